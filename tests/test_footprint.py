"""The memory an instance asks for: one scale counter a pattern (safe mode: one
a pattern and category) and no slots beyond those asked for, so that a shape
that fits a budget is not refused for a layout's sake. Sizes are chosen so
that partials and counters are whole allocation classes."""
import ctypes

import pytest

import iqtree2_amd as ia
from iqtree2_amd import _capi


def footprint(nstates, ncat, P, nslots, unknown, precision, safe):
    d = _capi.PlkInstanceDesc(ntaxa=8, nstates=nstates, ncat=ncat, npatterns=P, nslots=nslots, state_unknown=unknown,
                              precision=precision, safe_numeric=int(safe))
    return _capi.lib().plk_instance_footprint(ctypes.byref(d))


@pytest.mark.parametrize("safe", [False, True])
@pytest.mark.parametrize("precision,elem,count", [(ia.PREC_F64, 8, 2), (ia.PREC_F32, 4, 4)])
@pytest.mark.parametrize("nstates,unknown", [(4, 18), (20, 23)])
@pytest.mark.parametrize("ncat", [1, 2, 4, 8])
def test_slots_and_counters(nstates, unknown, ncat, precision, elem, count, safe):
    P, few, many = 8192, 8, 16
    grown = footprint(nstates, ncat, P, many, unknown, precision, safe) - footprint(nstates, ncat, P, few, unknown,
                                                                                    precision, safe)
    partials = (many - few) * P * nstates * ncat * elem
    counters = (many - few) * P * (ncat if safe else 1) * count
    # and the op list of eight more nodes, with its tables
    assert partials + counters <= grown <= partials + counters + (1 << 20)
