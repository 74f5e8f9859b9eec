"""A slot's values and counters as the interface gives them, of more patterns
than are fetched at a time: an alignment whose columns repeat gives the same
bits in every repeat, and with and without the values. 160 taxa far apart, so
that counters are not zero."""
import numpy as np
import pytest

import iqtree2_amd as ia

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seq_type,precision,ncat,safe,repeats",
                         [(ia.DNA, ia.PREC_F64, 8, False, 300), (ia.DNA, ia.PREC_F32, 4, True, 700),
                          (ia.DNA, ia.PREC_F64, 1, False, 2500), (ia.PROTEIN, ia.PREC_F64, 4, True, 150),
                          (ia.PROTEIN, ia.PREC_F64, 2, False, 270), (ia.PROTEIN, ia.PREC_F32, 4, False, 150)])
def test_pieces(ctx, seq_type, precision, ncat, safe, repeats):
    print(f"seq_type={seq_type} precision={precision} ncat={ncat} safe={safe} repeats={repeats}", flush=True)
    w = ia.Workload(seq_type=seq_type, ntaxa=160, nsite=150, ncat=ncat, mean_len=2.0, gap_frac=0.1, seed=9)
    P = 113
    m = w.model_arrays()
    tree = ia.PhyloTree(None, w)
    ops, node, dad = tree.plan_full(*tree.branches()[3])
    tree.close()
    out = []
    for r in (1, repeats):
        inst = ia.Instance(ctx, w.ntaxa, w.nstates, ncat, P * r, w.ntaxa, w.state_unknown, precision, safe)
        inst.set_patterns(np.tile(w.get("states")[:, :P], r), np.ones(P * r), np.zeros(P * r))
        inst.set_model(m["eval"], m["evec"], m["inv_evec"], m["tip"], m["rates"], m["props"])
        inst.likelihood_branch(ops, node, dad, 0.1)
        slot = int(ops["dad_slot"][-1])
        values, counts = inst.read_partial(slot)
        none, again = inst.read_partial(slot, partial=False)
        assert none is None
        np.testing.assert_array_equal(counts, again)
        out.append((values, counts))
        inst.close()
    for one, many in zip(*out):
        assert np.count_nonzero(one)
        np.testing.assert_array_equal(np.tile(one, (repeats,) + (1,) * (one.ndim - 1)), many)
