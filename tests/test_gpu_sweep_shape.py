"""Workgroups of a device Newton pass: one a CU for a 4-state tree of up to four
tiles a CU, else two, and as many as PLK_SWEEP_BLOCKS_PER_CU says where it is
set, whatever the size. A pass is reproducible to the bit with the same
workgroups; with others its sums are added in another order."""
import numpy as np
import pytest

import iqtree2_amd as ia
from test_gpu_parity import context_with

pytestmark = pytest.mark.gpu


def sweep(ctx, w):
    tree = ia.PhyloTree(ctx, w)
    lnl, n = tree.optimize_all_branches(iterations=1, tolerance=1e-3, max_nr=100)
    out = np.array([lnl] + [tree.get_length(a, b) for a, b in tree.branches()])
    tree.close()
    return n, out


def test_workgroups_per_cu(ctx):
    # 8 categories: tiles of 32 patterns, 296 of them: more than one and fewer than two a CU
    w = ia.Workload(seq_type=ia.DNA, ntaxa=20, nsite=13000, ncat=8, mean_len=0.3, seed=4)
    assert 256 < w.npatterns / 32 < 512
    n, values = sweep(ctx, w)
    for blocks in (1, 2):
        other = context_with({"PLK_SWEEP_BLOCKS_PER_CU": str(blocks)})
        try:
            m, got = sweep(other, w)
        finally:
            other.close()
        assert m == n
        np.testing.assert_allclose(got, values, rtol=1e-9, atol=1e-12)
        assert np.array_equal(got, values) == (blocks == 1)
