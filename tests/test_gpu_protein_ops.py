"""The 20-state traversal in double storage: op lists in every order a caller
may give, pattern counts around a wavefront's two sixteens, every category
count, both counter modes, rescaling beside patterns that have a +I mass and
are never rescaled, and alphabets whose tip lookups do and do not fit the staged
tables. Counters bit-exact and values to 1e-10 of the pattern's
largest against the oracle: a value is a chain of at most a few hundred
roundings of 1.1e-16, times the twenty terms of its sums."""
import numpy as np
import pytest

import iqtree2_amd as ia
from oracle.binding import OracleTree
from test_gpu_dna_ops import any_order
from test_gpu_parity import compare_partials

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ncat", [1, 2, 4, 8])
@pytest.mark.parametrize("safe", [False, True])
@pytest.mark.parametrize("npat,taxa,unknown", [(1, 3, 23), (17, 5, 40), (33, 30, 23), (129, 12, 24), (257, 6, 25)])
def test_orders_and_edges(ctx, ncat, safe, npat, taxa, unknown):
    print(f"ncat={ncat} safe={safe} npat={npat} taxa={taxa} unknown={unknown}", flush=True)
    w = ia.Workload(seq_type=ia.PROTEIN, ntaxa=taxa, nsite=max(npat, 4), ncat=ncat, mean_len=2.0, alpha=0.5,
                    gap_frac=0.1, seed=7 + npat)
    P = min(npat, w.npatterns)
    rng = np.random.default_rng(npat)
    m = w.model_arrays()
    # an alphabet of `unknown` states: some of the sequences' in new names
    states, tip = np.ascontiguousarray(w.get("states")[:, :P]), np.asarray(m["tip"]).reshape(-1, 20)
    more = unknown - w.state_unknown
    gap = states == w.state_unknown
    renamed = (states < more) & (rng.random(states.shape) < 0.5)
    states[renamed] += w.state_unknown
    states[gap] = unknown
    tip = np.concatenate([tip[:-1], tip[:more], tip[-1:]])
    args = (states, rng.integers(1, 5, P).astype(np.float64), np.zeros(P))
    inst = ia.Instance(ctx, taxa, 20, ncat, P, taxa, unknown, safe_numeric=safe)
    orc = OracleTree(taxa, 20, ncat, P, taxa, unknown, safe, 1)
    for x in (inst, orc):
        x.set_patterns(*args)
        x.set_model(m["eval"], m["evec"], m["inv_evec"], tip, m["rates"], m["props"])
    tree = ia.PhyloTree(None, w)
    try:
        for a, b in tree.branches()[::max(1, taxa // 3)]:
            ops, node, dad = tree.plan_full(a, b)
            length = tree.get_length(a, b)
            for trial in (ops, any_order(ops, rng), np.concatenate([any_order(ops, rng), ops])):
                lg, pg = inst.likelihood_branch(trial, node, dad, length, want_pattern_lh=True)
                lo, po = orc.likelihood_branch(ops, node, dad, length, want_pattern_lh=True)
                assert abs(lg - lo) <= 1e-9 * abs(lo)
                np.testing.assert_allclose(pg, po, rtol=0, atol=1e-9)
                compare_partials(inst, orc, ops)
    finally:
        tree.close()
        inst.close()


@pytest.mark.parametrize("ncat", [1, 2, 4, 8])
@pytest.mark.parametrize("safe", [False, True])
def test_rescaling_beside_invariable_sites(ctx, ncat, safe):
    print(f"ncat={ncat} safe={safe}", flush=True)
    w = ia.Workload(seq_type=ia.PROTEIN, ntaxa=120, nsite=80, ncat=ncat, mean_len=1.0, alpha=1.0, seed=78)
    P = min(70, w.npatterns)
    massed = np.arange(P) % 3 == 1
    m = w.model_arrays()
    inst = ia.Instance(ctx, 120, 20, ncat, P, 120, w.state_unknown, safe_numeric=safe)
    orc = OracleTree(120, 20, ncat, P, 120, w.state_unknown, safe, 2)
    for x in (inst, orc):
        x.set_patterns(np.ascontiguousarray(w.get("states")[:, :P]), np.ones(P), 0.01 * massed)
        x.set_model(m["eval"], m["evec"], m["inv_evec"], m["tip"], m["rates"], m["props"])
    tree = ia.PhyloTree(None, w)
    try:
        ops, node, dad = tree.plan_full(*tree.branches()[30])
        lg, pg = inst.likelihood_branch(ops, node, dad, 0.1, want_pattern_lh=True)
        lo, po = orc.likelihood_branch(ops, node, dad, 0.1, want_pattern_lh=True)
        assert abs(lg - lo) <= 1e-9 * abs(lo)
        np.testing.assert_allclose(pg, po, rtol=0, atol=1e-9)
        compare_partials(inst, orc, ops)
        counts = [inst.read_partial(int(op["dad_slot"]))[1] for op in ops]
        assert not any(c[massed].any() for c in counts)
        assert max(int(c.max()) for c in counts) > 0
    finally:
        tree.close()
        inst.close()
