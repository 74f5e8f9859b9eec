"""The 4-state traversal on the matrix cores: op lists in every order a caller
may give (a child from the last step, the one before, or memory; a slot written
twice), pattern counts around the wavefront's chunks, every category count,
both counter modes and storages; rescaling beside patterns that have a +I mass
and are never rescaled; and slots gigabytes apart.
Double storage: counters bit-exact and values to 1e-10 of the pattern's largest
against the oracle: a value is a chain of at most a few hundred roundings of
1.1e-16. Float storage rescales by other powers of two: every order gives the
planner's bits, and its pattern lnL is the oracle's to 2e-4 (40 steps of ten
roundings of 6e-8, in a basis of condition below ten), lnL to 2e-6 of itself."""
import numpy as np
import pytest

import iqtree2_amd as ia
from oracle.binding import OracleTree
from test_gpu_parity import compare_partials

pytestmark = pytest.mark.gpu


def any_order(ops, rng):
    """The ops in a random order that keeps children before their dads."""
    left, done, out = list(range(len(ops))), set(), []
    writes = {int(o["dad_slot"]) for o in ops}
    while left:
        free = [k for k in left if all(ops[k][c + "_tip"] or int(ops[k][c + "_id"]) in done or
                                       int(ops[k][c + "_id"]) not in writes for c in ("c0", "c1"))]
        k = free[int(rng.integers(len(free)))]
        left.remove(k)
        done.add(int(ops[k]["dad_slot"]))
        out.append(k)
    return ops[out]


@pytest.mark.parametrize("ncat", [1, 2, 4, 8])
@pytest.mark.parametrize("safe", [False, True])
@pytest.mark.parametrize("precision", [ia.PREC_F64, ia.PREC_F32])
@pytest.mark.parametrize("npat,taxa", [(1, 3), (15, 4), (64, 5), (257, 40)])
def test_orders_and_edges(ctx, ncat, safe, precision, npat, taxa):
    print(f"ncat={ncat} safe={safe} precision={precision} npat={npat} taxa={taxa}", flush=True)
    w = ia.Workload(seq_type=ia.DNA, ntaxa=taxa, nsite=max(npat, 4), ncat=ncat, mean_len=2.0, alpha=0.5, gap_frac=0.1,
                    seed=31 + npat)
    P = min(npat, w.npatterns)
    rng = np.random.default_rng(npat)
    m = w.model_arrays()
    freq = rng.integers(1, 5, P).astype(np.float64)
    args = (np.ascontiguousarray(w.get("states")[:, :P]), freq, np.zeros(P))
    inst = ia.Instance(ctx, taxa, 4, ncat, P, taxa, w.state_unknown, precision, safe)
    f64 = precision == ia.PREC_F64
    orc = OracleTree(taxa, 4, ncat, P, taxa, w.state_unknown, safe, 1)
    for x in (inst, orc):
        x.set_patterns(*args)
        x.set_model(m["eval"], m["evec"], m["inv_evec"], m["tip"], m["rates"], m["props"])
    tree = ia.PhyloTree(None, w)
    try:
        for a, b in tree.branches()[::max(1, taxa // 5)]:
            ops, node, dad = tree.plan_full(a, b)
            length = tree.get_length(a, b)
            lo, po = orc.likelihood_branch(ops, node, dad, length, want_pattern_lh=True)
            first = None
            # in the last list every slot is written twice
            for trial in (ops, any_order(ops, rng), np.concatenate([any_order(ops, rng), ops])):
                lg, pg = inst.likelihood_branch(trial, node, dad, length, want_pattern_lh=True)
                assert abs(lg - lo) <= (1e-9 if f64 else 2e-6) * abs(lo)
                np.testing.assert_allclose(pg, po, rtol=0, atol=1e-9 if f64 else 2e-4)
                if f64:
                    compare_partials(inst, orc, ops)
                slots = [inst.read_partial(int(op["dad_slot"])) for op in ops]
                first = first or slots
                for (v, c), (v0, c0) in zip(slots, first):
                    np.testing.assert_array_equal(v, v0)
                    np.testing.assert_array_equal(c, c0)
    finally:
        tree.close()
        inst.close()


@pytest.mark.parametrize("ncat", [1, 2, 4, 8])
@pytest.mark.parametrize("safe", [False, True])
@pytest.mark.parametrize("precision", [ia.PREC_F64, ia.PREC_F32])
def test_rescaling_beside_invariable_sites(ctx, ncat, safe, precision):
    """160 taxa far apart: every pattern falls below the threshold; those with
    a +I mass are not rescaled, the others beside them are. Float storage, where
    they underflow: the counters of the others as without any mass."""
    print(f"ncat={ncat} safe={safe} precision={precision}", flush=True)
    w = ia.Workload(seq_type=ia.DNA, ntaxa=160, nsite=100, ncat=ncat, mean_len=2.0, alpha=1.0, seed=77)
    P = min(90, w.npatterns)
    massed = np.arange(P) % 3 == 1
    m = w.model_arrays()
    args = (np.ascontiguousarray(w.get("states")[:, :P]), np.ones(P))
    inst = ia.Instance(ctx, 160, 4, ncat, P, 160, w.state_unknown, precision, safe)
    other = ia.Instance(ctx, 160, 4, ncat, P, 160, w.state_unknown, precision, safe)
    orc = OracleTree(160, 4, ncat, P, 160, w.state_unknown, safe, 2)
    for x, mass in ((inst, 0.01 * massed), (orc, 0.01 * massed), (other, np.zeros(P))):
        x.set_patterns(*args, mass)
        x.set_model(m["eval"], m["evec"], m["inv_evec"], m["tip"], m["rates"], m["props"])
    tree = ia.PhyloTree(None, w)
    try:
        ops, node, dad = tree.plan_full(*tree.branches()[40])
        for x in (inst, other, orc):
            x.likelihood_branch(ops, node, dad, 0.1)
        most = 0
        for op in ops:
            (v, c), (v0, c0) = (x.read_partial(int(op["dad_slot"])) for x in (inst, other))
            assert not c[massed].any()
            np.testing.assert_array_equal(c[~massed], c0[~massed])
            np.testing.assert_array_equal(v[~massed], v0[~massed])
            most = max(most, int(np.abs(c).max()))
        assert most > 0
        if precision == ia.PREC_F64:
            compare_partials(inst, orc, ops)
    finally:
        tree.close()
        inst.close()
        other.close()


@pytest.mark.parametrize("precision,nslots", [(ia.PREC_F64, (1 << 21) + 3), (ia.PREC_F32, (1 << 22) + 3)])
def test_far_chunks(ctx, precision, nslots):
    """The same bits from an instance whose slots are gigabytes apart."""
    w = ia.Workload(seq_type=ia.DNA, ntaxa=9, nsite=300, ncat=1, mean_len=0.3, gap_frac=0.05, seed=3)
    tree = ia.PhyloTree(None, w)
    a, b = tree.branches()[4]
    ops, node, dad = tree.plan_full(a, b)
    length = tree.get_length(a, b)
    tree.close()
    out = []
    for n in (w.ntaxa, nslots):
        print(f"precision={precision} slots={n}", flush=True)
        inst = ia.Instance(ctx, w.ntaxa, 4, 1, w.npatterns, n, w.state_unknown, precision)
        m = w.model_arrays()
        inst.set_patterns(w.get("states"), w.get("freq"), w.get("invar"))
        inst.set_model(m["eval"], m["evec"], m["inv_evec"], m["tip"], m["rates"], m["props"])
        far = ops.copy()
        shift = n - w.ntaxa          # slots at the end of the range
        far["dad_slot"] += shift
        for c in ("c0", "c1"):
            far[c + "_id"] += np.where(far[c + "_tip"] == 0, shift, 0).astype(np.int32)
        ends = [ia.end(e.is_tip, e.id + (0 if e.is_tip else shift)) for e in (node, dad)]
        lnl, pat = inst.likelihood_branch(far, *ends, length, want_pattern_lh=True)
        part, count = inst.read_partial(int(far["dad_slot"][-1]))
        batch = ia.likelihood_branch_batch(ctx, [(inst, far, *ends, length)])[0]
        out.append((lnl, pat, part, count, batch))
        inst.close()
    for x, y in zip(*out):
        np.testing.assert_array_equal(x, y)
