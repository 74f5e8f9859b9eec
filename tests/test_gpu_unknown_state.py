"""The unknown state at a tip: its transition is 1 for every state, whatever
the caller's row of tip vectors for it holds, in the reversible and the
state-basis traversals. Toward the root the matrix is transposed, and a
product with a row of ones would give its column sums instead.
Counters bit-exact and values to 1e-10 of the pattern's largest against the
oracle: a value is a chain of at most a few hundred roundings of 1.1e-16."""
import numpy as np
import pytest

import iqtree2_amd as ia
from oracle.binding import OracleTree
from refmath import indicators
from statebasis import categories, nonrev_model, plan
from test_gpu_parity import compare_partials
from test_oracle_nonrev import internal_branches

pytestmark = pytest.mark.gpu

ALPHABETS = [(ia.DNA, 18), (ia.PROTEIN, 23), (ia.PROTEIN, 24), (ia.PROTEIN, 25), (ia.PROTEIN, 40)]


def alignment(seq_type, unknown, ncat):
    """(workload, states): some of the sequences' states in the names that a
    larger alphabet has between the workload's and its unknown state."""
    w = ia.Workload(seq_type=seq_type, ntaxa=14, nsite=150, ncat=ncat, mean_len=0.4, gap_frac=0.3, seed=unknown + ncat)
    st = w.get("states").copy()
    if unknown != w.state_unknown:
        st[st == w.state_unknown] = unknown
    rng = np.random.default_rng(unknown)
    st[rng.random(st.shape) < 0.15] = unknown
    st[:2, ::3] = unknown
    return w, st


def tips(w, rows, unknown):
    """`rows` for an alphabet of `unknown` states: the new ones as the first."""
    more = unknown - w.state_unknown
    return np.concatenate([rows[:-1], rows[:max(more, 0)], rows[-1:]])


@pytest.mark.parametrize("ncat", [1, 2, 4, 8])
@pytest.mark.parametrize("seq_type,unknown", ALPHABETS)
def test_toward_the_root(ctx, seq_type, unknown, ncat):
    print(f"seq_type={seq_type} unknown={unknown} ncat={ncat}", flush=True)
    w, st = alignment(seq_type, unknown, ncat)
    nm = nonrev_model(w.nstates, 1, ncat, False, seed=3)
    assert len(categories(nm)) == ncat
    tip = tips(w, indicators(seq_type, w.nstates, w.state_unknown), unknown)
    inst = ia.Instance(ctx, w.ntaxa, w.nstates, ncat, st.shape[1], w.ntaxa, unknown)
    orc = OracleTree(w.ntaxa, w.nstates, ncat, st.shape[1], w.ntaxa, unknown, False, 2)
    for x in (inst, orc):
        x.set_patterns(st, w.get("freq"), np.zeros(st.shape[1]))
        x.set_model_nonrev(nm, tip, False)
    try:
        for a, b in internal_branches(w)[::3]:
            ops, node, dad, length = plan(w.ntaxa, w.edges(), a, b)
            ops = ops.copy()
            for c in ("c0", "c1"):
                ops[c + "_tip"][ops[c + "_tip"] == 1] = 3          # a tip, toward the root
            lg, pg = inst.likelihood_branch(ops, node, dad, length, want_pattern_lh=True)
            lo, po = orc.likelihood_branch(ops, node, dad, length, want_pattern_lh=True)
            compare_partials(inst, orc, ops)
            assert abs(lg - lo) <= 1e-9 * abs(lo)
            np.testing.assert_allclose(pg, po, rtol=0, atol=1e-9)
    finally:
        inst.close()


@pytest.mark.parametrize("ncat", [1, 2, 4, 8])
@pytest.mark.parametrize("seq_type,unknown", ALPHABETS)
def test_row_of_the_unknown_state_is_not_read(ctx, seq_type, unknown, ncat):
    print(f"seq_type={seq_type} unknown={unknown} ncat={ncat}", flush=True)
    w, st = alignment(seq_type, unknown, ncat)
    m = w.model_arrays()
    rows = tips(w, np.asarray(m["tip"]).reshape(-1, w.nstates), unknown)
    other = rows.copy()
    other[-1] = 7.0
    orc = OracleTree(w.ntaxa, w.nstates, ncat, st.shape[1], w.ntaxa, unknown, False, 2)
    insts = [ia.Instance(ctx, w.ntaxa, w.nstates, ncat, st.shape[1], w.ntaxa, unknown) for _ in range(2)]
    for x, tip in zip((orc, *insts), (rows, rows, other)):
        x.set_patterns(st, w.get("freq"), w.get("invar"))
        x.set_model(m["eval"], m["evec"], m["inv_evec"], tip, m["rates"], m["props"])
    tree = ia.PhyloTree(None, w)
    try:
        # a tip at the branch's end is another matter: there the row is the state's vector
        a, b = next(e for e in internal_branches(w) if min(e) >= w.ntaxa)
        ops, node, dad = tree.plan_full(a, b)
        length = tree.get_length(a, b)
        out = [x.likelihood_branch(ops, node, dad, length, want_pattern_lh=True) for x in (orc, *insts)]
        assert abs(out[1][0] - out[0][0]) <= 1e-9 * abs(out[0][0])
        assert out[1][0] == out[2][0]
        np.testing.assert_array_equal(out[1][1], out[2][1])
        compare_partials(insts[0], orc, ops)
        compare_partials(insts[1], orc, ops)
    finally:
        tree.close()
        for x in insts:
            x.close()
