"""The bytes that a profile charges to a traversal: child partials and counters
only where the kernel reads them, not where it still has them from the last
step (4 states: the last two)."""
import pytest

import iqtree2_amd as ia

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seq_type,precision,kept", [(ia.DNA, ia.PREC_F64, 2), (ia.DNA, ia.PREC_F32, 2),
                                                     (ia.PROTEIN, ia.PREC_F64, 1), (ia.PROTEIN, ia.PREC_F32, 0)])
def test_children_in_registers(ctx, seq_type, precision, kept):
    w = ia.Workload(seq_type=seq_type, ntaxa=30, nsite=200, ncat=4, seed=8)
    tree = ia.PhyloTree(None, w)
    a, b = next(e for e in tree.branches() if min(e) >= w.ntaxa)
    ops, node, dad = tree.plan_full(a, b)
    length = tree.get_length(a, b)
    tree.close()
    elem, count = (4, 4) if precision == ia.PREC_F32 else (8, 2)
    slot = w.nstates * 4 * elem + count
    expected = 0
    for o, op in enumerate(ops):
        have = {int(x["dad_slot"]) for x in ops[max(0, o - kept):o]}
        for c in ("c0", "c1"):
            expected += 1 if op[c + "_tip"] else 0 if int(op[c + "_id"]) in have else slot
        expected += slot
    inst = ia.Instance.from_workload(ctx, w, precision=precision)
    ctx.profile_start()
    inst.likelihood_branch(ops, node, dad, length)
    prof = ctx.profile_stop()
    inst.close()
    if seq_type == ia.DNA:
        got = prof["traverse+lnl"]["bytes"] / w.npatterns - 2 * slot - 24      # the branch's ends, weight, +I mass, lnL
    else:
        got = prof["traverse_mfma"]["bytes"] / w.npatterns
    assert got == pytest.approx(expected, rel=1e-9)
