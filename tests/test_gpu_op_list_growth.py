"""Op lists longer than the buffers of the last one, under a budget that holds
some of the new buffers only: the call is refused, the next short list runs in
buffers of its own, and the long one is refused again."""
import numpy as np
import pytest

import iqtree2_amd as ia

pytestmark = pytest.mark.gpu

PLK_ERR_NOMEM = 2
LONG = 4000


def instance(ctx, seq_type, precision):
    w = ia.Workload(seq_type=seq_type, ntaxa=12, nsite=90, ncat=4, seed=5)
    tree = ia.PhyloTree(None, w)
    a, b = next(e for e in tree.branches() if min(e) >= w.ntaxa)
    ops, node, dad = tree.plan_full(a, b)
    args = (node, dad, tree.get_length(a, b))
    tree.close()
    inst = ia.Instance.from_workload(ctx, w, precision=precision, safe_numeric=seq_type == ia.CODON)
    w.close()
    long = np.tile(ops, LONG // len(ops))
    return inst, ops, long, args


@pytest.mark.parametrize("seq_type,precision", [(ia.DNA, ia.PREC_F64), (ia.DNA, ia.PREC_F32), (ia.PROTEIN, ia.PREC_F64),
                                                (ia.PROTEIN, ia.PREC_F32), (ia.CODON, ia.PREC_F64)])
def test_refused_growth(seq_type, precision):
    with_room = ia.Context(0)
    inst, ops, long, args = instance(with_room, seq_type, precision)
    before = with_room.memory()[0]
    lnl = inst.likelihood_branch(ops, *args)
    short = with_room.memory()[0]
    assert inst.likelihood_branch(long, *args) == lnl
    whole = with_room.memory()[0]
    with_room.close()
    assert before < short < whole
    # the last one holds all but the last buffer
    budgets = sorted({short + (whole - short) * k // 6 for k in range(1, 6)} | {whole - 1})
    for budget in budgets:
        print(f"seq_type={seq_type} precision={precision} budget={budget} of {whole}", flush=True)
        ctx = ia.Context(0, hbm_budget=budget)
        try:
            inst, ops, long, args = instance(ctx, seq_type, precision)
            assert inst.likelihood_branch(ops, *args) == lnl
            for _ in range(2):
                with pytest.raises(ia.PlkError) as e:
                    inst.likelihood_branch(long, *args)
                assert e.value.status == PLK_ERR_NOMEM
                assert inst.likelihood_branch(ops, *args) == lnl
        finally:
            ctx.close()
