"""Order of equal keys in the plan's task sort (qlt_plan_build): several hundred
tasks per output block, so that tasks of one block lie in different 256-task
chunks of the counting sort, and more than 32768 tasks in runs of equal keys,
which the radix sort takes.  The order inside a block decides which task is the
first to touch it (beta).  Integers: equal to the oracle's plan, field by field."""
import numpy as np
import pytest

from oracle import oracle as O
from tensortoolkit_amd.blocksparse import IN, OUT, BlockSparseTensor, ContractionPlan, Index

pytestmark = pytest.mark.gpu


def _pair(legs, sectors, groups):
    """Two tensors joined by two legs whose charges add up to those of `legs` legs
    of `sectors` charges each: `groups` tasks per output block."""
    left = [Index(tuple((q,) for q in range(sectors)), tuple(1 + q % 3 for q in range(sectors)), IN)
            for _ in range(legs)]
    top = legs * (sectors - 1)
    mid = Index(tuple((q,) for q in range(groups)), (1,) * groups, OUT)
    aux = Index(tuple((q - top,) for q in range(groups + top)), (1,) * (groups + top), IN)
    a = BlockSparseTensor.allowed_blocks([*left, aux, mid], (0,))
    b = BlockSparseTensor.allowed_blocks([mid.inverse(), aux.inverse(), *(x.inverse() for x in left)], (0,))
    return ContractionPlan(a, b, [legs, legs + 1], [1, 0]), O.OraclePlan(a, b, [legs, legs + 1], [1, 0])


# legs, sectors, groups, tasks: one block over three chunks and a remainder, blocks
# that begin inside chunks, the last count of the counting sort and counts beyond
@pytest.mark.parametrize("legs,sectors,groups,count", [
    (1, 1, 257, 257), (1, 1, 771, 771), (1, 2, 300, 600), (1, 5, 511, 2555), (2, 3, 300, 5700),
    (2, 4, 744, 32736), (2, 4, 745, 32780), (2, 8, 128, 44032)])
def test_equal_keys_keep_generation_order(qlt, legs, sectors, groups, count):
    print(f"case: plan sort ties {legs} {sectors} {groups} = {count} tasks", flush=True)
    plan, ref = _pair(legs, sectors, groups)
    got, exp = plan.tasks(), ref.tasks()
    assert len(got) == count
    assert len(np.unique(exp["c_blk_idx"])) * groups == count
    for name in got.dtype.names:
        np.testing.assert_array_equal(got[name], exp[name])
