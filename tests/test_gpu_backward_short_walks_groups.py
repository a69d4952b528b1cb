"""The backward of short walks, without a launch in front, where a group has many heads of
few rows: their row dots are taken in one run over the group.  Against 64-bit arithmetic,
and with several batch entries - a group's heads do not lie one behind the other then - bit
for bit the call with the launch in front."""
import pytest

from .test_gpu_backward_halved_steps import MODES, _case
from .test_gpu_backward_short_walks import test_same_bits_as_with_the_launch_in_front as same_bits

pytestmark = pytest.mark.gpu
# head, group, q_seq, k_seq: the edges of a run of rows (32 and 16 at a time by 256 threads)
# fall within heads, between them, and on the last
SHAPES = [(64, 128, 1, 100), (64, 127, 1, 128), (64, 16, 8, 128), (64, 5, 25, 64), (64, 11, 3, 70), (64, 8, 16, 1),
          (128, 16, 8, 128), (128, 128, 1, 64), (128, 9, 14, 128)]


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("mode", sorted(MODES))
@pytest.mark.parametrize("head,group,q_seq,k_seq", SHAPES)
def test_groups_of_many_heads(dtype, mode, head, group, q_seq, k_seq):
    print("case bwd short groups", dtype, mode, head, group, q_seq, k_seq, flush=True)
    _case(mode, head, group, 2, q_seq, k_seq, dtype, False)


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("mode", ["none", "causal"])
@pytest.mark.parametrize("head,group,q_seq,k_seq", SHAPES)
def test_groups_of_several_batch_entries(dtype, mode, head, group, q_seq, k_seq):
    same_bits(dtype, mode, head, group, q_seq, k_seq)
