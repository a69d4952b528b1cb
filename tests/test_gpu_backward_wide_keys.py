"""Key-owning workgroups that hold dK and dV at head 128 (a launch of more than
512 workgroups under an analytic mask) against the same entries in launches that
keep the two apart: walks of less than 13 steps, which both take in one group of
wavefronts, so the sums are the same and the gradients agree bit for bit.  Sizes at the edges of a step of 64 queries and of a workgroup's 128 keys."""
import pytest
import torch

from nntile_amd import hip_sdpa
from . import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("mode", ["none", "causal"])
@pytest.mark.parametrize("q_seq,k_seq,entries,group", [
    (1, 1, 180, 1), (63, 129, 180, 1), (64, 128, 180, 1), (65, 127, 180, 1), (200, 130, 130, 1),
    (129, 257, 128, 1), (130, 70, 96, 4)])
def test_both_gradients_in_one_workgroup(dtype, mode, q_seq, k_seq, entries, group, head=128, part=8):
    print("case bwd wide", dtype, mode, q_seq, k_seq, entries, group, flush=True)
    m = hip_sdpa.MASK_NONE if mode == "none" else hip_sdpa.MASK_CAUSAL
    offset = k_seq - q_seq
    batch = entries * group
    torch.manual_seed(q_seq + k_seq)
    kind = {"bf16": torch.bfloat16, "fp16": torch.float16}[dtype]
    K, V = (torch.randn(entries, k_seq, head, device="cuda").to(kind) for _ in range(2))
    Q, G = (torch.randn(batch, q_seq, head, device="cuda").to(kind) for _ in range(2))
    lse, A = H.fresh_outputs(batch, q_seq, head, dtype)

    # the batch entries of one key-value head side by side: [n_head_kv, group], n_batch = 1
    def call(first, last):
        q = slice(first * group, last * group)
        args = [t.contiguous() for t in (K[first:last], Q[q], V[first:last])]
        l, a = H.fresh_outputs((last - first) * group, q_seq, head, dtype)
        hip_sdpa.sdpa_fwd_tile(args[0], args[1], None, l, args[2], a, m, n_batch=1, kv_group=group,
                               causal_offset=offset, flags=hip_sdpa.OVERWRITE)
        out = [torch.full_like(t, float("nan")) for t in args]
        hip_sdpa.sdpa_bwd_tile(*args, a, G[q].contiguous(), None, l, *out, m, n_batch=1,
                               kv_group=group, causal_offset=offset, flags=hip_sdpa.OVERWRITE)
        torch.cuda.synchronize()
        return out

    whole = call(0, entries)
    parts = [call(i, min(i + part, entries)) for i in range(0, entries, part)]
    for i, name in enumerate(("dK", "dQ", "dV")):
        want = torch.cat([p[i] for p in parts])
        assert torch.isfinite(want).all(), name
        assert torch.equal(whole[i], want), name
