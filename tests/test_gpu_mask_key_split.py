"""Masks given as values at head 64: from sixteen key steps on a launch of few
workgroups walks them in two groups of wavefronts, scanned by workgroups of the same
launch.  Sizes at that line, against 64-bit arithmetic."""
import numpy as np
import pytest
import torch

from nntile_amd import hip_sdpa
from . import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("kind", ["causal", "window", "full", "late"])
@pytest.mark.parametrize("seq,batch", [(960, 2), (1023, 2), (1024, 3), (1025, 2), (1100, 4)])
def test_tasks_of_head_64_at_sixteen_key_steps(dtype, kind, seq, batch):
    print("case key split", dtype, kind, seq, batch, flush=True)
    head = 64
    i, j = np.arange(seq)[:, None], np.arange(seq)[None, :]
    seen = {"causal": j <= i, "window": np.abs(i - j) <= 32, "full": (i >= 0) & (j >= 0),
            "late": j >= 200 + i // 8}[kind]
    (Q, K, V), f32 = H.make_qkv(9, batch, seq, seq, head, dtype)
    q, k, v = (torch.from_numpy(x).double() for x in f32)
    s = (q @ k.transpose(1, 2) / head ** 0.5).masked_fill(~torch.from_numpy(seen), float("-inf"))
    want, want_lse = torch.softmax(s, dim=2) @ v, torch.logsumexp(s, dim=2)
    lse, A = H.fresh_outputs(batch, seq, head, dtype)
    scratch = torch.empty(batch, seq, device="cuda")
    hip_sdpa.flash_sdpa_fwd(K.cuda(), Q.cuda(), H.additive_mask(seen, dtype).cuda(), lse, V.cuda(), A,
                            scratch, torch.empty_like(A))
    torch.cuda.synchronize()
    row, off = H.row_errors(H.to_np(A), want.numpy(), H.to_np(lse), want_lse.numpy())
    assert off < H.LSE_TOL[dtype], off
    assert row < H.ROW_TOL[dtype], row
