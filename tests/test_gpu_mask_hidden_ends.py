"""Masks given as values whose first or last key steps are hidden for every
query of a workgroup: those steps are not walked.  Every tile type and
workgroup form, rows of any length, more steps than the scan has bits for,
against float64 arithmetic."""
import numpy as np
import pytest
import torch

from nntile_amd import hip_sdpa
from . import helpers as H

pytestmark = pytest.mark.gpu


def _mask(kind, q_seq, k_seq):
    i = np.arange(q_seq)[:, None]
    j = np.arange(k_seq)[None, :]
    if kind == "last":                      # one key of the last step
        return np.broadcast_to(j == k_seq - 1, (q_seq, k_seq)).copy()
    if kind == "middle":                    # a band away from both ends
        return (j >= k_seq // 3 + i % 5) & (j < k_seq // 2 + i % 3)
    if kind == "upper":                     # nothing for the first queries, the end for the others
        return (i >= q_seq // 2) & (j > k_seq // 4)
    return (j + 1 < 70) | (j == k_seq // 2 + i)     # the start and a moving key


@pytest.mark.parametrize("dtype", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("form", ["additive", "bool"])
@pytest.mark.parametrize("kind", ["last", "middle", "upper", "start"])
@pytest.mark.parametrize("q_seq,k_seq,head", [(33, 200, 64), (130, 333, 128), (40, 14, 64),
                                              (64, 2300, 64), (140, 4500, 32)])
@pytest.mark.parametrize("flags", [0, hip_sdpa.FORM_SHARED, hip_sdpa.FORM_SPLIT])
def test_hidden_ends(dtype, form, kind, q_seq, k_seq, head, flags):
    print("case hidden ends", dtype, form, kind, q_seq, k_seq, head, flags, flush=True)
    batch = 2
    (Q, K, V), f32 = H.make_qkv(71, batch, q_seq, k_seq, head, dtype)
    vis = _mask(kind, q_seq, k_seq)
    m = (H.additive_mask(vis, dtype) if form == "additive" else torch.from_numpy(vis.copy())).cuda()
    mode = hip_sdpa.MASK_ADDITIVE if form == "additive" else hip_sdpa.MASK_BOOL
    lse = torch.full((batch, q_seq), float("nan"), device="cuda")
    A = torch.full((batch, q_seq, head), float("nan"), dtype=Q.dtype, device="cuda")
    hip_sdpa.sdpa_fwd_tile(K.cuda(), Q.cuda(), m, lse, V.cuda(), A, mode,
                           flags=flags | hip_sdpa.OVERWRITE)
    torch.cuda.synchronize()
    q, k, v = (torch.from_numpy(np.ascontiguousarray(x)).double() for x in f32)
    s = q @ k.transpose(1, 2).contiguous() / head ** 0.5
    s = s.masked_fill(~torch.from_numpy(vis), float("-inf"))
    want_lse = torch.logsumexp(s, dim=-1)
    want = torch.nan_to_num(torch.softmax(s, dim=-1)) @ v
    seen = torch.from_numpy(vis.any(axis=1))
    assert torch.equal(torch.isneginf(lse.cpu()), (~seen)[None].expand(batch, -1))
    assert (A.cpu()[:, ~seen] == 0).all()
    tol = {"fp32": 1e-5, "bf16": 1e-2, "fp16": 2e-3}[dtype]
    assert H.rel_fro(H.to_np(A), want.numpy()) < tol
    assert H.rel_fro(lse.cpu()[:, seen].numpy(), want_lse[:, seen].numpy()) < 1e-4
