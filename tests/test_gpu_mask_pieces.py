"""Masks given as values reach the lanes that apply them as pieces of eight
elements, moved back and shifted where a row ends inside one: row lengths around
a piece, a half step and a step, with values of every kind in each place."""
import numpy as np
import pytest
import torch

from nntile_amd import hip_sdpa
from . import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("form", ["additive", "bool"])
@pytest.mark.parametrize("q_seq,k_seq", [(1, 1), (3, 2), (33, 7), (16, 8), (17, 9), (40, 31), (64, 33),
                                         (65, 63), (31, 64), (130, 65), (129, 71), (48, 72), (97, 129),
                                         (128, 191), (200, 201)])
def test_every_element_of_a_row_is_applied_in_its_place(dtype, form, q_seq, k_seq):
    print("case pieces", dtype, form, q_seq, k_seq, flush=True)
    batch, head = 2, 64
    (Q, K, V), f32 = H.make_qkv(5, batch, q_seq, k_seq, head, dtype)
    rng = np.random.default_rng(1000 * q_seq + k_seq)
    seen = rng.random((q_seq, k_seq)) < 0.6
    if form == "additive":
        # (values that are exact in both tile types)
        values = np.where(seen, rng.integers(-8, 9, (q_seq, k_seq)) / 4.0, -np.inf)
        m = torch.from_numpy(values).to(H.TORCH_DT[dtype]).cuda()
    else:
        values = np.where(seen, 0.0, -np.inf)
        m = torch.from_numpy(seen).cuda()
    mode = hip_sdpa.MASK_ADDITIVE if form == "additive" else hip_sdpa.MASK_BOOL
    q, k, v = (torch.from_numpy(x).double() for x in f32)
    s = q @ k.transpose(1, 2) / head ** 0.5 + torch.from_numpy(values)
    want_lse = torch.logsumexp(s, dim=2)
    want = torch.nan_to_num(torch.softmax(s, dim=2)) @ v
    lse, A = H.fresh_outputs(batch, q_seq, head, dtype)
    hip_sdpa.sdpa_fwd_tile(K.cuda(), Q.cuda(), m, lse, V.cuda(), A, mode, flags=hip_sdpa.OVERWRITE)
    torch.cuda.synchronize()
    # (the bounds of the other tests: a value in another's place moves a row's
    # logsumexp by tenths, a rounding by 1e-6 of it)
    row, off = H.row_errors(H.to_np(A), want.numpy(), H.to_np(lse), want_lse.numpy())
    assert off < H.LSE_TOL[dtype], off
    assert row < H.ROW_TOL[dtype], row
