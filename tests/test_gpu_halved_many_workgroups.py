"""Halved steps in launches of more than 256 workgroups of 64 queries: the incomplete
second round of them is dealt in reverse over the runs that the XCDs get.  Every row
written, once: from outputs that hold NaN, against the 128-query form of the same call;
masks given as values also with the workgroups that scan them in front, bit for bit the call
whose workgroups scan for themselves."""
import pytest
import torch

from nntile_amd import hip_sdpa
from . import helpers as H

pytestmark = pytest.mark.gpu


def _inputs(head, batch, seq, dtype, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn(batch, seq, head, generator=gen, device="cuda").to(H.TORCH_DT[dtype]) for _ in range(3)]


def _nan_outputs(Q):
    return torch.full(Q.shape[:2], float("nan"), device="cuda"), torch.full_like(Q, float("nan"))


def _tile(K, Q, V, mask, mode, form, **kw):
    lse, A = _nan_outputs(Q)
    hip_sdpa.sdpa_fwd_tile(K, Q, mask, lse, V, A, mode, flags=form | hip_sdpa.OVERWRITE, **kw)
    torch.cuda.synchronize()
    return lse, A


def _close(got, want, dtype):
    row, off = H.row_errors(H.to_np(got[1]), H.to_np(want[1]), H.to_np(got[0]), H.to_np(want[0]))
    assert off < H.LSE_TOL[dtype], off
    assert row < H.ROW_TOL[dtype], row


def _same(a, b):
    assert torch.equal(a[0], b[0])
    assert torch.equal(a[1].view(torch.int16), b[1].view(torch.int16))


# 257, 300, 511, 513, 768 and 510 workgroups; batches that are and are not multiples of 8
@pytest.mark.parametrize("mode", ["causal", "none"])
@pytest.mark.parametrize("head,batch,seq,dtype", [
    (64, 257, 60, "bf16"), (64, 100, 190, "fp16"), (64, 73, 400, "bf16"), (64, 57, 570, "bf16"), (64, 64, 760, "fp16"),
    (64, 96, 500, "bf16"), (128, 257, 64, "fp16"), (128, 60, 310, "bf16"), (128, 73, 448, "fp16"), (128, 64, 512, "bf16"),
    (128, 51, 630, "bf16")])
def test_every_row_is_written(mode, head, batch, seq, dtype):
    print("case many", mode, head, batch, seq, dtype, flush=True)
    K, Q, V = _inputs(head, batch, seq, dtype, batch + seq)
    m = hip_sdpa.MASK_CAUSAL if mode == "causal" else hip_sdpa.MASK_NONE
    _close(_tile(K, Q, V, None, m, hip_sdpa.FORM_HALVED), _tile(K, Q, V, None, m, hip_sdpa.FORM_SHARED), dtype)


# launches that take the form by themselves, so that the call with a scratch, whose form
# cannot be asked for, has it too; blocks of 64 rows by fours make a number of scanning
# workgroups that is rounded up to a multiple of 8 (odd numbers of blocks)
@pytest.mark.parametrize("kind", ["causal", "window", "late"])
@pytest.mark.parametrize("head,batch,seq,dtype", [
    (64, 100, 190, "bf16"), (64, 72, 400, "fp16"), (64, 51, 600, "bf16"), (64, 64, 760, "bf16"), (64, 96, 500, "fp16"),
    (128, 16, 1537, "bf16"), (128, 11, 1600, "fp16"), (128, 3, 330, "bf16")])
def test_with_scanning_workgroups_in_front(kind, head, batch, seq, dtype):
    print("case many values", kind, head, batch, seq, dtype, flush=True)
    K, Q, V = _inputs(head, batch, seq, dtype, batch + seq)
    i, j = torch.arange(seq, device="cuda")[:, None], torch.arange(seq, device="cuda")[None, :]
    seen = {"causal": j <= i, "window": (i - j).abs() <= 32, "late": (j >= 70 + i // 8) | (j == i)}[kind]
    mask = H.additive_mask(seen.cpu().numpy(), dtype).cuda()
    lse, A = _nan_outputs(Q)
    lse.fill_(float("-inf"))
    hip_sdpa.flash_sdpa_fwd(K, Q, mask, lse, V, A, torch.empty_like(lse), torch.empty_like(A))
    torch.cuda.synchronize()
    _same((lse, A), _tile(K, Q, V, mask, hip_sdpa.MASK_ADDITIVE, hip_sdpa.FORM_HALVED))
    _close((lse, A), _tile(K, Q, V, mask, hip_sdpa.MASK_ADDITIVE, hip_sdpa.FORM_SHARED), dtype)
