"""fp32 tiles of head 64 on the fp16 matrix units in workgroups of two query blocks
and four key blocks (NNTILE_HIP_SDPA_FORM_HALVED; what launches of few workgroups and
a thousand keys take): against 64-bit arithmetic at the edges of its steps of 128 keys,
no further off than with two key blocks, and the values that pieces do not carry."""
import pytest
import torch

from nntile_amd import hip_sdpa
from . import helpers as H
from .test_gpu_fp32_on_fp16_units import FP32, call, draw, reference, rel

pytestmark = pytest.mark.gpu

TWO_BY_FOUR, TWO_BY_TWO = hip_sdpa.FORM_HALVED, hip_sdpa.FORM_WIDE | hip_sdpa.FORM_SPLIT


# one key; a key block's edges; a step's; odd and even numbers of passes; a last row
# of one query
@pytest.mark.parametrize("mode", ["none", "causal", "additive", "bool"])
@pytest.mark.parametrize("q_seq,k_seq", [(1, 1), (33, 31), (64, 97), (65, 128), (70, 129), (129, 384), (64, 385),
                                         (200, 1000)])
def test_against_64_bits(mode, q_seq, k_seq):
    print("case 2x4", mode, q_seq, k_seq, flush=True)
    Q, K, V = draw(q_seq * 7 + k_seq, 3, q_seq, k_seq, 64)
    offset = k_seq - q_seq
    q, k = torch.arange(q_seq)[:, None], torch.arange(k_seq)[None]
    seen, m, mm = None, None, hip_sdpa.MASK_NONE
    if mode == "causal":
        seen, mm = k <= q + offset, hip_sdpa.MASK_CAUSAL
    elif mode != "none":        # a window, and rows that see nothing
        seen = ((k - q - offset).abs() <= 70) & (q % 17 != 3)
        mm = hip_sdpa.MASK_ADDITIVE if mode == "additive" else hip_sdpa.MASK_BOOL
        m = (H.additive_mask(seen.numpy(), "fp32") if mode == "additive" else seen.clone()).cuda()
    A, lse = call(Q, K, V, mm, TWO_BY_FOUR, m, offset)
    wantA, want = reference(Q, K, V, seen)
    hidden = torch.isinf(want)
    assert torch.equal(torch.isinf(lse), hidden) and (A[hidden] == 0).all()
    if not bool(hidden.all()):
        # (the bounds of the other forms)
        assert rel(A[~hidden], wantA[~hidden]) < 1e-6
        assert float((lse[~hidden] - want[~hidden]).abs().max()) < 1e-6 * (1 + float(want[~hidden].abs().max()))


@pytest.mark.parametrize("mean", [0.0, 1.0])
@pytest.mark.parametrize("batch,seq", [(12, 1024), (6, 2000), (3, 4100), (16, 1000)])
def test_no_further_off_than_with_two_key_blocks(batch, seq, mean):
    """A wavefront walks half as many keys, so its sums are the shorter ones; 5 % for the
    scatter of the norms.  By themselves the launches take this form."""
    Q, K, V = draw(seq, batch, seq, seq, 64)
    V += mean
    seen = torch.ones(seq, seq, dtype=torch.bool).tril()
    for mode, mask in ((hip_sdpa.MASK_CAUSAL, seen), (hip_sdpa.MASK_NONE, None)):
        wantA, want = reference(Q[:2], K[:2], V[:2], mask)
        A, lse = call(Q, K, V, mode, TWO_BY_FOUR)
        A0, lse0 = call(Q, K, V, mode, 0)
        assert torch.equal(A0, A) and torch.equal(lse0, lse)
        A2, lse2 = call(Q, K, V, mode, TWO_BY_TWO)
        four, two = rel(A[:2], wantA), rel(A2[:2], wantA)
        print("%d x %d mean %g mode %d: %.2e, two key blocks %.2e; lse %.2e, %.2e" % (
            batch, seq, mean, mode, four, two, rel(lse[:2], want), rel(lse2[:2], want)), flush=True)
        assert four < 1.05 * two
        assert rel(lse[:2], want) < 1.05 * rel(lse2[:2], want)


@pytest.mark.parametrize("what", ["large later", "small later", "tiny rows", "infinite key"])
def test_values_that_pieces_do_not_carry(what):
    Q, K, V = draw(31, 2, 130, 700, 64)
    if what == "large later":
        V[:, 300:] *= 1e4
    elif what == "small later":
        V[:, 128:] *= 1e-6
        K[:, :128] = -Q[:, :1] * 30
    elif what == "tiny rows":
        K[:, 1:] *= 1e-3
        V[:, :, 5] *= 1e-9
    else:
        K[0, 600, 3] = float("inf")
    A, lse = call(Q, K, V, hip_sdpa.MASK_NONE, TWO_BY_FOUR)
    A32, lse32 = call(Q, K, V, hip_sdpa.MASK_NONE, FP32)
    if what == "infinite key":
        assert torch.equal(torch.isnan(A), torch.isnan(A32)) and torch.equal(torch.isnan(lse), torch.isnan(lse32))
        return
    wantA, want = reference(Q, K, V, None)
    # (within twice the error of fp32 products, as the other forms; each channel by itself)
    for d in range(64):
        assert rel(A[:, :, d], wantA[:, :, d]) < 2 * rel(A32[:, :, d], wantA[:, :, d]) + 1e-7, d
    assert rel(lse, want) < 2 * rel(lse32, want)
