"""fp32 tiles on the fp16 matrix units: values that two fp16 pieces under a common
power of two do not carry, in every place where they can hide."""
import math

import pytest
import torch

from nntile_amd import hip_sdpa

pytestmark = pytest.mark.gpu

S, P, W = hip_sdpa.FORM_SHARED, hip_sdpa.FORM_SPLIT, hip_sdpa.FORM_WIDE
# query blocks of 32 x key blocks of 32 of a workgroup
FORMS = {"2x2": W | P, "4x1": S, "4x2": W | S, "8x1": W}
FP32 = P        # the fp32 kernel


def draw(seed, batch, q_seq, k_seq, head):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn(batch, n, head, generator=g) for n in (q_seq, k_seq, k_seq)]


def call(Q, K, V, mode, flags):
    lse = torch.zeros(Q.shape[:2], device="cuda")
    A = torch.zeros_like(Q, device="cuda")
    hip_sdpa.sdpa_fwd_tile(K.cuda(), Q.cuda(), None, lse, V.cuda(), A, mode, flags=flags | hip_sdpa.OVERWRITE)
    torch.cuda.synchronize()
    return A.cpu(), lse.cpu()


def check(Q, K, V, form, mode=hip_sdpa.MASK_NONE):
    """By rows and by channels, against 64 bits, and against what fp32 products are
    off by: twice that in the mean, four times the largest (the bounds of the other
    ranges' test: sums of up to four times the keys in one accumulator)."""
    q, k, v = (t.double() for t in (Q, K, V))
    s = torch.matmul(q, k.transpose(1, 2).contiguous()) / math.sqrt(Q.shape[2])
    if mode == hip_sdpa.MASK_CAUSAL:
        s = s.masked_fill(torch.ones(s.shape[1:], dtype=torch.bool).triu(1), float("-inf"))
    want_lse = torch.logsumexp(s, 2)
    want = torch.matmul(torch.exp(s - want_lse[..., None]), v)
    (A, lse), (A32, lse32) = call(Q, K, V, mode, FORMS[form]), call(Q, K, V, mode, FP32)
    for dim in (1, 2):
        norm = want.norm(dim=dim).clamp_min(1e-300)
        err, err32 = ((x.double() - want).norm(dim=dim) / norm for x in (A, A32))
        print(form, dim, "mean %.2e, fp32 %.2e; largest %.2e, fp32 %.2e"
              % (err.mean(), err32.mean(), err.max(), err32.max()), flush=True)
        assert float(err.mean()) < 2 * float(err32.mean())
        assert float(err.max()) < 4 * float(err32.max())
    assert float((lse - want_lse).abs().max()) < 2 * float((lse32 - want_lse).abs().max()) + 1e-6


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("head", [64, 128])
@pytest.mark.parametrize("what", ["query 1e5", "query 1e7", "query 1e9", "half of the channels",
                                  "key 1e5", "key -1e6", "key -1e9", "later key -1e7"])
def test_scores_of_a_large_channel_against_a_small_one(form, head, what):
    print("case", form, head, what, flush=True)
    Q, K, V = draw(5, 2, 130, 700, head)
    if what == "half of the channels":
        Q[..., ::2] *= 1e5
        K[..., ::2] *= 1e-8
    elif what.startswith("query"):
        Q[..., 3] = float(what.split()[1])
        K[..., 3] = 0.0
    else:       # hidden keys by a channel of their own
        Q[..., 3] = 1.0
        K[..., 3] = 0.0
        K[:, (600 if "later" in what else 0)::4, 3] = float(what.split()[-1])
        if what == "key 1e5":       # (nothing hidden: the channel counts for nothing)
            Q[..., 3] = 0.0
    check(Q, K, V, form)


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("head", [64, 128])
@pytest.mark.parametrize("what", ["spread 1e5", "spread 1e7", "one channel 1e-9", "one channel 1e-13",
                                  "one channel small later", "one key small", "last row small", "large later"])
def test_values_of_any_size_in_any_channel(form, head, what):
    """Small values among large ones, in a channel, in some keys of it, in the one
    row of a ragged last step; values three bits above the first step's."""
    print("case", form, head, what, flush=True)
    Q, K, V = draw(6, 2, 130, 705 if "row" in what else 700, head)
    mode = hip_sdpa.MASK_NONE
    if what.startswith("spread"):
        V *= torch.logspace(0, -round(math.log10(float(what.split()[1]))), head)
    elif what == "one channel small later":
        V[:, 200:, 7] *= 1e-8
        K[:, :200] = -Q[:, :1] * 30         # ... which the first query does not see
    elif what.startswith("one channel"):
        V[..., 7] *= float(what.split()[-1])
    elif what == "one key small":           # the first query's only key
        V[:, 0] *= 1e-10
        mode = hip_sdpa.MASK_CAUSAL
    elif what == "last row small":
        V[:, 704] *= 1e-12
        K[:, 704] = Q[:, 0] * 30            # ... the first query's only key
    elif what == "large later":
        V[:, 40:] *= 8
        K[:, 0] = Q[:, 0] * 30
        V[:, 0] *= 1e-4
    check(Q, K, V, form, mode)


def walks_again(Q, K, V, form):
    """Whether every workgroup takes its keys with fp32 instructions: with an
    infinite value in channel 0, which makes all of them, the other channels have the
    same bits.  (A workgroup that stays with the pieces does not: other sums.)"""
    V1 = V.clone()
    V1[:, 3, 0] = float("inf")
    A, A1 = (call(Q, K, v, hip_sdpa.MASK_NONE, FORMS[form])[0] for v in (V, V1))
    assert not torch.isfinite(A1[..., 0]).any()
    return [torch.equal(a[:, 1:], a1[:, 1:]) for a, a1 in zip(A.flatten(0, 1).split(32), A1.flatten(0, 1).split(32))]


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("head", [64, 128])
@pytest.mark.parametrize("what", ["plain", "last channel small", "small spread", "small values",
                                  "large values", "zero channel", "no value", "one more key",
                                  "zeros first", "zeros first, small", "zeros first, large"])
def test_what_the_pieces_carry_is_not_taken_again(form, head, what):
    print("case", form, head, what, flush=True)
    Q, K, V = draw(7, 2, 128, 769 if "key" in what else 768, head)
    if what == "last channel small":
        V[..., head - 1] *= 1e-3
    elif what == "small spread":
        V *= torch.logspace(-2, 0, head)
    elif what == "small values":
        V *= 1e-9
        K *= 1e-9
    elif what == "large values":
        V *= 1e9
        K *= 20
    elif what == "zero channel":
        V[..., 1:4] = 0.0
    elif what == "no value":
        V[:, 32:64] = 0.0
    elif what.startswith("zeros first"):    # padding in front, a whole step of any form
        V *= 0.01 if "small" in what else 6.0 if "large" in what else 0.4
        K[:, :64] = 0.0
        V[:, :64] = 0.0
    assert not any(walks_again(Q, K, V, form))


@pytest.mark.parametrize("form", FORMS)
def test_what_is_taken_again_can_be_told(form):
    Q, K, V = draw(8, 2, 128, 768, 64)
    V[..., 7] *= 1e-9
    assert all(walks_again(Q, K, V, form))


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("head", [64, 128])
@pytest.mark.parametrize("gap", [6, 8, 10, 12])
@pytest.mark.parametrize("value", [1e-3, 0.0, 1.0])
def test_a_first_key_that_takes_most_of_every_row(form, head, gap, value):
    """Scores of the first key `gap` above the others', and little in its values (as
    in models that park what a row does not need at the first token): the output is
    that of the others' probabilities, exp(-gap) and less."""
    print("case", form, head, gap, value, flush=True)
    Q, K, V = draw(9, 2, 130, 700, head)
    Q[..., 0] = 1.0
    K[..., 0] = 0.0
    K[:, 0] = 0.0
    K[:, 0, 0] = gap * math.sqrt(head)
    V[:, 0] *= value
    check(Q, K, V, form)
    check(Q, K, V, form, hip_sdpa.MASK_CAUSAL)


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("head", [64, 128])
@pytest.mark.parametrize("k_seq", [769, 770, 773, 774, 33, 37])
def test_a_few_small_values_in_the_last_rows_are_not_taken_again(form, head, k_seq):
    """A last group of one or two rows (of a later step, of the first one) some of
    whose channels are below 2^-2 at the power of two of the first step."""
    print("case", form, head, k_seq, flush=True)
    Q, K, V = draw(10, 2, 128, k_seq, head)
    V[:, -1, ::9] = 1e-4
    V[:, -2, ::9] *= 1e-4 if k_seq % 2 == 0 else 1.0
    assert not any(walks_again(Q, K, V, form))
    V[..., 7] *= 1e-9
    assert all(walks_again(Q, K, V, form))
    check(Q, K, V, form)
