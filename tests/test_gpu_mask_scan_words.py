"""The scan of a mask that a call does once, in the memory it is lent for it
(scratch_lse), against the scan that every workgroup does for itself without:
the same bits, whatever that memory held before - words of earlier calls,
constants, single words that carry the tag of the call to come - and at the
edges of the sizes that are scanned so."""
import time

import numpy as np
import pytest
import torch

from nntile_amd import hip_sdpa
from . import helpers as H
from . import test_gpu_mask_scan_once as large

pytestmark = pytest.mark.gpu


def _mask(kind, seq):
    if kind == "holes" and seq < 200:       # open but for the first query's last key
        m = np.ones((seq, seq), bool)
        m[0, seq - 1] = False
        return m
    return large._mask(kind, seq)


class _Call:
    def __init__(self, seed, kind, seq, head, batch, dtype="bf16"):
        (Q, K, V), _ = H.make_qkv(seed, batch, seq, seq, head, dtype)
        self.vis = _mask(kind, seq)
        self.args = [t.cuda() for t in (K, Q, H.additive_mask(self.vis, dtype), V)]
        self.shape = (batch, seq, head, dtype)
        self.rows = torch.from_numpy(self.vis.any(axis=1)).cuda()
        self.want = self()

    def __call__(self, scratch=None):
        K, Q, mask, V = self.args
        lse, A = H.fresh_outputs(*self.shape)
        hip_sdpa.flash_sdpa_fwd(K, Q, mask, lse, V, A, scratch_lse=scratch)
        return lse, A

    def same(self, got):
        # (rows that see nothing leave A as it was, NaN here)
        return torch.equal(got[0], self.want[0]) and torch.equal(
            got[1][:, self.rows].view(torch.int16), self.want[1][:, self.rows].view(torch.int16))


def _uppers(scratch):
    return (scratch.cpu().numpy().view(np.uint64).ravel() >> np.uint64(32)).astype(np.int64)


@pytest.mark.parametrize("kind", ["causal", "upper"])
def test_single_words_under_the_next_tag_are_not_taken(kind):
    """Whatever the words look like, their upper halves advance by the same step
    from call to call: one word at a time, in every block, is given the upper half
    that the next call's will have, above a lower half that says nothing was found."""
    seq, head, batch = 1024, 64, 2
    call = _Call(41, kind, seq, head, batch)
    scratch = torch.zeros(batch, seq, device="cuda")
    tags = []
    for _ in range(2):
        scratch.zero_()
        assert call.same(call(scratch))
        tags.append(_uppers(scratch))
    n = int(np.count_nonzero(scratch.cpu().numpy().view(np.uint64)))
    blocks = seq // 128
    per_block = n // blocks
    assert n > 0 and per_block * blocks == n
    step = (tags[1] - tags[0]) % (1 << 32)
    last, taken = tags[1], []
    for i in range(per_block):
        words = np.zeros(batch * seq // 2, np.uint64)
        at = np.arange(blocks) * per_block + i
        words[at] = ((last + step) % (1 << 32)).astype(np.uint64)[at] << np.uint64(32)
        scratch.copy_(torch.from_numpy(words.view(np.float32)).view(batch, seq))
        if not call.same(call(scratch)):
            taken.append(i)
        last = _uppers(scratch)
    assert not taken, "words taken for this call's: %s of %d" % (taken, per_block)


@pytest.mark.parametrize("fill", [0.0, 1.0, float("-inf"), float("nan")])
def test_constants_in_the_scratch(fill):
    call = _Call(42, "causal", 640, 64, 2)
    scratch = torch.full((2, 640), fill, device="cuda")
    assert call.same(call(scratch))


def test_words_of_earlier_calls_with_other_masks():
    """Calls with different masks through one scratch, each right behind the other."""
    calls = [_Call(43 + i, kind, 768, 64, 2)
             for i, kind in enumerate(["causal", "full", "window", "upper", "holes", "random"])]
    scratch = torch.full((2, 768), float("nan"), device="cuda")
    for order in ((0, 1, 2, 3, 4, 5), (3, 0, 5, 1, 4, 2), (1, 1, 3, 3, 0, 2)):
        got = [(i, calls[i](scratch)) for i in order]
        for i, out in got:
            assert calls[i].same(out), i


@pytest.mark.parametrize("kind", ["causal", "full", "window", "holes", "random"])
@pytest.mark.parametrize("seq,head,batch", [
    (8, 64, 1), (9, 64, 7), (48, 64, 1), (65, 128, 2), (128, 64, 4), (129, 64, 1), (355, 128, 1),
    (355, 64, 5), (500, 64, 3), (1024, 64, 1)])
def test_small_masks(kind, seq, head, batch):
    """Rows of 16 bytes and just over, ranges without a step, one batch entry."""
    print("case", kind, seq, head, batch, flush=True)
    for dtype in ("bf16", "fp16"):
        call = _Call(49, kind, seq, head, batch, dtype)
        guard = 64
        memory = torch.full((batch * seq + guard,), float("nan"), device="cuda")
        scratch = memory[:batch * seq].view(batch, seq)
        assert call.same(call(scratch))
        assert torch.isnan(memory[batch * seq:]).all()


@pytest.mark.parametrize("short", [0, 4])
def test_the_smallest_scratch_of_the_codelet_body(short):
    """320 bytes for every 128 queries hold the scan; with less the scratch is left
    alone, and nothing behind it is written."""
    seq, head, batch, dtype = 400, 64, 3, "bf16"
    call = _Call(50, "causal", seq, head, batch, dtype)
    floats = 4 * 320 // 4
    memory = torch.full((floats + 64,), float("nan"), device="cuda")
    scratch = memory[:floats - short // 4]
    K, Q, mask, V = call.args
    lse, A = H.fresh_outputs(batch, seq, head, dtype)
    hip_sdpa.flash_sdpa_fwd_codelet(K, Q, mask, lse, V, A, scratch_lse=scratch)
    torch.cuda.synchronize()
    assert call.same((lse, A))
    written = ~torch.isnan(memory)
    assert not bool(written[floats - short // 4:].any())
    assert bool(written.any()) == (short == 0)


def test_two_streams_that_share_a_scratch():
    """Calls that overwrite each other's words: workgroups that start late find those
    of the other call and scan for themselves, after a wait of some 20 us, not one
    that stalls the device."""
    seq, head, batch, calls = 128, 64, 2048, 10
    gen = torch.Generator(device="cuda").manual_seed(51)
    Q, K, V = (torch.randn(batch, seq, head, generator=gen, device="cuda").bfloat16()
               for _ in range(3))
    masks = [H.additive_mask(_mask(kind, seq), "bf16").cuda() for kind in ("causal", "window")]
    scratch = torch.zeros(batch, seq, device="cuda")

    def outputs():
        return torch.full((batch, seq), float("-inf"), device="cuda"), torch.zeros_like(Q)

    want = []
    for mask in masks:
        want.append(outputs())
        hip_sdpa.flash_sdpa_fwd(K, Q, mask, want[-1][0], V, want[-1][1])
    got = [[outputs() for _ in range(calls)] for _ in masks]
    streams = [torch.cuda.Stream() for _ in masks]
    torch.cuda.synchronize()
    t0 = time.monotonic()
    for i in range(calls):
        for mask, stream, outs in zip(masks, streams, got):
            hip_sdpa.flash_sdpa_fwd(K, Q, mask, outs[i][0], V, outs[i][1], scratch_lse=scratch,
                                    stream=stream)
    torch.cuda.synchronize()
    seconds = time.monotonic() - t0
    print("%d calls in %.1f ms" % (2 * calls, 1e3 * seconds), flush=True)
    for outs, (lse, A) in zip(got, want):
        for l, a in outs:
            assert torch.equal(l, lse) and torch.equal(a.view(torch.int16), A.view(torch.int16))
    # 2048 workgroups, 512 at a time, 21 us of waiting each at the most: 0.1 ms a call
    # beside its work; a call that waits out a second once is far above this
    assert seconds < 0.5
