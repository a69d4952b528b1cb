"""The reference-signature call with its scratch tile: an additive mask is
scanned once per call by the first workgroups of the launch (into the scratch
logsumexp tile) instead of once per batch entry by the attention kernel's
workgroups.  Both ways produce the same bits about the mask, so the results
must be identical bit for bit, whatever the mask holds; and they must agree
with the CPU checker."""
import numpy as np
import pytest
import torch

from nntile_amd import hip_sdpa, synth
from . import helpers as H

pytestmark = pytest.mark.gpu


def _mask(kind, seq):
    i = np.arange(seq)[:, None]
    j = np.arange(seq)[None, :]
    if kind == "causal":
        return j <= i
    if kind == "full":
        return np.ones((seq, seq), bool)
    if kind == "window":
        return np.abs(i - j) <= 100
    if kind == "upper":                 # every query of the first blocks sees nothing
        return (j <= i) & (i >= 200)
    if kind == "holes":                 # open but for single hidden elements
        m = np.ones((seq, seq), bool)
        m[5, 70] = m[seq - 1, 0] = m[130, seq - 1] = False
        m[:, 0] = True
        return m
    rng = np.random.Generator(np.random.PCG64(7))
    m = rng.random((seq, seq)) < 0.5
    m[:, 0] = True
    return m


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("kind", ["causal", "full", "window", "upper", "holes", "random"])
@pytest.mark.parametrize("seq,head,batch", [(1024, 64, 2), (768, 128, 3), (4160, 64, 2)])
def test_scan_once_equals_scan_per_workgroup(oracle, dtype, kind, seq, head, batch):
    # (4160 = 65 key steps: steps from 63 on share one bit of the scan)
    print("case", dtype, kind, seq, head, batch, flush=True)
    (Q, K, V), f32 = H.make_qkv(31, batch, seq, seq, head, dtype)
    vis = _mask(kind, seq)
    m = H.additive_mask(vis, dtype).cuda()
    Kd, Qd, Vd = K.cuda(), Q.cuda(), V.cuda()
    outs = []
    for with_scratch in (False, True):
        lse, A = H.fresh_outputs(batch, seq, head, dtype)
        scratch = torch.full((batch, seq), float("nan"), device="cuda") if with_scratch else None
        hip_sdpa.flash_sdpa_fwd(Kd, Qd, m, lse, Vd, A, scratch_lse=scratch)
        torch.cuda.synchronize()
        outs.append((lse, A))
    (lse0, A0), (lse1, A1) = outs
    assert torch.equal(lse0, lse1)
    rows = torch.from_numpy(vis.any(axis=1)).cuda()
    assert torch.equal(A0[:, rows].view(torch.int16), A1[:, rows].view(torch.int16))
    if seq <= 1024:
        qf, kf, vf = f32
        want, want_lse = oracle.sdpa_vanilla(kf, qf, vf, vis)
        r = vis.any(axis=1)
        assert H.rel_fro(H.to_np(A1)[:, r], want[:, r]) < H.TOL[dtype]
        assert H.rel_fro(H.to_np(lse1)[:, r], want_lse[:, r]) < H.TOL[dtype]
        assert np.all(np.isneginf(H.to_np(lse1)[:, ~r]))


def test_codelet_body_uses_its_scratch_buffer(oracle):
    # buffer 6 of the codelet is the scratch logsumexp tile; with and without
    # it the task's result is the same
    dtype, seq, head, batch = "bf16", 1024, 64, 4
    (Q, K, V), _ = H.make_qkv(33, batch, seq, seq, head, dtype)
    m = H.additive_mask(synth.causal_mask(seq, seq), dtype).cuda()
    Kd, Qd, Vd = K.cuda(), Q.cuda(), V.cuda()
    outs = []
    for with_scratch in (False, True):
        lse, A = H.fresh_outputs(batch, seq, head, dtype)
        s_lse = torch.empty((batch, seq), device="cuda") if with_scratch else None
        s_A = torch.empty_like(A) if with_scratch else None
        hip_sdpa.flash_sdpa_fwd_codelet(Kd, Qd, m, lse, Vd, A, s_lse, s_A)
        torch.cuda.synchronize()
        outs.append((lse, A))
    assert torch.equal(outs[0][0], outs[1][0])
    assert torch.equal(outs[0][1].view(torch.int16), outs[1][1].view(torch.int16))


def test_a_scratch_smaller_than_a_logsumexp_tile_is_refused_or_left_alone():
    """The tile call cannot know the size of its scratch (it takes it to be a
    logsumexp tile), so the Python wrapper refuses a smaller tensor before the
    call; the codelet body reads the size from the buffer's interface and
    leaves a smaller one untouched - same result as without it."""
    seq, head, batch, dtype = 1024, 64, 2, "bf16"
    (Q, K, V), _ = H.make_qkv(37, batch, seq, seq, head, dtype)
    m = H.additive_mask(_mask("window", seq), dtype).cuda()
    Kd, Qd, Vd = K.cuda(), Q.cuda(), V.cuda()
    lse, A = H.fresh_outputs(batch, seq, head, dtype)
    small = torch.full((batch * seq - 1,), float("nan"), device="cuda")
    with pytest.raises(ValueError):
        hip_sdpa.flash_sdpa_fwd(Kd, Qd, m, lse, Vd, A, scratch_lse=small)
    torch.cuda.synchronize()
    assert torch.isneginf(lse).all()          # nothing ran
    lse0, A0 = H.fresh_outputs(batch, seq, head, dtype)
    hip_sdpa.flash_sdpa_fwd_codelet(Kd, Qd, m, lse0, Vd, A0)
    lse1, A1 = H.fresh_outputs(batch, seq, head, dtype)
    tiny = torch.full((4,), float("nan"), device="cuda")      # less than the scan's table
    hip_sdpa.flash_sdpa_fwd_codelet(Kd, Qd, m, lse1, Vd, A1, scratch_lse=tiny)
    torch.cuda.synchronize()
    assert torch.isnan(tiny).all()            # left alone
    assert torch.equal(lse0, lse1) and torch.equal(A0.view(torch.int16), A1.view(torch.int16))


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("seq,batch", [(640, 100), (1000, 63), (640, 102), (640, 103)])
def test_every_block_where_the_scan_fills_the_second_round(dtype, seq, batch):
    """The workgroups that scan the mask do not count where the second 256
    attention workgroups are dealt in reverse: 500 + 40, 504 + 64 (not dealt so),
    510 + 40 and 515 + 40 workgroups, each against the same mask as a rule."""
    print("case", dtype, seq, batch, flush=True)
    head = 64
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seq + batch)
    Q, K, V = (torch.randn(batch, seq, head, generator=gen, device="cuda").to(H.TORCH_DT[dtype])
               for _ in range(3))
    m = H.additive_mask(_mask("causal", seq), dtype).cuda()
    lse = torch.full((batch, seq), float("-inf"), device="cuda")
    A = torch.zeros_like(Q)
    hip_sdpa.flash_sdpa_fwd(K, Q, m, lse, V, A, torch.empty_like(lse), torch.empty_like(Q))
    lse2 = torch.full((batch, seq), float("-inf"), device="cuda")
    A2 = torch.zeros_like(Q)
    hip_sdpa.sdpa_fwd_tile(K, Q, None, lse2, V, A2, hip_sdpa.MASK_CAUSAL)
    torch.cuda.synchronize()
    # the same steps in the same order: probabilities and outputs rounded alike
    # but for the scores' path through the mask addition (fp32, 2^-24 each)
    assert H.rel_fro(H.to_np(lse), H.to_np(lse2)) < 1e-6
    assert H.rel_fro(H.to_np(A), H.to_np(A2)) < H.TOL[dtype]
    worst = (A.float() - A2.float()).norm(dim=-1) / A2.float().norm(dim=-1)
    assert float(worst.max()) < H.ROW_TOL[dtype]
