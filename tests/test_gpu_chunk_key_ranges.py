"""A chunk against a filled cache with its key axis shared out over workgroups
(sdpa_fwd_tile_cache with a workspace) against the checker and against the
same call without: ragged rows and keys, ranges that a causal rule hides from
all or some rows, a running pair that is merged with, a workspace that holds
NaN before the call."""
import pytest
import torch

from nntile_amd import hip_sdpa, synth
from nntile_amd.kv_cache import KVCache
from . import helpers as H


@pytest.mark.parametrize("q_seq,k_seq,heads,head,mode,shared", [
    (100, 4000, 8, 128, hip_sdpa.MASK_CAUSAL, True), (100, 4000, 8, 32, hip_sdpa.MASK_CAUSAL, False),
    (100, 4000, 8, 128, hip_sdpa.MASK_BOOL, False), (100, 500, 8, 128, hip_sdpa.MASK_NONE, False),
    (100, 4000, 200, 128, hip_sdpa.MASK_NONE, False), (4000, 4000, 8, 64, hip_sdpa.MASK_NONE, False)])
def test_which_calls_are_shared_out(q_seq, k_seq, heads, head, mode, shared):
    """...and that the memory asked for holds a whole number of ranges, at least two."""
    a = hip_sdpa.TileArgs()
    a.batch, a.q_seq, a.head, a.k_seq, a.n_batch, a.kv_group, a.mask_mode = heads, q_seq, head, k_seq, 1, 1, mode
    need = hip_sdpa.lib().nntile_hip_sdpa_fwd_tile_cache_workspace_bytes(a)
    one = heads * q_seq * (head + 2) * 4
    assert (need >= 2 * one and need % one == 0) if shared else need == 0


CASES = [
    # q_seq, k_seq, capacity, n_batch, group, n_kv, head, offset behind k_seq - q_seq
    (17, 1537, 1537, 1, 4, 1, 128, 0),       # one key in the last step
    (129, 1500, 2048, 1, 1, 3, 128, 0),      # a second block of one row
    (100, 3000, 3001, 2, 2, 2, 64, 0),
    (33, 9000, 9001, 1, 1, 1, 64, 0),        # the most ranges
    (20, 2048, 2048, 2, 8, 8, 128, 0),       # two ranges fill the places exactly
    (70, 2000, 2000, 1, 2, 2, 128, -1200),   # ranges nobody sees
    (70, 2000, 2000, 1, 2, 2, 64, -1960),    # rows that see nothing
    (90, 1100, 1100, 1, 1, 2, 128, None)]    # no mask


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("overwrite", [True, False])
def test_shared_out_keys(oracle, dtype, case, overwrite):
    q_seq, k_seq, cap, n_batch, group, n_kv, head, shift = case
    print("case", dtype, case, overwrite, flush=True)
    batch, kvb = n_batch * group * n_kv, n_batch * n_kv
    (Q, K, V), (qf, kf, vf) = H.make_qkv(57, batch, q_seq, k_seq, head, dtype, kv_batch=kvb)
    mode = hip_sdpa.MASK_NONE if shift is None else hip_sdpa.MASK_CAUSAL
    offset = 0 if shift is None else k_seq - q_seq + shift
    Qd = Q.cuda()
    Kc = torch.full((kvb, cap, head), float("nan"), dtype=H.TORCH_DT[dtype], device="cuda")
    Vc = torch.full_like(Kc, float("nan"))
    Kc[:, :k_seq] = K.cuda()
    Vc[:, :k_seq] = V.cuda()
    need = hip_sdpa.tile_cache_workspace_bytes(k_seq, Qd, mode)
    assert need > 0
    flags = hip_sdpa.OVERWRITE if overwrite else 0
    out = []
    for nbytes in (need, need - 4, None):       # (too little: as without)
        ws = None if nbytes is None else torch.full((need // 4,), float("nan"), device="cuda").view(
            torch.uint8)[:nbytes]
        lse = torch.full((batch, q_seq), 1.5, device="cuda")
        A = torch.full((batch, q_seq, head), 0.25, dtype=Qd.dtype, device="cuda")
        hip_sdpa.sdpa_fwd_tile_cache(Kc, Vc, k_seq, Qd, None, lse, A, mode, n_batch, group,
                                     causal_offset=offset, flags=flags, workspace=ws)
        torch.cuda.synchronize()
        out.append((A.float(), lse))
    (A, lse), (A1, lse1), (A2, lse2) = out
    assert torch.equal(A1, A2) and torch.equal(lse1, lse2)
    # 16-bit: each call rounds the probabilities (against its own maxima) and
    # the output, by at most u = 2^-9 (2^-12) of a value: four independent
    # errors, 2u in the 2-norm; fp32: a few hundred roundings of 2^-24
    apart = H.rel_fro(H.to_np(A), H.to_np(A2))
    print("apart %.2e" % apart, flush=True)
    assert apart < {"bf16": 2.0 ** -8, "fp16": 2.0 ** -11, "fp32": 5e-6}[dtype]
    hidden = torch.isinf(lse2)
    assert torch.equal(hidden, torch.isinf(lse)) and torch.equal(A[hidden], A2[hidden])
    lse_apart = H.rel_fro(H.to_np(lse[~hidden]), H.to_np(lse2[~hidden]))
    assert lse_apart < 1e-6
    if overwrite and shift in (0, None):
        mask = None if shift is None else synth.causal_mask(q_seq, k_seq, offset)
        want, want_lse = oracle.sdpa_vanilla(kf, qf, vf, mask, n_batch=n_batch, kv_repeat=group)
        assert H.rel_fro(H.to_np(A), want) < H.TOL[dtype]
        assert H.rel_fro(H.to_np(lse), want_lse) < H.LSE_TOL[dtype]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bf16", "fp32"])
def test_a_cache_takes_chunks_of_any_length_on_a_side_stream(oracle, dtype):
    """Chunks that are shared out, that are not and single tokens in turn, each
    against the rows of one pass over the whole sequence."""
    head, group, n_kv, total = 64, 2, 2, 1500
    (Q, K, V), (qf, kf, vf) = H.make_qkv(58, group * n_kv, total, total, head, dtype, kv_batch=n_kv)
    want, _ = oracle.sdpa_vanilla(kf, qf, vf, synth.causal_mask(total, total, 0), n_batch=1,
                                  kv_repeat=group)
    cache = KVCache(total)
    side = torch.cuda.Stream()
    pos = 0
    Qd, Kd, Vd = Q.cuda(), K.cuda(), V.cuda()
    torch.cuda.synchronize()
    for i, rows in enumerate((1100, 90, 1, 40, 200, 1, 68)):
        cut = [t[:, pos:pos + rows].contiguous() for t in (Qd, Kd, Vd)]
        lse, A = H.fresh_outputs(group * n_kv, rows, head, dtype)
        stream = side if i % 2 else None
        torch.cuda.synchronize()
        cache.append_attend(cut[1], cut[2], cut[0], lse, A, 1, group, stream=stream)
        torch.cuda.synchronize()
        assert H.rel_fro(H.to_np(A), want[:, pos:pos + rows]) < H.TOL[dtype], (i, rows)
        pos += rows
    assert pos == total
