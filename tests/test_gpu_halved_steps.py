"""The 16-bit prefill kernel with workgroups of 64 queries whose wavefronts halve
every key step between them (NNTILE_HIP_SDPA_FORM_HALVED; what most launches of at
most one workgroup of 128 queries per CU take by themselves) against the checker
and beside the 128-query form of the same call."""
import numpy as np
import pytest
import torch

from nntile_amd import hip_sdpa, synth
from . import helpers as H

pytestmark = pytest.mark.gpu


def _tiles(x, step):
    return [x[:, s:s + step].contiguous().cuda() for s in range(0, x.shape[1], step)]


def _check(got, want, want_lse, dtype, name):
    A, lse = got
    assert H.rel_fro(A, want) < H.TOL[dtype], name
    assert H.rel_fro(lse, want_lse) < H.TOL[dtype], name
    H.check_rows(A, want, lse, want_lse, dtype, name)


# steps: one, two (the least of the pipelined loop), three to five (its loads run
# out in every parity), then those from which the keys are touched first
@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("head", [64, 128])
@pytest.mark.parametrize("q_seq,k_seq,q_tile,k_tile,n_batch,group,n_kv,causal", [
    (64, 20, 64, 20, 1, 1, 2, False),           # nothing for the second half of the step
    (33, 64, 33, 64, 1, 2, 2, False),           # one step; one row for the second pair
    (65, 97, 65, 97, 1, 1, 3, True),            # ragged in the second half, a row over
    (64, 128, 64, 128, 1, 1, 1, False),
    (70, 192, 70, 192, 2, 1, 1, False),
    (128, 257, 128, 257, 1, 1, 2, False),
    (130, 330, 130, 330, 1, 1, 2, True),
    (512, 512, 512, 512, 2, 1, 2, True),
    (1000, 1000, 384, 320, 1, 2, 2, True),      # ragged tiles, two XCDs' worth of sharing
    (1000, 1033, 512, 512, 8, 1, 1, False),     # touched: whole tiles and a ragged one
    (300, 1500, 300, 1500, 2, 4, 4, True),      # touched: heads of a group on one XCD
    (1100, 1100, 1100, 1100, 3, 1, 1, True),    # touched: one entry on several XCDs
    (64, 4160, 64, 4160, 1, 1, 2, True),        # 65 steps
])
def test_halved_steps(oracle, dtype, head, q_seq, k_seq, q_tile, k_tile, n_batch, group, n_kv, causal):
    print("case", dtype, head, q_seq, k_seq, q_tile, k_tile, n_batch, group, n_kv, causal, flush=True)
    batch = n_batch * group * n_kv
    offset = k_seq - q_seq
    (Q, K, V), (qf, kf, vf) = H.make_qkv(81, batch, q_seq, k_seq, head, dtype, kv_batch=n_batch * n_kv)
    mask = synth.causal_mask(q_seq, k_seq, offset) if causal else None
    want, want_lse = oracle.sdpa_vanilla(kf, qf, vf, mask, k_tile=k_tile, n_batch=n_batch,
                                         kv_repeat=group)
    mode = hip_sdpa.MASK_CAUSAL if causal else hip_sdpa.MASK_NONE
    Kt, Vt, Qt = _tiles(K, k_tile), _tiles(V, k_tile), _tiles(Q, q_tile)
    outs = {}
    for name, flags in (("four", hip_sdpa.FORM_SHARED), ("halved", hip_sdpa.FORM_HALVED),
                        ("overwrite", hip_sdpa.FORM_HALVED | hip_sdpa.OVERWRITE),
                        ("again", hip_sdpa.FORM_HALVED)):
        o = [H.fresh_outputs(batch, t.shape[1], head, dtype) for t in Qt]
        hip_sdpa.sdpa_fwd_grid(Kt, Qt, [x[0] for x in o], Vt, [x[1] for x in o], q_seq, k_seq, q_tile,
                               k_tile, mode, n_batch=n_batch, kv_group=group, causal_offset=offset,
                               flags=flags)
        torch.cuda.synchronize()
        outs[name] = (np.concatenate([H.to_np(x[1]) for x in o], axis=1),
                      np.concatenate([H.to_np(x[0]) for x in o], axis=1))
        _check(outs[name], want, want_lse, dtype, name)
    assert H.rel_fro(outs["halved"][0], outs["four"][0]) < H.TOL[dtype]
    for name in ("overwrite", "again"):         # no dependence on timing
        assert np.array_equal(outs["halved"][0], outs[name][0])
        assert np.array_equal(outs["halved"][1], outs[name][1])


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("form", ["additive", "bool"])
@pytest.mark.parametrize("head", [64, 128])
@pytest.mark.parametrize("q_seq,k_seq,pattern", [
    (64, 5, "holes"), (70, 30, "band"), (256, 1024, "causal"), (200, 712, "band"), (128, 520, "holes"),
    (130, 333, "band"), (130, 1001, "causal"), (256, 1024, "all_open"), (128, 576, "all_hidden"),
    (190, 1600, "holes"), (130, 4232, "band")])
def test_halved_steps_with_masks_given_as_values(oracle, dtype, form, head, q_seq, k_seq, pattern):
    print("case", dtype, form, head, q_seq, k_seq, pattern, flush=True)
    batch = 3
    i = np.arange(q_seq)[:, None]
    j = np.arange(k_seq)[None, :]
    mask = {"causal": j <= i + (k_seq - q_seq), "band": j <= (k_seq // 3 + 2 * i),
            "holes": ((j < 100) | (j >= 300)) & (i % 50 != 49) & (j >= 0),
            "all_hidden": (i < 0) & (j < 0), "all_open": (i >= 0) & (j >= 0)}[pattern]
    mask = np.ascontiguousarray(np.broadcast_to(mask, (q_seq, k_seq)))
    (Q, K, V), (qf, kf, vf) = H.make_qkv(83, batch, q_seq, k_seq, head, dtype)
    want, want_lse = oracle.sdpa_vanilla(kf, qf, vf, mask)
    m = (H.additive_mask(mask, dtype) if form == "additive" else torch.from_numpy(mask.copy())).cuda()
    mode = hip_sdpa.MASK_ADDITIVE if form == "additive" else hip_sdpa.MASK_BOOL
    vis = mask.any(axis=1)
    for name, flags in (("four", hip_sdpa.FORM_SHARED), ("halved", hip_sdpa.FORM_HALVED)):
        lse, A = H.fresh_outputs(batch, q_seq, head, dtype)
        hip_sdpa.sdpa_fwd_tile(K.cuda(), Q.cuda(), m, lse, V.cuda(), A, mode,
                               flags=flags | hip_sdpa.OVERWRITE)
        torch.cuda.synchronize()
        a, l = H.to_np(A), H.to_np(lse)
        assert np.all(a[:, ~vis] == 0) and np.all(np.isneginf(l[:, ~vis])), name
        if vis.any():
            assert H.rel_fro(a[:, vis], want[:, vis]) < H.TOL[dtype], name
            assert H.rel_fro(l[:, vis], want_lse[:, vis]) < H.TOL[dtype], name


@pytest.mark.parametrize("mode", [hip_sdpa.MASK_CAUSAL, hip_sdpa.MASK_ADDITIVE])
def test_halved_steps_merge_into_a_running_pair(oracle, mode):
    """Key tiles one call at a time: the halves are put together first, then merged with
    what is there; rows that see nothing of a tile keep their pair.  The additive calls
    go through the entry point whose scratch holds the scan of the mask, done for
    blocks of twice as many rows."""
    dtype, head, seq, k_tile, batch = "bf16", 128, 640, 320, 2
    (Q, K, V), (qf, kf, vf) = H.make_qkv(82, batch, seq, seq, head, dtype)
    mask = synth.causal_mask(seq, seq)
    want, want_lse = oracle.sdpa_vanilla(kf, qf, vf, mask, k_tile=k_tile)
    lse, A = H.fresh_outputs(batch, seq, head, dtype)
    for i, (kt, vt) in enumerate(zip(_tiles(K, k_tile), _tiles(V, k_tile))):
        if mode == hip_sdpa.MASK_CAUSAL:
            hip_sdpa.sdpa_fwd_tile(kt, Q.cuda(), None, lse, vt, A, mode, k_pos0=i * k_tile,
                                   flags=hip_sdpa.FORM_HALVED)
            continue
        for q0 in range(0, seq, k_tile):
            m = H.additive_mask(np.ascontiguousarray(mask[q0:q0 + k_tile, i * k_tile:(i + 1) * k_tile]),
                                dtype).cuda()
            l, a = lse[:, q0:q0 + k_tile].contiguous(), A[:, q0:q0 + k_tile].contiguous()
            hip_sdpa.flash_sdpa_fwd(kt, Q[:, q0:q0 + k_tile].contiguous().cuda(), m, l, vt, a,
                                    torch.empty_like(l), torch.empty_like(a))
            lse[:, q0:q0 + k_tile], A[:, q0:q0 + k_tile] = l, a
    torch.cuda.synchronize()
    assert H.rel_fro(H.to_np(A), want) < H.TOL[dtype]
    assert H.rel_fro(H.to_np(lse), want_lse) < H.TOL[dtype]


@pytest.mark.parametrize("overwrite", [True, False])
@pytest.mark.parametrize("where", [5, 40, 100])     # either half of the first step, the second step
def test_nan_in_one_half_shows(where, overwrite):
    (Q, K, V), _ = H.make_qkv(84, 2, 130, 200, 128, "bf16")
    Q, K, V = Q.cuda(), K.cuda(), V.cuda()
    bad = torch.arange(130, device="cuda") >= where
    K[1, where, 7] = float("nan")
    lse = torch.full((2, 130), 1.5, device="cuda")
    A = torch.full((2, 130, 128), 0.25, dtype=Q.dtype, device="cuda")
    hip_sdpa.sdpa_fwd_tile(K, Q, None, lse, V, A, hip_sdpa.MASK_CAUSAL,
                           flags=hip_sdpa.FORM_HALVED | (hip_sdpa.OVERWRITE if overwrite else 0))
    torch.cuda.synchronize()
    assert torch.isfinite(lse[0]).all() and torch.isfinite(A[0]).all()
    assert torch.isfinite(lse[1, ~bad]).all() and torch.isfinite(A[1, ~bad]).all()
    if overwrite:
        assert torch.isnan(lse[1, bad]).all() and torch.isnan(A[1, bad]).all()
    else:
        assert (lse[1, bad] == 1.5).all() and (A[1, bad] == 0.25).all()
