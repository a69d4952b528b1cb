"""A NaN among the scores of a row shows in that row whatever route the call
takes, and in no other row.  Where (lse, A) are overwritten both become NaN;
the split-key decode kernels carry it into a running pair too, the tile kernels
leave the pair of such a row as it was (the rule of accumulate_attn_output:
src/kernel/accumulate_attn_output/cuda.cu:43-50)."""
import pytest
import torch

from nntile_amd import hip_sdpa
from . import helpers as H

pytestmark = pytest.mark.gpu

# name, route, q_seq, k_seq, heads (a batch entry each), head, flags
ROUTES = [
    ("tile, keys shared", "tile", 100, 300, 2, 128, hip_sdpa.FORM_SHARED),
    ("tile, keys split", "tile", 100, 300, 2, 64, hip_sdpa.FORM_SPLIT),
    ("tile, wide", "tile", 300, 500, 2, 128, hip_sdpa.FORM_WIDE),
    ("chunk, one range", "cache", 100, 3000, 2, 128, None),
    ("chunk, key ranges", "ranges", 100, 3000, 2, 128, None),
    ("chunk, key ranges", "ranges", 70, 2000, 1, 64, None),
    ("decode, one split", "decode", 16, 190, 3, 128, 0),
    ("decode, one split", "decode", 5, 60, 3, 64, 0),
    ("decode, few splits", "decode", 16, 400, 3, 128, 0),
    ("decode, many splits", "decode", 16, 4000, 3, 64, 0),
    ("decode, few splits, second launch", "decode", 16, 400, 3, 64, hip_sdpa.DECODE_SEPARATE_MERGE),
    ("decode, many splits, second launch", "decode", 16, 4000, 3, 128, hip_sdpa.DECODE_SEPARATE_MERGE)]


def call(route, K, Q, V, lse, A, k_seq, flags):
    if route == "decode":
        n = K.shape[0]
        ws = torch.full((hip_sdpa.decode_workspace_bytes(K, Q, n, 1),), 0xff, dtype=torch.uint8, device="cuda")
        hip_sdpa.sdpa_fwd_decode(K, Q, None, lse, V, A, hip_sdpa.MASK_CAUSAL, n, 1, ws,
                                 causal_offset=k_seq - Q.shape[1], flags=flags)
    elif route == "tile":
        hip_sdpa.sdpa_fwd_tile(K, Q, None, lse, V, A, hip_sdpa.MASK_CAUSAL,
                               causal_offset=k_seq - Q.shape[1], flags=flags)
    else:
        need = hip_sdpa.tile_cache_workspace_bytes(k_seq, Q, hip_sdpa.MASK_CAUSAL)
        assert need > 0
        ws = torch.full((need,), 0xff, dtype=torch.uint8, device="cuda") if route == "ranges" else None
        hip_sdpa.sdpa_fwd_tile_cache(K, V, k_seq, Q, None, lse, A, hip_sdpa.MASK_CAUSAL,
                                     causal_offset=k_seq - Q.shape[1], flags=flags, workspace=ws)
    torch.cuda.synchronize()


@pytest.mark.parametrize("dtype,case", [
    (d, c) for d in ("bf16", "fp32") for c in ROUTES
    if d == "bf16" or c[6] != hip_sdpa.FORM_WIDE])      # (a form of the 16-bit kernel)
@pytest.mark.parametrize("where", ["query", "key", "infinite key"])
@pytest.mark.parametrize("overwrite", [True, False])
def test_nan_shows(dtype, case, where, overwrite):
    name, route, q_seq, k_seq, heads, head, extra = case
    print("case", dtype, name, where, overwrite, flush=True)
    (Q, K, V), _ = H.make_qkv(71, heads, q_seq, k_seq, head, dtype)
    Q, K, V = Q.cuda(), K.cuda(), V.cuda()
    bad = torch.zeros(heads, q_seq, dtype=torch.bool, device="cuda")
    Kn, Qn = K.clone(), Q.clone()
    if where == "query":
        bad[heads - 1, q_seq // 2] = True
        Qn[heads - 1, q_seq // 2] = float("nan")
    else:
        # the rows from q_seq // 2 on see this key, the others do not.  (An
        # infinite score is subtracted from itself.)
        bad[0, q_seq // 2:] = True
        if where == "key":
            Kn[0, k_seq - q_seq + q_seq // 2, 3] = float("nan")
        else:
            Kn[0, k_seq - q_seq + q_seq // 2, 3] = float("inf")
            Qn[0, :, 3] = Q[0, :, 3] = 1.0
    flags = (extra or 0) | (hip_sdpa.OVERWRITE if overwrite else 0)
    out = []
    for k, q in ((K, Q), (Kn, Qn)):
        lse = torch.full((heads, q_seq), 1.5, device="cuda")
        A = torch.full((heads, q_seq, head), 0.25, dtype=Q.dtype, device="cuda")
        call(route, k, q, V, lse, A, k_seq, flags)
        out.append((lse, A.float()))
    (lse0, A0), (lse, A) = out
    assert torch.isfinite(lse0).all() and torch.isfinite(A0).all()
    if not overwrite and route != "decode":
        assert (lse[bad] == 1.5).all() and (A[bad] == 0.25).all()
    else:
        assert torch.isnan(lse[bad]).all() and torch.isnan(A[bad]).all()
    # (which maximum a row is taken against may follow its neighbours: two
    # roundings of the probabilities and of the output, 2^-9 each)
    assert H.rel_fro(H.to_np(A[~bad]), H.to_np(A0[~bad])) < {"bf16": 2.0 ** -8,
                                                            "fp32": 5e-6}[dtype]
    assert H.rel_fro(H.to_np(lse[~bad]), H.to_np(lse0[~bad])) < 1e-6
