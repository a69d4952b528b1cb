"""The backward of small launches: workgroups of 64 rows whose wavefronts halve the
steps of a walk between them, with dK and dV in workgroups of their own and, at head
64, in one: sizes at the edges of a half (32 rows), of a workgroup and of a step,
written and added to, against 64-bit arithmetic."""
import numpy as np
import pytest
import torch

from nntile_amd import hip_sdpa
from . import helpers as H

pytestmark = pytest.mark.gpu
# (those of the other backward tests)
TOL = {"bf16": 1e-2, "fp16": 2e-3}
MODES = {"none": hip_sdpa.MASK_NONE, "causal": hip_sdpa.MASK_CAUSAL, "additive": hip_sdpa.MASK_ADDITIVE,
         "bool": hip_sdpa.MASK_BOOL}


def _case(mode, head, group, n_kv, q_seq, k_seq, dtype, add):
    (Q, K, V), (qf, kf, vf) = H.make_qkv(17, n_kv * group, q_seq, k_seq, head, dtype, kv_batch=n_kv)
    G, gf = H.rounded(np.random.default_rng(5).standard_normal(qf.shape), dtype)
    q, g = (torch.from_numpy(x).cuda().double().reshape(n_kv, group, q_seq, head) for x in (qf, gf))
    k, v = (torch.from_numpy(x).cuda().double()[:, None].expand(n_kv, group, k_seq, head).contiguous()
            for x in (kf, vf))
    i, j = np.arange(q_seq)[:, None], np.arange(k_seq)[None, :]
    offset = max(k_seq - q_seq, 0)
    # (the values hide whole steps, halves and parts of others, and nothing of the rest)
    band = (np.abs(i - j) < 40) | (j < 10) | ((i >= 128) & (j < 100))
    seen = {"none": (i >= 0) & (j >= 0), "causal": j <= i + offset, "additive": band, "bool": band}[mode]
    shown = torch.from_numpy(seen).cuda()
    kt, vt = k.transpose(-1, -2).contiguous(), v.transpose(-1, -2).contiguous()
    s = (q @ kt / head ** 0.5).masked_fill(~shown, float("-inf"))
    lse, P = torch.logsumexp(s, dim=-1), torch.softmax(s, dim=-1)
    A16 = (P @ v).reshape(-1, q_seq, head).to(H.TORCH_DT[dtype])
    D = (g * A16.double().reshape(q.shape)).sum(-1, keepdim=True)
    dS = P * (g @ vt - D) / head ** 0.5
    want = {"dK": (dS.transpose(-1, -2).contiguous() @ q).sum(1), "dQ": (dS @ k).reshape(-1, q_seq, head),
            "dV": (P.transpose(-1, -2).contiguous() @ g).sum(1)}
    out = {name: torch.full(t.shape, 0.5 if add else float("nan"), dtype=t.dtype, device="cuda")
           for name, t in (("dK", K), ("dQ", Q), ("dV", V))}
    mask = H.additive_mask(seen, dtype).cuda() if mode == "additive" else \
        torch.from_numpy(seen.copy()).cuda() if mode == "bool" else None
    hip_sdpa.sdpa_bwd_tile(K.cuda(), Q.cuda(), V.cuda(), A16, G.cuda(), mask,
                           lse.reshape(-1, q_seq).float(), out["dK"], out["dQ"], out["dV"], MODES[mode],
                           n_batch=1, kv_group=group, causal_offset=offset,
                           flags=0 if add else hip_sdpa.OVERWRITE)
    torch.cuda.synchronize()
    for name in want:
        err = H.rel_fro(H.to_np(out[name]), want[name].cpu().numpy() + (0.5 if add else 0.0))
        assert err < TOL[dtype], (name, err)


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("mode", sorted(MODES))
@pytest.mark.parametrize("head,group,q_seq,k_seq,add", [
    (64, 1, 1, 1, False), (64, 1, 32, 33, True), (64, 1, 33, 32, False), (64, 1, 64, 64, True),
    (64, 1, 65, 97, False), (64, 1, 200, 160, False), (64, 2, 300, 300, True), (64, 8, 70, 130, False),
    (128, 1, 33, 33, True), (128, 1, 64, 64, False), (128, 1, 97, 97, True), (128, 1, 300, 300, False),
    (128, 2, 161, 161, True), (128, 1, 840, 70, False), (128, 1, 70, 850, True), (128, 7, 129, 129, False)])
def test_dk_and_dv_apart(dtype, mode, head, group, q_seq, k_seq, add):
    print("case bwd halved", dtype, mode, head, group, q_seq, k_seq, add, flush=True)
    _case(mode, head, group, 2, q_seq, k_seq, dtype, add)


# head 64, more than 256 workgroups of 64 rows in three sets (mask values: 512)
@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("mode,group,n_kv,q_seq,k_seq,add", [
    ("none", 1, 90, 33, 33, False), ("causal", 1, 90, 64, 64, True), ("causal", 1, 50, 97, 97, False),
    ("none", 1, 40, 161, 130, True), ("causal", 1, 80, 130, 200, False), ("causal", 4, 40, 100, 100, True),
    ("none", 8, 20, 130, 90, False), ("causal", 8, 24, 200, 129, False),
    ("additive", 1, 180, 64, 64, True), ("additive", 1, 60, 161, 190, False), ("bool", 1, 100, 97, 100, False)])
def test_dk_and_dv_in_one_workgroup(dtype, mode, group, n_kv, q_seq, k_seq, add):
    print("case bwd halved both", dtype, mode, group, n_kv, q_seq, k_seq, add, flush=True)
    _case(mode, 64, group, n_kv, q_seq, k_seq, dtype, add)
