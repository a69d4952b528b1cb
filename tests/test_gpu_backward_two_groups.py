"""The backward of a launch whose workgroups have a CU each walks its steps in two
groups of wavefronts that add their sums in LDS: walks of an even and an odd number of
steps, of none or one for the second group, at the lengths where the form begins,
against 64-bit arithmetic."""
import numpy as np
import pytest
import torch

from nntile_amd import hip_sdpa
from . import helpers as H

pytestmark = pytest.mark.gpu
# (those of the other backward tests)
TOL = {"bf16": 1e-2, "fp16": 2e-3}


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("mode", ["none", "causal", "additive"])
@pytest.mark.parametrize("head,group,q_seq,k_seq", [
    (64, 1, 320, 320), (64, 1, 321, 321), (64, 1, 384, 385), (64, 1, 449, 64), (64, 1, 64, 449), (64, 3, 130, 70),
    (128, 1, 768, 100), (128, 1, 769, 130), (128, 1, 100, 833), (128, 4, 200, 129), (128, 7, 65, 65)])
def test_gradients_of_walks_shared_by_two_groups(dtype, mode, head, group, q_seq, k_seq):
    print("case two groups", dtype, mode, head, group, q_seq, k_seq, flush=True)
    n_kv = 2
    (Q, K, V), (qf, kf, vf) = H.make_qkv(7, n_kv * group, q_seq, k_seq, head, dtype, kv_batch=n_kv)
    G, gf = H.rounded(np.random.default_rng(3).standard_normal(qf.shape), dtype)
    q, g = (torch.from_numpy(x).double().reshape(n_kv, group, q_seq, head) for x in (qf, gf))
    k, v = (torch.from_numpy(x).double()[:, None] for x in (kf, vf))
    i, j = np.arange(q_seq)[:, None], np.arange(k_seq)[None, :]
    offset = max(k_seq - q_seq, 0)
    # (the values hide whole steps, parts of others and nothing of the rest)
    seen = {"none": (i >= 0) & (j >= 0), "causal": j <= i + offset,
            "additive": (np.abs(i - j) < 150) | (j < 10)}[mode]
    s = (q @ k.transpose(-1, -2) / head ** 0.5).masked_fill(~torch.from_numpy(seen), float("-inf"))
    lse, P = torch.logsumexp(s, dim=-1), torch.softmax(s, dim=-1)
    A = P @ v
    # (what the kernel is handed is the rounded output)
    A16 = A.reshape(-1, q_seq, head).to(H.TORCH_DT[dtype])
    D = (g * A16.double().reshape(A.shape)).sum(-1, keepdim=True)
    dS = P * (g @ v.transpose(-1, -2) - D) / head ** 0.5
    want = {"dK": (dS.transpose(-1, -2) @ q).sum(1), "dQ": (dS @ k).reshape(-1, q_seq, head),
            "dV": (P.transpose(-1, -2) @ g).sum(1)}
    out = {name: torch.full(t.shape, float("nan"), dtype=t.dtype, device="cuda")
           for name, t in (("dK", K), ("dQ", Q), ("dV", V))}
    m = {"none": hip_sdpa.MASK_NONE, "causal": hip_sdpa.MASK_CAUSAL, "additive": hip_sdpa.MASK_ADDITIVE}[mode]
    mask = H.additive_mask(seen, dtype).cuda() if mode == "additive" else None
    hip_sdpa.sdpa_bwd_tile(K.cuda(), Q.cuda(), V.cuda(), A16.cuda(), G.cuda(), mask,
                           lse.reshape(-1, q_seq).float().cuda(), out["dK"], out["dQ"], out["dV"], m, n_batch=1,
                           kv_group=group, causal_offset=offset, flags=hip_sdpa.OVERWRITE)
    torch.cuda.synchronize()
    for name in want:
        err = H.rel_fro(H.to_np(out[name]), want[name].numpy())
        assert err < TOL[dtype], (name, err)


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("mode", ["none", "causal"])
@pytest.mark.parametrize("head,group,n_kv,q_seq,k_seq", [
    (64, 4, 48, 200, 129), (64, 13, 35, 64, 70), (128, 4, 48, 200, 129), (128, 13, 35, 65, 128), (128, 5, 44, 140, 200),
    (64, 1, 60, 830, 130), (128, 1, 60, 800, 257)])
def test_both_gradients_by_two_groups(dtype, mode, head, group, n_kv, q_seq, k_seq):
    """Launches of more workgroups, where one set of them computes dK and dV (those of
    one head a group without a mask by one group of wavefronts): the call over all
    key-value heads against the same in small ones."""
    print("case two groups fused", dtype, mode, head, group, n_kv, q_seq, k_seq, flush=True)
    assert n_kv * (2 * -(-k_seq // 128) + group * -(-q_seq // 128)) > 512
    m = hip_sdpa.MASK_NONE if mode == "none" else hip_sdpa.MASK_CAUSAL
    offset = max(k_seq - q_seq, 0)
    kind = H.TORCH_DT[dtype]
    torch.manual_seed(q_seq + k_seq)
    K, V = (torch.randn(n_kv, k_seq, head, device="cuda").to(kind) for _ in range(2))
    Q, G = (torch.randn(n_kv * group, q_seq, head, device="cuda").to(kind) for _ in range(2))
    lse, A = H.fresh_outputs(n_kv * group, q_seq, head, dtype)
    hip_sdpa.sdpa_fwd_tile(K, Q, None, lse, V, A, m, n_batch=1, kv_group=group, causal_offset=offset,
                           flags=hip_sdpa.OVERWRITE)

    def call(lo, hi):
        q = slice(lo * group, hi * group)
        args = [t.contiguous() for t in (K[lo:hi], Q[q], V[lo:hi], A[q], G[q])]
        out = [torch.full_like(t, float("nan")) for t in args[:3]]
        hip_sdpa.sdpa_bwd_tile(*args, None, lse[q].contiguous(), *out, m, n_batch=1, kv_group=group,
                               causal_offset=offset, flags=hip_sdpa.OVERWRITE)
        torch.cuda.synchronize()
        return out

    whole = call(0, n_kv)
    parts = [call(i, min(i + 4, n_kv)) for i in range(0, n_kv, 4)]
    # one rounding to the tile type each (2^-8 and 2^-11 of a value at most) of fp32 sums
    # taken in another order
    bound = {"bf16": 2.0 ** -8, "fp16": 2.0 ** -11}[dtype]
    for i, name in enumerate(("dK", "dQ", "dV")):
        want = torch.cat([p[i] for p in parts]).float()
        assert torch.isfinite(want).all() and torch.isfinite(whole[i]).all(), name
        err = float((whole[i].float() - want).norm() / want.norm())
        assert err < bound, (name, err)
