"""The backward over a grid of tiles where one set of workgroups computes dK and dV
and two groups of wavefronts share a walk (more than 512 workgroups in three sets, at
most 256 that own keys - 192 and grouped heads without a mask - and a walk of 13 steps
and more): against 64-bit arithmetic, written and added to, and bit for bit the call
over one allocation."""
import pytest
import torch

from nntile_amd import hip_sdpa
from . import helpers as H

pytestmark = pytest.mark.gpu
# (those of the other backward tests)
TOL = {"bf16": 1e-2, "fp16": 2e-3}

# q_seq, k_seq, q_tile, k_tile, n_batch, group, n_kv, n_slabs
GROUPED = [
    (130, 300, 128, 256, 1, 8, 30, 1),      # ragged last tiles of 2 and 44 rows
    (130, 300, 128, 256, 1, 8, 15, 2),      # the same entries in two slabs
    (200, 129, 128, 128, 2, 4, 24, 1),
    (65, 70, 65, 70, 1, 13, 12, 3),         # one tile an axis
]
SINGLE = [
    (830, 130, 256, 128, 3, 1, 20, 1),      # walks of up to 13 steps over the queries
    (130, 900, 128, 384, 1, 1, 15, 2),      # of up to 15 over the keys
]


def _kv_of(batch, n_batch, group, device="cuda"):
    b = torch.arange(batch, device=device)
    return b % n_batch + n_batch * (b // (n_batch * group))


def _gradients(Q, K, V, A, G, mask, kv, lse):
    """dK, dQ, dV of one slab in 64 bits, from the rounded inputs and output."""
    q, k, v, a, g = (t.double() for t in (Q, K[kv], V[kv], A, G))
    scale = Q.shape[-1] ** -0.5
    s = torch.bmm(q, k.transpose(1, 2).contiguous()) * scale
    P = torch.exp(s.masked_fill(~mask, float("-inf")) - lse.double()[:, :, None])
    dP = torch.bmm(g, v.transpose(1, 2).contiguous())
    dS = P * (dP - (g * a).sum(-1, keepdim=True)) * scale
    dK, dV = (torch.zeros(K.shape, dtype=torch.float64, device=K.device) for _ in range(2))
    dK.index_add_(0, kv, torch.bmm(dS.transpose(1, 2).contiguous(), q))
    dV.index_add_(0, kv, torch.bmm(P.transpose(1, 2).contiguous(), g))
    return dK, torch.bmm(dS, k), dV


def _inputs(shape, head, dtype, mode, seed):
    """Per slab: K, Q, V, A, dA, lse, and the mask of the rule."""
    q_seq, k_seq, _, _, n_batch, group, n_kv, n_slabs = shape
    offset = max(k_seq - q_seq, 0)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    batch = n_batch * group * n_kv
    m = hip_sdpa.MASK_CAUSAL if mode == "causal" else hip_sdpa.MASK_NONE
    slabs = []
    for _ in range(n_slabs):
        Q, G = (torch.randn(batch, q_seq, head, generator=gen, device="cuda").to(H.TORCH_DT[dtype])
                for _ in range(2))
        K, V = (torch.randn(n_batch * n_kv, k_seq, head, generator=gen,
                            device="cuda").to(H.TORCH_DT[dtype]) for _ in range(2))
        lse, A = H.fresh_outputs(batch, q_seq, head, dtype)
        hip_sdpa.sdpa_fwd_tile(K, Q, None, lse, V, A, m, n_batch=n_batch, kv_group=group,
                               causal_offset=offset, flags=hip_sdpa.OVERWRITE)
        slabs.append((K, Q, V, A, G, lse))
    i = torch.arange(q_seq, device="cuda")[:, None]
    j = torch.arange(k_seq, device="cuda")[None, :]
    seen = (j <= i + offset) if mode == "causal" else torch.ones_like(j <= i)
    return slabs, seen, offset, m


def _split(t, tile):
    return [t[:, s:s + tile].contiguous() for s in range(0, t.shape[1], tile)]


def _join(tiles):
    return torch.cat(tiles, dim=1)


def _grid_call(slabs, start, shape, offset, m, flags):
    """dK, dQ, dV tiles (slab by slab) of one call over all slabs, from `start`."""
    q_seq, k_seq, q_tile, k_tile, n_batch, group, n_kv, n_slabs = shape
    ins = [[] for _ in range(6)]
    for s in slabs:
        for dst, t, tile in zip(ins, s, (k_tile, q_tile, k_tile, q_tile, q_tile, q_tile)):
            dst += _split(t, tile)
    out = [[x for s in start for x in _split(s[i].clone(), tile)]
           for i, tile in enumerate((k_tile, q_tile, k_tile))]
    hip_sdpa.sdpa_bwd_grid(*ins, *out, q_seq, k_seq, q_tile, k_tile, m, n_batch=n_batch,
                           kv_group=group, causal_offset=offset, flags=flags, n_slabs=n_slabs)
    torch.cuda.synchronize()
    per_slab = [len(x) // n_slabs for x in out]
    return [[_join(out[i][s * n:(s + 1) * n]) for i, n in enumerate(per_slab)]
            for s in range(n_slabs)]


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("head", [64, 128])
@pytest.mark.parametrize("mode,shape", [("causal", s) for s in GROUPED + SINGLE]
                         + [("none", s) for s in GROUPED])
def test_gradients_of_a_grid_by_two_groups(dtype, head, mode, shape):
    q_seq, k_seq, q_tile, k_tile, n_batch, group, n_kv, n_slabs = shape
    print("case bwd grid two groups", dtype, head, mode, shape, flush=True)
    n_dkv = n_slabs * n_batch * n_kv * -(-k_seq // 128)
    n_dq = n_slabs * n_batch * n_kv * group * -(-q_seq // 128)
    assert 2 * n_dkv + n_dq > 512 and n_dkv <= (256 if mode == "causal" else 192)
    assert max(-(-q_seq // 64) * group, -(-k_seq // 64)) >= 13
    slabs, seen, offset, m = _inputs(shape, head, dtype, mode, 61)
    kv = _kv_of(n_batch * group * n_kv, n_batch, group)
    for flags in (0, hip_sdpa.OVERWRITE):
        add = flags == 0
        start = [[(0.25 * torch.randn_like(s[i], dtype=torch.float32)).to(s[i].dtype) if add
                  else torch.full_like(s[i], float("nan")) for i in range(3)] for s in slabs]
        got = _grid_call(slabs, start, shape, offset, m, flags)
        for (K, Q, V, A, G, lse), st, g in zip(slabs, start, got):
            want = _gradients(Q, K, V, A, G, seen, kv, lse)
            for name, a, w, s in zip(("dK", "dQ", "dV"), g, want, st):
                w = w + s.double() if add else w
                err = float((a.double() - w).norm() / w.norm())
                assert err < TOL[dtype], (name, flags, err)
        if n_slabs == 1:
            K, Q, V, A, G, lse = slabs[0]
            one = [t.clone() for t in start[0]]
            hip_sdpa.sdpa_bwd_tile(K, Q, V, A, G, None, lse, *one, m, n_batch=n_batch,
                                   kv_group=group, causal_offset=offset, flags=flags)
            torch.cuda.synchronize()
            for a, o in zip(got[0], one):
                assert torch.equal(a.view(torch.int16), o.view(torch.int16)), flags


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("mode", ["causal", "none"])
def test_slabs_across_the_line_of_the_form(dtype, mode):
    """Two slabs of ten heads of 64, 1024 rows: each by itself is a launch of 240
    workgroups, whose walks two groups share, both together are one of 480 and walk in
    one group.  The sums are the same but for the order of their fp32 additions, so
    the gradients are equal but for their last rounding: half a step of the tile
    type's mantissa in each, 2^-8 and 2^-11 of a value in all at the most."""
    shape, head = (1024, 1024, 256, 512, 1, 1, 10, 2), 64
    slabs, seen, offset, m = _inputs(shape, head, dtype, mode, 62)
    start = [[torch.zeros_like(s[i]) for i in range(3)] for s in slabs]
    both = _grid_call(slabs, start, shape, offset, m, 0)
    for s, (slab, st) in enumerate(zip(slabs, start)):
        one, = _grid_call([slab], [st], shape[:-1] + (1,), offset, m, 0)
        for name, a, b in zip(("dK", "dQ", "dV"), both[s], one):
            assert torch.isfinite(a).all()
            err = float((a.float() - b.float()).norm() / b.float().norm())
            assert err < {"bf16": 2.0 ** -8, "fp16": 2.0 ** -11}[dtype], (name, err)
