"""Launches that keep two groups of wavefronts a workgroup beside the halved steps: the
forward with masks given as values whose keys outgrow an XCD's L2, scanned by workgroups of
the same launch, against 64-bit arithmetic; the backward over a grid whose workgroups of 64
rows would be too many, against 64-bit arithmetic and bit for bit the call over one
allocation; and gradients of slabs on either side of that line."""
import pytest
import torch

from nntile_amd import hip_sdpa
from . import helpers as H
from .test_gpu_backward_grid_two_groups import TOL, _gradients, _grid_call, _inputs, _kv_of

pytestmark = pytest.mark.gpu


# 240 and 245 workgroups of 128 queries, 47 and 97 key steps: two entries of head 64, three
# of head 128 on an XCD are more than 3 MiB of keys
@pytest.mark.parametrize("kind", ["causal", "window", "late"])
@pytest.mark.parametrize("head,batch,seq,dtype", [(128, 10, 3000, "bf16"), (64, 5, 6200, "fp16")])
def test_two_groups_behind_scanning_workgroups(kind, head, batch, seq, dtype):
    print("case two groups scanned", kind, head, batch, seq, dtype, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(seq)
    K, Q, V = (torch.randn(batch, seq, head, generator=gen, device="cuda").to(H.TORCH_DT[dtype]) for _ in range(3))
    i, j = torch.arange(seq, device="cuda")[:, None], torch.arange(seq, device="cuda")[None, :]
    seen = {"causal": j <= i, "window": (i - j).abs() <= 32, "late": (j >= 200 + i // 8) | (j == i)}[kind]
    mask = H.additive_mask(seen.cpu().numpy(), dtype).cuda()
    outs = []
    for scratch in (True, False):
        lse = torch.full((batch, seq), float("-inf"), device="cuda")
        A = torch.full_like(Q, float("nan"))
        hip_sdpa.flash_sdpa_fwd(K, Q, mask, lse, V, A, torch.empty_like(lse) if scratch else None)
        torch.cuda.synchronize()
        outs.append((lse, A))
    assert torch.equal(outs[0][0], outs[1][0])
    assert torch.equal(outs[0][1].view(torch.int16), outs[1][1].view(torch.int16))
    form = torch.full((batch, seq), float("nan"), device="cuda"), torch.full_like(Q, float("nan"))
    hip_sdpa.sdpa_fwd_tile(K, Q, mask, form[0], V, form[1], hip_sdpa.MASK_ADDITIVE,
                           flags=hip_sdpa.FORM_SPLIT | hip_sdpa.OVERWRITE)
    torch.cuda.synchronize()
    assert torch.equal(outs[0][1].view(torch.int16), form[1].view(torch.int16))
    for b in range(batch):
        s = (Q[b].double() @ K[b].double().t().contiguous() / head ** 0.5).masked_fill(~seen, float("-inf"))
        want, want_lse = torch.softmax(s, dim=1) @ V[b].double(), torch.logsumexp(s, dim=1)
        row, off = H.row_errors(H.to_np(outs[0][1][b]), want.cpu().numpy(), H.to_np(outs[0][0][b]),
                                want_lse.cpu().numpy())
        assert off < H.LSE_TOL[dtype], (b, off)
        assert row < H.ROW_TOL[dtype], (b, row)


# q_seq, k_seq, q_tile, k_tile, n_batch, group, n_kv, n_slabs
GRIDS = [
    (130, 300, 128, 256, 1, 8, 60, 1),      # ragged last tiles of 2 and 44 rows
    (130, 300, 128, 256, 1, 8, 30, 2),      # the same entries in two slabs
    (130, 200, 130, 200, 1, 8, 75, 1),      # one tile an axis
]


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("mode", ["causal", "none"])
@pytest.mark.parametrize("shape", GRIDS)
def test_gradients_of_a_grid_in_two_groups_at_head_64(dtype, mode, shape):
    q_seq, k_seq, q_tile, k_tile, n_batch, group, n_kv, n_slabs = shape
    print("case bwd grid, head 64", dtype, mode, shape, flush=True)
    entries = n_slabs * n_batch * n_kv
    # too many key blocks of 64 for halved steps, few enough of 128 for two groups
    assert entries * -(-k_seq // 64) > 256 and entries * -(-k_seq // 128) <= (256 if mode == "causal" else 192)
    assert entries * (-(-k_seq // 64) + group * -(-q_seq // 64)) > 1024 and group * -(-q_seq // 64) >= 13
    slabs, seen, offset, m = _inputs(shape, 64, dtype, mode, 63)
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
            hip_sdpa.sdpa_bwd_tile(K, Q, V, A, G, None, lse, *one, m, n_batch=n_batch, kv_group=group,
                                   causal_offset=offset, flags=flags)
            torch.cuda.synchronize()
            for a, o in zip(got[0], one):
                assert torch.equal(a.view(torch.int16), o.view(torch.int16)), flags


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("mode,heads", [("causal", 24), ("none", 16)])
def test_slabs_on_either_side_of_halved_steps(dtype, mode, heads):
    """Heads of 64, 1024 rows: one slab is a launch of 768 (512) workgroups of 64 rows,
    which halve their steps, two slabs together are twice as many and take whole ones.
    The sums are the same but for the order of their fp32 additions, so the gradients
    are equal but for their last rounding: half a step of the tile type's mantissa in each,
    2^-8 and 2^-11 of a value in all at the most."""
    shape, head = (1024, 1024, 256, 512, 1, 1, heads, 2), 64
    limit = 1024 if mode == "causal" else 512
    assert heads * 32 <= limit < 2 * heads * 32
    slabs, _, offset, m = _inputs(shape, head, dtype, mode, 64)
    start = [[torch.zeros_like(s[i]) for i in range(3)] for s in slabs]
    both = _grid_call(slabs, start, shape, offset, m, 0)
    for s, (slab, st) in enumerate(zip(slabs, start)):
        one, = _grid_call([slab], [st], shape[:-1] + (1,), offset, m, 0)
        for name, a, b in zip(("dK", "dQ", "dV"), both[s], one):
            assert torch.isfinite(a).all()
            err = float((a.float() - b.float()).norm() / b.float().norm())
            assert err < {"bf16": 2.0 ** -8, "fp16": 2.0 ** -11}[dtype], (name, err)
