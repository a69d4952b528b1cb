"""The backward whose walks are at most two blocks of 64: the gradient launch takes the row
dots and the classes of a mask's blocks itself.  Against 64-bit arithmetic at the edges of
the rule (128 queries of all heads of a group, 128 keys), and bit for bit against the same
rows as one of several slabs, which have the launch in front."""
import numpy as np
import pytest
import torch

from nntile_amd import hip_sdpa
from . import helpers as H
from .test_gpu_backward_halved_steps import MODES, _case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("mode", sorted(MODES))
@pytest.mark.parametrize("head,group,q_seq,k_seq,add", [
    (64, 1, 1, 128, False), (64, 1, 128, 1, True), (64, 1, 128, 128, False), (64, 1, 127, 65, True),
    (64, 2, 64, 128, True), (64, 2, 33, 100, False), (64, 128, 1, 90, False), (64, 2, 65, 128, False),
    (64, 1, 129, 128, False), (64, 1, 128, 129, True),
    (128, 1, 128, 128, True), (128, 1, 65, 127, False), (128, 4, 32, 128, False), (128, 3, 43, 64, True)])
def test_edges_of_the_rule(dtype, mode, head, group, q_seq, k_seq, add):
    print("case bwd short", dtype, mode, head, group, q_seq, k_seq, add, flush=True)
    _case(mode, head, group, 2, q_seq, k_seq, dtype, add)


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("mode", ["none", "causal"])
@pytest.mark.parametrize("head,group,q_seq,k_seq", [
    (64, 1, 128, 128), (64, 1, 50, 77), (64, 2, 64, 128), (128, 1, 128, 100), (128, 4, 31, 128)])
def test_same_bits_as_with_the_launch_in_front(dtype, mode, head, group, q_seq, k_seq):
    print("case bwd short slabs", dtype, mode, head, group, q_seq, k_seq, flush=True)
    kw = dict(n_batch=2, kv_group=group, causal_offset=max(k_seq - q_seq, 0), flags=hip_sdpa.OVERWRITE)
    ins_all, out_all, out_one = [[] for _ in range(6)], [[], [], []], [[], [], []]
    for s in range(2):
        (Q, K, V), _ = H.make_qkv(31 + s, 4 * group, q_seq, k_seq, head, dtype, kv_batch=4)
        rng = np.random.default_rng(7 + s)
        A, G = (H.rounded(rng.standard_normal(tuple(Q.shape)), dtype)[0] for _ in range(2))
        lse = torch.from_numpy(np.log1p(rng.random((4 * group, q_seq))).astype(np.float32)) + 3.0
        ins = [[x.cuda()] for x in (K, Q, V, A, G, lse)]
        one = [[torch.full(x.shape, float("nan"), dtype=x.dtype, device="cuda")] for x in (K, Q, V)]
        hip_sdpa.sdpa_bwd_grid(*ins, *one, q_seq, k_seq, q_seq, k_seq, MODES[mode], **kw)
        for dst, src in zip(ins_all, ins):
            dst += src
        for dst, src in zip(out_one, one):
            dst += src
        for dst, src in zip(out_all, one):
            dst.append(torch.empty_like(src[0]))
    hip_sdpa.sdpa_bwd_grid(*ins_all, *out_all, q_seq, k_seq, q_seq, k_seq, MODES[mode], n_slabs=2, **kw)
    torch.cuda.synchronize()
    for got, want, name in zip(out_all, out_one, ("dK", "dQ", "dV")):
        for s in range(2):
            assert not torch.isnan(want[s]).any(), (name, s)
            assert torch.equal(got[s].view(torch.int16), want[s].view(torch.int16)), (name, s)


@pytest.mark.parametrize("name", ["dQ", "dK", "dV"])
@pytest.mark.parametrize("grid", [False, True])
@pytest.mark.parametrize("head,rows", [(64, 128), (128, 100)])
def test_gradient_in_the_memory_of_A(head, rows, name, grid):
    # A is read before a gradient is written: the same bits as with memory of its own
    print("case bwd short into A", head, rows, name, grid, flush=True)
    batch = 6
    (Q, K, V), _ = H.make_qkv(41, batch, rows, rows, head, "bf16")
    rng = np.random.default_rng(11)
    A, G = (H.rounded(rng.standard_normal(tuple(Q.shape)), "bf16")[0] for _ in range(2))
    lse = torch.from_numpy(np.log1p(rng.random((batch, rows))).astype(np.float32)) + 3.0
    Q, K, V, A, G, lse = (x.cuda() for x in (Q, K, V, A, G, lse))

    def run(shared):
        a = A.clone()
        outs = [a if n == shared else torch.empty_like(a) for n in ("dK", "dQ", "dV")]
        if grid:
            hip_sdpa.sdpa_bwd_grid(*([x] for x in (K, Q, V, a, G, lse)), *([x] for x in outs), rows, rows,
                                   rows, rows, hip_sdpa.MASK_CAUSAL, flags=hip_sdpa.OVERWRITE)
        else:
            hip_sdpa.sdpa_bwd_tile(K, Q, V, a, G, None, lse, *outs, hip_sdpa.MASK_CAUSAL,
                                   flags=hip_sdpa.OVERWRITE)
        torch.cuda.synchronize()
        return outs

    for got, want in zip(run(name), run(None)):
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))
