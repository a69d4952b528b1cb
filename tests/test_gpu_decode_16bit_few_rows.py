"""The 16-bit decode of head 128 with at most 16 rows a unit, whose wavefronts share
the two halves of a step's keys and of the head: against 64-bit arithmetic at the
edges of half a step, of a step and of the direct form, with one half hidden, and one
row more than the form takes."""
import numpy as np
import pytest
import torch

from nntile_amd import hip_sdpa

pytestmark = pytest.mark.gpu

# Half an ulp each for the probabilities, the partial outputs and the results, which
# are independent: sqrt(3) of it in the 2-norm at most; a fourth for what the sums add.
ULP = {"bf16": 2.0 ** -8, "fp16": 2.0 ** -11}
DTYPE = {"bf16": torch.bfloat16, "fp16": torch.float16}


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("group,q_seq", [(1, 1), (4, 1), (3, 5), (4, 4), (1, 17)])
@pytest.mark.parametrize("mode", ["none", "causal", "first half", "second half", "running pair"])
def test_against_64_bits(dtype, group, q_seq, mode):
    n_batch, n_kv, head = 2, 3, 128
    for k_seq in (17, 31, 33, 64, 65, 97, 192, 193, 225, 1000):
        print("case", dtype, group, q_seq, mode, k_seq, flush=True)
        g = torch.Generator().manual_seed(k_seq)
        Q, K, V = [torch.randn(n_batch * n_kv * r, s, head, generator=g).to(DTYPE[dtype])
                   for r, s in ((group, q_seq), (1, k_seq), (1, k_seq))]
        # the batch index is nb + n_batch * (group member + group * kv head)
        kv = [b % n_batch + n_batch * (b // (n_batch * group)) for b in range(Q.shape[0])]
        s = torch.matmul(Q.double(), K[kv].double().transpose(1, 2).contiguous()) / np.sqrt(head)
        keys = torch.arange(k_seq)
        mask = None
        if mode == "causal":
            s = s.masked_fill(keys > torch.arange(q_seq)[:, None] + k_seq - q_seq, float("-inf"))
        elif mode.endswith("half"):     # the other 32 keys of every step hidden, and of row 0 all
            mask = ((keys // 32 % 2) == ("first", "second").index(mode.split()[0])).repeat(q_seq, 1)
            mask[0] &= q_seq == 1
            s = s.masked_fill(~mask, float("-inf"))
            mask = mask.cuda()
        lse0 = torch.full(Q.shape[:2], 0.5)
        A0 = torch.randn(Q.shape, generator=g).to(DTYPE[dtype])
        overwrite = mode != "running pair"
        if not overwrite:
            s = torch.cat((s, lse0[..., None].double()), 2)
        want_lse = torch.logsumexp(s, 2)
        w = torch.exp(s - want_lse[..., None]).nan_to_num(0.0)
        want = torch.matmul(w[..., :k_seq], V[kv].double())
        if not overwrite:
            want += w[..., k_seq:] * A0.double()
        lse, A, Kd, Qd = lse0.cuda(), A0.cuda(), K.cuda(), Q.cuda()
        ws = torch.empty(hip_sdpa.decode_workspace_bytes(Kd, Qd, n_batch, group), dtype=torch.uint8,
                         device="cuda")
        hip_sdpa.sdpa_fwd_decode(
            Kd, Qd, mask, lse, V.cuda(), A,
            hip_sdpa.MASK_BOOL if mask is not None else hip_sdpa.MASK_CAUSAL if mode == "causal"
            else hip_sdpa.MASK_NONE, n_batch, group, ws, causal_offset=k_seq - q_seq,
            flags=hip_sdpa.OVERWRITE if overwrite else 0)
        torch.cuda.synchronize()
        seen = torch.isfinite(want_lse)
        assert torch.equal(torch.isfinite(lse.cpu()), seen)
        assert not A.cpu()[~seen].any()
        if seen.any():      # (17 keys: the second half is beyond them)
            assert float((A.cpu().double() - want)[seen].norm() / want[seen].norm()) < ULP[dtype]
            assert float((lse.cpu().double() - want_lse)[seen].abs().max()) < 1e-5


@pytest.mark.parametrize("q_seq", [1, 17])
@pytest.mark.parametrize("units", [256, 257, 512, 513])
def test_units_of_one_round(units, q_seq):
    """More units than CUs that fit the chip's places without a key split, and one unit
    on either side."""
    k_seq, head = 300, 128
    print("case", units, q_seq, flush=True)
    g = torch.Generator().manual_seed(units)
    Q, K, V = [torch.randn(units, s, head, generator=g).to(torch.bfloat16) for s in (q_seq, k_seq, k_seq)]
    s = torch.matmul(Q.double(), K.double().transpose(1, 2).contiguous()) / np.sqrt(head)
    s = s.masked_fill(torch.arange(k_seq) > torch.arange(q_seq)[:, None] + k_seq - q_seq, float("-inf"))
    want_lse = torch.logsumexp(s, 2)
    want = torch.matmul(torch.exp(s - want_lse[..., None]), V.double())
    lse, A, Kd, Qd = torch.zeros(Q.shape[:2], device="cuda"), torch.zeros_like(Q).cuda(), K.cuda(), Q.cuda()
    ws = torch.empty(hip_sdpa.decode_workspace_bytes(Kd, Qd, units, 1), dtype=torch.uint8, device="cuda")
    hip_sdpa.sdpa_fwd_decode(Kd, Qd, None, lse, V.cuda(), A, hip_sdpa.MASK_CAUSAL, units, 1, ws,
                             causal_offset=k_seq - q_seq, flags=hip_sdpa.OVERWRITE)
    torch.cuda.synchronize()
    assert float((A.cpu().double() - want).norm() / want.norm()) < ULP["bf16"]
    assert float((lse.cpu().double() - want_lse).abs().max()) < 1e-5
