"""The fp32 decode with at most 16 or 32 rows a unit, whose wavefronts share a step's
two key blocks and the two halves of the head or of the rows: against 64-bit
arithmetic at the edges of a key block, of a step and of the direct form, with one
key block hidden, and one row more than the forms take."""
import numpy as np
import pytest
import torch

from nntile_amd import hip_sdpa

pytestmark = pytest.mark.gpu

# A score is a sum of up to 128 products rounded to 2^-24 of its running value, a few
# units at these inputs, so a probability is off by some 2^-22; over the keys these
# average out and the sums add about sqrt(keys) * 2^-24: below 1e-6 at 700 keys.
TOL = 1e-6


@pytest.mark.parametrize("head", [64, 128])
@pytest.mark.parametrize("group,q_seq", [(1, 1), (4, 1), (3, 5), (4, 4), (1, 17), (2, 16), (3, 11)])
@pytest.mark.parametrize("mode", ["none", "causal", "first block", "second block", "running pair"])
def test_against_64_bits(head, group, q_seq, mode):
    n_batch, n_kv = 2, 3
    for k_seq in (17, 31, 33, 96, 97, 128, 129, 300, 700):
        print("case", head, group, q_seq, mode, k_seq, flush=True)
        g = torch.Generator().manual_seed(k_seq)
        Q, K, V = [torch.randn(n_batch * n_kv * r, s, head, generator=g)
                   for r, s in ((group, q_seq), (1, k_seq), (1, k_seq))]
        # the batch index is nb + n_batch * (group member + group * kv head)
        kv = [b % n_batch + n_batch * (b // (n_batch * group)) for b in range(Q.shape[0])]
        s = torch.matmul(Q.double(), K[kv].double().transpose(1, 2).contiguous()) / np.sqrt(head)
        keys = torch.arange(k_seq)
        mask = None
        if mode == "causal":
            s = s.masked_fill(keys > torch.arange(q_seq)[:, None] + k_seq - q_seq, float("-inf"))
        elif mode.endswith("block"):    # the other 16 keys of every step hidden, and of row 0 all
            mask = ((keys // 16 % 2) == ("first", "second").index(mode.split()[0])).repeat(q_seq, 1)
            mask[0] &= q_seq == 1
            s = s.masked_fill(~mask, float("-inf"))
            mask = mask.cuda()
        lse0 = torch.full(Q.shape[:2], 0.5)
        A0 = torch.randn(Q.shape, generator=g)
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
        if seen.any():      # (17 keys and a row whose only block is the hidden one)
            assert float((A.cpu().double() - want)[seen].norm() / want[seen].norm()) < TOL
            assert float((lse.cpu().double() - want_lse)[seen].abs().max()) < TOL * 8
