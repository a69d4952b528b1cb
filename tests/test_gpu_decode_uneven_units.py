"""Decode calls whose (batch entry, kv head) units do not come in eights, and
the edges of the rule that splits their keys (one workgroup up to three steps
of 64 keys, a split per step up to eight, then two steps a split at least):
the merge in the launch and the merge as a second launch give the same bits,
and both agree with the tile kernel."""
import pytest
import torch

from nntile_amd import hip_sdpa
from . import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("head", [64, 128])
@pytest.mark.parametrize("n_batch,n_head_kv,group,q_seq", [(1, 1, 8, 1), (3, 1, 1, 5), (3, 3, 4, 4),
                                                           (4, 5, 4, 16), (1, 12, 1, 1)])
@pytest.mark.parametrize("k_seq", [1, 96, 129, 192, 193, 512, 513, 1100, 4200])
def test_merge_forms_agree(dtype, head, n_batch, n_head_kv, group, q_seq, k_seq):
    print("case uneven", dtype, head, n_batch, n_head_kv, group, q_seq, k_seq, flush=True)
    q_seq = min(q_seq, k_seq)
    units = n_batch * n_head_kv
    (Q, _, _), _ = H.make_qkv(61, units * group, q_seq, q_seq, head, dtype)
    (_, K, V), _ = H.make_qkv(62, units, k_seq, k_seq, head, dtype)
    Q, K, V = Q.cuda(), K.cuda(), V.cuda()
    offset = k_seq - q_seq
    ws = torch.empty(hip_sdpa.decode_workspace_bytes(K, Q, n_batch, group), dtype=torch.uint8,
                     device="cuda")
    outs = []
    for flags in (0, hip_sdpa.DECODE_SEPARATE_MERGE):
        lse, A = H.fresh_outputs(units * group, q_seq, head, dtype)
        for part in (0, 1):       # onto an empty pair, then onto its own result
            hip_sdpa.sdpa_fwd_decode(K, Q, None, lse, V, A, hip_sdpa.MASK_CAUSAL, n_batch, group, ws,
                                     causal_offset=offset, flags=flags)
        torch.cuda.synchronize()
        outs.append((lse, A))
    assert torch.equal(outs[0][0], outs[1][0])
    assert torch.equal(outs[0][1].view(torch.uint8), outs[1][1].view(torch.uint8))
    lse, A = H.fresh_outputs(units * group, q_seq, head, dtype)
    for part in (0, 1):
        hip_sdpa.sdpa_fwd_tile(K, Q, None, lse, V, A, hip_sdpa.MASK_CAUSAL, n_batch=n_batch,
                               kv_group=group, causal_offset=offset)
    torch.cuda.synchronize()
    tol = {"bf16": 1e-2, "fp16": 1e-3, "fp32": 1e-5}[dtype]
    assert H.rel_fro(H.to_np(outs[0][1]), H.to_np(A)) < tol
    assert H.rel_fro(outs[0][0].cpu().numpy(), lse.cpu().numpy()) < 1e-5
