"""Blocks of a mask given as values that hold exactly the rule `key <= query`
run without reading the mask; one element off the rule and the block's values
are read.  Against the same call without room for the classes (every value
read) on shapes at and off the block edges, and, for the rule itself, against
the call with the rule as a mode."""
import numpy as np
import pytest
import torch

from nntile_amd import hip_sdpa
from . import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["additive", "bool"])
@pytest.mark.parametrize("head", [32, 64, 128])
@pytest.mark.parametrize("q_seq,k_seq", [(64, 64), (128, 65), (197, 261), (3, 2), (130, 16), (66, 194),
                                          (130, 131)])
@pytest.mark.parametrize("flip", [None, (1, 0), (64, 64), (63, 64), (128, 15), (196, 196)])
def test_rule_blocks(form, head, q_seq, k_seq, flip, batch=2, dtype="fp16"):
    if flip is not None and (flip[0] >= q_seq or flip[1] >= k_seq):
        flip = (q_seq - 1, 0)
    print("case bwd rule", form, head, q_seq, k_seq, flip, flush=True)
    mask = np.arange(k_seq)[None, :] <= np.arange(q_seq)[:, None]
    if flip is not None:
        mask[flip] = not mask[flip]
    (Q, K, V), _ = H.make_qkv(51, batch, q_seq, k_seq, head, dtype)
    G = H.make_qkv(52, batch, q_seq, q_seq, head, dtype)[0][0].cuda()
    Q, K, V = Q.cuda(), K.cuda(), V.cuda()
    m = (H.additive_mask(mask, dtype) if form == "additive" else torch.from_numpy(mask.copy())).cuda()
    mode = hip_sdpa.MASK_ADDITIVE if form == "additive" else hip_sdpa.MASK_BOOL
    lse, A = H.fresh_outputs(batch, q_seq, head, dtype)
    hip_sdpa.sdpa_fwd_tile(K, Q, m, lse, V, A, mode, flags=hip_sdpa.OVERWRITE)

    def grads(mask_, mode_, ws):
        out = [torch.full_like(t, float("nan")) for t in (K, Q, V)]
        hip_sdpa.sdpa_bwd_tile(K, Q, V, A, G, mask_, lse, *out, mode_, flags=hip_sdpa.OVERWRITE,
                               workspace=ws)
        torch.cuda.synchronize()
        return [t.float() for t in out]

    small = torch.empty(4 * q_seq * batch, dtype=torch.uint8, device="cuda")
    got, want = grads(m, mode, None), grads(m, mode, small)
    others = [want] if flip is not None else [want, grads(None, hip_sdpa.MASK_CAUSAL, None)]
    for other in others:
        for g, w, name in zip(got, other, ("dK", "dQ", "dV")):
            assert torch.isfinite(g).all(), name
            assert (g - w).abs().max() <= 2e-3 * w.abs().max(), (name, (g - w).abs().max())
