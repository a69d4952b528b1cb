"""The native front-end of the binding refuses what is not a device tile with
the exceptions its Python wrappers document (no GPU needed)."""
import pytest
import torch

from nntile_amd import hip_sdpa as h
from nntile_amd.kv_cache import KVCache

T = torch.zeros(2, 8, 64, dtype=torch.bfloat16)
L = torch.zeros(2, 8)
CALLS = {
    "flash_sdpa_fwd": lambda t: h.flash_sdpa_fwd(t, t, None, L, t, t),
    "sdpa_fwd_tile": lambda t: h.sdpa_fwd_tile(t, t, None, L, t, t, h.MASK_NONE),
    "flash_sdpa_bwd": lambda t: h.flash_sdpa_bwd(t, t, t, t, t, t, L, t, t, t, t),
    "sdpa_bwd_tile": lambda t: h.sdpa_bwd_tile(t, t, t, t, t, None, L, t, t, t, h.MASK_NONE, workspace=L),
    "sdpa_fwd_decode": lambda t: h.sdpa_fwd_decode(t, t, None, L, t, t, h.MASK_NONE, 2, 1, L),
    "sdpa_fwd_decode_cache": lambda t: h.sdpa_fwd_decode_cache(t, t, 8, t, None, L, t, h.MASK_NONE, 2, 1, L),
    "sdpa_fwd_tile_cache": lambda t: h.sdpa_fwd_tile_cache(t, t, 8, t, None, L, t, h.MASK_NONE),
    "sdpa_fwd_decode_append_cache": lambda t: h.sdpa_fwd_decode_append_cache(
        t, t, t, t, 8, t, None, L, t, h.MASK_NONE, 2, 1, L),
    "kv_cache_append": lambda t: h.kv_cache_append(t, t, t, t, 0),
    "accumulate_attn_output": lambda t: h.accumulate_attn_output(L, t, L, t),
    "rope": lambda t: h.rope(L, L, t, t),
    "transpose": lambda t: h.transpose(1.0, t, t, 8, 128),
}


@pytest.mark.parametrize("name", sorted(CALLS))
def test_tensors_off_the_device_are_refused(name):
    with pytest.raises(ValueError, match="contiguous device tensors"):
        CALLS[name](T)


def test_objects_that_are_no_tensors_are_refused():
    with pytest.raises(TypeError, match="torch tensor"):
        h.transpose(1.0, [1, 2], T, 1, 2)


def test_a_step_into_a_cache_off_the_device_is_refused():
    cache = KVCache(16)
    cache.k = cache.v = torch.zeros(2, 16, 64, dtype=torch.bfloat16)
    one = torch.zeros(2, 1, 64, dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="contiguous device tensors"):
        cache.append_attend(one, one, one, torch.zeros(2, 1), one, 2, 1)
    assert len(cache) == 0
