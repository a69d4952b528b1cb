"""The native front-end of the binding refuses what is not a device tile with
the exceptions its Python wrappers document (no GPU needed)."""
import ctypes
import os
import re
import threading
import time
import types

import pytest
import torch

from nntile_amd import build as B
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


def test_the_interpreter_lock_is_released_during_the_c_call():
    """A prepared call of sem_timedwait, given up by this thread while another
    one is inside it: with the lock held, nobody could, and the wait would time
    out.  (A launch into a full queue blocks just so.)"""
    libc = ctypes.CDLL(None)
    sem = ctypes.create_string_buffer(64)       # (larger than any sem_t)
    assert libc.sem_init(sem, 0, 0) == 0
    until = (ctypes.c_long * 2)(int(time.time()) + 10, 0)
    call = h._native().Launch(ctypes.cast(libc.sem_timedwait, ctypes.c_void_p).value,
                              ctypes.addressof(until), ()).call
    inside, got = threading.Event(), []

    def wait():
        inside.set()
        got.append(call(types.SimpleNamespace(cuda_stream=ctypes.addressof(sem))))

    t = threading.Thread(target=wait)
    t.start()
    inside.wait()
    time.sleep(0.2)         # (long enough for the thread to be in the call)
    libc.sem_post(sem)
    t.join()
    assert got == [0]


def test_every_launch_goes_through_the_form_that_releases_the_lock():
    with open(os.path.join(B.CSRC, "front.cpp")) as f:
        text = f.read()
    called = set(re.findall(r"\b(nntile_hip_\w+)\(", text))
    assert called == {"nntile_hip_sdpa_fwd_decode_workspace_bytes_fp32",
                      "nntile_hip_sdpa_fwd_decode_workspace_bytes"}
    assert not re.search(r"_fns\[[^]]*\]\(|\)\(s\b|fn\(s\b", text)


def test_another_torch_makes_the_front_end_stale(monkeypatch):
    """It reads torch's C++ objects: built against another torch it is built
    again, and refused where that was not done."""
    monkeypatch.setattr(B, "_stale", lambda obj, src: False)     # (no source is newer)
    assert not B._front_stale()
    monkeypatch.setattr(torch, "__version__", "1.2.3")
    assert B._front_stale()
    monkeypatch.setattr(h, "_front", None)
    with pytest.raises(RuntimeError, match="another build of torch"):
        h._native()
    monkeypatch.undo()
    monkeypatch.setattr(h, "_front", None)
    assert h._native().TAG
