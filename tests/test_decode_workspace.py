"""The decode workspace sized once for the longest cache serves every shorter
one: the size never falls as the keys grow.  (Fewer splits for more keys - from
nine steps on a split takes two at least - must not show in it.)"""
import ctypes

import pytest

from nntile_amd import hip_sdpa


def sizes(fp32, units, group, q_seq, head, lengths):
    fn = getattr(hip_sdpa.lib(), "nntile_hip_sdpa_fwd_decode_workspace_bytes" + ("_fp32" if fp32 else ""))
    a = hip_sdpa.TileArgs()
    a.batch, a.q_seq, a.head, a.n_batch, a.kv_group = units * group, q_seq, head, 1, group
    for k in lengths:
        a.k_seq = k
        yield int(fn(ctypes.byref(a)))


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("head", [64, 128])
@pytest.mark.parametrize("units,group,q_seq", [(1, 1, 1), (8, 4, 1), (12, 1, 3), (36, 4, 16), (64, 4, 16),
                                               (200, 1, 1), (600, 1, 1)])
def test_size_never_falls_with_more_keys(fp32, head, units, group, q_seq):
    got = list(sizes(fp32, units, group, q_seq, head, range(1, 5000, 7)))
    assert got[0] > 0 and all(a <= b for a, b in zip(got, got[1:]))
