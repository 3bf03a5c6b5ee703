"""Scores near the lowest finite value.  The running max starts there and a
masked row counts as -inf, so rows of very negative but finite scores must
still give the softmax of those scores.  The scores are so far apart that the
softmax picks one row: the output is that row's v."""
import numpy as np
import pytest

from leap_amd.attention import HipAttention
from oracle import oracle as O
from tests.helpers import assert_close, normal, rng_for, rope_f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nh,nkv,hd,T", [
    (32, 8, 128, 20), (32, 8, 128, 64), (32, 8, 128, 700), (8, 8, 128, 65), (24, 8, 128, 130),
    (32, 4, 64, 33), (32, 4, 64, 600), (64, 8, 128, 300), (64, 8, 128, 3000), (128, 8, 128, 90),
])
@pytest.mark.parametrize("new_token", ["lowest", "highest"])
def test_very_negative_scores(hip_device, nh, nkv, hd, T, new_token):
    rng = rng_for(91, nh, nkv, hd, T)
    G, pos = nh // nkv, T - 1
    with HipAttention(nh, nkv, hd, T) as att:
        c, s = att.rope_download(pos, T)
        # every head of a group has the same q, so that one direction serves it
        qk = normal(rng, (nkv, hd), 1) * np.float32(1e15)
        q = np.repeat(qk, G, axis=0).reshape(-1)
        unit = (qk / np.linalg.norm(qk, axis=1, keepdims=True)).astype(np.float32)
        rot = rope_f32(unit.reshape(-1), c[0], s[0])
        # row t's score: -1e15 |q| ... times (2 + t mod 37), row 5 (or the last) the least negative
        f = (2.0 + np.arange(pos) % 37).astype(np.float32)
        f[min(5, pos - 1)] = 1.0
        k_rows = -(f[:, None] * np.float32(1e15)) * rot[None, :]
        v_rows = normal(rng, (pos, nkv * hd), hd)
        k = unit.reshape(-1) * np.float32(-1e17 if new_token == "lowest" else 1.0)
        v = normal(rng, nkv * hd, hd)
        att.kv_upload(0, 0, 0, k_rows, v_rows)
        out = att.step(0, pos, q, k, v)
        orc = O.Oracle(1, nh, nkv, hd, T)
        orc.key_cache[0, :pos], orc.value_cache[0, :pos] = k_rows, v_rows
        want, _ = orc.step(0, pos, q, k, v)
        picked = v_rows[min(5, pos - 1)] if new_token == "lowest" else v
        expect = np.repeat(picked.reshape(nkv, hd), G, axis=0).reshape(-1)
        assert np.array_equal(want, expect)
        assert_close(out, expect, rel=1e-6)
