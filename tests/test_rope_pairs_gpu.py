"""Rope over whole chunk pairs at its edges: one to thirty-two chunk pairs a row, token counts around a workgroup's tokens and
threads, a width whose pairs are no power of two (the row form), f32; against the CpuOps oracle within the bounds of
tests/test_qk_rope_gpu.py, and every element past the rotated width left exactly as it was (NaN payloads too)."""
import numpy as np
import pytest

import oracle
import roost_amd
from test_attention_gpu import from_dev, to_dev
from test_qk_rope_gpu import _data, assert_rows_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bf16,hq,hk,hd,rot", [(True, 8, 2, 256, 64), (True, 3, 1, 64, 16), (True, 32, 8, 128, 0),
                                               (True, 2, 2, 512, 512), (True, 4, 1, 256, 48), (False, 4, 2, 128, 32),
                                               (False, 2, 1, 64, 8)])
@pytest.mark.parametrize("tokens", [1, 7, 65, 1100])
def test_rope_pairs(session, bf16, hq, hk, hd, rot, tokens):
    rng = np.random.default_rng(hd + rot + tokens)
    q, k = _data(rng, tokens * hq * hd, bf16), _data(rng, tokens * hk * hd, bf16)
    width = rot or hd
    if width < hd:  # a quiet NaN with a payload in every row's last element
        for a, heads in ((q, hq), (k, hk)):
            a.view(np.uint16 if bf16 else np.uint32).reshape(tokens * heads, hd)[:, -1] = 0x7FE5 if bf16 else 0x7FE50001
    pos = rng.integers(0, 1 << 18, tokens).astype(np.int32)
    want_q, want_k = q.copy(), k.copy()
    oracle.rope(want_q, want_k, pos, tokens=tokens, q_heads=hq, kv_heads=hk, head_dim=hd, theta=1e7, rotary_dim=rot)
    dq, dk = to_dev(q, bf16), to_dev(k, bf16)
    roost_amd.rope(session, dq, dk, to_dev(pos), tokens=tokens, q_heads=hq, kv_heads=hk, head_dim=hd, theta=1e7,
                   rotary_dim=rot)
    for got, want, before in ((from_dev(dq, bf16), want_q, q), (from_dev(dk, bf16), want_k, k)):
        g, w, b = (np.ascontiguousarray(a.reshape(-1, hd)) for a in (got, want, before))
        assert np.array_equal(g[:, width:].copy().view(np.uint8), b[:, width:].copy().view(np.uint8))
        assert_rows_close(np.ascontiguousarray(g[:, :width]), np.ascontiguousarray(w[:, :width]), bf16, width, "rope")
