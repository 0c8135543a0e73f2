"""The bf16 decode kernel at the places where it can go wrong: contexts around its 16-token groups, every number of query
heads a wavefront serves (4, 8, 16; 32 as two of 16), every head dim, pages that hold whole groups and pages that do not,
windows that start inside a group, and scores large enough to move the running maximum many times. Against the CpuOps
oracle within the attention-bf16 class of tests/cases.py; the one-launch mixed step against float32 torch."""
import numpy as np
import pytest

import cases
import roost_amd
from test_attention_gpu import Dev, _plan_overlap, run_case, torch_reference

pytestmark = pytest.mark.gpu

EDGES = [1, 15, 16, 17, 31, 32, 33, 63, 100, 257, 1000]


@pytest.mark.parametrize("hq,hkv", [(4, 1), (16, 4), (8, 1), (32, 4), (16, 1), (64, 2)],
                         ids=["g4", "g4x4", "g8", "g8x4", "g16", "g32x2"])
@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("ps,hnd,window", [(16, False, -1), (64, True, 40), (12, False, 21)],
                         ids=["ps16", "ps64 HND window", "ps12 window"])
def test_decode_group_and_page_edges(session, hq, hkv, d, ps, hnd, window):
    rng = np.random.default_rng(d + hq + ps)
    # std 2: score magnitudes of up to about 60 in log2 units, so a context's running maximum moves again and again.
    b = cases.make_paged_batch(rng, EDGES, [1] * len(EDGES), page_size=ps, hnd=hnd, hq=hq, hkv=hkv, d=d, std=2.0)
    got = run_case(session, b, window_left=window)
    ref = cases.values(cases.oracle_attention(b, window_left=window), True)
    cases.assert_attention_class(got, ref, float(np.abs(cases.values(b.v_cache, True)).max()), what="decode")


# Few rows, cut by themselves into pieces that are resident at once (or not cut at all), with fewer KV heads per workgroup
# than the full batch takes, empty rows among them; 64 rows around the line to the even deal.
@pytest.mark.parametrize("kv_lens", [[1], [16], [300], [1500], [9000], [0, 40, 0, 3000, 0], [17] * 9, [700, 1, 0, 5000, 33],
                                     [450 + 7 * i for i in range(64)]], ids=lambda k: f"{len(k)}x{max(k)}")
@pytest.mark.parametrize("hq,hkv,d,hnd", [(8, 2, 256, False), (32, 8, 128, True), (64, 4, 64, False)])
def test_decode_few_rows(session, kv_lens, hq, hkv, d, hnd):
    rng = np.random.default_rng(sum(kv_lens) + d)
    b = cases.make_paged_batch(rng, kv_lens, [1] * len(kv_lens), hq=hq, hkv=hkv, d=d, hnd=hnd, std=1.0)
    causal = 0 not in kv_lens  # the oracle refuses a causal row without keys; a decode row sees every key either way
    got = run_case(session, b, causal=causal)
    ref = cases.values(cases.oracle_attention(b, causal), True)
    cases.assert_attention_class(got, ref, float(np.abs(cases.values(b.v_cache, True)).max()), what="decode")


@pytest.mark.parametrize("hq,hkv,d", [(32, 4, 128), (32, 2, 128), (16, 2, 256), (16, 4, 64)])
def test_mixed_launch_query_head_groups(session, hq, hkv, d):
    rng = np.random.default_rng(hq + d)
    kv = [int(x) for x in rng.integers(6000, 12000, size=24)] + [1300]
    b = cases.make_paged_batch(rng, kv, [1] * 24 + [256], hq=hq, hkv=hkv, d=d, std=0.5)
    dev = Dev(b)
    key = ("mixed groups", hq, hkv, d)
    session.launch(session.lib.entry(roost_amd.ATTENTION_VARIANT), dev.params(), key=key)
    assert _plan_overlap(session, key) == 1
    cases.assert_close(dev.result(), torch_reference(b), what="mixed step vs fp32 torch")
