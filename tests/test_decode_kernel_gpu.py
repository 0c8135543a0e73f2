"""The bf16 decode kernel at the places where it can go wrong: contexts around its 16-token groups, every number of query
heads a wavefront serves (4, 8, 16; 32 as two of 16), every head dim, pages that hold whole groups and pages that do not,
windows that start inside a group, and scores large enough to move the running maximum many times. Against the CpuOps
oracle within the attention-bf16 class of tests/cases.py; the one-launch mixed step against float32 torch."""
import ctypes as C
import dataclasses

import numpy as np
import pytest

import cases
import roost_amd
from test_attention_gpu import Dev, _plan_overlap, from_dev, run_case, to_dev, torch, torch_reference

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


def _staircase(rng, hq, hkv, d, rows, groups, v_bits):
    """Contexts whose 16-token groups each hold one visible key, its score a step above that of the group before (the step
    is left to q's first element); every value of V the same."""
    b = cases.make_paged_batch(rng, [16 * groups] * rows, [1] * rows, hq=hq, hkv=hkv, d=1, pool_factor=1.0)
    shape = b.k_cache.shape[:3] + (d,)
    k = np.zeros(shape, np.float32)
    k[..., 0] = -300.0
    for r in range(rows):
        k[b.kv_indices[b.kv_indptr[r]:b.kv_indptr[r + 1]], 0, :, 0] = np.arange(groups)[:, None]
    b.d, b.q = d, np.zeros((rows, hq, d), np.uint16)
    b.k_cache, b.v_cache = cases.bf16_bits(k), np.full(shape, v_bits, np.uint16)
    return b


@pytest.mark.parametrize("hq", [16, 32, 64, 128], ids=["g4", "g8", "g16", "g32"])
@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("v_bits", [0x3FFF, 0x7BFF], ids=["V 1.99", "V 2.65e36"])
def test_decode_rising_scores_keep_the_dominant_weight(session, hq, d, v_bits):
    """A head's largest weight is exactly 1 in bf16, whatever the scores before it. A wavefront's scores rise by a step of 2
    to 7.5 in log2 (another for every row and head) from each of its groups to the next, so the roundings of the other
    weights (2^-8 of each at most) move a row by at most 2^-8 * 2^-2: less than half a unit of V's last place (2^-9 of it,
    V's mantissa being full), and the output is V to the bit. A weight of up to 2^7.5 would also overflow: 2^7.5 * 2.65e36
    is past the largest float."""
    rng = np.random.default_rng(d + hq)
    rows, groups = 48, 64
    b = _staircase(rng, hq, 4, d, rows, groups, v_bits)
    dev = Dev(b)
    entry = session.lib.entry(roost_amd.ATTENTION_VARIANT)
    ws = session.prepare(entry, dev.params(), ("staircase", d, hq))
    words = np.frombuffer(C.string_at(ws.plan, ws.plan_bytes), np.uint64)
    waves = 4 // (int(words[5]) >> 32)  # wavefronts that take a head's groups in turn
    assert int(words[7]) * 2 * waves <= rows * groups, "the plan leaves a wavefront fewer than two groups"
    q = np.zeros(b.q.shape, np.float32)
    q[..., 0] = rng.uniform(2.0 / waves, 7.5 / waves, q.shape[:2]) * np.sqrt(d) / np.log2(np.e)
    dev.q.copy_(to_dev(cases.bf16_bits(q), True))
    session.run(entry, dev.params(), ws)
    got = from_dev(dev.out, True)
    assert (got == v_bits).all(), f"{(got != v_bits).sum()} of {got.size} outputs differ from V"


def _unwritten_is_nan(b, window, bad_page):
    """The batch with NaN wherever no query can look: page 0, pages of no sequence, a context's last page past its end and
    everything before its window. bad_page: one page in the middle of each context of three pages or more gets an id
    outside the pool. Returns the batch and one without those pages, whose result is the same (no window, not causal)."""
    nan = np.uint16(0x7FC0) if b.bf16 else np.float32(np.nan)
    b = dataclasses.replace(b, kv_indices=b.kv_indices + 1)
    rows = [(0, 2, 1, 3) if b.hnd else (0, 1, 2, 3)] * 2  # views with the token on axis 1
    pools = []
    for pool in (b.k_cache, b.v_cache):
        grown = np.full((pool.shape[0] + 1,) + pool.shape[1:], nan, pool.dtype)
        new, old = grown.transpose(rows[0]), pool.transpose(rows[0])
        for s, n in enumerate(b.kv_lens):
            for j in range(max(0, n - 1 - window) if window >= 0 else 0, n):
                page = b.kv_indices[b.kv_indptr[s] + j // b.page_size]
                new[page, j % b.page_size] = old[page - 1, j % b.page_size]
        pools.append(grown)
    b = dataclasses.replace(b, k_cache=pools[0], v_cache=pools[1])
    if not bad_page:
        return b, b
    idx, keep, lens = b.kv_indices.copy(), np.ones(b.kv_indices.size, bool), list(b.kv_lens)
    for s in range(b.batch):
        if b.kv_indptr[s + 1] - b.kv_indptr[s] >= 3:
            at = b.kv_indptr[s] + 1
            idx[at], keep[at] = (-1, pools[0].shape[0])[s % 2], False
            lens[s] -= b.page_size
    indptr = np.concatenate([[0], np.cumsum(keep)])[b.kv_indptr].astype(np.int32)
    without = dataclasses.replace(b, kv_indices=b.kv_indices[keep], kv_indptr=indptr, kv_lens=lens)
    return dataclasses.replace(b, kv_indices=idx), without


@pytest.mark.parametrize("hq,hkv,d,bf16", [(8, 2, 256, True), (32, 4, 128, True), (16, 1, 64, True), (8, 2, 256, False),
                                           (4, 1, 64, False)])
@pytest.mark.parametrize("ps,hnd,window,bad_page", [(16, False, -1, False), (12, False, -1, False), (64, True, 37, False),
                                                    (12, True, 21, False), (16, False, -1, True), (5, False, -1, True)])
def test_decode_reads_nothing_that_nobody_wrote(session, hq, hkv, d, bf16, ps, hnd, window, bad_page):
    """Cache rows outside the visible keys hold whatever the pool's memory held: NaN here. A masked key's weight is 0, but 0
    times NaN is NaN, so such rows must not enter the products."""
    rng = np.random.default_rng(d + hq + ps)
    b = cases.make_paged_batch(rng, EDGES + [2500], [1] * (len(EDGES) + 1), page_size=ps, hnd=hnd, hq=hq, hkv=hkv, d=d,
                               bf16=bf16)
    b, without = _unwritten_is_nan(b, window, bad_page)
    got = run_case(session, b, causal=not bad_page, window_left=window)
    ref = cases.values(cases.oracle_attention(without, not bad_page, window_left=window), bf16)
    if bf16:
        v = cases.values(b.v_cache, True)
        cases.assert_attention_class(got, ref, float(np.nanmax(np.abs(v))), what="decode")
    else:
        cases.assert_close(got, ref, 1e-5, 1e-5, what="f32 decode")


@pytest.mark.parametrize("kv_lens", [[16000], [300, 17, 120, 250], [1200] * 30])
def test_f32_decode_deal_at_head_dim_256(session, kv_lens):
    """The f32 kernel spills there and its steps are long: few rows are dealt out evenly all the same."""
    rng = np.random.default_rng(len(kv_lens))
    dev = Dev(cases.make_paged_batch(rng, kv_lens, [1] * len(kv_lens), bf16=False))
    ws = session.prepare(session.lib.entry(roost_amd.ATTENTION_VARIANT), dev.params(), ("f32 deal", len(kv_lens)))
    words = np.frombuffer(C.string_at(ws.plan, ws.plan_bytes), np.uint64)
    groups = sum(-(-n // 16) for n in kv_lens)
    per_range = -(-groups // (2 * torch().cuda.get_device_properties(0).multi_processor_count))
    assert int(words[5]) >> 32 == 2 and int(words[8]) == -(-groups // per_range)


@pytest.mark.parametrize("kv_lens,hq,hkv,d,by_row", [
    ([1500], 8, 2, 256, True), ([2400, 2500, 2600], 8, 2, 256, True), ([3000] * 10, 8, 2, 256, True),
    ([9000], 32, 8, 128, True), ([512 + 120 * i for i in range(64)], 8, 2, 256, False), ([6960] * 17, 8, 2, 256, False),
    ([15107] * 7, 8, 2, 256, None), ([1025] * 44, 32, 8, 128, None)],
                         ids=lambda k: f"{len(k)}x{max(k)}" if isinstance(k, list) else None)
def test_decode_deal(session, kv_lens, hq, hkv, d, by_row):
    """Few rows are cut row by row, with fewer KV heads per workgroup; calls that fill the chip are dealt out evenly; a long
    stream (200 MB) takes more than one workgroup per CU; and no call leaves a second workgroup on a few CUs only."""
    rng = np.random.default_rng(len(kv_lens))
    b = cases.make_paged_batch(rng, kv_lens, [1] * len(kv_lens), hq=hq, hkv=hkv, d=d)
    dev = Dev(b)
    ws = session.prepare(session.lib.entry(roost_amd.ATTENTION_VARIANT), dev.params(), ("deal", d, len(kv_lens)))
    words = np.frombuffer(C.string_at(ws.plan, ws.plan_bytes), np.uint64)
    heads_per_wg, ranges = int(words[5]) >> 32, int(words[8])
    workgroups = ranges * hkv // heads_per_wg  # 4 query heads per KV head: a wavefront serves one KV head
    cus = torch().cuda.get_device_properties(0).multi_processor_count
    assert not cus < workgroups <= cus * 3 // 2, f"{workgroups} workgroups on {cus} CUs"
    if by_row is not None:
        most = 2 if d == 256 else 4  # the even deal's
        assert (heads_per_wg < most) == by_row, (heads_per_wg, ranges)
    assert sum(kv_lens) * hkv * d * 4 < 200e6 or workgroups > cus, f"{workgroups} workgroups on {cus} CUs"
