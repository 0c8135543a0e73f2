"""The prefill plan's two late choices against float32 torch: the 12-wavefront, 96-token items of head dim 128 (item edges
around 32, 64 and 96 tokens, split and whole items, prefixes, both layouts), and short prompts cut into pieces of 2 to 7 tiles
while CUs are idle (piece edges, several pieces per item, every head dim)."""
import ctypes as C
import dataclasses

import numpy as np
import pytest

import cases
import roost_amd
from test_attention_gpu import Dev, from_dev, to_dev, torch, torch_reference

pytestmark = pytest.mark.gpu


def _words(session, key):
    ws = session._ws[(session.lib.entry(roost_amd.ATTENTION_VARIANT).variant_id, key)][3]
    return np.frombuffer(C.string_at(ws.plan, ws.plan_bytes), np.uint64)


def _run(session, b, key, **kw):
    """The result and, from the plan record: work items, merges, and its last word, the query tokens per item."""
    dev = Dev(b, **kw)
    entry = session.lib.entry(roost_amd.ATTENTION_VARIANT)
    session.launch(entry, dev.params(), key=key)
    words = _words(session, key)
    got = dev.result()
    assert not np.isnan(got).any()
    return got, int(words[7]), int(words[9]), int(words[-1])


@pytest.mark.parametrize("hq,hkv", [(32, 8), (64, 4)])
@pytest.mark.parametrize("new,pre", [([1791, 1889, 1984, 2000, 33, 2], [0, 5, 1000, 64, 0, 7]),
                                           ([4001, 97, 4096, 96, 3999, 95], [0, 0, 0, 31, 17, 900])])
@pytest.mark.parametrize("hnd,ps", [(False, 16), (True, 64)])
def test_wide_items(session, hq, hkv, new, pre, hnd, ps):
    rng = np.random.default_rng(sum(new) + hq)
    b = cases.make_paged_batch(rng, [a + p for a, p in zip(new, pre)], new, page_size=ps, hnd=hnd, hq=hq, hkv=hkv, d=128,
                               std=0.5)
    got, _, _, tokens = _run(session, b, ("wide", hq, sum(new), hnd))
    assert tokens == 96, "the plan did not take the wide items"
    if hnd:  # the reference reads NHD pools
        b = dataclasses.replace(b, k_cache=b.k_cache.transpose(0, 2, 1, 3), v_cache=b.v_cache.transpose(0, 2, 1, 3))
    cases.assert_close(got, torch_reference(b), what="wide prefill vs fp32 torch")


def _torch_options(b, causal, window, cap):
    """torch_reference with a window and a soft cap, and the base-2 log-sum-exp beside it."""
    t = torch()
    q, k, v = (t.from_numpy(cases.values(x, True).astype(np.float32)).cuda() for x in (b.q, b.k_cache, b.v_cache))
    out, lse = t.zeros(q.shape, device="cuda"), t.zeros(q.shape[:2], device="cuda")
    for s in range(b.batch):
        pages = t.from_numpy(b.kv_indices[b.kv_indptr[s]:b.kv_indptr[s + 1]].astype(np.int64)).cuda()
        n, rows = int(b.kv_lens[s]), slice(int(b.q_indptr[s]), int(b.q_indptr[s + 1]))
        ks, vs = (c[pages].reshape(-1, b.hkv, b.d)[:n] for c in (k, v))
        pos = t.arange(n - (rows.stop - rows.start), n, device="cuda")[:, None]
        key = t.arange(n, device="cuda")[None, :]
        hidden = (key > pos) & causal | (key < pos - window) & (window >= 0)
        for h in range(b.hq):
            sc = q[rows, h] @ ks[:, h // (b.hq // b.hkv)].T / float(np.sqrt(b.d))
            if cap:
                sc = cap * t.tanh(sc / cap)
            sc = sc.masked_fill(hidden, float("-inf"))
            out[rows, h] = t.softmax(sc, -1) @ vs[:, h // (b.hq // b.hkv)]
            lse[rows, h] = t.logsumexp(sc, -1) / float(np.log(2.0))
    return out.cpu().numpy(), lse.cpu().numpy()


@pytest.mark.parametrize("causal,window,cap", [(True, -1, 0.0), (True, 3000, 0.0), (False, -1, 0.0), (True, -1, 3.0)],
                         ids=["causal", "window", "not causal", "soft cap"])
def test_wide_items_options(session, causal, window, cap):
    """The 96-token items with every option, lse and the output gate on, whole items and (a chunk on 20,000 keys) merged
    ones. The lse bar is that of the other prefill kernels."""
    rng = np.random.default_rng(7)
    new, pre = [3901, 3800, 3700, 3600, 300], [0, 0, 64, 5, 20000]
    b = cases.make_paged_batch(rng, [a + p for a, p in zip(new, pre)], new, hq=32, hkv=8, d=128, std=1.0)
    dev = Dev(b, causal, with_lse=True, window_left=window, soft_cap=cap)
    key, params = ("wide options", causal, window, cap), dev.params()
    session.launch(session.lib.entry(roost_amd.ATTENTION_VARIANT), params, key=key)
    words = _words(session, key)
    assert int(words[-1]) == 96 and (int(words[9]) > 0 or window >= 0 or not causal), "no wide items, or none merged"
    out, lse = _torch_options(b, causal, window, cap)
    cases.assert_close(dev.result(), out, what="wide prefill vs fp32 torch")
    assert np.abs(from_dev(dev.lse) - lse).max() < 2e-3
    plain, gate = dev.out.clone(), to_dev(cases.bf16_bits(rng.standard_normal(b.q.shape).astype(np.float32)), True)
    roost_amd.sigmoid_mul(session, plain, gate, plain, rows=b.tokens, dim=b.hq * b.d)
    dev.out.fill_(float("nan"))
    sm = roost_amd.sigmoid_mul_params(dev.out, gate, dev.out, rows=b.tokens, dim=b.hq * b.d)
    roost_amd.paged_attention_gated(session, params, sm, key=key)
    assert np.array_equal(from_dev(dev.out, True), from_dev(plain, True)), "gated differs from attention then SigmoidMul"


@pytest.mark.parametrize("hq,hkv,new,pre,window", [(16, 4, [993, 1263], [987, 2501], 511),
                                                   (8, 2, [2490, 2096, 2803, 1375, 886], [10, 157, 146, 244, 62], -1)])
def test_wide_form_pays_for_the_pieces_it_cuts(session, hq, hkv, new, pre, window):
    """Calls whose 96-token items would be cut into more pieces than the 64-token ones, and lose more in partial rows than
    their tiles gain, take the latter."""
    rng = np.random.default_rng(sum(new))
    b = cases.make_paged_batch(rng, [a + p for a, p in zip(new, pre)], new, hq=hq, hkv=hkv, d=128, std=0.5)
    got, _, _, tokens = _run(session, b, ("narrow", sum(new)), window_left=window)
    assert tokens == 64
    cases.assert_close(got, _torch_options(b, True, window, 0.0)[0], what="prefill vs fp32 torch")


@pytest.mark.parametrize("hq,hkv,d", [(8, 2, 256), (8, 2, 128), (4, 1, 64)])
@pytest.mark.parametrize("new,pre", [([500], [0]), ([1025], [0]), ([1777], [0]), ([256], [4001]), ([64], [8000]),
                                     ([129, 2, 1, 300], [0, 640, 900, 33])])
def test_short_prompts_in_small_pieces(session, hq, hkv, d, new, pre):
    rng = np.random.default_rng(sum(new) + d)
    b = cases.make_paged_batch(rng, [a + p for a, p in zip(new, pre)], new, hq=hq, hkv=hkv, d=d, std=0.5)
    got, items, merges, tokens = _run(session, b, ("sparse", d, sum(new)))
    # Items that pieces of at least 8 tiles would leave are fewer; every one of these calls is cut further.
    tiles = [-(-(p + min(q + 64, a)) // 64) for a, p in zip(new, pre) if a > 1 for q in range(0, a, 64)]
    coarse = hkv * sum(-(-x // 8) for x in tiles)
    assert tokens == 64 and merges > 0 and coarse < items <= 256, (items, coarse, merges)
    cases.assert_close(got, torch_reference(b), what="short prompt vs fp32 torch")


def _near_ties(b, rng):
    """Queries of zeros, so that a row is the plain mean of the V rows it sees, and V one of two neighbouring bf16 values,
    1 and 1 + 2^-7, with another share of each in every dim. The means, in units of 2^-7 above 1."""
    share = rng.uniform(0.3, 0.7, (b.hkv, b.d))
    upper = rng.random(b.v_cache.shape) < share
    pages = [b.kv_indices[b.kv_indptr[s]:b.kv_indptr[s + 1]] for s in range(b.batch)]
    rows = [upper[p].reshape(-1, b.hkv, b.d)[:n] for p, n in zip(pages, b.kv_lens)]
    means = [np.cumsum(r, 0)[n - m:] / np.arange(n - m + 1, n + 1)[:, None, None]
             for r, n, m in zip(rows, b.kv_lens, b.q_lens)]
    b = dataclasses.replace(b, q=np.zeros_like(b.q), v_cache=np.where(upper, 0x3F81, 0x3F80).astype(np.uint16))
    return b, np.repeat(np.concatenate(means), b.hq // b.hkv, axis=1)


def _check_single_rounding(got, mean, rows):
    """The weights are exactly 1 and every sum is exact in fp32, so a row rounded once is the mean's neighbour, but for the
    last place of the division and of the merge (2^-18 of a unit here); a piece's mean rounded to bf16 first would land on
    the other neighbour in a few dims of a hundred."""
    sure = rows[:, None, None] & (np.abs(mean - 0.5) > 1e-3)
    want = 1.0 + np.where(mean > 0.5, 2.0 ** -7, 0.0)
    wrong = sure & (got != want)
    assert sure.mean() > 0.1 and not wrong.any(), f"{wrong.sum()} of {sure.sum()} elements were rounded more than once"


@pytest.mark.parametrize("hq,hkv,d", [(8, 2, 256), (8, 2, 128), (4, 1, 64)])
@pytest.mark.parametrize("new,pre", [([500], [0]), ([1025], [0]), ([129, 450, 300], [40, 0, 33])])
def test_items_cut_for_idle_cus_keep_fp32(session, hq, hkv, d, new, pre):
    """A prompt cut into small pieces because CUs would idle is as precise as a whole one."""
    rng = np.random.default_rng(sum(new) + d)
    b, mean = _near_ties(cases.make_paged_batch(rng, [a + p for a, p in zip(new, pre)], new, hq=hq, hkv=hkv, d=d), rng)
    got, _, merges, _ = _run(session, b, ("ties", d, sum(new)))
    assert merges > 0
    pos = np.concatenate([p + np.arange(a) for a, p in zip(new, pre)])
    _check_single_rounding(got, mean, pos < 512 - 64)  # items of up to 8 tiles


@pytest.mark.parametrize("hq,hkv,d,rows,kv,new,pre", [
    (16, 2, 256, 16, 5300, 535, 143), (32, 2, 128, 81, 5800, 117, 5350), (32, 2, 256, 7, 5800, 200, 264),
    (16, 1, 64, 64, 3000, 300, 700)], ids=["g8 d256", "g16 d128", "g16 d256", "g16 d64"])
def test_items_cut_beside_decode_ranges_keep_fp32(session, hq, hkv, d, rows, kv, new, pre):
    """Groups of 8 and more query heads: decode ranges that take a good part of a mixed step's one launch leave a prompt's
    items as precise as whole ones."""
    rng = np.random.default_rng(hq + d)
    lens = [kv - 37 * i % 1000 for i in range(rows)] + [new + pre]
    b, mean = _near_ties(cases.make_paged_batch(rng, lens, [1] * rows + [new], hq=hq, hkv=hkv, d=d), rng)
    key = ("mixed ties", d, hq)
    got, _, merges, _ = _run(session, b, key)
    assert int(_words(session, key)[5]) & 0xFFFFFFFF == 1 and merges > 0, "the plan did not cut the items of one launch"
    _check_single_rounding(got, mean, np.ones(rows + new, bool))


@pytest.mark.parametrize("hq,hkv,d,rows,kv,new,pre", [(32, 2, 256, 2, 9577, [190], 1769), (16, 2, 256, 24, 4350, [512], 4088),
                                                      (32, 2, 256, 89, 190, [123] * 3, 1100)])
def test_mixed_step_leaves_the_decode_ranges_enough_cus(session, hq, hkv, d, rows, kv, new, pre):
    """Groups of 8 and more query heads: a range's CU streams about 28 KB a microsecond, so with the pieces on most CUs the
    few that are left would take longer than both parts one after the other."""
    rng = np.random.default_rng(hq + rows)
    b = cases.make_paged_batch(rng, [kv] * rows + [n + pre for n in new], [1] * rows + new, hq=hq, hkv=hkv, d=d, std=0.5)
    key = ("mixed cus", hq, rows)
    got, items, _, _ = _run(session, b, key)
    cases.assert_close(got, torch_reference(b), what="mixed step vs fp32 torch")
    if int(_words(session, key)[5]) & 0xFFFFFFFF:
        tile_us, k_us = 3.7, rows * kv * (hq // min(hq // hkv, 16)) * d * 4 / 28e3
        longest = -(-(max(new) + pre) // 64)
        assert k_us / (256 - items) < k_us / 200 + longest * tile_us, f"{items} of 256 CUs hold pieces"
