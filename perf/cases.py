"""The calls a worker makes of this library, as cases to time and to compare.

A case is one attention call, one set of attention input ops, one GDN layer or one whole worker step, at the shapes of
the benchmark and the tests: paged attention over 16- to 64-token pages with 4 to 16 query heads per KV head, GDN layers
of 16 key heads, batches from one chat to 128 sequences. Lengths come from the case (`lengths` seeds them), values from
the seed given to prepare(). Plans and workspaces are made in prepare(), as a worker keeps them over the layers of a
step; the whole step plans in run(), once, as a worker does for every step.
"""
import ctypes
import math
import random

import numpy as np
import torch

import roost_amd
from roost_amd import abi

GDN_DIM = 128
CONV_WIDTH = 4
EPS = 1e-6
LLAMA3 = (8.0, 1.0, 4.0, 8192)


def _attention(**kw):
    case = {"kind": "attention", "rows": 0, "ctx_lo": 1, "ctx_hi": 1, "chunks": 0, "new_lo": 2, "new_hi": 2, "pre_lo": 0,
            "pre_hi": 0, "q_heads": 8, "kv_heads": 2, "head_dim": 256, "page": 16, "hnd": False, "f32": False,
            "gated": False, "window": -1, "soft_cap": 0.0, "lengths": 1}
    case.update(kw)
    return case


def _inputs(**kw):
    case = {"kind": "inputs", "tokens": 64, "pos_hi": 4096, "q_heads": 8, "kv_heads": 2, "head_dim": 256, "rotary": 64,
            "llama3": False, "page": 16, "fused": False, "lengths": 1}
    case.update(kw)
    return case


def _gdn(**kw):
    case = {"kind": "gdn", "entry": "layer", "rows": 0, "chunks": 0, "new_lo": 2, "new_hi": 2, "k_heads": 16,
            "v_heads": 16, "lengths": 1}
    case.update(kw)
    return case


def listed():
    return [
        # One chat, one token: the smallest attention call there is, bound by latency.
        dict(_attention(rows=1, ctx_lo=1500, ctx_hi=1500), name="decode-one"),
        # A full decode batch at the hybrid model's head shape (the benchmark's headline).
        dict(_attention(rows=64, ctx_lo=512, ctx_hi=8192, lengths=2), name="decode-batch"),
        # Decode of a model with 8 query heads per KV head and head dim 128, over ragged contexts.
        dict(_attention(rows=48, ctx_lo=256, ctx_hi=12000, q_heads=32, kv_heads=4, head_dim=128, lengths=3),
             name="decode-group8"),
        # One user's fresh prompt, an odd length.
        dict(_attention(chunks=1, new_lo=1777, new_hi=1777), name="prefill-prompt"),
        # Chunked prefill: eight ragged chunks on cached prefixes, the attention output gate folded in.
        dict(_attention(chunks=8, new_lo=256, new_hi=2048, pre_hi=6144, gated=True, lengths=3), name="prefill-chunks"),
        # Long fresh prompts of a 32-head model at head dim 128: the largest case.
        dict(_attention(chunks=4, new_lo=3500, new_hi=4096, q_heads=32, kv_heads=8, head_dim=128, lengths=4),
             name="prefill-long-128"),
        # What feeds the attention call in a prefill pass: QkNorm, partial Rope and CacheWrite of 8,192 tokens.
        dict(_inputs(tokens=8192, pos_hi=16384), name="attention-inputs"),
        # One GDN layer of a decode step over a handful of chats: bound by latency and launches.
        dict(_gdn(rows=6), name="gdn-decode-few"),
        # The same over a full batch: bound by the state it reads and writes.
        dict(_gdn(rows=128), name="gdn-decode-batch"),
        # One GDN layer over one user's prompt, through the variant that a worker names for every length.
        dict(_gdn(chunks=1, new_lo=1777, new_hi=1777), name="gdn-prompt"),
        # One GDN layer of a large prefill pass on the chunk variant.
        dict(_gdn(entry="chunk", chunks=4, new_lo=3800, new_hi=4096, lengths=4), name="gdn-prefill"),
        # One whole step of a hybrid layer group: 48 decode rows and 2 prompt chunks through the attention layer (input
        # ops, plan, gated attention) and three GDN layers.
        dict(kind="step", rows=48, ctx_lo=1024, ctx_hi=16384, chunks=2, new_lo=512, new_hi=512, pre_lo=4096, pre_hi=4096,
             lengths=5, name="worker-step"),
    ]


# ---- more cases of the same ranges --------------------------------------------------------------------------------------

HEADS = [(8, 2, 256), (8, 2, 256), (8, 2, 256), (16, 2, 256), (32, 8, 128), (32, 4, 128), (32, 2, 128), (16, 4, 64)]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "mixed", "inputs", "gdn", "gdn", "gdn-chunk", "step"])
    seed = rng.randrange(1, 1 << 20)
    if kind in ("decode", "prefill", "mixed"):
        hq, hkv, d = rng.choice(HEADS)
        c = _attention(q_heads=hq, kv_heads=hkv, head_dim=d, page=rng.choice([16, 16, 32, 64]),
                       hnd=rng.random() < 0.25, gated=rng.random() < 0.3, lengths=seed)
        if rng.random() < 0.12:
            c["window"] = rng.choice([511, 1023, 4095])
        if rng.random() < 0.08:
            c["soft_cap"] = 30.0
        if kind != "prefill":
            c["rows"], c["ctx_hi"] = _log(rng, 1, 128), _log(rng, 64, 16384)
            c["ctx_lo"] = max(1, c["ctx_hi"] // rng.choice([1, 4, 16]))
        if kind != "decode":
            c["chunks"] = rng.randint(1, 8) if kind == "prefill" else rng.randint(1, 3)
            c["new_hi"] = _log(rng, 32, 4096 if kind == "prefill" else 1024)
            c["new_lo"] = max(2, c["new_hi"] // rng.choice([1, 4]))
            c["pre_hi"] = 0 if rng.random() < 0.4 else _log(rng, 64, 8192)
        if kind == "decode" and rng.random() < 0.1:  # f32 is the parity configuration: a few short sequences
            c.update(f32=True, gated=False, head_dim=64, q_heads=8, kv_heads=2, rows=_log(rng, 1, 8),
                     ctx_hi=_log(rng, 32, 1024), ctx_lo=17)
        return c
    if kind == "inputs":
        tokens = _log(rng, 1, 8192)
        if rng.random() < 0.4:
            return _inputs(tokens=tokens, pos_hi=_log(rng, 64, 65536), q_heads=32, kv_heads=8, head_dim=128, rotary=0,
                           llama3=True, page=rng.choice([16, 64]), lengths=seed)
        fused = rng.random() < 0.3
        return _inputs(tokens=tokens, pos_hi=_log(rng, 64, 262144), rotary=0 if fused else 64, fused=fused, lengths=seed)
    if kind == "gdn":
        c = _gdn(v_heads=rng.choice([16, 16, 32]), lengths=seed)
        mix = rng.choice(["rows", "rows", "chunks", "both"])
        if mix != "chunks":
            c["rows"] = _log(rng, 1, 128)
        if mix != "rows":
            c["chunks"] = rng.randint(1, 4)
            c["new_hi"] = _log(rng, 16, 4096)
            c["new_lo"] = max(2, c["new_hi"] // rng.choice([1, 4]))
        return c
    if kind == "gdn-chunk":
        c = _gdn(entry="chunk", chunks=rng.randint(1, 6), new_hi=_log(rng, 64, 4096), v_heads=rng.choice([16, 16, 32]),
                 lengths=seed)
        c["new_lo"] = max(2, c["new_hi"] // rng.choice([1, 4]))
        return c
    hi = _log(rng, 256, 16384)
    return dict(kind="step", rows=_log(rng, 1, 64), ctx_lo=max(1, hi // 16), ctx_hi=hi, chunks=rng.randint(0, 3),
                new_lo=64, new_hi=_log(rng, 64, 1024), pre_lo=0, pre_hi=rng.choice([0, 1024, 4096]), lengths=seed)


def _cost(case):
    """A rough time: what the case must move and multiply, at rates the kernels reach."""
    w = work(case)
    return w["bytes"] / 4e12 + w["flops"] / (8e14 if case["kind"] == "attention" else 2e14)


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        c = _draw(rng)
        if _cost(c) <= most:
            return c


# ---- lengths and algorithmic work ---------------------------------------------------------------------------------------

def _lengths(case):
    """(context, new tokens) per sequence: the one-token rows, then the prompt chunks."""
    rng = random.Random(case["lengths"])
    kv, n = [], []
    for _ in range(case["rows"]):
        kv.append(rng.randint(case["ctx_lo"], case["ctx_hi"]) if "ctx_lo" in case else 1)
        n.append(1)
    for _ in range(case["chunks"]):
        new = rng.randint(case["new_lo"], case["new_hi"])
        kv.append(new + (rng.randint(case["pre_lo"], case["pre_hi"]) if "pre_lo" in case else 0))
        n.append(new)
    return kv, n


def _attention_work(case, kv, n):
    e = 4 if case["f32"] else 2
    hq, hkv, d = case["q_heads"], case["kv_heads"], case["head_dim"]
    seen, pairs = 0, 0
    for c, m in zip(kv, n):
        w = case["window"]
        if w < 0:
            seen += c
            pairs += m * (c - m) + m * (m + 1) // 2
        else:
            seen += min(c, m + w)
            pairs += sum(min(c - m + i + 1, w + 1) for i in range(m))
    nbytes = seen * hkv * d * 2 * e + sum(n) * hq * d * e * (3 if case["gated"] else 2)
    return {"bytes": nbytes, "flops": 4.0 * hq * d * pairs}


def _gdn_work(case, n):
    kh, vh, D = case["k_heads"], case["v_heads"], GDN_DIM
    tokens, ch = sum(n), (2 * case["k_heads"] + case["v_heads"]) * GDN_DIM
    # The projection, its gate columns and the output gate read, the output written; states once each way.
    nbytes = tokens * (ch + 2 * vh + 2 * vh * D) * 2
    nbytes += len(n) * 2 * (vh * D * D * 4 + ch * (CONV_WIDTH - 1) * 2)
    return {"bytes": nbytes, "flops": tokens * (6.0 * vh * D * D + 2.0 * CONV_WIDTH * ch)}


def work(case):
    if case["kind"] == "inputs":
        rows = case["q_heads"] + case["kv_heads"] * 2
        t, d = case["tokens"], case["head_dim"]
        # In place: q and k read and written, v read, k and v written to the cache.
        extra = 0 if case["fused"] else case["kv_heads"]
        return {"bytes": t * (2 * rows + extra) * d * 2 + 12 * t, "flops": 10.0 * t * rows * d}
    kv, n = _lengths(case)
    if case["kind"] == "attention":
        return _attention_work(case, kv, n)
    if case["kind"] == "gdn":
        return _gdn_work(case, n)
    a, i = _step_parts(case)
    parts = [_attention_work(a, kv, n), work(i)] + [_gdn_work(_gdn(), n)] * 3
    return {"bytes": sum(p["bytes"] for p in parts), "flops": sum(p["flops"] for p in parts)}


def _step_parts(case):
    names = ("rows", "ctx_lo", "ctx_hi", "chunks", "new_lo", "new_hi", "pre_lo", "pre_hi", "lengths")
    return (_attention(gated=True, **{k: case[k] for k in names}),
            _inputs(tokens=sum(_lengths(case)[1]), lengths=case["lengths"]))


# ---- inputs on the GPU --------------------------------------------------------------------------------------------------

class _Values:
    """Normal values on the GPU, from one seed."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)
        self.np = np.random.default_rng(seed)

    def f32(self, *shape, std=1.0):
        return torch.randn(shape, generator=self.g, device="cuda") * std

    def bf16(self, *shape, std=1.0):
        return self.f32(*shape, std=std).to(torch.bfloat16)


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _indptr(n):
    return np.concatenate([[0], np.cumsum(n)]).astype(np.int32)


def _paged(case, kv, n, v):
    """A paged batch: random disjoint page lists from a pool 1.25 times what the contexts need."""
    d, hq, hkv, ps = case["head_dim"], case["q_heads"], case["kv_heads"], case["page"]
    pages = [-(-c // ps) for c in kv]
    pool = math.ceil(sum(pages) * 1.25)
    s = {"kv": kv, "n": n, "tokens": sum(n)}
    s["kv_indices_h"] = v.np.permutation(pool)[:sum(pages)].astype(np.int32)
    s["q_indptr_h"], s["kv_indptr_h"] = _indptr(n), _indptr(pages)
    s["last_h"] = np.array([c - (p - 1) * ps for c, p in zip(kv, pages)], np.int32)
    shape = (pool, hkv, ps, d) if case["hnd"] else (pool, ps, hkv, d)
    make = v.f32 if case["f32"] else v.bf16
    s["q"] = make(s["tokens"], hq, d, std=0.5)
    s["k"], s["v"] = make(*shape, std=0.5), make(*shape, std=0.5)
    s["out"] = torch.empty_like(s["q"])
    s["params"] = roost_amd.paged_attention_params(
        s["q"], s["out"], s["k"], s["v"], _dev(s["q_indptr_h"]), _dev(s["kv_indptr_h"]), _dev(s["kv_indices_h"]),
        _dev(s["last_h"]), q_indptr_host=s["q_indptr_h"], kv_indptr_host=s["kv_indptr_h"],
        kv_last_page_len_host=s["last_h"], batch=len(kv), q_heads=hq, kv_heads=hkv, head_dim=d, page_size=ps,
        kv_layout=abi.LAYOUT_PAGED_HND if case["hnd"] else abi.LAYOUT_PAGED_NHD, window_left=case["window"],
        soft_cap=case["soft_cap"])
    if case["gated"]:
        s["gate"] = v.bf16(s["tokens"], hq * d, std=2.0)
        s["gate_params"] = roost_amd.sigmoid_mul_params(s["out"], s["gate"], s["out"], rows=s["tokens"], dim=hq * d)
    return s


def _slots(s, ps):
    """The slot of every new token (the last n positions of each sequence)."""
    out = []
    for i, (c, m) in enumerate(zip(s["kv"], s["n"])):
        pages = s["kv_indices_h"][s["kv_indptr_h"][i]:s["kv_indptr_h"][i + 1]].astype(np.int64)
        pos = np.arange(c - m, c)
        out.append(pages[pos // ps] * ps + pos % ps)
    return np.concatenate(out)


def _input_ops(case, v, positions, slots, k_cache, v_cache, q=None):
    t, hq, hkv, d = case["tokens"], case["q_heads"], case["kv_heads"], case["head_dim"]
    s = {"qw": 1 + v.bf16(d, std=0.1), "kw": 1 + v.bf16(d, std=0.1), "pos": _dev(positions.astype(np.int32)),
         "slots": _dev(slots), "k_cache": k_cache, "v_cache": v_cache,
         "theta": 5e5 if case["llama3"] else 1e7}
    heads = dict(tokens=t, q_heads=hq, kv_heads=hkv, head_dim=d)
    if case["fused"]:
        s["qkv"] = v.bf16(t, (hq + 2 * hkv) * d)
        s["q"] = torch.empty((t, hq, d), dtype=torch.bfloat16, device="cuda")
        s["calls"] = [(roost_amd.QKV_VARIANT, roost_amd.qkv_qk_norm_rope_cache_write_params(
            s["qkv"], s["q"], s["qw"], s["kw"], s["pos"], k_cache, v_cache, s["slots"], page_size=case["page"], eps=EPS,
            theta=s["theta"], **heads))]
        return s
    s["q"] = v.bf16(t, hq, d) if q is None else q
    s["k"], s["v"] = v.bf16(t, hkv, d), v.bf16(t, hkv, d, std=0.5)
    s["calls"] = [
        (roost_amd.QK_NORM_VARIANT, roost_amd.qk_norm_params(s["q"], s["k"], s["qw"], s["kw"], eps=EPS, **heads)),
        (roost_amd.ROPE_VARIANT, roost_amd.rope_params(s["q"], s["k"], s["pos"], theta=s["theta"],
                                                       rotary_dim=case["rotary"],
                                                       llama3=LLAMA3 if case["llama3"] else None, **heads)),
        (roost_amd.CACHE_WRITE_VARIANT, roost_amd.cache_write_params(s["k"], s["v"], k_cache, v_cache, s["slots"],
                                                                     kv_heads=hkv, head_dim=d, page_size=case["page"])),
    ]
    return s


def _gdn_layer(case, n, v, slots, pool, conv_state):
    """One hybrid layer's projections, weights and state slots, and the four ops' params."""
    kh, vh, D, T = case["k_heads"], case["v_heads"], GDN_DIM, sum(n)
    ch = (2 * kh + vh) * D
    s = {"x": v.bf16(T, ch), "w": v.bf16(ch, CONV_WIDTH, std=0.5), "bias": v.bf16(ch, std=0.3),
         "proj": v.bf16(T, 2 * vh, std=2.0), "a_log": v.f32(vh, std=0.5), "dt_bias": v.f32(vh),
         "z": v.bf16(T * vh, D), "nw": 1 + v.f32(D, std=0.2), "slots": _dev(np.asarray(slots, np.int32)),
         "state": pool, "conv_state": conv_state}
    cu_h = _indptr(n)
    cu = _dev(cu_h)
    y = torch.empty((T, ch), dtype=torch.bfloat16, device="cuda")
    o = torch.empty((T, vh, D), dtype=torch.bfloat16, device="cuda")
    s["out"] = torch.empty((T * vh, D), dtype=torch.bfloat16, device="cuda")
    conv = roost_amd.causal_conv1d_params(s["x"], s["w"], s["bias"], y, conv_state, s["slots"], cu, batch=len(n),
                                          tokens=T, channels=ch, width=CONV_WIDTH)
    reach = (T - 1) * 2 * vh + vh
    gates = roost_amd.gated_delta_rule_gates_params(s["proj"], s["proj"], s["a_log"], s["dt_bias"], None, None, tokens=T,
                                                    v_heads=vh, a_stride=2 * vh, b_stride=2 * vh, a_len=reach,
                                                    b_len=reach, a_offset=vh, b_offset=0)
    gdn = roost_amd.gated_delta_rule_params(
        y, y, y, None, None, o, pool, s["slots"], cu, batch=len(n), tokens=T, k_heads=kh, v_heads=vh, q_stride=ch,
        k_stride=ch, v_stride=ch, q_len=(T - 1) * ch + kh * D, k_len=(T - 1) * ch + kh * D,
        v_len=(T - 1) * ch + vh * D, q_offset=0, k_offset=kh * D, v_offset=2 * kh * D, cu_seqlens_host=cu_h)
    norm = roost_amd.gated_rms_norm_params(o, s["z"], s["nw"], s["out"], rows=T * vh, dim=D, eps=EPS)
    s["params"] = (conv, gates, gdn, norm)
    return s


def _gdn_pools(case, slots, v):
    ch = (2 * case["k_heads"] + case["v_heads"]) * GDN_DIM
    return v.f32(slots, case["v_heads"], GDN_DIM, GDN_DIM, std=0.01), v.bf16(slots, ch, CONV_WIDTH - 1)


def _inputs_alone(case, v):
    t, ps = case["tokens"], case["page"]
    pages = -(-t // ps) + 3
    shape = (pages, ps, case["kv_heads"], case["head_dim"])
    caches = [torch.zeros(shape, dtype=torch.bfloat16, device="cuda") for _ in range(2)]
    start = random.Random(case["lengths"]).randint(0, case["pos_hi"])
    return _input_ops(case, v, np.arange(start, start + t), v.np.permutation(pages * ps)[:t].astype(np.int64), *caches)


def _step(case, v):
    kv, n = _lengths(case)
    a, i = _step_parts(case)
    att = _paged(a, kv, n, v)
    pos = np.concatenate([np.arange(c - m, c) for c, m in zip(kv, n)])
    inp = _input_ops(i, v, pos, _slots(att, a["page"]), att["k"], att["v"], q=att["q"])
    g, b = _gdn(), len(n)
    pool, conv_state = _gdn_pools(g, 3 * b, v)
    layers = [_gdn_layer(g, n, v, range(k * b, (k + 1) * b), pool, conv_state) for k in range(3)]
    return {"attention": att, "inputs": inp, "layers": layers, "state": pool, "conv_state": conv_state}


def _build(case, seed):
    v = _Values(seed)
    if case["kind"] == "inputs":
        return _inputs_alone(case, v)
    if case["kind"] == "step":
        return _step(case, v)
    kv, n = _lengths(case)
    if case["kind"] == "attention":
        return _paged(case, kv, n, v)
    slots = v.np.permutation(len(n) + 2)[:len(n)]
    return _gdn_layer(case, n, v, slots, *_gdn_pools(case, len(n) + 2, v))


def prepare(case, seed):
    s = _build(case, seed)
    session = roost_amd.OpSession()
    s["kind"], s["session"] = case["kind"], session
    if case["kind"] == "attention":
        s["entry"] = session.lib.entry(roost_amd.ATTENTION_VARIANT)
        s["ws"] = session.prepare(s["entry"], s["params"], "gated")
    elif case["kind"] == "inputs":
        s["calls"] = [(session.lib.entry(variant), p) for variant, p in s["calls"]]
    elif case["kind"] == "gdn":
        s["chunk"] = case["entry"] == "chunk"
        if s["chunk"]:
            _, gates, gdn, _ = s["params"]
            ws = session.prepare(session.lib.entry(roost_amd.CHUNK_VARIANT), gdn, ("chunk-layer", 0), plan=False)
            status = session.lib.dll.roost_amd_gdn_chunk_layer_plan(
                session.ctx, ctypes.addressof(gates), ctypes.addressof(gdn), ctypes.addressof(ws),
                ctypes.c_void_p(session.stream_handle))
            if status != abi.OK:
                raise RuntimeError(session.lib.last_error())
        else:
            session.prepare(session.lib.entry(roost_amd.RECURRENT_VARIANT), s["params"][2], ("layer", 0))
    else:
        s["inputs"]["calls"] = [(session.lib.entry(variant), p) for variant, p in s["inputs"]["calls"]]
    return s


# ---- one pass -----------------------------------------------------------------------------------------------------------

def _caches(s):
    return {"q": s["q"], "k_cache": s["k_cache"], "v_cache": s["v_cache"]}


def run(s):
    session = s["session"]
    if s["kind"] == "attention":
        if "gate" in s:
            roost_amd.paged_attention_gated(session, s["params"], s["gate_params"], plan=False)
        else:
            session.run(s["entry"], s["params"], s["ws"])
        return {"out": s["out"]}
    if s["kind"] == "inputs":
        for entry, p in s["calls"]:
            session.run(entry, p, None)
        return _caches(s)
    if s["kind"] == "gdn":
        (roost_amd.gdn_chunk_layer if s["chunk"] else roost_amd.gdn_layer)(
            session, *s["params"], **({"plan": False} if s["chunk"] else {}))
        return {"out": s["out"], "state": s["state"], "conv_state": s["conv_state"]}
    for entry, p in s["inputs"]["calls"]:
        session.run(entry, p, None)
    roost_amd.paged_attention_gated(session, s["attention"]["params"], s["attention"]["gate_params"])
    for k, layer in enumerate(s["layers"]):
        roost_amd.gdn_layer(session, *layer["params"], key=k)
    return {"attention": s["attention"]["out"], "layers": [x["out"] for x in s["layers"]], "state": s["state"],
            "conv_state": s["conv_state"], **_caches(s["inputs"])}


# ---- tolerances and 64-bit results --------------------------------------------------------------------------------------

def tolerance(case):
    if case["kind"] == "attention" and case["f32"]:
        return {"rel": 1e-5}
    if case["kind"] == "inputs":  # every op rounds its results once: two implementations differ by a step on few values
        return {"rel": 5e-4, "max": 0.02}
    # bf16 results with fp32 sums: one rounding of each output (2e-3 in the 2-norm), another at each op's boundary.
    return {"rel": 1e-2, "max": 0.1}


def _round(x):
    """The bf16 value that an op of the chain hands to the next."""
    return x.to(torch.bfloat16).double()


def _exact_attention(case, s, q, k_cache, v_cache):
    hq, hkv, d, ps = case["q_heads"], case["kv_heads"], case["head_dim"], case["page"]
    group = hq // hkv
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    for i, (c, m) in enumerate(zip(s["kv"], s["n"])):
        pages = _dev(s["kv_indices_h"][s["kv_indptr_h"][i]:s["kv_indptr_h"][i + 1]]).long()
        t0 = int(s["q_indptr_h"][i])
        qpos = torch.arange(c - m, c, device="cuda")[:, None]
        kpos = torch.arange(c, device="cuda")[None, :]
        hidden = kpos > qpos
        if case["window"] >= 0:
            hidden = hidden | (kpos < qpos - case["window"])
        for h in range(hkv):
            if case["hnd"]:
                k, v = k_cache[pages, h], v_cache[pages, h]
            else:
                k, v = k_cache[pages][:, :, h], v_cache[pages][:, :, h]
            k, v = k.reshape(-1, d)[:c].double(), v.reshape(-1, d)[:c].double()
            for head in range(h * group, (h + 1) * group):
                x = q[t0:t0 + m, head].double() @ k.t() / math.sqrt(d)
                if case["soft_cap"]:
                    x = case["soft_cap"] * torch.tanh(x / case["soft_cap"])
                x = torch.softmax(x.masked_fill(hidden, -math.inf), dim=1)
                out[t0:t0 + m, head] = x @ v
    if case["gated"]:
        out = _round(out) * torch.sigmoid(s["gate"].double()).reshape(out.shape)
    return out


def _exact_inputs(case, s):
    """(q, k_cache, v_cache) after QkNorm, Rope and CacheWrite, each op's results rounded as it stores them."""
    t, hq, hkv, d = case["tokens"], case["q_heads"], case["kv_heads"], case["head_dim"]
    if case["fused"]:
        q, k, v = s["qkv"].double().reshape(t, hq + 2 * hkv, d).split([hq, hkv, hkv], dim=1)
    else:
        q, k, v = s["q"].double(), s["k"].double(), s["v"].double()
    rot = case["rotary"] or d
    half = rot // 2
    freq = s["theta"] ** (-2.0 * torch.arange(half, dtype=torch.float64, device="cuda") / rot)
    if case["llama3"]:
        factor, low, high, orig = LLAMA3
        wave = 2 * math.pi / freq
        smooth = (orig / wave - low) / (high - low)
        mixed = (1 - smooth) * freq / factor + smooth * freq
        freq = torch.where(wave < orig / high, freq, torch.where(wave > orig / low, freq / factor, mixed))
    angle = s["pos"].double()[:, None] * freq
    cos, sin = angle.cos()[:, None, :], angle.sin()[:, None, :]

    def one(x, w):
        x = _round(x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double())
        a, b = x[..., :half], x[..., half:rot]
        return _round(torch.cat([a * cos - b * sin, b * cos + a * sin, x[..., rot:]], dim=-1))

    q, k = one(q, s["qw"]), one(k, s["kw"])
    caches = []
    for cache, rows in ((s["k_cache"], k), (s["v_cache"], v)):
        c = cache.double().reshape(-1, hkv, d)
        c[s["slots"]] = rows
        caches.append(c.reshape(cache.shape))
    return q, caches[0], caches[1]


def _exact_gdn(case, n, s, state, conv_state):
    """The layer's output; its slots of `state` and `conv_state` (both in 64 bits) are updated in place. The values that
    the ops hand on in bf16 (convolution, beta, GDN output) are rounded there."""
    kh, vh, D = case["k_heads"], case["v_heads"], GDN_DIM
    slots, cu = s["slots"].long(), _indptr(n)
    x, w, bias = s["x"].double(), s["w"].double(), s["bias"].double()
    y = torch.empty_like(x)
    for i, m in enumerate(n):
        t0 = int(cu[i])
        ext = torch.cat([conv_state[slots[i]].t(), x[t0:t0 + m]])
        z = sum(ext[j:j + m] * w[:, j] for j in range(CONV_WIDTH)) + bias
        y[t0:t0 + m] = z * torch.sigmoid(z)
        conv_state[slots[i]] = ext[m:].t()
    y = _round(y)
    q, k, v = y.split([kh * D, kh * D, vh * D], dim=1)
    unit = lambda r: r * torch.rsqrt((r * r).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
    q = unit(q.reshape(-1, kh, D)).repeat_interleave(vh // kh, dim=1) / math.sqrt(D)
    k = unit(k.reshape(-1, kh, D)).repeat_interleave(vh // kh, dim=1)
    v = v.reshape(-1, vh, D)
    b, a = s["proj"].double().split(vh, dim=1)
    beta = _round(torch.sigmoid(b))
    decay = torch.exp(-torch.exp(s["a_log"].double()) * torch.nn.functional.softplus(a + s["dt_bias"].double()))
    o = torch.empty_like(v)
    S = state[slots]
    starts, lens = torch.tensor(cu[:-1].astype(np.int64), device="cuda"), np.asarray(n)
    for t in range(max(n)):
        live = torch.from_numpy(np.flatnonzero(lens > t)).cuda() if (lens <= t).any() else slice(None)
        at = starts[live] + t
        Sl = S[live] * decay[at][:, :, None, None]
        kt = k[at]
        d = beta[at][:, :, None] * (v[at] - (kt[:, :, None] @ Sl)[:, :, 0])
        Sl = Sl + kt[..., None] * d[:, :, None]
        o[at] = (q[at][:, :, None] @ Sl)[:, :, 0]
        S[live] = Sl
    state[slots] = S
    o = _round(o).reshape(-1, D)
    z = s["z"].double()
    return o * torch.rsqrt((o * o).mean(-1, keepdim=True) + EPS) * s["nw"].double() * (z * torch.sigmoid(z))


def exact(case, seed):
    s = _build(case, seed)
    if case["kind"] == "attention":
        return {"out": _exact_attention(case, s, s["q"], s["k"], s["v"])}
    if case["kind"] == "inputs":
        return dict(zip(("q", "k_cache", "v_cache"), _exact_inputs(case, s)))
    n = _lengths(case)[1]
    state, conv_state = s["state"].double(), s["conv_state"].double()
    if case["kind"] == "gdn":
        return {"out": _exact_gdn(case, n, s, state, conv_state), "state": state, "conv_state": conv_state}
    a, i = _step_parts(case)
    q, k_cache, v_cache = _exact_inputs(i, s["inputs"])
    return {"attention": _exact_attention(a, s["attention"], q, k_cache, v_cache),
            "layers": [_exact_gdn(_gdn(), n, x, state, conv_state) for x in s["layers"]], "state": state,
            "conv_state": conv_state, "q": q, "k_cache": k_cache, "v_cache": v_cache}
