"""The work that programs have this library do, as cases to time and to check.

Seven kinds, each through entry points that a program calls:

  model      one pass: the ubatch is planned (DeviceModel.plan) and run
             (DeviceModel.forward), as a serving loop does each step; logits
  product    lgmlh_mul_mat / lgmlh_mul_mat_ggml on repacked weights
  ffn        a layer's feed-forward: rms_norm, [gate | up], the gated unit,
             down with the residual
  moe        a layer's routed experts: rms_norm, router, routing, the grouped
             products, the weighted sum with the residual
  head       the output end of a pass: rms_norm, output product, greedy ids
  attention  lgmlh_paged_attention over a planned pass (the pool, or the
             sequences' rings with a window)
  flash      lgmlh_flash_attn on strided K / V rows with an explicit mask

Sizes are those of the repository's configurations (lgml_amd/workload.py: an
8B shape "c2", a Gemma-4-style shape "c4", a 30B-A3B MoE shape "c5"; the tiny
f32 model of the tests) and generic ones around them. Weights are N(0, 0.02)
in the ggml block layouts (lgmlh_gen_normal), activations N(0, 1), the KV
cells N(0, 1) in f16.
"""
import ctypes as C
import math
import random

import numpy as np
import torch

from lgml_amd import hip, runtime, workload

F32, Q8_0, Q4_K, Q6_K = hip.F32, hip.Q8_0, hip.Q4_K, hip.Q6_K
TYPES = {"f32": F32, "q8_0": Q8_0, "q4_K": Q4_K, "q6_K": Q6_K}
BITS = {"f32": 32.0, "q8_0": 8.5, "q4_K": 4.5, "q6_K": 6.5625}
DEV = "cuda"


# ---- the cases ----------------------------------------------------------------
def listed():
    return [
        # the smallest pass: the tiny f32 model, one decode step of 4 slots at
        # the contexts its prompts leave; launches and host work count
        dict(name="tiny decode pass", kind="model", shape="tiny", wtype="f32", layers=2, slots=4,
             lo=17, hi=300, chunk=0),
        # one decode step of 64 ragged slots through two layers and the head
        # of the 8B shape, the serving loop's ordinary pass
        dict(name="8B decode pass", kind="model", shape="c2", wtype="q4_K_M", layers=2, slots=64,
             lo=128, hi=4096, chunk=0),
        # the feed-forward of a decode step: two products of 64 rows
        dict(name="8B ffn decode", kind="ffn", rows=64, embd=4096, ff=14336, wtype="q4_K",
             act="ggml", gelu=False),
        # the Gemma-4-style shape's feed-forward on one 512-token prompt chunk
        dict(name="gemma ffn prefill", kind="ffn", rows=512, embd=2560, ff=10240, wtype="q8_0",
             act="ggml", gelu=True),
        # a small product of few and odd rows in f32-accurate arithmetic (a
        # V matrix, a handful of slots)
        dict(name="small product", kind="product", wtype="q6_K", act="exact", m=1024, k=4096,
             n=13, x="f32", residual=False),
        # the largest product of a mixed pass: a 512-token chunk beside 63
        # decode tokens
        dict(name="8B gate|up prefill", kind="product", wtype="q4_K", act="ggml", m=28672, k=4096,
             n=575, x="f32", residual=False),
        # the end of a decode step: logits of 64 rows and their greedy ids
        dict(name="8B head", kind="head", rows=64, embd=4096, vocab=128256, wtype="q6_K",
             act="ggml"),
        # decode attention of 64 ragged sequences, one layer
        dict(name="8B attention decode", kind="attention", heads=32, kv=8, dim=128, slots=64,
             lo=128, hi=4096, chunk=0, past=0, window=0),
        # attention of a mixed pass of the MoE shape: a 512-token chunk of a
        # long prompt beside 32 decoding sequences
        dict(name="MoE attention chunk", kind="attention", heads=32, kv=4, dim=128, slots=32,
             lo=256, hi=8192, chunk=512, past=3584, window=0),
        # routed experts of a decode step of 64 slots
        dict(name="MoE layer decode", kind="moe", rows=64, embd=2048, ff=768, experts=128, used=8,
             wtype="q4_K", act="ggml"),
        # routed experts of a prompt chunk
        dict(name="MoE layer prefill", kind="moe", rows=512, embd=2048, ff=768, experts=128,
             used=8, wtype="q4_K", act="ggml"),
        # attention outside the pool: a 512-token chunk of a lone sequence
        # over its contiguous cache under a causal mask
        dict(name="flash chunk", kind="flash", heads=32, kv=8, dim=128, rows=512, cells=2048,
             mask="causal", softcap=0.0, max_bias=0.0),
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _mult(rng, lo, hi, m):
    return m * _log(rng, lo // m, hi // m)


def draw(rng):
    """A case of the ranges above: every kind, from one row to a mixed pass
    of two prompt chunks, odd row counts among them."""
    kind = rng.choice(["product"] * 3 + ["attention"] * 2 + ["ffn", "moe", "flash", "model", "head"])
    act = rng.choice(["ggml", "ggml", "exact"])
    if kind == "product":
        ty = rng.choice(["q4_K", "q4_K", "q6_K", "q8_0", "f32"])
        res = rng.random() < 0.3
        if ty == "f32":  # routers, tiny models: any size
            m, k, n = _log(rng, 16, 2048), 8 * _log(rng, 8, 512), _log(rng, 1, 576)
            return dict(kind=kind, wtype=ty, act="exact", m=m, k=k, n=n, x="f32", residual=res)
        while True:
            m, k = _mult(rng, 256, 28672, 16), _mult(rng, 256, 14336, 256)
            n = _log(rng, 1, 1088)
            if m * k * n <= 28672 * 4096 * 512:
                return dict(kind=kind, wtype=ty, act=act, m=m, k=k, n=n,
                            x=rng.choice(["f32", "f32", "f16"]), residual=res)
    if kind == "attention":
        d = rng.choice([64, 128, 128, 256])
        kv, g = rng.choice([1, 2, 4, 8]), rng.choice([1, 2, 4, 8])
        window = 1024 if d == 256 and rng.random() < 0.5 else 0
        chunk = rng.choice([0, 0, _log(rng, 2, 512)])
        return dict(kind=kind, heads=kv * g, kv=kv, dim=d, slots=_log(rng, 1, 64),
                    lo=_log(rng, 1, 512), hi=_log(rng, 513, 4096), chunk=chunk,
                    past=_log(rng, 1, 4096) if chunk else 0, window=window)
    if kind == "ffn":
        while True:
            e, f, n = _mult(rng, 256, 4096, 256), _mult(rng, 256, 14336, 256), _log(rng, 1, 576)
            if 3 * e * f * n <= 28672 * 4096 * 512:
                return dict(kind=kind, rows=n, embd=e, ff=f, act=act,
                            wtype=rng.choice(["q4_K", "q6_K", "q8_0"]), gelu=rng.random() < 0.3)
    if kind == "moe":
        return dict(kind=kind, rows=_log(rng, 1, 512), embd=_mult(rng, 512, 2048, 256),
                    ff=_mult(rng, 256, 768, 256), experts=rng.choice([8, 32, 64, 128]),
                    used=rng.choice([2, 4, 8]), wtype=rng.choice(["q4_K", "q4_K", "q8_0"]), act=act)
    if kind == "flash":
        kv, g = rng.choice([1, 2, 4, 8]), rng.choice([1, 2, 4])
        n = _log(rng, 1, 512)
        return dict(kind=kind, heads=kv * g, kv=kv, dim=8 * rng.choice([2, 4, 8, 10, 12, 16, 16, 32]),
                    rows=n, cells=n + _log(rng, 1, 2048),
                    mask=rng.choice(["causal", "causal", "window", "none"]),
                    softcap=rng.choice([0.0, 0.0, 0.0, 30.0]), max_bias=0.0)
    if kind == "model":
        chunk = rng.choice([0, _log(rng, 2, 300)])
        return dict(kind=kind, shape="tiny", wtype=rng.choice(["f32", "f32", "q8_0"]),
                    layers=rng.randint(1, 4), slots=_log(rng, 1, 16), lo=_log(rng, 1, 64),
                    hi=_log(rng, 65, 600), chunk=chunk)
    return dict(kind="head", rows=_log(rng, 1, 64), embd=_mult(rng, 512, 4096, 256),
                vocab=_log(rng, 8192, 128256), wtype=rng.choice(["q4_K", "q6_K", "q8_0"]), act=act)


# ---- inputs -------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(DEV).manual_seed(seed)


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32)


def _raw(seed, wtype, rows, cols, sd=0.02):
    """N(0, sd) weights (rows, cols) in the ggml layout of wtype (uint8; f32
    as it is)."""
    ty = TYPES[wtype]
    if ty == F32:
        return _normal(_gen(seed), rows, cols) * sd
    L = hip.lib()
    t = torch.empty(L.lgmlh_row_size(ty, cols) * rows, dtype=torch.uint8, device=DEV)
    hip.check(L.lgmlh_gen_normal(seed, ty, rows, cols, 0.0, sd, t.data_ptr(), hip.stream()))
    return t


def _repacked(seed, wtype, rows, cols):
    raw = _raw(seed, wtype, rows, cols)
    if wtype == "f32":
        return raw
    L, ty = hip.lib(), TYPES[wtype]
    out = torch.empty(L.lgmlh_repacked_bytes(ty, rows, cols), dtype=torch.uint8, device=DEV)
    hip.check(L.lgmlh_repack(ty, rows, cols, raw.data_ptr(), out.data_ptr(), hip.stream()))
    torch.cuda.current_stream().synchronize()
    return out


def _bytes(n):
    return torch.empty(max(int(n), 1), dtype=torch.uint8, device=DEV)


def _out(*shape):
    return torch.empty(*shape, dtype=torch.float32, device=DEV)


def _lengths(c, seed):
    """The contexts of a pass's decoding sequences, uniform in [lo, hi] (both
    ends among them), and for a chunk one sequence more."""
    rng = random.Random(seed * 7919 + 5)
    ctx = [rng.randint(c["lo"], c["hi"]) for _ in range(c["slots"])]
    ctx[0], ctx[-1] = c["lo"], c["hi"]
    return ctx


def _tables(seq_n, past, seed, extra=0):
    """Block tables over a shuffled pool: (table, pool blocks)."""
    need = [(p + n + 63) // 64 for p, n in zip(past, seq_n)]
    order = np.random.default_rng(seed + 11).permutation(sum(need) + extra).astype(np.int32)
    tab, at = np.zeros((len(need), max(need)), np.int32), 0
    for s, n in enumerate(need):
        tab[s, :n] = order[at:at + n]
        at += n
    return tab, sum(need) + extra


def _prep_product(c, seed):
    g, L, ty = _gen(seed + 1), hip.lib(), TYPES[c["wtype"]]
    x = _normal(g, c["n"], c["k"])
    x = x.half() if c["x"] == "f16" else x
    ws = _bytes(L.lgmlh_mul_mat_workspace(ty, c["m"], c["k"], c["n"]))
    return dict(c=c, w=_repacked(seed, c["wtype"], c["m"], c["k"]), x=x, y=_out(c["n"], c["m"]),
                res=_normal(g, c["n"], c["m"]) if c["residual"] else None, ws=ws)


def _product(act, ty, w, m, k, x, n, y, res, ws):
    L = hip.lib()
    fn = L.lgmlh_mul_mat_ggml if act == "ggml" else L.lgmlh_mul_mat
    hip.check(fn(ty, w.data_ptr(), m, k, x.data_ptr(),
                 hip.F16 if x.dtype == torch.float16 else F32, n, y.data_ptr(),
                 hip.EPI_ADD if res is not None else hip.EPI_NONE, hip.ptr(res), ws.data_ptr(),
                 ws.numel(), hip.stream()))


def _run_product(s):
    c = s["c"]
    _product(c["act"], TYPES[c["wtype"]], s["w"], c["m"], c["k"], s["x"], c["n"], s["y"], s["res"],
             s["ws"])
    return s["y"]


def _prep_ffn(c, seed):
    g, L, ty, n, e, f = _gen(seed + 1), hip.lib(), TYPES[c["wtype"]], c["rows"], c["embd"], c["ff"]
    ws = max(L.lgmlh_mul_mat_workspace(ty, 2 * f, e, n), L.lgmlh_mul_mat_workspace(ty, e, f, n))
    return dict(c=c, x=_normal(g, n, e), norm=1 + 0.1 * _normal(g, e), xn=_out(n, e),
                gu=_out(n, 2 * f), h=_out(n, f), y=_out(n, e), ws=_bytes(ws),
                wgu=_repacked(seed, c["wtype"], 2 * f, e), wdown=_repacked(seed + 7, c["wtype"], e, f))


def _run_ffn(s):
    c, L, st = s["c"], hip.lib(), hip.stream()
    n, e, f, ty = c["rows"], c["embd"], c["ff"], TYPES[c["wtype"]]
    hip.check(L.lgmlh_rms_norm(s["x"].data_ptr(), n, e, 1e-5, s["norm"].data_ptr(),
                               s["xn"].data_ptr(), F32, st))
    _product(c["act"], ty, s["wgu"], 2 * f, e, s["xn"], n, s["gu"], None, s["ws"])
    unit = L.lgmlh_geglu if c["gelu"] else L.lgmlh_swiglu
    hip.check(unit(s["gu"].data_ptr(), n, f, s["h"].data_ptr(), F32, st))
    _product(c["act"], ty, s["wdown"], e, f, s["h"], n, s["y"], s["x"], s["ws"])
    return {"h": s["h"], "y": s["y"]}


def _prep_moe(c, seed):
    g, L, ty = _gen(seed + 1), hip.lib(), TYPES[c["wtype"]]
    t, e, f, ne, nu = c["rows"], c["embd"], c["ff"], c["experts"], c["used"]
    gate, up = _raw(seed, c["wtype"], ne * f, e), _raw(seed + 3, c["wtype"], ne * f, e)
    wgu, _ = runtime.repack_experts((gate, ty, ne * f), (up, ty, ne * f), ne, e)
    wdown, _ = runtime.repack_experts((_raw(seed + 7, c["wtype"], ne * e, f), ty, ne * e), None, ne, f)
    ws = max(L.lgmlh_mul_mat_id_workspace(ty, ne, 2 * f, e, t, 1, nu),
             L.lgmlh_mul_mat_id_workspace(ty, ne, e, f, t, nu, nu))
    return dict(c=c, x=_normal(g, t, e), norm=1 + 0.1 * _normal(g, e), xn=_out(t, e),
                router=_raw(seed + 9, "f32", ne, e, e ** -0.5), logits=_out(t, ne),
                ids=torch.zeros(t, nu, dtype=torch.int32, device=DEV), wts=_out(t, nu), wgu=wgu,
                wdown=wdown, gu=_out(t * nu, 2 * f), h=_out(t * nu, f), ye=_out(t * nu, e),
                y=_out(t, e), ws=_bytes(ws))


def _run_moe(s):
    c, L, st = s["c"], hip.lib(), hip.stream()
    t, e, f, ne, nu, ty = (c[k] for k in ("rows", "embd", "ff", "experts", "used", "wtype"))
    ty = TYPES[ty]
    hip.check(L.lgmlh_rms_norm(s["x"].data_ptr(), t, e, 1e-6, s["norm"].data_ptr(),
                               s["xn"].data_ptr(), F32, st))
    _product("exact", F32, s["router"], ne, e, s["xn"], t, s["logits"], None, s["ws"])
    hip.check(L.lgmlh_moe_route(s["logits"].data_ptr(), t, ne, nu, hip.GATING_SOFTMAX, 1, 1.0,
                                s["ids"].data_ptr(), s["wts"].data_ptr(), st))
    fn = L.lgmlh_mul_mat_id_ggml if c["act"] == "ggml" else L.lgmlh_mul_mat_id
    hip.check(fn(ty, s["wgu"].data_ptr(), ne, 2 * f, e, s["xn"].data_ptr(), F32, 1,
                 s["ids"].data_ptr(), t, nu, s["gu"].data_ptr(), s["ws"].data_ptr(),
                 s["ws"].numel(), st))
    hip.check(L.lgmlh_swiglu(s["gu"].data_ptr(), t * nu, f, s["h"].data_ptr(), F32, st))
    hip.check(fn(ty, s["wdown"].data_ptr(), ne, e, f, s["h"].data_ptr(), F32, nu,
                 s["ids"].data_ptr(), t, nu, s["ye"].data_ptr(), s["ws"].data_ptr(),
                 s["ws"].numel(), st))
    hip.check(L.lgmlh_moe_sum(s["ye"].data_ptr(), s["wts"].data_ptr(), t, nu, e, s["x"].data_ptr(),
                              s["y"].data_ptr(), st))
    return {"logits": s["logits"], "y": s["y"]}


def _prep_head(c, seed):
    g, L, ty, n = _gen(seed + 1), hip.lib(), TYPES[c["wtype"]], c["rows"]
    return dict(c=c, x=_normal(g, n, c["embd"]), norm=1 + 0.1 * _normal(g, c["embd"]),
                xn=_out(n, c["embd"]), w=_repacked(seed, c["wtype"], c["vocab"], c["embd"]),
                y=_out(n, c["vocab"]), ids=torch.zeros(n, dtype=torch.int32, device=DEV),
                ws=_bytes(L.lgmlh_mul_mat_workspace(ty, c["vocab"], c["embd"], n)))


def _run_head(s):
    c, L, st, n = s["c"], hip.lib(), hip.stream(), s["c"]["rows"]
    hip.check(L.lgmlh_rms_norm(s["x"].data_ptr(), n, c["embd"], 1e-5, s["norm"].data_ptr(),
                               s["xn"].data_ptr(), F32, st))
    _product(c["act"], TYPES[c["wtype"]], s["w"], c["vocab"], c["embd"], s["xn"], n, s["y"], None,
             s["ws"])
    hip.check(L.lgmlh_argmax(s["y"].data_ptr(), n, c["vocab"], s["ids"].data_ptr(), st))
    return {"logits": s["y"], "ids": s["ids"]}


RING = 24  # blocks of a sequence's ring: a 1024-token window and a 512-token chunk


def _attention_pass(c, seed):
    """(tokens, positions before them) per sequence: the decoding ones, then
    the chunk's."""
    past = _lengths(c, seed)
    seq_n = [1] * len(past)
    if c["chunk"]:
        seq_n.append(c["chunk"])
        past.append(c["past"])
    return seq_n, past


def _prep_attention(c, seed):
    g, L = _gen(seed + 1), hip.lib()
    seq_n, past = _attention_pass(c, seed)
    n, h, kv, d = sum(seq_n), c["heads"], c["kv"], c["dim"]
    ids = np.zeros(n, np.int32)
    if c["window"]:
        blocks = RING * len(seq_n)
        tab = np.random.default_rng(seed + 11).permutation(blocks).astype(np.int32)
        tab = tab.reshape(len(seq_n), RING)
        plan = runtime.Plan(seq_n, past, tab, ids, h, kv, blocks, 12, ring_tab=tab,
                            window=c["window"])
    else:
        tab, blocks = _tables(seq_n, past, seed)
        plan = runtime.Plan(seq_n, past, tab, ids, h, kv, blocks, 28 if d >= 256 else 12)
    ws = L.lgmlh_attention_workspace(C.byref(plan.info), d)
    return dict(c=c, plan=plan, tab=tab, q=_normal(g, n, h, d), out=_out(n, h, d), ws=_bytes(ws),
                k=_normal(g, blocks, kv, 64, d).half(), v=_normal(g, blocks, kv, d, 64).half())


def _run_attention(s):
    c = s["c"]
    hip.check(hip.lib().lgmlh_paged_attention(
        s["q"].data_ptr(), c["heads"], c["kv"], c["dim"], c["dim"] ** -0.5, s["k"].data_ptr(),
        s["v"].data_ptr(), C.byref(s["plan"].ub), s["out"].data_ptr(), s["ws"].data_ptr(),
        s["ws"].numel(), hip.stream()))
    return s["out"]


def _flash_mask(c):
    """The additive mask of a chunk at the end of its cells, f16 (1, rows, cells)."""
    if c["mask"] == "none":
        return None
    t, j = torch.arange(c["rows"], device=DEV)[:, None], torch.arange(c["cells"], device=DEV)[None]
    p = c["cells"] - c["rows"] + t
    vis = (j <= p) & (j > p - 256 if c["mask"] == "window" else j >= 0)
    return torch.where(vis, 0.0, -math.inf).half()[None].contiguous()


def _prep_flash(c, seed):
    g = _gen(seed + 1)
    h, kv, d, t, n = (c[k] for k in ("heads", "kv", "dim", "rows", "cells"))
    return dict(c=c, q=_normal(g, h, t, d), k=_normal(g, n, kv, d).half(),
                v=_normal(g, n, kv, d).half(), mask=_flash_mask(c), out=_out(t, h, d))


def _run_flash(s):
    c = s["c"]
    h, kv, d, t, n = (c[k] for k in ("heads", "kv", "dim", "rows", "cells"))
    masked = s["mask"] is not None
    hip.check(hip.lib().lgmlh_flash_attn(
        s["q"].data_ptr(), h, t, d, s["k"].data_ptr(), s["v"].data_ptr(), kv, n, kv * d, d, kv * d,
        d, hip.ptr(s["mask"]), 1 if masked else 0, t if masked else 0, d ** -0.5, c["max_bias"],
        c["softcap"], s["out"].data_ptr(), hip.stream()))
    return s["out"]


TINY = dict(arch="llama", n_embd=256, n_head=4, n_head_kv=2, head_dim=64, n_ff=688, n_vocab=512,
            rope_base=1e4, eps=1e-6, n_rot=64, rope_neox=0, attn_scale=0.0)


def _hp(c):
    hp = dict(TINY if c["shape"] == "tiny" else workload.SHAPES[c["shape"]], n_layer=c["layers"],
              wtype=c["wtype"], act_quant=c["wtype"] != "f32")
    if c["shape"] == "tiny" and c["wtype"] != "f32":
        hp["n_ff"] = 768  # whole blocks
    return hp


def _model_source(c, hp, seed):
    """A weights source of DeviceModel: one seed per matrix, in the order asked."""
    if c["wtype"] != "f32":
        return runtime.generated_weights(hp, seed, workload.policy(c["wtype"], hp["n_layer"]))
    at = [0]

    def get(name, layer, rows, cols):
        at[0] += 1
        sd = 1.0 if name == "tok_embd" else cols ** -0.5
        return _raw(seed * 1000 + at[0], "f32", rows, cols, sd), F32, rows

    return get


def _prep_model(c, seed):
    hp = _hp(c)
    past = _lengths(c, seed)
    seq_n = [1] * len(past)
    if c["chunk"]:
        seq_n.append(c["chunk"])
        past.append(past[0])
    tab, blocks = _tables(seq_n, past, seed, extra=len(past))
    m = runtime.DeviceModel(hp, _model_source(c, hp, seed), blocks * 64)
    g = _gen(seed + 1)
    for pool in m.kpools + m.vpools:
        pool.view(torch.float16).copy_(_normal(g, pool.numel() // 2))
    ids = np.random.default_rng(seed + 3).integers(0, hp["n_vocab"], sum(seq_n)).astype(np.int32)
    return dict(c=c, m=m, hp=hp, seq_n=seq_n, past=past, tab=tab, ids=ids)


def _run_model(s):
    plan = s["m"].plan(s["seq_n"], s["past"], s["tab"], s["ids"])
    return s["m"].forward(plan)


_PREPARE = dict(product=_prep_product, ffn=_prep_ffn, moe=_prep_moe, head=_prep_head,
                attention=_prep_attention, flash=_prep_flash, model=_prep_model)
_RUN = dict(product=_run_product, ffn=_run_ffn, moe=_run_moe, head=_run_head,
            attention=_run_attention, flash=_run_flash, model=_run_model)


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    return _RUN[state["c"]["kind"]](state)


# ---- what a pass cannot do without --------------------------------------------
def _mat(wtype, rows, cols):
    return BITS[wtype] / 8 * rows * cols


def _attention_work(seq_n, past, h, kv, d, window=0):
    cells = flops = 0
    for n, p in zip(seq_n, past):
        seen = [min(p + j + 1, window) if window else p + j + 1 for j in range(n)]
        cells += min(p + n, window + n - 1) if window else p + n
        flops += sum(seen)
    return dict(bytes=cells * kv * d * 4 + 8.0 * sum(seq_n) * h * d, flops=4.0 * flops * h * d)


def work(case):
    c, kind = case, case["kind"]
    if kind == "product":
        b = _mat(c["wtype"], c["m"], c["k"]) + c["n"] * c["k"] * (2 if c["x"] == "f16" else 4)
        b += 4.0 * c["n"] * c["m"] * (2 if c["residual"] else 1)
        return dict(bytes=b, flops=2.0 * c["m"] * c["k"] * c["n"])
    if kind == "ffn":
        n, e, f = c["rows"], c["embd"], c["ff"]
        return dict(bytes=_mat(c["wtype"], 3 * f, e) + 4.0 * n * (2 * e + f), flops=6.0 * n * e * f)
    if kind == "moe":
        t, e, f, ne, nu = (c[k] for k in ("rows", "embd", "ff", "experts", "used"))
        picked = ne * (1 - (1 - nu / ne) ** t)
        return dict(bytes=picked * _mat(c["wtype"], 3 * f, e) + 4.0 * (ne * e + t * (2 * e + ne)),
                    flops=2.0 * t * e * (ne + 3 * f * nu))
    if kind == "head":
        n, e, v = c["rows"], c["embd"], c["vocab"]
        return dict(bytes=_mat(c["wtype"], v, e) + 4.0 * n * (e + v), flops=2.0 * n * e * v)
    if kind == "attention":
        ctx = [(c["lo"] + c["hi"]) / 2] * c["slots"]
        if c["window"]:
            ctx = [min(p, c["window"]) for p in ctx]
        w = _attention_work([1] * c["slots"], ctx, c["heads"], c["kv"], c["dim"], c["window"])
        if c["chunk"]:
            k = _attention_work([c["chunk"]], [c["past"]], c["heads"], c["kv"], c["dim"], c["window"])
            w = {m: w[m] + k[m] for m in w}
        return w
    if kind == "flash":
        h, kv, d, t, n = (c[k] for k in ("heads", "kv", "dim", "rows", "cells"))
        seen = {"none": t * n, "causal": t * (n - t) + t * (t + 1) / 2,
                "window": t * min(256, n)}[c["mask"]]
        b = 4.0 * n * kv * d + 8.0 * t * h * d + (0 if c["mask"] == "none" else 2.0 * t * n)
        return dict(bytes=b, flops=4.0 * seen * h * d)
    hp, n = _hp(c), c["slots"] + c["chunk"]
    e, h, kv, d, f, v = (hp[k] for k in ("n_embd", "n_head", "n_head_kv", "head_dim", "n_ff", "n_vocab"))
    out = c["slots"] + (1 if c["chunk"] else 0)
    a = _attention_work([1] * c["slots"] + ([c["chunk"]] if c["chunk"] else []),
                        [(c["lo"] + c["hi"]) / 2] * c["slots"] + [c["lo"]], h, kv, d)
    values = c["layers"] * (e * (2 * h + 2 * kv) * d + 3 * e * f)
    return dict(bytes=workload.weight_bytes(hp) + c["layers"] * a["bytes"] + 4.0 * (n * e + out * v),
                flops=2.0 * n * values + 2.0 * out * e * v + c["layers"] * a["flops"])


# ---- tolerances -----------------------------------------------------------------
def tolerance(case):
    """Single products and attention: f32 sums in another order. Chains in
    ggml's arithmetic quantize an intermediate result, where a last-bit
    difference moves some quantized value by one step; whole passes repeat
    that per layer."""
    kind = case["kind"]
    if kind == "model":
        return {"rel": 5e-5, "max": 2e-3} if case["wtype"] == "f32" else {"rel": 0.02, "max": 0.5}
    if kind == "attention" or kind == "flash":
        return {"rel": 1e-5, "max": 4e-4}
    if kind == "product":
        return {"rel": 5e-6, "max": 2e-4}
    if kind == "head":
        return {"rel": 2e-4, "max": 1e-2, "differ": 0.0}
    return {"rel": 2e-3, "max": 0.1} if case["act"] == "ggml" else {"rel": 1e-5, "max": 1e-3}


# ---- the same in 64 bits ----------------------------------------------------------
def _f16_of(b):
    return b.contiguous().view(torch.float16).double()


def _dequant(raw, wtype, rows, cols):
    """The f64 values of a matrix in its ggml layout."""
    if wtype == "f32":
        return raw.double()
    if wtype == "q8_0":
        b = raw.view(rows * cols // 32, 34)
        return (_f16_of(b[:, :2]) * b[:, 2:].view(torch.int8).double()).view(rows, cols)
    nb = rows * cols // 256
    if wtype == "q4_K":
        b = raw.view(nb, 144)
        d, dmin = _f16_of(b[:, 0:2]), _f16_of(b[:, 2:4])
        s = b[:, 4:16].int()
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | (s[:, 0:4] >> 6 << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | (s[:, 4:8] >> 6 << 4)], 1)
        q = b[:, 16:].view(nb, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).view(nb, 8, 32).double()
        v = (d * sc)[:, :, None] * q - (dmin * mn)[:, :, None]
        return v.view(rows, cols)
    b = raw.view(nb, 210)
    ql, qh = b[:, :128].view(nb, 2, 2, 32), b[:, 128:192].view(nb, 2, 1, 32)
    lo = torch.cat([ql & 15, ql >> 4], 2)                       # (nb, 2, 4, 32)
    hi = torch.cat([(qh >> (2 * t)) & 3 for t in range(4)], 2)
    q = (lo | hi << 4).double() - 32
    sc = b[:, 192:208].view(torch.int8).double().repeat_interleave(16, 1)
    return (_f16_of(b[:, 208:]) * sc * q.view(nb, 256)).view(rows, cols)


def _over(a, b):
    """a / b in f32, rounded once (a number over or under a tensor may go
    by way of a rounded reciprocal)."""
    a = a if torch.is_tensor(a) else torch.full_like(b, a)
    return a / (b if torch.is_tensor(b) else torch.full_like(a, b))


def _quantized(x, wtype):
    """x (f32) as the weight type's activation blocks give it back, in f64."""
    if wtype == "q8_0":
        b = x.view(-1, 32)
        d = _over(b.abs().amax(1, keepdim=True), 127.0)
        i = torch.where(d != 0, _over(1.0, d), 0.0)
        v = b * i
        q = torch.sign(v) * torch.floor(v.abs().double() + 0.5)
        return (q * d.half().double()).view(x.shape)
    b = x.view(-1, 256)
    big = b.gather(1, b.abs().argmax(1, keepdim=True))
    i = torch.where(big != 0, _over(-127.0, big), 0.0)
    q = torch.clamp(torch.round(i * b), max=127.0)
    d = torch.where(big != 0, _over(1.0, i), 0.0)
    return (q.double() * d.double()).view(x.shape)


def _mul(x, raw, wtype, rows, cols, act):
    """x (f64) times the matrix, x taken as f32 rows."""
    x = _quantized(x.float(), wtype) if act == "ggml" and wtype != "f32" else x
    return x @ _dequant(raw, wtype, rows, cols).T


def _rms(x, w, eps):
    x = x.double()
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _glu(gu, f, gelu):
    g, u = gu[..., :f], gu[..., f:]
    if gelu:
        g = 0.5 * g * (1 + torch.tanh(math.sqrt(2 / math.pi) * (g + 0.044715 * g ** 3)))
    else:
        g = g / (1 + torch.exp(-g))
    return g * u


def _softmax_v(s, v):
    """softmax(s) v; a row of -inf gives zeros."""
    m = s.amax(-1, keepdim=True)
    p = torch.exp(s - torch.where(torch.isfinite(m), m, 0.0))
    return (p @ v) / p.sum(-1, keepdim=True).clamp_min(1e-300)


def _seq_attention(q, k, v, p0, scale, window=0):
    """q (H, n, D) at positions p0 .. over k, v (Hkv, p0 + n, D), causal."""
    n, g = q.shape[1], q.shape[0] // k.shape[0]
    s = q @ k.repeat_interleave(g, 0).transpose(1, 2) * scale
    p, j = p0 + torch.arange(n, device=DEV)[:, None], torch.arange(k.shape[1], device=DEV)[None]
    see = (j <= p) & (j > p - window) if window else j <= p
    return _softmax_v(torch.where(see, s, -math.inf), v.repeat_interleave(g, 0))


def _exact_attention(c, s, seed):
    seq_n, past = _attention_pass(c, seed)
    out, at = [], 0
    for i, (n, p) in enumerate(zip(seq_n, past)):
        pos = torch.arange(p + n, device=DEV)
        if c["window"]:
            tab = torch.from_numpy(s["tab"][i]).to(DEV).long()
            first = max(0, p + 1 - c["window"])
            pos = pos[first:]
            blk = tab[(pos // 64) % RING]
        else:
            first = 0
            blk = torch.from_numpy(s["tab"][i]).to(DEV).long()[pos // 64]
        k = s["k"][blk, :, pos % 64].double().transpose(0, 1)
        v = s["v"][blk, :, :, pos % 64].double().transpose(0, 1)
        q = s["q"][at:at + n].double().transpose(0, 1)
        o = _seq_attention(q, k, v, p - first, c["dim"] ** -0.5, c["window"])
        out.append(o.transpose(0, 1))
        at += n
    return torch.cat(out)


def _exact_moe(c, s, seed):
    t, e, f, ne, nu = (c[k] for k in ("rows", "embd", "ff", "experts", "used"))
    ty, act = c["wtype"], c["act"]
    xn = _rms(s["x"], s["norm"], 1e-6)
    logits = xn @ s["router"].double().T
    p = torch.softmax(logits, -1)
    ids = torch.sort(logits, dim=-1, descending=True, stable=True).indices[:, :nu]
    w = p.gather(1, ids)
    w = w / w.sum(1, keepdim=True).clamp_min(6.103515625e-5)
    gate, up, down = (_raw(seed + o, ty, ne * r, k) for o, r, k in ((0, f, e), (3, f, e), (7, e, f)))
    y = s["x"].double().clone()
    for x in range(ne):
        tok, slot = (ids == x).nonzero(as_tuple=True)
        if not len(tok):
            continue

        def part(raw, rows):
            n = raw.numel() // ne
            return raw.view(-1)[x * n:(x + 1) * n]
        gu = torch.cat([_mul(xn[tok], part(gate, f), ty, f, e, act),
                        _mul(xn[tok], part(up, f), ty, f, e, act)], 1)
        o = _mul(_glu(gu, f, False), part(down, e), ty, e, f, act)
        y.index_add_(0, tok, o * w[tok, slot][:, None])
    return {"logits": logits, "y": y}


def _exact_model(c, s, seed):
    """The f32 model: the pass in f64 over f16 KV (a pass's own k and v are
    kept in f16 too); rope angles are the f32 running product."""
    hp = s["hp"]
    e, h, kv, d, f = (hp[k] for k in ("n_embd", "n_head", "n_head_kv", "head_dim", "n_ff"))
    src, nl = _model_source(c, hp, seed), hp["n_layer"]
    mats = [{n: src(n, i, r, k)[0].double() for n, r, k in (
        ("wq", h * d, e), ("wk", kv * d, e), ("wv", kv * d, e), ("wo", e, h * d), ("gate", f, e),
        ("up", f, e), ("down", e, f))} for i in range(nl)]
    embd, outw = src("tok_embd", None, hp["n_vocab"], e)[0], src("output", None, hp["n_vocab"], e)[0]
    x = embd.double()[torch.from_numpy(s["ids"]).to(DEV).long()]
    pos = np.concatenate([p + np.arange(n) for n, p in zip(s["seq_n"], s["past"])])
    th = np.empty((len(pos), d // 2), np.float32)
    th[:, 0] = pos
    step = np.float32(math.pow(hp["rope_base"], -2.0 / d))
    for i in range(1, d // 2):
        th[:, i] = th[:, i - 1] * step
    th = torch.from_numpy(th).to(DEV).double()[:, None]
    ends = np.cumsum(s["seq_n"])

    def rope(a):  # pairs (2i, 2i + 1)
        u, w = a[..., 0::2], a[..., 1::2]
        return torch.stack([u * th.cos() - w * th.sin(), u * th.sin() + w * th.cos()], -1).flatten(-2)

    for i, m in enumerate(mats):
        y = _rms(x, torch.ones(e, device=DEV), hp["eps"])
        n = len(y)
        q, k = rope((y @ m["wq"].T).view(n, h, d)), rope((y @ m["wk"].T).view(n, kv, d))
        k, v = k.half().double(), (y @ m["wv"].T).view(n, kv, d).half().double()
        kp = s["m"].kpools[i].view(torch.float16).view(-1, kv, 64, d)
        vp = s["m"].vpools[i].view(torch.float16).view(-1, kv, d, 64)
        att = []
        for j, (cnt, p) in enumerate(zip(s["seq_n"], s["past"])):
            at = slice(ends[j] - cnt, ends[j])
            cells = torch.arange(p, device=DEV)
            blk = torch.from_numpy(s["tab"][j]).to(DEV).long()[cells // 64]
            ka = torch.cat([kp[blk, :, cells % 64].double(), k[at]]).transpose(0, 1)
            va = torch.cat([vp[blk, :, :, cells % 64].double(), v[at]]).transpose(0, 1)
            o = _seq_attention(q[at].transpose(0, 1), ka, va, p, d ** -0.5)
            att.append(o.transpose(0, 1).reshape(cnt, h * d))
        x = x + torch.cat(att) @ m["wo"].T
        y = _rms(x, torch.ones(e, device=DEV), hp["eps"])
        x = x + _glu(torch.cat([y @ m["gate"].T, y @ m["up"].T], 1), f, False) @ m["down"].T
    x = _rms(x[torch.from_numpy(ends - 1).to(DEV)], torch.ones(e, device=DEV), hp["eps"])
    return x @ outw.double().T


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "model" and c["wtype"] != "f32":
        return None  # ggml's arithmetic quantizes every layer's intermediate results
    s = prepare(case, seed)
    if kind == "product":
        y = _mul(s["x"].double(), _raw(seed, c["wtype"], c["m"], c["k"]), c["wtype"], c["m"], c["k"],
                 c["act"])
        return y + s["res"].double() if c["residual"] else y
    if kind == "ffn":
        n, e, f, ty = c["rows"], c["embd"], c["ff"], c["wtype"]
        xn = _rms(s["x"], s["norm"], 1e-5)
        h = _glu(_mul(xn, _raw(seed, ty, 2 * f, e), ty, 2 * f, e, c["act"]), f, c["gelu"])
        return {"h": h, "y": s["x"].double() + _mul(h, _raw(seed + 7, ty, e, f), ty, e, f, c["act"])}
    if kind == "head":
        y = _mul(_rms(s["x"], s["norm"], 1e-5), _raw(seed, c["wtype"], c["vocab"], c["embd"]),
                 c["wtype"], c["vocab"], c["embd"], c["act"])
        return {"logits": y, "ids": None}
    if kind == "flash":
        g, d = c["heads"] // c["kv"], c["dim"]
        k = s["k"].double().permute(1, 0, 2).repeat_interleave(g, 0)
        v = s["v"].double().permute(1, 0, 2).repeat_interleave(g, 0)
        x = s["q"].double() @ k.transpose(1, 2).contiguous() * d ** -0.5
        if c["softcap"]:
            x = c["softcap"] * torch.tanh(x / c["softcap"])
        x = x if s["mask"] is None else x + s["mask"].double()
        return _softmax_v(x, v).transpose(0, 1).contiguous()
    return {"attention": _exact_attention, "moe": _exact_moe, "model": _exact_model}[kind](c, s, seed)
