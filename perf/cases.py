"""The work a user of this framework has it do, as cases that can be measured.

A case is a dict of plain values; `listed()` holds the fixed ones, `draw(rng)` gives more of the
same ranges.  Six kinds of work, each through the public functions of kernels.py:

  proj       one quantised linear, called eagerly
  linears    the four GEMM launches of a decoder layer (q|k|v, o, gate|up, down), as a captured
             graph for decode and verification steps and eagerly for prompt chunks
  mlp        the W8A8 MLP block of a prompt chunk: quantise, gate|up, SiLU*mul + quantise, down
  attention  verification attention over the INT8 paged cache, as a captured graph
  chunk      a prompt chunk: append its K/V to the paged cache, then attend to the whole cache
  layer      a whole W8A8 decoder layer replayed from plan-buffer graphs (PlanGraphSet)

The shapes are the framework's own (hidden 4096, 1024 K/V channels, MLP 14336, 32 query heads
over 8 K/V heads, B * (k + 1) rows) and generic ones of the same make.
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "specdec-quant-triton_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import kernels as K  # noqa: E402
from specq.plan import PlanGraphSet  # noqa: E402

DEV = "cuda"
GROUP = 128  # INT4 scale group
PAGE = 16
F64 = torch.float64


# ----------------------------------------------------------------------------------------
# Cases
# ----------------------------------------------------------------------------------------
def listed():
    return [
        # The smallest call: one token through one projection, weight as the reference's scripts pass it.
        dict(name="proj_w8a8_decode", kind="proj", fmt="w8a8", M=1, N=4096, K=4096),
        # Odd sizes throughout: a short prompt's rows, channels and K that no tile divides.
        dict(name="proj_w8a8_ragged", kind="proj", fmt="w8a8", M=517, N=5000, K=3088),
        # Verification of 8 drafts for 8 sequences: every linear of a layer, the framework's main workload.
        dict(name="linears_w8a8_verify", kind="linears", fmt="w8a8", M=72, hidden=4096, kv=1024, ff=14336, graph=True),
        # The same step with INT4 weights and fp16 activations.
        dict(name="linears_w4a16_verify", kind="linears", fmt="w4a16", M=72, hidden=4096, kv=1024, ff=14336, graph=True),
        # INT4 weights on the INT8 path, 16 sequences of 9 tokens, on a wider layer with full K/V heads.
        dict(name="linears_w4a8_verify", kind="linears", fmt="w4a8", M=144, hidden=5120, kv=5120, ff=13824, graph=True),
        # A prompt chunk through an INT4 layer: the GEMMs are bound by the matrix cores here.
        dict(name="linears_w4a16_prefill", kind="linears", fmt="w4a16", M=1024, hidden=4096, kv=1024, ff=14336,
             graph=False),
        # A long prompt chunk through the INT8 MLP, with its two quantisations: the largest work.
        dict(name="mlp_w8a8_prefill", kind="mlp", M=2048, hidden=4096, ff=14336),
        # Attention of the verification step above, context 4096.
        dict(name="attn_verify", kind="attention", B=8, q_len=9, ctx=4096, ragged=False, H=32, H_KV=8, D=128,
             scale32=False),
        # Plain decoding of a full batch whose sequences have all lengths up to 8192.
        dict(name="attn_decode_ragged", kind="attention", B=32, q_len=1, ctx=8192, ragged=True, H=32, H_KV=8, D=128,
             scale32=True),
        # One sequence with a long context, 4 drafts.
        dict(name="attn_long", kind="attention", B=1, q_len=5, ctx=65536, ragged=False, H=32, H_KV=8, D=128,
             scale32=True),
        # Chunked prefill of two prompts: 256 new tokens each behind up to 3840 cached ones.
        dict(name="chunk_prefill", kind="chunk", B=2, q_len=256, ctx=4096, ragged=True, H=32, H_KV=8, D=128,
             scale32=True),
        # A whole decode step of one layer, replayed from plan graphs captured for up to 4 sequences.
        dict(name="layer_plan_decode", kind="layer", B=3, b_max=4, q_len=1, ctx=1024, hidden=4096, kv=1024, ff=14336),
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _dims(rng, fmt):
    """Hidden, K/V and MLP widths: whole 128-blocks for W4A16 (its scale groups), 16s for INT8."""
    step = 256 if fmt == "w4a16" else rng.choice((16, 128, 512))
    to = lambda x: max(step, x // step * step)  # noqa: E731
    hidden = to(_log(rng, 1024, 5120))
    return hidden, to(hidden // rng.choice((1, 2, 4, 8))), to(int(hidden * rng.uniform(2.5, 3.5)))


def _rows(rng):
    """The rows of a decode or verification step: B sequences of k + 1 tokens, at most 288."""
    return _log(rng, 1, 32) * (rng.randrange(9) + 1)


def _heads(rng):
    h_kv = rng.choice((2, 4, 8))
    return h_kv * rng.choice((1, 2, 4, 8)), h_kv, rng.choice((64, 128, 128))


def draw(rng):
    kind = rng.choice(("proj", "proj", "linears", "linears", "linears", "prefill", "mlp", "attention", "attention",
                       "chunk", "layer"))
    fmt = rng.choice(("w8a8", "w4a16", "w4a8"))
    if kind == "proj":
        step = 256 if fmt == "w4a16" else 16
        N, Kd = _log(rng, 256, 14336), max(step, _log(rng, 512, 8192) // step * step)
        return dict(kind="proj", fmt=fmt, M=min(_log(rng, 1, 2048), (1 << 37) // (N * Kd)), N=N, K=Kd)
    if kind in ("linears", "prefill"):
        hidden, kv, ff = _dims(rng, fmt)
        M = _rows(rng) if kind == "linears" else _log(rng, 256, 1024)
        return dict(kind="linears", fmt=fmt, M=M, hidden=hidden, kv=kv, ff=ff, graph=kind == "linears")
    if kind == "mlp":
        hidden, _, ff = _dims(rng, "w8a8")
        return dict(kind="mlp", M=_log(rng, 1, 2048), hidden=min(hidden, 4096), ff=min(ff, 14336))
    if kind == "attention":
        H, H_KV, D = _heads(rng)
        q_len = rng.randrange(1, min(9, 64 * H_KV // H) + 1)
        B = _log(rng, 1, 32)
        return dict(kind="attention", B=B, q_len=q_len, ctx=_log(rng, 64, 262144 // max(B, 4)),
                    ragged=rng.random() < 0.7, H=H, H_KV=H_KV, D=D, scale32=rng.random() < 0.5)
    if kind == "chunk":
        H, H_KV, D = _heads(rng)
        q_len = _log(rng, 16, 256)
        return dict(kind="chunk", B=rng.randrange(1, 3), q_len=q_len, ctx=_log(rng, q_len, 4096),
                    ragged=rng.random() < 0.7, H=H, H_KV=H_KV, D=D, scale32=rng.random() < 0.5)
    b_max = _log(rng, 1, 32)
    return dict(kind="layer", B=rng.randrange(1, b_max + 1), b_max=b_max, q_len=rng.choice((1, 3, 5, 9)),
                ctx=_log(rng, 64, 2048), hidden=4096, kv=1024, ff=14336)


# ----------------------------------------------------------------------------------------
# Inputs.  Weights and activations have the values of real ones: weights normal with a standard
# deviation of hidden^-1/2 quantised by the framework's formats, activations normal.
# ----------------------------------------------------------------------------------------
class _Gen:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(1000003 * int(seed) + 17)

    def normal(self, *shape):
        return torch.randn(shape, device=DEV, generator=self.g)

    def uniform(self, lo, hi, *shape):
        return torch.rand(shape, device=DEV, generator=self.g) * (hi - lo) + lo

    def act16(self, M, Kd):
        return self.normal(M, Kd).half()

    def act8(self, M, Kd):
        return K.quantize_act_int8(self.act16(M, Kd))

    def int8(self, N, Kd):
        """INT8 weight [N, K] and its fp32 channel scale."""
        w = (self.normal(N, Kd) * 30).round_().clamp_(-127, 127).to(torch.int8)
        return w, self.uniform(0.8, 1.2, N) / (30 * math.sqrt(Kd))

    def nibbles(self, N, Kd):
        return ((self.normal(N, Kd) * 2.3).round_().clamp_(-8, 7) + 8).to(torch.uint8)

    def perm(self, n):
        return torch.randperm(n, device=DEV, generator=self.g)


def _pack_u8(q):
    """Nibbles [N, K] as the reference packs them: byte j holds k = j and k = j + K/2."""
    half = q.shape[1] // 2
    return (q[:, :half] | (q[:, half:] << 4)).contiguous()


def _weight(gen, fmt, N, Kd):
    """(what the call takes as its weight, its scales, the integer weight for exact())."""
    if fmt == "w8a8":
        w, s = gen.int8(N, Kd)
        return K.pack_weight_int8(w), s, w
    q = gen.nibbles(N, Kd)
    if fmt == "w4a8":
        return K.pack_weight_w4a8(_pack_u8(q)), gen.uniform(0.8, 1.2, N) / (2.3 * math.sqrt(Kd)), q
    return K.pack_weight_int4(_pack_u8(q)), (gen.uniform(0.8, 1.2, N, Kd // GROUP) / (2.3 * math.sqrt(Kd))).half(), q


def _layer_shapes(c):
    """The launches of a layer: the widths that share an input, and that input's length."""
    h, kv, ff = c["hidden"], c["kv"], c["ff"]
    return [("qkv", (h, kv, kv), h), ("o", (h,), h), ("gate_up", (ff, ff), h), ("down", (h,), ff)]


def _cache(gen, c, lens):
    """A paged INT8 cache whose sequences' pages are shuffled over a pool with room for all at full length."""
    B, H_KV, D = len(lens), c["H_KV"], c["D"]
    per = [-(-n // PAGE) for n in lens]
    pool = B * max(per)
    ids = gen.perm(pool).to(torch.int32)
    bt = torch.zeros((B, max(per)), dtype=torch.int32, device=DEV)
    at = 0
    for b, n in enumerate(per):
        bt[b, :n] = ids[at:at + n]
        at += n
    kv = [torch.randint(-127, 128, (pool, PAGE, H_KV, D), dtype=torch.int8, device=DEV, generator=gen.g) for _ in "kv"]
    dt = torch.float32 if c["scale32"] else torch.float16
    sc = [gen.uniform(0.005, 0.02, pool, PAGE, H_KV).to(dt) for _ in "kv"]
    return kv + sc + [bt, torch.tensor(lens, dtype=torch.int32, device=DEV)]


def _lens(c, seed):
    """Context lengths, the new tokens among them: all `ctx`, or spread from an eighth of it up to it."""
    if not c["ragged"]:
        return [c["ctx"]] * c["B"]
    g = torch.Generator().manual_seed(seed + 5)
    lo = max(c["q_len"], c["ctx"] // 8)
    lens = torch.randint(lo, c["ctx"] + 1, (c["B"],), generator=g).tolist()
    lens[0] = c["ctx"]
    return lens


def _capture(fn):
    """fn() as a graph, warmed up once so that workspaces have their size."""
    fn()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = fn()
    return g, out


def _inputs(case, seed):
    """Everything of a case that the seed decides, before any graph."""
    c, gen, kind = case, _Gen(seed), case["kind"]
    s = {"case": c}
    if kind == "proj":
        if c["fmt"] == "w8a8":
            s["w"], s["sw"] = gen.int8(c["N"], c["K"])
        else:
            s["w"], s["sw"], s["q"] = _weight(gen, c["fmt"], c["N"], c["K"])
        s["x"] = (gen.act16(c["M"], c["K"]),) if c["fmt"] == "w4a16" else gen.act8(c["M"], c["K"])
    elif kind == "linears":
        s["w"] = {n: [_weight(gen, c["fmt"], N, Kd) for N in Ns] for n, Ns, Kd in _layer_shapes(c)}
        s["x"] = {n: (gen.act16(c["M"], Kd),) if c["fmt"] == "w4a16" else gen.act8(c["M"], Kd)
                  for n, _, Kd in _layer_shapes(c)}
    elif kind == "mlp":
        s["w"] = {n: [_weight(gen, "w8a8", N, Kd) for N in Ns]
                  for n, Ns, Kd in (("gate_up", (c["ff"], c["ff"]), c["hidden"]), ("down", (c["hidden"],), c["ff"]))}
        s["x"] = gen.act16(c["M"], c["hidden"])
    elif kind in ("attention", "chunk"):
        s["kv"] = _cache(gen, c, _lens(c, seed))
        s["q"] = gen.normal(c["B"], c["q_len"], c["H"], c["D"]).half()
        if kind == "chunk":
            s["new"] = [gen.normal(c["B"], c["q_len"], c["H_KV"], c["D"]).half() for _ in "kv"]
    else:
        d = 128
        s["c"] = dict(c, H=c["hidden"] // d, H_KV=c["kv"] // d, D=d, scale32=True)
        s["kv"] = _cache(gen, s["c"], [c["ctx"] + c["q_len"]] * c["b_max"])
        s["w"] = {n: [_weight(gen, "w8a8", N, Kd) for N in (Ns if n == "gate_up" else (sum(Ns),))]
                  for n, Ns, Kd in _layer_shapes(c)}
        s["x"] = gen.act16(c["b_max"] * c["q_len"], c["hidden"])
    return s


# ----------------------------------------------------------------------------------------
# The calls
# ----------------------------------------------------------------------------------------
def _matmul(fmt, x, w, sw, **kw):
    fn = {"w8a8": K.w8a8_matmul, "w4a16": K.w4a16_matmul, "w4a8": K.w4a8_matmul}[fmt]
    return fn(*x, w, sw, BLOCK_M=None, **kw)[0]


def _grouped(fmt, x, ws, **kw):
    pairs = [(w, sw) for w, sw, _ in ws]
    if len(pairs) == 1:
        return [_matmul(fmt, x, *pairs[0], **kw)]
    return (K.w4a16_matmul_grouped if fmt == "w4a16" else K.w8a8_matmul_grouped)(*x, pairs, BLOCK_M=None, **kw)[0]


def _run_linears(s):
    return {n: _grouped(s["case"]["fmt"], s["x"][n], s["w"][n]) for n in s["w"]}


def _run_attention(s):
    c = s["case"]
    return K.paged_attention(s["q"], *s["kv"], c["q_len"])[0]


class _Layer:
    """One decoder layer's launches at a given grid, on buffers of its own."""

    def __init__(self, s):
        self.s, c = s, s["c"]
        self.c, M = c, c["b_max"] * c["q_len"]
        e = lambda n, dt=torch.float16: torch.zeros((M, n), dtype=dt, device=DEV)  # noqa: E731
        q8 = lambda n: (e(n, torch.int8), torch.zeros((M,), device=DEV))  # noqa: E731
        self.xq, self.oq, self.mq, self.hq = q8(c["hidden"]), q8(c["hidden"]), q8(c["hidden"]), q8(c["ff"])
        self.qkv, self.att, self.o = e(c["hidden"] + 2 * c["kv"]), e(c["hidden"]), e(c["hidden"])
        self.gate, self.up, self.down = e(c["ff"]), e(c["ff"]), e(c["hidden"])

    def step(self, Bg, ql, plan):
        c, w, M = self.c, self.s["w"], Bg * ql
        kw = dict(plan=plan.gemm, grid_m_max=M)
        gk = dict(kw, BLOCK_M=None, plan_tiles=plan.tiles)
        at = lambda qs: (qs[0][:M], qs[1][:M])  # noqa: E731
        quant = lambda x, qs: K.quantize_act_int8_gpu(x[:M], q=qs[0][:M], s=qs[1][:M], **kw)  # noqa: E731
        quant(self.s["x"], self.xq)
        K.w8a8_matmul(*at(self.xq), *w["qkv"][0][:2], out=self.qkv[:M], **gk)
        h, kv = c["hidden"], c["kv"]
        new = self.qkv[:M].view(Bg, ql, -1, c["D"])
        q, k, v = new[:, :, :h // c["D"]], new[:, :, h // c["D"]:(h + kv) // c["D"]], new[:, :, (h + kv) // c["D"]:]
        kc, vc, ks, vs, bt, ln = self.s["kv"]
        K.paged_kv_append(k, v, kc, vc, ks, vs, bt[:Bg], ln[:Bg], ql, plan=plan.attn)
        K.paged_attention(q, kc, vc, ks, vs, bt[:Bg], ln[:Bg], ql, plan=plan.attn,
                          out=self.att[:M].view(Bg, ql, -1, c["D"]))
        quant(self.att, self.oq)
        K.w8a8_matmul(*at(self.oq), *w["o"][0][:2], out=self.o[:M], **gk)
        quant(self.o, self.mq)
        K.w8a8_matmul_grouped(*at(self.mq), [g[:2] for g in w["gate_up"]], outs=[self.gate[:M], self.up[:M]], **gk)
        K.silu_mul_quant_int8(self.gate[:M], self.up[:M], q=self.hq[0][:M], s=self.hq[1][:M], **kw)
        K.w8a8_matmul(*at(self.hq), *w["down"][0][:2], out=self.down[:M], **gk)

    def outputs(self, B):
        M = B * self.c["q_len"]
        return {"att": self.att[:M], "o": self.o[:M], "hq": self.hq[0][:M], "hs": self.hq[1][:M],
                "down": self.down[:M], "kc": self.s["kv"][0], "vc": self.s["kv"][1]}


def prepare(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    if kind == "attention" or (kind == "linears" and case["graph"]):
        s["graph"], s["out"] = _capture(lambda: (_run_attention if kind == "attention" else _run_linears)(s))
    elif kind == "layer":
        s["layer"] = _Layer(s)
        s["graph"] = PlanGraphSet(s["layer"].step, case["b_max"], [case["q_len"]], device=DEV)
    return s


def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind == "layer":
        s["graph"].replay(c["B"], c["q_len"])
        return s["layer"].outputs(c["B"])
    if "graph" in s:
        s["graph"].replay()
        return s["out"]
    if kind == "proj":
        return _matmul(c["fmt"], s["x"], s["w"], s["sw"])
    if kind == "linears":
        return _run_linears(s)
    if kind == "mlp":
        x = K.quantize_act_int8_gpu(s["x"])
        gate, up = _grouped("w8a8", x, s["w"]["gate_up"])
        h = K.silu_mul_quant_int8(gate, up)
        down = _grouped("w8a8", h, s["w"]["down"])[0]
        return {"q": x[0], "s": x[1], "gate": gate, "up": up, "hq": h[0], "hs": h[1], "down": down}
    kc, vc, ks, vs, bt, ln = s["kv"]
    K.paged_kv_append(*s["new"], kc, vc, ks, vs, bt, ln, c["q_len"])
    qpp = min(c["q_len"], 64 * c["H_KV"] // c["H"])
    out = K.paged_attention(s["q"], kc, vc, ks, vs, bt, ln, c["q_len"], QPP=qpp)[0]
    return {"out": out, "kc": kc, "vc": vc, "ks": ks, "vs": vs}


# ----------------------------------------------------------------------------------------
# What a pass cannot do without, and what its results may differ by
# ----------------------------------------------------------------------------------------
def _gemm_work(fmt, M, Ns, Kd):
    N = sum(Ns)
    wb = {"w8a8": N * Kd + 4 * N, "w4a8": N * Kd // 2 + 4 * N, "w4a16": N * Kd // 2 + 2 * N * Kd // GROUP}[fmt]
    xb = 2 * M * Kd if fmt == "w4a16" else M * Kd + 4 * M
    return wb + xb + 2 * M * N, 2 * M * N * Kd


def _attn_work(c, lens, written):
    """K/V bytes and scales of the visible tokens, Q and O; two products over the causal pairs."""
    H, H_KV, D, ql = c["H"], c["H_KV"], c["D"], c["q_len"]
    sb = 4 if c["scale32"] else 2
    b = sum(n * H_KV * (2 * D + 2 * sb) + 4 * (-(-n // PAGE)) + 4 for n in lens) + 4 * len(lens) * ql * H * D
    f = sum(4 * H * D * (ql * (n - ql) + ql * (ql + 1) // 2) for n in lens)
    if written:  # the new tokens' K/V read in fp16
        b += len(lens) * ql * H_KV * 4 * D
    return b, f


def work(case):
    c, kind = case, case["kind"]
    if kind == "proj":
        b, f = _gemm_work(c["fmt"], c["M"], (c["N"],), c["K"])
    elif kind == "linears":
        parts = [_gemm_work(c["fmt"], c["M"], Ns, Kd) for _, Ns, Kd in _layer_shapes(c)]
        b, f = (sum(p[i] for p in parts) for i in (0, 1))
    elif kind == "mlp":
        M, h, ff = c["M"], c["hidden"], c["ff"]
        parts = [_gemm_work("w8a8", M, (ff, ff), h), _gemm_work("w8a8", M, (h,), ff)]
        b = sum(p[0] for p in parts) + M * h * 3 + 4 * M + M * ff * 5 + 4 * M
        f = sum(p[1] for p in parts)
    elif kind in ("attention", "chunk"):
        b, f = _attn_work(c, _lens(c, 0), kind == "chunk")
    else:
        M, h, kv, ff = c["B"] * c["q_len"], c["hidden"], c["kv"], c["ff"]
        parts = [_gemm_work("w8a8", M, Ns, Kd) for _, Ns, Kd in _layer_shapes(c)]
        parts.append(_attn_work(dict(c, H=h // 128, H_KV=kv // 128, D=128, scale32=True),
                                [c["ctx"] + c["q_len"]] * c["B"], True))
        b = sum(p[0] for p in parts) + M * (9 * h + 5 * ff)
        f = sum(p[1] for p in parts)
    return {"bytes": b, "flops": f}


def tolerance(case):
    kind, fmt = case["kind"], case.get("fmt")
    if kind in ("proj", "linears"):
        # INT8 products sum exactly in INT32, and the epilogue's roundings are fixed; fp16
        # products sum in fp32 in any order before the one rounding to fp16, which moves one
        # value in some hundreds by its last bit.
        return {"rel": 1e-4} if fmt == "w4a16" else "exact"
    if kind in ("attention", "chunk"):
        # 3e-4 from 64 bits measured: probabilities and outputs in fp16.
        return {"rel": 1.2e-3, "differ": 1e-4}
    # Whole blocks: a last bit ahead of a quantisation moves INT8 values by one, which is 2e-3
    # of the MLP's output, and 3e-2 behind the three quantisations of the layer.
    return {"rel": 8e-3, "differ": 1e-2} if kind == "mlp" else {"rel": 8e-2, "differ": 0.3}


# ----------------------------------------------------------------------------------------
# The same in 64 bits.  Values that the entry points hand over in fp16 or INT8 are rounded there.
# ----------------------------------------------------------------------------------------
def _exact_gemm(fmt, x, w, sw):
    if fmt == "w4a16":
        deq = ((w.half() - 8).view(w.shape[0], -1, GROUP) * sw[..., None]).view(w.shape)  # fp16 by definition
        return x[0].to(F64) @ deq.to(F64).t()
    w = w.to(F64) - (8 if fmt == "w4a8" else 0)
    return (x[0].to(F64) @ w.t()) * x[1].to(F64)[:, None] * sw.to(F64)


def _exact_quant(x):
    s = x.abs().amax(-1).clamp(min=1e-8) / 127
    return torch.round(x / s[..., None]).clamp(-127, 127), s


def _exact_attention(c, q, kc, vc, ks, vs, bt, lens):
    B, ql, H, D = q.shape
    G = H // c["H_KV"]
    out = torch.zeros((B, ql, H, D), dtype=F64, device=DEV)
    for b, n in enumerate(lens):
        pos = torch.arange(n, device=DEV)
        pg, sl = bt[b, pos // PAGE].long(), pos % PAGE
        mask = pos[None, :] > (n - ql + torch.arange(ql, device=DEV))[:, None]
        for h in range(c["H_KV"]):
            k = kc[pg, sl, h].to(F64) * ks[pg, sl, h].to(F64)[:, None]
            v = vc[pg, sl, h].to(F64) * vs[pg, sl, h].to(F64)[:, None]
            qq = q[b, :, h * G:(h + 1) * G].to(F64)  # [ql, G, D]
            sc = (qq.reshape(ql * G, D) @ k.t()).view(ql, G, n) / math.sqrt(D)
            p = sc.masked_fill(mask[:, None, :], float("-inf")).softmax(-1)
            out[b, :, h * G:(h + 1) * G] = (p.reshape(ql * G, n) @ v).view(ql, G, D)
    return out


def _exact_append(new, kv, lens, ql):
    """The cache with the new tokens quantised into their pages, in place."""
    kc, vc, ks, vs, bt, _ = kv
    for x, cache, scale in ((new[0], kc, ks), (new[1], vc, vs)):
        q, s = _exact_quant(x.to(F64))
        for b, n in enumerate(lens):
            pos = torch.arange(n - ql, n, device=DEV)
            pg, sl = bt[b, pos // PAGE].long(), pos % PAGE
            cache[pg, sl] = q[b].to(cache.dtype)
            scale[pg, sl] = s[b].to(scale.dtype)


def exact(case, seed):
    c, s, kind = case, _inputs(case, seed), case["kind"]
    if kind == "proj":
        w = s["w"] if c["fmt"] == "w8a8" else s["q"]
        return _exact_gemm(c["fmt"], s["x"], w, s["sw"])
    if kind == "linears":
        return {n: [_exact_gemm(c["fmt"], s["x"][n], q, sw) for _, sw, q in s["w"][n]] for n in s["w"]}
    if kind == "attention":
        return _exact_attention(c, s["q"], *s["kv"][:5], _lens(c, seed))
    if kind == "chunk":
        _exact_append(s["new"], s["kv"], _lens(c, seed), c["q_len"])
        kc, vc, ks, vs = s["kv"][:4]
        return {"out": _exact_attention(c, s["q"], *s["kv"][:5], _lens(c, seed)),
                "kc": kc, "vc": vc, "ks": ks.to(F64), "vs": vs.to(F64)}

    def lin(x, ws):
        return [_exact_gemm("w8a8", x, q, sw) for _, sw, q in ws]

    def mlp(x):
        gate, up = lin(x, s["w"]["gate_up"])
        g16, u16 = gate.half().to(F64), up.half().to(F64)
        h = _exact_quant((torch.nn.functional.silu(g16) * u16).half().to(F64))
        return gate, up, h, lin(h, s["w"]["down"])[0]

    if kind == "mlp":
        x = _exact_quant(s["x"].to(F64))
        gate, up, h, down = mlp(x)
        return {"q": x[0], "s": x[1], "gate": gate, "up": up, "hq": h[0], "hs": h[1], "down": down}
    lc, B, ql = s["c"], c["B"], c["q_len"]
    lens, hd = [c["ctx"] + ql] * B, c["hidden"]
    qkv = lin(_exact_quant(s["x"][:B * ql].to(F64)), s["w"]["qkv"])[0].half().to(F64).view(B, ql, -1, lc["D"])
    nq, nkv = hd // lc["D"], c["kv"] // lc["D"]
    # The graphs are warmed up at b_max sequences, whose tokens the caches then hold; the slots
    # of sequences at or past B hold those of that pass.
    every = lin(_exact_quant(s["x"].to(F64)), s["w"]["qkv"])[0].half().to(F64).view(c["b_max"], ql, -1, lc["D"])
    _exact_append([every[:, :, nq:nq + nkv], every[:, :, nq + nkv:]], s["kv"], [c["ctx"] + ql] * c["b_max"], ql)
    att = _exact_attention(lc, qkv[:, :, :nq], *s["kv"][:5], lens).reshape(B * ql, hd)
    o = lin(_exact_quant(att.half().to(F64)), s["w"]["o"])[0]
    _, _, h, down = mlp(_exact_quant(o.half().to(F64)))
    return {"att": att, "o": o, "hq": h[0], "hs": h[1], "down": down, "kc": s["kv"][0], "vc": s["kv"][1]}
