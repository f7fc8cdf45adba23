"""The workloads that libqk's speed is judged on, through qwen.haiku_amd/qk.py.

They are what a program does with this library for one hybrid model with
Gated DeltaNet layers: decode steps of one token, the LM head with its pick,
prefill of short, ordinary and long prompts, and the host seam. Matrix
types per projection, the widths (hidden 1024, FFN 3584, 16 heads of 128,
vocabulary 248320) and the weight distribution are those of
qwen.haiku_amd/host/qwen_e2e.c; the samplers are bench.py's.

A program that decodes, or that prefills in chunks of one length, captures
its launches once in a HIP graph and replays it, as bench.py does: cases
with "graph" true hold that graph and a pass replays it. A long prompt, or
a whole one at once, is run eagerly: one library call after another.
"""
import ctypes as C
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _binding():
    if "qk_binding" not in sys.modules:
        spec = importlib.util.spec_from_file_location("qk_binding", os.path.join(ROOT, "qwen.haiku_amd", "qk.py"))
        mod = importlib.util.module_from_spec(spec)
        sys.modules["qk_binding"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["qk_binding"]


qk = _binding()
Q8_0, Q4_K, Q5_K, Q6_K = qk.Q8_0, qk.Q4_K, qk.Q5_K, qk.Q6_K
EPS = 1e-6
SAMPLERS = {
    "default": dict(temperature=0.7, top_k=40, top_p=0.9, min_p=0.05, repetition_penalty=1.25, repetition_window=64),
    "wide": dict(temperature=1.0, top_k=0, top_p=0.95, min_p=0.0, repetition_penalty=1.0, repetition_window=0),
    "long": dict(temperature=0.8, top_k=100, top_p=0.95, min_p=0.02, repetition_penalty=1.1, repetition_window=0),
}
_lib = None


def lib():
    global _lib
    if _lib is None:
        _lib = qk.QK().init(0)
    return _lib


# ---- the cases ------------------------------------------------------------------

def listed():
    return [
        # one decode step's device work in one DeltaNet layer (qk_decode.c):
        # norm, four in-projections, out-projection, norm, FFN
        dict(name="decode_layer", kind="decode", layers=1, hidden=1024, ffn=3584, vocab=0, topk=0, graph=True),
        # a whole decoded token of the 24-layer model: every layer, then the
        # output norm, the LM head, the greedy pick and the 40 best
        dict(name="decode_token", kind="decode", layers=24, hidden=1024, ffn=3584, vocab=248320, topk=40, graph=True),
        # the head alone, greedy with 40 alternatives (a program that shows log-probabilities)
        dict(name="head_greedy", kind="head", hidden=1024, vocab=248320, topk=40, sampler="", history=0, graph=True),
        # the head and the default sampler (top-k 40, nucleus, min-p, penalty over the last 64)
        dict(name="head_sampled", kind="head", hidden=1024, vocab=248320, topk=0, sampler="default", history=512,
             graph=True),
        # the head and the widest sampler (top-k off: 256 slots)
        dict(name="head_sampled_wide", kind="head", hidden=1024, vocab=248320, topk=0, sampler="wide", history=512,
             graph=True),
        # a layer's FFN over a short chat turn, over a prefill chunk, and over a long prompt
        dict(name="ffn_23", kind="ffn", tokens=23, hidden=1024, ffn=3584, graph=True),
        dict(name="ffn_512", kind="ffn", tokens=512, hidden=1024, ffn=3584, graph=True),
        dict(name="ffn_2048", kind="ffn", tokens=2048, hidden=1024, ffn=3584, graph=False),
        # a DeltaNet layer's projections around the mixer, an odd prompt length
        dict(name="mixer_proj_333", kind="proj", tokens=333, hidden=1024, inner=2048, heads=16, graph=True),
        # the chunked DeltaNet of one layer: a short ragged prompt, and 512 tokens
        dict(name="deltanet_100", kind="deltanet", tokens=100, heads=16, kdim=128, vdim=128, graph=True),
        dict(name="deltanet_512", kind="deltanet", tokens=512, heads=16, kdim=128, vdim=128, graph=False),
        # the drop-in: the reference's FFN matmuls of one decode step, host buffers in and out
        dict(name="seam_decode", kind="seam", tokens=1, hidden=1024, ffn=3584),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "head", "ffn", "ffn", "proj", "deltanet", "seam"])
    hidden = 256 * rng.randint(2, 10)
    if kind == "decode":
        return dict(kind=kind, layers=rng.randint(1, 3), hidden=hidden, ffn=256 * rng.randint(8, 28),
                    vocab=rng.choice([0, _log(rng, 2000, 150000)]), topk=rng.choice([0, 1, 40, 200]), graph=True)
    if kind == "head":
        hidden = 256 * rng.randint(2, 5)
        sampler = rng.choice(["", "default", "wide", "long"])
        return dict(kind=kind, hidden=hidden, vocab=_log(rng, 5000, 200000),
                    topk=0 if sampler else rng.randint(1, 256), sampler=sampler, history=_log(rng, 10, 2000),
                    graph=True)
    if kind == "ffn":
        return dict(kind=kind, tokens=_log(rng, 2, 1500), hidden=256 * rng.randint(2, 4), ffn=256 * rng.randint(6, 14),
                    graph=rng.random() < 0.6)
    if kind == "proj":
        return dict(kind=kind, tokens=_log(rng, 2, 1000), hidden=256 * rng.randint(2, 5), inner=256 * rng.randint(4, 9),
                    heads=rng.choice([8, 16, 24]), graph=rng.random() < 0.6)
    if kind == "deltanet":
        return dict(kind=kind, tokens=_log(rng, 3, 500), heads=rng.randint(4, 16), kdim=rng.choice([64, 96, 128]),
                    vdim=rng.choice([64, 128]), graph=rng.random() < 0.6)
    return dict(kind=kind, tokens=_log(rng, 1, 64), hidden=256 * rng.randint(2, 6), ffn=256 * rng.randint(6, 14))


# ---- inputs -----------------------------------------------------------------------

class Draws:
    """Seeded inputs on the GPU, drawn in one order by prepare() and exact()."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(self, *shape):
        return torch.randn(*shape, device="cuda", generator=self.g)

    def ints(self, lo, hi, *shape):
        return torch.randint(lo, hi + 1, shape, device="cuda", generator=self.g)

    def f16(self, n, scale):
        jitter = 0.75 + 0.5 * torch.rand(n, device="cuda", generator=self.g)
        return (scale * jitter).to(torch.float16)

    def norm_weight(self, k):
        return 1.0 + 0.02 * self.normal(k)

    def matrix(self, wtype, n, k, gain=1.0):
        """n rows of k/256 (k/32) GGUF blocks whose weights have mean about 0
        and standard deviation about gain / sqrt(k)."""
        sigma = gain / math.sqrt(k)
        if wtype == Q8_0:
            nb = n * (k // 32)
            d = self.f16(nb, sigma / 73.0).view(torch.uint8).view(nb, 2)
            q = self.ints(-127, 127, nb, 32).to(torch.int8).view(torch.uint8)
            return torch.cat([d, q], 1).reshape(n, -1).contiguous()
        nb = n * (k // 256)
        low = self.ints(0, 255, nb, 128).to(torch.uint8)
        if wtype == Q6_K:
            high = self.ints(0, 255, nb, 64).to(torch.uint8)
            sc = self.ints(-32, 31, nb, 16).to(torch.int8).view(torch.uint8)
            d = self.f16(nb, sigma / 340.0).view(torch.uint8).view(nb, 2)
            return torch.cat([low, high, sc, d], 1).reshape(n, -1).contiguous()
        # 6-bit scales over the upper two thirds of their range, mins at the
        # middle of the quants: w = d * sc * (q - mid)
        mid, unit = (7.5, 200.0) if wtype == Q4_K else (15.5, 400.0)
        sc = self.ints(20, 63, nb, 8).to(torch.uint8)
        mn = sc
        d = self.f16(nb, sigma / unit)
        dmin = (d.float() * mid).to(torch.float16)
        packed = torch.cat([(sc[:, :4] & 63) | ((sc[:, 4:] >> 4) << 6), (mn[:, :4] & 63) | ((mn[:, 4:] >> 4) << 6),
                            (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)], 1)
        parts = [d.view(torch.uint8).view(nb, 2), dmin.view(torch.uint8).view(nb, 2), packed]
        if wtype == Q5_K:
            parts.append(self.ints(0, 255, nb, 32).to(torch.uint8))
        return torch.cat(parts + [low], 1).reshape(n, -1).contiguous()


def _in_proj(hidden, inner, heads):
    """The four in-projections of a DeltaNet layer (type, rows)."""
    return [(Q5_K, 3 * inner), (Q4_K, inner), (Q8_0, heads), (Q8_0, heads)]


def _decode_inputs(case, seed):
    r, H, F = Draws(seed), case["hidden"], case["ffn"]
    d = dict(h=r.normal(1, H), layers=[])
    for _ in range(case["layers"]):
        d["layers"].append(dict(
            norm=r.norm_weight(H), ffn_norm=r.norm_weight(H),
            proj=[(t, n, r.matrix(t, n, H)) for t, n in _in_proj(H, 2048, 16)],
            mixed=0.5 * r.normal(1, 2048), out=r.matrix(Q5_K, H, 2048, 0.5),
            gate=r.matrix(Q4_K, F, H), up=r.matrix(Q4_K, F, H), down=r.matrix(Q6_K, H, F, 0.5)))
    if case["vocab"]:
        d["out_norm"], d["head"] = r.norm_weight(H), r.matrix(Q6_K, case["vocab"], H, 3.0)
    return d


def _head_inputs(case, seed):
    r, H, V = Draws(seed), case["hidden"], case["vocab"]
    d = dict(x=r.normal(1, H), head=r.matrix(Q6_K, V, H, 3.0))
    if case["sampler"]:
        d["history"] = r.ints(0, V - 1, case["history"]).to(torch.int32)
        d["rng"] = r.ints(1, (1 << 62) - 1, 2)
    return d


def _ffn_inputs(case, seed):
    r, M, H, F = Draws(seed), case["tokens"], case["hidden"], case["ffn"]
    return dict(h=r.normal(M, H), mix=0.5 * r.normal(M, H), norm=r.norm_weight(H), gate=r.matrix(Q4_K, F, H),
                up=r.matrix(Q4_K, F, H), down=r.matrix(Q6_K, H, F, 0.5))


def _proj_inputs(case, seed):
    r, M, H = Draws(seed), case["tokens"], case["hidden"]
    return dict(h=r.normal(M, H), prev=0.5 * r.normal(M, H), norm=r.norm_weight(H),
                proj=[(t, n, r.matrix(t, n, H)) for t, n in _in_proj(H, case["inner"], case["heads"])],
                mixed=0.5 * r.normal(M, case["inner"]), out=r.matrix(Q5_K, H, case["inner"], 0.5))


def _deltanet_inputs(case, seed):
    r, n, H, kd, vd = Draws(seed), case["tokens"], case["heads"], case["kdim"], case["vdim"]
    unit = torch.nn.functional.normalize
    return dict(q=unit(r.normal(n, H, kd), dim=2) / math.sqrt(kd), k=unit(r.normal(n, H, kd), dim=2),
                v=torch.nn.functional.silu(r.normal(n, H, vd)), g=-torch.nn.functional.softplus(r.normal(n, H)),
                beta=torch.sigmoid(r.normal(n, H)), state=0.05 * r.normal(H, kd, vd))


def _seam_inputs(case, seed):
    r, M, H, F = Draws(seed), case["tokens"], case["hidden"], case["ffn"]
    d = dict(x=r.normal(M, H), act=r.normal(M, F), gate=r.matrix(Q4_K, F, H), up=r.matrix(Q4_K, F, H),
             down=r.matrix(Q6_K, H, F, 0.5))
    return {k: v.cpu().numpy() for k, v in d.items()}


# ---- what a program keeps, and one pass -----------------------------------------------

def _f32(*shape):
    return torch.empty(*shape, dtype=torch.float32, device="cuda")


def _q8k(m, k):
    return torch.empty(m, (k // 256) * qk.Q8K_BYTES, dtype=torch.uint8, device="cuda")


def _decode(case, seed):
    L, d, H, F, layers = lib(), _decode_inputs(case, seed), case["hidden"], case["ffn"], case["layers"]
    gate, up, xq, aq, x, mix = _f32(F), _f32(F), _q8k(1, H), _q8k(1, F), _f32(1, H), _f32(1, H)
    rows = [n for _, n, _ in d["layers"][0]["proj"]]
    proj, h_in, h_out, ffn = _f32(layers, sum(rows)), _f32(1, H), _f32(layers, H), _f32(layers, H)
    h_last, logits = _f32(1, H), _f32(max(1, case["vocab"]))

    def step():
        h, delta = d["h"], None
        for i, w in enumerate(d["layers"]):
            h_i, f_i = h_out[i:i + 1], ffn[i:i + 1]
            L.add_rmsnorm_q8k(h, delta, w["norm"], EPS, h_out=h_in, x_out=x)
            L.matvec_group_f32([(t, m, n, H, x, y) for (t, n, m), y in zip(w["proj"], proj[i].split(rows))])
            # (the mixer between its projections runs in the caller's own code)
            L.matvec_group_f32([(Q5_K, w["out"], H, 2048, w["mixed"], mix)])
            L.add_rmsnorm_q8k(h_in, mix, w["ffn_norm"], EPS, h_out=h_i, xq=xq)
            L.matvec_group([(Q4_K, w["gate"], F, H, xq, gate), (Q4_K, w["up"], F, H, xq, up)])
            L.swiglu_q8k(gate.view(1, F), up.view(1, F), xq=aq)
            L.matvec(Q6_K, w["down"], H, F, aq, f_i)
            h, delta = h_i, f_i
        if not case["vocab"]:
            return [proj, h_out, ffn]
        L.add_rmsnorm_q8k(h, delta, d["out_norm"], EPS, h_out=h_last, xq=xq)
        return [proj, h_out, ffn, h_last] + list(L.lmhead(d["head"], case["vocab"], H, xq, case["topk"], logits=logits))

    return step, []


def _head(case, seed):
    L, d, H, V = lib(), _head_inputs(case, seed), case["hidden"], case["vocab"]
    logits, xq = _f32(V), L.quantize_q8k(d["x"])

    def step():
        if not case["sampler"]:
            return list(L.lmhead(d["head"], V, H, xq, case["topk"], logits=logits))
        L.lmhead(d["head"], V, H, xq, 0, logits=logits)
        token = L.sample(logits, SAMPLERS[case["sampler"]], d["rng"], d["history"])
        return [logits, token, d["rng"]]

    return step, [d["rng"]] if case["sampler"] else []


def _ffn(case, seed):
    L, d, M, H, F = lib(), _ffn_inputs(case, seed), case["tokens"], case["hidden"], case["ffn"]
    h, xq, gate, up, aq, y = _f32(M, H), _q8k(M, H), _f32(M, F), _f32(M, F), _q8k(M, F), _f32(M, H)
    # as the host seam keeps them: Q6_K repacked for prefill, Q4_K in its blocks
    planes = L.pack_planes(Q6_K, d["down"], H, F)

    def step():
        L.add_rmsnorm_q8k(d["h"], d["mix"], d["norm"], EPS, h_out=h, xq=xq)
        L.matmul(Q4_K, d["gate"], F, H, xq, M, gate)
        L.matmul(Q4_K, d["up"], F, H, xq, M, up)
        L.swiglu_q8k(gate, up, xq=aq)
        L.matmul_planes(Q6_K, planes, H, F, aq, M, y)
        return [h, y]

    return step, []


def _proj(case, seed):
    L, d, M, H, inner = lib(), _proj_inputs(case, seed), case["tokens"], case["hidden"], case["inner"]
    h, x, xq, x0 = _f32(M, H), _f32(M, H), _q8k(M, H), torch.empty(M, (H // 32) * 34, dtype=torch.uint8, device="cuda")
    mq, y = _q8k(M, inner), _f32(M, H)
    weights = [(t, n, L.pack_planes(t, m, n, H) if t == Q5_K else m, _f32(M, n)) for t, n, m in d["proj"]]
    out = L.pack_planes(Q5_K, d["out"], H, inner)

    def step():
        L.add_rmsnorm_q8k(d["h"], d["prev"], d["norm"], EPS, h_out=h, x_out=x, xq=xq)
        L.quantize_q8_0(x, x0)
        for t, n, w, b in weights:
            if t == Q5_K:
                L.matmul_planes(t, w, n, H, xq, M, b)
            else:
                L.matmul(t, w, n, H, x0 if t == Q8_0 else xq, M, b)
        L.quantize_q8k(d["mixed"], mq)
        L.matmul_planes(Q5_K, out, H, inner, mq, M, y)
        return [h] + [b for _, _, _, b in weights] + [y]

    return step, []


def _deltanet(case, seed):
    L, d = lib(), _deltanet_inputs(case, seed)
    out = _f32(case["tokens"], case["heads"], case["vdim"])

    def step():
        L.deltanet_chunked(d["q"], d["k"], d["v"], d["g"], d["beta"], d["state"], out)
        return [out, d["state"]]

    return step, [d["state"]]


class Seam:
    """Host weights registered with the library for as long as they live."""

    def __init__(self, case, seed):
        self.L, self.d, self.H, self.F = lib(), _seam_inputs(case, seed), case["hidden"], case["ffn"]
        for name, t, n, k in self.weights():
            self.L.register_weight(self.d[name], t, k, n)

    def weights(self):
        return ("gate", Q4_K, self.F, self.H), ("up", Q4_K, self.F, self.H), ("down", Q6_K, self.H, self.F)

    def __call__(self):
        return [self.L.matmul_host(t, self.d[name], n, k, self.d["act" if name == "down" else "x"])
                for name, t, n, k in self.weights()]

    def __del__(self):
        for name, *_ in self.weights():
            self.L.unregister_weight(self.d[name])


_capture_stream = None


class Captured:
    """step's launches in a HIP graph: an eager pass first, so that the
    library's scratch of that stream exists before the capture. The tensors
    that a pass carries on to the next get their first values back. Keeps
    step, and with it every buffer that the graph points at."""

    def __init__(self, step, carried):
        global _capture_stream
        if _capture_stream is None:
            _capture_stream = torch.cuda.Stream()
        s = _capture_stream
        first = [t.clone() for t in carried]
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            step()
            for t, v in zip(carried, first):
                t.copy_(v)
        s.synchronize()
        self.step, self.graph = step, torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph, stream=s):
            self.outputs = step()
        torch.cuda.current_stream().wait_stream(s)

    def __call__(self):
        self.graph.replay()
        return self.outputs


def prepare(case, seed):
    if case["kind"] == "seam":
        return Seam(case, seed)
    build = dict(decode=_decode, head=_head, ffn=_ffn, proj=_proj, deltanet=_deltanet)[case["kind"]]
    step, carried = build(case, seed)
    return Captured(step, carried) if case["graph"] else step


def run(state):
    return state()


# ---- what a pass cannot do without ------------------------------------------------------

def work(case):
    k = case["kind"]
    H, F, V, M = case.get("hidden"), case.get("ffn"), case.get("vocab"), case.get("tokens", 1)
    if k == "deltanet":
        heads, kd, vd = case["heads"], case["kdim"], case["vdim"]
        per = heads * (2 * kd + 2 * vd + 2)                    # q, k, v, out, g, beta of a token
        # of a token and head: the state decayed, read by k, updated, read by q
        return dict(bytes=4 * (M * per + 2 * heads * kd * vd), flops=7 * M * heads * kd * vd)
    mats, floats, layers = [], 0, 1
    if k == "decode":
        layers = case["layers"]
        mats = [(t, n, H) for t, n in _in_proj(H, 2048, 16)]
        mats += [(Q5_K, H, 2048), (Q4_K, F, H), (Q4_K, F, H), (Q6_K, H, F)]
        floats = 2048 + 2 * H + 2 * H + sum(n for _, n in _in_proj(H, 2048, 16))
    elif k == "ffn":
        mats, floats = [(Q4_K, F, H), (Q4_K, F, H), (Q6_K, H, F)], M * 4 * H + H
    elif k == "proj":
        ins = _in_proj(H, case["inner"], case["heads"])
        mats = [(t, n, H) for t, n in ins] + [(Q5_K, H, case["inner"])]
        floats = M * (4 * H + case["inner"] + sum(n for _, n in ins)) + H
    elif k == "seam":
        mats, floats = [(Q4_K, F, H), (Q4_K, F, H), (Q6_K, H, F)], M * (2 * H + 3 * F)
    nbytes = layers * (sum(n * qk.row_bytes(t, kk) for t, n, kk in mats) + 4 * floats)
    flops = layers * 2 * M * sum(n * kk for _, n, kk in mats)
    if V:
        nbytes += V * qk.row_bytes(Q6_K, H) + 4 * (V + H)
        flops += 2 * V * H
    return dict(bytes=nbytes, flops=flops)


def tolerance(case):
    # the library's contract: every result is the reference's bit for bit
    # (the integer sums are exact, each float operation has its place in one order)
    return "exact"


# ---- the same in 64 bits -----------------------------------------------------------------

def _dequant(wtype, raw, n, k):
    """(n, k) float64 weights of GGUF blocks."""
    b = raw.reshape(-1, qk.BLOCK_BYTES[wtype])

    def half(at):
        return b[:, at:at + 2].contiguous().view(torch.float16).to(torch.float64)

    if wtype == Q8_0:
        return (half(0) * b[:, 2:].contiguous().view(torch.int8).double()).reshape(n, k)
    if wtype == Q6_K:
        low, high = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 1, 32)
        nib = torch.cat([low & 15, low >> 4], 2)               # (halves, 4 runs, 32)
        two = torch.cat([(high >> s) & 3 for s in (0, 2, 4, 6)], 2)
        q = (nib | (two << 4)).to(torch.int32) - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double().repeat_interleave(16, 1)
        return (half(208) * sc * q.reshape(-1, 256).double()).reshape(n, k)
    p = b[:, 4:16]
    sc = torch.cat([p[:, :4] & 63, (p[:, 8:] & 15) | ((p[:, :4] >> 6) << 4)], 1).double().repeat_interleave(32, 1)
    mn = torch.cat([p[:, 4:8] & 63, (p[:, 8:] >> 4) | ((p[:, 4:8] >> 6) << 4)], 1).double().repeat_interleave(32, 1)
    low = b[:, -128:].reshape(-1, 4, 1, 32)
    q = torch.cat([low & 15, low >> 4], 2).reshape(-1, 8, 32)
    if wtype == Q5_K:
        bits = torch.stack([(b[:, 16:48] >> s) & 1 for s in range(8)], 1)
        q = q | (bits << 4)
    return (half(0) * sc * q.reshape(-1, 256).double() - half(2) * mn).reshape(n, k)


def _rounded(x, wtype):
    """x as the product sees it: quantized to int8 per block of 256 (32 beside Q8_0)."""
    size = 32 if wtype == Q8_0 else 256
    v = x.reshape(-1, size)
    if wtype == Q8_0:
        d = v.abs().amax(1, keepdim=True) / 127.0
        q = torch.where(d > 0, v / d, torch.zeros_like(v))
        q = torch.sign(q) * torch.floor(q.abs() + 0.5)
        d = d.to(torch.float16).double()
    else:
        top = v.gather(1, v.abs().argmax(1, keepdim=True))
        d = top / -127.0
        q = torch.where(d != 0, v / d, torch.zeros_like(v)).round().clamp(max=127)
    return (q * d).reshape(x.shape)


def _mm(wtype, raw, n, k, x):
    w = _dequant(wtype, raw, n, k)
    return _rounded(x, wtype) @ w.t()


def _rms(h, w):
    return h / torch.sqrt((h * h).mean(1, keepdim=True) + EPS) * w.double()


def _silu(x):
    return x / (1.0 + torch.exp(-x))


def _exact_ffn(d, h, H, F):
    x = _rms(h, d.get("ffn_norm", d.get("norm")))
    act = _silu(_mm(Q4_K, d["gate"], F, H, x)) * _mm(Q4_K, d["up"], F, H, x)
    return _mm(Q6_K, d["down"], H, F, act)


def _exact_decode(case, seed):
    d, H, F, V = _decode_inputs(case, seed), case["hidden"], case["ffn"], case["vocab"]
    h, proj, h_out, ffn = d["h"].double(), [], [], []
    for w in d["layers"]:
        x = _rms(h, w["norm"])
        proj.append(torch.cat([_mm(t, m, n, H, x) for t, n, m in w["proj"]], 1))
        h_out.append(h + _mm(Q5_K, w["out"], H, 2048, w["mixed"].double()))
        ffn.append(_exact_ffn(w, h_out[-1], H, F))
        h = h_out[-1] + ffn[-1]
    outs = [torch.cat(v) for v in (proj, h_out, ffn)]
    if not V:
        return outs
    logits = _mm(Q6_K, d["head"], V, H, _rms(h, d["out_norm"])).reshape(-1)
    return outs + [h, logits, None, None, logits.topk(case["topk"])[0] if case["topk"] else None]


def _exact_head(case, seed):
    d, H, V = _head_inputs(case, seed), case["hidden"], case["vocab"]
    logits = _mm(Q6_K, d["head"], V, H, d["x"].double()).reshape(-1)
    if not case["sampler"]:
        return [logits, None, None, logits.topk(case["topk"])[0]]
    sp = SAMPLERS[case["sampler"]]
    window = sp["repetition_window"] or case["history"]
    p = float(np.float32(sp["repetition_penalty"]))
    if p != 1.0:
        for i in d["history"][-window:].tolist():              # each occurrence penalizes once more
            logits[i] = logits[i] / p if logits[i] > 0 else logits[i] * p
    return [logits, None, None]


def _exact_deltanet(case, seed):
    d = {k: v.double() for k, v in _deltanet_inputs(case, seed).items()}
    S, outs = d["state"].clone(), []
    for t in range(case["tokens"]):
        S = S * torch.exp(d["g"][t])[:, None, None]
        err = (d["v"][t] - torch.matmul(d["k"][t][:, None, :], S)[:, 0]) * d["beta"][t][:, None]
        S = S + d["k"][t][:, :, None] * err[:, None, :]
        outs.append(torch.matmul(d["q"][t][:, None, :], S)[:, 0])
    return [torch.stack(outs), S]


def exact(case, seed):
    k = case["kind"]
    if k == "decode":
        return _exact_decode(case, seed)
    if k == "head":
        return _exact_head(case, seed)
    if k == "deltanet":
        return _exact_deltanet(case, seed)
    if k == "seam":
        d, H, F = _seam_inputs(case, seed), case["hidden"], case["ffn"]
        d = {name: torch.from_numpy(v).cuda() for name, v in d.items()}
        x, act = d["x"].double(), d["act"].double()
        return [_mm(Q4_K, d["gate"], F, H, x), _mm(Q4_K, d["up"], F, H, x), _mm(Q6_K, d["down"], H, F, act)]
    if k == "ffn":
        d = _ffn_inputs(case, seed)
        h = d["h"].double() + d["mix"].double()
        return [h, _exact_ffn(d, h, case["hidden"], case["ffn"])]
    d, H, inner = _proj_inputs(case, seed), case["hidden"], case["inner"]
    h = d["h"].double() + d["prev"].double()
    x = _rms(h, d["norm"])
    return [h] + [_mm(t, m, n, H, x) for t, n, m in d["proj"]] + [_mm(Q5_K, d["out"], H, inner, d["mixed"].double())]
