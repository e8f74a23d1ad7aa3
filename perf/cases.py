"""The work that a user of this package has it do, as cases for timing.

    decode-small   a decode step of a small model, call by call: launches and host time count
    decode-step    a decode step of a large model, replayed as a graph (the captured step is the plan a server keeps)
    verify-4       four rows through one layer: the verify step of speculative decoding
    tied-head      the output projection of a model whose embedding is tied: weights as they are on disk
    prompt-45      a short prompt of odd length against the deepest contraction of a layer
    prefill-512    the prompt chunk of the benchmark, Q4_K up projection
    prefill-777    a ragged chunk in Q6_K, the format mixed files keep their down projections in
    prefill-2048   a long chunk in Q8_0: the largest
    moe-1/48/512   the routed experts' FFN for one token, for a small batch, for a prompt chunk
    ingest         loading: GGUF tensor bytes on the host into the layout the kernels read

A case is a dict of plain values; `prepare` makes what a program holds before the call, `run` is one pass."""
import math

import numpy as np
import torch

import reinstinct_amd as rein
from reinstinct_amd import hip, quant, runtime
from reinstinct_amd._lib import init, lib

DENSE = ("q4_0", "q4_k", "q5_k", "q6_k", "q8_0", "iq4_xs", "iq3_s")
FMT = dict(rein.FORMATS, iq3_s=rein.IQ3_S)
DISK = dict(FMT, q3_k=quant.GGML_Q3_K, iq4_nl=quant.GGML_IQ4_NL, bf16=quant.GGML_BF16)
# What a mixed file keeps its value and down projections in, beside the format of the others
MIX = {"q4_k": "q6_k", "q5_k": "q6_k", "q8_0": "q8_0", "iq4_xs": "q5_k", "q4_0": "q4_0"}
MOST_WEIGHTS = 3 << 29         # weights of one case
MOST_WORK = 2 * 2048 * 5120 * 17408


def listed():
    layer = dict(kind="layers", rows=1, layers=1, graph=False, vocab=0)
    return [
        # hidden 2048 against 5632: every launch is a few microseconds
        dict(layer, name="decode-small", hidden=2048, kv=512, ffn=5632, fmt="q4_k"),
        # the 27B-class decoder of the benchmark, eight of its layers and its output head
        dict(layer, name="decode-step", hidden=5120, kv=1024, ffn=17408, fmt="q4_k", layers=8, graph=True, vocab=151936),
        dict(layer, name="verify-4", hidden=4096, kv=1024, ffn=14336, fmt="q5_k", rows=4),
        dict(kind="head", name="tied-head", fmt="q6_k", in_dim=2048, out_dim=151936),
        dict(kind="matmul", name="prompt-45", fmt="q5_k", in_dim=17408, out_dim=5120, rows=45),
        dict(kind="matmul", name="prefill-512", fmt="q4_k", in_dim=5120, out_dim=17408, rows=512),
        dict(kind="matmul", name="prefill-777", fmt="q6_k", in_dim=17408, out_dim=5120, rows=777),
        dict(kind="matmul", name="prefill-2048", fmt="q8_0", in_dim=5120, out_dim=17408, rows=2048),
        # the benchmark's expert FFN: 128 experts, eight of them for each token
        dict(kind="moe", name="moe-1", rows=1, hidden=2048, ffn=768, experts=128, used=8, fmt="q4_k", down="q6_k"),
        dict(kind="moe", name="moe-48", rows=48, hidden=2048, ffn=768, experts=128, used=8, fmt="q4_k", down="q6_k"),
        dict(kind="moe", name="moe-512", rows=512, hidden=2048, ffn=768, experts=128, used=8, fmt="q4_k", down="q6_k"),
        dict(kind="ingest", name="ingest", fmt="q4_k", in_dim=5120, out_dim=17408),
    ]


def _spread(rng, lo, hi, step=1):
    """a multiple of `step` between lo and hi, spread over the logarithm"""
    return min(hi, max(lo, int(math.exp(rng.uniform(math.log(lo), math.log(hi))) + step / 2) // step * step))


def draw(rng):
    while True:
        kind = rng.choice(["matmul"] * 5 + ["layers"] * 3 + ["moe"] * 3 + ["head", "ingest"])
        if kind == "matmul":         # from one row to a long prompt
            case = dict(kind=kind, fmt=rng.choice(DENSE), in_dim=_spread(rng, 1024, 18432, 256), out_dim=_spread(rng, 512, 32768, 32),
                        rows=_spread(rng, 1, 2048))
        elif kind == "layers":
            hidden = _spread(rng, 1024, 8192, 256)
            case = dict(kind=kind, fmt=rng.choice(sorted(MIX)), hidden=hidden, kv=max(128, hidden // rng.choice((1, 4, 8)) // 128 * 128),
                        ffn=_spread(rng, 5 * hidden // 2, 4 * hidden, 256) // 256 * 256, rows=rng.choice((1, 1, 2, 3, 4)),
                        layers=rng.randint(1, 8), graph=rng.random() < 0.5, vocab=rng.choice((0, _spread(rng, 32000, 256000))))
        elif kind == "moe":
            case = dict(kind=kind, rows=_spread(rng, 1, 1024), hidden=_spread(rng, 1024, 4096, 256), ffn=_spread(rng, 256, 1536, 256),
                        experts=rng.choice((32, 64, 128, 256)), used=rng.choice((2, 4, 6, 8)), fmt=rng.choice(("q4_k", "q5_k", "q8_0")),
                        down=rng.choice(("q5_k", "q6_k", "q8_0")))
        elif kind == "head":
            case = dict(kind=kind, fmt=rng.choice(("q4_k", "q5_k", "q6_k", "q8_0")), in_dim=_spread(rng, 1024, 5120, 256),
                        out_dim=_spread(rng, 32000, 256000))
        else:
            case = dict(kind=kind, fmt=rng.choice(sorted(DISK)), in_dim=_spread(rng, 1024, 17408, 256), out_dim=_spread(rng, 1024, 17408, 32))
        most = 5120 * 17408 if kind == "ingest" else MOST_WEIGHTS
        if sum(k * n for _, k, n in _matrices(case)) <= most and work(case)["flops"] <= MOST_WORK:
            return case


# ---- sizes

def _matrices(case):
    """(format, in_dim, out_dim) of every weight matrix"""
    fmt = case["fmt"]
    if case["kind"] == "layers":
        h, kv, ffn, second = case["hidden"], case["kv"], case["ffn"], MIX[fmt]
        layer = [(fmt, h, h), (fmt, h, kv), (second, h, kv), (fmt, h, h), (fmt, h, ffn), (fmt, h, ffn), (second, ffn, h)]
        return layer * case["layers"] + ([("q6_k", h, case["vocab"])] if case["vocab"] else [])
    if case["kind"] == "moe":
        h, ffn = case["hidden"], case["ffn"]
        return [(fmt, h, ffn), (fmt, h, ffn), (case["down"], ffn, h)] * case["experts"]
    return [(fmt, case["in_dim"], case["out_dim"])]


def _disk_bytes(fmt, k, n):
    return int(lib.rein_ingest_src_len(DISK[fmt], k, n))


def work(case):
    kind = case["kind"]
    mats = _matrices(case)
    if kind == "ingest":         # host: the tensor in, the layout out; no arithmetic to speak of
        (fmt, k, n), = mats
        return {"bytes": _disk_bytes(fmt, k, n) + quant.repacked_len(lib.rein_ingest_format(DISK[fmt]), k, n), "flops": 0}
    if kind == "head":
        (fmt, k, n), = mats
        return {"bytes": _disk_bytes(fmt, k, n) + 4 * k + 4 * n, "flops": 2 * k * n}
    weights = {m: quant.repacked_len(FMT[m[0]], m[1], m[2]) for m in set(mats)}
    rows = case["rows"]
    if kind == "moe":
        entries, experts = rows * case["used"], case["experts"]
        per_expert = sum(weights[m] for m in mats[:3])
        touched = experts * (1 - (1 - case["used"] / experts) ** rows)         # of a router that spreads its tokens
        return {"bytes": touched * per_expert + 4 * rows * (2 * case["hidden"] + experts),
                "flops": 2 * entries * sum(k * n for _, k, n in mats[:3])}
    if kind == "matmul":
        outer = sum(4 * rows * (k + n) for _, k, n in mats)
    else:         # in: the embedding, the attention's answers; out: Q, K, V of each layer, the hidden state, the logits
        h, kv = case["hidden"], case["kv"]
        outer = 4 * rows * (2 * h + case["layers"] * (2 * h + 2 * kv) + case["vocab"])
    return {"bytes": sum(weights[m] for m in mats) + outer, "flops": 2 * rows * sum(k * n for _, k, n in mats)}


def tolerance(case):
    if case["kind"] == "ingest":
        return "exact"
    # Dots of whole numbers, scaled and summed in 32-bit floats.  Where a result is quantized to eight bits for the next
    # product, a sum that differs in its last bit may land on the other side of a half step: few values, by 1/127 of their
    # block's largest.
    return {"rel": {"moe": 1e-3, "layers": 2e-3}.get(case["kind"], 1e-5)}


# ---- inputs

def _generator(seed):
    init()
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape, scale=1.0):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * scale


def _bytes(g, *shape):
    return torch.randint(0, 256, shape, generator=g, device="cuda", dtype=torch.uint8)


def _nibbles(g, *shape):
    """bytes of two 4-bit codes each, spread as those of quantized Gaussian weights are: 32 of them span the 16 codes"""
    lo, hi = (_randn(g, *shape).mul_(3.6).add_(7.5).round_().clamp_(0, 15).to(torch.uint8) for _ in range(2))
    return hi.mul_(16).add_(lo)


def _halves(g, *shape, mean, signed=False):
    """fp16 scales within 30 % of `mean`, as bytes"""
    v = (torch.rand(shape, generator=g, device="cuda") * 0.6 + 0.7) * mean
    if signed:
        v *= torch.randint(0, 2, shape, generator=g, device="cuda") * 2 - 1
    return v.to(torch.float16).view(torch.uint8)


def _codes(g, *shape, lo, hi):
    return torch.randint(lo, hi, shape, generator=g, device="cuda").to(torch.uint8)


def _int8(g, *shape, scale):
    return _randn(g, *shape).mul_(scale).round_().clamp_(-127, 127).to(torch.int8).view(torch.uint8)


def _slab(g, fmt, in_dim, out_dim, copies=1):
    """`copies` matrices ~N(0, 0.02) in the layout that the kernels read (quant.repack_for_matvec), made on the GPU: a plane of
    codes, those of extra bits and scales, one entry for each 32 weights, then one for each 256"""
    n_sub, padded, n_super = in_dim // 32, quant.repacked_n_sub_padded(in_dim), in_dim // 256
    sub, sup = (copies, out_dim, padded), (copies, out_dim, n_super)
    if fmt in ("q4_k", "q5_k"):
        levels = 15 if fmt == "q4_k" else 31
        planes = [_nibbles(g, *sub, 16)] + ([_bytes(g, *sub, 4)] if fmt == "q5_k" else []) + [_codes(g, *sub, 2, lo=36, hi=64)]
        supers = [torch.cat([_halves(g, *sup, 1, mean=0.1 / 63 / levels), _halves(g, *sup, 1, mean=0.05 / 63)], -1)]
    elif fmt == "q6_k":
        scales = _codes(g, *sub, 2, lo=72, hi=128) * (torch.randint(0, 2, (*sub, 2), generator=g, device="cuda") * 2 - 1).to(torch.int8)
        planes = [_nibbles(g, *sub, 16), _bytes(g, *sub, 8), scales.to(torch.int8).view(torch.uint8)]
        supers = [_halves(g, *sup, 1, mean=1.2e-5)]
    elif fmt == "q8_0":
        planes, supers = [_int8(g, *sub, 16, scale=60), _int8(g, *sub, 16, scale=60), _halves(g, *sub, 1, mean=3.3e-4)], []
    else:         # a nibble and a signed scale: Q4_0, IQ4_XS, IQ3_S
        mean = {"q4_0": 5e-3, "iq4_xs": 3.7e-4, "iq3_s": 2.8e-3}[fmt]
        planes, supers = [_nibbles(g, *sub, 16), _halves(g, *sub, 1, mean=mean, signed=True)], []
    for p in planes:
        p[:, :, n_sub:] = 0
    slab = torch.cat([p.reshape(copies, -1) for p in planes + supers], 1).contiguous()
    assert slab.shape[1] == quant.repacked_len(FMT[fmt], in_dim, out_dim)
    return slab


def _blocks(g, fmt, in_dim, out_dim):
    """the same as GGUF tensor bytes, on the GPU"""
    n = in_dim * out_dim
    if fmt == "bf16":
        return _randn(g, n, scale=0.02).to(torch.bfloat16).view(torch.uint8)
    b, s = n // 32, n // 256
    fields = {
        "q4_0": lambda: [_halves(g, b, 1, mean=5e-3, signed=True), _nibbles(g, b, 16)],
        "iq4_nl": lambda: [_halves(g, b, 1, mean=3.7e-4, signed=True), _nibbles(g, b, 16)],
        "q8_0": lambda: [_halves(g, b, 1, mean=3.3e-4), _int8(g, b, 32, scale=60)],
        "q4_k": lambda: [_halves(g, s, 1, mean=1e-4), _halves(g, s, 1, mean=8e-4), _bytes(g, s, 12), _nibbles(g, s, 128)],
        "q5_k": lambda: [_halves(g, s, 1, mean=5e-5), _halves(g, s, 1, mean=8e-4), _bytes(g, s, 12), _bytes(g, s, 32), _nibbles(g, s, 128)],
        "q6_k": lambda: [_nibbles(g, s, 128), _bytes(g, s, 64), _int8(g, s, 16, scale=90), _halves(g, s, 1, mean=1.2e-5)],
        "iq4_xs": lambda: [_halves(g, s, 1, mean=2e-5), _bytes(g, s, 6), _nibbles(g, s, 128)],
        "iq3_s": lambda: [_halves(g, s, 1, mean=2e-4), _bytes(g, s, 108)],
        "q3_k": lambda: [_bytes(g, s, 108), _halves(g, s, 1, mean=5e-4)],
    }[fmt]()
    raw = torch.cat(fields, 1).reshape(-1)
    assert raw.numel() == _disk_bytes(fmt, in_dim, out_dim)
    return raw


def _floats(*shape):
    return torch.empty(shape, device="cuda", dtype=torch.float32)


def _room(n_bytes):
    return torch.empty(max(int(n_bytes), 16), device="cuda", dtype=torch.uint8)


def _q8(n):
    return _room(n // 32 * 40)


class _Layers:
    """a decoder's layers without their attention: what it answers is an input here"""

    def __init__(self, case, g):
        self.rows, self.h, self.kv, self.ffn, self.vocab = (case[k] for k in ("rows", "hidden", "kv", "ffn", "vocab"))
        h, kv, ffn, rows = self.h, self.kv, self.ffn, self.rows
        f, second = FMT[case["fmt"]], FMT[MIX[case["fmt"]]]
        self.f, self.down_fmt = f, second
        self.qkv_fmts, self.qkv_dims, self.gu_fmts, self.gu_dims = [f, f, second], [h, kv, kv], [f, f], [ffn, ffn]
        self.embedding, self.attention = _randn(g, rows, h), _randn(g, rows, h)
        self.hidden, self.o, self.down = _floats(rows, h), _floats(rows, h), _floats(rows, h)
        self.gate, self.up = _floats(rows, ffn), _floats(rows, ffn)
        self.xq, self.xq_ffn = _q8(rows * h), _q8(rows * ffn)
        self.layers, self.keep = [], []
        for _ in range(case["layers"]):
            slabs = [_slab(g, n, k, m) for n, k, m in _matrices(dict(case, layers=1, vocab=0))]
            norms = [_randn(g, h, scale=0.1) + 1 for _ in range(2)]
            outs = [_floats(rows, n) for n in self.qkv_dims]
            self.keep.append((slabs, norms, outs))
            w = [s.data_ptr() for s in slabs]
            self.layers.append((norms[0].data_ptr(), w[:3], [o.data_ptr() for o in outs], w[3], norms[1].data_ptr(), w[4:6], w[6]))
        self.outputs = {"qkv": [k[2] for k in self.keep], "hidden": self.hidden, "down": self.down}
        if self.vocab:
            self.head, self.last, self.logits = _slab(g, "q6_k", h, self.vocab), _randn(g, h, scale=0.1) + 1, _floats(rows, self.vocab)
            self.outputs["logits"] = self.logits
        self.p = {k: getattr(self, k).data_ptr() for k in ("embedding", "attention", "hidden", "o", "down", "gate", "up", "xq", "xq_ffn")}
        self.stream = self.graph = None
        if case["graph"]:
            self.stream = hip.Stream()
            torch.cuda.synchronize()
            self.step()
            self.stream.synchronize()
            self.stream.begin_capture()
            self.step()
            self.graph = self.stream.end_capture().instantiate()

    def matvec(self, fmt, w, xq, y, in_dim, out_dim):
        if self.rows == 1:
            runtime.matvec_xq8(fmt, w, xq, y, in_dim, out_dim, self.stream)
        else:
            runtime.matvec_batched_xq8(fmt, w, xq, y, in_dim, out_dim, self.rows, self.stream)

    def step(self):
        p, s, rows, h = self.p, self.stream, self.rows, self.h
        lib.rein_memcpy_d2d_async(p["hidden"], p["embedding"], 4 * rows * h, s.raw if s else None)
        add = None
        for norm, w_qkv, y_qkv, w_o, norm2, w_gu, w_down in self.layers:
            runtime.add_rmsnorm_q8(p["hidden"], add, norm, None, p["xq"], h, rows, 1e-6, s)
            runtime.matvec_multi_xq8(self.qkv_fmts, w_qkv, y_qkv, self.qkv_dims, p["xq"], h, rows, s)
            runtime.quantize_q8(p["attention"], p["xq"], h, rows, s)
            self.matvec(self.f, w_o, p["xq"], p["o"], h, h)
            runtime.add_rmsnorm_q8(p["hidden"], p["o"], norm2, None, p["xq"], h, rows, 1e-6, s)
            runtime.matvec_multi_xq8(self.gu_fmts, w_gu, [p["gate"], p["up"]], self.gu_dims, p["xq"], h, rows, s)
            runtime.swiglu_q8(p["gate"], p["up"], None, p["xq_ffn"], rows * self.ffn, s)
            self.matvec(self.down_fmt, w_down, p["xq_ffn"], p["down"], self.ffn, h)
            add = p["down"]
        if self.vocab:
            runtime.add_rmsnorm_q8(p["hidden"], add, self.last.data_ptr(), None, p["xq"], h, rows, 1e-6, s)
            self.matvec(rein.Q6_K, self.head.data_ptr(), p["xq"], self.logits.data_ptr(), h, self.vocab)

    def run(self):
        if self.graph is not None:
            self.graph.launch(self.stream)
        else:
            self.step()
        return self.outputs


class _Matmul:
    """fp32 rows in, fp32 rows out, with the scratch that a program keeps"""

    def __init__(self, case, g):
        k, n, rows = case["in_dim"], case["out_dim"], case["rows"]
        fmt = FMT[case["fmt"]]
        self.w, self.x, self.y = _slab(g, case["fmt"], k, n), _randn(g, rows, k), _floats(rows, n)
        size = runtime.matmul_scratch_bytes(fmt, k, rows)
        self.scratch = _room(size)
        self.args = (fmt, self.w.data_ptr(), self.x.data_ptr(), self.y.data_ptr(), k, n, rows, self.scratch.data_ptr(), size)

    def run(self):
        runtime.matmul_ws(*self.args)
        return self.y


class _Head:
    def __init__(self, case, g):
        k, n = case["in_dim"], case["out_dim"]
        self.w, self.x, self.xq, self.y = _blocks(g, case["fmt"], k, n), _randn(g, k), _q8(k), _floats(n)
        self.quantize = (self.x.data_ptr(), self.xq.data_ptr(), k)
        self.matvec = (FMT[case["fmt"]], self.w.data_ptr(), self.xq.data_ptr(), self.y.data_ptr(), k, n)

    def run(self):
        runtime.quantize_q8(*self.quantize)
        runtime.matvec_ondisk_xq8(*self.matvec)
        return self.y


class _Moe:
    def __init__(self, case, g):
        rows, h, ffn, experts = (case[k] for k in ("rows", "hidden", "ffn", "experts"))
        self.x, self.logits, self.out = _randn(g, rows, h), _randn(g, rows, experts), _floats(rows, h)
        self.slabs = [_slab(g, f, k, n, experts) for f, k, n in _matrices(dict(case, experts=1))]
        self.scale = torch.ones(experts, device="cuda")
        shape = runtime.moe_shape(rows, h, experts, case["used"], ffn, FMT[case["fmt"]], FMT[case["down"]])
        self.workspace = _room(runtime.moe_workspace_bytes(shape))
        self.args = (shape, self.x.data_ptr(), self.logits.data_ptr(), *(s.data_ptr() for s in self.slabs), self.scale.data_ptr(),
                     self.workspace.data_ptr(), self.out.data_ptr())

    def run(self):
        runtime.moe_ffn(*self.args)
        return self.out


class _Ingest:
    def __init__(self, case, g):
        raw = _blocks(g, case["fmt"], case["in_dim"], case["out_dim"]).cpu().numpy()
        self.args = (DISK[case["fmt"]], np.ascontiguousarray(raw), case["in_dim"], case["out_dim"])

    def run(self):
        slab, fmt = quant.ingest_for_matvec(*self.args)
        return {"slab": slab, "format": fmt}


def prepare(case, seed):
    kind = {"layers": _Layers, "matmul": _Matmul, "head": _Head, "moe": _Moe, "ingest": _Ingest}[case["kind"]]
    state = kind(case, _generator(seed))
    torch.cuda.synchronize()
    return state


def run(state):
    return state.run()
