"""The work a user of this framework has it do, as cases that can be timed and compared.

A pass is what a program runs between two of its own decisions: one projection, one token of a
single-sequence decode, one token of every sequence of a batch, one chunk of a prompt.  It goes through
the Python binding (``jitllm_amd.projections``) on a torch stream, eagerly, over weights that lie on the
device as GGUF blocks; attention is not part of the framework, so what attention would hand to a
layer's output projection is an input.  ``listed()`` names the cases, ``draw()`` gives more of the same
ranges: the same four kinds of pass over model-like widths, row counts from 1 to 2048 and weight types
as files hold them.

Widths are those of the models that bench.py, the tests and the documents of this repository name; block scales are chosen so
that weights have a standard deviation near 0.03, as trained ones do, and activations are normal.
"""
from __future__ import annotations

import ctypes as C
import math

import torch

from jitllm_amd import _lib as L
from jitllm_amd.ggml import GGMLType
from jitllm_amd.projections import QuantizedBatchProjections, QuantizedProjections, TornadoWorkspace
from jitllm_amd.runtime import Context, FloatArray, HalfFloatArray, TornadoTensor

EPS = 1e-5

# dim, hidden, width of k and of v, layers, vocabulary
WIDTHS = {
    "0.5B": (896, 4864, 128, 24, 151936),    # the smallest Qwen2.5
    "1B": (2048, 8192, 512, 16, 128256),     # Llama-3.2-1B
    "3B": (3072, 8192, 1024, 28, 128256),    # Llama-3.2-3B
    "7B-a": (3584, 18944, 512, 28, 151936),  # Qwen2.5-7B
    "7B-b": (4096, 11008, 4096, 32, 32000),  # Llama-2-7B
    "8B-a": (4096, 14336, 1024, 32, 128256), # Llama-3-8B
    "8B-b": (4096, 12288, 1024, 36, 151936), # Qwen3-8B-like
    "14B": (5120, 13824, 1024, 48, 151936),  # Qwen2.5-14B
}

# what one type of file holds: (most tensors, v and down of every second layer, the vocabulary projection)
FILES = {
    "Q8_0": (GGMLType.Q8_0, GGMLType.Q8_0, GGMLType.Q8_0),
    "Q4_0": (GGMLType.Q4_0, GGMLType.Q4_0, GGMLType.Q6_K),
    "Q4_K": (GGMLType.Q4_K, GGMLType.Q4_K, GGMLType.Q4_K),
    "Q4_K_M": (GGMLType.Q4_K, GGMLType.Q6_K, GGMLType.Q6_K),
}


def _model(name, kind, widths, file, layers=None, rows=1, batch=None, half=False, resident=False, vocabulary=True):
    dim, hidden, kv, all_layers, vocab = WIDTHS[widths]
    return {"name": name, "kind": kind, "dim": dim, "hidden": hidden, "kv": kv, "layers": layers or all_layers,
            "vocab": vocab if vocabulary else 0, "file": file, "rows": rows, "batch": batch or rows, "half": half,
            "resident": resident}


def listed():
    return [
        # a single projection, the smallest unit of work: a call and a launch (a gate matrix of Llama-3.2-3B)
        {"name": "projection_8192_q8_0", "kind": "projection", "type": "Q8_0", "d": 8192, "n": 3072},
        # one greedy token, normalisations folded in: a small model, where every launch is short ...
        _model("token_0.5b_q8_0", "token", "0.5B", "Q8_0"),
        # ... the model the benchmark is quoted on ...
        _model("token_1b_q8_0", "token", "1B", "Q8_0"),
        # ... and the usual 4-bit files of 7-8 B models, one with rows of awkward length and mixed types
        _model("token_8b_q4_0", "token", "8B-a", "Q4_0"),
        _model("token_7b_q4_k_m", "token", "7B-a", "Q4_K_M"),
        # one token of every sequence of a batch: few and many sequences, fp32 activations as the
        # reference's batched decode passes them and fp16 ones as its batched plan does
        _model("batch_8_8b_q4_k", "batch", "8B-b", "Q4_K", rows=8),
        _model("batch_29_8b_q4_0", "batch", "8B-a", "Q4_0", rows=29, batch=32, half=True),
        _model("batch_64_1b_q8_0", "batch", "1B", "Q8_0", rows=64),
        # a prompt, or the chunk of one: a short odd one, the benchmark's 512 tokens over fp32 activations with
        # weights decoded on every call, and 2048 tokens with a kept fp16 copy
        _model("prompt_201_7b_q4_k_m", "prompt", "7B-b", "Q4_K_M", layers=8, rows=201, batch=256, half=True, vocabulary=False),
        _model("prompt_512_1b_q8_0", "prompt", "1B", "Q8_0", rows=512, vocabulary=False),
        _model("prompt_2048_1b_q8_0_kept", "prompt", "1B", "Q8_0", rows=2048, half=True, resident=True, vocabulary=False),
        _model("prompt_2048_8b_q4_k", "prompt", "8B-b", "Q4_K", layers=8, rows=2048, vocabulary=False),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


# no drawn case reads more weights or multiplies more than these (token_8b_q4_0 and prompt_2048_8b_q4_k)
MOST_BYTES, MOST_FLOPS = 4.4e9, 6.8e12


def draw(rng):
    kind = rng.choice(("projection", "token", "token", "batch", "batch", "prompt", "prompt"))
    if kind == "projection":
        return {"kind": kind, "type": rng.choice(("Q8_0", "Q4_0", "Q4_K", "Q6_K", "Q5_K", "Q4_1", "Q5_0", "IQ4_XS")),
                "d": int(_log(rng, 512, 32768)), "n": 256 * int(_log(rng, 4, 57))}
    file = rng.choice(tuple(FILES))
    if rng.random() < 0.6:
        dim, hidden, kv, layers, vocab = WIDTHS[rng.choice([k for k in WIDTHS if k != "0.5B" or file == "Q8_0"])]
    else:
        dim = 256 * int(_log(rng, 4, 21))
        hidden = 256 * int(dim / 256 * rng.uniform(2.5, 4))
        kv = dim // rng.choice((1, 4, 8)) // 64 * 64
        layers, vocab = rng.randint(8, 40), 64 * rng.randint(500, 2400)
    rows = {"token": 1, "batch": int(_log(rng, 2, 65)), "prompt": int(_log(rng, 65, 2049))}[kind]
    half = kind != "token" and rng.random() < 0.5
    case = {"kind": kind, "dim": dim, "hidden": hidden, "kv": kv, "layers": layers if kind != "prompt" else rng.randint(2, 8),
            "vocab": vocab if kind != "prompt" else 0, "file": file, "rows": rows,
            "batch": rows if kind == "token" or rng.random() < 0.5 else -(-rows // 64) * 64, "half": half,
            "resident": kind == "prompt" and rng.random() < 0.4}
    while case["layers"] > 1 and (_weight_bytes(case) > MOST_BYTES or work(case)["flops"] > MOST_FLOPS):
        case["layers"] -= 1
    return case


# ---- what a program has in hand ------------------------------------------------------------------

_context = None


def context() -> Context:
    """The program's one context, on a torch stream that is made the current one."""
    global _context
    if _context is None:
        stream = torch.cuda.Stream()
        torch.cuda.set_stream(stream)
        _context = Context(torch.cuda.current_device(), stream=stream.cuda_stream)
        _context.torch_stream = stream
    return _context


class Floats(FloatArray):
    """A FloatArray over memory of a torch tensor."""

    def __init__(self, ctx, tensor):
        assert tensor.dtype == torch.float32 and tensor.is_contiguous()
        self.ctx, self.tensor, self.ptr = ctx, tensor, C.c_void_p(tensor.data_ptr())
        self.size, self.nbytes = tensor.numel(), tensor.numel() * 4

    def free(self):
        self.tensor = self.ptr = None


class Halves(HalfFloatArray):
    """A HalfFloatArray over memory of a torch tensor."""

    def __init__(self, ctx, tensor):
        assert tensor.dtype == torch.float16 and tensor.is_contiguous()
        self.ctx, self.tensor, self.ptr = ctx, tensor, C.c_void_p(tensor.data_ptr())
        self.size, self.nbytes = tensor.numel(), tensor.numel() * 2

    free = Floats.free


class Tokens:
    """One token id on the device."""

    def __init__(self, tensor):
        self.tensor, self.ptr = tensor, C.c_void_p(tensor.data_ptr())


def _f16_field(raw, at, gen, lo, hi):
    d = torch.empty(raw.shape[0], device="cuda").uniform_(lo, hi, generator=gen)
    raw[:, at:at + 2] = d.to(torch.float16).view(torch.uint8).view(-1, 2)


def _blocks(t, rows, cols, gen):
    """Random GGUF blocks of a [rows x cols] weight: quants uniform, block scales as in the module text."""
    n = rows * (cols // t.block_elems)
    raw = torch.randint(0, 256, (n * t.block_bytes,), dtype=torch.uint8, device="cuda", generator=gen).view(n, t.block_bytes)
    if t == GGMLType.Q8_0:
        raw[:, 2:].clamp_(max=254)          # the quantiser's range is symmetric: -128 does not occur ...
        raw[:, 2:].sub_(127)                # ... -127 .. 127 as bytes
        _f16_field(raw, 0, gen, 1e-4, 6e-4)
    elif t == GGMLType.Q4_0:
        low, high = raw[:, 2:] & 15, raw[:, 2:] >> 4
        # 1 .. 15, evenly to both sides of 8: a bias of the weights would add up over the layers
        raw[:, 2:] = (low + 8 * (low == 0)) | ((high + 8 * (high == 0)) << 4)
        _f16_field(raw, 0, gen, 2e-3, 1e-2)
    elif t == GGMLType.Q5_0:
        _f16_field(raw, 0, gen, 1e-3, 5e-3)
    elif t == GGMLType.Q4_1:
        _f16_field(raw, 0, gen, 2e-3, 1e-2)
        _f16_field(raw, 2, gen, -7e-2, -2e-2)
    elif t == GGMLType.Q4_K:
        _f16_field(raw, 0, gen, 5e-5, 2e-4)
        _f16_field(raw, 2, gen, 4e-4, 1.5e-3)
    elif t == GGMLType.Q5_K:
        _f16_field(raw, 0, gen, 2.5e-5, 1e-4)
        _f16_field(raw, 2, gen, 4e-4, 1.5e-3)
    elif t == GGMLType.Q6_K:
        _f16_field(raw, 208, gen, 1e-5, 3e-5)
    else:
        _f16_field(raw, 0, gen, 1e-5, 5e-5)
    return raw.view(-1)


class Weight(TornadoTensor):
    """A weight whose blocks are a torch tensor's memory (jl_weight_wrap)."""

    def __init__(self, ctx, t, rows, cols, gen):
        self.blocks = _blocks(t, rows, cols, gen)
        h = C.c_void_p()
        L.check(ctx._lib.jl_weight_wrap(ctx.handle, int(t), C.c_void_p(self.blocks.data_ptr()), rows, cols, C.byref(h)))
        self.ctx, self.ggml_type, self.rows, self.cols, self.handle, self.nbytes = ctx, t, rows, cols, h, self.blocks.numel()


class Layer:
    pass


class State:
    pass


def prepare(case, seed):
    ctx = context()
    gen = torch.Generator(device="cuda").manual_seed(seed)
    s = State()
    s.kind, s.ctx = case["kind"], ctx

    def floats(*shape, scale=None):
        t = torch.zeros(shape, device="cuda") if scale is None else torch.randn(shape, device="cuda", generator=gen) * scale
        return Floats(ctx, t)

    def activations(*shape, scale=None):
        a = floats(*shape, scale=scale)
        return Halves(ctx, a.tensor.to(torch.float16)) if case["half"] else a

    if s.kind == "projection":
        s.w = Weight(ctx, GGMLType[case["type"]], case["d"], case["n"], gen)
        s.x, s.out = floats(case["n"], scale=1.0), floats(case["d"])
        s.proj = QuantizedProjections(ctx, TornadoWorkspace())
        torch.cuda.synchronize()
        return s

    dim, hidden, kv, vocab, rows, batch = (case[k] for k in ("dim", "hidden", "kv", "vocab", "rows", "batch"))
    main, other, head = FILES[case["file"]]
    s.dim, s.hidden, s.kv, s.vocab, s.rows = dim, hidden, kv, vocab, rows
    s.embedding = torch.randn((batch, dim), device="cuda", generator=gen)
    s.x = floats(batch, dim)                                   # the residual stream
    s.att = activations(batch, dim, scale=0.7)                 # what attention leaves for every layer
    if s.kind == "token":
        s.xb, s.scale = floats(dim), floats(1)
        s.q, s.hb = floats(dim), floats(hidden)
        s.k, s.v = torch.zeros((2, case["layers"], kv), device="cuda")
        s.token = Tokens(torch.zeros(1, dtype=torch.int32, device="cuda"))
        s.logits = floats(vocab)
        s.proj = QuantizedProjections(ctx, TornadoWorkspace(wrapX=s.x, wrapXb=s.xb, wrapHb=s.hb))
        s.out = {"x": s.x.tensor[0], "q": s.q.tensor, "k": s.k, "v": s.v, "hb": s.hb.tensor, "logits": s.logits.tensor,
                 "token": s.token.tensor}
    else:
        s.xb = activations(batch, dim, scale=1.0)              # normalised activations
        s.hb = activations(batch, hidden)
        s.qkv = torch.zeros((case["layers"], batch, dim + 2 * kv), device="cuda")
        s.proj = QuantizedBatchProjections(ctx, batch, max(dim, hidden), max(2 * hidden, dim + 2 * kv), resident=case["resident"])
        s.out = {"x": s.x.tensor[:rows], "qkv": s.qkv[:, :rows], "hb": s.hb.tensor[:rows]}
        if vocab:
            s.logits = floats(batch, vocab)
            s.head_proj = QuantizedBatchProjections(ctx, batch, dim, vocab)
            s.out["logits"] = s.logits.tensor[:rows]
    s.layers = []
    for i in range(case["layers"]):
        y = Layer()
        some = other if i % 2 == 0 else main
        y.wq, y.wk, y.wv = (Weight(ctx, t, d, dim, gen) for t, d in ((main, dim), (main, kv), (some, kv)))
        y.wo, y.w1, y.w3 = (Weight(ctx, main, d, dim, gen) for d in (dim, hidden, hidden))
        y.w2 = Weight(ctx, some, dim, hidden, gen)
        y.norm_att, y.norm_ffn = (Floats(ctx, 1 + 0.1 * torch.randn(dim, device="cuda", generator=gen)) for _ in range(2))
        y.same = main == some
        if s.kind == "token":
            y.k, y.v = Floats(ctx, s.k[i]), Floats(ctx, s.v[i])
        else:
            y.qkv = Floats(ctx, s.qkv[i])
        s.layers.append(y)
    if vocab:
        s.head = Weight(ctx, head, vocab, dim, gen)
        s.head_folds = head in (GGMLType.Q8_0, GGMLType.Q4_0, GGMLType.Q4_K)
        s.norm_out = Floats(ctx, 1 + 0.1 * torch.randn(dim, device="cuda", generator=gen))
    torch.cuda.synchronize()
    return s


def run(s):
    if s.kind == "projection":
        s.proj.floatMatvec(s.x, s.out, s.w, s.w.cols, s.w.rows)
        return s.out.tensor
    s.x.tensor.copy_(s.embedding)
    if s.kind == "token":
        _token(s)
    elif s.att.tensor.dtype == torch.float16:
        _rows_half(s)
    else:
        _rows_float(s)
    return s.out


def _token(s):
    p = s.proj
    for y in s.layers:
        if y.same:
            p.fusedRmsNormQKV(s.x, s.q, y.k, y.v, y.norm_att, None, y.wq, y.wk, y.wv, EPS)
        else:                                                  # no fused launch takes two types
            p.rmsScale(s.x, s.dim, EPS, s.scale)
            p.rmsApply(y.norm_att, s.scale, s.dim)
            p.matvec(s.q, y.wq, s.dim, s.dim)
            p.matvec(y.k, y.wk, s.dim, s.kv)
            p.matvec(y.v, y.wv, s.dim, s.kv)
        p.residualMatvec(s.att, y.wo, s.dim, s.dim)
        p.fullyFusedRmsNormGateUp(s.x, y.norm_ffn, EPS, y.w1, y.w3, s.dim, s.hidden)
        p.residualMatvec(s.hb, y.w2, s.hidden, s.dim)
    if s.head_folds:
        p.matvecArgmax(s.x, s.logits, s.head, s.dim, s.vocab, s.token, s.norm_out, None, EPS)
    else:
        p.rmsScale(s.x, s.dim, EPS, s.scale)
        p.rmsApply(s.norm_out, s.scale, s.dim)
        p.matvecArgmax(s.xb, s.logits, s.head, s.dim, s.vocab, s.token)


def _rows_half(s):
    """Layers as the fp16 plan runs them: the library's normalisation hands the projections fp16 rows."""
    p = s.proj
    for y in s.layers:
        p.rmsApplyFP16(s.x, y.norm_att, EPS, s.xb, s.dim, activeRows=s.rows)
        p.fusedQKV(s.xb, y.qkv, y.wq, y.wk, y.wv, s.rows)
        p.projection(s.att, s.x, y.wo, s.dim, s.dim, True, s.rows)
        p.rmsApplyFP16(s.x, y.norm_ffn, EPS, s.xb, s.dim, activeRows=s.rows)
        p.gateUp(s.xb, s.hb, y.w1, y.w3, s.dim, s.hidden, s.rows)
        p.projection(s.hb, s.x, y.w2, s.hidden, s.dim, True, s.rows)
    if s.vocab:
        p.rmsApplyFP16(s.x, s.norm_out, EPS, s.xb, s.dim, activeRows=s.rows)
        s.head_proj.projection(s.xb, s.logits, s.head, s.dim, s.vocab, False, s.rows)


def _rows_float(s):
    """The same over fp32 activations, whose normalisation is the caller's own: ``xb`` is given."""
    p = s.proj
    for y in s.layers:
        p.fusedQKV(s.xb, y.qkv, y.wq, y.wk, y.wv, s.rows)
        p.projection(s.att, s.x, y.wo, s.dim, s.dim, True, s.rows)
        p.gateUp(s.xb, s.hb, y.w1, y.w3, s.dim, s.hidden, s.rows)
        p.projection(s.hb, s.x, y.w2, s.hidden, s.dim, True, s.rows)
    if s.vocab:
        s.head_proj.projection(s.x, s.logits, s.head, s.dim, s.vocab, False, s.rows)


# ---- what a pass cannot do without ---------------------------------------------------------------

def _layer_weights(case):
    """(elements, bytes) of the layers' weights."""
    dim, hidden, kv, layers = (case[k] for k in ("dim", "hidden", "kv", "layers"))
    main, other, _ = FILES[case["file"]]
    fixed = dim * (2 * dim + kv + 2 * hidden)
    some = dim * (kv + hidden)
    second = (layers + 1) // 2
    return layers * (fixed + some), (layers * main.byte_size_for(fixed) + second * other.byte_size_for(some)
                                     + (layers - second) * main.byte_size_for(some))


def _weight_bytes(case):
    return _layer_weights(case)[1] + FILES[case["file"]][2].byte_size_for(case["vocab"] * case["dim"])


def work(case):
    if case["kind"] == "projection":
        d, n = case["d"], case["n"]
        return {"bytes": GGMLType[case["type"]].byte_size_for(d * n) + 4 * (d + n), "flops": 2 * d * n}
    dim, hidden, kv, layers, vocab, rows = (case[k] for k in ("dim", "hidden", "kv", "layers", "vocab", "rows"))
    act = 2 if case["half"] else 4
    elements = _layer_weights(case)[0] + dim * vocab
    # per row and layer: normalised x twice, attention's result, hb in and out, q|k|v out, x read and added to twice
    per_row = layers * (act * (3 * dim + 2 * hidden) + 4 * (dim + 2 * kv) + 16 * dim) + 4 * (dim + vocab)
    return {"bytes": _weight_bytes(case) + rows * per_row, "flops": 2 * rows * elements}


def tolerance(case):
    """About four times what a pass differs by from the same pass in float64 (whole models, all their outputs)."""
    if case["kind"] == "projection":
        return {"rel": 1.5e-6, "max": 1e-5}
    if case["kind"] == "token":
        # fp32 sums; the types with minimums take the difference of two large sums, and layers add up
        return {"rel": 1e-4, "max": 1e-3} if case["file"].startswith("Q4_K") else {"rel": 1.5e-5, "max": 1.2e-4}
    # operands rounded to fp16; with half, the normalised and hidden vectors between the calls as well
    return {"rel": 1.6e-2, "max": 0.16} if case["half"] else {"rel": 2.5e-3, "max": 0.04}
