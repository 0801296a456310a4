"""Batched projections on the kernel that decodes weights in registers (jl_gemm_reg.hip): every tiling of
every type it takes, at row counts and widths on and off the edges of its tiles, against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

from gpu_util import DECODED, IN_LOOP, IN_REGISTERS, STREAMED, last_gemm, magnitude, rel_err, say
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu

# operands rounded once to fp16 (2^-11 each, of the weight and of the activation) and fp32 sums
F16_BOUND = 2e-3
UNTOUCHED = np.float32(-12345.5)


@pytest.fixture(scope="module")
def ctx():
    from jitllm_amd.runtime import Context
    with Context(0) as c:
        yield c


def columns(d):
    """The output columns that are checked: all of a narrow weight; of a wide one both ends, where tiles
    and ragged last groups are, and a stride through the rest that meets every place in a tile."""
    if d <= 600:
        return np.arange(d)
    return np.unique(np.concatenate([np.arange(40), np.arange(d - 70, d), np.arange(0, d, 131)]))


def rows_of(raw, d, cols):
    return np.ascontiguousarray(raw.reshape(d, -1)[cols]).reshape(-1)


# (type, columns, weight rows side by side, activation rows, active, gate/up, residual), wherever the prices send
# them: one block of columns (a set of waves idle), odd block counts, rows of one group, weights whose last group
# overlaps the one before
CASES = [
    (O.Q4_0, 512, (14003,), 449, 449, False, False), (O.Q4_0, 256, (14003, 14003), 200, 200, True, False),
    (O.Q4_0, 256, (10001, 10001), 257, 257, True, False), (O.Q4_0, 256, (14003, 14003), 449, 449, True, False),
    (O.Q4_0, 512, (14003, 14003), 97, 97, True, False), (O.Q4_0, 512, (14003, 14003), 81, 81, True, False),
    (O.Q4_0, 512, (14003, 14003), 65, 65, True, False), (O.Q4_0, 512, (5005,), 300, 300, False, True),
    (O.Q4_0, 256, (14003, 14003), 97, 97, True, False), (O.Q4_0, 512, (10001,), 129, 129, False, False),
    (O.Q4_0, 256, (16,), 65, 65, False, True), (O.Q4_0, 256, (100, 17, 33), 65, 65, False, True),
    (O.Q8_0, 512, (14003,), 449, 449, False, False), (O.Q8_0, 256, (14003, 14003), 200, 200, True, False),
    (O.Q8_0, 256, (14003, 14003), 449, 449, True, False), (O.Q8_0, 256, (10001, 10001), 257, 257, True, False),
    (O.Q8_0, 512, (14003, 14003), 65, 65, True, False),
    (O.Q8_0, 512, (12001,), 257, 257, False, True), (O.Q8_0, 256, (12001, 12001), 200, 199, True, False),
    (O.Q8_0, 512, (3003, 3003), 257, 257, True, False), (O.Q8_0, 512, (3003, 17, 100), 65, 65, False, False),
    (O.Q4_K, 512, (14003, 14003), 511, 511, True, False), (O.Q4_K, 1280, (12001, 12001), 200, 200, True, False),
    (O.Q4_K, 512, (12001, 12001), 449, 449, True, False), (O.Q4_K, 2304, (16390, 16390), 65, 65, True, False),
    (O.Q4_K, 2816, (8200, 8200), 97, 97, True, False), (O.Q4_K, 2304, (4099, 4099), 255, 255, True, False),
    (O.Q4_K, 2304, (4099, 4099), 240, 240, True, False), (O.Q4_K, 2816, (2050, 2050), 384, 384, True, False),
    (O.Q4_K, 2816, (5005, 5005), 161, 161, True, False), (O.Q4_K, 2816, (1002, 1002), 449, 440, True, False),
    (O.Q6_K, 5888, (5005,), 200, 200, False, True),
    (O.Q6_K, 256, (33,), 128, 128, False, True), (O.Q6_K, 512, (4099,), 161, 161, False, False),
    (O.Q6_K, 768, (4099, 4099), 128, 128, True, False), (O.Q6_K, 2816, (40, 17), 140, 130, False, False),
    (O.Q6_K, 768, (100, 100), 160, 145, True, False),
]


# (tiling, type, columns, weight rows side by side, activation rows, gate/up, residual): every instance of the kernel,
# the shape chosen for it by the price list, with four blocks of columns and more to a set of waves -- each block's
# bytes come in two blocks before they are multiplied -- and an odd count, whose last block one of two sets does not have
TILINGS = [
    (0, O.Q8_0, 1280, (14003,), 449, False, False), (1, O.Q8_0, 1280, (12001,), 481, False, True),
    (2, O.Q8_0, 1280, (10001,), 481, False, False), (3, O.Q8_0, 1280, (4099, 4099), 385, True, False),
    (6, O.Q8_0, 1792, (5005,), 385, False, False), (7, O.Q8_0, 8448, (2050, 2050), 353, True, False),
    (8, O.Q8_0, 1280, (4099,), 385, False, False), (9, O.Q8_0, 2816, (1002, 1002), 353, True, False),
    (10, O.Q8_0, 4352, (1002, 1002), 225, True, False), (0, O.Q4_0, 1280, (14003,), 449, False, False),
    (1, O.Q4_0, 1280, (12001,), 481, False, True), (2, O.Q4_0, 1280, (10001,), 481, False, False),
    (3, O.Q4_0, 1280, (4099, 4099), 385, True, False), (4, O.Q4_0, 1792, (3003, 3003), 481, True, False),
    (5, O.Q4_0, 1792, (5005,), 481, False, True), (6, O.Q4_0, 1792, (4099,), 449, False, False),
    (7, O.Q4_0, 1792, (4099,), 353, False, True), (8, O.Q4_0, 1280, (4099,), 385, False, False),
    (9, O.Q4_0, 1792, (1002, 1002), 385, True, False), (10, O.Q4_0, 2816, (600, 600), 353, True, False),
    (0, O.Q4_K, 1280, (14003,), 449, False, False), (1, O.Q4_K, 1280, (12001,), 481, False, True),
    (2, O.Q4_K, 1280, (10001,), 481, False, False), (3, O.Q4_K, 1280, (10001,), 385, False, True),
    (4, O.Q4_K, 2304, (3003, 3003), 481, True, False), (5, O.Q4_K, 2304, (3003, 3003), 449, True, False),
    (6, O.Q4_K, 2816, (2050, 2050), 449, True, False), (7, O.Q4_K, 2816, (2050, 2050), 353, True, False),
    (8, O.Q4_K, 2816, (5005, 5005), 161, True, False), (9, O.Q4_K, 2816, (1002, 1002), 385, True, False),
    (7, O.Q6_K, 5888, (2050, 2050), 225, True, False), (8, O.Q6_K, 1792, (4099,), 385, False, False),
    (9, O.Q6_K, 1792, (600, 600), 417, True, False), (10, O.Q6_K, 1792, (33,), 129, False, False),
]


@pytest.mark.parametrize("t,n,ds,rows,active,dual,residual", CASES)
def test_weights_decoded_in_registers(ctx, t, n, ds, rows, active, dual, residual):
    check(ctx, t, n, ds, rows, active, dual, residual)


@pytest.mark.parametrize("tiling,t,n,ds,rows,dual,residual", TILINGS)
def test_every_tiling_beyond_its_first_blocks(ctx, tiling, t, n, ds, rows, dual, residual):
    check(ctx, t, n, ds, rows, rows, dual, residual)
    assert last_gemm(ctx) == IN_REGISTERS + tiling


def check(ctx, t, n, ds, rows, active, dual, residual):
    """Against the oracle for fp32 activations; binary16 ones of the same values give the same bits, a
    second call gives the same bits as the first, rows past the active ones stay as they were."""
    from jitllm_amd import _lib as L, synthetic
    from jitllm_amd.projections import QuantizedBatchProjections
    say("decode in registers", t, n, ds, rows, active, dual, residual)
    raws = [synthetic.weight(t, d, n, seed=7100 + i) for i, d in enumerate(ds)]
    ws = [ctx.load_weight(t, raw, d, n) for raw, d in zip(raws, ds)]
    X = synthetic.activations((rows, n), seed=7110).astype(np.float16).astype(np.float32)
    width = ds[0] if dual else sum(ds)
    base = synthetic.activations((rows, width), seed=7111) if residual else np.full((rows, width), UNTOUCHED, np.float32)
    proj = QuantizedBatchProjections(ctx, rows, n, sum(ds))
    ep = L.JL_SWIGLU if dual else L.JL_RESIDUAL if residual else L.JL_STORE
    outs = []
    for x in (ctx.from_numpy(X), ctx.from_numpy(X), ctx.half_from_numpy(X.astype(np.float16))):
        out = ctx.from_numpy(base.reshape(-1).copy())
        proj._gemm(ws, x, out, active, width, 0, ep)
        ctx.sync()
        outs.append(out.get().reshape(rows, width))
        out.free()
        x.free()
    for other in outs[1:]:
        assert np.array_equal(outs[0].view(np.uint32), other.view(np.uint32))
    got = outs[0]
    assert np.array_equal(got[active:], base[active:])
    if dual:
        cols = columns(width)
        parts = [rows_of(raw, width, cols) for raw in raws]
        g, u = (O.matmul_batch(t, part, X[:active], len(cols), n) for part in parts)
        mg, mu = (magnitude(t, part, X[:active], len(cols), n) for part in parts)
        # an error of gate enters with SiLU's slope (at most 1.1) times up, one of up with SiLU(gate) <= |gate|
        sig = 1.0 / (1.0 + np.exp(-g.astype(np.float64)))
        bound = F16_BOUND * (1.1 * mg * np.abs(u) + np.abs(g) * sig * mu + 1.1 * F16_BOUND * mg * mu) + 1e-5
        assert np.all(np.abs(got[:active, cols] - g * sig * u) <= bound)
    else:
        at = 0
        for raw, d in zip(raws, ds):
            cols = columns(d)
            part = rows_of(raw, d, cols)
            ref = O.matmul_batch(t, part, X[:active], len(cols), n)
            old = base[:active, at + cols]
            delta = got[:active, at + cols] - (old if residual else 0.0)
            mag = magnitude(t, part, X[:active], len(cols), n) + (np.abs(old) * 1e-4 if residual else 0.0)
            assert rel_err(delta, ref, mag) < F16_BOUND
            at += d
    proj.workspace.free()
    for w in ws:
        w.free()


def test_output_columns_off_the_vector_width(ctx):
    """An output that starts at an odd column of longer rows (no 16-byte stores), neighbours untouched."""
    from jitllm_amd import _lib as L, synthetic
    from jitllm_amd.projections import QuantizedBatchProjections
    t, n, d, rows, ldo, off = O.Q4_0, 256, 100, 70, 131, 3
    say("decode in registers, odd columns")
    raw = synthetic.weight(t, d, n, seed=7120)
    w = ctx.load_weight(t, raw, d, n)
    X = synthetic.activations((rows, n), seed=7121)
    proj = QuantizedBatchProjections(ctx, rows, n, d)
    out = ctx.float_array(rows * ldo, fill=UNTOUCHED)
    x = ctx.from_numpy(X)
    proj._gemm([w], x, out, rows, ldo, off, L.JL_STORE)
    ctx.sync()
    got = out.get().reshape(rows, ldo)
    assert np.all(got[:, :off] == UNTOUCHED) and np.all(got[:, off + d:] == UNTOUCHED)
    assert rel_err(got[:, off:off + d], O.matmul_batch(t, raw, X, d, n), magnitude(t, raw, X, d, n)) < F16_BOUND
    # rows of very different magnitudes: the row scale keeps each row's bits
    Y = X * np.exp2(np.linspace(-90, 90, rows)).astype(np.float32)[:, None]
    y = ctx.from_numpy(Y)
    proj._gemm([w], y, out, rows, ldo, off, L.JL_STORE)
    ctx.sync()
    got = out.get().reshape(rows, ldo)[:, off:off + d]
    assert rel_err(got, O.matmul_batch(t, raw, Y, d, n), magnitude(t, raw, Y, d, n)) < F16_BOUND
    proj.workspace.free()
    w.free()


# (type, columns, weight rows, activation rows, gate/up or residual, kernel): what measuring both kernels showed to be the faster
@pytest.mark.parametrize("t,n,ds,rows,epilogue,kernel", [
    (O.Q4_0, 4096, (12288, 12288), 128, "dual", IN_LOOP), (O.Q8_0, 2048, (8192, 8192), 161, "dual", IN_LOOP),
    (O.Q4_0, 12288, (4096,), 224, "residual", IN_LOOP), (O.Q4_0, 2048, (2048,), 234, "residual", STREAMED),
    (O.Q4_0, 4096, (4096,), 289, "residual", STREAMED), (O.Q8_0, 2048, (2048, 512, 512), 257, "", STREAMED),
    (O.Q6_K, 3584, (3584, 512, 512), 511, "", DECODED), (O.Q6_K, 13824, (5120,), 511, "residual", DECODED),
    (O.Q6_K, 4096, (14336, 14336), 480, "dual", STREAMED),
    (O.Q4_0, 4096, (12288, 12288), 161, "dual", IN_REGISTERS), (O.Q8_0, 4096, (11008, 11008), 129, "dual", IN_REGISTERS),
    (O.Q4_K, 4096, (11008, 11008), 201, "dual", IN_REGISTERS), (O.Q6_K, 11008, (4096,), 201, "residual", IN_REGISTERS)])
def test_calls_go_to_the_faster_kernel(ctx, t, n, ds, rows, epilogue, kernel):
    """Both forms of activations the same way: the results have the same bits."""
    from jitllm_amd import _lib as L
    from jitllm_amd.ggml import GGMLType
    from jitllm_amd.projections import QuantizedBatchProjections
    say("which kernel", t, n, ds, rows, epilogue)
    ws = [ctx.load_weight(t, np.zeros(GGMLType(t).byte_size_for(d * n), np.uint8), d, n) for d in ds]
    dual = epilogue == "dual"
    width = ds[0] if dual else sum(ds)
    proj = QuantizedBatchProjections(ctx, rows, n, sum(ds))
    out = ctx.float_array(rows * width)
    for x in (ctx.float_array(rows * n), ctx.half_from_numpy(np.zeros((rows, n), np.float16))):
        proj._gemm(ws, x, out, rows, width, 0, L.JL_SWIGLU if dual else L.JL_RESIDUAL if epilogue else L.JL_STORE)
        ctx.sync()
        ran = last_gemm(ctx)
        assert (ran if ran < IN_REGISTERS else IN_REGISTERS) == kernel
    proj.workspace.free()
    for w in ws:
        w.free()


@pytest.mark.parametrize("t", [O.Q4_0, O.Q4_K])
def test_swiglu_of_exact_sums_has_the_bits_of_the_kernel_that_decodes_in_its_loop(ctx, t):
    """One activation a row: a sum is one product, exact in any order, and gate/up's results differ by their SiLU
    alone.  A context that does not cut K runs the call on the kernel that had it before."""
    from jitllm_amd import _lib as L, synthetic
    from jitllm_amd.projections import QuantizedBatchProjections
    from jitllm_amd.runtime import Context
    n, d, rows = 1792, 12001, 201
    say("decode in registers, swiglu", t)
    raws = [synthetic.weight(t, d, n, seed=7160 + i) for i in range(2)]
    X = np.zeros((rows, n), np.float16)
    X[np.arange(rows), (np.arange(rows) * 89) % n] = np.linspace(-400, 400, rows)
    got = []
    for split_k in (True, False):
        with Context(0) as c:
            c.set_split_k(split_k)
            ws = [c.load_weight(t, raw, d, n) for raw in raws]
            proj = QuantizedBatchProjections(c, rows, n, 2 * d)
            out = c.float_array(rows * d)
            proj._gemm(ws, c.half_from_numpy(X), out, rows, d, 0, L.JL_SWIGLU)
            c.sync()
            got.append(out.get())
    assert np.any(got[0]) and np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))


# (type, weight rows side by side, activation rows, gate/up, residual): the tilings with one and with two sets of waves
@pytest.mark.parametrize("t,ds,rows,dual,residual", [
    (O.Q8_0, (3003, 3003), 257, True, False), (O.Q8_0, (14003,), 449, False, False),
    (O.Q4_0, (5005,), 300, False, True), (O.Q4_0, (10001, 17), 129, False, False)])
def test_rows_whose_blocks_lie_far_apart(ctx, t, ds, rows, dual, residual):
    """fp32 rows whose 256-column blocks differ by 2^30, under weights that are zero where the row is large: a
    single power of two for the row would leave nothing of the block that counts."""
    from jitllm_amd import _lib as L, synthetic
    from jitllm_amd.projections import QuantizedBatchProjections
    say("decode in registers, blocks far apart", t, ds, rows, dual, residual)
    n, block = 512, 34 if t == O.Q8_0 else 18
    raws = [np.array(synthetic.weight(t, d, n, seed=7140 + i)).reshape(d, n // 32, block) for i, d in enumerate(ds)]
    for raw in raws:
        raw[:, :8, :2] = 0                                     # the scales of the first 256 columns
    raws = [raw.reshape(-1) for raw in raws]
    X = synthetic.activations((rows, n), seed=7150)
    X[1::3, :256] *= np.float32(2.0 ** 30)
    X[2::6, 256:] = 0
    ws = [ctx.load_weight(t, raw, d, n) for raw, d in zip(raws, ds)]
    width = ds[0] if dual else sum(ds)
    base = synthetic.activations((rows, width), seed=7151) if residual else np.full((rows, width), UNTOUCHED, np.float32)
    proj = QuantizedBatchProjections(ctx, rows, n, sum(ds))
    outs = []
    for _ in range(2):
        out = ctx.from_numpy(base.reshape(-1).copy())
        proj._gemm(ws, ctx.from_numpy(X), out, rows, width, 0, L.JL_SWIGLU if dual else L.JL_RESIDUAL if residual else L.JL_STORE)
        ctx.sync()
        outs.append(out.get().reshape(rows, width))
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
    X[:, :256] = 0                                             # (what those columns add)
    at = 0
    if dual:
        cols = columns(width)
        g, u = (O.matmul_batch(t, rows_of(raw, width, cols), X, len(cols), n).astype(np.float64) for raw in raws)
        mg, mu = (magnitude(t, rows_of(raw, width, cols), X, len(cols), n) for raw in raws)
        sig = 1.0 / (1.0 + np.exp(-g))
        bound = F16_BOUND * (1.1 * mg * np.abs(u) + np.abs(g) * sig * mu + 1.1 * F16_BOUND * mg * mu) + 1e-5
        assert np.all(np.abs(outs[0][:, cols] - g * sig * u) <= bound)
        return
    for raw, d in zip(raws, ds):
        cols = columns(d)
        part = rows_of(raw, d, cols)
        old = base[:, at + cols].astype(np.float64) if residual else 0.0
        # (an fp32 sum with what was there is rounded once: half a unit in the last place of the result)
        bound = F16_BOUND * magnitude(t, part, X, len(cols), n) + 2.0 ** -24 * np.abs(outs[0][:, at + cols])
        assert np.all(np.abs(outs[0][:, at + cols] - old - O.matmul_batch(t, part, X, len(cols), n)) <= bound)
        at += d


@pytest.mark.parametrize("t,n,d,rows", [(O.Q8_0, 1280, 4099, 385), (O.Q4_0, 1280, 4099, 385), (O.Q4_K, 1280, 10001, 385),
                                        (O.Q6_K, 1792, 4099, 385)])
def test_binary16_subnormals_are_multiplied(ctx, t, n, d, rows):
    """Rows of binary16 subnormals, which no scale brings into the normal range on this kernel."""
    from jitllm_amd import synthetic
    from jitllm_amd.projections import QuantizedBatchProjections
    say("decode in registers, subnormals", t, n, d, rows)
    raw = synthetic.weight(t, d, n, seed=7170)
    w = ctx.load_weight(t, raw, d, n)
    X = np.random.default_rng(7171).integers(-1000, 1001, (rows, n)).astype(np.float64) * 2.0 ** -24
    proj = QuantizedBatchProjections(ctx, rows, n, d)
    out = ctx.float_array(rows * d)
    proj.projection(ctx.half_from_numpy(X.astype(np.float16)), out, w, n, d, False)
    ctx.sync()
    assert last_gemm(ctx) >= IN_REGISTERS
    cols = columns(d)
    part = rows_of(raw, d, cols)
    x = X.astype(np.float32)
    assert rel_err(out.get().reshape(rows, d)[:, cols], O.matmul_batch(t, part, x, len(cols), n), magnitude(t, part, x, len(cols), n)) < F16_BOUND
    w.free()


# columns, weight rows, activation rows of Q6_K calls that the weight-streaming kernel has, whatever the others cost
@pytest.mark.parametrize("n,d,rows", [(4096, 4096, 384), (8192, 4096, 511), (14336, 4096, 256), (4096, 12288, 408)])
def test_q6_k_sums_are_as_exact_as_the_streaming_kernels(ctx, n, d, rows):
    """Weights that no kernel but the decoding one rounds (|scale x quant| <= 2048) and binary16 activations: all
    of the error against float64 is that of the fp32 sums.  The same rows in a call of 64, which the
    weight-streaming kernel takes, are the measure: 12 800 values tell its error to 0.6 % (one over the root of
    twice as many), 3 % is five times that.  (In registers, result by result, the first three are 4, 20 and 39 %
    further off, and the fourth four times as far by way of a copy decoded to fp16.)"""
    from jitllm_amd import synthetic
    from jitllm_amd.projections import QuantizedBatchProjections
    say("decode in registers, q6_k sums", n, d, rows)
    raw = np.array(synthetic.weight(O.Q6_K, d, n, seed=7130)).reshape(-1, 210)
    raw[:, 192:208] = (raw[:, 192:208].view(np.int8) >> 1).view(np.uint8)
    X = synthetic.activations((rows, n), seed=7131).astype(np.float16)
    w = ctx.load_weight(O.Q6_K, raw.reshape(-1), d, n)
    x = ctx.half_from_numpy(X)
    proj = QuantizedBatchProjections(ctx, rows, n, d)
    cols = np.arange(7, d, d // 200)[:200]
    exact = X.astype(np.float64) @ O.dequant(O.Q6_K, rows_of(raw.reshape(-1), d, cols)).reshape(len(cols), n).astype(np.float64).T
    err = []
    for active in (64, rows):
        out = ctx.float_array(rows * d)
        proj.projection(x, out, w, n, d, False, active)
        ctx.sync()
        got = out.get().reshape(rows, d)[:active, cols].astype(np.float64)
        err.append(np.linalg.norm(got - exact[:active]) / np.linalg.norm(exact[:active]))
    print("error at 64 rows %.4e, at %d rows %.4e" % (err[0], rows, err[1]))
    assert err[1] <= 1.03 * err[0], err
    proj.workspace.free()
    w.free()
