"""What no comparison of results shows: what a call takes against another call of the same kernel, and how wide a grid is.

Times of one box are compared with each other, the least of several replays each: a call whose neighbour in size takes
a fifth less per column has lost something."""
import numpy as np
import pytest

from gpu_util import DECODED, last_gemm, last_grid, say
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from jitllm_amd.runtime import Context
    c = Context(0)
    yield c
    c.close()


@pytest.fixture(scope="module")
def hip():
    import bench
    return bench.Hip()


def least_us(ctx, hip, enqueue, calls=12, replays=12):
    """Microseconds of one of `calls` calls in a replayed graph, the least of `replays`."""
    enqueue()
    ctx.sync()
    exe = hip.capture(ctx.stream, lambda: [enqueue() for _ in range(calls)])
    begin, end = hip.event(), hip.event()
    try:
        best = float("inf")
        for _ in range(replays):
            hip.record(begin, ctx.stream)
            hip.launch(exe, ctx.stream)
            hip.record(end, ctx.stream)
            best = min(best, hip.elapsed_ms(begin, end) * 1e3 / calls)
        return best
    finally:
        ctx.sync()
        hip.destroy_event(begin)
        hip.destroy_event(end)
        hip.destroy_graph(exe)


@pytest.mark.parametrize("hidden,rows", [(13824, 524)])      # 256 x 128 tiles in three rounds
def test_rows_no_power_of_two_apart_cost_no_more_per_column(ctx, hip, hidden, rows):
    """The many-row kernel over a kept copy: 2560 columns and 2048.  With loads that a wave waits longer to issue where
    rows lie no power of two apart, and weights come from HBM, the first took 1.24 times as much a column; it takes 1.04
    times as much."""
    from jitllm_amd import synthetic
    from jitllm_amd.projections import QuantizedBatchProjections
    per_column = {}
    for k in (2048, 2560):
        say("per column", hidden, rows, k)
        raw = synthetic.weight(O.Q8_0, hidden, k, seed=2100)
        pairs = [[ctx.load_weight(O.Q8_0, raw, hidden, k) for _ in range(2)] for _ in range(4)]   # more than the caches hold
        x = ctx.half_from_numpy(np.random.default_rng(2101).standard_normal((rows, k)).astype(np.float16))
        hb = ctx.half_from_numpy(np.zeros((rows, hidden), np.float16))
        proj = QuantizedBatchProjections(ctx, rows, k, 2 * hidden, resident=True)
        per_column[k] = least_us(ctx, hip, lambda: [proj.gateUp(x, hb, *pair, k, hidden, rows) for pair in pairs]) / k
        assert last_gemm(ctx) == DECODED
        for w in sum(pairs, []):
            w.free()
    assert per_column[2560] < 1.14 * per_column[2048], per_column


@pytest.mark.parametrize("t,d,n,two,workgroups", [
    (O.Q8_0, 8192, 2048, True, 3),       # (four fit since its tiles come in by buffer loads; three are faster)
    (O.Q4_0, 8960, 768, True, 3),
    (O.Q6_K, 8192, 2048, True, 3),
    (O.Q8_0, 16384, 2048, False, 4),     # what the LDS holds
    (O.Q4_K, 32768, 768, False, 5),      # what 96 registers a lane allow
    (O.Q4_K, 24576, 1536, False, 5),
])
def test_workgroups_a_compute_unit(ctx, t, d, n, two, workgroups):
    """Launches of more tiles than the chip holds workgroups: gate/up takes three a compute unit, others as many as fit."""
    from jitllm_amd import _lib as L, synthetic
    say("workgroups", t, d, n, two)
    raw = synthetic.weight(t, d, n, seed=2110)
    w = [ctx.load_weight(t, raw, d, n) for _ in range(2 if two else 1)]
    x, out = ctx.from_numpy(synthetic.activations(n, seed=2111)), ctx.float_array(d)
    if two:
        L.check(ctx._lib.jl_gemv_gate_up(ctx.handle, w[0].handle, w[1].handle, x.ptr, out.ptr))
    else:
        L.check(ctx._lib.jl_gemv(ctx.handle, w[0].handle, x.ptr, out.ptr, L.JL_STORE))
    ctx.sync()
    units, _ = ctx.device_info()
    assert last_grid(ctx) == workgroups * units
    for weight in w:
        weight.free()
