"""The one-launch GEMV entries (y and SiLU(gate) * up straight from the GEMV,
the last workgroup of a column tile summing the K slices) against the same call
on a caller's stream, which clears, accumulates and converts in three launches:
the same fixed-point terms, so the same bits. Shapes at the edges of the column
tile (8 groups; 16 for large Q4 weights), of the K slice (64, 128, 256 rows), of the
slices per workgroup and with one workgroup per tile (no hand-over); then calls
of different shapes in a row on the one set of counters."""
import ctypes

import numpy as np
import pytest

from helpers import device

pytestmark = pytest.mark.gpu

SHAPES = [(1, 32), (33, 32), (64, 256), (65, 288), (1024, 224), (1025, 512), (2048, 512), (4096, 96), (4097, 2048),
          (11008, 256), (20000, 64)]


def _call(ctx, pkg, d, fmt, paired, w, x, y, k, n, stream):
    lib, h = ctx.lib, ctx.h
    if fmt == "q4":
        if paired:
            return lib.qora_hip_gate_up_q4(h, w[0], w[1], w[2], w[3], x, y, k, n, stream)
        return lib.qora_hip_gemv_q4(h, w[0], w[1], x, y, k, n, stream)
    if paired:
        return lib.qora_hip_gate_up_f16(h, w[0], w[1], x, y, k, n, stream)
    return lib.qora_hip_gemv_f16(h, w[0], x, y, k, n, stream)


def _weights(pkg, d, fmt, paired, k, n, seed):
    out = []
    for i in range(2 if paired else 1):
        if fmt == "q4":
            packed, scales = pkg.synth_q4(seed, i, k, n)
            out += [d.put(packed), d.put(scales)]
        else:
            out.append(d.put(pkg.synth_f16(seed, i, k * n, 0.02)))
    return out


@pytest.fixture
def side_stream():
    hip = ctypes.CDLL("libamdhip64.so.7")
    s = ctypes.c_void_p()
    assert hip.hipStreamCreate(ctypes.byref(s)) == 0
    yield s.value
    hip.hipStreamSynchronize(s)
    assert hip.hipStreamDestroy(s) == 0


@pytest.mark.parametrize("fmt", ["q4", "f16"])
@pytest.mark.parametrize("paired", [False, True])
def test_one_launch_matches_accumulated(ctx, pkg, side_stream, fmt, paired):
    shapes = SHAPES + ([(300, 8192), (2048, 11008), (4096, 4096)] if paired else [(4100, 8224), (256, 131104)])
    with device(ctx) as d:
        held = []
        for k, n in shapes:
            print(f"case {fmt} paired={paired} k={k} n={n}", flush=True)
            w = _weights(pkg, d, fmt, paired, k, n, k + n)
            x = d.put(pkg.synth_f32(5, k, k))
            y, want = d.empty(n * 4), d.empty(n * 4)
            ctx.check(_call(ctx, pkg, d, fmt, paired, w, x, want, k, n, side_stream))
            ctypes.CDLL("libamdhip64.so.7").hipDeviceSynchronize()
            ctx.check(_call(ctx, pkg, d, fmt, paired, w, x, y, k, n, None))
            held.append((k, n, w, x, y, d.get(want, n, np.uint32)))
            assert np.array_equal(d.get(y, n, np.uint32), held[-1][5]), (k, n)
        # back to back, nothing waited for between the shapes
        for k, n, w, x, y, want in held * 2:
            ctx.check(_call(ctx, pkg, d, fmt, paired, w, x, y, k, n, None))
        for k, n, w, x, y, want in held:
            assert np.array_equal(d.get(y, n, np.uint32), want), (k, n)


def test_captured_calls_match_eager(ctx, pkg):
    """An eager call, then the same call captured and replayed with eager
    calls between the replays (a captured call takes the three launches and
    shares no counter with them)."""
    k, n = 2048, 512
    with device(ctx) as d:
        w = _weights(pkg, d, "q4", False, k, n, 9)
        x, y, z = d.put(pkg.synth_f32(9, 3, k)), d.empty(n * 4), d.empty(n * 4)
        ctx.check(_call(ctx, pkg, d, "q4", False, w, x, y, k, n, None))
        want = d.get(y, n, np.uint32)
        ctx.capture_begin()
        ctx.check(_call(ctx, pkg, d, "q4", False, w, x, z, k, n, None))
        g = ctx.capture_end()
        try:
            for _ in range(3):
                ctx.h2d(z, np.zeros(n, np.float32))
                ctx.h2d(y, np.zeros(n, np.float32))
                ctx.graph_launch(g)
                ctx.check(_call(ctx, pkg, d, "q4", False, w, x, y, k, n, None))
                assert np.array_equal(d.get(y, n, np.uint32), want)
                assert np.array_equal(d.get(z, n, np.uint32), want)
        finally:
            ctx.graph_destroy(g)


@pytest.mark.parametrize("fmt", ["q4", "f16"])
@pytest.mark.parametrize("paired", [False, True])
def test_scratch_grows_on_a_caller_stream_behind_queued_work(pkg, side_stream, fmt, paired):
    """Calls on a caller's stream while the context's stream has work queued, from
    the first call of a context on and from one that outgrows its scratch on:
    nothing that the growth leaves on the context's stream, to run in the middle of
    them, may touch what they accumulate in."""
    ctx, hip, calls = pkg.HipContext(0), ctypes.CDLL("libamdhip64.so.7"), 300
    try:
        with device(ctx) as d:
            big = pkg.synth_q4(3, 1, 8192, 8192)
            bp, bs, bo = d.put(big[0]), d.put(big[1]), d.empty(8192 * 8192 * 4)
            for k, n in ((2048, 512), (512, 80000)):            # the second outgrows the first's scratch
                print(f"case growth {fmt} paired={paired} k={k} n={n}", flush=True)
                w = _weights(pkg, d, fmt, paired, k, n, 17)
                x, y = d.put(pkg.synth_f32(17, 3, k)), d.empty(n * 4 * calls)
                ctx.synchronize()
                for _ in range(16):                             # 256 MB written each: about 1 ms in all
                    ctx.check(ctx.lib.qora_hip_dequant_q4(ctx.h, bp, bs, 8192, 8192, bo, None))
                for i in range(calls):                          # 3 ms or more
                    ctx.check(_call(ctx, pkg, d, fmt, paired, w, x, y + i * n * 4, k, n, side_stream))
                assert hip.hipDeviceSynchronize() == 0
                got = d.get(y, (calls, n), np.uint32)
                want = d.empty(n * 4)
                ctx.check(_call(ctx, pkg, d, fmt, paired, w, x, want, k, n, None))
                assert (got == d.get(want, n, np.uint32)).all(), (k, n)
    finally:
        ctx.close()


def test_outgrown_scratch_serves_the_graphs_that_hold_it(pkg):
    """A call captured into a graph, then eager calls that outgrow the scratch the
    graph was recorded with, then its replays: the outgrown scratch is kept."""
    ctx = pkg.HipContext(0)
    try:
        with device(ctx) as d:
            k, n = 2048, 512
            w = _weights(pkg, d, "q4", False, k, n, 9)
            x, y, z = d.put(pkg.synth_f32(9, 3, k)), d.empty(n * 4), d.empty(n * 4)
            ctx.check(_call(ctx, pkg, d, "q4", False, w, x, y, k, n, None))
            want = d.get(y, n, np.uint32)
            ctx.capture_begin()
            ctx.check(_call(ctx, pkg, d, "q4", False, w, x, z, k, n, None))
            g = ctx.capture_end()
            try:
                for n2 in (80000, 400000):                      # each more than twice the scratch before it
                    w2 = _weights(pkg, d, "q4", False, 64, n2, 10)
                    y2 = d.empty(n2 * 4)
                    ctx.check(_call(ctx, pkg, d, "q4", False, w2, d.put(pkg.synth_f32(9, 4, 64)), y2, 64, n2, None))
                    hold = d.put(np.full(1 << 20, 0x5A5A5A5A, np.uint32))   # what a freed block would be given to
                    ctx.h2d(z, np.zeros(n, np.float32))
                    ctx.graph_launch(g)
                    ctx.check(_call(ctx, pkg, d, "q4", False, w, x, y, k, n, None))
                    assert np.array_equal(d.get(z, n, np.uint32), want)
                    assert np.array_equal(d.get(y, n, np.uint32), want)
                    assert (d.get(hold, 1 << 20, np.uint32) == 0x5A5A5A5A).all()
            finally:
                ctx.graph_destroy(g)
    finally:
        ctx.close()


def test_scratch_does_not_grow_in_a_capture_of_the_caller(pkg):
    """A caller that captures the context's stream itself, in the mode that allows
    allocations: calls whose scratch would have to grow are refused and leave no
    node in the graph; once an eager call has sized it, they are captured, and eager
    and replayed calls agree."""
    hip = ctypes.CDLL("libamdhip64.so.7")
    ctx = pkg.HipContext(0)
    stream = ctypes.c_void_p(ctx.lib.qora_hip_stream(ctx.h))
    graph, ex = ctypes.c_void_p(), ctypes.c_void_p()
    k, n, L = 2048, 512, 100
    try:
        with device(ctx) as d:
            w = _weights(pkg, d, "q4", False, k, n, 9)
            x, y, z = d.put(pkg.synth_f32(9, 3, k)), d.empty(n * 4), d.empty(n * 4)
            wid = ctx.upload(pkg.Weight(k=k, n=n, packed=pkg.synth_q4(9, 1, k, n)[0], scales=pkg.synth_q4(9, 1, k, n)[1]))
            kv = d.put(pkg.synth_f32(9, 4, L * 128))
            ctx.synchronize()
            assert hip.hipStreamBeginCapture(stream, 2) == 0          # hipStreamCaptureModeRelaxed
            assert _call(ctx, pkg, d, "q4", False, w, x, z, k, n, None) == pkg.QORA_HIP_E_STATE
            assert ctx.lib.qora_hip_gemm(ctx.h, wid, x, z, 1, None) == pkg.QORA_HIP_E_STATE
            assert ctx.lib.qora_hip_attn_decode(ctx.h, x, kv, kv, 0, L, 1, 1, 128, z, None) == pkg.QORA_HIP_E_STATE
            assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
            nodes = ctypes.c_size_t(99)
            assert hip.hipGraphGetNodes(graph, None, ctypes.byref(nodes)) == 0 and nodes.value == 0
            assert hip.hipGraphDestroy(graph) == 0
            ctx.check(_call(ctx, pkg, d, "q4", False, w, x, y, k, n, None))
            want = d.get(y, n, np.uint32)
            assert hip.hipStreamBeginCapture(stream, 2) == 0
            ctx.check(_call(ctx, pkg, d, "q4", False, w, x, z, k, n, None))
            assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
            assert hip.hipGraphInstantiate(ctypes.byref(ex), graph, None, None, 0) == 0
            for _ in range(3):
                ctx.h2d(z, np.zeros(n, np.float32))
                ctx.h2d(y, np.zeros(n, np.float32))
                assert hip.hipGraphLaunch(ex, stream) == 0
                ctx.check(_call(ctx, pkg, d, "q4", False, w, x, y, k, n, None))
                assert np.array_equal(d.get(y, n, np.uint32), want)
                assert np.array_equal(d.get(z, n, np.uint32), want)
            ctx.synchronize()
            assert hip.hipGraphExecDestroy(ex) == 0 and hip.hipGraphDestroy(graph) == 0
    finally:
        ctx.close()


def test_a_small_eager_call_sizes_captured_ones_up_to_65536_words(pkg):
    ctx = pkg.HipContext(0)
    try:
        with device(ctx) as d:
            small = _weights(pkg, d, "q4", False, 64, 32, 9)
            x = d.put(pkg.synth_f32(9, 3, 64))
            ctx.check(_call(ctx, pkg, d, "q4", False, small, x, d.empty(32 * 4), 64, 32, None))
            for paired, n in ((False, 65536), (True, 32768)):
                w = _weights(pkg, d, "q4", paired, 64, n, 11)
                y, z = d.empty(n * 4), d.empty(n * 4)
                ctx.capture_begin()
                rc = _call(ctx, pkg, d, "q4", paired, w, x, z, 64, n, None)
                g = ctx.capture_end()
                ctx.check(rc)
                ctx.check(_call(ctx, pkg, d, "q4", paired, w, x, y, 64, n, None))
                for _ in range(3):
                    ctx.h2d(z, np.zeros(n, np.float32))
                    ctx.graph_launch(g)
                    assert np.array_equal(d.get(z, n, np.uint32), d.get(y, n, np.uint32)), (paired, n)
                ctx.graph_destroy(g)
    finally:
        ctx.close()


@pytest.mark.parametrize("fmt,rows", [("q4", 16), ("f16", 8)])
def test_long_k_keeps_its_lanes_chains_short(ctx, pkg, fmt, rows):
    """However long K is, a lane adds up at most 16 rows (F16: 8) one by one in
    fp32. Every 2048th group of 32 rows weighs 1, the others half a unit in the last
    place of that: a chain that starts with a 1 loses the rest of its rows, so the
    error tells its length."""
    k, n = 100000, 64
    x = np.full(k, 2.0 ** -25, np.float32)
    x[np.arange(k) % 2048 < 32] = 1.0
    truth = x.astype(np.float64).sum()
    with device(ctx) as d:
        if fmt == "q4":
            w = [d.put(np.full(k * n // 2, 0x99, np.uint8)), d.put(np.full(k * n // 32, 1.0, np.float16))]   # q = 9, scale 1
        else:
            w = [d.put(np.full(k * n, 1.0, np.float16))]
        y = d.empty(n * 4)
        ctx.check(_call(ctx, pkg, d, fmt, False, w, d.put(x), y, k, n, None))
        got = d.get(y, n, np.float32).astype(np.float64)
    assert np.max(np.abs(got - truth)) <= rows * 2.0 ** -24 * truth
