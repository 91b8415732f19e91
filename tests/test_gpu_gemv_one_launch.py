"""The one-launch GEMV entries (y and SiLU(gate) * up straight from the GEMV,
the last workgroup of a column tile summing the K slices) against the same call
on a caller's stream, which clears, accumulates and converts in three launches:
the same fixed-point terms, so the same bits. Shapes at the edges of the column
tile (8 groups; 16 for wide Q4 pairs), of the K slice (64, 128, 256 rows), of the
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
    shapes = SHAPES + ([(300, 8192), (2048, 11008)] if paired else [])
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
