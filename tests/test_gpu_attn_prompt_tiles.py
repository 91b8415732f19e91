"""Prompt attention (qora_hip_attn_prefill) at the edges of its query tiles (four or
eight waves: 16 or 32 queries with four heads a KV head, up to 128 with one) and
64-key steps, f32 and f16 caches, against float64. 64 heads over 16 take the eight
waves from 113 tokens on. The bound is the prompt attention
tests' own kind: fp32 sums of products held to 22 bits, relative to max |v|."""
import ctypes

import numpy as np
import pytest

from helpers import device, rng

pytestmark = pytest.mark.gpu


def _truth(q, k, v, pos0, T, H, KVH, hd):
    out = np.empty((T, H, hd))
    q, k, v = q.reshape(T, H, hd), k.reshape(-1, KVH, hd), v.reshape(-1, KVH, hd)
    for h in range(H):
        g = h // (H // KVH)
        s = q[:, h] @ k[:, g].T / np.sqrt(hd)
        s[np.arange(pos0 + T)[None, :] > pos0 + np.arange(T)[:, None]] = -np.inf
        p = np.exp(s - s.max(1, keepdims=True))
        out[:, h] = p / p.sum(1, keepdims=True) @ v[:, g]
    return out.reshape(T, H * hd)


@pytest.mark.parametrize("kv_f16", [0, 1])
@pytest.mark.parametrize("H,KVH,hd", [(8, 2, 128), (4, 2, 64), (2, 2, 64), (2, 2, 128), (64, 16, 64)])
@pytest.mark.parametrize("T,pos0", [(1, 0), (16, 47), (17, 0), (31, 1), (32, 32), (33, 63), (65, 64), (128, 0), (129, 200),
                                    (1, 255), (20, 192), (60, 1111), (193, 0), (300, 5)])
def test_query_and_key_tile_edges(ctx, kv_f16, H, KVH, hd, T, pos0):
    r = rng(T * 7 + hd)
    q = r.standard_normal((T, H * hd)).astype(np.float32) * 2
    k, v = (r.standard_normal((pos0 + T, KVH * hd)).astype(np.float16 if kv_f16 else np.float32) for _ in range(2))
    if kv_f16:
        k.flat[::97] = np.float16(6e-8)         # subnormals
    truth = _truth(q.astype(np.float64), k.astype(np.float64), v.astype(np.float64), pos0, T, H, KVH, hd)
    with device(ctx) as d:
        out = d.empty(T * H * hd * 4)
        ctx.check(ctx.lib.qora_hip_attn_prefill(ctx.h, d.put(q), d.put(k), d.put(v), kv_f16, pos0, T, H, KVH, hd, out, None))
        got = d.get(out, (T, H * hd), np.float32)
    assert np.max(np.abs(got - truth)) <= 1e-5 * np.max(np.abs(v.astype(np.float64)))


def test_f16_cache_of_subnormals(ctx):
    """An f16 cache goes to the matrix cores as it is stored: subnormal keys and
    values count in full (scores here are of order one, from q near 2^20)."""
    r = rng(5)
    T, H, hd = 70, 4, 64
    k, v = ((r.integers(-900, 900, (T, hd)) * 2.0 ** -24).astype(np.float16) for _ in range(2))
    q = (r.standard_normal((T, H * hd)) * 2.0 ** 13).astype(np.float32)
    truth = _truth(q.astype(np.float64), k.astype(np.float64), v.astype(np.float64), 0, T, H, 1, hd)
    with device(ctx) as d:
        out = d.empty(T * H * hd * 4)
        ctx.check(ctx.lib.qora_hip_attn_prefill(ctx.h, d.put(q), d.put(k), d.put(v), 1, 0, T, H, 1, hd, out, None))
        got = d.get(out, (T, H * hd), np.float32)
    assert np.max(np.abs(got - truth)) <= 1e-5 * np.max(np.abs(v.astype(np.float64)))


def test_split_keys_come_out_as_whole_ones(ctx):
    """Calls on the context's stream split the keys over blocks (193 or more of
    them). Chunks merge in key order whichever block is last, so the bits are the
    same call after call; (512, 1600) takes the split's eight waves, and the split's
    counters are back at zero for the next shape."""
    r = rng(9)
    H, KVH, hd = 16, 4, 128
    for T, pos0 in ((40, 700), (257, 0), (16, 180), (512, 90), (512, 1600), (40, 700)):
        q = r.standard_normal((T, H * hd)).astype(np.float32)
        k, v = (r.standard_normal((pos0 + T, KVH * hd)).astype(np.float32) for _ in range(2))
        truth = _truth(q.astype(np.float64), k.astype(np.float64), v.astype(np.float64), pos0, T, H, KVH, hd)
        with device(ctx) as d:
            out = d.empty(T * H * hd * 4)
            args = (ctx.h, d.put(q), d.put(k), d.put(v), 0, pos0, T, H, KVH, hd, out)
            first = None
            for _ in range(4):
                ctx.check(ctx.lib.qora_hip_attn_prefill(*args, None))
                got = d.get(out, (T, H * hd), np.float32)
                first = got if first is None else first
                np.testing.assert_array_equal(got, first)
        assert np.max(np.abs(first - truth)) <= 1e-5 * np.max(np.abs(v))


def test_the_splits_workspace_comes_with_the_first_split_call(pkg):
    """Contexts that never split a prompt's keys hold no workspace for it."""
    hip = ctypes.CDLL("libamdhip64.so.7")

    def used(n, split):
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        ctxs = [pkg.HipContext(0) for _ in range(n)]
        H, KVH, hd = 16, 4, 128
        T = 300 if split else 60
        try:
            for c in ctxs:
                with device(c) as d:
                    x = d.empty(T * H * hd * 4)
                    c.check(c.lib.qora_hip_attn_prefill(c.h, x, x, x, 0, 0, T, H, KVH, hd, d.empty(T * H * hd * 4), None))
            assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
            return total.value - free.value
        finally:
            for c in ctxs:
                c.close()

    used(2, True)                                  # (what the process allocates once)
    base, unsplit, split = used(1, False), used(17, False), used(17, True)
    print("MB a context:", (unsplit - base) / 16 / 2 ** 20, (split - base) / 16 / 2 ** 20, flush=True)
    assert unsplit - base < 16 * 8 * 2 ** 20
    assert split - base >= 16 * 4 * 2 ** 20


def test_the_first_split_call_leaves_another_streams_capture_alone(pkg):
    """A context's first split call, on its own stream, while the caller captures
    another stream in the default mode: that capture still ends in a graph."""
    hip = ctypes.CDLL("libamdhip64.so.7")
    H, KVH, hd, T = 4, 1, 128, 300
    r = rng(12)
    q = r.standard_normal((T, H * hd)).astype(np.float32)
    k, v = (r.standard_normal((T, KVH * hd)).astype(np.float32) for _ in range(2))
    truth = _truth(q.astype(np.float64), k.astype(np.float64), v.astype(np.float64), 0, T, H, KVH, hd)
    ctx, other, graph = pkg.HipContext(0), ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipStreamCreateWithFlags(ctypes.byref(other), 1) == 0     # hipStreamNonBlocking
    try:
        with device(ctx) as d:
            out = d.empty(T * H * hd * 4)
            args = (ctx.h, d.put(q), d.put(k), d.put(v), 0, 0, T, H, KVH, hd, out)
            ctx.synchronize()
            assert hip.hipStreamBeginCapture(other, 0) == 0              # hipStreamCaptureModeGlobal
            rc = ctx.lib.qora_hip_attn_prefill(*args, None)
            end = hip.hipStreamEndCapture(other, ctypes.byref(graph))
            ctx.check(rc)
            assert end == 0
            assert hip.hipGraphDestroy(graph) == 0
            got = d.get(out, (T, H * hd), np.float32)
            assert np.max(np.abs(got - truth)) <= 1e-5 * np.max(np.abs(v))
            ctx.check(ctx.lib.qora_hip_attn_prefill(*args, None))
            np.testing.assert_array_equal(d.get(out, (T, H * hd), np.float32), got)
    finally:
        ctx.close()
        assert hip.hipStreamDestroy(other) == 0
