"""Kernel-level calls whose output lies over their input: the forms that write it
while other workgroups still read are not taken then, so the results are those of
separate buffers, call after call."""
import numpy as np
import pytest

from helpers import device, dequant_np, elem_err, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("paired", [False, True])
@pytest.mark.parametrize("fmt", ["q4", "f16"])
@pytest.mark.parametrize("k,n,off", [(2048, 2048, 0), (4096, 4096, 0), (2048, 512, 1024), (512, 8192, -4096)])
def test_gemv_over_its_input(ctx, pkg, fmt, paired, k, n, off):
    """y starts `off` floats past x."""
    lib, h = ctx.lib, ctx.h
    x = pkg.synth_f32(31, 1, k)
    with device(ctx) as d:
        if fmt == "q4":
            w = [d.put(a) for i in range(2 if paired else 1) for a in pkg.synth_q4(31, 2 + i, k, n)]
            fn = lib.qora_hip_gate_up_q4 if paired else lib.qora_hip_gemv_q4
        else:
            w = [d.put(pkg.synth_f16(31, 2 + i, k * n, 0.02)) for i in range(2 if paired else 1)]
            fn = lib.qora_hip_gate_up_f16 if paired else lib.qora_hip_gemv_f16
        buf, apart = d.empty((k + n + 2 * abs(off)) * 4), d.empty(n * 4)
        xb = buf + 4 * abs(off)
        yb = xb + 4 * off
        ctx.check(fn(h, *w, d.put(x), apart, k, n, None))
        want = d.get(apart, n, np.uint32)
        for _ in range(5):
            ctx.h2d(xb, x)
            ctx.check(fn(h, *w, xb, yb, k, n, None))
            assert np.array_equal(d.get(yb, n, np.uint32), want)


@pytest.mark.parametrize("fmt", ["q4", "f16"])
@pytest.mark.parametrize("T,k,n", [(16, 512, 33024), (5, 128, 128), (64, 256, 66048), (20, 2048, 2048), (70, 512, 512)])
def test_gemm_over_its_input(ctx, pkg, fmt, T, k, n):
    """x at the start of y: K split and unsplit, few tokens and more."""
    x = rng(T).standard_normal((T, k)).astype(np.float32)
    if fmt == "q4":
        packed, scales = pkg.synth_q4(32, n, k, n)
        W, wt = dequant_np(packed, scales, k, n), pkg.Weight(k=k, n=n, packed=packed, scales=scales)
    else:
        w = pkg.synth_f16(32, n, k * n, 0.02)
        W, wt = w.view(np.float16).astype(np.float64).reshape(k, n), pkg.Weight(k=k, n=n, data=w)
    wid = ctx.upload(wt)
    with device(ctx) as d:
        buf = d.empty(T * max(k, n) * 4)
        for _ in range(3):
            ctx.h2d(buf, x)
            ctx.check(ctx.lib.qora_hip_gemm(ctx.h, wid, buf, buf, T, None))
            y = d.get(buf, (T, n), np.float32)
            # the GEMM tests' bound: fp32 sums of products exact to 22 bits
            assert elem_err(y, x.astype(np.float64) @ W, np.abs(x.astype(np.float64)) @ np.abs(W)) <= 1e-5
    ctx.lib.qora_hip_release_weight(ctx.h, wid)


@pytest.mark.parametrize("kv_f16", [0, 1])
@pytest.mark.parametrize("L", [1, 40, 500, 2000])
def test_decode_attention_over_its_query_and_cache(ctx, kv_f16, L):
    H, KVH, hd = 16, 4, 128
    r = rng(L)
    q = r.standard_normal(H * hd).astype(np.float32)
    k, v = (r.standard_normal((L, KVH * hd)).astype(np.float16 if kv_f16 else np.float32) for _ in range(2))
    with device(ctx) as d:
        apart, qd = d.empty(H * hd * 4), d.empty(H * hd * 4)
        vd = d.empty(max(v.nbytes, H * hd * 4))
        kd = d.put(k)
        ctx.h2d(vd, v)
        ctx.check(ctx.lib.qora_hip_attn_decode(ctx.h, d.put(q), kd, vd, kv_f16, L, H, KVH, hd, apart, None))
        want = d.get(apart, H * hd, np.uint32)
        for out in (qd, vd):
            for _ in range(3):
                ctx.h2d(qd, q)
                ctx.h2d(vd, v)
                ctx.check(ctx.lib.qora_hip_attn_decode(ctx.h, qd, kd, vd, kv_f16, L, H, KVH, hd, out, None))
                assert np.array_equal(d.get(out, H * hd, np.uint32), want)


@pytest.mark.parametrize("T,pos0", [(40, 700), (257, 0), (20, 0)])
def test_prompt_attention_over_its_queries(ctx, T, pos0):
    """Each query block reads its rows before it, or the last of its key chunks,
    writes them."""
    H, KVH, hd = 16, 4, 128
    r = rng(T)
    q = r.standard_normal((T, H * hd)).astype(np.float32)
    k, v = (r.standard_normal((pos0 + T, KVH * hd)).astype(np.float32) for _ in range(2))
    with device(ctx) as d:
        kd, vd, out, qd = d.put(k), d.put(v), d.empty(q.nbytes), d.empty(q.nbytes)
        ctx.check(ctx.lib.qora_hip_attn_prefill(ctx.h, d.put(q), kd, vd, 0, pos0, T, H, KVH, hd, out, None))
        want = d.get(out, q.size, np.uint32)
        for _ in range(3):
            ctx.h2d(qd, q)
            ctx.check(ctx.lib.qora_hip_attn_prefill(ctx.h, qd, kd, vd, 0, pos0, T, H, KVH, hd, qd, None))
            assert np.array_equal(d.get(qd, q.size, np.uint32), want)
