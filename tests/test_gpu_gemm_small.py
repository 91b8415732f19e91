"""qora_hip_gemm at the edges of its routes: the few-token kernel (16, 32 and 64
token tiles, K slices of 128 to 512 rows, column blocks partly past the last
group, x and y off the 16- and 8-byte boundaries) and the packed path just above
it, against float64. The bound is the other GEMM tests': fp32 sums of products
exact to 22 bits."""
import numpy as np
import pytest

from helpers import device, elem_err, dequant_np, rel_err, rng

pytestmark = pytest.mark.gpu

TRUTH_TOL = 1e-5


def _weight(pkg, fmt, k, n, seed, spread):
    if fmt == "f16":
        w = pkg.synth_f16(seed, 1, k * n, 0.02)
        return pkg.Weight(k=k, n=n, data=w), w.view(np.float16).astype(np.float64).reshape(k, n)
    packed, scales = pkg.synth_q4(seed, 2, k, n)
    if spread:      # scales over a range of exponents, both signs
        r = rng(seed)
        scales = (r.choice([-1.0, 1.0], scales.size) * 2.0 ** r.integers(*spread, scales.size)).astype(np.float16)
        scales = scales.view(np.uint16)
    return pkg.Weight(k=k, n=n, packed=packed, scales=scales), dequant_np(packed, scales, k, n)


@pytest.mark.parametrize("fmt", ["q4", "f16"])
@pytest.mark.parametrize("T,k,n", [(1, 32, 32), (15, 544, 96), (16, 2048, 512), (17, 1056, 160), (32, 11008, 256),
                                   (33, 4096, 2080), (64, 2048, 2048), (65, 2080, 256), (66, 8224, 384)])
def test_gemm_few_tokens_vs_truth(ctx, pkg, fmt, T, k, n):
    print(f"case gemm {fmt} T={T} k={k} n={n}", flush=True)
    wt, W = _weight(pkg, fmt, k, n, T + k, None)
    wid = ctx.upload(wt)
    x = (rng(T).standard_normal((T, k)) * 2.0 ** rng(k).integers(-6, 6, (T, 1))).astype(np.float32)
    truth = x.astype(np.float64) @ W
    mag = np.abs(x.astype(np.float64)) @ np.abs(W)
    with device(ctx) as d:
        for off in (0, 4):          # bytes past an aligned address, of x and of y
            xd, yd = d.empty(x.nbytes + 16), d.empty(T * n * 4 + 16)
            ctx.h2d(xd + off, x)
            ctx.check(ctx.lib.qora_hip_gemm(ctx.h, wid, xd + off, yd + off, T, None))
            y = d.get(yd + off, (T, n), np.float32)
            assert rel_err(y, truth) <= TRUTH_TOL
            assert elem_err(y, truth, mag) <= TRUTH_TOL
    ctx.lib.qora_hip_release_weight(ctx.h, wid)


@pytest.mark.parametrize("spread", [(-24, 15), (-24, -18)])
@pytest.mark.parametrize("T", [5, 64, 65])
def test_gemm_scale_extremes(ctx, pkg, T, spread):
    """Scales from subnormal to 2^14 in one matrix, and subnormal ones only:
    the slice exponents keep every weight's two parts finite and exact."""
    k, n = 1024, 256
    wt, W = _weight(pkg, "q4", k, n, 77, spread)
    wid = ctx.upload(wt)
    x = rng(T).standard_normal((T, k)).astype(np.float32)
    with device(ctx) as d:
        y = d.empty(T * n * 4)
        ctx.check(ctx.lib.qora_hip_gemm(ctx.h, wid, d.put(x), y, T, None))
        got = d.get(y, (T, n), np.float32)
    assert elem_err(got, x.astype(np.float64) @ W, np.abs(x.astype(np.float64)) @ np.abs(W)) <= TRUTH_TOL
    ctx.lib.qora_hip_release_weight(ctx.h, wid)


def test_gemm_non_finite_row_stays_in_its_row(ctx, pkg):
    """A row of x with an infinity or NaN gives non-finite outputs in that row
    and leaves the others as they are."""
    k, n, T = 544, 160, 20
    wt, _ = _weight(pkg, "q4", k, n, 5, None)
    wid = ctx.upload(wt)
    x = rng(3).standard_normal((T, k)).astype(np.float32)
    with device(ctx) as d:
        y = d.empty(T * n * 4)
        ctx.check(ctx.lib.qora_hip_gemm(ctx.h, wid, d.put(x), y, T, None))
        want = d.get(y, (T, n), np.float32)
        for bad in (np.inf, np.nan):
            xb = x.copy()
            xb[7, 100] = bad
            ctx.check(ctx.lib.qora_hip_gemm(ctx.h, wid, d.put(xb), y, T, None))
            got = d.get(y, (T, n), np.float32)
            rows = np.arange(T) != 7
            assert np.array_equal(got[rows], want[rows])
            assert not np.isfinite(got[7]).all()
    ctx.lib.qora_hip_release_weight(ctx.h, wid)


@pytest.mark.parametrize("T,k,n", [(65, 96, 128), (130, 2048, 512), (200, 4128, 256), (512, 512, 1152), (129, 8192, 8192),
                                   (129, 8448, 8320)])
def test_gemm_f16_wide_vs_truth(ctx, pkg, T, k, n):
    """F16 weights whose width is a multiple of 128 above 64 tokens: 32- and
    64-token tiles, K split and unsplit."""
    wt, W = _weight(pkg, "f16", k, n, T, None)
    wid = ctx.upload(wt)
    x = rng(T).standard_normal((T, k)).astype(np.float32)
    with device(ctx) as d:
        y = d.empty(T * n * 4)
        ctx.check(ctx.lib.qora_hip_gemm(ctx.h, wid, d.put(x), y, T, None))
        got = d.get(y, (T, n), np.float32)
    truth = x.astype(np.float64) @ W
    assert rel_err(got, truth) <= TRUTH_TOL
    assert elem_err(got, truth, np.abs(x.astype(np.float64)) @ np.abs(W)) <= TRUTH_TOL
    ctx.lib.qora_hip_release_weight(ctx.h, wid)


def _captured(ctx, wid, x, y, T):
    ctx.capture_begin()
    rc = ctx.lib.qora_hip_gemm(ctx.h, wid, x, y, T, None)
    g = ctx.capture_end()
    ctx.check(rc)
    return g


@pytest.mark.parametrize("fmt,k,n", [("q4", 11008, 2048), ("f16", 11008, 2048), ("q4", 2048, 11008), ("f16", 2048, 11008),
                                     ("q4", 1024, 160), ("f16", 1024, 160)])
@pytest.mark.parametrize("eager", [64, 100, 200])
def test_an_eager_gemm_sizes_captured_ones_of_fewer_tokens(pkg, fmt, k, n, eager):
    """Once an eager call of a weight has run, calls with as many tokens or fewer
    are captured; their replays give the eager calls' bits."""
    ctx = pkg.HipContext(0)
    wt, _ = _weight(pkg, fmt, k, n, 3, None)
    try:
        wid = ctx.upload(wt)
        x = rng(4).standard_normal((eager, k)).astype(np.float32)
        with device(ctx) as d:
            xd, y, z = d.put(x), d.empty(eager * n * 4), d.empty(eager * n * 4)
            ctx.check(ctx.lib.qora_hip_gemm(ctx.h, wid, xd, y, eager, None))
            for T in (eager, 130, 65, 64, 63, 33, 32, 17, 16, 1):
                if T > eager:
                    continue
                print(f"case captured gemm {fmt} {k} {n} eager={eager} T={T}", flush=True)
                g = _captured(ctx, wid, xd, z, T)
                for _ in range(3):
                    ctx.h2d(z, np.zeros((T, n), np.float32))
                    ctx.graph_launch(g)
                    ctx.check(ctx.lib.qora_hip_gemm(ctx.h, wid, xd, y, T, None))
                    assert np.array_equal(d.get(z, (T, n), np.uint32), d.get(y, (T, n), np.uint32)), T
                ctx.graph_destroy(g)
    finally:
        ctx.close()


def test_a_captured_gemm_takes_what_another_weights_call_sized(pkg):
    """Scratch sized by another weight's call, between what the general path and the
    few-token kernel need: captured on the former."""
    ctx = pkg.HipContext(0)
    k, n, T = 11008, 2048, 64                    # 22.5 MB of partial sums; 19.9 MB on the general path
    wt, W = _weight(pkg, "f16", k, n, 3, None)
    x = rng(4).standard_normal((T, k)).astype(np.float32)
    try:
        other = ctx.upload(_weight(pkg, "f16", 45056, 32, 5, None)[0])
        wid = ctx.upload(wt)
        with device(ctx) as d:
            xo = d.put(np.zeros((100, 45056), np.float32))
            ctx.check(ctx.lib.qora_hip_gemm(ctx.h, other, xo, d.empty(100 * 32 * 4), 100, None))   # 20.3 MB
            xd, z = d.put(x), d.empty(T * n * 4)
            g = _captured(ctx, wid, xd, z, T)
            for _ in range(2):
                ctx.h2d(z, np.zeros((T, n), np.float32))
                ctx.graph_launch(g)
                got = d.get(z, (T, n), np.float32)
                assert elem_err(got, x.astype(np.float64) @ W, np.abs(x.astype(np.float64)) @ np.abs(W)) <= TRUTH_TOL
            ctx.graph_destroy(g)
    finally:
        ctx.close()


@pytest.mark.parametrize("fmt", ["q4", "f16"])
@pytest.mark.parametrize("T,k,n", [(33, 2048, 11008), (64, 4096, 8192), (17, 4096, 32768), (16, 4096, 32768), (64, 11008, 2048),
                                   (64, 8192, 11008)])
def test_gemm_few_tokens_on_both_sides_of_the_partial_sum_limit(ctx, pkg, fmt, T, k, n):
    """Wide and deep weights: the few-token kernel below the limit on its partial
    sums, the general path above (each format has cases on either side)."""
    wt, W = _weight(pkg, fmt, k, n, 6, None)
    wid = ctx.upload(wt)
    x = rng(T).standard_normal((T, k)).astype(np.float32)
    cols = np.r_[0:64, n // 2:n // 2 + 64, n - 64:n]
    with device(ctx) as d:
        y = d.empty(T * n * 4)
        ctx.check(ctx.lib.qora_hip_gemm(ctx.h, wid, d.put(x), y, T, None))
        got = d.get(y, (T, n), np.float32)
    Wc = W[:, cols]
    assert np.isfinite(got).all()
    assert elem_err(got[:, cols], x.astype(np.float64) @ Wc, np.abs(x.astype(np.float64)) @ np.abs(Wc)) <= TRUTH_TOL
    ctx.lib.qora_hip_release_weight(ctx.h, wid)


def test_f16_gemm_keeps_its_fp32_chains_short(ctx, pkg):
    """Above 128 tokens an F16 weight's sums run over 256 rows at a time, whatever the
    K slices: rounding then leaves 1.7e-7 of the result's norm here, and 4.0e-7 where a
    chain runs over a whole slice (1856 rows)."""
    k, n, T = 11008, 2048, 300
    wt, W = _weight(pkg, "f16", k, n, 8, None)
    wid = ctx.upload(wt)
    x = rng(8).standard_normal((T, k)).astype(np.float32)
    with device(ctx) as d:
        y = d.empty(T * n * 4)
        ctx.check(ctx.lib.qora_hip_gemm(ctx.h, wid, d.put(x), y, T, None))
        got = d.get(y, (T, n), np.float32)
    truth = x.astype(np.float64) @ W
    assert np.linalg.norm(got - truth) <= 2.5e-7 * np.linalg.norm(truth)
    ctx.lib.qora_hip_release_weight(ctx.h, wid)


def test_outgrown_workspaces_serve_the_graphs_that_hold_them(pkg):
    """A GEMM and a decode attention captured, then eager calls that outgrow their
    workspaces, then the replays: what a graph holds is kept."""
    ctx = pkg.HipContext(0)
    k, n, T, L, H, hd = 2048, 512, 16, 700, 4, 128
    try:
        wid = ctx.upload(_weight(pkg, "q4", k, n, 3, None)[0])
        big = ctx.upload(_weight(pkg, "q4", 4096, 4096, 4, None)[0])
        r = rng(5)
        with device(ctx) as d:
            x, kv = d.put(r.standard_normal((T, k)).astype(np.float32)), d.put(r.standard_normal((8 * L, H * hd)).astype(np.float32))
            y, z, a, b = (d.empty(T * n * 4) for _ in range(4))
            attn = lambda L, out: ctx.lib.qora_hip_attn_decode(ctx.h, x, kv, kv, 0, L, H, H, hd, out, None)
            ctx.check(ctx.lib.qora_hip_gemm(ctx.h, wid, x, y, T, None))
            ctx.check(attn(L, a))
            want, wa = d.get(y, (T, n), np.uint32), d.get(a, H * hd, np.uint32)
            ctx.capture_begin()
            rc = ctx.lib.qora_hip_gemm(ctx.h, wid, x, z, T, None) or attn(L, b)
            g = ctx.capture_end()
            ctx.check(rc)
            ctx.check(ctx.lib.qora_hip_gemm(ctx.h, big, d.put(np.ones((300, 4096), np.float32)), d.empty(300 * 4096 * 4), 300, None))
            ctx.check(attn(8 * L, a))
            hold = [d.put(np.full(1 << 18, 0x5A5A5A5A, np.uint32)) for _ in range(16)]   # what freed blocks would be given to
            for _ in range(3):
                ctx.h2d(z, np.zeros((T, n), np.float32))
                ctx.h2d(b, np.zeros(H * hd, np.float32))
                ctx.graph_launch(g)
                assert np.array_equal(d.get(z, (T, n), np.uint32), want)
                assert np.array_equal(d.get(b, H * hd, np.uint32), wa)
            for h in hold:
                assert (d.get(h, 1 << 18, np.uint32) == 0x5A5A5A5A).all()
            ctx.graph_destroy(g)
    finally:
        ctx.close()
