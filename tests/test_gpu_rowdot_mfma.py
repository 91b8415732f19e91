"""The Q4 row-dot on the matrix cores (widths 256, 512, 1024, 2048) at its edges:
rows around a tile of 16, inputs spanning 2^-18 .. 2^6, scales with both signs and
zeros, scales off a 4-byte boundary, inputs with an outlier, and non-finite
inputs, against float64. The bound is the row-dot tests' own: fp32 sums of
products of all 24 bits of x, each output against its own sum of |x w|."""
import numpy as np
import pytest

from helpers import device, elem_err, dequant_np, rel_err, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cols", [256, 512, 1024, 2048])
@pytest.mark.parametrize("rows", [1, 15, 16, 17, 63, 64, 65, 2047, 33000])
def test_rowdot_edges(ctx, pkg, rows, cols):
    print(f"case rowdot rows={rows} cols={cols}", flush=True)
    r = rng(rows + cols)
    packed, scales = pkg.synth_q4(3, rows, rows, cols)
    sc = scales.view(np.float16).copy()
    sc *= r.choice([-1, 0, 1, 1], sc.size).astype(np.float16)
    scales = sc.view(np.uint16)
    x = (r.standard_normal(cols) * 2.0 ** r.integers(-18, 7, cols)).astype(np.float32)
    W = dequant_np(packed, scales, rows, cols)
    truth = W @ x.astype(np.float64)
    with device(ctx) as d:
        wd, xd = d.put(packed), d.put(x)
        for off in (0, 2):
            sd, yd = d.empty(scales.nbytes + 16), d.empty(rows * 4)
            ctx.h2d(sd + off, scales)
            ctx.check(ctx.lib.qora_hip_gemv_q4_rowdot(ctx.h, wd, sd + off, xd, yd, rows, cols, None))
            y = d.get(yd, rows, np.float32)
            assert rel_err(y, truth) <= 1e-5 or np.max(np.abs(truth)) == 0
            assert elem_err(y, truth, np.abs(W) @ np.abs(x.astype(np.float64))) <= 1e-5


@pytest.mark.parametrize("cols", [256, 512, 1024, 2048])
@pytest.mark.parametrize("outlier", [1e3, 1e5, 1e7, 1e9, 2.0 ** 36, 2.0 ** 45, 1e30, 3e38])
@pytest.mark.parametrize("unit", [1.0, 2.0 ** -130])
def test_rowdot_keeps_every_bit_beside_an_outlier(ctx, pkg, cols, outlier, unit):
    """One large input whose weight is zero in every row: the others count with all
    their bits, up to the widest spread that the integer sum holds and past it
    (where x goes through fp32), and with the others subnormal. The row-dot in fp32
    stays within 1e-6 of the sum of |x w| at any outlier."""
    print(f"case rowdot outlier cols={cols} {outlier} {unit}", flush=True)
    rows = 77
    r = rng(cols)
    packed, scales = pkg.synth_q4(6, cols, rows, cols)
    packed = packed.reshape(rows, cols // 2).copy()
    packed[:, 50] = (packed[:, 50] & 0xF0) | 8                   # column 100
    x = (r.standard_normal(cols) * unit).astype(np.float32)
    x[100] = min(outlier * unit, 3e38)
    W = dequant_np(packed.reshape(-1), scales, rows, cols)
    assert not W[:, 100].any()
    with device(ctx) as d:
        yd = d.empty(rows * 4)
        ctx.check(ctx.lib.qora_hip_gemv_q4_rowdot(ctx.h, d.put(packed), d.put(scales), d.put(x), yd, rows, cols, None))
        y = d.get(yd, rows, np.float32)
    xd = x.astype(np.float64)
    # (results of subnormal size: fp32's last place there, 2^-149, for each of the sums)
    err = np.abs(y - W @ xd) - cols * 2.0 ** -149
    assert np.all(err <= 1e-6 * (np.abs(W) @ np.abs(xd)))


def test_rowdot_non_finite_inputs(ctx, pkg):
    rows, cols = 100, 512
    packed, scales = pkg.synth_q4(4, 4, rows, cols)
    W = dequant_np(packed, scales, rows, cols)
    x = rng(1).standard_normal(cols).astype(np.float32)
    with device(ctx) as d:
        wd, sd, yd = d.put(packed), d.put(scales), d.empty(rows * 4)
        for bad in (np.inf, -np.inf, np.nan):
            xb = x.copy()
            xb[77] = bad
            ctx.check(ctx.lib.qora_hip_gemv_q4_rowdot(ctx.h, wd, sd, d.put(xb), yd, rows, cols, None))
            y = d.get(yd, rows, np.float32)
            with np.errstate(invalid="ignore"):
                want = W[:, 77] * bad          # infinite, or NaN where the weight is 0 (or x NaN)
            assert np.array_equal(np.isnan(y), np.isnan(want))
            ok = ~np.isnan(want)
            assert np.array_equal(y[ok], want[ok])
        ctx.check(ctx.lib.qora_hip_gemv_q4_rowdot(ctx.h, wd, sd, d.put(np.zeros(cols, np.float32)), yd, rows, cols, None))
        assert not d.get(yd, rows, np.float32).any()
