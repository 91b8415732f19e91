"""The Q4 row-dot on the matrix cores (widths 256, 512, 1024, 2048) at its edges:
rows around a tile of 16, inputs spanning 2^-18 .. 2^6, scales with both signs and
zeros, scales off a 4-byte boundary, and non-finite inputs, against
float64. The bound is the row-dot tests' own (fp32 sums; x to 30 bits of its maximum)."""
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
            # (x is held to 2^-31 of its largest value: that much of every weight too)
            bound = 1e-5 * (np.abs(W) @ np.abs(x.astype(np.float64))) + 2.0 ** -30 * np.max(np.abs(x)) * np.abs(W).sum(1)
            assert np.all(np.abs(y - truth) <= bound + 1e-30)


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
