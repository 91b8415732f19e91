"""Decode attention (qora_hip_attn_decode) in one launch, its splits merged by the
last of each KV head: the bits of the two launches that a caller's stream takes
(the same sums in the same order), at the edges of a split (32 positions) and of
the rule (128 splits over all KV heads), call after call."""
import numpy as np
import pytest

from helpers import device, rng

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def side_stream():
    s = torch.cuda.Stream()
    yield s.cuda_stream
    torch.cuda.synchronize()


@pytest.mark.parametrize("kv_f16", [0, 1])
@pytest.mark.parametrize("H,KVH,hd", [(16, 4, 128), (2, 2, 64), (3, 1, 40), (4, 2, 104)])
@pytest.mark.parametrize("L", [1, 31, 32, 33, 64, 500, 1024, 1025, 2048, 2049])
def test_one_launch_has_the_two_launches_bits(ctx, side_stream, kv_f16, H, KVH, hd, L):
    r = rng(L + hd)
    q = r.standard_normal(H * hd).astype(np.float32) * 3
    k, v = (r.standard_normal((L, KVH * hd)).astype(np.float16 if kv_f16 else np.float32) for _ in range(2))
    with device(ctx) as d:
        out, want = d.empty(H * hd * 4), d.empty(H * hd * 4)
        args = (ctx.h, d.put(q), d.put(k), d.put(v), kv_f16, L, H, KVH, hd)
        ctx.check(ctx.lib.qora_hip_attn_decode(*args, want, side_stream))
        torch.cuda.synchronize()
        ref = d.get(want, H * hd, np.float32)
        for _ in range(3):
            ctx.check(ctx.lib.qora_hip_attn_decode(*args, out, None))
            np.testing.assert_array_equal(d.get(out, H * hd, np.float32), ref)
    kd, vd = (a.astype(np.float64).reshape(L, KVH, hd).repeat(H // KVH, 1) for a in (k, v))
    s = np.einsum("hd,lhd->hl", q.reshape(H, hd).astype(np.float64), kd) / np.sqrt(hd)
    p = np.exp(s - s.max(1, keepdims=True))
    truth = np.einsum("hl,lhd->hd", p / p.sum(1, keepdims=True), vd).reshape(-1)
    # scores to a few fp32 ulp of |q||k| ~ 3 hd / sqrt(hd): 1e-5 relative to max |v|
    assert np.max(np.abs(ref - truth)) <= 1e-5 * np.max(np.abs(vd))


@pytest.mark.parametrize("L", [2049, 4096, 6000, 8064, 8065, 8200, 12001])
def test_long_f16_heads_of_64_at_both_pass_lengths(ctx, L):
    """Splits of fewer than 128 positions take passes of 8, longer ones of 16; L - 1
    leaves the last pass of a split partly empty."""
    H, KVH, hd = 8, 2, 64
    r = rng(L)
    q = r.standard_normal(H * hd).astype(np.float32) * 3
    k, v = (r.standard_normal((L, KVH * hd)).astype(np.float16) for _ in range(2))
    with device(ctx) as d:
        qd, kd, vd, out = d.put(q), d.put(k), d.put(v), d.empty(H * hd * 4)
        for n in (L, L - 1):
            ctx.check(ctx.lib.qora_hip_attn_decode(ctx.h, qd, kd, vd, 1, n, H, KVH, hd, out, None))
            got = d.get(out, H * hd, np.float32)
            k64, v64 = (a[:n].astype(np.float64).reshape(n, KVH, hd).repeat(H // KVH, 1) for a in (k, v))
            s = np.einsum("hd,lhd->hl", q.reshape(H, hd).astype(np.float64), k64) / np.sqrt(hd)
            p = np.exp(s - s.max(1, keepdims=True))
            truth = np.einsum("hl,lhd->hd", p / p.sum(1, keepdims=True), v64).reshape(-1)
            # as above: scores to a few fp32 ulp
            assert np.max(np.abs(got - truth)) <= 1e-5 * np.max(np.abs(v64))
