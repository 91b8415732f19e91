"""The one-launch top-k draw (the last block to arrive merges and draws; penalties
as kernel arguments) against the oracle at the edges of its block count (1, 2, 3,
63 and 64 blocks of 2048 logits) and of the argument list (767 to 769 distinct
penalised tokens, and far more), and against the same calls on a caller's stream,
which run two launches. Same token and Rng state, draw for draw."""
import ctypes

import numpy as np
import pytest

from helpers import device, rng

pytestmark = pytest.mark.gpu

SP = dict(temperature=0.9, top_p=0.97, top_k=40, repetition_penalty=1.2, presence_penalty=0.7)


@pytest.mark.parametrize("vocab", [1, 63, 2048, 2049, 4096, 6000, 129024, 131072])
def test_block_counts(ctx, pkg, orc, vocab):
    print(f"case one-launch sample vocab={vocab}", flush=True)
    hip = ctypes.CDLL("libamdhip64.so.7")
    stream = ctypes.c_void_p()
    assert hip.hipStreamCreate(ctypes.byref(stream)) == 0
    r = rng(vocab)
    params = pkg.SampleParams(**SP)
    a = b = c = 0x9E3779B97F4A7C15
    try:
        with device(ctx) as d:
            for trial in range(12):
                lg = (r.standard_normal(vocab) * 3).astype(np.float32)
                hist = r.integers(0, vocab, size=int(r.integers(0, 200))).astype(np.uint32)
                dl = d.put(lg)
                tok, a = ctx.sample(dl, vocab, hist, params, a)
                want, b = orc.sample(lg, hist.tolist(), SP["temperature"], SP["top_p"], SP["top_k"],
                                     SP["repetition_penalty"], SP["presence_penalty"], b)
                assert (tok, a) == (want, b), trial
                st, tk = ctypes.c_uint64(c), ctypes.c_uint32()
                ctx.check(ctx.lib.qora_hip_sample(ctx.h, dl, vocab, hist.ctypes.data if hist.size else None, hist.size,
                                                  ctypes.byref(params), ctypes.byref(st), ctypes.byref(tk), stream))
                c = st.value
                assert (tk.value, c) == (want, b), trial
    finally:
        hip.hipStreamSynchronize(stream)
        assert hip.hipStreamDestroy(stream) == 0


@pytest.mark.parametrize("distinct", [767, 768, 769, 5000])
def test_penalty_list_sizes(ctx, pkg, orc, distinct):
    vocab = 128256
    r = rng(distinct)
    lg = (r.standard_normal(vocab) * 2).astype(np.float32)
    hist = r.permutation(vocab)[:distinct]
    lg[hist[-40:]] += 9.0                       # the penalised tokens compete
    hist = np.concatenate([hist, hist[-10:], [vocab + 5, 0xFFFFFFFF]]).astype(np.uint32)   # ids past the vocabulary are skipped
    params = pkg.SampleParams(**SP)
    a = b = 77
    with device(ctx) as d:
        dl = d.put(lg)
        for _ in range(20):
            tok, a = ctx.sample(dl, vocab, hist, params, a)
            want, b = orc.sample(lg, hist.tolist(), SP["temperature"], SP["top_p"], SP["top_k"],
                                 SP["repetition_penalty"], SP["presence_penalty"], b)
            assert (tok, a) == (want, b)


def test_a_long_history_costs_no_table_of_its_length(pkg, orc):
    """The look-up table goes by the distinct tokens, at most the vocabulary, not by
    the history's length, and stays small in the context."""
    def resident():
        with open("/proc/self/statm") as f:
            return int(f.read().split()[1]) * 4096

    vocab, n = 5000, 1 << 25
    ctx = pkg.HipContext(0)
    params = pkg.SampleParams(**SP)
    try:
        lg = (rng(1).standard_normal(vocab) * 3).astype(np.float32)
        hist = np.tile(np.arange(0, 4096, dtype=np.uint32), n // 4096)
        with device(ctx) as d:
            dl = d.put(lg)
            ctx.sample(dl, vocab, hist[:100], params, 5)
            before = resident()
            got = ctx.sample(dl, vocab, hist, params, 7)
            grown = resident() - before
            assert got == orc.sample(lg, hist[-4096:].tolist(), SP["temperature"], SP["top_p"], SP["top_k"],
                                     SP["repetition_penalty"], SP["presence_penalty"], 7)
            assert grown < 32 * 2 ** 20, grown        # (a table of the history's length: 256 MB)
    finally:
        ctx.close()


def test_first_calls_on_a_caller_stream_behind_queued_work(pkg, orc):
    """A context's first sampling calls, and those after its scratch grew, on a
    caller's stream while the context's stream has about 1 ms of work queued, then
    one on the context's stream: nothing that the growth leaves on the context's
    stream may touch the words the draws write."""
    hip = ctypes.CDLL("libamdhip64.so.7")
    stream = ctypes.c_void_p()
    assert hip.hipStreamCreateWithFlags(ctypes.byref(stream), 1) == 0     # hipStreamNonBlocking
    ctx = pkg.HipContext(0)
    params = pkg.SampleParams(**SP)
    a = b = 0x1234567890ABCDEF
    try:
        with device(ctx) as d:
            w = pkg.synth_q4(3, 1, 8192, 8192)
            wp, ws, wo = d.put(w[0]), d.put(w[1]), d.empty(8192 * 8192 * 4)
            for vocab in (5000, 128256):
                print(f"case sampling growth vocab={vocab}", flush=True)
                lg = (rng(vocab).standard_normal(vocab) * 3).astype(np.float32)
                hist = np.arange(0, 300, 7, dtype=np.uint32)
                dl = d.put(lg)
                for _ in range(16):
                    ctx.check(ctx.lib.qora_hip_dequant_q4(ctx.h, wp, ws, 8192, 8192, wo, None))
                for call in range(60):
                    s = stream if call < 59 else None
                    st, tk = ctypes.c_uint64(a), ctypes.c_uint32()
                    ctx.check(ctx.lib.qora_hip_sample(ctx.h, dl, vocab, hist.ctypes.data, hist.size,
                                                      ctypes.byref(params), ctypes.byref(st), ctypes.byref(tk), s))
                    a = st.value
                    want, b = orc.sample(lg, hist.tolist(), SP["temperature"], SP["top_p"], SP["top_k"],
                                         SP["repetition_penalty"], SP["presence_penalty"], b)
                    assert (tk.value, a) == (want, b), call
    finally:
        hip.hipDeviceSynchronize()
        ctx.close()
        assert hip.hipStreamDestroy(stream) == 0
