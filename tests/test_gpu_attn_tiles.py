"""The prefill attention launch at the edges of its query tiles, key chunks and waves, and on both sides of the
prompt length past which a block takes two query tiles."""
import ctypes as C

import numpy as np
import pytest


pytestmark = pytest.mark.gpu

E, H, D = 768, 12, 64


@pytest.mark.parametrize("T", [1, 15, 16, 17, 31, 32, 33, 47, 49, 127, 129, 159, 161, 255, 257, 927, 928, 929, 943, 945, 959, 961, 1023])
def test_attention_tile_edges(pkg, L, T):
    """Against float64 attention on the same fp16 values.  Each probability is rounded to fp16 (2^-11 of
    itself, 2^-24 where subnormal; the denominator sums the rounded ones) and so is the output: the weighted
    mean of values is off by at most 2 * 2^-11 + T * 2^-24 of the largest value, and the output's own 2^-11."""
    rng = np.random.default_rng(T)
    qkv = rng.standard_normal((T, 3 * E), dtype=np.float32)
    qkv[:, :2 * E] *= 1.2
    qkv = qkv.astype(np.float16)
    dq, da = pkg.Dev.from_numpy(qkv), pkg.Dev.from_numpy(np.full((T + 1, E), np.float16(7.0)))
    L.gpt2_attention_flash(da.ptr, dq.ptr, T, E, H, D)
    L.gpt2_sync()
    pkg.check("attention")
    got = da.numpy(np.float16, (T + 1, E)).astype(np.float64)
    assert (got[T] == 7.0).all()   # nothing past the last row
    q, k, v = (qkv[:, i * E:(i + 1) * E].astype(np.float64).reshape(T, H, D).transpose(1, 0, 2) for i in range(3))
    s = q @ k.transpose(0, 2, 1) / 8.0
    s[:, np.triu(np.ones((T, T), bool), 1)] = -np.inf
    p = np.exp(s - s.max(axis=2, keepdims=True))
    ref = (p / p.sum(axis=2, keepdims=True) @ v).transpose(1, 0, 2).reshape(T, E)
    assert np.abs(got[:T] - ref).max() <= (3 * 2.0 ** -11 + T * 2.0 ** -24) * np.abs(v).max()


@pytest.mark.parametrize("T", [15, 33, 928, 930])
def test_cache_fill_with_attention(pkg, L, synth, T):
    """The cache rows that the attention launch writes equal the separate scatter's, and no row past T is
    touched."""
    m = pkg.Model(synth.make_body(seed=31, plain=False))
    ids = pkg.Dev.from_numpy(synth.token_ids(T, seed=T))
    scr, kv = pkg.Scratch(T), pkg.KVCache(1024)
    caches = []
    L.gpt2_tune_prefill_lnfold(0)
    try:
        for fused in (1, 0):
            L.gpt2_tune_prefill_fused(fused)
            fill = np.full(kv.kv.bytes // 2, 0x3C00, np.uint16)
            assert L.gpt2_h2d(kv.kv.data, fill.ctypes.data, fill.nbytes) == 0
            L.gpt2_prefill_fill_cache(pkg.backend("flash"), C.byref(m.gpu), C.byref(kv.kv), ids.ptr, T, C.byref(scr.s), None)
            L.gpt2_sync()
            pkg.check("prefill")
            assert L.gpt2_d2h(fill.ctypes.data, kv.kv.data, fill.nbytes) == 0
            caches.append(fill.reshape(12, 2, H, 1024, D).copy())
        assert np.array_equal(caches[0], caches[1])
        assert (caches[0][:, :, :, T:] == 0x3C00).all()
    finally:
        L.gpt2_tune_prefill_fused(1)
        L.gpt2_tune_prefill_lnfold(-1)
        scr.free()
        kv.free()
        m.free()


@pytest.mark.parametrize("T", [1, 17, 130, 1000])
def test_prefill_with_unaligned_qkv_rows(pkg, L, synth, T):
    """A hand-built scratch whose qkv buffer starts 2 bytes past a 16-byte boundary: keys and values go through
    registers instead of direct-to-LDS loads; the same logits and cache rows bit for bit as on an aligned scratch.  (The skinny
    GEMM and the fold want aligned rows of C; both are off here, so that QKV itself has the same bits.)"""
    m = pkg.Model(synth.make_body(seed=33, plain=False))
    ids = pkg.Dev.from_numpy(synth.token_ids(T, seed=T))
    scr, kv = pkg.Scratch(T), pkg.KVCache(1024)
    odd, rows = pkg.GPT2ScratchGPU(), pkg.Dev(T * 3 * E * 2 + 32)
    C.memmove(C.byref(odd), C.byref(scr.s), C.sizeof(odd))
    odd.qkv = rows.ptr + 2
    logits = pkg.Dev(50257 * 2)
    caps = pkg.GPT2CapsGPU()
    caps.logits = logits.ptr
    out = []
    L.gpt2_tune_prefill_lnfold(0)
    L.gpt2_tune_gemm_skinny(0)
    try:
        for s in (scr.s, odd):
            cache = np.full(kv.kv.bytes // 2, 0x3C00, np.uint16)
            assert L.gpt2_h2d(kv.kv.data, cache.ctypes.data, cache.nbytes) == 0
            L.gpt2_prefill_fill_cache(pkg.backend("flash"), C.byref(m.gpu), C.byref(kv.kv), ids.ptr, T, C.byref(s), C.byref(caps))
            L.gpt2_sync()
            pkg.check("prefill")
            assert L.gpt2_d2h(cache.ctypes.data, kv.kv.data, cache.nbytes) == 0
            out.append((logits.numpy(np.uint16, (50257,)), cache.copy()))
        assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    finally:
        L.gpt2_tune_prefill_lnfold(-1)
        L.gpt2_tune_gemm_skinny(-1)
        scr.free()
        kv.free()
        m.free()
