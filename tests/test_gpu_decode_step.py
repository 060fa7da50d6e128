"""The multi-kernel decode step's kernels (csrc/decode_step.hip) against the step that buffers they do not take
run (the LayerNorm, gelu and residual inside the GEMVs), that step on each such kind of buffers, and decode
attention against float64 attention.

A step leaves the kernels of decode_step.hip when a buffer is not 16-byte aligned; a copy of one LayerNorm
gain at an odd address makes the same weights do so.  Both round to fp16 at the same points and differ in the order
of fp32 sums, so logits and cache rows are held to the gates of the persistent step against the
eager one: rel_err = max|a - b| / max|b| <= 1e-2, KL < 2e-3."""
import ctypes as C

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

V, E, H, D, MAXT = 50257, 768, 12, 64, 1024


@pytest.fixture(scope="module")
def model(pkg, synth):
    m = pkg.Model(synth.make_body(seed=77, plain=False))
    yield m
    m.free()


def random_cache(pkg, L, kv, pos, seed):
    """Rows [0, pos) ordinary keys and values; every later row NaN, which no step may read."""
    c = np.full((12, 2, H, MAXT, D), 0x7E00, np.uint16)
    c[:, :, :, :pos] = np.random.default_rng(seed).standard_normal((12, 2, H, pos, D), dtype=np.float32).astype(np.float16).view(np.uint16)
    assert L.gpt2_h2d(kv.kv.data, c.ctypes.data, c.nbytes) == 0
    kv.kv.len = pos


def step(pkg, L, gpu, kv, scr, backend, token, pos, captures=True):
    logits, caps = pkg.Dev(V * 2), pkg.Dev(14 * E * 2)
    L.gpt2_decode_step_cuda(pkg.backend(backend), C.byref(gpu), C.byref(kv.kv), token, pos, C.byref(scr), logits.ptr,
                            caps.ptr if captures else None)
    L.gpt2_sync()
    pkg.check("decode step")
    assert kv.kv.len == pos + 1
    cache = np.empty((12, 2, H, MAXT, D), np.uint16)
    assert L.gpt2_d2h(cache.ctypes.data, kv.kv.data, cache.nbytes) == 0
    return (oracle.f16_to_f32(logits.numpy(np.uint16, (V,))), oracle.f16_to_f32(caps.numpy(np.uint16, (14, E))), cache)


def rel_err(a, b):
    return float(np.abs(a.astype(np.float64) - b).max() / np.abs(b).max())


def kl(got, ref):
    p, q = (np.exp(x.astype(np.float64) - x.max()) for x in (ref, got))
    p, q = p / p.sum(), q / q.sum()
    return float((p * (np.log(p) - np.log(q))).sum())


def copied(pkg, gpu):
    w = pkg.GPT2WeightsGPU()
    C.memmove(C.byref(w), C.byref(gpu), C.sizeof(w))
    return w


@pytest.mark.parametrize("backend,keep", [("gemv", None), ("int8", None), ("int8", 0), ("int8", 3)])
def test_step_matches_general_sequence(pkg, L, model, backend, keep):
    """Positions at the edges of the key splits, waves and passes; keep 0: an INT8 head too; keep 3: every
    third matrix fp16 beside INT8 ones."""
    if backend == "int8":
        model.quantize(None if keep is None else [int(keep and i % keep == 0) for i in range(49)])
    odd = pkg.Dev(2 * E + 32)
    general = pkg.GPT2WeightsGPU()
    C.memmove(C.byref(general), C.byref(model.gpu), C.sizeof(general))
    assert L.gpt2_d2d(odd.ptr + 2, model.gpu.layers[7].ln1_g, 2 * E) == 0
    general.layers[7].ln1_g = odd.ptr + 2
    scr, kv = pkg.Scratch(1), pkg.KVCache(MAXT)
    try:
        for pos in (0, 1, 4, 5, 31, 33, 127, 129, 255, 512, 1000, 1023):
            token = (pos * 7919 + 3) % V
            random_cache(pkg, L, kv, pos, pos)
            got = step(pkg, L, model.gpu, kv, scr.s, backend, token, pos)
            random_cache(pkg, L, kv, pos, pos)
            ref = step(pkg, L, general, kv, scr.s, backend, token, pos)
            assert rel_err(got[0], ref[0]) <= 1e-2, pos
            p = np.exp(ref[0].astype(np.float64) - ref[0].max())
            q = np.exp(got[0].astype(np.float64) - got[0].max())
            assert float((p / p.sum() * (np.log(p / p.sum()) - np.log(q / q.sum()))).sum()) < 2e-3, pos
            assert np.array_equal(got[1][13], ref[1][13]), pos   # the embedding
            assert rel_err(got[1][:13], ref[1][:13]) <= 1e-2, pos
            same = np.ones(MAXT, bool)
            same[pos] = False
            assert np.array_equal(got[2][:, :, :, same], ref[2][:, :, :, same]), pos   # no other row touched
            assert rel_err(oracle.f16_to_f32(got[2][:, :, :, pos]), oracle.f16_to_f32(ref[2][:, :, :, pos])) <= 1e-2, pos
    finally:
        scr.free()
        kv.free()
        if backend == "int8":
            L.gpt2_quant_free(C.byref(model.q))
            model.q = None
            model.gpu.q = None


@pytest.mark.parametrize("backend", ["gemv", "int8"])
@pytest.mark.parametrize("kind", ["scratch", "bias", "matrix"])
def test_step_on_other_buffers(pkg, L, model, kind, backend):
    """Buffers that decode_step.hip's kernels do not take: a scratch without ln, ao and ff (the step without
    captures needs none of them), null biases, matrices at odd addresses.  Same gates against the step on buffers
    that they take; a captured step gives the eager one's bits."""
    if backend == "int8":
        model.quantize()
    ref_w, w, hold = model.gpu, model.gpu, []
    scr, kv = pkg.Scratch(1), pkg.KVCache(MAXT)
    bare = pkg.GPT2ScratchGPU()
    C.memmove(C.byref(bare), C.byref(scr.s), C.sizeof(bare))
    if kind == "scratch":
        bare.ln = bare.ao = bare.ff = None
    elif kind == "bias":
        zero = pkg.Dev.from_numpy(np.zeros(3072, np.uint16))
        hold.append(zero)
        ref_w, w = copied(pkg, model.gpu), copied(pkg, model.gpu)
        for layer in range(12):
            for name in ("qkv_b", "attn_proj_b", "fc_b", "proj_b"):
                setattr(ref_w.layers[layer], name, zero.ptr)
                setattr(w.layers[layer], name, None)
    else:
        w = copied(pkg, model.gpu)
        q = pkg.GPT2QWeightsGPU()
        if backend == "int8":
            C.memmove(C.byref(q), C.byref(model.q), C.sizeof(q))
            w.q = C.addressof(q)
        for layer, name, n in ((0, "qkv_w", 2304 * E), (3, "attn_proj_w", E * E), (5, "fc_w", 3072 * E), (11, "proj_w", 3072 * E)):
            slot = getattr(q.layers[layer], name) if backend == "int8" else None
            size, src = (n, slot.q) if slot else (2 * n, getattr(w.layers[layer], name))
            odd = pkg.Dev(size + 16)
            hold.append(odd)
            assert L.gpt2_d2d(odd.ptr + 2, src, size) == 0
            if slot:
                slot.q = odd.ptr + 2
            else:
                setattr(w.layers[layer], name, odd.ptr + 2)
    try:
        for pos in (0, 5, 130, 1000, 1023):
            token = (pos * 7919 + 3) % V
            random_cache(pkg, L, kv, pos, pos)
            ref = step(pkg, L, ref_w, kv, scr.s, backend, token, pos)
            random_cache(pkg, L, kv, pos, pos)
            got = step(pkg, L, w, kv, bare, backend, token, pos, captures=False)
            assert rel_err(got[0], ref[0]) <= 1e-2 and kl(got[0], ref[0]) < 2e-3, pos
            same = np.ones(MAXT, bool)
            same[pos] = False
            assert np.array_equal(got[2][:, :, :, same], ref[2][:, :, :, same]), pos   # no other row touched
            assert rel_err(oracle.f16_to_f32(got[2][:, :, :, pos]), oracle.f16_to_f32(ref[2][:, :, :, pos])) <= 1e-2, pos
            random_cache(pkg, L, kv, pos, pos)
            logits, tokens = pkg.Dev(V * 2), pkg.Dev(4 * MAXT)
            g = L.gpt2_decode_graph_create_mode(pkg.backend(backend), C.byref(w), C.byref(kv.kv), C.byref(bare), logits.ptr,
                                                tokens.ptr, pkg.DECODE_MULTI)
            pkg.check("graph")
            assert L.gpt2_decode_graph_set(g, token, pos) == 0 and L.gpt2_decode_graph_run(g, 1) == 0
            assert L.gpt2_decode_graph_sync(g, None, None) == 0
            L.gpt2_decode_graph_destroy(g)
            assert np.array_equal(oracle.f16_to_f32(logits.numpy(np.uint16, (V,))), got[0]), pos
    finally:
        scr.free()
        kv.free()
        if backend == "int8":
            L.gpt2_quant_free(C.byref(model.q))
            model.q = None
            model.gpu.q = None


@pytest.mark.parametrize("shared", [("ff", "ao"), ("qkv", "fc"), ("att", "fc"), ("ff", "fc"), ("ao", "qkv")])
def test_step_on_shared_scratch(pkg, L, model, shared):
    """A scratch whose buffers share memory where no value of the general step outlives another's: the kernels of
    decode_step.hip keep their partials in those buffers and must leave such a scratch alone."""
    scr, kv = pkg.Scratch(1), pkg.KVCache(MAXT)
    alias = pkg.GPT2ScratchGPU()
    C.memmove(C.byref(alias), C.byref(scr.s), C.sizeof(alias))
    setattr(alias, shared[0], getattr(alias, shared[1]))
    try:
        for pos in (3, 700):
            token = (pos * 7919 + 3) % V
            random_cache(pkg, L, kv, pos, pos)
            ref = step(pkg, L, model.gpu, kv, scr.s, "gemv", token, pos)
            random_cache(pkg, L, kv, pos, pos)
            got = step(pkg, L, model.gpu, kv, alias, "gemv", token, pos)
            assert rel_err(got[0], ref[0]) <= 1e-2 and kl(got[0], ref[0]) < 2e-3, pos
            assert rel_err(got[1], ref[1]) <= 1e-2, pos
    finally:
        scr.free()
        kv.free()


def test_step_scores_of_minus_infinity(pkg, L, model):
    """Keys whose score is -inf weigh nothing, whether they fill a wave's share, a split or the whole cache: same bits
    as keys of the lowest finite scores, whose weights are 0 too.  The q bias makes dim 0 of every query about 60."""
    b = np.full(2304, np.float16(0))
    b[:E:D] = 60.0
    bias, scr, kv = pkg.Dev.from_numpy(b), pkg.Scratch(1), pkg.KVCache(MAXT)
    w = copied(pkg, model.gpu)
    for layer in range(12):
        w.layers[layer].qkv_b = bias.ptr
    odd = pkg.Dev(2 * E + 32)
    assert L.gpt2_d2d(odd.ptr + 2, model.gpu.layers[7].ln1_g, 2 * E) == 0
    other = copied(pkg, w)   # takes the step of fused GEMVs
    other.layers[7].ln1_g = odd.ptr + 2
    try:
        for pos, keys in ((1, (0, 1)), (33, (0, 2)), (33, (9, 18)), (33, (32, 33)), (33, (0, 33)), (200, (8, 24)), (1023, (256, 512))):
            out = []
            for low in (np.float16(-np.inf), np.float16(-65504.0)):
                c = np.full((12, 2, H, MAXT, D), np.float16(np.nan))
                c[:, :, :, :pos] = np.random.default_rng(pos).standard_normal((12, 2, H, pos, D), dtype=np.float32)
                c[:, 0, :, keys[0]:keys[1], 0] = low
                for gpu in (w, other):
                    assert L.gpt2_h2d(kv.kv.data, c.ctypes.data, c.nbytes) == 0
                    kv.kv.len = pos
                    out.append(step(pkg, L, gpu, kv, scr.s, "gemv", 11, pos)[0])
            assert np.isfinite(out[0]).all(), (pos, keys)
            assert np.array_equal(out[0], out[2]) and np.array_equal(out[1], out[3]), (pos, keys)
    finally:
        scr.free()
        kv.free()


def test_attn_decode_edges(pkg, L):
    """Lengths around the 8-key slots and 16 waves, NaN past the length, peaked scores: against
    float64 attention on the same fp16 values.  Probabilities and sums are fp32, so the error is the fp16
    rounding of the output (half an ulp, 2^-11 of the value) and fp32 noise below it."""
    rng = np.random.default_rng(5)
    kv = pkg.KVCache(MAXT)
    try:
        k, v = (rng.standard_normal((H, MAXT, D), dtype=np.float32).astype(np.float16) for _ in range(2))
        q = (4.0 * rng.standard_normal((3 * E,), dtype=np.float32)).astype(np.float16)
        dq, out = pkg.Dev.from_numpy(q), pkg.Dev(2 * E)
        for n in (1, 2, 7, 8, 9, 63, 64, 65, 127, 128, 129, 500, 512, 777, 1023, 1024):
            c = np.full((12, 2, H, MAXT, D), np.float16(np.nan))
            c[3, 0, :, :n], c[3, 1, :, :n] = k[:, :n], v[:, :n]
            assert L.gpt2_h2d(kv.kv.data, c.ctypes.data, c.nbytes) == 0
            L.gpt2_attn_decode(out.ptr, dq.ptr, C.byref(kv.kv), 3, n)
            L.gpt2_sync()
            pkg.check("attn_decode")
            got = out.numpy(np.float16, (H, D)).astype(np.float64)
            s = np.einsum("hjd,hd->hj", k[:, :n].astype(np.float64), q[:E].reshape(H, D).astype(np.float64)) / 8.0
            p = np.exp(s - s.max(axis=1, keepdims=True))
            ref = np.einsum("hj,hjd->hd", p / p.sum(axis=1, keepdims=True), v[:, :n].astype(np.float64))
            assert np.abs(got - ref).max() <= 2.0 ** -11 * np.abs(ref).max() + 1e-5 * np.abs(v[:, :n]).max(), n
    finally:
        kv.free()


def test_attn_decode_longer_cache(pkg, L):
    """A hand-built cache of more than 1024 positions (gpt2_kv_alloc makes none): a wave then joins several passes of
    64 keys.  Keys that score -inf, a wave's first pass, its second and all but the last key: against float64
    attention with the same scores."""
    T = 2048
    rng = np.random.default_rng(6)
    arena = pkg.Dev(12 * 2 * H * T * D * 2)
    kv = pkg.GPT2KVCache(data=arena.ptr, bytes=arena.nbytes, maxT=T, nLayer=12, nHead=H, headDim=D, len=0)
    k, v = (rng.standard_normal((H, T, D), dtype=np.float32).astype(np.float16) for _ in range(2))
    q = (2.0 * rng.standard_normal((3 * E,), dtype=np.float32)).astype(np.float16)
    q[:E:D] = 2.0
    dq, out = pkg.Dev.from_numpy(q), pkg.Dev(2 * E)
    for n, low in ((1025, ()), (1100, ()), (2048, ()), (1100, (0, 64)), (1100, (64, 72)), (2048, (0, 2047)), (1100, (72, 400))):
        kn = k[:, :n].copy()
        if low:
            kn[:, low[0]:low[1], 0] = -np.inf
        plane = np.full((2, H, T, D), np.float16(np.nan))
        plane[0, :, :n], plane[1, :, :n] = kn, v[:, :n]
        assert L.gpt2_h2d(arena.at(5 * plane.nbytes), plane.ctypes.data, plane.nbytes) == 0
        L.gpt2_attn_decode(out.ptr, dq.ptr, C.byref(kv), 5, n)
        L.gpt2_sync()
        pkg.check("attn_decode")
        got = out.numpy(np.float16, (H, D)).astype(np.float64)
        s = np.einsum("hjd,hd->hj", kn.astype(np.float64), q[:E].reshape(H, D).astype(np.float64)) / 8.0
        p = np.exp(s - s.max(axis=1, keepdims=True))
        ref = np.einsum("hj,hjd->hd", p / p.sum(axis=1, keepdims=True), v[:, :n].astype(np.float64))
        assert np.abs(got - ref).max() <= 2.0 ** -11 * np.abs(ref).max() + 1e-5 * np.abs(v[:, :n]).max(), (n, low)
