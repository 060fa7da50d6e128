"""The trunk GEMMs at both sides of every length where the pick table changes tiles, plain and with the
fused epilogues that the prefill uses there."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = {"qkv": (2304, 768), "attn_proj": (768, 768), "fc": (3072, 768), "mlp_proj": (768, 3072)}
EDGES = (64, 96, 128, 160, 224, 256, 320, 448, 512, 640, 672, 704, 768, 832, 896, 960, 1024)


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("shape", list(SHAPES))
def test_trunk_gemm_at_pick_edges(pkg, L, shape, int8):
    """Against the float64 product of the same fp16 (INT8: code x scale) values.  The fp32 sums are off by less
    than 2^-14 of the result's spread here (3072 terms, each fp32 step 2^-24 of the partial sum) and the fp16
    output by half an ulp, 2^-11 of the value.  Fused gelu and residual epilogues give the bits of the plain
    product followed by gpt2_gelu / gpt2_add; rows past M stay untouched."""
    N, K = SHAPES[shape]
    rng = np.random.default_rng(N + K + int8)
    A = rng.standard_normal((1025, K), dtype=np.float32).astype(np.float16)
    W = (rng.standard_normal((N, K), dtype=np.float32) * np.float32(0.02)).astype(np.float16)
    b = (rng.standard_normal(N, dtype=np.float32) * np.float32(0.1)).astype(np.float16)
    R = rng.standard_normal((1025, N), dtype=np.float32).astype(np.float16)
    Wd, sp = W.astype(np.float64), None
    if int8:
        s = (np.abs(W.astype(np.float32)).max(axis=1) / np.float32(127.0)).astype(np.float32)
        q = np.clip(np.rint(W.astype(np.float32) / s[:, None]), -127, 127).astype(np.int8)
        Wd, sp = q.astype(np.float64) * s[:, None].astype(np.float64), pkg.Dev.from_numpy(s)
    ref = A.astype(np.float64) @ Wd.T + b.astype(np.float64)
    dA, dW, db, dR = (pkg.Dev.from_numpy(x) for x in (A, q if int8 else W, b, R))
    plain, fused, add = (pkg.Dev(1026 * N * 2) for _ in range(3))
    mark = np.full((1, N), np.float16(3.0))
    for M in sorted({m + d for m in EDGES for d in (0, 1)} | {33, 577, 1000}):
        assert L.gpt2_h2d(plain.at(M * N * 2), mark.ctypes.data, mark.nbytes) == 0
        if int8:
            L.gpt2_matmul_int8(plain.ptr, dA.ptr, dW.ptr, sp.ptr, db.ptr, M, N, K)
        else:
            L.gpt2_matmul_tiled(plain.ptr, dA.ptr, dW.ptr, db.ptr, M, N, K)
        L.gpt2_sync()
        pkg.check("%s M=%d" % (shape, M))
        got = plain.numpy(np.float16, (M + 1, N))
        assert (got[M] == 3.0).all(), M
        err = np.abs(got[:M].astype(np.float64) - ref[:M])
        assert (err <= 2.0 ** -11 * np.abs(ref[:M]) + 2.0 ** -14 * ref[:M].std()).all(), (M, err.max())
        if shape == "qkv" or M > 1024:
            continue
        epi = 1 if shape == "fc" else 2
        assert L.gpt2_d2d(add.ptr, plain.ptr, M * N * 2) == 0
        if epi == 1:
            L.gpt2_gelu(add.ptr, M * N)
        else:
            assert L.gpt2_d2d(add.ptr, dR.ptr, M * N * 2) == 0
            L.gpt2_add(add.ptr, plain.ptr, M * N)
        assert L.gpt2_tune_gemm_fused(fused.ptr, dA.ptr, dW.ptr, sp.ptr if int8 else None, db.ptr, M, N, K, epi,
                                      dR.ptr if epi == 2 else None) == 1, M
        L.gpt2_sync()
        pkg.check("%s fused M=%d" % (shape, M))
        assert np.array_equal(fused.numpy(np.uint16, (M, N)), add.numpy(np.uint16, (M, N))), M


@pytest.mark.parametrize("M,N,K", [(1345, 768, 768), (1350, 768, 3072), (673, 1500, 1024), (961, 1001, 768), (450, 2000, 2048), (193, 4096, 1024)])
def test_int8_gemm_about_one_tile_a_cu(pkg, L, M, N, K):
    """INT8 shapes with 256 64x64 tiles or just more, where the tile is picked for the INT8 weights alone: against the
    float64 product of the same code x scale values, bounds as above; rows past M stay untouched."""
    rng = np.random.default_rng(M + N + K)
    A = rng.standard_normal((M, K), dtype=np.float32).astype(np.float16)
    q = rng.integers(-127, 128, (N, K)).astype(np.int8)
    s = (rng.random(N, dtype=np.float32) + np.float32(0.5)) * np.float32(3e-4)
    b = (rng.standard_normal(N, dtype=np.float32) * np.float32(0.1)).astype(np.float16)
    ref = A.astype(np.float64) @ (q * s[:, None].astype(np.float64)).T + b.astype(np.float64)
    dA, dW, ds, db = (pkg.Dev.from_numpy(x) for x in (A, q, s, b))
    out = pkg.Dev.from_numpy(np.full((M + 1, N), np.float16(3.0)))
    L.gpt2_matmul_int8(out.ptr, dA.ptr, dW.ptr, ds.ptr, db.ptr, M, N, K)
    L.gpt2_sync()
    pkg.check("int8 gemm")
    got = out.numpy(np.float16, (M + 1, N))
    assert (got[M] == 3.0).all()
    err = np.abs(got[:M].astype(np.float64) - ref)
    assert (err <= 2.0 ** -11 * np.abs(ref) + 2.0 ** -14 * ref.std()).all(), err.max()
