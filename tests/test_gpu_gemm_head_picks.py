"""The GEMM with a vocabulary-sized N at both sides of every row count where its tiles change, with rows of the
output that start at every 2-byte offset."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROWS = (33, 64, 65, 127, 128, 129, 192, 193, 256, 257, 320, 321, 384, 385, 448, 449, 577)


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("N", [16384, 16385, 32771])
def test_head_gemm_at_pick_edges(pkg, L, N, int8):
    """Against the float64 product of the same fp16 (INT8: code x scale) values, K = 192: the fp32 sums are off
    by less than 192 * 2^-24 of the sum of the terms' magnitudes, bounded here by 2^-14 of the results' spread
    (a sum of 192 random terms spreads by 1/11 of that sum), and the fp16 output by half an ulp, 2^-11 of the
    value.  The value past the last row stays untouched."""
    K = 192
    rng = np.random.default_rng(N + int8)
    A = rng.standard_normal((max(ROWS), K), dtype=np.float32).astype(np.float16)
    W = (rng.standard_normal((N, K), dtype=np.float32) * np.float32(0.05)).astype(np.float16)
    b = (rng.standard_normal(N, dtype=np.float32) * np.float32(0.1)).astype(np.float16)
    Wd, sp = W.astype(np.float64), None
    if int8:
        s = (np.abs(W.astype(np.float32)).max(axis=1) / np.float32(127.0)).astype(np.float32)
        q = np.clip(np.rint(W.astype(np.float32) / s[:, None]), -127, 127).astype(np.int8)
        Wd, sp = q.astype(np.float64) * s[:, None].astype(np.float64), pkg.Dev.from_numpy(s)
    ref = A.astype(np.float64) @ Wd.T + b.astype(np.float64)
    tol = 2.0 ** -11 * np.abs(ref) + 2.0 ** -14 * ref.std()
    dA, dW, db = (pkg.Dev.from_numpy(x) for x in (A, q if int8 else W, b))
    out = pkg.Dev((max(ROWS) + 1) * N * 2)
    mark = np.full(N, np.float16(3.0))
    for M in ROWS:
        assert L.gpt2_h2d(out.at(M * N * 2), mark.ctypes.data, mark.nbytes) == 0
        if int8:
            L.gpt2_matmul_int8(out.ptr, dA.ptr, dW.ptr, sp.ptr, db.ptr, M, N, K)
        else:
            L.gpt2_matmul_tiled(out.ptr, dA.ptr, dW.ptr, db.ptr, M, N, K)
        L.gpt2_sync()
        pkg.check("N=%d M=%d" % (N, M))
        got = out.numpy(np.float16, (M + 1, N))
        assert (got[M] == 3.0).all(), M
        err = np.abs(got[:M].astype(np.float64) - ref[:M])
        assert (err <= tol[:M]).all(), (M, err.max())
