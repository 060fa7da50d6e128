// gemm_skinny.hip -- C = A . W^T (+ bias) for a few rows of A (short prompts), on the MFMA units
// (gfx950).  Same contract as gpt2_matmul_tiled / gpt2_matmul_int8 (cuda/kernels_tiled.cu:24-53,
// cuda/kernels_quant.cu:38-67) for the GPT-2 trunk shapes (K = 768 or 3072, N a multiple of 16).
//
// With M in the tens the product is a weight stream, as the M = 1 GEMV is: W is 0.6-4.7 MB and the
// MFMA work is a fraction of a microsecond.  The tile pipeline (operands staged through an LDS ring,
// one barrier per k-tile, 32-column tiles: 24-96 work-groups for these shapes) spends several round
// trips where one suffices.  Here:
//   * A work-group owns 16 rows of W (one MFMA row block) and 16 rows of A; its four waves split K.
//     Grid = (N / 16) x ceil(M / 16): 48-192 work-groups per 16 rows of A.
//   * A wave brings its quarter of the rows of W and of A to LDS with direct loads of whole 128-byte pieces
//     of a row (64 bytes of int8 codes), all issued at once (one memory round trip; K = 3072 fp16: W
//     through a ring of six k-tiles, refilled as they are consumed), and multiplies each 64-wide k-tile as
//     it lands.  Loaded as fragments straight from memory, neighbouring lanes were rows apart and an
//     instruction took the address unit four times as long.  us per launch, fragments -> LDS: mlp-proj
//     fp16 M = 16 5.7 -> 3.7 (host-bound now), traced in the prefill 7.0 -> 5.2; INT8 M = 48 4.8 -> 4.1;
//     the whole prefill fp16 T = 17 330 -> 297, INT8 319 -> 304.
//   * What a wave multiplies it loaded itself, so nothing but its own loads is waited for (with the
//     LayerNorm prologue, A is normalized in registers, written to LDS and published by a barrier).  The
//     four waves' sums are added in LDS in wave order; wave 0 runs the epilogue: scale (INT8), bias,
//     then the elementwise op as the unfused sequence would apply it (epi_out).
//   * The LayerNorm prologue (QKV after LN1, fc after LN2) normalizes the block's 16 rows with the
//     LayerNorm kernel's arithmetic (ln_rows768: ln_row768's operations row by row, the rows'
//     reductions interleaved), so the result is bit-identical to the LayerNorm launch followed by
//     this kernel.  Its rows are loaded before the weights and normalized while the weight stream
//     is in flight.
#include <type_traits>

#include "common.h"

namespace g2 {

constexpr int SKN_W = 4;      // waves per work-group: K split four ways
constexpr int SKN_MB = 16;    // rows of A per work-group (the MFMA's B columns)
[[maybe_unused]] constexpr int SKN_TILE = SKN_MB * 128;   // LDS bytes per 64-wide k-tile of the A block

// f(t) for t = T0 .. T1 - 1, t a compile-time constant.
template <int T0, int T1, class F>
__device__ __forceinline__ void unroll_tiles(F f) {
    if constexpr (T0 < T1) {
        f(std::integral_constant<int, T0>{});
        unroll_tiles<T0 + 1, T1>(f);
    }
}

template <int K, bool QW, int EPI, bool LNP>
__device__ __forceinline__ void gemm_skinny_wg(uint16_t *__restrict__ C, const uint16_t *__restrict__ A,
                                               const void *__restrict__ Wv, const float *__restrict__ Ws,
                                               const uint16_t *__restrict__ bias, int M, int N, int nbn,
                                               const uint16_t *resid, const uint16_t *__restrict__ ln_g,
                                               const uint16_t *__restrict__ ln_b) {
#if defined(__HIP_DEVICE_COMPILE__)   // LDS address-space pointers exist only in the device pass
    constexpr int KT = K / 64;              // 64-wide k-tiles of the A block
    constexpr int WT = KT / SKN_W;          // a wave's share of them
    constexpr int WTILE = QW ? 1024 : 2048; // LDS bytes of a k-tile of the W block
    constexpr int WR = (QW || WT <= 6) ? WT : 6;   // W k-tiles in a wave's ring (fp16 K = 3072: all do not fit)
    constexpr int WI = WTILE / 1024, AI = 2;   // load instructions per k-tile: W, A
    static_assert(KT % SKN_W == 0, "a wave's share of K is whole 64-wide tiles");
    static_assert(!LNP || (K == GPT2_N_EMBD && EPI != EPI_RESID), "the LayerNorm prologue: K = 768, no residual");
    static_assert(WT * (AI + WI) < 64, "a wave's loads are counted");
    // A block [KT][16 rows][128 B] and the waves' W rings [WR][16 rows][128 or 64 B] (16-byte chunk c of row r
    // at slot c ^ (r & 7), or c ^ (r / 4 & 3)), then the sums of waves 1..3.  One LDS object: with several, the
    // compiler waits for every direct load in flight ahead of the first fragment read.
    __shared__ __attribute__((aligned(1024))) char lds[KT * SKN_TILE + SKN_W * WR * WTILE + (SKN_W - 1) * 64 * 16];
    f32x4 *const red = reinterpret_cast<f32x4 *>(lds + KT * SKN_TILE + SKN_W * WR * WTILE);

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lrow = lane & 15, g = lane >> 4;
    const int nb = blockIdx.x % nbn, mb = blockIdx.x / nbn;
    const int n0 = nb * 16, m0 = mb * SKN_MB;
    char *const xs = lds + wave * WT * SKN_TILE;                         // this wave's A tiles
    char *const ws = lds + KT * SKN_TILE + wave * WR * WTILE;            // and W ring

    // Loads, in this order (they complete in issue order): the LayerNorm prologue's rows and gamma / beta
    // (L2-resident, needed first), the epilogue operands, then the k-tiles.  Compiler barriers keep it.
    f16x4 lg[3], lb[3], lx[4][3];   // LayerNorm prologue: rows wave + 4 r; lane l: elements 256 i + 4 l ..
    if constexpr (LNP) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint16_t *xr = A + (size_t)min(m0 + wave + 4 * r, M - 1) * K;
#pragma unroll
            for (int i = 0; i < 3; ++i) lx[r][i] = *reinterpret_cast<const f16x4 *>(xr + 256 * i + 4 * lane);
        }
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            lg[i] = *reinterpret_cast<const f16x4 *>(ln_g + 256 * i + 4 * lane);
            lb[i] = *reinterpret_cast<const f16x4 *>(ln_b + 256 * i + 4 * lane);
        }
        asm volatile("" ::: "memory");
    }
    // the lane's outputs C[m][nbase .. nbase+3]: scales, bias and residual (rows past M read row M-1
    // and store nothing; the residual may alias C: this lane alone writes those elements)
    const int nbase = n0 + 4 * g, m = m0 + lrow;
    float sc[4];
    uint32_t bs[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        sc[i] = 1.f;
        if constexpr (QW) sc[i] = Ws[nbase + i];
        bs[i] = *(bias ? bias + nbase + i : A);
    }
    uint2 rs = {0u, 0u};
    if constexpr (EPI == EPI_RESID) rs = *reinterpret_cast<const uint2 *>(resid + (size_t)min(m, M - 1) * N + nbase);
    asm volatile("" ::: "memory");
    // k-tile t of this wave's share: A rows 8 q .. + 7 (lane l slot l & 7 of row 8 q + l / 8), W the same
    // way or, int8, 16 rows of 64 bytes an instruction (lane l slot l & 3 of row l / 4); N % 16 == 0, so
    // every row of W exists
    const int r8 = lane >> 3, c8 = ((lane & 7) ^ r8) * 8;
    const int r4 = lane >> 2, c4 = ((lane & 3) ^ ((r4 >> 2) & 3)) * 16;
    auto issue_a = [&](int t) {
#pragma unroll
        for (int q = 0; q < 2; ++q)
            __builtin_amdgcn_global_load_lds(A + (size_t)min(m0 + 8 * q + r8, M - 1) * K + 64 * (wave * WT + t) + c8,
                                             G2_LDS(xs + t * SKN_TILE + 1024 * q), 16, 0, 0);
    };
    auto issue_w = [&](int t) {
        const int k0 = 64 * (wave * WT + t);
        char *dst = ws + (t % WR) * WTILE;
        if constexpr (QW) {
            __builtin_amdgcn_global_load_lds(reinterpret_cast<const int8_t *>(Wv) + (size_t)(n0 + r4) * K + k0 + c4,
                                             G2_LDS(dst), 16, 0, 0);
        } else {
#pragma unroll
            for (int q = 0; q < 2; ++q)
                __builtin_amdgcn_global_load_lds(reinterpret_cast<const uint16_t *>(Wv) + (size_t)(n0 + 8 * q + r8) * K + k0 + c8,
                                                 G2_LDS(dst + 1024 * q), 16, 0, 0);
        }
    };
    if constexpr (LNP) {
        // The prologue form takes W through registers, lane for lane what the direct loads would have put in
        // LDS: with direct loads in flight the compiler counts no ordinary load exactly, and the LayerNorm
        // would start when W has landed instead of running meanwhile.
        i32x4 wl[WT * WI];
#pragma unroll
        for (int t = 0; t < WT; ++t)
#pragma unroll
            for (int q = 0; q < WI; ++q) {
                const int k0 = 64 * (wave * WT + t);
                wl[t * WI + q] = QW ? *reinterpret_cast<const i32x4 *>(reinterpret_cast<const int8_t *>(Wv) + (size_t)(n0 + r4) * K + k0 + c4)
                                    : *reinterpret_cast<const i32x4 *>(reinterpret_cast<const uint16_t *>(Wv) +
                                                                       (size_t)(n0 + 8 * q + r8) * K + k0 + c8);
            }
        asm volatile("" ::: "memory");
        // the LayerNorm's inputs pass through here, so none of its arithmetic is scheduled ahead of
        // the loads above (the compiler would otherwise issue the weight loads after it)
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int i = 0; i < 3; ++i) asm volatile("" : "+v"(lx[r][i]) : : "memory");
        // normalized as the LayerNorm kernel does, written where a direct-to-LDS load would have put them
        f16x4 o[4][3];
        ln_rows768<4>(lx, lg, lb, o);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = wave + 4 * r;
#pragma unroll
            for (int i = 0; i < 3; ++i)   // element 256 i + 4 lane: k-tile 4 i + lane / 16, chunk (lane & 15) / 2
                *reinterpret_cast<f16x4 *>(lds + (4 * i + (lane >> 4)) * SKN_TILE + row * 128 +
                                           ((((lane & 15) >> 1) ^ (row & 7)) << 4) + (lane & 1) * 8) = o[r][i];
        }
        asm volatile("" ::: "memory");   // W is waited for here, not inside the LayerNorm
#pragma unroll
        for (int i = 0; i < WT * WI; ++i) *reinterpret_cast<i32x4 *>(ws + 1024 * i + 16 * lane) = wl[i];
        lds_barrier();
    } else {
#pragma unroll
        for (int t = 0; t < WR; ++t) {
            issue_a(t);
            issue_w(t);
        }
#pragma unroll
        for (int t = WR; t < WT; ++t) issue_a(t);
    }

    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    auto consume = [&](int t) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int c = 4 * s + g;   // 16-byte chunk of the lane's eight k
            f16x8 w;
            if constexpr (QW) {
                const char *p = ws + (t % WR) * WTILE + lrow * 64 + (((c >> 1) ^ ((lrow >> 2) & 3)) << 4) + 8 * (c & 1);
                w = i8x8_to_f16x8(*reinterpret_cast<const uint2 *>(p));
            } else {
                w = *reinterpret_cast<const f16x8 *>(ws + (t % WR) * WTILE + lrow * 128 + ((c ^ (lrow & 7)) << 4));
            }
            const f16x8 x = *reinterpret_cast<const f16x8 *>(xs + t * SKN_TILE + lrow * 128 + ((c ^ (lrow & 7)) << 4));
            acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(w, x, acc, 0, 0, 0);
        }
    };
    // tile t has landed when at most the loads issued behind its last one are outstanding: the rest of the
    // first WR tiles, the later A tiles, and the refills since
    static_assert(WT == WR || WT == 2 * WR, "every slot of the ring is refilled once, or never");
    unroll_tiles<0, WT>([&](auto tc) {
        constexpr int t = decltype(tc)::value;
        if constexpr (!LNP) {
            wait_vm<t < WR ? (WR - 1 - t) * (AI + WI) + (WT - WR) * AI + (WT > WR ? t * WI : 0) : (WT - 1 - t) * WI>();
            asm volatile("" ::: "memory");
        }
        consume(t);
        if constexpr (t + WR < WT) {
            // the slot's fragments have been read before the refill goes out
            asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(acc) : : "memory");
            issue_w(t + WR);
        }
    });
    // lane holds D[n0 + 4g + i][m0 + lrow]; waves 1..3 hand theirs to wave 0, added in wave order
    if (wave > 0) red[(wave - 1) * 64 + lane] = acc;
    lds_barrier();
    if (wave != 0) return;
#pragma unroll
    for (int w = 0; w < SKN_W - 1; ++w) acc += red[w * 64 + lane];
    if (m >= M) return;
    uint16_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float v = acc[i];
        if constexpr (QW) v = v * sc[i];
        const uint16_t r = (uint16_t)((i < 2 ? rs.x : rs.y) >> (16 * (i & 1)));
        o[i] = epi_out<EPI>(v + (bias ? h2f((uint16_t)bs[i]) : 0.f), r);
    }
    *reinterpret_cast<uint2 *>(C + (size_t)m * N + nbase) =
        uint2{(uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16)};
#endif
}

// The pointers reach the body as __restrict__ parameters of an inlined function, so the compiler knows that
// its LDS reads do not alias the direct loads in flight (it would wait for them ahead of every read).
template <int K, bool QW, int EPI, bool LNP>
__global__ __launch_bounds__(64 * SKN_W) void k_gemm_skinny(uint16_t *__restrict__ C, const uint16_t *__restrict__ A,
                                                            const void *__restrict__ Wv, const float *__restrict__ Ws,
                                                            const uint16_t *__restrict__ bias, int M, int N, int nbn,
                                                            const uint16_t *resid, const uint16_t *__restrict__ ln_g,
                                                            const uint16_t *__restrict__ ln_b) {
    gemm_skinny_wg<K, QW, EPI, LNP>(C, A, Wv, Ws, bias, M, N, nbn, resid, ln_g, ln_b);
}

typedef void (*SkinnyFn)(uint16_t *, const uint16_t *, const void *, const float *, const uint16_t *, int, int, int,
                         const uint16_t *, const uint16_t *, const uint16_t *);

// [K = 768, 3072][fp16, INT8][epilogue: none, gelu, residual, LayerNorm + none, LayerNorm + gelu]
#define G2_SKN(K, QW) \
    {k_gemm_skinny<K, QW, EPI_NONE, false>, k_gemm_skinny<K, QW, EPI_GELU, false>, k_gemm_skinny<K, QW, EPI_RESID, false>, \
     K == GPT2_N_EMBD ? k_gemm_skinny<GPT2_N_EMBD, QW, EPI_NONE, true> : nullptr,                                       \
     K == GPT2_N_EMBD ? k_gemm_skinny<GPT2_N_EMBD, QW, EPI_GELU, true> : nullptr}
static const SkinnyFn kSkinny[2][2][5] = {{G2_SKN(768, false), G2_SKN(768, true)},
                                          {G2_SKN(3072, false), G2_SKN(3072, true)}};

// Rows of A up to which the skinny kernel takes the trunk shapes.  Whole prefill on MI355X, interleaved A/B,
// tiles with the LayerNorm fold over the skinny kernel with its prologue: INT8 weights 1.38 at T = 8, 1.36 at
// 16, 1.20 at 24-32, 1.13 at 40-48, 1.07 at 64, 1.03 at 80, 0.86 at 96; fp16 1.32 at 8-16, 1.22 at 24-32, 1.13 at
// 40-48, 1.10 at 64, 1.04 at 80, 0.93 at 96.  The limits are lower than those crossings: they were set when
// the kernel took its operands as fragments from memory (fp16 then lost from 40 rows on).
// gpt2_tune_gemm_skinny overrides both (0: never).
static int g_skinny_max = -1;    // -1: the measured default per weight format
static int g_skinny_calls = 0;   // launches so far (test hook)
int skinny_max_m(bool qw) { return g_skinny_max >= 0 ? g_skinny_max : (qw ? 64 : 32); }

// C = A . W^T (+ bias), then epi (EPI_GELU; EPI_RESID: C = resid + product, resid may be C); with
// ln_g / ln_b, A is first normalized row by row (LayerNorm, K = 768).  Returns false (nothing
// launched) outside its domain: M in [2, skinny_max_m(qw)], K 768 or 3072, N % 16 == 0, 16-byte
// aligned A and W, 8-byte aligned C (and residual, gamma, beta).
bool gemm_skinny(uint16_t *C, const uint16_t *A, const void *W, const float *Ws, const uint16_t *bias, int M, int N,
                 int K, bool qw, int epi, const uint16_t *resid, const uint16_t *ln_g, const uint16_t *ln_b) {
    if (M < 2 || M > skinny_max_m(qw) || N <= 0 || N % 16 || (K != 768 && K != 3072)) return false;
    if (!A || !W || !C || !aligned16(A) || !aligned16(W) || ((uintptr_t)C & 7u) || (qw && !Ws)) return false;
    int e = epi == EPI_NONE ? 0 : epi == EPI_GELU ? 1 : epi == EPI_RESID ? 2 : -1;
    if (e < 0 || (e == 2 && (!resid || ((uintptr_t)resid & 7u)))) return false;
    if (ln_g || ln_b) {
        if (!ln_g || !ln_b || e == 2 || K != GPT2_N_EMBD || (((uintptr_t)ln_g | (uintptr_t)ln_b) & 7u)) return false;
        e += 3;
    }
    const SkinnyFn fn = kSkinny[K == 768 ? 0 : 1][qw ? 1 : 0][e];
    if (!fn) return false;
    const int nbn = N / 16;
    hipLaunchKernelGGL(fn, dim3(nbn * cdiv(M, SKN_MB)), dim3(64 * SKN_W), 0, stream(), C, A, W, Ws, bias, M, N, nbn,
                       resid, ln_g, ln_b);
    check_launch("k_gemm_skinny");
    ++g_skinny_calls;
    return true;
}

}  // namespace g2

// Tuning/test hooks (no reference counterpart): the largest M the skinny kernel takes (0: off, -1:
// the default), the limit in force for fp16 (qw = 0) or INT8 weights, and the number of its
// launches so far.
extern "C" void gpt2_tune_gemm_skinny(int max_m) { g2::g_skinny_max = max_m < 0 ? -1 : max_m; }
extern "C" int gpt2_tune_gemm_skinny_max(int qw) { return g2::skinny_max_m(qw != 0); }
extern "C" int gpt2_tune_gemm_skinny_calls(void) { return g2::g_skinny_calls; }
