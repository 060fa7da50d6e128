// attn_prefill.hip -- the causal prefill attention launch (gfx950): one work-group per block of 16 or 32
// queries of one head.  Replaces the reference's fused attention (cuda/kernels_fused.cu:58-140; semantics of
// cpu/forward_cpu.c:83-116).
//
// The fragment layout, softmax and results are attn_block's (attn_prefill.h, the block of the persistent
// prefill).  What differs is how keys and values arrive: by direct-to-LDS loads of whole 128-byte rows,
// eight rows an instruction, one 32-key chunk ahead of the one in use.  attn_block loads key fragments straight from
// qkv, where neighbouring lanes lie 4608 bytes apart and an instruction takes the address unit four times
// as long; that, not memory, bounded it (6.7 us at 512 queries against 5.0, 10.0 against 6.8 at 777).
// The 16-byte chunks of a row are XOR-swizzled by the row (by choosing what each lane fetches), so neither
// the key reads nor the transposing value reads meet a bank conflict.  A wave's ring is its own: no
// barrier until the waves' states are merged.
// MI355X, us a launch, one / two tiles of 16 queries a block: T = 256 3.7 / 4.5, 512 5.0 / 5.9, 777 6.8 /
// 7.8, 896 7.9 / 8.3, 1024 9.5 / 8.9 (from 13.4).  Two tiles halve the key and value bytes per query but also
// the work-groups (708 of one tile at 929 queries, 360 of two; the chip holds 512): the two cross between 896 and
// 1024, and at 928 the one-tile launch takes 8.5 where the two-tile one at 929 takes 8.8.
#include "attn_prefill.h"

namespace g2 {

constexpr int AF_CK = 32;                       // keys per chunk
constexpr int AF_W = 4;                         // waves: chunk c goes to wave c % 4
constexpr int AF_TILE = AF_CK * 128;            // bytes of a chunk's keys (or values)
[[maybe_unused]] constexpr int AF_RING = 2 * 2 * AF_TILE;   // a wave's two stages of keys and values
constexpr int AF_T2 = 928;                      // prompts longer than this take two query tiles a block

// Eight halves from p; aligned: p is 16-byte aligned.
template <bool ALIGNED>
__device__ __forceinline__ f16x8 load_half8(const uint16_t *p) {
    f16x8 v;
    if constexpr (ALIGNED) v = *reinterpret_cast<const f16x8 *>(p);
    else __builtin_memcpy(&v, p, 16);
    return v;
}

// The pointers are __restrict__ parameters of an inlined function, which tells the compiler that the LDS
// reads below do not alias the direct loads in flight (it would wait for them ahead of every read).
// DIRECT = false takes keys and values through registers, for a qkv that is not 16-byte aligned: direct-to-LDS
// loads of 16 bytes are only issued at 16-byte aligned addresses.  Same values in the same places, same bits.
template <int QT, bool DIRECT>
__device__ __forceinline__ void attn_tiles(uint16_t *__restrict__ att, const uint16_t *__restrict__ qkv, int T,
                                           uint16_t *__restrict__ Kc, uint16_t *__restrict__ Vc, int maxT, int h, int qb) {
#if defined(__HIP_DEVICE_COMPILE__)   // LDS address-space pointers exist only in the device pass
    constexpr int E = GPT2_N_EMBD, D = GPT2_HEAD_DIM, S3 = 3 * GPT2_N_EMBD;
    constexpr int QB = 16 * QT;                  // queries of the block
    static_assert(D == 64 && AF_CK == 32 && AF_CK % QB == 0, "the layout, and the mask below, are for these sizes");
    __shared__ __attribute__((aligned(1024))) char smem[AF_W * AF_RING];
    constexpr int MRG_O = QT * 4 * 64 * 16;      // a wave's merge state: [query tile][dim group][lane] f32x4
    static_assert(AF_W * (MRG_O + 2 * QB * 4) <= AF_W * AF_RING, "the merge reuses the rings");

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int jq = lane & 15, g = lane >> 4;
    const int q0 = qb * QB;
    const int nc = q0 / AF_CK + 1;               // chunks over keys [0, last query]
    char *const ring = smem + wave * AF_RING;
    const uint16_t *Kb = qkv + E + h * D, *Vb = qkv + 2 * E + h * D;

    // chunk c into stage s: instruction i brings rows 8 i .. + 7, lane l chunk (l & 7) ^ (l >> 3) of row
    // 8 i + l / 8; rows past T read the last row (masked: they lie past every stored query)
    const int lr = lane >> 3, lc = ((lane & 7) ^ lr) * 8;
    auto issue = [&](int c, int s) {
        char *dst = ring + s * 2 * AF_TILE;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const size_t row = (size_t)min(c * AF_CK + 8 * i + lr, T - 1) * S3 + lc;
            if constexpr (DIRECT) __builtin_amdgcn_global_load_lds(Kb + row, G2_LDS(dst + 1024 * i), 16, 0, 0);
            else *reinterpret_cast<f16x8 *>(dst + 1024 * i + 16 * lane) = load_half8<false>(Kb + row);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const size_t row = (size_t)min(c * AF_CK + 8 * i + lr, T - 1) * S3 + lc;
            if constexpr (DIRECT) __builtin_amdgcn_global_load_lds(Vb + row, G2_LDS(dst + AF_TILE + 1024 * i), 16, 0, 0);
            else *reinterpret_cast<f16x8 *>(dst + AF_TILE + 1024 * i + 16 * lane) = load_half8<false>(Vb + row);
        }
    };

    // The wave's first two chunks, then the queries, then the rows that the cache fill copies (a thread one
    // 16-byte chunk of K and of V, with one tile the upper half of the threads repeats the lower's; stored at the end).
    if (wave < nc) issue(wave, 0);
    if (wave + AF_W < nc) issue(wave + AF_W, 1);
    asm volatile("" ::: "memory");
    f16x8 qf[QT][2];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
        const uint16_t *Qp = qkv + (size_t)min(q0 + 16 * qt + jq, T - 1) * S3 + h * D;
        qf[qt][0] = load_half8<DIRECT>(Qp + 8 * g);
        qf[qt][1] = load_half8<DIRECT>(Qp + 32 + 8 * g);
    }
    const int ft = q0 + ((threadIdx.x >> 3) & (QB - 1)), fd = (threadIdx.x & 7) * 8;
    f16x8 fk = {}, fv = {};
    static_assert(64 * AF_W >= QB * 8, "a thread per 16-byte chunk");
    if (Kc) {
        const uint16_t *src = qkv + (size_t)min(ft, T - 1) * S3 + E + h * D + fd;
        fk = load_half8<DIRECT>(src);
        fv = load_half8<DIRECT>(src + E);
    }
    asm volatile("" ::: "memory");

    float m[QT], lsum[QT];
    f32x4 o[QT][4];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
        m[qt] = -INFINITY;
        lsum[qt] = 0.f;
#pragma unroll
        for (int dg = 0; dg < 4; ++dg) o[qt][dg] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    constexpr float SL2 = 0.125f * 1.4426950408889634f;     // 1/sqrt(64) * log2(e)

    int stage = 0;
    for (int c = wave; c < nc; c += AF_W) {
        if (c + AF_W < nc) wait_vm<8>();
        else wait_vm<0>();
        asm volatile("" ::: "memory");
        const char *kt = ring + stage * 2 * AF_TILE, *vt = kt + AF_TILE;
        // ---- scores of keys 32 c + 16 t + 4 g + r for query q0 + 16 qt + jq
        f32x4 s[QT][2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const char *kr = kt + (16 * t + jq) * 128;
            const f16x8 k0 = *reinterpret_cast<const f16x8 *>(kr + ((g ^ (jq & 7)) << 4));
            const f16x8 k1 = *reinterpret_cast<const f16x8 *>(kr + (((4 + g) ^ (jq & 7)) << 4));
#pragma unroll
            for (int qt = 0; qt < QT; ++qt) {
                s[qt][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(k0, qf[qt][0], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                s[qt][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(k1, qf[qt][1], s[qt][t], 0, 0, 0);
            }
        }
        // Only the last chunk reaches past a query of the block; its first key reaches past none, so every
        // query has a finite score in every chunk.
        if (c == nc - 1) {
#pragma unroll
            for (int qt = 0; qt < QT; ++qt)
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (c * AF_CK + 16 * t + 4 * g + r > q0 + 16 * qt + jq) s[qt][t][r] = -INFINITY;
        }
        f16x8 pb[QT];
        float corr[QT];
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) {
            float mx = fmaxf(fmaxf(fmaxf(s[qt][0][0], s[qt][0][1]), fmaxf(s[qt][0][2], s[qt][0][3])),
                             fmaxf(fmaxf(s[qt][1][0], s[qt][1][1]), fmaxf(s[qt][1][2], s[qt][1][3])));
            mx = group_max(mx);
            const float mnew = fmaxf(m[qt], mx * SL2);
            corr[qt] = exp2_raw(m[qt] - mnew);   // 0 on the wave's first chunk
            m[qt] = mnew;
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) pb[qt][4 * t + r] = (f16)exp2_raw(fmaf(s[qt][t][r], SL2, -mnew));
            // the denominator sums exactly the fp16 probabilities the MFMA multiplies
            float ps = 0.f;
#pragma unroll
            for (int e = 0; e < 8; e += 2) ps = __builtin_amdgcn_fdot2(f16x2{pb[qt][e], pb[qt][e + 1]}, f16x2{1, 1}, ps, false);
            lsum[qt] = fmaf(lsum[qt], corr[qt], ps);
        }
        // ---- O^T += V^T . P: the k-slots of lane group g are keys 4g .. + 3 and 16 + 4g .. + 3, those that
        // the lane holds P for; lane jq = 4 r + a names 4 dims of key (base + r) and receives dim jq of 4 keys
        const int vr = jq >> 2, row = 4 * g + vr;
#pragma unroll
        for (int dg = 0; dg < 4; ++dg) {
            const int ch = 2 * dg + ((jq & 3) >> 1), sub = 8 * (jq & 1);
            const f16x4 lo = tr_read(vt + row * 128 + ((ch ^ (row & 7)) << 4) + sub);
            const f16x4 hi = tr_read(vt + (16 + row) * 128 + ((ch ^ (row & 7)) << 4) + sub);
            const f16x8 va = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
            for (int qt = 0; qt < QT; ++qt)
                o[qt][dg] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va, pb[qt], o[qt][dg] * corr[qt], 0, 0, 0);
        }
        // the stage is refilled once its reads are done
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (c + 2 * AF_W < nc) issue(c + 2 * AF_W, stage);
        stage ^= 1;
    }
    // ---- merge the waves' states: wave w finishes dims 16 w .. + 15 of every query
    lds_barrier();   // the rings are idle
    float *const mrg_m = reinterpret_cast<float *>(smem + AF_W * MRG_O), *const mrg_l = mrg_m + AF_W * QB;
    f32x4 *const mrg_o = reinterpret_cast<f32x4 *>(smem);   // [wave][query tile][dim group][lane]
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
        const float l = group_sum(lsum[qt]);
        if (g == 0) {
            mrg_m[wave * QB + 16 * qt + jq] = m[qt];
            mrg_l[wave * QB + 16 * qt + jq] = l;
        }
#pragma unroll
        for (int dg = 0; dg < 4; ++dg) mrg_o[((wave * QT + qt) * 4 + dg) * 64 + lane] = o[qt][dg];
    }
    if (Kc && ft < T) {
        const size_t at = ((size_t)h * maxT + ft) * D + fd;
        *reinterpret_cast<f16x8 *>(Kc + at) = fk;
        *reinterpret_cast<f16x8 *>(Vc + at) = fv;
    }
    lds_barrier();
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
        float mw[AF_W], lw[AF_W], mmax = -INFINITY;
#pragma unroll
        for (int u = 0; u < AF_W; ++u) {
            mw[u] = mrg_m[u * QB + 16 * qt + jq];
            lw[u] = mrg_l[u * QB + 16 * qt + jq];
            mmax = (lw[u] != 0.f) ? fmaxf(mmax, mw[u]) : mmax;   // wave 0 always has keys
        }
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        float L = 0.f;
#pragma unroll
        for (int u = 0; u < AF_W; ++u) {
            const float f = (lw[u] != 0.f) ? exp2_raw(mw[u] - mmax) : 0.f;
            L += lw[u] * f;
            acc += mrg_o[((u * QT + qt) * 4 + wave) * 64 + lane] * f;
        }
        const int q = q0 + 16 * qt + jq;
        if (q < T) {
            const float inv = 1.0f / L;
            *reinterpret_cast<uint2 *>(att + (size_t)q * E + h * D + 16 * wave + 4 * g) =
                uint2{(uint32_t)f2h(acc[0] * inv) | ((uint32_t)f2h(acc[1] * inv) << 16),
                      (uint32_t)f2h(acc[2] * inv) | ((uint32_t)f2h(acc[3] * inv) << 16)};
        }
    }
#endif
}

template <int QT, bool DIRECT>
__global__ __launch_bounds__(64 * AF_W) void k_attn_prefill(uint16_t *__restrict__ att, const uint16_t *__restrict__ qkv,
                                                            int T, uint16_t *__restrict__ Kc, uint16_t *__restrict__ Vc,
                                                            int maxT) {
    // XCD-aware assignment (work-group b runs on XCD b % 8): XCD x takes every query block of head
    // x and every other block of head 8 + x/2, so its L2 holds the keys and values of 1.5 heads
    // instead of all 12.  Within an XCD the blocks go heaviest first (qi = rank from the last block).
    const int nb = (T + 16 * QT - 1) / (16 * QT);
    int h, qi;
    {
        const int x = blockIdx.x & 7, k = blockIdx.x >> 3, i3 = k / 3, r3 = k - 3 * i3;
        if (r3 < 2) {
            h = x;
            qi = 2 * i3 + r3;
        } else {
            h = 8 + (x >> 1);
            qi = 2 * i3 + (x & 1);
        }
    }
    if (qi >= nb) return;                      // the grid is rounded up (whole work-group leaves)
    attn_tiles<QT, DIRECT>(att, qkv, T, Kc, Vc, maxT, h, nb - 1 - qi);
}

// Kc, Vc (optional): the layer's K and V cache planes ([H][maxT][D]), filled with this prompt's rows
// (the prefill scatter of cuda/kvcache.cu:66-81, done inside the attention launch).
void attention_prefill(uint16_t *att, const uint16_t *qkv, int T, uint16_t *Kc, uint16_t *Vc, int maxT) {
    static_assert(GPT2_N_HEAD == 12, "the XCD assignment covers 12 heads on 8 XCDs");
    // gpt2_attention_flash refuses an unaligned qkv; a prefill's own scratch may have one
    const bool direct = aligned16(qkv);
    const int qt = direct && T > AF_T2 ? 2 : 1;
    const auto fn = !direct ? k_attn_prefill<1, false> : qt == 2 ? k_attn_prefill<2, true> : k_attn_prefill<1, true>;
    hipLaunchKernelGGL(fn, dim3(8 * 3 * cdiv(cdiv(T, 16 * qt), 2)), dim3(64 * AF_W), 0, stream(), att, qkv, T, Kc, Vc, maxT);
    check_launch("k_attn_prefill");
}

}  // namespace g2
