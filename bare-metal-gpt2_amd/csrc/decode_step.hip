// decode_step.hip -- the kernels of the multi-kernel decode step (gpt2_decode_step_cuda and the
// GPT2_DECODE_MULTI graph) for the backends whose GEMV slots are this library's GEMVs (gfx950).
//
// One token is four launches a layer and one for the head (cuda/kvcache.cu:233-269 in the reference):
//   k_step_attn   LN1, q/k/v, K/V append and a quarter of one head's attention: 48 work-groups
//   k_step_proj   merge of the quarters, attn-proj rows, bias, residual
//   k_step_fc     LN2, fc rows, bias, gelu
//   k_step_mlp    mlp-proj rows, bias, residual
//   k_step_head   LN_f and the rows of the tied head
// Layer 0's k_step_attn also embeds the token.  Every launch here is bound by latency, not by bytes (a
// layer's weights are 14 MB in fp16: 2.8 us at the copy rate, spread over four launches), so what the
// design keeps short is the chain inside a launch: every load a work-group needs (activations first,
// then weights, then keys and values) is issued before the first wait, each dot product runs on
// registers already loaded, and one token's attention of a head runs on four CUs instead of one.
//
// Weights come ahead of their launch: no launch fills 256 CUs (k_step_attn runs on 48), so each carries
// extra work-groups that only read what later launches will read, on the XCD that will read it
// (work-group b runs on XCD b % 8, in every launch; a clean line stays in its XCD's L2 across
// launches: 97 ns a dependent load in the next launch against 380 from memory).  A work-group placed
// elsewhere would cost only the speed.
//
// The quarters of a head meet in memory: k_step_attn leaves (m, l, c[64], its part of q.k_new) in fp32
// and its slice of v_new in buffers of the caller's scratch that the step has no other use for at that
// point (StepPart), so steps on different scratch never share a word.
//
// Numerics: fp16 activations between the launches, fp32 inside, LayerNorm through ln_row768 (the LayerNorm
// kernel's arithmetic); a matmul's scale, bias, gelu and residual apply in fp32 ahead of its one rounding;
// softmax weights and partial contexts stay fp32 throughout.
#include <cmath>

#include "attn.h"
#include "common.h"
#include "decode_step.h"

namespace g2 {

constexpr int SP_E = GPT2_N_EMBD, SP_D = GPT2_HEAD_DIM, SP_H = GPT2_N_HEAD, SP_S = STEP_SPLITS;
constexpr int SP_KS = SP_D / SP_S;              // rows of k_new and v_new per split
constexpr int SP_R = SP_D + 2 * SP_KS;          // q/k/v rows a split computes: q (64), its k and v slices
constexpr int SP_WAVES = 8;                     // waves of k_step_attn with rows and keys (wave 0 has the LayerNorm)
constexpr int SP_KEYS = (GPT2_N_CTX + SP_S * SP_WAVES - 1) / (SP_S * SP_WAVES);   // keys per wave, at most
constexpr int SP_U = SP_R / SP_WAVES / 4;       // passes of four rows per wave
static_assert(SP_U * SP_WAVES * 4 == SP_R && SP_KEYS % 8 == 0 && SP_S == 4, "step layout");

// Four weight rows of 768 in a wave, 16 lanes a row: lane j of a row holds its 16-byte chunks j, j + 16, ..,
// so a load instruction reads 256 contiguous bytes of each row.  (As MFMA A-fragments, lane = row,
// neighbouring lanes lie 1536 bytes apart and an instruction takes four times the cycles of the address
// unit: 3.0 us against 1.1 to issue k_step_attn's loads.)  The products are few (72 v_dot2 a lane there).
template <bool QW>
struct Rows4 {
    static constexpr int NL = QW ? 3 : 6;
    i32x4 w[NL];
    __device__ __forceinline__ void load(const void *W, size_t row, int lane) {
        const char *src = reinterpret_cast<const char *>(W) + row * SP_E * (QW ? 1 : 2) + (lane & 15) * 16;
#pragma unroll
        for (int i = 0; i < NL; ++i) w[i] = *reinterpret_cast<const i32x4 *>(src + 256 * i);
    }
    __device__ __forceinline__ float dot(const f16x8 (&x)[6]) const {   // every lane of the row gets the sum
        float acc = 0.f;
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            if constexpr (QW) acc = dot16q(w[i], x[2 * i], x[2 * i + 1], acc);
            else acc = dot8(w[i], x[i], acc);
        }
        return row16_sum(acc);
    }
};
// The elements of x that meet a lane's chunks.
template <bool QW>
__device__ __forceinline__ void load_x(f16x8 (&x)[6], const f16 *xn, int lane) {
    const int j = lane & 15;
#pragma unroll
    for (int v = 0; v < 6; ++v)
        x[v] = *reinterpret_cast<const f16x8 *>(xn + (QW ? (j + 16 * (v >> 1)) * 16 + (v & 1) * 8 : (j + 16 * v) * 8));
}

// The LayerNorm of a 768-wide row by one wave (lane l: elements 256 i + 4 l .. + 3), left in LDS.  It has a
// wave to itself: a wave that first issues its share of the weight loads cannot look at x before
// the last of them is accepted.
struct LnRow {
    f16x4 x[3], g[3], b[3];
    __device__ __forceinline__ void load(const uint16_t *row, const uint16_t *gamma, const uint16_t *beta, int lane) {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            x[i] = *reinterpret_cast<const f16x4 *>(row + 256 * i + 4 * lane);
            g[i] = *reinterpret_cast<const f16x4 *>(gamma + 256 * i + 4 * lane);
            b[i] = *reinterpret_cast<const f16x4 *>(beta + 256 * i + 4 * lane);
        }
    }
    __device__ __forceinline__ void normalize(f16 *xn, int lane) {
        f16x4 o[3];
        ln_row768(x, g, b, o);
#pragma unroll
        for (int i = 0; i < 3; ++i) *reinterpret_cast<f16x4 *>(xn + 256 * i + 4 * lane) = o[i];
    }
};

// Reads bytes [0, bytes) of p (both multiples of 16) into the L2, the work-group's threads each up to N
// 16-byte pieces, all in flight at once.
template <int N>
__device__ __forceinline__ void read_ahead(const char *p, int bytes) {
    i32x4 v[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int at = ((int)threadIdx.x + (int)blockDim.x * i) * 16;
        v[i] = *reinterpret_cast<const i32x4 *>(p + min(at, bytes - 16));
    }
#pragma unroll
    for (int i = 0; i < N; ++i) asm volatile("" ::"v"(v[i]));   // the loads have a user
}

// Row r of the q/k/v rows of (head h, split sp) in the [2304][768] weight: rows 0-63 the head's q, then the
// split's slices of k and of v.
static_assert(SP_KS == 16 && SP_D == 64, "a slice is 16 rows");
__device__ __forceinline__ int step_qkv_row(int h, int sp, int r) {
    const int b = r >> 4;
    return h * SP_D + 16 * (b < 4 ? b : sp) + SP_E * max(b - 3, 0) + (r & 15);
}

// Reads ahead what the six (head, split) work-groups of XCD i % 8 in the next k_step_attn will read of the
// q/k/v weight: its own head's 3 x 64 rows, the shared head's 64 q rows and half of its k and v rows, 320
// rows in 16 shares (two launches of 64 work-groups: `part` 0 and 1, i = 0 .. 63).  At least 256 threads.
__device__ __forceinline__ void read_qkv_ahead(const char *W, int row_bytes, int part, int i) {
    constexpr int ROWS = 20, N = (ROWS * 96 + 255) / 256;
    const int xcd = i & 7, pieces = row_bytes / 16;   // 96, or 48 of int8 codes
    i32x4 v[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const int p = min((int)(threadIdx.x + 256 * j), ROWS * pieces - 1);
        const int r = (8 * part + (i >> 3)) * ROWS + p / pieces, q = r - 3 * SP_D;
        const int own = xcd * SP_D + (r / SP_D) * SP_E + r % SP_D;
        const int other = (8 + (xcd >> 1)) * SP_D +
                          (q < SP_D ? q : (q < SP_D + 32 ? SP_E : 2 * SP_E) + 32 * (xcd & 1) + ((q - SP_D) & 31));
        v[j] = *reinterpret_cast<const i32x4 *>(W + (size_t)(q < 0 ? own : other) * row_bytes + p % pieces * 16);
    }
#pragma unroll
    for (int j = 0; j < N; ++j) asm volatile("" ::"v"(v[j]));
}

// LN1, the head's q and this split's slices of k_new and v_new (96 rows, twelve a wave), their
// append to the cache, and attention over the split's share of the earlier keys.  The new key joins in
// k_step_proj as one more partial (m = q.k_new / 8, l = 1, c = v_new), so no work-group needs all of
// k_new or v_new.  48 work-groups, the splits of a head on as few XCDs as 12 heads on 8 allow (b % 8 is
// the XCD), so the q rows that they share come through one L2.
// MI355X, one layer at position 512, fp16, under the tracer: 6.0 us, where the q/k/v GEMV with its LayerNorm
// prologue (5.8) and a work-group per head (11.2) took 17.0.  Bound by the 147 KB of weight rows that each
// of the 48 CUs takes in (2.2 us).
template <bool QW>
__global__ __launch_bounds__(64 * (SP_WAVES + 1)) void k_step_attn(uint16_t *x, const uint16_t *__restrict__ wte,
                                                             const uint16_t *__restrict__ wpe,
                                                             const uint16_t *__restrict__ ln_g,
                                                             const uint16_t *__restrict__ ln_b,
                                                             const void *__restrict__ W, const float *__restrict__ Ws,
                                                             const uint16_t *__restrict__ bias, uint16_t *Kc, uint16_t *Vc,
                                                             int maxT, StepArg st, StepPart part, StepAhead ahead) {
    __shared__ __attribute__((aligned(16))) f16 xn[SP_E];
    __shared__ __attribute__((aligned(16))) f16 qkv[SP_R];
    __shared__ __attribute__((aligned(16))) float cw[SP_WAVES][SP_D];
    __shared__ float sm[SP_WAVES], sl[SP_WAVES];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (blockIdx.x >= SP_H * SP_S) {   // what work-group i of the three launches that follow will read
        const int i = blockIdx.x - SP_H * SP_S;
        read_ahead<1>(ahead.proj + (size_t)i * ahead.proj_bytes, ahead.proj_bytes);
        read_ahead<3>(ahead.fc + (size_t)i * ahead.fc_bytes, ahead.fc_bytes);
        read_ahead<3>(ahead.mlp + (size_t)i * ahead.mlp_bytes, ahead.mlp_bytes);
        return;
    }
    const int xcd = blockIdx.x & 7, slot8 = blockIdx.x >> 3;
    const int h = slot8 < SP_S ? xcd : 8 + (xcd >> 1);
    const int sp = slot8 < SP_S ? slot8 : 2 * (xcd & 1) + slot8 - SP_S;
    // the arguments in one batch of scalar loads: left to itself the compiler fetches each group where
    // it is first used, a chain of eight scalar round trips ahead of the last vector load
    asm volatile("" ::"s"(x), "s"(wte), "s"(wpe), "s"(ln_g), "s"(ln_b), "s"(W), "s"(Ws), "s"(bias), "s"(Kc), "s"(Vc), "s"(maxT));
    const int pos = __builtin_amdgcn_readfirstlane(st.p());
    if ((unsigned)pos >= (unsigned)maxT) return;   // uniform over the grid
    const size_t hoff = (size_t)h * maxT * SP_D;

    const int rw = wave - 1;   // row and key wave
    Rows4<QW> wr[SP_U];
    float sc[SP_U];
    uint16_t bs[SP_U];
    auto row_of = [&](int u) { return (rw * SP_U + u) * 4 + (lane >> 4); };
    // Keys of this wave: eight lanes read one 128-byte row of K and of V, so an instruction covers
    // eight whole rows; rows past the wave's last key read that key and count for nothing.
    const int per = (pos + SP_S - 1) / SP_S;
    const int j0 = min(pos, sp * per), j1 = min(pos, j0 + per);
    const int pw = (j1 - j0 + SP_WAVES - 1) / SP_WAVES;
    const int w0 = min(j1, j0 + pw * max(rw, 0)), w1 = min(j1, w0 + pw);
    const int slot = lane >> 3, dg = (lane & 7) * 8;
    constexpr int NT = SP_KEYS / 8;
    const int nt = (w1 - w0 + 7) >> 3;   // wave-uniform
    f16x8 kr[NT], vr[NT];
    if (wave == 0) {
        // Layer 0 takes the token's embedding for x (an id out of range embeds as wpe alone) and leaves
        // it there: split 0 of head h stores its 64 elements.
        LnRow ln;
        if (wte) {
            const int id = __builtin_amdgcn_readfirstlane(st.tok());
            const bool in_vocab = (unsigned)id < (unsigned)GPT2_VOCAB;
            ln.load(wte + (size_t)(in_vocab ? id : 0) * SP_E, ln_g, ln_b, lane);
            const uint16_t *prow = wpe + (size_t)min(pos, GPT2_N_CTX - 1) * SP_E;
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const f16x4 pe = *reinterpret_cast<const f16x4 *>(prow + 256 * i + 4 * lane);
#pragma unroll
                for (int c = 0; c < 4; ++c) ln.x[i][c] = (f16)((in_vocab ? (float)ln.x[i][c] : 0.f) + (float)pe[c]);
                if (sp == 0 && h >> 2 == i && lane >> 4 == (h & 3)) *reinterpret_cast<f16x4 *>(x + 256 * i + 4 * lane) = ln.x[i];
            }
        } else {
            ln.load(x, ln_g, ln_b, lane);
        }
        ln.normalize(xn, lane);
    } else {
#pragma unroll
        for (int u = 0; u < SP_U; ++u) wr[u].load(W, step_qkv_row(h, sp, row_of(u)), lane);
#pragma unroll
        for (int u = 0; u < SP_U; ++u) {
            const int row = step_qkv_row(h, sp, row_of(u));
            sc[u] = 1.f;
            if constexpr (QW) sc[u] = Ws[row];
            bs[u] = bias[row];
        }
    }
    lds_barrier();

    // ---- q, k, v rows, twelve a wave; the k and v slices also go to the cache, v_new to the merge
    if (wave > 0) {
        // the keys and values, behind the weights (ahead of the barrier they would hold it up: the
        // address unit takes 40 bytes a cycle)
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const size_t key = (size_t)max(0, min(w0 + slot + 8 * t, w1 - 1));
            if (t < nt) {
                kr[t] = *reinterpret_cast<const f16x8 *>(Kc + hoff + key * SP_D + dg);
                vr[t] = *reinterpret_cast<const f16x8 *>(Vc + hoff + key * SP_D + dg);
            }
        }
        f16x8 xr[6];
        load_x<QW>(xr, xn, lane);
        float dot[SP_U];
#pragma unroll
        for (int u = 0; u < SP_U; ++u) dot[u] = wr[u].dot(xr);
        if ((lane & 15) == 0) {
#pragma unroll
            for (int u = 0; u < SP_U; ++u) {
                const int r = row_of(u), i = r & (SP_KS - 1);
                const uint16_t o = f2h(dot[u] * sc[u] + h2f(bs[u]));
                qkv[r] = __builtin_bit_cast(f16, o);
                if (r >= SP_D) ((r < SP_D + SP_KS ? Kc : Vc) + hoff + (size_t)pos * SP_D + SP_KS * sp)[i] = o;
                if (r >= SP_D + SP_KS) part.v[h * SP_D + SP_KS * sp + i] = o;
            }
        }
    }
    lds_barrier();

    // ---- attention of q over the wave's keys: a key's score is the sum of its eight lanes
    float m_w = -INFINITY, l_w = 0.f, c[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (wave > 0 && w0 < w1) {
        const f16x8 q = *reinterpret_cast<const f16x8 *>(qkv + dg);
        float s[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            s[t] = -INFINITY;
            if (t < nt) s[t] = key_score(q, kr[t], w0 + slot + 8 * t < w1);
        }
        key_softmax<NT>(s, m_w, l_w);
#pragma unroll
        for (int t = 0; t < NT; ++t)
            if (t < nt) add_value(c, s[t], vr[t], w0 + slot + 8 * t < w1);
    }
    if (wave > 0) {
        reduce_values(c);
        if (lane < 8) {
            *reinterpret_cast<float4 *>(&cw[rw][8 * lane]) = float4{c[0], c[1], c[2], c[3]};
            *reinterpret_cast<float4 *>(&cw[rw][8 * lane + 4]) = float4{c[4], c[5], c[6], c[7]};
        }
        if (lane == 0) {
            sm[rw] = m_w;
            sl[rw] = l_w;
        }
    } else {   // this split's part of q.k_new
        const float pq = lane < SP_KS ? (float)qkv[SP_KS * sp + lane] * (float)qkv[SP_D + lane] : 0.f;
        const float d = row16_sum(pq);
        if (lane == 0) part.mls[h * 3 * SP_S + 2 * SP_S + sp] = d;
    }
    lds_barrier();
    const int rec = h * SP_S + sp;
    if (wave == 0) {   // lane = dimension
        float mw[SP_WAVES], lw[SP_WAVES], mx = -INFINITY;
#pragma unroll
        for (int w = 0; w < SP_WAVES; ++w) {
            mw[w] = sm[w];
            lw[w] = sl[w];
            mx = lw[w] != 0.f ? fmaxf(mx, mw[w]) : mx;
        }
        float L = 0.f, cc = 0.f;
#pragma unroll
        for (int w = 0; w < SP_WAVES; ++w) {
            const float f = lw[w] != 0.f ? __expf(mw[w] - mx) : 0.f;
            L += lw[w] * f;
            cc += cw[w][lane] * f;
        }
        part.record(rec)[lane] = cc;
        if (lane == 0) {
            part.mls[h * 3 * SP_S + sp] = mx;
            part.mls[h * 3 * SP_S + SP_S + sp] = L;
        }
    }
}

// The merge of the four splits and the new key, then attn-proj rows: a wave per row, four rows a
// work-group (192 work-groups), x[row] += row . att + bias.  The merge is repeated by every work-group:
// 16 KB of partials from L2 in one round trip, against a launch for doing it once.
template <bool QW>
__global__ __launch_bounds__(256) void k_step_proj(uint16_t *x, const void *__restrict__ W, const float *__restrict__ Ws,
                                                   const uint16_t *__restrict__ bias, StepPart part,
                                                   const uint16_t *kv_next, int maxT, StepArg st) {
    __shared__ __attribute__((aligned(16))) f16 att[SP_E];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (blockIdx.x >= SP_E / 4) {   // the next layer's keys and values, each head's on the XCDs that attend it
        const int i = blockIdx.x - SP_E / 4, xcd = i & 7, part8 = i >> 3;   // parts 0-3: K and V halves; 4-7: shared head
        const int pos = __builtin_amdgcn_readfirstlane(st.p()), keys = min(max(pos, 1), maxT), half = (keys + 1) / 2;
        const int h = part8 < 4 ? xcd : 8 + (xcd >> 1);
        const int v = (part8 >> 1) & 1, hf = part8 < 4 ? part8 & 1 : xcd & 1;
        const int from = min(hf * half, keys - 1), count = min(half, keys - from);
        if (part8 >= 4 && (part8 & 1)) return;
        const uint16_t *plane = kv_next + ((size_t)v * SP_H + h) * maxT * SP_D + (size_t)from * SP_D;
        read_ahead<GPT2_N_CTX / 2 * 128 / 16 / 256>(reinterpret_cast<const char *>(plane), count * 2 * SP_D);
        return;
    }
    const int row = blockIdx.x * 4 + wave;
    constexpr int TM = SP_E / 4;           // threads that merge, four elements each
    const int e = 4 * min(tid, TM - 1), h = e / SP_D;
    f32x4 c[SP_S];
#pragma unroll
    for (int s = 0; s < SP_S; ++s) c[s] = *reinterpret_cast<const f32x4 *>(part.record(h * SP_S + s) + e % SP_D);
    const f32x4 m = *reinterpret_cast<const f32x4 *>(part.mls + h * 3 * SP_S);
    const f32x4 l = *reinterpret_cast<const f32x4 *>(part.mls + h * 3 * SP_S + SP_S);
    const f32x4 d = *reinterpret_cast<const f32x4 *>(part.mls + h * 3 * SP_S + 2 * SP_S);
    const f16x4 vn = *reinterpret_cast<const f16x4 *>(part.v + e);
    uint2 wr[3];   // elements 256 i + 4 lane .. + 3 of the row
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const char *src = reinterpret_cast<const char *>(W) + ((size_t)row * SP_E + 256 * i + 4 * lane) * (QW ? 1 : 2);
        if constexpr (QW) wr[i] = uint2{*reinterpret_cast<const uint32_t *>(src), 0u};
        else wr[i] = *reinterpret_cast<const uint2 *>(src);
    }
    float sc = 1.f;
    if constexpr (QW) sc = Ws[row];
    const uint16_t bs = bias[row], rs = x[row];
    asm volatile("" ::: "memory");   // the row's loads stay ahead of the merge
    if (tid < TM) {
        const float spos = ((d[0] + d[1]) + (d[2] + d[3])) * 0.125f;
        float mx = spos;
#pragma unroll
        for (int s = 0; s < SP_S; ++s) mx = l[s] != 0.f ? fmaxf(mx, m[s]) : mx;
        const float fpos = __expf(spos - mx);
        float L = fpos;
        f32x4 o = {fpos * (float)vn[0], fpos * (float)vn[1], fpos * (float)vn[2], fpos * (float)vn[3]};
#pragma unroll
        for (int s = 0; s < SP_S; ++s) {
            const float f = l[s] != 0.f ? __expf(m[s] - mx) : 0.f;
            L += f * l[s];
            o += f * c[s];
        }
        const float inv = 1.0f / L;
        *reinterpret_cast<f16x4 *>(att + e) = f16x4{(f16)(o[0] * inv), (f16)(o[1] * inv), (f16)(o[2] * inv), (f16)(o[3] * inv)};
    }
    lds_barrier();
    float acc = 0.f;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const f16x4 a = *reinterpret_cast<const f16x4 *>(att + 256 * i + 4 * lane);
        f16x2 w0, w1;
        if constexpr (QW) {
            i8x4_to_f16x4_v(wr[i].x, w0, w1);
        } else {
            w0 = __builtin_bit_cast(f16x2, wr[i].x);
            w1 = __builtin_bit_cast(f16x2, wr[i].y);
        }
        acc = __builtin_amdgcn_fdot2(w0, f16x2{a[0], a[1]}, acc, false);
        acc = __builtin_amdgcn_fdot2(w1, f16x2{a[2], a[3]}, acc, false);
    }
    acc = wave_sum(acc);
    if (lane == 0) x[row] = f2h(acc * sc + h2f(bs) + h2f(rs));
}

// LN2, then 16 fc rows a work-group (192 work-groups), four a wave; gelu(row . xn + bias).  Bound by the
// chain x -> LayerNorm -> dot (1.2 us of the launch).  With the LayerNorm in a GEMV prologue, each lane
// normalized the 48 elements that it multiplied by, behind 24 loads of parameters: 6.2 us under the
// tracer against 3.0 here (fp16; 3.5 with the next layer's q/k/v rows read ahead, which saves 0.5 a layer).
template <bool QW>
__global__ __launch_bounds__(320) void k_step_fc(uint16_t *__restrict__ out, const uint16_t *__restrict__ x,
                                                 const uint16_t *__restrict__ ln_g, const uint16_t *__restrict__ ln_b,
                                                 const void *__restrict__ W, const float *__restrict__ Ws,
                                                 const uint16_t *__restrict__ bias, const char *qkv_next,
                                                 int qkv_row_bytes) {
    __shared__ __attribute__((aligned(16))) f16 xn[SP_E];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (blockIdx.x >= GPT2_FFN_DIM / 16) {
        read_qkv_ahead(qkv_next, qkv_row_bytes, 0, blockIdx.x - GPT2_FFN_DIM / 16);
        return;
    }
    const int row = blockIdx.x * 16 + 4 * max(wave - 1, 0) + (lane >> 4);
    Rows4<QW> wr;
    float sc = 1.f;
    uint16_t bs = 0;
    if (wave == 0) {
        LnRow ln;
        ln.load(x, ln_g, ln_b, lane);
        ln.normalize(xn, lane);
    } else {
        wr.load(W, row, lane);
        if constexpr (QW) sc = Ws[row];
        bs = bias[row];
    }
    lds_barrier();
    if (wave == 0) return;
    f16x8 xr[6];
    load_x<QW>(xr, xn, lane);
    const float v = wr.dot(xr);
    if ((lane & 15) == 0) out[row] = f2h(gelu_tanh(v * sc + h2f(bs)));
}

// mlp-proj rows, a wave per row and four rows a work-group (192 work-groups), x[row] += row . h + bias.  One
// memory round trip: 2.6 us under the tracer (3.0 with its rows not read ahead).
template <bool QW>
__global__ __launch_bounds__(256) void k_step_mlp(uint16_t *x, const uint16_t *__restrict__ hid, const void *__restrict__ W,
                                                  const float *__restrict__ Ws, const uint16_t *__restrict__ bias,
                                                  const char *qkv_next, int qkv_row_bytes) {
    constexpr int CPL = QW ? 3 : 6, K = GPT2_FFN_DIM;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (blockIdx.x >= SP_E / 4) {
        read_qkv_ahead(qkv_next, qkv_row_bytes, 1, blockIdx.x - SP_E / 4);
        return;
    }
    const int row = blockIdx.x * 4 + wave;
    f16x8 xr[6];
#pragma unroll
    for (int v = 0; v < 6; ++v)
        xr[v] = *reinterpret_cast<const f16x8 *>(hid + (QW ? (lane + 64 * (v >> 1)) * 16 + (v & 1) * 8 : (lane + 64 * v) * 8));
    i32x4 w[CPL];
#pragma unroll
    for (int i = 0; i < CPL; ++i)
        w[i] = *reinterpret_cast<const i32x4 *>(reinterpret_cast<const char *>(W) + (size_t)row * K * (QW ? 1 : 2) + (lane + 64 * i) * 16);
    float sc = 1.f;
    if constexpr (QW) sc = Ws[row];
    const uint16_t bs = bias[row], rs = x[row];
    asm volatile("" ::: "memory");
    float acc = 0.f;
#pragma unroll
    for (int i = 0; i < CPL; ++i) {
        if constexpr (QW) acc = dot16q(w[i], xr[2 * i], xr[2 * i + 1], acc);
        else acc = dot8(w[i], xr[i], acc);
    }
    acc = wave_sum(acc);
    if (lane == 0) x[row] = f2h(acc * sc + h2f(bs) + h2f(rs));
}

// LN_f, then the head: 16 rows a wave in four passes of four rows, three passes in flight behind the
// LayerNorm's loads.  786 work-groups, all resident at once (at most 128 registers a lane), so the
// LayerNorm is paid once per 64 rows and beside the weight stream: 16.1 us for 77 MB under the tracer
// (4.8 TB/s) against 20.8 with the LayerNorm in every 16-row work-group's prologue.  Row sums are added in
// the order of gpt2_gemv_*'s default forms.
constexpr int SH_PASS = 4, SH_AHEAD = 3, SH_ROWS = 4 * SH_PASS;
template <bool QW>
__global__ __launch_bounds__(256, 4) void k_step_head(uint16_t *__restrict__ out, const uint16_t *__restrict__ x,
                                                      const uint16_t *__restrict__ ln_g, const uint16_t *__restrict__ ln_b,
                                                      const void *__restrict__ W, const float *__restrict__ Ws, int N) {
    __shared__ __attribute__((aligned(16))) f16 xn[SP_E];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r0 = (blockIdx.x * 4 + wave) * SH_ROWS + (lane >> 4);
    Rows4<QW> wr[SH_AHEAD];
    float sc[SH_PASS];
    if (wave == 0) {
        LnRow ln;
        ln.load(x, ln_g, ln_b, lane);
        ln.normalize(xn, lane);
    }
#pragma unroll
    for (int u = 0; u < SH_AHEAD; ++u) wr[u].load(W, min(r0 + 4 * u, N - 1), lane);
#pragma unroll
    for (int u = 0; u < SH_PASS; ++u) {
        sc[u] = 1.f;
        if constexpr (QW) sc[u] = Ws[min(r0 + 4 * u, N - 1)];
    }
    lds_barrier();
    f16x8 xr[6];
    load_x<QW>(xr, xn, lane);
#pragma unroll
    for (int u = 0; u < SH_PASS; ++u) {
        const float v = wr[u % SH_AHEAD].dot(xr);
        if (u + SH_AHEAD < SH_PASS) wr[u % SH_AHEAD].load(W, min(r0 + 4 * (u + SH_AHEAD), N - 1), lane);
        const int r = r0 + 4 * u;
        if ((lane & 15) == 0 && r < N) out[r] = f2h(QW ? v * sc[u] : v);
    }
}

// ------------------------------------------------------------------ host launchers
// Bytes of a weight row of k elements.
static int row_bytes(const StepMat &m, int k) { return m.s ? k : 2 * k; }

void step_attn(uint16_t *x, const uint16_t *wte, const uint16_t *wpe, const uint16_t *ln_g, const uint16_t *ln_b,
               const StepMat &w, uint16_t *Kc, uint16_t *Vc, int maxT, StepArg st, const StepPart &part,
               const StepMat &proj, const StepMat &fc, const StepMat &mlp) {
    static_assert(SP_H * SP_S == 48, "the XCD assignment covers 12 heads of four splits on 8 XCDs");
    static_assert(SP_E / 4 == GPT2_FFN_DIM / 16, "a reading-ahead work-group per work-group of the next launches");
    const StepAhead a = {(const char *)proj.w, (const char *)fc.w, (const char *)mlp.w, 4 * row_bytes(proj, SP_E),
                         16 * row_bytes(fc, SP_E), 4 * row_bytes(mlp, GPT2_FFN_DIM)};
    hipLaunchKernelGGL(w.s ? k_step_attn<true> : k_step_attn<false>, dim3(SP_H * SP_S + SP_E / 4), dim3(64 * (SP_WAVES + 1)), 0,
                       stream(), x, wte, wpe, ln_g, ln_b, w.w, w.s, w.b, Kc, Vc, maxT, st, part, a);
    check_launch("k_step_attn");
}

void step_proj(uint16_t *x, const StepMat &w, const StepPart &part, const uint16_t *kv_next, int maxT, StepArg st) {
    hipLaunchKernelGGL(w.s ? k_step_proj<true> : k_step_proj<false>, dim3(SP_E / 4 + (kv_next ? 64 : 0)), dim3(256), 0,
                       stream(), x, w.w, w.s, w.b, part, kv_next, maxT, st);
    check_launch("k_step_proj");
}

void step_fc(uint16_t *out, const uint16_t *x, const uint16_t *ln_g, const uint16_t *ln_b, const StepMat &w,
             const StepMat *qkv_next) {
    hipLaunchKernelGGL(w.s ? k_step_fc<true> : k_step_fc<false>, dim3(GPT2_FFN_DIM / 16 + (qkv_next ? 64 : 0)), dim3(320), 0,
                       stream(), out, x, ln_g, ln_b, w.w, w.s, w.b, qkv_next ? (const char *)qkv_next->w : nullptr,
                       qkv_next ? row_bytes(*qkv_next, SP_E) : 0);
    check_launch("k_step_fc");
}

void step_mlp(uint16_t *x, const uint16_t *hid, const StepMat &w, const StepMat *qkv_next) {
    hipLaunchKernelGGL(w.s ? k_step_mlp<true> : k_step_mlp<false>, dim3(SP_E / 4 + (qkv_next ? 64 : 0)), dim3(256), 0, stream(),
                       x, hid, w.w, w.s, w.b, qkv_next ? (const char *)qkv_next->w : nullptr,
                       qkv_next ? row_bytes(*qkv_next, SP_E) : 0);
    check_launch("k_step_mlp");
}

void step_head(uint16_t *out, const uint16_t *x, const uint16_t *ln_g, const uint16_t *ln_b, const StepMat &w, int N) {
    hipLaunchKernelGGL(w.s ? k_step_head<true> : k_step_head<false>, dim3(cdiv(cdiv(N, SH_ROWS), 4)), dim3(256), 0,
                       stream(), out, x, ln_g, ln_b, w.w, w.s, N);
    check_launch("k_step_head");
}

}  // namespace g2
