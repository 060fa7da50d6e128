// decode_step.h -- launchers of the multi-kernel decode step's kernels (decode_step.hip).
#pragma once

#include "common.h"

namespace g2 {

constexpr int STEP_SPLITS = 4;   // key splits per head (k_step_attn)

// Where k_step_attn leaves each split's partial for k_step_proj, in the caller's scratch buffers (sized
// for at least one token, dead between the two launches):
//   48 records of 64 floats (unnormalized context of head h, split s: record 4 h + s) in fc, qkv, att;
//   the heads' m, l and parts of q.k_new ([head][3][4] floats) in ao; v_new (768 halves) in ff.
struct StepPart {
    float *rec[3];
    float *mls;
    uint16_t *v;
    static constexpr int N0 = GPT2_FFN_DIM / 2 / GPT2_HEAD_DIM;        // records in fc
    static constexpr int N1 = GPT2_QKV_DIM / 2 / GPT2_HEAD_DIM;        // in qkv
    static constexpr int N2 = GPT2_N_EMBD / 2 / GPT2_HEAD_DIM;         // in att
    static_assert(N0 + N1 + N2 >= GPT2_N_HEAD * STEP_SPLITS, "the records fit the scratch of one token");
    static_assert(GPT2_N_HEAD * 3 * STEP_SPLITS * 2 <= GPT2_N_EMBD, "m, l and q.k_new fit ao");
    __device__ __forceinline__ float *record(int i) const {
        float *base = i < N0 ? rec[0] : i < N0 + N1 ? rec[1] : rec[2];
        return base + (size_t)(i < N0 ? i : i < N0 + N1 ? i - N0 : i - N0 - N1) * GPT2_HEAD_DIM;
    }
};

// A weight matrix: fp16 rows, or int8 codes with row scales s; b its bias (fp16; the head has none).
struct StepMat {
    const void *w;
    const float *s;
    const uint16_t *b;
};

// What k_step_attn's spare work-groups read ahead: weights, and the bytes of them that one work-group of
// the later launch reads.
struct StepAhead {
    const char *proj, *fc, *mlp;
    int proj_bytes, fc_bytes, mlp_bytes;
};

// wte != nullptr (layer 0): the row is the token's embedding, which the launch also stores in x.  All
// pointers 16-byte aligned (scales: 4, biases: 2).  proj, fc, mlp: the same layer's later matrices;
// kv_next and qkv_next (may be null): the next layer's K plane (V follows it) and q/k/v matrix.
void step_attn(uint16_t *x, const uint16_t *wte, const uint16_t *wpe, const uint16_t *ln_g, const uint16_t *ln_b,
               const StepMat &w, uint16_t *Kc, uint16_t *Vc, int maxT, StepArg st, const StepPart &part,
               const StepMat &proj, const StepMat &fc, const StepMat &mlp);
void step_proj(uint16_t *x, const StepMat &w, const StepPart &part, const uint16_t *kv_next, int maxT, StepArg st);
void step_fc(uint16_t *out, const uint16_t *x, const uint16_t *ln_g, const uint16_t *ln_b, const StepMat &w,
             const StepMat *qkv_next);
void step_mlp(uint16_t *x, const uint16_t *hid, const StepMat &w, const StepMat *qkv_next);
void step_head(uint16_t *out, const uint16_t *x, const uint16_t *ln_g, const uint16_t *ln_b, const StepMat &w, int N);

}  // namespace g2
