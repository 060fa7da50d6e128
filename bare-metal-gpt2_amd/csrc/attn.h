// attn.h -- single-query attention over the K/V cache, shared by the decode attention kernels (ops.hip,
// decode_step.hip).
//
// A wave holds up to 8 NT keys: key slot s = lane / 8 of step t is key 8 t + s, and lane l of the slot
// holds dims 8 (l & 7) .. + 7 of the key and of its value, so one load instruction reads eight whole
// 128-byte rows of the cache.  (A lane per key, reading its own row 16 bytes at a time, touches 64 rows
// per instruction and every row again by the next seven.)
#pragma once

#include <cmath>

#include "common.h"

namespace g2 {

// A value from the lane eight further on (mod 16) of the same 16-lane row: the row's other key slot.
__device__ __forceinline__ float other_slot(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xF, 0xF, true));   // row_ror:8
}

// q . k / 8 of the lane's key slot, the eight lanes' parts summed (every lane of the slot gets it); -inf
// where the slot holds no key (`on` false).
__device__ __forceinline__ float key_score(const f16x8 q, const f16x8 k, bool on) {
    float d = __builtin_amdgcn_fdot2(f16x2{q[0], q[1]}, f16x2{k[0], k[1]}, 0.f, false);
    d = __builtin_amdgcn_fdot2(f16x2{q[2], q[3]}, f16x2{k[2], k[3]}, d, false);
    d = __builtin_amdgcn_fdot2(f16x2{q[4], q[5]}, f16x2{k[4], k[5]}, d, false);
    d = __builtin_amdgcn_fdot2(f16x2{q[6], q[7]}, f16x2{k[6], k[7]}, d, false);
    // quad_perm xor 1, xor 2, then the other quad of the eight (row_half_mirror)
    d += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(d), 0xB1, 0xF, 0xF, true));
    d += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(d), 0x4E, 0xF, 0xF, true));
    d += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(d), 0x141, 0xF, 0xF, true));
    return on ? d * 0.125f : -INFINITY;
}

// The softmax weights of a wave's scores against their maximum m, in place, and their sum l (both the
// same in every lane).  If no score is above -inf (keys that score -inf, not only absent ones), m is -inf and
// the weights and l are 0, as if the wave had no keys: another wave's keys may decide.
template <int NT>
__device__ __forceinline__ void key_softmax(float (&s)[NT], float &m, float &l) {
    float mx = s[0];
#pragma unroll
    for (int t = 1; t < NT; ++t) mx = fmaxf(mx, s[t]);
    mx = fmaxf(mx, other_slot(mx));
    m = fmaxf(fmaxf(lane_f(mx, 0), lane_f(mx, 16)), fmaxf(lane_f(mx, 32), lane_f(mx, 48)));
    const float base = m == -INFINITY ? 0.f : m;
    float sum = 0.f;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        s[t] = __expf(s[t] - base);
        sum += s[t];
    }
    sum += other_slot(sum);
    l = cross_rows_sum(sum);
}

// c += p v on the lane's eight dims; a slot without a key adds nothing, whatever v holds.
__device__ __forceinline__ void add_value(float (&c)[8], float p, const f16x8 v, bool on) {
    const i32x4 b = __builtin_bit_cast(i32x4, v);
    const f16x8 u = __builtin_bit_cast(f16x8, i32x4{on ? b[0] : 0, on ? b[1] : 0, on ? b[2] : 0, on ? b[3] : 0});
#pragma unroll
    for (int e = 0; e < 8; ++e) c[e] = __builtin_fmaf(p, (float)u[e], c[e]);
}

// Sum over the wave's eight key slots: every lane ends with dims 8 (lane & 7) .. + 7.
__device__ __forceinline__ void reduce_values(float (&c)[8]) {
#pragma unroll
    for (int e = 0; e < 8; ++e) c[e] = group_sum(c[e] + other_slot(c[e]));
}

}  // namespace g2
