// The decision of a two-layer decider on one row, by one wave: shared by the kernel that only decides and the one that
// goes on with the rows that are hard.
#pragma once
#include <hip/hip_runtime.h>

#include "duo_device.h"
#include "row_keys.h"
#include "tah_duo.h"

namespace tah {

struct DeciderTailParams {
    const __bf16 *h, *w2, *b2;
    int64_t h_rs;
    int32_t width;
    float threshold;
    const uint8_t* active;
    const int32_t* pos;
    uint8_t* hard;
    int32_t *hard_i, *slot, *q_pos;
};

inline DeciderTailParams decider_params(const tah_decider_tail_args& a) {
    DeciderTailParams p;
    p.h = static_cast<const __bf16*>(a.hidden); p.w2 = static_cast<const __bf16*>(a.w2); p.b2 = static_cast<const __bf16*>(a.b2);
    p.h_rs = a.hidden_row_stride; p.width = a.width; p.threshold = a.threshold;
    p.active = a.active; p.pos = a.pos; p.hard = a.hard; p.hard_i = a.hard_i32; p.slot = a.slot; p.q_pos = a.q_pos;
    return p;
}

inline int check_decider(const tah_decider_tail_args& a) {
    if (a.rows < 0 || a.rows > 65535 || a.width <= 0 || a.width % 8 != 0) return TAH_E_SHAPE;
    if (a.rows == 0) return TAH_OK;
    if (!a.hidden || !a.w2 || !a.hard || (a.q_pos && !a.pos)) return TAH_E_NULL;
    if ((reinterpret_cast<uintptr_t>(a.hidden) & 15) || (reinterpret_cast<uintptr_t>(a.w2) & 15) || a.hidden_row_stride % 8 != 0) return TAH_E_ALIGN;
    return TAH_OK;
}

// z = bf16(h . w2) (float32 sum), + b2 in bf16, sigmoid in float32, > threshold, and active; the same in every lane
__device__ __forceinline__ bool decide_row(const DeciderTailParams& p, int row, int lane) {
    float s = 0.f;
    for (int c = 8 * lane; c < p.width; c += 8 * kWave) {
        const u32x4 a = *reinterpret_cast<const u32x4*>(p.h + (int64_t)row * p.h_rs + c);
        const u32x4 b = *reinterpret_cast<const u32x4*>(p.w2 + c);
#pragma unroll
        for (int q = 0; q < 4; ++q)
            s += __uint_as_float(a[q] << 16) * __uint_as_float(b[q] << 16) + __uint_as_float(a[q] & 0xffff0000u) * __uint_as_float(b[q] & 0xffff0000u);
    }
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) s += __shfl_xor(s, m);
    float z = round_bf16(s);
    if (p.b2) z = round_bf16(z + (float)p.b2[0]);
    const float prob = 1.0f / (1.0f + fast_exp2(-z * kLog2e));
    return prob > p.threshold && (p.active == nullptr || p.active[row] != 0);
}

// what the second latent iteration is told about the row (one lane)
__device__ __forceinline__ void put_decision(const DeciderTailParams& p, int row, bool hard) {
    p.hard[row] = hard ? 1 : 0;
    if (p.hard_i) p.hard_i[row] = hard ? 1 : 0;
    if (p.slot) p.slot[row] = hard ? row : -1;
    if (p.q_pos) p.q_pos[row] = hard ? p.pos[row] : -1;
}

}  // namespace tah
