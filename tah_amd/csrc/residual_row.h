// A row of the residual stream on its way past a norm: the sum with a sublayer's normed result and the norm and short convolution in
// front of the next sublayer.  Shared by residual_norm_kernel (row_norm.hip), which writes what the next launch reads, by
// norm_linear_kernel (linear_rows.hip), whose workgroups each make the rows' operand for themselves, and by
// moe_norm_route_kernel (moe.hip), whose workgroup goes on to choose its row's experts.
#pragma once
#include "mixer_device.h"

namespace tah {
namespace {

constexpr int kRowThreads = 256;  // threads to a row
constexpr int kMaxGroups = 256;

// LDS of one row's threads
template <int U, bool GROUPS>
struct ResidualLds {
    float red[kRowThreads / kWave], unit_sums[GROUPS ? U * kRowThreads : 1], group_sum[GROUPS ? kMaxGroups : 1];
};

// Sum of a row's values over its group, one partial sum s[u] per thread and unit, for each of the thread's units.
// GROUPS: several groups of group_units units each, added up inside a wave where the groups divide it; else through LDS:
// `unit_sums` of as many floats as the row has units, `group_sum` of as many as it has groups.  `red`: a float per wave.
// tid: among the row's threads.  A workgroup whose threads make several rows calls it with all of them.
template <int U, bool GROUPS>
__device__ __forceinline__ void group_sums(float (&s)[U], int tid, int units, int groups, int group_units, ResidualLds<U, GROUPS>& lds) {
    if constexpr (!GROUPS) {
        float t = 0.f;
#pragma unroll
        for (int u = 0; u < U; ++u) t += s[u];
        t = wave_sum(t);
        if (tid % kWave == 0) lds.red[tid / kWave] = t;
        __syncthreads();
        t = 0.f;
#pragma unroll
        for (int w = 0; w < kRowThreads / kWave; ++w) t += lds.red[w];
        __syncthreads();
#pragma unroll
        for (int u = 0; u < U; ++u) s[u] = t;
    } else if (group_units <= kWave && (group_units & (group_units - 1)) == 0) {
        for (int d = group_units / 2; d >= 1; d >>= 1) {
#pragma unroll
            for (int u = 0; u < U; ++u) s[u] += __shfl_xor(s[u], d);
        }
    } else {
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (tid + u * kRowThreads < units) lds.unit_sums[tid + u * kRowThreads] = s[u];
        __syncthreads();
        for (int g = tid / kWave; g < groups; g += kRowThreads / kWave) {
            float t = 0.f;
            for (int i = tid % kWave; i < group_units; i += kWave) t += lds.unit_sums[g * group_units + i];
            t = wave_sum(t);
            if (tid % kWave == 0) lds.group_sum[g] = t;
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int g = (tid + u * kRowThreads) / group_units;
            s[u] = lds.group_sum[g < groups ? g : groups - 1];  // (columns behind the last group hold zeros)
        }
    }
}

// Sum of the squares of a unit's columns.  The roundings are written out: left to the compiler, one kernel fused the first square
// into the sum and another the second, the last bit of a norm hung on that, and two kernels that must agree did not have to.
__device__ __forceinline__ float sum_of_squares(const float (&v)[8]) {
    float s = fmaf(v[0], v[0], v[1] * v[1]);
#pragma unroll
    for (int i = 2; i < 8; ++i) s = fmaf(v[i], v[i], s);
    return s;
}

// What tah_residual_norm does with one row, by kRowThreads threads.  U: units of eight columns per thread.  kEarly: a few rows are a
// chain of trips to memory and little else, so a thread asks for everything at once: row, norms, convolution, the expert rows as soon
// as their indices are there and the convolution's inputs as soon as the position is.  (Threads whose columns lie behind the
// row's end read the row's start and use none of it.)
// write: the row's results go to memory, the residual row to x_out.  meanwhile(): called when the loads that wait for no other are on
// their way (a wave's loads return in order: what it asks for comes before the convolution's inputs and the experts' rows).
// emit(c, v): columns c ... c + 7 of the operand that comes out of it, the normed row or without next_coef the residual row.
template <class E, int U, bool GROUPS, bool kEarly, class Meanwhile, class Emit>
__device__ __forceinline__ void residual_row(const tah_residual_norm_args& p, int row, int tid, ResidualLds<U, GROUPS>& lds, bool write, float* x_out,
                                             Meanwhile meanwhile, Emit emit) {
    constexpr int kExpertsAhead = kEarly ? 8 : 1, kTaps = 4;
    const int units = p.cols / 8, group_units = GROUPS ? p.group_cols / 8 : units;
    const float count = GROUPS ? (float)(p.width / p.groups) : (float)p.width;
    float y[U][8], x[U][8];
    const bool add = p.y || p.experts, few_taps = kEarly && p.conv && p.taps <= kTaps;
    Eight<float> x_in[U], coef[kEarly ? U : 1], next_coef[kEarly ? U : 1], conv_w[kEarly ? U : 1][kTaps];
    Eight<E> y_in[U], conv_in[kEarly ? U : 1][kTaps];
    int at[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int c = 8 * (tid + u * kRowThreads);
        at[u] = c < p.cols ? c : 0;
        x_in[u].load(p.x + (int64_t)row * p.cols + at[u]);
        if (p.y) y_in[u].load(static_cast<const E*>(p.y) + (int64_t)row * p.y_row_stride + at[u]);
    }
    const float ys = p.y_scale ? p.y_scale[row] : 1.0f;
    const int slot = p.conv ? p.slot[row] : -1, pos = p.conv ? p.pos[row] : -1;
    if constexpr (kEarly) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (add) coef[u].load(p.coef + at[u]);
            if (p.next_coef) next_coef[u].load(p.next_coef + at[u]);
            if (few_taps) {
#pragma unroll
                for (int d = 0; d < kTaps; ++d) conv_w[u][d].load(p.conv + (int64_t)(d < p.taps ? p.taps - 1 - d : 0) * p.cols + at[u]);
            }
        }
    }
    meanwhile();
    const bool live = slot >= 0 && slot < p.nslots && pos >= 0;
    E* const rings = p.conv ? static_cast<E*>(p.conv_state) + (int64_t)(live ? slot : 0) * p.taps * p.cols : nullptr;
    if constexpr (kEarly) {
        if (few_taps) {
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int d = 1; d < kTaps; ++d)
                    conv_in[u][d].load(rings + (int64_t)(live && d < p.taps && d <= pos ? (pos - d) % p.taps : 0) * p.cols + at[u]);
        }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
        for (int i = 0; i < 8; ++i) y[u][i] = 0.f;
    if (p.y) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < 8; ++i) y[u][i] = y_in[u][i] * ys;
    }
    if (p.experts) {
        for (int j0 = 0; j0 < p.top; j0 += kExpertsAhead) {
            float w[kExpertsAhead];
            int64_t from[kExpertsAhead];
            Eight<E> v[kExpertsAhead][U];
#pragma unroll
            for (int k = 0; k < kExpertsAhead; ++k) {
                const int64_t j = (int64_t)row * p.top + (j0 + k < p.top ? j0 + k : j0);
                w[k] = p.weight[j];
                from[k] = ((int64_t)p.index[j] * p.index_scale + (int64_t)row * p.index_row) * p.experts_row_stride;
            }
#pragma unroll
            for (int k = 0; k < kExpertsAhead; ++k)
#pragma unroll
                for (int u = 0; u < U; ++u) v[k][u].load(static_cast<const E*>(p.experts) + from[k] + at[u]);
#pragma unroll
            for (int k = 0; k < kExpertsAhead; ++k)
                if (j0 + k < p.top) {
#pragma unroll
                    for (int u = 0; u < U; ++u)
#pragma unroll
                        for (int i = 0; i < 8; ++i) y[u][i] += w[k] * v[k][u][i];
                }
        }
    }
    float s[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const bool in = 8 * (tid + u * kRowThreads) < p.cols;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            x[u][i] = in ? x_in[u][i] : 0.f;
            y[u][i] = in ? y[u][i] : 0.f;
        }
    }
    if (add) {
#pragma unroll
        for (int u = 0; u < U; ++u) s[u] = sum_of_squares(y[u]);
        group_sums<U, GROUPS>(s, tid, units, p.groups, group_units, lds);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int c = 8 * (tid + u * kRowThreads);
        float sx = 0.f;
        if (c < p.cols) {
            if (add) {
                const float r = 1.0f / sqrtf(s[u] / count + p.eps);
                if constexpr (!kEarly) coef[0].load(p.coef + c);
#pragma unroll
                for (int i = 0; i < 8; ++i) x[u][i] += y[u][i] * r * coef[kEarly ? u : 0][i];
                if (write) store8(x_out + (int64_t)row * p.cols + c, x[u]);
            } else if (write && x_out != p.x) {
                store8(x_out + (int64_t)row * p.cols + c, x[u]);
            }
            sx = sum_of_squares(x[u]);
            if (write && p.xe) store8(static_cast<E*>(p.xe) + (int64_t)row * p.cols + c, x[u]);
            if (write && p.x_packed) static_cast<bf16x8*>(p.x_packed)[rows_form_unit(row, c)] = to_bf16x8(x[u]);
            if (!p.next_coef) emit(c, x[u]);
        }
        s[u] = sx;
    }
    if (!p.next_coef) return;
    group_sums<U, GROUPS>(s, tid, units, p.groups, group_units, lds);
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int c = 8 * (tid + u * kRowThreads);
        if (c < p.cols) {
            const float rx = 1.0f / sqrtf(s[u] / count + p.eps);
            float k[8];
            if constexpr (!kEarly) next_coef[0].load(p.next_coef + c);
#pragma unroll
            for (int i = 0; i < 8; ++i) k[i] = next_coef[kEarly ? u : 0][i] * (x[u][i] * rx);
            if (p.conv) {
                E* const ring = rings + c;
#pragma unroll
                for (int i = 0; i < 8; ++i) k[i] = (float)(E)k[i];
                if (live && write) store8(ring + (int64_t)(pos % p.taps) * p.cols, k);  // (in the place of a token no row reads any more)
                if (kEarly && few_taps) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) k[i] += conv_w[kEarly ? u : 0][0][i] * k[i];
#pragma unroll
                    for (int d = 1; d < kTaps; ++d)
                        if (live && d < p.taps && d <= pos) {
#pragma unroll
                            for (int i = 0; i < 8; ++i) k[i] += conv_w[kEarly ? u : 0][d][i] * conv_in[kEarly ? u : 0][d][i];
                        }
                } else {
                    float h[8], w[8];
                    load8(p.conv + (int64_t)(p.taps - 1) * p.cols + c, w);
#pragma unroll
                    for (int i = 0; i < 8; ++i) k[i] += w[i] * k[i];
                    for (int d = 1; live && d < p.taps && d <= pos; ++d) {
                        load8(ring + (int64_t)((pos - d) % p.taps) * p.cols, h);
                        load8(p.conv + (int64_t)(p.taps - 1 - d) * p.cols + c, w);
#pragma unroll
                        for (int i = 0; i < 8; ++i) k[i] += w[i] * h[i];
                    }
                }
            }
            if (write && p.normed) store8(static_cast<E*>(p.normed) + (int64_t)row * p.cols + c, k);
            if (write && p.normed_packed) static_cast<bf16x8*>(p.normed_packed)[rows_form_unit(row, c)] = to_bf16x8(k);
            emit(c, k);
        }
    }
}

// What tah_residual_norm's arguments have to be, sizes of a row apart.
inline int check_residual(const tah_residual_norm_args& a) {
    if (a.rows < 0 || a.width <= 0 || a.cols < a.width || a.cols % 8 != 0 || (a.dtype != TAH_DT_BF16 && a.dtype != TAH_DT_F32) || a.top < 0)
        return TAH_E_SHAPE;
    if (a.groups <= 0 || a.groups > kMaxGroups || a.width % a.groups != 0 ||
        (a.groups > 1 && (a.group_cols % 8 != 0 || a.group_cols < a.width / a.groups || (int64_t)a.groups * a.group_cols > a.cols)))
        return TAH_E_SHAPE;
    if (a.conv && (a.taps <= 0 || a.nslots <= 0)) return TAH_E_SHAPE;
    if ((a.x_packed || a.normed_packed) && (a.rows > 32 || a.cols % 32 != 0)) return TAH_E_SHAPE;
    if (a.rows == 0) return TAH_OK;
    if (!a.x || ((a.y || a.experts) && !a.coef) || (a.experts && (!a.index || !a.weight))) return TAH_E_NULL;
    if ((a.normed || a.normed_packed || a.conv) && !a.next_coef) return TAH_E_NULL;
    if (a.conv && (!a.conv_state || !a.slot || !a.pos)) return TAH_E_NULL;
    const void* ptrs[] = {a.y, a.experts, a.coef, a.next_coef, a.x, a.xe, a.x_packed, a.normed, a.normed_packed, a.conv, a.conv_state};
    for (const void* q : ptrs)
        if (!aligned_16(q)) return TAH_E_ALIGN;
    if ((a.y && (a.y_row_stride % 8 != 0 || a.y_row_stride < a.cols)) ||
        (a.experts && (a.experts_row_stride % 8 != 0 || a.experts_row_stride < a.cols)))
        return TAH_E_ALIGN;
    return TAH_OK;
}

}  // namespace
}  // namespace tah
