// Linear layers of a decode step, gfx950: y = x W^T for at most 32 rows (one token per sequence) against a weight
// of 8 to 50 MB.  The work is streaming W from HBM once; everything here serves having all of it in flight with
// as few cache-line requests as possible:
//
//  * W is re-ordered once, when the model is loaded, into the order the matrix instruction wants it: tiles of
//    16 output columns x 32 k, each stored as the 64 16-byte operands of the 64 lanes of one
//    v_mfma_f32_16x16x32_bf16 step (lane l: column l % 16, k = 8 (l / 16) ... + 8).  A wave's load instruction
//    then reads 1 KiB that lies together, and a column tile's k steps follow each other in memory.
//  * The rows are kept in the same form ([k / 32][2 row halves][64 lanes][8]): the kernels that produce them
//    (these linear layers, the attention merge, tah_linear_pack_rows) write it, so the rows' operand is one
//    1 KiB load per step and row half as well.  Reading either operand from a row-major matrix costs one cache
//    line request per row and lane group, and those, not the bytes, bound such a kernel.
//  * One workgroup = one group of output columns over all of K; its eight waves split K and meet in LDS.  A
//    wave issues the loads of a whole chunk of steps (up to 24 KiB) before the first multiply.
//  * Epilogues: + residual (in place is fine), or the MLP's act_fn(gate) * up with the input RMSNorm's per-row
//    factor (the norm's weight is expected inside W): the sum of squares of a row comes from the operands the
//    waves load anyway.  A LayerNorm of the rows folds in the same way (the learned decider's blocks,
//    tah/model/iter_decider.py:139-152): with W' = W diag(gamma), W' LN(x) = (W' x - mean(x) W' 1) / std(x) + W beta,
//    so the kernel needs the row's sum and sum of squares, the row sums of W' and a bias that carries W beta.
//    ReLU or GELU (the exact one, nn.GELU's default) last.  Results are written row-major and/or in the packed rows
//    form for the next layer.
//
// Measured at 32 rows inside a captured step (MI355X): q|k|v 16 MB 6.0 us, o 8 MB 5.1 us, gate|up + SiLU 50 MB
// 12.3 us, down 25 MB 9.6 us, against 14 / 8.4 / 16 + 5 / 15 us for the library GEMMs and the SiLU kernel.  What
// is left besides the weight stream (7.5 TB/s once started) is about 4 us of launch, first-byte latency and
// reduction per kernel, and the rows' operand: every workgroup reads all 32 x K of it from L2, which the
// per-CU L1 fill rate (about 100 GB/s) makes 1 us per 128 KB.  Splitting K over workgroups would cut that, but
// the hand-over between workgroups (device-scope fence + counter, last one reduces) cost 7 us per split when
// tried: the fence writes back and invalidates the whole L2 of the XCD.  One to eight rows: 5.2 / 4.6 / 11.5 / 7.6 us
// (kFold, H8 below), 5.7 / 5.1 / 11.7 / 9.6 without those.
#include <hip/hip_runtime.h>

#include <utility>

#include "residual_row.h"

namespace tah {
namespace {

constexpr int kLinWaves = 8;
constexpr int kLinThreads = kLinWaves * kWave;
constexpr int kLinRows = 32;    // rows per call: two 16-row halves of the MFMA's row operand
constexpr int kTileCols = 16;   // output columns of one weight tile
constexpr int kStepK = 32;      // k of one MFMA step; a tile step is 16 x 32 bf16 = 1 KiB
constexpr int kGroup24 = 24;    // gate|up: output columns per workgroup when n % 24 == 0 (256 workgroups for n = 6144)

// kPlainNorm: plain with the rows' RMSNorm factor; kPlainLayerNorm: with the rows' mean and deviation
enum Epi { kPlain = 0, kPlainNorm = 1, kGateUp16 = 2, kGateUp24 = 3, kPlainLayerNorm = 4 };

struct LinParams {
    const bf16x8* w;   // packed weight
    const bf16x8* x;   // packed rows
    const __bf16* res; // row-major residual or null
    const __bf16* bias; // [n] added to the product (rounded to bf16 first, as a GEMM's output is) or null
    const float* colsum; // kPlainLayerNorm: [n] sums of the packed weight's rows over k
    int32_t act;       // TAH_ACT_*
    __bf16* y;         // row-major result or null
    bf16x8* yp;        // packed result or null
    int64_t res_rs, y_rs;
    int32_t rows, n, k;
    float eps;
    int32_t norm;
    int32_t groups;  // column groups (workgroups per row half)
    // products of the same sizes in one launch (grid.y): operands `batch index * stride` elements further on
    int64_t w_bs, x_bs, y_bs, yp_bs;
    int32_t yp_col_step;    // columns a product's packed result is moved by (results side by side in one rows form)
    const int32_t* select;  // run only products whose index is listed here, or null
    int32_t n_select;
    int32_t grid_y, batches; // workgroups along y: one per product or, by_list, one per entry of a list that is shorter than the
    bool by_list;            // products are: seven of eight of 64 experts' workgroups would start only to leave (one row, eight experts of
                             // 2048 x 768, in a captured sequence: gate|up 10.3 -> 8.8 us a launch, down 8.4 -> 5.4; eight rows 10.9 -> 9.5, 9.2 -> 5.7)
    float c0, c1;           // constants of the activation
    // a second layer over the same rows, with the same norm, as the column groups from groups1 on (or w2 == null): tah_linear_beside
    const bf16x8* w2;
    const __bf16* bias2;
    __bf16* y2;
    int64_t y2_rs;
    int32_t act2, groups1;
};

// 16-byte unit of the packed rows form that holds row r, columns k ... k + 7 (k % 8 == 0)
__device__ __host__ __forceinline__ int64_t packed_rows_unit(int r, int k) {
    return ((int64_t)(k / kStepK) * 2 + r / 16) * 64 + (r % 16) + 16 * ((k % kStepK) / 8);
}

__device__ __forceinline__ float silu_f(float x) { return x / (1.0f + fast_exp2(-x * kLog2e)); }

// x[s][0] of step s: lane c of a k group takes what lane c + kRows * (s % kPer) of the group loaded (lanes past the group's end: 0)
typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4;
template <int kRows, int kShift>
__device__ __forceinline__ bf16x8 from_lane_above(bf16x8 v) {
    if constexpr (kShift == 0) return v;
    else {
        u32x4 u = __builtin_bit_cast(u32x4, v);
#pragma unroll
        for (int q = 0; q < 4; ++q) u[q] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)u[q], 0x100 + kShift, 0xf, 0xf, true);  // row_shl
        return __builtin_bit_cast(bf16x8, u);
    }
}
template <int kPer, int kRows, class X, int... S>
__device__ __forceinline__ void take_steps(const bf16x8* together, X& x, std::integer_sequence<int, S...>) {
    ((x[S][0] = from_lane_above<kRows, kRows * (S % kPer)>(together[S / kPer])), ...);
}


// NC: weight tiles per workgroup (1 plain, 2 or 3 for gate|up).  CH: steps per chunk of loads.  PW: steps per wave
// when K is known at compile time (K = 32 * 8 * PW), 0: any K % 32 == 0.  NH: row halves per workgroup -- 2: all 32
// rows; 1: sixteen rows, the grid holds a workgroup per (column group, half) (or only the first half when there
// are at most 16 rows).  A layer with few column groups (n = 2048: 128) then fills the chip, and every compute
// unit pulls half of the rows' operand; the second reader of a weight tile is placed on the same XCD, whose L2 has
// it or is fetching it.
// H8 (one tile, sixteen rows, K known): a workgroup takes eight of the tile's sixteen columns, so a layer whose tiles would
// occupy half of the compute units occupies all.  A load then covers two k steps of the eight columns (lanes c < 8 the
// even one, the others the odd one: 128 contiguous bytes each), and each loaded operand is multiplied twice, by either
// step's rows; of the first product the columns below 8 count, of the second those from 8 on.  At one to eight rows o
// (8 MB) takes 5.05 -> 4.65 us, down (25 MB) 9.6 -> 7.6, with the rows' operand folded (below); down at sixteen rows 9.5 -> 8.5.
template <int NC, int CH, int EPI, int PW, int NH, bool H8 = false, int kFold = 0>
__global__ __launch_bounds__(kLinThreads) void linear_rows_kernel(const LinParams p) {
    __shared__ __align__(16) float red[kLinWaves][NC][16 * NH][kTileCols];
    __shared__ float ssq[kLinWaves][16 * NH];
    __shared__ float ssum[EPI == kPlainLayerNorm ? kLinWaves : 1][16 * NH];
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int c = lane % 16, kg = lane / 16;
    int batch = blockIdx.y;
    if (p.select) {  // (every wave looks for itself: the answer is the same in all of them)
        bool hit = false;
        if (p.by_list) {
            const int at = batch;
            batch = p.select[at];
            for (int i = lane; i < at; i += kWave) hit |= p.select[i] == batch;  // listed before: that workgroup's
            if (__ballot(hit) != 0 || batch < 0 || batch >= p.batches) return;
        } else {
            for (int i = lane; i < p.n_select; i += kWave) hit |= p.select[i] == batch;
            if (__ballot(hit) == 0) return;
        }
    }
    const bf16x8* pw = p.w + batch * (p.w_bs / 8);
    const bf16x8* const px = p.x + batch * (p.x_bs / 8);
    int group = blockIdx.x, half = 0;
    if (NH == 1 && (int)gridDim.x == 2 * p.groups) {
        if (p.groups % 8 == 0) {  // workgroups go to the XCDs round robin: i and i + 8 share one
            group = (blockIdx.x / 16) * 8 + blockIdx.x % 8;
            half = (blockIdx.x / 8) % 2;
        } else {
            group = blockIdx.x / 2;
            half = blockIdx.x % 2;
        }
    }
    const __bf16* bias = p.bias;
    __bf16* y = p.y + batch * p.y_bs;
    int64_t y_rs = p.y_rs;
    int act = p.act;
    if constexpr (NC == 2 && EPI == kPlainNorm) {
        if (p.w2 && group >= p.groups1) {  // (uniform)
            group -= p.groups1;
            pw = p.w2;
            bias = p.bias2;
            y = p.y2;
            y_rs = p.y2_rs;
            act = p.act2;
        }
    }
    // The epilogue's own operands (residual, bias: 16 bytes each for a thread that writes results) are asked for here:
    // requested behind the reduction they would cost the kernel one trip to memory each, one after the other.
    constexpr bool kGateEpi = EPI == kGateUp16 || EPI == kGateUp24;
    constexpr int kEpiUnits = H8 ? 1 : EPI == kGateUp24 ? 3 : (kGateEpi ? 2 : 2 * NC);
    constexpr int kCols = H8 ? 8 : NC * kTileCols;  // a plain layer's columns per workgroup
    bf16x8 res_early = {0, 0, 0, 0, 0, 0, 0, 0}, bias_early = {0, 0, 0, 0, 0, 0, 0, 0};
    if constexpr (!kGateEpi) {
        const bool writer = (int)threadIdx.x < 16 * NH * kEpiUnits;
        const int erow = 16 * half + (writer ? (int)threadIdx.x / kEpiUnits : 0);
        const int en0 = group * kCols + 8 * (writer ? (int)threadIdx.x % kEpiUnits : 0);
        const bool live_row = erow < p.rows;
        // (addresses picked by selects, so that no load sits under a branch)
        const __bf16* ra = (p.res && live_row) ? p.res + (int64_t)erow * p.res_rs + en0 : reinterpret_cast<const __bf16*>(px);
        const __bf16* ba = bias ? bias + en0 : reinterpret_cast<const __bf16*>(px);
        res_early = *reinterpret_cast<const bf16x8*>(ra);
        bias_early = *reinterpret_cast<const bf16x8*>(ba);
    }
    const int steps = p.k / kStepK;
    const int per_wave = PW > 0 ? PW : (steps + kLinWaves - 1) / kLinWaves;
    int nst = steps - wave * per_wave;
    nst = nst < 0 ? 0 : (nst > per_wave ? per_wave : nst);
    const int s0 = nst > 0 ? wave * per_wave : 0;  // a wave without steps still points at valid memory
    const bf16x8* wb[NC];
#pragma unroll
    for (int t = 0; t < NC; ++t)
        wb[t] = H8 ? pw + ((int64_t)(group / 2) * steps + s0 + c / 8) * 64 + 16 * kg + 8 * (group % 2) + c % 8
                   : pw + ((int64_t)(group * NC + t) * steps + s0) * 64 + lane;
    // kFold: the lanes of rows past the last one read row 0's operand again instead of their zeros (their results are not used):
    // with up to eight rows a load then touches a half to a quarter of the bytes (gate|up at one to eight rows 11.7 -> 11.5 us).
    // Folded further where a wave's steps are one chunk: with one, two, four or eight rows (the next of these) the sixteen lanes of a k
    // group hold sixteen, eight, four or two steps of them, so 24 steps take 2, 3, 6 or 12 loads instead of 24 -- behind those the
    // weights' own would wait -- and a lane gets its step from its neighbours inside the vector pipe: down 8.2 -> 7.6 us at one to
    // eight rows (of a bound of 7.0, the same kernel with two of its operand loads), q|k|v 5.7 -> 5.2.
    constexpr int kFoldRows = kFold > 0 && kFold < 16 ? kFold : 16, kPerLoad = kFoldRows < 16 ? 16 / kFoldRows : 0;
    static_assert(kPerLoad == 0 || (CH == PW && NH == 1), "one chunk");
    const bf16x8* xb = px + (int64_t)s0 * 128 + 64 * half + (kPerLoad ? (c / kFoldRows) * 128 + 16 * kg + c % kFoldRows : kFold ? 16 * kg + (c < p.rows ? c : 0) : lane);

    struct Buf {
        bf16x8 w[H8 ? CH / 2 : CH][NC], x[CH][NH];
    };
    f32x4 acc[NC][H8 ? 2 : NH];  // (H8: of the even and of the odd steps)
#pragma unroll
    for (int t = 0; t < NC; ++t)
#pragma unroll
        for (int h = 0; h < (H8 ? 2 : NH); ++h) acc[t][h] = f32x4{0.f, 0.f, 0.f, 0.f};
    float ss0 = 0.f, ss1 = 0.f, sm0 = 0.f, sm1 = 0.f;
    const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
    // Loads of chunk ch.  Without a compile-time K a step past the wave's share reads step 0 of the wave's range
    // (valid memory) and is multiplied by rows of zeros: no branch sits between the loads.
    auto issue = [&](int ch, Buf& b) __attribute__((always_inline)) {
        // the rows' operand first: it comes from L2 and is there long before the weights are, and a wave's loads
        // return in order -- behind the weight loads it would only arrive after their trip to HBM (down 11.2 -> 9.6 us)
        bf16x8 together[kPerLoad ? (CH + kPerLoad - 1) / kPerLoad : 1];
        if constexpr (kPerLoad > 0) {
#pragma unroll
            for (int j = 0; j < (CH + kPerLoad - 1) / kPerLoad; ++j) {
                int back = j * kPerLoad + c / kFoldRows - (CH - 1);  // a last load's steps past the chunk: the last step again
                back = back > 0 ? back : 0;
                together[j] = xb[(j * kPerLoad - back) * 128];
            }
        } else {
#pragma unroll
            for (int s = 0; s < CH; ++s) {
                const int st = ch * CH + s;
                const int64_t sti = (PW > 0 || st < nst) ? st : 0;
                b.x[s][0] = xb[sti * 128];
                if constexpr (NH == 2) b.x[s][1] = xb[sti * 128 + 64];
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < CH; s += H8 ? 2 : 1) {
            const int st = ch * CH + s;
            const int64_t sti = (PW > 0 || st < nst) ? st : 0;
#pragma unroll
            for (int t = 0; t < NC; ++t) b.w[H8 ? s / 2 : s][t] = __builtin_nontemporal_load(wb[t] + sti * 64);
        }
        if constexpr (kPerLoad > 0) {  // each step's rows move to the lanes of the first rows while the weights are on their way
            __builtin_amdgcn_sched_barrier(0);
            take_steps<kPerLoad, kFoldRows>(together, b.x, std::make_integer_sequence<int, CH>{});
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto multiply = [&](int ch, Buf& b) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < CH; ++s) {
            const bool ok = PW > 0 || ch * CH + s < nst;
            const bf16x8 a0 = ok ? b.x[s][0] : zero8, a1 = ok ? b.x[s][NH - 1] : zero8;
            if constexpr (EPI != kPlain) {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float u = (float)a0[i], v = (float)a1[i];
                    ss0 += u * u;
                    ss1 += v * v;
                    if constexpr (EPI == kPlainLayerNorm) {
                        sm0 += u;
                        sm1 += v;
                    }
                }
            }
#pragma unroll
            for (int t = 0; t < NC; ++t) {
                if constexpr (H8) {
                    acc[t][s % 2] = mfma16(a0, b.w[s / 2][t], acc[t][s % 2]);
                } else {
                    acc[t][0] = mfma16(a0, b.w[s][t], acc[t][0]);
                    if constexpr (NH == 2) acc[t][1] = mfma16(a1, b.w[s][t], acc[t][1]);
                }
            }
        }
    };
    if constexpr (PW > 0) {
        static_assert(PW == 0 || PW % CH == 0, "chunks divide a wave's steps");
        constexpr int kChunks = PW > 0 ? PW / CH : 1;
        Buf b[2];
        issue(0, b[0]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ch = 0; ch < kChunks; ++ch) {
            if (ch + 1 < kChunks) issue(ch + 1, b[(ch + 1) % 2]);
            __builtin_amdgcn_sched_barrier(0);
            multiply(ch, b[ch % 2]);
        }
    } else {
        Buf b0, b1;
        const int nch = (nst + CH - 1) / CH;
        issue(0, b0);
        __builtin_amdgcn_sched_barrier(0);
        for (int ch = 0; ch < nch; ch += 2) {
            if (ch + 1 < nch) issue(ch + 1, b1);
            __builtin_amdgcn_sched_barrier(0);
            multiply(ch, b0);
            __builtin_amdgcn_sched_barrier(0);
            if (ch + 2 < nch) issue(ch + 2, b0);
            __builtin_amdgcn_sched_barrier(0);
            if (ch + 1 < nch) multiply(ch + 1, b1);  // never multiply a buffer that was not loaded
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // ---- the eight K slices meet in LDS ------------------------------------------------------------------
    // accumulator (tile t, half h, register r) of lane (c, kg) is row 16 h + 4 kg + r, column c of tile t
#pragma unroll
    for (int t = 0; t < NC; ++t)
#pragma unroll
        for (int h = 0; h < NH; ++h)
#pragma unroll
            for (int r = 0; r < 4; ++r) red[wave][t][16 * h + 4 * kg + r][c] = (H8 && c >= 8) ? acc[t][NH][r] : acc[t][h][r];
    if constexpr (EPI != kPlain) {
        // a lane's squares cover its 8 of every 32 k of rows c and 16 + c: add the four k groups
        ss0 += __shfl_xor(ss0, 16);
        ss0 += __shfl_xor(ss0, 32);
        ss1 += __shfl_xor(ss1, 16);
        ss1 += __shfl_xor(ss1, 32);
        if (kg == 0) {
            ssq[wave][c] = ss0;
            if constexpr (NH == 2) ssq[wave][16 + c] = ss1;
        }
        if constexpr (EPI == kPlainLayerNorm) {
            sm0 += __shfl_xor(sm0, 16);
            sm0 += __shfl_xor(sm0, 32);
            sm1 += __shfl_xor(sm1, 16);
            sm1 += __shfl_xor(sm1, 32);
            if (kg == 0) {
                ssum[wave][c] = sm0;
                if constexpr (NH == 2) ssum[wave][16 + c] = sm1;
            }
        }
    }
    __syncthreads();

    // ---- epilogue: one thread per (row, 8 output columns) -------------------------------------------------
    constexpr bool kGate = EPI == kGateUp16 || EPI == kGateUp24;
    constexpr int kUnits = H8 ? 1 : EPI == kGateUp24 ? 3 : (kGate ? 2 : 2 * NC);  // 8-column units of output per row and workgroup
    if (threadIdx.x >= 16 * NH * kUnits) return;
    const int lrow = threadIdx.x / kUnits, unit = threadIdx.x % kUnits;  // row inside the workgroup's rows
    const int row = 16 * half + lrow;
    // where the unit's gate (or plain) and up sums sit: tile and first column inside it
    int gt = kGate ? 0 : unit / 2, gc = kGate ? 8 * unit : 8 * (unit % 2), ut = 1, uc = 8 * unit;
    if constexpr (EPI == kGateUp24) {  // tiles: gate 0-15 | gate 16-23, up 16-23 | up 0-15
        gt = unit == 2 ? 1 : 0;
        gc = unit == 1 ? 8 : 0;
        ut = unit == 2 ? 1 : 2;
        uc = unit == 0 ? 0 : 8;
    }
    float sg[8], su[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) sg[i] = su[i] = 0.f;
#pragma unroll
    for (int w = 0; w < kLinWaves; ++w) {
        const f32x4 lo = *reinterpret_cast<const f32x4*>(&red[w][gt][lrow][gc]);
        const f32x4 hi = *reinterpret_cast<const f32x4*>(&red[w][gt][lrow][gc + 4]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            sg[i] += lo[i];
            sg[4 + i] += hi[i];
        }
        if constexpr (H8) {  // the odd steps' sums
            const f32x4 olo = *reinterpret_cast<const f32x4*>(&red[w][0][lrow][8]);
            const f32x4 ohi = *reinterpret_cast<const f32x4*>(&red[w][0][lrow][12]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                sg[i] += olo[i];
                sg[4 + i] += ohi[i];
            }
        }
        if constexpr (kGate) {
            const f32x4 ulo = *reinterpret_cast<const f32x4*>(&red[w][ut][lrow][uc]);
            const f32x4 uhi = *reinterpret_cast<const f32x4*>(&red[w][ut][lrow][uc + 4]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                su[i] += ulo[i];
                su[4 + i] += uhi[i];
            }
        }
    }
    const int n0 = group * (EPI == kGateUp24 ? kGroup24 : (kGate ? kTileCols : kCols)) + 8 * unit;
    const bool live = row < p.rows;
    bf16x8 out = zero8;
    if (live) {
        float rin = 1.0f;
        if constexpr (EPI != kPlain) {
            if (p.norm) {
                float ss = 0.f;
#pragma unroll
                for (int w = 0; w < kLinWaves; ++w) ss += ssq[w][lrow];
                if constexpr (EPI == kPlainLayerNorm) {
                    float sm = 0.f;
#pragma unroll
                    for (int w = 0; w < kLinWaves; ++w) sm += ssum[w][lrow];
                    const float mean = sm / (float)p.k;
                    const float var = fmaxf(ss / (float)p.k - mean * mean, 0.f);
                    rin = __builtin_amdgcn_rsqf(var + p.eps);
                    const f32x4 c0 = *reinterpret_cast<const f32x4*>(p.colsum + n0), c1 = *reinterpret_cast<const f32x4*>(p.colsum + n0 + 4);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        sg[i] -= mean * c0[i];
                        sg[4 + i] -= mean * c1[i];
                    }
                } else {
                    rin = __builtin_amdgcn_rsqf(ss / (float)p.k + p.eps);
                }
            }
        }
        if constexpr (kGate) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                // the projections' own rounding to bf16, the activation's, the product's (Qwen3MLP.forward)
                const float g = (float)(__bf16)(sg[i] * rin), u = (float)(__bf16)(su[i] * rin);
                out[i] = p.act == TAH_ACT_CLAMPED_GATE ? (__bf16)clamped_gate(g, u, p.c0, p.c1) : (__bf16)((float)(__bf16)silu_f(g) * u);
            }
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) out[i] = (__bf16)(sg[i] * rin);
            if (bias) {
#pragma unroll
                for (int i = 0; i < 8; ++i) out[i] = (__bf16)((float)out[i] + (float)bias_early[i]);
            }
            if (p.res) {
#pragma unroll
                for (int i = 0; i < 8; ++i) out[i] = (__bf16)((float)out[i] + (float)res_early[i]);
            }
            if (act == TAH_ACT_RELU) {
#pragma unroll
                for (int i = 0; i < 8; ++i) out[i] = (float)out[i] > 0.f ? out[i] : (__bf16)0.f;
            } else if (act == TAH_ACT_GELU) {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float v = (float)out[i];
                    out[i] = (__bf16)(0.5f * v * (1.0f + erff(v * 0.70710678118654752f)));
                }
            } else if (act == TAH_ACT_GELU_TANH) {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float v = (float)out[i];
                    out[i] = (__bf16)(0.5f * v * (1.0f + tanhf(0.7978845608028654f * (v + 0.044715f * v * v * v))));
                }
            } else if (act == TAH_ACT_XIELU) {
#pragma unroll
                for (int i = 0; i < 8; ++i) out[i] = (__bf16)xielu((float)out[i], p.c0, p.c1);
            }
        }
        if (p.y) *reinterpret_cast<bf16x8*>(y + (int64_t)row * y_rs + n0) = out;
    }
    if (p.yp) {
        bf16x8* const yp = p.yp + batch * (p.yp_bs / 8);
        const int nc = n0 + batch * p.yp_col_step;
        yp[packed_rows_unit(row, nc)] = out;  // rows past the last one stay zero for the next layer
        if (NH == 1 && (int)gridDim.x == p.groups) yp[packed_rows_unit(16 + lrow, nc)] = zero8;  // nobody computes the second half
    }
}

// An output head (n >= kWideFromCols plain columns, K = 256 PW) for more than sixteen rows: a resident workgroup per
// compute unit walks a range of column groups.  Its waves keep their slices of the rows' operand in registers -- read per
// group it is as many bytes as the weights and shares the L1's fill rate with them -- and ask for the next group's weights
// before they multiply and reduce this one's.  151936 x 2048, 32 rows: 116 -> 105 us (5.4 -> 5.9 TB/s), 24 rows
// 114 -> 105, inside a step 102 (6.1 TB/s); groups dealt out round robin instead of ranges 107.6 (two workgroups then write the halves of a line).
// With sixteen rows the operand is half of that and many workgroups, two or three to a compute unit, stream better (93
// against 98 us): they keep linear_rows_kernel.
template <int EPI, int PW>
__global__ __launch_bounds__(kLinThreads) void linear_wide_kernel(const LinParams p) {
    static_assert(EPI == kPlain || EPI == kPlainNorm, "plain layers");
    constexpr int NC = 2, NH = 2;
    __shared__ __align__(16) float red[kLinWaves][NC][16 * NH][kTileCols];
    __shared__ float ssq[kLinWaves][16 * NH];
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int c = lane % 16, kg = lane / 16;
    constexpr int steps = kLinWaves * PW;
    bf16x8 x[PW][NH];
    {
        const bf16x8* xb = p.x + (int64_t)wave * PW * 128 + lane;
#pragma unroll
        for (int s = 0; s < PW; ++s)
#pragma unroll
            for (int h = 0; h < NH; ++h) x[s][h] = xb[s * 128 + 64 * h];
    }
    struct Buf {
        bf16x8 w[PW][NC];
    };
    auto issue = [&](int g, Buf& b) __attribute__((always_inline)) {
        const bf16x8* wb = p.w + ((int64_t)g * NC * steps + wave * PW) * 64 + lane;
#pragma unroll
        for (int s = 0; s < PW; ++s)
#pragma unroll
            for (int t = 0; t < NC; ++t) b.w[s][t] = __builtin_nontemporal_load(wb + (int64_t)(t * steps + s) * 64);
    };
    // one thread per (row, 8 output columns)
    constexpr int kUnits = 2 * NC;
    const bool writer = (int)threadIdx.x < 16 * NH * kUnits;
    const int row = threadIdx.x / kUnits, unit = threadIdx.x % kUnits;
    float rin = 1.0f;
    auto finish = [&](int g, Buf& b) __attribute__((always_inline)) {
        f32x4 acc[NC][NH];
#pragma unroll
        for (int t = 0; t < NC; ++t)
#pragma unroll
            for (int h = 0; h < NH; ++h) acc[t][h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < PW; ++s)
#pragma unroll
            for (int t = 0; t < NC; ++t)
#pragma unroll
                for (int h = 0; h < NH; ++h) acc[t][h] = mfma16(x[s][h], b.w[s][t], acc[t][h]);
        __syncthreads();  // the group before has been read
#pragma unroll
        for (int t = 0; t < NC; ++t)
#pragma unroll
            for (int h = 0; h < NH; ++h)
#pragma unroll
                for (int r = 0; r < 4; ++r) red[wave][t][16 * h + 4 * kg + r][c] = acc[t][h][r];
        __syncthreads();
        if (!writer || row >= p.rows) return;
        float sum[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) sum[i] = 0.f;
#pragma unroll
        for (int w = 0; w < kLinWaves; ++w) {
            const f32x4 lo = *reinterpret_cast<const f32x4*>(&red[w][unit / 2][row][8 * (unit % 2)]);
            const f32x4 hi = *reinterpret_cast<const f32x4*>(&red[w][unit / 2][row][8 * (unit % 2) + 4]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                sum[i] += lo[i];
                sum[4 + i] += hi[i];
            }
        }
        bf16x8 out;
#pragma unroll
        for (int i = 0; i < 8; ++i) out[i] = (__bf16)(sum[i] * rin);
        *reinterpret_cast<bf16x8*>(p.y + (int64_t)row * p.y_rs + (int64_t)g * NC * kTileCols + 8 * unit) = out;
    };
    // (no workgroup is without a group)
    int g = (int)((int64_t)blockIdx.x * p.groups / gridDim.x);
    const int end = (int)((int64_t)(blockIdx.x + 1) * p.groups / gridDim.x);
    Buf buf[2];
    issue(g, buf[0]);
    if constexpr (EPI == kPlainNorm) {
        float ss[NH];
#pragma unroll
        for (int h = 0; h < NH; ++h) {
            ss[h] = 0.f;
#pragma unroll
            for (int s = 0; s < PW; ++s)
#pragma unroll
                for (int i = 0; i < 8; ++i) ss[h] += (float)x[s][h][i] * (float)x[s][h][i];
            ss[h] += __shfl_xor(ss[h], 16);
            ss[h] += __shfl_xor(ss[h], 32);
            if (kg == 0) ssq[wave][16 * h + c] = ss[h];
        }
        __syncthreads();
        if (writer) {
            float t = 0.f;
#pragma unroll
            for (int w = 0; w < kLinWaves; ++w) t += ssq[w][row];
            rin = __builtin_amdgcn_rsqf(t / (float)p.k + p.eps);
        }
    }
    while (true) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int next = g + 1;
            if (next < end) {
                issue(next, buf[(i + 1) % 2]);
                __builtin_amdgcn_sched_barrier(0);
                finish(g, buf[i]);
                ++g;
            } else {
                finish(g, buf[i]);
                return;
            }
        }
    }
}

// ---- a layer's four linear layers in one launch ------------------------------------------------------------
// o + residual, gate|up + SiLU, down + residual and the next layer's q|k|v of at most eight rows.  As four launches each of
// them pays its start, the first bytes' way and its reduction with the memory pipe empty; here the next phase's weights,
// which depend on nothing, are on their way while a phase's results travel between the workgroups.  2048 / 6144 / 4096 (100 MB) in a
// captured sequence of layers, against four launches: 24.1 us at one row (28.0), 24.0 at two (28.3), 24.4 at three and four (28.2),
// 25.5 at five and eight (28.9, 28.4); the weights alone take 16 us at 6.2 TB/s.  What bounds it
// now: the three hand-overs, each from the last workgroup's sums to the first product of the next phase 3.5 to 4 us (a store that has arrived 0.7 to 1, the slowest workgroup another 1, bit and poll 1.5, the rows 0.7), of which the weights
// asked for ahead hide one and parts of two.  From nine rows on it is four launches (31 us): the ninth wave's lanes hold ten rows of
// gate|up's results, and everybody reads the rows' operand past the L2s (eight rows already lose 1.4 us).  A form for them is not
// built, so what it would take is not known.  Nor is one for other layer sizes: K per wave is a template argument, and 2048 / 2048 /
// 6144 is the layer that this library's generation workloads have.
//  * A workgroup takes the same tile number of every phase (2048 / 6144: 256 tiles in each, one to a compute unit).  Eight waves
//    multiply as in linear_rows_kernel (same slices of K, same order of sums: the same bits); a ninth reduces, stores and
//    waits for the other workgroups, so that no wait for a store or a flag stands behind the weights' loads.
//  * A tile's results and then its bit in `arrived` are stored with device_store, past the XCDs' own L2 caches; readers use
//    device_load.  No fence: that would write back and invalidate the L2.
//  * Every wait ends, whatever is resident: a workgroup that has waited kChainLook polls looks which of the missing tiles belong to
//    workgroups that have not begun (another stream's work holds their compute units) and computes one of them after the other; after
//    kChainPolls polls it computes whatever is missing.  Those that wait start at different tiles (chain_pick).  All that
//    such a tile reads is there (the phase before it is complete, or the waiting workgroup would not be here), and its
//    result is the same bits whoever stores it and however often, because no result lies on an operand or on another
//    result (tah_linear_chain refuses such calls).  So one workgroup alone would finish the launch.
//    Two engines of eight layers on two streams, a tick of each: 480 us at one row (454 as four launches a layer), 557 to 609 at
//    eight (480); one such engine alone 290 and 324 (330 and 350).  When every workgroup waited its 128 polls and all took the same
//    tile: 483 to 573 and 672 to 1275.  kChainLook = 3, 5, 16: the same within those ranges.
//  * `arrived` is zero at the start; the words of the next launch (`clear`) are zeroed on the way.
constexpr int kChainTiles = TAH_LINEAR_CHAIN_TILES;  // tiles of a phase at most
// `arrived`: a bit per tile, four to a word, every word on a line of its own: a line's writes take their turns among the reads of
// everybody who waits (32 tiles to a line 31.4 us a launch, sixteen 27.6, eight 25.0, four 24.0; a byte per tile on two lines 38.5)
constexpr int kChainBits = 4, kChainLine = 32, kChainPhaseWords = kChainTiles / kChainBits * kChainLine;
static_assert(3 * kChainPhaseWords == TAH_LINEAR_CHAIN_WORDS, "header");
constexpr int kChainThreads = kLinThreads + kWave;
constexpr int kChainBegun = 1;    // word of a line, phase 0: the workgroups of these tiles have begun
#ifdef TAH_CPU_EMU
constexpr int kChainPolls = 2, kChainLook = 1;  // (workgroups run one after another there)
#else
constexpr int kChainPolls = 128;  // about 150 us: several times a whole launch
constexpr int kChainLook = 8;     // about 9 us: twice what a hand-over takes
#endif
constexpr int kChainSleep = 1;    // x 64 cycles between polls

struct ChainParams {
    const bf16x8 *w0, *w1, *w2, *w3;  // packed weights
    const bf16x8* x0;                 // packed rows: attention output
    unsigned long long *x1, *x2, *x3; // results on their way to the next phase (handed_over)
    bf16x8* out_packed;               // packed rows of `out`, or null
    const __bf16* res;                // rows the o layer adds to
    __bf16 *mid, *out, *y;            // row-major: o + residual, down + residual, q|k|v
    int64_t res_rs, mid_rs, out_rs, y_rs;
    uint32_t* arrived;
    int32_t* clear;
    int32_t rows, tiles0, tiles1, tiles2, tiles3, polls;
    float eps;
};

// Where columns col ... col + 3 of a row lie between two phases, in 8-byte words.  Nothing but the rows (rounded up to F), and
// a wave's 8-byte load of 64 operands' halves covers 512 bytes that lie together: every compute unit reads all of it past the L2s,
// and in the packed rows form (16 of 256 bytes used by one row) those requests took 1.5 us of a phase.
template <int F>
__device__ __forceinline__ int handed_over(int row, int col) {
    const int unit = (col / 8) * F + row;
    return ((unit / 64) * 2 + (col % 8) / 4) * 64 + unit % 64;
}
// While the ninth wave stores results and asks for others', a wave has this many loads of weights on their way at most: 32 KB per
// compute unit keep the memory busy, and those stores have no longer queue than that before them (all at once: they took 6.8 us to
// arrive, not 1.2).  o's weights at the start, q|k|v's second half and what is asked for again behind a tile of another workgroup go
// out all at once: the ninth wave has nothing to store then.
constexpr int kChainWindow = 4;

// A wave's part of one tile: PW steps of K, NC column tiles (H8: one, and half of its columns, as in linear_rows_kernel), rows
// folded to F.  kApart: even and odd steps are summed apart, as H8 does (a whole tile then leaves them in red's first two).
template <int PW, int NC, bool H8, int F, bool kApart = H8>
struct ChainTile {
    static_assert(NC == 1 || !kApart, "");
    static constexpr int kLoads = H8 ? PW / 2 : PW, kPer = 16 / F, kXLoads = (PW + kPer - 1) / kPer;
    bf16x8 w[kLoads][NC], x[kXLoads];
    float ss;
    f32x4 acc[NC][kApart ? 2 : 1];

    template <int kFrom, int kTo>
    __device__ __forceinline__ void ask_weights(const bf16x8* pw, int tile, int wave, int lane) {
        // (a base that is the same for the whole wave and 32-bit offsets: one address register for all loads)
        const int c = lane % 16, kg = lane / 16;
        constexpr int steps = kLinWaves * PW;
        const uint32_t own = 16 * (H8 ? 64 * (c / 8) + 16 * kg + c % 8 : lane);
#pragma unroll
        for (int i = kFrom; i < kTo; ++i)
#pragma unroll
            for (int t = 0; t < NC; ++t) {
                const bf16x8* at = H8 ? pw + ((int64_t)(tile / 2) * steps + wave * PW + 2 * i) * 64 + 8 * (tile % 2)
                                      : pw + ((int64_t)(tile * NC + t) * steps + wave * PW + i) * 64;
                uintptr_t base = reinterpret_cast<uintptr_t>(at);
                TAH_OPAQUE_S(base);
                w[i][t] = __builtin_nontemporal_load(reinterpret_cast<const TAH_GLOBAL bf16x8*>(reinterpret_cast<const TAH_GLOBAL char*>(base) + own));
            }
    }
    __device__ __forceinline__ void ask_weights(const bf16x8* pw, int tile, int wave, int lane) { ask_weights<0, kLoads>(pw, tile, wave, lane); }
    // the same with at most kChainWindow of the wave's loads on their way
    template <int kFrom, int kTo>
    __device__ __forceinline__ void trickle_weights(const bf16x8* pw, int tile, int wave, int lane) {
        if constexpr (kFrom < kTo) {
            __builtin_amdgcn_sched_barrier(0);
            TAH_WAIT_VMEM_N(kChainWindow - NC);
            ask_weights<kFrom, kFrom + 1>(pw, tile, wave, lane);
            __builtin_amdgcn_sched_barrier(0);
            trickle_weights<kFrom + 1, kTo>(pw, tile, wave, lane);
        }
    }
    __device__ __forceinline__ static int step_of(int j, int c) {
        const int step = j * kPer + c / F;
        return (j + 1) * kPer > PW && step >= PW ? PW - 1 : step;  // a last load's steps past the slice: the last step again
    }
    __device__ __forceinline__ void ask_rows(const bf16x8* px, int wave, int lane) {
        const int c = lane % 16, kg = lane / 16;
#pragma unroll
        for (int j = 0; j < kXLoads; ++j) x[j] = px[wave * PW * 128 + (uint32_t)(step_of(j, c) * 128 + 16 * kg + c % F)];
    }
    __device__ __forceinline__ void ask_rows(const unsigned long long* px, int wave, int lane) {
        const int c = lane % 16, kg = lane / 16;
        typedef __attribute__((__vector_size__(2 * sizeof(unsigned long long)))) unsigned long long u64x2;
#pragma unroll
        for (int j = 0; j < kXLoads; ++j) {
            const uint32_t at = handed_over<F>(c % F, 32 * (wave * PW + step_of(j, c)) + 8 * kg);
            u64x2 v;
            v[0] = device_load(px + at);
            v[1] = device_load(px + at + 64);
            x[j] = __builtin_bit_cast(bf16x8, v);
        }
    }
    __device__ __forceinline__ void start() {
        ss = 0.f;
#pragma unroll
        for (int t = 0; t < NC; ++t)
#pragma unroll
            for (int h = 0; h < (kApart ? 2 : 1); ++h) acc[t][h] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    template <bool kNorm, int S>
    __device__ __forceinline__ void step() {
        const bf16x8 a = from_lane_above<F, F * (S % kPer)>(x[S / kPer]);
        if constexpr (kNorm) {
#pragma unroll
            for (int i = 0; i < 8; ++i) ss += (float)a[i] * (float)a[i];
        }
#pragma unroll
        for (int t = 0; t < NC; ++t) {
            constexpr int half = kApart ? S % 2 : 0;
            acc[t][half] = mfma16(a, w[H8 ? S / 2 : S][t], acc[t][half]);
        }
    }
    template <bool kNorm, int kFrom, int... S>
    __device__ __forceinline__ void steps(std::integer_sequence<int, S...>) { (step<kNorm, kFrom + S>(), ...); }
    template <bool kNorm, int kFrom, int kTo>
    __device__ __forceinline__ void multiply() { steps<kNorm, kFrom>(std::make_integer_sequence<int, kTo - kFrom>{}); }
    template <bool kNorm>
    __device__ __forceinline__ void park(float (*red)[3][16][kTileCols], float (*ssq)[16], int wave, int lane) {
        const int c = lane % 16, kg = lane / 16;
#pragma unroll
        for (int t = 0; t < NC; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (4 * kg < F) {
                    red[wave][t][4 * kg + r][c] = (H8 && c >= 8) ? acc[t][H8 ? 1 : 0][r] : acc[t][0][r];
                    if constexpr (kApart && !H8) red[wave][1][4 * kg + r][c] = acc[t][1][r];
                }
        if constexpr (kNorm) {
            ss += __shfl_xor(ss, 16);
            ss += __shfl_xor(ss, 32);
            if (kg == 0) ssq[wave][c] = ss;
        }
    }
};

// One of the tiles that `take` names (a lane's kChainBits of them), -1: none.  Workgroups that see the same ones take different ones as
// far as there are any, so that what is missing gets less by as many tiles as there are workgroups that wait (each the first one: they
// all computed the same tile, a hundred missing ones took a hundred turns).
__device__ __forceinline__ int chain_pick(uint32_t take) {
    unsigned long long has[kChainBits];
    int total = 0;
#pragma unroll
    for (int b = 0; b < kChainBits; ++b) {
        has[b] = __ballot((take >> b & 1u) != 0);
        total += __builtin_popcountll(has[b]);
    }
    if (total == 0) return -1;
    int nth = (int)blockIdx.x % total, tile = -1;
#pragma unroll
    for (int b = 0; b < kChainBits; ++b) {
        const int n = __builtin_popcountll(has[b]);
        if (tile < 0 && nth < n) {
            for (int i = 0; i < nth; ++i) has[b] &= has[b] - 1;
            tile = kChainBits * __builtin_ctzll(has[b]) + b;
        }
        nth -= n;
    }
    return tile;
}

// LDS between the waves of a workgroup: loads from memory stay on their way across it
__device__ __forceinline__ void chain_barrier() {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    TAH_WAIT_LDS();
    __builtin_amdgcn_s_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// PWO, PWH, PWF: query columns, hidden size and MLP width over 256.  NEXT: the q|k|v phase (kNextApart: of so few columns that
// linear_rows takes eight at a time and sums even and odd steps apart).
enum { kNextNone, kNextWhole, kNextApart };
template <int F, int PWO, int PWH, int PWF, int NEXT>
__global__ __launch_bounds__(kChainThreads) void linear_chain_kernel(const ChainParams p) {
    __shared__ __align__(16) float red[kLinWaves][3][16][kTileCols];
    __shared__ float ssq[kLinWaves][16];
    __shared__ int command;  // a tile of the phase before to compute, or -1: go on
    const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
    const int tile = blockIdx.x;
    using O = ChainTile<PWO, 1, true, F>;
    using GateUp = ChainTile<PWH, 3, false, F>;
    using Down = ChainTile<PWF, 1, true, F>;
    constexpr bool kNext = NEXT != kNextNone;
    using Qkv = ChainTile<PWH, 1, false, F, NEXT == kNextApart>;
    // (a workgroup without a tile in a phase multiplies another's and stores nothing)
    const int t0 = tile < p.tiles0 ? tile : 0, t1 = tile < p.tiles1 ? tile : 0, t2 = tile < p.tiles2 ? tile : 0, t3 = tile < p.tiles3 ? tile : 0;

    if (wave < kLinWaves) {
        // until the phase before is complete, with tiles that others should have computed; the weights on their way are asked for
        // again behind those (they share registers with them)
        auto wait = [&](auto help, auto ask_again) __attribute__((always_inline)) {
            chain_barrier();
            int missing = command;
            if (missing >= 0) {
                do {
                    help(missing);
                    chain_barrier();
                    chain_barrier();
                    missing = command;
                } while (missing >= 0);
                ask_again();
            }
        };
        auto help0 = [&](int missing) __attribute__((always_inline)) {
            O o;
            o.ask_rows(p.x0, wave, lane);
            o.ask_weights(p.w0, missing, wave, lane);
            o.start();
            o.template multiply<false, 0, PWO>();
            o.template park<false>(red, ssq, wave, lane);
        };
        auto help1 = [&](int missing) __attribute__((always_inline)) {
            GateUp g;
            g.ask_rows(p.x1, wave, lane);
            g.ask_weights(p.w1, missing, wave, lane);
            g.start();
            g.template multiply<true, 0, PWH>();
            g.template park<true>(red, ssq, wave, lane);
        };
        auto help2 = [&](int missing) __attribute__((always_inline)) {
            Down d;
            d.ask_rows(p.x2, wave, lane);
            d.ask_weights(p.w2, missing, wave, lane);
            d.start();
            d.template multiply<false, 0, PWF>();
            d.template park<false>(red, ssq, wave, lane);
        };
        constexpr int kDownAhead = Down::kLoads / 3, kQkvAhead = kNext ? Qkv::kLoads / 2 : 0;  // (nine waves leave 168 registers)
        GateUp gu;
        Down down;
        Qkv qkv;
        {
            O o;
            o.ask_rows(p.x0, wave, lane);
            __builtin_amdgcn_sched_barrier(0);
            o.ask_weights(p.w0, t0, wave, lane);
            __builtin_amdgcn_sched_barrier(0);
            o.start();
            o.template multiply<false, 0, PWO>();
            o.template park<false>(red, ssq, wave, lane);
            chain_barrier();
            gu.template trickle_weights<0, PWH>(p.w1, t1, wave, lane);
            down.template trickle_weights<0, kDownAhead>(p.w2, t2, wave, lane);
        }
        wait(help0, [&]() __attribute__((always_inline)) { 
            gu.ask_weights(p.w1, t1, wave, lane);
            down.template ask_weights<0, kDownAhead>(p.w2, t2, wave, lane);
        });
        gu.ask_rows(p.x1, wave, lane);
        gu.start();
        gu.template multiply<true, 0, PWH>();
        gu.template park<true>(red, ssq, wave, lane);
        chain_barrier();
        down.template trickle_weights<kDownAhead, Down::kLoads>(p.w2, t2, wave, lane);
        qkv.template trickle_weights<0, kQkvAhead>(p.w3, t3, wave, lane);

        wait(help1, [&]() __attribute__((always_inline)) { 
            down.ask_weights(p.w2, t2, wave, lane);
            qkv.template ask_weights<0, kQkvAhead>(p.w3, t3, wave, lane);
        });
        down.ask_rows(p.x2, wave, lane);
        chain_barrier();
        if constexpr (kNext) qkv.template ask_weights<kQkvAhead, Qkv::kLoads>(p.w3, t3, wave, lane);
        __builtin_amdgcn_sched_barrier(0);
        down.start();
        down.template multiply<false, 0, PWF>();
        down.template park<false>(red, ssq, wave, lane);
        chain_barrier();

        if constexpr (kNext) {
            wait(help2, [&]() __attribute__((always_inline)) { qkv.ask_weights(p.w3, t3, wave, lane); });
            qkv.ask_rows(p.x3, wave, lane);
            qkv.start();
            qkv.template multiply<false, 0, PWH>();
            qkv.template park<false>(red, ssq, wave, lane);
            chain_barrier();
        }
        return;
    }

    // ---- the ninth wave: a lane per (row, 2 columns) of the eight-column tiles, per (row, 4 columns) of the others; all partial
    // sums are asked for before the first is added, in the order of linear_rows_kernel ----
    typedef __attribute__((__vector_size__(2 * sizeof(float)))) float f32x2;
    typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2;
    typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
    if (lane == 0) device_or(p.arrived + tile / kChainBits * kChainLine + kChainBegun, 1u << (tile % kChainBits));
    for (int i = (int)blockIdx.x * kWave + lane; i < TAH_LINEAR_CHAIN_WORDS; i += (int)gridDim.x * kWave) p.clear[i] = 0;
    // rows past the last one are zeros in the rows form that stays
    if (p.out_packed && tile < p.tiles2 && lane >= p.rows && lane < kLinRows) p.out_packed[packed_rows_unit(lane, 8 * tile)] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
    const int row2 = lane / 4, col2 = 2 * (lane % 4);
    const bool live2 = row2 < p.rows;
    auto sum_even_odd = [&](float* s) __attribute__((always_inline)) {
        f32x2 part[kLinWaves][2];
#pragma unroll
        for (int w = 0; w < kLinWaves; ++w)
#pragma unroll
            for (int odd = 0; odd < 2; ++odd) part[w][odd] = *reinterpret_cast<const f32x2*>(&red[w][0][row2][8 * odd + col2]);
        __builtin_amdgcn_sched_barrier(0);
        s[0] = s[1] = 0.f;
#pragma unroll
        for (int w = 0; w < kLinWaves; ++w)
#pragma unroll
            for (int odd = 0; odd < 2; ++odd) {
                s[0] += part[w][odd][0];
                s[1] += part[w][odd][1];
            }
    };
    auto ask4 = [&](f32x4 (&part)[kLinWaves], int t, int row, int col) __attribute__((always_inline)) {
#pragma unroll
        for (int w = 0; w < kLinWaves; ++w) part[w] = *reinterpret_cast<const f32x4*>(&red[w][t][row][col]);
    };
    auto sum4 = [&](const f32x4 (&part)[kLinWaves]) __attribute__((always_inline)) {
        f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < kLinWaves; ++w) s += part[w];
        return s;
    };
    auto announce = [&](int phase, int of) __attribute__((always_inline)) {
        device_settle();  // the results are there before the word that says so
        if (lane == 0) device_or(p.arrived + phase * kChainPhaseWords + of / kChainBits * kChainLine, 1u << (of % kChainBits));
    };
    auto hand_over2 = [&](unsigned long long* to, int of, bf16x2 o) __attribute__((always_inline)) {
        device_store(reinterpret_cast<uint32_t*>(to + handed_over<F>(row2, 8 * of + col2)) + (col2 % 4) / 2, __builtin_bit_cast(uint32_t, o));
    };
    auto plus = [&](const float* s, bf16x2 r) __attribute__((always_inline)) {
        bf16x2 o;
#pragma unroll
        for (int i = 0; i < 2; ++i) o[i] = (__bf16)((float)(__bf16)s[i] + (float)r[i]);
        return o;
    };
    auto finish0 = [&](int of, bf16x2 r) __attribute__((always_inline)) {
        bf16x2 o = r;
        if (live2) {
            float s[2];
            sum_even_odd(s);
            o = plus(s, r);
            hand_over2(p.x1, of, o);
            device_store(reinterpret_cast<uint32_t*>(p.mid + (int64_t)row2 * p.mid_rs + 8 * of + col2), __builtin_bit_cast(uint32_t, o));
        }
        announce(0, of);
        return o;
    };
    auto finish1 = [&](int of) __attribute__((always_inline)) {
        const int row = lane / 6, col = 4 * (lane % 6);
        if (row < p.rows) {
            // tiles: gate 0-15 | gate 16-23, up 16-23 | up 0-15
            const bool last = col >= 16;
            f32x4 g[kLinWaves], u[kLinWaves];
            float sq[kLinWaves];
            ask4(g, last ? 1 : 0, row, last ? col - 16 : col);
            ask4(u, last ? 1 : 2, row, last ? col - 8 : col);
#pragma unroll
            for (int w = 0; w < kLinWaves; ++w) sq[w] = ssq[w][row];
            __builtin_amdgcn_sched_barrier(0);
            const f32x4 sg = sum4(g), su = sum4(u);
            float ss = 0.f;
#pragma unroll
            for (int w = 0; w < kLinWaves; ++w) ss += sq[w];
            const float rin = __builtin_amdgcn_rsqf(ss / (float)(256 * PWH) + p.eps);
            bf16x4 o;
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = (__bf16)((float)(__bf16)silu_f((float)(__bf16)(sg[i] * rin)) * (float)(__bf16)(su[i] * rin));
            device_store(p.x2 + handed_over<F>(row, kGroup24 * of + col), __builtin_bit_cast(unsigned long long, o));
        }
        announce(1, of);
    };
    auto finish2 = [&](int of, bf16x2 r) __attribute__((always_inline)) {
        if (live2) {
            float s[2];
            sum_even_odd(s);
            const bf16x2 o = plus(s, r);
            if (kNext) hand_over2(p.x3, of, o);
            if (p.out_packed) *reinterpret_cast<bf16x2*>(reinterpret_cast<__bf16*>(p.out_packed + packed_rows_unit(row2, 8 * of)) + col2) = o;
            *reinterpret_cast<bf16x2*>(p.out + (int64_t)row2 * p.out_rs + 8 * of + col2) = o;
        }
        if (kNext) announce(2, of);
    };
    // until all tiles of a phase have arrived; a tile that does not come is computed here
    int look = kChainLook;
    auto wait = [&](int phase, int tiles, auto finish) __attribute__((always_inline)) {
        // a word per lane
        const int first = kChainBits * lane, mine = tiles - first < kChainBits ? tiles - first : kChainBits;
        const uint32_t* const word = p.arrived + phase * kChainPhaseWords + lane * kChainLine;
        uint32_t absent = mine > 0 ? (1u << mine) - 1u : 0u;
        for (int polls = 1;; ++polls) {
            if (absent != 0) absent &= ~device_load(word);  // (a word that is complete is not read again: reads are in the writers' way)
            if (__ballot(absent != 0) == 0) break;
            uint32_t take = 0;
            if (polls >= p.polls) take = absent;
            else if (polls >= look && absent != 0) take = absent & ~device_load(p.arrived + lane * kChainLine + kChainBegun);
            const int missing = chain_pick(take);
            if (missing >= 0) {
                if (lane == 0) command = missing;
                chain_barrier();
                chain_barrier();
                finish(missing);
                if (lane == missing / kChainBits) absent &= ~(1u << (missing % kChainBits));  // (the word may not say so yet)
                look = 1;  // (workgroups have not begun: looked for at once from now on)
            } else {
                TAH_SLEEP(kChainSleep);
            }
        }
        if (lane == 0) command = -1;
        chain_barrier();
        if (phase == 1) chain_barrier();  // (between the waves' loads of the rows and those of weights)
    };
    auto residual = [&](int of) __attribute__((always_inline)) {
        bf16x2 r = {0, 0};
        if (live2) r = *reinterpret_cast<const bf16x2*>(p.res + (int64_t)row2 * p.res_rs + 8 * of + col2);
        return r;
    };
    bf16x2 mid = residual(t0);
    chain_barrier();
    if (tile < p.tiles0) mid = finish0(tile, mid);
    wait(0, p.tiles0, [&](int of) __attribute__((always_inline)) { finish0(of, residual(of)); });
    chain_barrier();
    if (tile < p.tiles1) finish1(tile);
    wait(1, p.tiles1, finish1);
    chain_barrier();
    if (tile < p.tiles2) finish2(tile, mid);  // (tiles0 = tiles2: its own columns of o + residual are still here)
    if constexpr (kNext) {
        wait(2, p.tiles2, [&](int of) __attribute__((always_inline)) {
            uint32_t r = 0;
            if (live2) r = device_load(reinterpret_cast<const uint32_t*>(p.mid + (int64_t)row2 * p.mid_rs + 8 * of + col2));
            finish2(of, __builtin_bit_cast(bf16x2, r));
        });
        chain_barrier();
        const int row = lane / 4, col = 4 * (lane % 4);
        if (tile < p.tiles3 && row < p.rows) {
            f32x4 s = {0.f, 0.f, 0.f, 0.f}, part[kLinWaves], odd[kLinWaves];
            ask4(part, 0, row, col);
            if constexpr (NEXT == kNextApart) ask4(odd, 1, row, col);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int w = 0; w < kLinWaves; ++w) {
                s += part[w];
                if constexpr (NEXT == kNextApart) s += odd[w];
            }
            bf16x4 o;
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = (__bf16)s[i];
            *reinterpret_cast<bf16x4*>(p.y + (int64_t)row * p.y_rs + kTileCols * tile + col) = o;
        }
    }
}

// What a plain layer's tile leaves of at most two rows: sums, activation, row-major and / or rows form.
struct LinearOut {
    __bf16* y;
    bf16x8* yp;
    int64_t y_rs;
    int32_t act, rows;
    float c0, c1;
};
template <bool H8>
__device__ __forceinline__ void finish_plain_tile(const LinearOut& p, const float (*red)[3][16][kTileCols]) {
    // a lane per row (rows past the last one are zeros in the rows form) and eight columns
    constexpr int kUnits = H8 ? 1 : 2;
    if ((int)threadIdx.x >= kLinRows * kUnits) return;
    const int row = threadIdx.x % kLinRows, unit = threadIdx.x / kLinRows, n0 = (int)blockIdx.x * 8 * kUnits + 8 * unit;
    bf16x8 out = {0, 0, 0, 0, 0, 0, 0, 0};
    if (row < p.rows) {
        float s[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) s[i] = 0.f;
#pragma unroll
        for (int w = 0; w < kLinWaves; ++w)
#pragma unroll
            for (int half = 0; half < (H8 ? 2 : 1); ++half) {  // (H8: the even and the odd steps' sums)
                const f32x4 lo = *reinterpret_cast<const f32x4*>(&red[w][0][row][8 * (H8 ? half : unit)]);
                const f32x4 hi = *reinterpret_cast<const f32x4*>(&red[w][0][row][8 * (H8 ? half : unit) + 4]);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    s[i] += lo[i];
                    s[4 + i] += hi[i];
                }
            }
#pragma unroll
        for (int i = 0; i < 8; ++i) out[i] = (__bf16)s[i];
        if (p.act == TAH_ACT_GELU_TANH) {
#pragma unroll
            for (int i = 0; i < 8; ++i) out[i] = (__bf16)gelu_tanh_exact((float)out[i]);
        } else if (p.act == TAH_ACT_XIELU) {
#pragma unroll
            for (int i = 0; i < 8; ++i) out[i] = (__bf16)xielu((float)out[i], p.c0, p.c1);
        }
        if (p.y) *reinterpret_cast<bf16x8*>(p.y + (int64_t)row * p.y_rs + n0) = out;
    }
    if (p.yp) p.yp[packed_rows_unit(row, n0)] = out;
}

// ---- a norm of the residual stream and the linear layer behind it in one launch ----------------------------
// One or two rows: a decode step of such a model is a chain of launches of 4.4 us and more, most of it their start and the first trip to
// memory, and a norm of a few rows is a launch of its own for 8 KB.  Here every workgroup of the layer makes the normed rows for
// itself (28 KB a row, with experts 60, with a convolution 72) while its weights are on their way, and the first one stores what is kept: the
// new residual rows and the convolution's input.  Same arithmetic in the same order as tah_residual_norm and tah_linear_rows: the same bits.
// One row in a captured step of four layers, as two launches and as one: 2048 -> 6144 behind a plain norm 4.4 + 8.0 -> 8.9 us, 2048 -> 3616 behind
// a norm with convolution (and experts) 4.4 + 4.9 -> 7.9: a step 305.9 -> 298.8 us, two rows 329.8 -> 324.2; of the other design, 2048 -> 6144, 342.4 ->
// 334.9 and 369.1 -> 361.9.  Three and four rows: the rows' bytes cost more than the launch (350.5 -> 359.3, 369.6 -> 378.4).  More than two
// workgroups to a compute unit: the rows are made three times over (2048 -> 12352, one row: a step 334.9 -> 344.2).
constexpr int kNormLinearRows = 2, kNormLinearWorkgroups = 512;
constexpr int kNormLinearSteps = 8;  // K = 256 kNormLinearSteps = a thread's eight columns for 256 threads (no other width is built or measured)
struct NormLinear {
    tah_residual_norm_args n;
    float* x_out;
    const bf16x8* w;
    LinearOut out;
};

// kMore: with experts or a convolution, whose loads take the registers of a second workgroup on the compute unit
template <int F, bool GROUPS, bool H8, bool kMore>
__global__ __launch_bounds__(kLinThreads, kMore ? 2 : 4) void norm_linear_kernel(const NormLinear p) {
    constexpr int PW = kNormLinearSteps;
    static_assert(F <= kLinThreads / kRowThreads, "all rows at a time");
    using Tile = ChainTile<PW, 1, H8, F, H8>;
    __shared__ __align__(16) float red[kLinWaves][3][16][kTileCols];
    __shared__ __align__(16) bf16x8 rows_lds[PW * kLinWaves * 4 * F];  // [step][k group][row]
    __shared__ ResidualLds<1, GROUPS> lds[kLinThreads / kRowThreads];
    const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
    const int part = wave / (kRowThreads / kWave), c = lane % 16, kg = lane / 16;
    tah_residual_norm_args n = p.n;
    if constexpr (!kMore) {
        n.experts = nullptr;
        n.conv = nullptr;
    }
    Tile t;
    const int r = F == 1 ? 0 : part;  // (of one row both halves of the workgroup make it)
    const bool own = r < p.n.rows && (F > 1 || part == 0);
    residual_row<__bf16, 1, GROUPS, true>(
        n, r < p.n.rows ? r : p.n.rows - 1, threadIdx.x % kRowThreads, lds[part], blockIdx.x == 0 && own, p.x_out,
        [&]() __attribute__((always_inline)) {
            __builtin_amdgcn_sched_barrier(0);
            t.ask_weights(p.w, blockIdx.x, wave, lane);
            __builtin_amdgcn_sched_barrier(0);
        },
        [&](int col, const float (&v)[8]) __attribute__((always_inline)) {
            if (own) rows_lds[(col / kStepK * 4 + col % kStepK / 8) * F + r] = to_bf16x8(v);
        });
    __syncthreads();
#pragma unroll
    for (int j = 0; j < Tile::kXLoads; ++j) t.x[j] = rows_lds[((wave * PW + Tile::step_of(j, c)) * 4 + kg) * F + c % F];
    t.start();
    t.template multiply<false, 0, PW>();
    t.template park<false>(red, nullptr, wave, lane);
    __syncthreads();
    finish_plain_tile<H8>(p.out, red);
}

// ---- the parts of a windowed attention's split call and the output projection behind them in one launch -------
// One or two rows: merging a call's parts was a launch of 4.7 us for 42 KB a row, and the projection behind it another of 4.5. Here
// every workgroup of the projection merges the row for itself (a compute unit takes 42 KB in in 0.4 us), its weights on their way.  The
// same bits as window_merge_kernel and tah_linear_rows leave.  From three rows on the parts cost more than the launch: two launches.  Heads
// of 2048 columns together and no other width (K per wave is the template's, as in norm_linear_kernel: no other is built or measured):
// there, too, two launches.
// One row of 16 heads in five parts, 2048 -> 2048, in a captured step: 4.7 + 4.5 -> 5.5 us.
template <int F, bool H8>
__global__ __launch_bounds__(kLinThreads) void merge_linear_kernel(const MergeLinear p, const LinearOut out, const bf16x8* weights) {
    constexpr int PW = kNormLinearSteps, kCols = 4 * F, kAhead = 8;  // columns per thread; parts on their way
    using Tile = ChainTile<PW, 1, H8, F, H8>;
    __shared__ __align__(16) float red[kLinWaves][3][16][kTileCols];
    __shared__ __align__(16) bf16x8 rows_lds[PW * kLinWaves * 4 * F];  // [step][k group][row]
    const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
    const int c = lane % 16, kg = lane / 16;
    constexpr int kPerRow = kLinThreads / F;
    const int r = (int)threadIdx.x / kPerRow, col = kCols * ((int)threadIdx.x % kPerRow), h = col / p.value_dim, vs = p.value_dim + 4;
    const int row = r < out.rows ? r : out.rows - 1;
    const float* const base = p.part + ((int64_t)row * p.heads + h) * p.splits * vs;
    const int x = col % p.value_dim;
    f32x4 v[kAhead][F];
    float vm[kAhead], vl[kAhead];
    auto ask = [&](int s0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            const float* const at = base + (int64_t)(s0 + i < p.splits ? s0 + i : p.splits - 1) * vs;
#pragma unroll
            for (int f = 0; f < F; ++f) v[i][f] = *reinterpret_cast<const f32x4*>(at + x + 4 * f);
            vm[i] = at[p.value_dim];
            vl[i] = at[p.value_dim + 1];
        }
    };
    ask(0);
    const __bf16 gate = p.gate ? p.gate[(int64_t)row * p.gate_rs + h] : (__bf16)0.f;
    Tile t;
    __builtin_amdgcn_sched_barrier(0);
    t.ask_weights(weights, blockIdx.x, wave, lane);
    __builtin_amdgcn_sched_barrier(0);
    PartsSum<kCols> sum;
    for (int s0 = 0;;) {
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            if (s0 + i >= p.splits) continue;
            float w[kCols];
#pragma unroll
            for (int e = 0; e < kCols; ++e) w[e] = v[i][e / 4][e % 4];
            sum.add(vm[i], vl[i], w);
        }
        s0 += kAhead;
        if (s0 >= p.splits) break;
        ask(s0);
    }
    const float inv = sum.factor(p.gate != nullptr, (float)gate);
    if (r < out.rows) {
        __bf16* const to = reinterpret_cast<__bf16*>(&rows_lds[(col / kStepK * 4 + col % kStepK / 8) * F + r]) + col % 8;
#pragma unroll
        for (int f = 0; f < F; ++f) {
            bf16x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = (__bf16)(sum.y[4 * f + e] * inv);
            *reinterpret_cast<bf16x4*>(to + 4 * f) = o;
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < Tile::kXLoads; ++j) t.x[j] = rows_lds[((wave * PW + Tile::step_of(j, c)) * 4 + kg) * F + c % F];
    t.start();
    t.template multiply<false, 0, PW>();
    t.template park<false>(red, nullptr, wave, lane);
    __syncthreads();
    finish_plain_tile<H8>(out, red);
}

// what is left of a launch without rows: the words of the next one
__global__ __launch_bounds__(kLinThreads) void linear_chain_clear_kernel(int32_t* clear) {
    for (int i = threadIdx.x; i < TAH_LINEAR_CHAIN_WORDS; i += kLinThreads) clear[i] = 0;
}

template <int PWO, int PWH, int PWF>
void launch_chain(const ChainParams& p, int next, hipStream_t st) {
    int tiles = p.tiles0 > p.tiles1 ? p.tiles0 : p.tiles1;
    tiles = tiles > p.tiles3 ? tiles : p.tiles3;
    const auto run = [&](auto fold) {
        constexpr int F = decltype(fold)::value;
        const dim3 grid(tiles), block(kChainThreads);
        if (next == kNextApart) hipLaunchKernelGGL((linear_chain_kernel<F, PWO, PWH, PWF, kNextApart>), grid, block, 0, st, p);
        else if (next) hipLaunchKernelGGL((linear_chain_kernel<F, PWO, PWH, PWF, kNextWhole>), grid, block, 0, st, p);
        else hipLaunchKernelGGL((linear_chain_kernel<F, PWO, PWH, PWF, kNextNone>), grid, block, 0, st, p);
    };
    if (p.rows <= 1) run(std::integral_constant<int, 1>{});
    else if (p.rows <= 2) run(std::integral_constant<int, 2>{});
    else if (p.rows <= 4) run(std::integral_constant<int, 4>{});
    else run(std::integral_constant<int, 8>{});
}

// ---- re-ordering -----------------------------------------------------------------------------------------
// Weight row behind column slot c of tile t of the packed order.
__device__ __host__ inline int64_t packed_weight_row(int kind, int n, int tile, int c) {
    if (kind == TAH_LINEAR_PLAIN) return (int64_t)tile * kTileCols + c;
    if (n % kGroup24 == 0) {  // groups of 24 output columns: gate 0-15 | gate 16-23, up 16-23 | up 0-15
        const int g = tile / 3, t = tile % 3;
        if (t == 0) return (int64_t)kGroup24 * g + c;
        if (t == 2) return (int64_t)n + kGroup24 * g + c;
        return c < 8 ? (int64_t)kGroup24 * g + 16 + c : (int64_t)n + kGroup24 * g + 16 + (c - 8);
    }
    const int g = tile / 2;  // groups of 16 output columns: gate | up
    return (tile % 2 ? (int64_t)n : 0) + (int64_t)kTileCols * g + c;
}

__global__ __launch_bounds__(256) void pack_weight_kernel(const __bf16* w, int64_t w_rs, bf16x8* out, int kind, int n, int k, int64_t units) {
    const int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (u >= units) return;
    const int steps = k / kStepK;
    const int lane = (int)(u % 64);
    const int64_t ts = u / 64;
    const int step = (int)(ts % steps), tile = (int)(ts / steps);
    const int64_t row = packed_weight_row(kind, n, tile, lane % 16);
    out[u] = *reinterpret_cast<const bf16x8*>(w + row * w_rs + step * kStepK + 8 * (lane / 16));
}

__global__ __launch_bounds__(256) void pack_rows_kernel(const __bf16* x, int64_t x_rs, bf16x8* out, int rows, int k) {
    const int u = blockIdx.x * 256 + threadIdx.x;  // (step, half, lane)
    if (u >= k / kStepK * 128) return;
    const int lane = u % 64, half = (u / 64) % 2, step = u / 128;
    const int row = 16 * half + lane % 16;
    bf16x8 v = {0, 0, 0, 0, 0, 0, 0, 0};
    if (row < rows) v = *reinterpret_cast<const bf16x8*>(x + (int64_t)row * x_rs + step * kStepK + 8 * (lane / 16));
    out[u] = v;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// Sixteen rows per workgroup when there are no more, or when the column groups alone would leave half of the
// 256 compute units idle.
constexpr int kSplitRowsBelowGroups = 129;
constexpr int kWideFromCols = 16384;  // plain layers from this many output columns on take 32 columns per workgroup

template <int EPI, int PW>
void launch_wide(LinParams& p, int groups, hipStream_t st) {
    constexpr int kResident = 256;  // a workgroup per compute unit
    p.groups = groups;
    hipLaunchKernelGGL((linear_wide_kernel<EPI, PW>), dim3(groups < kResident ? groups : kResident), dim3(kLinThreads), 0, st, p);
}

// few rows: the rows operand folded as far as their number allows
template <int NC, int CH, int EPI, int PW, bool H8>
void launch_folded(const LinParams& p, int workgroups, hipStream_t st) {
    const dim3 grid(workgroups, p.grid_y), block(kLinThreads);
    if constexpr (PW > 0 && NC != 2) {
        const auto run = [&](auto fold) { hipLaunchKernelGGL((linear_rows_kernel<NC, CH, EPI, PW, 1, H8, decltype(fold)::value>), grid, block, 0, st, p); };
        if constexpr (CH == PW) {
            if (p.rows <= 1) return run(std::integral_constant<int, 1>{});
            if (p.rows <= 2) return run(std::integral_constant<int, 2>{});
            if (p.rows <= 4) return run(std::integral_constant<int, 4>{});
            if (p.rows <= 8) return run(std::integral_constant<int, 8>{});
        }
        run(std::integral_constant<int, 16>{});
    }
}

template <int NC, int CH, int EPI, int PW>
void launch(LinParams& p, int groups, int batch, hipStream_t st) {
    p.groups = groups;
    if constexpr (NC == 1 && EPI == kPlain && PW > 0 && PW % 2 == 0) {
        // (from nine rows on the doubled reads of the rows' operand outweigh it for short sums: K = 2048, sixteen rows 5.1 ->
        // 5.5 us, where K = 4096 gains 7.6 -> 7.0 and K = 6144 9.5 -> 8.8)
        if (groups * batch < kSplitRowsBelowGroups && (p.rows <= 8 || (p.rows <= 16 && PW >= 16))) {
            p.groups = 2 * groups;
            launch_folded<1, PW, kPlain, PW, true>(p, p.groups, st);
            return;
        }
    }
    if (NC != 2 && PW > 0 && p.rows <= 8)  // (two tiles share the operand: nothing to gain)
        launch_folded<NC, CH, EPI, PW, false>(p, groups, st);
    else if (p.rows <= 16)
        hipLaunchKernelGGL((linear_rows_kernel<NC, CH, EPI, PW, 1>), dim3(groups, p.grid_y), dim3(kLinThreads), 0, st, p);
    else if (groups * batch < kSplitRowsBelowGroups)
        hipLaunchKernelGGL((linear_rows_kernel<NC, CH, EPI, PW, 1>), dim3(2 * groups, p.grid_y), dim3(kLinThreads), 0, st, p);
    else
        hipLaunchKernelGGL((linear_rows_kernel<NC, CH, EPI, PW, 2>), dim3(groups, p.grid_y), dim3(kLinThreads), 0, st, p);
}

}  // namespace
}  // namespace tah

extern "C" int tah_linear_pack_weight(const void* w, int64_t w_row_stride, void* packed, int32_t n, int32_t k, int32_t kind,
                                      tah_stream_t stream) {
    using namespace tah;
    if (kind != TAH_LINEAR_PLAIN && kind != TAH_LINEAR_GATE_UP) return TAH_E_SHAPE;
    if (n < 0 || k < 0 || k % kStepK != 0 || w_row_stride < k) return TAH_E_SHAPE;
    if (kind == TAH_LINEAR_PLAIN ? n % kTileCols != 0 : (n % kGroup24 != 0 && n % kTileCols != 0)) return TAH_E_SHAPE;
    if (n == 0 || k == 0) return TAH_OK;
    if (!w || !packed) return TAH_E_NULL;
    if (!aligned16(w) || !aligned16(packed) || w_row_stride % 8 != 0) return TAH_E_ALIGN;
    const int64_t total_rows = kind == TAH_LINEAR_GATE_UP ? 2 * (int64_t)n : n;
    const int64_t units = total_rows * k / 8;
    if ((units + 255) / 256 > 0x7fffffff) return TAH_E_SHAPE;
    hipLaunchKernelGGL(pack_weight_kernel, dim3((unsigned)((units + 255) / 256)), dim3(256), 0, static_cast<hipStream_t>(stream),
                       static_cast<const __bf16*>(w), w_row_stride, static_cast<bf16x8*>(packed), (int)kind, (int)n, (int)k, units);
    return hipGetLastError() == hipSuccess ? TAH_OK : TAH_E_LAUNCH;
}

extern "C" int tah_linear_pack_rows(const void* x, int64_t x_row_stride, void* x_packed, int32_t rows, int32_t k, tah_stream_t stream) {
    using namespace tah;
    if (rows < 0 || rows > kLinRows || k < 0 || k % kStepK != 0) return TAH_E_SHAPE;
    if (k == 0) return TAH_OK;
    if (!x_packed || (rows > 0 && !x)) return TAH_E_NULL;
    if (!aligned16(x) || !aligned16(x_packed) || (rows > 1 && x_row_stride % 8 != 0)) return TAH_E_ALIGN;
    const int units = k / kStepK * 128;
    hipLaunchKernelGGL(pack_rows_kernel, dim3((units + 255) / 256), dim3(256), 0, static_cast<hipStream_t>(stream),
                       static_cast<const __bf16*>(x), x_row_stride, static_cast<bf16x8*>(x_packed), (int)rows, (int)k);
    return hipGetLastError() == hipSuccess ? TAH_OK : TAH_E_LAUNCH;
}

namespace tah {
namespace {
// beside: a second layer of the same rows in the launch (tah_linear_beside has checked it), or null
int run_linear_rows(const tah_linear_rows_args* a, const tah_linear_rows_args* beside, tah_stream_t stream) {
    if (a->kind != TAH_LINEAR_PLAIN && a->kind != TAH_LINEAR_GATE_UP) return TAH_E_SHAPE;
    if (a->rows < 0 || a->rows > kLinRows || a->n < 0 || a->k < 0 || a->k % kStepK != 0) return TAH_E_SHAPE;
    const bool gate_up = a->kind == TAH_LINEAR_GATE_UP;
    const bool g24 = gate_up && a->n % kGroup24 == 0;
    if (!g24 && a->n % kTileCols != 0) return TAH_E_SHAPE;
    if (a->activation != TAH_ACT_NONE && a->activation != TAH_ACT_RELU && a->activation != TAH_ACT_GELU &&
        a->activation != TAH_ACT_GELU_TANH && a->activation != TAH_ACT_XIELU && a->activation != TAH_ACT_CLAMPED_GATE)
        return TAH_E_SHAPE;
    if (!gate_up && a->activation == TAH_ACT_CLAMPED_GATE) return TAH_E_SHAPE;
    if (a->input_norm != TAH_NORM_NONE && a->input_norm != TAH_NORM_RMS && a->input_norm != TAH_NORM_LAYER) return TAH_E_SHAPE;
    if (gate_up && (a->residual || a->bias || (a->activation != TAH_ACT_NONE && a->activation != TAH_ACT_CLAMPED_GATE) || a->input_norm == TAH_NORM_LAYER)) return TAH_E_SHAPE;
    if (a->input_norm == TAH_NORM_LAYER && !a->ln_colsum && a->n > 0 && a->k > 0) return TAH_E_NULL;
    const int batch = a->batch > 1 ? a->batch : 1;
    if (a->batch < 0 || a->batch > 65535 || a->n_select < 0) return TAH_E_SHAPE;
    if (batch > 1 && (a->residual || a->bias || a->input_norm != TAH_NORM_NONE)) return TAH_E_SHAPE;
    // the packed rows form holds whole steps of 32 columns: a result of its own, or all results side by side
    if (a->out_packed && (a->out_packed_col_step ? a->out_packed_col_step % 8 != 0 || a->out_packed_col_step < a->n : a->n % kStepK != 0))
        return TAH_E_SHAPE;
    if ((a->w_batch_stride | a->x_batch_stride | a->out_batch_stride | a->out_packed_batch_stride) % 8 != 0) return TAH_E_ALIGN;
    if (a->n == 0 || a->k == 0 || (a->rows == 0 && !a->out_packed)) return TAH_OK;
    if (!a->w_packed || !a->x_packed || (!a->out && !a->out_packed)) return TAH_E_NULL;
    if (!aligned16(a->w_packed) || !aligned16(a->x_packed) || !aligned16(a->out) || !aligned16(a->out_packed) || !aligned16(a->residual) ||
        !aligned16(a->bias) || (a->input_norm == TAH_NORM_LAYER && !aligned16(a->ln_colsum)) ||
        (a->out && a->out_row_stride % 8 != 0) || (a->residual && a->residual_row_stride % 8 != 0))
        return TAH_E_ALIGN;
    if ((a->out && a->out_row_stride < a->n) || (a->residual && a->residual_row_stride < a->n)) return TAH_E_SHAPE;
    LinParams p{};
    p.w = static_cast<const bf16x8*>(a->w_packed);
    p.x = static_cast<const bf16x8*>(a->x_packed);
    p.res = static_cast<const __bf16*>(a->residual);
    p.bias = static_cast<const __bf16*>(a->bias);
    p.act = a->activation;
    p.c0 = a->act_c[0]; p.c1 = a->act_c[1];
    p.colsum = a->input_norm == TAH_NORM_LAYER ? a->ln_colsum : nullptr;
    p.y = static_cast<__bf16*>(a->out);
    p.yp = static_cast<bf16x8*>(a->out_packed);
    p.res_rs = a->residual_row_stride;
    p.y_rs = a->out_row_stride;
    p.rows = a->rows;
    p.n = a->n;
    p.k = a->k;
    p.eps = a->norm_eps;
    p.norm = a->input_norm;
    p.w_bs = a->w_batch_stride; p.x_bs = a->x_batch_stride; p.y_bs = a->out_batch_stride; p.yp_bs = a->out_packed_batch_stride;
    p.yp_col_step = a->out_packed_col_step;
    p.select = a->n_select > 0 ? a->batch_select : nullptr;
    p.n_select = a->n_select;
    p.batches = batch;
    p.by_list = p.select && a->n_select < batch;
    p.grid_y = p.by_list ? a->n_select : batch;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int steps = a->k / kStepK;
    const int pw = steps % kLinWaves == 0 ? steps / kLinWaves : 0;  // compile-time K for the sizes of the end-to-end model
    if (!gate_up && a->input_norm != TAH_NORM_LAYER && a->n >= kWideFromCols && a->n % (2 * kTileCols) == 0) {
        // an output head: two tiles per workgroup, the rows' operand is read half as often
        int groups = a->n / (2 * kTileCols);
        if (beside) {
            p.w2 = static_cast<const bf16x8*>(beside->w_packed);
            p.bias2 = static_cast<const __bf16*>(beside->bias);
            p.y2 = static_cast<__bf16*>(beside->out);
            p.y2_rs = beside->out_row_stride;
            p.act2 = beside->activation;
            p.groups1 = groups;
            groups += beside->n / (2 * kTileCols);
        }
        if (pw == 8 && p.rows > 16 && batch == 1 && p.y && !p.yp && !p.res && !p.bias && p.act == TAH_ACT_NONE && !p.select) {
            if (p.norm) launch_wide<kPlainNorm, 8>(p, groups, st);
            else launch_wide<kPlain, 8>(p, groups, st);
        } else if (p.norm) {
            if (pw == 8) launch<2, 2, kPlainNorm, 8>(p, groups, batch, st);
            else launch<2, 2, kPlainNorm, 0>(p, groups, batch, st);
        } else {
            if (pw == 8) launch<2, 2, kPlain, 8>(p, groups, batch, st);
            else launch<2, 2, kPlain, 0>(p, groups, batch, st);
        }
    } else if (!gate_up && a->input_norm == TAH_NORM_LAYER) {
        launch<1, 4, kPlainLayerNorm, 0>(p, a->n / kTileCols, batch, st);
    } else if (!gate_up && batch > 1 && a->n % (2 * kTileCols) == 0 && a->n / (2 * kTileCols) * batch >= kSplitRowsBelowGroups) {
        // many products of one size: two tiles per workgroup halve the workgroups and the reads of the rows' operand
        const int groups = a->n / (2 * kTileCols);
        if (pw == 2) launch<2, 2, kPlain, 2>(p, groups, batch, st);
        else if (pw == 3) launch<2, 3, kPlain, 3>(p, groups, batch, st);
        else if (pw == 4) launch<2, 4, kPlain, 4>(p, groups, batch, st);
        else if (pw == 8) launch<2, 4, kPlain, 8>(p, groups, batch, st);
        else launch<2, 2, kPlain, 0>(p, groups, batch, st);
    } else if (!gate_up) {
        const int groups = a->n / kTileCols;
        if (p.norm) {
            if (pw == 8) launch<1, 8, kPlainNorm, 8>(p, groups, batch, st);
            else launch<1, 4, kPlainNorm, 0>(p, groups, batch, st);
        } else if (pw == 8) launch<1, 8, kPlain, 8>(p, groups, batch, st);
        else if (pw == 16) launch<1, 8, kPlain, 16>(p, groups, batch, st);
        else if (pw == 24) launch<1, 8, kPlain, 24>(p, groups, batch, st);
        else launch<1, 4, kPlain, 0>(p, groups, batch, st);
    } else if (g24) {
        const int groups = a->n / kGroup24;
        if (pw == 8) launch<3, 4, kGateUp24, 8>(p, groups, batch, st);
        else launch<3, 2, kGateUp24, 0>(p, groups, batch, st);
    } else {
        const int groups = a->n / kTileCols;
        if (pw == 8) launch<2, 4, kGateUp16, 8>(p, groups, batch, st);
        else launch<2, 2, kGateUp16, 0>(p, groups, batch, st);
    }
    return hipGetLastError() == hipSuccess ? TAH_OK : TAH_E_LAUNCH;
}

}  // namespace
}  // namespace tah

extern "C" int tah_linear_rows(const tah_linear_rows_args* a, tah_stream_t stream) {
    if (!a) return TAH_E_NULL;
    return tah::run_linear_rows(a, nullptr, stream);
}

// (More than sixteen rows: the resident workgroups of the head walk ranges of column groups, and with a second layer's among them 32
// prompts and 96 tokens took 79.6 instead of 77.4 ms.)
extern "C" int tah_linear_beside_supported(int32_t rows, int32_t n, int32_t k, int32_t beside) {
    using namespace tah;
    return rows >= 0 && rows <= 16 && n >= kWideFromCols && n % (2 * kTileCols) == 0 && k > 0 && k % kStepK == 0 && beside > 0 && beside % (2 * kTileCols) == 0;
}

extern "C" int tah_linear_beside(const tah_linear_rows_args* a, const tah_linear_rows_args* b, tah_stream_t stream) {
    using namespace tah;
    if (!a || !b) return TAH_E_NULL;
    if (!tah_linear_beside_supported(a->rows, a->n, a->k, b->n) || a->kind != TAH_LINEAR_PLAIN || a->batch > 1 || a->residual || a->bias || a->out_packed || a->n_select != 0 ||
        a->activation != TAH_ACT_NONE || a->input_norm != TAH_NORM_RMS)
        return TAH_E_SHAPE;
    if (b->kind != TAH_LINEAR_PLAIN || b->batch < 0 || b->batch > 1 || b->residual || b->out_packed || b->n_select != 0 ||
        (b->activation != TAH_ACT_NONE && b->activation != TAH_ACT_RELU) || b->input_norm != TAH_NORM_RMS || b->rows != a->rows || b->k != a->k ||
        b->norm_eps != a->norm_eps || b->out_row_stride < b->n)
        return TAH_E_SHAPE;
    if (a->rows == 0) return TAH_OK;
    if (!a->out || !a->x_packed || !a->w_packed || !b->w_packed || !b->out) return TAH_E_NULL;
    if (b->x_packed != a->x_packed) return TAH_E_SHAPE;
    // (in two calls a result that lies on another, or on what the second one reads, has an order)
    const auto result = [&](const tah_linear_rows_args* l) { return RowSpan{l->out, 2ll * l->n, 2 * l->out_row_stride, l->rows}; };
    const RowSpan written[] = {result(a), result(b)};
    const RowSpan read[] = {one_span(a->x_packed, 64ll * a->k), one_span(a->w_packed, 2ll * a->n * a->k), one_span(b->w_packed, 2ll * b->n * b->k),
                            one_span(b->bias, 2ll * b->n)};
    if (spans_meet(written[0], written[1])) return TAH_E_SHAPE;
    for (const RowSpan& w : written)
        for (const RowSpan& r : read)
            if (spans_meet(w, r)) return TAH_E_SHAPE;
    if (!aligned16(b->w_packed) || !aligned16(b->out) || !aligned16(b->bias) || b->out_row_stride % 8 != 0) return TAH_E_ALIGN;
    return run_linear_rows(a, b, stream);
}

extern "C" int tah_norm_linear_supported(int32_t rows, int32_t cols, int32_t n) {
    using namespace tah;
    return rows >= 1 && rows <= kNormLinearRows && cols == kNormLinearSteps * kLinWaves * kStepK && n > 0 && n % kTileCols == 0 &&
           n / kTileCols <= kNormLinearWorkgroups;
}

namespace tah {
namespace {
// What a plain layer's arguments say beside its sizes, as tah_norm_linear and the merge's projection take them.
int check_plain(const tah_linear_rows_args& a) {
    if (a.kind != TAH_LINEAR_PLAIN || a.batch > 1 || a.residual || a.bias || a.input_norm != TAH_NORM_NONE || a.n_select != 0 ||
        (a.activation != TAH_ACT_NONE && a.activation != TAH_ACT_GELU_TANH && a.activation != TAH_ACT_XIELU) || (a.out_packed && a.n % kStepK != 0) ||
        (a.out && a.out_row_stride < a.n))
        return TAH_E_SHAPE;
    if (!a.w_packed || (!a.out && !a.out_packed)) return TAH_E_NULL;
    if (!aligned16(a.w_packed) || !aligned16(a.out) || !aligned16(a.out_packed) || (a.out && a.out_row_stride % 8 != 0)) return TAH_E_ALIGN;
    return TAH_OK;
}
LinearOut linear_out(const tah_linear_rows_args& a) {
    return LinearOut{static_cast<__bf16*>(a.out), static_cast<bf16x8*>(a.out_packed), a.out_row_stride, a.activation, a.rows, a.act_c[0], a.act_c[1]};
}
}  // namespace

bool merge_linear_fits(int rows, int k, int n) { return tah_norm_linear_supported(rows, k, n) != 0; }

int merge_linear(const MergeLinear& p, const tah_linear_rows_args& a, hipStream_t st) {
    if (const int rc = check_plain(a)) return rc;
    if (!merge_linear_fits(a.rows, a.k, a.n) || a.k != p.heads * p.value_dim) return TAH_E_SHAPE;
    const bool h8 = a.n / kTileCols < kSplitRowsBelowGroups;  // (as tah_linear_rows takes such a layer)
    const auto launch = [&](auto fold, auto half) {
        hipLaunchKernelGGL((merge_linear_kernel<decltype(fold)::value, decltype(half)::value>), dim3(a.n / (h8 ? 8 : kTileCols)), dim3(kLinThreads), 0, st, p,
                           linear_out(a), static_cast<const bf16x8*>(a.w_packed));
    };
    const auto run = [&](auto fold) { h8 ? launch(fold, std::true_type{}) : launch(fold, std::false_type{}); };
    if (a.rows <= 1) run(std::integral_constant<int, 1>{});
    else run(std::integral_constant<int, 2>{});
    return hipGetLastError() == hipSuccess ? TAH_OK : TAH_E_LAUNCH;
}
}  // namespace tah

extern "C" int tah_norm_linear(const tah_residual_norm_args* norm, float* x_out, const tah_linear_rows_args* a, tah_stream_t stream) {
    using namespace tah;
    if (!norm || !a || !x_out) return TAH_E_NULL;
    if (const int rc = check_residual(*norm)) return rc;
    if (!tah_norm_linear_supported(norm->rows, norm->cols, a->n) || norm->dtype != TAH_DT_BF16 || a->rows != norm->rows || a->k != norm->cols) return TAH_E_SHAPE;
    // (what a workgroup of another tile still reads: nothing but x_out, the convolution's input and the layer's result is written)
    if (norm->xe || norm->x_packed || norm->normed || norm->normed_packed) return TAH_E_SHAPE;
    if (const int rc = check_plain(*a)) return rc;
    if (!aligned16(x_out)) return TAH_E_ALIGN;
    struct Range { const char* at; int64_t bytes; };
    const auto of = [](const void* q, int64_t bytes) { return Range{static_cast<const char*>(q), q ? bytes : 0}; };
    const int64_t last = norm->rows - 1;
    const Range written[] = {of(x_out, 4ll * norm->rows * norm->cols), of(a->out, 2 * (last * a->out_row_stride + a->n)), of(a->out_packed, 64ll * a->n)};
    // (how far the experts' rows reach only their indices say)
    const int64_t choices = norm->experts ? 4ll * norm->rows * norm->top : 0, per_row = norm->conv ? 4ll * norm->rows : 0;
    const int64_t taps = norm->conv ? (int64_t)norm->taps * norm->cols : 0;
    const Range read[] = {of(norm->x, 4ll * norm->rows * norm->cols), of(norm->y, 2 * (last * norm->y_row_stride + norm->cols)),
                          of(norm->coef, 4ll * norm->cols), of(norm->next_coef, 4ll * norm->cols), of(a->w_packed, 2ll * a->n * a->k),
                          of(norm->y_scale, 4ll * norm->rows), of(norm->index, choices), of(norm->weight, choices), of(norm->slot, per_row),
                          of(norm->pos, per_row), of(norm->conv, 4 * taps), of(norm->conv_state, 2 * taps * norm->nslots)};
    const auto meet = [](const Range& x, const Range& y) { return x.bytes > 0 && y.bytes > 0 && x.at < y.at + y.bytes && y.at < x.at + x.bytes; };
    for (const Range& w : written)
        for (const Range& r : read)
            if (meet(w, r)) return TAH_E_SHAPE;
    NormLinear p{};
    p.n = *norm;
    p.x_out = x_out;
    p.w = static_cast<const bf16x8*>(a->w_packed);
    p.out = linear_out(*a);
    const bool h8 = a->n / kTileCols < kSplitRowsBelowGroups;  // (as tah_linear_rows takes such a layer)
    const auto launch = [&](auto fold, auto groups, auto half, auto more) {
        hipLaunchKernelGGL((norm_linear_kernel<decltype(fold)::value, decltype(groups)::value, decltype(half)::value, decltype(more)::value>),
                           dim3(a->n / (h8 ? 8 : kTileCols)), dim3(kLinThreads), 0, static_cast<hipStream_t>(stream), p);
    };
    const auto run = [&](auto fold, auto groups, auto half) {
        norm->conv || norm->experts ? launch(fold, groups, half, std::true_type{}) : launch(fold, groups, half, std::false_type{});
    };
    const auto by_tile = [&](auto fold, auto groups) { h8 ? run(fold, groups, std::true_type{}) : run(fold, groups, std::false_type{}); };
    const auto by_groups = [&](auto fold) { norm->groups > 1 ? by_tile(fold, std::true_type{}) : by_tile(fold, std::false_type{}); };
    if (norm->rows <= 1) by_groups(std::integral_constant<int, 1>{});
    else by_groups(std::integral_constant<int, 2>{});
    return hipGetLastError() == hipSuccess ? TAH_OK : TAH_E_LAUNCH;
}

extern "C" int tah_linear_chain_supported(int32_t rows, int32_t hidden, int32_t o_cols, int32_t ff, int32_t qkv_cols) {
    using namespace tah;
    if (rows < 1 || rows > 8 || qkv_cols < 0 || qkv_cols % kTileCols != 0 || qkv_cols > kTileCols * kChainTiles) return 0;
#ifdef TAH_CPU_EMU
    if (hidden == 512 && o_cols == 512 && ff == 1536) return 1;  // (a size the execution on the CPU gets through)
#endif
    return hidden == 2048 && o_cols == 2048 && ff == 6144;
}

extern "C" int tah_linear_chain(const tah_linear_chain_args* a, tah_stream_t stream) {
    using namespace tah;
    if (!a) return TAH_E_NULL;
    if (a->rows == 0) {
        if (!a->clear) return TAH_OK;
        if (reinterpret_cast<uintptr_t>(a->clear) % sizeof(int32_t) != 0) return TAH_E_ALIGN;
        hipLaunchKernelGGL(linear_chain_clear_kernel, dim3(1), dim3(kLinThreads), 0, static_cast<hipStream_t>(stream), a->clear);
        return hipGetLastError() == hipSuccess ? TAH_OK : TAH_E_LAUNCH;
    }
    const bool next = a->wqkv_packed != nullptr;
    if (!tah_linear_chain_supported(a->rows, a->hidden, a->o_cols, a->ff, next ? a->qkv_cols : 0) || (next && a->qkv_cols == 0)) return TAH_E_SHAPE;
    const void* needed[] = {a->wo_packed, a->wgu_packed, a->wdown_packed, a->attn_packed, a->residual, a->mid, a->out, a->handover, a->arrived, a->clear, next ? a->qkv : a->out, next ? a->wqkv_packed : a->out};
    for (const void* q : needed) {
        if (!q) return TAH_E_NULL;
        if (!aligned16(q)) return TAH_E_ALIGN;
    }
    if (!aligned16(a->out_packed)) return TAH_E_ALIGN;
    if ((a->residual_row_stride | a->mid_row_stride | a->out_row_stride) % 8 != 0 || (next && a->qkv_row_stride % 8 != 0)) return TAH_E_ALIGN;
    if (a->residual_row_stride < a->hidden || a->mid_row_stride < a->hidden || a->out_row_stride < a->hidden || (next && a->qkv_row_stride < a->qkv_cols))
        return TAH_E_SHAPE;
    // what a phase writes may be written again while later phases run: no result may lie on an operand or on another result
    struct Range { const char* at; int64_t bytes; };
    const auto rows_of = [&](const void* q, int64_t stride, int64_t cols) { return Range{static_cast<const char*>(q), 2 * ((a->rows - 1) * stride + cols)}; };
    const int64_t word_bytes = (int64_t)TAH_LINEAR_CHAIN_WORDS * 4;
    const Range none{nullptr, 0};
    const Range written[] = {rows_of(a->mid, a->mid_row_stride, a->hidden), rows_of(a->out, a->out_row_stride, a->hidden),
                             {static_cast<const char*>(a->handover), (int64_t)TAH_LINEAR_CHAIN_HANDOVER_BYTES(a->hidden, a->ff)},
                             {reinterpret_cast<const char*>(a->arrived), word_bytes}, {reinterpret_cast<const char*>(a->clear), word_bytes},
                             a->out_packed ? Range{static_cast<const char*>(a->out_packed), 64 * (int64_t)a->hidden} : none,
                             next ? rows_of(a->qkv, a->qkv_row_stride, a->qkv_cols) : none};
    const auto weight_of = [](const void* w, int64_t n, int64_t k) { return Range{static_cast<const char*>(w), 2 * n * k}; };
    const Range read[] = {rows_of(a->residual, a->residual_row_stride, a->hidden), {static_cast<const char*>(a->attn_packed), 64 * (int64_t)a->o_cols},
                          weight_of(a->wo_packed, a->hidden, a->o_cols), weight_of(a->wgu_packed, 2 * (int64_t)a->ff, a->hidden),
                          weight_of(a->wdown_packed, a->hidden, a->ff), next ? weight_of(a->wqkv_packed, a->qkv_cols, a->hidden) : none};
    const auto meet = [](const Range& x, const Range& y) { return x.bytes > 0 && y.bytes > 0 && x.at < y.at + y.bytes && y.at < x.at + x.bytes; };
    for (int i = 0; i < 7; ++i) {
        for (int j = i + 1; j < 7; ++j)
            if (meet(written[i], written[j])) return TAH_E_SHAPE;
        for (const Range& q : read)
            if (meet(written[i], q)) return TAH_E_SHAPE;
    }
    ChainParams p{};
    p.w0 = static_cast<const bf16x8*>(a->wo_packed);
    p.w1 = static_cast<const bf16x8*>(a->wgu_packed);
    p.w2 = static_cast<const bf16x8*>(a->wdown_packed);
    p.w3 = static_cast<const bf16x8*>(a->wqkv_packed);
    p.x0 = static_cast<const bf16x8*>(a->attn_packed);
    p.x1 = static_cast<unsigned long long*>(a->handover);
    p.x2 = p.x1 + 2 * (int64_t)a->hidden;  // (eight rows' 8-byte words of each)
    p.x3 = p.x2 + 2 * (int64_t)a->ff;
    p.out_packed = static_cast<bf16x8*>(a->out_packed);
    p.res = static_cast<const __bf16*>(a->residual);
    p.mid = static_cast<__bf16*>(a->mid);
    p.out = static_cast<__bf16*>(a->out);
    p.y = static_cast<__bf16*>(a->qkv);
    p.res_rs = a->residual_row_stride;
    p.mid_rs = a->mid_row_stride;
    p.out_rs = a->out_row_stride;
    p.y_rs = a->qkv_row_stride;
    p.arrived = reinterpret_cast<uint32_t*>(a->arrived);
    p.clear = a->clear;
    p.rows = a->rows;
    p.tiles0 = p.tiles2 = a->hidden / 8;
    p.tiles1 = a->ff / kGroup24;
    p.tiles3 = next ? a->qkv_cols / kTileCols : 0;
    p.polls = a->polls > 0 ? a->polls : kChainPolls;
    p.eps = a->norm_eps;
    const int form = !next ? kNextNone : p.tiles3 < kSplitRowsBelowGroups ? kNextApart : kNextWhole;
    hipStream_t st = static_cast<hipStream_t>(stream);
#ifdef TAH_CPU_EMU
    if (a->hidden == 512) {
        launch_chain<2, 2, 6>(p, form, st);
        return TAH_OK;
    }
#endif
    launch_chain<8, 8, 24>(p, form, st);
    return hipGetLastError() == hipSuccess ? TAH_OK : TAH_E_LAUNCH;
}
