// Hard-token index build and row gather/scatter (integer / byte work, exact).
//
// The index build is a single-workgroup stream compaction: 1024 threads, each
// owning 16 consecutive mask bytes per pass, a wave-shuffle + LDS block scan per
// pass, and a running carry.  Row-major order of the True entries is the packing
// order the model's forward loop uses for iteration-2 rows.
#include <hip/hip_runtime.h>

#include "duo_device.h"
#include "tah_duo.h"

namespace tah {
namespace {

constexpr int kScanThreads = 1024;
constexpr int kPerThread = 16;

__global__ __launch_bounds__(kScanThreads) void hard_index_kernel(const uint8_t* mask, int B, int S, int32_t* pos_out,
                                                                  int32_t* flat_out, int32_t* seq_out, int32_t* cu_out,
                                                                  int32_t* rank_out, int32_t* spans_out) {
    __shared__ int wave_tot[kScanThreads / kWave];
    __shared__ int carry_s;
    const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    const int64_t total = (int64_t)B * S;
    if (tid == 0) carry_s = 0;
    // a mask without columns has no element (b, 0) to carry a row's boundary: every boundary is 0
    if (S == 0)
        for (int b = tid; b < B; b += kScanThreads) cu_out[b] = 0;
    __syncthreads();
    for (int64_t chunk = 0; chunk < total; chunk += (int64_t)kScanThreads * kPerThread) {
        const int64_t f0 = chunk + (int64_t)tid * kPerThread;
        uint8_t m[kPerThread];
        int cnt = 0;
#pragma unroll
        for (int i = 0; i < kPerThread; ++i) {
            m[i] = (f0 + i < total) ? mask[f0 + i] : 0;
            cnt += m[i] != 0;
        }
        // inclusive scan of cnt across the wave, then across waves
        int inc = cnt;
#pragma unroll
        for (int d = 1; d < kWave; d <<= 1) {
            const int y = __shfl_up(inc, d);
            if (lane >= d) inc += y;
        }
        if (lane == kWave - 1) wave_tot[wave] = inc;
        __syncthreads();
        int wave_off = 0;
        for (int w = 0; w < wave; ++w) wave_off += wave_tot[w];
        int chunk_total = 0;
        for (int w = 0; w < kScanThreads / kWave; ++w) chunk_total += wave_tot[w];
        const int carry = carry_s;
        int run = carry + wave_off + inc - cnt;  // True entries before flat index f0
#pragma unroll
        for (int i = 0; i < kPerThread; ++i) {
            const int64_t f = f0 + i;
            if (f < total) {
                const int b = (int)(f / S), s = (int)(f - (int64_t)b * S);
                if (s == 0) cu_out[b] = run;
                if (rank_out) rank_out[f] = m[i] ? run : -1;
                if (m[i]) {
                    if (pos_out) pos_out[run] = s;
                    if (flat_out) flat_out[run] = (int32_t)f;
                    if (seq_out) seq_out[run] = b;
                    ++run;
                }
            }
        }
        __syncthreads();
        if (tid == 0) carry_s = carry + chunk_total;
        __syncthreads();
    }
    if (tid == 0) cu_out[B] = carry_s;
    if (!spans_out) return;  // (uniform)
    // every row as (flat index of its first True entry, that plus their number), then whether some row's do not lie together
    __shared__ int broken;
    if (tid == 0) broken = 0;
    __syncthreads();  // (and the boundaries and indices written above are there)
    for (int b = tid; b < B; b += kScanThreads) {
        const int lo = cu_out[b], n = cu_out[b + 1] - lo;
        const int first = n > 0 ? flat_out[lo] : b * S, last = n > 0 ? flat_out[lo + n - 1] : first - 1;
        spans_out[2 * b] = first;
        spans_out[2 * b + 1] = first + n;
        if (last - first + 1 != n) broken = 1;
    }
    __syncthreads();
    if (tid == 0) spans_out[2 * B] = broken;
}

// The right-padded (B, width) form of a mask's entries as tables: left[b * width + j] = flat index of row b's j-th entry, back[f] = place of
// entry f in that form, both -1 where there is none, and the form's padding.
__global__ __launch_bounds__(256) void left_index_kernel(const int32_t* cu, const int32_t* flat, const int32_t* rank, int B, int S, int width,
                                                         int32_t* left, int32_t* back, uint8_t* pad) {
    const int64_t at0 = (int64_t)blockIdx.x * 256 + threadIdx.x;  // (the last workgroup's may lie past 2^31)
    if (at0 >= (int64_t)B * (S > width ? S : width)) return;
    const int i = (int)at0;
    if (i < B * width) {
        const int b = i / width, at = cu[b] + i % width;
        const bool there = at < cu[b + 1];
        left[i] = there ? flat[at] : -1;
        pad[i] = there ? 0 : 1;
    }
    if (i < B * S) {
        const int r = rank[i], b = i / S;
        back[i] = r >= 0 && r - cu[b] < width ? b * width + r - cu[b] : -1;
    }
}

__global__ void pad_rows_kernel(const int32_t* cu, const int32_t* seq_of, int n, const int32_t* n_dev, int width,
                                int32_t* out, int32_t* overflow) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (n_dev && *n_dev < n) n = *n_dev;
    if (r < n) {
        const int b = seq_of[r];
        const int rank = r - cu[b];
        out[r] = rank < width ? b * width + rank : -1;  // an entry that does not fit its row is dropped by the copy
        if (rank >= width && overflow) *overflow = 1;
    }
}

template <typename V>
__global__ void rows_copy_kernel(const unsigned char* src, const int32_t* src_rows, unsigned char* dst,
                                 const int32_t* dst_rows, const uint8_t* dst_enable, int n, const int32_t* n_dev,
                                 int vec_per_row, int64_t src_stride, int64_t dst_stride, int row_base) {
    const int r = blockIdx.y;
    if (r >= n || (n_dev && row_base + r >= *n_dev)) return;
    const int64_t sr = src_rows ? src_rows[r] : row_base + r;
    const int64_t dr = dst_rows ? dst_rows[r] : row_base + r;
    if (sr < 0 || dr < 0) return;  // dropped entry (see pad_rows_kernel)
    if (dst_enable && !dst_enable[dr]) return;
    const V* s = reinterpret_cast<const V*>(src + sr * src_stride);
    V* d = reinterpret_cast<V*>(dst + dr * dst_stride);
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < vec_per_row; i += gridDim.x * blockDim.x) d[i] = s[i];
}

struct alignas(16) V16 { uint32_t x[4]; };
typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4;

// Rows of up to TAH_SELECT_TENSORS tensors by one table: row r of a result is row index[r] of its source, zeros where that is negative.
// What bounds it is the launch for a step's packed rows (three tensors of 1284 rows of 4, 2 and 2 KB: 6.6 us) and memory beyond; as clears and copies of
// every tensor by itself, three tensors were six launches, and the host's time for them stood between a model's two iterations.
struct SelectRows {
    tah_select_rows t[TAH_SELECT_TENSORS];
    int32_t unit[TAH_SELECT_TENSORS];  // bytes moved at a time
};
template <typename V>
__device__ __forceinline__ void select_rows(const tah_select_rows& t, const int32_t* index, int rows) {
    const int per_row = (int)(t.row_bytes / (int64_t)sizeof(V));
    const unsigned char* const src = static_cast<const unsigned char*>(t.src);
    unsigned char* const dst = static_cast<unsigned char*>(t.dst);
    if (per_row < kWave / 2) {  // short rows: as many as fit to a wave
        const int in_wave = kWave / per_row, lane = threadIdx.x % kWave, mine = lane / per_row, c = lane - mine * per_row;
        for (int64_t r0 = ((int64_t)blockIdx.x * 4 + threadIdx.x / kWave) * in_wave; r0 < rows; r0 += (int64_t)gridDim.x * 4 * in_wave) {
            const int64_t r = r0 + mine;
            if (mine >= in_wave || r >= rows) continue;
            const int from = index[r];
            V v = {};
            if (from >= 0) v = reinterpret_cast<const V*>(src + from * t.src_stride_bytes)[c];
            reinterpret_cast<V*>(dst + r * t.row_bytes)[c] = v;
        }
        return;
    }
    for (int64_t r = (int64_t)blockIdx.x * 4 + threadIdx.x / kWave; r < rows; r += (int64_t)gridDim.x * 4) {  // a wave to a row
        const int from = index[r];
        const V* const s = reinterpret_cast<const V*>(src + from * t.src_stride_bytes);
        V* const d = reinterpret_cast<V*>(dst + r * t.row_bytes);
        for (int c = threadIdx.x % kWave; c < per_row; c += 4 * kWave) {
            V v[4] = {};
            if (from >= 0) {  // (the same for the whole wave; its loads are on their way together)
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = s[c + i * kWave < per_row ? c + i * kWave : c];
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (c + i * kWave < per_row) d[c + i * kWave] = v[i];
        }
    }
}
__global__ __launch_bounds__(256) void select_rows_kernel(const SelectRows p, const int32_t* index, int rows, const int32_t* n_dev) {
    if (n_dev && *n_dev < rows) rows = *n_dev;
    const tah_select_rows t = p.t[blockIdx.y];
    switch (p.unit[blockIdx.y]) {  // (uniform)
        case 16: select_rows<u32x4>(t, index, rows); break;
        case 8: select_rows<uint64_t>(t, index, rows); break;
        case 4: select_rows<uint32_t>(t, index, rows); break;
        case 2: select_rows<uint16_t>(t, index, rows); break;
        default: select_rows<uint8_t>(t, index, rows); break;
    }
}

// Rows that belong to no sequence, set to zero: one launch for all tensors of a call.  Memory-bound, and only those rows are written (a
// clear of the whole result in front of the kernel that fills it writes the others twice).
struct GapRows {
    tah_gap_rows t[TAH_GAP_TENSORS];
};
__global__ __launch_bounds__(256) void zero_gaps_kernel(const GapRows p, int nseq) {
    const tah_gap_rows t = p.t[blockIdx.z];
    for (int g = blockIdx.y; g <= nseq; g += gridDim.y) {  // the rows between sequence g - 1 and sequence g
        const int64_t lo = g > 0 ? t.pairs[2 * g - 1] : 0, hi = g < nseq ? t.pairs[2 * g] : t.total;
        u32x4* const rows = static_cast<u32x4*>(t.rows);
        const int64_t end = (hi < t.total ? hi : t.total) * (t.row_bytes / 16);
        for (int64_t i = (lo > 0 ? lo : 0) * (t.row_bytes / 16) + (int64_t)blockIdx.x * 256 + threadIdx.x; i < end; i += (int64_t)gridDim.x * 256)
            rows[i] = u32x4{0u, 0u, 0u, 0u};
    }
}

template <typename V>
int launch_copy(const void* src, const int32_t* src_rows, void* dst, const int32_t* dst_rows, const uint8_t* dst_enable, int n,
                const int32_t* n_dev, int64_t row_bytes, int64_t src_stride, int64_t dst_stride, hipStream_t st) {
    const int vec = (int)(row_bytes / (int64_t)sizeof(V));
    int gx = (vec + 255) / 256;
    gx = gx < 1 ? 1 : (gx > 64 ? 64 : gx);
    for (int r0 = 0; r0 < n; r0 += 65535) {  // grid.y limit
        const int nr = n - r0 < 65535 ? n - r0 : 65535;
        hipLaunchKernelGGL(rows_copy_kernel<V>, dim3(gx, nr), dim3(256), 0, st, static_cast<const unsigned char*>(src),
                           src_rows ? src_rows + r0 : nullptr, static_cast<unsigned char*>(dst),
                           dst_rows ? dst_rows + r0 : nullptr, dst_enable, nr, n_dev, vec, src_stride, dst_stride, r0);
    }
    return hipGetLastError() == hipSuccess ? TAH_OK : TAH_E_LAUNCH;
}

}  // namespace
}  // namespace tah

extern "C" int tah_hard_index_build(const uint8_t* mask, int32_t B, int32_t S, int32_t* pos_out, int32_t* flat_out,
                                    int32_t* seq_out, int32_t* cu_out, tah_stream_t stream) {
    using namespace tah;
    if (B < 0 || S < 0) return TAH_E_SHAPE;
    if (!cu_out || (!mask && (int64_t)B * S > 0)) return TAH_E_NULL;
    if ((int64_t)B * S >= (int64_t)1 << 31) return TAH_E_SHAPE;
    hipLaunchKernelGGL(hard_index_kernel, dim3(1), dim3(kScanThreads), 0, static_cast<hipStream_t>(stream), mask, B, S,
                       pos_out, flat_out, seq_out, cu_out, nullptr, nullptr);
    return hipGetLastError() == hipSuccess ? TAH_OK : TAH_E_LAUNCH;
}

extern "C" int tah_mask_index_build(const tah_mask_index_args* a, tah_stream_t stream) {
    using namespace tah;
    if (!a) return TAH_E_NULL;
    if (a->B < 0 || a->S < 0 || (int64_t)a->B * a->S >= (int64_t)1 << 31) return TAH_E_SHAPE;
    if (!a->cu || ((int64_t)a->B * a->S > 0 && (!a->mask || (a->spans && !a->flat)))) return TAH_E_NULL;
    hipLaunchKernelGGL(hard_index_kernel, dim3(1), dim3(kScanThreads), 0, static_cast<hipStream_t>(stream), a->mask, a->B, a->S, a->pos, a->flat,
                       a->seq, a->cu, a->rank, a->spans);
    return hipGetLastError() == hipSuccess ? TAH_OK : TAH_E_LAUNCH;
}

extern "C" int tah_left_index_build(const int32_t* cu, const int32_t* flat, const int32_t* rank, int32_t B, int32_t S, int32_t width,
                                    int32_t* left, int32_t* back, uint8_t* pad, tah_stream_t stream) {
    using namespace tah;
    if (B < 0 || S < 0 || width < 0 || (int64_t)B * S >= (int64_t)1 << 31 || (int64_t)B * width >= (int64_t)1 << 31) return TAH_E_SHAPE;
    const int n = B * (S > width ? S : width);
    if (n == 0) return TAH_OK;
    if (!cu || (B * S > 0 && (!flat || !rank || !back)) || (B * width > 0 && (!left || !pad))) return TAH_E_NULL;
    hipLaunchKernelGGL(left_index_kernel, dim3((unsigned)(((int64_t)n + 255) / 256)), dim3(256), 0, static_cast<hipStream_t>(stream), cu, flat, rank, B, S, width, left,
                       back, pad);
    return hipGetLastError() == hipSuccess ? TAH_OK : TAH_E_LAUNCH;
}

extern "C" int tah_rows_select(const tah_select_rows* tensors, int32_t n, const int32_t* index, int32_t rows, const int32_t* n_dev,
                               tah_stream_t stream) {
    using namespace tah;
    if (n < 0 || n > TAH_SELECT_TENSORS || rows < 0) return TAH_E_SHAPE;
    if (n == 0 || rows == 0) return TAH_OK;
    if (!tensors || !index) return TAH_E_NULL;
    SelectRows p{};
    int used = 0;
    int64_t most = 0;
    for (int i = 0; i < n; ++i) {
        const tah_select_rows& t = tensors[i];
        if (t.row_bytes < 0) return TAH_E_SHAPE;
        if (t.row_bytes == 0) continue;
        if (!t.dst) return TAH_E_NULL;
        // (a source without rows may come without a pointer: nothing points into it)
        const uintptr_t all = reinterpret_cast<uintptr_t>(t.src) | reinterpret_cast<uintptr_t>(t.dst) | (uintptr_t)t.row_bytes | (uintptr_t)t.src_stride_bytes;
        const int unit = all % 16 == 0 ? 16 : all % 8 == 0 ? 8 : all % 4 == 0 ? 4 : all % 2 == 0 ? 2 : 1;
        if (t.row_bytes / unit >= (int64_t)1 << 31) return TAH_E_SHAPE;
        p.t[used] = t;
        p.unit[used++] = unit;
        const int64_t per_row = t.row_bytes / unit, waves = per_row < 32 ? (rows + 64 / per_row - 1) / (64 / per_row) : rows;
        most = waves > most ? waves : most;
    }
    if (used == 0) return TAH_OK;
    const int64_t blocks = (most + 3) / 4;
    hipLaunchKernelGGL(select_rows_kernel, dim3((unsigned)(blocks < 8192 ? blocks : 8192), used), dim3(256), 0, static_cast<hipStream_t>(stream), p,
                       index, rows, n_dev);
    return hipGetLastError() == hipSuccess ? TAH_OK : TAH_E_LAUNCH;
}

extern "C" int tah_pad_rows_build(const int32_t* cu, const int32_t* seq_of, int32_t n, const int32_t* n_dev, int32_t width,
                                  int32_t* out, int32_t* overflow, tah_stream_t stream) {
    using namespace tah;
    if (n < 0 || width < 0) return TAH_E_SHAPE;
    if (n == 0) return TAH_OK;
    if (!cu || !seq_of || !out) return TAH_E_NULL;
    hipLaunchKernelGGL(pad_rows_kernel, dim3((n + 255) / 256), dim3(256), 0, static_cast<hipStream_t>(stream), cu, seq_of, n,
                       n_dev, width, out, overflow);
    return hipGetLastError() == hipSuccess ? TAH_OK : TAH_E_LAUNCH;
}

extern "C" int tah_rows_copy(const void* src, const int32_t* src_rows, void* dst, const int32_t* dst_rows,
                             const uint8_t* dst_enable, int32_t n, const int32_t* n_dev, int64_t row_bytes,
                             int64_t src_stride_bytes, int64_t dst_stride_bytes, tah_stream_t stream) {
    using namespace tah;
    if (n < 0 || row_bytes < 0) return TAH_E_SHAPE;
    if (n == 0 || row_bytes == 0) return TAH_OK;
    if (!src || !dst) return TAH_E_NULL;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const uintptr_t bits = reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst) | (uintptr_t)row_bytes |
                           (uintptr_t)src_stride_bytes | (uintptr_t)dst_stride_bytes;
    if (bits % 16 == 0) return launch_copy<V16>(src, src_rows, dst, dst_rows, dst_enable, n, n_dev, row_bytes, src_stride_bytes, dst_stride_bytes, st);
    if (bits % 8 == 0) return launch_copy<uint64_t>(src, src_rows, dst, dst_rows, dst_enable, n, n_dev, row_bytes, src_stride_bytes, dst_stride_bytes, st);
    if (bits % 4 == 0) return launch_copy<uint32_t>(src, src_rows, dst, dst_rows, dst_enable, n, n_dev, row_bytes, src_stride_bytes, dst_stride_bytes, st);
    if (bits % 2 == 0) return launch_copy<uint16_t>(src, src_rows, dst, dst_rows, dst_enable, n, n_dev, row_bytes, src_stride_bytes, dst_stride_bytes, st);
    return launch_copy<uint8_t>(src, src_rows, dst, dst_rows, dst_enable, n, n_dev, row_bytes, src_stride_bytes, dst_stride_bytes, st);
}

extern "C" int tah_zero_gaps(const tah_gap_rows* tensors, int32_t n, int32_t nseq, tah_stream_t stream) {
    using namespace tah;
    if (n < 0 || n > TAH_GAP_TENSORS || nseq < 0) return TAH_E_SHAPE;
    if (n == 0) return TAH_OK;
    if (!tensors) return TAH_E_NULL;
    GapRows p{};
    int used = 0;
    for (int i = 0; i < n; ++i) {
        const tah_gap_rows& t = tensors[i];
        if (t.total < 0 || t.row_bytes < 0) return TAH_E_SHAPE;
        if (t.total == 0 || t.row_bytes == 0) continue;
        if (!t.rows || (nseq > 0 && !t.pairs)) return TAH_E_NULL;
        if ((reinterpret_cast<uintptr_t>(t.rows) & 15) || t.row_bytes % 16) return TAH_E_ALIGN;
        p.t[used++] = t;
    }
    if (used == 0) return TAH_OK;
    hipLaunchKernelGGL(zero_gaps_kernel, dim3(64, nseq < 1023 ? nseq + 1 : 1024, used), dim3(256), 0, static_cast<hipStream_t>(stream), p, nseq);
    return hipGetLastError() == hipSuccess ? TAH_OK : TAH_E_LAUNCH;
}
