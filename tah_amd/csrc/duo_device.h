// Device-side helpers shared by the duo-causal attention kernels (gfx950, wave64).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace tah {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

// LDS addressed through pointers that carry the LDS address space and start at LDS address 0.  A kernel that
// declares no static LDS object has its dynamic LDS at address 0; a pointer made from that integer (instead of
// the extern array's symbol, whose zero the compiler only learns after instruction selection) lets constant
// parts of an offset fold into the instructions' immediate fields -- no `v_add_u32 v, 0, v` per access -- and
// needs no generic-to-LDS conversion (a compare and a select each) where an address goes into m0.
#ifdef TAH_CPU_EMU
typedef unsigned char lds_byte;
typedef float lds_float;
typedef int lds_int;
#define TAH_LDS_ZERO_BASED(name, decl) unsigned char* const name = decl
#define TAH_LDS_CAST(T, p) (reinterpret_cast<T*>(p))
#else
typedef __attribute__((address_space(3))) unsigned char lds_byte;
typedef __attribute__((address_space(3))) float lds_float;
typedef __attribute__((address_space(3))) int lds_int;
#define TAH_LDS_ZERO_BASED(name, decl) \
    tah::lds_byte* const name = reinterpret_cast<tah::lds_byte*>(static_cast<uintptr_t>(0)); (void)decl
#define TAH_LDS_CAST(T, p) (reinterpret_cast<__attribute__((address_space(3))) T*>(p))
#endif

// Words that workgroups on different XCDs hand to each other inside one launch: device-scope relaxed atomics, which pass by
// the caches that are not shared.  Order between them is the caller's (device_settle between a store and what announces it).
#ifdef TAH_CPU_EMU
template <class T> inline void device_store(T* p, T v) { __atomic_store(p, &v, __ATOMIC_SEQ_CST); }
template <class T> inline T device_load(const T* p) { T v; __atomic_load(const_cast<T*>(p), &v, __ATOMIC_SEQ_CST); return v; }
inline int device_add(int32_t* p, int v) { return __atomic_fetch_add(p, v, __ATOMIC_SEQ_CST); }
inline void device_or(uint32_t* p, uint32_t v) {  // (one thread of a block calls it)
    __atomic_fetch_or(p, v, __ATOMIC_SEQ_CST);
    emu::g_ors.push_back(p);
}
inline void device_max(unsigned long long* p, unsigned long long v) {
    for (unsigned long long now = device_load(p); now < v && !__atomic_compare_exchange_n(p, &now, v, false, __ATOMIC_SEQ_CST, __ATOMIC_SEQ_CST);) {}
}
#else
template <class T> __device__ __forceinline__ void device_store(T* p, T v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
template <class T> __device__ __forceinline__ T device_load(const T* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ int device_add(int32_t* p, int v) { return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ void device_or(uint32_t* p, uint32_t v) { __hip_atomic_fetch_or(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ void device_max(unsigned long long* p, unsigned long long v) { __hip_atomic_fetch_max(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
#endif

// Memory that a call's rows take up, on the host: `rows` rows of `bytes`, `stride` bytes apart (nothing where `at` is null).
struct RowSpan {
    const void* at;
    int64_t bytes, stride;
    int32_t rows;
};
inline RowSpan one_span(const void* at, int64_t bytes) { return RowSpan{at, bytes, bytes, 1}; }
// Whether two of them share a byte (columns of one array side by side do not; otherwise a gap between rows counts as taken).
inline bool spans_meet(const RowSpan& x, const RowSpan& y) {
    if (!x.at || !y.at || x.bytes <= 0 || y.bytes <= 0 || x.rows <= 0 || y.rows <= 0) return false;
    const int64_t from = reinterpret_cast<intptr_t>(x.at), other = reinterpret_cast<intptr_t>(y.at);
    if (other >= from + (x.rows - 1) * x.stride + x.bytes || from >= other + (y.rows - 1) * y.stride + y.bytes) return false;
    if (x.rows > 1 && y.rows > 1 && x.stride == y.stride && x.stride >= x.bytes && x.stride >= y.bytes) {
        const int64_t d = ((other - from) % x.stride + x.stride) % x.stride;
        return d < x.bytes || x.stride - d < y.bytes;
    }
    return true;
}

#ifndef TAH_WAIT_VMEM
// s_waitcnt vmcnt(0) (expcnt/lgkmcnt untouched) as a builtin, so the compiler's own wait-count
// bookkeeping also learns that no ordinary load is pending past this point.
#define TAH_WAIT_VMEM() __builtin_amdgcn_s_waitcnt(0x0F70)
#endif
#ifdef TAH_CPU_EMU
#define TAH_WAIT_LDS() ((void)0)
#define TAH_SLEEP(n) ((void)0)
#define TAH_OPAQUE_S(p) ((void)0)
#define TAH_APART() ((void)0)
#define TAH_GLOBAL
#else
#define TAH_WAIT_LDS() __builtin_amdgcn_s_waitcnt(0xC07F)  // s_waitcnt lgkmcnt(0), loads from memory stay on their way
#define TAH_SLEEP(n) __builtin_amdgcn_s_sleep(n)
#define TAH_APART() asm volatile("; apart")  // no instruction: keeps what stands in one branch from being merged with its like in the other
#define TAH_OPAQUE_S(p) asm volatile("" : "+s"(p))  // a value that stays in scalar registers, apart from those it was made of
#define TAH_GLOBAL __attribute__((address_space(1)))
#endif
// What this thread has stored or added for other workgroups is there.  The wait alone says nothing to the compiler about memory:
// the fences, which cost no instruction, keep what stands before it before it and what stands behind it behind it.
__device__ __forceinline__ void device_settle() {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    TAH_WAIT_VMEM();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

constexpr int kWave = 64;
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;
constexpr float kNegInf = -__builtin_inff();

// v_mfma_f32_32x32x16_bf16: D(32x32) += A(32x16) * B(16x32).
// lane l: A[i = l%32][k = 8*(l/32) + 0..7], B[k = 8*(l/32) + 0..7][j = l%32],
// D reg r: [i = 8*(r/4) + 4*(l/32) + r%4][j = l%32].
__device__ __forceinline__ f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// Row index inside a 32-row MFMA accumulator tile held by (lane half h, reg r).
__device__ __forceinline__ constexpr int acc_row(int h, int r) { return 8 * (r / 4) + 4 * h + (r % 4); }

// x *= a with the product forced into x's own register, so that an accumulator rescaled inside a
// rarely taken branch is not copied to a second register set on the common path.
#ifndef TAH_MUL_INPLACE
#define TAH_MUL_INPLACE(x, a) asm volatile("v_mul_f32 %0, %1, %0" : "+v"(x) : "v"(a))
#endif

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float fast_log2(float x) { return __builtin_amdgcn_logf(x); }
__device__ __forceinline__ float fast_rcp(float x) { return __builtin_amdgcn_rcpf(x); }

__device__ __forceinline__ bf16x8 ld_global_16B(const __bf16* p) { return *reinterpret_cast<const bf16x8*>(p); }
__device__ __forceinline__ void st_global_16B(__bf16* p, bf16x8 v) { *reinterpret_cast<bf16x8*>(p) = v; }

// Asynchronous global -> LDS copy of 16 bytes per lane (global_load_lds_dwordx4): lane l's bytes
// land at lds_wave_base + 16*l; lds_wave_base must be wave-uniform.  Issued through inline
// assembly on purpose: the compiler then does not order later LDS reads of *other* tiles behind
// this copy (it cannot prove they do not alias and would wait for vmcnt(0) in the middle of the
// compute phase).  Completion is tracked by vmcnt: TAH_WAIT_VMEM() before the barrier that
// publishes the tile.
#ifndef TAH_ASYNC_COPY_16B
#define TAH_ASYNC_COPY_16B(gsrc, lds_wave_base)                                                                    \
    do {                                                                                                           \
        const unsigned tah_m0_ = __builtin_amdgcn_readfirstlane(                                                   \
            (unsigned)(uintptr_t)(__attribute__((address_space(3))) void*)(lds_wave_base));                        \
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"                             \
                     :                                                                                             \
                     : "s"(tah_m0_), "v"(gsrc)                                                                     \
                     : "memory");  /* m0 is reserved: the compiler reloads it before each own use */                                                                            \
    } while (0)
#endif
__device__ __forceinline__ void async_copy_16B(const void* gsrc, unsigned char* lds_wave_base) {
    TAH_ASYNC_COPY_16B(gsrc, lds_wave_base);
}
// Same copy addressed as wave-uniform base + per-lane 32-bit byte offset: the base lives in scalar
// registers and advances with scalar arithmetic, the lane offsets can be loop invariant.
#ifndef TAH_ASYNC_COPY_16B_SO
#define TAH_ASYNC_COPY_16B_SO(sbase, voff, lds_wave_base)                                                          \
    do {                                                                                                           \
        const unsigned tah_m0_ = __builtin_amdgcn_readfirstlane(                                                   \
            (unsigned)(uintptr_t)(__attribute__((address_space(3))) void*)(lds_wave_base));                        \
        const uint64_t tah_b_ = (uint64_t)(uintptr_t)(sbase);                                                      \
        /* the builtin returns int: narrow to 32 bits unsigned before widening, or bit 31 smears upward */      \
        const uint64_t tah_sb_ = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((unsigned)tah_b_) |            \
                                 ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((unsigned)(tah_b_ >> 32)) << 32); \
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"                              \
                     :                                                                                             \
                     : "s"(tah_m0_), "v"(voff), "s"(tah_sb_)                                                       \
                     : "memory");                                                                                  \
    } while (0)
#endif
__device__ __forceinline__ void async_copy_16B(const void* sbase, uint32_t voff, unsigned char* lds_wave_base) {
    TAH_ASYNC_COPY_16B_SO(sbase, voff, lds_wave_base);
}
// The same copy for data that is read once (streaming: the lines are not kept in the L2).
#ifndef TAH_ASYNC_COPY_16B_SO_NT
#define TAH_ASYNC_COPY_16B_SO_NT(sbase, voff, lds_wave_base)                                                       \
    do {                                                                                                           \
        const unsigned tah_m0_ = __builtin_amdgcn_readfirstlane(                                                   \
            (unsigned)(uintptr_t)(__attribute__((address_space(3))) void*)(lds_wave_base));                        \
        const uint64_t tah_b_ = (uint64_t)(uintptr_t)(sbase);                                                      \
        const uint64_t tah_sb_ = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((unsigned)tah_b_) |            \
                                 ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((unsigned)(tah_b_ >> 32)) << 32); \
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt"                           \
                     :                                                                                             \
                     : "s"(tah_m0_), "v"(voff), "s"(tah_sb_)                                                       \
                     : "memory");                                                                                  \
    } while (0)
#endif
__device__ __forceinline__ void async_copy_16B_stream(const void* sbase, uint32_t voff, unsigned char* lds_wave_base) {
    TAH_ASYNC_COPY_16B_SO_NT(sbase, voff, lds_wave_base);
}
#ifndef TAH_CPU_EMU
__device__ __forceinline__ void async_copy_16B_stream(const void* sbase, uint32_t voff, lds_byte* lds_wave_base) {
    TAH_ASYNC_COPY_16B_SO_NT(sbase, voff, lds_wave_base);
}
#endif
// Same with 4 bytes per lane (global_load_lds_dword): lane l's dword lands at lds_wave_base + 4*l.
#ifndef TAH_ASYNC_COPY_4B
#define TAH_ASYNC_COPY_4B(gsrc, lds_wave_base)                                                                     \
    do {                                                                                                           \
        const unsigned tah_m0_ = __builtin_amdgcn_readfirstlane(                                                   \
            (unsigned)(uintptr_t)(__attribute__((address_space(3))) void*)(lds_wave_base));                        \
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off"                               \
                     :                                                                                             \
                     : "s"(tah_m0_), "v"(gsrc)                                                                     \
                     : "memory");                                                                                  \
    } while (0)
#endif
__device__ __forceinline__ void async_copy_4B(const void* gsrc, void* lds_wave_base) {
    TAH_ASYNC_COPY_4B(gsrc, lds_wave_base);
}
// 4 bytes per lane from wave-uniform base + per-lane 32-bit byte offset.
#ifndef TAH_ASYNC_COPY_4B_SO
#define TAH_ASYNC_COPY_4B_SO(sbase, voff, lds_wave_base)                                                           \
    do {                                                                                                           \
        const unsigned tah_m0_ = __builtin_amdgcn_readfirstlane(                                                   \
            (unsigned)(uintptr_t)(__attribute__((address_space(3))) void*)(lds_wave_base));                        \
        const uint64_t tah_b_ = (uint64_t)(uintptr_t)(sbase);                                                      \
        const uint64_t tah_sb_ = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((unsigned)tah_b_) |            \
                                 ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((unsigned)(tah_b_ >> 32)) << 32); \
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"                                \
                     :                                                                                             \
                     : "s"(tah_m0_), "v"(voff), "s"(tah_sb_)                                                       \
                     : "memory");                                                                                  \
    } while (0)
#endif
__device__ __forceinline__ void async_copy_4B(const void* sbase, uint32_t voff, void* lds_wave_base) {
    TAH_ASYNC_COPY_4B_SO(sbase, voff, lds_wave_base);
}
#ifndef TAH_CPU_EMU
// the same copies with the destination given as an LDS-address-space pointer
__device__ __forceinline__ void async_copy_16B(const void* sbase, uint32_t voff, lds_byte* lds_wave_base) {
    TAH_ASYNC_COPY_16B_SO(sbase, voff, lds_wave_base);
}
__device__ __forceinline__ void async_copy_4B(const void* sbase, uint32_t voff, lds_float* lds_wave_base) {
    TAH_ASYNC_COPY_4B_SO(sbase, voff, lds_wave_base);
}
#endif
// acc (16 floats of an MFMA accumulator) *= a, executed only if the wave-uniform `cond` is non-zero.
// The branch lives inside the assembly so that the compiler sees one unconditional in-place update:
// a C++ `if` around accumulator updates makes it keep two copies of the accumulators.
#ifndef TAH_SCALE16_IF
#define TAH_SCALE16_IF(acc, a, cond)                                                                               \
    asm volatile(                                                                                                  \
        "s_cmp_eq_u32 %[cd], 0\n\t"                                                                                \
        "s_cbranch_scc1 .Ltah_skip_%=\n\t"                                                                         \
        "v_mul_f32 %[o0], %[al], %[o0]\n\tv_mul_f32 %[o1], %[al], %[o1]\n\t"                                       \
        "v_mul_f32 %[o2], %[al], %[o2]\n\tv_mul_f32 %[o3], %[al], %[o3]\n\t"                                       \
        "v_mul_f32 %[o4], %[al], %[o4]\n\tv_mul_f32 %[o5], %[al], %[o5]\n\t"                                       \
        "v_mul_f32 %[o6], %[al], %[o6]\n\tv_mul_f32 %[o7], %[al], %[o7]\n\t"                                       \
        "v_mul_f32 %[o8], %[al], %[o8]\n\tv_mul_f32 %[o9], %[al], %[o9]\n\t"                                       \
        "v_mul_f32 %[o10], %[al], %[o10]\n\tv_mul_f32 %[o11], %[al], %[o11]\n\t"                                   \
        "v_mul_f32 %[o12], %[al], %[o12]\n\tv_mul_f32 %[o13], %[al], %[o13]\n\t"                                   \
        "v_mul_f32 %[o14], %[al], %[o14]\n\tv_mul_f32 %[o15], %[al], %[o15]\n"                                     \
        ".Ltah_skip_%=:"                                                                                           \
        : [o0] "+v"((acc)[0]), [o1] "+v"((acc)[1]), [o2] "+v"((acc)[2]), [o3] "+v"((acc)[3]),                      \
          [o4] "+v"((acc)[4]), [o5] "+v"((acc)[5]), [o6] "+v"((acc)[6]), [o7] "+v"((acc)[7]),                      \
          [o8] "+v"((acc)[8]), [o9] "+v"((acc)[9]), [o10] "+v"((acc)[10]), [o11] "+v"((acc)[11]),                  \
          [o12] "+v"((acc)[12]), [o13] "+v"((acc)[13]), [o14] "+v"((acc)[14]), [o15] "+v"((acc)[15])               \
        : [al] "v"(a), [cd] "s"(cond)                                                                              \
        : "scc")
#endif
// Empty statement that counts as a use of four register values at this point of the program.
#ifndef TAH_KEEP_HERE4
#define TAH_KEEP_HERE4(a, b, c, d) asm volatile("" ::"v"(a), "v"(b), "v"(c), "v"(d))
#endif
// Makes two register values opaque to the optimiser at this point, so that what is derived from them
// afterwards is computed here (and not hoisted out of a loop into registers of its own).
#ifndef TAH_OPAQUE2
#define TAH_OPAQUE2(a, b) asm volatile("" : "+v"(a), "+v"(b))
#endif
#ifndef TAH_OPAQUE1
#define TAH_OPAQUE1(a) asm volatile("" : "+v"(a))
#endif
// Occupancy the kernel is written for; lets the scheduler spend registers on latency hiding.
// Between LDS writes of a wave and reads, by the same wave, of what its other lanes wrote: the lanes run
// in lockstep and the LDS serves a wave's requests in order, so all that is needed is that the compiler
// keeps the accesses in program order.
#ifndef TAH_WAVE_LDS_SYNC
#define TAH_WAVE_LDS_SYNC()                                      \
    do {                                                         \
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");   \
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");   \
    } while (0)
#endif
#ifndef TAH_WAVES_PER_EU
#define TAH_WAVES_PER_EU(lo, hi) __attribute__((amdgpu_waves_per_eu(lo, hi)))
#endif
#ifndef TAH_WAIT_VMEM_N
// s_waitcnt vmcnt(n), n <= 63: all but the n most recently issued loads / asynchronous copies have landed
#define TAH_WAIT_VMEM_N(n) __builtin_amdgcn_s_waitcnt(0x0F70 | ((n) & 15) | ((n) >> 4 << 14))
#endif

// LDS tile of R rows x 128 bf16 (256 B per row, 16 chunks of 16 B).  The chunk index is XORed
// with a 4-bit function of the row that (a) takes 16 different values over 16 consecutive rows,
// so 16 lanes reading the same logical chunk of consecutive rows (MFMA A operand, b128) touch 16
// different bank groups, and (b) moves 4 consecutive rows into 4 different aligned groups of 4
// chunks, so a transpose read (4 rows x 64 contiguous bytes per half-wave) is conflict-free too.
__device__ __forceinline__ constexpr int row_swizzle(int row) { return ((row & 3) << 2) | ((row >> 2) & 3); }
__device__ __forceinline__ int rowmajor128_off(int row, int chunk) { return row * 256 + ((chunk ^ row_swizzle(row)) << 4); }

// LDS tile of R rows x 64 bf16 (128 B per row, 8 chunks of 16 B), swizzled likewise.
__device__ __forceinline__ int rowmajor64_off(int row, int chunk) { return row * 128 + ((chunk ^ ((row >> 1) & 7)) << 4); }

// ds_read_b64_tr_b16: each lane supplies the LDS address of 4 consecutive bf16 (a row fragment).
// Within each group of 16 lanes the fragments form a flat array G[64] in lane order and lane i
// of the group receives G[i], G[16+i], G[32+i], G[48+i].  With lane r of the group pointing at
// element [row0 + r/4][col0 + 4*(r%4)] of a row-major tile, lane i ends up with
// [row0 + t][col0 + i] for t = 0..3: four rows of one column, i.e. a transposed fragment.
__device__ __forceinline__ bf16x4 lds_read_tr16(const unsigned char* p) {
    typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;
    return __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)p);
}
#ifndef TAH_CPU_EMU
__device__ __forceinline__ bf16x4 lds_read_tr16(const lds_byte* p) {
    typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;
    return __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)p);
}
#endif

// MFMA operand whose contraction index runs over the ROWS of a row-major [rows][128] bf16 LDS
// tile (rowmajor128_off layout): returns, for this lane, the 8 values
// tile[row16 + 8*a + 4*half + b][col32 + lane%32], a = 0..1, b = 0..3, in slot order 4*a + b --
// the slot order in which a 32x32 accumulator (lane half, reg) enumerates its rows, so that an
// accumulator converted to bf16 is directly the other operand of the same MFMA.
__device__ __forceinline__ bf16x8 lds_read_rows_as_k(const unsigned char* tile, int row16, int col32, int lane) {
    const int half = lane >> 5, r = lane & 15, grp = (lane >> 4) & 1;
    const int col = col32 + 16 * grp + 4 * (r & 3);
    const int row = row16 + 4 * half + (r >> 2);
    const bf16x4 lo = lds_read_tr16(tile + rowmajor128_off(row, col >> 3) + (col & 7) * 2);
    const bf16x4 hi = lds_read_tr16(tile + rowmajor128_off(row + 8, col >> 3) + (col & 7) * 2);
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

// Storage slot of key `key` (0..63) inside a transposed 64-key row.  The PV
// MFMA contracts over keys; operand slot (half h, j) of 16-key step s must hold
// the same key as S^T accumulator (half h, reg 8*(s%2)+j), i.e. key
// 16s + 8*(j/4) + 4h + j%4.  Storing key 16s+8a+4h+b at slot 16s+8h+4a+b makes
// each lane's 8 operand keys one contiguous 16-byte chunk.
__device__ __forceinline__ constexpr int pv_slot(int key) {
    return (key & ~12) | ((key & 4) << 1) | ((key & 8) >> 1);
}

// max over the two lanes l and l^32 (v_permlane32_swap: no LDS traffic)
__device__ __forceinline__ float wave_max_xor32(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float wave_sum_xor32(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// the same over lanes l and l^16 (v_permlane16_swap)
__device__ __forceinline__ float wave_max_xor16(float x) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float wave_sum_xor16(float x) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// Sum over a wave in every lane, in the pairs of a shuffle tree from 32 down to 1 (the same bits) without its trips through LDS.  Behind the
// pairs 32, 16 and 8 apart lanes that differ in those bits hold the same number, so turning a row by 4, 2 and 1 is the pairs that far apart.
__device__ __forceinline__ float wave_sum_tree(float x) {
    x = wave_sum_xor16(wave_sum_xor32(x));
    const auto turned = [](float v, auto by) {
        return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + decltype(by)::value, 0xf, 0xf, true));  // row_ror
    };
    x += turned(x, std::integral_constant<int, 8>{});
    x += turned(x, std::integral_constant<int, 4>{});
    x += turned(x, std::integral_constant<int, 2>{});
    return x + turned(x, std::integral_constant<int, 1>{});
}

// x of one lane, the same one for the whole wave
__device__ __forceinline__ int lane_value(int x, int lane) {
#ifdef TAH_CPU_EMU
    return __shfl(x, lane);
#else
    return __builtin_amdgcn_readlane(x, lane);
#endif
}
__device__ __forceinline__ float lane_value(float x, int lane) { return __int_as_float(lane_value(__float_as_int(x), lane)); }

// Largest / smallest of a wave, in every lane, without a trip through LDS (each of the six exchanges of a shuffle tree is one).
template <class T, class F>
__device__ __forceinline__ T wave_quick(T x, F pick) {
    const auto from = [](T v, auto ctrl) {
        return __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), decltype(ctrl)::value, 0xf, 0xf, true));
    };
    x = pick(x, from(x, std::integral_constant<int, 0xB1>{}));   // quad_perm [1,0,3,2]
    x = pick(x, from(x, std::integral_constant<int, 0x4E>{}));   // quad_perm [2,3,0,1]
    x = pick(x, from(x, std::integral_constant<int, 0x141>{}));  // row_half_mirror
    x = pick(x, from(x, std::integral_constant<int, 0x140>{}));  // row_mirror
    const auto at = [&](int lane) { return lane_value(x, lane); };
    return pick(pick(at(0), at(16)), pick(at(32), at(48)));
}
__device__ __forceinline__ int wave_reduce_max(int x) { return wave_quick(x, [](int a, int b) { return a > b ? a : b; }); }
__device__ __forceinline__ int wave_reduce_min(int x) { return wave_quick(x, [](int a, int b) { return a < b ? a : b; }); }
// Sum over this lane and those below it, likewise.
__device__ __forceinline__ int wave_prefix_sum(int x) {
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);   // row_shr:1, 2, 4, 8: inside sixteen lanes
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
    return x;
}

// Element i of an int32 array that no kernel of this library writes (sequence boundaries), read with
// a wave-uniform index: through the constant address space, i.e. with a scalar load when the address is
// uniform — a fraction of the latency of a vector load, which matters in the serial walk over the
// boundaries at the start of a workgroup.
#ifndef TAH_CONST_AS
#define TAH_CONST_AS __attribute__((address_space(4)))
#endif
__device__ __forceinline__ int32_t const_i32(const int32_t* a, int i) { return ((const TAH_CONST_AS int32_t*)a)[i]; }

// Boundaries of a wave's 64 sequences from b0 on, one per lane (no sequence: an empty one).  Asked for without a branch, so that a
// kernel can have those of all its streams on their way at once.  Sequence b's rows are cu[b << shift] ... cu[(b << shift) + 1]: shift 0
// for sequences one behind the other, 1 for (first row, one past the last) pairs with rows between sequences that belong to none.  nseq > b0.
struct LaneBounds {
    int lo, hi;
};
__device__ __forceinline__ LaneBounds lane_bounds(const int32_t* cu, int b0, int nseq, int shift) {
    const int b = b0 + (int)(threadIdx.x % kWave);
    const bool there = b < nseq;
    LaneBounds x;
    const int at = (there ? b : b0) << shift;
    x.lo = cu[at];
    x.hi = cu[at + 1];
    x.lo = there ? x.lo : 0;
    x.hi = there ? x.hi : 0;
    return x;
}

// Locate tile `slot` among sequences with the boundaries lane_bounds reads, `bm` rows
// per tile.  On success fills seq/row0/row_end and returns true; otherwise
// subtracts the number of tiles in this stream from `slot` and returns false.
// Every lane of the wave must call it with the same arguments: the lanes take 64 sequences at a time (one pair of
// loads and a prefix sum over the lanes), so that a batch of hundreds of short sequences costs a workgroup a few
// steps and not one scalar load pair per sequence.  `first`: lane_bounds(cu, 0, nseq, shift), nseq > 0.
__device__ __forceinline__ bool find_tile(const int32_t* cu, int shift, int nseq, int bm, int& slot, int& seq, int& row0, int& row_end, LaneBounds first) {
    for (int b0 = 0; b0 < nseq; b0 += kWave) {
        const LaneBounds x = b0 == 0 ? first : lane_bounds(cu, b0, nseq, shift);
        const int n = (x.hi - x.lo + bm - 1) / bm;
        const int incl = wave_prefix_sum(n);  // tiles of sequences b0 .. b
        const int tot = lane_value(incl, kWave - 1);
        if (slot < tot) {
            const int src = __builtin_ctzll(__ballot(slot < incl));  // the first sequence whose tiles reach past `slot`
            const int lo_s = lane_value(x.lo, src), hi_s = lane_value(x.hi, src);
            seq = b0 + src;
            row0 = lo_s + (slot - (lane_value(incl, src) - lane_value(n, src))) * bm;
            row_end = row0 + bm < hi_s ? row0 + bm : hi_s;
            return true;
        }
        slot -= tot;
    }
    return false;
}
__device__ __forceinline__ bool find_tile(const int32_t* cu, int shift, int nseq, int bm, int& slot, int& seq, int& row0, int& row_end) {
    return nseq > 0 && find_tile(cu, shift, nseq, bm, slot, seq, row0, row_end, lane_bounds(cu, 0, nseq, shift));
}

// The first 64 sequences' boundaries in both streams of a varlen call, asked for at once: a workgroup's start is a chain of trips to
// memory, and which tile it is, where its sequence's keys lie and how many there are then follow from one of them.
struct CallBounds {
    LaneBounds q1, k1, q2, k2;
};
template <class P>
__device__ __forceinline__ CallBounds call_bounds(const P& p) {
    CallBounds x;
    x.q1 = lane_bounds(p.s1.cu_q, 0, p.nseq, p.s1.q_shift);
    x.k1 = lane_bounds(p.s1.cu_k, 0, p.nseq, p.s1.k_shift);
    x.q2 = lane_bounds(p.s2.cu_q, 0, p.nseq, p.s2.q_shift);
    x.k2 = lane_bounds(p.s2.cu_k, 0, p.nseq, p.s2.k_shift);
    return x;
}
// Boundaries that a call may come without (no queries, no keys that anybody looks at): call_bounds reads the depth-0 keys' in their place.
// (Chosen on the host: a choice between pointers in a kernel became a branch with a trip to the arguments inside.)
template <class P>
void fill_absent_bounds(P& p, bool k2) {
    auto same = [&](const int32_t*& cu, int32_t& shift) {
        cu = p.s1.cu_k;
        shift = p.s1.k_shift;
    };
    if (p.s1.total_q == 0) same(p.s1.cu_q, p.s1.q_shift);
    if (p.s2.total_q == 0) same(p.s2.cu_q, p.s2.q_shift);
    if (!k2) same(p.s2.cu_k, p.s2.k_shift);
}
// Those of one sequence (the same one for the whole wave)
__device__ __forceinline__ LaneBounds bounds_at(const LaneBounds& first, const int32_t* cu, int shift, int seq) {
    LaneBounds x;
    x.lo = seq < kWave ? lane_value(first.lo, seq % kWave) : const_i32(cu, seq << shift);
    x.hi = seq < kWave ? lane_value(first.hi, seq % kWave) : const_i32(cu, (seq << shift) + 1);
    return x;
}

// ---------------------------------------------------------------------------
// Launch-order table of a varlen call (built by tah_duo_schedule_build): the tiles of both depths sorted
// by the number of tile steps they run, heaviest first, so that a launch of few, unequal workgroups per
// compute unit ends with the light ones.  int32 words: a header, then one (x, y) pair per launch slot of
// the query-tile kernels (forward, dQ), then one pair per slot of the key-tile kernel (dK/dV).
//   x = the tile's number in the order find_tile counts them (the depth-0 stream's tiles sequence by sequence, then
//       the depth-1 stream's); y = 0 (reserved).
// Every number below the list's length appears exactly once (those past the last tile at the end), so whatever
// boundaries a call has, walking the list visits each of its tiles once: a table built for other boundaries of the
// same sizes costs the intended order, never a tile.
// ---------------------------------------------------------------------------
constexpr int32_t kSchedMagic = 0x54414853;
constexpr int kSchedHeaderWords = 16;
enum { kSchedNseq = 1, kSchedGroup, kSchedTotalQ1, kSchedTotalQ2, kSchedTotalK1, kSchedTotalK2, kSchedQSlots, kSchedKSlots };
constexpr int kSchedKeyTile = 128;  // keys per workgroup of the dK/dV kernel

// launch slots of a kernel that tiles the rows of both streams by `bm` (an upper bound on
// sum_b ceil(len_b / bm) that needs no device read)
inline __host__ __device__ int sched_slots(int nseq, int bm, int total_1, int total_2) {
    return (total_1 > 0 ? total_1 / bm + nseq : 0) + (total_2 > 0 ? total_2 / bm + nseq : 0);
}

// The tile number that launch slot `idx` takes from the table, if the table was built for this call's sizes and this
// kernel's grid (true); otherwise the caller keeps its own order (false).
__device__ __forceinline__ bool sched_lookup(const int32_t* sched, bool key_tiles, int nseq, int group, int total_q1,
                                             int total_q2, int total_k1, int total_k2, int slots, int idx, int& slot) {
    if (!sched) return false;
    // (all of the header is asked for before any of it is compared)
    int h[kSchedKSlots + 1];
#pragma unroll
    for (int i = 0; i <= kSchedKSlots; ++i) h[i] = const_i32(sched, i);
    const int other = (h[0] ^ kSchedMagic) | (h[kSchedNseq] ^ nseq) | (h[kSchedGroup] ^ group) | (h[kSchedTotalQ1] ^ total_q1) |
                      (h[kSchedTotalQ2] ^ total_q2) | (h[kSchedTotalK1] ^ total_k1) | (h[kSchedTotalK2] ^ total_k2) |
                      (h[key_tiles ? kSchedKSlots : kSchedQSlots] ^ slots);
    if (other != 0) return false;
    const int base = kSchedHeaderWords + (key_tiles ? 2 * h[kSchedQSlots] : 0);
    const int x = const_i32(sched, base + 2 * idx);
    if (x < 0 || x >= slots) return false;  // (not a table this library wrote)
    slot = x;
    return true;
}

}  // namespace tah
