// Device-side building blocks shared by the attention-JVP kernels (gfx950 / CDNA4 only).
//
// Streaming (the tile algebra is described in sjvp_w16.hpp)
// ---------
// The looped side of a kernel lives in LDS stage slabs: unpadded [32][HD] 16-bit, XOR-swizzled in units of 16
// bytes, which keeps both LDS access patterns (row-major 16-byte reads, and the 4-row x 32-byte
// footprint of a transposing read) free of bank conflicts.  The kernels fill a ring of such
// stages with the LDS-DMA form of the global load (global_load_lds_dwordx4: 16 bytes per lane
// straight into LDS, no registers), issued ahead of use and retired with explicit
// s_waitcnt vmcnt(n); because every lane of an LDS-DMA load supplies its own global address, the
// swizzle costs nothing at copy time.  Rows that do not start on 16-byte boundaries, and fp32 rows, go through
// registers instead (sjvp_staged16.hpp).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sjvp {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef uint16_t elem_t;  // storage type of one 16-bit element, whatever its format

constexpr int kStageRows = 32;       // rows of the looped axis per stage
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

struct Bf16 {
    static __device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                      __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
        bf16x2 v = {(__bf16)lo, (__bf16)hi};
        return __builtin_bit_cast(uint32_t, v);
    }
    static __device__ __forceinline__ float to_float(elem_t x) {
        return __builtin_bit_cast(float, (uint32_t)x << 16);
    }
    // a.lo * b.lo + a.hi * b.hi + c on a packed pair, accumulated in fp32 (v_dot2c_f32_bf16)
    static __device__ __forceinline__ float dot2(uint32_t a, uint32_t b, float c) {
        return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, a), __builtin_bit_cast(bf16x2, b), c,
                                               false);
    }
};

struct Fp16 {
    static __device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                     __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
        f16x2 v = {(_Float16)lo, (_Float16)hi};
        return __builtin_bit_cast(uint32_t, v);
    }
    static __device__ __forceinline__ float to_float(elem_t x) {
        return (float)__builtin_bit_cast(_Float16, x);
    }
    static __device__ __forceinline__ float dot2(uint32_t a, uint32_t b, float c) {
        return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, a), __builtin_bit_cast(f16x2, b), c, false);
    }
};

// A [B,H,L,D] view: base pointer and element strides; the last dimension has unit stride.
struct TensorView {
    const elem_t* ptr;
    int64_t sb, sh, sl;
    __device__ __forceinline__ const elem_t* head(int b, int h) const {
        return ptr + b * sb + h * sh;
    }
};

struct OutView {
    elem_t* ptr;
    int64_t sb, sh, sl;
    __device__ __forceinline__ elem_t* head(int b, int h) const { return ptr + b * sb + h * sh; }
};

// cos / sin tables of a rotary position embedding folded into a kernel (see sjvp_w16.hpp)
struct RopeTables {
    const float* cos;  // [rows][32] fp32, row stride cs (multiple of 4, 16-byte aligned base); null: no rotation
    const float* sin;
    int64_t cs;
    int rows;          // rows of the tables (positions beyond are clamped; their data is zero padding)
};

// Workgroup barrier.  __syncthreads() leaves the wait for this wave's own LDS writes to the compiler,
// and at the head of a loop the compiler has been seen to hoist that wait into the loop's preheader
// only, so that a wave reached the barrier with the LDS write that ends its loop body still queued
// and another wave read the old value behind the barrier (one 16 x 16 tile of dQ in one of some ten
// thousand).  The explicit s_waitcnt lgkmcnt(0) is kept by the compiler wherever the barrier goes.
__device__ __forceinline__ void workgroup_barrier() {
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0); vmcnt and expcnt untouched
    __syncthreads();
}
// The same with a vote: true if `pred` holds for any thread of the workgroup.
__device__ __forceinline__ bool workgroup_barrier_or(bool pred) {
    __builtin_amdgcn_s_waitcnt(0xC07F);
    return __syncthreads_or(pred) != 0;
}

// Exchange through LDS among the lanes of ONE wave: the wave's LDS instructions run in order, but the compiler sees
// lanes one by one, and where the reads stand under a condition it may send the lanes outside it ahead, to
// writes that come behind the reads (seen: the next tensor's tile of the row stores written by the lanes
// without a row before the others had read the last one).  No instruction.
__device__ __forceinline__ void wave_exchange() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float fast_log2(float x) { return __builtin_amdgcn_logf(x); }

// ---------------------------------------------------------------------------------------------
// LDS stage slab: [32 rows][HD] elements, 16-byte chunk c of row r stored at chunk position
// c ^ swz(r).  The LDS has 64 banks of 4 bytes, i.e. 256 bytes per bank row, and serves a 16-byte
// read of 16 lanes per cycle: swz is chosen so that 16 consecutive slab rows read at one logical
// chunk (the A operand of a score tile) land in 16 distinct 16-byte positions of a bank row
// (measured on gfx950: 546 bytes/clk per CU against 315 with a swizzle that repeats every 8 rows).
// The transposing reads (4 rows x 32 bytes per group of 16 lanes) run at their full rate with it too.
// (A variant that also separates the four rows of a transposing read into distinct 32-byte positions
// measured worse: more conflict cycles on the hardware counter and 2 % less throughput.)
// swz has period 16 in the row.
template <int HD>
__device__ __forceinline__ int swz(int row) {
    if constexpr (HD == 32) return (row >> 2) & 3;  // four 64-byte rows per bank row
    if constexpr (HD == 64) return (row >> 1) & 7;  // two 128-byte rows per bank row
    return row & 15;                                // one 256-byte row per bank row
}

template <int HD>
struct Slab {
    static constexpr int elems = kStageRows * HD;
    static constexpr int chunks = kStageRows * HD / 8;  // 16-byte chunks
};

// LDS byte address of a pointer into shared memory: the low half of its flat address.
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
    return (uint32_t)(uintptr_t)p;
}

// LDS-DMA: each active lane copies 16 bytes from its global address to LDS byte address
// base + 16 * lane_id (base must be wave-uniform).  Completion is tracked by vmcnt only.  M0 carries
// the LDS base; nothing else in these kernels uses M0 (gfx9 LDS instructions do not need it).
__device__ __forceinline__ void dma16(const void* gptr, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off"
                 :
                 : "v"(gptr), "s"(__builtin_amdgcn_readfirstlane(lds_base))
                 : "memory");
}
// 4-byte form: LDS byte address base + 4 * lane_id.
__device__ __forceinline__ void dma4(const void* gptr, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dword %0, off"
                 :
                 : "v"(gptr), "s"(__builtin_amdgcn_readfirstlane(lds_base))
                 : "memory");
}

// s_waitcnt vmcnt(ahead * SPT + EXTRA): at most `ahead` later stages (SPT vector-memory instructions each,
// SPT a compile-time constant) of this wave's copies may still be outstanding afterwards.  Loads and
// LDS-DMA copies retire in issue order, so everything issued before those stages has landed.
// EXTRA counts other vector-memory instructions (stores) known to have been issued after them.
// `ahead` is wave-uniform and small (at most the ring depth); counts beyond the 6-bit field are
// clamped, which only makes the wait stricter.
template <int SPT, int EXTRA = 0>
__device__ __forceinline__ void wait_stages(int ahead) {
#define SJVP_VMCNT(n) __builtin_amdgcn_s_waitcnt((((n) > 63 ? 63 : (n)) & 15) | ((((n) > 63 ? 63 : (n)) >> 4) << 14) | 0x0F70)
    switch (ahead) {
        case 0: SJVP_VMCNT(EXTRA); break;
        case 1: SJVP_VMCNT(SPT + EXTRA); break;
        case 2: SJVP_VMCNT(2 * SPT + EXTRA); break;
        case 3: SJVP_VMCNT(3 * SPT + EXTRA); break;
        case 4: SJVP_VMCNT(4 * SPT + EXTRA); break;
        case 5: SJVP_VMCNT(5 * SPT + EXTRA); break;
        case 6: SJVP_VMCNT(6 * SPT + EXTRA); break;
        default: SJVP_VMCNT(7 * SPT + EXTRA); break;
    }
#undef SJVP_VMCNT
}

}  // namespace sjvp
