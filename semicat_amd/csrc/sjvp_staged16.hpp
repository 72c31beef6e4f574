// Copies of the 16-wide kernels for tensors that the LDS-DMA copies of sjvp_w16.hpp cannot read (gfx950): 16-bit
// rows that do not start on 16-byte boundaries (odd head dimensions, offset pointers), and fp32 rows whose
// elements are rounded to 16 bits on their way into LDS.  A stage goes through registers: its loads are issued
// where the LDS-DMA form issues its copies, one stage ahead, and written to LDS behind the arithmetic of the
// stage before, so that they travel under it.
//
// Rows are read in pieces of eight elements with loads of 16 (or twice 16) bytes at whatever alignment they have.
// The piece that reaches beyond column D is read as the LAST eight elements of the row (D >= 16) and
// shifted, so no load leaves a row, and columns >= D arrive as zeros.
//
// Measured, forward + backward (one element at a time through one stage of LDS under 32-wide tiles before):
//   bf16 B=8 H=8 L=300 D=36 158 -> 54 us (as the aligned D = 40), B=64 H=12 L=128 D=20 174 -> 57,
//   B=8 H=16 L=512 D=100 1579 -> 325; fp32 rows B=64 H=12 L=128 D=64 248 -> 139 us, B=128 H=12 L=256 1637 -> 745.
// The shorter life of a stage in registers (one ahead instead of a ring of two or three) costs 15 % against the
// LDS-DMA form; what is left is bound as that one is.
#pragma once
#include <type_traits>

#include "sjvp_w16.hpp"

namespace sjvp {

// How a 16-wide kernel meets the caller's tensors: 16-byte aligned 16-bit rows through LDS-DMA; 16-bit rows of any
// alignment; fp32 rows (pointers passed as elem_t*, strides in 2-byte units).
enum : int { kIoDma = 0, kIoAny = 1, kIoF32 = 2 };

// Eight consecutive elements as they lie in memory.
template <int IO>
struct Raw8 {
    u32x4 a[IO == kIoF32 ? 2 : 1];
    __device__ __forceinline__ void load(const elem_t* row, int col) {
        __builtin_memcpy(a, row + (IO == kIoF32 ? 2 : 1) * col, sizeof(a));
    }
    __device__ __forceinline__ void zero() {
#pragma unroll
        for (int i = 0; i < (IO == kIoF32 ? 2 : 1); ++i) a[i] = u32x4{0u, 0u, 0u, 0u};
    }
    template <typename T>
    __device__ __forceinline__ u32x4 get() const {
        if constexpr (IO == kIoF32) {
            const f32x4 lo = __builtin_bit_cast(f32x4, a[0]), hi = __builtin_bit_cast(f32x4, a[1]);
            return u32x4{T::pack2(lo[0], lo[1]), T::pack2(lo[2], lo[3]), T::pack2(hi[0], hi[1]), T::pack2(hi[2], hi[3])};
        } else {
            return a[0];
        }
    }
};

// Column from which the piece of columns d .. d+7 is read, and the shift that brings it into place.
__device__ __forceinline__ int piece_col(int d, int D) { return d + 8 <= D ? d : D - 8; }
__device__ __forceinline__ int piece_shift(int d, int D) { return min(d - piece_col(d, D), 8); }

// Elements s .. 7 of v, followed by zeros.
__device__ __forceinline__ u32x4 shift_down(u32x4 v, int s) {
    if (s & 4) v = u32x4{v[2], v[3], 0u, 0u};
    if (s & 2) v = u32x4{v[1], v[2], v[3], 0u};
    if (s & 1) v = u32x4{(v[0] >> 16) | (v[1] << 16), (v[1] >> 16) | (v[2] << 16), (v[2] >> 16) | (v[3] << 16), v[3] >> 16};
    if (s & 8) v = u32x4{0u, 0u, 0u, 0u};
    return v;
}

// B operands (all head-dimension chunks of 32) of one owned row of fp32 elements.
template <typename T, int HD, int IO>
__device__ __forceinline__ void staged_b_operands16(u32x4* out, const elem_t* row, int g, int D, bool valid) {
    Raw8<IO> raw[HD / 32];
#pragma unroll
    for (int c = 0; c < HD / 32; ++c) {
        raw[c].zero();
        if (valid) raw[c].load(row, piece_col(32 * c + 8 * g, D));
    }
#pragma unroll
    for (int c = 0; c < HD / 32; ++c) {
        out[c] = raw[c].template get<T>();
        if (D != HD) out[c] = shift_down(out[c], piece_shift(32 * c + 8 * g, D));
    }
}
// 16-bit rows of any alignment: the pieces are requested here, as they lie in a row that exists (own_row), and made operands by
// finish_b_operands16 once all of a wave's rows have been requested.  Made operands one row after the other, each row is
// awaited before the next is requested: forward + backward, in turn / together, B=8 H=8 L=300 D=36 56.7 / 54.0 us, B=64 H=12 L=128
// D=20 61.9 / 56.5, B=100 H=9 30 x 20 D=36 72.0 / 62.3, B=8 H=16 L=512 D=100 354 / 337.
__device__ __forceinline__ int64_t own_row(int64_t row, int L) { return row < L ? row : L - 1; }
template <int HD, int IO>
__device__ __forceinline__ void finish_b_operands16(u32x4* out, int g, int D, bool valid) {
    if constexpr (IO == kIoAny) {
#pragma unroll
        for (int c = 0; c < HD / 32; ++c) {
            if (D != HD) out[c] = shift_down(out[c], piece_shift(32 * c + 8 * g, D));
            if (!valid) out[c] = u32x4{0u, 0u, 0u, 0u};
        }
    }
}

// CopyPlan (sjvp_w16.hpp) through registers: issue() requests the next window, commit() writes it to the region it
// was issued for, slab j of the window PITCH elements behind slab j - 1.
template <typename T, int HD, int NS, int NT, int IO, int PITCH = Slab<HD>::elems>
struct StagedPlan {
    static constexpr int chunks = Slab<HD>::chunks;
    static constexpr int total = NS * chunks;
    static constexpr int N = (total + NT - 1) / NT;
    static_assert(chunks % 64 == 0 && (NT % chunks == 0 || chunks % NT == 0), "powers of two");
    const elem_t* src[N];  // first column this thread reads of its row in the next window
    int64_t adv[N];        // elements from one window to the next (wave-uniform)
    int row[N];
    int pos8;              // element offset of this thread's first chunk position
    int shift;             // of every chunk: a thread's positions are the same columns of successive slabs or rows
    bool shifted;          // wave-uniform: D does not fill the slabs
    elem_t* region;
    bool pending;
    Raw8<IO> raw[N];

    __device__ __forceinline__ void init(int tid, int D, Src t0, Src t1, Src t2 = Src{nullptr, 0}, Src t3 = Src{nullptr, 0},
                                         Src t4 = Src{nullptr, 0}, Src t5 = Src{nullptr, 0}) {
        static_assert(NS <= 6, "at most six tensors per copy");
        constexpr int CH = HD / 8;
        const int q0 = tid % chunks;
        const int c8 = 8 * ((q0 % CH) ^ swz<HD>(q0 / CH));
        static_assert(NT >= chunks || (NT / CH) % 16 == 0, "parts of a slab start at multiples of 16 rows");
        const int j0 = __builtin_amdgcn_readfirstlane(tid / chunks);
        const int col = (IO == kIoF32 ? 2 : 1) * piece_col(c8, D);
        shift = piece_shift(c8, D);
        shifted = D != HD;
        pos8 = j0 * PITCH + 8 * q0;
        pending = false;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int j = NT >= chunks ? j0 + (NT / chunks) * i : i / (chunks / NT);
            const int r = NT >= chunks ? q0 / CH : q0 / CH + (NT / CH) * (i % (chunks / NT));
            // the tensor of slab j: one of SPI neighbours, chosen by the (wave-uniform) slab of position 0
            constexpr int SPI = NT >= chunks ? NT / chunks : 1;
            const Src ts[6] = {t0, t1, t2, t3, t4, t5};
            const int first = NT >= chunks ? SPI * i : i / (chunks / NT);
            Src s = ts[first < NS ? first : 0];
#pragma unroll
            for (int k = 1; k < SPI; ++k)
                if (first + k < NS && j0 == k) s = ts[first + k < NS ? first + k : 0];
            row[i] = j < NS ? r : 1 << 30;  // a position beyond the last slab has no row
            src[i] = s.ptr + (int64_t)r * s.sl + col;
            adv[i] = 32 * s.sl;
        }
    }
    // Windows first, first + step, ... instead of all of them.
    __device__ __forceinline__ void take(int first, int step) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            src[i] += first * adv[i];
            adv[i] *= step;
        }
    }
    // Request the next window for `to`; rows_left of its rows exist (zeros beyond).
    __device__ __forceinline__ void issue(elem_t* to, int rows_left) {
        region = to;
        pending = true;
        if (total % NT == 0 && rows_left >= kStageRows) {
#pragma unroll
            for (int i = 0; i < N; ++i) raw[i].load(src[i], 0);
        } else {
#pragma unroll
            for (int i = 0; i < N; ++i) {
                raw[i].zero();
                if (row[i] < rows_left) raw[i].load(src[i], 0);
            }
        }
#pragma unroll
        for (int i = 0; i < N; ++i) src[i] += adv[i];
    }
    __device__ __forceinline__ void commit() {
        if (!pending) return;  // wave-uniform
        pending = false;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            if (total % NT != 0 && row[i] >= kStageRows) continue;
            u32x4 v = raw[i].template get<T>();
            if (shifted) v = shift_down(v, shift);
            constexpr int PPS = NT >= chunks ? 1 : chunks / NT;    // positions per slab
            constexpr int SPI = NT >= chunks ? NT / chunks : 1;    // slabs from one position to the next
            *reinterpret_cast<u32x4*>(region + pos8 + (i / PPS) * SPI * PITCH + (i % PPS) * 8 * NT) = v;
        }
    }
};

// B operands (all head-dimension chunks of 32) of one owned row, straight from global memory (kIoAny: own_row of it, to be finished).
// (GROUPED: the zeros come as one register group.  Joined with the loaded piece element by element, as the compiler may do, the
// piece is awaited as soon as it is requested.  Row-owned kernel at D = 80, 1476 queries on 10 keys: 278 -> 245 us; the forward
// of few workgroups, whose pieces were not affected, loses by it: 333 x 205, D = 48 8.9 -> 9.8 us.)
template <typename T, int HD, int IO, bool GROUPED = false>
__device__ __forceinline__ void load_b_operands16(u32x4* out, const elem_t* row, int g, int D, bool valid) {
    if constexpr (IO == kIoF32) return staged_b_operands16<T, HD, IO>(out, row, g, D, valid);
    if constexpr (IO == kIoAny) {
#pragma unroll
        for (int c = 0; c < HD / 32; ++c) __builtin_memcpy(&out[c], row + piece_col(32 * c + 8 * g, D), sizeof(out[c]));
        return;
    }
#pragma unroll
    for (int c = 0; c < HD / 32; ++c) {
        u32x4 piece = {0u, 0u, 0u, 0u};
        if constexpr (GROUPED) asm volatile("" : "+v"(piece));
        if (valid && 32 * c + 8 * g < D) piece = *reinterpret_cast<const u32x4*>(row + 32 * c + 8 * g);
        out[c] = piece;
    }
}

// The same from a uniform slice pointer and the lane's byte offset in the slice: whole rows of HD elements
// that all exist, no predicates, one 32-bit offset for every tensor of equal strides.
template <int HD>
__device__ __forceinline__ void load_b_operands16_at(u32x4* out, const elem_t* slice, uint32_t lane_bytes) {
    const char* base = reinterpret_cast<const char*>(slice);
#pragma unroll
    for (int c = 0; c < HD / 32; ++c) out[c] = *reinterpret_cast<const u32x4*>(base + lane_bytes + 64 * c);
}

// One 16-byte piece (columns 8c ..) of a 16-bit row of any alignment, masked at D.
__device__ __forceinline__ void store_piece(elem_t* dst, u32x4 v, int d, int D) {
    if (d + 8 <= D) {
        __builtin_memcpy(dst, &v, sizeof(v));
    } else {
#pragma unroll
        for (int e = 0; e < 7; ++e)
            if (d + e < D) dst[e] = (elem_t)(v[e >> 1] >> (16 * (e & 1)));
    }
}
// Four consecutive fp32 elements at columns d .., masked at D.
__device__ __forceinline__ void store_f32x4(elem_t* row, f32x4 v, int d, int D) {
    float* dst = reinterpret_cast<float*>(row) + d;
    if (d + 4 <= D) {
        __builtin_memcpy(dst, &v, sizeof(v));
    } else {
#pragma unroll
        for (int e = 0; e < 3; ++e)
            if (d + e < D) dst[e] = v[e];
    }
}

// One spelling for both kinds of plan.
template <int HD, int NS, int NT, typename... S>
__device__ __forceinline__ void init_plan(CopyPlan<HD, NS, 1, NT>& plan, int tid, int D, const void* sink, S... srcs) {
    plan.init(tid, 0, D, sink, srcs...);
}
template <typename T, int HD, int NS, int NT, int IO, int P, typename... S>
__device__ __forceinline__ void init_plan(StagedPlan<T, HD, NS, NT, IO, P>& plan, int tid, int D, const void*, S... srcs) {
    plan.init(tid, D, srcs...);
}
template <int HD, int NS, int NT>
__device__ __forceinline__ void issue_plan(CopyPlan<HD, NS, 1, NT>& plan, elem_t* slot, int rows_left, bool whole) {
    plan.issue(slot, rows_left, whole);
}
template <typename T, int HD, int NS, int NT, int IO, int P>
__device__ __forceinline__ void issue_plan(StagedPlan<T, HD, NS, NT, IO, P>& plan, elem_t* slot, int rows_left, bool) {
    plan.issue(slot, rows_left);
}

// store_tile16 (sjvp_w16.hpp) for rows of any alignment: 16-bit rows leave through the wave's staging tile as there,
// fp32 rows unrounded straight from the accumulators (four lanes hold 64 consecutive bytes of a row).
template <typename T, int HD, int IO, int DT = HD / 16>
__device__ __forceinline__ void staged_store_tile16(elem_t* stage, elem_t* gp, int64_t sl, int row0, int L, int D,
                                                    const f32x4* acc, float mul, int lane) {
    const int n = lane & 15, g = lane >> 4;
    if constexpr (IO == kIoF32) {
        if (row0 + n >= L) return;
        elem_t* row = gp + (int64_t)(row0 + n) * sl;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) store_f32x4(row, acc[dt] * mul, 16 * dt + 4 * g, D);
    } else {
        constexpr int P = StoreStage16<HD>::pitch;
        wave_exchange();  // the tile's last readers are done
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            u32x2 val = {T::pack2(acc[dt][0] * mul, acc[dt][1] * mul), T::pack2(acc[dt][2] * mul, acc[dt][3] * mul)};
            *reinterpret_cast<u32x2*>(stage + n * P + 16 * dt + 4 * g) = val;
        }
        wave_exchange();
        constexpr int CH = HD / 8;
        constexpr int RPI = 64 / CH;
#pragma unroll
        for (int it = 0; it < (16 + RPI - 1) / RPI; ++it) {
            const int r = it * RPI + lane / CH;
            const int c = lane % CH;
            if ((RPI <= 16 || r < 16) && row0 + r < L && 8 * c < D) {
                const u32x4 v = *reinterpret_cast<const u32x4*>(stage + r * P + 8 * c);
                store_piece(gp + (int64_t)(row0 + r) * sl + 8 * c, v, 8 * c, D);
            }
        }
    }
}

// The wave's 16 rows of an output tensor, whatever its storage.
template <typename T, int HD, int IO, bool ROPE = false, int DT = HD / 16>
__device__ __forceinline__ void store_rows16(elem_t* stage, elem_t* gp, int64_t sl, int row0, int L, int D,
                                             const f32x4* acc, float mul, int lane, const RopeTables* rt = nullptr) {
    if constexpr (IO == kIoDma) store_tile16<T, HD, ROPE, DT>(stage, gp, sl, row0, L, D, acc, mul, lane, rt);
    else staged_store_tile16<T, HD, IO, DT>(stage, gp, sl, row0, L, D, acc, mul, lane);
}

}  // namespace sjvp
