// fp32 kernels for problems that fill the chip (gfx950): the contractions of sjvp_f32.hpp on the bf16 matrix pipe,
// with every fp32 operand as a sum of three bf16 values.
//
// x = x0 + x1 + x2 with x0 = bf16(x), x1 = bf16(x - x0), x2 = bf16(x - x0 - x1): 24 significant bits, all of an fp32
// number's from 2^-110 on (bf16 ends at 2^-133; no instruction on the way flushes subnormals).
// Of the nine products of two such operands the three smallest (below 2^-25 of the whole) are left out; the other six are exact in the matrix unit and summed there in fp32, small ones first.  v_mfma_f32_16x16x32_bf16 adds 32 of them
// per rounding step of the accumulator where v_mfma_f32_16x16x4_f32 adds four, so the error against fp64 is smaller: sums of
// 32 / 64 / 512 / 4096 products of normal numbers 3.8e-8 / 9.1e-8 / 3.4e-7 / 1.0e-6 relative, on the fp32 unit 1.0e-7 /
// 1.4e-7 / 4.1e-7 / 1.2e-6.  What was computed in fp32 outside the contractions (exponentials, row sums, statistics,
// accumulators) is here too.
//
// What bounds it: six products at 16 times the rate are 2.7 times as fast as the fp32 unit, if splitting the operands
// (11 vector instructions per pair) stays beside it.  So the streamed side is split once per workgroup, on its way from
// registers to LDS, where it lies as three slabs per tensor in the layout of the 16-bit kernels (sjvp_w16.hpp: row reads
// for the score-like tiles, transposing reads for the output ones); the owned side is split once, and each tile
// once, before the output contractions that it enters.
//
// Measured, forward + backward, the fp32 unit's kernels / these: B=8 H=16 L=1024 D=64 4492 / 2177 us (the matrix pipe busy
// 48, 54 and 52 % of the forward's, row and column kernel's cycles), without tangents 1895 / 853, B=64 H=12 L=128
// D=64 512 / 308, B=8 H=12 L=500 D=32 567 / 257, B=8 H=16 L=512 D=128 2137 / 1466, B=8 H=12 L=500
// D=96 1904 / 886, B=4 H=16 300 queries on 700 keys D=80 1039 / 702.  What is left between the contractions is the split of the
// stage and of the tiles, softmax and barriers.
// Error against fp64 at B=16 H=8 L=512 D=64, worst output: 7.4e-7 / 4.7e-7; over 120 shapes every output's is 0.42 to 1.00 of the unit's.
// (A float as a sum of bfloat16 values, and which of the products matter: G. Henry, P. T. P. Tang, A. Heinecke, "Leveraging the bfloat16 artificial
// intelligence datatype for higher-precision computations", ARITH 2019.)
//
// Numbers that the split does not hold (infinities, NaN) or whose products could overflow one by one where their sum does
// not (2^59 and above) are left to the fp32 unit: a wave that met one, in its own rows, in a stage or in its tiles, computes its
// 16 rows again as the kernels of sjvp_f32.hpp do, behind its loop (inside it the second form costs the first one 60
// registers).  So infinite and overflowing scores come out as they do there.
// So are small numbers, where eight neighbours in a row, or an owned row's tiles of the whole streamed axis, are not all zero and all below
// 2^-100.  (Beside larger ones what a number loses, at most 2^-134, is nothing.)  Gradients of cotangents at 2^-118 have errors up to 5.3e-7 there, in
// three parts 8.5e-5 (the unit alone 4.4e-7: the scores meet the log-sum-exp of the other form's).
// Such waves pay for both forms: where all of a call's are, it takes 1.4 to 1.6 times as long as on the unit alone at D = 64, 2.6 to 3 times at D = 128.
#pragma once
#include "sjvp_f32.hpp"
#include "sjvp_staged16.hpp"

namespace sjvp {

// One operand of a matrix instruction in three parts.
struct Op3 {
    u32x4 p[3];
};
// c0 += a0 b0 and c1 += a1 b1, in turn: an instruction does not wait for the one ahead of it.
__device__ __forceinline__ void mfma6(const Op3& a0, const Op3& b0, f32x4& c0, const Op3& a1, const Op3& b1, f32x4& c1) {
    constexpr int pa[6] = {2, 1, 0, 1, 0, 0}, pb[6] = {0, 1, 2, 0, 1, 0};
#pragma unroll
    for (int i = 0; i < 6; ++i) {
        c0 = Bf16::mfma16(a0.p[pa[i]], b0.p[pb[i]], c0);
        c1 = Bf16::mfma16(a1.p[pa[i]], b1.p[pb[i]], c1);
    }
}

// The same into accumulators that live through the loop: the five small products are summed beside them, which leaves two
// roundings at the accumulator's size per 32 products in the place of six.  (Six, in the column kernel of eight waves: 288 heads, 2000 queries on
// 70 keys, D = 64, dtK, dtV 7.6e-7 against fp64, so 4.5e-7, the fp32 unit's split groups 5.5e-7; forward + backward 1.3 % shorter.)
__device__ __forceinline__ void mfma6_onto(const Op3& a0, const Op3& b0, f32x4& c0, const Op3& a1, const Op3& b1, f32x4& c1) {
    constexpr int pa[5] = {2, 1, 0, 1, 0}, pb[5] = {0, 1, 2, 0, 1};
    f32x4 t0 = {0.f, 0.f, 0.f, 0.f}, t1 = t0;
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        t0 = Bf16::mfma16(a0.p[pa[i]], b0.p[pb[i]], t0);
        t1 = Bf16::mfma16(a1.p[pa[i]], b1.p[pb[i]], t1);
    }
    c0 = Bf16::mfma16(a0.p[0], b0.p[0], c0);
    c1 = Bf16::mfma16(a1.p[0], b1.p[0], c1);
    c0 += t0;
    c1 += t1;
}

// The largest of `most` and the magnitudes of x and y; NaN if one is.
__device__ __forceinline__ float most_of(float most, float x, float y) {
    return __builtin_elementwise_maximum(__builtin_elementwise_maximum(most, fabsf(x)), fabsf(y));
}
// Numbers whose largest magnitude is `most` are for the fp32 unit if that is 2^59 or more, or NaN, or below 2^-100 but not zero.  (By the bits:
// those of magnitudes are in their order, and one less puts zero on the other end.)
constexpr uint32_t kLeast = 0x0d800000u, kMost = 0x5d000000u;
__device__ __forceinline__ uint32_t bits_less_one(float most) { return __builtin_bit_cast(uint32_t, most) - 1u; }
// Groups of numbers, each by its largest magnitude.  (Both ends are compared once for all of a thread's groups: three vector instructions less for
// every group but one; forward + backward at B=8 H=12 L=500 D=96 904 / 886 us, B=4 H=16 300 on 700 D=80 714 / 698, D <= 64 the same.)
struct Met {
    uint32_t least = ~0u;
    float most = 0.f;
    __device__ __forceinline__ void add(float group) {
        least = min(least, bits_less_one(group));
        most = __builtin_elementwise_maximum(most, group);
    }
    __device__ __forceinline__ bool special() const { return (least < kLeast - 1u) | (__builtin_bit_cast(uint32_t, most) >= kMost); }
};
// A row of tiles as one group, `most` by the lanes of one n; wave-uniform.
__device__ __forceinline__ bool tiles_out_of_range(float most) {
    most = most_of(most, __shfl_xor(most, 16, 64), 0.f);
    most = most_of(most, __shfl_xor(most, 32, 64), 0.f);
    Met m;
    m.add(most);
    return __builtin_amdgcn_ballot_w64(m.special()) != 0;
}

// Element i (two neighbours x, y) of the three parts.  What a part leaves over is exact in fp32, and the dot product with
// (-1, 0) or (0, -1) takes it from the packed pair as it is: seven instructions where unpacking and subtracting are eleven.
// (A neighbour that is infinite or NaN makes it NaN: such rows go to the fp32 unit.  The zero beside -1 is a negative one: the pair (-1, +0) is among the constants that
// the compiler writes as the inline operand -1.0, which the instruction reads as the pair (0, -1).)
__device__ __forceinline__ void split3(Op3& o, int i, float x, float y) {
    constexpr uint32_t kLow = 0x8000bf80u, kHigh = 0xbf800000u;
    const uint32_t p0 = Bf16::pack2(x, y);
    x = Bf16::dot2(p0, kLow, x);
    y = Bf16::dot2(p0, kHigh, y);
    const uint32_t p1 = Bf16::pack2(x, y);
    x = Bf16::dot2(p1, kLow, x);
    y = Bf16::dot2(p1, kHigh, y);
    o.p[0][i] = p0;
    o.p[1][i] = p1;
    o.p[2][i] = Bf16::pack2(x, y);
}
// Two score-like tiles of a stage (32 streamed rows) as the B operand of an output contraction.
__device__ __forceinline__ Op3 split_tiles(const f32x4& t0, const f32x4& t1) {
    Op3 o;
    split3(o, 0, t0[0], t0[1]);
    split3(o, 1, t0[2], t0[3]);
    split3(o, 2, t1[0], t1[1]);
    split3(o, 3, t1[2], t1[3]);
    return o;
}
// `most` collects the largest magnitude of the tiles of all stages.
__device__ __forceinline__ Op3 split_tiles(const f32x4& t0, const f32x4& t1, float& most) {
    most = most_of(most_of(most_of(most_of(most, t0[0], t0[1]), t0[2], t0[3]), t1[0], t1[1]), t1[2], t1[3]);
    return split_tiles(t0, t1);
}

// Eight consecutive fp32 elements from column `col` of a row of D (>= 16); those beyond D become zero.  Read as the row's last
// eight where they do not all exist, and shifted (piece_col, piece_shift).
struct F32x8 {
    f32x4 a[2];
    __device__ __forceinline__ void load(const float* at) { __builtin_memcpy(a, at, sizeof(a)); }
    __device__ __forceinline__ void zero() { a[0] = a[1] = f32x4{0.f, 0.f, 0.f, 0.f}; }
    __device__ __forceinline__ float operator[](int i) const { return a[i >> 2][i & 3]; }
    __device__ __forceinline__ void shift(int s) {
        if (s & 4) a[0] = a[1], a[1] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (s & 2) a[0] = f32x4{a[0][2], a[0][3], a[1][0], a[1][1]}, a[1] = f32x4{a[1][2], a[1][3], 0.f, 0.f};
        if (s & 1) a[0] = f32x4{a[0][1], a[0][2], a[0][3], a[1][0]}, a[1] = f32x4{a[1][1], a[1][2], a[1][3], 0.f};
        if (s & 8) zero();
    }
    __device__ __forceinline__ Op3 split(Met& m) const {
        Op3 o;
        float most = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            most = most_of(most, (*this)[2 * i], (*this)[2 * i + 1]);
            split3(o, i, (*this)[2 * i], (*this)[2 * i + 1]);
        }
        m.add(most);
        return o;
    }
};

// The owned row of the lane: columns 32 c + 8 g .. + 7 (zeros beyond D and for a row that does not exist).
template <int KC>
__device__ __forceinline__ void own_load(F32x8* x, const float* row, int g, int D, bool valid) {
#pragma unroll
    for (int c = 0; c < KC; ++c) {
        x[c].zero();
        if (valid) x[c].load(row + piece_col(32 * c + 8 * g, D));
    }
}
template <int KC>
__device__ __forceinline__ void own_cut(F32x8* x, int g, int D) {
    if (D != 32 * KC)
#pragma unroll
        for (int c = 0; c < KC; ++c) x[c].shift(piece_shift(32 * c + 8 * g, D));
}
template <int KC>
__device__ __forceinline__ void own_split(Op3* o, const F32x8* x, Met& m) {
#pragma unroll
    for (int c = 0; c < KC; ++c) o[c] = x[c].split(m);
}
template <int KC>
__device__ __forceinline__ float own_dot(const F32x8* x, const F32x8* y, float sum) {
#pragma unroll
    for (int c = 0; c < KC; ++c)
#pragma unroll
        for (int i = 0; i < 8; ++i) sum = fmaf(x[c][i], y[c][i], sum);
    return sum;
}

// A stage of 32 rows of NS tensors through registers: issue() requests it, commit() writes the three parts of every element to
// the buffer, tensor s part p at slab 3 s + p.  Columns of the slab that no tile reads (beyond DT tiles) are written too.
struct Src32 {
    const float* ptr;
    int64_t sl;
};
template <int HD, int NS, int NT>
struct TriPlan {
    static constexpr int CH = HD / 8;
    static constexpr int chunks = Slab<HD>::chunks;
    static constexpr int total = NS * chunks;
    static constexpr int N = (total + NT - 1) / NT;
    static_assert(NT % chunks == 0 || chunks % NT == 0, "powers of two");
    static_assert(NT >= chunks || (NT / CH) % 16 == 0, "parts of a slab start at multiples of 16 rows");
    const float* src[N];
    int64_t adv[N];
    int row[N];
    int q0, j0, sh, col;
    bool shifted;
    F32x8 raw[N];

    __device__ __forceinline__ void init(int tid, int D, Src32 t0, Src32 t1, Src32 t2 = Src32{nullptr, 0}, Src32 t3 = Src32{nullptr, 0}) {
        q0 = tid % chunks;
        j0 = __builtin_amdgcn_readfirstlane(tid / chunks);
        const int c8 = 8 * ((q0 % CH) ^ swz<HD>(q0 / CH));
        col = piece_col(c8, D);
        sh = piece_shift(c8, D);
        shifted = D != HD;
        const Src32 ts[4] = {t0, t1, t2, t3};
        constexpr int SPI = NT >= chunks ? NT / chunks : 1;  // slabs from one position to the next
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int first = NT >= chunks ? SPI * i : i / (chunks / NT);
            const int j = NT >= chunks ? j0 + first : first;
            const int r = NT >= chunks ? q0 / CH : q0 / CH + (NT / CH) * (i % (chunks / NT));
            Src32 s = ts[first < NS ? first : 0];
#pragma unroll
            for (int k = 1; k < SPI; ++k)
                if (first + k < NS && j0 == k) s = ts[first + k < NS ? first + k : 0];
            row[i] = j < NS ? r : 1 << 30;  // a position beyond the last slab has no row
            src[i] = s.ptr + (int64_t)r * s.sl + col;
            adv[i] = 32 * s.sl;
        }
    }
    __device__ __forceinline__ void issue(int rows_left) {
        if (total % NT == 0 && rows_left >= kStageRows) {
#pragma unroll
            for (int i = 0; i < N; ++i) raw[i].load(src[i]);
        } else {
#pragma unroll
            for (int i = 0; i < N; ++i) {
                raw[i].zero();
                if (row[i] < rows_left) raw[i].load(src[i]);
            }
        }
#pragma unroll
        for (int i = 0; i < N; ++i) src[i] += adv[i];
    }
    // Whether elements of this thread's were some for the fp32 unit.
    __device__ __forceinline__ bool commit(elem_t* buffer) {
        constexpr int SE = Slab<HD>::elems;
        Met m;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            if (total % NT != 0 && row[i] >= kStageRows) continue;
            if (shifted) raw[i].shift(sh);
            const Op3 o = raw[i].split(m);
            constexpr int PPS = NT >= chunks ? 1 : chunks / NT;
            constexpr int SPI = NT >= chunks ? NT / chunks : 1;
            const int slab = NT >= chunks ? j0 + i * SPI : i / PPS;
            elem_t* at = buffer + 3 * slab * SE + 8 * q0 + (i % PPS) * 8 * NT;
#pragma unroll
            for (int u = 0; u < 3; ++u) *reinterpret_cast<u32x4*>(at + u * SE) = o.p[u];
        }
        return m.special();
    }
};

// Operands from the three slabs of a tensor.
template <int HD>
__device__ __forceinline__ Op3 rows3(const elem_t* slabs, int t, int c, int n, int g) {
    constexpr int SE = Slab<HD>::elems;
    return Op3{lds_a_rows16<HD>(slabs, t, c, n, g), lds_a_rows16<HD>(slabs + SE, t, c, n, g), lds_a_rows16<HD>(slabs + 2 * SE, t, c, n, g)};
}
template <int HD>
__device__ __forceinline__ Op3 cols3(const elem_t* slabs, int d0, int lane) {
    constexpr int SE = Slab<HD>::elems;
    return Op3{lds_a_tr16<HD>(slabs, d0, lane), lds_a_tr16<HD>(slabs + SE, d0, lane), lds_a_tr16<HD>(slabs + 2 * SE, d0, lane)};
}

// x[d] += Y'[d] tile, and z[d] += Y'[d] more; tile d of the columns from `col` on.
template <int HD, int DT>
__device__ __forceinline__ void tri_out(const elem_t* slabs, int lane, const Op3& tile, f32x4* x, const Op3& more, f32x4* z, int col = 0) {
#pragma unroll
    for (int d = 0; d < DT; ++d) {
        const Op3 a = cols3<HD>(slabs, col + 16 * d, lane);
        mfma6_onto(a, tile, x[d], a, more, z[d]);
    }
}
template <int HD, int DT>
__device__ __forceinline__ void tri_out(const elem_t* slabs, int lane, const Op3& tile, f32x4* x, int col = 0) {
#pragma unroll
    for (int d = 0; d + 1 < DT; d += 2)
        mfma6_onto(cols3<HD>(slabs, col + 16 * d, lane), tile, x[d], cols3<HD>(slabs, col + 16 * d + 16, lane), tile, x[d + 1]);
    if constexpr (DT % 2 != 0) {
        const Op3 a = cols3<HD>(slabs, col + 16 * DT - 16, lane);
        f32x4 t0 = {0.f, 0.f, 0.f, 0.f}, t1 = t0;
        t0 = Bf16::mfma16(a.p[2], tile.p[0], t0);
        t1 = Bf16::mfma16(a.p[1], tile.p[1], t1);
        t0 = Bf16::mfma16(a.p[0], tile.p[2], t0);
        t1 = Bf16::mfma16(a.p[1], tile.p[0], t1);
        t0 = Bf16::mfma16(a.p[0], tile.p[1], t0);
        x[DT - 1] = Bf16::mfma16(a.p[0], tile.p[0], x[DT - 1]);
        x[DT - 1] += t0 + t1;
    }
}

// Workgroups of NW waves, 16 owned rows each.  LDS: one or two buffers of a stage, a word per buffer that names the stage if
// it holds elements for the fp32 unit.
template <int HD, int NS>
struct TriSmem {
    static constexpr int buffer = 3 * NS * Slab<HD>::elems;
    static constexpr int buffers = 2 * buffer * (int)sizeof(elem_t) <= 128 * 1024 ? 2 : 1;
    static constexpr int flags = buffers * buffer * (int)sizeof(elem_t);
    static constexpr int bytes = flags + 16;
};

// The stages of the streamed axis: `compute(buffer, first row, special)` once for each.
template <int HD, int NS, int NT, typename F>
__device__ __forceinline__ void tri_walk(unsigned char* smem, TriPlan<HD, NS, NT>& plan, int L, F&& compute) {
    using SM = TriSmem<HD, NS>;
    elem_t* buffers = reinterpret_cast<elem_t*>(smem);
    volatile int* flag = reinterpret_cast<volatile int*>(smem + SM::flags);
    const int ns = (L + kStageRows - 1) / kStageRows;
    if (threadIdx.x < 2) flag[threadIdx.x] = 0;
    auto commit = [&](int i) {
        const int b = SM::buffers == 2 ? i & 1 : 0;
        if (__builtin_amdgcn_ballot_w64(plan.commit(buffers + b * SM::buffer)) != 0 && (threadIdx.x & 63) == 0) flag[b] = i + 1;
    };
    plan.issue(L);
    workgroup_barrier();  // the flags are cleared
    commit(0);
    if constexpr (SM::buffers == 2) {
        // Waves w and w + 4 share a SIMD.  One of them splits its share of the next stage ahead of its contractions, the other behind
        // them, so that the vector instructions of one run beside the matrix instructions of the other.
        const bool early = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) < NT / 128;
        auto next = [&](int i) {
            if (i + 1 < ns) commit(i + 1);
            if (i + 2 < ns) plan.issue(L - (i + 2) * kStageRows);
        };
        if (ns > 1) plan.issue(L - kStageRows);
#pragma unroll 1
        for (int i = 0; i < ns; ++i) {
            workgroup_barrier();  // the stage is there, the one before it consumed
            if (early) next(i);
            compute(buffers + (i & 1) * SM::buffer, i * kStageRows, __builtin_amdgcn_readfirstlane(flag[i & 1]) == i + 1);
            if (!early) next(i);
        }
    } else {
#pragma unroll 1
        for (int i = 0; i < ns; ++i) {
            if (i > 0) {
                workgroup_barrier();  // the last stage is consumed
                commit(i);
            }
            workgroup_barrier();  // this one is there
            if (i + 1 < ns) plan.issue(L - (i + 1) * kStageRows);
            compute(buffers, i * kStageRows, __builtin_amdgcn_readfirstlane(flag[0]) == i + 1);
        }
    }
}

template <int NW>
__device__ __forceinline__ F32Place tri_place(int blocks, int H) {
    F32Place w;
    w.part = 0;
    w.lane = threadIdx.x & 63;
    w.n = w.lane & 15;
    w.g = w.lane >> 4;
    const int id = xcd_linear_id((int)blockIdx.x, (int)gridDim.x);
    w.bh = id / blocks;
    w.b = w.bh / H;
    w.h = w.bh % H;
    w.row0 = (id % blocks) * 16 * NW + 16 * __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    return w;
}

// The lane's row of an output: registers j of tile d are columns 16 d + 4 g + j.
template <int DT>
__device__ __forceinline__ void tri_store(float* row, const f32x4* acc, float mul, int D, int g, bool valid) {
    if (!valid) return;
#pragma unroll
    for (int d = 0; d < DT; ++d) store_f32x4(reinterpret_cast<elem_t*>(row), acc[d] * mul, 16 * d + 4 * g, D);
}
template <int T>
__device__ __forceinline__ void zero_tiles(f32x4* acc) {
#pragma unroll
    for (int t = 0; t < T; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
}

// ---------------------------------------------------------------------------------------------
// Forward: O, TO, lse, mu, li (fwd_f32_kernel in sjvp_f32.hpp has the formulas).
template <int HD, int DT, bool JVP, int NW>
__global__ __launch_bounds__(64 * NW, HD == 32 ? 2 : NW / 4) void fwd_f32x3_kernel(const FwdParamsF32 p) {
    constexpr int NS = JVP ? 4 : 2, NT = 64 * NW, KC = (DT + 1) / 2, SE = Slab<HD>::elems;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const F32Place w = tri_place<NW>(p.blocks, p.H);
    const int qrow = w.row0 + w.n;
    const bool qvalid = qrow < p.Lq, active = w.row0 < p.Lq;
    const int64_t so = (int64_t)w.bh * p.Lr + qrow;  // rows below Lr exist (a multiple of 128)
    auto no_query = [&]() {  // the statistic rows of a group without queries get what a zero query row produces
        if (w.g != 0) return;
        p.lse[so] = fast_log2((float)p.Lk) * kLn2;
        if constexpr (JVP) p.mu[so] = 0.f;
        if (p.li) p.li[so] = (float)p.Lk;
    };
    if (w.row0 - 16 * (int)(threadIdx.x >> 6) >= p.Lq) return no_query();  // the whole workgroup
    const float *kb = p.k.head(w.b, w.h), *vb = p.v.head(w.b, w.h);
    const float *tkb = JVP ? p.tk.head(w.b, w.h) : nullptr, *tvb = JVP ? p.tv.head(w.b, w.h) : nullptr;
    const float* q_own = p.q.head(w.b, w.h) + (int64_t)qrow * p.q.sl;
    const float* tq_own = JVP ? p.tq.head(w.b, w.h) + (int64_t)qrow * p.tq.sl : nullptr;
    TriPlan<HD, NS, NT> plan;
    if constexpr (JVP) plan.init(threadIdx.x, p.D, Src32{kb, p.k.sl}, Src32{vb, p.v.sl}, Src32{tkb, p.tk.sl}, Src32{tvb, p.tv.sl});
    else plan.init(threadIdx.x, p.D, Src32{kb, p.k.sl}, Src32{vb, p.v.sl});
    Op3 q[KC], tq[KC];
    bool met;  // an element for the fp32 unit (wave-uniform)
    {
        F32x8 x[KC], tx[KC];
        own_load<KC>(x, q_own, w.g, p.D, qvalid);
        if constexpr (JVP) own_load<KC>(tx, tq_own, w.g, p.D, qvalid);
        Met m;
        own_cut<KC>(x, w.g, p.D);
        own_split<KC>(q, x, m);
        if constexpr (JVP) {
            own_cut<KC>(tx, w.g, p.D);
            own_split<KC>(tq, tx, m);
        }
        met = __builtin_amdgcn_ballot_w64(m.special()) != 0;
    }
    f32x4 acc[DT], tacc[DT];
    zero_tiles<DT>(acc);
    zero_tiles<DT>(tacc);
    const float sl2 = p.scale * kLog2e;
    float pt_most = 0.f;  // (the probabilities are at most 1, and one of a row is)
    float m_i = -INFINITY, l_i = 0.f, mu_i = 0.f;  // maximum (log2 units), exp-sum, sum p * S_dot of the lane's keys

    tri_walk<HD, NS, NT>(smem_raw, plan, p.Lk, [&](const elem_t* buf, int k0, bool stage_special) {
        met = met || stage_special;
        if (!active) return;
        f32x4 s[2], ts[2];
        zero_tiles<2>(s);
        zero_tiles<2>(ts);
        // the score contractions go first: a wave that is through with them has vector work that runs beside another's (row and
        // column kernel, without / with: B=8 H=12 L=500 D=32 85 and 117 / 78 and 113 us, B=8 H=8 L=256 D=64 36.2 and 45.9 / 35.2 and
        // 45.0, L=1024 688 and 957 / 685 and 944; the forward 68.0 / 67.6, 504 / 502)
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int c = 0; c < KC; ++c) {
            const Op3 a0 = rows3<HD>(buf, 0, c, w.n, w.g), a1 = rows3<HD>(buf, 1, c, w.n, w.g);
            mfma6(a0, q[c], s[0], a1, q[c], s[1]);
            if constexpr (JVP) {
                mfma6(a0, tq[c], ts[0], a1, tq[c], ts[1]);
                mfma6(rows3<HD>(buf + 6 * SE, 0, c, w.n, w.g), q[c], ts[0], rows3<HD>(buf + 6 * SE, 1, c, w.n, w.g), q[c], ts[1]);
            }
        }
        __builtin_amdgcn_s_setprio(0);
        s[0] *= sl2;
        s[1] *= sl2;
        if (k0 + kStageRows > p.Lk) {  // wave-uniform
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (k0 + 16 * t + 4 * w.g + j >= p.Lk) s[t][j] = -INFINITY;
        }
        const float mloc = fmaxf(fmaxf(fmaxf(s[0][0], s[0][1]), fmaxf(s[0][2], s[0][3])), fmaxf(fmaxf(s[1][0], s[1][1]), fmaxf(s[1][2], s[1][3])));
        if (__builtin_amdgcn_ballot_w64(mloc > m_i) != 0) {  // wave-uniform
            const float m_new = fmaxf(m_i, group_max(mloc));
            const float alpha = m_i < m_new ? fast_exp2(m_i - m_new) : 1.f;  // (both may be -inf, see below)
            m_i = m_new;
            l_i *= alpha;
            mu_i *= alpha;
#pragma unroll
            for (int d = 0; d < DT; ++d) {
                acc[d] *= alpha;
                if constexpr (JVP) tacc[d] *= alpha;
            }
        }
        // a row whose keys so far all score -inf has no maximum yet, and no probability
        const float base = m_i == -INFINITY ? 0.f : m_i;
        f32x4 pt[2];
        zero_tiles<2>(pt);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                s[t][j] = fast_exp2(s[t][j] - base);
                l_i += s[t][j];
                if constexpr (JVP) {
                    pt[t][j] = s[t][j] * (ts[t][j] * p.scale);
                    mu_i += pt[t][j];
                }
            }
        const Op3 pb = split_tiles(s[0], s[1]);
        Op3 ptb;
        if constexpr (JVP) ptb = split_tiles(pt[0], pt[1], pt_most);
        if constexpr (JVP) {
            tri_out<HD, DT>(buf + 3 * SE, w.lane, pb, acc, ptb, tacc);
            tri_out<HD, DT>(buf + 9 * SE, w.lane, pb, tacc);
        } else {
            tri_out<HD, DT>(buf + 3 * SE, w.lane, pb, acc);
        }
    });
    if (!active) return no_query();
    if constexpr (JVP) met = met || tiles_out_of_range(pt_most);
    if (__builtin_expect(met, 0)) return fwd_f32_wave<HD, JVP, 1, kColumnsCut>(p, w, nullptr, nullptr);
    const float l = group_sum(l_i), mu_un = group_sum(mu_i);
    const float inv_l = 1.0f / l, mu = mu_un * inv_l;
    if (w.g == 0) {
        // a padded query row (all-zero q, q_dot) yields log(Lk), 0, Lk by itself
        p.lse[so] = (m_i + fast_log2(l)) * kLn2;
        if constexpr (JVP) p.mu[so] = mu;
        if (p.li) p.li[so] = l;
    }
    tri_store<DT>(p.o.head(w.b, w.h) + (int64_t)qrow * p.o.sl, acc, inv_l, p.D, w.g, qvalid);
    if constexpr (JVP) {
        // TO = (sum (p S_dot) v + sum p v_dot - mu_un O_un) / l   (ryu_triton.py:274-275)
#pragma unroll
        for (int d = 0; d < DT; ++d) tacc[d] -= mu * acc[d];
        tri_store<DT>(p.to.head(w.b, w.h) + (int64_t)qrow * p.to.sl, tacc, inv_l, p.D, w.g, qvalid);
    }
}

// ---------------------------------------------------------------------------------------------
// Row-owned backward: dQ (, dQ_dot) and the row sums for the column-owned kernel.
template <int HD, int DT, bool HAS_DO, bool HAS_G, int NW>
__global__ __launch_bounds__(64 * NW, HD == 32 ? 2 : NW / 4) void bwd_row_f32x3_kernel(const BwdParamsF32 p) {
    constexpr int NS = HAS_G ? 4 : 2, NT = 64 * NW, KC = (DT + 1) / 2, SE = Slab<HD>::elems;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const F32Place w = tri_place<NW>(p.q_blocks, p.H);
    const int qrow = w.row0 + w.n;
    const bool qvalid = qrow < p.Lq, active = w.row0 < p.Lq;
    const float *kb = p.k.head(w.b, w.h), *vb = p.v.head(w.b, w.h);
    const float *tkb = HAS_G ? p.tk.head(w.b, w.h) : nullptr, *tvb = HAS_G ? p.tv.head(w.b, w.h) : nullptr;
    auto own_row = [&](const F32In& t) { return t.head(w.b, w.h) + (int64_t)qrow * t.sl; };
    const float *q_own = own_row(p.q), *tq_own = HAS_G ? own_row(p.tq) : nullptr;
    const float *g_own = HAS_G ? own_row(p.dTO) : nullptr, *do_own = HAS_DO ? own_row(p.dO) : nullptr;
    TriPlan<HD, NS, NT> plan;
    if constexpr (HAS_G) plan.init(threadIdx.x, p.D, Src32{kb, p.k.sl}, Src32{vb, p.v.sl}, Src32{tkb, p.tk.sl}, Src32{tvb, p.tv.sl});
    else plan.init(threadIdx.x, p.D, Src32{kb, p.k.sl}, Src32{vb, p.v.sl});
    Op3 q[KC], tq[KC], g[KC], dO[KC];
    float s4 = 0.f, s7d = 0.f;
    bool met;  // an element for the fp32 unit (wave-uniform)
    {
        F32x8 x[KC], o[KC];
        Met m;
        auto fetch = [&](F32x8* to, const float* row) {
            own_load<KC>(to, row, w.g, p.D, qvalid);
            own_cut<KC>(to, w.g, p.D);
        };
        fetch(o, own_row(p.o));
        if constexpr (HAS_DO) {
            fetch(x, do_own);
            s7d = own_dot<KC>(x, o, s7d);
            own_split<KC>(dO, x, m);
        }
        if constexpr (HAS_G) {
            fetch(x, g_own);
            s4 = own_dot<KC>(x, o, s4);
            fetch(o, own_row(p.to));
            s7d = own_dot<KC>(x, o, s7d);
            own_split<KC>(g, x, m);
            fetch(x, tq_own);
            own_split<KC>(tq, x, m);
        }
        fetch(x, q_own);
        own_split<KC>(q, x, m);
        met = __builtin_amdgcn_ballot_w64(m.special()) != 0;
    }
    s4 = group_sum(s4);
    s7d = group_sum(s7d);
    f32x4 dq[DT], dtq[DT];
    zero_tiles<DT>(dq);
    zero_tiles<DT>(dtq);
    const int64_t so = (int64_t)w.bh * p.Lr + qrow;
    float lse2 = 0.f, mu = 0.f;
    if (active) {  // (rows below Lr exist)
        lse2 = p.lse[so] * kLog2e;
        if constexpr (HAS_G) mu = p.mu[so];
        if (w.g == 0) {
            p.lse2[so] = lse2;
            p.s4[so] = s4;
            p.s7d[so] = s7d;
        }
    }
    const float sl2 = p.scale * kLog2e;
    float ds_most = 0.f, dts_most = 0.f;

    tri_walk<HD, NS, NT>(smem_raw, plan, p.Lk, [&](const elem_t* buf, int k0, bool stage_special) {
        met = met || stage_special;
        if (!active) return;
        f32x4 s[2], ts[2], wt[2], xy[2];
        zero_tiles<2>(s);
        zero_tiles<2>(ts);
        zero_tiles<2>(wt);
        zero_tiles<2>(xy);
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int c = 0; c < KC; ++c) {
            auto rows = [&](int tensor, int t) { return rows3<HD>(buf + 3 * tensor * SE, t, c, w.n, w.g); };
            const Op3 a0 = rows(0, 0), a1 = rows(0, 1);
            mfma6(a0, q[c], s[0], a1, q[c], s[1]);
            if constexpr (HAS_G) {
                mfma6(a0, tq[c], ts[0], a1, tq[c], ts[1]);
                mfma6(rows(2, 0), q[c], ts[0], rows(2, 1), q[c], ts[1]);
            }
            const Op3 v0 = rows(1, 0), v1 = rows(1, 1);
            if constexpr (HAS_DO) mfma6(v0, dO[c], xy[0], v1, dO[c], xy[1]);
            if constexpr (HAS_G) {
                mfma6(v0, g[c], wt[0], v1, g[c], wt[1]);
                mfma6(rows(3, 0), g[c], xy[0], rows(3, 1), g[c], xy[1]);
            }
        }
        __builtin_amdgcn_s_setprio(0);
        f32x4 ds[2], dts[2];
        zero_tiles<2>(dts);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float pj = fast_exp2(fmaf(s[t][j], sl2, -lse2));
                if constexpr (HAS_G) {
                    const float nn = fmaf(ts[t][j], p.scale, -mu);
                    dts[t][j] = pj * (wt[t][j] - s4);
                    ds[t][j] = fmaf(dts[t][j], nn, pj * (xy[t][j] - s7d));
                } else {
                    ds[t][j] = pj * (xy[t][j] - s7d);
                }
            }
        if (k0 + kStageRows > p.Lk) {  // keys that do not exist contribute nothing
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const bool kvalid = k0 + 16 * t + 4 * w.g + j < p.Lk;
                    ds[t][j] = kvalid ? ds[t][j] : 0.f;
                    dts[t][j] = kvalid ? dts[t][j] : 0.f;
                }
        }
        const Op3 dsb = split_tiles(ds[0], ds[1], ds_most);
        Op3 dtsb;
        if constexpr (HAS_G) dtsb = split_tiles(dts[0], dts[1], dts_most);
        if constexpr (HAS_G) {
            tri_out<HD, DT>(buf, w.lane, dsb, dq, dtsb, dtq);
            tri_out<HD, DT>(buf + 6 * SE, w.lane, dtsb, dq);
        } else {
            tri_out<HD, DT>(buf, w.lane, dsb, dq);
        }
    });
    if (!active) return;
    met = met || tiles_out_of_range(ds_most) || tiles_out_of_range(dts_most);
    if (__builtin_expect(met, 0)) return bwd_row_f32_wave<HD, HAS_DO, HAS_G, 1, kColumnsCut>(p, w, nullptr);
    tri_store<DT>(p.dq.head(w.b, w.h) + (int64_t)qrow * p.dq.sl, dq, p.scale, p.D, w.g, qvalid);
    if constexpr (HAS_G) tri_store<DT>(p.dtq.head(w.b, w.h) + (int64_t)qrow * p.dtq.sl, dtq, p.scale, p.D, w.g, qvalid);
}

// ---------------------------------------------------------------------------------------------
// The same with tangents at D > 64, by pairs of waves: four owned tensors in three parts and the accumulators are more registers than
// leave a second wave room on its SIMD.  The pair shares 16 owned rows; one wave owns two tensors o, o_dot and streams y1, y2 against them,
//     x1 = y1 o, x2 = y1 o_dot + y2 o,
// here q, q_dot against k, k_dot and G, dO against v, v_dot: three contractions of both.  They exchange what the other one's element-wise
// part needs through LDS.  dQ, dQ_dot need all of it: each wave takes half of their columns.  One wave per SIMD with everything / pairs:
// B=8 H=16 L=512 D=128 552 / 480 us, B=8 H=12 L=500 D=96 325 / 289, B=32 H=8 L=128 D=80 74 / 66.
constexpr int kPairs = 4;  // of a workgroup: 64 owned rows
template <int HD, int NS>
constexpr int pair_smem() { return TriSmem<HD, NS>::bytes + kPairs * 2 * 4 * 64 * (int)sizeof(f32x4); }

// Whether a wave of the pair met an element for the fp32 unit.
template <int HD, int NS>
__device__ __forceinline__ bool pair_met(unsigned char* smem, bool met, int wave, int lane) {
    volatile int* flag = reinterpret_cast<volatile int*>(smem + TriSmem<HD, NS>::bytes);
    workgroup_barrier();  // the last stage's tiles are read
    if (lane == 0) flag[wave] = met;
    workgroup_barrier();
    return __builtin_expect(met || __builtin_amdgcn_readfirstlane(flag[wave ^ kPairs]) != 0, 0);
}

// The forms of the pairs on the fp32 unit, for rows whose numbers the split does not hold: operands are read where they are used.
// Score-like tile: streamed rows (the lane's `row` of L) times the owned one.
template <int HD>
__device__ __forceinline__ f32x4 unit_dot(const BwdParamsF32& p, const F32Place& w, const F32In& rows, int row, int L, const F32In& own, int own_row,
                                          int own_L) {
    __builtin_amdgcn_sched_barrier(0);
    f32x4 a[HD / 16], b[HD / 16], c = {0.f, 0.f, 0.f, 0.f};
    f32_load_own<HD, false, true>(a, rows.head(w.b, w.h), rows.sl, row, L, p.D, w.g);
    f32_load_own<HD, false, true>(b, own.head(w.b, w.h), own.sl, own_row, own_L, p.D, w.g);
#pragma unroll
    for (int m = 0; m < HD / 16; ++m)
#pragma unroll
        for (int e = 0; e < 4; ++e) c = mfma_f32(a[m][e], b[m][e], c);
    return c;
}
// Output-side operand of a streamed row.
template <int HD>
__device__ __forceinline__ void unit_cols(float* y, const BwdParamsF32& p, const F32Place& w, const F32In& x, int row, int L) {
    __builtin_amdgcn_sched_barrier(0);
    f32_load_cols<HD, false, true>(y, x.head(w.b, w.h), x.sl, row, L, p.D, w.n);
    f32_cut_cols<HD, false, true>(y, p.D, w.n);
    f32_zero_unless<F32Cols<HD>::tiles>(y, row < L);
}

// dQ, dQ_dot of 16 rows.
template <int HD, bool HAS_DO>
__device__ __forceinline__ void bwd_row_f32_unit(const BwdParamsF32& p, const F32Place& w, float s4, float s7d) {
    constexpr int T = F32Cols<HD>::tiles;
    const int qrow = w.row0 + w.n;
    const bool qvalid = qrow < p.Lq;
    const int64_t so = (int64_t)w.bh * p.Lr + qrow;
    const float lse2 = p.lse[so] * kLog2e, mu = p.mu[so];
    f32x4 acc[T], tacc[T];
    zero_tiles<T>(acc);
    zero_tiles<T>(tacc);
#pragma unroll 1
    for (int k0 = 0; k0 < p.Lk; k0 += kF32Rows) {
        int own_row = qrow;  // read anew for every tile: kept through the loop, the owned rows are more registers than there are
        asm volatile("" : "+v"(own_row));
        auto dot = [&](const F32In& rows, const F32In& own) { return unit_dot<HD>(p, w, rows, k0 + w.n, p.Lk, own, own_row, p.Lq); };
        const f32x4 s = dot(p.k, p.q), ts = dot(p.k, p.tq) + dot(p.tk, p.q), wt = dot(p.v, p.dTO);
        f32x4 xy = dot(p.tv, p.dTO);
        if constexpr (HAS_DO) xy = dot(p.v, p.dO) + xy;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int row = k0 + 4 * w.g + j;
            const float pj = fast_exp2(fmaf(s[j], p.scale * kLog2e, -lse2));
            float dts = pj * (wt[j] - s4), ds = fmaf(dts, fmaf(ts[j], p.scale, -mu), pj * (xy[j] - s7d));
            dts = row < p.Lk ? dts : 0.f;
            ds = row < p.Lk ? ds : 0.f;
            float y[T];
            unit_cols<HD>(y, p, w, p.k, row, p.Lk);
#pragma unroll
            for (int t = 0; t < T; ++t) {
                acc[t] = mfma_f32(y[t], ds, acc[t]);
                tacc[t] = mfma_f32(y[t], dts, tacc[t]);
            }
            unit_cols<HD>(y, p, w, p.tk, row, p.Lk);
#pragma unroll
            for (int t = 0; t < T; ++t) acc[t] = mfma_f32(y[t], dts, acc[t]);
        }
    }
    f32_store<HD, false, 1>(nullptr, p.dq.head(w.b, w.h) + (int64_t)qrow * p.dq.sl, acc, p.scale, w, p.D, qvalid);
    f32_store<HD, false, 1>(nullptr, p.dtq.head(w.b, w.h) + (int64_t)qrow * p.dtq.sl, tacc, p.scale, w, p.D, qvalid);
}

template <int HD, int DT, bool HAS_DO>
__global__ __launch_bounds__(128 * kPairs, 2) void bwd_row_f32x3_pair_kernel(const BwdParamsF32 p) {
    constexpr int NS = 4, NT = 128 * kPairs, KC = (DT + 1) / 2, SE = Slab<HD>::elems, HT = DT / 2;
    static_assert(DT % 2 == 0, "half of the columns each");
    extern __shared__ __align__(16) unsigned char smem_raw[];
    F32Place w = tri_place<kPairs>(p.q_blocks, p.H);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), role = wave / kPairs;  // 0: k, 1: v
    w.row0 -= role * 16 * kPairs;
    f32x4* exchange = reinterpret_cast<f32x4*>(smem_raw + TriSmem<HD, NS>::bytes) + (wave % kPairs) * 512 + w.lane;
    f32x4 *mine = exchange + 256 * role, *other = exchange + 256 * (1 - role);
    const int qrow = w.row0 + w.n;
    const bool qvalid = qrow < p.Lq, active = w.row0 < p.Lq;
    TriPlan<HD, NS, NT> plan;
    {
        auto src = [&](const F32In& t) { return Src32{t.head(w.b, w.h), t.sl}; };
        plan.init(threadIdx.x, p.D, src(p.k), src(p.v), src(p.tk), src(p.tv));
    }
    const int64_t so = (int64_t)w.bh * p.Lr + qrow;  // rows below Lr exist
    Op3 own[KC], town[KC];
    float c1 = 0.f, c2 = 0.f;  // of the row: log-sum-exp (log2 units) and mu, or s4 and s7d
    bool met;                  // an element for the fp32 unit (wave-uniform)
    {
        F32x8 x[KC], o[KC];
        Met m;
        auto fetch = [&](F32x8* to, const F32In& t) {
            own_load<KC>(to, t.head(w.b, w.h) + (int64_t)qrow * t.sl, w.g, p.D, qvalid);
            own_cut<KC>(to, w.g, p.D);
        };
        if (role == 0) {
            fetch(x, p.q);
            own_split<KC>(own, x, m);
            fetch(x, p.tq);
            own_split<KC>(town, x, m);
            if (active) {
                c1 = p.lse[so] * kLog2e;
                c2 = p.mu[so];
                if (w.g == 0) p.lse2[so] = c1;
            }
        } else {
            fetch(o, p.o);
            if constexpr (HAS_DO) {
                fetch(x, p.dO);
                c2 = own_dot<KC>(x, o, c2);
                own_split<KC>(town, x, m);
            }
            fetch(x, p.dTO);
            c1 = own_dot<KC>(x, o, c1);
            fetch(o, p.to);
            c2 = own_dot<KC>(x, o, c2);
            own_split<KC>(own, x, m);
            c1 = group_sum(c1);
            c2 = group_sum(c2);
            if (active && w.g == 0) {
                p.s4[so] = c1;
                p.s7d[so] = c2;
            }
        }
        met = __builtin_amdgcn_ballot_w64(m.special()) != 0;
    }
    f32x4 dq[HT], dtq[HT];
    zero_tiles<HT>(dq);
    zero_tiles<HT>(dtq);
    const int col = 16 * HT * role;
    const float sl2 = p.scale * kLog2e;
    float ds_most = 0.f, dts_most = 0.f;

    tri_walk<HD, NS, NT>(smem_raw, plan, p.Lk, [&](const elem_t* buf, int k0, bool stage_special) {
        met = met || stage_special;
        const elem_t *y1 = buf + role * 3 * SE, *y2 = y1 + 6 * SE;
        f32x4 x1[2], x2[2];
        zero_tiles<2>(x1);
        zero_tiles<2>(x2);
        if (active) {
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int c = 0; c < KC; ++c) {
                const Op3 a0 = rows3<HD>(y1, 0, c, w.n, w.g), a1 = rows3<HD>(y1, 1, c, w.n, w.g);
                mfma6(a0, own[c], x1[0], a1, own[c], x1[1]);
                if (HAS_DO || role == 0) mfma6(a0, town[c], x2[0], a1, town[c], x2[1]);
                mfma6(rows3<HD>(y2, 0, c, w.n, w.g), own[c], x2[0], rows3<HD>(y2, 1, c, w.n, w.g), own[c], x2[1]);
            }
            __builtin_amdgcn_s_setprio(0);
            // P and N, or W - s4 and XY - s7d
#pragma unroll
            for (int t = 0; t < 2; ++t) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (role == 0) {
                        x1[t][j] = fast_exp2(fmaf(x1[t][j], sl2, -c1));
                        x2[t][j] = fmaf(x2[t][j], p.scale, -c2);
                    } else {
                        x1[t][j] -= c1;
                        x2[t][j] -= c2;
                    }
                mine[64 * t] = x1[t];
                mine[64 * (2 + t)] = x2[t];
            }
        }
        workgroup_barrier();
        if (!active) return;
        f32x4 ds[2], dts[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const f32x4 z1 = other[64 * t], z2 = other[64 * (2 + t)];
            const f32x4 pr = role ? z1 : x1[t], nn = role ? z2 : x2[t], wt = role ? x1[t] : z1, xy = role ? x2[t] : z2;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                dts[t][j] = pr[j] * wt[j];
                ds[t][j] = fmaf(dts[t][j], nn[j], pr[j] * xy[j]);
            }
        }
        if (k0 + kStageRows > p.Lk) {  // keys that do not exist contribute nothing
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const bool kvalid = k0 + 16 * t + 4 * w.g + j < p.Lk;
                    ds[t][j] = kvalid ? ds[t][j] : 0.f;
                    dts[t][j] = kvalid ? dts[t][j] : 0.f;
                }
        }
        const Op3 dsb = split_tiles(ds[0], ds[1], ds_most), dtsb = split_tiles(dts[0], dts[1], dts_most);
        tri_out<HD, HT>(buf, w.lane, dsb, dq, dtsb, dtq, col);
        tri_out<HD, HT>(buf + 6 * SE, w.lane, dtsb, dq, col);
    });
    met = met || tiles_out_of_range(ds_most) || tiles_out_of_range(dts_most);
    if (pair_met<HD, NS>(smem_raw, met, wave, w.lane)) {
        if (active && role == 1) bwd_row_f32_unit<HD, HAS_DO>(p, w, c1, c2);
        return;
    }
    if (!active) return;
    tri_store<HT>(p.dq.head(w.b, w.h) + (int64_t)qrow * p.dq.sl + col, dq, p.scale, p.D - col, w.g, qvalid);
    tri_store<HT>(p.dtq.head(w.b, w.h) + (int64_t)qrow * p.dtq.sl + col, dtq, p.scale, p.D - col, w.g, qvalid);
}

// ---------------------------------------------------------------------------------------------
// Column-owned backward: dK, dV (, dK_dot, dV_dot).
template <int HD, int DT, bool HAS_DO, bool HAS_G, int NW>
__global__ __launch_bounds__(64 * NW, HD == 32 ? 2 : NW / 4) void bwd_col_f32x3_kernel(const BwdParamsF32 p) {
    constexpr int NS = HAS_G ? (HAS_DO ? 4 : 3) : 2, NT = 64 * NW, KC = (DT + 1) / 2, SE = Slab<HD>::elems;
    // slabs: Q, then Q_dot, G (HAS_G), then dO (HAS_DO)
    constexpr int kTq = 3, kG = 6, kDo = HAS_G ? 9 : 3;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const F32Place w = tri_place<NW>(p.k_blocks, p.H);
    const int krow = w.row0 + w.n;
    const bool kvalid = krow < p.Lk, active = w.row0 < p.Lk;
    const float* qb = p.q.head(w.b, w.h);
    const float* tqb = HAS_G ? p.tq.head(w.b, w.h) : nullptr;
    const float* gb = HAS_G ? p.dTO.head(w.b, w.h) : nullptr;
    const float* dob = HAS_DO ? p.dO.head(w.b, w.h) : nullptr;
    auto own_row = [&](const F32In& t) { return t.head(w.b, w.h) + (int64_t)krow * t.sl; };
    const float *k_own = own_row(p.k), *v_own = own_row(p.v);
    const float *tk_own = HAS_G ? own_row(p.tk) : nullptr, *tv_own = HAS_G ? own_row(p.tv) : nullptr;
    TriPlan<HD, NS, NT> plan;
    if constexpr (HAS_G && HAS_DO) plan.init(threadIdx.x, p.D, Src32{qb, p.q.sl}, Src32{tqb, p.tq.sl}, Src32{gb, p.dTO.sl}, Src32{dob, p.dO.sl});
    else if constexpr (HAS_G) plan.init(threadIdx.x, p.D, Src32{qb, p.q.sl}, Src32{tqb, p.tq.sl}, Src32{gb, p.dTO.sl});
    else plan.init(threadIdx.x, p.D, Src32{qb, p.q.sl}, Src32{dob, p.dO.sl});
    Op3 k[KC], v[KC], tk[KC], tv[KC];
    bool met;  // an element for the fp32 unit (wave-uniform)
    {
        F32x8 x[KC];
        Met m;
        auto fetch = [&](Op3* to, const float* row) {
            own_load<KC>(x, row, w.g, p.D, kvalid);
            own_cut<KC>(x, w.g, p.D);
            own_split<KC>(to, x, m);
        };
        fetch(k, k_own);
        fetch(v, v_own);
        if constexpr (HAS_G) {
            fetch(tk, tk_own);
            fetch(tv, tv_own);
        }
        met = __builtin_amdgcn_ballot_w64(m.special()) != 0;
    }
    f32x4 dk[DT], dv[DT], dtk[DT], dtv[DT];
    zero_tiles<DT>(dk);
    zero_tiles<DT>(dv);
    zero_tiles<DT>(dtk);
    zero_tiles<DT>(dtv);
    const int64_t so = (int64_t)w.bh * p.Lr + 4 * w.g;  // rows below Lr exist in every statistic
    const float sl2 = p.scale * kLog2e;
    float ds_most = 0.f, dts_most = 0.f, pr_most = 0.f, pn_most = 0.f;

    tri_walk<HD, NS, NT>(smem_raw, plan, p.Lq, [&](const elem_t* buf, int q0, bool stage_special) {
        met = met || stage_special;
        if (!active) return;
        f32x4 s[2], ts[2], wt[2], xy[2];
        zero_tiles<2>(s);
        zero_tiles<2>(ts);
        zero_tiles<2>(wt);
        zero_tiles<2>(xy);
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int c = 0; c < KC; ++c) {
            auto rows = [&](int slab, int t) { return rows3<HD>(buf + slab * SE, t, c, w.n, w.g); };
            const Op3 a0 = rows(0, 0), a1 = rows(0, 1);
            mfma6(a0, k[c], s[0], a1, k[c], s[1]);
            if constexpr (HAS_G) {
                mfma6(a0, tk[c], ts[0], a1, tk[c], ts[1]);
                mfma6(rows(kTq, 0), k[c], ts[0], rows(kTq, 1), k[c], ts[1]);
                const Op3 g0 = rows(kG, 0), g1 = rows(kG, 1);
                mfma6(g0, v[c], wt[0], g1, v[c], wt[1]);
                mfma6(g0, tv[c], xy[0], g1, tv[c], xy[1]);
            }
            if constexpr (HAS_DO) mfma6(rows(kDo, 0), v[c], xy[0], rows(kDo, 1), v[c], xy[1]);
        }
        __builtin_amdgcn_s_setprio(0);
        f32x4 pr[2], pn[2], ds[2], dts[2];
        zero_tiles<2>(pn);
        zero_tiles<2>(dts);
        const bool ragged = q0 + kStageRows > p.Lq;  // wave-uniform
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int64_t at = so + q0 + 16 * t;
            const f32x4 lse2 = *reinterpret_cast<const f32x4*>(p.lse2 + at);
            const f32x4 s7d = *reinterpret_cast<const f32x4*>(p.s7d + at);
            f32x4 mu = {0.f, 0.f, 0.f, 0.f}, s4 = mu;
            if constexpr (HAS_G) {
                s4 = *reinterpret_cast<const f32x4*>(p.s4 + at);
                mu = *reinterpret_cast<const f32x4*>(p.mu + at);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float pj = kvalid ? fast_exp2(fmaf(s[t][j], sl2, -lse2[j])) : 0.f;  // a padded key contributes nothing
                pr[t][j] = pj;
                if constexpr (HAS_G) {
                    const float nn = fmaf(ts[t][j], p.scale, -mu[j]);
                    dts[t][j] = pj * (wt[t][j] - s4[j]);
                    ds[t][j] = fmaf(dts[t][j], nn, pj * (xy[t][j] - s7d[j]));
                    pn[t][j] = pj * nn;
                } else {
                    ds[t][j] = pj * (xy[t][j] - s7d[j]);
                }
            }
            if (ragged) {  // nor does a query that does not exist
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const bool qvalid = q0 + 16 * t + 4 * w.g + j < p.Lq;
                    pr[t][j] = qvalid ? pr[t][j] : 0.f;
                    pn[t][j] = qvalid ? pn[t][j] : 0.f;
                    ds[t][j] = qvalid ? ds[t][j] : 0.f;
                    dts[t][j] = qvalid ? dts[t][j] : 0.f;
                }
            }
        }
        {
            const Op3 dsb = split_tiles(ds[0], ds[1], ds_most);
            Op3 dtsb;
            if constexpr (HAS_G) dtsb = split_tiles(dts[0], dts[1], dts_most);
            if constexpr (HAS_G) {
                tri_out<HD, DT>(buf, w.lane, dsb, dk, dtsb, dtk);
                tri_out<HD, DT>(buf + kTq * SE, w.lane, dtsb, dk);
            } else {
                tri_out<HD, DT>(buf, w.lane, dsb, dk);
            }
        }
        {
            const Op3 prb = split_tiles(pr[0], pr[1], pr_most);
            Op3 pnb;
            if constexpr (HAS_G) pnb = split_tiles(pn[0], pn[1], pn_most);
            if constexpr (HAS_G) tri_out<HD, DT>(buf + kG * SE, w.lane, pnb, dv, prb, dtv);
            if constexpr (HAS_DO) tri_out<HD, DT>(buf + kDo * SE, w.lane, prb, dv);
        }
    });
    if (!active) return;
    met = met || tiles_out_of_range(ds_most) || tiles_out_of_range(pr_most) || tiles_out_of_range(dts_most) || tiles_out_of_range(pn_most);
    if (__builtin_expect(met, 0)) return bwd_col_f32_wave<HD, HAS_DO, HAS_G, 1, kColumnsCut>(p, w, nullptr);
    tri_store<DT>(p.dk.head(w.b, w.h) + (int64_t)krow * p.dk.sl, dk, p.scale, p.D, w.g, kvalid);
    tri_store<DT>(p.dv.head(w.b, w.h) + (int64_t)krow * p.dv.sl, dv, 1.0f, p.D, w.g, kvalid);
    if constexpr (HAS_G) {
        tri_store<DT>(p.dtk.head(w.b, w.h) + (int64_t)krow * p.dtk.sl, dtk, p.scale, p.D, w.g, kvalid);
        tri_store<DT>(p.dtv.head(w.b, w.h) + (int64_t)krow * p.dtv.sl, dtv, 1.0f, p.D, w.g, kvalid);
    }
}

// ---------------------------------------------------------------------------------------------
// By pairs of waves, as the row kernel's: one wave owns k, k_dot and the gradients of them, the other v, v_dot and theirs.  With
// t1, t2 the tiles (dS_dot, dS or P, P_dot) the output contractions are three of both waves too, and nothing is done twice:
//     d(o_dot) = t1^T y1, d(o) = t2^T y1 + t1^T y2.
// The two gradients of a wave.
template <int HD, bool HAS_DO>
__device__ __forceinline__ void bwd_col_f32_half(const BwdParamsF32& p, const F32Place& w, int role) {
    constexpr int T = F32Cols<HD>::tiles;
    const int krow = w.row0 + w.n;
    const bool kvalid = krow < p.Lk;
    f32x4 acc[T], tacc[T];
    zero_tiles<T>(acc);
    zero_tiles<T>(tacc);
    const int64_t so = (int64_t)w.bh * p.Lr + 4 * w.g;
#pragma unroll 1
    for (int q0 = 0; q0 < p.Lq; q0 += kF32Rows) {
        int own_row = krow;  // read anew for every tile: kept through the loop, the owned rows are more registers than there are
        asm volatile("" : "+v"(own_row));
        auto dot = [&](const F32In& rows, const F32In& own) { return unit_dot<HD>(p, w, rows, q0 + w.n, p.Lq, own, own_row, p.Lk); };
        const f32x4 s = dot(p.q, p.k), ts = dot(p.tq, p.k) + dot(p.q, p.tk);
        f32x4 wt = {0.f, 0.f, 0.f, 0.f}, xy = wt, t1, t2;
        if (role == 0) {
            wt = dot(p.dTO, p.v);
            xy = dot(p.dTO, p.tv);
            if constexpr (HAS_DO) xy = dot(p.dO, p.v) + xy;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t at = so + q0 + j;
            const float pj = kvalid ? fast_exp2(fmaf(s[j], p.scale * kLog2e, -p.lse2[at])) : 0.f;
            const float nn = fmaf(ts[j], p.scale, -p.mu[at]), dts = pj * (wt[j] - p.s4[at]);
            t1[j] = role ? pj : dts;
            t2[j] = role ? pj * nn : fmaf(dts, nn, pj * (xy[j] - p.s7d[at]));
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int row = q0 + 4 * w.g + j;
            const bool qvalid = row < p.Lq;
            t1[j] = qvalid ? t1[j] : 0.f;
            t2[j] = qvalid ? t2[j] : 0.f;
            float y[T];
            auto cols = [&](const F32In& x) { unit_cols<HD>(y, p, w, x, row, p.Lq); };
            if (role) cols(p.dTO);
            else cols(p.q);
#pragma unroll
            for (int t = 0; t < T; ++t) {
                acc[t] = mfma_f32(y[t], t2[j], acc[t]);
                tacc[t] = mfma_f32(y[t], t1[j], tacc[t]);
            }
            if (HAS_DO || role == 0) {
                if (role) cols(p.dO);
                else cols(p.tq);
#pragma unroll
                for (int t = 0; t < T; ++t) acc[t] = mfma_f32(y[t], t1[j], acc[t]);
            }
        }
    }
    const F32Out &d = role ? p.dv : p.dk, &td = role ? p.dtv : p.dtk;
    const float mul = role ? 1.0f : p.scale;
    f32_store<HD, false, 1>(nullptr, d.head(w.b, w.h) + (int64_t)krow * d.sl, acc, mul, w, p.D, kvalid);
    f32_store<HD, false, 1>(nullptr, td.head(w.b, w.h) + (int64_t)krow * td.sl, tacc, mul, w, p.D, kvalid);
}

template <int HD, int DT, bool HAS_DO>
__global__ __launch_bounds__(128 * kPairs, 2) void bwd_col_f32x3_pair_kernel(const BwdParamsF32 p) {
    constexpr int NS = HAS_DO ? 4 : 3, NT = 128 * kPairs, KC = (DT + 1) / 2, SE = Slab<HD>::elems;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    F32Place w = tri_place<kPairs>(p.k_blocks, p.H);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), role = wave / kPairs;  // 0: k, 1: v
    w.row0 -= role * 16 * kPairs;
    f32x4* exchange = reinterpret_cast<f32x4*>(smem_raw + TriSmem<HD, NS>::bytes) + (wave % kPairs) * 512 + w.lane;
    f32x4 *mine = exchange + 256 * role, *other = exchange + 256 * (1 - role);
    const int krow = w.row0 + w.n;
    const bool kvalid = krow < p.Lk, active = w.row0 < p.Lk;
    TriPlan<HD, NS, NT> plan;
    {
        auto src = [&](const F32In& t) { return Src32{t.head(w.b, w.h), t.sl}; };
        if constexpr (HAS_DO) plan.init(threadIdx.x, p.D, src(p.q), src(p.tq), src(p.dTO), src(p.dO));
        else plan.init(threadIdx.x, p.D, src(p.q), src(p.tq), src(p.dTO));
    }
    Op3 own[KC], town[KC];
    bool met;  // an element for the fp32 unit (wave-uniform)
    {
        F32x8 x[KC];
        Met m;
        auto fetch = [&](Op3* to, const F32In& t) {
            own_load<KC>(x, t.head(w.b, w.h) + (int64_t)krow * t.sl, w.g, p.D, kvalid);
            own_cut<KC>(x, w.g, p.D);
            own_split<KC>(to, x, m);
        };
        fetch(own, role ? p.v : p.k);
        fetch(town, role ? p.tv : p.tk);
        met = __builtin_amdgcn_ballot_w64(m.special()) != 0;
    }
    f32x4 acc[DT], tacc[DT];
    zero_tiles<DT>(acc);
    zero_tiles<DT>(tacc);
    const int64_t so = (int64_t)w.bh * p.Lr + 4 * w.g;  // rows below Lr exist in every statistic
    const float sl2 = p.scale * kLog2e;
    float t1_most = 0.f, t2_most = 0.f;

    tri_walk<HD, NS, NT>(smem_raw, plan, p.Lq, [&](const elem_t* buf, int q0, bool stage_special) {
        met = met || stage_special;
        const elem_t *y1 = buf + role * 6 * SE, *y2 = y1 + 3 * SE;
        const bool has_y2 = HAS_DO || role == 0;
        f32x4 x1[2], x2[2];
        zero_tiles<2>(x1);
        zero_tiles<2>(x2);
        if (active) {
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int c = 0; c < KC; ++c) {
                const Op3 a0 = rows3<HD>(y1, 0, c, w.n, w.g), a1 = rows3<HD>(y1, 1, c, w.n, w.g);
                mfma6(a0, own[c], x1[0], a1, own[c], x1[1]);
                mfma6(a0, town[c], x2[0], a1, town[c], x2[1]);
                if (has_y2) mfma6(rows3<HD>(y2, 0, c, w.n, w.g), own[c], x2[0], rows3<HD>(y2, 1, c, w.n, w.g), own[c], x2[1]);
            }
            __builtin_amdgcn_s_setprio(0);
            // x1, x2 become P and N, or W - s4 and XY - s7d; what the other wave needs of them goes to it
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const int64_t at = so + q0 + 16 * t;
                const f32x4 c1 = *reinterpret_cast<const f32x4*>((role ? p.s4 : p.lse2) + at);
                const f32x4 c2 = *reinterpret_cast<const f32x4*>((role ? p.s7d : p.mu) + at);
                f32x4 second;
                if (role == 0) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        // a key or a query that does not exist contributes nothing
                        const bool valid = kvalid && q0 + 16 * t + 4 * w.g + j < p.Lq;
                        const float pj = valid ? fast_exp2(fmaf(x1[t][j], sl2, -c1[j])) : 0.f;
                        const float nn = fmaf(x2[t][j], p.scale, -c2[j]);
                        x1[t][j] = pj;
                        x2[t][j] = nn;
                        second[j] = valid ? pj * nn : 0.f;
                    }
                } else {
                    x1[t] -= c1;
                    x2[t] -= c2;
                    second = x2[t];
                }
                mine[64 * t] = x1[t];
                mine[64 * (2 + t)] = second;
            }
        }
        workgroup_barrier();
        if (!active) return;
        f32x4 t1[2], t2[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            t1[t] = other[64 * t];
            t2[t] = other[64 * (2 + t)];
            if (role == 0)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const bool valid = kvalid && q0 + 16 * t + 4 * w.g + j < p.Lq;
                    const float dts = x1[t][j] * t1[t][j], ds = fmaf(dts, x2[t][j], x1[t][j] * t2[t][j]);
                    t1[t][j] = valid ? dts : 0.f;
                    t2[t][j] = valid ? ds : 0.f;
                }
        }
        const Op3 b1 = split_tiles(t1[0], t1[1], t1_most), b2 = split_tiles(t2[0], t2[1], t2_most);
        tri_out<HD, DT>(y1, w.lane, b2, acc, b1, tacc);
        if (has_y2) tri_out<HD, DT>(y2, w.lane, b1, acc);
    });
    met = met || tiles_out_of_range(t1_most) || tiles_out_of_range(t2_most);
    const bool unit = pair_met<HD, NS>(smem_raw, met, wave, w.lane);
    if (!active) return;
    if (unit) return bwd_col_f32_half<HD, HAS_DO>(p, w, role);
    const F32Out &d = role ? p.dv : p.dk, &td = role ? p.dtv : p.dtk;
    const float mul = role ? 1.0f : p.scale;
    tri_store<DT>(d.head(w.b, w.h) + (int64_t)krow * d.sl, acc, mul, p.D, w.g, kvalid);
    tri_store<DT>(td.head(w.b, w.h) + (int64_t)krow * td.sl, tacc, mul, p.D, w.g, kvalid);
}

}  // namespace sjvp
