// fp32 mode of the attention-JVP path (gfx950): fp32 tensors in and out, every product, sum and
// exponential in fp32.  This is the correctness mode of the library (the reference's fp32 math path,
// semicat/jvp_utils/ryu_triton.py:426-454, meets 1e-5 against fp64; the 16-bit kernels cannot).
//
// All contractions run on v_mfma_f32_16x16x4_f32 (full fp32 products and sums):
//     C[y][x] += sum_k A[y][k] B[k][x],  A: lane l holds row y = l % 16, k = l / 16;  B: column x = l % 16, same k;
//     C: lane l holds column x = l % 16 and, in register j < 4, row y = 4 (l/16) + j.
// A wavefront owns 16 rows of one sequence axis (x) and walks over the other (y) in tiles of 16.
//   * Score-like tiles: element e of the lane's float4 at columns 16 m + 4 (l/16) of a row is step (m, e) of
//     the contraction, on both sides: the k order is permuted, but equally for A and B, and one 16-byte load
//     feeds four matrix instructions.  The tile's registers are rows y = 4 (l/16) + j of column x, so row
//     statistics are per-lane scalars and ...
//   * ... output contractions OUT^T[d][x] += sum_y Y[y][d] T[y][x] take register j of the tile as the B operand
//     (k = l/16 stands for y = 4 (l/16) + j) and, as A, element e of the float4 at columns 4 (l%16) of row
//     y: sub-tile e of the output holds columns d = 4 c + e, and a lane ends up with 16 consecutive columns of
//     output row x.  No shuffle, no LDS, no transposition.
//
// Problems that fill the chip go to the kernels of sjvp_f32x3.hpp (the rule is in sjvp_f32.hip); these serve the smaller ones, short
// axes, and waves that hold numbers which those cannot take.
//
// What bounds it: the matrix pipe (157 TFLOP/s in fp32), once a wave's operand loads are out of its way.  A
// 16-byte load serves 4 to 8 matrix instructions of 32 cycles each, so the operands come straight from global
// memory (L1 / L2: at most 21 bytes per clock and CU at D = 64, where the L1 delivers 64) and the loops have no
// barrier; the loads of a tile are issued a whole contraction ahead of their use (f32_walk), for which the
// backward kernels take the registers of one wave per SIMD (two waves of 256 registers with the same
// prefetch spilled or waited: row-owned kernel 2104 against 1560 us, column-owned 2340 against 1922, at B=8 H=16
// L=1024 D=64; without the prefetch, two waves, 3713 for both).
//
// SPLIT > 1 (problems with few rows): the SPLIT waves of a workgroup share ONE group of 16 owned rows and take
// every SPLIT-th tile each; their partial sums are added in LDS at the end, in a fixed order.  SPLIT = 1: four
// waves, each with a group of its own.  (SPLIT = 8 measured no faster: 63.5 against 58.5 us at B=2 H=4 L=256.)
//
// Measured, forward + backward, the earlier form on the vector ALUs / this one: B=2 H=4 L=256 D=64 333 / 51 us; B=64
// H=12 L=128 D=64 901 / 525 us; B=8 H=16 L=1024 D=64 8.80 / 4.50 ms (103 TFLOP/s of executed products);
// B=8 H=16 L=512 D=128 7.15 / 2.54 ms.
#pragma once
#include "sjvp_w16.hpp"

namespace sjvp {

constexpr int kF32Waves = 4;
constexpr int kF32Threads = 64 * kF32Waves;
constexpr int kF32Rows = 16;  // rows of one wave's tile, owned and streamed

struct F32In {
    const float* ptr;
    int64_t sb, sh, sl;
    __device__ __forceinline__ const float* head(int b, int h) const { return ptr + b * sb + h * sh; }
};
struct F32Out {
    float* ptr;
    int64_t sb, sh, sl;
    __device__ __forceinline__ float* head(int b, int h) const { return ptr + b * sb + h * sh; }
};

struct FwdParamsF32 {
    F32In q, k, v, tq, tk, tv;
    F32Out o, to;
    float* lse;
    float* mu;
    float* li;  // may be null
    int H, Lq, Lk, D, Lr;
    int blocks;  // workgroups per (batch, head) pair
    float scale;
};

struct BwdParamsF32 {
    F32In q, k, v, tq, tk, tv, o, to, dO, dTO;
    F32Out dq, dk, dv, dtq, dtk, dtv;
    const float* lse;
    const float* mu;
    float* lse2;  // workspace [B*H][Lr]
    float* s4;
    float* s7d;
    int H, Lq, Lk, D, Lr;
    int q_blocks, k_blocks;  // workgroups per (batch, head) pair of the row-owned, column-owned launch
    float scale;
};

__device__ __forceinline__ f32x4 mfma_f32(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Where a wave works: its (batch, head) pair, its 16 owned rows and its place in the split.
struct F32Place {
    int b, h, bh, row0, part, lane, n, g;
};
template <int SPLIT>
__device__ __forceinline__ F32Place f32_place(int blocks, int H) {
    F32Place w;
    w.lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    w.n = w.lane & 15;
    w.g = w.lane >> 4;
    // the workgroups of one pair, which stream the same rows, run on one XCD
    const int id = xcd_linear_id((int)blockIdx.x, (int)gridDim.x);
    w.bh = id / blocks;
    w.b = w.bh / H;
    w.h = w.bh % H;
    w.row0 = (id % blocks) * (SPLIT > 1 ? kF32Rows : kF32Rows * kF32Waves) + (SPLIT > 1 ? 0 : wave * kF32Rows);
    w.part = SPLIT > 1 ? wave : 0;
    return w;
}

// How the columns of a row fill the head dimension HD that a kernel is compiled for.  An instance each: with the forms in
// one kernel the registers of the cutting one spill into the loop of the one that has nothing to cut (backward at D = 128
// 8 % longer).  Forward + backward at B=64 H=12 L=128, with single loads and the selects at the load / as here: D = 65 3396 /
// 1072 us, 127 4675 / 1138, 68 1567 / 977, 64 off the 16-byte grid 722 / 511.
enum F32Columns {
    kColumnsAll,    // D == HD
    kColumnsWhole,  // HD / 2 <= D < HD, D % 4 == 0: a piece of W columns exists or does not
    kColumnsCut,    // HD / 2 <= D < HD
};

// W consecutive elements from column `col` of a row, as one load (fp32 needs no more than 4-byte alignment for it).
// MASK: columns >= D become zero in two steps, so that the second one can be put where the load has arrived
// anyway.  f32_ld reads W elements of the row in any case: a piece beyond D stands at column 0 (VEC: D % 4 == 0), or
// every piece that does not lie below D whole is read as the row's last W elements.  f32_cut moves what
// exists of the piece to its place and zeroes the rest.
template <int W>
struct F32Vec {
    typedef float type __attribute__((ext_vector_type(W), aligned(4)));
};
template <int W, bool VEC, bool MASK>
__device__ __forceinline__ void f32_ld(float* x, const float* row, int col, int D) {
    const int at = !MASK ? col : VEC ? (col < D ? col : 0) : min(col, D - W);  // D >= 16
    const typename F32Vec<W>::type v = *reinterpret_cast<const typename F32Vec<W>::type*>(row + at);
#pragma unroll
    for (int e = 0; e < W; ++e) x[e] = v[e];
}
template <int W, bool VEC>
__device__ __forceinline__ void f32_cut(float* x, int col, int D) {
    const int n = D - col;  // columns of the piece that exist, W or more: all
#pragma unroll
    for (int e = 0; e < W; ++e) {
        if constexpr (VEC) {
            x[e] = n > 0 ? x[e] : 0.f;
        } else {
            float y = n >= W ? x[e] : 0.f;  // column col + e was read into x[e + W - n]
#pragma unroll
            for (int t = e + 1; t < W; ++t) y = n == W - (t - e) ? x[t] : y;
            x[e] = y;
        }
    }
}
__device__ __forceinline__ const float* f32_row(const float* base, int64_t sl, int row, int L) {
    return base + (int64_t)(row < L ? row : L - 1) * sl;  // rows beyond L stand for the last one: the caller masks
}

// Score-side operand of 16 rows: element (m, e) of lane l = X[row][16 m + 4 (l/16) + e], to be cut where MASK.
template <int HD, bool VEC, bool MASK>
__device__ __forceinline__ void f32_load_rows(f32x4* x, const float* base, int64_t sl, int row, int L, int D, int g) {
    const float* p = f32_row(base, sl, row, L);
#pragma unroll
    for (int m = 0; m < HD / 16; ++m) {
        float v[4];
        f32_ld<4, VEC, MASK>(v, p, 16 * m + 4 * g, D);
        x[m] = f32x4{v[0], v[1], v[2], v[3]};
    }
}
template <int HD, bool VEC, bool MASK>
__device__ __forceinline__ void f32_cut_rows(f32x4* x, int D, int g) {
    if constexpr (MASK) {
        // (a class holds the head dimensions above half of HD: those pieces are whole)
#pragma unroll
        for (int m = HD / 32; m < HD / 16; ++m) {
            if (!VEC && 16 * m + 16 <= D) continue;  // wave-uniform; the few selects of VEC cost less than a branch
            float v[4] = {x[m][0], x[m][1], x[m][2], x[m][3]};
            f32_cut<4, VEC>(v, 16 * m + 4 * g, D);
            x[m] = f32x4{v[0], v[1], v[2], v[3]};
        }
    }
}
// The same for owned rows, cut, and zero beyond L.
template <int HD, bool VEC, bool MASK>
__device__ __forceinline__ void f32_load_own(f32x4* x, const float* base, int64_t sl, int row, int L, int D, int g) {
    f32_load_rows<HD, VEC, MASK>(x, base, sl, row, L, D, g);
    f32_cut_rows<HD, VEC, MASK>(x, D, g);
#pragma unroll
    for (int m = 0; m < HD / 16; ++m)
        if (row >= L) x[m] = f32x4{0.f, 0.f, 0.f, 0.f};
}

// Output-side operand: columns of one row as sub-tiles of the output, W elements per lane and group of 16 W
// columns (W = 4, or 2 for HD = 32): d = 16 W mm + W c + e, c = lane % 16.
template <int HD>
struct F32Cols {
    static constexpr int W = HD == 32 ? 2 : 4;
    static constexpr int MM = HD / (16 * W);
    static constexpr int tiles = W * MM;  // 16-wide sub-tiles: HD / 16
};
template <int HD, bool VEC, bool MASK>
__device__ __forceinline__ void f32_load_cols(float* x, const float* base, int64_t sl, int row, int L, int D, int c) {
    constexpr int W = F32Cols<HD>::W;
    const float* p = f32_row(base, sl, row, L);
#pragma unroll
    for (int mm = 0; mm < F32Cols<HD>::MM; ++mm) f32_ld<W, VEC, MASK>(x + W * mm, p, 16 * W * mm + W * c, D);
}
template <int HD, bool VEC, bool MASK>
__device__ __forceinline__ void f32_cut_cols(float* x, int D, int c) {
    if constexpr (MASK) {
        constexpr int W = F32Cols<HD>::W, mm = F32Cols<HD>::MM - 1;  // the others lie below half of HD
        f32_cut<W, VEC>(x + W * mm, 16 * W * mm + W * c, D);
    }
}
// Zero the operand of a row that does not exist (its tile entries are zero, but 0 * inf is not).
template <int T>
__device__ __forceinline__ void f32_zero_unless(float* x, bool valid) {
#pragma unroll
    for (int t = 0; t < T; ++t) x[t] = valid ? x[t] : 0.f;
}

// One row of an output tensor from the lane's accumulators: registers j of sub-tile (mm, e) are columns
// 16 W mm + 4 W g + W j + e.  Store the W columns of register j.
template <int HD, bool VEC>
__device__ __forceinline__ void f32_store_cols(float* row, const float* x, int mm, int j, int g, int D, bool valid) {
    constexpr int W = F32Cols<HD>::W;
    const int col = 16 * W * mm + 4 * W * g + W * j;
    if (!valid) return;
    if (col + W <= D) {
        typename F32Vec<W>::type v;
#pragma unroll
        for (int e = 0; e < W; ++e) v[e] = x[e];
        *reinterpret_cast<typename F32Vec<W>::type*>(row + col) = v;
    } else if constexpr (!VEC) {
#pragma unroll
        for (int e = 0; e < W; ++e)
            if (col + e < D) row[col + e] = x[e];
    }
}

// The wave's tiles of the streamed axis: `load(row)` requests the score-side operands of a tile, `tile(row, next)`
// consumes them and, once its score tiles are formed, requests those of the next tile (`next` < L), so that
// they arrive under the output contractions; the output-side operands of a tile are requested before its score
// contractions.
template <int SPLIT, typename L0, typename F>
__device__ __forceinline__ void f32_walk(const F32Place& w, int L, L0&& load, F&& tile) {
    constexpr int step = SPLIT * kF32Rows;
    int y0 = w.part * kF32Rows;
    if (y0 < L) load(y0);
    for (; y0 < L; y0 += step) tile(y0, y0 + step);
}

// Store the transposed accumulators of a group of 16 owned rows, times mul (of the lane's row).  With SPLIT the
// waves' partial sums are added first, through `red` (one tensor at a time, [wave][register][lane]), and wave w
// stores the W columns of register u % 4 of sub-tiles u / 4, u = w, w + SPLIT, ...
template <int HD, bool VEC, int SPLIT>
__device__ __forceinline__ void f32_store(float* red, float* row, const f32x4* acc, float mul, const F32Place& w,
                                          int D, bool valid) {
    constexpr int W = F32Cols<HD>::W, MM = F32Cols<HD>::MM, T = F32Cols<HD>::tiles;
    if constexpr (SPLIT == 1) {
#pragma unroll
        for (int mm = 0; mm < MM; ++mm)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float x[W];
#pragma unroll
                for (int e = 0; e < W; ++e) x[e] = acc[W * mm + e][j] * mul;
                f32_store_cols<HD, VEC>(row, x, mm, j, w.g, D, valid);
            }
    } else {
        workgroup_barrier();  // the previous tensor has been read
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j) red[((w.part * T + t) * 4 + j) * 64 + w.lane] = acc[t][j];
        workgroup_barrier();
#pragma unroll
        for (int u0 = 0; u0 < 4 * MM; u0 += SPLIT) {
            const int u = u0 + w.part, mm = u >> 2, j = u & 3;  // wave-uniform
            if (4 * MM % SPLIT != 0 && u >= 4 * MM) break;
            float x[W];
#pragma unroll
            for (int e = 0; e < W; ++e) {
                float s = 0.f;
#pragma unroll
                for (int v = 0; v < SPLIT; ++v) s += red[((v * T + W * mm + e) * 4 + j) * 64 + w.lane];
                x[e] = s * mul;
            }
            f32_store_cols<HD, VEC>(row, x, mm, j, w.g, D, valid);
        }
    }
}
template <int HD, int SPLIT>
constexpr int f32_red_floats() { return SPLIT > 1 ? SPLIT * HD / 16 * 4 * 64 : 1; }

// ---------------------------------------------------------------------------------------------
// Forward (ryu_triton.py:188-291 in fp32): O, TO, lse, mu, li.
// (`red`, `stat`: LDS for the sums of a split group.)
template <int HD, bool JVP, int SPLIT, F32Columns COLS>
__device__ __forceinline__ void fwd_f32_wave(const FwdParamsF32& p, const F32Place& w, float* red, float* stat) {
    constexpr int M = HD / 16, T = HD / 16;
    constexpr bool VEC = COLS != kColumnsCut, MASK = COLS != kColumnsAll;
    const int qrow = w.row0 + w.n;
    const bool qvalid = qrow < p.Lq;
    const int64_t so = (int64_t)w.bh * p.Lr + qrow;  // rows below Lr exist
    if (w.row0 >= p.Lq) {
        // no query in this group: its statistic rows get what a zero query row produces
        if (w.g == 0 && w.part == 0) {
            p.lse[so] = fast_log2((float)p.Lk) * kLn2;
            if constexpr (JVP) p.mu[so] = 0.f;
            if (p.li) p.li[so] = (float)p.Lk;
        }
        return;
    }
    f32x4 q[M], tq[M];
    f32_load_own<HD, VEC, MASK>(q, p.q.head(w.b, w.h), p.q.sl, qrow, p.Lq, p.D, w.g);
    if constexpr (JVP) f32_load_own<HD, VEC, MASK>(tq, p.tq.head(w.b, w.h), p.tq.sl, qrow, p.Lq, p.D, w.g);
    f32x4 acc[T], tacc[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        tacc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const float* kb = p.k.head(w.b, w.h);
    const float* vb = p.v.head(w.b, w.h);
    const float* tkb = JVP ? p.tk.head(w.b, w.h) : nullptr;
    const float* tvb = JVP ? p.tv.head(w.b, w.h) : nullptr;
    const float sl2 = p.scale * kLog2e;
    float m_i = -INFINITY, l_i = 0.f, mu_i = 0.f;  // maximum (log2 units), exp-sum, sum p * S_dot of the lane's keys

    f32x4 kr[M], tkr[M];
    auto load = [&](int k0) {
        f32_load_rows<HD, VEC, MASK>(kr, kb, p.k.sl, k0 + w.n, p.Lk, p.D, w.g);
        if constexpr (JVP) f32_load_rows<HD, VEC, MASK>(tkr, tkb, p.tk.sl, k0 + w.n, p.Lk, p.D, w.g);
    };
    f32_walk<SPLIT>(w, p.Lk, load, [&](int k0, int next) {
        const bool ragged = k0 + kF32Rows > p.Lk;  // wave-uniform
        float v[4][T], tv[4][T];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            f32_load_cols<HD, VEC, MASK>(v[j], vb, p.v.sl, k0 + 4 * w.g + j, p.Lk, p.D, w.n);
            if constexpr (JVP) f32_load_cols<HD, VEC, MASK>(tv[j], tvb, p.tv.sl, k0 + 4 * w.g + j, p.Lk, p.D, w.n);
        }
        __builtin_amdgcn_sched_barrier(0);
        f32_cut_rows<HD, VEC, MASK>(kr, p.D, w.g);
        if constexpr (JVP) f32_cut_rows<HD, VEC, MASK>(tkr, p.D, w.g);
        f32x4 s = {0.f, 0.f, 0.f, 0.f}, ts = s, ts2 = s;
#pragma unroll
        for (int m = 0; m < M; ++m)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                s = mfma_f32(kr[m][e], q[m][e], s);
                if constexpr (JVP) {
                    ts = mfma_f32(kr[m][e], tq[m][e], ts);
                    ts2 = mfma_f32(tkr[m][e], q[m][e], ts2);
                }
            }
        __builtin_amdgcn_sched_barrier(0);
        if (next < p.Lk) load(next);
        s *= sl2;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            f32_cut_cols<HD, VEC, MASK>(v[j], p.D, w.n);
            if constexpr (JVP) f32_cut_cols<HD, VEC, MASK>(tv[j], p.D, w.n);
        }
        if (ragged) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const bool kvalid = k0 + 4 * w.g + j < p.Lk;
                s[j] = kvalid ? s[j] : -INFINITY;
                f32_zero_unless<T>(v[j], kvalid);
                if constexpr (JVP) f32_zero_unless<T>(tv[j], kvalid);
            }
        }
        const float mloc = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
        if (__builtin_amdgcn_ballot_w64(mloc > m_i) != 0) {  // wave-uniform
            const float m_new = fmaxf(m_i, group_max(mloc));
            const float alpha = m_i < m_new ? fast_exp2(m_i - m_new) : 1.f;  // (both may be -inf, see below)
            m_i = m_new;
            l_i *= alpha;
            mu_i *= alpha;
#pragma unroll
            for (int t = 0; t < T; ++t) {
                acc[t] *= alpha;
                if constexpr (JVP) tacc[t] *= alpha;
            }
        }
        // A row whose keys so far all score -inf (products that overflow) has no maximum yet, and no probability: a
        // wave of a split group may hold nothing but such keys.
        const float base = m_i == -INFINITY ? 0.f : m_i;
        f32x4 pt = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            s[j] = fast_exp2(s[j] - base);
            l_i += s[j];
            if constexpr (JVP) {
                pt[j] = s[j] * ((ts[j] + ts2[j]) * p.scale);
                mu_i += pt[j];
            }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
            for (int t = 0; t < T; ++t) {
                acc[t] = mfma_f32(v[j][t], s[j], acc[t]);
                if constexpr (JVP) tacc[t] = mfma_f32(v[j][t], pt[j], tacc[t]);
            }
            if constexpr (JVP)
#pragma unroll
                for (int t = 0; t < T; ++t) tacc[t] = mfma_f32(tv[j][t], s[j], tacc[t]);
        }
    });
    float l = group_sum(l_i), mu_un = group_sum(mu_i);
    if constexpr (SPLIT > 1) {
        // bring the waves' sums to one maximum (a wave without keys has m = -inf, factor 0)
        if (w.g == 0) {
            stat[(3 * w.part + 0) * kF32Rows + w.n] = m_i;
            stat[(3 * w.part + 1) * kF32Rows + w.n] = l;
            stat[(3 * w.part + 2) * kF32Rows + w.n] = mu_un;
        }
        workgroup_barrier();
        float m_all = -INFINITY;
#pragma unroll
        for (int v = 0; v < SPLIT; ++v) m_all = fmaxf(m_all, stat[3 * v * kF32Rows + w.n]);
        l = 0.f;
        mu_un = 0.f;
#pragma unroll
        for (int v = 0; v < SPLIT; ++v) {
            const float f = fast_exp2(stat[3 * v * kF32Rows + w.n] - m_all);
            l += f * stat[(3 * v + 1) * kF32Rows + w.n];
            mu_un += f * stat[(3 * v + 2) * kF32Rows + w.n];
        }
        const float f = fast_exp2(m_i - m_all);
        m_i = m_all;
#pragma unroll
        for (int t = 0; t < T; ++t) {
            acc[t] *= f;
            if constexpr (JVP) tacc[t] *= f;
        }
    }
    const float inv_l = 1.0f / l;
    const float mu = mu_un * inv_l;
    if (w.g == 0 && w.part == 0) {
        // a padded query row (all-zero q, q_dot) yields log(Lk), 0, Lk by itself
        p.lse[so] = (m_i + fast_log2(l)) * kLn2;
        if constexpr (JVP) p.mu[so] = mu;
        if (p.li) p.li[so] = l;
    }
    f32_store<HD, VEC, SPLIT>(red, p.o.head(w.b, w.h) + (int64_t)qrow * p.o.sl, acc, inv_l, w, p.D, qvalid);
    if constexpr (JVP) {
        // TO = (sum (p S_dot) v + sum p v_dot - mu_un O_un) / l   (ryu_triton.py:274-275)
#pragma unroll
        for (int t = 0; t < T; ++t) tacc[t] -= mu * acc[t];
        f32_store<HD, VEC, SPLIT>(red, p.to.head(w.b, w.h) + (int64_t)qrow * p.to.sl, tacc, inv_l, w, p.D, qvalid);
    }
}
template <int HD, bool JVP, int SPLIT, F32Columns COLS>
__global__ __launch_bounds__(kF32Threads, HD == 128 ? 1 : 2) void fwd_f32_kernel(const FwdParamsF32 p) {
    __shared__ float red[f32_red_floats<HD, SPLIT>()];
    __shared__ float stat[SPLIT > 1 ? SPLIT * 3 * kF32Rows : 1];
    fwd_f32_wave<HD, JVP, SPLIT, COLS>(p, f32_place<SPLIT>(p.blocks, p.H), red, stat);
}

// ---------------------------------------------------------------------------------------------
// Row-owned backward: dQ (, dQ_dot) and the row sums for the column-owned kernel.
template <int HD, bool HAS_DO, bool HAS_G, int SPLIT, F32Columns COLS>
__device__ __forceinline__ void bwd_row_f32_wave(const BwdParamsF32& p, const F32Place& w, float* red) {
    constexpr int M = HD / 16, T = HD / 16;
    constexpr bool VEC = COLS != kColumnsCut, MASK = COLS != kColumnsAll;
    if (w.row0 >= p.Lq) return;
    const int qrow = w.row0 + w.n;
    const bool qvalid = qrow < p.Lq;

    f32x4 q[M], tq[M], g[M], dO[M], dq[T], dtq[T];
    float s4 = 0.f, s7d = 0.f;
    f32_load_own<HD, VEC, MASK>(q, p.q.head(w.b, w.h), p.q.sl, qrow, p.Lq, p.D, w.g);
    if constexpr (HAS_G) {
        f32_load_own<HD, VEC, MASK>(tq, p.tq.head(w.b, w.h), p.tq.sl, qrow, p.Lq, p.D, w.g);
        f32_load_own<HD, VEC, MASK>(g, p.dTO.head(w.b, w.h), p.dTO.sl, qrow, p.Lq, p.D, w.g);
    }
    if constexpr (HAS_DO) f32_load_own<HD, VEC, MASK>(dO, p.dO.head(w.b, w.h), p.dO.sl, qrow, p.Lq, p.D, w.g);
    {
        f32x4 o[M], to[M];
        f32_load_own<HD, VEC, MASK>(o, p.o.head(w.b, w.h), p.o.sl, qrow, p.Lq, p.D, w.g);
        if constexpr (HAS_G) f32_load_own<HD, VEC, MASK>(to, p.to.head(w.b, w.h), p.to.sl, qrow, p.Lq, p.D, w.g);
#pragma unroll
        for (int m = 0; m < M; ++m)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if constexpr (HAS_G) {
                    s4 = fmaf(g[m][e], o[m][e], s4);
                    s7d = fmaf(g[m][e], to[m][e], s7d);
                }
                if constexpr (HAS_DO) s7d = fmaf(dO[m][e], o[m][e], s7d);
            }
    }
    s4 = group_sum(s4);
    s7d = group_sum(s7d);
#pragma unroll
    for (int t = 0; t < T; ++t) {
        dq[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        dtq[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const int64_t so = (int64_t)w.bh * p.Lr + qrow;
    const float lse2 = p.lse[so] * kLog2e;
    const float mu = HAS_G ? p.mu[so] : 0.f;
    if (w.g == 0 && w.part == 0) {
        p.lse2[so] = lse2;
        p.s4[so] = s4;
        p.s7d[so] = s7d;
    }
    const float* kb = p.k.head(w.b, w.h);
    const float* vb = p.v.head(w.b, w.h);
    const float* tkb = HAS_G ? p.tk.head(w.b, w.h) : nullptr;
    const float* tvb = HAS_G ? p.tv.head(w.b, w.h) : nullptr;
    const float sl2 = p.scale * kLog2e;

    f32x4 kr[M], tkr[M], vr[M], tvr[M];
    auto load = [&](int k0) {
        f32_load_rows<HD, VEC, MASK>(kr, kb, p.k.sl, k0 + w.n, p.Lk, p.D, w.g);
        if constexpr (HAS_G) f32_load_rows<HD, VEC, MASK>(tkr, tkb, p.tk.sl, k0 + w.n, p.Lk, p.D, w.g);
        f32_load_rows<HD, VEC, MASK>(vr, vb, p.v.sl, k0 + w.n, p.Lk, p.D, w.g);
        if constexpr (HAS_G) f32_load_rows<HD, VEC, MASK>(tvr, tvb, p.tv.sl, k0 + w.n, p.Lk, p.D, w.g);
    };
    f32_walk<SPLIT>(w, p.Lk, load, [&](int k0, int next) {
        const bool ragged = k0 + kF32Rows > p.Lk;  // wave-uniform
        float kc[4][T], tkc[4][T];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            f32_load_cols<HD, VEC, MASK>(kc[j], kb, p.k.sl, k0 + 4 * w.g + j, p.Lk, p.D, w.n);
            if constexpr (HAS_G)
                f32_load_cols<HD, VEC, MASK>(tkc[j], tkb, p.tk.sl, k0 + 4 * w.g + j, p.Lk, p.D, w.n);
        }
        __builtin_amdgcn_sched_barrier(0);
        f32_cut_rows<HD, VEC, MASK>(kr, p.D, w.g);
        f32_cut_rows<HD, VEC, MASK>(vr, p.D, w.g);
        if constexpr (HAS_G) {
            f32_cut_rows<HD, VEC, MASK>(tkr, p.D, w.g);
            f32_cut_rows<HD, VEC, MASK>(tvr, p.D, w.g);
        }
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        f32x4 s = zero, ts = zero, ts2 = zero, wt = zero, xy = zero, xy2 = zero;
#pragma unroll
        for (int m = 0; m < M; ++m)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                s = mfma_f32(kr[m][e], q[m][e], s);
                if constexpr (HAS_G) {
                    ts = mfma_f32(kr[m][e], tq[m][e], ts);
                    ts2 = mfma_f32(tkr[m][e], q[m][e], ts2);
                }
            }
#pragma unroll
        for (int m = 0; m < M; ++m)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if constexpr (HAS_DO) xy = mfma_f32(vr[m][e], dO[m][e], xy);
                if constexpr (HAS_G) {
                    wt = mfma_f32(vr[m][e], g[m][e], wt);
                    xy2 = mfma_f32(tvr[m][e], g[m][e], xy2);
                }
            }
        __builtin_amdgcn_sched_barrier(0);
        if (next < p.Lk) load(next);
        f32x4 ds, dts = zero;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float pj = fast_exp2(fmaf(s[j], sl2, -lse2));
            if constexpr (HAS_G) {
                const float nn = fmaf(ts[j] + ts2[j], p.scale, -mu);
                dts[j] = pj * (wt[j] - s4);
                ds[j] = fmaf(dts[j], nn, pj * (xy[j] + xy2[j] - s7d));
            } else {
                ds[j] = pj * (xy[j] - s7d);
            }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            f32_cut_cols<HD, VEC, MASK>(kc[j], p.D, w.n);
            if constexpr (HAS_G) f32_cut_cols<HD, VEC, MASK>(tkc[j], p.D, w.n);
        }
        if (ragged) {  // keys that do not exist contribute nothing
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const bool kvalid = k0 + 4 * w.g + j < p.Lk;
                ds[j] = kvalid ? ds[j] : 0.f;
                dts[j] = kvalid ? dts[j] : 0.f;
                f32_zero_unless<T>(kc[j], kvalid);
                if constexpr (HAS_G) f32_zero_unless<T>(tkc[j], kvalid);
            }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
            for (int t = 0; t < T; ++t) {
                dq[t] = mfma_f32(kc[j][t], ds[j], dq[t]);
                if constexpr (HAS_G) dtq[t] = mfma_f32(kc[j][t], dts[j], dtq[t]);
            }
            if constexpr (HAS_G)
#pragma unroll
                for (int t = 0; t < T; ++t) dq[t] = mfma_f32(tkc[j][t], dts[j], dq[t]);
        }
    });
    f32_store<HD, VEC, SPLIT>(red, p.dq.head(w.b, w.h) + (int64_t)qrow * p.dq.sl, dq, p.scale, w, p.D, qvalid);
    if constexpr (HAS_G)
        f32_store<HD, VEC, SPLIT>(red, p.dtq.head(w.b, w.h) + (int64_t)qrow * p.dtq.sl, dtq, p.scale, w, p.D, qvalid);
}
template <int HD, bool HAS_DO, bool HAS_G, int SPLIT, F32Columns COLS>
__global__ __launch_bounds__(kF32Threads, HD == 128 || (HD == 64 && HAS_G) ? 1 : 2) void bwd_row_f32_kernel(const BwdParamsF32 p) {
    __shared__ float red[f32_red_floats<HD, SPLIT>()];
    bwd_row_f32_wave<HD, HAS_DO, HAS_G, SPLIT, COLS>(p, f32_place<SPLIT>(p.q_blocks, p.H), red);
}

// ---------------------------------------------------------------------------------------------
// Column-owned backward: dK, dV (, dK_dot, dV_dot).
template <int HD, bool HAS_DO, bool HAS_G, int SPLIT, F32Columns COLS>
__device__ __forceinline__ void bwd_col_f32_wave(const BwdParamsF32& p, const F32Place& w, float* red) {
    constexpr int M = HD / 16, T = HD / 16;
    constexpr bool VEC = COLS != kColumnsCut, MASK = COLS != kColumnsAll;
    if (w.row0 >= p.Lk) return;
    const int krow = w.row0 + w.n;
    const bool kvalid = krow < p.Lk;

    f32x4 k[M], v[M], tk[M], tv[M], dk[T], dv[T], dtk[T], dtv[T];
    f32_load_own<HD, VEC, MASK>(k, p.k.head(w.b, w.h), p.k.sl, krow, p.Lk, p.D, w.g);
    f32_load_own<HD, VEC, MASK>(v, p.v.head(w.b, w.h), p.v.sl, krow, p.Lk, p.D, w.g);
    if constexpr (HAS_G) {
        f32_load_own<HD, VEC, MASK>(tk, p.tk.head(w.b, w.h), p.tk.sl, krow, p.Lk, p.D, w.g);
        f32_load_own<HD, VEC, MASK>(tv, p.tv.head(w.b, w.h), p.tv.sl, krow, p.Lk, p.D, w.g);
    }
#pragma unroll
    for (int t = 0; t < T; ++t) {
        dk[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        dv[t] = dk[t];
        dtk[t] = dk[t];
        dtv[t] = dk[t];
    }
    const float* qb = p.q.head(w.b, w.h);
    const float* tqb = HAS_G ? p.tq.head(w.b, w.h) : nullptr;
    const float* gb = HAS_G ? p.dTO.head(w.b, w.h) : nullptr;
    const float* dob = HAS_DO ? p.dO.head(w.b, w.h) : nullptr;
    const int64_t so = (int64_t)w.bh * p.Lr + 4 * w.g;  // rows below Lr exist in every statistic
    const float sl2 = p.scale * kLog2e;

    f32x4 qr[M], tqr[M], gr[M], dor[M];
    auto load = [&](int q0) {
        f32_load_rows<HD, VEC, MASK>(qr, qb, p.q.sl, q0 + w.n, p.Lq, p.D, w.g);
        if constexpr (HAS_G) f32_load_rows<HD, VEC, MASK>(tqr, tqb, p.tq.sl, q0 + w.n, p.Lq, p.D, w.g);
    };
    f32_walk<SPLIT>(w, p.Lq, load, [&](int q0, int next) {
        const bool ragged = q0 + kF32Rows > p.Lq;  // wave-uniform
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        const f32x4 lse2 = *reinterpret_cast<const f32x4*>(p.lse2 + so + q0);
        const f32x4 s7d = *reinterpret_cast<const f32x4*>(p.s7d + so + q0);
        f32x4 mu = zero, s4 = zero;
        if constexpr (HAS_G) {
            s4 = *reinterpret_cast<const f32x4*>(p.s4 + so + q0);
            mu = *reinterpret_cast<const f32x4*>(p.mu + so + q0);
        }
        // output-side operands of row 4 g + j: Q, [G, Q_dot], [dO]; those of j + 1 are requested ahead of j's
        // contractions (all four at once do not fit the registers)
        float cq[2][T], cg[2][T], ctq[2][T], cdo[2][T];
        auto load_cols = [&](int j, int u) {
            const int row = q0 + 4 * w.g + j;
            f32_load_cols<HD, VEC, MASK>(cq[u], qb, p.q.sl, row, p.Lq, p.D, w.n);
            if constexpr (HAS_G) {
                f32_load_cols<HD, VEC, MASK>(cg[u], gb, p.dTO.sl, row, p.Lq, p.D, w.n);
                f32_load_cols<HD, VEC, MASK>(ctq[u], tqb, p.tq.sl, row, p.Lq, p.D, w.n);
            }
            if constexpr (HAS_DO) f32_load_cols<HD, VEC, MASK>(cdo[u], dob, p.dO.sl, row, p.Lq, p.D, w.n);
        };
        // G and dO rows are first used behind the Q, Q_dot contractions: no need to hold them from the last tile
        if constexpr (HAS_G) f32_load_rows<HD, VEC, MASK>(gr, gb, p.dTO.sl, q0 + w.n, p.Lq, p.D, w.g);
        if constexpr (HAS_DO) f32_load_rows<HD, VEC, MASK>(dor, dob, p.dO.sl, q0 + w.n, p.Lq, p.D, w.g);
        load_cols(0, 0);
        __builtin_amdgcn_sched_barrier(0);
        f32_cut_rows<HD, VEC, MASK>(qr, p.D, w.g);
        if constexpr (HAS_G) f32_cut_rows<HD, VEC, MASK>(tqr, p.D, w.g);
        f32x4 s = zero, ts = zero, ts2 = zero, wt = zero, xy = zero, xy2 = zero;
#pragma unroll
        for (int m = 0; m < M; ++m)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                s = mfma_f32(qr[m][e], k[m][e], s);
                if constexpr (HAS_G) {
                    ts = mfma_f32(tqr[m][e], k[m][e], ts);
                    ts2 = mfma_f32(qr[m][e], tk[m][e], ts2);
                }
            }
        if constexpr (HAS_G) f32_cut_rows<HD, VEC, MASK>(gr, p.D, w.g);
        if constexpr (HAS_DO) f32_cut_rows<HD, VEC, MASK>(dor, p.D, w.g);
#pragma unroll
        for (int m = 0; m < M; ++m)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if constexpr (HAS_G) {
                    wt = mfma_f32(gr[m][e], v[m][e], wt);
                    xy2 = mfma_f32(gr[m][e], tv[m][e], xy2);
                }
                if constexpr (HAS_DO) xy = mfma_f32(dor[m][e], v[m][e], xy);
            }
        __builtin_amdgcn_sched_barrier(0);
        load_cols(1, 1);
        if (next < p.Lq) load(next);
        f32x4 pr, pn = zero, ds, dts = zero;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float pj = kvalid ? fast_exp2(fmaf(s[j], sl2, -lse2[j])) : 0.f;  // a padded key contributes nothing
            pr[j] = pj;
            if constexpr (HAS_G) {
                const float nn = fmaf(ts[j] + ts2[j], p.scale, -mu[j]);
                dts[j] = pj * (wt[j] - s4[j]);
                ds[j] = fmaf(dts[j], nn, pj * (xy[j] + xy2[j] - s7d[j]));
                pn[j] = pj * nn;
            } else {
                ds[j] = pj * (xy[j] - s7d[j]);
            }
        }
        if (ragged) {  // nor does a query that does not exist
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const bool qvalid = q0 + 4 * w.g + j < p.Lq;
                pr[j] = qvalid ? pr[j] : 0.f;
                pn[j] = qvalid ? pn[j] : 0.f;
                ds[j] = qvalid ? ds[j] : 0.f;
                dts[j] = qvalid ? dts[j] : 0.f;
            }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int u = j & 1;
            f32_cut_cols<HD, VEC, MASK>(cq[u], p.D, w.n);
            if constexpr (HAS_G) {
                f32_cut_cols<HD, VEC, MASK>(cg[u], p.D, w.n);
                f32_cut_cols<HD, VEC, MASK>(ctq[u], p.D, w.n);
            }
            if constexpr (HAS_DO) f32_cut_cols<HD, VEC, MASK>(cdo[u], p.D, w.n);
            if (ragged) {
                const bool qvalid = q0 + 4 * w.g + j < p.Lq;
                f32_zero_unless<T>(cq[u], qvalid);
                if constexpr (HAS_G) {
                    f32_zero_unless<T>(cg[u], qvalid);
                    f32_zero_unless<T>(ctq[u], qvalid);
                }
                if constexpr (HAS_DO) f32_zero_unless<T>(cdo[u], qvalid);
            }
#pragma unroll
            for (int t = 0; t < T; ++t) {
                dk[t] = mfma_f32(cq[u][t], ds[j], dk[t]);
                if constexpr (HAS_G) {
                    dtk[t] = mfma_f32(cq[u][t], dts[j], dtk[t]);
                    dv[t] = mfma_f32(cg[u][t], pn[j], dv[t]);
                    dtv[t] = mfma_f32(cg[u][t], pr[j], dtv[t]);
                }
            }
#pragma unroll
            for (int t = 0; t < T; ++t) {
                if constexpr (HAS_G) dk[t] = mfma_f32(ctq[u][t], dts[j], dk[t]);
                if constexpr (HAS_DO) dv[t] = mfma_f32(cdo[u][t], pr[j], dv[t]);
            }
            if (j < 2) load_cols(j + 2, u);
        }
    });
    f32_store<HD, VEC, SPLIT>(red, p.dk.head(w.b, w.h) + (int64_t)krow * p.dk.sl, dk, p.scale, w, p.D, kvalid);
    f32_store<HD, VEC, SPLIT>(red, p.dv.head(w.b, w.h) + (int64_t)krow * p.dv.sl, dv, 1.0f, w, p.D, kvalid);
    if constexpr (HAS_G) {
        f32_store<HD, VEC, SPLIT>(red, p.dtk.head(w.b, w.h) + (int64_t)krow * p.dtk.sl, dtk, p.scale, w, p.D, kvalid);
        f32_store<HD, VEC, SPLIT>(red, p.dtv.head(w.b, w.h) + (int64_t)krow * p.dtv.sl, dtv, 1.0f, w, p.D, kvalid);
    }
}
template <int HD, bool HAS_DO, bool HAS_G, int SPLIT, F32Columns COLS>
__global__ __launch_bounds__(kF32Threads, HD == 128 || (HD == 64 && HAS_G) ? 1 : 2) void bwd_col_f32_kernel(const BwdParamsF32 p) {
    __shared__ float red[f32_red_floats<HD, SPLIT>()];
    bwd_col_f32_wave<HD, HAS_DO, HAS_G, SPLIT, COLS>(p, f32_place<SPLIT>(p.k_blocks, p.H), red);
}

}  // namespace sjvp
