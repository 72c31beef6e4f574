// Translation unit: the fp32 kernels of the correctness mode.
#include "sjvp_f32.hpp"
#include "sjvp_launch.hpp"

namespace sjvp {
namespace {

// Waves per group of 16 owned rows: 4 where that shortens the launch.  A SIMD holds one or two of these
// waves and the matrix pipe is what they share, so a launch takes as many rounds as there are waves per SIMD
// (1024 of them); a wave of a split group works a quarter as long, plus its prologue and its share of the
// reduction, which made the whole launch 1.3 times as long at equal rounds (forward + backward at D = 64, L = 256,
// split / not: 1024 groups 200 / 154 us; 1152 groups 241 / 298; 1536 groups 293 / 303; 128 groups 51 / 155).
constexpr int64_t kSimds = 1024;

inline int split(int BH, int rows, int streamed) {
    const int64_t groups = (int64_t)BH * ((rows + kF32Rows - 1) / kF32Rows);
    const int64_t whole = 4 * ((groups + kSimds - 1) / kSimds), quarter = (4 * groups + kSimds - 1) / kSimds;
    return streamed > kF32Rows && 13 * quarter < 10 * whole ? 4 : 1;
}
inline int blocks(int rows, int split) {
    const int per = split > 1 ? kF32Rows : kF32Rows * kF32Waves;
    return (rows + per - 1) / per;
}

template <int HD, bool JVP, bool VEC>
int fwd_one(FwdParamsF32 p, int BH, hipStream_t stream) {
    const int sp = split(BH, p.Lq, p.Lk);
    p.blocks = blocks(p.Lr, sp);  // the statistics cover rows below Lr
    const int grid = BH * p.blocks;
    if (sp == 4) return launch(fwd_f32_kernel<HD, JVP, 4, VEC>, grid, 0, stream, p, kF32Threads);
    return launch(fwd_f32_kernel<HD, JVP, 1, VEC>, grid, 0, stream, p, kF32Threads);
}

template <int HD, bool HAS_DO, bool HAS_G, bool VEC>
int row_one(BwdParamsF32 p, int BH, hipStream_t stream) {
    const int sp = split(BH, p.Lq, p.Lk);
    p.q_blocks = blocks(p.Lq, sp);
    const int grid = BH * p.q_blocks;
    if (sp == 4) return launch(bwd_row_f32_kernel<HD, HAS_DO, HAS_G, 4, VEC>, grid, 0, stream, p, kF32Threads);
    return launch(bwd_row_f32_kernel<HD, HAS_DO, HAS_G, 1, VEC>, grid, 0, stream, p, kF32Threads);
}

template <int HD, bool HAS_DO, bool HAS_G, bool VEC>
int col_one(BwdParamsF32 p, int BH, hipStream_t stream) {
    const int sp = split(BH, p.Lk, p.Lq);
    p.k_blocks = blocks(p.Lk, sp);
    const int grid = BH * p.k_blocks;
    if (sp == 4) return launch(bwd_col_f32_kernel<HD, HAS_DO, HAS_G, 4, VEC>, grid, 0, stream, p, kF32Threads);
    return launch(bwd_col_f32_kernel<HD, HAS_DO, HAS_G, 1, VEC>, grid, 0, stream, p, kF32Threads);
}

template <int HD, bool HAS_DO, bool HAS_G, bool VEC>
int bwd_one(const BwdParamsF32& p, int BH, int parts, hipStream_t stream) {
    if (parts & SJVP_BWD_ROW) {
        const int rc = row_one<HD, HAS_DO, HAS_G, VEC>(p, BH, stream);
        if (rc != SJVP_OK) return rc;
    }
    return parts & SJVP_BWD_COL ? col_one<HD, HAS_DO, HAS_G, VEC>(p, BH, stream) : SJVP_OK;
}

template <int HD, bool VEC>
int bwd_mode(const BwdParamsF32& p, int BH, bool has_do, bool has_g, int parts, hipStream_t stream) {
    if (has_do && has_g) return bwd_one<HD, true, true, VEC>(p, BH, parts, stream);
    if (has_g) return bwd_one<HD, false, true, VEC>(p, BH, parts, stream);
    return bwd_one<HD, true, false, VEC>(p, BH, parts, stream);
}

template <bool VEC>
int fwd_hd(const FwdParamsF32& p, int BH, bool jvp, hipStream_t stream) {
    if (p.D <= 32) return jvp ? fwd_one<32, true, VEC>(p, BH, stream) : fwd_one<32, false, VEC>(p, BH, stream);
    if (p.D <= 64) return jvp ? fwd_one<64, true, VEC>(p, BH, stream) : fwd_one<64, false, VEC>(p, BH, stream);
    return jvp ? fwd_one<128, true, VEC>(p, BH, stream) : fwd_one<128, false, VEC>(p, BH, stream);
}

template <bool VEC>
int bwd_hd(const BwdParamsF32& p, int BH, bool has_do, bool has_g, int parts, hipStream_t stream) {
    if (p.D <= 32) return bwd_mode<32, VEC>(p, BH, has_do, has_g, parts, stream);
    if (p.D <= 64) return bwd_mode<64, VEC>(p, BH, has_do, has_g, parts, stream);
    return bwd_mode<128, VEC>(p, BH, has_do, has_g, parts, stream);
}

}  // namespace

int fwd_f32(const FwdParamsF32& p, int BH, bool jvp, bool vec, hipStream_t stream) {
    return vec ? fwd_hd<true>(p, BH, jvp, stream) : fwd_hd<false>(p, BH, jvp, stream);
}

int bwd_f32(const BwdParamsF32& p, int BH, bool has_do, bool has_g, int parts, bool vec, hipStream_t stream) {
    return vec ? bwd_hd<true>(p, BH, has_do, has_g, parts, stream) : bwd_hd<false>(p, BH, has_do, has_g, parts, stream);
}

}  // namespace sjvp
