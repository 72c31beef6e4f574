// Translation unit: the fp32 kernels of the correctness mode.
#include <type_traits>

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

template <int HD, bool JVP, F32Columns COLS>
int fwd_one(FwdParamsF32 p, int BH, hipStream_t stream) {
    const int sp = split(BH, p.Lq, p.Lk);
    p.blocks = blocks(p.Lr, sp);  // the statistics cover rows below Lr
    const int grid = BH * p.blocks;
    if (sp == 4) return launch(fwd_f32_kernel<HD, JVP, 4, COLS>, grid, 0, stream, p, kF32Threads);
    return launch(fwd_f32_kernel<HD, JVP, 1, COLS>, grid, 0, stream, p, kF32Threads);
}

template <int HD, bool HAS_DO, bool HAS_G, F32Columns COLS>
int row_one(BwdParamsF32 p, int BH, hipStream_t stream) {
    const int sp = split(BH, p.Lq, p.Lk);
    p.q_blocks = blocks(p.Lq, sp);
    const int grid = BH * p.q_blocks;
    if (sp == 4) return launch(bwd_row_f32_kernel<HD, HAS_DO, HAS_G, 4, COLS>, grid, 0, stream, p, kF32Threads);
    return launch(bwd_row_f32_kernel<HD, HAS_DO, HAS_G, 1, COLS>, grid, 0, stream, p, kF32Threads);
}

template <int HD, bool HAS_DO, bool HAS_G, F32Columns COLS>
int col_one(BwdParamsF32 p, int BH, hipStream_t stream) {
    const int sp = split(BH, p.Lk, p.Lq);
    p.k_blocks = blocks(p.Lk, sp);
    const int grid = BH * p.k_blocks;
    if (sp == 4) return launch(bwd_col_f32_kernel<HD, HAS_DO, HAS_G, 4, COLS>, grid, 0, stream, p, kF32Threads);
    return launch(bwd_col_f32_kernel<HD, HAS_DO, HAS_G, 1, COLS>, grid, 0, stream, p, kF32Threads);
}

template <int HD, bool HAS_DO, bool HAS_G, F32Columns COLS>
int bwd_one(const BwdParamsF32& p, int BH, int parts, hipStream_t stream) {
    if (parts & SJVP_BWD_ROW) {
        const int rc = row_one<HD, HAS_DO, HAS_G, COLS>(p, BH, stream);
        if (rc != SJVP_OK) return rc;
    }
    return parts & SJVP_BWD_COL ? col_one<HD, HAS_DO, HAS_G, COLS>(p, BH, stream) : SJVP_OK;
}

// Calls f with the compiled head dimension and the form of its columns as constants.
template <int HD, typename F>
int by_columns(int D, F&& f) {
    constexpr std::integral_constant<int, HD> hd{};
    if (D == HD) return f(hd, std::integral_constant<F32Columns, kColumnsAll>{});
    if (D % 4 == 0) return f(hd, std::integral_constant<F32Columns, kColumnsWhole>{});
    return f(hd, std::integral_constant<F32Columns, kColumnsCut>{});
}
template <typename F>
int by_head(int D, F&& f) {
    return D <= 32 ? by_columns<32>(D, f) : D <= 64 ? by_columns<64>(D, f) : by_columns<128>(D, f);
}

}  // namespace

int fwd_f32(const FwdParamsF32& p, int BH, bool jvp, hipStream_t stream) {
    return by_head(p.D, [&](auto hd, auto cols) {
        constexpr int HD = decltype(hd)::value;
        constexpr F32Columns COLS = decltype(cols)::value;
        return jvp ? fwd_one<HD, true, COLS>(p, BH, stream) : fwd_one<HD, false, COLS>(p, BH, stream);
    });
}

int bwd_f32(const BwdParamsF32& p, int BH, bool has_do, bool has_g, int parts, hipStream_t stream) {
    return by_head(p.D, [&](auto hd, auto cols) {
        constexpr int HD = decltype(hd)::value;
        constexpr F32Columns COLS = decltype(cols)::value;
        if (has_do && has_g) return bwd_one<HD, true, true, COLS>(p, BH, parts, stream);
        if (has_g) return bwd_one<HD, false, true, COLS>(p, BH, parts, stream);
        return bwd_one<HD, true, false, COLS>(p, BH, parts, stream);
    });
}

}  // namespace sjvp
