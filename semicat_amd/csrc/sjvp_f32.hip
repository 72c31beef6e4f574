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

// Waves of a workgroup for which the kernels on the bf16 matrix pipe (sjvp_f32x3.hpp) take the launch, 0 where the ones on the
// fp32 unit keep it.  `rows`: owned rows of a (batch, head) pair (padded in the forward), `streamed`: the other axis.
//
// Four waves while every workgroup of 64 rows has a compute unit, else eight, whose workgroups split the streamed side once
// for 128 rows (D = 64, L = 256, 1024 / 2048 groups of 16 rows, four / eight: forward 28 / 36 and 54 / 40 us, row kernel 37 / 47 and
// 71 / 54, column 47 / 63 and 91 / 71).  The backward at D <= 32 (two workgroups of four share a unit: row kernel, 2048 and 2304
// groups, 33 / 32 and 48 / 57) and without tangents (D = 64: 27 / 25 and 34 / 44) keeps to four, so does all of D > 64.
//
// A launch costs rounds of workgroups times streamed tiles; per tile, in fortieths of what a round of the fp32 unit's whole
// groups takes: 28 (four waves; D > 64: 32) or 37 (eight), the forward without tangents 40 and 50; the fp32 unit's 40, 13 for each
// round of split groups.  Both sides in us, fp32 unit / here, L = 256: D = 64 512 groups 26 / 27 forward, 37 / 34 row, 40 / 44 column;
// 640 31 / 26, 54 / 33, 59 / 41; 4096 142 / 78, 201 / 105, 250 / 139; D = 80 640 62 / 50, 90 / 60, 113 / 57; D = 128
// 448 44 / 51, 70 / 70, 73 / 71, 576 64 / 53, 104 / 70, 108 / 72; D = 32 without tangents, forward, 640 9.0 / 11.2, 2048 17 / 13.
inline int x3_waves(int BH, int groups_of, int rows, int streamed, int D, bool forward, bool tangents, int split) {
    const int units = compute_units();
    const int64_t four = (int64_t)BH * ((rows + 63) / 64), eight = (int64_t)BH * ((rows + 127) / 128);
    const int waves = D > 64 || four <= units || (!forward && (D <= 32 || !tangents)) ? 4 : 8;
    // tenths; workgroups of four that share a compute unit (48 KB of LDS, or less) add 0.7 of a round each
    int64_t rounds = ((waves == 4 ? four : eight) + units - 1) / units;
    rounds = waves == 4 && (D <= 32 || (D <= 64 && !tangents)) ? 7 * rounds + 3 : 10 * rounds;
    const int per_tile = forward && !tangents ? (waves == 4 ? 40 : 50) : D > 64 ? 32 : waves == 4 ? 28 : 37;
    const int64_t groups = (int64_t)BH * ((groups_of + kF32Rows - 1) / kF32Rows);
    const int64_t unit = split == 4 ? 13 * ((4 * groups + kSimds - 1) / kSimds) : 40 * ((groups + kSimds - 1) / kSimds);
    const int64_t tiles = (streamed + kF32Rows - 1) / kF32Rows, stages = (streamed + kStageRows - 1) / kStageRows;
    return 2 * stages * rounds * per_tile < 10 * tiles * unit ? waves : 0;
}
inline int blocks(int rows, int split) {
    const int per = split > 1 ? kF32Rows : kF32Rows * kF32Waves;
    return (rows + per - 1) / per;
}

template <int HD, bool JVP, F32Columns COLS>
int fwd_one(FwdParamsF32 p, int BH, hipStream_t stream) {
    const int sp = split(BH, p.Lq, p.Lk);
    if (const int waves = x3_waves(BH, p.Lq, p.Lr, p.Lk, p.D, true, JVP, sp)) return fwd_f32x3(p, BH, JVP, waves, stream);
    p.blocks = blocks(p.Lr, sp);  // the statistics cover rows below Lr
    const int grid = BH * p.blocks;
    if (sp == 4) return launch(fwd_f32_kernel<HD, JVP, 4, COLS>, grid, 0, stream, p, kF32Threads);
    return launch(fwd_f32_kernel<HD, JVP, 1, COLS>, grid, 0, stream, p, kF32Threads);
}

template <int HD, bool HAS_DO, bool HAS_G, F32Columns COLS>
int row_one(BwdParamsF32 p, int BH, hipStream_t stream) {
    const int sp = split(BH, p.Lq, p.Lk);
    if (const int waves = x3_waves(BH, p.Lq, p.Lq, p.Lk, p.D, false, HAS_G, sp))
        return bwd_f32x3(p, BH, HAS_DO, HAS_G, SJVP_BWD_ROW, waves, stream);
    p.q_blocks = blocks(p.Lq, sp);
    const int grid = BH * p.q_blocks;
    if (sp == 4) return launch(bwd_row_f32_kernel<HD, HAS_DO, HAS_G, 4, COLS>, grid, 0, stream, p, kF32Threads);
    return launch(bwd_row_f32_kernel<HD, HAS_DO, HAS_G, 1, COLS>, grid, 0, stream, p, kF32Threads);
}

template <int HD, bool HAS_DO, bool HAS_G, F32Columns COLS>
int col_one(BwdParamsF32 p, int BH, hipStream_t stream) {
    const int sp = split(BH, p.Lk, p.Lq);
    if (const int waves = x3_waves(BH, p.Lk, p.Lk, p.Lq, p.D, false, HAS_G, sp))
        return bwd_f32x3(p, BH, HAS_DO, HAS_G, SJVP_BWD_COL, waves, stream);
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
