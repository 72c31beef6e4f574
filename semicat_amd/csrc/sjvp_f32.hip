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

// The kernels on the bf16 matrix pipe (sjvp_f32x3.hpp) take all launches on a shape or none: the backward forms the
// scores again, and against the log-sum-exp of the other set's scores its error grows (dQ of 200 queries on 32 keys, D = 100: 1.18 times
// the fp32 unit's, by one set 0.99).  A backward does not know whether its forward had tangents (for a cotangent on O alone it is
// given none), so the rule asks the shape alone.  `rows`: owned rows of a (batch, head) pair (padded in the forward), `streamed`: the other axis.
//
// Four waves while every workgroup of 64 rows has a compute unit, else eight, whose workgroups split the streamed side once
// for 128 rows (D = 64, L = 256, 1024 / 2048 groups of 16 rows, four / eight: forward 28 / 36 and 54 / 40 us, row kernel 37 / 47 and
// 71 / 54, column 47 / 63 and 91 / 71).  The backward at D <= 32 (two workgroups of four share a unit: row kernel, 2048 and 2304
// groups, 33 / 32 and 48 / 57) and without tangents (D = 64: 27 / 25 and 34 / 44) keeps to four, so does all of D > 64.
//
// A launch costs rounds of workgroups times streamed tiles; per tile, in fortieths of what a round of the fp32 unit's whole
// groups takes: 28 (four waves; D > 64: 32) or 37 (eight), the forward without tangents 40 and 50, the backward by pairs of waves 25
// (D > 96 on more than 256 rows: 27); the fp32 unit's 40, 13 for each round of split groups.
// Both sides in us, fp32 unit / here, L = 256: D = 64 512 groups 26 / 27 forward, 37 / 34 row, 40 / 44 column; 640 31 / 26, 54 / 33, 59 / 41; 4096 142 / 78, 201 / 105, 250 / 139; D = 80 384 42 / 50, 61 / 53, 74 / 56,
// 640 62 / 50, 90 / 53, 113 / 57; D = 128 384 43 / 51, 70 / 61, 73 / 70 (L = 1024: 125 / 187, 202 / 206, 218 / 239), 576 64 / 53, 104 / 62,
// 108 / 72; D = 32 without tangents, forward, 640 9.0 / 11.2, 2048 17 / 13.
inline int x3_width(int BH, int rows, int D, bool forward, bool tangents, int units = compute_units()) {
    const int64_t four = (int64_t)BH * ((rows + 63) / 64);
    return D > 64 || four <= units || (!forward && (D <= 32 || !tangents)) ? 4 : 8;
}
// What a launch saves there, in tenths of fortieths.
inline int64_t x3_saves(int BH, int groups_of, int rows, int streamed, int D, bool forward, bool tangents, int units) {
    const int waves = x3_width(BH, rows, D, forward, tangents, units);
    // tenths; workgroups of four that share a compute unit (48 KB of LDS, or less) add 0.7 of a round each
    int64_t rounds = ((int64_t)BH * ((rows + 16 * waves - 1) / (16 * waves)) + units - 1) / units;
    rounds = waves == 4 && (D <= 32 || (D <= 64 && !tangents)) ? 7 * rounds + 3 : 10 * rounds;
    const int pairs = D > 96 && streamed > 256 ? 27 : 25;
    const int per_tile = forward && !tangents ? (waves == 4 ? 40 : 50) : D > 64 ? (!forward && tangents ? pairs : 32) : waves == 4 ? 28 : 37;
    const int64_t groups = (int64_t)BH * ((groups_of + kF32Rows - 1) / kF32Rows);
    const int64_t unit = split(BH, groups_of, streamed) == 4 ? 13 * ((4 * groups + kSimds - 1) / kSimds) : 40 * ((groups + kSimds - 1) / kSimds);
    const int64_t tiles = (streamed + kF32Rows - 1) / kF32Rows, stages = (streamed + kStageRows - 1) / kStageRows;
    return 10 * tiles * unit - 2 * stages * rounds * per_tile;
}
// Where the launches of plain calls (the forward without tangents, or a cotangent on O alone) gain, or those of a call with tangents, whose costs
// are nearer to what is measured: at D <= 64 only if no launch of theirs leaves more than half of the compute units without a workgroup.
// Forward + backward with and without tangents, fp32 unit / here, us, at shapes where the two kinds' costs disagree:
//   plain launches gain, 46 shapes: with tangents 0.81 on average (0.56 to 1.19), plain 0.78: 332 heads, 144 x 144, D = 48 397 / 281 and
//   145 / 100; the worst, 300 heads, 3170 queries on 24 keys, D = 64 1592 / 1903 and 691 / 605;
//   launches with tangents gain, 80 shapes: 60 heads, 259 x 259, D = 48 321 / 153 and 125 / 82; 120 heads, 803 x 803, D = 128 5470 / 3742 and
//   2428 / 1596; the worst, 186 heads, 44 on 1663, D = 100 1539 / 1694 and 618 / 739; with half of the units idle at D > 64, 104 heads, 59 on
//   424, D = 100 295 / 293 and 122 / 136, 35 heads, 280 on 154, D = 80 220 / 140 and 89 / 74; stays on the unit: 78 heads, 52 on 3516,
//   D = 20 505 / 564 and 204 / 313; 24 heads, 250 on 2586, D = 16 349 / 350 and 142 / 193.
inline bool x3_takes(int BH, int Lq, int Lr, int Lk, int D) {
    const int units = compute_units();  // asks the runtime for the device: once
    auto gains = [&](bool tangents) {  // by the contractions of forward, row and column launch: 6, 9 and 12, without tangents 2, 3 and 4
        return 2 * x3_saves(BH, Lq, Lr, Lk, D, true, tangents, units) + 3 * x3_saves(BH, Lq, Lq, Lk, D, false, tangents, units) +
                   4 * x3_saves(BH, Lk, Lk, Lq, D, false, tangents, units) > 0;
    };
    const int64_t fewest = (int64_t)BH * (((Lq < Lk ? Lq : Lk) + 63) / 64);
    return gains(false) || (gains(true) && (D > 64 || 2 * fewest >= units));
}
inline int blocks(int rows, int split) {
    const int per = split > 1 ? kF32Rows : kF32Rows * kF32Waves;
    return (rows + per - 1) / per;
}

template <int HD, bool JVP, F32Columns COLS>
int fwd_one(FwdParamsF32 p, int BH, hipStream_t stream) {
    const int sp = split(BH, p.Lq, p.Lk);
    if (x3_takes(BH, p.Lq, p.Lr, p.Lk, p.D)) return fwd_f32x3(p, BH, JVP, x3_width(BH, p.Lr, p.D, true, JVP), stream);
    p.blocks = blocks(p.Lr, sp);  // the statistics cover rows below Lr
    const int grid = BH * p.blocks;
    if (sp == 4) return launch(fwd_f32_kernel<HD, JVP, 4, COLS>, grid, 0, stream, p, kF32Threads);
    return launch(fwd_f32_kernel<HD, JVP, 1, COLS>, grid, 0, stream, p, kF32Threads);
}

template <int HD, bool HAS_DO, bool HAS_G, F32Columns COLS>
int row_one(BwdParamsF32 p, int BH, hipStream_t stream) {
    const int sp = split(BH, p.Lq, p.Lk);
    if (x3_takes(BH, p.Lq, p.Lr, p.Lk, p.D))
        return bwd_f32x3(p, BH, HAS_DO, HAS_G, SJVP_BWD_ROW, x3_width(BH, p.Lq, p.D, false, HAS_G), stream);
    p.q_blocks = blocks(p.Lq, sp);
    const int grid = BH * p.q_blocks;
    if (sp == 4) return launch(bwd_row_f32_kernel<HD, HAS_DO, HAS_G, 4, COLS>, grid, 0, stream, p, kF32Threads);
    return launch(bwd_row_f32_kernel<HD, HAS_DO, HAS_G, 1, COLS>, grid, 0, stream, p, kF32Threads);
}

template <int HD, bool HAS_DO, bool HAS_G, F32Columns COLS>
int col_one(BwdParamsF32 p, int BH, hipStream_t stream) {
    const int sp = split(BH, p.Lk, p.Lq);
    if (x3_takes(BH, p.Lq, p.Lr, p.Lk, p.D))
        return bwd_f32x3(p, BH, HAS_DO, HAS_G, SJVP_BWD_COL, x3_width(BH, p.Lk, p.D, false, HAS_G), stream);
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
