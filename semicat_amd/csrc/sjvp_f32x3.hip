// Translation unit: the fp32 kernels on the bf16 matrix pipe.
#include <type_traits>

#include "sjvp_f32x3.hpp"

#include "sjvp_launch.hpp"

namespace sjvp {
namespace {

template <int HD, int DT, bool JVP, int NW>
int fwd_one(FwdParamsF32 p, int BH, hipStream_t stream) {
    p.blocks = p.Lr / (16 * NW);
    return launch(fwd_f32x3_kernel<HD, DT, JVP, NW>, BH * p.blocks, TriSmem<HD, JVP ? 4 : 2>::bytes, stream, p, 64 * NW);
}

template <int HD, int DT, bool HAS_DO, bool HAS_G, int NW>
int row_one(BwdParamsF32 p, int BH, hipStream_t stream) {
    if constexpr (HD == 128 && HAS_G) {
        p.q_blocks = (p.Lq + 16 * kPairs - 1) / (16 * kPairs);
        return launch(bwd_row_f32x3_pair_kernel<HD, DT, HAS_DO>, BH * p.q_blocks, pair_smem<HD, 4>(), stream, p, 128 * kPairs);
    } else {
        p.q_blocks = (p.Lq + 16 * NW - 1) / (16 * NW);
        return launch(bwd_row_f32x3_kernel<HD, DT, HAS_DO, HAS_G, NW>, BH * p.q_blocks, TriSmem<HD, HAS_G ? 4 : 2>::bytes, stream, p, 64 * NW);
    }
}

template <int HD, int DT, bool HAS_DO, bool HAS_G, int NW>
int col_one(BwdParamsF32 p, int BH, hipStream_t stream) {
    if constexpr (HD == 128 && HAS_G) {
        p.k_blocks = (p.Lk + 16 * kPairs - 1) / (16 * kPairs);
        return launch(bwd_col_f32x3_pair_kernel<HD, DT, HAS_DO>, BH * p.k_blocks, pair_smem<HD, HAS_DO ? 4 : 3>(), stream, p, 128 * kPairs);
    } else {
        p.k_blocks = (p.Lk + 16 * NW - 1) / (16 * NW);
        return launch(bwd_col_f32x3_kernel<HD, DT, HAS_DO, HAS_G, NW>, BH * p.k_blocks, TriSmem<HD, HAS_G ? (HAS_DO ? 4 : 3) : 2>::bytes, stream, p, 64 * NW);
    }
}

// Calls f with the waves of a workgroup (TWO: one of both forms, else four).
template <bool TWO, typename F>
int by_waves(int waves, F&& f) {
    if constexpr (TWO) {
        if (waves == 8) return f(std::integral_constant<int, 8>{});
    }
    return f(std::integral_constant<int, 4>{});
}

template <typename F>
int by_head(int D, F&& f) {
    using std::integral_constant;
    if (D <= 16) return f(integral_constant<int, 32>{}, integral_constant<int, 1>{});
    if (D <= 32) return f(integral_constant<int, 32>{}, integral_constant<int, 2>{});
    if (D <= 48) return f(integral_constant<int, 64>{}, integral_constant<int, 3>{});
    if (D <= 64) return f(integral_constant<int, 64>{}, integral_constant<int, 4>{});
    if (D <= 96) return f(integral_constant<int, 128>{}, integral_constant<int, 6>{});
    return f(integral_constant<int, 128>{}, integral_constant<int, 8>{});
}

}  // namespace

int fwd_f32x3(const FwdParamsF32& p, int BH, bool jvp, int waves, hipStream_t stream) {
    return by_head(p.D, [&](auto hd, auto dt) {
        constexpr int HD = decltype(hd)::value, DT = decltype(dt)::value;
        return by_waves<HD <= 64>(waves, [&](auto nw) {
            constexpr int NW = decltype(nw)::value;
            return jvp ? fwd_one<HD, DT, true, NW>(p, BH, stream) : fwd_one<HD, DT, false, NW>(p, BH, stream);
        });
    });
}

int bwd_f32x3(const BwdParamsF32& p, int BH, bool has_do, bool has_g, int part, int waves, hipStream_t stream) {
    return by_head(p.D, [&](auto hd, auto dt) {
        constexpr int HD = decltype(hd)::value, DT = decltype(dt)::value;
        auto go = [&](auto d, auto g) {
            constexpr bool DO = decltype(d)::value, G = decltype(g)::value;
            return by_waves<HD == 64 && G>(waves, [&](auto nw) {
                constexpr int NW = decltype(nw)::value;
                if (part == SJVP_BWD_ROW) return row_one<HD, DT, DO, G, NW>(p, BH, stream);
                return col_one<HD, DT, DO, G, NW>(p, BH, stream);
            });
        };
        if (has_do && has_g) return go(std::true_type{}, std::true_type{});
        if (has_g) return go(std::false_type{}, std::true_type{});
        return go(std::true_type{}, std::false_type{});
    });
}

}  // namespace sjvp
