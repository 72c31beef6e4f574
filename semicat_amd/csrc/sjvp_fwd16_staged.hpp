// Launch of the 16-wide forward on tensors whose stages are copied through registers (IO = kIoAny, kIoF32,
// sjvp_staged16.hpp).
#pragma once
#include "sjvp_fwd16.hpp"
#include "sjvp_launch.hpp"

namespace sjvp {

template <typename T, int HD, int IO, int DT = HD / 16>
int fwd16_staged_hd(const FwdParams& p, int grid, bool jvp, hipStream_t stream) {
    // the smallest rings whose LDS also holds the store staging tiles
    constexpr int RJ = 2, RP = 4;
    constexpr int OCC = HD == 128 || IO == kIoF32 ? 2 : 4;
    if constexpr (HD <= 64 && IO != kIoF32) {
        const int split = p.Lk > kOwned16 ? split_rows(grid, (p.Lk + kStageRows - 1) / kStageRows, 4, false) : 1;
        FwdParams ps = p;
        ps.q_blocks *= split;
        auto go = [&](auto jvp_tag, auto split_tag) {
            constexpr bool JVP = decltype(jvp_tag)::value;
            constexpr int SPLIT = decltype(split_tag)::value;
            return launch(fwd16_kernel<T, HD, 2 * SPLIT, JVP, 2, SPLIT, false, IO, 1, SPLIT, DT>, grid * SPLIT,
                          Fwd16Smem<HD, 2 * SPLIT, JVP, SPLIT, false, SPLIT>::bytes, stream, ps, kThreads16);
        };
        constexpr std::integral_constant<int, 2> two{};
        constexpr std::integral_constant<int, 4> four{};
        if (split == 2) return jvp ? go(std::true_type{}, two) : go(std::false_type{}, two);
        if (split == 4) return jvp ? go(std::true_type{}, four) : go(std::false_type{}, four);
    }
    if (jvp)
        return launch(fwd16_kernel<T, HD, RJ, true, OCC, 1, false, IO, 1, 1, DT>, grid,
                      Fwd16Smem<HD, RJ, true, 1, false>::bytes, stream, p, kThreads16);
    return launch(fwd16_kernel<T, HD, RP, false, OCC, 1, false, IO, 1, 1, DT>, grid,
                  Fwd16Smem<HD, RP, false, 1, false>::bytes, stream, p, kThreads16);
}

template <typename T, int IO>
int fwd16_staged(const FwdParams& p, int grid, bool jvp, hipStream_t stream) {
    if constexpr (IO != kIoF32) {
        if (p.D <= 16) return fwd16_staged_hd<T, 32, IO, 1>(p, grid, jvp, stream);
    }
    if (p.D <= 32) return fwd16_staged_hd<T, 32, IO>(p, grid, jvp, stream);
    if constexpr (IO != kIoF32) {
        if (p.D <= 48) return fwd16_staged_hd<T, 64, IO, 3>(p, grid, jvp, stream);
    }
    if (p.D <= 64) return fwd16_staged_hd<T, 64, IO>(p, grid, jvp, stream);
    if constexpr (IO != kIoF32) {
        if (p.D <= 96) return fwd16_staged_hd<T, 128, IO, 6>(p, grid, jvp, stream);
    }
    return fwd16_staged_hd<T, 128, IO>(p, grid, jvp, stream);
}

}  // namespace sjvp
