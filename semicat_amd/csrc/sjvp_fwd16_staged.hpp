// Launch of the 16-wide forward on tensors whose stages are copied through registers (IO = kIoAny, kIoF32,
// sjvp_staged16.hpp).
#pragma once
#include "sjvp_fwd16.hpp"
#include "sjvp_launch.hpp"

namespace sjvp {

template <typename T, int HD, int IO>
int fwd16_staged_hd(const FwdParams& p, int grid, bool jvp, hipStream_t stream) {
    // the smallest rings whose LDS also holds the store staging tiles
    constexpr int RJ = 2, RP = 4;
    constexpr int OCC = HD == 128 || IO == kIoF32 ? 2 : 4;
    if (jvp)
        return launch(fwd16_kernel<T, HD, RJ, true, OCC, 1, false, IO>, grid, Fwd16Smem<HD, RJ, true, 1, false>::bytes,
                      stream, p, kThreads16);
    return launch(fwd16_kernel<T, HD, RP, false, OCC, 1, false, IO>, grid, Fwd16Smem<HD, RP, false, 1, false>::bytes,
                  stream, p, kThreads16);
}

template <typename T, int IO>
int fwd16_staged(const FwdParams& p, int grid, bool jvp, hipStream_t stream) {
    if (p.D <= 32) return fwd16_staged_hd<T, 32, IO>(p, grid, jvp, stream);
    if (p.D <= 64) return fwd16_staged_hd<T, 64, IO>(p, grid, jvp, stream);
    return fwd16_staged_hd<T, 128, IO>(p, grid, jvp, stream);
}

}  // namespace sjvp
