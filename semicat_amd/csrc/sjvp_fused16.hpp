// Launches of the single-launch backward (short key axes), for every way the tensors may lie in memory (IO,
// sjvp_staged16.hpp).
#pragma once
#include "sjvp_bwd16.hpp"
#include "sjvp_launch.hpp"

namespace sjvp {

constexpr int kRingFused = 3;

template <typename T, int HD, bool HAS_DO, bool HAS_G, int IO>
int fused_mode(const BwdParams& p, int BH, hipStream_t stream) {
    if constexpr (HD == 64 && IO == kIoDma) {
        if (p.rope.cos)  // rotary embedding folded in
            return launch(bwd_fused16_kernel<T, HD, kRingFused, HAS_DO, HAS_G, true>, BH,
                          Fused16Smem<HD, kRingFused, HAS_DO, HAS_G>::bytes, stream, p, kThreads16);
    }
    return launch(bwd_fused16_kernel<T, HD, kRingFused, HAS_DO, HAS_G, false, IO>, BH,
                  Fused16Smem<HD, kRingFused, HAS_DO, HAS_G>::bytes, stream, p, kThreads16);
}

template <typename T, int HD, int IO>
int fused_hd(const BwdParams& p, int BH, bool has_do, bool has_g, hipStream_t stream) {
    if (has_do && has_g) return fused_mode<T, HD, true, true, IO>(p, BH, stream);
    if (has_g) return fused_mode<T, HD, false, true, IO>(p, BH, stream);
    return fused_mode<T, HD, true, false, IO>(p, BH, stream);
}

template <typename T, int IO>
int bwd_fused16(const BwdParams& p, int BH, bool has_do, bool has_g, hipStream_t stream) {
    if (p.D <= 32) return fused_hd<T, 32, IO>(p, BH, has_do, has_g, stream);
    return fused_hd<T, 64, IO>(p, BH, has_do, has_g, stream);
}

}  // namespace sjvp
