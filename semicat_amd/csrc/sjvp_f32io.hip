// Translation unit: the 16-wide forward and single-launch backward on fp32 tensors with bf16 arithmetic: inputs are rounded to bf16 on their
// way into registers and LDS and results are stored as fp32, which folds the casts that
// semicat/jvp_utils/functional.py:318-322,330-331 performs around the op for fp32 callers.
#include "sjvp_fused16.hpp"
#include "sjvp_fwd16_staged.hpp"

namespace sjvp {

int fwd_f32io(const FwdParams& p, int grid, bool jvp, hipStream_t stream) {
    return fwd16_staged<Bf16, kIoF32>(p, grid, jvp, stream);
}

int bwd_fused_f32io(const BwdParams& p, int BH, bool has_do, bool has_g, hipStream_t stream) {
    return bwd_fused16<Bf16, kIoF32>(p, BH, has_do, has_g, stream);
}

}  // namespace sjvp
