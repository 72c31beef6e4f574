// Translation unit: the 16-wide forward on fp32 tensors with bf16 arithmetic: inputs are rounded to bf16 on their
// way into registers and LDS and results are stored as fp32, which folds the casts that
// semicat/jvp_utils/functional.py:318-322,330-331 performs around the op for fp32 callers.
#include "sjvp_fwd16_staged.hpp"

namespace sjvp {

int fwd_f32io(const FwdParams& p, int grid, bool jvp, hipStream_t stream) {
    return fwd16_staged<Bf16, kIoF32>(p, grid, jvp, stream);
}

}  // namespace sjvp
