// Translation unit: 16-wide forward on 16-bit rows of any alignment for one element type (SJVP_T).
#include "sjvp_fwd16_staged.hpp"

namespace sjvp {

template <>
int fwd_any<SJVP_T>(const FwdParams& p, int grid, bool jvp, hipStream_t stream) {
    return fwd16_staged<SJVP_T, kIoAny>(p, grid, jvp, stream);
}

}  // namespace sjvp
