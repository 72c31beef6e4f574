// Translation unit: single-launch backward (short key axes) for one element type (SJVP_T).
#include "sjvp_fused16.hpp"

namespace sjvp {

template <>
int bwd_fused<SJVP_T>(const BwdParams& p, int BH, bool has_do, bool has_g, hipStream_t stream) {
    return bwd_fused16<SJVP_T, kIoDma>(p, BH, has_do, has_g, stream);
}

}  // namespace sjvp
