// Translation unit: 16-wide row-owned + column-owned backward pair on 16-byte aligned rows for one element type
// (SJVP_T).
#include "sjvp_pair16.hpp"

namespace sjvp {

template <>
int bwd_pair_vec<SJVP_T>(const BwdParams& p, int BH, bool has_do, bool has_g, int parts, hipStream_t stream) {
    return bwd_pair16<SJVP_T, kIoDma>(p, BH, has_do, has_g, parts, stream);
}

}  // namespace sjvp
