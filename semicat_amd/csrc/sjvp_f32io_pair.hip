// Translation unit: the 16-wide backward pair on fp32 tensors with bf16 arithmetic (see sjvp_f32io.hip).
#include "sjvp_pair16.hpp"

namespace sjvp {

int bwd_pair_f32io(const BwdParams& p, int BH, bool has_do, bool has_g, int parts, hipStream_t stream) {
    return bwd_pair16<Bf16, kIoF32>(p, BH, has_do, has_g, parts, stream);
}

}  // namespace sjvp
