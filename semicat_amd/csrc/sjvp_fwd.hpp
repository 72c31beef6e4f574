// Parameters of the attention-JVP forward kernels (sjvp_fwd16.hpp), gfx950.
#pragma once
#include "sjvp_device.hpp"

namespace sjvp {

struct FwdParams {
    TensorView q, k, v, tq, tk, tv;
    OutView o, to;
    float* lse;
    float* mu;
    float* li;
    int H, Lq, Lk, D, Lr;
    int q_blocks;  // workgroups per (batch, head): Lr / 128
    float scale;
    int vec;  // all tensors 16-byte aligned, strides % 8 == 0, D % 8 == 0
    RopeTables rope;  // rotation of q, k (and their tangents) as they are loaded; cos == null: none
};

// The reference maximum of the online softmax is only raised when a new tile exceeds it by more
// than this many log2 units.  Any reference point is valid as long as exp2 stays in range: the
// unnormalised probabilities are then bounded by 2^kMaxSlack instead of 1 and the final division
// by the exp-sum is unaffected.  This keeps the accumulator rescale out of almost every tile.
constexpr float kMaxSlack = 6.0f;

}  // namespace sjvp
