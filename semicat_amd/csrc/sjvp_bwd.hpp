// Attention-JVP backward kernels (gfx950): gradients of q, k, v, q_dot, k_dot, v_dot for
// cotangents dO (on O) and G = dTO (on the tangent output), either of which may be absent.
//
// With P = exp(S - lse), N = S_dot - mu, W = G V^T, XY = G V_dot^T + dO V^T and the row sums
// s4 = rowsum(G*O), s7d = rowsum(G*TO) + rowsum(dO*O):
//     dS_dot = P*(W - s4)                    (semicat/jvp_utils/flash_jvp_backward.py:251-257)
//     dS     = dS_dot*N + P*(XY - s7d)       (flash_jvp_backward.py:1364-1407 plus the primal term
//                                             of semicat/jvp_utils/flash_attn_triton.py:606)
//     P_dot  = P*N                           (flash_jvp_backward.py:947-954)
//     dV_dot = P^T G            dV = P_dot^T G + P^T dO
//     dK_dot = s dS_dot^T Q     dK = s (dS^T Q + dS_dot^T Q_dot)
//     dQ_dot = s dS_dot K       dQ = s (dS K + dS_dot K_dot)
// The reference spends eight launches and 35 tile contractions on this; here it is one launch (sjvp_bwd16.hpp, short
// key axes) or two (sjvp_bwd16x.hpp): a row-owned one -> dQ, dQ_dot, which also forms s4 and s7d for its rows
// from O, TO, dO, G (O(L*D) work instead of five contractions) and leaves them, with lse in log2 units, in the
// workspace, and a column-owned one -> dK, dV, dK_dot, dV_dot.  Each gradient is accumulated in fp32 registers
// by exactly one wavefront and written once, so the result is deterministic and never round-trips through
// 16-bit partial sums.
#pragma once
#include "sjvp_device.hpp"

namespace sjvp {

struct BwdParams {
    TensorView q, k, v, tq, tk, tv, o, to, dO, dTO;
    OutView dq, dk, dv, dtq, dtk, dtv;
    const float* lse;
    const float* mu;
    float* lse2;  // workspace [B*H][Lr]  lse * log2(e)
    float* s4;    // workspace [B*H][Lr]  rowsum(G*O)
    float* s7d;   // workspace [B*H][Lr]  rowsum(G*TO) + rowsum(dO*O)
    int H, Lq, Lk, D, Lr;
    // Set by the host where every query-side input (q, q_dot, o, o_dot, dO, dO_dot as present) has q's strides,
    // resp. every key-side input k's, and a row's byte offset inside its (batch, head) slice fits 31 bits: the
    // 16-wide row-owned and column-owned kernels then address their own rows from one offset.
    int q_side_uniform, k_side_uniform;
    int col_workgroups;  // workgroups of the column-owned pass in a launch that also holds others (set by its launcher)
    float scale;
    int vec;
    RopeTables rope;  // q, k (and tangents) are rotated as they are loaded, their gradients rotated back
    int* flags;        // workspace [B*H][Lr/64]: row-owned workgroups whose rows need the second launch
    int rowfix;        // second launch of the row-owned kernel: 0 never, 1 flagged workgroups, 2 always
    float rowfix_tau;  // a residue counts once it exceeds this fraction of the row's absolute tile sum
};

}  // namespace sjvp
