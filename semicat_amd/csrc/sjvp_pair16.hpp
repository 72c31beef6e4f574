// Launches of the 16-wide row-owned + column-owned backward pair, for every way the tensors may lie in memory
// (IO, sjvp_staged16.hpp).
#pragma once
#include "sjvp_bwd16x.hpp"
#include "sjvp_launch.hpp"

namespace sjvp {

template <typename T, int HD, bool HAS_DO, bool HAS_G, int IO, int DT>
int pair_mode(const BwdParams& p, int BH, int parts, hipStream_t stream) {
    // the row-owned kernel first (besides dQ, dQ_dot it leaves the row sums in the workspace), then
    // the column-owned one; workgroups of four waves own 64 positions
    constexpr int XR = HD == 128 || IO != kIoDma ? 2 : 3;  // ring depth (staged copies run one stage ahead)
    int rc = SJVP_OK;
    bool rides = false;
    if (parts & SJVP_BWD_ROW) {
        // (fp32 rows at HD = 128 are staged in 64 registers: one wave per SIMD, or they spill)
        constexpr int OCC = HD == 128 && IO == kIoF32 ? 1 : HD == 128 || IO != kIoDma ? 2 : 3;
        const int grid = BH * (p.Lr / kXOwned16);
        constexpr int smem = Row16Smem<HD, XR, HAS_G>::bytes;
        // "always": a launch that measures the row-sum residues, then one that computes with the corrected
        // sums; otherwise the pass itself and, unless switched off, a second launch in which the workgroups
        // whose residues call for it run again
        // Without the cotangent on TO a wave has registers for 32 queries, which every operand read from LDS then
        // serves: 78 -> 68 us at B=8 H=16 L=1024 D=64, 120 -> 105 at D=128.  Half as many waves: from four workgroups
        // of 64 queries per compute unit on (1024 of them 0.76 to 1.01 of the time, 512 1.03 to 1.13), and from 256
        // keys on (128 of them 1.02).
        bool wide = false;
        if constexpr (!HAS_G && IO == kIoDma) wide = p.rowfix != 2 && grid >= 4 * compute_units() && p.Lk >= 256;
        int split = 1;
        if constexpr (HD <= 64 && IO != kIoF32) {
            constexpr int MOST = IO == kIoDma ? 4 : 2;  // (four parts' staged copies do not fit the registers)
            if (p.rowfix != 2) split = split_rows(grid, (p.Lk + kStageRows - 1) / kStageRows, MOST, true);
            if (split == 2)
                rc = launch(bwd_row16_kernel<T, HD, 4, HAS_DO, HAS_G, 2, 0, IO, 1, 2, DT>, grid * 2,
                            Row16Smem<HD, 4, HAS_G, 2>::bytes, stream, p, kXThreads16);
            if constexpr (MOST == 4) {
                if (split == 4)
                    rc = launch(bwd_row16_kernel<T, HD, 8, HAS_DO, HAS_G, 2, 0, IO, 1, 4, DT>, grid * 4,
                                Row16Smem<HD, 8, HAS_G, 4>::bytes, stream, p, kXThreads16);
            }
        }
        if (split > 1) {
            // done above
        } else if (wide) {
            if constexpr (!HAS_G && IO == kIoDma)
                rc = launch(bwd_row16_kernel<T, HD, XR, HAS_DO, HAS_G, HD == 128 ? 2 : 3, 0, IO, 2, 1, DT>, grid / 2, smem, stream,
                            p, kXThreads16);
        } else if (p.rowfix == 2) rc = launch(bwd_row16_kernel<T, HD, XR, HAS_DO, HAS_G, OCC, 1, IO, 1, 1, DT>, grid, smem, stream, p, kXThreads16);
        else rc = launch(bwd_row16_kernel<T, HD, XR, HAS_DO, HAS_G, OCC, 0, IO, 1, 1, DT>, grid, smem, stream, p, kXThreads16);
        // The second launch does not depend on the column-owned pass.  Where nearly all of its workgroups leave
        // at once (repair of flagged workgroups only), they ride at the end of that launch instead of paying for
        // one of their own.
        // (not at D = 128 with the cotangent on O only: the row-owned body needs more registers than that
        // column-owned kernel, which would lose a resident workgroup per compute unit to it; nor on fp32 rows there)
        rides = p.rowfix == 1 && (parts & SJVP_BWD_COL) && (HD != 128 || (HAS_G && IO != kIoF32));
        if (rc == SJVP_OK && p.rowfix != 0 && !rides)
            rc = launch(bwd_row16_kernel<T, HD, XR, HAS_DO, HAS_G, OCC, 2, IO, 1, 1, DT>, grid, smem, stream, p, kXThreads16);
    }
    if (rc != SJVP_OK || !(parts & SJVP_BWD_COL)) return rc;
    const int grid = BH * ((p.Lk + kXOwned16 - 1) / kXOwned16);
    using CS = Col16Smem<HD, XR, HAS_DO, HAS_G>;
    if constexpr (HD == 128) {
        // eight waves: wave pairs share 16 keys, split the score-side tiles by query tile and the
        // gradients by head-dimension half (one launch, nothing computed twice)
        constexpr int PR = 2;  // ring depths 2, 3, 4 measure the same (the kernel is issue-bound)
        using PS = Col16pSmem<HD, PR, HAS_DO, HAS_G>;
        if (rides) {
            BwdParams pr = p;
            pr.col_workgroups = grid;
            constexpr int smem = PS::bytes > Row16Smem<HD, XR, HAS_G>::bytes ? PS::bytes : Row16Smem<HD, XR, HAS_G>::bytes;
            return launch(bwd_col16p_repair_kernel<T, HD, PR, XR, HAS_DO, HAS_G, IO, DT>, grid + BH * (p.Lr / kXOwned16), smem,
                          stream, pr, kThreads16);
        }
        return launch(bwd_col16p_kernel<T, HD, PR, HAS_DO, HAS_G, IO, DT>, grid, PS::bytes, stream, p, kThreads16);
    } else {
        if constexpr (HD <= 64 && IO != kIoF32) {
            constexpr int MOST = IO == kIoDma ? 4 : 2;
            // (whether or not the second row launch rides along: dK, dV are the same bits with the repair off, or in a call
            // for this part alone; as in the row launch, "always" keeps to whole workgroups)
            const int split = p.rowfix != 2 ? split_rows(grid, (p.Lq + kStageRows - 1) / kStageRows, MOST, IO == kIoDma) : 1;
            auto go = [&](auto split_tag) {
                constexpr int SPLIT = decltype(split_tag)::value;
                constexpr int OWNED = kXOwned16 / SPLIT;
                BwdParams pr = p;
                pr.col_workgroups = BH * ((p.Lk + OWNED - 1) / OWNED);
                constexpr int row = Row16Smem<HD, XR, HAS_G>::bytes, col = Col16Smem<HD, 2 * SPLIT, HAS_DO, HAS_G, SPLIT>::bytes;
                if (!rides)
                    return launch(bwd_col16_kernel<T, HD, 2 * SPLIT, HAS_DO, HAS_G, 2, IO, 1, SPLIT, DT>, pr.col_workgroups, col,
                                  stream, pr, kXThreads16);
                return launch(bwd_col16_repair_kernel<T, HD, 2 * SPLIT, HAS_DO, HAS_G, 2, IO, 1, SPLIT, XR, DT>,
                              pr.col_workgroups + BH * (p.Lr / kXOwned16), col > row ? col : row, stream, pr, kXThreads16);
            };
            if (split == 2) return go(std::integral_constant<int, 2>{});
            if constexpr (MOST == 4) {
                if (split == 4) return go(std::integral_constant<int, 4>{});
            }
        }
        // 32 keys per wave where the accumulators leave room for them (as in the row-owned launch): 92 -> 80 us at B=8
        // H=16 L=1024 D=64, cotangent on O only, from two workgroups of 64 keys per compute unit on (512 of them 0.96 to
        // 1.01 of the time, 256 1.16 to 1.23); at D = 32 with both cotangents 129 -> 112 us, from 1024 workgroups and
        // 512 queries on (1024 and 256: 0.97 to 1.04).
        if constexpr (IO == kIoDma && (!HAS_G || HD == 32)) {
            const int rounds = grid / compute_units();
            if (rides && (HAS_G ? rounds >= 4 && p.Lq >= 512 : rounds >= 2 && p.Lq >= 256)) {
                BwdParams pr = p;
                pr.col_workgroups = BH * ((p.Lk + 2 * kXOwned16 - 1) / (2 * kXOwned16));
                constexpr int smem = CS::bytes > Row16Smem<HD, XR, HAS_G>::bytes ? CS::bytes : Row16Smem<HD, XR, HAS_G>::bytes;
                return launch(bwd_col16_repair_kernel<T, HD, XR, HAS_DO, HAS_G, 2, IO, 2, 1, XR, DT>,
                              pr.col_workgroups + BH * (p.Lr / kXOwned16), smem, stream, pr, kXThreads16);
            }
        }
        if (rides) {
            BwdParams pr = p;
            pr.col_workgroups = grid;
            constexpr int smem = CS::bytes > Row16Smem<HD, XR, HAS_G>::bytes ? CS::bytes : Row16Smem<HD, XR, HAS_G>::bytes;
            return launch(bwd_col16_repair_kernel<T, HD, XR, HAS_DO, HAS_G, 2, IO, 1, 1, XR, DT>,
                          grid + BH * (p.Lr / kXOwned16), smem, stream, pr, kXThreads16);
        }
        return launch(bwd_col16_kernel<T, HD, XR, HAS_DO, HAS_G, 2, IO, 1, 1, DT>, grid, CS::bytes, stream, p, kXThreads16);
    }
}

template <typename T, int HD, int IO, int DT = HD / 16>
int pair_hd(const BwdParams& p, int BH, bool has_do, bool has_g, int parts, hipStream_t stream) {
    if (has_do && has_g) return pair_mode<T, HD, true, true, IO, DT>(p, BH, parts, stream);
    if (has_g) return pair_mode<T, HD, false, true, IO, DT>(p, BH, parts, stream);
    return pair_mode<T, HD, true, false, IO, DT>(p, BH, parts, stream);
}

template <typename T, int IO>
int bwd_pair16(const BwdParams& p, int BH, bool has_do, bool has_g, int parts, hipStream_t stream) {
    if constexpr (IO != kIoF32) {
        if (p.D <= 16) return pair_hd<T, 32, IO, 1>(p, BH, has_do, has_g, parts, stream);
    }
    if (p.D <= 32) return pair_hd<T, 32, IO>(p, BH, has_do, has_g, parts, stream);
    if constexpr (IO != kIoF32) {
        if (p.D <= 48) return pair_hd<T, 64, IO, 3>(p, BH, has_do, has_g, parts, stream);
    }
    if (p.D <= 64) return pair_hd<T, 64, IO>(p, BH, has_do, has_g, parts, stream);
    if constexpr (IO != kIoF32) {
        if (p.D <= 96) return pair_hd<T, 128, IO, 6>(p, BH, has_do, has_g, parts, stream);
    }
    return pair_hd<T, 128, IO>(p, BH, has_do, has_g, parts, stream);
}

}  // namespace sjvp
