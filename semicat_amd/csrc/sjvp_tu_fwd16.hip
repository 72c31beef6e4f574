// Translation unit: 16-wide forward kernels for one element type (SJVP_T = Bf16 or Fp16).
#include "sjvp_fwd16.hpp"
#include "sjvp_launch.hpp"

namespace sjvp {
namespace {

// Ring depths (stages of 32 keys in flight) per head-dimension class, sized to the LDS a workgroup
// may take when two of them are to share the 160 KB of a CU.
constexpr int kRingJvp = 2;     // with tangents (four slabs per stage)
constexpr int kRingPrimal = 4;  // primal only (two slabs per stage)
// key-axis length from which the forward takes two stages per barrier
constexpr int kFwdPairedFrom = 256;

template <typename T, int HD, int R, bool JVP, int OCC, int SPB = 1, bool ROPE = false, int DT = HD / 16>
int fwd16_one(const FwdParams& p, int grid, hipStream_t stream) {
    constexpr int smem = Fwd16Smem<HD, R, JVP, SPB>::bytes;
    // Without tangents a wave has registers for 32 queries, which every operand read from LDS then serves: 53 -> 48 us at
    // B=8 H=16 L=1024 D=64, 141 -> 134 at B=8 H=8 L=2048 D=128.  Half as many waves: from as many workgroups on as the
    // chip holds (D <= 64: 1024 of them 0.90 to 1.01 of the time, 512 0.97 to 1.08; D = 128: 512 of them from 1024 keys
    // on 0.95 to 0.98, with 256 to 512 keys 1.01 to 1.07).
    if constexpr (!JVP && SPB == 2) {
        const int rounds = grid / compute_units();
        if (HD == 128 ? rounds >= 2 && p.Lk >= 1024 : rounds >= 4)
            return launch(fwd16_kernel<T, HD, R, JVP, HD == 128 ? 2 : 4, SPB, ROPE, kIoDma, 2, 1, DT>, grid, smem, stream, p,
                          kThreads16 / 2);
    }
    if constexpr (HD <= 64 && !ROPE) {
        // (D > 64 is left whole: with tangents at D = 128 the sums of eight waves do not fit the LDS (168 KB); the other forms
        // would fit and have not been measured.  Up to 128 keys the folded rotation is an alternative to this launch, and
        // both round alike.)
        const int split = p.Lk > kOwned16 ? split_rows(grid, (p.Lk + kStageRows - 1) / kStageRows, 4, false) : 1;
        FwdParams ps = p;
        ps.q_blocks *= split;
        if (split == 2)
            return launch(fwd16_kernel<T, HD, 4, JVP, 4, 2, false, kIoDma, 1, 2, DT>, grid * 2,
                          Fwd16Smem<HD, 4, JVP, 2, true, 2>::bytes, stream, ps, kThreads16);
        if (split == 4)
            return launch(fwd16_kernel<T, HD, 8, JVP, 4, 4, false, kIoDma, 1, 4, DT>, grid * 4,
                          Fwd16Smem<HD, 8, JVP, 4, true, 4>::bytes, stream, ps, kThreads16);
    }
    return launch(fwd16_kernel<T, HD, R, JVP, OCC, SPB, ROPE, kIoDma, 1, 1, DT>, grid, smem, stream, p, kThreads16);
}

template <typename T, int HD, int DT = HD / 16>
int fwd16_hd(const FwdParams& p, int grid, bool jvp, hipStream_t stream) {
    // two stages in flight and at most 128 registers: two workgroups (sixteen waves) share a CU, which
    // overlaps one's copies with the other's arithmetic; HD = 128 needs the whole register budget
    constexpr int OCC = HD == 128 ? 2 : 4;
    if constexpr (HD == 64 && DT == 4) {
        if (p.rope.cos)  // rotary embedding folded in (short key axes only, checked by the caller)
            return jvp ? fwd16_one<T, HD, kRingJvp, true, OCC, 1, true>(p, grid, stream)
                       : fwd16_one<T, HD, kRingPrimal, false, OCC, 1, true>(p, grid, stream);
    }
    // long key axes: two stages per barrier over a ring of four slots in the same LDS footprint
    if (p.Lk >= kFwdPairedFrom)
        return jvp ? fwd16_one<T, HD, 4, true, OCC, 2, false, DT>(p, grid, stream) : fwd16_one<T, HD, 4, false, OCC, 2, false, DT>(p, grid, stream);
    return jvp ? fwd16_one<T, HD, kRingJvp, true, OCC, 1, false, DT>(p, grid, stream)
               : fwd16_one<T, HD, kRingPrimal, false, OCC, 1, false, DT>(p, grid, stream);
}

}  // namespace

template <>
int fwd_vec<SJVP_T>(const FwdParams& p, int grid, bool jvp, hipStream_t stream) {
    if (p.D <= 16) return fwd16_hd<SJVP_T, 32, 1>(p, grid, jvp, stream);
    if (p.D <= 32) return fwd16_hd<SJVP_T, 32>(p, grid, jvp, stream);
    if (p.D <= 48) return fwd16_hd<SJVP_T, 64, 3>(p, grid, jvp, stream);
    if (p.D <= 64) return fwd16_hd<SJVP_T, 64>(p, grid, jvp, stream);
    if (p.D <= 96) return fwd16_hd<SJVP_T, 128, 6>(p, grid, jvp, stream);
    return fwd16_hd<SJVP_T, 128>(p, grid, jvp, stream);
}

}  // namespace sjvp
