// Host-side launch plumbing shared by the translation units of the library: the kernels are
// instantiated per element type in separate units (compiled in parallel), each exporting the
// selection functions declared here; sjvp_api.hip validates arguments and calls them.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>

#include "../../include/sjvp.h"
#include "sjvp_bwd.hpp"
#include "sjvp_f32.hpp"
#include "sjvp_fwd.hpp"

namespace sjvp {

// Launch with the status of this launch only (not the thread's sticky last error).
// A kernel that needs more than 64 KB of LDS has its limit raised first.  K is a function pointer
// type shared by many kernels, so the (kernel, device) pairs already served are remembered in a small
// table: the attribute call, which costs host time on every launch otherwise, runs once per pair.
inline bool lds_limit_raised(const void* kernel, int smem_bytes) {
    constexpr int kSlots = 512;
    struct Slot {
        std::atomic<const void*> kernel{nullptr};
        std::atomic<int> bytes{0};
    };
    static Slot table[kSlots][8];  // open addressing over kernels, by device (devices beyond 8 are not cached)
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return false;
    Slot* hit = nullptr;
    if (dev >= 0 && dev < 8) {
        size_t h = (reinterpret_cast<uintptr_t>(kernel) >> 4) % kSlots;
        for (int probe = 0; probe < kSlots; ++probe, h = (h + 1) % kSlots) {
            Slot& s = table[h][dev];
            const void* cur = s.kernel.load(std::memory_order_acquire);
            if (cur == kernel) {
                if (s.bytes.load(std::memory_order_acquire) >= smem_bytes) return true;
                hit = &s;
                break;
            }
            if (cur == nullptr) {
                const void* expected = nullptr;
                if (s.kernel.compare_exchange_strong(expected, kernel, std::memory_order_acq_rel) || expected == kernel) {
                    hit = &s;
                    break;
                }
            }
        }
    }
    if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, smem_bytes) != hipSuccess) return false;
    if (hit) hit->bytes.store(smem_bytes, std::memory_order_release);
    return true;
}

template <typename K, typename P>
int launch(K kernel, int grid, int smem_bytes, hipStream_t stream, const P& params, int threads) {
    if (smem_bytes > 64 * 1024 && !lds_limit_raised(reinterpret_cast<const void*>(kernel), smem_bytes))
        return SJVP_ERR_LAUNCH;
    P copy = params;
    void* args[] = {&copy};
    const hipError_t rc = hipLaunchKernel(reinterpret_cast<const void*>(kernel), dim3(grid), dim3(threads), args,
                                          (size_t)smem_bytes, stream);
    return rc == hipSuccess ? SJVP_OK : SJVP_ERR_LAUNCH;
}

constexpr int kMaxDevices = 64;

// Compute units of the current device (looked up once per device; 256 for a whole MI355X, fewer for a partition of one).
inline int compute_units() {
    static std::atomic<int> cached[kMaxDevices] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 256;
    int n = cached[dev].load(std::memory_order_relaxed);
    if (n == 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 1) n = 256;
        cached[dev].store(n, std::memory_order_relaxed);
    }
    return n;
}

// Waves that share a group of 16 owned rows (SPLIT of the 16-wide kernels) in a launch of `grid` workgroups that would walk
// `stages` stages each, on `units` compute units.  A workgroup of a launch that does not fill the chip is a serial chain of
// stages; split, it is as many times shorter, plus the exchange of the sums.  So: while every split workgroup still has
// a compute unit of its own, or two share one (`pairs`) and the chain is long.  Times of the split launch over the whole
// one at D = 64: all have a unit 0.49 to 0.89; two to a unit, 16 or 32 stages 0.81 to 0.95, 7 stages 1.05; more 1.1 to 3.5
// (the forward, whose workgroups have eight waves, 1.1 to 1.3 already with two).  The shortest chains that are split, us whole /
// split: row kernel 4 stages in two 8.6 / 7.0, 5 in four 9.8 / 7.6; column kernel 4 in two 8.2 / 6.9, 5 in four 8.8 / 6.6;
// forward 5 in four 8.5 / 7.2, 5 in two 8.9 / 8.4, 6 in two 9.7 / 8.2; rows of odd lengths, row kernel 4 in two
// 11.6 / 9.8, column kernel 10.6 / 9.3.
// Forward + backward, whole / split: B=1 H=8 L=256 33.7 / 21.6 us, B=1 H=4 L=2048 173 / 96, B=1 H=12 L=512 without tangents
// 34.5 / 24.4, B=4 H=6 333 x 205 D=48 cotangent on TO 40.2 / 35.1, B=2 H=12 L=300 D=36 50.8 / 44.1.
inline int split_rows(int64_t grid, int stages, int most, bool pairs, int units = compute_units()) {
    if (most >= 4 && 4 * grid <= units && stages > 4) return 4;
    if (2 * grid <= units && stages > 3) return 2;
    return pairs && grid <= units && stages >= 12 ? 2 : 1;
}

// Forward: stages by LDS-DMA (16-byte aligned rows), or through registers (any alignment).
template <typename T> int fwd_vec(const FwdParams& p, int grid, bool jvp, hipStream_t stream);
template <typename T> int fwd_any(const FwdParams& p, int grid, bool jvp, hipStream_t stream);

// Backward: the single launch (short key axes, D <= 64; 16-byte aligned 16-bit rows: bwd_select keeps others away from it),
// and the row + column pair on rows as above.
template <typename T> int bwd_fused(const BwdParams& p, int BH, bool has_do, bool has_g, hipStream_t stream);
template <typename T> int bwd_pair_vec(const BwdParams& p, int BH, bool has_do, bool has_g, int parts, hipStream_t stream);
template <typename T> int bwd_pair_any(const BwdParams& p, int BH, bool has_do, bool has_g, int parts, hipStream_t stream);

// fp32 tensors with bf16 arithmetic (the cast folded into the loads and stores; rows of any alignment).
// The views carry fp32 pointers cast to elem_t* and strides counted in 2-byte units.
int fwd_f32io(const FwdParams& p, int grid, bool jvp, hipStream_t stream);
int bwd_fused_f32io(const BwdParams& p, int BH, bool has_do, bool has_g, hipStream_t stream);
int bwd_pair_f32io(const BwdParams& p, int BH, bool has_do, bool has_g, int parts, hipStream_t stream);

// fp32 correctness mode: forward, and the row-owned + column-owned backward pair.
int fwd_f32(const FwdParamsF32& p, int BH, bool jvp, hipStream_t stream);
int bwd_f32(const BwdParamsF32& p, int BH, bool has_do, bool has_g, int parts, hipStream_t stream);
// The same on the bf16 matrix pipe, operands in three parts (sjvp_f32x3.hpp), with four or eight waves in a workgroup; the
// two above choose.  `part`: SJVP_BWD_ROW or SJVP_BWD_COL.
int fwd_f32x3(const FwdParamsF32& p, int BH, bool jvp, int waves, hipStream_t stream);
int bwd_f32x3(const BwdParamsF32& p, int BH, bool has_do, bool has_g, int part, int waves, hipStream_t stream);

}  // namespace sjvp
