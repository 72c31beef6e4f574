// Translation unit: dense tensors between fp32 and a 16-bit type, up to 16 of them in one launch.
//
// Pure streaming: 6 bytes per element.  A workgroup takes 8192 consecutive elements of one tensor, a thread eight at a
// time: two 16-byte loads and one 16-byte store, or the other way round.  Rounds to nearest even, as PyTorch's casts do.
// Measured on sixteen tensors of 6.3 M elements, what the float32 callers of the op at B=64 H=12 L=128 D=64 cast (604 MB):
// 124 us in four launches (6, 2, 2, 6), 4.9 TB/s, where a large copy reaches 5.1 to 5.3; PyTorch's multi-tensor copies take
// 178 us in six.  The op with its casts 252 -> 198 us of kernels.
#include "sjvp_launch.hpp"

namespace {

using namespace sjvp;

constexpr int kThreads = 256, kPerThread = 8, kSteps = 4;
constexpr int kPerBlock = kThreads * kPerThread * kSteps;

struct CastParams {
    const void* x[SJVP_CAST_MAX];
    void* y[SJVP_CAST_MAX];
    int64_t count[SJVP_CAST_MAX];
    int end[SJVP_CAST_MAX];  // workgroups up to and including the tensor
};

template <typename T, bool WIDEN>
__device__ __forceinline__ void cast_one(const void* x, void* y, int64_t i) {
    if constexpr (WIDEN) {
        static_cast<float*>(y)[i] = T::to_float(static_cast<const elem_t*>(x)[i]);
    } else {
        static_cast<elem_t*>(y)[i] = (elem_t)(T::pack2(static_cast<const float*>(x)[i], 0.f) & 0xffffu);
    }
}

// T: the 16-bit type; WIDEN: from it to fp32
template <typename T, bool WIDEN>
__global__ __launch_bounds__(kThreads) void cast_kernel(const CastParams p) {
    int k = 0;
    while ((int)blockIdx.x >= p.end[k]) ++k;  // the grid ends with the last tensor's workgroups
    const int block = (int)blockIdx.x - (k ? p.end[k - 1] : 0);
    const void* x = p.x[k];
    void* y = p.y[k];
    const int64_t count = p.count[k];
    const bool aligned = ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(y)) & 15u) == 0;
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
        const int64_t i = (int64_t)block * kPerBlock + (s * kThreads + (int)threadIdx.x) * kPerThread;
        if (aligned && i + kPerThread <= count) {
            if constexpr (WIDEN) {
                const u32x4 v = *reinterpret_cast<const u32x4*>(static_cast<const elem_t*>(x) + i);
                f32x4 lo, hi;
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    lo[2 * e] = T::to_float((elem_t)(v[e] & 0xffffu));
                    lo[2 * e + 1] = T::to_float((elem_t)(v[e] >> 16));
                    hi[2 * e] = T::to_float((elem_t)(v[2 + e] & 0xffffu));
                    hi[2 * e + 1] = T::to_float((elem_t)(v[2 + e] >> 16));
                }
                f32x4* out = reinterpret_cast<f32x4*>(static_cast<float*>(y) + i);
                out[0] = lo;
                out[1] = hi;
            } else {
                const f32x4* in = reinterpret_cast<const f32x4*>(static_cast<const float*>(x) + i);
                const f32x4 lo = in[0], hi = in[1];
                *reinterpret_cast<u32x4*>(static_cast<elem_t*>(y) + i) =
                    u32x4{T::pack2(lo[0], lo[1]), T::pack2(lo[2], lo[3]), T::pack2(hi[0], hi[1]), T::pack2(hi[2], hi[3])};
            }
        } else {
            for (int e = 0; e < kPerThread; ++e)
                if (i + e < count) cast_one<T, WIDEN>(x, y, i + e);
        }
    }
}

}  // namespace

extern "C" int sjvp_cast(int n, const void* const* x, void* const* y, const int64_t* count, int in_dtype, int out_dtype,
                         void* stream) {
    if (!x || !y || !count) return SJVP_ERR_NULL;
    if (n < 1 || n > SJVP_CAST_MAX) return SJVP_ERR_SHAPE;
    const bool widen = out_dtype == SJVP_FP32;
    const int half = widen ? in_dtype : out_dtype;
    if ((!widen && in_dtype != SJVP_FP32) || (half != SJVP_BF16 && half != SJVP_FP16)) return SJVP_ERR_DTYPE;
    CastParams p{};
    int64_t blocks = 0;
    for (int i = 0; i < n; ++i) {
        if (count[i] < 0) return SJVP_ERR_SHAPE;
        if (count[i] > 0 && (!x[i] || !y[i])) return SJVP_ERR_NULL;
        p.x[i] = x[i];
        p.y[i] = y[i];
        p.count[i] = count[i];
        blocks += (count[i] + kPerBlock - 1) / kPerBlock;
        if (blocks > 0x7fffffffLL) return SJVP_ERR_SHAPE;
        p.end[i] = (int)blocks;
    }
    if (blocks == 0) return SJVP_OK;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (half == SJVP_BF16)
        return widen ? launch(cast_kernel<Bf16, true>, (int)blocks, 0, s, p, kThreads)
                     : launch(cast_kernel<Bf16, false>, (int)blocks, 0, s, p, kThreads);
    return widen ? launch(cast_kernel<Fp16, true>, (int)blocks, 0, s, p, kThreads)
                 : launch(cast_kernel<Fp16, false>, (int)blocks, 0, s, p, kThreads);
}
