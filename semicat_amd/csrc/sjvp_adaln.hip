// The element-wise parts of an adaLN-modulated transformer block (semicat/net/duo.py:101-166) with their
// forward-mode tangents and the reverse mode of both:
//
//   y = a gate + x                     gated residual            (skipped when a is absent: y = x)
//   h = LN(y; w, b) (1 + scale) + shift    LayerNorm, modulation     (skipped when w is absent)
//
// x, a [B,S,W]; gate, scale, shift [B,W] (rows of one modulation projection, any row stride); bf16 storage, fp32
// arithmetic, each output rounded once.  gelu_kernel is the MLP's tanh GELU in the same manner.
//
// Bound by memory (forward with tangents: 4 rows read, 4 written per position) and, at the sizes of a training
// step, by launches: PyTorch's forward-mode LayerNorm alone is some twenty kernels and twice as many in reverse.
// A wave owns whole rows, kept in registers from the load to the store (W <= 1024: 4 to 16 columns per lane, in
// pieces of 4 = 8 bytes, so that 768 columns are three full pieces per lane), so row statistics are wave
// reductions without a barrier and a row is read once.  In reverse mode a workgroup owns up to 16 rows of one
// sample and every lane keeps the column sums of its columns in registers over its rows; six of them are
// enough for the gradients of gate, scale, shift, their tangents, w and b.  They leave as one partial row per
// workgroup, which two small launches reduce in a fixed order (no atomics: results repeat bit by bit).
// Measured at W = 768, S = 128, gated residual + norm: forward with tangents (B = 16, 25 MB) 15.9 us, reverse (38 MB)
// 27.3; reverse without tangents (B = 48, 57 MB) 25.1 us = 2.3 TB/s.  The reverse is short of waves (one or two
// workgroups per compute unit) and waits for its chain of row reductions.  gelu_kernel averages 12.8 us forward and
// 21.2 us in reverse over the step's two shares.  In the place of PyTorch's kernels: LM1B training step 98 -> 67 ms.
#include <type_traits>

#include "../../include/sjvp.h"
#include "sjvp_device.hpp"

namespace sjvp {
namespace {

constexpr int kWaves = 4;
constexpr int kSums = 6;  // dh.xhat + dth.txhat | dh | dth.xhat | dth | dy.a + dty.ta | dty.a
constexpr int kMaxW = 1024;

struct AdaParams {
    sjvp_adaln t;
    int rows_per_block, chunks;  // reverse mode
    float* col_partial;          // [B][2][W]: each sample's share of dw, db
};

// Sum over the wave, in every lane: DPP moves within rows of 16 lanes, then one read of each row.  Six exchanges through
// LDS, each waiting for the one before, took longer: W = 768, S = 128, B = 16, reverse of the norm 13.1 -> 8.9 us, of
// gated residual + norm 15.9 -> 14.2, with tangents 28.8 -> 27.3; forward (B = 48) 16.0 -> 13.7.
__device__ __forceinline__ float wave_sum(float v) {
    auto dpp = [&](auto ctrl) {
        return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), decltype(ctrl)::value, 0xF,
                                                                     0xF, true));
    };
    v += dpp(std::integral_constant<int, 0xB1>{});   // quad_perm [1,0,3,2]
    v += dpp(std::integral_constant<int, 0x4E>{});   // quad_perm [2,3,0,1]
    v += dpp(std::integral_constant<int, 0x141>{});  // row_half_mirror
    v += dpp(std::integral_constant<int, 0x140>{});  // row_mirror
    auto row = [&](int lane) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane)); };
    return (row(0) + row(16)) + (row(32) + row(48));
}

// One lane's columns of a row: piece i holds columns 4 (lane + 64 i) ...
template <int NV>
struct Row {
    float v[NV * 4];
    __device__ __forceinline__ void zero() {
#pragma unroll
        for (int i = 0; i < NV * 4; ++i) v[i] = 0.f;
    }
    __device__ __forceinline__ void load(const void* base, int64_t at, int lane, int W) {
        const elem_t* p = static_cast<const elem_t*>(base);
        zero();
        if (!p) return;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int c = 4 * (lane + 64 * i);
            if (c < W) {
                const u32x2 r = *reinterpret_cast<const u32x2*>(p + at + c);
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    v[4 * i + 2 * j] = Bf16::to_float((elem_t)(r[j] & 0xffffu));
                    v[4 * i + 2 * j + 1] = Bf16::to_float((elem_t)(r[j] >> 16));
                }
            }
        }
    }
    __device__ __forceinline__ void load32(const float* p, int lane, int W) {
        zero();
        if (!p) return;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int c = 4 * (lane + 64 * i);
            if (c < W) {
                const f32x4 r = *reinterpret_cast<const f32x4*>(p + c);
#pragma unroll
                for (int j = 0; j < 4; ++j) v[4 * i + j] = r[j];
            }
        }
    }
    __device__ __forceinline__ void store(void* base, int64_t at, int lane, int W) const {
        elem_t* p = static_cast<elem_t*>(base);
        if (!p) return;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int c = 4 * (lane + 64 * i);
            if (c < W)
                *reinterpret_cast<u32x2*>(p + at + c) =
                    u32x2{Bf16::pack2(v[4 * i], v[4 * i + 1]), Bf16::pack2(v[4 * i + 2], v[4 * i + 3])};
        }
    }
    // the values that a store and a load would leave
    __device__ __forceinline__ void round() {
#pragma unroll
        for (int i = 0; i < NV * 4; ++i) v[i] = Bf16::to_float((elem_t)(Bf16::pack2(v[i], 0.f) & 0xffffu));
    }
};

// xhat = (y - mean) / sqrt(var + eps); columns beyond W stay 0.  Two passes over registers.
template <int NV>
__device__ __forceinline__ float normalise(const Row<NV>& y, Row<NV>& xhat, int lane, int W, float eps) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < NV * 4; ++i) s += y.v[i];
    const float mean = wave_sum(s) / W;
    float q = 0.f;
#pragma unroll
    for (int i = 0; i < NV * 4; ++i) {
        xhat.v[i] = 4 * (lane + 64 * (i / 4)) < W ? y.v[i] - mean : 0.f;
        q += xhat.v[i] * xhat.v[i];
    }
    const float r = 1.f / sqrtf(wave_sum(q) / W + eps);
#pragma unroll
    for (int i = 0; i < NV * 4; ++i) xhat.v[i] *= r;
    return r;
}

// r (t - mean t - xhat mean(xhat t)): the derivative of xhat, symmetric in its direction; returns mean(xhat t).
template <int NV>
__device__ __forceinline__ float project(const Row<NV>& t, const Row<NV>& xhat, Row<NV>& out, float r, int lane,
                                         int W) {
    float s = 0.f, d = 0.f;
#pragma unroll
    for (int i = 0; i < NV * 4; ++i) {
        s += t.v[i];
        d += t.v[i] * xhat.v[i];
    }
    const float mean = wave_sum(s) / W, dot = wave_sum(d) / W;
#pragma unroll
    for (int i = 0; i < NV * 4; ++i)
        out.v[i] = 4 * (lane + 64 * (i / 4)) < W ? r * (t.v[i] - mean - xhat.v[i] * dot) : 0.f;
    return dot;
}

template <int NV, bool GATE, bool NORM, bool JVP>
__global__ __launch_bounds__(64 * kWaves) void adaln_fwd_kernel(AdaParams p) {
    const sjvp_adaln& t = p.t;
    const int lane = threadIdx.x & 63, W = t.W;
    const int64_t row = (int64_t)blockIdx.x * kWaves + (threadIdx.x >> 6);
    if (row >= (int64_t)t.B * t.S) return;
    const int64_t b = row / t.S, at = row * W;
    Row<NV> y, ty, m;
    y.load(t.x, at, lane, W);
    if constexpr (JVP) ty.load(t.tx, at, lane, W);
    if constexpr (GATE) {
        Row<NV> a, g;
        a.load(t.a, at, lane, W);
        g.load(t.gate, b * t.mod_stride[0], lane, W);
#pragma unroll
        for (int i = 0; i < NV * 4; ++i) y.v[i] += a.v[i] * g.v[i];
        y.round();
        y.store(t.y, at, lane, W);
        if constexpr (JVP) {
            m.load(t.tgate, b * t.mod_stride[1], lane, W);
#pragma unroll
            for (int i = 0; i < NV * 4; ++i) ty.v[i] += a.v[i] * m.v[i];
            a.load(t.ta, at, lane, W);
#pragma unroll
            for (int i = 0; i < NV * 4; ++i) ty.v[i] += a.v[i] * g.v[i];
            ty.round();
            ty.store(t.ty, at, lane, W);
        }
    }
    if constexpr (NORM) {
        Row<NV> xhat, w, bias, sc, h;
        w.load32(t.w, lane, W);
        bias.load32(t.b, lane, W);
        sc.load(t.scale, b * t.mod_stride[2], lane, W);
        m.load(t.shift, b * t.mod_stride[4], lane, W);
        const float r = normalise(y, xhat, lane, W, t.eps);
#pragma unroll
        for (int i = 0; i < NV * 4; ++i) h.v[i] = (xhat.v[i] * w.v[i] + bias.v[i]) * (1.f + sc.v[i]) + m.v[i];
        h.store(t.h, at, lane, W);
        if constexpr (JVP) {
            Row<NV> txhat;
            project(ty, xhat, txhat, r, lane, W);
            m.load(t.tshift, b * t.mod_stride[5], lane, W);
            h.load(t.tscale, b * t.mod_stride[3], lane, W);
#pragma unroll
            for (int i = 0; i < NV * 4; ++i)
                h.v[i] = txhat.v[i] * w.v[i] * (1.f + sc.v[i]) + (xhat.v[i] * w.v[i] + bias.v[i]) * h.v[i] + m.v[i];
            h.store(t.th, at, lane, W);
        }
    }
}

template <int NV, bool GATE, bool NORM, bool JVP>
__global__ __launch_bounds__(64 * kWaves) void adaln_bwd_kernel(AdaParams p) {
    __shared__ float lds[kWaves][NV * 256];
    const sjvp_adaln& t = p.t;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, W = t.W;
    const int64_t b = blockIdx.x / p.chunks;
    const int chunk = blockIdx.x % p.chunks;
    const int end = min(t.S, (chunk + 1) * p.rows_per_block);
    Row<NV> sums[kSums], w, bias, sc, tsc, g, tg;
#pragma unroll
    for (int s = 0; s < kSums; ++s) sums[s].zero();
    if constexpr (NORM) {
        w.load32(t.w, lane, W);
        bias.load32(t.b, lane, W);
        sc.load(t.scale, b * t.mod_stride[2], lane, W);
        if constexpr (JVP) tsc.load(t.tscale, b * t.mod_stride[3], lane, W);
    }
    if constexpr (GATE) {
        g.load(t.gate, b * t.mod_stride[0], lane, W);
        if constexpr (JVP) tg.load(t.tgate, b * t.mod_stride[1], lane, W);
    }
    for (int s = chunk * p.rows_per_block + wave; s < end; s += kWaves) {
        const int64_t at = (b * t.S + s) * W;
        // every load of the row is issued ahead of its first reduction
        Row<NV> dy, dty, u, dh, e, ty, a, ta;
        if constexpr (NORM) {
            u.load(GATE ? t.y : t.x, at, lane, W);
            if constexpr (JVP) ty.load(GATE ? t.ty : t.tx, at, lane, W);
            dh.load(t.dh, at, lane, W);
            if constexpr (JVP) e.load(t.dth, at, lane, W);
        }
        dy.load(t.dy, at, lane, W);
        if constexpr (JVP) dty.load(t.dty, at, lane, W);
        if constexpr (GATE) {
            a.load(t.a, at, lane, W);
            if constexpr (JVP) ta.load(t.ta, at, lane, W);
        }
        if constexpr (NORM) {
            Row<NV> xhat;
            const float r = normalise(u, xhat, lane, W, t.eps);
#pragma unroll
            for (int i = 0; i < NV * 4; ++i) {
                sums[0].v[i] += dh.v[i] * xhat.v[i];
                sums[1].v[i] += dh.v[i];
                dh.v[i] *= (1.f + sc.v[i]) * w.v[i];  // now the gradient of xhat
            }
            if constexpr (JVP) {
                Row<NV> txhat;
                const float c1 = project(ty, xhat, txhat, r, lane, W);
#pragma unroll
                for (int i = 0; i < NV * 4; ++i) {
                    sums[0].v[i] += e.v[i] * txhat.v[i];
                    sums[2].v[i] += e.v[i] * xhat.v[i];
                    sums[3].v[i] += e.v[i];
                    dh.v[i] += e.v[i] * tsc.v[i] * w.v[i];
                    e.v[i] *= (1.f + sc.v[i]) * w.v[i];  // now the gradient of txhat
                }
                Row<NV> pe;
                const float c2 = project(e, xhat, pe, r, lane, W);
                // txhat = r (ty - mean - xhat c1), xhat = r (y - mean).  PyTorch's reverse mode of the forward-mode
                // LayerNorm holds the statistics mean and r of y constant here; so does this, so that the layer's
                // gradients are the same whichever way it is computed.  r (ty - mean) = txhat + r c1 xhat.
#pragma unroll
                for (int i = 0; i < NV * 4; ++i) {
                    dty.v[i] += pe.v[i];
                    dy.v[i] -= r * (r * c1 * e.v[i] + c2 * (txhat.v[i] + r * c1 * xhat.v[i]));
                }
            }
            Row<NV> pd;
            project(dh, xhat, pd, r, lane, W);
#pragma unroll
            for (int i = 0; i < NV * 4; ++i) dy.v[i] += pd.v[i];
        }
        dy.store(t.dx, at, lane, W);
        if constexpr (JVP) dty.store(t.dtx, at, lane, W);
        if constexpr (GATE) {
            Row<NV> da;
#pragma unroll
            for (int i = 0; i < NV * 4; ++i) {
                sums[4].v[i] += dy.v[i] * a.v[i];
                da.v[i] = dy.v[i] * g.v[i];
            }
            if constexpr (JVP) {
#pragma unroll
                for (int i = 0; i < NV * 4; ++i) {
                    sums[5].v[i] += dty.v[i] * a.v[i];
                    da.v[i] += dty.v[i] * tg.v[i];
                }
#pragma unroll
                for (int i = 0; i < NV * 4; ++i) {
                    sums[4].v[i] += dty.v[i] * ta.v[i];
                    dty.v[i] *= g.v[i];
                }
                dty.store(t.dta, at, lane, W);
            }
            da.store(t.da, at, lane, W);
        }
    }
#pragma unroll
    for (int s = 0; s < kSums; ++s) {
        if (s < 4 ? (!NORM || (s > 1 && !JVP)) : (!GATE || (s > 4 && !JVP))) continue;
#pragma unroll
        for (int i = 0; i < NV; ++i)
            *reinterpret_cast<f32x4*>(&lds[wave][4 * (lane + 64 * i)]) =
                f32x4{sums[s].v[4 * i], sums[s].v[4 * i + 1], sums[s].v[4 * i + 2], sums[s].v[4 * i + 3]};
        workgroup_barrier();
        float* out = t.workspace + ((int64_t)blockIdx.x * kSums + s) * W;
        for (int c = threadIdx.x; c < W; c += 64 * kWaves)
            out[c] = (lds[0][c] + lds[1][c]) + (lds[2][c] + lds[3][c]);
        workgroup_barrier();
    }
}

// One thread per (sample, column): the partial rows of a sample's workgroups, then what the sums stand for.
template <bool gate, bool norm, bool jvp>
__global__ __launch_bounds__(64) void adaln_mod_kernel(AdaParams p) {
    const sjvp_adaln& t = p.t;
    const int c = blockIdx.x * 64 + threadIdx.x, W = t.W;
    const int64_t b = blockIdx.y;
    if (c >= W) return;
    float s[kSums] = {};
    const float* in = t.workspace + b * p.chunks * kSums * W + c;
#pragma unroll 4
    for (int k = 0; k < p.chunks; ++k, in += (int64_t)kSums * W) {
#pragma unroll
        for (int i = 0; i < kSums; ++i)
            if (i < 4 ? (norm && (i < 2 || jvp)) : (gate && (i < 5 || jvp))) s[i] += in[(int64_t)i * W];
    }
    auto put = [&](void* out, float v) {
        if (out) static_cast<elem_t*>(out)[b * W + c] = (elem_t)(Bf16::pack2(v, 0.f) & 0xffffu);
    };
    auto mod = [&](const void* in, int64_t stride) {
        return in ? Bf16::to_float(static_cast<const elem_t*>(in)[b * stride + c]) : 0.f;
    };
    if (gate) {
        put(t.dgate, s[4]);
        put(t.dtgate, s[5]);
    }
    if (norm) {
        const float w = t.w[c], bias = t.b ? t.b[c] : 0.f;
        const float sc = 1.f + mod(t.scale, t.mod_stride[2]), tsc = mod(t.tscale, t.mod_stride[3]);
        put(t.dscale, w * s[0] + bias * s[1]);
        put(t.dshift, s[1]);
        put(t.dtscale, w * s[2] + bias * s[3]);
        put(t.dtshift, s[3]);
        p.col_partial[(b * 2) * W + c] = sc * s[0] + tsc * s[2];
        p.col_partial[(b * 2 + 1) * W + c] = sc * s[1] + tsc * s[3];
    }
}

// dw and db: 32 columns per workgroup, eight threads per column over the samples.
__global__ __launch_bounds__(256) void adaln_col_kernel(AdaParams p) {
    __shared__ float lds[8][32];
    const sjvp_adaln& t = p.t;
    const int W = t.W, c = blockIdx.x * 32 + (threadIdx.x & 31), k = threadIdx.x >> 5;
    float s = 0.f;
    if (c < W)
        for (int b = k; b < t.B; b += 8) s += p.col_partial[((int64_t)b * 2 + blockIdx.y) * W + c];
    lds[k][threadIdx.x & 31] = s;
    workgroup_barrier();
    if (k == 0 && c < W) {
#pragma unroll
        for (int i = 1; i < 8; ++i) s += lds[i][threadIdx.x];
        float* out = blockIdx.y ? t.db : t.dw;
        if (out) out[c] = s;
    }
}

struct Gelu {
    float g, g1, g2;  // value, first and second derivative
};
// 0.5 u (1 + tanh(k (u + c u^3)))
__device__ __forceinline__ Gelu gelu(float u) {
    const float k = 0.7978845608028654f, c = 0.044715f;
    const float z1 = k * (1.f + 3.f * c * u * u), z2 = 6.f * k * c * u;
    const float T = 1.f - 2.f / (__expf(2.f * k * (u + c * u * u * u)) + 1.f), d = 1.f - T * T;
    // (z1^2 alone overflows from 1e10 on, where d is 0)
    return {0.5f * u * (1.f + T), 0.5f * (1.f + T) + 0.5f * u * d * z1, d * (z1 + 0.5f * u * z2) - u * T * (d * z1) * z1};
}

__device__ __forceinline__ void load8(const void* base, int64_t at, float* v) {
    if (!base) {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = 0.f;
        return;
    }
    const u32x4 r = *reinterpret_cast<const u32x4*>(static_cast<const elem_t*>(base) + at);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[2 * i] = Bf16::to_float((elem_t)(r[i] & 0xffffu));
        v[2 * i + 1] = Bf16::to_float((elem_t)(r[i] >> 16));
    }
}
__device__ __forceinline__ void store8(void* base, int64_t at, const float* v) {
    if (!base) return;
    u32x4 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = Bf16::pack2(v[2 * i], v[2 * i + 1]);
    *reinterpret_cast<u32x4*>(static_cast<elem_t*>(base) + at) = r;
}

// forward: y = g(u), ty = g'(u) tu;  reverse: y = du, ty = dtu from the cotangents dy, dty (either may be absent).
// Streaming, 16 bytes per lane and tensor.
template <bool REVERSE>
__global__ __launch_bounds__(256) void gelu_kernel(const void* u, const void* tu, const void* dy, const void* dty,
                                                   void* y, void* ty, int64_t n8) {
    const int64_t i8 = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i8 >= n8) return;
    float x[8], tx[8], a[8], ta[8];
    load8(u, i8 * 8, x);
    load8(tu, i8 * 8, tx);
    if constexpr (REVERSE) {
        load8(dy, i8 * 8, a);
        load8(dty, i8 * 8, ta);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const Gelu f = gelu(x[i]);
        if constexpr (REVERSE) {
            // an absent tangent must not bring in a second derivative
            x[i] = a[i] * f.g1 + (tu && dty ? ta[i] * tx[i] * f.g2 : 0.f);
            tx[i] = ta[i] * f.g1;
        } else {
            x[i] = f.g;
            tx[i] *= f.g1;
        }
    }
    store8(y, i8 * 8, x);
    store8(ty, i8 * 8, tx);
}

// Launch with the status of this launch only (not the thread's sticky last error); the arguments take the types of the
// kernel's parameters.
template <int THREADS = 256, typename... P>
int launch(void (*kernel)(P...), dim3 grid, void* stream, std::type_identity_t<P>... params) {
    void* args[] = {&params...};
    const hipError_t rc = hipLaunchKernel(reinterpret_cast<const void*>(kernel), grid, dim3(THREADS), args, 0,
                                          static_cast<hipStream_t>(stream));
    return rc == hipSuccess ? SJVP_OK : SJVP_ERR_LAUNCH;
}

bool misaligned(const void* p, int bytes) { return reinterpret_cast<uintptr_t>(p) % bytes != 0; }

int check(const sjvp_adaln* t) {
    if (!t || !t->x || (!t->a && !t->w) || (t->a && !t->gate) || (t->w && (!t->scale || !t->shift)))
        return SJVP_ERR_NULL;
    if (t->B < 1 || t->S < 1 || t->W < 4 || t->W > kMaxW || t->W % 4 || t->B > 65535 ||
        (int64_t)t->B * t->S > 0x7fffffffLL)
        return SJVP_ERR_SHAPE;
    const void* p16[] = {t->x,   t->tx,  t->a,  t->ta,  t->gate, t->tgate, t->scale, t->tscale, t->shift, t->tshift,
                         t->y,   t->ty,  t->h,  t->th,  t->dy,   t->dty,   t->dh,    t->dth,    t->dx,    t->dtx,
                         t->da,  t->dta};
    for (const void* p : p16)
        if (misaligned(p, 8)) return SJVP_ERR_SHAPE;
    if (misaligned(t->w, 16) || misaligned(t->b, 16)) return SJVP_ERR_SHAPE;
    for (int64_t s : t->mod_stride)
        if (s % 4) return SJVP_ERR_SHAPE;
    return SJVP_OK;
}

int rows_per_block(const sjvp_adaln& t) {
    // 16 rows keep the partial sums at a tenth of the traffic; with too few of them to occupy the chip, 8
    return (int64_t)t.B * ((t.S + 15) / 16) >= 256 ? 16 : 8;
}
int chunks_of(const sjvp_adaln& t) { return (t.S + rows_per_block(t) - 1) / rows_per_block(t); }

// Calls f with the number of 256-column pieces of a row as a constant.
template <typename F>
int by_width(int W, F&& f) {
    switch ((W + 255) / 256) {
        case 1: return f(std::integral_constant<int, 1>{});
        case 2: return f(std::integral_constant<int, 2>{});
        case 3: return f(std::integral_constant<int, 3>{});
        default: return f(std::integral_constant<int, 4>{});
    }
}

template <bool REVERSE, bool JVP>
int run(const AdaParams& p, dim3 grid, void* stream) {
    return by_width(p.t.W, [&](auto nv) {
        constexpr int NV = decltype(nv)::value;
        if constexpr (REVERSE) {
            if (p.t.a && p.t.w) return launch(adaln_bwd_kernel<NV, true, true, JVP>, grid, stream, p);
            if (p.t.a) return launch(adaln_bwd_kernel<NV, true, false, JVP>, grid, stream, p);
            return launch(adaln_bwd_kernel<NV, false, true, JVP>, grid, stream, p);
        } else {
            if (p.t.a && p.t.w) return launch(adaln_fwd_kernel<NV, true, true, JVP>, grid, stream, p);
            if (p.t.a) return launch(adaln_fwd_kernel<NV, true, false, JVP>, grid, stream, p);
            return launch(adaln_fwd_kernel<NV, false, true, JVP>, grid, stream, p);
        }
    });
}

}  // namespace
}  // namespace sjvp

extern "C" {

using namespace sjvp;

size_t sjvp_adaln_workspace_floats(const sjvp_adaln* t) {
    if (check(t) != SJVP_OK) return 0;
    return ((size_t)t->B * chunks_of(*t) * kSums + (size_t)t->B * 2) * t->W;
}

int sjvp_adaln_fwd(const sjvp_adaln* t, int jvp, void* stream) {
    const int rc = check(t);
    if (rc != SJVP_OK) return rc;
    if ((t->a && (!t->y || (jvp && !t->ty))) || (t->w && (!t->h || (jvp && !t->th)))) return SJVP_ERR_NULL;
    AdaParams p{*t, 0, 0, nullptr};
    const dim3 grid((unsigned)(((int64_t)t->B * t->S + kWaves - 1) / kWaves));
    return jvp ? run<false, true>(p, grid, stream) : run<false, false>(p, grid, stream);
}

int sjvp_adaln_bwd(const sjvp_adaln* t, int jvp, void* stream) {
    int rc = check(t);
    if (rc != SJVP_OK) return rc;
    if (!t->workspace || (t->a && t->w && (!t->y || (jvp && !t->ty)))) return SJVP_ERR_NULL;
    AdaParams p{*t, rows_per_block(*t), chunks_of(*t), nullptr};
    p.col_partial = t->workspace + (size_t)t->B * p.chunks * kSums * t->W;
    const dim3 grid((unsigned)(t->B * p.chunks)), per_column((t->W + 63) / 64, t->B);
    rc = jvp ? run<true, true>(p, grid, stream) : run<true, false>(p, grid, stream);
    if (rc != SJVP_OK) return rc;
    auto columns = [&](auto j) {
        constexpr bool J = decltype(j)::value;
        if (t->a && t->w) return launch<64>(adaln_mod_kernel<true, true, J>, per_column, stream, p);
        if (t->a) return launch<64>(adaln_mod_kernel<true, false, J>, per_column, stream, p);
        return launch<64>(adaln_mod_kernel<false, true, J>, per_column, stream, p);
    };
    rc = jvp ? columns(std::true_type{}) : columns(std::false_type{});
    if (rc != SJVP_OK || !t->w || (!t->dw && !t->db)) return rc;
    return launch(adaln_col_kernel, dim3((t->W + 31) / 32, 2), stream, p);
}

int sjvp_gelu(const void* u, const void* tu, const void* dy, const void* dty, void* y, void* ty, int64_t n,
              int reverse, void* stream) {
    if (!u || (!y && !ty)) return SJVP_ERR_NULL;
    if (n < 8 || n % 8 || n / 8 > (int64_t)0x7fffffff * 256) return SJVP_ERR_SHAPE;
    for (const void* p : {u, tu, dy, dty, (const void*)y, (const void*)ty})
        if (misaligned(p, 16)) return SJVP_ERR_SHAPE;
    const dim3 grid((unsigned)((n / 8 + 255) / 256));
    return reverse ? launch(gelu_kernel<true>, grid, stream, u, tu, dy, dty, y, ty, n / 8)
                   : launch(gelu_kernel<false>, grid, stream, u, tu, dy, dty, y, ty, n / 8);
}

}  // extern "C"
