// family.hip -- ops of the other model families the reference runs through
// the same kernel layer: GELU (tanh form, Gemma), GELU-erf, LayerNorm
// (Whisper, Nomic), causal depthwise conv1d (LFM2) and the 3-tap conv1d
// (Whisper's front end).  Each output follows the reference's operation
// order (lanes, pairwise reductions, fused multiply-adds) bit for bit:
//
//   cactus_gelu_f16 / _erf             kernel_nn.cpp:46-150
//   fast_tanh_f32x4                    kernel_utils.h:143-163
//   compute_layernorm_node             graph_ops_nn.cpp:373-457
//   cactus_conv1d_causal_depthwise_f16 kernel_conv.cpp:15-110
//   cactus_conv1d_f16_k3               kernel_conv.cpp:112-236
//
// These are memory-light element or row operations off the Qwen3 path; one
// thread per output (one lane per row for LayerNorm's sequential sums) keeps
// the reference's order with no cross-lane reduction.  tanhf (the GELU tail)
// and erff are evaluated in double and rounded once to float, the same
// libm boundary as cactus_expf.
#include "hip_common.h"
#include "pointwise_device.h"

namespace cactus_hip {

__device__ __forceinline__ float fast_tanh_f(float x) {
    if (x > 4.5f) return 1.0f;
    if (x < -4.5f) return -1.0f;
    const float x2 = x * x;
    const float num = 27.0f + x2;
    const float den = __builtin_fmaf(9.0f, x2, 27.0f);
    return x * (num / den);
}

struct GeluOp {
    __device__ uint16_t operator()(uint16_t a, uint16_t, bool body) const {
        const float s2pi = 0.7978845608028654f, coeff = 0.044715f;
        const float x = h2f(a);
        float g;
        if (body) {
            const float x3 = (x * x) * x;
            const float inner = s2pi * __builtin_fmaf(coeff, x3, x);
            g = (0.5f * x) * (1.0f + fast_tanh_f(inner));
        } else {
            const float inner = s2pi * __builtin_fmaf((coeff * x) * x, x, x);
            g = (0.5f * x) * (1.0f + (float)tanh((double)inner));
        }
        return f2h(g);
    }
};

// erf(z) in double, rounded to float: |z| Q(z^2) with Q the degree-20
// Chebyshev interpolant of erf(sqrt(t)) / sqrt(t) on [0, 16] (its nodes
// evaluated to 50 digits), as a polynomial in u = t / 8 - 1; |z| >= 4 rounds
// to 1.  Absolute error below 2e-11, and the float equals the rounded double
// erf for the z of every fp16 input (all 63488 checked), so GELU's bits are
// the library call's.  Branch-free: 1500 x 5120 values take 11.7 us, the
// FP64 FMAs' issue (32.6 us with the library's erf, whose ranges diverge
// within a wave).
__device__ __forceinline__ float erf_f(float z) {
    constexpr double q[21] = {
    3.53530995644114998e-01, -1.76576233212071720e-01, 1.31675116723653618e-01,
    -1.07710449040000530e-01, 9.02090009164634721e-02, -7.47277260711611685e-02,
    5.98867995441831544e-02, -4.57664819493776923e-02, 3.30614691469805974e-02,
    -2.24661834254027103e-02, 1.43457370256611406e-02, -8.63003774965729990e-03,
    4.86462751615975453e-03, -2.53035653071606104e-03, 1.27232419626191733e-03,
    -6.73086548474439083e-04, 2.99180998130682454e-04, -7.23168414684691668e-05,
    3.10743840355647092e-05, -3.67141020877584886e-05, 1.32555242082359632e-05};
    const double a = fmin(fabs((double)z), 4.0);   // NaN gives 4; the caller's x * 0.5f carries it on
    const double u = __builtin_fma(a * a, 0.125, -1.0);
    double r = q[20];
#pragma unroll
    for (int i = 19; i >= 0; i--) r = __builtin_fma(r, u, q[i]);
    return __builtin_copysignf((float)(r * a), z);
}

struct GeluErfOp {
    __device__ uint16_t operator()(uint16_t a, uint16_t, bool) const {
        const float inv_sqrt2 = 0.70710678118654752440f;
        const float x = h2f(a);
        return f2h((x * 0.5f) * (1.0f + erf_f(x * inv_sqrt2)));
    }
};

// LayerNorm: the mean and variance are sequential sums over a row, so a row
// takes two dependent chains whatever the machine: 2 F steps of one FMA
// latency.  A workgroup stages LN_ROWS rows in LDS as fp32; one lane per row
// of its first wave adds them up from 16-byte LDS reads, sixteen values ahead
// of the chain, the four waves subtract the mean in place, and the chain
// lanes then run the variance over the differences: nothing but the chain's
// own instruction is left on the serial path.  1500 x 1280: 17 us; 196 us
// with the chains reading two bytes at a time from global memory.
constexpr int LN_ROWS = 4;
constexpr int LN_PAD = 32;   // floats readable past the last row

// s + x[0] + ... + x[F - 1] in that order (SQ: the same of squares, fused)
template <bool SQ>
__device__ __forceinline__ float ln_chain(const float* x, int F) {
    const f32x4* x4 = reinterpret_cast<const f32x4*>(x);
    float s = 0.0f;
    auto add = [&](float v) { s = SQ ? __builtin_fmaf(v, v, s) : s + v; };
    f32x4 v0[4], v1[4];
    // reads run up to 32 floats past the row (into the next row or the
    // allocation's LN_PAD) and are not used
    auto load = [&](int b, f32x4 (&v)[4]) {
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = x4[4 * b + j];
    };
    auto run = [&](const f32x4 (&v)[4]) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            add(v[j].x);
            add(v[j].y);
            add(v[j].z);
            add(v[j].w);
        }
    };
    const int nb = F / 16;
    load(0, v0);
    int b = 0;
    for (; b + 2 <= nb; b += 2) {
        // the reads stay a whole group ahead of the chain (the scheduler
        // would otherwise place them just before their use)
        load(b + 1, v1);
        __builtin_amdgcn_sched_barrier(0);
        run(v0);
        load(b + 2, v0);
        __builtin_amdgcn_sched_barrier(0);
        run(v1);
    }
    if (b < nb) run(v0);
    for (int i = nb * 16; i < F; i++) add(x[i]);
    return s;
}

__global__ void __launch_bounds__(256) layer_norm_rows_kernel(const uint16_t* __restrict__ x,
                                                              const uint16_t* __restrict__ w,
                                                              const uint16_t* __restrict__ b, uint16_t* __restrict__ y,
                                                              size_t rows, int F, float eps) {
    extern __shared__ __align__(16) float ln_row[];   // [LN_ROWS][FS], LN_PAD
    __shared__ float st[LN_ROWS];
    const int tid = threadIdx.x;
    const int FS = ((F + 3) & ~3) + 4;   // rows four banks apart
    const size_t r0 = (size_t)blockIdx.x * LN_ROWS;
    const int nr = (int)(rows - r0 < (size_t)LN_ROWS ? rows - r0 : (size_t)LN_ROWS);
    const bool vec = (F & 7) == 0 && (((uintptr_t)x | (uintptr_t)w | (uintptr_t)b | (uintptr_t)y) & 15) == 0;
    const int nc = F / 8;
    if (vec) {
        for (int u = tid; u < nr * nc; u += 256) {
            const int r = u / nc, c = u - r * nc;
            const i32x4 v = reinterpret_cast<const i32x4*>(x + (r0 + r) * F)[c];
            f32x4* d = reinterpret_cast<f32x4*>(ln_row + r * FS + 8 * c);
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const uint32_t p = (uint32_t)v[2 * h], q = (uint32_t)v[2 * h + 1];
                d[h] = (f32x4){h2f((uint16_t)(p & 0xFFFFu)), h2f((uint16_t)(p >> 16)), h2f((uint16_t)(q & 0xFFFFu)),
                               h2f((uint16_t)(q >> 16))};
            }
        }
    } else {
        for (int u = tid; u < nr * F; u += 256) {
            const int r = u / F, i = u - r * F;
            ln_row[r * FS + i] = h2f(x[(r0 + r) * F + i]);
        }
    }
    __syncthreads();
    if (tid < nr) st[tid] = ln_chain<false>(ln_row + tid * FS, F) / (float)F;
    __syncthreads();
    for (int r = 0; r < nr; r++) {
        const float mean = st[r];
        for (int i = tid; i < F; i += 256) ln_row[r * FS + i] -= mean;
    }
    __syncthreads();
    if (tid < nr) {
        const float var = ln_chain<true>(ln_row + tid * FS, F) / (float)F;
        st[tid] = 1.0f / __builtin_sqrtf(var + eps);
    }
    __syncthreads();
    if (vec) {
        for (int u = tid; u < nr * nc; u += 256) {
            const int r = u / nc, c = u - r * nc;
            const float inv = st[r];
            const f32x4* d = reinterpret_cast<const f32x4*>(ln_row + r * FS + 8 * c);
            const i32x4 wv = reinterpret_cast<const i32x4*>(w)[c], bv = reinterpret_cast<const i32x4*>(b)[c];
            i32x4 o;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const f32x4 dv = d[e >> 1];
                const uint32_t we = (uint32_t)wv[e], be = (uint32_t)bv[e];
                const float d0 = e & 1 ? dv.z : dv.x, d1 = e & 1 ? dv.w : dv.y;
                const uint32_t lo = f2h(__builtin_fmaf(d0 * inv, h2f((uint16_t)(we & 0xFFFFu)), h2f((uint16_t)(be & 0xFFFFu))));
                const uint32_t hi = f2h(__builtin_fmaf(d1 * inv, h2f((uint16_t)(we >> 16)), h2f((uint16_t)(be >> 16))));
                o[e] = (int)(lo | (hi << 16));
            }
            reinterpret_cast<i32x4*>(y + (r0 + r) * F)[c] = o;
        }
    } else {
        for (int u = tid; u < nr * F; u += 256) {
            const int r = u / F, i = u - r * F;
            y[(r0 + r) * F + i] = f2h(__builtin_fmaf(ln_row[r * FS + i] * st[r], h2f(w[i]), h2f(b[i])));
        }
    }
}

// rows beyond the LDS: one lane per row for the chains, straight from global
// memory, then the row's outputs by its wave
__global__ void __launch_bounds__(256) layer_norm_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
                                                         const uint16_t* __restrict__ b, uint16_t* __restrict__ y,
                                                         size_t rows, size_t F, float eps) {
    __shared__ float stats[4][2];
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const size_t r = (size_t)blockIdx.x * 4 + wv;
    if (r >= rows) return;   // the whole wave leaves: no barrier below
    const uint16_t* xr = x + r * F;
    if (lane == 0) {
        float mean = 0.0f;
        for (size_t i = 0; i < F; i++) mean += h2f(xr[i]);
        mean /= (float)F;
        float var = 0.0f;
        for (size_t i = 0; i < F; i++) {
            const float d = h2f(xr[i]) - mean;
            var = __builtin_fmaf(d, d, var);
        }
        var /= (float)F;
        stats[wv][0] = mean;
        stats[wv][1] = 1.0f / __builtin_sqrtf(var + eps);
    }
    wave_lds_order();
    const float mean = stats[wv][0], inv = stats[wv][1];
    for (size_t i = lane; i < F; i += 64)
        y[r * F + i] = f2h(__builtin_fmaf((h2f(xr[i]) - mean) * inv, h2f(w[i]), h2f(b[i])));
}

// x [N][L][C], w [C][K]; thread per output (n, t, c)
__global__ void conv1d_causal_dw_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
                                        uint16_t* __restrict__ y, size_t N, size_t L, size_t C, size_t K,
                                        size_t dil) {
    const size_t total = N * L * C;
    for (size_t o = (size_t)blockIdx.x * blockDim.x + threadIdx.x; o < total; o += (size_t)gridDim.x * blockDim.x) {
        const size_t c = o % C, t = (o / C) % L, n = o / (C * L);
        const uint16_t* wc = w + c * K;
        float lane[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        size_t k = 0;
        for (; k + 8 <= K; k += 8) {
#pragma unroll
            for (int h = 0; h < 2; h++) {
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const size_t kk = k + 4 * h + j;
                    const long long a = (long long)t - (long long)(kk * dil);
                    const float xv = a >= 0 ? h2f(x[(n * L + (size_t)a) * C + c]) : 0.0f;
                    lane[j] = __builtin_fmaf(xv, h2f(wc[K - 1 - kk]), lane[j]);
                }
            }
        }
        float acc = (lane[0] + lane[1]) + (lane[2] + lane[3]);
        for (; k < K; k++) {
            const long long a = (long long)t - (long long)(k * dil);
            if (a >= 0) acc = __builtin_fmaf(h2f(wc[K - 1 - k]), h2f(x[(n * L + (size_t)a) * C + c]), acc);
        }
        y[o] = f2h(acc);
    }
}

// x [N][C_in][L], w [C_out][C_in][3], y [N][C_out][out_len]; thread per output
__global__ void conv1d_k3_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
                                 uint16_t* __restrict__ y, size_t N, size_t L, size_t Cin, size_t Cout,
                                 size_t stride, size_t out_len) {
    const size_t total = N * Cout * out_len;
    for (size_t o = (size_t)blockIdx.x * blockDim.x + threadIdx.x; o < total; o += (size_t)gridDim.x * blockDim.x) {
        const size_t oi = o % out_len, oc = (o / out_len) % Cout, n = o / (out_len * Cout);
        const size_t t = oi * stride;
        float a0 = 0.0f, a1 = 0.0f, a2 = 0.0f, a3 = 0.0f;
        for (size_t ic = 0; ic < Cin; ic++) {
            const uint16_t* xc = x + (n * Cin + ic) * L;
            const uint16_t* wc = w + (oc * Cin + ic) * 3;
            const float xm = t >= 1 ? h2f(xc[t - 1]) : 0.0f;
            const float x0 = h2f(xc[t]);
            const float xp = t + 1 < L ? h2f(xc[t + 1]) : 0.0f;
            a0 = __builtin_fmaf(xm, h2f(wc[0]), a0);
            a1 = __builtin_fmaf(x0, h2f(wc[1]), a1);
            a2 = __builtin_fmaf(xp, h2f(wc[2]), a2);
            a3 = __builtin_fmaf(0.0f, 0.0f, a3);
        }
        y[o] = f2h((a0 + a2) + (a1 + a3));
    }
}

static unsigned blocks_for(size_t n, unsigned block) {
    size_t g = (n + block - 1) / block;
    if (g < 1) g = 1;
    if (g > 65535) g = 65535;
    return (unsigned)g;
}

}  // namespace cactus_hip

using namespace cactus_hip;

extern "C" {

int cactus_hip_gelu_f16(const uint16_t* in, uint16_t* out, size_t n, void* stream) {
    if (n == 0) return CACTUS_HIP_OK;
    CH_REQUIRE(in && out, "gelu: null pointer");
    return launch_pointwise<GeluOp, false>("gelu", in, nullptr, out, n, stream);
}

int cactus_hip_gelu_erf_f16(const uint16_t* in, uint16_t* out, size_t n, void* stream) {
    if (n == 0) return CACTUS_HIP_OK;
    CH_REQUIRE(in && out, "gelu_erf: null pointer");
    return launch_pointwise<GeluErfOp, false>("gelu_erf", in, nullptr, out, n, stream);
}

int cactus_hip_layer_norm_f16(const uint16_t* x, const uint16_t* weight, const uint16_t* bias, uint16_t* y,
                              size_t rows, size_t features, float eps, void* stream) {
    if (rows == 0) return CACTUS_HIP_OK;
    CH_REQUIRE(features > 0, "layer_norm: LayerNorm requires non-empty input tensor");
    CH_REQUIRE(x && weight && bias && y, "layer_norm: null pointer");
    CH_REQUIRE(rows / 4 < (1u << 31), "layer_norm: too many rows");
    const size_t smem = (LN_ROWS * (((features + 3) & ~(size_t)3) + 4) + LN_PAD) * sizeof(float);
    if (smem <= 64 * 1024) {   // features <= 4084: the default dynamic LDS limit
        hipLaunchKernelGGL(layer_norm_rows_kernel, dim3((unsigned)((rows + LN_ROWS - 1) / LN_ROWS)), dim3(256), smem,
                           as_stream(stream), x, weight, bias, y, rows, (int)features, eps);
        return check_launch("layer_norm");
    }
    hipLaunchKernelGGL(layer_norm_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, as_stream(stream), x,
                       weight, bias, y, rows, features, eps);
    return check_launch("layer_norm");
}

int cactus_hip_conv1d_causal_depthwise_f16(const uint16_t* input, const uint16_t* weight, uint16_t* output,
                                           size_t N, size_t L, size_t C, size_t K, size_t dilation,
                                           void* stream) {
    if (N == 0 || L == 0 || C == 0) return CACTUS_HIP_OK;
    CH_REQUIRE(input && weight && output, "conv1d_causal_depthwise: null pointer");
    CH_REQUIRE(K > 0 && dilation > 0, "conv1d_causal_depthwise: kernel size and dilation must be positive");
    hipLaunchKernelGGL(conv1d_causal_dw_kernel, dim3(blocks_for(N * L * C, 256)), dim3(256), 0, as_stream(stream),
                       input, weight, output, N, L, C, K, dilation);
    return check_launch("conv1d_causal_depthwise");
}

int cactus_hip_conv1d_f16_k3(const uint16_t* input, const uint16_t* weight, uint16_t* output, size_t N, size_t L,
                             size_t C_in, size_t C_out, size_t stride, void* stream) {
    if (N == 0 || C_out == 0) return CACTUS_HIP_OK;
    CH_REQUIRE(input && weight && output, "conv1d_k3: null pointer");
    CH_REQUIRE(L > 0 && stride > 0 && C_in > 0, "conv1d_k3: length, stride and input channels must be positive");
    const size_t out_len = (L - 1) / stride + 1;
    hipLaunchKernelGGL(conv1d_k3_kernel, dim3(blocks_for(N * C_out * out_len, 256)), dim3(256), 0,
                       as_stream(stream), input, weight, output, N, L, C_in, C_out, stride, out_len);
    return check_launch("conv1d_k3");
}

}  // extern "C"
