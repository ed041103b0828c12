// pointwise_device.h -- one kernel for the element-by-element fp16 ops.
//
// y[i] = f(a[i], b[i], i < body) with body = 8 floor(n / 8), the vector part
// of the reference's loops (its scalar tail uses other functions).  Bound by
// HBM where there are many values: a thread moves eight per 16-byte load
// when every pointer is 16-byte aligned.  Short calls are bound by one
// thread's chain of evaluations, so a thread takes two values (4-byte loads)
// below PW_WIDE values: SiLU of 1920 values 1.64 us with one each, 1.92 with
// eight; of 576000 values 3.04 and 3.0.  Whole chunks are body values: only
// the last n % 8 see body = false.  Values whose address is not aligned to a
// chunk go one at a time.
#pragma once
#include "hip_common.h"

#include <type_traits>

namespace cactus_hip {

constexpr size_t PW_WIDE = (size_t)1 << 19;

template <class F, int V, bool BINARY>
__device__ __forceinline__ void pointwise(const uint16_t* a, const uint16_t* b, uint16_t* y, size_t n) {
    const F f{};
    const size_t tid = (size_t)blockIdx.x * 256 + threadIdx.x;
    const size_t step = (size_t)gridDim.x * 256;
    const size_t body = n / 8 * 8;
    const bool vec = (((uintptr_t)a | (uintptr_t)y | (BINARY ? (uintptr_t)b : 0)) & (2 * V - 1)) == 0;
    if (vec) {
        typedef uint32_t chunk __attribute__((ext_vector_type(V / 2)));
        for (size_t c = tid; c < body / V; c += step) {
            const chunk av = reinterpret_cast<const chunk*>(a)[c];
            chunk bv = av, yv;
            if (BINARY) bv = reinterpret_cast<const chunk*>(b)[c];
#pragma unroll
            for (int w = 0; w < V / 2; w++) {
                const uint32_t lo = f((uint16_t)(av[w] & 0xFFFFu), (uint16_t)(bv[w] & 0xFFFFu), true);
                const uint32_t hi = f((uint16_t)(av[w] >> 16), (uint16_t)(bv[w] >> 16), true);
                yv[w] = lo | (hi << 16);
            }
            reinterpret_cast<chunk*>(y)[c] = yv;
        }
    }
    for (size_t i = (vec ? body : 0) + tid; i < n; i += step) y[i] = f(a[i], BINARY ? b[i] : (uint16_t)0, i < body);
}

// no more arguments than the op has: each costs host time in every launch
template <class F, int V>
__global__ void __launch_bounds__(256) unary_kernel(const uint16_t* a, uint16_t* y, size_t n) {
    pointwise<F, V, false>(a, nullptr, y, n);
}
template <class F, int V>
__global__ void __launch_bounds__(256) binary_kernel(const uint16_t* a, const uint16_t* b, uint16_t* y, size_t n) {
    pointwise<F, V, true>(a, b, y, n);
}

// launches F over n values (b: null for a unary op)
template <class F, bool BINARY>
int launch_pointwise(const char* what, const uint16_t* a, const uint16_t* b, uint16_t* y, size_t n, void* stream) {
    const uintptr_t at = (uintptr_t)a | (uintptr_t)y | (BINARY ? (uintptr_t)b : 0);
    const bool wide = n >= PW_WIDE && (at & 15) == 0;
    const size_t v = wide ? 8 : (at & 3) == 0 ? 2 : 1;
    size_t blocks = ((n + v - 1) / v + 255) / 256;
    if (blocks > 65535) blocks = 65535;
    const dim3 grid((unsigned)blocks), block(256);
    if constexpr (BINARY) {
        if (wide) hipLaunchKernelGGL((binary_kernel<F, 8>), grid, block, 0, as_stream(stream), a, b, y, n);
        else hipLaunchKernelGGL((binary_kernel<F, 2>), grid, block, 0, as_stream(stream), a, b, y, n);
    } else {
        if (wide) hipLaunchKernelGGL((unary_kernel<F, 8>), grid, block, 0, as_stream(stream), a, y, n);
        else hipLaunchKernelGGL((unary_kernel<F, 2>), grid, block, 0, as_stream(stream), a, y, n);
    }
    return check_launch(what);
}

}  // namespace cactus_hip
