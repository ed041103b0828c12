// pointwise_device.h -- one kernel for the element-by-element fp16 ops.
//
// y[i] = f(a[i], b[i], i < body) with body = 8 floor(n / 8), the vector part
// of the reference's loops (its scalar tail uses other functions).  Bound by
// HBM, so a thread moves eight values per 16-byte load when every pointer is
// 16-byte aligned, one at a time otherwise.  Whole chunks
// are body values: only the last n % 8 see body = false.
#pragma once
#include "hip_common.h"

namespace cactus_hip {

template <bool BINARY, class F>
__global__ void __launch_bounds__(256) pointwise_kernel(const uint16_t* a, const uint16_t* b, uint16_t* y, size_t n,
                                                        F f) {
    const size_t tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t step = (size_t)gridDim.x * blockDim.x;
    const size_t body = n / 8 * 8;
    const bool vec = (((uintptr_t)a | (uintptr_t)y | (BINARY ? (uintptr_t)b : 0)) & 15) == 0;
    if (vec) {
        for (size_t c = tid; c < body / 8; c += step) {
            const i32x4 av = reinterpret_cast<const i32x4*>(a)[c];
            i32x4 bv = {0, 0, 0, 0};
            if (BINARY) bv = reinterpret_cast<const i32x4*>(b)[c];
            i32x4 yv;
#pragma unroll
            for (int w = 0; w < 4; w++) {
                const uint32_t aw = (uint32_t)av[w], bw = (uint32_t)bv[w];
                const uint32_t lo = f((uint16_t)(aw & 0xFFFFu), (uint16_t)(bw & 0xFFFFu), true);
                const uint32_t hi = f((uint16_t)(aw >> 16), (uint16_t)(bw >> 16), true);
                yv[w] = (int)(lo | (hi << 16));
            }
            reinterpret_cast<i32x4*>(y)[c] = yv;
        }
    }
    for (size_t i = (vec ? body : 0) + tid; i < n; i += step) y[i] = f(a[i], BINARY ? b[i] : (uint16_t)0, i < body);
}

// launches f over n values (b: null for a unary op)
template <bool BINARY, class F>
int launch_pointwise(const char* what, const uint16_t* a, const uint16_t* b, uint16_t* y, size_t n, void* stream, F f) {
    const bool vec = (((uintptr_t)a | (uintptr_t)y | (BINARY ? (uintptr_t)b : 0)) & 15) == 0;
    size_t blocks = ((vec ? (n + 7) / 8 : n) + 255) / 256;
    if (blocks > 65535) blocks = 65535;
    hipLaunchKernelGGL((pointwise_kernel<BINARY, F>), dim3((unsigned)blocks), dim3(256), 0, as_stream(stream), a, b, y,
                       n, f);
    return check_launch(what);
}

}  // namespace cactus_hip
