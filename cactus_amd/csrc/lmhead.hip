// lmhead.hip -- FP16 matmul with FP16 accumulation (a4) and the fused
// LM-head + greedy-sample path (a4 + a14).
//
// Reference arithmetic (kernel_gemm.cpp:17-126): for each output, eight fp16
// lanes; lane j accumulates k = j (mod 8) in increasing k with fp16 FMA; the
// result is ((l0+l4)+(l2+l6)) + ((l1+l5)+(l3+l7)) in fp16.
//
// Three kernels: a few activation rows (f16_rows_kernel, one pass over the
// weights bound by HBM), more rows (f16_tile_kernel, bound by the packed FP16
// FMA rate), and the LM head with the argmax (f16_argmax_kernel).
#include "lm_device.h"

#include <algorithm>
#include <type_traits>

namespace cactus_hip {

struct LmArgs {
    const uint16_t* a;   // [M][K]
    const uint16_t* b;   // [N][K]
    uint16_t* c;         // [M][N] (may be null when only the argmax is wanted)
    int M, K, N;
    float* part_val;     // per-workgroup argmax partials (fused path)
    uint32_t* part_idx;
    uint32_t* counter;
    uint32_t* token;
};

// ------------------------------------------------ a few activation rows
// M <= 4 rows in one pass over the weights: bound by HBM for large N (the
// LM head of a sampled decode step), by load latency for small N.  A wave
// owns 16 weight rows; lane (c, j) = (lane / 4, lane % 4) runs chain pair j
// (chains 2j, 2j + 1) of row c, so a 16-row wave has 64 lanes busy and four
// times the waves of a lane per row are in flight (the 151936-row head: 9496
// waves; with a lane per row 2374, two or three per SIMD).  A stage is
// 16 rows x 256 values, loaded as whole 512-byte row pieces, two stages ahead
// (16 KB in flight per wave); it passes through the wave's own LDS slice
// (row stride 528 bytes: the 64 dwords of a step lie in 64 banks), no
// workgroup barrier after the activation rows are staged.  M=1 K=1024
// N=151936: 102 -> 47.8 us (6.5 TB/s) against the row-per-lane form that
// loaded, waited and then used each 64-value stage.
constexpr int LMR_KS = 256;                      // k-values per stage
constexpr int LMR_STRIDE = LMR_KS * 2 + 16;      // bytes per staged row
constexpr int LMR_TILE = 16;                     // weight rows per wave

template <int MR>
__global__ void __launch_bounds__(LM_THREADS) f16_rows_kernel(LmArgs p) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int K = p.K, N = p.N;
    const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int n0 = ((int)blockIdx.x * (LM_THREADS / 64) + wid) * LMR_TILE;
    const int nstage = (K + LMR_KS - 1) / LMR_KS, npc = K / 8;
    unsigned char* as = smem;                                                     // [MR][K] fp16
    unsigned char* st = smem + (size_t)MR * K * 2 + wid * LMR_TILE * LMR_STRIDE;  // this wave's stage

    // piece u = 64 i + lane of a stage: row u / 32, 16-byte piece u % 32;
    // rows and pieces past the end read the last one and are never used
    constexpr int NI = LMR_TILE * (LMR_KS / 8) / 64;
    const uint16_t* src[NI];
#pragma unroll
    for (int i = 0; i < NI; i++) src[i] = p.b + (size_t)min(n0 + 2 * i + (lane >> 5), N - 1) * K;
    auto load = [&](int s, i32x4 (&w)[NI]) {
        const int pc = min(s * (LMR_KS / 8) + (lane & 31), npc - 1);
#pragma unroll
        for (int i = 0; i < NI; i++)
            w[i] = __builtin_nontemporal_load(reinterpret_cast<const i32x4*>(src[i] + (size_t)pc * 8));
    };
    // the activation rows' first pieces are the oldest loads: the wait for
    // them leaves the weights in flight
    const i32x4* a4 = reinterpret_cast<const i32x4*>(p.a);
    const int a_pc = min((int)threadIdx.x, MR * npc - 1);
    const i32x4 av = a4[a_pc];
    __builtin_amdgcn_sched_barrier(0);
    i32x4 w0[NI], w1[NI];
    load(0, w0);
    load(1, w1);
    reinterpret_cast<i32x4*>(as)[a_pc] = av;
    for (int i = threadIdx.x + LM_THREADS; i < MR * npc; i += LM_THREADS) reinterpret_cast<i32x4*>(as)[i] = a4[i];
    __syncthreads();

    h2v acc[MR];
#pragma unroll
    for (int m = 0; m < MR; m++) acc[m] = (h2v){(f16)0.0f, (f16)0.0f};
    const unsigned char* bl = st + (lane >> 2) * LMR_STRIDE + (lane & 3) * 4;
    const unsigned char* al = as + (lane & 3) * 4;
    auto stage = [&](int s, i32x4 (&w)[NI]) {
#pragma unroll
        for (int i = 0; i < NI; i++)
            *reinterpret_cast<i32x4*>(st + (2 * i + (lane >> 5)) * LMR_STRIDE + (lane & 31) * 16) = w[i];
        wave_lds_order();
        load(s + 2, w);   // branch-free (past the end: the last piece again), so the waits stay exact
        const int nc = min(LMR_KS / 8, npc - s * (LMR_KS / 8));
        const unsigned char* ak = al + (size_t)s * (LMR_KS * 2);
        auto step = [&](int ch) {
            const h2v b = as_h2(*reinterpret_cast<const uint32_t*>(bl + ch * 16));
#pragma unroll
            for (int m = 0; m < MR; m++)
                acc[m] = __builtin_elementwise_fma(
                    as_h2(*reinterpret_cast<const uint32_t*>(ak + (size_t)m * K * 2 + ch * 16)), b, acc[m]);
        };
        if (nc == LMR_KS / 8) {
#pragma unroll
            for (int ch = 0; ch < LMR_KS / 8; ch++) step(ch);
        } else {
            for (int ch = 0; ch < nc; ch++) step(ch);
        }
        wave_lds_order();
    };
    int s = 0;
    for (; s + 2 <= nstage; s += 2) {
        stage(s, w0);
        stage(s + 1, w1);
    }
    if (s < nstage) stage(s, w0);
    // hsum_f16x8 over the quad's four chain pairs: (p0 + p2) + (p1 + p3),
    // then the two halves (fp16 addition commutes)
    const int n = n0 + (lane >> 2);
#pragma unroll
    for (int m = 0; m < MR; m++) {
        auto dpp = [](h2v v, auto ctrl) {
            const int b = __builtin_bit_cast(int, v);
            return __builtin_bit_cast(h2v, __builtin_amdgcn_update_dpp(b, b, decltype(ctrl)::value, 0xF, 0xF, false));
        };
        h2v t = acc[m] + dpp(acc[m], std::integral_constant<int, 0x4E>{});   // lane ^ 2
        t = t + dpp(t, std::integral_constant<int, 0xB1>{});                 // lane ^ 1
        const f16 r = t.x + t.y;
        if ((lane & 3) == m && n < N) p.c[(size_t)m * N + n] = __builtin_bit_cast(uint16_t, r);
    }
}

// ------------------------------------------------ many activation rows
// Each output is eight dependent fp16 chains (no matrix instruction rounds to
// fp16 after every product), so the packed FP16 FMA rate bounds this kernel:
// four instructions per output and 8 k-values.  A lane owns one weight row
// (output column) and TM activation rows; a wave is 64 columns x TM rows and
// the workgroup's four waves share the columns' 128-value LDS stages (double
// buffered; the next stage is in registers while this one is used).  The
// activation values are uniform over the wave: scalar loads feed the FMAs'
// scalar operand, so a step costs one LDS read per 4 TM FMAs.  M=100 K=1024
// N=3072: 1462 us in 25 four-row passes over the weights before, 16 us now
// (4 us of FMA issue at the full rate).
constexpr int LMT_KS = 128;                      // k-values per stage
constexpr int LMT_STRIDE = LMT_KS * 2 + 16;      // bytes per staged column (17 16-byte slots: conflict-free reads)

template <int TM>
__global__ void __launch_bounds__(LM_THREADS) f16_tile_kernel(const uint16_t* __restrict__ a,
                                                              const uint16_t* __restrict__ b,
                                                              uint16_t* __restrict__ c, int M, int K, int N) {
    __shared__ __align__(16) unsigned char sb[2][64 * LMT_STRIDE];
    const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int cols = (N + 63) / 64;
    const int n0 = ((int)blockIdx.x % cols) * 64;
    const int m0 = ((int)blockIdx.x / cols * 4 + wid) * TM;
    const int nstage = (K + LMT_KS - 1) / LMT_KS, npc = K / 8;
    // the wave's activation rows (rows past M repeat the last one)
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    typedef const __attribute__((address_space(4))) u32x4* sptr;
    sptr ar[TM];
#pragma unroll
    for (int m = 0; m < TM; m++) ar[m] = (sptr)(uintptr_t)(a + (size_t)min(m0 + m, M - 1) * K);

    // piece u = 256 i + tid of a stage: column u / 16, 16-byte piece u % 16;
    // columns and pieces past the end read the last one and are never used
    constexpr int NI = 64 * (LMT_KS / 8) / LM_THREADS;
    const uint16_t* src[NI];
#pragma unroll
    for (int i = 0; i < NI; i++) src[i] = b + (size_t)min(n0 + 16 * i + ((int)threadIdx.x >> 4), N - 1) * K;
    i32x4 w[NI];
    auto load = [&](int s) {
        const int pc = min(s * (LMT_KS / 8) + ((int)threadIdx.x & 15), npc - 1);
#pragma unroll
        for (int i = 0; i < NI; i++) w[i] = *reinterpret_cast<const i32x4*>(src[i] + (size_t)pc * 8);
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int i = 0; i < NI; i++)
            *reinterpret_cast<i32x4*>(sb[buf] + (16 * i + ((int)threadIdx.x >> 4)) * LMT_STRIDE + (threadIdx.x & 15) * 16) = w[i];
    };
    h2v acc[TM][4];
#pragma unroll
    for (int m = 0; m < TM; m++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[m][j] = (h2v){(f16)0.0f, (f16)0.0f};
    load(0);
    store(0);
    __syncthreads();
    for (int s = 0; s < nstage; s++) {
        if (s + 1 < nstage) load(s + 1);
        const unsigned char* bl = sb[s & 1] + lane * LMT_STRIDE;
        const int c0 = s * (LMT_KS / 8), nc = min(LMT_KS / 8, npc - c0);
        auto step = [&](int ch) {
            const uint4 bv = *reinterpret_cast<const uint4*>(bl + ch * 16);
#pragma unroll
            for (int m = 0; m < TM; m++) {
                const u32x4 av = ar[m][c0 + ch];
                f16_step(acc[m], make_uint4(av.x, av.y, av.z, av.w), bv);
            }
        };
        int ch = 0;
        for (; ch + 4 <= nc; ch += 4) {
#pragma unroll
            for (int u = 0; u < 4; u++) step(ch + u);
        }
        for (; ch < nc; ch++) step(ch);
        // buffer (s + 1) & 1 was last read in stage s - 1, before the barrier that ended it
        if (s + 1 < nstage) store((s + 1) & 1);
        __syncthreads();
    }
    const int n = n0 + lane;
    if (n < N) {
#pragma unroll
        for (int m = 0; m < TM; m++)
            if (m0 + m < M) c[(size_t)(m0 + m) * N + n] = f16_hsum(acc[m]);
    }
}

// LM head + argmax, one activation row: one lane owns one output row and
// keeps its eight chains as four packed halves (v_pk_fma_f16 does two chains
// per instruction).  A wave stages 64 rows x 64 k-values (8 KiB) through LDS
// with coalesced 16-byte loads, then every lane walks its own row out of LDS.
// The activation row is broadcast from LDS.
__global__ void __launch_bounds__(LM_THREADS) f16_argmax_kernel(LmArgs p) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int K = p.K;
    const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63;
    uint16_t* as = reinterpret_cast<uint16_t*>(smem);                       // [K]
    unsigned char* stage = smem + K * 2 + wid * LM_ROWS_PER_WAVE * LM_ROW_STRIDE;

    for (int i = threadIdx.x; i < K; i += LM_THREADS) as[i] = p.a[i];
    __syncthreads();

    const int row0 = (blockIdx.x * (LM_THREADS / 64) + wid) * LM_ROWS_PER_WAVE;
    const int my_row = row0 + lane;
    h2v acc[4];
#pragma unroll
    for (int j = 0; j < 4; j++) acc[j] = (h2v){(f16)0.0f, (f16)0.0f};

    for (int k0 = 0; k0 < K; k0 += LM_KC) {    // K % 8 == 0 (checked by the entry point)
        const int cpr = min(LM_KC, K - k0) / 8;   // 16-byte chunks per row in this step
        // stage 64 rows x kc values: lane -> (row, chunk) coalesced
        for (int i = lane; i < LM_ROWS_PER_WAVE * cpr; i += 64) {
            const int r = i / cpr, ch = i % cpr;
            uint4 v = make_uint4(0, 0, 0, 0);
            if (row0 + r < p.N)
                v = *reinterpret_cast<const uint4*>(p.b + (size_t)(row0 + r) * K + k0 + ch * 8);
            *reinterpret_cast<uint4*>(stage + r * LM_ROW_STRIDE + ch * 16) = v;
        }
        wave_lds_order();
        for (int ch = 0; ch < cpr; ch++) {
            const uint4 bv = *reinterpret_cast<const uint4*>(stage + lane * LM_ROW_STRIDE + ch * 16);
            const uint4 av = *reinterpret_cast<const uint4*>(as + k0 + ch * 8);
            f16_step(acc, av, bv);
        }
        wave_lds_order();
    }
    float best = -__builtin_inff();
    uint32_t best_i = 0xFFFFFFFFu;
    if (my_row < p.N) {
        const uint16_t r = f16_hsum(acc);
        if (p.c) p.c[my_row] = r;
        best = h2f(r);
        best_i = (uint32_t)my_row;
    }
    // workgroup (max, first index), then the last workgroup reduces all
    __shared__ float bv_s[LM_THREADS];
    __shared__ uint32_t bi_s[LM_THREADS];
    __shared__ bool last;
    bv_s[threadIdx.x] = best;
    bi_s[threadIdx.x] = best_i;
    __syncthreads();
    for (int w = LM_THREADS / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
            const float ov = bv_s[threadIdx.x + w];
            const uint32_t oi = bi_s[threadIdx.x + w];
            const float mv = bv_s[threadIdx.x];
            const uint32_t mi = bi_s[threadIdx.x];
            bool take = oi != 0xFFFFFFFFu &&
                        (mi == 0xFFFFFFFFu || ov > mv || (ov == mv && oi < mi));
            if (take) { bv_s[threadIdx.x] = ov; bi_s[threadIdx.x] = oi; }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        p.part_val[blockIdx.x] = bv_s[0];
        p.part_idx[blockIdx.x] = bi_s[0];
        __threadfence();
        const uint32_t done = atomicAdd(p.counter, 1u);
        last = (done == gridDim.x - 1);
    }
    __syncthreads();
    if (last) {
        __threadfence();
        float bv = -__builtin_inff();
        uint32_t bi = 0xFFFFFFFFu;
        for (unsigned i = threadIdx.x; i < gridDim.x; i += LM_THREADS) {
            const float v = p.part_val[i];
            const uint32_t ix = p.part_idx[i];
            if (ix != 0xFFFFFFFFu && (bi == 0xFFFFFFFFu || v > bv || (v == bv && ix < bi))) {
                bv = v; bi = ix;
            }
        }
        bv_s[threadIdx.x] = bv;
        bi_s[threadIdx.x] = bi;
        __syncthreads();
        for (int w = LM_THREADS / 2; w > 0; w >>= 1) {
            if ((int)threadIdx.x < w) {
                const float ov = bv_s[threadIdx.x + w];
                const uint32_t oi = bi_s[threadIdx.x + w];
                const float mv = bv_s[threadIdx.x];
                const uint32_t mi = bi_s[threadIdx.x];
                bool take = oi != 0xFFFFFFFFu &&
                            (mi == 0xFFFFFFFFu || ov > mv || (ov == mv && oi < mi));
                if (take) { bv_s[threadIdx.x] = ov; bi_s[threadIdx.x] = oi; }
            }
            __syncthreads();
        }
        if (threadIdx.x == 0) {
            *p.token = bi_s[0] == 0xFFFFFFFFu ? 0u : bi_s[0];
            *p.counter = 0u;  // leave the counter ready for the next call
        }
    }
}

// Any-K / any-alignment form: one thread per output, scalar loads, same
// lane order and final tree.
__global__ void f16_matmul_scalar_kernel(const uint16_t* __restrict__ a,
                                         const uint16_t* __restrict__ b, uint16_t* __restrict__ c,
                                         int M, int K, int N) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (size_t)M * N) return;
    const int m = (int)(t / N), n = (int)(t % N);
    const uint16_t* ar = a + (size_t)m * K;
    const uint16_t* br = b + (size_t)n * K;
    h2v acc[4];
    for (int j = 0; j < 4; j++) acc[j] = (h2v){(f16)0.0f, (f16)0.0f};
    const int K8 = (K / 8) * 8;
    for (int k = 0; k < K8; k += 8) {
        uint4 av, bv;
        av.x = (uint32_t)ar[k] | ((uint32_t)ar[k + 1] << 16);
        av.y = (uint32_t)ar[k + 2] | ((uint32_t)ar[k + 3] << 16);
        av.z = (uint32_t)ar[k + 4] | ((uint32_t)ar[k + 5] << 16);
        av.w = (uint32_t)ar[k + 6] | ((uint32_t)ar[k + 7] << 16);
        bv.x = (uint32_t)br[k] | ((uint32_t)br[k + 1] << 16);
        bv.y = (uint32_t)br[k + 2] | ((uint32_t)br[k + 3] << 16);
        bv.z = (uint32_t)br[k + 4] | ((uint32_t)br[k + 5] << 16);
        bv.w = (uint32_t)br[k + 6] | ((uint32_t)br[k + 7] << 16);
        f16_step(acc, av, bv);
    }
    for (int k = K8; k < K; k++) {
        const float r = __builtin_fmaf(h2f(ar[k]), h2f(br[k]), (float)acc[0].x);
        acc[0].x = hbits(f2h(r));
    }
    c[t] = f16_hsum(acc);
}

// ------------------------------------------------ per-(device, stream) scratch
// one buffer: the completion counter (zeroed when the buffer is made; the
// last workgroup of every call leaves it at zero), then the per-workgroup
// partial maxima and their indices
struct LmScratch {
    float* val = nullptr;
    uint32_t* idx = nullptr;
    uint32_t* counter = nullptr;
};

static int lm_scratch(void* stream, size_t blocks, LmScratch* out) {
    void* p = nullptr;
    int rc = stream_scratch(SCR_LM, stream, 256 + 8 * blocks, true, &p);
    if (rc) return rc;
    out->counter = static_cast<uint32_t*>(p);
    out->val = reinterpret_cast<float*>(static_cast<char*>(p) + 256);
    out->idx = reinterpret_cast<uint32_t*>(out->val + blocks);
    return CACTUS_HIP_OK;
}

static size_t lm_smem(int K) {
    return (size_t)K * 2 + (size_t)(LM_THREADS / 64) * LM_ROWS_PER_WAVE * LM_ROW_STRIDE;
}

template <int MR>
static int launch_rows(const LmArgs& p, hipStream_t st) {
    constexpr size_t kStages = (size_t)(LM_THREADS / 64) * LMR_TILE * LMR_STRIDE;
    const size_t smem = (size_t)MR * p.K * 2 + kStages;
    if (smem > 64 * 1024) {
        // beyond the default 64 KiB of dynamic LDS: the limit is raised once, to what the largest K needs
        static const hipError_t attr =
            hipFuncSetAttribute((const void*)f16_rows_kernel<MR>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)((size_t)MR * LM_MAX_K * 2 + kStages));
        if (attr != hipSuccess)
            return fail(CACTUS_HIP_ERUNTIME, std::string("hipFuncSetAttribute: ") + hipGetErrorString(attr));
    }
    hipLaunchKernelGGL(f16_rows_kernel<MR>, dim3(ceil_div(p.N, (LM_THREADS / 64) * LMR_TILE)), dim3(LM_THREADS), smem,
                       st, p);
    return check_launch("matmul_f16");
}

template <int TM>
static int launch_tile(const LmArgs& p, hipStream_t st) {
    // a launch holds fewer than 2^32 threads: 2^23 workgroups of rows at a time
    const size_t cols = ceil_div(p.N, 64);
    const size_t step = 4 * TM * std::max<size_t>(((size_t)1 << 23) / cols, 1);
    for (size_t m0 = 0; m0 < (size_t)p.M; m0 += step) {
        const int M = (int)std::min<size_t>(step, p.M - m0);
        hipLaunchKernelGGL(f16_tile_kernel<TM>, dim3((unsigned)(cols * ceil_div(M, 4 * TM))), dim3(LM_THREADS), 0, st,
                           p.a + m0 * p.K, p.b, p.c + m0 * p.N, M, p.K, p.N);
        const int rc = check_launch("matmul_f16");
        if (rc) return rc;
    }
    return CACTUS_HIP_OK;
}

}  // namespace cactus_hip

using namespace cactus_hip;

extern "C" {

int cactus_hip_matmul_f16(const uint16_t* a, const uint16_t* b_transposed, uint16_t* c, size_t M,
                          size_t K, size_t N, void* stream) {
    if (M == 0 || N == 0) return CACTUS_HIP_OK;
    CH_REQUIRE(a && b_transposed && c, "matmul_f16: null pointer");
    CH_REQUIRE(K <= (size_t)LM_MAX_K, "matmul_f16: K > 8192 not supported");
    CH_REQUIRE(M < (1u << 30) && N < (1u << 30), "matmul_f16: shape too large");
    if (((uintptr_t)b_transposed & 15) != 0 || K % 8 != 0 || ((uintptr_t)a & 15) != 0) {
        const size_t outs = M * N;
        hipLaunchKernelGGL(f16_matmul_scalar_kernel, dim3(ceil_div(outs, 256)), dim3(256), 0,
                           as_stream(stream), a, b_transposed, c, (int)M, (int)K, (int)N);
        return check_launch("matmul_f16");
    }
    if (K == 0) return cactus_hip_memset(c, 0, M * N * 2, stream);   // empty sums
    LmArgs p{};
    p.a = a; p.b = b_transposed; p.c = c; p.M = (int)M; p.K = (int)K; p.N = (int)N;
    const hipStream_t st = as_stream(stream);
    switch (M) {
        case 1: return launch_rows<1>(p, st);
        case 2: return launch_rows<2>(p, st);
        case 3: return launch_rows<3>(p, st);
        case 4: return launch_rows<4>(p, st);
        default: break;
    }
    // rows per wave: more share each LDS read, fewer give more waves
    const size_t cols = ceil_div(N, 64);
    if (cols * ceil_div(M, 8) >= 4096) return launch_tile<8>(p, st);
    if (cols * ceil_div(M, 4) >= 1024) return launch_tile<4>(p, st);
    return launch_tile<2>(p, st);
}

int cactus_hip_lm_head_argmax_f16(const uint16_t* a, const uint16_t* b_transposed,
                                  uint16_t* logits, uint32_t* token, size_t K, size_t N,
                                  void* stream) {
    CH_REQUIRE(token, "lm_head_argmax: null token pointer");
    if (N == 0) return cactus_hip_memset(token, 0, 4, stream);
    CH_REQUIRE(a && b_transposed, "lm_head_argmax: null pointer");
    CH_REQUIRE(K <= (size_t)LM_MAX_K, "lm_head_argmax: K > 8192 not supported");
    CH_REQUIRE(N < (1u << 30), "lm_head_argmax: N too large");
    CH_REQUIRE(((uintptr_t)b_transposed & 15) == 0 && K % 8 == 0,
               "lm_head_argmax: b must be 16-byte aligned with K a multiple of 8");
    const unsigned blocks = ceil_div(N, (LM_THREADS / 64) * LM_ROWS_PER_WAVE);
    LmScratch s;
    int rc = lm_scratch(stream, blocks, &s);
    if (rc) return rc;
    LmArgs p{};
    p.a = a; p.b = b_transposed; p.c = logits; p.M = 1; p.K = (int)K; p.N = (int)N;
    p.part_val = s.val; p.part_idx = s.idx; p.counter = s.counter; p.token = token;
    hipLaunchKernelGGL(f16_argmax_kernel, dim3(blocks), dim3(LM_THREADS), lm_smem((int)K), as_stream(stream), p);
    return check_launch("lm_head_argmax");
}

}  // extern "C"
