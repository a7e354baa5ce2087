// C[M, N] = A[M, K] B[N, K]^T for few rows of A (a decode step's projections), fp16 with fp32
// accumulation, for gfx950.
//
// The product reads B once and is bound by that stream, so the split serves the loads: a workgroup
// takes 16 rows of B, its W waves an equal share of K each, and keeps kUnroll 16-byte loads of B a
// lane in flight. v_mfma_f32_16x16x32_f16 does the sums: row = row of B, column = row of A (up to
// 16; columns past M repeat row M - 1 and are dropped), so M up to 16 costs what M = 1 does, and no
// sum crosses lanes. The waves meet in LDS, in wave order.
#include <hip/hip_runtime.h>

#include "launch_rules.h"
#include "fhip_common.h"
#include "fhip_internal.h"

using namespace fhip;

namespace {

constexpr int kRows = 16;  // rows of B per workgroup
constexpr int kWaves = 8;  // 4 waves, or 8 or 16 loads in flight, measured within 5%; 16 waves 5 .. 10% slower
constexpr int kLoads = 4;  // 16-byte loads of B a lane in flight
typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef float f4_t __attribute__((ext_vector_type(4)));

template <int W, int kUnroll>
__global__ __launch_bounds__(64 * W) void matmul_skinny_kernel(uint16_t* __restrict__ c,
                                                               const uint16_t* __restrict__ a,
                                                               const uint16_t* __restrict__ b, int m,
                                                               int n, int k) {
    __shared__ __attribute__((aligned(16))) float part[W][16][kRows + 4];  // [wave][row of A][row of B]
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, kg = lane >> 4;
    const int64_t n0 = (int64_t)blockIdx.x * kRows;
    const int64_t row = min(n0 + r, (int64_t)n - 1);
    const uint16_t* bp = b + row * k + 8 * kg;
    const uint16_t* ap = a + (int64_t)min(r, m - 1) * k + 8 * kg;
    const int steps = (k + 31) / 32, per = (steps + W - 1) / W;  // 32-wide steps, and per wave
    const int s0 = wave * per, s1 = min(steps, s0 + per);
    f4_t d = {0.0f, 0.0f, 0.0f, 0.0f};
    const int full = min(s1, k / 32);  // steps that lie within K whole
    int s = s0;
    for (; s + kUnroll <= full; s += kUnroll) {
        u32x4 bv[kUnroll], av[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) bv[u] = ld16_stream(bp + 32 * (s + u));
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) av[u] = ld16(ap + 32 * (s + u));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < kUnroll; ++u)
            d = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, bv[u]),
                                                       __builtin_bit_cast(h8_t, av[u]), d, 0, 0, 0);
    }
    for (; s < s1; ++s) {
        u32x4 bv = {0u, 0u, 0u, 0u}, av = {0u, 0u, 0u, 0u};
        if (32 * s + 8 * kg < k) {  // K is a multiple of 8: a lane's 8 are all in or all out
            bv = ld16_stream(bp + 32 * s);
            av = ld16(ap + 32 * s);
        }
        d = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, bv),
                                                   __builtin_bit_cast(h8_t, av), d, 0, 0, 0);
    }
    *(f4_t*)&part[wave][r][4 * kg] = d;  // column r, rows 4 kg .. 4 kg + 3
    __syncthreads();
    for (int i = threadIdx.x; i < m * kRows; i += 64 * W) {
        const int col = i / kRows, rr = i % kRows;
        float sum = 0.0f;
#pragma unroll
        for (int w = 0; w < W; ++w) sum += part[w][col][rr];
        if (n0 + rr < n) c[(int64_t)col * n + n0 + rr] = (uint16_t)f2h(sum);
    }
}

}  // namespace

namespace fhip_internal {

bool matmul_skinny_takes(const void* c, const void* a, const void* b, int m, int n, int k) {
    return fhip_rules::matmul_skinny(m, n, k) && fhip_host::aligned16(a) && fhip_host::aligned16(b);
}

int matmul_skinny(void* c, const void* a, const void* b, int m, int n, int k, hipStream_t s) {
    const unsigned wgs = (unsigned)ceil_div(n, kRows);
    hipLaunchKernelGGL((matmul_skinny_kernel<kWaves, kLoads>), dim3(wgs), dim3(64 * kWaves), 0, s,
                       (uint16_t*)c, (const uint16_t*)a, (const uint16_t*)b, m, n, k);
    return hipGetLastError();
}

}  // namespace fhip_internal
