// Router: logits GEMV (exact fp64 accumulation, one bf16 rounding), bias add in
// bf16, sqrt(softplus) scores, stable top-k and renormalised weights.
// Restates compute_expert_affinity_with_bias (router.py:22-36).
//
// One launch in one of two forms:
//  - m <= 8: a wave per expert row sums the tokens one after the other in fp64
//    FMAs (router_kernel; latency bound, the 2 MiB gate matrix is read once);
//  - m > 8: tiles of tokens x experts on v_mfma_f64_16x16x4_f64
//    (router_mfma_kernel).
// In both, the last block of the tokens (of a tile's tokens) to finish selects
// the top-k of each of them with (score desc, index asc) order == torch.sort(stable=True).
#include <math.h>

#include "hsmoe_common.h"
#include "hsmoe_internal.h"
#include "hsmoe_route.h"

namespace hsmoe {
namespace {

constexpr int kTok = kRouterTok;
constexpr int kLogitWaves = 4;  // expert rows per logits workgroup
constexpr size_t kCounterBytes = 4096;  // arrival counters: one per 16 or 32 tokens
constexpr int64_t kMaxRows = 8192;
static_assert(kMaxRows / 16 * 4 <= kCounterBytes, "a counter per tile of tokens");

// m <= kTok tokens.  Block b: wave w computes the logits of expert 4b + w for
// the tokens -- lane l holds columns 8l + 512c .. +8 of the row for every c,
// all loads issued before the math.  The last block (agent-scope arrival
// counter) runs the top-k of the tokens, one token per wave, and re-arms the
// counter.
__global__ void __launch_bounds__(64 * kLogitWaves)
    router_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, const float* __restrict__ bias,
                  int m, int64_t d, int64_t n_exp, int top_k, float scaling, uint16_t* __restrict__ logits_out,
                  float* __restrict__ stage, unsigned* __restrict__ counters, int64_t* __restrict__ idx_out,
                  float* __restrict__ w_out) {
  extern __shared__ __align__(16) uint16_t xs[];  // [m][d]
  __shared__ int s_last;
  const int wave = threadIdx.x >> 6;
  const int64_t e = (int64_t)blockIdx.x * kLogitWaves + wave;
  // the gate rows do not depend on x: issue their loads before staging x
  uint4 wv[kMaxChunks];
  if (e < n_exp) load_gate_row(w, e, d, wv);
  for (int64_t q = threadIdx.x; q < m * d / 8; q += blockDim.x)
    reinterpret_cast<uint4*>(xs)[q] = reinterpret_cast<const uint4*>(x)[q];
  __syncthreads();
  if (e < n_exp) router_row(wv, xs, m, d, e, n_exp, bias, logits_out ? logits_out + e : nullptr, stage + e);
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (threadIdx.x == 0)
    s_last = __hip_atomic_fetch_add(counters, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
  __syncthreads();
  if (!s_last) return;
  for (int t = wave; t < m; t += kLogitWaves)
    wave_topk(stage + t * n_exp, n_exp, top_k, scaling, idx_out + t * top_k, w_out + t * top_k);
  if (threadIdx.x == 0) __hip_atomic_store(counters, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Tiles of 16 kT tokens x 16 kT experts on the fp64 matrix cores, the columns
// split over the workgroup's kW waves (wave w: columns w d/kW ..), whose
// partial sums are added in wave order through LDS.  Products of bf16 values
// are exact in fp64, so a logit is the row's exact sum rounded once whenever
// that sum is exact in fp64, as in router_kernel.
// Operand layout of v_mfma_f64_16x16x4_f64: A[i][k] in lane 16k + i, B[k][j] in
// lane 16k + j, D[4q + lane / 16][lane % 16] in element q.  The k of an
// instruction may be any four columns as long as A and B agree: lane (i, kq)
// reads 32 bytes of its row at column 64 s + 16 kq, and instruction e of the
// 16 that follow takes element e of every lane, so the four lanes of a row read
// one 128-byte line.
// Bound: the fp64 matrix rate (2 m E d flops: 110 us at m = 4096, E = 256,
// d = 4096 on 78.6 TFLOP/s); the FMA form converted both operands for every
// product and re-read the gate per 8 tokens.  Measured per call, E = 256, d =
// 4096, FMA form -> this one: m = 4096 1800 -> 199 us, m = 509 245 -> 41,
// m = 32 37 -> 19.
typedef __attribute__((__vector_size__(4 * sizeof(double)))) double f64x4;

__device__ __forceinline__ double bf16_elem64(const uint4 (&q)[2], int e) {
  const uint4& h = q[e >> 3];
  const int f = e & 7;
  const uint32_t w = f < 2 ? h.x : f < 4 ? h.y : f < 6 ? h.z : h.w;
  return (double)__uint_as_float((f & 1) ? (w & 0xffff0000u) : (w << 16));
}

template <int kT, int kW>
__global__ void __launch_bounds__(64 * kW)
    router_mfma_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, const float* __restrict__ bias,
                       int m, int d, int n_exp, int top_k, float scaling, uint16_t* __restrict__ logits_out,
                       float* __restrict__ stage, unsigned* __restrict__ counters, int64_t* __restrict__ idx_out,
                       float* __restrict__ w_out) {
  constexpr int kRows = 16 * kT;
  __shared__ double s_part[kW][kT * kT][4][64];
  __shared__ int s_last;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i = lane & 15, kq = lane >> 4;
  const int t0 = blockIdx.y * kRows, e0 = blockIdx.x * kRows;
  const int kc = d / kW, k0 = wave * kc + 16 * kq;  // this lane's first column
  const uint16_t *xp[kT], *wp[kT];                  // rows past the end read the last row; their sums are dropped
#pragma unroll
  for (int t = 0; t < kT; ++t) {
    xp[t] = x + (int64_t)min(t0 + 16 * t + i, m - 1) * d + k0;
    wp[t] = w + (int64_t)min(e0 + 16 * t + i, n_exp - 1) * d + k0;
  }
  f64x4 acc[kT][kT];
#pragma unroll
  for (int a = 0; a < kT; ++a)
#pragma unroll
    for (int b = 0; b < kT; ++b) acc[a][b] = f64x4{0.0, 0.0, 0.0, 0.0};
  uint4 xa[kT][2], wa[kT][2], xb[kT][2], wb[kT][2];
  auto load = [&](uint4 (&xv)[kT][2], uint4 (&wv)[kT][2], int c) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < kT; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        xv[t][h] = ldg<uint4>(xp[t] + c + 8 * h);
        wv[t][h] = ldg<uint4>(wp[t] + c + 8 * h);
      }
  };
  auto mul = [&](const uint4 (&xv)[kT][2], const uint4 (&wv)[kT][2]) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      double xe[kT], we[kT];
#pragma unroll
      for (int t = 0; t < kT; ++t) {
        xe[t] = bf16_elem64(xv[t], e);
        we[t] = bf16_elem64(wv[t], e);
      }
#pragma unroll
      for (int a = 0; a < kT; ++a)
#pragma unroll
        for (int b = 0; b < kT; ++b)
          acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(xe[a], we[b], acc[a][b], 0, 0, 0);
    }
  };
  load(xa, wa, 0);
  for (int c = 0; c < kc; c += 128) {  // the next 64 columns are in flight while these are multiplied
    if (c + 64 < kc) load(xb, wb, c + 64);
    mul(xa, wa);
    if (c + 64 >= kc) break;
    if (c + 128 < kc) load(xa, wa, c + 128);
    mul(xb, wb);
  }
#pragma unroll
  for (int a = 0; a < kT; ++a)
#pragma unroll
    for (int b = 0; b < kT; ++b)
#pragma unroll
      for (int q = 0; q < 4; ++q) s_part[wave][a * kT + b][q][lane] = acc[a][b][q];
  __syncthreads();
  for (int n = threadIdx.x; n < kRows * kRows; n += 64 * kW) {
    const int l = n & 63, q = (n >> 6) & 3, ab = n >> 8;
    double sum = 0.0;
#pragma unroll
    for (int v = 0; v < kW; ++v) sum += s_part[v][ab][q][l];
    const int64_t t = t0 + 16 * (ab / kT) + 4 * q + (l >> 4);
    const int64_t e = e0 + 16 * (ab % kT) + (l & 15);
    if (t < m && e < n_exp) {
      const float score = router_score(sum, bias, e, logits_out ? logits_out + t * n_exp + e : nullptr);
      __hip_atomic_store(stage + t * n_exp + e, score, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (threadIdx.x == 0)
    s_last = __hip_atomic_fetch_add(&counters[blockIdx.y], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
             gridDim.x - 1;
  __syncthreads();
  if (!s_last) return;
  for (int64_t t = t0 + wave; t < min(t0 + kRows, m); t += kW)
    wave_topk(stage + t * n_exp, n_exp, top_k, scaling, idx_out + t * top_k, w_out + t * top_k);
  if (threadIdx.x == 0) __hip_atomic_store(&counters[blockIdx.y], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int kT, int kW>
void launch_mfma(const uint16_t* x, const uint16_t* gate, const float* bias, int64_t m, int64_t d, int64_t n_exp,
                 int top_k, float scaling, uint16_t* logits, float* stage, unsigned* counters, int64_t* idx, float* w,
                 hipStream_t st) {
  const dim3 grid((unsigned)((n_exp + 16 * kT - 1) / (16 * kT)), (unsigned)((m + 16 * kT - 1) / (16 * kT)));
  hipLaunchKernelGGL((router_mfma_kernel<kT, kW>), grid, dim3(64 * kW), 0, st, x, gate, bias, (int)m, (int)d,
                     (int)n_exp, top_k, scaling, logits, stage, counters, idx, w);
}

}  // namespace
}  // namespace hsmoe

using namespace hsmoe;

extern "C" size_t hsmoe_router_workspace_size(int64_t m, int64_t n_experts) {
  if (m < 0 || n_experts < 0) return 0;
  // [chunk arrival counters, fixed 4 KiB | staged fp32 scores [m][n_experts]]
  return kCounterBytes + (size_t)(((m * n_experts * 4) + 255) / 256 * 256);
}

extern "C" int hsmoe_router_topk(const void* x, const void* gate_w, const float* bias, int64_t m, int64_t d,
                                 int64_t n_experts, int top_k, float scaling, int64_t* idx_out, float* w_out,
                                 void* logits_out, void* workspace, size_t workspace_bytes, hsmoe_stream_t stream) {
  if (!x || !gate_w || !idx_out || !w_out || m < 0 || d <= 0 || n_experts <= 0)
    return fail(HSMOE_ERR_ARG, "hsmoe_router_topk: null pointer or bad size");
  if (n_experts > 1024 || top_k < 1 || top_k > 16 || top_k > n_experts)
    return fail(HSMOE_ERR_SHAPE, "hsmoe_router_topk: need 1 <= top_k <= min(16, n_experts) and n_experts <= 1024");
  if (d % 512 != 0 || d > 8192 || !aligned(x, 16) || !aligned(gate_w, 16))
    return fail(HSMOE_ERR_SHAPE,
                "hsmoe_router_topk: d must be a multiple of 512 (<= 8192) and x/gate_w 16-byte aligned");
  if (m > kMaxRows) return fail(HSMOE_ERR_SHAPE, "hsmoe_router_topk: m must be <= %lld", (long long)kMaxRows);
  if (!workspace || workspace_bytes < hsmoe_router_workspace_size(m, n_experts) || !aligned(workspace, 256))
    return fail(HSMOE_ERR_WORKSPACE, "hsmoe_router_topk: zero-filled 256-byte aligned workspace of %zu bytes needed",
                hsmoe_router_workspace_size(m, n_experts));
  if (m == 0) return HSMOE_OK;
  unsigned* counters = (unsigned*)workspace;
  float* stage = (float*)((char*)workspace + kCounterBytes);
  if (m > kTok) {
    auto go = [&](auto launch) {
      launch((const uint16_t*)x, (const uint16_t*)gate_w, bias, m, d, n_experts, top_k, scaling,
             (uint16_t*)logits_out, stage, counters, idx_out, w_out, (hipStream_t)stream);
    };
    // 16 x 16 tiles below 2.5 of them per CU; from there on 32 x 32 ones, which
    // convert half as many operands per product but take 2.5 times as long each
    // and leave CUs without one.  us with 16 / 32, d = 4096: 256 experts and
    // m = 256 / 509 / 640 / 700 / 1024: 23 / 51, 41 / 53, 54 / 53, 57 / 53,
    // 77 / 53; 64 experts and m = 800 / 2000 / 2700 / 4096: 19 / 48, 38 / 50,
    // 55 / 50, 72 / 50; 8 experts and m = 4096: 20 / 48 (the FMA form 63).
    const int64_t tiles = (n_experts + 15) / 16 * ((m + 15) / 16);
    if (2 * tiles < 5 * device_cus()) go(launch_mfma<1, 8>);
    else go(launch_mfma<2, 8>);
    return check_launch("hsmoe_router_topk");
  }
  const dim3 grid((unsigned)((n_experts + kLogitWaves - 1) / kLogitWaves));
  const size_t lds = (size_t)m * d * 2;
  hipLaunchKernelGGL(router_kernel, grid, dim3(64 * kLogitWaves), lds, (hipStream_t)stream, (const uint16_t*)x,
                     (const uint16_t*)gate_w, bias, (int)m, d, n_experts, top_k, scaling, (uint16_t*)logits_out, stage,
                     counters, idx_out, w_out);
  return check_launch("hsmoe_router_topk");
}
