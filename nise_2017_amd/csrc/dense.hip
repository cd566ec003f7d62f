// Absorption vectors through dense per-frame propagators U (the exact
// exponential, src/propagate.c:60-125): one wave per vector.
//
// What bounds it is the chain of tmax dependent steps: a batch has a few
// hundred vectors, far fewer than the chip has wave slots, so a step's
// latency decides.  A wave therefore keeps everything of its vector to
// itself (no barrier, no other wave's frames): lane (a, g) = (lane % NP, lane
// / NP) holds row a of the frame's U for the column pairs g, g + 64 / NP, ...
// in registers, reads the state from its own LDS row (broadcast 16-byte
// reads, two columns each), and refills every register with the next
// frame's entry as soon as it is used, so U's latency hides behind a whole
// step.  The partial sums of the 64 / NP column groups meet by DPP.
// Measured (N = 28, 150 samples of 300 steps, 450 vectors): 3.77 ms for the
// earlier kernel, whose 256-thread workgroups walked the frames of 21 samples
// with two barriers a frame (9 us each), 0.154 ms here.
#include <algorithm>
#include <vector>

#include "lanes.h"
#include "nise_internal.h"

namespace nise {

// NP: rows (a power of two >= N, at most 64); PPL: column pairs per lane.
template <int NP, int PPL>
__device__ __forceinline__ void dense_run(const DiaSys &S, int v, float2 *psi) {
  constexpr int G = 64 / NP;
  const int N = S.N, T = S.tmax, Pr = (N + 1) >> 1, nU = Pr * N;
  const int lane = threadIdx.x & 63, a = lane % NP, g = lane / NP;
  const bool row = a < N;
  const int64_t fs = (int64_t)(S.begin + v / 3) * S.sample;
  // entries past N stay zero: U's pad column and the clamped pairs below
  // meet a zero
  for (int i = lane; i < 2 * G * PPL; i += 64) psi[i] = make_float2(0.f, 0.f);
  const float4 *U = reinterpret_cast<const float4 *>(S.U) + (fs - S.f_lo) * nU;
  const float *mu = S.mu_rec + (S.mu_stride ? fs * S.mu_stride : 0) + 1 + (int64_t)(v % 3) * N + min(a, N - 1);
  // entry i of the lane's row in a frame's U (pairs past the last clamped);
  // with one column group the pair is wave-uniform: a scalar offset
  const uint32_t ac = (uint32_t)min(a, N - 1);
  uint32_t idx[G > 1 ? PPL : 1];
#pragma unroll
  for (int i = 0; i < PPL; ++i)
    if constexpr (G > 1) idx[i] = min(g + G * i, Pr - 1) * N + ac;
  auto load = [&](const float4 *Uf, int i) {
    if constexpr (G > 1) return gld(Uf + idx[i]);
    else return gld(Uf + min(i, Pr - 1) * N + ac);
  };
  float4 u[PPL];
#pragma unroll
  for (int i = 0; i < PPL; ++i) u[i] = load(U, i);
  float m = gld(mu);
  float2 p = make_float2(m, 0.f);
  double2 *out = S.partial + (int64_t)v * T;
  for (int t = 0; t < T; ++t) {
    // response mu(f).psi (src/absorption.c:205-212), summed over the rows
    const float rr = group_sum<NP>(row ? m * p.x : 0.f), ri = group_sum<NP>(row ? m * p.y : 0.f);
    if (lane == 0) gst(out + t, make_double2((double)rr, (double)ri));
    if (t == T - 1) break;
    mu += S.mu_stride;
    m = gld(mu);
    if (row && g == 0) psi[a] = p;
    // psi <- U psi (src/propagate.c:109-119); the refills read frame fs + t
    // + 1 <= fs + T - 1, which the tables hold
    U += nU;
    float2 y0 = make_float2(0.f, 0.f), y1 = make_float2(0.f, 0.f);
#pragma unroll
    for (int i = 0; i < PPL; ++i) {
      const float4 c = *reinterpret_cast<const float4 *>(psi + 2 * (g + G * i));
      const float4 w = u[i];
      u[i] = load(U, i);
      y0.x = fmaf(w.x, c.x, y0.x), y0.y = fmaf(w.x, c.y, y0.y);
      y1.x = fmaf(w.z, c.z, y1.x), y1.y = fmaf(w.z, c.w, y1.y);
      y0.x = fmaf(-w.y, c.y, y0.x), y0.y = fmaf(w.y, c.x, y0.y);
      y1.x = fmaf(-w.w, c.w, y1.x), y1.y = fmaf(w.w, c.z, y1.y);
      // eight state reads in flight: hoisting all 32 of an N = 64 row spills
      if ((i & 7) == 7) __builtin_amdgcn_sched_barrier(0);
    }
    p = make_float2(y0.x + y1.x, y0.y + y1.y);
    if constexpr (G > 1) p = make_float2(stride_sum<NP>(p.x), stride_sum<NP>(p.y));
  }
}

// Workgroup: the three polarisations of sample wmap.y / 3 of system wmap.x,
// one wave each (they read the same U at about the same time, through the
// same L1).  Row classes of 8, 16, 32 and 64; a lane's pairs cover N.
constexpr int kDensePsi = 64;  // LDS state entries per wave
__global__ void __launch_bounds__(192) __attribute__((amdgpu_waves_per_eu(2)))
dense_vectors_kernel(const DiaSys *sys, const int2 *wmap,
                                                            unsigned long long *times) {
  __shared__ __align__(16) float2 psi[3][kDensePsi];
  const unsigned long long t_start = __builtin_amdgcn_s_memrealtime();
  const int2 wm0 = wmap[blockIdx.x];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const DiaSys S = sys[__builtin_amdgcn_readfirstlane(wm0.x)];
  const int v = __builtin_amdgcn_readfirstlane(wm0.y) + wave;
  const int N = S.N;
  if (N <= 8) dense_run<8, 1>(S, v, psi[wave]);
  else if (N <= 16) dense_run<16, 2>(S, v, psi[wave]);
  else if (N <= 24) dense_run<32, 6>(S, v, psi[wave]);
  else if (N <= 32) dense_run<32, 8>(S, v, psi[wave]);
  else if (N <= 40) dense_run<64, 20>(S, v, psi[wave]);
  else if (N <= 48) dense_run<64, 24>(S, v, psi[wave]);
  else if (N <= 56) dense_run<64, 28>(S, v, psi[wave]);
  else dense_run<64, 32>(S, v, psi[wave]);
  __syncthreads();
  if (threadIdx.x == 0 && times) {
    times[2 * blockIdx.x] = t_start;
    times[2 * blockIdx.x + 1] = __builtin_amdgcn_s_memrealtime();
  }
}

// sys / wmap: device copies, one workgroup per (system, sample), N <= 64.
int launch_dense_vectors(const DiaSys *sys, const int2 *wmap, int nwg, hipStream_t st, unsigned long long *times) {
  if (nwg == 0) return NISE_OK;
  hipLaunchKernelGGL(dense_vectors_kernel, dim3((unsigned)nwg), dim3(192), 0, st, sys, wmap, times);
  NISE_HIP_CHECK(hipGetLastError());
  return NISE_OK;
}

}  // namespace nise
