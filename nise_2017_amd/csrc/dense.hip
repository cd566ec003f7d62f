// Absorption vectors through dense per-frame propagators U: the exact
// exponential (src/propagate.c:60-125), and the Trotter scheme where a run has
// too few vectors to fill the chip with sweeps (dense_pays).  N <= 32: one
// wave per vector.
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
#include <cmath>
#include <vector>

#include "lanes.h"
#include "nise_internal.h"

namespace nise {

// NP: rows (a power of two >= N, at most 32); PPL: column pairs per lane.
template <int NP, int PPL>
__device__ __forceinline__ void dense_run(const DiaSys &S, int v, float2 *psi) {
  constexpr int G = 64 / NP;
  const int N = S.N, T = S.tmax, Pr = (N + 1) >> 1, nU = Pr * N;
  const int lane = threadIdx.x & 63, a = lane % NP, g = lane / NP;
  const bool row = a < N;
  const int64_t fs = (int64_t)(S.begin + v / 3) * S.sample + S.t0;  // frame of step t0
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
  if (S.t0) p = gld(S.state + (int64_t)v * N + min(a, N - 1));
  double2 *out = S.partial + (int64_t)v * T;
  for (int t = S.t0;; ++t) {
    if (S.hist) {  // checkpoint rows as the conveyor writes them (RowsArgs)
      const int hr = t % S.hist_every == 0 ? t / S.hist_every : t == T - 1 ? t / S.hist_every + 1 : -1;
      if (hr >= 0 && row && g == 0) gst(S.hist + ((int64_t)v * S.nck + hr) * N + a, p);
    }
    // response mu(f).psi (src/absorption.c:205-212), summed over the rows
    const float rr = group_sum<NP>(row ? m * p.x : 0.f), ri = group_sum<NP>(row ? m * p.y : 0.f);
    if (lane == 0) gst(out + t, make_double2((double)rr, (double)ri));
    if (t == T - 1) break;
    const bool more = t + 1 < S.t1;
    mu += more ? S.mu_stride : 0;
    m = gld(mu);
    if (row && g == 0) psi[a] = p;
    // psi <- psi + (U - I) psi (src/propagate.c:109-119); the refills read the frame of
    // step t + 1 < t1, which the tables hold (at the end of a segment the same
    // frame again, not used)
    U += more ? nU : 0;
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
    }
    p = make_float2(p.x + stride_sum<NP>(y0.x + y1.x), p.y + stride_sum<NP>(y0.y + y1.y));
    if (!more) {  // the segment's end: its state
      if (row && g == 0) gst(S.state + (int64_t)v * N + a, p);
      break;
    }
  }
}

// Workgroup: the three polarisations of sample wmap.y of system wmap.x,
// one wave each (they read the same U at about the same time, through the
// same L1).  Row classes of 8, 16 and 32; a lane's pairs cover N.
constexpr int kDensePsi = 32;  // LDS state entries per wave
__global__ void __launch_bounds__(192)
dense_vectors_kernel(const DiaSys *sys, const int2 *wmap, unsigned long long *times) {
  __shared__ __align__(16) float2 psi[3][kDensePsi];
  const unsigned long long t_start = __builtin_amdgcn_s_memrealtime();
  const int2 wm0 = wmap[blockIdx.x];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const DiaSys S = sys[__builtin_amdgcn_readfirstlane(wm0.x)];
  const int v = 3 * __builtin_amdgcn_readfirstlane(wm0.y) + wave;
  const int N = S.N;
  if (N <= 8) dense_run<8, 1>(S, v, psi[wave]);
  else if (N <= 16) dense_run<16, 2>(S, v, psi[wave]);
  else if (N <= 24) dense_run<32, 6>(S, v, psi[wave]);
  else dense_run<32, 8>(S, v, psi[wave]);
  __syncthreads();
  if (threadIdx.x == 0 && times) {
    times[2 * blockIdx.x] = t_start;
    times[2 * blockIdx.x + 1] = __builtin_amdgcn_s_memrealtime();
  }
}

// ---------------------------------------------------------------------------
// N = 33 .. 128: one workgroup of eight waves per sample.  Lane (h, r) =
// (lane / 32, lane % 32) of wave w holds rows r, r + 32, ... of the column
// pairs 2 w + h, + 16, ... in registers and applies them to the sample's
// three vectors, so each entry of U is loaded once per sample and step (a
// wave per vector loads it three times: at N = 110 the L1 alone would take
// 4,500 cycles a step).  The waves' partial sums meet in LDS, thread (x, a)
// adds them and forms its part of the next response: two barriers a step.
// ---------------------------------------------------------------------------
constexpr int kWideWaves = 8, kWideSlices = 2 * kWideWaves;
template <int RPL, int PPL>
struct WideLds {
  float2 psi[3][2 * kWideSlices * PPL];
  float2 part[kWideWaves][3][32 * RPL];
  float2 red[2][kWideWaves];
};
template <int RPL, int PPL>
__device__ __forceinline__ void wide_run(const DiaSys &S, int s, unsigned char *smem) {
  WideLds<RPL, PPL> &L = *reinterpret_cast<WideLds<RPL, PPL> *>(smem);
  constexpr int NR = 32 * RPL;
  const int N = S.N, T = S.tmax, Pr = (N + 1) >> 1, nU = Pr * N, tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, h = lane >> 5, r = lane & 31;
  const int64_t fs = (int64_t)(S.begin + s) * S.sample + S.t0;  // frame of step t0
  // entries past N stay zero: U's pad column and the clamped pairs meet a zero
  for (int i = tid; i < 3 * 2 * kWideSlices * PPL; i += 64 * kWideWaves) (&L.psi[0][0])[i] = make_float2(0.f, 0.f);
  const float4 *U = reinterpret_cast<const float4 *>(S.U) + (fs - S.f_lo) * nU;
  uint32_t po[PPL], ro[RPL];
#pragma unroll
  for (int i = 0; i < PPL; ++i) po[i] = (uint32_t)(min(2 * wave + h + kWideSlices * i, Pr - 1) * N);
#pragma unroll
  for (int k = 0; k < RPL; ++k) ro[k] = (uint32_t)min(r + 32 * k, N - 1);
  float4 u[PPL][RPL];
#pragma unroll
  for (int i = 0; i < PPL; ++i)
#pragma unroll
    for (int k = 0; k < RPL; ++k) u[i][k] = gld(U + po[i] + ro[k]);
  // thread (x, a): site a of polarisation x
  const int x = tid / NR, a = tid - x * NR;
  const bool own = x < 3 && a < N;
  const float *mu = S.mu_rec + (S.mu_stride ? fs * S.mu_stride : 0) + 1 + (own ? (int64_t)x * N + a : 0);
  float m = gld(mu);
  float2 p = make_float2(own ? m : 0.f, 0.f);
  const int64_t srow = own ? (int64_t)(3 * s + x) * N + a : 0;
  if (S.t0 && own) p = gld(S.state + srow);
  __syncthreads();
  double2 *out = S.partial + (int64_t)s * T;
  for (int t = S.t0;; ++t) {
    if (S.hist) {
      const int hr = t % S.hist_every == 0 ? t / S.hist_every : t == T - 1 ? t / S.hist_every + 1 : -1;
      if (hr >= 0 && own) gst(S.hist + ((int64_t)(3 * s + x) * S.nck + hr) * N + a, p);
    }
    // publish psi(t) and this wave's part of the response mu(f).psi
    if (own) L.psi[x][a] = p;
    const float rr = group_sum<64>(own ? m * p.x : 0.f), ri = group_sum<64>(own ? m * p.y : 0.f);
    if (lane == 0) L.red[t & 1][wave] = make_float2(rr, ri);
    __syncthreads();
    if (tid == 0) {
      double2 z = make_double2(0.0, 0.0);
      for (int w = 0; w < kWideWaves; ++w) z.x += (double)L.red[t & 1][w].x, z.y += (double)L.red[t & 1][w].y;
      gst(out + t, z);
    }
    if (t == T - 1) break;
    const bool more = t + 1 < S.t1;
    mu += more ? S.mu_stride : 0;
    m = gld(mu);
    U += more ? nU : 0;  // the refills: the frame of step t + 1 < t1
    float2 y[3][RPL];
#pragma unroll
    for (int v = 0; v < 3; ++v)
#pragma unroll
      for (int k = 0; k < RPL; ++k) y[v][k] = make_float2(0.f, 0.f);
#pragma unroll
    for (int i = 0; i < PPL; ++i) {
      float4 c[3];
#pragma unroll
      for (int v = 0; v < 3; ++v)
        c[v] = *reinterpret_cast<const float4 *>(&L.psi[v][2 * (2 * wave + h + kWideSlices * i)]);
#pragma unroll
      for (int k = 0; k < RPL; ++k) {
        const float4 w = u[i][k];
        u[i][k] = gld(U + po[i] + ro[k]);
#pragma unroll
        for (int v = 0; v < 3; ++v) {
          float2 &z = y[v][k];
          z.x = fmaf(w.x, c[v].x, z.x), z.y = fmaf(w.x, c[v].y, z.y);
          z.x = fmaf(-w.y, c[v].y, z.x), z.y = fmaf(w.y, c[v].x, z.y);
          z.x = fmaf(w.z, c[v].z, z.x), z.y = fmaf(w.z, c[v].w, z.y);
          z.x = fmaf(-w.w, c[v].w, z.x), z.y = fmaf(w.w, c[v].z, z.y);
        }
      }
    }
#pragma unroll
    for (int v = 0; v < 3; ++v)
#pragma unroll
      for (int k = 0; k < RPL; ++k) {
        const float2 z = make_float2(add_xor32(y[v][k].x), add_xor32(y[v][k].y));
        if (h == 0) L.part[wave][v][r + 32 * k] = z;
      }
    __syncthreads();
    if (own) {
      float2 q[kWideWaves];
#pragma unroll
      for (int w = 0; w < kWideWaves; ++w) q[w] = L.part[w][x][a];
#pragma unroll
      for (int st = 1; st < kWideWaves; st <<= 1)
#pragma unroll
        for (int w = 0; w < kWideWaves; w += 2 * st) q[w].x += q[w + st].x, q[w].y += q[w + st].y;
      p.x += q[0].x, p.y += q[0].y;
    }
    if (!more) {
      if (own) gst(S.state + srow, p);
      break;
    }
  }
}

// Workgroup: sample wmap.y of system wmap.x.  Up to three rows per lane two
// workgroups share a CU (333 samples of a 77-site lattice on 256 CUs: propagators and
// this 1.05 ms, 1.14 with one workgroup per CU).
template <int RPL, int PPL>
__global__ void __launch_bounds__(64 * kWideWaves) __attribute__((amdgpu_waves_per_eu(RPL < 4 ? 4 : 2)))
dense_wide_kernel(const DiaSys *sys, const int2 *wmap, unsigned long long *times) {
  __shared__ __align__(16) unsigned char smem[sizeof(WideLds<RPL, PPL>)];
  const unsigned long long t_start = __builtin_amdgcn_s_memrealtime();
  const int2 wm = wmap[blockIdx.x];
  const DiaSys S = sys[__builtin_amdgcn_readfirstlane(wm.x)];
  wide_run<RPL, PPL>(S, __builtin_amdgcn_readfirstlane(wm.y), smem);
  if (threadIdx.x == 0 && times) {
    times[2 * blockIdx.x] = t_start;
    times[2 * blockIdx.x + 1] = __builtin_amdgcn_s_memrealtime();
  }
}

// Kernel by size: a wave per vector up to N = 32 (a row's half in a lane's
// registers), above it the wide kernel, which reads U once for the three
// vectors (exact propagators, 200 steps, wave and wide, ms: N = 64, 100
// samples 0.87 and 0.51, 1,500 samples 5.6 and 4.1; N = 48, 1,500 samples 3.4
// and 2.9; N = 36, 1,500 samples 2.4 and 2.6).
constexpr int kDenseWaveN = 32;
int dense_class(int N) { return N <= kDenseWaveN ? 0 : N <= 64 ? 1 : N <= 96 ? 2 : 3; }

// sys / wmap: device copies.
int launch_dense(int cls, const DiaSys *sys, const int2 *wmap, int nwg, hipStream_t st, unsigned long long *times) {
  if (nwg == 0) return NISE_OK;
  const void *fn = cls == 0 ? (const void *)dense_vectors_kernel : cls == 1 ? (const void *)dense_wide_kernel<2, 2>
                 : cls == 2 ? (const void *)dense_wide_kernel<3, 3> : cls == 3 ? (const void *)dense_wide_kernel<4, 4> : nullptr;
  if (!fn) return set_error("dense propagators: bad class %d", cls), NISE_ERR_ARG;
  void *kargs[] = {&sys, &wmap, &times};
  NISE_HIP_CHECK(hipLaunchKernel(fn, dim3((unsigned)nwg), dim3(cls ? 64 * kWideWaves : 192), kargs, 0, st));
  return NISE_OK;
}

// Costs in cycles of a Trotter run on the row conveyor and through per-frame
// propagators.  A conveyor wave walks tmax frames of nlayers dependent LDS
// round trips, each with its share of the sites, and all waves together are
// bound by LDS instructions; propagators are rotation sweeps on the N columns of
// every frame (independent of each other, so they fill the chip) and one product
// per vector step, a chain of tmax of them or bound by all vectors' products.
// The constants are fits.
struct RunCost {
  double rows, load;       // a conveyor wave's chain; the waves, in chips full
  double build;            // U of every frame
  double chain, work;      // the products: one vector's chain, all vectors' work
};
static RunCost run_cost(const TrotterRun &r) {
  const int R = rows_for(r.N, r.Kreal, r.nasap);
  const double N = r.N, T = r.T, S = (double)r.S, G = 64.0 / R;
  const double sweep = std::max({(double)r.nasap, (double)r.Kreal / R, 8.0}) * r.m;
  RunCost c;
  c.rows = T * (176.0 * sweep + 180.0 * N / R + 300.0), c.load = 3.0 * S / G / 3400.0;
  c.build = (double)r.F * std::ceil((N + (r.N & 1)) / G) / 256.0 * (21.0 * sweep + 150.0);
  if (dense_class(r.N) == 0) c.chain = T * (500.0 + 24.0 * N), c.work = T * 3.0 * S / 1024.0 * (200.0 + 12.0 * N);
  else c.chain = T * (1000.0 + 40.0 * N), c.work = S / 256.0 * c.chain;
  return c;
}
constexpr double kLaunches = 20000.0;  // of the propagators
double rows_cost(const TrotterRun &r) {
  const RunCost c = run_cost(r);
  return c.rows * (1.0 + c.load);
}

double dense_cost(const TrotterRun &r) {
  const RunCost c = run_cost(r);
  return kLaunches + c.build + std::max(c.chain, c.work);
}

static bool dense_fits(const TrotterRun &r) {
  return (int64_t)r.T * r.m <= kDenseMaxSweeps && r.N <= kDenseMaxN && r.F < (1 << 30) &&
         (double)dense_u_bytes(r.N, r.F) <= kDenseMaxBytes;
}

// A run by itself: propagators where they take less than 0.85 of the conveyor's
// time (kernels, ms, conveyor and propagators: N = 25 lattice, 1,500 samples 1.56
// and 0.59; N = 77, 333 samples 2.60 and 1.05; N = 64, 800 samples 2.43 and 1.24,
// 1,500 samples 2.72 and 3.4; N = 121, 800 samples 4.50 and 4.41.  Over 512 plans
// of lattices, 4 to 126 sites, 4 to 200 steps, 1 to 4 substeps, 4 to 2,500 samples,
// the choice is slower than the conveyor in two, by 8%).
bool dense_pays(const TrotterRun &r, double cost) { return dense_fits(r) && cost < 0.85 * rows_cost(r); }
bool dense_pays(const TrotterRun &r) { return dense_pays(r, dense_cost(r)); }

// Which Trotter runs of a batch go through propagators: those that pay by
// themselves, U of all of them within kDenseBatchBytes.  But runs that share the
// conveyor's launch fill the chip together, which gains little per run beside
// many others: only the longest of them, or none, where that takes less than
// three quarters of the time (propagators are the nearer to 64 bits, and beside a
// conveyor that leaves the chip idle they run on a second stream: half of the
// shorter side is counted; above 96 sites one workgroup fills a CU, and the
// products take 1.3 of run_cost's).  Whole calls, ms, all on the conveyor and all
// through propagators, lattices with 100 samples: N = 100, 256 steps, 1 of them
// 4.5 and 1.0, 4 4.7 and 2.7, 16 6.2 and 9.2, 48 9.4 and 26; N = 64, 200 steps, 8
// of them 3.0 and 1.7, 48 5.0 and 9.8; N = 25, 256 steps, 48 of them 4.6 and 3.9.
void dense_choice(const std::vector<TrotterRun> &runs, std::vector<char> &dense) {
  const size_t n = runs.size();
  dense.assign(n, 0);
  std::vector<RunCost> c(n);
  std::vector<size_t> order(n), pay;
  double load = 0.0, bytes = 0.0, stay = 0.0;  // stay: the longest chain that keeps the conveyor
  for (size_t i = 0; i < n; ++i) c[i] = run_cost(runs[i]), order[i] = i, load += c[i].load;
  std::stable_sort(order.begin(), order.end(), [&](size_t x, size_t y) { return c[x].rows > c[y].rows; });
  for (size_t i : order) {
    const double u = (double)dense_u_bytes(runs[i].N, runs[i].F);
    if (dense_pays(runs[i]) && bytes + u <= kDenseBatchBytes) pay.push_back(i), bytes += u;
    else stay = std::max(stay, c[i].rows);
  }
  double build = 0.0, chain[4] = {}, work[4] = {}, best = 0.0, total = 0.0;
  size_t keep = 0;
  for (size_t j = 0; j <= pay.size(); ++j) {  // the first j through propagators
    const double rows = std::max(stay, j < pay.size() ? c[pay[j]].rows : 0.0) * (1.0 + load);
    double props = build;
    for (int q = 0; q < 4; ++q) props += std::max(chain[q], work[q]);
    total = std::max(rows, props) + 0.5 * std::min(rows, props);
    if (j == 0 || total < best) best = total, keep = j;
    if (j == pay.size()) break;
    const RunCost &x = c[pay[j]];
    const int k = dense_class(runs[pay[j]].N);
    load -= x.load, build += x.build + (j ? 0.0 : kLaunches);
    chain[k] = std::max(chain[k], x.chain), work[k] += x.work * (k == 3 ? 1.3 : 1.0);
  }
  if (best >= 0.75 * total) keep = pay.size();
  for (size_t j = 0; j < keep; ++j) dense[pay[j]] = 1;
}

}  // namespace nise
