// Absorption vectors of nearest-neighbour chains (every kept coupling joins
// sites j and j + 1), forward and adjoint, as a systolic array over frames.
//
// A chain's sweep is one dependent sequence of rotations (0,1), (1,2), ...
// per frame, so the row conveyor gives a vector one lane and walks
// tmax (N - 1) LDS round trips; a thousand samples are 47 waves.  But rotation
// (j, j+1) of frame f + 1 needs only sites up to j + 1 of frame f.  Here R
// lanes share a vector: lane q holds sweep n = q, q + R, ... of the vector's
// sequence and runs two sites behind lane q - 1, which hands it each finished
// site in a register (wave_shr DPP); lane 0 takes lane R - 1's sites, which
// wait in LDS.  The pair being rotated lives in registers.  Every operation
// and its rounding are the row conveyor's with one row (src/propagate.c:
// 843-899), so the forward results are bit for bit the same.
//
// A frame's table entry of site j is one record of 32 bytes: the half-step
// phase D_j, (cos, sin) and f J of the pair (j - 1, j), and the dipoles of j;
// a lane reads its records in order, kAhead steps before their use, and the
// lanes of a wave cover R frames, so the records' 128-byte lines are used from
// L1.  What bounds it is the instruction issue of a lone wave (about 100
// instructions a step forward, 200 backward, 7 cycles each) times tmax / R (N + 1)
// steps: a thousand samples are one wave per SIMD.  Measured, with tables and sums
// (N = 128, 1,000 samples of 256 steps): forward 6.14 ms in the row conveyor,
// 0.68 here; backward 14.4 and 0.84 ms.  N = 16, 200 samples of 128 steps: 0.45
// and 0.145 ms (0.128 through propagators, dense.hip, whose rounding differs
// and which fall behind from N = 32 or 1,000 samples on: 0.37 and 0.19 ms).
#include <algorithm>
#include <vector>

#include "nise_internal.h"

namespace nise {

__device__ __forceinline__ uint32_t lane_below(uint32_t x) {  // lane - 1's x (lane 0: 0)
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x138, 0xF, 0xF, false);
}
__device__ __forceinline__ float2 lane_below(float2 p) {
  return make_float2(__uint_as_float(lane_below(__float_as_uint(p.x))), __uint_as_float(lane_below(__float_as_uint(p.y))));
}
__device__ __forceinline__ double lane_below(double d) {
  const unsigned long long u = __double_as_longlong(d);
  const uint32_t lo = lane_below((uint32_t)u), hi = lane_below((uint32_t)(u >> 32));
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// A copy of x in a register of its own: without it the compiler keeps the
// record that Dc, ... come from (or what is left to compute from it) in place,
// lets its refill land elsewhere and moves it home at the end of the unrolled
// steps, waiting for the loads just issued.
__device__ __forceinline__ float own(float x) {
  float y;
  asm volatile("v_mov_b32 %0, %1" : "=v"(y) : "v"(x));
  return y;
}
__device__ __forceinline__ float2 own(float2 x) { return make_float2(own(x.x), own(x.y)); }

// Records of every frame: rec[2 (row N + j)] = (D_j, cos, sin), + 1 = (f J,
// mu_x, mu_y, mu_z); the arithmetic of frame_tables_kernel.
__global__ void __launch_bounds__(256) chain_tables_kernel(FrameSource s, int N, int64_t f_lo, int64_t nfr, float fac,
                                                           const float *mu_rec, int64_t mu_stride, float4 *rec) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= nfr * N) return;
  const int64_t f = f_lo + e / N;
  const int j = (int)(e % N);
  // src/propagate.c:863-866
  float h = site_energy(s, N, f, j);
  if (s.delta) h = __fadd_rn(h, s.delta[j]);
  const double arg = 0.5 * (double)h * (double)fac;
  const float J = j ? kept_coupling(s, N, f, j - 1, j) : 0.f;
  float co = 1.f, si = 0.f;
  if (J != 0.f) {  // src/propagate.c:879-882
    const float Jf = __fmul_rn(__fmul_rn(J, s.cscale), fac);
    si = (float)(-sin((double)Jf));
    co = (float)sqrt((double)__fsub_rn(1.0f, __fmul_rn(si, si)));
  }
  const float *mu = mu_rec + (mu_stride ? f * mu_stride : 0) + 1 + j;
  gst(rec + 2 * e, make_float4((float)cos(arg), (float)(-sin(arg)), co, si));
  gst(rec + 2 * e + 1, make_float4(__fmul_rn(J, fac), gld(mu), gld(mu + N), gld(mu + 2 * N)));
}

int launch_chain_tables(const FrameSource &src, int N, int64_t f_lo, int64_t nfr, float fac, const float *mu_rec,
                        int64_t mu_stride, float4 *rec, hipStream_t st) {
  hipLaunchKernelGGL(chain_tables_kernel, dim3((unsigned)((nfr * N + 255) / 256)), dim3(256), 0, st, src, N, f_lo, nfr,
                     fac, mu_rec, mu_stride, rec);
  NISE_HIP_CHECK(hipGetLastError());
  return NISE_OK;
}

// Steps between a lane's sweeps: N + 1 (site N - 1 leaves at step N), and at
// least 2 R + 2, by when lane R - 1 has stored what lane 0 reads one step
// ahead.
__host__ __device__ inline int chain_period(int N, int R) { return N + 1 > 2 * R + 2 ? N + 1 : 2 * R + 2; }

// A lane's sweep: substep sub of step t (no division per sweep: with m = 1,
// R and m uniform, step() is two adds).
struct Sweep {
  int t, sub;
  __device__ Sweep(int n, int m) : t(n / m), sub(n - n / m * m) {}
  __device__ void step(int R, int m) {
    const int d = R / m;  // uniform
    t += d, sub += R - d * m;
    if (sub >= m) sub -= m, ++t;
  }
};

constexpr int kAhead = 4;  // steps from a record's load to its use (L2 latency; 8 registers a step backward)

// Forward of the vectors [group V, group V + V) of one system.
template <int R>
__device__ __forceinline__ void chain_run(const ChainArgs &A, int group, unsigned char *smem) {
  constexpr int V = 64 / R;
  const int N = A.N, T = A.T, m = A.m, P = chain_period(N, R), M = (T - 1) * m + 1;
  const int lane = threadIdx.x, vs = min(lane / R, V - 1), q = lane - vs * R;  // lanes past V R: q >= R, idle
  const int v = group * V + vs, vv = min(v, A.nvec - 1), x = vv % 3;
  const bool has = q < R && v < A.nvec;
  const uint32_t row0 = (uint32_t)((int64_t)(A.begin + vv / 3) * A.sample - A.f_lo);
  float2 *ret = reinterpret_cast<float2 *>(smem) + vs * N;  // lane R - 1's sites for lane 0

  // sweep n: substep n % m of relative time n / m; sweep M - 1 only responds
  int j = -2 * q;
  Sweep w(q, m);
  bool resp;
  float2 *hp;
  auto sweep = [&] {
    resp = has && w.sub == 0 && w.t < T;
    hp = nullptr;
    if (A.hist && resp) {
      const int c = w.t / A.hist_every;
      const bool on = c * A.hist_every == w.t;
      if (on || w.t == T - 1) hp = A.hist + ((int64_t)v * A.nck + c + !on) * N;
    }
  };
  sweep();
  // records in flight: jp, wp, base run kAhead steps ahead of j, w
  int jp = j;
  Sweep wp = w;
  uint32_t base = (row0 + (uint32_t)min(wp.t, T - 1)) * (uint32_t)N;
  float4 ra[kAhead];
  float rm[kAhead];
  auto fetch = [&](int k) {
    const float4 *r = A.rec + 2 * (base + (uint32_t)min(max(jp, 0), N - 1));
    ra[k] = gld(r);
    rm[k] = gld(reinterpret_cast<const float *>(r) + 5 + x);
    if (++jp == P) {
      jp = 0, wp.step(R, m);
      base = (row0 + (uint32_t)min(wp.t, T - 1)) * (uint32_t)N;
    }
  };
#pragma unroll
  for (int k = 0; k < kAhead; ++k) fetch(k);

  const int steps = (M - 1) / R * P + 2 * ((M - 1) % R) + N;
  float2 carry = make_float2(0.f, 0.f), out = carry, back = carry, Dc = carry;
  float rr = 0.f, ri = 0.f;
  bool first = q == 0;  // sweep 0
  for (int k0 = 0; k0 < steps; k0 += kAhead) {
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
      const float2 D = make_float2(ra[k].x, ra[k].y);
      const float co = ra[k].z, si = ra[k].w, mm = rm[k];
      float2 p = lane_below(out);
      p = q == 0 ? back : p;
      back = ret[(unsigned)(j + 1) < (unsigned)N ? j + 1 : 0];  // lane 0's of the next step
      if (first) p = make_float2(mm, 0.f);  // psi(0) = mu (src/absorption.c:92-146)
      rr = __fadd_rn(j == 0 ? 0.f : rr, __fmul_rn(mm, p.x));
      ri = __fadd_rn(j == 0 ? 0.f : ri, __fmul_rn(mm, p.y));
      if (hp && (unsigned)j < (unsigned)N) gst(hp + j, p);
      // site j enters: opening half-phase, rotation with site j - 1, whose
      // closing half-phase follows (j == N: site N - 1 leaves)
      float2 pb = cmul_diag(p, D), pa = carry;
      const float2 p0 = pb;
      rotate_pair(pa, pb, co, si);
      pa = j == N ? carry : pa;
      carry = own(j == 0 ? p0 : pb);
      out = cmul_diag(pa, Dc);
      Dc = own(D);
      if (q == R - 1 && j >= 1 && j <= N) ret[j - 1] = out;
      if (j == N - 1 && resp) gst(A.partial + (int64_t)v * T + w.t, make_double2((double)rr, (double)ri));
      if (++j == P) j = 0, first = false, w.step(R, m), sweep();
      fetch(k);
      __builtin_amdgcn_wave_barrier();  // other lanes' LDS accesses keep their order
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

template <int R>
__global__ void __launch_bounds__(64) chain_kernel(ChainArgs A) {
  extern __shared__ __align__(16) unsigned char smem[];
  chain_run<R>(A, blockIdx.x, smem);
}

// The chains of a batch, each with its own R: workgroup = group wmap.y of
// system wmap.x, with its start and end on the device clock.  One launch, because
// one system's few waves leave the chip idle (48 chains of 64 sites, 100 samples of
// 256 steps, whole call: one launch after the other 12.8 ms, the row conveyor 6.7,
// this 2.5).
__global__ void __launch_bounds__(64) chain_batch_kernel(const ChainArgs *sys, const int2 *wmap,
                                                         unsigned long long *times) {
  extern __shared__ __align__(16) unsigned char smem[];
  const unsigned long long t_start = __builtin_amdgcn_s_memrealtime();
  const int2 wm = wmap[blockIdx.x];
  const ChainArgs A = sys[__builtin_amdgcn_readfirstlane(wm.x)];
  const int group = __builtin_amdgcn_readfirstlane(wm.y);
  if (A.R == 21) chain_run<21>(A, group, smem);
  else if (A.R == 10) chain_run<10>(A, group, smem);
  else chain_run<5>(A, group, smem);
  if (threadIdx.x == 0) {
    times[2 * blockIdx.x] = t_start;
    times[2 * blockIdx.x + 1] = __builtin_amdgcn_s_memrealtime();
  }
}

// Backward (the recursion of adjoint.hip): sweep n undoes substep n, counted
// from the last, of the vectors' T - 1 steps; sites enter from N - 1 down.
// With phi and chi a site hands on its offset gradient, summed in FP64 over
// the sweeps; past the last sweep the lanes only pass it through.
template <int R>
__global__ void __launch_bounds__(64) chain_adjoint_kernel(ChainArgs A) {
  constexpr int V = 64 / R;
  extern __shared__ __align__(16) unsigned char smem[];
  const int N = A.N, T = A.T, m = A.m, P = chain_period(N, R), M = (T - 1) * m;
  const int lane = threadIdx.x, vs = min(lane / R, V - 1), q = lane - vs * R;
  const int v = blockIdx.x * V + vs, vv = min(v, A.nvec - 1), x = vv % 3;
  const bool has = q < R && v < A.nvec;
  auto row_of = [&](int vec) { return (uint32_t)((int64_t)(A.begin + vec / 3) * A.sample - A.f_lo); };
  const uint32_t row0 = row_of(vv);
  float4 *st0 = reinterpret_cast<float4 *>(smem);                  // [V][N] (phi, chi)
  double *ac0 = reinterpret_cast<double *>(st0 + (size_t)V * N);   // [V][N]
  float2 *gs = reinterpret_cast<float2 *>(ac0 + (size_t)V * N);    // [T]
  for (int i = lane; i < T; i += 64) gs[i] = gld(A.g + i);
  {  // psi(T-1) and lambda(T-1) = g(T-1) mu(T-1)
    const float2 gl = gld(A.g + (T - 1));
    for (int i = lane; i < V * N; i += 64) {
      const int vec = min(blockIdx.x * V + i / N, A.nvec - 1), site = i % N;
      const float2 p = gld(A.ck + ((int64_t)vec * A.nck + A.nck - 1) * N + site);
      const float mm = gld(reinterpret_cast<const float *>(A.rec + 2 * ((row_of(vec) + T - 1) * (uint32_t)N + site)) + 5 + vec % 3);
      st0[i] = make_float4(p.x, p.y, __fmul_rn(gl.x, mm), __fmul_rn(gl.y, mm));
      ac0[i] = 0.0;
    }
  }
  __builtin_amdgcn_wave_barrier();
  float4 *st = st0 + vs * N;
  double *ac = ac0 + vs * N;
  const float hf = 0.5f * A.fac;

  int s = -2 * q;  // local step s: site N - 1 - s enters, N - s leaves
  bool real, fin, reset;
  float2 gv;
  Sweep w(q, m);  // w.t steps and w.sub substeps undone before this sweep
  auto sweep = [&] {
    const int t = T - 2 - w.t;
    real = has && t >= 0;
    fin = real && w.sub == m - 1;
    reset = fin && t % A.every == 0;
    gv = gs[max(t, 0)];
  };
  sweep();
  int sp = s;
  Sweep wp = w;
  uint32_t base;
  const float2 *ckp;  // checkpoint row of the sweep being fetched, or null
  auto source = [&] {
    const int t = T - 2 - wp.t, tc = max(t, 0);
    base = (row0 + (uint32_t)tc) * (uint32_t)N;
    ckp = t >= 0 && wp.sub == m - 1 && tc % A.every == 0 ? A.ck + ((int64_t)vv * A.nck + tc / A.every) * N : nullptr;
  };
  source();
  float4 ra[kAhead], rb[kAhead];
  float2 rk[kAhead];
  auto fetch = [&](int k) {
    const int site = min(max(N - 1 - sp, 0), N - 1);
    const float4 *r = A.rec + 2 * (base + (uint32_t)site);
    ra[k] = gld(r), rb[k] = gld(r + 1);
    rk[k] = gld(ckp ? ckp + site : A.ck);  // the other lanes read one common entry
    if (++sp == P) sp = 0, wp.step(R, m), source();
  };
#pragma unroll
  for (int k = 0; k < kAhead; ++k) fetch(k);

  const int steps = M ? (M - 1) / R * P + 2 * (R - 1) + N + 1 : 0;
  float4 out = make_float4(0.f, 0.f, 0.f, 0.f), back = st[N - 1], cb = out;
  double oacc = 0.0, bacc = 0.0, cacc = 0.0, cg = 0.0;
  // the record of the site that entered last
  float2 Dc = make_float2(1.f, 0.f), cs = Dc, kc = Dc;
  float jc = 0.f, mc = 0.f;
  for (int k0 = 0; k0 < steps; k0 += kAhead) {
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
      const float4 r = ra[k], r1 = rb[k];
      const float2 ck = rk[k];
      float2 phi = lane_below(make_float2(out.x, out.y)), chi = lane_below(make_float2(out.z, out.w));
      double acc = lane_below(oacc);
      phi = q == 0 ? make_float2(back.x, back.y) : phi, chi = q == 0 ? make_float2(back.z, back.w) : chi;
      acc = q == 0 ? bacc : acc;
      const int nx = (unsigned)(s + 1) < (unsigned)N ? N - 2 - s : N - 1;  // enters lane 0 at the next step
      back = st[nx], bacc = ac[nx];
      // site a = N - 1 - s enters: closing half-phase undone
      const float2 D = make_float2(r.x, r.y);
      acc += (double)(real ? hf * im_cj(chi, phi) : 0.f);
      const float2 pa0 = cmul_conj_d(phi, D), xa0 = cmul_conj_d(chi, D);
      // rotation with site b = a + 1 undone (s == 0, N: none)
      float2 pa = pa0, xa = xa0, pb = make_float2(cb.x, cb.y), xb = make_float2(cb.z, cb.w);
      const float cf = jc * (im_cj(xa, pb) + im_cj(xb, pa));
      cg += (double)(real && s > 0 && s < N ? cf : 0.f);
      rotate_back(pa, pb, cs.x, cs.y);
      rotate_back(xa, xb, cs.x, cs.y);
      const bool end = s == N, top = s == 0;
      pb = end ? make_float2(cb.x, cb.y) : pb, xb = end ? make_float2(cb.z, cb.w) : xb;
      // site b leaves: opening half-phase undone, response term, checkpoint
      oacc = cacc + (double)(real ? hf * im_cj(xb, pb) : 0.f);
      pb = cmul_conj_d(pb, Dc), xb = cmul_conj_d(xb, Dc);
      const float2 xg = make_float2(__fadd_rn(xb.x, __fmul_rn(gv.x, mc)), __fadd_rn(xb.y, __fmul_rn(gv.y, mc)));
      xb = fin ? xg : xb;
      pb = reset ? kc : pb;
      out = make_float4(pb.x, pb.y, xb.x, xb.y);
      pa = top ? pa0 : pa, xa = top ? xa0 : xa;
      cb = make_float4(pa.x, pa.y, xa.x, xa.y), cacc = acc;
      Dc = own(D), cs = own(make_float2(r.z, r.w)), jc = own(r1.x), kc = own(ck);
      mc = own(x == 0 ? r1.y : x == 1 ? r1.z : r1.w);
      if (q == R - 1 && s >= 1 && s <= N) st[N - s] = out, ac[N - s] = oacc;
      if (++s == P) s = 0, w.step(R, m), sweep();
      fetch(k);
      __builtin_amdgcn_wave_barrier();  // other lanes' LDS accesses keep their order
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) cg += __shfl_xor(cg, off);
  for (int i = lane; i < N; i += 64) {
    double d = 0.0;
    for (int u = 0; u < V; ++u) d += ac0[u * N + i];
    gst(A.part_delta + (int64_t)blockIdx.x * N + i, d);
  }
  if (lane == 0) gst(A.part_c + blockIdx.x, cg);
}

// LDS of a workgroup, forward and backward.
static size_t chain_smem_fwd(int N, int R) { return (size_t)(64 / R) * N * 8; }
static size_t chain_smem(int N, int T, int R) { return (size_t)(64 / R) * N * 24 + (size_t)T * 8; }

// Steps of a launch, times the waves that share a SIMD.
static double chain_steps(int N, int T, int m, int64_t nvec, int R) {
  const int64_t M = (int64_t)(T - 1) * m + 1;
  return ((double)((M - 1) / R) * chain_period(N, R) + 2 * R + N) *
         std::max(1.0, (double)((nvec + 64 / R - 1) / (64 / R)) / 1024.0);
}

// Fewer lanes per vector where a short chain would leave lanes idle (the
// period is at least 2 R + 2 steps): the R with the fewest steps.  nvec: all
// vectors of the launch.
int chain_rows(int N, int T, int m, int64_t nvec, int64_t nfr) {
  if (nfr * N >= (int64_t)1 << 30) return 0;  // 32-bit record indexes
  if (((int64_t)(T - 1) * m + 1) * (N + 1) >= (int64_t)1 << 30) return 0;
  int best = 0;
  double cost = 0.0;
  for (int R : {21, 10, 5}) {
    if (chain_smem(N, T, R) > 160 * 1024) continue;
    const double c = chain_steps(N, T, m, nvec, R);
    if (!best || c < cost) best = R, cost = c;
  }
  return best;
}

// (a step takes about 700 cycles: N = 128, 1,000 samples of 256 steps, 1,600 steps
// in 0.55 ms; N = 16, 200 samples of 128, 286 in 0.09)
bool chain_pays(const TrotterRun &r, int R, int windows, int per) {
  return windows * (20000.0 + 700.0 * chain_steps(r.N, r.T, r.m, 3 * (int64_t)per, R)) < rows_cost(r);
}

static int launch_chain_fn(const void *fn, const ChainArgs &a, size_t smem, hipStream_t st) {
  const int nwg = chain_groups(a.nvec, a.R);
  if (nwg <= 0) return NISE_OK;
  if (!fn || smem > 160 * 1024) return set_error("chain: N=%d with %d lanes per vector", a.N, a.R), NISE_ERR_ARG;
  NISE_HIP_CHECK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
  ChainArgs args = a;
  void *kargs[] = {&args};
  NISE_HIP_CHECK(hipLaunchKernel(fn, dim3((unsigned)nwg), dim3(64), kargs, smem, st));
  return NISE_OK;
}

int launch_chain(const ChainArgs &a, hipStream_t st) {
  return launch_chain_fn(a.R == 21 ? (const void *)chain_kernel<21> : a.R == 10 ? (const void *)chain_kernel<10>
                         : a.R == 5 ? (const void *)chain_kernel<5> : nullptr, a, chain_smem_fwd(a.N, a.R), st);
}

int launch_chain_adjoint(const ChainArgs &a, double *out, hipStream_t st) {
  const int rc = launch_chain_fn(a.R == 21 ? (const void *)chain_adjoint_kernel<21>
                                 : a.R == 10 ? (const void *)chain_adjoint_kernel<10>
                                 : a.R == 5 ? (const void *)chain_adjoint_kernel<5> : nullptr, a,
                                 chain_smem(a.N, a.T, a.R), st);
  if (rc) return rc;
  return launch_adjoint_reduce(a.part_delta, a.part_c, chain_groups(a.nvec, a.R), a.N, out, st);
}

// Workgroups of a batch's chains, the longest first.
void chain_batch_map(const std::vector<ChainArgs> &sys, std::vector<int2> &wmap) {
  std::vector<int> order(sys.size());
  for (size_t i = 0; i < sys.size(); ++i) order[i] = (int)i;
  auto steps = [&](int i) {
    const ChainArgs &a = sys[i];
    return ((int64_t)(a.T - 1) * a.m / a.R + 1) * chain_period(a.N, a.R);
  };
  std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return steps(x) > steps(y); });
  wmap.clear();
  for (int i : order)
    for (int g = 0; g < chain_groups(sys[i].nvec, sys[i].R); ++g) wmap.push_back(make_int2(i, g));
}

// sys_h / nwg: host descriptors and chain_batch_map's size; sys / wmap: device copies.
int launch_chain_batch(const std::vector<ChainArgs> &sys_h, const ChainArgs *sys, const int2 *wmap, int nwg,
                       hipStream_t st, unsigned long long *times) {
  if (nwg <= 0) return NISE_OK;
  size_t smem = 0;
  for (const ChainArgs &a : sys_h) {
    smem = std::max(smem, chain_smem_fwd(a.N, a.R));
    if (smem > 160 * 1024 || !(a.R == 21 || a.R == 10 || a.R == 5))
      return set_error("chain: N=%d with %d lanes per vector", a.N, a.R), NISE_ERR_ARG;
  }
  const void *fn = (const void *)chain_batch_kernel;
  NISE_HIP_CHECK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
  void *kargs[] = {&sys, &wmap, &times};
  NISE_HIP_CHECK(hipLaunchKernel(fn, dim3((unsigned)nwg), dim3(64), kargs, smem, st));
  return NISE_OK;
}

bool chain_mask(int N, const std::vector<uint8_t> &mask) {
  int64_t k = 0, near = 0, all = 0;
  for (int a = 0; a < N; ++a)
    for (int b = a + 1; b < N; ++b, ++k)
      if (mask[k]) ++all, near += b == a + 1;
  return all && near == all;
}

}  // namespace nise
