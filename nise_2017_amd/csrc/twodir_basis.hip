// 2DIR / 2DUVvis through one-exciton basis vectors (no waiting time, Trotter
// scheme).
//
// Every term of the response (src/calc_2DIR.c:184-506) is linear in the t1
// seed L0[x0][t1] (mu_x0(tj - t1) propagated to tj) or in its conjugate:
//   kI[m](t3, t1)  = sum_i conj(L0[x0][t1]_i) VI_m(t3)_i
//   kII[m](t3, t1) = sum_i L0[x0][t1]_i VII_m(t3)_i
// with, for the item m = (x0, x1, x2, x3), U(t3) the one-exciton propagator
// from tj to tj + t3, M_x = U mu_x(tj), r_x3 = U^T mu_x3(tj + t3), q_y,x3 =
// mu_x3(tj + t3) . M_y and mu+ / mu- the transitions to and from the
// two-exciton states (propagator U2):
//   VI  = - mu_x1(tj) q_x2,x3 - mu_x2(tj) q_x1,x3 + U^+ mu-_x3 U2 mu+_x2 mu_x1(tj)
//   VII = - mu_x1(tj) q_x2,x3 - (mu_x1(tj) . mu_x2(tj)) r_x3 + W_m,
//   W_m,i = M_x1^+ mu-_x3 U2 mu+_x2 e_i
// (ground-state bleach, stimulated emission, excited-state absorption).  The
// vectors that must be propagated per sample are therefore the N columns of
// U, the 3 N two-exciton vectors mu+_x2 e_i and the nine mu+_x2 mu_x1, in
// place of 3 T1 + 3 one-exciton and 9 T1 + 9 two-exciton vectors: at N = 32
// and T1 = 64 35 and 105 against 195 and 585.  The sum over samples, seeds
// and items is one matrix product with FP64 sums.
//
// Stages: singles_seeds_kernel (L0), singles_basis_kernel (columns of U and
// M), dbl_basis_kernel (W and mu- U2 mu+ mu), combine_kernel (VI, VII summed
// over the items of each x0 with the three lab weights, in FP64),
// contract_kernel (the product with L0), finish_kernel (sum over sample
// chunks, lifetime factor).  Measured at N = 32, T1 = T3 = 64, 200 samples:
// 4.3 ms per call, 19.3 with every vector propagated; N = 7 (T1 48, T3 40, 60
// samples) 0.51 and 2.24 ms.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "doubles_dev.h"
#include "lanes.h"
#include "nise_internal.h"
#include "persist_dev.h"
#include "twodir_basis.h"

namespace nise {

struct BasisArgs {
  int N, T1, T3, S, s0, sample, m;
  int do_gb, do_se, do_ea, es;
  float anh;                // fixed anharmonicity (0: per-frame records)
  int64_t f_lo;
  const float *mu_rec;
  int64_t mu_stride;        // 0: static dipoles
  const float *over_rec;    // overtone dipole records when anh == 0
  const float2 *diag;       // [frame - f_lo][N] half-step phases
  const float2 *cs;         // [frame - f_lo][Kp] (cos, sin) in the program's order
  const uint32_t *prog;     // [Kp] rotation words in groups (sweep_program)
  int Kp;
  float2 *L0;               // [S][3][N][T1]
  float2 *UB;               // [S][T3][N][N + 3]: columns of U, then M_x
  int K2;
  const uint32_t *ab2;      // kept couplings (lexicographic)
  const float2 *D2;         // [frame - f_lo][N2]
  const float4 *cs2;        // [frame - f_lo][K2]
  float2 *W;                // [S][T3][27][N], (x1 x2 x3)
  float2 *Lr;               // [S][T3][27][N] mu-_x3 U2 mu+_x2 mu_x1
  double2 *V;               // [S][T3][3][N][6]: kI of the three lab weights, then kII
  const float *wpl;         // [3][21]
};

__device__ __forceinline__ int64_t tj_of(const BasisArgs &A, int s) { return (int64_t)(A.s0 + s) * A.sample + A.T1; }
__device__ __forceinline__ const float *mu_of(const BasisArgs &A, int64_t f, int x) {
  return A.mu_rec + (A.mu_stride ? f * A.mu_stride : 0) + 1 + (int64_t)x * A.N;
}

// ---------------------------------------------------------------------------
// One-exciton sweeps with one vector per lane.  All 64 vectors of a wave are
// at the same frame, so a rotation is wave-uniform: its sites are a scalar
// program word; the state is psi[site][lane] in LDS.  A wave has a SIMD to
// itself, so the chain of LDS round trips sets the time: the rotations run in
// the layered order (build_schedule: a layer's rotations share no site), up
// to kGroup of a layer per group, whose reads are all in flight together.
// (Keeping site a in registers over its lexicographic chain and reading ahead
// of the last store needs branches between the reads; it ran 9 us a frame at
// the N = 32 ring against 7 here.)
//
// The rotation takes the reference's rounded (cos, sin) (src/propagate.c
// :879-882), so that the norm drift which the rounded cosine of a static
// coupling causes is the reference's; the products are fused, the small one
// (sin) rounded first, which leaves about one rounding per value.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void rot_fma(float2 &pa, float2 &pb, float co, float si) {
  const float ax = fmaf(co, pa.x, -(si * pb.y)), ay = fmaf(co, pa.y, si * pb.x);
  pb = make_float2(fmaf(co, pb.x, -(si * pa.y)), fmaf(co, pb.y, si * pa.x));
  pa = make_float2(ax, ay);
}
__device__ __forceinline__ float2 cmul_f(float2 c, float2 u) {
  return make_float2(fmaf(-c.y, u.y, c.x * u.x), fmaf(c.y, u.x, c.x * u.y));
}

constexpr int kGroup = 4;
// Groups of the layered schedule: kGroup words a | b << 8 each, the first
// with the group's rotation count << 16; unused words are dummy pairs on the
// scratch site N.  pairs: the same entries as a | b << 16 for the tables.
void sweep_program(const Schedule &s, std::vector<uint32_t> &prog, std::vector<uint32_t> &pairs) {
  prog.clear(), pairs.clear();
  const uint32_t N = (uint32_t)s.N;
  for (int l = 0; l < s.nlayers(); ++l)
    for (int r = s.layer_off[l]; r < s.layer_off[l + 1]; r += kGroup) {
      const int n = std::min(kGroup, s.layer_off[l + 1] - r);
      for (int u = 0; u < kGroup; ++u) {
        const uint32_t a = u < n ? s.ab[r + u] & 0xffffu : N, b = u < n ? s.ab[r + u] >> 16 : N;
        prog.push_back(a | b << 8 | (u == 0 ? (uint32_t)n << 16 : 0u));
        pairs.push_back(a | b << 16);
      }
    }
}

// Words and coefficients reach the sweep in segments of 64 entries, one per
// lane, and from there by v_readlane: no memory wait inside a segment.  The
// segment after the one in use (the first of the next frame's after the last)
// is in flight.  (Scalar loads of the words waited about 200 cycles in every
// group; scalar loads of the coefficients missed their cache in every frame.)
struct Segment {
  uint32_t w;
  float2 c;
};
__device__ __forceinline__ Segment load_segment(const BasisArgs &A, int lane, int64_t row, int k0) {
  if (A.Kp == 0) return Segment{0u, make_float2(1.f, 0.f)};
  const int k = min(k0 + lane, A.Kp - 1);
  return Segment{gld(A.prog + k), gld(A.cs + row * A.Kp + k)};
}
__device__ __forceinline__ float lane_f(float x, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
}

// The first M rotations of the group at entry l of the segment.
template <int M>
__device__ __forceinline__ void rot_group(float2 *col, const Segment &s, int l) {
  float2 *qa[M], *qb[M], pa[M], pb[M];
#pragma unroll
  for (int u = 0; u < M; ++u) {
    const uint32_t w = __builtin_amdgcn_readlane(s.w, l + u);
    qa[u] = col + (int)(w & 0xffu) * 64, qb[u] = col + (int)((w >> 8) & 0xffu) * 64;
    pa[u] = *qa[u], pb[u] = *qb[u];
  }
#pragma unroll
  for (int u = 0; u < M; ++u) {
    rot_fma(pa[u], pb[u], lane_f(s.c.x, l + u), lane_f(s.c.y, l + u));
    *qa[u] = pa[u], *qb[u] = pb[u];
  }
}

// One sweep of table row `row` over the wave's vectors (its first segment in
// T, on return the first segment of row `nrow`).
__device__ __forceinline__ void sweep(const BasisArgs &A, Segment &T, float2 *psi, int lane, int64_t row, int64_t nrow) {
  float2 *col = psi + lane;
  for (int k0 = 0; k0 < A.Kp; k0 += 64) {
    const Segment s = T;
    const bool more = k0 + 64 < A.Kp;
    T = load_segment(A, lane, more ? row : nrow, more ? k0 + 64 : 0);
    const int n = min(64, A.Kp - k0);
    for (int l = 0; l < n; l += kGroup) {
      const int m = (int)(__builtin_amdgcn_readlane(s.w, l) >> 16);
      if (m == 1) rot_group<1>(col, s, l);
      else if (m == 2) rot_group<2>(col, s, l);
      else rot_group<kGroup>(col, s, l);  // three rotations: the fourth on the scratch site
    }
  }
}

// LDS of a one-exciton wave: the vectors, the phases of two frames and one
// dipole row.
struct SinglesLds {
  float2 *psi, *D;  // [N + 1][64], [2][64]
  float *mu;        // [64]
};
static size_t singles_smem(int N) { return (size_t)(N + 1) * 512 + 2 * 512 + 256; }
__device__ __forceinline__ SinglesLds singles_lds(unsigned char *smem, int N) {
  SinglesLds L;
  L.psi = reinterpret_cast<float2 *>(smem), L.D = L.psi + (size_t)(N + 1) * 64;
  L.mu = reinterpret_cast<float *>(L.D + 128);
  return L;
}
// The per-site pass: p = psi Dp (not at FIRST), p = at(site, p), psi = p Dc
// (not at LAST), in batches whose LDS reads are all issued before the first
// store (the compiler keeps a read of D behind a store of psi).  The last
// batch runs past N on the scratch site (D and mu hold 64 entries).
constexpr int kSiteB = 8;
template <bool FIRST, bool LAST, class At>
__device__ __forceinline__ void site_batches(const SinglesLds &L, const float2 *Dp, const float2 *Dc, int lane, int N,
                                             At at) {
  for (int k0 = 0; k0 < N; k0 += kSiteB) {
    float2 p[kSiteB], dp[kSiteB], dc[kSiteB];
#pragma unroll
    for (int u = 0; u < kSiteB; ++u) {
      p[u] = L.psi[min(k0 + u, N) * 64 + lane];
      if constexpr (!FIRST) dp[u] = Dp[k0 + u];
      if constexpr (!LAST) dc[u] = Dc[k0 + u];
    }
#pragma unroll
    for (int u = 0; u < kSiteB; ++u) {
      if constexpr (!FIRST) p[u] = cmul_f(p[u], dp[u]);
      p[u] = at(k0 + u, p[u]);
    }
    if constexpr (!LAST) {
#pragma unroll
      for (int u = 0; u < kSiteB; ++u) L.psi[min(k0 + u, N) * 64 + lane] = cmul_f(p[u], dc[u]);
    }
  }
}

// The substeps of a frame (its opening and closing half-phases are the
// callers'): psi *= D^2 between them.
__device__ __forceinline__ void frame_sweeps(const BasisArgs &A, Segment &T, const SinglesLds &L, const float2 *D,
                                             int lane, int64_t row, int64_t nrow) {
  for (int sub = 0; sub < A.m; ++sub) {
    if (sub)
      for (int k = 0; k < A.N; ++k) L.psi[k * 64 + lane] = cmul_f(cmul_f(L.psi[k * 64 + lane], D[k]), D[k]);
    sweep(A, T, L.psi, lane, row, sub + 1 < A.m ? row : nrow);
  }
}

// L0[s][x][k][t1]: mu_x(tj - t1) through frames tj - t1 .. tj - 1
// (src/calc_2DIR.c:215-239); one wave per (sample, x, 64 values of t1).  A
// lane's column is zero until its own start frame.  The phases and dipoles
// of the next frame are in flight during a frame.
__global__ void __launch_bounds__(64) singles_seeds_kernel(BasisArgs A) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int s = blockIdx.x, x = blockIdx.y, lane = threadIdx.x, N = A.N, T1 = A.T1;
  const SinglesLds L = singles_lds(smem, N);
  const int t1 = blockIdx.z * 64 + lane, tl = min(T1 - 1, (int)blockIdx.z * 64 + 63), lc = min(lane, N - 1);
  const int64_t tj = tj_of(A, s), f0 = tj - tl;
  for (int k = 0; k <= N; ++k) L.psi[k * 64 + lane] = make_float2(0.f, 0.f);
  Segment T = load_segment(A, lane, f0 - A.f_lo, 0);
  float2 dn = gld(A.diag + (f0 - A.f_lo) * N + lc);
  float mn = gld(mu_of(A, f0, x) + lc);
  for (int64_t f = f0; f <= tj; ++f) {
    const int64_t row = f - A.f_lo;
    const bool start = tj - f == t1, first = f == f0, last = f == tj;
    float2 *Dc = L.D + (f & 1) * 64;
    const float2 *Dp = L.D + ((f + 1) & 1) * 64;
    Dc[lane] = dn, L.mu[lane] = mn;
    if (!last) dn = gld(A.diag + (row + 1) * N + lc), mn = gld(mu_of(A, f + 1, x) + lc);
    // closing half-phase of f - 1, start, opening half-phase of f
    auto pass = [&](auto fst, auto lst) {
      constexpr bool kF = decltype(fst)::value, kL = decltype(lst)::value;
      site_batches<kF, kL>(L, Dp, Dc, lane, N, [&](int k, float2 p) {
        p = start ? make_float2(L.mu[k], 0.f) : p;
        if (kL && t1 < T1 && k < N) gst(A.L0 + (((int64_t)s * 3 + x) * N + k) * T1 + t1, p);
        return p;
      });
    };
    if (first && last) pass(std::true_type{}, std::true_type{});
    else if (first) pass(std::true_type{}, std::false_type{});
    else if (last) pass(std::false_type{}, std::true_type{});
    else pass(std::false_type{}, std::false_type{});
    if (last) break;
    frame_sweeps(A, T, L, Dc, lane, row, row + 1);
  }
}

// UB[s][t3][k][c]: column c of U(t3) for c < N, M_x(t3) for c = N + x; one
// wave per sample (N + 3 <= 64 columns).
__global__ void __launch_bounds__(64) singles_basis_kernel(BasisArgs A) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int s = blockIdx.x, c = threadIdx.x, lane = c, N = A.N, T3 = A.T3, NC = N + 3;
  const SinglesLds L = singles_lds(smem, N);
  const int64_t tj = tj_of(A, s), row0 = tj - A.f_lo;
  const int lc = min(lane, N - 1);
  for (int k = 0; k <= N; ++k) {
    float v = c == k && k < N ? 1.f : 0.f;
    if (c >= N && c < NC && k < N) v = gld(mu_of(A, tj, c - N) + k);
    L.psi[k * 64 + lane] = make_float2(v, 0.f);
  }
  Segment T = load_segment(A, lane, row0, 0);
  float2 dn = gld(A.diag + row0 * N + lc);
  for (int t3 = 0; t3 < T3; ++t3) {
    const int64_t row = row0 + t3;
    const bool last = t3 == T3 - 1;
    float2 *Dc = L.D + (t3 & 1) * 64;
    const float2 *Dp = L.D + ((t3 + 1) & 1) * 64;
    Dc[lane] = dn;
    if (!last) dn = gld(A.diag + (row + 1) * N + lc);
    float2 *out = A.UB + ((int64_t)s * T3 + t3) * N * NC + c;
    auto pass = [&](auto fst) {
      site_batches<decltype(fst)::value, false>(L, Dp, Dc, lane, N, [&](int k, float2 p) {
        if (c < NC && k < N) gst(out + (int64_t)k * NC, p);
        return p;
      });
    };
    if (t3 == 0) pass(std::true_type{});
    else pass(std::false_type{});
    if (last) break;
    frame_sweeps(A, T, L, Dc, lane, row, min(row + 1, row0 + T3 - 1));
  }
}

// ---------------------------------------------------------------------------
// Two-exciton basis vectors in LDS for every t3 (the rotation table and step
// rows of persist_dev.h).  A wave holds VW = 64 / NP vectors of one kind:
//   kind x2 = 0, 1, 2: mu+_x2 e_i, i = i0 .. i0 + nv - 1; per t3 it forms
//     W[x1 x2 x3][i] for all x1, x3;
//   kind 3: mu+_x2 mu_x1(tj) for the pairs v = x1 x2 = i0 .. ; per t3 it
//     stores mu-_x3 of each.
// Lane (k, c) = (lane / VW, lane % VW) contracts row k of vector c with the
// dipoles of frame tj + t3 (broadcast reads of the staged rows).
// ---------------------------------------------------------------------------
constexpr int kPre = 4;
struct BasisLayout {
  size_t ix, d2, cs, mu, psi, total;
};
__host__ __device__ inline BasisLayout basis_layout(int N, int VW, int K2, int npw) {
  const size_t N2 = (size_t)N * (N + 1) / 2;
  BasisLayout L;
  size_t o = 0;
  L.ix = o, o += rot_table_bytes(N, 64 / VW, K2);
  L.d2 = o, o += N2 * 8, o = (o + 15) & ~(size_t)15;
  L.cs = o, o += (size_t)K2 * 48;
  L.mu = o, o += (size_t)N * 16;
  L.psi = o, o += (size_t)npw * (N2 + 2) * VW * 8;
  L.total = o;
  return L;
}
// Waves per sample: N / VW per x2, and the nine vectors of kind 3.
__host__ __device__ inline int basis_waves(int N, int VW) { return 3 * ((N + VW - 1) / VW) + (9 + VW - 1) / VW; }

// rot_entry (persist_dev.h) with fused products.
__device__ __forceinline__ void rot_entry_fma(char *base, const char *cs, uint2 e) {
  float2 *a1 = reinterpret_cast<float2 *>(base + (e.x & 0xffffu));
  float2 *a2 = reinterpret_cast<float2 *>(base + (e.x >> 16));
  const float2 q = *reinterpret_cast<const float2 *>(base + (e.y & 0xffffu));
  const float4 cf = *reinterpret_cast<const float4 *>(cs + (e.y >> 16));
  float2 p1 = *a1, p2 = *a2;
  p1 = make_float2(fmaf(-cf.y, q.y, cf.x * p1.x), fmaf(cf.y, q.x, cf.x * p1.y));
  rot_fma(p1, p2, cf.z, cf.w);
  *a2 = p2;
  *a1 = p1;
}
template <int NP>
__device__ __forceinline__ void rot_sweep(float2 *psi, int total, const uint2 *ix, const float4 *csL, int q, int c0) {
  if (total == 0) return;
  char *base = reinterpret_cast<char *>(psi) + q * 8;
  const char *cs = reinterpret_cast<const char *>(csL);
  const uint2 *e = ix + c0;
  uint2 e0 = e[0];
  int j = 0;
  for (; j + 1 < total; j += 2) {  // entries read one rotation ahead
    const uint2 e1 = e[(j + 1) * NP];
    rot_entry_fma(base, cs, e0);
    e0 = e[(j + 2) * NP];
    rot_entry_fma(base, cs, e1);
  }
  if (j < total) rot_entry_fma(base, cs, e0);
  asm volatile("" ::: "memory");
}
template <int VW>
__device__ __forceinline__ void phase_pass(float2 *psi, const float2 *d2, int N2, int lane) {
  if constexpr (VW == 1) {
    for (int j = lane; j < N2; j += 64) psi[j] = cmul_f(psi[j], d2[j]);
  } else {
    float4 *p4 = reinterpret_cast<float4 *>(psi);
    for (int j = lane; j < N2 * (VW / 2); j += 64) {
      const float2 d = d2[j / (VW / 2)];
      const float4 v = p4[j];
      const float2 lo = cmul_f(make_float2(v.x, v.y), d), hi = cmul_f(make_float2(v.z, v.w), d);
      p4[j] = make_float4(lo.x, lo.y, hi.x, hi.y);
    }
  }
  asm volatile("" ::: "memory");
}

template <int NP>
__global__ void __launch_bounds__(256) dbl_basis_kernel(BasisArgs A, int npw, int nwg_s) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int VW = 64 / NP;
  const int N = A.N, N2 = N * (N + 1) / 2, K2 = A.K2, T3 = A.T3, t = threadIdx.x;
  const int wave = t >> 6, lane = t & 63;
  const BasisLayout Ly = basis_layout(N, VW, K2, npw);
  uint2 *ixL = reinterpret_cast<uint2 *>(smem + Ly.ix);
  float2 *d2 = reinterpret_cast<float2 *>(smem + Ly.d2);
  float4 *csL = reinterpret_cast<float4 *>(smem + Ly.cs);
  float4 *muL = reinterpret_cast<float4 *>(smem + Ly.mu);  // [N] mu_0..2(tl)
  float2 *psi = reinterpret_cast<float2 *>(smem + Ly.psi) + (size_t)wave * (N2 + 2) * VW;
  const int nt = blockDim.x;
  // this wave's vectors
  const int s = blockIdx.x / nwg_s, w = (blockIdx.x % nwg_s) * npw + wave, nbw = (N + VW - 1) / VW;
  const int kind = __builtin_amdgcn_readfirstlane(min(w / nbw, 3));
  const int i0 = (w - kind * nbw) * VW;
  const int nv = __builtin_amdgcn_readfirstlane(max(0, min(VW, (kind < 3 ? N : 9) - i0)));
  const int64_t tj = tj_of(A, s);
  // mu+ (src/NISE_subs.c:485-509): |aa> gets over_a c_a, |ab> mu_a c_b + mu_b c_a
  for (int j = lane; j < N2; j += 64) {
    int a = 0, rem = j;
    while (rem >= N - a) { rem -= N - a; ++a; }
    const int b = a + rem;
    for (int q = 0; q < VW; ++q) {
      float v = 0.f;
      if (q < nv) {
        const int x2 = kind < 3 ? kind : (i0 + q) % 3;
        const float *dip = mu_of(A, tj, x2), *cv = mu_of(A, tj, kind < 3 ? 0 : (i0 + q) / 3);
        const float ca = kind < 3 ? (a == i0 + q ? 1.f : 0.f) : cv[a], cb = kind < 3 ? (b == i0 + q ? 1.f : 0.f) : cv[b];
        if (a == b) {
          const float ov = A.es ? 0.f
                           : A.anh != 0.f ? __fmul_rn(kSqrt2, dip[a])
                                          : A.over_rec[tj * (1 + 3 * (int64_t)N) + 1 + (int64_t)x2 * N + a];
          v = A.es ? 0.f : __fmul_rn(ov, ca);
        } else {
          v = __fadd_rn(__fmul_rn(dip[a], cb), __fmul_rn(dip[b], ca));
        }
      }
      psi[j * VW + q] = make_float2(v, 0.f);
    }
  }
  init_special_states<VW>(psi, N2, lane);
  build_rot_table<NP>(ixL, A.ab2, N, K2, A.es != 0);
  const int q = lane % VW, k = lane / VW, nkb = (N + NP - 1) / NP;
  auto mu_row = [&](int64_t f) {
    const float *m = mu_of(A, f, 0);
    return t < N ? make_float4(gld(m + t), gld(m + N + t), gld(m + 2 * N + t), 0.f) : make_float4(0.f, 0.f, 0.f, 0.f);
  };
  {
    const float4 m = mu_row(tj);  // (N <= 61 < threads)
    if (t < N) muL[t] = m;
  }
  __syncthreads();
  for (int t3 = 0; t3 < T3; ++t3) {
    const int64_t tl = tj + t3, row = tl - A.f_lo;
    const bool last = t3 + 1 == T3;
    // the step's rows and the next frame's dipoles, in flight during the
    // contraction (the first kPre entries of a thread; longer rows load the
    // rest in place)
    float2 pd[kPre];
    float4 pc, pm;
    if (!last) {
#pragma unroll
      for (int u = 0; u < kPre; ++u)
        if (t + u * nt < N2) pd[u] = gld(A.D2 + row * N2 + t + u * nt);
      if (t < K2) pc = gld(A.cs2 + row * K2 + t);
      pm = mu_row(tl + 1);
    }
    if (nv > 0) {
      // W sums over the row blocks of N > 64 lanes' worth of sites
      float2 acc[9];
#pragma unroll
      for (int j = 0; j < 9; ++j) acc[j] = make_float2(0.f, 0.f);
      for (int kb = 0; kb < nkb; ++kb) {
        const int kk = kb * NP + k, kc = min(kk, N - 1);
        // row kc of the vector: elements (i, kc) at kc + rs(i) for i <= kc,
        // rs(kc) + i above; all with the dipole weight, then the diagonal
        // corrected to the overtone dipole (src/NISE_subs.c:552-575)
        float mk[3], ov[3];
        float2 M[3];
        const int64_t ob = tl * (1 + 3 * (int64_t)N) + 1;
#pragma unroll
        for (int x = 0; x < 3; ++x) {
          mk[x] = gld(mu_of(A, tl, x) + kc);
          ov[x] = A.es ? 0.f : A.anh != 0.f ? __fmul_rn(kSqrt2, mk[x]) : gld(A.over_rec + ob + (int64_t)x * N + kc);
          M[x] = gld(A.UB + (((int64_t)s * T3 + t3) * N + kc) * (N + 3) + N + x);
        }
        const char *fb = reinterpret_cast<const char *>(psi + q);
        int o = kc * VW * 8;
        float2 r[3];
#pragma unroll
        for (int x = 0; x < 3; ++x) r[x] = make_float2(0.f, 0.f);
#pragma unroll 4
        for (int i = 0; i < N; ++i) {
          const float2 f = *reinterpret_cast<const float2 *>(fb + o);
          const float4 m = muL[i];
          r[0].x = fmaf(m.x, f.x, r[0].x), r[0].y = fmaf(m.x, f.y, r[0].y);
          r[1].x = fmaf(m.y, f.x, r[1].x), r[1].y = fmaf(m.y, f.y, r[1].y);
          r[2].x = fmaf(m.z, f.x, r[2].x), r[2].y = fmaf(m.z, f.y, r[2].y);
          o += i < kc ? (N - i - 1) * VW * 8 : VW * 8;
        }
        const float2 fd = psi[(((kc * (2 * N - kc - 1)) >> 1) + kc) * VW + q];
#pragma unroll
        for (int x = 0; x < 3; ++x) {
          const float d = __fsub_rn(ov[x], mk[x]);
          r[x].x = fmaf(d, fd.x, r[x].x), r[x].y = fmaf(d, fd.y, r[x].y);
        }
        if (kind == 3) {
          if (q < nv && kk < N) {
            float2 *out = A.Lr + (((int64_t)s * T3 + t3) * 27 + (i0 + q) * 3) * N + kk;
            gst(out, r[0]), gst(out + N, r[1]), gst(out + 2 * N, r[2]);
          }
        } else {
          if (kk >= N) M[0] = M[1] = M[2] = make_float2(0.f, 0.f);
#pragma unroll
          for (int x1 = 0; x1 < 3; ++x1)
#pragma unroll
            for (int x3 = 0; x3 < 3; ++x3) {  // conj(M_x1) r_x3
              float2 &z = acc[x1 * 3 + x3];
              z.x = fmaf(M[x1].x, r[x3].x, fmaf(M[x1].y, r[x3].y, z.x));
              z.y = fmaf(M[x1].x, r[x3].y, fmaf(-M[x1].y, r[x3].x, z.y));
            }
        }
      }
      if (kind < 3) {
#pragma unroll
        for (int j = 0; j < 9; ++j) {
          const float2 z = make_float2(stride_sum<VW>(acc[j].x), stride_sum<VW>(acc[j].y));
          if (k == 0 && q < nv)
            gst(A.W + (((int64_t)s * T3 + t3) * 27 + ((j / 3) * 3 + kind) * 3 + j % 3) * N + i0 + q, z);
        }
      }
    }
    if (last) break;  // the state after the last t3 is not used
    __syncthreads();  // the previous step has read d2 and cs, this contraction muL
#pragma unroll
    for (int u = 0; u < kPre; ++u)
      if (t + u * nt < N2) d2[t + u * nt] = pd[u];
    for (int e = t + kPre * nt; e < N2; e += nt) d2[e] = gld(A.D2 + row * N2 + e);
    for (int e = t; e < K2; e += nt) {
      const float4 c = e == t ? pc : gld(A.cs2 + row * K2 + e);
      csL[3 * e] = make_float4(1.f, 0.f, c.x, c.y);
      csL[3 * e + 1] = make_float4(1.f, 0.f, c.z, c.w);
      csL[3 * e + 2] = make_float4(c.z, c.w, c.z, c.w);
    }
    if (t < N) muL[t] = pm;
    __syncthreads();
    for (int sub = 0; sub < (nv > 0 ? A.m : 0); ++sub) {
      phase_pass<VW>(psi, d2, N2, lane);
      rot_sweep<NP>(psi, K2 * nkb, ixL, csL, q, k);
      phase_pass<VW>(psi, d2, N2, lane);
    }
  }
}

// ---------------------------------------------------------------------------
// V[s][t3][x0][i][6]: kI and kII vectors of the file comment, summed over the
// items of x0 with the three lab weights in FP64.  One workgroup per (s, t3).
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) combine_kernel(BasisArgs A) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int s = blockIdx.x, t3 = blockIdx.y, N = A.N, NC = N + 3, t = threadIdx.x;
  float2 *U = reinterpret_cast<float2 *>(smem);  // [N][NC]
  float2 *q = U + (size_t)N * NC;                // [3][NC] mu_x3(tl) . columns
  float2 *lr = q + 3 * NC;                       // [27][N]
  float *mj = reinterpret_cast<float *>(lr + 27 * N);  // [3][N] mu(tj)
  float *ml = mj + 3 * N;                              // [3][N] mu(tl)
  float *g = ml + 3 * N;                               // [9] mu_a(tj) . mu_b(tj)
  float *wl = g + 9;                                   // [3][21]
  const int64_t tj = tj_of(A, s), tl = tj + t3, st = (int64_t)s * A.T3 + t3;
  stage_lds<4>(U, A.UB + st * N * NC, N * NC);
  if (A.do_ea) stage_lds<4>(lr, A.Lr + st * 27 * N, 27 * N);
  for (int e = t; e < 3 * N; e += 256) mj[e] = gld(mu_of(A, tj, 0) + e), ml[e] = gld(mu_of(A, tl, 0) + e);
  for (int e = t; e < 63; e += 256) wl[e] = gld(A.wpl + e);
  __syncthreads();
  for (int e = t; e < 3 * NC; e += 256) {
    const int x = e / NC, c = e % NC;
    float2 z = make_float2(0.f, 0.f);
    for (int k = 0; k < N; ++k) {
      const float2 u = U[k * NC + c];
      z.x = fmaf(ml[x * N + k], u.x, z.x), z.y = fmaf(ml[x * N + k], u.y, z.y);
    }
    q[e] = z;
  }
  if (t >= 192 && t < 201) {
    const int a = (t - 192) / 3, b = (t - 192) % 3;
    float z = 0.f;
    for (int k = 0; k < N; ++k) z = fmaf(mj[a * N + k], mj[b * N + k], z);
    g[t - 192] = z;
  }
  __syncthreads();
  // thread (x0, i): the items of x0 in turn
  for (int e = t; e < 3 * N; e += 256) {
    const int x0 = e / N, i = e % N;
    double2 v[6];
#pragma unroll
    for (int j = 0; j < 6; ++j) v[j] = make_double2(0.0, 0.0);
    // EA kI: U^+ l for the seven items at once (every column entry read once)
    float2 y[7];
#pragma unroll
    for (int j = 0; j < 7; ++j) y[j] = make_float2(0.f, 0.f);
    int lo[7], n = 0;
    for (int m = 0; m < 21; ++m)
      if (c_polar[m][0] == x0) {
        const int o = ((c_polar[m][1] * 3 + c_polar[m][2]) * 3 + c_polar[m][3]) * N;
#pragma unroll
        for (int j = 0; j < 7; ++j)
          if (j == n) lo[j] = o;
        ++n;
      }
    if (A.do_ea)
      for (int k = 0; k < N; ++k) {
        const float2 u = U[k * NC + i];
#pragma unroll
        for (int j = 0; j < 7; ++j) {
          const float2 l = lr[lo[j] + k];
          y[j].x = fmaf(u.x, l.x, fmaf(u.y, l.y, y[j].x));
          y[j].y = fmaf(u.x, l.y, fmaf(-u.y, l.x, y[j].y));
        }
      }
    n = 0;
    for (int m = 0; m < 21; ++m) {
      if (c_polar[m][0] != x0) continue;
      const int x1 = c_polar[m][1], x2 = c_polar[m][2], x3 = c_polar[m][3];
      double ar = 0.0, ai = 0.0, br = 0.0, bi = 0.0;
      if (A.do_gb) {  // src/calc_2DIR.c:272-275
        const float2 z = q[x3 * NC + N + x2];
        const double d = (double)mj[x1 * N + i];
        ar -= d * z.x, ai -= d * z.y, br -= d * z.x, bi -= d * z.y;
      }
      if (A.do_se) {  // :397-400
        const float2 z = q[x3 * NC + N + x1], r = q[x3 * NC + i];
        const double d = (double)mj[x2 * N + i], gg = (double)g[x1 * 3 + x2];
        ar -= d * z.x, ai -= d * z.y;
        br -= gg * r.x, bi -= gg * r.y;
      }
      if (A.do_ea) {  // :465-469
        float2 yy = y[0];
#pragma unroll
        for (int j = 1; j < 7; ++j)
          if (j == n) yy = y[j];
        const float2 ww = gld(A.W + (st * 27 + (x1 * 3 + x2) * 3 + x3) * N + i);
        ar += yy.x, ai += yy.y, br += ww.x, bi += ww.y;
      }
      ++n;
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        const double w = (double)wl[p * 21 + m];
        v[p].x += w * ar, v[p].y += w * ai, v[3 + p].x += w * br, v[3 + p].y += w * bi;
      }
    }
    double2 *out = A.V + ((st * 3 + x0) * N + i) * 6;
#pragma unroll
    for (int j = 0; j < 6; ++j) gst(out + j, v[j]);
  }
}

// part[chunk][12][t3][t1]: sum over the chunk's samples, x0 and i of
// conj(L0) V (kI) and L0 V (kII); one wave per (t3, 64 values of t1, chunk),
// one t1 per lane, V wave-uniform (scalar loads).
__global__ void __launch_bounds__(64) contract_kernel(BasisArgs A, int per, double *part) {
  const int t3 = blockIdx.x, lane = threadIdx.x, N = A.N, T1 = A.T1, T3 = A.T3;
  const int t1 = blockIdx.y * 64 + lane, tc = min(t1, T1 - 1), ch = blockIdx.z;
  double2 z[6];
#pragma unroll
  for (int j = 0; j < 6; ++j) z[j] = make_double2(0.0, 0.0);
  const int s1 = min(A.S, (ch + 1) * per);
  for (int s = ch * per; s < s1; ++s) {
    const double2 *v = A.V + ((int64_t)s * T3 + t3) * 18 * N;
    const float2 *l0 = A.L0 + (int64_t)s * 3 * N * T1 + tc;
#pragma unroll 4
    for (int e = 0; e < 3 * N; ++e) {
      const float2 lf = gld(l0 + (int64_t)e * T1);
      const double lx = lf.x, ly = lf.y;
#pragma unroll
      for (int j = 0; j < 3; ++j) {  // conj(L0) V
        const double2 a = cld(v + e * 6 + j);
        z[j].x = fma(a.x, lx, z[j].x), z[j].y = fma(a.y, lx, z[j].y);
        z[j].x = fma(a.y, ly, z[j].x), z[j].y = fma(-a.x, ly, z[j].y);
      }
#pragma unroll
      for (int j = 3; j < 6; ++j) {  // L0 V
        const double2 a = cld(v + e * 6 + j);
        z[j].x = fma(a.x, lx, z[j].x), z[j].y = fma(a.y, lx, z[j].y);
        z[j].x = fma(-a.y, ly, z[j].x), z[j].y = fma(a.x, ly, z[j].y);
      }
    }
  }
  if (t1 >= T1) return;
  // plane 4 p + {0, 1}: Im, Re of kI; 4 p + {2, 3}: of kII
  const int64_t plane = (int64_t)T3 * T1;
  double *o = part + (int64_t)ch * 12 * plane + (int64_t)t3 * T1 + t1;
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    o[(4 * p) * plane] = z[p].y, o[(4 * p + 1) * plane] = z[p].x;
    o[(4 * p + 2) * plane] = z[3 + p].y, o[(4 * p + 3) * plane] = z[3 + p].x;
  }
}

// R += lt(t3, t1) * (chunks in ascending order)
__global__ void finish_kernel(const double *part, int nc, int64_t plane, const float *lt, double *R) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= 12 * plane) return;
  double a = 0.0;
  for (int c = 0; c < nc; ++c) a += part[(int64_t)c * 12 * plane + e];
  R[e] += a * (double)lt[e % plane];
}

// ---------------------------------------------------------------------------
// Host side.
// ---------------------------------------------------------------------------
static int basis_npw(int N, int VW, int K2) {
  // as the per-vector kernel: the most resident waves per CU, at most 4
  int npw = 0;
  double best = 0;
  const int nw = basis_waves(N, VW);
  for (int w = 1; w <= 4; ++w) {
    const size_t L = basis_layout(N, VW, K2, w).total;
    if (L > 160 * 1024) break;
    const double score = (double)(160 * 1024 / L) * w * nw / (double)((nw + w - 1) / w * w);
    if (score > best * 1.0001) best = score, npw = w;
  }
  return npw;
}

// Taken where it propagates fewer vectors: 3 N + 9 two-exciton vectors
// against 9 T1 + 9 (and N + 3 one-exciton against 3 T1 + 3), with the
// two-exciton rotation table in LDS; N <= 61 keeps a sample's one-exciton
// columns in one wave.  Near the line it is still the faster one (N = 45, T1 =
// T3 = 16, 50 samples: 1.45 against 1.81 ms; N = 60, T1 = T3 = 24, 40 samples:
// 4.3 against 5.8).  Windows below 16 steps keep every vector's own
// propagation: they take a few hundred microseconds either way, and follow
// the reference's FP32 values of each vector bit for bit.
bool basis_path(const t_non *non, int K2, bool do_ea) {
  const int N = non->singles;
  if (non->propagation != 1 || non->tmax2 != 0 || N > 61 || non->tmax1 < 16 || N + 3 > 3 * non->tmax1) return false;
  const int VW = 64 / doubles_np(N);
  return !do_ea || (rot_table_fits(N, VW, K2) && basis_npw(N, VW, K2) > 0);
}

namespace {
struct BasisBufs {
  DevBuf par, diag, cs, L0, UB, W, Lr, V, part, D2, cs2, Rd;
};
}  // namespace

int run_basis(const BasisCall &c, float *R12) {
  static thread_local BasisBufs B;
  const t_non *non = c.non;
  const int N = non->singles, T1 = non->tmax1, T3 = non->tmax3, N2 = N * (N + 1) / 2;
  const int K2 = (int)c.lex.size(), total = c.end - non->begin;
  const int64_t nfr = c.f_hi - c.f_lo, plane = (int64_t)T3 * T1;
  hipStream_t st = c.st;
  int rc;
  // parameters in one upload: weights, lifetime factors, rotation program, couplings
  Schedule sch;
  build_schedule(N, c.mask, sch);
  std::vector<uint32_t> prog, pairs;
  sweep_program(sch, prog, pairs);
  std::vector<uint32_t> par(64 + plane + 2 * prog.size() + K2);
  float *wh = reinterpret_cast<float *>(par.data()), *lth = wh + 64;
  for (int p = 0; p < 3; ++p)
    for (int m = 0; m < 21; ++m) wh[p * 21 + m] = polarweight_h(p, m);
  for (int t3 = 0; t3 < T3; ++t3)
    for (int t1 = 0; t1 < T1; ++t1)
      lth[(size_t)t3 * T1 + t1] =
          (non->lifetime > 0) ? (float)exp(-(double)(t1 + t3) * non->deltat / (2 * non->lifetime)) : 1.0f;
  if (!prog.empty()) std::memcpy(par.data() + 64 + plane, prog.data(), prog.size() * 4);
  if (!pairs.empty()) std::memcpy(par.data() + 64 + plane + prog.size(), pairs.data(), pairs.size() * 4);
  if (K2) std::memcpy(par.data() + 64 + plane + 2 * prog.size(), c.lex.data(), (size_t)K2 * 4);
  if ((rc = B.par.alloc(par.size() * 4))) return rc;
  NISE_HIP_CHECK(hipMemcpy(B.par.p, par.data(), par.size() * 4, hipMemcpyHostToDevice));
  BasisArgs A;
  std::memset(&A, 0, sizeof(A));
  A.N = N, A.T1 = T1, A.T3 = T3, A.sample = non->sample, A.m = non->ts;
  A.do_gb = c.do_gb, A.do_se = c.do_se, A.do_ea = c.do_ea, A.es = c.es, A.anh = non->anharmonicity;
  A.f_lo = c.f_lo, A.mu_rec = c.mu_rec, A.mu_stride = c.mu_stride, A.over_rec = c.over_rec;
  A.wpl = B.par.as<float>();
  const float *lt = A.wpl + 64;
  A.prog = B.par.as<uint32_t>() + 64 + plane, A.Kp = (int)prog.size();
  A.ab2 = A.prog + 2 * prog.size(), A.K2 = K2;
  const float fac = trotter_factor(non->deltat, 1, non->ts);
  sch.K = A.Kp;  // the tables in the program's order, padding as dummy pairs
  if ((rc = B.diag.alloc((size_t)nfr * N * 8)) || (rc = B.cs.alloc((size_t)nfr * std::max(A.Kp, 1) * 8))) return rc;
  if ((rc = launch_frame_tables(c.src, N, sch, A.prog + prog.size(), fac, c.f_lo, nfr, B.diag.as<float2>(), B.cs.as<float2>(), st)))
    return rc;
  A.diag = B.diag.as<float2>(), A.cs = B.cs.as<float2>();
  const int np = doubles_np(N), VW = 64 / np;
  if (c.do_ea) {
    if ((rc = B.D2.alloc((size_t)nfr * N2 * 8)) || (rc = B.cs2.alloc((size_t)nfr * std::max(K2, 1) * 16))) return rc;
    if ((rc = launch_doubles_tables(c.src, N, K2, A.ab2, fac, c.es ? 0.f : non->anharmonicity, c.es ? nullptr : c.anh_rec,
                                    c.f_lo, nfr, B.D2.as<float2>(), B.cs2.as<float4>(), st)))
      return rc;
    A.D2 = B.D2.as<float2>(), A.cs2 = B.cs2.as<float4>();
  }
  if ((rc = B.Rd.alloc((size_t)12 * plane * 8))) return rc;
  NISE_HIP_CHECK(hipMemsetAsync(B.Rd.p, 0, (size_t)12 * plane * 8, st));
  const double per_sample = 24.0 * T1 * N + 8.0 * T3 * N * (N + 3) + (c.do_ea ? 432.0 * T3 * N : 0.0) + 288.0 * T3 * N;
  const int chunk = (int)std::max(1.0, std::min<double>({(double)total, 65535.0, 8.0e9 / per_sample}));
  const size_t ssm = singles_smem(N);
  for (int c0 = 0; c0 < total; c0 += chunk) {
    const int S = std::min(chunk, total - c0);
    A.S = S, A.s0 = non->begin + c0;
    // samples per contraction wave: about 4,096 waves in all
    const int nt = (T1 + 63) / 64, per = std::max(1, (int)((int64_t)S * T3 * nt / 4096));
    const int nc = (S + per - 1) / per;
    if ((rc = B.L0.alloc((size_t)S * 3 * N * T1 * 8)) || (rc = B.UB.alloc((size_t)S * T3 * N * (N + 3) * 8)) ||
        (rc = B.V.alloc((size_t)S * T3 * 18 * N * 16)) || (rc = B.part.alloc((size_t)nc * 12 * plane * 8)))
      return rc;
    if (c.do_ea && ((rc = B.W.alloc((size_t)S * T3 * 27 * N * 8)) || (rc = B.Lr.alloc((size_t)S * T3 * 27 * N * 8))))
      return rc;
    A.L0 = B.L0.as<float2>(), A.UB = B.UB.as<float2>(), A.V = B.V.as<double2>();
    A.W = B.W.as<float2>(), A.Lr = B.Lr.as<float2>();
    hipLaunchKernelGGL(singles_seeds_kernel, dim3(S, 3, nt), dim3(64), ssm, st, A);
    NISE_HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(singles_basis_kernel, dim3(S), dim3(64), ssm, st, A);
    NISE_HIP_CHECK(hipGetLastError());
    if (c.do_ea) {
      int npw = basis_npw(N, VW, K2), nwg_s = (basis_waves(N, VW) + npw - 1) / npw;
      const size_t psm = basis_layout(N, VW, K2, npw).total;
      const void *fn = np == 8 ? (const void *)dbl_basis_kernel<8>
                     : np == 16 ? (const void *)dbl_basis_kernel<16>
                     : np == 32 ? (const void *)dbl_basis_kernel<32> : (const void *)dbl_basis_kernel<64>;
      NISE_HIP_CHECK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)psm));
      void *kargs[] = {&A, &npw, &nwg_s};
      NISE_HIP_CHECK(hipLaunchKernel(fn, dim3((unsigned)(S * nwg_s)), dim3(64 * npw), kargs, psm, st));
    }
    const size_t csm = (size_t)N * (N + 3) * 8 + (size_t)3 * (N + 3) * 8 + (size_t)27 * N * 8 + (size_t)6 * N * 4 + 72 * 4;
    NISE_HIP_CHECK(hipFuncSetAttribute((const void *)combine_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)csm));
    hipLaunchKernelGGL(combine_kernel, dim3(S, T3), dim3(256), csm, st, A);
    NISE_HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(contract_kernel, dim3(T3, nt, nc), dim3(64), 0, st, A, per, B.part.as<double>());
    NISE_HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(finish_kernel, dim3((unsigned)((12 * plane + 255) / 256)), dim3(256), 0, st, B.part.as<double>(), nc,
                       plane, lt, B.Rd.as<double>());
    NISE_HIP_CHECK(hipGetLastError());
  }
  std::vector<double> h((size_t)12 * plane);
  NISE_HIP_CHECK(hipMemcpyAsync(h.data(), B.Rd.p, h.size() * 8, hipMemcpyDeviceToHost, st));
  NISE_HIP_CHECK(hipStreamSynchronize(st));
  for (size_t i = 0; i < h.size(); ++i) R12[i] = (float)h[i];
  return NISE_OK;
}

}  // namespace nise
