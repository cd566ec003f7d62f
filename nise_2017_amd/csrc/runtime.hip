// Host runtime of libnise_hip: error state, device buffers, the layered
// rotation schedule, device and stream setup.
#include <algorithm>
#include <cstdarg>
#include <cstdlib>
#include <cstring>
#include <mutex>

#include "nise_internal.h"

namespace nise {

static thread_local char g_err[1024] = "";

void set_error(const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
}

const char *get_error() { return g_err; }

int DevBuf::alloc(size_t n) {
  if (n <= bytes && p) return NISE_OK;
  release();
  if (n == 0) return NISE_OK;
  hipError_t e = hipMalloc(&p, n);
  if (e != hipSuccess) {
    p = nullptr;
    (void)hipGetLastError();  // or the next launch check, of a run that did without, would report it
    set_error("hipMalloc(%zu) failed: %s", n, hipGetErrorString(e));
    return NISE_ERR_NOMEM;
  }
  bytes = n;
  return NISE_OK;
}

void DevBuf::release() {
  if (p) (void)hipFree(p);
  p = nullptr;
  bytes = 0;
}

// ASAP layering of the lexicographic rotation sequence: rotation k goes to
// layer 1 + max(last layer touching a_k, last layer touching b_k).  Every
// site therefore sees its rotations in the original order, and rotations of
// one layer share no site.
void build_schedule(int N, const std::vector<uint8_t> &mask, Schedule &s) {
  s.N = N;
  s.ab.clear();
  std::vector<int> la, lb, lay;
  std::vector<int> last(N, -1);
  int nl = 0;
  int64_t p = 0;
  for (int a = 0; a < N; ++a)
    for (int b = a + 1; b < N; ++b, ++p) {
      if (!mask[p]) continue;
      int l = 1 + (last[a] > last[b] ? last[a] : last[b]);
      last[a] = last[b] = l;
      la.push_back(a), lb.push_back(b), lay.push_back(l);
      if (l + 1 > nl) nl = l + 1;
    }
  s.K = s.Kreal = (int)la.size();
  s.layer_off.assign(nl + 1, 0);
  for (int l : lay) s.layer_off[l + 1]++;
  for (int l = 0; l < nl; ++l) s.layer_off[l + 1] += s.layer_off[l];
  std::vector<int> fill(s.layer_off.begin(), s.layer_off.end() - 1);
  s.ab.assign(s.K, 0);
  for (int k = 0; k < s.K; ++k)  // stable within a layer
    s.ab[fill[lay[k]]++] = (uint32_t)la[k] | ((uint32_t)lb[k] << 16);
}

// LDS bank cost of a layer's row order: a row's G vectors occupy 2G consecutive
// dwords, so in B banks its run falls in block slot mod (B / 2G); per group
// of lanes the busiest block bounds the passes of an access.  The grouping
// the hardware uses for 8-byte accesses is not pinned here, so the cost is
// summed over 32-lane groups on 64 banks and 16-lane groups on 32 banks
// (a grouping of all 64 lanes does not depend on the row order).
struct BankModel {
  int nblk = 0, rpg = 0;  // blocks, rows per lane group
};

// Rotations of one layer touch disjoint sites, so their order across the R
// rows is free.  Each of the layer's n rotations goes to the lane group (of
// the finer model; a coarser group holds whole finer ones) where it raises the
// busiest blocks least, ties to the emptiest group; then one pass of swaps
// between groups lowers the cost, only of entries in a busiest block and with
// each swap's gain read from the block counts.  (Four passes over all pairs,
// each swap evaluated over its groups' rows, took 90% of a schedule's time for
// a cost 1% lower: N = 256 lattice, R = 16, 22 ms against 5 and cost 5,795
// against 5,855; N = 384, R = 32, 94 ms against 13 and 4,663 against 4,675.)
struct LayerBanks {
  int nm = 0, fine = 1, R = 1;
  BankModel bm[2];
  uint8_t cnt[2][2][64][64];  // [model][side][group][block] entries
  uint8_t hist[2][2][64][66]; // [..][count] blocks that hold so many
  uint8_t top[2][2][64];      // the busiest block's count
  int group(int k, int row) const { return row / bm[k].rpg; }
  int block(int k, int d, uint32_t e) const { return (int)(d ? e >> 16 : e & 0xffffu) & (bm[k].nblk - 1); }
  void init(int R_) {
    R = R_, nm = 0;
    const int G = 64 / R;
    for (const auto &m : {std::make_pair(64, 32), std::make_pair(32, 16)}) {
      const int span = 2 * G, rpg = std::max(1, m.second / G);
      if (span <= m.first && rpg < R) bm[nm].nblk = m.first / span, bm[nm++].rpg = rpg;
    }
    if (nm) fine = bm[nm - 1].rpg;
  }
  void clear() {
    for (int k = 0; k < nm; ++k)
      for (int d = 0; d < 2; ++d)
        for (int g = 0; g < R / bm[k].rpg; ++g) {
          std::memset(cnt[k][d][g], 0, bm[k].nblk);
          std::memset(hist[k][d][g], 0, sizeof(hist[k][d][g]));
          hist[k][d][g][0] = (uint8_t)bm[k].nblk, top[k][d][g] = 0;
        }
  }
  void add(int row, uint32_t e, int by) {
    for (int k = 0; k < nm; ++k)
      for (int d = 0; d < 2; ++d) {
        const int g = group(k, row);
        uint8_t &c = cnt[k][d][g][block(k, d, e)], *h = hist[k][d][g];
        --h[c], c = (uint8_t)(c + by), ++h[c];
        uint8_t &t = top[k][d][g];
        if (c > t) t = c;
        while (t && !h[t]) --t;
      }
  }
  // the group's top with entry `out` replaced by `in` (~0u: none)
  int top_after(int k, int d, int g, uint32_t out, uint32_t in) const {
    int t = top[k][d][g];
    const uint8_t *c = cnt[k][d][g];
    const int bo = out == ~0u ? -1 : block(k, d, out), bi = in == ~0u ? -1 : block(k, d, in);
    if (bo == bi) return t;
    if (bo >= 0 && c[bo] == t && hist[k][d][g][t] == 1) --t;
    return bi >= 0 ? std::max(t, c[bi] + 1) : t;
  }
  bool hot(int row, uint32_t e) const {
    for (int k = 0; k < nm; ++k)
      for (int d = 0; d < 2; ++d) {
        const int g = group(k, row), t = top[k][d][g];
        if (t > 1 && cnt[k][d][g][block(k, d, e)] == t) return true;
      }
    return false;
  }
};
static void assign_rows(LayerBanks &B, std::vector<uint32_t> &e, int n) {
  if (!B.nm) return;
  const int R = B.R, ng = R / B.fine;
  int used[64] = {};
  uint32_t out[64];
  for (int q = 0; q < R; ++q) out[q] = ~0u;
  B.clear();
  for (int i = 0; i < n; ++i) {
    int best = -1, bc = 0;
    for (int f = 0; f < ng; ++f) {
      if (used[f] == B.fine) continue;
      int c = 0;
      for (int k = 0; k < B.nm; ++k) {
        const int g = B.group(k, f * B.fine);
        for (int d = 0; d < 2; ++d) c += B.cnt[k][d][g][B.block(k, d, e[i])] >= B.top[k][d][g];
      }
      c = c * 64 + used[f];
      if (best < 0 || c < bc) best = f, bc = c;
    }
    const int row = best * B.fine + used[best]++;
    out[row] = e[i];
    B.add(row, e[i], 1);
  }
  for (int i = 0; i < R; ++i) {
    if (out[i] == ~0u || !B.hot(i, out[i])) continue;
    for (int j = 0; j < R; ++j) {
      if (j / B.fine == i / B.fine) continue;
      int gain = 0;
      for (int k = 0; k < B.nm; ++k) {
        const int gi = B.group(k, i), gj = B.group(k, j);
        if (gi == gj) continue;
        for (int d = 0; d < 2; ++d)
          gain += B.top[k][d][gi] + B.top[k][d][gj] - B.top_after(k, d, gi, out[i], out[j]) -
                  B.top_after(k, d, gj, out[j], out[i]);
      }
      if (gain <= 0) continue;
      B.add(i, out[i], -1);
      if (out[j] != ~0u) B.add(j, out[j], -1), B.add(i, out[j], 1);
      B.add(j, out[i], 1);
      std::swap(out[i], out[j]);
      break;
    }
  }
  e.assign(out, out + R);
}

// Layers of at most R rotations by list scheduling on the dependency graph
// of the lexicographic sweep: a rotation follows the previous rotation on
// each of its two sites, so every site keeps its order.  Layer by layer, the
// ready rotations with the longest remaining chain (ties: lexicographic
// order) fill the R rows; this keeps the layer count near
// max(critical path, rotations / R).  The rows of a layer are then ordered
// to spread its LDS accesses over the banks (assign_rows).  Each layer is
// padded to exactly R entries; the padding entry of row q is the dummy pair
// (N + q, N + q),
// which the table kernel turns into an identity and the kernels apply to a
// scratch site.  The layer count is padded to a multiple of kMinLayers.
void build_schedule_rows(int N, const std::vector<uint8_t> &mask, int R, Schedule &s) {
  constexpr int kMinLayers = 8;
  s.N = N;
  std::vector<uint32_t> rot;  // lexicographic order
  int64_t p = 0;
  for (int a = 0; a < N; ++a)
    for (int b = a + 1; b < N; ++b, ++p)
      if (mask[p]) rot.push_back((uint32_t)a | ((uint32_t)b << 16));
  const int K = (int)rot.size();
  // successors: the next rotation on each site of rotation k
  std::vector<int> succ(2 * (size_t)K, -1), npred(K, 0), height(K, 1), lastk(N, -1);
  for (int k = 0; k < K; ++k) {
    const int site[2] = {(int)(rot[k] & 0xffffu), (int)(rot[k] >> 16)};
    for (int e = 0; e < 2; ++e) {
      const int j = lastk[site[e]];
      if (j >= 0) {
        succ[2 * (size_t)j + ((int)(rot[j] & 0xffffu) == site[e] ? 0 : 1)] = k;
        ++npred[k];
      }
      lastk[site[e]] = k;
    }
  }
  for (int k = K - 1; k >= 0; --k)
    for (int e = 0; e < 2; ++e) {
      const int j = succ[2 * (size_t)k + e];
      if (j >= 0) height[k] = std::max(height[k], height[j] + 1);
    }
  auto later = [&](int x, int y) { return height[x] != height[y] ? height[x] < height[y] : x > y; };
  std::vector<int> ready;
  for (int k = 0; k < K; ++k)
    if (!npred[k]) ready.push_back(k);
  std::make_heap(ready.begin(), ready.end(), later);
  std::vector<std::vector<uint32_t>> layers;
  std::vector<int> fresh;
  while (!ready.empty()) {
    std::vector<uint32_t> L;
    fresh.clear();
    while ((int)L.size() < R && !ready.empty()) {
      std::pop_heap(ready.begin(), ready.end(), later);
      const int k = ready.back();
      ready.pop_back();
      L.push_back(rot[k]);
      for (int e = 0; e < 2; ++e) {
        const int j = succ[2 * (size_t)k + e];
        if (j >= 0 && --npred[j] == 0) fresh.push_back(j);  // ready from the next layer on
      }
    }
    layers.push_back(std::move(L));
    for (int j : fresh) {
      ready.push_back(j);
      std::push_heap(ready.begin(), ready.end(), later);
    }
  }
  // at least kMinLayers layers, and a multiple of them (the kernel's
  // operand ring runs across sweeps)
  const size_t nl = std::max<size_t>(kMinLayers, (layers.size() + kMinLayers - 1) / kMinLayers * kMinLayers);
  layers.resize(nl);
  s.Kreal = K;
  s.K = (int)layers.size() * R;
  s.ab.clear();
  s.layer_off.assign(1, 0);
  std::vector<uint32_t> e(R);
  static thread_local LayerBanks banks;
  if (R >= 4 && R <= 64) banks.init(R);
  for (auto &L : layers) {
    for (int q = 0; q < R; ++q) e[q] = q < (int)L.size() ? L[q] : ~0u;
    if (R >= 4 && R <= 64) assign_rows(banks, e, (int)L.size());
    for (int q = 0; q < R; ++q)
      s.ab.push_back(e[q] != ~0u ? e[q] : (uint32_t)(N + q) | ((uint32_t)(N + q) << 16));
    s.layer_off.push_back((int)s.ab.size());
  }
}

void pack_schedule_rows(const Schedule &asap, int R, Schedule &s) {
  constexpr int kMinLayers = 8;
  const int N = asap.N;
  s.N = N, s.Kreal = asap.Kreal;
  s.ab.clear();
  s.layer_off.assign(1, 0);
  auto pad = [&]() {
    for (int q = (int)s.ab.size() % R; q && q < R; ++q) s.ab.push_back((uint32_t)(N + q) | ((uint32_t)(N + q) << 16));
  };
  for (int l = 0; l < asap.nlayers(); ++l) {
    s.ab.insert(s.ab.end(), asap.ab.begin() + asap.layer_off[l], asap.ab.begin() + asap.layer_off[l + 1]);
    pad();
  }
  while (s.ab.empty() || s.ab.size() % ((size_t)R * kMinLayers))
    for (int q = 0; q < R; ++q) s.ab.push_back((uint32_t)(N + q) | ((uint32_t)(N + q) << 16));
  s.K = (int)s.ab.size();
  for (int k = R; k <= s.K; k += R) s.layer_off.push_back(k);
}

static std::once_flag g_dev_once;
static int g_dev_status = NISE_OK;

int ensure_device() {
  std::call_once(g_dev_once, [] {
    int n = 0;
    hipError_t e = hipGetDeviceCount(&n);
    if (e != hipSuccess || n < 1) {
      g_dev_status = NISE_ERR_HIP;
      return;
    }
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, 0) != hipSuccess) {
      g_dev_status = NISE_ERR_HIP;
      return;
    }
    if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0) {
      fprintf(stderr, "libnise_hip: built for gfx950, device is %s\n", prop.gcnArchName);
    }
  });
  if (g_dev_status != NISE_OK) set_error("no usable HIP device");
  return g_dev_status;
}

// One non-blocking stream per host thread: the drop-in symbols may be called
// concurrently from OpenMP threads (src/propagate.c:1541-1548).
hipStream_t default_stream() {
  static thread_local hipStream_t st = nullptr;
  if (!st) {
    if (hipStreamCreateWithFlags(&st, hipStreamNonBlocking) != hipSuccess) st = nullptr;
  }
  return st;
}

// A second stream of the calling thread (default priority), for work that
// is independent of the default stream's and may overlap it.
hipStream_t aux_stream() {
  static thread_local hipStream_t st = nullptr;
  if (!st) {
    if (hipStreamCreateWithFlags(&st, hipStreamNonBlocking) != hipSuccess) st = nullptr;
  }
  return st;
}

}  // namespace nise

extern "C" const char *nise_last_error(void) { return nise::get_error(); }
extern "C" const char *nise_version(void) { return "nise-mi355x 0.1 (gfx950)"; }
