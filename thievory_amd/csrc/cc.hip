// cc.hip -- connected components of a symmetric graph by union-find with
// neighbour sampling (Afforest: Sutton, Ben-Nun, Bader, IPDPS 2018).
//
// The reference computes CC by min-label propagation along out-edges until
// no label changes (cc/cc.cu:71-614, cc_kernels.cu:50-66); on a symmetric
// graph its fixpoint labels every vertex with the smallest id of its
// component.  Union-find with "larger root under smaller" hooking (uf.hpp)
// ends with exactly those labels, and reads far fewer edges:
//   1. link every vertex to its first two neighbours (a vertex whose list is
//      on the host to its parent hint, when the store holds hints: its
//      neighbour of largest degree, one HBM word and no request over the
//      link), compress.  Where the hints alone form a giant tree -- the graph
//      has hubs, at which their trees meet -- every vertex links its hint only:
//      the start makes a smaller hint the vertex's parent at once, a larger
//      one is linked (R-MAT 23, edge factor 32, labels left in HBM: 0.53 ms
//      with two records a vertex, 310 us of it this step; 0.25 with the hints);
//   2. sample 1024 vertices: the most frequent root is the giant component;
//   3. link the remaining lists of the vertices outside it (its own
//      members need nothing more: an edge to a non-member is linked from
//      the other side, which the graph's symmetry guarantees; a list with no
//      more records than step 1 linked is done), compress.
// Directed graphs keep label propagation (the labels there are not
// components).
#include <algorithm>
#include <unordered_map>

#include "internal.hpp"
#include "scan.hpp"
#include "uf.hpp"

namespace thv {

namespace {

constexpr int UBS = 256;
constexpr uint32_t CC_SAMPLES = 1024;

// The start: every vertex its own parent, or (hint given) its parent hint
// where that is a smaller id -- parents point to smaller ids, so the trees
// are sound without a link.  cnt[1]: hints taken; cnt[0..2] start at zero.
__global__ void __launch_bounds__(UBS) k_cc_start(uint32_t *comp, const uint32_t *hint,
                                                  uint64_t n) {
  for (uint64_t v = blockIdx.x * (uint64_t)UBS + threadIdx.x; v < n;
       v += (uint64_t)gridDim.x * UBS) {
    const uint32_t h = hint ? hint[v] : NO_HINT;  // NO_HINT is past every id
    comp[v] = h < v ? h : (uint32_t)v;
  }
}

// Step 1 with hints: the larger ones are linked.
__global__ void __launch_bounds__(UBS) k_cc_hint(const uint32_t *hint, uint64_t n, uint32_t *comp,
                                                 uint32_t *err, uint32_t steps,
                                                 unsigned long long *cnt) {
  __shared__ unsigned long long sh[UBS / 64];
  unsigned long long taken = 0;
  for (uint64_t v = blockIdx.x * (uint64_t)UBS + threadIdx.x; v < n;
       v += (uint64_t)gridDim.x * UBS) {
    const uint32_t h = hint[v];
    taken += h != NO_HINT;
    if (h != NO_HINT && h > v) uf_link((uint32_t)v, h, comp, err, steps);
  }
  taken = block_sum<UBS>(taken, sh);
  if (threadIdx.x == 0 && taken) atomicAdd(&cnt[1], taken);
}

// Step 1 from the lists, one vertex per thread: its first two records, then
// the links; with hints (nullable), a host list's vertex links its hint instead.
template <int REC>
__global__ void __launch_bounds__(UBS)
k_cc_first(const uint64_t *eptr, const uint32_t *deg, const uint32_t *rbit, const uint32_t *hint,
           uint64_t n, uint32_t *comp, uint32_t *err, uint32_t steps, unsigned long long *cnt) {
  __shared__ unsigned long long sh[UBS / 64];
  unsigned long long rd[2] = {0, 0};  // records read (host, HBM); a hint counts as HBM
  for (uint64_t v = blockIdx.x * (uint64_t)UBS + threadIdx.x; v < n;
       v += (uint64_t)gridDim.x * UBS) {
    const uint32_t d = deg[v];
    if (!d) continue;
    if (hint && !((rbit[v >> 5] >> (v & 31)) & 1u)) {
      uf_link((uint32_t)v, hint[v], comp, err, steps);  // d > 0: a neighbour
      rd[1] += 1;
      continue;
    }
    const unsigned long long b = eptr[v];
    const uint32_t w0 = *reinterpret_cast<const uint32_t *>(b);
    const uint32_t w1 = d > 1 ? *reinterpret_cast<const uint32_t *>(b + REC) : w0;
    uf_link((uint32_t)v, w0, comp, err, steps);
    if (d > 1) uf_link((uint32_t)v, w1, comp, err, steps);
    rd[(rbit[v >> 5] >> (v & 31)) & 1u] += d > 1 ? 2 : 1;
  }
  const unsigned long long h = block_sum<UBS>(rd[0], sh);
  const unsigned long long m = block_sum<UBS>(rd[1], sh);
  if (threadIdx.x == 0) {
    if (h) atomicAdd(&cnt[0], h);
    if (m) atomicAdd(&cnt[1], m);
  }
}

// Every vertex to its root.  A vertex's own lane alone writes its parent, at
// every hop, so the lanes that walk the same chain jump over each other's
// hops: a chain of n takes some log n of them, where lanes that write only
// their roots walked about sqrt(2 n).  CC of a path of
// 2^20 vertices, half of its lists in HBM: 4.6 ms on the device with one write
// at the end, 0.2.
__global__ void __launch_bounds__(UBS) k_cc_compress(uint32_t *comp, uint64_t n, uint32_t *err,
                                                     uint32_t steps) {
  for (uint64_t v = blockIdx.x * (uint64_t)UBS + threadIdx.x; v < n;
       v += (uint64_t)gridDim.x * UBS) {
    uint32_t p = uf_load(&comp[v]);
    for (uint32_t step = 0;; step++) {
      const uint32_t g = uf_load(&comp[p]);
      if (g == p) break;
      if (step >= steps) {
        atomicOr(err, 1u);
        break;
      }
      uf_store(&comp[v], g);
      p = g;
    }
  }
}

__global__ void k_cc_sample(const uint32_t *comp, uint64_t n, uint32_t *out) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < CC_SAMPLES) out[i] = comp[mix64(i) % n];
}

// A sampled vertex, following hints: where they end (a pair that name each
// other, or a vertex without one; the vertex itself when that takes more than
// HOPS), its degree and whether its list is in HBM.
struct HintSample {
  uint32_t root, deg, hbm;
};
constexpr uint32_t HOPS = 64;
__global__ void k_hint_sample(const uint32_t *hint, const uint32_t *deg, const uint32_t *rbit,
                              uint64_t n, HintSample *out) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= CC_SAMPLES) return;
  const uint32_t v = (uint32_t)(mix64(i) % n);
  uint32_t u = v, root = v;
  for (uint32_t k = 0; k < HOPS; k++) {
    const uint32_t h = hint[u];
    if (h == NO_HINT || hint[h] == u) {
      root = min(u, h);
      break;
    }
    u = h;
  }
  out[i] = {root, deg[v], (rbit[v >> 5] >> (v & 31)) & 1u};
}

// Vertices whose remaining lists are linked in step 3: a root other than
// the giant's, and more records than step 1 linked (of a list on the host, of
// one in HBM).  One lane per vertex; lanes 0 and 32 write the wave's two
// bitmap words.
__global__ void __launch_bounds__(UBS)
k_cc_rest(const uint32_t *comp, const uint32_t *deg, const uint32_t *rbit, uint32_t linked_host,
          uint32_t linked_hbm, uint64_t n, uint32_t giant, uint32_t *bits, uint64_t words) {
  const uint32_t lane = threadIdx.x & 63;
  for (uint64_t v = blockIdx.x * (uint64_t)UBS + threadIdx.x; v - lane < words * 32;
       v += (uint64_t)gridDim.x * UBS) {
    bool sel = false;
    if (v < n) {
      const uint32_t linked = (rbit[v >> 5] >> (v & 31)) & 1u ? linked_hbm : linked_host;
      sel = deg[v] > linked && comp[v] != giant;
    }
    const unsigned long long b = __ballot(sel);
    if ((lane == 0 || lane == 32) && v >> 5 < words) bits[v >> 5] = (uint32_t)(b >> lane);
  }
}

int grid_for(uint64_t n, int cap) {
  return (int)std::max<uint64_t>(1, std::min<uint64_t>((n + UBS - 1) / UBS, (uint64_t)cap));
}

}  // namespace

// From a sample, once for the hints of a store: whether the lists outside the
// giant tree of hints hold no more records than two of every list in HBM,
// which are what CC reads instead (a record takes some 50-70 ps either way).
// Random graph of degree 8, 2^20 vertices, device ms from the hints / from two
// records: in HBM 0.78 / 0.32, half of it 0.90 / 0.29; R-MAT 23, edge factor 32,
// 0.25 / 0.53.
static bool hint_trees_meet(Graph &g, hipStream_t s) {
  DevMem &buf = g.ws.qs.slist;
  static_assert(CC_SAMPLES * sizeof(HintSample) <= TILE * 4, "a tile holds the sample");
  if (buf.bytes < CC_SAMPLES * sizeof(HintSample)) fail(THV_ESTATE, "sample buffer too small");
  hipLaunchKernelGGL(k_hint_sample, dim3(CC_SAMPLES / UBS), dim3(UBS), 0, s,
                     g.store.d_hint.as<uint32_t>(), g.d_deg.as<uint32_t>(),
                     g.store.d_rbit.as<uint32_t>(), g.n, buf.as<HintSample>());
  HIPC(hipGetLastError());
  std::vector<HintSample> hs(CC_SAMPLES);
  HIPC(hipMemcpyAsync(hs.data(), buf.p, CC_SAMPLES * sizeof(HintSample), hipMemcpyDeviceToHost, s));
  HIPC(hipStreamSynchronize(s));
  std::unordered_map<uint32_t, uint32_t> freq;
  uint32_t giant = 0, best = 0;
  for (const HintSample &x : hs)
    if (x.deg && ++freq[x.root] > best) {
      best = freq[x.root];
      giant = x.root;
    }
  uint64_t rest = 0, two = 0;
  for (const HintSample &x : hs) {
    if (x.deg > 1 && x.root != giant) rest += x.deg;
    if (x.hbm) two += std::min(x.deg, 2u);
  }
  return rest <= two;
}

bool cc_union_find(Graph &g, thv_stats *st) {
  Workspace &w = g.ws;
  hipStream_t s = g.stream;
  const uint64_t n = g.n, words = bitmap_words(n);
  uint32_t *comp = w.val.as<uint32_t>();
  unsigned long long *aux = w.aux.as<unsigned long long>();
  uint32_t *err = reinterpret_cast<uint32_t *>(aux + 2);
  launch_fill_u32(reinterpret_cast<uint32_t *>(aux), 0u, 6, s);  // [0], [1] records, [2] error
  const uint64_t t0 = now_ns();
  const int grid = grid_for(n, 16 * g.cus);
  const uint32_t steps = g.uf_max_steps;
  const uint64_t *eptr = g.store.d_eptr.as<uint64_t>();
  const uint32_t *deg = g.d_deg.as<uint32_t>(), *rbit = g.store.d_rbit.as<uint32_t>();
  const uint32_t *hint = g.store.d_hint.as<uint32_t>();  // null without hints
  if (hint && g.store.hints_meet < 0) g.store.hints_meet = hint_trees_meet(g, s);
  const bool by_hint = hint && g.store.hints_meet > 0;
  hipLaunchKernelGGL(k_cc_start, dim3(grid), dim3(UBS), 0, s, comp, by_hint ? hint : nullptr, n);
  const int lgrid = grid_for(n, 4 * g.cus);  // ends with an atomic per block
  if (by_hint) {
    // the start's trees may be one chain (consecutive ids of one degree): no
    // link is to walk it (a path of 100,000 vertices, a leaf of a smaller id
    // on each: 19.4 ms on the device without this pass, 0.9 with it, 1.2 from
    // two records a vertex; R-MAT 23 the same within 0.05)
    hipLaunchKernelGGL(k_cc_compress, dim3(grid), dim3(UBS), 0, s, comp, n, err, steps);
    hipLaunchKernelGGL(k_cc_hint, dim3(lgrid), dim3(UBS), 0, s, hint, n, comp, err, steps, aux);
  } else if (g.rec == 8)
    hipLaunchKernelGGL(k_cc_first<8>, dim3(grid), dim3(UBS), 0, s, eptr, deg, rbit, hint, n, comp,
                       err, steps, aux);
  else
    hipLaunchKernelGGL(k_cc_first<4>, dim3(grid), dim3(UBS), 0, s, eptr, deg, rbit, hint, n, comp,
                       err, steps, aux);
  hipLaunchKernelGGL(k_cc_compress, dim3(grid), dim3(UBS), 0, s, comp, n, err, steps);
  // the sample lands in the probe's short-list buffer (unused here; at
  // least one tile = 16 KB, CC_SAMPLES x 4 = 4 KB), then on the host
  static_assert(CC_SAMPLES * 4 <= TILE * 4, "sample buffer");
  if (w.qs.slist.bytes < CC_SAMPLES * 4) fail(THV_ESTATE, "CC sample buffer too small");
  uint32_t *samp = w.qs.slist.as<uint32_t>();
  hipLaunchKernelGGL(k_cc_sample, dim3(CC_SAMPLES / UBS), dim3(UBS), 0, s, comp, n, samp);
  std::vector<uint32_t> hs(CC_SAMPLES);
  HIPC(hipMemcpyAsync(hs.data(), samp, CC_SAMPLES * 4, hipMemcpyDeviceToHost, s));
  HIPC(hipStreamSynchronize(s));
  std::unordered_map<uint32_t, uint32_t> freq;
  uint32_t giant = hs[0], best = 0;
  for (uint32_t c : hs)
    if (++freq[c] > best) {
      best = freq[c];
      giant = c;
    }
  // step 3: the rest of the lists outside the giant component
  uint32_t *bits = w.front[0].as<uint32_t>();
  hipLaunchKernelGGL(k_cc_rest, dim3(grid), dim3(UBS), 0, s, comp, deg, rbit, hint ? 1u : 2u,
                     by_hint ? 1u : 2u, n, giant, bits, words);
  LevelCtr *c = w.qs.ctr.as<LevelCtr>();
  launch_compact(g, w.qs, bits, c, s);
  ExpandArgs a = expand_args(g, w.qs);
  a.ctr = c;
  a.val = comp;
  a.err = err;
  a.uf_steps = steps;
  HIPC(hipEventRecord(w.ev[0], s));
  launch_expand(g, A_CC_LINK, a, s);
  HIPC(hipEventRecord(w.ev[1], s));
  hipLaunchKernelGGL(k_cc_compress, dim3(grid), dim3(UBS), 0, s, comp, n, err, steps);
  LevelSide ps;
  ps.pub_src = c;
  ps.pub = w.h_ctr_dev;
  ps.npub = 1;
  ps.xsrc = aux;
  ps.xpub = w.h_aux_dev;
  ps.nx = 3;
  launch_publish(ps, s);
  HIPC(hipStreamSynchronize(s));
  if (w.h_aux[2]) return false;  // a link hit its step guard: not trusted
  if (st) {
    const LevelCtr &h = w.h_ctr[0];
    float ms = 0;
    HIPC(hipEventElapsedTime(&ms, w.ev[0], w.ev[1]));
    const uint64_t rec = (uint64_t)g.rec;
    const uint64_t first = w.h_aux[0] + w.h_aux[1];
    st->edges_traversed = first + h.qw[0] + h.qw[1];
    st->edges_examined = st->edges_traversed;
    st->host_bytes = (w.h_aux[0] + h.qw[0]) * rec;
    // records in HBM, 8 bytes of comp traffic per linked record, the degree
    // and first address of every vertex and comp twice per compress pass
    st->hbm_bytes = (w.h_aux[1] + h.qw[1]) * rec + 8 * st->edges_traversed + 12 * n + 16 * n;
    st->iterations = 2;
    st->expand_launches = 1;
    st->expand_ms = ms;
    st->ms = (now_ns() - t0) * 1e-6;
  }
  return true;
}

}  // namespace thv
