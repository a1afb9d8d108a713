// wide.hip -- graphs with 64-bit vertex ids (2^32 - 1 vertices or more).
//
// The reference declares BFS64 / CC64 / SSSP64 for CSR<uint64> but leaves
// them empty (src/bfs/bfs.cu:544, src/cc/cc.cu:616, src/sssp/sssp.cu:572),
// and its file format stores 4-byte destinations (graph.cuh:754), so a
// graph past 2^32 vertices enters only through this API.  Such graphs are
// usually sparse in their id space, so the edge lists are kept by listed
// vertex: the sorted ids of the k vertices with edges, their list offsets
// (k + 1) and u64 destinations (with u32 weights for SSSP).  Values follow
// the reference's conventions (BFS 1 + hops, CC the least id reaching the
// vertex, SSSP min(n + 1, 1 + distance); unreached n + 1).
//
// A vertex that is neither listed nor a destination keeps its initial value
// (CC: its id), so only the others have one in memory: the graph's vertices
// are numbered 0..N-1 on loading (the listed ones in id order, then the
// destinations without a list), the records name those numbers, and values
// are N x u64.  The caller's n x u64 array is made from them on request.
// (A dense array of 4.4e9 values was filled and digested in 12.6 ms of a
// 17 ms call, and every access to it missed the TLB.)
//
// Store: the listed vertices are cut into greedy runs of at most
// partition_edges edges (one oversize list alone, graph.cuh:270-304); the
// densest runs go to an HBM slab while the budget allows, the rest stay in
// mapped pinned host memory read zero-copy; eptr[j] is the address of
// listed vertex j's first record either way.
//
// Traversal: top-down over a queue of list segments of at most 256 records
// (a hub's list is shared by many waves), 16 lanes per segment with four
// records each in flight: most lists have some 16 records.  SSSP over R-MAT
// 18 (10.6M records relaxed) took 4.0 ms with a wave per list and an append
// per wave, 0.75 this way.  BFS claims a vertex with atomicCAS on
// its value and the winner appends its segments to the next queue; CC and
// SSSP lower values with atomicMin and append a vertex the first time it
// improves in a level (a stamp per vertex holds the last level that queued
// it).  Appends go out block by block, through LDS.
#include <algorithm>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_select.hpp>

#include "internal.hpp"
#include "scan.hpp"
#include "wide.hpp"

namespace thv {

namespace {

constexpr int WBS = 256;
// The expansion's blocks are few and large (one per CU): every block ends
// with an atomic on the next queue's counter, and those take turns, some 60
// ns each when the line moves between XCDs (with 8,192 waves each claiming
// its own places that was all a level of R-MAT 18 took: 0.5 ms).
constexpr int XBS = 1024;
constexpr uint64_t NOWHERE = ~0ull;
// a queue item: a vertex number and which segment of its list
constexpr uint32_t ITEM_BITS = 40;
constexpr uint64_t ITEM_MASK = (1ull << ITEM_BITS) - 1;
constexpr uint32_t SEG_MIN = 256;
constexpr uint32_t WG = 16;         // lanes per item
constexpr uint32_t WU = 4;          // records per lane in flight

// Number of id v among `ids` (k sorted ids), or NOWHERE.
__host__ __device__ inline uint64_t number_in(const uint64_t *ids, uint64_t k, uint64_t v) {
  uint64_t lo = 0, n = k;
  if (!k || ids[0] > v) return NOWHERE;
  while (n > 1) {  // ids[lo] <= v
    const uint64_t h = n >> 1;
    if (ids[lo + h] <= v) lo += h;
    n -= h;
  }
  return ids[lo] == v ? lo : NOWHERE;
}

struct WideArgs {
  const uint64_t *uid, *loff, *eptr;
  uint64_t k, none;
  int rec;                      // 8: u64 number; 16: {u64 number, u32 w, pad}
  uint32_t seg_shift;           // log2 of the records per segment
  const uint64_t *q;            // this level's items
  const unsigned long long *qn;
  uint64_t *nq;                 // next queue and its count
  unsigned long long *nqn;
  unsigned long long *found;    // set when the level finds a vertex, listed or not
  unsigned long long *edges;    // per block, edges scanned (stats)
  uint64_t *val;
  uint32_t *stamp;              // CC/SSSP: the last level that queued the vertex
  uint32_t level;               //   this level + 1
  uint64_t level_value;         // BFS: value of the vertices this level finds
};

// A wave's items on their way to the next queue: gathered in LDS and copied
// out when the buffer is full, and at the block's end.
constexpr uint32_t QBUF = 512;
struct ItemBuf {
  uint64_t *buf;  // QBUF items of this wave
  uint32_t n;     // wave-uniform
  bool found;     // a vertex was found (wave-uniform)
};

__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ uint64_t claim(unsigned long long *count, uint32_t n) {
  unsigned long long base = 0;
  if (lane_id() == 0) base = atomicAdd(count, (unsigned long long)n);
  return __shfl(base, 0, 64);
}

__device__ __forceinline__ void flush(const WideArgs &a, ItemBuf &b) {
  if (!b.n) return;
  wave_lds_sync();
  const uint64_t base = claim(a.nqn, b.n);
  for (uint32_t i = lane_id(); i < b.n; i += 64) a.nq[base + i] = b.buf[i];
  b.n = 0;
  wave_lds_sync();
}

// Appends the list segments of the vertices w[u] of the lanes with take[u]
// (none for a vertex without a list).  Every lane of the wave takes part.
template <uint32_t U>
__device__ __forceinline__ void append(const WideArgs &a, ItemBuf &b, const bool (&take)[U],
                                       const uint64_t (&w)[U]) {
  bool any = false;
#pragma unroll
  for (uint32_t u = 0; u < U; u++) any |= take[u];
  if (!wave_ballot(any)) return;
  b.found = true;
  uint64_t l0[U], l1[U];
#pragma unroll
  for (uint32_t u = 0; u < U; u++) {
    const uint64_t j = take[u] && w[u] < a.k ? w[u] : a.k;  // loff has k + 1 entries
    l0[u] = a.loff[j];
    l1[u] = a.loff[j < a.k ? j + 1 : j];
  }
  uint32_t c[U], sum = 0;
#pragma unroll
  for (uint32_t u = 0; u < U; u++) {
    c[u] = (uint32_t)((l1[u] - l0[u] + (1ull << a.seg_shift) - 1) >> a.seg_shift);
    sum += c[u];
  }
  const uint32_t inc = wave_incl_scan(sum);
  const uint32_t tot = (uint32_t)__builtin_amdgcn_readlane((int)inc, 63);
  uint32_t at = inc - sum;
  uint64_t base = 0;
  const bool direct = tot > QBUF;  // long lists: straight to the queue
  if (direct) base = claim(a.nqn, tot);
  else if (b.n + tot > QBUF) flush(a, b);
#pragma unroll
  for (uint32_t u = 0; u < U; u++) {
    for (uint32_t i = 0; i < c[u]; i++, at++) {
      const uint64_t item = (uint64_t)i << ITEM_BITS | w[u];
      if (direct) a.nq[base + at] = item;
      else b.buf[b.n + at] = item;
    }
  }
  if (!direct) b.n += tot;
}

// The block's end: what its waves still hold goes out with one atomic.
struct BlockEnd {
  unsigned long long base;
  uint32_t n[XBS / 64], found[XBS / 64];
};
__device__ __forceinline__ bool flush_block(const WideArgs &a, ItemBuf &b, BlockEnd &e) {
  const uint32_t wv = threadIdx.x >> 6;
  if (lane_id() == 0) {
    e.n[wv] = b.n;
    e.found[wv] = b.found;
  }
  __syncthreads();
  uint32_t at = 0, tot = 0;
  bool found = false;
  for (uint32_t i = 0; i < XBS / 64; i++) {
    at += i < wv ? e.n[i] : 0u;
    tot += e.n[i];
    found |= e.found[i] != 0;
  }
  if (threadIdx.x == 0 && tot) e.base = atomicAdd(a.nqn, (unsigned long long)tot);
  __syncthreads();
  for (uint32_t i = lane_id(); i < b.n; i += 64) a.nq[e.base + at + i] = b.buf[i];
  return found;
}

// CC's first queue: every list's first segment in the order of the ids, so that
// the least labels set out first (a random graph of degree 16 took a third
// round, half as many edges again, whenever vertex 0 came late), then the
// longer lists' other segments.  *nqn is k before.
__global__ void __launch_bounds__(XBS) k_wide_all(WideArgs a) {
  const uint64_t T = (uint64_t)gridDim.x * XBS;
  for (uint64_t j = (uint64_t)blockIdx.x * XBS + threadIdx.x; j - lane_id() < a.k; j += T) {
    uint32_t more = 0;
    if (j < a.k) {
      a.nq[j] = j;
      more = (uint32_t)((a.loff[j + 1] - a.loff[j] - 1) >> a.seg_shift);  // lists are not empty
    }
    if (!wave_ballot(more != 0)) continue;
    const uint32_t inc = wave_incl_scan(more);
    const uint64_t at = claim(a.nqn, (uint32_t)__builtin_amdgcn_readlane((int)inc, 63)) + inc - more;
    for (uint32_t i = 0; i < more; i++) a.nq[at + i] = (uint64_t)(i + 1) << ITEM_BITS | j;
  }
}

template <int ALGO, int REC>
__global__ void __launch_bounds__(XBS) k_wide_expand(WideArgs a) {
  __shared__ uint64_t buf[XBS / 64][QBUF];
  __shared__ BlockEnd end;
  __shared__ unsigned long long sh[XBS / 64];
  constexpr uint32_t IPW = 64 / WG;  // items per wave and step
  const uint32_t lane = threadIdx.x & 63, gl = lane & (WG - 1), gi = lane / WG;
  ItemBuf ib{buf[threadIdx.x >> 6], 0, false};
  const uint64_t step = (uint64_t)gridDim.x * (XBS / 64) * IPW;
  const uint64_t total = *a.qn;
  unsigned long long scanned = 0;
  for (uint64_t q0 = ((uint64_t)blockIdx.x * (XBS / 64) + (threadIdx.x >> 6)) * IPW; q0 < total;
       q0 += step) {
    uint64_t e = 0, d = 0, vv = 0;
    unsigned long long base = 0;
    if (q0 + gi < total) {
      const uint64_t item = a.q[q0 + gi], j = item & ITEM_MASK;
      e = (item >> ITEM_BITS) << a.seg_shift;
      d = min(a.loff[j + 1] - a.loff[j], e + (1ull << a.seg_shift));
      base = a.eptr[j];
      if (ALGO != THV_ALGO_BFS) vv = a.val[j];
      if (gl == 0) scanned += d - e;
    }
    for (; wave_ballot(e < d); e += WG * WU) {  // wave-uniform: the appends need every lane
      uint64_t w[WU], nv[WU], cur[WU];
#pragma unroll
      for (uint32_t u = 0; u < WU; u++) {
        const uint64_t x = e + u * WG + gl;
        w[u] = NOWHERE;
        nv[u] = ALGO == THV_ALGO_BFS ? a.level_value : vv;
        if (x < d) {
          typedef const __attribute__((address_space(1))) uint64_t *gp;
          typedef const __attribute__((address_space(1))) uint32_t *gp32;
          w[u] = *reinterpret_cast<gp>(base + x * REC);
          if (ALGO == THV_ALGO_SSSP) nv[u] += *reinterpret_cast<gp32>(base + x * REC + 8);
        }
      }
#pragma unroll
      for (uint32_t u = 0; u < WU; u++) cur[u] = a.val[w[u] != NOWHERE ? w[u] : 0];
      bool take[WU];
#pragma unroll
      for (uint32_t u = 0; u < WU; u++) {
        take[u] = false;
        if (w[u] == NOWHERE) continue;
        unsigned long long *p = reinterpret_cast<unsigned long long *>(&a.val[w[u]]);
        if (ALGO == THV_ALGO_BFS) {
          if (cur[u] == a.none) take[u] = atomicCAS(p, a.none, nv[u]) == a.none;
        } else if (nv[u] < cur[u]) {
          take[u] = nv[u] < atomicMin(p, (unsigned long long)nv[u]);
        }
      }
      if (ALGO != THV_ALGO_BFS) {
#pragma unroll
        for (uint32_t u = 0; u < WU; u++)
          if (take[u]) take[u] = atomicMax(&a.stamp[w[u]], a.level) < a.level;
      }
      append(a, ib, take, w);
    }
  }
  const bool found = flush_block(a, ib, end);
  scanned = block_sum<XBS>(scanned, sh);
  if (threadIdx.x == 0) {
    if (scanned) a.edges[blockIdx.x] += scanned;  // this block's own count
    if (found) *a.found = 1;
  }
}

// The level's end: the next queue's count and whether it found vertices to
// the host; this queue's count and the flag cleared.
__global__ void k_wide_end(unsigned long long *qn, const unsigned long long *nqn,
                           unsigned long long *found, unsigned long long *host) {
  *qn = 0;
  host[0] = *nqn;
  host[1] = *found;
  *found = 0;
  __threadfence_system();
}

// The start of a run: every value `none` (CC: the vertex's id) but the
// source's 1, no stamps, the counters clear; the queue holds the source's
// segments (CC: as many as there are lists, k_wide_all's).
__global__ void __launch_bounds__(WBS)
k_wide_init(WideArgs a, uint64_t N, bool ids, uint64_t src, unsigned long long *ctr,
            uint32_t nctr) {
  __shared__ uint64_t buf[QBUF];
  const uint64_t T = (uint64_t)gridDim.x * WBS;
  for (uint64_t i = (uint64_t)blockIdx.x * WBS + threadIdx.x; i < N; i += T) {
    a.val[i] = i == src ? 1ull : ids ? a.uid[i] : a.none;
    if (a.stamp) a.stamp[i] = 0;
  }
  if (blockIdx.x == 0) {
    for (uint32_t i = threadIdx.x; i < nctr; i += WBS) ctr[i] = 0;
    __threadfence();
    __syncthreads();
    if (ids && threadIdx.x == 0) *a.nqn = a.k;
    if (threadIdx.x < 64 && src < a.k) {
      ItemBuf ib{buf, 0, false};
      const bool take[1] = {threadIdx.x == 0};
      const uint64_t w[1] = {src};
      append(a, ib, take, w);
      flush(a, ib);
    }
  }
}

// Digest of the values in memory: sum of mix64(mix64(id) + value) over those
// other than `none` (mod 2^64), their count and the largest; own (CC): each
// term less its initial value's, mix64(mix64(id) + id).
__global__ void __launch_bounds__(WBS) k_wide_digest(const uint64_t *val, const uint64_t *uid,
                                                    uint64_t N, uint64_t none, bool own,
                                                    unsigned long long *out) {
  __shared__ unsigned long long sh[WBS / 64];
  unsigned long long h = 0, c = 0, mx = 0;
  for (uint64_t i = blockIdx.x * (uint64_t)WBS + threadIdx.x; i < N;
       i += (uint64_t)gridDim.x * WBS) {
    const uint64_t x = val[i];
    if (x == none) continue;
    const uint64_t v = uid[i], hv = mix64(v);
    h += mix64(hv + x);
    if (own) h -= mix64(hv + v);
    c++;
    mx = x > mx ? x : mx;
  }
  const unsigned long long hs = block_sum<WBS>(h, sh), cs = block_sum<WBS>(c, sh);
  unsigned long long m = mx;
  for (int d = 32; d >= 1; d >>= 1) {
    const unsigned long long o = __shfl_xor(m, d, 64);
    m = o > m ? o : m;
  }
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (uint32_t w = 1; w < WBS / 64; w++) m = sh[w] > m ? sh[w] : m;
    if (hs) atomicAdd(&out[0], hs);
    if (cs) atomicAdd(&out[1], cs);
    if (m) atomicMax(&out[2], m);
  }
}

// Sum of mix64(mix64(v) + v) over v < n: CC's digest with every vertex its
// own label.  Bound by the 64-bit multiplies.
__global__ void __launch_bounds__(WBS) k_wide_own(uint64_t n, unsigned long long *out) {
  __shared__ unsigned long long sh[WBS / 64];
  unsigned long long h = 0;
  for (uint64_t v = blockIdx.x * (uint64_t)WBS + threadIdx.x; v < n;
       v += (uint64_t)gridDim.x * WBS)
    h += mix64(mix64(v) + v);
  h = block_sum<WBS>(h, sh);
  if (threadIdx.x == 0) atomicAdd(out, h);
}

// Values of the given vertices; one without a number has its initial value
// (lone: the source of the last run when it has none, value 1).
__global__ void k_wide_gather(const uint64_t *val, const uint64_t *uid, uint64_t k, uint64_t N,
                              bool ids, uint64_t none, uint64_t lone, const uint64_t *at,
                              uint64_t cnt, uint64_t *out) {
  for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < cnt;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const uint64_t v = at[i];
    uint64_t j = number_in(uid, k, v);
    if (j == NOWHERE) {
      j = number_in(uid + k, N - k, v);
      if (j != NOWHERE) j += k;
    }
    out[i] = j != NOWHERE ? val[j] : v == lone ? 1ull : ids ? v : none;
  }
}

// A piece [v0, v0 + cnt) of the caller's dense array: initial values, then
// the numbered vertices uid[a, b) that lie in it.
__global__ void k_wide_fill(uint64_t *p, uint64_t v0, uint64_t cnt, bool ids, uint64_t none,
                            uint64_t lone) {
  for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < cnt;
       i += (uint64_t)gridDim.x * blockDim.x)
    p[i] = v0 + i == lone ? 1ull : ids ? v0 + i : none;
}
__global__ void k_wide_scatter(uint64_t *p, uint64_t v0, const uint64_t *uid, const uint64_t *val,
                               uint64_t a, uint64_t b) {
  for (uint64_t i = a + blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < b;
       i += (uint64_t)gridDim.x * blockDim.x)
    p[uid[i] - v0] = val[i];
}

// ---- loading -------------------------------------------------------------------

// Records of destinations dst[0, cnt): their numbers (and weights).  Without
// `extra`, a destination that is not listed goes to `miss`; with it, every
// one is found.
__global__ void __launch_bounds__(WBS)
k_wide_number(const uint64_t *dst, const uint32_t *w, uint64_t cnt, const uint64_t *ids,
              uint64_t k, const uint64_t *extra, uint64_t x, int rec, unsigned char *out,
              uint64_t *miss, unsigned long long *nmiss) {
  for (uint64_t i = blockIdx.x * (uint64_t)WBS + threadIdx.x; i < cnt;
       i += (uint64_t)gridDim.x * WBS) {
    const uint64_t v = dst[i];
    uint64_t j = number_in(ids, k, v);
    if (j == NOWHERE) {
      if (extra) j = k + number_in(extra, x, v);
      else miss[atomicAdd(nmiss, 1ull)] = v;
    }
    if (rec == 8) {
      reinterpret_cast<uint64_t *>(out)[i] = j;
    } else {
      ulonglong2 r;
      r.x = j;
      r.y = w[i];
      reinterpret_cast<ulonglong2 *>(out)[i] = r;
    }
  }
}

int grid_of(uint64_t n, int cap) {
  return (int)std::max<uint64_t>(1, std::min<uint64_t>((n + WBS - 1) / WBS, (uint64_t)cap));
}

}  // namespace

Graph64::~Graph64() {
  if (stream) {
    (void)hipStreamSynchronize(stream);
    (void)hipStreamDestroy(stream);
  }
  if (h_ctr) (void)hipHostFree(h_ctr);
}

// The n keys of a, sorted, each once, to b (n places); a is scratch.  Returns
// how many.  count: a device word.
static uint64_t sorted_unique(uint64_t *a, uint64_t *b, uint64_t n, unsigned long long *count,
                              DevMem &tmp, hipStream_t s) {
  rocprim::double_buffer<uint64_t> db(a, b);
  size_t bytes = 0, ubytes = 0;
  HIPC(rocprim::radix_sort_keys(nullptr, bytes, db, (size_t)n, 0u, 64u, s));
  HIPC(rocprim::unique(nullptr, ubytes, a, b, count, (size_t)n, rocprim::equal_to<uint64_t>(), s));
  bytes = std::max(bytes, ubytes);
  if (tmp.bytes < bytes) tmp.alloc(bytes);
  HIPC(rocprim::radix_sort_keys(tmp.p, bytes, db, (size_t)n, 0u, 64u, s));
  HIPC(rocprim::unique(tmp.p, bytes, db.current(), db.alternate(), count, (size_t)n,
                       rocprim::equal_to<uint64_t>(), s));
  unsigned long long u = 0;
  HIPC(hipMemcpyAsync(&u, count, 8, hipMemcpyDeviceToHost, s));
  if (db.alternate() != b)
    HIPC(hipMemcpyAsync(b, db.alternate(), n * 8, hipMemcpyDeviceToDevice, s));
  HIPC(hipStreamSynchronize(s));
  return u;
}

// Numbers the destinations and writes the records (in mapped pinned host
// memory): pieces of the array go to the GPU, which finds each destination
// among the listed ids.  Those of a piece that are not listed are sorted and
// made unique there and merged into `extra`; such a piece's records are written
// once extra is complete.
static void number_destinations(Graph64 &g, const uint64_t *dst, const uint32_t *w) {
  constexpr uint64_t PIECE = 16ull << 20;
  const uint64_t piece = std::max<uint64_t>(1, std::min(PIECE, g.m));
  hipStream_t s = g.stream;
  // destinations, missing ones, weights, counts of missing and of unique ones
  const uint64_t at_miss = piece * 8, at_n = at_miss + piece * 8, at_w = at_n + 16;
  DevMem buf, keys, tmp, extra;
  uint64_t x = 0;  // ids in extra
  buf.alloc(at_w + (w ? piece * 4 : 0));
  unsigned char *b = buf.as<unsigned char>();
  uint64_t *d_dst = reinterpret_cast<uint64_t *>(b);
  uint64_t *d_miss = reinterpret_cast<uint64_t *>(b + at_miss);
  unsigned long long *d_n = reinterpret_cast<unsigned long long *>(b + at_n);
  uint32_t *d_w = w ? reinterpret_cast<uint32_t *>(b + at_w) : nullptr;
  std::vector<uint8_t> again(div_up(std::max<uint64_t>(g.m, 1), piece), 0);
  unsigned char *rec = static_cast<unsigned char *>(g.h_edges.dev);
  const int grid = grid_of(piece, 16 * g.cus);
  uint64_t held = UINT64_MAX;  // the piece that is in the buffer
  // writes a piece's records; how many of its destinations are missing
  auto number = [&](uint64_t e0, uint64_t cnt, bool final) {
    if (held != e0) {
      HIPC(hipMemcpy(d_dst, dst + e0, cnt * 8, hipMemcpyHostToDevice));
      if (w) HIPC(hipMemcpy(d_w, w + e0, cnt * 4, hipMemcpyHostToDevice));
      held = e0;
    }
    launch_fill_u32(reinterpret_cast<uint32_t *>(d_n), 0u, 2, s);
    hipLaunchKernelGGL(k_wide_number, dim3(grid), dim3(WBS), 0, s, d_dst, d_w, cnt,
                       g.d_uid.as<uint64_t>(), g.k, final ? extra.as<uint64_t>() : nullptr, x, g.rec,
                       rec + e0 * g.rec, d_miss, d_n);
    HIPC(hipGetLastError());
    unsigned long long n = 0;
    HIPC(hipMemcpyAsync(&n, d_n, 8, hipMemcpyDeviceToHost, s));
    HIPC(hipStreamSynchronize(s));
    return (uint64_t)n;
  };
  for (uint64_t e0 = 0; e0 < g.m; e0 += piece) {
    const uint64_t n = number(e0, std::min(piece, g.m - e0), false);
    if (!n) continue;
    again[e0 / piece] = 1;
    if (keys.bytes < n * 8) keys.alloc(n * 8);
    const uint64_t u = sorted_unique(d_miss, keys.as<uint64_t>(), n, d_n + 1, tmp, s);
    if (!x) {
      extra.swap(keys);
      x = u;
    } else {  // with those of earlier pieces
      DevMem both;
      both.alloc((x + u) * 8);
      uint64_t *p = both.as<uint64_t>();
      HIPC(hipMemcpyAsync(p, extra.p, x * 8, hipMemcpyDeviceToDevice, s));
      HIPC(hipMemcpyAsync(p + x, keys.p, u * 8, hipMemcpyDeviceToDevice, s));
      HIPC(hipStreamSynchronize(s));
      if (extra.bytes < (x + u) * 8) extra.alloc((x + u) * 8);
      x = sorted_unique(p, extra.as<uint64_t>(), x + u, d_n + 1, tmp, s);
    }
  }
  g.N = g.k + x;
  if (g.N > ITEM_MASK) fail(THV_ENOTSUP, "more than 2^40 vertices with edges");
  if (!x) return;
  DevMem uid;
  uid.alloc(g.N * 8);
  if (g.k) HIPC(hipMemcpyAsync(uid.p, g.d_uid.p, g.k * 8, hipMemcpyDeviceToDevice, s));
  HIPC(hipMemcpyAsync(uid.as<uint64_t>() + g.k, extra.p, x * 8, hipMemcpyDeviceToDevice, s));
  for (uint64_t e0 = 0; e0 < g.m; e0 += piece)
    if (again[e0 / piece]) number(e0, std::min(piece, g.m - e0), true);
  g.h_extra.resize(x);
  HIPC(hipMemcpy(g.h_extra.data(), extra.p, x * 8, hipMemcpyDeviceToHost));
  HIPC(hipStreamSynchronize(s));
  g.d_uid.swap(uid);
}

Graph64 *graph64_from_lists(uint64_t n, uint64_t k, const uint64_t *ids, const uint64_t *loff,
                            const uint64_t *dst, const uint32_t *w) {
  if (n == 0 || n == UINT64_MAX) fail(THV_EINVAL, "vertex count out of range");
  if (k > n) fail(THV_EINVAL, "more listed vertices than vertices");
  if (k && (!ids || !loff)) fail(THV_EINVAL, "null list arrays");
  if (k == 0 && loff && loff[0] != 0) fail(THV_EINVAL, "offsets must start at 0");
  const uint64_t m = k ? loff[k] : 0;
  if (m && !dst) fail(THV_EINVAL, "null destinations");
  if (k && loff[0] != 0) fail(THV_EINVAL, "offsets must start at 0");
  uint64_t longest = 0;
  for (uint64_t j = 0; j < k; j++) {
    if (ids[j] >= n) fail(THV_EINVAL, "listed id out of range");
    if (j && ids[j] <= ids[j - 1]) fail(THV_EINVAL, "listed ids must be strictly ascending");
    if (loff[j + 1] <= loff[j]) fail(THV_EINVAL, "a listed vertex needs at least one edge");
    longest = std::max(longest, loff[j + 1] - loff[j]);
  }
  for (uint64_t e = 0; e < m; e++)
    if (dst[e] >= n) fail(THV_EINVAL, "destination out of range");
  std::unique_ptr<Graph64> g(new Graph64());
  g->n = n;
  g->k = k;
  g->m = m;
  g->rec = w ? 16 : 8;
  // segments of SEG_MIN records, longer where a list would have too many
  g->seg_shift = (uint32_t)__builtin_ctz(SEG_MIN);
  while ((longest >> g->seg_shift) >= (1ull << (64 - ITEM_BITS))) g->seg_shift++;
  if (k) g->h_ids.assign(ids, ids + k);
  if (k) g->h_loff.assign(loff, loff + k + 1);
  else g->h_loff.assign(1, 0);
  HIPC(hipGetDevice(&g->device));
  hipDeviceProp_t prop;
  HIPC(hipGetDeviceProperties(&prop, g->device));
  g->cus = prop.multiProcessorCount;
  HIPC(hipStreamCreateWithFlags(&g->stream, hipStreamNonBlocking));
  HIPC(hipHostMalloc((void **)&g->h_ctr, 8 * 8, hipHostMallocMapped | hipHostMallocCoherent));
  memset(g->h_ctr, 0, 8 * 8);
  HIPC(hipHostGetDevicePointer((void **)&g->h_ctr_dev, g->h_ctr, 0));
  g->h_edges.alloc(std::max<uint64_t>(m, 1) * g->rec);
  g->d_uid.alloc(std::max<uint64_t>(k, 1) * 8);
  if (k) HIPC(hipMemcpy(g->d_uid.p, ids, k * 8, hipMemcpyHostToDevice));
  g->d_loff.alloc((k + 1) * 8);
  HIPC(hipMemcpy(g->d_loff.p, g->h_loff.data(), (k + 1) * 8, hipMemcpyHostToDevice));
  number_destinations(*g, dst, w);
  graph64_store(*g, UINT64_MAX, 1u << 16);
  return g.release();
}

void graph64_store(Graph64 &g, uint64_t budget, uint32_t part_edges) {
  if (part_edges == 0) fail(THV_EINVAL, "partition_edges must be > 0");
  HIPC(hipStreamSynchronize(g.stream));
  // greedy runs of listed vertices with at most part_edges edges
  std::vector<uint64_t> pj{0};
  uint64_t cur = 0;
  for (uint64_t j = 0; j < g.k; j++) {
    const uint64_t d = g.h_loff[j + 1] - g.h_loff[j];
    if (cur + d <= part_edges || j == pj.back()) {
      cur += d;
    } else {
      pj.push_back(j);
      cur = d;
    }
  }
  pj.push_back(g.k);
  const uint64_t P = pj.size() - 1;
  // densest runs first (edges per listed vertex), whole, while they fit
  std::vector<uint64_t> order(P);
  for (uint64_t p = 0; p < P; p++) order[p] = p;
  auto edges_of = [&](uint64_t p) { return g.h_loff[pj[p + 1]] - g.h_loff[pj[p]]; };
  auto dens = [&](uint64_t p) {
    return (double)edges_of(p) / (double)std::max<uint64_t>(1, pj[p + 1] - pj[p]);
  };
  std::stable_sort(order.begin(), order.end(),
                   [&](uint64_t a, uint64_t b) { return dens(a) > dens(b); });
  std::vector<uint8_t> res(P, 0);
  uint64_t used = 0;
  for (uint64_t p : order) {
    const uint64_t b = edges_of(p) * g.rec;
    if (budget != UINT64_MAX && used + b > budget) continue;
    res[p] = 1;
    used += b;
  }
  g.slab.alloc(std::max<uint64_t>(used, 8));
  std::vector<uint64_t> eptr(std::max<uint64_t>(g.k, 1));
  const unsigned char *host = static_cast<const unsigned char *>(g.h_edges.dev);
  uint64_t at = 0, dev_edges = 0;
  uint32_t pdev = 0;
  for (uint64_t p = 0; p < P; p++) {
    const uint64_t e0 = g.h_loff[pj[p]], ne = edges_of(p);
    if (res[p] && ne) {
      HIPC(hipMemcpy(static_cast<unsigned char *>(g.slab.p) + at,
                     static_cast<const unsigned char *>(g.h_edges.p) + e0 * g.rec, ne * g.rec,
                     hipMemcpyHostToDevice));
      for (uint64_t j = pj[p]; j < pj[p + 1]; j++)
        eptr[j] = (uint64_t)(static_cast<unsigned char *>(g.slab.p) + at +
                             (g.h_loff[j] - e0) * g.rec);
      at += ne * g.rec;
      dev_edges += ne;
      pdev++;
    } else {
      for (uint64_t j = pj[p]; j < pj[p + 1]; j++) eptr[j] = (uint64_t)(host + g.h_loff[j] * g.rec);
    }
  }
  g.d_eptr.alloc(eptr.size() * 8);
  HIPC(hipMemcpy(g.d_eptr.p, eptr.data(), eptr.size() * 8, hipMemcpyHostToDevice));
  g.P = (uint32_t)P;
  g.Pdev = pdev;
  g.dev_edges = dev_edges;
  g.budget = budget;
}

// Counters (u64), on lines of their own: the queues', the found flag, the
// digest, then the blocks' edges.
constexpr uint32_t CTR_Q = 0, CTR_FOUND = 32, CTR_DIGEST = 48, CTR_EDGES = 64;

static void ensure_work(Graph64 &g) {
  const uint64_t qcap = g.k + (g.m >> g.seg_shift) + 1;
  if (g.val.p) return;
  // The ids of a graph are bounded by the memory their n values would take:
  // they are never all there, but CC's digest visits every id (2^60 of them
  // would take years).
  size_t fr = 0, tot = 0;
  drop_idle_engines();
  HIPC(hipMemGetInfo(&fr, &tot));
  if (g.n > fr / 8)
    fail(THV_ENOMEM, "the values of " + std::to_string(g.n) + " vertices exceed the " +
                         std::to_string(fr) + " bytes of free device memory");
  for (auto &q : g.q) q.alloc(qcap * 8);
  g.ctr.alloc((CTR_EDGES + g.cus) * 8);
  g.stamp.alloc(std::max<uint64_t>(g.N, 1) * 4);
  g.val.alloc(std::max<uint64_t>(g.N, 1) * 8);
}

// The number of id v, or NOWHERE (neither listed nor a destination).
static uint64_t number_of(const Graph64 &g, uint64_t v) {
  const uint64_t j = number_in(g.h_ids.data(), g.k, v);
  if (j != NOWHERE) return j;
  const uint64_t x = number_in(g.h_extra.data(), g.h_extra.size(), v);
  return x != NOWHERE ? g.k + x : NOWHERE;
}

// The caller's dense array, a piece of it at a time.
static void dense_values(Graph64 &g, uint64_t *out) {
  constexpr uint64_t PIECE = 8ull << 20;
  const uint64_t piece = std::min(PIECE, g.n);
  hipStream_t s = g.stream;
  const bool ids = g.last_algo == THV_ALGO_CC;
  const uint64_t *uid = g.d_uid.as<uint64_t>();
  DevMem d;
  d.alloc(piece * 8);
  for (uint64_t v0 = 0; v0 < g.n; v0 += piece) {
    const uint64_t cnt = std::min(piece, g.n - v0);
    hipLaunchKernelGGL(k_wide_fill, dim3(grid_of(cnt, 8 * g.cus)), dim3(WBS), 0, s,
                       d.as<uint64_t>(), v0, cnt, ids, g.n + 1, g.lone);
    auto scatter = [&](const std::vector<uint64_t> &h, uint64_t first) {
      const uint64_t a = std::lower_bound(h.begin(), h.end(), v0) - h.begin();
      const uint64_t b = std::lower_bound(h.begin(), h.end(), v0 + cnt) - h.begin();
      if (a < b)
        hipLaunchKernelGGL(k_wide_scatter, dim3(grid_of(b - a, 8 * g.cus)), dim3(WBS), 0, s,
                           d.as<uint64_t>(), v0, uid, g.val.as<uint64_t>(), first + a, first + b);
    };
    scatter(g.h_ids, 0);
    scatter(g.h_extra, g.k);
    HIPC(hipGetLastError());
    HIPC(hipStreamSynchronize(s));
    g.rb.copy(out + v0, d.p, cnt * 8, s);
  }
}

template <int ALGO>
static void launch_wide(Graph64 &g, const WideArgs &a, uint64_t items, hipStream_t s) {
  const int grid = (int)std::max<uint64_t>(
      1, std::min<uint64_t>(div_up(items, XBS / WG), g.cus));
  if (g.rec == 16)
    hipLaunchKernelGGL((k_wide_expand<ALGO, 16>), dim3(grid), dim3(XBS), 0, s, a);
  else
    hipLaunchKernelGGL((k_wide_expand<ALGO, 8>), dim3(grid), dim3(XBS), 0, s, a);
}

void run_wide(Graph64 &g, int algo, uint64_t src, uint64_t *out, thv_stats *st,
              uint64_t *digest3) {
  if (algo != THV_ALGO_CC && src >= g.n) fail(THV_EINVAL, "source vertex out of range");
  if (algo == THV_ALGO_SSSP && g.rec != 16)
    fail(THV_ENOTSUP, "SSSP needs weights (build the graph with them)");
  ensure_work(g);
  hipStream_t s = g.stream;
  const bool cc = algo == THV_ALGO_CC;
  const uint64_t none = g.n + 1;
  unsigned long long *ctr = g.ctr.as<unsigned long long>();
  if (st) memset(st, 0, sizeof *st);
  const uint64_t at = cc ? NOWHERE : number_of(g, src);
  g.last_algo = algo;
  g.lone = !cc && at == NOWHERE ? src : NOWHERE;
  WideArgs a;
  memset(&a, 0, sizeof a);
  a.uid = g.d_uid.as<uint64_t>();
  a.loff = g.d_loff.as<uint64_t>();
  a.eptr = g.d_eptr.as<uint64_t>();
  a.k = g.k;
  a.none = none;
  a.rec = g.rec;
  a.seg_shift = g.seg_shift;
  a.val = g.val.as<uint64_t>();
  a.stamp = algo == THV_ALGO_BFS ? nullptr : g.stamp.as<uint32_t>();
  unsigned long long *qn[2] = {ctr + CTR_Q, ctr + CTR_Q + 16};
  a.edges = ctr + CTR_EDGES;
  a.found = ctr + CTR_FOUND;
  a.nq = g.q[0].as<uint64_t>();
  a.nqn = qn[0];
  hipLaunchKernelGGL(k_wide_init, dim3(grid_of(g.N, 8 * g.cus)), dim3(WBS), 0, s, a, g.N, cc, at,
                     ctr, CTR_EDGES + (uint32_t)g.cus);
  if (cc) {
    const int grid = (int)std::max<uint64_t>(1, std::min<uint64_t>(div_up(g.k, XBS), g.cus));
    hipLaunchKernelGGL(k_wide_all, dim3(grid), dim3(XBS), 0, s, a);
  }
  HIPC(hipGetLastError());
  HIPC(hipStreamSynchronize(s));
  const uint64_t t0 = now_ns();
  int cur = 0;
  uint64_t levels = 0;
  // the first queue's items, for its grid (an upper bound will do)
  uint64_t items = cc ? g.k + (g.m >> g.seg_shift)
                      : at < g.k ? div_up(g.h_loff[at + 1] - g.h_loff[at], 1ull << g.seg_shift) : 0;
  for (uint64_t L = 0;; L++) {
    levels++;
    if (!items) break;  // vertices without lists: a level that finds nothing
    a.q = g.q[cur].as<uint64_t>();
    a.qn = qn[cur];
    a.nq = g.q[cur ^ 1].as<uint64_t>();
    a.nqn = qn[cur ^ 1];
    a.level_value = L + 2;
    a.level = (uint32_t)(L + 1);
    if (algo == THV_ALGO_BFS) launch_wide<THV_ALGO_BFS>(g, a, items, s);
    else if (cc) launch_wide<THV_ALGO_CC>(g, a, items, s);
    else launch_wide<THV_ALGO_SSSP>(g, a, items, s);
    hipLaunchKernelGGL(k_wide_end, dim3(1), dim3(1), 0, s, qn[cur], qn[cur ^ 1], a.found,
                       g.h_ctr_dev);
    HIPC(hipGetLastError());
    HIPC(hipStreamSynchronize(s));
    items = g.h_ctr[0];
    if (!g.h_ctr[1]) break;
    cur ^= 1;
  }
  const double ms = (now_ns() - t0) * 1e-6;
  uint64_t dg[3] = {0, 0, 0}, edges = 0;
  if (st) {
    std::vector<unsigned long long> e(g.cus);
    HIPC(hipMemcpyAsync(e.data(), ctr + CTR_EDGES, e.size() * 8, hipMemcpyDeviceToHost, s));
    HIPC(hipStreamSynchronize(s));
    for (unsigned long long x : e) edges += x;
  }
  if (digest3 || st) {
    if (g.N)
      hipLaunchKernelGGL(k_wide_digest, dim3(grid_of(g.N, 2 * g.cus)), dim3(WBS), 0, s,
                         g.val.as<uint64_t>(), g.d_uid.as<uint64_t>(), g.N,
                         cc ? UINT64_MAX : none, cc, ctr + CTR_DIGEST);
    if (cc && digest3)
      hipLaunchKernelGGL(k_wide_own, dim3(grid_of(g.n, 8 * g.cus)), dim3(WBS), 0, s, g.n, ctr + CTR_DIGEST);
    HIPC(hipGetLastError());
    HIPC(hipMemcpyAsync(g.h_ctr + 4, ctr + CTR_DIGEST, 3 * 8, hipMemcpyDeviceToHost, s));
    HIPC(hipStreamSynchronize(s));
    memcpy(dg, g.h_ctr + 4, sizeof dg);
    if (cc) {  // every vertex has a label; one without a number its own
      dg[1] = g.n;
      uint64_t v = g.n;
      auto i = g.h_ids.size(), j = g.h_extra.size();
      while (v-- > 0) {  // the largest id that has no number
        if (i && g.h_ids[i - 1] == v) i--;
        else if (j && g.h_extra[j - 1] == v) j--;
        else break;
      }
      if (v != UINT64_MAX) dg[2] = std::max(dg[2], v);
    } else if (g.lone != NOWHERE) {
      dg[0] += mix64(mix64(g.lone) + 1);
      dg[1] += 1;
      dg[2] = std::max<uint64_t>(dg[2], 1);
    }
  }
  if (digest3) memcpy(digest3, dg, sizeof dg);
  if (out) dense_values(g, out);
  if (st) {
    st->ms = ms;
    st->iterations = (uint32_t)levels;
    st->edges_traversed = edges;
    st->edges_examined = edges;
    st->reached = dg[1];
    st->expand_launches = (uint32_t)levels;
  }
}

void wide_gather(Graph64 &g, const uint64_t *at, uint64_t k, uint64_t *out) {
  if (g.last_algo < 0) fail(THV_ESTATE, "no values yet: run an algorithm first");
  for (uint64_t i = 0; i < k; i++)
    if (at[i] >= g.n) fail(THV_EINVAL, "vertex out of range");
  if (k == 0) return;
  // a buffer of up to 2^20 ids and values stays with the graph
  constexpr uint64_t KEEP = 1ull << 20;
  DevMem own;
  DevMem &d = k <= KEEP ? g.at : own;
  if (d.bytes < k * 16) d.alloc(k * 16);
  uint64_t *d_at = d.as<uint64_t>(), *d_out = d_at + k;
  HIPC(hipMemcpy(d_at, at, k * 8, hipMemcpyHostToDevice));
  hipLaunchKernelGGL(k_wide_gather, dim3(grid_of(k, 16 * g.cus)), dim3(WBS), 0, g.stream,
                     g.val.as<uint64_t>(), g.d_uid.as<uint64_t>(), g.k, g.N,
                     g.last_algo == THV_ALGO_CC, g.n + 1, g.lone, d_at, k, d_out);
  HIPC(hipGetLastError());
  HIPC(hipStreamSynchronize(g.stream));
  HIPC(hipMemcpy(out, d_out, k * 8, hipMemcpyDeviceToHost));
}

}  // namespace thv
