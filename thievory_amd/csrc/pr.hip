// pr.hip -- PageRank's edge kernels and the push mode's hub table.
//
// Reference: PR32_PUSH's and PR32's edge kernels (src/pr/pr_kernels.cu:
// 539-542 atomicAdd(res[w], delta[v]); 45-51 sum[v] += contrib[u]).
//
// Both walk the level's work space (chunk.hpp), host and HBM chunks
// interleaved.  Push takes chunks of PR_CHUNK edges, one wave per chunk: the
// wave stages the chunk's queue entries in its own slice of LDS, marks their
// starts in a bit mask and finds each edge's entry by a popcount rank, eight
// edges per lane in flight.  Waves share nothing but the hub sums, so there
// is no barrier in the loop.
#include <algorithm>

#include "chunk.hpp"

namespace thv {

namespace {

constexpr uint32_t PC = PR_CHUNK;
constexpr uint32_t PE = PC / 64;  // edges per lane
constexpr uint32_t PW = PC / 32;  // mask words

// Orders this wave's LDS accesses: lanes read what other lanes wrote.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A wave's staging area: NE entries at a time (a chunk with more, which
// needs lists of fewer than PC / NE records on average, takes several
// windows).
template <uint32_t NE>
struct PrStage {
  unsigned long long base[NE];  // address of the entry's record for edge 0 of the work space
  float f[NE];                  // the source's delta
  uint32_t mask[PW], pre[PW];
};

// Stages entries [i, i + ne) of a chunk: starts marked, bases kept; edges
// before *lo belong to earlier windows, edges from *hi to later ones.
// Returns the entries staged.
template <int REC, uint32_t NE>
__device__ __forceinline__ void stage(const PrArgs &a, PrStage<NE> &s, const ChunkInfo &ci, int q,
                                      uint32_t first, uint32_t ne, uint32_t lane, uint32_t *lo,
                                      uint32_t *hi) {
  const uint32_t *__restrict__ qv = a.qv[q];
  const unsigned long long *__restrict__ qe = a.qe[q];
  if (lane < PW) s.mask[lane] = 0;
  wave_lds_sync();
  for (uint32_t t = lane; t < ne; t += 64) {
    const uint32_t v = qv[ci.i0 + first + t];
    const unsigned long long b = qe[ci.i0 + first + t];
    const unsigned long long r = chunk_rel(b, ci.e0);
    if (r < PC) {
      atomicOr(&s.mask[r >> 5], 1u << (r & 31));
      s.base[t] = a.eptr[v] - b * REC;
      s.f[t] = a.src[v];
    }
  }
  *lo = first ? (uint32_t)chunk_rel(qe[ci.i0 + first], ci.e0) : 0u;
  const bool more = first + ne < ci.nent;
  const unsigned long long h = more ? chunk_rel(qe[ci.i0 + first + ne], ci.e0) : ci.len;
  *hi = (uint32_t)min(h, (unsigned long long)ci.len);
  wave_lds_sync();
  const uint32_t pc = lane < PW ? __popc(s.mask[lane]) : 0u;
  uint32_t inc = pc;
#pragma unroll
  for (uint32_t d = 1; d < PW; d <<= 1) {
    const uint32_t y = __shfl_up(inc, d, 64);
    if (lane >= d) inc += y;
  }
  if (lane < PW) s.pre[lane] = inc - pc;
  wave_lds_sync();
}

// The records of the staged entries' edges: neighbour and entry of edge
// lane + 64 j, for the edges in [lo, hi); VNONE elsewhere.
constexpr uint32_t VNONE = 0xFFFFFFFFu;
template <int REC, uint32_t NE>
__device__ __forceinline__ void records(const PrStage<NE> &s, const ChunkInfo &ci, uint32_t lane,
                                        uint32_t lo, uint32_t hi, uint32_t (&nb)[PE],
                                        uint32_t (&ent)[PE]) {
#pragma unroll
  for (uint32_t j = 0; j < PE; j++) {
    const uint32_t l = j * 64 + lane;
    nb[j] = VNONE;
    ent[j] = 0;
    if (l >= lo && l < hi) {
      const uint32_t k = chunk_rank(s.mask, s.pre, l);
      ent[j] = k;
      nb[j] = *reinterpret_cast<const __attribute__((address_space(1))) uint32_t *>(
          s.base[k] + (ci.e0 + l) * REC);
    }
  }
}

// Push: an atomic add in HBM per record runs at about 11.6 G/s (2.64 ms for
// 31M edges over 2M vertices, all in HBM), whatever feeds it.  So the
// destinations that receive the most records (hubs: up to PR_HUBS, dense
// indices from a bitmap with prefix counts) are summed in LDS, one 1024-
// thread block per CU so that the table is as large as LDS allows, and
// each block adds its sums to a compact array (consecutive addresses: some
// 20 times fewer memory operations than scattered ones).  On that graph
// 32,768 hubs receive 61% of the records; 2,048, 22%.  It takes 0.77 ms, and
// with a 25% HBM budget 1.74 against 2.67: the host's 92 MB at 53 GB/s, the
// link's rate.
constexpr int PBS = 1024;
constexpr uint32_t PUSH_NE = 128;
struct PushShared {
  float acc[PR_HUBS];
  PrStage<PUSH_NE> st[PBS / 64];
};
static_assert(sizeof(PushShared) <= 160 * 1024, "one block per CU");

template <int REC>
__global__ void __launch_bounds__(PBS) k_pr_push(PrArgs a) {
  __shared__ PushShared sh;
  const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  for (uint32_t t = threadIdx.x; t < a.nhubs; t += PBS) sh.acc[t] = 0.0f;
  __syncthreads();
  PrStage<PUSH_NE> &s = sh.st[wv];
  const ChunkSrc cs = chunk_src(a.ctr, PC);
  const uint32_t nw = gridDim.x * (PBS / 64);
  for (uint32_t c = blockIdx.x * (PBS / 64) + wv; c < cs.total; c += nw) {
    int q;
    uint32_t cc;
    chunk_pick(cs, c, q, cc);
    const ChunkInfo ci = chunk_info<PC>(cs, a.qc, q, cc);
    for (uint32_t first = 0; first < ci.nent; first += PUSH_NE) {
      uint32_t lo, hi, w[PE], ent[PE];
      stage<REC>(a, s, ci, q, first, min(PUSH_NE, ci.nent - first), lane, &lo, &hi);
      records<REC>(s, ci, lane, lo, hi, w, ent);
      uint2 tab[PE];  // the destination's word of the hub bitmap and the hubs before it
#pragma unroll
      for (uint32_t j = 0; j < PE; j++) tab[j] = a.hubtab[w[j] != VNONE ? w[j] >> 5 : 0];
#pragma unroll
      for (uint32_t j = 0; j < PE; j++) {
        if (w[j] == VNONE) continue;
        const float d = s.f[ent[j]];
        const uint32_t bit = 1u << (w[j] & 31);
        if (tab[j].x & bit) atomicAdd(&sh.acc[tab[j].y + __popc(tab[j].x & (bit - 1))], d);
        else unsafeAtomicAdd(&a.dst[w[j]], d);
      }
      wave_lds_sync();
    }
  }
  __syncthreads();
  // blocks start at different places, so they seldom meet on a line
  const uint32_t turn = a.nhubs ? (uint32_t)((uint64_t)blockIdx.x * a.nhubs / gridDim.x) & ~63u : 0u;
  for (uint32_t t = threadIdx.x; t < a.nhubs; t += PBS) {
    const uint32_t i = t + turn < a.nhubs ? t + turn : t + turn - a.nhubs;
    const float x = sh.acc[i];
    if (x != 0.0f) unsafeAtomicAdd(&a.hubacc[i], x);
  }
}

// Pull: one 256-thread block per chunk of 256 EPT edges, staged as in
// expand.hip.  The gather of contributions bounds it: of 62M gathers over 4M
// vertices (16 MB of contributions) 85% miss the CU's L1 and its address
// unit is busy 78% of the time; without the gathers the kernel takes 146
// us, without the sums 375, as it is 424.  Where a wave's 64 edges all belong
// to one list its sum is made in registers: an LDS add per edge to one
// address takes a turn per lane (610 us).  More waves per CU (5, 6, 8 per
// SIMD) or a wave per chunk without barriers gather no faster (440-570 us),
// and smaller chunks split more lines of the host's lists between CUs.
constexpr int LBS = 256;

// Sum over the wave, in lane 63 (row shifts, then row broadcasts).
template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp_add(float x) {
  return x + __int_as_float(
                 __builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, ROWS, 0xf, false));
}
__device__ __forceinline__ float wave_sum63(float x) {
  x = dpp_add<0x111, 0xf>(x);
  x = dpp_add<0x112, 0xf>(x);
  x = dpp_add<0x114, 0xf>(x);
  x = dpp_add<0x118, 0xf>(x);
  x = dpp_add<0x142, 0xa>(x);
  return dpp_add<0x143, 0xc>(x);
}

template <int REC, int EPT>
__global__ void __launch_bounds__(LBS) k_pr_pull(PrArgs a) {
  constexpr uint32_t C = LBS * EPT, NW = C / 32;
  __shared__ uint32_t s_mask[NW], s_pre[NW];
  __shared__ unsigned long long s_base[C + 1];
  __shared__ uint32_t s_v[C + 1];
  __shared__ float s_f[C + 1];
  const uint32_t tid = threadIdx.x, lane = tid & 63;
  const ChunkSrc cs = chunk_src(a.ctr, C);
  for (uint32_t c = blockIdx.x; c < cs.total; c += gridDim.x) {
    int q;
    uint32_t cc;
    chunk_pick(cs, c, q, cc);
    const ChunkInfo ci = chunk_info<C>(cs, a.qc, q, cc);
    const uint32_t *__restrict__ qv = a.qv[q];
    const unsigned long long *__restrict__ qe = a.qe[q];
    for (uint32_t t = tid; t < NW; t += LBS) s_mask[t] = 0;
    __syncthreads();
    for (uint32_t t = tid; t < ci.nent; t += LBS) {
      const uint32_t v = qv[ci.i0 + t];
      const unsigned long long b = qe[ci.i0 + t];
      const unsigned long long r = chunk_rel(b, ci.e0);
      s_v[t] = VNONE;  // starts in the next chunk
      if (r < C) {
        atomicOr(&s_mask[r >> 5], 1u << (r & 31));
        s_base[t] = a.eptr[v] - b * REC;
        s_v[t] = v;
        s_f[t] = 0.0f;
      }
    }
    __syncthreads();
    chunk_prefix<NW>(s_mask, s_pre);
    __syncthreads();
    uint32_t u[EPT], ent[EPT];
#pragma unroll
    for (int j = 0; j < EPT; j++) {
      const uint32_t l = tid + j * LBS;
      u[j] = VNONE;
      ent[j] = 0;
      if (l < ci.len) {
        const uint32_t k = chunk_rank(s_mask, s_pre, l);
        ent[j] = k;
        u[j] = *reinterpret_cast<const __attribute__((address_space(1))) uint32_t *>(
            s_base[k] + (ci.e0 + l) * REC);
      }
    }
    float x[EPT];
#pragma unroll
    for (int j = 0; j < EPT; j++) x[j] = a.src[u[j] != VNONE ? u[j] : 0];
#pragma unroll
    for (int j = 0; j < EPT; j++) {
      const bool in = u[j] != VNONE;
      const uint32_t k0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)ent[j]);
      if (__all(in && ent[j] == k0)) {
        const float t = wave_sum63(x[j]);
        if (lane == 63) atomicAdd(&s_f[k0], t);
      } else if (in) {
        atomicAdd(&s_f[ent[j]], x[j]);
      }
    }
    __syncthreads();
    for (uint32_t t = tid; t < ci.nent; t += LBS) {
      const uint32_t v = s_v[t];
      if (v == VNONE) continue;
      // a list with entries on both sides in the chunk is this block's alone
      if (t > 0 && t + 1 < ci.nent) a.dst[v] = s_f[t];
      else unsafeAtomicAdd(&a.dst[v], s_f[t]);
    }
    __syncthreads();
  }
}

// ---- hub table ---------------------------------------------------------------

// Destinations of every 16th run of 16 records (a 64-byte line of 4-byte
// ones), from the host copy of the edge array.
constexpr uint32_t HUB_RUN = 16, HUB_STEP = 16;
__global__ void __launch_bounds__(256) k_hub_sample(const uint32_t *rec, uint32_t stride,
                                                    uint64_t m, uint32_t *cnt) {
  const uint64_t runs = m / HUB_RUN / HUB_STEP + 1, T = gridDim.x * 256ull;
  for (uint64_t t = blockIdx.x * 256ull + threadIdx.x; t < runs * HUB_RUN; t += T) {
    const uint64_t e = t / HUB_RUN * HUB_RUN * HUB_STEP + t % HUB_RUN;
    if (e < m) atomicAdd(&cnt[rec[e * stride]], 1u);
  }
}

// hist[c]: vertices sampled c times (the last bin: that often or more).
constexpr uint32_t HUB_BINS = 1024;
__global__ void __launch_bounds__(256) k_hub_hist(const uint32_t *cnt, uint64_t n,
                                                  uint32_t *hist) {
  __shared__ uint32_t h[HUB_BINS];
  for (uint32_t i = threadIdx.x; i < HUB_BINS; i += 256) h[i] = 0;
  __syncthreads();
  const uint64_t T = gridDim.x * 256ull;
  for (uint64_t v = blockIdx.x * 256ull + threadIdx.x; v < n; v += T) {
    const uint32_t c = cnt[v];
    if (c) atomicAdd(&h[min(c, HUB_BINS - 1)], 1u);
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < HUB_BINS; i += 256)
    if (h[i]) atomicAdd(&hist[i], h[i]);
}

// The hubs: every vertex sampled at least `all` times, and `room` of those
// sampled `some` times.  A wave takes 64 vertices; its hubs get the next
// indices (in no order).  used[0]: indices given, used[1]: room taken.
__global__ void __launch_bounds__(256) k_hub_table(const uint32_t *cnt, uint64_t n, uint32_t all,
                                                   uint32_t some, uint32_t room, uint32_t *used,
                                                   uint2 *tab, uint64_t words) {
  const uint32_t lane = threadIdx.x & 63;
  const uint64_t T = gridDim.x * 256ull;
  for (uint64_t v = blockIdx.x * 256ull + threadIdx.x; v - lane < words * 32; v += T) {
    const uint32_t c = v < n ? min(cnt[v], HUB_BINS - 1) : 0u;
    bool hub = c >= all;
    const unsigned long long bs = wave_ballot(c == some && c < all && c > 0);
    if (bs) {
      uint32_t at = 0;
      if (lane == 0) at = atomicAdd(&used[1], (uint32_t)__popcll(bs));
      at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at) + lanes_below(bs);
      if (((bs >> lane) & 1ull) && at < room) hub = true;
    }
    const unsigned long long b = wave_ballot(hub);
    uint32_t base = 0;
    if (lane == 0 && b) base = atomicAdd(&used[0], (uint32_t)__popcll(b));
    base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
    if ((lane & 31) == 0 && (v >> 5) < words) {
      const uint32_t lo = (uint32_t)b, hi = (uint32_t)(b >> 32);
      tab[v >> 5] = lane ? make_uint2(hi, base + __popc(lo)) : make_uint2(lo, base);
    }
  }
}

}  // namespace

// A sampled vertex receives 16 records on average for each time it was
// seen; the table takes the PR_HUBS most often seen ones (all vertices,
// where there are no more than that).
void ensure_pr_hubs(Graph &g) {
  if (g.hubs_built) return;
  hipStream_t s = g.stream;
  const uint64_t n = g.n, words = bitmap_words(n);
  DevMem cnt, aux;  // hist, then used[2]
  cnt.alloc((n + 1) * 4);
  aux.alloc((HUB_BINS + 2) * 4);
  uint32_t *hist = aux.as<uint32_t>(), *used = hist + HUB_BINS;
  launch_fill_u32(cnt.as<uint32_t>(), n <= PR_HUBS ? 1u : 0u, n, s);
  launch_fill_u32(hist, 0u, HUB_BINS + 2, s);
  const uint32_t grid = (uint32_t)(8 * g.cus);
  uint32_t all = 1, some = 0, room = 0, h[HUB_BINS] = {};
  if (n > PR_HUBS) {
    if (g.m)
      hipLaunchKernelGGL(k_hub_sample, dim3(grid), dim3(256), 0, s,
                         static_cast<const uint32_t *>(g.h_edges.dev), (uint32_t)g.rec / 4, g.m,
                         cnt.as<uint32_t>());
    hipLaunchKernelGGL(k_hub_hist, dim3(grid), dim3(256), 0, s, cnt.as<uint32_t>(), n, hist);
    HIPC(hipMemcpyAsync(h, hist, sizeof h, hipMemcpyDeviceToHost, s));
    HIPC(hipStreamSynchronize(s));
    uint32_t have = 0;
    all = HUB_BINS;  // more than any count: none
    while (all > 1 && have + h[all - 1] <= PR_HUBS) have += h[--all];
    some = all - 1;  // 0: every sampled vertex is in
    room = PR_HUBS - have;
  }
  g.d_hubtab.alloc(words * 8);
  g.d_hubacc.alloc(PR_HUBS * 4);
  launch_fill_u32(g.d_hubacc.as<uint32_t>(), 0u, PR_HUBS, s);
  hipLaunchKernelGGL(k_hub_table, dim3(grid), dim3(256), 0, s, cnt.as<uint32_t>(), n, all, some,
                     room, used, g.d_hubtab.as<uint2>(), words);
  HIPC(hipGetLastError());
  HIPC(hipMemcpyAsync(&g.nhubs, used, 4, hipMemcpyDeviceToHost, s));
  HIPC(hipStreamSynchronize(s));
  if (g.nhubs > PR_HUBS) fail(THV_ESTATE, "hub table overflow");
  g.hubs_built = true;
}

void launch_pr(Graph &g, bool push, const PrArgs &a, hipStream_t s) {
  if (!a.src || !a.dst || !a.ctr || (push && (!a.hubtab || !a.hubacc)))
    fail(THV_ESTATE, "PageRank launch: missing array");
  const bool r8 = g.rec == 8;
  if (push) {
    const uint64_t chunks = g.m / PC + 2;  // both queues' last chunks may be partial
    const uint32_t grid = (uint32_t)std::min<uint64_t>(div_up(chunks, PBS / 64), g.cus);
    if (r8) hipLaunchKernelGGL(k_pr_push<8>, dim3(grid), dim3(PBS), 0, s, a);
    else hipLaunchKernelGGL(k_pr_push<4>, dim3(grid), dim3(PBS), 0, s, a);
  } else {
    const uint32_t grid = (uint32_t)(g.shape.blocks_per_cu * g.cus);
    const bool e4 = g.shape.ept == 4;
    if (g.shape.ept != 4 && g.shape.ept != 8) fail(THV_EINVAL, "unsupported edges-per-thread");
    if (r8 && e4) hipLaunchKernelGGL((k_pr_pull<8, 4>), dim3(grid), dim3(LBS), 0, s, a);
    else if (r8) hipLaunchKernelGGL((k_pr_pull<8, 8>), dim3(grid), dim3(LBS), 0, s, a);
    else if (e4) hipLaunchKernelGGL((k_pr_pull<4, 4>), dim3(grid), dim3(LBS), 0, s, a);
    else hipLaunchKernelGGL((k_pr_pull<4, 8>), dim3(grid), dim3(LBS), 0, s, a);
  }
  HIPC(hipGetLastError());
}

}  // namespace thv
