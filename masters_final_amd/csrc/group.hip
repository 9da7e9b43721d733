// Stable grouping of ensemble labels by cluster on gfx950: the member lists
// of the K-Means centroid update (KMeans.py:709-754 sums a cluster's points
// in point order) and of the co-association plan.
//
// Labels of a partition only meet clusters of that partition, so one counting
// sort per partition takes the place of radix passes over (cluster, point)
// pairs, up to some thousand clusters a partition (radix_items):
//  * histogram: one workgroup per (chunk of points, partition) counts its
//    labels in LDS and writes a column of the table T[cluster][chunk];
//  * one exclusive scan of T in (cluster, chunk) order gives every chunk its
//    first output position in every cluster;
//  * placement: one wavefront per (chunk, partition) walks its points in
//    order, 64 at a time, with the clusters' next positions in LDS. Lanes of
//    one step with the same label are ranked by a match mask (one ballot per
//    label bit), so the order inside a cluster is the point order.
// The labels are read twice and the ids written once; the table is at most a
// quarter of the labels. Bound by the placement: its 4-byte stores land on as
// many lines as there are clusters, and its LDS chain (a read and a write of
// the next positions per 64 points) is spread over a few thousand wavefronts.
// 500,000 points x 16 partitions (16,600 clusters): histogram 29, scan 13,
// placement 100 us (0.08 G points/us), against 0.85 ms for keys with global
// counts and two 8-bit radix passes of (cluster, point) pairs; 10,000 x 100:
// 25 us against 110.
#include "group.hpp"

#include "prims.hpp"
#include "sort.hpp"

namespace eac {
namespace {

constexpr int kGH = 256;       // histogram threads
constexpr int kGRange = 4096;  // clusters per LDS table; more take further grid layers

// Chunk b = blockIdx.x of partition p = blockIdx.y, clusters [z * kGRange, ...)
// of it: T[(k_off[p] + c) * nch + b] = labels c of the chunk.
__global__ __launch_bounds__(kGH) void k_group_hist(const int32_t* __restrict__ labels, int64_t n,
                                                    int P, const int64_t* __restrict__ k_off,
                                                    int64_t chunk, int64_t nch,
                                                    int32_t* __restrict__ T, int64_t last,
                                                    unsigned int* __restrict__ bad) {
  extern __shared__ int32_t s_dyn[];
  int32_t* const s_g = s_dyn;
  const int64_t i0 = (int64_t)blockIdx.x * chunk;
  const int64_t i1 = i0 + chunk < n ? i0 + chunk : n;
  const int32_t z0 = (int32_t)blockIdx.z * kGRange;
  if (blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0 && threadIdx.x == 0) T[last] = 0;
  for (int p = blockIdx.y; p < P; p += gridDim.y) {
    const int64_t kb = k_off[p];
    const int32_t k = (int32_t)(k_off[p + 1] - kb);
    const int32_t kz = k - z0 < kGRange ? k - z0 : kGRange;
    if (kz <= 0 && !(k <= 0 && z0 == 0)) continue;  // uniform over the block
    for (int c = threadIdx.x; c < kz; c += kGH) s_g[c] = 0;
    __syncthreads();
    const int32_t* lp = labels + (int64_t)p * n;
    for (int64_t i = i0 + threadIdx.x; i < i1; i += kGH) {
      const int32_t l = lp[i];
      if (l >= k) {
        if (bad && z0 == 0) atomicOr(bad, 1u);
      } else if (l >= z0 && l - z0 < kz) {
        atomicAdd(&s_g[l - z0], 1);
      }
    }
    __syncthreads();
    for (int c = threadIdx.x; c < kz; c += kGH)
      T[(kb + z0 + c) * nch + blockIdx.x] = s_g[c];
    __syncthreads();
  }
}

// Places chunk blockIdx.x of partition blockIdx.y; the first chunk's wave also
// writes the clusters' starts.
__global__ __launch_bounds__(kWave) void k_group_place(
    const int32_t* __restrict__ labels, int64_t n, int P, const int64_t* __restrict__ k_off,
    int64_t chunk, int64_t nch, const int32_t* __restrict__ T, int64_t last,
    uint32_t* __restrict__ members, uint32_t* __restrict__ start, int32_t* __restrict__ pos) {
  extern __shared__ int32_t s_dyn[];
  // next position of each cluster: lanes read what other lanes of the wavefront
  // wrote a step before, so every access is made, in order
  volatile int32_t* const s_g = s_dyn;
  const int ln = threadIdx.x;
  const int64_t i0 = (int64_t)blockIdx.x * chunk;
  const int64_t i1 = i0 + chunk < n ? i0 + chunk : n;
  const int32_t z0 = (int32_t)blockIdx.z * kGRange;
  const uint64_t lt = lanemask_lt();
  if (blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0 && ln == 0)
    start[k_off[P]] = (uint32_t)T[last];
  for (int p = blockIdx.y; p < P; p += gridDim.y) {
    const int64_t kb = k_off[p];
    const int32_t k = (int32_t)(k_off[p + 1] - kb);
    const int32_t kz = k - z0 < kGRange ? k - z0 : kGRange;
    if (kz <= 0 && z0 > 0) continue;
    __syncthreads();
    for (int c = ln; c < kz; c += kWave) {
      const int32_t at = T[(kb + z0 + c) * nch + blockIdx.x];
      s_g[c] = at;
      if (blockIdx.x == 0) start[kb + z0 + c] = (uint32_t)at;
    }
    __syncthreads();
    int bits = 0;
    while ((kz - 1) >> bits > 0) ++bits;
    const int32_t* lp = labels + (int64_t)p * n;
    int32_t* pp = pos ? pos + (int64_t)p * n : nullptr;
    constexpr int U = 4;  // label loads in flight
    for (int64_t b = i0; b < i1; b += U * kWave) {
      int32_t lab[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t i = b + u * kWave + ln;
        lab[u] = i < i1 ? lp[i] : -1;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t i = b + u * kWave + ln;
        const bool valid = lab[u] >= z0 && lab[u] < k && lab[u] - z0 < kz;
        const uint32_t c = (uint32_t)(lab[u] - z0);
        uint64_t peers = __ballot(valid);
        for (int q = 0; q < bits; ++q) {
          const bool one = (c >> q) & 1u;
          const uint64_t bal = __ballot(one);
          peers &= one ? bal : ~bal;
        }
        uint32_t at = 0;
        if (valid) {
          const int rank = __popcll(peers & lt);
          at = (uint32_t)s_g[c] + rank;
          // the lane ranked last moves the cluster's position on (the reads
          // of this step come first: one wavefront's LDS operations complete
          // in the order they are made)
          if ((peers >> ln) == 1ull) s_g[c] = (int32_t)at + 1;
          members[at] = (uint32_t)i;
        }
        if (pp && i < i1 && (valid || (z0 == 0 && (lab[u] < 0 || lab[u] >= k))))
          pp[i] = valid ? (int32_t)at : -1;
      }
    }
  }
}

// ---- many clusters a partition: the radix sort of (cluster, point).
// key: global cluster, ktot for points left out (sorted last); value: p * n + i.
__global__ void k_group_keys(const int32_t* __restrict__ labels, int64_t n, int P,
                             const int64_t* __restrict__ k_off, uint32_t* __restrict__ key,
                             uint32_t* __restrict__ val, unsigned int* __restrict__ bad) {
  const uint32_t ktot = (uint32_t)k_off[P];
  for (int p = blockIdx.y; p < P; p += gridDim.y) {
    const int64_t kb = k_off[p], k = k_off[p + 1] - kb;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
      const int64_t t = (int64_t)p * n + i;
      const int32_t l = labels[t];
      if (l >= k && bad) atomicOr(bad, 1u);
      key[t] = l < 0 || l >= k ? ktot : (uint32_t)(kb + l);
      val[t] = (uint32_t)t;
    }
  }
}
// start[c] = the first sorted key that is at least c.
__global__ void k_group_starts(const uint32_t* __restrict__ skey, int64_t items, int64_t ktot,
                               uint32_t* __restrict__ start) {
  for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c <= ktot;
       c += (int64_t)gridDim.x * blockDim.x) {
    int64_t lo = 0, hi = items;
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if (skey[mid] < (uint64_t)c) lo = mid + 1; else hi = mid;
    }
    start[c] = (uint32_t)lo;
  }
}
// sorted values (members, in place) to point ids and positions.
__global__ void k_group_members(const uint32_t* __restrict__ skey, int64_t items, uint32_t n,
                                uint32_t ktot, uint32_t* __restrict__ members,
                                int32_t* __restrict__ pos) {
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < items;
       q += (int64_t)gridDim.x * blockDim.x) {
    const uint32_t v = members[q];
    members[q] = v % n;
    if (pos) pos[v] = skey[q] < ktot ? (int32_t)q : -1;
  }
}

}  // namespace

GroupShape group_shape(int64_t n, int P, int64_t ktot) {
  // at least 512 points a wavefront, a table of at most a quarter of the
  // labels, and about 8192 wavefronts in all
  GroupShape g;
  const int64_t items = (int64_t)P * n;
  g.chunk = 512;
  if (g.chunk < 4 * ktot / P) g.chunk = 4 * ktot / P;
  if (g.chunk < items / 8192) g.chunk = items / 8192;
  g.chunk = (g.chunk + kWave - 1) / kWave * kWave;
  g.nch = (n + g.chunk - 1) / g.chunk;
  g.table = ktot * g.nch + 1;
  return g;
}

// The most labels that ktot clusters in P partitions are sorted by radix
// passes for (0: none). A chunk of the counting sort has at least four times as
// many points as its table has clusters, and one wavefront walks it: 0.044 us
// a cluster, beside 40 us and 1e-5 us a label that the radix passes cost more.
// One partition of 100,000 points, a whole centroid update: 1000 clusters 91 us
// by counting and 84 by radix, 24,000 1069 and 91; 16 partitions of 1,000,000:
// 4000 483 and 604, 12,000 855 and 758.
static int64_t radix_items(int P, int64_t ktot) {
  const int64_t over = ktot / P - 800;
  if (over <= 0 || ktot >= INT32_MAX) return 0;
  return over < INT32_MAX / 2200 ? over * 2200 : INT32_MAX;
}

size_t group_ws_bytes(int64_t n, int P, int64_t ktot) {
  const GroupShape g = group_shape(n, P, ktot);
  Arena ar(nullptr, 0, true);
  ar.take<int32_t>(g.table);
  const size_t counting = ar.used + scan_ws_bytes(g.table, 4) + 256;
  // (a workspace also serves fewer points, which may take the radix passes)
  const int64_t most = radix_items(P, ktot), items = (int64_t)P * n < most ? (int64_t)P * n : most;
  if (items <= 0) return counting;
  Arena rar(nullptr, 0, true);
  for (int q = 0; q < 3; ++q) rar.take<uint32_t>(items);
  const size_t radix = rar.used + radix_sort_ws_bytes(items, 4, 4) + 256;
  return radix > counting ? radix : counting;
}

int group_by_cluster(const int32_t* labels, int64_t n, int P, const int64_t* d_koff,
                     const int64_t* h_koff, uint32_t* members, uint32_t* start, int32_t* pos,
                     unsigned int* bad, Arena& ar, hipStream_t s) {
  const int64_t ktot = h_koff[P];
  const int64_t items = (int64_t)P * n;
  if (items <= radix_items(P, ktot)) {
    uint32_t* key = ar.take<uint32_t>(items);
    uint32_t* val = ar.take<uint32_t>(items);
    uint32_t* skey = ar.take<uint32_t>(items);
    if (ar.overflow()) return fail(EAC_ERR_WORKSPACE, "group: workspace too small");
    const int py = P < 65535 ? P : 65535;
    k_group_keys<<<dim3(grid_for(n, 256 * 4, 4096), py), 256, 0, s>>>(labels, n, P, d_koff, key,
                                                                      val, bad);
    EAC_LAUNCH_CHECK();
    EAC_TRY((radix_sort<uint32_t, uint32_t>(key, skey, val, members, items, 0,
                                            bits_for((uint64_t)ktot), ar, s)));
    k_group_starts<<<grid_for(ktot + 1, 256, 4096), 256, 0, s>>>(skey, items, ktot, start);
    EAC_LAUNCH_CHECK();
    k_group_members<<<grid_for(items, 256 * 4, 8192), 256, 0, s>>>(
        skey, items, (uint32_t)n, (uint32_t)ktot, members, pos);
    EAC_LAUNCH_CHECK();
    return EAC_OK;
  }
  const GroupShape g = group_shape(n, P, ktot);
  if (g.nch > INT32_MAX || g.table >= (int64_t)INT32_MAX * 4)
    return fail(EAC_ERR_UNSUPPORTED, "group: too many labels");
  int64_t kmax = 1;
  for (int p = 0; p < P; ++p)
    if (h_koff[p + 1] - h_koff[p] > kmax) kmax = h_koff[p + 1] - h_koff[p];
  const int64_t layers = (kmax + kGRange - 1) / kGRange;
  if (layers > 65535) return fail(EAC_ERR_UNSUPPORTED, "group: a partition of too many clusters");
  int32_t* T = ar.take<int32_t>(g.table);
  if (ar.overflow()) return fail(EAC_ERR_WORKSPACE, "group: workspace too small");
  const dim3 grid((unsigned)g.nch, P < 65535 ? P : 65535, (unsigned)layers);
  const size_t lds = (size_t)(kmax < kGRange ? kmax : kGRange) * sizeof(int32_t);
  k_group_hist<<<grid, kGH, lds, s>>>(labels, n, P, d_koff, g.chunk, g.nch, T, g.table - 1, bad);
  EAC_LAUNCH_CHECK();
  EAC_TRY((scan_excl<int32_t, int32_t>(T, T, g.table, 0, nullptr, ar, s)));
  k_group_place<<<grid, kWave, lds, s>>>(labels, n, P, d_koff, g.chunk, g.nch, T, g.table - 1,
                                         members, start, pos);
  EAC_LAUNCH_CHECK();
  return EAC_OK;
}

}  // namespace eac
