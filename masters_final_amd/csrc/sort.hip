// Stable LSD radix sort of 32/64-bit unsigned keys with optional 32/64-bit
// values, 8 bits per pass.
//
// Used for the canonical (weight, min, max) order of forest edges in the
// lifetime cuts (the reference sorts MST weights with numpy's unstable
// argsort, MyML/MyML/EAC/eac.py:232 and MyML/MyML/graph/singlelink.py:27),
// for the row order of graphs rebuilt from edge lists
// (MyML/MyML/graph/build.py:49-93) and for per-graph grouping in the batched
// single-link path.
//
// Per pass: (1) per-tile digit histograms (digit-major table), (2) one
// exclusive scan of the table gives every (digit, tile) its output offset,
// (3) each tile ranks its keys stably and scatters them. A wavefront takes
// consecutive keys of its tile, all loaded before the first is ranked; the
// rank among the wavefront's earlier keys is a match mask built from 8 ballots
// (peers with the same digit) and its own LDS counters, so the tile meets only
// to add up its wavefronts' counts. The tile grows with the count so that the
// table stays within one launch of the scan (up to a million keys). 925,000
// 64-bit keys, a pass: 6 + 6 + 14 us (before, with a barrier per 256 keys and
// two scan launches: 7 + 11 + 16), bound by the launches' latency and the
// scattered writes; 30,000 keys: 4 + 5 + 5 (5 + 5 + 12).
//
// A few thousand keys are placed by their ranks instead (k_rank_sort).
#include "prims.hpp"
#include "sort.hpp"

namespace eac {
namespace {

constexpr int kRadix = 256;

// Keys per tile: threads and keys a thread.
struct RadixTile {
  int rb, ri;
};
inline RadixTile radix_tile(int64_t n) {
  if (n <= 128 * 1024) return {256, 4};
  if (n <= 128 * 2048) return {256, 8};
  if (n <= 128 * 4096) return {256, 16};
  return {512, 16};
}
inline int64_t radix_tiles(int64_t n) {
  const RadixTile t = radix_tile(n);
  return (n + t.rb * t.ri - 1) / (t.rb * t.ri);
}

template <typename K>
__device__ __forceinline__ uint32_t digit_of(K k, int shift) {
  return (uint32_t)((k >> shift) & (K)0xff);
}

template <typename K, int RB, int RI>
__global__ __launch_bounds__(RB) void k_hist(const K* __restrict__ keys, int64_t n, int shift,
                                             int32_t ntiles, int32_t* __restrict__ table) {
  __shared__ int32_t h[kRadix];
  const int t = threadIdx.x;
  K key[RI];
  const int64_t base = (int64_t)blockIdx.x * (RB * RI);
#pragma unroll
  for (int j = 0; j < RI; ++j) {
    const int64_t i = base + j * RB + t;
    key[j] = i < n ? keys[i] : (K)0;
  }
  if (t < kRadix) h[t] = 0;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < RI; ++j)
    if (base + j * RB + t < n) atomicAdd(&h[digit_of(key[j], shift)], 1);
  __syncthreads();
  if (t < kRadix) table[(int64_t)t * ntiles + blockIdx.x] = h[t];
}

template <typename K, typename V, bool HAS_V, int RB, int RI>
__global__ __launch_bounds__(RB) void k_scatter(const K* __restrict__ kin,
                                                const V* __restrict__ vin, K* __restrict__ kout,
                                                V* __restrict__ vout, int64_t n, int shift,
                                                int32_t ntiles,
                                                const int32_t* __restrict__ offs) {
  constexpr int NW = RB / kWave;
  __shared__ int32_t s_cnt[NW][kRadix];  // a wavefront's keys of a digit so far
  const int t = threadIdx.x, w = t / kWave, l = lane_id();
  const int64_t base = (int64_t)blockIdx.x * (RB * RI) + (int64_t)w * (kWave * RI) + l;
  K key[RI];
  V val[HAS_V ? RI : 1];
#pragma unroll
  for (int j = 0; j < RI; ++j) {
    const int64_t i = base + j * kWave;
    key[j] = i < n ? kin[i] : (K)0;
    if (HAS_V && i < n) val[j] = vin[i];
  }
  int32_t off = t < kRadix ? offs[(int64_t)t * ntiles + blockIdx.x] : 0;
  volatile int32_t* const mine = s_cnt[w];
#pragma unroll
  for (int q = 0; q < kRadix / kWave; ++q) mine[q * kWave + l] = 0;
  const uint64_t lt = lanemask_lt();
  int32_t pos[RI];
#pragma unroll
  for (int j = 0; j < RI; ++j) {
    const bool valid = base + j * kWave < n;
    const uint32_t d = digit_of(key[j], shift);
    uint64_t peers = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const uint64_t bal = __ballot((d >> b) & 1u);
      peers &= ((d >> b) & 1u) ? bal : ~bal;
    }
    const int rank = __popcll(peers & lt);
    // (one wavefront's LDS accesses keep their order)
    const int32_t before = mine[d];
    pos[j] = before + rank;
    if (valid && rank == 0) mine[d] = before + __popcll(peers);
  }
  __syncthreads();
  if (t < kRadix) {  // the tile's offset of the digit, then every wavefront's
#pragma unroll
    for (int ww = 0; ww < NW; ++ww) {
      const int32_t c = s_cnt[ww][t];
      s_cnt[ww][t] = off;
      off += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < RI; ++j) {
    if (base + j * kWave >= n) continue;
    const int64_t o = (int64_t)s_cnt[w][digit_of(key[j], shift)] + pos[j];
    kout[o] = key[j];
    if (HAS_V) vout[o] = val[j];
  }
}

// Stable placement by rank: a workgroup takes 64 keys, one a lane, and every
// wavefront counts the keys before them among a sixteenth of all, which it
// reads as scalars: smaller ones, and equal ones that come earlier. n^2
// comparisons in one launch: 8,000 64-bit keys 22 us, where every pass of the
// radix sort takes three launches and 14 us at these counts. So it is used
// while n^2 <= 4e7 per pass.
constexpr int64_t kRankN = 16384;
inline bool rank_fits(int64_t n, int passes) {
  return n <= kRankN && n * n <= (int64_t)40000000 * passes;
}
template <typename K, typename V, bool HAS_V>
__global__ __launch_bounds__(1024) void k_rank_sort(const K* __restrict__ kin,
                                                    const V* __restrict__ vin,
                                                    K* __restrict__ kout, V* __restrict__ vout,
                                                    int64_t n, int begin, int end) {
  __shared__ int32_t s_rank[kWave];
  const int l = lane_id(), w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int i0 = blockIdx.x * kWave, i = i0 + l, m = (int)n;
  constexpr int kBits = 8 * sizeof(K);
  // the bits [begin, end) in order: the others shifted out
  const int up = kBits - end, down = kBits - end + begin;
  auto word = [&](K k) { return (K)((K)(k << up) >> down); };
  const K own = i < m ? kin[i] : (K)0;
  const K k = word(own);
  if (threadIdx.x < kWave) s_rank[threadIdx.x] = 0;
  __syncthreads();
  const int per = (m + 15) / 16, a = w * per, b = a + per < m ? a + per : m;
  int32_t rank = 0;
  const int b1 = b < i0 ? b : i0, a3 = a > i0 + kWave ? a : i0 + kWave;
#pragma unroll 8
  for (int j = a; j < b1; ++j) rank += word(kin[j]) <= k;
  for (int j = a > i0 ? a : i0; j < b && j < i0 + kWave; ++j) {
    const K o = word(kin[j]);
    rank += o < k || (o == k && j < i);
  }
#pragma unroll 8
  for (int j = a3; j < b; ++j) rank += word(kin[j]) < k;
  atomicAdd(&s_rank[l], rank);
  __syncthreads();
  if (w == 0 && i < m) {
    kout[s_rank[l]] = own;
    if (HAS_V) vout[s_rank[l]] = vin[i];
  }
}

template <typename T>
__global__ void k_copy(const T* __restrict__ a, T* __restrict__ b, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    b[i] = a[i];
}

}  // namespace

// Table entries of any count up to n (a sort may be smaller than its
// workspace's count, and smaller counts have smaller tiles).
static size_t radix_table(int64_t n) {
  int64_t most = 0;
  for (int64_t top : {(int64_t)128 * 1024, (int64_t)128 * 2048, (int64_t)128 * 4096, n}) {
    const int64_t t = radix_tiles(top < n ? top : n);
    most = t > most ? t : most;
  }
  return (size_t)most * kRadix;
}

size_t radix_sort_ws_bytes(int64_t n, int key_bytes, int val_bytes) {
  const size_t table = radix_table(n);
  Arena ar(nullptr, 0, true);
  ar.take<char>((size_t)n * key_bytes);
  if (val_bytes) ar.take<char>((size_t)n * val_bytes);
  ar.take<int32_t>(table);
  return ar.used + scan_ws_bytes((int64_t)table, 4) + 1024;
}

template <typename K, typename V, int RB, int RI>
static int radix_pass(const K* kin, const V* vin, K* kout, V* vout, int64_t n, int shift,
                      int32_t ntiles, int32_t* table, Arena& ar, hipStream_t s) {
  constexpr bool HAS_V = !std::is_same<V, NoValue>::value;
  const size_t mark = ar.used;  // each pass's scan reuses the same scratch
  k_hist<K, RB, RI><<<ntiles, RB, 0, s>>>(kin, n, shift, ntiles, table);
  EAC_LAUNCH_CHECK();
  EAC_TRY((scan_excl<int32_t, int32_t>(table, table, (int64_t)ntiles * kRadix, 0, nullptr, ar,
                                       s)));
  ar.used = mark;
  k_scatter<K, V, HAS_V, RB, RI><<<ntiles, RB, 0, s>>>(kin, vin, kout, vout, n, shift, ntiles,
                                                       table);
  EAC_LAUNCH_CHECK();
  return EAC_OK;
}

template <typename K, typename V>
int radix_sort(const K* kin, K* kout, const V* vin, V* vout, int64_t n, int begin_bit,
               int end_bit, Arena& ar, hipStream_t s) {
  constexpr bool HAS_V = !std::is_same<V, NoValue>::value;
  if (n <= 0) return EAC_OK;
  if (begin_bit < 0 || end_bit > (int)(8 * sizeof(K)) || begin_bit > end_bit)
    return fail(EAC_ERR_ARG, "radix_sort: bad bit range");
  const int64_t ntiles64 = radix_tiles(n);
  if (ntiles64 * kRadix > INT32_MAX) return fail(EAC_ERR_ARG, "radix_sort: too many keys");
  const int32_t ntiles = (int32_t)ntiles64;
  K* kbuf = ar.take<K>(n);
  V* vbuf = HAS_V ? ar.take<V>(n) : nullptr;
  int32_t* table = ar.take<int32_t>((size_t)ntiles * kRadix);
  if (ar.overflow()) return fail(EAC_ERR_WORKSPACE, "radix_sort: workspace too small");
  int passes = (end_bit - begin_bit + 7) / 8;
  if (passes == 0) {
    if (kout != kin) {
      k_copy<K><<<grid_for(n, 256, 4096), 256, 0, s>>>(kin, kout, n);
      EAC_LAUNCH_CHECK();
    }
    if (HAS_V && vout != vin) {
      k_copy<V><<<grid_for(n, 256, 4096), 256, 0, s>>>(vin, vout, n);
      EAC_LAUNCH_CHECK();
    }
    return EAC_OK;
  }
  if (rank_fits(n, passes)) {
    // (a last digit may reach past end_bit: the radix passes sort by it too)
    const int top = begin_bit + 8 * passes;
    k_rank_sort<K, V, HAS_V><<<grid_for(n, kWave), 1024, 0, s>>>(
        kin, vin, kout, vout, n, begin_bit, top < (int)(8 * sizeof(K)) ? top : 8 * (int)sizeof(K));
    EAC_LAUNCH_CHECK();
    return EAC_OK;
  }
  // ping-pong so that the last pass writes kout/vout
  const K* src_k = kin;
  const V* src_v = vin;
  const RadixTile tile = radix_tile(n);
  for (int p = 0; p < passes; ++p) {
    const int shift = begin_bit + 8 * p;
    const bool to_out = ((passes - 1 - p) % 2) == 0;
    K* dk = to_out ? kout : kbuf;
    V* dv = to_out ? vout : vbuf;
    if (tile.rb == 512)
      EAC_TRY((radix_pass<K, V, 512, 16>(src_k, src_v, dk, dv, n, shift, ntiles, table, ar, s)));
    else if (tile.ri == 16)
      EAC_TRY((radix_pass<K, V, 256, 16>(src_k, src_v, dk, dv, n, shift, ntiles, table, ar, s)));
    else if (tile.ri == 8)
      EAC_TRY((radix_pass<K, V, 256, 8>(src_k, src_v, dk, dv, n, shift, ntiles, table, ar, s)));
    else
      EAC_TRY((radix_pass<K, V, 256, 4>(src_k, src_v, dk, dv, n, shift, ntiles, table, ar, s)));
    src_k = dk;
    src_v = dv;
  }
  return EAC_OK;
}

template int radix_sort<uint64_t, NoValue>(const uint64_t*, uint64_t*, const NoValue*, NoValue*,
                                           int64_t, int, int, Arena&, hipStream_t);
template int radix_sort<uint32_t, NoValue>(const uint32_t*, uint32_t*, const NoValue*, NoValue*,
                                           int64_t, int, int, Arena&, hipStream_t);
template int radix_sort<uint32_t, uint32_t>(const uint32_t*, uint32_t*, const uint32_t*,
                                            uint32_t*, int64_t, int, int, Arena&, hipStream_t);
template int radix_sort<uint32_t, uint64_t>(const uint32_t*, uint32_t*, const uint64_t*,
                                            uint64_t*, int64_t, int, int, Arena&, hipStream_t);
template int radix_sort<uint64_t, uint32_t>(const uint64_t*, uint64_t*, const uint32_t*,
                                            uint32_t*, int64_t, int, int, Arena&, hipStream_t);

}  // namespace eac

// ------------------------------------------------------------------ C ABI
extern "C" size_t eac_sort_workspace_bytes(int64_t n, int32_t key_bytes, int32_t val_bytes) {
  return eac::radix_sort_ws_bytes(n < 1 ? 1 : n, key_bytes, val_bytes);
}

extern "C" int eac_radix_sort_u64(const uint64_t* keys_in, uint64_t* keys_out,
                                  const uint32_t* vals_in, uint32_t* vals_out, int64_t n,
                                  int32_t begin_bit, int32_t end_bit, void* ws, size_t ws_bytes,
                                  void* stream) {
  if (n < 0) return eac::fail(EAC_ERR_ARG, "sort: negative length");
  if (n == 0) return EAC_OK;
  if (!keys_in || !keys_out || (!vals_in) != (!vals_out))
    return eac::fail(EAC_ERR_ARG, "sort: null array");
  size_t need = eac::radix_sort_ws_bytes(n, 8, vals_in ? 4 : 0);
  if (!ws || ws_bytes < need)
    return eac::fail(EAC_ERR_WORKSPACE, "sort: workspace %zu < %zu bytes", ws_bytes, need);
  eac::Arena ar(ws, ws_bytes);
  hipStream_t s = (hipStream_t)stream;
  if (vals_in)
    return eac::radix_sort<uint64_t, uint32_t>(keys_in, keys_out, vals_in, vals_out, n,
                                               begin_bit, end_bit, ar, s);
  return eac::radix_sort<uint64_t, eac::NoValue>(keys_in, keys_out, nullptr, nullptr, n,
                                                 begin_bit, end_bit, ar, s);
}
