// Sparse co-association matrix of an ensemble of partitions (EAC) on gfx950.
//
// Reference: MyML/MyML/EAC/sparse.py EAC_CSR (:12-304): for every partition
// and cluster, every pair of members gets +1 (update_cluster_fp_condensed
// :445-465 for the first partition, update_cluster_sorted_surgical_condensed
// :956-1040 with binary_search_interval :1069-1099 for the others); the
// condensed form keeps the upper triangle (col > row), rows sorted by column;
// _condense (:212-225, condense_eac_csr :336-349) packs the rows with a
// sequential offset sum; make_diassoc (:295-311) turns counts into
// (max + 1) - count. The reference caps each row at max_assocs and silently
// drops associations beyond it (sparse.py:501-503, :995-997); the default
// build here is exact (no cap, int64 row offsets), and a capacity-capped
// selection (eac_coassoc_cap, at the end of this file) reproduces the
// reference's lossy matrix from the exact one plus per-entry partition ranks.
//
// MI355X design:
//  * Plan: a stable counting sort by cluster (group.hip) turns labels
//    [P][n] into member lists (ascending point id per cluster) plus each
//    point's position in its list. A point's later co-members in partition p
//    are then the suffix of its cluster's list after its own position: no
//    search and no pair materialisation.
//  * Count/fill: one workgroup per row (rows handed out by atomic counters).
//    Columns are covered in windows of 16384; each window has a dense array
//    of byte counters (16 KiB of LDS, seven workgroups per compute unit; u16
//    beyond 255 partitions). Per window every partition's suffix cursor
//    advances over the members inside the window (flattened over partitions
//    so that lanes stream consecutive members), each member an LDS atomic
//    increment. The window is then read in column order: pass 1 counts
//    non-zeros (row nnz, max count), pass 2 writes (col, value) after a block
//    scan, so rows come out sorted without a per-row sort. Bound: vector
//    issue (0.6 instructions per unit and cycle, about 37 per 64 visits).
//    Byte counters and windows emitted by set bit instead of by column took
//    the whole build of 200,003 points x 64 partitions (4.6 G visits, 905 M
//    entries) from 36.8 to 10.7 ms, and of 10,000 x 100 from 0.67 to 0.51.
//  * Row offsets: exclusive scan of the per-row nnz into int64 (nnz > 2^31
//    for the large ensembles).
#include <cstring>
#include <vector>

#include "group.hpp"
#include "prims.hpp"

namespace eac {
namespace {

constexpr int kCB = 256;       // threads per row workgroup
constexpr int kWin = 32768;    // columns per LDS window (two u16 counters per u32 word)
constexpr int kMaxP = 1024;    // partitions staged in LDS
constexpr int kMaxRanges = 8;  // contiguous row ranges (one per XCD)
constexpr int kStripes = 32;   // interleaved row ranges of a small matrix
constexpr int kCtrPad = 16;    // row counters 128 bytes apart
constexpr int kCtrSum = kStripes * kCtrPad;  // after the counters: the sampled nnz sum
constexpr int kCtrs = kCtrSum + 2;

// Window table: wtab[g * (nw + 1) + w] = first position in cluster g's
// member list whose member is >= w * win (windows aligned to multiples of
// win), so a window's end in every partition is one load instead of a
// search; one lower bound per entry over the cluster's ascending list.
__global__ void k_win_table(const int32_t* __restrict__ members,
                            const int32_t* __restrict__ cstart, int64_t ktot, int win, int nw,
                            int32_t* __restrict__ wtab) {
  const int64_t ts = nw + 1;
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < ktot * ts;
       q += (int64_t)gridDim.x * blockDim.x) {
    const int64_t g = q / ts;
    const int64_t at = (q - g * ts) * win;
    int32_t lo = cstart[g], hi = cstart[g + 1];
    while (lo < hi) {
      const int32_t mid = lo + ((hi - lo) >> 1);
      if (members[mid] < at) lo = mid + 1; else hi = mid;
    }
    wtab[q] = lo;
  }
}

// 64-bit words of a window's run-start bitmap: the flattened path covers
// windows of up to 128 members per partition on average (32 beyond 256
// partitions, where the bitmap would crowd out the counters).
__host__ __device__ inline int co_bm_words(int P) {
  return P <= 256 ? 2 * P + 2 : ((P / 2 + 1) + 1) & ~1;
}

// Window counters are bytes while every count fits one: a pair meets at most
// once per partition, so P <= 255; u16 beyond.
inline bool co_bytes(int P) { return P <= 255; }

struct CoPlan {
  const int32_t* labels;
  int64_t n;
  int P;
  const int64_t* k_off;   // [P+1] device
  const int32_t* members;
  const int32_t* pos;     // [P*n]
  const int32_t* cstart;  // [ktot+1] start of each global cluster in members
  const int32_t* wtab;    // window table (nullptr: search the window ends)
  int nw;                 // windows of the table: ceil(n / win)
  const int32_t* first;   // ranked fill: the partition processed first (device)
  int ranges;             // row ranges with a counter each: contiguous ones
                          // (1..kMaxRanges), or interleaved (-kStripes)
  int64_t row_stride;     // > 1: only rows 0, stride, 2*stride, ... (a sample)
};

// Outputs of the row kernel (pointers a pass does not use are null).
struct CoOut {
  unsigned long long* row_ctr;  // row counters kCtrPad apart, zeroed
  int32_t* row_nnz;             // PASS 0, 2, 3: nnz of each row
  unsigned int* max_count;      // PASS 0, 2, 3: largest count
  unsigned long long* nnz_sum;  // PASS 0: sum of the visited rows' nnz
  const int64_t* indptr;        // PASS 1: row offsets
  int32_t w_offset;             // PASS 1: data = w_offset - count when non-zero
  int32_t* col;                 // PASS 1: columns
  int32_t* val;                 // PASS 1: counts (or w_offset - count)
  int32_t* rank;                // PASS 1 with RANK: first partition rank
  uint32_t* pool;               // PASS 2, 3: staged entries (count << 16 | column - c0)
  uint64_t* seg;                // PASS 2, 3: per (row, window) offset << 16 | entries
  unsigned long long* pool_ctr; // PASS 2: next free pool chunk
  int64_t pool_cap;             // PASS 2: pool entries
  int64_t pool_chunk;           // PASS 2: entries per chunk (>= win)
  unsigned int* overflow;       // PASS 2: set when the pool ran out
};

// Staged entries are taken from the pool in chunks (one global atomic per
// chunk) of up to this many, or 16 windows when that is more. A pool of
// co_pairs entries needs no chunks: row i's entries of columns from c on start
// at co_pair_at(i, c), after a place for every pair before them.
constexpr int64_t kPoolChunk = 65536;
__host__ __device__ inline int64_t co_pairs(int64_t n, int full_rows) {
  return full_rows ? n * (n - 1) : n * (n - 1) / 2;
}
__host__ __device__ inline int64_t co_pair_at(int64_t i, int64_t c, int64_t n, int full_rows) {
  if (full_rows) return i * (n - 1) + c - (c > i ? 1 : 0);
  return i * (n - 1) - i * (i - 1) / 2 + (c > i + 1 ? c - (i + 1) : 0);
}

// Segment-table slot of (row i, first window of the row): rows keep the
// windows from w0(i) = (i + 1) / win on (every window with full rows), so
// the table packs them with sum_{r < i} (nw - w0(r)) slots before row i;
// sum_{m=1..i} floor(m / win) = win * q (q - 1) / 2 + q (i - q win + 1)
// with q = floor(i / win).
__host__ __device__ inline int64_t seg_base(int64_t i, int64_t win, int64_t nw, int full_rows) {
  if (full_rows) return i * nw;
  const int64_t q = i / win;
  return i * nw - (win * q * (q - 1) / 2 + q * (i - q * win + 1));
}

// The partition the reference processes first: the one with the fewest
// non-empty clusters, the first such (sparse.py:158: np.argmin over the
// cluster-list lengths; clusters are the labels present, partition.py:73-86).
// One block; cstart gives every global cluster's member count.
__global__ __launch_bounds__(256) void k_first_partition(const int32_t* __restrict__ cstart,
                                                         const int64_t* __restrict__ k_off,
                                                         int P, int32_t* __restrict__ first) {
  __shared__ unsigned long long s_best;
  if (threadIdx.x == 0) s_best = ~0ull;
  __syncthreads();
  for (int p = threadIdx.x; p < P; p += blockDim.x) {
    uint32_t nonempty = 0;
    for (int64_t g = k_off[p]; g < k_off[p + 1]; ++g) nonempty += cstart[g + 1] > cstart[g];
    atomicMin(&s_best, ((unsigned long long)nonempty << 32) | (unsigned)p);
  }
  __syncthreads();
  if (threadIdx.x == 0) first[0] = (int32_t)(s_best & 0xffffffffu);
}

// Window counters of type CT (u8 or u16): the words they take (a multiple of
// four, read 16 bytes at a time) and how a lane reads them.
__host__ __device__ inline int co_cnt_words(int win, int bytes) {
  return ((win * bytes + 15) / 16) * 4;
}
template <typename CT>
struct CoCnt {
  static constexpr int kB = (int)sizeof(CT);
  static constexpr int kPerWord = 4 / kB;   // columns per 32-bit word
  static constexpr int kPerGroup = 16 / kB; // columns per 16-byte group
  static constexpr int kPerLane = 2 * kPerGroup;  // columns a lane emits at a time
  // emission steps of a full window (kWin columns over kCB lanes): unrolled
  static constexpr int kIters = kWin / kPerLane / kCB;
  // one count for window column jj
  static __device__ __forceinline__ void add(uint32_t* cnt, int jj) {
    if (kB == 1) atomicAdd(&cnt[jj >> 2], 1u << ((jj & 3) * 8));
    else atomicAdd(&cnt[jj >> 1], 1u << ((jj & 1) * 16));
  }
  // bit c of the result: column c of the group has a non-zero counter. The
  // high bit of each counter of ((x & lo) + lo) | x is set iff the counter
  // is non-zero (lo: all bits but the high one); a byte dot product with
  // the weights 1, 2, 4, 8 gathers a word's four flags (times 128).
  static __device__ __forceinline__ uint32_t mask(const uint4& x) {
    const uint32_t w[4] = {x.x, x.y, x.z, x.w};
    if (kB == 1) {
      uint32_t m = 0;
#pragma unroll
      for (int q = 3; q >= 0; --q) {
        const uint32_t u =
            (((w[q] & 0x7f7f7f7fu) + 0x7f7f7f7fu) | w[q]) & 0x80808080u;
        m = (m << 4) + __builtin_amdgcn_udot4(u, 0x08040201u, 0u, false);
      }
      return m >> 7;
    }
    uint32_t m = 0;
#pragma unroll
    for (int q = 3; q >= 0; --q) {
      const uint32_t u = (((w[q] & 0x7fff7fffu) + 0x7fff7fffu) | w[q]) & 0x80008000u;
      m = (m << 2) | (u >> 31 << 1) | ((u >> 15) & 1u);
    }
    return m;
  }
  static __device__ __forceinline__ uint32_t max_of(const uint4& x, uint32_t mx) {
    const uint32_t w[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (kB == 1) {
        mx = max(mx, max(w[q] & 0xffu, w[q] >> 24));
        mx = max(mx, max((w[q] >> 8) & 0xffu, (w[q] >> 16) & 0xffu));
      } else {
        mx = max(mx, max(w[q] & 0xffffu, w[q] >> 16));
      }
    }
    return mx;
  }
};

// One row: walk every partition's co-members > i (or all co-members != i for
// full rows) window by window. PASS 0: per-row nnz and max count. PASS 1:
// write (col, value) at indptr[i]. RANK (PASS 1 only): also write, per entry,
// the processing rank of the first partition in which the pair co-occurs
// (0 = the partition pl.first[0], then the others in index order), kept in a
// second LDS window with one atomicMin per pair visit. PASS 2 (one-pass
// build): each window's entries go to the workgroup's current pool chunk as
// (count << 16 | column - c0), the window's (pool offset, entries) to the
// segment table, and the row's nnz and the max count as in PASS 0; a
// workgroup that finds the pool used up sets the overflow flag and stops.
// PASS 3: the same with a place for every pair in the pool (co_pair_at).
// U: member loads in flight per lane while visiting (4 or 8, a tuning knob).
template <int PASS, bool RANK, int U, typename CT>
__global__ __launch_bounds__(kCB) void k_coassoc_rows(CoPlan pl, int full_rows, int win,
                                                      CoOut out) {
  using Cnt = CoCnt<CT>;
  constexpr bool STAGE = PASS >= 2;
  unsigned long long* __restrict__ row_ctr = out.row_ctr;
  const int64_t* __restrict__ indptr = out.indptr;
  const int32_t w_offset = out.w_offset;
  int32_t* __restrict__ out_col = out.col;
  int32_t* __restrict__ out_val = out.val;
  int32_t* __restrict__ out_rank = out.rank;
  // launch-time LDS: this window's run-start bitmap (co_bm_words(P) entries
  // of 16 bytes: 64 bits, then the run starts marked in the words before),
  // the window counters, with RANK the rank window (win words), then per
  // partition the next member position, the cluster end, this window's
  // member end and the flattened-range prefix (P + 1), the row's global
  // cluster, this window's member position minus flattened index, each
  // partition's rank; per run (non-empty partition range of this window) the
  // position delta and the partition's rank
  extern __shared__ __align__(16) uint32_t s_dyn[];
  uint4* s_bm = reinterpret_cast<uint4*>(s_dyn);
  const int bmw = co_bm_words(pl.P);
  const int cwords = co_cnt_words(win, Cnt::kB);
  uint32_t* s_cnt = s_dyn + 4 * bmw;
  uint32_t* s_rank = s_cnt + cwords;
  int32_t* s_cur = reinterpret_cast<int32_t*>(s_cnt + cwords + (RANK ? win : 0));
  int32_t* s_end = s_cur + pl.P;
  int32_t* s_hi = s_end + pl.P;
  int32_t* s_pre = s_hi + pl.P;
  int32_t* s_g = s_pre + pl.P + 1;  // global cluster of the row in each partition
  int32_t* s_d = s_g + pl.P;        // this window: member position - flattened index
  int32_t* s_prank = s_d + pl.P;
  int32_t* s_dr = s_prank + pl.P;   // per run: member position - flattened index
  int32_t* s_rp = s_dr + pl.P;      // per run: rank of its partition
  const uint4* s4 = reinterpret_cast<const uint4*>(s_cnt);
  typedef CT __attribute__((may_alias)) CtAlias;
  const CtAlias* s_ct = reinterpret_cast<const CtAlias*>(s_cnt);
  __shared__ uint32_t s_tmp[kCB / kWave + 1];
  __shared__ int64_t s_row;
  __shared__ unsigned long long s_chunk;
  __shared__ unsigned int s_max;
  const int t = threadIdx.x;
  const int wv = __builtin_amdgcn_readfirstlane(t / kWave), ln = lane_id();
  const int64_t n = pl.n;
  const int P = pl.P;
  // the window is cleared once here; afterwards every window clears the
  // groups it used while reading them, so a clean window costs no pass
  for (int v = t; v < cwords; v += kCB) s_cnt[v] = 0;
  if (RANK) {
    for (int v = t; v < win; v += kCB) s_rank[v] = ~0u;
    const int f = pl.first[0];
    for (int p = t; p < P; p += kCB) s_prank[p] = p == f ? 0 : (p < f ? p + 1 : p);
  }
  // Rows are taken in the order of partition 0's member list (points
  // grouped by their partition-0 cluster) when every point is assigned
  // there: rows in flight at the same time then share most of their
  // clusters, so their member runs are read from cache. The output does not
  // depend on the order (each row writes its own segment).
  // The row order is cut into pl.ranges contiguous ranges with a counter
  // each; workgroup b starts on range b % ranges. Workgroups are dispatched
  // to the XCDs round-robin, so with 8 ranges each XCD (own L2) works
  // through its own stretch of the order and its resident rows share their
  // clusters' member lists in that L2. A workgroup whose range is used up
  // moves on to the next ranges (thread 0 keeps the cursor).
  // A small matrix (its member lists fit every L2) is bound by the counters
  // instead: atomics on one address serialise at about 16 ns each, 160 us
  // for 10,000 rows. There pl.ranges = -kStripes: row r belongs to range
  // r mod kStripes, so the ranges cost alike, and a workgroup whose range is
  // used up is done (10,000 rows x 100 partitions: the count pass 163 us
  // with one counter).
  const int32_t* order = nullptr;
  {
    const int32_t a = pl.cstart[pl.k_off[0]], b = pl.cstart[pl.k_off[1]];
    if ((int64_t)(b - a) == n) order = pl.members + a;
  }
  // a sample (row_stride > 1) takes rows 0, stride, 2 * stride, ...
  const int64_t stride = pl.row_stride > 1 ? pl.row_stride : 1;
  const int64_t nrows = (n + stride - 1) / stride;
  if (stride > 1) order = nullptr;
  const int nctr = pl.ranges < 0 ? -pl.ranges : pl.ranges;
  int xr = (int)(blockIdx.x % (unsigned)nctr), tries = 0;
  // PASS 2: the workgroup's pool chunk [chunk_pos, chunk_end) (uniform)
  int64_t chunk_pos = 0, chunk_end = 0;
  uint32_t mx_row = 0;  // largest count this lane met
  if (t == 0) s_max = 0;
  for (;;) {
    if (t == 0) {
      int64_t r = nrows;
      if (pl.ranges < 0) {
        r = xr + nctr * (int64_t)atomicAdd(&row_ctr[xr * kCtrPad], 1ull);
        if (r > nrows) r = nrows;
      } else {
        while (tries < nctr) {
          const int64_t lo = nrows * xr / nctr, hi = nrows * (xr + 1) / nctr;
          const int64_t q = lo + (int64_t)atomicAdd(&row_ctr[xr * kCtrPad], 1ull);
          if (q < hi) {
            r = q;
            break;
          }
          xr = xr + 1 == nctr ? 0 : xr + 1;
          ++tries;
        }
      }
      s_row = r;
    }
    __syncthreads();
    const int64_t r = s_row;
    if (r >= nrows) break;
    const int64_t i = order ? (int64_t)order[r] : r * stride;
    for (int p = t; p < P; p += kCB) {
      int32_t q = pl.pos[(int64_t)p * n + i];
      if (q < 0) {  // unassigned in partition p
        s_cur[p] = 0;
        s_end[p] = 0;
      } else {
        int64_t g = pl.k_off[p] + pl.labels[(int64_t)p * n + i];
        s_cur[p] = full_rows ? pl.cstart[g] : q + 1;
        s_end[p] = pl.cstart[g + 1];
        s_g[p] = (int32_t)g;
      }
    }
    int64_t row_base = PASS == 1 ? indptr[i] : 0;
    int64_t written = 0;
    // PASS 2: the row's first segment-table slot and its first window
    const int64_t w_first = full_rows ? 0 : (i + 1) / win;
    const int64_t seg0 = STAGE ? seg_base(i, win, pl.nw, full_rows) : 0;
    uint32_t nnz_local = 0;
    const int self = full_rows ? (int)i : -1;  // full rows skip the diagonal
    // windows aligned to multiples of win (columns <= i get no counts)
    for (int64_t c0 = full_rows ? 0 : ((i + 1) / win) * win; c0 < n; c0 += win) {
      const int64_t c1 = c0 + win < n ? c0 + win : n;
      for (int v = t; v < bmw; v += kCB) s_bm[v] = make_uint4(0u, 0u, 0u, 0u);
      // members of this window: [cur, hi) with member < c1 (lists ascending);
      // the last window takes every remaining member, no search. Otherwise
      // an exponential probe from cur (a window holds few members of each
      // partition), then a binary search inside the bracket.
      if (c1 == n) {
        for (int p = t; p < P; p += kCB) s_hi[p] = s_end[p];
      } else if (pl.wtab) {
        const int64_t w1 = c1 / win;
        for (int p = t; p < P; p += kCB)
          s_hi[p] = s_cur[p] >= s_end[p] ? s_end[p]
                                         : pl.wtab[(int64_t)s_g[p] * (pl.nw + 1) + w1];
      } else {
        for (int p = t; p < P; p += kCB) {
          int32_t lo = s_cur[p], hi = s_end[p];
          for (int32_t step = 16; lo < hi; step <<= 1) {
            const int32_t b = hi - lo > step ? lo + step : hi;
            if (pl.members[b - 1] < c1) {
              lo = b;  // all of [lo, b) lie in the window
            } else {
              hi = b;
              break;
            }
          }
          while (lo < hi) {
            int32_t mid = (lo + hi) >> 1;
            if (pl.members[mid] < c1) lo = mid + 1; else hi = mid;
          }
          s_hi[p] = lo;
        }
      }
      __syncthreads();
      // flattened ranges: prefix of (hi - cur) over partitions; the runs
      // (non-empty ranges) in partition order, each start but the first
      // marked one index early in the bitmap over the flattened indices
      // (short windows), and per bitmap word the marks before it: the marks
      // below flattened index f are then the number of f's run. One
      // wavefront: its LDS operations complete in order, so its bitmap reads
      // see its own marks.
      if (wv == 0) {
        int32_t carry = 0, rcarry = 0;
        const uint64_t below = (1ull << ln) - 1ull;
        for (int p0 = 0; p0 < P; p0 += kWave) {
          int p = p0 + ln;
          int32_t len = p < P ? s_hi[p] - s_cur[p] : 0;
          int32_t inc = (int32_t)wave_incl_scan_dpp((uint32_t)len);
          const uint64_t ne = __ballot(len > 0);
          if (p < P) {
            const int32_t pre = carry + inc - len;
            s_pre[p] = pre;
            s_d[p] = s_cur[p] - pre;
            if (len > 0) {
              const int r = rcarry + __popcll(ne & below);
              s_dr[r] = s_cur[p] - pre;
              if (RANK) s_rp[r] = s_prank[p];
              if (pre > 0 && pre <= 64 * bmw) {
                const int b = pre - 1;
                atomicOr(&s_dyn[(b >> 6) * 4 + ((b >> 5) & 1)], 1u << (b & 31));
              }
            }
          }
          carry += __builtin_amdgcn_readlane(inc, kWave - 1);
          rcarry += __popcll(ne);
        }
        if (ln == 0) s_pre[P] = carry;
        if (carry <= 64 * bmw) {  // the bitmap covers the window: word prefix counts
          const int W = (carry + 63) >> 6;
          int32_t wc = 0;
          for (int w0 = 0; w0 < W; w0 += kWave) {
            const int w = w0 + ln;
            const int32_t c = w < W ? __popc(s_dyn[4 * w]) + __popc(s_dyn[4 * w + 1]) : 0;
            const int32_t ci = (int32_t)wave_incl_scan_dpp((uint32_t)c);
            if (w < W) s_dyn[4 * w + 2] = (uint32_t)(wc + ci - c);
            wc += __builtin_amdgcn_readlane(ci, kWave - 1);
          }
        }
      }
      __syncthreads();
      const int32_t tot = s_pre[P];
      const int c0i = (int)c0;
      auto visit = [&](int32_t j, int32_t rk) {
        const int jj = j - c0i;
        Cnt::add(s_cnt, jj);
        if (RANK) atomicMin(&s_rank[jj], (uint32_t)rk);
      };
      // Flattened member index f -> member position f + delta of its run; U
      // member loads in flight per lane, consecutive lanes on consecutive f
      // (coalesced). While the bitmap covers the window (up to 128 members
      // per partition on average) each wavefront takes U * 64 consecutive f
      // per step and f's run is the number of marks below f: those in the
      // words before (one broadcast read with the word) plus a masked bit
      // count. Longer windows: the flattened range is split evenly over the
      // wavefronts and each walks its runs one after the other with
      // wave-uniform bounds, U * 64 members of a run per step (on average
      // at least two steps' worth of lanes per run, so few are idle, and no
      // per-member search). Whole steps run without a bounds check.
      if (tot > 64 * bmw) {
        const int32_t share = (tot + kCB / kWave - 1) / (kCB / kWave);
        const int32_t fa = wv * share, fb = fa + share < tot ? fa + share : tot;
        int p = 0;
        if (fa < fb) {
          int hi = P;  // s_pre[p] <= fa < s_pre[hi]
          while (hi - p > 1) {
            const int mid = (p + hi) >> 1;
            if (s_pre[mid] <= fa) p = mid; else hi = mid;
          }
        }
        for (int32_t f = fa; f < fb;) {
          const int32_t re = __builtin_amdgcn_readfirstlane(s_pre[p + 1]);
          const int32_t* __restrict__ mp =
              pl.members + __builtin_amdgcn_readfirstlane(s_d[p]);
          const int32_t rk = RANK ? s_prank[p] : 0;
          const int32_t e = re < fb ? re : fb;
          int32_t j[U];
          for (; f + U * kWave <= e; f += U * kWave) {
#pragma unroll
            for (int u = 0; u < U; ++u) j[u] = mp[f + u * kWave + ln];
#pragma unroll
            for (int u = 0; u < U; ++u)
              if (!full_rows || j[u] != self) visit(j[u], rk);
          }
          if (f < e) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
              const int32_t q = f + u * kWave + ln;
              j[u] = q < e ? mp[q] : -1;
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
              if (j[u] >= 0 && j[u] != self) visit(j[u], rk);
          }
          f = e;
          ++p;
        }
      } else {
        // member position and rank slot of flattened index base + 64 u + lane
        auto place = [&](int32_t base, int u, int32_t& rk) {
          const uint4 w = s_bm[(base >> 6) + u];
          const uint32_t r = __builtin_amdgcn_mbcnt_hi(w.y, __builtin_amdgcn_mbcnt_lo(w.x, w.z));
          if (RANK) rk = s_rp[r];
          return base + u * kWave + ln + s_dr[r];
        };
        int32_t base = wv * U * kWave;
        for (; base + U * kWave <= tot; base += U * kCB) {
          int32_t j[U], rk[U];
#pragma unroll
          for (int u = 0; u < U; ++u) j[u] = pl.members[place(base, u, rk[u])];
#pragma unroll
          for (int u = 0; u < U; ++u)
            if (!full_rows || j[u] != self) visit(j[u], rk[u]);
        }
        if (base < tot) {
          int32_t j[U], rk[U];
#pragma unroll
          for (int u = 0; u < U; ++u) {
            j[u] = -1;
            if (base + u * kWave + ln < tot) j[u] = pl.members[place(base, u, rk[u])];
          }
#pragma unroll
          for (int u = 0; u < U; ++u)
            if (j[u] >= 0 && j[u] != self) visit(j[u], rk[u]);
        }
      }
      __syncthreads();
      for (int p2 = t; p2 < P; p2 += kCB) s_cur[p2] = s_hi[p2];
      // read the window 16 bytes of counters per lane and load (the groups
      // past the window's width stay zero), clearing the groups it used
      const int width = (int)(c1 - c0);
      const int groups = (width + Cnt::kPerGroup - 1) / Cnt::kPerGroup;
      uint4* s4w = reinterpret_cast<uint4*>(s_cnt);
      if (PASS == 0) {
        uint32_t c = 0;
        for (int g = t; g < groups; g += kCB) {
          const uint4 x = s4[g];
          if (x.x | x.y | x.z | x.w) {
            s4w[g] = make_uint4(0u, 0u, 0u, 0u);
            c += __popc(Cnt::mask(x));
            mx_row = Cnt::max_of(x, mx_row);
          }
        }
        nnz_local += c;
      } else {  // PASS 1, 2 and 3
        // Wave w emits lane pieces (two groups each) [w*RG, (w+1)*RG) in
        // column order. First the non-zero masks of its pieces (kept in
        // registers: a window has few entries, about one column in twenty
        // on the large ensembles, so reading the counters is most of the
        // work), then per 64 pieces one prefix sum and a loop that takes the
        // set bits of each lane's mask one by one, so the instructions
        // follow the entries and not the columns.
        const int pieces = (groups + 1) >> 1;
        const int RG = ((pieces + 4 * kWave - 1) / (4 * kWave)) * kWave;
        const int ga = wv * RG, gb = (wv + 1) * RG < pieces ? (wv + 1) * RG : pieces;
        uint32_t mk[Cnt::kIters];
        uint32_t c = 0;
#pragma unroll
        for (int it = 0; it < Cnt::kIters; ++it) {
          mk[it] = 0;
          if (ga + it * kWave < gb) {  // uniform
            const int g = 2 * (ga + it * kWave + ln);
            if (g < groups) {
              mk[it] = Cnt::mask(s4[g]);
              if (g + 1 < groups) mk[it] |= Cnt::mask(s4[g + 1]) << Cnt::kPerGroup;
            }
            c += __popc(mk[it]);
          }
        }
        c = __builtin_amdgcn_readlane(wave_incl_scan_dpp(c), kWave - 1);
        if (ln == 0) s_tmp[wv] = c;
        __syncthreads();
        int64_t o = row_base + written;
        uint32_t wtot = 0;
        for (int q = 0; q < kCB / kWave; ++q) {
          if (q < wv) o += s_tmp[q];
          wtot += s_tmp[q];
        }
        if (STAGE) {  // block-uniform: wtot, chunk_pos, chunk_end
          if (PASS == 3) {
            chunk_pos = co_pair_at(i, c0, n, full_rows);
          } else if (chunk_pos + (int64_t)wtot > chunk_end) {
            if (t == 0) s_chunk = atomicAdd(out.pool_ctr, (unsigned long long)out.pool_chunk);
            __syncthreads();
            chunk_pos = (int64_t)s_chunk;
            chunk_end = chunk_pos + out.pool_chunk;
            if (chunk_end > out.pool_cap) {
              if (t == 0) atomicOr(out.overflow, 1u);
              return;  // the whole workgroup: the caller rebuilds in two passes
            }
          }
          o += chunk_pos - row_base - written;
          if (t == 0)
            out.seg[seg0 + c0 / win - w_first] =
                wtot ? ((uint64_t)chunk_pos << 16) | (uint64_t)wtot : 0ull;
          chunk_pos += wtot;
        }
        uint32_t* __restrict__ po = STAGE ? out.pool + o : nullptr;
        int32_t* __restrict__ pc = PASS == 1 ? out_col + o : nullptr;
        int32_t* __restrict__ pv = PASS == 1 ? out_val + o : nullptr;
        int32_t* __restrict__ pr = PASS == 1 && RANK ? out_rank + o : nullptr;
        uint32_t done = 0;  // entries this wave wrote before (uniform)
#pragma unroll
        for (int it = 0; it < Cnt::kIters; ++it) {
          if (ga + it * kWave >= gb) break;  // uniform
          uint32_t m = mk[it];
          if (__ballot(m != 0u) == 0ull) continue;
          const uint32_t cnt = __popc(m);
          const uint32_t incl = wave_incl_scan_dpp(cnt);
          uint32_t at = done + incl - cnt;
          const uint32_t here = __builtin_amdgcn_readlane(incl, kWave - 1);
          const int g = 2 * (ga + it * kWave + ln);
          const int colg = g * Cnt::kPerGroup;
          const uint32_t m0 = m;
          if (PASS == 1 && here > kWave * Cnt::kPerLane / 6) {
            // More than a sixth are entries: by column, 64 neighbours at a time,
            // so that a store covers a few lines and not one a lane (bit by bit,
            // 50,000 points, both visits: 0.9 full 14.3 and 3.7 ms, 0.4 4.5 and
            // 2.0, 0.23 1.97 and 1.42; but 0.12 1.07 and 1.10).
            const int lim = groups * Cnt::kPerGroup;
            int col = (ga + it * kWave) * Cnt::kPerLane + ln;
            for (int q = 0; q < Cnt::kPerLane; ++q, col += kWave) {
              const uint32_t v = col < lim ? s_ct[col] : 0u;
              const uint64_t full = __ballot(v != 0u);
              if (v) {
                at = done + __builtin_amdgcn_mbcnt_hi(
                                (uint32_t)(full >> 32),
                                __builtin_amdgcn_mbcnt_lo((uint32_t)full, 0u));
                pc[at] = c0i + col;
                pv[at] = w_offset ? w_offset - (int32_t)v : (int32_t)v;
                if (RANK) {
                  pr[at] = (int32_t)s_rank[col];
                  s_rank[col] = ~0u;
                }
              }
              done += __popcll(full);
            }
            m = 0;
          } else {
            done += here;
          }
          while (m) {
            const int col = colg + __builtin_ctz(m);
            m &= m - 1u;
            const uint32_t v = s_ct[col];
            if (STAGE) {
              po[at] = (v << 16) | (uint32_t)col;
              mx_row = max(mx_row, v);
            } else {
              pc[at] = c0i + col;
              pv[at] = w_offset ? w_offset - (int32_t)v : (int32_t)v;
              if (RANK) {
                pr[at] = (int32_t)s_rank[col];
                s_rank[col] = ~0u;
              }
            }
            ++at;
          }
          if (m0 & ((1u << Cnt::kPerGroup) - 1u)) s4w[g] = make_uint4(0u, 0u, 0u, 0u);
          if (m0 >> Cnt::kPerGroup) s4w[g + 1] = make_uint4(0u, 0u, 0u, 0u);
        }
        written += wtot;
      }
      __syncthreads();
    }
    if (PASS == 0) {
      uint32_t rt;
      (void)block_excl_scan<uint32_t>(nnz_local, s_tmp, &rt);
      if (t == 0) {
        out.row_nnz[i] = (int32_t)rt;
        if (out.nnz_sum) atomicAdd(out.nnz_sum, (unsigned long long)rt);
      }
    }
    if (STAGE && t == 0) out.row_nnz[i] = (int32_t)written;
    __syncthreads();
  }
  if (PASS != 1) {
    if (mx_row) atomicMax(&s_max, mx_row);
    __syncthreads();
    if (t == 0 && s_max) atomicMax(out.max_count, s_max);
  }
}

// One-pass build, last step: copies each row's staged segments, in window
// order, to indices/data at indptr[i] (one wavefront per row; the segment
// headers are wave-uniform loads).
// With ctl (the capturable build's device results: nnz, max count, error
// bits) nothing is written when an error bit is set, and w_offset = -1
// takes max count + 1 from ctl.
__global__ __launch_bounds__(256) void k_coassoc_compact(
    const unsigned char* __restrict__ stage, const int64_t* __restrict__ indptr, int64_t n,
    int32_t w_offset, int32_t* __restrict__ out_col, int32_t* __restrict__ out_val,
    const int64_t* __restrict__ ctl = nullptr) {
  if (ctl) {
    if (ctl[2] != 0) return;
    if (w_offset == -1) w_offset = (int32_t)ctl[1] + 1;
  }
  const int64_t* hdr = reinterpret_cast<const int64_t*>(stage);
  const int win = (int)hdr[0], nw = (int)hdr[1], full_rows = (int)hdr[5];
  const uint64_t* __restrict__ seg = reinterpret_cast<const uint64_t*>(stage + 256);
  const uint32_t* __restrict__ pool = reinterpret_cast<const uint32_t*>(stage + hdr[4]);
  const int l = lane_id();
  const int64_t waves = (int64_t)gridDim.x * (blockDim.x / kWave);
  for (int64_t i = (int64_t)blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave; i < n;
       i += waves) {
    const int64_t w_first = full_rows ? 0 : (i + 1) / win;
    const uint64_t* sg = seg + seg_base(i, win, nw, full_rows);
    int64_t dst = indptr[i];
    for (int64_t w = w_first; w < nw; ++w) {
      const uint64_t h = sg[w - w_first];
      const int cnt = (int)(h & 0xffffu);
      if (!cnt) continue;
      const uint32_t* src = pool + (h >> 16);
      const int32_t c0 = (int32_t)(w * win);
      for (int e = l; e < cnt; e += kWave) {
        const uint32_t x = src[e];
        const int32_t c = (int32_t)(x >> 16);
        out_col[dst + e] = c0 + (int32_t)(x & 0xffffu);
        out_val[dst + e] = w_offset ? w_offset - c : c;
      }
      dst += cnt;
    }
  }
}

struct CoBufs {
  int64_t* k_off;
  int32_t* wtab;     // [items] window table, when it fits
  int32_t* members;
  int32_t* pos;
  int32_t* cstart;
  int32_t* row_nnz;
  unsigned long long* ctr;  // [kCtrs]: row counters, [kCtrSum] sampled nnz sum
  unsigned int* misc;  // [0] bad label, [1] max count
};

CoBufs carve_co(Arena& ar, int64_t n, int P, int64_t ktot) {
  CoBufs b;
  int64_t items = (int64_t)P * n;
  b.k_off = ar.take<int64_t>(P + 1);
  b.members = ar.take<int32_t>(items);
  b.pos = ar.take<int32_t>(items);
  b.cstart = ar.take<int32_t>(ktot + 2);
  b.row_nnz = ar.take<int32_t>(n + 1);
  b.ctr = ar.take<unsigned long long>(kCtrs + 2);  // one fill clears both
  b.misc = reinterpret_cast<unsigned int*>(b.ctr + kCtrs);
  b.wtab = ar.take<int32_t>(items);
  return b;
}

int d2h(void* host, const void* dev, size_t bytes, hipStream_t s) {
  void* pin = pinned_scratch(bytes);
  if (!pin) return fail(EAC_ERR_HIP, "pinned host allocation failed");
  EAC_HIP_CHECK(hipMemcpyAsync(pin, dev, bytes, hipMemcpyDeviceToHost, s));
  EAC_HIP_CHECK(hipStreamSynchronize(s));
  memcpy(host, pin, bytes);
  return EAC_OK;
}

// Several small reads behind one wait (a wait costs 10 us, a copy 2).
struct HostRead {
  void* host;
  const void* dev;
  size_t bytes;
};
template <int N>
int d2h_all(const HostRead (&r)[N], hipStream_t s) {
  constexpr size_t kSlot = 64;
  char* pin = static_cast<char*>(pinned_scratch(N * kSlot));
  if (!pin) return fail(EAC_ERR_HIP, "pinned host allocation failed");
  for (int i = 0; i < N; ++i) {
    if (r[i].bytes > kSlot) return fail(EAC_ERR_ARG, "coassoc: host read too long");
    EAC_HIP_CHECK(hipMemcpyAsync(pin + i * kSlot, r[i].dev, r[i].bytes, hipMemcpyDeviceToHost, s));
  }
  EAC_HIP_CHECK(hipStreamSynchronize(s));
  for (int i = 0; i < N; ++i) memcpy(r[i].host, pin + i * kSlot, r[i].bytes);
  return EAC_OK;
}

int co_check(const int32_t* labels, int64_t n, const int64_t* h_koff, int32_t P) {
  if (n < 1 || P < 1) return fail(EAC_ERR_ARG, "coassoc: need n, P >= 1");
  if (P > kMaxP) return fail(EAC_ERR_UNSUPPORTED, "coassoc: more than %d partitions", kMaxP);
  if (!labels || !h_koff) return fail(EAC_ERR_ARG, "coassoc: null array");
  if (h_koff[0] != 0) return fail(EAC_ERR_ARG, "coassoc: k_off[0] must be 0");
  for (int p = 0; p < P; ++p)
    if (h_koff[p + 1] < h_koff[p]) return fail(EAC_ERR_ARG, "coassoc: k_off not ascending");
  if ((int64_t)P * n >= (int64_t)INT32_MAX)
    return fail(EAC_ERR_UNSUPPORTED, "coassoc: P*n too large");
  return EAC_OK;
}

}  // namespace
// Columns per LDS window (even, <= kWin): the whole row range when n is
// small (fewer LDS bytes, more resident workgroups), else 16384 (16 KiB of
// byte counters: seven workgroups per compute unit; 200,003 points x 64
// partitions, whole build: 13.0 / 11.8 / 11.0 / 11.0 / 12.3 ms at 8192 /
// 12288 / 16384 / 24576 / 32768), or the EAC_TUNE_CO_WINDOW setting (the
// autotuner trades windows per row against workgroups per compute unit).
int co_window(int64_t n) {
  int w = tune_value(EAC_TUNE_CO_WINDOW);
  if (w <= 0) w = 16384;
  if (w > kWin) w = kWin;
  const int64_t need = ((n + 63) / 64) * 64;
  if (need < w) w = (int)need;
  return w < 64 ? 64 : (w & ~1);
}
// Member loads in flight per lane in the pair visits (EAC_TUNE_CO_UNROLL:
// 4 by default, or 8).
inline int co_unroll() { return tune_value(EAC_TUNE_CO_UNROLL) == 8 ? 8 : 4; }
// Row ranges of the co-association row loop (EAC_TUNE_CO_RANGES: 1..8
// contiguous ones; default one per XCD, or kStripes interleaved ranges below
// 65536 rows, see the row kernel).
inline int co_ranges(int64_t n) {
  const int r = tune_value(EAC_TUNE_CO_RANGES);
  if (r > 0 && r <= kMaxRanges) return r;
  return n < 65536 ? -kStripes : kMaxRanges;
}
inline size_t co_lds(int win, int P, bool rank = false) {
  return (size_t)(4 * co_bm_words(P) + co_cnt_words(win, co_bytes(P) ? 1 : 2) +
                  (rank ? win : 0) + 9 * P + 1) * 4;
}
// The ranked fill keeps a 4-byte rank per column next to the counters: its
// window is at most half as wide.
constexpr int kWinRank = kWin / 2;

// Builds the window table when it fits its buffer; returns nullptr otherwise
// (the rows then search their window ends).
int32_t* build_win_table(const CoBufs& B, int64_t n, int P, int64_t ktot, int win, int* nw,
                         hipStream_t s) {
  *nw = (int)((n + win - 1) / win);
  const int64_t items = (int64_t)P * n, entries = ktot * (int64_t)(*nw + 1);
  if (*nw < 2 || entries > items) return nullptr;  // one window needs no table
  k_win_table<<<grid_for(entries, 256, 16384), 256, 0, s>>>(B.members, B.cstart, ktot, win, *nw,
                                                            B.wtab);
  if (hipGetLastError() != hipSuccess) return nullptr;
  return B.wtab;
}
// The row kernel with the counter width for P and the unroll knob.
using CoRowsFn = void (*)(CoPlan, int, int, CoOut);
template <int PASS, bool RANK = false>
CoRowsFn co_rows_fn(int P) {
  if constexpr (RANK) {
    return co_bytes(P) ? k_coassoc_rows<PASS, true, 4, uint8_t>
                       : k_coassoc_rows<PASS, true, 4, uint16_t>;
  } else {
    if (co_unroll() == 8)
      return co_bytes(P) ? k_coassoc_rows<PASS, false, 8, uint8_t>
                         : k_coassoc_rows<PASS, false, 8, uint16_t>;
    return co_bytes(P) ? k_coassoc_rows<PASS, false, 4, uint8_t>
                       : k_coassoc_rows<PASS, false, 4, uint16_t>;
  }
}
// Every workgroup resident at once (rows are handed out dynamically).
template <int PASS, bool RANK = false>
int co_grid(int win, int P) {
  int dev = 0, cus = 256, per = 1;
  if (hipGetDevice(&dev) == hipSuccess)
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  // allow launch-time LDS beyond 64 KB (the window of large graphs)
  const size_t lds = co_lds(win, P, RANK);
  const void* fn = reinterpret_cast<const void*>(co_rows_fn<PASS, RANK>(P));
  (void)hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, fn, kCB, lds) != hipSuccess || per < 1)
    per = 1;
  return cus * per;
}

}  // namespace eac

// ------------------------------------------------------------------ C ABI
using namespace eac;

extern "C" size_t eac_coassoc_workspace_bytes(int64_t n, int32_t P, int64_t k_total) {
  if (n < 1) n = 1;
  if (P < 1) P = 1;
  Arena ar(nullptr, 0, true);
  (void)carve_co(ar, n, P, k_total);
  const size_t s1 = group_ws_bytes(n, P, k_total);
  const size_t s2 = scan_ws_bytes(n + 1, 8);
  return ar.used + (s1 > s2 ? s1 : s2) + 4096;
}

namespace eac {
namespace {
// The member plan in ws (shared by every pass over the same labels): member
// lists, cluster starts, each point's position in its cluster's list; zeroes
// the row counters and flags.
int co_plan_build(const int32_t* labels, int64_t n, const int64_t* h_koff, int32_t P,
                  void* ws, size_t ws_bytes, CoBufs* out, size_t* mark_out, Arena& ar,
                  hipStream_t s, const int64_t* d_koff = nullptr) {
  EAC_TRY(co_check(labels, n, h_koff, P));
  const int64_t ktot = h_koff[P];
  size_t need = eac_coassoc_workspace_bytes(n, P, ktot);
  if (!ws || ws_bytes < need)
    return fail(EAC_ERR_WORKSPACE, "coassoc: workspace %zu < %zu bytes", ws_bytes, need);
  CoBufs B = carve_co(ar, n, P, ktot);
  const size_t mark = ar.used;
  const int64_t items = (int64_t)P * n;
  if (d_koff) {  // already on the device: a device copy (capturable)
    EAC_HIP_CHECK(hipMemcpyAsync(B.k_off, d_koff, sizeof(int64_t) * (P + 1),
                                 hipMemcpyDeviceToDevice, s));
  } else {
    EAC_TRY(put_i64(B.k_off, h_koff, P + 1, s));
  }
  EAC_TRY(fill<int64_t>((int64_t*)B.ctr, kCtrs + 2, 0, s));
  int pr = prof_begin(EAC_PROF_CO_PLAN, 16 * items, s);
  EAC_TRY(group_by_cluster(labels, n, P, B.k_off, h_koff, reinterpret_cast<uint32_t*>(B.members),
                           reinterpret_cast<uint32_t*>(B.cstart), B.pos, B.misc, ar, s));
  ar.used = mark;
  prof_end(pr, s);
  *out = B;
  *mark_out = mark;
  return EAC_OK;
}

template <int PASS, bool RANK = false>
int co_launch(const CoPlan& pl, int full_rows, int win, const CoOut& o, hipStream_t s) {
  co_rows_fn<PASS, RANK>(pl.P)<<<co_grid<PASS, RANK>(win, pl.P), kCB, co_lds(win, pl.P, RANK),
                                 s>>>(pl, full_rows, win, o);
  EAC_LAUNCH_CHECK();
  return EAC_OK;
}
}  // namespace
}  // namespace eac

// Pass 1: builds the member plan in ws (keep ws unchanged for the fill),
// writes indptr[n+1] (int64) and returns nnz and the largest count.
extern "C" int eac_coassoc_count(const int32_t* labels, int64_t n, const int64_t* h_koff,
                                 int32_t P, int32_t full_rows, int64_t* indptr, int64_t* h_nnz,
                                 int32_t* h_max_count, void* ws, size_t ws_bytes, void* stream) {
  EAC_TRY(co_check(labels, n, h_koff, P));
  if (!indptr) return fail(EAC_ERR_ARG, "coassoc: null indptr");
  hipStream_t s = (hipStream_t)stream;
  const int64_t ktot = h_koff[P];
  Arena ar(ws, ws_bytes);
  CoBufs B;
  size_t mark = 0;
  EAC_TRY(co_plan_build(labels, n, h_koff, P, ws, ws_bytes, &B, &mark, ar, s));
  const int win = co_window(n);
  int nw = 0;
  const int32_t* wtab = build_win_table(B, n, P, ktot, win, &nw, s);
  CoPlan pl{labels, n, P, B.k_off, B.members, B.pos, B.cstart, wtab, nw, nullptr, co_ranges(n), 1};
  CoOut o{};
  o.row_ctr = B.ctr;
  o.row_nnz = B.row_nnz;
  o.max_count = B.misc + 1;
  int pr2 = prof_begin(EAC_PROF_CO_COUNT, 0, s);
  EAC_TRY(co_launch<0>(pl, full_rows, win, o, s));
  prof_end(pr2, s);
  EAC_TRY((scan_excl<int32_t, int64_t>(B.row_nnz, indptr, n + 1, 0, nullptr, ar, s)));
  ar.used = mark;
  unsigned int misc[4];
  int64_t nnz = 0;
  EAC_TRY(d2h_all<2>({{misc, B.misc, sizeof(misc)}, {&nnz, indptr + n, sizeof(nnz)}}, s));
  prof_flush();
  if (misc[0]) return fail(EAC_ERR_ARG, "coassoc: label >= k of its partition");
  if (h_nnz) *h_nnz = nnz;
  if (h_max_count) *h_max_count = (int32_t)misc[1];
  return EAC_OK;
}

// Pass 2 (same ws as pass 1): indices[nnz] (int32 columns, ascending per
// row) and data[nnz] = count, or w_offset - count when w_offset != 0
// (make_diassoc, sparse.py:295-311, with w_offset = max + 1).
namespace eac {
namespace {
int coassoc_fill(const int32_t* labels, int64_t n, const int64_t* h_koff, int32_t P,
                 int32_t full_rows, const int64_t* indptr, int32_t w_offset, int32_t* indices,
                 int32_t* data, int32_t* rank, void* ws, size_t ws_bytes, hipStream_t s) {
  EAC_TRY(co_check(labels, n, h_koff, P));
  if (!indptr || !indices || !data) return fail(EAC_ERR_ARG, "coassoc: null output");
  const int64_t ktot = h_koff[P];
  size_t need = eac_coassoc_workspace_bytes(n, P, ktot);
  if (!ws || ws_bytes < need)
    return fail(EAC_ERR_WORKSPACE, "coassoc: workspace %zu < %zu bytes", ws_bytes, need);
  Arena ar(ws, ws_bytes);
  CoBufs B = carve_co(ar, n, P, ktot);
  EAC_TRY(fill<int64_t>((int64_t*)B.ctr, kCtrs, 0, s));
  int64_t nnz = 0;
  EAC_TRY(d2h(&nnz, indptr + n, sizeof(int64_t), s));
  int win = co_window(n);
  if (rank && win > kWinRank) win = kWinRank;
  int nw = 0;
  const int32_t* wtab = build_win_table(B, n, P, ktot, win, &nw, s);
  int32_t* d_first = reinterpret_cast<int32_t*>(B.misc + 2);
  CoPlan pl{labels, n, P, B.k_off, B.members, B.pos, B.cstart, wtab, nw, d_first, co_ranges(n), 1};
  CoOut o{};
  o.row_ctr = B.ctr;
  o.indptr = indptr;
  o.w_offset = w_offset;
  o.col = indices;
  o.val = data;
  o.rank = rank;
  int pr = prof_begin(EAC_PROF_CO_FILL, 8 * nnz + 8 * (n + 1), s);
  if (rank) {
    k_first_partition<<<1, 256, 0, s>>>(B.cstart, B.k_off, P, d_first);
    EAC_LAUNCH_CHECK();
    EAC_TRY((co_launch<1, true>(pl, full_rows, win, o, s)));
  } else {
    EAC_TRY(co_launch<1>(pl, full_rows, win, o, s));
  }
  prof_end(pr, s);
  EAC_HIP_CHECK(hipStreamSynchronize(s));
  prof_flush();
  return EAC_OK;
}
}  // namespace
}  // namespace eac

extern "C" int eac_coassoc_fill(const int32_t* labels, int64_t n, const int64_t* h_koff,
                                int32_t P, int32_t full_rows, const int64_t* indptr,
                                int32_t w_offset, int32_t* indices, int32_t* data, void* ws,
                                size_t ws_bytes, void* stream) {
  return coassoc_fill(labels, n, h_koff, P, full_rows, indptr, w_offset, indices, data, nullptr,
                      ws, ws_bytes, (hipStream_t)stream);
}

// Pass 2 with, per entry, the processing rank of the first partition in
// which the pair co-occurs (the input of the capacity-capped selection).
extern "C" int eac_coassoc_fill_ranked(const int32_t* labels, int64_t n, const int64_t* h_koff,
                                       int32_t P, int32_t full_rows, const int64_t* indptr,
                                       int32_t* indices, int32_t* data, int32_t* rank, void* ws,
                                       size_t ws_bytes, void* stream) {
  if (!rank) return fail(EAC_ERR_ARG, "coassoc: null rank output");
  return coassoc_fill(labels, n, h_koff, P, full_rows, indptr, 0, indices, data, rank, ws,
                      ws_bytes, (hipStream_t)stream);
}

// ------------------------------------------------------- one-pass build
// The count pass visits every pair once only to size the output; the
// one-pass build visits them once: the plan plus a sampled count estimate
// the nnz, the caller allocates a staging buffer from it, the staged pass
// writes every window's entries (4 bytes each) to chunks of that buffer
// and the row sizes, and a compaction copies the segments into the CSR.
// A pool that turns out too small is reported (h_nnz = -1): the caller
// then runs eac_coassoc_count + eac_coassoc_fill.
namespace eac {
namespace {
// staging buffer: header (int64: win, nw, pool counter, overflow flag,
// pool byte offset, full_rows), then the segment table, then the pool
// (4-byte entries). The compaction takes the layout from the header.
constexpr size_t kStageHdr = 256;
__global__ void k_stage_header(int64_t* hdr, int win, int nw, int64_t pool_at, int full_rows) {
  if (threadIdx.x == 0) {
    hdr[0] = win;
    hdr[1] = nw;
    hdr[2] = 0;
    hdr[3] = 0;
    hdr[4] = pool_at;
    hdr[5] = full_rows;
  }
}
struct StageLayout {
  int win, nw;
  int64_t slots;     // segment-table entries
  size_t pool_at;    // byte offset of the pool
  int64_t chunk;     // pool entries per chunk: n / 8 rounded up to a power
                     // of two, at most kPoolChunk, and at least 16 windows
                     // (a chunk loses at most one window's width at its end)
};
StageLayout stage_layout(int64_t n, int full_rows) {
  StageLayout L;
  L.win = co_window(n);
  L.nw = (int)((n + L.win - 1) / L.win);
  L.slots = seg_base(n, L.win, L.nw, full_rows);
  L.pool_at = kStageHdr + (((size_t)L.slots * 8 + 255) & ~(size_t)255);
  int64_t c = 1;
  while (c < n / 8 && c < kPoolChunk) c <<= 1;
  L.chunk = c < 16 * (int64_t)L.win ? 16 * (int64_t)L.win : c;
  return L;
}
// Entries per chunk for a staging buffer of these bytes, -1: it does not hold
// one. 0: a place for every pair (PASS 3), for the bytes
// eac_coassoc_stage_bytes gives for that, or rounded up to a page (a larger
// buffer was sized as entries and chunks).
int64_t stage_chunk(const StageLayout& L, int64_t n, int full_rows, size_t stage_bytes) {
  const size_t all = L.pool_at + (size_t)co_pairs(n, full_rows) * 4;
  if (stage_bytes >= all && stage_bytes < all + 4096) return 0;
  return stage_bytes >= L.pool_at + (size_t)L.chunk * 4 ? L.chunk : -1;
}
}  // namespace
}  // namespace eac

// The plan alone (as eac_coassoc_count builds it); a label of k or more of its
// partition is an error. Keep ws for eac_coassoc_stage.
extern "C" int eac_coassoc_plan(const int32_t* labels, int64_t n, const int64_t* h_koff,
                                int32_t P, void* ws, size_t ws_bytes, void* stream) {
  EAC_TRY(co_check(labels, n, h_koff, P));
  hipStream_t s = (hipStream_t)stream;
  Arena ar(ws, ws_bytes);
  CoBufs B;
  size_t mark = 0;
  EAC_TRY(co_plan_build(labels, n, h_koff, P, ws, ws_bytes, &B, &mark, ar, s));
  unsigned int misc[4];
  EAC_TRY(d2h(misc, B.misc, sizeof(misc), s));
  if (misc[0]) return fail(EAC_ERR_ARG, "coassoc: label >= k of its partition");
  return EAC_OK;
}

// Plan (as eac_coassoc_count) plus the count pass over rows 0, stride,
// 2 * stride, ...: h_estimate = their nnz sum x (rows / sampled rows),
// rounded up. Keep ws for eac_coassoc_stage.
extern "C" int eac_coassoc_estimate(const int32_t* labels, int64_t n, const int64_t* h_koff,
                                    int32_t P, int32_t full_rows, int64_t sample_stride,
                                    int64_t* h_estimate, void* ws, size_t ws_bytes,
                                    void* stream) {
  EAC_TRY(co_check(labels, n, h_koff, P));
  if (sample_stride < 1) return fail(EAC_ERR_ARG, "coassoc: sample stride must be >= 1");
  if (!h_estimate) return fail(EAC_ERR_ARG, "coassoc: null estimate");
  hipStream_t s = (hipStream_t)stream;
  const int64_t ktot = h_koff[P];
  Arena ar(ws, ws_bytes);
  CoBufs B;
  size_t mark = 0;
  EAC_TRY(co_plan_build(labels, n, h_koff, P, ws, ws_bytes, &B, &mark, ar, s));
  const int win = co_window(n);
  int nw = 0;
  const int32_t* wtab = build_win_table(B, n, P, ktot, win, &nw, s);
  CoPlan pl{labels, n, P,  B.k_off,     B.members,    B.pos, B.cstart,
            wtab,   nw, nullptr, co_ranges(n), sample_stride};
  CoOut o{};
  o.row_ctr = B.ctr;
  o.row_nnz = B.row_nnz;
  o.max_count = B.misc + 1;
  o.nnz_sum = B.ctr + kCtrSum;
  int pr = prof_begin(EAC_PROF_CO_COUNT, 0, s);
  EAC_TRY(co_launch<0>(pl, full_rows, win, o, s));
  prof_end(pr, s);
  unsigned int misc[4];
  unsigned long long sum = 0;
  EAC_TRY(d2h_all<2>({{misc, B.misc, sizeof(misc)}, {&sum, B.ctr + kCtrSum, sizeof(sum)}}, s));
  prof_flush();
  if (misc[0]) return fail(EAC_ERR_ARG, "coassoc: label >= k of its partition");
  const int64_t rows = (n + sample_stride - 1) / sample_stride;
  *h_estimate = (int64_t)(((long double)sum * n + rows - 1) / rows);
  return EAC_OK;
}

// Bytes of the staging buffer with room for pool_entries staged entries
// beyond the partly used chunks of the workgroups, or for every pair and no
// more (the segment table and the chunk size depend on n, full_rows and the
// window knob).
extern "C" size_t eac_coassoc_stage_bytes(int64_t n, int32_t full_rows, int32_t P,
                                          int64_t pool_entries) {
  if (n < 1) n = 1;
  if (P < 1) P = 1;
  if (pool_entries < 0) pool_entries = 0;
  const StageLayout L = stage_layout(n, full_rows);
  const int64_t pairs = co_pairs(n, full_rows);
  if (pool_entries >= pairs) return L.pool_at + (size_t)pairs * 4;
  const int64_t grid = co_grid<2>(L.win, P);
  return L.pool_at + (size_t)(pool_entries + (grid + 1) * L.chunk) * 4;
}

// Staged pass (ws from eac_coassoc_estimate): writes indptr[n+1] and, in
// stage, every row's window segments; h_nnz = nnz and h_max_count the
// largest count, or h_nnz = -1 when the pool was too small.
extern "C" int eac_coassoc_stage(const int32_t* labels, int64_t n, const int64_t* h_koff,
                                 int32_t P, int32_t full_rows, int64_t* indptr, void* stage,
                                 size_t stage_bytes, int64_t* h_nnz, int32_t* h_max_count,
                                 void* ws, size_t ws_bytes, void* stream) {
  EAC_TRY(co_check(labels, n, h_koff, P));
  if (!indptr || !stage || !h_nnz) return fail(EAC_ERR_ARG, "coassoc: null argument");
  const int64_t ktot = h_koff[P];
  size_t need = eac_coassoc_workspace_bytes(n, P, ktot);
  if (!ws || ws_bytes < need)
    return fail(EAC_ERR_WORKSPACE, "coassoc: workspace %zu < %zu bytes", ws_bytes, need);
  const StageLayout SL = stage_layout(n, full_rows);
  const int64_t chunk = stage_chunk(SL, n, full_rows, stage_bytes);
  if (chunk < 0)
    return fail(EAC_ERR_WORKSPACE, "coassoc: staging buffer %zu < %zu bytes", stage_bytes,
                SL.pool_at + (size_t)SL.chunk * 4);
  hipStream_t s = (hipStream_t)stream;
  Arena ar(ws, ws_bytes);
  CoBufs B = carve_co(ar, n, P, ktot);
  const size_t mark = ar.used;
  unsigned char* st = static_cast<unsigned char*>(stage);
  int64_t* hdr = reinterpret_cast<int64_t*>(st);
  k_stage_header<<<1, 64, 0, s>>>(hdr, SL.win, SL.nw, (int64_t)SL.pool_at, full_rows);
  EAC_LAUNCH_CHECK();
  EAC_TRY(fill<int64_t>((int64_t*)B.ctr, kCtrs + 2, 0, s));
  int nw = 0;
  const int32_t* wtab = build_win_table(B, n, P, ktot, SL.win, &nw, s);
  CoPlan pl{labels, n, P, B.k_off, B.members, B.pos, B.cstart, wtab, nw, nullptr, co_ranges(n), 1};
  CoOut o{};
  o.row_ctr = B.ctr;
  o.row_nnz = B.row_nnz;
  o.max_count = B.misc + 1;
  o.seg = reinterpret_cast<uint64_t*>(st + kStageHdr);
  o.pool = reinterpret_cast<uint32_t*>(st + SL.pool_at);
  o.pool_ctr = reinterpret_cast<unsigned long long*>(hdr + 2);
  o.pool_cap = (int64_t)((stage_bytes - SL.pool_at) / 4);
  o.pool_chunk = chunk;
  o.overflow = reinterpret_cast<unsigned int*>(hdr + 3);
  int pr = prof_begin(EAC_PROF_CO_STAGE, 0, s);
  // (PASS 3 apart: the choice inside PASS 2 cost its emission 1.7%)
  EAC_TRY(chunk ? co_launch<2>(pl, full_rows, SL.win, o, s)
                : co_launch<3>(pl, full_rows, SL.win, o, s));
  prof_end(pr, s);
  EAC_TRY((scan_excl<int32_t, int64_t>(B.row_nnz, indptr, n + 1, 0, nullptr, ar, s)));
  ar.used = mark;
  unsigned int misc[4];
  int64_t tail[2] = {0, 0};  // overflow flag (hdr[3])
  int64_t nnz = 0;
  EAC_TRY(d2h_all<3>({{misc, B.misc, sizeof(misc)},
                      {tail, hdr + 2, sizeof(tail)},
                      {&nnz, indptr + n, sizeof(nnz)}},
                     s));
  prof_flush();
  *h_nnz = tail[1] ? -1 : nnz;
  if (h_max_count) *h_max_count = (int32_t)misc[1];
  return EAC_OK;
}

// Compaction of a staged build: indices[nnz] / data[nnz] as
// eac_coassoc_fill writes them (data = count, or w_offset - count).
extern "C" int eac_coassoc_compact(int64_t n, const int64_t* indptr, const void* stage,
                                   size_t stage_bytes, int32_t w_offset, int32_t* indices,
                                   int32_t* data, void* stream) {
  if (n < 1) return fail(EAC_ERR_ARG, "coassoc: need n >= 1");
  if (!indptr || !stage || !indices || !data) return fail(EAC_ERR_ARG, "coassoc: null argument");
  if (stage_bytes < kStageHdr)
    return fail(EAC_ERR_WORKSPACE, "coassoc: staging buffer %zu < %zu bytes", stage_bytes,
                kStageHdr);
  hipStream_t s = (hipStream_t)stream;
  int pr = prof_begin(EAC_PROF_CO_COMPACT, 0, s);
  const int64_t blocks = (n + 3) / 4;
  k_coassoc_compact<<<(unsigned)(blocks < 65536 ? blocks : 65536), 256, 0, s>>>(
      static_cast<const unsigned char*>(stage), indptr, n, w_offset, indices, data, nullptr);
  EAC_LAUNCH_CHECK();
  prof_end(pr, s);
  EAC_HIP_CHECK(hipStreamSynchronize(s));
  prof_flush();
  return EAC_OK;
}

// ------------------------------------------- capturable one-pass build
// Results of the capturable build in the caller's device int64[4]: nnz,
// largest count, error bits (1: pool too small, 2: more than cap_nnz
// entries, 4: a label >= k of its partition), 0.
namespace eac {
namespace {
__global__ void k_co_finish(const int64_t* __restrict__ indptr, int64_t n,
                            const unsigned int* __restrict__ misc,
                            const int64_t* __restrict__ hdr, int64_t cap_nnz,
                            int64_t* __restrict__ out) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  const int64_t nnz = indptr[n];
  int64_t err = 0;
  if (hdr[3]) err |= 1;
  if (nnz > cap_nnz) err |= 2;
  if (misc[0]) err |= 4;
  out[0] = nnz;
  out[1] = (int64_t)misc[1];
  out[2] = err;
  out[3] = 0;
}
}  // namespace
}  // namespace eac

// The one-pass build with no host read, copy or synchronisation (for
// capture in a HIP graph): the member plan from d_koff (h_koff still gives
// the sizes), the staged pass into `stage` (eac_coassoc_stage_bytes of the
// pool the caller can afford; no estimate), the row offsets, and the
// compaction into indices/data of capacity cap_nnz. w_offset as in
// eac_coassoc_fill, or -1 for (largest count + 1) taken on the device.
// d_out (device int64[4]): nnz, largest count, error bits (1: pool too
// small, 2: nnz > cap_nnz, 4: label >= k; no entry is written then).
extern "C" int eac_coassoc_graph(const int32_t* labels, int64_t n, const int64_t* h_koff,
                                 const int64_t* d_koff, int32_t P, int32_t full_rows,
                                 int32_t w_offset, int64_t* indptr, int32_t* indices,
                                 int32_t* data, int64_t cap_nnz, void* stage,
                                 size_t stage_bytes, int64_t* d_out, void* ws, size_t ws_bytes,
                                 void* stream) {
  EAC_TRY(co_check(labels, n, h_koff, P));
  if (!d_koff || !indptr || !indices || !data || !stage || !d_out)
    return fail(EAC_ERR_ARG, "coassoc graph: null argument");
  if (w_offset < -1) return fail(EAC_ERR_ARG, "coassoc graph: w_offset < -1");
  const int64_t ktot = h_koff[P];
  const StageLayout SL = stage_layout(n, full_rows);
  const int64_t chunk = stage_chunk(SL, n, full_rows, stage_bytes);
  if (chunk < 0)
    return fail(EAC_ERR_WORKSPACE, "coassoc graph: staging buffer %zu < %zu bytes", stage_bytes,
                SL.pool_at + (size_t)SL.chunk * 4);
  hipStream_t s = (hipStream_t)stream;
  Arena ar(ws, ws_bytes);
  CoBufs B;
  size_t mark = 0;
  EAC_TRY(co_plan_build(labels, n, h_koff, P, ws, ws_bytes, &B, &mark, ar, s, d_koff));
  unsigned char* st = static_cast<unsigned char*>(stage);
  int64_t* hdr = reinterpret_cast<int64_t*>(st);
  k_stage_header<<<1, 64, 0, s>>>(hdr, SL.win, SL.nw, (int64_t)SL.pool_at, full_rows);
  EAC_LAUNCH_CHECK();
  int nw = 0;
  const int32_t* wtab = build_win_table(B, n, P, ktot, SL.win, &nw, s);
  CoPlan pl{labels, n, P, B.k_off, B.members, B.pos, B.cstart, wtab, nw, nullptr, co_ranges(n), 1};
  CoOut o{};
  o.row_ctr = B.ctr;
  o.row_nnz = B.row_nnz;
  o.max_count = B.misc + 1;
  o.seg = reinterpret_cast<uint64_t*>(st + kStageHdr);
  o.pool = reinterpret_cast<uint32_t*>(st + SL.pool_at);
  o.pool_ctr = reinterpret_cast<unsigned long long*>(hdr + 2);
  o.pool_cap = (int64_t)((stage_bytes - SL.pool_at) / 4);
  o.pool_chunk = chunk;
  o.overflow = reinterpret_cast<unsigned int*>(hdr + 3);
  int pr = prof_begin(EAC_PROF_CO_STAGE, 0, s);
  // (PASS 3 apart: the choice inside PASS 2 cost its emission 1.7%)
  EAC_TRY(chunk ? co_launch<2>(pl, full_rows, SL.win, o, s)
                : co_launch<3>(pl, full_rows, SL.win, o, s));
  prof_end(pr, s);
  EAC_TRY((scan_excl<int32_t, int64_t>(B.row_nnz, indptr, n + 1, 0, nullptr, ar, s)));
  ar.used = mark;
  k_co_finish<<<1, 64, 0, s>>>(indptr, n, B.misc, hdr, cap_nnz, d_out);
  EAC_LAUNCH_CHECK();
  int pr2 = prof_begin(EAC_PROF_CO_COMPACT, 0, s);
  const int64_t blocks = (n + 3) / 4;
  k_coassoc_compact<<<(unsigned)(blocks < 65536 ? blocks : 65536), 256, 0, s>>>(
      st, indptr, n, w_offset, indices, data, d_out);
  EAC_LAUNCH_CHECK();
  prof_end(pr2, s);
  return EAC_OK;
}

// ------------------------------------------------ capacity-capped selection
// The reference's EAC_CSR gives row r a fixed capacity (cap_off[r+1] -
// cap_off[r] condensed, max_assocs with full rows) and, processing the
// partitions in their order (the one with the fewest clusters first), adds
// a new column to a row only while the row is below capacity; a column met
// when the row is full is discarded, and discarded again at each later
// co-occurrence (sparse.py:956-1040 / :866-950). Rows never shrink, so a row
// keeps exactly the first `cap` of its columns in the order (rank of the
// first partition with the pair, column), and each kept column ends with
// its full count. From the exact matrix with per-entry ranks, the kept set
// of a row is {rank < R*} plus the first `need` columns of rank R*, where
// R* is the smallest rank whose cumulative entry count reaches cap. Full
// rows above id 405109 keep only the first partition's entries at count 1
// (the update returns before them, sparse.py:877-878). A first partition
// that gives a row more entries than its capacity makes the reference write
// past the row: reported as an error.
namespace eac {
namespace {
constexpr int kCapB = 256;
constexpr int64_t kDebugRow = 405109;

__global__ __launch_bounds__(kCapB) void k_cap_select(const int64_t* __restrict__ indptr,
                                                      const int32_t* __restrict__ rank,
                                                      int64_t n, int P, int full_rows,
                                                      const int64_t* __restrict__ cap_off,
                                                      int64_t max_assocs,
                                                      int32_t* __restrict__ kept,
                                                      int32_t* __restrict__ rstar,
                                                      int32_t* __restrict__ need,
                                                      unsigned long long* __restrict__ bad_row) {
  extern __shared__ int32_t s_hist[];  // P bins
  __shared__ int32_t s_tmp[kCapB / kWave + 1];
  __shared__ int32_t s_sel[2];
  const int t = threadIdx.x;
  for (int64_t i = blockIdx.x; i < n; i += gridDim.x) {
    const int64_t a = indptr[i], b = indptr[i + 1], total = b - a;
    const int64_t cap = full_rows ? max_assocs : cap_off[i + 1] - cap_off[i];
    const bool debug_row = full_rows && i > kDebugRow;
    if (total <= cap && !debug_row) {  // block-uniform: the row fits
      if (t == 0) {
        kept[i] = (int32_t)total;
        rstar[i] = INT32_MAX;
        need[i] = 0;
      }
      continue;
    }
    for (int v = t; v < P; v += kCapB) s_hist[v] = 0;
    if (t == 0) { s_sel[0] = 0; s_sel[1] = 0; }
    __syncthreads();
    for (int64_t e = a + t; e < b; e += kCapB) {
      const int32_t R = rank[e];
      if ((uint32_t)R < (uint32_t)P) atomicAdd(&s_hist[R], 1);
      else atomicAdd(&bad_row[3], 1ull);  // a rank outside [0, P): rejected by the caller
    }
    __syncthreads();
    const int32_t n0 = s_hist[0];
    if (t == 0 && n0 > cap) atomicMin(bad_row, (unsigned long long)i);
    if (debug_row) {
      if (t == 0) {
        kept[i] = n0;
        rstar[i] = 1;  // keep rank 0 only
        need[i] = 0;
      }
    } else {
      // contiguous bins per thread, block scan of their sums
      const int per = (P + kCapB - 1) / kCapB;
      const int b0 = t * per, b1 = b0 + per < P ? b0 + per : P;
      int32_t mine = 0;
      for (int r = b0; r < b1; ++r) mine += s_hist[r];
      int32_t tot;
      int32_t cum = block_excl_scan<int32_t>(mine, s_tmp, &tot);
      for (int r = b0; r < b1; ++r) {
        if (cum < cap && cum + s_hist[r] >= cap) {
          s_sel[0] = r;
          s_sel[1] = (int32_t)(cap - cum);
        }
        cum += s_hist[r];
      }
      __syncthreads();
      if (t == 0) {
        kept[i] = (int32_t)cap;
        rstar[i] = cap > 0 ? s_sel[0] : 0;
        need[i] = cap > 0 ? s_sel[1] : 0;
      }
    }
    __syncthreads();
  }
}

__global__ __launch_bounds__(kCapB) void k_cap_compact(
    const int64_t* __restrict__ indptr, const int32_t* __restrict__ indices,
    const int32_t* __restrict__ count, const int32_t* __restrict__ rank, int64_t n,
    int full_rows, const int32_t* __restrict__ rstar, const int32_t* __restrict__ need,
    const int64_t* __restrict__ out_off, int32_t* __restrict__ out_col,
    int32_t* __restrict__ out_val, unsigned long long* __restrict__ discarded,
    unsigned int* __restrict__ max_kept) {
  __shared__ int32_t s_tmp[kCapB / kWave + 1];
  const int t = threadIdx.x;
  unsigned long long disc = 0;
  unsigned int mx = 0;
  for (int64_t i = blockIdx.x; i < n; i += gridDim.x) {
    const int64_t a = indptr[i], b = indptr[i + 1], o = out_off[i];
    const int32_t rs = rstar[i], nd = need[i];
    const bool debug_row = full_rows && i > kDebugRow;
    if (rs == INT32_MAX) {  // the whole row is kept
      for (int64_t e = a + t; e < b; e += kCapB) {
        const int32_t v = count[e];
        out_col[o + (e - a)] = indices[e];
        out_val[o + (e - a)] = v;
        mx = (unsigned)v > mx ? (unsigned)v : mx;
      }
      continue;
    }
    int32_t carry_star = 0, carry_keep = 0;
    for (int64_t base = a; base < b; base += kCapB) {  // block-uniform trip count
      const int64_t e = base + t;
      const bool valid = e < b;
      const int32_t R = valid ? rank[e] : INT32_MAX;
      const int32_t is_star = valid && R == rs;
      int32_t star_tot, keep_tot;
      const int32_t idx = carry_star + block_excl_scan<int32_t>(is_star, s_tmp, &star_tot);
      const int32_t keep = valid && (R < rs || (is_star && idx < nd));
      const int32_t pos = carry_keep + block_excl_scan<int32_t>(keep, s_tmp, &keep_tot);
      if (keep) {
        const int32_t v = debug_row ? 1 : count[e];
        out_col[o + pos] = indices[e];
        out_val[o + pos] = v;
        mx = (unsigned)v > mx ? (unsigned)v : mx;
      } else if (valid && !debug_row) {
        disc += (unsigned long long)count[e];
      }
      carry_star += star_tot;
      carry_keep += keep_tot;
    }
  }
  disc = wave_sum(disc);
  for (int off = kWave / 2; off > 0; off >>= 1) {
    const unsigned int o2 = __shfl_xor(mx, off, kWave);
    mx = o2 > mx ? o2 : mx;
  }
  if (lane_id() == 0) {
    if (disc) atomicAdd(discarded, disc);
    if (mx) atomicMax(max_kept, mx);
  }
}

struct CapBufs {
  int32_t* kept;
  int32_t* rstar;
  int32_t* need;
  unsigned long long* misc;  // [0] bad row (min), [1] discarded, [2] max kept, [3] bad ranks
};

CapBufs carve_cap(Arena& ar, int64_t n) {
  CapBufs c;
  c.kept = ar.take<int32_t>(n + 1);
  c.rstar = ar.take<int32_t>(n);
  c.need = ar.take<int32_t>(n);
  c.misc = ar.take<unsigned long long>(4);
  return c;
}
}  // namespace
}  // namespace eac

extern "C" size_t eac_coassoc_cap_workspace_bytes(int64_t n) {
  if (n < 1) n = 1;
  Arena ar(nullptr, 0, true);
  (void)carve_cap(ar, n);
  return ar.used + scan_ws_bytes(n + 1, 8) + 4096;
}

extern "C" int eac_coassoc_cap(const int64_t* indptr, const int32_t* indices,
                               const int32_t* count, const int32_t* rank, int64_t n, int32_t P,
                               int32_t full_rows, const int64_t* cap_off, int64_t max_assocs,
                               int64_t out_capacity, int64_t* out_indptr, int32_t* out_indices,
                               int32_t* out_data, int64_t* h_out, void* ws, size_t ws_bytes,
                               void* stream) {
  if (n < 1 || P < 1 || P > kMaxP) return fail(EAC_ERR_ARG, "coassoc cap: need n >= 1, 1 <= P <= %d", kMaxP);
  if (!indptr || !count || !rank || !out_indptr || (!full_rows && !cap_off))
    return fail(EAC_ERR_ARG, "coassoc cap: null array");
  if (full_rows && max_assocs < 0) return fail(EAC_ERR_ARG, "coassoc cap: max_assocs < 0");
  const size_t need_ws = eac_coassoc_cap_workspace_bytes(n);
  if (!ws || ws_bytes < need_ws)
    return fail(EAC_ERR_WORKSPACE, "coassoc cap: workspace %zu < %zu bytes", ws_bytes, need_ws);
  hipStream_t s = (hipStream_t)stream;
  Arena ar(ws, ws_bytes);
  CapBufs B = carve_cap(ar, n);
  const size_t mark = ar.used;
  uint64_t* misc64 = reinterpret_cast<uint64_t*>(B.misc);
  EAC_TRY(fill<uint64_t>(misc64, 4, 0ull, s));
  EAC_TRY(fill<uint64_t>(misc64, 1, ~0ull, s));
  EAC_TRY(fill<int32_t>(B.kept + n, 1, 0, s));
  const int g = grid_for(n, 1, 4096);
  k_cap_select<<<g, kCapB, sizeof(int32_t) * P, s>>>(indptr, rank, n, P, full_rows, cap_off,
                                                     max_assocs, B.kept, B.rstar, B.need, B.misc);
  EAC_LAUNCH_CHECK();
  EAC_TRY((scan_excl<int32_t, int64_t>(B.kept, out_indptr, n + 1, 0, nullptr, ar, s)));
  ar.used = mark;
  unsigned long long bad[4] = {0, 0, 0, 0};
  int64_t total = 0;
  EAC_TRY(d2h(bad, B.misc, sizeof(bad), s));
  EAC_TRY(d2h(&total, out_indptr + n, sizeof(total), s));
  if (bad[3]) return fail(EAC_ERR_ARG, "coassoc cap: %llu ranks outside [0, P)", bad[3]);
  if (bad[0] != ~0ull)
    return fail(EAC_ERR_VALUE,
                "coassoc cap: the first partition gives row %llu more entries than its "
                "capacity (the reference writes past the row)", bad[0]);
  if (total > out_capacity)
    return fail(EAC_ERR_ARG, "coassoc cap: %lld kept entries exceed the output capacity %lld",
                (long long)total, (long long)out_capacity);
  if (total > 0 && (!out_indices || !out_data))
    return fail(EAC_ERR_ARG, "coassoc cap: null output");
  k_cap_compact<<<g, kCapB, 0, s>>>(indptr, indices, count, rank, n, full_rows, B.rstar, B.need,
                                    out_indptr, out_indices, out_data, B.misc + 1,
                                    reinterpret_cast<unsigned int*>(B.misc + 2));
  EAC_LAUNCH_CHECK();
  unsigned long long misc[3];
  EAC_TRY(d2h(misc, B.misc, sizeof(misc), s));
  if (h_out) {
    h_out[0] = total;
    h_out[1] = (int64_t)misc[1];
    h_out[2] = (int64_t)(unsigned int)misc[2];
    h_out[3] = -1;
  }
  return EAC_OK;
}
