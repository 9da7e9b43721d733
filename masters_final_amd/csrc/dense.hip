// Dense co-association (EAC_FULL) and single linkage over it, for small n.
//
// Reference: MyML/MyML/EAC/full.py:8-181 (EAC_FULL: counts of every pair of
// samples, condensed or n x n, make_diassoc val - count),
// MyML/MyML/EAC/eac.py:337-391 (full_sl_lifetime: SLINK, the lifetime rule
// lifetime_n_clusters on the float32 heights, labels from Z),
// MyML/MyML/cluster/linkage.py:144-149 (SL: the SLINK wrapper returning the
// float32 linkage matrix Z) and :303-357 (labels_from_Z_numba: the first
// n - n_clusters merges, clusters numbered by first occurrence),
// scipy_numba/scipy_numba/cluster/_hierarchy_eac.py:842-927 (SLINK and
// from_pointer_representation).
//
// MI355X design:
//  * Counts: the labels of 32 partitions become bit planes of a sample, so
//    one three-input operation a plane compares 32 labels of a pair; tiles of
//    64 x 128 pairs, the planes of both sides staged in LDS, 4 x 8 counts a
//    thread in registers.
//  * The single-linkage dendrogram is the minimum spanning tree's merges in
//    height order. The dense graph is complete, so Borůvka needs at most
//    bits(n - 1) rounds; each round streams the n x n matrix at most once (a
//    wavefront per row, the columns' component ids in LDS), and up to 12,288
//    points one workgroup does the rest of it in LDS. Keys (weight word, min
//    id, max id) are a strict total order: the tree is unique and a mutual
//    choice is the only cycle (the smaller root stays root). A flag on the
//    device ends the rounds.
//  * The lifetime rule runs in one workgroup over the sorted heights; the
//    labels of the cut are a parallel union-find, up to 16,384 points in one
//    workgroup's LDS (roots are component
//    minima, so a scan of the root flags numbers components by first
//    occurrence). The linkage matrix Z, when asked for, is built by one
//    thread from the sorted tree edges with a union-find in LDS; rows of
//    equal height come in (height, min id, max id) order.
#include <algorithm>

#include "prims.hpp"
#include "sort.hpp"

namespace eac {
namespace {

constexpr int kDT = 64;    // samples a tile side (label words, square copy)
constexpr int kCC = 128;   // columns of a count tile (its rows: kDT)
constexpr int kStage = 32; // partitions a label word holds
constexpr int64_t kDenseMaxN = 65536;  // 16-bit ids in the Borůvka keys

__host__ __device__ __forceinline__ int64_t cidx(int64_t n, int64_t i, int64_t j) {
  return n * i - (i * (i + 1)) / 2 + (j - i - 1);  // i < j
}

// Labels as bit planes: of 32 partitions, word 0 holds the bits of those that
// list the sample (label >= 0) and word 1 + b their labels' bits b. Two
// samples' unequal partitions are then not(both listed) or an or over the
// planes of x ^ y: one three-input operation a plane for 32 comparisons, where
// comparing labels takes a compare and an add each.
constexpr int kPlanes = 32;  // listed, and the 31 bits of a label

// The 32 labels of sample x from partition p0 on, as words (w[0] listed,
// w[1 + b] plane b). Returns the or of the labels.
__device__ __forceinline__ uint32_t label_words(const int32_t* __restrict__ labels, int64_t n,
                                                int P, int p0, int64_t x, uint32_t (&w)[kPlanes],
                                                uint32_t& listed) {
  uint32_t any = 0;
  listed = 0;
#pragma unroll
  for (int p = 0; p < kStage; ++p)
    w[p] = x < n && p0 + p < P ? (uint32_t)labels[(int64_t)(p0 + p) * n + x] : ~0u;
#pragma unroll
  for (int p = 0; p < kStage; ++p) {
    const bool in = (int32_t)w[p] >= 0;
    listed |= in ? 1u << p : 0u;
    w[p] = in ? w[p] : 0u;
    any |= w[p];
  }
  // bit b of label p becomes bit p of word b: the 32 x 32 bit-matrix
  // transposition by halves of Hacker's Delight (Warren, section 7-3), blocks
  // of 16, 8, 4, 2 and 1 swapped across the diagonal
#pragma unroll
  for (int j = 16, m = 0xffff; j > 0; j >>= 1, m ^= m << j) {
#pragma unroll
    for (int k = 0; k < 32; ++k) {
      if (k & j) continue;
      const uint32_t t = ((w[k] >> j) ^ w[k + j]) & (uint32_t)m;
      w[k + j] ^= t;
      w[k] ^= t << j;
    }
  }
  return any;
}

// planes[stage][kPlanes][npad] and, per 64 samples, the bits in use.
__global__ __launch_bounds__(kDT) void k_label_planes(const int32_t* __restrict__ labels,
                                                      int64_t n, int P, int64_t npad,
                                                      uint32_t* __restrict__ planes,
                                                      int32_t* __restrict__ bits) {
  const int64_t x = (int64_t)blockIdx.x * kDT + threadIdx.x;
  uint32_t w[kPlanes], listed;
  uint32_t any = label_words(labels, n, P, blockIdx.y * kStage, x, w, listed);
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) any |= __shfl_xor(any, off, kWave);
  const int nb = any ? 32 - __builtin_clz(any) : 0;
  uint32_t* out = planes + (int64_t)blockIdx.y * kPlanes * npad + x;
  out[0] = listed;
#pragma unroll
  for (int b = 0; b < kPlanes - 1; ++b)
    if (b < nb) out[(int64_t)(1 + b) * npad] = w[b];
  if (threadIdx.x == 0) bits[(int64_t)blockIdx.y * gridDim.x + blockIdx.x] = nb;
}

// Counts of a tile of 64 rows and 128 columns, 4 x 8 pairs a thread, from the
// planes, or (PLANES false: the caller's workspace has no room for them) from
// labels the workgroup transposes itself, which takes longer than the counting.
// A row of tiles stays on one XCD, so neighbouring tiles' pieces of a line meet
// in its L2. Bound by the vector units: (planes + 2) operations a pair and 32
// partitions. 8,000 samples, 100 partitions of 50 to 200 clusters: 68 us and 6
// for the planes, where comparing labels one by one took 212. ADD: the matrix receives the sums of its own values and the counts
// (uint8 wraps as numpy's += does), and no maximum is taken.
template <typename T, bool ADD, bool PLANES>
__global__ __launch_bounds__(256, PLANES ? 4 : 2) void k_dense_counts(
    const int32_t* __restrict__ labels, int64_t n, int P, int condensed,
    const uint32_t* __restrict__ planes, const int32_t* __restrict__ bits, int64_t npad,
    T* __restrict__ out, unsigned int* __restrict__ max_count) {
  // workgroups go to the XCDs in turn (eight a column of tiles): rows of tiles
  // up and down over them
  const int turn = blockIdx.y, xcd = blockIdx.x % 8, tj = blockIdx.x / 8;
  const int ti = turn * 8 + (turn & 1 ? 7 - xcd : xcd);
  const int64_t i0 = (int64_t)ti * kDT, j0 = (int64_t)tj * kCC;
  if (i0 >= n || j0 + kCC <= i0) return;  // below the diagonal (block-uniform)
  __shared__ __align__(16) uint32_t s_r[kPlanes][kDT];
  __shared__ __align__(16) uint32_t s_c[kPlanes][kCC];
  __shared__ unsigned int s_mx, s_any;
  const int t = threadIdx.x, ty = t / 16, tx = t % 16;
  const int stages = (P + kStage - 1) / kStage;
  const int64_t i = i0 + ty * 4, j = j0 + tx * 8;
  uint32_t cnt[4][8];  // unequal or not listed
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 8; ++b) cnt[a][b] = 0;
  if (t == 0) s_mx = 0;
  // the matrix's own values, on their way during the counting
  T old[4][8];
  auto whole = [&](int a) { return i + a < n && j > i + a && j + 8 <= n; };
  auto row = [&](int a) { return out + (condensed ? cidx(n, i + a, j) : (i + a) * n + j); };
  if (ADD) {
#pragma unroll
    for (int a = 0; a < 4; ++a)
      if (whole(a)) __builtin_memcpy(old[a], row(a), sizeof(old[a]));
  }
  auto count = [&](int pl0, int nb) {
    uint32_t ne[4][8], r[4], c[8];
    auto read = [&](int pl) {
      *reinterpret_cast<uint4*>(r) = *reinterpret_cast<const uint4*>(&s_r[pl][ty * 4]);
      *reinterpret_cast<uint4*>(c) = *reinterpret_cast<const uint4*>(&s_c[pl][tx * 8]);
      *reinterpret_cast<uint4*>(c + 4) = *reinterpret_cast<const uint4*>(&s_c[pl][tx * 8 + 4]);
    };
    read(pl0);
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 8; ++b) ne[a][b] = ~(r[a] & c[b]);
    for (int pl = pl0 + 1; pl <= pl0 + nb; ++pl) {
      read(pl);
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 8; ++b) ne[a][b] |= r[a] ^ c[b];
    }
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 8; ++b) cnt[a][b] += __popc(ne[a][b]);
  };
  for (int st = 0; st < stages; ++st) {
    int nb;
    if constexpr (PLANES) {
      const int64_t tiles = npad / kDT, ct = j0 / kDT;
      const int32_t* bt = bits + (int64_t)st * tiles;
      const int nr = bt[ti], c0 = bt[ct], c1 = ct + 1 < tiles ? bt[ct + 1] : -1;
      nb = max(max(c0, c1), nr);
      const uint32_t* src = planes + (int64_t)st * kPlanes * npad;
      __syncthreads();  // the previous stage is counted
      for (int v = t; v < (nb + 1) * kDT; v += 256) {
        const int pl = v / kDT, x = v % kDT;
        s_r[pl][x] = pl <= nr ? src[pl * npad + i0 + x] : 0u;
      }
      for (int v = t; v < (nb + 1) * kCC; v += 256) {
        const int pl = v / kCC, x = v % kCC;
        s_c[pl][x] = pl <= (x < kDT ? c0 : c1) ? src[pl * npad + j0 + x] : 0u;
      }
    } else {
      __syncthreads();  // the previous stage is counted
      if (t == 0) s_any = 0;
      __syncthreads();
      uint32_t w[kPlanes], listed, any = 0;
      if (t < kDT + kCC)
        any = label_words(labels, n, P, st * kStage, t < kDT ? i0 + t : j0 + t - kDT, w, listed);
      if (any) atomicOr(&s_any, any);
      __syncthreads();
      nb = s_any ? 32 - __builtin_clz(s_any) : 0;
      if (t < kDT + kCC) {
        uint32_t* dst = t < kDT ? &s_r[0][t] : &s_c[0][t - kDT];
        const int ld = t < kDT ? kDT : kCC;
        dst[0] = listed;
#pragma unroll
        for (int b = 0; b < kPlanes - 1; ++b)
          if (b < nb) dst[(1 + b) * ld] = w[b];
      }
    }
    __syncthreads();
    count(0, nb);
  }
  unsigned int mx = 0;
  const uint32_t all = 32u * stages;
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    if (i + a >= n) break;
    T v[8];
#pragma unroll
    for (int b = 0; b < 8; ++b) v[b] = (T)(all - cnt[a][b]);  // uint8 wraps as numpy's += 1 does
    T* to = row(a);
    if (whole(a)) {  // eight neighbours at once, whatever their alignment
#pragma unroll
      for (int b = 0; b < 8; ++b) {
        if (ADD) v[b] = (T)(v[b] + old[a][b]);
        else mx = max(mx, (unsigned)v[b]);
      }
      __builtin_memcpy(to, v, sizeof(v));
    } else {
#pragma unroll
      for (int b = 0; b < 8; ++b) {
        if (j + b >= n) continue;
        if (j + b > i + a) {
          to[b] = ADD ? (T)(v[b] + to[b]) : v[b];
          mx = max(mx, (unsigned)v[b]);
        } else if (!ADD && !condensed && j + b == i + a) {
          to[b] = (T)0;
        }
      }
    }
  }
  if (!condensed) {  // the mirrored entries, four neighbours a column
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      if (j + b >= n) break;
      T v[4];
#pragma unroll
      for (int a = 0; a < 4; ++a) v[a] = (T)(all - cnt[a][b]);
      T* to = out + (j + b) * n + i;
      if (i + 4 <= j + b) {
        if (ADD) {
          T o[4];
          __builtin_memcpy(o, to, sizeof(o));
#pragma unroll
          for (int a = 0; a < 4; ++a) v[a] = (T)(v[a] + o[a]);
        }
        __builtin_memcpy(to, v, sizeof(v));
      } else {
#pragma unroll
        for (int a = 0; a < 4; ++a)
          if (i + a < j + b) to[a] = ADD ? (T)(v[a] + to[a]) : v[a];
      }
    }
  }
  if (ADD || !max_count) return;  // uniform
  for (int off = kWave / 2; off > 0; off >>= 1) {
    const unsigned int o = __shfl_xor(mx, off, kWave);
    mx = o > mx ? o : mx;
  }
  if (lane_id() == 0 && mx) atomicMax(&s_mx, mx);
  __syncthreads();
  // (a plain read first: the tiles' maxima are mostly not larger)
  if (t == 0 && s_mx > *(volatile unsigned int*)max_count) atomicMax(max_count, s_mx);
}

// make_diassoc_1d / _2d (full.py:98-112): a[i] = val - a[i], stored in the
// matrix dtype (integer types wrap, as the reference's store does). With top
// (the largest value, see k_dense_max) val = int(*top) + 1. 16 bytes a lane
// where the array is aligned.
template <typename T>
struct alignas(16) Pack16 {
  T v[16 / sizeof(T)];
};
template <typename T>
__device__ __forceinline__ T diassoc_of(T a, double val) {
  if (T(0.5) == T(0))  // integer type: int64 arithmetic, modular store
    return (T)((int64_t)val - (int64_t)a);
  return (T)(val - (double)a);
}
template <typename T>
__global__ void k_dense_diassoc(T* __restrict__ a, int64_t len, double val,
                                const unsigned long long* __restrict__ top) {
  constexpr int V = 16 / sizeof(T);
  if (top) {
    const long long w = (long long)(*top - 0x8000000000000000ull);
    val = (double)(w + 1);
  }
  const bool vec = (reinterpret_cast<uintptr_t>(a) & 15) == 0;
  const int64_t head = vec ? len / V : 0, stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t t0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  Pack16<T>* p = reinterpret_cast<Pack16<T>*>(a);
  for (int64_t i = t0; i < head; i += stride) {
    Pack16<T> x = p[i];
#pragma unroll
    for (int u = 0; u < V; ++u) x.v[u] = diassoc_of(x.v[u], val);
    p[i] = x;
  }
  for (int64_t i = head * V + t0; i < len; i += stride) a[i] = diassoc_of(a[i], val);
}

// Largest int(value) of the array into *top (biased by 2^63 so that unsigned
// order is signed order; cleared by the caller).
template <typename T>
__global__ __launch_bounds__(1024) void k_dense_max(const T* __restrict__ a, int64_t len,
                                                   unsigned long long* __restrict__ top) {
  constexpr int V = 16 / sizeof(T);
  const bool vec = (reinterpret_cast<uintptr_t>(a) & 15) == 0;
  const int64_t head = vec ? len / V : 0, stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t t0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const Pack16<T>* p = reinterpret_cast<const Pack16<T>*>(a);
  T m = a[0];
  for (int64_t i = t0; i < head; i += stride) {
    const Pack16<T> x = p[i];
#pragma unroll
    for (int u = 0; u < V; ++u) m = x.v[u] > m ? x.v[u] : m;
  }
  for (int64_t i = head * V + t0; i < len; i += stride) m = a[i] > m ? a[i] : m;
  __shared__ unsigned long long s_w[1024 / kWave];
  unsigned long long w = (unsigned long long)(long long)m + 0x8000000000000000ull;
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) {
    const unsigned long long o = __shfl_xor(w, off, kWave);
    w = o > w ? o : w;
  }
  if (lane_id() == 0) s_w[threadIdx.x / kWave] = w;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int u = 1; u < 1024 / kWave; ++u) w = s_w[u] > w ? s_w[u] : w;
    // (a plain read first: same-address atomics serialise, and most are not larger)
    if (w > *(volatile unsigned long long*)top) atomicMax(top, w);
  }
}

// Row stride of the square copy: rows on 64 bytes, so the row scans read
// whole aligned pieces; the padding holds the largest weight word.
__host__ __device__ inline int64_t sq_stride(int64_t n) { return (n + 63) & ~int64_t(63); }

// Square copy of a condensed matrix (both triangles; the diagonal is not
// read): 64 x 64 tiles through LDS so both the row-major read and the
// transposed write are coalesced, four columns a lane.
template <typename T>
__global__ __launch_bounds__(256) void k_square_from_condensed(const T* __restrict__ cond,
                                                               int64_t n, T pad,
                                                               T* __restrict__ sq) {
  const int ti = blockIdx.y, tj = blockIdx.x;
  if (ti > tj) return;
  struct alignas(4 * sizeof(T)) Four {
    T v[4];
  };
  __shared__ T s[kDT][kDT + 4 / sizeof(T)];
  const int64_t i0 = (int64_t)ti * kDT, j0 = (int64_t)tj * kDT, ld = sq_stride(n);
  for (int v = threadIdx.x; v < kDT * kDT / 4; v += 256) {
    const int a = v / (kDT / 4), b = (v % (kDT / 4)) * 4;
    const int64_t i = i0 + a, j = j0 + b;
    Four x;
    if (i < n && j > i && j + 4 <= n) {
      __builtin_memcpy(&x, cond + cidx(n, i, j), sizeof(x));
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        x.v[u] = pad;
        if (i < n && j + u < n && j + u > i) x.v[u] = cond[cidx(n, i, j + u)];
        else if (i < n && j + u < n && j + u < i) x.v[u] = cond[cidx(n, j + u, i)];  // diagonal tile
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) s[a][b + u] = x.v[u];
    if (i < n) *reinterpret_cast<Four*>(sq + i * ld + j) = x;
  }
  if (ti == tj) return;
  __syncthreads();
  for (int v = threadIdx.x; v < kDT * kDT / 4; v += 256) {
    const int a = v / (kDT / 4), b = (v % (kDT / 4)) * 4;  // row j0 + a, columns i0 + b ...
    const int64_t j = j0 + a;
    Four x;
#pragma unroll
    for (int u = 0; u < 4; ++u) x.v[u] = s[b + u][a];
    if (j < n) *reinterpret_cast<Four*>(sq + j * ld + i0 + b) = x;  // (i0 + 63 < n here)
  }
}

// Order-preserving 32-bit word of a weight.
__device__ __forceinline__ uint32_t wword(uint8_t w) { return w; }
__device__ __forceinline__ uint32_t wword(uint16_t w) { return w; }
__device__ __forceinline__ uint32_t wword(int32_t w) { return (uint32_t)w ^ 0x80000000u; }
__device__ __forceinline__ uint32_t wword(float w) {
  const uint32_t b = __float_as_uint(w);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
// float32 value of a weight word (the reference's float32 Z heights)
template <typename T>
__device__ __forceinline__ float wvalue(uint32_t x);
template <>
__device__ __forceinline__ float wvalue<uint8_t>(uint32_t x) { return (float)x; }
template <>
__device__ __forceinline__ float wvalue<uint16_t>(uint32_t x) { return (float)x; }
template <>
__device__ __forceinline__ float wvalue<int32_t>(uint32_t x) {
  return (float)(int32_t)(x ^ 0x80000000u);
}
template <>
__device__ __forceinline__ float wvalue<float>(uint32_t x) {
  return __uint_as_float((x & 0x80000000u) ? (x & 0x7fffffffu) : ~x);
}

// One Borůvka step's minima: for every row u the lightest (weight, column) to
// another component. Among equal weights the smallest column is also the
// smallest (min id, max id) key, so a row needs no more than its columns in
// order. A wavefront per row; the columns' component ids (16 bits) sit in LDS
// once per workgroup. 16 bytes of weights a lane and load: for one-byte
// weights three vector operations a column (64 M columns of 8,000 points: 5 us
// of issue a round, 14 of memory at the copy rate; measured 18, with one byte
// a lane and load 64). ld: row stride of sq.
// A row whose last minimum still leads to another component keeps it: the
// columns it may choose from only get fewer. minv must start as all ones.
// done[0]: set when one component is left.
constexpr int kRowB = 1024;
template <typename T>
__global__ __launch_bounds__(kRowB) void k_dense_rowmin(const T* __restrict__ sq, int64_t n,
                                                        int64_t ld,
                                                        const uint16_t* __restrict__ comp,
                                                        unsigned long long* __restrict__ minv,
                                                        const int32_t* __restrict__ done) {
  if (done[0]) return;  // uniform over the grid
  extern __shared__ __align__(16) uint16_t s_comp[];
  constexpr int V = 16 / sizeof(T), Q = 4;  // columns a piece, pieces in flight
  typedef uint32_t Raw __attribute__((ext_vector_type(4)));
  typedef uint16_t U16x2 __attribute__((ext_vector_type(2)));
  const int64_t nv = (n + V - 1) / V * V;
  const int w = threadIdx.x / kWave, l = lane_id();
  const int64_t full = ld >= nv ? nv : n / V * V;  // columns covered by whole pieces
  Raw x[Q];
  auto load = [&](int64_t u, int64_t g) {
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int64_t v0 = g + ((int64_t)q * kWave + l) * V;
      // (rows of an n x n matrix start on any byte)
      if (v0 < full) __builtin_memcpy(&x[q], sq + u * ld + v0, sizeof(Raw));
    }
  };
  int64_t u = (int64_t)blockIdx.x * (kRowB / kWave) + w;
  const int64_t step = (int64_t)gridDim.x * (kRowB / kWave);
  if (u < n) load(u, 0);  // on its way while the ids are staged
  for (int64_t v = threadIdx.x; v < nv; v += kRowB) s_comp[v] = v < n ? comp[v] : 0xffffu;
  __syncthreads();
  for (bool first = true; u < n; u += step, first = false) {
    const uint32_t cu = s_comp[u], cu2 = cu << 16 | cu;
    const unsigned long long was = minv[u];
    if (was != ~0ull) {
      const uint32_t a = (was >> 16) & 0xffffu, b = was & 0xffffu;
      if (s_comp[a == (uint32_t)u ? b : a] != cu) continue;  // uniform over the wavefront
    }
    const T* row = sq + u * ld;
    unsigned long long best = ~0ull;  // weight word << 16 | column
    for (int64_t g = 0; g < full; g += Q * kWave * V) {
      if (!first || g) load(u, g);
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int64_t v0 = g + ((int64_t)q * kWave + l) * V;
        if (v0 >= full) continue;
        if constexpr (sizeof(T) == 1) {
          // two columns a word: (weight << 8 | position in the piece), all ones
          // where the column is in the row's own component
          const uint4 c0 = *reinterpret_cast<const uint4*>(s_comp + v0);
          const uint4 c1 = *reinterpret_cast<const uint4*>(s_comp + v0 + 8);
          const uint32_t c[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
          U16x2 m = {0xffff, 0xffff};
#pragma unroll
          for (int e = 0; e < 16; e += 2) {
            const U16x2 d = __builtin_bit_cast(U16x2, c[e >> 1] ^ cu2);
            const U16x2 own = __builtin_elementwise_min(d, U16x2{1, 1}) - U16x2{1, 1};
            const uint32_t wb = __builtin_amdgcn_perm(
                0u, x[q][e >> 2], (uint32_t)(e & 2 ? 0x030c020cu : 0x010c000cu));
            const U16x2 k = __builtin_bit_cast(
                U16x2, wb | __builtin_bit_cast(uint32_t, own) | (uint32_t)(e | (e + 1) << 16));
            m = __builtin_elementwise_min(m, k);
          }
          const uint32_t k16 = m.x < m.y ? m.x : m.y;
          if (k16 != 0xffffu) {
            const unsigned long long k =
                ((unsigned long long)(k16 >> 8) << 16) | (uint32_t)(v0 + (k16 & 15u));
            best = k < best ? k : best;
          }
        } else {
          T tv[V];
          __builtin_memcpy(tv, &x[q], 16);
#pragma unroll
          for (int e = 0; e < V; ++e) {
            const unsigned long long k =
                ((unsigned long long)wword(tv[e]) << 16) | (uint32_t)(v0 + e);
            best = s_comp[v0 + e] != cu && k < best ? k : best;
          }
        }
      }
    }
    for (int64_t v = full + l; v < n; v += kWave) {
      const unsigned long long k = ((unsigned long long)wword(row[v]) << 16) | (uint32_t)v;
      best = s_comp[v] != cu && k < best ? k : best;
    }
    best = wave_min_u64(best);
    if (l == 0) {
      const uint64_t v = best & 0xffffu;
      // (a column past n is padding: no other component is left)
      const uint64_t lo = (uint64_t)u < v ? (uint64_t)u : v, hi = (uint64_t)u < v ? v : (uint64_t)u;
      minv[u] = best == ~0ull || (int64_t)v >= n
                    ? ~0ull
                    : ((best >> 16) << 32) | (lo << 16) | hi;
    }
  }
}

// The rest of a round for n <= kMergeN in one workgroup: every component's
// lightest key (64-bit minima in LDS, each tried only when it improves the
// value read, since atomics on one address serialise), the hooking (of a
// mutual choice the smaller root stays) and the new component ids.
// done[1] counts the edges of the tree: n - 1 end the rounds. A thread's
// vertices stay in registers over the steps. 7 us at 8,000 vertices, bound by
// the latency of its five steps; the separate launches took 15 and a fill.
constexpr int64_t kMergeN = 12288;  // 8 + 2 bytes of LDS a vertex
__global__ __launch_bounds__(1024) void k_dense_merge(int64_t n, uint16_t* __restrict__ comp,
                                                      const unsigned long long* __restrict__ minv,
                                                      unsigned long long* __restrict__ tree,
                                                      int32_t* __restrict__ done) {
  if (done[0]) return;
  extern __shared__ __align__(16) unsigned long long s_best[];
  uint16_t* s_par = reinterpret_cast<uint16_t*>(s_best + n);
  __shared__ int s_hooked;
  constexpr int U = kMergeN / 1024;
  const int t = threadIdx.x, m = (int)n;
  unsigned long long k[U];
  uint32_t c[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int v = u * 1024 + t;
    k[u] = v < m ? minv[v] : ~0ull;
    c[u] = v < m ? comp[v] : 0u;
    if (v < m) {
      s_best[v] = ~0ull;
      s_par[v] = (uint16_t)v;
    }
  }
  if (t == 0) s_hooked = 0;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (u * 1024 < m && k[u] < *(volatile unsigned long long*)&s_best[c[u]])
      atomicMin(&s_best[c[u]], k[u]);
  }
  __syncthreads();
  int hooked = 0;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int r = u * 1024 + t;
    if (r < m && c[u] == (uint32_t)r) {
      const unsigned long long b = s_best[r];
      if (b != ~0ull) {
        const uint32_t ca = comp[(b >> 16) & 0xffffu], cb = comp[b & 0xffffu];
        const uint32_t other = ca == (uint32_t)r ? cb : ca;
        if (s_best[other] != b || (uint32_t)r > other) {
          s_par[r] = (uint16_t)other;
          tree[r] = b;
          ++hooked;
        }
      }
    }
  }
  hooked = (int)wave_sum((unsigned int)hooked);
  if (lane_id() == 0 && hooked) atomicAdd(&s_hooked, hooked);
  __syncthreads();
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int v = u * 1024 + t;
    if (v < m) {
      uint32_t x = c[u];
      for (uint32_t y; (y = s_par[x]) != x;) x = y;
      comp[v] = (uint16_t)x;  // (the hooking's reads of comp are behind the barrier)
    }
  }
  if (t == 0) {
    const int total = done[1] + s_hooked;
    done[1] = total;
    if (total >= m - 1) done[0] = 1;
  }
}

// The same for larger n: component minima in memory (best, all ones before
// the first round and again after each hooking), then hooking, then ids.
__global__ void k_dense_best(int64_t n, const uint16_t* __restrict__ comp,
                             const unsigned long long* __restrict__ minv,
                             unsigned long long* __restrict__ best,
                             const int32_t* __restrict__ done) {
  if (done[0]) return;
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= n) return;
  const unsigned long long k = minv[v];
  unsigned long long* b = best + comp[v];
  if (k < __hip_atomic_load(b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMin(b, k);
}
__global__ void k_dense_hook(int64_t n, const uint16_t* __restrict__ comp,
                             const unsigned long long* __restrict__ best,
                             int32_t* __restrict__ parent, unsigned long long* __restrict__ tree,
                             int32_t* __restrict__ done) {
  if (done[0]) return;
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n || comp[r] != (uint32_t)r) return;
  const unsigned long long b = best[r];
  if (b == ~0ull) return;
  const uint32_t ca = comp[(b >> 16) & 0xffffu], cb = comp[b & 0xffffu];
  const uint32_t other = ca == (uint32_t)r ? cb : ca;
  if (best[other] == b && (uint32_t)r < other) return;  // mutual choice: the smaller root stays
  parent[r] = (int32_t)other;
  tree[r] = b;
  const unsigned long long hooked = __ballot(1);
  if (lane_id() == (int)__builtin_ctzll(hooked)) atomicAdd(&done[1], __popcll(hooked));
}
__global__ void k_dense_flatten(int64_t n, const int32_t* __restrict__ parent,
                                uint16_t* __restrict__ comp,
                                unsigned long long* __restrict__ best,
                                const int32_t* __restrict__ done) {
  if (done[0]) return;
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= n) return;
  int32_t x = comp[v];
  while (parent[x] != x) x = parent[x];
  comp[v] = (uint16_t)x;
  best[v] = ~0ull;
}
// After a round of the larger form: n - 1 edges end the rounds.
__global__ void k_dense_round_end(int64_t n, int32_t* __restrict__ done) {
  if (done[1] >= n - 1) done[0] = 1;
}

__global__ void k_dense_init(int64_t n, uint16_t* __restrict__ comp, int32_t* __restrict__ parent,
                             unsigned long long* __restrict__ best,
                             unsigned long long* __restrict__ minv,
                             unsigned long long* __restrict__ tree,
                             unsigned long long* __restrict__ sorted, int32_t* __restrict__ done) {
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v == 0) {
    done[0] = n < 2;
    done[1] = 0;
  }
  if (v >= n) return;
  comp[v] = (uint16_t)v;
  parent[v] = (int32_t)v;
  best[v] = minv[v] = tree[v] = sorted[v] = ~0ull;
}

__global__ void k_iota(int32_t* __restrict__ a, int64_t n) {
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v < n) a[v] = (int32_t)v;
}

// Lifetime rule of eac.py:366-391 on the float32 heights of the n - 1 sorted
// tree edges (one workgroup): st[0] = clusters, st[1] = merges to apply,
// st[2] = 1 where numpy raises ValueError (fewer than two heights, or no
// lifetime within 1e-8 of zero).
template <typename T>
__global__ __launch_bounds__(1024) void k_dense_lifetime(const unsigned long long* __restrict__ sk,
                                                         int64_t n, int32_t n_clusters,
                                                         int64_t* __restrict__ st) {
  __shared__ unsigned long long s_arg[1024 / kWave], s_above[1024 / kWave];
  __shared__ unsigned int s_zero[1024 / kWave];
  const int t = threadIdx.x, w = t / kWave;
  if (n_clusters > 0) {
    if (t == 0) {
      st[0] = n_clusters;
      st[1] = n - n_clusters > 0 ? n - n_clusters : 0;
      st[2] = 0;
    }
    return;
  }
  if (n < 3) {
    if (t == 0) { st[0] = 0; st[1] = 0; st[2] = 1; }
    return;
  }
  const int64_t nl = n - 2;  // lifetimes
  // per lane, then per wave, then over the waves: (lifetime word, n - index),
  // whose maximum is the first largest lifetime, and the smallest lifetime
  // close to zero (all ones: none)
  unsigned long long arg = 0;
  unsigned int zero = ~0u;
  for (int64_t i = t; i < nl; i += blockDim.x) {
    const float w0 = wvalue<T>((uint32_t)(sk[i] >> 32)), w1 = wvalue<T>((uint32_t)(sk[i + 1] >> 32));
    const float lt = w1 - w0;  // >= 0: heights ascend
    const uint32_t bits = __float_as_uint(lt);  // non-negative floats order as integers
    const unsigned long long k = ((unsigned long long)bits << 32) | (unsigned long long)(nl - i);
    arg = k > arg ? k : arg;
    if (fabs((double)lt) <= 1e-8) zero = bits < zero ? bits : zero;
  }
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) {
    const unsigned long long o = __shfl_xor(arg, off, kWave);
    arg = o > arg ? o : arg;
    zero = min(zero, (unsigned)__shfl_xor(zero, off, kWave));
  }
  if (lane_id() == 0) {
    s_arg[w] = arg;
    s_zero[w] = zero;
  }
  __syncthreads();
  for (int u = 0; u < 1024 / kWave; ++u) {
    arg = s_arg[u] > arg ? s_arg[u] : arg;
    zero = min(zero, s_zero[u]);
  }
  const int64_t m = nl - (int64_t)(arg & 0xffffffffull);
  const float th = __uint_as_float((uint32_t)(arg >> 32));
  const float wm = wvalue<T>((uint32_t)(sk[m] >> 32));
  unsigned long long above = 0;
  for (int64_t i = t; i < n - 1; i += blockDim.x) above += wvalue<T>((uint32_t)(sk[i] >> 32)) > wm;
  above = wave_sum(above);
  if (lane_id() == 0) s_above[w] = above;
  __syncthreads();
  if (t == 0) {
    above = 0;
    for (int u = 0; u < 1024 / kWave; ++u) above += s_above[u];
    if (zero == ~0u) {
      st[0] = 0; st[1] = 0; st[2] = 1;
      return;
    }
    int64_t nc = above == 0 ? 1 : (int64_t)above + 1;
    if (th < 2.0f * __uint_as_float(zero)) nc = 1;
    st[0] = nc;
    st[1] = n - nc;
    st[2] = 0;
  }
}

__device__ __forceinline__ int32_t uf_find(int32_t* parent, int32_t x) {
  for (;;) {
    const int32_t p = parent[x];
    if (p == x) return x;
    const int32_t g = parent[p];
    if (g != p) parent[x] = g;  // path halving (a benign race: g is an ancestor)
    x = p;
  }
}

// Union of the endpoints of the first st[1] sorted edges (ends decoded from
// the key, or from node pairs in idx when given); the larger root hooks
// under the smaller, so every root is its component's smallest vertex.
__global__ void k_uf_link(const unsigned long long* __restrict__ sk, const int32_t* __restrict__ ends,
                          const int64_t* __restrict__ st, int32_t* __restrict__ parent) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= st[1]) return;
  int32_t a, b;
  if (ends) {
    a = ends[2 * e];
    b = ends[2 * e + 1];
  } else {
    a = (int32_t)((sk[e] >> 16) & 0xffffu);
    b = (int32_t)(sk[e] & 0xffffu);
  }
  for (;;) {
    a = uf_find(parent, a);
    b = uf_find(parent, b);
    if (a == b) return;
    if (a > b) { const int32_t t = a; a = b; b = t; }
    if (atomicCAS(&parent[b], b, a) == b) return;
  }
}

__global__ void k_uf_roots(int64_t n, int32_t* __restrict__ parent, int32_t* __restrict__ flag) {
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= n) return;
  const int32_t r = uf_find(parent, (int32_t)v);
  flag[v] = r == (int32_t)v;
}

__global__ void k_uf_labels(int64_t n, int32_t* __restrict__ parent, const int32_t* __restrict__ rank,
                            int32_t* __restrict__ labels) {
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= n) return;
  labels[v] = rank[uf_find(parent, (int32_t)v)];
}

// The cut's labels for n <= kOneGroupN in one workgroup. Rounds: every edge
// between two roots hooks the larger under the smaller (the smallest of
// several), then every vertex goes to its root; an edge within a component is
// dropped. The edges and roots stay in registers (16 of each a thread: the
// limit), the forest in LDS. 31 us at 8,000 points, five launches 57.
constexpr int64_t kOneGroupN = 16384;
__global__ __launch_bounds__(1024) void k_uf_one(const unsigned long long* __restrict__ sk,
                                                 const int32_t* __restrict__ ends,
                                                 const int64_t* __restrict__ st, int64_t n,
                                                 int32_t* __restrict__ labels) {
  extern __shared__ __align__(16) int32_t s_p[];
  __shared__ int32_t s_tmp[1024 / kWave + 1];
  constexpr int U = kOneGroupN / 1024;
  const int t = threadIdx.x, m = (int)n;
  const int64_t merges = st[1] < n - 1 ? st[1] : n - 1;
  uint32_t e[U], root[U];  // two vertices a word; ~0: no edge
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int64_t v = u * 1024 + t;
    if (v < n) s_p[v] = (int32_t)v;
    e[u] = ~0u;
    if (v < merges)
      e[u] = ends ? ((uint32_t)ends[2 * v] << 16) | (uint32_t)ends[2 * v + 1] : (uint32_t)sk[v];
  }
  __syncthreads();
  for (;;) {
    bool any = false;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (u * 1024 < m && e[u] != ~0u) {
        const uint32_t a = (uint32_t)s_p[e[u] >> 16], b = (uint32_t)s_p[e[u] & 0xffffu];
        root[u] = (a > b ? a : b) << 16 | (a > b ? b : a);
        if (a == b) e[u] = ~0u;
        any |= a != b;
      }
    }
    if (!__syncthreads_or(any)) break;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (u * 1024 < m && e[u] != ~0u) {
        const int32_t low = (int32_t)(root[u] & 0xffffu);
        int32_t* at = &s_p[root[u] >> 16];
        if (low < *(volatile int32_t*)at) atomicMin(at, low);  // (atomics on one word serialise)
      }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int v = u * 1024 + t;
      if (v < m) {
        int32_t x = s_p[v];
        for (int32_t y; (y = s_p[x]) != x;) x = y;
        s_p[v] = x;  // (others may read either: both are ancestors)
      }
    }
    __syncthreads();
  }
  // roots (component minima) in vertex order get the ranks 0, 1, ...
  const int per = (m + 1023) / 1024, v0 = t * per, v1 = v0 + per < m ? v0 + per : m;
  int32_t cnt = 0;
  for (int v = v0; v < v1; ++v) cnt += s_p[v] == v;
  int32_t total;
  int32_t rank = block_excl_scan<int32_t>(cnt, s_tmp, &total);
  for (int v = v0; v < v1; ++v)
    if (s_p[v] == v) s_p[v] = ~rank++;
  __syncthreads();
  for (int v = t; v < m; v += 1024) {
    const int32_t r = s_p[v];
    labels[v] = ~(r < 0 ? r : s_p[r]);
  }
}

// Linkage matrix from the sorted tree edges: one thread, union-find with the
// cluster's node id and size at its root (in LDS when 12 n bytes fit).
template <typename T, bool LDS>
__global__ void k_dense_linkage(const unsigned long long* __restrict__ sk, int64_t n,
                                int32_t* __restrict__ g_par, int32_t* __restrict__ g_nid,
                                int32_t* __restrict__ g_size, float* __restrict__ Z) {
  extern __shared__ int32_t s_uf[];
  int32_t* par = LDS ? s_uf : g_par;
  int32_t* nid = LDS ? s_uf + n : g_nid;
  int32_t* size = LDS ? s_uf + 2 * n : g_size;
  for (int64_t v = threadIdx.x; v < n; v += blockDim.x) {
    par[v] = (int32_t)v;
    nid[v] = (int32_t)v;
    size[v] = 1;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  for (int64_t i = 0; i + 1 < n; ++i) {
    const unsigned long long k = sk[i];
    int32_t a = (int32_t)((k >> 16) & 0xffffu), b = (int32_t)(k & 0xffffu);
    while (par[a] != a) { par[a] = par[par[a]]; a = par[a]; }
    while (par[b] != b) { par[b] = par[par[b]]; b = par[b]; }
    const int32_t ia = nid[a], ib = nid[b];
    const int32_t sz = size[a] + size[b];
    Z[4 * i + 0] = (float)(ia < ib ? ia : ib);
    Z[4 * i + 1] = (float)(ia < ib ? ib : ia);
    Z[4 * i + 2] = wvalue<T>((uint32_t)(k >> 32));
    Z[4 * i + 3] = (float)sz;
    if (size[a] < size[b]) { const int32_t t = a; a = b; b = t; }
    par[b] = a;
    size[a] = sz;
    nid[a] = (int32_t)(n + i);
  }
}

// labels_from_Z on a given Z: the leaf reached by following left children
// from every internal node (pointer jumping, one workgroup), then the union
// of the first `merges` rows' two sides.
__global__ __launch_bounds__(1024) void k_z_leftleaf(const float* __restrict__ Z, int64_t n,
                                                     int32_t* __restrict__ rep,
                                                     int32_t* __restrict__ bad) {
  __shared__ int s_changed;
  for (int64_t i = threadIdx.x; i + 1 < n; i += blockDim.x) {
    const float l = Z[4 * i];
    const int64_t li = (int64_t)l;
    if (!(l >= 0.0f) || (float)li != l || li >= n + i) {  // not a node formed before row i
      atomicOr(bad, 1);
      rep[i] = 0;
    } else {
      rep[i] = (int32_t)li;
    }
  }
  __syncthreads();
  for (;;) {
    if (threadIdx.x == 0) s_changed = 0;
    __syncthreads();
    for (int64_t i = threadIdx.x; i + 1 < n; i += blockDim.x) {
      const int32_t r = rep[i];
      if (r >= n) {
        rep[i] = rep[r - n];
        s_changed = 1;
      }
    }
    __syncthreads();
    if (!s_changed) break;
    __syncthreads();
  }
}

__global__ void k_z_ends(const float* __restrict__ Z, int64_t n, const int64_t* __restrict__ st,
                         const int32_t* __restrict__ rep, int32_t* __restrict__ ends,
                         int32_t* __restrict__ bad) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= st[1]) return;
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const float x = Z[4 * i + s];
    const int64_t xi = (int64_t)x;
    int32_t leaf = 0;
    if (!(x >= 0.0f) || (float)xi != x || xi >= n + i) atomicOr(bad, 1);
    else leaf = xi < n ? (int32_t)xi : rep[xi - n];
    ends[2 * i + s] = leaf;
  }
}

// Non-zero associations per row (full.py:83-95 get_degree with
// full_get_assoc_degree :190-212 / full_condensed_assoc_degree :214-226: a
// condensed row counts only its columns j > i). A wavefront per row, 16 bytes
// a lane between the row's aligned ends; one atomic on the total per
// workgroup (same-address atomics serialise: one per row made this 107 us at
// 8,000 rows, now 12).
template <typename T>
__global__ __launch_bounds__(1024) void k_dense_degree(const T* __restrict__ mat, int64_t n,
                                                      int condensed, int32_t* __restrict__ degree,
                                                      unsigned long long* __restrict__ nnz) {
  constexpr int V = 16 / sizeof(T);
  __shared__ unsigned long long s_w[1024 / kWave];
  const int l = lane_id(), w = threadIdx.x / kWave;
  unsigned long long total = 0;
  for (int64_t i = (int64_t)blockIdx.x * (1024 / kWave) + w; i < n;
       i += (int64_t)gridDim.x * (1024 / kWave)) {
    const T* row = condensed ? (i + 1 < n ? mat + cidx(n, i, i + 1) : mat) : mat + i * n;
    const int64_t len = condensed ? n - 1 - i : n;
    int64_t head = (int64_t)((16 - (reinterpret_cast<uintptr_t>(row) & 15)) & 15) / sizeof(T);
    if (head > len) head = len;
    const int64_t body = (len - head) / V;
    unsigned int c = 0;
    for (int64_t j = l; j < head; j += kWave) c += row[j] != (T)0;
    const Pack16<T>* p = reinterpret_cast<const Pack16<T>*>(row + head);
    for (int64_t j = l; j < body; j += kWave) {
      const Pack16<T> x = p[j];
#pragma unroll
      for (int u = 0; u < V; ++u) c += x.v[u] != (T)0;
    }
    for (int64_t j = head + body * V + l; j < len; j += kWave) c += row[j] != (T)0;
    c = wave_sum(c);
    if (l == 0) degree[i] = (int32_t)c;
    total += c;
  }
  if (l == 0) s_w[w] = total;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int u = 1; u < 1024 / kWave; ++u) total += s_w[u];
    if (total) atomicAdd(nnz, total);
  }
}

int elem_bytes(int32_t dtype) {
  switch (dtype) {
    case EAC_W_U8: return 1;
    case EAC_W_U16: return 2;
    case EAC_W_I32: return 4;
    case EAC_W_F32: return 4;
    default: return 0;
  }
}

struct DenseBufs {
  void* sq;        // square copy (condensed input only)
  uint16_t* comp;
  int32_t* parent;
  unsigned long long* best;
  unsigned long long* minv;
  unsigned long long* tree;
  unsigned long long* sorted;
  int64_t* st;     // lifetime state (3); st[3]: two ints, tree complete / its edges
  int32_t* flag;
  int32_t* rank;
  int32_t* misc;
};

DenseBufs carve_dense(Arena& ar, int64_t n, int eb, bool condensed) {
  DenseBufs b;
  b.sq = condensed ? static_cast<void*>(ar.take<uint8_t>((size_t)n * sq_stride(n) * eb)) : nullptr;
  b.comp = ar.take<uint16_t>(n);
  b.parent = ar.take<int32_t>(n);
  b.best = ar.take<unsigned long long>(n);
  b.minv = ar.take<unsigned long long>(n);
  b.tree = ar.take<unsigned long long>(n);
  b.sorted = ar.take<unsigned long long>(n);
  b.st = ar.take<int64_t>(4);
  b.flag = ar.take<int32_t>(n + 1);
  b.rank = ar.take<int32_t>(n + 1);
  b.misc = ar.take<int32_t>(4);
  return b;
}

int dense_check(const void* d, int32_t dtype, int64_t n) {
  if (!d) return fail(EAC_ERR_ARG, "dense: null matrix");
  if (!elem_bytes(dtype)) return fail(EAC_ERR_ARG, "dense: dtype %d not supported", dtype);
  if (n < 1 || n > kDenseMaxN) return fail(EAC_ERR_UNSUPPORTED, "dense: n = %lld outside [1, %lld]",
                                           (long long)n, (long long)kDenseMaxN);
  return EAC_OK;
}

template <typename T>
int launch_rowmin(const void* sq, int64_t n, int64_t ld, const DenseBufs& B, hipStream_t s) {
  const size_t lds = (size_t)((n + 15) & ~int64_t(15)) * 2;
  (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k_dense_rowmin<T>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  k_dense_rowmin<T><<<grid_for(n, kRowB / kWave, 1024), kRowB, lds, s>>>(
      static_cast<const T*>(sq), n, ld, B.comp, B.minv, reinterpret_cast<int32_t*>(B.st + 3));
  EAC_LAUNCH_CHECK();
  return EAC_OK;
}

// Rounds that always complete the tree, and those enqueued before the first
// read-back: components at least halve in each, and equal weights (counts)
// keep them from falling much faster (8 rounds of at most 14 at 8,000 points),
// while a round with nothing left costs two launches that return at once.
int dense_rounds(int64_t n) { return bits_for((uint64_t)(n > 1 ? n - 1 : 1)) + 1; }
int dense_batch(int64_t n) { return (dense_rounds(n) * 3 + 3) / 4; }

// The square form of the matrix and the rounds' start.
int dense_begin(const void* dists, int32_t dtype, int64_t n, int32_t condensed, DenseBufs& B,
                const void** sq, hipStream_t s) {
  *sq = dists;
  if (condensed) {
    const int tiles = (int)((n + kDT - 1) / kDT);
    const dim3 g(tiles, tiles);
    switch (dtype) {
      case EAC_W_U8:
        k_square_from_condensed<uint8_t><<<g, 256, 0, s>>>(static_cast<const uint8_t*>(dists), n,
                                                          0xffu, static_cast<uint8_t*>(B.sq));
        break;
      case EAC_W_U16:
        k_square_from_condensed<uint16_t><<<g, 256, 0, s>>>(
            static_cast<const uint16_t*>(dists), n, 0xffffu, static_cast<uint16_t*>(B.sq));
        break;
      default:  // the largest word: 2^31 - 1, or a NaN's bits
        k_square_from_condensed<uint32_t><<<g, 256, 0, s>>>(
            static_cast<const uint32_t*>(dists), n, 0x7fffffffu, static_cast<uint32_t*>(B.sq));
        break;
    }
    EAC_LAUNCH_CHECK();
    *sq = B.sq;
  }
  k_dense_init<<<grid_for(n, 256), 256, 0, s>>>(n, B.comp, B.parent, B.best, B.minv, B.tree,
                                                 B.sorted, reinterpret_cast<int32_t*>(B.st + 3));
  EAC_LAUNCH_CHECK();
  return EAC_OK;
}

// Borůvka rounds [r0, r1) over the dense matrix, then the tree edges sorted
// into B.sorted (n - 1 keys, then ~0).
int dense_tree(const void* sq, int32_t dtype, int64_t n, int32_t condensed, int r0, int r1,
               DenseBufs& B, Arena& ar, hipStream_t s) {
  const int64_t ld = condensed ? sq_stride(n) : n;
  const int gv = grid_for(n, 256);
  int32_t* done = reinterpret_cast<int32_t*>(B.st + 3);
  for (int r = r0; r < r1 && n > 1; ++r) {
    switch (dtype) {
      case EAC_W_U8: EAC_TRY(launch_rowmin<uint8_t>(sq, n, ld, B, s)); break;
      case EAC_W_U16: EAC_TRY(launch_rowmin<uint16_t>(sq, n, ld, B, s)); break;
      case EAC_W_I32: EAC_TRY(launch_rowmin<int32_t>(sq, n, ld, B, s)); break;
      default: EAC_TRY(launch_rowmin<float>(sq, n, ld, B, s)); break;
    }
    if (n <= kMergeN) {
      const size_t lds = (size_t)n * 10 + 16;
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k_dense_merge),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      k_dense_merge<<<1, 1024, lds, s>>>(n, B.comp, B.minv, B.tree, done);
    } else {
      k_dense_best<<<gv, 256, 0, s>>>(n, B.comp, B.minv, B.best, done);
      k_dense_hook<<<gv, 256, 0, s>>>(n, B.comp, B.best, B.parent, B.tree, done);
      k_dense_flatten<<<gv, 256, 0, s>>>(n, B.parent, B.comp, B.best, done);
      k_dense_round_end<<<1, 1, 0, s>>>(n, done);
    }
    EAC_LAUNCH_CHECK();
  }
  const size_t mark = ar.used;
  // (weight words of narrow types leave the top bits zero; the absent key's
  // remaining bits still sort it last)
  EAC_TRY((radix_sort<uint64_t, NoValue>(reinterpret_cast<const uint64_t*>(B.tree),
                                          reinterpret_cast<uint64_t*>(B.sorted), nullptr, nullptr,
                                          n, 0, 32 + 8 * elem_bytes(dtype), ar, s)));
  ar.used = mark;
  return EAC_OK;
}

template <typename T>
void launch_lifetime(const unsigned long long* sk, int64_t n, int32_t nc, int64_t* st,
                     hipStream_t s) {
  k_dense_lifetime<T><<<1, 1024, 0, s>>>(sk, n, nc, st);
}

template <typename T>
int launch_linkage(const unsigned long long* sk, int64_t n, int32_t* par, int32_t* nid,
                   int32_t* size, float* Z, hipStream_t s) {
  const size_t lds = (size_t)12 * n;
  if (lds <= 150 * 1024) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k_dense_linkage<T, true>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    k_dense_linkage<T, true><<<1, 256, lds, s>>>(sk, n, par, nid, size, Z);
  } else {
    k_dense_linkage<T, false><<<1, 256, 0, s>>>(sk, n, par, nid, size, Z);
  }
  EAC_LAUNCH_CHECK();
  return EAC_OK;
}

int d2h_small(void* host, const void* dev, size_t bytes, hipStream_t s) {
  EAC_HIP_CHECK(hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, s));
  EAC_HIP_CHECK(hipStreamSynchronize(s));
  return EAC_OK;
}

// Labels of the first st[1] merges (edges from sk, or node pairs in ends).
int cut_labels(const unsigned long long* sk, const int32_t* ends, int64_t n, DenseBufs& B,
               int32_t* labels, Arena& ar, hipStream_t s) {
  if (n <= kOneGroupN) {
    const size_t lds = (size_t)n * 4;
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k_uf_one),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    k_uf_one<<<1, 1024, lds, s>>>(sk, ends, B.st, n, labels);
    EAC_LAUNCH_CHECK();
    return EAC_OK;
  }
  const int gv = grid_for(n, 256);
  k_iota<<<gv, 256, 0, s>>>(B.parent, n);
  k_uf_link<<<gv, 256, 0, s>>>(sk, ends, B.st, B.parent);
  k_uf_roots<<<gv, 256, 0, s>>>(n, B.parent, B.flag);
  EAC_LAUNCH_CHECK();
  const size_t mark = ar.used;
  EAC_TRY((scan_excl<int32_t, int32_t>(B.flag, B.rank, n, 0, nullptr, ar, s)));
  ar.used = mark;
  k_uf_labels<<<gv, 256, 0, s>>>(n, B.parent, B.rank, labels);
  EAC_LAUNCH_CHECK();
  return EAC_OK;
}

size_t dense_ws(int64_t n, int32_t dtype, bool condensed) {
  Arena ar(nullptr, 0, true);
  (void)carve_dense(ar, n, elem_bytes(dtype) ? elem_bytes(dtype) : 4, condensed);
  const size_t a = radix_sort_ws_bytes(n, 8, 0), b = scan_ws_bytes(n + 1, 4);
  return ar.used + (a > b ? a : b) + 3 * sizeof(int32_t) * (size_t)n + 4096;
}

}  // namespace
}  // namespace eac

using namespace eac;

namespace {
size_t coassoc_dense_ws(int64_t n, int32_t P) {
  const int64_t tiles = (n + kDT - 1) / kDT;
  const int64_t stages = ((int64_t)P + kStage - 1) / kStage;
  return 256 + 4 * (size_t)(stages * tiles) * (kPlanes * kDT + 1);
}

template <typename T, bool ADD>
void launch_counts(const int32_t* labels, int64_t n, int32_t P, int32_t condensed,
                   const uint32_t* planes, const int32_t* bits, void* out, unsigned int* mx,
                   hipStream_t s) {
  const int64_t tiles = (n + kDT - 1) / kDT;
  // (two dimensions: one takes fewer than 2^32 threads, n = 370,727)
  const dim3 g((unsigned)(8 * ((n + kCC - 1) / kCC)), (unsigned)((tiles + 7) / 8));
  auto f = planes ? k_dense_counts<T, ADD, true> : k_dense_counts<T, ADD, false>;
  f<<<g, 256, 0, s>>>(labels, n, P, condensed, planes, bits, tiles * kDT, static_cast<T*>(out), mx);
}

template <bool ADD>
int coassoc_dense(const int32_t* labels, int64_t n, int32_t P, int32_t condensed, int32_t dtype,
                  void* out, int64_t* h_max, void* ws, size_t ws_bytes, void* stream) {
  hipStream_t s = (hipStream_t)stream;
  if (!labels || !out) return fail(EAC_ERR_ARG, "coassoc dense: null array");
  if (n < 1 || P < 1) return fail(EAC_ERR_ARG, "coassoc dense: need n, P >= 1");
  if (n > (int64_t)1 << 20) return fail(EAC_ERR_UNSUPPORTED, "coassoc dense: n too large");
  if (!ws || ws_bytes < 256) return fail(EAC_ERR_WORKSPACE, "coassoc dense: workspace < 256 bytes");
  // [0]: the maximum; then, where the workspace has the room, the planes
  unsigned int* mx = h_max ? static_cast<unsigned int*>(ws) : nullptr;
  if (mx) EAC_TRY(fill<int32_t>(reinterpret_cast<int32_t*>(mx), 1, 0, s));
  const int64_t tiles = (n + kDT - 1) / kDT, npad = tiles * kDT;
  const int stages = (P + kStage - 1) / kStage;
  uint32_t* planes = nullptr;
  int32_t* bits = nullptr;
  if (ws_bytes >= coassoc_dense_ws(n, P) && stages <= 65535) {
    planes = static_cast<uint32_t*>(ws) + 64;
    bits = reinterpret_cast<int32_t*>(planes + (int64_t)stages * kPlanes * npad);
    k_label_planes<<<dim3((unsigned)tiles, stages), kDT, 0, s>>>(labels, n, P, npad, planes, bits);
    EAC_LAUNCH_CHECK();
  }
  switch (dtype) {
    case EAC_W_U8: launch_counts<uint8_t, ADD>(labels, n, P, condensed, planes, bits, out, mx, s); break;
    case EAC_W_U16: launch_counts<uint16_t, ADD>(labels, n, P, condensed, planes, bits, out, mx, s); break;
    case EAC_W_I32: launch_counts<int32_t, ADD>(labels, n, P, condensed, planes, bits, out, mx, s); break;
    case EAC_W_F32: launch_counts<float, ADD>(labels, n, P, condensed, planes, bits, out, mx, s); break;
    default: return fail(EAC_ERR_ARG, "coassoc dense: dtype %d not supported", dtype);
  }
  EAC_LAUNCH_CHECK();
  if (h_max) {
    unsigned int v = 0;
    EAC_TRY(d2h_small(&v, mx, sizeof(v), s));
    *h_max = v;
  }
  return EAC_OK;
}

int diassoc(void* mat, int64_t len, int32_t dtype, double val, const unsigned long long* top,
            hipStream_t s) {
  const int g = grid_for(len, 256 * 16, 4096);
  switch (dtype) {
    case EAC_W_U8: k_dense_diassoc<uint8_t><<<g, 256, 0, s>>>((uint8_t*)mat, len, val, top); break;
    case EAC_W_U16: k_dense_diassoc<uint16_t><<<g, 256, 0, s>>>((uint16_t*)mat, len, val, top); break;
    case EAC_W_I32: k_dense_diassoc<int32_t><<<g, 256, 0, s>>>((int32_t*)mat, len, val, top); break;
    case EAC_W_F32: k_dense_diassoc<float><<<g, 256, 0, s>>>((float*)mat, len, val, top); break;
    default: return fail(EAC_ERR_ARG, "dense diassoc: dtype %d not supported", dtype);
  }
  EAC_LAUNCH_CHECK();
  return EAC_OK;
}
}  // namespace

extern "C" size_t eac_coassoc_dense_workspace_bytes(int64_t n, int32_t P) {
  return n < 1 || P < 1 ? 256 : coassoc_dense_ws(n, P);
}

extern "C" int eac_coassoc_dense(const int32_t* labels, int64_t n, int32_t P, int32_t condensed,
                                 int32_t dtype, void* out, int64_t* h_max, void* ws,
                                 size_t ws_bytes, void* stream) {
  return coassoc_dense<false>(labels, n, P, condensed, dtype, out, h_max, ws, ws_bytes, stream);
}

extern "C" int eac_coassoc_dense_add(const int32_t* labels, int64_t n, int32_t P,
                                     int32_t condensed, int32_t dtype, void* inout, void* ws,
                                     size_t ws_bytes, void* stream) {
  return coassoc_dense<true>(labels, n, P, condensed, dtype, inout, nullptr, ws, ws_bytes, stream);
}

extern "C" int eac_dense_diassoc(void* mat, int64_t len, int32_t dtype, double val,
                                 void* stream) {
  if (len < 0 || (len > 0 && !mat)) return fail(EAC_ERR_ARG, "dense diassoc: bad array");
  if (len == 0) return EAC_OK;
  return diassoc(mat, len, dtype, val, nullptr, (hipStream_t)stream);
}

extern "C" int eac_dense_diassoc_max(void* mat, int64_t len, int32_t dtype, void* ws,
                                     size_t ws_bytes, void* stream) {
  hipStream_t s = (hipStream_t)stream;
  if (len < 1 || !mat) return fail(EAC_ERR_ARG, "dense diassoc: bad array");
  if (!ws || ws_bytes < 256) return fail(EAC_ERR_WORKSPACE, "dense diassoc: workspace < 256 bytes");
  uint64_t* w = static_cast<uint64_t*>(ws);
  EAC_TRY(fill<uint64_t>(w, 1, 0ull, s));
  unsigned long long* top = reinterpret_cast<unsigned long long*>(w);
  const int g = grid_for(len, 1024 * 16, 512);
  switch (dtype) {
    case EAC_W_U8: k_dense_max<uint8_t><<<g, 1024, 0, s>>>((const uint8_t*)mat, len, top); break;
    case EAC_W_U16: k_dense_max<uint16_t><<<g, 1024, 0, s>>>((const uint16_t*)mat, len, top); break;
    case EAC_W_I32: k_dense_max<int32_t><<<g, 1024, 0, s>>>((const int32_t*)mat, len, top); break;
    default: return fail(EAC_ERR_ARG, "dense diassoc: dtype %d not supported", dtype);
  }
  EAC_LAUNCH_CHECK();
  return diassoc(mat, len, dtype, 0.0, top, s);
}

extern "C" int eac_dense_degree(const void* mat, int32_t dtype, int64_t n, int32_t condensed,
                                int32_t* degree, int64_t* h_nnz, void* ws, size_t ws_bytes,
                                void* stream) {
  hipStream_t s = (hipStream_t)stream;
  if (!mat || !degree || n < 1) return fail(EAC_ERR_ARG, "dense degree: bad arguments");
  if (!ws || ws_bytes < 256) return fail(EAC_ERR_WORKSPACE, "dense degree: workspace < 256 bytes");
  uint64_t* nnz = static_cast<uint64_t*>(ws);
  EAC_TRY(fill<uint64_t>(nnz, 1, 0ull, s));
  unsigned long long* c = reinterpret_cast<unsigned long long*>(nnz);
  const int g = grid_for(n, 1024 / kWave, 512);
  switch (dtype) {
    case EAC_W_U8: k_dense_degree<uint8_t><<<g, 1024, 0, s>>>((const uint8_t*)mat, n, condensed, degree, c); break;
    case EAC_W_U16: k_dense_degree<uint16_t><<<g, 1024, 0, s>>>((const uint16_t*)mat, n, condensed, degree, c); break;
    case EAC_W_I32: k_dense_degree<int32_t><<<g, 1024, 0, s>>>((const int32_t*)mat, n, condensed, degree, c); break;
    case EAC_W_F32: k_dense_degree<float><<<g, 1024, 0, s>>>((const float*)mat, n, condensed, degree, c); break;
    default: return fail(EAC_ERR_ARG, "dense degree: dtype %d not supported", dtype);
  }
  EAC_LAUNCH_CHECK();
  if (h_nnz) {
    uint64_t v = 0;
    EAC_TRY(d2h_small(&v, nnz, sizeof(v), s));
    *h_nnz = (int64_t)v;
  }
  return EAC_OK;
}

extern "C" size_t eac_dense_sl_workspace_bytes(int64_t n, int32_t dtype, int32_t condensed) {
  if (n < 1) n = 1;
  return dense_ws(n, dtype, condensed != 0);
}

extern "C" int eac_full_sl_lifetime(const void* dists, int32_t dtype, int64_t n,
                                    int32_t condensed, int32_t n_clusters, float* Z,
                                    int32_t* labels, int64_t* h_out, void* ws, size_t ws_bytes,
                                    void* stream) {
  hipStream_t s = (hipStream_t)stream;
  EAC_TRY(dense_check(dists, dtype, n));
  if (!labels) return fail(EAC_ERR_ARG, "full_sl_lifetime: null labels");
  if (n_clusters < 0) return fail(EAC_ERR_ARG, "full_sl_lifetime: n_clusters < 0");
  const size_t need = dense_ws(n, dtype, condensed != 0);
  if (!ws || ws_bytes < need)
    return fail(EAC_ERR_WORKSPACE, "full_sl_lifetime: workspace %zu < %zu bytes", ws_bytes, need);
  Arena ar(ws, ws_bytes);
  DenseBufs B = carve_dense(ar, n, elem_bytes(dtype), condensed != 0);
  const void* sq = nullptr;
  EAC_TRY(dense_begin(dists, dtype, n, condensed, B, &sq, s));
  int64_t st[4] = {0, 0, 0, 0};
  const size_t mark = ar.used;
  // the usual number of rounds, the sort and the rule go out together; the
  // read-back says whether the tree was complete
  for (int r0 = 0, rounds = dense_batch(n);;
       r0 = rounds, rounds = dense_rounds(n)) {
    ar.used = mark;
    EAC_TRY(dense_tree(sq, dtype, n, condensed, r0, rounds, B, ar, s));
    switch (dtype) {
      case EAC_W_U8: launch_lifetime<uint8_t>(B.sorted, n, n_clusters, B.st, s); break;
      case EAC_W_U16: launch_lifetime<uint16_t>(B.sorted, n, n_clusters, B.st, s); break;
      case EAC_W_I32: launch_lifetime<int32_t>(B.sorted, n, n_clusters, B.st, s); break;
      default: launch_lifetime<float>(B.sorted, n, n_clusters, B.st, s); break;
    }
    EAC_LAUNCH_CHECK();
    EAC_TRY(d2h_small(st, B.st, sizeof(st), s));
    if ((int32_t)st[3] || rounds >= dense_rounds(n)) break;
  }
  if (Z && n > 1) {
    int32_t* par = ar.take<int32_t>(n);
    int32_t* nid = ar.take<int32_t>(n);
    int32_t* size = ar.take<int32_t>(n);
    switch (dtype) {
      case EAC_W_U8: EAC_TRY(launch_linkage<uint8_t>(B.sorted, n, par, nid, size, Z, s)); break;
      case EAC_W_U16: EAC_TRY(launch_linkage<uint16_t>(B.sorted, n, par, nid, size, Z, s)); break;
      case EAC_W_I32: EAC_TRY(launch_linkage<int32_t>(B.sorted, n, par, nid, size, Z, s)); break;
      default: EAC_TRY(launch_linkage<float>(B.sorted, n, par, nid, size, Z, s)); break;
    }
  }
  if (st[2]) return fail(EAC_ERR_VALUE, "full_sl_lifetime: the lifetime rule raises (no lifetime "
                                       "within 1e-8 of zero, or fewer than two heights)");
  const int64_t nc = st[0];
  if (h_out) {
    h_out[0] = nc;
    h_out[1] = nc > 1 ? 0 : 1;
  }
  if (nc > 1) EAC_TRY(cut_labels(B.sorted, nullptr, n, B, labels, ar, s));
  return EAC_OK;
}

extern "C" int eac_slink(const void* dists, int32_t dtype, int64_t n, int32_t condensed,
                         float* Z, void* ws, size_t ws_bytes, void* stream) {
  hipStream_t s = (hipStream_t)stream;
  EAC_TRY(dense_check(dists, dtype, n));
  if (!Z) return fail(EAC_ERR_ARG, "slink: null Z");
  const size_t need = dense_ws(n, dtype, condensed != 0);
  if (!ws || ws_bytes < need)
    return fail(EAC_ERR_WORKSPACE, "slink: workspace %zu < %zu bytes", ws_bytes, need);
  if (n < 2) return EAC_OK;
  Arena ar(ws, ws_bytes);
  DenseBufs B = carve_dense(ar, n, elem_bytes(dtype), condensed != 0);
  const void* sq = nullptr;
  EAC_TRY(dense_begin(dists, dtype, n, condensed, B, &sq, s));
  EAC_TRY(dense_tree(sq, dtype, n, condensed, 0, dense_rounds(n), B, ar, s));
  int32_t* par = ar.take<int32_t>(n);
  int32_t* nid = ar.take<int32_t>(n);
  int32_t* size = ar.take<int32_t>(n);
  switch (dtype) {
    case EAC_W_U8: EAC_TRY(launch_linkage<uint8_t>(B.sorted, n, par, nid, size, Z, s)); break;
    case EAC_W_U16: EAC_TRY(launch_linkage<uint16_t>(B.sorted, n, par, nid, size, Z, s)); break;
    case EAC_W_I32: EAC_TRY(launch_linkage<int32_t>(B.sorted, n, par, nid, size, Z, s)); break;
    default: EAC_TRY(launch_linkage<float>(B.sorted, n, par, nid, size, Z, s)); break;
  }
  return EAC_OK;
}

extern "C" size_t eac_labels_from_Z_workspace_bytes(int64_t n) {
  if (n < 1) n = 1;
  Arena ar(nullptr, 0, true);
  (void)carve_dense(ar, n, 4, false);
  (void)ar.take<int32_t>(n);      // rep
  (void)ar.take<int32_t>(2 * n);  // ends
  return ar.used + scan_ws_bytes(n + 1, 4) + 4096;
}

extern "C" int eac_labels_from_Z(const float* Z, int64_t n, int32_t n_clusters, int32_t* labels,
                                 void* ws, size_t ws_bytes, void* stream) {
  hipStream_t s = (hipStream_t)stream;
  if (n < 1 || (n > 1 && !Z) || !labels) return fail(EAC_ERR_ARG, "labels_from_Z: bad arguments");
  if (n_clusters < 1 || n_clusters > n)
    return fail(EAC_ERR_ARG, "labels_from_Z: n_clusters %d outside [1, n]", n_clusters);
  const size_t need = eac_labels_from_Z_workspace_bytes(n);
  if (!ws || ws_bytes < need)
    return fail(EAC_ERR_WORKSPACE, "labels_from_Z: workspace %zu < %zu bytes", ws_bytes, need);
  Arena ar(ws, ws_bytes);
  DenseBufs B = carve_dense(ar, n, 4, false);
  int32_t* rep = ar.take<int32_t>(n);
  int32_t* ends = ar.take<int32_t>(2 * n);
  EAC_TRY(fill<int32_t>(B.misc, 1, 0, s));
  int64_t st[2] = {n_clusters, n - n_clusters};
  EAC_HIP_CHECK(hipMemcpyAsync(B.st, st, sizeof(st), hipMemcpyHostToDevice, s));
  if (n > 1) {
    k_z_leftleaf<<<1, 1024, 0, s>>>(Z, n, rep, B.misc);
    k_z_ends<<<grid_for(n, 256), 256, 0, s>>>(Z, n, B.st, rep, ends, B.misc);
    EAC_LAUNCH_CHECK();
  }
  EAC_TRY(cut_labels(nullptr, ends, n, B, labels, ar, s));
  int32_t bad = 0;
  EAC_TRY(d2h_small(&bad, B.misc, sizeof(bad), s));
  if (bad) return fail(EAC_ERR_ARG, "labels_from_Z: Z holds a node id that is not a leaf or an "
                                    "earlier row");
  return EAC_OK;
}
