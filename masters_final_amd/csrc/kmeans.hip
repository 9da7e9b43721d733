// K-Means labeling and centroid update for gfx950.
//
// Reference: MyML/MyML/cluster/KMeans.py:117-189 (K_Means.fit),
// KMeans.py:453-490 (py_label/numba_label: direct squared differences, strict
// < so the lowest k wins exact ties), KMeans.py:586-629 (the CUDA labeling
// kernel) and KMeans.py:709-754 (centroid recomputation: float32 sums in
// point order, division by the count in double, empty clusters reseeded with
// the points of smallest distance).
//
// Labeling modes (all batched over P partitions that share the data, each
// with its own centroid range [k_off[p], k_off[p+1]) of one centroid array):
//  * F32: plain FP32 direct difference, one thread per point, centroid tiles
//    staged in LDS (the "plain per-call FP32" path).
//  * F64: FP64 direct difference in ascending dimension order with strict <,
//    i.e. the oracle's arithmetic; exact by construction.
//  * BF16X3: the distance ||x||^2 - 2 x.c + ||c||^2 with the contraction on
//    MFMA. Each operand is split into two 16-bit halves (x = xh + xl + ex);
//    16x16x32 MFMAs of xh.ch + xh.cl + xl.ch accumulate in fp32. The halves
//    are f16 after a power-of-two scaling: 22 bits of every coordinate
//    against the 16 of two bf16 halves, at the same rate (2^-23 rather than
//    2^-17 left over: 0.16% of a 500,000-point ensemble re-scored instead of
//    0.33%, 0.19% of 4 M x 64-d points). The epilogue keeps the two best
//    groups of four centroids per point. A rigorous per-point bound E on
//    |approx - FP64 oracle| (split residuals, fp32 accumulation with a
//    truncation-safe 2^-23 unit, oracle rounding) certifies the group when the
//    margin exceeds 2 E, and its four candidates are compared in FP64; every
//    other point is re-scored in FP64 against all centroids of its partition.
//    Labels and distances therefore equal the FP64 oracle's.
//    Large single labelings of more than 32 dimensions run as a cascade: one
//    product first (a third of the MFMAs, a wider bound), all three only for
//    the rows it cannot certify (1% on the 64-d workload).
//    4,194,304 x 64-d points, 2048 centroids: 4.00 -> 1.9 ms a pass (the
//    single product 1.54, of which the group's FP64 comparison is a third;
//    bound by vector issue), 300,007 x 37-d, 501 centroids: 239 -> 155 us.
#include <algorithm>
#include <cfloat>
#include <climits>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "group.hpp"
#include "prims.hpp"
#include "sort.hpp"

namespace eac {
namespace {

// ------------------------------------------------- split-f16 MFMA labeling
// Layout of the split rows (points in registers, centroids in memory and
// LDS). Every operand is scaled by a power of two (the centroids of a partition
// by their largest coordinate, the points of a workgroup by that of most of
// its rows, see kApart) into f16's normal range and split into two f16 halves,
// v = h + l + e; halves below f16's smallest normal value are zero, so no
// product meets a subnormal. Three products h.h + h.l + l.h make the
// contraction. For d where it saves MFMA steps the three pieces are laid end to
// end over one K axis of 3 d entries (points: h, l, h; centroids: h, h, l), 32
// entries a step: ceil(3 d / 32) steps; otherwise (3 d close to a multiple of
// 96) h and l are kept as rows of KB = ceil(d / 32) fragments and used twice:
// 3 KB steps from 2 KB fragments.
struct LabelLayout {
  int KS;      // MFMA steps (32 entries each)
  bool split;  // two rows of KS / 3 fragments
  int NF;      // fragments per row (32 halves each)
};
inline LabelLayout label_layout(int d, bool want_split = false) {
  LabelLayout L;
  const int packed = (3 * d + 31) / 32, KB = (d + 31) / 32;
  L.split = want_split || packed >= 3 * KB || packed == 3 || packed > 8 || packed == 6;
  L.KS = L.split ? 3 * KB : packed;
  L.NF = L.split ? 2 * KB : packed;
  return L;
}

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
// LDS rows are written as 16-bit words and read as fragments
typedef f16x8 f16x8_lds __attribute__((may_alias));
typedef f32x4 f32x4_u __attribute__((aligned(4)));  // rows need no more than their own alignment
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 u32x4_lds __attribute__((may_alias));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef f16x4 f16x4_lds __attribute__((may_alias));

// Power-of-two scale that takes a largest magnitude m into [2^14, 2^15)
// (1 for 0, infinity and NaN; exponents are kept within 2^+-60, so products of
// two scales and their inverses stay finite and normal).
__device__ __forceinline__ float pow2_scale(float m) {
  const int e = (int)((__float_as_uint(m) >> 23) & 255u);
  if (e == 255 || m == 0.0f) return 1.0f;
  int s = 127 + 14 - (e - 127);  // biased exponent of the scale
  s = s < 127 - 60 ? 127 - 60 : s > 127 + 60 ? 127 + 60 : s;
  return __uint_as_float((uint32_t)s << 23);
}
__device__ __forceinline__ _Float16 f16_half(float v) {
  return fabsf(v) < 6.103515625e-05f ? (_Float16)0.0f : (_Float16)v;
}
__device__ __forceinline__ uint16_t f16_bits(_Float16 h) { return __builtin_bit_cast(uint16_t, h); }

// Per-partition statistics of the centroids as float bits (non-negative
// floats order like their bit patterns): maxima of ||c||, ||ch||, ||cl||,
// ||ec|| (unscaled), and of |c_j| (the scale).
constexpr int kStat = 5;

// Largest |c_j| of each partition (grid.y over partitions).
__global__ __launch_bounds__(256) void k_cent_max(const float* __restrict__ C, int d,
                                                  const int64_t* __restrict__ k_off, int P,
                                                  unsigned int* __restrict__ pstat) {
  for (int p = blockIdx.y; p < P; p += gridDim.y) {
    const int64_t a = k_off[p] * d, b = k_off[p + 1] * d;
    unsigned int m = 0;
    for (int64_t i = a + (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < b;
         i += (int64_t)gridDim.x * blockDim.x)
      m = max(m, __float_as_uint(C[i]) & 0x7fffffffu);
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) m = max(m, (unsigned)__shfl_xor(m, off, kWave));
    if (lane_id() == 0 && m) atomicMax(&pstat[p * kStat + 4], m);
  }
}

// Splits every centroid into its layout row Cf [ktot][NF * 32] (zero padded),
// writes ||c||^2 and (Ct, nullable) the transposed copy, and reduces the norm
// maxima. Sixteen lanes per centroid; grid.y over partitions.
__global__ __launch_bounds__(256) void k_cent_prep(const float* __restrict__ C, int64_t ktot, int d,
                                                   LabelLayout L,
                                                   const int64_t* __restrict__ k_off, int P,
                                                   uint16_t* __restrict__ Cf,
                                                   float* __restrict__ Ct,
                                                   float* __restrict__ ncf,
                                                   unsigned int* __restrict__ pstat) {
  __shared__ unsigned int s_v[256 / kWave][4];
  const int sub = threadIdx.x & 15;
  const int RH = L.NF * 32;
  for (int p = blockIdx.y; p < P; p += gridDim.y) {
    const int64_t kb = k_off[p], ke = k_off[p + 1];
    const float sc = pow2_scale(__uint_as_float(pstat[p * kStat + 4])), inv = 1.0f / sc;
    unsigned int v[4] = {0u, 0u, 0u, 0u};
    for (int64_t c = kb + (int64_t)blockIdx.x * 16 + threadIdx.x / 16; c < ke;
         c += (int64_t)gridDim.x * 16) {
      double n2 = 0, h2 = 0, l2 = 0, e2 = 0;
      uint16_t* row = Cf + c * RH;
      for (int j = sub; j < d; j += 16) {
        const float x = C[c * d + j], y = x * sc;
        const _Float16 h = f16_half(y);
        const float r = y - (float)h;  // exact
        const _Float16 l = f16_half(r);
        const float e = r - (float)l;  // exact
        if (L.split) {
          row[j] = f16_bits(h);
          row[RH / 2 + j] = f16_bits(l);
        } else {
          row[j] = f16_bits(h);
          row[d + j] = f16_bits(h);
          row[2 * d + j] = f16_bits(l);
        }
        if (Ct) Ct[(int64_t)j * ktot + c] = x;  // transposed copy for the re-scoring
        const double hd = (double)(float)h * inv, ld = (double)(float)l * inv;
        const double ed = (double)e * inv;
        n2 += (double)x * x;
        h2 += hd * hd;
        l2 += ld * ld;
        e2 += ed * ed;
      }
      if (L.split) {
        for (int j = d + sub; j < RH / 2; j += 16) row[j] = row[RH / 2 + j] = 0;
      } else {
        for (int j = 3 * d + sub; j < RH; j += 16) row[j] = 0;
      }
#pragma unroll
      for (int off = 1; off < 16; off <<= 1) {
        n2 += __shfl_xor(n2, off, kWave);
        h2 += __shfl_xor(h2, off, kWave);
        l2 += __shfl_xor(l2, off, kWave);
        e2 += __shfl_xor(e2, off, kWave);
      }
      if (sub == 0) ncf[c] = (float)n2;
      // norms rounded up so the bound stays rigorous (a NaN or infinity
      // keeps the largest bits: its partition's points are all re-scored)
      v[0] = max(v[0], __float_as_uint((float)sqrt(n2) * (1.f + 1e-6f)) & 0x7fffffffu);
      v[1] = max(v[1], __float_as_uint((float)sqrt(h2) * (1.f + 1e-6f)) & 0x7fffffffu);
      v[2] = max(v[2], __float_as_uint((float)sqrt(l2) * (1.f + 1e-6f)) & 0x7fffffffu);
      v[3] = max(v[3], __float_as_uint((float)sqrt(e2) * (1.f + 1e-6f)) & 0x7fffffffu);
    }
    // one atomic per statistic and block (same-address atomics serialise)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
#pragma unroll
      for (int off = 16; off < kWave; off <<= 1)
        v[q] = max(v[q], (unsigned)__shfl_xor(v[q], off, kWave));
    }
    __syncthreads();
    if (lane_id() == 0)
#pragma unroll
      for (int q = 0; q < 4; ++q) s_v[threadIdx.x / kWave][q] = v[q];
    __syncthreads();
    if (threadIdx.x < 4) {
      unsigned int m = 0;
      for (int u = 0; u < 256 / kWave; ++u) m = max(m, s_v[u][threadIdx.x]);
      if (m) atomicMax(&pstat[p * kStat + threadIdx.x], m);
    }
  }
}

constexpr int kLB = 256;       // threads per labeling block (4 waves)
constexpr int kBN = 64;        // centroids per LDS tile
constexpr int kFlagSlots = 64; // flag list regions (one counter each)
constexpr int kGrp = 4;        // consecutive centroids of a candidate group

// Rigorous bound on |approx - oracle| for one point and one partition, for
// D' = ||c||^2 - 2 x.c (||x||^2 is common to a point's centroids) accumulated
// from ||c||^2 on: the three products of the split, or (TERMS = 1) only xh.ch,
// where x.c - xh.ch = (x - xh).c + xh.(c - ch). rs: the point's ||x||, ||xh||,
// ||xl|| and ||ex|| (TERMS = 1: ||x - xh||), st: the partition's maxima.
template <int TERMS>
__device__ __forceinline__ float point_bound(const float* rs, const float* st, int d) {
  const float u = 5.9604645e-08f;            // 2^-24
  const float ut = 1.1920929e-07f;           // 2^-23: fp32 accumulation, any rounding
  const float xn = rs[0], xhn = rs[1], xln = rs[2], exn = rs[3];
  const float Cn = st[0], Chn = st[1], Cln = st[2], Cen = st[3];
  // nonzero products per dot and the starting value (the padding is zero in
  // both operands; adding an exact zero neither rounds nor truncates)
  const float nterms = (float)(TERMS * d + 1);
  const float gam = nterms * ut / (1.f - nterms * ut);
  const float cross =
      TERMS == 1
          ? gam * xhn * Chn + exn * Cn + xhn * (Cln + Cen)
          : gam * (xhn * (Chn + Cln) + xln * Chn) + xhn * Cen + xln * (Cln + Cen) + exn * Cn;
  const float epi = (gam + 6.f * u) * Cn * Cn + 6.f * u * xn * xn;
  const float orc = 4.f * d * 1.1102230e-16f * (xn + Cn) * (xn + Cn);
  return (2.f * cross + epi + orc) * 1.0001f + 1e-30f;
}

// The nearest of a group's kGrp consecutive centroids for 16 points of a
// wave, in the oracle's FP64 arithmetic (ascending dimensions, strict <, lowest
// index on ties). Four lanes per point, one per candidate, each adding its own
// chain in order; row and g are the lane's point and its group's first
// centroid. The rows go through LDS, 16 dimensions at a time: a point's lanes
// load its row and its candidates' rows 64 bytes a row, the next stage's
// loads in flight during the current sums, and every lane reads back its own
// row; straight from memory the lanes would take 16 bytes of 64 different
// lines per load. sf: kRsLds floats of the wave; d >= 4. V4: d is a multiple
// of four, so every piece lies on 16 bytes of LDS.
constexpr int kRsD = 16;          // dimensions per stage
constexpr int kRsS = kRsD + 4;    // LDS row stride: 16-byte reads of neighbouring rows on other banks
constexpr int kRsLds = (kWave + kWave / kGrp) * kRsS + 4;
template <bool V4>
__device__ __forceinline__ void resolve16(const float* __restrict__ X, int d,
                                          const float* __restrict__ C, int64_t kb, int64_t ke,
                                          int64_t row, int32_t g, float* __restrict__ sf,
                                          double& best, int32_t& bk) {
#pragma clang fp contract(off)  // the oracle's separately rounded products and sums
  using Piece = std::conditional_t<V4, f32x4, f32x4_u>;  // 16-byte LDS stores with V4
  const int l = lane_id(), pt = l / kGrp, q = l % kGrp;
  const int32_t k = (int32_t)(ke - kb);
  // A point's four lanes load its rows together: lane q 16 bytes at 16 q of
  // each candidate's row and of the point's, the last piece of a row moved
  // back to end with it (its overlap with the piece before is the same
  // values; it may start up to three floats before the stage, in the row
  // before's padding). Byte offsets inside the partition's centroids
  // (direct_f64 keeps them in range): half the registers of addresses.
  float* sc = sf + 4;
  float* sx = sc + kWave * kRsS;
  const char* cb = reinterpret_cast<const char*>(C + kb * d);
  const uint32_t d4 = (uint32_t)d * 4;
  uint32_t cr[kGrp];
#pragma unroll
  for (int u = 0; u < kGrp; ++u) cr[u] = __umul24((uint32_t)min(g + u, k - 1), d4);
  const float* xp = X + row * d;
  f32x4 cv[kGrp], xv;
  int at = 0;  // where the loaded pieces belong, relative to the stage
  auto load = [&](int j0) {
    const int j = min(j0 + 4 * q, d - 4);
    at = j - j0;
#pragma unroll
    for (int u = 0; u < kGrp; ++u)
      cv[u] = *reinterpret_cast<const f32x4_u*>(cb + (uint32_t)(cr[u] + 4 * j));
    xv = *reinterpret_cast<const f32x4_u*>(xp + j);
  };
  load(0);
  double acc = 0.0;
  for (int j0 = 0; j0 < d; j0 += kRsD) {
    const int dd = d - j0 < kRsD ? d - j0 : kRsD;
    __builtin_amdgcn_wave_barrier();  // one wavefront: its LDS operations keep their order
#pragma unroll
    for (int u = 0; u < kGrp; ++u)
      *reinterpret_cast<Piece*>(sc + (pt * kGrp + u) * kRsS + at) = cv[u];
    *reinterpret_cast<Piece*>(sx + pt * kRsS + at) = xv;
    __builtin_amdgcn_wave_barrier();
    if (j0 + kRsD < d) load(j0 + kRsD);
    const float* ca = sc + l * kRsS;
    const float* xa = sx + pt * kRsS;
    auto add = [&](float xe, float ce) {
      const double e = (double)xe - (double)ce;
      acc = acc + e * e;
    };
    if (dd == kRsD) {
#pragma unroll 2
      for (int j = 0; j < kRsD; j += 4) {
        const f32x4 xe = *reinterpret_cast<const f32x4*>(xa + j);
        const f32x4 ce = *reinterpret_cast<const f32x4*>(ca + j);
#pragma unroll
        for (int u = 0; u < 4; ++u) add(xe[u], ce[u]);
      }
    } else {
#pragma unroll 1
      for (int j = 0; j < dd; ++j) add(xa[j], ca[j]);
    }
  }
  // lanes hold ascending candidates: strictly smaller wins, else the lower
  best = acc;
  bk = g + q < k ? g + q : INT_MAX;
#pragma unroll
  for (int off = 1; off < kGrp; off <<= 1) {
    const double ob = __shfl_xor(best, off, kWave);
    const int32_t ok = __shfl_xor(bk, off, kWave);
    if (ok != INT_MAX && (bk == INT_MAX || ob < best || (ob == best && ok < bk))) {
      best = ob;
      bk = ok;
    }
  }
}

// One wave labels MB blocks of 16 points against every centroid of the
// block's partitions. The centroids are the rows of the MFMA result and the
// points its columns, so a lane holds four consecutive centroids of one point
// per 16 x 16 tile: their largest value (two operations) is all that enters
// the running top two, with the group's number for an index, and the MFMAs
// start from -||c||^2 / 2 (one value per row: a broadcast read of four), so the
// accumulators are compared as they come. Per element that is 1.5 vector
// operations (half a maximum, and a quarter of compare, med3 and two
// selects), against 5 when every element adds its ||c||^2 and carries its own
// index, and three registers of running state per point block instead of
// twelve. The margin is then between groups: when the second group's maximum
// is more than 2 E below the first's, the FP64 oracle's nearest centroid is
// one of the first group's four, and resolve16 picks it in FP64; every other
// point is flagged for the re-scoring. labels receives 4 x the group (FUSE:
// the label).
// Centroid tiles are double buffered in LDS and shared by the block's four
// waves; each fragment read feeds MB MFMAs.
// TERMS = 1: only xh.ch (from the h rows of a split layout), a third of the
// MFMAs with point_bound<1>, for the first pass of a cascade. LIST: the points
// are the rows of a flag list. FUSE (one partition): the group is resolved in
// the kernel and labels and dists are final.
//
// The points' scale: one for the workgroup, so that a tile's accumulators start
// from one value per centroid, whatever the point. Where the rows' largest
// coordinates lie within 2^kApart of each other (ordinary data) it is the
// largest row's. f16's smallest normal value cuts low halves off at 2^-14; the
// largest coordinate of the smallest such row is 2^2 or more, so 2^-16 of it
// stay, what two bf16 halves would leave. Where some lie further apart (a fill
// value, a heavy tail) the scale is the one that leaves the fewest rows to the
// re-scoring, by scale_cost: rows below it have wider bounds, rows above it
// overflow to infinite halves, so that their norms and bounds are infinite or
// NaN. An outlier then costs itself and not the rows beside it: with one row in
// 128 2^40 times the others, 300,007 x 37-d and 501 centroids take 196 us (168
// without; 1633 when the largest row's scale served all), 1,000,000 x 64-d and
// 2048 centroids 1.7 ms (0.72; 27.7).
constexpr int kApart = 12;
// The cost of a scale with exponent e for the rows' own exponents (hist: rows
// by exponent, upto: rows with this exponent or a smaller one): the share of
// 256 rows like it that the bound cannot certify, 2^(k - 13) of them for a row
// whose own scale is 2^k times this one (300,007 x 37-d: 0.2% at k = 0, 1% at
// 14). A row that overflows counts twice: it is far from everything, and the
// re-scoring's screen seldom spares such a row a centroid.
template <typename U32>
__device__ __forceinline__ uint32_t scale_cost(int e, const U32* hist, const U32* upto) {
  uint32_t cost = e > 1 ? 512u * upto[e - 2] : 0u;
  for (int k = kApart + 1; k <= kApart + 8; ++k)
    if (e + k < 256) cost += hist[e + k] << (k - 13);
  return cost + 256u * (upto[255] - upto[min(e + kApart + 8, 255)]);
}
constexpr uint64_t kFlagRow = (1ull << 40) - 1;
template <int KS, bool SPLIT, int MB, int WPE, int TERMS = 3, bool FUSE = false,
          bool LIST = false>
__global__ __launch_bounds__(kLB) __attribute__((amdgpu_waves_per_eu(WPE)))
void k_label_f16x3(
    const float* __restrict__ X, int64_t row0, int64_t n, int d, const float* __restrict__ C,
    const uint16_t* __restrict__ Cf, const float* __restrict__ ncf,
    const int64_t* __restrict__ k_off, int P, const unsigned int* __restrict__ pstat,
    const uint64_t* __restrict__ list, int32_t* __restrict__ labels, float* __restrict__ dists,
    uint64_t* __restrict__ flags, unsigned long long* __restrict__ nflag, int64_t region) {
  static_assert(TERMS == 3 || SPLIT, "one product needs separate h rows");
  constexpr int KB = KS / TERMS;                              // split: fragments of h
  constexpr int NF = TERMS == 1 ? KS : SPLIT ? 2 * KB : KS;   // fragments per row
  constexpr int RH = NF * 32;     // halves per centroid row
  constexpr int LROW = RH + 8;    // padded LDS row
  // two centroid tiles; with FUSE the resolving's rows afterwards
  constexpr int kTiles = 2 * kBN * LROW * 2, kRs = FUSE ? (kLB / kWave) * kRsLds * 4 : 0;
  __shared__ __align__(16) unsigned char s_raw[kTiles > kRs ? kTiles : kRs];
  uint16_t* s_c = reinterpret_cast<uint16_t*>(s_raw);
  __shared__ __align__(16) float s_nc[2][kBN];
  __shared__ float s_st[4 * MB * 16][4];  // row statistics of point_bound
  constexpr int kRows = (kLB / kWave) * MB * 16;  // rows of a workgroup
  __shared__ uint32_t s_rng[kLB / kWave], s_key[2][kLB / kWave];
  // the exponents of the scales the rows would have alone, how many have each
  // and how many up to each (before the tiles need the room)
  static_assert((kRows + 512) * 4 <= kTiles && kLB == 256, "an exponent a thread");
  typedef uint32_t __attribute__((may_alias)) u32_lds;
  u32_lds* s_ex = reinterpret_cast<u32_lds*>(s_raw);
  u32_lds *s_hist = s_ex + kRows, *s_upto = s_hist + 256;
  const int t = threadIdx.x;
  const int w = t / kWave;
  const int l = lane_id();
  const int lr = l & 15;  // point inside a 16-block / centroid row (A layout)
  const int lq = l >> 4;  // k-group (operands) / centroid quad (result)
  const int64_t p0 = row0 + ((int64_t)blockIdx.x * (kLB / kWave) + w) * (MB * 16);
  auto row_id = [&](int64_t r) { return LIST ? (int64_t)(list[r] & kFlagRow) : r; };
  // partitions of this block (grid.y splits them)
  const int pa = (int)((int64_t)P * blockIdx.y / gridDim.y);
  const int pz = (int)((int64_t)P * (blockIdx.y + 1) / gridDim.y);

  // Point fragments and row statistics, one block of 16 rows at a time: four
  // lanes per row split its scaled coordinates into the wave's sixteen rows of the second centroid buffer (free until the first tile is done), from which
  // the fragments are read back. (Split straight into the fragments, the
  // loads and conditions of all blocks together spill.)
  f16x8 pf[MB][NF];
  // largest exponent and largest 255 - exponent of the rows' scales
  typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
  u16x2 rng = {0, 0};
  // coordinates are loaded four at a time (the last piece of a row moved back
  // to end with it), halves stored eight bytes at a time where d allows
  const bool x4 = (d & 3) == 0;
#pragma unroll 1
  for (int pb = 0; pb < MB; ++pb) {
    const int64_t row = p0 + pb * 16 + (l >> 2);
    const float* xr = X + row_id(row < n ? row : n - 1) * d;
    float mx = 0.f;
    for (int j = 4 * (l & 3); j < d; j += 16) {
      const f32x4 v = *reinterpret_cast<const f32x4_u*>(xr + min(j, d - 4));
      mx = fmaxf(fmaxf(mx, fabsf(v[0])), fmaxf(fabsf(v[1]), fmaxf(fabsf(v[2]), fabsf(v[3]))));
    }
    // the four lanes of a row (quad permutations: lane ^ 1, lane ^ 2)
    mx = fmaxf(mx, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(mx), 0xb1, 0xf,
                                                              0xf, true)));
    mx = fmaxf(mx, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(mx), 0x4e, 0xf,
                                                              0xf, true)));
    // (0: zeros, which any scale takes)
    const uint32_t ex = mx == 0.f ? 0u : __float_as_uint(pow2_scale(mx)) >> 23;
    if ((l & 3) == 0) s_ex[(w * MB + pb) * 16 + (l >> 2)] = ex;
    if (ex) rng = __builtin_elementwise_max(rng, u16x2{(uint16_t)ex, (uint16_t)(255u - ex)});
  }
#pragma unroll
  for (int off = 4; off < kWave; off <<= 1)
    rng = __builtin_elementwise_max(
        rng, __builtin_bit_cast(
                 u16x2, __shfl_xor(__builtin_bit_cast(uint32_t, rng), off, kWave)));
  if (l == 0) s_rng[w] = __builtin_bit_cast(uint32_t, rng);
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kLB / kWave; ++u)
    rng = __builtin_elementwise_max(rng, __builtin_bit_cast(u16x2, s_rng[u]));
  uint32_t ex = rng.x ? 255u - rng.y : 127u;
  if (rng.x > ex + kApart) {  // uniform over the block
    s_hist[t] = 0;
    __syncthreads();
    if (t < kRows && s_ex[t]) atomicAdd((uint32_t*)&s_hist[s_ex[t]], 1u);
    __syncthreads();
    uint32_t upto = wave_incl_scan_dpp((uint32_t)s_hist[t]);
    if (l == kWave - 1) s_key[0][w] = upto;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kLB / kWave; ++u) upto += u < w ? s_key[0][u] : 0u;
    s_upto[t] = upto;
    __syncthreads();
    uint32_t key = s_hist[t] ? scale_cost(t, s_hist, s_upto) << 8 | (uint32_t)t : ~0u;
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) key = min(key, __shfl_xor(key, off, kWave));
    if (l == 0) s_key[1][w] = key;
    __syncthreads();  // (and the tiles may have their room)
#pragma unroll
    for (int u = 0; u < kLB / kWave; ++u) key = min(key, s_key[1][u]);
    ex = key & 255u;
  }
  const float sx = __uint_as_float(ex << 23);
  const float isx = 1.0f / sx;  // exact: powers of two
  uint16_t* sw = s_c + kBN * LROW + w * 16 * LROW;
#pragma unroll
  for (int pb = 0; pb < MB; ++pb) {
    const int64_t row = p0 + pb * 16 + (l >> 2);
    const bool ok = row < n;
    const float* xr = X + row_id(ok ? row : n - 1) * d;
    uint16_t* sr = sw + (l >> 2) * LROW;
    float s2 = 0, sh = 0, sl = 0, se = 0;
    const float sy = ok ? sx : 0.f;  // (rows past the end: zeros)
    // one coordinate's halves, its share of the norms added
    auto split = [&](float x, _Float16& h, _Float16& lo) {
      const float y = x * sy;
      h = f16_half(y);
      const float r = y - (float)h;  // exact
      s2 += y * y;
      sh += (float)h * (float)h;
      if constexpr (TERMS == 1) {
        lo = (_Float16)0.f;
        se += r * r;
      } else {
        lo = f16_half(r);
        const float e = r - (float)lo;  // exact
        sl += (float)lo * (float)lo;
        se += e * e;
      }
    };
    if (x4) {
      for (int j = 4 * (l & 3); j < d; j += 16) {
        const f32x4 v = *reinterpret_cast<const f32x4_u*>(xr + j);
        f16x4 h, lo;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          _Float16 a, b;
          split(v[u], a, b);
          h[u] = a;
          lo[u] = b;
        }
        *reinterpret_cast<f16x4_lds*>(&sr[j]) = h;
        if constexpr (TERMS == 3 && SPLIT) {
          *reinterpret_cast<f16x4_lds*>(&sr[RH / 2 + j]) = lo;
        } else if constexpr (TERMS == 3) {
          *reinterpret_cast<f16x4_lds*>(&sr[d + j]) = lo;
          *reinterpret_cast<f16x4_lds*>(&sr[2 * d + j]) = h;
        }
      }
    } else {
      for (int j = 4 * (l & 3); j < d; j += 16) {
        const int jc = min(j, d - 4);
        const f32x4 v = *reinterpret_cast<const f32x4_u*>(xr + jc);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int ju = jc + u;
          if (ju < j) continue;  // the piece before has it
          _Float16 h, lo;
          split(v[u], h, lo);
          sr[ju] = f16_bits(h);
          if constexpr (TERMS == 3 && SPLIT) {
            sr[RH / 2 + ju] = f16_bits(lo);
          } else if constexpr (TERMS == 3) {
            sr[d + ju] = f16_bits(lo);
            sr[2 * d + ju] = f16_bits(h);
          }
        }
      }
    }
    if constexpr (TERMS == 1) {
      for (int j = d + (l & 3); j < RH; j += 4) sr[j] = 0;
    } else if constexpr (SPLIT) {
      for (int j = d + (l & 3); j < RH / 2; j += 4) sr[j] = sr[RH / 2 + j] = 0;
    } else {
      for (int j = 3 * d + (l & 3); j < RH; j += 4) sr[j] = 0;
    }
#pragma unroll
    for (int off = 1; off < 4; off <<= 1) {
      s2 += __shfl_xor(s2, off, kWave);
      sh += __shfl_xor(sh, off, kWave);
      sl += __shfl_xor(sl, off, kWave);
      se += __shfl_xor(se, off, kWave);
    }
    if ((l & 3) == 0) {  // norms rounded up: the bound stays rigorous
      float* st = s_st[w * MB * 16 + pb * 16 + (l >> 2)];
      const float up = (1.f + 4e-5f) * isx;
      // d squares that went to zero (below the smallest normal value) are less
      const float gone = (float)d * 1.17549435e-38f;
      st[0] = sqrtf(s2 + gone) * up;
      st[1] = sqrtf(sh + gone) * up;
      st[2] = sqrtf(sl + gone) * up;
      st[3] = sqrtf(se + gone) * up;
    }
#pragma unroll
    for (int f = 0; f < NF; ++f)
      pf[pb][f] = *reinterpret_cast<const f16x8_lds*>(&sw[lr * LROW + f * 32 + lq * 8]);
    asm volatile("" ::: "memory");  // the next block overwrites the rows
  }

  // Centroid tiles of the block's partitions in sequence, double buffered in
  // LDS: the next tile is fetched into registers before the current one is
  // multiplied and stored to the other buffer after it, so one barrier per
  // tile and the L2 latency overlaps the MFMAs.
  constexpr int VPR = RH / 8;                       // uint4 per row
  constexpr int VPG = (TERMS == 1 ? 2 : 1) * VPR;   // the same in memory (h and l rows)
  static_assert((kBN * VPR) % kLB == 0 && kBN <= kLB, "a tile splits evenly over the block");
  constexpr int NV = kBN * VPR / kLB;
  u32x4 pv[NV];
  float pnc;
  float ncs = 0.f;  // -||c||^2 / 2 in the accumulators' scale
  // Rows past the partition repeat its last centroid (every partition has
  // one; the host checks k >= 1) and start from -inf, so the epilogue never
  // takes them. Fetch and store
  // are branch-free: the loads are unconditional, every thread loads a norm
  // (kLB / kBN threads store the same value to each entry) and the defaults
  // are chosen when the tile is stored. A register write to a load's
  // destination next to the load, or a load skipped on some lanes, would make
  // the wave wait for the new tile there, before the MFMAs, and undo the
  // double buffering. Row indices are 32-bit offsets from the tile's first
  // centroid.
  int32_t f_rem = 0;
  auto fetch = [&](int64_t c0, int64_t kend) {
    const int32_t rem = (int32_t)(kend - c0 < kBN ? kend - c0 : kBN);  // >= 1 rows left
    const u32x4* bh = reinterpret_cast<const u32x4*>(Cf + c0 * (VPG * 8));
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int v = t + i * kLB;
      const int32_t r = min(v / VPR, rem - 1);
      pv[i] = bh[r * VPG + v % VPR];
    }
    pnc = ncf[c0 + min(t % kBN, rem - 1)];
    f_rem = rem;
  };
  auto stash = [&](int b) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int v = t + i * kLB;
      *reinterpret_cast<u32x4_lds*>(&s_c[b * kBN * LROW + (v / VPR) * LROW + (v % VPR) * 8]) =
          pv[i];
    }
    s_nc[b][t % kBN] = (t % kBN) < f_rem ? pnc * ncs : -INFINITY;
  };
  auto part_scale = [&](int q) { return pow2_scale(__uint_as_float(pstat[q * kStat + 4])); };
  int p = pa, buf = 0;
  if (pa >= pz) return;  // uniform over the block
  int64_t c0 = k_off[pa];
  float scp = part_scale(pa);
  ncs = -0.5f * sx * scp;
  fetch(c0, k_off[pa + 1]);
  stash(0);
  __syncthreads();
  for (; p < pz; ++p) {
    const int64_t kbeg = k_off[p], kend = k_off[p + 1];
    const float isc = 1.0f / scp;
    float d1[MB], d2[MB];
    int32_t k1[MB];
#pragma unroll
    for (int pb = 0; pb < MB; ++pb) {
      d1[pb] = -FLT_MAX;
      d2[pb] = -FLT_MAX;
      k1[pb] = -kGrp;
    }
    for (c0 = kbeg; c0 < kend; c0 += kBN) {
      // the next tile: this partition's, else the next partition's first
      int64_t nc0 = c0 + kBN, nend = kend;
      if (nc0 >= kend && p + 1 < pz) {
        nc0 = kend;
        nend = k_off[p + 2];
        scp = part_scale(p + 1);
        ncs = -0.5f * sx * scp;
      }
      const bool more = nc0 < nend;
      if (more) fetch(nc0, nend);
      const uint16_t* sc = s_c + buf * kBN * LROW;
      const int32_t gb = __builtin_amdgcn_readfirstlane((int32_t)(c0 - kbeg));
#pragma unroll
      for (int cb = 0; cb < kBN / 16; ++cb) {
        f16x8 af[NF];
#pragma unroll
        for (int f = 0; f < NF; ++f)
          af[f] = *reinterpret_cast<const f16x8_lds*>(&sc[(cb * 16 + lr) * LROW + f * 32 + lq * 8]);
        const f32x4 nc = *reinterpret_cast<const f32x4*>(&s_nc[buf][cb * 16 + lq * 4]);
        f32x4 acc[MB];
#pragma unroll
        for (int pb = 0; pb < MB; ++pb) acc[pb] = nc;  // (the first MFMA's addend)
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          // split rows: h.h, h.l, l.h per fragment
          const int a = SPLIT && TERMS == 3 ? (s % 3 == 1 ? KB + s / 3 : s / 3) : s;
          const int b = SPLIT && TERMS == 3 ? (s % 3 == 2 ? KB + s / 3 : s / 3) : s;
#pragma unroll
          for (int pb = 0; pb < MB; ++pb)
            acc[pb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[a], pf[pb][b], acc[pb], 0, 0, 0);
        }
        // x.c - ||c||^2 / 2 of four consecutive centroids, their maximum, and
        // the running top two of the groups
        const int32_t id = gb + cb * 16;  // uniform; the lane's quad comes at the end
#pragma unroll
        for (int pb = 0; pb < MB; ++pb) {
          // (the NaN-propagating maximum: the other one costs an instruction
          // per accumulator that quiets signalling NaNs)
          const float m3 = __builtin_elementwise_maximum(
              __builtin_elementwise_maximum(acc[pb][0], acc[pb][1]), acc[pb][2]);
          const float m = __builtin_elementwise_maximum(m3, acc[pb][3]);
          const bool take = m > d1[pb];
          d2[pb] = __builtin_amdgcn_fmed3f(d1[pb], d2[pb], m);
          d1[pb] = take ? m : d1[pb];
          k1[pb] = take ? id : k1[pb];
        }
      }
      // the epilogue stays ahead of the tile store: its VALU work covers the
      // latency of the next tile's loads (left alone, the compiler sinks it
      // below the store and the barrier, which then wait right after the MFMAs)
#pragma unroll
      for (int pb = 0; pb < MB; ++pb)
        asm volatile("" : "+v"(d1[pb]), "+v"(d2[pb]), "+v"(k1[pb])::"memory");
      if (more) {
        stash(buf ^ 1);  // last read in the previous tile, before its barrier
        __syncthreads();
        buf ^= 1;
      }
    }
    // merge the four lanes of a point (lower group on equal maxima), then lane
    // (lq, lr) finishes point block lq
    float st[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) st[q] = __uint_as_float(pstat[p * kStat + q]);
    float D1 = 0.f, D2 = 0.f;
    int32_t K1 = -1;
#pragma unroll
    for (int pb = 0; pb < MB; ++pb) {
      float a1 = d1[pb], a2 = d2[pb];
      int32_t k = k1[pb] < 0 ? INT_MAX : k1[pb] + kGrp * lq;
#pragma unroll
      for (int off = 16; off < 64; off <<= 1) {
        const float o1 = __shfl_xor(a1, off, kWave);
        const float o2 = __shfl_xor(a2, off, kWave);
        const int32_t ok = __shfl_xor(k, off, kWave);
        a2 = fmaxf(fmaxf(a2, o2), fminf(a1, o1));
        const bool take = o1 > a1 || (o1 == a1 && ok < k);
        a1 = take ? o1 : a1;
        k = take ? ok : k;
      }
      if (lq == pb) {
        D1 = a1;
        D2 = a2;
        K1 = k;
      }
    }
    const bool mine = l < MB * 16 && p0 + l < n;
    const int64_t row = row_id(mine ? p0 + l : row0);
    const int32_t g = K1 == INT_MAX ? 0 : K1;  // first centroid of the group
    bool flagged = false;
    if (mine) {
      const float E = point_bound<TERMS>(s_st[w * MB * 16 + l], st, d);
      const float margin = (D1 - D2) * (2.f * isx * isc);  // in squared distance
      // no group taken (all values infinite or NaN): re-scored as well
      flagged = !(margin > 2.f * E) || K1 == INT_MAX;
      if (!FUSE) labels[(int64_t)p * n + row] = g;
    }
    // append flagged (p, row) pairs: one atomic per wave
    const uint64_t fm = __ballot(flagged);
    if (fm) {
      // flags go to one of kFlagSlots regions (by block): counters on one
      // address would serialise one atomic per wave and partition
      const int slot = blockIdx.x % kFlagSlots;
      unsigned long long base = 0;
      if (l == 0) base = atomicAdd(&nflag[slot], (unsigned long long)__popcll(fm));
      base = __shfl(base, 0, kWave);
      if (flagged) {
        const unsigned long long o = base + __popcll(fm & lanemask_lt());
        if (o < (unsigned long long)region)
          flags[(int64_t)slot * region + (int64_t)o] = ((uint64_t)p << 40) | (uint64_t)row;
      }
    }
    if constexpr (FUSE) {
      // one partition: pick the nearest of the group right here, 16 points at
      // a time, while the other waves multiply (the rows were read when the
      // wave started and come from the last-level cache)
      __syncthreads();  // the centroid tiles are consumed: their LDS is free
      float* sf = reinterpret_cast<float*>(s_raw) + w * kRsLds;
#pragma unroll 1
      for (int it = 0; it < MB; ++it) {
        const int src = it * 16 + l / kGrp;
        const int32_t gi = __shfl(g, src, kWave);
        const int64_t ri = __shfl(row, src, kWave);
        const bool ok = __shfl((int)mine, src, kWave);
        double best;
        int32_t bk;
        if (x4) resolve16<true>(X, d, C, kbeg, kend, ri, gi, sf, best, bk);
        else resolve16<false>(X, d, C, kbeg, kend, ri, gi, sf, best, bk);
        if (ok && l % kGrp == 0) {
          labels[ri] = bk;
          if (dists) dists[ri] = (float)best;
        }
      }
      return;  // (the only partition: the fragments need not outlive the tiles)
    }
  }
}

// acc + diff^2 with separately rounded multiply and add in FP64 (the
// oracle's arithmetic: no fused multiply-add), plain expression otherwise.
// HIP's __dmul_rn / __dadd_rn are plain operators that the compiler may
// contract into one fma; the pragma keeps the two roundings.
__device__ __forceinline__ double sq_acc(double acc, double diff) {
#pragma clang fp contract(off)
  return acc + diff * diff;
}
__device__ __forceinline__ float sq_acc(float acc, float diff) {
  return __builtin_fmaf(diff, diff, acc);
}

// Squared distance of two float rows in FP64, accumulated in ascending
// dimension order (the oracle's arithmetic); 16-byte loads when both rows
// are 16-byte aligned and d is a multiple of 4.
__device__ __forceinline__ double dist2_f64(const float* __restrict__ x,
                                           const float* __restrict__ c, int d, bool vec4) {
  double acc = 0.0;
  if (vec4) {
    const float4* x4 = reinterpret_cast<const float4*>(x);
    const float4* c4 = reinterpret_cast<const float4*>(c);
    for (int j = 0; j < d / 4; ++j) {
      const float4 xv = x4[j], cv = c4[j];
      acc = sq_acc(acc, (double)xv.x - (double)cv.x);
      acc = sq_acc(acc, (double)xv.y - (double)cv.y);
      acc = sq_acc(acc, (double)xv.z - (double)cv.z);
      acc = sq_acc(acc, (double)xv.w - (double)cv.w);
    }
  } else {
    int j = 0;
    for (; j + 8 <= d; j += 8) {  // eight loads in flight, then the chain
      float xv[8], cv[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        xv[u] = x[j + u];
        cv[u] = c[j + u];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) acc = sq_acc(acc, (double)xv[u] - (double)cv[u]);
    }
    for (; j < d; ++j) acc = sq_acc(acc, (double)x[j] - (double)c[j]);
  }
  return acc;
}

// The screen's bounds: R (relative, as a factor on the smallest screened
// value) and A (absolute underflow slack), see k_rescore_tiled.
__device__ __forceinline__ void screen_bounds(int d, float& R, float& A) {
  const double ug = 1.1920928955078125e-07, u64 = 1.1102230246251565e-16;
  const double gs = (d + 2) * ug / (1.0 - (d + 2) * ug);
  const double g64 = (d + 2) * 2 * u64 / (1.0 - (d + 2) * 2 * u64);
  R = (float)((1.0 + gs) * (1.0 + g64) / ((1.0 - gs) * (1.0 - g64)) * (1.0 + 1e-6));
  A = (float)d * 4.7e-38f;  // >= d * 2^-124
}

// The re-scorings' full pass over a subset of the centroids, which includes the
// partition's first when `first`: strict < in ascending order. A NaN never
// replaces a distance, and nothing replaces a NaN of the first centroid, which
// stands here as -infinity (rescored_dist gives it back).
__device__ __forceinline__ void full_min(double a, bool first, int32_t c, double& best,
                                         int32_t& bk) {
  if (first && a != a) a = -(double)INFINITY;
  if (a < best || (bk < 0 && a == a)) {
    best = a;
    bk = c;
  }
}
__device__ __forceinline__ float rescored_dist(double best) {
  return best == -(double)INFINITY ? __builtin_nanf("") : (float)best;
}

// Re-scoring of few flagged points (d <= 128): a block takes up to F flags of
// one partition at a time. Its threads hold U centroids each, read from the
// transposed copy Ct [d][ktot] (64 consecutive floats per load), and walk the
// dimensions with the F points' coordinates broadcast from LDS, so each
// centroid value loaded serves F points and each coordinate U centroids. FP32
// screen, then FP64 for the candidates, by the bounds of k_rescore_tiled; a
// thread that may hold more candidates than it kept makes the block score
// every centroid in FP64.
// The flags are a list (nflag or *d_nflag of them), or (cnt) still lie in the
// regions of the labeling; then kFewMax or more are left alone.
// BS threads: 256 while flags are few, and the workgroups for them too; many
// flags of partitions of up to kRfOneK centroids, most of which would leave
// lanes of four wavefronts idle, go by one wavefront each, four times as many
// workgroups at a time. 30,000 x 100-d points with 14,000 to 27,000 flags, 10
// partitions of 30 centroids: a call 366 and 263 us, 150: 486 and 374, 600: 756
// and 626, 1500: 1138 and 1219; one of 100,000 x 64-d with 22,000 to 47,000
// flags, 40: 210 and 128, 500: 385 and 224, 1000: 407 and 388; but with 200
// flags, 100 centroids 102 and 114, 500 123 and 136.
constexpr int kRfF = 4;
constexpr int64_t kFewMax = 8192, kRfOneK = 600;
template <int F, int BS>
__global__ __launch_bounds__(BS, 4) void k_rescore_few(
    const float* __restrict__ X, int64_t n, int d, const float* __restrict__ C,
    const float* __restrict__ Ct, int64_t ktot, const int64_t* __restrict__ k_off,
    const uint64_t* __restrict__ list, int64_t nflag, int32_t* __restrict__ labels,
    float* __restrict__ dists, const int64_t* __restrict__ d_nflag,
    const unsigned long long* __restrict__ cnt, int64_t region) {
  constexpr int U = 4;  // centroids per thread and pass
  constexpr int NW = BS / kWave;
  __shared__ float s_x[128 * F];
  __shared__ uint64_t s_f[F];
  __shared__ float s_min[F][NW];
  __shared__ double s_best[F][NW];
  __shared__ int32_t s_bk[F][NW];
  __shared__ unsigned long long s_pre[kFlagSlots + 1];
  const int t = threadIdx.x, w = t / kWave, l = lane_id();
  if (d_nflag) nflag = *d_nflag;  // count left on the device (capturable calls)
  if (cnt) {  // the flags lie in their regions: entries before each
    if (t < kWave) {
      const uint32_t c = (uint32_t)cnt[l];
      const uint32_t incl = wave_incl_scan(c);
      s_pre[l] = incl - c;
      if (l == kWave - 1) s_pre[kFlagSlots] = incl;
    }
    __syncthreads();
    nflag = (int64_t)s_pre[kFlagSlots];
    if (nflag >= kFewMax) return;  // left to the host (uniform over the grid)
  }
  auto flag_at = [&](int64_t f) {
    if (!cnt) return list[f];
    int lo = 0, hi = kFlagSlots;  // slot with s_pre[lo] <= f < s_pre[lo + 1]
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (s_pre[mid] <= (unsigned long long)f) lo = mid; else hi = mid;
    }
    return list[(int64_t)lo * region + (f - (int64_t)s_pre[lo])];
  };
  float R, A;
  screen_bounds(d, R, A);
  for (int64_t f0 = (int64_t)blockIdx.x * F; f0 < nflag; f0 += (int64_t)gridDim.x * F) {
    const int nf = nflag - f0 < F ? (int)(nflag - f0) : F;
    if (t < nf) s_f[t] = flag_at(f0 + t);
    __syncthreads();
    for (int done = 0; done < nf;) {  // runs of one partition (block-uniform)
      const int p = (int)(s_f[done] >> 40);
      int end = done + 1;
      while (end < nf && (int)(s_f[end] >> 40) == p) ++end;
      const int64_t kbeg = k_off[p], kend = k_off[p + 1];
      const float* x[F];
#pragma unroll
      for (int q = 0; q < F; ++q) {
        const int f = done + q < end ? done + q : done;  // a missing flag repeats one
        x[q] = X + (int64_t)(s_f[f] & kFlagRow) * d;
      }
      __syncthreads();  // the previous run's rows and results are consumed
      for (int j = t; j < d; j += BS)
#pragma unroll
        for (int q = 0; q < F; ++q) s_x[j * F + q] = x[q][j];
      __syncthreads();
      float v1[F], v2[F];
      int32_t k1[F];
#pragma unroll
      for (int q = 0; q < F; ++q) {
        v1[q] = INFINITY;
        v2[q] = INFINITY;
        k1[q] = -1;
      }
      const bool any = kbeg + t < kend;  // this thread has a centroid
      bool full = false;
      for (int64_t c0 = kbeg; c0 < kend; c0 += BS * U) {
        // U centroids a thread, every coordinate of theirs for all F points
        float a[U][F];
        const float* ct[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int64_t c = c0 + u * BS + t;
          ct[u] = Ct + (c < kend ? c : kend - 1);
#pragma unroll
          for (int q = 0; q < F; ++q) a[u][q] = 0.f;
        }
        const int nu = kend - c0 >= BS * U ? U : (int)((kend - c0 + BS - 1) / BS);  // uniform
        auto pass = [&](auto full_u) {
#pragma unroll 4
          for (int j = 0; j < d; ++j) {
            float cv[U];
#pragma unroll
            for (int u = 0; u < U; ++u)
              if (full_u.value || u < nu) cv[u] = ct[u][(int64_t)j * ktot];
#pragma unroll
            for (int u = 0; u < U; ++u)
              if (full_u.value || u < nu) {
#pragma unroll
                for (int q = 0; q < F; ++q) {
                  const float e = s_x[j * F + q] - cv[u];
                  a[u][q] = fmaf(e, e, a[u][q]);
                }
              }
          }
        };
        if (nu == U) pass(std::true_type{});
        else pass(std::false_type{});
        if (c0 == kbeg && t == 0) {  // a NaN of the first centroid decides
#pragma unroll
          for (int q = 0; q < F; ++q) full = full || a[0][q] != a[0][q];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int64_t c = c0 + u * BS + t;
          if (c < kend) {
#pragma unroll
            for (int q = 0; q < F; ++q) {
              const bool lt1 = a[u][q] < v1[q];
              v2[q] = __builtin_amdgcn_fmed3f(v1[q], v2[q], a[u][q]);
              k1[q] = lt1 ? (int32_t)(c - kbeg) : k1[q];
              v1[q] = lt1 ? a[u][q] : v1[q];
            }
          }
        }
      }
#pragma unroll
      for (int q = 0; q < F; ++q) {
        float m = v1[q];
#pragma unroll
        for (int off = kWave / 2; off > 0; off >>= 1) m = fminf(m, __shfl_xor(m, off, kWave));
        if (l == 0) s_min[q][w] = m;
      }
      __syncthreads();
      double best[F];
      int32_t bk[F];
#pragma unroll
      for (int q = 0; q < F; ++q) {
        float m = s_min[q][0];
#pragma unroll
        for (int u = 1; u < NW; ++u) m = fminf(m, s_min[q][u]);
        const float T = (m + A) * R + A;
        best[q] = DBL_MAX;
        bk[q] = -1;
        if (k1[q] >= 0 && v1[q] <= T) {
          best[q] = dist2_f64(x[q], C + (kbeg + k1[q]) * d, d, false);
          bk[q] = k1[q];
        }
        // (NaN screens take the full pass)
        full = full || (any && (k1[q] < 0 || !(v2[q] > T)));
      }
      if (__syncthreads_or(full)) {
#pragma unroll
        for (int q = 0; q < F; ++q) {
          best[q] = DBL_MAX;
          bk[q] = -1;
        }
        for (int64_t c = kbeg + t; c < kend; c += BS) {
#pragma unroll
          for (int q = 0; q < F; ++q) {
            full_min(dist2_f64(x[q], C + c * d, d, false), c == kbeg, (int32_t)(c - kbeg),
                     best[q], bk[q]);
          }
        }
      }
#pragma unroll
      for (int q = 0; q < F; ++q) {
#pragma unroll
        for (int off = kWave / 2; off > 0; off >>= 1) {
          const double ob = __shfl_xor(best[q], off, kWave);
          const int32_t ok = __shfl_xor(bk[q], off, kWave);
          if (ok >= 0 && (bk[q] < 0 || ob < best[q] || (ob == best[q] && ok < bk[q]))) {
            best[q] = ob;
            bk[q] = ok;
          }
        }
        if (l == 0) {
          s_best[q][w] = best[q];
          s_bk[q][w] = bk[q];
        }
      }
      __syncthreads();
      if (t < end - done) {
        double b = s_best[t][0];
        int32_t k = s_bk[t][0];
        for (int u = 1; u < NW; ++u) {
          const double ob = s_best[t][u];
          const int32_t ok = s_bk[t][u];
          if (ok >= 0 && (k < 0 || ob < b || (ob == b && ok < k))) {
            b = ob;
            k = ok;
          }
        }
        const int64_t o =
            (int64_t)p * n + (int64_t)(s_f[done + t] & kFlagRow);
        labels[o] = k;
        if (dists) dists[o] = rescored_dist(b);
      }
      __syncthreads();  // the shared results are consumed
      done = end;
    }
    __syncthreads();  // and the flags
  }
}

// FP64 re-scoring with the partition's centroids staged in LDS, for flags
// sorted by partition: a block takes 64 flags; four threads per flag split
// the centroids (c = s, s+4, ... ascending, two chains at a time) and read
// them from LDS tiles shared by all 64 flags, so each centroid is read from
// memory once per 64 flagged points instead of once per point.
//
// Screen first: the FP32 direct difference S = sum fl(x_j - c_j)^2 (fused
// multiply-add) is within a factor (1 +- g) of the exact distance D, g =
// gamma_{d+2} (d + 2 roundings, unit 2^-23 for safety), plus an absolute
// underflow slack A; the oracle's FP64 sum is within (1 +- g64) of D. With m
// the smallest screened value, a centroid whose screened value exceeds
// T = (m + A) R + A, R = (1+g)(1+g64) / ((1-g)(1-g64)), has an oracle distance
// strictly above the oracle distance of the true nearest centroid, so it can
// be neither the oracle's minimum nor tied with it. Each thread keeps its two
// smallest screened values; the candidates (screened value <= T, usually one
// per flag) are re-scored with the oracle's FP64 arithmetic, lowest index on
// equal values (the oracle's first minimum). A flag where some thread's
// second-smallest value is also <= T may have more candidates than were kept:
// the block then re-scores its run in FP64 against every centroid, strict < in
// ascending order inside a subset, lowest index among equal minima across the
// four subsets.
constexpr int kRtF = 64;  // flags per block
constexpr int kRtS = 4;   // threads per flag
constexpr int kRtT = 64;  // centroids per LDS tile
// point rows: stride d + 1 (lanes read different rows: conflict-free);
// centroid rows: stride rounded up to 4 floats, zero padded (every lane of a
// wave reads the same row: broadcast 16-byte reads)
inline int rescore_cstride(int d) { return (d + 3) & ~3; }
inline size_t rescore_tiled_lds(int d) {
  return ((size_t)kRtF * (d + 1) + (size_t)kRtT * rescore_cstride(d)) * sizeof(float);
}
// DX > 0: the screen keeps the point's d <= DX coordinates in registers.
template <int DX>
__global__ __launch_bounds__(kRtF * kRtS) void k_rescore_tiled(
    const float* __restrict__ X, int64_t n, int d, const float* __restrict__ C,
    const int64_t* __restrict__ k_off, const uint64_t* __restrict__ flags, int64_t nflag,
    int32_t* __restrict__ labels, float* __restrict__ dists,
    const int64_t* __restrict__ d_nflag = nullptr) {
  extern __shared__ __align__(16) float s_dyn[];
  __shared__ double s_best[kRtS][kRtF];
  __shared__ int32_t s_bk[kRtS][kRtF];
  __shared__ float s_v1[kRtS][kRtF];
  constexpr uint64_t kRowMask = (1ull << 40) - 1;
  const int RS = d + 1;
  const int RC = (d + 3) & ~3;
  float* s_x = s_dyn;
  float* s_c = s_dyn + kRtF * RS;  // 16-byte aligned: kRtF * RS * 4 = 256 (d + 1) bytes
  const int t = threadIdx.x, g = t & (kRtF - 1), sub = t / kRtF;
  if (d_nflag) nflag = *d_nflag;  // count left on the device: tiles in a loop
  for (int64_t f0 = (int64_t)blockIdx.x * kRtF; f0 < nflag; f0 += (int64_t)gridDim.x * kRtF) {
  const int cnt = nflag - f0 < kRtF ? (int)(nflag - f0) : kRtF;
  float R, A;
  screen_bounds(d, R, A);
  for (int done = 0; done < cnt;) {  // runs of one partition (block-uniform)
    const int p = (int)(flags[f0 + done] >> 40);
    int end = done + 1;
    while (end < cnt && (int)(flags[f0 + end] >> 40) == p) ++end;
    for (int v = t; v < (end - done) * d; v += kRtF * kRtS) {
      const int r = v / d, j = v - r * d;
      s_x[r * RS + j] = X[(int64_t)(flags[f0 + done + r] & kRowMask) * d + j];
    }
    const bool active = g >= done && g < end;
    const float* xa = s_x + (active ? g - done : 0) * RS;
    const int64_t kbeg = k_off[p], kend = k_off[p + 1];
    // pass 1: FP32 screen, two smallest values per thread
    float v1 = INFINITY, v2 = INFINITY;
    int64_t k1 = -1;
    auto keep = [&](float v, int64_t k) {
      const bool lt1 = v < v1;
      v2 = __builtin_amdgcn_fmed3f(v1, v2, v);
      k1 = lt1 ? k : k1;
      v1 = lt1 ? v : v1;
    };
    // staged centroid rows, zero padded to RC columns
    auto stage = [&](int64_t c0, int rows) {
      for (int v = t; v < rows * RC; v += kRtF * kRtS) {
        const int r = v / RC, j = v - r * RC;
        s_c[v] = j < d ? C[(c0 + r) * d + j] : 0.f;
      }
    };
    constexpr int NX = DX > 0 ? DX : 1;
    float xr[NX];
    bool full = false;
    __syncthreads();  // the point rows are staged
    if constexpr (DX > 0) {
#pragma unroll
      for (int j = 0; j < NX; ++j) xr[j] = j < d ? xa[j] : 0.f;
    }
    const int nq = RC / 4;
    // screened value of one staged row (padding adds exact zeros)
    auto screen = [&](const float* cr) {
      float a = 0.f;
      if constexpr (DX > 0) {
        const float4* c4 = reinterpret_cast<const float4*>(cr);
#pragma unroll
        for (int q = 0; q < NX / 4; ++q) {
          if (q < nq) {
            const float4 u = c4[q];
            float e = xr[4 * q] - u.x;
            a = fmaf(e, e, a);
            e = xr[4 * q + 1] - u.y;
            a = fmaf(e, e, a);
            e = xr[4 * q + 2] - u.z;
            a = fmaf(e, e, a);
            e = xr[4 * q + 3] - u.w;
            a = fmaf(e, e, a);
          }
        }
      } else {
        for (int j = 0; j < d; ++j) {
          const float e = xa[j] - cr[j];
          a = fmaf(e, e, a);
        }
      }
      return a;
    };
    for (int64_t c0 = kbeg; c0 < kend; c0 += kRtT) {
      const int rows = kend - c0 < kRtT ? (int)(kend - c0) : kRtT;
      __syncthreads();  // the rows are staged, the previous tile is consumed
      stage(c0, rows);
      __syncthreads();
      if (!active) continue;
      if (c0 == kbeg && sub == 0) {  // a NaN of the first centroid decides
        const float a0 = screen(s_c);
        full = a0 != a0;
      }
      int c = sub;
      for (; c + kRtS < rows; c += 2 * kRtS) {
        const float a0 = screen(s_c + c * RC);
        const float a1 = screen(s_c + (c + kRtS) * RC);
        keep(a0, c0 + c);
        keep(a1, c0 + c + kRtS);
      }
      for (; c < rows; c += kRtS) keep(screen(s_c + c * RC), c0 + c);
    }
    s_v1[sub][g] = v1;
    __syncthreads();
    {
      float m = s_v1[0][g];
      for (int q = 1; q < kRtS; ++q) m = fminf(m, s_v1[q][g]);
      const float T = (m + A) * R + A;
      double best = DBL_MAX;
      int32_t bk = -1;
      if (active && k1 >= 0 && v1 <= T) {
        best = dist2_f64(xa, C + k1 * d, d, false);
        bk = (int32_t)(k1 - kbeg);
      }
      full = full || (active && (k1 < 0 || !(v2 > T)));  // (NaN screens take the full pass)
      s_best[sub][g] = best;
      s_bk[sub][g] = bk;
    }
    // pass 2 (rare): every centroid in FP64 for the whole run
    if (__syncthreads_or(full)) {
      double best = DBL_MAX;
      int32_t bk = -1;
      for (int64_t c0 = kbeg; c0 < kend; c0 += kRtT) {
        const int rows = kend - c0 < kRtT ? (int)(kend - c0) : kRtT;
        __syncthreads();
        stage(c0, rows);
        __syncthreads();
        if (!active) continue;
        for (int c = sub; c < rows; c += kRtS) {
          const float* ca = s_c + c * RC;
          double a0 = 0.0;
          for (int j = 0; j < d; ++j) a0 = sq_acc(a0, (double)xa[j] - (double)ca[j]);
          full_min(a0, c0 + c == kbeg, (int32_t)(c0 + c - kbeg), best, bk);
        }
      }
      s_best[sub][g] = best;
      s_bk[sub][g] = bk;
      __syncthreads();
    }
    if (active && sub == 0) {
      double b = s_best[0][g];
      int32_t k = s_bk[0][g];
      for (int q = 1; q < kRtS; ++q) {
        const double ob = s_best[q][g];
        const int32_t ok = s_bk[q][g];
        if (ok >= 0 && (k < 0 || ob < b || (ob == b && ok < k))) { b = ob; k = ok; }
      }
      const int64_t o = (int64_t)p * n + (int64_t)(flags[f0 + g] & kRowMask);
      labels[o] = k;
      if (dists) dists[o] = rescored_dist(b);
    }
    __syncthreads();
    done = end;
  }
  }  // tiles
}

// Concatenates the kFlagSlots flag regions (counts cnt[slot]) into one list.
__global__ void k_gather_flags(const uint64_t* __restrict__ regions, int64_t region,
                               const unsigned long long* __restrict__ cnt,
                               uint64_t* __restrict__ out, int64_t total,
                               const int64_t* __restrict__ d_total = nullptr) {
  __shared__ unsigned long long s_pre[kFlagSlots + 1];
  if (d_total) total = *d_total;
  if (threadIdx.x == 0) {
    unsigned long long a = 0;
    for (int q = 0; q < kFlagSlots; ++q) {
      s_pre[q] = a;
      a += cnt[q];
    }
    s_pre[kFlagSlots] = a;
  }
  __syncthreads();
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    int lo = 0, hi = kFlagSlots;  // slot q with s_pre[q] <= i < s_pre[q+1]
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (s_pre[mid] <= (unsigned long long)i) lo = mid; else hi = mid;
    }
    out[i] = regions[(int64_t)lo * region + (i - (int64_t)s_pre[lo])];
  }
}

// resolve16 for every (point, partition): labels holds the group's first
// centroid and receives the label, dists (nullable) its distance as float32
// like the reference's dists array. A block takes kPG partitions (grid.y over
// partition groups) with the partitions innermost, so a point's row is read
// from memory once per group and from cache for the other partitions.
constexpr int kPG = 8;
template <bool V4>
__global__ __launch_bounds__(256) void k_resolve(const float* __restrict__ X, int64_t n, int d,
                                                 const float* __restrict__ C,
                                                 const int64_t* __restrict__ k_off, int P,
                                                 int32_t* __restrict__ labels,
                                                 float* __restrict__ dists) {
  constexpr int PW = kWave / kGrp;  // points per wave
  __shared__ __align__(16) float s_rs[256 / kWave][kRsLds];
  const int w = threadIdx.x / kWave, l = lane_id();
  const int64_t step = (int64_t)gridDim.x * (256 / kGrp);
  for (int pg = blockIdx.y * kPG; pg < P; pg += gridDim.y * kPG) {
    const int pe = P - pg < kPG ? P : pg + kPG;
    // wave-uniform trip count
    for (int64_t i0 = ((int64_t)blockIdx.x * (256 / kWave) + w) * PW; i0 < n; i0 += step) {
      const int64_t i = i0 + l / kGrp;
      const bool valid = i < n;
      const int64_t row = valid ? i : n - 1;
      int32_t g = labels[(int64_t)pg * n + row];
      for (int p = pg; p < pe; ++p) {
        const int32_t gn = p + 1 < pe ? labels[(int64_t)(p + 1) * n + row] : 0;  // in flight
        double best;
        int32_t bk;
        resolve16<V4>(X, d, C, k_off[p], k_off[p + 1], row, g, s_rs[w], best, bk);
        if (valid && l % kGrp == 0) {
          labels[(int64_t)p * n + i] = bk;
          if (dists) dists[(int64_t)p * n + i] = (float)best;
        }
        g = gn;
      }
    }
  }
}

// The smaller one, a NaN left out.
__device__ __forceinline__ float min_of(float a, float b) { return __builtin_fminf(a, b); }
__device__ __forceinline__ double min_of(double a, double b) { return __builtin_fmin(a, b); }

// Direct-difference labeling: one thread per (PT points, partition), blocks of
// 256 PT points x one partition (grid.y over partitions, so a small data set
// with many partitions still fills the chip). The point sits in registers
// (DX = d exactly for d <= 4, else zero padded to DX: padding adds exact
// zeros) and the partition's centroids are staged in LDS, already converted
// to T, a tile of at most 16 KiB at a time. T = float: plain FP32; T =
// double: the oracle's FP64 arithmetic (ascending dimensions, strict <).
// PT points a lane (i and i + 256): a centroid read from LDS serves them all,
// and their chains of rounded operations overlap.
// Vector issue bounds it. Up to four dimensions the comparison costs as much
// as the distance, so it is made on the minimum of four (NaN rows fill the
// last four; a minimum leaves NaNs out, as the strict < does), and the best
// four of a tile are computed once more for the lowest index that gives the
// minimum. 10,000 points, 100 partitions of 50 to 100 centroids in 2-D in
// FP64: 35 us with one point a lane, 31 with two, 26 in fours. 300,000 points
// and 300 centroids, a call in FP64 (FP32), one by one and in fours: 62 and 51
// us in 1-D (53 and 47), 94 and 85 in 4-D (61 and 58), but 124 and 136 in 8-D,
// 223 and 234 in 16-D (111 and 128), where the loads of four rows stall. Beyond
// 64 dimensions the point alone fills the registers and a centroid is taken at a
// time: 200,000 x 128-d and 500 centroids in FP64 5.42 ms, two at a time 5.64.
template <typename T, int DX, int PT>
__global__ __launch_bounds__(256) void k_label_direct(const float* __restrict__ X, int64_t n,
                                                      int d, const float* __restrict__ C,
                                                      const int64_t* __restrict__ k_off, int P,
                                                      int32_t* __restrict__ labels,
                                                      float* __restrict__ dists) {
  constexpr int kTileRaw = 16384 / (DX * (int)sizeof(T));
  constexpr int kTile = kTileRaw > 256 ? 256 : kTileRaw;
  constexpr bool kFours = DX <= 4;
  __shared__ T s_c[kTile * DX];
  const int64_t i0 = (int64_t)blockIdx.x * (256 * PT) + threadIdx.x;
  T xr[PT][DX];
#pragma unroll
  for (int q = 0; q < PT; ++q)
#pragma unroll
    for (int j = 0; j < DX; ++j)
      xr[q][j] = (i0 + q * 256 < n && j < d) ? (T)X[(i0 + q * 256) * d + j] : T(0);
  auto dist_to = [&](int q, int r) {  // point q to the tile's row r
    T v = 0;
#pragma unroll
    for (int j = 0; j < DX; ++j) v = sq_acc(v, xr[q][j] - s_c[r * DX + j]);
    return v;
  };
  for (int p = blockIdx.y; p < P; p += gridDim.y) {
    const int64_t kbeg = k_off[p], kend = k_off[p + 1];
    T best[PT];
    int32_t bl[PT];
#pragma unroll
    for (int q = 0; q < PT; ++q) {
      best[q] = 0;
      bl[q] = -1;
    }
    for (int64_t c0 = kbeg; c0 < kend; c0 += kTile) {
      const int rows = (int)((kend - c0) < kTile ? (kend - c0) : kTile);
      const int stored = kFours ? (rows + 3) & ~3 : rows;
      __syncthreads();
      for (int v = threadIdx.x; v < stored * DX; v += blockDim.x) {
        const int r = v / DX, j = v - (v / DX) * DX;
        s_c[v] = r < rows ? (j < d ? (T)C[(c0 + r) * d + j] : T(0)) : (T)__builtin_nanf("");
      }
      __syncthreads();
      int r = 0;
      if (c0 == kbeg) {  // the first centroid wins whatever its distance is (a NaN stays)
#pragma unroll
        for (int q = 0; q < PT; ++q) {
          best[q] = dist_to(q, 0);
          bl[q] = 0;
        }
        r = kFours ? 0 : 1;
      }
      const int base = (int)(c0 - kbeg);
      if constexpr (kFours) {
        int bg[PT];  // the tile's best four, -1: none better than before
#pragma unroll
        for (int q = 0; q < PT; ++q) bg[q] = -1;
        for (; r < rows; r += 4) {
#pragma unroll
          for (int q = 0; q < PT; ++q) {
            T v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = dist_to(q, r + u);
            const T m = min_of(min_of(v[0], v[1]), min_of(v[2], v[3]));
            const bool less = m < best[q];
            best[q] = less ? m : best[q];
            bg[q] = less ? r : bg[q];
          }
        }
#pragma unroll
        for (int q = 0; q < PT; ++q)
          if (bg[q] >= 0) {
            int at = 0;
#pragma unroll
            for (int u = 3; u > 0; --u) at = dist_to(q, bg[q] + u) == best[q] ? u : at;
            at = dist_to(q, bg[q]) == best[q] ? 0 : at;
            bl[q] = base + bg[q] + at;
          }
      } else {
#pragma unroll (DX > 64 ? 1 : 2)
        for (; r < rows; ++r) {
#pragma unroll
          for (int q = 0; q < PT; ++q) {
            const T v = dist_to(q, r);
            const bool less = v < best[q];
            best[q] = less ? v : best[q];
            bl[q] = less ? base + r : bl[q];
          }
        }
      }
    }
#pragma unroll
    for (int q = 0; q < PT; ++q) {
      const int64_t i = i0 + q * 256;
      if (i < n) {
        labels[(int64_t)p * n + i] = bl[q];
        if (dists) dists[(int64_t)p * n + i] = (float)best[q];
      }
    }
  }
}

// numpy's float32 sum of one short row v[0..d), d <= 128 (numpy's add
// reduction along the last axis: 0 + the pairwise sum of the row; a row of
// at most PW_BLOCKSIZE = 128 elements is one leaf: fewer than 8 elements
// summed in order from 0, otherwise eight partial sums over v[j], v[j+8],
// ... up to the last multiple of 8, combined as ((r0+r1)+(r2+r3)) +
// ((r4+r5)+(r6+r7)), then the remaining elements added in order). Every
// operation is a separately rounded float32 addition.
// (x - c) ** 2 in float32: a rounded difference, then a rounded square; the
// pragma keeps the square from being fused into the row sum's additions.
__device__ __forceinline__ float np_square_diff(float x, float c) {
#pragma clang fp contract(off)
  const float df = x - c;
  return df * df;
}

template <int DX>
__device__ __forceinline__ float np_row_sum(const float* v, int d) {
#pragma clang fp contract(off)
  if (d < 8) {
    float r = 0.0f;
#pragma unroll
    for (int j = 0; j < (DX < 8 ? DX : 8); ++j)
      if (j < d) r = __fadd_rn(r, v[j]);
    return r;
  }
  float r[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) r[j] = j < DX ? v[j < DX ? j : 0] : 0.0f;
  const int full = d - (d & 7);
#pragma unroll
  for (int i = 8; i + 8 <= DX; i += 8)
    if (i < full) {
#pragma unroll
      for (int j = 0; j < 8; ++j) r[j] = __fadd_rn(r[j], v[i + j]);
    }
  float res = __fadd_rn(__fadd_rn(__fadd_rn(r[0], r[1]), __fadd_rn(r[2], r[3])),
                        __fadd_rn(__fadd_rn(r[4], r[5]), __fadd_rn(r[6], r[7])));
#pragma unroll
  for (int i = 0; i < DX; ++i)
    if (i >= full && i < d) res = __fadd_rn(res, v[i]);
  return __fadd_rn(0.0f, res);
}

// Labeling in numpy's float32 arithmetic (KMeans.py:493-522 np_label):
// dist_c = ((x - c) ** 2).sum(axis=1) with a float32 difference, a float32
// square and numpy's row sum (np_row_sum); a centroid replaces the best one
// only when strictly closer (labels[dist < best_dist] = c), so the lowest k
// wins ties. Same grid and LDS staging as k_label_direct.
template <int DX>
__global__ __launch_bounds__(256) void k_label_np(const float* __restrict__ X, int64_t n, int d,
                                                  const float* __restrict__ C,
                                                  const int64_t* __restrict__ k_off, int P,
                                                  int32_t* __restrict__ labels,
                                                  float* __restrict__ dists) {
  constexpr int kTile = 16384 / (DX * 4) > 256 ? 256 : 16384 / (DX * 4);
  __shared__ float s_c[kTile * DX];
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool valid = i < n;
  float xr[DX];
#pragma unroll
  for (int j = 0; j < DX; ++j) xr[j] = (valid && j < d) ? X[i * d + j] : 0.0f;
  for (int p = blockIdx.y; p < P; p += gridDim.y) {
    const int64_t kbeg = k_off[p], kend = k_off[p + 1];
    float best = 0.0f;
    int32_t bl = -1;
    for (int64_t c0 = kbeg; c0 < kend; c0 += kTile) {
      const int rows = (int)((kend - c0) < kTile ? (kend - c0) : kTile);
      __syncthreads();
      for (int v = threadIdx.x; v < rows * DX; v += blockDim.x) {
        const int r = v / DX, j = v - (v / DX) * DX;
        s_c[v] = j < d ? C[(c0 + r) * d + j] : 0.0f;
      }
      __syncthreads();
      if (valid) {
        for (int r = 0; r < rows; ++r) {
          float sq[DX];
#pragma unroll
          for (int j = 0; j < DX; ++j) sq[j] = np_square_diff(xr[j], s_c[r * DX + j]);
          const float dist = np_row_sum<DX>(sq, d);
          if (bl < 0 || dist < best) { best = dist; bl = (int32_t)(c0 + r - kbeg); }
        }
      }
    }
    if (valid) {
      labels[(int64_t)p * n + i] = bl;
      if (dists) dists[(int64_t)p * n + i] = best;
    }
  }
}

int launch_np(const float* X, int64_t n, int d, const float* C, const int64_t* k_off, int P,
              int32_t* labels, float* dists, hipStream_t s) {
  const dim3 g(grid_for(n, 256), P < 65535 ? P : 65535);
  if (d == 1) k_label_np<1><<<g, 256, 0, s>>>(X, n, d, C, k_off, P, labels, dists);
  else if (d == 2) k_label_np<2><<<g, 256, 0, s>>>(X, n, d, C, k_off, P, labels, dists);
  else if (d <= 4) k_label_np<4><<<g, 256, 0, s>>>(X, n, d, C, k_off, P, labels, dists);
  else if (d <= 8) k_label_np<8><<<g, 256, 0, s>>>(X, n, d, C, k_off, P, labels, dists);
  else if (d <= 16) k_label_np<16><<<g, 256, 0, s>>>(X, n, d, C, k_off, P, labels, dists);
  else if (d <= 32) k_label_np<32><<<g, 256, 0, s>>>(X, n, d, C, k_off, P, labels, dists);
  else if (d <= 64) k_label_np<64><<<g, 256, 0, s>>>(X, n, d, C, k_off, P, labels, dists);
  else if (d <= 128) k_label_np<128><<<g, 256, 0, s>>>(X, n, d, C, k_off, P, labels, dists);
  else return fail(EAC_ERR_UNSUPPORTED, "kmeans numpy arithmetic: d=%d > 128", d);
  EAC_LAUNCH_CHECK();
  return EAC_OK;
}

// numpy's float32 sum of each partition's dists: the inertia of
// KMeans.py:164 (new_inertia = self._dists.sum()). numpy's add reduction
// starts from 0 and visits the array in chunks of its buffer size (8192
// elements), adding each chunk's pairwise sum in order
// (numpy/_core/src/umath/loops_utils.h.src @TYPE@_pairwise_sum,
// PW_BLOCKSIZE 128): a range of len < 8 is summed sequentially from 0; len
// <= 128 keeps eight partial sums over a[j], a[j+8], ... combined as
// ((r0+r1)+(r2+r3))+((r4+r5)+(r6+r7)), then adds the tail in order; longer
// ranges split at n2 = len/2 rounded down to a multiple of 8. Every addition
// is a float32 addition, so the result is numpy's to the bit.
//
// The tree of a chunk is a pure function of its length. The shorter half n2
// grows with len, so the leftmost node of a depth is its shortest, and T, the
// first depth at which that one is a leaf (len <= 128), has all its 2^T <= 64
// nodes. Halves differ by at most 15, so the lengths of a depth by less than
// 30, and a node of depth T that is no leaf (len < 158) has two leaves: depth
// T is computed node by node and the rest is a full binary tree.
constexpr int kNpBuf = 8192;

// A leaf's sum by eight lanes (lane j holds the partial sum over a[j],
// a[j+8], ...), all of a lane's loads in flight at once; the result is that of
// lane 0, whose additions take their operands in numpy's order.
__device__ __forceinline__ float np_leaf(const float* __restrict__ a, int len, int j) {
  float res = 0.0f;
  if (len >= 8) {
    constexpr int Q = 128 / 8;
    const int m = len >> 3;
    float e[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) e[q] = q < m ? a[8 * q + j] : 0.0f;
    res = e[0];
#pragma unroll
    for (int q = 1; q < Q; ++q)
      if (q < m) res = __fadd_rn(res, e[q]);
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) res = __fadd_rn(res, __shfl_xor(res, o));
  }
  for (int i = len & ~7; i < len; ++i) res = __fadd_rn(res, a[i]);
  return res;
}

// One workgroup per (chunk, row): csum[row * nchunks + chunk]. Eight lanes a
// node of depth T, so that a full chunk is read at once, 32 bytes a node, and
// its sum waits for one round trip to memory; the 2^T sums are one
// wavefront's. 100 rows of 10,000: 4.5 us (a lane a leaf and a walk of the
// tree in LDS: 9.8).
constexpr int kNpT = 512;
__global__ __launch_bounds__(kNpT) void k_np_chunk_sums(const float* __restrict__ x, int64_t n,
                                                        int64_t nchunks,
                                                        float* __restrict__ csum) {
  __shared__ float v[kWave];
  const int64_t c = blockIdx.x;
  const int64_t row = blockIdx.y;
  const int64_t base = c * kNpBuf;
  const int len0 = (int)(n - base < kNpBuf ? n - base : kNpBuf);
  const float* a = x + row * n + base;
  int T = 0;
  for (int l = len0; l > 128; l = (l >> 1) & ~7) ++T;
  const int g = threadIdx.x >> 3, j = threadIdx.x & 7;
  if (g < 1 << T) {
    int len = len0;
    for (int q = T - 1; q >= 0; --q) {
      const int n2 = (len >> 1) & ~7;
      if ((g >> q) & 1) {
        a += n2;
        len -= n2;
      } else {
        len = n2;
      }
    }
    const int n2 = len > 128 ? (len >> 1) & ~7 : len;
    float r = np_leaf(a, n2, j);
    if (len > n2) r = __fadd_rn(r, np_leaf(a + n2, len - n2, j));
    if (j == 0) v[g] = r;
  }
  __syncthreads();
  if (threadIdx.x < kWave) {
    float r = (int)threadIdx.x < 1 << T ? v[threadIdx.x] : 0.0f;
    for (int o = 1; o < 1 << T; o <<= 1) r = __fadd_rn(r, __shfl_xor(r, o));
    if (threadIdx.x == 0) csum[row * nchunks + c] = r;
  }
}

// ((0 + csum[0]) + csum[1]) + ...
__device__ __forceinline__ float np_finish(const float* __restrict__ csum, int64_t nchunks) {
  float r = 0.0f;
  for (int64_t c = 0; c < nchunks; ++c) r = __fadd_rn(r, csum[c]);
  return r;
}
__global__ void k_np_finish(const float* __restrict__ csum, int64_t nchunks, int64_t rows,
                            float* __restrict__ out) {
  const int64_t row = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (row >= rows) return;
  out[row] = np_finish(csum + row * nchunks, nchunks);
}

int64_t np_chunks(int64_t n) { return n > 0 ? (n + kNpBuf - 1) / kNpBuf : 0; }

// chunk sums of `rows` rows of length n: csum holds rows * np_chunks(n)
int np_chunk_sums(const float* x, int64_t n, int64_t rows, float* csum, hipStream_t s) {
  const int64_t nc = np_chunks(n);
  if (nc > 0) {
    for (int64_t r0 = 0; r0 < rows; r0 += 65535) {
      const int64_t rr = rows - r0 < 65535 ? rows - r0 : 65535;
      k_np_chunk_sums<<<dim3((unsigned)nc, (unsigned)rr), kNpT, 0, s>>>(x + r0 * n, n, nc,
                                                                          csum + r0 * nc);
      EAC_LAUNCH_CHECK();
    }
  }
  return EAC_OK;
}

// numpy float32 sums of `rows` rows of length n; csum holds rows * np_chunks(n)
int np_sum_rows(const float* x, int64_t n, int64_t rows, float* csum, float* out,
                hipStream_t s) {
  EAC_TRY(np_chunk_sums(x, n, rows, csum, s));
  k_np_finish<<<grid_for(rows, 256), 256, 0, s>>>(csum, np_chunks(n), rows, out);
  EAC_LAUNCH_CHECK();
  return EAC_OK;
}

template <typename T>
int launch_direct(const float* X, int64_t n, int d, const float* C, const int64_t* k_off, int P,
                  int32_t* labels, float* dists, hipStream_t s) {
  const int py = P < 65535 ? P : 65535;
  const dim3 g(grid_for(n, 256), py);
  // two points a lane while that still leaves every unit two workgroups
  if (d <= 4 && (int64_t)grid_for(n, 512) * py >= 512) {
    const dim3 g2(grid_for(n, 512), py);
    if (d == 1) k_label_direct<T, 1, 2><<<g2, 256, 0, s>>>(X, n, d, C, k_off, P, labels, dists);
    else if (d == 2) k_label_direct<T, 2, 2><<<g2, 256, 0, s>>>(X, n, d, C, k_off, P, labels, dists);
    else if (d == 3) k_label_direct<T, 3, 2><<<g2, 256, 0, s>>>(X, n, d, C, k_off, P, labels, dists);
    else k_label_direct<T, 4, 2><<<g2, 256, 0, s>>>(X, n, d, C, k_off, P, labels, dists);
    EAC_LAUNCH_CHECK();
    return EAC_OK;
  }
  if (d == 1) k_label_direct<T, 1, 1><<<g, 256, 0, s>>>(X, n, d, C, k_off, P, labels, dists);
  else if (d == 2) k_label_direct<T, 2, 1><<<g, 256, 0, s>>>(X, n, d, C, k_off, P, labels, dists);
  else if (d == 3) k_label_direct<T, 3, 1><<<g, 256, 0, s>>>(X, n, d, C, k_off, P, labels, dists);
  else if (d == 4) k_label_direct<T, 4, 1><<<g, 256, 0, s>>>(X, n, d, C, k_off, P, labels, dists);
  else if (d <= 8) k_label_direct<T, 8, 1><<<g, 256, 0, s>>>(X, n, d, C, k_off, P, labels, dists);
  else if (d <= 16) k_label_direct<T, 16, 1><<<g, 256, 0, s>>>(X, n, d, C, k_off, P, labels, dists);
  else if (d <= 32) k_label_direct<T, 32, 1><<<g, 256, 0, s>>>(X, n, d, C, k_off, P, labels, dists);
  else if (d <= 64) k_label_direct<T, 64, 1><<<g, 256, 0, s>>>(X, n, d, C, k_off, P, labels, dists);
  else if (d <= 128) k_label_direct<T, 128, 1><<<g, 256, 0, s>>>(X, n, d, C, k_off, P, labels, dists);
  else return fail(EAC_ERR_UNSUPPORTED, "kmeans direct: d=%d > 128", d);
  EAC_LAUNCH_CHECK();
  return EAC_OK;
}

// ------------------------------------------------------- centroid update
// new[c][j] = fp32 sequential sum over members in point order, / count in
// double (KMeans.py:736-745). One workgroup per centroid and group of up to
// 128 dimensions (grid.y over partitions). The members' rows are gathered by
// all lanes, a stage of rows ahead in registers, and stored transposed in
// LDS; lane j then adds dimension j's values in member order, four rows per
// LDS read. The additions of one sum cannot be split (their order is part of
// the result), so the longest cluster bounds the launch: LDS reads and adds
// for it instead of a dependent gather per 16 members (500,000 x 16-d points,
// 16 partitions of 32 to 2048 clusters: 612 -> 213 us). Small clusters take
// one wavefront (BS = 64), so more of them are in flight (10,000 x 2-d, 100
// partitions: 28 -> 15 us).
// upd (nullable): partitions whose centroids stay. eflag (nullable): 1 for an
// empty cluster; n_empty counts them.
// V4: rows are read 16 bytes at a time (d a multiple of 4, X 16-byte aligned).
constexpr int kSumDims = 2 * kWave;
template <int BS>
struct SumStage {
  static constexpr int kFloats = BS == kWave ? 1024 : 8192;
  static constexpr int kRows = BS == kWave ? 256 : 1024;
};
template <int BS, bool V4>
__global__ __launch_bounds__(BS) void k_centroid_sums(
    const float* __restrict__ X, int d, const uint32_t* __restrict__ members,
    const uint32_t* __restrict__ start, const int64_t* __restrict__ k_off, int P,
    const int32_t* __restrict__ upd, int32_t* __restrict__ eflag, int32_t* __restrict__ n_empty,
    float* __restrict__ Cout) {
  constexpr int kFloats = SumStage<BS>::kFloats, kRows = SumStage<BS>::kRows;
  constexpr int W = V4 ? 4 : 1;
  constexpr int NV = kFloats / W / BS;  // row pieces a lane holds
  constexpr int NM = kRows / BS;        // member ids a lane holds
  __shared__ __align__(16) float s_x[kFloats + 4 * kSumDims];
  __shared__ uint32_t s_m[kRows];
  const int t = threadIdx.x;
  for (int p = blockIdx.y; p < P; p += gridDim.y) {
    const int64_t kb = k_off[p], ke = k_off[p + 1];
    const bool run = !upd || upd[p];
    for (int64_t c = kb + blockIdx.x; c < ke; c += gridDim.x) {
      const uint32_t m0 = start[c];
      const uint32_t cnt = start[c + 1] - m0;
      if (t == 0) {
        if (eflag) eflag[c] = cnt == 0;
        if (cnt == 0) atomicAdd(n_empty, 1);
      }
      if (cnt == 0 || !run) continue;  // uniform over the block
      const uint32_t* m = members + m0;
      for (int j0 = 0; j0 < d; j0 += kSumDims) {
        const int dd = d - j0 < kSumDims ? d - j0 : kSumDims;
        const int pw = dd / W;  // pieces per row
        int rs = (kFloats / dd) & ~3;
        if (rs > kRows) rs = kRows;
        // column stride: 16-byte aligned, neighbouring columns on other banks (a
        // multiple of 32 would have them all on one)
        if (((rs + 4) & 31) == 0) rs -= 4;
        const int rsp = rs + 4;
        const int dr = BS / pw, dp = BS - dr * pw;  // a step of BS pieces: rows, pieces
        uint32_t mi[NM];
        float4 xv[V4 ? NV : 1];
        float xs[V4 ? 1 : NV];
        auto ids = [&](uint32_t b) {  // member ids of the stage at b
#pragma unroll
          for (int i = 0; i < NM; ++i) {
            const uint32_t r = b + i * BS + t;
            mi[i] = r < cnt ? m[r] : 0u;
          }
        };
        auto keep_ids = [&]() {
#pragma unroll
          for (int i = 0; i < NM; ++i) s_m[i * BS + t] = mi[i];
        };
        // q rows named by s_m, into registers, and from there into LDS. A stage
        // that fills the registers takes no branch (the pieces past its end are
        // its last row's again), so that all its ids are read and all its loads
        // sent before the first wait: 100,000 points in one cluster, 37-d 4.5 ms
        // with a branch a piece, now 1.5, 61-d 6.1 and 2.5, 64-d (16 bytes a
        // piece) 3.1 and 1.6.
        auto walk = [&](int q, auto&& piece) {
          int r = t / pw, j = t - (t / pw) * pw;
          auto step = [&](int i) {
            piece(i, r < q ? r : q - 1, j);
            r += dr;
            j += dp;
            if (j >= pw) {
              j -= pw;
              ++r;
            }
          };
          if (q * pw > (NV - 1) * BS) {
#pragma unroll
            for (int i = 0; i < NV; ++i) step(i);
          } else {
#pragma unroll
            for (int i = 0; i < NV; ++i)
              if (i * BS < q * pw) step(i);  // uniform
          }
        };
        auto rows = [&](int q) {
          walk(q, [&](int i, int r, int j) {
            const float* src = X + (int64_t)s_m[r] * d + j0 + j * W;
            if constexpr (V4) xv[i] = *reinterpret_cast<const float4*>(src);
            else xs[i] = *src;
          });
        };
        auto keep_rows = [&](int q) {
          walk(q, [&](int i, int r, int j) {
            if constexpr (V4) {
              float* col = s_x + (j * 4) * rsp + r;
              col[0] = xv[i].x;
              col[rsp] = xv[i].y;
              col[2 * rsp] = xv[i].z;
              col[3 * rsp] = xv[i].w;
            } else {
              s_x[j * rsp + r] = xs[i];
            }
          });
        };
        auto take = [&](uint32_t b) {
          return (int)(cnt - b < (uint32_t)rs ? cnt - b : (uint32_t)rs);
        };
        float s0 = 0.f;
        int q = take(0);
        __syncthreads();  // the previous centroid's sums are done
        ids(0);
        keep_ids();
        __syncthreads();
        rows(q);
        if (cnt > (uint32_t)rs) ids(rs);
        for (uint32_t b = 0; b < cnt; b += rs) {
          q = take(b);
          keep_rows(q);
          const bool more = b + rs < cnt;
          if (more) {
            __syncthreads();  // this stage's ids are consumed
            keep_ids();
          }
          __syncthreads();  // the stage's rows and the next one's ids are in LDS
          if (more) {
            rows(take(b + rs));
            if (b + 2 * rs < cnt) ids(b + 2 * rs);
          }
          if (t < dd) {
            const float* col = s_x + t * rsp;
            int r = 0;
            for (; r + 16 <= q; r += 16) {
              float4 v[4];
#pragma unroll
              for (int u = 0; u < 4; ++u) v[u] = *reinterpret_cast<const float4*>(col + r + 4 * u);
#pragma unroll
              for (int u = 0; u < 4; ++u) {
                s0 = s0 + v[u].x;
                s0 = s0 + v[u].y;
                s0 = s0 + v[u].z;
                s0 = s0 + v[u].w;
              }
            }
            for (; r < q; ++r) s0 = s0 + col[r];
          }
          if (more) __syncthreads();  // the stage's rows are summed
        }
        if (t < dd) Cout[c * d + j0 + t] = (float)((double)s0 / (double)cnt);
      }
    }
  }
}

// KMeans.py:117-189 stopping rule of iteration `it` for every partition
// still running: new_inertia = numpy float32 sum of the dists (the chunk sums
// csum[p] added up in order),
// err = |new_inertia - previous| in float32 (previous starts at +inf); stop
// when err <= tol (compared in float32, as numpy compares a float32 scalar
// with a Python float) or it >= max_iter, else mark the partition for a
// centroid update. any[0] = some partition continues; any[1] (the update's
// count of empty clusters) is cleared.
__global__ void k_converge(const float* __restrict__ csum, int64_t nchunks,
                           float* __restrict__ prev, int32_t* __restrict__ active, int32_t* __restrict__ iters,
                           int32_t* __restrict__ upd, int P, int it, int max_iter, float tol,
                           int32_t* __restrict__ any) {
  __shared__ int s_any;
  if (threadIdx.x == 0) s_any = 0;
  __syncthreads();
  for (int p = threadIdx.x; p < P; p += blockDim.x) {
    upd[p] = 0;
    if (!active[p]) continue;
    iters[p] = it;
    const float inertia = np_finish(csum + p * nchunks, nchunks);
    const float err = fabsf(__fsub_rn(inertia, prev[p]));
    prev[p] = inertia;
    if (err <= tol || it >= max_iter) {
      active[p] = 0;
      continue;
    }
    upd[p] = 1;
    s_any = 1;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    any[0] = s_any;
    any[1] = 0;
  }
}

__global__ void k_fit_init(float* __restrict__ prev, int32_t* __restrict__ active,
                           int32_t* __restrict__ iters, int P) {
  for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < P; p += gridDim.x * blockDim.x) {
    prev[p] = INFINITY;
    active[p] = 1;
    iters[p] = 0;
  }
}

// keys (dist bits << 32 | index) of one partition: ascending = (dist, index)
__global__ void k_dist_keys(const float* __restrict__ dists, int64_t n,
                            uint64_t* __restrict__ keys) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    keys[i] = ((uint64_t)__float_as_uint(dists[i]) << 32) | (uint64_t)i;
}

// empty clusters c of one partition (ascending) take the points of the
// smallest (dist, index), in that order
__global__ void k_reseed(const float* __restrict__ X, int d, const uint64_t* __restrict__ sorted,
                         const int32_t* __restrict__ eflag, const int32_t* __restrict__ erank,
                         int64_t kbeg, int64_t kend, const int32_t* __restrict__ upd,
                         float* __restrict__ Cnew) {
  if (upd && !*upd) return;  // a stopped partition keeps its centroids
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < (kend - kbeg) * d;
       t += (int64_t)gridDim.x * blockDim.x) {
    int64_t c = kbeg + t / d;
    int j = (int)(t % d);
    if (!eflag[c]) continue;
    int32_t r = erank[c] - erank[kbeg];
    uint32_t src = (uint32_t)(sorted[r] & 0xffffffffu);
    Cnew[c * d + j] = X[(int64_t)src * d + j];
  }
}

// ----------------------------------------- capturable fit (no host reads)
// Total of the flag regions (clamped to the list), error bit 1 when a
// region or the list overflowed. One wavefront.
__global__ void k_flags_total(const unsigned long long* __restrict__ cnt, int64_t region,
                              int64_t cap, int64_t* __restrict__ d_nf,
                              unsigned int* __restrict__ err) {
  const int l = lane_id();
  const unsigned long long c = l < kFlagSlots ? cnt[l] : 0ull;
  const bool over = (int64_t)c > region;
  unsigned long long tot = c;
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) tot += __shfl_xor(tot, off, kWave);
  const bool any_over = __ballot(over) != 0ull;
  if (l == 0) {
    if (any_over || (int64_t)tot > cap) atomicOr(err, 1u);
    d_nf[0] = (int64_t)tot < cap ? (int64_t)tot : cap;
  }
}

// Counting sort of the flags by partition (flag = partition << 40 | row),
// stable-free but deterministic: kSortBlocks workgroups each take the same
// grid-stride share of the flags in both passes; pass 1 counts its share's
// flags per partition in LDS (bcount[p][b]); a scan of bcount in (partition,
// workgroup) order gives offsets; pass 2 places the share's flags
// from LDS cursors started at those offsets. No global atomics (their
// serialisation on a few hot partitions dominated).
constexpr int kSortBlocks = 256;
constexpr int kSortMaxP = 4096;  // partitions counted in LDS
__global__ __launch_bounds__(256) void k_flag_bcount(const uint64_t* __restrict__ flags,
                                                     int64_t nf, const int64_t* __restrict__ d_nf,
                                                     int P, int32_t* __restrict__ bcount) {
  __shared__ int32_t h[kSortMaxP];
  for (int p = threadIdx.x; p < P; p += blockDim.x) h[p] = 0;
  __syncthreads();
  if (d_nf) nf = *d_nf;
  for (int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; f < nf;
       f += (int64_t)gridDim.x * blockDim.x) {
    const int p = (int)(flags[f] >> 40);
    if (p < P) atomicAdd(&h[p], 1);
  }
  __syncthreads();
  for (int p = threadIdx.x; p < P; p += blockDim.x) bcount[(int64_t)p * gridDim.x + blockIdx.x] = h[p];
}
__global__ __launch_bounds__(256) void k_flag_bscatter(const uint64_t* __restrict__ flags,
                                                       int64_t nf,
                                                       const int64_t* __restrict__ d_nf, int P,
                                                       const int32_t* __restrict__ boff,
                                                       uint64_t* __restrict__ out) {
  __shared__ int32_t cur[kSortMaxP];
  for (int p = threadIdx.x; p < P; p += blockDim.x)
    cur[p] = boff[(int64_t)p * gridDim.x + blockIdx.x];
  __syncthreads();
  if (d_nf) nf = *d_nf;
  for (int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; f < nf;
       f += (int64_t)gridDim.x * blockDim.x) {
    const uint64_t fl = flags[f];
    const int p = (int)(fl >> 40);
    if (p < P) out[atomicAdd(&cur[p], 1)] = fl;
  }
}

// Device reseeding of every partition's empty clusters (the same rule as
// k_dist_keys + radix sort + k_reseed): the r-th empty cluster of partition
// p (ascending) takes the point of the r-th smallest key (dist bits << 32 |
// index). One workgroup per partition with empties: the e-th smallest key by
// a radix select (eight 8-bit digit passes over the partition's dists), the
// e keys at or below it collected in LDS and ranked among themselves. More
// than kMaxReseed empties in one partition set error bit 2.
constexpr int kMaxReseed = 2048;
__global__ __launch_bounds__(1024) void k_reseed_dev(
    const float* __restrict__ X, int d, const float* __restrict__ dists, int64_t n,
    const int64_t* __restrict__ k_off, int P, const int32_t* __restrict__ eflag,
    const int32_t* __restrict__ erank, const int32_t* __restrict__ upd,
    float* __restrict__ Cnew, unsigned int* __restrict__ err) {
  __shared__ unsigned int hist[256];
  __shared__ unsigned long long s_sel[kMaxReseed];
  __shared__ int32_t s_emp[kMaxReseed];
  __shared__ unsigned long long s_prefix;
  __shared__ int64_t s_want;
  __shared__ int s_nsel;
  const int t = threadIdx.x;
  for (int p = blockIdx.x; p < P; p += gridDim.x) {
    const int64_t kb = k_off[p], ke = k_off[p + 1];
    const int64_t e = (int64_t)erank[ke] - erank[kb];
    if (e == 0 || (upd && !upd[p])) continue;  // uniform over the block
    if (e > n || e > kMaxReseed) {
      if (t == 0) atomicOr(err, 2u);
      continue;
    }
    const float* dp = dists + (int64_t)p * n;
    if (t == 0) {
      s_prefix = 0ull;
      s_want = e;  // rank (1-based) of the wanted key among those left
    }
    for (int shift = 56; shift >= 0; shift -= 8) {
      for (int b = t; b < 256; b += blockDim.x) hist[b] = 0u;
      __syncthreads();
      const unsigned long long pre = s_prefix;
      for (int64_t i = t; i < n; i += blockDim.x) {
        const unsigned long long key =
            ((unsigned long long)__float_as_uint(dp[i]) << 32) | (unsigned long long)i;
        if (shift == 56 || ((key ^ pre) >> (shift + 8)) == 0ull)
          atomicAdd(&hist[(key >> shift) & 255u], 1u);
      }
      __syncthreads();
      if (t == 0) {
        int64_t want = s_want, cum = 0;
        int b = 0;
        for (; b < 255 && cum + (int64_t)hist[b] < want; ++b) cum += hist[b];
        s_want = want - cum;
        s_prefix = pre | ((unsigned long long)b << shift);
      }
      __syncthreads();
    }
    const unsigned long long T = s_prefix;  // the e-th smallest key (keys are unique)
    if (t == 0) s_nsel = 0;
    for (int64_t c = kb + t; c < ke; c += blockDim.x)
      if (eflag[c]) s_emp[erank[c] - erank[kb]] = (int32_t)c;
    __syncthreads();
    for (int64_t i = t; i < n; i += blockDim.x) {
      const unsigned long long key =
          ((unsigned long long)__float_as_uint(dp[i]) << 32) | (unsigned long long)i;
      if (key <= T) {
        const int at = atomicAdd(&s_nsel, 1);
        if (at < kMaxReseed) s_sel[at] = key;
      }
    }
    __syncthreads();
    const int ns = s_nsel < (int)e ? s_nsel : (int)e;
    for (int j = t; j < ns; j += blockDim.x) {
      const unsigned long long key = s_sel[j];
      int r = 0;
      for (int q = 0; q < ns; ++q) r += s_sel[q] < key;
      const int64_t c = s_emp[r];
      const int64_t pt = (int64_t)(key & 0xffffffffull);
      for (int jj = 0; jj < d; ++jj) Cnew[c * d + jj] = X[pt * d + jj];
    }
    __syncthreads();
  }
}

// Running totals of a capturable fit: info[0] += flags re-scored,
// info[1] += empty clusters reseeded (device; one thread), counted only
// while some partition still runs (any[0], the last stopping-rule result),
// as the fit that stops when none does counts them.
__global__ void k_fit_tally(int64_t* __restrict__ info, const int64_t* __restrict__ d_nf,
                            const int32_t* __restrict__ erank, int64_t ktot,
                            const int32_t* __restrict__ any) {
  if (threadIdx.x == 0 && blockIdx.x == 0 && any[0]) {
    if (d_nf) info[0] += *d_nf;
    if (erank) info[1] += erank[ktot];
  }
}

int d2h(void* host, const void* dev, size_t bytes, hipStream_t s) {
  void* pin = pinned_scratch(bytes);
  if (!pin) return fail(EAC_ERR_HIP, "pinned host allocation failed");
  EAC_HIP_CHECK(hipMemcpyAsync(pin, dev, bytes, hipMemcpyDeviceToHost, s));
  EAC_HIP_CHECK(hipStreamSynchronize(s));
  memcpy(host, pin, bytes);
  return EAC_OK;
}

struct LabelBufs {
  int64_t* k_off;
  uint16_t* Cf;  // split rows of the centroids
  float* Ct;  // centroids transposed: [d][ktot]
  float* ncf;
  unsigned int* pstat;        // [P][kStat]; cleared with nflag, which follows it
  uint64_t* flags_r;  // kFlagSlots regions of `region` flags
  uint64_t* flags;    // the flags of all regions, contiguous
  unsigned long long* nflag;  // per-region counts
  int32_t* bcount;            // [P][kSortBlocks] flags per (partition, sorting workgroup)
  float* csum;                // numpy-order chunk sums of the dists
  int64_t flag_cap;
  int64_t region;
};

LabelBufs carve_label(Arena& ar, int64_t n, int d, int64_t ktot, int P) {
  LabelBufs b;
  const int NF = std::max(label_layout(d).NF, label_layout(d, true).NF);
  b.k_off = ar.take<int64_t>(P + 1);
  b.Cf = ar.take<uint16_t>((size_t)ktot * NF * 32 + 64);
  b.Ct = ar.take<float>((size_t)ktot * d);
  b.ncf = ar.take<float>(ktot);
  b.nflag = ar.take<unsigned long long>(kFlagSlots + ((size_t)P * kStat + 1) / 2);
  b.pstat = reinterpret_cast<unsigned int*>(b.nflag + kFlagSlots);
  b.flag_cap = (int64_t)P * n;
  // a region holds every (partition, row) its blocks can flag
  const int64_t nblocks = (n + kLB - 1) / kLB;
  b.region = ((nblocks + kFlagSlots - 1) / kFlagSlots) * kLB * (int64_t)P;
  b.flags_r = ar.take<uint64_t>((size_t)kFlagSlots * b.region);
  b.flags = ar.take<uint64_t>(b.flag_cap);
  b.bcount = ar.take<int32_t>((size_t)std::min(P, kSortMaxP) * kSortBlocks);
  b.csum = ar.take<float>((size_t)P * np_chunks(n) + 1);
  return b;
}

}  // namespace

size_t kmeans_label_ws_bytes(int64_t n, int d, int64_t ktot, int P) {
  Arena ar(nullptr, 0, true);
  (void)carve_label(ar, n, d, ktot, P);
  return ar.used + scan_ws_bytes((int64_t)std::min(P, kSortMaxP) * kSortBlocks, 4) + 4096;
}

// Device-side state of a capturable fit: flag count, running totals (info[0]
// flags re-scored, info[1] clusters reseeded), error bits.
struct KmGraph {
  const int32_t* any;  // some partition still runs (the labeling counts only then)
  int64_t* d_nf;
  int64_t* info;
  unsigned int* err;
};

// The labeling kernel for a layout: point blocks per wave (four where the
// point fragments leave the registers for it, two for wide rows and for
// inputs of too few points to fill the chip otherwise) and waves per SIMD
// (EAC_TUNE_KM_WAVES, or the built-in choice, for the layouts of d = 11 ... 21 and
// d = 54 ... 64).
struct LabelCall {
  const float* X;
  int64_t row0, n;  // rows [row0, n), or entries of `list`
  int d;
  const float* C;
  const uint16_t* Cf;
  const float* ncf;
  const int64_t* k_off;
  int P;
  const unsigned int* pstat;
  const uint64_t* list;
  int32_t* labels;
  float* dists;
  uint64_t* flags;
  unsigned long long* nflag;
  int64_t region;
};
template <int KS, bool SPLIT, int MB, int WPE, int TERMS = 3, bool FUSE = false,
          bool LIST = false>
void label_go(const LabelCall& a, hipStream_t s) {
  const int64_t gx = (a.n - a.row0 + 64 * MB - 1) / (64 * MB);
  int64_t gy = FUSE || gx >= 1536 ? 1 : (1536 + gx - 1) / gx;
  if (gy > a.P) gy = a.P;
  if (gy > 65535) gy = 65535;
  k_label_f16x3<KS, SPLIT, MB, WPE, TERMS, FUSE, LIST>
      <<<dim3((unsigned)gx, (unsigned)gy), kLB, 0, s>>>(a.X, a.row0, a.n, a.d, a.C, a.Cf, a.ncf,
                                                        a.k_off, a.P, a.pstat, a.list, a.labels,
                                                        a.dists, a.flags, a.nflag, a.region);
}
template <int KS, bool SPLIT, bool FUSE>
void label_sized(const LabelCall& a, bool wide, hipStream_t s) {
  if constexpr (KS == 2 || (KS == 6 && SPLIT)) {
    switch (tune_value(EAC_TUNE_KM_WAVES)) {
      case 2: return wide ? label_go<KS, SPLIT, 4, 2, 3, FUSE>(a, s)
                          : label_go<KS, SPLIT, 2, 2, 3, FUSE>(a, s);
      case 3: return wide ? label_go<KS, SPLIT, 4, 3, 3, FUSE>(a, s)
                          : label_go<KS, SPLIT, 2, 3, 3, FUSE>(a, s);
      case 4: return wide ? label_go<KS, SPLIT, 4, 4, 3, FUSE>(a, s)
                          : label_go<KS, SPLIT, 2, 4, 3, FUSE>(a, s);
    }
  }
  constexpr int W = KS <= 3 ? 4 : 3;
  return wide ? label_go<KS, SPLIT, 4, W, 3, FUSE>(a, s)
              : label_go<KS, SPLIT, 2, W, 3, FUSE>(a, s);
}
template <bool FUSE>
int launch_label(const LabelLayout& L, const LabelCall& a, hipStream_t s) {
  const bool wide = (a.n - a.row0) * a.P >= 256 * 1536;
  if (L.split) {
    switch (L.KS) {
      case 3: label_sized<3, true, FUSE>(a, wide, s); break;
      case 6: label_sized<6, true, FUSE>(a, wide, s); break;
      case 9: label_go<9, true, 2, 2, 3, FUSE>(a, s); break;
      default: label_go<12, true, 2, 2, 3, FUSE>(a, s); break;
    }
  } else {
    switch (L.KS) {
      case 1: label_sized<1, false, FUSE>(a, wide, s); break;
      case 2: label_sized<2, false, FUSE>(a, wide, s); break;
      case 4: label_sized<4, false, FUSE>(a, wide, s); break;
      case 5: label_sized<5, false, FUSE>(a, wide, s); break;
      case 7: label_go<7, false, 2, 2, 3, FUSE>(a, s); break;
      default: label_go<8, false, 2, 2, 3, FUSE>(a, s); break;
    }
  }
  EAC_LAUNCH_CHECK();
  return EAC_OK;
}
// The cascade's passes (split layouts of two to four fragments, one
// partition): the single product over rows, and all three over a list.
int launch_single(const LabelLayout& L, const LabelCall& a, hipStream_t s) {
  switch (L.KS) {
    case 6: label_go<2, true, 4, 4, 1, true>(a, s); break;
    case 9: label_go<3, true, 4, 3, 1, true>(a, s); break;
    default: label_go<4, true, 4, 3, 1, true>(a, s); break;
  }
  EAC_LAUNCH_CHECK();
  return EAC_OK;
}
int launch_listed(const LabelLayout& L, const LabelCall& a, hipStream_t s) {
  switch (L.KS) {
    case 6: label_go<6, true, 2, 3, 3, true, true>(a, s); break;
    case 9: label_go<9, true, 2, 2, 3, true, true>(a, s); break;
    default: label_go<12, true, 2, 2, 3, true, true>(a, s); break;
  }
  EAC_LAUNCH_CHECK();
  return EAC_OK;
}

// Flags in all regions (read back).
int read_flags(const LabelBufs& B, unsigned long long* nf, hipStream_t s) {
  unsigned long long hcnt[kFlagSlots];
  EAC_TRY(d2h(hcnt, B.nflag, sizeof(hcnt), s));
  *nf = 0;
  for (int q = 0; q < kFlagSlots; ++q) {
    if ((int64_t)hcnt[q] > B.region) return fail(EAC_ERR_HIP, "kmeans: flag list overflow");
    *nf += hcnt[q];
  }
  if ((int64_t)*nf > B.flag_cap) return fail(EAC_ERR_HIP, "kmeans: flag list overflow");
  return EAC_OK;
}
// The gathered flags (their number on the host, or at d_nf) sorted by
// partition into the regions, which the gathering has emptied.
int sort_flags(const LabelBufs& B, int P, int64_t nf, const int64_t* d_nf, Arena& ar,
               hipStream_t s) {
  k_flag_bcount<<<kSortBlocks, 256, 0, s>>>(B.flags, nf, d_nf, P, B.bcount);
  EAC_LAUNCH_CHECK();
  const size_t mark = ar.used;
  EAC_TRY((scan_excl<int32_t, int32_t>(B.bcount, B.bcount, (int64_t)P * kSortBlocks, 0, nullptr,
                                       ar, s)));
  ar.used = mark;
  k_flag_bscatter<<<kSortBlocks, 256, 0, s>>>(B.flags, nf, d_nf, P, B.bcount, B.flags_r);
  EAC_LAUNCH_CHECK();
  return EAC_OK;
}
int gather_flags(const LabelBufs& B, unsigned long long nf, hipStream_t s) {
  k_gather_flags<<<grid_for((int64_t)nf, 256, 65536), 256, 0, s>>>(B.flags_r, B.region, B.nflag,
                                                                   B.flags, (int64_t)nf);
  EAC_LAUNCH_CHECK();
  return EAC_OK;
}

// Whether BF16X3 takes the plain FP64 labeling (the same labels and
// distances). It must where resolve16 does not reach: fewer than four
// dimensions, or a partition beyond its 32-bit offsets (2^23 rows of up to 512
// bytes). From 16 dimensions on it never does (it pays only for toy sizes
// there). In between the cheaper one, from measured times: a thread of the
// direct kernel walks its partition's centroids in sequence (c1 us each,
// whatever n is; 40 us a call with no centroid to speak of), a full chip does
// a (point, centroid) pair in c2 us; the MFMA path costs 28 us more a call
// (60 with several partitions: sorted flags, a separate resolving) and about
// 0.075e-6 us a pair and MFMA step. E.g. d = 8: 30,000 points, k = 100: 51 us
// direct, 68 MFMA; k = 500: 101 and 73; 300,000 points, k = 2000: 631 and 149.
bool direct_f64(int64_t n, int d, const int64_t* h_koff, int P) {
  if (d < 4) return true;
  int64_t kmax = 1;
  for (int p = 0; p < P; ++p) kmax = std::max(kmax, h_koff[p + 1] - h_koff[p]);
  if (kmax >= (int64_t)1 << 23) return true;
  if (d >= 16) return false;
  const int dx = d <= 4 ? 0 : d <= 8 ? 1 : 2;
  const double c1[] = {0.083, 0.125, 0.29}, c2[] = {0.59e-6, 0.99e-6, 1.9e-6};
  const double pairs = (double)n * (double)h_koff[P];
  const double direct = std::max((double)kmax * c1[dx], pairs * c2[dx]);
  return direct <= (P == 1 ? 28.0 : 60.0) + pairs * 0.075e-6 * label_layout(d).KS;
}

// Label all partitions; dists (nullable) receive FP64-exact distances for
// the F64 / BF16X3 modes and fp32 distances for F32; csum_out (nullable)
// the numpy float32 chunk sums of each partition's dists.
// With g (capturable calls) nothing is read back: the flag count stays on
// the device and sizes the re-scoring from there.
int kmeans_label(const float* X, int64_t n, int d, const float* C, const int64_t* h_koff,
                 int P, int mode, int32_t* labels, float* dists, const float** csum_out,
                 int64_t* n_rescored, Arena& ar, hipStream_t s,
                 const int64_t* d_koff = nullptr, const KmGraph* kg = nullptr) {
  const int64_t ktot = h_koff[P];
  LabelBufs B = carve_label(ar, n, d, ktot, P);
  if (ar.overflow()) return fail(EAC_ERR_WORKSPACE, "kmeans: workspace too small");
  if (d_koff) {
    B.k_off = const_cast<int64_t*>(d_koff);  // read only
  } else {
    EAC_TRY(put_i64(B.k_off, h_koff, P + 1, s));
  }
  if (n_rescored) *n_rescored = 0;
  if (mode != EAC_KM_F32 && mode != EAC_KM_F64 && mode != EAC_KM_F32_NUMPY &&
      mode != EAC_KM_BF16X3)
    return fail(EAC_ERR_ARG, "kmeans: unknown mode %d", mode);
  if (mode != EAC_KM_BF16X3 || direct_f64(n, d, h_koff, P)) {
    int pr = prof_begin(EAC_PROF_KM_LABEL, 2 * n * (int64_t)d * ktot, s);
    if (mode == EAC_KM_F32_NUMPY)
      EAC_TRY(launch_np(X, n, d, C, B.k_off, P, labels, dists, s));
    else if (mode == EAC_KM_F32)
      EAC_TRY(launch_direct<float>(X, n, d, C, B.k_off, P, labels, dists, s));
    else
      EAC_TRY(launch_direct<double>(X, n, d, C, B.k_off, P, labels, dists, s));
    prof_end(pr, s);
    if (csum_out) {
      if (!dists) return fail(EAC_ERR_ARG, "kmeans: inertia needs dists");
      EAC_TRY(np_chunk_sums(dists, n, P, B.csum, s));
      *csum_out = B.csum;
    }
    return EAC_OK;
  }
  if (d > 128) return fail(EAC_ERR_UNSUPPORTED, "kmeans bf16x3: d=%d > 128", d);
  if (csum_out && !dists) return fail(EAC_ERR_ARG, "kmeans: inertia needs dists");
  // The cascade pays where the three products take long (its read-backs
  // cost about 40 us) and two thirds of the MFMAs are to be saved: one
  // partition of more than 32 dimensions.
  const bool cascade = !kg && P == 1 && d > 32 && n * ktot * ((d + 31) / 32) >= (int64_t)5e8;
  const LabelLayout L = label_layout(d, cascade);
  EAC_TRY(fill<uint64_t>((uint64_t*)B.nflag, kFlagSlots + ((int64_t)P * kStat + 1) / 2, 0ull, s));
  {
    const int py = P < 65535 ? P : 65535;
    const int gm = grid_for(ktot * d / P, 4096, 64), gp = grid_for(ktot / P, 64, 256);
    k_cent_max<<<dim3(gm, py), 256, 0, s>>>(C, d, B.k_off, P, B.pstat);
    EAC_LAUNCH_CHECK();
    k_cent_prep<<<dim3(gp, py), 256, 0, s>>>(C, ktot, d, L, B.k_off, P, B.Cf, B.Ct, B.ncf,
                                             B.pstat);
    EAC_LAUNCH_CHECK();
  }
  int pr = prof_begin(EAC_PROF_KM_LABEL, 2 * n * (int64_t)d * ktot, s);
  LabelCall call{X,       0,      n,        d,      C,     B.Cf,      B.ncf,   B.k_off,
                 P,       B.pstat, nullptr, labels, dists, B.flags_r, B.nflag, B.region};
  if (cascade) {
    // The single product first, on a sample: when it certifies most points
    // the rest follow it and only the flagged rows take the three products.
    const int64_t ns = n < 65536 ? n : 65536;
    unsigned long long nf1 = 0;
    call.n = ns;
    EAC_TRY(launch_single(L, call, s));
    EAC_TRY(read_flags(B, &nf1, s));
    const bool single = nf1 * 4 <= (unsigned long long)ns;
    call.n = n;
    if (single) {
      call.row0 = ns;
      if (ns < n) {
        EAC_TRY(launch_single(L, call, s));
        EAC_TRY(read_flags(B, &nf1, s));
      }
      if (nf1 > 0) {
        EAC_TRY(gather_flags(B, nf1, s));
        EAC_TRY(fill<uint64_t>((uint64_t*)B.nflag, kFlagSlots, 0ull, s));
        call.row0 = 0;
        call.n = (int64_t)nf1;
        call.list = B.flags;
        EAC_TRY(launch_listed(L, call, s));
      }
    } else {
      EAC_TRY(fill<uint64_t>((uint64_t*)B.nflag, kFlagSlots, 0ull, s));
      EAC_TRY(launch_label<true>(L, call, s));
    }
  } else if (P == 1) {
    EAC_TRY(launch_label<true>(L, call, s));
  } else {
    EAC_TRY(launch_label<false>(L, call, s));
  }
  prof_end(pr, s);
  if (P > 1) {
    const int pgs = (P + kPG - 1) / kPG;
    const dim3 gr(grid_for(n, 256 / kGrp, 16384), pgs < 65535 ? pgs : 65535);
    if ((d & 3) == 0) k_resolve<true><<<gr, 256, 0, s>>>(X, n, d, C, B.k_off, P, labels, dists);
    else k_resolve<false><<<gr, 256, 0, s>>>(X, n, d, C, B.k_off, P, labels, dists);
    EAC_LAUNCH_CHECK();
  }
  if (kg) {
    // flags gathered, sorted by partition and re-scored with device counts
    // (grids sized for the whole list, blocks past the count exit at once)
    k_flags_total<<<1, kWave, 0, s>>>(B.nflag, B.region, B.flag_cap, kg->d_nf, kg->err);
    EAC_LAUNCH_CHECK();
    const int gp = grid_for(B.flag_cap, 256, 4096);
    k_gather_flags<<<gp, 256, 0, s>>>(B.flags_r, B.region, B.nflag, B.flags, 0, kg->d_nf);
    EAC_LAUNCH_CHECK();
    const uint64_t* fl = B.flags;
    const bool tiled = rescore_tiled_lds(d) <= 64 * 1024;
    if (tiled && P > 1 && P <= kSortMaxP) {
      EAC_TRY(sort_flags(B, P, 0, kg->d_nf, ar, s));
      fl = B.flags_r;
    }
    int pr2 = prof_begin(EAC_PROF_KM_RESCORE, 0, s);
    if (tiled) {
      const size_t lds = rescore_tiled_lds(d);
      int dev = 0, cus = 256;
      if (hipGetDevice(&dev) == hipSuccess)
        (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
      // as many workgroups as the eager launch of a few million flags
      // would have; those past the device count exit at once
      const int64_t tiles = (B.flag_cap + kRtF - 1) / kRtF;
      const unsigned nb = (unsigned)(tiles < 64 * (int64_t)cus ? tiles : 64 * (int64_t)cus);
      auto go = [&](auto kern) {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        kern<<<nb, kRtF * kRtS, lds, s>>>(X, n, d, C, B.k_off, fl, 0, labels, dists, kg->d_nf);
      };
      if (d <= 16) go(k_rescore_tiled<16>);
      else if (d <= 32) go(k_rescore_tiled<32>);
      else if (d <= 64) go(k_rescore_tiled<64>);
      else go(k_rescore_tiled<0>);
    } else {
      const int gr = grid_for(B.flag_cap, kRfF, 16384);
      k_rescore_few<kRfF, 256><<<gr, 256, 0, s>>>(X, n, d, C, B.Ct, ktot, B.k_off, B.flags, 0,
                                                  labels, dists, kg->d_nf, nullptr, 0);
    }
    EAC_LAUNCH_CHECK();
    prof_end(pr2, s);
    k_fit_tally<<<1, 64, 0, s>>>(kg->info, kg->d_nf, nullptr, 0, kg->any);
    EAC_LAUNCH_CHECK();
  } else {
  // One partition: the re-scoring of fewer than kFewMax flags needs no sorting and
  // follows without a read-back, straight from the regions.
  if (P == 1) {
    int pr2 = prof_begin(EAC_PROF_KM_RESCORE, 0, s);
    k_rescore_few<kRfF, 256><<<1024, 256, 0, s>>>(X, n, d, C, B.Ct, ktot, B.k_off, B.flags_r, 0,
                                                  labels, dists, nullptr, B.nflag, B.region);
    EAC_LAUNCH_CHECK();
    prof_end(pr2, s);
  }
  unsigned long long nf = 0;
  EAC_TRY(read_flags(B, &nf, s));
  if (nf > 0 && (P > 1 || nf >= (unsigned long long)kFewMax)) {
    EAC_TRY(gather_flags(B, nf, s));
    int pr2 = prof_begin(EAC_PROF_KM_RESCORE, 3 * (int64_t)nf * d * (ktot / P), s);
    // Many flags (at least 1024 blocks of 64) and d <= 127 (LDS tiles up to
    // 64 KiB): the LDS-tiled re-scoring. Few flags: a block per kRfF of them
    // over the transposed centroids (more parallelism per flag). Both want
    // neighbouring flags in one partition: from 4096 flags on they are
    // sorted by partition.
    const uint64_t* fl = B.flags;
    bool tiled = nf >= (unsigned long long)kRtF * 1024 && rescore_tiled_lds(d) <= 64 * 1024;
    bool sorted_flags = P == 1;
    if (P > 1 && P <= kSortMaxP && nf >= 4096) {
      EAC_TRY(sort_flags(B, P, (int64_t)nf, nullptr, ar, s));
      fl = B.flags_r;
      sorted_flags = true;
    }
    if (tiled) {
      const size_t lds = rescore_tiled_lds(d);
      const unsigned nb = (unsigned)(((int64_t)nf + kRtF - 1) / kRtF);
      auto go = [&](auto kern) {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        kern<<<nb, kRtF * kRtS, lds, s>>>(X, n, d, C, B.k_off, fl, (int64_t)nf, labels, dists,
                                          nullptr);
      };
      if (d <= 16) go(k_rescore_tiled<16>);
      else if (d <= 32) go(k_rescore_tiled<32>);
      else if (d <= 64) go(k_rescore_tiled<64>);
      else go(k_rescore_tiled<0>);
    } else {
      auto go = [&](auto kern, int f, int bs) {
        kern<<<grid_for((int64_t)nf, f, 65536), bs, 0, s>>>(X, n, d, C, B.Ct, ktot, B.k_off, fl,
                                                            (int64_t)nf, labels, dists, nullptr,
                                                            nullptr, 0);
      };
      if (sorted_flags && ktot <= kRfOneK * P) go(k_rescore_few<kRfF, kWave>, kRfF, kWave);
      else if (sorted_flags) go(k_rescore_few<kRfF, 256>, kRfF, 256);
      else go(k_rescore_few<1, 256>, 1, 256);
    }
    EAC_LAUNCH_CHECK();
    prof_end(pr2, s);
  }
  if (n_rescored) *n_rescored = (int64_t)nf;
  }  // read-back path
  if (csum_out) {
    EAC_TRY(np_chunk_sums(dists, n, P, B.csum, s));
    *csum_out = B.csum;
  }
  return EAC_OK;
}

struct UpdateBufs {
  int32_t* eflag;  // [ktot + 1]: 1 for an empty cluster (the last entry is scanned, but no result holds it)
  int32_t* erank;  // [ktot + 1]
  uint64_t* dk;
  uint64_t* dks;
  size_t mark;     // arena position of the scratch after these
};

size_t kmeans_update_ws_bytes(int64_t n, int d, int64_t ktot, int P) {
  Arena ar(nullptr, 0, true);
  ar.take<int64_t>(P + 1);
  ar.take<int32_t>(2);
  ar.take<uint32_t>((int64_t)P * n);
  ar.take<uint32_t>(ktot + 1);
  ar.take<int32_t>(ktot + 1);
  ar.take<int32_t>(ktot + 1);
  ar.take<uint64_t>(n);
  ar.take<uint64_t>(n);
  size_t a = ar.used;
  size_t grp = group_ws_bytes(n, P, ktot);
  size_t sort_b = radix_sort_ws_bytes(n, 8, 0);
  size_t scan_b = scan_ws_bytes(ktot + 1, 8);
  size_t m = grp > sort_b ? grp : sort_b;
  m = m > scan_b ? m : scan_b;
  return a + m + 4096;
}

// New centroids of every partition (KMeans.py:709-754) into Cout, except
// those of partitions with upd[p] == 0 (upd nullable); *n_empty (device,
// cleared by the caller) += clusters without a point, which U->eflag marks
// for the reseeding. Nothing is read back.
int kmeans_update(const float* X, int64_t n, int d, const int32_t* labels, const int64_t* h_koff,
                  const int64_t* d_koff, int P, float* Cout, const int32_t* upd, int32_t* n_empty,
                  UpdateBufs* U, Arena& ar, hipStream_t s) {
  const int64_t ktot = h_koff[P];
  const int64_t items = (int64_t)P * n;
  if (items > (int64_t)UINT32_MAX || ktot >= (int64_t)UINT32_MAX)
    return fail(EAC_ERR_UNSUPPORTED, "kmeans update: P*n or k too large");
  uint32_t* members = ar.take<uint32_t>(items);
  uint32_t* start = ar.take<uint32_t>(ktot + 1);
  U->eflag = ar.take<int32_t>(ktot + 1);
  U->erank = ar.take<int32_t>(ktot + 1);
  U->dk = ar.take<uint64_t>(n);
  U->dks = ar.take<uint64_t>(n);
  U->mark = ar.used;
  if (ar.overflow()) return fail(EAC_ERR_WORKSPACE, "kmeans update: workspace too small");
  EAC_TRY(group_by_cluster(labels, n, P, d_koff, h_koff, members, start, nullptr, nullptr, ar, s));
  ar.used = U->mark;
  int64_t kmax = 1;
  for (int p = 0; p < P; ++p)
    if (h_koff[p + 1] - h_koff[p] > kmax) kmax = h_koff[p + 1] - h_koff[p];
  // small clusters (up to 1024 coordinates on average): one wavefront each
  const bool small = d <= kWave && items / ktot * d <= SumStage<kWave>::kFloats;
  const bool v4 = (d & 3) == 0 && (reinterpret_cast<uintptr_t>(X) & 15) == 0;
  const dim3 grid((unsigned)(kmax < 65536 ? kmax : 65536), P < 65535 ? P : 65535);
  auto go = [&](auto kern, int bs) {
    kern<<<grid, bs, 0, s>>>(X, d, members, start, d_koff, P, upd, U->eflag, n_empty, Cout);
  };
  if (small && v4) go(k_centroid_sums<kWave, true>, kWave);
  else if (small) go(k_centroid_sums<kWave, false>, kWave);
  else if (v4) go(k_centroid_sums<256, true>, 256);
  else go(k_centroid_sums<256, false>, 256);
  EAC_LAUNCH_CHECK();
  return EAC_OK;
}

// Empty clusters (total of them, known on the host) take the points of
// smallest (dist, index) of their partition in ascending cluster order.
int kmeans_reseed(const float* X, int64_t n, int d, const float* dists, const int64_t* h_koff,
                  int P, float* Cout, const int32_t* upd, int32_t total, const UpdateBufs& U,
                  Arena& ar, hipStream_t s) {
  if (total == 0) return EAC_OK;
  const int64_t ktot = h_koff[P];
  ar.used = U.mark;
  EAC_TRY((scan_excl<int32_t, int32_t>(U.eflag, U.erank, ktot + 1, 0, nullptr, ar, s)));
  ar.used = U.mark;
  std::vector<int32_t> er(ktot + 1);
  EAC_TRY(d2h(er.data(), U.erank, sizeof(int32_t) * (ktot + 1), s));
  for (int p = 0; p < P; ++p) {
    const int64_t e = er[h_koff[p + 1]] - er[h_koff[p]];
    if (e == 0) continue;
    if (e > n) return fail(EAC_ERR_ARG, "kmeans update: more empty clusters than points");
    k_dist_keys<<<grid_for(n, 256, 4096), 256, 0, s>>>(dists + (int64_t)p * n, n, U.dk);
    EAC_LAUNCH_CHECK();
    EAC_TRY((radix_sort<uint64_t, NoValue>(U.dk, U.dks, nullptr, nullptr, n, 0, 64, ar, s)));
    ar.used = U.mark;
    k_reseed<<<grid_for((h_koff[p + 1] - h_koff[p]) * d, 256, 4096), 256, 0, s>>>(
        X, d, U.dks, U.eflag, U.erank, h_koff[p], h_koff[p + 1], upd ? upd + p : nullptr, Cout);
    EAC_LAUNCH_CHECK();
  }
  return EAC_OK;
}

}  // namespace eac

// ------------------------------------------------------------------ C ABI
using namespace eac;

extern "C" size_t eac_kmeans_workspace_bytes(int64_t n, int32_t d, int64_t k_total, int32_t P) {
  if (n < 1) n = 1;
  if (k_total < 1) k_total = 1;
  if (P < 1) P = 1;
  size_t a = kmeans_label_ws_bytes(n, d, k_total, P);
  size_t b = kmeans_update_ws_bytes(n, d, k_total, P);
  // fit: labels/dists/centroids are caller buffers; the per-partition state
  // (previous inertia, offsets, active, iterations, update flags, two
  // counters), each rounded up to 256 bytes
  Arena fa(nullptr, 0, true);
  fa.take<float>(P);
  fa.take<int64_t>(P + 1);
  fa.take<int32_t>(P);
  fa.take<int32_t>(P);
  fa.take<int32_t>(P);
  fa.take<int32_t>(2);
  size_t c = fa.used + 4096;
  return (a > b ? a : b) + c;
}

static int km_check(const float* X, int64_t n, int32_t d, const float* C, const int64_t* h_koff,
                    int32_t P) {
  if (n < 1 || d < 1 || P < 1) return fail(EAC_ERR_ARG, "kmeans: need n, d, P >= 1");
  if (!X || !C || !h_koff) return fail(EAC_ERR_ARG, "kmeans: null array");
  if (h_koff[0] != 0) return fail(EAC_ERR_ARG, "kmeans: k_off[0] must be 0");
  for (int p = 0; p < P; ++p)
    if (h_koff[p + 1] <= h_koff[p]) return fail(EAC_ERR_ARG, "kmeans: partition %d has k < 1", p);
  if (n >= (1ll << 40) || P >= (1 << 23)) return fail(EAC_ERR_UNSUPPORTED, "kmeans: n or P too large");
  return EAC_OK;
}

extern "C" int eac_kmeans_label(const float* X, int64_t n, int32_t d, const float* C,
                                const int64_t* h_koff, int32_t P, int32_t mode, int32_t* labels,
                                float* dists, int64_t* h_out, void* ws, size_t ws_bytes,
                                void* stream) {
  EAC_TRY(km_check(X, n, d, C, h_koff, P));
  if (!labels) return fail(EAC_ERR_ARG, "kmeans: null labels");
  size_t need = eac_kmeans_workspace_bytes(n, d, h_koff[P], P);
  if (!ws || ws_bytes < need)
    return fail(EAC_ERR_WORKSPACE, "kmeans: workspace %zu < %zu bytes", ws_bytes, need);
  Arena ar(ws, ws_bytes);
  hipStream_t s = (hipStream_t)stream;
  int64_t nres = 0;
  EAC_TRY(kmeans_label(X, n, d, C, h_koff, P, mode, labels, dists, nullptr, &nres, ar, s));
  EAC_HIP_CHECK(hipStreamSynchronize(s));
  prof_flush();
  if (h_out) h_out[0] = nres;
  return EAC_OK;
}

extern "C" int eac_kmeans_update(const float* X, int64_t n, int32_t d, const int32_t* labels,
                                 const float* dists, const int64_t* h_koff, int32_t P,
                                 float* C_new, int64_t* h_out, void* ws, size_t ws_bytes,
                                 void* stream) {
  if (!labels || !dists || !C_new) return fail(EAC_ERR_ARG, "kmeans update: null array");
  EAC_TRY(km_check(X, n, d, C_new, h_koff, P));
  size_t need = eac_kmeans_workspace_bytes(n, d, h_koff[P], P);
  if (!ws || ws_bytes < need)
    return fail(EAC_ERR_WORKSPACE, "kmeans update: workspace %zu < %zu bytes", ws_bytes, need);
  Arena ar(ws, ws_bytes);
  hipStream_t s = (hipStream_t)stream;
  int64_t* k_off = ar.take<int64_t>(P + 1);
  int32_t* d_ctl = ar.take<int32_t>(2);
  EAC_TRY(put_i64(k_off, h_koff, P + 1, s));
  EAC_TRY(fill<int32_t>(d_ctl, 2, 0, s));
  UpdateBufs U;
  EAC_TRY(kmeans_update(X, n, d, labels, h_koff, k_off, P, C_new, nullptr, d_ctl + 1, &U, ar, s));
  int32_t ctl[2];
  EAC_TRY(d2h(ctl, d_ctl, sizeof(ctl), s));
  EAC_TRY(kmeans_reseed(X, n, d, dists, h_koff, P, C_new, nullptr, ctl[1], U, ar, s));
  EAC_HIP_CHECK(hipStreamSynchronize(s));
  if (h_out) h_out[0] = ctl[1];
  return EAC_OK;
}

// ------------------------------------------------- capturable batched fit
namespace eac {
namespace {
// KmGraph buffers (the flag count); info and err are the caller's device
// arrays.
KmGraph carve_graph(Arena& ar, int64_t n, int P, int64_t* info, unsigned int* err) {
  KmGraph g;
  g.d_nf = ar.take<int64_t>(1);
  g.info = info;
  g.err = err;
  g.any = nullptr;
  return g;
}
__global__ void k_graph_init(int64_t* info, unsigned int* err) {
  if (threadIdx.x == 0) {
    info[0] = 0;
    info[1] = 0;
    err[0] = 0u;
  }
}
}  // namespace
}  // namespace eac

extern "C" size_t eac_kmeans_fit_graph_workspace_bytes(int64_t n, int32_t d, int64_t k_total,
                                                       int32_t P) {
  if (n < 1) n = 1;
  if (P < 1) P = 1;
  Arena ga(nullptr, 0, true);
  (void)carve_graph(ga, n, P, nullptr, nullptr);
  return eac_kmeans_workspace_bytes(n, d, k_total, P) + ga.used + 4096;
}

// eac_kmeans_fit for capture in a HIP graph: no host read, no host copy, no
// synchronisation. d_koff: the partition offsets already on the device;
// exactly max_iter labelings run (a partition that meets the stopping rule
// keeps its centroids, so its later labelings repeat, and its iteration
// count in d_iters stops); d_info (device int64[2]) receives the flags
// re-scored and the clusters reseeded, d_err (device uint32) error bits
// (1: flag list overflow, 2: more than 2048 empty clusters in one
// partition): the labels are valid when d_err is 0 after the replay.
extern "C" int eac_kmeans_fit_graph(const float* X, int64_t n, int32_t d, float* C_inout,
                                    const int64_t* h_koff, const int64_t* d_koff, int32_t P,
                                    int32_t max_iter, double tol, int32_t mode, int32_t* labels,
                                    float* dists, int32_t* d_iters, int64_t* d_info,
                                    uint32_t* d_err, void* ws, size_t ws_bytes, void* stream) {
  EAC_TRY(km_check(X, n, d, C_inout, h_koff, P));
  if (!labels || !dists || !d_koff || !d_iters || !d_info || !d_err)
    return fail(EAC_ERR_ARG, "kmeans fit graph: null array");
  if (max_iter < 1) return fail(EAC_ERR_ARG, "kmeans fit graph: max_iter < 1");
  const int64_t ktot = h_koff[P];
  size_t need = eac_kmeans_fit_graph_workspace_bytes(n, d, ktot, P);
  if (!ws || ws_bytes < need)
    return fail(EAC_ERR_WORKSPACE, "kmeans fit graph: workspace %zu < %zu bytes", ws_bytes,
                need);
  hipStream_t s = (hipStream_t)stream;
  Arena ar(ws, ws_bytes);
  KmGraph g = carve_graph(ar, n, P, d_info, d_err);
  float* prev = ar.take<float>(P);
  int32_t* active = ar.take<int32_t>(P);
  int32_t* upd = ar.take<int32_t>(P);
  int32_t* d_any = ar.take<int32_t>(2);
  if (ar.overflow()) return fail(EAC_ERR_WORKSPACE, "kmeans fit graph: workspace too small");
  const size_t mark = ar.used;
  g.any = d_any;
  k_graph_init<<<1, 64, 0, s>>>(d_info, d_err);
  EAC_LAUNCH_CHECK();
  EAC_TRY(fill<int32_t>(d_any, 1, 1, s));  // the first labeling always counts
  k_fit_init<<<grid_for(P, 256, 1024), 256, 0, s>>>(prev, active, d_iters, P);
  EAC_LAUNCH_CHECK();
  for (int it = 1; it <= max_iter; ++it) {
    ar.used = mark;
    int64_t nres = 0;
    const float* csum = nullptr;
    EAC_TRY(kmeans_label(X, n, d, C_inout, h_koff, P, mode, labels, dists, &csum, &nres, ar,
                         s, d_koff, &g));
    k_converge<<<1, 1024, 0, s>>>(csum, np_chunks(n), prev, active, d_iters, upd, P, it, max_iter,
                                  (float)tol, d_any);
    EAC_LAUNCH_CHECK();
    if (it >= max_iter) break;
    ar.used = mark;
    UpdateBufs U;
    EAC_TRY(kmeans_update(X, n, d, labels, h_koff, d_koff, P, C_inout, upd, d_any + 1, &U, ar, s));
    EAC_TRY((scan_excl<int32_t, int32_t>(U.eflag, U.erank, ktot + 1, 0, nullptr, ar, s)));
    k_reseed_dev<<<P < 4096 ? P : 4096, 1024, 0, s>>>(X, d, dists, n, d_koff, P, U.eflag, U.erank,
                                                      upd, C_inout, g.err);
    EAC_LAUNCH_CHECK();
    k_fit_tally<<<1, 64, 0, s>>>(g.info, nullptr, U.erank, ktot, g.any);
    EAC_LAUNCH_CHECK();
  }
  return EAC_OK;
}

extern "C" size_t eac_sum_f32_workspace_bytes(int64_t n, int64_t rows) {
  if (n < 0 || rows < 0) return 0;
  return ((size_t)rows * (size_t)np_chunks(n) + 1) * sizeof(float) + 256;
}

// numpy's float32 x[r].sum() of every row (KMeans.py:164 inertia).
extern "C" int eac_sum_f32_rows(const float* x, int64_t n, int64_t rows, float* out, void* ws,
                                size_t ws_bytes, void* stream) {
  if (n < 0 || rows < 0) return fail(EAC_ERR_ARG, "sum_f32: negative size");
  if (rows == 0) return EAC_OK;
  if (!out || (n > 0 && !x)) return fail(EAC_ERR_ARG, "sum_f32: null array");
  if (n >= (1ll << 40)) return fail(EAC_ERR_UNSUPPORTED, "sum_f32: n too large");
  const size_t need = eac_sum_f32_workspace_bytes(n, rows);
  if (!ws || ws_bytes < need)
    return fail(EAC_ERR_WORKSPACE, "sum_f32: workspace %zu < %zu bytes", ws_bytes, need);
  EAC_TRY(np_sum_rows(x, n, rows, static_cast<float*>(ws), out, (hipStream_t)stream));
  return EAC_OK;
}

// KMeans.py:117-189 per partition: label, count the iteration, stop when
// |sum(dists) - previous| <= tol or iters >= max_iter, otherwise recompute the
// centroids. Partitions stop independently; a stopped partition keeps its
// labels and centroids. labels/dists: [P][n]; C_inout: initial centroids in,
// final centroids out. h_iters[P] (host): iterations run per partition.
// h_out (host): [0] points re-scored in FP64 (all iterations), [1] empty
// clusters re-seeded (all iterations).
extern "C" int eac_kmeans_fit(const float* X, int64_t n, int32_t d, float* C_inout,
                              const int64_t* h_koff, int32_t P, int32_t max_iter, double tol,
                              int32_t mode, int32_t* labels, float* dists, int32_t* h_iters,
                              int64_t* h_out, void* ws, size_t ws_bytes, void* stream) {
  EAC_TRY(km_check(X, n, d, C_inout, h_koff, P));
  if (!labels || !dists) return fail(EAC_ERR_ARG, "kmeans fit: null labels/dists");
  if (max_iter < 1) return fail(EAC_ERR_ARG, "kmeans fit: max_iter < 1");
  const int64_t ktot = h_koff[P];
  size_t need = eac_kmeans_workspace_bytes(n, d, ktot, P);
  if (!ws || ws_bytes < need)
    return fail(EAC_ERR_WORKSPACE, "kmeans fit: workspace %zu < %zu bytes", ws_bytes, need);
  hipStream_t s = (hipStream_t)stream;
  Arena ar(ws, ws_bytes);
  float* prev = ar.take<float>(P);
  int64_t* d_koff = ar.take<int64_t>(P + 1);
  int32_t* active = ar.take<int32_t>(P);
  int32_t* d_iters = ar.take<int32_t>(P);
  int32_t* upd = ar.take<int32_t>(P);
  int32_t* d_any = ar.take<int32_t>(2);
  if (ar.overflow()) return fail(EAC_ERR_WORKSPACE, "kmeans fit: workspace too small");
  const size_t mark = ar.used;
  // the partition offsets go up once; the stopping rule runs on the device
  // and the update follows it unread (a stopped partition's centroids stay),
  // so an iteration costs one read-back: does any partition continue, and
  // did a cluster lose all its points?
  EAC_TRY(put_i64(d_koff, h_koff, P + 1, s));
  k_fit_init<<<grid_for(P, 256, 1024), 256, 0, s>>>(prev, active, d_iters, P);
  EAC_LAUNCH_CHECK();
  int64_t tot_res = 0, tot_empty = 0;
  for (int it = 1; it <= max_iter; ++it) {
    // label every partition (stopped ones relabel identically: unchanged
    // centroids, deterministic kernels)
    int64_t nres = 0;
    ar.used = mark;
    const float* csum = nullptr;
    EAC_TRY(kmeans_label(X, n, d, C_inout, h_koff, P, mode, labels, dists, &csum, &nres, ar, s,
                         d_koff));
    tot_res += nres;
    k_converge<<<1, 1024, 0, s>>>(csum, np_chunks(n), prev, active, d_iters, upd, P, it, max_iter,
                                  (float)tol, d_any);
    EAC_LAUNCH_CHECK();
    if (it >= max_iter) break;  // every partition stops at max_iter
    ar.used = mark;
    UpdateBufs U;
    EAC_TRY(kmeans_update(X, n, d, labels, h_koff, d_koff, P, C_inout, upd, d_any + 1, &U, ar, s));
    int32_t ctl[2];
    EAC_TRY(d2h(ctl, d_any, sizeof(ctl), s));
    if (!ctl[0]) break;
    tot_empty += ctl[1];
    EAC_TRY(kmeans_reseed(X, n, d, dists, h_koff, P, C_inout, upd, ctl[1], U, ar, s));
  }
  if (h_iters) EAC_TRY(d2h(h_iters, d_iters, sizeof(int32_t) * P, s));
  EAC_HIP_CHECK(hipStreamSynchronize(s));
  prof_flush();
  if (h_out) { h_out[0] = tot_res; h_out[1] = tot_empty; }
  return EAC_OK;
}
