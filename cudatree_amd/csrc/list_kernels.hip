// list_kernels.hip -- split search from the nodes' sample lists.
//
// A node evaluates max_features of the F features, yet a schedule over sorted
// rows moves all F rows at every level to have the few it will read in order.
// Here a node keeps one row, the list of its samples in ascending order, and
// the order of an evaluated feature is made when it is
// needed: the words (value index << kLabBits | label) of the node's samples
// are gathered from the feature's column and sorted on the chip.  Samples of
// equal value may leave the sort in any order: a split lies between two
// different values, so its counts, threshold and sides do not depend on it,
// and the trees are those of the sorted rows, bit for bit.
//
// What bounds it: the sort's and the scan's VALU work (a bitonic network of
// two instructions a step, about 120 a 64-sample tile at n = 1,024) and the
// gathers of the words, a cache line a sample at sparse nodes, from columns
// that the workgroup kernels' feature order keeps in L2; against that, sorted
// rows cost 9 bytes of HBM traffic a sample and kept row.  Fits, rows / lists:
// 20,000 x 4,096, 100 trees, 64 of 4,096 features a node 233 / 47 ms (reshuffle
// 170 / 0.6); 200,000 x 256, 200 trees 299 / 138; 1,000,000 x 64 of 256
// levels, 100 classes, 100 trees 690 / 273.
//
// Ascending lists make the gathers of a large node walk its columns in order,
// several samples a cache line (with the lists in feature 0's order the counts
// of 1,000,000 x 64 took 105 ms a fit, ascending 56, when this came in; the marks
// 33 and 23).
//
// Per (node, feature), by the node's size n:
//   up to kListWave           one wave, sorted in its registers   (k_list_scan)
//   up to kListWg[0], [1]     one workgroup of 4 / 16 waves, sorted in
//                             registers and LDS                   (k_list_wg)
//   more                      one workgroup of 16 waves streams the feature's
//                             presorted row of all N samples and keeps the
//                             node's                              (k_list_wg)
//   a feature of few values   above kListWave: one workgroup counts the
//                             node's samples by value and class   (k_list_wg)
#include "device_util.h"
#include "internal.h"

namespace cta {

// ---- tables of the training set --------------------------------------------------
// Made by the first list fit on a training set from its presorted rows: for
// every feature the distinct-value index of each sample (equal floats, +0 and
// -0 included, share one), as words with the sample's label, and the distinct
// values in ascending order.  Three passes over tiles of kCodeTile positions,
// as the value code columns are built: value changes and their in-tile
// prefix, a per-feature scan of the tile totals (k_code_tscan), the scatter.

// pre[f][r]: value changes in position r's tile up to r; tsum[f][tile]: all of
// the tile's; bad[f]: two adjacent distinct values fail the candidate test.
template <class IdxT>
__global__ __launch_bounds__(kCodeThreads) void k_list_flags(const IdxT *rows, const float *XT, uint32_t N,
                                                              uint32_t ntiles, uint32_t *pre, uint32_t *tsum,
                                                              uint32_t *bad) {
  __shared__ uint32_t ws[kCodeThreads / 64];
  const uint32_t f = blockIdx.y, tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
  const IdxT *row = rows + (size_t)f * N;
  const float *x = XT + (size_t)f * N;
  const uint32_t r0 = blockIdx.x * kCodeTile + tid * kCodeItems;
  float v[kCodeItems + 1];
#pragma unroll
  for (int j = 0; j <= kCodeItems; ++j) {
    // (position r0 + j - 1; before the first, the first again: no change)
    const uint32_t r = r0 + (uint32_t)j;
    v[j] = x[sample_of(row[min(r ? r - 1u : 0u, N - 1u)])];
  }
  uint32_t fl[kCodeItems], ts = 0, isbad = 0;
#pragma unroll
  for (int j = 0; j < kCodeItems; ++j) {
    fl[j] = r0 + (uint32_t)j < N && v[j] != v[j + 1] ? 1u : 0u;
    if (fl[j] && !gap_ok(v[j], v[j + 1])) isbad = 1;
    ts += fl[j];
  }
  if (isbad) atomicOr(&bad[f], 1u);
  const uint32_t inc = wave_incl_scan(ts);
  if (lane == 63) ws[wave] = inc;
  __syncthreads();
  uint32_t run = inc - ts;
  for (uint32_t w = 0; w < wave; ++w) run += ws[w];
#pragma unroll
  for (int j = 0; j < kCodeItems; ++j) {
    run += fl[j];
    if (r0 + (uint32_t)j < N) pre[(size_t)f * N + r0 + j] = run;
  }
  if (tid == kCodeThreads - 1) tsum[(size_t)f * ntiles + blockIdx.x] = run;
}

// rank[f][sample] = value index << kLabBits | label, and the distinct values
// of feature f from dval[voff[f]].
template <class IdxT, class LabT>
__global__ __launch_bounds__(kCodeThreads) void k_list_tables(const IdxT *rows, const float *XT, const LabT *y,
                                                               const uint32_t *pre, const uint32_t *tsum, uint32_t N,
                                                               uint32_t ntiles, const uint64_t *voff, uint32_t *rank,
                                                               float *dval) {
  const uint32_t f = blockIdx.y;
  const uint32_t base = tsum[(size_t)f * ntiles + blockIdx.x];
  const IdxT *row = rows + (size_t)f * N;
  const uint32_t *pf = pre + (size_t)f * N;
  float *v = dval + voff[f];
#pragma unroll
  for (int j = 0; j < kCodeItems; ++j) {
    const uint32_t r = blockIdx.x * kCodeTile + (uint32_t)j * kCodeThreads + threadIdx.x;
    if (r >= N) continue;
    const IdxT e = row[r];
    const uint32_t s = sample_of(e), p = pf[r];
    uint32_t lab;
    if constexpr (sizeof(IdxT) == 4) lab = (uint32_t)e >> kIdBits;
    else lab = (uint32_t)y[s];
    rank[(size_t)f * N + s] = (base + p) << kLabBits | lab;
    // the first sample of its value: the prefix rose at r (at a tile's first
    // position it is the position's own flag)
    const bool first = r == 0 || p != (r % kCodeTile ? pf[r - 1] : 0u);
    if (first) v[base + p] = XT[(size_t)f * N + s];
  }
}

// Row entries of all samples in ascending order (the list of a node that
// holds every sample).
template <class IdxT, class LabT>
__global__ void k_list_all(const LabT *y, uint32_t N, IdxT *out) {
  for (uint32_t s = blockIdx.x * blockDim.x + threadIdx.x; s < N; s += gridDim.x * blockDim.x) {
    if constexpr (sizeof(IdxT) == 4) out[s] = (IdxT)(s | ((uint32_t)y[s] << kIdBits));
    else out[s] = (IdxT)s;
  }
}

// gapw[f] (1 before): value indices at least that far apart pass the
// candidate test, whatever lies between them.  A feature whose adjacent
// values all pass it keeps 1; past kGapMax the test is always made on the
// values.
constexpr uint32_t kGapMax = 64;
__global__ __launch_bounds__(kCodeThreads) void k_list_gapw(const float *dval, const uint64_t *voff, const uint32_t *D,
                                                             const uint32_t *bad, uint32_t *gapw) {
  const uint32_t f = blockIdx.y;
  if (!bad[f]) return;
  const float *v = dval + voff[f];
  const uint32_t n = D[f];
  uint32_t most = 1;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i + 1 < n; i += gridDim.x * blockDim.x) {
    const float x = v[i];
    uint32_t w = 1;
    while (w < kGapMax && i + w < n && !gap_ok(x, v[i + w])) ++w;
    most = max(most, w < kGapMax ? w : 0xFFFFFFFFu);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) most = max(most, (uint32_t)__shfl_xor((int)most, o, kWave));
  if (lane_id() == 0 && most > 1) atomicMax(&gapw[f], most);
}

// ---- bitonic sort of 64 E words in a wave's registers ----------------------------
// Position u * 64 + lane is k[u] of that lane, so strides of 64 and more are
// exchanges between registers of a lane, smaller ones between lanes.

// The middle of three (v_med3_u32): with c = 0 the lower of a and b, with
// c = ~0 the higher.
__device__ __forceinline__ uint32_t med3(uint32_t a, uint32_t b, uint32_t c) {
  return max(min(a, b), min(max(a, b), c));
}

// Compare-exchange with lane ^ T: the higher word where `hi` is ~0, the lower
// where it is 0.
template <int T>
__device__ __forceinline__ uint32_t cmpx(uint32_t v, uint32_t hi) {
  if constexpr (T == 1 || T == 2 || T == 8) {
    // quad_perm [1,0,3,2], quad_perm [2,3,0,1], row_ror:8
    constexpr int ctrl = T == 1 ? 0xB1 : T == 2 ? 0x4E : 0x128;
    return med3(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, ctrl, 0xF, 0xF, true), hi);
  } else if constexpr (T == 4) {
    // row_shl:4 into banks 0 and 2, row_shr:4 into banks 1 and 3
    int p = __builtin_amdgcn_update_dpp(0, (int)v, 0x104, 0xF, 0x5, false);
    p = __builtin_amdgcn_update_dpp(p, (int)v, 0x114, 0xF, 0xA, false);
    return med3(v, (uint32_t)p, hi);
  } else if constexpr (T == 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    return med3(r[0], r[1], hi);
  } else {
    static_assert(T == 32, "lane strides are powers of two below 64");
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return med3(r[0], r[1], hi);
  }
}

constexpr int ilog2(int v) { return v <= 1 ? 0 : 1 + ilog2(v / 2); }

// The strides T, T / 2, ..., 1 of the merge of size S (positions with bit S
// set descend).  M[b]: ~0 in the lanes with bit b set.
template <int E, int S, int T>
__device__ __forceinline__ void bitonic_steps(uint32_t (&k)[E], const uint32_t (&M)[6]) {
  if constexpr (T >= 64) {
    constexpr int d = T / 64;
#pragma unroll
    for (int u = 0; u < E; ++u) {
      if (u & d) continue;
      const uint32_t lo = min(k[u], k[u + d]), hi = max(k[u], k[u + d]);
      const bool asc = !(u & (S / 64));
      k[u] = asc ? lo : hi;
      k[u + d] = asc ? hi : lo;
    }
  } else {
#pragma unroll
    for (int u = 0; u < E; ++u) {
      uint32_t hi = M[ilog2(T)];
      if constexpr (S < 64) hi ^= M[ilog2(S) % 6];
      else if (u & (S / 64)) hi = ~hi;
      k[u] = cmpx<T>(k[u], hi);
    }
  }
  if constexpr (T > 1) bitonic_steps<E, S, T / 2>(k, M);
}

template <int E, int S = 2>
__device__ __forceinline__ void wave_sort(uint32_t (&k)[E], const uint32_t (&M)[6]) {
  bitonic_steps<E, S, S / 2>(k, M);
  if constexpr (S < 64 * E) wave_sort<E, S * 2>(k, M);
}

__device__ __forceinline__ void lane_masks(uint32_t (&M)[6]) {
  const uint32_t lane = lane_id();
#pragma unroll
  for (int b = 0; b < 6; ++b) M[b] = 0u - ((lane >> b) & 1u);
}

// ---- scores --------------------------------------------------------------------
// The score of a split is num / den, num = S_L nR + S_R nL and den = nL nR (see
// q_cmp).  S_L <= nL^2 and S_R <= nR^2, so in a node of n samples
// num <= nL nR n <= n^3 / 4 and den <= n^2 / 4: smaller nodes take narrower
// products, and the comparisons stay exact.
constexpr unsigned __int128 most_num(unsigned __int128 n) { return n * n * n / 4; }
static_assert(most_num(CTA_MAX_SAMPLES) >> 64 == 0, "a score's numerator in 64 bits");
static_assert(most_num(kListWave) >> 32 == 0, "and of one wave's nodes in 32");
struct Small {  // n <= 1,024: num <= 2^28, den <= 2^18, products in 64 bits
  using Num = uint32_t;
  using Den = uint32_t;
  using Sum = uint32_t;
  static __device__ __forceinline__ int cmp(uint32_t n1, uint32_t d1, uint32_t n2, uint32_t d2) {
    const uint64_t a = (uint64_t)n1 * d2, b = (uint64_t)n2 * d1;
    return a > b ? 1 : a < b ? -1 : 0;
  }
};
struct Mid {  // n <= 32,768: num <= 2^43, den <= 2^28, products in 96 bits
  using Num = uint64_t;
  using Den = uint32_t;
  using Sum = uint32_t;
  static __device__ __forceinline__ int cmp(uint64_t n1, uint32_t d1, uint64_t n2, uint32_t d2) {
    const uint64_t al = (n1 & 0xFFFFFFFFull) * d2, bl = (n2 & 0xFFFFFFFFull) * d1;
    const uint64_t ah = (n1 >> 32) * d2 + (al >> 32), bh = (n2 >> 32) * d1 + (bl >> 32);
    if (ah != bh) return ah > bh ? 1 : -1;
    const uint32_t x = (uint32_t)al, y = (uint32_t)bl;
    return x > y ? 1 : x < y ? -1 : 0;
  }
};

struct Large {  // any node: products in 128 bits
  using Num = uint64_t;
  using Den = uint64_t;
  using Sum = uint64_t;
  static __device__ __forceinline__ int cmp(uint64_t n1, uint64_t d1, uint64_t n2, uint64_t d2) {
    return q_cmp(n1, d1, n2, d2);
  }
};

// A lane's best split so far (num = 0: none; a split's num is positive).
template <class A>
struct Best {
  typename A::Num num = 0;
  typename A::Den den = 1;
  uint32_t pos = 0;
  int32_t feat = 0x7FFFFFFF;
  uint32_t lo = 0, hi = 0;  // value indices on both sides
};

template <class A>
__device__ __forceinline__ bool beats(const Best<A> &a, const Best<A> &b) {
  const int c = A::cmp(a.num, a.den, b.num, b.den);
  if (c) return c > 0;
  if (a.feat != b.feat) return a.feat < b.feat;
  return a.pos < b.pos;
}

template <class T>
__device__ __forceinline__ T readlane_of(T v, uint32_t lane) {
  if constexpr (sizeof(T) == 8) return (uint64_t)readlane((uint32_t)(v >> 32), lane) << 32 | readlane((uint32_t)v, lane);
  else return readlane(v, lane);
}
template <int kCtrl, int kRowMask, class T>
__device__ __forceinline__ T dpp_of(T v) {
  if constexpr (sizeof(T) == 8) return Move64{}.template operator()<kCtrl, kRowMask>(v);
  else return dpp<kCtrl, kRowMask>(v);
}

template <class A>
__device__ __forceinline__ Best<A> shfl_best(const Best<A> &b, uint32_t lane) {
  Best<A> r;
  r.num = readlane_of(b.num, lane);
  r.den = readlane_of(b.den, lane);
  r.pos = readlane(b.pos, lane);
  r.feat = (int32_t)readlane((uint32_t)b.feat, lane);
  r.lo = readlane(b.lo, lane);
  r.hi = readlane(b.hi, lane);
  return r;
}

struct MoveBest {
  template <int kCtrl, int kRowMask, class A>
  static __device__ __forceinline__ Best<A> move(const Best<A> &b) {
    Best<A> r;
    r.num = dpp_of<kCtrl, kRowMask>(b.num);  // a lane without a source reads num = 0: beaten by any split
    r.den = dpp_of<kCtrl, kRowMask>(b.den);
    r.pos = dpp<kCtrl, kRowMask>(b.pos);
    r.feat = (int32_t)dpp<kCtrl, kRowMask>((uint32_t)b.feat);
    r.lo = dpp<kCtrl, kRowMask>(b.lo);
    r.hi = dpp<kCtrl, kRowMask>(b.hi);
    return r;
  }
};

// The wave's best split, in every lane.
template <class A>
__device__ __forceinline__ Best<A> wave_best_of(Best<A> b) {
  auto step = [&](const Best<A> &o) {
    if (o.num != 0 && (b.num == 0 || beats(o, b))) b = o;
  };
  step(MoveBest::move<kDppRowShr + 1, 0xF>(b));
  step(MoveBest::move<kDppRowShr + 2, 0xF>(b));
  step(MoveBest::move<kDppRowShr + 4, 0xF>(b));
  step(MoveBest::move<kDppRowShr + 8, 0xF>(b));
  step(MoveBest::move<kDppBcast15, 0xA>(b));
  step(MoveBest::move<kDppBcast31, 0xC>(b));
  return shfl_best(b, kWave - 1);
}

__device__ __forceinline__ uint32_t label_bits(uint32_t K) {
  return K > 1 ? 32u - (uint32_t)__builtin_clz(K - 1u) : 1u;
}

// What a feature's split scan needs besides its sorted words: adjacent words
// are a candidate when their value indices differ by gapw or more, or differ
// and the values pass the candidate test.
struct FeatVals {
  uint32_t gapw;
  const float *v;
};
template <class IdxT, class LabT>
__device__ __forceinline__ FeatVals feat_vals(const FitArgs<IdxT, LabT> &a, uint32_t f) {
  return {uniform(a.gapw[f]), a.dval + a.voff[f]};
}
__device__ __forceinline__ bool splits(const FeatVals &fv, uint32_t i, uint32_t j) {
  const uint32_t d = j - i;
  if (d == 0) return false;
  return d >= fv.gapw || gap_ok(fv.v[i], fv.v[j]);
}

// The split scan of a node of n samples over one feature's words in ascending
// order, 64 positions at a time: the class counts before the next position in
// cv (kRegs: lane k holds class k) or carry[] (LDS), the class totals in tv /
// tot[], SL = sum c^2 and D = sum t c before it, T2 = sum t^2.  (A node of at
// most 32,768 samples keeps these sums below 2^32.)
template <class A, bool kRegs>
struct Scan {
  using Sum = typename A::Sum;
  uint32_t n, nbits;
  uint32_t cv, tv;
  uint32_t *carry;
  const uint32_t *tot;
  Sum SL, D, T2;
  int32_t f;
  FeatVals fv;

  // Lane l's position p holds word x, the next one y (lanes with `valid` set).
  __device__ __forceinline__ void tile(uint32_t x, uint32_t y, bool valid, uint32_t p, Best<A> &best) {
    const uint32_t lane = lane_id();
    const uint32_t lab = x & kLabMask, i = x >> kLabBits, j = y >> kLabBits;
    // earlier lanes with the same label, and the label's total
    uint32_t cprev = 0, dD = 0;
    uint64_t rem = ballot(valid);
    if constexpr (kRegs) {
      while (rem) {
        const uint32_t L = readlane(lab, (uint32_t)__ffsll((unsigned long long)rem) - 1u);
        const uint64_t mm = ballot(valid && lab == L);
        const uint32_t b0 = readlane(cv, L), tL = readlane(tv, L);
        if (valid && lab == L) {
          cprev = b0 + mbcnt(mm);
          dD = tL;
        }
        if (lane == L) cv += (uint32_t)__popcll(mm);
        rem &= ~mm;
      }
    } else {
      uint64_t same = rem;
      for (uint32_t b = 0; b < nbits; ++b) {
        const uint32_t bit = (lab >> b) & 1u;
        const uint64_t mb = ballot(bit != 0u);
        same &= bit ? mb : ~mb;
      }
      if (valid) {
        cprev = carry[lab] + mbcnt(same);
        dD = tot[lab];
      }
      wave_sync();
      if (valid && (same >> lane) == 1ull) carry[lab] = cprev + 1u;
      wave_sync();
    }
    const uint32_t iS = wave_incl_scan(valid ? 2u * cprev + 1u : 0u);
    const uint32_t iD = wave_incl_scan(dD);
    const Sum SLp = SL + iS, Dp = D + iD;
    SL += readlane(iS, kWave - 1);
    D += readlane(iD, kWave - 1);
    if (valid && p + 1u < n && splits(fv, i, j)) {
      const uint32_t nL = p + 1u, nR = n - nL;
      const Sum SR = T2 + SLp - 2u * Dp;
      using Num = typename A::Num;
      const Num num = (Num)SLp * nR + (Num)SR * nL;
      const typename A::Den den = (typename A::Den)nL * nR;
      const int c = A::cmp(num, den, best.num, best.den);
      // (positions rise within a feature, so an equal score stays with the
      // earlier one; another feature's wins with the lower id)
      if (c > 0 || (c == 0 && f < best.feat)) {
        best.num = num;
        best.den = den;
        best.pos = p;
        best.feat = f;
        best.lo = i;
        best.hi = j;
      }
    }
  }

  // Positions [p0, p1) of the sorted words w (LDS); `after`: the word at p1,
  // when p1 < n.
  __device__ __forceinline__ void words(const uint32_t *w, uint32_t p0, uint32_t p1, uint32_t after, Best<A> &best) {
    for (uint32_t pb = p0; pb < p1; pb += kWave) {
      const uint32_t p = pb + lane_id();
      const uint32_t x = w[min(p, p1 - 1u)], y = p + 1u < p1 ? w[p + 1u] : after;
      tile(x, y, p < p1, p, best);
    }
  }
};

template <class A>
__device__ __forceinline__ ScanRes to_res(const Best<A> &b) {
  ScanRes r;
  r.num = b.num;
  r.den = b.den;
  r.pos = b.pos;
  r.feat = b.feat;
  r.lo = b.lo;
  r.hi = b.hi;
  return r;
}

// ---- small nodes: one wave -------------------------------------------------------
// The wave's LDS: 64 x kListE words, then the class counts and totals.
__host__ __device__ __forceinline__ uint32_t list_wave_words(uint32_t K) {
  return kListWave + 2u * K;
}

// The features [first, first + count) evaluated at a node of at most 64 E
// samples.  The next feature's words are gathered while this one's are
// scanned.
template <int E, bool kRegs, class IdxT, class LabT>
__device__ __forceinline__ void list_features(const FitArgs<IdxT, LabT> &a, const IdxT *list, uint32_t n,
                                              const int32_t *feats, uint32_t first, uint32_t count, uint32_t nbits,
                                              uint32_t tv, uint32_t *w, uint32_t *carry, const uint32_t *tot,
                                              uint32_t T2, Best<Small> &best) {
  const uint32_t lane = lane_id(), K = (uint32_t)a.K;
  uint32_t M[6];
  lane_masks(M);
  uint32_t id[E], nx[E];
#pragma unroll
  for (int u = 0; u < E; ++u) id[u] = sample_of(list[min((uint32_t)u * kWave + lane, n - 1u)]);
  uint32_t f = uniform((uint32_t)feats[first]);
  auto gather = [&](uint32_t ff) {
    const uint32_t *col = a.rank + (size_t)ff * (uint32_t)a.N;
#pragma unroll
    for (int u = 0; u < E; ++u) nx[u] = col[id[u]];
  };
  gather(f);
  for (uint32_t j = 0; j < count; ++j) {
    uint32_t k[E];
#pragma unroll
    for (int u = 0; u < E; ++u) k[u] = (uint32_t)u * kWave + lane < n ? nx[u] : 0xFFFFFFFFu;
    const uint32_t fn = uniform((uint32_t)feats[min(first + j + 1u, first + count - 1u)]);
    if (j + 1 < count) gather(fn);
    wave_sort<E>(k, M);
    wave_sync();
#pragma unroll
    for (int u = 0; u < E; ++u) w[(uint32_t)u * kWave + lane] = k[u];
    if constexpr (!kRegs)
      for (uint32_t c = lane; c < K; c += kWave) carry[c] = 0;
    wave_sync();
    Scan<Small, kRegs> sc = {n, nbits, 0u, tv, carry, tot, 0u, 0u, T2, (int32_t)f, feat_vals(a, f)};
    sc.words(w, 0, n, 0u, best);
    f = fn;
  }
}

// The same at a node of at most P = 16 or 32 samples: 64 / P features side by
// side, one in each group of P lanes, which sort, count and sum among
// themselves; no word goes through LDS.  (A 64-lane tile for a node of 16
// samples or fewer, 70% of the nodes at 1,000,000 x 64 with 100 classes, left
// three lanes of four idle: small nodes' scans there 60 -> 48 ms a fit, at
// 20,000 x 4,096 18.7 -> 14.2 ms.)
template <int P, class IdxT, class LabT>
__device__ __forceinline__ void list_features_packed(const FitArgs<IdxT, LabT> &a, const IdxT *list, uint32_t n,
                                                     const int32_t *feats, uint32_t first, uint32_t count,
                                                     uint32_t nbits, const uint32_t *tot, uint32_t T2,
                                                     Best<Small> &best) {
  static_assert(P == 16 || P == 32, "groups are whole rows of 16 lanes");
  constexpr uint32_t G = kWave / P;
  const uint32_t lane = lane_id(), g = lane / P, i = lane % P;
  const uint64_t group = (P == 32 ? 0xFFFFFFFFull : 0xFFFFull) << (g * P);
  uint32_t M[6];
  lane_masks(M);
  const uint32_t id = sample_of(list[min(i, n - 1u)]);
  auto feature = [&](uint32_t j) { return (uint32_t)feats[first + min(j + g, count - 1u)]; };
  auto gather = [&](uint32_t f) { return a.rank[(size_t)f * (uint32_t)a.N + id]; };
  uint32_t f = feature(0), nx = gather(f);
  for (uint32_t j = 0; j < count; j += G) {
    const bool valid = i < n && j + g < count;
    uint32_t k[1] = {i < n ? nx : 0xFFFFFFFFu};
    const uint32_t fn = feature(j + G < count ? j + G : j);
    if (j + G < count) nx = gather(fn);
    const FeatVals fv = {a.gapw[f], a.dval + a.voff[f]};
    bitonic_steps<1, 2, 1>(k, M);
    bitonic_steps<1, 4, 2>(k, M);
    bitonic_steps<1, 8, 4>(k, M);
    if constexpr (P == 32) bitonic_steps<1, 16, 8>(k, M);
    bitonic_steps<1, 64, P / 2>(k, M);  // (the last merge ascends in every group)
    const uint32_t x = k[0], y = wave_next(x), lab = x & kLabMask;
    uint64_t same = ballot(valid) & group;
    for (uint32_t b = 0; b < nbits; ++b) {
      const uint32_t bit = (lab >> b) & 1u;
      const uint64_t mb = ballot(bit != 0u);
      same &= bit ? mb : ~mb;
    }
    uint32_t sS = valid ? 2u * mbcnt(same) + 1u : 0u, sD = valid ? tot[lab] : 0u;
    sS += dpp<kDppRowShr + 1>(sS);
    sD += dpp<kDppRowShr + 1>(sD);
    sS += dpp<kDppRowShr + 2>(sS);
    sD += dpp<kDppRowShr + 2>(sD);
    sS += dpp<kDppRowShr + 4>(sS);
    sD += dpp<kDppRowShr + 4>(sD);
    sS += dpp<kDppRowShr + 8>(sS);
    sD += dpp<kDppRowShr + 8>(sD);
    if constexpr (P == 32) {  // the first row's total to the group's second
      sS += dpp<kDppBcast15, 0xA>(sS);
      sD += dpp<kDppBcast15, 0xA>(sD);
    }
    const uint32_t lo = x >> kLabBits, hi = y >> kLabBits;
    if (valid && i + 1u < n && splits(fv, lo, hi)) {
      const uint32_t nL = i + 1u, nR = n - nL, SR = T2 + sS - 2u * sD;
      const uint32_t num = sS * nR + SR * nL, den = nL * nR;
      const int c = Small::cmp(num, den, best.num, best.den);
      if (c > 0 || (c == 0 && (int32_t)f < best.feat)) {
        best.num = num;
        best.den = den;
        best.pos = i;
        best.feat = (int32_t)f;
        best.lo = lo;
        best.hi = hi;
      }
    }
    f = fn;
  }
}

// A wave per task: some of the evaluated features of a node of at most
// kListWave samples (tasks of a class on its XCD's workgroups, as in k_scan).
template <class IdxT, class LabT, bool kRegs>
__global__ __launch_bounds__(kBlock) void k_list_scan(FitArgs<IdxT, LabT> a) {
  if (a.ctl->err) return;  // a list overflowed: the fit fails, nothing more is read
  extern __shared__ uint32_t smem[];
  const uint32_t lane = lane_id();
  const uint32_t K = (uint32_t)a.K, nbits = label_bits(K);
  uint32_t *w = smem + (threadIdx.x / kWave) * list_wave_words(K);
  uint32_t *carry = w + kListWave, *tot = carry + K;
  const uint32_t cls = blockIdx.x % kXcd;
  const uint32_t cn = lane < kXcd ? a.ctl->n_cls[lane] : 0u;
  const uint32_t cbase = wave_incl_scan(cn) - cn;
  const uint32_t lo = readlane(cbase, cls), hi = min(lo + readlane(cn, cls), a.cap_scan);
  const uint32_t nwc = (gridDim.x / kXcd) * kWavesPerBlock;
  for (uint32_t item = lo + (blockIdx.x / kXcd) * kWavesPerBlock + threadIdx.x / kWave; item < hi; item += nwc) {
    const Task tk = a.scan_tasks[item];
    const uint32_t i = uniform(tk.node);
    const FNode nd = a.front[i];
    const uint32_t n = uniform(nd.n);
    uint32_t tv = 0, t2 = 0;
    wave_sync();
    for (uint32_t k = lane; k < K; k += kWave) {
      const uint32_t v = a.cnt[(size_t)i * K + k];
      if (kRegs) tv = v;
      tot[k] = v;
      t2 += v * v;
    }
    wave_sync();
    const uint32_t T2 = wave_sum32(t2);
    const uint32_t first = uniform(tk.first_count & 0xFFFFu), count = uniform(tk.first_count >> 16);
    const IdxT *list = rows_of(a, nd.src, nd.tree, 0) + nd.start;
    const int32_t *feats = a.feats + (size_t)i * a.m;
    Best<Small> best;
    if (n <= 16) {
      list_features_packed<16>(a, list, n, feats, first, count, nbits, tot, T2, best);
    } else if (n <= 32) {
      list_features_packed<32>(a, list, n, feats, first, count, nbits, tot, T2, best);
    } else if (n <= 64) list_features<1, kRegs>(a, list, n, feats, first, count, nbits, tv, w, carry, tot, T2, best);
    else if (n <= 128) list_features<2, kRegs>(a, list, n, feats, first, count, nbits, tv, w, carry, tot, T2, best);
    else if (n <= 256) list_features<4, kRegs>(a, list, n, feats, first, count, nbits, tv, w, carry, tot, T2, best);
    else if (n <= 512) list_features<8, kRegs>(a, list, n, feats, first, count, nbits, tv, w, carry, tot, T2, best);
    else list_features<16, kRegs>(a, list, n, feats, first, count, nbits, tv, w, carry, tot, T2, best);
    best = wave_best_of(best);
    if (lane == 0) a.res[a.aux[i].scan_base + first / a.aux[i].fpt] = to_res(best);
  }
}

// ---- larger nodes: one workgroup -------------------------------------------------
// kWg = 0: 4 waves, up to 4,096 samples; kWg = 1: 16 waves, up to 32,768;
// kWg = 2: 16 waves, any size, from the presorted row; kWg = 3 / 4: 16 / 4
// waves, counted by value and class.
// LDS: the words (kWg = 2: the node's sample set as N bits, then a queue of
// kQueue words per wave; kWg = 3, 4: the table), (W + 1) x K class counts (per
// wave, totals), the waves' results of 8 words each, the next task.
constexpr uint32_t kQueue = 2 * kWave;
__host__ __device__ __forceinline__ uint32_t list_body_words(int wg, uint32_t N, uint32_t hist_max) {
  return wg == 0   ? kListWg[0]
         : wg == 1 ? kListWg[1]
         : wg == 2 ? (N + 31u) / 32u + (uint32_t)kListWaves[2] * kQueue
         : wg == 3 ? hist_max
                   : kHistSmall;
}
__host__ __device__ __forceinline__ uint32_t list_wg_words(int wg, uint32_t K, uint32_t N, uint32_t hist_max) {
  const uint32_t W = (uint32_t)kListWaves[wg];
  return list_body_words(wg, N, hist_max) + (W + 1u) * K + W * 8u + 8u;
}

// The words of the node's samples in ascending order into `w` (W x E x 64
// places, unused ones ~0): every wave sorts its 64 E words, then bitonic
// merges of 2, 4, .. W waves.  A wave that has to leave a descending run
// works on complemented words.
template <int W, int E, class IdxT>
__device__ __forceinline__ void wg_sort(const IdxT *list, uint32_t n, const uint32_t *col, uint32_t *w) {
  const uint32_t lane = lane_id(), wave = uniform(threadIdx.x / kWave);
  const uint32_t base = wave * (E * kWave) + lane;
  uint32_t M[6];
  lane_masks(M);
  uint32_t k[E];
#pragma unroll
  for (int u = 0; u < E; ++u) k[u] = sample_of(list[min(base + (uint32_t)u * kWave, n - 1u)]);
#pragma unroll
  for (int u = 0; u < E; ++u) k[u] = col[k[u]];
  uint32_t flip = (wave & 1u) ? 0xFFFFFFFFu : 0u;
#pragma unroll
  for (int u = 0; u < E; ++u) k[u] = (base + (uint32_t)u * kWave < n ? k[u] : 0xFFFFFFFFu) ^ flip;
  wave_sort<E>(k, M);
#pragma unroll 1
  for (uint32_t r = 2; r <= (uint32_t)W; r <<= 1) {
    const uint32_t nf = (wave & r) ? 0xFFFFFFFFu : 0u;  // (the last merge ascends: wave < W)
#pragma unroll
    for (int u = 0; u < E; ++u) k[u] ^= flip ^ nf;
    flip = nf;
#pragma unroll 1
    for (uint32_t t = r >> 1; t; t >>= 1) {
      __syncthreads();
#pragma unroll
      for (int u = 0; u < E; ++u) w[base + (uint32_t)u * kWave] = k[u];
      __syncthreads();
      const uint32_t ob = base ^ (t * (E * kWave));
      if (wave & t) {
#pragma unroll
        for (int u = 0; u < E; ++u) k[u] = max(k[u], w[ob + (uint32_t)u * kWave]);
      } else {
#pragma unroll
        for (int u = 0; u < E; ++u) k[u] = min(k[u], w[ob + (uint32_t)u * kWave]);
      }
    }
    bitonic_steps<E, 64 * E, 32 * E>(k, M);
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < E; ++u) w[base + (uint32_t)u * kWave] = k[u];
  __syncthreads();
}

// The waves' class counts in cnt[W][K] become each wave's starting counts.
template <int W>
__device__ __forceinline__ void wg_prefix(uint32_t *cnt, uint32_t K) {
  __syncthreads();
  for (uint32_t k = threadIdx.x; k < K; k += W * kWave) {
    uint32_t run = 0;
    for (int v = 0; v < W; ++v) {
      const uint32_t c = cnt[v * K + k];
      cnt[v * K + k] = run;
      run += c;
    }
  }
  __syncthreads();
}

// Adds the labels of the lanes with `valid` set to the wave's counts (those
// of one label by its last lane).
__device__ __forceinline__ void count_labels(uint32_t *own, uint32_t lab, bool valid, uint32_t nbits) {
  uint64_t same = ballot(valid);
  for (uint32_t b = 0; b < nbits; ++b) {
    const uint32_t bit = (lab >> b) & 1u;
    const uint64_t mb = ballot(bit != 0u);
    same &= bit ? mb : ~mb;
  }
  if (valid && (same >> lane_id()) == 1ull) own[lab] += (uint32_t)__popcll(same);
  wave_sync();
}

// The wave's scan state at its starting counts `own`; returns the samples
// before it.
template <class A, bool kRegs>
__device__ __forceinline__ uint32_t scan_start(Scan<A, kRegs> &sc, uint32_t *own, const uint32_t *tot, uint32_t K,
                                               uint32_t n, uint32_t f, const FeatVals &fv) {
  const uint32_t lane = lane_id();
  uint64_t sl = 0, dd = 0, t2 = 0;
  uint32_t before = 0, cv = 0, tv = 0;
  for (uint32_t k = lane; k < K; k += kWave) {
    const uint32_t c = own[k], t = tot[k];
    if (kRegs) {
      cv = c;
      tv = t;
    }
    before += c;
    sl += (uint64_t)c * c;
    dd += (uint64_t)t * c;
    t2 += (uint64_t)t * t;
  }
  using Sum = typename A::Sum;
  if constexpr (sizeof(Sum) == 8) {
    sc.SL = wave_sum64(sl);
    sc.D = wave_sum64(dd);
    sc.T2 = wave_sum64(t2);
  } else {
    sc.SL = wave_sum32((uint32_t)sl);
    sc.D = wave_sum32((uint32_t)dd);
    sc.T2 = wave_sum32((uint32_t)t2);
  }
  sc.n = n;
  sc.nbits = label_bits(K);
  sc.cv = cv;
  sc.tv = tv;
  sc.carry = own;
  sc.tot = tot;
  sc.f = (int32_t)f;
  sc.fv = fv;
  wave_sync();
  return wave_sum32(before);
}

// Entry of a wave's best split in the waves' results: num, den, pos, lo, hi.
template <class A>
__device__ __forceinline__ void put_best(uint32_t *t, const Best<A> &b) {
  t[0] = (uint32_t)b.num;
  t[1] = (uint32_t)((uint64_t)b.num >> 32);
  t[2] = (uint32_t)b.den;
  t[3] = (uint32_t)((uint64_t)b.den >> 32);
  t[4] = b.pos;
  t[5] = b.lo;
  t[6] = b.hi;
}

// The wave with the best entry (positions rise with the waves, so an equal
// score stays with the earlier one); W: none.
template <class A, int W>
__device__ __forceinline__ uint32_t best_entry(const uint32_t *tail) {
  uint32_t win = W;
  uint64_t wnum = 0, wden = 1;
#pragma unroll 1
  for (uint32_t v = 0; v < (uint32_t)W; ++v) {
    const uint64_t num = (uint64_t)tail[v * 8u + 1u] << 32 | tail[v * 8u];
    const uint64_t den = (uint64_t)tail[v * 8u + 3u] << 32 | tail[v * 8u + 2u];
    if (A::cmp((typename A::Num)num, (typename A::Den)den, (typename A::Num)wnum, (typename A::Den)wden) > 0) {
      win = v;
      wnum = num;
      wden = den;
    }
  }
  return uniform(win);
}

// Result entry of a task: the entry t of the winning wave, or none.
__device__ __forceinline__ void put_res(ScanRes *res, const uint32_t *t, uint32_t f, bool found) {
  ScanRes r;
  r.num = found ? (uint64_t)t[1] << 32 | t[0] : 0ull;
  r.den = found ? (uint64_t)t[3] << 32 | t[2] : 1ull;
  r.pos = t[4];
  r.feat = (int32_t)f;
  r.lo = t[5];
  r.hi = t[6];
  *res = r;
}

// Split scan of the n sorted words in LDS: every wave takes 64 E of them, its
// starting class counts from the counts of the waves before it.  Writes the
// result entry and the left class counts of the best split (left[0, K)).
template <int W, int E, bool kRegs, class IdxT, class LabT>
__device__ __forceinline__ void wg_scan(const FitArgs<IdxT, LabT> &a, uint32_t n, uint32_t f, const uint32_t *w,
                                        uint32_t *cnt, const uint32_t *tot, uint32_t *tail, ScanRes *res,
                                        uint32_t *left) {
  const uint32_t lane = lane_id(), wave = uniform(threadIdx.x / kWave), K = (uint32_t)a.K;
  constexpr uint32_t C = E * kWave;
  const uint32_t p0 = min(wave * C, n), p1 = min(p0 + C, n), nbits = label_bits(K);
  uint32_t *own = cnt + wave * K;
  for (uint32_t c = threadIdx.x; c < W * K; c += W * kWave) cnt[c] = 0;
  __syncthreads();
  for (uint32_t pb = p0; pb < p1; pb += kWave) {
    const uint32_t p = pb + lane;
    count_labels(own, w[min(p, p1 - 1u)] & kLabMask, p < p1, nbits);
  }
  wg_prefix<W>(cnt, K);
  Scan<Mid, kRegs> sc;
  scan_start(sc, own, tot, K, n, f, feat_vals(a, f));
  Best<Mid> best;
  if (p0 < p1) sc.words(w, p0, p1, p1 < n ? w[p1] : 0u, best);
  if (kRegs && lane < K) own[lane] = sc.cv;  // the counts at the end of the chunk, as in LDS
  best = wave_best_of(best);
  if (lane == 0) put_best(tail + wave * 8u, best);
  __syncthreads();
  const uint32_t win = best_entry<Mid, W>(tail);
  bool found = win < (uint32_t)W;
  const uint32_t *t = tail + (found ? win : 0u) * 8u;
  const uint32_t pos = t[4];
  if (found) {
    // the entry has to name the words at the split: the sides of the samples
    // follow from its indices, the children's sizes from its position
    found = pos + 1u < n && w[min(pos, n - 1u)] >> kLabBits == t[5] && w[min(pos + 1u, n - 1u)] >> kLabBits == t[6];
    if (!found && threadIdx.x == 0) a.ctl->bad = 1u;
  }
  if (threadIdx.x == 0) put_res(res, t, f, found);
  if (!found) return;  // (the whole workgroup)
  // left class counts: those before the winning wave's chunk (where the wave
  // before it ended) and the chunk's words up to the split
  uint32_t *acc = cnt + win * K;  // its end counts are no longer needed
  for (uint32_t k = threadIdx.x; k < K; k += W * kWave) acc[k] = win ? cnt[(win - 1u) * K + k] : 0u;
  __syncthreads();
  for (uint32_t p = win * C + threadIdx.x; p <= pos; p += W * kWave) atomicAdd(&acc[w[p] & kLabMask], 1u);
  __syncthreads();
  for (uint32_t k = threadIdx.x; k < K; k += W * kWave) left[k] = acc[k];
}

// Split scan of a node of any size: the waves stream equal shares of the
// feature's presorted row of all N samples and keep the node's, whose set is
// in LDS as N bits.  Twice: for the waves' class counts, then for the scan,
// which takes 64 kept words at a time from a queue of the wave.  Streaming
// costs about 50 VALU instructions per 64 row entries whether they are kept
// or not, the scan about 250 per 64 kept, so it pays while a node holds more
// than a small share of the samples: 200,000 x 256, 200 trees, nodes above
// 32,768 samples (30% of the evaluated elements) 38 ms where moving their
// rows took 60 and scanning them 30, and 29 since tasks run in feature order.
template <int W, bool kRegs, class IdxT, class LabT>
__device__ __forceinline__ void wg_filter(const FitArgs<IdxT, LabT> &a, const IdxT *list, uint32_t n, uint32_t f,
                                          uint32_t *set, uint32_t *cnt, const uint32_t *tot, uint32_t *tail,
                                          ScanRes *res, uint32_t *left) {
  const uint32_t lane = lane_id(), wave = uniform(threadIdx.x / kWave), K = (uint32_t)a.K, N = (uint32_t)a.N;
  const uint32_t nbits = label_bits(K), Wb = (N + 31u) / 32u;
  const IdxT *row = a.presorted + (size_t)f * N;
  const uint32_t *col = a.rank + (size_t)f * N;
  uint32_t *q = set + Wb + wave * kQueue, *own = cnt + wave * K;
  constexpr int U = 4;
  for (uint32_t c = threadIdx.x; c < Wb; c += W * kWave) set[c] = 0;
  for (uint32_t c = threadIdx.x; c < W * K; c += W * kWave) cnt[c] = 0;
  __syncthreads();
  for (uint32_t p = threadIdx.x; p < n; p += U * W * kWave) {
    uint32_t s[U];
#pragma unroll
    for (int u = 0; u < U; ++u) s[u] = sample_of(list[min(p + (uint32_t)u * (W * kWave), n - 1u)]);
#pragma unroll
    for (int u = 0; u < U; ++u) atomicOr(&set[s[u] >> 5], 1u << (s[u] & 31u));  // (the last one again past the end)
  }
  __syncthreads();
  // this wave's share of the row, whole tiles of U x 64
  const uint32_t share = (N + W * U * kWave - 1u) / (W * U * kWave) * (U * kWave);
  const uint32_t r0 = min(wave * share, N), r1 = min(r0 + share, N);
  uint32_t firstw = 0xFFFFFFFFu;  // the wave's first kept word
  for (uint32_t rb = r0; rb < r1; rb += U * kWave) {
    uint32_t e[U];
    load_row_batch(row, rb, r1, e);
    uint32_t lab[U];
    bool in[U];
#pragma unroll
    for (int u = 0; u < U; ++u) lab[u] = a.label((IdxT)e[u]);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t s = sample_of((IdxT)e[u]);
      in[u] = rb + (uint32_t)u * kWave + lane < r1 && (set[s >> 5] >> (s & 31u) & 1u) != 0u;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint64_t mk = ballot(in[u]);
      if (!mk) continue;
      if (firstw == 0xFFFFFFFFu)
        firstw = uniform(col[sample_of((IdxT)readlane(e[u], (uint32_t)__ffsll((unsigned long long)mk) - 1u))]);
      count_labels(own, lab[u], in[u], nbits);
    }
  }
  if (lane == 0) tail[wave * 8u + 7u] = firstw;
  wg_prefix<W>(cnt, K);
  uint32_t after = 0;  // the first kept word of the waves behind
#pragma unroll 1
  for (uint32_t v = W; v-- > wave + 1u;) {
    const uint32_t x = tail[v * 8u + 7u];
    if (x != 0xFFFFFFFFu) after = x;
  }
  Scan<Large, kRegs> sc;
  const uint32_t p0 = scan_start(sc, own, tot, K, n, f, feat_vals(a, f));
  Best<Large> best;
  uint32_t qn = 0, qd = 0;  // words queued, words scanned
  for (uint32_t rb = r0; rb < r1; rb += U * kWave) {
    uint32_t e[U], x[U];
    load_row_batch(row, rb, r1, e);
    bool in[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t s = sample_of((IdxT)e[u]);
      in[u] = rb + (uint32_t)u * kWave + lane < r1 && (set[s >> 5] >> (s & 31u) & 1u) != 0u;
      x[u] = 0;
      if (in[u]) x[u] = col[s];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint64_t mk = ballot(in[u]);
      if (in[u]) q[(qn + mbcnt(mk)) % kQueue] = x[u];
      qn += (uint32_t)__popcll(mk);
      wave_sync();
      if (qn - qd > kWave) {  // a whole tile and the word after it
        sc.tile(q[(qd + lane) % kQueue], q[(qd + lane + 1u) % kQueue], true, p0 + qd + lane, best);
        qd += kWave;
        wave_sync();
      }
    }
  }
  if (qn != qd) {
    const uint32_t m = qn - qd;  // at most 64
    const uint32_t y = lane + 1u < m ? q[(qd + lane + 1u) % kQueue] : after;
    sc.tile(q[(qd + lane) % kQueue], y, lane < m, p0 + qd + lane, best);
  }
  if (kRegs && lane < K) own[lane] = sc.cv;  // the counts at the end of the share, as in LDS
  best = wave_best_of(best);
  if (lane == 0) put_best(tail + wave * 8u, best);
  __syncthreads();
  const uint32_t win = best_entry<Large, W>(tail);
  bool found = win < (uint32_t)W;
  const uint32_t *t = tail + (found ? win : 0u) * 8u;
  const uint32_t pos = t[4], lo = t[5];
  if (found) {
    // left class counts: those before the winning wave's share and its kept
    // samples up to the split's value
    uint32_t *acc = cnt + win * K;
    for (uint32_t k = threadIdx.x; k < K; k += W * kWave) acc[k] = win ? cnt[(win - 1u) * K + k] : 0u;
    __syncthreads();
    for (uint32_t r = win * share + threadIdx.x; r < min((win + 1u) * share, N); r += W * kWave) {
      const uint32_t s = sample_of(row[r]);
      if (!(set[s >> 5] >> (s & 31u) & 1u)) continue;
      const uint32_t x = col[s];
      if (x >> kLabBits <= lo) atomicAdd(&acc[x & kLabMask], 1u);
    }
    __syncthreads();
    uint32_t sum = 0;
    for (uint32_t k = lane; k < K; k += kWave) sum += acc[k];
    // (they have to be the samples up to the split's position)
    found = wave_sum32(sum) == pos + 1u;
    if (!found && threadIdx.x == 0) a.ctl->bad = 1u;
    for (uint32_t k = threadIdx.x; k < K; k += W * kWave) left[k] = acc[k];
  }
  if (threadIdx.x == 0) put_res(res, t, f, found);
}

// Inclusive prefix sums over groups of V = 16, 32 or 64 lanes.
template <int V>
__device__ __forceinline__ uint32_t group_incl_scan(uint32_t v) {
  if constexpr (V == 64) return wave_incl_scan(v);
  v += dpp<kDppRowShr + 1>(v);
  v += dpp<kDppRowShr + 2>(v);
  v += dpp<kDppRowShr + 4>(v);
  v += dpp<kDppRowShr + 8>(v);
  if constexpr (V == 32) v += dpp<kDppBcast15, 0xA>(v);
  return v;
}

// Split scan of a node over a feature of D <= 64 W values: the samples counted
// by value and class in LDS (table h, hist_stride(K) words a value), then the
// candidates between adjacent present values scored from the running class
// counts, a lane a value.  No order of the samples is needed: per sample it
// takes the value's code, the label and one LDS atomic.  The table's part is
// as long as the samples' at small nodes (at 1,000,000 x 64 of 256 levels, 100
// classes, 9,300 samples a task), so all waves share it: V = 16, 32 or 64
// values a wave, the wave's lanes over 64 / V classes at a time, and the left
// counts summed by every wave (64 values a wave and the left counts by one
// thread a class 52 ms, this way 39).
template <int W, int V, class IdxT, class LabT>
__device__ __forceinline__ void wg_hist(const FitArgs<IdxT, LabT> &a, const IdxT *list, uint32_t n, uint32_t f,
                                        uint32_t *h, uint32_t *cnt, const uint32_t *tot, uint32_t *tail, ScanRes *res,
                                        uint32_t *left) {
  const uint32_t lane = lane_id(), wave = uniform(threadIdx.x / kWave), K = (uint32_t)a.K;
  const uint32_t Kp = hist_stride(K), D = uniform(a.ndist[f]);
  for (uint32_t c = threadIdx.x; c < D * Kp; c += W * kWave) h[c] = 0;
  __syncthreads();
  IndexCol col = index_col(a, f);
  col.kind = uniform(col.kind);
  constexpr int U = 8;
  for (uint32_t p = threadIdx.x; p < n; p += U * W * kWave) {
    uint32_t e[U], x[U], l[U];
#pragma unroll
    for (int u = 0; u < U; ++u) e[u] = (uint32_t)list[min(p + (uint32_t)u * (W * kWave), n - 1u)];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t s = sample_of((IdxT)e[u]);
      l[u] = a.label((IdxT)e[u]);
      x[u] = col.at(s);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (p + (uint32_t)u * (W * kWave) < n) atomicAdd(&h[x[u] * Kp + l[u]], 1u);
  }
  __syncthreads();
  // class counts of the wave's V values, then those before them
  constexpr uint32_t G = kWave / V;
  const uint32_t v0 = min(wave * V, D), v1 = min(v0 + V, D);
  uint32_t *own = cnt + wave * K;
  for (uint32_t k = lane; k < K; k += kWave) {
    uint32_t s = 0;
    for (uint32_t v = v0; v < v1; ++v) s += h[v * Kp + k];
    own[k] = s;
  }
  wg_prefix<W>(cnt, K);
  // a lane a value and every G-th class, summed over the G groups of V lanes
  const uint32_t g = lane / V, v = v0 + lane % V;
  const bool valid = v < v1;
  uint64_t SL = 0, Dd = 0, T2 = 0;
  uint32_t here = 0, nL = 0;
  if (v0 < v1)
    for (uint32_t k0 = 0; k0 < K; k0 += G) {
      const uint32_t k = k0 + g;
      const uint32_t x = valid && k < K ? h[v * Kp + k] : 0u, t = k < K ? tot[k] : 0u;
      const uint32_t c = (k < K ? own[k] : 0u) + group_incl_scan<V>(x);
      here += x;
      nL += c;
      SL += (uint64_t)c * c;
      Dd += (uint64_t)t * c;
      T2 += (uint64_t)t * t;
    }
#pragma unroll
  for (int o = V; o < kWave; o <<= 1) {
    here += (uint32_t)__shfl_xor((int)here, o, kWave);
    nL += (uint32_t)__shfl_xor((int)nL, o, kWave);
    SL += (uint64_t)__shfl_xor((unsigned long long)SL, o, kWave);
    Dd += (uint64_t)__shfl_xor((unsigned long long)Dd, o, kWave);
    T2 += (uint64_t)__shfl_xor((unsigned long long)T2, o, kWave);
  }
  here = g == 0 ? here : 0u;  // (the first group goes on)
  const uint64_t present = ballot(here != 0u);
  if (lane == 0) tail[wave * 8u + 7u] = present ? v0 + (uint32_t)__ffsll((unsigned long long)present) - 1u : 0xFFFFFFFFu;
  __syncthreads();
  // the next present value: in the wave's, else the first of the waves behind
  uint32_t nx = 0xFFFFFFFFu;
#pragma unroll 1
  for (uint32_t w = W; w-- > wave + 1u;) {
    const uint32_t x = tail[w * 8u + 7u];
    if (x != 0xFFFFFFFFu) nx = x;
  }
  const uint64_t later = lane == kWave - 1 ? 0ull : present >> (lane + 1u);
  if (later) nx = v + (uint32_t)__ffsll((unsigned long long)later);
  const FeatVals fv = feat_vals(a, f);
  Best<Large> best;
  if (here != 0u && nx != 0xFFFFFFFFu && splits(fv, v, nx)) {
    const uint64_t l = nL, r = (uint64_t)n - nL, SR = T2 + SL - 2 * Dd;
    best.num = SL * r + SR * l;
    best.den = l * r;
    best.pos = nL - 1u;
    best.feat = (int32_t)f;
    best.lo = v;
    best.hi = nx;
  }
  best = wave_best_of(best);
  if (lane == 0) put_best(tail + wave * 8u, best);
  __syncthreads();
  const uint32_t win = best_entry<Large, W>(tail);
  bool found = win < (uint32_t)W;
  const uint32_t *t = tail + (found ? win : 0u) * 8u;
  if (found) {
    // left class counts: those before the winning wave's values and theirs up
    // to the split (they have to be the samples up to the split's position)
    const uint32_t last = min(t[5], D - 1u);
    uint32_t *acc = cnt + win * K;
    for (uint32_t k = lane; k < K; k += kWave) {
      uint32_t s = 0;
      for (uint32_t x = win * V + wave; x <= last; x += W) s += h[x * Kp + k];
      if (s) atomicAdd(&acc[k], s);
    }
    __syncthreads();
    if (wave == 0) {
      uint32_t sum = 0;
      for (uint32_t k = lane; k < K; k += kWave) {
        left[k] = acc[k];
        sum += acc[k];
      }
      found = wave_sum32(sum) == t[4] + 1u;
      if (!found && lane == 0) a.ctl->bad = 1u;
    }
  }
  if (threadIdx.x == 0) put_res(res, t, f, found);
}

template <int kWg, int E, bool kRegs, class IdxT, class LabT>
__device__ __forceinline__ void wg_task(const FitArgs<IdxT, LabT> &a, const IdxT *list, uint32_t n, uint32_t f,
                                        uint32_t *w, uint32_t *cnt, const uint32_t *tot, uint32_t *tail, ScanRes *res,
                                        uint32_t *left) {
  constexpr int W = kListWaves[kWg];
  wg_sort<W, E>(list, n, a.rank + (size_t)f * (uint32_t)a.N, w);
  wg_scan<W, E, kRegs>(a, n, f, w, cnt, tot, tail, res, left);
}

// A workgroup per (node, feature).  The tasks are in feature order; the c-th
// eighth of them (class c) belongs to the G workgroups of XCD c, so that the
// ones in flight share few columns in its L2: each starts with the task
// of its own number, and any beyond the G-th are taken one at a time by
// whoever is free, workgroups of other classes too -- nodes differ in size by
// orders of magnitude, so no fixed split would be even.  A level with few
// tasks costs its idle workgroups no atomics.
template <class IdxT, class LabT, int kWg, bool kRegs>
__global__ __launch_bounds__(kListWaves[kWg] * kWave) void k_list_wg(FitArgs<IdxT, LabT> a) {
  if (a.ctl->err) return;  // a list overflowed: the fit fails, nothing more is read
  constexpr int W = kListWaves[kWg];
  extern __shared__ uint32_t smem[];
  const uint32_t K = (uint32_t)a.K;
  uint32_t *w = smem, *cnt = w + list_body_words(kWg, (uint32_t)a.N, a.hist_max), *tot = cnt + W * K, *tail = tot + K, *next = tail + W * 8u;
  const uint32_t G = gridDim.x / kXcd, total = min(uniform(a.ctl->n_wg[kWg]), a.cap_wg[kWg]);
  bool own = true;
  for (uint32_t turn = 0; turn < kXcd;) {
    const uint32_t cls = (blockIdx.x + turn) % kXcd;
    const uint32_t first = (uint32_t)((uint64_t)total * cls / kXcd);
    const uint32_t count = (uint32_t)((uint64_t)total * (cls + 1u) / kXcd) - first;
    uint32_t item = blockIdx.x / kXcd;
    if (!own) {
      if (count <= G) {
        ++turn;
        continue;
      }
      __syncthreads();
      if (threadIdx.x == 0) *next = G + atomicAdd(&a.ctl->wg_next[kWg][cls], 1u);
      __syncthreads();
      item = uniform(*next);
    }
    own = false;
    if (item >= count) {
      if (count > G) ++turn;  // (else the loop's next round does it)
      continue;
    }
    __syncthreads();  // (the last task's LDS is free)
    const Task tk = a.wg_tasks[kWg][first + item];
    const uint32_t i = uniform(tk.node), j = uniform(tk.first_count & 0xFFFFu);
    const FNode nd = a.front[i];
    const uint32_t n = uniform(nd.n);
    const uint32_t f = uniform((uint32_t)a.feats[(size_t)i * a.m + j]);
    const IdxT *list = rows_of(a, nd.src, nd.tree, 0) + nd.start;
    for (uint32_t k = threadIdx.x; k < K; k += W * kWave) tot[k] = a.cnt[(size_t)i * K + k];
    ScanRes *res = a.res + a.aux[i].scan_base + j;
    uint32_t *left = a.hist + a.aux[i].hist_base + (size_t)j * K;
    if constexpr (kWg == 0) {
      if (n <= 2048) wg_task<kWg, 8, kRegs>(a, list, n, f, w, cnt, tot, tail, res, left);
      else wg_task<kWg, 16, kRegs>(a, list, n, f, w, cnt, tot, tail, res, left);
    } else if constexpr (kWg >= 3) {
      const uint32_t D = uniform(a.ndist[f]);
      if (D <= W * 16u) wg_hist<W, 16>(a, list, n, f, w, cnt, tot, tail, res, left);
      else if (D <= W * 32u) wg_hist<W, 32>(a, list, n, f, w, cnt, tot, tail, res, left);
      else wg_hist<W, 64>(a, list, n, f, w, cnt, tot, tail, res, left);
    } else if constexpr (kWg == 2) {
      wg_filter<W, kRegs>(a, list, n, f, w, cnt, tot, tail, res, left);
    } else {
      if (n <= 8192) wg_task<kWg, 8, kRegs>(a, list, n, f, w, cnt, tot, tail, res, left);
      else if (n <= 16384) wg_task<kWg, 16, kRegs>(a, list, n, f, w, cnt, tot, tail, res, left);
      else wg_task<kWg, 32, kRegs>(a, list, n, f, w, cnt, tot, tail, res, left);
    }
  }
}

}  // namespace cta
