// mk_sample.hip — on-device sampling of the next token from the decode
// step's fp32 logits (libmk.so, MI355X / gfx950).
//
// The reference exposes sampling through NxDI's on-device sampler:
// --top-k / --top-p / --temperature / --global-topk / --on-device-sampling
// (main.py:57-61, 85, 129-130) with per-sequence parameters built by
// prepare_sampling_params(batch_size, top_k, top_p, temperature)
// (main.py:195-206). HF generation semantics are followed:
//   * greedy (top_k == 1, or temperature <= 0): the argmax, lowest index on ties;
//   * otherwise: x = logits / temperature; keep every token whose x is >= the
//     top_k-th largest x (ties at the threshold kept, as TopKLogitsWarper);
//     top_k <= 0 or > MK_SAMPLE_MAX_TOPK means the global cap
//     MK_SAMPLE_MAX_TOPK (NxDI's global top-k); then nucleus filtering over
//     the kept tokens' softmax: in descending order, a token is kept while
//     the probability mass before it is < top_p (TopPLogitsWarper: the top
//     token always stays); then a draw from the renormalised distribution.
// The draw is an inverse CDF over the kept tokens in descending order of x
// (ties by ascending index) with u = Philox4x32-10(key = seed, counter =
// (counter[row], row, 0, 0)), first output word >> 8 times 2^-24. Passing a
// sequence's position as its counter gives every step of every sequence its
// own reproducible u with no RNG state on the device.
//
// How a row is sampled. What bounds it is one workgroup's path through a row
// of 128256 logits: one CU reads at most about 42 GB/s from memory (12 us for
// the row), and the exact radix select read the row five times, with LDS
// histogram atomics that mostly hit two or three bins (a row's floats share
// few exponents) and a serial scan of 256 bins: 172 us at batch 1, 189 us at
// batch 32. So the row is read once, by many workgroups, and only its best
// tokens are looked at again:
//   1. mk_group_max_kernel (with scratch): the row as at most 8192 groups of
//      4 * 2^s consecutive logits (16 for 128256); the largest key of each
//      group to scratch. Without scratch, and in rows of up to SOLO logits, the
//      row's one workgroup does this itself, into LDS (a greedy row's just takes
//      the argmax);
//   2. mk_sample_kernel, one 1024-thread workgroup per row: a key L that at
//      least k group maxima reach, from a histogram of the maxima over 2048
//      equal key ranges (bisection within one range where that is too coarse).
//      At least k logits are then >= L, so the top-k set lies in the groups
//      whose maximum is >= L: a little over k of them, the only ones read again;
//   3. their logits >= L go to LDS and are sorted (descending key, ascending
//      index): into the same kind of key ranges, then by counting within a
//      range; the k-th of them is the threshold, ties included;
//   4. softmax numerators in that order, an inclusive prefix sum (fixed tree:
//      bitwise repeatable), the nucleus cut and the draw.
// A row whose logits >= L do not fit in LDS (many of the best ones in the same
// few groups) takes an exact radix select over the whole row instead, and
// candidates of which many share a key range a bitonic sort.
// Measured (128256 logits, back to back): batch 1, top-k 50: 177 -> 13.2 us;
// batch 32 with top-k up to 1024: 190 -> 22.0 us. Of that mk_group_max_kernel takes
// 3.8 and 4.6 us, mk_sample_kernel 9.8 and 18.0; with bisection alone for L and a
// bitonic sort throughout it took 18 and 41 us.
#include <hip/hip_runtime.h>

#include <stdint.h>
#include <string.h>

#include "mk.h"

namespace {

constexpr int ST = 1024;                 // threads per workgroup
constexpr int CAND = MK_SAMPLE_CAND;     // candidate slots (top-k set incl. ties)
constexpr int MAXK = MK_SAMPLE_MAX_TOPK;

struct SParams {
  const float* logits;
  const float* params;   // [batch][3]: top_k, top_p, temperature
  const int32_t* counter;
  int32_t* tokens;
  float* uniforms;
  unsigned long long seed;
  int vocab, stride;
};

// Order-preserving key of an fp32 value (larger float -> larger key); NaN -> 0.
__device__ __forceinline__ uint32_t okey(float f) {
  const uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return 0u;
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float key_to_float(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// Philox4x32-10 (Salmon, Moraes, Dror, Shaw, SC'11): 10 rounds of
// (hi, lo) = M * c products mixed with the key, key bumped by the Weyl
// constants between rounds. Returns the first output word.
__device__ __forceinline__ uint32_t philox_first(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3, uint32_t k0,
                                                 uint32_t k1) {
  constexpr uint32_t M0 = 0xD2511F53u, M1 = 0xCD9E8D57u, W0 = 0x9E3779B9u, W1 = 0xBB67AE85u;
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    const uint64_t p0 = (uint64_t)M0 * c0, p1 = (uint64_t)M1 * c2;
    const uint32_t hi0 = (uint32_t)(p0 >> 32), lo0 = (uint32_t)p0, hi1 = (uint32_t)(p1 >> 32), lo1 = (uint32_t)p1;
    const uint32_t n0 = hi1 ^ c1 ^ k0, n2 = hi0 ^ c3 ^ k1;
    c0 = n0;
    c1 = lo1;
    c2 = n2;
    c3 = lo0;
    k0 += W0;
    k1 += W1;
  }
  return c0;
}

constexpr int SORT = 4096;               // logits the sort in LDS holds
constexpr int BINS = 2048;               // key ranges of a histogram
constexpr int CROWD = 32;                // candidates in one key range that are still ordered by counting
constexpr int NG = 8;                    // group maxima per thread
constexpr int MAX_GROUPS = NG * ST;
// Longest row that its own workgroup reads alone, with scratch too. The first
// kernel costs 2 us and its launch; one workgroup's pass over 32768 logits is about
// as long. With scratch against without, batch 1: 8192 logits greedy 6.3, 3.4 us,
// top-k 50 11.9, 10.7; 32768 greedy 6.4, 6.0, top-k 50 13.4, 13.7; 48000 6.7, 7.6
// and 13.9, 16.6 (and a call without it takes 4 us less of the host's time).
constexpr int SOLO = 32768;
constexpr int GT = 256;                  // threads of the group maximum kernel
constexpr int GSEG = 4;                  // 256-logit segments per wave of it

// Logits per group: 4 * 2^s, the smallest that gives at most MAX_GROUPS groups.
// 0: a row that is sampled without groups (it fits the sort as a whole, or is
// so long that a group would span more than the 64 lanes x 4 logits of one load).
__host__ __device__ inline int group_size(int vocab) {
  if (vocab <= SORT || vocab > 256 * MAX_GROUPS) return 0;
  int gs = 4;
  while ((vocab + gs - 1) / gs > MAX_GROUPS) gs *= 2;
  return gs;
}
static_assert(SORT / 4 >= MAXK && MAX_GROUPS / 2 >= MAXK, "at least k groups, in groups of 4 and of more");

struct SLds {
  uint32_t hist[BINS];             // counts of a histogram, then its start offsets
  unsigned long long cand[SORT];   // (key << 32) | (0xffffffff - index)
  unsigned long long tmp[SORT];    // the candidates by key range (the row's own group maxima before that)
  float csum[2][CAND];             // prefix sums of the softmax numerators, alternating by step
  unsigned long long best[ST / 64];
  uint32_t cnt[2][ST / 64];        // counts of each wave, alternating by step
  uint32_t wmin[ST / 64], wmax[ST / 64];
  uint16_t glist[MAX_GROUPS];      // the groups that hold candidates
  uint32_t prefix, need, ncand, nties, ngl, crowded;
  int bin, at_bin, n, nkeep, pick;
};

// Steps within each 16-lane row by DPP, then the four rows through v_readlane
// (a lane shuffle would be an LDS round trip per step).
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, false);
}
__device__ __forceinline__ uint32_t lane_u32(uint32_t v, int l) { return (uint32_t)__builtin_amdgcn_readlane((int)v, l); }
__device__ __forceinline__ uint32_t umax(uint32_t a, uint32_t b) { return a > b ? a : b; }
__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
  v = umax(v, dpp_u32<0xb1>(v));    // quad_perm [1,0,3,2]
  v = umax(v, dpp_u32<0x4e>(v));    // quad_perm [2,3,0,1]
  v = umax(v, dpp_u32<0x124>(v));   // row_ror:4
  v = umax(v, dpp_u32<0x128>(v));   // row_ror:8
  return umax(umax(lane_u32(v, 0), lane_u32(v, 16)), umax(lane_u32(v, 32), lane_u32(v, 48)));
}
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v) {
  const int lane = threadIdx.x & 63;
  v += dpp_u32<0x111>(v);   // row_shr:1, zeros shifted in
  v += dpp_u32<0x112>(v);
  v += dpp_u32<0x114>(v);
  v += dpp_u32<0x118>(v);
  const uint32_t r0 = lane_u32(v, 15), r1 = lane_u32(v, 31), r2 = lane_u32(v, 47);
  return v + (lane >= 16 ? r0 : 0u) + (lane >= 32 ? r1 : 0u) + (lane >= 48 ? r2 : 0u);
}

// Keys of the 4 logits i .. i+3 of a row (0 past its end). One 16-byte load
// where the row is 16-byte aligned and all 4 are in it.
__device__ __forceinline__ void keys4(const float* x, int i, int V, bool vec, uint32_t (&k)[4]) {
  if (vec && i + 4 <= V) {
    const float4 v = *reinterpret_cast<const float4*>(x + i);
    k[0] = okey(v.x);
    k[1] = okey(v.y);
    k[2] = okey(v.z);
    k[3] = okey(v.w);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) k[e] = i + e < V ? okey(x[i + e]) : 0u;
  }
}
__device__ __forceinline__ bool aligned16(const float* x) { return (reinterpret_cast<uintptr_t>(x) & 15u) == 0; }

// The largest key of each group in the 256-logit segments seg, seg + step, ..
// (NSEG of them at once in flight) of a row, by one wave: a lane holds 4
// logits of a segment, a group is gs / 4 neighbouring lanes.
template <int NSEG, class Store>
__device__ __forceinline__ void group_max(const float* x, int V, int gs, int seg, int step, Store&& store) {
  const int lane = threadIdx.x & 63;
  const bool vec = aligned16(x);
  uint32_t k[NSEG][4];
#pragma unroll
  for (int s = 0; s < NSEG; ++s) keys4(x, (seg + s * step) * 256 + lane * 4, V, vec, k[s]);
#pragma unroll
  for (int s = 0; s < NSEG; ++s) {
    uint32_t m = umax(umax(k[s][0], k[s][1]), umax(k[s][2], k[s][3]));
    for (int o = 1; o < gs / 4; o <<= 1) m = umax(m, (uint32_t)__shfl_xor((int)m, o, 64));
    const int i = (seg + s * step) * 256 + lane * 4;
    if ((i & (gs - 1)) == 0 && i < V) store(i >> __builtin_ctz(gs), m);
  }
}

__global__ void __launch_bounds__(GT) mk_group_max_kernel(const float* logits, int V, int stride, int gs,
                                                          uint32_t* gmax, int ngroups) {
  const float* x = logits + (size_t)blockIdx.x * stride;
  uint32_t* out = gmax + (size_t)blockIdx.x * ngroups;
  const int waves = gridDim.y * (GT / 64), wave = blockIdx.y * (GT / 64) + (threadIdx.x >> 6);
  group_max<GSEG>(x, V, gs, wave, waves, [&](int g, uint32_t m) { out[g] = m; });
}

// Inclusive prefix sum of the first n <= CAND floats of a[0] (Hillis-Steele,
// fixed order), between the two arrays in turn. Returns the one with the sums.
__device__ const float* prefix_sum(float (*a)[CAND], int n) {
  int from = 0;
  for (int off = 1; off < n; off <<= 1, from ^= 1) {
    for (int i = threadIdx.x; i < n; i += ST) a[from ^ 1][i] = i >= off ? a[from][i] + a[from][i - off] : a[from][i];
    __syncthreads();
  }
  return a[from];
}

// Key ranges: range (key - from) >> shift, below BINS for every key in [from, to].
__device__ __forceinline__ int bin_shift(uint32_t from, uint32_t to) {
  const uint32_t w = to - from;
  const int bits = w ? 32 - __builtin_clz(w) : 0;
  return bits > 11 ? bits - 11 : 0;
}
static_assert(BINS == 1 << 11 && BINS == 2 * ST, "two ranges per thread");

// L.hist from counts per range (range r's count at BINS - 1 - r: descending keys)
// to the number of entries in higher ranges. f(i, before, count) is called for
// this thread's two places i. A barrier before it and after it included.
template <class F>
__device__ __forceinline__ void scan_bins(SLds& L, F&& f) {
  const int t = threadIdx.x, wave = t >> 6;
  __syncthreads();
  const uint32_t c0 = L.hist[2 * t], c1 = L.hist[2 * t + 1];
  const uint32_t incl = wave_incl_scan(c0 + c1);
  if ((t & 63) == 63) L.cnt[0][wave] = incl;
  __syncthreads();
  uint32_t before = incl - c0 - c1;
#pragma unroll
  for (int w = 0; w < ST / 64; ++w) before += w < wave ? L.cnt[0][w] : 0u;
  L.hist[2 * t] = before;
  L.hist[2 * t + 1] = before + c0;
  f(2 * t, before, c0);
  f(2 * t + 1, before + c0, c1);
  __syncthreads();
}

// Descending bitonic sort of the first `size` (a power of two, >= 2) entries of
// cand; every thread takes part, a barrier before it and after it included.
// The 64 compare-exchanges of a wave cover 128 consecutive entries while the
// stride is at most 64, so only the wider steps need the workgroup's barrier
// (LDS accesses of one wave complete in order): 14 barriers instead of 66 for
// 2048 entries.
__device__ void sort_desc(unsigned long long* cand, int size) {
  __syncthreads();
  for (int len = 2; len <= size; len <<= 1) {
    for (int stride = len >> 1; stride > 0; stride >>= 1) {
      for (int i = threadIdx.x; i < size / 2; i += ST) {
        const int lo = 2 * i - (i & (stride - 1)), hi = lo + stride;
        const bool desc = (lo & len) == 0;
        const unsigned long long a = cand[lo], b = cand[hi];
        if ((a < b) == desc) {
          cand[lo] = b;
          cand[hi] = a;
        }
      }
      const int next = stride > 1 ? stride >> 1 : len;   // the next step's stride
      if (stride > 64 || next > 64) __syncthreads();
      else asm volatile("" ::: "memory");
    }
  }
  __syncthreads();
}

// Sum over the workgroup of the count of v >= t among each thread's NG keys
// (slot: 0 or 1, alternating between calls, so one barrier serves each).
__device__ __forceinline__ uint32_t count_ge(const uint32_t (&v)[NG], uint32_t t, SLds& L, int slot) {
  uint32_t c = 0u;
#pragma unroll
  for (int j = 0; j < NG; ++j) c += (uint32_t)__popcll(__ballot(v[j] >= t));
  if ((threadIdx.x & 63) == 0) L.cnt[slot][threadIdx.x >> 6] = c;
  __syncthreads();
  uint32_t s = 0u;
#pragma unroll
  for (int w = 0; w < ST / 64; ++w) s += L.cnt[slot][w];
  return s;
}

// The candidates of a row's top k in L.cand (L.ncand of them, unsorted; all
// logits at or above the k-th largest unless more than CAND tie with it), from
// the group maxima gm (NG per thread: groups threadIdx.x + j * ST, 0 past the
// last; at least k groups); low and top: keys no candidate is below or above.
// False: they do not fit, L.cand holds nothing of use; at least k logits reach low.
__device__ bool gather_top(const float* x, int V, int gs, int ngroups, int k, const uint32_t (&gm)[NG], SLds& L,
                           uint32_t& low, uint32_t& top) {
  const int t = threadIdx.x, wave = t >> 6;
  uint32_t inv = 0u, mx = 0u;   // (inv: the largest of ~key, for the smallest key)
#pragma unroll
  for (int j = 0; j < NG; ++j)
    if (t + j * ST < ngroups) {
      inv = umax(inv, ~gm[j]);
      mx = umax(mx, gm[j]);
    }
  inv = wave_max(inv);
  mx = wave_max(mx);
  if ((t & 63) == 0) {
    L.wmin[wave] = inv;
    L.wmax[wave] = mx;
  }
  if (t == 0) L.ncand = L.ngl = 0u;
  L.hist[t] = L.hist[t + ST] = 0u;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < ST / 64; ++w) {
    inv = umax(inv, L.wmin[w]);
    mx = umax(mx, L.wmax[w]);
  }
  const uint32_t mn = ~inv;
  top = mx;
  const int sh = bin_shift(mn, mx);
#pragma unroll
  for (int j = 0; j < NG; ++j)
    if (t + j * ST < ngroups) atomicAdd(&L.hist[BINS - 1 - ((gm[j] - mn) >> sh)], 1u);
  scan_bins(L, [&](int i, uint32_t before, uint32_t count) {
    if (before < (uint32_t)k && before + count >= (uint32_t)k) {
      L.bin = BINS - 1 - i;
      L.at_bin = (int)(before + count);
    }
  });
  // lo: a key at least k maxima reach; hi: one that fewer than k reach (the
  // edges of the range that holds the k-th maximum). Bisected further until lo
  // is reached by few more than k (or exactly, lo + 1 == hi: then the maxima
  // tie at lo). Every thread follows the same values.
  const uint32_t enough = (uint32_t)k + (uint32_t)k / 16u + 64u;
  unsigned long long lo = (unsigned long long)mn + ((unsigned long long)L.bin << sh), hi = lo + (1ull << sh);
  if (hi > (unsigned long long)mx + 1ull) hi = (unsigned long long)mx + 1ull;
  uint32_t at_lo = (uint32_t)L.at_bin;
  for (int slot = 0; at_lo > enough && hi - lo > 1ull; slot ^= 1) {
    const unsigned long long mid = lo + (hi - lo) / 2ull;
    const uint32_t c = count_ge(gm, (uint32_t)mid, L, slot);
    if (c >= (uint32_t)k) {
      lo = mid;
      at_lo = c;
    } else {
      hi = mid;
    }
  }
  // with many maxima tied at lo, the logits above lo are gathered first (all
  // of them in fewer than k groups), then ties as far as they are kept
  const bool ties = at_lo > enough;
  const uint32_t L0 = (uint32_t)lo, first = ties ? (uint32_t)hi : L0;
  low = L0;
  auto list_groups = [&](uint32_t from, uint32_t below) {
#pragma unroll
    for (int j = 0; j < NG; ++j)
      if (t + j * ST < ngroups && gm[j] >= from && gm[j] <= below) {
        const uint32_t s = atomicAdd(&L.ngl, 1u);
        L.glist[s] = (uint16_t)(t + j * ST);
      }
  };
  const bool vec = aligned16(x);
  // logits with from <= key <= below of the listed groups, up to `most` entries in all
  auto gather = [&](uint32_t from, uint32_t below, uint32_t most) {
    const int lg = __builtin_ctz(gs) - 2, total = (int)L.ngl << lg;   // 2^lg 4-logit pieces per group
    for (int w = t; w < total; w += ST) {
      if (*(volatile uint32_t*)&L.ncand >= most) break;
      const int i = (int)L.glist[w >> lg] * gs + (w & ((1 << lg) - 1)) * 4;
      uint32_t kx[4];
      keys4(x, i, V, vec, kx);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (i + e < V && kx[e] >= from && kx[e] <= below) {
          const uint32_t s = atomicAdd(&L.ncand, 1u);
          if (s < most && s < (uint32_t)SORT)
            L.cand[s] = ((unsigned long long)kx[e] << 32) | (0xffffffffu - (uint32_t)(i + e));
        }
    }
  };
  list_groups(first, 0xffffffffu);
  __syncthreads();
  gather(first, 0xffffffffu, SORT + 1u);
  __syncthreads();
  if (L.ncand > (uint32_t)SORT) {   // (so more than k logits reach `first`)
    low = first;
    return false;
  }
  if (ties && L.ncand < (uint32_t)k) {   // the k-th largest logit is lo itself
    list_groups(L0, L0);                 // (behind the groups above lo, which may hold ties too)
    __syncthreads();
    gather(L0, L0, (uint32_t)CAND);
    __syncthreads();
    if (t == 0 && L.ncand > (uint32_t)CAND) L.ncand = (uint32_t)CAND;
    __syncthreads();
  }
  return true;
}

// The same by an exact radix select over the whole row: 4 passes of 8-bit count
// histograms over the keys find the k-th largest, then the logits above it and
// as many ties as there is room for are gathered. At least k keys reach `from`;
// those below it are not counted (the histogram's atomics on the one or two
// ranges that hold most of a row are what takes the time: a mask that leaves
// 5000 logits side by side, top-k 1024: 265 -> 160 us, sorted logits 287 -> 184).
__device__ void radix_top(const float* x, int V, int k, uint32_t from, SLds& L) {
  const int t = threadIdx.x;
  if (t == 0) {
    L.prefix = 0u;
    L.need = (uint32_t)k;
    L.ncand = L.nties = 0u;
  }
  uint32_t mask = 0u;
  for (int shift = 24; shift >= 0; shift -= 8) {
    for (int i = t; i < 256; i += ST) L.hist[i] = 0u;
    __syncthreads();
    const uint32_t prefix = L.prefix;
    for (int i = t; i < V; i += ST) {
      const uint32_t kx = okey(x[i]);
      if (kx >= from && (kx & mask) == prefix) atomicAdd(&L.hist[(kx >> shift) & 255u], 1u);
    }
    __syncthreads();
    if (t == 0) {
      uint32_t cum = 0u, need = L.need;
      int d = 255;
      for (; d > 0; --d) {
        if (cum + L.hist[d] >= need) break;
        cum += L.hist[d];
      }
      L.need = need - cum;
      L.prefix = prefix | ((uint32_t)d << shift);
    }
    mask |= 255u << shift;
    __syncthreads();
  }
  const uint32_t thr = L.prefix, above = (uint32_t)k - L.need;   // key of the k-th largest logit, and how many are above it
  for (int i = t; i < V; i += ST) {
    const uint32_t kx = okey(x[i]);
    if (kx < thr) continue;
    const uint32_t s = kx > thr ? atomicAdd(&L.ncand, 1u) : above + atomicAdd(&L.nties, 1u);
    if (s < (uint32_t)CAND) L.cand[s] = ((unsigned long long)kx << 32) | (0xffffffffu - (uint32_t)i);
  }
  __syncthreads();
  if (t == 0) L.ncand = above + L.nties < (uint32_t)CAND ? above + L.nties : (uint32_t)CAND;
  __syncthreads();
}

// The first n candidates of L.cand, all keys in [low, top], in descending order.
// Each goes to its key range (the higher ranges' entries before it, in any order
// within the range), then to its place there by counting the larger ones of the
// range: entries are distinct, so the order is one. 2048 ranges hold at most a
// few each, unless the keys are crowded: ties, one far outlier, or logits of both
// signs (a row sorted whole, up to SORT logits; between 2 and -2 lie as many keys as
// beyond them). Then the bitonic sort: 4096 logits 38 us in all.
__device__ void sort_cand(int n, uint32_t low, uint32_t top, SLds& L) {
  const int t = threadIdx.x, sh = bin_shift(low, top);
  L.hist[t] = L.hist[t + ST] = 0u;
  if (t == 0) L.crowded = 0u;
  __syncthreads();
  unsigned long long c[SORT / ST];
  uint32_t place[SORT / ST];
#pragma unroll
  for (int j = 0; j < SORT / ST; ++j) {
    const int i = t + j * ST;
    if (i < n) {
      c[j] = L.cand[i];
      place[j] = atomicAdd(&L.hist[BINS - 1 - (((uint32_t)(c[j] >> 32) - low) >> sh)], 1u);
    }
  }
  scan_bins(L, [&](int, uint32_t, uint32_t count) {
    if (count > CROWD) L.crowded = 1u;
  });
  if (L.crowded) {
    int size = 2;
    while (size < n) size <<= 1;
    for (int i = n + t; i < size; i += ST) L.cand[i] = 0ull;
    sort_desc(L.cand, size);
    return;
  }
#pragma unroll
  for (int j = 0; j < SORT / ST; ++j)
    if (t + j * ST < n) L.tmp[L.hist[BINS - 1 - (((uint32_t)(c[j] >> 32) - low) >> sh)] + place[j]] = c[j];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < SORT / ST; ++j)
    if (t + j * ST < n) {
      const int b = BINS - 1 - (int)(((uint32_t)(c[j] >> 32) - low) >> sh);
      const int i0 = (int)L.hist[b], i1 = b + 1 < BINS ? (int)L.hist[b + 1] : n;
      int at = i0;
      for (int i = i0; i < i1; ++i) at += L.tmp[i] > c[j] ? 1 : 0;
      L.cand[at] = c[j];
    }
  __syncthreads();
}

// gmax: the rows' group maxima (mk_group_max_kernel), or null: the workgroup
// finds its row's itself.
__global__ void __launch_bounds__(ST) mk_sample_kernel(SParams p, const uint32_t* gmax, int gs) {
  __shared__ SLds L;
  const int row = blockIdx.x, t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const float* x = p.logits + (size_t)row * p.stride;
  const float pk = p.params[row * 3 + 0], pp = p.params[row * 3 + 1], temp = p.params[row * 3 + 2];
  const int V = p.vocab, ngroups = gs ? (V + gs - 1) / gs : 0;
  const uint32_t ctr = p.counter ? (uint32_t)p.counter[row] : 0u;
  int k = (int)pk;
  const bool greedy = k == 1 || !(temp > 0.f);
  if (k <= 0 || k > MAXK) k = MAXK;
  if (k > V) k = V;

  uint32_t gm[NG];
#pragma unroll
  for (int j = 0; j < NG; ++j) gm[j] = 0u;
  if (gs && (gmax || !greedy)) {
    const uint32_t* src = gmax + (size_t)row * ngroups;
    if (!gmax) {   // into the sort's LDS, not in use yet
      uint32_t* own = reinterpret_cast<uint32_t*>(L.tmp);
      static_assert(MAX_GROUPS * sizeof(uint32_t) <= sizeof(L.tmp), "group maxima in LDS");
      const int nseg = (V + 255) / 256, nw = ST / 64;
      auto put = [&](int g, uint32_t m) { own[g] = m; };
      if (nseg <= 4 * nw) group_max<4>(x, V, gs, wave, nw, put);
      else if (nseg <= 8 * nw) group_max<8>(x, V, gs, wave, nw, put);
      else
        for (int s0 = wave; s0 < nseg; s0 += 16 * nw) group_max<16>(x, V, gs, s0, nw, put);
      __syncthreads();
#pragma unroll
      for (int j = 0; j < NG; ++j)
        if (t + j * ST < ngroups) gm[j] = own[t + j * ST];
      __syncthreads();
    } else {
#pragma unroll
      for (int j = 0; j < NG; ++j)
        if (t + j * ST < ngroups) gm[j] = src[t + j * ST];
    }
  }

  if (greedy) {   // argmax, lowest index on ties
    unsigned long long b = 0xffffffffull;   // key 0 (NaN), index 0
    auto take = [&](uint32_t key, int i) {
      const unsigned long long kv = ((unsigned long long)key << 32) | (0xffffffffu - (uint32_t)i);
      b = kv > b ? kv : b;
    };
    if (gmax) {   // the first group with the largest maximum, by its first index
#pragma unroll
      for (int j = 0; j < NG; ++j)
        if (t + j * ST < ngroups) take(gm[j], (t + j * ST) * gs);
    } else {
      const bool vec = aligned16(x);
      for (int i = 4 * t; i < V; i += 4 * ST) {
        uint32_t kx[4];
        keys4(x, i, V, vec, kx);
#pragma unroll
        for (int e = 0; e < 4; ++e) take(kx[e], i + e);   // (past the row: key 0, behind index 0's)
      }
    }
    for (int o = 32; o >= 1; o >>= 1) {
      const unsigned long long v = __shfl_xor(b, o, 64);
      b = v > b ? v : b;
    }
    if (lane == 0) L.best[wave] = b;
    __syncthreads();
    if (wave == 0) {
      unsigned long long m = L.best[0];
      for (int w = 1; w < ST / 64; ++w) m = L.best[w] > m ? L.best[w] : m;
      int at = (int)(0xffffffffu - (uint32_t)(m & 0xffffffffull));
      if (gmax) {   // the first logit of that group with its maximum
        const uint32_t best = (uint32_t)(m >> 32);
        for (int o = 0; o < gs; o += 64) {
          const int i = at + o + lane;
          const unsigned long long hit = __ballot(o + lane < gs && i < V && okey(x[i]) == best);
          if (hit) {
            at += o + (int)__ffsll(hit) - 1;
            break;
          }
        }
      }
      if (lane == 0) {
        p.tokens[row] = at;
        if (p.uniforms) p.uniforms[row] = -1.f;
      }
    }
    return;
  }

  // the candidates of the top k in L.cand
  uint32_t low = 0u, top = 0xffffffffu;
  if (!gs && V <= SORT) {
    for (int i = t; i < V; i += ST) L.cand[i] = ((unsigned long long)okey(x[i]) << 32) | (0xffffffffu - (uint32_t)i);
    if (t == 0) L.ncand = (uint32_t)V;
    __syncthreads();
  } else if (!gs || !gather_top(x, V, gs, ngroups, k, gm, L, low, top)) {
    const uint32_t from = low;   // (gather_top's, or 0)
    low = 0u;
    top = 0xffffffffu;
    __syncthreads();
    radix_top(x, V, k, from, L);
  }
  // sorted descending (key, then ascending index); the k-th and its ties are kept
  const int nc = (int)L.ncand;
  sort_cand(nc, low, top, L);
  const uint32_t thr = (uint32_t)(L.cand[k - 1] >> 32);
  for (int i = k - 1 + t; i < nc; i += ST)
    if ((uint32_t)(L.cand[i] >> 32) == thr && (i + 1 == nc || (uint32_t)(L.cand[i + 1] >> 32) != thr)) L.n = i + 1;
  __syncthreads();
  const int n = L.n < CAND ? L.n : CAND;

  // softmax numerators in sorted order, prefix sums, nucleus cut, draw
  const float m = key_to_float((uint32_t)(L.cand[0] >> 32)) / temp;
  for (int i = t; i < n; i += ST) L.csum[0][i] = __expf(key_to_float((uint32_t)(L.cand[i] >> 32)) / temp - m);
  if (t == 0) L.nkeep = 0;
  __syncthreads();
  const float* csum = prefix_sum(L.csum, n);
  const float Z = csum[n - 1];
  // kept: position 0, and j >= 1 while csum[j-1] < top_p * Z
  const float cut = (pp > 0.f && pp < 1.f) ? pp * Z : 2.f * Z;
  int mine = 0;
#pragma unroll
  for (int j = 0; j < CAND / ST; ++j) {
    const int i = t + j * ST;
    mine += __popcll(__ballot(i < n && (i == 0 || csum[i - 1] < cut)));
  }
  if (lane == 0 && mine) atomicAdd(&L.nkeep, mine);
  __syncthreads();
  const int nkeep = L.nkeep;
  const uint32_t w = philox_first(ctr, (uint32_t)row, 0u, 0u, (uint32_t)p.seed, (uint32_t)(p.seed >> 32));
  const float u = (float)(w >> 8) * (1.0f / 16777216.0f);
  const float target = u * csum[nkeep - 1];
  if (t == 0) L.pick = nkeep - 1;   // target at the very top (rounding): the last kept token
  __syncthreads();
  // the first j with csum[j] > target: csum is nondecreasing, so exactly one j has
  // csum[j] > target >= csum[j-1]
  for (int j = t; j < nkeep; j += ST)
    if (csum[j] > target && (j == 0 || !(csum[j - 1] > target))) L.pick = j;
  __syncthreads();
  if (t == 0) {
    p.tokens[row] = (int32_t)(0xffffffffu - (uint32_t)(L.cand[L.pick] & 0xffffffffull));
    if (p.uniforms) p.uniforms[row] = u;
  }
}

thread_local char s_msg[256] = "";

}  // namespace

extern "C" {

const char* mk_sample_last_error(void) { return s_msg; }

size_t mk_sample_scratch_bytes(int32_t batch, int32_t vocab) {
  const int gs = vocab > SOLO ? group_size(vocab) : 0;
  return gs && batch > 0 ? (size_t)batch * ((vocab + gs - 1) / gs) * sizeof(uint32_t) : 0;
}

int mk_sample(const mk_sample_args* a) { return mk_sample_with_scratch(a, nullptr, 0); }

int mk_sample_with_scratch(const mk_sample_args* a, void* scratch, size_t scratch_bytes) {
  if (!a || !a->logits || !a->params || !a->tokens_out) {
    strcpy(s_msg, "args, logits, params or tokens_out is NULL");
    return MK_ERR_NULL;
  }
  if (a->batch < 1 || a->vocab < 1 || a->vocab_stride < a->vocab) {
    strcpy(s_msg, "batch >= 1, vocab >= 1 and vocab_stride >= vocab required");
    return MK_ERR_SHAPE;
  }
  if (scratch && (scratch_bytes < mk_sample_scratch_bytes(a->batch, a->vocab) ||
                  (reinterpret_cast<uintptr_t>(scratch) & 3u))) {
    strcpy(s_msg, "scratch smaller than mk_sample_scratch_bytes, or not 4-byte aligned");
    return MK_ERR_WORKSPACE;
  }
  SParams p;
  p.logits = a->logits;
  p.params = a->params;
  p.counter = a->counter;
  p.tokens = a->tokens_out;
  p.uniforms = a->uniforms_out;
  p.seed = a->seed;
  p.vocab = a->vocab;
  p.stride = a->vocab_stride;
  hipStream_t st = static_cast<hipStream_t>(a->stream);
  const int gs = group_size(a->vocab);
  uint32_t* gmax = gs && a->vocab > SOLO ? static_cast<uint32_t*>(scratch) : nullptr;
  if (gmax) {
    const int nseg = (a->vocab + 255) / 256, per = GSEG * (GT / 64);
    hipLaunchKernelGGL(mk_group_max_kernel, dim3(a->batch, (nseg + per - 1) / per), dim3(GT), 0, st, a->logits,
                       a->vocab, a->vocab_stride, gs, gmax, (a->vocab + gs - 1) / gs);
  }
  hipLaunchKernelGGL(mk_sample_kernel, dim3(a->batch), dim3(ST), 0, st, p, (const uint32_t*)gmax, gs);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    strncpy(s_msg, hipGetErrorString(e), sizeof(s_msg) - 1);
    return MK_ERR_HIP;
  }
  return MK_OK;
}

}  // extern "C"
