// Token top-k from blocks of bf16 scores: the selection half of the non-lazy DINO-feature path.
//
// ref: saf3r/patch/utils.py:54-184 (compute_qk_topk_indices_batched: per-frame torch.topk of bf16
//      q.k scores, optional exclusion of frame 0 with strided first-frame samples prepended, and a
//      cap on the number of kept keys), saf3r/patch/patch_vggt.py:313-357 (its caller).
//
// Scores are bf16 bit patterns; a key is ranked by the score, ties go to the lower key index. The
// 16-bit order key of a score is its sortable transform (larger score -> larger key, -0 < +0).
//   frame stage: one wave per (row, frame) holds the frame's scores in registers, finds the k-th
//                largest order key with wave-wide counts, and writes the k keys in increasing key order;
//   cap stage:   one work-group per row takes the best `cap` of a candidate list (the frame stage's
//                output, or every key of the row when selection is not per frame) the same way,
//                in list order, which is increasing key order.
#include <cmath>
#include <type_traits>

#include "common.h"

namespace saf3r {

typedef short s16x2 __attribute__((ext_vector_type(2)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

constexpr int kMaxPerFrame = 4096;  // frame stage: at most 33 words of two keys per lane

struct FrameTopkParams {
  const uint16_t* scores;
  int64_t srs;        // score row stride (elements)
  int rows, F, P, f0;  // f0: first frame selected from (1 excludes frame 0)
  int k;              // keys per frame
  int32_t* out;       // frame stage output (idx or candidate list)
  int64_t ors;        // its row stride
  int ocol;           // first column written
  int lanes;          // lane maxima the first threshold guess aims at
  int window;         // whether a threshold with k .. kCands keys is searched for (see frame_window)
  uint16_t* okey;     // candidate order keys (cap stage input), row stride ors, or null
};

struct CapParams {
  const uint16_t* scores;  // dense mode: the score rows
  int64_t srs;
  int64_t dense_base;      // dense mode: first key, dense_n: key count
  int64_t dense_n;
  const int32_t* cidx;     // list mode: candidate keys and their order keys
  const uint16_t* ckey;
  int64_t crs;
  int64_t n;               // list mode: candidates per row
  int rows, cap;
  int32_t* out;
  int64_t ors;
  int ocol;
};

__device__ inline uint32_t sortable16(uint16_t b) { return (uint32_t)(b ^ ((b & 0x8000u) ? 0xFFFFu : 0x8000u)); }

// Byte-histogram step of a radix select over keys held by the caller: counts[256] in LDS; returns
// the bin holding the rank-`need` largest key and, through above, the number of keys above it.
template <int NT>
__device__ inline int radix_bin(uint32_t* counts, int need, int* above, int lane, uint32_t* scan) {
  // NT threads cooperate; thread t owns bins 256 - (t + 1) * (256 / NT) .. (from the top)
  constexpr int per = 256 / NT;
  uint32_t s = 0;
#pragma unroll
  for (int i = 0; i < per; ++i) s += counts[255 - (lane * per + i)];
  scan[lane] = s;
  __syncthreads();
  // exclusive prefix over threads from the top (small: NT <= 256)
  uint32_t pre = 0;
  for (int t = 0; t < lane; ++t) pre += scan[t];
  int bin = -1, ab = 0;
  if ((int)pre < need && (int)(pre + s) >= need) {
    uint32_t acc = pre;
#pragma unroll
    for (int i = 0; i < per; ++i) {
      const uint32_t c = counts[255 - (lane * per + i)];
      if ((int)(acc + c) >= need) {
        bin = 255 - (lane * per + i);
        ab = (int)acc;
        break;
      }
      acc += c;
    }
  }
  __syncthreads();
  if (bin >= 0) {
    scan[0] = (uint32_t)bin;
    scan[1] = (uint32_t)ab;
  }
  __syncthreads();
  *above = (int)scan[1];
  const int b = (int)scan[0];
  __syncthreads();
  return b;
}

// base + the set lanes of m below this one
__device__ __forceinline__ int lanes_before(uint64_t m, int base) {
  return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, (uint32_t)base));
}

// x over the wave by DPP within rows of 16 lanes and the row / half swaps, as a wave-uniform value
template <typename Op>
__device__ __forceinline__ uint32_t wave_reduce_u32(uint32_t x, Op op) {
  auto mov = [](uint32_t y, auto ctl) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)y, decltype(ctl)::value, 0xF, 0xF, true);
  };
  x = op(x, mov(x, std::integral_constant<int, 0xB1>{}));   // quad_perm [1, 0, 3, 2]
  x = op(x, mov(x, std::integral_constant<int, 0x4E>{}));   // quad_perm [2, 3, 0, 1]
  x = op(x, mov(x, std::integral_constant<int, 0x141>{}));  // mirror of 8
  x = op(x, mov(x, std::integral_constant<int, 0x128>{}));  // rotation by 8 of 16
  const auto a = __builtin_amdgcn_permlane16_swap(x, x, false, false);
  x = op((uint32_t)a[0], (uint32_t)a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(x, x, false, false);
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)op((uint32_t)b[0], (uint32_t)b[1]));
}

// ---- frame stage, k <= 4 in short frames: four waves, one (row, frame) each ----
// Every lane keeps the four best of its keys as composites (order key << 16 | 0xFFFF - position: larger is
// better, equal scores by the lower position; 0 for none), descending; six exchanges merge the lists of
// the wave, and the k winners are written in increasing key order. Bound by VALU issue.
// Frames of up to 1407 keys: there the lists beat the threshold search below (16384 rows x 8 frames, top-4, us,
// search / lists: 256 keys 79 / 40, 512 75 / 50, 1036 83 / 67, 1369 90 / 78; five different scores
// 63 / 40, 67 / 49, 104 / 67, 114 / 78), beyond they would hold more words than they save.
constexpr int kListMax = 4;
constexpr int kListWords = 11;  // per lane
__device__ __forceinline__ void list_sort(uint32_t (&c)[kListMax]) {  // a bitonic list, descending
  const uint32_t a = max(c[0], c[2]), b = max(c[1], c[3]), d = min(c[0], c[2]), e = min(c[1], c[3]);
  c[0] = max(a, b);
  c[1] = min(a, b);
  c[2] = max(d, e);
  c[3] = min(d, e);
}

template <int NR, int NF>
__global__ __launch_bounds__(256) void frame_list_kernel(FrameTopkParams p) {
  const int lane = tid_x() & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid_x() >> 6);
  const int row = bid_y();
  const int fs = bid_x() * 4 + w;  // selected-frame index
  if (fs >= p.F - p.f0) return;
  const int64_t s0 = (int64_t)(p.f0 + fs) * p.P;  // first key of the frame in the row
  const int off = (int)(s0 & 1);                  // the span starts at the word of key s0
  const uint32_t* words = reinterpret_cast<const uint32_t*>(p.scores + (int64_t)row * p.srs + (s0 - off));
  const int last = (off + p.P - 1) >> 1;          // last word with a key of the frame
  const int k = p.k;
  uint32_t key[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) key[r] = words[r < NF ? lane + 64 * r : min(lane + 64 * r, last)];
  uint32_t c[kListMax] = {0, 0, 0, 0};
  const int j0 = 2 * lane - off;
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const s16x2 b = __builtin_bit_cast(s16x2, key[r]);
    key[r] ^= __builtin_bit_cast(uint32_t, b >> (short)15) | 0x80008000u;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint32_t j = (uint32_t)(j0 + 128 * r + h);
      uint32_t y = (h ? key[r] & 0xFFFF0000u : key[r] << 16) | (0xFFFFu - j);
      if ((r == 0 && h == 0) || r >= NF - 1)  // other positions are inside the frame
        y = j < (uint32_t)p.P ? y : 0u;
#pragma unroll
      for (int i = kListMax - 1; i > 0; --i) c[i] = max(c[i], min(c[i - 1], y));
      c[0] = max(c[0], y);
    }
  }
  auto merge = [&](const uint32_t (&x)[kListMax], const uint32_t (&y)[kListMax]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kListMax; ++i) c[i] = max(x[i], y[kListMax - 1 - i]);
    list_sort(c);
  };
  auto step = [&](auto ctl) __attribute__((always_inline)) {
    uint32_t x[kListMax], y[kListMax];
#pragma unroll
    for (int i = 0; i < kListMax; ++i) {
      x[i] = c[i];
      y[i] = (uint32_t)__builtin_amdgcn_mov_dpp((int)c[i], decltype(ctl)::value, 0xF, 0xF, true);
    }
    merge(x, y);
  };
  step(std::integral_constant<int, 0xB1>{});   // quad_perm [1, 0, 3, 2]
  step(std::integral_constant<int, 0x4E>{});   // quad_perm [2, 3, 0, 1]
  step(std::integral_constant<int, 0x141>{});  // mirror of 8
  step(std::integral_constant<int, 0x128>{});  // rotation by 8 of 16
  uint32_t x[kListMax], y[kListMax];
#pragma unroll
  for (int i = 0; i < kListMax; ++i) {
    const auto s = __builtin_amdgcn_permlane16_swap(c[i], c[i], false, false);
    x[i] = s[0];
    y[i] = s[1];
  }
  merge(x, y);
#pragma unroll
  for (int i = 0; i < kListMax; ++i) {
    const auto s = __builtin_amdgcn_permlane32_swap(c[i], c[i], false, false);
    x[i] = s[0];
    y[i] = s[1];
  }
  merge(x, y);
  // lane i < k: winner i, written behind the winners of lower positions
  uint32_t mine = 0;
#pragma unroll
  for (int i = 0; i < kListMax; ++i)
    if (i == lane) mine = c[i];
  int rank = 0;
#pragma unroll
  for (int i = 0; i < kListMax; ++i) rank += i < k && (c[i] & 0xFFFFu) > (mine & 0xFFFFu) ? 1 : 0;
  if (lane < k) {
    const int64_t at = (int64_t)row * p.ors + (int64_t)fs * k + rank;
    p.out[at + p.ocol] = (int32_t)(s0 + (0xFFFFu - (mine & 0xFFFFu)));
    if (p.okey) p.okey[at] = (uint16_t)(mine >> 16);
  }
}

// ---- frame stage: four waves, one (row, frame) each ----
// A lane holds NR words of two scores: word lane + 64 r of the frame's span, so element order (r,
// lane, half) is increasing key order. Words up to NF are whole (the caller picks NR by the frame's
// length); positions outside the frame hold order key 0, which no threshold of the search counts
// (its thresholds are >= 1; a real key 0, the lowest, only matters at threshold 0).
//   1. A threshold with k .. kCands keys at or above it: a first guess from the lanes' largest keys
//      (one compare and ballot per bisection step), then counts of all keys until one falls into
//      the window, mostly one or two. A count is one compare per key (the upper half of a word
//      compares as the word) and scalar adds.
//   2. Those candidates, (order key, position) in one word, into LDS in key order, two per lane.
//   3. The exact k-th key by bisection over the candidates, and the k kept ones written out in key
//      order, equal keys lowest first.
// A row whose counts jump over the window (many equal scores) takes every key above the one they jump at
// and the first of those equal to it. Without a window (frame_window): the exact threshold over all keys.
// Bound by VALU issue (the loads alone would take half the time): about 260 instructions per row and
// frame of 1036 keys at k = 64. It replaced one bisection over unpacked keys (24 registers for 1036
// keys, 9 rounds of two instructions per key): 4096 rows x 32 frames x 1036 keys, top-64 279 -> 97 us,
// 128 x 1369 keys 1070 -> 392 us.
constexpr int kCands = 128;
template <int NR, int NF>
__global__ __launch_bounds__(256) void frame_select_kernel(FrameTopkParams p) {
  __shared__ uint32_t cands[4][kCands];
  const int lane = tid_x() & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid_x() >> 6);
  const int row = bid_y();
  const int nfr = p.F - p.f0;
  const int fs = bid_x() * 4 + w;  // selected-frame index
  if (fs >= nfr) return;              // whole wave: no work-group barrier below
  const int64_t s0 = (int64_t)(p.f0 + fs) * p.P;  // first key of the frame in the row
  const int off = (int)(s0 & 1);                  // the span starts at the word of key s0
  const uint32_t* words = reinterpret_cast<const uint32_t*>(p.scores + (int64_t)row * p.srs + (s0 - off));
  const int last = (off + p.P - 1) >> 1;          // last word with a key of the frame
  const int k = p.k;
  uint32_t key[NR];  // order keys: larger score -> larger key
#pragma unroll
  for (int r = 0; r < NR; ++r) key[r] = words[r < NF ? lane + 64 * r : min(lane + 64 * r, last)];
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    if (r >= NF - 1) {
      if (lane + 64 * r > last) key[r] = 0xFFFFFFFFu;  // bits 0xFFFF: order key 0
      if (lane + 64 * r == last && ((off + p.P) & 1)) key[r] |= 0xFFFF0000u;
    }
    if (r == 0 && off && lane == 0) key[0] |= 0xFFFFu;
    const s16x2 b = __builtin_bit_cast(s16x2, key[r]);
    key[r] ^= __builtin_bit_cast(uint32_t, b >> (short)15) | 0x80008000u;
  }
  auto count_ge = [&](uint32_t t) {  // keys >= t (1 <= t <= 0xFFFF), wave-wide
    int c = 0;
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      c += __popcll(__builtin_amdgcn_ballot_w64((uint16_t)key[r] >= (uint16_t)t));
      c += __popcll(__builtin_amdgcn_ballot_w64(key[r] >= (t << 16)));
    }
    return c;
  };
  int32_t* o = p.out + (int64_t)row * p.ors + p.ocol + (int64_t)fs * k;
  uint16_t* ok = p.okey ? p.okey + (int64_t)row * p.ors + (int64_t)fs * k : nullptr;
  u16x2 mx = __builtin_bit_cast(u16x2, key[0]);
#pragma unroll
  for (int r = 1; r < NR; ++r) mx = __builtin_elementwise_max(mx, __builtin_bit_cast(u16x2, key[r]));
  const uint32_t lmax = max((uint32_t)mx[0], (uint32_t)mx[1]);
  const uint32_t top = wave_reduce_u32(lmax, [](uint32_t a, uint32_t b) { return max(a, b); });
  uint32_t t = 1;
  uint32_t thr = 0;  // the k-th largest key, where the counts jump over the window at it (0: the lowest key)
  int n = -1;
  if (p.window) {
    if (p.P > kCands) {
      uint32_t a = 1, b = top;
      t = wave_reduce_u32(lmax, [](uint32_t x, uint32_t y) { return min(x, y); });
      if (k <= 64) a = max(t, 1u);  // every lane's largest key reaches it
      t = (a + b + 1) >> 1;
      for (uint32_t x = a, y = b; x < y;) {
        const int c = __popcll(__builtin_amdgcn_ballot_w64(lmax >= t));
        if (c > p.lanes + 2) x = t;
        else if (c < p.lanes - 2) y = t - 1;
        else break;
        t = (x + y + 1) >> 1;
      }
      // count(a) >= k unless a = 1; stops with a = b where the counts jump over the window
      for (;;) {
        const int c = count_ge(t);
        if (c >= k && c <= kCands) {
          n = c;
          break;
        }
        if (c < k) b = t - 1;
        else a = t;
        if (a >= b) {  // the one threshold left
          const int ca = a == t ? c : count_ge(a);
          if (ca >= k && ca <= kCands) {
            n = ca;
            t = a;
          } else if (ca >= k) {
            thr = a;  // count(a + 1) < k
          }
          break;
        }
        t = (a + b + 1) >> 1;
      }
    } else {
      n = count_ge(1);
      if (n < k) n = -1;  // the k-th key is the lowest order key, which counts leave out
    }
  }
  if (n >= 0) {
    uint32_t* cw = cands[w];
    const int j0 = 2 * lane - off;
    int base = 0;
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const bool h0 = (uint16_t)key[r] >= (uint16_t)t, h1 = key[r] >= (t << 16);
      const uint64_t m0 = __builtin_amdgcn_ballot_w64(h0), m1 = __builtin_amdgcn_ballot_w64(h1);
      const int at = lanes_before(m1, lanes_before(m0, base));
      if (h0) cw[at] = (key[r] << 16) | (uint32_t)(j0 + 128 * r);
      if (h1) cw[at + (h0 ? 1 : 0)] = (key[r] & 0xFFFF0000u) | (uint32_t)(j0 + 128 * r + 1);
      base += __popcll(m0) + __popcll(m1);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const uint32_t x0 = lane < n ? cw[lane] : 0u, x1 = 64 + lane < n ? cw[64 + lane] : 0u;
    uint32_t lo = t, hi = top;  // count(lo) >= k
    int above = 0;                // keys above hi
    int c_lo = n;
    while (lo < hi && c_lo != k) {
      const uint32_t mid = (lo + hi + 1) >> 1;
      const int c = __popcll(__builtin_amdgcn_ballot_w64(x0 >= (mid << 16))) +
                    __popcll(__builtin_amdgcn_ballot_w64(x1 >= (mid << 16)));
      if (c >= k) {
        lo = mid;
        c_lo = c;
      } else {
        hi = mid - 1;
        above = c;
      }
    }
    // every candidate at or above lo, except the last of those equal to it where they are too many
    // (then the search ended with lo = hi, so that `above` counts the keys above lo)
    int skip_from = c_lo == k ? 0x7FFFFFFF : k - above;  // rank among the equal ones from which they drop out
    int out_base = 0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint32_t x = h ? x1 : x0;
      bool take = x >= (lo << 16);
      const uint64_t meq = __builtin_amdgcn_ballot_w64(take && (x >> 16) == lo);
      take = take && ((x >> 16) != lo || lanes_before(meq, 0) < skip_from);
      if (skip_from != 0x7FFFFFFF) skip_from -= (int)__popcll(meq);
      const uint64_t mt = __builtin_amdgcn_ballot_w64(take);
      const int at = lanes_before(mt, out_base);
      if (take) {
        o[at] = (int32_t)(s0 + (x & 0xFFFFu));
        if (ok) ok[at] = (uint16_t)(x >> 16);
      }
      out_base += __popcll(mt);
    }
    return;
  }
  // no window: the exact threshold over all keys, the largest t with at least k keys at or above it
  if (!p.window) {
#pragma unroll 1
    for (int bit = 15; bit >= 0; --bit) {
      const uint32_t c = thr | (1u << bit);
      if (count_ge(c) >= k) thr = c;
    }
  }
  int need = k - (thr < 0xFFFFu ? count_ge(thr + 1) : 0);  // keys equal to thr to keep, lowest first
  int base = 0;
  int ln = lane;
  asm volatile("" : "+v"(ln));  // positions formed here, not held through the search
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const int j = 2 * (ln + 64 * r) - off;  // position of the lower half
    const uint32_t k0 = key[r] & 0xFFFFu, k1 = key[r] >> 16;
    const bool in0 = (uint32_t)j < (uint32_t)p.P, in1 = (uint32_t)(j + 1) < (uint32_t)p.P;
    const bool e0 = in0 && k0 == thr, e1 = in1 && k1 == thr;
    const uint64_t me0 = __builtin_amdgcn_ballot_w64(e0), me1 = __builtin_amdgcn_ballot_w64(e1);
    const int rank = lanes_before(me1, lanes_before(me0, 0));
    const bool t0 = k0 > thr || (e0 && rank < need);
    const bool t1 = k1 > thr || (e1 && rank + (e0 ? 1 : 0) < need);
    const uint64_t m0 = __builtin_amdgcn_ballot_w64(t0), m1 = __builtin_amdgcn_ballot_w64(t1);
    const int at = lanes_before(m1, lanes_before(m0, base));
    if (t0) {
      o[at] = (int32_t)(s0 + j);
      if (ok) ok[at] = (uint16_t)k0;
    }
    if (t1) {
      o[at + (t0 ? 1 : 0)] = (int32_t)(s0 + j + 1);
      if (ok) ok[at + (t0 ? 1 : 0)] = (uint16_t)k1;
    }
    base += __popcll(m0) + __popcll(m1);
    need -= (int)(__popcll(me0) + __popcll(me1));
  }
}

// ---- cap stage: one work-group per row ----
__device__ inline void cap_item(const CapParams& p, int row, int64_t i, uint32_t* key, int32_t* idx) {
  if (p.cidx) {
    *idx = p.cidx[(int64_t)row * p.crs + i];
    *key = p.ckey[(int64_t)row * p.crs + i];
  } else {
    *idx = (int32_t)(p.dense_base + i);
    *key = sortable16(p.scores[(int64_t)row * p.srs + p.dense_base + i]);
  }
}

__global__ __launch_bounds__(256) void cap_select_kernel(CapParams p) {
  __shared__ uint32_t hist[256];
  __shared__ uint32_t scan[256];
  __shared__ uint32_t wsum[4];
  const int tid = tid_x(), lane = tid & 63, w = tid >> 6;
  const int row = bid_x();
  const int64_t n = p.cidx ? p.n : p.dense_n;
  const int m = p.cap;
  hist[tid] = 0;
  __syncthreads();
  for (int64_t i = tid; i < n; i += 256) {
    uint32_t k;
    int32_t x;
    cap_item(p, row, i, &k, &x);
    atomicAdd(&hist[k >> 8], 1u);
  }
  __syncthreads();
  int above1 = 0;
  const int b1 = radix_bin<256>(hist, m, &above1, tid, scan);
  hist[tid] = 0;
  __syncthreads();
  for (int64_t i = tid; i < n; i += 256) {
    uint32_t k;
    int32_t x;
    cap_item(p, row, i, &k, &x);
    if ((int)(k >> 8) == b1) atomicAdd(&hist[k & 255], 1u);
  }
  __syncthreads();
  int above2 = 0;
  const int b2 = radix_bin<256>(hist, m - above1, &above2, tid, scan);
  const uint32_t t = ((uint32_t)b1 << 8) | (uint32_t)b2;
  const int need_eq = m - above1 - above2;
  // ordered compaction over the list in chunks of 256 (block prefix of ballots)
  int base = 0, eq_seen = 0;
  int32_t* o = p.out + (int64_t)row * p.ors + p.ocol;
  for (int64_t c0 = 0; c0 < n; c0 += 256) {
    const int64_t i = c0 + tid;
    uint32_t k = 0;
    int32_t x = 0;
    const bool valid = i < n;
    if (valid) cap_item(p, row, i, &k, &x);
    const bool eq = valid && k == t;
    // rank of eq among the list's eq items before i
    const uint64_t me = __ballot(eq);
    const int in_wave_eq = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(me >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)me, 0));
    if (lane == 0) wsum[w] = __popcll(me);
    __syncthreads();
    int eq_before = eq_seen;
    for (int v = 0; v < w; ++v) eq_before += wsum[v];
    const int eq_tot = wsum[0] + wsum[1] + wsum[2] + wsum[3];
    __syncthreads();
    const bool sel = valid && (k > t || (eq && eq_before + in_wave_eq < need_eq));
    const uint64_t ms = __ballot(sel);
    const int in_wave = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(ms >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)ms, 0));
    if (lane == 0) wsum[w] = __popcll(ms);
    __syncthreads();
    int before = base;
    for (int v = 0; v < w; ++v) before += wsum[v];
    const int tot = wsum[0] + wsum[1] + wsum[2] + wsum[3];
    __syncthreads();
    if (sel) o[before + in_wave] = x;
    base += tot;
    eq_seen += eq_tot;
  }
}

__global__ __launch_bounds__(256) void first_samples_kernel(int32_t* idx, int64_t idx_stride, int n, int stride) {
  int32_t* o = idx + (int64_t)bid_x() * idx_stride;
  for (int i = tid_x(); i < n; i += 256) o[i] = i * stride;
}

}  // namespace saf3r

using namespace saf3r;

// Whether the frame stage searches for a window of k .. kCands keys. The closer k comes to kCands, the more counts
// it takes to hit the window, and frames with few different scores jump over it; the exact threshold takes
// 16 counts whatever the scores. The line is fitted to (us, 16384 rows x 8 frames of normal scores in bf16, window /
// exact): 160 keys k = 64 77 / 82, 96 129 / 82; 256 keys k = 80 107 / 100; 512 keys k = 80 120 / 142, 96 152 / 142; 768 keys
// k = 96 165 / 182; 1036 keys k = 112 213 / 225, 128 284 / 225; 1369 keys k = 112 229 / 263, 128 317 / 263.
static bool frame_window(int per_frame, int k) {
  return per_frame <= kCands || k <= std::min(112, std::max(64, 48 + per_frame / 16));
}

extern "C" int saf3r_frame_topk_scores(const void* scores, int64_t score_stride, int rows, int frames, int per_frame,
                                       int exclude_first, int first_stride, int per_frame_mode, int topk, int cap,
                                       int32_t* idx, int64_t idx_stride, int32_t* cand_idx, uint16_t* cand_key,
                                       void* stream) {
  if (int e = injected("saf3r_frame_topk_scores")) return e;
  if (!scores || !idx) return fail(SAF3R_ERR_INVALID, "saf3r_frame_topk_scores: null pointer");
  if (rows < 0 || frames <= 0 || per_frame <= 0 || topk <= 0 || first_stride < 0 || rows > 65535)
    return fail(SAF3R_ERR_INVALID, "saf3r_frame_topk_scores: bad shape");
  const int64_t nk = (int64_t)frames * per_frame;
  if (nk > 0x7fffffff || score_stride < nk) return fail(SAF3R_ERR_INVALID, "saf3r_frame_topk_scores: bad score stride");
  const int f0 = exclude_first ? 1 : 0;
  const int nfr = frames - f0;
  const int fsel = exclude_first && first_stride > 0 ? (per_frame + first_stride - 1) / first_stride : 0;
  if (exclude_first && first_stride <= 0)
    return fail(SAF3R_ERR_INVALID, "saf3r_frame_topk_scores: first_stride must be positive with exclude_first");
  // keys drawn from the frames after the optional frame 0, before the cap
  int64_t rest;
  if (per_frame_mode) rest = (int64_t)min(topk, per_frame) * nfr;
  else rest = min((int64_t)topk, nk - (int64_t)f0 * per_frame);
  const int64_t kept = cap > 0 ? min(rest, (int64_t)cap) : rest;
  if (idx_stride < fsel + kept) return fail(SAF3R_ERR_INVALID, "saf3r_frame_topk_scores: idx_stride too small");
  if (per_frame_mode && per_frame > kMaxPerFrame)
    return fail(SAF3R_ERR_UNSUPPORTED, "saf3r_frame_topk_scores: per_frame must be <= %d", kMaxPerFrame);
  if (score_stride % 8 || (uintptr_t)scores % 16)
    return fail(SAF3R_ERR_INVALID, "saf3r_frame_topk_scores: score rows must be 16-byte aligned (stride %% 8)");
  const bool capped = kept < rest;
  if (per_frame_mode && nfr > 0 && capped && (!cand_idx || !cand_key))
    return fail(SAF3R_ERR_INVALID, "saf3r_frame_topk_scores: the cap needs the candidate buffers");
  if (rows == 0) return SAF3R_OK;
  hipStream_t st = (hipStream_t)stream;
  if (fsel > 0) {
    // the guaranteed first-frame samples 0, s, 2s, ... in the first columns of every row
    hipLaunchKernelGGL(first_samples_kernel, dim3(rows), dim3(256), 0, st, idx, idx_stride, fsel, first_stride);
    if (int e = check_launch("saf3r_frame_topk_scores")) return e;
  }
  if (per_frame_mode && nfr > 0) {
    const int k = min(topk, per_frame);
    FrameTopkParams p;
    p.scores = (const uint16_t*)scores;
    p.srs = score_stride;
    p.rows = rows;
    p.F = frames;
    p.P = per_frame;
    p.f0 = f0;
    p.k = k;
    p.out = capped ? cand_idx : idx;
    p.ors = capped ? rest : idx_stride;
    p.ocol = capped ? 0 : fsel;
    p.okey = capped ? cand_key : nullptr;
    p.window = frame_window(per_frame, k);
    const dim3 grid((nfr + 3) / 4, rows);
    // m keys at or above a threshold, spread at random, reach 64 (1 - e^(-m / 64)) of the lane
    // maxima: aim at the middle of the window
    p.lanes = (int)(64.0 * (1.0 - std::exp(-std::sqrt((double)std::min(k, kCands) * kCands) / 64.0)));
    const int words = per_frame / 2 + 1;  // of a frame's span, at most
#define SAF3R_FRAME(KERNEL, NR, NF) hipLaunchKernelGGL((KERNEL<NR, NF>), grid, dim3(256), 0, st, p)
    if (k <= kListMax && words <= 64 * kListWords) {
      if (words <= 64 * 2) SAF3R_FRAME(frame_list_kernel, 2, 0);
      else if (words <= 64 * 3) SAF3R_FRAME(frame_list_kernel, 3, 1);
      else if (words <= 64 * 5) SAF3R_FRAME(frame_list_kernel, 5, 2);
      else if (words <= 64 * 7) SAF3R_FRAME(frame_list_kernel, 7, 4);
      else if (words <= 64 * 9) SAF3R_FRAME(frame_list_kernel, 9, 6);
      else SAF3R_FRAME(frame_list_kernel, 11, 8);
    } else if (words <= 64 * 2) SAF3R_FRAME(frame_select_kernel, 2, 0);
    else if (words <= 64 * 3) SAF3R_FRAME(frame_select_kernel, 3, 1);
    else if (words <= 64 * 5) SAF3R_FRAME(frame_select_kernel, 5, 2);
    else if (words <= 64 * 7) SAF3R_FRAME(frame_select_kernel, 7, 4);
    else if (words <= 64 * 9) SAF3R_FRAME(frame_select_kernel, 9, 6);
    else if (words <= 64 * 11) SAF3R_FRAME(frame_select_kernel, 11, 8);
    else if (words <= 64 * 13) SAF3R_FRAME(frame_select_kernel, 13, 10);
    else if (words <= 64 * 17) SAF3R_FRAME(frame_select_kernel, 17, 12);
    else if (words <= 64 * 25) SAF3R_FRAME(frame_select_kernel, 25, 16);
    else SAF3R_FRAME(frame_select_kernel, 33, 24);
#undef SAF3R_FRAME
    if (int e = check_launch("saf3r_frame_topk_scores")) return e;
    if (!capped) return SAF3R_OK;
  }
  if (kept <= 0) return SAF3R_OK;
  CapParams c;
  c.scores = (const uint16_t*)scores;
  c.srs = score_stride;
  c.dense_base = (int64_t)f0 * per_frame;
  c.dense_n = nk - c.dense_base;
  c.cidx = per_frame_mode ? cand_idx : nullptr;
  c.ckey = per_frame_mode ? cand_key : nullptr;
  c.crs = rest;
  c.n = rest;
  c.rows = rows;
  c.cap = (int)kept;
  c.out = idx;
  c.ors = idx_stride;
  c.ocol = fsel;
  hipLaunchKernelGGL(cap_select_kernel, dim3(rows), dim3(256), 0, st, c);
  return check_launch("saf3r_frame_topk_scores");
}
