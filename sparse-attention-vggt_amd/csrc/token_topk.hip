// Per-frame token top-k of q.k: the lazy selector of the reference dino_topk heads.
//
// ref: saf3r/triton/fused_qk_topk.py:26-102 (bf16 q.k with fp32 accumulation per 64-key tile;
//      composite key = sortable fp32 bits << 32 | reversed index so ties go to the lower index;
//      running per-frame top-k; frame-major flush in descending order, -1 for empty slots),
//      :120-217 (API: q [B, Nq, D], k [B, Nk, D], Nk = frames * num_toks_per_img, output
//      int32 [B, Nq, frames * min(topk, num_toks_per_img)] of key indices).
// A 256-thread workgroup owns 128 queries (32 per wave). Key tiles of 64 keys are staged in LDS,
// scored with v_mfma_f32_32x32x16_bf16 (S^T = K . Q^T); a lane holds one query and 32 keys of each
// tile, and keeps a running top-k of the keys of its half; the two lane halves of a query merge
// their lists when the frame ends. Each frame is scored twice (see token_topk_kernel).
#include <algorithm>
#include <type_traits>

#include "common.h"

namespace saf3r {

struct TopkParams {
  const __bf16* qptr;
  int64_t q_rs, q_base, q_rpf, q_frs;
  const __bf16* kptr;
  int64_t k_rs, k_base, k_rpf, k_frs;
  int nq, F, P, ke;
  int kmode;  // key row of (frame f, token j): 1 = frame f row j (rows_per_frame == P), 0 = flat row f*P + j, 2 = general
  int64_t k_fst;  // kmode 0 and 1: rows from frame f to frame f + 1 (P or frame_row_stride)
  int32_t* idx;
  int fgroups;  // frame groups of the selection launch (grid.y)
};

__device__ inline const __bf16* rows_at(const __bf16* ptr, int64_t rs, int64_t base, int64_t rpf, int64_t frs,
                                        int64_t r) {
  int64_t f = r / rpf;
  return ptr + (base + f * frs + (r - f * rpf)) * rs;
}


__device__ inline uint64_t partner_u64(uint64_t x) {
  uint32_t lo = (uint32_t)x, hi = (uint32_t)(x >> 32);
  auto rl = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
  auto rh = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
  const bool upper = (tid_x() & 63) >= 32;
  uint32_t plo = upper ? (uint32_t)rl[0] : (uint32_t)rl[1];
  uint32_t phi = upper ? (uint32_t)rh[0] : (uint32_t)rh[1];
  return ((uint64_t)phi << 32) | plo;
}

// the float bits of a sortable key
__device__ __forceinline__ uint32_t fkey_bits(uint32_t k) { return k ^ (~(uint32_t)((int32_t)k >> 31) | 0x80000000u); }

// Candidate buffer of pass 2: per lane up to kCand candidates (float bits << 32 | key index), entry i
// of thread tid at cbuf[i * 256 + tid] (a lane's entries all sit in its own bank pair: no conflicts
// whatever the fill levels), emptied into the lane's running top-K at the end of each frame. A lane
// with more candidates than that in one frame (ties, or neighbouring keys that share a group) loses
// the rest and has its frame scanned again at the frame's end (see token_topk_kernel).
template <int K>
constexpr int cand_cap() { return K <= 8 ? 12 : 24; }
constexpr int kGroup = 8;  // candidates whose wave masks are formed together
constexpr int kStep = 2;   // candidates that share a wave-uniform branch
constexpr int kStages = 3;  // K tiles in flight: the tile of step t + 2 loads while step t computes

// K-th largest of the running float list t (descending, -inf = empty) after inserting x.
template <int K>
__device__ inline void fmax_insert(float (&t)[K], float x) {
  bool c[K];
#pragma unroll
  for (int i = 0; i < K; ++i) c[i] = x > t[i];
#pragma unroll
  for (int i = K - 1; i > 0; --i) t[i] = c[i - 1] ? t[i - 1] : (c[i] ? x : t[i]);
  t[0] = c[0] ? x : t[0];
}

// Two passes per key frame over the same bf16 MFMA scores (the score of a (query, key) pair is the
// same sequence of MFMAs in both, so the same fp32 value):
//   pass 1: every lane keeps the maximum of G groups of its candidates; the K-th largest of the 2G
//           group maxima of a query (its two lane halves) is a lower bound tau of the query's K-th
//           best score in the frame (they are 2G >= K distinct candidates);
//   pass 2: only candidates with score >= tau (or unordered: a NaN never drops out) are appended to
//           the lane's LDS buffer; a candidate costs one compare, and two share a wave-uniform branch
//           unless some lane of the wave keeps one (one branch each: 2 - 5% slower, one for four: the
//           same). A lane whose buffer overflowed is served at the frame's end by a scan of its wave
//           over the frame's key rows in global memory (same MFMAs, so the same scores) with the K-th
//           best of its buffered candidates as the bound, which rises as better ones are found.
// The second 32 keys of a tile go to the groups in a rotated order (G <= 16): with the same order in
// both halves, the keys of one image column shared a group on grids 32 patches wide and neighbouring
// ones on grids of 33, tau fell and frames overflowed (24 frames of 19 x 33, top-8: 153 us against 226).
// Queries past the last one keep nothing: as ties at 0 they overflowed on every frame, which cost
// the last work-group of each frame group twice its time (48 x 1369 tokens, top-4, with single-frame
// groups allowed: 1727 us against 1415).
// A few candidates per query and frame pass (about 3 of 1369 for top-4 of N(0,1) scores), so the
// composite-key insertion that dominates a one-pass selection runs a few times per frame instead
// of for every candidate. Key tiles stream through a 3-stage LDS ring filled by LDS-DMA loads
// issued two steps ahead (rows past the frame's end load a valid row; their scores are masked).
// Step t reads its K fragments, selects over the scores of step t - 1 while those reads are in
// flight, then issues its MFMAs into the same registers; the two waves of a SIMD alternate their
// VALU and MFMA phases.
template <int K, int G, bool FLAT>
__global__ __launch_bounds__(256, K <= 8 ? 3 : 2) void token_topk_kernel(TopkParams p) {
  // G groups per lane: 2G >= K maxima per query
  __shared__ __align__(16) char ring[kStages][8192];
  constexpr int kCand = cand_cap<K>();
  __shared__ uint64_t cbuf[(kCand + 1) * 256];
  const int tid = tid_x(), lane = tid & 63, half = lane >> 5, col = lane & 31;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t q0 = (int64_t)bid_x() * 128;
  const int64_t qi = q0 + 32 * w + col;
  const bool qvalid = qi < p.nq;

  bf16x8 qfrag[4];
  {
    const u32x4* qs = reinterpret_cast<const u32x4*>(
        rows_at(p.qptr, p.q_rs, p.q_base, p.q_rpf, p.q_frs, qvalid ? qi : 0) + 32 * half);
#pragma unroll
    for (int s = 0; s < 4; ++s) qfrag[s] = __builtin_bit_cast(bf16x8, qvalid ? qs[s] : u32x4{0, 0, 0, 0});
  }

  const int tiles_pf = (p.P + 63) / 64;
  // frame f: pass 1 over its tiles, then pass 2, for the frames [f_lo, f_hi) of this work-group's
  // frame group (bid_y of p.fgroups: the split only evens out the tail of the launch)
  const int f_lo = __builtin_amdgcn_readfirstlane(p.F * bid_y() / p.fgroups);
  const int f_hi = __builtin_amdgcn_readfirstlane(p.F * (bid_y() + 1) / p.fgroups);
  const int total = (f_hi - f_lo) * 2 * tiles_pf;
  // LDS chunk position P = 256 j + 64 w + lane of a tile (instruction j of wave w) holds key row
  // P / 8, global 16-byte chunk (P % 8) ^ swz8(row): the swizzle that makes the MFMA fragment
  // reads conflict-free is applied on the load side
  int rowj[2], chj[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int P = 256 * j + 64 * w + lane;
    rowj[j] = P >> 3;
    chj[j] = (P & 7) ^ swz8(rowj[j]);
  }
  int iu = 0, ips = 0;  // tile and pass of the next step to issue
  int64_t ifr = f_lo;  // its frame
  // FLAT (kmode 0 and 1): frame f's rows are k_fst rows apart, so a tile's address is a uniform
  // base plus a fixed 32-bit lane offset (the last tile of a frame clamps its rows to the frame's
  // last row: its own offsets); otherwise every row goes through the general row mapping
  const char* kb0 = reinterpret_cast<const char*>(p.kptr + p.k_base * p.k_rs);
  const int64_t fbytes = p.k_fst * p.k_rs * 2, tbytes = 64 * p.k_rs * 2;
  uint32_t lo[2], lo_last[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    lo[j] = (uint32_t)(rowj[j] * p.k_rs * 2 + 16 * chj[j]);
    const int rl = min(64 * (tiles_pf - 1) + rowj[j], p.P - 1) - 64 * (tiles_pf - 1);
    lo_last[j] = (uint32_t)(rl * p.k_rs * 2 + 16 * chj[j]);
  }
  // the tile of sequence step `step` (the next one) into its stage; past the last step the last
  // frame's last tile is loaded again into a stage nobody reads, so every step waits on the same
  // count of loads
  // tile address of the next step to issue (FLAT), advanced by additions; stage of that step
  const char* itb = kb0 + f_lo * fbytes;
  int ist = 0;
  auto issue = [&](int step) __attribute__((always_inline)) {
    char* st = ring[ist];
    ist = ist == kStages - 1 ? 0 : ist + 1;
    if constexpr (FLAT) {
      const char* tb = itb;
      const bool last = iu == tiles_pf - 1;
#pragma unroll
      for (int j = 0; j < 2; ++j)
        dma16s(tb, last ? lo_last[j] : lo[j], __builtin_amdgcn_readfirstlane(lds_addr(st + 4096 * j + 1024 * w)));
    } else {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int pp = min(64 * iu + rowj[j], p.P - 1);
        const __bf16* row = rows_at(p.kptr, p.k_rs, p.k_base, p.k_rpf, p.k_frs, ifr * p.P + pp);
        dma16(row + 8 * chj[j], __builtin_amdgcn_readfirstlane(lds_addr(st + 4096 * j + 1024 * w)));
      }
    }
    if (step + 1 < total) {
      itb += tbytes;
      if (++iu == tiles_pf) {
        iu = 0;
        ifr += ips;
        itb -= tiles_pf * tbytes;
        if (ips) itb += fbytes;
        ips ^= 1;
      }
    }
  };

  uint64_t a[K];  // the lane's running top-K of its half of the frame (composite keys, 0 = empty)
#pragma unroll
  for (int t = 0; t < K; ++t) a[t] = 0;
  float gmax[G];  // this lane's group maxima over the tiles of pass 1 so far
#pragma unroll
  for (int g = 0; g < G; ++g) gmax[g] = -__builtin_inff();
  float tau = -__builtin_inff();
  // LDS byte address of this lane's next entry, row n for n candidates so far in the frame (rows
  // from kCand on are written to row kCand, the spare row that absorbs writes past the buffer)
  const uint32_t wa0 = lds_addr(cbuf) + 8 * tid, wspare = wa0 + 2048 * kCand;
  uint32_t wa = wa0;
  auto count = [&]() { return (int)((wa - wa0) >> 11); };
  auto flush = [&]() __attribute__((always_inline)) {
    const int n = min(count(), kCand);
    for (int i = 0; i < n; ++i) {
      const uint64_t ent = cbuf[i * 256 + tid];
      topk_insert<K>(a, ckey(__builtin_bit_cast(float, (uint32_t)(ent >> 32)), (uint32_t)ent));
    }
    wa = wa0;
  };
  // candidate e of this lane: key 32*(e>>4) + 8*((e&15)>>2) + 4*half + (e&3) of the tile
  auto kpos = [](int e) { return 32 * (e >> 4) + 8 * ((e & 15) >> 2) + (e & 3); };
  int f = f_lo, ps = 0, u = 0;  // frame, pass and tile of the step being selected
  // Frame f again, for the lanes flagged `over` (their a[] holds the best K of the buffered ones). K
  // fragments come from global memory (this lane's rows col of each half tile, chunks 4 half ..
  // 4 half + 3), the next ones loading while these are scored; the MFMAs run as in the main loop.
  // Keys come in increasing order, so once a[] is full only a higher score than its last can enter.
  auto direct = [&](bool over) __attribute__((always_inline)) {
    int cl = col, hf = half;
    asm volatile("" : "+v"(cl), "+v"(hf));  // addresses formed here, not held through the main loop
    float bound = over ? fmaxf(tau, __builtin_bit_cast(float, fkey_bits((uint32_t)(a[K - 1] >> 32)))) : __builtin_inff();
    if (over) {
#pragma unroll
      for (int e = 0; e < K; ++e) a[e] = 0;
    }
    auto fetch = [&](int h2, u32x4 (&t)[4]) __attribute__((always_inline)) {  // rows 32 h2 + col
      const int r = min(32 * h2 + cl, p.P - 1);
      const __bf16* row;
      if constexpr (FLAT) row = reinterpret_cast<const __bf16*>(kb0 + f * fbytes) + (int64_t)r * p.k_rs;
      else row = rows_at(p.kptr, p.k_rs, p.k_base, p.k_rpf, p.k_frs, (int64_t)f * p.P + r);
#pragma unroll
      for (int s = 0; s < 4; ++s) t[s] = reinterpret_cast<const u32x4*>(row + 32 * hf)[s];
    };
    u32x4 t[4];
    fetch(0, t);
#pragma unroll 1
    for (int h2 = 0; h2 < 2 * tiles_pf; ++h2) {
      f32x16 d = {};
#pragma unroll
      for (int s = 0; s < 4; ++s)
        d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, t[s]), qfrag[s], d, 0, 0, 0);
      fetch(h2 + 1, t);  // (past the end: the last row again)
      const int pb = 32 * h2 + 4 * hf;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int pp = pb + kpos(e);
        const bool keep = over && !(d[e] < bound) && pp < p.P;
        if (__builtin_amdgcn_ballot_w64(keep)) {
          topk_insert<K>(a, keep ? ckey(d[e], (uint32_t)pp) : 0);
          // (a NaN bound keeps every candidate; the insertion decides)
          if (a[K - 1]) bound = __builtin_bit_cast(float, fkey_bits((uint32_t)(a[K - 1] >> 32) + 1));
        }
      }
    }
  };
  // PADDED: the frame's last tile holds positions past the frame's end, which never count
  auto select = [&](auto padded_tag, const f32x16& s0, const f32x16& s1) __attribute__((always_inline)) {
    constexpr bool PADDED = decltype(padded_tag)::value;
    const int pbase = 64 * u + 4 * half;
    const int lim = p.P - pbase;  // candidate e is a key of the frame when kpos(e) < lim
    auto sc = [&](int e) { return e < 16 ? s0[e] : s1[e - 16]; };
    if (ps == 0) {
#pragma unroll
      for (int e = 0; e < 32; ++e) {
        const int g = G <= 16 && e >= 16 ? (e + 9) % G : e % G;
        gmax[g] = fmaxf(gmax[g], (!PADDED || kpos(e) < lim) ? sc(e) : -__builtin_inff());
      }
    } else {
#pragma unroll
      for (int e0 = 0; e0 < 32; e0 += kGroup) {
        // the wave masks of a group of candidates first, then one uniform branch each: the compares' latency
        // is paid once per group
        uint64_t bm[kGroup];
#pragma unroll
        for (int i = 0; i < kGroup; ++i)  // >= tau, or unordered
          bm[i] = __builtin_amdgcn_ballot_w64(!(sc(e0 + i) < tau) && (!PADDED || kpos(e0 + i) < lim));
#pragma unroll
        for (int i0 = 0; i0 < kGroup; i0 += kStep) {
          uint64_t any = bm[i0];
#pragma unroll
          for (int i = i0 + 1; i < i0 + kStep; ++i) any |= bm[i];
          if (any) {
            // every lane writes its next entry; only the lanes that keep the candidate advance
#pragma unroll
            for (int i = i0; i < i0 + kStep; ++i) {
              const int e = e0 + i;
              const bool keep = !(sc(e) < tau) && (!PADDED || kpos(e) < lim);
              const uint32_t at = min(wa, wspare);
              wa += keep ? 2048u : 0u;
              auto* ew = reinterpret_cast<__attribute__((address_space(3))) uint32_t*>(at);
              ew[0] = (uint32_t)(pbase + kpos(e));
              ew[1] = __builtin_bit_cast(uint32_t, sc(e));
            }
          }
        }
      }
    }
  };
  // the end of a pass over frame f
  auto pass_end = [&]() __attribute__((always_inline)) {
    if (ps == 0) {
      // K-th largest of this query's 2G group maxima (this lane's and its partner half's)
      float top[K];
#pragma unroll
      for (int i = 0; i < K; ++i) top[i] = -__builtin_inff();
#pragma unroll
      for (int g = 0; g < G; ++g) {
        uint32_t b = __builtin_bit_cast(uint32_t, gmax[g]);
        auto r = __builtin_amdgcn_permlane32_swap(b, b, false, false);
        const float other = __builtin_bit_cast(float, (uint32_t)(half ? r[0] : r[1]));
        fmax_insert<K>(top, gmax[g]);
        fmax_insert<K>(top, other);
        gmax[g] = -__builtin_inff();
      }
      // lanes past the last query score 0 everywhere: they keep nothing (as ties they would fill
      // their buffers over and over)
      tau = qvalid ? top[K - 1] : __builtin_inff();
    } else {
      // empty the buffer (and scan the frame again for overflowed lanes), merge the partner half's
      // list, then write this frame's indices
      const bool over = count() > kCand;
      flush();
      if (__builtin_amdgcn_ballot_w64(over)) direct(over);
      uint64_t b[K];
#pragma unroll
      for (int e = 0; e < K; ++e) b[e] = partner_u64(a[e]);
#pragma unroll
      for (int e = 0; e < K; ++e)
        if (b[e] > a[K - 1]) topk_insert<K>(a, b[e]);
      if (qvalid && half == 0) {
        int32_t* o = p.idx + qi * ((int64_t)p.F * p.ke) + (int64_t)f * p.ke;
#pragma unroll
        for (int e = 0; e < K; ++e)
          if (e < p.ke) o[e] = a[e] ? (int32_t)(f * p.P + ckey_index(a[e])) : -1;
      }
#pragma unroll
      for (int e = 0; e < K; ++e) a[e] = 0;
      tau = -__builtin_inff();
      ++f;
    }
    u = 0;
    ps ^= 1;
  };

  wait_vm<0>();  // q fragments landed; from here vmcnt counts ring loads only
  for (int s = 0; s < kStages - 1; ++s) issue(s);
  f32x16 s0 = {}, s1 = {};  // scores of the previous step
  int rst = 0;  // stage of step t
  for (int t = 0; t <= total; ++t) {
    bf16x8 ka[4], kbf[4];
    const char* kb = ring[0];
    auto read_k = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int chn = 4 * half + s;
        const int r0 = col, r1 = 32 + col;
        ka[s] = *reinterpret_cast<const bf16x8*>(&kb[r0 * 128 + ((chn ^ swz8(r0)) << 4)]);
        kbf[s] = *reinterpret_cast<const bf16x8*>(&kb[r1 * 128 + ((chn ^ swz8(r1)) << 4)]);
      }
    };
    if (t < total) {
      wait_vm<2 * (kStages - 2)>();  // tile t landed: only the loads of step t + 1 are pending
      barrier_only();                // every wave's share of tile t is in LDS; every wave is done with tile t-1
      issue(t + kStages - 1);
      kb = ring[rst];
      rst = rst == kStages - 1 ? 0 : rst + 1;
      read_k();
    }
    if (t > 0) {
      if (64 * u + 64 > p.P) select(std::true_type{}, s0, s1);
      else select(std::false_type{}, s0, s1);
      if (++u == tiles_pf) {
        pass_end();
        if (t < total) read_k();  // read again rather than held in 32 registers meanwhile
      }
    }
    if (t < total) {
      // S^T = K . Q^T over the staged tile: keys 0..31 in s0, 32..63 in s1
      s0 = f32x16{};
      s1 = f32x16{};
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        s0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka[s], qfrag[s], s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kbf[s], qfrag[s], s1, 0, 0, 0);
      }
    }
  }
  wait_vm<0>();  // the trailing loads into unread stages land before the work-group's LDS is released
}

static int gpu_cus() {
  int cus = 0, dev = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
    cus = 256;
  return cus;
}

// Frame groups: every work-group walks all frames of its queries, so with few, long work-groups the
// launch ends with a partly idle last round. The frames split into g groups (one work-group per
// query block and group): the largest g of at most 16 whose rounds of resident work-groups (`per_cu`
// per CU) are within 2% of the fullest (at 128 frames x 1369 tokens, top-4: g = 16, 10.5 ms against
// 10.9 with g = 5 and 13.2 with one group). Groups of single frames are allowed: with at least 8
// frames a group, 16 x 1036 tokens took 735 us against 257, 4 x 1036 413 against 107.
static int frame_groups(int64_t nb, int frames, int per_cu) {
  const int64_t slots = (int64_t)gpu_cus() * per_cu;
  const int gmax = std::max(1, std::min(16, frames));
  auto eff = [&](int g) {
    const int64_t wgs = nb * g, rounds = (wgs + slots - 1) / slots;
    return (double)wgs / (double)(rounds * slots);
  };
  double best_eff = 0.0;
  for (int g = 1; g <= gmax; ++g) best_eff = std::max(best_eff, eff(g));
  for (int g = gmax; g >= 1; --g)
    if (eff(g) >= best_eff - 0.02) return g;
  return 1;
}

template <int K, int G>
static int launch_topk(TopkParams p, hipStream_t st) {
  const int64_t nb = (p.nq + 127) / 128;
  p.fgroups = frame_groups(nb, p.F, K <= 8 ? 3 : 2);
  const dim3 grid((unsigned)nb, (unsigned)p.fgroups);
  if (p.kmode == 2) hipLaunchKernelGGL((token_topk_kernel<K, G, false>), grid, dim3(256), 0, st, p);
  else hipLaunchKernelGGL((token_topk_kernel<K, G, true>), grid, dim3(256), 0, st, p);
  return check_launch("saf3r_token_topk");
}

// ---- per-frame top-k for 16 < k <= 128 (the reference's range): score rows in LDS ----
constexpr int kLargeMaxP = 4096;  // frame length of that path (values of a row held by one wave)
constexpr int kRowWaves = 16;

// x of lane (lane ^ D)
template <int CTL>
__device__ __forceinline__ uint32_t dpp32(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, CTL, 0xF, 0xF, true);
}
template <int D>
__device__ __forceinline__ uint32_t lane_xor(uint32_t x, int lane) {
  if constexpr (D == 1) return dpp32<0xB1>(x);
  else if constexpr (D == 2) return dpp32<0x4E>(x);
  else if constexpr (D == 4) return dpp32<0x1B>(dpp32<0x141>(x));  // the mirror of 8 lanes (^ 7), then of 4 (^ 3)
  else if constexpr (D == 8) return dpp32<0x128>(x);
  else if constexpr (D == 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    return (lane & 16) ? (uint32_t)r[0] : (uint32_t)r[1];
  } else {
    const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    return (lane & 32) ? (uint32_t)r[0] : (uint32_t)r[1];
  }
}
template <int D>
__device__ __forceinline__ uint64_t lane_xor(uint64_t x, int lane) {
  return ((uint64_t)lane_xor<D>((uint32_t)(x >> 32), lane) << 32) | lane_xor<D>((uint32_t)x, lane);
}

// x of 32 bits over the wave, as a wave-uniform value
template <typename T, typename Op>
__device__ __forceinline__ T wave_reduce32(T x, Op op) {
  auto at = [](uint32_t y) { return __builtin_bit_cast(T, y); };
  auto bits = [](T y) { return __builtin_bit_cast(uint32_t, y); };
  x = op(x, at(dpp32<0xB1>(bits(x))));
  x = op(x, at(dpp32<0x4E>(bits(x))));
  x = op(x, at(dpp32<0x141>(bits(x))));
  x = op(x, at(dpp32<0x128>(bits(x))));
  const auto a = __builtin_amdgcn_permlane16_swap(bits(x), bits(x), false, false);
  x = op(at((uint32_t)a[0]), at((uint32_t)a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(bits(x), bits(x), false, false);
  x = op(at((uint32_t)b[0]), at((uint32_t)b[1]));
  return at((uint32_t)__builtin_amdgcn_readfirstlane((int)bits(x)));
}

// One compare-exchange of a bitonic network over the wave: runs of M lanes, distance D
// (the lanes that keep the larger value as a literal mask: compares per lane would be hoisted out of
// the caller's loops, 42 scalar registers)
constexpr uint64_t keep_max(int M, int D, bool desc) {
  uint64_t m = 0;
  for (int l = 0; l < 64; ++l)
    if ((((l & M) == 0) == ((l & D) == 0)) == desc) m |= 1ull << l;
  return m;
}
template <int M, int D, bool DESC, typename T>
__device__ __forceinline__ void lane_cas(T& x, int lane) {
  constexpr uint64_t keep = keep_max(M, D, DESC);
  const T y = lane_xor<D>(x, lane);
  x = __builtin_amdgcn_inverse_ballot_w64(~(__builtin_amdgcn_ballot_w64(x > y) ^ keep)) ? x : y;
}
// runs of M lanes, each bitonic, to sorted runs (M = 64: the whole wave, descending for DESC)
template <int M, int D, bool DESC, typename T>
__device__ __forceinline__ void lane_merge(T& x, int lane) {
  lane_cas<M, D, DESC>(x, lane);
  if constexpr (D > 1) lane_merge<M, D / 2, DESC>(x, lane);
}
template <bool DESC, int M = 2, typename T>
__device__ __forceinline__ void lane_sort(T& x, int lane) {
  lane_merge<M, M / 2, DESC>(x, lane);
  if constexpr (M < 64) lane_sort<DESC, 2 * M>(x, lane);
}
// x, y (empty entries 0) of a wave's n entries, the 64 best descending in x; the rest in y for `both`
template <typename T>
__device__ __forceinline__ void lane_sort128(T& x, T& y, int n, bool both, int lane) {
  lane_sort<true>(x, lane);
  if (n > 64) {  // wave-uniform
    lane_sort<false>(y, lane);
    const T big = x > y ? x : y;
    y = x > y ? y : x;
    x = big;
    lane_merge<64, 32, true>(x, lane);
    if (both) lane_merge<64, 32, true>(y, lane);
  }
}

// base + the set lanes of m below this one
__device__ __forceinline__ int lanes_before(uint64_t m, int base) {
  return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, (uint32_t)base));
}
// A work-group owns QR queries (16, or 8 of the 16 matrix columns for long frames) and walks the
// frames of its group. Per frame: the waves share out the frame's 16-key tiles, score them on the
// matrix core (v_mfma_f32_16x16x32_bf16, S^T = K . Q^T) and put the fp32 scores into LDS rows,
// one row per query (a tile's loads read whole 128-byte rows and reach the A fragments through a
// swizzled LDS stage: fragments read straight from global memory touch 16 rows per 16 lanes, which
// the address unit takes four times as long for); then every wave selects whole rows, a lane holding NV scores of its row:
//   - a threshold with k .. CAP scores at or above it: a first guess from the lane maxima (one compare
//     and ballot per bisection step), then wave-wide counts of all scores until the count falls into
//     the window, which mostly takes one or two;
//   - those candidates, as composite keys, into the row's own LDS space, then a bitonic sort over
//     the wave (DPP exchanges) and the k best written out in order.
// A row whose counts jump over the window (more than CAP - k equal scores, or infinities), or that holds a NaN
// (the matrix core hands every NaN on as -NaN, the lowest key), takes the exact threshold on the sortable
// keys, equal keys from the lowest index on.
// CAP is 64 for k <= 32 (one sorted register per lane), else 128 (two, merged).
// The next frame's fragments load while the rows of this one are selected (NV <= 24; longer frames
// have no registers for it).
// Bound by the VALU of the selection and the loads' latency: a work-group of 16 waves fills a CU
// (its LDS rows take 74 KB at 1036 keys and 90 KB at 1369), scoring takes 220 us of 500 at
// 16 x 1036 tokens, top-64, and the 128-entry sort 80 us. The prefetch takes the registers to their limit of 128:
// none spilled at 1036 keys, 42 at 1369, 157 at 4096 (most of them of the exact path). It replaced a
// dump of every score to a workspace in HBM and a radix select of eight digit passes over LDS bins per row:
// 1630 -> 500 us there, 21.9 -> 6.2 ms at 48 x 1369 tokens. A 64-bit sort of (score, index)
// took 220 VALU instructions against 82, fragments loaded without the LDS stage 50 us more.
template <int NV, bool FLAT>
__global__ __launch_bounds__(64 * kRowWaves) void topk_rows_kernel(TopkParams p) {
  constexpr int QR = NV <= 24 ? 16 : 8;
  constexpr int kTiles = NV / 4 + (NV % 4 != 0);  // 16-key tiles of a wave
  const int cap = p.ke <= 32 ? 64 : 128;
  // m scores at or above a threshold, spread at random, reach 64 (1 - e^(-m / 64)) of the lane
  // maxima: aim at the middle of the window
  const int lanes = (int)(64.f * (1.f - __expf(-sqrtf((float)p.ke * cap) / 64.f)));
  constexpr bool kPrefetch = NV <= 24;
  // row stride = 4 (mod 64) words: the 16-byte score stores of the 16 query columns take distinct banks
  // (NV = 64 has no LDS left for it)
  __shared__ __align__(16) float rows[QR][NV * 64 + (NV < 64 ? 4 : 0)];
  // a wave's tile on its way from coalesced loads to A fragments: 16 rows of 8 chunks, swizzled
  __shared__ __align__(16) char stage[kRowWaves][2048];
  static_assert(sizeof(rows) / QR >= 128 * 8, "a row's candidates fit its LDS space");
  const int tid = tid_x(), lane = tid & 63, col = lane & 15, kq = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t q0 = (int64_t)bid_x() * QR;
  bf16x8 qf[2];
  {
    const int64_t qi = q0 + col;
    const bool ok = col < QR && qi < p.nq;
    const u32x4* qs = reinterpret_cast<const u32x4*>(rows_at(p.qptr, p.q_rs, p.q_base, p.q_rpf, p.q_frs, ok ? qi : 0));
#pragma unroll
    for (int s = 0; s < 2; ++s) qf[s] = __builtin_bit_cast(bf16x8, ok ? qs[4 * s + kq] : u32x4{0, 0, 0, 0});
  }
  const int f_lo = __builtin_amdgcn_readfirstlane((int)((int64_t)p.F * bid_y() / p.fgroups));
  const int f_hi = __builtin_amdgcn_readfirstlane((int)((int64_t)p.F * (bid_y() + 1) / p.fgroups));
  const char* kb0 = reinterpret_cast<const char*>(p.kptr + p.k_base * p.k_rs);
  const int64_t fbytes = p.k_fst * p.k_rs * 2;
  const int krow = (int)p.k_rs * 2;  // FLAT: a frame's rows stay below 2^31 bytes
  // tile w + 16 i of frame f: lane l holds chunk l % 8 of rows l / 8 and 8 + l / 8, so that a load
  // reads whole rows (rows past the frame's end read its last row)
  const int lrow = lane >> 3, lchk = lane & 7;
  auto load_tile = [&](int f, int i, u32x4 (&kt)[2]) __attribute__((always_inline)) {
    int lrow = lane >> 3;
    asm volatile("" : "+v"(lrow));  // offsets computed anew, not held across the frame loop
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int j = min(16 * (w + kRowWaves * i) + 8 * h + lrow, p.P - 1);
      if constexpr (FLAT) {
        const char* fb = kb0 + f * fbytes;  // wave-uniform, plus a 32-bit lane offset
        kt[h] = *reinterpret_cast<const u32x4*>(fb + (uint32_t)(j * krow + 16 * lchk));
      } else {
        const __bf16* row = rows_at(p.kptr, p.k_rs, p.k_base, p.k_rpf, p.k_frs, (int64_t)f * p.P + j);
        kt[h] = reinterpret_cast<const u32x4*>(row)[lchk];
      }
    }
  };
  auto score_tile = [&](int i, const u32x4 (&kt)[2]) __attribute__((always_inline)) {
    char* st = stage[w];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int r = 8 * h + lrow;
      *reinterpret_cast<u32x4*>(st + r * 128 + ((lchk ^ swz8(r)) << 4)) = kt[h];
    }
    f32x4 d = {};
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const bf16x8 kf = *reinterpret_cast<const bf16x8*>(st + col * 128 + (((4 * s + kq) ^ swz8(col)) << 4));
      d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[s], d, 0, 0, 0);
    }
    const int tile = w + kRowWaves * i;
    if (16 * tile + 16 > p.P) {  // positions past the frame's end never reach a threshold
      int left = p.P - 16 * tile - 4 * kq;
      asm volatile("" : "+v"(left));
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (r >= left) d[r] = -__builtin_inff();
    }
    if (tile < 4 * NV && col < QR) *reinterpret_cast<f32x4*>(&rows[col][16 * tile + 4 * kq]) = d;
  };
  u32x4 kt[kPrefetch ? kTiles : 1][2];
  auto prefetch = [&](int f) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kTiles; ++i) load_tile(f, i, kt[i]);
  };
  if constexpr (kPrefetch) prefetch(f_lo);

  for (int f = f_lo; f < f_hi; ++f) {
    if constexpr (kPrefetch) {
#pragma unroll
      for (int i = 0; i < kTiles; ++i) score_tile(i, kt[i]);
    } else {
#pragma unroll 2
      for (int i = 0; i < kTiles; ++i) {
        load_tile(f, i, kt[0]);
        score_tile(i, kt[0]);
      }
    }
    __syncthreads();
    if constexpr (kPrefetch)
      if (f + 1 < f_hi) prefetch(f + 1);
    for (int r = w; r < QR; r += kRowWaves) {
      if (q0 + r >= p.nq) break;
      float* row = rows[r];
      // opaque per row: keeps the compiler from holding NV key indices and compares in registers
      // across the frame loop
      int ln = lane;
      asm volatile("" : "+v"(ln));
      u32x2* buf = reinterpret_cast<u32x2*>(row);  // candidates: score bits, key index
      float v[NV];  // score of key lane + 64 i
#pragma unroll
      for (int i = 0; i < NV; ++i) v[i] = row[ln + 64 * i];
      auto count = [&](float t) {  // scores at or above t, wave-wide
        int c = 0;
#pragma unroll
        for (int i = 0; i < NV; ++i) c += __popcll(__builtin_amdgcn_ballot_w64(!(v[i] < t)));
        return c;
      };
      // the counts take a NaN of either sign for the best, the key order has -NaN last: to the exact threshold
      // (two scores a compare: 519 -> 522 us at 16 x 1036 tokens, top-64)
      uint64_t nans = 0;
#pragma unroll
      for (int i = 0; i < NV; i += 2) nans |= __builtin_amdgcn_ballot_w64(__builtin_isunordered(v[i], v[i + 1]));
      float t = -0x1.fffffep127f;  // P <= cap: every finite score is a candidate
      bool found = false;
      float lo = -__builtin_inff(), hi = __builtin_inff();
      if (!nans && p.P <= cap) {
        const int c = count(t);
        found = c >= p.ke && c <= cap;
      } else if (!nans) {
        float lmax = v[0];
#pragma unroll
        for (int i = 1; i < NV; ++i) lmax = fmaxf(lmax, v[i]);
        hi = wave_reduce32(lmax, [](float a, float b) { return fmaxf(a, b); });
        lo = wave_reduce32(lmax, [](float a, float b) { return fminf(a, b); });
        if (p.ke > 64) lo -= 2.f * (hi - lo);  // 64 scores reach the least lane maximum: look below it
        // first guess: the value that about `lanes` of the 64 lane maxima reach
        float a = lo, b = hi;
        t = 0.5f * a + 0.5f * b;
        for (int step = 0; step < 10; ++step) {
          const int c = __popcll(__builtin_amdgcn_ballot_w64(!(lmax < t)));
          if (c > lanes + 2) a = t;
          else if (c < lanes - 2) b = t;
          else break;
          t = 0.5f * a + 0.5f * b;
        }
        for (int step = 0; step < 32; ++step) {
          if (!(t > lo && t < hi)) break;
          const int c = count(t);
          if (c < p.ke) hi = t;
          else if (c > cap) lo = t;
          else {
            found = true;
            break;
          }
          t = 0.5f * lo + 0.5f * hi;
        }
      }
      int n = 0;  // candidates, in increasing key index
      // (likely: otherwise the exact path's values take registers of this one: 6 x 1369 tokens, top-32 115 us
      // against 100, 2 x 4096 219 against 127)
      if (__builtin_expect(found, 1)) {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
          const bool take = !(v[i] < t);
          const uint64_t m = __builtin_amdgcn_ballot_w64(take);
          const int at = lanes_before(m, n);
          if (take) buf[at] = u32x2{__builtin_bit_cast(uint32_t, v[i]), (uint32_t)(ln + 64 * i)};
          n += __popcll(m);
        }
      } else {
        asm volatile("" : "+v"(ln));
        uint32_t u[NV];  // sortable keys, 0 past the frame's end
#pragma unroll
        for (int i = 0; i < NV; ++i) u[i] = ln + 64 * i < p.P ? fkey(v[i]) : 0;
        auto count_keys = [&](uint32_t x) {
          int c = 0;
#pragma unroll
          for (int i = 0; i < NV; ++i) c += __popcll(__builtin_amdgcn_ballot_w64(u[i] >= x));
          return c;
        };
        // The ke-th largest key: at least ke keys are >= thr, fewer above last. First the search's bounds (the counts
        // took both zeros as equal), then the best key up to `last`, which is it where few scores differ
        // (16 x 1036 tokens, top-64, all scores equal 1335 -> 715 us, five values 1600 -> 1000: it was 32 counts
        // from the top bit down), with three halvings between its tries.
        const uint32_t from = fkey(lo == 0.f ? -0.f : lo), to = fkey(hi == 0.f ? 0.f : hi);
        uint32_t thr = 0, last = 0xFFFFFFFFu;
#pragma unroll 1
        for (int step = -2; thr < last; ++step) {
          uint32_t x = step == -2 ? from : step == -1 ? to : thr + ((last - thr) >> 1) + 1;
          const bool best = step >= 0 && (step & 3) == 0;
          if (best) {
            x = 0;
#pragma unroll
            for (int i = 0; i < NV; ++i) x = max(x, u[i] <= last ? u[i] : 0u);
            x = wave_reduce32(x, [](uint32_t a, uint32_t b) { return max(a, b); });
          }
          if (count_keys(x) >= p.ke) {
            thr = x;
            if (best) break;
          } else {
            last = x - 1;
          }
        }
        int need = p.ke;  // keys equal to thr to take
#pragma unroll
        for (int i = 0; i < NV; ++i) need -= __popcll(__builtin_amdgcn_ballot_w64(u[i] > thr));
#pragma unroll
        for (int i = 0; i < NV; ++i) {
          const bool eq = u[i] == thr && ln + 64 * i < p.P;
          const uint64_t meq = __builtin_amdgcn_ballot_w64(eq);
          const bool take = u[i] > thr || (eq && lanes_before(meq, 0) < need);
          const uint64_t m = __builtin_amdgcn_ballot_w64(take);
          const int at = lanes_before(m, n);
          if (take) buf[at] = u32x2{fkey_bits(u[i]), (uint32_t)(ln + 64 * i)};
          n += __popcll(m);
          need -= min(need, (int)__popcll(meq));
        }
        t = __builtin_bit_cast(float, fkey_bits(thr));
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      int32_t* o = p.idx + (q0 + r) * ((int64_t)p.F * p.ke) + (int64_t)f * p.ke;
      const u32x2 c0 = buf[lane], c1 = buf[64 + lane];  // (entries from n on are not used)
      const uint32_t k0 = fkey(__builtin_bit_cast(float, c0[0])), k1 = fkey(__builtin_bit_cast(float, c1[0]));
      const uint32_t kt0 = fkey(t);
      const bool in0 = lane < n, in1 = 64 + lane < n;
      if (!__builtin_amdgcn_ballot_w64((in0 && (k0 - kt0) >> 25) || (in1 && (k1 - kt0) >> 25))) {
        // every candidate within 2^25 float steps of the threshold: one 32-bit word orders them by
        // score, then by slot (slots are in key order), with the slot in its low 7 bits
        uint32_t x = in0 ? ((k0 - kt0) << 7) | (uint32_t)(127 - lane) : 0u;
        uint32_t y = in1 ? ((k1 - kt0) << 7) | (uint32_t)(63 - lane) : 0u;
        lane_sort128(x, y, n, p.ke > 64, lane);
        if (lane < p.ke) o[lane] = f * p.P + (int)buf[127 - (x & 127)][1];
        if (64 + lane < p.ke) o[64 + lane] = f * p.P + (int)buf[127 - (y & 127)][1];
      } else {
        uint64_t x = in0 ? ((uint64_t)k0 << 32) | (0xFFFFFFFEu - c0[1]) : 0;
        uint64_t y = in1 ? ((uint64_t)k1 << 32) | (0xFFFFFFFEu - c1[1]) : 0;
        lane_sort128(x, y, n, p.ke > 64, lane);
        if (lane < p.ke) o[lane] = f * p.P + (int)ckey_index(x);
        if (64 + lane < p.ke) o[64 + lane] = f * p.P + (int)ckey_index(y);
      }
    }
    __syncthreads();
  }
}

// Bytes of one query's workspace share (frames x frame length rounded up to 64, fp32).
static int64_t large_row_bytes(int frames, int per_frame) { return (int64_t)frames * (64 * ((per_frame + 63) / 64)) * 4; }

// Queries per chunk: a workspace of at most 1 GiB in whole work-groups of 128 queries (at least one).
static int64_t large_chunk_rows(int n_q, int frames, int per_frame) {
  int64_t nqc = ((int64_t)1 << 30) / large_row_bytes(frames, per_frame) / 128 * 128;
  if (nqc < 128) nqc = 128;
  const int64_t nq128 = ((int64_t)n_q + 127) / 128 * 128;
  return nqc < nq128 ? nqc : nq128;
}

template <int NV, bool FLAT = true>
static void launch_rows(const TopkParams& p, dim3 grid, hipStream_t st) {
  hipLaunchKernelGGL((topk_rows_kernel<NV, FLAT>), grid, dim3(64 * kRowWaves), 0, st, p);
}

// Top-k of LDS score rows.
static int launch_topk_rows(TopkParams p, hipStream_t st) {
  const int nv = (p.P + 63) / 64;
  const int qr = nv <= 24 ? 16 : 8;
  const int64_t nb = ((int64_t)p.nq + qr - 1) / qr;
  p.fgroups = frame_groups(nb, p.F, 1);
  const dim3 grid((unsigned)nb, (unsigned)p.fgroups);
  if (p.kmode == 2) {  // the general row map: four lengths
    if (nv <= 8) launch_rows<8, false>(p, grid, st);
    else if (nv <= 24) launch_rows<24, false>(p, grid, st);
    else if (nv <= 32) launch_rows<32, false>(p, grid, st);
    else launch_rows<64, false>(p, grid, st);
  } else if (nv <= 4) launch_rows<4>(p, grid, st);
  else if (nv <= 6) launch_rows<6>(p, grid, st);
  else if (nv <= 8) launch_rows<8>(p, grid, st);
  else if (nv <= 10) launch_rows<10>(p, grid, st);
  else if (nv <= 12) launch_rows<12>(p, grid, st);
  else if (nv <= 14) launch_rows<14>(p, grid, st);
  else if (nv <= 16) launch_rows<16>(p, grid, st);
  else if (nv <= 18) launch_rows<18>(p, grid, st);
  else if (nv <= 20) launch_rows<20>(p, grid, st);
  else if (nv <= 22) launch_rows<22>(p, grid, st);
  else if (nv <= 24) launch_rows<24>(p, grid, st);
  else if (nv <= 32) launch_rows<32>(p, grid, st);
  else if (nv <= 48) launch_rows<48>(p, grid, st);
  else launch_rows<64>(p, grid, st);
  return check_launch("saf3r_token_topk");
}

// Whether a top-k of at most 16 takes the LDS rows. They start a work-group per 16 queries and frame
// group and need no second pass, so small launches end sooner; the two-pass kernel does less work
// per key and wins once it fills the chip. Measured in rounds of 16 queries x 1 frame per CU (us,
// rows / two passes): top-4 2 x 1036 tokens (1 round) 15 / 29, 3 x 1036 (2.3) 21 / 29, 4 x 1036 (4)
// 40 / 29, 3 x 1369 (3) 47 / 36; top-8 3 x 1036 21 / 35, 4 x 1036 41 / 35; top-16 5 x 1036 (6.3)
// 54 / 57, 5 x 1369 (8.4) 81 / 73, 16 x 1036 418 / 274. Short frames leave the two-pass bound of a
// top-16 weak (64 groups of P / 64 keys): 16 x 256 42 / 79, 64 x 256 553 / 1050.
// The two sum a score's products in different orders (16x16x32 and 32x32x16 MFMAs), so keys whose scores are
// within that rounding can change places between a small call and a large one.
static bool topk_takes_rows(const TopkParams& p) {
  if (p.kmode == 2 || p.P > 1536) return false;
  if (p.ke > 8 && p.P <= 512) return true;
  const int64_t tasks = ((int64_t)p.nq + 15) / 16 * p.F;
  return tasks <= (int64_t)gpu_cus() * (p.ke <= 4 ? 2 : p.ke <= 8 ? 3 : 6);
}

}  // namespace saf3r

using namespace saf3r;

// Shape checks shared by saf3r_token_topk and its workspace query.
static int topk_shape(const char* who, int n_q, int frames, int per_frame, int topk) {
  if (n_q < 0 || frames <= 0 || per_frame <= 0) return fail(SAF3R_ERR_INVALID, "%s: bad shape", who);
  if (topk < 1) return fail(SAF3R_ERR_INVALID, "%s: topk must be >= 1", who);
  const int ke = topk < per_frame ? topk : per_frame;
  if (ke > 128) return fail(SAF3R_ERR_UNSUPPORTED, "%s: min(topk, per_frame) must be <= 128 (got %d)", who, ke);
  if (ke > 16 && (per_frame > kLargeMaxP || frames > 65535))
    return fail(SAF3R_ERR_UNSUPPORTED, "%s: topk > 16 needs per_frame <= %d and frames <= 65535", who, kLargeMaxP);
  return SAF3R_OK;
}

extern "C" int64_t saf3r_token_topk_workspace_bytes(int n_q, int frames, int per_frame, int topk) {
  if (topk_shape("saf3r_token_topk_workspace_bytes", n_q, frames, per_frame, topk)) return -1;
  const int ke = topk < per_frame ? topk : per_frame;
  if (ke <= 16 || n_q == 0) return 0;
  return large_chunk_rows(n_q, frames, per_frame) * large_row_bytes(frames, per_frame);
}

extern "C" int saf3r_token_topk(const saf3r_rows* q, const saf3r_rows* k, int n_q, int frames, int per_frame,
                                int topk, int32_t* idx, void* workspace, int64_t workspace_bytes, void* stream) {
  if (int e = injected("saf3r_token_topk")) return e;
  if (!q || !k || !q->ptr || !k->ptr || !idx) return fail(SAF3R_ERR_INVALID, "saf3r_token_topk: null pointer");
  if (int e = topk_shape("saf3r_token_topk", n_q, frames, per_frame, topk)) return e;
  const int ke = topk < per_frame ? topk : per_frame;
  if (workspace_bytes < 0) return fail(SAF3R_ERR_INVALID, "saf3r_token_topk: negative workspace size");
  if (q->row_stride % 8 || k->row_stride % 8 || ((uintptr_t)q->ptr | (uintptr_t)k->ptr) % 16 ||
      q->rows_per_frame <= 0 || k->rows_per_frame <= 0)
    return fail(SAF3R_ERR_INVALID, "saf3r_token_topk: rows must be 16-byte aligned, row stride %% 8");
  if (n_q == 0) return SAF3R_OK;
  TopkParams p;
  p.qptr = (const __bf16*)q->ptr;
  p.q_rs = q->row_stride;
  p.q_base = q->base_row;
  p.q_rpf = q->rows_per_frame;
  p.q_frs = q->frame_row_stride;
  p.kptr = (const __bf16*)k->ptr;
  p.k_rs = k->row_stride;
  p.k_base = k->base_row;
  p.k_rpf = k->rows_per_frame;
  p.k_frs = k->frame_row_stride;
  p.kmode = k->rows_per_frame == per_frame ? 1 : k->rows_per_frame >= (int64_t)frames * per_frame ? 0 : 2;
  p.k_fst = p.kmode == 1 ? k->frame_row_stride : per_frame;
  // the flat form addresses a frame's rows with 32-bit lane offsets from a tile base
  if (p.kmode != 2 && ((int64_t)per_frame + 64) * k->row_stride * 2 >= ((int64_t)1 << 31)) p.kmode = 2;
  p.nq = n_q;
  p.F = frames;
  p.P = per_frame;
  p.ke = ke;
  p.idx = idx;
  p.fgroups = 1;
  hipStream_t st = (hipStream_t)stream;
  if (ke > 16) {  // the workspace is checked as the ABI states and not used
    const int64_t row_bytes = large_row_bytes(p.F, p.P);
    if (!workspace || workspace_bytes / row_bytes < 128)
      return fail(SAF3R_ERR_INVALID,
                  "saf3r_token_topk: min(topk, per_frame) > 16 needs a workspace of at least %lld bytes "
                  "(saf3r_token_topk_workspace_bytes), got %lld",
                  (long long)(128 * row_bytes), (long long)(workspace ? workspace_bytes : 0));
    return launch_topk_rows(p, st);
  }
  if (topk_takes_rows(p)) return launch_topk_rows(p, st);
  if (p.ke <= 1) return launch_topk<1, 8>(p, st);
  if (p.ke <= 2) return launch_topk<2, 8>(p, st);
  // short frames: 16 groups of a lane (64 x 256 tokens, top-4: 149 us against 245 with 8), whose
  // registers cost long ones 5% (128 x 1369: 9.68 ms against 9.21)
  if (p.ke <= 4) return p.P <= 512 ? launch_topk<4, 16>(p, st) : launch_topk<4, 8>(p, st);
  if (p.ke <= 8) return launch_topk<8, 16>(p, st);
  return launch_topk<16, 32>(p, st);
}
