// On-device token selection by one wave (generator.py:178-207 of the reference, with the
// Gumbel-max / Philox draw that replaces torch.multinomial).
#pragma once
#include <type_traits>
#include "qtts_common.h"
#include "qtts_poll.h"

// forced: a call from the persistent kernels would pass their by-value launch arguments through scratch
#define QTTS_SEL_INLINE __attribute__((always_inline))

namespace qtts {

struct SelParams {
  int do_sample;
  float temperature;
  int top_k;
  float top_p;
  uint64_t seed;
  int frame_step;
  int group;
};

// Keep the better of two (value, index) candidates: larger value, lower index on ties.
__device__ __forceinline__ void best_merge(float& bv, int& bi, float ov, int oi) {
  if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
}

// LDS scratch of one selection: the short list (and a slot per lane for the writes that it does not
// take); for draws in place, every logit by id and its probability (top-p).
// Entries are words key << 16 | id.
constexpr int SEL_CAP = 256;
struct SelScratch {
  uint32_t list[SEL_CAP + 64];
  alignas(16) uint32_t all[MAXV];
  double p[MAXV];
};

// Order-preserving 16-bit key of a bf16 value and back (-inf is SEL_NINF, +inf SEL_PINF; NaNs lie outside, by their sign).
constexpr uint32_t SEL_NINF = 0x007fu, SEL_PINF = 0xff80u;
__device__ __forceinline__ uint32_t bfkey(float f) { return fkey(f) >> 16; }
__device__ __forceinline__ float bfkey_value(uint32_t k) {
  return __uint_as_float(((k & 0x8000u) ? (k ^ 0x8000u) : (k ^ 0xffffu)) << 16);
}
// the key's logit over the temperature, rounded to bf16 as the reference's bf16 logits / temperature
// (generator.py:189): non-decreasing in the key
__device__ __forceinline__ float sel_scaled(uint32_t key, float temperature) { return rbf(bfkey_value(key) / temperature); }

// Lowest key whose scaled value is that of `key`: neighbouring logits can fall together when they are
// scaled, and top-k keeps ties of the scaled values. Mostly `key` itself; a few steps down otherwise,
// then (temperatures that overflow or flush most values together) a binary search.
__device__ __forceinline__ uint32_t sel_lowest_tie(uint32_t key, float temperature) {
  if (key <= SEL_NINF) return key;
  const uint32_t sk = bfkey(sel_scaled(key, temperature));
  uint32_t k = key;
  for (int it = 0; it < 4; ++it) {
    if (k <= SEL_NINF + 1u || bfkey(sel_scaled(k - 1u, temperature)) != sk) return k;
    --k;
  }
  uint32_t lo = SEL_NINF + 1u;
  while (lo < k) {
    const uint32_t mid = (lo + k) >> 1;
    if (bfkey(sel_scaled(mid, temperature)) >= sk) k = mid; else lo = mid + 1u;
  }
  return k;
}

// k-th largest key (k >= 1) of the wave's 64 N words, found bit by bit on ballots: no LDS, no shuffles.
template <int N>
__device__ __forceinline__ uint32_t sel_kth(const uint32_t (&w)[N], int k) {
  uint32_t t = 0u;
#pragma unroll 1
  for (int b = 31; b >= 16; --b) {
    const uint32_t cand = t | (1u << b);
    int c = 0;
#pragma unroll
    for (int j = 0; j < N; ++j) c += __popcll(__ballot(w[j] >= cand));
    if (c >= k) t = cand;
  }
  return t >> 16;
}

// Greedy selection by words: larger value (-0 counts as +0, a NaN is below -inf), then lower id.
__device__ __forceinline__ uint32_t greedy_word(float x, int id) {
  static_assert(MAXV <= 4096, "12-bit ids");
  return (x != x ? 0u : bfkey(x + 0.0f) << 12) | (uint32_t)(4095 - id);
}
__device__ __forceinline__ int greedy_id(uint32_t best, int n) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) best = max(best, (uint32_t)__shfl_xor((int)best, o, 64));
  return min(4095 - (int)(best & 4095u), n - 1);
}

// Temperature / top-k / top-p / Gumbel-max over n <= MAXV masked logits (bf16 values; suppressed ids
// = -inf) by one wave, which holds them in registers as words key << 16 | id (0 past n, below every
// value's). Returns the same id on every lane.
//
// One wave at a time can issue about one instruction per 4 cycles, so the work is kept to a few
// instructions per logit and the expensive parts to the ids still in the running. For top_k <= 63 the
// k-th largest of the 64 lane maxima is a lower bound of the k-th largest logit: the ids that reach it (94 of
// 2048 on average at 50, 164 at 60, 228 at 63, where 256 is passed in a quarter of the draws) go to a short
// list of at most SEL_CAP, and the temperature division, the exact threshold, the Philox draws (one pass of 64
// lanes for 64 ids) and the logarithms run on that list alone. A larger top_k, or ties that overflow the list,
// search the threshold on the registers. No top_k, or one past SEL_CAP ids, draws in place, the words in LDS by
// id so that four neighbours share a Philox block (a frame of unlimited draws 1,577 -> 1,347 us, 8 of them
// 2,115 -> 1,907). A threshold search over 32-bit keys in LDS and a draw in every lane pass that held a kept id
// took 93 us for a code-predictor head of 2048 (top-k 50), 15 of them a frame.
constexpr int SEL_NJ = MAXV / 64;          // words per lane
// Largest top_k for the list. At 64 the bound is the smallest lane maximum, more than half of the lists overflow
// and are searched again (us, list : search: 63 a frame 1,031 : 1,071, a backbone step 482 : 490, 8 frames
// 1,657 : 1,653; 64 1,072 : 1,064, 492 : 490, 1,683 : 1,648)
constexpr int SEL_LIST_K = 63;
__device__ __forceinline__ int wave_sample(const uint32_t (&w)[SEL_NJ], int n, const SelParams& sp, SelScratch* sc) {
  const int lane = opaque((int)threadIdx.x & 63);
  const float T = sp.temperature;
  constexpr int NJ = SEL_NJ, NG = 16;      // words in groups that a smaller n skips
  static_assert(NJ % NG == 0 && MAXV <= 4096, "word groups, 12-bit ids");
  auto count = [&](uint32_t key) QTTS_SEL_INLINE {         // ids with a key >= `key`
    int c = 0;
#pragma unroll
    for (int g = 0; g < NJ; g += NG) {
      if (64 * g >= n) break;
#pragma unroll
      for (int j = g; j < g + NG; ++j) c += __popcll(__ballot(w[j] >= (key << 16)));
    }
    return c;
  };
  // ids with a key >= `key` to the list, in any order; returns how many there are (the list is whole up to
  // SEL_CAP). Every lane writes each time, to its own spare slot where its word is not taken: no branches.
  auto collect = [&](uint32_t key) QTTS_SEL_INLINE {
    int c = 0;
#pragma unroll
    for (int g = 0; g < NJ; g += NG) {
      if (64 * g >= n) break;
#pragma unroll
      for (int j = g; j < g + NG; ++j) {
        const bool in = w[j] >= (key << 16);
        const uint64_t m = __ballot(in);
        const uint32_t at = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, (uint32_t)c));
        sc->list[in && at < (uint32_t)SEL_CAP ? at : (uint32_t)(SEL_CAP + lane)] = w[j];
        c += __popcll(m);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    return c;
  };
  // top-p: keep x when the probability mass of strictly larger kept values is <= top_p: the smallest
  // scaled key t with sum_{key > t} p <= top_p z (the sum is non-increasing in t)
  auto top_p_key = [&](double z, auto&& mass_above) QTTS_SEL_INLINE {
    uint32_t lo = 0u, hi = 0xffffu;
#pragma unroll 1
    while (lo < hi) {
      const uint32_t mid = (lo + hi) >> 1;
      if (mass_above(mid) <= (double)sp.top_p * z) hi = mid; else lo = mid + 1u;
    }
    return lo;
  };
  // the running ids of the list's c entries, 64 R of them at most, of which top-k keeps k (0: all of
  // them), as scaled words; returns how many
  auto finish = [&](auto r_, int c, int k) QTTS_SEL_INLINE {
    constexpr int R = decltype(r_)::value;
    uint32_t x[R];                         // scaled key << 16 | id; 0: out of the running
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const uint32_t e = sc->list[lane + 64 * r];
      x[r] = lane + 64 * r < c ? (bfkey(sel_scaled(e >> 16, T)) << 16) | (e & 0xffffu) : 0u;
    }
    // ties of the scaled values are kept, scaled values that overflow to -inf are not
    const uint32_t thr = max(k > 0 ? sel_kth<R>(x, k) : 0u, SEL_NINF + 1u);
#pragma unroll
    for (int r = 0; r < R; ++r) x[r] = x[r] >= (thr << 16) ? x[r] : 0u;
    if (sp.top_p < 1.0f) {
      float m = -INFINITY;
#pragma unroll
      for (int r = 0; r < R; ++r) m = x[r] != 0u ? fmaxf(m, bfkey_value(x[r] >> 16)) : m;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
      double p[R], z = 0.0;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        p[r] = x[r] != 0u ? exp((double)bfkey_value(x[r] >> 16) - (double)m) : 0.0;
        z += p[r];
      }
      z = wave_sum_d(z);
      const uint32_t pth = top_p_key(z, [&](uint32_t t) QTTS_SEL_INLINE {
        double acc = 0.0;
#pragma unroll
        for (int r = 0; r < R; ++r) acc += (x[r] >> 16) > t ? p[r] : 0.0;
        return wave_sum_d(acc);
      });
#pragma unroll
      for (int r = 0; r < R; ++r) x[r] = (x[r] >> 16) >= pth ? x[r] : 0u;
    }
    // the ids still in the running move together, so that as few passes as possible draw for them
    int n_in = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const uint64_t m = __ballot(x[r] != 0u);
      const uint32_t at = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, (uint32_t)n_in));
      sc->list[x[r] != 0u ? at : (uint32_t)(SEL_CAP + lane)] = x[r];
      n_in += __popcll(m);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    return n_in;
  };
  auto finish_list = [&](int c, int k) QTTS_SEL_INLINE {
    return c <= 128 ? finish(std::integral_constant<int, 2>{}, c, k) : finish(std::integral_constant<int, SEL_CAP / 64>{}, c, k);
  };

  const bool limited = sp.top_k > 0 && sp.top_k < n;
  const bool reversed = __builtin_signbit(T);   // the scaled values fall as the keys rise: everything on scaled words
  int n_in = -1;                           // words to draw from in the list
  double best = -INFINITY;
  int bi = 0x7fffffff;
  auto draw = [&](uint32_t e, double u) QTTS_SEL_INLINE {
    const int id = (int)(e & 0xffffu);
    const double g = (double)bfkey_value(e >> 16) - log(-log(u));
    if (g > best || (g == best && id < bi)) { best = g; bi = id; }
  };
  if (limited && sp.top_k <= SEL_LIST_K && !reversed) {
    uint32_t lmax[1] = {0u};
#pragma unroll
    for (int j = 0; j < NJ; ++j) lmax[0] = max(lmax[0], w[j]);
    uint32_t low = sel_kth<1>(lmax, sp.top_k);
    // down to the lowest logit that the temperature may tie with it: the scaled values are as widely
    // spaced, to a factor of two, as the logits, so that at most 3 neighbours fall together where
    // nothing overflows or vanishes
    const float a = fabsf(bfkey_value(low));
    constexpr float BIG = 1152921504606846976.0f;   // 2^60
    if (a > 1.0f / BIG && a < BIG && T > 1.0f / BIG && T < BIG) low = max(low - 4u, SEL_NINF + 1u);
    else low = sel_lowest_tie(low, T);
    if (low > SEL_NINF) {
      const int c = collect(low);
      if (c <= SEL_CAP) n_in = finish_list(c, sp.top_k);
    }
  }
  if (n_in < 0) {
    uint32_t thr = 0u;                     // the lowest logit key that top-k keeps
    if (limited && !reversed) {
#pragma unroll 1
      for (int b = 15; b >= 0; --b)
        if (count(thr | (1u << b)) >= sp.top_k) thr |= 1u << b;
      thr = sel_lowest_tie(thr, T);
    }
    // a NaN that is kept makes the mass under top-p no number, also one with its sign bit set (below -inf)
    const bool no_mass = !reversed && sp.top_p < 1.0f && thr < SEL_NINF && (thr == 0u ? n : count(thr)) > count(SEL_NINF);
    thr = max(thr, reversed ? 0u : SEL_NINF + 1u);   // suppressed ids are never drawn
    const int c = no_mass ? 0 : (limited && sp.top_k <= SEL_CAP && !reversed ? collect(thr) : SEL_CAP + 1);
    if (c <= SEL_CAP) {
      n_in = finish_list(c, 0);
    } else {
      // every scaled word in LDS by its id (0: not kept), so that the loops below stay rolled
      sc->all[0] = 0u;
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        if (w[j] != 0u) sc->all[w[j] & 0xffffu] = w[j];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll 1
      for (int i = lane; i < n; i += 64) {
        const uint32_t e = sc->all[i];
        const float v = sel_scaled(e >> 16, T);
        sc->all[i] = e != 0u && e >= (thr << 16) && v != -INFINITY ? (bfkey(v) << 16) | (e & 0xffffu) : 0u;
      }
      if (reversed && limited) {
        uint32_t k = 0u;
#pragma unroll 1
        for (int b = 15; b >= 0; --b) {
          const uint32_t cand = k | (1u << b);
          int kept = 0;
#pragma unroll 1
          for (int i = lane; i < n; i += 64) kept += __popcll(__ballot(sc->all[i] >= (cand << 16)));
          if (kept >= sp.top_k) k = cand;
        }
#pragma unroll 1
        for (int i = lane; i < n; i += 64)
          if (sc->all[i] < (k << 16)) sc->all[i] = 0u;
      }
      n_in = 0;
      if (sp.top_p < 1.0f) {
        float m = -INFINITY;
        for (int i = lane; i < n; i += 64)
          if (sc->all[i] != 0u) m = fmaxf(m, bfkey_value(sc->all[i] >> 16));
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
        double z = 0.0;
        for (int i = lane; i < n; i += 64) {
          const double pi = sc->all[i] != 0u ? exp((double)bfkey_value(sc->all[i] >> 16) - (double)m) : 0.0;
          sc->p[i] = pi;
          z += pi;
        }
        z = wave_sum_d(z);
        const uint32_t pth = top_p_key(z, [&](uint32_t t) QTTS_SEL_INLINE {
          double acc = 0.0;
          for (int i = lane; i < n; i += 64) acc += (sc->all[i] >> 16) > t ? sc->p[i] : 0.0;
          return wave_sum_d(acc);
        });
        for (int i = lane; i < n; i += 64)
          if ((sc->all[i] >> 16) < pth) sc->all[i] = 0u;
      }
      // (four neighbouring ids share a Philox block)
#pragma unroll 1
      for (int i = 4 * lane; i < n; i += 256) {
        const u32x4 e4 = *reinterpret_cast<const u32x4*>(&sc->all[i]);
        if ((e4.x | e4.y | e4.z | e4.w) == 0u) continue;
        uint64_t c[4];
        sampler_block(c, sp.seed, sp.frame_step, sp.group, i);
#pragma unroll 1
        for (int q = 0; q < 4; ++q) {
          const uint32_t e = sc->all[i + q];
          if (e != 0u) draw(e, sampler_word(c, q));
        }
      }
    }
  }
#pragma unroll 1
  for (int i = lane; i < n_in; i += 64) {
    const uint32_t e = sc->list[i];
    draw(e, sampler_uniform(sp.seed, sp.frame_step, sp.group, (int)(e & 0xffffu)));
  }
  auto merge = [&](double ov, int oi) QTTS_SEL_INLINE {
    if (ov > best || (ov == best && oi < bi)) { best = ov; bi = oi; }
  };
  merge(xlane_d<0>(best), (int)xlane<0>((uint32_t)bi));
  merge(xlane_d<1>(best), (int)xlane<1>((uint32_t)bi));
  merge(xlane_d<2>(best), (int)xlane<2>((uint32_t)bi));
  merge(xlane_d<3>(best), (int)xlane<3>((uint32_t)bi));
  merge(xlane_d<4>(best), (int)xlane<4>((uint32_t)bi));
  merge(xlane_d<5>(best), (int)xlane<5>((uint32_t)bi));
  bi = __builtin_amdgcn_readfirstlane(bi);
  if (bi != 0x7fffffff) return bi;
  // nothing to draw from (every id suppressed, or a probability mass that is no number): the largest logit, the
  // lowest id on ties (-0 counts as +0). Keys above +inf's are NaNs'.
  const int nans = count(SEL_PINF + 1u);
  uint32_t bk = 0u;
#pragma unroll 1
  for (int b = 15; b >= 0; --b)
    if (count(bk | (1u << b)) > nans) bk |= 1u << b;
  const uint32_t tie = bk == 0x8000u ? 0x7fffu : bk;
  int lo = 0x7fffffff;
#pragma unroll
  for (int j = 0; j < NJ; ++j)
    if ((w[j] >> 16) - tie <= bk - tie && bk >= SEL_NINF) lo = min(lo, (int)(w[j] & 0xffffu));
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) lo = min(lo, __shfl_xor(lo, o, 64));
  return lo == 0x7fffffff ? 0 : lo;
}

// Selection from a head's logit slots, for the persistent decode kernels: n tagged slots at byte `off` of
// the workspace polled straight into the key registers, masked, and drawn from (or the largest taken).
// The kernels are instantiated apart for greedy and for sampled launches: with both selections in one
// kernel, the key registers raise the pressure of the whole step loop (the backbone's spills 9 -> 39 dwords).
struct HeadMask {
  int tail;                // ids [tail, n) are suppressed but for `eos` (n: none)
  int eos;
  int drop;                // one more suppressed id, or -1
  float penalty;           // on the ids in pen_bits, 1.0: none (bf16 arithmetic, generator.py:161-167)
};
// use(j, id, x) for the lane's j-th masked logit (16 per 1024 ids).
// MASKED = false: no id is suppressed or penalised (code-predictor heads).
template <bool MASKED, typename F>
__device__ __forceinline__ void head_logits(const Poll& P, uint32_t off, int n, uint32_t tag, const HeadMask& hm,
                                            const uint32_t* pen_bits, F use) {
  const int lane = opaque((int)threadIdx.x & 63);
  // 1024 slots at a time: 8 pairs per lane, two batches in flight
  auto part = [&](auto p_) QTTS_SEL_INLINE {
    constexpr int P0 = decltype(p_)::value;
    if (1024 * P0 >= n) return;
    float v[16];           // (a timed-out poll leaves the error word set and these as they are)
#pragma unroll
    for (int j = 0; j < 16; ++j) v[j] = 0.0f;
    const uint32_t o = off + 8u * 1024u * P0;
    poll_regs<8>(P, min(n - 1024 * P0, 1024) >> 1, tag, v, [o](int i) { return o + 16u * (uint32_t)i; });
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int id = 1024 * P0 + 2 * (lane + 64 * (j >> 1)) + (j & 1);
      float x = v[j];
      if constexpr (MASKED) {
        if (hm.penalty != 1.0f && id < n && ((pen_bits[id >> 5] >> (id & 31)) & 1u)) x = rbf(x > 0.f ? x / hm.penalty : x * hm.penalty);
        if ((id >= hm.tail && id != hm.eos) || id == hm.drop) x = -INFINITY;
      }
      use(16 * P0 + j, id, x);
    }
  };
  static_assert(MAXV == 3 * 1024, "head parts");
  part(std::integral_constant<int, 0>{});
  part(std::integral_constant<int, 1>{});
  part(std::integral_constant<int, 2>{});
}
template <bool MASKED>
__device__ __forceinline__ int head_argmax(const Poll& P, uint32_t off, int n, uint32_t tag, const HeadMask& hm,
                                           const uint32_t* pen_bits) {
  uint32_t best = 0u;
  head_logits<MASKED>(P, off, n, tag, hm, pen_bits, [&](int, int id, float x) QTTS_SEL_INLINE {
    best = max(best, id < n ? greedy_word(x, id) : 0u);
  });
  return greedy_id(best, n);
}
template <bool MASKED>
__device__ __forceinline__ int head_sample(const Poll& P, uint32_t off, int n, uint32_t tag, const SelParams& sp,
                                           const HeadMask& hm, const uint32_t* pen_bits, SelScratch* sc) {
  uint32_t w[SEL_NJ];
#pragma unroll
  for (int j = 0; j < SEL_NJ; ++j) w[j] = 0u;
  head_logits<MASKED>(P, off, n, tag, hm, pen_bits,
                      [&](int j, int id, float x) QTTS_SEL_INLINE { w[j] = id < n ? (bfkey(x) << 16) | (uint32_t)id : 0u; });
  return wave_sample(w, n, sp, sc);
}

}  // namespace qtts
