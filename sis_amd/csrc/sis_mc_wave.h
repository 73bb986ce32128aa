// Limit-rule Monte Carlo of the performance mode: one wavefront resolves
// one connected component of the formed-pair graph, with the component's
// pairs and nucleotides held in registers (ballots and lane shuffles; no
// LDS round trips in the loop).  The algorithm per iteration is that of
// src/force_bp_limit_triplet.F90:259-330 restricted to the component:
//   pick a nucleotide with excess uniformly (ascending id order), list its
//   formed pairs in list order, shuffle them with the reference's swap
//   sweep, choose the pair to delete by the Metropolis sweep on energies,
//   delete it and update the two counts.
// Restricting to a component keeps the distribution: the uniform choice
// among all excess nucleotides, conditioned on the component, is uniform in
// it, and deletions never change counts outside the component.
#pragma once
#include "sis_device.h"

namespace sis {

constexpr int MCW_ITEMS = 2;   // pairs per lane   -> 128 pairs per component
constexpr int MCW_NODES = 4;   // nodes per lane   -> 256 nucleotides
// ints of wave scratch (LDS) for `items` pairs per lane
constexpr int mcw_lds(int items) { return 6 * 64 * items + 64; }
constexpr int MCW_LDS = mcw_lds(MCW_ITEMS);
// the large form: components of up to 256 pairs (the bucket capacity)
constexpr int MCB_ITEMS = 4, MCB_NODES = 8;
constexpr int MCB_LDS = mcw_lds(MCB_ITEMS);

__device__ __forceinline__ int lane_id() { return __lane_id(); }

__device__ __forceinline__ double philox_u(uint64_t seed, int r, int64_t step, int root, uint32_t draw) {
  U4 o = philox(U4{(uint32_t)step, (uint32_t)(step >> 32) ^ 0x4d43u, (uint32_t)root, draw},
                (uint32_t)seed, (uint32_t)(seed >> 32) ^ (0x5bd1e995u * (uint32_t)(r + 1)));
  return u01(o.x, o.y);
}

// Broadcasts from a lane chosen by a wave-uniform index go through
// v_readlane, and writes to one lane are a per-lane select: register
// traffic, no LDS round trip.
__device__ __forceinline__ int bcast(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }
__device__ __forceinline__ double bcast(double v, int lane) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)b, lane), hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned int)lo);
}
__device__ __forceinline__ int setlane(int v, int x, int lane) { return __lane_id() == lane ? x : v; }
__device__ __forceinline__ unsigned long long bcast64(unsigned long long v, int lane) {
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)v, lane);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(v >> 32), lane);
  return ((unsigned long long)hi << 32) | lo;
}
// Inclusive prefix sum over the 64 lanes.
__device__ __forceinline__ int wave_incl_scan(int v) {
  const int L = __lane_id();
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int t = __shfl_up(v, d);
    if (L >= d) v += t;
  }
  return v;
}

// Set bits of m below this lane (prefix population count).
__device__ __forceinline__ int below(unsigned long long m) {
  return __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
}
// Orders LDS writes of this wave before its later LDS reads of other lanes' words.
__device__ __forceinline__ void wave_lds_fence() { __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront"); }

// Prefix sum, minimum and maximum over the 64 lanes by DPP row shifts and
// row broadcasts: register traffic, no LDS round trip.
template <typename F>
__device__ __forceinline__ int wave_scan(int v, int id, F f) {
  v = f(v, __builtin_amdgcn_update_dpp(id, v, 0x111, 0xf, 0xf, false));   // row_shr:1
  v = f(v, __builtin_amdgcn_update_dpp(id, v, 0x112, 0xf, 0xf, false));   // row_shr:2
  v = f(v, __builtin_amdgcn_update_dpp(id, v, 0x114, 0xf, 0xf, false));   // row_shr:4
  v = f(v, __builtin_amdgcn_update_dpp(id, v, 0x118, 0xf, 0xf, false));   // row_shr:8
  v = f(v, __builtin_amdgcn_update_dpp(id, v, 0x142, 0xa, 0xf, false));   // row_bcast:15
  return f(v, __builtin_amdgcn_update_dpp(id, v, 0x143, 0xc, 0xf, false));  // row_bcast:31
}
__device__ __forceinline__ int wave_min(int v) {
  return bcast(wave_scan(v, 0x7fffffff, [](int a, int b) { return a < b ? a : b; }), 63);
}
__device__ __forceinline__ int wave_max(int v) {
  return bcast(wave_scan(v, (int)0x80000000, [](int a, int b) { return a > b ? a : b; }), 63);
}

// Ranks of the values v[k] (where ok[k]) among the distinct values held by
// the wave, ascending; returns how many distinct ones there are, or -1 when
// they span more than the 2,048 bits of the bitmap (bm, pre: 64 ints of LDS
// each).  A bit per value, a prefix count over the 64 words and two LDS
// reads a value: a few hundred cycles whatever the number of values, where
// comparing each with all others took thousands.
template <int K>
__device__ __forceinline__ int wave_rank(const int (&v)[K], const bool (&ok)[K], int *bm, int *pre, int (&rank)[K]) {
  const int L = lane_id();
  int lo = 0x7fffffff, hi = -1;
#pragma unroll
  for (int k = 0; k < K; k++)
    if (ok[k]) {
      lo = v[k] < lo ? v[k] : lo;
      hi = v[k] > hi ? v[k] : hi;
    }
  lo = wave_min(lo);
  hi = wave_max(hi);
  if (hi - lo >= 2048) return -1;
  bm[L] = 0;
  wave_lds_fence();
#pragma unroll
  for (int k = 0; k < K; k++)
    if (ok[k]) atomicOr(&bm[(v[k] - lo) >> 5], 1 << ((v[k] - lo) & 31));
  wave_lds_fence();
  const int c = __popc((unsigned)bm[L]);
  const int inc = wave_scan(c, 0, [](int a, int b) { return a + b; });
  pre[L] = inc - c;
  wave_lds_fence();
#pragma unroll
  for (int k = 0; k < K; k++) {
    const int d = ok[k] ? v[k] - lo : 0;
    rank[k] = pre[d >> 5] + __popc((unsigned)bm[d >> 5] & ((1u << (d & 31)) - 1u));
  }
  wave_lds_fence();
  return bcast(inc, 63);
}

// wave_rank for values of any span (a component between chains whose beads
// are numbered far apart): every value compared with all `nv` (value k of
// lane L is number L + 64 k; all: nv rounded up to 4 ints of LDS, first: as
// many).  Kept rolled: a launch meets this code cold, and the fetch of an
// unrolled body took longer than the loop (17,000 cycles against 25,000 for
// a 26-pair component).
template <int K>
__device__ __forceinline__ int wave_rank_any(const int (&v)[K], int nv, int *all, int *first, int (&rank)[K]) {
  constexpr int NONE = 0x7fffffff;
  const int L = lane_id();
  const int n4 = (nv + 3) & ~3;
  bool f[K];
#pragma unroll
  for (int k = 0; k < K; k++) {
    const int t = L + 64 * k;
    f[k] = t < nv;
    rank[k] = 0;
    if (t < n4) all[t] = t < nv ? v[k] : NONE;
  }
  wave_lds_fence();
  for (int j = 0; j < nv; j++) {
    const int x = all[j];
#pragma unroll
    for (int k = 0; k < K; k++)
      if (j < L + 64 * k && x == v[k]) f[k] = false;
  }
  int nn = 0;
#pragma unroll
  for (int k = 0; k < K; k++) {
    const int t = L + 64 * k;
    if (t < n4) first[t] = f[k] ? v[k] : NONE;
    nn += __popcll(__ballot(f[k]));
  }
  wave_lds_fence();
  for (int j = 0; j < nv; j++) {
    const int x = first[j];
#pragma unroll
    for (int k = 0; k < K; k++) rank[k] += x < v[k];
  }
  wave_lds_fence();
  return nn;
}

// The pick among nact active nucleotides, ceil(u nact) - 1, with the draw
// of lane o (wu, its upper 32 bits wh): floor(u nact) unless the product is
// a whole number, which the upper 32 bits exclude except next to one.
__device__ __forceinline__ int mc_pick(unsigned wh, double wu, int nact, int o) {
  const uint64_t pr = (uint64_t)(unsigned)bcast((int)wh, o) * (unsigned)nact;
  if ((unsigned)pr - 2u <= 0xffffffe0u - (unsigned)nact) return (int)(pr >> 32);
  return bcast((int)ceil(wu * nact), o) - 1;
}

// The Monte Carlo loop of mc_component_wave over its pair slots (IT chunks
// of 64: endpoints ua, ub as nucleotide slots, energies en) and nucleotides
// (ND chunks of 64: excess counts cnt).  live: the pairs left at the end.
// Uniform arguments; all 64 lanes call it.  Returns false on an
// inconsistent state.
//
// One deletion is a serial chain of scalar and lane operations on one
// wavefront, which issues an instruction every four to eight cycles, so its
// time is the number of instructions on it: live pairs are scalar masks,
// nothing is worked out ahead (answers kept per nucleotide for the draws to
// come took more instructions than they saved), the pick is mc_pick's
// 32-bit multiply for an FP64 product, ceiling and conversion, and a
// sequence of up to 8 pairs is packed in 64 bits.
template <int IT, int ND>
__device__ __forceinline__ bool mc_sweep(int rk, int root, double beta, uint64_t seed, int64_t step, int *sseq,
                                         const int (&ua)[IT], const int (&ub)[IT], const double (&en)[IT],
                                         int (&cnt)[ND], unsigned long long (&live)[IT]) {
  const int L = lane_id();
  // energy of pair slot `slot` (wave-uniform)
  auto ene_of = [&](int slot) {
    double x = en[0];
#pragma unroll
    for (int k = 1; k < IT; k++) x = (slot >> 6) == k ? en[k] : x;
    return bcast(x, slot & 63);
  };
  uint32_t draw = 0, w0 = (uint32_t)-64;
  double wu = 0.0, wl = 0.0;
  unsigned wh = 0;
  unsigned long long g2 = 0;
  for (;;) {
    // active nucleotides (excess > 0) in ascending id order
    unsigned long long am[ND];
    int pc[ND], nact = 0;
#pragma unroll
    for (int q = 0; q < ND; q++) {
      am[q] = __ballot(cnt[q] > 0);
      pc[q] = __popcll(am[q]);
      nact += pc[q];
    }
    if (nact == 0) return true;
    // draws: a window of 64 counters, lane i holding draw w0 + i, its
    // logarithm (Metropolis test: log u < dE beta) and its upper 32 bits;
    // g2: draws above one half (the swap target of a two-pair sequence).
    // It holds any sequence of up to eight pairs.
    if ((int)(draw - w0) > 64 - 16) {
      w0 = draw;
      wu = philox_u(seed, rk, step, root, w0 + (uint32_t)L);
      wl = log(wu);
      wh = (unsigned)(wu * 4294967296.0);
      g2 = __ballot(wu > 0.5);
    }
    const int o = (int)(draw - w0);
    int want = mc_pick(wh, wu, nact, o);
    unsigned long long amq = am[0];
    int base = 0;
#pragma unroll
    for (int q = 1; q < ND; q++) {
      const bool next = base == 64 * (q - 1) && want >= pc[q - 1];
      want = next ? want - pc[q - 1] : want;
      amq = next ? am[q] : amq;
      base = next ? 64 * q : base;
    }
    const int ntd = base + __builtin_ctzll(__ballot(below(amq) == want) & amq);
    // its pairs in list order
    unsigned long long sm[IT];
    int ns = 0;
#pragma unroll
    for (int k = 0; k < IT; k++) {
      sm[k] = (__ballot(ua[k] == ntd) | __ballot(ub[k] == ntd)) & live[k];
      ns += __popcll(sm[k]);
    }
    if (ns == 0) return false;
    if (ns > 64) ns = 64;
    int del;
    if (ns == 2) {
      // two pairs: the swap sweep leaves them reversed exactly when both
      // swap draws fall on the same side of one half
      int la = -1, lb = -1;
#pragma unroll
      for (int k = IT - 1; k >= 0; k--)
        if (sm[k]) la = 64 * k + __builtin_ctzll(sm[k]);
#pragma unroll
      for (int k = 0; k < IT; k++)
        if (sm[k]) lb = 64 * k + 63 - __builtin_clzll(sm[k]);
      const unsigned t = (unsigned)(g2 >> (o + 1)) & 3u;
      const bool flip = t == 0u || t == 3u;
      const int s0 = flip ? lb : la, s1 = flip ? la : lb;
      const double e0 = ene_of(s0), w = bcast(wl, o + 3);
      double ev = en[0];
#pragma unroll
      for (int k = 1; k < IT; k++) ev = (s1 >> 6) == k ? en[k] : ev;
      const bool acc = (__ballot(w < (ev - e0) * beta) >> (s1 & 63)) & 1ull;
      del = acc ? s1 : s0;
    } else if (ns <= 8) {
      // short sequence: kept in scalar registers, entry m in bits
      // 8m..8m+7 (slots < 256)
      uint64_t sp = 0;
      int m = 0;
#pragma unroll
      for (int k = 0; k < IT; k++)
        for (unsigned long long mk = sm[k]; mk; mk &= mk - 1) {
          sp |= (uint64_t)(64 * k + __builtin_ctzll(mk)) << m;
          m += 8;
        }
      const int swv = 8 * ((int)ceil(wu * ns) - 1);
      // reference shuffle: for i = 1..n swap(i, ceil(rnd*n))
      for (int i = 0; i < 8 * ns; i += 8) {
        const int sw = bcast(swv, o + 1 + (i >> 3));
        const uint64_t x = ((sp >> i) ^ (sp >> sw)) & 0xffull;   // swap entries i and sw
        sp ^= (x << i) | (x << sw);
      }
      // Metropolis sweep on the energies of the sequence's pairs
      del = (int)(sp & 0xffull);
      double edel = ene_of(del);
      for (int i = 1; i < ns; i++) {
        const int si = (int)((sp >> (8 * i)) & 0xffull);
        const double ej = ene_of(si);
        if (bcast(wl, o + ns + i) < (ej - edel) * beta) { del = si; edel = ej; }
      }
    } else {
      // long sequence: entry m in lane m (through LDS)
#pragma unroll
      for (int k = 0, m0 = 0; k < IT; k++) {
        const int m = m0 + below(sm[k]);
        if (((sm[k] >> L) & 1ull) && m < 64) sseq[m] = 64 * k + L;
        m0 += __popcll(sm[k]);
      }
      wave_lds_fence();
      int seqv = L < ns ? sseq[L] : 0;
      // lane i: the i-th swap target, and the logarithm of the draw that
      // decides on entry i
      const double us = philox_u(seed, rk, step, root, draw + 1u + (uint32_t)L);
      const double ul = log(philox_u(seed, rk, step, root, draw + (uint32_t)(ns + L)));
      const int swl = (int)ceil(us * ns) - 1;
      for (int i = 0; i < ns; i++) {
        const int sw = bcast(swl, i);
        const int ti = bcast(seqv, i), ts = bcast(seqv, sw);
        seqv = setlane(seqv, ts, i);
        seqv = setlane(seqv, ti, sw);
      }
      del = bcast(seqv, 0);
      double edel = ene_of(del);
      for (int i = 1; i < ns; i++) {
        const int si = bcast(seqv, i);
        const double ej = ene_of(si);
        if (bcast(ul, i) < (ej - edel) * beta) { del = si; edel = ej; }
      }
      wave_lds_fence();
    }
    // draws used: 1 (pick) + ns (shuffle) + ns - 1 (Metropolis) = 2 ns
    draw += 2u * (uint32_t)ns;
    int a = ua[0], b = ub[0];
#pragma unroll
    for (int k = 1; k < IT; k++) {
      a = (del >> 6) == k ? ua[k] : a;
      b = (del >> 6) == k ? ub[k] : b;
    }
    const int da = bcast(a, del & 63), db = bcast(b, del & 63);
#pragma unroll
    for (int k = 0; k < IT; k++) live[k] &= (del >> 6) == k ? ~(1ull << (del & 63)) : ~0ull;
#pragma unroll
    for (int q = 0; q < ND; q++) cnt[q] -= (L + 64 * q == da) + (L + 64 * q == db);
  }
}

// The same loop for components of at most 64 pairs and 128 nucleotides, one
// pair and two nucleotides a lane: the live pairs are one 64-bit mask, and
// a sequence of up to 8 pairs a 4-bit permutation of their ranks.  1,250
// cycles a deletion (34 deletions of a 40-pair component in 42,000), 1,700
// with the FP64 pick and 2,000 with answers worked out ahead.  Its loops stay rolled: unrolled ones gained 5% on such a
// component and lost 30% on one of five pairs, to instruction fetch.
// Returns false if a nucleotide has more than 8 formed
// pairs or the state is inconsistent (the caller then runs the general loop
// from the start, which gives the same result).
__device__ __forceinline__ bool mc_sweep64(int rk, int root, int n, double beta, uint64_t seed, int64_t step,
                                           int ua, int ub, double en, int cnt0, int cnt1, unsigned long long &live) {
  const int L = lane_id();
  live = __ballot(L < n);
  uint32_t draw = 0, w0 = (uint32_t)-64;
  double wu = 0.0, wl = 0.0;
  unsigned wh = 0;
  unsigned long long g2 = 0;
  for (;;) {
    const unsigned long long a0 = __ballot(cnt0 > 0), a1 = __ballot(cnt1 > 0);
    const int p0 = __popcll(a0), nact = p0 + __popcll(a1);
    if (nact == 0) return true;
    if ((int)(draw - w0) > 64 - 16) {   // the window holds any sequence of up to eight pairs
      w0 = draw;
      wu = philox_u(seed, rk, step, root, w0 + (uint32_t)L);
      wl = log(wu);
      wh = (unsigned)(wu * 4294967296.0);
      g2 = __ballot(wu > 0.5);
    }
    const int o = (int)(draw - w0);
    const int want0 = mc_pick(wh, wu, nact, o);
    const bool upper = want0 >= p0;
    const unsigned long long am = upper ? a1 : a0;
    const int want = upper ? want0 - p0 : want0;
    const int ntd = __builtin_ctzll(__ballot(below(am) == want) & am) + (upper ? 64 : 0);
    const unsigned long long sm = (__ballot(ua == ntd) | __ballot(ub == ntd)) & live;
    const int ns = __popcll(sm);
    if (ns == 0 || ns > 8) return false;
    int del;
    if (ns == 2) {
      // two pairs: the swap sweep leaves them reversed exactly when both
      // swap draws fall on the same side of one half
      const int la = __builtin_ctzll(sm), lb = 63 - __builtin_clzll(sm);
      const unsigned t = (unsigned)(g2 >> (o + 1)) & 3u;
      const bool flip = t == 0u || t == 3u;
      const int s0 = flip ? lb : la, s1 = flip ? la : lb;
      const double e0 = bcast(en, s0), w = bcast(wl, o + 3);
      const bool acc = (__ballot(w < (en - e0) * beta) >> s1) & 1ull;
      del = acc ? s1 : s0;
    } else {
      // ntd's pairs in list order are the set bits of sm in lane order (rank
      // 0..ns-1); perm holds the rank at each sequence slot, 4 bits a slot
      const int swv = 4 * ((int)ceil(wu * ns) - 1);
      uint32_t perm = 0x76543210u;
      for (int i = 0; i < ns; i++) {
        const int sw = bcast(swv, o + 1 + i);
        const uint32_t x = ((perm >> (4 * i)) ^ (perm >> sw)) & 15u;
        perm ^= (x << (4 * i)) | (x << sw);
      }
      const int rkl = below(sm);
      del = __builtin_ctzll(__ballot(rkl == (int)(perm & 15u)) & sm);
      double edel = bcast(en, del);
      for (int i = 1; i < ns; i++) {
        const int si = __builtin_ctzll(__ballot(rkl == (int)((perm >> (4 * i)) & 15u)) & sm);
        const double ej = bcast(en, si);
        if (bcast(wl, o + ns + i) < (ej - edel) * beta) { del = si; edel = ej; }
      }
    }
    draw += 2u * (uint32_t)ns;
    live &= ~(1ull << del);
    const int da = bcast(ua, del), db = bcast(ub, del);
    cnt0 -= (L == da) + (L == db);
    cnt1 -= (L + 64 == da) + (L + 64 == db);
  }
}

// Resolve the component whose formed pairs are seg[0..n) (candidate ids,
// any order).  Must be called by all 64 lanes of a wave with uniform
// arguments; ws is mcw_lds(IT) ints of LDS private to the wave (8-byte
// aligned).  Returns false if the component exceeds the capacity of 64*IT
// pairs or its state is inconsistent, having written nothing.  The result
// does not depend on IT (same draws, same decisions).  r indexes the
// per-replica arrays; rk keys the random stream.
// Layout: pair slot t (candidate-id order) lives in lane t % 64, chunk
// t / 64; nucleotide slot u (ascending id) in lane u % 64, chunk u / 64;
// the pair sequence of one iteration holds entry m in lane m.
template <int IT = MCW_ITEMS, int ND = MCW_NODES>
__device__ __forceinline__ bool mc_component_wave(const Params &P, const Ptrs &D, int r, int rk, int root,
                                                  const int *seg, int n, double beta, uint64_t seed,
                                                  int64_t step, int *ws) {
  constexpr int NONE = 0x7fffffff;
  constexpr int NP = 64 * IT;
  static_assert(NP <= 256 && ND <= 8 && ND == 2 * IT, "pair slots are packed in 8 bits, nucleotide slots in 9");
  const int L = lane_id();
  const int N = P.N;
  // uniform by contract; said so to the compiler, so that loop counters
  // and lane indices stay scalar
  n = __builtin_amdgcn_readfirstlane(n);
  root = __builtin_amdgcn_readfirstlane(root);
  if (n > NP) return false;
  // ---- pairs in candidate-id order (= reference list order)
  int *ssort = ws + 128;   // after the two 64-word arrays of wave_rank, inside its any-span arrays
  int raw[IT], rank[IT];
  bool ok[IT];
#pragma unroll
  for (int k = 0; k < IT; k++) {
    const int t = L + 64 * k;
    ok[k] = t < n;
    raw[k] = ok[k] ? seg[t] : NONE;
  }
  if (wave_rank(raw, ok, ws, ws + 64, rank) < 0) wave_rank_any(raw, n, ws, ws + NP, rank);
#pragma unroll
  for (int k = 0; k < IT; k++)
    if (ok[k]) ssort[rank[k]] = raw[k];
  wave_lds_fence();
  int gb[IT], ua[IT], ub[IT], e2[2 * IT], u2[2 * IT];
  bool ok2[2 * IT];
  double en[IT];
  bool bad = false;
#pragma unroll
  for (int k = 0; k < IT; k++) {
    gb[k] = ok[k] ? ssort[L + 64 * k] : NONE;
    e2[2 * k] = e2[2 * k + 1] = -1;
    ok2[2 * k] = ok2[2 * k + 1] = ok[k];
    en[k] = 0.0;
    if (ok[k]) {
      const int *mp = D.bp_mp + (size_t)gb[k] * 8;
      e2[2 * k] = mp[0] - 1;
      e2[2 * k + 1] = mp[1] - 1;
      en[k] = D.ene_bp[gb[k]];
      bad = bad || e2[2 * k] < 0 || e2[2 * k] >= N || e2[2 * k + 1] < 0 || e2[2 * k + 1] >= N;
    }
  }
  wave_lds_fence();
  // a candidate naming a bead outside the system means corrupted MC state:
  // report it (flags[7]) instead of indexing with it
  if (__ballot(bad)) {
    if (L == 0) D.flags[7] = 1;
    return true;
  }
  // ---- distinct nucleotides in ascending id order, with their counts
  int *snode = ws + 128;
  int nn = wave_rank(e2, ok2, ws, ws + 64, u2);
  if (nn < 0) {
    // endpoint number L + 64 j of lane L in wave_rank_any's numbering:
    // pairs of chunk k first by their lower, then their upper nucleotide
    int v[2 * IT], w[2 * IT];
#pragma unroll
    for (int k = 0; k < IT; k++) {
      v[k] = ok[k] ? e2[2 * k] : N;      // slots beyond n hold one value
      v[IT + k] = ok[k] ? e2[2 * k + 1] : N;   // above every bead id
    }
    nn = wave_rank_any(v, 2 * NP, ws + 64, ws + 64 + 2 * NP, w) - (n < NP ? 1 : 0);
#pragma unroll
    for (int k = 0; k < IT; k++) {
      u2[2 * k] = w[k];
      u2[2 * k + 1] = w[IT + k];
    }
  }
#pragma unroll
  for (int j = 0; j < 2 * IT; j++)
    if (ok2[j]) snode[u2[j]] = e2[j];   // equal values write the same word
  wave_lds_fence();
  int cnt[ND];
#pragma unroll
  for (int q = 0; q < ND; q++) {
    const int u = L + 64 * q;
    cnt[q] = u < nn ? D.nt_cnt[(size_t)r * N + snode[u]] : 0;
  }
  wave_lds_fence();
#pragma unroll
  for (int k = 0; k < IT; k++) {
    ua[k] = ok[k] ? u2[2 * k] : -1;
    ub[k] = ok[k] ? u2[2 * k + 1] : -1;
  }
  unsigned long long live[IT];
#pragma unroll
  for (int k = 0; k < IT; k++) live[k] = __ballot(ok[k]);
  // half the nucleotide chunks do for nearly all components
  bool done = false;
  if constexpr (IT == 1) {
    done = mc_sweep64(rk, root, n, beta, seed, step, ua[0], ub[0], en[0], cnt[0], cnt[1], live[0]);
    live[0] = done ? live[0] : __ballot(ok[0]);
  }
  if (done) {
  } else if (IT > 1 && nn <= 32 * ND) {
    int c[ND / 2];
#pragma unroll
    for (int q = 0; q < ND / 2; q++) c[q] = cnt[q];
    done = mc_sweep<IT, ND / 2>(rk, root, beta, seed, step, ws, ua, ub, en, c, live);
  } else {
    done = mc_sweep<IT, ND>(rk, root, beta, seed, step, ws, ua, ub, en, cnt, live);
  }
  if (!done) return false;
  // write back the pairs deleted here
#pragma unroll
  for (int k = 0; k < IT; k++)
    if (ok[k] && !((live[k] >> L) & 1ull)) D.bp_status[gb[k]] = 0;
  return true;
}

// The wavefront forms by size: one pair per lane up to 64 pairs, MCW_ITEMS
// above.  ws holds MCW_LDS ints.
__device__ __forceinline__ bool mc_component_wave_any(const Params &P, const Ptrs &D, int r, int rk, int root,
                                                      const int *seg, int n, double beta, uint64_t seed,
                                                      int64_t step, int *ws) {
  if (n <= 64) return mc_component_wave<1, 2>(P, D, r, rk, root, seg, n, beta, seed, step, ws);
  return mc_component_wave(P, D, r, rk, root, seg, n, beta, seed, step, ws);
}
// The same up to the bucket capacity.  ws holds MCB_LDS ints.
__device__ __forceinline__ bool mc_component_wave_big(const Params &P, const Ptrs &D, int r, int rk, int root,
                                                      const int *seg, int n, double beta, uint64_t seed,
                                                      int64_t step, int *ws) {
  if (n <= 64 * MCW_ITEMS) return mc_component_wave_any(P, D, r, rk, root, seg, n, beta, seed, step, ws);
  return mc_component_wave<MCB_ITEMS, MCB_NODES>(P, D, r, rk, root, seg, n, beta, seed, step, ws);
}

// ---------------------------------------------------------------------
// A component of two pairs (the usual smallest one) by one lane: with one
// pair allowed per nucleotide they share the only nucleotide in excess, so
// its pick is certain and one deletion resolves it, by the draws the sweep
// would use (1 and 2: swaps, 3: Metropolis).  Draws and decision are those
// of mc_component_wave; many such components resolve in parallel, one per
// lane.  Returns false for any other component or an inconsistent one.
constexpr int MCL_PAIRS = 2;

__device__ __forceinline__ bool mc_component_lane(const Ptrs &D, int max_bp, int N, int rk, int root, const int *seg,
                                                  int n, double beta, uint64_t seed, int64_t step) {
  if (n != 2 || max_bp != 1) return false;
  const int g0 = seg[0], g1 = seg[1];
  const int a = g0 < g1 ? g0 : g1, b = g0 < g1 ? g1 : g0;
  const int *ma = D.bp_mp + (size_t)a * 8, *mb = D.bp_mp + (size_t)b * 8;
  const int a0 = ma[0], a1 = ma[1], b0 = mb[0], b1 = mb[1];
  if (a0 < 1 || a0 > N || a1 < 1 || a1 > N || b0 < 1 || b0 > N || b1 < 1 || b1 > N) {
    D.flags[7] = 1;
    return true;
  }
  if ((a0 == b0) + (a0 == b1) + (a1 == b0) + (a1 == b1) != 1) return false;
  const bool h1 = philox_u(seed, rk, step, root, 1u) > 0.5, h2 = philox_u(seed, rk, step, root, 2u) > 0.5;
  const double w = log(philox_u(seed, rk, step, root, 3u));
  const double ea = D.ene_bp[a], eb = D.ene_bp[b];
  // both swap draws on the same side of one half: the pairs are reversed
  const bool flip = h1 == h2;
  const double e0 = flip ? eb : ea, e1 = flip ? ea : eb;
  const bool second = w < (e1 - e0) * beta;
  D.bp_status[second == flip ? a : b] = 0;
  return true;
}

}  // namespace sis
