// Phase kernels of the SIS MD step (one thread per bead, per candidate or
// per component).  Included by sis_gpu.hip.
#pragma once
#include "sis_device.h"
#include "sis_mc_wave.h"

namespace sis {

// ---------------------------------------------------------------------
// pbc_wrap (src/pbc.F90:196-226) for replicas with mask[r] != 0.
// pbc_wrap of the replicas being rebuilt (src/pbc.F90:196-226), and their
// electrostatic cutoff for the new lists (src/neighbor_list.F90:80-82)
__global__ void k_wrap(Params P, Ptrs D, const int *mask) {
  int i = blockIdx.x * blockDim.x + threadIdx.x, r = blockIdx.y;
  if (i < 8 && r == 0) D.flags[i] = 0;   // (a block has more than eight threads)
  if (mask && !mask[r]) return;
  if (i == 0) D.ele_cut[r] = rebuild_ele_cut(P, D, r);
  if (i >= P.N || !P.pbc) return;
  const double *box = D.box + 3 * r;
  double4 &p = D.pos[(size_t)r * P.N + i];
  double v[3] = {p.x, p.y, p.z};
  for (int k = 0; k < 3; k++) {
    double L = box[k];
    if (v[k] > L) v[k] = v[k] - L * ((double)(int)((v[k] - L) / L) + 1);
    else if (v[k] < 0.0) v[k] = v[k] + L * ((double)(int)((0.0 - v[k]) / L) + 1);
  }
  p.x = v[0]; p.y = v[1]; p.z = v[2];
}

// ---------------------------------------------------------------------
// Base-pair eligibility of replica-local beads i < j (0-based) and the
// triplet-table index: the pair rules of src/init_bp.F90:184-313 (models
// 3/4/5); with a secondary-structure file only its pairs are considered
// (lines 206-209).  Returns table index (0 = not eligible); *bpt receives
// the BPT type.
__device__ __forceinline__ int is_comp(int a, int b) {
  return (a == SQ_A && b == SQ_U) || (a == SQ_U && (b == SQ_A || b == SQ_G)) ||
         (a == SQ_G && (b == SQ_C || b == SQ_U)) || (a == SQ_C && b == SQ_G);
}
__device__ __forceinline__ int hkey(int w, int x, int u, int z, int y, int v) {
  if (x < y) return 1 + w + x * 4 + u * 16 + z * 64 + y * 256 + v * 1024;
  return 1 + v + y * 4 + z * 16 + u * 64 + x * 256 + w * 1024;
}
__device__ __forceinline__ int bp_eligible(const Params &P, const Ptrs &D, int i, int j, int *bpt) {
  *bpt = 0;
  if (D.ss_off) {
    const int a = i < j ? i : j, b = i < j ? j : i;
    int lo = D.ss_off[a], hi = D.ss_off[a + 1];
    while (lo < hi) {
      const int m = (lo + hi) >> 1;
      if (D.ss_partner[m] < b) lo = m + 1; else hi = m;
    }
    if (lo == D.ss_off[a + 1] || D.ss_partner[lo] != b) return 0;
  }
  Topo ti = D.topo[i], tj = D.topo[j];
  int li = ti.loc, lj = tj.loc, ni = ti.len, nj = tj.len;
  bool ic = topo_circ(ti), jc = topo_circ(tj);
  int ipre = li - 1, inxt = li + 1, jpre = lj - 1, jnxt = lj + 1;
  if (ic) { if (li == 1) ipre = ni; if (li == ni) inxt = 1; }
  else if (li == 1 || li == ni) return 0;
  if (jc) { if (lj == 1) jpre = nj; if (lj == nj) jnxt = 1; }
  else if (lj == 1 || lj == nj) return 0;
  auto sq = [&](const Topo &t, int l) { return topo_seq(D.topo[t.start + l - 1]); };
  int s_i = topo_seq(ti), s_j = topo_seq(tj);
  int s_ipre = sq(ti, ipre), s_inxt = sq(ti, inxt), s_jpre = sq(tj, jpre), s_jnxt = sq(tj, jnxt);
  int p1 = is_comp(s_ipre, s_jnxt), p2 = is_comp(s_inxt, s_jpre);
  if (!ic && ipre == 1) p1 = 0;
  if (!jc && jnxt == nj) p1 = 0;
  if (!ic && inxt == ni) p2 = 0;
  if (!jc && jpre == 1) p2 = 0;
  int L = P.bp_min_loop;
  if (ti.start == tj.start) {
    if (li + L >= lj) return 0;
    if (li + 1 + L >= lj - 1) p2 = 0;
    if (ic) {
      if (lj + L >= li + ni) return 0;
      if (lj + 1 + L >= li - 1 + ni) p1 = 0;
    }
  }
  if ((P.bp_model >= 3) && !p1 && !p2) return 0;
  int t = 0;
  if (s_i == SQ_G && s_j == SQ_C) t = 1; else if (s_i == SQ_C && s_j == SQ_G) t = 4;
  else if (s_i == SQ_A && s_j == SQ_U) t = 2; else if (s_i == SQ_U && s_j == SQ_A) t = 5;
  else if (s_i == SQ_G && s_j == SQ_U) t = 3; else if (s_i == SQ_U && s_j == SQ_G) t = 6;
  *bpt = t;
  if (P.bp_model != 5) return t;
  int key;
  if (!p1) key = hkey(SQ_U, s_i, s_inxt, SQ_U, s_j, s_jpre);
  else if (!p2) key = hkey(s_ipre, s_i, SQ_U, s_jnxt, s_j, SQ_U);
  else key = hkey(s_ipre, s_i, s_inxt, s_jnxt, s_j, s_jpre);
  return D.bp3_hash[key];
}

// Pair criteria of src/neighbor_list.F90:123-223 for replica-local beads
// a != b of replica r: which of a's lists b belongs to (w: WCA, e:
// Debye-Hueckel, bp: base-pair candidate, owned by the lower bead).
struct PairHit {
  bool w, e, bp;
};
// whether the pair is within reach of any list, and its squared distance.
// Not so for a NaN distance, which none of the criteria would take: a run
// that has blown up rebuilds in every step and need not look at them.
__device__ __forceinline__ bool pair_near(const Params &P, const Ptrs &D, int r, int a, int b, const double4 &pa,
                                          const double4 &pb, double ele_cut2, double &d2) {
  const double4 &plo = a < b ? pa : pb;
  const double4 &phi = a < b ? pb : pa;
  double vx, vy, vz;
  pbc_vec(D.box + 3 * r, P.pbc, plo.x, plo.y, plo.z, phi.x, phi.y, phi.z, vx, vy, vz);
  d2 = dot_nc(vx, vy, vz, vx, vy, vz);
  return d2 <= ele_cut2 || d2 <= P.wca_nl_cut2 || d2 <= P.bp_nl_cut2;
}
// the lists of a near pair
__device__ __forceinline__ PairHit pair_rules(const Params &P, const Ptrs &D, int a, int b, double d2, double ele_cut2) {
  PairHit h{false, false, false};
  const int lo = a < b ? a : b, hi = a < b ? b : a;
  Topo tl = D.topo[lo], th = D.topo[hi];
  bool same = tl.start == th.start;
  int il = tl.loc, jl = th.loc, n = tl.len;
  bool circ = topo_circ(tl);
  // the analysis lists take no circular wrap into their exclusions
  // (src/list_exv.F90:34-38, src/list_ele.F90:35-46)
  const bool nl_rule = P.list_rule == 0;
  // WCA
  if (topo_seq(tl) != SQ_D && topo_seq(th) != SQ_D && d2 <= P.wca_nl_cut2) {
    h.w = true;
    if (same) {
      if (il + 2 >= jl) h.w = false;
      else if (nl_rule && circ && jl + 2 >= il + n) h.w = false;
    }
  }
  // Debye-Hueckel
  if (P.ele_on && d2 <= ele_cut2 && topo_charged(tl) && topo_charged(th)) {
    h.e = true;
    // list_ele tests the chain-local indices of every chain pair, the
    // neighbour list those of one chain only
    if (same || !nl_rule) {
      if (jl == il + 1 && P.ele_excl_bond) h.e = false;
      if (jl == il + 2 && P.ele_excl_angl) h.e = false;
    }
    if (same && nl_rule) {
      if (circ) {
        if (il == 1) {
          if (jl == n && P.ele_excl_bond) h.e = false;
          if (jl == n - 1 && P.ele_excl_angl) h.e = false;
        } else if (il == 2) {
          if (jl == n && P.ele_excl_angl) h.e = false;
        }
      }
    }
  }
  // base-pair candidates, owned by the lower bead; list_bp starts jmp at
  // imp + bp_min_loop + 1 over the whole system (src/list_bp.F90:41-42).
  // Candidates beyond the neighbour cutoff are left out in both rules:
  // they can form no pair, so no energy, force or limit-MC choice sees them.
  if (a < b && P.bp_model > 0 && d2 <= P.bp_nl_cut2 && (nl_rule || b >= a + P.bp_min_loop + 1)) {
    int bt;
    h.bp = bp_eligible(P, D, a, b, &bt) > 0;
  }
  return h;
}

// entries a's lists hold so far
struct SearchOut {
  int ne, nw, nb;
};
// b tested and appended to a's lists by one thread; most pairs are far, and
// end at one branch (with the tests of h behind it too, a search of 150 beads
// in a workgroup took 208 us for 195)
__device__ __forceinline__ void pair_test(const Params &P, const Ptrs &D, int r, int a, int b,
                                          const double4 &pa, const double4 &pb, double ele_cut2,
                                          SearchOut &o) {
  const int N = P.N;
  double d2;
  if (!pair_near(P, D, r, a, b, pa, pb, ele_cut2, d2)) return;
  const PairHit h = pair_rules(P, D, a, b, d2, ele_cut2);
  if (h.w) {
    if (o.nw < D.maxw) D.nb_wca[((size_t)r * D.maxw + o.nw) * N + a] = b;
    o.nw++;
  }
  if (h.e) {
    if (o.ne < D.maxnb) D.nb_ele[((size_t)r * D.maxnb + o.ne) * N + a] = b;
    o.ne++;
  }
  if (h.bp) {
    if (o.nb < D.maxbpb) D.bp_tmp[((size_t)r * N + a) * D.maxbpb + o.nb] = b;
    o.nb++;
  }
}

__device__ __forceinline__ void search_finish(const Params &P, const Ptrs &D, int r, int a,
                                              SearchOut &o) {
  size_t g = (size_t)r * P.N + a;
  D.n_ele[g] = o.ne;
  D.n_wca[g] = o.nw;
  int nb = o.nb < D.maxbpb ? o.nb : D.maxbpb;
  D.n_bp_tmp[g] = nb;
  // sort this bead's BP partners so the global list follows the
  // reference order (chain_i, chain_j, i, j)
  int *t = D.bp_tmp + g * D.maxbpb;
  for (int x = 1; x < nb; x++) {
    int v = t[x], y = x - 1;
    while (y >= 0 && t[y] > v) { t[y + 1] = t[y]; y--; }
    t[y + 1] = v;
  }
  if (o.ne > D.maxnb || o.nw > D.maxw || o.nb > D.maxbpb) {
    D.flags[0] = 1;
    atomicMax(&D.flags[2], o.ne);
    atomicMax(&D.flags[3], o.nw);
    atomicMax(&D.flags[4], o.nb);
  }
}

// The searches give a bead a wavefront: 64 candidates are tested at a time
// and appended in candidate order by prefix counts of ballots.  (A thread
// per bead walked its candidates one by one, each through dependent loads
// of its cell, position, topology and eligibility, with a few hundred
// threads in flight: 420 us for 9,400 beads, 68 us for 47.)
constexpr int SEARCH_WAVES = 4;
struct WaveSearch {
  SearchOut o;
  int *bp;   // 64 ints of LDS: the first base-pair partners
  __device__ __forceinline__ void add(const Params &P, const Ptrs &D, int r, int a, int b, const PairHit &h) {
    const int N = P.N;
    const unsigned long long mw = __ballot(h.w), me = __ballot(h.e), mb = __ballot(h.bp);
    const int kw = o.nw + below(mw), ke = o.ne + below(me), kb = o.nb + below(mb);
    if (h.w && kw < D.maxw) D.nb_wca[((size_t)r * D.maxw + kw) * N + a] = b;
    if (h.e && ke < D.maxnb) D.nb_ele[((size_t)r * D.maxnb + ke) * N + a] = b;
    if (h.bp) {
      if (kb < 64) bp[kb] = b;
      else if (kb < D.maxbpb) D.bp_tmp[((size_t)r * N + a) * D.maxbpb + kb] = b;
    }
    o.nw += __popcll(mw);
    o.ne += __popcll(me);
    o.nb += __popcll(mb);
  }
  // counts, partners in ascending order, capacity flags.  sorted: the
  // candidates came in ascending order
  __device__ __forceinline__ void finish(const Params &P, const Ptrs &D, int r, int a, bool sorted) {
    const int L = lane_id();
    const size_t g = (size_t)r * P.N + a;
    const int nb = o.nb < D.maxbpb ? o.nb : D.maxbpb, n = nb < 64 ? nb : 64;
    int *t = D.bp_tmp + g * D.maxbpb;
    wave_lds_fence();
    const int v = L < n ? bp[L] : 0x7fffffff;
    int rank = L;
    if (!sorted && nb <= 64) {
      rank = 0;
      for (int k = 0; k < n; k++) rank += bcast(v, k) < v;
    }
    if (L < n) t[rank] = v;
    if (L == 0) {
      D.n_ele[g] = o.ne;
      D.n_wca[g] = o.nw;
      D.n_bp_tmp[g] = nb;
      // the sizes to grow to.  A first search may overflow at every bead: a
      // maximum already there is only read (an atomic for each of 32,768
      // beads on one word took 2.4 ms)
      auto grow = [&](int k, int n) {
        if (__hip_atomic_load(&D.flags[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < n) atomicMax(&D.flags[k], n);
      };
      if (o.ne > D.maxnb || o.nw > D.maxw || o.nb > D.maxbpb) {
        grow(0, 1);
        grow(2, o.ne);
        grow(3, o.nw);
        grow(4, o.nb);
      }
    }
    if (!sorted && nb > 64) {
      // more than a wavefront holds: in memory, by one lane
      __threadfence();
      if (L == 0)
        for (int x = 1; x < nb; x++) {
          const int w = __hip_atomic_load(t + x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          int y = x - 1, u;
          while (y >= 0 && (u = __hip_atomic_load(t + y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) > w) {
            __hip_atomic_store(t + y + 1, u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            y--;
          }
          __hip_atomic_store(t + y + 1, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
  }
};

// All-pairs search (small systems or small boxes).
__global__ void __launch_bounds__(64 * SEARCH_WAVES) k_search_brute(Params P, Ptrs D, const int *mask) {
  __shared__ int s_bp[SEARCH_WAVES][64];
  const int N = P.N, L = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t g = (int64_t)blockIdx.x * SEARCH_WAVES + w;
  if (g >= (int64_t)P.R * N) return;
  const int r = (int)(g / N), a = (int)(g - (int64_t)r * N);
  if (L == 0) D.n_inc[g] = 0;
  if (mask && !mask[r]) return;
  const double4 *x = D.pos + (size_t)r * N;
  const double4 pa = x[a];
  const double ec = D.ele_cut[r] + P.nl_margin, ele_cut2 = P.ele_on ? ec * ec : 0.0;
  WaveSearch S{{0, 0, 0}, s_bp[w]};
  for (int b0 = 0; b0 < N; b0 += 64) {
    const int b = b0 + L;
    PairHit h{false, false, false};
    double d2;
    if (b < N && b != a && pair_near(P, D, r, a, b, pa, x[b], ele_cut2, d2)) h = pair_rules(P, D, a, b, d2, ele_cut2);
    S.add(P, D, r, a, b, h);
  }
  S.finish(P, D, r, a, true);
}

// Cell list: assignment / fill / per-cell sort / search.
__device__ __forceinline__ int cell_index(const Ptrs &D, int r, const double4 &p) {
  const double *box = D.box + 3 * r;
  int cx = (int)(p.x * D.ncell_x / box[0]), cy = (int)(p.y * D.ncell_y / box[1]),
      cz = (int)(p.z * D.ncell_z / box[2]);
  cx = min(max(cx, 0), D.ncell_x - 1);
  cy = min(max(cy, 0), D.ncell_y - 1);
  cz = min(max(cz, 0), D.ncell_z - 1);
  return (cz * D.ncell_y + cy) * D.ncell_x + cx;
}
__global__ void k_cell_count(Params P, Ptrs D, const int *mask) {
  int i = blockIdx.x * blockDim.x + threadIdx.x, r = blockIdx.y;
  if (i >= P.N || (mask && !mask[r])) return;
  int c = cell_index(D, r, D.pos[(size_t)r * P.N + i]);
  D.cell_of[(size_t)r * P.N + i] = c;
  atomicAdd(&D.cell_cnt[(size_t)r * D.ncell + c], 1);
}
__global__ void k_cell_fill(Params P, Ptrs D, const int *mask, int *fill) {
  int i = blockIdx.x * blockDim.x + threadIdx.x, r = blockIdx.y;
  if (i >= P.N || (mask && !mask[r])) return;
  size_t cg = (size_t)r * D.ncell + D.cell_of[(size_t)r * P.N + i];
  int slot = atomicAdd(&fill[cg], 1);
  D.cell_beads[D.cell_start[cg] + slot] = i;
}
// beads of a cell in ascending order: every bead counts the smaller ones of
// its cell (an insertion sort by a thread per cell took as long as its
// fullest cell: 74 us for 9,400 beads)
__global__ void k_cell_sort(Params P, Ptrs D, const int *mask, const int *filled) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x, r = blockIdx.y;
  if (i >= P.N || (mask && !mask[r])) return;
  const size_t cg = (size_t)r * D.ncell + D.cell_of[(size_t)r * P.N + i];
  const int s = D.cell_start[cg], e = D.cell_start[cg + 1];
  int rank = 0;
  for (int q = s; q < e; q++) rank += filled[q] < i;
  D.cell_beads[s + rank] = i;
}
// Cell-list search: lanes 0..26 read the bounds of the neighbouring cells,
// then the wavefront takes their beads 64 at a time in cell order.
__global__ void __launch_bounds__(64 * SEARCH_WAVES) k_search_cell(Params P, Ptrs D, const int *mask) {
  __shared__ int s_bp[SEARCH_WAVES][64], s_at[SEARCH_WAVES][28], s_off[SEARCH_WAVES][28];
  const int N = P.N, L = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t g = (int64_t)blockIdx.x * SEARCH_WAVES + w;
  if (g >= (int64_t)P.R * N) return;
  const int r = (int)(g / N), a = (int)(g - (int64_t)r * N);
  if (L == 0) D.n_inc[g] = 0;
  if (mask && !mask[r]) return;
  const double4 *x = D.pos + (size_t)r * N;
  const double4 pa = x[a];
  const double ec = D.ele_cut[r] + P.nl_margin, ele_cut2 = P.ele_on ? ec * ec : 0.0;
  const int c = D.cell_of[g];
  const int cx = c % D.ncell_x, cy = (c / D.ncell_x) % D.ncell_y, cz = c / (D.ncell_x * D.ncell_y);
  int at = 0, cnt = 0;
  if (L < 27) {
    const int nx = (cx + L % 3 - 1 + D.ncell_x) % D.ncell_x, ny = (cy + (L / 3) % 3 - 1 + D.ncell_y) % D.ncell_y,
              nz = (cz + L / 9 - 1 + D.ncell_z) % D.ncell_z;
    const size_t cg = (size_t)r * D.ncell + (nz * D.ncell_y + ny) * D.ncell_x + nx;
    at = D.cell_start[cg];
    cnt = D.cell_start[cg + 1] - at;
  }
  const int inc = wave_scan(cnt, 0, [](int p, int q) { return p + q; });
  const int total = bcast(inc, 26);
  if (L < 27) {
    s_at[w][L] = at;
    s_off[w][L] = inc - cnt;   // candidates before this cell
  }
  wave_lds_fence();
  WaveSearch S{{0, 0, 0}, s_bp[w]};
  for (int k0 = 0; k0 < total; k0 += 64) {
    const int k = k0 + L;
    PairHit h{false, false, false};
    int b = -1;
    if (k < total) {
      int lo = 0, hi = 26;   // the last cell with at most k candidates before it
      while (lo < hi) {
        const int m = (lo + hi + 1) >> 1;
        if (s_off[w][m] <= k) lo = m; else hi = m - 1;
      }
      b = D.cell_beads[s_at[w][lo] + k - s_off[w][lo]];
      double d2;
      if (b != a && pair_near(P, D, r, a, b, pa, x[b], ele_cut2, d2)) h = pair_rules(P, D, a, b, d2, ele_cut2);
    }
    S.add(P, D, r, a, b, h);
  }
  S.finish(P, D, r, a, false);
}

// ---------------------------------------------------------------------
// Exclusive scan (three passes) over n ints.
template <int B>
__global__ void k_scan_blocks(const int *in, int *out, int *bsum, int64_t n) {
  __shared__ int s[B];
  int64_t i = (int64_t)blockIdx.x * B + threadIdx.x;
  int v = i < n ? in[i] : 0;
  s[threadIdx.x] = v;
  __syncthreads();
  for (int off = 1; off < B; off <<= 1) {
    int t = threadIdx.x >= off ? s[threadIdx.x - off] : 0;
    __syncthreads();
    s[threadIdx.x] += t;
    __syncthreads();
  }
  if (i < n) out[i] = s[threadIdx.x] - v;
  if (threadIdx.x == B - 1) bsum[blockIdx.x] = s[B - 1];
}
template <int B>
__global__ void __launch_bounds__(B) k_scan_bsum(int *bsum, int nb, int *total, int *out_end) {
  __shared__ int s[B];
  const int t = threadIdx.x;
  int acc = 0;
  for (int k0 = 0; k0 < nb; k0 += B) {
    const int v = k0 + t < nb ? bsum[k0 + t] : 0;
    s[t] = v;
    __syncthreads();
    for (int off = 1; off < B; off <<= 1) {
      const int u = t >= off ? s[t - off] : 0;
      __syncthreads();
      s[t] += u;
      __syncthreads();
    }
    if (k0 + t < nb) bsum[k0 + t] = acc + s[t] - v;
    acc += s[B - 1];
    __syncthreads();
  }
  if (t == 0) {
    *total = acc;
    if (out_end) *out_end = acc;
  }
}
template <int B>
__global__ void k_scan_add(int *out, const int *bsum, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * B + threadIdx.x;
  if (i < n) out[i] += bsum[blockIdx.x];
}

// ---------------------------------------------------------------------
// Fill the BP candidate list (src/neighbor_list.F90:183-223) and scatter
// incidences.  bp_mp holds replica-local 1-based ids as the reference.
__global__ void k_bp_fill(Params P, Ptrs D, const int *mask) {
  int a = blockIdx.x * blockDim.x + threadIdx.x, r = blockIdx.y;
  if (a >= P.N || (mask && !mask[r])) return;
  const int N = P.N;
  size_t g = (size_t)r * N + a;
  int nb = D.n_bp_tmp[g], off = D.bp_off[g];
  Topo ti = D.topo[a];
  for (int k = 0; k < nb; k++) {
    int b = D.bp_tmp[g * D.maxbpb + k];
    int gb = off + k;
    if (gb >= D.maxbp) { D.flags[0] = 1; continue; }
    Topo tj = D.topo[b];
    int i = ti.loc, j = tj.loc, imp = a + 1, jmp = b + 1;
    int mp[7];
    mp[0] = imp;
    mp[1] = jmp;
    if (P.list_rule == 0) {
      mp[2] = (i == 1) ? imp + ti.len - 1 : imp - 1;
      mp[3] = (j == 1) ? jmp + tj.len - 1 : jmp - 1;
      mp[4] = (i == ti.len) ? imp + 1 - ti.len : imp + 1;
      // the reference compares j with the length of chain i here
      // (src/neighbor_list.F90:212); kept unless it leaves the system
      int m6 = (j == ti.len) ? jmp + 1 - tj.len : jmp + 1;
      if (P.fix_h4 || m6 < 1 || m6 > N) m6 = (j == tj.len) ? jmp + 1 - tj.len : jmp + 1;
      mp[5] = m6;
    } else {
      // list_bp wraps the neighbours of circular chains only and takes
      // each bead's own chain length (src/list_bp.F90:60-82)
      const bool ic = topo_circ(ti), jc = topo_circ(tj);
      mp[2] = (ic && i == 1) ? imp + ti.len - 1 : imp - 1;
      mp[3] = (jc && j == 1) ? jmp + tj.len - 1 : jmp - 1;
      mp[4] = (ic && i == ti.len) ? imp + 1 - ti.len : imp + 1;
      mp[5] = (jc && j == tj.len) ? jmp + 1 - tj.len : jmp + 1;
    }
    int bt;
    int h = bp_eligible(P, D, a, b, &bt);
    mp[6] = bt;
    int *dst = D.bp_mp + (size_t)gb * 8;
    for (int q = 0; q < 7; q++) dst[q] = mp[q];
    dst[7] = r;
    // the triplet table exists for model 5 only, other models read zeros
    // (src/init_bp.F90:39, src/neighbor_list.F90:220-221)
    D.bp_coef[2 * (size_t)gb] = P.bp_model == 5 ? D.bp3_dH[h] : 0.0;
    D.bp_coef[2 * (size_t)gb + 1] = P.bp_model == 5 ? D.bp3_dS[h] : 0.0;
    // reference list order: (chain_i, chain_j, i, j) for the neighbour list
    // (src/neighbor_list.F90:99-114), (imp, jmp) for list_bp
    // (src/list_bp.F90:41-42)
    if (P.list_rule == 0)
      D.bp_key[gb] = (((unsigned long long)(r * (int64_t)P.nchains + D.chain_id[a]) * P.nchains +
                       D.chain_id[b]) * P.maxlen + (i - 1)) * P.maxlen + (j - 1);
    else
      D.bp_key[gb] = ((unsigned long long)r * N + a) * N + b;
    D.bp_val[gb] = gb;
  }
}
// gather the candidate records into key order
__global__ void k_bp_permute(Ptrs D, int total, const int *order, int *mp_out, double *coef_out) {
  int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= total) return;
  int o = order[p];
  for (int q = 0; q < 8; q++) mp_out[(size_t)p * 8 + q] = D.bp_mp[(size_t)o * 8 + q];
  coef_out[2 * (size_t)p] = D.bp_coef[2 * (size_t)o];
  coef_out[2 * (size_t)p + 1] = D.bp_coef[2 * (size_t)o + 1];
}
// nbp_total < 0: the count of the current lists, read from the device (the
// end of the candidates' scan; graph replays launch over the capacity)
__device__ __forceinline__ int bp_count(const Params &P, const Ptrs &D, int nbp_total) {
  return nbp_total >= 0 ? nbp_total : D.bp_off[(size_t)P.R * P.N];
}

// incidences of each candidate on its six beads
__global__ void k_bp_inc(Params P, Ptrs D, int total) {
  int gb = blockIdx.x * blockDim.x + threadIdx.x;
  if (gb >= min(bp_count(P, D, total), D.maxbp)) return;
  const int *mp = D.bp_mp + (size_t)gb * 8;
  int r = mp[7];
  const int N = P.N;
  for (int q = 0; q < 6; q++) {
    size_t gq = (size_t)r * N + (mp[q] - 1);
    int slot = atomicAdd(&D.n_inc[gq], 1);
    if (slot < D.maxinc) D.inc[((size_t)r * D.maxinc + slot) * N + (mp[q] - 1)] = gb * 8 + q;
    else { D.flags[0] = 1; atomicMax(&D.flags[6], slot + 1); }
  }
}
// deterministic incidence order: each bead's list sorted by (candidate,
// role), in LDS up to 32 entries
__global__ void __launch_bounds__(64) k_inc_sort(Params P, Ptrs D, const int *mask) {
  __shared__ int s[32][64];
  const int t = threadIdx.x, a = blockIdx.x * 64 + t, r = blockIdx.y;
  if (a >= P.N || (mask && !mask[r])) return;
  const size_t g = (size_t)r * P.N + a;
  const int n = min(D.n_inc[g], D.maxinc);
  const size_t base = (size_t)r * D.maxinc * P.N + a, st = P.N;
  if (n <= 32) {
    for (int x = 0; x < n; x++) s[x][t] = D.inc[base + x * st];
    for (int x = 1; x < n; x++) {
      const int v = s[x][t];
      int y = x - 1;
      while (y >= 0 && s[y][t] > v) { s[y + 1][t] = s[y][t]; y--; }
      s[y + 1][t] = v;
    }
    for (int x = 0; x < n; x++) D.inc[base + x * st] = s[x][t];
  } else {
    for (int x = 1; x < n; x++) {
      int v = D.inc[base + x * st], y = x - 1;
      while (y >= 0 && D.inc[base + y * st] > v) { D.inc[base + (y + 1) * st] = D.inc[base + y * st]; y--; }
      D.inc[base + (y + 1) * st] = v;
    }
  }
  D.nt_cnt[g] = -P.max_bp_per_nt;
}

// per-nucleotide formed-pair counter, reset before each BP evaluation
__global__ void k_reset_cnt(Params P, Ptrs D, const int *mask) {
  int i = blockIdx.x * blockDim.x + threadIdx.x, r = blockIdx.y;
  if (i >= P.N || (mask && !mask[r])) return;
  D.nt_cnt[(size_t)r * P.N + i] = -P.max_bp_per_nt;
}

__device__ __forceinline__ int uf_find(int *p, int x) {
  while (true) {
    int q = p[x];
    if (q == x) return x;
    int qq = p[q];
    if (qq != q) atomicCAS(&p[x], q, qq);
    x = q;
  }
}

// one conflict component for the nucleotides a and b of a formed pair
// (larger root linked under the smaller)
__device__ __forceinline__ void uf_join(int *p, int a, int b) {
  while (true) {
    a = uf_find(p, a);
    b = uf_find(p, b);
    if (a == b) return;
    if (a > b) { int t = a; a = b; b = t; }
    if (atomicCAS(&p[b], b, a) == b) return;
  }
}

// ---------------------------------------------------------------------
// BP evaluation per candidate (src/force_bp_limit_triplet.F90:85-256 and
// src/force_bp_triplet.F90).  mc[r]: MC step for replica r.  ecT (may be
// null): temperature override per replica (energy at another condition).
template <typename T>
__global__ void k_bp_eval(Params P, Ptrs D, int nbp_total, const int *mc, const double *ecT,
                          const int *mask, int do_union) {
  int gb = blockIdx.x * blockDim.x + threadIdx.x;
  if (gb >= bp_count(P, D, nbp_total)) return;
  const int *mp = D.bp_mp + (size_t)gb * 8;
  int r = mp[7];
  if (mask && !mask[r]) return;
  const int N = P.N;
  D.bp_status[gb] = 0;
  D.ene_bp[gb] = 0.0;
  if (!mc[r] && P.nstep_bp_mc > 0 && !D.bp_status_mc[gb]) return;
  double tK = ecT ? ecT[r] : D.tK[r];
  // model 5: dG = dH - T dS of the triplet; models 1/3: U0 exp(-u) alone
  // (src/force_bp.F90:203)
  double dG = 1.0;
  if (P.bp_model == 5) {
    dG = D.bp_coef[2 * (size_t)gb] - tK * D.bp_coef[2 * (size_t)gb + 1];
    if (dG >= 0.0) return;
  }
  const double *box = D.box + 3 * r;
  const double4 *x = D.pos + (size_t)r * N;
  double4 p1 = x[mp[0] - 1], p2 = x[mp[1] - 1];
  V3<double> v12 = pvec(P, box, p1, p2), v13 = pvec(P, box, p1, x[mp[2] - 1]),
             v15 = pvec(P, box, p1, x[mp[4] - 1]), v42 = pvec(P, box, x[mp[3] - 1], p2),
             v62 = pvec(P, box, x[mp[5] - 1], p2);
  const BpPara &bp = D.bpp[mp[6]];
  T u;
  V3<T> fb[6];
  if (!bp_geom<T>(bp, v12, v13, v15, v42, v62, u, fb)) return;
  double e = bp.U0 * dG * exp(-(double)u);
  if (e <= P.bp_cutoff_energy) {
    D.bp_status[gb] = 1;
    D.ene_bp[gb] = e;
    double *fo = D.for_bp + (size_t)gb * 18;
    for (int q = 0; q < 6; q++) {
      fo[3 * q] = e * (double)fb[q].x;
      fo[3 * q + 1] = e * (double)fb[q].y;
      fo[3 * q + 2] = e * (double)fb[q].z;
    }
    atomicAdd(&D.nt_cnt[(size_t)r * N + mp[0] - 1], 1);
    atomicAdd(&D.nt_cnt[(size_t)r * N + mp[1] - 1], 1);
    // performance-form MC: one conflict component for the pair's nucleotides
    if (do_union && mc[r]) uf_join(D.comp + (size_t)r * N, mp[0] - 1, mp[1] - 1);
  }
}

// one base-pair candidate (src/force_bp_limit_triplet.F90:85-256);
// returns 1 if formed
template <typename T>
__device__ __forceinline__ int bp_eval_one(const Params &P, const Ptrs &D, int gb, int mc,
                                           const double4 *xr = nullptr, const int *mpl = nullptr,
                                           int *ntc = nullptr) {
  const int *mp = mpl ? mpl : D.bp_mp + (size_t)gb * 8;   // mpl: the same record staged in LDS
  const int r = mp[7];
  const int N = P.N;
  D.bp_status[gb] = 0;
  D.ene_bp[gb] = 0.0;
  if (!mc && P.nstep_bp_mc > 0 && !D.bp_status_mc[gb]) return 0;
  double tK = D.tK[r];
  double dG = 1.0;   // models 1/3: U0 exp(-u) (src/force_bp.F90:203)
  if (P.bp_model == 5) {
    dG = D.bp_coef[2 * (size_t)gb] - tK * D.bp_coef[2 * (size_t)gb + 1];
    if (dG >= 0.0) return 0;
  }
  const double *box = D.box + 3 * r;
  const double4 *x = xr ? xr : D.pos + (size_t)r * N;
  double4 p1 = x[mp[0] - 1], p2 = x[mp[1] - 1];
  V3<double> v12 = pvec(P, box, p1, p2), v13 = pvec(P, box, p1, x[mp[2] - 1]),
             v15 = pvec(P, box, p1, x[mp[4] - 1]), v42 = pvec(P, box, x[mp[3] - 1], p2),
             v62 = pvec(P, box, x[mp[5] - 1], p2);
  const BpPara &bp = D.bpp[mp[6]];
  T u;
  V3<T> fb[6];
  if (!bp_geom<T>(bp, v12, v13, v15, v42, v62, u, fb)) return 0;
  double e = bp.U0 * dG * exp(-(double)u);
  if (!(e <= P.bp_cutoff_energy)) return 0;   // also rejects a NaN energy
  D.bp_status[gb] = 1;
  D.ene_bp[gb] = e;
  double *fo = D.for_bp + (size_t)gb * 18;
  for (int q = 0; q < 6; q++) {
    fo[3 * q] = e * (double)fb[q].x;
    fo[3 * q + 1] = e * (double)fb[q].y;
    fo[3 * q + 2] = e * (double)fb[q].z;
  }
  int *cnt = ntc ? ntc : D.nt_cnt + (size_t)r * N;   // ntc: this replica's counts in LDS
  atomicAdd(&cnt[mp[0] - 1], 1);
  atomicAdd(&cnt[mp[1] - 1], 1);
  return 1;
}

// ---------------------------------------------------------------------
// Limit MC, parity form: the serial algorithm of
// src/force_bp_limit_triplet.F90:259-330 on the injected MT words of the
// replica, one thread.  Consumes words exactly as genrand_double3 /
// genrand_double1 would.
__global__ void k_mc_serial(Params P, Ptrs D, const int *mc, const double *ecT, int *ntlist,
                            int *bpseq, const int *mask) {
  if (threadIdx.x != 0) return;
  int r = blockIdx.x;
  if (mask && !mask[r]) return;
  if (!mc[r]) return;
  const int N = P.N;
  double tK = ecT ? ecT[r] : D.tK[r];
  double beta = mc_beta(P, tK, ecT == nullptr);
  int b0 = D.bp_off[(size_t)r * N], nb = D.bp_off[(size_t)(r + 1) * N] - b0;
  const uint32_t *w = D.tape + D.tape_off[r];
  int64_t pos = D.tape_pos[r], lim = D.tape_off[r + 1] - D.tape_off[r];
  int *cnt = D.nt_cnt + (size_t)r * N;
  int *nl = ntlist + (size_t)r * (N + 1);
  int *bs = bpseq + b0 + r;
  for (;;) {
    int nnt = 0;
    for (int k = 0; k < N; k++) if (cnt[k] > 0) nl[++nnt] = k + 1;
    if (nnt == 0) break;
    if (pos + 2 > lim) { D.flags[1] = 1; break; }
    double rnd = mt_d3(w[pos], w[pos + 1]); pos += 2;
    int ntd = nl[(int)ceil(rnd * nnt)];
    int ns = 0;
    for (int k = 0; k < nb; k++) {
      int gb = b0 + k;
      if (D.bp_status[gb]) {
        const int *mp = D.bp_mp + (size_t)gb * 8;
        if (mp[0] == ntd || mp[1] == ntd) bs[++ns] = gb;
      }
    }
    for (int k = 1; k <= ns; k++) {
      if (pos + 2 > lim) { D.flags[1] = 1; break; }
      rnd = mt_d3(w[pos], w[pos + 1]); pos += 2;
      int sw = (int)ceil(rnd * ns);
      int sv = bs[k]; bs[k] = bs[sw]; bs[sw] = sv;
    }
    if (ns == 0) { D.flags[1] = 2; break; }
    int del = bs[1];
    for (int k = 2; k <= ns; k++) {
      int jb = bs[k];
      double ratio = exp((D.ene_bp[jb] - D.ene_bp[del]) * beta);
      if (pos + 2 > lim) { D.flags[1] = 1; break; }
      rnd = mt_d1(w[pos], w[pos + 1]); pos += 2;
      if (rnd < ratio) del = jb;
    }
    D.bp_status[del] = 0;
    const int *mp = D.bp_mp + (size_t)del * 8;
    cnt[mp[0] - 1] -= 1;
    cnt[mp[1] - 1] -= 1;
  }
  D.tape_pos[r] = pos;
}

// Limit MC, performance form.  The excess-removal process of the reference
// decomposes over connected components of the formed-pair graph: a step
// only changes counts inside the component of the chosen nucleotide, and
// the uniform choice among all excess nucleotides restricted to one
// component is uniform within it.  Each component is therefore resolved
// independently with its own counter-RNG stream.
// Performance-form components: union-find roots, pairs bucketed per root
// (capacity SEGCAP per component), one wavefront per component with excess.
constexpr int SEGCAP = 256;
__global__ void k_comp_init(Params P, Ptrs D, int *seg_n, int *has_exc, const int *mask) {
  int i = blockIdx.x * blockDim.x + threadIdx.x, r = blockIdx.y;
  if (i >= P.N || (mask && !mask[r])) return;
  size_t g = (size_t)r * P.N + i;
  D.comp[g] = i;
  seg_n[g] = 0;
  has_exc[g] = 0;
}
// the per-step state of the performance-form MC in one pass: formed-pair
// counts (k_reset_cnt), union-find parents and buckets (k_comp_init), and
// the list of components with excess (its count in exc_list[0])
__global__ void k_mc_reset(Params P, Ptrs D, int *seg_n, int *has_exc, int *exc_list, const int *mask) {
  int i = blockIdx.x * blockDim.x + threadIdx.x, r = blockIdx.y;
  if (i == 0 && r == 0) exc_list[0] = 0;
  if (i >= P.N || (mask && !mask[r])) return;
  size_t g = (size_t)r * P.N + i;
  D.nt_cnt[g] = -P.max_bp_per_nt;
  D.comp[g] = i;
  seg_n[g] = 0;
  has_exc[g] = 0;
}
// formed pair gb into the bucket of its component; the component listed if
// it has excess (exc_list: [0] count, then replica * N + root)
__device__ __forceinline__ void seg_fill_one(const Params &P, const Ptrs &D, int gb, int *seg_n, int *seg, int *has_exc,
                                             int *exc_list) {
  const int *mp = D.bp_mp + (size_t)gb * 8;
  const int r = mp[7], N = P.N;
  int a = mp[0] - 1, b = mp[1] - 1;
  // the counts (final since the evaluation) are loaded before the dependent
  // chain of the root walk and the bucket atomic, not after it
  const bool exc = D.nt_cnt[(size_t)r * N + a] > 0 || D.nt_cnt[(size_t)r * N + b] > 0;
  int root = uf_find(D.comp + (size_t)r * N, a);
  size_t gr = (size_t)r * N + root;
  int slot = atomicAdd(&seg_n[gr], 1);
  if (slot < SEGCAP) seg[gr * SEGCAP + slot] = gb;
  if (exc && atomicExch(&has_exc[gr], 1) == 0) exc_list[1 + atomicAdd(&exc_list[0], 1)] = (int)gr;   // listed once
}
__global__ void k_seg_fill(Params P, Ptrs D, int nbp_total, int *seg_n, int *seg, int *has_exc,
                           const int *mc, const int *mask, int *exc_list) {
  int gb = blockIdx.x * blockDim.x + threadIdx.x;
  if (gb >= nbp_total || !D.bp_status[gb]) return;
  const int r = D.bp_mp[(size_t)gb * 8 + 7];
  if ((mask && !mask[r]) || !mc[r]) return;
  seg_fill_one(P, D, gb, seg_n, seg, has_exc, exc_list);
}
// serial fallback for a component larger than one wave holds: the same
// algorithm on global memory by one lane
// The arrays it touches come by value so that the callers' parameter
// structs stay in registers.
struct McArrays {
  const int *bp_mp;
  uint8_t *bp_status;
  const double *ene_bp;
  int *nt_cnt, *flags;
};
__device__ __noinline__ void mc_component_serial(const McArrays D, const int N, int r, int rk, int root, int *seg,
                                                 int n, double beta, uint64_t seed, int64_t step) {
  int *cnt = D.nt_cnt + (size_t)r * N;
  for (int t = 0; t < n; t++) {
    const int *mp = D.bp_mp + (size_t)seg[t] * 8;
    if (mp[0] < 1 || mp[0] > N || mp[1] < 1 || mp[1] > N) { D.flags[7] = 1; return; }
  }
  for (int x = 1; x < n; x++) {
    int v = seg[x], y = x - 1;
    while (y >= 0 && seg[y] > v) { seg[y + 1] = seg[y]; y--; }
    seg[y + 1] = v;
  }
  uint32_t draw = 0x10000u;
  int sq[64];
  for (int iter = 0; iter <= n; iter++) {
    // active nucleotides = endpoints with count > 0, ascending id
    int nact = 0, prev = -1;
    while (true) {
      int nxt = 0x7fffffff;
      for (int t = 0; t < n; t++) {
        const int *mp = D.bp_mp + (size_t)seg[t] * 8;
        int a = mp[0] - 1, b = mp[1] - 1;
        if (a > prev && a < nxt && cnt[a] > 0) nxt = a;
        if (b > prev && b < nxt && cnt[b] > 0) nxt = b;
      }
      if (nxt == 0x7fffffff) break;
      nact++;
      prev = nxt;
    }
    if (nact == 0) return;
    int pick = (int)ceil(philox_u(seed, rk, step, root, draw++) * nact), ntd = -1;
    prev = -1;
    for (int c = 0; c < pick; c++) {
      int nxt = 0x7fffffff;
      for (int t = 0; t < n; t++) {
        const int *mp = D.bp_mp + (size_t)seg[t] * 8;
        int a = mp[0] - 1, b = mp[1] - 1;
        if (a > prev && a < nxt && cnt[a] > 0) nxt = a;
        if (b > prev && b < nxt && cnt[b] > 0) nxt = b;
      }
      prev = nxt;
    }
    ntd = prev;
    int ns = 0;
    for (int t = 0; t < n && ns < 64; t++) {
      int gb = seg[t];
      const int *mp = D.bp_mp + (size_t)gb * 8;
      if (D.bp_status[gb] && (mp[0] - 1 == ntd || mp[1] - 1 == ntd)) sq[ns++] = gb;
    }
    if (ns == 0) { D.flags[1] = 2; return; }
    for (int i = 0; i < ns; i++) {
      int sw = (int)ceil(philox_u(seed, rk, step, root, draw++) * ns) - 1;
      int t = sq[i]; sq[i] = sq[sw]; sq[sw] = t;
    }
    int del = sq[0];
    for (int i = 1; i < ns; i++) {
      double ratio = exp((D.ene_bp[sq[i]] - D.ene_bp[del]) * beta);
      if (philox_u(seed, rk, step, root, draw++) < ratio) del = sq[i];
    }
    D.bp_status[del] = 0;
    const int *mp = D.bp_mp + (size_t)del * 8;
    cnt[mp[0] - 1] -= 1;
    cnt[mp[1] - 1] -= 1;
  }
}
__device__ __forceinline__ McArrays mc_arrays(const Ptrs &D) {
  return McArrays{D.bp_mp, D.bp_status, D.ene_bp, D.nt_cnt, D.flags};
}

// Scratch (ints) that mc_component_huge needs for a replica with nc
// candidates and N beads.
__device__ __forceinline__ size_t mc_huge_ints(int nc, int N) {
  const size_t pc = (size_t)((nc + 1) & ~1);
  const size_t nw = (size_t)(N + 31) / 32;
  return 8 * pc + ((nw + (size_t)N + 1) & ~(size_t)1) + 2 * (size_t)((N + 63) / 64);
}

// A component of any size (those above the bucket capacity SEGCAP): one
// wavefront, the state of the sweep in global scratch.  The sweep is that
// of mc_component_wave (an excess nucleotide picked uniformly in ascending
// id order, its formed pairs in list order, the reference's shuffle and
// Metropolis sweep, one deletion per iteration), on its own draws:
//   - the component's formed pairs come from a scan of the replica's
//     candidates [g0, g1) in order (list order kept), keeping those whose
//     union-find root is `root`;
//   - its nucleotides are listed in ascending id order through a bitmap
//     over bead ids;
//   - active nucleotides are 64-bit masks, updated on each deletion;
//   - each iteration's sequence is a ballot scan over the pairs, staged
//     through sseq (64 ints of LDS).
// comp is the replica's union-find array; scr holds cap ints.  Returns
// false if cap is too small.  Must be called by all 64 lanes of a wave
// with uniform arguments.
__device__ __noinline__ bool mc_component_huge(const McArrays D, const int N, int r, int rk, int root, int *comp,
                                               int g0, int g1, double beta, uint64_t seed, int64_t step, int *scr,
                                               size_t cap, int *sseq) {
  const int L = lane_id();
  root = __builtin_amdgcn_readfirstlane(root);
  const int nc = g1 - g0;
  if (mc_huge_ints(nc, N) > cap) return false;
  const size_t pc = (size_t)((nc + 1) & ~1);
  const int nw = (N + 31) / 32;
  int *hp = scr, *ha = hp + pc, *hb = ha + pc, *hua = hb + pc, *hub = hua + pc, *hal = hub + pc;
  double *he = reinterpret_cast<double *>(hal + pc);
  uint32_t *bm = reinterpret_cast<uint32_t *>(he + pc);
  int *hn = reinterpret_cast<int *>(bm + nw);
  unsigned long long *am = reinterpret_cast<unsigned long long *>(hn + ((nw + N + 1) & ~1) - nw);
  int *cnt = D.nt_cnt + (size_t)r * N;
  // ---- the component's formed pairs, in candidate order
  int n = 0;
  bool bad = false;
  for (int g = g0; g < g1; g += 64) {
    const int gb = g + L;
    bool in = false;
    int a = 0, b = 0;
    if (gb < g1 && D.bp_status[gb]) {
      const int *mp = D.bp_mp + (size_t)gb * 8;
      a = mp[0] - 1;
      b = mp[1] - 1;
      if (a < 0 || a >= N || b < 0 || b >= N) bad = true;
      else in = uf_find(comp, a) == root;
    }
    const unsigned long long m = __ballot(in);
    if (in) {
      const int t = n + below(m);
      hp[t] = gb; ha[t] = a; hb[t] = b; hua[t] = 0; hub[t] = 0; hal[t] = 1;
      he[t] = D.ene_bp[gb];
    }
    n += __popcll(m);
  }
  if (__ballot(bad)) {
    if (L == 0) D.flags[7] = 1;
    return true;
  }
  // ---- its nucleotides in ascending id order
  for (int w = L; w < nw; w += 64) bm[w] = 0u;
  __threadfence();
  for (int t = L; t < n; t += 64) {
    atomicOr(&bm[ha[t] >> 5], 1u << (ha[t] & 31));
    atomicOr(&bm[hb[t] >> 5], 1u << (hb[t] & 31));
  }
  __threadfence();
  int U = 0;
  for (int w0 = 0; w0 < nw; w0 += 64) {
    const int w = w0 + L;
    const uint32_t bits = w < nw ? bm[w] : 0u;
    const int c = __popc(bits), inc = wave_incl_scan(c);
    int k = U + inc - c;
    for (uint32_t x = bits; x; x &= x - 1) hn[k++] = 32 * w + __ffs(x) - 1;
    U += bcast(inc, 63);
  }
  __threadfence();
  // node index of each endpoint, then the active masks
  for (int t = L; t < n; t += 64) {
    int v = ha[t], lo = 0, hi = U;
    while (lo < hi) { const int mid = (lo + hi) >> 1; if (hn[mid] < v) lo = mid + 1; else hi = mid; }
    hua[t] = lo;
    v = hb[t]; lo = 0; hi = U;
    while (lo < hi) { const int mid = (lo + hi) >> 1; if (hn[mid] < v) lo = mid + 1; else hi = mid; }
    hub[t] = lo;
  }
  const int nuw = (U + 63) / 64;
  for (int u0 = 0; u0 < U; u0 += 64) {
    const int u = u0 + L;
    const unsigned long long m = __ballot(u < U && cnt[hn[u < U ? u : 0]] > 0);
    if (L == 0) am[u0 >> 6] = m;
  }
  __threadfence();
  // ---- the sweep: one deletion per iteration
  uint32_t draw = 0;
  for (int iter = 0; iter <= n; iter++) {
    int nact = 0;
    for (int w0 = 0; w0 < nuw; w0 += 64) {
      const int w = w0 + L;
      nact += bcast(wave_incl_scan(w < nuw ? __popcll(am[w]) : 0), 63);
    }
    if (nact == 0) break;
    const int pick = __builtin_amdgcn_readfirstlane((int)ceil(philox_u(seed, rk, step, root, draw) * nact));
    int ntu = -1, acc = 0;
    for (int w0 = 0; w0 < nuw && ntu < 0; w0 += 64) {
      const int w = w0 + L;
      const unsigned long long m = w < nuw ? am[w] : 0ull;
      const int c = __popcll(m), inc = wave_incl_scan(c), tot = bcast(inc, 63);
      if (acc + tot >= pick) {
        const int want = pick - acc - 1;
        const unsigned long long sel = __ballot(c > 0 && want >= inc - c && want < inc);
        const int ln = __ffsll((long long)sel) - 1;
        if (ln < 0) break;
        const unsigned long long mw = bcast64(m, ln);
        const int k = want - (bcast(inc, ln) - bcast(c, ln));
        const unsigned long long hit = __ballot(((mw >> L) & 1ull) && below(mw) == k);
        ntu = 64 * (w0 + ln) + __ffsll((long long)hit) - 1;
      }
      acc += tot;
    }
    ntu = __builtin_amdgcn_readfirstlane(ntu);
    if (ntu < 0 || ntu >= U) {   // masks and counts disagree: corrupted state
      if (L == 0) D.flags[7] = 1;
      return true;
    }
    const int ntd = __builtin_amdgcn_readfirstlane(hn[ntu]);
    // formed pairs of ntd in list order (the first 64)
    int ns = 0;
    for (int t0 = 0; t0 < n && ns < 64; t0 += 64) {
      const int t = t0 + L;
      const bool hit = t < n && hal[t] && (ha[t] == ntd || hb[t] == ntd);
      const unsigned long long m = __ballot(hit);
      if (hit) {
        const int k = ns + below(m);
        if (k < 64) sseq[k] = t;
      }
      ns += __popcll(m);
    }
    if (ns == 0) {
      if (L == 0) D.flags[1] = 2;
      return true;
    }
    if (ns > 64) ns = 64;
    wave_lds_fence();
    int seqv = L < ns ? sseq[L] : 0;
    // draws after the pick: shuffle 1..ns, Metropolis ns+1..2ns-1
    const int swl = L < ns ? (int)ceil(philox_u(seed, rk, step, root, draw + 1u + (uint32_t)L) * ns) - 1 : 0;
    const double lgl = (L >= 1 && L < ns) ? log(philox_u(seed, rk, step, root, draw + (uint32_t)(ns + L))) : 0.0;
    for (int i = 0; i < ns; i++) {
      const int sw = bcast(swl, i);
      const int ti = bcast(seqv, i), ts = bcast(seqv, sw);
      seqv = setlane(seqv, ts, i);
      seqv = setlane(seqv, ti, sw);
    }
    const double ev = L < ns ? he[seqv] : 0.0;
    int del = bcast(seqv, 0);
    double edel = bcast(ev, 0);
    for (int i = 1; i < ns; i++) {
      const double ej = bcast(ev, i);
      if (bcast(lgl, i) < (ej - edel) * beta) { del = bcast(seqv, i); edel = ej; }
    }
    draw += 2u * (uint32_t)ns;
    if (L == 0) {
      hal[del] = 0;
      D.bp_status[hp[del]] = 0;
      if (atomicSub(&cnt[ha[del]], 1) <= 1) atomicAnd(&am[hua[del] >> 6], ~(1ull << (hua[del] & 63)));
      if (atomicSub(&cnt[hb[del]], 1) <= 1) atomicAnd(&am[hub[del] >> 6], ~(1ull << (hub[del] & 63)));
    }
    __threadfence();
  }
  return true;
}

// Per-phase form: the components of replica r above SEGCAP pairs, by one
// wavefront (64 threads) after the others are resolved
__device__ __forceinline__ void mc_huge_replica(const Params &P, const Ptrs &D, int r, const int *seg_n, int *seg,
                                                const int *has_exc, const double *ecT, uint64_t seed, int64_t step) {
  const int L = threadIdx.x, N = P.N;
  __shared__ int sseq[64];
  const double tK = ecT ? ecT[r] : D.tK[r];
  const double beta = mc_beta(P, tK, ecT == nullptr);
  const int g0 = D.bp_off[(size_t)r * N], g1 = D.bp_off[(size_t)(r + 1) * N];
  int *scr = seg + (size_t)r * N * SEGCAP;
  for (int u0 = 0; u0 < N; u0 += 64) {
    const int root = u0 + L;
    bool h = false;
    if (root < N) {
      const size_t gr = (size_t)r * N + root;
      h = has_exc[gr] && seg_n[gr] > SEGCAP;
    }
    for (unsigned long long m = __ballot(h); m; m &= m - 1) {
      const int rt = bcast(root, __ffsll((long long)m) - 1);
      if (!mc_component_huge(mc_arrays(D), N, r, r, rt, D.comp + (size_t)r * N, g0, g1, beta, seed, step, scr,
                             (size_t)N * SEGCAP, sseq))
        if (L == 0) D.flags[5] = 1;
    }
  }
}
// ... for the replicas that k_mc_list marked
__global__ void __launch_bounds__(64) k_mc_huge(Params P, Ptrs D, const int *seg_n, int *seg, const int *has_exc,
                                                int *huge, const double *ecT, uint64_t seed, int64_t step) {
  const int r = blockIdx.x;
  if (!huge[r]) return;
  mc_huge_replica(P, D, r, seg_n, seg, has_exc, ecT, seed, step);
  if (threadIdx.x == 0) huge[r] = 0;
}
// one conflict component (root of replica r) resolved by a wavefront with
// MCB_LDS ints of LDS: one lane, the whole wave, or the serial fallback; a
// component above the bucket capacity is flagged in huge[r] (returns true)
__device__ __forceinline__ bool mc_one_component(const Params &P, const Ptrs &D, int r, int root, int *seg_n,
                                                 int *seg, const double *ecT, uint64_t seed, int64_t step,
                                                 int *huge, int *ws) {
  const int L = lane_id();
  size_t gr = (size_t)r * P.N + root;
  int n = seg_n[gr];
  double tK = ecT ? ecT[r] : D.tK[r];
  double beta = mc_beta(P, tK, ecT == nullptr);
  if (n > SEGCAP) {
    if (L == 0) huge[r] = 1;
    return true;
  }
  int *sg = seg + gr * SEGCAP;
  if (n <= MCL_PAIRS) {   // two pairs: one lane, same result
    if (L == 0 && !mc_component_lane(D, P.max_bp_per_nt, P.N, r, root, sg, n, beta, seed, step))
      mc_component_serial(mc_arrays(D), P.N, r, r, root, sg, n, beta, seed, step);
    return false;
  }
  if (!mc_component_wave_big(P, D, r, r, root, sg, n, beta, seed, step, ws) && L == 0) mc_component_serial(mc_arrays(D), P.N, r, r, root, sg, n, beta, seed, step);
  return false;
}

// The components listed by k_seg_fill (exc_list: [0] count, then
// replica * N + root), a grid-stride loop of 64-thread blocks.
__global__ void __launch_bounds__(64) k_mc_list(Params P, Ptrs D, int *seg_n, int *seg, const int *exc_list,
                                                const double *ecT, uint64_t seed, int64_t step, int *huge) {
  const int n = exc_list[0];
  __shared__ __align__(16) int ws[MCB_LDS];
  for (int k = blockIdx.x; k < n; k += gridDim.x) {
    const int gr = exc_list[1 + k];
    const int r = gr / P.N, root = gr - r * P.N;
    mc_one_component(P, D, r, root, seg_n, seg, ecT, seed, step, huge, ws);
  }
}

// ---------------------------------------------------------------------
// Parity noise: 3N (or `count`) normals per replica with the polar
// Box-Muller of src/rnd_boxmuller.F90 on the replica's MT words, replicas
// in order, sharing one cached value as the reference does.
__global__ void k_noise_parity(Params P, Ptrs D, int count, int dest, const int *mask) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  for (int r = 0; r < P.R; r++) {
    if (mask && !mask[r]) continue;
    const uint32_t *w = D.tape + D.tape_off[r];
    int64_t pos = D.tape_pos[r], lim = D.tape_off[r + 1] - D.tape_off[r];
    double *out = D.noise + (size_t)r * P.N * 3;
    for (int k = 0; k < count; k++) {
      double val;
      if (D.bm_cache[0] == 0.0) {
        D.bm_cache[0] = 1.0;
        double vx, vy, r2;
        for (;;) {
          if (pos + 4 > lim) { D.flags[1] = 1; D.tape_pos[r] = pos; return; }
          vx = 2.0 * mt_d1(w[pos], w[pos + 1]) - 1.0;
          vy = 2.0 * mt_d1(w[pos + 2], w[pos + 3]) - 1.0;
          pos += 4;
          r2 = vx * vx + vy * vy;
          if (r2 < 1.0 && r2 > 0.0) break;
        }
        double rf = sqrt(-2.0 * log(r2) / r2);
        D.bm_cache[1] = vx * rf;
        val = vy * rf;
      } else {
        D.bm_cache[0] = 0.0;
        val = D.bm_cache[1];
      }
      out[k] = val;
    }
    D.tape_pos[r] = pos;
  }
  (void)dest;
}

// ---------------------------------------------------------------------
// GJF-2GJ update of one bead (src/job_md.F90:415-444), or the
// Ermak-McCammon Brownian step (lines 446-456) when P.bd; g = r*N + a.
// Returns |move|^2.
//
// The Brownian move says which of its two products is rounded on its own:
// left to the compiler it depends on the code around it, and a run at a step
// where a bond is stiff (see k_step_force) turns that last bit into another
// trajectory.  It is the force's product, but for z in the kernels that keep
// the state through many steps (Z_NOISE: persistent, batched, jobs) the
// noise's: the forms that runs of either kind have had all along.
template <bool Z_NOISE = false>
__device__ __forceinline__ double move_bead(const Params &P, const Ptrs &D, size_t g, int a,
                                            const V3<double> &F, double n0, double n1, double n2) {
  const double cr = D.md_cr[g], ca = D.md_a[a];
  const double4 p = D.pos[g];
  double4 mv = D.move[g];
  double dx, dy, dz;
  if (P.bd) {
    // dx = (h/gamma) F + sqrt(2 kT h/gamma) xi; velocities are not used
    dx = __builtin_fma(cr, n0, ca * F.x);
    dy = __builtin_fma(cr, n1, ca * F.y);
    dz = Z_NOISE ? __builtin_fma(ca, F.z, cr * n2) : __builtin_fma(cr, n2, ca * F.z);
  } else {
    const double cf = D.md_cf[a], cx = D.md_cx[a];
    double4 v = D.vel[g];
    const double4 ac = D.acc[g];
    const double b0 = cr * n0, b1 = cr * n1, b2 = cr * n2;
    v.x = ca * v.x + cf * F.x + (ac.x + b0);
    v.y = ca * v.y + cf * F.y + (ac.y + b1);
    v.z = ca * v.z + cf * F.z + (ac.z + b2);
    dx = cx * v.x; dy = cx * v.y; dz = cx * v.z;
    D.vel[g] = v;
    D.acc[g] = double4{b0, b1, b2, 0.0};
  }
  D.frc[g] = double4{F.x, F.y, F.z, 0.0};
  mv.x += dx; mv.y += dy; mv.z += dz;
  D.move[g] = mv;
  // other beads still read D.pos in this pass: write the next buffer
  D.pos_out[g] = double4{p.x + dx, p.y + dy, p.z + dz, p.w};
  return dot_nc(mv.x, mv.y, mv.z, mv.x, mv.y, mv.z);
}

// Lane-split owner-computes: LPB lanes share bead a; lane l takes items
// l, l+LPB, ... of the bead's work list [bonded terms | WCA neighbours |
// DH neighbours | BP incidences]; partial forces are reduced with lane
// shuffles (FP64).
// Bonded terms of bead a (owner-computes): lane l of an LPB-lane group
// takes terms l, l+LPB, ... of [2 bonds | 3 angles | 4 dihedrals]
// (src/list_local.F90:24-104 enumerates the same terms).  FP64 always.
__device__ __forceinline__ V3<double> bonded_part(const Params &P, const Ptrs &D, int r, int a,
                                                  int l, int LPB, const double4 *xr = nullptr) {
  const int N = P.N;
  const double *box = D.box + 3 * r;
  const double4 *x = xr ? xr : D.pos + (size_t)r * N;
  const Topo ta = D.topo[a];
  const int loc = ta.loc, n = ta.len, st = ta.start;
  const bool circ = topo_circ(ta);
  const int nbond = P.dih_type ? 9 : 5;
  V3<double> F{0.0, 0.0, 0.0};
  for (int it = l; it < nbond; it += LPB) {
    const int m = it < 2 ? 2 : (it < 5 ? 3 : 4);
    const int p = it < 2 ? it : (it < 5 ? it - 2 : it - 5);
    int s0 = loc - p;
    bool ok;
    if (circ) { ok = n >= m; if (s0 < 1) s0 += n; }
    else ok = s0 >= 1 && s0 + m - 1 <= n;
    if (!ok) continue;
    auto bead = [&](int k) { int q = s0 + k; if (q > n) q -= n; return st + q - 1; };
    if (m == 2) {
      F = F + bond_force_p(P, pvec(P, box, x[bead(0)], x[bead(1)]), p);
    } else if (m == 3) {
      const double4 p1 = x[bead(1)];
      F = F + angle_force_p(P, pvec(P, box, x[bead(0)], p1), pvec(P, box, x[bead(2)], p1), p);
    } else {
      const double4 p1 = x[bead(1)], p2 = x[bead(2)];
      F = F + dih_force_p(P, pvec(P, box, x[bead(0)], p1), pvec(P, box, p2, p1),
                          pvec(P, box, p2, x[bead(3)]), p);
    }
  }
  return F;
}

// Pair terms of bead a: WCA and DH over the full neighbour lists in T,
// 6-bead BP forces gathered through the incidence list; FP64 sums.
// Pair forces on bead a, lane l of LPB: WCA and Debye-Hueckel neighbours
// (pair_nb), then the formed base pairs it takes part in (pair_bp), both
// accumulated onto F in that order.  pair_part is the two in sequence.
constexpr int PAIR_U = 4;   // neighbours a lane works on at a time
template <typename T>
__device__ __forceinline__ V3<double> pair_nb(const Params &P, const Ptrs &D, int r, int a, int l, int LPB,
                                              const double4 *xr, V3<double> F) {
  const int N = P.N;
  const double *box = D.box + 3 * r;
  const double4 *x = xr ? xr : D.pos + (size_t)r * N;
  const double4 pa = x[a];
  const size_t g = (size_t)r * N + a;
  const int nw = min(D.n_wca[g], D.maxw);
  const int ne = P.ele_on ? min(D.n_ele[g], D.maxnb) : 0;
  const T coef = (T)D.ele_coef[r], rc2 = (T)(D.ele_cut[r] * D.ele_cut[r]), rl = (T)(1.0 / D.lambdaD[r]);
  // neighbours in batches of PAIR_U: their index and position loads are all
  // issued before the arithmetic, and the arithmetic of a batch is
  // independent up to the sums; the summation order is unchanged
  const int *nbw = D.nb_wca + (size_t)r * D.maxw * N + a;
  for (int k0 = l; k0 < nw; k0 += PAIR_U * LPB) {
    int id[PAIR_U];
    double4 pb[PAIR_U];
    V3<T> f[PAIR_U];
#pragma unroll
    for (int u = 0; u < PAIR_U; u++) {
      const int k = k0 + u * LPB;
      id[u] = k < nw ? nbw[(size_t)k * N] : -1;
    }
#pragma unroll
    for (int u = 0; u < PAIR_U; u++) pb[u] = x[id[u] >= 0 ? id[u] : a];
#pragma unroll
    for (int u = 0; u < PAIR_U; u++) f[u] = wca_force<T>(P, cvt<T>(pvec(P, box, pa, pb[u])), id[u] >= 0);
#pragma unroll
    for (int u = 0; u < PAIR_U; u++) F = add_nc(F, cvt<double>(f[u]));
  }
  const int *nbe = D.nb_ele + (size_t)r * D.maxnb * N + a;
  for (int k0 = l; k0 < ne; k0 += PAIR_U * LPB) {
    int id[PAIR_U];
    double4 pb[PAIR_U];
    V3<T> f[PAIR_U];
#pragma unroll
    for (int u = 0; u < PAIR_U; u++) {
      const int k = k0 + u * LPB;
      id[u] = k < ne ? nbe[(size_t)k * N] : -1;
    }
#pragma unroll
    for (int u = 0; u < PAIR_U; u++) pb[u] = x[id[u] >= 0 ? id[u] : a];
#pragma unroll
    for (int u = 0; u < PAIR_U; u++) f[u] = dh_force<T>(coef, rc2, rl, cvt<T>(pvec(P, box, pa, pb[u])), id[u] >= 0);
#pragma unroll
    for (int u = 0; u < PAIR_U; u++) F = add_nc(F, cvt<double>(f[u]));
  }
  return F;
}

__device__ __forceinline__ V3<double> pair_bp(const Params &P, const Ptrs &D, int r, int a, int l, int LPB,
                                              V3<double> F) {
  const int N = P.N;
  const size_t g = (size_t)r * N + a;
  const int ni = min(D.n_inc[g], D.maxinc);
  const int *inc = D.inc + (size_t)r * D.maxinc * N + a;
  for (int k = l; k < ni; k += LPB) {
    int e = inc[(size_t)k * N], gb = e >> 3, role = e & 7;
    if (D.bp_status[gb]) {
      const double *fo = D.for_bp + (size_t)gb * 18 + 3 * role;
      F.x += fo[0]; F.y += fo[1]; F.z += fo[2];
    }
  }
  return F;
}

// pair_bp of a bead by one lane: incidences in batches of four, their
// loads issued before the sums
__device__ __forceinline__ V3<double> pair_bp4(const Params &P, const Ptrs &D, int r, int a, V3<double> F) {
  const int N = P.N;
  const int ni = min(D.n_inc[(size_t)r * N + a], D.maxinc);
  const int *inc = D.inc + (size_t)r * D.maxinc * N + a;
  for (int k0 = 0; k0 < ni; k0 += 4) {
    int e[4];
    bool on[4];
#pragma unroll
    for (int u = 0; u < 4; u++) e[u] = k0 + u < ni ? inc[(size_t)(k0 + u) * N] : -1;
#pragma unroll
    for (int u = 0; u < 4; u++) on[u] = e[u] >= 0 && D.bp_status[e[u] >> 3];
#pragma unroll
    for (int u = 0; u < 4; u++)
      if (on[u]) {
        const double *fo = D.for_bp + (size_t)(e[u] >> 3) * 18 + 3 * (e[u] & 7);
        F.x += fo[0]; F.y += fo[1]; F.z += fo[2];
      }
  }
  return F;
}

template <typename T>
__device__ __forceinline__ V3<double> pair_part(const Params &P, const Ptrs &D, int r, int a, int l,
                                                int LPB, const double4 *xr = nullptr) {
  return pair_bp(P, D, r, a, l, LPB, pair_nb<T>(P, D, r, a, l, LPB, xr, V3<double>{0.0, 0.0, 0.0}));
}

// The three normal draws of bead a on `step` (counter RNG; rk keys the
// replica's stream)
__device__ __forceinline__ void noise_normals(uint64_t seed, int rk, int64_t step, int a, double &n0, double &n1,
                                              double &n2) {
  uint32_t k1 = (uint32_t)(seed >> 32) ^ (0x9e3779b9u * (uint32_t)(rk + 1));
  U4 o = philox(U4{(uint32_t)step, (uint32_t)(step >> 32), (uint32_t)a, 0x6e6f6973u}, (uint32_t)seed, k1);
  U4 o2 = philox(U4{(uint32_t)step, (uint32_t)(step >> 32), (uint32_t)a, 0x6e6f6974u}, (uint32_t)seed, k1);
  double u1 = u01(o.x, o.y), u2 = u01(o.z, o.w), u3 = u01(o2.x, o2.y), u4 = u01(o2.z, o2.w);
  double rr = sqrt(-2.0 * log(u1)), r2 = sqrt(-2.0 * log(u3));
  n0 = rr * cos(6.283185307179586 * u2);
  n1 = rr * sin(6.283185307179586 * u2);
  n2 = r2 * cos(6.283185307179586 * u4);
}

// One bead's update with its noise draws (the injected MT words in the
// parity form, else the counter RNG); r indexes the per-replica arrays,
// rk keys the random stream.
template <bool Z_NOISE = false>
__device__ __forceinline__ double gjf_update(const Params &P, const Ptrs &D, int r, int rk, int a,
                                             const V3<double> &F, int parity, uint64_t seed,
                                             int64_t step) {
  size_t g = (size_t)r * P.N + a;
  double n0, n1, n2;
  if (parity) {
    const double *nz = D.noise + g * 3;
    n0 = nz[0]; n1 = nz[1]; n2 = nz[2];
  } else {
    noise_normals(seed, rk, step, a, n0, n1, n2);
  }
  return move_bead<Z_NOISE>(P, D, g, a, F, n0, n1, n2);
}

template <int LPB>
__device__ __forceinline__ V3<double> group_sum(V3<double> F) {
#pragma unroll
  for (int off = LPB / 2; off > 0; off >>= 1) {
    F.x += __shfl_xor(F.x, off, LPB);
    F.y += __shfl_xor(F.y, off, LPB);
    F.z += __shfl_xor(F.z, off, LPB);
  }
  return F;
}

// bonded forces per bead into D.fbond (FP64)
template <int LPB, int B>
__global__ void __launch_bounds__(B) k_bonded(Params P, Ptrs D, const int *mask) {
  const int grp = threadIdx.x / LPB, l = threadIdx.x % LPB;
  const int a = blockIdx.x * (B / LPB) + grp, r = blockIdx.y;
  const bool act = a < P.N && !(mask && !mask[r]);
  V3<double> F{0.0, 0.0, 0.0};
  if (act) F = bonded_part(P, D, r, a, l, LPB);
  F = group_sum<LPB>(F);
  if (act && l == 0) D.fbond[(size_t)r * P.N + a] = double4{F.x, F.y, F.z, 0.0};
}

// top two of (a1 >= a2) and (b1 >= b2): the two largest values of the four
__device__ __forceinline__ void top2_merge(double &m1, double &m2, double b1, double b2) {
  const double n1 = m1 > b1 ? m1 : b1;
  const double n2 = m1 > b1 ? (m2 > b1 ? m2 : b1) : (m1 > b2 ? m1 : b2);
  m1 = n1;
  m2 = n2;
}

// Workgroups are dispatched to the eight XCDs in turn (linear ID mod 8),
// each XCD with its own L2.  xcd_tile maps a linear workgroup ID to a tile
// so that XCD x takes the x-th contiguous slice of the n tiles: the
// position and list gathers of one XCD's workgroups then fall mostly on
// beads its own L2 already holds.  One-to-one for any n.
__device__ __forceinline__ int xcd_tile(int id, int n) {
  const int q = n >> 3, rem = n & 7, x = id & 7;
  return x * q + min(x, rem) + (id >> 3);
}

// Force of every bead and its update in one pass: LPB lanes a bead over the
// pair lists, the base-pair incidences and the bonded terms.  g_own: the
// bead this thread updated (unchanged if none).
template <typename T, int LPB, int B>
__device__ __forceinline__ void force_lanes(const Params &P, const Ptrs &D, int integrate, int parity, uint64_t seed,
                                            int64_t step, const int *mask, int bonded_inline, double *top2, int &g_own) {
  __shared__ double s1[B / LPB], s2[B / LPB];
  const int grp = threadIdx.x / LPB, l = threadIdx.x % LPB;
  // tile (bx, r) of this workgroup: grid x = tiles of a replica, y = replicas
  const int tile = xcd_tile(blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y);
  const int bx = tile % gridDim.x, r = tile / gridDim.x;
  const int a = bx * (B / LPB) + grp;
  const int N = P.N;
  const bool act = a < N && !(mask && !mask[r]);
  // bonded forces here (bonded_inline) or from k_bonded's D.fbond (which
  // external terms add to): the same lanes and sums either way
  V3<double> Fb{0.0, 0.0, 0.0};
  if (bonded_inline) {
    if (act) Fb = bonded_part(P, D, r, a, l, LPB);
    Fb = group_sum<LPB>(Fb);
  }
  V3<double> F{0.0, 0.0, 0.0};
  if (act) F = pair_part<T>(P, D, r, a, l, LPB);
  F = group_sum<LPB>(F);
  double d2 = 0.0;
  if (act && l == 0) {
    size_t g = (size_t)r * N + a;
    const double4 fb = bonded_inline ? double4{Fb.x, Fb.y, Fb.z, 0.0} : D.fbond[g];
    F.x += fb.x; F.y += fb.y; F.z += fb.z;
    D.nt_cnt[g] = -P.max_bp_per_nt;
    g_own = (int)g;
    if (!integrate) D.frc[g] = double4{F.x, F.y, F.z, 0.0};
    else d2 = gjf_update(P, D, r, r, a, F, parity, seed, step);
  }
  if (!integrate) return;
  if (l == 0) { s1[grp] = d2; s2[grp] = 0.0; }
  __syncthreads();
  for (int off = (B / LPB) / 2; off > 0; off >>= 1) {
    if (threadIdx.x < off) {
      double a1 = s1[threadIdx.x], a2 = s2[threadIdx.x], b1 = s1[threadIdx.x + off], b2 = s2[threadIdx.x + off];
      s1[threadIdx.x] = a1 > b1 ? a1 : b1;
      s2[threadIdx.x] = a1 > b1 ? (a2 > b1 ? a2 : b1) : (a1 > b2 ? a1 : b2);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    top2[((size_t)r * gridDim.x + bx) * 2] = s1[0];
    top2[((size_t)r * gridDim.x + bx) * 2 + 1] = s2[0];
  }
}
template <typename T, int LPB, int B>
__global__ void __launch_bounds__(B) k_force_lanes(Params P, Ptrs D, int integrate, int parity, uint64_t seed,
                                                  int64_t step, const int *mask, int bonded_inline) {
  int g;
  force_lanes<T, LPB, B>(P, D, integrate, parity, seed, step, mask, bonded_inline, D.blk_top2, g);
}


// skin test per replica (src/job_md.F90:376-395): sqrt(d2max) +
// sqrt(d2max_2nd) > nl_margin over the top-2 displacements of nblk blocks
// (top2), reduced by a workgroup (the top two are the same values in any
// order).
template <int B>
__global__ void __launch_bounds__(B) k_skin(Params P, Ptrs D, const double *top2, int nblk) {
  __shared__ double s1[B], s2[B];
  const int r = blockIdx.x, t = threadIdx.x;
  double m1 = 0.0, m2 = 0.0;
  for (int b = t; b < nblk; b += B) top2_merge(m1, m2, top2[((size_t)r * nblk + b) * 2], top2[((size_t)r * nblk + b) * 2 + 1]);
  s1[t] = m1;
  s2[t] = m2;
  __syncthreads();
  for (int off = B / 2; off > 0; off >>= 1) {
    if (t < off) {
      double a1 = s1[t], a2 = s2[t];
      top2_merge(a1, a2, s1[t + off], s2[t + off]);
      s1[t] = a1;
      s2[t] = a2;
    }
    __syncthreads();
  }
  if (t == 0) D.rebuild_flag[r] = (sqrt(s1[0]) + sqrt(s2[0]) > P.nl_margin) ? 1 : 0;
}

// Bead state between the host's xyz(3, nmp, nrep) and the device's double4.
// The copy over PCIe is the bound; packed here, it moves 24 bytes a bead and
// the host does no loop of its own (one core packing 94,000 beads into a
// vector of 32-byte rows took longer than the copy: 100 steps with state in
// and out 45.6 -> 43.7 ms).
__global__ void k_state_in(const double *src, double4 *dst, size_t n) {
  const size_t g = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g < n) dst[g] = double4{src[3 * g], src[3 * g + 1], src[3 * g + 2], 0.0};
}
__global__ void k_state_out(const double4 *src, double *dst, size_t n) {
  const size_t g = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= n) return;
  const double4 v = src[g];
  dst[3 * g] = v.x; dst[3 * g + 1] = v.y; dst[3 * g + 2] = v.z;
}

__global__ void k_clear_move(Params P, Ptrs D, const int *mask) {
  int i = blockIdx.x * blockDim.x + threadIdx.x, r = blockIdx.y;
  if (i >= P.N || (mask && !mask[r])) return;
  D.move[(size_t)r * P.N + i] = double4{0, 0, 0, 0};
}

// velocities / initial noise terms (src/job_md.F90:157-176); parity uses
// the noise buffer filled twice (velocities then accelerations).
__global__ void k_init_vel(Params P, Ptrs D, int which, int parity, uint64_t seed,
                           const int *mask) {
  int a = blockIdx.x * blockDim.x + threadIdx.x, r = blockIdx.y;
  if (a >= P.N || (mask && !mask[r])) return;
  size_t g = (size_t)r * P.N + a;
  double n0, n1, n2;
  if (parity) {
    n0 = D.noise[3 * g]; n1 = D.noise[3 * g + 1]; n2 = D.noise[3 * g + 2];
  } else {
    U4 o = philox(U4{0xffffffffu, (uint32_t)which, (uint32_t)a, 0x696e6974u}, (uint32_t)seed,
                  (uint32_t)(seed >> 32) ^ (0x9e3779b9u * (uint32_t)(r + 1)));
    U4 o2 = philox(U4{0xfffffffeu, (uint32_t)which, (uint32_t)a, 0x696e6974u}, (uint32_t)seed,
                   (uint32_t)(seed >> 32) ^ (0x9e3779b9u * (uint32_t)(r + 1)));
    double rr = sqrt(-2.0 * log(u01(o.x, o.y))), r2 = sqrt(-2.0 * log(u01(o2.x, o2.y)));
    n0 = rr * cos(6.283185307179586 * u01(o.z, o.w));
    n1 = rr * sin(6.283185307179586 * u01(o.z, o.w));
    n2 = r2 * cos(6.283185307179586 * u01(o2.z, o2.w));
  }
  if (which == 0) {
    const double BOLTZ = 1.380649e-23 * ((1.0 / 4184.0) * 6.02214076e23);
    double c = sqrt(D.tK[r] * BOLTZ / D.mass[a]);
    D.vel[g] = double4{c * n0, c * n1, c * n2, 0.0};
  } else {
    double cr = D.md_cr[g];
    D.acc[g] = double4{cr * n0, cr * n1, cr * n2, 0.0};
  }
}

// rescale velocities of replica r by f (replica exchange,
// src/replica_exchange.F90:175-213)
__global__ void k_scale_vel(Params P, Ptrs D, int r, double f, int divide) {
  int a = blockIdx.x * blockDim.x + threadIdx.x;
  if (a >= P.N) return;
  double4 &v = D.vel[(size_t)r * P.N + a];
  if (divide) { v.x = v.x / f; v.y = v.y / f; v.z = v.z / f; }
  else { v.x = f * v.x; v.y = f * v.y; v.z = f * v.z; }
}

// ---------------------------------------------------------------------
// Energy terms of bead a of replica r into e[1..6] (src/energy_sumup.F90
// and the terms): 1 bond, 2 angle, 3 dihedral, 4 BP, 5 WCA, 6 DH.  Each
// term is counted once: on the first bead of a bonded term, the lower bead
// of a pair, the owner (role 0) of a base-pair candidate.  coef / rlam: the
// DH coefficient and inverse Debye length to use; bp_masked: sum only the
// pairs that survived the limit MC (src/energy_bp_limit_triplet.F90:195),
// else all formed ones (src/energy_bp_triplet.F90:88).
// Lane l of LPB takes its share of the bead's terms.
__device__ __forceinline__ void bead_energy(const Params &P, const Ptrs &D, int r, int a, double coef,
                                            double rc, int bp_masked, const double4 *x, double e[7], int l = 0,
                                            int LPB = 1) {
  const int N = P.N;
  const double *box = D.box + 3 * r;
  Topo ta = D.topo[a];
  int loc = ta.loc, n = ta.len, st = ta.start;
  bool circ = topo_circ(ta);
  auto at = [&](int k) { int l = loc + k; if (l > n) l -= n; return st + l - 1; };
  // bond starting at this bead
  if (l == 0 && (circ || loc + 1 <= n)) {
    V3<double> v = pvec(P, box, x[at(0)], x[at(1)]);
    double d = sqrt(dot(v, v));
    e[1] += 0.5 * P.bond_k * ((d - P.bond_r0) * (d - P.bond_r0));
  }
  if (l == 1 % LPB && ((circ && n >= 3) || loc + 2 <= n)) {
    V3<double> v12 = pvec(P, box, x[at(0)], x[at(1)]), v32 = pvec(P, box, x[at(2)], x[at(1)]);
    double co = dot(v32, v12) / sqrt(dot(v12, v12) * dot(v32, v32));
    if (P.angl_reb) {
      e[2] += 0.5 * P.angl_k * ((co - P.angl_co0) * (co - P.angl_co0)) / (1.0 - co * co);
    } else {
      if (co > 1.0) co = 1.0; else if (co < -1.0) co = -1.0;
      double t = acos(co);
      e[2] += 0.5 * P.angl_k * ((t - P.angl_t0) * (t - P.angl_t0));
    }
  }
  if (l == 2 % LPB && P.dih_type && ((circ && n >= 4) || loc + 3 <= n)) {
    V3<double> v12 = pvec(P, box, x[at(1)], x[at(0)]), v23 = pvec(P, box, x[at(2)], x[at(1)]),
               v34 = pvec(P, box, x[at(3)], x[at(2)]);
    V3<double> c1 = cross(v12, v23), c2 = cross(v23, v34);
    double dih = atan2(sqrt(dot(v23, v23)) * dot(v12, c2), dot(c1, c2));
    if (P.dih_type == 2) e[3] -= P.dih_k * exp(-0.5 * P.dih_w * ((dih - P.dih_p0) * (dih - P.dih_p0)));
    else e[3] += P.dih_k * (1.0 + cos(dih + P.dih_p0));
  }
  size_t g = (size_t)r * N + a;
  {
    int ni = min(D.n_inc[g], D.maxinc);
    const int *inc = D.inc + (size_t)r * D.maxinc * N + a;
    for (int k = l; k < ni; k += LPB) {
      int q = inc[(size_t)k * N];
      if ((q & 7) == 0 && (D.bp_status[q >> 3] || !bp_masked)) e[4] += D.ene_bp[q >> 3];
    }
  }
  {
    int nw = min(D.n_wca[g], D.maxw);
    const int *nb = D.nb_wca + (size_t)r * D.maxw * N + a;
    for (int k = l; k < nw; k += LPB) {
      int b = nb[(size_t)k * N];
      if (b < a) continue;
      V3<double> v = pvec(P, box, x[a], x[b]);
      double d = sqrt(dot(v, v));
      if (d >= P.wca_sigma) continue;
      d = P.wca_sigma / d;
      double d6 = d * d * d * d * d * d;
      e[5] += P.wca_eps * (d6 * d6 - 2 * d6 + 1.0);
    }
  }
  if (P.ele_on) {
    int ne = min(D.n_ele[g], D.maxnb);
    const int *nb = D.nb_ele + (size_t)r * D.maxnb * N + a;
    for (int k = l; k < ne; k += LPB) {
      int b = nb[(size_t)k * N];
      if (b < a) continue;
      V3<double> v = pvec(P, box, x[a], x[b]);
      double dist = sqrt(dot(v, v));
      if (dist > D.ele_cut[r]) continue;
      e[6] += coef / dist * exp(-dist * rc);
    }
  }
}

// Energies (src/energy_sumup.F90): per-block partial sums of bead_energy,
// ENE_LPB lanes a bead (one lane walked its lists in 33 us for 47 beads),
// reduced in a fixed order.  r_only >= 0: one replica, grid.y = 1, its DH
// coefficient and Debye length by value (coef1, lam1) and its partial
// sums in slot 0 of `partial`.
constexpr int ENE_LPB = 4;
template <int B>
__global__ void __launch_bounds__(B *ENE_LPB) k_energy(Params P, Ptrs D, const double *ecT,
                                              const double *eCoef, const double *eLam,
                                              double *partial, const int *mask, int bp_masked,
                                              int r_only, double coef1, double lam1) {
  __shared__ double s[7][B];
  const int t = threadIdx.x / ENE_LPB, l = threadIdx.x % ENE_LPB;
  int a = blockIdx.x * B + t, r = r_only >= 0 ? r_only : blockIdx.y;
  const int slot = r_only >= 0 ? 0 : r;
  const int N = P.N;
  double e[7] = {0, 0, 0, 0, 0, 0, 0};
  if (a < N && !(mask && !mask[r])) {
    double coef = r_only >= 0 ? coef1 : (eCoef ? eCoef[r] : D.ele_coef[r]);
    double rc = 1.0 / (r_only >= 0 ? lam1 : (eLam ? eLam[r] : D.lambdaD[r]));
    bead_energy(P, D, r, a, coef, rc, bp_masked, D.pos + (size_t)r * N, e, l, ENE_LPB);
  }
  (void)ecT;
  for (int k = 1; k < 7; k++) {
    for (int off = 1; off < ENE_LPB; off <<= 1) e[k] += __shfl_xor(e[k], off);
    if (l == 0) s[k][t] = e[k];
  }
  __syncthreads();
  for (int off = B / 2; off > 0; off >>= 1) {
    if (threadIdx.x < off)
      for (int k = 1; k < 7; k++) s[k][threadIdx.x] += s[k][threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0)
    for (int k = 1; k < 7; k++) partial[((size_t)slot * gridDim.x + blockIdx.x) * 8 + k] = s[k][0];
}
// energy_kinetic (src/energy_kinetic.F90:16-29): 0.5 sum m |v|^2 of
// replica blockIdx.x, one workgroup per replica, FP64 tree sum.
template <int B>
__global__ void __launch_bounds__(B) k_kinetic(Params P, Ptrs D, double *out) {
  __shared__ double s[B];
  const int r = blockIdx.x, N = P.N;
  double e = 0.0;
  for (int a = threadIdx.x; a < N; a += B) {
    const double4 v = D.vel[(size_t)r * N + a];
    e += D.mass[a] * (v.x * v.x + v.y * v.y + v.z * v.z);
  }
  s[threadIdx.x] = e;
  __syncthreads();
  for (int off = B / 2; off > 0; off >>= 1) {
    if (threadIdx.x < off) s[threadIdx.x] += s[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[r] = 0.5 * s[0];
}

// ext: stage, tweezers, Rg and restraint energies [4*R], or null.
// r_only >= 0: that replica alone, partial sums and output in slot 0.
__global__ void k_energy_reduce(const double *partial, int nblk, double *out, const double *ext, int r_only) {
  const int r = r_only >= 0 ? r_only : blockIdx.x, slot = r_only >= 0 ? 0 : r;
  if (threadIdx.x != 0) return;
  double e[11] = {0};
  for (int b = 0; b < nblk; b++)
    for (int k = 1; k < 7; k++) e[k] += partial[((size_t)slot * nblk + b) * 8 + k];
  if (ext)
    for (int k = 0; k < 4; k++) e[7 + k] = ext[4 * r + k];
  double t = 0.0;
  for (int k = 1; k <= 10; k++) t += e[k];
  e[0] = t;
  for (int k = 0; k < 11; k++) out[(size_t)slot * 16 + k] = e[k];
}

}  // namespace sis
