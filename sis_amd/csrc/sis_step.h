// Kernels of the per-phase form's device-driven batches of steps: four
// launches a step (five with a conflict component above the bucket
// capacity), no host round trip inside a batch.
//
//   k_step_bp    skin decision of the step; base-pair evaluation per
//                candidate (+ union of formed pairs); bonded forces and noise
//                of every bead; the pair forces of a small system when the
//                limit MC is off (k_step_pair after it: of a large one)
//   k_step_seg   formed pairs bucketed by conflict component
//   k_step_mc    limit MC, one wavefront per component with excess; the pair
//                forces
//   k_step_move  base-pair forces gathered, GJF-2GJ (or Brownian) update,
//                displacement top-2, reset of the step's scratch
//
// The base-pair chain (evaluation, buckets, deletion chains) is bound by
// latency: a few hundred wavefronts of dependent FP64, atomics and lane
// reads on a chip with room for thousands.  The pair, bonded and noise work
// needs only the positions, so it runs beside that chain in the same
// launches, on blocks after those of the chain (the dispatcher starts those
// first), and what it gives is kept for the last launch: 64 B a bead more
// traffic.  Bonded terms are worked out once per term, a thread per term
// and tile, instead of once per bead they act on with one lane in eight
// active, and the noise once per bead with every lane active.  With the
// skin test, the resets and the large-component pass inside these launches
// a step takes four launches where it took seven.  Before and after, one
// MI355X, microseconds a step: 64 nt FP64 45 -> 28, 397 nt FP32 72 -> 54,
// 9,400 beads FP64 82 -> 61, 94,000 beads FP32 141 -> 100.
#pragma once
#include "sis_kernels.h"

namespace sis {

constexpr int STEP_B = 256;                 // threads of every block here
constexpr int BEAD_TILE = STEP_B - 3;       // beads of a bead tile (terms start up to three beads before it)
constexpr int PAIR_LPB = 8;                 // lanes per bead of a pair tile
constexpr int PAIR_TILE = STEP_B / PAIR_LPB;
constexpr int GRAPH_STEPS = 16;   // steps of a batch; even: the positions end in the buffer they started in

// Where the pair tiles run with the limit MC: beside the deletion chains of
// k_step_mc.  Microseconds a step with a share of them beside the evaluation
// and beside the buckets instead (0.4 and 0.15, then 1 and 0, then none):
// 94,000 beads FP32 119, 149, 106, FP64 130, 158, 116; 9,400 beads FP64 71.7,
// 70.9, 69.7; 397 nt FP32 61.1, 60.4, 60.2; 64 x 128 nt FP32 90.0, 91.5, 90.4.
// The evaluation needs 198 VGPRs and its blocks run two waves a SIMD, a pair
// tile among them too; k_step_mc needs 133 and waits for few long chains.
//
// Without the limit MC there is no k_step_mc.  Few tiles run beside the
// evaluation in k_step_bp, which spares a launch; from PAIR_OWN_LAUNCH on they
// have one to themselves (k_step_pair) and with it more waves a SIMD.
// Microseconds a step in k_step_bp / alone, FP64 and FP32: 256 tiles 30.5 /
// 34.8 and 27.4 / 32.0, 588 tiles 35.1 / 36.1 and 32.0 / 31.7, 940 tiles 44.2 /
// 39.7 and 41.0 / 34.5, 2,938 tiles (94,000 beads) 103 / 75 and 92 / 64.
constexpr int PAIR_OWN_LAUNCH = 640;

// Blocks of k_step_mc that take components (a wavefront each): a cap, as the
// listed ones are far fewer than the wavefronts there may be.  94,000 beads
// (about 3,400 listed a step) FP32 / FP64: 256 blocks 106.6 / 113.7, 512 104.3
// / 114.1, 1,024 105.4 / 115.9, 2,048 106.8 / 117.2, 4,096 107.0 / 117.2;
// smaller systems the same with any of them.
constexpr int STEP_MC_BLOCKS = 512;

// Device words that steer the batches (written back to the host as they are).
struct StepWords {
  int64_t step0;        // steps completed before the current batch
  int64_t stop;         // stop once this step is completed
  int64_t done;         // steps completed when they halted
  int64_t force_step;   // the step whose replicas with force_mc do the limit MC (after a rebuild)
  int64_t huge_step;    // the step that met a component above the bucket capacity (with huge_any)
  int halt;             // 1: this step and all after it do nothing
  int huge_any;         // such a component was met
};

// Arguments of one launch of step j (0-based) of a batch of nj.
struct StepArgs {
  StepWords *w;
  const int *force_mc;       // [R]
  int *huge;                 // [R] replicas with a component above the bucket capacity
  int *seg_n, *seg, *has_exc, *exc_list;
  double4 *fpair, *noise;    // [R*N] pair forces and normal draws of the step
  double *top2;              // [R*nblk*2] displacement maxima of k_step_move's blocks
  uint64_t seed;
  int nblk;                  // blocks of k_step_move per replica
  int ncand, nbead;          // leading blocks of k_step_bp: candidates, then bead tiles (multiples of 8)
  int nlist;                 // leading blocks of k_step_mc (a multiple of 8)
  int npair;                 // pair tiles per replica
  int ntile;                 // pair tiles of this launch: all R * npair or none
  int circ;                  // 1: some chain is circular (bonded terms per bead)
  int sep_huge;              // 1: k_step_huge runs in every step
  int j, nj;
};

// limit MC of replica r on `step`: every nstep_MC steps and after a rebuild
// (src/job_md.F90:364-394)
__device__ __forceinline__ bool step_mc(const Params &P, const StepArgs &A, int r, int64_t step) {
  if (P.nstep_bp_mc <= 0) return false;
  return step % P.nstep_bp_mc == 0 || (step == A.w->force_step && A.force_mc[r]);
}

// The skin test of the last step for replica r, of all R in turn
// (src/job_md.F90:376-395: sqrt(d2max) + sqrt(d2max_2nd) > nl_margin), from the
// maxima that k_step_move left.  The maxima meet in the order of k_skin's tree,
// which matters for a run that has blown up: a NaN maximum gives way to what it
// is compared with, and that order lets every other block count.  Returns
// whether one fires, to some threads of the block.  s: 2 x STEP_B doubles.
__device__ __forceinline__ bool skin_fires(const Params &P, const StepArgs &A, double *s) {
  const int t = threadIdx.x, L = t & 63, n = A.nblk;
  // blocks b, b + stride, ... of replica r
  auto take = [&](int r, int b, int stride, double &m1, double &m2) {
    m1 = m2 = 0.0;
    for (; b < n; b += stride) {
      const double *q = A.top2 + ((size_t)r * n + b) * 2;
      top2_merge(m1, m2, q[0], q[1]);
    }
  };
  bool fire = false;
  double m1, m2, x1, x2;
  if (n <= 4) {
    // a thread for each replica
    for (int r = t; r < P.R; r += STEP_B) {
      double m[4][2];
#pragma unroll
      for (int b = 0; b < 4; b++) {
        take(r, b, 4, m[b][0], m[b][1]);
        top2_merge(m[b][0], m[b][1], 0.0, 0.0);   // the empty rest of the tree
      }
      top2_merge(m[0][0], m[0][1], m[2][0], m[2][1]);
      top2_merge(m[1][0], m[1][1], m[3][0], m[3][1]);
      top2_merge(m[0][0], m[0][1], m[1][0], m[1][1]);
      if (sqrt(m[0][0]) + sqrt(m[0][1]) > P.nl_margin) fire = true;
    }
    return fire;
  }
  if (n <= 64) {
    // a wavefront for each replica
    for (int r = t >> 6; r < P.R; r += STEP_B / 64) {
      take(r, L, 64, m1, m2);
      top2_merge(m1, m2, 0.0, 0.0);
      for (int off = 32; off > 0; off >>= 1) {
        x1 = __shfl_xor(m1, off);
        x2 = __shfl_xor(m2, off);
        top2_merge(m1, m2, x1, x2);
      }
      if (L == 0 && sqrt(m1) + sqrt(m2) > P.nl_margin) fire = true;
    }
    return fire;
  }
  for (int r = 0; r < P.R; r++) {
    if (n <= 1024) {
      take(r, t, STEP_B, m1, m2);
    } else {   // k_skin<1024>
      take(r, t, 1024, m1, m2);
      take(r, t + 512, 1024, x1, x2);
      top2_merge(m1, m2, x1, x2);
      double y1, y2;
      take(r, t + 256, 1024, x1, x2);
      take(r, t + 768, 1024, y1, y2);
      top2_merge(x1, x2, y1, y2);
      top2_merge(m1, m2, x1, x2);
    }
    s[t] = m1;
    s[STEP_B + t] = m2;
    __syncthreads();
    if (t < 64) {
      top2_merge(m1, m2, s[t + 128], s[STEP_B + t + 128]);
      x1 = s[t + 64];
      x2 = s[STEP_B + t + 64];
      top2_merge(x1, x2, s[t + 192], s[STEP_B + t + 192]);
      top2_merge(m1, m2, x1, x2);
      for (int off = 32; off > 0; off >>= 1) {
        x1 = __shfl_xor(m1, off);
        x2 = __shfl_xor(m2, off);
        top2_merge(m1, m2, x1, x2);
      }
      if (t == 0 && sqrt(m1) + sqrt(m2) > P.nl_margin) fire = true;
    }
    __syncthreads();
  }
  return fire;
}

// Whether step j does nothing: an earlier step of the batch halted, the
// stop is reached, a component waits for k_step_huge, or the skin test of
// the last step asks for a rebuild.  Every block of k_step_bp works it out from
// the maxima k_step_move left (a few KB; a launch of its own took longer);
// block 0 notes it for the other launches and the host.  Called by every
// thread.
__device__ __forceinline__ bool step_halted(const Params &P, const StepArgs &A, double *s) {
  // (a block that starts late may see the word block 0 has just written:
  // its own answer would be the same)
  const bool before = A.w->halt != 0;
  const int64_t at = A.w->step0 + A.j;   // steps completed
  int64_t done = at;
  bool h = before;
  if (!h && !A.sep_huge && A.w->huge_any) {
    // that step waits for its update (step0 may be stale here: a batch whose
    // last step waits has not committed)
    h = true;
    done = A.w->huge_step - 1;
  }
  h = __syncthreads_or(h || at >= A.w->stop) != 0;   // one answer for the block
  if (!h) h = __syncthreads_or(skin_fires(P, A, s)) != 0;
  if (blockIdx.x == 0 && threadIdx.x == 0 && h && !before) {
    A.w->done = done;
    A.w->halt = 1;
  }
  return h;
}

// Bonded forces and noise of a tile of beads of replica r.  Thread t takes
// the bond, angle and dihedral that start at bead b = first - 3 + t; the
// forces on a term's beads go through LDS (one kind of term at a time,
// component-major: no bank conflicts) and each bead adds those of the terms
// it belongs to, so every term is worked out once and the sums keep a fixed
// order.
__device__ __forceinline__ void bead_tile(const Params &P, const Ptrs &D, const StepArgs &A, int r, int tile,
                                          int64_t step, double (*sf)[STEP_B]) {
  const int N = P.N, t = threadIdx.x, b = tile * BEAD_TILE - 3 + t;
  const double *box = D.box + 3 * r;
  const double4 *x = D.pos + (size_t)r * N;
  const bool own = t >= 3 && b < N;
  V3<double> F{0.0, 0.0, 0.0};
  if (A.circ) {
    if (own) F = bonded_part(P, D, r, b, 0, 1);
  } else {
    int left = 0;   // beads of the chain after b
    double4 x0{0, 0, 0, 0}, x1 = x0, x2 = x0, x3 = x0;
    if (b >= 0 && b < N) {
      const Topo tb = D.topo[b];
      left = tb.len - tb.loc;
      x0 = x[b];
      if (left > 0) x1 = x[b + 1];
      if (left > 1) x2 = x[b + 2];
      if (left > 2) x3 = x[b + 3];
    }
    const V3<double> z{0.0, 0.0, 0.0}, v01 = pvec(P, box, x0, x1), v21 = pvec(P, box, x2, x1),
                     v23 = pvec(P, box, x2, x3);
    auto put = [&](int k, const V3<double> &f) { sf[3 * k][t] = f.x; sf[3 * k + 1][t] = f.y; sf[3 * k + 2][t] = f.z; };
    auto get = [&](int k, int u) { return V3<double>{sf[3 * k][u], sf[3 * k + 1][u], sf[3 * k + 2][u]}; };
    // bond: force on the second bead, its negative on the first
    put(0, left > 0 ? bond_force_p(P, v01, 1) : z);
    {
      V3<double> f0 = z, f2 = z;
      if (left > 1) {
        f0 = angle_force_p(P, v01, v21, 0);
        f2 = angle_force_p(P, v01, v21, 2);
      }
      put(1, f0);
      put(2, f2);
    }
    __syncthreads();
    if (own)
      F = get(0, t - 1) - get(0, t) + get(1, t) - (get(1, t - 1) + get(2, t - 1)) + get(2, t - 2);
    if (P.dih_type) {
      V3<double> f0 = z, f1 = z, f2 = z;
      if (left > 2) {
        f0 = dih_force_p(P, v01, v21, v23, 0);
        f1 = dih_force_p(P, v01, v21, v23, 1);
        f2 = dih_force_p(P, v01, v21, v23, 2);
      }
      __syncthreads();
      put(0, f0);
      put(1, f1);
      put(2, f2);
      __syncthreads();
      // the fourth force is what the other three leave
      if (own)
        F = F + get(0, t) + get(1, t - 1) + get(2, t - 2) - (get(0, t - 3) + get(1, t - 3) + get(2, t - 3));
    }
  }
  if (!own) return;
  const size_t g = (size_t)r * N + b;
  D.fbond[g] = double4{F.x, F.y, F.z, 0.0};
  double n0, n1, n2;
  noise_normals(A.seed, r, step, b, n0, n1, n2);
  A.noise[g] = double4{n0, n1, n2, 0.0};
}

// WCA and Debye-Hueckel forces of pair tile `tile` (PAIR_TILE beads of one
// replica, PAIR_LPB lanes each)
template <typename T>
__device__ __forceinline__ void pair_tile(const Params &P, const Ptrs &D, const StepArgs &A, int tile) {
  const int r = tile / A.npair, a = (tile - r * A.npair) * PAIR_TILE + threadIdx.x / PAIR_LPB;
  const int l = threadIdx.x % PAIR_LPB;
  V3<double> F{0.0, 0.0, 0.0};
  if (a < P.N) F = pair_nb<T>(P, D, r, a, l, PAIR_LPB, nullptr, F);
  F = group_sum<PAIR_LPB>(F);
  if (a < P.N && l == 0) A.fpair[(size_t)r * P.N + a] = double4{F.x, F.y, F.z, 0.0};
}

// this launch's pair tile of block `id` after `first` leading blocks (a
// multiple of 8: the block's XCD keeps a contiguous slice of the tiles, see
// xcd_tile)
template <typename T>
__device__ __forceinline__ void pair_block(const Params &P, const Ptrs &D, const StepArgs &A, int first) {
  const int id = blockIdx.x - first;
  if (id < A.ntile) pair_tile<T>(P, D, A, xcd_tile(id, A.ntile));
}

template <typename T>
__global__ void __launch_bounds__(STEP_B) k_step_bp(Params P, Ptrs D, StepArgs A) {
  __shared__ double sf[9][STEP_B];
  if (step_halted(P, A, sf[0])) return;   // (two rows of it)
  const int64_t step = A.w->step0 + A.j + 1;
  const int blk = blockIdx.x;
  if (blk < A.ncand) {
    if (blk == 0 && threadIdx.x == 0) A.exc_list[0] = 0;
    const int gb = blk * STEP_B + threadIdx.x;
    if (gb >= bp_count(P, D, -1)) return;
    const int *mp = D.bp_mp + (size_t)gb * 8;
    const int r = mp[7];
    const int mc = step_mc(P, A, r, step) ? 1 : 0;
    if (bp_eval_one<T>(P, D, gb, mc) && mc) uf_join(D.comp + (size_t)r * P.N, mp[0] - 1, mp[1] - 1);
  } else if (blk < A.ncand + A.nbead) {
    const int k = blk - A.ncand, per = (P.N + BEAD_TILE - 1) / BEAD_TILE;
    if (k < per * P.R) {
      __syncthreads();   // sf is free
      bead_tile(P, D, A, k / per, k % per, step, sf);
    }
  } else {
    pair_block<T>(P, D, A, A.ncand + A.nbead);
  }
}

__global__ void __launch_bounds__(STEP_B) k_step_seg(Params P, Ptrs D, StepArgs A) {
  if (A.w->halt) return;
  const int gb = blockIdx.x * STEP_B + threadIdx.x;
  if (gb >= bp_count(P, D, -1) || !D.bp_status[gb]) return;
  const int r = D.bp_mp[(size_t)gb * 8 + 7];
  if (step_mc(P, A, r, A.w->step0 + A.j + 1)) seg_fill_one(P, D, gb, A.seg_n, A.seg, A.has_exc, A.exc_list);
}

// the pair tiles alone
template <typename T>
__global__ void __launch_bounds__(STEP_B) k_step_pair(Params P, Ptrs D, StepArgs A) {
  if (A.w->halt) return;
  pair_block<T>(P, D, A, 0);
}

template <typename T>
__global__ void __launch_bounds__(STEP_B) k_step_mc(Params P, Ptrs D, StepArgs A) {
  __shared__ __align__(16) int ws[STEP_B / 64][MCB_LDS];
  if (A.w->halt) return;
  if ((int)blockIdx.x >= A.nlist) {
    pair_block<T>(P, D, A, A.nlist);
    return;
  }
  const int64_t step = A.w->step0 + A.j + 1;
  const int n = A.exc_list[0], wave = threadIdx.x >> 6;
  // components dealt block by block: the listed ones of a small system
  // spread over the compute units
  for (int k = blockIdx.x + wave * A.nlist; k < n; k += A.nlist * (STEP_B / 64)) {
    const int gr = A.exc_list[1 + k];
    const int r = gr / P.N, root = gr - r * P.N;
    if (mc_one_component(P, D, r, root, A.seg_n, A.seg, nullptr, A.seed, step, A.huge, ws[wave])) {
      A.w->huge_step = step;   // every wavefront that meets one writes the same values
      A.w->huge_any = 1;
    }
  }
}

// components above the bucket capacity, one wavefront per replica that has
// them (k_step_mc marks it)
__global__ void __launch_bounds__(64) k_step_huge(Params P, Ptrs D, StepArgs A) {
  const int r = blockIdx.x;
  if (A.w->halt || !A.huge[r]) return;
  mc_huge_replica(P, D, r, A.seg_n, A.seg, A.has_exc, nullptr, A.seed, A.w->step0 + A.j + 1);
  if (threadIdx.x == 0) A.huge[r] = 0;
}

// bp_status_MC = bp_status for the replicas that did the MC this step
// (src/job_md.F90:399-401); launched when the MC does not run in every step
__global__ void __launch_bounds__(STEP_B) k_step_keep(Params P, Ptrs D, StepArgs A) {
  if (A.w->halt || (!A.sep_huge && A.w->huge_any)) return;
  const int gb = blockIdx.x * STEP_B + threadIdx.x;
  if (gb >= bp_count(P, D, -1)) return;
  if (step_mc(P, A, D.bp_mp[(size_t)gb * 8 + 7], A.w->step0 + A.j + 1)) D.bp_status_mc[gb] = D.bp_status[gb];
}

__global__ void __launch_bounds__(STEP_B) k_step_move(Params P, Ptrs D, StepArgs A) {
  __shared__ double s[STEP_B / 64][2];
  if (A.w->halt || (!A.sep_huge && A.w->huge_any)) return;
  const int N = P.N, a = blockIdx.x * STEP_B + threadIdx.x, r = blockIdx.y, t = threadIdx.x;
  double m1 = 0.0, m2 = 0.0;
  if (a < N) {
    const size_t g = (size_t)r * N + a;
    const double4 fp = A.fpair[g], fb = D.fbond[g], nz = A.noise[g];
    V3<double> F = pair_bp4(P, D, r, a, V3<double>{fp.x, fp.y, fp.z});
    F.x += fb.x; F.y += fb.y; F.z += fb.z;
    D.nt_cnt[g] = -P.max_bp_per_nt;
    if (P.nstep_bp_mc > 0) {
      D.comp[g] = a;
      A.seg_n[g] = 0;
      A.has_exc[g] = 0;
    }
    m1 = move_bead(P, D, g, a, F, nz.x, nz.y, nz.z);
    if (!(m1 > 0.0)) m1 = 0.0;   // a bead gone to NaN does not hide the others
  }
  for (int off = 32; off > 0; off >>= 1) top2_merge(m1, m2, __shfl_xor(m1, off), __shfl_xor(m2, off));
  if ((t & 63) == 0) { s[t >> 6][0] = m1; s[t >> 6][1] = m2; }
  __syncthreads();
  if (t != 0) return;
  for (int w = 1; w < STEP_B / 64; w++) top2_merge(m1, m2, s[w][0], s[w][1]);
  double *q = A.top2 + ((size_t)r * A.nblk + blockIdx.x) * 2;
  q[0] = m1;
  q[1] = m2;
  // the last step of the batch commits it (no block here reads step0)
  if (A.j == A.nj - 1 && blockIdx.x == 0 && r == 0) A.w->step0 += A.nj;
}

// Brownian dynamics: pair, bonded and base-pair forces and the update in one
// launch (force_lanes), in place of the tiles of the other launches and of
// k_step_move.  Its positions move by h/gamma times the force with no
// inertia in between, and where a bond is stiff for the step (h k / gamma
// near or above 2) such a run amplifies the last bit of every sum, so these
// runs keep the order of summation and the rounding that steps launched one
// by one have (add_nc, move_bead).
template <typename T>
__global__ void __launch_bounds__(STEP_B) k_step_force(Params P, Ptrs D, StepArgs A) {
  if (A.w->halt || (!A.sep_huge && A.w->huge_any)) return;
  int g = -1;
  force_lanes<T, PAIR_LPB, STEP_B>(P, D, 1, 0, A.seed, A.w->step0 + A.j + 1, nullptr, 1, A.top2, g);
  if (g >= 0 && P.nstep_bp_mc > 0) {
    D.comp[g] = g % P.N;
    A.seg_n[g] = 0;
    A.has_exc[g] = 0;
  }
}
// the end of such a batch (the blocks of k_step_force read step0)
__global__ void k_step_commit(StepArgs A) {
  if (A.w->halt || (!A.sep_huge && A.w->huge_any)) return;
  A.w->step0 += A.nj;
}

}  // namespace sis
