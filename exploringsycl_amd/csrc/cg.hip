// libteahip.so: the CG solve (TeaLeaf/c_kernels/sycl/cg.cpp) and the shared
// solver kernels (TeaLeaf/c_kernels/sycl/solver_methods.cpp).
//
// Every FP64 expression below is evaluated in the reference's operand order
// and the library is compiled with -ffp-contract=off, so each product and sum
// rounds on its own; together with the reference's reduction tree
// (span_reduce on the device, the last passes on the host) the results are
// bitwise those of the
// FP64 CPU restatement.

#include <hip/hip_runtime.h>

#include "tea_hip_impl.h"

namespace tea {
namespace {

// The 5-point operator of TeaLeaf/shared.h:59-63 at cell i, given the
// operand at the cell (c) and at its left/right/bottom/top neighbours.
__device__ inline double smvp(double c, double l, double r, double b, double t,
                              const double* __restrict__ kx,
                              const double* __restrict__ ky, int i, int x) {
  const double kx0 = kx[i], kx1 = kx[i + 1];
  const double ky0 = ky[i], ky1 = ky[i + x];
  const double diag = (1.0 + (kx1 + kx0)) + (ky1 + ky0);
  return (diag * c - (kx1 * r + kx0 * l)) - (ky1 * t + ky0 * b);
}

// ---- cg_init (cg.cpp:7-134) ----------------------------------------------

struct InitUBody {
  double* __restrict__ p;
  double* __restrict__ r;
  double* __restrict__ u;
  double* __restrict__ w;
  const double* __restrict__ density;
  const double* __restrict__ energy;
  int coefficient, x, y;
  __device__ void operator()(int i, int kk, int jj) const {
    p[i] = 0.0;
    r[i] = 0.0;
    u[i] = energy[i] * density[i];
    if (jj > 0 && jj < y - 1 && kk > 0 && kk < x - 1)
      w[i] = coefficient == TEA_CONDUCTIVITY ? density[i] : 1.0 / density[i];
  }
};

struct InitKBody {
  const double* __restrict__ w;
  double* __restrict__ kx;
  double* __restrict__ ky;
  double rx, ry;
  int x, y, h;
  __device__ void operator()(int i, int kk, int jj) const {
    if (jj >= h && jj < y - 1 && kk >= h && kk < x - 1) {
      kx[i] = rx * (w[i - 1] + w[i]) / (2.0 * w[i - 1] * w[i]);
      ky[i] = ry * (w[i - x] + w[i]) / (2.0 * w[i - x] * w[i]);
    }
  }
};

struct InitOthersBody {
  const double* __restrict__ kx;
  const double* __restrict__ ky;
  double* __restrict__ p;
  double* __restrict__ r;
  const double* __restrict__ u;
  double* __restrict__ w;
  int x;
  __device__ void operator()(int i, int, int, double (&out)[1]) const {
    const double s = smvp(u[i], u[i - 1], u[i + 1], u[i - x], u[i + x], kx, ky,
                          i, x);
    w[i] = s;
    const double rr = u[i] - s;
    r[i] = rr;
    p[i] = rr;
    out[0] = rr * rr;
  }
};

// ---- one launch per reference kernel -------------------------------------

struct CalcWBody {  // cg.cpp:137-195
  const double* __restrict__ p;
  const double* __restrict__ kx;
  const double* __restrict__ ky;
  double* __restrict__ w;
  int x;
  __device__ void operator()(int i, int, int, double (&out)[1]) const {
    const double pc = p[i];
    const double s = smvp(pc, p[i - 1], p[i + 1], p[i - x], p[i + x], kx, ky,
                          i, x);
    w[i] = s;
    out[0] = s * pc;
  }
};

struct CalcURBody {  // cg.cpp:198-254
  double* __restrict__ u;
  double* __restrict__ r;
  const double* __restrict__ p;
  const double* __restrict__ w;
  double alpha;
  __device__ void operator()(int i, int, int, double (&out)[1]) const {
    u[i] = u[i] + alpha * p[i];
    const double rn = r[i] - alpha * w[i];
    r[i] = rn;
    out[0] = rn * rn;
  }
};

struct CalcPBody {  // cg.cpp:257-281
  double* __restrict__ p;
  const double* __restrict__ r;
  double beta;
  Geo g;
  __device__ void operator()(int i, int kk, int jj) const {
    if (interior(g, kk, jj)) p[i] = beta * p[i] + r[i];
  }
};

// ---- fused iteration ------------------------------------------------------
//
// Kernel 1 (fused_w), in one pass over the grid:
//   u += alpha_prev * p_old                  (deferred from cg_calc_ur)
//   p_new = beta * p_old + r                 (deferred cg_calc_p)
//   p_new, u on the depth-1 halo ring         (deferred run_local_halos)
//   w = A p_new,  pw = sum p_new . w          (cg_calc_w)
// reads p_old, r, u, kx, ky and writes p_new, u, w: 8 words per cell.
// p_new at a neighbour is recomputed from p_old and r there; a neighbour on
// the halo ring is the reflection of the cell itself, so its p_new is pc.
// Kernel 2 (fused_r): r -= alpha w, rrn = r.r (3 words per cell).
// Together 11 words = 88 bytes per cell per iteration against the
// reference's 13 (calc_w 4 + calc_ur 6 + calc_p 3).

template <bool CONSUME>
__device__ inline double ra_scalar(const RaScalar& s, double value) {
  if (!CONSUME) return s.dev ? *s.dev : value;
  double sum[1];
  const double rro = s.rro_dev ? *s.rro_dev : s.rro;
  consume_sums<1>(s.sub, s.nblk, sum);
  const double q = s.inverse ? sum[0] / rro : rro / sum[0];
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (s.sum_dev) *s.sum_dev = s.inverse ? sum[0] : q;
    s.out[0] = sum[0];
    s.out[1] = q;
  }
  return q;
}

// Cells of one thread are visited in batches of BATCH: all loads of a batch
// are issued before any of its arithmetic and stores, so each wave keeps
// BATCH cells' worth of reads in flight (loads cannot move past the stores
// of the previous batch, as the compiler cannot prove the arrays distinct).
// BATCH trades reads in flight per wave against waves per SIMD.
template <bool APPLY_P, int kBatch>
__global__ __launch_bounds__(kBlock) void fused_w_kernel(Geo g, FusedWArgs a,
                                                         double* partials,
                                                         int nspan,
                                                         int single_group) {
  const int span = xcd_span(blockIdx.x, gridDim.x);
  const int base = span * kSpan;
  const int x = g.x;
  const int xl = g.h, xr = g.x - g.h - 1, yb = g.h, yt = g.y - g.h - 1;
  const double* __restrict__ P = a.p_old;
  const double* __restrict__ R = a.r;
  const double* __restrict__ KX = a.kx;
  const double* __restrict__ KY = a.ky;
  double prod[1][kItems];

#pragma unroll
  for (int b0 = 0; b0 < kItems; b0 += kBatch) {
    int ci[kBatch], ck[kBatch], cj[kBatch];
    bool in[kBatch];
    double po[kBatch], pl[kBatch], pr[kBatch], pb[kBatch], pt[kBatch];
    double rc[kBatch], rl[kBatch], rr[kBatch], rb[kBatch], rt[kBatch];
    double uc[kBatch], kx0[kBatch], kx1[kBatch], ky0[kBatch], ky1[kBatch];
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      const int e = base + (b0 + j) * kBlock + threadIdx.x;
      const int jj = e < g.n ? (int)g.dx.div((uint32_t)e) : 0;
      ci[j] = e;
      cj[j] = jj;
      ck[j] = e - jj * x;
      in[j] = e < g.n && interior(g, ck[j], jj);
    }
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      const int i = in[j] ? ci[j] : x + 1;  // any interior-safe index
      po[j] = P[i];
      pl[j] = P[i - 1];
      pr[j] = P[i + 1];
      pb[j] = P[i - x];
      pt[j] = P[i + x];
      if (APPLY_P) {
        rc[j] = R[i];
        rl[j] = R[i - 1];
        rr[j] = R[i + 1];
        rb[j] = R[i - x];
        rt[j] = R[i + x];
      }
      kx0[j] = KX[i];
      kx1[j] = KX[i + 1];
      ky0[j] = KY[i];
      ky1[j] = KY[i + x];
      uc[j] = a.apply_u ? a.u[i] : 0.0;
    }
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      const int i = ci[j], kk = ck[j], jj = cj[j];
      double pc, l, rgt, bot, top;
      if (APPLY_P) {
        // p_new = beta p_old + r, here and at the four neighbours; a
        // neighbour on the reflective halo ring is this cell's mirror image.
        pc = a.beta * po[j] + rc[j];
        l = kk == xl ? pc : a.beta * pl[j] + rl[j];
        rgt = kk == xr ? pc : a.beta * pr[j] + rr[j];
        bot = jj == yb ? pc : a.beta * pb[j] + rb[j];
        top = jj == yt ? pc : a.beta * pt[j] + rt[j];
      } else {
        pc = po[j];
        l = pl[j];
        rgt = pr[j];
        bot = pb[j];
        top = pt[j];
      }
      const double diag = (1.0 + (kx1[j] + kx0[j])) + (ky1[j] + ky0[j]);
      const double s = (diag * pc - (kx1[j] * rgt + kx0[j] * l)) -
                       (ky1[j] * top + ky0[j] * bot);
      prod[0][b0 + j] = in[j] ? s * pc : 0.0;
      if (!in[j]) continue;
      a.w[i] = s;
      const bool L = kk == xl, Rr = kk == xr, B = jj == yb, T = jj == yt;
      const bool edge = L | Rr | B | T;
      if (a.apply_u) {
        const double un = uc[j] + a.alpha * po[j];
        a.u[i] = un;
        if (a.ring && edge) {
          if (L) a.u[i - 1] = un;
          if (Rr) a.u[i + 1] = un;
          if (B) a.u[i - x] = un;
          if (T) a.u[i + x] = un;
          if (L && B) a.u[i - 1 - x] = un;
          if (Rr && B) a.u[i + 1 - x] = un;
          if (L && T) a.u[i - 1 + x] = un;
          if (Rr && T) a.u[i + 1 + x] = un;
        }
      }
      if (APPLY_P) {
        double* __restrict__ Q = a.p_new;
        Q[i] = pc;
        if (edge) {
          // With the halo refresh folded in, the ring gets the new values;
          // without it, p keeps its old halo.
          if (L) Q[i - 1] = a.ring ? pc : pl[j];
          if (Rr) Q[i + 1] = a.ring ? pc : pr[j];
          if (B) Q[i - x] = a.ring ? pc : pb[j];
          if (T) Q[i + x] = a.ring ? pc : pt[j];
          if (L && B) Q[i - 1 - x] = a.ring ? pc : P[i - 1 - x];
          if (Rr && B) Q[i + 1 - x] = a.ring ? pc : P[i + 1 - x];
          if (L && T) Q[i - 1 + x] = a.ring ? pc : P[i - 1 + x];
          if (Rr && T) Q[i + 1 + x] = a.ring ? pc : P[i + 1 + x];
        }
      }
    }
  }
  span_reduce<1>(prod, partials, nspan, span, single_group != 0);
}

// ---- two cells per lane --------------------------------------------------
//
// Every cell pair (2m, 2m+1) starts on a 16-byte boundary, so p, r, u, kx and
// ky are read with one 16-byte load per pair (the rows above and below too,
// at 8-byte alignment when x is odd), and the left/right neighbours come from
// the adjacent lanes (lane l-1 holds 2m-1, lane l+1 holds 2m+2); only lanes
// 0 and 63 load theirs.  A wave covers 128 consecutive cells = two groups
// of the reduction tree (lanes 0-31 and 32-63); a 256-thread block covers a
// 4096-cell span in 8 slots of 512 cells.  The first tree level is the
// in-lane pair sum, then the butterfly runs over each 32-lane half.

__device__ inline void span_reduce_pairs(double (&v)[kSlots], double* partials,
                                         int nspan, int span,
                                         bool single_group) {
  double (&vv)[1][kSlots] = *reinterpret_cast<double (*)[1][kSlots]>(&v);
  span_reduce_pairs_n<1>(vv, partials, nspan, span, single_group);
}

// One cell pair of the fused iteration: its indices, its loads and its
// arithmetic, shared by the span-per-block and pair-per-thread kernels so
// both evaluate every cell identically.
struct FusedPair {
  int e0, kk, jj;
  bool in0, in1, any;
  double2 P0, Pt, Pb, R0, Rt, Rb, KX, KY, KYt, U, H, H2;
  // Wave-edge neighbours: lane 0 holds p and r at e0 - 1, lane 63 p, r and
  // kx at e0 + 2 (the other lanes take theirs from adjacent lanes).
  double PN, RN, KXN;
};

__device__ inline void fused_pair_index(const Geo& g, int e, FusedPair& s) {
  const int row = e < g.n ? (int)g.dx.div((uint32_t)e) : 0;
  s.e0 = e;
  s.jj = row;
  s.kk = e - row * g.x;
  s.in0 = e < g.n && interior(g, s.kk, row);
  s.in1 = e < g.n && interior(g, s.kk + 1, row);
  s.any = s.in0 || s.in1;
}

// The pair's own p, r and kx are also the left/right neighbours the adjacent
// lanes take by shuffle, so they are read whenever the pair is in range; the
// rows above and below only for interior pairs.
template <bool APPLY_P, int UM>
__device__ inline void fused_pair_load(const Geo& g, const FusedWArgs& a,
                                       FusedPair& s) {
  const int x = g.x;
  const double* __restrict__ P = a.p_old;
  const double* __restrict__ R = a.r;
  const int ic = s.e0 < g.n ? s.e0 : safe_pair(x);
  const int ir = s.any ? s.e0 : safe_pair(x);
  s.P0 = ld2(P, ic);
  s.Pt = ld2u(P, ir + x);
  s.Pb = ld2u(P, ir - x);
  if (APPLY_P) {
    s.R0 = ld2(R, ic);
    s.Rt = ld2u(R, ir + x);
    s.Rb = ld2u(R, ir - x);
  }
  s.KX = ld2(a.kx, ic);
  s.KY = ld2(a.ky, ir);
  s.KYt = ld2u(a.ky, ir + x);
  if (UM == 3 || (UM == 1 && a.apply_u)) s.U = ld2_nt(a.u, ir, g.nt);
  if (UM == 3) {
    s.H = ld2_nt(a.p_h, ir, g.nt);
    s.H2 = ld2_nt(a.p_h2, ir, g.nt);
  }
  // Issued with the pair's own loads so the wave waits once; ir - 1 and
  // ir + 2 are in range (ir is an interior pair's index or the safe one).
  // Lanes 0 and 63 share each load instruction, at their own addresses
  // (lane 0's kx value is not used).
  const int lane = threadIdx.x & (kWave - 1);
  if (lane == 0 || lane == kWave - 1) {
    const int ni = lane == 0 ? ir - 1 : ir + 2;
    s.PN = P[ni];
    if (APPLY_P) s.RN = R[ni];
    s.KXN = a.kx[ni];
  }
}

// Computes and stores the pair (w, u, p_new and their halo ring) and returns
// the in-lane pair sum of p_new . w (the first level of the reduction tree).
template <bool APPLY_P, int UM>
__device__ inline double fused_pair_compute(const Geo& g, const FusedWArgs& a,
                                            const FusedPair& s, int lane, double beta) {
  const int x = g.x;
  const int xl = g.h, xr = g.x - g.h - 1, yb = g.h, yt = g.y - g.h - 1;
  const double* __restrict__ P = a.p_old;
  const int i = s.e0;
  // Neighbours across the pair boundary, from the adjacent lanes.
  double pl = from_prev_lane(s.P0.y), pr = from_next_lane(s.P0.x);
  double rl = 0.0, rr = 0.0;
  if (APPLY_P) {
    rl = from_prev_lane(s.R0.y);
    rr = from_next_lane(s.R0.x);
  }
  double kxr = from_next_lane(s.KX.x);
  if (lane == 0) {
    pl = s.PN;
    if (APPLY_P) rl = s.RN;
  }
  if (lane == kWave - 1) {
    pr = s.PN;
    if (APPLY_P) rr = s.RN;
    kxr = s.KXN;
  }
  const int ka = s.kk, kb = s.kk + 1, row = s.jj;
  double ca, cb, la, ra, lb, rb2, ba, ta, bb, tb;
  if (APPLY_P) {
    ca = beta * s.P0.x + s.R0.x;
    cb = beta * s.P0.y + s.R0.y;
    la = ka == xl ? ca : beta * pl + rl;
    ra = ka == xr ? ca : cb;
    lb = kb == xl ? cb : ca;
    rb2 = kb == xr ? cb : beta * pr + rr;
    ba = row == yb ? ca : beta * s.Pb.x + s.Rb.x;
    ta = row == yt ? ca : beta * s.Pt.x + s.Rt.x;
    bb = row == yb ? cb : beta * s.Pb.y + s.Rb.y;
    tb = row == yt ? cb : beta * s.Pt.y + s.Rt.y;
  } else {
    ca = s.P0.x;
    cb = s.P0.y;
    la = pl;
    ra = cb;
    lb = ca;
    rb2 = pr;
    ba = s.Pb.x;
    ta = s.Pt.x;
    bb = s.Pb.y;
    tb = s.Pt.y;
  }
  const double kxa0 = s.KX.x, kxa1 = s.KX.y, kxb0 = s.KX.y, kxb1 = kxr;
  const double diag_a = (1.0 + (kxa1 + kxa0)) + (s.KYt.x + s.KY.x);
  const double diag_b = (1.0 + (kxb1 + kxb0)) + (s.KYt.y + s.KY.y);
  const double sa = (diag_a * ca - (kxa1 * ra + kxa0 * la)) -
                    (s.KYt.x * ta + s.KY.x * ba);
  const double sb = (diag_b * cb - (kxb1 * rb2 + kxb0 * lb)) -
                    (s.KYt.y * tb + s.KY.y * bb);
  const double psum = (s.in0 ? sa * ca : 0.0) + (s.in1 ? sb * cb : 0.0);
  if (!s.any) return psum;
  st2(a.w, i, s.in0, s.in1, sa, sb);
  double ua = 0.0, ub = 0.0;
  const bool apply_u = UM == 3 || (UM == 1 && a.apply_u);
  if (apply_u) {
    const double alpha = a.alpha_dev ? *a.alpha_dev : a.alpha;
    ua = s.U.x;
    ub = s.U.y;
    if (UM == 3) {
      ua = (ua + a.alpha_h * s.H.x) + a.alpha_h2 * s.H2.x;
      ub = (ub + a.alpha_h * s.H.y) + a.alpha_h2 * s.H2.y;
    }
    ua = ua + alpha * s.P0.x;
    ub = ub + alpha * s.P0.y;
    st2_nt(a.u_out, i, s.in0, s.in1, ua, ub, g.nt);
  }
  if (APPLY_P) st2_nt(a.p_new, i, s.in0, s.in1, ca, cb, g.nt);
  // Halo ring of boundary-adjacent cells (rare; per cell).  With the halo
  // refresh folded in it takes the new values; without, p (and u, where it
  // goes to another buffer) keeps its old ring.
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int ic = i + c, kc = ka + c;
    if (!(c == 0 ? s.in0 : s.in1) || !(kc == xl || kc == xr || row == yb || row == yt)) continue;
    if (a.ring) {
      if (apply_u) ring_store(a.u_out, ic, kc, row, x, xl, xr, yb, yt, c == 0 ? ua : ub);
      if (APPLY_P) ring_store(a.p_new, ic, kc, row, x, xl, xr, yb, yt, c == 0 ? ca : cb);
      continue;
    }
    for (int dj = row == yb ? -1 : 0; dj <= (row == yt ? 1 : 0); ++dj)
      for (int dk = kc == xl ? -1 : 0; dk <= (kc == xr ? 1 : 0); ++dk) {
        if (dj == 0 && dk == 0) continue;
        const int q = ic + dj * x + dk;
        if (apply_u && a.u_out != a.u) a.u_out[q] = a.u[q];
        if (APPLY_P) a.p_new[q] = P[q];
      }
  }
  return psum;
}

// One span per block, 8 pairs per thread in batches of SB.
template <bool APPLY_P, int SB>
__global__ __launch_bounds__(kBlock) void fused_w2_kernel(Geo g, FusedWArgs a,
                                                          double* partials,
                                                          int nspan,
                                                          int single_group) {
  const int span = xcd_span(blockIdx.x, gridDim.x);
  const int base = span * kSpan;
  const int lane = threadIdx.x & (kWave - 1);
  double psum[kSlots];
#pragma unroll
  for (int s0 = 0; s0 < kSlots; s0 += SB) {
    FusedPair s[SB];
#pragma unroll
    for (int j = 0; j < SB; ++j)
      fused_pair_index(g, base + (s0 + j) * (2 * kBlock) + 2 * threadIdx.x, s[j]);
#pragma unroll
    for (int j = 0; j < SB; ++j) fused_pair_load<APPLY_P, 1>(g, a, s[j]);
#pragma unroll
    for (int j = 0; j < SB; ++j)
      psum[s0 + j] = fused_pair_compute<APPLY_P, 1>(g, a, s[j], lane, a.beta);
  }
  span_reduce_pairs(psum, partials, nspan, span, single_group != 0);
}

// One pair per thread: a 256-thread block covers 512 cells (8 groups of the
// reduction tree) and stores their 8-leaf subtree sum.  Small blocks
// keep 4x more waves per SIMD in flight than the span-per-block kernel.
// With CONSUME beta is formed from the sums of the r-step before it.
// UM: 0 leaves u alone, 1 adds alpha p_old where a.apply_u, 3 the two held
// updates and its own, each rounded as when made one by one.  u's read and
// write are 16 of the pass's 64 bytes per cell; with two passes of three
// leaving it to the third they move 48, 48 and 80 (the third also reads the
// two held p).
template <bool APPLY_P, int KS, int UM, bool CONSUME>
__global__ __launch_bounds__(kBlock * KS) void fused_w1_kernel(Geo g, FusedWArgs a, RaScalar sc,
                                                               double* sub, int nblk, int S) {
  int tid;
  const int blk = stacked_block<KS, kBlock>(S, &tid, g.bands);
  const int lane = threadIdx.x & (kWave - 1);
  FusedPair s;
  fused_pair_index(g, blk < nblk ? blk * kPairBlock + 2 * tid : g.n, s);
  fused_pair_load<APPLY_P, UM>(g, a, s);
  const double beta = ra_scalar<CONSUME>(sc, a.beta);
  const double v[1] = {fused_pair_compute<APPLY_P, UM>(g, a, s, lane, beta)};
  block_sums_pairs<1, KS>(v, sub, nblk, blk, tid);
}

// Launches fused_w1_kernel with stack_factor(c) blocks one row apart per
// workgroup (stacked_block, tea_hip_impl.h): their rows above and below come
// mostly from the CU's L1.  FP64 iteration with one, two and four blocks per
// workgroup: 4096^2 252.2, 250.3, 261.6 us; 1000^2 20.4, 20.1, 23.0.
template <bool APPLY_P, int UM, bool CONSUME>
void launch_fused_w1(tea_hip_chunk* c, const FusedWArgs& a, const RaScalar& sc) {
  const int S = stack_rows(c), ks = stack_factor(c);
  const auto kernel = ks == 1   ? fused_w1_kernel<APPLY_P, 1, UM, CONSUME>
                      : ks == 2 ? fused_w1_kernel<APPLY_P, 2, UM, CONSUME>
                                : fused_w1_kernel<APPLY_P, 4, UM, CONSUME>;
  hipLaunchKernelGGL(kernel, stacked_grid(c, ks), dim3(ks * kBlock), 0, c->stream, c->geo, a, sc,
                     c->sub, c->nblk, S);
}

int launch_cg_step(tea_hip_chunk* c, const CgStep& s, const RaScalar& sc) {
  Timed t(c, K_CG_FUSED_W);
  const bool consume = sc.sub != nullptr;
  if (!s.apply_p)
    launch_fused_w1<false, 1, false>(c, s.a, sc);
  else if (s.um == 0)
    consume ? launch_fused_w1<true, 0, true>(c, s.a, sc)
            : launch_fused_w1<true, 0, false>(c, s.a, sc);
  else if (s.um == 1)
    consume ? launch_fused_w1<true, 1, true>(c, s.a, sc)
            : launch_fused_w1<true, 1, false>(c, s.a, sc);
  else
    consume ? launch_fused_w1<true, 3, true>(c, s.a, sc)
            : launch_fused_w1<true, 3, false>(c, s.a, sc);
  TEA_HIP_TRY(hipGetLastError());
  return TEA_HIP_OK;
}

__global__ __launch_bounds__(kBlock) void fused_r2_kernel(
    Geo g, double* __restrict__ r, const double* __restrict__ w, double alpha,
    double* partials, int nspan, int single_group) {
  const int span = xcd_span(blockIdx.x, gridDim.x);
  const int base = span * kSpan;
  double2 rv[kSlots], wv[kSlots];
  bool in0[kSlots], in1[kSlots];
#pragma unroll
  for (int k = 0; k < kSlots; ++k) {
    const int e = base + k * (2 * kBlock) + 2 * threadIdx.x;
    const int row = e < g.n ? (int)g.dx.div((uint32_t)e) : 0;
    const int kk = e - row * g.x;
    in0[k] = e < g.n && interior(g, kk, row);
    in1[k] = e < g.n && interior(g, kk + 1, row);
    const int i = (in0[k] || in1[k]) ? e : 0;
    rv[k] = ld2_nt(r, i);
    wv[k] = ld2_nt(w, i);
  }
  double psum[kSlots];
#pragma unroll
  for (int k = 0; k < kSlots; ++k) {
    const double ra = rv[k].x - alpha * wv[k].x;
    const double rb = rv[k].y - alpha * wv[k].y;
    psum[k] = (in0[k] ? ra * ra : 0.0) + (in1[k] ? rb * rb : 0.0);
    st2_nt(r, base + k * (2 * kBlock) + 2 * threadIdx.x, in0[k], in1[k], ra, rb);
  }
  span_reduce_pairs(psum, partials, nspan, span, single_group != 0);
}

// fused_r2's arithmetic with one pair per thread; the block stores its
// 8-leaf subtree of r.r (see fused_w1_kernel).  The new r goes to r_out (r
// itself, or a spare buffer when the iteration runs ahead).
template <bool CONSUME>
__global__ __launch_bounds__(kBlock) void fused_r1_kernel(
    Geo g, const double* r, double* r_out, const double* __restrict__ w, double value,
    RaScalar sc, double* sub, int nblk) {
  const int blk = band_index(g.bands);
  const int e = blk * kPairBlock + 2 * threadIdx.x;
  const int row = e < g.n ? (int)g.dx.div((uint32_t)e) : 0;
  const int kk = e - row * g.x;
  const bool in0 = e < g.n && interior(g, kk, row);
  const bool in1 = e < g.n && interior(g, kk + 1, row);
  const int i = (in0 || in1) ? e : 0;
  const double2 rv = ld2_nt(r, i, g.nt), wv = ld2_nt(w, i, g.nt);
  const double alpha = ra_scalar<CONSUME>(sc, value);
  const double ra = rv.x - alpha * wv.x;
  const double rb = rv.y - alpha * wv.y;
  const double v[1] = {(in0 ? ra * ra : 0.0) + (in1 ? rb * rb : 0.0)};
  st2_nt(r_out, e, in0, in1, ra, rb, g.nt);
  block_sums_pairs<1>(v, sub, nblk, blk, threadIdx.x);
}

// r -= alpha w and r.r: all 16 cells' loads first, then the updates.
__global__ __launch_bounds__(kBlock) void fused_r_kernel(
    Geo g, double* __restrict__ r, const double* __restrict__ w, double alpha,
    double* partials, int nspan, int single_group) {
  const int span = xcd_span(blockIdx.x, gridDim.x);
  const int base = span * kSpan;
  double rv[kItems], wv[kItems];
  bool in[kItems];
#pragma unroll
  for (int k = 0; k < kItems; ++k) {
    const int e = base + k * kBlock + threadIdx.x;
    const int jj = e < g.n ? (int)g.dx.div((uint32_t)e) : 0;
    in[k] = e < g.n && interior(g, e - jj * g.x, jj);
    const int i = in[k] ? e : 0;
    rv[k] = r[i];
    wv[k] = w[i];
  }
  double prod[1][kItems];
#pragma unroll
  for (int k = 0; k < kItems; ++k) {
    const double rn = rv[k] - alpha * wv[k];
    prod[0][k] = in[k] ? rn * rn : 0.0;
    if (in[k]) r[base + k * kBlock + threadIdx.x] = rn;
  }
  span_reduce<1>(prod, partials, nspan, span, single_group != 0);
}

struct ApplyPendingBody {
  double* __restrict__ u;
  double* __restrict__ p;
  const double* __restrict__ r;
  double alpha, beta;
  int apply_u, apply_p;
  Geo g;
  __device__ void operator()(int i, int kk, int jj) const {
    if (!interior(g, kk, jj)) return;
    const double po = p[i];
    if (apply_u) u[i] = u[i] + alpha * po;
    if (apply_p) p[i] = beta * po + r[i];
  }
};

// ---- shared solver kernels (solver_methods.cpp) ---------------------------

struct CopyUBody {
  const double* __restrict__ u;
  double* __restrict__ u0;
  Geo g;
  __device__ void operator()(int i, int kk, int jj) const {
    if (interior(g, kk, jj)) u0[i] = u[i];
  }
};

struct ResidualBody {
  const double* __restrict__ u;
  const double* __restrict__ u0;
  double* __restrict__ r;
  const double* __restrict__ kx;
  const double* __restrict__ ky;
  Geo g;
  __device__ void operator()(int i, int kk, int jj) const {
    if (!interior(g, kk, jj)) return;
    const int x = g.x;
    r[i] = u0[i] - smvp(u[i], u[i - 1], u[i + 1], u[i - x], u[i + x], kx, ky,
                        i, x);
  }
};

struct NormBody {
  const double* __restrict__ b;
  __device__ void operator()(int i, int, int, double (&out)[1]) const {
    const double v = b[i];
    out[0] = v * v;
  }
};

// The 2-norm over cell pairs, one pair per lane (more than one group): 8 bytes
// per cell, the sum tree's first level in-lane.
__global__ __launch_bounds__(kBlock) void norm_pair_kernel(
    Geo g, const double* __restrict__ b, double* sub, int nblk) {
  const int blk = band_index(g.bands);
  const PairAt q = pair_at(g, blk * kPairBlock + 2 * threadIdx.x);
  const double2 v = ld2_nt(b, q.ic, g.nt);
  const double s[1] = {(q.in0 ? v.x * v.x : 0.0) + (q.in1 ? v.y * v.y : 0.0)};
  block_sums_pairs<1>(s, sub, nblk, blk, threadIdx.x);
}

struct FinaliseBody {
  const double* __restrict__ u;
  const double* __restrict__ density;
  double* __restrict__ energy;
  Geo g;
  __device__ void operator()(int i, int kk, int jj) const {
    if (interior(g, kk, jj)) energy[i] = u[i] / density[i];
  }
};

template <class Body>
int launch_each(tea_hip_chunk* c, int kid, const Body& body) {
  {
    Timed t(c, kid);
    hipLaunchKernelGGL((each_kernel<Body>), flat_grid(c->geo.n), dim3(kBlock),
                       0, c->stream, c->geo, body);
  }
  TEA_HIP_TRY(hipGetLastError());
  return TEA_HIP_OK;
}

template <class Body>
int launch_span1(tea_hip_chunk* c, int kid, const Body& body, double* out) {
  return sum_over_cells<1>(c, kid, body, out);
}

// The cells outside the interior of up to kFrames buffers from others
// (blockIdx.y the pair): the h rows below and above it, then its rows' h cells
// left and right of it.
constexpr int kFrames = 6;
struct FramePairs {
  const double* src[kFrames];
  double* dst[kFrames];
};
__global__ __launch_bounds__(kBlock) void copy_frame_kernel(Geo g, FramePairs f) {
  const int rows = 2 * g.h * g.x, sides = 2 * g.h * (g.y - 2 * g.h);
  int k = blockIdx.x * kBlock + threadIdx.x;
  if (k >= rows + sides) return;
  int i;
  if (k < rows) {
    i = k < rows / 2 ? k : k + (g.y - 2 * g.h) * g.x;
  } else {
    k -= rows;
    const int row = k / (2 * g.h), q = k - row * (2 * g.h);
    i = (g.h + row) * g.x + (q < g.h ? q : g.x - 2 * g.h + q);
  }
  f.dst[blockIdx.y][i] = f.src[blockIdx.y][i];
}

int copy_frames(tea_hip_chunk* c, const FramePairs& f, int n) {
  if (n == 0) return TEA_HIP_OK;
  const Geo& g = c->geo;
  const long cells = 2L * g.h * g.x + 2L * g.h * (g.y - 2 * g.h);
  hipLaunchKernelGGL(copy_frame_kernel, dim3((unsigned)((cells + kBlock - 1) / kBlock), n),
                     dim3(kBlock), 0, c->stream, g, f);
  TEA_HIP_TRY(hipGetLastError());
  return TEA_HIP_OK;
}

// Makes the spare p buffers' cells outside the interior equal to p's (the
// fused kernel writes only the interior and the ring).
int sync_p_alt(tea_hip_chunk* c) {
  if (c->p_alt_synced) return TEA_HIP_OK;
  FramePairs f{};
  int n = 0;
  for (double* b : c->p_alt)
    if (b) {
      f.src[n] = c->field[TEA_FIELD_P];
      f.dst[n++] = b;
    }
  TEA_RETURN_IF(copy_frames(c, f, n));
  c->p_alt_synced = true;
  return TEA_HIP_OK;
}

// The spare p buffers that held updates need (none: updates are not held).
void ensure_p_ring(tea_hip_chunk* c) {
  if (!c->hold_ok || c->p_ring_off || c->p_alt[2]) return;
  const size_t bytes = pair_bytes(c->geo.n, sizeof(double));
  if (!dev_alloc(c, &c->p_alt[1], bytes) || !dev_alloc(c, &c->p_alt[2], bytes)) {
    dev_free(c, c->p_alt[1]);
    c->p_ring_off = true;
    return;
  }
  c->p_alt_synced = false;
}

// ---- run-ahead of the fused CG iteration ----------------------------------
//
// The drop-in API returns p.w and r.r to the host, which forms alpha =
// rro / pw and beta = rrn / rro before the next pass can start
// (TeaLeaf/drivers/cg_driver.c:87-113): two host round trips per iteration,
// each costing the wait for the finisher's values, the host's arithmetic and
// a launch (about 13.5 us of a 272 us iteration at 4096^2).  The device
// forms the same scalars itself, and the next passes of the iteration are
// already queued, writing only spare buffers.  On grids of at most
// kConsumeBlocks blocks the next pass sums and divides (RaScalar), and its
// first block hands the host the values; beyond, a finisher does both
// (finish_out, core.hip):
//   the r-step: r - alpha w into r_alt, and r.r;
//   the w-step: u + alpha p into u_alt (or held), p = beta p + r into a spare
//     p with the U/P halo ring, w = A p into w_alt, p.w.
// cg_calc_w leaves the r-step and the w-step behind its own pass queued,
// cg_calc_ur the r-step after that: two passes ahead, as a pass of a small
// grid (4-6 us) is over before the host has seen its scalar.
// The host's next call takes a pass over (exchanging the buffers) when its
// scalar is bitwise the one the device used (read back with the sums) and,
// for the w-step, the deferred work is exactly the u and p updates and the
// U/P ring the pass applied; anything else drops the run-ahead, which wrote
// nothing but spare buffers, device scalars and its own host slots.  The
// results are those of the iteration without it, bit for bit.  Each step's
// sum and scalar go to one of two host slot sets, alternating, so the next
// step is queued before the host has read the last one.

constexpr int kRaW = 0, kRaRStep = 1;  // slot kinds

// x even: the passes take odd x too, and mixed precision runs ahead there, but
// FP64 CG's run-ahead has been measured and tested at even x only.
bool ra_possible(const tea_hip_chunk* c) {
  return c->ra_enabled && !c->ra_off && c->fused && c->poll && c->pairs && c->geo.x % 2 == 0 &&
         c->ra_rro_known && c->ra_fail < 3 && use_pair_blocks(c, 1) && use_pair_blocks(c, 2);
}

// Offset of a slot in ra_host.
int ra_slot(int kind, int i) { return 2 * (2 * kind + i); }

// Whether the run-ahead's buffers are there (else there is no run-ahead).
bool ensure_ra(tea_hip_chunk* c) {
  if (c->ra_host) return true;
  const size_t bytes = pair_bytes(c->geo.n, sizeof(double));
  bool ok = true;
  for (double** b : {&c->r_alt, &c->w_alt, &c->u_alt}) ok = ok && (*b || dev_alloc(c, b, bytes));
  ok = ok && (c->ra_dev || dev_alloc(c, &c->ra_dev, 3 * sizeof(double)));
  if (ok) c->ra_host = host_slots(8, &c->ra_host_dev);
  if (c->ra_host) return true;
  dev_free(c, c->r_alt);
  dev_free(c, c->w_alt);
  if (!c->mra_host) dev_free(c, c->u_alt);
  c->ra_off = true;
  return false;
}

// The next pass forms the scalar of the pass before it (RaScalar::sub).
bool ra_consume(const tea_hip_chunk* c) { return c->nblk <= kConsumeBlocks; }

// Arms a step's host slot for the pass or finisher about to be launched.
int ra_arm(tea_hip_chunk* c, int kind, int i) {
  if (c->ra_dirty) {
    // A dropped run-ahead may still be queued and write these slots.
    TEA_HIP_TRY(hipStreamSynchronize(c->stream));
    c->ra_dirty = false;
  }
  arm_host_values(c->ra_host + ra_slot(kind, i), 2);
  return TEA_HIP_OK;
}

// Where the pass after a w-step (kind kRaW) or r-step takes its scalar from;
// rro is the value, or what the w-step before left on the device.
RaScalar ra_scalar_of(const tea_hip_chunk* c, int kind, int i, double rro, bool from_dev) {
  RaScalar sc;
  sc.out = c->ra_host_dev + ra_slot(kind, i);
  if (!ra_consume(c)) {
    sc.dev = c->ra_dev + kind;
    return sc;
  }
  sc.sub = kind == kRaW ? c->sub : c->sub2;
  sc.nblk = c->nblk;
  sc.inverse = kind == kRaW ? 0 : 1;
  sc.rro = rro;
  sc.rro_dev = from_dev ? c->ra_dev + 2 : nullptr;
  sc.sum_dev = c->ra_dev + (kind == kRaW ? 0 : 2);
  return sc;
}

// The finisher of a w-step or r-step just queued (grids above kConsumeBlocks
// blocks).  Either way the step counts as one cg_ra_finish launch in the
// statistics.
int ra_finish(tea_hip_chunk* c, int kind, int i, double rro, bool from_dev) {
  if (ra_consume(c)) {
    if (c->timing && c->time_kernel[K_CG_RA_FINISH]) c->launches[K_CG_RA_FINISH] += 1;
    return TEA_HIP_OK;
  }
  TEA_RETURN_IF(ra_arm(c, kind, i));
  return launch_span_finish_ra(c, 1, c->ra_host_dev + ra_slot(kind, i),
                               RaTail{rro, from_dev ? 1 : 0, kind, c->ra_dev});
}

// Waits for a slot's sum and scalar.
int ra_wait(tea_hip_chunk* c, int kind, int i, double* sum, double* scalar) {
  const double* h = c->ra_host + ra_slot(kind, i);
  TEA_RETURN_IF(wait_host_values(c, h, 2));
  *sum = h[0];
  *scalar = h[1];
  return TEA_HIP_OK;
}

void ra_mismatch(tea_hip_chunk* c) {
  c->ra_r = c->ra_w = false;
  c->ra_dirty = true;
  c->ra_fail += 1;
}

template <class T>
void swap_ptr(T*& a, T*& b) {
  T* t = a;
  a = b;
  b = t;
}

// The w-step for the deferred work (ahead: behind the r-step in flight, for
// the whole of an iteration's deferred work, its alpha and beta on the
// device).  With all of it deferred, u's update is held over two steps.
int plan_cg_w(tea_hip_chunk* c, bool ahead, CgStep* s) {
  double** f = c->field;
  const bool ride = c->hold_ok && c->p_alt[2] &&
                    (ahead || (c->pend_u && c->pend_p && c->pend_halo));
  if (c->uh && !ride) TEA_RETURN_IF(apply_held_u(c));
  *s = CgStep{};
  s->apply_p = ahead || c->pend_p;
  if (s->apply_p) TEA_RETURN_IF(sync_p_alt(c));
  double* p_new = c->p_alt[0];
  for (double* b : c->p_alt) {
    if (!b || (c->uh > 0 && b == c->uh_p[0]) || (c->uh > 1 && b == c->uh_p[1])) continue;
    p_new = b;
    break;
  }
  s->a = FusedWArgs{f[TEA_FIELD_P], p_new, ahead ? c->r_alt : f[TEA_FIELD_R], f[TEA_FIELD_U],
                    ahead ? c->w_alt : f[TEA_FIELD_W], f[TEA_FIELD_KX], f[TEA_FIELD_KY],
                    c->pend_alpha, c->pend_beta, ahead || c->pend_u ? 1 : 0,
                    ahead || c->pend_halo ? 1 : 0, ahead ? c->u_alt : f[TEA_FIELD_U],
                    ahead ? c->ra_dev : nullptr, nullptr, nullptr, 0.0, 0.0};
  if (!ride) return TEA_HIP_OK;
  if (c->uh == 2) {
    s->um = 3;
    s->a.p_h = c->uh_p[0];
    s->a.alpha_h = c->uh_alpha[0];
    s->a.p_h2 = c->uh_p[1];
    s->a.alpha_h2 = c->uh_alpha[1];
    return TEA_HIP_OK;
  }
  s->um = 0;
  s->hold = c->uh + 1;
  for (int i = 0; i < c->uh; ++i) {
    s->hold_p[i] = c->uh_p[i];
    s->hold_alpha[i] = c->uh_alpha[i];
  }
  s->hold_p[c->uh] = f[TEA_FIELD_P];
  return TEA_HIP_OK;
}

// The chunk's state once a w-step has been asked for (or taken over), its u
// update's factor alpha.
void commit_cg_step(tea_hip_chunk* c, const CgStep& s, double alpha) {
  double** f = c->field;
  c->pend_u = c->pend_p = c->pend_halo = false;
  c->uh = s.hold;
  for (int i = 0; i < s.hold; ++i) {
    c->uh_p[i] = s.hold_p[i];
    c->uh_alpha[i] = i == s.hold - 1 ? alpha : s.hold_alpha[i];
  }
  if (s.um && s.a.apply_u && s.a.u_out != s.a.u) swap_ptr(f[TEA_FIELD_U], c->u_alt);
  if (s.a.w != f[TEA_FIELD_W]) swap_ptr(f[TEA_FIELD_W], c->w_alt);
  if (!s.apply_p) return;
  for (double*& b : c->p_alt)
    if (b == s.a.p_new) {
      swap_ptr(f[TEA_FIELD_P], b);
      break;
    }
}

// Queues the r-step behind the newest w-step.  rro: r.r before it, the value
// where the host has it.
int ra_queue_r(tea_hip_chunk* c, double rro, bool from_dev) {
  if (ra_consume(c)) TEA_RETURN_IF(ra_arm(c, kRaW, c->ra_wi));
  const RaScalar sc = ra_scalar_of(c, kRaW, c->ra_wi, rro, from_dev);
  {
    Timed t(c, K_CG_FUSED_R);
    hipLaunchKernelGGL(sc.sub ? fused_r1_kernel<true> : fused_r1_kernel<false>, pair_grid(c),
                       dim3(kBlock), 0, c->stream, c->geo, c->field[TEA_FIELD_R], c->r_alt,
                       c->ra_w ? c->w_alt : c->field[TEA_FIELD_W], 0.0, sc,
                       sc.sub ? c->sub2 : c->sub, c->nblk);
  }
  TEA_HIP_TRY(hipGetLastError());
  c->ra_ri ^= 1;
  TEA_RETURN_IF(ra_finish(c, kRaRStep, c->ra_ri, rro, from_dev));
  c->ra_r = true;
  return TEA_HIP_OK;
}

// Queues the next w-step behind the r-step in flight (r.r before that step:
// ra_rro).
int ra_queue_w(tea_hip_chunk* c) {
  TEA_RETURN_IF(plan_cg_w(c, true, &c->ra_step));
  if (ra_consume(c)) TEA_RETURN_IF(ra_arm(c, kRaRStep, c->ra_ri));
  TEA_RETURN_IF(
      launch_cg_step(c, c->ra_step, ra_scalar_of(c, kRaRStep, c->ra_ri, c->ra_rro, false)));
  c->ra_wi ^= 1;
  TEA_RETURN_IF(ra_finish(c, kRaW, c->ra_wi, 0.0, true));
  c->ra_w = true;
  return TEA_HIP_OK;
}

struct HeldUBody {
  double* __restrict__ u;
  const double* __restrict__ p0;
  const double* __restrict__ p1;
  double a0, a1;
  int n;
  Geo g;
  __device__ void operator()(int i, int kk, int jj) const {
    if (!interior(g, kk, jj)) return;
    double v = u[i] + a0 * p0[i];
    if (n == 2) v = v + a1 * p1[i];
    u[i] = v;
  }
};

}  // namespace

int ra_discard(tea_hip_chunk* c) {
  if (c->ra_r || c->ra_w) {
    c->ra_r = c->ra_w = false;
    c->ra_dirty = true;
  }
  return TEA_HIP_OK;
}

int apply_held_u(tea_hip_chunk* c) {
  if (c->uh == 0) return TEA_HIP_OK;
  TEA_RETURN_IF(ra_discard(c));
  const int n = c->uh;
  c->uh = 0;
  TEA_RETURN_IF(launch_each(c, K_CG_APPLY_PENDING,
                            HeldUBody{c->field[TEA_FIELD_U], c->uh_p[0], c->uh_p[n - 1],
                                      c->uh_alpha[0], c->uh_alpha[n - 1], n, c->geo}));
  static const int ext[4] = {-1, -1, -1, -1};
  int fields[TEA_HALO_NUM] = {0};
  fields[TEA_HALO_U] = 1;
  return launch_halos(c, 1, ext, fields);
}

int apply_pending(tea_hip_chunk* c) {
  TEA_RETURN_IF(drop_ahead(c, kAheadNone));
  c->mra_synced = false;
  TEA_RETURN_IF(apply_cg_pending(c));
  return flush_held(c);
}

int apply_cg_pending(tea_hip_chunk* c) {
  TEA_RETURN_IF(ra_discard(c));
  if (c->hold) TEA_RETURN_IF(apply_mp_hold(c));
  TEA_RETURN_IF(apply_held_u(c));
  if (!c->pend_u && !c->pend_p && !c->pend_halo) return TEA_HIP_OK;
  double** f = c->field;
  const bool halo_u = c->pend_u;  // the deferred ring update includes U
  if (c->pend_u || c->pend_p) {
    ApplyPendingBody body{f[TEA_FIELD_U], f[TEA_FIELD_P], f[TEA_FIELD_R],
                          c->pend_alpha, c->pend_beta, c->pend_u ? 1 : 0,
                          c->pend_p ? 1 : 0, c->geo};
    TEA_RETURN_IF(launch_each(c, K_CG_APPLY_PENDING, body));
    if (c->pend_p) c->p_alt_synced = false;
  }
  const bool halo = c->pend_halo;
  c->pend_u = c->pend_p = c->pend_halo = false;
  if (halo) {
    static const int ext[4] = {-1, -1, -1, -1};
    int fields[TEA_HALO_NUM] = {0};
    fields[TEA_HALO_U] = halo_u ? 1 : 0;
    fields[TEA_HALO_P] = 1;
    TEA_RETURN_IF(launch_halos(c, 1, ext, fields));
    c->p_alt_synced = false;
  }
  return TEA_HIP_OK;
}

}  // namespace tea

using namespace tea;

extern "C" {

int tea_hip_cg_init(tea_hip_chunk* c, int coefficient, double rx, double ry,
                    double* rro) {
  TEA_ENTER(c);
  TEA_CHECK_ARG(rro != nullptr, "null rro");
  TEA_CHECK_ARG(coefficient == TEA_CONDUCTIVITY ||
                    coefficient == TEA_RECIP_CONDUCTIVITY,
                "unknown conductivity model");
  TEA_RETURN_IF(apply_pending(c));
  c->faces_ok_u = c->faces_ok_p = false;
  double** f = c->field;
  const Geo g = c->geo;
  TEA_RETURN_IF(launch_each(
      c, K_CG_INIT_U,
      InitUBody{f[TEA_FIELD_P], f[TEA_FIELD_R], f[TEA_FIELD_U], f[TEA_FIELD_W],
                f[TEA_FIELD_DENSITY], f[TEA_FIELD_ENERGY], coefficient, g.x,
                g.y}));
  TEA_RETURN_IF(launch_each(c, K_CG_INIT_K,
                            InitKBody{f[TEA_FIELD_W], f[TEA_FIELD_KX],
                                      f[TEA_FIELD_KY], rx, ry, g.x, g.y, g.h}));
  c->p_alt_synced = false;
  TEA_RETURN_IF(launch_span1(c, K_CG_INIT_OTHERS,
                             InitOthersBody{f[TEA_FIELD_KX], f[TEA_FIELD_KY],
                                            f[TEA_FIELD_P], f[TEA_FIELD_R],
                                            f[TEA_FIELD_U], f[TEA_FIELD_W], g.x},
                             rro));
  // The host's first rro (TeaLeaf/drivers/cg_driver.c:45-52), for the
  // run-ahead's first alpha.
  c->ra_rro = *rro;
  c->ra_rro_known = true;
  c->ra_fail = 0;
  return TEA_HIP_OK;
}

int tea_hip_cg_calc_w(tea_hip_chunk* c, double* pw) {
  TEA_ENTER_RA(c);
  TEA_CHECK_ARG(pw != nullptr, "null pw");
  double** f = c->field;
  const Geo g = c->geo;
  if (c->ra_r || c->ra_w) {
    // The w-step in flight applied exactly the deferred work: take it over.
    if (c->ra_w && c->pend_u && c->pend_p && c->pend_halo && !c->held && c->pre_halo < 0 &&
        c->pend_alpha == c->ra_alpha && c->pend_beta == c->ra_beta) {
      commit_cg_step(c, c->ra_step, c->pend_alpha);
      c->taken[0] += 1;
      c->ra_w = false;
      c->ra_fail = 0;
      const int slot = c->ra_wi;
      TEA_RETURN_IF(ra_queue_w(c));  // its r-step is queued already
      return ra_wait(c, kRaW, slot, pw, &c->ra_alpha);
    }
    ra_mismatch(c);
  }
  TEA_FLUSH_HELD(c);
  if (!c->fused) {
    TEA_RETURN_IF(apply_pending(c));
    return launch_span1(c, K_CG_CALC_W,
                        CalcWBody{f[TEA_FIELD_P], f[TEA_FIELD_KX],
                                  f[TEA_FIELD_KY], f[TEA_FIELD_W], g.x},
                        pw);
  }
  // The run-ahead's buffers before those of the held updates, which gain less.
  const bool pair_blocks = use_pair_blocks(c, 1);
  const bool ahead = pair_blocks && ra_possible(c) && ensure_ra(c);
  if (pair_blocks) ensure_p_ring(c);
  const double alpha = c->pend_alpha;
  CgStep s;
  TEA_RETURN_IF(plan_cg_w(c, false, &s));
  const bool apply_p = s.apply_p;
  const FusedWArgs& args = s.a;
  int plen = c->nspan;
  if (pair_blocks) {
    if (ahead) {
      // Start a run-ahead: the spare buffers take the cells outside the
      // interior (and the ring) that no pass writes.
      TEA_RETURN_IF(copy_frames(c, FramePairs{{f[TEA_FIELD_R], f[TEA_FIELD_U], f[TEA_FIELD_W]},
                                              {c->r_alt, c->u_alt, c->w_alt}}, 3));
    }
    TEA_RETURN_IF(launch_cg_step(c, s, RaScalar{}));
    commit_cg_step(c, s, alpha);
    if (ahead) {
      c->ra_wi ^= 1;
      TEA_RETURN_IF(ra_finish(c, kRaW, c->ra_wi, c->ra_rro, false));
      TEA_RETURN_IF(ra_queue_r(c, c->ra_rro, false));
      const int slot = c->ra_wi;
      TEA_RETURN_IF(ra_queue_w(c));
      return ra_wait(c, kRaW, slot, pw, &c->ra_alpha);
    }
    TEA_RETURN_IF(launch_span_finish(c, 1, &plen, 0, true));
    return finish_reduction_n(c, 1, plen, pw);
  } else {
    Timed t(c, K_CG_FUSED_W);
    const int sg = c->ngroup == 1 ? 1 : 0;
#define TEA_FUSED_W(AP, B)                                                   \
  hipLaunchKernelGGL((fused_w_kernel<AP, B>), span_grid(c), dim3(kBlock), 0, \
                     c->stream, g, args, c->partials, c->nspan, sg)
#define TEA_FUSED_W2(AP, B)                                                   \
  hipLaunchKernelGGL((fused_w2_kernel<AP, B>), span_grid(c), dim3(kBlock), 0, \
                     c->stream, g, args, c->partials, c->nspan, sg)
    if (c->pairs) {
      if (!apply_p) TEA_FUSED_W2(false, 2);
      else if (c->batch == 1) TEA_FUSED_W2(true, 1);
      else if (c->batch == 2) TEA_FUSED_W2(true, 2);
      else TEA_FUSED_W2(true, 4);
    } else {
      if (!apply_p) TEA_FUSED_W(false, 4);
      else if (c->batch == 2) TEA_FUSED_W(true, 2);
      else if (c->batch == 8) TEA_FUSED_W(true, 8);
      else TEA_FUSED_W(true, 4);
    }
#undef TEA_FUSED_W
#undef TEA_FUSED_W2
  }
  TEA_HIP_TRY(hipGetLastError());
  commit_cg_step(c, s, alpha);
  return finish_reduction_n(c, 1, plen, pw);
}

int tea_hip_cg_calc_ur(tea_hip_chunk* c, double alpha, double* rrn) {
  TEA_ENTER_RA(c);
  TEA_CHECK_ARG(rrn != nullptr, "null rrn");
  double** f = c->field;
  if (c->ra_r || c->ra_w) {
    // The r-step in flight used the device's alpha: take it over when the
    // host's is the same.
    if (c->ra_r && c->ra_w && alpha == c->ra_alpha && !c->pend_u && !c->pend_p &&
        !c->pend_halo && !c->held && c->pre_halo < 0) {
      swap_ptr(f[TEA_FIELD_R], c->r_alt);
      c->taken[0] += 1;
      c->pend_u = true;
      c->pend_alpha = alpha;
      c->ra_r = false;
      const int slot = c->ra_ri;
      // The r-step of the w-step in flight, before waiting for this r.r.
      TEA_RETURN_IF(ra_queue_r(c, 0.0, true));
      TEA_RETURN_IF(ra_wait(c, kRaRStep, slot, rrn, &c->ra_beta));
      c->ra_rro = *rrn;
      c->ra_fail = 0;
      return TEA_HIP_OK;
    }
    ra_mismatch(c);
  }
  TEA_FLUSH_HELD(c);
  // Held u updates alone may stay held: this step leaves u and p alone.
  if (!c->fused || c->pend_u || c->pend_p || c->pend_halo) TEA_RETURN_IF(apply_pending(c));
  if (!c->fused)
    return launch_span1(c, K_CG_CALC_UR,
                        CalcURBody{f[TEA_FIELD_U], f[TEA_FIELD_R],
                                   f[TEA_FIELD_P], f[TEA_FIELD_W], alpha},
                        rrn);
  int rlen = c->nspan;
  if (use_pair_blocks(c, 2)) {
    {
      Timed t(c, K_CG_FUSED_R);
      hipLaunchKernelGGL(fused_r1_kernel<false>, pair_grid(c), dim3(kBlock), 0,
                         c->stream, c->geo, f[TEA_FIELD_R], f[TEA_FIELD_R], f[TEA_FIELD_W],
                         alpha, RaScalar{}, c->sub, c->nblk);
    }
    TEA_HIP_TRY(hipGetLastError());
    TEA_RETURN_IF(launch_span_finish(c, 1, &rlen, 0, true));
  } else {
    Timed t(c, K_CG_FUSED_R);
    if (c->pairs)
      hipLaunchKernelGGL(fused_r2_kernel, span_grid(c), dim3(kBlock), 0,
                         c->stream, c->geo, f[TEA_FIELD_R], f[TEA_FIELD_W],
                         alpha, c->partials, c->nspan, c->ngroup == 1 ? 1 : 0);
    else
      hipLaunchKernelGGL(fused_r_kernel, span_grid(c), dim3(kBlock), 0,
                         c->stream, c->geo, f[TEA_FIELD_R], f[TEA_FIELD_W],
                         alpha, c->partials, c->nspan, c->ngroup == 1 ? 1 : 0);
  }
  TEA_HIP_TRY(hipGetLastError());
  TEA_RETURN_IF(finish_reduction_n(c, 1, rlen, rrn));
  c->pend_u = true;
  c->pend_alpha = alpha;
  c->ra_rro = *rrn;  // the host's next rro (TeaLeaf/drivers/cg_driver.c:113)
  return TEA_HIP_OK;
}

int tea_hip_cg_calc_p(tea_hip_chunk* c, double beta) {
  TEA_ENTER_RA(c);
  // Only deferred: a run-ahead w-step stays in flight for cg_calc_w.
  if (c->held || c->pre_halo >= 0) TEA_FLUSH_HELD(c);
  double** f = c->field;
  if (!c->fused || c->pend_p || c->pend_halo) TEA_RETURN_IF(apply_pending(c));
  if (!c->fused) {
    c->p_alt_synced = false;
    return launch_each(c, K_CG_CALC_P,
                       CalcPBody{f[TEA_FIELD_P], f[TEA_FIELD_R], beta, c->geo});
  }
  c->pend_p = true;
  c->pend_beta = beta;
  return TEA_HIP_OK;
}

int tea_hip_copy_u(tea_hip_chunk* c) {
  TEA_ENTER(c);
  TEA_RETURN_IF(apply_pending(c));
  double** f = c->field;
  return launch_each(c, K_COPY_U,
                     CopyUBody{f[TEA_FIELD_U], f[TEA_FIELD_U0], c->geo});
}

int tea_hip_calculate_residual(tea_hip_chunk* c) {
  TEA_ENTER(c);
  TEA_RETURN_IF(apply_pending(c));
  double** f = c->field;
  return launch_each(c, K_CALC_RESIDUAL,
                     ResidualBody{f[TEA_FIELD_U], f[TEA_FIELD_U0],
                                  f[TEA_FIELD_R], f[TEA_FIELD_KX],
                                  f[TEA_FIELD_KY], c->geo});
}

int tea_hip_calculate_2norm(tea_hip_chunk* c, const double* buffer,
                            double* norm) {
  TEA_ENTER_HELD(c);
  TEA_CHECK_ARG(norm != nullptr, "null norm");
  int fid = -1;
  for (int f = 0; f < TEA_NUM_FIELDS; ++f)
    if (buffer == c->field[f] && c->field_len[f] >= (size_t)c->geo.n) fid = f;
  TEA_CHECK_ARG(fid >= 0, "buffer is not an x*y field of this chunk");
  // Deferred work can move the field to its second buffer: name it by field.
  TEA_RETURN_IF(apply_pending(c));
  const double* b = c->field[fid];
  if (!use_pair_blocks(c, 1))
    return launch_span1(c, K_CALC_2NORM, NormBody{b}, norm);
  {
    Timed t(c, K_CALC_2NORM);
    hipLaunchKernelGGL(norm_pair_kernel, pair_grid(c), dim3(kBlock), 0,
                       c->stream, c->geo, b, c->sub, c->nblk);
  }
  TEA_HIP_TRY(hipGetLastError());
  int len = c->nspan;
  TEA_RETURN_IF(launch_span_finish(c, 1, &len, 0, true));
  return finish_reduction_n(c, 1, len, norm);
}

int tea_hip_finalise(tea_hip_chunk* c) {
  TEA_ENTER(c);
  TEA_RETURN_IF(apply_pending(c));
  double** f = c->field;
  return launch_each(c, K_FINALISE,
                     FinaliseBody{f[TEA_FIELD_U], f[TEA_FIELD_DENSITY],
                                  f[TEA_FIELD_ENERGY], c->geo});
}

}  // extern "C"
