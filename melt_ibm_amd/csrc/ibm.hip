// Immersed-boundary kernels of the RK3 substep on gfx950:
//  - narrow-band signed-distance tagging (genSDF.f90) with a deterministic
//    arg-min (smallest distance, then lowest face index: the reference's
//    "first face wins"), so tags equal the serial CPU result bit for bit;
//  - init-time ray tagging (pencil_rayTag.f90, rayAux.f90);
//  - MLS shape functions (mlsWeight.f90), interpolation and force spreading
//    (mlsForce.f90, forc1-3.f90, forctemp.f90).  Spreading accumulates each
//    contribution as a 128-bit fixed-point integer, so the sum over faces is
//    exact and independent of scheduling order;
//  - MLS gradient probes for the heat flux (mls_heatFlux.f90) and the surface
//    loads (mls_structLoads.f90).
// All of this scales with the number of triangles, not with N^3.
#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>

#include "common.h"
#include "fixed128.h"

namespace {

constexpr double WCON = 0.3, WSCL = 1.5;  // initmls.f90:12-13

__device__ inline double gco(const Grid& g, int dim, int centre, int i) {
  if (dim == 0) return centre ? gxm(g, i) : gxc(g, i);
  if (dim == 1) return centre ? gym(g, i) : gyc(g, i);
  return centre ? gzm(g, i) : gzc(g, i);
}

__device__ inline double mls_gaussian(double r) {  // geom.f90:24-36
  if (r > 1.0) return 0.0;
  double t = r / WCON;
  return det_exp(-(t * t));
}
__device__ inline double mls_gauss_deriv(double r) {  // geom.f90:38-53
  if (r > 1.0) return 0.0;
  double t = r / WCON;
  return -2.0 * r / (WCON * WCON) * det_exp(-(t * t));
}

// A(i,j) += (w p_j) p_i : DGEMM('N','T',4,4,1,w,p,4,p,4,1,A,4)
__device__ inline void rank1(double A[16], double w, const double p[4]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    double temp = w * p[j];
#pragma unroll
    for (int i = 0; i < 4; ++i) A[i + 4 * j] = A[i + 4 * j] + temp * p[i];
  }
}

// MLS shape function over the 3x3x3 support i0..i0+2, j0.., k0.. (wght1/2/3/temp,
// mlsWeight.f90:48-412); c[d] selects face (0) or centre (1) coordinates.
// sink(inw, phi) receives the 27 values in the reference's k, j, i order.
template <class Sink>
__device__ int mls_phi(const Grid& g, const double pos[3], int i0, int j0, int k0, const int c[3], Sink sink) {
  double A[16];
#pragma unroll
  for (int q = 0; q < 16; ++q) A[q] = 0.0;
  // separable Gaussian factors, evaluated once per axis
  double xs[3], ys[3], zs[3], wx[3], wy[3], wz[3];
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    xs[q] = gco(g, 0, c[0], i0 + q);
    wx[q] = mls_gaussian(fabs(xs[q] - pos[0]) / (WSCL / g.dx1));
    ys[q] = gco(g, 1, c[1], j0 + q);
    wy[q] = mls_gaussian(fabs(ys[q] - pos[1]) / (WSCL / g.dx2));
    zs[q] = gco(g, 2, c[2], k0 + q);
    wz[q] = mls_gaussian(fabs(zs[q] - pos[2]) / (WSCL / g.dx3));
  }
#pragma unroll 1
  for (int kq = 0; kq < 3; ++kq)
#pragma unroll
    for (int jq = 0; jq < 3; ++jq) {
      double w23 = wy[jq] * wz[kq];
#pragma unroll
      for (int iq = 0; iq < 3; ++iq) {
        double wtx = wx[iq] * w23;
        double p[4] = {1.0, xs[iq], ys[jq], zs[kq]};
        rank1(A, wtx, p);
      }
    }
  int info = lu_inverse<4>(A);
  if (info) return info;
  double ptx[4] = {1.0, pos[0], pos[1], pos[2]}, ptxA[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    double s = 0.0;
#pragma unroll
    for (int l = 0; l < 4; ++l) s = s + (1.0 * A[l + 4 * j]) * ptx[l];
    ptxA[j] = s;
  }
#pragma unroll 1
  for (int kq = 0; kq < 3; ++kq)
#pragma unroll
    for (int jq = 0; jq < 3; ++jq) {
      double w23 = wy[jq] * wz[kq];
#pragma unroll
      for (int iq = 0; iq < 3; ++iq) {
        double wtx = wx[iq] * w23;
        double b[4] = {wtx * 1.0, wtx * xs[iq], wtx * ys[jq], wtx * zs[kq]};
        double s = 0.0;
#pragma unroll
        for (int l = 0; l < 4; ++l) s = s + (1.0 * b[l]) * ptxA[l];
        sink(9 * kq + 3 * jq + iq, s);
      }
    }
  return 0;
}

// The weight derivative of one axis; inv = 1 / scale.
__device__ inline double dweight(double dist, double nrm, double inv) {
  if (nrm < 2.220446049250313e-16) return 0.0;  // EPSILON(1.0d0)
  return mls_gauss_deriv(nrm) * copysign(inv, dist);   // dist / |dist| / scale
}

// Order the LDS accesses of one wave (its lanes run in step).
__device__ inline void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Exchange area of the 64 probes of a k_probes_grad block.
struct GradShared {
  double crd[9][64], w[9][64], dw[9][64];   // coordinate, weight and its derivative of (axis, point) pair 3 axis + point
  double A[16][64];                         // moment matrix, then its inverse
  double pg[4][64];                         // probe position, then gamma
  int info[64];                             // -1: no probe
};

// MLS gradient at a probe (wght_gradT mls_heatFlux.f90:85-300 and
// wght_gradP/U/V/W mls_structLoads.f90:380-1297), computed by the 4 lanes of
// one probe: lane 0 accumulates the moment matrix A, lane 1+d the derivative
// matrix dA/dx_d; one wave inverts the block's 64 matrices, a lane each (a
// different wave from block to block, for the SIMDs' sake); lanes 1..3 form
// gradient component d in the reference's point order, so every value rounds
// as in the single-thread formulation.
// kz: grid indices used for the z coordinate (the reference uses k1-1, k1,
// k1); ke: field planes (1-based, ghost-plane semantics) k1-1, k1, k1+1.
// Must be reached by every thread of the block (it contains barriers);
// active = 0 lanes only take part in the barriers.  Returns the LU info of A
// on lanes 1..3 (0 elsewhere); with COEF the 27 shape-function derivatives of
// component lane-1 go to coef[q cstride], otherwise *grad_d receives their sum
// against the field.
//
// Bound by its FP64 instructions: 4350 a wave and 88 us for six probes of 20480
// faces on 128^3 with every lane forming all nine coordinates and the inverse,
// a branch per point for the lane's weight and a wrap per point of the field; 2970
// and 60 us this way (with COEF, 5120 faces beside the explicit pass: 25 -> 18).
template <bool COEF, typename R>
__device__ __forceinline__ int mls_grad_lanes(const Grid& g, GradShared& sh, const R* __restrict__ fld, const double pos[3], int ic, int jc,
                                              const int kz[3], const int ke[3], const int c[3], int lane, bool active, double* grad_d,
                                              double* coef, size_t cstride) {
  const int slot = threadIdx.x >> 2;
  double M[16];   // column 0 only stands for row 0 too: (w 1) p_i and (w p_i) 1 round alike
  if (active) {
    // pair p = 3 axis + point is evaluated on lane p % 4 of the probe's lanes
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      const int pp = lane + 4 * r, ax = pp / 3, q = pp - 3 * ax;
      if (pp >= 9) continue;
      // selects, not an indexed pick (which would put the arrays in scratch)
      const int i = ax == 0 ? ic - 1 + q : ax == 1 ? jc - 1 + q : q == 0 ? kz[0] : q == 1 ? kz[1] : kz[2];
      const double n = ax == 0 ? (double)g.n1 : ax == 1 ? (double)g.n2 : (double)g.n3;
      const double len = ax == 0 ? g.xlen : ax == 1 ? g.ylen : g.zlen;
      const double pc = ax == 0 ? pos[0] : ax == 1 ? pos[1] : pos[2];
      const double sc = WSCL / (ax == 0 ? g.dx1 : ax == 1 ? g.dx2 : g.dx3);
      const bool centre = (ax == 0 ? c[0] : ax == 1 ? c[1] : c[2]) != 0;
      double x = len * ((double)(i - 1) / n);          // gco(g, ax, centre, i)
      if (centre) x = (x + len * ((double)i / n)) * 0.5;
      const double nrm = fabs(pc - x) / sc;
      sh.crd[pp][slot] = x;
      sh.w[pp][slot] = mls_gaussian(nrm);
      sh.dw[pp][slot] = dweight(pc - x, nrm, 1.0 / sc);
    }
    wave_lds_fence();
    // this lane's factors: the derivative's on its own axis
    const double(*fx)[64] = lane == 1 ? sh.dw : sh.w;
    const double(*fy)[64] = lane == 2 ? sh.dw : sh.w;
    const double(*fz)[64] = lane == 3 ? sh.dw : sh.w;
    double xs[3], ys[3], f1[3], f2[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      xs[q] = sh.crd[q][slot]; ys[q] = sh.crd[3 + q][slot];
      f1[q] = fx[q][slot]; f2[q] = fy[3 + q][slot];
    }
#pragma unroll
    for (int q = 0; q < 16; ++q) M[q] = 0.0;
#pragma unroll 1
    for (int nk = 0; nk < 3; ++nk) {
      const double zk = sh.crd[6 + nk][slot], f3 = fz[6 + nk][slot];
      // lane 0: w1 (w2 w3); the others: (f1 f2) f3
      double G[3], H[3];
#pragma unroll
      for (int q = 0; q < 3; ++q) { G[q] = lane == 0 ? f3 : f1[q]; H[q] = lane == 0 ? f1[q] : f3; }
#pragma unroll
      for (int jq = 0; jq < 3; ++jq)
#pragma unroll
        for (int iq = 0; iq < 3; ++iq) {
          const double wgt = (f2[jq] * G[iq]) * H[iq];
          const double p[3] = {xs[iq], ys[jq], zk};
          M[0] = M[0] + wgt;
#pragma unroll
          for (int j = 0; j < 3; ++j) {
            const double temp = wgt * p[j];
            M[j + 1] = M[j + 1] + temp;
#pragma unroll
            for (int i = 0; i < 3; ++i) M[i + 1 + 4 * (j + 1)] = M[i + 1 + 4 * (j + 1)] + temp * p[i];
          }
        }
    }
#pragma unroll
    for (int j = 1; j < 4; ++j) M[4 * j] = M[j];
  }
  if (lane == 0) {
    sh.info[slot] = active ? 0 : -1;
    if (active) {
#pragma unroll
      for (int q = 0; q < 16; ++q) sh.A[q][slot] = M[q];
#pragma unroll
      for (int q = 0; q < 3; ++q) sh.pg[q][slot] = pos[q];
    }
  }
  __syncthreads();
  if ((threadIdx.x >> 6) == (blockIdx.x & 3)) {
    const int t = threadIdx.x & 63;
    if (sh.info[t] == 0) {
      double A[16], gam[4];
#pragma unroll
      for (int q = 0; q < 16; ++q) A[q] = sh.A[q][t];
      sh.info[t] = lu_inverse<4>(A);
      const double ptx[4] = {1.0, sh.pg[0][t], sh.pg[1][t], sh.pg[2][t]};
#pragma unroll
      for (int i = 0; i < 4; ++i) gam[i] = 0.0;
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) gam[i] = gam[i] + ptx[j] * A[i + 4 * j];
#pragma unroll
      for (int q = 0; q < 16; ++q) sh.A[q][t] = A[q];
#pragma unroll
      for (int q = 0; q < 4; ++q) sh.pg[q][t] = gam[q];
    }
  }
  __syncthreads();
  if (!active || lane == 0) return 0;
  if (const int info = sh.info[slot]) return info;
  const int d = lane - 1;
  double gam[4], pv[4], dg[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) { gam[i] = sh.pg[i][slot]; pv[i] = i == d + 1 ? 1.0 : 0.0; }   // unit vector e_(d+1), in registers
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    double t = -1.0 * gam[j];
#pragma unroll
    for (int i = 0; i < 4; ++i) pv[i] = pv[i] + t * M[i + 4 * j];
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) dg[i] = 0.0;
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) dg[i] = dg[i] + pv[j] * sh.A[i + 4 * j][slot];
  const double(*fx)[64] = lane == 1 ? sh.dw : sh.w;
  const double(*fy)[64] = lane == 2 ? sh.dw : sh.w;
  const double(*fz)[64] = lane == 3 ? sh.dw : sh.w;
  double xs[3], ys[3], w1[3], w2[3], f1[3], f2[3];
  int ci[3] = {0, 0, 0}, cj[3] = {0, 0, 0};
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    xs[q] = sh.crd[q][slot]; ys[q] = sh.crd[3 + q][slot];
    w1[q] = sh.w[q][slot]; w2[q] = sh.w[3 + q][slot];
    f1[q] = fx[q][slot]; f2[q] = fy[3 + q][slot];
    if (!COEF) { ci[q] = pmod(ic - 2 + q, g.n1); cj[q] = pmod(jc - 2 + q, g.n2); }
  }
  double s = 0.0;
#pragma unroll 1
  for (int nk = 0; nk < 3; ++nk) {
    const double zk = sh.crd[6 + nk][slot], w3k = sh.w[6 + nk][slot], f3 = fz[6 + nk][slot];
    const int kk = COEF ? 0 : pmod((nk == 0 ? ke[0] : nk == 1 ? ke[1] : ke[2]) - 1, g.n3);
#pragma unroll
    for (int jq = 0; jq < 3; ++jq) {
      const R* line = COEF ? nullptr : fld + cidx(g, 0, cj[jq], kk);
#pragma unroll
      for (int iq = 0; iq < 3; ++iq) {
        double wtx = w1[iq] * (w2[jq] * w3k);
        double p[4] = {1.0, xs[iq], ys[jq], zk};
        double dw = f1[iq] * f2[jq] * f3;
        double acc = 0.0;
#pragma unroll
        for (int l = 0; l < 4; ++l) acc = acc + (wtx * p[l]) * dg[l];
#pragma unroll
        for (int l = 0; l < 4; ++l) acc = acc + (dw * p[l]) * gam[l];
        if constexpr (COEF) coef[(size_t)(9 * nk + 3 * jq + iq) * cstride] = acc;   // geometry only
        else s = s + acc * (double)line[ci[iq]];
      }
    }
  }
  *grad_d = s;
  return 0;
}

// ---------------------------------------------------- 128-bit accumulation
// acc_split / acc_value (fixed128.h) hold each contribution exactly as a
// 64.64 fixed-point integer; the atomics add the two words with carry.  The
// high word changes only when the running sum crosses a multiple of 2^64
// (for a small negative contribution its all-ones high word and the carry
// cancel), so its atomic is issued only when hi + carry is not zero.
__device__ inline void acc_add_split(unsigned long long* w /* [lo, hi] */, unsigned long long lo, unsigned long long hi) {
  if ((lo | hi) == 0) return;
  unsigned long long old = atomicAdd(&w[0], lo);
  unsigned long long carry = (old + lo < old) ? 1ull : 0ull;
  if (hi + carry) atomicAdd(&w[1], hi + carry);
}
__device__ inline void acc_add(unsigned long long* w, double v) {
  unsigned long long lo, hi;
  acc_split(v, lo, hi);
  acc_add_split(w, lo, hi);
}

__device__ inline long long win_slot(const int org[3], const int E[3], int iu, int ju, int ku) {
  int a = iu - org[0], b = ju - org[1], c = ku - org[2];
  if (a < 0 || b < 0 || c < 0 || a >= E[0] || b >= E[1] || c >= E[2]) return -1;
  return (long long)a + (long long)E[0] * ((long long)b + (long long)E[1] * c);
}

struct Win3 { int e[3]; };

// ------------------------------------------------------------ windows
// Face base indices floor(x*dx)+1 (unwrapped) bound every cell the MLS
// supports (base-1..base+2) and the tagging band (base-2..base+2) touch.
// Min / max of the face base indices over all live faces: one block per 256
// faces, wave shuffles and then integer atomics (order-independent; shared
// atomics of 256 threads on one address serialise, 15 -> 5 us for the tagging's
// set-up).
__device__ void window_box_block(const Grid& g, const double* __restrict__ bar, const unsigned char* __restrict__ gf, int nf, melt_window* win,
                                 int blk) {
  __shared__ int mn[3][4], mx[3][4];
  const int f = blk * 256 + (int)threadIdx.x, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const bool live = f < nf && !gf[f];
  const double dx[3] = {g.dx1, g.dx2, g.dx3};
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const int b = live ? (int)floor(bar[3 * f + d] * dx[d]) + 1 : 0;
    int lo = live ? b : INT_MAX, hi = live ? b : INT_MIN;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      lo = min(lo, __shfl_xor(lo, o, 64));
      hi = max(hi, __shfl_xor(hi, o, 64));
    }
    if (lane == 0) { mn[d][w] = lo; mx[d][w] = hi; }
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    const int d = threadIdx.x;
    atomicMin(&win->bmin[d], min(min(mn[d][0], mn[d][1]), min(mn[d][2], mn[d][3])));
    atomicMax(&win->bmax[d], max(max(mx[d][0], mx[d][1]), max(mx[d][2], mx[d][3])));
  }
}
__global__ __launch_bounds__(256) void k_window_box(Grid g, const double* __restrict__ bar, const unsigned char* __restrict__ gf, int nf,
                                                    melt_window* win) {
  window_box_block(g, bar, gf, nf, win, blockIdx.x);
}

// Initial state of the windows: no box placed yet, empty extents.
__global__ void k_window_reset(melt_window* win, int n) {
  for (int w = 0; w < n; ++w) {
    for (int d = 0; d < 3; ++d) {
      win[w].org[d] = 0; win[w].prev_org[d] = 0;
      win[w].bmin[d] = INT_MAX; win[w].bmax[d] = INT_MIN;
    }
    win[w].prev_valid = 0;
    win[w].pad = 0;
  }
}

// Place the forcing (which & 1: win[0]) and / or tagging (which & 2: win[1])
// box from the face extent in win[0].bmin/bmax (one thread).
__device__ void window_place(melt_window* win, const Win3& ef, const Win3& et, int which, int* err) {
  const int* mn = win[0].bmin;
  const int* mx = win[0].bmax;
  if (which & 1) {  // forcing window
    melt_window& w = win[0];
    for (int d = 0; d < 3; ++d) {
      w.org[d] = mn[d] - 2;
      if (mx[d] + 3 - w.org[d] >= ef.e[d]) raise_error(err, MELT_ERR_WINDOW);
    }
  }
  if (which & 2) {  // tagging window
    melt_window& w = win[1];
    if (w.prev_valid >= 0) {
      for (int d = 0; d < 3; ++d) w.prev_org[d] = w.org[d];
      w.prev_valid = w.pad;
    }
    for (int d = 0; d < 3; ++d) {
      w.org[d] = mn[d] - 2;
      if (mx[d] + 2 - w.org[d] >= et.e[d]) raise_error(err, MELT_ERR_WINDOW);
    }
    w.pad = 1;  // current box is valid from now on
  }
}
// Reset the extent for the next call.
__device__ void window_reset_extent(melt_window* win) {
  for (int d = 0; d < 3; ++d) { win[0].bmin[d] = INT_MAX; win[0].bmax[d] = INT_MIN; }
}
__global__ void k_window_final(melt_window* win, Win3 ef, Win3 et, int which, int* err) {
  window_place(win, ef, et, which, err);
  window_reset_extent(win);
}

// ------------------------------------------------------------ narrow band
// genSDF.f90:85-234, Eberly's point-triangle distance.  The regions' cases
// select one quotient, so a wave whose points lie in several regions divides
// once (0/1 and 1/1 stand for the parameters 0 and 1).
struct TriEdges {   // of one face, formed once
  double V0[3], E0[3], E1[3], a, b, c, det;
};
__device__ inline TriEdges tri_edges(const double* V0, const double* V1, const double* V2) {
  TriEdges T;
  for (int d = 0; d < 3; ++d) { T.V0[d] = V0[d]; T.E0[d] = V1[d] - V0[d]; T.E1[d] = V2[d] - V0[d]; }
  const double* E0 = T.E0;
  const double* E1 = T.E1;
  T.a = E0[0] * E0[0] + E0[1] * E0[1] + E0[2] * E0[2];
  T.b = E0[0] * E1[0] + E0[1] * E1[1] + E0[2] * E1[2];
  T.c = E1[0] * E1[0] + E1[1] * E1[1] + E1[2] * E1[2];
  T.det = T.a * T.c - T.b * T.b;
  return T;
}
__device__ double dist_point_tri(const double P[3], const TriEdges& T) {
  const double a = T.a, b = T.b, c = T.c, det = T.det;
  double DE[3];
  for (int d = 0; d < 3; ++d) DE[d] = T.V0[d] - P[d];
  const double d = T.E0[0] * DE[0] + T.E0[1] * DE[1] + T.E0[2] * DE[2];
  const double e = T.E1[0] * DE[0] + T.E1[1] * DE[1] + T.E1[2] * DE[2];
  double s = b * e - c * d, t = b * d - a * e;
  const bool in = s + t <= det, sn = s < 0.0, tn = t < 0.0;
  // past the edge opposite V0: the parameter t1 of the corner tested first
  const double t0 = sn ? b + d : b + e, t1 = sn ? c + e : a + d;
  const bool far = !in && (!(sn || tn) || t1 > t0);          // on that edge
  const bool edge1 = in ? sn && !(tn && d < 0.0) : sn;       // else on E1 (s = 0) or E0 (t = 0)
  const double g = edge1 ? e : d, h = edge1 ? c : a;
  const bool inner = in && !sn && !tn;
  double num, den;
  if (inner) { num = 1.0; den = det; }
  else if (far) {
    num = sn || tn ? t1 - t0 : c + e - b - d;
    den = a - 2.0 * b + c;
    const bool zero = !(sn || tn) && num <= 0.0, one = num >= den;
    if (zero || one) { num = zero ? 0.0 : 1.0; den = 1.0; }
  } else {
    const bool one = in ? !(g >= 0.0) && -g >= h : t1 <= 0.0, zero = !one && g >= 0.0;
    num = one ? 1.0 : zero ? 0.0 : -g;
    den = one || zero ? 1.0 : h;
  }
  const double q = num / den;
  if (inner) { s = s * q; t = t * q; }
  else if (far) {
    const bool on_t = !sn && tn;   // the quotient is t there, s elsewhere
    s = on_t ? 1.0 - q : q;
    t = on_t ? q : 1.0 - q;
  } else { s = edge1 ? 0.0 : q; t = edge1 ? q : 0.0; }
  double r[3];
  for (int k = 0; k < 3; ++k) r[k] = (T.V0[k] + s * T.E0[k] + t * T.E1[k]) - P[k];
  return sqrt(r[0] * r[0] + r[1] * r[1] + r[2] * r[2]);
}

// The tagging's set-up in one launch: blocks [0, nbox) reduce the face
// extent (as k_window_box), the other 256 set sdf to 999 over the window the
// previous tagging wrote (that tagging's cells are re-tagged from scratch)
// and clear the per-cell keys.  This runs before window_place moves the
// tagging window, so it takes the previous window from where its update leaves
// it (prev_org := org, prev_valid := pad, while prev_valid >= 0).
template <typename R>
__global__ __launch_bounds__(256) void k_tag_prepare(Grid g, const double* __restrict__ bar, const unsigned char* __restrict__ gf, int nf,
                                                     int nbox, melt_window* win, R* __restrict__ sdf, Win3 et,
                                                     unsigned long long* __restrict__ key, int* __restrict__ face, size_t ncell) {
  if ((int)blockIdx.x < nbox) {
    window_box_block(g, bar, gf, nf, win, blockIdx.x);
    return;
  }
  // (window cells are below 2^30: 32-bit indices)
  const unsigned t0 = (blockIdx.x - (unsigned)nbox) * 256u + threadIdx.x, step = (gridDim.x - (unsigned)nbox) * 256u;
  const melt_window& w = win[1];
  const bool moved = w.prev_valid >= 0;
  if ((moved ? w.pad : w.prev_valid) > 0) {
    const int o0 = moved ? w.org[0] : w.prev_org[0], o1 = moved ? w.org[1] : w.prev_org[1], o2 = moved ? w.org[2] : w.prev_org[2];
    const unsigned e0 = (unsigned)et.e[0], e1 = (unsigned)et.e[1], n = e0 * e1 * (unsigned)et.e[2];
    for (unsigned s = t0; s < n; s += step) {
      const unsigned r = s / e0, c = r / e1;
      sdf[widx(g, o0 + (int)(s - r * e0), o1 + (int)(r - c * e1), o2 + (int)c)] = R(999.0);
    }
  }
  for (unsigned s = t0; s < ncell; s += step) {
    key[s] = ~0ull;
    face[s] = INT_MAX;
  }
}

struct MeshArgs {
  const double* __restrict__ xyzv;
  const double* __restrict__ bar;
  const double* __restrict__ nor;
  const int* __restrict__ vof;
  const unsigned char* __restrict__ gf;
  int nf;
};

// A block's open-addressing table of window cells in LDS: `slot` of a cell,
// claimed on first use, or -1 once PROBES neighbours are taken by others (the
// caller then works on the cell in memory).  Neighbouring faces share most of
// their stencil cells, whatever the mesh's order makes of the group's extent,
// so one update per cell and block leaves the CU instead of one per (face, cell).
template <int N>
struct CellTable {
  static constexpr int PROBES = 8, RUN = 8;   // RUN neighbours of a line stay together: 128 bytes of accumulators
  static_assert((N & (N - 1)) == 0, "a power of two");
  int cell[N];   // -1: free
  __device__ int slot(int s) {
    unsigned h = ((unsigned)s / RUN * 2654435761u >> (32 - __builtin_ctz(N / RUN))) * RUN + (unsigned)s % RUN;
#pragma unroll 1
    for (int q = 0; q < PROBES; ++q) {
      int have = cell[h];
      if (have == -1) have = atomicCAS(&cell[h], -1, s);
      if (have == -1 || have == s) return (int)h;
      h = (h + RUN) & (N - 1);
    }
    return -1;
  }
};

// Passes of the narrow-band tagging over groups of FPB faces.
//
// k_tag_band: distance of every (face, band cell) of a group, the min per cell
// and the lowest face among the minima in LDS first, then one update of the
// cell's key; the group's winners are left as records for the other two passes.
// A group that touches more cells than its table or its records hold updates
// the keys entry by entry and leaves its distances instead (count < 0).
// k_tag_pass MODE 1: lowest face among the minima of all groups; 2: write sdf
// and VOFp.
// Neighbouring faces share most of their cells: a key update per entry (2.56 M
// atomics for 20480 faces) and two more passes over all entries took 51 + 11 +
// 20 us on 128^3; per group 28 + 5 + 9, the first bound by the distances'
// arithmetic (36 before a wave's regions shared one division and the band's
// coordinates were formed once per face).
//
// The window follows from the extent k_tag_prepare reduced: k_tag_band and mode
// 1 take its origin straight from there, one thread of mode 1 places the
// windows (no thread before mode 2 reads the placed origin), and one of mode 2
// resets the extent (mode 2 reads the placed origin), so no launch of its own does.
struct TagRecord {
  unsigned long long key;   // the distance's bits
  int cell, face;
};

// A group's share of the distances' memory: up to 125 distances a face, or
// records, and behind the distances of all faces the groups' record counts.
template <int FPB>
struct TagGroup {
  double* dist;
  int* count;
  int f0, nface;
  __device__ TagGroup(double* dst, int nf, int group) {
    f0 = group * FPB;
    nface = min(FPB, nf - f0);
    dist = dst + (size_t)f0 * 125;
    count = reinterpret_cast<int*>(dst + (size_t)nf * 125) + group;
  }
  __device__ TagRecord* records() const { return reinterpret_cast<TagRecord*>(dist); }
  __device__ int capacity() const { return nface * 125 / 2; }
};

template <int FPB, int CELLS>
struct BandShared {
  CellTable<CELLS> tab;
  unsigned long long kmin[CELLS];
  int fmin[CELLS];
  TriEdges tri[FPB];
  double crd[FPB][15];   // the band's x, y and z (a division each)
  int base[FPB][3];
  bool alive[FPB];
  int used, full;
};
struct BandArgs {
  const melt_window* __restrict__ win;
  Win3 et;
  unsigned long long* __restrict__ key;
  double* __restrict__ dst;
};

template <int FPB, int T, int CELLS>
__device__ void tag_band_block(const Grid& g, const MeshArgs& M, const BandArgs& B, BandShared<FPB, CELLS>& sh, int group, int* err) {
  constexpr int E = (FPB * 125 + T - 1) / T;   // entries per thread
  const TagGroup<FPB> G(B.dst, M.nf, group);
  const int t = threadIdx.x, n = G.nface * 125;
  if (t < FPB) {
    const int f = G.f0 + t;
    const bool live = t < G.nface && !M.gf[f];
    sh.alive[t] = live;
    if (live) {
      const int* v = &M.vof[3 * f];
      sh.tri[t] = tri_edges(&M.xyzv[3 * v[0]], &M.xyzv[3 * v[1]], &M.xyzv[3 * v[2]]);
    }
  }
  for (int u = t; u < G.nface * 15; u += T) {
    const int r = u / 15, m = u - 15 * r, d = m / 5, o = m - 5 * d;
    const double x = M.bar[3 * (G.f0 + r) + d];
    const int i0 = (int)floor(x * (d == 0 ? g.dx1 : d == 1 ? g.dx2 : g.dx3)) + 1, i = i0 + o - 2;
    sh.crd[r][m] = d == 0 ? gxm(g, i) : d == 1 ? gym(g, i) : gzm(g, i);
    if (o == 0) sh.base[r][d] = i0;
  }
  for (int q = t; q < CELLS; q += T) { sh.tab.cell[q] = -1; sh.kmin[q] = ~0ull; sh.fmin[q] = INT_MAX; }
  if (t == 0) { sh.used = 0; sh.full = 0; }
  __syncthreads();
  int org[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) org[d] = B.win[0].bmin[d] - 2;
  unsigned long long dk[E];
  int cell[E], slot[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int id = t + e * T, r = id / 125, q = id - 125 * r;
    cell[e] = slot[e] = -1;
    dk[e] = 0ull;
    if (id >= n || !sh.alive[r]) continue;
    const int oi = q % 5, oj = (q / 5) % 5, ok = q / 25;
    const long long s = win_slot(org, B.et.e, sh.base[r][0] + oi - 2, sh.base[r][1] + oj - 2, sh.base[r][2] + ok - 2);
    if (s < 0) { raise_error(err, MELT_ERR_WINDOW); continue; }
    const double P[3] = {sh.crd[r][oi], sh.crd[r][5 + oj], sh.crd[r][10 + ok]};
    dk[e] = (unsigned long long)__double_as_longlong(dist_point_tri(P, sh.tri[r]));
    cell[e] = (int)s;   // window cells are below 2^30
    slot[e] = sh.tab.slot((int)s);
    if (slot[e] >= 0) atomicMin(&sh.kmin[slot[e]], dk[e]);
    else sh.full = 1;
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < E; ++e)
    if (slot[e] >= 0 && sh.kmin[slot[e]] == dk[e]) atomicMin(&sh.fmin[slot[e]], G.f0 + (t + e * T) / 125);
  for (int q0 = 0; q0 < CELLS; q0 += T) {
    const unsigned long long m = __ballot(sh.tab.cell[q0 + t] >= 0);
    if ((t & 63) == 0 && m) atomicAdd(&sh.used, (int)__popcll(m));
  }
  __syncthreads();
  const int count = sh.used;
  if (sh.full || count > G.capacity()) {
    if (t == 0) *G.count = -1;
#pragma unroll
    for (int e = 0; e < E; ++e)
      if (cell[e] >= 0) {
        G.dist[t + e * T] = __longlong_as_double((long long)dk[e]);
        atomicMin(&B.key[cell[e]], dk[e]);
      }
    return;
  }
  __syncthreads();
  if (t == 0) { *G.count = count; sh.used = 0; }
  __syncthreads();
  for (int q0 = 0; q0 < CELLS; q0 += T) {
    const int q = q0 + t, c = sh.tab.cell[q];
    const unsigned long long m = __ballot(c >= 0);
    int at = 0;
    if ((t & 63) == 0 && m) at = atomicAdd(&sh.used, (int)__popcll(m));
    at = __shfl(at, 0, 64) + (int)__popcll(m & ((1ull << (t & 63)) - 1ull));
    if (c >= 0) {
      G.records()[at] = TagRecord{sh.kmin[q], c, sh.fmin[q]};
      atomicMin(&B.key[c], sh.kmin[q]);
    }
  }
}

template <int FPB, int T, int CELLS>
__global__ __launch_bounds__(T) void k_tag_band(Grid g, MeshArgs M, BandArgs B, int* err) {
  __shared__ BandShared<FPB, CELLS> sh;
  tag_band_block<FPB, T, CELLS>(g, M, B, sh, blockIdx.x, err);
}

template <int MODE, int FPB, typename R>
__global__ __launch_bounds__(256) void k_tag_pass(Grid g, MeshArgs M, melt_window* __restrict__ win, Win3 ef, Win3 et, int which,
                                                  const unsigned long long* __restrict__ key, int* __restrict__ face,
                                                  double* __restrict__ dst, R* __restrict__ sdf, R* __restrict__ vofp, double pi, int* err) {
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (MODE == 1) window_place(win, ef, et, which, err);
    else window_reset_extent(win);
  }
  const TagGroup<FPB> G(dst, M.nf, blockIdx.x);
  int org[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) org[d] = MODE == 2 ? win[1].org[d] : win[0].bmin[d] - 2;
  const int count = *G.count;
  for (int id = threadIdx.x; id < (count >= 0 ? count : G.nface * 125); id += 256) {
    int f, s, i, j, k;
    unsigned long long dk;
    if (count >= 0) {
      const TagRecord rec = G.records()[id];
      dk = rec.key; s = rec.cell; f = rec.face;
      const int r = s / et.e[0], c = r / et.e[1];
      i = org[0] + (s - r * et.e[0]); j = org[1] + (r - c * et.e[1]); k = org[2] + c;
    } else {
      const int q = id % 125;
      f = G.f0 + id / 125;
      if (M.gf[f]) continue;
      const double* pos = &M.bar[3 * f];
      i = (int)floor(pos[0] * g.dx1) + 1 + q % 5 - 2;
      j = (int)floor(pos[1] * g.dx2) + 1 + (q / 5) % 5 - 2;
      k = (int)floor(pos[2] * g.dx3) + 1 + q / 25 - 2;
      const long long w = win_slot(org, et.e, i, j, k);
      if (w < 0) continue;   // reported by k_tag_band
      s = (int)w;
      dk = (unsigned long long)__double_as_longlong(G.dist[id]);
    }
    if constexpr (MODE == 1) {
      if (key[s] == dk) atomicMin(&face[s], f);
    } else if (face[s] == f) {
      const double dist = __longlong_as_double((long long)dk);
      const double* pos = &M.bar[3 * f];
      double P[3] = {gxm(g, i), gym(g, j), gzm(g, k)};
      const double* n = &M.nor[3 * f];
      double dot = n[0] * (pos[0] - P[0]) + n[1] * (pos[1] - P[1]) + n[2] * (pos[2] - P[2]);
      double sgn = signbit(dot) ? -1.0 : 1.0;
      double sg = dist * (-sgn);
      size_t c = widx(g, i, j, k);
      sdf[c] = (R)sg;
      double eps = 1.0 / g.dx1, v;  // sdf_to_VOF genSDF.f90:237-255
      if (sg <= -eps) v = 0.0;
      else if (sg >= eps) v = 1.0;
      else v = 0.5 * (1.0 + sg * g.dx1 + (1.0 / pi) * det_sin(pi * sg * g.dx1));
      vofp[c] = (R)v;
    }
  }
}

// ------------------------------------------------------------ ray tagging
__device__ bool edge_sq(double y1, double z1, double y2, double z2, double ymin, double ymax, double zmin, double zmax) {
  double t, y, z;  // rayAux.f90:139-190
  if (y1 != y2) {
    t = (ymin - y1) / (y2 - y1);
    if (t >= 0.0 && t <= 1.0) { z = z1 + t * (z2 - z1); if (z >= zmin && z <= zmax) return true; }
    t = (ymax - y1) / (y2 - y1);
    if (t >= 0.0 && t <= 1.0) { z = z1 + t * (z2 - z1); if (z >= zmin && z <= zmax) return true; }
  }
  if (z1 != z2) {
    t = (zmin - z1) / (z2 - z1);
    if (t >= 0.0 && t <= 1.0) { y = y1 + t * (y2 - y1); if (y >= ymin && y <= ymax) return true; }
    t = (zmax - z1) / (z2 - z1);
    if (t >= 0.0 && t <= 1.0) { y = y1 + t * (y2 - y1); if (y >= ymin && y <= ymax) return true; }
  }
  return false;
}

__device__ bool yz_range(const double* V0, const double* V1, const double* V2, double ymin, double ymax, double zmin, double zmax) {
  double yv[3] = {V0[1], V1[1], V2[1]}, zv[3] = {V0[2], V1[2], V2[2]};  // rayAux.f90:86-113
  for (int i = 0; i < 3; ++i)
    if (yv[i] >= ymin && yv[i] <= ymax && zv[i] >= zmin && zv[i] <= zmax) return true;
  double ymx = fmax(fmax(yv[0], yv[1]), yv[2]), ymn = fmin(fmin(yv[0], yv[1]), yv[2]);
  double zmx = fmax(fmax(zv[0], zv[1]), zv[2]), zmn = fmin(fmin(zv[0], zv[1]), zv[2]);
  if (ymx < ymin || ymn > ymax || zmx < zmin || zmn > zmax) return false;
  for (int i = 0; i < 3; ++i) {
    int j = (i + 1) % 3;
    if (edge_sq(yv[i], zv[i], yv[j], zv[j], ymin, ymax, zmin, zmax)) return true;
  }
  return false;
}

struct Box { int lo[3], hi[3]; };

__global__ __launch_bounds__(256) void k_pencil_build(Grid g, MeshArgs M, Box bx, int* __restrict__ count, int* __restrict__ list, int buff,
                                                      int* err) {
  int js = bx.hi[1] - bx.lo[1] + 1, ks = bx.hi[2] - bx.lo[2] + 1;
  size_t np = (size_t)js * ks;
  size_t id = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= np * M.nf) return;
  int f = (int)(id % M.nf);
  size_t p = id / M.nf;
  if (M.gf[f]) return;
  int j = bx.lo[1] + (int)(p % js), k = bx.lo[2] + (int)(p / js);
  double ymin = gym(g, j) - 0.5 / g.dx2, ymax = gym(g, j) + 0.5 / g.dx2;
  double zmin = gzm(g, k) - 0.5 / g.dx3, zmax = gzm(g, k) + 0.5 / g.dx3;
  const double* V0 = &M.xyzv[3 * M.vof[3 * f + 0]];
  const double* V1 = &M.xyzv[3 * M.vof[3 * f + 1]];
  const double* V2 = &M.xyzv[3 * M.vof[3 * f + 2]];
  if (yz_range(V0, V1, V2, ymin, ymax, zmin, zmax)) {
    int n = atomicAdd(&count[p], 1);
    if (n < buff) list[p * buff + n] = f;
    else raise_error(err, MELT_ERR_PENCIL_OVERFLOW);
  }
}

// rayTriangle_intersect (rayAux.f90:9-83).  A near-parallel ray re-enters with
// an origin shifted by (0, 0.1/dx2, -0.1/dx3); the caller then re-applies its own
// barycentric tests on top of the callee's verdict.  Evaluated here level by
// level from the innermost call outwards.
__device__ bool ray_tri(const Grid& g, const double C0[3], const double Q[3], const double* V0, const double* V1, const double* V2,
                        double ip[3], int* err) {
  const double EPS = 1.e-18;
  const int MAXD = 8;
  double Cs[MAXD + 1][3];
  int L = 0;
  Cs[0][0] = C0[0]; Cs[0][1] = C0[1]; Cs[0][2] = C0[2];
  double e1[3], e2[3];
  for (int d = 0; d < 3; ++d) { e1[d] = V1[d] - V0[d]; e2[d] = V2[d] - V0[d]; }
  // find the first level whose ray is not parallel
  for (;;) {
    double r[3] = {Q[0] - Cs[L][0], Q[1] - Cs[L][1], Q[2] - Cs[L][2]}, p[3];
    dcross(p, r, e2);
    double a = e1[0] * p[0] + e1[1] * p[1] + e1[2] * p[2];
    if (!(a > -EPS && a <= EPS)) break;
    if (L == MAXD) { raise_error(err, MELT_ERR_RAY_RECURSION); return false; }
    Cs[L + 1][0] = Cs[L][0]; Cs[L + 1][1] = Cs[L][1] + 0.1 / g.dx2; Cs[L + 1][2] = Cs[L][2] - 0.1 / g.dx3;
    ++L;
  }
  bool hit = true;
  for (int lev = L; lev >= 0; --lev) {
    const double* C = Cs[lev];
    double r[3], s[3], p[3], q1[3];
    for (int d = 0; d < 3; ++d) { r[d] = Q[d] - C[d]; s[d] = C[d] - V0[d]; }
    dcross(p, r, e2);
    double a = e1[0] * p[0] + e1[1] * p[1] + e1[2] * p[2];
    if (lev == L) hit = true;  // intersect = .true. at entry of the innermost call
    double f = 1.0 / a;
    double u = f * (s[0] * p[0] + s[1] * p[1] + s[2] * p[2]);
    if (u < EPS || u > 1.0) hit = false;
    dcross(q1, s, e1);
    double v = f * (r[0] * q1[0] + r[1] * q1[1] + r[2] * q1[2]);
    if (v < EPS || (u + v) > 1.0) hit = false;
    double t = f * (e2[0] * q1[0] + e2[1] * q1[1] + e2[2] * q1[2]);
    if (t < 0.0 || t > 1.0) hit = false;
    if (hit)
      for (int d = 0; d < 3; ++d) ip[d] = C[d] + t * r[d];
  }
  return hit;
}

__device__ double ray_tag_cell(const Grid& g, const MeshArgs& M, double xlen, const double Q[3], const int* list, int n, int* err) {
  double C[3] = {-xlen * 10.0, Q[1], Q[2]};  // pencil_rayTag.f90:402
  int cnt = 0;
  double xmin = Q[0] - 0.5 / g.dx1, xmax = Q[0] + 0.5 / g.dx1;
  for (int t = 0; t < n; ++t) {
    int f = list[t];
    if (M.gf[f]) continue;
    const double* V0 = &M.xyzv[3 * M.vof[3 * f + 0]];
    const double* V1 = &M.xyzv[3 * M.vof[3 * f + 1]];
    const double* V2 = &M.xyzv[3 * M.vof[3 * f + 2]];
    double mn = fmin(fmin(V0[0], V1[0]), V2[0]), mx = fmax(fmax(V0[0], V1[0]), V2[0]);  // triangleXIntersect
    if (!(mx < xmin || mn > xmax)) {
      if ((V0[0] >= xmin && V0[0] <= xmax) || (V1[0] >= xmin && V1[0] <= xmax) || (V2[0] >= xmin && V2[0] <= xmax)) return 0.5;
    }
    double ip[3] = {0.0, 0.0, 0.0};
    if (ray_tri(g, C, Q, V0, V1, V2, ip, err)) {
      bool inside = ip[0] >= xmin && ip[0] <= xmax && ip[1] >= Q[1] - 0.5 / g.dx2 && ip[1] <= Q[1] + 0.5 / g.dx2 && ip[2] >= Q[2] - 0.5 / g.dx3 &&
                    ip[2] <= Q[2] + 0.5 / g.dx3;
      if (inside) return 0.5;
      cnt += 1;
    }
  }
  return (cnt % 2 == 0) ? 1.0 : 0.0;
}

// pencil_tagCells (pencil_rayTag.f90:189-291): every wrapped cell of the box
// visits its unwrapped preimages in the reference's order (i, then j, then k)
// and keeps the first value below 1.
template <typename R>
__global__ __launch_bounds__(256) void k_pencil_tag(Grid g, MeshArgs M, Box bx, const int* __restrict__ count, const int* __restrict__ list,
                                                    int buff, R* __restrict__ vofp, double xlen, int* err) {
  int ext[3], cov[3];
  int nn[3] = {g.n1, g.n2, g.n3};
  for (int d = 0; d < 3; ++d) { ext[d] = bx.hi[d] - bx.lo[d] + 1; cov[d] = min(ext[d], nn[d]); }
  size_t id = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= (size_t)cov[0] * cov[1] * cov[2]) return;
  int ta = (int)(id % cov[0]), tb = (int)((id / cov[0]) % cov[1]), tc = (int)(id / ((size_t)cov[0] * cov[1]));
  int js = ext[1];
  double cur = 1.0;
  for (int i = bx.lo[0] + ta; i <= bx.hi[0]; i += g.n1)
    for (int j = bx.lo[1] + tb; j <= bx.hi[1]; j += g.n2)
      for (int kk = bx.lo[2] + tc; kk <= bx.hi[2]; kk += g.n3) {
        double Q[3] = {gxm(g, i), gym(g, j), gzm(g, kk)};
        size_t p = (size_t)(j - bx.lo[1]) + (size_t)js * (kk - bx.lo[2]);
        int n = min(count[p], buff);
        double v = ray_tag_cell(g, M, xlen, Q, &list[p * buff], n, err);
        if (!(cur < 1.0)) cur = v;
      }
  vofp[widx(g, bx.lo[0] + ta, bx.lo[1] + tb, bx.lo[2] + tc)] = (R)cur;
}

__global__ __launch_bounds__(256) void k_vbox(const double* __restrict__ xyzv, const unsigned char* __restrict__ gv, int nv, double* out) {
  __shared__ double mn[3][256], mx[3][256];
  double a[3] = {INFINITY, INFINITY, INFINITY}, b[3] = {-INFINITY, -INFINITY, -INFINITY};
  for (int v = threadIdx.x; v < nv; v += blockDim.x) {
    if (gv[v]) continue;
    for (int d = 0; d < 3; ++d) { a[d] = fmin(a[d], xyzv[3 * v + d]); b[d] = fmax(b[d], xyzv[3 * v + d]); }
  }
  for (int d = 0; d < 3; ++d) { mn[d][threadIdx.x] = a[d]; mx[d][threadIdx.x] = b[d]; }
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w)
      for (int d = 0; d < 3; ++d) {
        mn[d][threadIdx.x] = fmin(mn[d][threadIdx.x], mn[d][threadIdx.x + w]);
        mx[d][threadIdx.x] = fmax(mx[d][threadIdx.x], mx[d][threadIdx.x + w]);
      }
    __syncthreads();
  }
  if (threadIdx.x == 0)
    for (int d = 0; d < 3; ++d) { out[d] = mn[d][0]; out[3 + d] = mx[d][0]; }
}

template <typename R>
__global__ __launch_bounds__(256) void k_fill(R* __restrict__ p, double v, size_t n) {
  for (size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x; c < n; c += (size_t)gridDim.x * blockDim.x) p[c] = (R)v;
}

// ------------------------------------------------------------ MLS forcing
__global__ __launch_bounds__(256) void k_centroid_idx(Grid g, const double* __restrict__ bar, const unsigned char* __restrict__ gf, int nf,
                                                      int* __restrict__ pind) {
  int f = blockIdx.x * blockDim.x + threadIdx.x;  // findCentroidIndices.f90:16-48
  if (f >= nf || gf[f]) return;
  const double* p = &bar[3 * f];
  int* o = &pind[6 * f];
  o[0] = (int)floor(p[0] * g.dx1) + 1; o[3] = fnint(p[0] * g.dx1) + 1;
  o[1] = (int)floor(p[1] * g.dx2) + 1; o[4] = fnint(p[1] * g.dx2) + 1;
  int k1 = (int)floor(p[2] * g.dx3) + 1, kst = fnint(p[2] * g.dx3) + 1;
  o[2] = pmod(k1 - 1, g.n3) + 1; o[5] = pmod(kst - 1, g.n3) + 1;
}

struct PhiOut { double* q[4]; };  // ptxAB_q1, ptxAB_q2, ptxAB_temp, ptxAB_q3

// component c: 0 = wght1 (u), 1 = wght2 (v), 2 = wghttemp (T), 3 = wght3 (w).
// With find, the face's cell indices are formed here as k_centroid_idx
// forms them (findCentroidIndices.f90:16-48) and component 0 stores them;
// otherwise they are read from pind.
__device__ __forceinline__ void mls_weights_item(const Grid& g, const double* __restrict__ bar, const unsigned char* __restrict__ gf, int nf,
                                                 int* __restrict__ pind, int find, const PhiOut& out, int id, int* err) {
  if (id >= nf * 4) return;
  int f = id >> 2, comp = id & 3;
  if (gf[f]) return;
  const double* pos = &bar[3 * f];
  int k1 = (int)floor(pos[2] * g.dx3) + 1, kst = fnint(pos[2] * g.dx3) + 1;
  int p[6];
  if (find) {
    p[0] = (int)floor(pos[0] * g.dx1) + 1; p[3] = fnint(pos[0] * g.dx1) + 1;
    p[1] = (int)floor(pos[1] * g.dx2) + 1; p[4] = fnint(pos[1] * g.dx2) + 1;
    p[2] = pmod(k1 - 1, g.n3) + 1; p[5] = pmod(kst - 1, g.n3) + 1;
    if (comp == 0)
      for (int q = 0; q < 6; ++q) pind[6 * f + q] = p[q];
  } else {
    for (int q = 0; q < 6; ++q) p[q] = pind[6 * f + q];
  }
  int i0, j0, k0, c[3];
  if (comp == 0) { i0 = p[3] - 1; j0 = p[1] - 1; k0 = k1 - 1; c[0] = 0; c[1] = 1; c[2] = 1; }
  else if (comp == 1) { i0 = p[0] - 1; j0 = p[4] - 1; k0 = k1 - 1; c[0] = 1; c[1] = 0; c[2] = 1; }
  else if (comp == 2) { i0 = p[0] - 1; j0 = p[1] - 1; k0 = k1 - 1; c[0] = 1; c[1] = 1; c[2] = 1; }
  else { i0 = p[0] - 1; j0 = p[1] - 1; k0 = kst - 1; c[0] = 1; c[1] = 1; c[2] = 0; }
  double* o = &out.q[comp][27 * (size_t)f];
  if (mls_phi(g, pos, i0, j0, k0, c, [&](int q, double v) { o[q] = v; })) raise_error(err, MELT_ERR_SINGULAR_MLS);
}

__global__ __launch_bounds__(64) void k_mls_weights(Grid g, const double* __restrict__ bar, const unsigned char* __restrict__ gf, int nf,
                                                    int* __restrict__ pind, int find, PhiOut out, int* err) {
  mls_weights_item(g, bar, gf, nf, pind, find, out, blockIdx.x * blockDim.x + threadIdx.x, err);
}

constexpr int FORCE_CELLS = 1024;   // table of k_mls_force: 20 KiB of LDS
constexpr int FORCE_FACES = 64;     // faces per block, at most

template <typename R>
struct ForceArgs {
  const R* fld[4];        // vx, vy, temp, vz
  const double* phi[4];
  const double* vel_tri;
  const double* cfac;
  double tmelt;
  const double* bar;
  const unsigned char* gf;
  int nf, fpb;   // fpb: faces per block
  const int* pind;
  const melt_window* win;
  Win3 ef;
  unsigned long long* acc;
  size_t cells;
};

// forc1/forc2/forctemp/forc3 (forc1.f90:28-65): Um = sum q phi, spread
// cfac (V - Um) phi.  32 lanes per face: lane l < 27 loads stencil point l and
// its weight, every lane forms Um from the 27 products in the reference's
// point order (so Um rounds exactly as the serial loop), and lane l adds its
// contribution to the exact 64.64 accumulators.  A block takes fpb faces of one
// component and sums them per cell in LDS first (integer words: the sums do not
// depend on the order).  Bound by updates of the accumulators in memory, whose
// atomics no cache takes: 77 us for 20480 faces on 128^3 with an update per
// face and cell, 38 with a table whose every cell hashes by itself (16 of them the
// flush, each update a transaction of its own), 27 with eight cells of a line
// kept together.
template <int T>
struct ForceShared {
  CellTable<FORCE_CELLS> tab;
  unsigned long long sum[FORCE_CELLS][2];
  alignas(16) double prods[T / 32][28];
  int site[FORCE_FACES][6];       // centre of the stencil: wrapped, 0-based; from the window's origin
  double face[FORCE_FACES][2];    // V, cfac
  bool alive[FORCE_FACES];
};
template <typename R, int T>
__device__ __forceinline__ void mls_force_block(const Grid& g, const ForceArgs<R>& F, ForceShared<T>& sh, int block, int* err) {
  const int t = threadIdx.x, l = t & 31, comp = block & 3, f0 = (int)(block >> 2) * F.fpb;
  if (t < F.fpb) {
    const int f = f0 + t;
    const bool live = f < F.nf && !F.gf[f];
    sh.alive[t] = live;
    if (live) {
      const int* p = &F.pind[6 * f];
      const double z = F.bar[3 * f + 2] * g.dx3;
      const int i0 = p[comp == 0 ? 3 : 0], j0 = p[comp == 1 ? 4 : 1], kw = p[comp == 3 ? 5 : 2];
      const int ku = comp == 3 ? fnint(z) + 1 : (int)floor(z) + 1;
      sh.site[t][0] = pmod(i0 - 1, g.n1); sh.site[t][1] = pmod(j0 - 1, g.n2); sh.site[t][2] = pmod(kw - 1, g.n3);
      sh.site[t][3] = i0 - F.win[0].org[0]; sh.site[t][4] = j0 - F.win[0].org[1]; sh.site[t][5] = ku - F.win[0].org[2];
      sh.face[t][0] = comp == 2 ? F.tmelt : F.vel_tri[3 * f + (comp == 3 ? 2 : comp)];
      sh.face[t][1] = F.cfac[f];
    }
  }
  for (int q = t; q < FORCE_CELLS; q += T) { sh.tab.cell[q] = -1; sh.sum[q][0] = 0ull; sh.sum[q][1] = 0ull; }
  __syncthreads();
  unsigned long long* const out = F.acc + (size_t)comp * F.cells * 2;
  const R* __restrict__ fld = F.fld[comp];
  const double* __restrict__ phi = F.phi[comp];
  const int di = l % 3 - 1, dj = (l / 3) % 3 - 1, dk = l / 9 - 1;
  double* const pr = sh.prods[t >> 5];
  auto wrap = [](int i, int n) { return i < 0 ? i + n : i >= n ? i - n : i; };
  // the loads of the next face are in flight while this one is summed
  auto load = [&](int r, double& ph, R& val) {
    ph = 0.0;
    val = R(0);
    if (r >= F.fpb || l >= 27 || !sh.alive[r]) return;
    const int* st = sh.site[r];
    ph = phi[27 * (size_t)(f0 + r) + l];
    val = fld[wrap(st[0] + di, g.n1) + g.n1 * (wrap(st[1] + dj, g.n2) + g.n2 * wrap(st[2] + dk, g.n3))];
  };
  double ph_next;
  R val_next;
  load(t >> 5, ph_next, val_next);
  for (int r = t >> 5; r < F.fpb; r += T / 32) {
    const double ph = ph_next;
    const R val = val_next;
    load(r + T / 32, ph_next, val_next);
    if (!sh.alive[r]) continue;   // all 32 lanes alike
    if (l < 27) pr[l] = (double)val * ph;
    wave_lds_fence();
    double Um = 0.0;
#pragma unroll
    for (int q = 0; q < 27; ++q) Um = Um + pr[q];
    wave_lds_fence();
    if (l >= 27) continue;
    const double v = sh.face[r][1] * (sh.face[r][0] - Um) * ph;
    const int a = sh.site[r][3] + di, b = sh.site[r][4] + dj, c = sh.site[r][5] + dk;
    if (a < 0 || b < 0 || c < 0 || a >= F.ef.e[0] || b >= F.ef.e[1] || c >= F.ef.e[2]) { raise_error(err, MELT_ERR_WINDOW); continue; }
    const int sl = a + F.ef.e[0] * (b + F.ef.e[1] * c);   // window cells are below 2^30
    const int h = sh.tab.slot(sl);
    acc_add(h >= 0 ? sh.sum[h] : &out[(size_t)sl * 2], v);
  }
  __syncthreads();
  for (int q = threadIdx.x; q < FORCE_CELLS; q += T)
    if (sh.tab.cell[q] >= 0) acc_add_split(&out[(size_t)sh.tab.cell[q] * 2], sh.sum[q][0], sh.sum[q][1]);
}
template <typename R, int T>
__global__ __launch_bounds__(T) void k_mls_force(Grid g, ForceArgs<R> F, int* err) {
  __shared__ ForceShared<T> sh;
  mls_force_block<R, T>(g, F, sh, blockIdx.x, err);
}

// Drain the accumulators: mode 0 adds the forces to the fields (velocity
// without its mean, which the projection subtracts later) and sums the
// velocity forces exactly per block; mode 1 stores them into the for_* fields.
template <typename R>
__global__ __launch_bounds__(256) void k_force_apply(Grid g, const melt_window* __restrict__ win, Win3 ef, unsigned long long* __restrict__ acc,
                                                     size_t cells, R* __restrict__ vx, R* __restrict__ vy, R* __restrict__ t,
                                                     R* __restrict__ vz, int mode, unsigned long long* __restrict__ part) {
  __shared__ unsigned long long slo[3][256], shi[3][256];
  unsigned long long mlo[3] = {0, 0, 0}, mhi[3] = {0, 0, 0};
  R* dst[4] = {vx, vy, t, vz};
  for (size_t s = (size_t)blockIdx.x * blockDim.x + threadIdx.x; s < cells; s += (size_t)gridDim.x * blockDim.x) {
    int a = (int)(s % ef.e[0]), b = (int)((s / ef.e[0]) % ef.e[1]), c = (int)(s / ((size_t)ef.e[0] * ef.e[1]));
    size_t cell = widx(g, win[0].org[0] + a, win[0].org[1] + b, win[0].org[2] + c);
    for (int comp = 0; comp < 4; ++comp) {
      unsigned long long* w = acc + ((size_t)comp * cells + s) * 2;
      unsigned long long lo = w[0], hi = w[1];
      if ((lo | hi) == 0) continue;
      w[0] = 0; w[1] = 0;
      double v = acc_value(lo, hi);
      if (mode == 0) dst[comp][cell] = dst[comp][cell] + v;
      else dst[comp][cell] = v;
      if (comp != 2) {
        int m = comp == 3 ? 2 : comp;
        acc_add_words(mlo[m], mhi[m], lo, hi);
      }
    }
  }
  if (!part) return;
  for (int m = 0; m < 3; ++m) { slo[m][threadIdx.x] = mlo[m]; shi[m][threadIdx.x] = mhi[m]; }
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w)
      for (int m = 0; m < 3; ++m) {
        unsigned long long l1 = slo[m][threadIdx.x], l2 = slo[m][threadIdx.x + w];
        unsigned long long nl = l1 + l2;
        shi[m][threadIdx.x] = shi[m][threadIdx.x] + shi[m][threadIdx.x + w] + (nl < l1 ? 1ull : 0ull);
        slo[m][threadIdx.x] = nl;
      }
    __syncthreads();
  }
  if (threadIdx.x == 0)
    for (int m = 0; m < 3; ++m) { part[(blockIdx.x * 3 + m) * 2] = slo[m][0]; part[(blockIdx.x * 3 + m) * 2 + 1] = shi[m][0]; }
}

// Exact sum of the per-block partial force sums (integer adds: any order
// gives the same words), divided by the cell count.
__global__ __launch_bounds__(256) void k_fmean_final(const unsigned long long* __restrict__ part, int nb, double ncell,
                                                     double* __restrict__ mean) {
  __shared__ unsigned long long slo[3][256], shi[3][256];
  unsigned long long lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0};
  for (int b = threadIdx.x; b < nb; b += blockDim.x)
    for (int m = 0; m < 3; ++m) acc_add_words(lo[m], hi[m], part[(b * 3 + m) * 2], part[(b * 3 + m) * 2 + 1]);
  for (int m = 0; m < 3; ++m) { slo[m][threadIdx.x] = lo[m]; shi[m][threadIdx.x] = hi[m]; }
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w)
      for (int m = 0; m < 3; ++m) {
        unsigned long long l = slo[m][threadIdx.x], h = shi[m][threadIdx.x];
        acc_add_words(l, h, slo[m][threadIdx.x + w], shi[m][threadIdx.x + w]);
        slo[m][threadIdx.x] = l; shi[m][threadIdx.x] = h;
      }
    __syncthreads();
  }
  if (threadIdx.x < 3) mean[threadIdx.x] = acc_value(slo[threadIdx.x][0], shi[threadIdx.x][0]) / ncell;
}

// velforce.f90:21-51 on full fields (per-routine entry point)
template <typename R>
__global__ __launch_bounds__(256) void k_sum3(const R* __restrict__ a, const R* __restrict__ b, const R* __restrict__ c,
                                              size_t n, double* __restrict__ part) {
  __shared__ double s[3][256];
  double x = 0.0, y = 0.0, z = 0.0;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    x = x + a[i]; y = y + b[i]; z = z + c[i];
  }
  s[0][threadIdx.x] = x; s[1][threadIdx.x] = y; s[2][threadIdx.x] = z;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w)
      for (int m = 0; m < 3; ++m) s[m][threadIdx.x] = s[m][threadIdx.x] + s[m][threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0)
    for (int m = 0; m < 3; ++m) part[blockIdx.x * 3 + m] = s[m][0];
}
__global__ void k_sum3_final(const double* __restrict__ part, int nb, double ncell, double* __restrict__ mean) {
  int m = threadIdx.x;
  if (m >= 3) return;
  double s = 0.0;
  for (int b = 0; b < nb; ++b) s = s + part[b * 3 + m];
  mean[m] = s / ncell;
}
template <typename R>
__global__ __launch_bounds__(256) void k_add_force(R* __restrict__ q, const R* __restrict__ f, const double* __restrict__ mean, int m,
                                                   size_t n) {
  size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  q[c] = mean ? q[c] + f[c] - mean[m] : q[c] + f[c];
}

template <typename R>
__global__ __launch_bounds__(256) void k_sub_mean(R* __restrict__ q, const double* __restrict__ mean, int m, size_t n) {
  size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  q[c] = q[c] - mean[m];
}

// ------------------------------------------------------------ probes
// kind 0/1: +/- temperature probe (findProbeIndices.f90 + wght_gradT);
// kind 2: pressure (wght_press); 3..6: grad p, grad u, grad v, grad w.
template <typename R>
struct ProbeArgs {
  const R* temp;
  const R* pr;
  const R* vx;
  const R* vy;
  const R* vz;
  const double* bar;
  const double* nor;
  const unsigned char* gf;
  int nf;
  double h, pec;
  int heat, loads;  // imelt == 1 (kinds 0, 1) / imlsstr == 1 (kinds 2..6)
};

// Probe point of face f on the fluid (kind != 1) or solid (kind 1) side:
// bar +- h n/|n| (mls_heatFlux.f90:33-60, mls_structLoads.f90:40-80).
template <typename R>
__device__ inline void probe_pos(const ProbeArgs<R>& P, int f, int kind, double pos[3]) {
  const double* nor = &P.nor[3 * f];
  const double* bar = &P.bar[3 * f];
  double s = fnorm2(nor, 3);
  double sg = kind == 1 ? -1.0 : 1.0;
  for (int d = 0; d < 3; ++d) pos[d] = sg > 0 ? bar[d] + P.h * nor[d] / s : bar[d] - P.h * nor[d] / s;
}

// Where gradient probe `kind` of face f samples: its position, the stencil
// origin (ic, jc), the z coordinates' grid indices kz and field planes ke
// (findProbeIndices.f90:9-76), the staggering of the field and the field.
template <typename R>
struct ProbeSite {
  double pos[3];
  int ic, jc, kz[3], ke[3], cc[3];
  int icent, jcent, kw;
  const R* fld;
};
template <typename R>
__device__ inline void probe_site(const Grid& g, const ProbeArgs<R>& P, int f, int kind, ProbeSite<R>& S) {
  probe_pos(P, f, kind, S.pos);
  const double* pos = S.pos;
  int icent = (int)floor(pos[0] * g.dx1) + 1, jcent = (int)floor(pos[1] * g.dx2) + 1;
  int istag = fnint(pos[0] * g.dx1) + 1, jstag = fnint(pos[1] * g.dx2) + 1;
  int k1 = (int)floor(pos[2] * g.dx3) + 1, kst = fnint(pos[2] * g.dx3) + 1;
  int kw = pmod(k1 - 1, g.n3) + 1, kws = pmod(kst - 1, g.n3) + 1;
  S.icent = icent; S.jcent = jcent; S.kw = kw;
  S.ic = icent; S.jc = jcent;
  S.cc[0] = S.cc[1] = S.cc[2] = 1;
  S.kz[0] = k1 - 1; S.kz[1] = k1; S.kz[2] = k1;
  S.ke[0] = kw - 1; S.ke[1] = kw; S.ke[2] = kw + 1;
  if (kind <= 1) {
    S.fld = P.temp;
  } else if (kind == 3) {
    S.fld = P.pr;
  } else if (kind == 4) {
    S.fld = P.vx; S.ic = istag; S.cc[0] = 0;
  } else if (kind == 5) {
    S.fld = P.vy; S.jc = jstag; S.cc[1] = 0;
  } else {
    S.fld = P.vz; S.cc[2] = 0;
    S.kz[0] = kst - 1; S.kz[1] = kst; S.kz[2] = kst;
    S.ke[0] = kws - 1; S.ke[1] = kws; S.ke[2] = kws + 1;
  }
}

__device__ __forceinline__ int grad_kind(int q) { return q < 2 ? q : q + 1; }  // 0, 1, 3, 4, 5, 6

// Slots of the stored shape-function derivatives.  The pressure-gradient
// probe (kind 3) samples the same point as the fluid-side temperature probe
// (kind 0, bar + h n) on the same cell-centred stencil, so with both heat flux
// and loads on it shares kind 0's slot: kinds 0, 1, 4, 5, 6.
__device__ __forceinline__ int coef_kind(int cs, int heat, int loads) {
  return heat && loads ? (cs < 2 ? cs : cs + 2) : heat ? cs : cs + 3;
}
__device__ __forceinline__ int coef_slot(int kind, int heat, int loads) {
  return heat && loads ? (kind < 2 ? kind : kind == 3 ? 0 : kind - 2) : heat ? kind : kind - 3;
}

__device__ inline double* probe_out(double* out, int f, int kind, int d) {
  double* o = &out[(size_t)PRB_N * f];
  return &o[(kind == 0 ? PRB_GT0 : kind == 1 ? PRB_GT1 : kind == 3 ? PRB_GP : kind == 4 ? PRB_GU : kind == 5 ? PRB_GV : PRB_GW) + d];
}

// Gradient probes: kinds 0/1 (temperature, fluid/solid side), 3 (pressure),
// 4/5/6 (u, v, w); item = kind slot x nf + face, 4 lanes per item.  With
// COEF (the fused substep) only the geometry part runs: lane 1+d stores the
// 27 shape-function derivatives of component d at coef[q * 3 nitems + 3 item
// + d], and k_force_probes later sums them against the field in the same
// order; without it the lanes sum against the field directly.  Either way
// the values round as in the single-thread formulation.
// With ppw (and COEF) the blocks from gradient block count nblk on store the pressure
// interpolation's 27 shape functions of one face per thread at ppw[q nf + f].
template <typename R>
struct GradArgs {
  ProbeArgs<R> P;
  double* __restrict__ out;
  int* __restrict__ pind;
  int klo, nkinds;
  double* __restrict__ coef;
  double* __restrict__ ppw;
  int nblk;
};
template <bool COEF, typename R>
__device__ __forceinline__ void probes_grad_block(const Grid& g, const GradArgs<R>& Q, GradShared& sh, int block, int* err) {
  const ProbeArgs<R>& P = Q.P;
  double* __restrict__ out = Q.out;
  int* __restrict__ pind = Q.pind;
  double* __restrict__ coef = Q.coef;
  double* __restrict__ ppw = Q.ppw;
  const int klo = Q.klo, nkinds = Q.nkinds, nblk = Q.nblk;
  if (COEF && block >= nblk) {
    const int f = (block - nblk) * 256 + (int)threadIdx.x;
    if (f >= P.nf || P.gf[f]) return;
    int icent, jcent, kw;
    if (pressure_phi(g, P, f, icent, jcent, kw, [&](int q, double phi) { ppw[(size_t)q * P.nf + f] = phi; })) raise_error(err, MELT_ERR_SINGULAR_MLS);
    return;
  }
  const int id = block * 256 + (int)threadIdx.x;
  const int item = id >> 2, lane = id & 3;
  const int nitem = P.nf * nkinds;   // with coef: items over the coefficient slots
  const bool inrange = item < nitem;
  const int f = inrange ? item % P.nf : 0;
  const int q = inrange ? item / P.nf : 0;
  const int kind = COEF ? coef_kind(q, P.heat, P.loads) : grad_kind(klo + q);
  const bool active = inrange && !P.gf[f];
  ProbeSite<R> S;
  S.pos[0] = S.pos[1] = S.pos[2] = 0.0;
  S.ic = S.jc = 1;
  for (int q = 0; q < 3; ++q) { S.kz[q] = 1; S.ke[q] = 1; S.cc[q] = 1; }
  S.fld = P.temp;
  if (active) {
    probe_site(g, P, f, kind, S);
    if (!COEF && kind <= 1 && lane == 0) { int* pi = &pind[6 * f + 3 * kind]; pi[0] = S.icent; pi[1] = S.jcent; pi[2] = S.kw; }
  }
  double gd = 0.0;
  const size_t cs = (size_t)3 * nitem;
  double* cf = COEF && lane > 0 ? coef + (size_t)3 * item + (lane - 1) : nullptr;
  int info = mls_grad_lanes<COEF>(g, sh, S.fld, S.pos, S.ic, S.jc, S.kz, S.ke, S.cc, lane, active, &gd, cf, cs);
  if (!active || lane == 0) return;
  if (info) { raise_error(err, MELT_ERR_SINGULAR_MLS); return; }
  if (!COEF) *probe_out(out, f, kind, lane - 1) = gd;
}
template <bool COEF, typename R>
__global__ __launch_bounds__(256) void k_probes_grad(Grid g, GradArgs<R> Q, int* err) {
  __shared__ GradShared sh;
  probes_grad_block<COEF, R>(g, Q, sh, blockIdx.x, err);
}

// What the coming substep needs of the moved faces, in one launch: the band
// distances of the tagging (as k_tag_band), the forcing's cell indices and
// shape functions (k_mls_weights) and the probes' geometry part
// (k_probes_grad).  On one stream each of the three would leave most of a small
// mesh's chip idle for its own latency: 1280 faces 7 + 10 + 13 us apart, 15 together.
template <int FPB, int CELLS, typename R>
__global__ __launch_bounds__(256) void k_faces_next(Grid g, MeshArgs M, BandArgs B, GradArgs<R> Q, int ngrad, int nwgt, int* __restrict__ pind,
                                                    PhiOut phi, int* err) {
  constexpr size_t bytes = sizeof(GradShared) > sizeof(BandShared<FPB, CELLS>) ? sizeof(GradShared) : sizeof(BandShared<FPB, CELLS>);
  __shared__ __align__(16) unsigned char mem[bytes];
  const int b = blockIdx.x;
  if (b < ngrad) probes_grad_block<true, R>(g, Q, *reinterpret_cast<GradShared*>(mem), b, err);
  else if (b < ngrad + nwgt) mls_weights_item(g, M.bar, M.gf, M.nf, pind, 1, phi, (b - ngrad) * 256 + (int)threadIdx.x, err);
  else tag_band_block<FPB, 256, CELLS>(g, M, B, *reinterpret_cast<BandShared<FPB, CELLS>*>(mem), b - ngrad - nwgt, err);
}

// The field part of the probes of the fused substep: one thread per (item,
// component) sums the stored shape-function derivatives against the field
// values in the reference's point order (and records the heat-flux probes'
// cell indices, as the probes do); with ppw one more thread per face sums the
// stored shape functions of the pressure probe, whose moment matrix and
// inverse (11 us of latency) thereby leave the path to the forcing.
template <typename R>
struct ApplyArgs {
  ProbeArgs<R> P;
  const double* __restrict__ coef;
  const double* __restrict__ ppw;
  double* __restrict__ out;
  int* __restrict__ pind;
  int klo, nkinds, ncoef;
};
template <typename R>
__device__ __forceinline__ void probes_apply_item(const Grid& g, const ApplyArgs<R>& Q, int id) {
  const ProbeArgs<R>& P = Q.P;
  const double* __restrict__ coef = Q.coef;
  const double* __restrict__ ppw = Q.ppw;
  double* __restrict__ out = Q.out;
  int* __restrict__ pind = Q.pind;
  const int klo = Q.klo, nkinds = Q.nkinds, ncoef = Q.ncoef;
  const int nitem = P.nf * nkinds;
  if (id >= 3 * nitem) {
    const int f = id - 3 * nitem;
    if (!ppw || f >= P.nf || P.gf[f]) return;
    double pos[3];
    probe_pos(P, f, 2, pos);
    const int icent = (int)floor(pos[0] * g.dx1) + 1, jcent = (int)floor(pos[1] * g.dx2) + 1;
    const int kw = pmod((int)floor(pos[2] * g.dx3), g.n3) + 1;
    double pp = 0.0;
#pragma unroll
    for (int q = 0; q < 27; ++q)
      pp = pp + P.pr[widx(g, icent - 1 + q % 3, jcent - 1 + (q / 3) % 3, kw - 1 + q / 9)] * ppw[(size_t)q * P.nf + f];
    out[(size_t)PRB_N * f + PRB_P] = pp;
    return;
  }
  const int item = id / 3, d = id - 3 * item;
  const int f = item % P.nf, kind = grad_kind(klo + item / P.nf);
  if (P.gf[f]) return;
  ProbeSite<R> S;
  probe_site(g, P, f, kind, S);
  if (kind <= 1 && d == 0) { int* pi = &pind[6 * f + 3 * kind]; pi[0] = S.icent; pi[1] = S.jcent; pi[2] = S.kw; }
  const size_t cs = (size_t)3 * P.nf * ncoef;
  const double* c = coef + (size_t)3 * ((size_t)coef_slot(kind, P.heat, P.loads) * P.nf + f) + d;
  double s = 0.0;
#pragma unroll 1
  for (int nk = 0; nk < 3; ++nk) {
    const int kk = nk == 0 ? S.ke[0] : nk == 1 ? S.ke[1] : S.ke[2];   // registers, not scratch
#pragma unroll
    for (int jq = 0; jq < 3; ++jq)
#pragma unroll
      for (int iq = 0; iq < 3; ++iq) {
        double acc = c[(size_t)(9 * nk + 3 * jq + iq) * cs];
        double val = S.fld[widx(g, S.ic - 1 + iq, S.jc - 1 + jq, kk)];
        s = s + acc * val;
      }
  }
  *probe_out(out, f, kind, d) = s;
}

// The forcing's spreading and the field part of the probes read the same
// provisional fields and nothing of each other: blocks of one launch.
template <typename R, int T>
__global__ __launch_bounds__(T) void k_force_probes(Grid g, ForceArgs<R> F, ApplyArgs<R> Q, int nforce, int* err) {
  __shared__ ForceShared<T> sh;
  const int b = blockIdx.x;
  if (b < nforce) mls_force_block<R, T>(g, F, sh, b, err);
  else probes_apply_item<R>(g, Q, (b - nforce) * T + (int)threadIdx.x);
}

// Shape functions of the pressure interpolation probe (kind 2, wght_press) of
// face f: sink(q, phi) in the reference's point order.
template <typename R, class Sink>
__device__ __forceinline__ int pressure_phi(const Grid& g, const ProbeArgs<R>& P, int f, int& icent, int& jcent, int& kw, Sink sink) {
  double pos[3];
  probe_pos(P, f, 2, pos);
  icent = (int)floor(pos[0] * g.dx1) + 1; jcent = (int)floor(pos[1] * g.dx2) + 1;
  const int k1 = (int)floor(pos[2] * g.dx3) + 1;
  kw = pmod(k1 - 1, g.n3) + 1;
  const int cc[3] = {1, 1, 1};
  return mls_phi(g, pos, icent - 1, jcent - 1, k1 - 1, cc, sink);
}

// Pressure interpolation probe (kind 2), one thread per face.
template <typename R>
__global__ __launch_bounds__(64) void k_probes_point(Grid g, ProbeArgs<R> P, double* __restrict__ out, int* err) {
  int f = blockIdx.x * blockDim.x + threadIdx.x;
  if (f >= P.nf || P.gf[f]) return;
  double pp = 0.0;
  const R* pr = P.pr;
  int icent, jcent, kw;
  int info = pressure_phi(g, P, f, icent, jcent, kw, [&](int q, double phi) {
    int kk = q / 9, j = jcent - 1 + (q / 3) % 3, i = icent - 1 + q % 3;
    pp = pp + pr[widx(g, i, j, kw - 1 + kk)] * phi;
  });
  if (info) { raise_error(err, MELT_ERR_SINGULAR_MLS); return; }
  out[(size_t)PRB_N * f + PRB_P] = pp;
}

inline unsigned nb(size_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

MeshArgs mesh_args(melt_ctx* ctx) {
  MeshArgs M;
  M.xyzv = ctx->d_lag[MELT_L_XYZV]; M.bar = ctx->d_lag[MELT_L_TRI_BAR]; M.nor = ctx->d_lag[MELT_L_TRI_NOR];
  M.vof = ctx->d_vof; M.gf = ctx->d_gf; M.nf = ctx->nf;
  return M;
}

}  // namespace

// ----------------------------------------------------------------- host
// sphereTagging (tagType 0, sphereTagging.f90:5-549): the level set of
// Kempe & Froehlich (2012) for a rigid sphere of radius rad_p.  A thread owns
// one (i, j, kk) of the bounding box of get_bbox_inds (tagCells.f90:31-62,
// lim from k_vbox, all three axes scaled by dx1 as there), unwrapped in x and
// y; kk is folded into the domain with the centre shifted by zlen
// (get_periodic_indices, tagCells.f90:68-84).  Each of VOFp, VOFx, VOFy, VOFz
// is 1 - alpha over the 8 corners of its control volume (level_setc2, 12, 22,
// 32), alpha = sum (-phi) H(-phi) / sum |phi|, phi the distance to the centre
// minus rad_p (geom.f90:56-80), corners in the reference's i, j, k order.
__device__ inline double sphere_phi(double x, double y, double z, const double c[3], double rad) {
  const double dx = x - c[0], dy = y - c[1], dz = z - c[2];
  return sqrt(dx * dx + dy * dy + dz * dz) - rad;
}

template <int XS, int YS, int ZS>   // per axis: 0 corners at the faces (c, c+1), 1 at the centres (c-1, c)
__device__ inline double sphere_alpha(const Grid& g, int ic, int jc, int kc, const double c[3], double rad) {
  double alpha = 0.0, tot = 0.0;
  for (int a = 0; a < 2; ++a) {
    const int i = XS ? ic - 1 + a : ic + a;
    const double x = XS ? gxm(g, i) : gxc(g, i);
    for (int b = 0; b < 2; ++b) {
      const int j = YS ? jc - 1 + b : jc + b;
      const double y = YS ? gym(g, j) : gyc(g, j);
      for (int d = 0; d < 2; ++d) {
        const int k = ZS ? kc - 1 + d : kc + d;
        const double z = ZS ? gzm(g, k) : gzc(g, k);
        const double phi = sphere_phi(x, y, z, c, rad);
        alpha = alpha + (-phi) * (-phi >= 0.0 ? 1.0 : 0.0);
        tot = tot + fabs(phi);
      }
    }
  }
  return alpha / tot;
}

template <typename R>
__global__ __launch_bounds__(256) void k_sphere_tag(Grid g, const double* __restrict__ lim, const melt_body* __restrict__ body, double rad,
                                                    R* __restrict__ vofp, R* __restrict__ vofx, R* __restrict__ vofy, R* __restrict__ vofz,
                                                    int* err) {
  int lo[3], hi[3];
  for (int d = 0; d < 3; ++d) {
    lo[d] = (int)floor(lim[d] * g.dx1) + 1 - 2;
    hi[d] = (int)floor(lim[3 + d] * g.dx1) + 1 + 2;
  }
  const int ext[3] = {hi[0] - lo[0] + 1, hi[1] - lo[1] + 1, hi[2] - lo[2] + 1};
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t == 0 && (ext[0] > g.n1 || ext[1] > g.n2 || ext[2] > g.n3)) raise_error(err, MELT_ERR_WINDOW);  // a cell would be visited twice
  if (t >= (size_t)g.n1 * g.n2 * g.n3) return;
  const int di = (int)(t % g.n1), dj = (int)((t / g.n1) % g.n2), dk = (int)(t / ((size_t)g.n1 * g.n2));
  if (di >= ext[0] || dj >= ext[1] || dk >= ext[2]) return;
  const int i = lo[0] + di, j = lo[1] + dj;
  int k = lo[2] + dk;
  double c[3] = {body->pos_cm[0], body->pos_cm[1], body->pos_cm[2]};
  if (k >= g.n3 + 1) { k = k - g.n3; c[2] = c[2] - g.zlen; }
  if (k < 1) { k = k + g.n3; c[2] = c[2] + g.zlen; }
  if (k < 1 || k > g.n3) return;
  const size_t o = (size_t)pmod(i - 1, g.n1) + (size_t)g.n1 * ((size_t)pmod(j - 1, g.n2) + (size_t)g.n2 * (k - 1));
  vofp[o] = (R)(1.0 - sphere_alpha<0, 0, 0>(g, i, j, k, c, rad));
  vofx[o] = (R)(1.0 - sphere_alpha<1, 0, 0>(g, i, j, k, c, rad));
  vofy[o] = (R)(1.0 - sphere_alpha<0, 1, 0>(g, i, j, k, c, rad));
  vofz[o] = (R)(1.0 - sphere_alpha<0, 0, 1>(g, i, j, k, c, rad));
}

template <typename R>
static int sphere_tag_t(melt_ctx* ctx) {
  const Grid g = make_grid(ctx);
  Win3 ef{{ctx->fwin[0], ctx->fwin[1], ctx->fwin[2]}}, et{{ctx->twin[0], ctx->twin[1], ctx->twin[2]}};
  hipLaunchKernelGGL(k_window_box, dim3(nb(ctx->nf, 256)), dim3(256), 0, ctx->stream, g, ctx->d_lag[MELT_L_TRI_BAR], ctx->d_gf, ctx->nf,
                     ctx->d_win);
  hipLaunchKernelGGL(k_window_final, dim3(1), dim3(1), 0, ctx->stream, ctx->d_win, ef, et, ctx->force_window_from_tag ? 3 : 2,
                     ctx->d_err);
  hipLaunchKernelGGL(k_vbox, dim3(1), dim3(256), 0, ctx->stream, ctx->d_lag[MELT_L_XYZV], ctx->d_gv, ctx->nv, ctx->d_sbox);
  for (int id = MELT_VOFP; id <= MELT_VOFZ; ++id)
    hipLaunchKernelGGL(k_fill<R>, dim3(1024), dim3(256), 0, ctx->stream, fld<R>(ctx, id), 1.0, ctx->nc);
  hipLaunchKernelGGL(k_sphere_tag<R>, dim3(nb(ctx->nc, 256)), dim3(256), 0, ctx->stream, g, ctx->d_sbox, ctx->d_body, ctx->rad_p,
                     fld<R>(ctx, MELT_VOFP), fld<R>(ctx, MELT_VOFX), fld<R>(ctx, MELT_VOFY), fld<R>(ctx, MELT_VOFZ), ctx->d_err);
  MELT_HIP(hipGetLastError());
  if (ctx->h_body.initial_tag) {   // no ray tagging in this mode: the flag only gates graph capture
    ctx->h_body.initial_tag = 0;
    MELT_HIP(hipMemcpyAsync(&ctx->d_body->initial_tag, &ctx->h_body.initial_tag, sizeof(int), hipMemcpyHostToDevice, ctx->stream));
    MELT_HIP(hipStreamSynchronize(ctx->stream));
  }
  return 0;
}

template <typename R>
static int ray_tag_init_t(melt_ctx* ctx) {
  Grid g = make_grid(ctx);
  hipLaunchKernelGGL(k_vbox, dim3(1), dim3(256), 0, ctx->stream, ctx->d_lag[MELT_L_XYZV], ctx->d_gv, ctx->nv, ctx->d_sbox);
  MELT_HIP(hipGetLastError());
  double lim[6];
  MELT_HIP(hipMemcpyAsync(lim, ctx->d_sbox, sizeof lim, hipMemcpyDeviceToHost, ctx->stream));
  MELT_HIP(hipStreamSynchronize(ctx->stream));
  Box bx;  // get_bbox_inds tagCells.f90:31-62 (the reference scales all three axes by dx1)
  for (int d = 0; d < 3; ++d) {
    bx.lo[d] = (int)floor(lim[d] * ctx->dx1) + 1 - 2;
    bx.hi[d] = (int)floor(lim[3 + d] * ctx->dx1) + 1 + 2;
  }
  for (int id = MELT_VOFP; id <= MELT_VOFZ; ++id)
    hipLaunchKernelGGL(k_fill<R>, dim3(1024), dim3(256), 0, ctx->stream, fld<R>(ctx, id), 1.0, ctx->nc);
  MELT_HIP(hipGetLastError());
  int js = bx.hi[1] - bx.lo[1] + 1, ks = bx.hi[2] - bx.lo[2] + 1;
  // BUFF_SIZE: n1m as the reference sets it (pencil_rayTag.f90:84) unless the
  // caller sized it (tuning key pbuf); tags do not depend on it below overflow
  int buff = ctx->tune[TUNE_PBUF] > 0 ? ctx->tune[TUNE_PBUF] : ctx->n1;
  size_t np = (size_t)js * ks;
  if (np * buff > ctx->plist_cap) {
    if (ctx->d_plist) hipFree(ctx->d_plist);
    if (ctx->d_pcount) hipFree(ctx->d_pcount);
    MELT_HIP(hipMalloc(&ctx->d_plist, sizeof(int) * np * buff));
    MELT_HIP(hipMalloc(&ctx->d_pcount, sizeof(int) * np));
    ctx->plist_cap = np * buff;
  }
  MELT_HIP(hipMemsetAsync(ctx->d_pcount, 0, sizeof(int) * np, ctx->stream));
  MeshArgs M = mesh_args(ctx);
  hipLaunchKernelGGL(k_pencil_build, dim3(nb(np * ctx->nf, 256)), dim3(256), 0, ctx->stream, g, M, bx, ctx->d_pcount, ctx->d_plist, buff,
                     ctx->d_err);
  MELT_HIP(hipGetLastError());
  size_t cov = 1;
  int nn[3] = {ctx->n1, ctx->n2, ctx->n3};
  for (int d = 0; d < 3; ++d) cov *= (size_t)std::min(bx.hi[d] - bx.lo[d] + 1, nn[d]);
  hipLaunchKernelGGL(k_pencil_tag<R>, dim3(nb(cov, 256)), dim3(256), 0, ctx->stream, g, M, bx, ctx->d_pcount, ctx->d_plist, buff,
                     fld<R>(ctx, MELT_VOFP), ctx->cfg.xlen, ctx->d_err);
  MELT_HIP(hipGetLastError());
  return 0;
}

template <typename R>
static ProbeArgs<R> probe_args(melt_ctx* ctx) {
  ProbeArgs<R> P;
  P.temp = fld<R>(ctx, MELT_TEMP); P.pr = fld<R>(ctx, MELT_PR); P.vx = fld<R>(ctx, MELT_VX); P.vy = fld<R>(ctx, MELT_VY); P.vz = fld<R>(ctx, MELT_VZ);
  P.bar = ctx->d_lag[MELT_L_TRI_BAR]; P.nor = ctx->d_lag[MELT_L_TRI_NOR]; P.gf = ctx->d_gf; P.nf = ctx->nf;
  P.h = ctx->h_body.h_eulerian; P.pec = ctx->cfg.ren * ctx->cfg.prandtl;
  P.heat = ctx->cfg.imelt == 1;
  P.loads = ctx->cfg.imlsstr == 1;
  return P;
}

template <typename R>
static int probe_coef_slots(const ProbeArgs<R>& P) { return P.heat && P.loads ? 5 : P.heat ? 2 : P.loads ? 4 : 0; }

// Where the pressure probe's shape functions sit in d_pcoef (27 x 18 doubles per
// face): behind the gradient slots (27 x 15 at most).
template <typename R>
static double* probe_ppw(melt_ctx* ctx, const ProbeArgs<R>& P) {
  return P.loads ? ctx->d_pcoef + (size_t)27 * 3 * probe_coef_slots(P) * ctx->nf : nullptr;
}

// The geometry part of the probes: its arguments, and its blocks (0: no probes).
template <typename R>
static GradArgs<R> coef_args(melt_ctx* ctx, int* blocks) {
  const ProbeArgs<R> P = probe_args<R>(ctx);
  const int klo = P.heat ? 0 : 2, khi = P.loads ? 6 : 2, ncoef = probe_coef_slots(P);
  const int ngrad = (int)nb((size_t)ctx->nf * ncoef * 4, 256), npr = P.loads ? (int)nb(ctx->nf, 256) : 0;
  *blocks = khi > klo ? ngrad + npr : 0;
  return {P, ctx->d_probe, ctx->d_pind, klo, ncoef, ctx->d_pcoef, probe_ppw(ctx, P), ngrad};
}

// The field part of the probes of the fused substep: its arguments and its threads.
template <typename R>
static ApplyArgs<R> apply_args(melt_ctx* ctx, int* pind) {
  const ProbeArgs<R> P = probe_args<R>(ctx);
  const int klo = P.heat ? 0 : 2, khi = P.loads ? 6 : 2;
  return {P, ctx->d_pcoef, probe_ppw(ctx, P), ctx->d_probe, pind, klo, std::max(0, khi - klo), probe_coef_slots(P)};
}
template <typename R>
static size_t apply_items(const ApplyArgs<R>& Q) {
  return Q.nkinds ? (size_t)Q.P.nf * Q.nkinds * 3 + (Q.P.loads ? Q.P.nf : 0) : 0;
}

static PhiOut phi_out(melt_ctx* ctx) {
  return {{ctx->d_lag[MELT_L_PTXAB_Q1], ctx->d_lag[MELT_L_PTXAB_Q2], ctx->d_lag[MELT_L_PTXAB_TEMP], ctx->d_lag[MELT_L_PTXAB_Q3]}};
}

template <typename R>
static int ibm_tag_t(melt_ctx* ctx, bool wgt, bool coef) {  // tagCells.f90:4-27 (tagType 1) + interp_vof when not fused
  if (!ctx->has_geom) return melt_fail(ctx, MELT_ERR_NO_GEOMETRY, "tagCells", "no geometry");
  if (ctx->cfg.tagtype == 0) return sphere_tag_t<R>(ctx);
  Grid g = make_grid(ctx);
  if (ctx->h_body.initial_tag) {
    int rc = ray_tag_init_t<R>(ctx);
    if (rc) return rc;
    ctx->h_body.initial_tag = 0;
    MELT_HIP(hipMemcpyAsync(&ctx->d_body->initial_tag, &ctx->h_body.initial_tag, sizeof(int), hipMemcpyHostToDevice, ctx->stream));
  }
  Win3 ef{{ctx->fwin[0], ctx->fwin[1], ctx->fwin[2]}}, et{{ctx->twin[0], ctx->twin[1], ctx->twin[2]}};
  // face extent, reset of the previous window, cleared keys: one launch
  const int nbox = (int)nb(ctx->nf, 256);
  hipLaunchKernelGGL(k_tag_prepare<R>, dim3(nbox + 256), dim3(256), 0, ctx->stream, g, ctx->d_lag[MELT_L_TRI_BAR], ctx->d_gf, ctx->nf, nbox,
                     ctx->d_win, fld<R>(ctx, MELT_SDF), et, ctx->d_tkey, ctx->d_tface, ctx->twin_cells);
  // the fused substep places the forcing window from the same extent (the
  // faces do not move between tagging and forcing)
  const int which = ctx->force_window_from_tag ? 3 : 2;
  MeshArgs M = mesh_args(ctx);
  const BandArgs B{ctx->d_win, et, ctx->d_tkey, ctx->d_tdist};
  int ngrad = 0;
  const GradArgs<R> Q = coef_args<R>(ctx, &ngrad);
  const int nwgt = (int)nb((size_t)ctx->nf * 4, 256);
  if (!coef) ngrad = 0;
#define TAG_PASSES(FPB, T, CELLS)                                                                                                       \
  do {                                                                                                                                  \
    const unsigned groups = nb(ctx->nf, FPB);                                                                                           \
    if (wgt)                                                                                                                            \
      hipLaunchKernelGGL((k_faces_next<FPB, CELLS, R>), dim3(ngrad + nwgt + groups), dim3(256), 0, ctx->stream, g, M, B, Q, ngrad, nwgt, \
                         ctx->d_pind, phi_out(ctx), ctx->d_err);                                                                        \
    else                                                                                                                                \
      hipLaunchKernelGGL((k_tag_band<FPB, T, CELLS>), dim3(groups), dim3(T), 0, ctx->stream, g, M, B, ctx->d_err);                       \
    hipLaunchKernelGGL((k_tag_pass<1, FPB, R>), dim3(groups), dim3(256), 0, ctx->stream, g, M, ctx->d_win, ef, et, which, ctx->d_tkey,   \
                       ctx->d_tface, ctx->d_tdist, fld<R>(ctx, MELT_SDF), fld<R>(ctx, MELT_VOFP), ctx->pi, ctx->d_err);                  \
    hipLaunchKernelGGL((k_tag_pass<2, FPB, R>), dim3(groups), dim3(256), 0, ctx->stream, g, M, ctx->d_win, ef, et, which, ctx->d_tkey,   \
                       ctx->d_tface, ctx->d_tdist, fld<R>(ctx, MELT_SDF), fld<R>(ctx, MELT_VOFP), ctx->pi, ctx->d_err);                  \
  } while (0)
  // As many faces a group as keep the chip's blocks busy (20480 faces on 128^3:
  // 16 a group 42 us for the three passes, 8 50; 5120 faces: 8 22, 16 27; 1280: 4
  // 16, 8 17), with twice the cells a group of neighbours touches in its table
  // (16 faces with 1024 cells often leave their distances: 62).  Beside the lines: a
  // tagCells call of 9680 faces 46 us with 16 or 8, 11520 48 and 51, 14580 53 and 57; a
  // step at 128^3 with 8000 faces 1.08 ms with 16, 1.05 with 8; with 2420 and 2880 4 and 8
  // are level.
  if (ctx->nf > 8192) TAG_PASSES(16, 512, 2048);
  else if (ctx->nf > 2560) TAG_PASSES(8, 512, 1024);
  else TAG_PASSES(4, 512, 512);
#undef TAG_PASSES
  MELT_HIP(hipGetLastError());
  return 0;
}

int ibm_find_centroid_indices(melt_ctx* ctx) {
  hipLaunchKernelGGL(k_centroid_idx, dim3(nb(ctx->nf, 256)), dim3(256), 0, ctx->stream, make_grid(ctx), ctx->d_lag[MELT_L_TRI_BAR], ctx->d_gf,
                     ctx->nf, ctx->d_pind);
  MELT_HIP(hipGetLastError());
  return 0;
}

int ibm_weights(melt_ctx* ctx, bool find) {
  const PhiOut o = phi_out(ctx);
  hipLaunchKernelGGL(k_mls_weights, dim3(nb((size_t)ctx->nf * 4, 64)), dim3(64), 0, ctx->stream, make_grid(ctx), ctx->d_lag[MELT_L_TRI_BAR],
                     ctx->d_gf, ctx->nf, ctx->d_pind, find ? 1 : 0, o, ctx->d_err);
  MELT_HIP(hipGetLastError());
  return 0;
}

// Interpolation + spreading into the exact accumulators (mlsForce.f90, forc*);
// with_probes (the fused substep, their coefficients ready): also the field part of
// the gradient and pressure probes, their cell indices into pind2.
template <typename R>
static int ibm_force_scatter_t(melt_ctx* ctx, bool with_probes) {
  Grid g = make_grid(ctx);
  Win3 ef{{ctx->fwin[0], ctx->fwin[1], ctx->fwin[2]}}, et{{ctx->twin[0], ctx->twin[1], ctx->twin[2]}};
  if (!ctx->force_window_from_tag) {
    hipLaunchKernelGGL(k_window_box, dim3(nb(ctx->nf, 256)), dim3(256), 0, ctx->stream, g, ctx->d_lag[MELT_L_TRI_BAR], ctx->d_gf, ctx->nf,
                       ctx->d_win);
    hipLaunchKernelGGL(k_window_final, dim3(1), dim3(1), 0, ctx->stream, ctx->d_win, ef, et, 1, ctx->d_err);
  }
  ForceArgs<R> F;
  F.fld[0] = fld<R>(ctx, MELT_VX); F.fld[1] = fld<R>(ctx, MELT_VY); F.fld[2] = fld<R>(ctx, MELT_TEMP); F.fld[3] = fld<R>(ctx, MELT_VZ);
  const PhiOut phi = phi_out(ctx);
  for (int q = 0; q < 4; ++q) F.phi[q] = phi.q[q];
  F.vel_tri = ctx->d_lag[MELT_L_VEL_TRI]; F.cfac = ctx->d_lag[MELT_L_CFAC]; F.tmelt = ctx->cfg.tmelt;
  F.bar = ctx->d_lag[MELT_L_TRI_BAR]; F.gf = ctx->d_gf; F.nf = ctx->nf; F.pind = ctx->d_pind;
  F.win = ctx->d_win; F.ef = ef; F.acc = ctx->d_acc; F.cells = ctx->fwin_cells;
  const ApplyArgs<R> Q = apply_args<R>(ctx, ctx->d_pind2);
  const size_t items = with_probes ? apply_items(Q) : 0;
#define MLS_FORCE(T, FPB)                                                                                                              \
  do {                                                                                                                                 \
    F.fpb = FPB;                                                                                                                       \
    const unsigned nforce = 4 * nb(ctx->nf, FPB);                                                                                      \
    if (items)                                                                                                                         \
      hipLaunchKernelGGL((k_force_probes<R, T>), dim3(nforce + nb(items, T)), dim3(T), 0, ctx->stream, g, F, Q, (int)nforce, ctx->d_err); \
    else                                                                                                                               \
      hipLaunchKernelGGL((k_mls_force<R, T>), dim3(nforce), dim3(T), 0, ctx->stream, g, F, ctx->d_err);                                 \
  } while (0)
  // Many faces: as many per block as share their cells best (20480 faces: 64
  // per block 27 us, 32 46, one update per face and cell 77).  Fewer faces: more
  // blocks (5120 faces with the probes: 32 by 256 threads 15 us, 16 24, 32 by 512, of
  // which a CU holds two, 24), and more faces at a time (1280 faces alone: 16 by
  // 512 threads 6.7 us, 8 by 256 8.1, 64 15.6).  Beside the lines, a step: 96^3 with
  // 2420 faces 0.71 ms with 16 by 512, 0.69 with 32 by 256, with 2880 0.70 and 0.69; 128^3 in
  // FP32 with 8000 0.76 with 64 or 32, with 8820 0.81 with 64, 0.82 with 32.
  if (ctx->nf > 8192) MLS_FORCE(256, 64);
  else if (ctx->nf > 2560) MLS_FORCE(256, 32);
  else MLS_FORCE(512, 16);
#undef MLS_FORCE
  MELT_HIP(hipGetLastError());
  return 0;
}

static unsigned drain_blocks(const melt_ctx* ctx) { return (unsigned)std::min<size_t>(512, nb(ctx->fwin_cells, 256)); }

// The exact mean of the velocity forces into d_fmean, for the projection
// (velforce.f90:21-51 with the uniform shift deferred), from the block sums of
// ibm_force_drain (d_red[64..3136), which the Lagrangian update's sums leave alone).
int ibm_force_mean(melt_ctx* ctx) {
  hipLaunchKernelGGL(k_fmean_final, dim3(1), dim3(256), 0, ctx->stream, reinterpret_cast<unsigned long long*>(ctx->d_red + 64),
                     (int)drain_blocks(ctx), (double)((long long)ctx->n1 * ctx->n2 * ctx->n3), ctx->d_fmean);
  MELT_HIP(hipGetLastError());
  return 0;
}

// Drain the accumulators.  apply_now = 1 (fused substep): forces go straight
// into u, v, w, T, and the block sums of the velocity forces are left for
// ibm_force_mean; 0: the folded for_* fields are written (per-routine API, mlsForce output).
template <typename R>
static int ibm_force_drain_t(melt_ctx* ctx, int apply_now) {
  Grid g = make_grid(ctx);
  Win3 ef{{ctx->fwin[0], ctx->fwin[1], ctx->fwin[2]}};
  const unsigned blocks = drain_blocks(ctx);
  unsigned long long* part = reinterpret_cast<unsigned long long*>(ctx->d_red + 64);
  if (apply_now) {
    hipLaunchKernelGGL(k_force_apply<R>, dim3(blocks), dim3(256), 0, ctx->stream, g, ctx->d_win, ef, ctx->d_acc, ctx->fwin_cells, fld<R>(ctx, MELT_VX),
                       fld<R>(ctx, MELT_VY), fld<R>(ctx, MELT_TEMP), fld<R>(ctx, MELT_VZ), 0, part);
  } else {
    for (int id = MELT_FOR_XC; id <= MELT_FOR_TEMP; ++id)
      hipLaunchKernelGGL(k_fill<R>, dim3(1024), dim3(256), 0, ctx->stream, fld<R>(ctx, id), 0.0, ctx->nc);
    hipLaunchKernelGGL(k_force_apply<R>, dim3(blocks), dim3(256), 0, ctx->stream, g, ctx->d_win, ef, ctx->d_acc, ctx->fwin_cells,
                       fld<R>(ctx, MELT_FOR_XC), fld<R>(ctx, MELT_FOR_YC), fld<R>(ctx, MELT_FOR_TEMP), fld<R>(ctx, MELT_FOR_ZC), 1, nullptr);
  }
  MELT_HIP(hipGetLastError());
  return 0;
}

// u -= fbar over the whole field (the shift the fused substep defers to the
// projection), for callers that stop after particle.
template <typename R>
static int ibm_sub_mean_t(melt_ctx* ctx) {
  const int q[3] = {MELT_VX, MELT_VY, MELT_VZ};
  for (int m = 0; m < 3; ++m)
    hipLaunchKernelGGL(k_sub_mean<R>, dim3(nb(ctx->nc, 256)), dim3(256), 0, ctx->stream, fld<R>(ctx, q[m]), ctx->d_fmean, m, ctx->nc);
  MELT_HIP(hipGetLastError());
  return 0;
}

template <typename R>
static int ibm_velforce_t(melt_ctx* ctx, int /*defer*/) {  // velforce.f90 on full for_* fields
  unsigned blocks = (unsigned)std::min<size_t>(1024, nb(ctx->nc, 256));
  double* part = ctx->d_red + 64;
  hipLaunchKernelGGL(k_sum3<R>, dim3(blocks), dim3(256), 0, ctx->stream, fld<R>(ctx, MELT_FOR_XC), fld<R>(ctx, MELT_FOR_YC), fld<R>(ctx, MELT_FOR_ZC), ctx->nc,
                     part);
  hipLaunchKernelGGL(k_sum3_final, dim3(1), dim3(64), 0, ctx->stream, part, (int)blocks, (double)((long long)ctx->n1 * ctx->n2 * ctx->n3),
                     ctx->d_fmean);
  const int q[3] = {MELT_VX, MELT_VY, MELT_VZ}, fo[3] = {MELT_FOR_XC, MELT_FOR_YC, MELT_FOR_ZC};
  for (int m = 0; m < 3; ++m)
    hipLaunchKernelGGL(k_add_force<R>, dim3(nb(ctx->nc, 256)), dim3(256), 0, ctx->stream, fld<R>(ctx, q[m]), fld<R>(ctx, fo[m]), ctx->d_fmean, m, ctx->nc);
  MELT_HIP(hipGetLastError());
  return 0;
}

template <typename R>
static int ibm_tempforce_t(melt_ctx* ctx) {  // tempforce.f90
  hipLaunchKernelGGL(k_add_force<R>, dim3(nb(ctx->nc, 256)), dim3(256), 0, ctx->stream, fld<R>(ctx, MELT_TEMP), fld<R>(ctx, MELT_FOR_TEMP), nullptr, 0,
                     ctx->nc);
  MELT_HIP(hipGetLastError());
  return 0;
}

// The geometry part of the probes (shape-function derivatives and the pressure
// probe's shape functions into d_pcoef): reads only the faces and the grid, so
// the fused substep runs it beside the explicit pass.
template <typename R>
static int ibm_probe_coefs_t(melt_ctx* ctx) {
  int blocks = 0;
  const GradArgs<R> Q = coef_args<R>(ctx, &blocks);
  if (blocks) hipLaunchKernelGGL((k_probes_grad<true, R>), dim3(blocks), dim3(256), 0, ctx->stream, make_grid(ctx), Q, ctx->d_err);
  MELT_HIP(hipGetLastError());
  return 0;
}

// The probes outside the fused substep: geometry and field part at once.
template <typename R>
static int ibm_probes_t(melt_ctx* ctx) {
  ProbeArgs<R> P = probe_args<R>(ctx);
  int klo = P.heat ? 0 : 2, khi = P.loads ? 6 : 2;
  if (khi > klo) {
    const int ngrad = (int)nb((size_t)ctx->nf * (khi - klo) * 4, 256);
    const GradArgs<R> Q{P, ctx->d_probe, ctx->d_pind, klo, khi - klo, nullptr, nullptr, ngrad};
    hipLaunchKernelGGL((k_probes_grad<false, R>), dim3(ngrad), dim3(256), 0, ctx->stream, make_grid(ctx), Q, ctx->d_err);
    if (P.loads)
      hipLaunchKernelGGL(k_probes_point<R>, dim3(nb(ctx->nf, 64)), dim3(64), 0, ctx->stream, make_grid(ctx), P, ctx->d_probe, ctx->d_err);
  }
  MELT_HIP(hipGetLastError());
  return 0;
}

int ibm_window_reset(melt_ctx* ctx) {
  hipLaunchKernelGGL(k_window_reset, dim3(1), dim3(1), 0, ctx->stream, ctx->d_win, 2);
  MELT_HIP(hipGetLastError());
  return 0;
}

// ------------------------------------------------- precision dispatch
int ibm_tag(melt_ctx* ctx, bool wgt, bool coef) { return ctx->fp32 ? ibm_tag_t<float>(ctx, wgt, coef) : ibm_tag_t<double>(ctx, wgt, coef); }
int ibm_force_scatter(melt_ctx* ctx, bool with_probes) {
  return ctx->fp32 ? ibm_force_scatter_t<float>(ctx, with_probes) : ibm_force_scatter_t<double>(ctx, with_probes);
}
int ibm_force_drain(melt_ctx* ctx, int apply_now) { return ctx->fp32 ? ibm_force_drain_t<float>(ctx, apply_now) : ibm_force_drain_t<double>(ctx, apply_now); }
int ibm_sub_mean(melt_ctx* ctx) { return ctx->fp32 ? ibm_sub_mean_t<float>(ctx) : ibm_sub_mean_t<double>(ctx); }
int ibm_velforce(melt_ctx* ctx, int defer) { return ctx->fp32 ? ibm_velforce_t<float>(ctx, defer) : ibm_velforce_t<double>(ctx, defer); }
int ibm_tempforce(melt_ctx* ctx) { return ctx->fp32 ? ibm_tempforce_t<float>(ctx) : ibm_tempforce_t<double>(ctx); }
int ibm_probes(melt_ctx* ctx) { return ctx->fp32 ? ibm_probes_t<float>(ctx) : ibm_probes_t<double>(ctx); }
int ibm_probe_coefs(melt_ctx* ctx) { return ctx->fp32 ? ibm_probe_coefs_t<float>(ctx) : ibm_probe_coefs_t<double>(ctx); }
