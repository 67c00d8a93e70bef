// Diagnostics the reference's time loop calls around tschem (gcurv.f90:151-201):
// the time-step choice get_dt (cfl.f90:33-77) and the turbulence statistics
// of CalcDissipation (diss.f90:11-201).  Both read the fields once: get_dt is
// a max reduction (exact in any order), CalcDissipation a sum over the fluid
// cells taken in a fixed order (the planes of each thread's column, a fixed
// tree per block, a fixed tree over the block partials), so every run on a
// given grid gives the same bits.
#include <algorithm>
#include <cmath>

#include "common.h"

namespace {

constexpr int DISS_THREADS = 256;
constexpr int DISS_BLOCKS = 512;   // at most, 4 partials each in ctx->d_red (16384 doubles)

// Two neighbouring cells of a line, and with the cells left and right of them.
struct Pair { double a, b; };
struct Quad { double l, a, b, r; };
template <typename R>
__device__ inline Pair ld_pair(const R* __restrict__ p) {
  struct alignas(2 * sizeof(R)) Vec { R a, b; };
  const Vec v = *reinterpret_cast<const Vec*>(p);
  return {(double)v.a, (double)v.b};
}

// Per-cell terms of diss.f90:56-141, summed over cells with VOFp == 1
// (diss.f90:144-153): [0] tke, [1] diss, [2] chi, [3] the number of such cells.
// A thread takes two neighbouring columns (n1 is even, so their loads are
// aligned) of a tile of DISS_THREADS pairs and marches `dz` planes up them:
// what a plane shares with the next one stays in registers, the x neighbours
// come from the neighbouring lanes (a lane at the end of its wave or line
// loads them), and the indices need no division per cell.  The stencil's 36
// loads a cell kept the L1 busy, not the memory: one column per thread with
// every neighbour loaded (23 loads a cell) still took 109 M L1 accesses, 177 us
// of its 262 at 256^3 FP64 (440 with all 36); six aligned loads a cell take 172
// us, the five fields at the rate of a copy 141.  A block takes the (tile,
// segment) pairs its index and the grid's stride give, and an XCD
// neighbouring tiles, whose lines they share in its L2.
template <typename R>
__global__ __launch_bounds__(DISS_THREADS, 2) void k_diss_partial(Grid g, const R* __restrict__ vx, const R* __restrict__ vy,
                                                                  const R* __restrict__ vz, const R* __restrict__ te,
                                                                  const R* __restrict__ vof, double ren, double pec, int tiles, int dz,
                                                                  int items, double* __restrict__ part) {
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  const double udx1 = g.dx1, udx2 = g.dx2, udx3 = g.dx3;
  const int n1 = g.n1, plane = n1 * g.n2, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (int it = (int)xcd_block(blockIdx.x, gridDim.x); it < items; it += (int)gridDim.x) {
    const int seg = it / tiles, c0 = 2 * ((it - seg * tiles) * DISS_THREADS + (int)threadIdx.x);
    if (c0 >= plane) continue;
    const int j = c0 / n1, i = c0 - j * n1;
    const int djp = j + 1 == g.n2 ? n1 - plane : n1, djm = j == 0 ? plane - n1 : -n1;
    const int dl = i == 0 ? n1 - 1 : -1, dr = i + 2 == n1 ? 2 - n1 : 2;
    const bool el = lane == 0 || i == 0, er = lane == 63 || i + 2 == n1;
    auto left = [&](const Pair& p) { return __shfl_up(p.b, 1, 64); };
    auto right = [&](const Pair& p) { return __shfl_down(p.a, 1, 64); };
    auto pair = [&](const R* f, int o) { return ld_pair<R>(f + o); };
    auto quad = [&](const R* f, int o) {
      const Pair p = ld_pair<R>(f + o);
      Quad q{left(p), p.a, p.b, right(p)};
      if (el) q.l = (double)f[o + dl];
      if (er) q.r = (double)f[o + dr];
      return q;
    };
    const int k0 = seg * dz, k1 = min(k0 + dz, g.n3);
    int c = k0 * plane + c0;
    const int cm = k0 == 0 ? (g.n3 - 1) * plane + c0 : c - plane;
    // plane k (and k - 1): the values that a later plane reads again
    Quad x = quad(vx, c), xd = quad(vx, cm), y = quad(vy, c), yj = quad(vy, c + djp), z = quad(vz, c), t = quad(te, c);
    Pair yd = pair(vy, cm), yjd = pair(vy, cm + djp), zj = pair(vz, c + djp), zm = pair(vz, c + djm), td = pair(te, cm);
    for (int k = k0; k < k1; ++k) {
      const int u = k + 1 == g.n3 ? c0 : c + plane;
      const Pair xup = pair(vx, u), xjp = pair(vx, c + djp), xmp = pair(vx, c + djm), yup = pair(vy, u), yujp = pair(vy, u + djp);
      const Pair zup = pair(vz, u), zuj = pair(vz, u + djp), zum = pair(vz, u + djm), tup = pair(te, u);
      const Pair tj = pair(te, c + djp), tm = pair(te, c + djm), f = pair(vof, c);
      Quad xu{0.0, xup.a, xup.b, right(xup)}, xj{0.0, xjp.a, xjp.b, right(xjp)}, xm{0.0, xmp.a, xmp.b, right(xmp)};
      Quad yu{left(yup), yup.a, yup.b, right(yup)}, yuj{left(yujp), yujp.a, yujp.b, right(yujp)};
      Quad zu{left(zup), zup.a, zup.b, right(zup)}, tu{left(tup), tup.a, tup.b, right(tup)};
      if (el) {
        yu.l = (double)vy[u + dl]; yuj.l = (double)vy[u + djp + dl];
        zu.l = (double)vz[u + dl]; tu.l = (double)te[u + dl];
      }
      if (er) {
        xu.r = (double)vx[u + dr]; xj.r = (double)vx[c + djp + dr]; xm.r = (double)vx[c + djm + dr];
        yu.r = (double)vy[u + dr]; yuj.r = (double)vy[u + djp + dr];
        zu.r = (double)vz[u + dr]; tu.r = (double)te[u + dr];
      }
      // one cell; *i is the cell's right neighbour, *l its left one
      auto cell = [&](double xc, double xi, double xdc, double xdi, double xuc, double xui, double xjc, double xji, double xmc, double xmi,
                      double yl, double yc, double yi, double yjl, double yjc, double yji, double ydc, double yjdc, double yuc, double yujc,
                      double zl, double zc, double zi, double zul, double zuc, double zui, double zjc, double zujc, double zmc, double zumc,
                      double tl, double ti, double tjc, double tmc, double tuc, double tdc, double fc) {
        const double h11 = (xi - xc) * udx1;
        const double h12 = ((xjc + xji) - (xmc + xmi)) * 0.25 * udx2;
        const double h13 = ((xuc + xui) - (xdc + xdi)) * 0.25 * udx3;
        const double h21 = ((yi + yji) - (yl + yjl)) * 0.25 * udx1;
        const double h22 = (yjc - yc) * udx2;
        const double h23 = ((yuc + yujc) - (ydc + yjdc)) * 0.25 * udx3;
        const double h31 = ((zi + zui) - (zl + zul)) * 0.25 * udx1;
        const double h32 = ((zjc + zujc) - (zmc + zumc)) * 0.25 * udx2;
        const double h33 = (zuc - zc) * udx3;
        double tke = (xc * xc + xi * xi + yc * yc + yjc * yjc + zc * zc + zuc * zuc) * 0.5;
        tke = tke * 0.5;
        double d = h11 * h11 + h22 * h22 + h33 * h33 + 0.5 * ((h21 + h12) * (h21 + h12)) + 0.5 * ((h31 + h13) * (h31 + h13)) +
                   0.5 * ((h32 + h23) * (h32 + h23));
        d = d * 2.0 / ren;
        const double ax = 0.5 * g.dx1 * (ti - tl), ay = 0.5 * g.dx2 * (tjc - tmc), az = 0.5 * g.dx3 * (tuc - tdc);
        double chi = ax * ax + ay * ay + az * az;
        chi = chi / pec;
        if (fc == 1.0) {
          acc[0] += tke;
          acc[1] += d;
          acc[2] += chi;
          acc[3] += 1.0;
        }
      };
      cell(x.a, x.b, xd.a, xd.b, xu.a, xu.b, xj.a, xj.b, xm.a, xm.b, y.l, y.a, y.b, yj.l, yj.a, yj.b, yd.a, yjd.a, yu.a, yuj.a,
           z.l, z.a, z.b, zu.l, zu.a, zu.b, zj.a, zuj.a, zm.a, zum.a, t.l, t.b, tj.a, tm.a, tu.a, td.a, f.a);
      cell(x.b, x.r, xd.b, xd.r, xu.b, xu.r, xj.b, xj.r, xm.b, xm.r, y.a, y.b, y.r, yj.a, yj.b, yj.r, yd.b, yjd.b, yu.b, yuj.b,
           z.a, z.b, z.r, zu.a, zu.b, zu.r, zj.b, zuj.b, zm.b, zum.b, t.a, t.r, tj.b, tm.b, tu.b, td.b, f.b);
      xd = x; x = xu;
      yd = {y.a, y.b}; yjd = {yj.a, yj.b}; y = yu; yj = yuj;
      z = zu; zj = zuj; zm = zum;
      td = {t.a, t.b}; t = tu;
      c = u;
    }
  }
  __shared__ double red[4][DISS_THREADS / 64];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    double v = acc[q];
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    if (lane == 0) red[q][w] = v;
  }
  __syncthreads();
  if (threadIdx.x < 4) {
    double v = 0.0;
    for (int q = 0; q < DISS_THREADS / 64; ++q) v += red[threadIdx.x][q];
    part[4 * blockIdx.x + threadIdx.x] = v;
  }
}

// The block partials of one quantity per wave: a lane takes every 64th, in
// order, then a fixed tree (a single thread per quantity waited for each load
// in turn: 277 us for 2048 partials).
__global__ __launch_bounds__(256) void k_diss_final(const double* __restrict__ part, int nb, double* __restrict__ out) {
  const int q = threadIdx.x >> 6, lane = threadIdx.x & 63;
  double v = 0.0;
#pragma unroll 16
  for (int b = lane; b < nb; b += 64) v += part[4 * b + q];
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  if (lane == 0) out[q] = v;
}

template <typename R>
int launch_diss(melt_ctx* ctx, double* sums) {
  double* part = ctx->d_red;
  double* out = ctx->d_red + 4 * DISS_BLOCKS;
  const int tiles = (ctx->n1 * ctx->n2 / 2 + DISS_THREADS - 1) / DISS_THREADS;
  // as many segments as leave at most DISS_BLOCKS blocks, each a plane at least
  const int segs = std::max(1, std::min(ctx->n3, DISS_BLOCKS / tiles));
  const int dz = (ctx->n3 + segs - 1) / segs, items = tiles * ((ctx->n3 + dz - 1) / dz), nb = std::min(items, DISS_BLOCKS);
  hipLaunchKernelGGL(k_diss_partial<R>, dim3(nb), dim3(DISS_THREADS), 0, ctx->stream, make_grid(ctx), fld<R>(ctx, MELT_VX),
                     fld<R>(ctx, MELT_VY), fld<R>(ctx, MELT_VZ), fld<R>(ctx, MELT_TEMP), fld<R>(ctx, MELT_VOFP), ctx->cfg.ren,
                     ctx->cfg.ren * ctx->cfg.prandtl, tiles, dz, items, part);
  MELT_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_diss_final, dim3(1), dim3(256), 0, ctx->stream, part, nb, out);
  MELT_HIP(hipGetLastError());
  MELT_HIP(hipMemcpyAsync(sums, out, 4 * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
  MELT_HIP(hipStreamSynchronize(ctx->stream));
  return 0;
}

}  // namespace

int diag_dissipation(melt_ctx* ctx, double* sums) { return ctx->fp32 ? launch_diss<float>(ctx, sums) : launch_diss<double>(ctx, sums); }

// get_dt (cfl.f90:33-77): the largest advective CFL of the cells at the
// current dt, at least the viscous one 6 dt dx1^2 / Re, and dt scaled to cflfix.
extern "C" int melt_get_dt(melt_ctx* ctx, double cflfix, double* dt_out) {
  if (!ctx || !dt_out || !(ctx->dt > 0.0)) return MELT_ERR_ARG;
  double adv = 0.0;
  int rc = euler_reduce_max(ctx, 2, &adv, ctx->dt);
  if (rc) return rc;
  double buf = adv;
  const double visc = 6.0 / ctx->cfg.ren * ctx->dt * (ctx->dx1 * ctx->dx1);
  if (visc > buf) buf = visc;
  *dt_out = buf > 0.0 ? ctx->dt * cflfix / buf : ctx->dt;
  return 0;
}

// CalcDissipation (diss.f90:11-201): re-tags the cells of a moving body first
// (diss.f90:47-49), sums over the fully fluid cells and forms the statistics
// the reference writes to diss.txt (diss.f90:155-197):
// out = {diss_volAvg, kenerg, urms, eta, lambda_t, Re_L, re_lam, L_int,
//        chi_volAvg, kmax_eta, sumVOF}.
extern "C" int melt_dissipation(melt_ctx* ctx, double* out) {
  if (!ctx || !out) return MELT_ERR_ARG;
  const melt_config& c = ctx->cfg;
  const bool moving = c.imlsfor == 1 && (c.imlsstr == 1 || c.imelt == 1) && ctx->has_geom;
  int rc;
  if (moving && ((rc = ibm_tag(ctx)) || (c.tagtype != 0 && (rc = euler_launch_interp_vof(ctx))))) return rc;
  double s[4];
  if ((rc = diag_dissipation(ctx, s))) return rc;
  const double sumvof = s[3];
  const double kenerg = s[0] / sumvof;
  const double nu = 1.0 / c.ren;
  const double diss = s[1] / sumvof;
  const double chi = s[2] / sumvof;
  const double urms = sqrt(2.0 / 3.0 * kenerg);
  const double eta = pow(nu * nu * nu / diss, 0.25);
  const double kmax_eta = ctx->pi * ctx->dx1 * eta;
  const double re_l = kenerg * kenerg / (nu * diss);
  const double lambda_t = sqrt(15.0 * nu * (urms * urms) / diss);
  const double re_lam = urms * lambda_t / nu;
  const double l_int = sqrt(kenerg * kenerg * kenerg) / diss;
  const double v[11] = {diss, kenerg, urms, eta, lambda_t, re_l, re_lam, l_int, chi, kmax_eta, sumvof};
  for (int q = 0; q < 11; ++q) out[q] = v[q];
  return melt_sync(ctx);
}
