// Pressure Poisson solve of phcalc.f90:11-97 on gfx950.
//
// phi = L^{-1} dph with L the 7-point staggered Laplacian and the (0,0,0) mode
// set to zero: forward transforms in x (real-to-complex, fused with the
// divergence of divg.f90 in the fused substep), y and z, division by the
// modified wavenumbers -(ak3 + ak1 + ak2) (phini.f90:35-55) after the 1/N^3
// normalisation (phcalc.f90:48-60), and the inverse transforms.  Each transform
// is a radix-4/2/3 FFT of a tile of lines held in registers (32 to 512 points)
// or LDS, so each pass reads and writes the spectrum once.  The z pass does forward FFT, division
// and inverse FFT in one visit.
//
// The real transforms along x pack two real lines into one complex line
// (z = a + i b) and separate the two half spectra afterwards (inverse: the
// two Hermitian half spectra are packed the same way), which halves their LDS
// work.  Radix stages are templates, so every butterfly lives in registers.
//
// Spectrum layout: complex (n1hp x N2 x N3), kx fastest, n1hp = N1/2+1 rounded
// up to a multiple of 8 so every row starts on a 128-byte boundary.
#include <cmath>
#include <cstring>
#include <type_traits>

#include "common.h"

namespace {

template <typename T>
struct alignas(2 * sizeof(T)) cx {
  T x, y;
};
template <typename T>
__device__ __forceinline__ cx<T> mkc(T a, T b) {
  cx<T> r;
  r.x = a;
  r.y = b;
  return r;
}
template <typename T>
__device__ __forceinline__ cx<T> cadd(cx<T> a, cx<T> b) { return mkc<T>(a.x + b.x, a.y + b.y); }
template <typename T>
__device__ __forceinline__ cx<T> csub(cx<T> a, cx<T> b) { return mkc<T>(a.x - b.x, a.y - b.y); }
template <typename T>
__device__ __forceinline__ cx<T> cmul(cx<T> a, cx<T> b) { return mkc<T>(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }

constexpr int FFT_NT = 256;   // threads per FFT block
constexpr int FFT_EPT = 8;    // LDS elements per thread: a tile holds <= 2048 complex values

struct FftPlan {
  int N, nst;
  int radix[24];
};

// One Stockham stage of radix R over the tile: element (line l, position p)
// at s[l*ls + p*ps].  LFAST: consecutive butterflies run over lines (tile
// layouts with the line index contiguous) instead of positions.
template <typename T, int R, bool LFAST>
__device__ __forceinline__ void fft_stage(cx<T>* s, int nl, int ls, int ps, int N, int Ns, const cx<T>* __restrict__ tw, bool inv) {
  constexpr int Q = (FFT_EPT + R - 1) / R;  // butterflies per thread
  const int NR = N / R, nbf = nl * NR, tid = threadIdx.x, nt = blockDim.x;
  const int step = N / (Ns * R);
  cx<T> v[Q][R];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    int b = tid + q * nt;
    if (b < nbf) {
      int l = LFAST ? b % nl : b / NR;
      int j = LFAST ? b / nl : b % NR;
#pragma unroll
      for (int r = 0; r < R; ++r) v[q][r] = s[l * ls + (j + r * NR) * ps];
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    int b = tid + q * nt;
    if (b < nbf) {
      int l = LFAST ? b % nl : b / NR;
      int j = LFAST ? b / nl : b % NR;
      int k = j % Ns;
#pragma unroll
      for (int r = 1; r < R; ++r) {
        cx<T> w = tw[k * r * step];
        if (inv) w.y = -w.y;
        v[q][r] = cmul(v[q][r], w);
      }
      cx<T> y[R];
      if constexpr (R == 4) {
        cx<T> a0 = cadd(v[q][0], v[q][2]), a1 = csub(v[q][0], v[q][2]);
        cx<T> a2 = cadd(v[q][1], v[q][3]), d = csub(v[q][1], v[q][3]);
        cx<T> a3 = inv ? mkc<T>(-d.y, d.x) : mkc<T>(d.y, -d.x);  // +i d (backward) or -i d (forward)
        y[0] = cadd(a0, a2); y[1] = cadd(a1, a3); y[2] = csub(a0, a2); y[3] = csub(a1, a3);
      } else if constexpr (R == 2) {
        y[0] = cadd(v[q][0], v[q][1]); y[1] = csub(v[q][0], v[q][1]);
      } else {
        const T c = T(-0.5), sn = (inv ? T(1) : T(-1)) * T(0.86602540378443864676);
        cx<T> sm = cadd(v[q][1], v[q][2]), df = csub(v[q][1], v[q][2]);
        y[0] = cadd(v[q][0], sm);
        cx<T> t1 = mkc<T>(v[q][0].x + c * sm.x, v[q][0].y + c * sm.y);
        cx<T> t2 = mkc<T>(-sn * df.y, sn * df.x);  // i sn df
        y[1] = cadd(t1, t2); y[2] = csub(t1, t2);
      }
      int o = (j / Ns) * Ns * R + k;
#pragma unroll
      for (int r = 0; r < R; ++r) s[l * ls + (o + r * Ns) * ps] = y[r];
    }
  }
  __syncthreads();
}

// Unnormalised in-LDS FFT of nl lines (forward: exp(-i...), as FFTW_FORWARD).
// The tile must hold at most FFT_EPT * blockDim.x elements, be complete in LDS
// and visible (barrier) on entry; it is visible again on return.
template <typename T, bool LFAST>
__device__ void lds_fft(cx<T>* s, int nl, int ls, int ps, const FftPlan& P, const cx<T>* __restrict__ tw, bool inv) {
  int Ns = 1;
  for (int st = 0; st < P.nst; ++st) {
    const int R = P.radix[st];
    if (R == 4) fft_stage<T, 4, LFAST>(s, nl, ls, ps, P.N, Ns, tw, inv);
    else if (R == 2) fft_stage<T, 2, LFAST>(s, nl, ls, ps, P.N, Ns, tw, inv);
    else fft_stage<T, 3, LFAST>(s, nl, ls, ps, P.N, Ns, tw, inv);
    Ns *= R;
  }
}

template <typename T>
struct SpecArgs {
  Grid g;
  int n1h, n1hp;
  cx<T>* spec;
};

// x pass, forward: nl real lines (divergence divg.f90:17-20, or a stored field)
// -> bins 0..N1/2 of each, two lines per complex transform.  div_slots !=
// null: max |div u| in FP64 (divg.f90:36-50) is folded into those slots too.
template <typename Rf, typename T>
__global__ __launch_bounds__(FFT_NT) void k_fft_x_fwd(SpecArgs<T> S, FftPlan P, const cx<T>* __restrict__ tw, int nl,
                                                      const Rf* __restrict__ vx, const Rf* __restrict__ vy, const Rf* __restrict__ vz,
                                                      const Rf* __restrict__ src, T usdtal, const int* __restrict__ gate,
                                                      unsigned long long* __restrict__ div_slots) {
  if (gate && *gate == 0) return;
  extern __shared__ unsigned char smem[];
  cx<T>* sh = reinterpret_cast<cx<T>*>(smem);
  T* shr = reinterpret_cast<T*>(smem);
  const Grid& g = S.g;
  const int N = g.n1, ls = N + 1;
  unsigned t = xcd_block(blockIdx.x, gridDim.x);
  int jt, k;
  tiled_2d(t, g.n2 / nl, g.n3, 16, 8, jt, k);  // the divergence reads lines j+1 and planes k+1
  const int j0 = jt * nl;
  const T dx1 = (T)g.dx1, dx2 = (T)g.dx2, dx3 = (T)g.dx3;
  const int kp = k == g.n3 - 1 ? 0 : k + 1;
  double dmax = 0.0;
  for (int c = threadIdx.x; c < nl * N; c += blockDim.x) {
    int l = c / N, i = c % N, j = j0 + l;
    size_t idx = (size_t)i + (size_t)N * ((size_t)j + (size_t)g.n2 * k);
    T v;
    if (src) {
      v = (T)src[idx];
    } else {
      int ip = i == N - 1 ? 0 : i + 1, jp = j == g.n2 - 1 ? 0 : j + 1;
      const Rf x0 = vx[idx], x1 = vx[idx - i + ip], y0 = vy[idx], y1 = vy[(size_t)i + (size_t)N * ((size_t)jp + (size_t)g.n2 * k)];
      const Rf z0 = vz[idx], z1 = vz[(size_t)i + (size_t)N * ((size_t)j + (size_t)g.n2 * kp)];
      T dq = ((T)x1 - (T)x0) * dx1 + ((T)y1 - (T)y0) * dx2 + ((T)z1 - (T)z0) * dx3;
      v = dq * usdtal;
      if (div_slots)
        dmax = fmax(dmax, fabs(((double)x1 - (double)x0) * g.dx1 + ((double)y1 - (double)y0) * g.dx2 + ((double)z1 - (double)z0) * g.dx3));
    }
    shr[2 * ((l >> 1) * ls + i) + (l & 1)] = v;  // line 2p -> real part, 2p+1 -> imaginary part
  }
  if (div_slots) block_max_to_slots(dmax, div_slots);
  __syncthreads();
  lds_fft<T, false>(sh, nl / 2, ls, 1, P, tw, false);
  const int np = nl / 2;
  for (int c = threadIdx.x; c < np * S.n1hp; c += blockDim.x) {
    int pl = c / S.n1hp, m = c % S.n1hp;
    cx<T> a = mkc<T>(0, 0), b = mkc<T>(0, 0);
    if (m < S.n1h) {
      cx<T> z = sh[pl * ls + m], zr = sh[pl * ls + (m == 0 ? 0 : N - m)];
      // A = (Z[m] + conj Z[N-m]) / 2,  B = (Z[m] - conj Z[N-m]) / (2i)
      a = mkc<T>((z.x + zr.x) * T(0.5), (z.y - zr.y) * T(0.5));
      b = mkc<T>((z.y + zr.y) * T(0.5), (zr.x - z.x) * T(0.5));
    }
    size_t row = (size_t)S.n1hp * ((size_t)(j0 + 2 * pl) + (size_t)g.n2 * k);
    S.spec[row + m] = a;
    S.spec[row + S.n1hp + m] = b;
  }
}

// y pass: tile of nl kx-columns (the last tile may be partial) for one z plane.
template <typename T>
__global__ __launch_bounds__(FFT_NT) void k_fft_y(SpecArgs<T> S, FftPlan P, const cx<T>* __restrict__ tw, int nl, int inv,
                                                  const int* __restrict__ gate) {
  if (gate && *gate == 0) return;
  extern __shared__ unsigned char smem[];
  cx<T>* sh = reinterpret_cast<cx<T>*>(smem);
  const Grid& g = S.g;
  const int N = g.n2;
  unsigned t = xcd_block(blockIdx.x, gridDim.x);
  int ntm = (S.n1hp + nl - 1) / nl;
  int m0 = (t % ntm) * nl, k = t / ntm;
  size_t base = (size_t)m0 + (size_t)S.n1hp * (size_t)g.n2 * k;
  for (int c = threadIdx.x; c < nl * N; c += blockDim.x) {
    int l = c % nl, p = c / nl;
    sh[p * nl + l] = m0 + l < S.n1hp ? S.spec[base + l + (size_t)S.n1hp * p] : mkc<T>(0, 0);
  }
  __syncthreads();
  lds_fft<T, true>(sh, nl, 1, nl, P, tw, inv != 0);
  for (int c = threadIdx.x; c < nl * N; c += blockDim.x) {
    int l = c % nl, p = c / nl;
    if (m0 + l < S.n1hp) S.spec[base + l + (size_t)S.n1hp * p] = sh[p * nl + l];
  }
}

// z pass: forward FFT, 1/(N1 N2 N3), division by -(ak3+ak1+ak2) with the zero
// mode set to 0 (phcalc.f90:40-73), inverse FFT.
template <typename T>
__global__ __launch_bounds__(FFT_NT) void k_fft_z_solve(SpecArgs<T> S, FftPlan P, const cx<T>* __restrict__ tw, int nl,
                                                        const double* __restrict__ ak1, const double* __restrict__ ak2,
                                                        const double* __restrict__ ak3, double nrm, const int* __restrict__ gate) {
  if (gate && *gate == 0) return;
  extern __shared__ unsigned char smem[];
  cx<T>* sh = reinterpret_cast<cx<T>*>(smem);
  const Grid& g = S.g;
  const int N = g.n3;
  unsigned t = xcd_block(blockIdx.x, gridDim.x);
  int ntm = (S.n1hp + nl - 1) / nl;
  int m0 = (t % ntm) * nl, j = t / ntm;
  size_t plane = (size_t)S.n1hp * g.n2;
  size_t base = (size_t)m0 + (size_t)S.n1hp * j;
  for (int c = threadIdx.x; c < nl * N; c += blockDim.x) {
    int l = c % nl, p = c / nl;
    sh[p * nl + l] = m0 + l < S.n1hp ? S.spec[base + l + plane * p] : mkc<T>(0, 0);
  }
  __syncthreads();
  lds_fft<T, true>(sh, nl, 1, nl, P, tw, false);
  for (int c = threadIdx.x; c < nl * N; c += blockDim.x) {
    int l = c % nl, p = c / nl, m = m0 + l;
    cx<T> v = sh[p * nl + l];
    if (m < S.n1h) {
      double ev = -ak3[p] - ak1[m] - ak2[j];
      double vx = (double)v.x / nrm, vy = (double)v.y / nrm;
      if (m == 0 && j == 0 && p == 0) { vx = 0.0; vy = 0.0; }
      else { vx = vx / ev; vy = vy / ev; }
      v = mkc<T>((T)vx, (T)vy);
    } else {
      v = mkc<T>(0, 0);
    }
    sh[p * nl + l] = v;
  }
  __syncthreads();
  lds_fft<T, true>(sh, nl, 1, nl, P, tw, true);
  for (int c = threadIdx.x; c < nl * N; c += blockDim.x) {
    int l = c % nl, p = c / nl;
    if (m0 + l < S.n1hp) S.spec[base + l + plane * p] = sh[p * nl + l];
  }
}

// x pass, backward (complex-to-real with FFTW c2r semantics: the imaginary
// parts of bins 0 and N1/2 are ignored): the half spectra A, B of lines 2p,
// 2p+1 are packed as Z = A + iB over the full Hermitian range, one inverse
// FFT gives line 2p in the real and line 2p+1 in the imaginary part.
template <typename Rf, typename T>
__global__ __launch_bounds__(FFT_NT) void k_fft_x_bwd(SpecArgs<T> S, FftPlan P, const cx<T>* __restrict__ tw, int nl, Rf* __restrict__ dst,
                                                      const int* __restrict__ gate) {
  if (gate && *gate == 0) return;
  extern __shared__ unsigned char smem[];
  cx<T>* sh = reinterpret_cast<cx<T>*>(smem);
  const Grid& g = S.g;
  const int N = g.n1, ls = N + 1, np = nl / 2;
  unsigned t = xcd_block(blockIdx.x, gridDim.x);
  int ntj = g.n2 / nl;
  int j0 = (t % ntj) * nl, k = t / ntj;
  for (int c = threadIdx.x; c < np * S.n1h; c += blockDim.x) {
    int pl = c / S.n1h, m = c % S.n1h;
    size_t row = (size_t)S.n1hp * ((size_t)(j0 + 2 * pl) + (size_t)g.n2 * k);
    cx<T> a = S.spec[row + m], b = S.spec[row + S.n1hp + m];
    if (m == 0 || 2 * m == N) { a.y = T(0); b.y = T(0); }
    sh[pl * ls + m] = mkc<T>(a.x - b.y, a.y + b.x);                         // A + iB
    if (m > 0 && 2 * m < N) sh[pl * ls + (N - m)] = mkc<T>(a.x + b.y, b.x - a.y);  // conj(A) + i conj(B)
  }
  __syncthreads();
  lds_fft<T, false>(sh, np, ls, 1, P, tw, true);
  for (int c = threadIdx.x; c < nl * N; c += blockDim.x) {
    int l = c / N, i = c % N;
    cx<T> z = sh[(l >> 1) * ls + i];
    dst[(size_t)i + (size_t)N * ((size_t)(j0 + l) + (size_t)g.n2 * k)] = (Rf)((l & 1) ? z.y : z.x);
  }
}

// ---------------------------------------------------------------- register FFTs
// Lines of N = P*Q points are transformed in two stages with one LDS exchange
// (two barriers a component) between them instead of one per radix: thread
// b < Q of a line loads x[b + Q a], a < P, straight from HBM and transforms them
// in registers (stage A); thread k < P then receives the Q values of its k,
// finishes them in registers (stage B) and holds X[k + P q] for every q.
//
// 64 = 8 * 8 and 256 = 16 * 16: stage A is a P-point DFT and the twiddles
// W_N^(b k), stage B a second DFT, X[k1 + P k2] = sum_b W_Q^(b k2) W_N^(b k1)
// sum_a x[b + Q a] W_P^(a k1); the inverse runs the same steps from that layout
// in reverse.
//
// The other lengths group the radix stages of lds_fft: stage A is its first
// radices (product P), stage B the rest, each on the values a thread holds, with
// the same twiddles, butterflies and order, so the results are those of lds_fft
// to the last bit.  (In Stockham's order the first stages with product P
// combine x[b + Q a] only, and the stages after them, from Ns = P on, the
// elements k + P a only.)
//
// Where P and Q differ one stage runs on a part of the threads (whole waves);
// the passes are bound by HBM or, on small grids, by the chain of barriers, so
// the shorter chain is what counts.  All five passes of a solve against the
// staged transforms above, us (FP64 / FP32): 48^3 64 -> 37 / 58 -> 36, 96^3 98 ->
// 56 / 84 -> 44, 128^3 127 -> 82 / 106 -> 64, 192^3 258 -> 166 / 193 -> 109, 384^3
// 2009 -> 1272 / 1152 -> 700, 512^3 5138 -> 2716 / 2755 -> 1599 (384^3 FP64 moves
// 5.4 GB of spectrum and velocity: 1140 us at the rate of a copy).

// cos(pi m / 8) and sin(pi m / 8), m = 0..15 (W_16^m = cos - i sin forward)
template <typename T>
__device__ __forceinline__ cx<T> w16(int m, bool inv) {
  const T c1 = T(0.92387953251128675613), s1 = T(0.38268343236508977173), r = T(0.70710678118654752440);
  const T cs[16] = {T(1), c1, r, s1, T(0), -s1, -r, -c1, T(-1), -c1, -r, -s1, T(0), s1, r, c1};
  const T sn[16] = {T(0), s1, r, c1, T(1), c1, r, s1, T(0), -s1, -r, -c1, T(-1), -c1, -r, -s1};
  return mkc<T>(cs[m], inv ? sn[m] : -sn[m]);
}

// v * W_16^M with the exact forms for M = 0, 4, 8, 12
template <typename T, int M>
__device__ __forceinline__ cx<T> mul_w16(cx<T> v, bool inv) {
  constexpr int m = M % 16;
  if constexpr (m == 0) return v;
  else if constexpr (m == 8) return mkc<T>(-v.x, -v.y);
  else if constexpr (m == 4) return inv ? mkc<T>(-v.y, v.x) : mkc<T>(v.y, -v.x);    // +i v or -i v
  else if constexpr (m == 12) return inv ? mkc<T>(v.y, -v.x) : mkc<T>(-v.y, v.x);
  else return cmul(v, w16<T>(m, inv));
}

// DFT of R values in place, natural order (the butterflies of fft_stage)
template <typename T>
__device__ __forceinline__ void dft4(cx<T>& x0, cx<T>& x1, cx<T>& x2, cx<T>& x3, bool inv) {
  cx<T> a0 = cadd(x0, x2), a1 = csub(x0, x2), a2 = cadd(x1, x3), d = csub(x1, x3);
  cx<T> a3 = inv ? mkc<T>(-d.y, d.x) : mkc<T>(d.y, -d.x);
  x0 = cadd(a0, a2); x1 = cadd(a1, a3); x2 = csub(a0, a2); x3 = csub(a1, a3);
}
template <typename T, int R>
__device__ __forceinline__ void butterfly(cx<T> (&v)[R], bool inv) {
  if constexpr (R == 4) {
    dft4(v[0], v[1], v[2], v[3], inv);
  } else if constexpr (R == 2) {
    const cx<T> e = v[0], f = v[1];
    v[0] = cadd(e, f); v[1] = csub(e, f);
  } else {
    static_assert(R == 3, "radix 2, 3 or 4");
    const T c = T(-0.5), sn = (inv ? T(1) : T(-1)) * T(0.86602540378443864676);
    const cx<T> sm = cadd(v[1], v[2]), df = csub(v[1], v[2]);
    const cx<T> t1 = mkc<T>(v[0].x + c * sm.x, v[0].y + c * sm.y), t2 = mkc<T>(-sn * df.y, sn * df.x);   // t2 = i sn df
    v[0] = cadd(v[0], sm);
    v[1] = cadd(t1, t2); v[2] = csub(t1, t2);
  }
}

// P-point DFT (P = 8, 16) of v[0..P-1] in registers; result in natural order.
template <typename T, int P>
__device__ __forceinline__ void dft_reg(cx<T> (&v)[P], bool inv) {
  if constexpr (P == 16) {
    // a = 4 a1 + a0: DFT4 over a1, twiddle W_16^(a0 k0), DFT4 over a0
#pragma unroll
    for (int a0 = 0; a0 < 4; ++a0) dft4(v[a0], v[a0 + 4], v[a0 + 8], v[a0 + 12], inv);   // v[a0 + 4 k0]
    v[5] = mul_w16<T, 1>(v[5], inv); v[9] = mul_w16<T, 2>(v[9], inv); v[13] = mul_w16<T, 3>(v[13], inv);
    v[6] = mul_w16<T, 2>(v[6], inv); v[10] = mul_w16<T, 4>(v[10], inv); v[14] = mul_w16<T, 6>(v[14], inv);
    v[7] = mul_w16<T, 3>(v[7], inv); v[11] = mul_w16<T, 6>(v[11], inv); v[15] = mul_w16<T, 9>(v[15], inv);
    cx<T> o[16];
#pragma unroll
    for (int k0 = 0; k0 < 4; ++k0) {
      cx<T> x0 = v[4 * k0], x1 = v[4 * k0 + 1], x2 = v[4 * k0 + 2], x3 = v[4 * k0 + 3];
      dft4(x0, x1, x2, x3, inv);
      o[k0] = x0; o[k0 + 4] = x1; o[k0 + 8] = x2; o[k0 + 12] = x3;
    }
#pragma unroll
    for (int q = 0; q < 16; ++q) v[q] = o[q];
  } else {
    static_assert(P == 8, "register DFT of 8 or 16 points");
    // a = 2 a1 + a0: DFT4 over a1, twiddle W_8^(a0 k0) = W_16^(2 a0 k0), DFT2 over a0
    dft4(v[0], v[2], v[4], v[6], inv);
    dft4(v[1], v[3], v[5], v[7], inv);
    v[3] = mul_w16<T, 2>(v[3], inv); v[5] = mul_w16<T, 4>(v[5], inv); v[7] = mul_w16<T, 6>(v[7], inv);
    cx<T> o[8];
#pragma unroll
    for (int k0 = 0; k0 < 4; ++k0) {
      cx<T> e = v[2 * k0], f = v[2 * k0 + 1];
      o[k0] = cadd(e, f); o[k0 + 4] = csub(e, f);
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = o[q];
  }
}

// Radix of the next stage of a plan with M points left (make_plan's order).
constexpr int next_radix(int M) { return M % 4 == 0 ? 4 : M % 2 == 0 ? 2 : 3; }

// The stages of an N-point Stockham transform from Ns = P0 on, with product M, on
// the M values v[a] = element k0 + P0 a a thread holds (L: product of those done;
// k0 < P0 the thread's, 0 for the first stages).  The butterflies with twiddle 1
// skip the product (1 - 0 i), which changes no value.
template <typename T, int N, int P0, int M, int L = 1>
__device__ __forceinline__ void stockham(cx<T> (&v)[M], const cx<T>* tw, int k0, bool inv) {
  if constexpr (L < M) {
    constexpr int R = next_radix(M / L), step = N / (P0 * L * R);
    cx<T> o[M];
#pragma unroll
    for (int j = 0; j < M / R; ++j) {
      const int kk = j % L, k = k0 + P0 * kk;
      cx<T> x[R];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        x[r] = v[j + r * (M / R)];
        if (r > 0 && !(P0 == 1 && kk == 0)) {
          cx<T> w = tw[k * r * step];
          if (inv) w.y = -w.y;
          x[r] = cmul(x[r], w);
        }
      }
      butterfly<T, R>(x, inv);
#pragma unroll
      for (int r = 0; r < R; ++r) o[(j / L) * L * R + kk + r * L] = x[r];
    }
#pragma unroll
    for (int q = 0; q < M; ++q) v[q] = o[q];
    // (keeps the next stage's twiddles from being loaded, and held, before this one is done)
    if constexpr (M >= 24) __builtin_amdgcn_sched_barrier(0);
    stockham<T, N, P0, M, L * R>(v, tw, k0, inv);
  }
}

// P-point DFT and the twiddles W_N^(b k1) of the square lengths
template <typename T, int P>
__device__ __forceinline__ void dft_twiddle(cx<T> (&v)[P], const cx<T>* tw, int b, bool inv) {
  dft_reg<T, P>(v, inv);
#pragma unroll
  for (int k1 = 1; k1 < P; ++k1) {
    cx<T> w = tw[b * k1];
    if (inv) w.y = -w.y;
    v[k1] = cmul(v[k1], w);
  }
}

// Stage A of thread b and stage B of thread k.
template <typename T, int P, int Q>
__device__ __forceinline__ void stage_a(cx<T> (&v)[P], const cx<T>* tw, int b, bool inv) {
  if constexpr (P == Q) dft_twiddle<T, P>(v, tw, b, inv);
  else stockham<T, P * Q, 1, P>(v, tw, 0, inv);
}
template <typename T, int P, int Q>
__device__ __forceinline__ void stage_b(cx<T> (&u)[Q], const cx<T>* tw, int k, bool inv) {
  if constexpr (P == Q) dft_reg<T, Q>(u, inv);
  else stockham<T, P * Q, P, Q>(u, tw, k, inv);
}

constexpr int RF_NC = 8;   // kx columns per register-FFT block (8 x 16 B = one 128-byte line per row; 16 and 32 measured slower)

// LDS image of one block of NC lines: the exchange tile (per line P rows of
// pitch Q+1) and the N twiddles.
template <typename T, int P, int Q, int NC>
struct RegFftLds {
  // The exchanges move the real and then the imaginary parts through one
  // tile of T (half the LDS of a complex tile, so more blocks fit per CU).
  // Line c's tile starts at c * CS; CS = 2 mod 16 puts the 16 lanes of a
  // 64-bit access in distinct bank pairs in both thread layouts (y/z: 8
  // columns x 2 threads per lane group; x: the threads of one line).
  static constexpr int CS = P * (Q + 1) + ((2 - P * (Q + 1) % 16) + 16) % 16;
  T ex[NC * CS];
  cx<T> tw[P * Q];
};

// Thread (c, b) of stage A (b < Q) holds v[k1], k1 < P; thread (d, k) of stage B
// (k < P) receives u[q] = v[k] of thread (d, q), one component at a time.  The
// tile must be free on entry (callers put a barrier after any earlier read of
// it).  Every thread of the block calls this; those past their stage's count
// only take part in the barriers.
template <typename T, int P, int Q, int NC>
__device__ __forceinline__ void exchange_ab(const cx<T> (&v)[P], cx<T> (&u)[Q], RegFftLds<T, P, Q, NC>& L, int c, int b, bool inA, int d, int k,
                                            bool inB) {
  T* ea = L.ex + c * L.CS + b;
  const T* eb = L.ex + d * L.CS + k * (Q + 1);
  if (inA)
#pragma unroll
    for (int k1 = 0; k1 < P; ++k1) ea[k1 * (Q + 1)] = v[k1].x;
  __syncthreads();
  if (inB)
#pragma unroll
    for (int q = 0; q < Q; ++q) u[q].x = eb[q];
  __syncthreads();
  if (inA)
#pragma unroll
    for (int k1 = 0; k1 < P; ++k1) ea[k1 * (Q + 1)] = v[k1].y;
  __syncthreads();
  if (inB)
#pragma unroll
    for (int q = 0; q < Q; ++q) u[q].y = eb[q];
}
// The reverse: thread (c, b) receives v[k1] = u[b] of thread (c, k1).
template <typename T, int P, int Q, int NC>
__device__ __forceinline__ void exchange_ba(cx<T> (&v)[P], const cx<T> (&u)[Q], RegFftLds<T, P, Q, NC>& L, int c, int b, bool inA, int d, int k,
                                            bool inB) {
  const T* ea = L.ex + c * L.CS + b;
  T* eb = L.ex + d * L.CS + k * (Q + 1);
  if (inB)
#pragma unroll
    for (int q = 0; q < Q; ++q) eb[q] = u[q].x;
  __syncthreads();
  if (inA)
#pragma unroll
    for (int k1 = 0; k1 < P; ++k1) v[k1].x = ea[k1 * (Q + 1)];
  __syncthreads();
  if (inB)
#pragma unroll
    for (int q = 0; q < Q; ++q) eb[q] = u[q].y;
  __syncthreads();
  if (inA)
#pragma unroll
    for (int k1 = 0; k1 < P; ++k1) v[k1].y = ea[k1 * (Q + 1)];
}

// From stage B's order (thread b holds element b + P q in u[q]) to stage A's
// (thread b holds element b + Q a in v[a]).
template <typename T, int P, int Q, int NC>
__device__ __forceinline__ void reorder_ba(cx<T> (&v)[P], const cx<T> (&u)[Q], RegFftLds<T, P, Q, NC>& L, int c, int b, bool inA, bool inB) {
  T* e = L.ex + c * L.CS + b;
  if (inB)
#pragma unroll
    for (int q = 0; q < Q; ++q) e[P * q] = u[q].x;
  __syncthreads();
  if (inA)
#pragma unroll
    for (int a = 0; a < P; ++a) v[a].x = e[Q * a];
  __syncthreads();
  if (inB)
#pragma unroll
    for (int q = 0; q < Q; ++q) e[P * q] = u[q].y;
  __syncthreads();
  if (inA)
#pragma unroll
    for (int a = 0; a < P; ++a) v[a].y = e[Q * a];
}

// Threads of a block of NC lines.
constexpr int rf_threads(int P, int Q, int NC) { return NC * (P > Q ? P : Q); }

// Element b + q of column c of a block's lines (rows rs apart): a block-uniform
// base plus one 32-bit lane offset, so the P or Q addresses of a thread live in
// scalar registers (as 64-bit lane addresses they take 2 P vector registers).
template <typename T>
struct Column {
  char* base;
  size_t row;     // bytes from row to row
  unsigned off;   // of this thread (below 32 rows of 1024 x 520 bins: under 4 GiB)
  __device__ __forceinline__ Column(cx<T>* p, size_t rs, int c, int b)
      : base(reinterpret_cast<char*>(p)), row(rs * sizeof(cx<T>)), off((unsigned)(((size_t)b * rs + (size_t)c) * sizeof(cx<T>))) {}
  __device__ __forceinline__ cx<T>& at(int q) const { return *reinterpret_cast<cx<T>*>(base + row * (size_t)q + off); }
};

// y pass (N2 = P*Q): RF_NC kx columns per block.
template <typename T, int P, int Q, bool INV>
__global__ __launch_bounds__(rf_threads(P, Q, RF_NC)) void k_fft_y_reg(SpecArgs<T> S, const cx<T>* __restrict__ tw, const int* __restrict__ gate) {
  if (gate && *gate == 0) return;
  __shared__ RegFftLds<T, P, Q, RF_NC> L;
  constexpr int N = P * Q, NT = rf_threads(P, Q, RF_NC);
  const int t = threadIdx.x, c = t % RF_NC, b = t / RF_NC;
  const bool inA = b < Q, inB = b < P;
  const unsigned blk = xcd_block(blockIdx.x, gridDim.x);
  const int ntm = S.n1hp / RF_NC;
  const int m0 = (int)(blk % (unsigned)ntm) * RF_NC, k = (int)(blk / (unsigned)ntm);
  for (int q = t; q < N; q += NT) L.tw[q] = tw[q];
  const Column<T> col(S.spec + (size_t)m0 + (size_t)S.n1hp * N * k, (size_t)S.n1hp, c, b);
  cx<T> v[P], u[Q];
  if (inA)
#pragma unroll
    for (int a = 0; a < P; ++a) v[a] = col.at(Q * a);
  __syncthreads();   // twiddles
  if (inA) stage_a<T, P, Q>(v, L.tw, b, INV);
  exchange_ab<T, P, Q, RF_NC>(v, u, L, c, b, inA, c, b, inB);
  if (!inB) return;
  stage_b<T, P, Q>(u, L.tw, b, INV);
#pragma unroll
  for (int k2 = 0; k2 < Q; ++k2) col.at(P * k2) = u[k2];
}

// z pass with register FFTs: forward FFT, 1/(N1 N2 N3), division by
// -(ak3+ak1+ak2) with the zero mode set to 0 (phcalc.f90:40-73), inverse FFT.
template <typename T, int P, int Q>
__global__ __launch_bounds__(rf_threads(P, Q, RF_NC), P * Q == 512 ? 2 : 1) void k_fft_z_solve_reg(SpecArgs<T> S, const cx<T>* __restrict__ tw,
                                                                             const double* __restrict__ ak1, const double* __restrict__ ak2,
                                                                             const double* __restrict__ ak3, double nrm,
                                                                             const int* __restrict__ gate) {
  if (gate && *gate == 0) return;
  constexpr int N = P * Q, NT = rf_threads(P, Q, RF_NC);
  __shared__ RegFftLds<T, P, Q, RF_NC> L;
  __shared__ double lak[N];
  const int t = threadIdx.x, c = t % RF_NC, b = t / RF_NC;
  const bool inA = b < Q, inB = b < P;
  const unsigned blk = xcd_block(blockIdx.x, gridDim.x);
  const int ntm = S.n1hp / RF_NC;
  const int m0 = (int)(blk % (unsigned)ntm) * RF_NC, m = m0 + c, j = (int)(blk / (unsigned)ntm);
  const double a1 = ak1[m], a2 = ak2[j];   // (the padding bins n1h <= m < n1hp are below n1)
  for (int q = t; q < N; q += NT) {
    L.tw[q] = tw[q];
    lak[q] = ak3[q];
  }
  const Column<T> col(S.spec + (size_t)m0 + (size_t)S.n1hp * j, (size_t)S.n1hp * S.g.n2, c, b);
  cx<T> v[P], u[Q];
  if (inA)
#pragma unroll
    for (int a = 0; a < P; ++a) v[a] = col.at(Q * a);
  __syncthreads();
  if (inA) stage_a<T, P, Q>(v, L.tw, b, false);
  exchange_ab<T, P, Q, RF_NC>(v, u, L, c, b, inA, c, b, inB);
  if (inB) {
    stage_b<T, P, Q>(u, L.tw, b, false);
#pragma unroll
    for (int k2 = 0; k2 < Q; ++k2) {
      // selected, not branched over: a branch per point keeps every operand of
      // every division live (166 -> 138 registers at 256 points of FP64)
      const int p = b + P * k2;
      const double ev = -lak[p] - a1 - a2;
      const double vx = (double)u[k2].x / nrm / ev, vy = (double)u[k2].y / nrm / ev;
      const bool zero = m >= S.n1h || (m == 0 && j == 0 && p == 0);
      u[k2] = mkc<T>(zero ? T(0) : (T)vx, zero ? T(0) : (T)vy);
    }
  }
  if constexpr (P == Q) {   // back through the same steps in reverse
    if (inB) dft_twiddle<T, Q>(u, L.tw, b, true);   // over k2: u[n1] = W_N^-(k1 n1) Z[k1 = b][n1]
    __syncthreads();   // every thread has read its forward exchange
    exchange_ba<T, P, Q, RF_NC>(v, u, L, c, b, inA, c, b, inB);
    if (!inA) return;
    dft_reg<T, P>(v, true);   // over k1: v[n2] = x[b + Q n2]
#pragma unroll
    for (int n2 = 0; n2 < P; ++n2) col.at(Q * n2) = v[n2];
  } else {   // the points in natural order, then the same two stages
    __syncthreads();
    reorder_ba<T, P, Q, RF_NC>(v, u, L, c, b, inA, inB);
    if (inA) stage_a<T, P, Q>(v, L.tw, b, true);
    __syncthreads();   // the reordered values are read
    exchange_ab<T, P, Q, RF_NC>(v, u, L, c, b, inA, c, b, inB);
    if (!inB) return;
    stage_b<T, P, Q>(u, L.tw, b, true);
#pragma unroll
    for (int k2 = 0; k2 < Q; ++k2) col.at(P * k2) = u[k2];
  }
}

// Line pairs per block of the x passes: about 128 threads, and 2 NPB lines that
// divide N (the passes have n1 = n2).  256 points take 16 pairs, whose rows j+1
// the divergence reads once more per 32 lines instead of 16 (forward, FP64 125 ->
// 107 us, FP32 84 -> 70; at 192 16 pairs are slower, 40 -> 44 in FP32, at 128 and 384
// the same).
constexpr int x_pairs(int N) { return N == 64 || N == 256 ? 16 : N == 512 ? 4 : 8; }
// Threads of a forward x block: whole waves, since its maximum of |div u| shuffles
// over all 64 lanes of each (48 points: 8 pairs of 12 threads, 96, become 128).
constexpr int x_fwd_threads(int P, int Q) { return (rf_threads(P, Q, x_pairs(P * Q)) + 63) / 64 * 64; }
// Waves per SIMD the forward x pass asks for: 384 points in FP64 take 172 registers
// by themselves, four above what three waves leave (486 -> 400 us).
template <typename T>
constexpr int x_fwd_waves(int N) { return sizeof(T) == 8 && N == 384 ? 3 : 1; }

// x pass, forward, with register FFTs (N1 = P*Q): thread (c, b) of stage A owns
// line pair c of the block (lines j, j+1 packed as real and imaginary part,
// divergence formed at load as k_fft_x_fwd) and points b + Q a.  After the
// transform the two half spectra are separated with the mirror bins N-m,
// exchanged through LDS.
template <typename Rf, typename T, int P, int Q>
__global__ __launch_bounds__(x_fwd_threads(P, Q), x_fwd_waves<T>(P * Q)) void k_fft_x_fwd_reg(
    SpecArgs<T> S, const cx<T>* __restrict__ tw, const Rf* __restrict__ vx, const Rf* __restrict__ vy, const Rf* __restrict__ vz,
    const Rf* __restrict__ src, T usdtal, const int* __restrict__ gate, unsigned long long* __restrict__ div_slots) {
  if (gate && *gate == 0) return;
  constexpr int N = P * Q, NPB = x_pairs(N), NT = x_fwd_threads(P, Q), TB = NT / NPB;
  static_assert(N % (2 * NPB) == 0, "whole line pairs per block");
  static_assert(NT % 64 == 0 && NT % NPB == 0, "whole waves, and as many threads for each pair");
  __shared__ RegFftLds<T, P, Q, NPB> L;
  static_assert(NPB * N <= (int)(sizeof(L.ex) / sizeof(L.ex[0])), "mirror exchange fits the transpose tile");
  const Grid& g = S.g;
  // stage A: TB threads a line, b < Q; stage B: the first NPB * P threads, P a line
  const int t = threadIdx.x, b = t % TB, c = t / TB, kb = t % P, d = t / P;
  const bool inA = b < Q, inB = d < NPB;
  int jt, k;
  tiled_2d(xcd_block(blockIdx.x, gridDim.x), g.n2 / (2 * NPB), g.n3, 16, 8, jt, k);  // the divergence reads rows j+1 and planes k+1
  const int j = jt * 2 * NPB + 2 * c, kp = k == g.n3 - 1 ? 0 : k + 1;
  for (int q = t; q < N; q += NT) L.tw[q] = tw[q];
  const T dx1 = (T)g.dx1, dx2 = (T)g.dx2, dx3 = (T)g.dx3;
  double dmax = 0.0;
  cx<T> v[P], u[Q];
  if (inA) {
    // lines j0.. of the block start at a uniform base; a lane's two lines and
    // their y neighbours at 32-bit offsets from it (j is even and n2 is, so only
    // the row after the second line can wrap)
    const size_t line = (size_t)N * ((size_t)(j - 2 * c) + (size_t)g.n2 * k), up = (size_t)N * ((size_t)(j - 2 * c) + (size_t)g.n2 * kp);
    const int o = N * 2 * c + b, jw = j + 2 == g.n2 ? N * (2 - g.n2) : 2 * N;   // to the row after the second line
    const Rf *px = vx + line, *py = vy + line, *pz = vz + line, *pu = vz + up, *ps = src + line;
#pragma unroll
    for (int a = 0; a < P; ++a) {
      const int i = o + Q * a;
      T z[2];
      if (src) {
        z[0] = (T)ps[i];
        z[1] = (T)ps[i + N];
      } else {
        const int ip = a == P - 1 && b == Q - 1 ? i - (N - 1) : i + 1;
        const Rf y[3] = {py[i], py[i + N], py[i + jw]};
#pragma unroll
        for (int l = 0; l < 2; ++l) {
          const Rf x0 = px[i + l * N], x1 = px[ip + l * N], z0 = pz[i + l * N], z1 = pu[i + l * N];
          T dq = ((T)x1 - (T)x0) * dx1 + ((T)y[l + 1] - (T)y[l]) * dx2 + ((T)z1 - (T)z0) * dx3;
          z[l] = dq * usdtal;
          if (div_slots)
            dmax = fmax(dmax, fabs(((double)x1 - (double)x0) * g.dx1 + ((double)y[l + 1] - (double)y[l]) * g.dx2 + ((double)z1 - (double)z0) * g.dx3));
        }
      }
      v[a] = mkc<T>(z[0], z[1]);
    }
  }
  if (div_slots) block_max_to_slots(dmax, div_slots);
  __syncthreads();   // twiddles
  if (inA) stage_a<T, P, Q>(v, L.tw, b, false);
  exchange_ab<T, P, Q, NPB>(v, u, L, c, b, inA, d, kb, inB);
  if (inB) stage_b<T, P, Q>(u, L.tw, kb, false);   // u[k2] = Z[kb + P k2]
  // mirror bins Z[N-m] of the line pair through LDS, one component at a time;
  // a thread stores the bins kb + P k2 < n1hp, all but the last of them without
  // a test (the bin counts follow from N)
  constexpr int N1H = N / 2 + 1, N1HP = (N1H + 7) & ~7, KS = (N1HP + P - 1) / P;
  T* zs = L.ex + (inB ? d : 0) * N;
  T zrx[KS];
  __syncthreads();   // the exchange tile is read
  if (inB)
#pragma unroll
    for (int k2 = 0; k2 < Q; ++k2) zs[kb + P * k2] = u[k2].x;
  __syncthreads();
  if (inB)
#pragma unroll
    for (int k2 = 0; k2 < KS; ++k2) zrx[k2] = zs[k2 == 0 && kb == 0 ? 0 : N - kb - P * k2];
  __syncthreads();
  if (inB)
#pragma unroll
    for (int k2 = 0; k2 < Q; ++k2) zs[kb + P * k2] = u[k2].y;
  __syncthreads();
  if (!inB) return;
  cx<T>* out = S.spec + (size_t)N1HP * ((size_t)(jt * 2 * NPB) + (size_t)g.n2 * k);   // uniform; lanes at 32-bit offsets
  const int o = N1HP * 2 * d + kb;
#pragma unroll
  for (int k2 = 0; k2 < KS; ++k2) {
    const int m = kb + P * k2;
    if (P * k2 + P > N1HP && m >= N1HP) break;
    const cx<T> z = u[k2], zr = mkc<T>(zrx[k2], zs[k2 == 0 && kb == 0 ? 0 : N - m]);
    // A = (Z[m] + conj Z[N-m]) / 2,  B = (Z[m] - conj Z[N-m]) / (2i)
    cx<T> A = mkc<T>((z.x + zr.x) * T(0.5), (z.y - zr.y) * T(0.5));
    cx<T> B = mkc<T>((z.y + zr.y) * T(0.5), (zr.x - z.x) * T(0.5));
    if (P * k2 + P > N1H && m >= N1H) A = B = mkc<T>(0, 0);
    out[o + P * k2] = A;
    out[o + N1HP + P * k2] = B;
  }
}

// Z = A + iB of a line pair at bin m (FFTW c2r semantics as k_fft_x_bwd), the
// bins above N/2 as conj(A) + i conj(B) of the mirror bin; o: the pair's first
// bin, row: bins per line.  lo <= m <= hi are known at compile time, so which
// half a bin is in is only tested around N/2.
template <typename T, int N>
__device__ __forceinline__ cx<T> pair_bin(const cx<T>* __restrict__ in, int o, int row, int m, int lo, int hi) {
  const bool lower = hi <= N / 2 || (lo <= N / 2 && m <= N / 2);
  const int q = o + (lower ? m : N - m);
  cx<T> A = in[q], B = in[q + row];
  if (m == 0 || 2 * m == N) { A.y = T(0); B.y = T(0); }
  return lower ? mkc<T>(A.x - B.y, A.y + B.x) : mkc<T>(A.x + B.y, B.x - A.y);
}

// x pass, backward, with register FFTs: the line pairs' bins are packed
// (pair_bin) into the thread's order of the transform (in reverse from stage B
// for the square lengths, else from stage A), and line j comes from the real,
// line j+1 from the imaginary part.
template <typename Rf, typename T, int P, int Q>
__global__ __launch_bounds__(rf_threads(P, Q, x_pairs(P * Q))) void k_fft_x_bwd_reg(SpecArgs<T> S, const cx<T>* __restrict__ tw,
                                                                                    Rf* __restrict__ dst, const int* __restrict__ gate) {
  if (gate && *gate == 0) return;
  constexpr int N = P * Q, NPB = x_pairs(N), NT = rf_threads(P, Q, NPB), TB = NT / NPB;
  static_assert(N % (2 * NPB) == 0, "whole line pairs per block");
  __shared__ RegFftLds<T, P, Q, NPB> L;
  const Grid& g = S.g;
  const int t = threadIdx.x, b = t % TB, c = t / TB, kb = t % P, d = t / P;
  const bool inA = b < Q, inB = d < NPB;
  const unsigned blk = xcd_block(blockIdx.x, gridDim.x);
  const int ntj = g.n2 / (2 * NPB);
  const int j0 = (int)(blk % (unsigned)ntj) * 2 * NPB, k = (int)(blk / (unsigned)ntj);
  for (int q = t; q < N; q += NT) L.tw[q] = tw[q];
  constexpr int N1HP = (N / 2 + 8) & ~7;
  const cx<T>* in = S.spec + (size_t)N1HP * ((size_t)j0 + (size_t)g.n2 * k);   // uniform; lanes at 32-bit offsets
  Rf* out = dst + (size_t)N * ((size_t)j0 + (size_t)g.n2 * k);
  cx<T> v[P], u[Q];
  if constexpr (P == Q) {
    if (inB)
#pragma unroll
      for (int k2 = 0; k2 < Q; ++k2) u[k2] = pair_bin<T, N>(in, N1HP * 2 * d, N1HP, kb + P * k2, P * k2, P * k2 + P - 1);
    __syncthreads();   // twiddles
    if (inB) dft_twiddle<T, Q>(u, L.tw, kb, true);   // over k2: u[n1] = W_N^-(k1 n1) Z[k1 = kb][n1]
    exchange_ba<T, P, Q, NPB>(v, u, L, c, b, inA, d, kb, inB);
    if (!inA) return;
    dft_reg<T, P>(v, true);   // over k1: v[n2] = z[b + Q n2]
    const int o = N * 2 * c + b;
#pragma unroll
    for (int n2 = 0; n2 < P; ++n2) {
      out[o + Q * n2] = (Rf)v[n2].x;
      out[o + N + Q * n2] = (Rf)v[n2].y;
    }
  } else {
    if (inA)
#pragma unroll
      for (int a = 0; a < P; ++a) v[a] = pair_bin<T, N>(in, N1HP * 2 * c, N1HP, b + Q * a, Q * a, Q * a + Q - 1);
    __syncthreads();   // twiddles
    if (inA) stage_a<T, P, Q>(v, L.tw, b, true);
    exchange_ab<T, P, Q, NPB>(v, u, L, c, b, inA, d, kb, inB);
    if (!inB) return;
    stage_b<T, P, Q>(u, L.tw, kb, true);   // u[k2] = z[kb + P k2]
    const int o = N * 2 * d + kb;
#pragma unroll
    for (int k2 = 0; k2 < Q; ++k2) {
      out[o + P * k2] = (Rf)u[k2].x;
      out[o + N + P * k2] = (Rf)u[k2].y;
    }
  }
}

// Calls f(P, Q) (as integral constants) for a line length with a register FFT;
// false otherwise: shorter lines are bound by their launches either way, and
// 768 and 1024 points would hold 48 or more values a thread.
template <class F>
bool with_reg_fft(int n, F&& f) {
#define RF(NN, PP, QQ) case NN: f(std::integral_constant<int, PP>{}, std::integral_constant<int, QQ>{}); return true;
  switch (n) {
    RF(32, 4, 8) RF(48, 4, 12) RF(64, 8, 8) RF(96, 16, 6) RF(128, 16, 8) RF(192, 16, 12) RF(256, 16, 16) RF(384, 16, 24) RF(512, 16, 32)
    default: return false;
  }
#undef RF
}

bool make_plan(int N, FftPlan& P) {
  P.N = N;
  P.nst = 0;
  int m = N;
  while (m % 4 == 0) { P.radix[P.nst++] = 4; m /= 4; }
  while (m % 2 == 0) { P.radix[P.nst++] = 2; m /= 2; }
  while (m % 3 == 0) { P.radix[P.nst++] = 3; m /= 3; }
  return m == 1 && P.nst <= 24;
}

// Largest even divisor of n2 with (nl/2) * N1 complex values per tile.
int x_lines(int n1, int n2) {
  int cap = std::max(2, 2 * (FFT_EPT * FFT_NT) / n1);
  int best = 2;
  for (int d = 2; d <= std::min(cap, n2); d += 2)
    if (n2 % d == 0) best = d;
  return best;
}

}  // namespace

template <typename T>
int upload_twiddles(melt_ctx* ctx, int n, void** dst) {
  std::vector<cx<T>> h(n);
  for (int t = 0; t < n; ++t) {
    long double ang = 2.0L * 3.14159265358979323846264338327950288L * (long double)t / (long double)n;
    h[t].x = (T)cosl(ang);
    h[t].y = (T)-sinl(ang);
  }
  MELT_HIP(hipMalloc(dst, sizeof(cx<T>) * n));
  MELT_HIP(hipMemcpy(*dst, h.data(), sizeof(cx<T>) * n, hipMemcpyHostToDevice));
  return 0;
}

int poisson_init(melt_ctx* ctx) {
  int n[3] = {ctx->n1, ctx->n2, ctx->n3};
  void** tw[3] = {&ctx->tw1, &ctx->tw2, &ctx->tw3};
  double** ak[3] = {&ctx->ak1, &ctx->ak2, &ctx->ak3};
  double len[3] = {ctx->cfg.xlen, ctx->cfg.ylen, ctx->cfg.zlen};
  if (ctx->n2 % 2) return melt_fail(ctx, MELT_ERR_ARG, "poisson_init", "n2m must be even");
  for (int d = 0; d < 3; ++d) {
    FftPlan P;
    if (!make_plan(n[d], P)) return melt_fail(ctx, MELT_ERR_ARG, "poisson_init", "grid size must be 2^a 3^b");
    int rc = ctx->fp32 ? upload_twiddles<float>(ctx, n[d], tw[d]) : upload_twiddles<double>(ctx, n[d], tw[d]);
    if (rc) return rc;
    // phini.f90:35-55, 0-based index m -> reference index m+1
    std::vector<double> a(n[d]);
    int nm = n[d], nmh = nm / 2 + 1;
    for (int i = 1; i <= nm; ++i) {
      double ao = i <= nmh ? (double)(i - 1) * 2.0 * ctx->pi : -(double)(nm - i + 1) * 2.0 * ctx->pi;
      double r = (double)nm / len[d];
      a[i - 1] = 2.0 * (1.0 - cos(ao / nm)) * (r * r);
    }
    MELT_HIP(hipMalloc(ak[d], sizeof(double) * n[d]));
    MELT_HIP(hipMemcpy(*ak[d], a.data(), sizeof(double) * n[d], hipMemcpyHostToDevice));
  }
  size_t sz = 2 * ctx->esz * (size_t)ctx->n1hp * ctx->n2 * ctx->n3;
  MELT_HIP(hipMalloc(&ctx->spec, sz));
  MELT_HIP(hipMemset(ctx->spec, 0, sz));
  return 0;
}

// fused_divg = 1: dph := divergence / (al dt) is formed on the fly from the
// velocities (divg.f90) and never stored; 0: transforms MELT_DPH as phcalc.
// gate != null: every kernel returns at once unless *gate != 0 (the
// refinement solve of the precision form).  Rf is the field type, T the
// spectrum's (and the transforms' arithmetic).
template <typename Rf, typename T>
int solve_t(melt_ctx* ctx, int fused_divg, const int* gate, unsigned long long* div_slots) {
  SpecArgs<T> S;
  S.g = make_grid(ctx);
  S.n1h = ctx->n1h; S.n1hp = ctx->n1hp; S.spec = static_cast<cx<T>*>(ctx->spec);
  FftPlan Px, Py, Pz;
  make_plan(ctx->n1, Px); make_plan(ctx->n2, Py); make_plan(ctx->n3, Pz);
  const cx<T>* twx = static_cast<const cx<T>*>(ctx->tw1);
  const cx<T>* twy = static_cast<const cx<T>*>(ctx->tw2);
  const cx<T>* twz = static_cast<const cx<T>*>(ctx->tw3);
  hipEvent_t ev = nullptr;

  int nlx = x_lines(ctx->n1, ctx->n2);
  size_t shx = sizeof(cx<T>) * (size_t)(nlx / 2) * (ctx->n1 + 1);
  T usdtal = T(1.0 / (ctx->dt * ctx->al));
  unsigned gx = (unsigned)((ctx->n2 / nlx) * ctx->n3);
  const Rf* src = fused_divg ? nullptr : fld<Rf>(ctx, MELT_DPH);
  unsigned long long* dsl = fused_divg ? div_slots : nullptr;
  if (!gate) timing_begin(ctx, SLOT_DIVG_FFTX, &ev);
  if (!with_reg_fft(ctx->n1, [&](auto P, auto Q) {
        constexpr int p = decltype(P)::value, q = decltype(Q)::value, npb = x_pairs(p * q);
        hipLaunchKernelGGL((k_fft_x_fwd_reg<Rf, T, p, q>), dim3((unsigned)(ctx->n2 / (2 * npb) * ctx->n3)), dim3(x_fwd_threads(p, q)), 0,
                           ctx->stream, S, twx, fld<Rf>(ctx, MELT_VX), fld<Rf>(ctx, MELT_VY), fld<Rf>(ctx, MELT_VZ), src, usdtal, gate, dsl);
      }))
    hipLaunchKernelGGL((k_fft_x_fwd<Rf, T>), dim3(gx), dim3(FFT_NT), shx, ctx->stream, S, Px, twx, nlx, fld<Rf>(ctx, MELT_VX), fld<Rf>(ctx, MELT_VY),
                       fld<Rf>(ctx, MELT_VZ), src, usdtal, gate, dsl);
  MELT_HIP(hipGetLastError());
  if (!gate) timing_end(ctx, SLOT_DIVG_FFTX, ev);

  int nly = std::max(1, std::min(ctx->n1hp, (FFT_EPT * FFT_NT) / ctx->n2));
  size_t shy = sizeof(cx<T>) * (size_t)nly * ctx->n2;
  unsigned gy = (unsigned)(((ctx->n1hp + nly - 1) / nly) * ctx->n3);
  const unsigned gry = (unsigned)((ctx->n1hp / RF_NC) * ctx->n3), grz = (unsigned)((ctx->n1hp / RF_NC) * ctx->n2);
  auto fft_y = [&](auto inv) {
    if (!with_reg_fft(ctx->n2, [&](auto P, auto Q) {
          constexpr int p = decltype(P)::value, q = decltype(Q)::value;
          hipLaunchKernelGGL((k_fft_y_reg<T, p, q, decltype(inv)::value>), dim3(gry), dim3(rf_threads(p, q, RF_NC)), 0, ctx->stream, S, twy, gate);
        }))
      hipLaunchKernelGGL((k_fft_y<T>), dim3(gy), dim3(FFT_NT), shy, ctx->stream, S, Py, twy, nly, decltype(inv)::value ? 1 : 0, gate);
  };
  if (!gate) timing_begin(ctx, SLOT_FFTY, &ev);
  fft_y(std::false_type{});
  MELT_HIP(hipGetLastError());
  if (!gate) timing_end(ctx, SLOT_FFTY, ev);

  int nlz = std::max(1, std::min(ctx->n1hp, (FFT_EPT * FFT_NT) / ctx->n3));
  size_t shz = sizeof(cx<T>) * (size_t)nlz * ctx->n3;
  unsigned gz = (unsigned)(((ctx->n1hp + nlz - 1) / nlz) * ctx->n2);
  double nrm = (double)((long long)ctx->n1 * ctx->n2 * ctx->n3);
  if (!gate) timing_begin(ctx, SLOT_FFTZ_SOLVE, &ev);
  if (!with_reg_fft(ctx->n3, [&](auto P, auto Q) {
        constexpr int p = decltype(P)::value, q = decltype(Q)::value;
        hipLaunchKernelGGL((k_fft_z_solve_reg<T, p, q>), dim3(grz), dim3(rf_threads(p, q, RF_NC)), 0, ctx->stream, S, twz, ctx->ak1, ctx->ak2,
                           ctx->ak3, nrm, gate);
      }))
    hipLaunchKernelGGL((k_fft_z_solve<T>), dim3(gz), dim3(FFT_NT), shz, ctx->stream, S, Pz, twz, nlz, ctx->ak1, ctx->ak2, ctx->ak3, nrm, gate);
  MELT_HIP(hipGetLastError());
  if (!gate) timing_end(ctx, SLOT_FFTZ_SOLVE, ev);

  if (!gate) timing_begin(ctx, SLOT_IFFTY, &ev);
  fft_y(std::true_type{});
  MELT_HIP(hipGetLastError());
  if (!gate) timing_end(ctx, SLOT_IFFTY, ev);

  if (!gate) timing_begin(ctx, SLOT_IFFTX, &ev);
  if (!with_reg_fft(ctx->n1, [&](auto P, auto Q) {
        constexpr int p = decltype(P)::value, q = decltype(Q)::value, npb = x_pairs(p * q);
        hipLaunchKernelGGL((k_fft_x_bwd_reg<Rf, T, p, q>), dim3((unsigned)(ctx->n2 / (2 * npb) * ctx->n3)), dim3(rf_threads(p, q, npb)), 0,
                           ctx->stream, S, twx, fld<Rf>(ctx, MELT_DPH), gate);
      }))
    hipLaunchKernelGGL((k_fft_x_bwd<Rf, T>), dim3(gx), dim3(FFT_NT), shx, ctx->stream, S, Px, twx, nlx, fld<Rf>(ctx, MELT_DPH), gate);
  MELT_HIP(hipGetLastError());
  if (!gate) timing_end(ctx, SLOT_IFFTX, ev);
  return 0;
}

int poisson_solve(melt_ctx* ctx, int fused_divg, const int* gate, unsigned long long* div_slots) {
  return ctx->fp32 ? solve_t<float, float>(ctx, fused_divg, gate, div_slots) : solve_t<double, double>(ctx, fused_divg, gate, div_slots);
}
