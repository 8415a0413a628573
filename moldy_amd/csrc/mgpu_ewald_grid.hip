// Reciprocal-space Ewald sum on a grid (src/ewald.c:280-589): the
// same finite k set, weights and half-space sums as the direct sum, with the
// structure factors and the back-projection formed by spreading the charges
// over a grid with a compact window, transforming the grid, and dividing the
// window's transform out.
//
// The direct sums take N_k N_s complex products (1.3e10 at 132,872 sites);
// here a site meets w^3 grid points and the transforms cost about 4 n^3 (n/2)
// multiply-adds in all.  The k set is the direct path's, so nothing is
// truncated that the reference keeps: the window only approximates
// exp(i k.r), and its width is set so that the error lies at the rounding of
// the arithmetic (w = 16 in FP64, w = 8 in FP32; at least 4.6 and 4 grid
// points per shortest wave in each direction; the sampling theorem asks for 2).
//
//   window   phi(z) = exp(beta (sqrt(1 - z^2) - 1)), |z| <= 1, z = 2 d / w for a
//            grid distance d (the "exponential of semicircle" window of
//            Barnett, Magland and af Klinteberg, SIAM J. Sci. Comput. 41, C479,
//            2019).  beta = 2.6 w (FP64) and 2.7 w (FP32): past their 2.3 w,
//            because the Ewald weight exp(-k^2/4 alpha^2) damps the k next to
//            the cutoff, whose aliases a larger beta raises, while the
//            window's jump at its edge falls.  Its own error in the forces
//            of 4,054 salt water sites (all else in long double): 1.5e-15 at
//            2.5 w, 4e-16 at 2.6 w, 5e-16 at 2.65 w; for FP32 2.9e-7 at 2.6 w,
//            1.4e-7 at 2.7 w, 1.1e-7 at 2.75 w (1.2e-7 and rising in silica).
//            It is evaluated as one polynomial per grid offset.
//   spread   G(x,y,z) = sum_i q_i phi phi phi
//   forward  T(h,k,l) = sum_xyz G e^{+2 pi i (hx/nx + ky/ny + lz/nz)}, l >= 0, as
//            dense transforms of one axis at a time on the matrix cores: only the
//            modes of the k set's box are formed (a quarter of each axis), so
//            the dense form costs about what a full FFT would
//   k space  S = T / (phi^ phi^ phi^); energy, stress (ewald.c:539-553); W = coeff S / (phi^ phi^ phi^)
//   inverse  Phi(x,y,z) = Re sum W e^{-2 pi i (...)}
//   gather   F_i = -q_i grad sum_g Phi(g) phi phi phi, the gradient of the window's polynomials
//
// The transforms (and the window's polynomials) run in FP64 for both: in FP32
// the transforms' rounding alone made an error of 9.5e-7 in the forces of 729
// waters (4e-7 for all else), because the sums
// over the grid cancel; they are a small part of the pass.
//
// Every sum has a fixed order (a brick's sites are ranked by index before
// they are added), so results repeat bit for bit.
#include "mgpu_internal.h"
#include "mgpu_ewald_grid.h"

#include <algorithm>
#include <cmath>

using namespace mgpu;

namespace {

constexpr double PI_D = 3.14159265358979323846;
constexpr int GB = 8;               // brick edge in grid points

// Window width and polynomial degree of each arithmetic.
template <class R> struct Win;
template <> struct Win<double> {
   static constexpr int W = 16, DEG = 15;
   static constexpr double BETA = 2.6 * W;
};
template <> struct Win<float> {
   static constexpr int W = 8, DEG = 10;
   static constexpr double BETA = 2.7 * W;
};
// A site's spread weights: three rows of W + 2, a zero at either end for every
// grid point outside the window.
template <class R> constexpr int WROW = Win<R>::W + 2;

typedef double dbl4 __attribute__((ext_vector_type(4)));
// 16x16x4 matrix product: A row (B column) lane % 16 at k = lane / 16; item v
// of D is row lane / 16 + 4 v of column lane % 16.
__device__ __forceinline__ dbl4 mma(double a, double b, dbl4 c) {
   return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
template <class R> struct Vec;
template <> struct Vec<double> {
   using T2 = double2;
};
template <> struct Vec<float> {
   using T2 = float2;
};

// The wave's own LDS writes before its reads.
__device__ __forceinline__ void wave_lds_sync() {
   __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
   __builtin_amdgcn_wave_barrier();
   __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ------------------------------------------------------------ binning
struct GBinArgs {
   double hinv[9];
   int n[3], nb[3];      // grid points, bricks
   int ns, nsp, w, cap;
   const double *site;
   int4 *sa;             // per site: anchor (first grid point of the window, wrapped) and brick
   double *sx;           // per site: polynomial argument per axis, [3][nsp]
   int *cnt, *bucket;    // per brick: sites seen; [brick][cap] the first cap of them
};

// Anchor a = ceil(u - w/2) and the polynomials' argument 2 (a - (u - w/2)) - 1
// of each axis, u the grid coordinate; sites counted into the bricks of
// their anchors.  The fractional coordinate is formed as a sum of two doubles
// and the argument with one fma from the anchor: the position within the
// window then carries no rounding of the size of the box (which would be a
// phase error growing with |h|, as the trig recurrence of the direct sum has).
__device__ __forceinline__ void b_g_bin(int bx, int nbx, const GBinArgs &a) {
#pragma clang fp contract(off)
   const int i = bx * 256 + threadIdx.x;
   if (i >= a.ns) return;
   const double r[3] = {a.site[i], a.site[a.nsp + i], a.site[2 * (size_t)a.nsp + i]};
   int an[3];
#pragma unroll
   for (int d = 0; d < 3; d++) {
      double hi = 0, lo = 0;
#pragma unroll
      for (int c = 0; c < 3; c++) {
         const double p = a.hinv[3 * d + c] * r[c];
         lo += __builtin_fma(a.hinv[3 * d + c], r[c], -p);
         const double t = hi + p, z = t - hi;
         lo += (hi - (t - z)) + (p - z);
         hi = t;
      }
      hi -= rint(hi);
      // a coordinate that is not finite is put into the origin's brick, and its
      // argument stays NaN: its weights, and with them all sums, are NaN then,
      // as the direct sum's are
      const double n = a.n[d], hw = 0.5 * a.w, c = ceil(__builtin_fma(n, fabs(hi) <= 0.5 ? hi : 0.0, -hw));
      an[d] = (int)c;
      if (an[d] < 0) an[d] += a.n[d];
      a.sx[(size_t)d * a.nsp + i] = 2.0 * (__builtin_fma(-n, hi, c + hw) - n * lo) - 1.0;
   }
   const int b = ((an[0] / GB) * a.nb[1] + an[1] / GB) * a.nb[2] + an[2] / GB;
   a.sa[i] = make_int4(an[0], an[1], an[2], b);
   const int slot = atomicAdd(&a.cnt[b], 1);
   if (slot < a.cap) a.bucket[(size_t)b * a.cap + slot] = i;
}
__global__ __launch_bounds__(256) void k_g_bin(GBinArgs a) { b_g_bin(blockIdx.x, gridDim.x, a); }

// Exclusive prefix sum of the brick counts, one block.
__device__ __forceinline__ void b_g_scan(int bx, int nbx, int nb, const int *__restrict__ cnt,
                                         int *__restrict__ start) {
   __shared__ int ws[4];
   const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
   const int per = (nb + 255) / 256, b0 = min(t * per, nb), b1 = min(b0 + per, nb);
   int s = 0;
   for (int b = b0; b < b1; b++) s += cnt[b];
   const int inc = wave_incl_scan(s, lane);
   if (lane == 63) ws[wv] = inc;
   __syncthreads();
   int off = inc - s;
   for (int q = 0; q < wv; q++) off += ws[q];
   for (int b = b0; b < b1; b++) {
      start[b] = off;
      off += cnt[b];
   }
   if (t == 255) start[nb] = off;
}
__global__ __launch_bounds__(256) void k_g_scan(int nb, const int *__restrict__ cnt, int *__restrict__ start) {
   b_g_scan(blockIdx.x, gridDim.x, nb, cnt, start);
}

// ------------------------------------------------------------ weights
struct GWtArgs {
   int nb, ns, nsp, cap;
   const int4 *sa;
   const double *sx, *chg;
   const int *bucket, *start;
   int *cnt;             // cleared for the next pass
   const double *poly;   // [DEG + 1][W]
   void *wt;             // R [ns][3][W + 2]
   int4 *anc;            // brick order: anchor and site index
   double4 *fr;          // [ns]: arguments and charge
};

// One wave per brick: its sites in index order, each with its anchor,
// arguments and spread weights (the charge in the x row).  A brick with more
// than cap sites collects them by a walk over all sites.
template <class R>
__device__ __forceinline__ void b_g_weights(int bx, int nbx, const GWtArgs &a) {
   constexpr int W = Win<R>::W, DEG = Win<R>::DEG, WR = WROW<R>, NL = 3 * WR;
   extern __shared__ double gw_lds[];
   const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
   const int b = bx * 4 + wave;
   if (b >= a.nb) return;   // wave-uniform; no block barrier in this kernel
   double *xs = gw_lds + wave * 4 * a.cap;                  // the ranked sites' arguments and charges
   int *list = (int *)(gw_lds + 16 * a.cap) + wave * a.cap;
   const int m = a.cnt[b], s0 = a.start[b];
   // lanes d WR + 1 + p: the polynomial of offset p on axis d
   double c[DEG + 1];
   const int wd = min(lane / WR, 2), wp = lane % WR - 1;
#pragma unroll
   for (int k = 0; k <= DEG; k++) c[k] = lane < NL && wp >= 0 && wp < W ? a.poly[k * W + wp] : 0.0;
   auto place = [&](int i, int pos) {
      const int4 s = a.sa[i];
      a.anc[pos] = make_int4(s.x, s.y, s.z, i);
      const double4 f = make_double4(a.sx[i], a.sx[(size_t)a.nsp + i], a.sx[2 * (size_t)a.nsp + i], a.chg[i]);
      a.fr[pos] = f;
      return f;
   };
   auto weights = [&](double x, double q, int pos) {
      double v = c[DEG];
#pragma unroll
      for (int k = DEG - 1; k >= 0; k--) v = v * x + c[k];
      if (wd == 0) v *= q;
      if (lane < NL) ((R *)a.wt)[(size_t)pos * NL + lane] = (R)v;
   };
   if (m <= a.cap) {
      for (int t = lane; t < m; t += 64) list[t] = a.bucket[(size_t)b * a.cap + t];
      wave_lds_sync();
      for (int t = lane; t < m; t += 64) {
         const int i = list[t];
         int r = 0;
         for (int q = 0; q < m; q++) r += list[q] < i;
         const double4 f = place(i, s0 + r);
         xs[4 * r] = f.x;
         xs[4 * r + 1] = f.y;
         xs[4 * r + 2] = f.z;
         xs[4 * r + 3] = f.w;
      }
      wave_lds_sync();
      for (int t = 0; t < m; t++) weights(xs[4 * t + wd], xs[4 * t + 3], s0 + t);
   } else {
      int r = 0;
      for (int i0 = 0; i0 < a.ns; i0 += 64) {
         const int i = i0 + lane;
         const bool in = i < a.ns && a.sa[i].w == b;
         unsigned long long mk = __ballot(in);
         if (in) place(i, s0 + r + __popcll(mk & ((1ull << lane) - 1)));
         for (; mk; mk &= mk - 1, r++) {
            const int j = i0 + __builtin_ctzll(mk);
            weights(a.sx[(size_t)wd * a.nsp + j], a.chg[j], s0 + r);
         }
      }
   }
   if (lane == 0) a.cnt[b] = 0;
}
template <class R> __global__ __launch_bounds__(256) void k_g_weights(GWtArgs a) {
   b_g_weights<R>(blockIdx.x, gridDim.x, a);
}

// ------------------------------------------------------------ spread
struct GSpArgs {
   int n[3], nb[3];
   int ntz, per;         // z tiles of 16, blocks of each XCD
};

typedef float flt4 __attribute__((ext_vector_type(4)));
template <class R> struct SpM;
template <> struct SpM<double> {
   using V = dbl4;
   static __device__ __forceinline__ V mul(double a, double b, V c) { return mma(a, b, c); }
   static __device__ __forceinline__ int row(int g, int v) { return g + 4 * v; }
};
template <> struct SpM<float> {
   using V = flt4;
   static __device__ __forceinline__ V mul(float a, float b, V c) {
      return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
   }
   static __device__ __forceinline__ int row(int g, int v) { return 4 * g + v; }
};

// What bounds it: the matrix cores (the tiles of 8 x 8 x 16 multiply 4.5 times the
// points the windows hold; 42% of their FP64 peak) and the operands' addresses.
// 132,872 sites: 175 us FP64, 44 us FP32 (450 and 206 with one site a wave at a
// time, its x weights as scalar loads: scalar issue bound it).
// One block per tile of 8 x 8 x 16 grid points, as a product over the sites
// whose windows reach it: rows (x, y) with q wx wy, columns z with wz, four
// sites a step (lane / 16), four row tiles of 16.  Those sites have their
// anchors in the 3 (W = 16) or 2 (W = 8) bricks per axis up to the tile's (one
// more in z), each row of bricks along z one run of the brick-ordered sites, two
// where it wraps; the four waves take every fourth group of four.  Weights are
// read one group ahead.
template <class R>
__device__ __forceinline__ void b_g_spread(int bx, int nbx, const GSpArgs &a, const R *__restrict__ wt,
                                           const int4 *__restrict__ anc, const int *__restrict__ start,
                                           R *__restrict__ G) {
   constexpr int W = Win<R>::W, WR = WROW<R>, NK = W > GB + 1 ? 3 : 2, NR = NK * NK * 2;
   using V = typename SpM<R>::V;
   __shared__ R red[4][1024];
   const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
   const int m = lane & 15, g = lane >> 4;
   const int nby = a.nb[1], nbz = a.nb[2];
   const int t = (bx & 7) * a.per + (bx >> 3);
   if (t >= a.nb[0] * nby * a.ntz) return;   // block-uniform, before any barrier
   const int Bx = t / (nby * a.ntz), By = t / a.ntz - nby * Bx, Tz = t - a.ntz * (By + nby * Bx);
   // run r = (x brick, y brick, wrapped part): lane r holds its sites and its
   // tile origin less the image shift, per axis
   int rs = 0, re = 0, ox = 0, oy = 0, oz = 0;
   if (lane < NR) {
      const int q = lane >> 1, wrap = lane & 1;
      int cx = Bx - q / NK, cy = By - q % NK;
      ox = GB * Bx;
      oy = GB * By;
      oz = 2 * GB * Tz;
      if (cx < 0) {
         cx += a.nb[0];
         ox += a.n[0];
      }
      if (cy < 0) {
         cy += nby;
         oy += a.n[1];
      }
      const int zlo = 2 * Tz - (NK - 1), zhi = min(2 * Tz + 2, nbz);   // bricks [zlo, zhi)
      int z0 = max(zlo, 0), z1 = zhi;
      if (wrap) {
         z0 = zlo + nbz;
         z1 = zlo < 0 ? nbz : z0;
         oz += a.n[2];
      }
      const int cb = (cx * nby + cy) * nbz;
      rs = z1 > z0 ? start[cb + z0] : 0;
      re = z1 > z0 ? start[cb + z1] : 0;
   }
   V acc[4];
#pragma unroll
   for (int c = 0; c < 4; c++) acc[c] = V{0, 0, 0, 0};
   int r = -1, base = 0, end = 0, rx = 0, ry = 0, rz = 0;
   auto next = [&]() {   // the wave's next group of sites; false past the last run
      base += 16;
      while (base >= end) {
         if (++r == NR) return false;
         base = __builtin_amdgcn_readlane(rs, r) + 4 * wave;
         end = __builtin_amdgcn_readlane(re, r);
      }
      rx = __builtin_amdgcn_readlane(ox, r);
      ry = __builtin_amdgcn_readlane(oy, r);
      rz = __builtin_amdgcn_readlane(oz, r);
      return true;
   };
   // a group's anchors are loaded two groups ahead, its weights one
   struct Op {
      R wx[4], wy, wz;
   };
   int4 A = make_int4(0, 0, 0, 0);
   int jc = 0, px = 0, py = 0, pz = 0;
   auto fetch_anchor = [&]() {
      const int j = base + g;
      jc = min(j, end - 1);                       // a group holds at least one site
      px = rx + (m >> 3);
      py = ry + (m & 7);
      pz = j < end ? rz + m : -(1 << 20);          // off the window: no weight
      A = anc[jc];
   };
   auto fetch = [&](Op &o) {
      const R *w = wt + (size_t)jc * (3 * WR) + 1;
      const int dx = px - A.x;
      o.wy = w[WR + min(max(py - A.y, -1), W)];
      o.wz = w[2 * WR + min(max(pz - A.z, -1), W)];
#pragma unroll
      for (int c = 0; c < 4; c++) o.wx[c] = w[min(max(dx + 2 * c, -1), W)];
   };
   bool have = next(), more = false;
   Op P, Q;
   if (have) {
      fetch_anchor();
      fetch(P);
      more = next();
      if (more) fetch_anchor();
   }
   auto step = [&](const Op &o, Op &ahead) {
      R av[4];
#pragma unroll
      for (int c = 0; c < 4; c++) av[c] = o.wx[c] * o.wy;
      have = more;
      if (have) {
         fetch(ahead);
         more = next();
         if (more) fetch_anchor();
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = 0; c < 4; c++) acc[c] = SpM<R>::mul(av[c], o.wz, acc[c]);
   };
   while (have) {
      step(P, Q);
      if (!have) break;
      step(Q, P);
   }
   // row of tile c: x = 2 c + row / 8, y = row % 8
#pragma unroll
   for (int c = 0; c < 4; c++)
#pragma unroll
      for (int v = 0; v < 4; v++) red[wave][(16 * c + SpM<R>::row(g, v)) * 16 + m] = acc[c][v];
   __syncthreads();
   const int z = 2 * GB * Tz + m;
   if (z < a.n[2])
      for (int q = threadIdx.x >> 4; q < 64; q += 16) {
         const int o = q * 16 + m;
         const int x = GB * Bx + (q >> 3), y = GB * By + (q & 7);
         G[((size_t)x * a.n[1] + y) * a.n[2] + z] = ((red[0][o] + red[1][o]) + red[2][o]) + red[3][o];
      }
}
template <class R>
__global__ __launch_bounds__(256) void k_g_spread(GSpArgs a, const R *__restrict__ wt, const int4 *__restrict__ anc,
                                                  const int *__restrict__ start, R *__restrict__ G) {
   b_g_spread<R>(blockIdx.x, gridDim.x, a, wt, anc, start, G);
}

// ------------------------------------------------------------ transforms
struct GzArgs {
   int nlines, K, lda;        // rows of the input, its K and row stride (elements)
   int ncols, ldt, ldo;       // columns out, table row stride, output row stride
   int nmt, ngrp;             // row tiles, column groups
};

// out[line][col] = sum_k in[line][k] tab[k][col]: the z transforms, both
// ways.  A wave takes 16 lines by NT column tiles; lane (row, g) reads
// elements 2 g, 2 g + 1 of each 8 (the table's rows taken alike).  The table
// has zero rows up to a multiple of 8 and zero columns up to whole groups.
template <class RI, class RO, int NT>
__device__ __forceinline__ void b_gz(int bx, int nbx, const GzArgs &a, const RI *__restrict__ in,
                                     const double *__restrict__ tab, RO *__restrict__ out) {
   using T2 = typename Vec<RI>::T2;
   const int lane = threadIdx.x & 63, m = lane & 15, g = lane >> 4;
   const int t = bx * 4 + (threadIdx.x >> 6);
   if (t >= a.nmt * a.ngrp) return;
   const int mt = t / a.ngrp, c0 = (t - mt * a.ngrp) * NT * 16 + m;
   const RI *ap = in + (size_t)min(mt * 16 + m, a.nlines - 1) * a.lda;
   dbl4 acc[NT];
#pragma unroll
   for (int c = 0; c < NT; c++) acc[c] = dbl4{0, 0, 0, 0};
   // operands one step ahead (past the end: the last step's again)
   struct Op {
      T2 a;
      double b0[NT], b1[NT];
   };
   const int klast = (a.K + 7) / 8 * 8 - 8;
   auto load = [&](Op &o, int k0) {
      const int k = min(k0, klast) + 2 * g;
      o.a = *(const T2 *)(ap + min(k, a.K - 2));   // K is even
      const double *tp = tab + (size_t)k * a.ldt + c0;
#pragma unroll
      for (int c = 0; c < NT; c++) {
         o.b0[c] = tp[16 * c];
         o.b1[c] = tp[a.ldt + 16 * c];
      }
   };
   auto step = [&](const Op &o) {
#pragma unroll
      for (int c = 0; c < NT; c++) {
         acc[c] = mma(o.a.x, o.b0[c], acc[c]);
         acc[c] = mma(o.a.y, o.b1[c], acc[c]);
      }
   };
   Op p, q;
   load(p, 0);
   for (int k0 = 0; k0 <= klast; k0 += 16) {
      load(q, k0 + 8);
      __builtin_amdgcn_sched_barrier(0);
      step(p);
      load(p, k0 + 16);
      __builtin_amdgcn_sched_barrier(0);
      if (k0 + 8 <= klast) step(q);
   }
#pragma unroll
   for (int v = 0; v < 4; v++) {
      const int line = mt * 16 + g + 4 * v;
      if (line >= a.nlines) continue;
#pragma unroll
      for (int c = 0; c < NT; c++)
         if (c0 + 16 * c < a.ncols) out[(size_t)line * a.ldo + c0 + 16 * c] = (RO)acc[c][v];
   }
}
template <class RI, class RO, int NT>
__global__ __launch_bounds__(256) void k_gz(GzArgs a, const RI *__restrict__ in, const double *__restrict__ tab,
                                            RO *__restrict__ out) {
   b_gz<RI, RO, NT>(blockIdx.x, gridDim.x, a, in, tab, out);
}

struct GcArgs {
   int nbatch, nmt, nct;             // batches, row tiles, column tiles
   int K, M, N, ldt;                 // contraction length, rows with an image, columns, table row stride
   int off, qoff, mq;                // output index of row m: off + m, and qoff - m for 0 < m < mq
   size_t inb, ink, inc, outb, outm, outc;
};

// out[b][index(m)][n] = sum_k E[m][k] in[b][k][n] over complex planes (real at
// 0, imaginary at inc / outc), with the mirrored row conj(E[m]) from the same
// four real products: the x and y transforms, both ways.  A wave takes one
// 16 x 16 tile.
__device__ __forceinline__ void b_gc(int bx, int nbx, const GcArgs &a, const double *__restrict__ in,
                                     const double *__restrict__ er, const double *__restrict__ ei, double *__restrict__ out) {
   const int lane = threadIdx.x & 63, m = lane & 15, g = lane >> 4;
   const int t = bx * 4 + (threadIdx.x >> 6);
   if (t >= a.nbatch * a.nmt * a.nct) return;
   const int b = t / (a.nmt * a.nct), r = t - b * (a.nmt * a.nct), ct = r / a.nmt, mt = r - ct * a.nmt;
   const int n = ct * 16 + m;
   const double *ip = in + b * a.inb + min(n, a.N - 1);
   const double *rp = er + mt * 16 + m, *xp = ei + mt * 16 + m;
   dbl4 rr{0, 0, 0, 0}, ii{0, 0, 0, 0}, ri{0, 0, 0, 0}, ir{0, 0, 0, 0};
   // operands of eight k, one step ahead (past the end: the last step's again)
   struct Op {
      double br[2], bi[2], ar[2], ai[2];
   };
   const int klast = (a.K + 7) / 8 * 8 - 8;
   auto load = [&](Op &o, int k0) {
#pragma unroll
      for (int u = 0; u < 2; u++) {
         const int k = min(k0, klast) + 4 * u + g, kc = min(k, a.K - 1);   // the table's rows past K are zero
         o.br[u] = ip[kc * a.ink];
         o.bi[u] = ip[kc * a.ink + a.inc];
         o.ar[u] = rp[(size_t)k * a.ldt];
         o.ai[u] = xp[(size_t)k * a.ldt];
      }
   };
   auto step = [&](const Op &o) {
#pragma unroll
      for (int u = 0; u < 2; u++) {
         rr = mma(o.ar[u], o.br[u], rr);
         ii = mma(o.ai[u], o.bi[u], ii);
         ri = mma(o.ar[u], o.bi[u], ri);
         ir = mma(o.ai[u], o.br[u], ir);
      }
   };
   Op p, q;
   load(p, 0);
   for (int k0 = 0; k0 <= klast; k0 += 16) {
      load(q, k0 + 8);
      __builtin_amdgcn_sched_barrier(0);
      step(p);
      load(p, k0 + 16);
      __builtin_amdgcn_sched_barrier(0);
      if (k0 + 8 <= klast) step(q);
   }
   if (n >= a.N) return;
#pragma unroll
   for (int v = 0; v < 4; v++) {
      const int mm = mt * 16 + g + 4 * v;
      if (mm >= a.M) continue;
      double *o = out + b * a.outb + (size_t)(a.off + mm) * a.outm + n;
      o[0] = rr[v] - ii[v];
      o[a.outc] = ri[v] + ir[v];
      if (mm > 0 && mm < a.mq) {
         o = out + b * a.outb + (size_t)(a.qoff - mm) * a.outm + n;
         o[0] = rr[v] + ii[v];
         o[a.outc] = ri[v] - ir[v];
      }
   }
}
__global__ __launch_bounds__(256) void k_gc(GcArgs a, const double *__restrict__ in, const double *__restrict__ er,
                                            const double *__restrict__ ei, double *__restrict__ out) {
   b_gc(blockIdx.x, gridDim.x, a, in, er, ei, out);
}

// ------------------------------------------------------------ k space
struct GkArgs {
   int hmax, kmax, lmax;
   double vol, r4a, c2;
   const KRow *rows;
   const int *rowmap;              // [hmax + 1][2 kmax + 1]: row of (h, k) or -1
   const double *dx, *dy, *dz;     // 1 / phi^ per |h|, |k|, |l|
   double *bpart;                  // [blocks][8]
};

// Per mode (h, k, l >= 0): energy and stress of the k vector it stands for
// (itself, or its inverse where the half-space set holds that), and the
// weight of the inverse transform in its place; modes outside the set become
// zero.
__device__ __forceinline__ void b_gk(int bx, int nbx, const GkArgs &a, double *__restrict__ T) {
   __shared__ double ws[4][8];
   const int L = a.lmax + 1, NKk = 2 * a.kmax + 1, P = NKk * L;
   const int e = bx * 256 + threadIdx.x;
   double v[7] = {0, 0, 0, 0, 0, 0, 0};
   if (e < (2 * a.hmax + 1) * P) {
      const int hs = e / P, q = e - hs * P, ks = q / L, l = q - ks * L, h = hs - a.hmax;
      int r = h >= 0 ? a.rowmap[h * NKk + ks] : -1, ll = l;
      if (r >= 0 && !(l >= a.rows[r].l0 && l < a.rows[r].l0 + a.rows[r].nl)) r = -1;
      if (r < 0 && l > 0 && h <= 0) {
         r = a.rowmap[-h * NKk + 2 * a.kmax - ks];
         ll = -l;
         if (r >= 0 && !(ll >= a.rows[r].l0 && ll < a.rows[r].l0 + a.rows[r].nl)) r = -1;
      }
      double *p = T + (size_t)hs * 2 * P + q;
      double wr = 0, wi = 0;
      if (r >= 0) {
         const KRow Q = a.rows[r];
         const double dec = a.dx[h < 0 ? -h : h] * a.dy[ks < a.kmax ? a.kmax - ks : ks - a.kmax] * a.dz[l];
         const double c = dec * p[0], s = dec * p[P];
         const double kx = Q.kx, ky = Q.ky, kz = Q.kzt + ll * a.c2;
         const double ksq = kx * kx + ky * ky + kz * kz;
         const double coeff = 2.0 / ((0.25 / PI_D) * a.vol) * exp(ksq * a.r4a) / ksq;
         const double coeff2 = 2.0 * (1.0 - ksq * a.r4a) / ksq;
         const double pe_k = 0.5 * coeff * (c * c + s * s);
         v[0] = pe_k;
         v[1] = pe_k - pe_k * coeff2 * kx * kx;
         v[2] = -pe_k * coeff2 * kx * ky;
         v[3] = -pe_k * coeff2 * kx * kz;
         v[4] = pe_k - pe_k * coeff2 * ky * ky;
         v[5] = -pe_k * coeff2 * ky * kz;
         v[6] = pe_k - pe_k * coeff2 * kz * kz;
         wr = coeff * dec * c;
         wi = coeff * dec * s;
      }
      p[0] = wr;
      p[P] = wi;
   }
   const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
   for (int q = 0; q < 7; q++) {
      const double t = wave_sum(v[q]);
      if (lane == 0) ws[wv][q] = t;
   }
   __syncthreads();
   if (threadIdx.x < 8)
      a.bpart[8 * (size_t)bx + threadIdx.x] =
          threadIdx.x == 7 ? 0.0
                           : ws[0][threadIdx.x] + ws[1][threadIdx.x] + ws[2][threadIdx.x] + ws[3][threadIdx.x];
}
__global__ __launch_bounds__(256) void k_gk(GkArgs a, double *__restrict__ T) {
   b_gk(blockIdx.x, gridDim.x, a, T);
}

// ------------------------------------------------------------ gather
struct GGaArgs {
   int n[3], nb[3];
   int ntz, per;         // z tiles, blocks of each XCD
   double m[9];          // force = q sum_d G_d m[d]: 2 n_d hinv[d]
   int nsp, add;         // add: accumulate into out
};
// Anchors per tile: 8 x 8 x GaT::TZ; the grid points their windows meet are
// staged in LDS, RX x RX rows of RZ (a power of two).
template <class R> struct GaT;
template <> struct GaT<double> {
   static constexpr int TZ = 16, RX = 23, RZ = 32, NW = 16;
};
template <> struct GaT<float> {
   static constexpr int TZ = 8, RX = 15, RZ = 16, NW = 4;
};

// What bounds it: LDS reads in FP64 (32 KB a site) and the chain of one site
// (polynomials, window, wave sum).  132,872 sites: 230 us FP64, 57 us FP32 (331 and 78
// reading the grid from L2).
// One block per tile of anchors: the tile's sites are one run of the
// brick-ordered sites, and every grid point their windows meet is read once
// into LDS (read per site, a site's window of 2 x 128-byte lines a row is 64 KB
// from L2 in FP64, 8.7 GB at 132,872 sites).  A wave per site in turn: a lane
// holds a (y, z) of the window and walks x; the weights and their derivatives
// come from one polynomial a lane through LDS.  Rows are turned by W elements
// (every second one in FP64, second four in FP32) so that the rows a wave reads
// together lie on different banks.
template <class R>
__device__ __forceinline__ void b_g_gather(int bx, int nbx, const GGaArgs &a, const R *__restrict__ G,
                                           const double *__restrict__ poly, const int4 *__restrict__ anc,
                                           const double4 *__restrict__ fr, const int *__restrict__ start,
                                           double *__restrict__ out) {
   constexpr int W = Win<R>::W, DEG = Win<R>::DEG, NL = 3 * W, LY = 64 / W, NJ = W / LY;
   constexpr int TZ = GaT<R>::TZ, RX = GaT<R>::RX, RZ = GaT<R>::RZ, NW = GaT<R>::NW, YS = W == 16 ? 0 : 2;
   using T2 = typename Vec<R>::T2;
   __shared__ R sg[RX * RX * RZ];
   __shared__ T2 sv[NW][NL];
   const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
   const int wd = lane / W, wp = lane % W;
   const int t = (bx & 7) * a.per + (bx >> 3);
   if (t >= a.nb[0] * a.nb[1] * a.ntz) return;   // block-uniform, before any barrier
   const int Bx = t / (a.nb[1] * a.ntz), By = t / a.ntz - a.nb[1] * Bx, Tz = t - a.ntz * (By + a.nb[1] * Bx);
   const int cb = (Bx * a.nb[1] + By) * a.nb[2];
   const int s0 = start[cb + Tz * (TZ / GB)], s1 = start[cb + min((Tz + 1) * (TZ / GB), a.nb[2])];
   if (s1 == s0) return;   // block-uniform
   {
      const int z = threadIdx.x % RZ;
      int zz = TZ * Tz + z;
      if (zz >= a.n[2]) zz -= a.n[2];
      if (z < TZ + W - 1) {
#pragma unroll
         for (int u = 0; u < (RX * RX * RZ + 64 * NW - 1) / (64 * NW); u++) {
            const int r = threadIdx.x / RZ + u * (64 * NW / RZ);
            if (r >= RX * RX) break;
            int xx = GB * Bx + r / RX, yy = GB * By + r % RX;
            if (xx >= a.n[0]) xx -= a.n[0];
            if (yy >= a.n[1]) yy -= a.n[1];
            sg[r * RZ + ((z + W * (((r % RX) >> YS) & 1)) & (RZ - 1))] = G[((size_t)xx * a.n[1] + yy) * a.n[2] + zz];
         }
      }
   }
   double c[DEG + 1];
#pragma unroll
   for (int k = 0; k <= DEG; k++) c[k] = lane < NL ? poly[k * W + wp] : 0.0;
   int4 An = anc[min(s0 + wave, s1 - 1)];
   double4 fn = fr[min(s0 + wave, s1 - 1)];
   __syncthreads();
   for (int pos = s0 + wave; pos < s1; pos += NW) {   // wave-uniform
      const int4 A = An;
      const double4 f = fn;
      An = anc[min(pos + NW, s1 - 1)];
      fn = fr[min(pos + NW, s1 - 1)];
      const double x = wd == 0 ? f.x : wd == 1 ? f.y : f.z;
      double v = c[DEG], dv = 0;
#pragma unroll
      for (int k = DEG - 1; k >= 0; k--) {
         dv = dv * x + v;
         v = v * x + c[k];
      }
      wave_lds_sync();
      if (lane < NL) {
         T2 w;
         w.x = (R)v;
         w.y = (R)dv;
         sv[wave][lane] = w;
      }
      wave_lds_sync();
      const int lx = A.x - GB * Bx, lz = A.z - TZ * Tz + wp;
      const R *gp[NJ];
#pragma unroll
      for (int j = 0; j < NJ; j++) {
         const int y = A.y - GB * By + j * LY + wd;
         gp[j] = sg + (lx * RX + y) * RZ + ((lz + W * ((y >> YS) & 1)) & (RZ - 1));
      }
      // FP32: the grid less its value at the window's middle, whose force is zero:
      // the potential (the site's own charge's for the most part) changes by a
      // fifth over the window, and the weights' rounding meets only that
      R mid = 0;
      if constexpr (sizeof(R) == 4) {
         const int y = A.y - GB * By + W / 2, z = A.z - TZ * Tz + W / 2;
         mid = sg[((lx + W / 2) * RX + y) * RZ + ((z + W * ((y >> YS) & 1)) & (RZ - 1))];
      }
      R a0[NJ], a1[NJ];
#pragma unroll
      for (int j = 0; j < NJ; j++) a0[j] = a1[j] = 0;
#pragma unroll
      for (int i = 0; i < W; i++) {
         const T2 wx = sv[wave][i];
#pragma unroll
         for (int j = 0; j < NJ; j++) {
            R gv = gp[j][i * RX * RZ];
            if constexpr (sizeof(R) == 4) gv -= mid;
            a0[j] += wx.x * gv;
            a1[j] += wx.y * gv;
         }
      }
      double px = 0, py = 0, p0 = 0;
#pragma unroll
      for (int j = 0; j < NJ; j++) {
         const T2 wy = sv[wave][W + j * LY + wd];
         px += (double)wy.x * (double)a1[j];
         py += (double)wy.y * (double)a0[j];
         p0 += (double)wy.x * (double)a0[j];
      }
      const T2 wz = sv[wave][2 * W + wp];
      double gx = px * (double)wz.x, gy = py * (double)wz.x, gz = p0 * (double)wz.y;
      wave_sum3(gx, gy, gz, lane);
      if (lane < 3) {
         const double fc = f.w * (gx * a.m[lane] + gy * a.m[3 + lane] + gz * a.m[6 + lane]);
         double *op = out + (size_t)lane * a.nsp + A.w;
         *op = a.add ? *op + fc : fc;
      }
   }
}
template <class R>
__global__ __launch_bounds__(64 * GaT<R>::NW) void k_g_gather(GGaArgs a, const R *__restrict__ G,
                                                              const double *__restrict__ poly,
                                                              const int4 *__restrict__ anc,
                                                              const double4 *__restrict__ fr,
                                                              const int *__restrict__ start,
                                                              double *__restrict__ out) {
   b_g_gather<R>(blockIdx.x, gridDim.x, a, G, poly, anc, fr, start, out);
}

// force += the gathered forces, once the real-space pass has added its own.
__device__ __forceinline__ void b_g_add(int bx, int nbx, int ns, int nsp, const double *__restrict__ f,
                                        double *__restrict__ force) {
   const int i = bx * 256 + threadIdx.x;
   if (i >= ns) return;
#pragma unroll
   for (int c = 0; c < 3; c++) force[(size_t)c * nsp + i] += f[(size_t)c * nsp + i];
}
__global__ __launch_bounds__(256) void k_g_add(int ns, int nsp, const double *__restrict__ f,
                                               double *__restrict__ force) {
   b_g_add(blockIdx.x, gridDim.x, ns, nsp, f, force);
}

// ------------------------------------------------------------ the plan
typedef long double ld;
const ld PI_L = 3.14159265358979323846264338327950288L;

int up(int v, int m) { return (v + m - 1) / m * m; }

ld window(ld z, ld beta) {
   const ld y = 1.0L - z * z;
   return y > 0 ? expl(beta * (sqrtl(y) - 1.0L)) : (y == 0 ? expl(-beta) : 0.0L);
}

// The window's polynomials: for offset p and argument x in [-1, 1], z = (p +
// (x + 1)/2) / (w/2) - 1; Chebyshev interpolation of degree deg, as monomials.
template <class R> std::vector<double> window_polys() {
   constexpr int W = Win<R>::W, N = Win<R>::DEG + 1;
   const ld beta = Win<R>::BETA;
   ld T[N][N] = {}, cs[4 * N];
   T[0][0] = 1;
   T[1][1] = 1;
   for (int k = 2; k < N; k++)
      for (int j = 0; j < N; j++) T[k][j] = (j > 0 ? 2 * T[k - 1][j - 1] : 0) - T[k - 2][j];
   for (int q = 0; q < 4 * N; q++) cs[q] = cosl(q * PI_L / (2 * N));
   std::vector<double> out((size_t)N * W);
   for (int p = 0; p < W; p++) {
      ld f[N], mono[N] = {};
      for (int j = 0; j < N; j++) f[j] = window((p + (cs[2 * j + 1] + 1) / 2) / (W / 2.0L) - 1, beta);
      for (int k = 0; k < N; k++) {
         ld c = 0;
         for (int j = 0; j < N; j++) c += f[j] * cs[k * (2 * j + 1) % (4 * N)];
         c *= (k ? 2.0L : 1.0L) / N;
         for (int j = 0; j < N; j++) mono[j] += c * T[k][j];
      }
      for (int k = 0; k < N; k++) out[(size_t)k * W + p] = (double)mono[k];
   }
   return out;
}

// 1 / phi^(m), phi^(m) = int phi(2 d / w) cos(2 pi m d / n) dd, m = 0 .. mmax, by
// the tanh-sinh rule (the window has square-root ends); cos(m t) by the
// three-term recurrence.
void window_inverse(int w, ld beta, int n, int mmax, std::vector<double> &out) {
   const ld h = 0.0275L;
   std::vector<ld> sum(mmax + 1, 0);
   for (int j = 0; j <= 120; j++) {
      const ld t = j * h, u = PI_L / 2 * sinhl(t), ch = coshl(u);
      const ld wt = (j ? 2 : 1) * h * PI_L / 2 * coshl(t) / (ch * ch) * expl(beta * (1 / ch - 1));
      const ld c1 = cosl(PI_L * w / n * tanhl(u));
      ld c0 = 1, c = c1;
      sum[0] += wt;
      for (int m = 1; m <= mmax; m++) {
         sum[m] += wt * c;
         const ld cn = 2 * c1 * c - c0;
         c0 = c;
         c = cn;
      }
   }
   for (int m = 0; m <= mmax; m++) out.push_back((double)(1 / (sum[m] * w / 2)));
}

// Table [rows][ldt] of sign times cos or sin (2 pi r c / n) for r < nr, c < nc (r
// taken from r0), zero elsewhere.  co holds cos(2 pi j / n); n is a multiple of 4.
void trig_table(std::vector<double> &out, const std::vector<double> &co, int n, int rows, int ldt, int r0, int nr,
                int nc, bool sine, double sign) {
   const size_t o = out.size();
   out.resize(o + (size_t)rows * ldt, 0.0);
   for (int r = 0; r < nr; r++) {
      const int step = ((r0 + r) % n + n) % n;
      int q = sine ? 3 * n / 4 : 0;   // sin x = cos(x - pi/2)
      double *row = &out[o + (size_t)r * ldt];
      for (int c = 0; c < nc; c++) {
         row[c] = sign * co[q];
         q += step;
         if (q >= n) q -= n;
      }
   }
}

std::vector<double> roots(int n) {
   std::vector<double> co(n);
   for (int j = 0; j < n; j++) co[j] = 4 * j == n || 4 * j == 3 * n ? 0.0 : (double)cosl(2 * PI_L * j / n);
   return co;
}

}  // namespace

GridGeom mgpu::grid_geom(int ns, int nsp, int hmax, int kmax, int lmax, const double h[9], const double hinv[9],
                         double vol, double alpha, double kc, bool fp64) {
   GridGeom g;
   g.ns = ns; g.nsp = nsp; g.fp64 = fp64;
   g.m[0] = hmax; g.m[1] = kmax; g.m[2] = lmax;
   for (int d = 0; d < 3; d++) {
      // grid points per shortest wave along this cell vector (kc |h_d| / 2 pi
      // waves): the aliases of the modes next to the cutoff are down by
      // phi^(n - m) / phi^(m) = 1.4e-11 at 4.6 (FP64), 1.1e-4 at 4 (FP32), before
      // the weight's own 1e-6
      const double wv = kc / (2 * PI_D) * sqrt(h[d] * h[d] + h[3 + d] * h[3 + d] + h[6 + d] * h[6 + d]);
      g.n[d] = (int)std::min(1e6, std::max(3.0 * GB, ceil((fp64 ? 4.6 : 4.0) * wv / GB) * GB));
      g.nb[d] = g.n[d] / GB;
   }
   for (int i = 0; i < 9; i++) g.hinv[i] = hinv[i];
   g.vol = vol; g.alpha = alpha;
   g.w = fp64 ? Win<double>::W : Win<float>::W;
   // a brick's bucket holds four times the mean count and what a dense liquid's
   // or solid's 0.2 sites an A^3 put there (a droplet's bricks are full while the mean
   // is low), up to 448 (LDS of the weights kernel)
   const long nbr = (long)g.nb[0] * g.nb[1] * g.nb[2];
   const double fill = std::max(4.0 * (ns / nbr + 1), std::min(0.2 * vol / nbr, (double)ns));
   g.cap = up((int)std::min(448.0, std::max(64.0, fill)), 64);
   return g;
}

namespace {
// Where the grid beats the direct sum: its thirteen launches cost a floor that
// N_k N_s products must outweigh, its transforms depend on the grid alone, and
// with coarse points a tile of them holds so many sites that few blocks do the
// spreading and gathering.  MD step, direct against grid, us:
//   products    FP64 8,800 water sites (5.4e7) 216 and 226, 10,800 (8.2e7) 314 and 285,
//               16,384 (1.9e8) 344 and 256, 132,872 salt water (1.3e10) 7,870 and 1,112; mixed 14,400
//               water (1.5e8) 171 and 174, 12,288 silica (2.2e8) 166 and 157, 32,000 water
//               (7.2e8) 254 and 215, 132,872 1,336 and 635
//   transforms  few sites in a wide box or at a high cutoff: mixed 700 sites, 6.6e9
//               multiply-adds, 3.4e8 products 265 and 514, 4,000, 6e8, 3e8 184 and 199, 8,000, 2.7e8,
//               3.6e8 181 and 190, 16,000, 3e8, 5.4e8 203 and 196.  The FP64 direct sum slows as the
//               transforms grow: 700, 1.4e9, 8.1e7 310 and 298, 9.6e9, 3.4e8 4,184 and 887, 2,400,
//               4.5e8, 1.1e8 224 and 238, 8,000, 3.8e8, 3.6e8 365 and 272: no term
//   points      alpha 0.15 (FP64 1.8 A^3 a point, mixed 2.8): a droplet of 16,000 sites, 1.8e8
//               products, FP64 367 and 420, 6.1e8 mixed 244 and 309; 80,000 sites, 1.9e9 mixed 559 and 500
bool grid_pays(const GridGeom &g, int nk) {
   const double direct = (double)nk * g.ns, L = g.m[2] + 1;
   double points = 1;
   for (int d = 0; d < 3; d++) points *= g.n[d];
   const double macs = 2 * (points * 2 * L + 4.0 * g.n[0] * g.n[1] * (g.m[1] + 1) * L +
                            4.0 * g.n[0] * (g.m[0] + 1) * (2 * g.m[1] + 1) * L);
   const double coarse = g.vol / points / (g.fp64 ? 0.45 : 0.69);
   return direct > (g.fp64 ? 8e7 : std::max(2e8, 1e8 + macs)) * std::max(1.0, coarse);
}
}  // namespace

bool mgpu::grid_applies(const GridGeom &g, int nsxf, int nk, double kc, const std::vector<KRow> &rows) {
   // frameworks need two structure factors a k; the window's width counts on
   // the Gaussian damping of the last k (measured to 9.9e-6; the reference's
   // automatic parameters give their accuracy here, 1.013e-5 by default, and take
   // the direct sum); one row per (h, k) is the reference's set
   if (nsxf != g.ns || g.ns < 1 || rows.empty()) return false;
   if (!(exp(-kc * kc / (4 * g.alpha * g.alpha)) <= 1e-5)) return false;
   for (size_t r = 1; r < rows.size(); r++)
      if (rows[r].h == rows[r - 1].h && rows[r].k == rows[r - 1].k) return false;
   for (int d = 0; d < 3; d++)
      if (g.n[d] > 512 || g.n[d] < 4 * g.m[d]) return false;
   return grid_pays(g, nk);
}

GridSizes mgpu::grid_sizes(const GridGeom &g) {
   GridSizes z;
   const size_t rs = g.fp64 ? 8 : 4, ns = g.ns;
   const size_t L = g.m[2] + 1, P = (2 * g.m[1] + 1) * L;
   const size_t nb = (size_t)g.nb[0] * g.nb[1] * g.nb[2];
   size_t off = 0;
   auto take = [&](size_t bytes) {
      const size_t o = off;
      off += (bytes + 255) & ~(size_t)255;
      return o;
   };
   z.sa = take(16 * ns);
   z.sx = take(8 * 3 * (size_t)g.nsp);
   z.cnt = take(4 * nb);
   z.start = take(4 * (nb + 1));
   z.bucket = take(4 * nb * g.cap);
   z.anc = take(16 * ns);
   z.fr = take(32 * ns);
   z.wt = take(3 * (size_t)(g.w + 2) * rs * ns);
   z.G = take(rs * g.n[0] * g.n[1] * g.n[2]);
   z.T1 = take(8 * g.n[0] * g.n[1] * 2 * L);
   z.T2 = take(8 * g.n[0] * 2 * P);
   z.T3 = take(8 * (2 * g.m[0] + 1) * 2 * P);
   z.nred = (int)(((2 * g.m[0] + 1) * P + 255) / 256);
   z.bpart = take(8 * 8 * (size_t)z.nred);
   z.fout = take(8 * 3 * (size_t)g.nsp);
   z.bytes = off;
   return z;
}

namespace {
// Column tiles of a z transform: groups of NT <= 5 tiles.
void z_split(int ncols, int &nt, int &ngrp) {
   const int tiles = (ncols + 15) / 16;
   ngrp = (tiles + 4) / 5;
   nt = (tiles + ngrp - 1) / ngrp;
}

template <class R> void build_tables(const GridGeom &g, GridTables &t) {
   const int W = Win<R>::W, L = g.m[2] + 1;
   std::vector<double> tab, dec;
   for (int d = 0; d < 3; d++) {
      int same = 0;   // an earlier axis of the same grid and box
      while (same < d && (g.n[same] != g.n[d] || g.m[same] != g.m[d])) same++;
      t.dec_off[d] = same < d ? t.dec_off[same] : dec.size();
      if (same == d) window_inverse(W, Win<R>::BETA, g.n[d], g.m[d], dec);
   }
   int nt, ng;
   {   // z: forward [z][c L + l], inverse [c L + l][z]
      const int n = g.n[2];
      const std::vector<double> co = roots(n);
      z_split(2 * L, nt, ng);
      t.zf_ld = nt * ng * 16;
      t.zf = tab.size();
      tab.resize(t.zf + (size_t)n * t.zf_ld, 0.0);
      z_split(n, nt, ng);
      t.zi_ld = nt * ng * 16;
      t.zi = tab.size();
      tab.resize(t.zi + (size_t)up(2 * L, 8) * t.zi_ld, 0.0);
      for (int l = 0; l < L; l++)
         for (int z = 0, q = 0, q3 = 3 * n / 4; z < n; z++) {
            const double c = co[q], s = co[q3];
            if ((q += l) >= n) q -= n;
            if ((q3 += l) >= n) q3 -= n;
            tab[t.zf + (size_t)z * t.zf_ld + l] = c;
            tab[t.zf + (size_t)z * t.zf_ld + L + l] = s;
            tab[t.zi + (size_t)l * t.zi_ld + z] = c;
            tab[t.zi + (size_t)(L + l) * t.zi_ld + z] = s;
         }
   }
   for (int d = 0; d < 2; d++) {   // x, y: forward e^{+} [n][m], inverse e^{-} [2 m + 1][n/2 + 1]
      const int n = g.n[d], m = g.m[d];
      const std::vector<double> co = roots(n);
      t.f_ld[d] = up(m + 1, 16);
      t.fr[d] = tab.size();
      trig_table(tab, co, n, n, t.f_ld[d], 0, n, m + 1, false, 1.0);
      t.fi[d] = tab.size();
      trig_table(tab, co, n, n, t.f_ld[d], 0, n, m + 1, true, 1.0);
      t.i_ld[d] = up(n / 2 + 1, 16);
      const int kr = up(2 * m + 1, 8);
      t.ir[d] = tab.size();
      trig_table(tab, co, n, kr, t.i_ld[d], -m, 2 * m + 1, n / 2 + 1, false, 1.0);
      t.ii[d] = tab.size();
      trig_table(tab, co, n, kr, t.i_ld[d], -m, 2 * m + 1, n / 2 + 1, true, -1.0);
   }
   t.dec = tab.size();
   tab.insert(tab.end(), dec.begin(), dec.end());
   t.poly = tab.size();
   static const std::vector<double> poly = window_polys<R>();   // the window's, the same for every grid
   tab.insert(tab.end(), poly.begin(), poly.end());
   t.data = std::move(tab);
}
}  // namespace

void mgpu::grid_tables(const GridGeom &g, GridTables &t) {
   if (g.fp64) build_tables<double>(g, t);
   else build_tables<float>(g, t);
}

void mgpu::grid_rowmap(const GridGeom &g, const std::vector<KRow> &rows, std::vector<int> &map) {
   map.assign((size_t)(g.m[0] + 1) * (2 * g.m[1] + 1), -1);
   for (size_t r = 0; r < rows.size(); r++) map[(size_t)rows[r].h * (2 * g.m[1] + 1) + rows[r].k + g.m[1]] = (int)r;
}

namespace {
template <class RI, class RO, int NT>
void gz_launch(std::vector<LaunchRec> *rec, hipStream_t st, unsigned grid, const GzArgs &a, const RI *in,
               const double *tab, RO *out) {
   glaunch<k_gz<RI, RO, NT>, b_gz<RI, RO, NT>, 256>(rec, st, grid, 256, 0, a, in, tab, out);
}

template <class RI, class RO>
void z_pass(std::vector<LaunchRec> *rec, hipStream_t st, int nlines, int K, int ncols, int ldt, const RI *in,
            const double *tab, RO *out) {
   GzArgs a;
   int nt;
   a.nlines = nlines; a.K = K; a.lda = K; a.ncols = ncols; a.ldt = ldt; a.ldo = ncols;
   z_split(ncols, nt, a.ngrp);
   a.nmt = (nlines + 15) / 16;
   const unsigned grid = (a.nmt * a.ngrp + 3) / 4;
   switch (nt) {
   case 1: gz_launch<RI, RO, 1>(rec, st, grid, a, in, tab, out); break;
   case 2: gz_launch<RI, RO, 2>(rec, st, grid, a, in, tab, out); break;
   case 3: gz_launch<RI, RO, 3>(rec, st, grid, a, in, tab, out); break;
   case 4: gz_launch<RI, RO, 4>(rec, st, grid, a, in, tab, out); break;
   default: gz_launch<RI, RO, 5>(rec, st, grid, a, in, tab, out); break;
   }
}

void c_pass(std::vector<LaunchRec> *rec, hipStream_t st, GcArgs a, const double *in, const double *er,
            const double *ei, double *out) {
   a.nmt = (a.M + 15) / 16;
   a.nct = (a.N + 15) / 16;
   const unsigned grid = (unsigned)(((long)a.nbatch * a.nmt * a.nct + 3) / 4);
   glaunch<k_gc, b_gc, 256>(rec, st, grid, 256, 0, a, in, er, ei, out);
}

// The stages of a pass on explicit storage.
template <class R> struct Stages {
   mgpu_engine *e;
   std::vector<LaunchRec> *rec;
   const GridGeom &g;
   const GridTables &t;
   const GridBufs &b;
   const GridSizes z;
   const double *tab, *poly;
   size_t L, P;
   int4 *anc;
   int *cnt, *start;
   R *G;
   double *T1, *T2, *T3;

   Stages(mgpu_engine *e_, std::vector<LaunchRec> *rec_, const GridGeom &g_, const GridTables &t_, const GridBufs &b_)
       : e(e_), rec(rec_), g(g_), t(t_), b(b_), z(grid_sizes(g_)), tab(b_.tab), poly(b_.tab + t_.poly) {
      uint8_t *B = b.base;
      L = g.m[2] + 1;
      P = (2 * g.m[1] + 1) * L;
      anc = (int4 *)(B + z.anc);
      cnt = (int *)(B + z.cnt);
      start = (int *)(B + z.start);
      G = (R *)(B + z.G);
      T1 = (double *)(B + z.T1);
      T2 = (double *)(B + z.T2);
      T3 = (double *)(B + z.T3);
   }

   // the sites into bricks, with their spread weights times w
   void sites(const double *w) {
      hipStream_t st = e->stream;
      const int nbr = g.nb[0] * g.nb[1] * g.nb[2];
      uint8_t *B = b.base;
      GBinArgs a;
      for (int i = 0; i < 9; i++) a.hinv[i] = g.hinv[i];
      for (int d = 0; d < 3; d++) { a.n[d] = g.n[d]; a.nb[d] = g.nb[d]; }
      a.ns = g.ns; a.nsp = g.nsp; a.w = g.w; a.cap = g.cap;
      a.site = b.site; a.sa = (int4 *)(B + z.sa); a.sx = (double *)(B + z.sx); a.cnt = cnt;
      a.bucket = (int *)(B + z.bucket);
      glaunch<k_g_bin, b_g_bin, 256>(rec, st, (g.ns + 255) / 256, 256, 0, a);
      glaunch<k_g_scan, b_g_scan, 256>(rec, st, 1, 256, 0, nbr, cnt, start);
      GWtArgs q;
      q.nb = nbr; q.ns = g.ns; q.nsp = g.nsp; q.cap = g.cap;
      q.sa = a.sa; q.sx = a.sx; q.chg = w; q.bucket = a.bucket; q.start = start; q.cnt = cnt;
      q.poly = poly; q.wt = B + z.wt; q.anc = anc; q.fr = (double4 *)(B + z.fr);
      glaunch<k_g_weights<R>, b_g_weights<R>, 256>(rec, st, (nbr + 3) / 4, 256, (size_t)g.cap * (16 * 8 + 4 * 4), q);
   }

   void spread() {
      GSpArgs s;
      for (int d = 0; d < 3; d++) { s.n[d] = g.n[d]; s.nb[d] = g.nb[d]; }
      s.ntz = (g.nb[2] + 1) / 2;
      s.per = (g.nb[0] * g.nb[1] * s.ntz + 7) / 8;
      glaunch<k_g_spread<R>, b_g_spread<R>, 256>(rec, e->stream, 8 * s.per, 256, 0, s, (const R *)(b.base + z.wt), anc,
                                                 start, G);
   }

   void forward() {
      hipStream_t st = e->stream;
      GcArgs c;
      z_pass<R, double>(rec, st, g.n[0] * g.n[1], g.n[2], 2 * L, t.zf_ld, G, tab + t.zf, T1);
      c.nbatch = g.n[0]; c.K = g.n[1]; c.M = g.m[1] + 1; c.N = L; c.ldt = t.f_ld[1];
      c.off = c.qoff = g.m[1]; c.mq = g.m[1] + 1;
      c.inb = (size_t)g.n[1] * 2 * L; c.ink = 2 * L; c.inc = L; c.outb = 2 * P; c.outm = L; c.outc = P;
      c_pass(rec, st, c, T1, tab + t.fr[1], tab + t.fi[1], T2);
      c.nbatch = 1; c.K = g.n[0]; c.M = g.m[0] + 1; c.N = P; c.ldt = t.f_ld[0];
      c.off = c.qoff = g.m[0]; c.mq = g.m[0] + 1;
      c.inb = 0; c.ink = 2 * P; c.inc = P; c.outb = 0; c.outm = 2 * P; c.outc = P;
      c_pass(rec, st, c, T2, tab + t.fr[0], tab + t.fi[0], T3);
   }

   void inverse() {
      hipStream_t st = e->stream;
      GcArgs c;
      c.nbatch = 1; c.K = 2 * g.m[0] + 1; c.M = g.n[0] / 2 + 1; c.N = P; c.ldt = t.i_ld[0];
      c.off = 0; c.qoff = g.n[0]; c.mq = g.n[0] / 2;
      c.inb = 0; c.ink = 2 * P; c.inc = P; c.outb = 0; c.outm = 2 * P; c.outc = P;
      c_pass(rec, st, c, T3, tab + t.ir[0], tab + t.ii[0], T2);
      c.nbatch = g.n[0]; c.K = 2 * g.m[1] + 1; c.M = g.n[1] / 2 + 1; c.N = L; c.ldt = t.i_ld[1];
      c.off = 0; c.qoff = g.n[1]; c.mq = g.n[1] / 2;
      c.inb = 2 * P; c.ink = L; c.inc = P; c.outb = (size_t)g.n[1] * 2 * L; c.outm = 2 * L; c.outc = L;
      c_pass(rec, st, c, T2, tab + t.ir[1], tab + t.ii[1], T1);
      z_pass<double, R>(rec, st, g.n[0] * g.n[1], 2 * L, g.n[2], t.zi_ld, T1, tab + t.zi, G);
   }

   void gather(double *out, bool add) {
      GGaArgs a;
      for (int d = 0; d < 3; d++) {
         a.n[d] = g.n[d];
         a.nb[d] = g.nb[d];
         // k = h a* + k b* + l c* as ewald.c:445-447 forms it: c* along z only (a
         // barostat's h may be tilted from that by a little)
         for (int q = 0; q < 3; q++) a.m[3 * d + q] = d == 2 && q < 2 ? 0.0 : 2.0 * g.n[d] * g.hinv[3 * d + q];
      }
      constexpr int TB = GaT<R>::TZ / GB;
      a.ntz = (g.nb[2] + TB - 1) / TB;
      a.per = (g.nb[0] * g.nb[1] * a.ntz + 7) / 8;
      a.nsp = g.nsp;
      a.add = add;
      glaunch<k_g_gather<R>, b_g_gather<R>, 64 * GaT<R>::NW>(rec, e->stream, 8 * a.per, 64 * GaT<R>::NW, 0, a, G, poly,
                                                             anc, (const double4 *)(b.base + z.fr), start, out);
   }

   const double *dec(int d) const { return tab + t.dec + t.dec_off[d]; }
};

template <class R>
void pass(mgpu_engine *e, std::vector<LaunchRec> *rec, const GridGeom &g, const GridTables &t, const GridBufs &b,
          bool join) {
   Stages<R> s(e, rec, g, t, b);
   mgpu_engine *pe = b.prof ? e : nullptr;
   {
      ProfScope ps(pe, "ewald_grid_spread");
      s.sites(b.w);
      s.spread();
   }
   {
      ProfScope ps(pe, "ewald_grid_forward");
      s.forward();
   }
   {
      ProfScope ps(pe, "ewald_grid_kspace");
      GkArgs k;
      k.hmax = g.m[0]; k.kmax = g.m[1]; k.lmax = g.m[2];
      k.vol = g.vol; k.r4a = -1.0 / (4.0 * g.alpha * g.alpha); k.c2 = 2 * PI_D * g.hinv[8];
      k.rows = b.rows; k.rowmap = b.rowmap;
      k.dx = s.dec(0); k.dy = s.dec(1); k.dz = s.dec(2);
      k.bpart = (double *)(b.base + s.z.bpart);
      glaunch<k_gk, b_gk, 256>(rec, e->stream, s.z.nred, 256, 0, k, s.T3);
   }
   {
      ProfScope ps(pe, "ewald_grid_inverse");
      s.inverse();
   }
   {
      ProfScope ps(pe, "ewald_grid_gather");
      // straight into the forces when no other stream is adding to them
      const bool direct = !(join && e->join_pending);
      double *fout = (double *)(b.base + s.z.fout);
      s.gather(direct ? b.force : fout, direct);
      if (!direct) {
         join_side(e);
         glaunch<k_g_add, b_g_add, 256>(rec, e->stream, (g.ns + 255) / 256, 256, 0, g.ns, g.nsp, fout, b.force);
      }
   }
}

// Place of k vector k's mode in the dense box, and whether it is held as
// its inverse (l < 0).
struct GxArgs {
   int nk, hmax, kmax, lmax;
   const KRow *rows;
   const int *krow;
   const double *dx, *dy, *dz;
};
__device__ __forceinline__ size_t mode_of(const GxArgs &a, int k, bool &conj, double &dec) {
   const KRow R = a.rows[a.krow[k]];
   const int l = R.l0 + (k - R.kstart), L = a.lmax + 1, P = (2 * a.kmax + 1) * L;
   conj = l < 0;
   const int h = conj ? -R.h : R.h, kk = conj ? -R.k : R.k, ll = conj ? -l : l;
   dec = a.dx[R.h] * a.dy[R.k < 0 ? -R.k : R.k] * a.dz[ll];
   return (size_t)(h + a.hmax) * 2 * P + (kk + a.kmax) * L + ll;
}
// cs[k] = S(k) from the transformed grid.
__global__ __launch_bounds__(256) void k_g_sf(GxArgs a, const double *__restrict__ T, double2 *__restrict__ cs) {
   const int k = blockIdx.x * 256 + threadIdx.x;
   if (k >= a.nk) return;
   bool conj;
   double dec;
   const size_t o = mode_of(a, k, conj, dec);
   const double s = dec * T[o + (2 * a.kmax + 1) * (a.lmax + 1)];
   cs[k] = make_double2(dec * T[o], conj ? -s : s);
}
// The inverse transform's weights coeff S from cs, into a cleared T.
__global__ __launch_bounds__(256) void k_g_fill(GxArgs a, const double4 *__restrict__ kc, const double2 *__restrict__ cs,
                                                double *__restrict__ T) {
   const int k = blockIdx.x * 256 + threadIdx.x;
   if (k >= a.nk) return;
   bool conj;
   double dec;
   const size_t o = mode_of(a, k, conj, dec);
   const double w = dec * kc[k].w;
   T[o] = w * cs[k].x;
   T[o + (2 * a.kmax + 1) * (a.lmax + 1)] = conj ? -w * cs[k].y : w * cs[k].y;
}
}  // namespace

void mgpu::grid_pass(mgpu_engine *e, std::vector<LaunchRec> *rec, const GridGeom &g, const GridTables &t,
                     const GridBufs &b, bool join) {
   if (g.fp64) pass<double>(e, rec, g, t, b, join);
   else pass<float>(e, rec, g, t, b, join);
}

void mgpu::grid_clear(mgpu_engine *e, const GridGeom &g, uint8_t *base) {
   const GridSizes z = grid_sizes(g);
   zero_async(e, base + z.cnt, 4 * (size_t)g.nb[0] * g.nb[1] * g.nb[2]);
}

// What the tables and the place of the brick counts depend on.
static void table_key(const GridGeom &g, int key[8]) {
   for (int d = 0; d < 3; d++) {
      key[d] = g.n[d];
      key[3 + d] = g.m[d];
   }
   key[6] = g.fp64;
   key[7] = g.ns;
}

std::shared_ptr<const GridTables> mgpu::grid_host_tables(mgpu_engine *e, const GridGeom &g) {
   int key[8];
   table_key(g, key);
   if (e->grid_tab && memcmp(key, e->grid_key, sizeof key) == 0) return e->grid_tab;
   if (!e->grid_host_tab || memcmp(key, e->grid_host_key, sizeof key) != 0) {
      e->grid_host_tab.reset();
      auto t = std::make_shared<GridTables>();
      grid_tables(g, *t);
      e->grid_host_tab = t;
      memcpy(e->grid_host_key, key, sizeof key);
   }
   return e->grid_host_tab;
}

// The grid of the engine's geometry and precision; whether it is to be used.
static bool engine_grid(const mgpu_engine *e, GridGeom &g) {
   g = grid_geom(e->nsites, e->nsp, e->hmax, e->kmax, e->lmax, e->h, e->hinv, host_det(e->h), e->alpha, e->k_cutoff,
                 e->precision == MGPU_FP64);
   return grid_applies(g, e->nsitesxf, e->nk, e->k_cutoff, e->rows);
}

bool mgpu::grid_chosen(const mgpu_engine *e) {
   GridGeom g;
   return engine_grid(e, g);
}

// The engine's plan for its geometry and precision, made where it is missing
// or stale; false where the direct sum is to run.
static bool grid_plan(mgpu_engine *e, GridGeom &g) {
   if (!engine_grid(e, g)) return false;
   const GridSizes z = grid_sizes(g);
   // the plan: tables of the grid's sizes, the k set's row map, and the
   // cleared parts of the scratch block
   int key[8];
   table_key(g, key);
   const bool same = e->grid_tab && memcmp(key, e->grid_key, sizeof key) == 0;
   if (e->capturing && (!same || e->grid_version != e->geom_version))
      throw StatusError{MGPU_E_STATE, "gridded Ewald plan changed during capture"};
   if (!same) {
      auto t = std::make_shared<GridTables>();
      grid_tables(g, *t);
      e->d_gtab.reserve(t->data.size());
      HIPCHK(hipMemcpyAsync(e->d_gtab.p, t->data.data(), t->data.size() * sizeof(double), hipMemcpyHostToDevice, e->stream));
      HIPCHK(hipStreamSynchronize(e->stream));
      e->grid_tab = t;
      memcpy(e->grid_key, key, sizeof key);
      // a step captured with the old tables (another precision's, say) is stale
      e->geom_version++;
   }
   if (e->d_grid.reserve(z.bytes) || !same) grid_clear(e, g, e->d_grid.p);
   if (!same || e->grid_version != e->geom_version) {
      std::vector<int> map;
      grid_rowmap(g, e->rows, map);
      e->d_growmap.reserve(map.size());
      HIPCHK(hipMemcpyAsync(e->d_growmap.p, map.data(), sizeof(int) * map.size(), hipMemcpyHostToDevice, e->stream));
      HIPCHK(hipStreamSynchronize(e->stream));
      e->grid_version = e->geom_version;
   }
   return true;
}

static GridBufs grid_bufs(mgpu_engine *e) {
   GridBufs b;
   b.site = e->d_site.p; b.w = e->d_chg_site.p; b.force = e->d_force_site.p;
   b.rows = e->d_rows.p; b.rowmap = e->d_growmap.p; b.tab = e->d_gtab.p; b.base = e->d_grid.p; b.prof = true;
   return b;
}

bool mgpu::run_ewald_grid(mgpu_engine *e) {
   GridGeom g;
   if (!grid_plan(e, g)) return false;
   const GridSizes z = grid_sizes(g);
   e->d_out.reserve(OUT_SIZE);
   grid_pass(e, e->rec, g, *e->grid_tab, grid_bufs(e), true);
   const double *bpart = (const double *)(e->d_grid.p + z.bpart);
   if (e->defer_recip) {   // the glue adds them (eval_forces_device)
      e->recip_part = bpart;
      e->recip_rows = z.nred;
   } else {
      reduce_cols(e, bpart, z.nred, 8, e->d_out.p + OUT_RECIP);
   }
   return true;
}

static GxArgs mode_args(mgpu_engine *e, const Stages<double> &s) {
   return GxArgs{e->nk, s.g.m[0], s.g.m[1], s.g.m[2], e->d_rows.p, e->d_krow.p, s.dec(0), s.dec(1), s.dec(2)};
}

bool mgpu::grid_weighted_sf(mgpu_engine *e, const double *w, double2 *cs) {
   GridGeom g;
   if (e->precision != MGPU_FP64 || !grid_plan(e, g)) return false;
   const GridBufs b = grid_bufs(e);
   Stages<double> s(e, nullptr, g, *e->grid_tab, b);
   s.sites(w);
   s.spread();
   s.forward();
   k_g_sf<<<(e->nk + 255) / 256, 256, 0, e->stream>>>(mode_args(e, s), s.T3, cs);
   return true;
}

bool mgpu::grid_backproject(mgpu_engine *e, const double *w, const double4 *kc, const double2 *cs, double *out) {
   GridGeom g;
   if (e->precision != MGPU_FP64 || !grid_plan(e, g)) return false;
   const GridBufs b = grid_bufs(e);
   Stages<double> s(e, nullptr, g, *e->grid_tab, b);
   s.sites(w);
   zero_async(e, s.T3, sizeof(double) * (2 * g.m[0] + 1) * 2 * s.P);
   k_g_fill<<<(e->nk + 255) / 256, 256, 0, e->stream>>>(mode_args(e, s), kc, cs, s.T3);
   s.inverse();
   s.gather(out, true);
   return true;
}
