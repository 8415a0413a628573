// Reciprocal-space Ewald sum, FP64 path (restates src/ewald.c:280-589).
//
// Per call: per-site trig tables by the reference's recurrence (trig_recur,
// ewald.c:148-193, z table premultiplied by q as at ewald.c:475-481), the
// structure factors S(k) for the reference's half-space k set, the energy
// and stress per k (ewald.c:539-553), and the force back-projection
// (ewald.c:557-579).  Framework sites (the last ns - nsitesxf sites) enter
// S(k) separately so that frame-frame terms are excluded as in the reference.
//
// S(k): a complex GEMM of the (h,k) rows against the l columns on the FP64
// matrix cores, per chunk of sites; chunk partials are reduced in a fixed
// order (deterministic).
//
// Forces: one thread per site walks the rows; exp(i l c*.r) is advanced along
// a row by multiplication with exp(i c*.r), and exp(i k b*.r) along a run of
// rows of one h, so the inner loop touches no memory except the per-k
// weights (uniform loads).
#include "mgpu_internal.h"
#include "mgpu_ewald_grid.h"

#include <algorithm>
#include <cmath>
#include <mutex>
#include <string>

using namespace mgpu;

namespace {

constexpr double PI_D = 3.14159265358979323846;

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
   return make_double2(a.x * b.x - a.y * b.y, a.y * b.x + a.x * b.y);
}

struct TrigArgs {
   double ks[9];     // rows a*, b*, c* (2 pi h^-1)
   int hmax, kmax, lmax, ns, nsp;
};

// trig_recur for the three axes; z tables multiplied by q.
__global__ void k_trig(TrigArgs a, const double *__restrict__ site, const double *__restrict__ chg,
                       double2 *__restrict__ tx, double2 *__restrict__ ty, double2 *__restrict__ tz,
                       double2 *__restrict__ tz1) {
   int i = blockIdx.x * blockDim.x + threadIdx.x;
   if (i >= a.ns) return;
   double x = site[i], y = site[a.nsp + i], z = site[2 * a.nsp + i], q = chg[i];
   const int nmax[3] = {a.hmax, a.kmax, a.lmax};
   double2 *tb[3] = {tx, ty, tz};
#pragma unroll
   for (int ax = 0; ax < 3; ax++) {
      double2 *t = tb[ax];
      double w = ax == 2 ? q : 1.0;
      t[i] = make_double2(w, 0.0);
      if (nmax[ax] >= 1) {
         double kr = a.ks[3 * ax] * x + a.ks[3 * ax + 1] * y + a.ks[3 * ax + 2] * z;
         double s1, c1;
         sincos(kr, &s1, &c1);
         if (ax == 2) tz1[i] = make_double2(c1, s1);
         double cm = c1, sm = s1;
         t[(size_t)a.nsp + i] = make_double2(c1 * w, s1 * w);
         for (int n = 2; n <= nmax[ax]; n++) {
            double cc = cm * c1 - sm * s1;
            double ss = sm * c1 + cm * s1;
            cm = cc;
            sm = ss;
            t[(size_t)n * a.nsp + i] = make_double2(cc * w, ss * w);
         }
      } else if (ax == 2) {
         double s1, c1;
         double kr = a.ks[6] * x + a.ks[7] * y + a.ks[8] * z;
         sincos(kr, &s1, &c1);
         tz1[i] = make_double2(c1, s1);
      }
   }
}

typedef double dbl4 __attribute__((ext_vector_type(4)));

struct SkArgs {
   int nk, ns, nsp, nsxf, nrows, lmax;
   int nca, ncb;       // site chunks over [0, nsxf) and over the framework sites [nsxf, ns)
   int nrb;            // row blocks of 64 rows
   const KRow *rows;
   const double2 *tx, *ty, *tz;
   double *part;       // [nca + ncb][nk][4]: (C, S) of a chunk in slots 0-1 or, framework, 2-3
};

// S(k) as a complex GEMM on the FP64 matrix cores.  Rows are the (h,k) rows
// of the k set (A_r(i) = exp(i(h a* + k b*).r_i)), columns the l >= 0 of the
// q-weighted table Z_l(i) = q_i exp(i l c*.r_i), and the sum runs over a
// chunk of sites.  Four real products RR = sum Ar Zr, II = sum Ai Zi,
// RI = sum Ar Zi, IR = sum Ai Zr give both signs of l:
// S(h,k,+l) = (RR - II) + i(RI + IR) and, as Z_{-l} = conj Z_l (qsincos,
// ewald.c:108-121), S(h,k,-l) = (RR + II) + i(IR - RI).  A workgroup is four
// waves, one 16-row tile each, over NC 16-column tiles starting at
// l = 48 blockIdx.y.  v_mfma_f64_16x16x4f64 takes site i0 + 4s + lane/16 with row (column)
// lane%16 in its A (B) operand and leaves D[lane/16 + 4v][lane%16] in item
// v (both checked on gfx950 with integer operands).  The workgroups of one chunk go to one XCD (workgroup ids are dealt
// round robin over the 8 XCDs), so that the chunk's X, Y and Z rows come from
// HBM about once.  Each k of the chunk is stored exactly once.
template <int NC>
__global__ __launch_bounds__(256) void k_sfac(SkArgs a) {
   const int nchunks = a.nca + a.ncb;
   const int L = blockIdx.x, s8 = L >> 3;
   const int chunk = (L & 7) * (nchunks >> 3) + s8 / a.nrb;
   const int rb = s8 % a.nrb;
   const bool fwc = chunk >= a.nca;
   int c0, c1;
   if (!fwc) {
      c0 = (int)((long)a.nsxf * chunk / a.nca);
      c1 = (int)((long)a.nsxf * (chunk + 1) / a.nca);
   } else {
      const long nf = a.ns - a.nsxf, c = chunk - a.nca;
      c0 = a.nsxf + (int)(nf * c / a.ncb);
      c1 = a.nsxf + (int)(nf * (c + 1) / a.ncb);
   }
   const int lane = threadIdx.x & 63, m = lane & 15, kq = lane >> 4;
   const int rt = rb * 4 + (threadIdx.x >> 6);
   // this lane's operand row and columns; rows past the end read the last
   // row and columns past lmax read row lmax: their outputs are never stored
   const KRow R = a.rows[min(rt * 16 + m, a.nrows - 1)];
   const double2 *xp = a.tx + (size_t)R.h * a.nsp;
   const double2 *yp = a.ty + (size_t)(R.k < 0 ? -R.k : R.k) * a.nsp;
   const double ysg = R.k < 0 ? -1.0 : 1.0;
   const int lb = 48 * blockIdx.y;
   const double2 *zp[NC];
#pragma unroll
   for (int c = 0; c < NC; c++) zp[c] = a.tz + (size_t)min(lb + m + 16 * c, a.lmax) * a.nsp;
   dbl4 acc[NC][4];
#pragma unroll
   for (int c = 0; c < NC; c++)
#pragma unroll
      for (int q = 0; q < 4; q++) acc[c][q] = dbl4{0, 0, 0, 0};
   const int nstep = (c1 - c0 + 3) >> 2;
   const int ilast = max(c1 - 1, 0);
   int i = c0 + kq;
   // operands one step ahead; indexes clamped into the chunk, the sites past
   // its end weighted by zero
   int ic = min(i, ilast);
   double2 xn = xp[ic], yn = yp[ic], zn[NC];
#pragma unroll
   for (int c = 0; c < NC; c++) zn[c] = zp[c][ic];
   for (int st = 0; st < nstep; st++) {
      const double2 x = xn, y = yn;
      double2 z[NC];
#pragma unroll
      for (int c = 0; c < NC; c++) z[c] = zn[c];
      const double wgt = i < c1 ? 1.0 : 0.0;
      i += 4;
      ic = min(i, ilast);
      xn = xp[ic];
      yn = yp[ic];
#pragma unroll
      for (int c = 0; c < NC; c++) zn[c] = zp[c][ic];
      const double yi = ysg * y.y;
      const double ar = (x.x * y.x - x.y * yi) * wgt, ai = (x.y * y.x + x.x * yi) * wgt;
#pragma unroll
      for (int c = 0; c < NC; c++) {
         acc[c][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, z[c].x, acc[c][0], 0, 0, 0);
         acc[c][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, z[c].y, acc[c][1], 0, 0, 0);
         acc[c][2] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, z[c].y, acc[c][2], 0, 0, 0);
         acc[c][3] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, z[c].x, acc[c][3], 0, 0, 0);
      }
   }
   // store: item v of this lane is row rt*16 + kq + 4v, column l = lb + m + 16c
#pragma unroll
   for (int v = 0; v < 4; v++) {
      const int rr = rt * 16 + kq + 4 * v;
      if (rr >= a.nrows) continue;
      const KRow Q = a.rows[rr];
#pragma unroll
      for (int c = 0; c < NC; c++) {
         const int l = lb + m + 16 * c;
         if (l > a.lmax) continue;
         const double RR = acc[c][0][v], II = acc[c][1][v], RI = acc[c][2][v], IR = acc[c][3][v];
         double2 *p;
         if (l >= Q.l0 && l < Q.l0 + Q.nl) {
            p = (double2 *)(a.part + ((size_t)chunk * a.nk + Q.kstart + (l - Q.l0)) * 4);
            const double2 val = make_double2(RR - II, RI + IR), zero = make_double2(0, 0);
            p[0] = fwc ? zero : val;
            p[1] = fwc ? val : zero;
         }
         if (l > 0 && -l >= Q.l0 && -l < Q.l0 + Q.nl) {
            p = (double2 *)(a.part + ((size_t)chunk * a.nk + Q.kstart + (-l - Q.l0)) * 4);
            const double2 val = make_double2(RR + II, IR - RI), zero = make_double2(0, 0);
            p[0] = fwc ? zero : val;
            p[1] = fwc ? val : zero;
         }
      }
   }
}

struct EkArgs {
   int nk, nchunks, nrows;
   double vol, r4a, c2;
   const KRow *rows;
   const int *krow;
   const double *part;
   double *w;       // [nk][4]: Wc, Ws (all sites), Wcn, Wsn (framework sites)
   double *bpart;   // [nblocks][8]
};

// Per k: sum the chunk partials, energy, stress, weights (ewald.c:506-553).
__global__ __launch_bounds__(256) void k_ewald_k(EkArgs a) {
   __shared__ double ws[4][8];
   int k = blockIdx.x * 256 + threadIdx.x;
   double pe = 0, s00 = 0, s01 = 0, s02 = 0, s11 = 0, s12 = 0, s22 = 0;
   if (k < a.nk) {
      double scn = 0, ssn = 0, scf = 0, ssf = 0;
      for (int c = 0; c < a.nchunks; c++) {
         const double *p = a.part + ((size_t)c * a.nk + k) * 4;
         scn += p[0]; ssn += p[1]; scf += p[2]; ssf += p[3];
      }
      KRow R = a.rows[a.krow[k]];
      int l = R.l0 + (k - R.kstart);
      double kx = R.kx, ky = R.ky, kz = R.kzt + l * a.c2;
      double ksq = kx * kx + ky * ky + kz * kz;
      double coeff = 2.0 / ((0.25 / PI_D) * a.vol) * exp(ksq * a.r4a) / ksq;
      double coeff2 = 2.0 * (1.0 - ksq * a.r4a) / ksq;
      double pe_k = 0.5 * coeff * (scn * (scn + scf + scf) + ssn * (ssn + ssf + ssf));
      pe = pe_k;
      s00 = pe_k - pe_k * coeff2 * kx * kx;
      s01 = -pe_k * coeff2 * kx * ky;
      s02 = -pe_k * coeff2 * kx * kz;
      s11 = pe_k - pe_k * coeff2 * ky * ky;
      s12 = -pe_k * coeff2 * ky * kz;
      s22 = pe_k - pe_k * coeff2 * kz * kz;
      double *w = a.w + 4 * (size_t)k;
      w[0] = coeff * (scn + scf);
      w[1] = coeff * (ssn + ssf);
      w[2] = coeff * scn;
      w[3] = coeff * ssn;
   }
   double v[7] = {pe, s00, s01, s02, s11, s12, s22};
   int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
   for (int q = 0; q < 7; q++) {
      double t = wave_sum(v[q]);
      if (lane == 0) ws[wv][q] = t;
   }
   __syncthreads();
   if (threadIdx.x < 7) {
      double t = ws[0][threadIdx.x] + ws[1][threadIdx.x] + ws[2][threadIdx.x] + ws[3][threadIdx.x];
      a.bpart[8 * (size_t)blockIdx.x + threadIdx.x] = t;
   }
}

struct EfArgs {
   int ns, nsp, nsxf, nrows;
   double c2;
   const KRow *rows;
   const int *rpart;        // [npart+1] row ranges of the partitions
   const double *w;
   const double2 *tx, *ty, *tz, *tz1;
   const double2 *ty1;      // row k = 1 of ty (row 0 when kmax = 0, where it is never used)
   double *fpart;           // [npart][3][nsp]
};

// Force back-projection (ewald.c:557-579): one thread per site, the rows
// split over blockIdx.y so that enough waves are resident to hide the
// latency of the l recurrence; partials are summed in a fixed order.
__global__ __launch_bounds__(256) void k_ewald_force(EfArgs a) {
   int i = blockIdx.x * 256 + threadIdx.x;
   if (i >= a.ns) return;
   const int part = blockIdx.y;
   const bool fw = i >= a.nsxf;
   const int wo = fw ? 2 : 0;
   const double2 z1 = a.tz1[i];
   double fx = 0, fy = 0, fz = 0;
   int hcur = -1, kcur = 0;
   double2 xh = make_double2(1, 0), A = make_double2(1, 0);
   const double2 y1 = a.ty1[i];   // exp(i b*.r)
   for (int r = a.rpart[part]; r < a.rpart[part + 1]; r++) {
      const KRow R = a.rows[r];
      if (R.h == hcur && R.k == kcur + 1) {
         A = cmul(A, y1);                 // next k of the same h: exp(i (h a* + k b*).r) by recurrence
      } else {
         if (R.h != hcur) xh = a.tx[(size_t)R.h * a.nsp + i];
         int ak = R.k < 0 ? -R.k : R.k;
         double2 yk = a.ty[(size_t)ak * a.nsp + i];
         if (R.k < 0) yk.y = -yk.y;
         A = cmul(xh, yk);
      }
      hcur = R.h;
      kcur = R.k;
      int al0 = R.l0 < 0 ? -R.l0 : R.l0;
      double2 z = a.tz[(size_t)al0 * a.nsp + i];
      if (R.l0 < 0) z.y = -z.y;
      const double *w = a.w + 4 * (size_t)R.kstart + wo;
      // along the run of l: e = q exp(i k.r) advanced by exp(i c*.r), and
      // sum_l kz_l fc_l = (kzt + l0 c2) sum fc + c2 sum (l - l0) fc
      double2 e = cmul(A, z);
      double sf = 0, sq = 0, dq = 0;
      for (int q = 0; q < R.nl; q++) {
         const double wc = w[4 * q], wsn = w[4 * q + 1];
         const double fc = e.y * wc - e.x * wsn;
         sf += fc;
         sq += dq * fc;
         dq += 1.0;
         e = cmul(e, z1);
      }
      fx += R.kx * sf;
      fy += R.ky * sf;
      fz += (R.kzt + R.l0 * a.c2) * sf + a.c2 * sq;
   }
   double *fp = a.fpart + (size_t)part * 3 * a.nsp;
   fp[i] = fx;
   fp[a.nsp + i] = fy;
   fp[2 * a.nsp + i] = fz;
}

// ---------------- back-projection on the FP64 matrix cores
// With P[r,i] = sum_l Z[l,i] conj W[r,l] and Q[r,i] = sum_l l Z[l,i] conj W[r,l]
// over the row's run of l (ewald.c:557-566), the force is
//   F_i = sum_r Im(A[r,i] ((kx, ky, kzt)(r) P[r,i] + (0, 0, c2) Q[r,i])),
// A[r,i] = exp(i(h a* + k b*).r_i).  As Z[-l] = conj Z[l], the columns are
// l >= 0 only: the K = 2 NC real columns are Zr[0..NC) then Zi[0..NC), and the
// weights of W[r,+l] and W[r,-l] fold onto them (four kinds: Re P, Im P,
// Re Q, Im Q).  v_mfma_f64_16x16x4f64 with the weights as the A operand
// (row = lane % 16, column 4s + lane / 16) and Z as the B operand (site =
// lane % 16) leaves rows lane/16 + 4v of one site in item v, so each lane
// sums the forces of one site.

// Z operand, site-major: row i = Zr[0..NC) then Zi[0..NC) of site i (zeros
// past lmax and past ns), one 64-site tile per block through LDS.
__global__ __launch_bounds__(64) void k_zt64(int ns, int nsp, int lmax, int nc, const double2 *__restrict__ tz,
                                             double *__restrict__ zt) {
   extern __shared__ double szt[];   // [64][2 nc + 1]
   const int K2 = 2 * nc, RS = K2 + 1, base = blockIdx.x * 64, t = threadIdx.x, i = base + t;
   for (int l = 0; l < nc; l++) {
      double2 z = make_double2(0, 0);
      if (l <= lmax && i < ns) z = tz[(size_t)l * nsp + i];
      szt[t * RS + l] = z.x;
      szt[t * RS + nc + l] = z.y;
   }
   __syncthreads();
   for (int q = t; q < 64 * K2; q += 64) {
      const int row = q / K2, c = q - row * K2;
      zt[(size_t)(base + row) * K2 + c] = szt[row * RS + c];
   }
}

// Folded weight operands, lane-ordered: element [kind][tile][s][g][lc] is
// kind's weight of row 16 tile + lc at column 4 s + g.  wo selects the
// per-k weights (Wc, Ws) or, for framework sites, (Wcn, Wsn).
__global__ void k_w64(int nrows, int nrows16, int nc, int ksteps, int wo, const KRow *__restrict__ rows,
                      const double *__restrict__ w, double *__restrict__ wt) {
   const int K2 = 2 * nc;
   const int idx = blockIdx.x * blockDim.x + threadIdx.x;
   if (idx >= nrows16 * K2) return;
   const int r = idx / K2, kk = idx - r * K2;
   const int part = kk >= nc, l = kk - part * nc;
   double wpr = 0, wpi = 0, wmr = 0, wmi = 0;
   if (r < nrows) {
      const KRow R = rows[r];
      if (l >= R.l0 && l < R.l0 + R.nl) {
         const double *q = w + 4 * (size_t)(R.kstart + l - R.l0) + wo;
         wpr = q[0];
         wpi = q[1];
      }
      if (l > 0 && -l >= R.l0 && -l < R.l0 + R.nl) {
         const double *q = w + 4 * (size_t)(R.kstart - l - R.l0) + wo;
         wmr = q[0];
         wmi = q[1];
      }
   }
   double v[4];
   if (!part) { v[0] = wpr + wmr; v[1] = -(wpi + wmi); v[2] = l * (wpr - wmr); v[3] = l * (wmi - wpi); }
   else { v[0] = wpi - wmi; v[1] = wpr - wmr; v[2] = l * (wpi + wmi); v[3] = l * (wpr + wmr); }
   const int tile = r >> 4, lc = r & 15, s = kk >> 2, g = kk & 3;
   const size_t ntile = (size_t)nrows16 / 16;
#pragma unroll
   for (int kind = 0; kind < 4; kind++)
      wt[((kind * ntile + tile) * ksteps + s) * 64 + g * 16 + lc] = v[kind];
}

struct Ef64Args {
   int s0, s1, nsp, nrows, nrows16, kmax, nparts;
   double c2;
   const KRow *rows;
   const double *zt;      // [nsp][4 KST]
   const double *wt;      // [4][ntile][KST][64]
   const double2 *tx, *ty;
   double *fpart;         // [nparts][3][nsp]
};

// Four waves of 32 sites (two 16-site tiles) per workgroup, the row tiles of
// one partition (blockIdx.x % nparts, consecutive workgroups on different
// partitions so that each XCD's L2 keeps one partition's weights).  Per row
// tile: 8 KST MFMAs, then the epilogue, where each lane advances
// A = exp(i(h a* + k b*).r) of its four rows at its site by exp(16 i b*.r)
// along a run of one h, or takes it from the tables at a new run.
template <int KST>
__global__ __launch_bounds__(256) void k_force64(Ef64Args a) {
   constexpr int K2 = 4 * KST;
   const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4, lc = lane & 15;
   const int part = blockIdx.x % a.nparts;
   const int base = a.s0 + (blockIdx.x / a.nparts) * 128 + 32 * wave;
   const int ntile_all = a.nrows16 / 16;
   const int rt0 = part * ntile_all / a.nparts, rt1 = (part + 1) * ntile_all / a.nparts;
   int site[2];
   double zb[2][KST];
   double2 y16[2];
#pragma unroll
   for (int m = 0; m < 2; m++) {
      const int i = base + 16 * m + lc;
      site[m] = i < a.s1 ? i : a.s1 - 1;   // past s1: the last site again, never stored
      const double *zr = a.zt + (size_t)site[m] * K2 + g;
#pragma unroll
      for (int s = 0; s < KST; s++) zb[m][s] = zr[4 * s];
      y16[m] = a.kmax >= 16 ? a.ty[(size_t)16 * a.nsp + site[m]] : make_double2(1, 0);
   }
   double f[2][3] = {{0, 0, 0}, {0, 0, 0}};
   double2 ph[2][4];
   int cur_h[4], cur_k[4];
#pragma unroll
   for (int v = 0; v < 4; v++) {
      cur_h[v] = -1;
      cur_k[v] = 0;
      ph[0][v] = ph[1][v] = make_double2(1, 0);
   }
   const size_t kstride = (size_t)ntile_all * KST * 64;
   for (int rt = rt0; rt < rt1; rt++) {
      dbl4 acc[2][4];
#pragma unroll
      for (int m = 0; m < 2; m++)
#pragma unroll
         for (int kd = 0; kd < 4; kd++) acc[m][kd] = dbl4{0, 0, 0, 0};
      const double *wb = a.wt + (size_t)rt * KST * 64 + lane;
#pragma unroll
      for (int s = 0; s < KST; s++) {
         double wv[4];
#pragma unroll
         for (int kd = 0; kd < 4; kd++) wv[kd] = wb[kd * kstride + s * 64];
#pragma unroll
         for (int kd = 0; kd < 4; kd++)
#pragma unroll
            for (int m = 0; m < 2; m++)
               acc[m][kd] = __builtin_amdgcn_mfma_f64_16x16x4f64(wv[kd], zb[m][s], acc[m][kd], 0, 0, 0);
      }
#pragma unroll
      for (int v = 0; v < 4; v++) {
         const int r = rt * 16 + g + 4 * v;
         if (r >= a.nrows) continue;
         const KRow R = a.rows[r];
         if (R.h == cur_h[v] && R.k == cur_k[v] + 16) {
#pragma unroll
            for (int m = 0; m < 2; m++) ph[m][v] = cmul(ph[m][v], y16[m]);
         } else {
            const int ak = R.k < 0 ? -R.k : R.k;
#pragma unroll
            for (int m = 0; m < 2; m++) {
               const double2 x = a.tx[(size_t)R.h * a.nsp + site[m]];
               double2 y = a.ty[(size_t)ak * a.nsp + site[m]];
               if (R.k < 0) y.y = -y.y;
               ph[m][v] = cmul(x, y);
            }
         }
         cur_h[v] = R.h;
         cur_k[v] = R.k;
#pragma unroll
         for (int m = 0; m < 2; m++) {
            const double Ar = ph[m][v].x, Ai = ph[m][v].y;
            const double t1 = Ar * acc[m][1][v] + Ai * acc[m][0][v];
            const double t2 = Ar * acc[m][3][v] + Ai * acc[m][2][v];
            f[m][0] += R.kx * t1;
            f[m][1] += R.ky * t1;
            f[m][2] += R.kzt * t1 + a.c2 * t2;
         }
      }
   }
   // the four lanes of a site (g = 0..3) hold rows g + 4v: sum them
#pragma unroll
   for (int m = 0; m < 2; m++)
#pragma unroll
      for (int c = 0; c < 3; c++) {
         double t = f[m][c];
         t += __shfl_xor(t, 16, 64);
         t += __shfl_xor(t, 32, 64);
         f[m][c] = t;
      }
   if (g == 0) {
#pragma unroll
      for (int m = 0; m < 2; m++) {
         const int i = base + 16 * m + lc;
         if (i < a.s1) {
            double *fp = a.fpart + (size_t)part * 3 * a.nsp;
            fp[i] = f[m][0];
            fp[a.nsp + i] = f[m][1];
            fp[2 * a.nsp + i] = f[m][2];
         }
      }
   }
}

__global__ void k_add_parts(int ns, int nsp, int npart, const double *__restrict__ fpart,
                            double *__restrict__ force) {
   int i = blockIdx.x * 256 + threadIdx.x;
   if (i >= ns) return;
   for (int c = 0; c < 3; c++) {
      double s = 0.0;
      for (int p = 0; p < npart; p++) s += fpart[((size_t)p * 3 + c) * nsp + i];
      force[(size_t)c * nsp + i] += s;
   }
}


}  // namespace

// ---------------- the FP64 reciprocal pass on explicit storage
// The pass runs on one set of device buffers: the engine's own (mgpu_ewald,
// eval_forces, the adjoint), or regions of the library's static scratch
// array (mgpu_ewald_noalloc).  Both launch the same kernels with the same
// shapes, so their results are bit-identical.
namespace {

struct Ew64Geom {
   int ns, nsp, nsxf, nk, nrows, hmax, kmax, lmax;
   double hinv[9], vol, alpha;
};

struct Ew64Bufs {
   const double *site;           // [3][nsp]
   const double *w;              // [nsp] z-table weights (the charges)
   double *force;                // [3][nsp], accumulated
   const KRow *rows;             // [nrows]
   const int *krow;              // [nk]
   const int *rpart;             // [npart + 1] row partitions
   int npart;
   double2 *tx, *ty, *tz;        // trig tables
   double *sk;                   // S(k) chunk partials
   double *wk;                   // [nk][4] weights
   double *red;                  // [nkb][8] per-block energy/stress sums
   double *out;                  // [7] pe, stress upper triangle
   double *fpart, *zt64, *w64;   // back-projection partials and operands
   double *rtmp;                 // reduction partials
   unsigned *count;              // reduction completion count (zero between passes)
   bool prof;                    // event timing of the stages
};

// Element counts of every buffer of one pass (nch S(k) chunks).
struct Ew64Sizes {
   size_t tx, ty, tz, sk, wk, red, rtmp, fpart, zt64, w64;
   int nch, nkb, kst;
};

int sk_chunks(int ncu, int nrows, int ns) {
   const int nrb = (nrows + 63) / 64;
   int nch = (4 * ncu + nrb - 1) / std::max(nrb, 1);
   nch = std::min(nch, std::max(8, ns / 256));
   return std::max(8, (nch + 7) / 8 * 8);
}

// Column steps of the matrix-core back-projection for this lmax (2 KST >=
// lmax + 1 columns of each of Zr and Zi), or 0 past lmax 47, where the
// per-site walk runs instead.
int force64_ksteps(int lmax) {
   for (int kst : {8, 12, 16, 20, 24})
      if (2 * kst >= lmax + 1) return kst;
   return 0;
}

Ew64Sizes ew64_sizes(const Ew64Geom &g, int ncu, int npart) {
   Ew64Sizes z;
   const size_t nsp = g.nsp;
   z.tx = (g.hmax + 1) * nsp;
   z.ty = (g.kmax + 1) * nsp;
   z.tz = (g.lmax + 1) * nsp + nsp;
   z.nch = sk_chunks(ncu, g.nrows, g.ns);
   z.sk = (size_t)z.nch * g.nk * 4 + 4;
   z.wk = (size_t)g.nk * 4 + 4;
   z.nkb = (g.nk + 255) / 256;
   z.red = (size_t)z.nkb * 8 + 16;
   z.rtmp = (size_t)reduce_cols_blocks(z.nkb) * 8 + 16;
   z.kst = force64_ksteps(g.lmax);
   if (z.kst == 0) {
      z.fpart = (size_t)npart * 3 * nsp;
      z.zt64 = z.w64 = 0;
   } else {
      const int K2 = 4 * z.kst, nrows16 = (g.nrows + 15) / 16 * 16, ntile = nrows16 / 16;
      const int nparts = std::max(1, std::min(npart, ntile));
      z.fpart = (size_t)nparts * 3 * nsp;
      z.zt64 = nsp * K2;
      z.w64 = (size_t)(g.nsxf < g.ns ? 2 : 1) * 4 * nrows16 * K2;
   }
   return z;
}

// Row partitions of the force pass with about equal numbers of k vectors.
std::vector<int> row_partition(const std::vector<KRow> &rows, int nk, int want) {
   const int nrows = (int)rows.size();
   const int npart = std::max(1, std::min(want, nrows / 8));
   std::vector<int> rp(npart + 1, nrows);
   rp[0] = 0;
   int p = 1;
   for (int q = 0; q < nrows && p < npart; q++)
      if ((long)rows[q].kstart * npart >= (long)p * nk) rp[p++] = q;
   for (; p < npart; p++) rp[p] = nrows;
   return rp;
}

// Trig tables (FP64) for the sites, the z table weighted by b.w.
void ew64_tables(mgpu_engine *e, const Ew64Geom &g, const Ew64Bufs &b) {
   TrigArgs t;
   for (int i = 0; i < 9; i++) t.ks[i] = 2 * PI_D * g.hinv[i];
   t.hmax = g.hmax; t.kmax = g.kmax; t.lmax = g.lmax; t.ns = g.ns; t.nsp = g.nsp;
   ProfScope ps(b.prof ? e : nullptr, "ewald_trig");
   k_trig<<<(g.ns + 255) / 256, 256, 0, e->stream>>>(t, b.site, b.w, b.tx, b.ty, b.tz,
                                                   b.tz + (size_t)(g.lmax + 1) * g.nsp);
}

// S(k) chunk partials of the trig tables into b.sk, sites from nsxf on
// counted as framework; returns the number of chunks.  About four
// workgroups per CU in all, chunks of at least 256 sites, a multiple of 8
// chunks (one XCD each).
int ew64_sfac(mgpu_engine *e, const Ew64Geom &g, const Ew64Bufs &b, int nsxf) {
   const int ns = g.ns, nrb = (g.nrows + 63) / 64;
   const int nch = sk_chunks(e->ncu, g.nrows, ns);
   int ncb = 0;
   if (nsxf == 0)
      ncb = nch;
   else if (nsxf < ns)
      ncb = std::min(nch - 1, std::max(1, (int)std::lround((double)nch * (ns - nsxf) / ns)));
   SkArgs s;
   s.nk = g.nk; s.ns = ns; s.nsp = g.nsp; s.nsxf = nsxf; s.nrows = g.nrows; s.lmax = g.lmax;
   s.nca = nch - ncb; s.ncb = ncb; s.nrb = nrb;
   s.rows = b.rows; s.tx = b.tx; s.ty = b.ty; s.tz = b.tz; s.part = b.sk;
   const int ncol = g.lmax + 1;
   const dim3 grid(nrb * nch, (ncol + 47) / 48);
   switch (std::min(3, (ncol + 15) / 16)) {
   case 1: k_sfac<1><<<grid, 256, 0, e->stream>>>(s); break;
   case 2: k_sfac<2><<<grid, 256, 0, e->stream>>>(s); break;
   default: k_sfac<3><<<grid, 256, 0, e->stream>>>(s); break;
   }
   return nch;
}

// b.force[3][nsp] += the back-projection of the weights b.wk over the trig
// tables (sites from nsxf on with the framework weights), summed over the
// row partitions in partition order; join_side before the sum when asked
// (the real-space pass on the side stream adds into the same forces).
void ew64_backproject(mgpu_engine *e, const Ew64Geom &g, const Ew64Bufs &b, int nsxf, double *out, bool join) {
   const int ns = g.ns, nsp = g.nsp;
   const int kst = force64_ksteps(g.lmax);
   if (kst == 0) {
      const int npart = b.npart;
      EfArgs ef;
      ef.ns = ns; ef.nsp = nsp; ef.nsxf = nsxf; ef.nrows = g.nrows;
      ef.c2 = 2 * PI_D * g.hinv[8];
      ef.rows = b.rows; ef.rpart = b.rpart; ef.w = b.wk;
      ef.tx = b.tx; ef.ty = b.ty; ef.tz = b.tz;
      ef.tz1 = b.tz + (size_t)(g.lmax + 1) * nsp;
      ef.ty1 = b.ty + (g.kmax > 0 ? nsp : 0);
      ef.fpart = b.fpart;
      dim3 grid((ns + 255) / 256, npart);
      k_ewald_force<<<grid, 256, 0, e->stream>>>(ef);
      if (join) join_side(e);
      k_add_parts<<<(ns + 255) / 256, 256, 0, e->stream>>>(ns, nsp, npart, b.fpart, out);
      return;
   }
   const int nc = 2 * kst, K2 = 4 * kst;
   const int nrows16 = (g.nrows + 15) / 16 * 16, ntile = nrows16 / 16;
   const int nparts = std::max(1, std::min(b.npart, ntile));
   k_zt64<<<nsp / 64, 64, sizeof(double) * 64 * (K2 + 1), e->stream>>>(ns, nsp, g.lmax, nc, b.tz, b.zt64);
   const size_t wsz = (size_t)4 * nrows16 * K2;
   const bool fw = nsxf < ns;
   const int nw = (nrows16 * K2 + 255) / 256;
   k_w64<<<nw, 256, 0, e->stream>>>(g.nrows, nrows16, nc, kst, 0, b.rows, b.wk, b.w64);
   if (fw) k_w64<<<nw, 256, 0, e->stream>>>(g.nrows, nrows16, nc, kst, 2, b.rows, b.wk, b.w64 + wsz);
   Ef64Args a;
   a.nsp = nsp; a.nrows = g.nrows; a.nrows16 = nrows16; a.kmax = g.kmax; a.nparts = nparts;
   a.c2 = 2 * PI_D * g.hinv[8];
   a.rows = b.rows; a.zt = b.zt64; a.tx = b.tx; a.ty = b.ty; a.fpart = b.fpart;
   auto run = [&](int s0, int s1, const double *wt) {
      if (s1 <= s0) return;
      a.s0 = s0; a.s1 = s1; a.wt = wt;
      const dim3 grid((unsigned)(((s1 - s0 + 127) / 128) * nparts));
      switch (kst) {
      case 8: k_force64<8><<<grid, 256, 0, e->stream>>>(a); break;
      case 12: k_force64<12><<<grid, 256, 0, e->stream>>>(a); break;
      case 16: k_force64<16><<<grid, 256, 0, e->stream>>>(a); break;
      case 20: k_force64<20><<<grid, 256, 0, e->stream>>>(a); break;
      default: k_force64<24><<<grid, 256, 0, e->stream>>>(a); break;
      }
   };
   run(0, nsxf, b.w64);
   run(nsxf, ns, fw ? b.w64 + wsz : b.w64);
   if (join) join_side(e);
   k_add_parts<<<(ns + 255) / 256, 256, 0, e->stream>>>(ns, nsp, nparts, b.fpart, out);
}

// The whole pass: tables, S(k), per-k energy/stress/weights, their sums
// into b.out[0..6], and the forces into b.force.
void ew64_pass(mgpu_engine *e, const Ew64Geom &g, const Ew64Bufs &b, bool join) {
   ew64_tables(e, g, b);
   int nchunks;
   {
      ProfScope ps(b.prof ? e : nullptr, "ewald_sfac");
      nchunks = ew64_sfac(e, g, b, g.nsxf);
   }
   const int nkb = (g.nk + 255) / 256;
   EkArgs ek;
   ek.nk = g.nk; ek.nchunks = nchunks; ek.nrows = g.nrows;
   ek.vol = g.vol;
   ek.r4a = -1.0 / (4.0 * g.alpha * g.alpha);
   ek.c2 = 2 * PI_D * g.hinv[8];
   ek.rows = b.rows; ek.krow = b.krow; ek.part = b.sk; ek.w = b.wk;
   ek.bpart = b.red;
   {
      ProfScope ps(b.prof ? e : nullptr, "ewald_kspace");
      k_ewald_k<<<nkb, 256, 0, e->stream>>>(ek);
   }
   reduce_cols_into(nullptr, e->stream, b.red, nkb, 8, b.out, b.rtmp, b.count);
   {
      ProfScope ps(b.prof ? e : nullptr, "ewald_force");
      ew64_backproject(e, g, b, g.nsxf, b.force, join);
   }
}

Ew64Geom engine_geom(const mgpu_engine *e) {
   Ew64Geom g;
   g.ns = e->nsites; g.nsp = e->nsp; g.nsxf = e->nsitesxf; g.nk = e->nk; g.nrows = e->nrows;
   g.hmax = e->hmax; g.kmax = e->kmax; g.lmax = e->lmax;
   for (int i = 0; i < 9; i++) g.hinv[i] = e->hinv[i];
   g.vol = host_det(e->h);
   g.alpha = e->alpha;
   return g;
}

}  // namespace

// Row partitions of the force pass, a host table uploaded when the k set
// changes
static void ewald_plan(mgpu_engine *e) {
   if (e->ew_plan_version != e->geom_version) {
      const std::vector<int> rp = row_partition(e->rows, e->nk, e->tune_npart);
      const int npart = (int)rp.size() - 1;
      e->d_rpart.reserve(npart + 1);
      HIPCHK(hipMemcpyAsync(e->d_rpart.p, rp.data(), sizeof(int) * (npart + 1), hipMemcpyHostToDevice, e->stream));
      HIPCHK(hipStreamSynchronize(e->stream));
      e->ew_npart = npart;
      e->ew_plan_version = e->geom_version;
   }
}

// The engine's buffers for a pass with z-table weights w, sized for its
// geometry (the reduction storage is d_rtmp, as reduce_cols uses it).
static Ew64Bufs engine_bufs(mgpu_engine *e, const Ew64Geom &g, const double *w) {
   const Ew64Sizes z = ew64_sizes(g, e->ncu, e->ew_npart);
   e->d_tx.reserve(z.tx);
   e->d_ty.reserve(z.ty);
   e->d_tz.reserve(z.tz);
   e->d_sk.reserve(z.sk);
   e->d_wk.reserve(z.wk);
   e->d_red.reserve(z.red);
   e->d_fpart.reserve(z.fpart);
   if (z.zt64) e->d_zt64.reserve(z.zt64);
   if (z.w64) e->d_w64.reserve(z.w64);
   e->d_out.reserve(OUT_SIZE);
   if (e->d_rtmp.reserve(z.rtmp + 1)) zero_async(e, e->d_rtmp.p, 8);
   Ew64Bufs b;
   b.site = e->d_site.p; b.w = w; b.force = e->d_force_site.p;
   b.rows = e->d_rows.p; b.krow = e->d_krow.p; b.rpart = e->d_rpart.p; b.npart = e->ew_npart;
   b.tx = e->d_tx.p; b.ty = e->d_ty.p; b.tz = e->d_tz.p;
   b.sk = e->d_sk.p; b.wk = e->d_wk.p; b.red = e->d_red.p; b.out = e->d_out.p + OUT_RECIP;
   b.fpart = e->d_fpart.p; b.zt64 = e->d_zt64.p; b.w64 = e->d_w64.p;
   b.count = (unsigned *)e->d_rtmp.p; b.rtmp = e->d_rtmp.p + 1;
   b.prof = true;
   return b;
}

// Engine-bound forms used by the charge adjoint: tables weighted by w, the
// S(k) partials, and the back-projection of d_wk into out.
static void ewald_tables(mgpu_engine *e, const double *w) {
   const Ew64Geom g = engine_geom(e);
   ew64_tables(e, g, engine_bufs(e, g, w));
}

static int sfac_partials(mgpu_engine *e, int nsxf) {
   const Ew64Geom g = engine_geom(e);
   return ew64_sfac(e, g, engine_bufs(e, g, e->d_chg_site.p), nsxf);
}

static void backproject_fp64(mgpu_engine *e, int nsxf, double *out, bool join) {
   const Ew64Geom g = engine_geom(e);
   ew64_backproject(e, g, engine_bufs(e, g, e->d_chg_site.p), nsxf, out, join);
}

void mgpu::run_ewald_fp64(mgpu_engine *e) {
   ewald_plan(e);
   const Ew64Geom g = engine_geom(e);
   ew64_pass(e, g, engine_bufs(e, g, e->d_chg_site.p), true);
}

// ---------------- the pass without allocation (mgpu_ewald_noalloc)
// Its device storage is one fixed array in the code object: each GPU the
// library runs on holds its own copy until the process ends.  Host code
// never uses the array's name as an address (in host code it is only a
// stand-in); it uses the device address hipGetSymbolAddress returns for
// each device, taken once per device by scratch_init.  Every call on a GPU
// shares that GPU's copy and leaves its contents behind: what must start at
// zero (the reduction's completion count) is cleared by a kernel at every
// call, and calls that overlap on one GPU race.
static __device__ __align__(256) unsigned char scratch[MGPU_NOALLOC_BYTES];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
unsigned char *g_scratch_dev[kMaxDevices] = {};
}  // namespace

void mgpu::scratch_init(int device) {
   if (device < 0 || device >= kMaxDevices) throw StatusError{MGPU_E_ARG, "device index out of range"};
   std::lock_guard<std::mutex> lock(g_scratch_mu);
   if (g_scratch_dev[device]) return;
   void *p = nullptr;
   HIPCHK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
   g_scratch_dev[device] = (unsigned char *)p;
}

void mgpu::ewald_noalloc(mgpu_engine *e, const double h[9], const double *site, int ld, const double *chg,
                         double *site_force, double out7[7], mgpu_ew_info *info) {
   unsigned char *base = nullptr;
   {
      std::lock_guard<std::mutex> lock(g_scratch_mu);
      if (e->device >= 0 && e->device < kMaxDevices) base = g_scratch_dev[e->device];
   }
   if (!base) throw StatusError{MGPU_E_STATE, "no scratch address for this device (mgpu_create not called)"};
   Ew64Geom g;
   host_invert(h, g.hinv);
   KSet ks;
   build_kset(h, g.hinv, e->k_cutoff, ks);
   const std::vector<int> rp = row_partition(ks.rows, ks.nk, e->tune_npart);
   const int npart = (int)rp.size() - 1;
   g.ns = e->nsites; g.nsp = e->nsp; g.nsxf = e->nsitesxf; g.nk = ks.nk; g.nrows = (int)ks.rows.size();
   g.hmax = ks.hmax; g.kmax = ks.kmax; g.lmax = ks.lmax;
   g.vol = host_det(h);
   g.alpha = e->alpha;
   // the same choice of sum as mgpu_ewald's, unless only the direct sum's buffers fit
   const GridGeom gg = grid_geom(g.ns, g.nsp, g.hmax, g.kmax, g.lmax, h, g.hinv, g.vol, g.alpha, e->k_cutoff, true);
   const GridSizes gz = grid_sizes(gg);
   bool grid = gz.bytes <= (size_t)MGPU_NOALLOC_BYTES && grid_applies(gg, g.nsxf, g.nk, e->k_cutoff, ks.rows);
   std::shared_ptr<const GridTables> gt;
   std::vector<int> gmap;
   if (grid) {
      gt = grid_host_tables(e, gg);
      grid_rowmap(gg, ks.rows, gmap);
   }
   const Ew64Sizes z = ew64_sizes(g, e->ncu, npart);
   // the regions, 256-byte aligned
   const size_t nsp = g.nsp;
   size_t off = 0, oSite, oForce, oChg, oRows, oOut, oRtmp, oKrow = 0, oRpart = 0, oTx = 0, oTy = 0, oTz = 0, oSk = 0,
          oWk = 0, oRed = 0, oFpart = 0, oZt = 0, oW64 = 0, oGrid = 0, oGtab = 0, oGmap = 0;
   int nred = 0;
   auto carve = [&] {
      off = 0;
      auto take = [&](size_t bytes) {
         const size_t o = off;
         off += (bytes + 255) & ~(size_t)255;
         return o;
      };
      oSite = take(sizeof(double) * 3 * nsp);
      oForce = take(sizeof(double) * 3 * nsp);
      oChg = chg ? take(sizeof(double) * nsp) : 0;
      oRows = take(sizeof(KRow) * (g.nrows + 1));
      oOut = take(sizeof(double) * 8);
      if (grid) {
         oGrid = take(gz.bytes);
         oGtab = take(sizeof(double) * gt->data.size());
         oGmap = take(sizeof(int) * gmap.size());
      } else {
         oKrow = take(sizeof(int) * (g.nk + 1));
         oRpart = take(sizeof(int) * (npart + 1));
         oTx = take(sizeof(double2) * z.tx);
         oTy = take(sizeof(double2) * z.ty);
         oTz = take(sizeof(double2) * z.tz);
         oSk = take(sizeof(double) * z.sk);
         oWk = take(sizeof(double) * z.wk);
         oRed = take(sizeof(double) * z.red);
         oFpart = take(sizeof(double) * z.fpart);
         oZt = take(sizeof(double) * z.zt64);
         oW64 = take(sizeof(double) * z.w64);
      }
      nred = grid ? gz.nred : z.nkb;
      oRtmp = take(sizeof(double) * ((size_t)reduce_cols_blocks(nred) * 8 + 17));
   };
   carve();
   if (grid && off > (size_t)MGPU_NOALLOC_BYTES) {
      grid = false;
      carve();
   }
   if (off > (size_t)MGPU_NOALLOC_BYTES)
      throw StatusError{MGPU_E_CAPACITY, "mgpu_ewald_noalloc: this system needs " + std::to_string(off >> 20) +
                                             " MiB of scratch; the limit is " +
                                             std::to_string(MGPU_NOALLOC_BYTES >> 20) + " MiB"};
   Ew64Bufs b;
   double *dsite = (double *)(base + oSite);
   b.site = dsite;
   b.force = (double *)(base + oForce);
   b.w = chg ? (const double *)(base + oChg) : e->d_chg_site.p;
   b.rows = (const KRow *)(base + oRows);
   b.krow = (const int *)(base + oKrow);
   b.rpart = (const int *)(base + oRpart);
   b.npart = npart;
   b.tx = (double2 *)(base + oTx); b.ty = (double2 *)(base + oTy); b.tz = (double2 *)(base + oTz);
   b.sk = (double *)(base + oSk); b.wk = (double *)(base + oWk); b.red = (double *)(base + oRed);
   b.out = (double *)(base + oOut);
   b.fpart = (double *)(base + oFpart); b.zt64 = (double *)(base + oZt); b.w64 = (double *)(base + oW64);
   b.count = (unsigned *)(base + oRtmp);
   b.rtmp = (double *)(base + oRtmp) + 1;
   b.prof = false;
   hipStream_t st = e->stream;
   zero_async(e, b.count, 8);
   for (int c = 0; c < 3; c++) {
      HIPCHK(hipMemcpyAsync(dsite + c * nsp, site + (size_t)c * ld, sizeof(double) * g.ns, hipMemcpyHostToDevice, st));
      HIPCHK(hipMemcpyAsync(b.force + c * nsp, site_force + (size_t)c * ld, sizeof(double) * g.ns,
                            hipMemcpyHostToDevice, st));
   }
   if (chg) HIPCHK(hipMemcpyAsync(base + oChg, chg, sizeof(double) * g.ns, hipMemcpyHostToDevice, st));
   HIPCHK(hipMemcpyAsync(base + oRows, ks.rows.data(), sizeof(KRow) * g.nrows, hipMemcpyHostToDevice, st));
   if (grid) {
      HIPCHK(hipMemcpyAsync(base + oGtab, gt->data.data(), sizeof(double) * gt->data.size(), hipMemcpyHostToDevice, st));
      HIPCHK(hipMemcpyAsync(base + oGmap, gmap.data(), sizeof(int) * gmap.size(), hipMemcpyHostToDevice, st));
      grid_clear(e, gg, base + oGrid);
      GridBufs gb;
      gb.site = dsite; gb.w = b.w; gb.force = b.force; gb.rows = b.rows; gb.rowmap = (const int *)(base + oGmap);
      gb.tab = (const double *)(base + oGtab); gb.base = base + oGrid; gb.prof = false;
      grid_pass(e, nullptr, gg, *gt, gb, false);
      reduce_cols_into(nullptr, st, (const double *)(base + oGrid + gz.bpart), nred, 8, b.out, b.rtmp, b.count);
   } else {
      HIPCHK(hipMemcpyAsync(base + oKrow, ks.krow.data(), sizeof(int) * g.nk, hipMemcpyHostToDevice, st));
      HIPCHK(hipMemcpyAsync(base + oRpart, rp.data(), sizeof(int) * (npart + 1), hipMemcpyHostToDevice, st));
      ew64_pass(e, g, b, false);
   }
   for (int c = 0; c < 3; c++)
      HIPCHK(hipMemcpyAsync(site_force + (size_t)c * ld, b.force + c * nsp, sizeof(double) * g.ns,
                            hipMemcpyDeviceToHost, st));
   HIPCHK(hipMemcpyAsync(out7, b.out, sizeof(double) * 7, hipMemcpyDeviceToHost, st));
   HIPCHK(hipStreamSynchronize(st));
   if (info) {
      info->hmax = ks.hmax; info->kmax = ks.kmax; info->lmax = ks.lmax; info->nhkl = ks.nk;
      info->nsitesxf = e->nsitesxf;
      info->self_energy = e->self_energy; info->sheet_energy = e->sheet_energy;
   }
}

// ============================ charge adjoint ============================
// With E = 1/2 sum_k coeff (C^2 + S^2), C + iS = sum_j q_j exp(i k.r_j) and
// F_i = q_i sum_k coeff k (C sin_i - S cos_i) (ewald.c:539-579), the charge
// derivatives by site id a use the id-restricted sums C_a + iS_a =
// sum_{j in a} exp(i k.r_j):
//   dE/dq_a       = sum_k coeff (C C_a + S S_a)
//   dF_i/dq_a     = [id_i = a] phi_i + q_i sum_k coeff k (C_a sin_i - S_a cos_i)
// with phi_i = sum_k coeff k (C sin_i - S cos_i), so that for a cotangent v
//   sum_i v_i.dF_i/dq_a = sum_{i in a} v_i.phi_i + sum_k coeff (C_a T_S - S_a T_C),
//   T_C + i T_S = sum_i q_i (v_i.k) exp(i k.r_i).
namespace {

__global__ void k_sf_sum(int nk, int nchunks, const double *__restrict__ part, double2 *__restrict__ out) {
   int k = blockIdx.x * blockDim.x + threadIdx.x;
   if (k >= nk) return;
   double c = 0, s = 0;
   for (int q = 0; q < nchunks; q++) {
      const double *p = part + ((size_t)q * nk + k) * 4;
      c += p[0];
      s += p[1];
   }
   out[k] = make_double2(c, s);
}

struct KcArgs {
   int nk;
   double vol, r4a, c2;
   const KRow *rows;
   const int *krow;
};

// coeff and k of every k vector (ewald.c:506-531)
__global__ void k_kcoeff(KcArgs a, double4 *__restrict__ out) {
   int k = blockIdx.x * blockDim.x + threadIdx.x;
   if (k >= a.nk) return;
   KRow R = a.rows[a.krow[k]];
   int l = R.l0 + (k - R.kstart);
   double kx = R.kx, ky = R.ky, kz = R.kzt + l * a.c2;
   double ksq = kx * kx + ky * ky + kz * kz;
   out[k] = make_double4(kx, ky, kz, 2.0 / ((0.25 / PI_D) * a.vol) * exp(ksq * a.r4a) / ksq);
}

__global__ void k_weights_w(int nk, const double4 *__restrict__ kc, const double2 *__restrict__ cs,
                            double *__restrict__ w) {
   int k = blockIdx.x * blockDim.x + threadIdx.x;
   if (k >= nk) return;
   double c = kc[k].w;
   w[4 * (size_t)k] = c * cs[k].x;
   w[4 * (size_t)k + 1] = c * cs[k].y;
   w[4 * (size_t)k + 2] = c * cs[k].x;
   w[4 * (size_t)k + 3] = c * cs[k].y;
}

__global__ void k_site_weight(int ns, int mode, int id, const int *__restrict__ stype,
                              const double *__restrict__ chg, const double *__restrict__ v, int nsp,
                              double *__restrict__ w) {
   int i = blockIdx.x * blockDim.x + threadIdx.x;
   if (i >= nsp) return;
   double x = 0.0;
   if (i < ns) {
      if (mode == 0) x = stype[i] == id ? 1.0 : 0.0;       // indicator of site id
      else if (mode == 1) x = 1.0;                         // unit weights
      else x = chg[i] * v[(size_t)(mode - 2) * nsp + i];  // q v_x, q v_y, q v_z
   }
   w[i] = x;
}

// per k: columns 2a (dE/dq_a) and 2a+1 (the k part of the cotangent product)
__global__ __launch_bounds__(256) void k_charge_k(int nk, int nid, const double4 *__restrict__ kc,
                                                  const double2 *__restrict__ csq,
                                                  const double2 *__restrict__ csa,
                                                  const double2 *__restrict__ csv, int have_v,
                                                  double *__restrict__ part) {
   __shared__ double ws[4][2 * MGPU_MAX_ID];
   int k = blockIdx.x * 256 + threadIdx.x;
   const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
   double4 K = k < nk ? kc[k] : make_double4(0, 0, 0, 0);
   double2 cq = k < nk ? csq[k] : make_double2(0, 0);
   double tc = 0, tsn = 0;
   if (k < nk && have_v) {
      double2 vx = csv[k], vy = csv[(size_t)nk + k], vz = csv[2 * (size_t)nk + k];
      tc = K.x * vx.x + K.y * vy.x + K.z * vz.x;
      tsn = K.x * vx.y + K.y * vy.y + K.z * vz.y;
   }
   for (int a = 0; a < nid; a++) {
      double2 ca = k < nk ? csa[(size_t)a * nk + k] : make_double2(0, 0);
      double de = K.w * (cq.x * ca.x + cq.y * ca.y);
      double dv = K.w * (ca.x * tsn - ca.y * tc);
      de = wave_sum(de);
      dv = wave_sum(dv);
      if (lane == 0) { ws[w][2 * a] = de; ws[w][2 * a + 1] = dv; }
   }
   __syncthreads();
   if (threadIdx.x < 2 * nid)
      part[(size_t)blockIdx.x * 2 * nid + threadIdx.x] =
          ws[0][threadIdx.x] + ws[1][threadIdx.x] + ws[2][threadIdx.x] + ws[3][threadIdx.x];
}

// per site id a: sum_{i in a} v_i.phi_i
__global__ __launch_bounds__(256) void k_vphi(int ns, int nsp, int nid, const int *__restrict__ stype,
                                              const double *__restrict__ v, const double *__restrict__ phi,
                                              double *__restrict__ part) {
   __shared__ double ws[4][MGPU_MAX_ID];
   int i = blockIdx.x * 256 + threadIdx.x;
   const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
   double x = 0;
   int t = -1;
   if (i < ns) {
      t = stype[i];
      x = v[i] * phi[i] + v[nsp + i] * phi[nsp + i] + v[2 * (size_t)nsp + i] * phi[2 * (size_t)nsp + i];
   }
   for (int a = 0; a < nid; a++) {
      double y = wave_sum(t == a ? x : 0.0);
      if (lane == 0) ws[w][a] = y;
   }
   __syncthreads();
   if (threadIdx.x < nid)
      part[(size_t)blockIdx.x * nid + threadIdx.x] =
          ws[0][threadIdx.x] + ws[1][threadIdx.x] + ws[2][threadIdx.x] + ws[3][threadIdx.x];
}

__global__ void k_colsum(int nrows, int ncols, const double *__restrict__ part, double *__restrict__ out) {
   int c = blockIdx.x * blockDim.x + threadIdx.x;
   if (c >= ncols) return;
   double t = 0;
   for (int r = 0; r < nrows; r++) t += part[(size_t)r * ncols + c];
   out[c] = t;
}

// dS = sum_a dq_a (C_a, S_a)
__global__ void k_dir_sf(int nk, int nid, const double *__restrict__ dq, const double2 *__restrict__ csa,
                         double2 *__restrict__ out) {
   int k = blockIdx.x * blockDim.x + threadIdx.x;
   if (k >= nk) return;
   double c = 0, s = 0;
   for (int a = 0; a < nid; a++) {
      double2 x = csa[(size_t)a * nk + k];
      c += dq[a] * x.x;
      s += dq[a] * x.y;
   }
   out[k] = make_double2(c, s);
}

// jvp_i += dq_{id_i} phi_i
__global__ void k_jvp_phi(int ns, int nsp, const int *__restrict__ stype, const double *__restrict__ dq,
                          const double *__restrict__ phi, double *__restrict__ out) {
   int i = blockIdx.x * blockDim.x + threadIdx.x;
   if (i >= ns) return;
   double d = dq[stype[i]];
   for (int c = 0; c < 3; c++) out[(size_t)c * nsp + i] += d * phi[(size_t)c * nsp + i];
}

}  // namespace

// sum_i w_i exp(i k.r_i) for every k into cs[nk]
static void weighted_sf(mgpu_engine *e, const double *w, double2 *cs) {
   if (grid_weighted_sf(e, w, cs)) return;
   ewald_tables(e, w);
   const int nchunks = sfac_partials(e, e->nsites);
   k_sf_sum<<<(e->nk + 255) / 256, 256, 0, e->stream>>>(e->nk, nchunks, e->d_sk.p, cs);
}

// out[3][nsp] += w_i sum_k coeff k (C sin_i - S cos_i) with (C, S) = cs
static void backproject(mgpu_engine *e, const double *w, const double4 *kc, const double2 *cs, double *out) {
   if (grid_backproject(e, w, kc, cs, out)) return;
   e->d_wk.reserve((size_t)e->nk * 4 + 4);
   k_weights_w<<<(e->nk + 255) / 256, 256, 0, e->stream>>>(e->nk, kc, cs, e->d_wk.p);
   ewald_tables(e, w);
   backproject_fp64(e, e->nsites, out, false);
}

void mgpu::ewald_charge_adjoint(mgpu_engine *e, const double *v, const double *dq_dev, double *dE, double *vjp,
                                double *jvp) {
   if (e->nsitesxf < e->nsites)
      throw StatusError{MGPU_E_CAPACITY, "charge derivatives of the Ewald sum with a framework"};
   ewald_plan(e);
   const int nk = e->nk, nid = e->max_id, nsp = e->nsp, ns = e->nsites;
   const int nb = (nsp + 255) / 256;
   // scratch: coeff/k, C+iS for q, each id, q v_x..z, direction; phi; weights;
   // partial sums and the sums per id
   size_t off = 0;
   auto take = [&](size_t bytes) { size_t o = off; off += (bytes + 255) & ~(size_t)255; return o; };
   const size_t oKc = take(sizeof(double4) * nk), oQ = take(sizeof(double2) * nk),
                oA = take(sizeof(double2) * nk * (size_t)nid), oV = take(sizeof(double2) * nk * 3),
                oD = take(sizeof(double2) * nk), oPhi = take(sizeof(double) * 3 * nsp),
                oW = take(sizeof(double) * nsp), oP = take(sizeof(double) * (size_t)std::max(nk, nsp) / 256 * 2 * nid + 64 * nid),
                oO = take(sizeof(double) * 2 * nid);
   e->d_adj.reserve(off);
   uint8_t *B = e->d_adj.p;
   double4 *kc = (double4 *)(B + oKc);
   double2 *csq = (double2 *)(B + oQ), *csa = (double2 *)(B + oA), *csv = (double2 *)(B + oV),
           *csd = (double2 *)(B + oD);
   double *phi = (double *)(B + oPhi), *w = (double *)(B + oW), *part = (double *)(B + oP), *outc = (double *)(B + oO);
   KcArgs ka{nk, host_det(e->h), -1.0 / (4.0 * e->alpha * e->alpha), 2 * PI_D * e->hinv[8], e->d_rows.p, e->d_krow.p};
   k_kcoeff<<<(nk + 255) / 256, 256, 0, e->stream>>>(ka, kc);
   weighted_sf(e, e->d_chg_site.p, csq);
   // an id without sites (id 0 in every Moldy system) has zero sums
   std::vector<char> used(nid, 0);
   for (int t : e->site_type) used[t] = 1;
   zero_async(e, csa, sizeof(double2) * nk * (size_t)nid);
   for (int a = 0; a < nid; a++) {
      if (!used[a]) continue;
      k_site_weight<<<nb, 256, 0, e->stream>>>(ns, 0, a, e->d_site_type.p, e->d_chg_site.p, nullptr, nsp, w);
      weighted_sf(e, w, csa + (size_t)a * nk);
   }
   if (v)
      for (int c = 0; c < 3; c++) {
         k_site_weight<<<nb, 256, 0, e->stream>>>(ns, 2 + c, 0, e->d_site_type.p, e->d_chg_site.p, v, nsp, w);
         weighted_sf(e, w, csv + (size_t)c * nk);
      }
   // phi_i: unit site weights against the charges' structure factors
   zero_async(e, phi, sizeof(double) * 3 * nsp);
   k_site_weight<<<nb, 256, 0, e->stream>>>(ns, 1, 0, e->d_site_type.p, e->d_chg_site.p, nullptr, nsp, w);
   backproject(e, w, kc, csq, phi);
   // dE/dq and the k part of the cotangent product
   const int nkb = (nk + 255) / 256;
   k_charge_k<<<nkb, 256, 0, e->stream>>>(nk, nid, kc, csq, csa, csv, v != nullptr, part);
   k_colsum<<<1, 64, 0, e->stream>>>(nkb, 2 * nid, part, outc);
   std::vector<double> h2(2 * nid), hv(nid, 0.0);
   HIPCHK(hipMemcpyAsync(h2.data(), outc, sizeof(double) * 2 * nid, hipMemcpyDeviceToHost, e->stream));
   HIPCHK(hipStreamSynchronize(e->stream));
   if (v) {
      k_vphi<<<nb, 256, 0, e->stream>>>(ns, nsp, nid, e->d_site_type.p, v, phi, part);
      k_colsum<<<1, 64, 0, e->stream>>>(nb, nid, part, outc);
      HIPCHK(hipMemcpyAsync(hv.data(), outc, sizeof(double) * nid, hipMemcpyDeviceToHost, e->stream));
      HIPCHK(hipStreamSynchronize(e->stream));
   }
   for (int a = 0; a < nid; a++) {
      if (dE) dE[a] = h2[2 * a];
      if (vjp) vjp[a] = h2[2 * a + 1] + hv[a];
   }
   if (jvp && dq_dev) {
      k_dir_sf<<<nkb, 256, 0, e->stream>>>(nk, nid, dq_dev, csa, csd);
      backproject(e, e->d_chg_site.p, kc, csd, jvp);
      k_jvp_phi<<<(ns + 255) / 256, 256, 0, e->stream>>>(ns, nsp, e->d_site_type.p, dq_dev, phi, jvp);
   }
}
