// Real-space site-site forces (the work of force_inner + kernel + mk_forces,
// src/force.c:784-1005, src/kernel.c:157-463).
//
// Each site gathers its interactions with every site in the full neighbour
// shell of its cell (the reference's half-shell offsets plus their mirror
// images), so each unordered pair is evaluated from both ends and no
// atomics are needed.  The pair set is the
// reference's: pair (i,j) is present iff j lies in a cell offset by a
// half-shell vector from i's cell (or the reverse), j != i, and not both are
// framework sites (src/force.c:541-566, 904-912).  Energies and the virial
// are accumulated once per visit with weight 1/2; the virial is the pair form
// sum f r_a r_b, which equals the reference's sum r_i F_i + sum R_n g_n
// (src/force.c:973-997) when site_force starts at zero.
//
// Link cells hold about one site at the reference's subcell (r_c/5), so
// the work is spread as one thread per (site, part of the shell): many
// short, independent loops over L2-resident cell-ordered positions keep
// enough waves in flight to hide the gather latency.  The number of parts
// (4 to 256) grows as the system shrinks, so small boxes still fill the GPU.
#include "mgpu_internal.h"
#include "mgpu_pair.h"

#include <type_traits>

using namespace mgpu;

namespace {

struct RSArgs {
   int ncells, nx, ny, nz, nfull, max_id, nsp, strict_sub;
   int lognq;          // log2 of the shell parts per site
   int skip_intra_u;   // FP32: drop minimum-image intramolecular pair energies
   double alpha, norm, cutsq, cut100sq, half_box_sq;
   double reloc[81];
   const int *css;
   const int4 *off;
   const float4 *offD;
   const double4 *cpos;
   const float4 *cposf;
   const int2 *cmeta;
   const int *corig;
   const int *ccell;
   int nsites;
   // z-columns of the shell for the load-balanced pass
   int ncol, own_col;
   int bit_words;         // words of piece-start bits in a window of candidates
   int spw;               // sites of a wave
   const int4 *cols;      // dx, dy, dz lo, dz hi
   const float4 *colD;    // h (dx/nx, dy/ny, 0)
   const int *ccz;        // z index of each cell-ordered site's cell
   // the half of the columns for the Newton-3 pass and its partial forces
   int nhcol, pstride;
   const int4 *hcols;
   const float4 *hcolD;
   void *rsp;
   float cvx, cvy, cvz;   // h (0, 0, 1/nz)
   const double *potpar;
   double *force;
   double *part;
   int *tooclose;
};

template <class R> struct Pos;
template <> struct Pos<double> {
   static __device__ __forceinline__ void load(const RSArgs &a, int j, double &x, double &y,
                                               double &z, double &q) {
      double4 v = a.cpos[j];
      x = v.x; y = v.y; z = v.z; q = v.w;
   }
};
template <> struct Pos<float> {
   static __device__ __forceinline__ void load(const RSArgs &a, int j, float &x, float &y,
                                               float &z, float &q) {
      float4 v = a.cposf[j];
      x = v.x; y = v.y; z = v.z; q = v.w;
   }
};

// One thread per (site i, part q of the full shell): part q takes offsets
// o = q, q + nq, ... (own cell in part 0) and walks the sites of each
// neighbour cell.  The nq threads of a site are adjacent lanes (and, past
// 64, adjacent waves of one block) and combine their forces with shuffles
// and LDS; energy and virial go to one partial per wavefront.

// The bodies take their arguments as A: by value from the direct kernels
// (the code they compiled to before the bodies were split out), by
// reference into the table from a grouped launch (by value there they would
// be copied to scratch memory).
template <class R, int PT, bool COUL, class A = const RSArgs &>
__device__ __forceinline__ void b_realspace(int bx, int nbx, A a) {
   __shared__ R spot[MGPU_MAX_ID * MGPU_MAX_ID * MGPU_NPOTP];
   __shared__ double sreloc[81];
   const int npp = a.max_id * a.max_id * MGPU_NPOTP;
   for (int t = threadIdx.x; t < npp; t += blockDim.x) spot[t] = (R)a.potpar[t];
   for (int t = threadIdx.x; t < 81; t += blockDim.x) sreloc[t] = a.reloc[t];
   __syncthreads();

   const int lane = threadIdx.x & 63;
   const int t = bx * blockDim.x + threadIdx.x;
   const int nq = 1 << a.lognq;
   const int p = t >> a.lognq, qtr = t & (nq - 1);
   const bool have = p < a.nsites;
   const int pi = have ? p : 0;
   const int cell = a.ccell[pi];
   const int ix = cell / (a.ny * a.nz), iy = cell / a.nz - a.ny * ix, iz = cell - a.nz * (iy + a.ny * ix);
   R xi, yi, zi, qi;
   Pos<R>::load(a, pi, xi, yi, zi, qi);
   const int2 mi2 = a.cmeta[pi];
   const int ti = mi2.x & 0xff, fwi = mi2.x >> 8, mi = mi2.y;
   const R *prow = &spot[ti * a.max_id * MGPU_NPOTP];
   const R norm = (R)a.norm, alpha = (R)a.alpha;
   // per-cell partials in R, the running sums in FP64
   double gx = 0, gy = 0, gz = 0, v[7] = {0, 0, 0, 0, 0, 0, 0};
   // neighbour cell of offset o: index and periodic shift
   auto cell_of = [&](int o, int &jc, R &shx, R &shy, R &shz) {
      const int4 d = a.off[o];
      int ex = ix + d.x, ey = iy + d.y, ez = iz + d.z;
      int sx = ex < 0 ? -1 : (ex >= a.nx ? 1 : 0);
      int sy = ey < 0 ? -1 : (ey >= a.ny ? 1 : 0);
      int sz = ez < 0 ? -1 : (ez >= a.nz ? 1 : 0);
      jc = (ez - sz * a.nz) + a.nz * ((ey - sy * a.ny) + a.ny * (ex - sx * a.nx));
      if (sizeof(R) == 8) {
         const int code = 9 * (sx + 1) + 3 * (sy + 1) + (sz + 1);
         shx = (R)sreloc[3 * code]; shy = (R)sreloc[3 * code + 1]; shz = (R)sreloc[3 * code + 2];
      } else {
         const float4 D = a.offD[o];
         shx = D.x; shy = D.y; shz = D.z;
      }
   };
   // software pipeline over offsets: the next offset's cell and site range
   // are fetched while this one's sites are walked
   int jcn = 0, jn0 = 0, jn1 = 0;
   R snx = 0, sny = 0, snz = 0;
   if (have && qtr < a.nfull) {
      cell_of(qtr, jcn, snx, sny, snz);
      jn0 = a.css[jcn];
      jn1 = a.css[jcn + 1];
   }
   for (int o = qtr; have && o < a.nfull; o += nq) {
      R fx = 0, fy = 0, fz = 0, ep = 0, w00 = 0, w01 = 0, w02 = 0, w11 = 0, w12 = 0, w22 = 0;
      const int j0 = jn0, j1 = jn1;
      const R shx = snx, shy = sny, shz = snz;
      if (o + nq < a.nfull) {
         cell_of(o + nq, jcn, snx, sny, snz);
         jn0 = a.css[jcn];
         jn1 = a.css[jcn + 1];
      }
      for (int j = j0; j < j1; j++) {
         // the site's metadata and position are fetched together
         const int2 mj = a.cmeta[j];
         R xj, yj, zj, qj;
         Pos<R>::load(a, j, xj, yj, zj, qj);
         // one wait for both loads (else the position load sinks below the
         // checks and waits on its own)
         asm volatile("" ::"v"(xj), "v"(yj), "v"(zj), "v"(qj), "v"(mj.x));
         if (o == 0 && j == p) continue;
         const int tj = mj.x & 0xff, fwj = mj.x >> 8;
         if (fwi & fwj) continue;
         R rx = xj - xi + shx, ry = yj - yi + shy, rz = zj - zi + shz;
         R rsq = rx * rx + ry * ry + rz * rz;
         if (rsq < R(0.25) && mi != mj.y) {
            int io = a.corig[p], jo = a.corig[j];
            if (io < jo) {
               int slot = atomicAdd(a.tooclose, 1);
               if (slot < 16) {
                  a.tooclose[1 + 2 * slot] = io;
                  a.tooclose[2 + 2 * slot] = jo;
               }
            }
         }
         if (a.strict_sub && rsq > (R)a.cutsq) rsq = (R)a.cut100sq;
         R u, f;
         pair_term<R, PT, COUL>(rsq, qi * qj, norm, alpha, prow + tj * MGPU_NPOTP, u, f);
         // The minimum-image intramolecular pairs of rigid molecules sum to
         // eintra, which the FP64 path subtracts again; the FP32 path leaves
         // both out so their large cancelling energies never meet FP32
         // rounding.  Forces are kept.
         if (sizeof(R) == 4 && a.skip_intra_u && mi == mj.y && rsq < (R)a.half_box_sq) u = 0;
         fx -= f * rx;
         fy -= f * ry;
         fz -= f * rz;
         ep += u;
         w00 += f * rx * rx; w01 += f * rx * ry; w02 += f * rx * rz;
         w11 += f * ry * ry; w12 += f * ry * rz; w22 += f * rz * rz;
      }
      gx += (double)fx; gy += (double)fy; gz += (double)fz;
      v[0] += (double)ep;
      v[1] += (double)w00; v[2] += (double)w01; v[3] += (double)w02;
      v[4] += (double)w11; v[5] += (double)w12; v[6] += (double)w22;
   }
   // forces: the nq parts of a site sit in adjacent lanes, and for nq > 64
   // in adjacent waves of the block, summed in wave order through LDS
   const int nql = nq < 64 ? nq : 64;
   for (int m = 1; m < nql; m <<= 1) {
      gx += __shfl_xor(gx, m, 64);
      gy += __shfl_xor(gy, m, 64);
      gz += __shfl_xor(gz, m, 64);
   }
   if (nq > 64) {
      __shared__ double sred[4][3];
      const int wv = threadIdx.x >> 6;
      if (lane == 0) { sred[wv][0] = gx; sred[wv][1] = gy; sred[wv][2] = gz; }
      __syncthreads();
      if (qtr == 0) {
         for (int w = wv + 1; w < wv + nq / 64; w++) { gx += sred[w][0]; gy += sred[w][1]; gz += sred[w][2]; }
      }
   }
   if (have && qtr == 0) {
      const int io = a.corig[p];
      a.force[io] += gx;
      a.force[a.nsp + io] += gy;
      a.force[2 * a.nsp + io] += gz;
   }
#pragma unroll
   for (int q = 0; q < 7; q++) v[q] = wave_sum(v[q]);
   if (lane == 0) {
      double *pp = a.part + 8 * (size_t)(t >> 6);
      pp[0] = 0.5 * v[0];
      for (int q = 1; q < 7; q++) pp[q] = 0.5 * v[q];
      pp[7] = 0;
   }
}
template <class R, int PT, bool COUL>
__global__ __launch_bounds__(256) void k_realspace(RSArgs a) {
   b_realspace<R, PT, COUL, RSArgs>(blockIdx.x, gridDim.x, a);
}

// Load-balanced variant: a wave takes spw consecutive sites in turn.  The full
// shell is cut into z-columns of cells; a column's cells are consecutive in
// cell order, so its sites form one run of the cell-ordered arrays (two when
// it wraps through the periodic boundary in z).  The lanes build the site's
// runs ("pieces", at most two per column), wave prefix sums give each piece's
// first candidate, and the candidates are then dealt to the lanes 64 at a
// time, each lane finding its piece by the number of piece starts up to its
// candidate.  Every lane does a pair per step whatever the cell occupancies,
// where the per-offset walk above waits on the fullest cell of the wave at
// every offset.  The pair set and the pair term are the walk's; only the
// summation order differs.
//
// What bounds it: vector issue.  Beside the pairs (about 11 steps of 64 a
// site) the work of a site itself counts, so the columns' cells and shifts are
// kept while the sites stay in one column of cells (the sites are in cell
// order), a candidate's shift comes from its piece's record in LDS, the scans run on DPP, the piece starts of a window are held
// one word a lane, and energy and virial stay in the lanes over the wave's
// sites.  132,872 salt water sites: FP32 292 -> 239 us, FP64 563 -> 474
// (at the vector issue rate: about 90 vector instructions a step in FP32, 165 in FP64);
// 108,000 argon atoms 200 -> 128 us.
constexpr int RSB_SPW = 4;      // most sites of a wave
constexpr int RSB_NBW = 32;     // 64-bit words of piece-start bits per wave: a window of 2048 candidates

// Dynamic LDS of the balanced kernel, for maxp = 2 ncol pieces per site and
// npp potential parameters: reloc (FP64), per wave the piece-start bits, the
// pieces' shifts and their candidates' offsets, then the potential table.
template <class R> constexpr int RSB_ND = sizeof(R) == 4 ? 4 : 3;   // FP32: shift and z offset
template <class R> __host__ __device__ __forceinline__ size_t rsb_lds_bytes(int maxp, int npp) {
   return 82 * 8 + 4 * RSB_NBW * 8 + 4 * (size_t)maxp * RSB_ND<R> * sizeof(R) + 4 * (size_t)((maxp + 3) / 4 * 4) * 4 +
          (size_t)npp * sizeof(R);
}

// Inclusive scan over the wave on DPP: shifts within rows of 16, then each
// row's last lane to the next row and lane 31 to the upper half.
__device__ __forceinline__ int dpp_scan(int x) {
   x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);
   x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);
   x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);
   x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);
   x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, true);
   x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, true);
   return x;
}

// S64 (FP32 pairs): a lane adds every pair's force, energy and virial in FP64, as
// the walk adds each cell's, instead of keeping FP32 sums over the 11 or so pairs of a
// site that it meets.  Forces of 216 to 912 waters against FP64: 1.6 to 2.3% closer,
// as the walk's to 0.1%; the kernel alone 2,048 sites 12 us either way, 132,872 sites
// 222 and 232 us.
// MC: groups of 64 columns (2 holds the shell of a near-cubic cell at the
// reference's subcell, about 110 columns; 4 the most, 256).
template <class R, int PT, bool COUL, int MC, bool S64, class A = const RSArgs &>
__device__ __forceinline__ void b_realspace_bal(int bx, int nbx, A a) {
   constexpr bool F4 = sizeof(R) == 4;
   constexpr int ND = RSB_ND<R>;
   using S = typename std::conditional<S64, double, R>::type;
   extern __shared__ __attribute__((aligned(16))) unsigned char rsb_lds[];
   const int npp = a.max_id * a.max_id * MGPU_NPOTP, maxp = 2 * a.ncol;
   const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
   // carved in the order of rsb_lds_bytes
   unsigned char *lp = rsb_lds;
   double *sreloc = (double *)lp;
   lp += 82 * 8;
   unsigned long long *sbits = (unsigned long long *)lp + wave * RSB_NBW;   // piece-start bits
   lp += 4 * RSB_NBW * 8;
   R *sD = (R *)lp + wave * maxp * ND;             // a piece's shift (FP32: and z offset)
   lp += 4 * (size_t)maxp * ND * sizeof(R);
   int *sj = (int *)lp + wave * ((maxp + 3) / 4 * 4);   // site index less candidate index
   lp += 4 * (size_t)((maxp + 3) / 4 * 4) * 4;
   R *spot = (R *)lp;
   for (int t = threadIdx.x; t < npp; t += blockDim.x) spot[t] = (R)a.potpar[t];
   if (!F4)
      for (int t = threadIdx.x; t < 81; t += blockDim.x) sreloc[t] = a.reloc[t];
   __syncthreads();   // the only block barrier

   const int row = bx * 4 + wave, p0 = row * a.spw, p1 = min(p0 + a.spw, a.nsites);
   const R norm = (R)a.norm, alpha = (R)a.alpha;
   double v[7] = {0, 0, 0, 0, 0, 0, 0};
   // columns lane, lane + 64, ...: first cell and dz range at the present
   // (ix, iy), and the shift (FP32) or the periodic image code (FP64)
   int ccol = -1, cb[MC], zr[MC], code[MC];   // zr: dz range, low | high << 16
   float Dx[MC], Dy[MC], Dz[MC];
   for (int p = p0; p < p1; p++) {   // wave-uniform
      const int iz = a.ccz[p], col0 = a.ccell[p] - iz;
      if (col0 != ccol) {
         ccol = col0;
         const int ixy = col0 / a.nz, ix = ixy / a.ny, iy = ixy - a.ny * ix;
#pragma unroll
         for (int m = 0; m < MC; m++) {
            const int c = lane + 64 * m;
            if (c < a.ncol) {
               const int4 col = a.cols[c];
               const int ex = ix + col.x, ey = iy + col.y;
               const int sx = ex < 0 ? -1 : (ex >= a.nx ? 1 : 0), sy = ey < 0 ? -1 : (ey >= a.ny ? 1 : 0);
               cb[m] = a.nz * ((ey - sy * a.ny) + a.ny * (ex - sx * a.nx));
               zr[m] = (col.z & 0xffff) | (col.w << 16);
               if (F4) {
                  const float4 D = a.colD[c];
                  Dx[m] = D.x;
                  Dy[m] = D.y;
                  Dz[m] = D.z;
               } else {
                  code[m] = 9 * (sx + 1) + 3 * (sy + 1) + 1;
               }
            }
         }
      }
      R xi, yi, zi, qi;
      Pos<R>::load(a, p, xi, yi, zi, qi);
      const int2 mi2 = a.cmeta[p];
      const int ti = mi2.x & 0xff, fwi = mi2.x >> 8, mi = mi2.y;
      const R *prow = &spot[ti * a.max_id * MGPU_NPOTP];

      // pieces of this lane's columns: first site, count (second of a column: past the wrap)
      int pj[2 * MC], pn[2 * MC];
      int cnt = 0, tot = 0;
#pragma unroll
      for (int m = 0; m < MC; m++) {
         pn[2 * m] = pn[2 * m + 1] = 0;
         if (lane + 64 * m < a.ncol) {
            const int ez0 = iz + (short)zr[m], ez1 = iz + (zr[m] >> 16);
            const int s0 = ez0 < 0 ? -1 : (ez0 >= a.nz ? 1 : 0), s1 = ez1 < 0 ? -1 : (ez1 >= a.nz ? 1 : 0);
            const int za = ez0 - s0 * a.nz, zb = s1 == s0 ? ez1 - s0 * a.nz : a.nz - 1;
            pj[2 * m] = a.css[cb[m] + za];
            pn[2 * m] = a.css[cb[m] + zb + 1] - pj[2 * m];
            if (s1 != s0) {
               pj[2 * m + 1] = a.css[cb[m]];
               pn[2 * m + 1] = a.css[cb[m] + ez1 - s1 * a.nz + 1] - pj[2 * m + 1];
            }
            cnt += (pn[2 * m] > 0) + (pn[2 * m + 1] > 0);
            tot += pn[2 * m] + pn[2 * m + 1];
         }
      }
      // non-empty pieces, packed in lane order
      const int icnt = dpp_scan(cnt), itot = dpp_scan(tot);
      const int total = __builtin_amdgcn_readlane(itot, 63);
      int cself = -1;   // the site itself among its own column's candidates
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      {
         int k = icnt - cnt, st = itot - tot;
#pragma unroll
         for (int m = 0; m < MC; m++)
            {
#pragma unroll
               for (int w = 0; w < 2; w++) {
                  const int n = pn[2 * m + w], j = pj[2 * m + w];
                  if (n > 0) {
                     sj[k] = j - st;
                     const int ez = iz + (w ? zr[m] >> 16 : (int)(short)zr[m]), s = ez < 0 ? -1 : (ez >= a.nz ? 1 : 0);
                     if (F4) {
                        // z offset: turns a site's cell z index into dz
                        ((float4 *)sD)[k] = make_float4(Dx[m], Dy[m], Dz[m], (float)(s * a.nz - iz));
                     } else {
                        const double *rl = sreloc + 3 * (code[m] + s);
                        sD[3 * k] = (R)rl[0];
                        sD[3 * k + 1] = (R)rl[1];
                        sD[3 * k + 2] = (R)rl[2];
                     }
                     if (lane + 64 * m == a.own_col && p >= j && p < j + n) cself = p - j + st;
                     k++;
                     st += n;
                  }
               }
            }
      }
      cself = __builtin_amdgcn_readlane(cself, a.own_col & 63);

      S fx = 0, fy = 0, fz = 0;
      R ep = 0, w00 = 0, w01 = 0, w02 = 0, w11 = 0, w12 = 0, w22 = 0;
      int nst = -1;   // piece starts before the batch, less one
      // windows of candidates: a bit per piece start, then the window's batches of 64
      for (int wbase = 0; wbase < total; wbase += 64 * a.bit_words) {   // uniform
         if (lane < RSB_NBW) sbits[lane] = 0;
         __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
         __builtin_amdgcn_wave_barrier();
         __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
         {
            int st = itot - tot - wbase;
#pragma unroll
            for (int q = 0; q < 2 * MC; q++) {
                  if (pn[q] > 0) {
                     if ((unsigned)st < 64u * a.bit_words) atomicOr(&sbits[st >> 6], 1ull << (st & 63));
                     st += pn[q];
                  }
               }
         }
         __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
         __builtin_amdgcn_wave_barrier();
         __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
         const unsigned long long wl = sbits[lane & (RSB_NBW - 1)];
         const int wlo = (int)(unsigned)wl, whi = (int)(unsigned)(wl >> 32);
         const int wend = min(total, wbase + 64 * a.bit_words);
         for (int base = wbase; base < wend; base += 64) {
            // piece of a candidate: the starts at or before it, less one.  Bits
            // 1 .. lane of the word are the bits below lane of the word halved.
            const int wi = (base - wbase) >> 6;
            const unsigned long long w =
                (unsigned)__builtin_amdgcn_readlane(wlo, wi) |
                ((unsigned long long)(unsigned)__builtin_amdgcn_readlane(whi, wi) << 32);
            const unsigned long long h = w >> 1;
            const int k = __builtin_amdgcn_mbcnt_hi(
                (unsigned)(h >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)h, nst + (int)(w & 1)));
            nst += __popcll(w);
            const int c = base + lane;
            const bool act = c < total;
            const int j = act ? c + sj[k] : p;
            const int2 mj = a.cmeta[j];
            R xj, yj, zj, qj;
            Pos<R>::load(a, j, xj, yj, zj, qj);
            R rx, ry, rz;
            if (F4) {
               const float4 D = ((const float4 *)sD)[k];
               const float dz = (float)a.ccz[j] + D.w;
               rx = xj - xi + (R)(D.x + dz * a.cvx);
               ry = yj - yi + (R)(D.y + dz * a.cvy);
               rz = zj - zi + (R)(D.z + dz * a.cvz);
            } else {
               rx = xj - xi + sD[3 * k];
               ry = yj - yi + sD[3 * k + 1];
               rz = zj - zi + sD[3 * k + 2];
            }
            const int tj = mj.x & 0xff, fwj = mj.x >> 8;
            const bool skip = !act || c == cself || (fwi & fwj);
            R rsq = rx * rx + ry * ry + rz * rz;
            if (!skip && rsq < R(0.25) && mi != mj.y) {
               int io = a.corig[p], jo = a.corig[j];
               if (io < jo) {
                  int slot = atomicAdd(a.tooclose, 1);
                  if (slot < 16) {
                     a.tooclose[1 + 2 * slot] = io;
                     a.tooclose[2 + 2 * slot] = jo;
                  }
               }
            }
            if (a.strict_sub && rsq > (R)a.cutsq) rsq = (R)a.cut100sq;
            if (skip) rsq = R(1);   // a finite stand-in; its terms are dropped below
            R u, f;
            pair_term<R, PT, COUL>(rsq, qi * qj, norm, alpha, prow + tj * MGPU_NPOTP, u, f);
            if (F4 && a.skip_intra_u && mi == mj.y && rsq < (R)a.half_box_sq) u = 0;
            if (skip) {
               u = 0;
               f = 0;
            }
            const R gx = f * rx, gy = f * ry, gz = f * rz;
            if constexpr (S64) {
               fx -= (double)gx; fy -= (double)gy; fz -= (double)gz;
               v[0] += (double)u;
               v[1] += (double)(gx * rx); v[2] += (double)(gx * ry); v[3] += (double)(gx * rz);
               v[4] += (double)(gy * ry); v[5] += (double)(gy * rz); v[6] += (double)(gz * rz);
            } else {
               // from f, so that the product is not rounded by itself
               fx -= f * rx; fy -= f * ry; fz -= f * rz;
               ep += u;
               w00 += gx * rx; w01 += gx * ry; w02 += gx * rz;
               w11 += gy * ry; w12 += gy * rz; w22 += gz * rz;
            }
         }
      }
      double gx = (double)fx, gy = (double)fy, gz = (double)fz;
      wave_sum3(gx, gy, gz, lane);
      if constexpr (!S64) {
         v[0] += (double)ep;
         v[1] += (double)w00; v[2] += (double)w01; v[3] += (double)w02;
         v[4] += (double)w11; v[5] += (double)w12; v[6] += (double)w22;
      }
      if (lane < 3) a.force[(size_t)lane * a.nsp + a.corig[p]] += lane == 0 ? gx : lane == 1 ? gy : gz;
   }
   double *pp = a.part + 8 * (size_t)row;
#pragma unroll
   for (int q = 0; q < 7; q++) v[q] = wave_sum(v[q]);
   if (lane == 0) {
      for (int q = 0; q < 7; q++) pp[q] = 0.5 * v[q];
      pp[7] = 0;
   }
}
// Waves a SIMD the registers are held to (the compiler would take 133 in FP64 and
// 87 in FP32 for two groups of columns, three and five waves).
template <class R, int MC> constexpr int RSB_WPE = MC == 2 ? (sizeof(R) == 8 ? 4 : 6) : (sizeof(R) == 8 ? 3 : 4);
template <class R, int PT, bool COUL, int MC, bool S64>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(RSB_WPE<R, MC>))) void k_realspace_bal(RSArgs a) {
   b_realspace_bal<R, PT, COUL, MC, S64, RSArgs>(blockIdx.x, gridDim.x, a);
}

// Tiled Newton-3 variant: every pair once.  The full shell is symmetric,
// so its half (the own column from dz = 0, in the own cell only the sites
// after i, and the columns with (dx, dy) after (0, 0)) holds each unordered
// pair and image once.  One block per z-column of cells (ix, iy) takes the
// column's sites as i, 64 at a time (lane l: site l of the pass).  The half
// columns are dealt to the four waves in turn.  For each, the wave copies
// its j-column into LDS, RSN_MAXJ sites at a time; every lane forms its run
// of j there (the cells iz + lo .. iz + hi, across the periodic wrap in z,
// as parts at the images -1, 0, +1), and the pairs of all the wave's runs are
// dealt to its lanes 64 at a time (each pair's run found from a bit per run
// start, as in the balanced kernel).  The force on j is added to the chunk's
// LDS slot for j (ds_add, one wave per slot); the force on i is summed over
// the run's lanes (a segmented scan) into the wave's FP64 slot for i.  A
// chunk's j slots then go to row hc (the half column) of a partial array in
// which every (half column, site) has exactly one writer (the tile whose
// column plus that offset is the site's column); the four waves' i slots,
// in wave order, go to row H.  k_rs_fold adds each site's H + 1 rows in
// order, so the result does not depend on timing.  Energy and virial take
// weight 1.
constexpr int RSN_MAXJ = 64;   // j-sites staged per wave at a time
constexpr int RSN_NBW = 64;    // run-start words per wave: up to 64 runs of RSN_MAXJ pairs

template <class R> struct Stage;
template <> struct Stage<float> {
   using V = float4;
   static __device__ __forceinline__ V load(const RSArgs &a, int j) { return a.cposf[j]; }
};
template <> struct Stage<double> {
   using V = double4;
   static __device__ __forceinline__ V load(const RSArgs &a, int j) { return a.cpos[j]; }
};

// Dynamic LDS of the Newton-3 kernel, in carving order: per wave the staged
// j positions, the pass's i positions, per wave the j metadata, the i
// metadata, per wave the j force slots (R), per wave the i force slots
// (FP64), per wave the run table and the run-start bits, reloc, then the
// potential table.
__host__ __device__ __forceinline__ size_t rsn_lds_bytes(int npp, int rsize) {
   return (4 * (size_t)RSN_MAXJ + 64) * 4 * rsize + (4 * (size_t)RSN_MAXJ + 64) * 8 +
          4 * 3 * (size_t)RSN_MAXJ * rsize + 4 * 3 * 64 * 8 + 4 * 64 * 8 + 4 * (size_t)RSN_NBW * 8 + 84 * 8 +
          (size_t)npp * rsize;
}

// Segmented inclusive sum over lanes seg0 .. lane (all lanes of a segment
// share seg0), on the DPP data paths instead of LDS permutes: shifts by 1, 2,
// 4, 8 within rows of 16, then each row's last lane to the next row (rows 1
// and 3) and lane 31 to rows 2 and 3.  Lanes without a source read 0.
template <int CTRL, int ROWS> __device__ __forceinline__ float dpp0(float x) {
   return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, ROWS, 0xf, true));
}
template <int CTRL, int ROWS> __device__ __forceinline__ double dpp0(double x) {
   const long long b = __builtin_bit_cast(long long, x);
   const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWS, 0xf, true);
   const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xf, true);
   return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned)lo);
}
template <class T> __device__ __forceinline__ void seg_scan3(T &x, T &y, T &z, int lane, int seg0) {
#define RSN_STEP(CTRL, ROWS, COND)                                                         \
   {                                                                                      \
      const T ux = dpp0<CTRL, ROWS>(x), uy = dpp0<CTRL, ROWS>(y), uz = dpp0<CTRL, ROWS>(z); \
      if (COND) {                                                                         \
         x += ux;                                                                         \
         y += uy;                                                                         \
         z += uz;                                                                         \
      }                                                                                   \
   }
   RSN_STEP(0x111, 0xf, lane - 1 >= seg0)
   RSN_STEP(0x112, 0xf, lane - 2 >= seg0)
   RSN_STEP(0x114, 0xf, lane - 4 >= seg0)
   RSN_STEP(0x118, 0xf, lane - 8 >= seg0)
   RSN_STEP(0x142, 0xa, seg0 < (lane & ~15))
   RSN_STEP(0x143, 0xc, seg0 < 32)
#undef RSN_STEP
}

template <class R, int PT, bool COUL, class A = const RSArgs &>
__device__ __forceinline__ void b_realspace_n3(int bx, int nbx, A a) {
   using V = typename Stage<R>::V;
   extern __shared__ __attribute__((aligned(32))) unsigned char rsn_lds[];
   const int npp = a.max_id * a.max_id * MGPU_NPOTP;
   const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
   unsigned char *lp = rsn_lds;
   V *jpos = (V *)lp + wave * RSN_MAXJ;
   lp += 4 * (size_t)RSN_MAXJ * sizeof(V);
   V *ipos = (V *)lp;
   lp += 64 * sizeof(V);
   int2 *jmeta = (int2 *)lp + wave * RSN_MAXJ;
   lp += 4 * (size_t)RSN_MAXJ * 8;
   int2 *imeta = (int2 *)lp;
   lp += 64 * 8;
   R *fj = (R *)lp + wave * 3 * RSN_MAXJ;
   lp += 4 * 3 * (size_t)RSN_MAXJ * sizeof(R);
   double *fiall = (double *)lp;
   double *fi = fiall + wave * 3 * 64;
   lp += 4 * 3 * 64 * 8;
   int2 *srun = (int2 *)lp + wave * 64;
   lp += 4 * 64 * 8;
   unsigned long long *sbits = (unsigned long long *)lp + wave * RSN_NBW;
   lp += 4 * (size_t)RSN_NBW * 8;
   double *sreloc = (double *)lp;
   lp += 84 * 8;
   R *spot = (R *)lp;
   double *pp = a.part + 8 * ((size_t)bx * 4 + wave);
   R *P = (R *)a.rsp;
   const size_t ps = (size_t)a.pstride;

   // blocks go to the XCDs in turn: give each XCD a contiguous range of
   // columns, whose j-columns overlap, so that they meet in its L2
   const int ncolxy = a.nx * a.ny, per = (ncolxy + 7) >> 3;
   const int t = (int)(bx & 7) * per + (int)(bx >> 3);
   if (t >= ncolxy) {   // block-uniform; no barrier has been passed
      if (lane < 8) pp[lane] = 0.0;
      return;
   }
   for (int k = threadIdx.x; k < npp; k += blockDim.x) spot[k] = (R)a.potpar[k];
   for (int k = threadIdx.x; k < 81; k += blockDim.x) sreloc[k] = a.reloc[k];

   const int ix = t / a.ny, iy = t - a.ny * ix;
   const int ifirst = a.css[a.nz * t], ni = a.css[a.nz * t + a.nz] - ifirst;
   const R norm = (R)a.norm, alpha = (R)a.alpha;
   double v[7] = {0, 0, 0, 0, 0, 0, 0};
   // at least one pass, so that every j chunk of every half column is
   // written (zeros for a column without sites)
   const int npass = ni > 64 ? (ni + 63) >> 6 : 1;
   for (int pass = 0; pass < npass; pass++) {   // block-uniform
      const int i0 = pass * 64;
      const bool iact = i0 + lane < ni;
      if (wave == 0) {
         const int p = ifirst + (iact ? i0 + lane : 0);
         ipos[lane] = Stage<R>::load(a, p);
         const int2 m = a.cmeta[p];
         imeta[lane] = make_int2((m.x & 0x1ff) | (a.ccz[p] << 12), m.y);
      }
      fi[lane] = 0.0;
      fi[64 + lane] = 0.0;
      fi[128 + lane] = 0.0;
      __syncthreads();
      const int izi = imeta[lane].x >> 12;
      for (int c = wave; c < a.nhcol; c += 4) {   // wave-uniform
         const int4 col = a.hcols[c];
         const int ex = ix + col.x, ey = iy + col.y;
         const int sx = ex < 0 ? -1 : (ex >= a.nx ? 1 : 0), sy = ey < 0 ? -1 : (ey >= a.ny ? 1 : 0);
         const int cbj = a.nz * ((ey - sy * a.ny) + a.ny * (ex - sx * a.nx));
         const int jfirst = a.css[cbj], nj = a.css[cbj + a.nz] - jfirst;
         if (nj == 0) continue;
         // the lane's run [vs, ve) in image-major order (image s at
         // (s + 1) nj); in the own column it starts after i itself
         int vs = 0, ve = 0;
         if (iact) {
            const int zh = izi + col.w + 1;
            const int sh = zh < 0 ? -1 : (zh >= a.nz ? 1 : 0);
            ve = (sh + 1) * nj + a.css[cbj + zh - sh * a.nz] - jfirst;
            if (c == 0) {
               vs = nj + i0 + lane + 1;
            } else {
               const int zl = izi + col.z;
               const int sl = zl < 0 ? -1 : (zl >= a.nz ? 1 : 0);
               vs = (sl + 1) * nj + a.css[cbj + zl - sl * a.nz] - jfirst;
            }
         }
         R shx[3], shy[3], shz[3];
         float4 D = make_float4(0.f, 0.f, 0.f, 0.f);
         if (sizeof(R) == 8) {
#pragma unroll
            for (int s = 0; s < 3; s++) {
               const int code = 9 * (sx + 1) + 3 * (sy + 1) + s;
               shx[s] = (R)sreloc[3 * code];
               shy[s] = (R)sreloc[3 * code + 1];
               shz[s] = (R)sreloc[3 * code + 2];
            }
         } else {
            D = a.hcolD[c];
         }
         for (int k0 = 0; k0 < nj; k0 += RSN_MAXJ) {   // wave-uniform
            const int nch = min(nj - k0, RSN_MAXJ);
            // the previous chunk's reads and adds are done before the slices
            // are refilled
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            if (lane < nch) {
               const int jg = jfirst + k0 + lane;
               jpos[lane] = Stage<R>::load(a, jg);
               const int2 m = a.cmeta[jg];
               jmeta[lane] = make_int2((m.x & 0x1ff) | (a.ccz[jg] << 12), m.y);
            }
            fj[lane] = R(0);
            fj[RSN_MAXJ + lane] = R(0);
            fj[2 * RSN_MAXJ + lane] = R(0);
            sbits[lane] = 0ull;
            // the run's parts in this chunk, image by image
            int lo[3], n[3];
#pragma unroll
            for (int s = 0; s < 3; s++) {
               const int b = s * nj + k0;
               lo[s] = max(vs, b);
               n[s] = max(0, min(ve, b + nch) - lo[s]);
               lo[s] = n[s] > 0 ? lo[s] - b : 0;   // LDS index of the part's first site (< RSN_MAXJ)
            }
            const int cnt = n[0] + n[1] + n[2];
            const int icnt = wave_incl_scan(cnt, lane), irun = wave_incl_scan(cnt > 0 ? 1 : 0, lane);
            const int total = __shfl(icnt, 63, 64);
            const int st = icnt - cnt;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            if (cnt > 0) {
               srun[irun - 1] = make_int2(lane | (lo[0] << 6) | (lo[1] << 12) | (lo[2] << 18),
                                          n[0] | ((n[0] + n[1]) << 7) | (st << 14));
               atomicOr(&sbits[st >> 6], 1ull << (st & 63));
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            R ep = 0, w00 = 0, w01 = 0, w02 = 0, w11 = 0, w12 = 0, w22 = 0;
            int nst = 0;
            for (int base = 0; base < total; base += 64) {
               const int g = base + lane;
               const bool valid = g < total;
               // run = run starts at or before g, less one (bits past the
               // total are clear)
               const unsigned long long wd = sbits[base >> 6];
               const int below = __builtin_amdgcn_mbcnt_hi((unsigned)(wd >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)wd, 0));
               const int k = nst + below + (int)((wd >> lane) & 1ull) - 1;
               nst += __popcll(wd);
               const int2 r = srun[k];
               const int il = r.x & 63, n0 = r.y & 127, n01 = (r.y >> 7) & 127, rst = r.y >> 14;
               const int off = g - rst;
               const int s = off < n0 ? 0 : (off < n01 ? 1 : 2);
               int l = s == 0 ? ((r.x >> 6) & 63) + off
                              : (s == 1 ? ((r.x >> 12) & 63) + off - n0 : ((r.x >> 18) & 63) + off - n01);
               if (!valid) l = 0;
               const V pi = ipos[il];
               const int2 mi = imeta[il];
               const V pj = jpos[l];
               const int2 mj = jmeta[l];
               const int ti = mi.x & 0xff, fwi = (mi.x >> 8) & 1, tj = mj.x & 0xff, fwj = (mj.x >> 8) & 1;
               R rx, ry, rz;
               if (sizeof(R) == 4) {
                  const int dz = (mj.x >> 12) + (s - 1) * a.nz - (mi.x >> 12);
                  rx = (R)pj.x - (R)pi.x + (R)(D.x + (float)dz * a.cvx);
                  ry = (R)pj.y - (R)pi.y + (R)(D.y + (float)dz * a.cvy);
                  rz = (R)pj.z - (R)pi.z + (R)(D.z + (float)dz * a.cvz);
               } else {
                  rx = (R)pj.x - (R)pi.x + shx[s];
                  ry = (R)pj.y - (R)pi.y + shy[s];
                  rz = (R)pj.z - (R)pi.z + shz[s];
               }
               const bool skip = !valid || (fwi & fwj);
               R rsq = rx * rx + ry * ry + rz * rz;
               if (!skip && rsq < R(0.25) && mi.y != mj.y) {
                  const int io = a.corig[ifirst + i0 + il], jo = a.corig[jfirst + k0 + l];
                  const int slot = atomicAdd(a.tooclose, 1);
                  if (slot < 16) {
                     a.tooclose[1 + 2 * slot] = min(io, jo);
                     a.tooclose[2 + 2 * slot] = max(io, jo);
                  }
               }
               if (a.strict_sub && rsq > (R)a.cutsq) rsq = (R)a.cut100sq;
               if (skip) rsq = R(1);   // a finite stand-in; its terms are dropped below
               R u, f;
               pair_term<R, PT, COUL>(rsq, (R)pi.w * (R)pj.w, norm, alpha,
                                      &spot[(ti * a.max_id + tj) * MGPU_NPOTP], u, f);
               if (sizeof(R) == 4 && a.skip_intra_u && mi.y == mj.y && rsq < (R)a.half_box_sq) u = 0;
               if (skip) {
                  u = 0;
                  f = 0;
               }
               // the force on j; minus it on i
               const R gx = f * rx, gy = f * ry, gz = f * rz;
               ep += u;
               w00 += gx * rx; w01 += gx * ry; w02 += gx * rz;
               w11 += gy * ry; w12 += gy * rz; w22 += gz * rz;
               if (valid) {
                  atomicAdd(&fj[l], gx);
                  atomicAdd(&fj[RSN_MAXJ + l], gy);
                  atomicAdd(&fj[2 * RSN_MAXJ + l], gz);
               }
               // segmented sum over the run's lanes (lanes past the total
               // belong to the last run and add zeros); a run ends where the
               // next position starts a run, at the total or at lane 63
               const int seg0 = max(rst - base, 0);
               R hx = gx, hy = gy, hz = gz;
               seg_scan3(hx, hy, hz, lane, seg0);
               const bool last = lane == 63 || ((wd >> (lane + 1)) & 1ull) || g + 1 == total;
               if (last) {
                  fi[il] -= (double)hx;
                  fi[64 + il] -= (double)hy;
                  fi[128 + il] -= (double)hz;
               }
            }
            v[0] += (double)ep;
            v[1] += (double)w00; v[2] += (double)w01; v[3] += (double)w02;
            v[4] += (double)w11; v[5] += (double)w12; v[6] += (double)w22;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            // the chunk's j slots to row c (one writer; a later pass of the
            // same block adds)
            if (lane < nch) {
               const size_t o = (size_t)c * 3 * ps + jfirst + k0 + lane;
               if (pass == 0) {
                  P[o] = fj[lane];
                  P[o + ps] = fj[RSN_MAXJ + lane];
                  P[o + 2 * ps] = fj[2 * RSN_MAXJ + lane];
               } else {
                  P[o] += fj[lane];
                  P[o + ps] += fj[RSN_MAXJ + lane];
                  P[o + 2 * ps] += fj[2 * RSN_MAXJ + lane];
               }
            }
         }
      }
      __syncthreads();
      // the i sums of the four waves, in wave order, to row H
      if (wave == 0 && iact) {
         double hx = 0, hy = 0, hz = 0;
#pragma unroll
         for (int w = 0; w < 4; w++) {
            hx += fiall[w * 192 + lane];
            hy += fiall[w * 192 + 64 + lane];
            hz += fiall[w * 192 + 128 + lane];
         }
         const size_t o = (size_t)a.nhcol * 3 * ps + ifirst + i0 + lane;
         P[o] = (R)hx;
         P[o + ps] = (R)hy;
         P[o + 2 * ps] = (R)hz;
      }
      __syncthreads();   // before the next pass refills the i slots
   }
#pragma unroll
   for (int q = 0; q < 7; q++) v[q] = wave_sum(v[q]);
   if (lane == 0) {
      for (int q = 0; q < 7; q++) pp[q] = v[q];
      pp[7] = 0;
   }
}
template <class R, int PT, bool COUL>
__global__ __launch_bounds__(256) void k_realspace_n3(RSArgs a) {
   b_realspace_n3<R, PT, COUL, RSArgs>(blockIdx.x, gridDim.x, a);
}

// Site forces of the Newton-3 pass: each cell-ordered site adds its rows
// 0 .. H of the partial array in order.
template <class R>
__device__ __forceinline__ void b_rs_fold(int bx, int nbx, const R *__restrict__ P, int nrows, int nsites, int nsp,
                                          const int *__restrict__ corig, double *__restrict__ force) {
   const int s = bx * blockDim.x + threadIdx.x;
   if (s >= nsites) return;
   const size_t ps = (size_t)nsites;
   double fx = 0, fy = 0, fz = 0;
   for (int h = 0; h < nrows; h++) {
      const R *row = P + (size_t)h * 3 * ps + s;
      fx += (double)row[0];
      fy += (double)row[ps];
      fz += (double)row[2 * ps];
   }
   const int io = corig[s];
   force[io] += fx;
   force[nsp + io] += fy;
   force[2 * nsp + io] += fz;
}
template <class R>
__global__ __launch_bounds__(256) void k_rs_fold(const R *__restrict__ P, int nrows, int nsites, int nsp,
                                                 const int *__restrict__ corig, double *__restrict__ force) {
   b_rs_fold<R>(blockIdx.x, gridDim.x, P, nrows, nsites, nsp, corig, force);
}

template <class R, int PT, bool COUL, int MC>
void launch_bal(std::vector<LaunchRec> *rec, bool s64, unsigned g, unsigned b, hipStream_t s, size_t shm,
                const RSArgs &a) {
   auto run = [&](auto S) {
      constexpr bool S64 = decltype(S)::value;
      glaunch<k_realspace_bal<R, PT, COUL, MC, S64>, b_realspace_bal<R, PT, COUL, MC, S64>, 256, RSB_WPE<R, MC>>(
          rec, s, g, b, shm, a);
   };
   if constexpr (sizeof(R) == 4) {
      if (s64) return run(std::true_type{});
   }
   run(std::false_type{});
}

template <class R, bool COUL>
void launch_pt(std::vector<LaunchRec> *rec, int pt, int kind, bool s64, unsigned g, unsigned b, hipStream_t s,
               const RSArgs &a) {
   const int npp = a.max_id * a.max_id * MGPU_NPOTP;
   const size_t shm = kind == 1   ? rsb_lds_bytes<R>(2 * a.ncol, npp)
                      : kind == 2 ? rsn_lds_bytes(npp, sizeof(R))
                                  : 0;
#define RS_CASE(n)                                                                                     \
   case n:                                                                                             \
      if (kind == 1) {                                                                                 \
         if (a.ncol <= 128)                                                                            \
            launch_bal<R, n, COUL, 2>(rec, s64, g, b, s, shm, a);                                      \
         else                                                                                          \
            launch_bal<R, n, COUL, 4>(rec, s64, g, b, s, shm, a);                                      \
      } else if (kind == 2)                                                                            \
         glaunch<k_realspace_n3<R, n, COUL>, b_realspace_n3<R, n, COUL>, 256>(rec, s, g, b, shm, a);   \
      else                                                                                             \
         glaunch<k_realspace<R, n, COUL>, b_realspace<R, n, COUL>, 256>(rec, s, g, b, 0, a);           \
      break;
   switch (pt) {
      RS_CASE(0) RS_CASE(1) RS_CASE(2) RS_CASE(3) RS_CASE(4) RS_CASE(6)
   default: throw StatusError{MGPU_E_PTYPE, "unknown potential type"};
   }
#undef RS_CASE
}

}  // namespace

void mgpu::run_realspace(mgpu_engine *e) {
   int nc = e->ncells;
   // waves over the sites (load-balanced over the shell's z-columns) from one
   // site a CU: a step of 24 replicas of 256 to 2,048 waters took 0.24 + 0.16 ms here
   // with the walk below 4,096 sites, and single runs of 864 to 2,800 sites are 5 to 10
   // us a step shorter (132 to 123 FP64 at 864).  Below, or when the shell does not
   // split into columns, shell parts per site: at least 4, more (up to 256, four
   // waves of one 256-thread block) until the grid holds about 16 waves per CU
   // the tiled Newton-3 kernel (one block per z-column of cells) on request
   const bool tile = e->rs_nhcol > 0 && e->rs_mode == MGPU_RS_TILED;
   const bool bal = !tile && e->rs_ncol > 0 &&
                    (e->rs_mode == MGPU_RS_BALANCED || e->rs_mode == MGPU_RS_BALANCED_SEARCH ||
                     (e->rs_mode == MGPU_RS_AUTO && e->nsites >= e->ncu));
   e->rs_last_bal = bal || tile;
   int lognq = 2;
   while (lognq < 8 && (long)e->nsites << lognq < 16L * 64 * e->ncu) lognq++;
   // sites of a wave: more share the columns and the partial row (132,872 salt
   // water sites, FP32: 291, 252, 239, 246 us at 1, 2, 4, 8; 24,000 silica, FP64: 84 and
   // 76 at 1 and 2), as long as about 16 waves a CU remain
   int spw = 1;
   while (spw < RSB_SPW && (long)e->nsites >= 32L * spw * e->ncu) spw *= 2;
   const long nthreads = tile ? 256L * 8 * ((e->nx * e->ny + 7) / 8) : bal ? 64L * ((e->nsites + spw - 1) / spw) : (long)e->nsites << lognq;
   const int nblk = (int)((nthreads + 255) / 256), nwaves = nblk * 4;
   const int kind = tile ? 2 : bal ? 1 : 0;
   e->d_cell_part.reserve((size_t)nwaves * 8 + 8);
   RSArgs a;
   a.ncells = nc; a.nx = e->nx; a.ny = e->ny; a.nz = e->nz; a.nfull = e->n_full;
   a.lognq = lognq;
   a.max_id = e->max_id; a.nsp = e->nsp;
   a.strict_sub = e->strict && !e->molpbc;
   a.alpha = e->alpha;
   a.norm = 2.0 * e->alpha / sqrt(3.14159265358979323846);
   a.cutsq = e->cutoff * e->cutoff;
   a.cut100sq = 10000.0 * a.cutsq;
   a.skip_intra_u = e->precision == MGPU_MIXED && e->intra_exact;
   a.half_box_sq = e->half_box * e->half_box;
   int k = 0;
   for (int ii = -1; ii <= 1; ii++)
      for (int jj = -1; jj <= 1; jj++)
         for (int kk = -1; kk <= 1; kk++, k++) {
            // reloc_v, src/force.c:1284-1293
            a.reloc[3 * k] = e->h[0] * ii + e->h[1] * jj + e->h[2] * kk;
            a.reloc[3 * k + 1] = e->h[3] * ii + e->h[4] * jj + e->h[5] * kk;
            a.reloc[3 * k + 2] = e->h[6] * ii + e->h[7] * jj + e->h[8] * kk;
         }
   a.css = e->d_cell_site_start.p;
   a.off = e->d_off.p;
   a.offD = e->d_offD.p;
   a.cpos = e->d_cpos.p;
   a.cposf = e->d_cposf.p;
   a.cmeta = e->d_cmeta.p;
   a.corig = e->d_corig.p;
   a.ccell = e->d_ccell.p;
   a.nsites = e->nsites;
   a.ncol = e->rs_ncol; a.own_col = e->rs_own_col;
   a.bit_words = e->rs_mode == MGPU_RS_BALANCED_SEARCH ? 1 : RSB_NBW;
   a.spw = spw;
   a.cols = e->d_rscol.p; a.colD = e->d_rscolD.p; a.ccz = e->d_ccz.p;
   a.cvx = (float)(e->h[2] / e->nz); a.cvy = (float)(e->h[5] / e->nz); a.cvz = (float)(e->h[8] / e->nz);
   a.nhcol = e->rs_nhcol; a.pstride = e->nsites;
   a.hcols = e->d_rshcol.p; a.hcolD = e->d_rshcolD.p;
   const size_t rsize = e->precision == MGPU_FP64 ? 8 : 4;
   if (tile) e->d_rspart.reserve(((size_t)(e->rs_nhcol + 1) * 3 * e->nsites * rsize + 7) / 8 + 1);
   a.rsp = e->d_rspart.p;
   a.potpar = e->d_potpar.p;
   a.force = e->d_force_site.p;
   a.part = e->d_cell_part.p;
   a.tooclose = e->d_iflags.p + 1;
   const unsigned g = nblk, b = 256;
   bool coul = e->alpha > 0.0;
   // FP64 sums of the FP32 pairs below 16 sites a CU, where the walk, which has
   // them, was the choice by speed before the balanced kernel was, and on to 32,
   // where they cost nothing either (8,192 sites 22 us both ways; 24,000 water sites 45
   // and 47, 48,000 81 and 85): replicas of up to 2,048 waters then share one launch
   // (24 of them, 238 and 258 us a step: there they are enough to be issue bound)
   const bool s64 = (long)e->nsites <= 32L * e->ncu;
   {
      ProfScope ps(e, "realspace");
      if (e->precision == MGPU_FP64) {
         if (coul) launch_pt<double, true>(e->rec, e->ptype, kind, s64, g, b, e->stream, a);
         else launch_pt<double, false>(e->rec, e->ptype, kind, s64, g, b, e->stream, a);
      } else {
         if (coul) launch_pt<float, true>(e->rec, e->ptype, kind, s64, g, b, e->stream, a);
         else launch_pt<float, false>(e->rec, e->ptype, kind, s64, g, b, e->stream, a);
      }
      if (tile) {
         const int fb = (e->nsites + 255) / 256;
         if (e->precision == MGPU_FP64)
            glaunch<k_rs_fold<double>, b_rs_fold<double>, 256>(e->rec, e->stream, fb, 256, 0, (const double *)a.rsp,
                                                               a.nhcol + 1, e->nsites, e->nsp, e->d_corig.p,
                                                               e->d_force_site.p);
         else
            glaunch<k_rs_fold<float>, b_rs_fold<float>, 256>(e->rec, e->stream, fb, 256, 0, (const float *)a.rsp,
                                                             a.nhcol + 1, e->nsites, e->nsp, e->d_corig.p,
                                                             e->d_force_site.p);
      }
   }
   e->d_out.reserve(OUT_SIZE);
   if (e->defer_real && nwaves <= 2048) {
      // few rows: the glue adds them beside its own (16 loads a thread at the
      // most), where a column sum is a launch of 7.5 us (864 argon atoms)
      e->real_part = e->d_cell_part.p;
      e->real_rows = nwaves;
   } else {
      reduce_cols(e, e->d_cell_part.p, nwaves, 8, e->d_out.p + OUT_REAL);
   }
}
