// Parameter adjoint of eval_forces' potential energy and site forces (FP64):
// derivatives with respect to every pair type's potential parameters and
// every site id's charge.  This has no counterpart in the reference; it
// differentiates exactly what src/force.c:784-1005 (with kernel.c),
// src/ewald.c:280-589 and the constant terms of src/accel.c:293-329 and
// src/force.c:1158-1168 compute.
//
// Real space: a wave takes a few sites of one id in turn.  For each it
// lists the neighbour sites of the force kernel's full shell in LDS and deals
// them to its lanes 64 at a time; each lane forms u, dforceij and their
// derivatives with respect to the pair type's parameters and q_i q_j, and
// keeps its sums by the neighbour's site id in a lane-private column of LDS.
// Each unordered pair is seen from both ends with weight 1/2.  A wave's
// columns are added at its end, and a second kernel folds the waves' sums
// into the parameter vector, both in a fixed order.  For a site-force
// cotangent v the pair (i, j) contributes dforceij * (v_j - v_i).(r_j - r_i),
// since F_i = forceij (r_i - r_j) (mk_forces, src/force.c:717-743).
//
// Reciprocal space: see ewald_charge_adjoint (mgpu_ewald.hip).
// Constant terms (intramolecular correction, distant potential, self and
// sheet energies): differentiated on the host with the same Dual pair term.
#include "mgpu_internal.h"
#include "mgpu_pair.h"

#include <math.h>
#include <algorithm>

using namespace mgpu;

namespace {

constexpr double PI_D = 3.14159265358979323846;
constexpr int ADJ_QCAP = 320;     // neighbour queue: 63 left over and 64 lanes of ADJ_EMIT
constexpr int ADJ_EMIT = 4;       // sites a lane lists at once

struct AdjArgs {
   int nsites, nx, ny, nz, nfull, max_id, npar, nsp, strict_sub;
   int nslot;              // slots of a wave: half of them for dE, the others for the cotangent (none without v)
   double alpha, norm, cutsq, cut100sq;
   double reloc[81];
   const int *css;
   const int4 *off;
   const double4 *cpos;
   const int2 *cmeta;
   const int *corig;
   const int *ccell;
   const int *pos;         // site -> position in cell order
   const int4 *chunk;      // per wave: first and end of its sites in bysite, their id
   const int *bysite;      // sites ordered by id
   const double *potpar;   // [max_id][max_id][8]
   const double *v;        // cotangent [3][nsp] or null
   const double *dpar;     // direction [max_id][max_id][8] or null
   const double *dq;       // direction [max_id] or null
   const double *chg_id;   // [max_id]
   double *part;           // [waves][nslot]
   double *jvp;            // [3][nsp] accumulated, or null
};

// Parameters of each potential form (src/kernel.c:75-84).
__host__ __device__ constexpr int form_npar(int pt) {
   return pt == 0 ? 2 : pt == 1 ? 3 : pt == 2 ? 4 : pt == 3 ? 6 : pt == 4 ? 3 : 7;
}

// Derivatives of pair_term's u and forceij with respect to the form's
// parameters (du, df) and the charge product (uq, fq).  Both are linear in
// q_i q_j, so uq and fq do not depend on it.
template <int PT, bool COUL>
__device__ __forceinline__ void pair_grad(double rsq, double norm, double alpha, const double *__restrict__ p,
                                          double *du, double *df, double &uq, double &fq) {
   double r = 0, r_r = 0, r2r;
   uq = fq = 0;
   if (COUL || PT != 0) {
      r = sqrt(rsq);
      r_r = 1.0 / r;
      r2r = r_r * r_r;
   } else {
      r2r = 1.0 / rsq;
   }
   if (COUL) {
      const double ar = alpha * r, t = 1.0 / (1.0 + AS_P * ar), et = exp(-(ar * ar));
      uq = t * (AS_A1 + t * (AS_A2 + t * (AS_A3 + t * (AS_A4 + t * AS_A5)))) * et * r_r;
      fq = r2r * (uq + norm * et);
   }
   const double r4 = r2r * r2r, r6 = r2r * r4;
   if (PT == 0) {
      const double x = p[1] * p[1] * r2r, s6 = x * x * x, s12 = s6 * s6;
      const double d6 = 6.0 * p[1] * r2r * (x * x), d12 = 2.0 * s6 * d6;   // with respect to p[1]
      du[0] = s12 - s6;
      du[1] = p[0] * (d12 - d6);
      df[0] = 6.0 * r2r * (2.0 * s12 - s6);
      df[1] = 6.0 * r2r * p[0] * (2.0 * d12 - d6);
   } else if (PT == 1) {
      const double e = exp(-p[2] * r), pe = p[1] * e;
      du[0] = -r6;
      du[1] = e;
      du[2] = -r * pe;
      df[0] = -6.0 * r2r * r6;
      df[1] = p[2] * e * r_r;
      df[2] = pe * r_r * (1.0 - p[2] * r);
   } else if (PT == 2) {
      const double e1 = exp(-p[1] * r), e2 = exp(-p[3] * r);
      du[0] = e1;
      du[1] = -r * p[0] * e1;
      du[2] = -e2;
      du[3] = r * p[2] * e2;
      df[0] = p[1] * e1 * r_r;
      df[1] = p[0] * e1 * r_r * (1.0 - p[1] * r);
      df[2] = -p[3] * e2 * r_r;
      df[3] = -p[2] * e2 * r_r * (1.0 - p[3] * r);
   } else if (PT == 3) {
      const double e1 = exp(-p[1] * r), r8 = r4 * r4, r12 = r6 * r6;
      du[0] = e1;
      du[1] = -r * p[0] * e1;
      du[2] = r12;
      du[3] = -r4;
      du[4] = -r6;
      du[5] = -r8;
      df[0] = p[1] * e1 * r_r;
      df[1] = p[0] * e1 * r_r * (1.0 - p[1] * r);
      df[2] = 12.0 * r2r * r12;
      df[3] = -4.0 * r2r * r4;
      df[4] = -6.0 * r2r * r6;
      df[5] = -8.0 * r2r * r8;
   } else if (PT == 4) {
      const double r12 = r6 * r6;
      du[0] = r4;
      du[1] = r6;
      du[2] = r12;
      df[0] = 4.0 * r2r * r4;
      df[1] = 6.0 * r2r * r6;
      df[2] = 12.0 * r2r * r12;
   } else {
      const double a = p[1] - r, b = r - p[6];
      const double e1 = exp(a * p[2]), e2 = exp(-2.0 * p[5] * b), e3 = exp(-p[5] * b);
      du[0] = e1;
      du[1] = p[0] * p[2] * e1;
      du[2] = p[0] * a * e1;
      du[3] = -r6;
      du[4] = e2 - 2.0 * e3;
      du[5] = 2.0 * p[4] * b * (e3 - e2);
      du[6] = 2.0 * p[4] * p[5] * (e2 - e3);
      df[0] = r_r * p[2] * e1;
      df[1] = r_r * p[2] * p[2] * p[0] * e1;
      df[2] = r_r * p[0] * e1 * (1.0 + p[2] * a);
      df[3] = -6.0 * r2r * r6;
      df[4] = 2.0 * r_r * p[5] * (e2 - e3);
      df[5] = 2.0 * r_r * p[4] * ((e2 - e3) + p[5] * b * (e3 - 2.0 * e2));
      df[6] = 2.0 * r_r * p[5] * p[4] * p[5] * (2.0 * e2 - e3);
   }
}

// Slots of a wave (E half, then V half):
//   [b*(npar+1) + k]   sum over neighbours of id b of 1/2 du/dp_k (k < npar)
//   [b*(npar+1)+npar]  sum over neighbours of id b of 1/2 du/d(qq) q_i
//   [nid*(npar+1)]     sum over all neighbours of 1/2 du/d(qq) q_j
// LDS: the lanes' slots [slot][lane] (a lane's own column: no conflicts),
// the neighbour queue, and the parameter rows of the wave's id.
//
// Bound by the FP64 pair terms and their LDS sums.  24,000 silica sites take
// 0.22 ms and 2,916 water sites 0.05 ms; one thread a site, each walking its
// own shell with all eight derivatives whatever the form, took 2.3 ms and
// 4.1 ms (46 one-wave blocks at 2,916 sites).
template <int PT, bool COUL>
__global__ __launch_bounds__(64) void k_adj_real(AdjArgs a) {
   constexpr int NP = form_npar(PT);
   extern __shared__ double adj_lds[];
   const int lane = threadIdx.x;
   double *acc = adj_lds;
   double *prow = acc + (size_t)a.nslot * 64;
   int2 *q = (int2 *)(prow + (size_t)a.max_id * MGPU_NPOTP);
   const int4 ch = a.chunk[blockIdx.x];
   const int ti = ch.z, ns1 = a.npar + 1, self_slot = a.max_id * ns1, half = self_slot + 1;
   const int np = a.npar < NP ? a.npar : NP;
   for (int t = 0; t < a.nslot; t++) acc[t * 64 + lane] = 0.0;
   for (int t = lane; t < a.max_id * MGPU_NPOTP; t += 64) prow[t] = a.potpar[(size_t)ti * a.max_id * MGPU_NPOTP + t];
   __syncthreads();
   double se = 0, sv = 0;   // the wave's self slots
   for (int s = ch.x; s < ch.y; s++) {   // wave-uniform
      const int io = a.bysite[s], p = a.pos[io], cell = a.ccell[p];
      const int ix = cell / (a.ny * a.nz), iy = cell / a.nz - a.ny * ix, iz = cell - a.nz * (iy + a.ny * ix);
      const double4 Pi = a.cpos[p];
      const int fwi = a.cmeta[p].x >> 8;
      double vi[3] = {0, 0, 0};
      if (a.v) { vi[0] = a.v[io]; vi[1] = a.v[a.nsp + io]; vi[2] = a.v[2 * (size_t)a.nsp + io]; }
      double jx = 0, jy = 0, jz = 0;
      // one queued neighbour (position j, image code | own-cell bit << 5)
      auto pair = [&](int2 e) {
         const int j = e.x, code = e.y & 31;
         const int2 mj = a.cmeta[j];
         const int tj = mj.x & 0xff, fwj = mj.x >> 8;
         if (((e.y >> 5) && j == p) || (fwi & fwj)) return;
         const double4 Pj = a.cpos[j];
         const double rx = Pj.x - Pi.x + a.reloc[3 * code], ry = Pj.y - Pi.y + a.reloc[3 * code + 1],
                      rz = Pj.z - Pi.z + a.reloc[3 * code + 2];
         double rsq = rx * rx + ry * ry + rz * rz;
         if (a.strict_sub && rsq > a.cutsq) rsq = a.cut100sq;
         double du[NP], df[NP], uq, fq;
         pair_grad<PT, COUL>(rsq, a.norm, a.alpha, prow + tj * MGPU_NPOTP, du, df, uq, fq);
         double *eb = acc + (size_t)(tj * ns1) * 64 + lane;
#pragma unroll
         for (int k = 0; k < NP; k++)
            if (k < np) eb[64 * k] += 0.5 * du[k];
         eb[64 * a.npar] += 0.5 * uq * Pi.w;
         se += 0.5 * uq * Pj.w;
         if (a.v) {
            const int jo = a.corig[j];
            const double w = 0.5 * ((a.v[jo] - vi[0]) * rx + (a.v[a.nsp + jo] - vi[1]) * ry +
                                    (a.v[2 * (size_t)a.nsp + jo] - vi[2]) * rz);
            double *vb = eb + (size_t)half * 64;
#pragma unroll
            for (int k = 0; k < NP; k++)
               if (k < np) vb[64 * k] += df[k] * w;
            vb[64 * a.npar] += fq * Pi.w * w;
            sv += fq * Pj.w * w;
         }
         if (a.jvp) {
            const double *dp = a.dpar + (size_t)(ti * a.max_id + tj) * MGPU_NPOTP;
            double g = fq * (a.dq[ti] * a.chg_id[tj] + a.dq[tj] * a.chg_id[ti]);
#pragma unroll
            for (int k = 0; k < NP; k++)
               if (k < np) g += dp[k] * df[k];
            jx -= g * rx;
            jy -= g * ry;
            jz -= g * rz;
         }
      };
      int qn = 0;   // queued neighbours, wave-uniform
      for (int o0 = 0; o0 < a.nfull; o0 += 64) {
         const int o = o0 + lane;
         int j = 0, j1 = 0, code = 0;
         if (o < a.nfull) {
            const int4 d = a.off[o];
            const int ex = ix + d.x, ey = iy + d.y, ez = iz + d.z;
            const int sx = ex < 0 ? -1 : (ex >= a.nx ? 1 : 0), sy = ey < 0 ? -1 : (ey >= a.ny ? 1 : 0),
                      sz = ez < 0 ? -1 : (ez >= a.nz ? 1 : 0);
            const int jc = (ez - sz * a.nz) + a.nz * ((ey - sy * a.ny) + a.ny * (ex - sx * a.nx));
            j = a.css[jc];
            j1 = a.css[jc + 1];
            code = (9 * (sx + 1) + 3 * (sy + 1) + (sz + 1)) | (o == 0) << 5;
         }
         // every lane lists up to ADJ_EMIT of its cell's sites; full batches
         // are evaluated at once, the rest moves to the front of the queue
         while (__any(j < j1)) {
            const int m = min(j1 - j, ADJ_EMIT);
            const int incl = wave_incl_scan(m, lane);
            for (int t = 0; t < m; t++) q[qn + incl - m + t] = make_int2(j + t, code);
            j += m;
            qn += __shfl(incl, 63, 64);
            __syncthreads();
            int b = 0;
            for (; qn - b >= 64; b += 64) pair(q[b + lane]);
            qn -= b;
            const int2 rest = q[b + (lane < qn ? lane : 0)];
            __syncthreads();
            if (lane < qn) q[lane] = rest;
            __syncthreads();
         }
      }
      if (lane < qn) pair(q[lane]);
      __syncthreads();
      if (a.jvp) {
         jx = wave_sum(jx);
         jy = wave_sum(jy);
         jz = wave_sum(jz);
         if (lane == 0) {
            a.jvp[io] += jx;
            a.jvp[a.nsp + io] += jy;
            a.jvp[2 * (size_t)a.nsp + io] += jz;
         }
      }
   }
   acc[(size_t)self_slot * 64 + lane] = se;
   if (a.v) acc[(size_t)(half + self_slot) * 64 + lane] = sv;
   __syncthreads();
   // lane s adds slot s over the lanes, each from its own start (no conflicts)
   for (int s = lane; s < a.nslot; s += 64) {
      double t = 0;
      for (int k = 0; k < 64; k++) t += acc[s * 64 + ((k + lane) & 63)];
      a.part[(size_t)blockIdx.x * a.nslot + s] = t;
   }
}

// Site -> position in cell order.
__global__ void k_adj_pos(int ns, const int *__restrict__ corig, int *__restrict__ pos) {
   const int p = blockIdx.x * blockDim.x + threadIdx.x;
   if (p < ns) pos[corig[p]] = p;
}

// The waves' slots folded into theta: one block per theta entry and half
// (blockIdx.y: 0 dE, 1 the cotangent part), the waves in a fixed order.  One
// thread per entry walking all 24,000 sites took 22 ms; this takes 18 us.
__global__ __launch_bounds__(256) void k_adj_fold(int nw, int max_id, int npar, int nslot, int half,
                                                  const int4 *__restrict__ chunk, const double *__restrict__ part,
                                                  double *__restrict__ out) {
   __shared__ double ws[4];
   const int ntypes = max_id * (max_id + 1) / 2, ns1 = npar + 1;
   const int col = blockIdx.x;
   double s = 0.0;
   if (col < ntypes * npar) {
      int t = col / npar, k = col - t * npar, a = 0;
      while (t >= max_id - a) { t -= max_id - a; a++; }
      const int b = a + t;
      for (int c = threadIdx.x; c < nw; c += 256) {
         const int ti = chunk[c].z;
         const double *r = part + (size_t)c * nslot + blockIdx.y * half;
         if (ti == a) s += r[b * ns1 + k];
         if (a != b && ti == b) s += r[a * ns1 + k];
      }
   } else {
      const int a = col - ntypes * npar;
      for (int c = threadIdx.x; c < nw; c += 256) {
         const double *r = part + (size_t)c * nslot + blockIdx.y * half;
         if (chunk[c].z == a) s += r[max_id * ns1];
         s += r[a * ns1 + npar];
      }
   }
   s = wave_sum(s);
   if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = s;
   __syncthreads();
   if (threadIdx.x == 0) out[(size_t)blockIdx.y * gridDim.x + col] = ws[0] + ws[1] + ws[2] + ws[3];
}

template <int PT, bool COUL> void launch_adj(unsigned g, size_t shm, hipStream_t s, const AdjArgs &a) {
   allow_lds((const void *)k_adj_real<PT, COUL>, shm);
   k_adj_real<PT, COUL><<<g, 64, shm, s>>>(a);
}

template <bool COUL> void launch_adj_pt(int pt, unsigned g, size_t shm, hipStream_t s, const AdjArgs &a) {
   switch (pt) {
   case 0: launch_adj<0, COUL>(g, shm, s, a); break;
   case 1: launch_adj<1, COUL>(g, shm, s, a); break;
   case 2: launch_adj<2, COUL>(g, shm, s, a); break;
   case 3: launch_adj<3, COUL>(g, shm, s, a); break;
   case 4: launch_adj<4, COUL>(g, shm, s, a); break;
   case 6: launch_adj<6, COUL>(g, shm, s, a); break;
   default: throw StatusError{MGPU_E_PTYPE, "unknown potential type"};
   }
}

// ---------------------------------------------------------------- host
using D1 = Dual<1>;

template <int PT> D1 pair_u_pt(double rsq, D1 qq, double alpha, const D1 *p) {
   D1 u, f;
   if (alpha > 0.0)
      pair_term<D1, PT, true>(D1(rsq), qq, D1(2.0 * alpha / sqrt(PI_D)), D1(alpha), p, u, f);
   else
      pair_term<D1, PT, false>(D1(rsq), qq, D1(0.0), D1(alpha), p, u, f);
   return u;
}

D1 pair_u(int pt, double rsq, D1 qq, double alpha, const D1 *p) {
   switch (pt) {
   case 0: return pair_u_pt<0>(rsq, qq, alpha, p);
   case 1: return pair_u_pt<1>(rsq, qq, alpha, p);
   case 2: return pair_u_pt<2>(rsq, qq, alpha, p);
   case 3: return pair_u_pt<3>(rsq, qq, alpha, p);
   case 4: return pair_u_pt<4>(rsq, qq, alpha, p);
   case 6: return pair_u_pt<6>(rsq, qq, alpha, p);
   default: throw StatusError{MGPU_E_PTYPE, "unknown potential type"};
   }
}

D1 texp(D1 x) { return Math<D1>::exp_(x); }

// dist_pot, src/kernel.c:103-151, in Dual arithmetic
D1 dist_pot_d(const D1 *p, double rc, int pt) {
   auto sq = [](D1 x) { return x * x; };
   auto cu = [](D1 x) { return x * x * x; };
   const double rc3 = rc * rc * rc;
   switch (pt) {
   case 0: return p[0] * cu(sq(p[1]) * (1.0 / rc)) * (1.0 / 3.0);
   case 1:
      if (p[2].v > 1e-7)
         return p[0] * (1.0 / (3.0 * rc3)) -
                p[1] * texp(-p[2] * rc) *
                    (rc * rc * Math<D1>::rcp(p[2]) + 2 * rc * Math<D1>::rcp(sq(p[2])) + 2.0 * Math<D1>::rcp(cu(p[2])));
      return p[0] * (1.0 / (3.0 * rc3));
   case 2:
      if (p[3].v > 1e-7)
         return p[2] * (rc * rc * Math<D1>::rcp(p[3]) + 2 * rc * Math<D1>::rcp(sq(p[3])) + 2.0 * Math<D1>::rcp(cu(p[3]))) *
                texp(-p[3] * rc);
      return D1(0.0);
   case 3: {
      D1 tail = -p[2] * (1.0 / (9.0 * rc3 * rc3 * rc3)) + p[3] * (1.0 / rc) + p[4] * (1.0 / (3.0 * rc3)) +
                p[5] * (1.0 / (5.0 * rc * rc * rc3));
      if (p[1].v > 1e-7)
         return -p[0] * texp(-p[1] * rc) *
                    (rc * rc * Math<D1>::rcp(p[1]) + 2 * rc * Math<D1>::rcp(sq(p[1])) + 2.0 * Math<D1>::rcp(cu(p[1]))) +
                tail;
      return tail;
   }
   case 6:
      if (p[5].v != 0.0)
         return p[3] * (1.0 / (3.0 * rc3)) +
                2.0 * p[4] *
                    (rc * rc * Math<D1>::rcp(p[5]) + 2 * rc * Math<D1>::rcp(sq(p[5])) + 2.0 * Math<D1>::rcp(cu(p[5]))) *
                    texp(-p[5] * (rc - p[6]));
      return p[3] * (1.0 / (3.0 * rc3));
   case 4: return -p[0] * (1.0 / rc) - p[1] * (1.0 / (3.0 * rc3)) - p[2] * (1.0 / (9.0 * rc3 * rc3 * rc3));
   default: return D1(0.0);
   }
}

double err_fn_host(double x) {   // src/auxil.c:586-593
   double t = 1.0 / (1.0 + AS_P * x);
   if (x >= 0.0) return 1.0 - t * (AS_A1 + t * (AS_A2 + t * (AS_A3 + t * (AS_A4 + t * AS_A5)))) * exp(-x * x);
   return -err_fn_host(-x);
}

// Derivatives of the constant terms of pe[0] + pe[1]: -eintra + dist/V
// (potential parameters and charges) and -self + sheet/V (charges).
void static_grad(mgpu_engine *e, int npar, double *g) {
   const int nid = e->max_id, ntypes = nid * (nid + 1) / 2;
   const double vol = host_det(e->h);
   auto tcol = [&](int a, int b) {
      int lo = std::min(a, b), hi = std::max(a, b), t = 0;
      for (int x = 0; x < lo; x++) t += nid - x;
      return t + (hi - lo);
   };
   std::vector<double> q(e->site_charge);
   // one theta entry at a time: seed it, evaluate the terms in Dual<1>
   const int ntheta = ntypes * npar + nid;
   for (int th = 0; th < ntheta; th++) {
      const bool is_q = th >= ntypes * npar;
      const int qa = is_q ? th - ntypes * npar : -1;
      int ta = -1, tb = -1, tk = -1;
      if (!is_q) {
         int t = th / npar;
         tk = th - t * npar;
         int a = 0;
         while (t >= nid - a) { t -= nid - a; a++; }
         ta = a;
         tb = a + t;
      }
      auto par = [&](int a, int b, D1 *out) {
         const double *pp = e->potpar.data() + MGPU_NPOTP * (a * nid + b);
         bool hit = !is_q && tcol(a, b) == tcol(ta, tb);
         for (int k = 0; k < MGPU_NPOTP; k++) out[k] = D1::seed(pp[k], hit && k == tk ? 0 : -1);
      };
      auto chg = [&](int a) { return D1::seed(q[a], a == qa ? 0 : -1); };
      double total = 0.0;
      // -eintra, src/force.c:654-668 and 1158-1168
      for (int s = 0; s < e->nspecies; s++) {
         if (e->spec_fw[s]) continue;
         const int ns = e->spec_nsites[s];
         const int *id = e->spec_site_id.data() + e->spec_off[s];
         const double *pf = e->spec_pf.data() + 3 * e->spec_off[s];
         double ei = 0.0;
         for (int b = 0; b < ns; b++)
            for (int a = b + 1; a < ns; a++) {
               double d2 = 0;
               for (int c = 0; c < 3; c++) d2 += (pf[3 * a + c] - pf[3 * b + c]) * (pf[3 * a + c] - pf[3 * b + c]);
               double d = sqrt(d2);
               D1 p[MGPU_NPOTP];
               par(id[b], id[a], p);
               ei += pair_u(e->ptype, d * d, chg(id[a]) * chg(id[b]), e->alpha, p).d[0];
            }
         total -= e->spec_nmols[s] * ei;
      }
      // dist / V, src/accel.c:293-329 (potential parameters only)
      if (!is_q) {
         std::vector<long> count(nid, 0);
         for (int sp = 0; sp < e->nspecies; sp++)
            for (int is = 0; is < e->spec_nsites[sp]; is++)
               count[e->spec_site_id[e->spec_off[sp] + is]] += e->spec_nmols[sp];
         for (int a = 1; a < nid; a++)
            for (int b = 1; b < nid; b++) {
               D1 p[MGPU_NPOTP];
               par(a, b, p);
               total -= 2 * PI_D * count[a] * count[b] * dist_pot_d(p, e->cutoff, e->ptype).d[0] / vol;
            }
      }
      // -self + sheet / V, src/ewald.c:367-425 (charges only)
      if (is_q && e->alpha > 0) {
         double dself = 0.0, sq = 0.0;
         int ssite = 0, s = 0;
         std::vector<double> chs;
         for (int sp = 0; sp < e->nspecies; sp++)
            for (int m = 0; m < e->spec_nmols[sp]; m++)
               for (int is = 0; is < e->spec_nsites[sp]; is++) chs.push_back(q[e->spec_site_id[e->spec_off[sp] + is]]);
         for (; s < e->nspecies && !e->spec_fw[s]; s++) {
            const int ns = e->spec_nsites[s];
            const int *id = e->spec_site_id.data() + e->spec_off[s];
            const double *pf = e->spec_pf.data() + 3 * e->spec_off[s];
            double intra = 0.0;
            for (int a = 0; a < ns; a++)
               for (int b = a + 1; b < ns; b++) {
                  double d2 = 0;
                  for (int c = 0; c < 3; c++) d2 += (pf[3 * a + c] - pf[3 * b + c]) * (pf[3 * a + c] - pf[3 * b + c]);
                  double r = sqrt(d2);
                  double dqq = (id[a] == qa ? q[id[b]] : 0.0) + (id[b] == qa ? q[id[a]] : 0.0);
                  intra += dqq * err_fn_host(e->alpha * r) / r;
               }
            dself += e->spec_nmols[s] * intra;
            ssite += ns * e->spec_nmols[s];
         }
         long na = 0;
         for (int i = 0; i < ssite; i++) {
            sq += chs[i];
            if (e->site_type[i] == qa) na++;
         }
         dself += e->alpha / sqrt(PI_D) * 2.0 * q[qa] * na;
         total -= dself;
         double sqall = sq;
         long naall = na;
         for (int i = ssite; i < e->nsites; i++) {
            sqall += chs[i];
            if (e->site_type[i] == qa) naall++;
         }
         const double conv_q = 4.07497263794495e-14 * 1.e-3 * 1.05482230112e-05 / 1.60217733e-19;
         if (fabs(sqall) * conv_q > 1.0e-5)
            total -= PI_D * 2.0 * sqall * naall / (2.0 * e->alpha * e->alpha) / vol;
      }
      g[th] += total;
   }
}

}  // namespace

int mgpu::adjoint_ntheta(const mgpu_engine *e) {
   const int nid = e->max_id;
   return nid * (nid + 1) / 2 * e->npar + nid;
}

void mgpu::run_adjoint(mgpu_engine *e, const double *v_host, const double *dtheta, double *dE, double *vjp,
                       double *jvp_host) {
   if (e->surface_dipole && e->alpha > 1e-7)
      throw StatusError{MGPU_E_CAPACITY, "the parameter adjoint does not include the surface-dipole term"};
   const int nid = e->max_id, npar = e->npar, ntypes = nid * (nid + 1) / 2;
   const int ntheta = ntypes * npar + nid, ns = e->nsites, nsp = e->nsp;
   // slots of a wave: half for dE, half for the cotangent when there is one
   const int half = nid * (npar + 1) + 1, nslot = v_host ? 2 * half : half;
   const size_t shm = sizeof(double) * (64 * (size_t)nslot + nid * MGPU_NPOTP) + sizeof(int2) * ADJ_QCAP;
   if (shm > 160 * 1024) throw StatusError{MGPU_E_CAPACITY, "too many site ids for the adjoint"};
   // the sites by id, cut into waves of one id each: about two rounds of the
   // waves that fit on the CUs (LDS), at most 16 sites a wave
   std::vector<int> bysite(ns), first(nid + 1, 0);
   for (int t : e->site_type) first[t + 1]++;
   for (int t = 0; t < nid; t++) first[t + 1] += first[t];
   {
      std::vector<int> at(first);
      for (int i = 0; i < ns; i++) bysite[at[e->site_type[i]]++] = i;
   }
   const int resident = e->ncu * std::max(1, std::min(16, (int)(160 * 1024 / shm)));
   const int per = std::max(1, std::min(16, ns / (2 * resident)));
   std::vector<int4> chunk;
   for (int t = 0; t < nid; t++)
      for (int s = first[t]; s < first[t + 1]; s += per)
         chunk.push_back(make_int4(s, std::min(s + per, first[t + 1]), t, 0));
   const int nw = (int)chunk.size();
   // device inputs
   size_t off = 0;
   auto take = [&](size_t bytes) { size_t o = off; off += (bytes + 255) & ~(size_t)255; return o; };
   const size_t oPart = take(sizeof(double) * (size_t)nw * nslot), oV = take(sizeof(double) * 3 * nsp),
                oJ = take(sizeof(double) * 3 * nsp), oDP = take(sizeof(double) * nid * nid * MGPU_NPOTP),
                oDQ = take(sizeof(double) * nid), oQ = take(sizeof(double) * nid), oT = take(sizeof(double) * 2 * ntheta),
                oPos = take(sizeof(int) * ns), oBy = take(sizeof(int) * ns), oCh = take(sizeof(int4) * nw);
   e->d_adj_real.reserve(off);
   uint8_t *B = e->d_adj_real.p;
   double *part = (double *)(B + oPart), *dv = (double *)(B + oV), *dj = (double *)(B + oJ),
          *ddp = (double *)(B + oDP), *ddq = (double *)(B + oDQ), *dqid = (double *)(B + oQ),
          *dth = (double *)(B + oT);
   int *pos = (int *)(B + oPos), *dby = (int *)(B + oBy);
   int4 *dch = (int4 *)(B + oCh);
   std::vector<double> hdp((size_t)nid * nid * MGPU_NPOTP, 0.0), hdq(nid, 0.0);
   if (dtheta) {
      for (int a = 0; a < nid; a++)
         for (int b = a; b < nid; b++) {
            int col = 0;
            for (int x = 0; x < a; x++) col += nid - x;
            col += b - a;
            for (int k = 0; k < npar; k++) {
               hdp[(size_t)(a * nid + b) * MGPU_NPOTP + k] = dtheta[col * npar + k];
               hdp[(size_t)(b * nid + a) * MGPU_NPOTP + k] = dtheta[col * npar + k];
            }
         }
      for (int a = 0; a < nid; a++) hdq[a] = dtheta[ntypes * npar + a];
   }
   HIPCHK(hipMemcpyAsync(ddp, hdp.data(), sizeof(double) * hdp.size(), hipMemcpyHostToDevice, e->stream));
   HIPCHK(hipMemcpyAsync(ddq, hdq.data(), sizeof(double) * nid, hipMemcpyHostToDevice, e->stream));
   HIPCHK(hipMemcpyAsync(dqid, e->site_charge.data(), sizeof(double) * nid, hipMemcpyHostToDevice, e->stream));
   HIPCHK(hipMemcpyAsync(dby, bysite.data(), sizeof(int) * ns, hipMemcpyHostToDevice, e->stream));
   HIPCHK(hipMemcpyAsync(dch, chunk.data(), sizeof(int4) * nw, hipMemcpyHostToDevice, e->stream));
   zero_async(e, dv, sizeof(double) * 3 * nsp);
   if (v_host)
      for (int c = 0; c < 3; c++)
         HIPCHK(hipMemcpyAsync(dv + (size_t)c * nsp, v_host + (size_t)c * ns, sizeof(double) * ns,
                               hipMemcpyHostToDevice, e->stream));
   zero_async(e, dj, sizeof(double) * 3 * nsp);
   // sites and cells of force_calc
   launch_make_sites(e, e->molpbc ? 1 : 0);
   zero_async(e, e->d_iflags.p, sizeof(int) * 48);
   run_binning(e, false);
   AdjArgs a;
   a.nsites = ns; a.nx = e->nx; a.ny = e->ny; a.nz = e->nz; a.nfull = e->n_full;
   a.max_id = nid; a.npar = npar; a.nsp = nsp; a.strict_sub = e->strict && !e->molpbc; a.nslot = nslot;
   a.alpha = e->alpha; a.norm = 2.0 * e->alpha / sqrt(PI_D);
   a.cutsq = e->cutoff * e->cutoff; a.cut100sq = 10000.0 * a.cutsq;
   int k = 0;
   for (int ii = -1; ii <= 1; ii++)
      for (int jj = -1; jj <= 1; jj++)
         for (int kk = -1; kk <= 1; kk++, k++) {
            a.reloc[3 * k] = e->h[0] * ii + e->h[1] * jj + e->h[2] * kk;
            a.reloc[3 * k + 1] = e->h[3] * ii + e->h[4] * jj + e->h[5] * kk;
            a.reloc[3 * k + 2] = e->h[6] * ii + e->h[7] * jj + e->h[8] * kk;
         }
   a.css = e->d_cell_site_start.p; a.off = e->d_off.p; a.cpos = e->d_cpos.p; a.cmeta = e->d_cmeta.p;
   a.corig = e->d_corig.p; a.ccell = e->d_ccell.p; a.potpar = e->d_potpar.p;
   a.pos = pos; a.bysite = dby; a.chunk = dch;
   a.v = v_host ? dv : nullptr;
   a.dpar = ddp; a.dq = ddq; a.chg_id = dqid; a.part = part;
   a.jvp = (jvp_host && dtheta) ? dj : nullptr;
   k_adj_pos<<<(ns + 255) / 256, 256, 0, e->stream>>>(ns, e->d_corig.p, pos);
   {
      ProfScope ps(e, "adjoint_real");
      if (e->alpha > 0.0) launch_adj_pt<true>(e->ptype, nw, shm, e->stream, a);
      else launch_adj_pt<false>(e->ptype, nw, shm, e->stream, a);
   }
   if (!v_host) zero_async(e, dth + ntheta, sizeof(double) * ntheta);
   k_adj_fold<<<dim3(ntheta, v_host ? 2 : 1), 256, 0, e->stream>>>(nw, nid, npar, nslot, half, dch, part, dth);
   std::vector<double> h(2 * (size_t)ntheta);
   HIPCHK(hipMemcpyAsync(h.data(), dth, sizeof(double) * 2 * ntheta, hipMemcpyDeviceToHost, e->stream));
   int fl[41];
   HIPCHK(hipMemcpyAsync(fl, e->d_iflags.p, sizeof fl, hipMemcpyDeviceToHost, e->stream));
   HIPCHK(hipStreamSynchronize(e->stream));
   if (fl[0] & FLAG_BIN_RANGE) throw StatusError{MGPU_E_BIN_RANGE, "Co-ordinate out of range in BIN (fill_cells)"};
   if (fl[0] & FLAG_BIN_ROUND) throw StatusError{MGPU_E_BIN_ROUND, "Rounding problem in BIN (fill_cells)"};
   std::vector<double> ge(h.begin(), h.begin() + ntheta), gv(h.begin() + ntheta, h.end());
   if (e->alpha > 1e-7) {
      std::vector<double> qe(nid, 0.0), qv(nid, 0.0);
      ewald_charge_adjoint(e, v_host ? dv : nullptr, ddq, qe.data(), qv.data(), a.jvp ? dj : nullptr);
      for (int q = 0; q < nid; q++) {
         ge[ntypes * npar + q] += qe[q];
         gv[ntypes * npar + q] += qv[q];
      }
   }
   static_grad(e, npar, ge.data());
   if (dE) std::copy(ge.begin(), ge.end(), dE);
   if (vjp) std::copy(gv.begin(), gv.end(), vjp);
   if (jvp_host) {
      if (!dtheta) {
         std::fill(jvp_host, jvp_host + 3 * (size_t)ns, 0.0);
      } else {
         for (int c = 0; c < 3; c++)
            HIPCHK(hipMemcpyAsync(jvp_host + (size_t)c * ns, dj + (size_t)c * nsp, sizeof(double) * ns,
                                  hipMemcpyDeviceToHost, e->stream));
         HIPCHK(hipStreamSynchronize(e->stream));
      }
   }
}
