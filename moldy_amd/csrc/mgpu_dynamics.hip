// Molecular-dynamics step on the device: do_step of src/accel.c:626-827 with
// the leapfrog splitting of src/leapfrog.c (centre-of-mass update with the
// metric G^-1, momentum kicks, the symplectic quaternion rotations of
// leapf_quat_a/leapf_quat_b), the Nose-Poincare thermostat and the
// Parrinello-Rahman / uniform-dilation barostat, in FP64.  At constant cell
// every launch of a step has fixed arguments and the whole step can be
// captured in a hipGraph; under the barostat the host reads the new h after
// the first cell half step and rebuilds the cell-dependent plans.
//
// Device layout: one thread per molecule; momenta mom[nmols][3] (scaled,
// mom = h^T p), principal angular momenta amom[nmols_r][4]; the integrator
// scalars (s, p_s, H_0, record counter, h, hmom) and per-species kinetic
// sums live in e->d_scal so that no value goes back to the host inside a
// constant-cell step.
#include "mgpu_internal.h"

#include <algorithm>
#include <cmath>
#include <cstring>

using namespace mgpu;

namespace {

constexpr double INERTIA_MIN = 1.0e-14;   // src/leapfrog.c:75
constexpr double QTOL = 1.0e-4;           // src/leapfrog.c:72
constexpr double DMIN = 2.2250738585072014e-308;

// d_scal slots: thermostat, record row, per-species KE sums (4 a species),
// cell h and hmom (row-major), per-species momentum dyads (6 a species)
// S_INIT: the next step sets H_0 (so that the step itself is the same captured graph)
enum { S_TS = 0, S_TSMOM = 1, S_H0 = 2, S_ROW = 3, S_INIT = 4, S_KE = 8, S_H = 64, S_HMOM = 73, S_DY = 82 };
constexpr int MAX_SPEC = 14;              // S_KE + 4 * MAX_SPEC <= S_H
constexpr int SCAL_SIZE = MGPU_SCAL_SIZE;            // S_DY + 6 * MAX_SPEC <= SCAL_SIZE
constexpr int TRACE_W = 8;                // ke_t, ke_r, pe0, pe1, ts, tsmom, H_0, det(h)

struct SpecDyn {
   double mass, I[3], rI[3], fw;
};

__device__ __forceinline__ void qmul(const double *p, const double *q, double *r) {
   double p0 = p[0], p1 = p[1], p2 = p[2], p3 = p[3];
   double q0 = q[0], q1 = q[1], q2 = q[2], q3 = q[3];
   r[0] = p0 * q0 - p1 * q1 - p2 * q2 - p3 * q3;
   r[1] = p1 * q0 + p0 * q1 - p3 * q2 + p2 * q3;
   r[2] = p2 * q0 + p3 * q1 + p0 * q2 - p1 * q3;
   r[3] = p3 * q0 - p2 * q1 + p1 * q2 + p0 * q3;
}

// rot_substep, src/leapfrog.c:238-244
__device__ __forceinline__ void rot_substep(const double *rot, double *L, double *q) {
   double rc[4] = {rot[0], -rot[1], -rot[2], -rot[3]};
   qmul(rc, L, L);
   qmul(L, rot, L);
   qmul(q, rot, q);
}

// Element i of three values by selection: an array indexed by a variable is
// put into LDS (64 KB a block of k_coords, which left two blocks a CU).
__device__ __forceinline__ double pick3(const double *x, int i) { return i == 0 ? x[0] : i == 1 ? x[1] : x[2]; }

// make_rot, src/leapfrog.c:193-208: rotation about a principal axis
__device__ __forceinline__ void rot_axis(double step, int axis, const double *L, double rinertia, double *rot) {
   double s, c;
   sincos(0.5 * step * rinertia * pick3(L + 1, axis), &s, &c);
   rot[0] = c;
   rot[1] = axis == 0 ? s : 0.0;
   rot[2] = axis == 1 ? s : 0.0;
   rot[3] = axis == 2 ? s : 0.0;
}

// make_rot_amom, src/leapfrog.c:213-231: rotation about L
__device__ __forceinline__ void rot_amom(double step, const double *L, double rinertia, double *rot) {
   double samom = sqrt(L[1] * L[1] + L[2] * L[2] + L[3] * L[3]);
   double ramom = 1.0 / (samom + 8 * DMIN);
   double s, c;
   sincos(0.5 * step * rinertia * samom, &s, &c);
   rot[0] = c;
   rot[1] = s * ramom * L[1];
   rot[2] = s * ramom * L[2];
   rot[3] = s * ramom * L[3];
}

struct CoordArgs {
   int nmols;
   double step;          // the half step of leapf_all_coords
   double Gi[9];         // (h^T h)^-1
   int do_com;           // centre-of-mass update in this launch
   int ph_lo, ph_hi;     // rotation sub-steps [ph_lo, ph_hi) of the splitting
   int variant_a;        // leapf_quat_a (else leapf_quat_b)
   int saxis;            // near-symmetry axis of leapf_quat_b
   int normalise;        // normalise after the last sub-step
};

// leapf_all_coords (src/accel.c:360-372): leapf_com (leapfrog.c:133-146) and
// the sub-steps [ph_lo, ph_hi) of leapf_quat_b (leapfrog.c:255-338: 0 half
// delta about o1, 1 precession about the symmetry axis and spin about L, 2
// half delta about o1) or leapf_quat_a (leapfrog.c:345-392: axes 0,1,2,1,0
// with weights 1/2,1/2,1,1/2,1/2), then normalise (leapfrog.c:96-113).
// One molecule m (no restrict: the fused kernels write mom and amom first).
__device__ __forceinline__ void coords_one(int m, const CoordArgs &a, const int *mol_spec, const int *mol_quat,
                                           const SpecDyn *sd, const double *scal, const double *mom, double *cm,
                                           double *quat, double *amom, int *flags) {
   const int sp = mol_spec[m];
   const SpecDyn S = sd[sp];
   const double ts = scal[S_TS];
   if (a.do_com) {
      const double c = a.step / (S.mass * ts);
      double A[9];
#pragma unroll
      for (int i = 0; i < 9; i++) A[i] = c * a.Gi[i];
      double *r = cm + 3 * m;
      const double *p = mom + 3 * m;
      double y0 = r[0] + A[0] * p[0] + A[1] * p[1] + A[2] * p[2];
      double y1 = r[1] + A[3] * p[0] + A[4] * p[1] + A[5] * p[2];
      double y2 = r[2] + A[6] * p[0] + A[7] * p[1] + A[8] * p[2];
      // escape, leapfrog.c:117-128
      r[0] = y0 - floor(y0 + 0.5);
      r[1] = y1 - floor(y1 + 0.5);
      r[2] = y2 - floor(y2 + 0.5);
   }
   const int iq = mol_quat[m];
   if (iq < 0 || a.ph_hi <= a.ph_lo) return;
   double q[4], L[4], rot[4];
#pragma unroll
   for (int k = 0; k < 4; k++) { q[k] = quat[4 * iq + k]; L[k] = amom[4 * iq + k]; }
   const double stepdts = a.step / ts;
   for (int ph = a.ph_lo; ph < a.ph_hi; ph++) {
      if (a.variant_a) {
         const int ax = ph == 0 || ph == 4 ? 0 : (ph == 2 ? 2 : 1);
         const double w = ph == 2 ? 1.0 : 0.5;
         rot_axis(w * stepdts, ax, L, pick3(S.rI, ax), rot);
         rot_substep(rot, L, q);
      } else {
         const int s = a.saxis, o1 = (s + 1) % 3, o2 = (s + 2) % 3;
         if (ph == 1) {
            rot_axis(stepdts, s, L, pick3(S.rI, s) - pick3(S.rI, o2), rot);
            rot_substep(rot, L, q);
            rot_amom(stepdts, L, pick3(S.rI, o2), rot);
            qmul(q, rot, q);
         } else {
            rot_axis(0.5 * stepdts, o1, L, pick3(S.rI, o1) - pick3(S.rI, o2), rot);
            rot_substep(rot, L, q);
         }
      }
   }
   if (a.normalise) {
      double n = sqrt(q[0] * q[0] + q[1] * q[1] + q[2] * q[2] + q[3] * q[3]);
      if (fabs(n - 1.0) > QTOL) {
         atomicOr(flags, FLAG_QNORM);
         atomicCAS(flags + 40, 0, m + 1);
      }
#pragma unroll
      for (int k = 0; k < 4; k++) q[k] /= n;
   }
#pragma unroll
   for (int k = 0; k < 4; k++) { quat[4 * iq + k] = q[k]; amom[4 * iq + k] = L[k]; }
}
__device__ __forceinline__ void b_coords(int bx, int nbx, const CoordArgs &a, const int *mol_spec,
                                         const int *mol_quat, const SpecDyn *sd, const double *scal,
                                         const double *mom, double *cm, double *quat, double *amom, int *flags) {
   const int m = bx * 256 + threadIdx.x;
   if (m < a.nmols) coords_one(m, a, mol_spec, mol_quat, sd, scal, mom, cm, quat, amom, flags);
}
__global__ __launch_bounds__(256) void k_coords(CoordArgs a, const int *__restrict__ mol_spec, const int *__restrict__ mol_quat,
                         const SpecDyn *__restrict__ sd, const double *__restrict__ scal,
                         const double *__restrict__ mom, double *__restrict__ cm, double *__restrict__ quat,
                         double *__restrict__ amom, int *__restrict__ flags) {
   b_coords(blockIdx.x, gridDim.x, a, mol_spec, mol_quat, sd, scal, mom, cm, quat, amom, flags);
}

struct MomArgs {
   int nmols;
   double step;          // the half step of leapf_all_momenta
   double hT[9];         // h^T
   int zero_fw;          // zero framework momenta afterwards (accel.c:752-757)
};

// leapf_all_momenta, src/accel.c:376-388 (leapf_mom, leapf_amom)
__device__ __forceinline__ void mom_one(int m, const MomArgs &a, const int *mol_spec, const int *mol_quat,
                                        const SpecDyn *sd, const double *scal, const double *force,
                                        const double *torque, double *mom, double *amom) {
   const double c = a.step * scal[S_TS];
   double A[9];
#pragma unroll
   for (int i = 0; i < 9; i++) A[i] = c * a.hT[i];
   double *p = mom + 3 * m;
   const double *f = force + 3 * m;
   double y0 = p[0] + A[0] * f[0] + A[1] * f[1] + A[2] * f[2];
   double y1 = p[1] + A[3] * f[0] + A[4] * f[1] + A[5] * f[2];
   double y2 = p[2] + A[6] * f[0] + A[7] * f[1] + A[8] * f[2];
   if (a.zero_fw && sd[mol_spec[m]].fw != 0.0) y0 = y1 = y2 = 0.0;
   p[0] = y0; p[1] = y1; p[2] = y2;
   const int iq = mol_quat[m];
   if (iq >= 0) {
      amom[4 * iq + 1] += c * torque[3 * iq];
      amom[4 * iq + 2] += c * torque[3 * iq + 1];
      amom[4 * iq + 3] += c * torque[3 * iq + 2];
   }
}
__device__ __forceinline__ void b_momenta(int bx, int nbx, const MomArgs &a, const int *mol_spec,
                                          const int *mol_quat, const SpecDyn *sd, const double *scal,
                                          const double *force, const double *torque, double *mom, double *amom) {
   const int m = bx * 256 + threadIdx.x;
   if (m < a.nmols) mom_one(m, a, mol_spec, mol_quat, sd, scal, force, torque, mom, amom);
}
__global__ __launch_bounds__(256) void k_momenta(MomArgs a, const int *mol_spec, const int *mol_quat,
                                                 const SpecDyn *sd, const double *scal, const double *force,
                                                 const double *torque, double *mom, double *amom) {
   b_momenta(blockIdx.x, gridDim.x, a, mol_spec, mol_quat, sd, scal, force, torque, mom, amom);
}

// The second momentum half step and, without a thermostat's scalars between
// them, the coordinate half step after it: one launch for two.
__device__ __forceinline__ void b_mom_coords(int bx, int nbx, const MomArgs &a, const CoordArgs &c,
                                             const int *mol_spec, const int *mol_quat, const SpecDyn *sd,
                                             const double *scal, const double *force, const double *torque,
                                             double *mom, double *cm, double *quat, double *amom, int *flags) {
   const int m = bx * 256 + threadIdx.x;
   if (m >= a.nmols) return;
   mom_one(m, a, mol_spec, mol_quat, sd, scal, force, torque, mom, amom);
   coords_one(m, c, mol_spec, mol_quat, sd, scal, mom, cm, quat, amom, flags);
}
__global__ __launch_bounds__(256) void k_mom_coords(MomArgs a, CoordArgs c, const int *mol_spec, const int *mol_quat,
                                                    const SpecDyn *sd, const double *scal, const double *force,
                                                    const double *torque, double *mom, double *cm, double *quat,
                                                    double *amom, int *flags) {
   b_mom_coords(blockIdx.x, gridDim.x, a, c, mol_spec, mol_quat, sd, scal, force, torque, mom, cm, quat, amom, flags);
}

struct KeArgs {
   int nmols, nspec;
   double hiT[9];        // (h^-1)^T: real momenta
};

// Per-species sums of |p_real|^2 and amom_k^2 (k = 1..3): columns 4s+0..3
// of a [nblocks][4 nspec] partial array (trans_ke and rot_ke numerators,
// src/algorith.c:221-259).  Deterministic: wave sums, fixed block order.
__device__ __forceinline__ void b_ke_part(int bx, int nbx, const KeArgs &a, const int *mol_spec,
                                          const int *mol_quat, const double *mom, const double *amom, double *part) {
   __shared__ double ws[4][4 * MAX_SPEC];
   int m = bx * 256 + threadIdx.x;
   double v[4] = {0, 0, 0, 0};
   int sp = -1;
   if (m < a.nmols) {
      sp = mol_spec[m];
      const double *q = mom + 3 * m;
      double p0 = a.hiT[0] * q[0] + a.hiT[1] * q[1] + a.hiT[2] * q[2];
      double p1 = a.hiT[3] * q[0] + a.hiT[4] * q[1] + a.hiT[5] * q[2];
      double p2 = a.hiT[6] * q[0] + a.hiT[7] * q[1] + a.hiT[8] * q[2];
      v[0] = p0 * p0 + p1 * p1 + p2 * p2;
      const int iq = mol_quat[m];
      if (iq >= 0) {
         v[1] = amom[4 * iq + 1] * amom[4 * iq + 1];
         v[2] = amom[4 * iq + 2] * amom[4 * iq + 2];
         v[3] = amom[4 * iq + 3] * amom[4 * iq + 3];
      }
   }
   const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
   for (int s = 0; s < a.nspec; s++)
      for (int k = 0; k < 4; k++) {
         double t = wave_sum(sp == s ? v[k] : 0.0);
         if (lane == 0) ws[w][4 * s + k] = t;
      }
   __syncthreads();
   const int nc = 4 * a.nspec;
   if (threadIdx.x < nc)
      part[(size_t)bx * nc + threadIdx.x] =
          ws[0][threadIdx.x] + ws[1][threadIdx.x] + ws[2][threadIdx.x] + ws[3][threadIdx.x];
}
__global__ __launch_bounds__(256) void k_ke_part(KeArgs a, const int *__restrict__ mol_spec,
                                                 const int *__restrict__ mol_quat, const double *__restrict__ mom,
                                                 const double *__restrict__ amom, double *__restrict__ part) {
   b_ke_part(blockIdx.x, gridDim.x, a, mol_spec, mol_quat, mom, amom, part);
}

// The first momentum half step and the kinetic sums of what it leaves.
__device__ __forceinline__ void b_mom_ke(int bx, int nbx, const MomArgs &a, const KeArgs &k, const int *mol_spec,
                                         const int *mol_quat, const SpecDyn *sd, const double *scal,
                                         const double *force, const double *torque, double *mom, double *amom,
                                         double *part) {
   const int m = bx * 256 + threadIdx.x;
   if (m < a.nmols) mom_one(m, a, mol_spec, mol_quat, sd, scal, force, torque, mom, amom);
   b_ke_part(bx, nbx, k, mol_spec, mol_quat, mom, amom, part);   // each thread its own molecule again
}
__global__ __launch_bounds__(256) void k_mom_ke(MomArgs a, KeArgs k, const int *mol_spec, const int *mol_quat,
                                                const SpecDyn *sd, const double *scal, const double *force,
                                                const double *torque, double *mom, double *amom, double *part) {
   b_mom_ke(blockIdx.x, gridDim.x, a, k, mol_spec, mol_quat, sd, scal, force, torque, mom, amom, part);
}

// Per-species sums of the real-momentum dyad p p^T (energy_dyad,
// src/algorith.c:261-285): columns 6s + {xx, xy, xz, yy, yz, zz}.
__device__ __forceinline__ void b_dyad_part(int bx, int nbx, const KeArgs &a, const int *__restrict__ mol_spec,
                                            const double *__restrict__ mom, double *__restrict__ part) {
   __shared__ double ws[4][6 * MAX_SPEC];
   int m = bx * 256 + threadIdx.x;
   double v[6] = {0, 0, 0, 0, 0, 0};
   int sp = -1;
   if (m < a.nmols) {
      sp = mol_spec[m];
      const double *q = mom + 3 * m;
      double p0 = a.hiT[0] * q[0] + a.hiT[1] * q[1] + a.hiT[2] * q[2];
      double p1 = a.hiT[3] * q[0] + a.hiT[4] * q[1] + a.hiT[5] * q[2];
      double p2 = a.hiT[6] * q[0] + a.hiT[7] * q[1] + a.hiT[8] * q[2];
      v[0] = p0 * p0; v[1] = p0 * p1; v[2] = p0 * p2;
      v[3] = p1 * p1; v[4] = p1 * p2; v[5] = p2 * p2;
   }
   const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
   for (int s = 0; s < a.nspec; s++)
      for (int k = 0; k < 6; k++) {
         double t = wave_sum(sp == s ? v[k] : 0.0);
         if (lane == 0) ws[w][6 * s + k] = t;
      }
   __syncthreads();
   const int nc = 6 * a.nspec;
   if (threadIdx.x < nc)
      part[(size_t)bx * nc + threadIdx.x] =
          ws[0][threadIdx.x] + ws[1][threadIdx.x] + ws[2][threadIdx.x] + ws[3][threadIdx.x];
}
__global__ __launch_bounds__(256) void k_dyad_part(KeArgs a, const int *__restrict__ mol_spec,
                                                   const double *__restrict__ mom, double *__restrict__ part) {
   b_dyad_part(blockIdx.x, gridDim.x, a, mol_spec, mom, part);
}

// Column sums of the partials into out[0 .. nc), one block: 256 / nc threads a
// column each add every such row in order, then those sums are added in
// order.  (One thread a column took 25 to 48 us for 135 to 422 rows, a load's
// latency each.)
__device__ __forceinline__ void b_col_sum(int bx, int nbx, int nblocks, int nc, const double *part, double *out) {
   __shared__ double s[256];
   const int per = 256 / nc, c = (int)threadIdx.x % nc, q = (int)threadIdx.x / nc;
   double t = 0.0;
   if (q < per)
      for (int b = q; b < nblocks; b += per) t += part[(size_t)b * nc + c];
   s[threadIdx.x] = t;
   __syncthreads();
   if ((int)threadIdx.x < nc) {
      double u = 0.0;
      for (int k = 0; k < per; k++) u += s[k * nc + threadIdx.x];
      out[threadIdx.x] = u;
   }
}
__global__ __launch_bounds__(256) void k_col_sum(int nblocks, int nc, const double *__restrict__ part,
                                                 double *__restrict__ out) {
   b_col_sum(blockIdx.x, gridDim.x, nblocks, nc, part, out);
}

enum {
   OP_THERM_IN = 0,     // leapf_nose_therm then the log term (accel.c:680-682)
   OP_THERM_OUT,        // the log term then leapf_nose_therm (accel.c:788-789)
   OP_TSMOM_TRANS,      // tsmom += 1/2 step KE_trans (accel.c:698-699, 765-766)
   OP_TSMOM_ROT,        // tsmom += 1/2 h rot_ke (leapfrog.c:298-299, 317-318)
   OP_TSMOM_AXES,       // tsmom += w * stepdts2 * rI_k * sum amom_k^2 (leapfrog.c:364-381)
   OP_RECORD,           // KE at the H_0 point, H_0, trace row (accel.c:714-724)
   OP_TSMOM_PE,         // tsmom -= step (pe - H_0) (accel.c:759-760)
   OP_RESET_ROW,
   OP_GLEAP_CELL,       // gleap_cell at a half step (accel.c:688-690, 777-779)
   OP_HMOM_KIN,         // update_hmom with stress_kin at a half step (accel.c:700-704, 767-771)
   OP_HMOM_VIR          // update_hmom with the virial at a full step (accel.c:760-761)
};

struct ScalArgs {
   int op, nspec, init_h0, trace_cap;
   int ke_rows;          // rows of kinetic partials to sum into S_KE first (0: none)
   double step, ttmass, pmass, gkt;
   double w[3];                 // per-axis weights (OP_TSMOM_AXES), order of addition
   int axes[3], naxes;
   int const_temp, const_pressure, uniform, strain_mask;
   double pressure;
};

// 3x3 helpers in the index order of src/algorith.c (det, mk_sigma,
// trace_sqr) and src/leapfrog.c (ke_cell).
__device__ double det3(const double *a) {
   double d = 0.0;
   for (int i = 0, j = 1, k = 2; i < 3; i++, j = (j + 1) % 3, k = (k + 1) % 3)
      d += a[i] * (a[3 + j] * a[6 + k] - a[3 + k] * a[6 + j]);
   return d;
}

__device__ void mk_sigma(const double *h, double *sg) {
   for (int i = 0, j = 1, k = 2; i < 3; i++, j = (j + 1) % 3, k = (k + 1) % 3)
      for (int l = 0, m = 1, n = 2; l < 3; l++, m = (m + 1) % 3, n = (n + 1) % 3)
         sg[3 * i + l] = h[3 * j + m] * h[3 * k + n] - h[3 * k + m] * h[3 * j + n];
}

__device__ double sum_sq9(const double *m) {
   double t = 0.0;
   for (int i = 0; i < 9; i++) t += m[i] * m[i];
   return t;
}

// leapf_hmom, src/leapfrog.c:415-430: pressure term, strain mask in
// row-major bit order
__device__ void leapf_hmom(double step, double *hmom, const double *sigma, double s, double pressure, int mask) {
   const double r = 0.5 * step * s * pressure;
   for (int i = 0; i < 9; i++) {
      if (mask & 1) hmom[i] = 0.0;
      else hmom[i] -= r * sigma[i];
      mask >>= 1;
   }
}

__device__ void hmom_pressure(const ScalArgs &a, double step, double s, const double *h, double *hmom) {
   if (a.uniform) {
      const double vol = det3(h);
      leapf_hmom(step, hmom, h, 3.0 * vol * s / sum_sq9(h), a.pressure, a.strain_mask);
   } else {
      double sg[9];
      mk_sigma(h, sg);
      leapf_hmom(step, hmom, sg, s, a.pressure, a.strain_mask);
   }
}

// update_hmom, src/leapfrog.c:516-531; sp is a stress times the volume
__device__ void update_hmom(const ScalArgs &a, double step, double s, const double *h, const double *sp,
                            double *hmom) {
   double t[9];
   if (a.uniform) {
      const double c = step * s * (sp[0] + sp[4] + sp[8]) / sum_sq9(h);
      for (int i = 0; i < 9; i++) t[i] = c * h[i];
   } else {
      double sg[9];
      const double vol = det3(h);
      mk_sigma(h, sg);
      for (int i = 0; i < 3; i++)
         for (int j = 0; j < 3; j++) {
            double x = 0.0;
            for (int k = 0; k < 3; k++) x += sp[3 * i + k] * sg[3 * k + j];
            t[3 * i + j] = x;
         }
      const double c = step * s / vol;
      for (int i = 0; i < 9; i++) t[i] *= c;
   }
   for (int i = 0; i < 9; i++) hmom[i] += t[i];
}

__device__ double ke_trans(const ScalArgs &a, const SpecDyn *sd, const double *scal) {
   double ts = scal[S_TS], ke = 0.0;
   for (int s = 0; s < a.nspec; s++) ke += scal[S_KE + 4 * s] / (2.0 * sd[s].mass * ts * ts);
   return ke;
}

__device__ double ke_rot(const ScalArgs &a, const SpecDyn *sd, const double *scal, int s) {
   double ts = scal[S_TS], ke = 0.0;
   for (int i = 0; i < 3; i++)
      if (sd[s].I[i] > INERTIA_MIN) ke += scal[S_KE + 4 * s + 1 + i] / sd[s].I[i];
   return 0.5 * ke / (ts * ts);
}

__device__ __forceinline__ void b_scalar(int bx, int nbx, const ScalArgs &a, const SpecDyn *sd, const int *spec_rdof,
                                         const double *res, const double *part, double *scal, double *trace) {
   if (bx != 0) return;
   if (a.ke_rows > 0) {
      b_col_sum(0, 1, a.ke_rows, 4 * a.nspec, part, scal + S_KE);
      __syncthreads();
   }
   if (threadIdx.x != 0) return;
   double &ts = scal[S_TS], &tsmom = scal[S_TSMOM];
   switch (a.op) {
      case OP_THERM_IN:
      case OP_THERM_OUT: {
         const double h = 0.5 * a.step;
         if (a.op == OP_THERM_OUT) tsmom -= h * a.gkt * (1.0 + log(ts));
         const double scale = 1.0 + tsmom * h / (2.0 * a.ttmass);   // leapfrog.c:468-474
         tsmom /= scale;
         ts *= scale * scale;
         if (a.op == OP_THERM_IN) tsmom -= h * a.gkt * (1.0 + log(ts));
         break;
      }
      case OP_TSMOM_TRANS: tsmom += 0.5 * a.step * ke_trans(a, sd, scal); break;
      case OP_TSMOM_ROT:
         for (int s = 0; s < a.nspec; s++)
            if (spec_rdof[s] > 0) tsmom += 0.5 * a.step * ke_rot(a, sd, scal, s);
         break;
      case OP_TSMOM_AXES: {
         const double stepdts2 = a.step / (ts * ts);
         for (int s = 0; s < a.nspec; s++)
            if (spec_rdof[s] > 0)
               for (int k = 0; k < a.naxes; k++)
                  tsmom += a.w[k] * stepdts2 * sd[s].rI[a.axes[k]] * scal[S_KE + 4 * s + 1 + a.axes[k]];
         break;
      }
      case OP_RECORD: {
         double kt = ke_trans(a, sd, scal), kr = 0.0;
         for (int s = 0; s < a.nspec; s++)
            if (spec_rdof[s] > 0) kr += ke_rot(a, sd, scal, s);
         const double pe0 = res[0], pe1 = res[1];
         const double vol = det3(scal + S_H);
         if (scal[S_INIT] != 0.0) {
            scal[S_H0] = (kt + kr) + (pe0 + pe1) + tsmom * tsmom / (2.0 * a.ttmass) + a.gkt * log(ts) +
                         0.5 / a.pmass * sum_sq9(scal + S_HMOM);
            if (a.const_pressure) scal[S_H0] += a.pressure * vol;
         }
         int row = (int)scal[S_ROW];
         if (row < a.trace_cap) {
            double *t = trace + (size_t)row * TRACE_W;
            t[0] = kt; t[1] = kr; t[2] = pe0; t[3] = pe1; t[4] = ts; t[5] = tsmom; t[6] = scal[S_H0];
            t[7] = vol;
         }
         scal[S_ROW] = row + 1;
         scal[S_INIT] = 0.0;
         break;
      }
      case OP_TSMOM_PE: tsmom -= a.step * (res[0] + res[1] - scal[S_H0]); break;
      case OP_RESET_ROW:
         scal[S_ROW] = 0.0;
         scal[S_INIT] = a.init_h0 ? 1.0 : 0.0;
         break;
      case OP_GLEAP_CELL: {
         // gleap_cell, src/leapfrog.c:475-508, at step = a.step / 2
         const double st = 0.5 * a.step;
         double *h = scal + S_H, *hm = scal + S_HMOM;
         hmom_pressure(a, st, ts, h, hm);
         if (a.const_temp) tsmom -= 0.5 * st * (0.5 / a.pmass * sum_sq9(hm) + a.pressure * det3(h));
         const double r = st * ts / a.pmass;   // leapf_h
         for (int i = 0; i < 9; i++) h[i] += r * hm[i];
         if (a.const_temp) tsmom -= 0.5 * st * (0.5 / a.pmass * sum_sq9(hm) + a.pressure * det3(h));
         hmom_pressure(a, st, ts, h, hm);
         break;
      }
      case OP_HMOM_KIN: {
         // stress_kin (accel.c:349-355): sum over species of dyad / (m s^2)
         double kd[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
         const int ij[9] = {0, 1, 2, 1, 3, 4, 2, 4, 5};
         for (int s = 0; s < a.nspec; s++) {
            const double d = sd[s].mass * ts * ts;
            for (int q = 0; q < 9; q++) kd[q] += scal[S_DY + 6 * s + ij[q]] / d;
         }
         update_hmom(a, 0.5 * a.step, ts, scal + S_H, kd, scal + S_HMOM);
         break;
      }
      case OP_HMOM_VIR: update_hmom(a, a.step, ts, scal + S_H, res + 5, scal + S_HMOM); break;
   }
}
__global__ __launch_bounds__(256) void k_scalar(ScalArgs a, const SpecDyn *sd, const int *spec_rdof,
                                                const double *res, const double *part, double *scal, double *trace) {
   b_scalar(blockIdx.x, gridDim.x, a, sd, spec_rdof, res, part, scal, trace);
}

void matmul3(const double *a, const double *b, double *c) {
   for (int i = 0; i < 3; i++)
      for (int j = 0; j < 3; j++) {
         double t = 0;
         for (int k = 0; k < 3; k++) t += a[3 * i + k] * b[3 * k + j];
         c[3 * i + j] = t;
      }
}

ScalArgs scal_args(mgpu_engine *e, int op) {
   ScalArgs a{};
   a.op = op;
   a.nspec = e->nspecies;
   a.trace_cap = e->trace_cap;
   a.step = e->dyn_step;
   a.ttmass = e->dyn_ttmass;
   a.pmass = e->dyn_pmass;
   a.gkt = e->dyn_gkt;
   a.const_temp = e->dyn_const_temp;
   a.const_pressure = e->dyn_const_pressure;
   a.uniform = e->dyn_const_pressure > 0 && e->dyn_const_pressure % 2 == 0;   // accel.c:657
   a.strain_mask = e->dyn_strain_mask;
   a.pressure = e->dyn_pressure;
   return a;
}

void scalar_op(mgpu_engine *e, const ScalArgs &a) {
   glaunch<k_scalar, b_scalar, 256>(e->rec, e->stream, 1, 256, 0, a, (const SpecDyn *)e->d_spec_dyn.p,
                                    e->d_spec_rdof.p, e->d_out.p + OUT_RES, e->d_red.p, e->d_scal.p, e->d_trace.p);
}

KeArgs ke_args(mgpu_engine *e) {
   KeArgs k;
   k.nmols = e->nmols;
   k.nspec = e->nspecies;
   for (int i = 0; i < 3; i++)
      for (int j = 0; j < 3; j++) k.hiT[3 * i + j] = e->hinv[3 * j + i];
   return k;
}

// The kinetic sums, then the scalar update that needs them (which adds the
// partials itself: one launch for two).
void ke_scalar(mgpu_engine *e, ScalArgs a) {
   a.ke_rows = (e->nmols + 255) / 256;
   glaunch<k_ke_part, b_ke_part, 256>(e->rec, e->stream, a.ke_rows, 256, 0, ke_args(e), e->d_mol_spec.p,
                                      e->d_mol_quat.p, e->d_mom.p, e->d_amom.p, e->d_red.p);
   scalar_op(e, a);
}

void dyad_sums(mgpu_engine *e) {
   const int nb = (e->nmols + 255) / 256, nc = 6 * e->nspecies;
   glaunch<k_dyad_part, b_dyad_part, 256>(e->rec, e->stream, nb, 256, 0, ke_args(e), e->d_mol_spec.p, e->d_mom.p,
                                          e->d_red.p);
   glaunch<k_col_sum, b_col_sum, 256>(e->rec, e->stream, 1, 256, 0, nb, nc, e->d_red.p, e->d_scal.p + S_DY);
}

// Arguments of a leapf_all_coords half step in one launch.
CoordArgs coord_args(mgpu_engine *e) {
   CoordArgs c{};
   c.nmols = e->nmols;
   c.step = 0.5 * e->dyn_step;
   double ht[9], G[9];
   for (int i = 0; i < 3; i++)
      for (int j = 0; j < 3; j++) ht[3 * i + j] = e->h[3 * j + i];
   matmul3(ht, e->h, G);
   host_invert(G, c.Gi);
   c.variant_a = e->dyn_nosym;
   c.saxis = e->dyn_saxis;
   c.do_com = 1;
   c.ph_hi = e->nmols_r ? (e->dyn_nosym ? 5 : 3) : 0;
   c.normalise = 1;
   return c;
}

// The thermostat's rotational terms come between the rotation sub-steps.
bool split_coords(const mgpu_engine *e) { return e->dyn_const_temp && e->nmols_r > 0; }

// One leapf_all_coords half step, with the thermostat's rotational terms
// between the rotation sub-steps when the thermostat is on.
void coords_half(mgpu_engine *e) {
   CoordArgs c = coord_args(e);
   const int nb = (e->nmols + 255) / 256;
   const int nph = e->dyn_nosym ? 5 : 3;
   auto launch = [&](int com, int lo, int hi) {
      c.do_com = com;
      c.ph_lo = lo;
      c.ph_hi = hi;
      c.normalise = hi == nph;
      glaunch<k_coords, b_coords, 256>(e->rec, e->stream, nb, 256, 0, c, e->d_mol_spec.p, e->d_mol_quat.p,
                                        (const SpecDyn *)e->d_spec_dyn.p, e->d_scal.p, e->d_mom.p, e->d_cm.p,
                                        e->d_quat.p, e->d_amom.p, e->d_iflags.p);
   };
   if (!split_coords(e)) {
      launch(1, 0, c.ph_hi);
      return;
   }
   if (!e->dyn_nosym) {
      launch(1, 0, 1);
      ScalArgs a = scal_args(e, OP_TSMOM_ROT);
      a.step = c.step;
      ke_scalar(e, a);
      launch(0, 1, 2);
      ke_scalar(e, a);
      launch(0, 2, 3);
   } else {
      // leapf_quat_a: sums after sub-steps 0, 1 and 3
      launch(1, 0, 1);
      ScalArgs a = scal_args(e, OP_TSMOM_AXES);
      a.step = c.step;
      a.naxes = 2; a.axes[0] = 0; a.axes[1] = 1; a.w[0] = 0.25; a.w[1] = 0.25;
      ke_scalar(e, a);
      launch(0, 1, 2);
      a.naxes = 1; a.axes[0] = 2; a.w[0] = 0.5;
      ke_scalar(e, a);
      launch(0, 2, 4);
      a.naxes = 2; a.axes[0] = 1; a.axes[1] = 0; a.w[0] = 0.25; a.w[1] = 0.25;
      ke_scalar(e, a);
      launch(0, 4, 5);
   }
}

MomArgs mom_args(mgpu_engine *e, bool zero_fw) {
   MomArgs m{};
   m.nmols = e->nmols;
   m.step = 0.5 * e->dyn_step;
   for (int i = 0; i < 3; i++)
      for (int j = 0; j < 3; j++) m.hT[3 * i + j] = e->h[3 * j + i];
   m.zero_fw = zero_fw;
   return m;
}

// The first momentum half step, the kinetic sums and the step's record.
void momenta_record(mgpu_engine *e) {
   ScalArgs a = scal_args(e, OP_RECORD);
   a.ke_rows = (e->nmols + 255) / 256;
   glaunch<k_mom_ke, b_mom_ke, 256>(e->rec, e->stream, a.ke_rows, 256, 0, mom_args(e, false), ke_args(e),
                                    e->d_mol_spec.p, e->d_mol_quat.p, (const SpecDyn *)e->d_spec_dyn.p, e->d_scal.p,
                                    e->d_mforce.p, e->d_mtorque.p, e->d_mom.p, e->d_amom.p, e->d_red.p);
   scalar_op(e, a);
}

// The second momentum half step.
void momenta_half(mgpu_engine *e) {
   glaunch<k_momenta, b_momenta, 256>(e->rec, e->stream, (e->nmols + 255) / 256, 256, 0, mom_args(e, true),
                                      e->d_mol_spec.p, e->d_mol_quat.p, (const SpecDyn *)e->d_spec_dyn.p, e->d_scal.p,
                                      e->d_mforce.p, e->d_mtorque.p, e->d_mom.p, e->d_amom.p);
}

// The second momentum half step and the coordinate half step after it, with
// no thermostat between them.
void momenta_coords(mgpu_engine *e) {
   glaunch<k_mom_coords, b_mom_coords, 256>(
       e->rec, e->stream, (e->nmols + 255) / 256, 256, 0, mom_args(e, true), coord_args(e), e->d_mol_spec.p,
       e->d_mol_quat.p, (const SpecDyn *)e->d_spec_dyn.p, e->d_scal.p, e->d_mforce.p, e->d_mtorque.p, e->d_mom.p,
       e->d_cm.p, e->d_quat.p, e->d_amom.p, e->d_iflags.p);
}

}  // namespace

void mgpu::md_setup(mgpu_engine *e, const mgpu_dynamics *d) {
   if (e->nspecies > MAX_SPEC) throw StatusError{MGPU_E_CAPACITY, "more than 14 species in the MD step"};
   // a zero step is a static run (positions held, forces evaluated each step)
   if (!(d->step >= 0)) throw StatusError{MGPU_E_ARG, "step must not be negative"};
   if (d->const_temp && !(d->ttmass > 0)) throw StatusError{MGPU_E_ARG, "ttmass must be positive"};
   if (d->const_pressure < 0 || d->const_pressure > 2)
      throw StatusError{MGPU_E_ARG, "const_pressure must be 0, 1 or 2"};
   if (!(d->pmass > 0)) throw StatusError{MGPU_E_ARG, "pmass must be positive"};
   std::vector<SpecDyn> sd(e->nspecies);
   e->spec_mass.assign(d->spec_mass, d->spec_mass + e->nspecies);
   e->spec_inertia.assign(d->spec_inertia, d->spec_inertia + 3 * e->nspecies);
   int saxis = 0;
   bool first = true;
   for (int s = 0; s < e->nspecies; s++) {
      if (!(d->spec_mass[s] > 0)) throw StatusError{MGPU_E_ARG, "species mass must be positive"};
      SpecDyn &S = sd[s];
      S.mass = d->spec_mass[s];
      const double *I = d->spec_inertia + 3 * s;
      for (int i = 0; i < 3; i++) {
         S.I[i] = I[i];
         // leapfrog.c:263-269
         S.rI[i] = (e->spec_rdof[s] > 0 && !(I[i] / (I[(i + 1) % 3] + I[(i + 2) % 3]) < INERTIA_MIN)) ? 1.0 / I[i]
                                                                                                     : 0.0;
      }
      S.fw = e->spec_fw[s] ? 1.0 : 0.0;
      if (e->spec_rdof[s] > 0 && first) {
         // near-symmetry axis, leapfrog.c:275-290; the reference keeps the
         // first species' choice for all later ones (a static)
         double idmin = 1.0e37;
         for (int i = 0; i < 3; i++) {
            double idiff = fabs(S.rI[(i + 1) % 3] - S.rI[(i + 2) % 3]);
            if (idiff < idmin) { idmin = idiff; saxis = i; }
         }
         first = false;
      }
   }
   e->dyn_step = d->step;
   e->dyn_ttmass = d->ttmass;
   e->dyn_pmass = d->pmass;
   e->dyn_gkt = d->gkt;
   e->dyn_const_temp = d->const_temp != 0;
   e->dyn_nosym = d->nosymmetric_rot != 0;
   e->dyn_const_pressure = d->const_pressure;
   e->dyn_pressure = d->pressure;
   e->dyn_strain_mask = d->strain_mask;
   for (int i = 0; i < 9; i++) e->hmom[i] = 0.0;
   e->dyn_saxis = saxis;
   e->d_spec_dyn.reserve(sizeof(SpecDyn) / sizeof(double) * e->nspecies);
   HIPCHK(hipMemcpy(e->d_spec_dyn.p, sd.data(), sizeof(SpecDyn) * sd.size(), hipMemcpyHostToDevice));
   e->d_mom.reserve(3 * (size_t)e->nmols + 3);
   e->d_amom.reserve(4 * (size_t)std::max(e->nmols_r, 1));
   e->d_scal.reserve(SCAL_SIZE);
   const int nb = (e->nmols + 255) / 256;
   e->d_red.reserve((size_t)nb * 6 * MAX_SPEC + 64);
   e->have_dyn = true;
   e->geom_version++;   // captured steps hold the integrator's arguments
}

void mgpu::md_set_scalars(mgpu_engine *e, const double thermo[3]) {
   double v[SCAL_SIZE] = {0};
   v[S_TS] = thermo[0];
   v[S_TSMOM] = thermo[1];
   v[S_H0] = thermo[2];
   for (int i = 0; i < 9; i++) {
      v[S_H + i] = e->h[i];
      v[S_HMOM + i] = e->hmom[i];
   }
   const double *src[1] = {v};
   double *dst[1] = {e->d_scal.p};
   const size_t n[1] = {SCAL_SIZE};
   upload_pinned(e, PIN_SCAL, 1, src, dst, n);
   memcpy(e->cell_loaded, v + S_H, sizeof e->cell_loaded);
   e->cell_valid = true;
}

// The host's h and hmom into the device slots (start of a run), unless the
// slots already hold them.
void mgpu::md_load_cell(mgpu_engine *e) {
   double v[18];
   for (int i = 0; i < 9; i++) {
      v[i] = e->h[i];
      v[9 + i] = e->hmom[i];
   }
   if (e->cell_valid && memcmp(v, e->cell_loaded, sizeof v) == 0) return;
   HIPCHK(hipMemcpyAsync(e->d_scal.p + S_H, v, sizeof v, hipMemcpyHostToDevice, e->stream));
   HIPCHK(hipStreamSynchronize(e->stream));
   memcpy(e->cell_loaded, v, sizeof v);
   e->cell_valid = true;
}

void mgpu::md_fetch_cell(mgpu_engine *e, double h[9], double hmom[9]) {
   double v[18];
   HIPCHK(hipMemcpyAsync(v, e->d_scal.p + S_H, sizeof v, hipMemcpyDeviceToHost, e->stream));
   HIPCHK(hipStreamSynchronize(e->stream));
   for (int i = 0; i < 9; i++) {
      if (h) h[i] = v[i];
      if (hmom) hmom[i] = v[9 + i];
   }
}

void mgpu::md_thermo(const double v[4], double thermo[3]) {
   thermo[0] = v[S_TS];
   thermo[1] = v[S_TSMOM];
   thermo[2] = v[S_H0];
}

void mgpu::md_reset_record(mgpu_engine *e, int cap, bool init_h0) {
   e->d_trace.reserve((size_t)std::max(cap, 1) * TRACE_W);
   e->trace_cap = (int)(e->d_trace.n / TRACE_W);   // what a captured step may fill in a longer call
   ScalArgs a = scal_args(e, OP_RESET_ROW);
   a.init_h0 = init_h0;
   scalar_op(e, a);
}

// do_step, src/accel.c:626-827, at constant h, enqueued on e->stream with
// no host synchronisation.
void mgpu::md_step_launch(mgpu_engine *e) {
   const bool therm = e->dyn_const_temp;
   if (therm) {
      scalar_op(e, scal_args(e, OP_THERM_IN));
      ke_scalar(e, scal_args(e, OP_TSMOM_TRANS));
   }
   coords_half(e);
   eval_forces_device(e, false);
   momenta_record(e);
   if (!therm) {
      momenta_coords(e);
      return;
   }
   momenta_half(e);
   scalar_op(e, scal_args(e, OP_TSMOM_PE));
   ke_scalar(e, scal_args(e, OP_TSMOM_TRANS));
   coords_half(e);
   scalar_op(e, scal_args(e, OP_THERM_OUT));
}

// do_step with the barostat (const_pressure branches of src/accel.c:686-779).
// The cell half step runs on the device; the host then reads h, rebuilds the
// link cells and the k-vector set for it and enqueues the rest of the step.
void mgpu::md_step_pressure(mgpu_engine *e) {
   const bool therm = e->dyn_const_temp;
   if (therm) scalar_op(e, scal_args(e, OP_THERM_IN));
   scalar_op(e, scal_args(e, OP_GLEAP_CELL));
   double h[9];
   md_fetch_cell(e, h, nullptr);
   set_geometry(e, h);
   if (therm) {
      ke_scalar(e, scal_args(e, OP_TSMOM_TRANS));
   }
   dyad_sums(e);
   scalar_op(e, scal_args(e, OP_HMOM_KIN));
   coords_half(e);
   eval_forces_device(e, false);
   momenta_record(e);
   momenta_half(e);
   if (therm) scalar_op(e, scal_args(e, OP_TSMOM_PE));
   scalar_op(e, scal_args(e, OP_HMOM_VIR));
   if (therm) {
      ke_scalar(e, scal_args(e, OP_TSMOM_TRANS));
   }
   dyad_sums(e);
   scalar_op(e, scal_args(e, OP_HMOM_KIN));
   coords_half(e);
   scalar_op(e, scal_args(e, OP_GLEAP_CELL));
   if (therm) scalar_op(e, scal_args(e, OP_THERM_OUT));
}

int mgpu::md_trace_width() { return TRACE_W; }
