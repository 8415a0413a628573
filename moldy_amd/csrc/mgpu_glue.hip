// eval_forces glue on the GPU (restates src/accel.c:398-617 around the
// boundary calls): make_sites (src/algorith.c:169-217), the dipole and
// surface-dipole term (accel.c:542-558), mol_force/mol_torque
// (algorith.c:111-163) and the site-to-molecular virial correction
// (accel.c:575-599).  Sums are per-block partials reduced in a fixed order.
#include "mgpu_internal.h"

using namespace mgpu;

namespace {

struct MsArgs {
   double h[9], hinv[9];
   int ns, nsp, mode;   // mode 0: wrap every site; 1: wrap none; 2: wrap framework only
};

// Binning by make_sites (k_bin's work, src/force.c:119-137): the first site
// of each binning entry takes the entry's cell, from the site position it
// has just formed (one-site entries) or its molecule's centre (molecular
// entries), and a slot in the cell's bucket.
struct MsBin {
   const int *site_entry, *entry_isite, *entry_mol;
   int *e_cell, *c_count, *bucket, *flags;
   int on, nx, ny, nz, ncells, cap;
   double eps;
};

#pragma clang fp contract(off)
__device__ __forceinline__ void b_make_sites(int bx, int nbx, const MsArgs &a, const int *__restrict__ site_mol,
                                             const int *__restrict__ mol_first, const int *__restrict__ mol_spec,
                                             const int *__restrict__ mol_quat, const int *__restrict__ spec_off,
                                             const int *__restrict__ spec_fw, const double *__restrict__ pf,
                                             const double *__restrict__ cm, const double *__restrict__ quat,
                                             double *__restrict__ site, double *__restrict__ zero_f, const MsBin &b) {
   int i = bx * blockDim.x + threadIdx.x;
   if (i >= a.ns) return;
   if (zero_f) {   // the evaluation's site forces start at zero
      zero_f[i] = 0.0;
      zero_f[a.nsp + i] = 0.0;
      zero_f[2 * a.nsp + i] = 0.0;
   }
   int m = site_mol[i], sp = mol_spec[m], iq = mol_quat[m];
   const double *p = pf + 3 * (spec_off[sp] + (i - mol_first[m]));
   const double *c = cm + 3 * m;
   // centre of mass: mat_vec_mul(h, c_of_m_s)
   double c0 = a.h[0] * c[0] + a.h[1] * c[1] + a.h[2] * c[2];
   double c1 = a.h[3] * c[0] + a.h[4] * c[1] + a.h[5] * c[2];
   double c2 = a.h[6] * c[0] + a.h[7] * c[1] + a.h[8] * c[2];
   double x, y, z;
   if (iq >= 0) {
      // q_to_rot, src/quaterns.c:129-154, then mat_vec_mul
      const double *qq = quat + 4 * iq;
      double q0 = qq[0], q1 = qq[1], q2 = qq[2], q3 = qq[3];
      double a01 = 2.0 * q0 * q1, a02 = 2.0 * q0 * q2, a03 = 2.0 * q0 * q3;
      double a12 = 2.0 * q1 * q2, a13 = 2.0 * q1 * q3, a23 = 2.0 * q2 * q3;
      double r01 = a12 - a03, r02 = a13 + a02, r10 = a12 + a03, r12 = a23 - a01;
      double r20 = a13 - a02, r21 = a23 + a01;
      q0 = q0 * q0; q1 = q1 * q1; q2 = q2 * q2; q3 = q3 * q3;
      double r00 = q0 + q1 - q2 - q3, r11 = q0 - q1 + q2 - q3, r22 = q0 - q1 - q2 + q3;
      double s0 = r00 * p[0] + r01 * p[1] + r02 * p[2];
      double s1 = r10 * p[0] + r11 * p[1] + r12 * p[2];
      double s2 = r20 * p[0] + r21 * p[1] + r22 * p[2];
      x = s0 + c0; y = s1 + c1; z = s2 + c2;
   } else {
      x = p[0] + c0; y = p[1] + c1; z = p[2] + c2;
   }
   bool wrap = a.mode == 0 || (a.mode == 2 && spec_fw[sp]);
   if (wrap) {
      double tx = floor(a.hinv[0] * x + a.hinv[1] * y + a.hinv[2] * z + 0.5);
      double ty = floor(a.hinv[3] * x + a.hinv[4] * y + a.hinv[5] * z + 0.5);
      double tz = floor(a.hinv[6] * x + a.hinv[7] * y + a.hinv[8] * z + 0.5);
      x -= a.h[0] * tx + a.h[1] * ty + a.h[2] * tz;
      y -= a.h[3] * tx + a.h[4] * ty + a.h[5] * tz;
      z -= a.h[6] * tx + a.h[7] * ty + a.h[8] * tz;
   }
   site[i] = x;
   site[a.nsp + i] = y;
   site[2 * a.nsp + i] = z;
   if (b.on) {
      const int en = b.site_entry[i];
      if (b.entry_isite[en] == i) {
         double s0, s1, s2;
         if (b.entry_mol[en] < 0) {
            // mat_vec_mul, src/matrix.c:81-83 (left-to-right, no contraction)
            s0 = a.hinv[0] * x + a.hinv[1] * y + a.hinv[2] * z;
            s1 = a.hinv[3] * x + a.hinv[4] * y + a.hinv[5] * z;
            s2 = a.hinv[6] * x + a.hinv[7] * y + a.hinv[8] * z;
         } else {
            s0 = c[0];
            s1 = c[1];
            s2 = c[2];
         }
         int flag = 0;
         const int cell = cellbin_dev(s2, b.nz, (double)b.nz, b.eps, &flag) +
                          b.nz * (cellbin_dev(s1, b.ny, (double)b.ny, b.eps, &flag) +
                                  b.ny * cellbin_dev(s0, b.nx, (double)b.nx, b.eps, &flag));
         if (flag) atomicOr(b.flags, flag);
         b.e_cell[en] = cell;
         const int slot = atomicAdd(&b.c_count[cell], 1);
         if (slot < b.cap) b.bucket[(size_t)slot * b.ncells + cell] = en;
      }
   }
}
__global__ void k_make_sites(MsArgs a, const int *__restrict__ site_mol, const int *__restrict__ mol_first,
                             const int *__restrict__ mol_spec, const int *__restrict__ mol_quat,
                             const int *__restrict__ spec_off, const int *__restrict__ spec_fw,
                             const double *__restrict__ pf, const double *__restrict__ cm,
                             const double *__restrict__ quat, double *__restrict__ site, double *__restrict__ zero_f,
                             MsBin b) {
   b_make_sites(blockIdx.x, gridDim.x, a, site_mol, mol_first, mol_spec, mol_quat, spec_off, spec_fw, pf, cm, quat,
                site, zero_f, b);
}
#pragma clang fp contract(on)

// Block partial sums of NV per-item values, to row `row` of out.
template <int NV>
__device__ void block_partial(double (&v)[NV], double *out, int row) {
   __shared__ double ws[4][NV];
   int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
   for (int q = 0; q < NV; q++) {
      double t = wave_sum(v[q]);
      if (lane == 0) ws[w][q] = t;
   }
   __syncthreads();
   if (threadIdx.x < NV)
      out[(size_t)row * NV + threadIdx.x] =
          ws[0][threadIdx.x] + ws[1][threadIdx.x] + ws[2][threadIdx.x] + ws[3][threadIdx.x];
}

__device__ __forceinline__ void b_dipole(int bx, int nbx, int ns, int nsp, const double *__restrict__ site,
                                         const double *__restrict__ chg, double *__restrict__ part) {
   int i = bx * 256 + threadIdx.x;
   double v[3] = {0, 0, 0};
   if (i < ns) {
      double q = chg[i];
      v[0] = site[i] * q; v[1] = site[nsp + i] * q; v[2] = site[2 * nsp + i] * q;
   }
   block_partial<3>(v, part, bx);
}
__global__ __launch_bounds__(256) void k_dipole(int ns, int nsp, const double *__restrict__ site,
                                                const double *__restrict__ chg, double *__restrict__ part) {
   b_dipole(blockIdx.x, gridDim.x, ns, nsp, site, chg, part);
}

// Surface-dipole force, src/accel.c:545-552: f_i -= 4 pi / (3V) q_i M.
__device__ __forceinline__ void b_surface(int bx, int nbx, int ns, int nsp, double c, const double *__restrict__ dip,
                                          const double *__restrict__ chg, double *__restrict__ f) {
   int i = bx * 256 + threadIdx.x;
   if (i >= ns) return;
   double q = chg[i];
   f[i] -= c * dip[0] * q;
   f[nsp + i] -= c * dip[1] * q;
   f[2 * nsp + i] -= c * dip[2] * q;
}
__global__ void k_surface(int ns, int nsp, double c, const double *__restrict__ dip, const double *__restrict__ chg,
                          double *__restrict__ f) {
   b_surface(blockIdx.x, gridDim.x, ns, nsp, c, dip, chg, f);
}

struct AsmArgs {
   double vol, pe_real_shift, dist_vol, distp_vol, self_energy, sheet_vol;
   int recip, surface;
};

// Energies, dipole and stress of eval_forces from the reduced sums
// (src/accel.c:526-606), one thread.
__device__ void assemble(const AsmArgs &a, double *__restrict__ out) {
   const double PI_D = 3.14159265358979323846;
   double pe0 = out[OUT_REAL] + a.pe_real_shift;
   double pe1 = 0.0, dip[3] = {0, 0, 0}, st_r[6] = {0, 0, 0, 0, 0, 0};
   if (a.recip) {
      pe1 += out[OUT_RECIP] - a.self_energy + a.sheet_vol;
      for (int q = 0; q < 6; q++) st_r[q] = out[OUT_RECIP + 1 + q];
      st_r[0] += a.sheet_vol;
      st_r[3] += a.sheet_vol;
      st_r[5] += a.sheet_vol;
      for (int c = 0; c < 3; c++) dip[c] = out[OUT_DIP + c];
      if (a.surface) pe1 += 2.0 * PI_D / (3.0 * a.vol) * (dip[0] * dip[0] + dip[1] * dip[1] + dip[2] * dip[2]);
   }
   double st[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
   const int up[6][2] = {{0, 0}, {0, 1}, {0, 2}, {1, 1}, {1, 2}, {2, 2}};
   for (int q = 0; q < 6; q++) st[3 * up[q][0] + up[q][1]] = out[OUT_REAL + 1 + q] + st_r[q];
   const double *corr = out + OUT_CORR;
   for (int i = 0; i < 3; i++) {
      for (int j = i + 1; j < 3; j++) st[3 * j + i] = st[3 * i + j];
      for (int j = 0; j < 3; j++) st[3 * i + j] -= corr[3 * i + j] - corr[9 + 3 * i + j];
   }
   for (int i = 0; i < 3; i++) st[4 * i] += a.distp_vol;
   double *r = out + OUT_RES;
   r[0] = pe0 + a.dist_vol;
   r[1] = pe1;
   for (int c = 0; c < 3; c++) r[2 + c] = dip[c];
   for (int q = 0; q < 9; q++) r[5 + q] = st[q];
}

__device__ __forceinline__ void b_assemble(int bx, int nbx, const AsmArgs &a, double *__restrict__ out) {
   if (threadIdx.x == 0 && bx == 0) assemble(a, out);
}
__global__ void k_assemble(AsmArgs a, double *__restrict__ out) {
   b_assemble(blockIdx.x, gridDim.x, a, out);
}

struct MfArgs {
   int nmols, nsp;
};

// mol_force and mol_torque for one molecule per thread.
__device__ __forceinline__ void b_mol_ft(int bx, int nbx, const MfArgs &a, const int *__restrict__ mol_first,
                                         const int *__restrict__ mol_spec, const int *__restrict__ mol_quat,
                                         const int *__restrict__ spec_off, const int *__restrict__ spec_ns,
                                         const double *__restrict__ pf, const double *__restrict__ quat,
                                         const double *__restrict__ f, double *__restrict__ mforce,
                                         double *__restrict__ mtorque) {
   int m = bx * blockDim.x + threadIdx.x;
   if (m >= a.nmols) return;
   int sp = mol_spec[m], i0 = mol_first[m], n = spec_ns[sp], iq = mol_quat[m];
   double F0 = 0, F1 = 0, F2 = 0;
   for (int s = 0; s < n; s++) F0 += f[i0 + s];
   for (int s = 0; s < n; s++) F1 += f[a.nsp + i0 + s];
   for (int s = 0; s < n; s++) F2 += f[2 * a.nsp + i0 + s];
   mforce[3 * m] = F0; mforce[3 * m + 1] = F1; mforce[3 * m + 2] = F2;
   if (iq < 0) return;
   const double *qq = quat + 4 * iq;
   double q0 = qq[0], q1 = qq[1], q2 = qq[2], q3 = qq[3];
   double a01 = 2.0 * q0 * q1, a02 = 2.0 * q0 * q2, a03 = 2.0 * q0 * q3;
   double a12 = 2.0 * q1 * q2, a13 = 2.0 * q1 * q3, a23 = 2.0 * q2 * q3;
   double r[9];
   r[1] = a12 - a03; r[2] = a13 + a02; r[3] = a12 + a03; r[5] = a23 - a01; r[6] = a13 - a02;
   r[7] = a23 + a01;
   q0 = q0 * q0; q1 = q1 * q1; q2 = q2 * q2; q3 = q3 * q3;
   r[0] = q0 + q1 - q2 - q3; r[4] = q0 - q1 + q2 - q3; r[8] = q0 - q1 - q2 + q3;
   const double *p = pf + 3 * spec_off[sp];
   double t[3] = {0, 0, 0};
   for (int s = 0; s < n; s++) {
      double fs0 = f[i0 + s], fs1 = f[a.nsp + i0 + s], fs2 = f[2 * a.nsp + i0 + s];
      double pf0 = r[0] * fs0 + r[3] * fs1 + r[6] * fs2;   // inverse rotation
      double pf1 = r[1] * fs0 + r[4] * fs1 + r[7] * fs2;
      double pf2 = r[2] * fs0 + r[5] * fs1 + r[8] * fs2;
      const double *ps = p + 3 * s;
      t[0] += ps[1] * pf2 - ps[2] * pf1;
      t[1] += ps[2] * pf0 - ps[0] * pf2;
      t[2] += ps[0] * pf1 - ps[1] * pf0;
   }
   mtorque[3 * iq] = t[0]; mtorque[3 * iq + 1] = t[1]; mtorque[3 * iq + 2] = t[2];
}
__global__ void k_mol_ft(MfArgs a, const int *__restrict__ mol_first, const int *__restrict__ mol_spec,
                         const int *__restrict__ mol_quat, const int *__restrict__ spec_off,
                         const int *__restrict__ spec_ns, const double *__restrict__ pf,
                         const double *__restrict__ quat, const double *__restrict__ f, double *__restrict__ mforce,
                         double *__restrict__ mtorque) {
   b_mol_ft(blockIdx.x, gridDim.x, a, mol_first, mol_spec, mol_quat, spec_off, spec_ns, pf, quat, f, mforce, mtorque);
}

// Per-site terms of the virial correction: non-framework sites contribute
// f_i s_j, framework sites f_i p_j (principal-frame coordinates).
__device__ __forceinline__ void b_vir_sites(int bx, int nbx, int ns, int nsp, int nsxf,
                                            const int *__restrict__ site_mol, const int *__restrict__ mol_first,
                                            const int *__restrict__ mol_spec, const int *__restrict__ spec_off,
                                            const double *__restrict__ pf, const double *__restrict__ site,
                                            const double *__restrict__ f, double *__restrict__ part) {
   int i = bx * 256 + threadIdx.x;
   double v[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
   if (i < ns) {
      double fa[3] = {f[i], f[nsp + i], f[2 * nsp + i]};
      double sa[3];
      if (i < nsxf) {
         sa[0] = site[i]; sa[1] = site[nsp + i]; sa[2] = site[2 * nsp + i];
      } else {
         int m = site_mol[i];
         const double *p = pf + 3 * (spec_off[mol_spec[m]] + (i - mol_first[m]));
         sa[0] = p[0]; sa[1] = p[1]; sa[2] = p[2];
      }
#pragma unroll
      for (int a = 0; a < 3; a++)
#pragma unroll
         for (int b = 0; b < 3; b++) v[3 * a + b] = fa[a] * sa[b];
   }
   block_partial<9>(v, part, bx);
}
__global__ __launch_bounds__(256) void k_vir_sites(int ns, int nsp, int nsxf, const int *__restrict__ site_mol,
                                                   const int *__restrict__ mol_first,
                                                   const int *__restrict__ mol_spec, const int *__restrict__ spec_off,
                                                   const double *__restrict__ pf, const double *__restrict__ site,
                                                   const double *__restrict__ f, double *__restrict__ part) {
   b_vir_sites(blockIdx.x, gridDim.x, ns, nsp, nsxf, site_mol, mol_first, mol_spec, spec_off, pf, site, f, part);
}

// Molecular terms: F_i R_j over non-framework molecules, R = h c_of_m.
__device__ __forceinline__ void b_vir_mols(int bx, int nbx, int nmolsxf, double h0, double h1, double h2, double h3,
                                           double h4, double h5, double h6, double h7, double h8,
                                           const double *__restrict__ cm, const double *__restrict__ mforce,
                                           double *__restrict__ part) {
   int m = bx * 256 + threadIdx.x;
   double v[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
   if (m < nmolsxf) {
      const double *c = cm + 3 * m;
      double R[3] = {h0 * c[0] + h1 * c[1] + h2 * c[2], h3 * c[0] + h4 * c[1] + h5 * c[2],
                     h6 * c[0] + h7 * c[1] + h8 * c[2]};
      const double *F = mforce + 3 * m;
#pragma unroll
      for (int a = 0; a < 3; a++)
#pragma unroll
         for (int b = 0; b < 3; b++) v[3 * a + b] = F[a] * R[b];
   }
   block_partial<9>(v, part, bx);
}
__global__ __launch_bounds__(256) void k_vir_mols(int nmolsxf, double h0, double h1, double h2, double h3, double h4,
                                                  double h5, double h6, double h7, double h8,
                                                  const double *__restrict__ cm, const double *__restrict__ mforce,
                                                  double *__restrict__ part) {
   b_vir_mols(blockIdx.x, gridDim.x, nmolsxf, h0, h1, h2, h3, h4, h5, h6, h7, h8, cm, mforce, part);
}


// The glue without the surface-dipole term in two launches.  k_glue_parts:
// blocks 0 .. nb-1 take sites (the second make_sites in registers, its
// sites stored, and per block the dipole sums q r and the site virial terms
// f s, or f p for framework sites); blocks nb .. nb+nmb-1 take molecules
// (mol_force, mol_torque and per block the molecular virial terms F R).
// k_glue_sum adds each column's block partials in a fixed order and
// assembles the results (the work of k_assemble).
constexpr int GLUE_S = 12;   // site partial columns: dipole (3), site virial (9)
constexpr int GLUE_M = 9;    // molecule partial columns: molecular virial

struct GlueArgs {
   MsArgs ms;
   MfArgs mf;
   int nb, nsxf, nmolsxf;
};

#pragma clang fp contract(off)
__device__ __forceinline__ void site_pos2(const MsArgs &a, int i, int m, int sp, int iq, const double *p,
                                          const double *__restrict__ cm, const double *__restrict__ quat,
                                          bool fw, double &x, double &y, double &z) {
   // k_make_sites with mode 2 (wrap framework sites only), same operations
   const double *c = cm + 3 * m;
   double c0 = a.h[0] * c[0] + a.h[1] * c[1] + a.h[2] * c[2];
   double c1 = a.h[3] * c[0] + a.h[4] * c[1] + a.h[5] * c[2];
   double c2 = a.h[6] * c[0] + a.h[7] * c[1] + a.h[8] * c[2];
   if (iq >= 0) {
      const double *qq = quat + 4 * iq;
      double q0 = qq[0], q1 = qq[1], q2 = qq[2], q3 = qq[3];
      double a01 = 2.0 * q0 * q1, a02 = 2.0 * q0 * q2, a03 = 2.0 * q0 * q3;
      double a12 = 2.0 * q1 * q2, a13 = 2.0 * q1 * q3, a23 = 2.0 * q2 * q3;
      double r01 = a12 - a03, r02 = a13 + a02, r10 = a12 + a03, r12 = a23 - a01;
      double r20 = a13 - a02, r21 = a23 + a01;
      q0 = q0 * q0; q1 = q1 * q1; q2 = q2 * q2; q3 = q3 * q3;
      double r00 = q0 + q1 - q2 - q3, r11 = q0 - q1 + q2 - q3, r22 = q0 - q1 - q2 + q3;
      double s0 = r00 * p[0] + r01 * p[1] + r02 * p[2];
      double s1 = r10 * p[0] + r11 * p[1] + r12 * p[2];
      double s2 = r20 * p[0] + r21 * p[1] + r22 * p[2];
      x = s0 + c0; y = s1 + c1; z = s2 + c2;
   } else {
      x = p[0] + c0; y = p[1] + c1; z = p[2] + c2;
   }
   if (fw) {
      double tx = floor(a.hinv[0] * x + a.hinv[1] * y + a.hinv[2] * z + 0.5);
      double ty = floor(a.hinv[3] * x + a.hinv[4] * y + a.hinv[5] * z + 0.5);
      double tz = floor(a.hinv[6] * x + a.hinv[7] * y + a.hinv[8] * z + 0.5);
      x -= a.h[0] * tx + a.h[1] * ty + a.h[2] * tz;
      y -= a.h[3] * tx + a.h[4] * ty + a.h[5] * tz;
      z -= a.h[6] * tx + a.h[7] * ty + a.h[8] * tz;
   }
}
#pragma clang fp contract(on)

__device__ __forceinline__ void b_glue_parts(int bx, int nbx, const GlueArgs &g, const int *__restrict__ site_mol,
                                             const int *__restrict__ mol_first, const int *__restrict__ mol_spec,
                                             const int *__restrict__ mol_quat, const int *__restrict__ spec_off,
                                             const int *__restrict__ spec_ns, const int *__restrict__ spec_fw,
                                             const double *__restrict__ pf, const double *__restrict__ cm,
                                             const double *__restrict__ quat, const double *__restrict__ chg,
                                             const double *__restrict__ f, double *__restrict__ site,
                                             double *__restrict__ mforce, double *__restrict__ mtorque,
                                             double *__restrict__ part_s, double *__restrict__ part_m) {
   const int nsp = g.ms.nsp;
   if ((int)bx < g.nb) {   // block-uniform role
      const int i = bx * 256 + threadIdx.x;
      double v[GLUE_S];
#pragma unroll
      for (int q = 0; q < GLUE_S; q++) v[q] = 0.0;
      if (i < g.ms.ns) {
         const int m = site_mol[i], sp = mol_spec[m], iq = mol_quat[m];
         const double *p = pf + 3 * (spec_off[sp] + (i - mol_first[m]));
         double x, y, z;
         site_pos2(g.ms, i, m, sp, iq, p, cm, quat, spec_fw[sp] != 0, x, y, z);
         site[i] = x;
         site[nsp + i] = y;
         site[2 * nsp + i] = z;
         const double q = chg[i];
         v[0] = x * q; v[1] = y * q; v[2] = z * q;
         const double fa[3] = {f[i], f[nsp + i], f[2 * nsp + i]};
         const double sa[3] = {i < g.nsxf ? x : p[0], i < g.nsxf ? y : p[1], i < g.nsxf ? z : p[2]};
#pragma unroll
         for (int a = 0; a < 3; a++)
#pragma unroll
            for (int b = 0; b < 3; b++) v[3 + 3 * a + b] = fa[a] * sa[b];
      }
      block_partial<GLUE_S>(v, part_s, bx);
   } else {
      const int mb = bx - g.nb, m = mb * 256 + threadIdx.x;
      double v[GLUE_M];
#pragma unroll
      for (int q = 0; q < GLUE_M; q++) v[q] = 0.0;
      if (m < g.mf.nmols) {
         // mol_force, mol_torque: as k_mol_ft
         int sp = mol_spec[m], i0 = mol_first[m], n = spec_ns[sp], iq = mol_quat[m];
         double F0 = 0, F1 = 0, F2 = 0;
         for (int s = 0; s < n; s++) F0 += f[i0 + s];
         for (int s = 0; s < n; s++) F1 += f[nsp + i0 + s];
         for (int s = 0; s < n; s++) F2 += f[2 * nsp + i0 + s];
         mforce[3 * m] = F0; mforce[3 * m + 1] = F1; mforce[3 * m + 2] = F2;
         if (iq >= 0) {
            const double *qq = quat + 4 * iq;
            double q0 = qq[0], q1 = qq[1], q2 = qq[2], q3 = qq[3];
            double a01 = 2.0 * q0 * q1, a02 = 2.0 * q0 * q2, a03 = 2.0 * q0 * q3;
            double a12 = 2.0 * q1 * q2, a13 = 2.0 * q1 * q3, a23 = 2.0 * q2 * q3;
            double r[9];
            r[1] = a12 - a03; r[2] = a13 + a02; r[3] = a12 + a03; r[5] = a23 - a01; r[6] = a13 - a02;
            r[7] = a23 + a01;
            q0 = q0 * q0; q1 = q1 * q1; q2 = q2 * q2; q3 = q3 * q3;
            r[0] = q0 + q1 - q2 - q3; r[4] = q0 - q1 + q2 - q3; r[8] = q0 - q1 - q2 + q3;
            const double *p = pf + 3 * spec_off[sp];
            double t[3] = {0, 0, 0};
            for (int s = 0; s < n; s++) {
               double fs0 = f[i0 + s], fs1 = f[nsp + i0 + s], fs2 = f[2 * nsp + i0 + s];
               double pf0 = r[0] * fs0 + r[3] * fs1 + r[6] * fs2;   // inverse rotation
               double pf1 = r[1] * fs0 + r[4] * fs1 + r[7] * fs2;
               double pf2 = r[2] * fs0 + r[5] * fs1 + r[8] * fs2;
               const double *ps = p + 3 * s;
               t[0] += ps[1] * pf2 - ps[2] * pf1;
               t[1] += ps[2] * pf0 - ps[0] * pf2;
               t[2] += ps[0] * pf1 - ps[1] * pf0;
            }
            mtorque[3 * iq] = t[0]; mtorque[3 * iq + 1] = t[1]; mtorque[3 * iq + 2] = t[2];
         }
         if (m < g.nmolsxf) {
            // F R over non-framework molecules, R = h c_of_m (as k_vir_mols)
            const double *c = cm + 3 * m;
            const double *h = g.ms.h;
            const double R[3] = {h[0] * c[0] + h[1] * c[1] + h[2] * c[2], h[3] * c[0] + h[4] * c[1] + h[5] * c[2],
                                 h[6] * c[0] + h[7] * c[1] + h[8] * c[2]};
            const double F[3] = {F0, F1, F2};
#pragma unroll
            for (int a = 0; a < 3; a++)
#pragma unroll
               for (int b = 0; b < 3; b++) v[3 * a + b] = F[a] * R[b];
         }
      }
      block_partial<GLUE_M>(v, part_m, mb);
   }
}
__global__ __launch_bounds__(256) void k_glue_parts(GlueArgs g, const int *__restrict__ site_mol,
                                                    const int *__restrict__ mol_first,
                                                    const int *__restrict__ mol_spec,
                                                    const int *__restrict__ mol_quat,
                                                    const int *__restrict__ spec_off, const int *__restrict__ spec_ns,
                                                    const int *__restrict__ spec_fw, const double *__restrict__ pf,
                                                    const double *__restrict__ cm, const double *__restrict__ quat,
                                                    const double *__restrict__ chg, const double *__restrict__ f,
                                                    double *__restrict__ site, double *__restrict__ mforce,
                                                    double *__restrict__ mtorque, double *__restrict__ part_s,
                                                    double *__restrict__ part_m) {
   b_glue_parts(blockIdx.x, gridDim.x, g, site_mol, mol_first, mol_spec, mol_quat, spec_off, spec_ns, spec_fw, pf, cm,
                quat, chg, f, site, mforce, mtorque, part_s, part_m);
}

// One block: each of the 21 columns is summed by 48 threads over the rows
// q, q + 48, ... in order, then those 48 sums in order; thread 0 assembles.
// With rpart set, also the reciprocal pass's 8 sums (OUT_RECIP) from its
// rrows rows of per-block partials: 128 threads a column add every 128th
// row in order, then those 128 sums in order (before the assembly reads them);
// with qpart set, the real-space pass's (OUT_REAL) likewise.
__device__ __forceinline__ void b_glue_sum(int bx, int nbx, const AsmArgs &a, int nb, int nmb,
                                           const double *__restrict__ part_s, const double *__restrict__ part_m,
                                           const double *__restrict__ rpart, int rrows,
                                           const double *__restrict__ qpart, int qrows, double *__restrict__ out) {
   constexpr int NC = GLUE_S + GLUE_M, NT = 48, RT = 128;
   __shared__ double sp[NC][NT];
   __shared__ double col[NC];
   __shared__ double rp[8][RT], qp[8][RT];
   const int t = threadIdx.x;
   if (rpart) {
      const int c = t / RT, q = t - c * RT;
      double acc = 0.0;
      for (int r = q; r < rrows; r += RT) acc += rpart[(size_t)r * 8 + c];
      rp[c][q] = acc;
   }
   if (qpart) {
      const int c = t / RT, q = t - c * RT;
      double acc = 0.0;
      for (int r = q; r < qrows; r += RT) acc += qpart[(size_t)r * 8 + c];
      qp[c][q] = acc;
   }
   if (t < NC * NT) {
      const int c = t / NT, q = t - c * NT;
      double acc = 0.0;
      if (c < GLUE_S)
         for (int r = q; r < nb; r += NT) acc += part_s[(size_t)r * GLUE_S + c];
      else
         for (int r = q; r < nmb; r += NT) acc += part_m[(size_t)r * GLUE_M + (c - GLUE_S)];
      sp[c][q] = acc;
   }
   __syncthreads();
   if (t < NC) {
      double acc = 0.0;
      for (int q = 0; q < NT; q++) acc += sp[t][q];
      col[t] = acc;
   } else if (rpart && t >= 32 && t < 40) {
      double acc = 0.0;
      for (int q = 0; q < RT; q++) acc += rp[t - 32][q];
      out[OUT_RECIP + (t - 32)] = acc;
   } else if (qpart && t >= 64 && t < 72) {
      double acc = 0.0;
      for (int q = 0; q < RT; q++) acc += qp[t - 64][q];
      out[OUT_REAL + (t - 64)] = acc;
   }
   __syncthreads();
   if (t == 0) {
      for (int c = 0; c < 3; c++) out[OUT_DIP + c] = col[c];
      for (int c = 0; c < 9; c++) out[OUT_CORR + c] = col[3 + c];
      for (int c = 0; c < 9; c++) out[OUT_CORR + 9 + c] = col[GLUE_S + c];
      assemble(a, out);
   }
}
__global__ __launch_bounds__(1024) void k_glue_sum(AsmArgs a, int nb, int nmb, const double *__restrict__ part_s,
                                                   const double *__restrict__ part_m, const double *__restrict__ rpart,
                                                   int rrows, const double *__restrict__ qpart, int qrows,
                                                   double *__restrict__ out) {
   b_glue_sum(blockIdx.x, gridDim.x, a, nb, nmb, part_s, part_m, rpart, rrows, qpart, qrows, out);
}

}  // namespace

void mgpu::launch_make_sites(mgpu_engine *e, int mode, bool zero_forces, bool bin) {
   MsArgs a;
   for (int i = 0; i < 9; i++) { a.h[i] = e->h[i]; a.hinv[i] = e->hinv[i]; }
   a.ns = e->nsites; a.nsp = e->nsp; a.mode = mode;
   MsBin b{};
   if (bin) {
      prepare_binning(e);
      b.site_entry = e->d_site_entry.p; b.entry_isite = e->d_entry_isite.p; b.entry_mol = e->d_entry_mol.p;
      b.e_cell = e->d_entry_cell.p; b.c_count = e->d_cell_count.p; b.bucket = e->d_cell_bucket.p;
      b.flags = e->d_iflags.p;
      b.on = 1; b.nx = e->nx; b.ny = e->ny; b.nz = e->nz; b.ncells = e->ncells; b.cap = e->bin_cap;
      b.eps = 8.0 * 2.220446049250313e-16;   // 8 * precision(), src/force.c:437
   }
   ProfScope ps(e, "make_sites");
   glaunch<k_make_sites, b_make_sites, 1024>(e->rec, e->stream, (e->nsites + 255) / 256, 256, 0, a, e->d_site_mol.p,
                                             e->d_mol_first.p, e->d_mol_spec.p, e->d_mol_quat.p, e->d_spec_off.p,
                                             e->d_spec_fw.p, e->d_pf.p, e->d_cm.p, e->d_quat.p, e->d_site.p,
                                             zero_forces ? e->d_force_site.p : nullptr, b);
}

// Everything of eval_forces after the two boundary calls, on the device.
void mgpu::run_glue(mgpu_engine *e) {
   ProfScope ps(e, "glue");
   const int ns = e->nsites, nsp = e->nsp;
   const int nb = (ns + 255) / 256, nmb = (e->nmols + 255) / 256;
   const double PI_D = 3.14159265358979323846;
   double vol = host_det(e->h);
   e->d_red.reserve((size_t)(nb + nmb) * 9 + 64);
   e->d_out.reserve(OUT_SIZE);
   double *out = e->d_out.p;
   const bool recip = e->alpha > 1e-7;
   AsmArgs aa;
   aa.vol = vol;
   aa.pe_real_shift = (e->precision == MGPU_MIXED && e->intra_exact) ? 0.0 : -e->eintra;
   aa.dist_vol = e->dist / vol;
   aa.distp_vol = e->distp / vol;
   aa.self_energy = e->self_energy;
   aa.sheet_vol = e->sheet_energy / vol;
   aa.recip = recip;
   aa.surface = e->surface_dipole;
   if (!e->surface_dipole) {
      // two launches: the per-site and per-molecule terms, then the sums
      GlueArgs g;
      for (int i = 0; i < 9; i++) { g.ms.h[i] = e->h[i]; g.ms.hinv[i] = e->hinv[i]; }
      g.ms.ns = ns; g.ms.nsp = nsp; g.ms.mode = 2;
      g.mf.nmols = e->nmols; g.mf.nsp = nsp;
      g.nb = nb; g.nsxf = e->nsitesxf; g.nmolsxf = e->nmolsxf;
      const int nmb1 = std::max(nmb, 1);
      e->d_red.reserve((size_t)nb * GLUE_S + (size_t)nmb1 * GLUE_M + 64);
      double *part_s = e->d_red.p, *part_m = e->d_red.p + (size_t)nb * GLUE_S;
      glaunch<k_glue_parts, b_glue_parts, 256>(e->rec, e->stream, nb + nmb1, 256, 0, g, e->d_site_mol.p,
                                               e->d_mol_first.p, e->d_mol_spec.p, e->d_mol_quat.p, e->d_spec_off.p,
                                               e->d_spec_nsites.p, e->d_spec_fw.p, e->d_pf.p, e->d_cm.p, e->d_quat.p,
                                               e->d_chg_site.p, e->d_force_site.p, e->d_site.p, e->d_mforce.p,
                                               e->d_mtorque.p, part_s, part_m);
      glaunch<k_glue_sum, b_glue_sum, 1024>(e->rec, e->stream, 1, 1024, 0, aa, nb, nmb1, part_s, part_m,
                                            e->recip_part, e->recip_rows, e->real_part, e->real_rows, out);
      e->recip_part = e->real_part = nullptr;
      return;
   }
   // second make_sites: MOLPBC for molecules, SITEPBC for frameworks (accel.c:536-541)
   launch_make_sites(e, 2);
   if (recip) {
      glaunch<k_dipole, b_dipole, 256>(e->rec, e->stream, nb, 256, 0, ns, nsp, e->d_site.p, e->d_chg_site.p,
                                       e->d_red.p);
      reduce_cols(e, e->d_red.p, nb, 3, out + OUT_DIP);
      if (e->surface_dipole)
         glaunch<k_surface, b_surface, 1024>(e->rec, e->stream, nb, 256, 0, ns, nsp, 4.0 * PI_D / (3.0 * vol),
                                             out + OUT_DIP, e->d_chg_site.p, e->d_force_site.p);
   }
   MfArgs mf{e->nmols, nsp};
   glaunch<k_mol_ft, b_mol_ft, 1024>(e->rec, e->stream, nmb, 256, 0, mf, e->d_mol_first.p, e->d_mol_spec.p,
                                     e->d_mol_quat.p, e->d_spec_off.p, e->d_spec_nsites.p, e->d_pf.p, e->d_quat.p,
                                     e->d_force_site.p, e->d_mforce.p, e->d_mtorque.p);
   glaunch<k_vir_sites, b_vir_sites, 256>(e->rec, e->stream, nb, 256, 0, ns, nsp, e->nsitesxf, e->d_site_mol.p,
                                          e->d_mol_first.p, e->d_mol_spec.p, e->d_spec_off.p, e->d_pf.p, e->d_site.p,
                                          e->d_force_site.p, e->d_red.p);
   int nmxb = (e->nmolsxf + 255) / 256;
   if (nmxb == 0) nmxb = 1;
   double *mpart = e->d_red.p + (size_t)nb * 9;
   glaunch<k_vir_mols, b_vir_mols, 256>(e->rec, e->stream, nmxb, 256, 0, e->nmolsxf, e->h[0], e->h[1], e->h[2],
                                        e->h[3], e->h[4], e->h[5], e->h[6], e->h[7], e->h[8], e->d_cm.p,
                                        e->d_mforce.p, mpart);
   reduce_cols(e, e->d_red.p, nb, 9, out + OUT_CORR);
   reduce_cols(e, mpart, nmxb, 9, out + OUT_CORR + 9);
   glaunch<k_assemble, b_assemble, 1024>(e->rec, e->stream, 1, 64, 0, aa, out);
}

// Zero fill by a kernel: memset nodes must stay out of captured graphs.
__device__ __forceinline__ void b_zero(int bx, int nbx, uint32_t *__restrict__ p, size_t n4) {
   for (size_t i = bx * (size_t)blockDim.x + threadIdx.x; i < n4; i += (size_t)nbx * blockDim.x)
      p[i] = 0u;
}
__global__ void k_zero(uint32_t *__restrict__ p, size_t n4) {
   b_zero(blockIdx.x, gridDim.x, p, n4);
}

void mgpu::zero_async(mgpu_engine *e, void *p, size_t bytes) {
   if (bytes % 4) throw StatusError{MGPU_E_ARG, "zero_async: size not a multiple of 4"};
   size_t n4 = bytes / 4;
   if (!n4) return;
   int nb = (int)std::min<size_t>(1024, (n4 + 255) / 256);
   // always launched, never recorded: in a force evaluation or MD step it
   // only clears freshly allocated memory, which a grouped step's recording
   // pass allocates (and must clear) once, outside the recorded launches
   k_zero<<<nb, 256, 0, e->stream>>>((uint32_t *)p, n4);
}
