/*
 * moldy_amd.h -- C ABI of the MI355X force engine (libmoldy_amd.so).
 *
 * Plain pointers and sizes only.  All entry points return 0 on success or a
 * MGPU_E* status; mgpu_last_error() gives the message.  Arrays are FP64 in
 * Moldy's program units.  Site arrays are structure-of-arrays [3][ld] (the
 * layout of eval_forces' site/site_force blocks, src/accel.c:422-426); h is
 * the 3x3 cell matrix, row-major, upper triangular (columns a, b, c).
 *
 * The Moldy-signature drop-ins force_calc()/ewald()/poteval() are in
 * moldy_force.h; they are implemented on top of these calls.
 */
#ifndef MOLDY_AMD_H
#define MOLDY_AMD_H

#ifdef __cplusplus
extern "C" {
#endif

typedef struct mgpu_engine mgpu_engine;

enum {
   MGPU_OK = 0,
   MGPU_E_ARG = 1,        /* bad argument                                     */
   MGPU_E_HIP = 2,        /* HIP runtime error                                */
   MGPU_E_BIN_RANGE = 3,  /* "Co-ordinate out of range in BIN", force.c:130   */
   MGPU_E_BIN_ROUND = 4,  /* "Rounding problem in BIN",        force.c:134    */
   MGPU_E_CUTOFF = 5,     /* CUTOFF fatal,                     force.c:206    */
   MGPU_E_TONAB = 6,      /* TONAB fatal,                      force.c:562    */
   MGPU_E_MULTIFW = 7,    /* multiple frameworks,              force.c:1219   */
   MGPU_E_PTYPE = 8,      /* UNKPTY,                           kernel.c:186   */
   MGPU_E_STATE = 9,      /* call order (no system set, ...)                  */
   MGPU_E_CAPACITY = 10,  /* a fixed-capacity limit of this engine exceeded   */
   MGPU_E_QNORM = 11      /* QNORM2 fatal, quaternion norm off by > 1e-4,
                             src/leapfrog.c:104-106                            */
};

enum { MGPU_FP64 = 0, MGPU_MIXED = 1 };

/* System description: the content of system_mt, spec_mt[], site_mt[] charges,
 * pot_mt[] and the contr_mt fields the path reads (src/structs.h:27-161).
 * Species are ordered with frameworks last (src/input.c:95-117). */
typedef struct {
   int nsites, nmols, nspecies, max_id, ptype, n_potpar;
   const int    *spec_nmols;      /* [nspecies]                                */
   const int    *spec_nsites;     /* [nspecies]                                */
   const int    *spec_framework;  /* [nspecies]                                */
   const int    *spec_rdof;       /* [nspecies]                                */
   const int    *spec_site_id;    /* concatenated per-species site ids         */
   const double *spec_p_f_sites;  /* concatenated principal-frame sites [..][3]*/
   const double *site_charge;     /* [max_id] charge per site id               */
   const double *potpar;          /* [max_id*max_id][8], pot_mt.p              */
   double cutoff, subcell, alpha, k_cutoff;
   int strict_cutoff, molpbc, surface_dipole;
} mgpu_system;

/* Diagnostics of one real-space call (the notes/warnings Moldy prints). */
typedef struct {
   int nx, ny, nz, n_nabors;      /* subcells; half-shell offsets (Moldy prints 2x) */
   int n_too_close;               /* TOOCLS pairs, force.c:944                  */
   int too_close_i[16], too_close_j[16];
   long n_list_entries;           /* sum of site-neighbour-list lengths         */
   int max_cell_sites;
   double eintra;                 /* intramolecular correction, force.c:1167    */
} mgpu_fc_info;

typedef struct {
   int hmax, kmax, lmax, nhkl, nsitesxf;
   double self_energy, sheet_energy;
} mgpu_ew_info;

/* ---- lifetime ---- */
int  mgpu_create(mgpu_engine **eng, int device);
void mgpu_destroy(mgpu_engine *eng);
const char *mgpu_last_error(const mgpu_engine *eng);
int  mgpu_set_system(mgpu_engine *eng, const mgpu_system *sys);
int  mgpu_set_precision(mgpu_engine *eng, int precision);
/* Nonzero (the default): the device-resident evaluation runs the real-space
 * pass on a second stream beside the Ewald sum (results bit-identical to the
 * serial order).  No counterpart in the reference, whose force_calc and
 * ewald run one after the other on the CPU. */
int  mgpu_set_overlap(mgpu_engine *eng, int on);

/* Real-space kernel: 0 automatic (the load-balanced kernel from one site a
 * CU), 1 the per-offset walk, 2 the load-balanced kernel (a wave takes sites
 * in turn, each over the shell's z-columns of cells) wherever the shell splits into columns, else the walk; 3 as 2 with
 * the candidates assigned to their column runs in windows of 64 instead of 2048,
 * the path taken by sites with more than 2048 candidates; 4 the tiled
 * Newton-3 kernel (every pair once, as force.c:717-778: one block per
 * z-column of cells, half of the shell's columns staged in LDS, the force on
 * j summed through a partial array in a fixed order) wherever the shell
 * splits into columns, else the walk; it is slower than 2 on MI355X and is
 * never chosen automatically.  All give the reference's pair set; only the
 * summation order differs.
 * mgpu_realspace_balanced reports whether the last real-space pass used one
 * of the column kernels (2, 3 or 4).  No counterpart in the reference. */
#define MGPU_RS_AUTO 0
#define MGPU_RS_WALK 1
#define MGPU_RS_BALANCED 2
#define MGPU_RS_BALANCED_SEARCH 3
#define MGPU_RS_TILED 4
int  mgpu_set_realspace_mode(mgpu_engine *eng, int mode);
int  mgpu_realspace_balanced(const mgpu_engine *eng);

/* ---- the boundary, host buffers (replaces src/force.c:1108 force_calc) ----
 * site/site_force: [3][ld]; c_of_m_frac: [nmols][3] (read when molpbc);
 * chg: [nsites].  Accumulates into site_force, *pe and the upper triangle of
 * stress (row-major 3x3), as the reference does. */
int mgpu_force_calc(mgpu_engine *eng, const double h[9], const double *site, int ld,
                    const double *c_of_m_frac, const double *chg, double *site_force,
                    double *pe, double stress[9], mgpu_fc_info *info);

/* ---- the boundary, host buffers (replaces src/ewald.c:280 ewald) ---- */
int mgpu_ewald(mgpu_engine *eng, const double h[9], const double *site, int ld,
               const double *chg, double *site_force, double *pe, double stress[9],
               mgpu_ew_info *info);

/* ---- the reciprocal-space sum without device allocation ----
 * No counterpart in the reference.  For callers that cannot allocate
 * device memory (code under stream capture, tight serving loops, harnesses
 * that forbid hipMalloc): the arguments, semantics and results of
 * mgpu_ewald, FP64 only, with every device buffer it needs taken from one
 * static array of MGPU_NOALLOC_BYTES (64 MiB) that each GPU holds from the
 * engine's creation until the process ends: copies of site, chg and
 * site_force, the k rows, and for the direct sum trig tables,
 * structure-factor partials, weights and back-projection partials, for the
 * gridded sum its grid, half-transformed modes, the sites' window weights and
 * the transforms' tables.  The call makes no device allocation (host memory
 * for the k set and the tables is the usual heap's); a system whose buffers
 * do not fit returns MGPU_E_CAPACITY with the size it needs.  Calls on one
 * GPU share its array: calls that overlap in time on one GPU race.  Results
 * are bit-identical to mgpu_ewald's (the same kernels, launch shapes and
 * summation order), except where mgpu_ewald takes the gridded sum and only
 * the direct sum's buffers fit: then the direct sum runs, and the two agree
 * to rounding. */
int mgpu_ewald_noalloc(mgpu_engine *eng, const double h[9], const double *site, int ld,
                       const double *chg, double *site_force, double *pe, double stress[9],
                       mgpu_ew_info *info);

/* ---- the caller, device resident (restates src/accel.c:398-617) ----
 * Upload h, scaled centre-of-mass coordinates [nmols][3] and quaternions
 * [nmols_r][4]; mgpu_eval_forces then runs make_sites, force_calc, ewald and
 * the glue on the GPU and returns pe[2], dip_mom[3] and the full stress[9].
 * Molecular forces/torques and site forces stay on the device until
 * mgpu_download_forces. */
int mgpu_upload_state(mgpu_engine *eng, const double h[9], const double *c_of_m_frac,
                      const double *quat);
int mgpu_eval_forces(mgpu_engine *eng, double pe[2], double dip_mom[3], double stress[9]);
int mgpu_download_forces(mgpu_engine *eng, double *force, double *torque,
                         double *site_xyz, double *site_force);
/* Host-side copies of the last call's diagnostics. */
int mgpu_last_info(const mgpu_engine *eng, mgpu_fc_info *fc, mgpu_ew_info *ew);
/* The system's constant terms, in program units, computed once by
 * mgpu_set_system: out = {dist, distp} (distant_const's potential and
 * pressure constants, src/accel.c:293-329; divide by V and V^2 as
 * src/accel.c:450-451 prints them), eintra (src/force.c:1158-1168), the
 * Ewald self energy and the sheet energy (src/ewald.c:367-421). */
int mgpu_statics(const mgpu_engine *eng, double out[5]);

/* ---- molecular dynamics on the device (do_step, src/accel.c:626-827) ----
 * The leapfrog splitting of src/leapfrog.c in FP64: centre-of-mass update
 * with the metric (h^T h)^-1, momentum half kicks, the symplectic rotation
 * of leapf_quat_b (or leapf_quat_a when nosymmetric_rot), when const_temp
 * the Nose-Poincare thermostat and, when const_pressure, the cell dynamics
 * of gleap_cell / update_hmom (src/leapfrog.c:475-531; 1 Parrinello-Rahman,
 * 2 uniform dilation).  Forces come from mgpu_eval_forces' device path at
 * the engine's precision. */
typedef struct {
   double step;                  /* control.step, program time units          */
   double ttmass;                /* control.ttmass                            */
   double pmass;                 /* control.pmass, the cell mass W            */
   double gkt;                   /* sys->d_of_f * kB * control.temp           */
   int const_temp;               /* 0, or nonzero = Nose-Poincare thermostat  */
   int nosymmetric_rot;          /* control.nosymmetric_rot                   */
   const double *spec_mass;      /* [nspecies] molecular masses               */
   const double *spec_inertia;   /* [nspecies][3] principal moments           */
   int const_pressure;           /* control.const_pressure: 0, 1 or 2         */
   double pressure;              /* control.pressure, program units           */
   int strain_mask;              /* control.strain_mask: bit 3i+j fixes h_ij  */
} mgpu_dynamics;

int mgpu_set_dynamics(mgpu_engine *eng, const mgpu_dynamics *dyn);
/* Scaled momenta mom[nmols][3] (mom = h^T p, as spec_mt.mom), principal
 * angular momenta amom[nmols_r][4] and thermo = {s, p_s, H_0}.  Positions and
 * h come from mgpu_upload_state. */
int mgpu_upload_momenta(mgpu_engine *eng, const double *mom, const double *amom,
                        const double thermo[3]);
/* Runs nsteps do_steps on the device.  init_H_0: evaluate H_0 on the first
 * step (accel.c:718-724).  use_graph: replay steps 2..nsteps from a captured
 * hipGraph (ignored under const_pressure: the cell, and with it the link
 * cells and the k-vector set, changes every step, so each step is launched
 * eagerly after the host reads the new h).  trace (optional, [nsteps][8])
 * receives per step: translational KE, rotational KE, pe[0], pe[1] at the
 * H_0 point, s, p_s, H_0, det(h).  pe and stress (optional) are those of the
 * last step's force evaluation. */
int mgpu_md_steps(mgpu_engine *eng, int nsteps, int init_H_0, int use_graph, double *trace,
                  double pe[2], double stress[9]);
int mgpu_download_dynamics(mgpu_engine *eng, double *c_of_m_frac, double *quat, double *mom,
                           double *amom, double thermo[3]);
/* The cell momentum sys->hmom[3][3] (zero after mgpu_set_dynamics), and the
 * cell h with its momentum after a run (h as advanced by the barostat; it
 * replaces the h of mgpu_upload_state for later calls). */
int mgpu_upload_cell_momentum(mgpu_engine *eng, const double hmom[9]);
int mgpu_download_cell(mgpu_engine *eng, double h[9], double hmom[9]);

/* ---- link cells and pair lists (bit-exact with src/force.c:426-569) ----
 * mgpu_cells: per entry (a site, or a molecule when molpbc) its cell, and the
 * cell lists in the reference's linked-list order as CSR.
 * mgpu_pairlist: for every cell the site neighbour list (nab, pbctrans) in the
 * reference's order, CSR over cells; call with nab == NULL to get the total. */
int mgpu_cells(mgpu_engine *eng, const double h[9], const double *site, int ld,
               const double *c_of_m_frac, int *dims3, int *entry_cell, int *cell_start,
               int *cell_entries);
int mgpu_pairlist(mgpu_engine *eng, const double h[9], const double *site, int ld,
                  const double *c_of_m_frac, int strict, double cutoff, long *total,
                  long *list_start, int *nab, int *pbctrans, int *nfnab);

/* ---- radial distribution functions (rdf_inner, src/force.c:1010-1103;
 * rdf_accum, src/rdf.c:94-108; run from force_calc at src/force.c:1302-1313).
 * Adds 1/density to rdf[block][bin] for every site pair closer than limit,
 * found with the strict neighbour list at limit over force_calc's cells;
 * block = init_rdf's (id_i, id_j) block order (src/rdf.c:71-89), so rdf is
 * [(max_id-1)*max_id/2][nbins] floats and may be Moldy's rdf_ptr() array.
 * Bins are exact: the pair distances are formed as the reference forms them
 * and the float additions are rounded as its loop rounds them. */
int mgpu_rdf(mgpu_engine *eng, const double h[9], const double *site, int ld,
             const double *c_of_m_frac, double limit, int nbins, float *rdf);

/* ---- parameter adjoint (no counterpart in the reference; for force
 * matching) ----
 * theta = the n_potpar parameters of every site-id pair type a <= b
 * (a, b = 0 .. max_id-1, row order), then the charge of every site id:
 * ntheta = max_id (max_id + 1) / 2 * n_potpar + max_id (mgpu_theta_count).
 * At the state of mgpu_upload_state, in FP64, for E = pe[0] + pe[1] and the
 * site forces F of mgpu_eval_forces:
 *   dE_dtheta[ntheta] = dE/dtheta (pair sums, intramolecular correction,
 *                       distant terms, Ewald sum, self and sheet energies);
 *   vjp[ntheta]       = sum_i v_i . dF_i/dtheta for the cotangent v[3][nsites];
 *   jvp[3][nsites]    = sum_t dtheta_t dF/dtheta_t for the direction dtheta.
 * Outputs may be NULL.  Charges cannot be differentiated with a framework or
 * with the surface-dipole term (MGPU_E_CAPACITY). */
int mgpu_theta_count(const mgpu_engine *eng, int *ntheta);
int mgpu_adjoint(mgpu_engine *eng, const double *v, const double *dtheta, double *dE_dtheta,
                 double *vjp, double *jvp);

/* ---- many replicas and the autotuner (no counterpart in the reference,
 * which runs one system per process) ----
 * A batch steps independent engines together (each prepared with
 * mgpu_set_dynamics, mgpu_upload_state and mgpu_upload_momenta; uneven sizes
 * and their own boxes and Ewald parameters allowed).  schedule:
 *   MGPU_SCHED_GRAPH          one hipGraph with a branch per replica, one
 *                             launch per step of the whole set;
 *   MGPU_SCHED_STREAM_GRAPHS  each replica's step graph on its own stream;
 *   MGPU_SCHED_STREAMS        eager launches on the replicas' streams;
 *   MGPU_SCHED_GROUPED        one launch per stage for all replicas (each
 *                             kernel's grid holds every replica's blocks,
 *                             the replica found from the block index), the
 *                             launches of a step in one hipGraph; mixed
 *                             precision (or no Ewald sum) and no surface
 *                             dipole, else MGPU_E_ARG;
 *   -1                        the batch's current choice (autotuned).
 * trace: [n_engines][nsteps][8] as mgpu_md_steps, or NULL.
 * mgpu_batch_autotune times every engine's launch shapes (mgpu_autotune) and
 * then each schedule over trial_steps MD steps, which advance the replicas,
 * with the engines' own real/reciprocal stream overlap and with it off;
 * ms_per_step[4] receives the best wall time per step of each schedule
 * (-1 for a schedule that does not apply).
 * mgpu_autotune picks e's launch shapes by timing its force evaluation:
 * the S(k) MFMA workgroup count and the MFMA back-projection grid (mixed;
 * returned in sk_blocks and npart: 0 = one workgroup per 128-site block,
 * r > 0 = r rounds of resident workgroups sharing the work equally), or the
 * FP64 back-projection row partitions (npart); both 0 where the evaluation
 * takes the gridded sum, which has no such shape (the overlap is tuned all
 * the same).  Results are identical up to the order of partial sums. */
enum { MGPU_SCHED_GRAPH = 0, MGPU_SCHED_STREAM_GRAPHS = 1, MGPU_SCHED_STREAMS = 2, MGPU_SCHED_GROUPED = 3 };
typedef struct mgpu_batch mgpu_batch;
int  mgpu_batch_create(mgpu_batch **batch, int device);
void mgpu_batch_destroy(mgpu_batch *batch);
const char *mgpu_batch_last_error(const mgpu_batch *batch);
int  mgpu_batch_add(mgpu_batch *batch, mgpu_engine *eng);
int  mgpu_batch_steps(mgpu_batch *batch, int nsteps, int init_H_0, int schedule, double *trace);
int  mgpu_batch_autotune(mgpu_batch *batch, int trial_steps, int *schedule, double ms_per_step[4]);
/* The grouped schedule's plan, once built: out[0] launches per step of the
 * whole batch, out[1] the launches the replicas' own steps make (summed).
 * MGPU_E_STATE before the grouped schedule has run. */
int  mgpu_batch_grouped_plan(const mgpu_batch *batch, long out[2]);
int  mgpu_autotune(mgpu_engine *eng, int reps, int *sk_blocks, int *npart);

/* ---- timing helpers for measurement ---- */
int mgpu_sync(mgpu_engine *eng);
/* Average device time (ms) of the named kernel over the calls since
 * mgpu_profile_reset, measured with HIP events on the engine's stream. */
int mgpu_profile_enable(mgpu_engine *eng, int on);
int mgpu_profile_reset(mgpu_engine *eng);
int mgpu_profile_get(const mgpu_engine *eng, const char *name, double *avg_ms, long *calls);
/* Sustained rate (TFLOP/s) of one FP16 matrix-core instruction on the
 * device: shape 16 = v_mfma_f32_16x16x32_f16 (the shape of the mixed Ewald
 * kernels), 32 = v_mfma_f32_32x32x16_f16; independent accumulator chains,
 * two, four and eight waves per SIMD, the best of them.  A measurement aid with no
 * counterpart in the reference. */
int mgpu_mfma_rate(int device, int shape, double *tflops);
/* The matrix-core work the mixed reciprocal sum issues for the engine's
 * current k set: out = {forward row tiles, sum over them of their 16-wide
 * l blocks, back-projection row tiles, sum over them of their l blocks}
 * (each GEMM multiplies a tile only over the blocks of l its rows reach).
 * A measurement aid with no counterpart in the reference; MGPU_E_STATE
 * before the first mixed evaluation. */
int mgpu_mfma_plan(const mgpu_engine *eng, long out[4]);

#ifdef __cplusplus
}
#endif
#endif
