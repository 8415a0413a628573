// Internal definitions shared by the engine's HIP translation units.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string>
#include <vector>
#include <map>
#include <memory>

#include "../../include/moldy_amd.h"
#include "mgpu_group.h"

#define MGPU_NPOTP 8
#define MGPU_MAX_ID 16          // site ids 0..15 (potential table in LDS)
#define MGPU_WAVE 64

namespace mgpu {

struct HipError {
   hipError_t err;
   const char *what;
   int line;
};

#define HIPCHK(x)                                                   \
   do {                                                             \
      hipError_t e_ = (x);                                          \
      if (e_ != hipSuccess) throw mgpu::HipError{e_, #x, __LINE__}; \
   } while (0)

struct StatusError {
   int code;
   std::string msg;
};

// Counts device (re)allocations of engine buffers: a captured graph holds raw
// pointers and is valid only while this is unchanged.
extern unsigned long g_alloc_epoch;

// Device buffer owned by the engine (grows, never shrinks).  reserve()
// returns true when it allocated fresh memory, whose contents are undefined
// (the allocator may hand back the address it just released).
template <class T> struct DBuf {
   T *p = nullptr;
   size_t n = 0;
   bool reserve(size_t m) {
      if (m <= n) return false;
      if (p) HIPCHK(hipFree(p));
      p = nullptr;
      size_t bytes = (m ? m : 1) * sizeof(T);
      HIPCHK(hipMalloc((void **)&p, bytes));
      n = m;
      g_alloc_epoch++;
      return true;
   }
   void free() {
      if (p) (void)hipFree(p);
      p = nullptr;
      n = 0;
   }
};

// Pinned host memory between the caller's arrays and the device.  An upload
// copies into its region (state, momenta, scalars: one allocation, so that
// they do not wait for one another) and returns with the transfers enqueued;
// the region is busy until its event.
enum { PIN_STATE = 0, PIN_MOM, PIN_SCAL, PIN_REGIONS };
struct PinBuf {
   double *p = nullptr;
   size_t n = 0;
   hipEvent_t ev[PIN_REGIONS] = {};
   bool busy[PIN_REGIONS] = {};
};

// Per-kernel event timing (HIP events on the engine stream).
struct KProf {
   double total_ms = 0;
   long calls = 0;
};

// Row of the reciprocal-lattice set: fixed (h,k), a contiguous run of l.
struct KRow {
   int h, k, l0, nl;     // l runs l0 .. l0+nl-1
   int kstart;           // index of (h,k,l0) in the reference's k order
   int pad;
   double kx, ky, kzt;   // kx, ky and kz at l = 0 (src/ewald.c:445-447)
};

}  // namespace mgpu

namespace mgpu {
struct GridTables;   // mgpu_ewald_grid.h
}

struct mgpu_engine {
   int device = 0;
   hipStream_t stream = nullptr;
   // Real-space pass of eval_forces on its own stream, concurrent with the
   // reciprocal pass; joined before the reciprocal forces are added.
   hipStream_t side = nullptr;
   hipEvent_t ev_fork = nullptr, ev_join = nullptr;
   bool join_pending = false;
   int overlap = 1;
   int precision = MGPU_FP64;
   std::string err;

   // ---- system (host copies) ----
   bool have_system = false;
   int nsites = 0, nmols = 0, nmols_r = 0, nspecies = 0, max_id = 0, ptype = 0, npar = 0;
   std::vector<int> spec_nmols, spec_nsites, spec_fw, spec_rdof, spec_site_id, spec_off;
   std::vector<double> spec_pf, site_charge, potpar;
   double cutoff = 0, subcell = 0, alpha = -1, k_cutoff = 0;
   int strict = 0, molpbc = 0, surface_dipole = 0;
   int nsitesxf = 0, nmolsxf = 0, fw_spec = -1;
   std::vector<int> site_type, site_mol, site_fw;      // per site
   std::vector<int> entry_isite, entry_num, entry_ftype, entry_mol;  // binning entries
   int nentries = 0, n_frame_types = 1;
   double eintra = 0, self_energy = 0, sheet_energy = 0, dist = 0, distp = 0;
   double max_intra = 0;       // largest intramolecular site distance
   double half_box = 0;        // half the smallest plane spacing of h
   bool intra_exact = false;   // every intramolecular pair is listed exactly once
   bool statics_done = false;
   int nsp = 0;        // padded site stride

   mgpu::PinBuf pin_up, pin_down;               // host staging of the uploads and the downloads

   // ---- static device data ----
   mgpu::DBuf<int> d_site_type, d_site_mol, d_site_fw;
   mgpu::DBuf<double> d_chg_site;             // per site, FP64
   mgpu::DBuf<int> d_entry_isite, d_entry_num, d_entry_ftype, d_entry_mol;
   mgpu::DBuf<int> d_site_entry;               // per site: its binning entry
   mgpu::DBuf<double> d_potpar;                // [max_id*max_id*8]
   mgpu::DBuf<int> d_mol_first, d_mol_spec, d_mol_quat;
   mgpu::DBuf<double> d_pf;                    // concatenated p_f_sites
   mgpu::DBuf<int> d_spec_off, d_spec_nsites, d_spec_rdof, d_spec_fw;

   // ---- dynamic device data ----
   double h[9] = {0}, hinv[9] = {0};
   mgpu::DBuf<double> d_site;                  // [3][nsp]
   mgpu::DBuf<double> d_force_site;            // [3][nsp]
   mgpu::DBuf<double> d_cm;                    // [nmols][3] scaled
   mgpu::DBuf<double> d_quat;                  // [nmols_r][4]
   mgpu::DBuf<double> d_mforce, d_mtorque;     // [nmols][3], [nmols_r][3]
   mgpu::DBuf<double> d_red;                   // reduction scratch
   mgpu::DBuf<double> d_out;                   // small result block
   mgpu::DBuf<double> d_rtmp;                  // column-sum partials
   mgpu::DBuf<double> d_rtmp_side;             // the same for the side stream
   mgpu::DBuf<int> d_iflags;                   // status flags / counters

   // ---- cells ----
   int nx = 0, ny = 0, nz = 0, ncells = 0;
   mgpu::DBuf<int> d_entry_cell, d_entry_off, d_cell_count, d_cell_start, d_cell_entries;
   mgpu::DBuf<int> d_cell_bucket;              // [bin_cap][ncells] entries by arrival slot
   int bin_cap = 8;                            // bucket slots per cell
   mgpu::DBuf<int2> d_chunk_sum;               // per chunk of cells: entries, sites; then prefix sums
   mgpu::DBuf<int> d_cell_site_start, d_scan_tmp;
   mgpu::DBuf<int> d_corig;                    // cell-ordered -> site index
   mgpu::DBuf<int> d_ccell;                    // cell-ordered -> cell index
   mgpu::DBuf<double4> d_cpos;                 // cell-ordered x,y,z,q (FP64)
   mgpu::DBuf<float4> d_cposf;                 // cell-local x,y,z,q (FP32)
   mgpu::DBuf<int2> d_cmeta;                   // type | fw<<8, mol
   // neighbour offsets (half shell in reference order, then the mirror)
   int n_half = 0, n_full = 0;
   std::vector<int> off_half;                  // [n_half][3]
   mgpu::DBuf<int4> d_off;                     // full shell: dx,dy,dz,0
   mgpu::DBuf<float4> d_offD;                  // h (dx/nx,dy/ny,dz/nz) as float
   // the full shell as z-columns of cells (dx, dy, dz lo, dz hi) and their
   // h (dx/nx, dy/ny, 0) as float, for the load-balanced real-space pass;
   // rs_ncol = 0 when the shell does not split into columns (see set_geometry)
   mgpu::DBuf<int4> d_rscol;
   mgpu::DBuf<float4> d_rscolD;
   int rs_ncol = 0, rs_own_col = 0;
   // the half of the columns the Newton-3 tiled pass walks: the own column
   // (dz >= 0) first, then the columns with (dx, dy) after (0, 0)
   mgpu::DBuf<int4> d_rshcol;
   mgpu::DBuf<float4> d_rshcolD;
   int rs_nhcol = 0;
   mgpu::DBuf<double> d_rspart;                // its partial forces, [nhcol + 1][3][nsites]
   int rs_mode = 0;                             // MGPU_RS_*
   int rs_last_bal = 0;                         // the last pass used the balanced kernel
   mgpu::DBuf<int> d_ccz;                      // cell-ordered -> z index of the cell
   mgpu::DBuf<int4> d_off_pl;                  // offsets of an explicit pair-list call
   mgpu::DBuf<int> d_pl_count, d_pl_start;     // pair-list CSR counts / starts
   mgpu::DBuf<int> d_pl_nab, d_pl_pbc, d_pl_nfnab;   // site neighbour lists (CSR)
   mgpu::DBuf<int> d_rdf_blk, d_rdf_hist;      // RDF block table, pair counts
   mgpu::DBuf<float> d_rdf_bins;               // RDF float bins
   double off_key[13] = {0};
   mgpu::DBuf<double> d_cell_part;             // per-cell energy/virial partials

   // ---- ewald ----
   int hmax = 0, kmax = 0, lmax = 0, nk = 0, nrows = 0;
   std::vector<mgpu::KRow> rows;
   std::vector<int> hkl;                        // [nk][3]
   double kset_key[10] = {0};
   mgpu::DBuf<mgpu::KRow> d_rows;
   mgpu::DBuf<int> d_krow;                      // row of each k
   mgpu::DBuf<double2> d_tx, d_ty, d_tz;        // trig tables [n+1][nsp]
   mgpu::DBuf<double> d_sk;                     // S(k) partial sums
   mgpu::DBuf<double> d_wk;                     // per-k weights
   mgpu::DBuf<int> d_rpart;                     // row partitions of the force pass
   mgpu::DBuf<double> d_fpart;                  // per-partition site forces
   mgpu::DBuf<double> d_zt64;                   // FP64 back-projection: site-major Z operand
   mgpu::DBuf<double> d_w64;                    // FP64 back-projection: folded weight operands
   mgpu::DBuf<uint8_t> d_adj;                   // scratch of the parameter adjoint (k space)
   mgpu::DBuf<uint8_t> d_adj_real;              // scratch of the parameter adjoint (real space)
   int sk_chunks = 0;

   // ---- mixed-precision ewald ----
   mgpu::DBuf<uint8_t> d_mix;                   // scratch for the MFMA path
   size_t mix_bytes = 0;
   // MFMA back-projection row order (k columns dealt to 16 row lanes), built
   // on the host from the k set when the geometry version changes
   std::vector<int> bp_src;                     // k row of each back-projection row, -1 padding
   std::vector<int2> bp_hk;                     // (h, k); h < 0 pads a lane's tail
   std::vector<float4> bp_k;                    // (kx, ky, kzt, 0), zero for padding
   std::vector<int> bp_step;                    // at a column start: index of the step from the lane's last column
   std::vector<int> bp_dsteps;                  // the distinct column steps d (q -> q + d)
   std::vector<int> bp_tile_nb;                 // per back-projection tile: blocks of 16 l reached
   std::vector<int2> fwd_hk;                    // forward row order (by l extent): (h, k), h < 0 padding
   std::vector<int> fwd_pos, fwd_tile_nb;       // each k row's forward position; per tile: blocks of 16 l
   int bp_version = -1;

   // ---- gridded ewald: tables of the grid's sizes (key: grid points, largest
   // |h| |k| |l|, FP64, sites), the k set's row map, scratch
   std::shared_ptr<const mgpu::GridTables> grid_tab;
   int grid_key[8] = {0};
   std::shared_ptr<const mgpu::GridTables> grid_host_tab;   // mgpu_ewald_noalloc's
   int grid_host_key[8] = {0};
   int grid_version = -1;
   mgpu::DBuf<double> d_gtab;
   mgpu::DBuf<uint8_t> d_grid;
   mgpu::DBuf<int> d_growmap;

   // ---- plan caching: uploads of k-set/slice metadata happen when the
   // geometry version changes, so a steady-state evaluation is launches only
   int geom_version = 0;
   int ew_plan_version = -1, mix_plan_version = -1;
   int ew_npart = 0;
   // launch shapes chosen by the autotuner (mgpu_autotune)
   int ncu = 256;                               // compute units of the device
   int tune_sk_blocks = 1024;                   // most S(k) MFMA workgroups (2 per CU resident)
   int tune_npart = 16;                         // FP64 back-projection row partitions
   int tune_force_parts = 1;                    // MFMA back-projection: rounds of resident workgroups (0: one per site block)
   void *mix_plan_ptr = nullptr;
   bool capturing = false;                      // inside hipStreamBeginCapture
   std::vector<mgpu::LaunchRec> *rec = nullptr; // record mode: grouped-launch records instead of launches
   // an evaluation whose glue sums the mixed reciprocal pass's partials
   // itself (one launch fewer): the pass leaves them here instead
   bool defer_recip = false;
   const double *recip_part = nullptr;
   int recip_rows = 0;
   // the same for a real-space pass of few rows
   bool defer_real = false;
   const double *real_part = nullptr;
   int real_rows = 0;

   // ---- molecular dynamics (device-resident state of the integrator) ----
   bool have_dyn = false;
   mgpu::DBuf<double> d_mom;                    // [nmols][3] scaled momenta
   mgpu::DBuf<double> d_amom;                   // [nmols_r][4] principal angular momenta
   mgpu::DBuf<double> d_scal;                   // integrator scalars and KE sums
   mgpu::DBuf<double> d_trace;                  // per-step record
   mgpu::DBuf<double> d_spec_dyn;               // per species: mass, I0..2, rI0..2, fw
   int trace_cap = 0;
   hipGraph_t graph = nullptr;
   hipGraphExec_t graph_exec = nullptr;
   int graph_version = -1, graph_precision = -1;
   unsigned long graph_epoch = 0;
   double dyn_step = 0, dyn_ttmass = 0, dyn_pmass = 0, dyn_gkt = 0;
   int dyn_const_temp = 0, dyn_nosym = 0, dyn_saxis = 0;
   int dyn_const_pressure = 0, dyn_strain_mask = 0;
   double dyn_pressure = 0;
   double hmom[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};   // cell momentum between runs
   double cell_loaded[18];                      // h, hmom as last put in the device slots
   bool cell_valid = false;                     // ... and still there
   std::vector<double> spec_mass, spec_inertia;

   // ---- diagnostics ----
   mgpu_fc_info last_fc{};
   mgpu_ew_info last_ew{};
   bool prof_on = false;
   std::map<std::string, mgpu::KProf> prof;
   std::vector<hipEvent_t> ev_pool;             // pairs: 2*slot, 2*slot+1
   std::vector<std::string> ev_names;           // pending slot names
   int ev_used = 0;
};

namespace mgpu {
// Slots of the small device result block e->d_out.
enum {
   OUT_REAL = 0,    // real space: pe (raw), virial upper triangle (6)
   OUT_RECIP = 8,   // reciprocal space: pe, stress upper triangle (6)
   OUT_DIP = 16,    // total dipole (3)
   OUT_CORR = 24,   // site- and molecule-virial corrections (9 + 9)
   OUT_RES = 48,    // eval_forces results: pe[2], dip[3], stress[9]
   OUT_TMP = 64,    // column sums copied to the host at once (16)
   OUT_SIZE = 80
};
// Flags block e->d_iflags: [0] error bits, [1] too-close count, [2..33] pairs,
// [40] first molecule whose quaternion norm failed.
enum { FLAG_BIN_RANGE = 1, FLAG_BIN_ROUND = 2, FLAG_QNORM = 4 };

// launch helpers implemented per translation unit
void launch_make_sites(mgpu_engine *e, int molflag_mode, bool zero_forces = false, bool bin = false);
// Link-cell binning.  prepare_binning sizes the binning buffers (and the
// bucket capacity) for the current grid; run_binning bins e->d_site, or,
// with entries_binned, takes the entry cells and bucket slots that
// make_sites (launch_make_sites with bin) has already written.
void prepare_binning(mgpu_engine *e);
void run_binning(mgpu_engine *e, bool entries_binned);
void run_realspace(mgpu_engine *e);          // -> d_out[OUT_REAL..]
void run_pairlist_count(mgpu_engine *e, int strict, double cutoff, const int *offs, int noff,
                        long *total, long *list_start_host);
void run_pairlist_fill(mgpu_engine *e, const int *offs, int noff, long total, int *nab,
                       int *pbctrans, int *nfnab);
void run_pairlist_fill_device(mgpu_engine *e, int noff, long total);
void run_rdf(mgpu_engine *e, double limit, int nbins, int noff, float *rdf_host);
void run_ewald_fp64(mgpu_engine *e);        // -> d_out[OUT_RECIP..]
void run_ewald_mixed(mgpu_engine *e);       // -> d_out[OUT_RECIP..]
bool run_ewald_grid(mgpu_engine *e);        // the same; false (nothing done) where the direct sum is to run
bool grid_chosen(const mgpu_engine *e);     // whether run_ewald_grid runs it
// The device part of eval_forces after the two boundary calls: second
// make_sites, dipole and surface term, molecular forces and torques, virial
// correction and the assembly of pe, dipole and stress into d_out[OUT_RES..].
void run_glue(mgpu_engine *e);
void eval_forces_device(mgpu_engine *e, bool clear_flags);
// Charge derivatives of the FP64 Ewald sum for the sites in d_site (no
// frameworks): dE[max_id], the cotangent product vjp[max_id] for the site
// force cotangent v (device [3][nsp], or null), and jvp (device [3][nsp],
// accumulated) for the charge direction dq (device [max_id]).
void ewald_charge_adjoint(mgpu_engine *e, const double *v, const double *dq_dev, double *dE, double *vjp,
                          double *jvp);
// Parameter adjoint (mgpu_adjoint.hip): theta = pair-type parameters then
// site-id charges; host arrays v[3][nsites], dtheta/dE/vjp[ntheta],
// jvp[3][nsites], each optional.
int adjoint_ntheta(const mgpu_engine *e);
void run_adjoint(mgpu_engine *e, const double *v, const double *dtheta, double *dE, double *vjp, double *jvp);
// molecular dynamics (mgpu_dynamics.hip)
void md_setup(mgpu_engine *e, const mgpu_dynamics *d);
// n[i] doubles from src[i] (host) to dst[i] (device) on e->stream through a
// region of pin_up, for k arrays; src may be reused on return.
void upload_pinned(mgpu_engine *e, int region, int k, const double *const *src, double *const *dst, const size_t *n);
// n[i] doubles from src[i] (device) to dst[i] (host), complete on return.
void download_pinned(mgpu_engine *e, int k, const double *const *src, double *const *dst, const size_t *n);
#define MGPU_SCAL_SIZE 192   // integrator scalars (mgpu_dynamics.hip)
void md_set_scalars(mgpu_engine *e, const double thermo[3]);
void md_thermo(const double scal[4], double thermo[3]);   // from the first integrator scalars
// A run of cap recorded steps; init_h0: its first step sets H_0.
void md_reset_record(mgpu_engine *e, int cap, bool init_h0);
void md_step_launch(mgpu_engine *e);
void md_load_cell(mgpu_engine *e);
void md_step_pressure(mgpu_engine *e);
void md_fetch_cell(mgpu_engine *e, double h[9], double hmom[9]);
void set_geometry(mgpu_engine *e, const double h[9]);
// Size of the static device scratch array of mgpu_ewald_noalloc.
#define MGPU_NOALLOC_BYTES (64u << 20)
// Takes (once per device, with that device current) the device address of
// the scratch array.
void scratch_init(int device);
// The FP64 reciprocal pass of mgpu_ewald with every device buffer in the
// scratch array: site, site_force and chg are host arrays as for mgpu_ewald
// (site_force accumulated); out7 receives the raw k-sum energy and stress
// upper triangle.  Throws MGPU_E_CAPACITY when the system does not fit.
void ewald_noalloc(mgpu_engine *e, const double h[9], const double *site, int ld, const double *chg,
                   double *site_force, double out7[7], mgpu_ew_info *info);
// The reference's half-space k set (src/ewald.c:441-461) for cell h within
// k_cutoff kc, as rows of one (h, k) and a contiguous run of l.
struct KSet {
   int hmax = 0, kmax = 0, lmax = 0, nk = 0;
   std::vector<KRow> rows;
   std::vector<int> hkl;     // [nk][3]
   std::vector<int> krow;    // row of each k
};
void build_kset(const double h[9], const double hinv[9], double kc, KSet &ks);
// Main stream waits for the side stream's real-space pass (if one is pending).
void join_side(mgpu_engine *e);
bool step_graph_current(const mgpu_engine *e);
void ensure_step_graph(mgpu_engine *e);
void autotune_engine(mgpu_engine *e, int reps, int *sk_blocks, int *npart);
void handle_flags(mgpu_engine *e, const int *fl);   // throws on error flags
int md_trace_width();
// Fill with zeros by a kernel (safe inside a captured graph).
void zero_async(mgpu_engine *e, void *p, size_t bytes);
void device_scan_int(mgpu_engine *e, const int *in, int *out, int n);  // exclusive, out[n]=total
void sum_cols(mgpu_engine *e, const double *in, int nrows, int ncols, double *host_out);
void reduce_cols(mgpu_engine *e, const double *in, int nrows, int ncols, double *out_dev);
// reduce_cols with the caller's storage: tmp holds reduce_cols_blocks(nrows)
// * ncols partials; *count must be zero at the launch and is zero after it.
int reduce_cols_blocks(int nrows);
void reduce_cols_into(std::vector<LaunchRec> *rec, hipStream_t st, const double *in, int nrows, int ncols,
                      double *out_dev, double *tmp, unsigned *count);
double host_det(const double a[9]);
void host_invert(const double a[9], double b[9]);

// Event timing that does not stall the stream: events come from a pool and
// are resolved when the profile is read (mgpu_profile_get).  A null engine
// times nothing.
struct ProfScope {
   mgpu_engine *e;
   const char *name;
   int slot = -1;
   ProfScope(mgpu_engine *e_, const char *n);
   ~ProfScope();
};
void prof_resolve(mgpu_engine *e);
}  // namespace mgpu

// ---------------------------------------------------------- device helpers
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
   for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
   return v;
}
__device__ __forceinline__ float wave_sumf(float v) {
#pragma unroll
   for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
   return v;
}
template <int CTRL> __device__ __forceinline__ double row_ror(double x) {
   const long long b = __builtin_bit_cast(long long, x);
   const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, false);
   const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, false);
   return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double lane_value(double x, int lane) {
   const long long b = __builtin_bit_cast(long long, x);
   const int lo = __builtin_amdgcn_readlane((int)b, lane), hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
   return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned)lo);
}
// Sums of x, y, z over the wave, in every lane: x and y share the halves of a
// register, z the odd rows of 16, so that 7 steps do for 18.
__device__ __forceinline__ void wave_sum3(double &x, double &y, double &z, int lane) {
   const bool hi = lane & 32, odd = lane & 16;
   const double u = (hi ? y : x) + __shfl_xor(hi ? x : y, 32, 64), v = z + __shfl_xor(z, 32, 64);
   double t = (odd ? v : u) + __shfl_xor(odd ? u : v, 16, 64);
   t += row_ror<0x128>(t);
   t += row_ror<0x124>(t);
   t += row_ror<0x122>(t);
   t += row_ror<0x121>(t);
   x = lane_value(t, 0);
   y = lane_value(t, 32);
   z = lane_value(t, 16);
}

// Cell index along one axis, restating cellbin (src/force.c:426-446): the
// 8*DBL_EPSILON edge clamp, floor((s+0.5)*n), and the reference's two error
// conditions as flag bits.
#pragma clang fp contract(off)
__device__ __forceinline__ int cellbin_dev(double rc, int nc, double fnc, double eps, int *flag) {
   if (rc < -0.5 + eps || rc >= 0.5 - eps) {
      if (rc < -0.5 + eps && rc >= -0.5 - eps)
         rc = -0.5;
      else if (rc >= 0.5 - eps && rc <= 0.5 + eps)
         rc = 0.5 - eps;
      else
         *flag |= mgpu::FLAG_BIN_RANGE;
   }
   int ib = (int)floor((rc + 0.5) * fnc);
   if (ib >= nc || ib < 0) {
      *flag |= mgpu::FLAG_BIN_ROUND;
      ib = ib < 0 ? 0 : nc - 1;
   }
   return ib;
}
#pragma clang fp contract(on)

__device__ __forceinline__ int wave_incl_scan(int v, int lane) {
#pragma unroll
   for (int o = 1; o < 64; o <<= 1) {
      int t = __shfl_up(v, o, 64);
      if (lane >= o) v += t;
   }
   return v;
}
