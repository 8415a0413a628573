// The gridded reciprocal-space Ewald sum (mgpu_ewald_grid.hip): its plan and
// the pass on explicit storage.
#pragma once
#include "mgpu_internal.h"

namespace mgpu {

struct GridGeom {
   int ns, nsp, w, cap;       // sites, site stride, window width, bucket slots of a brick
   int m[3], n[3], nb[3];     // largest |h|, |k|, |l|; grid points; bricks
   double hinv[9], vol, alpha;
   bool fp64;
};

// Byte offsets into the scratch block.
struct GridSizes {
   size_t sa, sx, cnt, start, bucket, anc, fr, wt, G, T1, T2, T3, bpart, fout, bytes;
   int nred;                  // rows of bpart
};

// Transform matrices, window transforms and window polynomials: offsets into
// data.
struct GridTables {
   std::vector<double> data;
   size_t zf, zi, fr[2], fi[2], ir[2], ii[2], dec, dec_off[3], poly;
   int zf_ld, zi_ld, f_ld[2], i_ld[2];
};

struct GridBufs {
   const double *site, *w;    // [3][nsp], [nsp] charges
   double *force;             // [3][nsp], accumulated
   const KRow *rows;
   const int *rowmap;
   const double *tab;         // GridTables::data on the device
   uint8_t *base;             // GridSizes::bytes
   bool prof;
};

GridGeom grid_geom(int ns, int nsp, int hmax, int kmax, int lmax, const double h[9], const double hinv[9], double vol,
                   double alpha, double kc, bool fp64);
// Whether the gridded sum takes this system (it can, and it pays).
bool grid_applies(const GridGeom &g, int nsxf, int nk, double kc, const std::vector<KRow> &rows);
GridSizes grid_sizes(const GridGeom &g);
void grid_tables(const GridGeom &g, GridTables &t);
// The host tables for g: the engine's plan's where they are the same, else kept
// on the engine from one call to the next (mgpu_ewald_noalloc: building them
// takes 0.14 ms at 72 points an axis, 0.7 ms at 168).
std::shared_ptr<const GridTables> grid_host_tables(mgpu_engine *e, const GridGeom &g);
void grid_rowmap(const GridGeom &g, const std::vector<KRow> &rows, std::vector<int> &map);
// Clears what a pass expects cleared (brick counts); a
// pass leaves it so.
void grid_clear(mgpu_engine *e, const GridGeom &g, uint8_t *base);
// The pass: per-block energy and stress sums at base + GridSizes::bpart
// ([nred][8]), forces into b.force (after join_side when asked).
void grid_pass(mgpu_engine *e, std::vector<LaunchRec> *rec, const GridGeom &g, const GridTables &t, const GridBufs &b,
               bool join);
// For the charge adjoint of an FP64 engine: cs[k] = sum_i w_i exp(i k.r_i), and
// out[3][nsp] += w_i sum_k coeff k (C sin_i - S cos_i) with (C, S) = cs and coeff
// kc[k].w; false (nothing done) where the direct sum is to run.
bool grid_weighted_sf(mgpu_engine *e, const double *w, double2 *cs);
bool grid_backproject(mgpu_engine *e, const double *w, const double4 *kc, const double2 *cs, double *out);

}  // namespace mgpu
