// Link-cell binning and site neighbour lists on the GPU.
//
// Binning restates fill_cells/cellbin (src/force.c:119-137, 426-486): the
// fractional coordinate s = h^-1 r is formed in the reference's operation
// order with FMA contraction off, then floor((s+0.5)*n) with the 8*DBL_EPSILON
// edge clamp.  Moldy pushes each entry on the head of its cell's linked list,
// so a cell lists its entries in decreasing entry order; the counting sort
// below reproduces exactly that order.  The cell-ordered site arrays written
// here feed the real-space kernel.
//
// The site neighbour lists restate site_neighbour_list (src/force.c:521-569):
// per reference cell, frame type by frame type, the half-shell offsets in
// list order (own cell excluded for the framework pass), each neighbour
// cell's entries in list order, and each entry's sites, tagged with the
// periodic image code 9*(sx+1)+3*(sy+1)+(sz+1).
#include "mgpu_internal.h"

#include <algorithm>

using namespace mgpu;


// ----------------------------------------------------------------- scan
static __global__ void k_scan_block(const int *__restrict__ in, int *__restrict__ out,
                                    int *__restrict__ bsum, int n) {
   __shared__ int ws[16];
   int i = blockIdx.x * 1024 + threadIdx.x;
   int v = i < n ? in[i] : 0;
   int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
   int inc = wave_incl_scan(v, lane);
   if (lane == 63) ws[w] = inc;
   __syncthreads();
   if (w == 0) {
      int t = lane < 16 ? ws[lane] : 0;
      int ti = wave_incl_scan(t, lane);
      if (lane < 16) ws[lane] = ti - t;
   }
   __syncthreads();
   int excl = inc - v + ws[w];
   if (i < n) out[i] = excl;
   if (threadIdx.x == 1023) bsum[blockIdx.x] = excl + v;
}

static __global__ void k_scan_sums(int *__restrict__ bsum, int nb, int *__restrict__ total) {
   // single block: exclusive scan of up to 1024*k block sums
   __shared__ int carry;
   if (threadIdx.x == 0) carry = 0;
   __syncthreads();
   for (int base = 0; base < nb; base += 1024) {
      __shared__ int ws[16];
      int i = base + threadIdx.x;
      int v = i < nb ? bsum[i] : 0;
      int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
      int inc = wave_incl_scan(v, lane);
      if (lane == 63) ws[w] = inc;
      __syncthreads();
      if (w == 0) {
         int t = lane < 16 ? ws[lane] : 0;
         int ti = wave_incl_scan(t, lane);
         if (lane < 16) ws[lane] = ti - t;
      }
      __syncthreads();
      int excl = inc - v + ws[w] + carry;
      if (i < nb) bsum[i] = excl;
      __syncthreads();
      if (threadIdx.x == 1023) carry = excl + v;
      __syncthreads();
   }
   if (threadIdx.x == 0) *total = carry;
}

static __global__ void k_scan_add(int *__restrict__ out, const int *__restrict__ bsum, int n,
                                  const int *__restrict__ total) {
   int i = blockIdx.x * 1024 + threadIdx.x;
   if (i < n) out[i] += bsum[blockIdx.x];
   if (i == 0) out[n] = *total;
}

void mgpu::device_scan_int(mgpu_engine *e, const int *in, int *out, int n) {
   int nb = (n + 1023) / 1024;
   e->d_scan_tmp.reserve((size_t)nb + 2);
   int *bsum = e->d_scan_tmp.p, *total = e->d_scan_tmp.p + nb;
   if (nb == 0) nb = 1;
   k_scan_block<<<nb, 1024, 0, e->stream>>>(in, out, bsum, n);
   k_scan_sums<<<1, 1024, 0, e->stream>>>(bsum, (n + 1023) / 1024, total);
   k_scan_add<<<nb, 1024, 0, e->stream>>>(out, bsum, n, total);
}

// ------------------------------------------------- column sums (two stages)
// out[c] = sum over rows of in[r*ncols + c], ncols <= 16, summed in a fixed
// order (per-block partials, then one block), so results are reproducible.
// Column sums of in[nrows][ncols] (ncols <= 16) into out[ncols] in one
// launch: every block writes its partial, and the last block to finish (an
// atomic count, reset by that block) adds the partials in block order, so
// the result does not depend on which block finishes last.
static __device__ __forceinline__ void b_rc(int bx, int nbx, const double *__restrict__ in, int nrows, int ncols,
                                            int chunk, unsigned *__restrict__ count, double *__restrict__ tmp,
                                            double *__restrict__ out) {
   __shared__ double ws[4][16];
   __shared__ double fin[256];
   __shared__ bool last;
   const int r0 = bx * chunk, r1 = min(nrows, r0 + chunk);
   double acc[16];
#pragma unroll
   for (int c = 0; c < 16; c++) acc[c] = 0.0;
   for (int r = r0 + (int)threadIdx.x; r < r1; r += 256)
#pragma unroll
      for (int c = 0; c < 16; c++)
         if (c < ncols) acc[c] += in[(size_t)r * ncols + c];
   const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
   for (int c = 0; c < 16; c++) {
      if (c >= ncols) break;
      double t = wave_sum(acc[c]);
      if (lane == 0) ws[w][c] = t;
   }
   __syncthreads();
   if (threadIdx.x < ncols)
      tmp[(size_t)bx * ncols + threadIdx.x] =
          ws[0][threadIdx.x] + ws[1][threadIdx.x] + ws[2][threadIdx.x] + ws[3][threadIdx.x];
   __threadfence();
   __syncthreads();
   if (threadIdx.x == 0) last = atomicAdd(count, 1u) == (unsigned)nbx - 1u;
   __syncthreads();
   if (last) {
      __threadfence();
      // per = 256 / ncols threads a column, thread q of them summing the
      // blocks q, q + per, ... in order; then the per sums in order
      const int per = 256 / ncols, c = (int)threadIdx.x % ncols, q = (int)threadIdx.x / ncols;
      double t = 0.0;
      if (q < per)
         for (unsigned b = q; b < (unsigned)nbx; b += per) t += tmp[(size_t)b * ncols + c];
      fin[threadIdx.x] = t;
      __syncthreads();
      if ((int)threadIdx.x < ncols) {
         double u = 0.0;
         for (int k = 0; k < per; k++) u += fin[k * ncols + threadIdx.x];
         out[threadIdx.x] = u;
      }
      if (threadIdx.x == 0) *count = 0u;
   }
}
static __global__ __launch_bounds__(256) void k_rc(const double *__restrict__ in, int nrows, int ncols, int chunk,
                                            unsigned *__restrict__ count, double *__restrict__ tmp,
                                            double *__restrict__ out) {
   b_rc(blockIdx.x, gridDim.x, in, nrows, ncols, chunk, count, tmp, out);
}

int mgpu::reduce_cols_blocks(int nrows) { return std::max(1, std::min(1024, (nrows + 255) / 256)); }

void mgpu::reduce_cols_into(std::vector<LaunchRec> *rec, hipStream_t st, const double *in, int nrows, int ncols,
                            double *out_dev, double *tmp, unsigned *count) {
   if (ncols > 16) throw StatusError{MGPU_E_ARG, "reduce_cols: more than 16 columns"};
   const int nb = reduce_cols_blocks(nrows);
   const int chunk = (nrows + nb - 1) / nb;
   glaunch<k_rc, b_rc, 256>(rec, st, nb, 256, 0, in, nrows, ncols, chunk, count, tmp, out_dev);
}

void mgpu::reduce_cols(mgpu_engine *e, const double *in, int nrows, int ncols, double *out_dev) {
   // d_rtmp: a completion count in its first slot, then the partials
   const bool fresh = e->d_rtmp.reserve((size_t)reduce_cols_blocks(nrows) * ncols + 16);
   unsigned *count = (unsigned *)e->d_rtmp.p;
   if (fresh) zero_async(e, count, 8);   // fresh memory: the count starts at zero
   reduce_cols_into(e->rec, e->stream, in, nrows, ncols, out_dev, e->d_rtmp.p + 1, count);
}

// ---------------------------------------------------------------- binning
#pragma clang fp contract(off)
// Three or four launches and no fills.
//  k_bin         one thread per entry: its cell and a slot in the cell's
//                bucket (slot-major: bucket[slot * ncells + cell]) from the
//                cell's atomic count.  In a force evaluation make_sites does
//                this instead, from the position or centre it has just formed
//                (k_make_sites with binning).
//  k_cell_csr    one thread per cell, one block per chunk of BIN_CHUNK
//                cells: the cell's entries in Moldy's list order (descending
//                entry index), block scans of the cells' entry and site
//                counts (positions within the chunk), each entry's position
//                and first site slot within the chunk, and the chunk's
//                totals.  It clears the cell counts for the next binning.
//  k_site_place  one thread per site, in site order, so that its reads are
//                coalesced: the slot is the chunk's first site slot plus the
//                entry's offset in the chunk plus the site's rank in its
//                entry.  The same grid adds the chunk offsets to cell_start
//                and cell_site_start and places the entries in cell_entries.
//                Up to BIN_PRE_LDS chunks, every block forms the chunks'
//                exclusive prefix sums in its LDS (a few KB of L2 reads a
//                block); beyond, one block (k_chunk_scan) forms them first.
// A cell holding more entries than its bucket takes its entries from
// entry_cell instead, scanned in descending order; the bucket holds four
// times the mean occupancy (at least 8), so this path is for pathological
// geometries only.  The cell counts are zero between binnings.  No atomic
// is shared beyond a cell: same-address atomics serialise (per-chunk atomic
// totals made k_bin six times slower), and a single-pass look-back over the
// chunks measured slower than the one-block scan, its status reads crossing
// the XCDs' L2s.
constexpr int BIN_CHUNK = 256;   // cells per chunk = threads per k_cell_csr block
constexpr int BIN_PRE_LDS = 2048; // chunks whose prefix sums k_site_place forms itself
constexpr int BIN_REG = 8;       // entries a cell sorts in registers

struct BinArgs {
   double hi[9];
   int nx, ny, nz, ne, nsp, ncells, cap;
   double eps;
};

static __device__ __forceinline__ void b_bin(int bx, int nbx, const BinArgs &a, const double *__restrict__ site,
                                      const double *__restrict__ cm, const int *__restrict__ e_isite,
                                      const int *__restrict__ e_mol, int *__restrict__ e_cell,
                                      int *__restrict__ c_count, int *__restrict__ bucket, int *__restrict__ flags) {
   const int e = bx * blockDim.x + threadIdx.x;
   if (e >= a.ne) return;
   double s0, s1, s2;
   const int m = e_mol[e];
   if (m < 0) {
      int is = e_isite[e];
      double r0 = site[is], r1 = site[a.nsp + is], r2 = site[2 * a.nsp + is];
      // mat_vec_mul, src/matrix.c:81-83 (left-to-right, no contraction)
      s0 = a.hi[0] * r0 + a.hi[1] * r1 + a.hi[2] * r2;
      s1 = a.hi[3] * r0 + a.hi[4] * r1 + a.hi[5] * r2;
      s2 = a.hi[6] * r0 + a.hi[7] * r1 + a.hi[8] * r2;
   } else {
      s0 = cm[3 * m];
      s1 = cm[3 * m + 1];
      s2 = cm[3 * m + 2];
   }
   int flag = 0;
   const int c = cellbin_dev(s2, a.nz, (double)a.nz, a.eps, &flag) +
                 a.nz * (cellbin_dev(s1, a.ny, (double)a.ny, a.eps, &flag) +
                         a.ny * cellbin_dev(s0, a.nx, (double)a.nx, a.eps, &flag));
   if (flag) atomicOr(flags, flag);
   e_cell[e] = c;
   const int slot = atomicAdd(&c_count[c], 1);
   if (slot < a.cap) bucket[(size_t)slot * a.ncells + c] = e;
}
static __global__ __launch_bounds__(256) void k_bin(BinArgs a, const double *__restrict__ site,
                                             const double *__restrict__ cm, const int *__restrict__ e_isite,
                                             const int *__restrict__ e_mol, int *__restrict__ e_cell,
                                             int *__restrict__ c_count, int *__restrict__ bucket,
                                             int *__restrict__ flags) {
   b_bin(blockIdx.x, gridDim.x, a, site, cm, e_isite, e_mol, e_cell, c_count, bucket, flags);
}
#pragma clang fp contract(on)

struct CsrArgs {
   int ncells, ne, cap;
};

static __device__ __forceinline__ void b_cell_csr(int bx, int nbx, const CsrArgs &a, int *__restrict__ c_count,
                                           const int *__restrict__ bucket, const int *__restrict__ e_cell,
                                           const int *__restrict__ e_num, int *__restrict__ c_start,
                                           int *__restrict__ c_site_start, int *__restrict__ e_rank,
                                           int *__restrict__ e_off, int2 *__restrict__ chunk_tot) {
   __shared__ int wsum[4][2];   // per wave: entries, sites
   const int t = threadIdx.x, lane = t & 63, w = t >> 6;
   const int c = bx * BIN_CHUNK + t;
   const size_t nc = (size_t)a.ncells;
   // this cell's entries, descending; its site count
   const int n = c < a.ncells ? c_count[c] : 0;
   int ent[BIN_REG], num[BIN_REG], nst = 0;
   if (n <= BIN_REG) {
#pragma unroll
      for (int i = 0; i < BIN_REG; i++) ent[i] = i < n ? bucket[i * nc + c] : -1;
      if (n > 1) {
#pragma unroll
         for (int i = 1; i < BIN_REG; i++)
#pragma unroll
            for (int j = i; j > 0; j--) {
               int x = ent[j - 1], y = ent[j];
               ent[j - 1] = max(x, y);
               ent[j] = min(x, y);
            }
      }
#pragma unroll
      for (int i = 0; i < BIN_REG; i++) {
         num[i] = i < n ? e_num[ent[i]] : 0;
         nst += num[i];
      }
   } else if (n <= a.cap) {
      for (int i = 0; i < n; i++) nst += e_num[bucket[i * nc + c]];
   } else {
      for (int q = a.ne - 1; q >= 0; q--)
         if (e_cell[q] == c) nst += e_num[q];
   }
   const int ie = wave_incl_scan(n, lane), is = wave_incl_scan(nst, lane);
   if (lane == 63) {
      wsum[w][0] = ie;
      wsum[w][1] = is;
   }
   __syncthreads();
   int cs = ie - n, ss = is - nst;
#pragma unroll
   for (int k = 0; k < 4; k++)
      if (k < w) {
         cs += wsum[k][0];
         ss += wsum[k][1];
      }
   if (t == BIN_CHUNK - 1) chunk_tot[bx] = make_int2(cs + n, ss + nst);
   if (c < a.ncells) {
      c_start[c] = cs;
      c_site_start[c] = ss;
      c_count[c] = 0;
   }
   if (n <= BIN_REG) {
#pragma unroll
      for (int i = 0; i < BIN_REG; i++)
         if (i < n) {
            e_rank[ent[i]] = cs + i;
            e_off[ent[i]] = ss;
            ss += num[i];
         }
   } else if (n <= a.cap) {
      // selection: the largest entry below the previous one
      int prev = a.ne;
      for (int i = 0; i < n; i++) {
         int best = -1;
         for (int k = 0; k < n; k++) {
            int v = bucket[k * nc + c];
            if (v < prev && v > best) best = v;
         }
         e_rank[best] = cs + i;
         e_off[best] = ss;
         ss += e_num[best];
         prev = best;
      }
   } else {
      int i = 0;
      for (int q = a.ne - 1; q >= 0; q--)
         if (e_cell[q] == c) {
            e_rank[q] = cs + i++;
            e_off[q] = ss;
            ss += e_num[q];
         }
   }
}
static __global__ __launch_bounds__(BIN_CHUNK) void k_cell_csr(CsrArgs a, int *__restrict__ c_count,
                                                        const int *__restrict__ bucket,
                                                        const int *__restrict__ e_cell, const int *__restrict__ e_num,
                                                        int *__restrict__ c_start, int *__restrict__ c_site_start,
                                                        int *__restrict__ e_rank, int *__restrict__ e_off,
                                                        int2 *__restrict__ chunk_tot) {
   b_cell_csr(blockIdx.x, gridDim.x, a, c_count, bucket, e_cell, e_num, c_start, c_site_start, e_rank, e_off,
              chunk_tot);
}

// One block of 1024: pre[k] = totals of the chunks before k, and
// pre[nchunk] = all of them.  Thread t sums a contiguous segment.
static __device__ __forceinline__ void b_chunk_scan(int bx, int nbx, int nchunk, const int2 *__restrict__ tot,
                                             int2 *__restrict__ pre) {
   __shared__ int ws[16][2];
   const int t = threadIdx.x, lane = t & 63, w = t >> 6;
   const int seg = (nchunk + 1023) / 1024, k0 = min(nchunk, t * seg), k1 = min(nchunk, k0 + seg);
   int se = 0, ss = 0;
   for (int k = k0; k < k1; k++) {
      const int2 v = tot[k];
      se += v.x;
      ss += v.y;
   }
   const int ie = wave_incl_scan(se, lane), is = wave_incl_scan(ss, lane);
   if (lane == 63) {
      ws[w][0] = ie;
      ws[w][1] = is;
   }
   __syncthreads();
   int be = ie - se, bs = is - ss;
   for (int k = 0; k < w; k++) {
      be += ws[k][0];
      bs += ws[k][1];
   }
   for (int k = k0; k < k1; k++) {
      pre[k] = make_int2(be, bs);
      const int2 v = tot[k];
      be += v.x;
      bs += v.y;
   }
   if (t == 1023) pre[nchunk] = make_int2(be, bs);
}
static __global__ __launch_bounds__(1024) void k_chunk_scan(int nchunk, const int2 *__restrict__ tot,
                                                            int2 *__restrict__ pre) {
   b_chunk_scan(blockIdx.x, gridDim.x, nchunk, tot, pre);
}

struct PlaceArgs {
   double h[9];
   int nx, ny, nz, nsites, nsp, ncells, ne, nchunk, pre_lds;
};

static __device__ __forceinline__ void b_site_place(int bx, int nbx, const PlaceArgs &a,
                                                    const int *__restrict__ site_entry,
                                                    const int *__restrict__ e_isite, const int *__restrict__ e_rank,
                                                    const int *__restrict__ e_off, const int *__restrict__ e_cell,
                                                    const int2 *__restrict__ tot, const int2 *pre,
                                                    const double *__restrict__ site, const double *__restrict__ chg,
                                                    const int *__restrict__ stype, const int *__restrict__ smol,
                                                    const int *__restrict__ sfw, int *__restrict__ c_start,
                                                    int *__restrict__ c_site_start, int *__restrict__ c_entries,
                                                    double4 *__restrict__ cpos, float4 *__restrict__ cposf,
                                                    int2 *__restrict__ cmeta, int *__restrict__ corig,
                                                    int *__restrict__ ccell, int *__restrict__ ccz) {
   // the chunks' exclusive prefix sums: from k_chunk_scan, or formed here
   // (thread q sums a contiguous segment, a block scan of the segment sums)
   __shared__ int2 spre[BIN_PRE_LDS + 1];
   __shared__ int ws[4][2];
   if (a.pre_lds) {
      const int q = threadIdx.x, lane = q & 63, w = q >> 6;
      const int seg = (a.nchunk + 255) / 256, k0 = min(a.nchunk, q * seg), k1 = min(a.nchunk, k0 + seg);
      int se = 0, ss = 0;
      for (int k = k0; k < k1; k++) {
         const int2 v = tot[k];
         se += v.x;
         ss += v.y;
      }
      const int ie = wave_incl_scan(se, lane), is = wave_incl_scan(ss, lane);
      if (lane == 63) {
         ws[w][0] = ie;
         ws[w][1] = is;
      }
      __syncthreads();
      int be = ie - se, bs = is - ss;
      for (int k = 0; k < w; k++) {
         be += ws[k][0];
         bs += ws[k][1];
      }
      for (int k = k0; k < k1; k++) {
         spre[k] = make_int2(be, bs);
         const int2 v = tot[k];
         be += v.x;
         bs += v.y;
      }
      if (q == 255) spre[a.nchunk] = make_int2(be, bs);
      __syncthreads();
      pre = spre;
   }
   const int t = bx * blockDim.x + threadIdx.x;
   if (t < a.ncells) {
      const int2 p = pre[t / BIN_CHUNK];
      c_start[t] += p.x;
      c_site_start[t] += p.y;
   } else if (t == a.ncells) {
      const int2 q = pre[(a.ncells + BIN_CHUNK - 1) / BIN_CHUNK];
      c_start[t] = q.x;
      c_site_start[t] = q.y;
   }
   if (t < a.ne) c_entries[pre[e_cell[t] / BIN_CHUNK].x + e_rank[t]] = t;
   if (t >= a.nsites) return;
   const int en = site_entry[t];
   const int c = e_cell[en];
   const int pos = pre[c / BIN_CHUNK].y + e_off[en] + (t - e_isite[en]);
   const double x = site[t], y = site[a.nsp + t], z = site[2 * a.nsp + t], q = chg[t];
   const int ty = stype[t], mo = smol[t], fw = sfw[t];
   int ix = c / (a.ny * a.nz), iy = c / a.nz - a.ny * ix, iz = c - a.nz * (iy + a.ny * ix);
   double f0 = (double)ix / a.nx - 0.5, f1 = (double)iy / a.ny - 0.5, f2 = (double)iz / a.nz - 0.5;
   double o0 = a.h[0] * f0 + a.h[1] * f1 + a.h[2] * f2;
   double o1 = a.h[3] * f0 + a.h[4] * f1 + a.h[5] * f2;
   double o2 = a.h[6] * f0 + a.h[7] * f1 + a.h[8] * f2;
   cpos[pos] = make_double4(x, y, z, q);
   cposf[pos] = make_float4((float)(x - o0), (float)(y - o1), (float)(z - o2), (float)q);
   cmeta[pos] = make_int2(ty | (fw << 8), mo);
   corig[pos] = t;
   ccell[pos] = c;
   ccz[pos] = iz;
}
static __global__ __launch_bounds__(256) void k_site_place(PlaceArgs a, const int *__restrict__ site_entry,
                                                    const int *__restrict__ e_isite, const int *__restrict__ e_rank,
                                                    const int *__restrict__ e_off, const int *__restrict__ e_cell,
                                                    const int2 *__restrict__ tot, const int2 *pre,
                                                    const double *__restrict__ site, const double *__restrict__ chg,
                                                    const int *__restrict__ stype, const int *__restrict__ smol,
                                                    const int *__restrict__ sfw, int *__restrict__ c_start,
                                                    int *__restrict__ c_site_start, int *__restrict__ c_entries,
                                                    double4 *__restrict__ cpos, float4 *__restrict__ cposf,
                                                    int2 *__restrict__ cmeta, int *__restrict__ corig,
                                                    int *__restrict__ ccell, int *__restrict__ ccz) {
   b_site_place(blockIdx.x, gridDim.x, a, site_entry, e_isite, e_rank, e_off, e_cell, tot, pre, site, chg, stype,
                smol, sfw, c_start, c_site_start, c_entries, cpos, cposf, cmeta, corig, ccell, ccz);
}

void mgpu::prepare_binning(mgpu_engine *e) {
   const int nc = e->ncells, ne = e->nentries;
   const int nchunk = (nc + BIN_CHUNK - 1) / BIN_CHUNK;
   int cap = 8;
   while (cap < 4.0 * ne / std::max(nc, 1) && cap < (1 << 16)) cap *= 2;
   e->bin_cap = cap;
   e->d_entry_cell.reserve(ne);
   e->d_entry_off.reserve(2 * (size_t)ne);   // entry site offsets, then positions, within the chunk
   e->d_cell_start.reserve(nc + 1);
   e->d_cell_site_start.reserve(nc + 1);
   e->d_cell_entries.reserve(ne + 1);
   e->d_cell_bucket.reserve((size_t)cap * nc);
   e->d_chunk_sum.reserve(2 * (size_t)nchunk + 1);   // totals, then prefix sums
   e->d_cpos.reserve(e->nsites + 1);
   e->d_cposf.reserve(e->nsites + 1);
   e->d_cmeta.reserve(e->nsites + 1);
   e->d_corig.reserve(e->nsites + 1);
   e->d_ccell.reserve(e->nsites + 1);
   e->d_ccz.reserve(e->nsites + 1);
   // the counts are cleared by the kernel that reads them; fresh memory
   // starts at zero
   if (e->d_cell_count.reserve(nc + 1)) zero_async(e, e->d_cell_count.p, sizeof(int) * (nc + 1));
}

// Bin the current site coordinates (e->d_site) and build the cell-ordered
// arrays.  Requires e->nx/ny/nz set and e->hinv valid; with entries_binned,
// prepare_binning and the binning make_sites have run since.
void mgpu::run_binning(mgpu_engine *e, bool entries_binned) {
   ProfScope ps(e, "binning");
   if (!entries_binned) prepare_binning(e);
   const int nc = e->ncells, ne = e->nentries, cap = e->bin_cap;
   const int nchunk = (nc + BIN_CHUNK - 1) / BIN_CHUNK;
   int *e_off = e->d_entry_off.p, *e_rank = e->d_entry_off.p + ne;
   int2 *tot = e->d_chunk_sum.p, *pre = e->d_chunk_sum.p + nchunk;
   if (!entries_binned) {
      BinArgs a;
      for (int i = 0; i < 9; i++) a.hi[i] = e->hinv[i];
      a.nx = e->nx; a.ny = e->ny; a.nz = e->nz; a.ne = ne; a.nsp = e->nsp; a.ncells = nc; a.cap = cap;
      a.eps = 8.0 * 2.220446049250313e-16;   // 8 * precision(), src/force.c:437
      glaunch<k_bin, b_bin, 256>(e->rec, e->stream, (ne + 255) / 256, 256, 0, a, e->d_site.p, e->d_cm.p,
                                 e->d_entry_isite.p, e->d_entry_mol.p, e->d_entry_cell.p, e->d_cell_count.p,
                                 e->d_cell_bucket.p, e->d_iflags.p);
   }
   CsrArgs ca;
   ca.ncells = nc; ca.ne = ne; ca.cap = cap;
   glaunch<k_cell_csr, b_cell_csr, BIN_CHUNK>(e->rec, e->stream, nchunk, BIN_CHUNK, 0, ca, e->d_cell_count.p,
                                              e->d_cell_bucket.p, e->d_entry_cell.p, e->d_entry_num.p,
                                              e->d_cell_start.p, e->d_cell_site_start.p, e_rank, e_off, tot);
   const bool pre_lds = nchunk <= BIN_PRE_LDS;
   if (!pre_lds) glaunch<k_chunk_scan, b_chunk_scan, 1024>(e->rec, e->stream, 1, 1024, 0, nchunk, tot, pre);
   PlaceArgs f;
   for (int i = 0; i < 9; i++) f.h[i] = e->h[i];
   f.nx = e->nx; f.ny = e->ny; f.nz = e->nz; f.nsites = e->nsites; f.nsp = e->nsp; f.ncells = nc; f.ne = ne;
   f.nchunk = nchunk; f.pre_lds = pre_lds;
   const int nt = std::max(std::max(e->nsites, nc + 1), ne);
   glaunch<k_site_place, b_site_place, 256>(e->rec, e->stream, (nt + 255) / 256, 256, 0, f, e->d_site_entry.p,
                                            e->d_entry_isite.p, e_rank, e_off, e->d_entry_cell.p, tot, pre,
                                            e->d_site.p, e->d_chg_site.p, e->d_site_type.p, e->d_site_mol.p,
                                            e->d_site_fw.p, e->d_cell_start.p, e->d_cell_site_start.p,
                                            e->d_cell_entries.p, e->d_cpos.p, e->d_cposf.p, e->d_cmeta.p,
                                            e->d_corig.p, e->d_ccell.p, e->d_ccz.p);
}

// ------------------------------------------------------ site neighbour lists
struct PLArgs {
   int nx, ny, nz, ncells, noff, nftypes;
};

// One wavefront per reference cell.  Lanes take offsets; each lane counts
// the sites its neighbour cell contributes for the current frame type, a
// wave prefix sum places them, and (fill mode) they are written.  The
// cell-ordered arrays hold each cell's sites contiguously in the reference's
// list order (entries in linked-list order, a molecule's sites in order), so
// a neighbour cell's contribution is its run of corig, filtered by the frame
// flag when a framework is present.  Without a framework the lanes then take
// the 64 offsets' output entries 64 at a time: a bit per run start marks
// where each non-empty run begins, an entry's run is the count of starts up
// to it (v_mbcnt), and every store is a whole wave's consecutive entries.
constexpr int PL_NBW = 8;   // 64-bit start words per wave: up to 512 entries per 64 offsets
template <bool FILL>
static __global__ __launch_bounds__(256) void k_pairlist(PLArgs a, const int4 *__restrict__ off,
                                                         const int *__restrict__ css,
                                                         const int *__restrict__ corig,
                                                         const int2 *__restrict__ cmeta,
                                                         int *__restrict__ count,
                                                         const int *__restrict__ lstart,
                                                         int *__restrict__ nab, int *__restrict__ pbct,
                                                         int *__restrict__ nfnab) {
   __shared__ int2 srun[4][64];                       // (first site - first entry, image code) of each run
   __shared__ unsigned long long sbit[4][PL_NBW];     // run starts
   int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
   int c = blockIdx.x * 4 + w;
   if (c >= a.ncells) return;   // wave-uniform; the LDS below is the wave's own
   int ix = c / (a.ny * a.nz), iy = c / a.nz - a.ny * ix, iz = c - a.nz * (iy + a.ny * ix);
   int base = FILL ? lstart[c] : 0;
   int nn = 0;
   for (int ft = 0; ft < a.nftypes; ft++) {
      for (int o0 = (ft == 0 ? 0 : 1); o0 < a.noff; o0 += 64) {
         int o = o0 + lane, cnt = 0, j0 = 0, j1 = 0, code = 0;
         if (o < a.noff) {
            int4 d = off[o];
            int ex = ix + d.x, ey = iy + d.y, ez = iz + d.z;
            int sx = ex < 0 ? -1 : (ex >= a.nx ? 1 : 0);
            int sy = ey < 0 ? -1 : (ey >= a.ny ? 1 : 0);
            int sz = ez < 0 ? -1 : (ez >= a.nz ? 1 : 0);
            int jc = (ez - sz * a.nz) + a.nz * ((ey - sy * a.ny) + a.ny * (ex - sx * a.nx));
            code = 9 * (sx + 1) + 3 * (sy + 1) + (sz + 1);
            j0 = css[jc];
            j1 = css[jc + 1];
            if (a.nftypes == 1) {
               cnt = j1 - j0;
            } else {
               for (int j = j0; j < j1; j++) cnt += (cmeta[j].x >> 8) == ft;
            }
         }
         int inc = wave_incl_scan(cnt, lane);
         const int tot = __shfl(inc, 63, 64);
         if (FILL && a.nftypes == 1 && tot <= 64 * PL_NBW) {
            const int st = inc - cnt;
            if (lane < PL_NBW) sbit[w][lane] = 0;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            const unsigned long long ne = __ballot(cnt > 0);
            if (cnt > 0) {
               const int rank = __builtin_amdgcn_mbcnt_hi((unsigned)(ne >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)ne, 0));
               srun[w][rank] = make_int2(j0 - st, code);
               atomicOr(&sbit[w][st >> 6], 1ull << (st & 63));
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            // run of entry q = starts at or before q, less one (the first
            // non-empty run starts at 0; bits past tot are clear)
            int nst = 0;
            for (int q0 = 0; q0 < tot; q0 += 64) {
               const unsigned long long bw = sbit[w][q0 >> 6];
               const int below = __builtin_amdgcn_mbcnt_hi((unsigned)(bw >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)bw, 0));
               const int k = nst + below + (int)((bw >> lane) & 1ull) - 1;
               nst += __popcll(bw);
               const int q = q0 + lane;
               if (q < tot) {
                  const int2 rd = srun[w][k];
                  nab[base + nn + q] = corig[q + rd.x];
                  pbct[base + nn + q] = rd.y;
               }
            }
            // the next offsets' writes to srun/sbit come after these reads
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
         } else if (FILL && cnt) {
            int p = base + nn + inc - cnt;
            for (int j = j0; j < j1; j++) {
               if (a.nftypes != 1 && (cmeta[j].x >> 8) != ft) continue;
               nab[p] = corig[j];
               pbct[p] = code;
               p++;
            }
         }
         nn += tot;
      }
      if (FILL && lane == 0) nfnab[2 * c + ft] = nn;
   }
   if (FILL && lane == 0 && a.nftypes == 1) nfnab[2 * c + 1] = nn;
   if (!FILL && lane == 0) count[c] = nn;
}

void mgpu::run_pairlist_count(mgpu_engine *e, int, double, const int *offs, int noff,
                              long *total, long *list_start_host) {
   std::vector<int4> h(noff);
   for (int i = 0; i < noff; i++) h[i] = make_int4(offs[3 * i], offs[3 * i + 1], offs[3 * i + 2], 0);
   e->d_off_pl.reserve(noff + 1);
   HIPCHK(hipMemcpyAsync(e->d_off_pl.p, h.data(), sizeof(int4) * noff, hipMemcpyHostToDevice, e->stream));
   int nc = e->ncells;
   e->d_pl_count.reserve(nc + 1);
   e->d_pl_start.reserve(nc + 1);
   PLArgs a{e->nx, e->ny, e->nz, nc, noff, e->n_frame_types};
   {
      ProfScope ps(e, "pairlist_count");
      k_pairlist<false><<<(nc + 3) / 4, 256, 0, e->stream>>>(a, e->d_off_pl.p, e->d_cell_site_start.p,
                                                             e->d_corig.p, e->d_cmeta.p, e->d_pl_count.p,
                                                             nullptr, nullptr, nullptr, nullptr);
      device_scan_int(e, e->d_pl_count.p, e->d_pl_start.p, nc);
   }
   std::vector<int> hs(nc + 1);
   HIPCHK(hipMemcpyAsync(hs.data(), e->d_pl_start.p, sizeof(int) * (nc + 1), hipMemcpyDeviceToHost, e->stream));
   HIPCHK(hipStreamSynchronize(e->stream));
   for (int i = 0; i <= nc; i++) list_start_host[i] = hs[i];
   *total = hs[nc];
}

void mgpu::run_pairlist_fill(mgpu_engine *e, const int *, int noff, long total, int *nab,
                             int *pbctrans, int *nfnab) {
   run_pairlist_fill_device(e, noff, total);
   int nc = e->ncells;
   if (nab) HIPCHK(hipMemcpyAsync(nab, e->d_pl_nab.p, sizeof(int) * total, hipMemcpyDeviceToHost, e->stream));
   if (pbctrans)
      HIPCHK(hipMemcpyAsync(pbctrans, e->d_pl_pbc.p, sizeof(int) * total, hipMemcpyDeviceToHost, e->stream));
   if (nfnab)
      HIPCHK(hipMemcpyAsync(nfnab, e->d_pl_nfnab.p, sizeof(int) * 2 * nc, hipMemcpyDeviceToHost, e->stream));
   HIPCHK(hipStreamSynchronize(e->stream));
}

// Site neighbour lists of every cell into engine buffers (CSR over cells by
// d_pl_start; counts from run_pairlist_count).
void mgpu::run_pairlist_fill_device(mgpu_engine *e, int noff, long total) {
   ProfScope ps(e, "pairlist_fill");
   int nc = e->ncells;
   e->d_pl_nab.reserve(total + 1);
   e->d_pl_pbc.reserve(total + 1);
   e->d_pl_nfnab.reserve(2 * (size_t)nc + 2);
   PLArgs a{e->nx, e->ny, e->nz, nc, noff, e->n_frame_types};
   k_pairlist<true><<<(nc + 3) / 4, 256, 0, e->stream>>>(a, e->d_off_pl.p, e->d_cell_site_start.p,
                                                         e->d_corig.p, e->d_cmeta.p, nullptr, e->d_pl_start.p,
                                                         e->d_pl_nab.p, e->d_pl_pbc.p, e->d_pl_nfnab.p);
}

// ------------------------------------------------- radial distributions
struct RdfArgs {
   int ncells, nbins, nb, max_id;
   double rbin;
   double reloc[81];
};

// rdf_inner (src/force.c:1010-1103) and rdf_accum (src/rdf.c:94-108): one
// wavefront per cell walks the cell's sites in list order with the
// reference's jmin/jmax rules, lanes take neighbours j, and every pair
// closer than limit counts once in hist[block(id_i, id_j)][bin].  The
// distance is formed in the reference's operation order without
// contraction, so bins are exact.
//
// A block counts in LDS (LDSH) and adds its non-zero bins to hist at its
// end; its waves take cells in strides of the grid.  Counting straight into
// hist, where the pairs meet in a few hundred words of L2, took 1.01 ms at
// 16,384 water sites (limit 8 A, 200 bins); this takes 0.07 ms.  Histograms past
// RDF_LDS_BINS counters still count in hist directly: they would leave room
// for one or two blocks on a CU, and their pairs meet less often.
constexpr int RDF_LDS_BINS = 12288;   // 48 KB: three blocks on a CU
#pragma clang fp contract(off)
template <bool LDSH>
static __global__ __launch_bounds__(256) void k_rdf(RdfArgs a, const int *__restrict__ c_start,
                                                    const int *__restrict__ c_entries,
                                                    const int *__restrict__ e_isite,
                                                    const int *__restrict__ e_num,
                                                    const int *__restrict__ e_ftype,
                                                    const int *__restrict__ lstart, const int *__restrict__ nab,
                                                    const int *__restrict__ pbct, const int *__restrict__ nfnab,
                                                    const int *__restrict__ stype, const int *__restrict__ blk,
                                                    const double *__restrict__ site, int nsp,
                                                    int *__restrict__ hist) {
   extern __shared__ int lhist[];
   const int lane = threadIdx.x & 63;
   if (LDSH) {
      for (int t = threadIdx.x; t < a.nb; t += 256) lhist[t] = 0;
      __syncthreads();
   }
   int *cnt = LDSH ? lhist : hist;
   for (int c = blockIdx.x * 4 + (threadIdx.x >> 6); c < a.ncells; c += gridDim.x * 4) {   // wave-uniform
      const int base = lstart[c], nnab = lstart[c + 1] - base, nf0 = nfnab[2 * c];
      int jmin = 0;
      for (int q = c_start[c]; q < c_start[c + 1]; q++) {
         const int en = c_entries[q], ft = e_ftype[en];
         int jmax;
         if (ft) {
            jmin = 0;
            jmax = nf0;
         } else {
            jmax = nnab;
         }
         const int i0 = e_isite[en], i1 = i0 + e_num[en];
         for (int i = i0; i < i1; i++) {
            if (!ft) jmin++;
            const double s0 = site[i], s1 = site[nsp + i], s2 = site[2 * nsp + i];
            const int *brow = blk + stype[i] * a.max_id;
            for (int j = jmin + lane; j < jmax; j += 64) {
               const int sj = nab[base + j], t = pbct[base + j];
               const double ax = site[sj] - s0 + a.reloc[3 * t];
               const double ay = site[nsp + sj] - s1 + a.reloc[3 * t + 1];
               const double az = site[2 * nsp + sj] - s2 + a.reloc[3 * t + 2];
               const double rsq = ax * ax + ay * ay + az * az;
               const int bin = (int)(a.rbin * sqrt(rsq));
               if (bin < a.nbins) atomicAdd(cnt + (size_t)brow[stype[sj]] * a.nbins + bin, 1);
            }
         }
      }
   }
   if (LDSH) {
      __syncthreads();
      for (int t = threadIdx.x; t < a.nb; t += 256)
         if (lhist[t]) atomicAdd(hist + t, lhist[t]);
   }
}

// n additions of r to x, each rounded as (float)((double)x + r).  Once a step
// starts and ends in one binade, every further step that ends in it adds the
// same multiple of its ulp: x is a multiple of the ulp, so r rounds to the
// ulp the same way each time (a tie too, as a step that ends in a tie leaves
// x even), and the steps up to the binade's end are taken at once.  About
// three single steps a binade are left: 0.009 ms, where the loop of n additions took
// 0.35 ms for bins of up to 2e5 counts.
static __device__ float repeat_add(float x, double r, int n) {
   while (n > 0) {
      const float y = (float)((double)x + r);
      n--;
      if (y == x) return y;   // further additions round back to y
      const unsigned bx = __float_as_uint(x), by = __float_as_uint(y);
      // positive normal numbers of one exponent, below infinity
      if (n > 0 && r > 0 && (bx >> 23) == (by >> 23) && by >= 0x00800000u && by < 0x7f000000u) {
         const float z = (float)((double)y + r);
         const double d = (double)z - (double)y;
         const double top = (double)__uint_as_float(((by >> 23) + 1) << 23);
         const double room = top - (double)y - r;
         if (room > 0 && d > 0) {
            const double q = floor(room / d);
            const int m = q < (double)n ? (int)q : n;
            x = (float)((double)y + (double)m * d);
            n -= m;
            continue;
         }
      }
      x = y;
   }
   return x;
}

// rdf_accum's float bins: n additions of 1/density to the float bin, each
// rounded as (float)(bin + invrho) the way the reference's loop rounds them.
static __global__ void k_rdf_float(int nb, double invrho, const int *__restrict__ hist,
                                   float *__restrict__ rdf) {
   int b = blockIdx.x * blockDim.x + threadIdx.x;
   if (b >= nb) return;
   rdf[b] = repeat_add(rdf[b], invrho, hist[b]);
}
#pragma clang fp contract(on)

void mgpu::run_rdf(mgpu_engine *e, double limit, int nbins, int noff, float *rdf_host) {
   const int nblk = (e->max_id - 1) * e->max_id / 2, nb = nblk * nbins;
   std::vector<int> blk((size_t)e->max_id * e->max_id, 0);
   for (int i = 1; i < e->max_id; i++)
      for (int j = 1; j < e->max_id; j++) {
         int lo = std::min(i, j), hi = std::max(i, j), k = 0;
         for (int t = 1; t < lo; t++) k += e->max_id - t;
         blk[(size_t)i * e->max_id + j] = k + (hi - lo);
      }
   e->d_rdf_blk.reserve(blk.size());
   e->d_rdf_hist.reserve(nb);
   e->d_rdf_bins.reserve(nb);
   HIPCHK(hipMemcpyAsync(e->d_rdf_blk.p, blk.data(), sizeof(int) * blk.size(), hipMemcpyHostToDevice, e->stream));
   HIPCHK(hipMemcpyAsync(e->d_rdf_bins.p, rdf_host, sizeof(float) * nb, hipMemcpyHostToDevice, e->stream));
   zero_async(e, e->d_rdf_hist.p, sizeof(int) * nb);
   RdfArgs a;
   a.ncells = e->ncells; a.nbins = nbins; a.nb = nb; a.max_id = e->max_id;
   a.rbin = nbins / limit;
   int k = 0;
   for (int ii = -1; ii <= 1; ii++)
      for (int jj = -1; jj <= 1; jj++)
         for (int kk = -1; kk <= 1; kk++, k++) {
            a.reloc[3 * k] = e->h[0] * ii + e->h[1] * jj + e->h[2] * kk;
            a.reloc[3 * k + 1] = e->h[3] * ii + e->h[4] * jj + e->h[5] * kk;
            a.reloc[3 * k + 2] = e->h[6] * ii + e->h[7] * jj + e->h[8] * kk;
         }
   (void)noff;
   {
      ProfScope ps(e, "rdf");
      auto run = [&](auto k, unsigned g, size_t shm) {
         k<<<g, 256, shm, e->stream>>>(a, e->d_cell_start.p, e->d_cell_entries.p, e->d_entry_isite.p, e->d_entry_num.p,
                                       e->d_entry_ftype.p, e->d_pl_start.p, e->d_pl_nab.p, e->d_pl_pbc.p,
                                       e->d_pl_nfnab.p, e->d_site_type.p, e->d_rdf_blk.p, e->d_site.p, e->nsp,
                                       e->d_rdf_hist.p);
      };
      const unsigned g = (e->ncells + 3) / 4;
      if (nb <= RDF_LDS_BINS) run(k_rdf<true>, std::min(g, 8u * e->ncu), sizeof(int) * nb);
      else run(k_rdf<false>, g, 0);
      const double invrho = 1.0 / (e->nsites / host_det(e->h));
      k_rdf_float<<<(nb + 255) / 256, 256, 0, e->stream>>>(nb, invrho, e->d_rdf_hist.p, e->d_rdf_bins.p);
   }
   HIPCHK(hipMemcpyAsync(rdf_host, e->d_rdf_bins.p, sizeof(float) * nb, hipMemcpyDeviceToHost, e->stream));
   HIPCHK(hipStreamSynchronize(e->stream));
}
