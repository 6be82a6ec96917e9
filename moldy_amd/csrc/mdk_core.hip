// mdk_core.hip -- libmoldy_hip: MOLDY's Fe force hot path on MI355X (gfx950).
//
// Device design (one system per handle, one HIP stream):
//  * per-atom state is FP64 SoA, kept SORTED BY CELL of a fine grid (cell
//    width >= interaction range + skin) so that neighbour gathers are local;
//    the sort is redone at every full-list rebuild.  slot_of/orig map between
//    the reference's atom order and the device order.
//  * the force path uses a FULL neighbour list (both directions) pruned at
//    r_int + skin, r_int = 3.72645 A being the outermost knot beyond which
//    V, V', phi and phi' are identically zero; per-atom sums are gathers (no
//    atomics, deterministic).  It is rebuilt on the reference's ntcm cadence
//    and whenever an atom may have moved more than skin/2.
//  * the reference half list at rnear (NLIST/NUMN) is built on request by a
//    separate kernel that reproduces the reference's link-cell grid, stencil
//    and bit-exact distance test.
//  * reductions (energies, virial, kinetic tensor, thermodynamic sums) are
//    per-block partials reduced in a fixed order by a finishing block: of its
//    own kernel, of the kick's, or an extra one of the next density pass.
//  * box/thermo tensors live on the device (BoxState, four copies in turn) so an
//    MD step needs no host round trip.
//  * systems of different sizes take different forms of list and passes: several
//    lanes per atom and few launches where latency counts, partners staged in LDS
//    where the gathers do.
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>
#include <limits.h>
#include <math.h>
#include <stdarg.h>
#include <stddef.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <string>
#include <vector>

#include "../../include/moldy_hip.h"
#include "mdk_brick.h"
#include "mdk_internal.h"
#include "mdk_wave.h"

// ---------------------------------------------------------------------------
// error handling
// ---------------------------------------------------------------------------
static thread_local char g_err[512] = "";
static int set_err(int code, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}
extern "C" const char *mdk_last_error(void) { return g_err; }

#define HIPCK(call)                                                                    \
  do {                                                                                 \
    hipError_t e_ = (call);                                                            \
    if (e_ != hipSuccess)                                                              \
      return set_err(MDK_ERR_HIP, "%s failed: %s (%s:%d)", #call, hipGetErrorString(e_), \
                     __FILE__, __LINE__);                                              \
  } while (0)
#define RCK(expr)          \
  do {                     \
    int r_ = (expr);       \
    if (r_ != MDK_OK) return r_; \
  } while (0)

#include "mdk_hostpot.h"

// ---------------------------------------------------------------------------
// context
// ---------------------------------------------------------------------------
enum {
  F_X0 = 0, F_Y0, F_Z0, F_X1, F_Y1, F_Z1, F_X2, F_Y2, F_Z2, F_FX, F_FY, F_FZ,
  F_RHO, F_AFRHO, F_DAFRHO, F_MASS, F_DEL2, F_X3, F_Y3, F_Z3, F_N
};

struct TimedEv {
  int cls;
  hipEvent_t a, b;
};

// monitor sample: [0] max squared displacement since the list was built,
// [1] max squared displacement of the next drift, then B0, b1 + b2 (the next
// drift's box change) and Bref (B0 at the list build), 9 each; [MON_STAMP] the
// step's stamp, written last (the host waits for it)
#define MON_STRIDE 32
#define MON_B0 2
#define MON_DB 11
#define MON_BREF 20
#define MON_STAMP 31
#define MDK_NSPEC 128  // species (atomic numbers) covered by the mass/del2 table

// list grid for cell-relative packing (gx == 0: absolute packing)
struct PackGeo {
  int gx, gy, gz;
  double ix, iy, iz;  // 1/g
};

// the reference's link cells, and where the atoms' go (ic null: not asked for)
struct LinkGrid {
  int nx, ny, nz;
  int *ic;
};

// Arguments of a step's finishing (k_finish_step, or deferred to the next
// density pass).
struct FinKick {
  BoxState *bs;
  BoxState *bout;  // the advanced copy of a fused drift: receives the same sums
  double *trace_row, *mon;
  double dt, bdel2, press, stamp;  // stamp: of the monitor sample (step index + 1)
};
// A deferred finishing: kind 1 the half kick's partials (NPART_KICK columns of
// nb), 2 those of a force pass fused with the kick (NPART_FIXED columns) and
// the embedding energies (nbe)
struct FinRide {
  int kind, nb, nbe;
  const double *part, *emb;
  FinKick kick;
};
// Flags of a deferred list build, copied to host-mapped memory with the build's
// stamp behind them (stamp 0: nothing to report).
struct ListReport {
  const int *flags;
  int *out, stamp;
};
// What a density pass does besides, in workgroups of its own
struct Rider {
  FinRide fin;
  ListReport list;
  int one_xcd;  // the pass's placement (place_of)
};

struct mdk_ctx {
  mdk_params p;
  int n;
  int pbc;                 // periodic dims mask from ivol (bit0 x, bit1 y, bit2 z)
  int device;
  hipStream_t stream;
  // per-atom state (sorted order): F_N doubles per atom, field-major
  double *atoms, *atoms_alt;
  int *zat, *zat_alt, *orig, *orig_alt, *slot_of;
  float *sref;             // fractional positions at the last full-list build
  double4 *pos4;           // packed positions (absolute or cell-relative) and F' for the pair kernels
  double4 *pos4_alt;       // the next step's, written by a force pass fused with the kick (fixed boxes)
  float4 *p4f_alt;
  int *img;                // integer image floor(s) fixed at the last full-list build
  bool pos4_valid;         // pos4 (and p4f) match the positions and box
  bool p4f_valid;          // p4f matches them (the FP32 lean passes read only p4f)
  bool masschk;            // some atom has mass <= 0.05: keep the per-pair mass test
  // mass and del2 as functions of the species when every atom of a species
  // carries the same values: spec_tab[2 z], spec_tab[2 z + 1] (device), used
  // by the kick and kinten instead of the per-atom fields; host copies of the
  // uploads (reference order) decide it
  double *spec_tab;
  bool spec_ok;
  double *h_mass, *h_del2;
  int *h_z;
  // reference link cells (1-based cell per atom, sorted order)
  int *ic;
  // parity half list in reference layout: numn_ref[nm] and nlist_ref[nm*nnbrs] (orig order)
  int *numn_ref, *nlist_ref;
  // full list
  int maxn;
  int *nbr, *numn;
  int *nact;  // per atom: list slots the force pass visits (set by the density pass)
  bool rel;     // positions packed cell-relative (block list) rather than absolute
  float4 *p4f;  // FP32 copy of the packed positions (FP32 form only)
  bool part_due;  // the next density pass reorders the new list (in-range partners first)
  int *cell_of, *cell_alt, *ic_alt;
  // counting sort: cell_count is zero between sorts (the scan clears it)
  int *cell_count, *cell_start, *cell_fill, *cell_btot, *members;
  int ncell_cap;
  int grid[3];
  int *dflags;             // [0] full-list overflow, [1] half-list overflow, [2] grid too coarse
  // list-kernel flags copied to host-mapped memory after a deferred build
  // ([0..3]), then the build's stamp ([4]), which the host waits for
  int *flags_host, *flags_map, list_stamp;
  bool list_pending;       // a deferred build whose flags the host has not checked yet
  bool report_due;         // ... and no density pass has been asked to report
  // cubes of 2 or 4 cells a side of the list build (lowest Morton key / cells),
  // for grid lblock_g and side lblock_side
  int *lblocks, nlblocks, lblocks_cap, lblock_g[3], lblock_side;
  // brick list (k_brick_list): its entries and their quads per atom, staged atoms
  // and extents of every brick
  bool brick, brick_bad;   // the list is one; bricks did not fit lately
  int brick_wait;          // lists planned since then
  bool brick_built;        // nbr16, bcnt, bstage and binfo hold a built list
  bool wide_valid;         // nbr, numn hold the brick list's pairs as well (ensure_wide_list)
  uint2 *nbr16;
  int *bcnt, *bstage;
  int4 *binfo;
  int brick_k;             // 2^k units of the staged positions per A
  int brick_cap, brick_nt; // staged atoms per brick, threads of its workgroup
  size_t bstage_cap, binfo_cap;
  long rebuilds;
  bool list_valid;
  bool half_valid;         // numn_ref/nlist_ref hold a reference half list
  bool x3_live;            // X3..Z3 may be non-zero (uploaded, or the predictor-corrector ran)
  // a step whose sums the next density pass completes (kind 0: none)
  FinRide ride;
  // reference link-cell chains (src/linkcell_m.F90:122-274) on the host in
  // reference atom order, 1-based: L0 per cell, LINK, IC; chains_exact is
  // false after relinks inside mdk_md_steps, which update only the device ic
  int *h_l0, *h_link, *h_ic, h_ncell;
  bool chains_exact;
  int *ref_key, *rank_orig, *rank_slot;  // device: cell keys and chain ranks
  int last_rebuild_step;
  // box state: four copies in turn (a step reads one and writes the next one or
  // two; the deferred half-kick sums still go to the last step's)
  BoxState *box;
  int cur;
  // partials
  // per-block partials, value-major: the force pass (also the fixed-box kick's),
  // the embedding energy and kinten (two buffers each: a kernel may read one
  // step's while it writes the next) and the half kick
  double *part_f, *emb2, *kin2, *part_k;
  char *small;                // the allocation of the partials and other small arrays
  int emb_slot, kin_slot;     // buffers that hold the current partials, and their blocks
  int emb_nb, kin_nb;
  double *stage_f, *stage_k;  // first-stage reductions of force()'s and scalev's partials
  unsigned *fin_cnt;          // arrival counters of k_finalize_force and k_fold, zeroed
  int nblk;
  int lanes, nbp;          // lanes per atom of the pair passes (pair_lanes) and their blocks
  int part_cap;            // blocks the partial arrays hold
  // host-mapped monitor ring: four step slots of MON_STRIDE doubles (layout there)
  double *mon_host, *mon_dev;
  double b0_lag[9];        // B0 of a completed step (from the monitor ring)
  long b0_lag_step;        // its step index, -1 when none
  bool drifted;            // the next step's drift was fused into the last kick
  bool kin_fresh;          // kinten's partial sums match the velocities and box of the next force
  long step_counter;
  // trace buffer on device
  double *trace_dev;
  int trace_cap;
  // potential
  PotDev pot;
  bool pot_set;
  double *tabs;
  float *fetab;   // interval table of the FP32 Fe-Fe pair terms (MDK_FE_TAB floats)
  bool fe_ok;     // fetab holds the current knots' table
  hostpot::Knots knots;
  int material;            // MDK_MAT_*: fetransmetal (knots) or iron_carbon (fec)
  int iverlet;             // md_steps integrator: 1 velocity Verlet, 0 predictor-corrector
  bool pc_primed;          // a correc or velocityverlet has run (predic is live)
  double snhv;             // Nose-Hoover velocity scaling accumulated by scalev
  double *red;             // 4 doubles: results of the scalev folds
  hostpot::FecCoef fec;
  double r_int_exact;      // interaction range of the exact functions
  // reference list threshold: r < rnear  <=>  r^2 < rnear2_exact (see near_threshold)
  double rnear2_exact;
  double r_list, skin;
  int ntc;
  // timing
  int timing_mask;          // kernel classes recorded with HIP events
  int timing_every;         // record one launch in this many per class
  long t_seen[TC_NCLASS];
  std::vector<TimedEv> evs;
  std::vector<hipEvent_t> evpool;
  double t_ms[TC_NCLASS];
  long t_cnt[TC_NCLASS];
  bool linked;
};

static inline double *fld(double *base, int f, int n) { return base + (size_t)f * n; }
static inline double *emb_buf(const mdk_ctx *c, int s) { return c->emb2 + (size_t)s * c->part_cap; }
static inline double *kin_buf(const mdk_ctx *c, int s) { return c->kin2 + (size_t)s * c->part_cap * NPART_KIN; }
static inline LinkGrid link_grid(const mdk_ctx *c, bool want) {
  return LinkGrid{c->p.nlcx, c->p.nlcy, c->p.nlcz, want ? c->ic : nullptr};
}
static inline int next_box(const mdk_ctx *c, int k = 1) { return (c->cur + k) & 3; }
static inline PackGeo pack_geo(const mdk_ctx *c) {
  PackGeo pg = {0, 0, 0, 0.0, 0.0, 0.0};
  if (c->rel) {
    pg.gx = c->grid[0]; pg.gy = c->grid[1]; pg.gz = c->grid[2];
    pg.ix = 1.0 / pg.gx; pg.iy = 1.0 / pg.gy; pg.iz = 1.0 / pg.gz;
  }
  return pg;
}
static inline float4 *p4f_of(const mdk_ctx *c) { return c->p.precision == MDK_PREC_FP32 ? c->p4f : nullptr; }
// the (mass, del2) species table when it holds, else the per-atom fields
static inline const double *spec_of(const mdk_ctx *c) { return c->spec_ok ? c->spec_tab : nullptr; }

// ---------------------------------------------------------------------------
// device helpers
// ---------------------------------------------------------------------------

// Block-reduce K sums (and the last KM entries as maxima) into
// part[k nb + b], block b of nb (value-major, so the finishing block's reads
// of one value across all blocks are contiguous).
template <int K, int KM, int BLOCK = MDK_BLOCK>
__device__ __forceinline__ void block_store(double (&v)[K], double *part, int nb, int b) {
  __shared__ double sh[BLOCK / 64][K];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  wave_reduce_all<K, KM>(v);
  if (lane == 0) {
#pragma unroll
    for (int k = 0; k < K; k++) sh[w][k] = v[k];
  }
  __syncthreads();
  if (threadIdx.x < K) {
    const int k = threadIdx.x;
    double s = sh[0][k];
    for (int q = 1; q < BLOCK / 64; q++) s = (k < K - KM) ? s + sh[q][k] : fmax(s, sh[q][k]);
    part[(size_t)k * nb + b] = s;
  }
}
template <int K, int KM, int BLOCK = MDK_BLOCK>
__device__ __forceinline__ void block_store(double (&v)[K], double *part) {
  block_store<K, KM, BLOCK>(v, part, gridDim.x, blockIdx.x);
}

// kinten's terms of one atom (src/thermostat_m.F90:127-177): tk(a,b) += m
// (B0 x1)_a x1_b, column-major in v[0..8], with B0 the box of the force
// evaluation the velocities x1 belong to
__device__ __forceinline__ void kin_terms(const double *b, double a1, double a2, double a3, double mi,
                                          double (&v)[9]) {
#pragma clang fp contract(off)  // the same rounding in every kernel that calls it
  const double mvx = (b[0] * a1 + b[3] * a2 + b[6] * a3) * mi;
  const double mvy = (b[1] * a1 + b[4] * a2 + b[7] * a3) * mi;
  const double mvz = (b[2] * a1 + b[5] * a2 + b[8] * a3) * mi;
  v[0] = a1 * mvx; v[1] = a1 * mvy; v[2] = a1 * mvz;
  v[3] = a2 * mvx; v[4] = a2 * mvy; v[5] = a2 * mvz;
  v[6] = a3 * mvx; v[7] = a3 * mvy; v[8] = a3 * mvz;
}

// XCD-aware tile order.  Workgroups are dispatched round-robin over the 8
// XCDs, each with its own L2; remapping physical block b to logical tile
// start(b%8) + b/8 gives every XCD one contiguous range of (cell-sorted)
// atoms, so its neighbour gathers stay inside its own L2.
#define MDK_NXCD 8
__device__ __forceinline__ int xcd_tile(int nb, int b) {
  const int q = nb / MDK_NXCD, r = nb % MDK_NXCD, x = b % MDK_NXCD;
  return x * q + min(x, r) + b / MDK_NXCD;
}
__device__ __forceinline__ int xcd_tile() { return xcd_tile(gridDim.x, blockIdx.x); }

// Placement of a pass: its workgroups nb and this one's index b among them.  The
// smallest systems keep to one XCD: workgroups go to the XCDs in turn, so with
// MDK_NXCD times as many the first of every MDK_NXCD share one and the others leave
// at once (idle).  What a pass leaves in that XCD's L2 is then there for the next,
// which would have to fetch it from memory on another.  Up to a workgroup per CU
// (ONE_XCD_BLOCKS); us per step, all XCDs : one -- 250 atoms NVE 14.4 : 13.6, NPT 19.1
// : 17.9, iron_carbon 29.5 : 27.6; 1024 atoms 14.6 : 13.8, 19.1 : 18.2, 26.0 : 25.0;
// 2000 atoms (63 workgroups) 13.6 : 13.9, 18.7 : 19.0, 25.4 : 26.4.
#define ONE_XCD_BLOCKS 32
struct Place {
  int nb, b;
  bool idle;
};
__device__ __forceinline__ Place place_of(int grid, int block, int one_xcd) {
  if (!one_xcd) return {grid, block, false};
  return {grid / MDK_NXCD, block / MDK_NXCD, block % MDK_NXCD != 0};
}

__device__ __forceinline__ void min_image(int pbc, double &dx, double &dy, double &dz) {
  if (pbc & 1) dx = dx - round(dx);
  if (pbc & 2) dy = dy - round(dy);
  if (pbc & 4) dz = dz - round(dz);
}

// Reference-order Cartesian separation squared (src/parrinellorahman_m.F90:167-172),
// no FMA: bit-identical to the reference's r*r before the square root.
__device__ __forceinline__ double sep2_exact(const double *b, double dx, double dy, double dz) {
#pragma clang fp contract(off)
  const double rx = b[0] * dx + b[3] * dy + b[6] * dz;
  const double ry = b[1] * dx + b[4] * dy + b[7] * dz;
  const double rz = b[2] * dx + b[5] * dy + b[8] * dz;
  return rx * rx + ry * ry + rz * rz;
}

// 3x3 helpers on column-major arrays (device, one thread)
__device__ void dev_invert(const double *a, double *b, int *status) {
#pragma clang fp contract(off)
  double det = TT(a, 1, 1) * (TT(a, 2, 2) * TT(a, 3, 3) - TT(a, 2, 3) * TT(a, 3, 2));
  det = det + TT(a, 2, 1) * (TT(a, 3, 2) * TT(a, 1, 3) - TT(a, 1, 2) * TT(a, 3, 3));
  det = det + TT(a, 3, 1) * (TT(a, 1, 2) * TT(a, 2, 3) - TT(a, 1, 3) * TT(a, 2, 2));
  TT(b, 1, 1) = TT(a, 2, 2) * TT(a, 3, 3) - TT(a, 2, 3) * TT(a, 3, 2);
  TT(b, 1, 2) = TT(a, 3, 1) * TT(a, 2, 3) - TT(a, 2, 1) * TT(a, 3, 3);
  TT(b, 1, 3) = TT(a, 2, 1) * TT(a, 3, 2) - TT(a, 3, 1) * TT(a, 2, 2);
  TT(b, 2, 1) = TT(a, 3, 2) * TT(a, 1, 3) - TT(a, 1, 2) * TT(a, 3, 3);
  TT(b, 2, 2) = TT(a, 1, 1) * TT(a, 3, 3) - TT(a, 1, 3) * TT(a, 3, 1);
  TT(b, 2, 3) = TT(a, 3, 1) * TT(a, 1, 2) - TT(a, 1, 1) * TT(a, 3, 2);
  TT(b, 3, 1) = TT(a, 1, 2) * TT(a, 2, 3) - TT(a, 1, 3) * TT(a, 2, 2);
  TT(b, 3, 2) = TT(a, 2, 1) * TT(a, 1, 3) - TT(a, 2, 3) * TT(a, 1, 1);
  TT(b, 3, 3) = TT(a, 1, 1) * TT(a, 2, 2) - TT(a, 1, 2) * TT(a, 2, 1);
  if (fabs(det) == 0.0) {
    *status = MDK_ERR_SINGULAR_BOX;
    return;
  }
  for (int k = 0; k < 9; k++) b[k] = b[k] / det;
}
__device__ void dev_matmul(const double *a, const double *b, double *c) {
#pragma clang fp contract(off)
  for (int i = 1; i <= 3; i++) {
    for (int j = 1; j <= 3; j++) TT(c, i, j) = 0.0;
    for (int k = 1; k <= 3; k++)
      for (int j = 1; j <= 3; j++) TT(c, i, j) = TT(c, i, j) + TT(a, i, k) * TT(b, k, j);
  }
}
__device__ double dev_volume(const double *b) {
#pragma clang fp contract(off)
  return TT(b, 1, 1) * (TT(b, 2, 2) * TT(b, 3, 3) - TT(b, 2, 3) * TT(b, 3, 2)) +
         TT(b, 2, 1) * (TT(b, 3, 2) * TT(b, 1, 3) - TT(b, 1, 2) * TT(b, 3, 3)) +
         TT(b, 3, 1) * (TT(b, 1, 2) * TT(b, 2, 3) - TT(b, 2, 2) * TT(b, 1, 3));
}


// A neighbour entry of nbr[] is j | code << 27.  The pair separation is
// r_ij = R_i - R_j + D[code] with R the packed positions (pos4):
//  * absolute packing (legacy list, any box): R = B0 (s - img) with the integer
//    image img fixed at the last rebuild, code = image shift (sx+1) + 3 (sy+1)
//    + 9 (sz+1) with s in {-1,0,1}^3, D = B0 (sx, sy, sz);
//  * cell-relative packing (block list): R = B0 (s - img - f) with f the
//    fractional centre of the atom's list cell, code = offset (dx+1) + 3 (dy+1)
//    + 9 (dz+1) of j's list cell (unwrapped) from i's, D = -B0 (dx/gx, dy/gy,
//    dz/gz).  |R| stays below a cell width, so an FP32 copy of R loses little
//    and one 16-byte gather carries a partner in the FP32 form.
// Codes 27..31 place the partner 1e6 A away: null entries that pad quads.
#define NBR_IDX_MASK 0x07FFFFFF
#define NBR_CODE_SHIFT 27
// Neighbour k of atom i lives at nbr[((k/4) n + i) 4 + k%4]: four consecutive
// entries of one atom form one 16-byte load, and consecutive atoms' quads are
// contiguous (coalesced dwordx4 loads).
__device__ __forceinline__ size_t nbr_at(int k, int i, int n) {
  return (((size_t)(k >> 2) * n + i) << 2) + (k & 3);
}
#define NBR_NULL_CODE 31
__device__ __forceinline__ void shift_table(const double *b, PackGeo pg, double (*S)[3]) {
  for (int c = threadIdx.x; c < 32; c += blockDim.x) {
    if (c >= 27) {
      S[c][0] = 1.0e6;
      S[c][1] = 0.0;
      S[c][2] = 0.0;
      continue;
    }
    double sx = (double)(c % 3 - 1), sy = (double)((c / 3) % 3 - 1), sz = (double)(c / 9 - 1);
    if (pg.gx) {
      sx = -sx * pg.ix;
      sy = -sy * pg.iy;
      sz = -sz * pg.iz;
    }
    S[c][0] = b[0] * sx + b[3] * sy + b[6] * sz;
    S[c][1] = b[1] * sx + b[4] * sy + b[7] * sz;
    S[c][2] = b[2] * sx + b[5] * sy + b[8] * sz;
  }
}
// inverse of a 3x3 column-major matrix (cofactors / determinant)
__device__ __forceinline__ void inv3(const double *b, double *bi) {
  const double c00 = TT(b, 2, 2) * TT(b, 3, 3) - TT(b, 2, 3) * TT(b, 3, 2);
  const double c01 = TT(b, 2, 3) * TT(b, 3, 1) - TT(b, 2, 1) * TT(b, 3, 3);
  const double c02 = TT(b, 2, 1) * TT(b, 3, 2) - TT(b, 2, 2) * TT(b, 3, 1);
  const double det = TT(b, 1, 1) * c00 + TT(b, 1, 2) * c01 + TT(b, 1, 3) * c02;
  const double id = 1.0 / det;
  TT(bi, 1, 1) = c00 * id;
  TT(bi, 2, 1) = c01 * id;
  TT(bi, 3, 1) = c02 * id;
  TT(bi, 1, 2) = (TT(b, 1, 3) * TT(b, 3, 2) - TT(b, 1, 2) * TT(b, 3, 3)) * id;
  TT(bi, 2, 2) = (TT(b, 1, 1) * TT(b, 3, 3) - TT(b, 1, 3) * TT(b, 3, 1)) * id;
  TT(bi, 3, 2) = (TT(b, 1, 2) * TT(b, 3, 1) - TT(b, 1, 1) * TT(b, 3, 2)) * id;
  TT(bi, 1, 3) = (TT(b, 1, 2) * TT(b, 2, 3) - TT(b, 1, 3) * TT(b, 2, 2)) * id;
  TT(bi, 2, 3) = (TT(b, 1, 3) * TT(b, 2, 1) - TT(b, 1, 1) * TT(b, 2, 3)) * id;
  TT(bi, 3, 3) = (TT(b, 1, 1) * TT(b, 2, 2) - TT(b, 1, 2) * TT(b, 2, 1)) * id;
}

// ---------------------------------------------------------------------------
// permutation / transfer kernels
// ---------------------------------------------------------------------------
__global__ void k_scatter_d(double *dst, const double *src, const int *slot_of, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[slot_of[i]] = src[i];
}
__global__ void k_gather_d(double *dst, const double *src, const int *slot_of, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[slot_of[i]];
}
__global__ void k_scatter_i(int *dst, const int *src, const int *slot_of, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[slot_of[i]] = src[i];
}
__global__ void k_gather_i(int *dst, const int *src, const int *slot_of, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[slot_of[i]];
}
__global__ void k_zero(double *a, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) a[i] = 0.0;
}
__global__ void k_iota(int *a, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) a[i] = i;
}
// ---------------------------------------------------------------------------
// cells: counting sort helpers
// ---------------------------------------------------------------------------
// Runs of equal keys within a wave (atoms arrive nearly sorted by cell): every
// lane learns its run's head lane and length, and only heads touch the
// counters, once per run.  Lanes past n form their own runs and are skipped.
struct KeyRun {
  int key, head, len;
  bool is_head;
};
__device__ __forceinline__ KeyRun key_run(int k) {  // k: the lane's key, -1 past n
  const int lane = threadIdx.x & 63;
  const int prev = __shfl_up(k, 1, 64);
  const bool head = lane == 0 || prev != k;
  const unsigned long long heads = __ballot(head);
  const unsigned long long above = lane == 63 ? 0ull : heads >> (lane + 1);
  const unsigned long long upto = lane == 63 ? heads : heads & ((2ull << lane) - 1ull);
  KeyRun r;
  r.key = k;
  r.is_head = head;
  r.len = above ? __builtin_ctzll(above) + 1 : 64 - lane;
  r.head = 63 - __builtin_clzll(upto);
  return r;
}
__global__ void k_count(const int *key, int n, int *count) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const KeyRun r = key_run(i < n ? key[i] : -1);
  if (r.is_head && r.key >= 0) atomicAdd(&count[r.key], r.len);
}
// exclusive scan of count[0..m) into start[0..m] (start[m] = total), clearing
// count for the next sort and fill for k_fill: one workgroup up to
// SCAN_ONE keys (a launch costs more than its eight keys per thread), else
// three passes: per-block scans of SCAN_CHUNK elements, a scan of the block
// totals, and the add-back.
#define SCAN_CHUNK 2048
#define SCAN_ONE 8192
__device__ __forceinline__ int block_exclusive_scan_1024(int v, int *sh, int &total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int inc = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int u = __shfl_up(inc, o, 64);
    if (lane >= o) inc += u;
  }
  if (lane == 63) sh[w] = inc;
  __syncthreads();
  int before = 0;
  total = 0;
#pragma unroll
  for (int q = 0; q < 16; q++) {
    const int x = sh[q];
    before += q < w ? x : 0;
    total += x;
  }
  __syncthreads();
  return before + inc - v;
}
__global__ void __launch_bounds__(1024) k_scan_one(int *count, int *start, int *fill, int m) {
  __shared__ int sh[16];
  const int per = (m + 1023) / 1024, b0 = min(m, (int)threadIdx.x * per), b1 = min(m, b0 + per);
  int c[SCAN_ONE / 1024], s = 0;
#pragma unroll
  for (int q = 0; q < SCAN_ONE / 1024; q++) {
    c[q] = b0 + q < b1 ? count[b0 + q] : 0;
    s += c[q];
  }
  int total, ex = block_exclusive_scan_1024(s, sh, total);
#pragma unroll
  for (int q = 0; q < SCAN_ONE / 1024; q++) {
    if (b0 + q < b1) {
      start[b0 + q] = ex;
      count[b0 + q] = 0;
      fill[b0 + q] = 0;
    }
    ex += c[q];
  }
  if (threadIdx.x == 0) start[m] = total;
}
__global__ void __launch_bounds__(1024) k_scan_a(int *count, int *start, int *fill, int *btot, int m) {
  __shared__ int sh[16];
  const int base = blockIdx.x * SCAN_CHUNK + 2 * threadIdx.x;
  const int c0 = base < m ? count[base] : 0, c1 = base + 1 < m ? count[base + 1] : 0;
  int total;
  const int ex = block_exclusive_scan_1024(c0 + c1, sh, total);
  if (base < m) {
    start[base] = ex;
    count[base] = 0;
    fill[base] = 0;
  }
  if (base + 1 < m) {
    start[base + 1] = ex + c0;
    count[base + 1] = 0;
    fill[base + 1] = 0;
  }
  if (threadIdx.x == 0) btot[blockIdx.x] = total;
}
__global__ void __launch_bounds__(1024) k_scan_b(int *btot, int nb, int *start, int m) {
  __shared__ int sh[16];
  int run = 0;
  for (int b0 = 0; b0 < nb; b0 += 1024) {
    int t = b0 + threadIdx.x;
    int v = t < nb ? btot[t] : 0;
    int total;
    int ex = block_exclusive_scan_1024(v, sh, total);
    if (t < nb) btot[t] = run + ex;
    run += total;
  }
  if (threadIdx.x == 0) start[m] = run;
}
__global__ void k_scan_c(int *start, const int *btot, int m) {
  int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < m) start[k] += btot[k / SCAN_CHUNK];
}
__global__ void k_fill(const int *key, int n, const int *start, int *fill, int *members) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const KeyRun r = key_run(i < n ? key[i] : -1);
  int base = 0;
  if (r.is_head && r.key >= 0) base = start[r.key] + atomicAdd(&fill[r.key], r.len);
  base = __shfl(base, r.head, 64);  // the run's slots follow its head's reservation
  if (i < n) members[base + ((int)(threadIdx.x & 63) - r.head)] = i;
}
// deterministic order inside each cell: ascending sort key (key[members] or members)
__global__ void k_sort_cells(const int *start, int m, int *members, const int *key) {
  int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= m) return;
  int b = start[c], e = start[c + 1];
  for (int i = b + 1; i < e; i++) {
    int v = members[i];
    int kv = key ? key[v] : v;
    int j = i - 1;
    while (j >= b) {
      int u = members[j];
      int ku = key ? key[u] : u;
      if (ku <= kv) break;
      members[j + 1] = u;
      j--;
    }
    members[j + 1] = v;
  }
}

// reference link cell of an atom (src/linkcell_m.F90:149-153), 1-based
__device__ __forceinline__ void put_link_cell(const LinkGrid &G, int i, double x, double y, double z) {
#pragma clang fp contract(off)
  const double hm = 0.4999999999;
  int ix = (int)((x - round(x) + hm) * (double)G.nx);
  int iy = (int)((y - round(y) + hm) * (double)G.ny);
  int iz = (int)((z - round(z) + hm) * (double)G.nz);
  // the reference's range is [0, nlc-1] for finite positions; clamp guards NaN
  ix = min(max(ix, 0), G.nx - 1);
  iy = min(max(iy, 0), G.ny - 1);
  iz = min(max(iz, 0), G.nz - 1);
  G.ic[i] = ix + G.nx * iy + G.nx * G.ny * iz + 1;
}
__global__ void k_ref_cells(const double *x0, const double *y0, const double *z0, int n, LinkGrid G) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) put_link_cell(G, i, x0[i], y0[i], z0[i]);
}
__global__ void k_minus1(const int *in, int *out, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = in[i] - 1;
}

// Reference half list (src/neighbourlist_m.F90:143-255): atom i lists j when
// j lies in i's own link cell after it in the cell's chain from L0 (rank =
// position in that chain) or in one of the 13 forward cells, and r < rnear
// with the reference's arithmetic; cells in the reference's stencil order and
// members in chain order (bin_atoms sorts them by rank), so NLIST(:, i) is the
// reference's, entry for entry.  Output in reference layout NLIST(nnbrs, nm),
// 1-based.
__global__ void k_half_list(const double *x0, const double *y0, const double *z0, const int *ic,
                            const int *orig, const int *rank, const int *cstart, const int *members, int n,
                            int nlcx, int nlcy, int nlcz, const BoxState *bs, double rn2,
                            int pbc, int nnbrs, int *numn_ref, int *nlist_ref, int *flags) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double *b = bs->b0;
  const int c = ic[i] - 1;
  const int cx = c % nlcx, cy = (c / nlcx) % nlcy, cz = c / (nlcx * nlcy);
  const double xi = x0[i], yi = y0[i], zi = z0[i];
  const int oi = orig[i], ri = rank[i];
  int cnt = 0;
  for (int dz = -1; dz <= 1; dz++) {
    int jz = (cz + dz + nlcz) % nlcz;
    for (int dy = -1; dy <= 1; dy++) {
      int jy = (cy + dy + nlcy) % nlcy;
      for (int dx = -1; dx <= 1; dx++) {
        int jx = (cx + dx + nlcx) % nlcx;
        // forward stencil of src/neighbourlist_m.F90:163-191
        bool fwd = (dz == 1) || (dz == 0 && dy == 1) || (dz == 0 && dy == 0 && dx == 1);
        bool own = (dz == 0 && dy == 0 && dx == 0);
        if (!fwd && !own) continue;
        int cj = jx + nlcx * (jy + nlcy * jz);
        for (int q = cstart[cj]; q < cstart[cj + 1]; q++) {
          int j = members[q];
          if (own && rank[j] <= ri) continue;
          double ddx = xi - x0[j], ddy = yi - y0[j], ddz = zi - z0[j];
          min_image(pbc, ddx, ddy, ddz);
          double r2 = sep2_exact(b, ddx, ddy, ddz);
          if (r2 < rn2) {
            cnt++;
            if (cnt <= nnbrs) nlist_ref[(size_t)oi * nnbrs + cnt - 1] = orig[j] + 1;
          }
        }
      }
    }
  }
  numn_ref[oi] = cnt;
  if (cnt > nnbrs) atomicOr(&flags[1], 1);
}

// Morton (Z-order) key of a fine-grid cell: consecutive keys form compact 3-D
// blocks, so atoms sorted by key have spatially local neighbourhoods.
__device__ __forceinline__ unsigned spread3(unsigned v) {
  v &= 0x3ff;
  v = (v | (v << 16)) & 0x030000FF;
  v = (v | (v << 8)) & 0x0300F00F;
  v = (v | (v << 4)) & 0x030C30C3;
  v = (v | (v << 2)) & 0x09249249;
  return v;
}
__device__ __forceinline__ unsigned compact3(unsigned v) {
  v &= 0x09249249;
  v = (v | (v >> 2)) & 0x030C30C3;
  v = (v | (v >> 4)) & 0x0300F00F;
  v = (v | (v >> 8)) & 0x030000FF;
  v = (v | (v >> 16)) & 0x000003FF;
  return v;
}
__device__ __forceinline__ int morton3(int x, int y, int z) {
  return (int)(spread3((unsigned)x) | (spread3((unsigned)y) << 1) | (spread3((unsigned)z) << 2));
}

// Packed position of atom i from fractional s - img (see the entry format).
// k: the atom's cell key (read only when pg.gx is set)
__device__ __forceinline__ double3 packed_pos_key(const double *b, PackGeo pg, unsigned k, double fx, double fy,
                                                  double fz) {
#pragma clang fp contract(off)  // the same packed positions from every kernel that writes them
  if (pg.gx) {
    fx -= ((double)compact3(k) + 0.5) * pg.ix;
    fy -= ((double)compact3(k >> 1) + 0.5) * pg.iy;
    fz -= ((double)compact3(k >> 2) + 0.5) * pg.iz;
  }
  return make_double3(b[0] * fx + b[3] * fy + b[6] * fz, b[1] * fx + b[4] * fy + b[7] * fz,
                      b[2] * fx + b[5] * fy + b[8] * fz);
}
// Image floors of an atom from its list cell: since the list was built it has
// moved less than half a skin, so the integer nearest to its position from the
// cell's centre is the floor of then (img), 12 bytes that the kick need not read.
// us per step without : with -- 2,000,000 atoms FP32 NVE 232.9 : 230.2, NPT 267.8 :
// 263.5.
__device__ __forceinline__ double3 near_image(PackGeo pg, unsigned k, double x, double y, double z) {
  return make_double3(rint(x - ((double)compact3(k) + 0.5) * pg.ix), rint(y - ((double)compact3(k >> 1) + 0.5) * pg.iy),
                      rint(z - ((double)compact3(k >> 2) + 0.5) * pg.iz));
}
__device__ __forceinline__ double3 packed_pos(const double *b, PackGeo pg, const int *cell, int i, double fx,
                                              double fy, double fz) {
  return packed_pos_key(b, pg, pg.gx ? (unsigned)cell[i] : 0u, fx, fy, fz);
}
__device__ __forceinline__ void store_packed(double4 *pos4, float4 *p4f, int i, double3 r, double w) {
  if (pos4) pos4[i] = make_double4(r.x, r.y, r.z, w);
  if (p4f) p4f[i] = make_float4((float)r.x, (float)r.y, (float)r.z, (float)w);
}


// fine-grid cell of an atom (fractional, folded into [0,1))
__device__ __forceinline__ int grid_cell(double x, double y, double z, int gx, int gy, int gz) {
  const double fx = x - floor(x), fy = y - floor(y), fz = z - floor(z);
  const int cx = min(max((int)(fx * gx), 0), gx - 1);
  const int cy = min(max((int)(fy * gy), 0), gy - 1);
  const int cz = min(max((int)(fz * gz), 0), gz - 1);
  return morton3(cx, cy, cz);
}
// The counting sort of a small system in one workgroup: cells, counts in LDS,
// start offsets, members (in any order within a cell; k_place ranks them).  Each
// thread keeps its atoms' cells and ranks in registers between the phases.
// Latency bound: 6.1 us at 2000 atoms against 2.4 + 2.2 + 2.4 and two launch gaps;
// even at 16,000 (14.6 us), where one workgroup's loads take over.
#define SORT_ONE_ATOMS 8192
#define SORT_ONE_CELLS 4096
__global__ void __launch_bounds__(1024) k_sort_one(const double *__restrict__ atoms, int n, int gx, int gy, int gz,
                                                   int m, int *__restrict__ cell, int *__restrict__ start,
                                                   int *__restrict__ members) {
  __shared__ int cnt[SORT_ONE_CELLS], sh[16];
  constexpr int NP = SORT_ONE_ATOMS / 1024, NC = SORT_ONE_CELLS / 1024;
  const int t = threadIdx.x;
#pragma unroll
  for (int q = 0; q < NC; q++) cnt[t + 1024 * q] = 0;
  __syncthreads();
  int kr[NP];  // cell | rank << 12
#pragma unroll
  for (int p0 = 0; p0 < NP; p0 += 4) {
    double x[4], y[4], z[4];
    if (1024 * p0 < n) {
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int i = min(t + 1024 * (p0 + u), n - 1);
        x[u] = atoms[i];
        y[u] = atoms[(size_t)n + i];
        z[u] = atoms[2 * (size_t)n + i];
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int i = t + 1024 * (p0 + u);
        if (i >= n) continue;
        const int key = grid_cell(x[u], y[u], z[u], gx, gy, gz);
        cell[i] = key;
        kr[p0 + u] = key | atomicAdd(&cnt[key], 1) << 12;
      }
    }
  }
  __syncthreads();
  int c[NC], s = 0;
#pragma unroll
  for (int q = 0; q < NC; q++) s += c[q] = cnt[NC * t + q];
  int total, ex = block_exclusive_scan_1024(s, sh, total);
#pragma unroll
  for (int q = 0; q < NC; q++) {
    cnt[NC * t + q] = ex;
    if (NC * t + q < m) start[NC * t + q] = ex;
    ex += c[q];
  }
  if (t == 0) start[m] = total;
  __syncthreads();
#pragma unroll
  for (int p0 = 0; p0 < NP; p0++) {
    const int i = t + 1024 * p0;
    if (i < n) members[cnt[kr[p0] & (SORT_ONE_CELLS - 1)] + (kr[p0] >> 12)] = i;
  }
}
// the same for larger systems: cells and their counts
__global__ void k_bin(const double *__restrict__ atoms, int n, int gx, int gy, int gz, int *__restrict__ cell,
                      int *__restrict__ count) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  int key = -1;
  if (i < n) {
    key = grid_cell(atoms[i], atoms[(size_t)n + i], atoms[2 * (size_t)n + i], gx, gy, gz);
    cell[i] = key;
  }
  const KeyRun r = key_run(key);
  if (r.is_head && key >= 0) atomicAdd(&count[key], r.len);
}

// The re-sort, one thread per atom: the atom's new slot is its rank by old slot
// among its cell's members, so the order is the same whatever order k_fill's
// atomics left them in.  It moves the per-atom fields that are read again
// (resort_fields), and sets what belongs to the new list: images, list cells,
// packed positions, reference positions, the reference box and the cleared list
// flags.  Bound by memory (about 350 B per atom).  Sorting the members, moving
// the fields, the integers and the reference cells, packing, clearing and
// copying took nine launches, 74 us at 524,288 atoms and 31 us at 2000, against
// 31 and 5 us for this kernel.
struct ResortSet {
  bool outs, third;  // FX..FZ and RHO; X3..Z3
};
__global__ void __launch_bounds__(MDK_BLOCK) k_place(
    double *__restrict__ dst, const double *__restrict__ src, const int *__restrict__ members,
    const int *__restrict__ cell, const int *__restrict__ start, int n, ResortSet rs, int *__restrict__ zdst,
    const int *__restrict__ zsrc, int *__restrict__ odst, const int *__restrict__ osrc, int *__restrict__ icdst,
    const int *__restrict__ icsrc, int *__restrict__ celldst, int *__restrict__ slot_of, int *__restrict__ img,
    float *__restrict__ sref, double4 *__restrict__ pos4, float4 *__restrict__ p4f, PackGeo pg, BoxState *bs,
    int *__restrict__ flags) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (blockIdx.x == 0) {
    if (threadIdx.x < 9) bs->bref[threadIdx.x] = bs->b0[threadIdx.x];
    if (threadIdx.x < 4) flags[threadIdx.x] = 0;
  }
  if (p >= n) return;
  const int v = members[p], key = cell[v], b = start[key], e = start[key + 1];
  int k = b;
  for (int q = b; q < e; q++) k += members[q] < v ? 1 : 0;
  constexpr int fl[13] = {F_X0, F_Y0, F_Z0, F_X1, F_Y1, F_Z1, F_X2, F_Y2, F_Z2, F_AFRHO, F_DAFRHO, F_MASS, F_DEL2};
  double f[13];
#pragma unroll
  for (int q = 0; q < 13; q++) f[q] = src[(size_t)fl[q] * n + v];
  const int z = zsrc[v], o = osrc[v], ic = icsrc[v];
#pragma unroll
  for (int q = 0; q < 13; q++) dst[(size_t)fl[q] * n + k] = f[q];
  if (rs.outs)
    for (int q : {F_FX, F_FY, F_FZ, F_RHO}) dst[(size_t)q * n + k] = src[(size_t)q * n + v];
  if (rs.third)
    for (int q : {F_X3, F_Y3, F_Z3}) dst[(size_t)q * n + k] = src[(size_t)q * n + v];
  zdst[k] = z;
  odst[k] = o;
  icdst[k] = ic;
  slot_of[o] = k;
  celldst[k] = key;
  const double mx = floor(f[0]), my = floor(f[1]), mz = floor(f[2]);
  img[3 * k] = (int)mx;
  img[3 * k + 1] = (int)my;
  img[3 * k + 2] = (int)mz;
  sref[3 * k] = (float)f[0];
  sref[3 * k + 1] = (float)f[1];
  sref[3 * k + 2] = (float)f[2];
  const double3 r = packed_pos_key(bs->b0, pg, (unsigned)key, f[0] - (int)mx, f[1] - (int)my, f[2] - (int)mz);
  store_packed(pos4, p4f, k, r, f[10]);
}

// Flags (flags[2]) a grid whose cells are narrower than the list radius in
// the current box (perpendicular widths) in any dimension the stencil spans.
__device__ void check_cell_width(const double *b, int gx, int gy, int gz, double rl2, int *flags) {
  const int gg[3] = {gx, gy, gz};
  const double vol = fabs(dev_volume(b));
  for (int d = 0; d < 3; d++) {
    const double *u = b + 3 * ((d + 1) % 3), *w = b + 3 * ((d + 2) % 3);
    const double cx = u[1] * w[2] - u[2] * w[1], cy = u[2] * w[0] - u[0] * w[2], cz = u[0] * w[1] - u[1] * w[0];
    const double width = vol / sqrt(cx * cx + cy * cy + cz * cz);
    if (gg[d] >= 3 && width / gg[d] < sqrt(rl2)) atomicMax(&flags[2], 1);
  }
}

// Neighbour list of atom i over its 27 stencil cells, gathering candidates
// from global memory (any grid; rounding images in dimensions with < 3 cells).
__device__ void list_one_atom(int i, const double4 *__restrict__ pos4, const double *atoms, const int *img,
                              const int *cell, const int *cstart, int n, int gx, int gy, int gz,
                              const double (*S)[3], double rl2, int pbc, bool rel, int maxn, int *nbr,
                              int *numn, int *flags) {
  const unsigned c = (unsigned)cell[i];
  const int cx = (int)compact3(c), cy = (int)compact3(c >> 1), cz = (int)compact3(c >> 2);
  const int sxr = gx >= 3 ? 1 : 0, syr = gy >= 3 ? 1 : 0, szr = gz >= 3 ? 1 : 0;
  const double4 pi = pos4[i];
  const double sxi = atoms[i] - img[3 * i], syi = atoms[(size_t)n + i] - img[3 * i + 1],
               szi = atoms[2 * (size_t)n + i] - img[3 * i + 2];
  int cnt = 0;
  for (int dz = -szr; dz <= szr; dz++) {
    int kz = cz + dz, wz = 0;
    if (kz < 0) { kz += gz; wz = 1; } else if (kz >= gz) { kz -= gz; wz = -1; }
    for (int dy = -syr; dy <= syr; dy++) {
      int ky = cy + dy, wy = 0;
      if (ky < 0) { ky += gy; wy = 1; } else if (ky >= gy) { ky -= gy; wy = -1; }
      for (int dx = -sxr; dx <= sxr; dx++) {
        int kx = cx + dx, wx = 0;
        if (kx < 0) { kx += gx; wx = 1; } else if (kx >= gx) { kx -= gx; wx = -1; }
        const int cj = morton3(kx, ky, kz);
        for (int j = cstart[cj]; j < cstart[cj + 1]; j++) {
          if (j == i) continue;
          int tx = wx, ty = wy, tz = wz;
          if (!sxr && (pbc & 1)) tx = -(int)round(sxi - (atoms[j] - img[3 * j]));
          if (!syr && (pbc & 2)) ty = -(int)round(syi - (atoms[(size_t)n + j] - img[3 * j + 1]));
          if (!szr && (pbc & 4)) tz = -(int)round(szi - (atoms[2 * (size_t)n + j] - img[3 * j + 2]));
          // open axes take the raw fractional difference: positions are folded
          // by img, so the shift restores img_i - img_j, which is -1, 0 or 1
          // for any pair closer than half the box
          if (!(pbc & 1)) tx = img[3 * i] - img[3 * j];
          if (!(pbc & 2)) ty = img[3 * i + 1] - img[3 * j + 1];
          if (!(pbc & 4)) tz = img[3 * i + 2] - img[3 * j + 2];
          if (tx < -1 || tx > 1 || ty < -1 || ty > 1 || tz < -1 || tz > 1) continue;
          // cell-relative packing: the cell offset (>= 3 cells per dimension)
          const int code = rel ? (dx + 1) + 3 * (dy + 1) + 9 * (dz + 1) : (tx + 1) + 3 * (ty + 1) + 9 * (tz + 1);
          const double4 pj = pos4[j];
          const double rx = pi.x - pj.x + S[code][0];
          const double ry = pi.y - pj.y + S[code][1];
          const double rz = pi.z - pj.z + S[code][2];
          const double r2 = rx * rx + ry * ry + rz * rz;
          if (r2 < rl2) {
            if (cnt < maxn) nbr[nbr_at(cnt, i, n)] = j | (code << NBR_CODE_SHIFT);
            cnt++;
          }
        }
      }
    }
  }
  numn[i] = min(cnt, maxn);
  if (cnt > maxn) atomicMax(&flags[0], cnt);
  for (int k = cnt; k < ((cnt + 3) & ~3) && k < maxn; k++)  // pad the last quad with null entries
    nbr[nbr_at(k, i, n)] = i | (NBR_NULL_CODE << NBR_CODE_SHIFT);
}

// Full neighbour list at r_list over the fine grid; atoms are already sorted by
// cell so cell c holds slots [cstart[c], cstart[c+1]).  Positions are the
// image-fixed Cartesian ones of pos4; the image shift of a candidate follows
// from the wrap of its cell (or from rounding in a dimension with one cell).
// nbr is column-major nbr[k*n + i] (index | shift code << 27).
__global__ void __launch_bounds__(MDK_BLOCK) k_full_list(
    const double4 *__restrict__ pos4, const double *atoms, const int *img, const int *cell,
    const int *cstart, int n, int gx, int gy, int gz, const BoxState *bs, double rl2, int pbc,
    int maxn, int *nbr, int *numn, int *flags) {
  __shared__ double S[32][3];
  double b[9];
#pragma unroll
  for (int k = 0; k < 9; k++) b[k] = bs->b0[k];
  const PackGeo absolute = {0, 0, 0, 0.0, 0.0, 0.0};
  shift_table(b, absolute, S);
  __syncthreads();
  if (blockIdx.x == 0 && threadIdx.x == 0) check_cell_width(b, gx, gy, gz, rl2, flags);
  int i = xcd_tile() * blockDim.x + threadIdx.x;
  if (i >= n) return;
  list_one_atom(i, pos4, atoms, img, cell, cstart, n, gx, gy, gz, S, rl2, pbc, false, maxn, nbr, numn, flags);
}

// Full neighbour list, a wave per atom (per consecutive atoms in turn): any
// grid and either packing.  The atom's 27 stencil cells are expanded into one
// candidate list in LDS (a lane per cell, offsets by a prefix sum; rounds of
// WLIST_CAP where a neighbourhood is larger), the lanes test 64 candidates at
// a time, and ballots rank the hits: partners within rc (the interaction range
// now, rin2) first, in list_one_atom's order, then the skin's (up to
// WLIST_SKIN of them wait in LDS, more stay among the first, which costs only
// efficiency), so the force pass stops after the in-range part and no density
// pass has to reorder the list (13 us a rebuild at 2000 atoms, 41 at 31,250 of
// iron_carbon).  Bound by latency where it is used: one lane per atom walked 182 to
// 488 candidates in a row of dependent loads (146 us for a 3456-atom slab, 111
// us for 250 atoms in one cell, 443 us for 31,250 iron_carbon atoms whose
// blocks exceed LIST_CAP; 27 us for 2000 atoms by blocks), against 10.0, 8.2,
// 57 and 6.6 us here.
#define WLIST_CAP 512
#define WLIST_SKIN 128
#define LIST_WAVE_BLK 16384
#define LIST_WAVE_ANY 131072
// set bits of a wave mask below this lane
__device__ __forceinline__ int lanes_below(unsigned long long mask) {
  return __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0));
}
__global__ void __launch_bounds__(64) k_full_list_wave(
    const double4 *__restrict__ pos4, const double *__restrict__ atoms, const int *__restrict__ img,
    const int *__restrict__ cell, const int *__restrict__ cstart, int n, int gx, int gy, int gz, PackGeo pg,
    const BoxState *bs, double rl2, double rin2, int pbc, int per, int maxn, int *nbr, int *numn, int *flags) {
  __shared__ double S[32][3];
  __shared__ int cand[WLIST_CAP], skin[WLIST_SKIN];
  const int lane = threadIdx.x, nw = gridDim.x - 1;
  const double *b = bs->b0;
  if ((int)blockIdx.x == nw) {  // the last block checks the grid
    if (lane == 0) check_cell_width(b, gx, gy, gz, rl2, flags);
    return;
  }
  shift_table(b, pg, S);
  const bool rel = pg.gx != 0;
  const int sxr = gx >= 3 ? 1 : 0, syr = gy >= 3 ? 1 : 0, szr = gz >= 3 ? 1 : 0;
  const int i0 = blockIdx.x * per, i1 = min(n, i0 + per);
  int have = -1, total = 0, cs = 0, cc = 0, off = 0;
  for (int i = i0; i < i1; i++) {
    const int key = __builtin_amdgcn_readfirstlane(cell[i]);
    const bool fresh = key != have;
    if (fresh) {
      have = key;
      cs = cc = 0;
      const int dx = lane % 3 - 1, dy = (lane / 3) % 3 - 1, dz = lane / 9 - 1;
      if (lane < 27 && abs(dx) <= sxr && abs(dy) <= syr && abs(dz) <= szr) {
        int kx = (int)compact3((unsigned)key) + dx, ky = (int)compact3((unsigned)key >> 1) + dy,
            kz = (int)compact3((unsigned)key >> 2) + dz;
        kx += kx < 0 ? gx : (kx >= gx ? -gx : 0);
        ky += ky < 0 ? gy : (ky >= gy ? -gy : 0);
        kz += kz < 0 ? gz : (kz >= gz ? -gz : 0);
        const int cj = morton3(kx, ky, kz);
        cs = cstart[cj];
        cc = cstart[cj + 1] - cs;
      }
      off = cc;  // prefix sum over the wave
#pragma unroll
      for (int o = 1; o < 32; o <<= 1) {
        const int u = __shfl_up(off, o, 64);
        if (lane >= o) off += u;
      }
      total = __shfl(off, 26, 64);
      off -= cc;
    }
    const double4 pi = pos4[i];
    const double si[3] = {atoms[i], atoms[(size_t)n + i], atoms[2 * (size_t)n + i]};
    const int ii[3] = {img[3 * i], img[3 * i + 1], img[3 * i + 2]};
    const unsigned cu = (unsigned)key;
    const int cx = (int)compact3(cu), cy = (int)compact3(cu >> 1), cz = (int)compact3(cu >> 2);
    int cnt = 0, held = 0;
    for (int base = 0; base < total; base += WLIST_CAP) {
      const int end = min(WLIST_CAP, total - base);
      if (fresh || total > WLIST_CAP) {
        __syncthreads();
        for (int k = max(0, base - off); k < cc && off + k < base + end; k++)
          cand[off + k - base] = (cs + k) | (lane << NBR_CODE_SHIFT);
        __syncthreads();  // one wave: orders its LDS accesses (and the shift table's)
      }
      for (int t0 = 0; t0 < end; t0 += 64) {
        const unsigned e = t0 + lane < end ? (unsigned)cand[t0 + lane] : (unsigned)i;
        const int j = (int)(e & NBR_IDX_MASK), c = (int)(e >> NBR_CODE_SHIFT);
        bool ok = j != i;
        int code = c;
        if (!rel) {  // image shift: from the cell's wrap, rounding, or an open axis's images
          int q[3];
          const int d[3] = {c % 3 - 1, (c / 3) % 3 - 1, c / 9 - 1}, ck[3] = {cx, cy, cz}, g[3] = {gx, gy, gz};
          const int sr[3] = {sxr, syr, szr};
#pragma unroll
          for (int a = 0; a < 3; a++) {
            const int k = ck[a] + d[a], w = k < 0 ? 1 : (k >= g[a] ? -1 : 0);
            const int ij = img[3 * j + a];
            if (!((pbc >> a) & 1)) q[a] = ii[a] - ij;
            else if (sr[a]) q[a] = w;
            else q[a] = -(int)round((si[a] - ii[a]) - (atoms[(size_t)a * n + j] - ij));
            ok = ok && q[a] >= -1 && q[a] <= 1;
          }
          code = ok ? (q[0] + 1) + 3 * (q[1] + 1) + 9 * (q[2] + 1) : 0;
        }
        const double4 pj = pos4[j];
        const double rx = pi.x - pj.x + S[code][0], ry = pi.y - pj.y + S[code][1], rz = pi.z - pj.z + S[code][2];
        const double r2 = rx * rx + ry * ry + rz * rz;
        const bool hit = ok && r2 < rl2;
        const unsigned long long out = __ballot(hit && !(r2 < rin2));
        const int h = held + lanes_below(out);
        const bool wait = hit && !(r2 < rin2) && h < WLIST_SKIN;
        const int entry = j | (code << NBR_CODE_SHIFT);
        if (wait) skin[h] = entry;
        held = min(WLIST_SKIN, held + __popcll(out));
        const unsigned long long mask = __ballot(hit && !wait);
        const int m = cnt + lanes_below(mask);
        if (hit && !wait && m < maxn) nbr[nbr_at(m, i, n)] = entry;
        cnt += __popcll(mask);
      }
    }
    __syncthreads();  // the held entries
    for (int q = lane; q < held; q += 64)
      if (cnt + q < maxn) nbr[nbr_at(cnt + q, i, n)] = skin[q];
    __syncthreads();  // read before the next atom's
    cnt += held;
    if (lane == 0) {
      numn[i] = min(cnt, maxn);
      if (cnt > maxn) atomicMax(&flags[0], cnt);
    }
    const int pad = cnt + lane;  // pad the last quad with null entries
    if (lane < 3 && pad < ((cnt + 3) & ~3) && pad < maxn) nbr[nbr_at(pad, i, n)] = i | (NBR_NULL_CODE << NBR_CODE_SHIFT);
  }
}

// Full neighbour list by 2x2x2-cell blocks (8 consecutive Morton keys, so one
// contiguous range of atoms), one wave per block, for cell-relative packing.
// The wave stages the atoms of the 4x4x4 cells around the block in LDS --
// positions relative to the centre of the block's first cell, in FP32 (the
// 1e-6 A rounding is immaterial against the skin) -- instead of gathering them
// from global memory.  Each lane then walks the 27 staged cells around its own
// atom's cell (about 155 candidates instead of all 368 staged ones), row by
// row; a partner's code is the offset of its cell.
// Fully periodic boxes with >= 4 cells per dimension (no staged cell occurs
// twice); a block whose neighbourhood exceeds LIST_CAP atoms uses the
// global-gather loop.  blocks[] lists the Morton key / 8 of every block that
// holds grid cells.
#define LIST_CAP 512
__global__ void __launch_bounds__(64) k_full_list_blk(
    const double4 *__restrict__ pos4, const double *atoms, const int *img, const int *cell,
    const int *__restrict__ cstart, const int *blocks, int n, PackGeo pg, const BoxState *bs,
    double rl2, int maxn, int *nbr, int *numn, int *flags) {
  __shared__ double S[32][3];
  __shared__ float4 cpos[LIST_CAP];
  __shared__ int hoff[64], hcnt[64];  // staged cell h: candidates [hoff, hoff + hcnt)
  const int lane = threadIdx.x, gx = pg.gx, gy = pg.gy, gz = pg.gz;
  const double *b = bs->b0;
  shift_table(b, pg, S);
  if (blockIdx.x == 0 && lane == 0) check_cell_width(b, gx, gy, gz, rl2, flags);
  const unsigned base = (unsigned)blocks[xcd_tile()] << 3;
  const int x0 = 2 * (int)compact3(base >> 3), y0 = 2 * (int)compact3(base >> 4), z0 = 2 * (int)compact3(base >> 5);
  const int a0 = cstart[base], a1 = cstart[base + 8];
  if (a1 <= a0) return;  // uniform: no atoms in this block
  // staged cell h = hx + 4 hy + 16 hz at (x0-1+hx, y0-1+hy, z0-1+hz): one per lane
  const int hx = lane & 3, hy = (lane >> 2) & 3, hz = lane >> 4;
  int x = x0 - 1 + hx, y = y0 - 1 + hy, z = z0 - 1 + hz;
  if (x < 0) x += gx; else if (x >= gx) x -= gx;
  if (y < 0) y += gy; else if (y >= gy) y -= gy;
  if (z < 0) z += gz; else if (z >= gz) z -= gz;
  const int key = morton3(x, y, z);
  const int cs = cstart[key], cnt = cstart[key + 1] - cs;
  int off = cnt;  // exclusive prefix sum over the wave
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int u = __shfl_up(off, o, 64);
    if (lane >= o) off += u;
  }
  const int total = __shfl(off, 63, 64);
  off -= cnt;
  hoff[lane] = off;
  hcnt[lane] = cnt;
  __syncthreads();  // shift table, cell ranges
  if (total > LIST_CAP) {
    for (int i = a0 + lane; i < a1; i += 64)
      list_one_atom(i, pos4, atoms, img, cell, cstart, n, gx, gy, gz, S, rl2, 7, true, maxn, nbr, numn, flags);
    return;
  }
  // centre of the staged cell from the centre of cell (x0,y0,z0): B0 (h - 1) / g
  const double fx = (hx - 1) * pg.ix, fy = (hy - 1) * pg.iy, fz = (hz - 1) * pg.iz;
  const double vx = b[0] * fx + b[3] * fy + b[6] * fz, vy = b[1] * fx + b[4] * fy + b[7] * fz,
               vz = b[2] * fx + b[5] * fy + b[8] * fz;
  for (int k = 0; k < cnt; k++) {
    const double4 p = pos4[cs + k];
    cpos[off + k] = make_float4((float)(p.x + vx), (float)(p.y + vy), (float)(p.z + vz), __int_as_float(cs + k));
  }
  __syncthreads();
  const float rl2f = (float)rl2;
  for (int i = a0 + lane; i < a1; i += 64) {
    const unsigned ck = (unsigned)cell[i];
    const int ax = (int)compact3(ck) - x0, ay = (int)compact3(ck >> 1) - y0, az = (int)compact3(ck >> 2) - z0;
    const double4 pd = pos4[i];
    const double ex = ax * pg.ix, ey = ay * pg.iy, ez = az * pg.iz;
    const float px = (float)(pd.x + (b[0] * ex + b[3] * ey + b[6] * ez)),
                py = (float)(pd.y + (b[1] * ex + b[4] * ey + b[7] * ez)),
                pz = (float)(pd.z + (b[2] * ex + b[5] * ey + b[8] * ez));
    const int h0 = ax + 4 * ay + 16 * az;  // staged cell at offset (-1,-1,-1) from the atom's
    int m = 0;
    // the three cells of a row along x are consecutive staged cells, so one
    // loop walks their candidates (about 17, instead of three loops of about
    // 6 whose lengths differ from lane to lane); a partner's cell offset, and
    // so its code, follows from where it lies in the row
    for (int dz = 0; dz < 3; dz++)
      for (int dy = 0; dy < 3; dy++) {
        const int h = h0 + 4 * dy + 16 * dz;  // the row's cell at dx = 0
        const int lo = hoff[h], m1 = hoff[h + 1], m2 = hoff[h + 2], hi = m2 + hcnt[h + 2];
        const int tagb = 3 * dy + 9 * dz;
        auto test = [&](const float4 q, int c) {
          const float rx = px - q.x, ry = py - q.y, rz = pz - q.z;
          const int j = __float_as_int(q.w);
          if (rx * rx + ry * ry + rz * rz < rl2f && j != i) {
            const int code = tagb + (c >= m1 ? 1 : 0) + (c >= m2 ? 1 : 0);
            if (m < maxn) nbr[nbr_at(m, i, n)] = j | (code << NBR_CODE_SHIFT);
            m++;
          }
        };
        // four candidates per trip: their LDS reads are in flight together;
        // the tests run in candidate order, so the list is the same
        int c = lo;
        for (; c + 4 <= hi; c += 4) {
          const float4 q0 = cpos[c], q1 = cpos[c + 1], q2 = cpos[c + 2], q3 = cpos[c + 3];
          test(q0, c);
          test(q1, c + 1);
          test(q2, c + 2);
          test(q3, c + 3);
        }
        for (; c < hi; c++) test(cpos[c], c);
      }
    numn[i] = min(m, maxn);
    if (m > maxn) atomicMax(&flags[0], m);
    for (int k = m; k < ((m + 3) & ~3) && k < maxn; k++)  // pad the last quad with null entries
      nbr[nbr_at(k, i, n)] = i | (NBR_NULL_CODE << NBR_CODE_SHIFT);
  }
}

// Brick list: the full list of the FP32 Fe path for large systems, by bricks of
// 4x4x4 cells (64 consecutive Morton keys, so one contiguous range of atoms), a
// workgroup of NT threads each and at most one atom a thread.  The pair passes
// keep the atoms of a brick and of the cells around it (6x6x6) in LDS, so the
// list holds LDS byte offsets of 16 bits instead of atom indices and cell codes.
//   binfo[b]   first atom, atoms, staged atoms of brick b (brick_extent)
//   bstage     b's staged atoms (brick_cap each): index | cell h << BRICK_H_SHIFT,
//              h = hx + 6 hy + 36 hz of the 6x6x6 cells; the brick's own atoms
//              come first, in order
//   nbr16      quad q of atom i (four entries) at [q n + i]: partners within
//              rin first, then those of the skin, then null slots (the one
//              behind the staged atoms)
//   bcnt[i]    quads
// Entries are found as in k_full_list_blk, a row of three cells at a time, as a
// bit mask of hits, so that the lanes append in step; the masks of the skin's
// entries wait in LDS until the others are written.
struct Quad16 {
  unsigned a, b;
  int m;
  __device__ __forceinline__ void push(unsigned e) {
    a = __builtin_amdgcn_alignbit(b, a, 16);
    b = __builtin_amdgcn_alignbit(e, b, 16);
    m++;
  }
};
template <int NT>
__global__ void __launch_bounds__(NT) k_brick_list(const float4 *__restrict__ p4f, const int *__restrict__ cell,
                                                   const int *__restrict__ cstart, const int *__restrict__ bricks,
                                                   int n, PackGeo pg, const BoxState *bs, double rl2, double rin2,
                                                   int maxq, int cap, uint2 *__restrict__ nbr16, int *bcnt,
                                                   int *__restrict__ bstage, int4 *binfo, int *flags) {
  extern __shared__ float4 cpos[];
  __shared__ int hoff[BRICK_CELLS + 1], wsum[NT / 64][2];
  __shared__ unsigned skin[9][NT];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6, bi = xcd_tile();
  const double *b = bs->b0;
  if (blockIdx.x == 0 && t == 0) check_cell_width(b, pg.gx, pg.gy, pg.gz, rl2, flags);
  const unsigned base = (unsigned)bricks[bi] << 6;
  const int x0 = (int)compact3(base), y0 = (int)compact3(base >> 1), z0 = (int)compact3(base >> 2);
  const int a0 = cstart[base], own = cstart[base + 64] - a0;
  // staged cell t = hx + 6 hy + 36 hz at (x0-1+hx, y0-1+hy, z0-1+hz), one per
  // thread; those more than one beyond the grid's end are nobody's neighbours
  const int hx = t % 6, hy = (t / 6) % 6, hz = t / 36;
  int cs = 0, cnt = 0;
  bool mine = false;
  if (t < BRICK_CELLS) {
    int x = x0 - 1 + hx, y = y0 - 1 + hy, z = z0 - 1 + hz;
    if (x <= pg.gx && y <= pg.gy && z <= pg.gz) {
      mine = hx >= 1 && hx <= 4 && x < pg.gx && hy >= 1 && hy <= 4 && y < pg.gy && hz >= 1 && hz <= 4 && z < pg.gz;
      x += x < 0 ? pg.gx : (x == pg.gx ? -pg.gx : 0);
      y += y < 0 ? pg.gy : (y == pg.gy ? -pg.gy : 0);
      z += z < 0 ? pg.gz : (z == pg.gz ? -pg.gz : 0);
      const int key = morton3(x, y, z);
      cs = cstart[key];
      cnt = cstart[key + 1] - cs;
    }
  }
  // exclusive prefix sums over the cells: of all atoms, and of the others' atoms
  int off = cnt, oth = mine ? 0 : cnt;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int u = __shfl_up(off, o, 64), v = __shfl_up(oth, o, 64);
    if (lane >= o) {
      off += u;
      oth += v;
    }
  }
  if (lane == 63) {
    wsum[w][0] = off;
    wsum[w][1] = oth;
  }
  off -= cnt;
  oth -= mine ? 0 : cnt;
  __syncthreads();
  int total = 0;
#pragma unroll
  for (int q = 0; q < NT / 64; q++) {
    off += q < w ? wsum[q][0] : 0;
    oth += q < w ? wsum[q][1] : 0;
    total += wsum[q][0];
  }
  if (t < BRICK_CELLS) hoff[t] = off;
  if (t == 0) hoff[BRICK_CELLS] = total;
  const int4 info = brick_extent(a0, own, total, NT, cap);
  if (t == 0) {
    binfo[bi] = info;
    if (own > NT) atomicMax(&flags[1], own);
    if (own > 0 && total >= cap) atomicMax(&flags[3], total + 1);
  }
  if (info.y == 0) return;  // uniform: no bstage words, and none counted
  // centre of the staged cell from the brick's centre, in FP32 positions (the
  // rounding is immaterial against the skin); .w = LDS offset in the pair passes
  const double fx = (hx - 2.5) * pg.ix, fy = (hy - 2.5) * pg.iy, fz = (hz - 2.5) * pg.iz;
  const double vx = b[0] * fx + b[3] * fy + b[6] * fz, vy = b[1] * fx + b[4] * fy + b[7] * fz,
               vz = b[2] * fx + b[5] * fy + b[8] * fz;
  const int slot0 = mine ? cs - a0 : own + oth;
#pragma unroll 2
  for (int k = 0; k < cnt; k++) {
    const float4 p = p4f[cs + k];
    cpos[off + k] = make_float4((float)(p.x + vx), (float)(p.y + vy), (float)(p.z + vz), __int_as_float((slot0 + k) << 4));
    bstage[(size_t)bi * cap + slot0 + k] = (int)((unsigned)(cs + k) | (unsigned)t << BRICK_H_SHIFT);
  }
  __syncthreads();
  if (t >= own) return;
  const int i = a0 + t;
  const unsigned ck = (unsigned)cell[i];
  const int ax = (int)compact3(ck) - x0, ay = (int)compact3(ck >> 1) - y0, az = (int)compact3(ck >> 2) - z0;
  const double ex = (ax - 1.5) * pg.ix, ey = (ay - 1.5) * pg.iy, ez = (az - 1.5) * pg.iz;
  const float4 pi = p4f[i];
  const float px = (float)(pi.x + (b[0] * ex + b[3] * ey + b[6] * ez)),
              py = (float)(pi.y + (b[1] * ex + b[4] * ey + b[7] * ez)),
              pz = (float)(pi.z + (b[2] * ex + b[5] * ey + b[8] * ez));
  const float rl2f = (float)rl2, rin2f = (float)rin2;
  const int h0 = ax + 6 * ay + 36 * az;  // the cell at offset (-1,-1,-1) from the atom's
  const unsigned self = (unsigned)t << 4, null = (unsigned)total << 4;
  Quad16 list = {0, 0, 0};
  auto put = [&](unsigned e) {
    list.push(e);
    if (!(list.m & 3) && list.m <= 4 * maxq) nbr16[(size_t)((list.m >> 2) - 1) * n + i] = make_uint2(list.a, list.b);
  };
  auto put_hits = [&](unsigned mask, int c0) {
    while (mask) {
      const unsigned e = (unsigned)__float_as_int(cpos[c0 + __builtin_ctz(mask)].w);
      mask &= mask - 1;
      if (e != self) put(e);
    }
  };
  for (int r = 0; r < 9; r++) {
    const int h = h0 + 6 * (r % 3) + 36 * (r / 3), hi = hoff[h + 3];
    const int lo = hoff[h];
    skin[r][t] = 0u;
    for (int c0 = lo; c0 < hi; c0 += 32) {
      const int m = min(32, hi - c0);
      unsigned hit = 0, near = 0;
      auto test = [&](const float4 q, int k) {
        const float rx = px - q.x, ry = py - q.y, rz = pz - q.z, r2 = rx * rx + ry * ry + rz * rz;
        hit |= r2 < rl2f ? 1u << k : 0u;
        near |= r2 < rin2f ? 1u << k : 0u;
      };
      int k = 0;
      for (; k + 4 <= m; k += 4) {  // four LDS reads in flight
        const float4 q0 = cpos[c0 + k], q1 = cpos[c0 + k + 1], q2 = cpos[c0 + k + 2], q3 = cpos[c0 + k + 3];
        test(q0, k);
        test(q1, k + 1);
        test(q2, k + 2);
        test(q3, k + 3);
      }
      for (; k < m; k++) test(cpos[c0 + k], k);
      put_hits(near, c0);
      if (c0 == lo) skin[r][t] = hit & ~near;
      else put_hits(hit & ~near, c0);
    }
  }
  for (int r = 0; r < 9; r++) put_hits(skin[r][t], hoff[h0 + 6 * (r % 3) + 36 * (r / 3)]);
  while (list.m & 3) put(null);
  const int nq = list.m >> 2;
  if (nq > maxq) atomicMax(&flags[0], list.m);
  bcnt[i] = nq > maxq ? 0 : nq;
}

// The brick list's pairs as entries of the general format, for the callers
// outside the FP32 Fe passes.
__global__ void __launch_bounds__(BRICK_THREADS_MAX) k_brick_expand(const int *__restrict__ cell, const int *__restrict__ bricks, int n,
                                                     int cap, const uint2 *__restrict__ nbr16,
                                                     const int *__restrict__ bcnt, const int *__restrict__ bstage,
                                                     const int4 *__restrict__ binfo, int maxn, int *nbr, int *numn) {
  const int bi = blockIdx.x;
  const int4 info = binfo[bi];
  if ((int)threadIdx.x >= info.y) return;
  const int i = info.x + threadIdx.x, nq = bcnt[i];
  const unsigned base = (unsigned)bricks[bi] << 6, ck = (unsigned)cell[i];
  // hx - 1 of the atom's own staged cell is its offset in the brick
  const int ax = (int)(compact3(ck) - compact3(base)), ay = (int)(compact3(ck >> 1) - compact3(base >> 1)),
            az = (int)(compact3(ck >> 2) - compact3(base >> 2));
  int m = 0;
  for (int q = 0; q < nq; q++) {
    const uint2 w = nbr16[(size_t)q * n + i];
    for (int u = 0; u < 4; u++) {
      const int slot = (int)(((u < 2 ? w.x : w.y) >> (16 * (u & 1))) & 0xffff) >> 4;
      if (slot >= info.z || m >= maxn) continue;
      const unsigned e = (unsigned)bstage[(size_t)bi * cap + slot];
      const int h = e >> BRICK_H_SHIFT, hx = h % 6, hy = (h / 6) % 6, hz = h / 36;
      const int code = (hx - ax) + 3 * (hy - ay) + 9 * (hz - az);
      nbr[nbr_at(m++, i, n)] = (int)(e & ((1u << BRICK_H_SHIFT) - 1)) | (code << NBR_CODE_SHIFT);
    }
  }
  numn[i] = m;
  for (; m & 3; m++)
    if (m < maxn) nbr[nbr_at(m, i, n)] = i | (NBR_NULL_CODE << NBR_CODE_SHIFT);
}

// ---------------------------------------------------------------------------
// MD-step kernels
// ---------------------------------------------------------------------------
// Box part of the drift, by one workgroup: copies the box state into the other
// buffer with b0 += b1 + b2 and b1 += b2 (src/quench_m.F90:574-589; one field
// per thread).
__device__ void drift_box(const BoxState *bin, BoxState *bout, int ivol) {
#pragma clang fp contract(off)
  const int nw = (int)(sizeof(BoxState) / sizeof(double));
  const double *src = (const double *)bin;
  double *dst = (double *)bout;
  for (int w = threadIdx.x; w < nw; w += blockDim.x) {
    const int f = w - (int)(offsetof(BoxState, b0) / sizeof(double));
    const int g = w - (int)(offsetof(BoxState, b1) / sizeof(double));
    double val = src[w];
    if (f >= 0 && f < 9) {  // b0 += b1 + b2 (component-wise, as the reference's two updates)
      const bool upd = ivol < 1 || (ivol == 4 && f == 8);
      if (upd) val = bin->b0[f] + (bin->b1[f] + bin->b2[f]);
    } else if (g >= 0 && g < 9) {
      const bool upd = ivol < 1 || (ivol == 4 && g == 8);
      if (upd) val = bin->b1[g] + bin->b2[g];
    }
    dst[w] = val;
  }
}

// velocityverlet drift (src/quench_m.F90:574-589): x0 += x1 + x2 (also into the
// packed copy); block 0 copies the box state into the other buffer, advancing
// b1 and b0 there (one field per thread).
__global__ void k_drift(double *__restrict__ atoms, double4 *__restrict__ pos4, float4 *__restrict__ p4f,
                        const int *__restrict__ img, const int *__restrict__ cell, PackGeo pg, int n,
                        const BoxState *__restrict__ bin, BoxState *__restrict__ bout, int ivol,
                        const int *__restrict__ zat, const double *__restrict__ spec, double *__restrict__ kin) {
#pragma clang fp contract(off)
  int i = xcd_tile() * blockDim.x + threadIdx.x;
  double kv[9] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  if (i < n) {
    double *x0 = atoms, *y0 = atoms + n, *z0 = atoms + 2 * (size_t)n;
    const double *x1 = atoms + 3 * (size_t)n, *y1 = atoms + 4 * (size_t)n, *z1 = atoms + 5 * (size_t)n;
    const double *x2 = atoms + 6 * (size_t)n, *y2 = atoms + 7 * (size_t)n, *z2 = atoms + 8 * (size_t)n;
    const double xn = x0[i] + (x1[i] + x2[i]);
    const double yn = y0[i] + (y1[i] + y2[i]);
    const double zn = z0[i] + (z1[i] + z2[i]);
    x0[i] = xn;
    y0[i] = yn;
    z0[i] = zn;
    // the box after this step's update (computed redundantly per thread)
    double b[9];
    for (int k = 0; k < 9; k++) {
      const bool upd = ivol < 1 || (ivol == 4 && k == 8);
      b[k] = upd ? bin->b0[k] + (bin->b1[k] + bin->b2[k]) : bin->b0[k];
    }
    const double3 r = packed_pos(b, pg, cell, i, xn - img[3 * i], yn - img[3 * i + 1], zn - img[3 * i + 2]);
    store_packed(pos4, p4f, i, r, 0.0);  // F' is stored by the density pass, which always runs next
    const int z = zat[i];
    if (z != 0) kin_terms(b, x1[i], y1[i], z1[i], spec ? spec[2 * z] : atoms[(size_t)F_MASS * n + i], kv);
  }
  if (blockIdx.x == 0) drift_box(bin, bout, ivol);
  block_store<9, 0>(kv, kin);
}

// predic (src/quench_m.F90:636-671): x0 += x1 + x2 + x3, x1 += 2 x2 + 3 x3,
// x2 += 3 x3, the box likewise for ivol 0 (all) or 4 (z only), packed
// positions with the predicted box; block 0 writes the predicted box state
// into bout.  primed == 0 leaves everything as it is (see mdk_predic).
__device__ __forceinline__ void predict_box(const BoxState *bin, double *b0, double *b1, double *b2, int ivol,
                                            int primed, int k) {
#pragma clang fp contract(off)
  const bool upd = primed && (ivol == 0 || (ivol == 4 && k == 8));
  b0[k] = upd ? bin->b0[k] + bin->b1[k] + bin->b2[k] + bin->b3[k] : bin->b0[k];
  b1[k] = upd ? bin->b1[k] + 2.0 * bin->b2[k] + 3.0 * bin->b3[k] : bin->b1[k];
  b2[k] = upd ? bin->b2[k] + 3.0 * bin->b3[k] : bin->b2[k];
}
__global__ void k_predic(double *__restrict__ atoms, double4 *__restrict__ pos4, float4 *__restrict__ p4f,
                         const int *__restrict__ img, const int *__restrict__ cell, PackGeo pg, int n,
                         const BoxState *__restrict__ bin, BoxState *__restrict__ bout, int ivol, int primed,
                         const int *__restrict__ zat, const double *__restrict__ spec, double *__restrict__ kin) {
#pragma clang fp contract(off)
  const int i = xcd_tile() * blockDim.x + threadIdx.x;
  double kv[9] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  if (i < n) {
    double *p = atoms;
    double x[3], v[3];
    for (int d = 0; d < 3; d++) {
      double *q0 = p + (size_t)(F_X0 + d) * n, *q1 = p + (size_t)(F_X1 + d) * n, *q2 = p + (size_t)(F_X2 + d) * n;
      const double *q3 = p + (size_t)(F_X3 + d) * n;
      double v0 = q0[i];
      if (primed) {
        const double v1 = q1[i], v2 = q2[i], v3 = q3[i];
        v0 = v0 + v1 + v2 + v3;
        q0[i] = v0;
        q1[i] = v1 + 2.0 * v2 + 3.0 * v3;
        q2[i] = v2 + 3.0 * v3;
      }
      x[d] = v0;
      v[d] = q1[i];
    }
    double b[9], bd1[9], bd2[9];
    for (int k = 0; k < 9; k++) predict_box(bin, b, bd1, bd2, ivol, primed, k);
    const double3 r = packed_pos(b, pg, cell, i, x[0] - img[3 * i], x[1] - img[3 * i + 1], x[2] - img[3 * i + 2]);
    store_packed(pos4, p4f, i, r, 0.0);  // F' is stored by the density pass, which always runs next
    const int z = zat[i];
    if (z != 0) kin_terms(b, v[0], v[1], v[2], spec ? spec[2 * z] : atoms[(size_t)F_MASS * n + i], kv);
  }
  if (blockIdx.x == 0) {  // the whole box state into bout, one field per thread
    const int nw = (int)(sizeof(BoxState) / sizeof(double));
    const double *src = (const double *)bin;
    double *dst = (double *)bout;
    for (int w = threadIdx.x; w < nw; w += blockDim.x) dst[w] = src[w];
    __syncthreads();
    if (threadIdx.x < 9) predict_box(bin, bout->b0, bout->b1, bout->b2, ivol, primed, threadIdx.x);
  }
  block_store<9, 0>(kv, kin);
}

// kinten's partial sums for the velocities and box as they are (a force
// evaluation that no drift, predictor or fused half kick has prepared)
__global__ void __launch_bounds__(MDK_BLOCK) k_kin(const double *__restrict__ atoms, const int *__restrict__ zat,
                                                   int n, const BoxState *__restrict__ bs,
                                                   const double *__restrict__ spec, double *__restrict__ kin) {
  const int i = xcd_tile() * blockDim.x + threadIdx.x;
  double kv[9] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  if (i < n) {
    const int z = zat[i];
    double b[9];
    for (int k = 0; k < 9; k++) b[k] = bs->b0[k];
    if (z != 0)
      kin_terms(b, atoms[(size_t)F_X1 * n + i], atoms[(size_t)F_Y1 * n + i], atoms[(size_t)F_Z1 * n + i],
                spec ? spec[2 * z] : atoms[(size_t)F_MASS * n + i], kv);
  }
  block_store<9, 0>(kv, kin);
}

// correc (src/quench_m.F90:682-759).  The coefficients are the reference's
// REAL(4) parameters (no d0 suffix): 1/6, 5/6, 1, 1/3 rounded to float.
// cc = del2 f - tgid x1 / 2 - x2 per atom (vacancies skipped); the box (ivol
// < 1: all, 4: z only) with cc = bdel2 fb - b2, in place by nine threads of
// block 0 (no other thread reads the box's b fields).
__global__ void k_correc(double *__restrict__ atoms, const int *__restrict__ zat, int n, BoxState *bs, int ivol,
                         double bdel2, const double *__restrict__ spec) {
#pragma clang fp contract(off)
  const double ct0 = (double)0.166666666666666667f, ct1 = (double)0.833333333333333333f;
  const double ct2 = (double)1.000000000000000000f, ct3 = (double)0.333333333333333333f;
  const int i = xcd_tile() * blockDim.x + threadIdx.x;
  if (i < n && zat[i] != 0) {
    const double *g = bs->tgid;
    const int z = zat[i];
    const double d2 = spec ? spec[2 * z + 1] : atoms[(size_t)F_DEL2 * n + i];
    const double x1 = atoms[(size_t)F_X1 * n + i], y1 = atoms[(size_t)F_Y1 * n + i], z1 = atoms[(size_t)F_Z1 * n + i];
    const double s[3] = {TT(g, 1, 1) * x1 + TT(g, 1, 2) * y1 + TT(g, 1, 3) * z1,
                         TT(g, 2, 1) * x1 + TT(g, 2, 2) * y1 + TT(g, 2, 3) * z1,
                         TT(g, 3, 1) * x1 + TT(g, 3, 2) * y1 + TT(g, 3, 3) * z1};
    for (int d = 0; d < 3; d++) {
      double *q0 = atoms + (size_t)(F_X0 + d) * n, *q1 = atoms + (size_t)(F_X1 + d) * n;
      double *q2 = atoms + (size_t)(F_X2 + d) * n, *q3 = atoms + (size_t)(F_X3 + d) * n;
      const double f = atoms[(size_t)(F_FX + d) * n + i];
      const double cc = d2 * f - 0.5 * s[d] - q2[i];
      q0[i] = q0[i] + cc * ct0;
      q1[i] = q1[i] + cc * ct1;
      q2[i] = q2[i] + cc * ct2;
      q3[i] = q3[i] + cc * ct3;
    }
  }
  if (blockIdx.x == 0 && threadIdx.x < 9) {
    const int k = threadIdx.x;
    if (ivol < 1 || (ivol == 4 && k == 8)) {
      const double cc = bdel2 * bs->fb[k] - bs->b2[k];
      bs->b0[k] = bs->b0[k] + ct0 * cc;
      bs->b1[k] = bs->b1[k] + ct1 * cc;
      bs->b2[k] = bs->b2[k] + ct2 * cc;
      bs->b3[k] = bs->b3[k] + ct3 * cc;
    }
  }
}

// geometry of pair (i,j): fractional separation (minimum image) and Cartesian
template <bool EXACT>
__device__ __forceinline__ double pair_geom(const double *b, int pbc, double xi, double yi, double zi,
                                            double xj, double yj, double zj, double &dx, double &dy,
                                            double &dz, double &rx, double &ry, double &rz) {
  dx = xi - xj;
  dy = yi - yj;
  dz = zi - zj;
  min_image(pbc, dx, dy, dz);
  rx = b[0] * dx + b[3] * dy + b[6] * dz;
  ry = b[1] * dx + b[4] * dy + b[7] * dz;
  rz = b[2] * dx + b[5] * dy + b[8] * dz;
  return rx * rx + ry * ry + rz * rz;
}

// r and 1/r from r^2: hardware reciprocal square root refined by Newton steps
// (two in FP64, one in FP32) instead of a square root followed by a division.
__device__ __forceinline__ void r_and_inv(double r2, double &r, double &ri) {
  double y = __builtin_amdgcn_rsq(r2);
  const double h = 0.5 * r2;
  y = y * (1.5 - h * y * y);
  y = y * (1.5 - h * y * y);
  ri = y;
  r = r2 * y;
}
__device__ __forceinline__ void r_and_inv(float r2, float &r, float &ri) {
  float y = __builtin_amdgcn_rsqf(r2);
  y = y * (1.5f - 0.5f * r2 * y * y);
  ri = y;
  r = r2 * y;
}

// Pair geometry: Cartesian minimum-image separation R'_i - R'_j + B0 shift (FP64)
// and its square in the arithmetic type T (the FP32 form rounds the components).
template <typename T>
__device__ __forceinline__ T pair_r2(const double (*S)[3], const double4 &pi, const double4 &pj,
                                     int code, T &rx, T &ry, T &rz) {
  rx = (T)(pi.x - pj.x + S[code][0]);
  ry = (T)(pi.y - pj.y + S[code][1]);
  rz = (T)(pi.z - pj.z + S[code][2]);
  return rx * rx + ry * ry + rz * rz;
}

// The same with the FP64 components kept (for FP64 accumulation of forces and
// virial); the arithmetic type T sees them rounded.
template <typename T>
__device__ __forceinline__ T pair_sep(const double (*S)[3], const double4 &pi, const double4 &pj,
                                      int code, double &dx, double &dy, double &dz, T &rx, T &ry,
                                      T &rz) {
  dx = pi.x - pj.x + S[code][0];
  dy = pi.y - pj.y + S[code][1];
  dz = pi.z - pj.z + S[code][2];
  rx = (T)dx;
  ry = (T)dy;
  rz = (T)dz;
  return rx * rx + ry * ry + rz * rz;
}


// Packed positions R (absolute or cell-relative, see the entry format) and the
// current F', for one 32-byte gather per neighbour (16 bytes for the FP32
// copy p4f, when given).
__global__ void k_pack(const double *atoms, const int *img, const BoxState *bs, int n, double4 *pos4, float4 *p4f,
                       const int *cell, PackGeo pg) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double x = atoms[i], y = atoms[(size_t)n + i], z = atoms[2 * (size_t)n + i];
  const double3 r = packed_pos(bs->b0, pg, cell, i, x - img[3 * i], y - img[3 * i + 1], z - img[3 * i + 2]);
  store_packed(pos4, p4f, i, r, atoms[(size_t)F_DAFRHO * n + i]);
}

// Neighbour j's packed position and F': the FP64 record, or (P32) the FP32
// copy of a cell-relative packing, widened exactly.
template <bool P32>
__device__ __forceinline__ double4 partner(const double4 *__restrict__ pos4, const float4 *__restrict__ p4f,
                                           unsigned j) {
  if constexpr (P32) {
    const float4 q = p4f[j];
    return make_double4(q.x, q.y, q.z, q.w);
  } else {
    return pos4[j];
  }
}

// Per-atom end of the density pass: rho, and with do_embed the embedding
// energy F(rho), F'(rho) (also into the packed positions for the force pass);
// returns atom i's embedding energy (0 without do_embed).
__device__ __forceinline__ double density_atom(double *atoms, double4 *pos4, float4 *p4f, int n, int i,
                                               double acc, const PotDev &P, int do_embed) {
  double *rho = atoms + (size_t)F_RHO * n, *af = atoms + (size_t)F_AFRHO * n, *daf = atoms + (size_t)F_DAFRHO * n;
  rho[i] = acc;
  if (!do_embed) return 0.0;
  double dfi = daf[i], pe = 0.0;
  if (acc > 1e-40) {  // src/potential_m.F90:161 leaves stale values below
    double f;
    mdk_embed_f(P, acc, f, dfi);
    af[i] = f;
    daf[i] = dfi;
    pe = f;
  }
  if (pos4) pos4[i].w = dfi;
  if (p4f) p4f[i].w = (float)dfi;
  return pe;
}
// ... and the block's embedding-energy partial
__device__ __forceinline__ void density_finish(double *atoms, double4 *pos4, float4 *p4f, int n, int i,
                                               double acc, const PotDev &P, int do_embed, double *part, int nb,
                                               int b) {
  double pe[1] = {i < n ? density_atom(atoms, pos4, p4f, n, i, acc, P, do_embed) : 0.0};
  if (do_embed) block_store<1, 0>(pe, part, nb, b);
}
// The density passes also complete the previous step's sums where their finishing
// was deferred, and report a new list's flags: MDK_NXCD extra workgroups come
// first, of which one does both (no launches of their own, and it ends before the
// others; whole rounds over the XCDs keep the others' atoms where the force pass
// has them).  DENS_BLOCKS defines this block's index bk of nb among the others.
template <int NT>
__device__ __forceinline__ void finish_ride(const FinRide &R);
__device__ __forceinline__ void report_list(const ListReport &L) {
  if (threadIdx.x != 0) return;
  for (int k = 0; k < 4; k++) L.out[k] = L.flags[k];
  __hip_atomic_store(&L.out[4], L.stamp, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
#define DENS_BLOCKS(R, NT)                                                                            \
  const int nride = R.fin.kind || R.list.stamp ? MDK_NXCD : 0;                                        \
  if ((int)blockIdx.x < nride) {                                                                      \
    if (blockIdx.x == 0 && R.list.stamp) report_list(R.list);                                         \
    if (blockIdx.x == 0 && R.fin.kind) finish_ride<NT>(R.fin);                                        \
    return;                                                                                           \
  }                                                                                                   \
  const Place place = place_of((int)gridDim.x - nride, (int)blockIdx.x - nride, R.one_xcd);           \
  if (place.idle) return;                                                                             \
  const int nb = place.nb, bk = place.b

// Appends entry e as slot m of atom i's list through a register quad; every
// fourth entry stores the quad with one 16-byte write.
__device__ __forceinline__ void quad_put(int *nbr, int i, int n, int e, int &m, int4 &qd) {
  const int sl = m & 3;
  qd.x = sl == 0 ? e : qd.x;
  qd.y = sl == 1 ? e : qd.y;
  qd.z = sl == 2 ? e : qd.z;
  qd.w = sl == 3 ? e : qd.w;
  if (sl == 3) *(int4 *)(nbr + nbr_at(m - 3, i, n)) = qd;
  m++;
}

// the partners of one quad of entries
template <bool P32>
__device__ __forceinline__ void quad_partners(const double4 *pos4, const float4 *p4f, const int4 &e, double4 (&pj)[4]) {
  pj[0] = partner<P32>(pos4, p4f, (unsigned)e.x & NBR_IDX_MASK);
  pj[1] = partner<P32>(pos4, p4f, (unsigned)e.y & NBR_IDX_MASK);
  pj[2] = partner<P32>(pos4, p4f, (unsigned)e.z & NBR_IDX_MASK);
  pj[3] = partner<P32>(pos4, p4f, (unsigned)e.w & NBR_IDX_MASK);
}

// Density pass (rhoset, src/dynamics_m.F90:497-579) fused with embed
// (src/potential_m.F90:148-169): rho_i = sum_j phi(r_ij) over the full list,
// L lanes per atom (pair_lanes); F, F' per atom; per-block embedding energy.
// F' is also stored in pos4[i].w for the force pass.
template <typename T, int POTM, bool P32, int L>
__global__ void __launch_bounds__(MDK_BLOCK) k_density(double *atoms, double4 *pos4, float4 *p4f, int n,
                                                       const int *__restrict__ nbr,
                                                       const int *__restrict__ numn, int maxn,
                                                       const BoxState *bs, PackGeo pg, PotDev P,
                                                       int do_embed, double *part, int *nact, Rider R) {
  DENS_BLOCKS(R, MDK_BLOCK);
  __shared__ double S[32][3];
  const int i = (xcd_tile(nb, bk) * (int)blockDim.x + (int)threadIdx.x) / L, g = threadIdx.x % L;
  // the atom's record, its first quad and (several lanes per atom: mostly its only
  // one) that quad's partners load before the barrier, and later quads' indices a
  // quad ahead: us per step before : after -- iron_carbon 31,250 atoms 47.3 : 45.9,
  // 78,608 85.9 : 83.0; FP64 Fe 78,608 46.8 : 44.8, 524,288 115.4 : 114.3
  double4 pi, pj[4];
  int4 e4 = make_int4(0, 0, 0, 0);
  int nn = 0;
  if (i < n) {
    pi = pos4[i];
    nn = numn[i];
    if (4 * g < maxn) e4 = *(const int4 *)(nbr + (((size_t)g * n + i) << 2));
  }
  if (L > 1 && 4 * g < nn) quad_partners<P32>(pos4, p4f, e4, pj);
  shift_table(bs->b0, pg, S);
  __syncthreads();
  double acc = 0.0;  // per-atom density accumulated in FP64 in both forms
  // list slots up to the end of the last quad holding a partner in range: with
  // a margin of 1e-4 A the force pass's own r of every later pair is beyond the
  // outermost knot, where all pair terms are exactly zero
  const T rc = (T)P.r_int + (T)1e-4, rc2 = rc * rc;
  int na = 0;
  if (i < n) {
    // one 16-byte index load and four independent gathers per quad (quads
    // are padded with null entries)
    for (int q = g; 4 * q < nn; q += L) {
      const unsigned e[4] = {(unsigned)e4.x, (unsigned)e4.y, (unsigned)e4.z, (unsigned)e4.w};
      if (L == 1 || q != g) quad_partners<P32>(pos4, p4f, e4, pj);
      // the next quad's indices load while this quad's partners arrive
      if (4 * (q + L) < nn) e4 = *(const int4 *)(nbr + (((size_t)(q + L) * n + i) << 2));
      T mn = rc2;  // one min chain per quad keeps the register footprint of the loop
#pragma unroll
      for (int u = 0; u < 4; u++) {
        T rx, ry, rz;
        const T r2 = pair_r2<T>(S, pi, pj[u], (int)(e[u] >> NBR_CODE_SHIFT), rx, ry, rz);
        T r, ri;
        r_and_inv(r2, r, ri);
        acc += (double)mdk_pair_phi<T, POTM>(P, r);
        mn = fmin(mn, r2);
      }
      na = mn < rc2 ? 4 * q + 4 : na;
    }
    acc = group_sum<L>(acc);
    na = group_max<L>(na);
    if (g == 0) nact[i] = na;
  }
  density_finish(atoms, pos4, p4f, n, g == 0 ? i : n, acc, P, do_embed, part, nb, bk);
}

// Density pass of the first step on a new list: as k_density, and it also
// reorders each atom's list in place -- the partners in range now (r^2 < rc2,
// the test k_density uses for nact) first, in list order, then the others --
// so that the force pass of this and the following steps stops after the
// in-range part.  Out-of-range entries wait in LDS (DENS_OBUF per lane, more
// stay in place, which costs only efficiency).  Each completed quad is written
// after its slots have been read (an atom's list belongs to its lane alone).
#define DENS_OBUF 16
template <typename T, int POTM, bool P32>
__global__ void __launch_bounds__(MDK_BLOCK) k_density_part(double *atoms, double4 *pos4, float4 *p4f, int n,
                                                            int *nbr, const int *__restrict__ numn,
                                                            const BoxState *bs, PackGeo pg, PotDev P,
                                                            int do_embed, double *part, int *nact, Rider R) {
  DENS_BLOCKS(R, MDK_BLOCK);
  __shared__ double S[32][3];
  __shared__ int obuf[DENS_OBUF][MDK_BLOCK];
  shift_table(bs->b0, pg, S);
  __syncthreads();
  const T rc = (T)P.r_int + (T)1e-4, rc2 = rc * rc;
  const int t = threadIdx.x, i = xcd_tile(nb, bk) * blockDim.x + t;
  double acc = 0.0;
  if (i < n) {
    const double4 pi = pos4[i];
    const int nn = numn[i];
    int m = 0, no = 0, last = 0;  // entries written back, entries held, end of the last in-range one
    int4 qd = make_int4(0, 0, 0, 0);
    for (int q = 0; 4 * q < nn; q++) {
      const int4 e4 = *(const int4 *)(nbr + (((size_t)q * n + i) << 2));
      const int e[4] = {e4.x, e4.y, e4.z, e4.w};
      double4 pj[4];
#pragma unroll
      for (int u = 0; u < 4; u++) pj[u] = partner<P32>(pos4, p4f, (unsigned)e[u] & NBR_IDX_MASK);
#pragma unroll
      for (int u = 0; u < 4; u++) {
        T rx, ry, rz;
        const T r2 = pair_r2<T>(S, pi, pj[u], (int)((unsigned)e[u] >> NBR_CODE_SHIFT), rx, ry, rz);
        T r, ri;
        r_and_inv(r2, r, ri);
        acc += (double)mdk_pair_phi<T, POTM>(P, r);
        if (4 * q + u < nn) {
          const bool in = r2 < rc2;
          if (in || no == DENS_OBUF) {
            quad_put(nbr, i, n, e[u], m, qd);
            if (in) last = m;
          } else {
            obuf[no++][t] = e[u];
          }
        }
      }
    }
    for (int u = 0; u < no; u++) quad_put(nbr, i, n, obuf[u][t], m, qd);
    if (m & 3) {  // the last quad's null entries
      const int nul = i | (NBR_NULL_CODE << NBR_CODE_SHIFT), sl = m & 3;
      qd.y = sl <= 1 ? nul : qd.y;
      qd.z = sl <= 2 ? nul : qd.z;
      qd.w = nul;
      *(int4 *)(nbr + nbr_at(m & ~3, i, n)) = qd;
    }
    nact[i] = (last + 3) & ~3;
  }
  density_finish(atoms, pos4, p4f, n, i, acc, P, do_embed, part, nb, bk);
}

enum { FIN_FORCE = 0, FIN_VV = 1, FIN_VV_THERM = 2, FIN_INIT = 3 };

// update_therm_avs box part (src/dynamics_m.F90:672-700)
__device__ void therm_box(BoxState &s, int ivol) {
#pragma clang fp contract(off)
  for (int k = 0; k < 9; k++) { s.tg[k] = 0.0; s.tgdot[k] = 0.0; }
  for (int i = 1; i <= 3; i++)
    for (int k = 1; k <= 3; k++)
      for (int j = 1; j <= 3; j++) {
        TT(s.tg, i, j) = TT(s.tg, i, j) + TT(s.b0, k, i) * TT(s.b0, k, j);
        if (ivol != 1)
          TT(s.tgdot, i, j) = TT(s.tgdot, i, j) + TT(s.b1, k, i) * TT(s.b0, k, j) + TT(s.b0, k, i) * TT(s.b1, k, j);
      }
  dev_invert(s.tg, s.tginv, &s.status);
  dev_matmul(s.tginv, s.tgdot, s.tgid);
  s.vol = dev_volume(s.b0);
  const double *b = s.b0, v = s.vol;
  TT(s.binv, 1, 1) = (TT(b, 2, 2) * TT(b, 3, 3) - TT(b, 2, 3) * TT(b, 3, 2)) / v;  // xx
  TT(s.binv, 1, 2) = (TT(b, 2, 3) * TT(b, 3, 1) - TT(b, 3, 3) * TT(b, 2, 1)) / v;  // xy
  TT(s.binv, 1, 3) = (TT(b, 2, 1) * TT(b, 3, 2) - TT(b, 3, 1) * TT(b, 2, 2)) / v;  // xz
  TT(s.binv, 2, 1) = (TT(b, 3, 2) * TT(b, 1, 3) - TT(b, 1, 2) * TT(b, 3, 3)) / v;  // yx
  TT(s.binv, 2, 2) = (TT(b, 1, 1) * TT(b, 3, 3) - TT(b, 1, 3) * TT(b, 3, 1)) / v;  // yy
  TT(s.binv, 2, 3) = (TT(b, 3, 1) * TT(b, 1, 2) - TT(b, 1, 1) * TT(b, 3, 2)) / v;  // yz
  TT(s.binv, 3, 1) = (TT(b, 1, 2) * TT(b, 2, 3) - TT(b, 2, 2) * TT(b, 1, 3)) / v;  // zx
  TT(s.binv, 3, 2) = (TT(b, 1, 3) * TT(b, 2, 1) - TT(b, 1, 1) * TT(b, 2, 3)) / v;  // zy
  TT(s.binv, 3, 3) = (TT(b, 1, 1) * TT(b, 2, 2) - TT(b, 1, 2) * TT(b, 2, 1)) / v;  // zz
}

// Stage-and-finish reduction for the finishing kernels, launched as p =
// ceil(nb / 64) blocks of one wave (MDK_FIN_BLOCK).  Block b folds per-block
// partials [64 b, 64 b + 64) lane-wise and across the wave in a fixed order;
// lane 0 writes the K results to stage[k*p + b] and increments the arrival
// counter with one agent-scope release/acquire, so each block makes a single
// L2 write-back and invalidate.  The last block to arrive folds the p stage
// columns the same way into out[] (every lane receives them), resets the
// counter and returns true; the others return false.
#define MDK_FIN_BLOCK 64
template <int K, int KM>
__device__ __forceinline__ void fold_columns(const double *part, int nb, int b0, int b1, double (&v)[K]) {
#pragma unroll
  for (int k = 0; k < K; k++) v[k] = (k < K - KM) ? 0.0 : -HUGE_VAL;
  for (int b = b0 + (int)threadIdx.x; b < b1; b += MDK_FIN_BLOCK) {
#pragma unroll
    for (int k = 0; k < K; k++) {
      const double x = part[(size_t)k * nb + b];
      v[k] = (k < K - KM) ? v[k] + x : fmax(v[k], x);
    }
  }
  wave_reduce_all<K, KM>(v);
}

template <int K, int KM>
__device__ bool stage_and_finish(const double *part, int nb, double *stage, unsigned *cnt, double (&out)[K]) {
  const int p = gridDim.x, b0 = blockIdx.x * 64;
  double v[K];
  fold_columns<K, KM>(part, nb, b0, min(nb, b0 + 64), v);
  int last = 0;
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < K; k++) stage[(size_t)k * p + blockIdx.x] = v[k];
    const unsigned prev = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
    last = prev + 1 == (unsigned)p;
  }
  // one wave: lane 0's verdict to all lanes, which are past lane 0's acquire
  if (!__builtin_amdgcn_readfirstlane(last)) return false;
  fold_columns<K, KM>(stage, p, 0, p, out);
  if (threadIdx.x == 0) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return true;
}

// force()'s partials and the blocks that wrote them
struct ForceParts {
  const double *pair, *emb, *kin;
  int nbp, nbe, nbk;
};
// column c of NSUM_FORCE: its nb values
__device__ __forceinline__ const double *force_column(const ForceParts &P, int c, int &nb) {
  nb = c < PART_EMB ? P.nbp : (c == PART_EMB ? P.nbe : P.nbk);
  return c < PART_EMB ? P.pair + (size_t)c * P.nbp : (c == PART_EMB ? P.emb : P.kin + (size_t)(c - PART_KIN) * P.nbk);
}

// Arguments of the finishing kernels of force().
struct FinForce {
  ForceParts part;
  double *stage;   // ceil(nbp / 64) x NSUM_FORCE first-stage sums
  unsigned *cnt;   // arrival counter, zero between launches
  BoxState *bs;
  int mode, ivol;
  double press, bdel2, dt;
  int one_xcd;     // placement (place_of) of the kernel that finishes and kicks
};

// The box fields and sums of force()'s completion, in LDS: the nine tensor
// threads index them with their own (ii,jj), which private arrays would turn
// into scratch accesses.  b0, b1, b2, tgid0: the box of this force evaluation
// (b1, b2 advanced by complete_force); the rest are results (tgd, tgn: tgdot
// with the old and the new b1).
struct ForceLds {
  double b0[9], b1[9], b2[9], tgid0[9], tg[9], tgd[9], tgn[9], tgi[9], sv[NSUM_FORCE], sbi[9];
  double tp[9], tk[9], tc[9], fb[9], tgid[9], binv[9], vol;
  int singular;
};
__device__ __forceinline__ void load_force_box(const BoxState *bs, ForceLds &s) {
  const int t = threadIdx.x;
  if (t < 9) {
    s.b0[t] = bs->b0[t];
    s.b1[t] = bs->b1[t];
    s.b2[t] = bs->b2[t];
    s.tgid0[t] = bs->tgid[t];
  }
  if (t == 0) s.singular = 0;
}
__device__ void prepare_force(const FinForce &F, ForceLds &s);
__device__ void complete_force(const FinForce &F, ForceLds &s);
__device__ void store_force(const FinForce &F, const ForceLds &s);

// Finishing kernel of force() for large systems, p blocks of one wave (spread
// over many CUs: seventeen columns of thousands of blocks are too much data
// for one), as stage_and_finish: each folds its part of every column, a lane a
// block (p >= the longest column / 64), the last to arrive folds the staged sums
// and completes force().  The partials are in flight during prepare_force.
__global__ void __launch_bounds__(MDK_FIN_BLOCK) k_finalize_force(FinForce F) {
  __shared__ ForceLds s;
  load_force_box(F.bs, s);
  const int p = gridDim.x, lane = threadIdx.x;
  double v[NSUM_FORCE];
#pragma unroll
  for (int c = 0; c < NSUM_FORCE; c++) {
    int nb;
    const double *q = force_column(F.part, c, nb);
    const int per = (nb + p - 1) / p, b = (int)blockIdx.x * per + lane;
    v[c] = lane < per && b < nb ? q[b] : 0.0;
  }
  prepare_force(F, s);
  wave_reduce_all<NSUM_FORCE, 0>(v);
  int last = 0;
  if (lane == 0) {
#pragma unroll
    for (int c = 0; c < NSUM_FORCE; c++) F.stage[(size_t)c * p + blockIdx.x] = v[c];
    const unsigned prev = __hip_atomic_fetch_add(F.cnt, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
    last = prev + 1 == (unsigned)p;
  }
  // one wave: lane 0's verdict to all lanes, which are past lane 0's acquire
  if (!__builtin_amdgcn_readfirstlane(last)) return;
  fold_columns<NSUM_FORCE, 0>(F.stage, p, 0, p, v);
  if (lane == 0) {
    __hip_atomic_store(F.cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int k = 0; k < NSUM_FORCE; k++) s.sv[k] = v[k];
  }
  __syncthreads();
  complete_force(F, s);
  store_force(F, s);
}

// The same for small systems (at most FIN_ONE_BLOCKS blocks of the pair
// passes), one workgroup: a wave per column, no second stage and no arrival
// counter.  Latency bound: one round trip for the partials, then the box
// algebra.  4.3 us against 7.2 for the two-stage form at 2000 atoms, 6.8 : 7.4
// at 31,250.
#define FIN_ONE_THREADS 1024
#define FIN_ONE_BLOCKS 1280
// Every column's sum by one wave (lanes in order, then the wave) into s.sv;
// the first loads of every column are in flight during prepare_force.
template <int NT>
__device__ __forceinline__ void fold_force_columns(const FinForce &F, ForceLds &s) {
  constexpr int NW = NT / 64, NQ = (NSUM_FORCE + NW - 1) / NW;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  double v[NQ];
#pragma unroll
  for (int q = 0; q < NQ; q++) {
    const int c = w + q * NW;
    int nb;
    const double *p = force_column(F.part, c, nb);
    v[q] = c < NSUM_FORCE && lane < nb ? p[lane] : 0.0;
  }
  prepare_force(F, s);
#pragma unroll
  for (int q = 0; q < NQ; q++) {
    const int c = w + q * NW;
    if (c >= NSUM_FORCE) continue;
    int nb;
    const double *p = force_column(F.part, c, nb);
#pragma unroll 4
    for (int b = lane + 64; b < nb; b += 64) v[q] += p[b];
    const double sum = wave_sum(v[q]);
    if (lane == 0) s.sv[c] = sum;
  }
}
__global__ void __launch_bounds__(FIN_ONE_THREADS) k_finalize_force_one(FinForce F) {
  __shared__ ForceLds s;
  load_force_box(F.bs, s);
  fold_force_columns<FIN_ONE_THREADS>(F, s);
  __syncthreads();
  complete_force(F, s);
  store_force(F, s);
}

// Completion of force() in LDS by one workgroup (threads 0..8 each own one
// tensor element (i,j)), in two parts.  prepare_force is what the box alone
// determines, while the partial sums are on their way: B0^-1, the volume, the
// cofactors, the metric tensor and its inverse.  It starts with a barrier (the
// box in LDS).
__device__ __forceinline__ void prepare_force(const FinForce &F, ForceLds &s) {
#pragma clang fp contract(off)  // therm_box's rounding: the step API and the fused step agree bit for bit
  const double(&b0)[9] = s.b0, (&b1)[9] = s.b1;
  const int t = threadIdx.x, ii = t % 3 + 1, jj = t / 3 + 1;  // element (ii,jj) of thread t < 9
  __syncthreads();
  const int other = blockDim.x > 64 ? 64 : 0;  // lanes of another wave where there is one
  if (t == other) inv3(b0, s.sbi);
  if (t >= 9) return;
  const int i1 = ii % 3 + 1, i2 = (ii + 1) % 3 + 1, j1 = jj % 3 + 1, j2 = (jj + 1) % 3 + 1;
  const double cof = TT(b0, i1, j1) * TT(b0, i2, j2) - TT(b0, i1, j2) * TT(b0, i2, j1);
  s.tc[t] = cof;  // cofactor matrix of b0 (dynamics_m.F90:365-373)
  const double vol = dev_volume(b0);
  if (t == 0) s.vol = vol;
  s.binv[t] = cof / vol;  // update_therm_avs's b0_XXdet ... (dynamics_m.F90:692-700)
  double tg[9], tgdv = 0.0;
#pragma unroll
  for (int c = 0; c < 9; c++) {
    double v = 0.0;
    for (int k = 1; k <= 3; k++) v += TT(b0, k, c % 3 + 1) * TT(b0, k, c / 3 + 1);
    tg[c] = v;
  }
  for (int k = 1; k <= 3; k++) tgdv = tgdv + TT(b0, k, ii) * TT(b1, k, jj) + TT(b1, k, ii) * TT(b0, k, jj);
  s.tgd[t] = tgdv;  // kinten's tgdot
#pragma unroll
  for (int c = 0; c < 9; c++)
    if (c == t) s.tg[t] = tg[c];
  const double det = TT(tg, 1, 1) * (TT(tg, 2, 2) * TT(tg, 3, 3) - TT(tg, 2, 3) * TT(tg, 3, 2)) +
                     TT(tg, 2, 1) * (TT(tg, 3, 2) * TT(tg, 1, 3) - TT(tg, 1, 2) * TT(tg, 3, 3)) +
                     TT(tg, 3, 1) * (TT(tg, 1, 2) * TT(tg, 2, 3) - TT(tg, 2, 2) * TT(tg, 1, 3));
  if (t == 0 && fabs(det) == 0.0) s.singular = 1;
  // inverse of tg, element (ii,jj): cofactor(jj,ii)/det, the cofactor of a
  // matrix element chosen by the thread (no dynamic index into registers)
  double c9[9];
#pragma unroll
  for (int c = 0; c < 9; c++) {
    const int r = c % 3 + 1, q = c / 3 + 1;  // element (r,q) of the inverse
    const int a1 = q % 3 + 1, a2 = (q + 1) % 3 + 1, d1 = r % 3 + 1, d2 = (r + 1) % 3 + 1;
    c9[c] = TT(tg, a1, d1) * TT(tg, a2, d2) - TT(tg, a1, d2) * TT(tg, a2, d1);
  }
  double ct = c9[0];
#pragma unroll
  for (int c = 1; c < 9; c++) ct = c == t ? c9[c] : ct;
  s.tgi[t] = ct / det;
}
// complete_force is the rest, after a barrier behind the sums sv: tp, tk, tc, fb
// (dynamics_m.F90:365-394), then per mode the velocity-Verlet box kick
// (quench_m.F90:595-604), the initial tgid/b2 (moldin.F90:452-477) or the
// update_therm_avs box part (dynamics_m.F90:672-700).  It ends with a barrier.
__device__ __forceinline__ void complete_force(const FinForce &F, ForceLds &s) {
#pragma clang fp contract(off)
  double(&b0)[9] = s.b0, (&b1)[9] = s.b1;
  const int mode = F.mode, ivol = F.ivol;
  const int t = threadIdx.x, ii = t % 3 + 1, jj = t / 3 + 1;
  if (t < 9) {
    // W = 1/2 sum r r^T fp (symmetric; sv[1..6] = xx yy zz xy xz yz) ->
    // tp(a,c) = sum_k W(a,k) B0^-1(c,k)
    double tpv = 0.0;
    for (int k = 1; k <= 3; k++) {
      const int w = ii == k ? ii : (ii + k == 3 ? 4 : (ii + k == 4 ? 5 : 6));
      tpv += s.sv[w] * TT(s.sbi, jj, k);
    }
    const double tkv = s.sv[PART_KIN + t] / (F.dt * F.dt);
    const double fbv = tkv + tpv - F.press * s.tc[t];
    s.tp[t] = tpv;
    s.tk[t] = tkv;
    s.fb[t] = fbv;
    if (mode == FIN_VV || mode == FIN_VV_THERM) {
      const bool upd = ivol < 1 || (ivol == 4 && t == 8);
      if (upd) {
        const double b2v = F.bdel2 * fbv;
        s.b2[t] = b2v;
        b1[t] = b1[t] + b2v;
      }
    } else if (mode == FIN_INIT) {
      s.b2[t] = F.bdel2 * fbv;
    }
  }
  __syncthreads();
  if (mode != FIN_VV_THERM && mode != FIN_INIT) return;
  // tgid = tginv tgdot, with update_therm_avs's tgdot of the new b1 (VV_THERM)
  // or kinten's (INIT, moldin's first tgid)
  if (t < 9) {
    double g = 0.0;
    for (int k = 1; k <= 3; k++) {
      double d = 0.0;
      if (mode == FIN_INIT) {
        d = s.tgd[3 * (jj - 1) + k - 1];
      } else if (ivol != 1) {
        for (int q = 1; q <= 3; q++) d = d + TT(b1, q, k) * TT(b0, q, jj) + TT(b0, q, k) * TT(b1, q, jj);
      }
      if (mode == FIN_VV_THERM && k == ii) s.tgn[t] = d;
      g += TT(s.tgi, ii, k) * d;
    }
    s.tgid[t] = g;
  }
  __syncthreads();
}
// ... and its results into the box state: only the fields that change
__device__ void store_force(const FinForce &F, const ForceLds &s) {
  BoxState *bs = F.bs;
  const int t = threadIdx.x, mode = F.mode;
  const bool vv = mode == FIN_VV || mode == FIN_VV_THERM, therm = mode == FIN_VV_THERM;
  if (t == 0) {
    bs->pe_emb = s.sv[PART_EMB];
    bs->pe = s.sv[PART_EMB] + s.sv[0];
    bs->vol = s.vol;
    if (s.singular) bs->status = MDK_ERR_SINGULAR_BOX;
  }
  if (t < 9) {
    bs->tp[t] = s.tp[t];
    bs->tk[t] = s.tk[t];
    bs->tc[t] = s.tc[t];
    bs->fb[t] = s.fb[t];
    if (mode != FIN_VV) {
      bs->tg[t] = s.tg[t];
      bs->tgdot[t] = therm ? s.tgn[t] : s.tgd[t];
    }
    if (vv) {
      bs->tgid_lag[t] = s.tgid0[t];
      bs->b1[t] = s.b1[t];
    }
    if (vv || mode == FIN_INIT) bs->b2[t] = s.b2[t];
    if (therm || mode == FIN_INIT) {
      bs->tginv[t] = s.tgi[t];
      bs->tgid[t] = s.tgid[t];
    }
    if (therm) bs->binv[t] = s.binv[t];
  }
}
// The box state after the fused finishing and kick (FIN_VV_THERM) into another
// copy, one word per thread: bin with the fields store_force would change; with
// drift also b0 += b1 + b2, b1 += b2 as drift_box.
__device__ void store_box(const FinForce &F, const ForceLds &s, BoxState *out, bool drift) {
#pragma clang fp contract(off)
  const double *src = (const double *)F.bs;
  double *dst = (double *)out;
  auto at = [](size_t off) { return (int)(off / sizeof(double)); };
  for (int w = threadIdx.x; w < (int)(sizeof(BoxState) / sizeof(double)); w += blockDim.x) {
    double val = src[w];
    auto field = [&](size_t off, const double *f) {
      const int k = w - at(off);
      if (k >= 0 && k < 9) val = f[k];
    };
    field(offsetof(BoxState, tp), s.tp);
    field(offsetof(BoxState, tk), s.tk);
    field(offsetof(BoxState, tc), s.tc);
    field(offsetof(BoxState, fb), s.fb);
    field(offsetof(BoxState, tg), s.tg);
    field(offsetof(BoxState, tgdot), s.tgn);
    field(offsetof(BoxState, tgid_lag), s.tgid0);
    field(offsetof(BoxState, tginv), s.tgi);
    field(offsetof(BoxState, tgid), s.tgid);
    field(offsetof(BoxState, binv), s.binv);
    field(offsetof(BoxState, b1), s.b1);
    field(offsetof(BoxState, b2), s.b2);
    if (w == at(offsetof(BoxState, pe_emb))) val = s.sv[PART_EMB];
    if (w == at(offsetof(BoxState, pe))) val = s.sv[PART_EMB] + s.sv[0];
    if (w == at(offsetof(BoxState, vol))) val = s.vol;
    if (drift) {
      const int f = w - at(offsetof(BoxState, b0)), g = w - at(offsetof(BoxState, b1));
      if (f >= 0 && f < 9 && (F.ivol < 1 || (F.ivol == 4 && f == 8))) val = s.b0[f] + (s.b1[f] + s.b2[f]);
      if (g >= 0 && g < 9 && (F.ivol < 1 || (F.ivol == 4 && g == 8))) val = s.b1[g] + s.b2[g];
    }
    if (w == at(offsetof(BoxState, status)) && s.singular) {
      const int st[2] = {MDK_ERR_SINGULAR_BOX, 0};
      memcpy(&val, st, sizeof(val));
    }
    dst[w] = val;
  }
}

// Completion of a step's sums by one workgroup of NT threads: s1,s2,s3, KE, box
// KE, TE, H, TH (moldin.F90:763-790), the trace row and the host-visible skin
// monitor.  Thread t folds blocks t, t + NT, ... in order, then the lanes of
// each wave and the waves in index order; one memory round trip.  After a
// fixed-box step (kind 2) the box, its metric and the forces' virial are as they
// were or not read before the next plain step: the energies change besides.  The
// tensors pass through LDS: in registers they would halve the occupancy of the
// density passes, which have this code in them.
template <int NT>
__device__ __forceinline__ void finish_ride(const FinRide &R) {
#pragma clang fp contract(off)
  __shared__ double sh[NT / 64][NPART_KICK], sb[4][9];
  const FinKick &F = R.kick;
  BoxState *bs = F.bs;
  const int t = threadIdx.x;
  if (t < 9) {
    sb[0][t] = bs->b0[t];
    sb[1][t] = bs->b1[t];
    sb[2][t] = bs->b2[t];
    sb[3][t] = bs->bref[t];
  }
  // columns: s1 or (kind 2) the embedding energy, s2 or the pair energy, s3, and two maxima
  const bool fixed = R.kind == 2;
  const double *col0 = fixed ? R.emb : R.part, *col1 = fixed ? R.part : R.part + R.nb;
  const int nb0 = fixed ? R.nbe : R.nb;
  double v[NPART_KICK] = {0.0, 0.0, 0.0, -HUGE_VAL, -HUGE_VAL};
  for (int b = t; b < R.nb; b += NT) {
    v[1] += col1[b];
    v[2] += col1[(size_t)R.nb + b];
    v[3] = fmax(v[3], col1[(size_t)2 * R.nb + b]);
    v[4] = fmax(v[4], col1[(size_t)3 * R.nb + b]);
  }
  for (int b = t; b < nb0; b += NT) v[0] += col0[b];
  wave_reduce_all<NPART_KICK, 2>(v);
  if ((t & 63) == 0) {
#pragma unroll
    for (int k = 0; k < NPART_KICK; k++) sh[t >> 6][k] = v[k];
  }
  __syncthreads();
  if (F.mon && t < 9) {  // the host forms the box strains from B0, b1 + b2 and Bref
    F.mon[MON_B0 + t] = sb[0][t];
    F.mon[MON_DB + t] = sb[1][t] + sb[2][t];
    F.mon[MON_BREF + t] = sb[3][t];
  }
  if (t < NPART_KICK) {
    double s = sh[0][t];
#pragma unroll 1
    for (int q = 1; q < NT / 64; q++) s = t < 3 ? s + sh[q][t] : fmax(s, sh[q][t]);
    sh[0][t] = s;
  }
  __syncthreads();
  if (t != 0) return;
#pragma unroll
  for (int k = 0; k < NPART_KICK; k++) v[k] = sh[0][k];
  double pe, vol;
  if (fixed) {
    pe = v[0] + v[1];
    vol = dev_volume(sb[0]);
    bs->pe_emb = v[0];
    bs->pe = pe;
    bs->vol = vol;
  } else {
    pe = bs->pe;
    vol = bs->vol;
  }
  const double ke = v[2] / (F.dt * F.dt) / 2.0;
  double bk = 0.0;
#pragma unroll 1
  for (int q = 0; q < 9; q++) {  // rows, then columns
    const double e = TT(sb[1], q / 3 + 1, q % 3 + 1);
    bk = bk + (e * e) / F.bdel2;
  }
  const double te = ke + pe, hh = te + F.press * vol, th = hh + bk;
  for (BoxState *o : {bs, F.bout}) {  // the fused drift's copy was taken before these sums
    if (!o) continue;
    if (!fixed) {
      o->s1 = v[0];
      o->s2 = v[1];
    }
    o->s3 = v[2];
    o->maxdisp2 = v[3];
    o->maxstep2 = v[4];
    o->ke = ke;
    o->boxke = bk;
    o->te = te;
    o->h = hh;
    o->th = th;
  }
  if (F.trace_row) {
    F.trace_row[0] = pe; F.trace_row[1] = ke; F.trace_row[2] = te;
    F.trace_row[3] = hh; F.trace_row[4] = th; F.trace_row[5] = vol;
  }
  if (F.mon) {
    F.mon[0] = v[3];
    F.mon[1] = v[4];
    __hip_atomic_store(&F.mon[MON_STAMP], F.stamp, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}
#define FINISH_THREADS 1024
__global__ void __launch_bounds__(FINISH_THREADS) k_finish_step(FinRide R) { finish_ride<FINISH_THREADS>(R); }

// What the half kick reads of one atom, and the tensors of the box it uses.
struct KickAtom {
  double x0, y0, z0, x1, y1, z1, x2, y2, z2, fx, fy, fz, m, d2;
  float r0, r1, r2;
  int z, im0, im1, im2;
  unsigned ck;
};
struct KickBox {
  const double *lag, *tgid, *binv, *b0, *b1, *b2;
};
// Every per-atom load is issued here, before the first store: the fields
// share one allocation, so a load written after a store to another field
// could not be moved ahead of it, and each would cost a round trip of its own.
// FORCE: with the force fields (a fused force pass has them in registers)
template <bool DRIFT, bool FORCE>
__device__ __forceinline__ KickAtom load_kick(const double *__restrict__ atoms, const int *__restrict__ zat, int n, int i,
                                              const float *__restrict__ sref, const int *__restrict__ img,
                                              const int *__restrict__ cell, const PackGeo &pg,
                                              const double *__restrict__ spec) {
  auto f = [&](int k) { return atoms[(size_t)k * n + i]; };
  KickAtom a;
  a.z = zat[i];
  a.x1 = f(F_X1); a.y1 = f(F_Y1); a.z1 = f(F_Z1);
  a.x2 = f(F_X2); a.y2 = f(F_Y2); a.z2 = f(F_Z2);
  a.fx = a.fy = a.fz = 0.0;
  if (FORCE) {
    a.fx = f(F_FX);
    a.fy = f(F_FY);
    a.fz = f(F_FZ);
  }
  a.x0 = f(F_X0); a.y0 = f(F_Y0); a.z0 = f(F_Z0);
  a.im0 = a.im1 = a.im2 = 0;
  a.ck = 0u;
  if (DRIFT) {
    if (pg.gx) {  // the images follow from the cell (near_image)
      a.ck = (unsigned)cell[i];
    } else {
      a.im0 = img[3 * i];
      a.im1 = img[3 * i + 1];
      a.im2 = img[3 * i + 2];
    }
  }
  a.r0 = a.r1 = a.r2 = 0.f;
  if (sref) {
    a.r0 = sref[3 * i];
    a.r1 = sref[3 * i + 1];
    a.r2 = sref[3 * i + 2];
  }
  // mass and del2 from the species table when they are functions of the
  // species: both rows (Fe and vacancies, the only ones) by uniform loads, so
  // that no load waits for the atom's species
  if (spec) {
    const double m26 = spec[2 * 26], d26 = spec[2 * 26 + 1], m0 = spec[0], d0 = spec[1];
    a.m = a.z == 0 ? m0 : m26;
    a.d2 = a.z == 0 ? d0 : d26;
  } else {
    a.m = f(F_MASS);
    a.d2 = f(F_DEL2);
  }
  return a;
}

// Velocity half-kick (src/quench_m.F90:604-622) of one atom, its sums of
// update_therm_avs (src/dynamics_m.F90:702-732) in v[0..2] and of the list-skin
// monitor in v[3..4].
// mode 0: VV kick + sums; 1: sums only; 2: initial accelerations (moldin.F90:461-472)
// DRIFT (mode 0 only) fuses the next step's drift: x0 += x1 + x2 with the new
// velocities, packed positions with the advanced box and kinten's terms of the
// next force evaluation in kv -- what k_drift would do at the start of the
// next step; where this step ends with a relink, the link cells of its positions
// come first.  FIXED: a box that does not move (no tgid term), without s1 and s2.
template <bool DRIFT, bool FIXED>
__device__ __forceinline__ void kick_atom(KickAtom a, const KickBox &B, int i, int n, int ivol, int mode, bool monitor,
                                          double *__restrict__ atoms, double4 *pos4, float4 *p4f, const PackGeo &pg,
                                          const LinkGrid &link, double (&v)[NPART_KICK], double (&kv)[9]) {
#pragma clang fp contract(off)
  double x1 = a.x1, y1 = a.y1, z1 = a.z1, x2 = a.x2, y2 = a.y2, z2 = a.z2;
  auto put = [&](int k, double val) { atoms[(size_t)k * n + i] = val; };
  const int z = a.z;
  if (mode == 0) {
    const double *g = B.lag;
    const double xd = x1 + x2, yd = y1 + y2, zd = z1 + z2;  // x1_dt2
    if (!(z == 0 || a.m < (double)0.1f)) {
      double sx = 0.0, sy = 0.0, sz = 0.0;
      if (!FIXED && ivol == 0) {
        sx = TT(g, 1, 1) * x1 + TT(g, 1, 2) * y1 + TT(g, 1, 3) * z1;
        sy = TT(g, 2, 1) * x1 + TT(g, 2, 2) * y1 + TT(g, 2, 3) * z1;
        sz = TT(g, 3, 1) * x1 + TT(g, 3, 2) * y1 + TT(g, 3, 3) * z1;
      }
      if (!FIXED && ivol == 4) sz = TT(g, 3, 3) * z1;
      x2 = a.d2 * a.fx - 0.5 * sx;
      y2 = a.d2 * a.fy - 0.5 * sy;
      z2 = a.d2 * a.fz - 0.5 * sz;
      put(F_X2, x2); put(F_Y2, y2); put(F_Z2, z2);
    }
    x1 = xd + x2; y1 = yd + y2; z1 = zd + z2;
    put(F_X1, x1); put(F_Y1, y1); put(F_Z1, z1);
  } else if (mode == 2) {
    if (z != 0) {
      const double *g = B.tgid;
      double a1 = TT(g, 1, 1) * x1 + TT(g, 1, 2) * y1 + TT(g, 1, 3) * z1;
      double a2 = TT(g, 2, 1) * x1 + TT(g, 2, 2) * y1 + TT(g, 2, 3) * z1;
      double a3 = TT(g, 3, 1) * x1 + TT(g, 3, 2) * y1 + TT(g, 3, 3) * z1;
      x2 = a.d2 * a.fx - 0.5 * a1;
      y2 = a.d2 * a.fy - 0.5 * a2;
      z2 = a.d2 * a.fz - 0.5 * a3;
      put(F_X2, x2); put(F_Y2, y2); put(F_Z2, z2);
    }
  }
  const double *b = B.b0;
  if (mode != 2 && z != 0) {
    const double *g = B.tgid, *bi = B.binv;
    if (!FIXED) {
      double sx = TT(g, 1, 1) * x1 + TT(g, 1, 2) * y1 + TT(g, 1, 3) * z1;
      double sy = TT(g, 2, 1) * x1 + TT(g, 2, 2) * y1 + TT(g, 2, 3) * z1;
      double sz = TT(g, 3, 1) * x1 + TT(g, 3, 2) * y1 + TT(g, 3, 3) * z1;
      double fxq = 2.0 * x2 + sx, fyq = 2.0 * y2 + sy, fzq = 2.0 * z2 + sz;
      double fxi = TT(bi, 1, 1) * fxq + TT(bi, 1, 2) * fyq + TT(bi, 1, 3) * fzq;
      double fyi = TT(bi, 2, 1) * fxq + TT(bi, 2, 2) * fyq + TT(bi, 2, 3) * fzq;
      double fzi = TT(bi, 3, 1) * fxq + TT(bi, 3, 2) * fyq + TT(bi, 3, 3) * fzq;
      double f2 = fxi * fxi + fyi * fyi + fzi * fzi;
      v[0] = f2;
      v[1] = f2 * f2;
    }
    double rx = TT(b, 1, 1) * x1 + TT(b, 1, 2) * y1 + TT(b, 1, 3) * z1;
    double ry = TT(b, 2, 1) * x1 + TT(b, 2, 2) * y1 + TT(b, 2, 3) * z1;
    double rz = TT(b, 3, 1) * x1 + TT(b, 3, 2) * y1 + TT(b, 3, 3) * z1;
    v[2] = a.m * (rx * rx + ry * ry + rz * rz);
  }
  if (monitor) {
    double ex = a.x0 - (double)a.r0, ey = a.y0 - (double)a.r1, ez = a.z0 - (double)a.r2;
    double qx = b[0] * ex + b[3] * ey + b[6] * ez, qy = b[1] * ex + b[4] * ey + b[7] * ez,
           qz = b[2] * ex + b[5] * ey + b[8] * ez;
    v[3] = qx * qx + qy * qy + qz * qz;
    double sx = x1 + x2, sy = y1 + y2, sz = z1 + z2;
    qx = b[0] * sx + b[3] * sy + b[6] * sz;
    qy = b[1] * sx + b[4] * sy + b[7] * sz;
    qz = b[2] * sx + b[5] * sy + b[8] * sz;
    v[4] = qx * qx + qy * qy + qz * qz;
  }
  if (DRIFT) {
    if (link.ic) put_link_cell(link, i, a.x0, a.y0, a.z0);
    const double xn = a.x0 + (x1 + x2), yn = a.y0 + (y1 + y2), zn = a.z0 + (z1 + z2);
    put(F_X0, xn);
    put(F_Y0, yn);
    put(F_Z0, zn);
    double bn[9];
    for (int k = 0; k < 9; k++) {
      const bool upd = !FIXED && (ivol < 1 || (ivol == 4 && k == 8));
      bn[k] = upd ? b[k] + (B.b1[k] + B.b2[k]) : b[k];
    }
    double3 im = make_double3(a.im0, a.im1, a.im2);
    if (pg.gx) im = near_image(pg, a.ck, xn, yn, zn);
    const double3 r = packed_pos_key(bn, pg, a.ck, xn - im.x, yn - im.y, zn - im.z);
    store_packed(pos4, p4f, i, r, 0.0);  // F' is stored by the density pass, which always runs next
    if (z != 0) kin_terms(bn, x1, y1, z1, a.m, kv);  // kinten of the next force evaluation
  }
}

// The half kick and drift of a force pass in a fixed box: inputs, the next
// step's packed positions, the partials (NPART_FIXED) and, where the next force
// evaluation finishes with kinten, its partials.
struct KickIo {
  const int *zat;
  const float *sref;
  const int *img, *cell;
  const double *spec;
  double4 *pos4;
  float4 *p4f;
  double *part, *kin;
  int ivol;
  LinkGrid link;
  int one_xcd;  // the pass's placement (place_of)
};
template <int NT>
__device__ __forceinline__ void fixed_kick(KickAtom a, const KickIo &K, const BoxState *bs, int i, int n, bool own,
                                           double pe, double fx, double fy, double fz, double *atoms,
                                           const PackGeo &pg, int nb, int bk) {
  double v[NPART_KICK] = {0.0, 0.0, 0.0, 0.0, 0.0}, kv[9] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  if (own) {
    const KickBox B = {nullptr, nullptr, nullptr, bs->b0, bs->b1, bs->b2};
    a.fx = fx;
    a.fy = fy;
    a.fz = fz;
    kick_atom<true, true>(a, B, i, n, K.ivol, 0, true, atoms, K.pos4, K.p4f, pg, K.link, v, kv);
  }
  double o[NPART_FIXED] = {pe, v[2], v[3], v[4]};
  block_store<NPART_FIXED, 2, NT>(o, K.part, nb, bk);
  if (K.kin) block_store<9, 0, NT>(kv, K.kin, nb, bk);
}

// Force pass (src/dynamics_m.F90:235-346); kinten's partial sums come from
// the kernel that last set the velocities (kin_terms).
// fp = -(V' + phi'(F'_i + F'_j))/r;  F_i = sum_j r_ij fp (Cartesian) and
// f_i = B0^-1 F_i;  the virial is accumulated as W = 1/2 sum r r^T fp (tp =
// W B0^-T in the finishing block, i.e. sum r_a s_b fp) and the pair energy as
// 1/2 sum V.  L lanes per atom (pair_lanes); MASSCHK keeps the
// reference's exclusion of pairs of immobile atoms from the virial.
// KICK (steps in a box that does not move, between two others of one call):
// the half kick and the next drift follow in the same kernel, from the force in
// registers -- the velocity update needs no sum over atoms there.  The forces
// themselves and the virial, which nothing reads before the next plain step,
// are not formed for memory.  It saves a launch, the finishing between the two,
// the force's round trip (48 B per atom) and idle memory pipes in the pair loop.
// us per NVE step, separate : fused -- 2000 atoms (FP64) 21.5 : 15.3, 31,250
// 32.2 : 25.7 (FP32 30.3 : 22.0), 524,288 117 : 95 (91 : 74); 3,456,000 FP32 force
// 135 + finishing 14 + kick 131 : 219.
template <typename T, bool MASSCHK, int POTM, bool P32, int L, bool KICK>
__global__ void __launch_bounds__(MDK_BLOCK)
k_force(double *atoms, const double4 *__restrict__ pos4, const float4 *__restrict__ p4f, int n, const int *__restrict__ nbr, const int *__restrict__ nvisit, int maxn, const BoxState *bs, PackGeo pg,
        PotDev P, double *part, const float *fetab, KickIo K) {
  __shared__ double S[32][3];
  // interval table of the FP32 Fe-Fe pair terms: bin records, then intervals
  __shared__ float4 fbin[MDK_FE_NB];
  __shared__ __align__(16) float fiv[8 * MDK_FE_NI];
  constexpr bool CUBIC = sizeof(T) == 4 && POTM == POT_FE;
  const Place place = place_of(gridDim.x, blockIdx.x, K.one_xcd);
  if (place.idle) return;
  const int i = (xcd_tile(place.nb, place.b) * (int)blockDim.x + (int)threadIdx.x) / L, g = threadIdx.x % L;
  double4 pi, pj[4];  // loaded ahead as in k_density
  int4 e4 = make_int4(0, 0, 0, 0);
  int nn = 0;  // list slots that can hold a partner in range
  if (i < n) {
    pi = pos4[i];
    nn = nvisit[i];
    if (4 * g < maxn) e4 = *(const int4 *)(nbr + (((size_t)g * n + i) << 2));
  }
  KickAtom ka;
  // small systems: the kick's loads arrive during the pair loop
  if (KICK && L > 1 && i < n && g == 0) ka = load_kick<true, false>(atoms, K.zat, n, i, K.sref, K.img, K.cell, pg, K.spec);
  if (L > 1 && 4 * g < nn) quad_partners<P32>(pos4, p4f, e4, pj);
  double b[9];
#pragma unroll
  for (int k = 0; k < 9; k++) b[k] = bs->b0[k];
  __shared__ double bi[9];  // B0^-1 for the fractional forces
  shift_table(b, pg, S);
  if (CUBIC) {
    const float4 *src = (const float4 *)fetab;
    if (threadIdx.x < MDK_FE_NB) fbin[threadIdx.x] = src[threadIdx.x];
    else if (threadIdx.x < MDK_FE_NB + 2 * MDK_FE_NI)
      ((float4 *)fiv)[threadIdx.x - MDK_FE_NB] = src[threadIdx.x];
  }
  if (threadIdx.x == 64) inv3(b, bi);
  __syncthreads();
  const double *mass = atoms + (size_t)F_MASS * n;
  double v[NPART_FORCE];
#pragma unroll
  for (int k = 0; k < NPART_FORCE; k++) v[k] = 0.0;
  double fxi = 0.0, fyi = 0.0, fzi = 0.0;  // Cartesian force on i
  if (i < n) {
    const T dfi = (T)pi.w;
    const double mi = MASSCHK ? mass[i] : 0.0;
    // sums of V and of r r^T fp; the factor 1/2 of both is applied once below
    double pe2 = 0.0, wxx = 0, wyy = 0, wzz = 0, wxy = 0, wxz = 0, wyz = 0;
    for (int q = g; 4 * q < nn; q += L) {
      const unsigned e[4] = {(unsigned)e4.x, (unsigned)e4.y, (unsigned)e4.z, (unsigned)e4.w};
      if (L == 1 || q != g) quad_partners<P32>(pos4, p4f, e4, pj);
      if (4 * (q + L) < nn) e4 = *(const int4 *)(nbr + (((size_t)(q + L) * n + i) << 2));
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const unsigned eu = e[u];
        const int j = (int)(eu & NBR_IDX_MASK);
        double dx, dy, dz;
        T rx, ry, rz;
        const T r2 = pair_sep<T>(S, pi, pj[u], (int)(eu >> NBR_CODE_SHIFT), dx, dy, dz, rx, ry, rz);
        T r, rr;
        r_and_inv(r2, r, rr);
        T vv, dv, dph;
        if constexpr (CUBIC) {
          mdk_fe_terms(P, fbin, fiv, r, vv, dv, dph);
        } else {
          mdk_pair_vdv<T, POTM>(P, r, vv, dv);
          dph = mdk_pair_dphi<T, POTM>(P, r);
        }
        const T fp = -dv * rr + (-T(1) * (dph * dfi + dph * (T)pj[u].w) * rr);
        const double fpd = (double)fp;
        // FP32 Fe-Fe form: the force and virial sums take the FP32 separation
        // (widened exactly), which frees the FP64 one early: 93 VGPRs and five
        // waves per SIMD instead of 106 and four; its rounding (6e-8 relative)
        // is far below the form's force error
        if constexpr (CUBIC) { dx = (double)rx; dy = (double)ry; dz = (double)rz; }
        const double gx = dx * fpd, gy = dy * fpd, gz = dz * fpd;
        pe2 += (double)vv;
        fxi += gx;
        fyi += gy;
        fzi += gz;
        if (!KICK && (!MASSCHK || mi + mass[j] > (double)0.1f)) {
          wxx += dx * gx; wyy += dy * gy; wzz += dz * gz;
          wxy += dx * gy; wxz += dx * gz; wyz += dy * gz;
        }
      }
    }
    v[0] = 0.5 * pe2;
    v[1] = 0.5 * wxx; v[2] = 0.5 * wyy; v[3] = 0.5 * wzz;
    v[4] = 0.5 * wxy; v[5] = 0.5 * wxz; v[6] = 0.5 * wyz;
  }
  if (L > 1 && i < n) {
    fxi = group_sum<L>(fxi);
    fyi = group_sum<L>(fyi);
    fzi = group_sum<L>(fzi);
  }
  // fractional force f = B0^-1 F (the reference's fx = sum s fp, Cartesian = B0 f)
  const double f0 = bi[0] * fxi + bi[3] * fyi + bi[6] * fzi, f1 = bi[1] * fxi + bi[4] * fyi + bi[7] * fzi,
               f2 = bi[2] * fxi + bi[5] * fyi + bi[8] * fzi;
  const bool own = i < n && g == 0;
  if constexpr (KICK) {
    if (L == 1 && own) ka = load_kick<true, false>(atoms, K.zat, n, i, K.sref, K.img, K.cell, pg, K.spec);
    fixed_kick<MDK_BLOCK>(ka, K, bs, i, n, own, v[0], f0, f1, f2, atoms, pg, place.nb, place.b);
  } else {
    if (own) {
      atoms[(size_t)F_FX * n + i] = f0;
      atoms[(size_t)F_FY * n + i] = f1;
      atoms[(size_t)F_FZ * n + i] = f2;
    }
    block_store<NPART_FORCE, 0>(v, part, place.nb, place.b);
  }
}

// ---------------------------------------------------------------------------
// FP32 Fe-Fe pair passes on cell-relative block lists (the FP32 form's main
// path).  Both atoms of a pair come from the 16-byte FP32 packed records and
// the separation (R_i - R_j) + D[code] is formed in FP32; r and 1/r come from
// the hardware reciprocal square root with one Newton step.  L lanes per atom
// (pair_lanes).
// ---------------------------------------------------------------------------
// D[code] as an unevaluated FP32 sum hi + lo: a rounded D would bias every
// separation of one cell offset the same way (pairs (i,j) and (j,i) alike),
// and that bias adds up in the energy; ((R_i - R_j) + hi) + lo does not.
__device__ __forceinline__ void shift_table_f32(const double (*S)[3], float4 *Sf, float4 *Sl) {
  for (int c = threadIdx.x; c < 32; c += blockDim.x) {
    const float hx = (float)S[c][0], hy = (float)S[c][1], hz = (float)S[c][2];
    Sf[c] = make_float4(hx, hy, hz, 0.f);
    Sl[c] = make_float4((float)(S[c][0] - hx), (float)(S[c][1] - hy), (float)(S[c][2] - hz), 0.f);
  }
}
__device__ __forceinline__ float pair_r2_f32(const float4 &pi, const float4 &pj, const float4 *Sf,
                                             const float4 *Sl, unsigned e, float &rx, float &ry, float &rz) {
  const float4 d = Sf[e >> NBR_CODE_SHIFT], dl = Sl[e >> NBR_CODE_SHIFT];
  rx = ((pi.x - pj.x) + d.x) + dl.x;
  ry = ((pi.y - pj.y) + d.y) + dl.y;
  rz = ((pi.z - pj.z) + d.z) + dl.z;
  return rx * rx + ry * ry + rz * rz;
}

__device__ __forceinline__ void quad_partners_f32(const float4 *p4f, const int4 &e, float4 (&pj)[4]) {
  pj[0] = p4f[(unsigned)e.x & NBR_IDX_MASK];
  pj[1] = p4f[(unsigned)e.y & NBR_IDX_MASK];
  pj[2] = p4f[(unsigned)e.z & NBR_IDX_MASK];
  pj[3] = p4f[(unsigned)e.w & NBR_IDX_MASK];
}

// Density pass (rhoset + embed, src/dynamics_m.F90:497-579,
// src/potential_m.F90:148-169): phi in FP32, each atom's density summed in
// FP64; nact[i] = list slots up to the end of the last quad holding a partner
// within r_int + 1e-4 A (the force pass's visit length).
template <int L>
__global__ void __launch_bounds__(MDK_BLOCK) k_density_f32(double *atoms, double4 *pos4, float4 *p4f, int n,
                                                           const int *__restrict__ nbr,
                                                           const int *__restrict__ numn, int maxn, const BoxState *bs,
                                                           PackGeo pg, PotDev P, int do_embed, double *part,
                                                           int *nact, Rider R) {
  DENS_BLOCKS(R, MDK_BLOCK);
  __shared__ double S[32][3];
  __shared__ float4 Sf[32], Sl[32];
  const int i = (xcd_tile(nb, bk) * (int)blockDim.x + (int)threadIdx.x) / L, g = threadIdx.x % L;
  float4 pi, pj[4];  // loaded ahead as in k_density
  int4 e4 = make_int4(0, 0, 0, 0);
  int nn = 0;
  if (i < n) {
    pi = p4f[i];
    nn = numn[i];
    if (4 * g < maxn) e4 = *(const int4 *)(nbr + (((size_t)g * n + i) << 2));
  }
  if (L > 1 && 4 * g < nn) quad_partners_f32(p4f, e4, pj);
  shift_table(bs->b0, pg, S);
  __syncthreads();
  shift_table_f32(S, Sf, Sl);
  __syncthreads();
  const float rc = (float)P.r_int + 1e-4f, rc2 = rc * rc;
  double acc = 0.0;
  if (i < n) {
    int na = 0;
    for (int q = g; 4 * q < nn; q += L) {
      const unsigned e[4] = {(unsigned)e4.x, (unsigned)e4.y, (unsigned)e4.z, (unsigned)e4.w};
      if (L == 1 || q != g) quad_partners_f32(p4f, e4, pj);
      // the next quad's indices load while this quad's partners arrive
      if (4 * (q + L) < nn) e4 = *(const int4 *)(nbr + (((size_t)(q + L) * n + i) << 2));
      float mn = rc2;
#pragma unroll
      for (int u = 0; u < 4; u++) {
        float rx, ry, rz;
        const float r2 = pair_r2_f32(pi, pj[u], Sf, Sl, e[u], rx, ry, rz);
        if (r2 < rc2) {  // phi is zero beyond r_int; the list's tail is out of range
          float r, ri;
          r_and_inv(r2, r, ri);
          acc += (double)mdk_pair_phi<float, POT_FE>(P, r);
        }
        mn = fminf(mn, r2);
      }
      na = mn < rc2 ? 4 * q + 4 : na;
    }
    acc = group_sum<L>(acc);
    na = group_max<L>(na);
    if (g == 0) nact[i] = na;
  }
  density_finish(atoms, pos4, p4f, n, g == 0 ? i : n, acc, P, do_embed, part, nb, bk);
}

// The lean path's density pass on a new list: k_density_f32's arithmetic (so
// the densities are those of every later pass on this list), and each atom's
// list reordered in place as k_density_part does -- partners within rc first,
// in list order, then the others (DENS_OBUF of them held in LDS, more stay in
// place) -- so that the force pass stops after the in-range part.
__global__ void __launch_bounds__(MDK_BLOCK) k_density_part_f32(double *atoms, float4 *p4f, int n, int *nbr,
                                                                const int *__restrict__ numn, const BoxState *bs,
                                                                PackGeo pg, PotDev P, int do_embed, double *part,
                                                                int *nact, Rider R) {
  DENS_BLOCKS(R, MDK_BLOCK);
  __shared__ double S[32][3];
  __shared__ float4 Sf[32], Sl[32];
  __shared__ int obuf[DENS_OBUF][MDK_BLOCK];
  shift_table(bs->b0, pg, S);
  __syncthreads();
  shift_table_f32(S, Sf, Sl);
  __syncthreads();
  const int t = threadIdx.x, i = xcd_tile(nb, bk) * blockDim.x + t;
  const float rc = (float)P.r_int + 1e-4f, rc2 = rc * rc;
  double acc = 0.0;
  if (i < n) {
    const float4 pi = p4f[i];
    const int nn = numn[i];
    int m = 0, no = 0, last = 0;  // entries written back, entries held, end of the last in-range one
    int4 qd = make_int4(0, 0, 0, 0);
    for (int q = 0; 4 * q < nn; q++) {
      const int4 e4 = *(const int4 *)(nbr + (((size_t)q * n + i) << 2));
      const int e[4] = {e4.x, e4.y, e4.z, e4.w};
      float4 pj[4];
#pragma unroll
      for (int u = 0; u < 4; u++) pj[u] = p4f[(unsigned)e[u] & NBR_IDX_MASK];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        float rx, ry, rz;
        const float r2 = pair_r2_f32(pi, pj[u], Sf, Sl, (unsigned)e[u], rx, ry, rz);
        if (r2 < rc2) {
          float r, ri;
          r_and_inv(r2, r, ri);
          acc += (double)mdk_pair_phi<float, POT_FE>(P, r);
        }
        if (4 * q + u < nn) {
          const bool in = r2 < rc2;
          if (in || no == DENS_OBUF) {
            quad_put(nbr, i, n, e[u], m, qd);
            if (in) last = m;
          } else {
            obuf[no++][t] = e[u];
          }
        }
      }
    }
    for (int u = 0; u < no; u++) quad_put(nbr, i, n, obuf[u][t], m, qd);
    if (m & 3) {  // the last quad's null entries
      const int nul = i | (NBR_NULL_CODE << NBR_CODE_SHIFT), sl = m & 3;
      qd.y = sl <= 1 ? nul : qd.y;
      qd.z = sl <= 2 ? nul : qd.z;
      qd.w = nul;
      *(int4 *)(nbr + nbr_at(m & ~3, i, n)) = qd;
    }
    nact[i] = (last + 3) & ~3;
  }
  density_finish(atoms, nullptr, p4f, n, i, acc, P, do_embed, part, nb, bk);
}

// Force pass (src/dynamics_m.F90:235-346): V, V' and phi' from the FP32 interval table, fp = -(V' + phi'(F'_i +
// F'_j))/r, F_i = sum r fp.  Each atom's force and the lane's pair energy and
// virial W = 1/2 sum r r^T fp are FP32 sums over the atom's few tens of terms;
// the sums over lanes, waves and workgroups are FP64.
template <int L, bool KICK>
__global__ void __launch_bounds__(MDK_BLOCK) k_force_f32(double *atoms, const float4 *__restrict__ p4f,
                                                         int n, const int *__restrict__ nbr,
                                                         const int *__restrict__ nvisit, int maxn, const BoxState *bs,
                                                         PackGeo pg, PotDev P, double *part, const float *fetab,
                                                         KickIo K) {
  __shared__ double S[32][3];
  __shared__ float4 Sf[32], Sl[32];
  __shared__ float4 fbin[MDK_FE_NB];
  __shared__ __align__(16) float fiv[8 * MDK_FE_NI];
  __shared__ double bi[9];
  const Place place = place_of(gridDim.x, blockIdx.x, K.one_xcd);
  if (place.idle) return;
  const int i = (xcd_tile(place.nb, place.b) * (int)blockDim.x + (int)threadIdx.x) / L, g = threadIdx.x % L;
  const bool own = i < n && g == 0;
  float4 pi, pj[4];  // loaded ahead as in k_density
  int4 e4 = make_int4(0, 0, 0, 0);
  int nn = 0;
  if (i < n) {
    pi = p4f[i];
    nn = nvisit[i];
    if (4 * g < maxn) e4 = *(const int4 *)(nbr + (((size_t)g * n + i) << 2));
  }
  KickAtom ka;
  if (KICK && L > 1 && own) ka = load_kick<true, false>(atoms, K.zat, n, i, K.sref, K.img, K.cell, pg, K.spec);
  if (L > 1 && 4 * g < nn) quad_partners_f32(p4f, e4, pj);
  double b[9];
#pragma unroll
  for (int k = 0; k < 9; k++) b[k] = bs->b0[k];
  shift_table(b, pg, S);
  {
    const float4 *src = (const float4 *)fetab;
    if (threadIdx.x < MDK_FE_NB) fbin[threadIdx.x] = src[threadIdx.x];
    else if (threadIdx.x < MDK_FE_NB + 2 * MDK_FE_NI) ((float4 *)fiv)[threadIdx.x - MDK_FE_NB] = src[threadIdx.x];
  }
  if (threadIdx.x == 128) inv3(b, bi);
  __syncthreads();
  shift_table_f32(S, Sf, Sl);
  __syncthreads();
  double v[NPART_FORCE];
#pragma unroll
  for (int k = 0; k < NPART_FORCE; k++) v[k] = 0.0;
  double f0 = 0.0, f1 = 0.0, f2 = 0.0;
  if (i < n) {
    float fx = 0.f, fy = 0.f, fz = 0.f;
    // sums of V and of r r^T fp (the factor 1/2 of both is applied once below)
    float pe2 = 0.f, wxx = 0.f, wyy = 0.f, wzz = 0.f, wxy = 0.f, wxz = 0.f, wyz = 0.f;
    for (int q = g; 4 * q < nn; q += L) {
      const unsigned e[4] = {(unsigned)e4.x, (unsigned)e4.y, (unsigned)e4.z, (unsigned)e4.w};
      if (L == 1 || q != g) quad_partners_f32(p4f, e4, pj);
      // the next quad's indices load while this quad's partners arrive
      if (4 * (q + L) < nn) e4 = *(const int4 *)(nbr + (((size_t)(q + L) * n + i) << 2));
#pragma unroll
      for (int u = 0; u < 4; u++) {
        float rx, ry, rz;
        const float r2 = pair_r2_f32(pi, pj[u], Sf, Sl, e[u], rx, ry, rz);
        float r, ri;
        r_and_inv(r2, r, ri);
        float vv, dv, dph;
        mdk_fe_terms(P, fbin, fiv, r, vv, dv, dph);
        const float fp = -(dv + dph * (pi.w + pj[u].w)) * ri;
        const float gx = rx * fp, gy = ry * fp, gz = rz * fp;
        fx += gx;
        fy += gy;
        fz += gz;
        pe2 += vv;
        if (!KICK) {
          wxx += rx * gx; wyy += ry * gy; wzz += rz * gz;
          wxy += rx * gy; wxz += rx * gz; wyz += ry * gz;
        }
      }
    }
    v[0] = 0.5 * (double)pe2;
    v[1] = 0.5 * (double)wxx; v[2] = 0.5 * (double)wyy; v[3] = 0.5 * (double)wzz;
    v[4] = 0.5 * (double)wxy; v[5] = 0.5 * (double)wxz; v[6] = 0.5 * (double)wyz;
    // fractional force f = B0^-1 F (the reference's fx = sum s fp, Cartesian = B0 f)
    const double Fx = group_sum<L>(fx), Fy = group_sum<L>(fy), Fz = group_sum<L>(fz);
    f0 = bi[0] * Fx + bi[3] * Fy + bi[6] * Fz;
    f1 = bi[1] * Fx + bi[4] * Fy + bi[7] * Fz;
    f2 = bi[2] * Fx + bi[5] * Fy + bi[8] * Fz;
  }
  if constexpr (KICK) {
    if (L == 1 && own) ka = load_kick<true, false>(atoms, K.zat, n, i, K.sref, K.img, K.cell, pg, K.spec);
    fixed_kick<MDK_BLOCK>(ka, K, bs, i, n, own, v[0], f0, f1, f2, atoms, pg, place.nb, place.b);
  } else {
    if (own) {
      atoms[(size_t)F_FX * n + i] = f0;
      atoms[(size_t)F_FY * n + i] = f1;
      atoms[(size_t)F_FZ * n + i] = f2;
    }
    block_store<NPART_FORCE, 0>(v, part, place.nb, place.b);
  }
}

// ---------------------------------------------------------------------------
// The same passes on a brick list.  The workgroup stages the brick's atoms and
// their surroundings once -- some 1090 records of 16 bytes for 324 atoms, read
// in order -- and every partner is then an LDS read of 16 bytes by a 16-bit
// offset.  With lists of atom indices the gathers kept the address units busy
// for 89 % of the density pass of a liquid (a line per lane); here the vector
// ALU is (67 %), and in the force pass with the kick memory (5.8 TB/s).  us at
// 3,456,000 atoms of liquid, indices : bricks -- density 168 : 121, force and
// kick 219 : 204, list with its first density pass 866 : 525; 524,288 atoms of
// crystal 23.7 : 22.0, force 21.5 : 23.6, list 141 : 101.
// Positions are staged as 32-bit fixed point about the brick's centre, so that
// partner differences are exact: with cells of 4 A a unit is 2^-25 A, a quarter
// of the FP32 record's own rounding, and the offset of a cell is rounded once,
// to 1e-8 of a cell (as FP32 numbers offsets of this size would bias every
// separation of one cell offset alike).
// ---------------------------------------------------------------------------
struct BrickArgs {
  const uint2 *nbr16;
  const int *bstage;
  const int4 *binfo;
  int cap;
  float scale, inv;  // units per A (a power of two) and its inverse
};
#define BRICK_NULL 0x3fffffff  // the null slot's coordinates: beyond every range from any atom
// Stages the atoms of brick bi with w = their F'.
template <int NT>
__device__ __forceinline__ void brick_stage(const BrickArgs &A, int bi, const int4 &info, const double *b,
                                            const PackGeo &pg, const float4 *__restrict__ p4f, int4 *st) {
  __shared__ int4 step[3][6], cell[BRICK_CELLS];  // centres of the 6x6x6 cells from the brick's, in units
  constexpr int NS = 3;                           // staged atoms per thread that load together
  const int t = threadIdx.x;
  const int *src = A.bstage + (size_t)bi * A.cap;
  unsigned e[NS];
#pragma unroll
  for (int u = 0; u < NS; u++) e[u] = t + u * NT < A.cap ? (unsigned)src[t + u * NT] : 0u;  // info is on its way
  if (t < 24 && (t & 7) < 6) {
    const int a = t >> 3, h = t & 7;
    const double f = (h - 2.5) * (a == 0 ? pg.ix : (a == 1 ? pg.iy : pg.iz)) * (double)A.scale;
    step[a][h] = make_int4((int)rint(b[3 * a] * f), (int)rint(b[3 * a + 1] * f), (int)rint(b[3 * a + 2] * f), 0);
  }
  float4 q[NS];
#pragma unroll
  for (int u = 0; u < NS; u++)
    if (t + u * NT < info.z) q[u] = p4f[e[u] & ((1u << BRICK_H_SHIFT) - 1)];
  __syncthreads();
  if (t < BRICK_CELLS) {
    const int4 x = step[0][t % 6], y = step[1][(t / 6) % 6], z = step[2][t / 36];
    cell[t] = make_int4(x.x + y.x + z.x, x.y + y.y + z.y, x.z + y.z + z.z, 0);
  }
  __syncthreads();
  auto put = [&](int s, unsigned e, const float4 &q) {
    const int4 c = cell[e >> BRICK_H_SHIFT];
    auto fix = [&](float x) { return (int)floorf(fmaf(x, A.scale, 0.5f)); };
    st[s] = make_int4(fix(q.x) + c.x, fix(q.y) + c.y, fix(q.z) + c.z, __float_as_int(q.w));
  };
#pragma unroll
  for (int u = 0; u < NS; u++)
    if (t + u * NT < info.z) put(t + u * NT, e[u], q[u]);
  for (int s = t + NS * NT; s < info.z; s += NT) {
    const unsigned es = (unsigned)src[s];
    put(s, es, p4f[es & ((1u << BRICK_H_SHIFT) - 1)]);
  }
  if (t == 0) st[info.z] = make_int4(BRICK_NULL, BRICK_NULL, BRICK_NULL, 0);
  __syncthreads();
}
// two partners: their LDS byte offsets are the halves of a word
__device__ __forceinline__ void brick_partners(const int4 *st, unsigned w, int4 (&pj)[2]) {
  const char *at = (const char *)st;
  pj[0] = *(const int4 *)(at + (w & 0xffff));
  pj[1] = *(const int4 *)(at + (w >> 16));
}

// k_density_f32 on a brick list; nact[i] = quads up to the last with a partner in
// range.
template <int NT>
__global__ void __launch_bounds__(NT) k_density_brick(double *atoms, float4 *p4f, int n, BrickArgs A,
                                                      const int *__restrict__ bcnt, const BoxState *bs, PackGeo pg,
                                                      PotDev P, int do_embed, double *part, int *nact, Rider R) {
  DENS_BLOCKS(R, NT);
  extern __shared__ int4 st[];
  const int bi = xcd_tile(nb, bk), t = threadIdx.x;
  const int4 info = A.binfo[bi];
  const int i = info.x + t;
  const bool own = t < info.y;
  int nq = 0;
  uint2 o = make_uint2(0, 0);
  if (own) {
    nq = bcnt[i];
    o = A.nbr16[i];
  }
  brick_stage<NT>(A, bi, info, bs->b0, pg, p4f, st);
  const float rc = (float)P.r_int + 1e-4f, rc2 = rc * rc, inv2 = A.inv * A.inv;
  double acc = 0.0, pe[1] = {0.0};
  if (own) {
    const int4 pi = st[t];
    int na = 0;
    for (int q = 0; q < nq; q++) {
      const uint2 w = o;
      // the next quad loads while this quad's partners arrive
      if (q + 1 < nq) o = A.nbr16[(size_t)(q + 1) * n + i];
      float mn = rc2;
#pragma unroll
      for (int half = 0; half < 2; half++) {
        int4 pj[2];
        brick_partners(st, half ? w.y : w.x, pj);
#pragma unroll
        for (int u = 0; u < 2; u++) {
          const float rx = (float)(pi.x - pj[u].x), ry = (float)(pi.y - pj[u].y), rz = (float)(pi.z - pj[u].z);
          const float r2 = (rx * rx + ry * ry + rz * rz) * inv2;
          if (r2 < rc2) {  // phi is zero beyond r_int; the skin is out of range
            float r, ri;
            r_and_inv(r2, r, ri);
            acc += (double)mdk_pair_phi<float, POT_FE>(P, r);
          }
          mn = fminf(mn, r2);
        }
      }
      na = mn < rc2 ? q + 1 : na;
    }
    nact[i] = na;
    pe[0] = density_atom(atoms, nullptr, p4f, n, i, acc, P, do_embed);
  }
  if (do_embed) block_store<1, 0, NT>(pe, part, nb, bk);
}

// k_force_f32 on a brick list
template <int NT, bool KICK>
__global__ void __launch_bounds__(NT, 8) k_force_brick(double *atoms, const float4 *__restrict__ p4f, int n, BrickArgs A,
                                                    const int *__restrict__ nvisit, const BoxState *bs, PackGeo pg,
                                                    PotDev P, double *part, const float *fetab, KickIo K) {
  extern __shared__ int4 st[];
  __shared__ float4 fbin[MDK_FE_NB];
  __shared__ __align__(16) float fiv[8 * MDK_FE_NI];
  __shared__ double bi9[9];
  const int bi = xcd_tile(), t = threadIdx.x;
  const int4 info = A.binfo[bi];
  const int i = info.x + t;
  const bool own = t < info.y;
  int nq = 0;
  uint2 o = make_uint2(0, 0);
  if (own) {
    nq = nvisit[i];
    o = A.nbr16[i];
  }
  {
    const float4 *src = (const float4 *)fetab;
    if (t < MDK_FE_NB) fbin[t] = src[t];
    else if (t < MDK_FE_NB + 2 * MDK_FE_NI) ((float4 *)fiv)[t - MDK_FE_NB] = src[t];
  }
  if (t == NT - 64) {
    double b[9];
#pragma unroll
    for (int k = 0; k < 9; k++) b[k] = bs->b0[k];
    inv3(b, bi9);
  }
  brick_stage<NT>(A, bi, info, bs->b0, pg, p4f, st);
  double v[NPART_FORCE];
#pragma unroll
  for (int k = 0; k < NPART_FORCE; k++) v[k] = 0.0;
  double f0 = 0.0, f1 = 0.0, f2 = 0.0;
  KickAtom ka;
  if (own) {
    const int4 pi = st[t];
    const float wi = __int_as_float(pi.w), inv2 = A.inv * A.inv;
    float fx = 0.f, fy = 0.f, fz = 0.f;
    float pe2 = 0.f, wxx = 0.f, wyy = 0.f, wzz = 0.f, wxy = 0.f, wxz = 0.f, wyz = 0.f;
    for (int q = 0; q < nq; q++) {
      const uint2 w = o;
      if (q + 1 < nq) o = A.nbr16[(size_t)(q + 1) * n + i];
#pragma unroll 1
      for (int half = 0; half < 2; half++) {
        int4 pj[2];
        brick_partners(st, half ? w.y : w.x, pj);
#pragma unroll
        for (int u = 0; u < 2; u++) {
          const float rx = (float)(pi.x - pj[u].x), ry = (float)(pi.y - pj[u].y), rz = (float)(pi.z - pj[u].z);
          const float r2 = (rx * rx + ry * ry + rz * rz) * inv2;
          float r, ri;
          r_and_inv(r2, r, ri);
          float vv, dv, dph;
          mdk_fe_terms(P, fbin, fiv, r, vv, dv, dph);
          const float fp = -(dv + dph * (wi + __int_as_float(pj[u].w))) * ri;
          // sums in units: scaled by inv (inv^2) below, a power of two
          const float gx = rx * fp, gy = ry * fp, gz = rz * fp;
          fx += gx;
          fy += gy;
          fz += gz;
          pe2 += vv;
          if (!KICK) {
            wxx += rx * gx; wyy += ry * gy; wzz += rz * gz;
            wxy += rx * gy; wxz += rx * gz; wyz += ry * gz;
          }
        }
      }
    }
    const double s1 = (double)A.inv, s2 = 0.5 * (double)inv2;
    v[0] = 0.5 * (double)pe2;
    v[1] = s2 * (double)wxx; v[2] = s2 * (double)wyy; v[3] = s2 * (double)wzz;
    v[4] = s2 * (double)wxy; v[5] = s2 * (double)wxz; v[6] = s2 * (double)wyz;
    // fractional force f = B0^-1 F (the reference's fx = sum s fp, Cartesian = B0 f)
    const double Fx = s1 * (double)fx, Fy = s1 * (double)fy, Fz = s1 * (double)fz;
    f0 = bi9[0] * Fx + bi9[3] * Fy + bi9[6] * Fz;
    f1 = bi9[1] * Fx + bi9[4] * Fy + bi9[7] * Fz;
    f2 = bi9[2] * Fx + bi9[5] * Fy + bi9[8] * Fz;
  }
  if constexpr (KICK) {
    if (own) ka = load_kick<true, false>(atoms, K.zat, n, i, K.sref, K.img, K.cell, pg, K.spec);
    fixed_kick<NT>(ka, K, bs, i, n, own, v[0], f0, f1, f2, atoms, pg, gridDim.x, blockIdx.x);
  } else {
    if (own) {
      atoms[(size_t)F_FX * n + i] = f0;
      atoms[(size_t)F_FY * n + i] = f1;
      atoms[(size_t)F_FZ * n + i] = f2;
    }
    block_store<NPART_FORCE, 0, NT>(v, part);
  }
}

// scalev (src/thermostat_m.F90:317-395), Nose-Hoover velocity scaling, as
// three passes with deterministic block partials: (1) sums of x1 over all
// atoms; (2) moving atoms (Z != 0, mass >= 0.1) lose the mean, partial
// kinetic sums m |B0 x1|^2; (3) moving atoms' x1 scaled by 1 + snhv (the
// host forms ke, snhf and snhv between (2) and (3)).
__global__ void __launch_bounds__(MDK_BLOCK) k_vsum(const double *__restrict__ atoms, int n, double *part) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double v[3] = {0.0, 0.0, 0.0};
  if (i < n)
    for (int d = 0; d < 3; d++) v[d] = atoms[(size_t)(F_X1 + d) * n + i];
  block_store<3, 0>(v, part);
}
__device__ __forceinline__ bool moving_atom(const double *atoms, const int *zat, const double *spec, int n, int i) {
  const int z = zat[i];
  const double m = spec ? spec[2 * z] : atoms[(size_t)F_MASS * n + i];
  return !(z == 0 || m < (double)0.1f);
}
__global__ void __launch_bounds__(MDK_BLOCK) k_vsub_ke(double *__restrict__ atoms, const int *__restrict__ zat, int n,
                                                       const double *__restrict__ mean, const BoxState *bs,
                                                       const double *__restrict__ spec, double *part) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double v[1] = {0.0};
  if (i < n && moving_atom(atoms, zat, spec, n, i)) {
    double x[3];
    for (int d = 0; d < 3; d++) {
      double *q = atoms + (size_t)(F_X1 + d) * n + i;
      x[d] = *q - mean[d];
      *q = x[d];
    }
    const double *b = bs->b0;
    const double rx = b[0] * x[0] + b[3] * x[1] + b[6] * x[2];
    const double ry = b[1] * x[0] + b[4] * x[1] + b[7] * x[2];
    const double rz = b[2] * x[0] + b[5] * x[1] + b[8] * x[2];
    const double m = spec ? spec[2 * zat[i]] : atoms[(size_t)F_MASS * n + i];
    v[0] = m * (rx * rx + ry * ry + rz * rz);
  }
  block_store<1, 0>(v, part);
}
__global__ void __launch_bounds__(MDK_BLOCK) k_vscale(double *__restrict__ atoms, const int *__restrict__ zat, int n,
                                                      const double *__restrict__ spec, double f) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && moving_atom(atoms, zat, spec, n, i))
    for (int d = 0; d < 3; d++) atoms[(size_t)(F_X1 + d) * n + i] *= f;
}
// fixed-order fold of K per-block partials into out[0..K-1]
template <int K>
__global__ void __launch_bounds__(MDK_FIN_BLOCK) k_fold(const double *part, int nb, double *stage, unsigned *cnt,
                                                        double *out) {
  double v[K];
  if (!stage_and_finish<K, 0>(part, nb, stage, cnt, v)) return;
  if (threadIdx.x == 0)
    for (int k = 0; k < K; k++) out[k] = v[k];
}

// update_therm_avs box part only (stand-alone entry point)
__global__ void k_therm_box(BoxState *bs, int ivol) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    BoxState s = *bs;
    therm_box(s, ivol);
    *bs = s;
  }
}

// The half kick over all atoms; with DRIFT block 0 writes the advanced box
// state into bout.  Every pointer is restrict-qualified: the box state is only
// read, so its uniform fields come through scalar loads instead of one vector
// load per lane.
template <bool DRIFT>
__global__ void __launch_bounds__(MDK_BLOCK) k_kick(double *__restrict__ atoms, const int *__restrict__ zat, int n,
                                                    const BoxState *__restrict__ bs, int ivol, int mode,
                                                    const float *__restrict__ sref, double *__restrict__ part,
                                                    double4 *__restrict__ pos4, float4 *__restrict__ p4f,
                                                    const int *__restrict__ img, const int *__restrict__ cell,
                                                    PackGeo pg, BoxState *__restrict__ bout,
                                                    const double *__restrict__ spec, double *__restrict__ kin, LinkGrid link) {
  const int i = xcd_tile() * blockDim.x + threadIdx.x;
  double v[NPART_KICK] = {0.0, 0.0, 0.0, 0.0, 0.0};
  double kv[9] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  if (i < n) {
    const KickAtom a = load_kick<DRIFT, true>(atoms, zat, n, i, sref, img, cell, pg, spec);
    const KickBox B = {bs->tgid_lag, bs->tgid, bs->binv, bs->b0, bs->b1, bs->b2};
    kick_atom<DRIFT, false>(a, B, i, n, ivol, mode, sref != nullptr, atoms, pos4, p4f, pg, link, v, kv);
  }
  if (DRIFT && blockIdx.x == 0) drift_box(bs, bout, ivol);
  block_store<NPART_KICK, 2>(v, part);
  if (DRIFT) block_store<9, 0>(kv, kin);
}

// Small systems: force()'s finishing and the half kick in one launch.  Every
// workgroup folds the partials and completes the box in its own LDS (the same
// bits everywhere), so no kernel boundary separates the sums from the atoms
// that need them; block 0 writes the box state into fin, and with DRIFT the
// advanced one into bout -- copies of their own, since other workgroups may
// still read F.bs.  The per-atom loads are issued first and arrive during the
// fold.  Latency bound: 9.0 us against 4.3 + 5.7 us and a launch gap of
// about 1.5 us for the two kernels at 2000 atoms.
template <bool DRIFT>
__global__ void __launch_bounds__(MDK_BLOCK) k_finish_kick(
    FinForce F, BoxState *__restrict__ fin, double *__restrict__ atoms, const int *__restrict__ zat, int n,
    const float *__restrict__ sref, double *__restrict__ part, double4 *__restrict__ pos4, float4 *__restrict__ p4f,
    const int *__restrict__ img, const int *__restrict__ cell, PackGeo pg, BoxState *__restrict__ bout,
    const double *__restrict__ spec, double *__restrict__ kin, LinkGrid link) {
  __shared__ ForceLds s;
  const Place place = place_of(gridDim.x, blockIdx.x, F.one_xcd);
  if (place.idle) return;
  const int i = xcd_tile(place.nb, place.b) * blockDim.x + threadIdx.x;
  KickAtom a;
  if (i < n) a = load_kick<DRIFT, true>(atoms, zat, n, i, sref, img, cell, pg, spec);
  load_force_box(F.bs, s);
  fold_force_columns<MDK_BLOCK>(F, s);
  __syncthreads();
  complete_force(F, s);
  double v[NPART_KICK] = {0.0, 0.0, 0.0, 0.0, 0.0};
  double kv[9] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  if (i < n) {
    const KickBox B = {s.tgid0, s.tgid, s.binv, s.b0, s.b1, s.b2};
    kick_atom<DRIFT, false>(a, B, i, n, F.ivol, 0, true, atoms, pos4, p4f, pg, link, v, kv);
  }
  if (blockIdx.x == 0) {
    store_box(F, s, fin, false);
    if (DRIFT) store_box(F, s, bout, true);
  }
  block_store<NPART_KICK, 2>(v, part, place.nb, place.b);
  if (DRIFT) block_store<9, 0>(kv, kin, place.nb, place.b);
}

// energy_calc (src/dynamics_m.F90:410-470): en_i = F(rho_i) + 1/2 sum_j V(r_ij)
// over atom i's full list (each pair once from each end, as the reference's
// half list adds V/2 to both ends).  The pair function is the exact one even
// when the force path uses tables: the reference calls vee_src there.
template <int POTM>
__global__ void __launch_bounds__(MDK_BLOCK) k_energy_calc(const double *atoms, const double4 *__restrict__ pos4,
                                                           int n, const int *__restrict__ nbr,
                                                           const int *__restrict__ numn, const BoxState *bs,
                                                           PackGeo pg, PotDev P, double *en) {
  __shared__ double S[32][3];
  shift_table(bs->b0, pg, S);
  __syncthreads();
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double4 pi = pos4[i];
  double s = 0.0;
  for (int k = 0; k < numn[i]; k++) {
    const unsigned e = (unsigned)nbr[nbr_at(k, i, n)];
    const double4 pj = pos4[e & NBR_IDX_MASK];
    double dx, dy, dz, rx, ry, rz;
    const double r = sqrt(pair_sep<double>(S, pi, pj, (int)(e >> NBR_CODE_SHIFT), dx, dy, dz, rx, ry, rz));
    double v, dv;
    mdk_pair_vdv<double, POTM>(P, r, v, dv);
    s += v / 2.0;
  }
  en[i] = atoms[(size_t)F_AFRHO * n + i] + s;
}

// Per-atom diagonal stress of the reference's force loop
// (src/dynamics_m.F90:279-283): stress_x(i) = sum of rx_ij fp_ij over atom i's
// own half-list partners j only (the partner gets nothing from that pair),
// with fp = -V'/r - (phi' F'_i + phi' F'_j)/r as the force loop forms it.
// One thread per atom in reference order; positions at the atom's current slot.
template <int POTM>
__global__ void __launch_bounds__(MDK_BLOCK) k_atomic_stress(const double *atoms, const int *slot_of, int n,
                                                             const int *numn_ref, const int *nlist_ref,
                                                             int nnbrs, const BoxState *bs, int pbc, PotDev P,
                                                             double *sx, double *sy, double *sz) {
#pragma clang fp contract(off)
  const int oi = blockIdx.x * blockDim.x + threadIdx.x;
  if (oi >= n) return;
  const double *b = bs->b0;
  const int i = slot_of[oi];
  const double *x0 = atoms, *y0 = atoms + n, *z0 = atoms + 2 * (size_t)n;
  const double *df = atoms + (size_t)F_DAFRHO * n;
  const double xi = x0[i], yi = y0[i], zi = z0[i], dfi = df[i];
  double ax = 0.0, ay = 0.0, az = 0.0;
  const int cnt = min(numn_ref[oi], nnbrs);
  for (int q = 0; q < cnt; q++) {
    const int j = slot_of[nlist_ref[(size_t)oi * nnbrs + q] - 1];
    double dx = xi - x0[j], dy = yi - y0[j], dz = zi - z0[j];
    min_image(pbc, dx, dy, dz);
    const double r = sqrt(sep2_exact(b, dx, dy, dz));
    const double rr = 1.0 / r;
    double v, dv;
    mdk_pair_vdv<double, POTM>(P, r, v, dv);
    const double dph = mdk_pair_dphi<double, POTM>(P, r);
    const double fp = -dv * rr + (-1.0 * (dph * dfi + dph * df[j]) * rr);
    ax += (b[0] * dx + b[3] * dy + b[6] * dz) * fp;
    ay += (b[1] * dx + b[4] * dy + b[7] * dz) * fp;
    az += (b[2] * dx + b[5] * dy + b[8] * dz) * fp;
  }
  sx[oi] = ax;
  sy[oi] = ay;
  sz[oi] = az;
}

// potential evaluation for mdk_eval_potential
__global__ void k_eval_pot(PotDev P, int which, const double *x, double *y, int cnt, const float *fetab) {
  int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= cnt) return;
  if (which >= 6) {  // the FP32 force pass's V, V', phi' (interval table)
    float v32, dv32, dph32;
    mdk_fe_terms(P, (const float4 *)fetab, fetab + 4 * MDK_FE_NB, (float)x[k], v32, dv32, dph32);
    y[k] = which == 6 ? v32 : (which == 7 ? dv32 : dph32);
    return;
  }
  double r = x[k], v = 0.0, dv = 0.0;
  const bool lk = P.use_lookup != 0, fec = P.material == MDK_MAT_IRON_CARBON;
  switch (which) {
    case 0:
    case 1:
      if (lk) mdk_pair_vdv<double, POT_TABLE>(P, r, v, dv);
      else if (fec) mdk_pair_vdv<double, POT_FEC>(P, r, v, dv);
      else mdk_pair_vdv<double>(P, r, v, dv);
      y[k] = which == 0 ? v : dv;
      break;
    case 2:
      y[k] = lk ? mdk_pair_phi<double, POT_TABLE>(P, r)
                : (fec ? mdk_pair_phi<double, POT_FEC>(P, r) : mdk_pair_phi<double>(P, r));
      break;
    case 3:
      y[k] = lk ? mdk_pair_dphi<double, POT_TABLE>(P, r)
                : (fec ? mdk_pair_dphi<double, POT_FEC>(P, r) : mdk_pair_dphi<double>(P, r));
      break;
    case 4: mdk_embed_f(P, r, v, dv); y[k] = v; break;
    case 5: mdk_embed_f(P, r, v, dv); y[k] = dv; break;
  }
}

// ---------------------------------------------------------------------------
// host orchestration
// ---------------------------------------------------------------------------
static inline int nblocks(long n) { return (int)((n + MDK_BLOCK - 1) / MDK_BLOCK); }

static hipEvent_t pooled_event(mdk_ctx *c) {
  hipEvent_t e;
  if (!c->evpool.empty()) {
    e = c->evpool.back();
    c->evpool.pop_back();
  } else {
    hipEventCreate(&e);
  }
  return e;
}
static void tbegin(mdk_ctx *c, int cls, TimedEv &te) {
  te.cls = -1;
  if (!((c->timing_mask >> cls) & 1)) return;
  if (c->timing_every > 1 && (c->t_seen[cls]++ % c->timing_every) != 0) return;
  te.cls = cls;
  te.a = pooled_event(c);
  te.b = pooled_event(c);
  hipEventRecord(te.a, c->stream);
}
// Events filled in by the kernel dispatch itself (hipExtLaunchKernel): the
// interval is the kernel's own execution, with no gap before or after it.
static void tbegin_ext(mdk_ctx *c, int cls, TimedEv &te) {
  te.cls = -1;
  if (!((c->timing_mask >> cls) & 1)) return;
  if (c->timing_every > 1 && (c->t_seen[cls]++ % c->timing_every) != 0) return;
  te.cls = cls;
  te.a = pooled_event(c);
  te.b = pooled_event(c);
}
static void tpush(mdk_ctx *c, TimedEv &te);
static void tend(mdk_ctx *c, TimedEv &te) {
  if (te.cls < 0) return;
  hipEventRecord(te.b, c->stream);
  tpush(c, te);
}
static void tpush(mdk_ctx *c, TimedEv &te) {
  if (te.cls < 0) return;
  c->evs.push_back(te);
  if (c->evs.size() > 4096) {  // resolve old ones to bound memory
    hipEventSynchronize(te.b);
    for (auto &e : c->evs) {
      float ms = 0.f;
      hipEventElapsedTime(&ms, e.a, e.b);
      c->t_ms[e.cls] += ms;
      c->t_cnt[e.cls] += 1;
      c->evpool.push_back(e.a);
      c->evpool.push_back(e.b);
    }
    c->evs.clear();
  }
}

static int check_launch(const char *what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_err(MDK_ERR_HIP, "launch %s: %s", what, hipGetErrorString(e));
  return MDK_OK;
}

static double near_threshold(double rn) {
  // smallest double q with sqrt(q) >= rn (host sqrt is correctly rounded), so
  // that sqrt(q) < rn <=> q < threshold without a device square root.
  double q = rn * rn;
  while (sqrt(q) >= rn) q = nextafter(q, 0.0);
  while (sqrt(q) < rn) q = nextafter(q, INFINITY);
  return q;
}

static int read_box(mdk_ctx *c, BoxState *out) {
  HIPCK(hipMemcpyAsync(out, c->box + c->cur, sizeof(BoxState), hipMemcpyDeviceToHost, c->stream));
  HIPCK(hipStreamSynchronize(c->stream));
  return MDK_OK;
}

// Fine grid from the current box: cells at least r_list wide (perpendicular width)
static void plan_grid(mdk_ctx *c, const double *b, int g[3], double margin) {
  double vol = fabs(TT(b, 1, 1) * (TT(b, 2, 2) * TT(b, 3, 3) - TT(b, 2, 3) * TT(b, 3, 2)) +
                    TT(b, 2, 1) * (TT(b, 3, 2) * TT(b, 1, 3) - TT(b, 1, 2) * TT(b, 3, 3)) +
                    TT(b, 3, 1) * (TT(b, 1, 2) * TT(b, 2, 3) - TT(b, 2, 2) * TT(b, 1, 3)));
  for (int d = 0; d < 3; d++) {
    int e1 = (d + 1) % 3, e2 = (d + 2) % 3;
    const double *u = b + 3 * e1, *w = b + 3 * e2;
    double cx = u[1] * w[2] - u[2] * w[1], cy = u[2] * w[0] - u[0] * w[2], cz = u[0] * w[1] - u[1] * w[0];
    double width = vol / sqrt(cx * cx + cy * cy + cz * cz);
    int nc = (int)floor(width / (c->r_list * margin));
    if (nc < 3) nc = 1;  // too few cells for a distinct 27-cell stencil: one cell in this dim
    if (nc > 256) nc = 256;
    g[d] = nc;
  }
}

static int ensure_cells(mdk_ctx *c, int m) {
  if (m <= c->ncell_cap) return MDK_OK;
  for (int **q : {&c->cell_count, &c->cell_start, &c->cell_fill, &c->cell_btot}) {
    if (*q) hipFree(*q);
    *q = nullptr;
  }
  c->ncell_cap = 0;
  int cap = std::max(m, 64);
  HIPCK(hipMalloc(&c->cell_count, sizeof(int) * cap));
  HIPCK(hipMalloc(&c->cell_start, sizeof(int) * (cap + 1)));
  HIPCK(hipMalloc(&c->cell_fill, sizeof(int) * cap));
  HIPCK(hipMalloc(&c->cell_btot, sizeof(int) * (cap / SCAN_CHUNK + 1)));
  HIPCK(hipMemsetAsync(c->cell_count, 0, sizeof(int) * cap, c->stream));
  c->ncell_cap = cap;
  return MDK_OK;
}

// start offsets of the counted cells, then the members in cell order (in any
// order within a cell)
static int scan_and_fill(mdk_ctx *c, const int *key, int m) {
  if (m <= SCAN_ONE) {
    k_scan_one<<<1, 1024, 0, c->stream>>>(c->cell_count, c->cell_start, c->cell_fill, m);
  } else {
    const int nb = (m + SCAN_CHUNK - 1) / SCAN_CHUNK;
    k_scan_a<<<nb, 1024, 0, c->stream>>>(c->cell_count, c->cell_start, c->cell_fill, c->cell_btot, m);
    k_scan_b<<<1, 1024, 0, c->stream>>>(c->cell_btot, nb, c->cell_start, m);
    k_scan_c<<<nblocks(m), MDK_BLOCK, 0, c->stream>>>(c->cell_start, c->cell_btot, m);
  }
  k_fill<<<nblocks(c->n), MDK_BLOCK, 0, c->stream>>>(key, c->n, c->cell_start, c->cell_fill, c->members);
  return check_launch("scan_and_fill");
}

// counting sort of atoms by key[] into cell_start/members, ascending sortkey
// within a cell
static int bin_atoms(mdk_ctx *c, const int *key, int m, const int *sortkey) {
  RCK(ensure_cells(c, m));
  k_count<<<nblocks(c->n), MDK_BLOCK, 0, c->stream>>>(key, c->n, c->cell_count);
  RCK(scan_and_fill(c, key, m));
  k_sort_cells<<<nblocks(m), MDK_BLOCK, 0, c->stream>>>(c->cell_start, m, c->members, sortkey);
  return check_launch("bin_atoms");
}

static int ensure_pos4(mdk_ctx *c);

// Morton-ordered list of the cubes of side^3 cells that hold cells of grid g
// (recomputed when either changes).
static int plan_list_blocks(mdk_ctx *c, const int g[3], int side) {
  if (c->lblocks && side == c->lblock_side && g[0] == c->lblock_g[0] && g[1] == c->lblock_g[1] &&
      g[2] == c->lblock_g[2])
    return MDK_OK;
  const int bx = (g[0] + side - 1) / side, by = (g[1] + side - 1) / side, bz = (g[2] + side - 1) / side;
  std::vector<int> keys;
  keys.reserve((size_t)bx * by * bz);
  for (int z = 0; z < bz; z++)
    for (int y = 0; y < by; y++)
      for (int x = 0; x < bx; x++) {
        unsigned k = 0;
        for (int bit = 0; bit < 10; bit++) {
          k |= (unsigned)((x >> bit) & 1) << (3 * bit);
          k |= (unsigned)((y >> bit) & 1) << (3 * bit + 1);
          k |= (unsigned)((z >> bit) & 1) << (3 * bit + 2);
        }
        keys.push_back((int)k);
      }
  std::sort(keys.begin(), keys.end());
  const int nb = (int)keys.size();
  if (nb > c->lblocks_cap) {
    if (c->lblocks) HIPCK(hipFree(c->lblocks));
    HIPCK(hipMalloc(&c->lblocks, sizeof(int) * nb));
    c->lblocks_cap = nb;
  }
  HIPCK(hipMemcpy(c->lblocks, keys.data(), sizeof(int) * nb, hipMemcpyHostToDevice));
  c->nlblocks = nb;
  c->lblock_g[0] = g[0]; c->lblock_g[1] = g[1]; c->lblock_g[2] = g[2];
  c->lblock_side = side;
  return MDK_OK;
}

// Fields a re-sort must carry.  Inside force (force_follows) the density and
// force passes rewrite RHO and FX..FZ of every atom before anything reads
// them; X3..Z3 are zero in both buffers until the predictor-corrector or an
// upload sets them (both buffers are cleared at create, and the scratch uses
// of the alternate buffer stay in its X0..Z0 columns).
static ResortSet resort_fields(const mdk_ctx *c, bool force_follows) {
  return ResortSet{!force_follows, c->x3_live};
}

// Which kernel builds the list: a wave per atom where the chip is not full
// with a lane per atom, or where the atoms of a 4x4x4-cell neighbourhood would
// not fit LIST_CAP; else a lane per atom, by blocks where the box allows it.
// Whole rebuilds, wave against lane per atom: by blocks 56 : 76 us at 2000
// atoms, 69 : 81 at 16,000, 84 : 85 at 31,250; open slabs 58 : 187 us at 2000,
// 118 : 192 at 65,536 and 176 : 211 at 128,000.
static bool list_by_waves(int n, bool blk, double per_cell) {
  return blk ? n <= LIST_WAVE_BLK || 64.0 * per_cell > 0.8 * LIST_CAP : n <= LIST_WAVE_ANY;
}

// Brick lists: the FP32 Fe passes of large periodic systems (one lane per atom),
// where a brick's atoms fit a workgroup's threads and their surroundings its
// LDS.  A brick's staging is paid once per workgroup, which smaller systems do not
// repeat often enough to hide.  us per step of the NPT crystal (NVE liquid), lists
// of indices : bricks -- 128,000 atoms 42.9 : 44.0 (29.9 : 32.2), 250,000 57.0 :
// 57.6 (41.9 : 40.8), 314,928 66.0 : 62.4 (50.2 : 47.9), 524,288 91.0 : 88.4 (73.4
// : 71.7), 746,496 117.7 : 107.5 (99 : 96), 1,024,000 166 : 143 (139 : 121).
#define BRICK_ATOMS 262144
static bool brick_size(const mdk_ctx *c) {
  return c->p.precision == MDK_PREC_FP32 && c->pbc == 7 && c->n >= BRICK_ATOMS && c->n < (1 << BRICK_H_SHIFT);
}
static bool lean_pot(const mdk_ctx *c);
// calls f with the number of threads of a brick's workgroup as a constant
template <typename F>
static void with_brick_threads(int nt, F f) {
  switch (nt) {
    case 320: f(std::integral_constant<int, 320>()); break;
    case 384: f(std::integral_constant<int, 384>()); break;
    case 448: f(std::integral_constant<int, 448>()); break;
    default: f(std::integral_constant<int, BRICK_THREADS_MAX>()); break;
  }
}
// the smallest workgroup that has a thread for each of m atoms (0: none)
static int brick_threads(double m) {
  for (int nt = 320; nt <= BRICK_THREADS_MAX; nt += 64)
    if (m <= nt) return nt;
  return 0;
}
// Whether grid g is listed by bricks; g then has whole bricks where their atoms
// still fit (524,288 atoms of bcc Fe: 11^3 bricks of 394 atoms instead of 12^3, of
// which 397 have a cell or two).  The threads are those of the mean brick and a
// few atoms more, or of the largest brick so far (a liquid's, which needs its size
// again and again: forgotten every 32 lists it cost 1.4 % of 3,456,000 atoms' steps).
// Bricks that did not fit any workgroup are tried again after BRICK_RETRY lists, so
// that a system which was uneven for a while returns to the better form; one that
// stays so builds a list in 32 twice.
#define BRICK_RETRY 32
static bool plan_bricks(mdk_ctx *c, int g[3]) {
  if (c->brick_bad && ++c->brick_wait > BRICK_RETRY) c->brick_bad = false;
  if (!brick_size(c) || !lean_pot(c) || c->lanes != 1 || c->brick_bad) return false;
  const int f[3] = {g[0] & ~3, g[1] & ~3, g[2] & ~3};
  auto atoms = [&](const int *q) { return 64.0 * c->n / ((double)q[0] * q[1] * q[2]); };
  const int *q = brick_threads(1.02 * atoms(f)) ? f : g;
  const int nt = brick_threads(1.02 * atoms(q)), nb = ((q[0] + 3) / 4) * ((q[1] + 3) / 4) * ((q[2] + 3) / 4);
  // (the partial sums have room for as many workgroups as the other passes have)
  if (nt == 0 || nb > c->part_cap || BRICK_CELLS * atoms(q) / 64.0 * 1.15 + 16 > BRICK_CAP_MAX) return false;
  c->brick_nt = std::max(c->brick_nt, nt);
  if (q == f) memcpy(g, f, sizeof(f));
  return true;
}
static int ensure_nbr(mdk_ctx *c) {
  if (!c->nbr) HIPCK(hipMalloc(&c->nbr, sizeof(int) * (size_t)c->maxn * c->n));
  return MDK_OK;
}
static int ensure_brick(mdk_ctx *c, double per_cell) {
  const int n = c->n;
  if (!c->nbr16) HIPCK(hipMalloc(&c->nbr16, sizeof(uint2) * (size_t)(c->maxn / 4) * n));
  if (!c->bcnt) HIPCK(hipMalloc(&c->bcnt, sizeof(int) * (size_t)n));
  // staged atoms with their null slot: the mean and some more for uneven cells
  if (!c->brick_cap) c->brick_cap = std::min(BRICK_CAP_MAX, (int)(BRICK_CELLS * per_cell * 1.15) + 16);
  const size_t need = (size_t)c->nlblocks * c->brick_cap;
  if (need > c->bstage_cap) {
    if (c->bstage) HIPCK(hipFree(c->bstage));
    c->bstage = nullptr;
    c->bstage_cap = 0;
    HIPCK(hipMalloc(&c->bstage, sizeof(int) * (need + need / 8)));
    c->bstage_cap = need + need / 8;
  }
  if ((size_t)c->nlblocks > c->binfo_cap) {
    if (c->binfo) HIPCK(hipFree(c->binfo));
    c->binfo = nullptr;
    c->binfo_cap = 0;
    HIPCK(hipMalloc(&c->binfo, sizeof(int4) * (size_t)c->nlblocks));
    c->binfo_cap = c->nlblocks;
  }
  return MDK_OK;
}
// after a build in which a brick's atoms (fl[1]) or their surroundings (fl[3]) did not fit
static void fit_bricks(mdk_ctx *c, const volatile int *fl) {
  const int nt = brick_threads(fl[1]);
  if (nt == 0 || fl[3] > BRICK_CAP_MAX) {
    c->brick_bad = true;
    c->brick_wait = 0;
  }
  c->brick_nt = std::max(c->brick_nt, nt);
  if (fl[3]) c->brick_cap = std::min(BRICK_CAP_MAX, fl[3] + fl[3] / 16);
}
static BrickArgs brick_args(const mdk_ctx *c) {
  return BrickArgs{c->nbr16, c->bstage, c->binfo, c->brick_cap, ldexpf(1.f, c->brick_k), ldexpf(1.f, -c->brick_k)};
}

// Full-list rebuild: fine grid from the current box, re-sort atoms by cell,
// build the list; grows the per-atom capacity and retries on overflow.
// defer: one attempt whose flags the caller checks after queueing the next
// kernels (confirm_list); otherwise every attempt is checked here.
static int rebuild_full(mdk_ctx *c, bool defer = false, bool force_follows = false) {
  const int n = c->n;
  c->list_valid = false;
  TimedEv te;
  tbegin(c, TC_REBUILD, te);
  // Grid from the box.  Inside the MD loop the box of a completed step comes
  // from the monitor ring (no host round trip before the build; cells planned
  // 1 % wider than the list radius cover the box change of a few steps);
  // otherwise it is read synchronously.  The host reads the list kernel's
  // flags before any force uses the list (here, or in confirm_list after the
  // density pass is queued): a list that overflowed grows its capacity and is
  // built again, and a grid found too narrow for the current box is planned
  // again from the exact box -- so no flagged list is ever used.
  bool lagged = c->rebuilds > 0 && c->b0_lag_step >= 0 && c->step_counter - c->b0_lag_step <= 4;
  for (int plan = 0; plan < 3; plan++) {
    double b0[9];
    if (lagged) {
      memcpy(b0, c->b0_lag, sizeof(b0));
    } else {
      BoxState bs;
      RCK(read_box(c, &bs));
      memcpy(b0, bs.b0, sizeof(b0));
    }
    int g[3];
    plan_grid(c, b0, g, lagged ? 1.01 : 1.0);
    // staged blocks and bricks need a fully periodic box with >= 4 cells per
    // dimension (and 26-bit atom indices); they pack positions cell-relative
    const bool blk = c->pbc == 7 && g[0] >= 4 && g[1] >= 4 && g[2] >= 4 && n < (1 << 26);
    c->rel = blk;
    c->brick = blk && plan_bricks(c, g);
    int p2 = 1;
    while (p2 < std::max(g[0], std::max(g[1], g[2]))) p2 <<= 1;
    const int m = p2 * p2 * p2;  // Morton key space
    c->grid[0] = g[0]; c->grid[1] = g[1]; c->grid[2] = g[2];
    RCK(ensure_cells(c, m));
    if (n <= SORT_ONE_ATOMS && m <= SORT_ONE_CELLS) {
      k_sort_one<<<1, 1024, 0, c->stream>>>(c->atoms, n, g[0], g[1], g[2], m, c->cell_of, c->cell_start, c->members);
      RCK(check_launch("k_sort_one"));
    } else {
      k_bin<<<nblocks(n), MDK_BLOCK, 0, c->stream>>>(c->atoms, n, g[0], g[1], g[2], c->cell_of, c->cell_count);
      RCK(scan_and_fill(c, c->cell_of, m));
    }
    const double rl2 = c->r_list * c->r_list;
    // physical re-sort of every per-atom array into cell order; images, list
    // cells and packed positions of the new list
    k_place<<<nblocks(n), MDK_BLOCK, 0, c->stream>>>(
        c->atoms_alt, c->atoms, c->members, c->cell_of, c->cell_start, n, resort_fields(c, force_follows), c->zat_alt,
        c->zat, c->orig_alt, c->orig, c->ic_alt, c->ic, c->cell_alt, c->slot_of, c->img, c->sref, c->pos4, p4f_of(c),
        pack_geo(c), c->box + c->cur, c->dflags);
    RCK(check_launch("k_place"));
    std::swap(c->atoms, c->atoms_alt);
    std::swap(c->zat, c->zat_alt);
    std::swap(c->orig, c->orig_alt);
    std::swap(c->ic, c->ic_alt);
    std::swap(c->cell_of, c->cell_alt);
    c->pos4_valid = c->p4f_valid = true;
    const double per_cell = (double)n / ((double)g[0] * g[1] * g[2]);
    const bool waves = !c->brick && list_by_waves(n, blk, per_cell);
    bool replan = false;
    for (int attempt = 0; attempt < 4; attempt++) {
      if (blk) RCK(plan_list_blocks(c, g, c->brick ? 4 : 2));
      c->nbp = c->brick ? c->nlblocks : nblocks((long)n * c->lanes);
      c->part_due = !waves && !c->brick;  // the other lists have their in-range partners first
      c->wide_valid = false;
      if (!c->brick) RCK(ensure_nbr(c));
      if (attempt > 0) HIPCK(hipMemsetAsync(c->dflags, 0, sizeof(int) * 4, c->stream));  // k_place cleared them
      if (waves) {
        const int per = n <= 8192 ? 1 : 4;
        const double rin = c->pot.r_int + 1e-4;  // the density pass's in-range test
        k_full_list_wave<<<(n + per - 1) / per + 1, 64, 0, c->stream>>>(
            c->pos4, c->atoms, c->img, c->cell_of, c->cell_start, n, g[0], g[1], g[2], pack_geo(c), c->box + c->cur,
            rl2, rin * rin, c->pbc, per, c->maxn, c->nbr, c->numn, c->dflags);
        RCK(check_launch("k_full_list_wave"));
      } else if (c->brick) {
        c->brick_built = false;
        RCK(ensure_brick(c, per_cell));
        // staged coordinates: three cells from the centre at most, below 2^29 units
        double ext = 0.0;
        for (int a = 0; a < 3; a++)
          ext = std::max(ext, fabs(b0[a]) / g[0] + fabs(b0[a + 3]) / g[1] + fabs(b0[a + 6]) / g[2]);
        c->brick_k = 29 - (ilogb(3.6 * ext) + 1);
        const double rin = c->pot.r_int + 1e-4;
        with_brick_threads(c->brick_nt, [&](auto nt) {
          k_brick_list<nt()><<<c->nlblocks, nt(), sizeof(float4) * c->brick_cap, c->stream>>>(
              c->p4f, c->cell_of, c->cell_start, c->lblocks, n, pack_geo(c), c->box + c->cur, rl2, rin * rin,
              c->maxn / 4, c->brick_cap, c->nbr16, c->bcnt, c->bstage, c->binfo, c->dflags);
        });
        RCK(check_launch("k_brick_list"));
        c->brick_built = true;
      } else if (blk) {
        k_full_list_blk<<<c->nlblocks, 64, 0, c->stream>>>(
            c->pos4, c->atoms, c->img, c->cell_of, c->cell_start, c->lblocks, n, pack_geo(c), c->box + c->cur,
            rl2, c->maxn, c->nbr, c->numn, c->dflags);
        RCK(check_launch("k_full_list_blk"));
      } else {
        k_full_list<<<nblocks(n), MDK_BLOCK, 0, c->stream>>>(
            c->pos4, c->atoms, c->img, c->cell_of, c->cell_start, n, g[0], g[1], g[2], c->box + c->cur, rl2,
            c->pbc, c->maxn, c->nbr, c->numn, c->dflags);
        RCK(check_launch("k_full_list"));
      }
      if (defer) {
        c->list_stamp = c->list_stamp == INT_MAX ? 1 : c->list_stamp + 1;
        c->report_due = true;  // by the density pass on it
        c->list_valid = true;
        c->list_pending = true;
        c->rebuilds++;
        c->last_rebuild_step = (int)c->step_counter;  // skin samples before this step predate the list
        tend(c, te);
        return MDK_OK;
      }
      int fl[4];
      HIPCK(hipMemcpyAsync(fl, c->dflags, sizeof(fl), hipMemcpyDeviceToHost, c->stream));
      HIPCK(hipStreamSynchronize(c->stream));
      if (fl[2] != 0) {
        if (!lagged) {
          tend(c, te);
          return set_err(MDK_ERR_STATE, "list cells narrower than the list radius");
        }
        replan = true;  // planned from a stale box: plan again from the exact one
        break;
      }
      if (fl[1] != 0 || fl[3] != 0) {  // a brick's atoms or surroundings did not fit
        fit_bricks(c, fl);
        replan = c->brick_bad;
        if (replan) break;
        continue;
      }
      if (fl[0] == 0) {
        c->list_valid = true;
        c->rebuilds++;
        c->last_rebuild_step = (int)c->step_counter;  // skin samples before this step predate the list
        tend(c, te);
        return MDK_OK;
      }
      // grow capacity to the observed maximum (+25%) and retry
      const int newmax = ((int)(fl[0] * 1.25) + 8 + 3) & ~3;
      c->brick_built = false;
      for (void **q : {(void **)&c->nbr, (void **)&c->nbr16}) {  // allocated again where needed
        if (*q) HIPCK(hipFree(*q));
        *q = nullptr;
      }
      c->maxn = newmax;
    }
    if (!replan) break;
    lagged = false;
  }
  tend(c, te);
  HIPCK(hipMemsetAsync(c->numn, 0, sizeof(int) * n, c->stream));
  return set_err(MDK_ERR_NBR_OVERFLOW, "full neighbour list overflow (max %d)", c->maxn);
}

// The FP32 form gathers the 16-byte FP32 copy of cell-relative packed
// positions (P32); absolute packing and the FP64 form gather the FP64 record.
static int pot_mode(const mdk_ctx *c);
// The FP32 form's lean kernels: Fe-Fe interval table, cell-relative lists, no
// immobile atoms (the per-pair mass test).
static bool lean_pot(const mdk_ctx *c) {
  return c->p.precision == MDK_PREC_FP32 && pot_mode(c) == POT_FE && !c->masschk;
}
static bool lean_path(const mdk_ctx *c) { return c->rel && lean_pot(c); }
// Lanes per atom of the pair passes.  With one lane per atom a system of a few
// thousand atoms keeps a few workgroups busy with a chain of four to seven
// (iron_carbon: sixteen) dependent index and partner loads; eight lanes take a
// quad of partners each, so the chain is one or two long and eight times as
// many waves hide it.  us per NPT step, one lane : eight lanes --
//   atoms         2000         16,000       31,250       65,536        128,000
//   Fe FP64       36.4 : 27.4  37.7 : 30.2  40.1 : 36.4  42.0 : 45.2   50.6 : 69.4
//   Fe FP32       34.5 : 28.0  35.4 : 29.3  38.1 : 33.9  39.5 : 39.6   44.2 : 59.4
//   iron_carbon   93.9 : 33.9  95.4 : 40.0  99.4 : 51.3  105.6 : 75.0  134.1 : 128.2
// so the line lies higher for the longer lists of ranges above 4.5 A.  The Fe passes
// take four and two lanes in between, whose lists of five or six quads leave fewer
// lanes idle; us per NVE step (NPT) --
//   Fe FP64   8192: 8 14.0 (21.4), 4 14.6 (21.1)     16,000: 8 16.8 (24.3), 4 15.3 (22.7)
//             31,250: 8 24.5 (31.5), 4 19.3 (28.7)   43,904: 4 22.2 (31.6), 2 22.3 (32.5), 1 23.4 (33.4)
//             78,608: 2 29.0 (40.8), 4 31.5 (42.1), 1 32.7 (45.2)
//             128,000: 1 32.4 (47.0), 2 36.6 (47.7)
//   Fe FP32   31,250: 8 20.5 (29.8), 4 17.7 (27.0)   65,536: 2 20.4 (31.8), 4 22.1 (31.8), 1 22.9 (36.4)
//             101,306: 2 25.2 (35.4), 1 25.3 (38.8)  128,000: 1 27.0 (41.7), 2 27.4 (38.3)
#define PAIR_8_ATOMS 8192
#define PAIR_4_ATOMS 48000
#define PAIR_2_ATOMS 110000
#define PAIR_LANES_ATOMS 40000
#define PAIR_LANES_ATOMS_LONG 131072
static int pair_lanes(int n, double r_list, bool fe) {
  if (fe) return n <= PAIR_8_ATOMS ? 8 : (n <= PAIR_4_ATOMS ? 4 : (n <= PAIR_2_ATOMS ? 2 : 1));
  return n <= (r_list > 4.5 ? PAIR_LANES_ATOMS_LONG : PAIR_LANES_ATOMS) ? 8 : 1;
}
// calls f with the lanes per atom as a constant; two and four are the Fe passes' alone
template <int POTM, typename F>
static void with_lanes(int lanes, F f) {
  if (lanes == 8) return f(std::integral_constant<int, 8>());
  if constexpr (POTM == POT_FE) {
    if (lanes == 4) return f(std::integral_constant<int, 4>());
    if (lanes == 2) return f(std::integral_constant<int, 2>());
  }
  f(std::integral_constant<int, 1>());
}
// after every change of the range
static void set_pair_lanes(mdk_ctx *c) {
  c->lanes = pair_lanes(c->n, c->r_list, pot_mode(c) == POT_FE && c->r_list <= 4.5);
  c->nbp = nblocks((long)c->n * c->lanes);
}

// the placement of the passes (place_of), and their grid
static int one_xcd(const mdk_ctx *c) { return c->lanes > 1 && c->nbp <= ONE_XCD_BLOCKS; }
static int placed(const mdk_ctx *c, int blocks) { return one_xcd(c) ? MDK_NXCD * blocks : blocks; }

// Takes the deferred finishing for this density pass and the buffer of its
// embedding-energy partials (the other one may still be read by the finishing).
static Rider take_ride(mdk_ctx *c, int do_embed, int blocks) {
  const Rider R = {c->ride, {c->dflags, c->flags_map, c->report_due ? c->list_stamp : 0}, one_xcd(c)};
  c->ride.kind = 0;
  c->report_due = false;
  if (do_embed) {
    c->emb_slot = 1 - c->emb_slot;
    c->emb_nb = blocks;
  }
  return R;
}

// The brick list's pairs in nbr and numn, for a caller that reads those.
static int ensure_wide_list(mdk_ctx *c) {
  if (!c->brick || !c->brick_built || c->wide_valid) return MDK_OK;
  RCK(ensure_nbr(c));
  k_brick_expand<<<c->nlblocks, c->brick_nt, 0, c->stream>>>(c->cell_of, c->lblocks, c->n, c->brick_cap, c->nbr16,
                                                             c->bcnt, c->bstage, c->binfo, c->maxn, c->nbr, c->numn);
  c->wide_valid = true;
  return check_launch("k_brick_expand");
}

static void lean_density(mdk_ctx *c, int do_embed) {
  const int blocks = c->part_due ? c->nblk : c->nbp;
  const Rider R = take_ride(c, do_embed, blocks);
  const int grid = placed(c, blocks) + (R.fin.kind || R.list.stamp ? MDK_NXCD : 0);
  double *pe = emb_buf(c, c->emb_slot);
  // F' goes to the FP32 records only: the FP64 copy is not kept on this path
  if (c->brick) {
    with_brick_threads(c->brick_nt, [&](auto nt) {
      k_density_brick<nt()><<<grid, nt(), sizeof(int4) * c->brick_cap, c->stream>>>(
          c->atoms, c->p4f, c->n, brick_args(c), c->bcnt, c->box + c->cur, pack_geo(c), c->pot, do_embed, pe, c->nact, R);
    });
    c->pos4_valid = false;
    return;
  }
#define MDK_DENS_F32_ARGS c->atoms, nullptr, c->p4f, c->n, c->nbr, c->numn, c->maxn, c->box + c->cur, pack_geo(c), c->pot, do_embed, pe, c->nact, R
  if (c->part_due)
    k_density_part_f32<<<grid, MDK_BLOCK, 0, c->stream>>>(c->atoms, c->p4f, c->n, c->nbr, c->numn, c->box + c->cur,
                                                          pack_geo(c), c->pot, do_embed, pe, c->nact, R);
  else
    with_lanes<POT_FE>(c->lanes,
                       [&](auto L) { k_density_f32<L()><<<grid, MDK_BLOCK, 0, c->stream>>>(MDK_DENS_F32_ARGS); });
#undef MDK_DENS_F32_ARGS
  c->pos4_valid = false;
  c->part_due = false;
}
// a force pass's fused kick, or only its placement
static KickIo kick_io(const mdk_ctx *c, const KickIo *K) {
  KickIo io = K ? *K : KickIo{};
  io.one_xcd = one_xcd(c);
  return io;
}
// a force pass, by the dispatch that fills in its events where it is timed
template <typename... A>
static void launch_timed(mdk_ctx *c, void (*k)(A...), int threads, size_t lds, hipEvent_t ea, hipEvent_t eb, A... args) {
  const int grid = placed(c, c->nbp);
  if (ea) hipExtLaunchKernelGGL(k, dim3(grid), dim3(threads), lds, c->stream, ea, eb, 0, args...);
  else k<<<grid, threads, lds, c->stream>>>(args...);
}
static void lean_force(mdk_ctx *c, const KickIo *K, hipEvent_t ea, hipEvent_t eb) {
  if (c->brick) {
    with_brick_threads(c->brick_nt, [&](auto nt) {
      auto k = K ? k_force_brick<nt(), true> : k_force_brick<nt(), false>;
      launch_timed(c, k, nt(), sizeof(int4) * c->brick_cap, ea, eb, c->atoms, (const float4 *)c->p4f, c->n, brick_args(c),
                   (const int *)c->nact, (const BoxState *)(c->box + c->cur), pack_geo(c), c->pot, c->part_f,
                   (const float *)c->fetab, kick_io(c, K));
    });
    return;
  }
  with_lanes<POT_FE>(c->lanes, [&](auto L) {
    auto k = K ? k_force_f32<L(), true> : k_force_f32<L(), false>;
    launch_timed(c, k, MDK_BLOCK, 0, ea, eb, c->atoms, (const float4 *)c->p4f, c->n, (const int *)c->nbr, (const int *)c->nact, c->maxn,
                 (const BoxState *)(c->box + c->cur), pack_geo(c), c->pot, c->part_f, (const float *)c->fetab,
                 kick_io(c, K));
  });
}

template <typename T, int POTM, bool P32>
static void density_dispatch_p(mdk_ctx *c, int do_embed) {
  const int blocks = c->part_due ? c->nblk : c->nbp;
  const Rider R = take_ride(c, do_embed, blocks);
  const int grid = placed(c, blocks) + (R.fin.kind || R.list.stamp ? MDK_NXCD : 0);
  double *pe = emb_buf(c, c->emb_slot);
#define MDK_DENS_REST c->box + c->cur, pack_geo(c), c->pot, do_embed, pe, c->nact, R
#define MDK_DENS_ARGS c->atoms, c->pos4, p4f_of(c), c->n, c->nbr, c->numn, c->maxn, MDK_DENS_REST
  if (c->part_due)
    k_density_part<T, POTM, P32><<<grid, MDK_BLOCK, 0, c->stream>>>(c->atoms, c->pos4, p4f_of(c), c->n, c->nbr, c->numn,
                                                                    MDK_DENS_REST);
  else
    with_lanes<POTM>(c->lanes,
                     [&](auto L) { k_density<T, POTM, P32, L()><<<grid, MDK_BLOCK, 0, c->stream>>>(MDK_DENS_ARGS); });
#undef MDK_DENS_ARGS
#undef MDK_DENS_REST
  c->part_due = false;
}
template <typename T, int POTM>
static void density_dispatch(mdk_ctx *c, int do_embed) {
  if constexpr (sizeof(T) == 4) {
    if (c->rel) return density_dispatch_p<T, POTM, true>(c, do_embed);
  }
  density_dispatch_p<T, POTM, false>(c, do_embed);
}
template <typename T, bool MC, int POTM, bool P32>
static void force_dispatch_p(mdk_ctx *c, const KickIo *K, hipEvent_t ea, hipEvent_t eb) {
  // tabulated pair terms interpolate across the range edge: those use the whole list
  with_lanes<POTM>(c->lanes, [&](auto L) {
    auto k = k_force<T, MC, POTM, P32, L(), false>;
    if constexpr (!MC) {  // the fused kick forms no virial, which alone needs the masses
      if (K) k = k_force<T, MC, POTM, P32, L(), true>;
    }
    launch_timed(c, k, MDK_BLOCK, 0, ea, eb, c->atoms, (const double4 *)c->pos4, (const float4 *)p4f_of(c), c->n, (const int *)c->nbr,
                 (const int *)(POTM == POT_TABLE ? c->numn : c->nact), c->maxn, (const BoxState *)(c->box + c->cur), pack_geo(c),
                 c->pot, c->part_f, (const float *)c->fetab, kick_io(c, K));
  });
}
template <typename T, bool MC, int POTM>
static void force_dispatch(mdk_ctx *c, const KickIo *K, hipEvent_t ea, hipEvent_t eb) {
  if constexpr (sizeof(T) == 4) {
    if (c->rel) return force_dispatch_p<T, MC, POTM, true>(c, K, ea, eb);
  }
  force_dispatch_p<T, MC, POTM, false>(c, K, ea, eb);
}
// lookup tables, iron_carbon (FP64 only: set-up refuses the FP32 form), the
// fetransmetal Fe-Fe knot counts, or any knot count
static int pot_mode(const mdk_ctx *c) {
  if (c->pot.use_lookup) return POT_TABLE;
  if (c->material == MDK_MAT_IRON_CARBON) return POT_FEC;
  if (c->pot.nv != MDK_FE_NV || c->pot.np != MDK_FE_NP) return POT_KNOTS;
  return (c->p.precision == MDK_PREC_FP32 && !c->fe_ok) ? POT_KNOTS : POT_FE;
}
template <typename T>
static void density_pot(mdk_ctx *c, int do_embed) {
  switch (pot_mode(c)) {
    case POT_TABLE: density_dispatch<T, POT_TABLE>(c, do_embed); break;
    case POT_FE: density_dispatch<T, POT_FE>(c, do_embed); break;
    case POT_FEC:
      if constexpr (sizeof(T) == 8) density_dispatch<T, POT_FEC>(c, do_embed);
      break;
    default: density_dispatch<T, POT_KNOTS>(c, do_embed); break;
  }
}
template <typename T, bool MC>
static void force_pot(mdk_ctx *c, const KickIo *K, hipEvent_t ea, hipEvent_t eb) {
  switch (pot_mode(c)) {
    case POT_TABLE: force_dispatch<T, MC, POT_TABLE>(c, K, ea, eb); break;
    case POT_FE: force_dispatch<T, MC, POT_FE>(c, K, ea, eb); break;
    case POT_FEC:
      if constexpr (sizeof(T) == 8) force_dispatch<T, MC, POT_FEC>(c, K, ea, eb);
      break;
    default: force_dispatch<T, MC, POT_KNOTS>(c, K, ea, eb); break;
  }
}

static int ensure_pos4(mdk_ctx *c) {
  if (c->pos4_valid) return MDK_OK;
  c->p4f_valid = true;
  k_pack<<<nblocks(c->n), MDK_BLOCK, 0, c->stream>>>(c->atoms, c->img, c->box + c->cur, c->n, c->pos4, p4f_of(c),
                                                     c->cell_of, pack_geo(c));
  c->pos4_valid = true;
  return check_launch("k_pack");
}

static int launch_density(mdk_ctx *c, int do_embed) {
  if (!(lean_path(c) && c->p4f_valid)) RCK(ensure_pos4(c));  // the lean passes read only the FP32 records
  TimedEv te;
  tbegin(c, TC_DENSITY, te);
  if (lean_path(c)) {
    lean_density(c, do_embed);
  } else if (c->p.precision == MDK_PREC_FP32) {
    density_pot<float>(c, do_embed);
  } else {
    density_pot<double>(c, do_embed);
  }
  tend(c, te);
  return check_launch("k_density");
}

// K: the fused kick of a fixed-box step, or null
static int launch_force(mdk_ctx *c, const KickIo *K = nullptr) {
  if (!K && !c->kin_fresh) {  // no drift, predictor or fused kick prepared kinten's sums
    k_kin<<<c->nblk, MDK_BLOCK, 0, c->stream>>>(c->atoms, c->zat, c->n, c->box + c->cur, spec_of(c),
                                                kin_buf(c, c->kin_slot));
    RCK(check_launch("k_kin"));
    c->kin_nb = c->nblk;
  }
  c->kin_fresh = false;  // consumed by this force evaluation
  TimedEv te;
  tbegin_ext(c, TC_FORCE, te);  // the force kernel's own start and end
  hipEvent_t ea = te.cls >= 0 ? te.a : nullptr, eb = te.cls >= 0 ? te.b : nullptr;
  const bool f32 = c->p.precision == MDK_PREC_FP32, mc = c->masschk && !K;
  if (lean_path(c)) {
    lean_force(c, K, ea, eb);
  } else if (f32) {
    if (mc) force_pot<float, true>(c, K, ea, eb); else force_pot<float, false>(c, K, ea, eb);
  } else {
    if (mc) force_pot<double, true>(c, K, ea, eb); else force_pot<double, false>(c, K, ea, eb);
  }
  tpush(c, te);
  return check_launch("k_force");
}

static FinForce fin_force(mdk_ctx *c, int fin_mode) {
  return FinForce{{c->part_f, emb_buf(c, c->emb_slot), kin_buf(c, c->kin_slot), c->nbp, c->emb_nb, c->kin_nb},
                  c->stage_f, c->fin_cnt, c->box + c->cur, fin_mode, c->p.ivol, c->p.press, c->p.bdel2, c->p.deltat, one_xcd(c)};
}
static int launch_finish(mdk_ctx *c, int fin_mode) {
  const FinForce F = fin_force(c, fin_mode);
  if (c->nbp <= FIN_ONE_BLOCKS) k_finalize_force_one<<<1, FIN_ONE_THREADS, 0, c->stream>>>(F);
  else k_finalize_force<<<(std::max(c->nbp, std::max(c->emb_nb, c->kin_nb)) + 63) / 64, MDK_FIN_BLOCK, 0, c->stream>>>(F);
  return check_launch("k_finalize_force");
}

// Completes a deferred finishing on its own (the last step of an MD call).
static int flush_ride(mdk_ctx *c) {
  if (!c->ride.kind) return MDK_OK;
  k_finish_step<<<1, FINISH_THREADS, 0, c->stream>>>(c->ride);
  c->ride.kind = 0;
  return check_launch("k_finish_step");
}

// FX..FZ of the last step of a call that stopped after one with a fused kick, which
// forms no forces for memory: from the packed records that its force pass read (the
// alternate ones by now, F' included) over the same list.
static int last_forces(mdk_ctx *c) {
  const bool fp64 = !lean_path(c), kin = c->kin_fresh;
  std::swap(c->p4f, c->p4f_alt);
  if (fp64) std::swap(c->pos4, c->pos4_alt);
  c->kin_fresh = true;  // no sums are wanted
  const int rc = launch_force(c);
  c->kin_fresh = kin;
  std::swap(c->p4f, c->p4f_alt);
  if (fp64) std::swap(c->pos4, c->pos4_alt);
  return rc;
}

// Waits until the device has written the stamp: a spin on host-mapped memory
// (an event wait wakes the host microseconds later); a stream that failed or
// drained without writing it ends the wait.
template <typename V>
static int wait_stamp(mdk_ctx *c, const volatile V *p, V stamp) {
  for (long spin = 1; *p != stamp; spin++) {
    if (spin & 0xffff) continue;
    const hipError_t e = hipStreamQuery(c->stream);
    if (e == hipErrorNotReady || *p == stamp) continue;
    if (e != hipSuccess) return set_err(MDK_ERR_HIP, "waiting for the device: %s", hipGetErrorString(e));
    return set_err(MDK_ERR_HIP, "the device did not report a finished step");
  }
  std::atomic_thread_fence(std::memory_order_acquire);
  return MDK_OK;
}

// Checks the flags of a deferred build (the density pass on it is queued and
// may run meanwhile; a flagged list yields wrong values but valid indices).
// A flagged build is discarded: the list is built again with every attempt
// checked (grown capacity, grid from the exact box) and the density pass
// repeated, before any force uses it.
static int confirm_list(mdk_ctx *c) {
  if (!c->list_pending) return MDK_OK;
  c->list_pending = false;
  const volatile int *fl = c->flags_host;
  RCK(wait_stamp(c, fl + 4, c->list_stamp));
  if (fl[0] == 0 && fl[1] == 0 && fl[2] == 0 && fl[3] == 0) return MDK_OK;
  HIPCK(hipStreamSynchronize(c->stream));
  if (fl[1] || fl[3]) fit_bricks(c, fl);  // the exact box's grid may differ and not show it
  c->rebuilds--;
  c->b0_lag_step = -1;
  RCK(rebuild_full(c, false, true));
  return launch_density(c, 1);
}

// force() bookkeeping of src/dynamics_m.F90:186-198 plus the skin criterion
// kick: with the fixed-box kick and drift in the force pass (kin: and kinten's
// sums for the next force evaluation; link: and this step's link cells)
static int force_body(mdk_ctx *c, bool skin_due, bool kick = false, bool kin = false, bool link = false) {
  if (!c->pot_set) return set_err(MDK_ERR_STATE, "potential not set");
  c->ntc = c->ntc + 1;
  bool ref_due = (c->ntc == 1);
  if (c->ntc == c->p.ntcm) c->ntc = 0;
  bool due = !c->list_valid || skin_due || (ref_due && c->p.rebuild == 0);
  if (due) RCK(rebuild_full(c, true, true));
  RCK(launch_density(c, 1));
  RCK(confirm_list(c));
  if (!kick) return launch_force(c);
  // FP32 systems outside the Fe path read the FP64 records as well
  if (!lean_path(c) && !c->pos4_alt) HIPCK(hipMalloc((void **)&c->pos4_alt, sizeof(double4) * (size_t)c->n));
  const KickIo K = {c->zat, c->sref, c->img, c->cell_of, spec_of(c), lean_path(c) ? nullptr : c->pos4_alt,
                    c->p.precision == MDK_PREC_FP32 ? c->p4f_alt : nullptr, c->part_f,
                    kin ? kin_buf(c, c->kin_slot) : nullptr, c->p.ivol, link_grid(c, link), 0};
  return launch_force(c, &K);
}
static int force_and_finish(mdk_ctx *c, int fin_mode, bool skin_due) {
  RCK(force_body(c, skin_due));
  return launch_finish(c, fin_mode);
}

// Half kick (mode 0), sums only (1) or initial accelerations (2).  With
// fuse_drift (mode 0) the kernel also performs the next step's drift; the
// finishing block then completes this step's sums on the current box copy and
// the next md_step skips its drift.
// defer (mode 0): the sums' finishing is left to the next density pass (or
// flush_ride).
static int launch_kick(mdk_ctx *c, int mode, double *trace_row_dev, double *mon, bool fuse_drift = false,
                       bool defer = false, bool link = false) {
  TimedEv te;
  tbegin(c, TC_KICK, te);
  const int nxt = next_box(c);
  const bool fused = fuse_drift && mode == 0;
  if (fused)
    k_kick<true><<<c->nblk, MDK_BLOCK, 0, c->stream>>>(
        c->atoms, c->zat, c->n, c->box + c->cur, c->p.ivol, mode, c->sref, c->part_k,
        lean_path(c) ? nullptr : c->pos4, p4f_of(c), c->img, c->cell_of, pack_geo(c), c->box + nxt, spec_of(c),
        kin_buf(c, c->kin_slot), link_grid(c, link));
  else
    k_kick<false><<<c->nblk, MDK_BLOCK, 0, c->stream>>>(
        c->atoms, c->zat, c->n, c->box + c->cur, c->p.ivol, mode, c->sref, c->part_k, nullptr, nullptr,
        nullptr, nullptr, pack_geo(c), nullptr, spec_of(c), nullptr, link_grid(c, false));
  tend(c, te);
  RCK(check_launch("k_kick"));
  if (mode != 2) {  // initial accelerations have no sums
    const FinKick F = {c->box + c->cur, fused ? c->box + nxt : nullptr, trace_row_dev, mon, c->p.deltat, c->p.bdel2,
                       c->p.press, (double)(c->step_counter + 1)};
    if (defer && mode == 0) {
      c->ride = FinRide{1, c->nblk, 0, c->part_k, nullptr, F};
    } else {
      k_finish_step<<<1, FINISH_THREADS, 0, c->stream>>>(FinRide{1, c->nblk, 0, c->part_k, nullptr, F});
      RCK(check_launch("k_finish_step"));
    }
  }
  if (fused) {
    c->pos4_valid = !lean_path(c);
    c->p4f_valid = true;
    c->cur = nxt;
    c->drifted = true;
    c->kin_fresh = true;
    c->kin_nb = c->nblk;
  }
  return MDK_OK;
}

// force()'s finishing and the half kick of a small system in one launch (the
// MD loop); the kick's sums stay pending as with a deferred launch_kick.
// Every workgroup folds the partials of every workgroup of the pair passes, so what
// it saves (a launch and the gap) is lost where the product of the two numbers is
// large.  us per NPT step, two kernels : one, FP64 (FP32) --
//   eight lanes per atom  2000 22.2 : 19.3 (22.7 : 20.0)    8192 24.0 : 21.5 (24.5 : 22.4)
//   four                  16,000 24.3 : 23.1 (24.7 : 23.1)  31,250, product 60,000: 28.8 : 28.3 (27.3 : 27.3)
//                         39,366, 95,000: 31.0 : 31.2 (28.6 : 28.7)  47,096, 136,000: 32.0 : 32.6 (29.5 : 30.0)
//   two                   54,000, 89,000: 32.4 : 32.7 (30.4 : 30.8)  78,608, 189,000: 38.5 : 39.7 (33.9 : 35.2)
//   one                   128,000, 250,000: 44.0 : 45.9 (39.0 : 40.3)  159,014, 387,000: 53.7 : 54.5 (42.6 : 44.4)
//   eight, iron_carbon    16,000, 31,500: 32.9 : 32.6  21,296, 56,000: 38.0 : 37.9  27,648, 93,000: 43.0 : 43.9
#define FIN_KICK_FOLDS 64000
static int launch_finish_kick(mdk_ctx *c, double *trace_row_dev, double *mon, bool fuse_drift, bool link) {
  const FinForce F = fin_force(c, FIN_VV_THERM);
  BoxState *fin = c->box + next_box(c), *nxt = c->box + next_box(c, 2);
  TimedEv te;
  tbegin(c, TC_KICK, te);
  auto k = fuse_drift ? k_finish_kick<true> : k_finish_kick<false>;
  k<<<placed(c, c->nblk), MDK_BLOCK, 0, c->stream>>>(F, fin, c->atoms, c->zat, c->n, c->sref, c->part_k,
                                          lean_path(c) ? nullptr : c->pos4, p4f_of(c), c->img, c->cell_of,
                                          pack_geo(c), nxt, spec_of(c), kin_buf(c, 1 - c->kin_slot), link_grid(c, link));
  tend(c, te);
  RCK(check_launch("k_finish_kick"));
  c->ride = FinRide{1, c->nblk, 0, c->part_k, nullptr,
                    FinKick{fin, fuse_drift ? nxt : nullptr, trace_row_dev, mon, c->p.deltat, c->p.bdel2, c->p.press,
                            (double)(c->step_counter + 1)}};
  if (fuse_drift) {
    c->kin_slot = 1 - c->kin_slot;
    c->kin_nb = c->nblk;
    c->pos4_valid = !lean_path(c);
    c->p4f_valid = true;
    c->cur = next_box(c, 2);
    c->drifted = true;
    c->kin_fresh = true;
  } else {
    c->cur = next_box(c);
  }
  return MDK_OK;
}

static int launch_drift(mdk_ctx *c) {
  if (c->drifted) {  // performed by the previous step's fused kick
    c->drifted = false;
    return MDK_OK;
  }
  TimedEv te;
  tbegin(c, TC_DRIFT, te);
  const int nxt = next_box(c);
  k_drift<<<c->nblk, MDK_BLOCK, 0, c->stream>>>(c->atoms, lean_path(c) ? nullptr : c->pos4, p4f_of(c), c->img,
                                                c->cell_of, pack_geo(c), c->n, c->box + c->cur, c->box + nxt,
                                                c->p.ivol, c->zat, spec_of(c), kin_buf(c, c->kin_slot));
  c->pos4_valid = !lean_path(c);
  c->p4f_valid = true;
  c->kin_fresh = true;
  c->kin_nb = c->nblk;
  tend(c, te);
  c->cur = nxt;
  return check_launch("k_drift");
}

// Reads the monitor sample of step s-3 (its kernels have completed or the
// host waits for them): the box for the next grid plan and the skin bound.
// In the MD loop a step's sample is completed by the next step's density pass,
// so the host stays about two steps ahead of the GPU.
static int poll_monitor(mdk_ctx *c, const double **sample) {
  const long s = c->step_counter;
  *sample = nullptr;
  if (s < 3) return MDK_OK;
  const long probe = s - 3;
  const double *m = c->mon_host + MON_STRIDE * (int)(probe & 3);
  RCK(wait_stamp(c, (const volatile double *)m + MON_STAMP, (double)(probe + 1)));
  for (int k = 0; k < 9; k++) c->b0_lag[k] = m[MON_B0 + k];
  c->b0_lag_step = probe;
  *sample = m;
  return MDK_OK;
}

// Frobenius norm of A Bref^-1 - s I for the monitor's Bref (column-major 3x3)
static double strain_norm(const double *a, const double *bref, double s) {
  const double det = bref[0] * (bref[4] * bref[8] - bref[7] * bref[5]) -
                     bref[3] * (bref[1] * bref[8] - bref[7] * bref[2]) +
                     bref[6] * (bref[1] * bref[5] - bref[4] * bref[2]);
  double inv[9];  // cofactors / determinant, column-major
  inv[0] = (bref[4] * bref[8] - bref[7] * bref[5]) / det;
  inv[3] = -(bref[3] * bref[8] - bref[6] * bref[5]) / det;
  inv[6] = (bref[3] * bref[7] - bref[6] * bref[4]) / det;
  inv[1] = -(bref[1] * bref[8] - bref[7] * bref[2]) / det;
  inv[4] = (bref[0] * bref[8] - bref[6] * bref[2]) / det;
  inv[7] = -(bref[0] * bref[7] - bref[6] * bref[1]) / det;
  inv[2] = (bref[1] * bref[5] - bref[4] * bref[2]) / det;
  inv[5] = -(bref[0] * bref[5] - bref[3] * bref[2]) / det;
  inv[8] = (bref[0] * bref[4] - bref[3] * bref[1]) / det;
  double e2 = 0.0;
  for (int i = 0; i < 3; i++)
    for (int j = 0; j < 3; j++) {
      double x = (i == j) ? -s : 0.0;
      for (int k = 0; k < 3; k++) x += a[i + 3 * k] * inv[k + 3 * j];
      e2 += x * x;
    }
  return sqrt(e2);
}
// box strain since the list was built (B0 Bref^-1 - I) and that of the next
// drift's box change ((b1 + b2) Bref^-1)
static double strain_since_build(const double *m) { return strain_norm(m + MON_B0, m + MON_BREF, 1.0); }
static double strain_of_step(const double *m) { return strain_norm(m + MON_DB, m + MON_BREF, 0.0); }

// The list a step uses holds every pair within the potential's range while
// each atom has moved less than d and the box has strained by less than e
// (monitor sample: d^2 = m[0], e = strain_since_build) since the list was
// built, with 2 d + e r_list < skin: no pair separation has then changed by
// the skin.
static double skin_used(const mdk_ctx *c, const double *m) {
  return sqrt(fmax(m[0], 0.0)) + 0.5 * strain_since_build(m) * c->r_list;  // against skin / 2
}
static int skin_violation(const mdk_ctx *c, const double *m, long step) {
  return set_err(MDK_ERR_SKIN,
                 "step %ld: an atom moved %.4g A and the box strained %.3g since the list was built "
                 "(bound: skin/2 = %.4g A); pairs may have been missed",
                 step, sqrt(fmax(m[0], 0.0)), strain_since_build(m), 0.5 * c->skin);
}

// Checks the completed sample of step s-3 against the skin bound (an error if
// it was exceeded), then decides whether the next force evaluation could see
// it exceeded: that sample's displacement and strain plus four times its
// step's (m[1]: squared displacement of the next drift, strain_of_step: that
// of the next drift's box change) -- three drifts since the sample and one
// to spare.
static int skin_check(mdk_ctx *c, bool *due) {
  const double *m;
  RCK(poll_monitor(c, &m));
  *due = !c->list_valid;
  if (!m) return MDK_OK;
  if (skin_used(c, m) >= 0.5 * c->skin) return skin_violation(c, m, c->step_counter - 3);
  if (c->step_counter - c->last_rebuild_step < 4) return MDK_OK;  // the sample predates the list
  const double stp = sqrt(fmax(m[1], 0.0)) + 0.5 * strain_of_step(m) * c->r_list;
  *due = *due || skin_used(c, m) + 4.0 * stp >= 0.5 * c->skin;
  return MDK_OK;
}

static int launch_predic(mdk_ctx *c) {
  c->x3_live = true;
  TimedEv te;
  tbegin(c, TC_DRIFT, te);
  const int nxt = next_box(c);
  k_predic<<<c->nblk, MDK_BLOCK, 0, c->stream>>>(c->atoms, c->pos4, p4f_of(c), c->img, c->cell_of, pack_geo(c),
                                                 c->n, c->box + c->cur, c->box + nxt, c->p.ivol,
                                                 c->pc_primed ? 1 : 0, c->zat, spec_of(c), kin_buf(c, c->kin_slot));
  tend(c, te);
  c->pos4_valid = c->p4f_valid = true;
  c->kin_fresh = true;
  c->kin_nb = c->nblk;
  c->cur = nxt;
  return check_launch("k_predic");
}

static int launch_correc(mdk_ctx *c) {
  c->x3_live = true;
  TimedEv te;
  tbegin(c, TC_KICK, te);
  k_correc<<<c->nblk, MDK_BLOCK, 0, c->stream>>>(c->atoms, c->zat, c->n, c->box + c->cur, c->p.ivol,
                                                 c->p.bdel2, spec_of(c));
  tend(c, te);
  c->pos4_valid = c->p4f_valid = false;  // positions and box moved
  c->pc_primed = true;
  return check_launch("k_correc");
}

// One moldin step with iverlet = 0 (src/moldin.F90:754-758): PREDIC, FORCE,
// CORREC, then update_therm_avs (box part, then the sums with the monitor).
static int md_step_gear(mdk_ctx *c, double *trace_row_dev) {
  bool skin_due;
  RCK(skin_check(c, &skin_due));
  RCK(launch_predic(c));
  RCK(force_and_finish(c, FIN_FORCE, skin_due));
  RCK(launch_correc(c));
  k_therm_box<<<1, 64, 0, c->stream>>>(c->box + c->cur, c->p.ivol);
  RCK(check_launch("k_therm_box"));
  int slot = (int)(c->step_counter & 3);
  RCK(launch_kick(c, 1, trace_row_dev, c->mon_dev + MON_STRIDE * slot));
  c->step_counter++;
  return MDK_OK;
}

// One moldin step; its sums are finished by the next step's density pass,
// mdk_md_steps finishes the last one itself.  more: steps of the call that follow.
static int md_step(mdk_ctx *c, double *trace_row_dev, int more) {
  if (c->iverlet == 0) return md_step_gear(c, trace_row_dev);
  bool skin_due;
  RCK(skin_check(c, &skin_due));
  c->pc_primed = true;  // velocityverlet refreshes quench_m's parameter copy
  RCK(launch_drift(c));
  double *mon = c->mon_dev + MON_STRIDE * (int)(c->step_counter & 3);
  // the next drift follows in the same launch, after the relink's part where ntc
  // wraps in this force (moldin.F90:791): us per step, with separate passes at every
  // tenth step : without -- 2000 atoms NVE 15.5 : 14.8, 31,250 25.4 : 23.6 (NPT 32.6 :
  // 31.2), 524,288 95.6 : 91.1 (114.4 : 112.6; FP32 69.6 : 65.9, 87.9 : 86.5)
  const bool fuse = more > 0, link = fuse && c->ntc + 1 == c->p.ntcm;
  if (fuse && c->p.ivol >= 1 && c->p.ivol != 4) {
    // a box that does not move: the kick and the drift ride in the force pass
    // (kinten's sums only where the next step takes the plain passes)
    const bool plain_next = more == 1;
    RCK(force_body(c, skin_due, true, plain_next, link));
    c->ride = FinRide{2, c->nbp, c->emb_nb, c->part_f, emb_buf(c, c->emb_slot),
                      FinKick{c->box + c->cur, nullptr, trace_row_dev, mon, c->p.deltat, c->p.bdel2, c->p.press,
                              (double)(c->step_counter + 1)}};
    std::swap(c->p4f, c->p4f_alt);
    if (!lean_path(c)) std::swap(c->pos4, c->pos4_alt);
    c->pos4_valid = !lean_path(c);
    c->p4f_valid = true;
    c->drifted = true;
    c->kin_fresh = plain_next;
    c->kin_nb = c->nbp;
  } else {
    RCK(force_body(c, skin_due));
    if ((long)c->nblk * c->nbp <= FIN_KICK_FOLDS) {
      RCK(launch_finish_kick(c, trace_row_dev, mon, fuse, link));
    } else {
      RCK(launch_finish(c, FIN_VV_THERM));
      RCK(launch_kick(c, 0, trace_row_dev, mon, fuse, true, link));
    }
  }
  if (link) c->chains_exact = false;  // as relink_in_loop, whose cells the kick wrote
  c->step_counter++;
  return MDK_OK;
}

static int check_device_status(mdk_ctx *c) {
  BoxState bs;
  RCK(read_box(c, &bs));
  if (bs.status != 0) return set_err(bs.status, "singular box matrix in matrix_invert");
  return MDK_OK;
}

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------
static mdk_ctx *H(void *h) { return (mdk_ctx *)h; }

extern "C" int mdk_create(void **handle, const mdk_params *p) {
  if (!handle || !p) return set_err(MDK_ERR_BAD_ARG, "null argument");
  if (p->nm < 1 || p->nnbrs < 1 || p->ntcm < 1 || p->nlcx < 3 || p->nlcy < 3 || p->nlcz < 3 ||
      p->deltat <= 0.0 || p->rnear <= 0.0)
    return set_err(MDK_ERR_BAD_ARG, "bad parameters (nm=%d nnbrs=%d ntcm=%d)", p->nm, p->nnbrs, p->ntcm);
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return set_err(MDK_ERR_NO_DEVICE, "no HIP device");
  void *mem = ::operator new(sizeof(mdk_ctx));
  memset(mem, 0, sizeof(mdk_ctx));
  mdk_ctx *c = (mdk_ctx *)mem;
  new (&c->evs) std::vector<TimedEv>();
  new (&c->evpool) std::vector<hipEvent_t>();
  c->p = *p;
  c->n = p->nm;
  c->iverlet = 1;  // velocity Verlet unless mdk_set_integrator selects the predictor-corrector
  const int n = c->n;
  switch (p->ivol) {
    case 0: case 1: case 4: c->pbc = 7; break;
    case 2: c->pbc = 3; break;
    case 5: c->pbc = 4; break;
    default: c->pbc = 0; break;
  }
  hipGetDevice(&c->device);
  c->maxn = ((p->max_full > 0 ? p->max_full : 64) + 3) & ~3;

  c->skin = p->rskin > 0.0 ? p->rskin : 0.3;
  c->rnear2_exact = near_threshold(p->rnear);
  c->nblk = nblocks(n);
  set_pair_lanes(c);  // until a potential is set
  int rc = MDK_OK;
#define ALLOC(ptr, bytes)                                                          \
  do {                                                                             \
    if (hipMalloc((void **)&(ptr), (bytes)) != hipSuccess) {                       \
      rc = set_err(MDK_ERR_HIP, "hipMalloc %zu bytes failed", (size_t)(bytes));    \
      goto fail;                                                                   \
    }                                                                              \
  } while (0)
  if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
    rc = set_err(MDK_ERR_HIP, "stream create failed");
    goto fail;
  }
  ALLOC(c->atoms, sizeof(double) * (size_t)F_N * n);
  ALLOC(c->atoms_alt, sizeof(double) * (size_t)F_N * n);
  ALLOC(c->zat, sizeof(int) * n);
  ALLOC(c->zat_alt, sizeof(int) * n);
  ALLOC(c->orig, sizeof(int) * n);
  ALLOC(c->orig_alt, sizeof(int) * n);
  ALLOC(c->slot_of, sizeof(int) * n);
  ALLOC(c->sref, sizeof(float) * 3 * (size_t)n);
  ALLOC(c->ic, sizeof(int) * n);
  ALLOC(c->numn_ref, sizeof(int) * n);
  ALLOC(c->nlist_ref, sizeof(int) * (size_t)n * p->nnbrs);
  // the list's entries, in the form that the list will most likely have
  if (brick_size(c)) {
    ALLOC(c->nbr16, sizeof(uint2) * (size_t)(c->maxn / 4) * n);
    ALLOC(c->bcnt, sizeof(int) * n);
  } else {
    ALLOC(c->nbr, sizeof(int) * (size_t)c->maxn * n);
  }
  ALLOC(c->numn, sizeof(int) * n);
  ALLOC(c->nact, sizeof(int) * n);
  ALLOC(c->cell_of, sizeof(int) * n);
  ALLOC(c->cell_alt, sizeof(int) * n);
  ALLOC(c->ic_alt, sizeof(int) * n);
  ALLOC(c->ref_key, sizeof(int) * n);
  ALLOC(c->rank_orig, sizeof(int) * n);
  ALLOC(c->rank_slot, sizeof(int) * n);
  ALLOC(c->members, sizeof(int) * n);
  ALLOC(c->pos4, sizeof(double4) * (size_t)n);
  if (p->precision == MDK_PREC_FP32) ALLOC(c->p4f, sizeof(float4) * (size_t)n);
  if (p->ivol >= 1 && p->ivol != 4) {  // the next step's packed positions (fixed-box steps)
    if (p->precision == MDK_PREC_FP32) ALLOC(c->p4f_alt, sizeof(float4) * (size_t)n);
    else ALLOC(c->pos4_alt, sizeof(double4) * (size_t)n);
  }
  ALLOC(c->img, sizeof(int) * 3 * (size_t)n);
  c->part_cap = nblocks((long)n * pair_lanes(n, INFINITY, false));
  {  // the small arrays share one allocation
    const size_t cap = c->part_cap, nb = c->nblk;
    const struct {
      void **p;
      size_t bytes;
    } part[] = {{(void **)&c->part_f, sizeof(double) * NPART_FORCE * cap},
                {(void **)&c->emb2, sizeof(double) * 2 * cap},
                {(void **)&c->kin2, sizeof(double) * 2 * NPART_KIN * cap},
                {(void **)&c->part_k, sizeof(double) * NPART_KICK * nb},
                {(void **)&c->stage_f, sizeof(double) * (cap / 64 + 1) * NSUM_FORCE},
                {(void **)&c->stage_k, sizeof(double) * (nb / 64 + 1) * NPART_KICK},
                {(void **)&c->fin_cnt, sizeof(unsigned) * 2},
                {(void **)&c->red, sizeof(double) * 4},
                {(void **)&c->spec_tab, sizeof(double) * 2 * MDK_NSPEC},
                {(void **)&c->dflags, sizeof(int) * 4},
                {(void **)&c->box, sizeof(BoxState) * 4}};
    size_t sum = 0;
    for (const auto &q : part) sum += (q.bytes + 255) & ~(size_t)255;
    ALLOC(c->small, sum);
    char *at = c->small;
    for (const auto &q : part) {
      *q.p = at;
      at += (q.bytes + 255) & ~(size_t)255;
    }
  }
  if (hipMemset(c->fin_cnt, 0, sizeof(unsigned) * 2) != hipSuccess) {
    rc = set_err(MDK_ERR_HIP, "counter initialisation failed");
    goto fail;
  }
  // the monitor ring and the list flags behind it
  if (hipHostMalloc((void **)&c->mon_host, sizeof(double) * 4 * MON_STRIDE + sizeof(int) * 8, hipHostMallocMapped) !=
          hipSuccess ||
      hipHostGetDevicePointer((void **)&c->mon_dev, c->mon_host, 0) != hipSuccess) {
    rc = set_err(MDK_ERR_HIP, "mapped host buffer failed");
    goto fail;
  }
  c->flags_host = (int *)(c->mon_host + 4 * MON_STRIDE);
  c->flags_map = (int *)(c->mon_dev + 4 * MON_STRIDE);
  hipMemsetAsync(c->atoms, 0, sizeof(double) * (size_t)F_N * n, c->stream);
  // both buffers start at zero: a re-sort leaves X3..Z3 unmoved while they
  // are zero in both (x3_live false; scratch uses of atoms_alt stay in X0..Z0)
  hipMemsetAsync(c->atoms_alt, 0, sizeof(double) * (size_t)F_N * n, c->stream);
  hipMemsetAsync(c->zat, 0, sizeof(int) * n, c->stream);
  hipMemsetAsync(c->box, 0, sizeof(BoxState) * 4, c->stream);
  hipMemsetAsync(c->ic, 0, sizeof(int) * n, c->stream);
  hipMemsetAsync(c->img, 0, sizeof(int) * 3 * (size_t)n, c->stream);
  hipMemsetAsync(c->numn_ref, 0, sizeof(int) * n, c->stream);
  hipMemsetAsync(c->numn, 0, sizeof(int) * n, c->stream);
  hipMemsetAsync(c->nact, 0, sizeof(int) * n, c->stream);
  k_iota<<<nblocks(n), MDK_BLOCK, 0, c->stream>>>(c->orig, n);
  k_iota<<<nblocks(n), MDK_BLOCK, 0, c->stream>>>(c->slot_of, n);
  memset(c->mon_host, 0, sizeof(double) * 4 * MON_STRIDE);
  memset(c->flags_host, 0, sizeof(int) * 8);
  c->b0_lag_step = -1;
  if (hipStreamSynchronize(c->stream) != hipSuccess) {
    rc = set_err(MDK_ERR_HIP, "init sync failed");
    goto fail;
  }
  *handle = c;
  return MDK_OK;
fail:
  mdk_destroy(c);
  return rc;
#undef ALLOC
}

extern "C" int mdk_destroy(void *h) {
  mdk_ctx *c = H(h);
  if (!c) return MDK_OK;
  if (c->stream) hipStreamSynchronize(c->stream);
  void *ptrs[] = {c->pos4, c->p4f, c->pos4_alt, c->p4f_alt, c->img, c->atoms, c->atoms_alt, c->zat, c->zat_alt, c->orig, c->orig_alt, c->slot_of,
                  c->sref, c->ic, c->numn_ref, c->nlist_ref, c->nbr, c->numn, c->nact, c->cell_of, c->cell_alt, c->ic_alt,
                  c->cell_btot, c->members, c->small, c->nbr16, c->bcnt, c->bstage, c->binfo, c->cell_count,
                  c->cell_start, c->cell_fill, c->tabs, c->trace_dev, c->lblocks, c->fetab,
                  c->ref_key, c->rank_orig, c->rank_slot};
  for (void *q : ptrs)
    if (q) hipFree(q);
  if (c->mon_host) hipHostFree(c->mon_host);
  free(c->h_mass);
  free(c->h_del2);
  free(c->h_z);
  free(c->h_l0);
  free(c->h_link);
  free(c->h_ic);
  for (auto &e : c->evs) {
    hipEventDestroy(e.a);
    hipEventDestroy(e.b);
  }
  for (auto e : c->evpool) hipEventDestroy(e);
  if (c->stream) hipStreamDestroy(c->stream);
  c->evs.~vector();
  c->evpool.~vector();
  ::operator delete(c);
  return MDK_OK;
}

extern "C" int mdk_set_potential(void *h, int nv, const double *av, const double *rv, int np,
                                 const double *ap, const double *rp) {
  mdk_ctx *c = H(h);
  if (!c || nv < 1 || nv > MDK_MAXV || np < 1 || np > MDK_MAXP || !av || !rv || !ap || !rp)
    return set_err(MDK_ERR_BAD_ARG, "bad potential coefficients");
  hostpot::Knots &k = c->knots;
  memset(&k, 0, sizeof(k));
  k.nv = nv;
  k.np = np;
  for (int i = 0; i < nv; i++) { k.av[i] = av[i]; k.rv[i] = rv[i]; }
  for (int i = 0; i < np; i++) { k.ap[i] = ap[i]; k.rp[i] = rp[i]; }
  hostpot::set_up(k);
  PotDev &P = c->pot;
  const int keep_lookup = P.use_lookup, keep_n = P.nlookup;
  const double rint = hostpot::fill_potdev(P, k);
  float fetab[MDK_FE_TAB];
  c->fe_ok = hostpot::build_fe_table(k, fetab, P.fe_binh, P.fe_binc);
  if (c->fe_ok) {
    if (!c->fetab) HIPCK(hipMalloc(&c->fetab, sizeof(fetab)));
    HIPCK(hipMemcpy(c->fetab, fetab, sizeof(fetab), hipMemcpyHostToDevice));
  }
  c->material = MDK_MAT_FETRANSMETAL;
  c->r_int_exact = rint;
  c->r_list = rint + c->skin;
  set_pair_lanes(c);
  c->pot_set = true;
  c->list_valid = false;
  if (keep_lookup) return mdk_set_lookup(h, keep_n > 0 ? keep_n : 5000);
  return MDK_OK;
}

extern "C" int mdk_set_iron_carbon(void *h, const double *iron_in) {
  mdk_ctx *c = H(h);
  if (!c) return set_err(MDK_ERR_BAD_ARG, "null handle");
  if (c->p.precision == MDK_PREC_FP32)
    return set_err(MDK_ERR_BAD_ARG, "the FP32 form is built for the fetransmetal potential");
  PotDev &P = c->pot;
  const int keep_lookup = P.use_lookup, keep_n = P.nlookup;
  hostpot::fec_coef(c->fec, iron_in);
  memset(&c->knots, 0, sizeof(c->knots));
  c->material = MDK_MAT_IRON_CARBON;
  const double rint = hostpot::fill_potdev_fec(P, c->fec);
  c->r_int_exact = rint;
  c->r_list = rint + c->skin;
  set_pair_lanes(c);
  c->pot_set = true;
  c->list_valid = false;
  if (keep_lookup) return mdk_set_lookup(h, keep_n > 0 ? keep_n : 5000);
  return MDK_OK;
}

extern "C" int mdk_set_lookup(void *h, int nlookup) {
  mdk_ctx *c = H(h);
  if (!c || !c->pot_set) return set_err(MDK_ERR_STATE, "set the potential before the lookup tables");
  PotDev &P = c->pot;
  if (nlookup <= 0) {
    P.use_lookup = 0;
    P.r_int = c->r_int_exact;
    c->r_list = P.r_int + c->skin;
    set_pair_lanes(c);
    c->list_valid = false;
    return MDK_OK;
  }
  hostpot::Material mat;
  mat.id = c->material;
  mat.k = c->knots;
  mat.f = c->fec;
  // src/lookup_m.F90:161-251 with the material's range (src/fetransmetal.F90:589-593,
  // src/iron_carbon.F90:93 through get_supported_potential_range) and potential_m's rho range (:185)
  P.nlookup = nlookup;
  P.r_min = 0.0; P.r_max = mat.range();
  P.vp_range = P.r_max - P.r_min;
  P.vp_reciprange = 1.0 / P.vp_range;
  P.vp_recipnlkp = 1.0 / (double)nlookup;
  P.vp_recipstep = (double)nlookup / P.vp_range;
  P.rho_min = 0.0; P.rho_max = 10000.0;
  P.e_range = P.rho_max - P.rho_min;
  P.e_reciprange = 1.0 / P.e_range;
  P.e_recipnlkp = 1.0 / (double)nlookup;
  P.e_recipstep = (double)nlookup / P.e_range;
  const size_t m = (size_t)nlookup + 1;
  std::vector<double> t(6 * m);
  size_t last = 0;  // last node where a pair table is nonzero
  for (size_t i = 0; i < m; i++) {
    double r = P.r_min + (double)i * P.vp_range * P.vp_recipnlkp;
    t[0 * m + i] = mat.vee(r);
    t[1 * m + i] = mat.dvee(r);
    t[2 * m + i] = mat.phi(r);
    t[3 * m + i] = mat.dphi(r);
    if (t[i] != 0.0 || t[m + i] != 0.0 || t[2 * m + i] != 0.0 || t[3 * m + i] != 0.0) last = i;
    double rh = P.rho_min + (double)i * P.e_range * P.e_recipnlkp;
    t[4 * m + i] = mat.emb(rh);
    t[5 * m + i] = mat.demb(rh);
  }
  // interpolation reaches one node beyond the last nonzero one: the list must
  // hold those pairs (two nodes of margin for the rounding of the index)
  P.r_int = std::max(c->r_int_exact, std::min(P.r_max, P.r_min + (double)(last + 2) * P.vp_range * P.vp_recipnlkp));
  c->r_list = P.r_int + c->skin;
  c->list_valid = false;
  if (c->tabs) hipFree(c->tabs);
  HIPCK(hipMalloc(&c->tabs, sizeof(double) * 6 * m));
  HIPCK(hipMemcpy(c->tabs, t.data(), sizeof(double) * 6 * m, hipMemcpyHostToDevice));
  P.tab_v = c->tabs; P.tab_dv = c->tabs + m; P.tab_p = c->tabs + 2 * m;
  P.tab_dp = c->tabs + 3 * m; P.tab_e = c->tabs + 4 * m; P.tab_de = c->tabs + 5 * m;
  P.use_lookup = 1;
  set_pair_lanes(c);
  return MDK_OK;
}

extern "C" int mdk_potential_constants(void *h, double *out) {
  mdk_ctx *c = H(h);
  if (!c || !c->pot_set || !out) return set_err(MDK_ERR_STATE, "potential not set");
  if (c->material != MDK_MAT_FETRANSMETAL) return set_err(MDK_ERR_STATE, "set_up constants belong to fetransmetal");
  out[0] = c->knots.bc1; out[1] = c->knots.bc2;
  for (int i = 0; i < 4; i++) out[2 + i] = c->knots.sc[i];
  out[6] = c->knots.pcr; out[7] = c->knots.pcv;
  return MDK_OK;
}

extern "C" int mdk_eval_potential(void *h, int which, const double *x, double *y, int count) {
  mdk_ctx *c = H(h);
  if (!c || !c->pot_set) return set_err(MDK_ERR_STATE, "potential not set");
  if (which < 0 || which > 8 || count < 0 || (count > 0 && (!x || !y))) return set_err(MDK_ERR_BAD_ARG, "bad eval args");
  if (which >= 6 && (!c->fe_ok || c->material != MDK_MAT_FETRANSMETAL))
    return set_err(MDK_ERR_BAD_ARG, "no FP32 interval table for this potential");
  if (count == 0) return MDK_OK;
  double *d = nullptr;
  HIPCK(hipMalloc(&d, sizeof(double) * 2 * (size_t)count));
  HIPCK(hipMemcpyAsync(d, x, sizeof(double) * count, hipMemcpyHostToDevice, c->stream));
  k_eval_pot<<<nblocks(count), MDK_BLOCK, 0, c->stream>>>(c->pot, which, d, d + count, count, c->fetab);
  int rc = check_launch("k_eval_pot");
  hipMemcpyAsync(y, d + count, sizeof(double) * count, hipMemcpyDeviceToHost, c->stream);
  hipStreamSynchronize(c->stream);
  hipFree(d);
  return rc;
}

extern "C" int mdk_energy_calc(void *h, double *en_atom) {
  mdk_ctx *c = H(h);
  if (!c || !en_atom) return set_err(MDK_ERR_BAD_ARG, "bad energy_calc arguments");
  if (!c->pot_set || !c->list_valid)
    return set_err(MDK_ERR_STATE, "energy_calc needs the neighbour list and densities of a force evaluation");
  const int n = c->n;
  RCK(ensure_pos4(c));
  RCK(ensure_wide_list(c));
  double *en = fld(c->atoms_alt, 1, n), *out = fld(c->atoms_alt, 0, n);
  const dim3 g(nblocks(n)), b(MDK_BLOCK);
  const BoxState *bs = c->box + c->cur;
  if (c->material == MDK_MAT_IRON_CARBON)
    k_energy_calc<POT_FEC><<<g, b, 0, c->stream>>>(c->atoms, c->pos4, n, c->nbr, c->numn, bs, pack_geo(c), c->pot, en);
  else if (c->pot.nv == MDK_FE_NV && c->pot.np == MDK_FE_NP)
    k_energy_calc<POT_FE><<<g, b, 0, c->stream>>>(c->atoms, c->pos4, n, c->nbr, c->numn, bs, pack_geo(c), c->pot, en);
  else
    k_energy_calc<POT_KNOTS><<<g, b, 0, c->stream>>>(c->atoms, c->pos4, n, c->nbr, c->numn, bs, pack_geo(c), c->pot, en);
  RCK(check_launch("k_energy_calc"));
  k_gather_d<<<nblocks(n), MDK_BLOCK, 0, c->stream>>>(out, en, c->slot_of, n);
  RCK(check_launch("k_gather_d"));
  HIPCK(hipMemcpyAsync(en_atom, out, sizeof(double) * n, hipMemcpyDeviceToHost, c->stream));
  HIPCK(hipStreamSynchronize(c->stream));
  return MDK_OK;
}

extern "C" int mdk_atomic_stress(void *h, double *sx, double *sy, double *sz) {
  mdk_ctx *c = H(h);
  if (!c || !sx || !sy || !sz) return set_err(MDK_ERR_BAD_ARG, "bad atomic_stress arguments");
  if (!c->pot_set || !c->half_valid)
    return set_err(MDK_ERR_STATE, "atomic_stress needs the reference half list and densities of a force evaluation");
  const int n = c->n;
  double *o = fld(c->atoms_alt, 0, n);  // three scratch columns
  const dim3 g(nblocks(n)), b(MDK_BLOCK);
  const BoxState *bs = c->box + c->cur;
#define MDK_STRESS_ARGS c->atoms, c->slot_of, n, c->numn_ref, c->nlist_ref, c->p.nnbrs, bs, c->pbc, c->pot, o, o + n, o + 2 * (size_t)n
  if (c->pot.use_lookup)
    k_atomic_stress<POT_TABLE><<<g, b, 0, c->stream>>>(MDK_STRESS_ARGS);
  else if (c->material == MDK_MAT_IRON_CARBON)
    k_atomic_stress<POT_FEC><<<g, b, 0, c->stream>>>(MDK_STRESS_ARGS);
  else if (c->pot.nv == MDK_FE_NV && c->pot.np == MDK_FE_NP)
    k_atomic_stress<POT_FE><<<g, b, 0, c->stream>>>(MDK_STRESS_ARGS);
  else
    k_atomic_stress<POT_KNOTS><<<g, b, 0, c->stream>>>(MDK_STRESS_ARGS);
#undef MDK_STRESS_ARGS
  RCK(check_launch("k_atomic_stress"));
  HIPCK(hipMemcpyAsync(sx, o, sizeof(double) * n, hipMemcpyDeviceToHost, c->stream));
  HIPCK(hipMemcpyAsync(sy, o + n, sizeof(double) * n, hipMemcpyDeviceToHost, c->stream));
  HIPCK(hipMemcpyAsync(sz, o + 2 * (size_t)n, sizeof(double) * n, hipMemcpyDeviceToHost, c->stream));
  HIPCK(hipStreamSynchronize(c->stream));
  return MDK_OK;
}

static const int field_map[MDK_NFIELDS] = {F_X0,  F_Y0,  F_Z0,   F_X1,     F_Y1,      F_Z1,   F_X2,
                                           F_Y2,  F_Z2,  F_FX,   F_FY,     F_FZ,      F_RHO,  F_AFRHO,
                                           F_DAFRHO, F_MASS, F_DEL2, F_X3, F_Y3, F_Z3};

// Species table of (mass, del2) when both are functions of the species.
static int keep_host_copy(double **dst, const double *src, int n) {
  if (!*dst) *dst = (double *)malloc(sizeof(double) * n);
  if (!*dst) return set_err(MDK_ERR_HIP, "host copy failed");
  memcpy(*dst, src, sizeof(double) * n);
  return MDK_OK;
}
static int update_species_table(mdk_ctx *c) {
  c->spec_ok = false;
  if (!c->h_mass || !c->h_del2 || !c->h_z) return MDK_OK;
  double tab[2 * MDK_NSPEC];
  bool seen[MDK_NSPEC] = {};
  for (int i = 0; i < c->n; i++) {
    const int z = c->h_z[i];
    if (z < 0 || z >= MDK_NSPEC) return MDK_OK;
    if (!seen[z]) {
      seen[z] = true;
      tab[2 * z] = c->h_mass[i];
      tab[2 * z + 1] = c->h_del2[i];
    } else if (memcmp(&tab[2 * z], &c->h_mass[i], sizeof(double)) != 0 ||
               memcmp(&tab[2 * z + 1], &c->h_del2[i], sizeof(double)) != 0) {
      return MDK_OK;  // per-atom values differ within a species
    }
  }
  for (int z = 0; z < MDK_NSPEC; z++)
    if (!seen[z]) tab[2 * z] = tab[2 * z + 1] = 0.0;
  HIPCK(hipMemcpy(c->spec_tab, tab, sizeof(tab), hipMemcpyHostToDevice));
  c->spec_ok = true;
  return MDK_OK;
}
extern "C" int mdk_upload(void *h, int field, const double *data) {
  mdk_ctx *c = H(h);
  if (!c || field < 0 || field >= MDK_NFIELDS || !data) return set_err(MDK_ERR_BAD_ARG, "bad upload");
  c->kin_fresh = false;  // velocities, masses or box may change: kinten's sums are recomputed
  const int n = c->n;
  double *tmp = fld(c->atoms_alt, 0, n);  // staging in the alternate buffer
  HIPCK(hipMemcpyAsync(tmp, data, sizeof(double) * n, hipMemcpyHostToDevice, c->stream));
  k_scatter_d<<<nblocks(n), MDK_BLOCK, 0, c->stream>>>(fld(c->atoms, field_map[field], n), tmp, c->slot_of, n);
  RCK(check_launch("k_scatter_d"));
  HIPCK(hipStreamSynchronize(c->stream));
  if (field <= MDK_Z0) {  // positions replaced: rebuild (from the exact box) before the next force
    c->list_valid = false;
    c->b0_lag_step = -1;
  }
  if (field <= MDK_Z0 || field == MDK_DAFRHO) c->pos4_valid = c->p4f_valid = false;
  if (field == MDK_X3 || field == MDK_Y3 || field == MDK_Z3) c->x3_live = true;
  if (field == MDK_MASS) {
    // the per-pair test m_i + m_j > 0.1 (REAL(4) literal) can only fail with a mass <= 0.05
    bool any = false;
    for (int i = 0; i < n; i++) any = any || !(data[i] > 0.05);
    c->masschk = any;
    if (c->brick && !lean_pot(c)) {  // the general passes take over this list
      RCK(ensure_wide_list(c));
      c->brick = false;
      c->nbp = nblocks((long)n * c->lanes);
    }
  }
  if (field == MDK_MASS || field == MDK_DEL2) {
    RCK(keep_host_copy(field == MDK_MASS ? &c->h_mass : &c->h_del2, data, n));
    RCK(update_species_table(c));
  }
  return MDK_OK;
}

extern "C" int mdk_download(void *h, int field, double *data) {
  mdk_ctx *c = H(h);
  if (!c || field < 0 || field >= MDK_NFIELDS || !data) return set_err(MDK_ERR_BAD_ARG, "bad download");
  const int n = c->n;
  double *tmp = fld(c->atoms_alt, 0, n);
  k_gather_d<<<nblocks(n), MDK_BLOCK, 0, c->stream>>>(tmp, fld(c->atoms, field_map[field], n), c->slot_of, n);
  RCK(check_launch("k_gather_d"));
  HIPCK(hipMemcpyAsync(data, tmp, sizeof(double) * n, hipMemcpyDeviceToHost, c->stream));
  HIPCK(hipStreamSynchronize(c->stream));
  return MDK_OK;
}

extern "C" int mdk_upload_species(void *h, const int *zn) {
  mdk_ctx *c = H(h);
  if (!c || !zn) return set_err(MDK_ERR_BAD_ARG, "bad species upload");
  c->kin_fresh = false;  // velocities, masses or box may change: kinten's sums are recomputed
  const int n = c->n;
  // the pair kernels evaluate the Fe-Fe functions: Fe atoms and vacancies only
  for (int i = 0; i < n; i++)
    if (zn[i] != 26 && zn[i] != 0) return set_err(MDK_ERR_BAD_ARG, "only Fe (Z=26) and vacancies (Z=0) are supported");
  HIPCK(hipMemcpyAsync(c->zat_alt, zn, sizeof(int) * n, hipMemcpyHostToDevice, c->stream));
  k_scatter_i<<<nblocks(n), MDK_BLOCK, 0, c->stream>>>(c->zat, c->zat_alt, c->slot_of, n);
  RCK(check_launch("k_scatter_i"));
  HIPCK(hipStreamSynchronize(c->stream));
  if (!c->h_z) c->h_z = (int *)malloc(sizeof(int) * n);
  if (!c->h_z) return set_err(MDK_ERR_HIP, "host copy failed");
  memcpy(c->h_z, zn, sizeof(int) * n);
  return update_species_table(c);
}

static double *box_field(BoxState &s, int which) {
  switch (which) {
    case MDK_B0: return s.b0;
    case MDK_B1: return s.b1;
    case MDK_B2: return s.b2;
    case MDK_TK: return s.tk;
    case MDK_TC: return s.tc;
    case MDK_TG: return s.tg;
    case MDK_TP: return s.tp;
    case MDK_TGINV: return s.tginv;
    case MDK_TGDOT: return s.tgdot;
    case MDK_TGID: return s.tgid;
    case MDK_FB: return s.fb;
    case MDK_B3: return s.b3;
    default: return nullptr;
  }
}

extern "C" int mdk_set_tensor(void *h, int which, const double *t9) {
  mdk_ctx *c = H(h);
  if (!c || !t9 || which < 0 || which >= MDK_NTENSORS) return set_err(MDK_ERR_BAD_ARG, "bad tensor");
  c->kin_fresh = false;  // velocities, masses or box may change: kinten's sums are recomputed
  BoxState s;
  RCK(read_box(c, &s));
  memcpy(box_field(s, which), t9, 9 * sizeof(double));
  if (which == MDK_B0) {
    const double *b = s.b0;
    s.vol = TT(b, 1, 1) * (TT(b, 2, 2) * TT(b, 3, 3) - TT(b, 2, 3) * TT(b, 3, 2)) +
            TT(b, 2, 1) * (TT(b, 3, 2) * TT(b, 1, 3) - TT(b, 1, 2) * TT(b, 3, 3)) +
            TT(b, 3, 1) * (TT(b, 1, 2) * TT(b, 2, 3) - TT(b, 2, 2) * TT(b, 1, 3));
    c->list_valid = false;
    c->pos4_valid = c->p4f_valid = false;
    c->b0_lag_step = -1;  // the next list is planned from this box, not a lagged one
  }
  HIPCK(hipMemcpyAsync(c->box + c->cur, &s, sizeof(s), hipMemcpyHostToDevice, c->stream));
  HIPCK(hipStreamSynchronize(c->stream));
  return MDK_OK;
}

extern "C" int mdk_get_tensor(void *h, int which, double *t9) {
  mdk_ctx *c = H(h);
  if (!c || !t9 || which < 0 || which >= MDK_NTENSORS) return set_err(MDK_ERR_BAD_ARG, "bad tensor");
  BoxState s;
  RCK(read_box(c, &s));
  memcpy(t9, box_field(s, which), 9 * sizeof(double));
  return MDK_OK;
}

extern "C" int mdk_get_scalars(void *h, double *out) {
  mdk_ctx *c = H(h);
  if (!c || !out) return set_err(MDK_ERR_BAD_ARG, "bad scalars");
  BoxState s;
  RCK(read_box(c, &s));
  out[MDK_S_PE] = s.pe; out[MDK_S_KE] = s.ke; out[MDK_S_VOL] = s.vol;
  out[MDK_S_S1] = s.s1; out[MDK_S_S2] = s.s2; out[MDK_S_S3] = s.s3;
  out[MDK_S_TE] = s.te; out[MDK_S_H] = s.h; out[MDK_S_TH] = s.th; out[MDK_S_BOXKE] = s.boxke;
  out[MDK_S_MAXDISP] = sqrt(fmax(s.maxdisp2, 0.0));
  return MDK_OK;
}

extern "C" int mdk_set_ntc(void *h, int ntc) {
  mdk_ctx *c = H(h);
  if (!c) return set_err(MDK_ERR_BAD_ARG, "null handle");
  c->ntc = ntc;
  return MDK_OK;
}
extern "C" int mdk_get_ntc(void *h, int *ntc) {
  mdk_ctx *c = H(h);
  if (!c || !ntc) return set_err(MDK_ERR_BAD_ARG, "null handle");
  *ntc = c->ntc;
  return MDK_OK;
}

// Reference cells of every atom in reference order (host), from the device ic.
static int ic_to_host(mdk_ctx *c, int *ico) {
  const int n = c->n;
  k_gather_i<<<nblocks(n), MDK_BLOCK, 0, c->stream>>>(c->ref_key, c->ic, c->slot_of, n);
  RCK(check_launch("k_gather_i"));
  HIPCK(hipMemcpyAsync(ico, c->ref_key, sizeof(int) * n, hipMemcpyDeviceToHost, c->stream));
  HIPCK(hipStreamSynchronize(c->stream));
  return MDK_OK;
}

static int chains_reserve(mdk_ctx *c) {
  const int m = c->p.nlcx * c->p.nlcy * c->p.nlcz;
  if (c->h_l0 && c->h_ncell == m) return MDK_OK;
  free(c->h_l0);
  c->h_l0 = (int *)calloc((size_t)m + 1, sizeof(int));
  if (!c->h_link) c->h_link = (int *)calloc((size_t)c->n + 1, sizeof(int));
  if (!c->h_ic) c->h_ic = (int *)calloc((size_t)c->n + 1, sizeof(int));
  if (!c->h_l0 || !c->h_link || !c->h_ic) return set_err(MDK_ERR_STATE, "out of host memory for the link-cell chains");
  c->h_ncell = m;
  return MDK_OK;
}

// linkup's chains (src/linkcell_m.F90:140-182): each cell's atoms in
// ascending order, the last linked back to the first
static void chains_linkup(mdk_ctx *c, const int *ico) {
  const int n = c->n, m = c->h_ncell;
  int *l0 = c->h_l0, *link = c->h_link;
  std::vector<int> last(m + 1, 0);
  for (int k = 0; k <= m; k++) l0[k] = 0;
  for (int i = 1; i <= n; i++) {
    const int ip = ico[i - 1];
    c->h_ic[i] = ip;
    if (last[ip]) link[last[ip]] = i; else l0[ip] = i;
    last[ip] = i;
  }
  for (int ip = 1; ip <= m; ip++)
    if (last[ip]) link[last[ip]] = l0[ip];
}

// relink's chain surgery (src/linkcell_m.F90:224-271), atoms in reference
// order: an atom whose cell changed leaves its old chain (the atom after it
// becomes that cell's starter) and enters its new cell right after the
// starter, becoming the starter itself.
static int chains_relink(mdk_ctx *c, const int *ico) {
  int *l0 = c->h_l0, *link = c->h_link, *icr = c->h_ic;
  for (int i = 1; i <= c->n; i++) {
    const int ip = ico[i - 1];
    if (ip == icr[i]) continue;
    const int me = icr[i];
    int j = l0[me], hops = 0;
    while (j > 0 && link[j] != i && hops++ < c->n) j = link[j];
    if (j <= 0 || link[j] != i) return set_err(MDK_ERR_STATE, "link-cell chains inconsistent at atom %d", i);
    link[j] = link[i];
    l0[me] = link[j];
    if (i == j) l0[me] = 0;
    j = l0[ip] == 0 ? i : l0[ip];
    link[i] = link[j];
    link[j] = i;
    icr[i] = ip;
    l0[ip] = i;
  }
  return MDK_OK;
}

// each atom's position in its cell's chain from L0, uploaded in reference order
static int chains_rank(mdk_ctx *c) {
  std::vector<int> rank(c->n, 0);
  for (int ip = 1; ip <= c->h_ncell; ip++) {
    const int s0 = c->h_l0[ip];
    if (!s0) continue;
    int i = s0, r = 0;
    do {
      rank[i - 1] = r++;
      i = c->h_link[i];
    } while (i != s0 && r <= c->n);
  }
  HIPCK(hipMemcpyAsync(c->rank_orig, rank.data(), sizeof(int) * c->n, hipMemcpyHostToDevice, c->stream));
  HIPCK(hipStreamSynchronize(c->stream));
  return MDK_OK;
}

static int launch_ref_cells(mdk_ctx *c) {
  const int n = c->n;
  k_ref_cells<<<nblocks(n), MDK_BLOCK, 0, c->stream>>>(c->atoms, c->atoms + n, c->atoms + 2 * (size_t)n, n,
                                                      link_grid(c, true));
  return check_launch("k_ref_cells");
}

extern "C" int mdk_linkup(void *h) {
  mdk_ctx *c = H(h);
  if (!c) return set_err(MDK_ERR_BAD_ARG, "null handle");
  RCK(launch_ref_cells(c));
  RCK(chains_reserve(c));
  std::vector<int> ico(c->n);
  RCK(ic_to_host(c, ico.data()));
  chains_linkup(c, ico.data());
  RCK(chains_rank(c));
  c->linked = true;
  c->chains_exact = true;
  return MDK_OK;
}

extern "C" int mdk_relink(void *h) {
  mdk_ctx *c = H(h);
  if (!c) return set_err(MDK_ERR_BAD_ARG, "null handle");
  if (!c->linked || !c->chains_exact) return mdk_linkup(h);
  RCK(launch_ref_cells(c));
  std::vector<int> ico(c->n);
  RCK(ic_to_host(c, ico.data()));
  RCK(chains_relink(c, ico.data()));
  return chains_rank(c);
}

// The relink at the wrap of ntc inside mdk_md_steps: the device ic only (no
// host round trip in the loop).  The chain order it would give is not
// tracked; the next chain query or half list starts from linkup's chains.
static int relink_in_loop(mdk_ctx *c) {
  RCK(launch_ref_cells(c));
  c->chains_exact = false;
  return MDK_OK;
}

extern "C" int mdk_get_linkcells(void *h, int *l0, int *link, int *ic) {
  mdk_ctx *c = H(h);
  if (!c) return set_err(MDK_ERR_BAD_ARG, "null handle");
  if (!c->linked) return set_err(MDK_ERR_STATE, "link cells not set (call linkup)");
  if (!c->chains_exact) RCK(mdk_linkup(h));
  if (ic) memcpy(ic, c->h_ic + 1, sizeof(int) * c->n);
  if (l0) memcpy(l0, c->h_l0 + 1, sizeof(int) * c->h_ncell);
  if (link) memcpy(link, c->h_link + 1, sizeof(int) * c->n);
  return MDK_OK;
}

extern "C" int mdk_update_neighbourlist(void *h) {
  mdk_ctx *c = H(h);
  if (!c) return set_err(MDK_ERR_BAD_ARG, "null handle");
  if (!c->linked || !c->chains_exact) RCK(mdk_linkup(h));
  const int n = c->n, m = c->p.nlcx * c->p.nlcy * c->p.nlcz;
  // bin by reference cell (0-based key), in-cell order by chain rank; the
  // device list's own cell keys (cell_of) are left alone
  k_minus1<<<nblocks(n), MDK_BLOCK, 0, c->stream>>>(c->ic, c->ref_key, n);
  k_gather_i<<<nblocks(n), MDK_BLOCK, 0, c->stream>>>(c->rank_slot, c->rank_orig, c->orig, n);
  RCK(check_launch("k_gather_i"));
  RCK(bin_atoms(c, c->ref_key, m, c->rank_slot));
  HIPCK(hipMemsetAsync(c->dflags, 0, sizeof(int) * 4, c->stream));
  k_half_list<<<nblocks(n), MDK_BLOCK, 0, c->stream>>>(
      c->atoms, c->atoms + n, c->atoms + 2 * (size_t)n, c->ic, c->orig, c->rank_slot, c->cell_start, c->members, n,
      c->p.nlcx, c->p.nlcy, c->p.nlcz, c->box + c->cur, c->rnear2_exact, c->pbc, c->p.nnbrs,
      c->numn_ref, c->nlist_ref, c->dflags);
  RCK(check_launch("k_half_list"));
  int fl[4];
  HIPCK(hipMemcpyAsync(fl, c->dflags, sizeof(fl), hipMemcpyDeviceToHost, c->stream));
  HIPCK(hipStreamSynchronize(c->stream));
  if (fl[1]) return set_err(MDK_ERR_NBR_OVERFLOW, "NEIGHBOURLIST: EXCESS NEIGHBOURS! (nnbrs=%d)", c->p.nnbrs);
  c->half_valid = true;
  return MDK_OK;
}

extern "C" int mdk_get_neighbourlist(void *h, int *numn, int *nlist) {
  mdk_ctx *c = H(h);
  if (!c) return set_err(MDK_ERR_BAD_ARG, "null handle");
  if (numn) HIPCK(hipMemcpy(numn, c->numn_ref, sizeof(int) * c->n, hipMemcpyDeviceToHost));
  if (nlist) HIPCK(hipMemcpy(nlist, c->nlist_ref, sizeof(int) * (size_t)c->n * c->p.nnbrs, hipMemcpyDeviceToHost));
  return MDK_OK;
}

extern "C" int mdk_get_pairs(void *h, long *count, int *pi, int *pj, long cap) {
  mdk_ctx *c = H(h);
  if (!c || !count) return set_err(MDK_ERR_BAD_ARG, "null argument");
  const int n = c->n, nn = c->p.nnbrs;
  std::vector<int> numn(n), nl((size_t)n * nn);
  RCK(mdk_get_neighbourlist(h, numn.data(), nl.data()));
  long k = 0;
  for (int i = 0; i < n; i++)
    for (int q = 0; q < std::min(numn[i], nn); q++) {
      if (pi && pj && k < cap) {
        pi[k] = i;
        pj[k] = nl[(size_t)i * nn + q] - 1;
      }
      k++;
    }
  *count = k;
  return MDK_OK;
}

extern "C" int mdk_force(void *h) {
  mdk_ctx *c = H(h);
  if (!c) return set_err(MDK_ERR_BAD_ARG, "null handle");
  RCK(force_and_finish(c, FIN_FORCE, false));
  HIPCK(hipStreamSynchronize(c->stream));
  return check_device_status(c);
}

extern "C" int mdk_rhoset(void *h) {
  mdk_ctx *c = H(h);
  if (!c || !c->pot_set) return set_err(MDK_ERR_STATE, "potential not set");
  if (!c->list_valid) RCK(rebuild_full(c));
  RCK(launch_density(c, 0));
  HIPCK(hipStreamSynchronize(c->stream));
  return MDK_OK;
}

extern "C" int mdk_embed(void *h, double *pe_embed) {
  mdk_ctx *c = H(h);
  if (!c || !c->pot_set) return set_err(MDK_ERR_STATE, "potential not set");
  if (!c->list_valid) RCK(rebuild_full(c));
  RCK(launch_density(c, 1));
  if (pe_embed) {
    const int nb = c->emb_nb;
    std::vector<double> part(nb);
    HIPCK(hipMemcpyAsync(part.data(), emb_buf(c, c->emb_slot), sizeof(double) * nb, hipMemcpyDeviceToHost, c->stream));
    HIPCK(hipStreamSynchronize(c->stream));
    double s = 0.0;
    for (double v : part) s += v;
    *pe_embed = s;
  }
  HIPCK(hipStreamSynchronize(c->stream));
  return MDK_OK;
}

extern "C" int mdk_kinten(void *h) { return mdk_force(h); }

extern "C" int mdk_md_init(void *h) {
  mdk_ctx *c = H(h);
  if (!c) return set_err(MDK_ERR_BAD_ARG, "null handle");
  RCK(force_and_finish(c, FIN_INIT, false));
  RCK(launch_kick(c, 2, nullptr, nullptr));
  HIPCK(hipStreamSynchronize(c->stream));
  return check_device_status(c);
}

extern "C" int mdk_velocityverlet(void *h) {
  mdk_ctx *c = H(h);
  if (!c) return set_err(MDK_ERR_BAD_ARG, "null handle");
  bool skin_due;
  RCK(skin_check(c, &skin_due));
  c->pc_primed = true;
  RCK(launch_drift(c));
  RCK(force_and_finish(c, FIN_VV, skin_due));
  // half kick without the thermodynamic sums' box part (tgid stays lagged)
  int slot = (int)(c->step_counter & 3);
  RCK(launch_kick(c, 0, nullptr, c->mon_dev + MON_STRIDE * slot));
  c->step_counter++;
  HIPCK(hipStreamSynchronize(c->stream));
  const double *m = c->mon_host + MON_STRIDE * slot;  // this step's sample
  if (skin_used(c, m) >= 0.5 * c->skin) return skin_violation(c, m, c->step_counter - 1);
  return check_device_status(c);
}

extern "C" int mdk_scalev(void *h, double nose, double rqke) {
  mdk_ctx *c = H(h);
  if (!c) return set_err(MDK_ERR_BAD_ARG, "null handle");
  c->kin_fresh = false;  // velocities, masses or box may change: kinten's sums are recomputed
  if (!(nose > 0.0)) return MDK_OK;  // only a positive nose acts (src/thermostat_m.F90:329)
  const int n = c->n, nb = nblocks(n);
  if (nb > c->nblk) return set_err(MDK_ERR_STATE, "partial buffers too small");
  const unsigned fb = (unsigned)((nb + 63) / 64);
  k_vsum<<<nb, MDK_BLOCK, 0, c->stream>>>(c->atoms, n, c->part_k);
  RCK(check_launch("k_vsum"));
  k_fold<3><<<fb, MDK_FIN_BLOCK, 0, c->stream>>>(c->part_k, nb, c->stage_k, c->fin_cnt + 1, c->red);
  RCK(check_launch("k_fold"));
  // mean over all atoms: sx / float(nm), a REAL(4) conversion of nm
  double s3[4];
  HIPCK(hipMemcpyAsync(s3, c->red, sizeof(double) * 3, hipMemcpyDeviceToHost, c->stream));
  HIPCK(hipStreamSynchronize(c->stream));
  const double fn = (double)(float)n;
  const double mean[3] = {s3[0] / fn, s3[1] / fn, s3[2] / fn};
  HIPCK(hipMemcpyAsync(c->red, mean, sizeof(mean), hipMemcpyHostToDevice, c->stream));
  k_vsub_ke<<<nb, MDK_BLOCK, 0, c->stream>>>(c->atoms, c->zat, n, c->red, c->box + c->cur, spec_of(c), c->part_k);
  RCK(check_launch("k_vsub_ke"));
  k_fold<1><<<fb, MDK_FIN_BLOCK, 0, c->stream>>>(c->part_k, nb, c->stage_k, c->fin_cnt + 1, c->red + 3);
  RCK(check_launch("k_fold"));
  HIPCK(hipMemcpyAsync(s3 + 3, c->red + 3, sizeof(double), hipMemcpyDeviceToHost, c->stream));
  HIPCK(hipStreamSynchronize(c->stream));
  const double ke = s3[3] / (c->p.deltat * c->p.deltat) / 2.0;
  double snhf = 0.0;
  if (ke > 0.0) snhf = (ke - rqke) / (nose * (double)n);
  c->snhv = c->snhv - snhf;
  k_vscale<<<nb, MDK_BLOCK, 0, c->stream>>>(c->atoms, c->zat, n, spec_of(c), 1.0 + c->snhv);
  RCK(check_launch("k_vscale"));
  HIPCK(hipStreamSynchronize(c->stream));
  return MDK_OK;
}

extern "C" int mdk_get_snhv(void *h, double *v) {
  mdk_ctx *c = H(h);
  if (!c || !v) return set_err(MDK_ERR_BAD_ARG, "bad snhv arguments");
  *v = c->snhv;
  return MDK_OK;
}

extern "C" int mdk_set_snhv(void *h, double v) {
  mdk_ctx *c = H(h);
  if (!c) return set_err(MDK_ERR_BAD_ARG, "null handle");
  c->snhv = v;
  return MDK_OK;
}

extern "C" int mdk_set_pressure(void *h, double press) {
  mdk_ctx *c = H(h);
  if (!c) return set_err(MDK_ERR_BAD_ARG, "null handle");
  c->p.press = press;
  return MDK_OK;
}

extern "C" int mdk_set_integrator(void *h, int iverlet) {
  mdk_ctx *c = H(h);
  if (!c || (iverlet != 0 && iverlet != 1)) return set_err(MDK_ERR_BAD_ARG, "iverlet must be 0 or 1");
  c->iverlet = iverlet;
  return MDK_OK;
}

extern "C" int mdk_predic(void *h) {
  mdk_ctx *c = H(h);
  if (!c) return set_err(MDK_ERR_BAD_ARG, "null handle");
  RCK(launch_predic(c));
  HIPCK(hipStreamSynchronize(c->stream));
  return MDK_OK;
}

extern "C" int mdk_correc(void *h) {
  mdk_ctx *c = H(h);
  if (!c) return set_err(MDK_ERR_BAD_ARG, "null handle");
  c->kin_fresh = false;  // velocities, masses or box may change: kinten's sums are recomputed
  RCK(launch_correc(c));
  HIPCK(hipStreamSynchronize(c->stream));
  return MDK_OK;
}

extern "C" int mdk_update_therm_avs(void *h, double *s1, double *s2, double *s3) {
  mdk_ctx *c = H(h);
  if (!c) return set_err(MDK_ERR_BAD_ARG, "null handle");
  k_therm_box<<<1, 64, 0, c->stream>>>(c->box + c->cur, c->p.ivol);
  RCK(check_launch("k_therm_box"));
  TimedEv te;
  tbegin(c, TC_KICK, te);
  k_kick<false><<<c->nblk, MDK_BLOCK, 0, c->stream>>>(
      c->atoms, c->zat, c->n, c->box + c->cur, c->p.ivol, 1, nullptr, c->part_k, nullptr, nullptr, nullptr,
      nullptr, pack_geo(c), nullptr, spec_of(c), nullptr, link_grid(c, false));
  tend(c, te);
  RCK(check_launch("k_kick"));
  const FinKick F = {c->box + c->cur, nullptr, nullptr, nullptr, c->p.deltat, c->p.bdel2, c->p.press, 0.0};
  k_finish_step<<<1, FINISH_THREADS, 0, c->stream>>>(FinRide{1, c->nblk, 0, c->part_k, nullptr, F});
  RCK(check_launch("k_finish_step"));
  BoxState s;
  RCK(read_box(c, &s));
  if (s1) *s1 = s.s1;
  if (s2) *s2 = s.s2;
  if (s3) *s3 = s.s3;
  if (s.status) return set_err(s.status, "singular box matrix in matrix_invert");
  return MDK_OK;
}

extern "C" int mdk_md_steps(void *h, int nsteps, double *trace) {
  mdk_ctx *c = H(h);
  if (!c || nsteps < 0) return set_err(MDK_ERR_BAD_ARG, "bad md_steps arguments");
  if (trace && nsteps > c->trace_cap) {
    if (c->trace_dev) hipFree(c->trace_dev);
    HIPCK(hipMalloc(&c->trace_dev, sizeof(double) * 6 * (size_t)nsteps));
    c->trace_cap = nsteps;
  }
  int rc = MDK_OK;
  for (int s = 0; s < nsteps && rc == MDK_OK; s++) {
    rc = md_step(c, trace ? c->trace_dev + 6 * (size_t)s : nullptr, nsteps - s - 1);
    // relink when the reference's ntc counter wraps (moldin.F90:791)
    if (rc == MDK_OK && c->ntc == 0 && !c->drifted) rc = relink_in_loop(c);
  }
  // the list is still the one of a fused last step if that step's sums are pending
  // and no rebuild has begun
  const bool fused = c->ride.kind == 2 && c->list_valid && !c->list_pending;
  const int rf = flush_ride(c);  // the last step's sums (also after a failed step)
  if (rc != MDK_OK) {
    if (fused) {
      char msg[sizeof(g_err)];
      memcpy(msg, g_err, sizeof(msg));
      if (last_forces(c) == MDK_OK) hipStreamSynchronize(c->stream);
      set_err(rc, "%s", msg);
    }
    return rc;
  }
  RCK(rf);
  if (trace && nsteps > 0)
    HIPCK(hipMemcpyAsync(trace, c->trace_dev, sizeof(double) * 6 * (size_t)nsteps, hipMemcpyDeviceToHost, c->stream));
  HIPCK(hipStreamSynchronize(c->stream));
  // the samples of the last three steps, not yet polled
  for (long st = std::max(c->step_counter - 3, c->step_counter - nsteps); st < c->step_counter; st++) {
    const double *m = c->mon_host + MON_STRIDE * (int)(st & 3);
    if (skin_used(c, m) >= 0.5 * c->skin) return skin_violation(c, m, st);
  }
  return check_device_status(c);
}

extern "C" int mdk_stats(void *h, long *rebuilds, long *full_pairs) {
  mdk_ctx *c = H(h);
  if (!c) return set_err(MDK_ERR_BAD_ARG, "null handle");
  if (rebuilds) *rebuilds = c->rebuilds;
  if (full_pairs) {
    RCK(ensure_wide_list(c));
    HIPCK(hipStreamSynchronize(c->stream));
    std::vector<int> nn(c->n);
    HIPCK(hipMemcpy(nn.data(), c->numn, sizeof(int) * c->n, hipMemcpyDeviceToHost));
    long s = 0;
    for (int v : nn) s += v;
    *full_pairs = s;
  }
  return MDK_OK;
}

extern "C" int mdk_timing(void *h, int mask) {
  mdk_ctx *c = H(h);
  if (!c) return set_err(MDK_ERR_BAD_ARG, "null handle");
  c->timing_mask = mask & ((1 << TC_NCLASS) - 1);
  for (int k = 0; k < TC_NCLASS; k++) c->t_seen[k] = 0;
  if (c->timing_mask) {
    for (int k = 0; k < TC_NCLASS; k++) { c->t_ms[k] = 0.0; c->t_cnt[k] = 0; }
    hipStreamSynchronize(c->stream);
    for (auto &e : c->evs) { c->evpool.push_back(e.a); c->evpool.push_back(e.b); }
    c->evs.clear();
  }
  return MDK_OK;
}

extern "C" int mdk_timing_every(void *h, int every) {
  mdk_ctx *c = H(h);
  if (!c || every < 1) return set_err(MDK_ERR_BAD_ARG, "bad timing stride");
  c->timing_every = every;
  return MDK_OK;
}

extern "C" int mdk_timing_read(void *h, double *ms, long *launches, int nclasses) {
  mdk_ctx *c = H(h);
  if (!c) return set_err(MDK_ERR_BAD_ARG, "null handle");
  HIPCK(hipStreamSynchronize(c->stream));
  for (auto &e : c->evs) {
    float t = 0.f;
    hipEventElapsedTime(&t, e.a, e.b);
    c->t_ms[e.cls] += t;
    c->t_cnt[e.cls] += 1;
    c->evpool.push_back(e.a);
    c->evpool.push_back(e.b);
  }
  c->evs.clear();
  for (int k = 0; k < nclasses && k < TC_NCLASS; k++) {
    if (ms) ms[k] = c->t_ms[k];
    if (launches) launches[k] = c->t_cnt[k];
  }
  return MDK_OK;
}

extern "C" int mdk_synchronize(void *h) {
  mdk_ctx *c = H(h);
  if (!c) return set_err(MDK_ERR_BAD_ARG, "null handle");
  HIPCK(hipStreamSynchronize(c->stream));
  return MDK_OK;
}
