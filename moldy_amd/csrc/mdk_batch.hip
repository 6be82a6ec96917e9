// mdk_batch.hip -- many independent periodic Fe cells evaluated together.
//
// Energies, forces and the 3x3 stress of thousands of cells of uneven atom
// counts (the force() evaluation of src/dynamics_m.F90:135-401 applied to each
// cell, with the Fe-Fe potential of src/fetransmetal.F90), and the adjoint
// with respect to the potential's knots.
//
// The unit of work is a tile: at most 64 consecutive atoms (one wave, one lane
// per atom) of one cell, in sub-cell order.  Every pass is one launch over all
// tiles of all cells, so the chip is full whatever the cells' sizes are and no
// pass waits for a large cell:
//   k_pack   packed positions and candidate records
//   k_list   neighbour list, densities, embedding
//   k_force  forces, pair energy and virial partials (and the loss's seeds)
//   k_cells  per-cell sums of the tiles' partials, in tile order
//   k_adjoint, k_fold, k_grad_out   gradient of a loss, or a seeded product
// Sums over atoms have a fixed order: lanes, then tiles, then cells.
//
// One workgroup per cell (whole cells from a work queue) was the earlier form:
// a 4000-atom cell kept one 256-thread workgroup busy for 1.19 ms while the
// rest of the chip was idle; 256 cells of 54..4000 atoms took 1191 us against
// 101 us now, loss and gradient of 1024 cells 1930 us against 513 us.
//
// Pair arithmetic is FP32 (or FP64), with FP64 accumulation of densities,
// energies and virials over atoms; positions are FP64.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "../../include/moldy_hip.h"
#include "mdk_hostpot.h"
#include "mdk_internal.h"
#include "mdk_wave.h"

namespace {

thread_local char b_err[512] = "";
int berr(int code, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(b_err, sizeof(b_err), fmt, ap);
  va_end(ap);
  return code;
}
#define BCK(call)                                                                        \
  do {                                                                                   \
    hipError_t e_ = (call);                                                              \
    if (e_ != hipSuccess)                                                                \
      return berr(MDK_ERR_HIP, "%s failed: %s (%s:%d)", #call, hipGetErrorString(e_),     \
                  __FILE__, __LINE__);                                                   \
  } while (0)

// A list entry is j | code << 27: j the partner's local atom index, code =
// (ox+1) + 3 (oy+1) + 9 (oz+1) with o the offset of j's sub-cell (unwrapped)
// from i's; along a dimension with one sub-cell o is j's periodic image.
// r_ij = (R_i - R_j) + D[code], R the position from the centre of the atom's
// sub-cell and D = -B (o / n).  Code 27 places the partner 1e6 A away, where
// every pair term is zero: it pads lists to a multiple of four entries.
#define NB_IDX_MASK 0x07FFFFFF
#define NB_CODE_SHIFT 27
#define NB_NULL_CODE 27
#define TILE 64

// gradient slots: a_k, r_k (MDK_MAXV each), A_k, R_k (MDK_MAXP each)
#define NGRAD_SLOTS (2 * MDK_MAXV + 2 * MDK_MAXP)
// partial sums of a tile: pair energy, virial (xx yy zz xy xz yz), embedding
// energy, sum |F - F_t|^2
#define NPART_TILE 9
#define PT_EMB 7
#define PT_FSQ 8
#define FOLD_CHUNKS 32  // first-stage blocks per gradient slot

// One cell.  nx, ny, nz: sub-cells per dimension (1, or >= 3, each at least the
// interaction range wide).  rows: >= 3 in every dimension, candidate records
// in rows along x with the wrapped neighbour cells repeated at both ends;
// otherwise one record per atom.
struct CellMeta {
  int a0, nc, tile0, ntile;
  int nx, ny, nz, rows;
  int est0;     // first entry of the cell's record offsets in est
  int rec0;     // first candidate record
  float ext;    // largest sum over cell vectors of a Cartesian component's magnitude
  int pad;
};

struct Tile {
  int cell, a0, cnt, il0;  // cell, first atom (global), atoms, first atom (within the cell)
};

struct BatchArgs {
  int ncell, natom, ntile, nrec, maxnb;
  const CellMeta *meta;
  const Tile *tiles;
  const double *box;     // 9 per cell, column-major
  const int *subc;       // per atom: local sub-cell index (x fastest)
  const int *est;        // record offsets (relative to rec0) of the cell's (extended) sub-cells
  const int2 *rsrc;      // per record: cell, local atom | ghost << 28 (0 none, 1 and 2: wrapped from above, below)
  const double *s;       // 3 per atom: fractional, wrapped into [0,1), sorted by sub-cell
  const int *perm;       // sorted atom -> caller's atom index
  float4 *rec;           // candidate records: FP32 position (Cartesian, or fractional without rows), local index
  double4 *pos4;         // FP64 form: position from the sub-cell's centre, F'
  float4 *p4f;           // FP32 form: the same in FP32, F'
  double *daf;           // FP32 form: F' in FP64
  int4 *nbr;             // per tile: quad q of lane l's entries at nbr[(tile maxnb / 4 + q) 64 + l]
  int *numn;
  double *rho;           // per caller atom
  double *part;          // NPART_TILE per tile
  double *out_e;         // per cell energy
  double *out_w;         // per cell virial W (6: xx yy zz xy xz yz), W = sum_pairs r r^T fp
  double *out_f;         // 3 per caller atom, Cartesian forces
  int *flags;            // [0] max neighbour count seen when over capacity
  int *flags_out;        // host-mapped copy, written by k_cells
  double rc;             // interaction range (outermost knot)
  const float *fetab;    // FP32 form: V, V', phi' interval table of the knots
  // adjoint
  const double *e_in;    // per cell: dL/dE_c (vector-Jacobian product) or target E_c (loss)
  const double *f_in;    // 3 per caller atom: dL/dF_i (product) or target F_i (loss)
  double4 *gvec;         // per sorted atom: the force seed dL/dF_i
  double *ecell;         // per cell: dL/dE_c of the loss
  double *part_g;        // gradient partials: slot k of tile t at [k ntile + t]
  double *out_loss;      // per cell loss
  double f_weight;       // loss weight of sum_i |F_i - F_t,i|^2 (0.1 / total atoms)
};

__device__ __forceinline__ void r_inv(double r2, double &r, double &ri) {
  double y = __builtin_amdgcn_rsq(r2);
  const double h = 0.5 * r2;
  y = y * (1.5 - h * y * y);
  y = y * (1.5 - h * y * y);
  ri = y;
  r = r2 * y;
}
__device__ __forceinline__ void r_inv(float r2, float &r, float &ri) {
  float y = __builtin_amdgcn_rsqf(r2);
  y = y * (1.5f - 0.5f * r2 * y * y);
  ri = y;
  r = r2 * y;
}

// pair functions for the potential's own 6 + 2 knots (FE) or any knot count
template <typename T, bool FE>
__device__ __forceinline__ T b_phi(const PotDev &P, T r) {
  return mdk_phi_n<T, FE ? MDK_FE_NP : MDK_MAXP>(P, r);
}

// Tile order: physical block b takes the tiles of logical block
// start(b mod 8) + b / 8, so each XCD works on one contiguous range of tiles
// and a cell's records stay in one L2.
__device__ __forceinline__ int logical_block() {
  const int nb = gridDim.x, b = blockIdx.x, q = nb / 8, r = nb % 8, x = b % 8;
  return x * q + min(x, r) + b / 8;
}

// This wave's tile and cell (wave-uniform; idle waves past the last tile take
// the last one with no atoms).
struct TileView {
  Tile t;
  CellMeta m;
  int index, il;  // tile index; this lane's local atom (valid when active)
  bool active;
};
template <int BLOCK>
__device__ __forceinline__ TileView tile_view(const BatchArgs &A) {
  TileView v;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  int ti = logical_block() * (BLOCK / TILE) + w;
  const bool real = ti < A.ntile;
  ti = real ? ti : A.ntile - 1;
  v.index = real ? ti : -1;
  v.t = A.tiles[ti];
  v.m = A.meta[v.t.cell];
  v.active = real && lane < v.t.cnt;
  v.il = v.t.il0 + lane;
  return v;
}

// The wave's 27 shifts D[code] = -B (o / n): FP64, or FP32 as an unevaluated
// sum hi + lo (a rounded shift would bias every pair of a code the same way).
template <typename T> struct Shifts;
template <> struct Shifts<double> {
  double d[28][3];
};
template <> struct Shifts<float> {
  float4 hi[28], lo[28];
};
template <typename T>
__device__ __forceinline__ void fill_shifts(const BatchArgs &A, const TileView &V, Shifts<T> &S) {
  const int k = threadIdx.x & 63;
  if (k > 27) return;
  const double *b = A.box + 9 * (size_t)V.t.cell;
  const double fx = -(double)(k % 3 - 1) / V.m.nx, fy = -(double)((k / 3) % 3 - 1) / V.m.ny,
               fz = -(double)(k / 9 - 1) / V.m.nz;
  double dx = b[0] * fx + b[3] * fy + b[6] * fz, dy = b[1] * fx + b[4] * fy + b[7] * fz,
         dz = b[2] * fx + b[5] * fy + b[8] * fz;
  if (k == NB_NULL_CODE) {
    dx = 1.0e6;
    dy = dz = 0.0;
  }
  if constexpr (sizeof(T) == 8) {
    S.d[k][0] = dx;
    S.d[k][1] = dy;
    S.d[k][2] = dz;
  } else {
    const float hx = (float)dx, hy = (float)dy, hz = (float)dz;
    S.hi[k] = make_float4(hx, hy, hz, 0.f);
    S.lo[k] = make_float4((float)(dx - (double)hx), (float)(dy - (double)hy), (float)(dz - (double)hz), 0.f);
  }
}

// packed record of either form
template <typename T> struct Rec;
template <> struct Rec<double> {
  using V = double4;
  static __device__ __forceinline__ double4 *of(const BatchArgs &A) { return A.pos4; }
};
template <> struct Rec<float> {
  using V = float4;
  static __device__ __forceinline__ float4 *of(const BatchArgs &A) { return A.p4f; }
};
__device__ __forceinline__ void pair_sep(const double4 &pi, const double4 &pj, const Shifts<double> &S, int code,
                                         double &x, double &y, double &z) {
  x = (pi.x - pj.x) + S.d[code][0];
  y = (pi.y - pj.y) + S.d[code][1];
  z = (pi.z - pj.z) + S.d[code][2];
}
__device__ __forceinline__ void pair_sep(const float4 &pi, const float4 &pj, const Shifts<float> &S, int code,
                                         float &x, float &y, float &z) {
  const float4 d = S.hi[code], l = S.lo[code];
  x = ((pi.x - pj.x) + d.x) + l.x;
  y = ((pi.y - pj.y) + d.y) + l.y;
  z = ((pi.z - pj.z) + d.z) + l.z;
}

// Candidate records and packed positions.  One thread per record; the record
// of an atom itself (no ghost) also writes the packed position.  Bound by
// memory: 24 B read and 32 (FP32) or 48 B written per atom.
template <typename T>
__global__ void __launch_bounds__(256) k_pack(BatchArgs A) {
  const int r = blockIdx.x * 256 + threadIdx.x;
  if (r >= A.nrec) return;
  const int2 src = A.rsrc[r];
  const CellMeta m = A.meta[src.x];
  const int il = src.y & 0x0FFFFFFF, ghost = src.y >> 28;
  const size_t a = (size_t)m.a0 + il;
  const double *b = A.box + 9 * (size_t)src.x;
  double x = A.s[3 * a], y = A.s[3 * a + 1], z = A.s[3 * a + 2];
  if (m.rows) {
    const double gx = ghost == 0 ? x : (ghost == 1 ? x - 1.0 : x + 1.0);
    A.rec[r] = make_float4((float)(b[0] * gx + b[3] * y + b[6] * z), (float)(b[1] * gx + b[4] * y + b[7] * z),
                           (float)(b[2] * gx + b[5] * y + b[8] * z), __int_as_float(il));
    if (ghost) return;
  } else {
    A.rec[r] = make_float4((float)x, (float)y, (float)z, __int_as_float(il));
  }
  const int sc = A.subc[a], cx = sc % m.nx, cy = (sc / m.nx) % m.ny, cz = sc / (m.nx * m.ny);
  x -= (cx + 0.5) / m.nx;
  y -= (cy + 0.5) / m.ny;
  z -= (cz + 0.5) / m.nz;
  const double px = b[0] * x + b[3] * y + b[6] * z, py = b[1] * x + b[4] * y + b[7] * z,
               pz = b[2] * x + b[5] * y + b[8] * z;
  if constexpr (sizeof(T) == 8) A.pos4[a] = make_double4(px, py, pz, 0.0);
  else A.p4f[a] = make_float4((float)px, (float)py, (float)pz, 0.f);
}

// This lane's list being written: entries through a register quad, every fourth
// stores it with one 16-byte write.
struct ListOut {
  int4 *nb;
  int maxnb, cnt;
  int a, b, c, d;
  __device__ __forceinline__ void put(int e) {
    a = b; b = c; c = d; d = e;
    cnt++;
    if (!(cnt & 3) && cnt <= maxnb) nb[((cnt >> 2) - 1) * TILE] = make_int4(a, b, c, d);
  }
};
// orders a wave's LDS accesses across its lanes
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// A walk finds partners by FP32 positions in the whole cell, whose rounding grows
// with the cell: a separation is off by at most 16 half-ulps of the extent (rows: 2
// for the record, 1 for the atom, 1 for the shifts, 5 for adding those, times
// sqrt(3); less by fractions), below 1e-6 of it, and by 1e-5 A of the FP32 square.
// So lists end that much past the range, at least 1e-4 A (pairs beyond the range add
// exact zeros).  FP64 lists end at the range: the few partners that are not inside it
// for certain are tested again, in FP64 and by the separation that the passes form.
// us per pass with one FP32 test against 1e-4 A : so -- 48 cells in FP64, list and
// adjoint 298 : 305; 1024 cells in FP32, loss and gradient 472 : 473.
#define LIST_MARGIN 1e-4
#define LIST_ROUND 1e-6
template <typename T> struct Range {
  float cand2, sure2;  // squares: candidates below, and in range for certain below
  double rc2;
  const double4 *pc;
  double4 pi;
  const Shifts<T> &S;
  __device__ __forceinline__ Range(const BatchArgs &A, const TileView &V, const Shifts<T> &S_) : S(S_) {
    const double off = LIST_ROUND * V.m.ext + 1e-5, c = A.rc + fmax(LIST_MARGIN, off), u = fmax(A.rc - off, 0.0);
    cand2 = (float)(c * c);
    if constexpr (sizeof(T) == 8) {
      sure2 = (float)(u * u);
      rc2 = A.rc * A.rc;
      pc = A.pos4 + V.m.a0;
      pi = pc[V.active ? V.il : 0];
    }
  }
  // whether candidate j with the FP32 square r2 belongs to the list
  __device__ __forceinline__ bool holds(float r2, int j, int code) const {
    if constexpr (sizeof(T) == 8) {
      if (r2 < sure2) return true;
      double x, y, z;
      pair_sep(pi, pc[j], S, code, x, y, z);
      return x * x + y * y + z * z < rc2;
    }
    return true;
  }
};

// Appends the partners of this lane's atom to its list (a whole wave calls; lanes
// past the tile's atoms only help to stage).
// The candidate records of a plane of rows pass through LDS in windows of at most
// LIST_WIN (a plane's rows of the tile's sub-cells mostly fit one), read in order,
// and each lane tests those of its three rows.  Read by every lane for itself, 16
// bytes at a time, they kept the address units busy for 83 % of the kernel; now the
// vector ALU binds (some 180 tests, 16 appended entries).  A row's hits are
// collected as a bit mask, so that the lanes append in step and one candidate in
// ten does not run the appending code for the others.  us before : after -- 1024
// cells, 1.27 M atoms 254 : 221, 256 cells 71 : 65, 48 cells in FP64 46.3 : 44.5.
// Windows of 256 records split planes (224, 72, 49), of 512 leave four waves per
// SIMD (241, 85, 41).  Candidates are visited in a fixed order (planes, windows,
// rows; then along x).
#define LIST_WIN 384
__device__ __forceinline__ int wave_max_i(int v) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) v = max(v, __shfl_xor(v, o, 64));
  return __builtin_amdgcn_readfirstlane(v);
}
template <typename T>
__device__ __forceinline__ void walk_rows(const BatchArgs &A, const TileView &V, const Range<T> &N, float4 *win,
                                          ListOut &out) {
  const double *b = A.box + 9 * (size_t)V.t.cell;
  const int lane = threadIdx.x & 63;
  const size_t a = (size_t)V.m.a0 + (V.active ? V.il : 0);
  const int nx = V.m.nx, ny = V.m.ny, nz = V.m.nz;
  const int sc = A.subc[a], cx = sc % nx, cy = (sc / nx) % ny, cz = sc / (nx * ny);
  const double sx = A.s[3 * a], sy = A.s[3 * a + 1], sz = A.s[3 * a + 2];
  const float px = (float)(b[0] * sx + b[3] * sy + b[6] * sz), py = (float)(b[1] * sx + b[4] * sy + b[7] * sz),
              pz = (float)(b[2] * sx + b[5] * sy + b[8] * sz);
  const float yx = (float)b[3], yy = (float)b[4], yz = (float)b[5], zx = (float)b[6], zy = (float)b[7],
              zz = (float)b[8];
  const int *est = A.est + V.m.est0;
  const int nrec = est[(nx + 2) * ny * nz];
  const float4 *rec = A.rec + V.m.rec0;
#pragma unroll 1
  for (int oz = -1; oz <= 1; oz++) {
    int kz = cz + oz;
    const float wz = kz < 0 ? 1.f : (kz >= nz ? -1.f : 0.f);
    kz += kz < 0 ? nz : (kz >= nz ? -nz : 0);
    int lo[3], m1[3], m2[3], hi[3];
    float wy[3];
#pragma unroll
    for (int y = 0; y < 3; y++) {
      int ky = cy + y - 1;
      wy[y] = ky < 0 ? 1.f : (ky >= ny ? -1.f : 0.f);
      ky += ky < 0 ? ny : (ky >= ny ? -ny : 0);
      const int *e = est + (size_t)(ky + ny * kz) * (nx + 2) + cx;  // sub-cell cx - 1 of an extended row
      lo[y] = e[0];
      m1[y] = e[1];
      m2[y] = e[2];
      hi[y] = V.active ? e[3] : 0;
    }
    // the wave's range of records (lanes past the tile's atoms have the first atom's)
    const int first = -wave_max_i(-min(lo[0], min(lo[1], lo[2]))), last = wave_max_i(max(hi[0], max(hi[1], hi[2])));
    for (int w0 = first; w0 < last; w0 += LIST_WIN) {
      const int w1 = min(last, w0 + LIST_WIN);
      bool any = false;
#pragma unroll
      for (int y = 0; y < 3; y++) any = any || max(lo[y], w0) < min(hi[y], w1);
      if (!__ballot(any)) continue;
      wave_sync();  // the last window has been read
#pragma unroll
      for (int u = 0; u < LIST_WIN / 64; u++)
        if (w0 + u * 64 < w1) win[u * 64 + lane] = rec[min(w0 + u * 64 + lane, nrec - 1)];
      wave_sync();
#pragma unroll
      for (int y = 0; y < 3; y++) {
        const float qx = px + wy[y] * yx + wz * zx, qy = py + wy[y] * yy + wz * zy, qz = pz + wy[y] * yz + wz * zz;
        const int end = min(hi[y], w1), base = 3 * y + 9 * (oz + 1);
        for (int c0 = max(lo[y], w0); c0 < end; c0 += 32) {
          const int m = min(32, end - c0);
          const float4 *q = win + (c0 - w0);
          unsigned hit = 0;
          auto sep2 = [&](const float4 &p) {
            const float ex = qx - p.x, ey = qy - p.y, ez = qz - p.z;
            return ex * ex + ey * ey + ez * ez;
          };
          auto test = [&](const float4 &p, int k) { hit |= sep2(p) < N.cand2 ? 1u << k : 0u; };
          int k = 0;
          for (; k + 4 <= m; k += 4) {  // four LDS reads in flight
            const float4 q0 = q[k], q1 = q[k + 1], q2 = q[k + 2], q3 = q[k + 3];
            test(q0, k);
            test(q1, k + 1);
            test(q2, k + 2);
            test(q3, k + 3);
          }
          for (; k < m; k++) test(q[k], k);
          while (hit) {
            const int h = __builtin_ctz(hit), c = c0 + h;
            const float4 p = q[h];
            const int j = __float_as_int(p.w);
            hit &= hit - 1;
            const int code = base + (c >= m1[y] ? 1 : 0) + (c >= m2[y] ? 1 : 0);
            if (j != V.il && N.holds(sep2(p), j, code)) out.put(j | (code << NB_CODE_SHIFT));
          }
        }
      }
    }
  }
}
// Any grid (some dimension with one sub-cell): the nearest image of the
// fractional separation.  An in-range pair's nearest image is the one its
// sub-cell offset names, since the cell is wider than twice the range.
template <typename T>
__device__ __forceinline__ void walk_any(const BatchArgs &A, const TileView &V, const Range<T> &N, ListOut &out) {
  const double *b = A.box + 9 * (size_t)V.t.cell;
  const size_t a = (size_t)V.m.a0 + V.il;
  const int nx = V.m.nx, ny = V.m.ny, nz = V.m.nz;
  const int rx = nx >= 3 ? 1 : 0, ry = ny >= 3 ? 1 : 0, rz = nz >= 3 ? 1 : 0;
  const int sc = A.subc[a], cx = sc % nx, cy = (sc / nx) % ny, cz = sc / (nx * ny);
  const float sx = (float)A.s[3 * a], sy = (float)A.s[3 * a + 1], sz = (float)A.s[3 * a + 2];
  float bf[9];
#pragma unroll
  for (int k = 0; k < 9; k++) bf[k] = (float)b[k];
  const int *est = A.est + V.m.est0;
  const float4 *rec = A.rec + V.m.rec0;
  for (int oz = -rz; oz <= rz; oz++) {
    const int kz = cz + oz < 0 ? cz + oz + nz : (cz + oz >= nz ? cz + oz - nz : cz + oz);
    for (int oy = -ry; oy <= ry; oy++) {
      const int ky = cy + oy < 0 ? cy + oy + ny : (cy + oy >= ny ? cy + oy - ny : cy + oy);
      for (int ox = -rx; ox <= rx; ox++) {
        const int kx = cx + ox < 0 ? cx + ox + nx : (cx + ox >= nx ? cx + ox - nx : cx + ox);
        const int cj = kx + nx * (ky + ny * kz);
        const int lo = est[cj], hi = est[cj + 1];
        for (int c = lo; c < hi; c += 4) {
          float4 q[4];
#pragma unroll
          for (int u = 0; u < 4; u++) q[u] = rec[c + u];
#pragma unroll
          for (int u = 0; u < 4; u++) {
            float ex = sx - q[u].x, ey = sy - q[u].y, ez = sz - q[u].z;
            const float tx = rintf(ex), ty = rintf(ey), tz = rintf(ez);
            ex -= tx; ey -= ty; ez -= tz;
            const float x = bf[0] * ex + bf[3] * ey + bf[6] * ez, y = bf[1] * ex + bf[4] * ey + bf[7] * ez,
                        z = bf[2] * ex + bf[5] * ey + bf[8] * ez;
            const int j = __float_as_int(q[u].w);
            const float r2 = x * x + y * y + z * z;
            if (r2 < N.cand2 && c + u < hi && j != V.il) {
              const int code = (rx ? ox : (int)tx) + 3 * (ry ? oy : (int)ty) + 9 * (rz ? oz : (int)tz) + 13;
              if (N.holds(r2, j, code)) out.put(j | (code << NB_CODE_SHIFT));
            }
          }
        }
      }
    }
  }
}

// Neighbour list at the interaction range, then the densities over it
// (src/dynamics_m.F90:497-579) and the embedding (src/potential_m.F90:148-169):
// rho, F' into the packed record's w, the tile's embedding energy.  Bound by
// VALU issue: about 150 to 250 candidate tests per atom, then some 16 density
// terms.  The densities are a second loop over the finished list: inside the
// walk the density code would run for almost every candidate trip, since some
// lane of the wave hits, while only one candidate in ten is a partner.
template <typename T, int BLOCK, bool FE>
__global__ void __launch_bounds__(BLOCK) k_list(BatchArgs A, PotDev P) {
  __shared__ Shifts<T> SH[BLOCK / TILE];
  __shared__ float4 win[BLOCK / TILE][LIST_WIN];
  const TileView V = tile_view<BLOCK>(A);
  Shifts<T> &S = SH[threadIdx.x >> 6];
  fill_shifts<T>(A, V, S);
  __syncthreads();
  double e_emb = 0.0;
  const int lane = threadIdx.x & 63;
  int4 *nb = A.nbr + (size_t)max(V.index, 0) * (A.maxnb / 4) * TILE + lane;
  ListOut out = {nb, A.maxnb, 0, 0, 0, 0, 0};
  const Range<T> N(A, V, S);
  if (V.m.rows) walk_rows<T>(A, V, N, win[threadIdx.x >> 6], out);
  else if (V.active) walk_any<T>(A, V, N, out);
  if (V.active) {
    const size_t a = (size_t)V.m.a0 + V.il;
    int cnt = out.cnt;
    if (cnt > A.maxnb) atomicMax(&A.flags[0], cnt);
    while (out.cnt & 3) out.put(V.il | (NB_NULL_CODE << NB_CODE_SHIFT));
    cnt = min(cnt, A.maxnb);
    A.numn[a] = cnt;
    const int end = (cnt + 3) & ~3;
    const typename Rec<T>::V *pc = Rec<T>::of(A) + V.m.a0;
    const typename Rec<T>::V pi = pc[V.il];
    double acc = 0.0;
    for (int k = 0; k < end; k += 4) {
      const int4 e4 = nb[(k >> 2) * TILE];
      const unsigned e[4] = {(unsigned)e4.x, (unsigned)e4.y, (unsigned)e4.z, (unsigned)e4.w};
      typename Rec<T>::V q[4];
#pragma unroll
      for (int u = 0; u < 4; u++) q[u] = pc[e[u] & NB_IDX_MASK];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        T dx, dy, dz, r, ri;
        pair_sep(pi, q[u], S, (int)(e[u] >> NB_CODE_SHIFT), dx, dy, dz);
        r_inv(dx * dx + dy * dy + dz * dz, r, ri);
        acc += (double)b_phi<T, FE>(P, r);
      }
    }
    A.rho[A.perm[a]] = acc;
    double f = 0.0, df = 0.0;
    if (acc > 1e-40) {
      mdk_embed_f(P, acc, f, df);
      e_emb = f;
    }
    if constexpr (sizeof(T) == 8) {
      A.pos4[a].w = df;
    } else {
      A.daf[a] = df;
      A.p4f[a].w = (float)df;
    }
  }
  e_emb = wave_sum(e_emb);
  if (V.index >= 0 && (threadIdx.x & 63) == 0) A.part[(size_t)V.index * NPART_TILE + PT_EMB] = e_emb;
}

// Forces and virial (src/dynamics_m.F90:235-346).  With LOSS, also the force
// seed dL/dF_i = 2 f_weight (F_i - F_t,i) into gvec and the tile's sum of
// |F_i - F_t,i|^2.  FP32 form: each atom's force, pair energy and virial terms
// are summed in FP32 over its partners (V, V' and phi' from the interval table
// with TAB, knot sums otherwise), over atoms in FP64; FP64 form: every term in
// FP64.  Four list entries per trip, their partner loads in flight together.
template <typename T, int BLOCK, bool FE, bool TAB, bool LOSS>
__global__ void __launch_bounds__(BLOCK) k_force(BatchArgs A, PotDev P) {
  __shared__ Shifts<T> SH[BLOCK / TILE];
  __shared__ float4 fbin[MDK_FE_NB];
  __shared__ __align__(16) float fiv[8 * MDK_FE_NI];
  if (TAB) {
    const float4 *src = (const float4 *)A.fetab;
    for (int t = threadIdx.x; t < MDK_FE_NB + 2 * MDK_FE_NI; t += BLOCK) {
      if (t < MDK_FE_NB) fbin[t] = src[t];
      else ((float4 *)fiv)[t - MDK_FE_NB] = src[t];
    }
  }
  const TileView V = tile_view<BLOCK>(A);
  Shifts<T> &S = SH[threadIdx.x >> 6];
  fill_shifts<T>(A, V, S);
  __syncthreads();
  constexpr int NS = LOSS ? 8 : 7;
  double v[NS];
#pragma unroll
  for (int k = 0; k < NS; k++) v[k] = 0.0;
  if (V.active) {
    const int lane = threadIdx.x & 63;
    const size_t a = (size_t)V.m.a0 + V.il;
    const int4 *nb = A.nbr + (size_t)V.index * (A.maxnb / 4) * TILE + lane;
    const int end = (A.numn[a] + 3) & ~3;
    const typename Rec<T>::V *pc = Rec<T>::of(A) + V.m.a0;
    const typename Rec<T>::V pi = pc[V.il];
    T fx = T(0), fy = T(0), fz = T(0), se = T(0), s0 = T(0), s1 = T(0), s2 = T(0), s3 = T(0), s4 = T(0), s5 = T(0);
    for (int k = 0; k < end; k += 4) {
      const int4 e4 = nb[(k >> 2) * TILE];
      const unsigned e[4] = {(unsigned)e4.x, (unsigned)e4.y, (unsigned)e4.z, (unsigned)e4.w};
      typename Rec<T>::V q[4];
#pragma unroll
      for (int u = 0; u < 4; u++) q[u] = pc[e[u] & NB_IDX_MASK];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        T dx, dy, dz, r, rr, vv, dv, dph;
        pair_sep(pi, q[u], S, (int)(e[u] >> NB_CODE_SHIFT), dx, dy, dz);
        r_inv(dx * dx + dy * dy + dz * dz, r, rr);
        if constexpr (TAB) {
          mdk_fe_terms(P, fbin, fiv, r, vv, dv, dph);
        } else {
          mdk_vee_n<T, FE ? MDK_FE_NV : MDK_MAXV>(P, r, vv, dv);
          dph = mdk_dphi_n<T, FE ? MDK_FE_NP : MDK_MAXP>(P, r);
        }
        const T fp = -dv * rr + (-T(1) * (dph * pi.w + dph * q[u].w) * rr);
        const T gx = dx * fp, gy = dy * fp, gz = dz * fp;
        se += vv;
        fx += gx; fy += gy; fz += gz;
        s0 += dx * gx; s1 += dy * gy; s2 += dz * gz;
        s3 += dx * gy; s4 += dx * gz; s5 += dy * gz;
      }
    }
    v[0] = 0.5 * (double)se;
    v[1] = 0.5 * (double)s0; v[2] = 0.5 * (double)s1; v[3] = 0.5 * (double)s2;
    v[4] = 0.5 * (double)s3; v[5] = 0.5 * (double)s4; v[6] = 0.5 * (double)s5;
    const size_t u = (size_t)A.perm[a];
    A.out_f[3 * u] = (double)fx;
    A.out_f[3 * u + 1] = (double)fy;
    A.out_f[3 * u + 2] = (double)fz;
    if constexpr (LOSS) {
      const double ex = (double)fx - A.f_in[3 * u], ey = (double)fy - A.f_in[3 * u + 1],
                   ez = (double)fz - A.f_in[3 * u + 2];
      v[7] = ex * ex + ey * ey + ez * ez;
      const double g = 2.0 * A.f_weight;
      A.gvec[a] = make_double4(g * ex, g * ey, g * ez, 0.0);
    }
  }
  wave_reduce_all<NS, 0>(v);
  if (V.index >= 0 && (threadIdx.x & 63) == 0) {
    double *p = A.part + (size_t)V.index * NPART_TILE;
#pragma unroll
    for (int k = 0; k < 7; k++) p[k] = v[k];
    if constexpr (LOSS) p[PT_FSQ] = v[7];
  }
}

// Per-cell sums over the cell's tiles (one wave per cell, lanes then the wave
// in a fixed order): energy, virial; with LOSS the cell's loss
// (E_c - E_t,c)^2 / N_c^2 + f_weight sum |F_i - F_t,i|^2 and its dL/dE_c.
template <bool LOSS>
__global__ void __launch_bounds__(256) k_cells(BatchArgs A) {
  const int c = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (blockIdx.x == 0 && threadIdx.x < 4) A.flags_out[threadIdx.x] = A.flags[threadIdx.x];
  if (c >= A.ncell) return;
  const CellMeta m = A.meta[c];
  double v[NPART_TILE];
#pragma unroll
  for (int k = 0; k < NPART_TILE; k++) v[k] = 0.0;
  for (int t = lane; t < m.ntile; t += 64) {
    const double *p = A.part + (size_t)(m.tile0 + t) * NPART_TILE;
#pragma unroll
    for (int k = 0; k < NPART_TILE; k++)
      if (LOSS || k != PT_FSQ) v[k] += p[k];
  }
  wave_reduce_all<NPART_TILE, 0>(v);
  const double e = v[0] + v[PT_EMB];
  if (lane == 0) A.out_e[c] = e;
  if (lane < 6) A.out_w[6 * (size_t)c + lane] = lane == 0 ? v[1] : lane == 1 ? v[2] : lane == 2 ? v[3] : lane == 3 ? v[4] : lane == 4 ? v[5] : v[6];
  if (LOSS && lane == 0) {
    const double inv_n2 = 1.0 / ((double)m.nc * (double)m.nc), de = e - A.e_in[c];
    A.ecell[c] = 2.0 * de * inv_n2;
    A.out_loss[c] = de * de * inv_n2 + A.f_weight * v[PT_FSQ];
  }
}

// force seeds of a vector-Jacobian product, into sorted order
__global__ void __launch_bounds__(256) k_seeds(BatchArgs A) {
  const int a = blockIdx.x * 256 + threadIdx.x;
  if (a >= A.natom) return;
  const size_t u = (size_t)A.perm[a];
  A.gvec[a] = make_double4(A.f_in[3 * u], A.f_in[3 * u + 1], A.f_in[3 * u + 2], 0.0);
}

// Adjoint.  With seeds e_c = dL/dE_c and G_i = dL/dF_i, F_i the
// force on atom i, r_ij = R_i - R_j and u_ij = (G_i - G_j) . r_ij / r:
//   dL/dtheta = sum_i sum_j { e_c [ V_theta/2 + F'_i phi_theta ]
//                             - [ V'_theta + (F'_i + F'_j) phi'_theta ] u_ij / 2
//                             - lambda_i phi_theta },
//   lambda_i = F''(rho_i) Q_i,  Q_i = sum_j phi'(r_ij) u_ij,  F'' = -2 F'^3,
// over the full list (every pair from both ends).  The lambda term is
// accumulated as lambda_i d(rho_i)/dtheta after the neighbour loop, so one
// pass over the list suffices.  The list and F' are those of the forward
// passes; G from gvec, e_c from seed (the loss's ecell, or the caller's).
// NV, NP: pair and density knot counts the per-lane FP64 gradient sums hold
// (6 and 2 for the Fe potential; the maxima for any other knot set).
template <typename T, int BLOCK, int NV, int NP>
__global__ void __launch_bounds__(BLOCK) k_adjoint(BatchArgs A, PotDev P, GradDev D, const double *__restrict__ seed) {
  __shared__ Shifts<T> SH[BLOCK / TILE];
  const TileView V = tile_view<BLOCK>(A);
  Shifts<T> &S = SH[threadIdx.x >> 6];
  fill_shifts<T>(A, V, S);
  __syncthreads();
  PotView<T> Q(P);
  double gv[2 * NV], gp[2 * NP];  // a_k then r_k; A_k then R_k
#pragma unroll
  for (int m = 0; m < 2 * NV; m++) gv[m] = 0.0;
#pragma unroll
  for (int m = 0; m < 2 * NP; m++) gp[m] = 0.0;
  if (V.active) {
    const int lane = threadIdx.x & 63;
    const size_t a = (size_t)V.m.a0 + V.il;
    const int4 *nb = A.nbr + (size_t)V.index * (A.maxnb / 4) * TILE + lane;
    const int nn = A.numn[a];
    const typename Rec<T>::V *pc = Rec<T>::of(A) + V.m.a0;
    const double4 *gc = A.gvec + V.m.a0;
    const typename Rec<T>::V pi = pc[V.il];
    double fi;  // F'_i in FP64
    if constexpr (sizeof(T) == 8) fi = pi.w;
    else fi = A.daf[a];
    const T fpi = (T)fi;
    const double4 gi = gc[V.il];
    const double ec = seed[V.t.cell];
    double q = 0.0, drA[NP], drR[NP];
#pragma unroll
    for (int m = 0; m < NP; m++) { drA[m] = 0.0; drR[m] = 0.0; }
    int4 e4 = make_int4(0, 0, 0, 0);
    for (int k = 0; k < nn; k++) {
      if (!(k & 3)) e4 = nb[(k >> 2) * TILE];
      const unsigned e = (unsigned)e4.x;
      e4.x = e4.y;
      e4.y = e4.z;
      e4.z = e4.w;
      const int jl = (int)(e & NB_IDX_MASK);
      const typename Rec<T>::V pj = pc[jl];
      const double4 gj = gc[jl];
      const T fpj = (T)pj.w;
      T dx, dy, dz, r, ri;
      pair_sep(pi, pj, S, (int)(e >> NB_CODE_SHIFT), dx, dy, dz);
      r_inv(dx * dx + dy * dy + dz * dz, r, ri);
      const T u = ((T)(gi.x - gj.x) * dx + (T)(gi.y - gj.y) * dy + (T)(gi.z - gj.z) * dz) * ri;
      const T dph = mdk_dphi_n<T, NP>(P, r);
      q += (double)(dph * u);
      const T cv = T(0.5) * (T)ec, cvp = T(-0.5) * u;
      const T cp = (T)ec * fpi, cpp = T(-0.5) * (fpi + fpj) * u;
      // pair parameters
      if (r > Q.bc2()) {
#pragma unroll
        for (int m = 0; m < NV; m++) {
          if (m < P.nv) {
            const T d = Q.rv(m) - r;
            if (d > T(0)) {
              const T d2 = d * d;
              gv[m] += (double)(cv * d2 * d - T(3) * cvp * d2);
              gv[NV + m] += (double)(Q.av(m) * (T(3) * cv * d2 - T(6) * cvp * d));
            }
          }
        }
      } else if (r > Q.bc1()) {
        // log-space Hermite join: only x2 and v2 depend on the knots
        const double h = P.bc2 - P.bc1, t = ((double)r - P.bc1) / h;
        const double t2 = t * t, t3 = t2 * t;
        const double sp = (2 * t3 - 3 * t2 + 1) * P.jx1 + (t3 - 2 * t2 + t) * P.jv1 * h +
                          (-2 * t3 + 3 * t2) * P.jx2 + (t3 - t2) * P.jv2 * h;
        const double ds = ((6 * t2 - 6 * t) * P.jx1 + (3 * t2 - 4 * t + 1) * P.jv1 * h +
                           (-6 * t2 + 6 * t) * P.jx2 + (3 * t2 - 2 * t) * P.jv2 * h) / h;
        const double ve = exp(sp), vpe = ds * ve;
        const double h01 = -2 * t3 + 3 * t2, h11 = (t3 - t2) * h;
        const double d01 = (-6 * t2 + 6 * t) / h, d11 = 3 * t2 - 2 * t;
#pragma unroll
        for (int m = 0; m < NV; m++) {
          if (m < P.nv) {
            const double sa = h01 * D.xa[m] + h11 * D.ya[m], sr = h01 * D.xr[m] + h11 * D.yr[m];
            const double pa = d01 * D.xa[m] + d11 * D.ya[m], pr = d01 * D.xr[m] + d11 * D.yr[m];
            gv[m] += (double)cv * (ve * sa) + (double)cvp * (pa * ve + vpe * sa);
            gv[NV + m] += (double)cv * (ve * sr) + (double)cvp * (pr * ve + vpe * sr);
          }
        }
      }
      // density parameters
      if (r < Q.pcr()) {
#pragma unroll
        for (int m = 0; m < NP; m++) {
          if (m < P.np) {
            gp[m] += (double)cp * D.cpa[m];
            gp[NP + m] += (double)cp * D.cpr[m];
            drA[m] += D.cpa[m];
            drR[m] += D.cpr[m];
          }
        }
      } else {
#pragma unroll
        for (int m = 0; m < NP; m++) {
          if (m < P.np) {
            const T d = Q.dp(m, r);
            if (d > T(0)) {
              const T d2 = d * d, pa = d2 * d, pr = T(3) * Q.ap(m) * d2;
              gp[m] += (double)(cp * pa - T(3) * cpp * d2);
              gp[NP + m] += (double)(cp * pr - T(6) * cpp * Q.ap(m) * d);
              drA[m] += (double)pa;
              drR[m] += (double)pr;
            }
          }
        }
      }
    }
    const double lam = -2.0 * fi * fi * fi * q;  // F''(rho_i) Q_i
#pragma unroll
    for (int m = 0; m < NP; m++) {
      gp[m] -= lam * drA[m];
      gp[NP + m] -= lam * drR[m];
    }
  }
  wave_reduce_all<2 * NV, 0>(gv);
  wave_reduce_all<2 * NP, 0>(gp);
  if (V.index >= 0 && (threadIdx.x & 63) == 0) {  // slots a_0..a_{nv-1}, r_0.., A_0..A_{np-1}, R_0..
    double *out = A.part_g + V.index;
    const size_t nt = A.ntile;
#pragma unroll
    for (int m = 0; m < NV; m++) {
      if (m < P.nv) {
        out[m * nt] = gv[m];
        out[(P.nv + m) * nt] = gv[NV + m];
      }
    }
#pragma unroll
    for (int m = 0; m < NP; m++) {
      if (m < P.np) {
        out[(2 * P.nv + m) * nt] = gp[m];
        out[(2 * P.nv + P.np + m) * nt] = gp[NP + m];
      }
    }
  }
}

// Gradient slots summed over tiles and the loss over cells, in a fixed order:
// block (k, y) folds part y of gridDim.y of slot k (k == nslot, launched only
// for the loss: the per-cell losses).  One part writes the results itself,
// several go through stage and k_grad_out.
__global__ void __launch_bounds__(256) k_fold(const double *part_g, const double *out_loss, int ntile, int ncell,
                                              int nslot, double *stage, double *grad, double *loss) {
  __shared__ double red[4];
  const int k = blockIdx.x, parts = gridDim.y;
  const double *src = k < nslot ? part_g + (size_t)k * ntile : out_loss;
  const int n = k < nslot ? ntile : ncell;
  const int lo = (int)((long)n * blockIdx.y / parts), hi = (int)((long)n * (blockIdx.y + 1) / parts);
  double s = 0.0;
  for (int i = lo + (int)threadIdx.x; i < hi; i += 256) s += src[i];
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    s = ((red[0] + red[1]) + red[2]) + red[3];
    if (parts > 1) stage[k * FOLD_CHUNKS + blockIdx.y] = s;
    else if (k < nslot) grad[k] = s;
    else *loss = s;
  }
}
__global__ void __launch_bounds__(64) k_grad_out(const double *stage, int parts, int nslot, int nval, double *grad,
                                                 double *loss) {
  const int k = threadIdx.x;
  if (k >= nval) return;
  double s = 0.0;
  for (int y = 0; y < parts; y++) s += stage[k * FOLD_CHUNKS + y];
  if (k < nslot) grad[k] = s;
  else *loss = s;
}
}  // namespace

// One captured launch sequence (forward, or loss + gradient).
struct GraphSlot {
  hipGraph_t graph;
  hipGraphExec_t gexec;
  bool valid;
  bool used;  // launched since the last change (captured from the second time on)
};

struct mdk_batch {
  int ncell, natom, precision, maxnb;
  hipStream_t stream;
  int device;
  // sub-cell plan: tiles, cells and candidate records for grid width rgrid
  int ntile, nrec;
  double rgrid;
  CellMeta *meta;
  Tile *tiles;
  int2 *rsrc;
  int *subc, *est, *perm, *numn, *flags, *flags_host, *flags_map;
  int4 *nbr;
  double *box, *s, *rho, *part, *out_e, *out_w, *out_f, *daf;
  float4 *rec;
  double4 *pos4;
  float4 *p4f;
  float *fetab;  // FP32 interval table of the current knots (when they admit one)
  bool fe_ok;
  // adjoint buffers: targets, product seeds, force seeds (sorted order),
  // gradient partials per tile, losses per cell, reduced results (host-mapped)
  double *e_tgt, *f_tgt, *e_seed, *f_seed, *ecell, *part_g, *out_loss, *stage, *res_host, *res_map;
  double4 *gvec;
  std::vector<int> h_off;                // first atom of each cell
  std::vector<double> h_box, h_s;        // boxes; wrapped fractional positions, caller's order
  PotDev pot;
  GradDev gd;
  hostpot::Knots knots;
  bool pot_set, targets_set, list_valid;
  int block, wg_per_cu;
  bool use_graph;
  GraphSlot g_eval, g_grad;
  double rc;
  double min_width;  // narrowest perpendicular cell width: the minimum image needs 2 rc below it
};

namespace {

template <typename T, int BLOCK, bool FE, bool TAB>
void launch_forward(mdk_batch *b, const BatchArgs &A, bool loss) {
  const int tg = (A.ntile + BLOCK / TILE - 1) / (BLOCK / TILE), cg = (A.ncell + 3) / 4;
  k_pack<T><<<(A.nrec + 255) / 256, 256, 0, b->stream>>>(A);
  k_list<T, BLOCK, FE><<<tg, BLOCK, 0, b->stream>>>(A, b->pot);
  if (loss) {
    k_force<T, BLOCK, FE, TAB, true><<<tg, BLOCK, 0, b->stream>>>(A, b->pot);
    k_cells<true><<<cg, 256, 0, b->stream>>>(A);
  } else {
    k_force<T, BLOCK, FE, TAB, false><<<tg, BLOCK, 0, b->stream>>>(A, b->pot);
    k_cells<false><<<cg, 256, 0, b->stream>>>(A);
  }
}
template <int BLOCK>
void forward_block(mdk_batch *b, const BatchArgs &A, bool loss) {
  const bool fe = b->pot.nv == MDK_FE_NV && b->pot.np == MDK_FE_NP;
  if (b->precision == MDK_PREC_FP64) {
    if (fe) launch_forward<double, BLOCK, true, false>(b, A, loss);
    else launch_forward<double, BLOCK, false, false>(b, A, loss);
  } else if (fe && b->fe_ok) {
    launch_forward<float, BLOCK, true, true>(b, A, loss);
  } else if (fe) {
    launch_forward<float, BLOCK, true, false>(b, A, loss);
  } else {
    launch_forward<float, BLOCK, false, false>(b, A, loss);
  }
}
void forward(mdk_batch *b, const BatchArgs &A, bool loss) {
  switch (b->block) {
    case 64: forward_block<64>(b, A, loss); break;
    case 128: forward_block<128>(b, A, loss); break;
    case 512: forward_block<512>(b, A, loss); break;
    default: forward_block<256>(b, A, loss); break;
  }
}
template <typename T, int BLOCK>
void adjoint_block(mdk_batch *b, const BatchArgs &A, const double *seed) {
  const int tg = (A.ntile + BLOCK / TILE - 1) / (BLOCK / TILE);
  if (b->pot.nv == MDK_FE_NV && b->pot.np == MDK_FE_NP)
    k_adjoint<T, BLOCK, MDK_FE_NV, MDK_FE_NP><<<tg, BLOCK, 0, b->stream>>>(A, b->pot, b->gd, seed);
  else
    k_adjoint<T, BLOCK, MDK_MAXV, MDK_MAXP><<<tg, BLOCK, 0, b->stream>>>(A, b->pot, b->gd, seed);
}
template <typename T>
void adjoint(mdk_batch *b, const BatchArgs &A, const double *seed) {
  switch (b->block) {
    case 64: adjoint_block<T, 64>(b, A, seed); break;
    case 128: adjoint_block<T, 128>(b, A, seed); break;
    case 512: adjoint_block<T, 512>(b, A, seed); break;
    default: adjoint_block<T, 256>(b, A, seed); break;
  }
}

BatchArgs args_of(mdk_batch *b) {
  BatchArgs A;
  A.ncell = b->ncell; A.natom = b->natom; A.ntile = b->ntile; A.nrec = b->nrec; A.maxnb = b->maxnb;
  A.meta = b->meta; A.tiles = b->tiles; A.box = b->box; A.subc = b->subc; A.est = b->est; A.rsrc = b->rsrc;
  A.s = b->s; A.perm = b->perm; A.rec = b->rec; A.pos4 = b->pos4; A.p4f = b->p4f; A.daf = b->daf; A.nbr = b->nbr;
  A.numn = b->numn; A.rho = b->rho; A.part = b->part; A.out_e = b->out_e; A.out_w = b->out_w; A.out_f = b->out_f;
  A.flags = b->flags; A.flags_out = b->flags_map;
  A.rc = b->rc;
  A.fetab = b->fetab;
  A.e_in = b->e_tgt; A.f_in = b->f_tgt; A.gvec = b->gvec; A.ecell = b->ecell; A.part_g = b->part_g;
  A.out_loss = b->out_loss; A.f_weight = 0.1 / (double)b->natom;
  return A;
}

int ngrad_of(const mdk_batch *b) { return 2 * b->knots.nv + 2 * b->knots.np; }

int launch_status() {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return berr(MDK_ERR_HIP, "batch launch: %s", hipGetErrorString(e));
  return MDK_OK;
}

int enqueue(mdk_batch *b) {
  forward(b, args_of(b), false);
  return launch_status();
}

// loss + gradient (vjp = false, from the targets) or the vector-Jacobian
// product with the seeds e_seed/f_seed (vjp = true, on the last forward's list
// and F'), then the fixed-order sums into grad[0..ngrad) and, for the loss, *loss
int enqueue_grad(mdk_batch *b, bool vjp, double *grad, double *loss) {
  BatchArgs A = args_of(b);
  const double *seed = b->ecell;
  if (vjp) {
    A.f_in = b->f_seed;
    seed = b->e_seed;
    k_seeds<<<(A.natom + 255) / 256, 256, 0, b->stream>>>(A);
  } else {
    forward(b, A, true);
  }
  if (b->precision == MDK_PREC_FP64) adjoint<double>(b, A, seed);
  else adjoint<float>(b, A, seed);
  // about 2048 tile values per first-stage block
  const int ng = ngrad_of(b), nval = ng + (vjp ? 0 : 1);
  const int parts = std::min(FOLD_CHUNKS, 1 + A.ntile / 2048);
  k_fold<<<dim3(nval, parts), 256, 0, b->stream>>>(b->part_g, b->out_loss, A.ntile, A.ncell, ng, b->stage, grad, loss);
  if (parts > 1) k_grad_out<<<1, 64, 0, b->stream>>>(b->stage, parts, ng, nval, grad, loss);
  return launch_status();
}

void drop_slot(GraphSlot &g) {
  if (g.valid) {
    hipGraphExecDestroy(g.gexec);
    hipGraphDestroy(g.graph);
    g.valid = false;
  }
  g.used = false;
}

void drop_graph(mdk_batch *b) {
  drop_slot(b->g_eval);
  drop_slot(b->g_grad);
}

// Captures the launches of enqueue (grad = false) or of the loss + gradient
// (grad = true) into a graph slot.
int capture(mdk_batch *b, bool grad) {
  GraphSlot &gs = grad ? b->g_grad : b->g_eval;
  drop_slot(gs);
  BCK(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
  int rc = grad ? enqueue_grad(b, false, b->res_map, b->res_map + ngrad_of(b)) : enqueue(b);
  hipGraph_t g = nullptr;
  hipError_t e = hipStreamEndCapture(b->stream, &g);
  if (rc != MDK_OK) {
    if (g) hipGraphDestroy(g);
    return rc;
  }
  if (e != hipSuccess) return berr(MDK_ERR_HIP, "capture: %s", hipGetErrorString(e));
  e = hipGraphInstantiate(&gs.gexec, g, nullptr, nullptr, 0);
  if (e != hipSuccess) {
    hipGraphDestroy(g);
    return berr(MDK_ERR_HIP, "graph instantiate: %s", hipGetErrorString(e));
  }
  gs.graph = g;
  gs.valid = true;
  return MDK_OK;
}

// Runs one of the two sequences: by its graph where it was launched before
// with the same potential and launch settings, else directly (a fit changes
// the potential before every launch, and a capture costs more than the six
// launches it replaces).
int launch_sequence(mdk_batch *b, bool grad) {
  GraphSlot &gs = grad ? b->g_grad : b->g_eval;
  if (b->use_graph && gs.used && !gs.valid) {
    int rc = capture(b, grad);
    if (rc != MDK_OK) return rc;
  }
  if (b->use_graph && gs.valid) {
    BCK(hipGraphLaunch(gs.gexec, b->stream));
  } else {
    int rc = grad ? enqueue_grad(b, false, b->res_map, b->res_map + ngrad_of(b)) : enqueue(b);
    if (rc != MDK_OK) return rc;
    gs.used = true;
  }
  b->list_valid = true;
  return MDK_OK;
}

void free_plan(mdk_batch *b) {
  void **p[] = {(void **)&b->meta, (void **)&b->tiles, (void **)&b->rsrc, (void **)&b->subc, (void **)&b->est,
                (void **)&b->perm, (void **)&b->s,     (void **)&b->rec,  (void **)&b->nbr,  (void **)&b->part,
                (void **)&b->part_g};
  for (void **q : p) {
    if (*q) hipFree(*q);
    *q = nullptr;
  }
  b->rgrid = 0.0;
}

// Perpendicular widths of a cell's box.
void widths(const double *B, double (&w)[3]) {
  const double vol = fabs(TT(B, 1, 1) * (TT(B, 2, 2) * TT(B, 3, 3) - TT(B, 2, 3) * TT(B, 3, 2)) +
                          TT(B, 2, 1) * (TT(B, 3, 2) * TT(B, 1, 3) - TT(B, 1, 2) * TT(B, 3, 3)) +
                          TT(B, 3, 1) * (TT(B, 1, 2) * TT(B, 2, 3) - TT(B, 2, 2) * TT(B, 1, 3)));
  for (int d = 0; d < 3; d++) {
    const double *u = B + 3 * ((d + 1) % 3), *v = B + 3 * ((d + 2) % 3);
    const double cx = u[1] * v[2] - u[2] * v[1], cy = u[2] * v[0] - u[0] * v[2], cz = u[0] * v[1] - u[1] * v[0];
    w[d] = vol / sqrt(cx * cx + cy * cy + cz * cz);
  }
}

// Sub-cells at least rgrid wide, atoms sorted by sub-cell, tiles and candidate
// records of every cell.
int plan(mdk_batch *b, double rgrid) {
  const int ncell = b->ncell, natom = b->natom;
  std::vector<CellMeta> meta(ncell);
  std::vector<Tile> tiles;
  std::vector<int> subc(natom), perm(natom), est;
  std::vector<int2> rsrc;
  std::vector<double> s(3 * (size_t)natom);
  rsrc.reserve((size_t)natom + natom / 2);
  tiles.reserve(natom / TILE + ncell);
  std::vector<int> key, start, fill;
  for (int c = 0; c < ncell; c++) {
    double w[3];
    widths(&b->h_box[9 * (size_t)c], w);
    int g[3];
    for (int d = 0; d < 3; d++) {
      const int k = (int)floor(std::min(w[d] / rgrid, 64.0));
      g[d] = k < 3 ? 1 : k;
    }
    const int a0 = b->h_off[c], nc = b->h_off[c + 1] - a0, nsc = g[0] * g[1] * g[2];
    CellMeta &m = meta[c];
    double ext = 0.0;
    for (const double *B = &b->h_box[9 * (size_t)c], *r = B; r < B + 3; r++)
      ext = std::max(ext, fabs(r[0]) + fabs(r[3]) + fabs(r[6]));
    m = CellMeta{a0, nc, (int)tiles.size(), (nc + TILE - 1) / TILE, g[0], g[1], g[2],
                 g[0] >= 3 && g[1] >= 3 && g[2] >= 3 ? 1 : 0, (int)est.size(), (int)rsrc.size(), (float)ext, 0};
    for (int i = 0; i < nc; i += TILE) tiles.push_back(Tile{c, a0 + i, std::min(TILE, nc - i), i});
    key.resize(nc);
    start.assign(nsc + 1, 0);
    for (int i = 0; i < nc; i++) {
      int q[3];
      for (int d = 0; d < 3; d++)
        q[d] = std::max(0, std::min((int)(b->h_s[3 * ((size_t)a0 + i) + d] * g[d]), g[d] - 1));
      key[i] = q[0] + g[0] * (q[1] + g[1] * q[2]);
      start[key[i] + 1]++;
    }
    for (int k = 0; k < nsc; k++) start[k + 1] += start[k];
    fill.assign(start.begin(), start.end() - 1);
    for (int i = 0; i < nc; i++) {
      const size_t k = (size_t)a0 + fill[key[i]]++;
      for (int d = 0; d < 3; d++) s[3 * k + d] = b->h_s[3 * ((size_t)a0 + i) + d];
      perm[k] = a0 + i;
      subc[k] = key[i];
    }
    auto add = [&](int sub, int ghost) {
      est.push_back((int)rsrc.size() - m.rec0);
      for (int i = start[sub]; i < start[sub + 1]; i++) rsrc.push_back(make_int2(c, i | (ghost << 28)));
    };
    for (int yz = 0; yz < g[1] * g[2]; yz++) {
      if (m.rows) add(g[0] * yz + g[0] - 1, 1);
      for (int x = 0; x < g[0]; x++) add(g[0] * yz + x, 0);
      if (m.rows) add(g[0] * yz, 2);
    }
    est.push_back((int)rsrc.size() - m.rec0);
  }
  BCK(hipStreamSynchronize(b->stream));  // launches in flight still read the previous plan
  free_plan(b);
  b->ntile = (int)tiles.size();
  b->nrec = (int)rsrc.size();
#define PALLOC(p, count)                                                                                        \
  do {                                                                                                          \
    if (hipMalloc((void **)&(p), sizeof(*(p)) * (size_t)(count)) != hipSuccess) {                               \
      free_plan(b);                                                                                             \
      return berr(MDK_ERR_HIP, "hipMalloc %zu bytes failed", sizeof(*(p)) * (size_t)(count));                   \
    }                                                                                                           \
  } while (0)
  PALLOC(b->meta, ncell);
  PALLOC(b->tiles, b->ntile);
  PALLOC(b->rsrc, b->nrec);
  PALLOC(b->subc, natom);
  PALLOC(b->est, est.size());
  PALLOC(b->perm, natom);
  PALLOC(b->s, 3 * (size_t)natom);
  PALLOC(b->rec, (size_t)b->nrec + 4);  // a walk loads up to three records past its last candidate
  PALLOC(b->nbr, (size_t)b->ntile * TILE * (b->maxnb / 4));
  PALLOC(b->part, (size_t)b->ntile * NPART_TILE);
  PALLOC(b->part_g, (size_t)b->ntile * NGRAD_SLOTS);
#undef PALLOC
  hipMemcpy(b->meta, meta.data(), sizeof(CellMeta) * ncell, hipMemcpyHostToDevice);
  hipMemcpy(b->tiles, tiles.data(), sizeof(Tile) * tiles.size(), hipMemcpyHostToDevice);
  hipMemcpy(b->rsrc, rsrc.data(), sizeof(int2) * rsrc.size(), hipMemcpyHostToDevice);
  hipMemcpy(b->subc, subc.data(), sizeof(int) * natom, hipMemcpyHostToDevice);
  hipMemcpy(b->est, est.data(), sizeof(int) * est.size(), hipMemcpyHostToDevice);
  hipMemcpy(b->perm, perm.data(), sizeof(int) * natom, hipMemcpyHostToDevice);
  hipMemset(b->rec + b->nrec, 0, sizeof(float4) * 4);
  if (hipMemcpy(b->s, s.data(), sizeof(double) * 3 * (size_t)natom, hipMemcpyHostToDevice) != hipSuccess) {
    free_plan(b);
    return berr(MDK_ERR_HIP, "upload failed");
  }
  b->rgrid = rgrid;
  return MDK_OK;
}

}  // namespace

extern "C" const char *mdk_batch_last_error(void) { return b_err; }

extern "C" int mdk_batch_destroy(void *h) {
  mdk_batch *b = (mdk_batch *)h;
  if (!b) return MDK_OK;
  if (b->stream) hipStreamSynchronize(b->stream);
  drop_graph(b);
  free_plan(b);
  void *p[] = {b->numn, b->flags, b->box, b->rho, b->out_e, b->out_w, b->out_f, b->daf, b->pos4, b->p4f,
               b->fetab, b->e_tgt, b->f_tgt, b->e_seed, b->f_seed, b->gvec, b->ecell, b->out_loss, b->stage};
  for (void *q : p)
    if (q) hipFree(q);
  if (b->flags_host) hipHostFree(b->flags_host);
  if (b->res_host) hipHostFree(b->res_host);
  if (b->stream) hipStreamDestroy(b->stream);
  delete b;
  return MDK_OK;
}

// Cells: natoms[c] atoms each, boxes 9 doubles per cell (column-major, columns
// are cell vectors), s = 3 fractional coordinates per atom, cells concatenated.
// The sub-cell plan is made by mdk_batch_set_potential, which knows the range.
extern "C" int mdk_batch_create(void **handle, int ncell, const int *natoms, const double *boxes,
                                const double *s, int precision) {
  if (!handle || ncell < 1 || !natoms || !boxes || !s) return berr(MDK_ERR_BAD_ARG, "bad batch arguments");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return berr(MDK_ERR_NO_DEVICE, "no HIP device");
  mdk_batch *b = new mdk_batch();
  b->ncell = ncell;
  b->precision = precision;
  b->maxnb = 48;
  b->block = 256;
  b->wg_per_cu = 4;
  b->use_graph = true;
  hipGetDevice(&b->device);
  b->h_off.assign(ncell + 1, 0);
  b->min_width = 1e300;
  for (int c = 0; c < ncell; c++) {
    if (natoms[c] < 1) {
      delete b;
      return berr(MDK_ERR_BAD_ARG, "cell %d has no atoms", c);
    }
    b->h_off[c + 1] = b->h_off[c] + natoms[c];
    double w[3];
    widths(boxes + 9 * (size_t)c, w);
    for (double x : w) b->min_width = std::min(b->min_width, x);
  }
  const int natom = b->h_off[ncell];
  b->natom = natom;
  b->h_box.assign(boxes, boxes + 9 * (size_t)ncell);
  b->h_s.resize(3 * (size_t)natom);
  for (size_t k = 0; k < 3 * (size_t)natom; k++) {
    double v = s[k] - floor(s[k]);
    if (v >= 1.0) v = 0.0;
    b->h_s[k] = v;
  }
  b->rc = 3.72645;  // replaced by the potential's outermost knot in set_potential
  const bool f64 = precision == MDK_PREC_FP64;
  int rc = MDK_OK;
#define BALLOC(p, bytes)                                                                \
  do {                                                                                  \
    if (hipMalloc((void **)&(p), (bytes)) != hipSuccess) {                              \
      rc = berr(MDK_ERR_HIP, "hipMalloc %zu bytes failed", (size_t)(bytes));            \
      goto fail;                                                                        \
    }                                                                                   \
  } while (0)
  if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess) {
    rc = berr(MDK_ERR_HIP, "stream create failed");
    goto fail;
  }
  BALLOC(b->box, sizeof(double) * 9 * (size_t)ncell);
  if (f64) {
    BALLOC(b->pos4, sizeof(double4) * (size_t)natom);
  } else {
    BALLOC(b->p4f, sizeof(float4) * (size_t)natom);
    BALLOC(b->daf, sizeof(double) * (size_t)natom);
  }
  BALLOC(b->fetab, sizeof(float) * MDK_FE_TAB);
  BALLOC(b->numn, sizeof(int) * (size_t)natom);
  BALLOC(b->rho, sizeof(double) * (size_t)natom);
  BALLOC(b->out_e, sizeof(double) * (size_t)ncell);
  BALLOC(b->out_w, sizeof(double) * 6 * (size_t)ncell);
  BALLOC(b->out_f, sizeof(double) * 3 * (size_t)natom);
  BALLOC(b->e_tgt, sizeof(double) * (size_t)ncell);
  BALLOC(b->f_tgt, sizeof(double) * 3 * (size_t)natom);
  BALLOC(b->e_seed, sizeof(double) * (size_t)ncell);
  BALLOC(b->f_seed, sizeof(double) * 3 * (size_t)natom);
  BALLOC(b->gvec, sizeof(double4) * (size_t)natom);
  BALLOC(b->ecell, sizeof(double) * (size_t)ncell);
  BALLOC(b->out_loss, sizeof(double) * (size_t)ncell);
  BALLOC(b->stage, sizeof(double) * (NGRAD_SLOTS + 1) * FOLD_CHUNKS);
  BALLOC(b->flags, sizeof(int) * 4);
  if (hipHostMalloc((void **)&b->flags_host, sizeof(int) * 4, hipHostMallocMapped) != hipSuccess ||
      hipHostGetDevicePointer((void **)&b->flags_map, b->flags_host, 0) != hipSuccess ||
      hipHostMalloc((void **)&b->res_host, sizeof(double) * (NGRAD_SLOTS + 1), hipHostMallocMapped) != hipSuccess ||
      hipHostGetDevicePointer((void **)&b->res_map, b->res_host, 0) != hipSuccess) {
    rc = berr(MDK_ERR_HIP, "mapped host buffer failed");
    goto fail;
  }
  memset(b->flags_host, 0, sizeof(int) * 4);
  hipMemset(b->flags, 0, sizeof(int) * 4);
  hipMemset(b->numn, 0, sizeof(int) * (size_t)natom);
  if (hipMemcpy(b->box, boxes, sizeof(double) * 9 * (size_t)ncell, hipMemcpyHostToDevice) != hipSuccess) {
    rc = berr(MDK_ERR_HIP, "upload failed");
    goto fail;
  }
  *handle = b;
  return MDK_OK;
fail:
  mdk_batch_destroy(b);
  return rc;
#undef BALLOC
}

extern "C" int mdk_batch_set_potential(void *h, int nv, const double *av, const double *rv, int np,
                                       const double *ap, const double *rp) {
  mdk_batch *b = (mdk_batch *)h;
  if (!b || nv < 1 || nv > MDK_MAXV || np < 1 || np > MDK_MAXP) return berr(MDK_ERR_BAD_ARG, "bad potential");
  hostpot::Knots &k = b->knots;
  memset(&k, 0, sizeof(k));
  k.nv = nv;
  k.np = np;
  for (int i = 0; i < nv; i++) { k.av[i] = av[i]; k.rv[i] = rv[i]; }
  for (int i = 0; i < np; i++) { k.ap[i] = ap[i]; k.rp[i] = rp[i]; }
  hostpot::set_up(k);
  const double rint = hostpot::fill_potdev(b->pot, k);
  hostpot::grad_consts(k, b->gd);
  // the FP32 form's interval table of V, V', phi' (knot sums where the knots
  // do not admit one); launches in flight still read the previous table
  float tab[MDK_FE_TAB];
  b->fe_ok = nv == MDK_FE_NV && np == MDK_FE_NP && b->precision != MDK_PREC_FP64 &&
             hostpot::build_fe_table(k, tab, b->pot.fe_binh, b->pot.fe_binc);
  if (b->fe_ok) {
    if (hipStreamSynchronize(b->stream) != hipSuccess ||
        hipMemcpyAsync(b->fetab, tab, sizeof(tab), hipMemcpyHostToDevice, b->stream) != hipSuccess ||
        hipStreamSynchronize(b->stream) != hipSuccess)
      return berr(MDK_ERR_HIP, "interval table upload failed");
  }
  if (rint > 4.5) return berr(MDK_ERR_BAD_ARG, "knots beyond 4.5 A are not supported by the batch grid");
  if (2.0 * rint >= b->min_width)
    return berr(MDK_ERR_BAD_ARG, "a cell is narrower (%.3f A) than twice the interaction range", b->min_width);
  // sub-cells as narrow as the list radius allows (a walk tests 27 of them per
  // atom: with cells sized for a 4.5 A range, 1.7 times as many candidates),
  // with 2 % to spare, so that the knots of a fit move without a new plan
  if (b->rgrid < rint + 1e-4 || b->rgrid > 1.25 * rint) {
    const int rc = plan(b, 1.02 * rint);
    if (rc != MDK_OK) {
      b->pot_set = false;
      return rc;
    }
  }
  b->rc = rint;
  b->pot_set = true;
  b->list_valid = false;
  drop_graph(b);  // the potential is a kernel argument of the captured launches
  return MDK_OK;
}

extern "C" int mdk_batch_config(void *h, int block, int wg_per_cu, int use_graph) {
  mdk_batch *b = (mdk_batch *)h;
  if (!b) return berr(MDK_ERR_BAD_ARG, "null handle");
  if (block != 64 && block != 128 && block != 256 && block != 512) return berr(MDK_ERR_BAD_ARG, "block must be 64..512");
  if (wg_per_cu < 1 || wg_per_cu > 32) return berr(MDK_ERR_BAD_ARG, "wg_per_cu out of range");
  b->block = block;
  b->wg_per_cu = wg_per_cu;
  b->use_graph = use_graph != 0;
  drop_graph(b);
  return MDK_OK;
}

extern "C" int mdk_batch_evaluate(void *h) {
  mdk_batch *b = (mdk_batch *)h;
  if (!b || !b->pot_set) return berr(MDK_ERR_STATE, "batch potential not set");
  return launch_sequence(b, false);
}

extern "C" int mdk_batch_synchronize(void *h) {
  mdk_batch *b = (mdk_batch *)h;
  if (!b) return berr(MDK_ERR_BAD_ARG, "null handle");
  BCK(hipStreamSynchronize(b->stream));
  const int over = *(volatile int *)b->flags_host;
  if (over) return berr(MDK_ERR_NBR_OVERFLOW, "batch neighbour capacity %d exceeded (%d)", b->maxnb, over);
  return MDK_OK;
}

// energy[ncell] (eV), virial[6*ncell] = sum over pairs of r r^T fp (xx yy zz xy xz yz;
// stress = -virial/volume), forces[3*natom] Cartesian (eV/A), rho[natom]; any may be NULL.
extern "C" int mdk_batch_results(void *h, double *energy, double *virial, double *forces, double *rho) {
  mdk_batch *b = (mdk_batch *)h;
  if (!b) return berr(MDK_ERR_BAD_ARG, "null handle");
  int rc = mdk_batch_synchronize(h);
  if (rc != MDK_OK) return rc;
  if (energy) BCK(hipMemcpy(energy, b->out_e, sizeof(double) * b->ncell, hipMemcpyDeviceToHost));
  if (virial) BCK(hipMemcpy(virial, b->out_w, sizeof(double) * 6 * (size_t)b->ncell, hipMemcpyDeviceToHost));
  if (forces) BCK(hipMemcpy(forces, b->out_f, sizeof(double) * 3 * (size_t)b->natom, hipMemcpyDeviceToHost));
  if (rho) BCK(hipMemcpy(rho, b->rho, sizeof(double) * b->natom, hipMemcpyDeviceToHost));
  return MDK_OK;
}

// Autotuner: times every block size with HIP events (best of `reps` replays)
// and keeps the fastest; returns the choice and its time.  Workgroups per CU
// follow from the block's registers (the grid covers every tile), so the
// setting is returned as it is.
extern "C" int mdk_batch_tune(void *h, int reps, int *best_block, int *best_wgpc, double *best_ms) {
  mdk_batch *b = (mdk_batch *)h;
  if (!b || !b->pot_set) return berr(MDK_ERR_STATE, "batch potential not set");
  hipEvent_t e0, e1;
  BCK(hipEventCreate(&e0));
  BCK(hipEventCreate(&e1));
  double best = 1e30;
  int bb = b->block;
  for (int bl : {128, 256, 512}) {
    b->block = bl;
    drop_graph(b);
    int rc = MDK_OK;
    for (int w = 0; w < 2 && rc == MDK_OK; w++) rc = mdk_batch_evaluate(h);  // warm-up (and capture)
    if (rc != MDK_OK) return rc;
    double t = 1e30;
    for (int r = 0; r < std::max(1, reps); r++) {
      BCK(hipEventRecord(e0, b->stream));
      rc = mdk_batch_evaluate(h);
      if (rc != MDK_OK) return rc;
      BCK(hipEventRecord(e1, b->stream));
      BCK(hipEventSynchronize(e1));
      float ms = 0.f;
      BCK(hipEventElapsedTime(&ms, e0, e1));
      t = std::min(t, (double)ms);
    }
    if (t < best) {
      best = t;
      bb = bl;
    }
  }
  hipEventDestroy(e0);
  hipEventDestroy(e1);
  b->block = bb;
  drop_graph(b);
  if (best_block) *best_block = bb;
  if (best_wgpc) *best_wgpc = b->wg_per_cu;
  if (best_ms) *best_ms = best;
  return mdk_batch_synchronize(h);
}

// Average time of `reps` replays (HIP events on the batch stream), ms.
extern "C" int mdk_batch_time(void *h, int reps, double *ms_avg) {
  mdk_batch *b = (mdk_batch *)h;
  if (!b || reps < 1) return berr(MDK_ERR_BAD_ARG, "bad arguments");
  hipEvent_t e0, e1;
  BCK(hipEventCreate(&e0));
  BCK(hipEventCreate(&e1));
  int rc = mdk_batch_evaluate(h);
  if (rc != MDK_OK) return rc;
  BCK(hipEventRecord(e0, b->stream));
  for (int r = 0; r < reps; r++) {
    rc = mdk_batch_evaluate(h);
    if (rc != MDK_OK) return rc;
  }
  BCK(hipEventRecord(e1, b->stream));
  BCK(hipEventSynchronize(e1));
  float ms = 0.f;
  BCK(hipEventElapsedTime(&ms, e0, e1));
  hipEventDestroy(e0);
  hipEventDestroy(e1);
  if (ms_avg) *ms_avg = ms / reps;
  return mdk_batch_synchronize(h);
}

extern "C" int mdk_batch_info(void *h, int *natom, int *block, int *wg_per_cu, long *pairs) {
  mdk_batch *b = (mdk_batch *)h;
  if (!b) return berr(MDK_ERR_BAD_ARG, "null handle");
  if (natom) *natom = b->natom;
  if (block) *block = b->block;
  if (wg_per_cu) *wg_per_cu = b->wg_per_cu;
  if (pairs) {
    std::vector<int> nn(b->natom);
    BCK(hipMemcpy(nn.data(), b->numn, sizeof(int) * b->natom, hipMemcpyDeviceToHost));
    long s = 0;
    for (int v : nn) s += v;
    *pairs = s;
  }
  return MDK_OK;
}

// ---------------------------------------------------------------------------
// Adjoint: d(loss)/d(knot parameters).  Gradient order: a_0..a_{nv-1},
// r_0..r_{nv-1}, A_0..A_{np-1}, R_0..R_{np-1} (2 nv + 2 np values).
// ---------------------------------------------------------------------------

// Targets of the loss: e_target[ncell] (eV) and f_target[3*natom] (Cartesian
// eV/A, the caller's atom order).
extern "C" int mdk_batch_set_targets(void *h, const double *e_target, const double *f_target) {
  mdk_batch *b = (mdk_batch *)h;
  if (!b || !e_target || !f_target) return berr(MDK_ERR_BAD_ARG, "bad arguments");
  BCK(hipMemcpyAsync(b->e_tgt, e_target, sizeof(double) * b->ncell, hipMemcpyHostToDevice, b->stream));
  BCK(hipMemcpyAsync(b->f_tgt, f_target, sizeof(double) * 3 * (size_t)b->natom, hipMemcpyHostToDevice,
                     b->stream));
  BCK(hipStreamSynchronize(b->stream));
  b->targets_set = true;
  return MDK_OK;
}

namespace {
int read_res(mdk_batch *b, int n, double *out) {
  int rc = mdk_batch_synchronize(b);
  if (rc != MDK_OK) return rc;
  for (int k = 0; k < n; k++) out[k] = ((volatile double *)b->res_host)[k];
  return MDK_OK;
}
int enqueue_loss_grad(mdk_batch *b) {
  if (!b->pot_set || !b->targets_set) return berr(MDK_ERR_STATE, "batch potential or targets not set");
  return launch_sequence(b, true);
}
}  // namespace

// loss = sum_c (E_c - E_t,c)^2 / N_c^2 + (0.1 / natom) sum_i |F_i - F_t,i|^2 and
// grad = d(loss)/d(knot parameters): the forward passes with the loss's seeds,
// the adjoint on their list and F', then a fixed-order reduction over tiles.
// Energies and forces of the forward part are left for mdk_batch_results.
extern "C" int mdk_batch_loss_grad(void *h, double *loss, double *grad) {
  mdk_batch *b = (mdk_batch *)h;
  if (!b) return berr(MDK_ERR_BAD_ARG, "null handle");
  int rc = enqueue_loss_grad(b);
  if (rc != MDK_OK) return rc;
  const int ng = ngrad_of(b);
  double r[NGRAD_SLOTS + 1];
  rc = read_res(b, ng + 1, r);
  if (rc != MDK_OK) return rc;
  if (grad) memcpy(grad, r, sizeof(double) * ng);
  if (loss) *loss = r[ng];
  return MDK_OK;
}

// Vector-Jacobian product: grad = sum_c dE[c] dE_c/dtheta + sum_i dF_i . dF_i/dtheta
// for seeds dE[ncell] and dF[3*natom] (Cartesian, caller's order), at the
// positions and potential of the last forward evaluation (mdk_batch_evaluate or
// mdk_batch_loss_grad; its neighbour list and F' are reused).
extern "C" int mdk_batch_vjp(void *h, const double *dE, const double *dF, double *grad) {
  mdk_batch *b = (mdk_batch *)h;
  if (!b || !dE || !dF || !grad) return berr(MDK_ERR_BAD_ARG, "bad arguments");
  if (!b->pot_set || !b->list_valid)
    return berr(MDK_ERR_STATE, "mdk_batch_vjp needs a forward evaluation with the current potential");
  BCK(hipMemcpyAsync(b->e_seed, dE, sizeof(double) * b->ncell, hipMemcpyHostToDevice, b->stream));
  BCK(hipMemcpyAsync(b->f_seed, dF, sizeof(double) * 3 * (size_t)b->natom, hipMemcpyHostToDevice,
                     b->stream));
  int rc = enqueue_grad(b, true, b->res_map, nullptr);
  if (rc != MDK_OK) return rc;
  return read_res(b, ngrad_of(b), grad);
}

// mdk_batch_loss_grad into caller device memory without allocating: the
// kernels are those of mdk_batch_loss_grad (no graph) on the handle's own
// buffers, so the results agree bit for bit.
extern "C" int mdk_batch_loss_grad_noalloc(void *h, double *loss, double *grad) {
  mdk_batch *b = (mdk_batch *)h;
  if (!b || !loss || !grad) return berr(MDK_ERR_BAD_ARG, "bad arguments");
  if (!b->pot_set || !b->targets_set) return berr(MDK_ERR_STATE, "batch potential or targets not set");
  if (b->ncell > MDK_NOALLOC_MAX_CELLS)
    return berr(MDK_ERR_BAD_ARG, "%d cells exceed the no-allocation limit of %d cells", b->ncell,
                MDK_NOALLOC_MAX_CELLS);
  const int rc = enqueue_grad(b, false, grad, loss);
  b->list_valid = true;
  return rc;
}

// Average time of `reps` loss + gradient launches (HIP events on the batch stream), ms.
extern "C" int mdk_batch_time_loss_grad(void *h, int reps, double *ms_avg) {
  mdk_batch *b = (mdk_batch *)h;
  if (!b || reps < 1) return berr(MDK_ERR_BAD_ARG, "bad arguments");
  hipEvent_t e0, e1;
  BCK(hipEventCreate(&e0));
  BCK(hipEventCreate(&e1));
  int rc = enqueue_loss_grad(b);
  if (rc != MDK_OK) return rc;
  BCK(hipEventRecord(e0, b->stream));
  for (int r = 0; r < reps; r++) {
    rc = enqueue_loss_grad(b);
    if (rc != MDK_OK) return rc;
  }
  BCK(hipEventRecord(e1, b->stream));
  BCK(hipEventSynchronize(e1));
  float ms = 0.f;
  BCK(hipEventElapsedTime(&ms, e0, e1));
  hipEventDestroy(e0);
  hipEventDestroy(e1);
  if (ms_avg) *ms_avg = ms / reps;
  return mdk_batch_synchronize(h);
}
