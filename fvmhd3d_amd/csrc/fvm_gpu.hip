// HIP implementation of the fvm_gpu.h C ABI: the reference-order ("parity")
// kernels of the Voronoi-face pipeline and the context that owns their device
// buffers.
//
// Device layout: every per-cell field is structure-of-arrays, component k of
// cell i at [k*np + i]; per-face records and geometry are rows.  Fields the
// reference stores as float (Fluid_flt, fvec3, FluidD) use the storage type S
// (float as shipped, double for the all-FP64 build); everything else is double.
//
// Sums that the reference accumulates face by face (flux scatter, area
// closure, predictor) run per cell over a CSR list of its active face-ends
// sorted by face_active_list position, i.e. in the reference's own order, so
// the results do not depend on scheduling (no atomics on data).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/fvm_gpu.h"
#include "fvm_internal.h"
#include "fvm_physics.h"

using namespace fvm;

namespace fvm {

// ---------------------------------------------------------------------------
// field table
// ---------------------------------------------------------------------------
enum { K_DOUBLE = 0, K_STORE = 1, K_INT = 2 };
struct FieldInfo {
  int width, kind;
};
static const FieldInfo kFields[FVM_NFIELDS] = {
    {10, K_DOUBLE},  // W
    {10, K_STORE},   // GRAD_X
    {10, K_STORE},   // GRAD_Y
    {10, K_STORE},   // GRAD_Z
    {10, K_STORE},   // DWDT
    {3, K_DOUBLE},   // POS
    {3, K_STORE},    // VEL
    {3, K_STORE},    // J
    {1, K_DOUBLE},   // TEND
    {1, K_INT},      // BND
    {1, K_INT},      // IS_NGB
    {1, K_INT},      // IS_ACTIVE
    {10, K_STORE},   // MINMAX_LO
    {10, K_STORE},   // MINMAX_HI
    {10, K_STORE},   // LIMITER
    {10, K_STORE},   // DU
    {3, K_STORE},    // DGRADPSI
    {1, K_STORE},    // DDIVB
    {10, K_DOUBLE},  // U
    {1, K_DOUBLE},   // MESH_VOLUME
    {1, K_DOUBLE},   // TBEG
    {3, K_DOUBLE},   // MESH_VEL
    {3, K_DOUBLE},   // ACC0
    {3, K_DOUBLE},   // ACC1
    {1, K_DOUBLE},   // DT_NEW
    {1, K_DOUBLE},   // DIVB
};

template <typename S> struct Cells {
  int np, nactive;
  double *w;
  S *x, *y, *z, *t;
  double *pos;
  S *vel, *J;
  double *tend;
  int *bnd, *is_ngb, *is_active;
  S *mm_lo, *mm_hi, *lim, *dU, *dgp, *ddivB;
  double *U, *mvol, *tbeg, *mvel, *acc0, *acc1, *dt_new, *divB;
};

struct MeshView {
  int nface, nfa;
  const int *s1, *s2;
  const double *cn;     // [nface][6]: centroid, n
  const int *coff, *cface;
  const int *cnbr;      // the other cell of each cell_face entry
  const double *cvol;
  const int *fact;        // face_active_list
  const int *soff, *sent; // per-cell active face-ends, entry = a<<1 | side
};

struct Phys {
  double gamma, courant, t_global;
  double L[3];
  int limiter;
};

#define FLD(p, k, i, n) (p)[(size_t)(k) * (size_t)(n) + (size_t)(i)]
// per-face records of the flux and predictor sweeps: one row of NREC doubles per
// active face, a whole 128-byte line, read by the 16 lanes of a cell at once
constexpr int NREC = 16;
#define REC(p, k, a) (p)[(size_t)(a) * NREC + (size_t)(k)]
// per-face geometry record: centroid[3] then area vector n[3]
#define GEO_C(M, d, f) (M).cn[(size_t)(f) * 6 + (size_t)(d)]
#define GEO_N(M, d, f) (M).cn[(size_t)(f) * 6 + 3 + (size_t)(d)]

__device__ __forceinline__ int gid() { return blockIdx.x * blockDim.x + threadIdx.x; }
// XCD-aware index of the cell and face sweeps: block b runs on XCD b mod 8
// and the 8 XCDs each take a contiguous eighth of the range, so neighbour
// gathers of nearby (Morton-ordered) cells share one XCD's L2.  gridDim.x is
// a multiple of 8 (LAUNCH_X); every thread still computes exactly one item.
__device__ __forceinline__ int xgid() {
  const int per = (int)gridDim.x >> 3;
  const int tile = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
  return tile * (int)blockDim.x + (int)threadIdx.x;
}

// Cell rows: what the face flux kernel reads of a cell, side by side.  Gathered
// from the fields (one array per variable), every value of a neighbour comes with
// a line of its own, and the launch is bound by the L2's bandwidth: 112 lines a
// face against 8.  2.1 M cells, 16.7 M faces, FP64: 3.29 ms, now 2.16 and 0.35 for
// the rows; the face states' W alone (predictor, reconstruction) gains too little
// for its rows (192 -> 165 + 14 and 291 -> 267 + 14 us on average).
// W[10], position[3], vel[3], then x[10], y[10], z[10], t[10]: 448 bytes.
constexpr int CROW_W = 16, CROW = 56;
__device__ __forceinline__ void ld_row(const double *__restrict__ p, int n, double *o) {
#pragma unroll
  for (int k = 0; k < n; k += 2) {
    const double2 v = *reinterpret_cast<const double2 *>(p + k);
    o[k] = v.x;
    o[k + 1] = v.y;
  }
}
// 64 cells a block through LDS: fields read 512 bytes at a time, all of a
// wavefront's in flight, rows written whole
template <typename S> __global__ void __launch_bounds__(256) k_cell_rows(Cells<S> C, double *__restrict__ rows) {
  __shared__ double tile[64 * (CROW + 1)];
  const int c0 = (int)blockIdx.x * 64, l = (int)threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int c = min(c0 + l, C.np - 1);
  double v[CROW / 4];
#pragma unroll
  for (int u = 0; u < CROW / 4; u++) {
    const int k = w + 4 * u;
    if (k < 10) v[u] = FLD(C.w, k, c, C.np);
    else if (k < 13) v[u] = FLD(C.pos, k - 10, c, C.np);
    else if (k < 16) v[u] = (double)FLD(C.vel, k - 13, c, C.np);
    else if (k < 26) v[u] = (double)FLD(C.x, k - 16, c, C.np);
    else if (k < 36) v[u] = (double)FLD(C.y, k - 26, c, C.np);
    else if (k < 46) v[u] = (double)FLD(C.z, k - 36, c, C.np);
    else v[u] = (double)FLD(C.t, k - 46, c, C.np);
  }
#pragma unroll
  for (int u = 0; u < CROW / 4; u++) tile[l * (CROW + 1) + w + 4 * u] = v[u];
  __syncthreads();
  const int m = min(64, C.np - c0) * CROW;
#pragma unroll
  for (int u = 0; u < 64 * CROW / 256; u++) {
    const int e = (int)threadIdx.x + 256 * u;
    if (e < m) rows[(size_t)c0 * CROW + e] = tile[e / CROW * (CROW + 1) + e % CROW];
  }
}

// ---------------------------------------------------------------------------
// layout conversion
// ---------------------------------------------------------------------------
template <typename S>
__global__ void k_aos_to_soa(const double *__restrict__ src, S *__restrict__ dst, int n, int width) {
  const int i = gid();
  if (i >= n) return;
  for (int k = 0; k < width; k++) FLD(dst, k, i, n) = (S)src[(size_t)i * width + k];
}
template <typename S>
__global__ void k_soa_to_aos(const S *__restrict__ src, double *__restrict__ dst, int n, int width) {
  const int i = gid();
  if (i >= n) return;
  for (int k = 0; k < width; k++) dst[(size_t)i * width + k] = (double)FLD(src, k, i, n);
}
__global__ void k_split_faces(const fvm_face *__restrict__ f, int n, int *s1, int *s2, double *cn) {
  const int i = gid();
  if (i >= n) return;
  const fvm_face F = f[i];
  s1[i] = F.s1;
  s2[i] = F.s2;
  for (int d = 0; d < 3; d++) {
    cn[(size_t)i * 6 + d] = F.centroid[d];
    cn[(size_t)i * 6 + 3 + d] = F.n[d];
  }
}

// ---------------------------------------------------------------------------
// The cell loops take 16 lanes per cell.  Reconstruction and slope limiter: the
// lanes first form the geometry of the cell's faces, one face a lane, into LDS,
// then lane k walks the faces for variable k in the reference's order.  Sums over
// face records (fluid update, predictor): lane k sums word k of the cell's
// records in the reference's order, a face-end being one 128-byte row.
// ---------------------------------------------------------------------------
// 16 lanes per cell.  Faces are staged FCH at a time: 24 covers all but the
// largest cells of random generators (15.5 faces on average), and the LDS
// leaves four blocks a CU.
constexpr int LC = 16, FCH = 24;
constexpr int GEO_D = 11;              // doubles of a staged face
constexpr int GEO_S = FCH * GEO_D + 3;  // of a cell's slice: four cells of a wavefront on distinct banks
__host__ __device__ constexpr long cell_lanes(long n) { return n * LC; }
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// largest of a per-cell count over the wavefront's four cells
__device__ __forceinline__ int wave_cells_max(int v) {
  v = max(v, __shfl_xor(v, 16));
  return __builtin_amdgcn_readfirstlane(max(v, __shfl_xor(v, 32)));
}

// System::computeReconstruction (computeReconstruction.cpp:42-264).
// Bound by the latency of its gathers (cell list -> face -> neighbour -> W) and
// of the FP64 geometry: with a face a lane each is paid once a cell instead of
// once a face, and the limiter's divisions once a variable.
// Measured (disk, 2.1 M cells, mean over the active sets of a 32-substep cycle): 295 us a
// launch; a thread per cell above 131,072 cells and a lane per (cell, variable)
// below took 925 and 117 us (521 us on average).  97,000 cells at once: 109 us
// against 284; 14,000 cells' active sets: 14.5 us against 57.
template <typename S>
__global__ void __launch_bounds__(256) k_reconstruction(Cells<S> C, MeshView M, Phys P) {
  __shared__ double geo[256 / LC][GEO_S];
  const int t = xgid();
  const int i = t / LC, k = t & (LC - 1), grp = (int)(threadIdx.x & 63) & ~(LC - 1);
  double *G = geo[threadIdx.x / LC];
  const int np = C.np;
  const bool live = i < C.nactive;
  const bool bad_cell = live && C.bnd[i] != NO_BOUNDARY;
  const int fb = live ? M.coff[i] : 0;
  const int deg = live && !bad_cell ? M.coff[i + 1] - fb : 0;
  const int wdeg = wave_cells_max(deg);
  const int kk = k < NF ? k : NF - 1;
  double Wi = 0.0, ipos[3] = {0.0, 0.0, 0.0};
  if (live) {
    Wi = FLD(C.w, kk, i, np);
    for (int d = 0; d < 3; d++) ipos[d] = FLD(C.pos, d, i, np);
  }

  double Wx = 0.0, Wy = 0.0, Wz = 0.0;
  S dmin = (S)0.0, dmax = (S)0.0;
  bool zero_flag = false;
  // geometry of faces [f0, f0 + FCH) of the list
  auto stage = [&](int f0) {
    for (int q = k; q < FCH; q += LC) {
      if (f0 + q >= deg) break;
      const int f = M.cface[fb + f0 + q];
      const int j = M.cnbr[fb + f0 + q];
      double cen[3];
      for (int d = 0; d < 3; d++) {
        double v = GEO_C(M, d, f) - ipos[d];
        if (v > 0.5 * P.L[d]) v -= P.L[d];
        else if (v < -0.5 * P.L[d]) v += P.L[d];
        cen[d] = v;
      }
      const double fn[3] = {GEO_N(M, 0, f), GEO_N(M, 1, f), GEO_N(M, 2, f)};
      const double area = dsqrt(fn[0] * fn[0] + fn[1] * fn[1] + fn[2] * fn[2]);
      const double cn = cen[0] * fn[0] + cen[1] * fn[1] + cen[2] * fn[2];
      const double sc = (cn < 0.0) ? (-1.0 / area) : (1.0 / area);
      const double normal[3] = {fn[0] * sc, fn[1] * sc, fn[2] * sc};
      const double dsh = cen[0] * normal[0] + cen[1] * normal[1] + cen[2] * normal[2];
      const double ids = (dsh != 0.0) ? 0.5 / dsh : 0.0;
      double *g = G + GEO_D * q;
      for (int d = 0; d < 3; d++) {
        const double drh = normal[d] * dsh;
        g[d] = drh;
        g[3 + d] = cen[d] - drh;
        g[6 + d] = cen[d];
      }
      g[9] = area * ids;
      g[10] = __longlong_as_double((long long)j);
      const int bj = C.bnd[j];
      zero_flag = zero_flag || (bj != NO_BOUNDARY && bj != INFLOW);
    }
  };

  for (int f0 = 0; f0 < wdeg; f0 += FCH) {
    if (f0 > 0) wave_sync();  // the last chunk is read
    stage(f0);
    wave_sync();
    const int n = min(deg - f0, FCH);
    // four neighbours' values in flight
    for (int q0 = 0; q0 < n; q0 += 4) {
      double wj[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int j = q0 + u < n ? (int)__double_as_longlong(G[GEO_D * (q0 + u) + 10]) : i;
        wj[u] = FLD(C.w, kk, j, np);
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
        if (q0 + u >= n) break;
        const double *g = G + GEO_D * (q0 + u);
        const double sum = wj[u] + Wi;
        const double diff = wj[u] - Wi;
        dmin = (S)smin((double)dmin, diff);
        dmax = (S)smax((double)dmax, diff);
        Wx += (sum * g[0] + diff * g[3]) * g[9];
        Wy += (sum * g[1] + diff * g[4]) * g[9];
        Wz += (sum * g[2] + diff * g[5]) * g[9];
      }
    }
  }
  // boundary cells, and cells with a face on a boundary other than an inflow
  zero_flag = bad_cell || ((__ballot(zero_flag) >> grp) & 0xffffull) != 0;
  if (live && zero_flag && k < NF) {
    FLD(C.x, k, i, np) = (S)0.0;
    FLD(C.y, k, i, np) = (S)0.0;
    FLD(C.z, k, i, np) = (S)0.0;
    FLD(C.t, k, i, np) = (S)0.0;
  }

  const double invV = 1.0 / (live ? M.cvol[i] : 1.0);
  Wx *= invV;
  Wy *= invV;
  Wz *= invV;
  // J = curl B from the B lanes of this cell
  const double yBZ = __shfl(Wy, grp + BZ), zBY = __shfl(Wz, grp + BY);
  const double zBX = __shfl(Wz, grp + BX), xBZ = __shfl(Wx, grp + BZ);
  const double xBY = __shfl(Wx, grp + BY), yBX = __shfl(Wy, grp + BX);
  const double told = live ? (double)FLD(C.t, kk, i, np) : 0.0;
  double limiter_min = 1.0;
  if (P.limiter != LIM_SHIPPED) {
    // the shipped Phi() returns 1 for every argument.  The reference's time
    // term, 0 * Wt * dt, only matters where Wt is not finite
    const double dWt = 0.0 * told;
    double lo = 0.0, hi = 0.0;
    for (int f0 = 0; f0 < wdeg; f0 += FCH) {
      if (wdeg > FCH) {  // otherwise the one chunk is still staged
        wave_sync();
        stage(f0);
        wave_sync();
      }
      const int n = min(deg - f0, FCH);
      for (int q = 0; q < n; q++) {
        const double *g = G + GEO_D * q;
        const double d = (Wx * g[6] + Wy * g[7] + Wz * g[8]) + dWt;
        lo = __builtin_fmin(lo, d);
        hi = __builtin_fmax(hi, d);
      }
    }
    limiter_min = limiter_of_extremes<false>(P.limiter, lo, hi, (double)dmin, (double)dmax);
  }
  if (!live || zero_flag || k >= NF) return;
  if (k < 3) FLD(C.J, k, i, np) = (S)(k == 0 ? yBZ - zBY : k == 1 ? zBX - xBZ : xBY - yBX);
  FLD(C.mm_lo, k, i, np) = (S)((double)dmin + Wi);
  FLD(C.mm_hi, k, i, np) = (S)((double)dmax + Wi);
  const double tau = 1.0 * limiter_min;
  FLD(C.t, k, i, np) = (S)(told * tau);
  FLD(C.x, k, i, np) = (S)(Wx * tau);
  FLD(C.y, k, i, np) = (S)(Wy * tau);
  FLD(C.z, k, i, np) = (S)(Wz * tau);
}

// ---------------------------------------------------------------------------
// slopeLimiter compute part (slopeLimiter.cpp:27-237) per cell over its active
// face-ends, then computeFluidUpdateI (computeFluidUpdate.cpp:25-75)
// ---------------------------------------------------------------------------
struct FaceGeo {
  double area, normal[3], dri[3], drj[3], dsh, dsl;
};
__device__ __forceinline__ void face_geo(const MeshView &M, const double *pos_i, int f, int np,
                                         FaceGeo &g) {
  (void)np;
  const double fn[3] = {GEO_N(M, 0, f), GEO_N(M, 1, f), GEO_N(M, 2, f)};
  g.area = dsqrt(fn[0] * fn[0] + fn[1] * fn[1] + fn[2] * fn[2]);
  const double ia = 1.0 / g.area;
  for (int d = 0; d < 3; d++) {
    g.normal[d] = fn[d] * ia;
    g.dri[d] = GEO_C(M, d, f) - pos_i[d];
  }
  g.dsh = g.dri[0] * g.normal[0] + g.dri[1] * g.normal[1] + g.dri[2] * g.normal[2];
  g.dsl = 2.0 * g.dsh;
  for (int d = 0; d < 3; d++) g.drj[d] = g.dri[d] - g.normal[d] * g.dsl;
}

// Bound like the reconstruction by its chain of gathers (face-end -> active face
// -> face -> both cells' tend, position, boundary flag) and the face geometry,
// paid once a cell here, one face-end a lane.
// Measured (as the reconstruction): 235 us a launch against 912 and 145 us (529 us
// on average) for a thread per cell above 131,072 cells and a lane per (cell,
// variable) below; 72 us against 249; 10.5 us against 41.
template <typename S>
__global__ void __launch_bounds__(256) k_slope_limiter(Cells<S> C, MeshView M, Phys P, unsigned long long *diag) {
  constexpr int D = 4;            // staged per face-end: offset of the centroid, time offset
  constexpr int SL = FCH * D + 3;
  __shared__ double geo[256 / LC][SL];
  const int t = xgid();
  const int c = t / LC, k = t & (LC - 1), grp = (int)(threadIdx.x & 63) & ~(LC - 1);
  double *G = geo[threadIdx.x / LC];
  const int np = C.np;
  const bool live = c < np;
  const int fb = live ? M.soff[c] : 0;
  const int deg = live ? M.soff[c + 1] - fb : 0;
  const int wdeg = wave_cells_max(deg);
  const int kk = k < NF ? k : NF - 1;
  double x = 0.0, y = 0.0, z = 0.0, tt = 0.0;
  if (live) {
    x = (double)FLD(C.x, kk, c, np);
    y = (double)FLD(C.y, kk, c, np);
    z = (double)FLD(C.z, kk, c, np);
    tt = (double)FLD(C.t, kk, c, np);
  }
  double at[3] = {0.0, 0.0, 0.0}, lo = 0.0, hi = 0.0;
  bool at_bnd = false;
  for (int f0 = 0; f0 < wdeg; f0 += FCH) {
    if (f0 > 0) wave_sync();
    for (int q = k; q < FCH; q += LC) {
      if (f0 + q >= deg) break;
      const int ent = M.sent[fb + f0 + q];
      const int side = ent & 1;
      const int f = M.fact[ent >> 1];
      const int i = M.s1[f], j = M.s2[f];
      const double dtI = C.tend[i] - P.t_global;
      const double dtJ = C.tend[j] - P.t_global;
      const double dth = 0.5 * smin(dtI, dtJ);
      const double pos_i[3] = {FLD(C.pos, 0, i, np), FLD(C.pos, 1, i, np), FLD(C.pos, 2, i, np)};
      FaceGeo g;
      face_geo(M, pos_i, f, np, g);
      for (int d = 0; d < 3; d++) {
        const double an = g.normal[d] * g.area;
        at[d] = side == 0 ? at[d] + an : at[d] - an;
        G[D * q + d] = side == 0 ? g.dri[d] : g.drj[d];
      }
      G[D * q + 3] = side == 0 ? dtI - dth : dtJ - dth;
      at_bnd = at_bnd || C.bnd[i] != NO_BOUNDARY || C.bnd[j] != NO_BOUNDARY;
    }
    wave_sync();
    if (P.limiter == LIM_SHIPPED) continue;  // Phi() == 1: the limiter stays 1
    const int n = min(deg - f0, FCH);
    for (int q = 0; q < n; q++) {
      const double *g = G + D * q;
      const double dWt = tt * g[3];
      const double dWx = x * g[0] + y * g[1] + z * g[2];
      const double dW = dWx + dWt;
      lo = __builtin_fmin(lo, dW);
      hi = __builtin_fmax(hi, dW);
    }
  }
  // a face on a boundary sets every limiter of the cell to 0
  at_bnd = ((__ballot(at_bnd) >> grp) & 0xffffull) != 0;
  for (int d = 0; d < 3; d++)
    for (int o = LC / 2; o > 0; o >>= 1) at[d] += __shfl_xor(at[d], o);
  if (!live) return;
  if (k == 0 && c < C.nactive && C.bnd[c] == NO_BOUNDARY) {
    const double aabs = dsqrt(at[0] * at[0] + at[1] * at[1] + at[2] * at[2]);
    if (!(aabs < 1.0e-10 * pow(M.cvol[c], 2.0 / 3.0))) atomicAdd(&diag[FVM_DIAG_CLOSURE], 1ULL);
  }
  if (k >= NF) return;
  double l = 1.0;
  if (P.limiter != LIM_SHIPPED) {
    const double wc = FLD(C.w, k, c, np);
    const double mlo = (double)FLD(C.mm_lo, k, c, np), mhi = (double)FLD(C.mm_hi, k, c, np);
    l = limiter_of_extremes<true>(P.limiter, lo, hi, smin(mlo - wc, 0.0), smax(mhi - wc, 0.0));
  }
  const S lim = at_bnd ? (S)0.0 : (S)l;
  FLD(C.lim, k, c, np) = lim;
  if (c < C.nactive || C.is_ngb[c]) {
    const double f = 1.0 * (double)lim;
    FLD(C.x, k, c, np) = (S)(x * f);
    FLD(C.y, k, c, np) = (S)(y * f);
    FLD(C.z, k, c, np) = (S)(z * f);
    FLD(C.t, k, c, np) = (S)(tt * f);
  }
}

// ---------------------------------------------------------------------------
// System::computeFluidUpdate face part (computeFluidUpdate.cpp:99-223): one
// thread per active face writes the face record
//   rec[0..9] = flux*dt*A, rec[10..12] = n*(psi*dt*A), rec[13] = Bn*dt*A,
//   rec[15] = 1 when i and j were swapped (s1 on a boundary), else 0
// ---------------------------------------------------------------------------
// computeFluidUpdate.cpp:99-209: the inputs of computeFlux for active face a
// (boundary swap, space-time extrapolation of both sides, face velocity)
// F: the face arithmetic (double: the reference's; float: the FP32 face
// states, formed from FP64 geometry, dt and dti as the fused FP32 path forms
// them)
template <typename F> struct FaceIn {
  int i, j, jbnd;
  bool sw;
  double dt, area, normal[3], wij[3];
  F Wi[NF], Wj[NF];
};

// ROWS: the cells' values from their rows (k_cell_rows)
template <typename S, typename F, bool ROWS>
__device__ __forceinline__ void face_inputs(const Cells<S> &C, const MeshView &M, const Phys &P,
                                            const double *__restrict__ rows, int a, unsigned long long *diag,
                                            FaceIn<F> &q) {
  const int np = C.np;
  const int f = M.fact[a];
  int i = M.s1[f], j = M.s2[f];
  const double fn[3] = {GEO_N(M, 0, f), GEO_N(M, 1, f), GEO_N(M, 2, f)};
  const double area = dsqrt(fn[0] * fn[0] + fn[1] * fn[1] + fn[2] * fn[2]);
  const double ia = 1.0 / area;
  double normal[3] = {fn[0] * ia, fn[1] * ia, fn[2] * ia};
  double hi[CROW_W], hj[CROW_W];  // W, position, vel of the two sides
  if constexpr (ROWS) {
    ld_row(rows + (size_t)CROW * i, CROW_W, hi);
    ld_row(rows + (size_t)CROW * j, CROW_W, hj);
  } else {
    for (int d = 0; d < 3; d++) hi[10 + d] = FLD(C.pos, d, i, np);
  }
  double dri[3];
  for (int d = 0; d < 3; d++) dri[d] = GEO_C(M, d, f) - hi[10 + d];
  const bool sw = C.bnd[i] != NO_BOUNDARY;
  if (sw) {
    const int tmp = i;
    i = j;
    j = tmp;
    if constexpr (ROWS)
      for (int k = 0; k < CROW_W; k++) {
        const double t = hi[k];
        hi[k] = hj[k];
        hj[k] = t;
      }
    for (int d = 0; d < 3; d++) {
      normal[d] = normal[d] * -1.0;
      dri[d] = dri[d] * -1.0;
    }
  }
  const double dtI = C.tend[i] - P.t_global;
  const double dtJ = C.tend[j] - P.t_global;
  const double dt = smin(dtI, dtJ);
  const double dti = dtI - 0.5 * dt;
  const double dtj = dtJ - 0.5 * dt;
  const double dsh = dri[0] * normal[0] + dri[1] * normal[1] + dri[2] * normal[2];
  const double dsl = 2.0 * dsh;
  if (diag && !(dsl > 0.0)) atomicAdd(&diag[FVM_DIAG_DSL], 1ULL);
  const double drj[3] = {dri[0] - normal[0] * dsl, dri[1] - normal[1] * dsl, dri[2] - normal[2] * dsl};

  F *Wi = q.Wi, *Wj = q.Wj;
  for (int k = 0; k < NF; k++) {
    Wi[k] = (F)(ROWS ? hi[k] : FLD(C.w, k, i, np));
    Wj[k] = (F)(ROWS ? hj[k] : FLD(C.w, k, j, np));
  }
  const int jbnd = C.bnd[j];
  if (jbnd == NO_BOUNDARY) {
    // W + (x dr_x + y dr_y + z dr_z + t dt), term by term in this order; FP32: the
    // half-step state W + t dt first, then the gradient terms, in FMAs
    const auto extrapolate = [&](const double *row, int c, const double *dr, double dt_, F *W) {
      if constexpr (std::is_same<F, double>::value) {
        double g[NF], v[NF];
        const auto term = [&](int o, const S *fld, double h) {
          if constexpr (ROWS) ld_row(row + o, NF, v);
          for (int k = 0; k < NF; k++) {
            const double p = (ROWS ? v[k] : (double)FLD(fld, k, c, np)) * h;
            g[k] = o == CROW_W ? p : g[k] + p;
          }
        };
        term(CROW_W, C.x, dr[0]);
        term(CROW_W + NF, C.y, dr[1]);
        term(CROW_W + 2 * NF, C.z, dr[2]);
        term(CROW_W + 3 * NF, C.t, dt_);
        for (int k = 0; k < NF; k++) W[k] += g[k];
      } else {
        double v[NF];
        const auto term = [&](int o, const S *fld, float h) {
          if constexpr (ROWS) ld_row(row + o, NF, v);
          for (int k = 0; k < NF; k++)
            W[k] = __builtin_fmaf((float)(ROWS ? v[k] : (double)FLD(fld, k, c, np)), h, W[k]);
        };
        term(CROW_W + 3 * NF, C.t, (float)dt_);
        term(CROW_W, C.x, (float)dr[0]);
        term(CROW_W + NF, C.y, (float)dr[1]);
        term(CROW_W + 2 * NF, C.z, (float)dr[2]);
      }
    };
    extrapolate(rows + (size_t)CROW * i, i, dri, dti, Wi);
    extrapolate(rows + (size_t)CROW * j, j, drj, dtj, Wj);
  }
  if (diag && (!(Wi[DENS] > F(0.0)) || !(Wi[ETHM] > F(0.0)) || !(Wj[DENS] > F(0.0)) || !(Wj[ETHM] > F(0.0))))
    atomicAdd(&diag[FVM_DIAG_POSITIVITY], 1ULL);

  if constexpr (!ROWS)
    for (int d = 0; d < 3; d++) {
      hi[13 + d] = (double)FLD(C.vel, d, i, np);
      hj[13 + d] = (double)FLD(C.vel, d, j, np);
    }
  const double *vi = hi + 13, *vj = hj + 13;
  const double vij[3] = {vj[0] + vi[0], vj[1] + vi[1], vj[2] + vi[2]};
  const double dvij[3] = {vj[0] - vi[0], vj[1] - vi[1], vj[2] - vi[2]};
  const double fij[3] = {dri[0] - normal[0] * dsh, dri[1] - normal[1] * dsh, dri[2] - normal[2] * dsh};
  const double fdv = dvij[0] * fij[0] + dvij[1] * fij[1] + dvij[2] * fij[2];
  const double rji[3] = {normal[0] * dsl, normal[1] * dsl, normal[2] * dsl};
  const double r = 1.0 / sqr(dsl);
  q.wij[0] = vij[0] * 0.5 - rji[0] * fdv * r;
  q.wij[1] = vij[1] * 0.5 - rji[1] * fdv * r;
  q.wij[2] = vij[2] * 0.5 - rji[2] * fdv * r;
  for (int d = 0; d < 3; d++) q.normal[d] = normal[d];
  q.i = i;
  q.j = j;
  q.jbnd = jbnd;
  q.sw = sw;
  q.dt = dt;
  q.area = area;
}

// F = float: the FP32 face arithmetic (face states and HLLD); the records
// times dt and area, and every sum over them, stay FP64
template <typename S, typename F, bool ROWS>
__global__ void __launch_bounds__(256) k_face_flux(Cells<S> C, MeshView M, Phys P, const double *rows, double *rec,
                                   unsigned long long *diag) {
  const int a = xgid();
  if (a >= M.nfa) return;
  FaceIn<F> q;
  face_inputs<S, F, ROWS>(C, M, P, rows, a, diag, q);
  F psi, Bn, flux[NF];
  F wij[3], nrm[3];
  for (int d = 0; d < 3; d++) {
    wij[d] = (F)q.wij[d];
    nrm[d] = (F)q.normal[d];
  }
  compute_flux<F>((F)P.gamma, wij, q.Wi, q.Wj, q.jbnd, nrm, psi, Bn, flux);

  const double tarea = q.dt * q.area;
  for (int k = 0; k < NF; k++) REC(rec, k, a) = (double)flux[k] * tarea;
  for (int d = 0; d < 3; d++) REC(rec, NF + d, a) = q.normal[d] * ((double)psi * tarea);
  REC(rec, NF + 3, a) = (double)Bn * tarea;
  REC(rec, 14, a) = 0.0;
  REC(rec, 15, a) = q.sw ? 1.0 : 0.0;
}

// the computeFlux inputs of active faces [first, first + count), in the
// batch layout of fvm_compute_flux
template <typename S>
__global__ void __launch_bounds__(256) k_face_states(Cells<S> C, MeshView M, Phys P, int first, int count, double *wij,
                                                     double *Wi, double *Wj, int *jbnd, double *normal) {
  const int q0 = gid();
  if (q0 >= count) return;
  FaceIn<double> q;
  face_inputs<S, double, false>(C, M, P, nullptr, first + q0, nullptr, q);
  for (int d = 0; d < 3; d++) {
    wij[3 * (size_t)q0 + d] = q.wij[d];
    normal[3 * (size_t)q0 + d] = q.normal[d];
  }
  for (int k = 0; k < NF; k++) {
    Wi[(size_t)NF * q0 + k] = q.Wi[k];
    Wj[(size_t)NF * q0 + k] = q.Wj[k];
  }
  jbnd[q0] = q.jbnd;
}

// The sum of word k = lane % 16 of cell c's face records over its active
// face-ends in face_active_list order (computeFluidUpdate.cpp:225-245,
// computePredictor.cpp:120-136): words 0-9 (flux) leave the i side and enter the
// j side, the others the other way round.  Every sum rounds to the storage type
// as the reference's does (words 10-12 are added in it, word 14 stays double).
// Four rows in flight.
template <typename S>
__device__ __forceinline__ double sum_records(const MeshView &M, const double *rec, int fb, int deg, int wdeg) {
  const int lane = (int)__lane_id(), k = lane & (LC - 1), grp = lane & ~(LC - 1);
  double acc = 0.0;
  for (int f0 = 0; f0 < wdeg; f0 += LC) {
    const int mine = f0 + k < deg ? M.sent[fb + f0 + k] : -1;
    const int wn = min(wdeg - f0, LC);
    for (int q0 = 0; q0 < wn; q0 += 4) {
      double r[4];
      int ent[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        ent[u] = __shfl(mine, grp + q0 + u);
        r[u] = ent[u] >= 0 ? REC(rec, k, ent[u] >> 1) : 0.0;
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const bool sw = __shfl(r[u], grp + 15) != 0.0;
        if (ent[u] < 0) continue;
        const bool is_i = ((ent[u] & 1) == 0) != sw;
        const double x = is_i == (k < NF) ? -r[u] : r[u];
        if constexpr (std::is_same<S, double>::value) {
          acc = acc + x;
        } else {
          acc = (k >= NF && k < NF + 3) ? (double)((S)acc + (S)x) : k == 14 ? acc + x : (double)(S)(acc + x);
        }
      }
    }
  }
  return acc;
}

// Bound by the records, one 128-byte row per face-end, most of them from L2 or
// further.
// Measured (disk, 2.1 M cells, mean over the active sets of a cycle): 89 us a launch; a
// thread per cell above 131,072 cells and a lane per (cell, variable) below, with
// 112-byte rows and the swap flag in an array of its own, took 200 us on average.
template <typename S>
__global__ void __launch_bounds__(256) k_scatter(Cells<S> C, MeshView M, const double *rec) {
  const int t = xgid();
  const int c = t / LC, k = t & (LC - 1);
  const int np = C.np;
  const bool live = c < np;
  const int fb = live ? M.soff[c] : 0, deg = live ? M.soff[c + 1] - fb : 0;
  const double acc = sum_records<S>(M, rec, fb, deg, wave_cells_max(deg));
  if (!live) return;
  if (k < NF) FLD(C.dU, k, c, np) = FLD(C.dU, k, c, np) + (S)acc;
  else if (k < NF + 3) FLD(C.dgp, k - NF, c, np) = FLD(C.dgp, k - NF, c, np) + (S)acc;
  else if (k == NF + 3) FLD(C.ddivB, 0, c, np) = FLD(C.ddivB, 0, c, np) + (S)acc;
}

// ---------------------------------------------------------------------------
// System::computePrimitives (computeFluidUpdate.cpp:347-542), one thread per
// active cell; the failed-mass fallback (:508-541) touches only its own cell
// and runs in the same thread.
// ---------------------------------------------------------------------------
__device__ __forceinline__ double ethm_from_entropy(double g, const double *W) {
  return W[ENTR] * pow(W[DENS], g) / (g - 1.0);
}
__device__ __forceinline__ double entropy_from_ethm(double g, const double *W) {
  return (g - 1.0) * W[ETHM] / pow(W[DENS], g);
}

template <typename S>
__global__ void __launch_bounds__(256) k_primitives(Cells<S> C, MeshView M, Phys P, int predictor_flag,
                                    unsigned long long *diag) {
  const int i = xgid();
  if (i >= C.nactive) return;
  const int np = C.np;
  const double g = P.gamma;
  double Ui[NF], wi[NF];
  for (int k = 0; k < NF; k++) {
    Ui[k] = FLD(C.U, k, i, np);
    wi[k] = FLD(C.w, k, i, np);
  }
  if (C.bnd[i] != NO_BOUNDARY) {
    to_primitive(Ui, C.mvol[i], wi);
    for (int k = 0; k < NF; k++) {
      FLD(C.x, k, i, np) = (S)0.0;
      FLD(C.y, k, i, np) = (S)0.0;
      FLD(C.z, k, i, np) = (S)0.0;
      FLD(C.t, k, i, np) = (S)0.0;
    }
    C.mvol[i] = M.cvol[i];
    to_conservative(wi, C.mvol[i], Ui);
    for (int k = 0; k < NF; k++) {
      FLD(C.w, k, i, np) = wi[k];
      FLD(C.U, k, i, np) = Ui[k];
    }
    return;
  }
  double Uc[NF];
  for (int k = 0; k < NF; k++) Uc[k] = Ui[k] + (double)FLD(C.dU, k, i, np);
  const double divB = (double)FLD(C.ddivB, 0, i, np);
  const double dPsi[3] = {(double)FLD(C.dgp, 0, i, np), (double)FLD(C.dgp, 1, i, np),
                          (double)FLD(C.dgp, 2, i, np)};
  const double dt = P.t_global - C.tbeg[i];
  C.divB[i] = dt > 0.0 ? divB / dt / M.cvol[i] : divB;

  double W1[NF];
  const bool failed = Uc[MASS] <= 0.0;
  if (!failed) {
    const double dth = 0.5 * dt;
    double Wh[NF];
    for (int k = 0; k < NF; k++) Wh[k] = wi[k] + (double)FLD(C.t, k, i, np) * dth;
    Uc[WBX] -= Wh[VELX] * divB;
    Uc[WBY] -= Wh[VELY] * divB;
    Uc[WBZ] -= Wh[VELZ] * divB;
    const double pres = pressure(g, Wh[ETHM]);
    const double B2 = Wh[BX] * Wh[BX] + Wh[BY] * Wh[BY] + Wh[BZ] * Wh[BZ];
    const double dcs2 = g * pres + B2;
    const double ch_sig = dsqrt(dcs2 / Wh[DENS]);
    Uc[WBX] -= dPsi[0];
    Uc[WBY] -= dPsi[1];
    Uc[WBZ] -= dPsi[2];
    Uc[MPSI] -= dcs2 * divB;
    if (!predictor_flag) {
      double a0[3], a1[3];
      for (int d = 0; d < 3; d++) {
        a0[d] = FLD(C.acc0, d, i, np);
        a1[d] = FLD(C.acc1, d, i, np);
      }
      const double M0 = Ui[MASS], M1 = Uc[MASS];
      double dmom[3];
      for (int d = 0; d < 3; d++) dmom[d] = ((a0[d] * M0 + a1[d] * M1) * 0.5) * dt;
      Uc[MOMX] += dmom[0];
      Uc[MOMY] += dmom[1];
      Uc[MOMZ] += dmom[2];
      const double mom0[3] = {Ui[MOMX], Ui[MOMY], Ui[MOMZ]};
      const double mom1[3] = {Uc[MOMX], Uc[MOMY], Uc[MOMZ]};
      Uc[ENER] += ((mom0[0] * a0[0] + mom0[1] * a0[1] + mom0[2] * a0[2]) +
                   (mom1[0] * a1[0] + mom1[1] * a1[1] + mom1[2] * a1[2])) *
                  dt * 0.5;
    }
    const double cr = 0.5;
    const double l_min = pow(M.cvol[i] / (4.0 * REF_PI / 3.0), 1.0 / 3.0);
    Uc[MPSI] *= exp(-cr * ch_sig / l_min * dt);
    to_primitive(Uc, M.cvol[i], W1);
    if (W1[ETHM] <= 0.0) {
      W1[ETHM] = ethm_from_entropy(g, W1);
      atomicAdd(&diag[FVM_DIAG_ETHM_FAILED], 1ULL);
    } else {
      W1[ENTR] = entropy_from_ethm(g, W1);
    }
    if (predictor_flag) {
      if (dt > 0.0)
        for (int k = 0; k < NF; k++) FLD(C.t, k, i, np) = (S)((W1[k] - wi[k]) / dt);
      else
        for (int k = 0; k < NF; k++) FLD(C.t, k, i, np) = (S)0.0;
      return;
    }
  } else {
    atomicAdd(&diag[FVM_DIAG_MASS_FAILED], 1ULL);
    double Ut[NF];
    for (int k = 0; k < NF; k++) W1[k] = wi[k] + (double)FLD(C.t, k, i, np) * dt;
    to_conservative(W1, C.mvol[i], Ut);
    to_primitive(Ut, M.cvol[i], W1);
    if (W1[ETHM] <= 0.0) W1[ETHM] = ethm_from_entropy(g, W1);
    else W1[ENTR] = entropy_from_ethm(g, W1);
  }
  C.mvol[i] = M.cvol[i];
  to_conservative(W1, M.cvol[i], Ui);
  for (int k = 0; k < NF; k++) {
    FLD(C.w, k, i, np) = W1[k];
    FLD(C.U, k, i, np) = Ui[k];
    FLD(C.dU, k, i, np) = (S)0.0;
  }
  for (int d = 0; d < 3; d++) FLD(C.dgp, d, i, np) = (S)0.0;
  FLD(C.ddivB, 0, i, np) = (S)0.0;
}

// ---------------------------------------------------------------------------
// System::computeTimestep (computeTimestep.cpp:6-62)
// ---------------------------------------------------------------------------
// Two phases a wavefront, as the predictor's cell update: 16 lanes per cell look
// over its faces (R rounds of four cells), then one lane per cell finishes the
// cell.  R is chosen on the host so that small sets still fill the chip
// (cell_rounds).
template <typename S, int R>
__global__ void __launch_bounds__(256) k_timestep(Cells<S> C, MeshView M, Phys P, unsigned long long *dtmin_bits) {
  __shared__ double arg[256 / 64][4 * R];
  const int lane = (int)threadIdx.x & 63, wv = (int)threadIdx.x >> 6, k = lane & (LC - 1);
  const int c0 = (xgid() >> 6) * (4 * R);  // the wavefront's first cell
  const int np = C.np;
  for (int r = 0; r < R; r++) {
    const int i = c0 + 4 * r + lane / LC;
    // min over faces of h / (cs + sqrt(a_f)) = h / (cs + sqrt(max a_f)): every
    // rounding is monotone
    double a = -1.0;
    if (i < C.nactive) {
      const double fac = C.bnd[i] != NO_BOUNDARY ? 0.0 : 1.0;
      const double iM = 1.0 / FLD(C.U, MASS, i, np);
      double v[3], pv[3];
      for (int d = 0; d < 3; d++) {
        v[d] = FLD(C.U, MOMX + d, i, np) * iM;  // Fluid::to_primitive
        pv[d] = FLD(C.mvel, d, i, np);
      }
      const int fe = M.coff[i + 1];
      for (int e = M.coff[i] + k; e < fe; e += LC) {
        const int j = M.cnbr[e];
        const double dvi[3] = {FLD(C.w, VELX, j, np) - v[0], FLD(C.w, VELY, j, np) - v[1], FLD(C.w, VELZ, j, np) - v[2]};
        const double dwi[3] = {(double)FLD(C.vel, 0, j, np) - pv[0], (double)FLD(C.vel, 1, j, np) - pv[1],
                               (double)FLD(C.vel, 2, j, np) - pv[2]};
        a = __builtin_fmax(a, (dwi[0] * dwi[0] + dwi[1] * dwi[1] + dwi[2] * dwi[2]) +
                                  fac * (dvi[0] * dvi[0] + dvi[1] * dvi[1] + dvi[2] * dvi[2]) + 1.0 / REF_HUGE);
      }
    }
    for (int o = LC / 2; o > 0; o >>= 1) a = __builtin_fmax(a, __shfl_xor(a, o));
    if (k == 0) arg[wv][4 * r + lane / LC] = a;
  }
  wave_sync();
  const int i = c0 + lane;
  double v = HUGE_VAL;  // no cell
  if (lane < 4 * R && i < C.nactive) {
    const double g = P.gamma;
    const double Volume = C.mvol[i];
    double Ui[NF], Wi[NF];
    for (int m = 0; m < NF; m++) Ui[m] = FLD(C.U, m, i, np);
    to_primitive(Ui, Volume, Wi);
    const double h = pow(Volume / (4.0 * REF_PI / 3.0), 1.0 / 3.0);
    const double pv[3] = {FLD(C.mvel, 0, i, np), FLD(C.mvel, 1, i, np), FLD(C.mvel, 2, i, np)};
    double csi = 0.0, vrel = 0.0;
    if (C.bnd[i] == NO_BOUNDARY) {
      const double Pi = pressure(g, Wi[ETHM]) * g;
      const double B2i = Wi[BX] * Wi[BX] + Wi[BY] * Wi[BY] + Wi[BZ] * Wi[BZ];
      csi = dsqrt((Pi + B2i) / Wi[DENS]);
      const double dv[3] = {Wi[VELX] - pv[0], Wi[VELY] - pv[1], Wi[VELZ] - pv[2]};
      vrel = dsqrt(dv[0] * dv[0] + dv[1] * dv[1] + dv[2] * dv[2]);
    }
    double dti = h / (csi + vrel + 1.0 / REF_HUGE);
    const double a = arg[wv][lane];
    if (a >= 0.0) dti = smin(dti, h / (csi + dsqrt(a)));
    dti = smin(dti, REF_HUGE);
    const double dtn = dti * P.courant;
    C.dt_new[i] = dtn;
    if (dtn >= 0.0) v = dtn;  // a cell without a timestep (NaN) leaves the others theirs
  }
  // min over active cells; dt > 0 so the IEEE bit patterns order like the
  // values.  Atomics on one address take their turn (about 10 ns each), so a
  // block adds one, and only while it lowers what it reads there
  for (int off = 32; off > 0; off >>= 1) v = smin(v, __shfl_xor(v, off));
  __shared__ double wmin[256 / 64];
  if (lane == 0) wmin[wv] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int m = 1; m < 256 / 64; m++) v = smin(v, wmin[m]);
    const unsigned long long bits = (unsigned long long)__double_as_longlong(v);
    if (bits < __hip_atomic_load(dtmin_bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      atomicMin(dtmin_bits, bits);
  }
}

// ---------------------------------------------------------------------------
// System::computePredictor (computePredictor.cpp:11-391)
// face part: record rec[0..9] = flux*A, [10..12] = n*(psi*A), [13] = Bn*A, [14] = dV,
// [15] = swapped
// ---------------------------------------------------------------------------
// F = float: the FP32 HLLD of the first-order states; the records stay FP64
template <typename S, typename F>
__global__ void __launch_bounds__(256) k_predictor_face(Cells<S> C, MeshView M, Phys P, double *rec,
                                        unsigned long long *diag) {
  const int a = xgid();
  if (a >= M.nfa) return;
  const int np = C.np;
  const int f = M.fact[a];
  int i = M.s1[f], j = M.s2[f];
  const double fn[3] = {GEO_N(M, 0, f), GEO_N(M, 1, f), GEO_N(M, 2, f)};
  const double area = dsqrt(fn[0] * fn[0] + fn[1] * fn[1] + fn[2] * fn[2]);
  const double ia = 1.0 / area;
  double normal[3] = {fn[0] * ia, fn[1] * ia, fn[2] * ia};
  double dri[3];
  for (int d = 0; d < 3; d++) dri[d] = GEO_C(M, d, f) - FLD(C.pos, d, i, np);
  const bool sw = C.bnd[i] != NO_BOUNDARY;
  if (sw) {
    const int tmp = i;
    i = j;
    j = tmp;
    for (int d = 0; d < 3; d++) {
      normal[d] = normal[d] * -1.0;
      dri[d] = dri[d] * -1.0;
    }
  }
  const double dsh = dri[0] * normal[0] + dri[1] * normal[1] + dri[2] * normal[2];
  const double dsl = 2.0 * dsh;
  if (!(dsl > 0.0)) atomicAdd(&diag[FVM_DIAG_DSL], 1ULL);
  const int jbnd = C.bnd[j];
  const int jw = (jbnd == NO_BOUNDARY || jbnd == INFLOW) ? j : i;
  double Wi[NF], Wj[NF];
  for (int k = 0; k < NF; k++) {
    Wi[k] = FLD(C.w, k, i, np);
    Wj[k] = FLD(C.w, k, jw, np);
  }
  const double vi[3] = {(double)FLD(C.vel, 0, i, np), (double)FLD(C.vel, 1, i, np), (double)FLD(C.vel, 2, i, np)};
  const double vj[3] = {(double)FLD(C.vel, 0, j, np), (double)FLD(C.vel, 1, j, np), (double)FLD(C.vel, 2, j, np)};
  const double vij[3] = {vj[0] + vi[0], vj[1] + vi[1], vj[2] + vi[2]};
  const double dvij[3] = {vj[0] - vi[0], vj[1] - vi[1], vj[2] - vi[2]};
  const double fij[3] = {dri[0] - normal[0] * dsh, dri[1] - normal[1] * dsh, dri[2] - normal[2] * dsh};
  const double fdv = dvij[0] * fij[0] + dvij[1] * fij[1] + dvij[2] * fij[2];
  const double rij[3] = {normal[0] * dsl, normal[1] * dsl, normal[2] * dsl};
  const double r = 1.0 / sqr(dsl);
  const double wij[3] = {vij[0] * 0.5 - rij[0] * fdv * r, vij[1] * 0.5 - rij[1] * fdv * r,
                         vij[2] * 0.5 - rij[2] * fdv * r};
  F psi, Bn, flux[NF];
  {
    F wf[3], nf[3], Wif[NF], Wjf[NF];
    for (int d = 0; d < 3; d++) {
      wf[d] = (F)wij[d];
      nf[d] = (F)normal[d];
    }
    for (int k = 0; k < NF; k++) {
      Wif[k] = (F)Wi[k];
      Wjf[k] = (F)Wj[k];
    }
    compute_flux<F>((F)P.gamma, wf, Wif, Wjf, jbnd, nf, psi, Bn, flux);
  }
  for (int k = 0; k < NF; k++) REC(rec, k, a) = (double)flux[k] * area;
  for (int d = 0; d < 3; d++) REC(rec, NF + d, a) = normal[d] * ((double)psi * area);
  REC(rec, NF + 3, a) = (double)Bn * area;
  REC(rec, NF + 4, a) = area * (rij[0] * wij[0] + rij[1] * wij[1] + rij[2] * wij[2]) / dsl;
  REC(rec, 15, a) = sw ? 1.0 : 0.0;
}

__device__ __forceinline__ int exp_of(double dt) {
  return (int)(((unsigned long long)__double_as_longlong(dt) >> 52) & 0xfff);
}
// Scheduler::get_dt(get_rung(dt)) (Scheduler.h:94-111)
__device__ __forceinline__ double rung_dt(double dtmax, int min_rung, double dt) {
  int rung = exp_of(dtmax) - exp_of(dt);
  if (rung < min_rung) rung = min_rung;
  const double dt_tick = dtmax / (double)(1ULL << 31);
  return dt_tick * (double)(1ULL << (31 - rung));
}

// Cell part, two phases a wavefront: the face sums with 16 lanes per cell (R
// rounds of four cells), then the cell update with one lane per cell.  Bound by
// the records in large sets, by the update's chain of divisions, exp and pow in
// small ones.
// Measured (same sets): 128 us a launch against 179 us for a thread per cell above
// 131,072 cells and a lane per (cell, variable) below; 97,000 cells at once: 57
// against 105 us.
template <typename S, int R>
__global__ void __launch_bounds__(256) k_predictor_cell(Cells<S> C, MeshView M, Phys P, const double *rec,
                                        double dtmax, int min_rung, unsigned long long *diag) {
  constexpr int ST = NREC + 1;  // a cell's sums in LDS
  __shared__ double sums[256 / 64][4 * R * ST];
  const int lane = (int)threadIdx.x & 63, wv = (int)threadIdx.x >> 6, k = lane & (LC - 1);
  const int c0 = (xgid() >> 6) * (4 * R);  // the wavefront's first cell
  const int np = C.np;
  for (int r = 0; r < R; r++) {
    const int i = c0 + 4 * r + lane / LC;
    const int fb = i < C.nactive ? M.soff[i] : 0, deg = i < C.nactive ? M.soff[i + 1] - fb : 0;
    sums[wv][(4 * r + lane / LC) * ST + k] = sum_records<S>(M, rec, fb, deg, wave_cells_max(deg));
  }
  wave_sync();
  const int c = c0 + lane;
  if (lane >= 4 * R || c >= C.nactive || C.bnd[c] != NO_BOUNDARY) return;
  const double *dU = &sums[wv][lane * ST];
  const double *dPsi = dU + NF;
  const double divB = dU[NF + 3], dV = dU[NF + 4];
  const double g = P.gamma;
  double U0[NF], W0[NF];
  for (int m = 0; m < NF; m++) U0[m] = FLD(C.U, m, c, np);
  to_primitive(U0, M.cvol[c], W0);
  double dtn = C.dt_new[c];
  while (U0[MASS] + dU[MASS] * dtn <= 0.0) dtn *= 0.5;
  C.dt_new[c] = dtn;
  const double dt = rung_dt(dtmax, min_rung, dtn) / 128;
  double Uc[NF];
  for (int m = 0; m < NF; m++) Uc[m] = U0[m] + dU[m] * dt;
  Uc[WBX] -= W0[VELX] * divB * dt;
  Uc[WBY] -= W0[VELY] * divB * dt;
  Uc[WBZ] -= W0[VELZ] * divB * dt;
  const double pres = pressure(g, W0[ETHM]);
  const double B2 = W0[BX] * W0[BX] + W0[BY] * W0[BY] + W0[BZ] * W0[BZ];
  const double dcs2 = g * pres + B2;
  const double ch_sig = dsqrt(dcs2 / W0[DENS]);
  Uc[WBX] -= dPsi[0] * dt;
  Uc[WBY] -= dPsi[1] * dt;
  Uc[WBZ] -= dPsi[2] * dt;
  Uc[MPSI] -= dcs2 * divB * dt;
  const double cr = 0.5;
  const double l_min = pow(M.cvol[c] / (4.0 * REF_PI / 3.0), 1.0 / 3.0);
  Uc[MPSI] *= exp(-cr * ch_sig / l_min * dt);
  double W1[NF];
  to_primitive(Uc, M.cvol[c] * exp(dV * dt / M.cvol[c]), W1);
  if (W1[ETHM] <= 0.0) {
    W1[ETHM] = ethm_from_entropy(g, W1);
    atomicAdd(&diag[FVM_DIAG_ETHM_FAILED], 1ULL);
  } else {
    W1[ENTR] = entropy_from_ethm(g, W1);
  }
  const double idt = 1.0 / dt;
  for (int m = 0; m < NF; m++) FLD(C.t, m, c, np) = (S)((W1[m] - W0[m]) * idt);
}

// ---------------------------------------------------------------------------
// batched System::computeFlux (FP64)
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_flux_batch(int n, double gamma, const double *wij, const double *Wi, const double *Wj,
                             const int *jbnd, const double *normal, double *psi, double *Bn, double *flux) {
  const int f = gid();
  if (f >= n) return;
  double w3[3], n3[3], L[NF], R[NF], F[NF];
  for (int d = 0; d < 3; d++) {
    w3[d] = wij[3 * (size_t)f + d];
    n3[d] = normal[3 * (size_t)f + d];
  }
  for (int k = 0; k < NF; k++) {
    L[k] = Wi[(size_t)NF * f + k];
    R[k] = Wj[(size_t)NF * f + k];
  }
  double p, b;
  compute_flux<double>(gamma, w3, L, R, jbnd[f], n3, p, b, F);
  psi[f] = p;
  Bn[f] = b;
  for (int k = 0; k < NF; k++) flux[(size_t)NF * f + k] = F[k];
}

// The same on a small batch in pinned host memory: in wij[n][3], Wi[n][10],
// Wj[n][10], normal[n][3], jbnd; out psi[n], B_n[n], flux[n][10].  A wavefront reads
// and writes its 64 faces' rows over the link in whole lines, all in flight,
// through LDS; one launch in place of two copies in, a launch and a copy out, each
// a few microseconds after the other (2048 faces: 64 -> 43 us a call).
__global__ void __launch_bounds__(64) k_flux_pinned(int n, double gamma, const double *in, const int *jbnd, double *out) {
  constexpr int W = 26;
  __shared__ double tile[64 * W];
  const int l = (int)threadIdx.x, f0 = (int)blockIdx.x * 64, m = min(64, n - f0);
  const int width[4] = {3, NF, NF, 3};
  {
    double v[W];
    int off = 0;
#pragma unroll
    for (int a = 0; a < 4; a++) {
      const double *p = in + (size_t)off * n + (size_t)width[a] * f0;
#pragma unroll
      for (int u = 0; u < width[a]; u++) v[off + u] = 64 * u + l < width[a] * m ? p[64 * u + l] : 0.0;
      off += width[a];
    }
#pragma unroll
    for (int u = 0; u < W; u++) tile[64 * u + l] = v[u];
  }
  const int jb = l < m ? jbnd[f0 + l] : NO_BOUNDARY;
  __syncthreads();
  double w3[3], n3[3], L[NF], R[NF], F[NF], p, b;
  for (int d = 0; d < 3; d++) {
    w3[d] = tile[3 * l + d];
    n3[d] = tile[64 * 23 + 3 * l + d];
  }
  for (int k = 0; k < NF; k++) {
    L[k] = tile[64 * 3 + NF * l + k];
    R[k] = tile[64 * 13 + NF * l + k];
  }
  __syncthreads();
  if (l < m) {
    compute_flux<double>(gamma, w3, L, R, jb, n3, p, b, F);
    out[f0 + l] = p;
    out[n + f0 + l] = b;
    for (int k = 0; k < NF; k++) tile[NF * l + k] = F[k];
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < NF; u++)
    if (64 * u + l < NF * m) out[2 * (size_t)n + (size_t)NF * f0 + 64 * u + l] = tile[64 * u + l];
}

// ---------------------------------------------------------------------------
// get_active_faces (Iterate.cpp:298-324) and the per-cell face-end lists
// ---------------------------------------------------------------------------
__global__ void k_fill_int(int *p, int v, int n) {
  const int i = gid();
  if (i < n) p[i] = v;
}
__global__ void k_set_u64(unsigned long long *p, unsigned long long v) {
  if (gid() == 0) *p = v;
}

// Cell lists from the face list as localMesh.cpp:586-589 builds them: every
// face is listed by its s1 and, when s2 is active, by its s2, in the order the
// faces were created (ascending index).  Count, scan, fill, then sort each
// cell's short list.
__global__ void k_csr_count(const int *__restrict__ s1, const int *__restrict__ s2, int nface, int nactive,
                            int *__restrict__ cnt) {
  const int f = gid();
  if (f >= nface) return;
  atomicAdd(&cnt[s1[f]], 1);
  if (s2[f] < nactive) atomicAdd(&cnt[s2[f]], 1);
}
__global__ void k_csr_fill(const int *__restrict__ s1, const int *__restrict__ s2, int nface, int nactive,
                           int *__restrict__ cursor, int *__restrict__ cface) {
  const int f = gid();
  if (f >= nface) return;
  cface[atomicAdd(&cursor[s1[f]], 1)] = f;
  if (s2[f] < nactive) cface[atomicAdd(&cursor[s2[f]], 1)] = f;
}
// the other cell of every cell_face entry
__global__ void k_cell_nbr(const int *__restrict__ coff, const int *__restrict__ cface, const int *__restrict__ s1,
                           const int *__restrict__ s2, int nactive, int *__restrict__ cnbr) {
  const int t = gid();
  const int i = t / LC;
  if (i >= nactive) return;
  for (int e = coff[i] + (t & (LC - 1)); e < coff[i + 1]; e += LC) {
    const int f = cface[e], a = s1[f];
    cnbr[e] = a == i ? s2[f] : a;
  }
}
// Distinct non-negative ints of a short list into ascending order by 16 lanes:
// every lane ranks its own entries against the whole list in LDS (up to
// LIST_LDS entries; longer lists are handled by the callers).  Negative entries
// are left out.
constexpr int LIST_LDS = 64;
template <typename F> __device__ __forceinline__ void rank_list(const int *list, int n, int k, F put) {
  for (int e = k; e < n; e += LC) {
    const int v = list[e];
    if (v < 0) continue;
    int rank = 0;
    for (int m = 0; m < n; m++) rank += (unsigned)list[m] < (unsigned)v ? 1 : 0;
    put(rank, v);
  }
}
__global__ void __launch_bounds__(256) k_csr_sort(const int *__restrict__ coff, int nactive, int *__restrict__ cface) {
  __shared__ int list[256 / LC][LIST_LDS + 1];
  const int t = gid();
  const int i = t / LC, k = t & (LC - 1);
  int *l = list[threadIdx.x / LC];
  const int b = i < nactive ? coff[i] : 0, e = i < nactive ? coff[i + 1] : 0, n = e - b;
  if (n <= LIST_LDS)
    for (int q = k; q < n; q += LC) l[q] = cface[b + q];
  wave_sync();
  if (n <= LIST_LDS) {
    rank_list(l, n, k, [&](int r, int v) { cface[b + r] = v; });
  } else if (k == 0) {
    for (int q = b + 1; q < e; q++) {
      const int v = cface[q];
      int m = q - 1;
      while (m >= b && cface[m] > v) {
        cface[m + 1] = cface[m];
        m--;
      }
      cface[m + 1] = v;
    }
  }
}
// first position of each face in the concatenated face lists of active,
// non-boundary cells
__global__ void k_face_firstpos(MeshView M, const int *bnd, int nactive, int *firstpos) {
  const int i = gid();
  if (i >= nactive || bnd[i] != NO_BOUNDARY) return;
  for (int e = M.coff[i]; e < M.coff[i + 1]; e++) atomicMin(&firstpos[M.cface[e]], e);
}
__global__ void k_face_firstflag(MeshView M, const int *bnd, int nactive, const int *firstpos, int *flag) {
  const int i = gid();
  if (i >= nactive) return;
  const bool ok = bnd[i] == NO_BOUNDARY;
  for (int e = M.coff[i]; e < M.coff[i + 1]; e++) flag[e] = (ok && firstpos[M.cface[e]] == e) ? 1 : 0;
}
// The same flags when every active cell lists all its faces (each face under
// s1 when s1 is active and under s2 when s2 is active): a face first appears
// in the lower-indexed of its two cells that are active and not on a
// boundary, since the lists are concatenated in cell order.
__global__ void k_face_firstflag_direct(MeshView M, const int *bnd, int nactive, int *flag) {
  const int t = gid();
  const int i = t / LC;
  if (i >= nactive) return;
  const bool ok = bnd[i] == NO_BOUNDARY;
  for (int e = M.coff[i] + (t & (LC - 1)); e < M.coff[i + 1]; e += LC) {
    const int j = M.cnbr[e];
    const bool earlier = j < i && j < nactive && bnd[j] == NO_BOUNDARY;
    flag[e] = (ok && !earlier) ? 1 : 0;
  }
}
__global__ void k_face_compact(MeshView M, const int *flag, const int *pos, int nref, int *fact, int *fpos) {
  const int e = gid();
  if (e < nref && flag[e]) {
    const int f = M.cface[e], a = pos[e];
    fact[a] = f;
    fpos[f] = a;
  }
}

// The face-end list of every cell, entries a << 1 | side in ascending order,
// from the cells' own face lists and the faces' places in the active list: no
// atomics, and no gathers beyond one list.  A cell without a list of its own (an
// inactive neighbour of a substep layout) walks its global list and takes the
// faces of the layout.  COUNT: the lengths; otherwise the lists.
// Measured (disk, 2.1 M cells, mean over the active sets of a cycle): 77 us for both
// passes; counting and filling over the active faces with atomics, then
// sorting, took 201 us (a 14,000-cell mesh's active sets: 10 against 51 us).
struct EndLists {
  int np, nactive;
  const int *coff, *cface, *s1, *fpos;
  const int *perm, *goff, *gface, *gmark, *gpos;  // substep layout (cells >= nactive), else null
};
__device__ __forceinline__ int end_entry(const EndLists &E, int c, int e) {
  int f;
  if (c < E.nactive) {
    f = E.cface[e];
  } else {
    const int gf = E.gface[e];
    if (!E.gmark[gf]) return -1;
    f = E.gpos[gf];
  }
  const int a = E.fpos[f];
  return a < 0 ? -1 : (a << 1) | (E.s1[f] == c ? 0 : 1);
}
template <bool COUNT>
__global__ void __launch_bounds__(256) k_end_lists(EndLists E, int *__restrict__ cnt, const int *__restrict__ soff,
                                                   int *__restrict__ sent) {
  __shared__ int list[256 / LC][LIST_LDS + 1];
  const int t = xgid();
  const int c = t / LC, k = t & (LC - 1);
  const bool live = c < E.np;
  int b = 0, n = 0;
  if (live) {
    const int g = c < E.nactive ? c : E.perm[c];
    const int *off = c < E.nactive ? E.coff : E.goff;
    b = off[g];
    n = off[g + 1] - b;
  }
  if constexpr (COUNT) {
    int m = 0;
    for (int q = k; q < n; q += LC) m += end_entry(E, c, b + q) >= 0 ? 1 : 0;
    for (int o = LC / 2; o > 0; o >>= 1) m += __shfl_xor(m, o);
    if (live && k == 0) cnt[c] = m;
  } else {
    int *l = list[threadIdx.x / LC];
    if (n <= LIST_LDS)
      for (int q = k; q < n; q += LC) l[q] = end_entry(E, c, b + q);
    wave_sync();
    if (!live) return;
    int *out = sent + soff[c];
    if (n <= LIST_LDS) {
      rank_list(l, n, k, [&](int r, int v) { out[r] = v; });
    } else {
      for (int q = k; q < n; q += LC) {
        const int v = end_entry(E, c, b + q);
        if (v < 0) continue;
        int rank = 0;
        for (int m = 0; m < n; m++) rank += (unsigned)end_entry(E, c, b + m) < (unsigned)v ? 1 : 0;
        out[rank] = v;
      }
    }
  }
}
// Consecutive active faces mostly share the cell whose list introduced them,
// so lanes with the same target add once per wavefront: the lowest such lane
// adds the lane count, and each lane takes base + its rank among them.  Every
// lane of the wavefront runs the loop (inactive ones with target -1).
__device__ __forceinline__ int wave_add(int *ctr, int t, bool want_pos) {
  const int lane = (int)(threadIdx.x & 63);
  unsigned long long left = __ballot(t >= 0);
  int pos = -1;
  while (left) {
    const int lead = __ffsll((long long)left) - 1;
    const int tv = __shfl(t, lead);
    const unsigned long long same = __ballot(t == tv);
    int base = 0;
    if (lane == lead) base = atomicAdd(&ctr[tv], __popcll(same));
    if (want_pos) {
      base = __shfl(base, lead);
      if (t == tv) pos = base + __popcll(same & ((1ull << lane) - 1ull));
    }
    left &= ~same;
  }
  return pos;
}
__global__ void k_end_count(MeshView M, int *cnt) {
  const int a = gid();
  int t1 = -1, t2 = -1;
  if (a < M.nfa) {
    const int f = M.fact[a];
    t1 = M.s1[f];
    t2 = M.s2[f];
  }
  wave_add(cnt, t1, false);
  wave_add(cnt, t2, false);
}
__global__ void k_end_fill(MeshView M, int *cursor, int *sent) {
  const int a = gid();
  int t1 = -1, t2 = -1;
  if (a < M.nfa) {
    const int f = M.fact[a];
    t1 = M.s1[f];
    t2 = M.s2[f];
  }
  const int p1 = wave_add(cursor, t1, true);
  const int p2 = wave_add(cursor, t2, true);
  if (a < M.nfa) {
    sent[p1] = (a << 1) | 0;
    sent[p2] = (a << 1) | 1;
  }
}
// order each cell's face-ends by face_active_list position (insertion sort of
// short segments) so that every sum runs in the reference's face order
// Each cell's face-end entries (a << 1 | side, all distinct) in ascending
// order.  Up to END_SORT_REG entries are sorted in registers by a fully
// unrolled odd-even transposition network (static indices, padded with
// INT_MAX); longer lists are insertion-sorted in place.  Distinct keys have
// one sorted order, so both give the same list.
constexpr int END_SORT_REG = 48;
__global__ void k_end_sort(const int *soff, int *sent, int n) {
  const int c = gid();
  if (c >= n) return;
  const int b = soff[c], e = soff[c + 1];
  const int deg = e - b;
  if (deg <= 1) return;
  if (deg <= END_SORT_REG) {
    int v[END_SORT_REG];
#pragma unroll
    for (int k = 0; k < END_SORT_REG; k++) v[k] = k < deg ? sent[b + k] : INT_MAX;
#pragma unroll
    for (int pass = 0; pass < END_SORT_REG; pass++) {
#pragma unroll
      for (int k = pass & 1; k + 1 < END_SORT_REG; k += 2) {
        const int lo = min(v[k], v[k + 1]), hi = max(v[k], v[k + 1]);
        v[k] = lo;
        v[k + 1] = hi;
      }
    }
#pragma unroll
    for (int k = 0; k < END_SORT_REG; k++)
      if (k < deg) sent[b + k] = v[k];
    return;
  }
  for (int p = b + 1; p < e; p++) {
    const int v = sent[p];
    int q = p - 1;
    while (q >= b && sent[q] > v) {
      sent[q + 1] = sent[q];
      q--;
    }
    sent[q + 1] = v;
  }
}

}  // namespace fvm

// ===========================================================================
// staging memory of fvm_compute_flux_noalloc
// ===========================================================================
// A file-scope device array: every GPU the library runs on holds its own copy
// (at its own address) until the process ends.  In host code the name
// `scratch` is only a host-side stand-in; the device address of each GPU's
// copy comes from hipGetSymbolAddress, called once per device by fvm_create
// with that device current, and only that address is ever passed to kernels
// or copies.
static __device__ __align__(256) unsigned char scratch[FVM_FLUX_NOALLOC_BYTES];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[kMaxDevices];  // device address of `scratch` per device, or null
}  // namespace

// device address of this device's copy of `scratch` (the caller has made the
// device current); looked up once per device
static int noalloc_scratch_init(int device) {
  if (device < 0 || device >= kMaxDevices) return FVM_EARG;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (g_scratch_ptr[device]) return FVM_OK;
  void *p = nullptr;
  if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return FVM_EHIP;
  g_scratch_ptr[device] = p;
  return FVM_OK;
}

static void *noalloc_scratch(int device) {
  if (device < 0 || device >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  return g_scratch_ptr[device];
}

// ===========================================================================
// context
// ===========================================================================
int fvm_fail(fvm_ctx *c, int code, const std::string &msg) {
  if (c) c->err = msg;
  return code;
}
static int fail(fvm_ctx *c, int code, const std::string &msg) { return fvm_fail(c, code, msg); }
#define HIPCHK(c, call) FVM_HIPCHK(c, call)

// the end of an entry point: wait for its work unless a substep defers it
static int finish(fvm_ctx *c) {
  if (!c->defer_sync) HIPCHK(c, hipStreamSynchronize(c->stream));
  return FVM_OK;
}

int fvm_ensure(fvm_ctx *c, DBuf &b, size_t bytes) {
  if (b.bytes >= bytes && b.p) return FVM_OK;
  if (b.p) HIPCHK(c, hipFree(b.p));
  b.p = nullptr;
  b.bytes = 0;
  if (bytes == 0) bytes = 8;
  hipError_t e = hipMalloc(&b.p, bytes);
  if (e != hipSuccess && &b != &c->crow && c->crow.p) {
    // the cell rows are optional: their memory goes to what cannot do without
    (void)hipGetLastError();
    fvm_release(c->crow);
    e = hipMalloc(&b.p, bytes);
  }
  if (e != hipSuccess) {
    b.p = nullptr;
    return fvm_fail(c, FVM_EHIP, std::string("hipMalloc(&b.p, bytes): ") + hipGetErrorString(e));
  }
  b.bytes = bytes;
  return FVM_OK;
}
static int ensure(fvm_ctx *c, DBuf &b, size_t bytes) { return fvm_ensure(c, b, bytes); }
void fvm_release(DBuf &b) {
  if (b.p) (void)hipFree(b.p);
  b.p = nullptr;
  b.bytes = 0;
}
static void release(DBuf &b) { fvm_release(b); }

static size_t store_size(const fvm_ctx *c) { return c->prm.storage == FVM_STORAGE_SHIPPED ? sizeof(float) : sizeof(double); }
static size_t field_bytes(const fvm_ctx *c, int f, int np) {
  const auto &fi = fvm::kFields[f];
  const size_t es = fi.kind == fvm::K_INT ? sizeof(int) : (fi.kind == fvm::K_STORE ? store_size(c) : sizeof(double));
  return es * (size_t)fi.width * (size_t)np;
}

template <typename S> static fvm::Cells<S> cells(fvm_ctx *c) {
  fvm::Cells<S> C;
  C.np = c->np;
  C.nactive = c->nactive;
  auto D = [&](int f) { return (double *)c->field[f].p; };
  auto St = [&](int f) { return (S *)c->field[f].p; };
  auto I = [&](int f) { return (int *)c->field[f].p; };
  C.w = D(FVM_FIELD_W);
  C.x = St(FVM_FIELD_GRAD_X);
  C.y = St(FVM_FIELD_GRAD_Y);
  C.z = St(FVM_FIELD_GRAD_Z);
  C.t = St(FVM_FIELD_DWDT);
  C.pos = D(FVM_FIELD_POS);
  C.vel = St(FVM_FIELD_VEL);
  C.J = St(FVM_FIELD_J);
  C.tend = D(FVM_FIELD_TEND);
  C.bnd = I(FVM_FIELD_BND);
  C.is_ngb = I(FVM_FIELD_IS_NGB);
  C.is_active = I(FVM_FIELD_IS_ACTIVE);
  C.mm_lo = St(FVM_FIELD_MINMAX_LO);
  C.mm_hi = St(FVM_FIELD_MINMAX_HI);
  C.lim = St(FVM_FIELD_LIMITER);
  C.dU = St(FVM_FIELD_DU);
  C.dgp = St(FVM_FIELD_DGRADPSI);
  C.ddivB = St(FVM_FIELD_DDIVB);
  C.U = D(FVM_FIELD_U);
  C.mvol = D(FVM_FIELD_MESH_VOLUME);
  C.tbeg = D(FVM_FIELD_TBEG);
  C.mvel = D(FVM_FIELD_MESH_VEL);
  C.acc0 = D(FVM_FIELD_ACC0);
  C.acc1 = D(FVM_FIELD_ACC1);
  C.dt_new = D(FVM_FIELD_DT_NEW);
  C.divB = D(FVM_FIELD_DIVB);
  return C;
}

static fvm::MeshView meshview(fvm_ctx *c) {
  fvm::MeshView M;
  M.nface = c->nface;
  M.nfa = c->nfa < 0 ? 0 : c->nfa;
  M.s1 = (const int *)c->m_s1.p;
  M.s2 = (const int *)c->m_s2.p;
  M.cn = (const double *)c->m_cn.p;
  M.coff = (const int *)c->m_coff.p;
  M.cface = (const int *)c->m_cface.p;
  M.cnbr = (const int *)c->m_cnbr.p;
  M.cvol = (const double *)c->m_cvol.p;
  M.fact = (const int *)c->m_fact.p;
  M.soff = (const int *)c->m_soff.p;
  M.sent = (const int *)c->m_sent.p;
  return M;
}

static fvm::Phys phys(const fvm_ctx *c) {
  fvm::Phys P;
  P.gamma = c->prm.gamma_gas;
  P.courant = c->prm.courant_no;
  P.t_global = c->t_global;
  for (int d = 0; d < 3; d++) P.L[d] = c->prm.domain_size[d];
  P.limiter = c->prm.limiter_mode;
  return P;
}

static inline unsigned nblk(long n, int bs = 256) { return (unsigned)((n + bs - 1) / bs); }

#define LAUNCH(c, kern, n, ...)                                                        \
  do {                                                                                 \
    if ((n) > 0) {                                                                     \
      hipLaunchKernelGGL(kern, dim3(nblk(n)), dim3(256), 0, (c)->stream, __VA_ARGS__); \
      HIPCHK(c, hipGetLastError());                                                    \
    }                                                                                  \
  } while (0)
// the same with the grid padded to a multiple of 8 blocks (kernels indexed by xgid)
#define LAUNCH_X(c, kern, n, ...)                                                        \
  do {                                                                                 \
    if ((n) > 0) {                                                                     \
      hipLaunchKernelGGL(kern, dim3((nblk(n) + 7u) & ~7u), dim3(256), 0, (c)->stream, __VA_ARGS__); \
      HIPCHK(c, hipGetLastError());                                                    \
    }                                                                                  \
  } while (0)

// LAUNCH_X timed as kernel `id` when fvm_kernel_timing is on: events around the
// launch on the context's stream, waited for, the elapsed time added up
#define LAUNCH_T(c, id, kern, n, ...)                                                   \
  do {                                                                                  \
    if ((n) > 0 && (c)->kt.on) HIPCHK(c, hipEventRecord((c)->kt.ev[0], (c)->stream));   \
    LAUNCH_X(c, kern, n, __VA_ARGS__);                                                  \
    if ((n) > 0 && (c)->kt.on) {                                                        \
      HIPCHK(c, hipEventRecord((c)->kt.ev[1], (c)->stream));                            \
      HIPCHK(c, hipEventSynchronize((c)->kt.ev[1]));                                    \
      float ms_ = 0.0f;                                                                 \
      HIPCHK(c, hipEventElapsedTime(&ms_, (c)->kt.ev[0], (c)->kt.ev[1]));               \
      (c)->kt.ms[id] += ms_;                                                            \
      (c)->kt.launches[id] += 1;                                                        \
    }                                                                                   \
  } while (0)

static int check_params(const fvm_params *p, std::string &why) {
  if (!p) { why = "params is NULL"; return FVM_EARG; }
  if (!(p->gamma_gas > 0.0)) { why = "gamma_gas must be > 0"; return FVM_EARG; }
  if (!(p->courant_no > 0.0)) { why = "courant_no must be > 0"; return FVM_EARG; }
  for (int d = 0; d < 3; d++)
    if (!(p->domain_size[d] > 0.0)) { why = "domain_size must be > 0"; return FVM_EARG; }
  if (p->limiter_mode < 0 || p->limiter_mode > 2) { why = "limiter_mode out of range"; return FVM_EARG; }
  if (p->storage != FVM_STORAGE_F64 && p->storage != FVM_STORAGE_SHIPPED) { why = "storage out of range"; return FVM_EARG; }
  return FVM_OK;
}

// Entry points: C linkage comes from the declarations in fvm_gpu.h.

int fvm_create(fvm_ctx **out, int device, const fvm_params *params) {
  if (!out) return FVM_EARG;
  *out = nullptr;
  std::string why;
  if (check_params(params, why) != FVM_OK) return FVM_EARG;
  fvm_ctx *c = nullptr;
  try {
    c = new fvm_ctx;
  } catch (...) {
    return FVM_EARG;
  }
  c->device = device;
  c->prm = *params;
  hipError_t e = hipSetDevice(device);
  if (e != hipSuccess) {
    delete c;
    return FVM_EHIP;
  }
  e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking);
  if (e != hipSuccess) {
    delete c;
    return FVM_EHIP;
  }
  if (ensure(c, c->diag, sizeof(unsigned long long) * FVM_NDIAG) != FVM_OK ||
      ensure(c, c->scalars, sizeof(unsigned long long) * 8) != FVM_OK) {
    (void)hipStreamDestroy(c->stream);
    delete c;
    return FVM_EHIP;
  }
  (void)hipMemsetAsync(c->diag.p, 0, c->diag.bytes, c->stream);
  fvm_xfer_ref();
  if (noalloc_scratch_init(device) != FVM_OK || hipHostMalloc((void **)&c->pin, (size_t)1 << 20, hipHostMallocDefault) != hipSuccess ||
      hipEventCreateWithFlags(&c->pin_ev[0], hipEventDisableTiming) != hipSuccess ||
      hipEventCreateWithFlags(&c->pin_ev[1], hipEventDisableTiming) != hipSuccess) {
    (void)fvm_destroy(c);
    return FVM_EHIP;
  }
  *out = c;
  return FVM_OK;
}

int fvm_destroy(fvm_ctx *c) {
  if (!c) return FVM_EARG;
  (void)hipSetDevice(c->device);
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  for (auto &b : c->field) release(b);
  for (DBuf *b : {&c->m_s1, &c->m_s2, &c->m_fpos, &c->m_cn, &c->m_coff, &c->m_cface, &c->m_cnbr, &c->m_cvol, &c->m_fact,
                  &c->m_soff, &c->m_sent, &c->rec, &c->crow, &c->tmp0, &c->tmp1, &c->tmp2, &c->stage,
                  &c->diag, &c->scalars})
    release(*b);
  fvm::scan_release(c->scan);
  fvm_fast_release(c);
  fvm_substep_release(c);
  for (hipEvent_t e : c->pin_ev)
    if (e) (void)hipEventDestroy(e);
  if (c->pin) (void)hipHostFree(c->pin);
  fvm_xfer_unref(c);
  for (hipEvent_t &e : c->kt.ev)
    if (e) (void)hipEventDestroy(e);
  if (c->stream) (void)hipStreamDestroy(c->stream);
  delete c;
  return FVM_OK;
}

int fvm_kernel_timing(fvm_ctx *c, int enable) {
  if (!c) return FVM_EARG;
  HIPCHK(c, hipSetDevice(c->device));
  for (hipEvent_t &e : c->kt.ev)
    if (!e) HIPCHK(c, hipEventCreate(&e));
  c->kt.on = enable != 0;
  for (int k = 0; k < FVM_NKT; k++) {
    c->kt.ms[k] = 0.0;
    c->kt.launches[k] = 0;
  }
  return FVM_OK;
}

int fvm_kernel_ms(fvm_ctx *c, double *ms, long long *launches, int n) {
  if (!c) return FVM_EARG;
  if (n < 0 || n > FVM_NKT || (n > 0 && (!ms || !launches))) return fvm_fail(c, FVM_EARG, "fvm_kernel_ms: bad n or null output");
  for (int k = 0; k < n; k++) {
    ms[k] = c->kt.ms[k];
    launches[k] = c->kt.launches[k];
  }
  return FVM_OK;
}

const char *fvm_last_error(const fvm_ctx *c) { return c ? c->err.c_str() : "null context"; }

int fvm_set_params(fvm_ctx *c, const fvm_params *p) {
  if (!c) return FVM_EARG;
  std::string why;
  if (check_params(p, why) != FVM_OK) return fail(c, FVM_EARG, why);
  if (c->have_mesh && p->storage != c->prm.storage)
    return fail(c, FVM_ESTATE, "storage mode cannot change after fvm_upload_mesh");
  c->prm = *p;
  return FVM_OK;
}

int fvm_set_time(fvm_ctx *c, double t) {
  if (!c) return FVM_EARG;
  c->t_global = t;
  return FVM_OK;
}

namespace fvm {
// Complete cell lists: every face appears exactly once in the list of its s1
// when s1 is active and exactly once in the list of its s2 when s2 is active
// (localMesh.cpp:586-589).  Checked per (cell, face) pair; the lists must
// already be known to hold only faces their cell owns.
bool lists_complete(int nactive, int nface, const fvm_face *faces, const int *cell_face_off, const int *cell_face) {
  try {
    std::vector<unsigned char> under1(nface, 0), under2(nface, 0);
    for (int i = 0; i < nactive; i++)
      for (int e = cell_face_off[i]; e < cell_face_off[i + 1]; e++) {
        const int f = cell_face[e];
        unsigned char &u = faces[f].s1 == i ? under1[f] : under2[f];
        if (u) return false;  // listed twice under the same cell
        u = 1;
      }
    for (int f = 0; f < nface; f++)
      if (under1[f] != (faces[f].s1 < nactive) || under2[f] != (faces[f].s2 < nactive)) return false;
  } catch (...) {
    return false;
  }
  return true;
}
}  // namespace fvm

int fvm_upload_mesh(fvm_ctx *c, int np, int nactive, int nimport_loc, int nface, const fvm_face *faces,
                    const int *cell_face_off, const int *cell_face, const double *cell_volume) {
  if (!c) return FVM_EARG;
  if (np <= 0 || nactive < 0 || nactive > np || nimport_loc < 0 || nactive + nimport_loc > np || nface < 0)
    return fail(c, FVM_EARG, "fvm_upload_mesh: inconsistent sizes");
  if ((nface > 0 && !faces) || !cell_face_off || (nactive > 0 && !cell_volume))
    return fail(c, FVM_EARG, "fvm_upload_mesh: NULL array");
  // host-side validation of every index the kernels will follow
  const int nref = cell_face_off[nactive];
  if (cell_face_off[0] != 0 || nref < 0 || (nref > 0 && !cell_face))
    return fail(c, FVM_EARG, "fvm_upload_mesh: bad cell_face_off");
  for (int i = 0; i < nactive; i++)
    if (cell_face_off[i + 1] < cell_face_off[i]) return fail(c, FVM_EARG, "fvm_upload_mesh: cell_face_off not monotone");
  for (int e = 0; e < nref; e++)
    if (cell_face[e] < 0 || cell_face[e] >= nface) return fail(c, FVM_EARG, "fvm_upload_mesh: cell_face index out of range");
  for (int f = 0; f < nface; f++)
    if (faces[f].s1 < 0 || faces[f].s1 >= np || faces[f].s2 < 0 || faces[f].s2 >= np || faces[f].s1 == faces[f].s2)
      return fail(c, FVM_EARG, "fvm_upload_mesh: face cell index out of range");
  for (int i = 0; i < nactive; i++)
    for (int e = cell_face_off[i]; e < cell_face_off[i + 1]; e++) {
      const fvm_face &F = faces[cell_face[e]];
      if (F.s1 != i && F.s2 != i) return fail(c, FVM_EARG, "fvm_upload_mesh: cell lists a face it does not own");
    }
  bool complete = fvm::lists_complete(nactive, nface, faces, cell_face_off, cell_face);
  (void)hipSetDevice(c->device);
  fvm_fast_release(c);   // the fused state belongs to the previous mesh
  c->have_mesh = false;  // until the new mesh is complete
  c->sub_layout = false;
  c->lists_complete = complete;
  const bool resize = np != c->np;
  c->np = np;
  c->nactive = nactive;
  c->nimport_loc = nimport_loc;
  c->nface = nface;
  c->nref = nref;
  c->nfa = -1;
  for (int f = 0; f < FVM_NFIELDS; f++) {
    const size_t bytes = field_bytes(c, f, np);
    if (resize || c->field[f].bytes < bytes) {
      int rc = ensure(c, c->field[f], bytes);
      if (rc) return rc;
      HIPCHK(c, hipMemsetAsync(c->field[f].p, 0, bytes, c->stream));
    }
  }
  int rc;
  if ((rc = ensure(c, c->m_s1, sizeof(int) * (size_t)nface)) || (rc = ensure(c, c->m_s2, sizeof(int) * (size_t)nface)) ||
      (rc = ensure(c, c->m_cn, sizeof(double) * 6 * (size_t)nface + 8)) ||
      (rc = ensure(c, c->m_coff, sizeof(int) * (size_t)(nactive + 1))) || (rc = ensure(c, c->m_cface, sizeof(int) * (size_t)nref)) ||
      (rc = ensure(c, c->m_cnbr, sizeof(int) * (size_t)nref)) ||
      (rc = ensure(c, c->m_cvol, sizeof(double) * (size_t)nactive)) || (rc = ensure(c, c->stage, sizeof(fvm_face) * (size_t)nface)))
    return rc;
  if (nface > 0) {
    if ((rc = fvm_to_device(c, c->stage.p, faces, sizeof(fvm_face) * (size_t)nface))) return rc;
    LAUNCH(c, fvm::k_split_faces, nface, (const fvm_face *)c->stage.p, nface, (int *)c->m_s1.p, (int *)c->m_s2.p,
           (double *)c->m_cn.p);
  }
  HIPCHK(c, hipMemcpyAsync(c->m_coff.p, cell_face_off, sizeof(int) * (size_t)(nactive + 1), hipMemcpyHostToDevice, c->stream));
  if (nref > 0 && (rc = fvm_to_device(c, c->m_cface.p, cell_face, sizeof(int) * (size_t)nref))) return rc;
  if (nactive > 0) HIPCHK(c, hipMemcpyAsync(c->m_cvol.p, cell_volume, sizeof(double) * (size_t)nactive, hipMemcpyHostToDevice, c->stream));
  LAUNCH(c, fvm::k_cell_nbr, fvm::cell_lanes(nactive), (const int *)c->m_coff.p, (const int *)c->m_cface.p,
         (const int *)c->m_s1.p, (const int *)c->m_s2.p, nactive, (int *)c->m_cnbr.p);
  HIPCHK(c, hipStreamSynchronize(c->stream));
  c->have_mesh = true;
  return FVM_OK;
}

int fvm_upload_faces(fvm_ctx *c, int np, int nactive, int nimport_loc, int nface, const fvm_face *faces,
                     const double *cell_volume) {
  if (!c) return FVM_EARG;
  if (np <= 0 || nactive < 0 || nactive > np || nimport_loc < 0 || nactive + nimport_loc > np || nface < 0)
    return fail(c, FVM_EARG, "fvm_upload_faces: inconsistent sizes");
  if ((nface > 0 && !faces) || (nactive > 0 && !cell_volume)) return fail(c, FVM_EARG, "fvm_upload_faces: NULL array");
  // every face is created by an active cell (its s1); s2 may be any local cell
  for (int f = 0; f < nface; f++)
    if (faces[f].s1 < 0 || faces[f].s1 >= nactive || faces[f].s2 < 0 || faces[f].s2 >= np || faces[f].s1 == faces[f].s2)
      return fail(c, FVM_EARG, "fvm_upload_faces: face cell index out of range (s1 must be active)");
  (void)hipSetDevice(c->device);
  fvm_fast_release(c);   // the fused state belongs to the previous mesh
  c->have_mesh = false;  // until the new mesh is complete
  c->sub_layout = false;
  c->lists_complete = true;  // built below, every face under each active cell
  const bool resize = np != c->np;
  for (int f = 0; f < FVM_NFIELDS; f++) {
    const size_t bytes = field_bytes(c, f, np);
    if (resize || c->field[f].bytes < bytes) {
      int rc = ensure(c, c->field[f], bytes);
      if (rc) return rc;
      HIPCHK(c, hipMemsetAsync(c->field[f].p, 0, bytes, c->stream));
    }
  }
  int rc;
  if ((rc = ensure(c, c->m_s1, sizeof(int) * (size_t)nface)) || (rc = ensure(c, c->m_s2, sizeof(int) * (size_t)nface)) ||
      (rc = ensure(c, c->m_cn, sizeof(double) * 6 * (size_t)nface + 8)) ||
      (rc = ensure(c, c->m_coff, sizeof(int) * (size_t)(nactive + 1))) || (rc = ensure(c, c->m_cface, sizeof(int) * 2 * (size_t)nface + 4)) ||
      (rc = ensure(c, c->m_cnbr, sizeof(int) * 2 * (size_t)nface + 4)) ||
      (rc = ensure(c, c->m_cvol, sizeof(double) * (size_t)nactive + 8)) || (rc = ensure(c, c->stage, sizeof(fvm_face) * (size_t)nface + 8)) ||
      (rc = ensure(c, c->tmp0, sizeof(int) * (size_t)(nactive + 1))) || (rc = ensure(c, c->tmp1, sizeof(int) * (size_t)(nactive + 1))))
    return rc;
  int *cnt = (int *)c->tmp0.p, *cursor = (int *)c->tmp1.p;
  LAUNCH(c, fvm::k_fill_int, nactive + 1, cnt, 0, nactive + 1);
  if (nface > 0) {
    if ((rc = fvm_to_device(c, c->stage.p, faces, sizeof(fvm_face) * (size_t)nface))) return rc;
    LAUNCH(c, fvm::k_split_faces, nface, (const fvm_face *)c->stage.p, nface, (int *)c->m_s1.p, (int *)c->m_s2.p,
           (double *)c->m_cn.p);
    LAUNCH(c, fvm::k_csr_count, nface, (const int *)c->m_s1.p, (const int *)c->m_s2.p, nface, nactive, cnt);
  }
  if (fvm::exclusive_scan(c->scan, cnt, (int *)c->m_coff.p, nactive + 1, c->stream))
    return fail(c, FVM_EHIP, "fvm_upload_faces: scan failed");
  int nref = 0;
  HIPCHK(c, hipMemcpyAsync(&nref, (int *)c->m_coff.p + nactive, sizeof(int), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipMemcpyAsync(cursor, c->m_coff.p, sizeof(int) * (size_t)(nactive + 1), hipMemcpyDeviceToDevice, c->stream));
  if (nface > 0) {
    LAUNCH(c, fvm::k_csr_fill, nface, (const int *)c->m_s1.p, (const int *)c->m_s2.p, nface, nactive, cursor,
           (int *)c->m_cface.p);
    LAUNCH(c, fvm::k_csr_sort, fvm::cell_lanes(nactive), (const int *)c->m_coff.p, nactive, (int *)c->m_cface.p);
    LAUNCH(c, fvm::k_cell_nbr, fvm::cell_lanes(nactive), (const int *)c->m_coff.p, (const int *)c->m_cface.p,
           (const int *)c->m_s1.p, (const int *)c->m_s2.p, nactive, (int *)c->m_cnbr.p);
  }
  if (nactive > 0) HIPCHK(c, hipMemcpyAsync(c->m_cvol.p, cell_volume, sizeof(double) * (size_t)nactive, hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  c->np = np;
  c->nactive = nactive;
  c->nimport_loc = nimport_loc;
  c->nface = nface;
  c->nref = nref;
  c->nfa = -1;
  c->have_mesh = true;
  return FVM_OK;
}

int fvm_download_cell_faces(fvm_ctx *c, int *cell_face_off, int *cell_face) {
  if (!c) return FVM_EARG;
  if (!c->have_mesh) return fail(c, FVM_ESTATE, "fvm_download_cell_faces before a mesh upload");
  if (!cell_face_off && !cell_face) return fail(c, FVM_EARG, "fvm_download_cell_faces: NULL arrays");
  (void)hipSetDevice(c->device);
  if (cell_face_off)
    HIPCHK(c, hipMemcpy(cell_face_off, c->m_coff.p, sizeof(int) * (size_t)(c->nactive + 1), hipMemcpyDeviceToHost));
  if (cell_face && c->nref > 0)
    HIPCHK(c, hipMemcpy(cell_face, c->m_cface.p, sizeof(int) * (size_t)c->nref, hipMemcpyDeviceToHost));
  return FVM_OK;
}

int fvm_upload_field(fvm_ctx *c, int field, const void *host, int np) {
  if (!c) return FVM_EARG;
  if (!c->have_mesh) return fail(c, FVM_ESTATE, "fvm_upload_field before fvm_upload_mesh");
  if (field < 0 || field >= FVM_NFIELDS) return fail(c, FVM_EARG, "fvm_upload_field: unknown field");
  if (np != c->np || !host) return fail(c, FVM_EARG, "fvm_upload_field: np mismatch or NULL");
  (void)hipSetDevice(c->device);
  const auto &fi = fvm::kFields[field];
  if (fi.kind == fvm::K_INT) {
    HIPCHK(c, hipMemcpyAsync(c->field[field].p, host, sizeof(int) * (size_t)np, hipMemcpyHostToDevice, c->stream));
  } else {
    const size_t bytes = sizeof(double) * (size_t)fi.width * (size_t)np;
    int rc = ensure(c, c->stage, bytes);
    if (rc) return rc;
    if ((rc = fvm_to_device(c, c->stage.p, host, bytes))) return rc;
    if (fi.kind == fvm::K_STORE && c->prm.storage == FVM_STORAGE_SHIPPED)
      LAUNCH(c, fvm::k_aos_to_soa<float>, np, (const double *)c->stage.p, (float *)c->field[field].p, np, fi.width);
    else
      LAUNCH(c, fvm::k_aos_to_soa<double>, np, (const double *)c->stage.p, (double *)c->field[field].p, np, fi.width);
  }
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return FVM_OK;
}

int fvm_download_field(fvm_ctx *c, int field, void *host, int np) {
  if (!c) return FVM_EARG;
  if (!c->have_mesh) return fail(c, FVM_ESTATE, "fvm_download_field before fvm_upload_mesh");
  if (field < 0 || field >= FVM_NFIELDS) return fail(c, FVM_EARG, "fvm_download_field: unknown field");
  if (np != c->np || !host) return fail(c, FVM_EARG, "fvm_download_field: np mismatch or NULL");
  (void)hipSetDevice(c->device);
  const auto &fi = fvm::kFields[field];
  if (fi.kind == fvm::K_INT) {
    HIPCHK(c, hipMemcpyAsync(host, c->field[field].p, sizeof(int) * (size_t)np, hipMemcpyDeviceToHost, c->stream));
  } else {
    const size_t bytes = sizeof(double) * (size_t)fi.width * (size_t)np;
    int rc = ensure(c, c->stage, bytes);
    if (rc) return rc;
    if (fi.kind == fvm::K_STORE && c->prm.storage == FVM_STORAGE_SHIPPED)
      LAUNCH(c, fvm::k_soa_to_aos<float>, np, (const float *)c->field[field].p, (double *)c->stage.p, np, fi.width);
    else
      LAUNCH(c, fvm::k_soa_to_aos<double>, np, (const double *)c->field[field].p, (double *)c->stage.p, np, fi.width);
    return fvm_to_host(c, host, c->stage.p, bytes);
  }
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return FVM_OK;
}

// Face-end lists of every cell over the current face_active_list: from the
// cells' lists when every cell has a complete one (fpos: the faces' places in
// the active list), otherwise by counting over the active faces
static int build_face_ends(fvm_ctx *c, bool from_lists) {
  const int np = c->np, nfa = c->nfa;
  int rc;
  if ((rc = ensure(c, c->m_soff, sizeof(int) * (size_t)(np + 1))) || (rc = ensure(c, c->m_sent, sizeof(int) * 2 * (size_t)nfa + 4)) ||
      (rc = ensure(c, c->tmp0, sizeof(int) * (size_t)(np + 1))))
    return rc;
  int *cnt = (int *)c->tmp0.p;
  if (from_lists) {
    fvm::EndLists E{};
    E.np = np;
    E.nactive = c->nactive;
    E.coff = (const int *)c->m_coff.p;
    E.cface = (const int *)c->m_cface.p;
    E.s1 = (const int *)c->m_s1.p;
    E.fpos = (const int *)c->m_fpos.p;
    if (c->sub_layout) {
      E.perm = (const int *)c->sub.perm.p;
      E.goff = (const int *)c->sub.goff.p;
      E.gface = (const int *)c->sub.gface.p;
      E.gmark = (const int *)c->sub.fmark.p;
      E.gpos = (const int *)c->sub.fpos.p;
    }
    LAUNCH_X(c, fvm::k_end_lists<true>, fvm::cell_lanes(np), E, cnt, nullptr, nullptr);
    if (fvm::exclusive_scan(c->scan, cnt, (int *)c->m_soff.p, np, c->stream, true)) return fail(c, FVM_EHIP, "scan failed");
    LAUNCH_X(c, fvm::k_end_lists<false>, fvm::cell_lanes(np), E, nullptr, (const int *)c->m_soff.p, (int *)c->m_sent.p);
    return FVM_OK;
  }
  HIPCHK(c, hipMemsetAsync(cnt, 0, sizeof(int) * (size_t)(np + 1), c->stream));
  fvm::MeshView M = meshview(c);
  LAUNCH(c, fvm::k_end_count, nfa, M, cnt);
  rc = fvm::exclusive_scan(c->scan, cnt, (int *)c->m_soff.p, np + 1, c->stream);
  if (rc) return fail(c, FVM_EHIP, "scan failed");
  HIPCHK(c, hipMemcpyAsync(cnt, c->m_soff.p, sizeof(int) * (size_t)(np + 1), hipMemcpyDeviceToDevice, c->stream));
  M = meshview(c);
  LAUNCH(c, fvm::k_end_fill, nfa, M, cnt, (int *)c->m_sent.p);
  LAUNCH(c, fvm::k_end_sort, np, (const int *)c->m_soff.p, (int *)c->m_sent.p, np);
  return FVM_OK;
}

int fvm_get_active_faces(fvm_ctx *c, int *nface_active) {
  if (!c || !nface_active) return FVM_EARG;
  if (!c->have_mesh) return fail(c, FVM_ESTATE, "fvm_get_active_faces before fvm_upload_mesh");
  (void)hipSetDevice(c->device);
  const int nref = c->nref;
  int rc;
  if ((rc = ensure(c, c->tmp1, sizeof(int) * ((size_t)std::max(c->nface, nref) + 1))) ||
      (rc = ensure(c, c->tmp2, sizeof(int) * ((size_t)nref + 1))) || (rc = ensure(c, c->tmp0, sizeof(int) * ((size_t)nref + 1))) ||
      (rc = ensure(c, c->m_fact, sizeof(int) * ((size_t)c->nface + 1))) ||
      (rc = ensure(c, c->m_fpos, sizeof(int) * ((size_t)c->nface + 1))))
    return rc;
  int *firstpos = (int *)c->tmp1.p, *flag = (int *)c->tmp2.p, *pos = (int *)c->tmp0.p, *fpos = (int *)c->m_fpos.p;
  fvm::MeshView M = meshview(c);
  if (c->lists_complete) {
    LAUNCH(c, fvm::k_face_firstflag_direct, fvm::cell_lanes(c->nactive), M, (const int *)c->field[FVM_FIELD_BND].p, c->nactive, flag);
  } else {
    LAUNCH(c, fvm::k_fill_int, c->nface, firstpos, INT_MAX, c->nface);
    LAUNCH(c, fvm::k_face_firstpos, c->nactive, M, (const int *)c->field[FVM_FIELD_BND].p, c->nactive, firstpos);
    LAUNCH(c, fvm::k_face_firstflag, c->nactive, M, (const int *)c->field[FVM_FIELD_BND].p, c->nactive, firstpos, flag);
  }
  // within a substep without boundary cells every face of its complete lists is
  // active: has_bnd tells what the layout was gathered from, which a caller may
  // have replaced since, on either side
  const bool all = c->lists_complete && c->sub_layout && c->defer_sync && !c->sub.has_bnd;
  int total = all ? c->nface : 0;
  if (!all) LAUNCH(c, fvm::k_fill_int, c->nface, fpos, -1, c->nface);
  if (nref > 0) {
    rc = fvm::exclusive_scan_flags(c->scan, flag, pos, nref, all ? nullptr : &total, c->stream);
    if (rc) return fail(c, FVM_EHIP, "flag scan failed");
    LAUNCH(c, fvm::k_face_compact, nref, M, flag, pos, nref, (int *)c->m_fact.p, fpos);
  }
  c->nfa = total;
  rc = build_face_ends(c, c->lists_complete && (c->nactive == c->np || c->sub_layout));
  if (rc) return rc;
  if ((rc = finish(c))) return rc;
  *nface_active = total;
  return FVM_OK;
}

int fvm_set_active_faces(fvm_ctx *c, int nfa, const int *face_active) {
  if (!c) return FVM_EARG;
  if (!c->have_mesh) return fail(c, FVM_ESTATE, "fvm_set_active_faces before fvm_upload_mesh");
  if (nfa < 0 || nfa > c->nface || (nfa > 0 && !face_active)) return fail(c, FVM_EARG, "fvm_set_active_faces: bad size");
  for (int a = 0; a < nfa; a++)
    if (face_active[a] < 0 || face_active[a] >= c->nface) return fail(c, FVM_EARG, "fvm_set_active_faces: index out of range");
  (void)hipSetDevice(c->device);
  int rc = ensure(c, c->m_fact, sizeof(int) * ((size_t)nfa + 1));
  if (rc) return rc;
  if (nfa > 0) HIPCHK(c, hipMemcpyAsync(c->m_fact.p, face_active, sizeof(int) * (size_t)nfa, hipMemcpyHostToDevice, c->stream));
  c->nfa = nfa;
  rc = build_face_ends(c, false);  // the list may name a face more than once
  if (rc) return rc;
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return FVM_OK;
}

int fvm_download_active_faces(fvm_ctx *c, int *face_active, int n) {
  if (!c) return FVM_EARG;
  if (c->nfa < 0) return fail(c, FVM_ESTATE, "no active face list");
  if (n != c->nfa || (n > 0 && !face_active)) return fail(c, FVM_EARG, "fvm_download_active_faces: size mismatch");
  (void)hipSetDevice(c->device);
  if (n > 0) HIPCHK(c, hipMemcpyAsync(face_active, c->m_fact.p, sizeof(int) * (size_t)n, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return FVM_OK;
}

// Rounds of four cells a wavefront takes in the two-phase cell kernels: as many
// as leave about four wavefronts for each of the 1024 SIMDs, since the second
// phase uses one lane per cell (16 rounds: all 64 lanes).
// Measured: the CFL kernel on 97,000 cells 33 us with 4 rounds (45 us as a thread
// per cell), on a 14,000-cell mesh's active sets 8 us with one (29 us).
static int cell_rounds(int n) { return n >= 262144 ? 16 : n >= 65536 ? 4 : 1; }
static long rounds_threads(int n, int R) { return ((long)n + 4 * R - 1) / (4 * R) * 64; }

#define DISPATCH(c, fn, ...)                                   \
  ((c)->prm.storage == FVM_STORAGE_SHIPPED ? fn<float>(__VA_ARGS__) : fn<double>(__VA_ARGS__))

template <typename S> static int do_reconstruction(fvm_ctx *c) {
  LAUNCH_T(c, FVM_KT_RECONSTRUCTION, fvm::k_reconstruction<S>, fvm::cell_lanes(c->nactive), cells<S>(c), meshview(c), phys(c));
  return finish(c);
}
int fvm_compute_reconstruction(fvm_ctx *c) {
  if (!c) return FVM_EARG;
  if (!c->have_mesh) return fail(c, FVM_ESTATE, "no mesh");
  (void)hipSetDevice(c->device);
  return DISPATCH(c, do_reconstruction, c);
}

template <typename S> static int do_limiter(fvm_ctx *c) {
  LAUNCH_T(c, FVM_KT_SLOPE_LIMITER, fvm::k_slope_limiter<S>, fvm::cell_lanes(c->np), cells<S>(c), meshview(c), phys(c),
           (unsigned long long *)c->diag.p);
  return finish(c);
}
int fvm_slope_limiter(fvm_ctx *c) {
  if (!c) return FVM_EARG;
  if (!c->have_mesh || c->nfa < 0) return fail(c, FVM_ESTATE, "no mesh or no active face list");
  (void)hipSetDevice(c->device);
  return DISPATCH(c, do_limiter, c);
}

static int read_diag(fvm_ctx *c, unsigned long long *h) {
  HIPCHK(c, hipMemcpyAsync(h, c->diag.p, sizeof(unsigned long long) * FVM_NDIAG, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return FVM_OK;
}

// The cells' rows for the face flux kernel, written on the context's stream, or
// null where it reads the fields: few faces, whose lines stay in the caches while
// the rows cost a launch (300 000 faces: 72 us, with rows 44 + 10; up to 100 000,
// FP32: 14.1, with rows 10.3 + 4.9), or no memory for the rows.
constexpr int ROWS_MIN_FACES = 131072;
bool fvm_cell_row_space(fvm_ctx *c, int np, int nfa) {
  if (nfa < ROWS_MIN_FACES) return false;
  if (ensure(c, c->crow, sizeof(double) * fvm::CROW * (size_t)np) == FVM_OK) return true;
  (void)hipGetLastError();
  return false;
}
template <typename S> static const double *cell_rows(fvm_ctx *c) {
  if (!fvm_cell_row_space(c, c->np, c->nfa)) return nullptr;
  hipLaunchKernelGGL((fvm::k_cell_rows<S>), dim3((unsigned)((c->np + 63) / 64)), dim3(256), 0, c->stream, cells<S>(c),
                     (double *)c->crow.p);
  return (const double *)c->crow.p;
}

template <typename S> static int do_fluid_update(fvm_ctx *c) {
  const int nfa = c->nfa;
  int rc;
  if ((rc = ensure(c, c->rec, sizeof(double) * fvm::NREC * (size_t)nfa))) return rc;
  unsigned long long before[FVM_NDIAG], after[FVM_NDIAG];
  if (!c->defer_sync && (rc = read_diag(c, before))) return rc;
  const double *rows = cell_rows<S>(c);
#define FLUX(F_, R_)                                                                                                   \
  LAUNCH_T(c, FVM_KT_FACE_FLUX, (fvm::k_face_flux<S, F_, R_>), nfa, cells<S>(c), meshview(c), phys(c), rows,             \
           (double *)c->rec.p, (unsigned long long *)c->diag.p)
  if (c->face32 && rows) FLUX(float, true);
  else if (c->face32) FLUX(float, false);
  else if (rows) FLUX(double, true);
  else FLUX(double, false);
#undef FLUX
  LAUNCH_T(c, FVM_KT_SCATTER, fvm::k_scatter<S>, fvm::cell_lanes(c->np), cells<S>(c), meshview(c), (const double *)c->rec.p);
  if (c->defer_sync) return FVM_OK;  // the substep compares the positivity count itself
  if ((rc = read_diag(c, after))) return rc;
  if (after[FVM_DIAG_POSITIVITY] != before[FVM_DIAG_POSITIVITY])
    return fail(c, FVM_EPOS, "computeFluidUpdate: non-positive density or thermal energy at a face");
  return FVM_OK;
}
int fvm_set_face_precision(fvm_ctx *c, int bits) {
  if (!c) return FVM_EARG;
  if (bits != 32 && bits != 64) return fail(c, FVM_EARG, "fvm_set_face_precision: bits must be 32 or 64");
  c->face32 = bits == 32;
  return FVM_OK;
}
int fvm_compute_fluid_update(fvm_ctx *c) {
  if (!c) return FVM_EARG;
  if (!c->have_mesh || c->nfa < 0) return fail(c, FVM_ESTATE, "no mesh or no active face list");
  (void)hipSetDevice(c->device);
  return DISPATCH(c, do_fluid_update, c);
}

template <typename S>
static int do_face_states(fvm_ctx *c, int first, int count, double *wij, double *Wi, double *Wj, int *jbnd,
                          double *normal) {
  const size_t N = (size_t)count;
  const size_t nd = (3 + 10 + 10 + 3) * N;
  int rc = ensure(c, c->stage, sizeof(double) * nd + sizeof(int) * N);
  if (rc) return rc;
  double *d_wij = (double *)c->stage.p, *d_Wi = d_wij + 3 * N, *d_Wj = d_Wi + 10 * N, *d_n = d_Wj + 10 * N;
  int *d_jb = (int *)(d_n + 3 * N);
  LAUNCH(c, fvm::k_face_states<S>, count, cells<S>(c), meshview(c), phys(c), first, count, d_wij, d_Wi, d_Wj, d_jb,
         d_n);
  HIPCHK(c, hipMemcpyAsync(wij, d_wij, sizeof(double) * 3 * N, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipMemcpyAsync(Wi, d_Wi, sizeof(double) * 10 * N, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipMemcpyAsync(Wj, d_Wj, sizeof(double) * 10 * N, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipMemcpyAsync(normal, d_n, sizeof(double) * 3 * N, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipMemcpyAsync(jbnd, d_jb, sizeof(int) * N, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return FVM_OK;
}
int fvm_get_face_states(fvm_ctx *c, int first, int count, double *wij, double *Wi, double *Wj, int *jbnd,
                        double *normal) {
  if (!c) return FVM_EARG;
  if (!c->have_mesh || c->nfa < 0) return fail(c, FVM_ESTATE, "no mesh or no active face list");
  if (first < 0 || count < 0 || first + count > c->nfa) return fail(c, FVM_EARG, "face range outside the active list");
  if (count == 0) return FVM_OK;
  if (!wij || !Wi || !Wj || !jbnd || !normal) return fail(c, FVM_EARG, "NULL array");
  (void)hipSetDevice(c->device);
  return DISPATCH(c, do_face_states, c, first, count, wij, Wi, Wj, jbnd, normal);
}

template <typename S> static int do_primitives(fvm_ctx *c, int flag) {
  LAUNCH_T(c, FVM_KT_PRIMITIVES, fvm::k_primitives<S>, c->nactive, cells<S>(c), meshview(c), phys(c), flag, (unsigned long long *)c->diag.p);
  return finish(c);
}
int fvm_compute_primitives(fvm_ctx *c, int predictor_flag) {
  if (!c) return FVM_EARG;
  if (!c->have_mesh) return fail(c, FVM_ESTATE, "no mesh");
  (void)hipSetDevice(c->device);
  return DISPATCH(c, do_primitives, c, predictor_flag);
}

template <typename S> static int do_timestep(fvm_ctx *c, double *dt_min) {
  unsigned long long *bits = (unsigned long long *)c->scalars.p;
  LAUNCH(c, fvm::k_set_u64, 1, bits, 0x7FF0000000000000ULL);  // +inf
  const int R = cell_rounds(c->nactive);
  const long nt = rounds_threads(c->nactive, R);
  if (R == 16) LAUNCH_T(c, FVM_KT_TIMESTEP, (fvm::k_timestep<S, 16>), nt, cells<S>(c), meshview(c), phys(c), bits);
  else if (R == 4) LAUNCH_T(c, FVM_KT_TIMESTEP, (fvm::k_timestep<S, 4>), nt, cells<S>(c), meshview(c), phys(c), bits);
  else LAUNCH_T(c, FVM_KT_TIMESTEP, (fvm::k_timestep<S, 1>), nt, cells<S>(c), meshview(c), phys(c), bits);
  if (c->defer_sync && !dt_min) return FVM_OK;
  unsigned long long h = 0;
  HIPCHK(c, hipMemcpyAsync(&h, bits, sizeof h, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  if (dt_min) std::memcpy(dt_min, &h, sizeof(double));
  return FVM_OK;
}
int fvm_compute_timestep(fvm_ctx *c, double *dt_min) {
  if (!c) return FVM_EARG;
  if (!c->have_mesh) return fail(c, FVM_ESTATE, "no mesh");
  (void)hipSetDevice(c->device);
  return DISPATCH(c, do_timestep, c, dt_min);
}

int fvm_compute_timestep_limiter(fvm_ctx *c) {
  // Sequential neighbour sweep of computeTimestep.cpp:64-110 (its result
  // depends on the visiting order): runs on the host next to the Scheduler.
  if (!c) return FVM_EARG;
  if (!c->have_mesh) return fail(c, FVM_ESTATE, "no mesh");
  try {
    const int np = c->np, nactive = c->nactive;
    std::vector<double> dt_new(np), tend(np), tbeg(np);
    std::vector<int> is_ngb(np), is_active(np), coff(nactive + 1), cface(c->nref), s1(c->nface), s2(c->nface);
    int rc;
    if ((rc = fvm_download_field(c, FVM_FIELD_DT_NEW, dt_new.data(), np)) || (rc = fvm_download_field(c, FVM_FIELD_TEND, tend.data(), np)) ||
        (rc = fvm_download_field(c, FVM_FIELD_TBEG, tbeg.data(), np)) || (rc = fvm_download_field(c, FVM_FIELD_IS_NGB, is_ngb.data(), np)) ||
        (rc = fvm_download_field(c, FVM_FIELD_IS_ACTIVE, is_active.data(), np)))
      return rc;
    HIPCHK(c, hipMemcpy(coff.data(), c->m_coff.p, sizeof(int) * (size_t)(nactive + 1), hipMemcpyDeviceToHost));
    if (c->nref) HIPCHK(c, hipMemcpy(cface.data(), c->m_cface.p, sizeof(int) * (size_t)c->nref, hipMemcpyDeviceToHost));
    if (c->nface) {
      HIPCHK(c, hipMemcpy(s1.data(), c->m_s1.p, sizeof(int) * (size_t)c->nface, hipMemcpyDeviceToHost));
      HIPCHK(c, hipMemcpy(s2.data(), c->m_s2.p, sizeof(int) * (size_t)c->nface, hipMemcpyDeviceToHost));
    }
    std::vector<double> dti(np, -fvm::REF_HUGE);
    for (int i = 0; i < nactive; i++) dti[i] = dt_new[i];
    for (int i = nactive; i < np; i++)
      if (is_ngb[i]) dti[i] = is_active[i] ? dt_new[i] : tend[i] - tbeg[i];
    const double scale_fac = 2.0;
    for (int i = 0; i < nactive; i++)
      for (int e = coff[i]; e < coff[i + 1]; e++) {
        const int f = cface[e];
        const int j = (i == s1[f]) ? s2[f] : s1[f];
        dti[j] = fvm::smin_h(dti[j], scale_fac * dti[i]);
        dti[i] = fvm::smin_h(dti[i], scale_fac * dti[j]);
      }
    for (int i = 0; i < np; i++)
      if (i < nactive || is_ngb[i]) dt_new[i] = dti[i];
    return fvm_upload_field(c, FVM_FIELD_DT_NEW, dt_new.data(), np);
  } catch (...) {
    return fail(c, FVM_EARG, "fvm_compute_timestep_limiter: host allocation failed");
  }
}

template <typename S> static int do_predictor(fvm_ctx *c, double dtmax, int min_rung) {
  const int nfa = c->nfa;
  int rc;
  if ((rc = ensure(c, c->rec, sizeof(double) * fvm::NREC * (size_t)nfa))) return rc;
  if (c->face32)
    LAUNCH_T(c, FVM_KT_PREDICTOR_FACE, (fvm::k_predictor_face<S, float>), nfa, cells<S>(c), meshview(c), phys(c),
             (double *)c->rec.p, (unsigned long long *)c->diag.p);
  else
    LAUNCH_T(c, FVM_KT_PREDICTOR_FACE, (fvm::k_predictor_face<S, double>), nfa, cells<S>(c), meshview(c), phys(c),
             (double *)c->rec.p, (unsigned long long *)c->diag.p);
  const int R = cell_rounds(c->nactive);
  const long nt = rounds_threads(c->nactive, R);
#define PRED(R_)                                                                                                      \
  LAUNCH_T(c, FVM_KT_PREDICTOR_CELL, (fvm::k_predictor_cell<S, R_>), nt, cells<S>(c), meshview(c), phys(c),             \
           (const double *)c->rec.p, dtmax, min_rung, (unsigned long long *)c->diag.p)
  if (R == 16) PRED(16);
  else if (R == 4) PRED(4);
  else PRED(1);
#undef PRED
  return finish(c);
}
int fvm_compute_predictor(fvm_ctx *c, double dtmax, int min_rung) {
  if (!c) return FVM_EARG;
  if (!c->have_mesh || c->nfa < 0) return fail(c, FVM_ESTATE, "no mesh or no active face list");
  if (!(dtmax > 0.0) || min_rung < 0 || min_rung > 31) return fail(c, FVM_EARG, "bad dtmax/min_rung");
  (void)hipSetDevice(c->device);
  return DISPATCH(c, do_predictor, c, dtmax, min_rung);
}

// faces [f0, f0 + n) of a batch through contiguous staging: in h (host, pinned)
// and d (device) the inputs of the n faces, then their outputs, in the batch's
// array order (FVM_FLUX_BYTES_PER_FACE a face)
namespace {
struct FluxBatch {
  const double *wij, *Wi, *Wj;
  const int *jbnd;
  const double *normal;
  double *psi, *Bn, *flux;
};
constexpr size_t FLUX_IN_D = 26, FLUX_OUT_D = 12;  // doubles in and out per face, and one int in
static_assert(FVM_FLUX_BYTES_PER_FACE == 8 * (FLUX_IN_D + FLUX_OUT_D) + 4, "face bytes");

// in and out of the staging: [n] faces' inputs, outputs, boundary kinds
struct FluxStage {
  double *in, *out;
  int *jb;
};
FluxStage flux_stage(char *h, size_t n) {
  double *in = (double *)h, *out = in + FLUX_IN_D * n;
  return {in, out, (int *)(out + FLUX_OUT_D * n)};
}
void flux_stage_in(const FluxBatch &b, size_t f0, size_t n, const FluxStage &s) {
  std::memcpy(s.in, b.wij + 3 * f0, 24 * n);
  std::memcpy(s.in + 3 * n, b.Wi + 10 * f0, 80 * n);
  std::memcpy(s.in + 13 * n, b.Wj + 10 * f0, 80 * n);
  std::memcpy(s.in + 23 * n, b.normal + 3 * f0, 24 * n);
  std::memcpy(s.jb, b.jbnd + f0, 4 * n);
}
void flux_stage_out(const FluxBatch &b, size_t f0, size_t n, const FluxStage &s) {
  std::memcpy(b.psi + f0, s.out, 8 * n);
  std::memcpy(b.Bn + f0, s.out + n, 8 * n);
  std::memcpy(b.flux + 10 * f0, s.out + 2 * n, 80 * n);
}

// outputs in memory that holds inputs: such a batch is taken up whole before any of
// its results come down, where pieces would read what earlier ones have replaced
bool flux_in_place(const FluxBatch &b, size_t n) {
  const std::pair<const void *, size_t> in[] = {{b.wij, 24 * n}, {b.Wi, 80 * n}, {b.Wj, 80 * n}, {b.jbnd, 4 * n}, {b.normal, 24 * n}},
                                        out[] = {{b.psi, 8 * n}, {b.Bn, 8 * n}, {b.flux, 80 * n}};
  for (const auto &o : out)
    for (const auto &i : in) {
      const uintptr_t a = (uintptr_t)o.first, c = (uintptr_t)i.first;
      if (a < c + i.second && c < a + o.second) return true;
    }
  return false;
}

// every array within reach of the DMA
bool flux_all_pinned(const FluxBatch &b) {
  for (const void *p : {(const void *)b.wij, (const void *)b.Wi, (const void *)b.Wj, (const void *)b.jbnd, (const void *)b.normal,
                        (const void *)b.psi, (const void *)b.Bn, (const void *)b.flux})
    if (fvm_pageable(p)) return false;
  return true;
}

hipError_t flux_chunk(double gamma, const FluxBatch &b, size_t f0, size_t n, char *h, char *d, hipStream_t st) {
  const FluxStage H = flux_stage(h, n), D = flux_stage(d, n);
  flux_stage_in(b, f0, n, H);
  hipError_t e = hipMemcpyAsync(D.in, H.in, 8 * FLUX_IN_D * n, hipMemcpyHostToDevice, st);
  if (e == hipSuccess) e = hipMemcpyAsync(D.jb, H.jb, 4 * n, hipMemcpyHostToDevice, st);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(fvm::k_flux_batch, dim3(nblk((long)n)), dim3(256), 0, st, (int)n, gamma, D.in, D.in + 3 * n, D.in + 13 * n,
                     D.jb, D.in + 23 * n, D.out, D.out + n, D.out + 2 * n);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  e = hipMemcpyAsync(H.out, D.out, 8 * FLUX_OUT_D * n, hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  if (e != hipSuccess) return e;
  flux_stage_out(b, f0, n, H);
  return hipSuccess;
}

// a small batch computed where it lies in pinned memory (h)
hipError_t flux_pinned(double gamma, const FluxBatch &b, size_t n, char *h, hipStream_t st) {
  const FluxStage H = flux_stage(h, n);
  flux_stage_in(b, 0, n, H);
  hipLaunchKernelGGL(fvm::k_flux_pinned, dim3((unsigned)((n + 63) / 64)), dim3(64), 0, st, (int)n, gamma, H.in, H.jb, H.out);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  if (e != hipSuccess) return e;
  flux_stage_out(b, 0, n, H);
  return hipSuccess;
}
// a batch in pieces of at most `piece` faces, in the two halves of h (`half` bytes
// each) in turn: the host fills one half and empties it again while the other
// half's piece is computed
hipError_t flux_pieces(double gamma, const FluxBatch &b, size_t n, size_t piece, char *h, size_t half, hipEvent_t *ev,
                       hipStream_t st) {
  hipError_t e = hipSuccess;
  const size_t np = (n + piece - 1) / piece;
  const auto stage = [&](size_t k) { return flux_stage(h + (k & 1) * half, std::min(piece, n - k * piece)); };
  size_t k = 0;
  for (; k <= np; k++) {
    if (k < np) {
      const size_t m = std::min(piece, n - k * piece);
      const FluxStage H = stage(k);
      flux_stage_in(b, k * piece, m, H);
      hipLaunchKernelGGL(fvm::k_flux_pinned, dim3((unsigned)((m + 63) / 64)), dim3(64), 0, st, (int)m, gamma, H.in, H.jb,
                         H.out);
      if ((e = hipGetLastError()) != hipSuccess || (e = hipEventRecord(ev[k & 1], st)) != hipSuccess) break;
    }
    if (k > 0) {
      if ((e = hipEventSynchronize(ev[(k - 1) & 1])) != hipSuccess) break;
      flux_stage_out(b, (k - 1) * piece, std::min(piece, n - (k - 1) * piece), stage(k - 1));
    }
  }
  if (e != hipSuccess) (void)hipStreamSynchronize(st);  // nothing may still use the halves
  return e;
}
}  // namespace
// faces that fit the context's pinned staging (1 MiB: 3400 faces) and of a chunk
// of a large batch (a transfer slot).  Batches from two chunks up go chunk by chunk
// over the transfer threads, uploads, kernels and downloads overlapping (60 000
// faces 542 us, in pieces 606; 32 000 367 in pieces); those between in pieces
// through the pinned staging (5000 faces 161 -> 76 us, 20 000 334 -> 237, against
// copies of pageable memory).
constexpr int FLUX_PIN = (1 << 20) / FVM_FLUX_BYTES_PER_FACE;
constexpr int FLUX_CHUNK = 16384;
// Batches in arrays that are pinned themselves go whole from about where the DMA's
// own copies overtake the host's into the staging (14 000 faces 172 us whole, 166 in
// pieces; 16 384 182 and 191; 20 000 204 and 231; 60 000 419 and by chunks 480).
constexpr int FLUX_WHOLE_PINNED = 16384;
static_assert((size_t)FLUX_CHUNK * FVM_FLUX_BYTES_PER_FACE <= fvm::kXferSlot, "a chunk fits a slot");

// the batched computeFlux, synchronous.  fixed: device staging with room for n faces
// (FVM_FLUX_BYTES_PER_FACE each), and nothing may be allocated; null: the context's
// staging, where the route has one (without the memory for it a batch goes in
// pieces), and the transfer threads, whose slots and streams are allocated on
// first use
static int flux_batch_staged(fvm_ctx *c, char *fixed, int n, const double *wij, const double *Wi, const double *Wj,
                             const int *jbnd, const double *normal, double *psi, double *Bn, double *flux) {
  const size_t N = (size_t)n;
  const FluxBatch b{wij, Wi, Wj, jbnd, normal, psi, Bn, flux};
  if (n <= FLUX_PIN) {
    HIPCHK(c, flux_pinned(c->prm.gamma_gas, b, N, c->pin, c->stream));
    return FVM_OK;
  }
  const bool in_place = flux_in_place(b, N);
  bool whole = fixed || in_place || (n >= FLUX_WHOLE_PINNED && flux_all_pinned(b));
  char *base = fixed;
  if (!fixed && (whole || n >= 2 * FLUX_CHUNK)) {
    const int rc = ensure(c, c->stage, (size_t)FVM_FLUX_BYTES_PER_FACE * N);
    if (rc && in_place) return rc;
    if (rc) {
      (void)hipGetLastError();
      whole = false;
    } else {
      base = (char *)c->stage.p;
    }
  }
  if (!whole && base) {
    hipError_t err = hipSuccess;
    HIPCHK(c, hipStreamSynchronize(c->stream));  // the staging may be in use by work before this call
    if (fvm_xfer_chunks(c, (n + FLUX_CHUNK - 1) / FLUX_CHUNK, [&](int k, char *slot, hipStream_t st) {
          const size_t f0 = (size_t)k * FLUX_CHUNK, m = std::min<size_t>(N - f0, FLUX_CHUNK);
          return flux_chunk(c->prm.gamma_gas, b, f0, m, slot, base + f0 * FVM_FLUX_BYTES_PER_FACE, st);
        }, &err)) {
      HIPCHK(c, err);
      return FVM_OK;
    }
  }
  if (!whole) {
    HIPCHK(c, flux_pieces(c->prm.gamma_gas, b, N, FLUX_PIN / 2, c->pin, (size_t)1 << 19, c->pin_ev, c->stream));
    return FVM_OK;
  }
  // whole through the device staging: fvm_compute_flux_noalloc past the pinned
  // staging (its fixed device array), batches computed in place and large ones in
  // pinned arrays
  double *d_wij = (double *)base, *d_Wi = d_wij + 3 * N, *d_Wj = d_Wi + 10 * N, *d_n = d_Wj + 10 * N, *d_psi = d_n + 3 * N,
         *d_Bn = d_psi + N, *d_flux = d_Bn + N;
  int *d_jb = (int *)(d_flux + 10 * N);
  HIPCHK(c, hipMemcpyAsync(d_wij, wij, sizeof(double) * 3 * N, hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipMemcpyAsync(d_Wi, Wi, sizeof(double) * 10 * N, hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipMemcpyAsync(d_Wj, Wj, sizeof(double) * 10 * N, hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipMemcpyAsync(d_n, normal, sizeof(double) * 3 * N, hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipMemcpyAsync(d_jb, jbnd, sizeof(int) * N, hipMemcpyHostToDevice, c->stream));
  LAUNCH(c, fvm::k_flux_batch, n, n, c->prm.gamma_gas, d_wij, d_Wi, d_Wj, d_jb, d_n, d_psi, d_Bn, d_flux);
  HIPCHK(c, hipMemcpyAsync(psi, d_psi, sizeof(double) * N, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipMemcpyAsync(Bn, d_Bn, sizeof(double) * N, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipMemcpyAsync(flux, d_flux, sizeof(double) * 10 * N, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return FVM_OK;
}

int fvm_compute_flux(fvm_ctx *c, int n, const double *wij, const double *Wi, const double *Wj, const int *jbnd,
                     const double *normal, double *psi, double *Bn, double *flux) {
  if (!c) return FVM_EARG;
  if (n < 0) return fail(c, FVM_EARG, "n < 0");
  if (n == 0) return FVM_OK;
  if (!wij || !Wi || !Wj || !jbnd || !normal || !psi || !Bn || !flux) return fail(c, FVM_EARG, "NULL array");
  (void)hipSetDevice(c->device);
  return flux_batch_staged(c, nullptr, n, wij, Wi, Wj, jbnd, normal, psi, Bn, flux);
}

int fvm_compute_flux_noalloc(fvm_ctx *c, int n, const double *wij, const double *Wi, const double *Wj,
                             const int *jbnd, const double *normal, double *psi, double *Bn, double *flux) {
  if (!c) return FVM_EARG;
  if (n < 0) return fail(c, FVM_EARG, "n < 0");
  if (n > FVM_FLUX_NOALLOC_MAX)
    return fail(c, FVM_EARG, "fvm_compute_flux_noalloc: n = " + std::to_string(n) + " exceeds FVM_FLUX_NOALLOC_MAX = " +
                                 std::to_string(FVM_FLUX_NOALLOC_MAX) + " faces");
  if (n == 0) return FVM_OK;
  if (!wij || !Wi || !Wj || !jbnd || !normal || !psi || !Bn || !flux) return fail(c, FVM_EARG, "NULL array");
  (void)hipSetDevice(c->device);
  char *base = (char *)noalloc_scratch(c->device);
  if (!base) return fail(c, FVM_ESTATE, "fvm_compute_flux_noalloc: no staging address for this device");
  return flux_batch_staged(c, base, n, wij, Wi, Wj, jbnd, normal, psi, Bn, flux);
}

int fvm_get_diagnostics(fvm_ctx *c, long long *out, int n) {
  if (!c || !out || n < 0) return FVM_EARG;
  (void)hipSetDevice(c->device);
  unsigned long long h[FVM_NDIAG];
  int rc = read_diag(c, h);
  if (rc) return rc;
  for (int k = 0; k < n && k < FVM_NDIAG; k++) out[k] = (long long)h[k];
  return FVM_OK;
}

int fvm_reset_diagnostics(fvm_ctx *c) {
  if (!c) return FVM_EARG;
  (void)hipSetDevice(c->device);
  HIPCHK(c, hipMemsetAsync(c->diag.p, 0, c->diag.bytes, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return FVM_OK;
}

int fvm_synchronize(fvm_ctx *c) {
  if (!c) return FVM_EARG;
  (void)hipSetDevice(c->device);
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return FVM_OK;
}

