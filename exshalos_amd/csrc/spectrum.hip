// Mass assignment and power-spectrum estimator (gfx950).
//
//  k_deposit     NGP / CIC / TSC scatter of particles (and of the copy
//                shifted by -Lb/2 for interlacing) with device-scope atomics
//                (gridmodule.c:9-53, 146-270); float atomics in FP32, double
//                atomics in FP64
//  k_deposit_tiles  the same weights for particles in Lagrangian lattice
//                order, accumulated per lattice tile in LDS (double) and
//                flushed with one coalesced atomic per touched cell
//  k_normalise   rho / rho_bar - 1 for unweighted grids (gridmodule.c:197-202)
//  k_bin_*       the same weights for particles in any order, listed by grid
//                tiles and summed per tile in LDS
//  k_power_lines, k_power_bins  one pass over the half-complex modes of one
//                tracer's or all tracers' grids:
//                interlacing combine, window deconvolution and Normk
//                (spectrum_h.c:112-157), the reference's mode mask and bin
//                index (powermodule.c:47-55), and the pair products times
//                P_2l(mu) (powermodule.c:66-72).  One tracer: each lane sums
//                along j and adds where its bin changes.  Several: along a
//                row the bin index never
//                decreases, so bins are summed by a segmented scan across
//                the 64 lanes and added by the segment's last lane into a
//                wave-private LDS accumulator.  Waves and blocks are then
//                reduced in a fixed order: the double sums are bit-for-bit
//                reproducible (of one tracer as far as the LDS adds the lanes
//                of one instruction in a fixed order).
#include "common.hpp"
#include "kernels.hpp"
#include "util.hpp"

#include <array>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <mutex>

namespace exh {

// ---------------------------------------------------------------------------
// deposit
// ---------------------------------------------------------------------------
// Periodic wrap into [0, L).  Values within one box length of the range
// take the reference's subtract/add loop (spectrum_h.c:18-28); farther
// values are reduced with floor first, so that the loop is bounded (the
// reference's loop does not terminate for huge or infinite values).  Where L
// is below the rounding of x / L * L (|x| beyond 1e7 boxes in float), the
// difference may lie anywhere and says nothing of the position: 0 is taken.
// Non-finite input is returned as it is, and the callers skip the tracer: a
// position that becomes so by the redshift-space shift is still seen by the
// test that follows its wrap.
template <typename T>
__device__ inline T wrap_while(T x, T L) {
  if (!isfinite(x)) return x;
  if (x >= (T)2 * L || x < -L) {
    const T r = x - floor(x / L) * L;
    x = r >= -L && r < (T)2 * L ? r : (T)0;
  }
  while (x >= L) x -= L;
  while (x < (T)0) x += L;
  return x;
}

// Hardware float/double atomic add (global_atomic_add_f32/f64).  HIP's
// atomicAdd(float*) defaults to a compare-and-swap loop, which serialises
// under the contention of neighbouring particles; the grids live in
// coarse-grained hipMalloc memory, where the hardware instruction is exact.
template <typename T>
__device__ inline void atomic_add_t(T* p, T v) {
  unsafeAtomicAdd(p, v);
}

template <typename T>
__device__ __forceinline__ bool finite3(const T* x) {
  return isfinite(x[0]) && isfinite(x[1]) && isfinite(x[2]);
}

template <typename T>
__device__ inline void dep_ngp(T* g, const T* x, int nd, T Ld, T m) {
  int xt[3];
  for (int a = 0; a < 3; a++) {
    xt[a] = (int)floor(x[a] / Ld);
    if (xt[a] == nd) xt[a] -= 1;
  }
  atomic_add_t(g + ((size_t)xt[0] * nd + xt[1]) * nd + xt[2], m);
}

template <typename T>
__device__ inline void dep_cic(T* g, const T* x, int nd, T Ld, T m) {
  int xt[3], o[3];
  T dx[3], t[3];
  for (int a = 0; a < 3; a++) {
    T q = x[a] / Ld;
    xt[a] = (int)floor(q);
    if (xt[a] == nd) xt[a] -= 1;
    dx[a] = (T)((double)q - ((double)xt[a] + 0.5));
    if (dx[a] >= (T)0) {
      o[a] = xt[a] + 1 == nd ? 0 : xt[a] + 1;
    } else {
      o[a] = xt[a] == 0 ? nd - 1 : xt[a] - 1;
      dx[a] = -dx[a];
    }
    t[a] = (T)(1.0 - (double)dx[a]);
  }
  const size_t n2 = (size_t)nd * nd;
  const size_t X0 = xt[0] * n2, X1 = o[0] * n2, Y0 = (size_t)xt[1] * nd, Y1 = (size_t)o[1] * nd;
  const size_t Z0 = xt[2], Z1 = o[2];
  atomic_add_t(g + X0 + Y0 + Z0, m * t[0] * t[1] * t[2]);
  atomic_add_t(g + X1 + Y0 + Z0, m * dx[0] * t[1] * t[2]);
  atomic_add_t(g + X0 + Y1 + Z0, m * t[0] * dx[1] * t[2]);
  atomic_add_t(g + X0 + Y0 + Z1, m * t[0] * t[1] * dx[2]);
  atomic_add_t(g + X1 + Y1 + Z0, m * dx[0] * dx[1] * t[2]);
  atomic_add_t(g + X1 + Y0 + Z1, m * dx[0] * t[1] * dx[2]);
  atomic_add_t(g + X0 + Y1 + Z1, m * t[0] * dx[1] * dx[2]);
  atomic_add_t(g + X1 + Y1 + Z1, m * dx[0] * dx[1] * dx[2]);
}

template <typename T>
__device__ inline void dep_tsc(T* g, const T* x, int nd, T Ld, T m) {
  int c[3];
  T w[3][3];
  for (int a = 0; a < 3; a++) {
    double u = (double)x[a] / (double)Ld - 0.5;
    double cf = floor(u + 0.5);
    double d = u - cf;
    c[a] = (int)cf;
    w[a][0] = (T)(0.5 * (0.5 - d) * (0.5 - d));
    w[a][1] = (T)(0.75 - d * d);
    w[a][2] = (T)(0.5 * (0.5 + d) * (0.5 + d));
  }
  for (int a = 0; a < 3; a++) {
    int ix = c[0] + a - 1;
    ix = ix < 0 ? ix + nd : (ix >= nd ? ix - nd : ix);
    for (int b = 0; b < 3; b++) {
      int iy = c[1] + b - 1;
      iy = iy < 0 ? iy + nd : (iy >= nd ? iy - nd : iy);
      T wab = m * w[0][a] * w[1][b];
      for (int e = 0; e < 3; e++) {
        int iz = c[2] + e - 1;
        iz = iz < 0 ? iz + nd : (iz >= nd ? iz - nd : iz);
        atomic_add_t(g + ((size_t)ix * nd + iy) * nd + iz, wab * w[2][e]);
      }
    }
  }
}

// Entries that were counted against those set aside: where there are more,
// nothing is listed and the atomics of k_deposit run in its place.
struct BinRoom {
  const int* total = nullptr;
  long long cap = 0;
  __device__ __forceinline__ bool over() const { return total && *total > cap; }
};

template <typename T, int WIN>
__global__ void k_deposit(const T* pos, const T* vel, const T* mass, const int* type,
                          long long np, int nd, T L, T Lb, int direction, T rsd, int nsub,
                          T* grid, unsigned long long* counts, BinRoom room) {
  if (room.total && !room.over()) return;  // the bins have done it
  const size_t ng = (size_t)nd * nd * nd;
  const T Ld = L / (T)nd;
  // particle counts per type (the normalisation's total mass): registers
  // for up to 4 types, an LDS histogram beyond; one atomic per block and
  // type at the end instead of one per particle on a single address
  __shared__ unsigned long long sh_cnt[64];
  unsigned long long reg_cnt[4] = {0, 0, 0, 0};
  const bool count = !mass && counts;
  const int ntype_reg = 4;
  if (threadIdx.x < 64) sh_cnt[threadIdx.x] = 0;
  __syncthreads();
  for (long long j = blockIdx.x * (long long)blockDim.x + threadIdx.x; j < np;
       j += (long long)gridDim.x * blockDim.x) {
    T x[3] = {pos[3 * j], pos[3 * j + 1], pos[3 * j + 2]};
    if (direction >= 0) x[direction] = wrap_while<T>(x[direction] + vel[3 * j + direction] * rsd, L);
    int t = type ? type[j] : 0;
    T m = mass ? mass[j] : (T)1;
    T p[3];
    for (int a = 0; a < 3; a++) p[a] = wrap_while<T>(x[a], L);
    if (!finite3(p)) continue;
    T* g = grid + (size_t)t * nsub * ng;
    if (WIN == 1) dep_ngp(g, p, nd, Ld, m);
    if (WIN == 2) dep_cic(g, p, nd, Ld, m);
    if (WIN == 5) dep_tsc(g, p, nd, Ld, m);
    if (nsub == 2) {
      T sh = (T)(-(double)Lb / 2.0);
      for (int a = 0; a < 3; a++) p[a] = wrap_while<T>(x[a] + sh, L);
      if (WIN == 1) dep_ngp(g + ng, p, nd, Ld, m);
      if (WIN == 2) dep_cic(g + ng, p, nd, Ld, m);
      if (WIN == 5) dep_tsc(g + ng, p, nd, Ld, m);
    }
    if (count) {
      if (t < ntype_reg) {
        for (int q = 0; q < ntype_reg; q++) reg_cnt[q] += (q == t);
      } else {
        atomicAdd(&sh_cnt[t], 1ull);
      }
    }
  }
  if (!count) return;
  for (int q = 0; q < ntype_reg; q++)
    if (reg_cnt[q]) atomicAdd(&sh_cnt[q], reg_cnt[q]);
  __syncthreads();
  if (threadIdx.x < 64 && sh_cnt[threadIdx.x]) atomicAdd(&counts[threadIdx.x], sh_cnt[threadIdx.x]);
}

// Spherical (window 3) and exponential (window 4) assignment
// (gridmodule.c:57-119): every cell of the cube of half-side
// times = floor(1/2 + R_eff / Ld) around the particle's cell whose centre lies
// within R_eff gets m (sphere, R_eff = R) or m exp(-r^2 / 2R^2) (R_eff =
// R R_times).  As in the reference, each offset is evaluated in double and
// stored in T, the periodic image is L - dx, and r^2 is summed in T.
// Returns the deposited weight.
__device__ inline int wrap_any(int x, int n) {
  int r = x % n;
  return r < 0 ? r + n : r;
}

template <typename T, bool EXPW>
__device__ inline double dep_sphere(T* g, const T* x, int nd, T L, T Ld, T R, T Rt, T m) {
  int xt[3];
  for (int a = 0; a < 3; a++) {
    xt[a] = (int)floor(x[a] / Ld);
    if (xt[a] == nd) xt[a] -= 1;
  }
  const int times = EXPW ? (int)floor(0.5 + (double)(R * Rt / Ld)) : (int)floor(0.5 + (double)(R / Ld));
  const T R2 = R * R, Re2 = R * R * Rt * Rt;
  const double halfL = (double)L / 2.0;
  auto offset = [&](int a, int c) {
    T d = (T)((double)x[a] - ((double)c + 0.5) * (double)Ld);
    if ((double)d > halfL) d = L - d;
    if ((double)d < -halfL) d = L + d;
    return d;
  };
  double M = 0.0;
  for (int i = -times; i <= times; i++) {
    const int ci = wrap_any(xt[0] + i, nd);
    const T d0 = offset(0, ci);
    for (int j = -times; j <= times; j++) {
      const int cj = wrap_any(xt[1] + j, nd);
      const T d1 = offset(1, cj);
      T* row = g + ((size_t)ci * nd + cj) * nd;
      for (int k = -times; k <= times; k++) {
        const int ck = wrap_any(xt[2] + k, nd);
        const T d2 = offset(2, ck);
        const T r2 = d0 * d0 + d1 * d1 + d2 * d2;
        if (!EXPW) {
          if (r2 <= R2) {
            atomic_add_t(row + ck, m);
            M += (double)m;
          }
        } else if (r2 <= Re2) {
          const T w = (T)exp(-0.5 * (double)r2 / (double)R / (double)R);
          atomic_add_t(row + ck, m * w);
          M += (double)m * (double)w;
        }
      }
    }
  }
  return M;
}

// One thread per particle; wsum[t * nsub + s] receives the deposited weight
// of each grid (the normalisation's total, in place of the particle count).
template <typename T, bool EXPW>
__global__ void k_deposit_sphere(const T* pos, const T* vel, const T* mass, const int* type,
                                 long long np, int nd, T L, T Lb, T R, T Rt, int direction, T rsd,
                                 int nsub, int ngrids, T* grid, double* wsum) {
  __shared__ double sh[128];
  const size_t ng = (size_t)nd * nd * nd;
  const T Ld = L / (T)nd;
  if (threadIdx.x < 128) sh[threadIdx.x] = 0.0;
  __syncthreads();
  for (long long j = blockIdx.x * (long long)blockDim.x + threadIdx.x; j < np;
       j += (long long)gridDim.x * blockDim.x) {
    T x[3] = {pos[3 * j], pos[3 * j + 1], pos[3 * j + 2]};
    if (direction >= 0) x[direction] = wrap_while<T>(x[direction] + vel[3 * j + direction] * rsd, L);
    const int t = type ? type[j] : 0;
    const T m = mass ? mass[j] : (T)1;
    T p[3];
    for (int a = 0; a < 3; a++) p[a] = wrap_while<T>(x[a], L);
    if (!finite3(p)) continue;
    T* g = grid + (size_t)t * nsub * ng;
    atomicAdd(&sh[t * nsub], dep_sphere<T, EXPW>(g, p, nd, L, Ld, R, Rt, m));
    if (nsub == 2) {
      const T sft = (T)(-(double)Lb / 2.0);
      for (int a = 0; a < 3; a++) p[a] = wrap_while<T>(x[a] + sft, L);
      atomicAdd(&sh[t * nsub + 1], dep_sphere<T, EXPW>(g + ng, p, nd, L, Ld, R, Rt, m));
    }
  }
  __syncthreads();
  if (threadIdx.x < ngrids && sh[threadIdx.x] != 0.0) atomicAdd(&wsum[threadIdx.x], sh[threadIdx.x]);
}

// ---------------------------------------------------------------------------
// LDS-privatised deposit for particles stored in Lagrangian lattice order
// (particle (i, j, k) of an nL^3 lattice at index (i nL + j) nL + k, as the
// LPT positions are).  One workgroup takes a TL^3 tile of the lattice: its
// particles, displaced by a smooth field, land in a compact Eulerian box.
// The block finds that box (cells relative to the tile centre, unwrapped
// across the periodic boundary), accumulates the window weights there with
// LDS atomics, and adds each touched cell to the grid with one coalesced
// global atomic (about 3 per particle for CIC at nd = nL instead of 8
// conflicting ones).  Tiles whose box exceeds the LDS deposit directly.
// The boxes accumulate in double for either grid precision: LDS float
// atomic adds (ds_add_f32) run at a small fraction of the rate of
// ds_add_f64 on gfx950, and the double sums round once when flushed.
// Weights are computed exactly as in dep_ngp/dep_cic/dep_tsc.
// ---------------------------------------------------------------------------
__device__ inline int rel_cell(int c, int qc, int nd) {
  int d = c - qc;
  if (d >= nd / 2) d -= nd;
  if (d < -nd / 2) d += nd;
  return d;
}

// Cells handled here lie within (-nd/2, 3nd/2) (a stencil neighbour, or a
// box cell a relative offset of less than nd/2 from a tile centre), so one
// conditional step wraps them exactly.
__device__ inline int wrap_cell(int c, int nd) { return c < 0 ? c + nd : (c >= nd ? c - nd : c); }

// Scaled coordinate of a wrapped position, the one division of a window
// evaluation: x / Ld for NGP and CIC, x / Ld - 0.5 in double for TSC.
template <typename T, int WIN>
__device__ inline auto scale_q(T x, T Ld) {
  if constexpr (WIN == 5)
    return (double)x / (double)Ld - 0.5;
  else
    return x / Ld;
}

// Cells and weights along one axis from the scaled coordinate, with the
// expressions of dep_ngp/dep_cic/dep_tsc.
template <typename T, int WIN, typename Q>
__device__ inline int stencil_q(Q q, int nd, int* cell, T* w) {
  if constexpr (WIN == 1) {
    int xt = (int)floor(q);
    if (xt == nd) xt -= 1;
    cell[0] = xt;
    w[0] = (T)1;
    return 1;
  } else if constexpr (WIN == 2) {
    int xt = (int)floor(q);
    if (xt == nd) xt -= 1;
    // dx = q - (xt + 1/2) and 1 - dx in T: both differences are exact in
    // double and round once, so T's correctly rounded subtraction gives the
    // reference's double-then-round values bit for bit
    T dx = q - ((T)xt + (T)0.5);
    int o;
    if (dx >= (T)0) {
      o = xt + 1 == nd ? 0 : xt + 1;
    } else {
      o = xt == 0 ? nd - 1 : xt - 1;
      dx = -dx;
    }
    cell[0] = xt;
    w[0] = (T)1 - dx;
    cell[1] = o;
    w[1] = dx;
    return 2;
  } else {
    const double u = q;
    const double cf = floor(u + 0.5);
    const double d = u - cf;
    const int c = (int)cf;
    cell[0] = wrap_cell(c - 1, nd);
    cell[1] = wrap_cell(c, nd);
    cell[2] = wrap_cell(c + 1, nd);
    w[0] = (T)(0.5 * (0.5 - d) * (0.5 - d));
    w[1] = (T)(0.75 - d * d);
    w[2] = (T)(0.5 * (0.5 + d) * (0.5 + d));
    return 3;
  }
}

// Cells and weights of one particle along one axis for window WIN.
template <typename T, int WIN>
__device__ inline int axis_stencil(T x, T Ld, int nd, int* cell, T* w) {
  return stencil_q<T, WIN>(scale_q<T, WIN>(x, Ld), nd, cell, w);
}

template <int N>
__device__ inline void block_minmax(int* v_min, int* v_max, int* sh) {
  // sh: 2 * N * (blockDim/64) ints; reduces N axes at once
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  for (int a = 0; a < N; a++) {
    int mn = v_min[a], mx = v_max[a];
    for (int o = 32; o > 0; o >>= 1) {
      mn = min(mn, __shfl_xor(mn, o, 64));
      mx = max(mx, __shfl_xor(mx, o, 64));
    }
    if (lane == 0) {
      sh[(2 * a) * nw + wave] = mn;
      sh[(2 * a + 1) * nw + wave] = mx;
    }
  }
  __syncthreads();
  for (int a = 0; a < N; a++) {
    int mn = sh[(2 * a) * nw], mx = sh[(2 * a + 1) * nw];
    for (int w = 1; w < nw; w++) {
      mn = min(mn, sh[(2 * a) * nw + w]);
      mx = max(mx, sh[(2 * a + 1) * nw + w]);
    }
    v_min[a] = mn;
    v_max[a] = mx;
  }
  __syncthreads();
}

static constexpr int TILE_L = 16;        // lattice tile side
static constexpr int TILE_THREADS = 1024;
static constexpr int TILE_PPT = TILE_L * TILE_L * TILE_L / TILE_THREADS;  // particles per thread

template <typename T, int WIN>
__global__ __launch_bounds__(TILE_THREADS) void k_deposit_tiles(
    const T* pos, const T* vel, const T* mass, int nL, int nd, int W, T L, T Lb, int direction,
    T rsd, int nsub, int cap, T* grid, unsigned long long* counts) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  double* box = (double*)lds_raw;
  __shared__ int red[2 * 3 * (TILE_THREADS / 64)];
  __shared__ unsigned long long nvalid;
  constexpr int NW = WIN == 1 ? 1 : (WIN == 2 ? 2 : 3);
  const size_t ng = (size_t)nd * nd * nd;
  const T Ld = L / (T)nd;
  const int nt = nL / TILE_L;
  const int tz = blockIdx.x % nt, ty = (blockIdx.x / nt) % nt, tx = blockIdx.x / (nt * nt);
  // tile centre in grid cells: the middle of the grid tile of the same index
  const int qc[3] = {tx * W + W / 2, ty * W + W / 2, tz * W + W / 2};
  if (threadIdx.x == 0) nvalid = 0;
  // particles of this thread: lanes along k (coalesced rows)
  T xs[TILE_PPT][3];
  T ms[TILE_PPT];
  bool ok[TILE_PPT];
  unsigned long long myvalid = 0;
  for (int p = 0; p < TILE_PPT; p++) {
    int lin = threadIdx.x + p * TILE_THREADS;
    int c = lin % TILE_L, b = (lin / TILE_L) % TILE_L, a = lin / (TILE_L * TILE_L);
    size_t j = ((size_t)(tx * TILE_L + a) * nL + (ty * TILE_L + b)) * nL + (tz * TILE_L + c);
    T x[3] = {pos[3 * j], pos[3 * j + 1], pos[3 * j + 2]};
    if (direction >= 0) x[direction] = wrap_while<T>(x[direction] + vel[3 * j + direction] * rsd, L);
    ok[p] = finite3(x);
    for (int q = 0; q < 3; q++) xs[p][q] = x[q];
    ms[p] = mass ? mass[j] : (T)1;
    myvalid += ok[p];
  }
  for (int s = 0; s < nsub; s++) {
    T* g = grid + (size_t)s * ng;
    const T sh = s == 0 ? (T)0 : (T)(-(double)Lb / 2.0);
    // box extent of this sub-grid's stencils
    int vmin[3] = {1 << 30, 1 << 30, 1 << 30}, vmax[3] = {-(1 << 30), -(1 << 30), -(1 << 30)};
    for (int p = 0; p < TILE_PPT; p++) {
      if (!ok[p]) continue;
      for (int q = 0; q < 3; q++) {
        T pa = wrap_while<T>(xs[p][q] + sh, L);
        int cell[3];
        T w[3];
        int n = axis_stencil<T, WIN>(pa, Ld, nd, cell, w);
        for (int u = 0; u < n; u++) {
          int r = rel_cell(cell[u], qc[q], nd);
          vmin[q] = min(vmin[q], r);
          vmax[q] = max(vmax[q], r);
        }
      }
    }
    block_minmax<3>(vmin, vmax, red);
    if (vmax[0] < vmin[0]) continue;  // no valid particle
    const int e0 = vmax[0] - vmin[0] + 1, e1 = vmax[1] - vmin[1] + 1, e2 = vmax[2] - vmin[2] + 1;
    const bool fits = (long long)e0 * e1 * e2 <= cap;
    if (fits) {
      const int vol = e0 * e1 * e2;
      for (int v = threadIdx.x; v < vol; v += TILE_THREADS) box[v] = 0.0;
      __syncthreads();
    }
    for (int p = 0; p < TILE_PPT; p++) {
      if (!ok[p]) continue;
      int cell[3][3];
      T w[3][3];
      for (int q = 0; q < 3; q++) {
        T pa = wrap_while<T>(xs[p][q] + sh, L);
        axis_stencil<T, WIN>(pa, Ld, nd, cell[q], w[q]);
      }
      for (int u = 0; u < NW; u++) {
        for (int b = 0; b < NW; b++) {
          T wab = ms[p] * w[0][u] * w[1][b];
          for (int c = 0; c < NW; c++) {
            T val = wab * w[2][c];
            const int lx = rel_cell(cell[0][u], qc[0], nd) - vmin[0];
            const int ly = rel_cell(cell[1][b], qc[1], nd) - vmin[1];
            const int lz = rel_cell(cell[2][c], qc[2], nd) - vmin[2];
            // the box bounds were taken over these same stencils; the
            // range test only guards the LDS index
            if (fits && (unsigned)lx < (unsigned)e0 && (unsigned)ly < (unsigned)e1 &&
                (unsigned)lz < (unsigned)e2) {
              atomicAdd(&box[(lx * e1 + ly) * e2 + lz], (double)val);
            } else {
              atomic_add_t(g + ((size_t)cell[0][u] * nd + cell[1][b]) * nd + cell[2][c], val);
            }
          }
        }
      }
    }
    if (fits) {
      __syncthreads();
      const int vol = e0 * e1 * e2;
      for (int v = threadIdx.x; v < vol; v += TILE_THREADS) {
        const double val = box[v];
        if (val == 0.0) continue;
        const int lz = v % e2, ly = (v / e2) % e1, lx = v / (e1 * e2);
        const int cx = wrap_cell(qc[0] + vmin[0] + lx, nd), cy = wrap_cell(qc[1] + vmin[1] + ly, nd),
                  cz = wrap_cell(qc[2] + vmin[2] + lz, nd);
        atomic_add_t(g + ((size_t)cx * nd + cy) * nd + cz, (T)val);
      }
      __syncthreads();
    }
  }
  if (!mass && counts) {
    atomicAdd(&nvalid, myvalid);
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(&counts[0], nvalid);
  }
}

// Window deposit: the tile's particles go into a fixed LDS window of
// E = W + 2 h cells per axis (W = grid cells per tile side, margin h), placed at
// the tile's mean displacement.  The mean is taken over one sampled
// particle per wave, so no pass over all particles precedes the deposit.  The
// rare stencil that leaves the window goes straight to the grid.  The
// window is flushed row by row, lanes along z, one global atomic per
// touched cell.
//
// A tile is PX x PY x PZ particles of the lattice and the window holds
// ACC sums (unsigned, float or double).
static constexpr int WIN_THREADS = 1024;
static constexpr int WIN_HALO = 4;  // default margin h

// Window sums: float or double (LDS float/double atomic adds), or unsigned
// 32-bit fixed point with 22 fraction bits (ds_add_u32; integer sums are
// exact, so the window does not depend on the order of the adds).  Fixed
// point serves unweighted deposits only, whose weights lie in [0, 1]: a
// cell holds 1023 particles' weight before the sum would wrap.  The adds
// return nothing; what a thread added is summed beside them, and the window's
// own total is compared with it.  Where they differ a cell wrapped, and the
// window is filled again with adds that return the old value: one that wraps
// carries 1024, exactly, to the grid's cell.
template <typename ACC>
struct WinAcc {
  static constexpr float SCALE = 1.f;
  template <typename T>
  __device__ static ACC to(T a, T w) {
    return (ACC)(a * w);
  }
  template <typename T>
  __device__ static T from(ACC a) {
    return (T)a;
  }
};
template <>
struct WinAcc<unsigned> {
  static constexpr float SCALE = 4194304.f;  // of the weights passed to `to`
  // a w, to the nearest
  template <typename T>
  __device__ static unsigned to(T a, T w) {
    return (unsigned)fmaf((float)a, (float)w, 0.5f);
  }
  template <typename T>
  __device__ static T from(unsigned a) {
    return (T)a * (T)(1.0 / 4194304.0);
  }
};

// First cell (possibly -1) and weights of the window along one axis: the
// values of stencil_q, in cell order.  CIC and TSC scale by the reciprocal of
// the cell size (their weights are continuous in the position, so the
// rounding of x / Ld against x * (1 / Ld) moves them by an ulp), TSC of a float
// grid in double, far below a float weight's rounding; NGP and TSC of a double
// grid divide as the reference does.
template <typename T, int WIN>
__device__ __forceinline__ int axis_window(T x, T Ld, T inv, double invd, int nd, T* w) {
  if constexpr (WIN == 1) {
    const int xt = (int)floor(x / Ld);
    w[0] = (T)1;
    return xt == nd ? xt - 1 : xt;
  } else if constexpr (WIN == 2) {
    const T q = x * inv;
    int xt = (int)floor(q);
    if (xt == nd) xt -= 1;
    const T dx = q - ((T)xt + (T)0.5);
    const T far = dx >= (T)0 ? dx : -dx, near = (T)1 - far;
    w[0] = dx >= (T)0 ? near : far;
    w[1] = dx >= (T)0 ? far : near;
    return dx >= (T)0 ? xt : xt - 1;
  } else {
    double u;
    if constexpr (sizeof(T) == 8)
      u = x / Ld - 0.5;
    else
      u = (double)x * invd - 0.5;
    const double cf = floor(u + 0.5);
    const double d = u - cf;
    w[0] = (T)(0.5 * (0.5 - d) * (0.5 - d));
    w[1] = (T)(0.75 - d * d);
    w[2] = (T)(0.5 * (0.5 + d) * (0.5 + d));
    return (int)cf - 1;
  }
}

// Bound by vector instructions (204 a particle and sub-grid for TSC) and LDS
// adds (6 cycles each with conflicts), with the flush's atomics close behind.
// One cell and one range test per axis, the fixed-point scale folded into the
// weights, adds without return values, the double division of a float grid's
// TSC as a product, and 64 registers in place of more than 64 (two workgroups
// per CU instead of one): 775 -> 637 us for 256^3 particles, TSC, interlaced,
// FP32.
template <typename T, int WIN, typename ACC, int PX, int PY, int PZ, bool KEEP>
__device__ __forceinline__ void deposit_window_tile(
    int tile, const T* pos, const T* vel, const T* mass, int nL, int nd, int Wx, int Wy, int Wz,
    int wh, T L, T Lb, int direction, T rsd, int nsub, T* grid, unsigned long long* counts) {
  constexpr int NW = WIN == 1 ? 1 : (WIN == 2 ? 2 : 3);
  constexpr int NWAVE = WIN_THREADS / 64;
  constexpr int PPT = PX * PY * PZ / WIN_THREADS;
  static_assert(PPT * WIN_THREADS == PX * PY * PZ, "tile must be a multiple of the block");
  extern __shared__ __align__(16) unsigned char lds_raw[];
  ACC* box = (ACC*)lds_raw;
  __shared__ float samp[3][NWAVE];
  __shared__ int wo_s[3];
  __shared__ long long diff_s[NWAVE];
  __shared__ unsigned long long nvalid;
  const size_t ng = (size_t)nd * nd * nd;
  const T Ld = L / (T)nd;
  const int nty = nL / PY, ntz = nL / PZ;
  const int W[3] = {Wx, Wy, Wz};
  const int Ex = Wx + 2 * wh, Ey = Wy + 2 * wh, Ez = Wz + 2 * wh, sx = Ey * Ez;
  const int tz = tile % ntz, ty = (tile / ntz) % nty, tx = tile / (ntz * nty);
  // tile centre in grid cells: the middle of the grid tile of the same index
  const int qc[3] = {tx * Wx + Wx / 2, ty * Wy + Wy / 2, tz * Wz + Wz / 2};
  if (threadIdx.x == 0) nvalid = 0;
  // particle p of this thread, after the redshift-space shift: kept in
  // registers, or read again for every filling (48 KB a tile, from the L2)
  auto load = [&](int p, T* x, T& m) {
    const int lin = threadIdx.x + p * WIN_THREADS;
    const int c = lin % PZ, b = (lin / PZ) % PY, a = lin / (PZ * PY);
    const size_t j = ((size_t)(tx * PX + a) * nL + (ty * PY + b)) * nL + (tz * PZ + c);
#pragma unroll
    for (int q = 0; q < 3; q++) x[q] = pos[3 * j + q];
    if (direction >= 0) {
      const T v = vel[3 * j + direction] * rsd;
#pragma unroll
      for (int q = 0; q < 3; q++)
        if (q == direction) x[q] = wrap_while<T>(x[q] + v, L);
    }
    m = mass ? mass[j] : (T)1;
  };
  T xk[KEEP ? PPT : 1][3], mk[KEEP ? PPT : 1];
  if constexpr (KEEP) {
#pragma unroll
    for (int p = 0; p < PPT; p++) load(p, xk[p], mk[p]);
  }
  unsigned myvalid = 0;
  // displacement (in cells) of each wave's first particle: its cell relative
  // to the tile centre minus its lattice point's offset from the centre
  if ((threadIdx.x & 63) == 0) {
    const int lin = threadIdx.x;
    const int lat[3] = {lin / (PZ * PY), (lin / PZ) % PY, lin % PZ};
    T x[3] = {xk[0][0], xk[0][1], xk[0][2]}, m;
    if constexpr (!KEEP) load(0, x, m);
#pragma unroll
    for (int q = 0; q < 3; q++) {
      float r = 1e30f;
      if (finite3(x)) {
        int cc = (int)floor(wrap_while<T>(x[q], L) / Ld);
        cc = cc < nd ? cc : nd - 1;
        r = (float)rel_cell(cc, qc[q], nd) -
            ((lat[q] + 0.5f) * (float)nd / (float)nL - 0.5f * (float)W[q]);
      }
      samp[q][threadIdx.x >> 6] = r;
    }
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    float sum = 0.f;
    int n = 0;
    for (int w = 0; w < NWAVE; w++) {
      const float v = samp[threadIdx.x][w];
      if (v < 1e29f) {
        sum += v;
        n++;
      }
    }
    const float mean = n ? sum / (float)n : 0.f;
    wo_s[threadIdx.x] = (int)floorf(mean + 0.5f) - W[threadIdx.x] / 2 - wh;
  }
  __syncthreads();
  const int wo[3] = {wo_s[0], wo_s[1], wo_s[2]};
  const int vol = Ex * sx;
  const T shift = (T)(-(double)Lb / 2.0);
  const T invLd = (T)1 / Ld;
  const double invd = 1.0 / (double)Ld;
  // the window's first cell, in [0, nd)
  int org[3];
#pragma unroll
  for (int q = 0; q < 3; q++) {
    org[q] = (qc[q] + wo[q]) % nd;
    org[q] += org[q] < 0 ? nd : 0;
  }
  constexpr bool FIXED = std::is_same<ACC, unsigned>::value;
  for (int s = 0; s < nsub; s++) {
    T* g = grid + (size_t)s * ng;
    unsigned added = 0;  // fixed point: this thread's sum, < 5 * 2^22 * PPT
    // the tile's particles into the window; `again`: the second filling, which
    // carries and leaves out what lies outside
    auto fill = [&](auto again) {
      for (int v = threadIdx.x; v < vol; v += WIN_THREADS) box[v] = (ACC)0;
      __syncthreads();
      T x[3], m;
      if constexpr (!KEEP) load(0, x, m);
#pragma unroll(KEEP ? PPT : 1)
      for (int p = 0; p < PPT; p++) {
        if constexpr (KEEP) {
          x[0] = xk[p][0], x[1] = xk[p][1], x[2] = xk[p][2], m = mk[p];
        }
        const T px[3] = {x[0], x[1], x[2]}, pm = m;
        if constexpr (!KEEP) {
          if (p + 1 < PPT) load(p + 1, x, m);
        }
        if (!finite3(px)) continue;
        if constexpr (!decltype(again)::value) myvalid += s == 0;
        int b[3], l[3];
        T w[3][NW];
#pragma unroll
        for (int q = 0; q < 3; q++) {
          T pa = s == 0 ? px[q] : px[q] + shift;
          if (!(pa >= (T)0 && pa < L)) pa = wrap_while<T>(pa, L);
          b[q] = axis_window<T, WIN>(pa, Ld, invLd, invd, nd, w[q]);
          l[q] = b[q] - org[q];
          l[q] += l[q] < 0 ? nd : 0;
        }
        if (l[0] + NW <= Ex && l[1] + NW <= Ey && l[2] + NW <= Ez) {
          ACC* row = box + l[0] * sx + l[1] * Ez + l[2];
#pragma unroll
          for (int u = 0; u < NW; u++) {
#pragma unroll
            for (int v = 0; v < NW; v++) {
              const T wab = pm * w[0][u] * w[1][v] * (T)WinAcc<ACC>::SCALE;
              ACC* r = row + u * sx + v * Ez;
#pragma unroll
              for (int k = 0; k < NW; k++) {
                const ACC val = WinAcc<ACC>::to(wab, w[2][k]);
                if constexpr (decltype(again)::value) {
                  const ACC old = atomicAdd(&r[k], val);
                  if (old + val < old)
                    atomic_add_t(g + ((size_t)wrap_cell(b[0] + u, nd) * nd +
                                      wrap_cell(b[1] + v, nd)) * nd + wrap_cell(b[2] + k, nd),
                                 (T)1024);
                } else {
                  atomicAdd(&r[k], val);
                  if constexpr (FIXED) added += val;
                }
              }
            }
          }
        } else if constexpr (!decltype(again)::value) {
          for (int u = 0; u < NW; u++)
            for (int v = 0; v < NW; v++) {
              const T wab = pm * w[0][u] * w[1][v];
              for (int k = 0; k < NW; k++)
                atomic_add_t(g + ((size_t)wrap_cell(b[0] + u, nd) * nd +
                                  wrap_cell(b[1] + v, nd)) * nd + wrap_cell(b[2] + k, nd),
                             wab * w[2][k]);
            }
        }
      }
      __syncthreads();
    };
    fill(std::false_type{});
    if constexpr (FIXED) {
      // the window's total less what was added; a multiple of 2^32 wrapped
      long long diff = -(long long)added;
      for (int v = threadIdx.x; v < vol; v += WIN_THREADS) diff += box[v];
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) diff += __shfl_xor(diff, o, 64);
      if ((threadIdx.x & 63) == 0) diff_s[threadIdx.x >> 6] = diff;
      __syncthreads();
      long long all = 0;
#pragma unroll
      for (int w = 0; w < NWAVE; w++) all += diff_s[w];
      if (all != 0) fill(std::true_type{});
    }
    // flush: (y, z) rows over the threads, z fastest in 32-lane groups
    const int lz0 = threadIdx.x & 31;
    for (int ly = threadIdx.x >> 5; ly < Ey; ly += WIN_THREADS / 32) {
      const int cy = wrap_cell(org[1] + ly, nd);
      for (int lz = lz0; lz < Ez; lz += 32) {
        const int cz = wrap_cell(org[2] + lz, nd);
        const ACC* bp = box + ly * Ez + lz;
        int cx = org[0];
        for (int lx = 0; lx < Ex; lx++) {
          const ACC val = bp[lx * sx];
          if (val != (ACC)0)
            atomic_add_t(g + ((size_t)cx * nd + cy) * nd + cz, WinAcc<ACC>::template from<T>(val));
          cx = cx + 1 == nd ? 0 : cx + 1;
        }
      }
    }
    __syncthreads();
  }
  if (!mass && counts) {
    atomicAdd(&nvalid, (unsigned long long)myvalid);
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(&counts[0], nvalid);
  }
}

// One workgroup per tile, or (EXH_DEPOSIT_WG) fewer workgroups that walk the
// tiles, leaving CUs to the kernels of other streams.
template <typename T, int WIN, typename ACC, int PX, int PY, int PZ, bool KEEP, int WAVES>
__global__ __launch_bounds__(WIN_THREADS, WAVES) void k_deposit_window(
    const T* pos, const T* vel, const T* mass, int nL, int nd, int Wx, int Wy, int Wz, int wh,
    T L, T Lb, int direction, T rsd, int nsub, T* grid, unsigned long long* counts, int ntiles) {
  for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    deposit_window_tile<T, WIN, ACC, PX, PY, PZ, KEEP>(tile, pos, vel, mass, nL, nd, Wx, Wy, Wz,
                                                       wh, L, Lb, direction, rsd, nsub, grid,
                                                       counts);
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Binned deposit for particles in any order.  k_deposit issues one global
// atomic per particle, cell and sub-grid, and those run at 26 G requests a
// second whatever they touch (2 M particles, CIC, interlaced, 256^3 FP32:
// 1.54 ms; binned 0.20 ms, of which the tiles' LDS atomics are the most).  Here
// the grid is cut into tiles of at most 16 to 24 cells an edge; every particle is
// listed with each tile that its stencils reach (1.4 on average for
// interlaced CIC and 16^3 tiles), and one workgroup per tile sums its
// particles in LDS, in double, and writes its own cells: no global atomic,
// no zeroed grid and no normalisation pass.
//
//  k_bin_count    tile counts of a block's particles in LDS, then one add per
//                 tile (in runs) that also gives the block its first place
//  k_bin_scatter  places from LDS counters; writes (x, y, z, weight)
//  k_bin_deposit  sums and writes a tile, or a part of one that holds more
//                 than BIN_PART entries into a slot of its own
//  k_bin_merge    adds up the parts of such a tile and writes it
// ---------------------------------------------------------------------------
static constexpr int BIN_MAX = 36864;   // bins (tiles x types): counters in LDS
static constexpr int BIN_PART = 16384;  // entries of a part
static constexpr long long BIN_ATOMICS = 1 << 20;  // fewest atomics to bin for
static constexpr long long BIN_NP = 1 << 27;       // particles (entries fit an int)
static constexpr long long BIN_READ = 4 << 20;     // most particles with 8 entries each
static constexpr size_t BIN_BYTES = 8ull << 30;    // most bytes set aside for a count not read

struct BinGeom {
  int nd, nt, ntile;  // cells and tiles per axis, tiles
  int ntype, bins;
  FastDiv dnd;
};

// Tile of cell c along an axis: tile t holds cells floor(t nd / nt) up to
// floor((t + 1) nd / nt).
__device__ __forceinline__ int bin_tile(const BinGeom& g, int c) {
  return (int)fdiv((unsigned)((c + 1) * g.nt - 1), g.dnd);
}
__device__ __forceinline__ int bin_start(const BinGeom& g, int t) {
  return (int)((long long)t * g.nd / g.nt);
}

template <typename T>
struct BinParticles {
  const T *pos, *vel, *mass;
  const int* type;
  long long np;
  T L, Lb, rsd;
  int direction, nsub;
};

template <typename T>
struct alignas(sizeof(T) * 4) BinEntry {
  T x, y, z, m;
};

// Particle j after the redshift-space shift; false where k_deposit skips it.
template <typename T>
__device__ __forceinline__ bool bin_particle(const BinParticles<T>& a, const BinGeom& g,
                                             long long j, T* x, int& t) {
  x[0] = a.pos[3 * j];
  x[1] = a.pos[3 * j + 1];
  x[2] = a.pos[3 * j + 2];
  if (a.direction >= 0) {
    const T v = a.vel[3 * j + a.direction] * a.rsd;
#pragma unroll
    for (int q = 0; q < 3; q++)
      if (q == a.direction) x[q] = wrap_while<T>(x[q] + v, a.L);
  }
  t = a.type ? a.type[j] : 0;
  return finite3(x) && (unsigned)t < (unsigned)g.ntype;
}

// The one or two tiles per axis that the particle's stencils reach (at most
// four neighbouring cells; every tile has at least eight where there are two).
template <typename T, int WIN>
__device__ __forceinline__ void bin_tiles(const BinParticles<T>& a, const BinGeom& g, const T* x,
                                          int* ta, int* tb) {
  const T Ld = a.L / (T)g.nd;
  const T sh = (T)(-(double)a.Lb / 2.0);
#pragma unroll
  for (int q = 0; q < 3; q++) {
    int cell[3];
    T w[3];
    const int n = axis_stencil<T, WIN>(wrap_while<T>(x[q], a.L), Ld, g.nd, cell, w);
    ta[q] = bin_tile(g, cell[0]);
    tb[q] = ta[q];
#pragma unroll
    for (int u = 1; u < n; u++) {
      const int t = bin_tile(g, cell[u]);
      if (t != ta[q]) tb[q] = t;
    }
    if (a.nsub == 2) {
      axis_stencil<T, WIN>(wrap_while<T>(x[q] + sh, a.L), Ld, g.nd, cell, w);
#pragma unroll
      for (int u = 0; u < n; u++) {
        const int t = bin_tile(g, cell[u]);
        if (t != ta[q]) tb[q] = t;
      }
    }
  }
}

template <typename F>
__device__ __forceinline__ void bin_each(const BinGeom& g, int t, const int* ta, const int* tb,
                                         const F& f) {
  for (int i = 0; i <= (tb[0] != ta[0]); i++)
    for (int j = 0; j <= (tb[1] != ta[1]); j++)
      for (int k = 0; k <= (tb[2] != ta[2]); k++)
        f(t * g.ntile + ((i ? tb[0] : ta[0]) * g.nt + (j ? tb[1] : ta[1])) * g.nt +
          (k ? tb[2] : ta[2]));
}

// counts[bin] += the block's entries of the bin; place[block][bin] = what it
// held before.  nvalid[type] += the block's particles.
template <typename T, int WIN>
__global__ __launch_bounds__(1024) void k_bin_count(BinParticles<T> a, BinGeom g, long long chunk,
                                                    int* counts, int* place,
                                                    unsigned long long* nvalid) {
  extern __shared__ int bin_lds[];
  __shared__ unsigned sh_cnt[64];
  for (int b = threadIdx.x; b < g.bins; b += blockDim.x) bin_lds[b] = 0;
  if (threadIdx.x < 64) sh_cnt[threadIdx.x] = 0;
  __syncthreads();
  const long long j0 = blockIdx.x * chunk, j1 = min(j0 + chunk, a.np);
  unsigned mine = 0;
  for (long long j = j0 + threadIdx.x; j < j1; j += blockDim.x) {
    T x[3];
    int t, ta[3], tb[3];
    if (!bin_particle(a, g, j, x, t)) continue;
    bin_tiles<T, WIN>(a, g, x, ta, tb);
    bin_each(g, t, ta, tb, [&](int b) { atomicAdd(&bin_lds[b], 1); });
    if (g.ntype == 1)
      mine++;
    else
      atomicAdd(&sh_cnt[t], 1u);
  }
  if (mine) atomicAdd(&sh_cnt[0], mine);
  __syncthreads();
  int* pl = place + (size_t)blockIdx.x * g.bins;
  for (int b = threadIdx.x; b < g.bins; b += blockDim.x) {
    const int h = bin_lds[b];
    pl[b] = h ? atomicAdd(&counts[b], h) : 0;
  }
  if (threadIdx.x < 64 && sh_cnt[threadIdx.x])
    atomicAdd(&nvalid[threadIdx.x], (unsigned long long)sh_cnt[threadIdx.x]);
}

template <typename T, int WIN>
__global__ __launch_bounds__(1024) void k_bin_scatter(BinParticles<T> a, BinGeom g,
                                                      long long chunk, const int* off,
                                                      const int* place, BinRoom room,
                                                      BinEntry<T>* out) {
  extern __shared__ int bin_lds[];
  if (room.over()) return;
  const int* pl = place + (size_t)blockIdx.x * g.bins;
  for (int b = threadIdx.x; b < g.bins; b += blockDim.x) bin_lds[b] = off[b] + pl[b];
  __syncthreads();
  const long long j0 = blockIdx.x * chunk, j1 = min(j0 + chunk, a.np);
  for (long long j = j0 + threadIdx.x; j < j1; j += blockDim.x) {
    T x[3];
    int t, ta[3], tb[3];
    if (!bin_particle(a, g, j, x, t)) continue;
    bin_tiles<T, WIN>(a, g, x, ta, tb);
    const BinEntry<T> e{x[0], x[1], x[2], a.mass ? a.mass[j] : (T)1};
    bin_each(g, t, ta, tb, [&](int b) { out[atomicAdd(&bin_lds[b], 1)] = e; });
  }
}

// Slots of the parts: slot[b] = parts of the split bins before b.
__global__ __launch_bounds__(256) void k_bin_parts(const int* counts, int bins, int* parts) {
  const int b = blockIdx.x * 256 + threadIdx.x;
  if (b < bins) parts[b] = counts[b] > BIN_PART ? (counts[b] + BIN_PART - 1) / BIN_PART : 0;
}

struct BinTile {
  int s[3], n[3];  // first cell and cells per axis
  int t;           // type
};
__device__ __forceinline__ BinTile bin_of(const BinGeom& g, int b) {
  BinTile r;
  r.t = b / g.ntile;
  const int q = b - r.t * g.ntile;
  const int c[3] = {q / (g.nt * g.nt), q / g.nt % g.nt, q % g.nt};
#pragma unroll
  for (int a = 0; a < 3; a++) {
    r.s[a] = bin_start(g, c[a]);
    r.n[a] = bin_start(g, c[a] + 1) - r.s[a];
  }
  return r;
}

// The tile's cells of one sub-grid from their sums; normalised without
// weights (delta = rho / rho_bar - 1).
template <typename T, typename F>
__device__ __forceinline__ void bin_write(const BinGeom& g, const BinTile& r, T* grid, bool norm,
                                          double mean, const F& sum) {
  const int cells = r.n[0] * r.n[1] * r.n[2];
  for (int c = threadIdx.x; c < cells; c += blockDim.x) {
    const int k = c % r.n[2], q = c / r.n[2], j = q % r.n[1], i = q / r.n[1];
    const double v = sum(c);
    grid[((size_t)(r.s[0] + i) * g.nd + r.s[1] + j) * g.nd + r.s[2] + k] =
        norm ? (T)(v / mean - 1.0) : (T)v;
  }
}

template <typename T, int WIN>
__global__ __launch_bounds__(256) void k_bin_deposit(BinGeom g, const BinEntry<T>* ent,
                                                     const int* off, const int* slot, T L, T Lb,
                                                     int nsub, bool norm,
                                                     const unsigned long long* nvalid,
                                                     double* partial, int pitch, BinRoom room,
                                                     T* grid) {
  extern __shared__ double bin_sum[];
  if (room.over()) return;
  constexpr int NW = WIN == 1 ? 1 : (WIN == 2 ? 2 : 3);
  int b = blockIdx.x, e0, e1, sl = -1;
  if (b < g.bins) {
    e0 = off[b];
    e1 = off[b + 1];
    if (slot[b + 1] > slot[b]) return;  // in parts
  } else {
    sl = b - g.bins;
    if (sl >= slot[g.bins]) return;
    int lo = 0, hi = g.bins;  // slot[lo] <= sl < slot[hi]
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (slot[mid] <= sl)
        lo = mid;
      else
        hi = mid;
    }
    b = lo;
    e0 = off[b] + (sl - slot[b]) * BIN_PART;
    e1 = min(e0 + BIN_PART, off[b + 1]);
  }
  const BinTile r = bin_of(g, b);
  const int cells = r.n[0] * r.n[1] * r.n[2];
  const T Ld = L / (T)g.nd;
  const T sh = (T)(-(double)Lb / 2.0);
  const size_t ng = (size_t)g.nd * g.nd * g.nd;
  const double mean = norm ? (double)nvalid[r.t] / (double)ng : 1.0;
  for (int sub = 0; sub < nsub; sub++) {
    for (int c = threadIdx.x; c < cells; c += 256) bin_sum[c] = 0.0;
    __syncthreads();
    for (int e = e0 + (int)threadIdx.x; e < e1; e += 256) {
      const BinEntry<T> p = ent[e];
      const T x[3] = {p.x, p.y, p.z};
      int l[3][3];
      T w[3][3];
#pragma unroll
      for (int q = 0; q < 3; q++) {
        int cell[3];
        axis_stencil<T, WIN>(wrap_while<T>(sub ? x[q] + sh : x[q], L), Ld, g.nd, cell, w[q]);
#pragma unroll
        for (int u = 0; u < NW; u++) {
          const int d = cell[u] - r.s[q];
          l[q][u] = (unsigned)d < (unsigned)r.n[q] ? d : -1;
        }
      }
#pragma unroll
      for (int u = 0; u < NW; u++) {
        if (l[0][u] < 0) continue;
#pragma unroll
        for (int v = 0; v < NW; v++) {
          if (l[1][v] < 0) continue;
          const int row = (l[0][u] * r.n[1] + l[1][v]) * r.n[2];
          const T wab = p.m * w[0][u] * w[1][v];
#pragma unroll
          for (int k = 0; k < NW; k++)
            if (l[2][k] >= 0) atomicAdd(&bin_sum[row + l[2][k]], (double)(wab * w[2][k]));
        }
      }
    }
    __syncthreads();
    if (sl >= 0) {
      double* o = partial + ((size_t)sl * nsub + sub) * pitch;
      for (int c = threadIdx.x; c < cells; c += 256) o[c] = bin_sum[c];
    } else {
      bin_write<T>(g, r, grid + (size_t)(r.t * nsub + sub) * ng, norm, mean,
                   [&](int c) { return bin_sum[c]; });
    }
    __syncthreads();
  }
}

// Block s: the parts from slot s on where s is the first slot of a bin.
template <typename T>
__global__ __launch_bounds__(256) void k_bin_merge(BinGeom g, const int* slot, int nsub, bool norm,
                                                   const unsigned long long* nvalid,
                                                   const double* partial, int pitch, BinRoom room,
                                                   T* grid) {
  const int sl = blockIdx.x;
  if (room.over()) return;
  if (sl >= slot[g.bins]) return;
  int lo = 0, hi = g.bins;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (slot[mid] <= sl)
      lo = mid;
    else
      hi = mid;
  }
  if (slot[lo] != sl) return;
  const int np = slot[lo + 1] - sl;
  const BinTile r = bin_of(g, lo);
  const size_t ng = (size_t)g.nd * g.nd * g.nd;
  const double mean = norm ? (double)nvalid[r.t] / (double)ng : 1.0;
  for (int sub = 0; sub < nsub; sub++)
    bin_write<T>(g, r, grid + (size_t)(r.t * nsub + sub) * ng, norm, mean, [&](int c) {
      double v = 0.0;
      for (int q = 0; q < np; q++) v += partial[((size_t)(sl + q) * nsub + sub) * pitch + c];
      return v;
    });
}

template <typename T>
__global__ void k_zero(T* g, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    g[i] = (T)0;
}

// The same for a 16-byte aligned array, with 16-byte stores (the values
// past the last whole 16 bytes one by one).
template <typename T>
__global__ void k_zero16(T* g, size_t n) {
  const size_t nv = n * sizeof(T) / 16;
  const size_t t0 = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  const size_t st = (size_t)gridDim.x * blockDim.x;
  uint4* v = reinterpret_cast<uint4*>(g);
  for (size_t i = t0; i < nv; i += st) v[i] = make_uint4(0u, 0u, 0u, 0u);
  for (size_t i = nv * 16 / sizeof(T) + t0; i < n; i += st) g[i] = (T)0;
}

// The grids of a deposit whose entries found no room, zeroed for the atomics.
template <typename T>
__global__ void k_zero_over(T* g, size_t n, BinRoom room) {
  if (!room.over()) return;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    g[i] = (T)0;
}

// grid (blockIdx.y) of ngrids: delta = rho / (M / ng) - 1
template <typename T>
__global__ void k_normalise(T* grid, size_t ng, int nsub, const unsigned long long* counts,
                            BinRoom room) {
  if (room.total && !room.over()) return;
  const double M = (double)counts[blockIdx.y / nsub];
  const double mean = M / (double)ng;
  T* g = grid + (size_t)blockIdx.y * ng;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < ng;
       i += (size_t)gridDim.x * blockDim.x)
    g[i] = (T)((double)g[i] / mean - 1.0);
}

// The same with 16-byte loads and stores, for 16-byte aligned grids whose
// size is a multiple of 16 bytes; each value's expression is unchanged.
template <typename T>
__global__ void k_normalise16(T* grid, size_t ng, int nsub, const unsigned long long* counts) {
  constexpr int W = 16 / (int)sizeof(T);
  const double M = (double)counts[blockIdx.y / nsub];
  const double mean = M / (double)ng;
  uint4* g = reinterpret_cast<uint4*>(grid + (size_t)blockIdx.y * ng);
  const size_t nv = ng / W;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < nv;
       i += (size_t)gridDim.x * blockDim.x) {
    uint4 u = g[i];
    T t[W];
    __builtin_memcpy(t, &u, 16);
#pragma unroll
    for (int e = 0; e < W; e++) t[e] = (T)((double)t[e] / mean - 1.0);
    __builtin_memcpy(&u, t, 16);
    g[i] = u;
  }
}

// grid (blockIdx.y): delta = rho / (W / ng) - 1, W the deposited weight
template <typename T>
__global__ void k_normalise_w(T* grid, size_t ng, const double* wsum) {
  const double mean = wsum[blockIdx.y] / (double)ng;
  T* g = grid + (size_t)blockIdx.y * ng;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < ng;
       i += (size_t)gridDim.x * blockDim.x)
    g[i] = (T)((double)g[i] / mean - 1.0);
}

// Side of the particle lattice when np is a perfect cube, else 0.
static int lattice_side(long long np) {
  if (np <= 0) return 0;
  long long n = (long long)std::llround(std::cbrt((double)np));
  for (long long m = n > 1 ? n - 1 : 1; m <= n + 1; m++)
    if (m * m * m == np) return (int)m;
  return 0;
}

// LDS bytes of the tiled deposit's Eulerian box: EXH_DEPOSIT_LDS_KB (0
// disables the tiled path), default 144 KB of the 160 KB per workgroup.
static int deposit_lds_bytes() {
  static int v = [] {
    const char* e = std::getenv("EXH_DEPOSIT_LDS_KB");
    int kb = e ? std::atoi(e) : 144;
    if (kb < 0) kb = 0;
    if (kb > 156) kb = 156;
    return kb * 1024;
  }();
  return v;
}

// The window deposit for lattice-ordered particles (EXH_DEPOSIT_WINDOW=0
// keeps the extent-sized boxes of k_deposit_tiles).
static bool deposit_window_enabled() {
  static const bool on = [] {
    const char* e = std::getenv("EXH_DEPOSIT_WINDOW");
    return !(e && std::atoi(e) == 0);
  }();
  return on;
}

// Workgroups of the window deposit (EXH_DEPOSIT_WG; 0 = one per tile).
static int deposit_workgroups() {
  static const int v = [] {
    const char* e = std::getenv("EXH_DEPOSIT_WG");
    const int n = e ? std::atoi(e) : 0;
    return n < 0 ? 0 : n;
  }();
  return v;
}

// Window margin h in cells (EXH_DEPOSIT_MARGIN, 1..8, default WIN_HALO).
static int deposit_window_margin() {
  static const int v = [] {
    const char* e = std::getenv("EXH_DEPOSIT_MARGIN");
    const int h = e ? std::atoi(e) : WIN_HALO;
    return h < 1 ? 1 : (h > 8 ? 8 : h);
  }();
  return v;
}

// Scratch of the allocation-free deposit (exh_grid_compute_noalloc): the
// per-type particle counts (64 words) or the per-grid deposited weights
// (128 doubles) that the normalisation reads.  Each device holds its own
// copy; host code takes its address once per device from
// hipGetSymbolAddress and never uses the array's name.  Calls that
// overlap on one device share it and race.
static __device__ __align__(256) unsigned long long scratch[NOALLOC_GRID_WORDS];

static std::mutex g_scratch_mu;
static void* g_scratch_ptr[NOALLOC_MAX_DEVICES] = {};

void* noalloc_grid_scratch(int device) {
  EXH_REQUIRE(device >= 0 && device < NOALLOC_MAX_DEVICES, EXH_ERR_ARG,
              "device %d out of range for the allocation-free entry point", device);
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[device]) {
    int cur = -1;
    EXH_CHECK_HIP(hipGetDevice(&cur));
    EXH_REQUIRE(cur == device, EXH_ERR_INTERNAL, "device %d is not current", device);
    void* p = nullptr;
    EXH_CHECK_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    EXH_REQUIRE(p != nullptr, EXH_ERR_HIP, "no address for the deposit scratch on device %d",
                device);
    g_scratch_ptr[device] = p;
  }
  return g_scratch_ptr[device];
}

// Tile shape of the window deposit (EXH_DEPOSIT_TILE: 16 = 16^3 particles,
// the default; 3216 = 32 x 16 x 16; 32 = 32 x 32 x 16) and its
// accumulator (EXH_DEPOSIT_ACC: 1 fixed point, the default for float grids
// without masses; 8 double; 4 float).  Two 16^3 workgroups of 55 KB and 64
// registers share a CU.  The whole call (zero, deposit, normalise) at nd = nL
// = 512, FP32, CIC, interlaced, LPT positions, takes 3.28 ms with 16^3 tiles,
// 3.28 with 32 x 16 x 16 and 3.02 with 32 x 32 x 16, whose windows issue the
// fewest atomics; small boxes leave CUs without one of the larger tiles (64^3:
// 52, 63 and 84 us), and beside the halo finder's sort larger workgroups hold
// CUs long enough to slow the sort.  16^3 tiles summed in double take 4.33 ms,
// in float 12.1 (ds_add_f32 runs far slower than ds_add_u32 or ds_add_f64).
struct WinShape {
  int px, py, pz;
};
static WinShape tile_shape(int t) {
  if (t == 32) return WinShape{32, 32, 16};
  if (t == 3216) return WinShape{32, 16, 16};
  return WinShape{16, 16, 16};
}
static WinShape deposit_window_shape() {
  static const WinShape v = [] {
    const char* e = std::getenv("EXH_DEPOSIT_TILE");
    return tile_shape(e ? std::atoi(e) : 16);
  }();
  return v;
}
static int deposit_window_acc() {
  static const int v = [] {
    const char* e = std::getenv("EXH_DEPOSIT_ACC");
    const int a = e ? std::atoi(e) : 1;
    return (a == 4 || a == 1) ? a : 8;
  }();
  return v;
}
// LDS of the window (the kernel's static shared memory takes < 1 KB of the
// 160 KB)
static constexpr int WIN_LDS_MAX = 159 * 1024;

template <typename T>
struct DepositWinArgs {
  const T *pos, *vel, *mass;
  int nL, nd, Wx, Wy, Wz, wh;
  T L, Lb;
  int direction;
  T rsd;
  int nsub;
  T* grid;
  unsigned long long* counts;
  int ntiles;
};

// Positions stay in registers where every CU has one tile at most, and with
// two sub-grids, which read them twice, also where one workgroup fills a CU
// anyway and there are few tiles a CU; else they are read again, in 64
// registers (WAVES = 8) where the window lets two workgroups share a CU.
// Whole call, read again against kept, us: FP32, CIC, two sub-grids, 96^3
// (216 tiles) 69.6 and 65.0; TSC, 256^3 638 and 664.  FP64, CIC, two
// sub-grids, 160^3 (1000 tiles) 206 and 193, 256^3 (4096) 671 and 681; one
// sub-grid, with weights, 256^3 326 and 372.  32 x 32 x 16 particles, FP32,
// CIC, two sub-grids, 192^3 (432 tiles) 246 and 239; one, 320^3 472 and 517.
template <typename T, int WN, typename ACC, int PX, int PY, int PZ>
static void launch_window(exh_ctx* c, unsigned nwg, int lds, const DepositWinArgs<T>& a) {
  constexpr bool MAY = sizeof(ACC) == 4 && PX * PY * PZ == 4 * WIN_THREADS;
  const bool two = MAY && lds <= WIN_LDS_MAX / 2;
  auto go = [&](auto k) {
    EXH_CHECK_HIP(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                      lds));
    hipLaunchKernelGGL(k, dim3(nwg), dim3(WIN_THREADS), lds, c->stream, a.pos, a.vel, a.mass, a.nL,
                       a.nd, a.Wx, a.Wy, a.Wz, a.wh, a.L, a.Lb, a.direction, a.rsd, a.nsub, a.grid,
                       a.counts, a.ntiles);
  };
  const bool keep = nwg <= 256 || (!two && a.nsub == 2 && nwg <= 2048);
  if (keep) return go(k_deposit_window<T, WN, ACC, PX, PY, PZ, true, 4>);
  if constexpr (MAY) {
    if (two) return go(k_deposit_window<T, WN, ACC, PX, PY, PZ, false, 8>);
  }
  go(k_deposit_window<T, WN, ACC, PX, PY, PZ, false, 4>);
}

template <typename T, int WN>
static void launch_window_shape(exh_ctx* c, int acc, const WinShape& ws, unsigned nwg, int lds,
                                const DepositWinArgs<T>& a) {
  if constexpr (sizeof(T) == 8) {
    if (ws.px == 32 && ws.py == 32) launch_window<T, WN, double, 32, 32, 16>(c, nwg, lds, a);
    else if (ws.px == 32) launch_window<T, WN, double, 32, 16, 16>(c, nwg, lds, a);
    else launch_window<T, WN, double, 16, 16, 16>(c, nwg, lds, a);
  } else if (ws.px == 32 && ws.py == 32) {
    if (acc == 1) launch_window<T, WN, unsigned, 32, 32, 16>(c, nwg, lds, a);
    else if (acc == 4) launch_window<T, WN, float, 32, 32, 16>(c, nwg, lds, a);
    else launch_window<T, WN, double, 32, 32, 16>(c, nwg, lds, a);
  } else if (ws.px == 32) {
    if (acc == 1) launch_window<T, WN, unsigned, 32, 16, 16>(c, nwg, lds, a);
    else if (acc == 4) launch_window<T, WN, float, 32, 16, 16>(c, nwg, lds, a);
    else launch_window<T, WN, double, 32, 16, 16>(c, nwg, lds, a);
  } else {
    if (acc == 1) launch_window<T, WN, unsigned, 16, 16, 16>(c, nwg, lds, a);
    else if (acc == 4) launch_window<T, WN, float, 16, 16, 16>(c, nwg, lds, a);
    else launch_window<T, WN, double, 16, 16, 16>(c, nwg, lds, a);
  }
}

template <typename T>
static void launch_window_any(exh_ctx* c, int window, int acc, const WinShape& ws, unsigned nwg,
                              int lds, const DepositWinArgs<T>& a) {
  if (window == 1) launch_window_shape<T, 1>(c, acc, ws, nwg, lds, a);
  if (window == 2) launch_window_shape<T, 2>(c, acc, ws, nwg, lds, a);
  if (window == 5) launch_window_shape<T, 5>(c, acc, ws, nwg, lds, a);
}

// Tiles of the binned deposit: the smallest edge (16, 20 or 24 cells) whose
// bins fit the LDS counters; 0 bins where none does.
static BinGeom bin_geom(const exh_ctx* c, int nd, int ntype) {
  const int most = c->tune_bin_max ? std::min(c->tune_bin_max, BIN_MAX) : BIN_MAX;
  BinGeom g{};
  g.nd = nd;
  g.ntype = ntype;
  for (int edge = 16; edge <= 24; edge += 4) {
    g.nt = (nd + edge - 1) / edge;
    const long long bins = (long long)g.nt * g.nt * g.nt * ntype;
    if (bins > most) continue;
    g.ntile = g.nt * g.nt * g.nt;
    g.bins = (int)bins;
    g.dnd = fast_div((unsigned)nd);
    return g;
  }
  return g;
}

// Whether the entries' buffer may take `bytes`: it has them, or they are at
// most a quarter of the memory that is free (the atomics need none).
static bool bin_fits(const exh_ctx* c, size_t bytes) {
  if (c->tune_bin_room) return bytes <= (size_t)c->tune_bin_room << 20;
  if (bytes <= c->cap[BUF_BIN_ENT]) return true;
  size_t avail = 0, total = 0;
  return hipMemGetInfo(&avail, &total) == hipSuccess &&
         bytes <= (avail + c->cap[BUF_BIN_ENT]) / 4;
}

// False where the entries find no room: nothing of the grid is written then.
//
// Up to BIN_READ particles, room for the most entries there can be (8 each) is
// set aside.  Above, the host reads their number, unless the call runs on the
// second stream, where it must go ahead of the halo finder: there 2 a particle
// are set aside (LPT particles of 4 Mpc/h cells have 1.3 with CIC and 1.6 with
// TSC), and the device goes over to the atomics where they do not suffice
// (200^3 chain, FP32, CIC: 3.3 ms in bins, 7.2 after an overflow, 8.0 with
// atomics alone).  Whether there is room is decided before the first launch,
// except for a number that is read where one entry a particle would fit.
// Chains of sides that the tiles do not divide, 8 entries a particle counted
// first against 2: FP64, 330^3 30.6 -> 13.1 ms (refused after the count), FP32,
// 350^3 10.2 ms both, 9.1 -> 5.0 GB held.
template <typename T, int WIN>
static bool run_binned(exh_ctx* c, const BinParticles<T>& a, const BinGeom& g, T* grid,
                       unsigned long long* counts) {
  const bool all = a.np <= (c->tune_bin_read ? c->tune_bin_read : BIN_READ);
  const bool read = !all && !(c->aux && c->stream == c->aux);
  const int edge = (g.nd + g.nt - 1) / g.nt, pitch = edge * edge * edge;
  long long most = 8 * a.np;  // a particle's stencils reach at most 8 tiles
  // a split bin has more than BIN_PART entries, so its parts hold at least
  // half of BIN_PART on average
  auto slots = [&]() { return (int)(2 * most / BIN_PART); };
  auto entry_bytes = [&]() { return ((size_t)most * sizeof(BinEntry<T>) + 255) & ~(size_t)255; };
  auto bytes = [&]() { return entry_bytes() + (size_t)slots() * a.nsub * pitch * 8; };
  if (read) {
    most = a.np;
  } else if (!all) {
    most = a.np * (c->tune_bin_entries ? c->tune_bin_entries : 32) / 16;
    if (bytes() > BIN_BYTES) return false;
  }
  if (!bin_fits(c, bytes())) return false;
  // particles per workgroup of the counting passes: at least 4 a thread, and
  // at least as many as there are counters to clear
  const long long chunk =
      std::max<long long>({4096, (a.np + 511) / 512, (long long)g.bins / 2});
  const unsigned nb = grid_for(a.np, (int)chunk);
  size_t off_b = 0;
  auto take = [&](size_t b) {
    const size_t r = off_b;
    off_b += (b + 255) & ~(size_t)255;
    return r;
  };
  const size_t o_cnt = take((size_t)g.bins * 4), o_off = take(((size_t)g.bins + 1) * 4),
               o_parts = take((size_t)g.bins * 4), o_slot = take(((size_t)g.bins + 1) * 4),
               o_place = take((size_t)nb * g.bins * 4);
  char* buf = (char*)ctx_buf(c, BUF_BINS, off_b);
  int* cnt = (int*)(buf + o_cnt);
  int* off = (int*)(buf + o_off);
  int* parts = (int*)(buf + o_parts);
  int* slot = (int*)(buf + o_slot);
  int* place = (int*)(buf + o_place);
  const int lds = g.bins * 4;
  hipLaunchKernelGGL(k_zero<int>, dim3(grid_for(g.bins, 256)), dim3(256), 0, c->stream, cnt,
                     (size_t)g.bins);
  auto kc = k_bin_count<T, WIN>;
  EXH_CHECK_HIP(hipFuncSetAttribute((const void*)kc, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    lds));
  hipLaunchKernelGGL(kc, dim3(nb), dim3(1024), lds, c->stream, a, g, chunk, cnt, place, counts);
  EXH_LAUNCH_CHECK();
  exclusive_scan<int>(c, cnt, off, g.bins, BUF_BIN_SCAN);
  hipLaunchKernelGGL(k_bin_parts, dim3(grid_for(g.bins, 256)), dim3(256), 0, c->stream, cnt,
                     g.bins, parts);
  EXH_LAUNCH_CHECK();
  exclusive_scan<int>(c, parts, slot, g.bins, BUF_BIN_SCAN);
  if (read) {
    int* h = (int*)ctx_pinned(c, 256);
    EXH_CHECK_HIP(hipMemcpyAsync(h, off + g.bins, 4, hipMemcpyDeviceToHost, c->stream));
    EXH_CHECK_HIP(hipStreamSynchronize(c->stream));
    most = h[0];
    if (!bin_fits(c, bytes())) return false;
  }
  const int nslot = slots();
  const size_t eb = entry_bytes();
  // tested on the device only where the entries may exceed it: every block of
  // the passes waits for the number first
  const bool test = !all && !read;
  const BinRoom lim = test ? BinRoom{off + g.bins, most} : BinRoom{};
  char* ebuf = (char*)ctx_buf(c, BUF_BIN_ENT, bytes());
  BinEntry<T>* ent = (BinEntry<T>*)ebuf;
  double* partial = (double*)(ebuf + eb);
  auto ks = k_bin_scatter<T, WIN>;
  EXH_CHECK_HIP(hipFuncSetAttribute((const void*)ks, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    lds));
  hipLaunchKernelGGL(ks, dim3(nb), dim3(1024), lds, c->stream, a, g, chunk, off, place, lim, ent);
  const int dlds = pitch * 8;
  const bool norm = !a.mass;
  auto kd = k_bin_deposit<T, WIN>;
  EXH_CHECK_HIP(hipFuncSetAttribute((const void*)kd, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    dlds));
  hipLaunchKernelGGL(kd, dim3((unsigned)(g.bins + nslot)), dim3(256), dlds, c->stream, g, ent, off,
                     slot, a.L, a.Lb, a.nsub, norm, counts, partial, pitch, lim, grid);
  if (nslot > 0)
    hipLaunchKernelGGL(k_bin_merge<T>, dim3((unsigned)nslot), dim3(256), 0, c->stream, g, slot,
                       a.nsub, norm, counts, partial, pitch, lim, grid);
  EXH_LAUNCH_CHECK();
  c->deposit_path = EXH_DEPOSIT_BINNED;
  c->bin_total = lim.total;
  c->bin_cap = lim.cap;
  if (test) {
    const size_t ng = (size_t)g.nd * g.nd * g.nd;
    hipLaunchKernelGGL(k_zero_over<T>, dim3(2048), dim3(256), 0, c->stream, grid,
                       ng * g.ntype * a.nsub, lim);
    hipLaunchKernelGGL((k_deposit<T, WIN>), dim3(std::min(grid_for(a.np, 256), 8192u)), dim3(256),
                       0, c->stream, a.pos, a.vel, a.mass, a.type, a.np, g.nd, a.L, a.Lb,
                       a.direction, a.rsd, a.nsub, grid, (unsigned long long*)nullptr, lim);
    if (norm)
      hipLaunchKernelGGL(k_normalise<T>, dim3(1024, g.ntype * a.nsub), dim3(256), 0, c->stream,
                         grid, ng, a.nsub, counts, lim);
    EXH_LAUNCH_CHECK();
  }
  return true;
}

template <typename T>
void run_grid(exh_ctx* c, const T* pos, const T* vel, const T* mass, const int* type,
              long long np, int ntype, int nd, double L, double Om0, double z, int direction,
              int window, double R, double R_times, int interlacing, int folds, T* grid,
              void* scratch_dev) {
  EXH_REQUIRE(window >= EXH_WINDOW_NGP && window <= EXH_WINDOW_TSC, EXH_ERR_UNSUPPORTED,
              "window %d: NGP (1), CIC (2), sphere (3), exponential (4) or TSC (5)", window);
  EXH_REQUIRE(window < 3 || window > 4 || (R > 0 && (window == 3 || R_times > 0)), EXH_ERR_ARG,
              "the sphere and exponential windows need R > 0 (and R_times > 0)");
  EXH_REQUIRE(nd > 0 && ntype >= 1 && folds >= 1, EXH_ERR_ARG, "bad grid arguments");
  EXH_REQUIRE(direction < 0 || vel != nullptr, EXH_ERR_ARG, "redshift space needs velocities");
  const int nsub = interlacing ? 2 : 1;
  const size_t ng = (size_t)nd * nd * nd;
  T Lf = (T)((T)L / (T)folds);
  T Lb = Lf / (T)nd;
  // reference: vel * (1+z)^3 / H(Om0, z) (gridmodule.c:167-169)
  T Hz = (T)(100.0 * std::sqrt((T)Om0 * std::pow(1.0 + (T)z, 3) + (1.0 - (T)Om0)));
  T rsd = (T)(std::pow(1.0 + (T)z, 3.0) / (double)Hz);
  unsigned long long* counts = scratch_dev ? (unsigned long long*)scratch_dev
                                           : (unsigned long long*)ctx_buf(c, BUF_GCNT, 64 * 8);
  EXH_REQUIRE(ntype <= 64, EXH_ERR_ARG, "at most 64 tracer types");
  c->deposit_path = 0;
  const int nL = window == 3 || window == 4 ? 0 : lattice_side(np);
  const int nt = nL / TILE_L;
  const bool tiles = type == nullptr && nL >= TILE_L && nL % TILE_L == 0 && nd % nt == 0 &&
                     deposit_lds_bytes() > 0;
  const int stencil = window == 1 ? 1 : (window == 2 ? 8 : 27);
  // Particles in any order: the binned deposit where the atomics of k_deposit
  // (particles x cells x sub-grids, 26 G/s) would take longer than the
  // binning's passes.  Measured with n particles in random order, atomics and
  // bins: CIC, two sub-grids, nd = 64, n = 20 k (the atomics) 54 us; 130 k:
  // 143 and 112; 400 k: 357 and 166; TSC, nd = 128, 40 k: 103 and 81.
  // A cube of particles is most likely a lattice in order, whose atomics
  // coalesce in part: CIC, 52^3: 77 and 92, two sub-grids 112 and 125; TSC,
  // 52^3: 165 and 120; 100^3 CIC 313 and 103, TSC 884 and 156.
  const long long atomics = np * stencil * nsub;
  if (window != 3 && window != 4 && !tiles && !scratch_dev && np <= BIN_NP &&
      atomics >= (nL > 0 ? 3 * BIN_ATOMICS : BIN_ATOMICS)) {
    const BinGeom g = bin_geom(c, nd, ntype);
    if (g.bins > 0) {
      TimedScope ts(c, window == 2 ? "cic_deposit" : (window == 1 ? "ngp_deposit" : "tsc_deposit"));
      hipLaunchKernelGGL(k_zero<unsigned long long>, dim3(1), dim3(64), 0, c->stream, counts,
                         (size_t)64);
      const BinParticles<T> a{pos, vel, mass, type, np, Lf, Lb, rsd, direction, nsub};
      const bool done = window == 1   ? run_binned<T, 1>(c, a, g, grid, counts)
                        : window == 2 ? run_binned<T, 2>(c, a, g, grid, counts)
                                      : run_binned<T, 5>(c, a, g, grid, counts);
      if (done) return;
    }
  }
  {
    TimedScope ts(c, "grid_zero");
    const size_t nz = ng * ntype * nsub;
    if (reinterpret_cast<uintptr_t>(grid) % 16 == 0)
      hipLaunchKernelGGL(k_zero16<T>, dim3(grid_for(nz * sizeof(T) / 16 + 1, 256 * 4)),
                         dim3(256), 0, c->stream, grid, nz);
    else
      hipLaunchKernelGGL(k_zero<T>, dim3(grid_for(nz, 256 * 8)), dim3(256), 0, c->stream, grid,
                         nz);
    hipLaunchKernelGGL(k_zero<unsigned long long>, dim3(1), dim3(64), 0, c->stream, counts,
                       (size_t)64);
    EXH_LAUNCH_CHECK();
  }
  unsigned gsz = grid_for(np, 256);
  if (gsz > 65536 * 4) gsz = 65536 * 4;
  // particles on a lattice whose side is a multiple of the tile side, with
  // a grid side divisible by the number of tiles per axis, are deposited
  // tile by tile through LDS (correct for any order; fast when the array is
  // in lattice order, as LPT particles are)
  if (window == 3 || window == 4) {
    // spherical / exponential windows: normalised by the deposited weight
    double* wsum = scratch_dev ? (double*)scratch_dev : (double*)ctx_buf(c, BUF_GCNT, 128 * 8);
    hipLaunchKernelGGL(k_zero<double>, dim3(1), dim3(128), 0, c->stream, wsum, (size_t)128);
    c->deposit_path = EXH_DEPOSIT_SPHERES;
    {
      TimedScope ts(c, window == 3 ? "sphere_deposit" : "exp_deposit");
      const unsigned gs = std::min(grid_for(np, 256), 65536u);
#define EXH_DEPS(E)                                                                              \
  hipLaunchKernelGGL((k_deposit_sphere<T, E>), dim3(gs), dim3(256), 0, c->stream, pos, vel, mass, \
                     type, np, nd, Lf, Lb, (T)R, (T)R_times, direction, rsd, nsub, ntype * nsub,  \
                     grid, wsum)
      if (window == 3) EXH_DEPS(false);
      if (window == 4) EXH_DEPS(true);
#undef EXH_DEPS
      EXH_LAUNCH_CHECK();
    }
    if (!mass) {
      TimedScope ts(c, "grid_normalise");
      hipLaunchKernelGGL(k_normalise_w<T>, dim3(grid_for(ng, 256 * 8), ntype * nsub), dim3(256),
                         0, c->stream, grid, ng, wsum);
      EXH_LAUNCH_CHECK();
    }
    return;
  }
  {
    TimedScope ts(c, window == 2 ? "cic_deposit" : (window == 1 ? "ngp_deposit" : "tsc_deposit"));
    const int W = tiles ? nd / nt : 0;
    const int wh = deposit_window_margin();
    // the window's tile shape and accumulator (EXH_DEPOSIT_TILE,
    // EXH_DEPOSIT_ACC), where the lattice and the grid divide into it and
    // the window fits the LDS; nd >= E keeps every window cell within
    // (-nd, 2nd), where the flush's single-step wrap is exact
    // (float windows for float grids only; the default shape when the
    // chosen one does not fit)
    WinShape ws = c->tune_deposit_tile ? tile_shape(c->tune_deposit_tile) : deposit_window_shape();
    int acc = sizeof(T) == 8 ? 8 : (c->tune_deposit_acc ? c->tune_deposit_acc : deposit_window_acc());
    if (acc == 1 && mass) acc = 8;  // fixed point holds weights in [0, 1] only
    int Wq[3] = {0, 0, 0}, win_lds = 0;
    auto fits = [&](const WinShape& w, int a) {
      if (!(tiles && deposit_window_enabled() && nL % w.px == 0 && nL % w.py == 0 &&
            nL % w.pz == 0))
        return false;
      const int pq[3] = {w.px, w.py, w.pz};
      long long cells = 1;
      for (int q = 0; q < 3; q++) {
        const int ntq = nL / pq[q];
        if (nd % ntq != 0) return false;
        Wq[q] = nd / ntq;
        if (nd < Wq[q] + 2 * wh) return false;
        cells *= Wq[q] + 2 * wh;
      }
      win_lds = (int)std::min<long long>(cells * (a == 1 ? 4 : a), 1 << 30);
      return win_lds <= WIN_LDS_MAX;
    };
    bool win = fits(ws, acc);
    if (!win && (ws.px != 16 || ws.py != 16 || ws.pz != 16)) {
      ws = WinShape{16, 16, 16};
      win = fits(ws, acc);
    }
    if (!win && acc != 8) {
      acc = 8;
      win = fits(ws, acc);
    }
    if (win) {
      const unsigned nblk = (unsigned)((nL / ws.px) * (nL / ws.py) * (nL / ws.pz));
      const unsigned nwg = deposit_workgroups() > 0 ? std::min(nblk, (unsigned)deposit_workgroups())
                                                    : nblk;
      const DepositWinArgs<T> da{pos, vel, mass, nL, nd, Wq[0], Wq[1], Wq[2], wh, Lf, Lb,
                                 direction, rsd, nsub, grid, counts, (int)nblk};
      launch_window_any<T>(c, window, acc, ws, nwg, win_lds, da);
      c->deposit_path = EXH_DEPOSIT_WINDOWS;
    } else if (tiles) {
      c->deposit_path = EXH_DEPOSIT_TILES;
      const int lds = deposit_lds_bytes();
      const int cap = lds / (int)sizeof(double);
      const unsigned nblk = (unsigned)nt * nt * nt;
#define EXH_DEPT(WN)                                                                           \
  do {                                                                                         \
    EXH_CHECK_HIP(hipFuncSetAttribute((const void*)k_deposit_tiles<T, WN>,                     \
                                      hipFuncAttributeMaxDynamicSharedMemorySize, lds));       \
    hipLaunchKernelGGL((k_deposit_tiles<T, WN>), dim3(nblk), dim3(TILE_THREADS), lds,          \
                       c->stream, pos, vel, mass, nL, nd, W, Lf, Lb, direction, rsd, nsub, cap, \
                       grid, counts);                                                          \
  } while (0)
      if (window == 1) EXH_DEPT(1);
      if (window == 2) EXH_DEPT(2);
      if (window == 5) EXH_DEPT(5);
#undef EXH_DEPT
    } else {
      c->deposit_path = EXH_DEPOSIT_ATOMICS;
#define EXH_DEP(W)                                                                         \
  hipLaunchKernelGGL((k_deposit<T, W>), dim3(gsz), dim3(256), 0, c->stream, pos, vel, mass, \
                     type, np, nd, Lf, Lb, direction, rsd, nsub, grid, counts, BinRoom{})
      if (window == 1) EXH_DEP(1);
      if (window == 2) EXH_DEP(2);
      if (window == 5) EXH_DEP(5);
#undef EXH_DEP
    }
    EXH_LAUNCH_CHECK();
  }
  if (!mass) {
    TimedScope ts(c, "grid_normalise");
    if (reinterpret_cast<uintptr_t>(grid) % 16 == 0 && (ng * sizeof(T)) % 16 == 0)
      hipLaunchKernelGGL(k_normalise16<T>, dim3(grid_for(ng * sizeof(T) / 16, 256 * 2),
                                                ntype * nsub),
                         dim3(256), 0, c->stream, grid, ng, nsub, counts);
    else
      hipLaunchKernelGGL(k_normalise<T>, dim3(grid_for(ng, 256 * 8), ntype * nsub), dim3(256),
                         0, c->stream, grid, ng, nsub, counts, BinRoom{});
    EXH_LAUNCH_CHECK();
  }
}

// ---------------------------------------------------------------------------
// power spectrum
// ---------------------------------------------------------------------------
struct PowerArgs {
  int nd, nz, ntype, nsub, Nk, ls, NPs, NV, direction, kbin;
  const double2* ex;  // per-axis phase e^{-i k Lb/2}: x/y [nd], z [nz]
  const double2* ez;
  const double* wx;   // per-axis window^-1 factors
  const double* wz;
  double Normk;
  int rwin;         // 3 (sphere) or 4 (exponential): window per mode, else 0
  double knT, RT;   // kn and R in the grid's precision
  // bin index arithmetic
  float knf, kminf, dkf;
  double kn, kmin, dk;
  FastDiv dz, dnd;  // divisions by nz and nd (flat mode index -> i, j, k)
};

__device__ inline double legendre_d(int l, double x) {
  if (l == 0) return 1.0;
  double p0 = 1.0, p1 = x;
  for (int n = 1; n < l; n++) {
    double p2 = ((2 * n + 1) * x * p1 - n * p0) / (n + 1);
    p0 = p1;
    p1 = p2;
  }
  return p1;
}

// One DPP move of a double (its two halves) across the wave; lanes without
// a source read 0.  Controls: row_shr:n = 0x110 + n (within rows of 16
// lanes), row_bcast:15 = 0x142 (lane 15 of each row to the next row),
// row_bcast:31 = 0x143 (lane 31 to rows 2 and 3).
template <int CTRL>
__device__ inline double dpp_d(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double(
      (long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned long long)(unsigned)lo));
}

// Inclusive segmented sum over a full wave: lane l gets x summed over lanes
// sstart .. l (sstart <= l, the start of l's segment), in a fixed order:
// shifts by 1, 2, 4 and 8 within rows of 16 lanes, then the last lane of
// row 0 into row 1 and of row 2 into row 3, then lane 31 into rows 2 and 3,
// each added only where the source lies in the lane's segment.  DPP moves
// run on the vector ALU; the cross-lane shuffles they replace went through
// the LDS crossbar.
__device__ inline double seg_scan_d(double x, int lane, int sstart) {
  const int rl = lane & 15, rs = lane & ~15;
  double y;
  y = dpp_d<0x111>(x);
  if (rl >= 1 && lane - 1 >= sstart) x += y;
  y = dpp_d<0x112>(x);
  if (rl >= 2 && lane - 2 >= sstart) x += y;
  y = dpp_d<0x114>(x);
  if (rl >= 4 && lane - 4 >= sstart) x += y;
  y = dpp_d<0x118>(x);
  if (rl >= 8 && lane - 8 >= sstart) x += y;
  y = dpp_d<0x142>(x);
  if ((rs == 16 || rs == 48) && sstart < rs) x += y;
  y = dpp_d<0x143>(x);
  if (rs >= 32 && sstart < 32) x += y;
  return x;
}

static constexpr int PW_MAXV = 64;  // max values per mode (pairs x multipoles + 1)

// Bin of half-complex mode (i, j, k), or -1: the reference's mode mask
// (powermodule.c:47-55) and bin index floor((|k| - k_min) / dk) in float
// (kbin 4, spectrum_h.c:39-48) or double (kbin 8); |k| and mu along the
// line of sight as the binning evaluates them.
__device__ inline int mode_bin(const PowerArgs& a, int i, int j, int k, double& kmod, double& mu) {
  const int nd = a.nd;
  const bool masked = (k == 0 || k == nd / 2) &&
                      ((i > nd / 2 && j > nd / 2) || (i == 0 || i == nd / 2) ||
                       (j == 0 || j == nd / 2) || (i > nd / 2 && j < nd / 2));
  if (masked) return -1;
  const int fi = (2 * i < nd) ? i : i - nd, fj = (2 * j < nd) ? j : j - nd;
  const int fk = (2 * k < nd) ? k : k - nd;
  int b;
  if (a.kbin == 4) {
    float kx = (float)fi * a.knf, ky = (float)fj * a.knf, kz = (float)fk * a.knf;
    float km = sqrtf(kx * kx + ky * ky + kz * kz);
    float tmp = (km - a.kminf) / a.dkf;
    b = (int)floorf(tmp);
    kmod = km;
    if (a.direction == 0) mu = (double)(kx / km);
    if (a.direction == 1) mu = (double)(ky / km);
    if (a.direction == 2) mu = (double)(kz / km);
  } else {
    double kx = fi * a.kn, ky = fj * a.kn, kz = fk * a.kn;
    double km = sqrt(kx * kx + ky * ky + kz * kz);
    b = (int)floor((km - a.kmin) / a.dk);
    kmod = km;
    if (a.direction == 0) mu = kx / km;
    if (a.direction == 1) mu = ky / km;
    if (a.direction == 2) mu = kz / km;
  }
  return (b < 0 || b >= a.Nk) ? -1 : b;
}

// W of the sphere (3) and exponential (4) windows at mode (fi, fj, fk), in
// the grid's precision with the reference's double intermediates
// (spectrum_h.c:60-67).
template <typename T>
__device__ inline T window_r(const PowerArgs& a, int fi, int fj, int fk) {
  const T kn = (T)a.knT, R = (T)a.RT;
  const T k1 = (T)fi * kn, k2 = (T)fj * kn, k3 = (T)fk * kn;
  if (a.rwin == 3) {
    const T kmod = (T)sqrt((double)(k1 * k1 + k2 * k2 + k3 * k3));
    const T kR = kmod * R;
    const T sc = kR != (T)0 ? (T)(sin((double)kR) / (double)kR) : (T)1;
    return (T)(3.0 / kmod / kmod / R / R * ((double)sc - cos((double)kR)));
  }
  const T kmod = k1 * k1 + k2 * k2 + k3 * k3;
  return (T)exp((double)(-kmod * R * R) / 2.0);
}

// The waves' LDS sums and counts added in a fixed order: one partial per block.
__device__ __forceinline__ void power_block_sums(const double* lds, int nw, int Nk, int NV,
                                                 double* part, unsigned* pcnt) {
  __syncthreads();
  double* out = part + (size_t)blockIdx.x * Nk * NV;
  unsigned* cout = pcnt + (size_t)blockIdx.x * Nk;
  for (int q = threadIdx.x; q < Nk * NV; q += blockDim.x) {
    double s = 0.0;
    for (int w = 0; w < nw; w++) s += lds[(size_t)w * Nk * NV + q];
    out[q] = s;
  }
  for (int q = threadIdx.x; q < Nk; q += blockDim.x) {
    unsigned s = 0;
    const unsigned* cbase = (const unsigned*)(lds + (size_t)nw * Nk * NV);
    for (int w = 0; w < nw; w++) s += cbase[(size_t)w * Nk + q];
    cout[q] = s;
  }
}

// Phase e^{-i theta} = e1 e2 e3 of a mode and the factor that undoes the window
// and normalises, the same for every tracer; F is the precision of the combine
// (float for the monopole of a float grid, else double).
template <typename F>
struct ModePhase {
  F er, ei, wk;
};
template <typename T, typename F, bool RWIN>
__device__ __forceinline__ ModePhase<F> mode_phase(const PowerArgs& a, int i, int j, int k,
                                                   const double2& e1d, const double2& e2d,
                                                   const double2& e3d) {
  const int nd = a.nd;
  ModePhase<F> m;
  if (RWIN && a.rwin) {
    const int fi = (2 * i < nd) ? i : i - nd, fj = (2 * j < nd) ? j : j - nd;
    const int fk = (2 * k < nd) ? k : k - nd;
    m.wk = (F)(a.Normk / (double)window_r<T>(a, fi, fj, fk));
  } else {
    m.wk = (F)a.wx[i] * (F)a.wx[j] * (F)a.wz[k] * (F)a.Normk;
  }
  const F x1 = (F)e1d.x, y1 = (F)e1d.y, x2 = (F)e2d.x, y2 = (F)e2d.y, x3 = (F)e3d.x,
          y3 = (F)e3d.y;
  const F pr = x1 * x2 - y1 * y2, pi = x1 * y2 + y1 * x2;
  m.er = pr * x3 - pi * y3;
  m.ei = pr * y3 + pi * x3;
  return m;
}

// A tracer's combined, deconvolved mode, (f1 + f2 e^{-i theta}) / 2 with two
// sub-grids.
template <typename F, typename C2>
__device__ __forceinline__ void mode_combine(const ModePhase<F>& m, int nsub, const C2& f1,
                                             const C2& f2, double& dr, double& di) {
  F re = (F)f1.x, im = (F)f1.y;
  if (nsub == 2) {
    re = (re + ((F)f2.x * m.er - (F)f2.y * m.ei)) * (F)0.5;
    im = (im + ((F)f2.x * m.ei + (F)f2.y * m.er)) * (F)0.5;
  }
  dr = (double)(re * m.wk);
  di = (double)(im * m.wk);
}

// One tracer, LS multipoles, a window that is a product over the axes; KB is
// the binning's precision.  Bound by vector instructions: with a segmented
// sum of every 64 modes and value (k_power_bins) the sums took most of them.
// Here a lane keeps one k and steps along j, sums the modes of its current bin
// in registers (a bin holds a few steps) and adds them to its wave's LDS sums
// when the bin changes; a wave's sums are its own, so the order of its
// instructions does not depend on timing.  Lanes that change to one bin at the
// same step meet in one ds_add_f64: that equal calls give equal bits rests on
// the LDS adding the lanes of an instruction in a fixed order, as it has in
// every run.  A wave takes 64 neighbouring k and `jlen` steps;
// the nz % 64 last k share a wave `rpw` rows at a time.  512^3, FP32,
// interlaced: monopole, binned in double, 620 -> 464 us; l_max = 4, binned in
// float, 1158 -> 520 us.
struct PowerLines {
  int jlen, kfull, rem, rpw, njs, njr;
};
template <typename T, int LS, int KB>
__global__ __launch_bounds__(256) void k_power_lines(PowerArgs a, PowerLines g,
                                                     const typename cplx<T>::type* gk,
                                                     double* part, unsigned* pcnt) {
  extern __shared__ double lds[];
  using C2 = typename cplx<T>::type;
  constexpr int NV = LS + 1, U = 4;
  using F = typename std::conditional<LS == 1 && sizeof(T) == 4, float, double>::type;
  a.kbin = KB;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int Nk = a.Nk, nd = a.nd, nz = a.nz;
  double* acc = lds + (size_t)wave * Nk * NV;
  unsigned* cacc = (unsigned*)(lds + (size_t)nw * Nk * NV) + (size_t)wave * Nk;
  for (int q = lane; q < Nk * NV; q += 64) acc[q] = 0.0;
  for (int q = lane; q < Nk; q += 64) cacc[q] = 0;
  __syncthreads();
  const size_t nh = (size_t)nd * nd * nz;
  const long long nfull = (long long)nd * g.kfull * g.njs;
  const long long ntask = nfull + (g.rem ? (long long)nd * g.njr : 0);
  const long long gw = (long long)blockIdx.x * nw + wave, tw = (long long)gridDim.x * nw;
  for (long long t = gw; t < ntask; t += tw) {
    int i, j, k, dj, jend;
    if (t < nfull) {
      const int r = (int)(t / g.kfull);
      k = (int)(t - (long long)r * g.kfull) * 64 + lane;
      i = r / g.njs;
      j = (r - i * g.njs) * g.jlen;
      dj = 1;
      jend = min(j + g.jlen, nd);
    } else {
      const int r = (int)(t - nfull), row = lane / g.rem;
      k = g.kfull * 64 + lane - row * g.rem;
      i = r / g.njr;
      const int j0 = (r - i * g.njr) * g.jlen * g.rpw;
      dj = g.rpw;
      jend = min(j0 + g.jlen * g.rpw, nd);
      j = row < g.rpw ? j0 + row : jend;
    }
    const double2 e1 = a.ex[i], e3 = a.ez[k];
    int cb = -1;  // the lane's bin and its sums
    unsigned cn = 0;
    double cs[NV];
    auto flush = [&]() {
      if (cb >= 0) {
#pragma unroll
        for (int v = 0; v < NV; v++) atomicAdd(&acc[(size_t)cb * NV + v], cs[v]);
        atomicAdd(&cacc[cb], cn);
      }
    };
    const C2* p = gk + ((size_t)i * nd + j) * nz + k;
    const size_t dp = (size_t)dj * nz;
    for (; j < jend; j += U * dj, p += U * dp) {
      C2 f1[U], f2[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const bool in = j + u * dj < jend;
        const C2* q = in ? p + u * dp : p;
        f1[u] = q[0];
        f2[u] = a.nsub == 2 ? q[nh] : f1[u];
      }
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int ju = j + u * dj;
        if (ju >= jend) break;
        double kmod = 0, mu = 0;
        const int b = mode_bin(a, i, ju, k, kmod, mu);
        if (b != cb) {
          flush();
          cb = b;
          cn = 0;
#pragma unroll
          for (int v = 0; v < NV; v++) cs[v] = 0.0;
        }
        if (b < 0) continue;
        double dr, di;
        mode_combine(mode_phase<T, F, false>(a, i, ju, k, e1, a.ex[ju], e3), a.nsub, f1[u], f2[u],
                     dr, di);
        const double P = dr * dr + di * di;
#pragma unroll
        for (int l = 0; l < LS; l++) cs[l] += P * legendre_d(2 * l, mu);
        cs[LS] += kmod;
        cn++;
      }
    }
    flush();
  }
  power_block_sums(lds, nw, Nk, NV, part, pcnt);
}

// Several tracers, more multipoles, or a window of |k|: segmented sums of 64 modes at a time.
template <typename T>
__global__ void k_power_bins(PowerArgs a, const typename cplx<T>::type* gk, double* part,
                             unsigned* pcnt) {
  extern __shared__ double lds[];
  using C2 = typename cplx<T>::type;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int NV = a.NV, Nk = a.Nk, LS = a.ls;
  double* acc = lds + (size_t)wave * Nk * NV;
  unsigned* cacc = (unsigned*)(lds + (size_t)nw * Nk * NV) + (size_t)wave * Nk;
  for (int q = lane; q < Nk * NV; q += 64) acc[q] = 0.0;
  for (int q = lane; q < Nk; q += 64) cacc[q] = 0;
  __syncthreads();
  const int nd = a.nd, nz = a.nz;
  const size_t nh = (size_t)nd * nd * nz;
  // waves walk 64-mode chunks of the flat mode index (a row of nd/2+1
  // modes would leave a chunk with one active lane); bins change at row
  // boundaries, which the segmented scan below handles like any change
  const long long nchunks = (long long)((nh + 63) / 64);
  const long long gw = (long long)blockIdx.x * nw + wave, tw = (long long)gridDim.x * nw;
  for (long long ch = gw; ch < nchunks; ch += tw) {
    const size_t id = (size_t)ch * 64 + lane;
    int i = 0, j = 0, k = nz;  // k = nz: no mode
    long long row = (long long)((nh - 1) / nz);
    if (id < nh) {
      if (nh < (1ull << 31)) {
        const unsigned r = fdiv((unsigned)id, a.dz);
        k = (int)((unsigned)id - r * (unsigned)nz);
        i = (int)fdiv(r, a.dnd);
        j = (int)(r - (unsigned)i * (unsigned)nd);
        row = r;
      } else {
        k = (int)(id % nz);
        const size_t r = id / nz;
        j = (int)(r % nd);
        i = (int)(r / nd);
        row = (long long)r;
      }
    }
    // the chunk's rows: within one row bins never decrease, so a bin has
    // at most one segment per row; tails update the accumulators one row
    // at a time (deterministically, without two lanes on one address)
    const long long row0 = __shfl(row, 0, 64);
    const int part = (int)(row - row0);
    const int nparts = (int)(__shfl(row, 63, 64) - row0) + 1;
    double kmod = 0, mu = 0;
    const int b = k < nz ? mode_bin(a, i, j, k, kmod, mu) : -1;
    const bool valid = b >= 0;
    // segment bookkeeping
    const int bprev = __shfl_up(b, 1, 64);
    const bool head = valid && (lane == 0 || bprev != b);
    const unsigned long long heads = __ballot(head);
    const unsigned long long upto = heads & (lane == 63 ? ~0ull : ((2ull << lane) - 1));
    const int sstart = upto ? 63 - __clzll((long long)upto) : 0;
    const int bnext = __shfl_down(b, 1, 64);
    const bool tail = valid && (lane == 63 || bnext != b);
    // combined modes of every tracer
    double dr[8], di[8];
    if (valid) {
      const double2 e1 = a.ex[i], e2 = a.ex[j], e3 = a.ez[k];
      const auto m = mode_phase<T, double, true>(a, i, j, k, e1, e2, e3);
      for (int t = 0; t < a.ntype; t++) {
        const C2* f = gk + (size_t)(t * a.nsub) * nh + id;
        const C2 f1 = f[0];
        C2 f2 = f1;
        if (a.nsub == 2) f2 = f[nh];
        mode_combine(m, a.nsub, f1, f2, dr[t], di[t]);
      }
    }
    // values: pair products x P_2l(mu), then |k|
    for (int v = 0; v < NV; v++) {
      double x = 0.0;
      if (valid) {
        if (v == NV - 1) {
          x = kmod;
        } else {
          int pair = v / LS, l2 = 2 * (v % LS);
          // pair index -> (l, m <= l) in the reference's order
          int l = 0;
          while ((l + 1) * (l + 2) / 2 <= pair) l++;
          int m = pair - l * (l + 1) / 2;
          x = (dr[l] * dr[m] + di[l] * di[m]) * legendre_d(l2, mu);
        }
      }
      x = seg_scan_d(x, lane, sstart);
      for (int p = 0; p < nparts; p++)
        if (tail && part == p) acc[(size_t)b * NV + v] += x;
    }
    for (int p = 0; p < nparts; p++)
      if (tail && part == p) cacc[b] += (unsigned)(lane - sstart + 1);
  }
  power_block_sums(lds, nw, Nk, NV, part, pcnt);
}

// One block per output value: 256 threads stride over the block partials,
// then a fixed-shape tree; the result does not depend on timing.
__global__ void k_power_reduce(const double* part, const unsigned* pcnt, int nblocks, int Nk,
                               int NV, double* sum, unsigned long long* cnt) {
  __shared__ double sd[256];
  __shared__ unsigned long long sc[256];
  const int q = blockIdx.x;
  const bool is_cnt = q >= Nk * NV;
  double s = 0.0;
  unsigned long long u = 0;
  for (int bl = threadIdx.x; bl < nblocks; bl += 256) {
    if (is_cnt)
      u += pcnt[(size_t)bl * Nk + (q - Nk * NV)];
    else
      s += part[(size_t)bl * Nk * NV + q];
  }
  sd[threadIdx.x] = s;
  sc[threadIdx.x] = u;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) {
      sd[threadIdx.x] += sd[threadIdx.x + w];
      sc[threadIdx.x] += sc[threadIdx.x + w];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    if (is_cnt)
      cnt[q - Nk * NV] = sc[0];
    else
      sum[q] = sd[0];
  }
}

template <typename T>
static double sinc_t(T x) {
  T r;
  if (x != (T)0)
    r = (T)(std::sin((double)x) / (double)x);
  else
    r = (T)1;
  return r;
}

// Binning arguments of the P(k) passes: per-axis tables with the
// reference's fft_real rounding of kn and Lb (uploaded to the context's
// table slot), window, Normk and the bin-edge arithmetic.
template <typename T>
static PowerArgs make_power_args(exh_ctx* c, int ntype, int nd, double L, int window, double R,
                                 int interlacing, int Nk, double k_min, double k_max, int l_max,
                                 int direction, int kbin_precision) {
  const int nsub = interlacing ? 2 : 1;
  const int nz = nd / 2 + 1;
  const int NPs = ntype * (ntype + 1) / 2, ls = l_max / 2 + 1;
  const int NV = NPs * ls + 1;

  // per-axis tables with the reference's fft_real rounding of kn and Lb
  T Lr = (T)L;
  T kn = (T)(2 * M_PI / (double)Lr);
  T Lb = Lr / (T)nd;
  T Normk = (T)std::pow((double)(Lr / (T)(nd * nd)), 3.0 / 2.0);
  // NGP, CIC, TSC: per-axis sinc powers; the sphere and exponential windows
  // are functions of |k|, evaluated per mode in the kernel
  int pw = (window == 0 || window == 3 || window == 4) ? 0 : (window == 1 ? 1 : (window == 2 ? 2 : 3));
  // ex [nd], ez [nz], wx [nd], wz [nz] in one array and one upload (four took
  // 5 us each of the 76 us of a 64^3 call)
  const size_t tn = 3 * ((size_t)nd + nz);
  std::vector<double> tab(tn);
  double2* ex = (double2*)tab.data();
  double2* ez = ex + nd;
  double* wx = (double*)(ez + nz);
  double* wz = wx + nd;
  for (int i = 0; i < nd; i++) {
    T kx = (2 * i < nd) ? (T)i * kn : (T)(i - nd) * kn;
    double th = (double)kx * (double)Lb / 2.0;
    ex[i] = make_double2(std::cos(th), -std::sin(th));
    wx[i] = 1.0 / std::pow(sinc_t<T>((T)((double)kx * (double)Lb / 2.0)), pw);
  }
  for (int k = 0; k < nz; k++) {
    T kz = (2 * k < nd) ? (T)k * kn : (T)(k - nd) * kn;
    double th = (double)kz * (double)Lb / 2.0;
    ez[k] = make_double2(std::cos(th), -std::sin(th));
    wz[k] = 1.0 / std::pow(sinc_t<T>((T)((double)kz * (double)Lb / 2.0)), pw);
  }
  double2* dex = (double2*)ctx_buf(c, BUF_PTAB, tn * 8);
  double2* dez = dex + nd;
  double* dwx = (double*)(dez + nz);
  double* dwz = dwx + nd;
  EXH_CHECK_HIP(hipMemcpyAsync(dex, tab.data(), tn * 8, hipMemcpyHostToDevice, c->stream));

  PowerArgs a{};
  a.nd = nd;
  a.nz = nz;
  a.ntype = ntype;
  a.nsub = nsub;
  a.Nk = Nk;
  a.ls = ls;
  a.NPs = NPs;
  a.NV = NV;
  a.direction = direction;
  a.kbin = kbin_precision;
  a.dz = fast_div((unsigned)nz);
  a.dnd = fast_div((unsigned)nd);
  a.ex = dex;
  a.ez = dez;
  a.wx = dwx;
  a.wz = dwz;
  a.Normk = (double)Normk;
  a.rwin = (window == 3 || window == 4) ? window : 0;
  a.knT = (double)kn;
  a.RT = (double)(T)R;
  // bin edges: fft_real arithmetic for kbin 4 (spectrum_h.c:39-48, powermodule.c:13)
  a.knf = (float)(2 * M_PI / (double)(float)L);
  a.kminf = (float)k_min;
  a.dkf = ((float)k_max - (float)k_min) / (float)Nk;
  a.kn = 2 * M_PI / L;
  a.kmin = k_min;
  a.dk = (k_max - k_min) / Nk;
  if (sizeof(T) == 4) {
    // the FP32 build rounds kn to float before use
    a.kn = (double)(float)a.kn;
  }
  return a;
}

template <typename T>
void run_power(exh_ctx* c, const T* grid, int ntype, int nd, double L, int window, double R,
               int interlacing, int Nk, double k_min, double k_max, int l_max, int direction,
               int kbin_precision, double* k_out, double* P_out, long long* count_out,
               bool deferred) {
  using C2 = typename cplx<T>::type;
  EXH_REQUIRE(nd >= 2 && nd % 2 == 0, EXH_ERR_ARG, "nd must be even");
  EXH_REQUIRE(ntype >= 1 && ntype <= 8, EXH_ERR_UNSUPPORTED, "1 to 8 tracer types supported");
  EXH_REQUIRE(Nk >= 1 && l_max >= 0, EXH_ERR_ARG, "bad binning");
  EXH_REQUIRE(window >= 0 && window <= 5, EXH_ERR_UNSUPPORTED, "window %d cannot be deconvolved",
              window);
  const int nsub = interlacing ? 2 : 1;
  const int nz = nd / 2 + 1;
  const size_t nh = (size_t)nd * nd * nz;
  const int NPs = ntype * (ntype + 1) / 2, ls = l_max / 2 + 1;
  const int NV = NPs * ls + 1;
  EXH_REQUIRE(NV <= PW_MAXV, EXH_ERR_UNSUPPORTED, "too many spectra x multipoles");
  C2* gk = (C2*)ctx_buf(c, BUF_GRIDK, nh * ntype * nsub * sizeof(C2));
  fft_r2c(c, nd, nd, nd, sizeof(T) == 4 ? 4 : 8, ntype * nsub, grid, gk);
  PowerArgs a = make_power_args<T>(c, ntype, nd, L, window, R, interlacing, Nk, k_min, k_max,
                                   l_max, direction, kbin_precision);

  // LDS: per wave Nk*NV doubles + Nk counters
  size_t per_wave = (size_t)Nk * NV * 8 + (size_t)Nk * 4;
  int waves = 4;
  while (waves > 1 && per_wave * waves > 60 * 1024) waves--;
  EXH_REQUIRE(per_wave <= 60 * 1024, EXH_ERR_UNSUPPORTED,
              "Nk x spectra x multipoles too large for the LDS accumulator (%zu bytes)", per_wave);
  // one tracer up to l = 4, no window of |k|: lines along j, at least 8 steps each and about one
  // for each of 8192 waves
  const bool lines = ntype == 1 && ls <= 3 && !a.rwin;
  PowerLines g{};
  long long nrows = (long long)nd * nd;
  if (lines) {
    g.kfull = nz / 64;
    g.rem = nz % 64;
    g.rpw = g.rem ? 64 / g.rem : 0;
    g.jlen = (int)std::min<long long>(std::max<long long>(8, nrows * std::max(g.kfull, 1) / 8192),
                                      128);
    g.njs = (nd + g.jlen - 1) / g.jlen;
    g.njr = g.rem ? (nd + g.jlen * g.rpw - 1) / (g.jlen * g.rpw) : 0;
    nrows = (long long)nd * (g.kfull * g.njs + g.njr);  // waves' tasks
  }
  int nblocks = (int)std::min<long long>((nrows + waves - 1) / waves, 2048);
  size_t poff = 0;
  auto ptake = [&](size_t bytes) {
    size_t r = poff;
    poff += (bytes + 255) & ~(size_t)255;
    return r;
  };
  size_t o_part = ptake((size_t)nblocks * Nk * NV * 8), o_pcnt = ptake((size_t)nblocks * Nk * 4),
         o_sum = ptake((size_t)Nk * NV * 8), o_cnt = ptake((size_t)Nk * 8);
  char* pbuf = (char*)ctx_buf(c, BUF_PART, poff);
  double* part = (double*)(pbuf + o_part);
  unsigned* pcnt = (unsigned*)(pbuf + o_pcnt);
  double* sum = (double*)(pbuf + o_sum);
  unsigned long long* cnt = (unsigned long long*)(pbuf + o_cnt);
  {
    TimedScope ts(c, "power_bins");
    if (lines) {
      auto k = ls == 1   ? (a.kbin == 4 ? k_power_lines<T, 1, 4> : k_power_lines<T, 1, 8>)
               : ls == 2 ? (a.kbin == 4 ? k_power_lines<T, 2, 4> : k_power_lines<T, 2, 8>)
                         : (a.kbin == 4 ? k_power_lines<T, 3, 4> : k_power_lines<T, 3, 8>);
      hipLaunchKernelGGL(k, dim3(nblocks), dim3(64 * waves), per_wave * waves, c->stream, a, g, gk,
                         part, pcnt);
    } else {
      hipLaunchKernelGGL(k_power_bins<T>, dim3(nblocks), dim3(64 * waves), per_wave * waves,
                         c->stream, a, gk, part, pcnt);
    }
    EXH_LAUNCH_CHECK();
  }
  {
    TimedScope ts(c, "power_reduce");
    hipLaunchKernelGGL(k_power_reduce, dim3((unsigned)(Nk * NV + Nk)), dim3(256), 0,
                       c->stream, part, pcnt, nblocks, Nk, NV, sum, cnt);
    EXH_LAUNCH_CHECK();
  }
  c->power_pending.o_sum = o_sum;
  c->power_pending.o_cnt = o_cnt;
  c->power_pending.Nk = Nk;
  c->power_pending.NV = NV;
  c->power_pending.NPs = NPs;
  c->power_pending.ls = ls;
  if (!deferred) power_copy_out(c, k_out, P_out, count_out);
}

// Copies the sums of the last run_power to the host (waits for the stream)
// and forms k, P and the mode counts per bin.
void power_copy_out(exh_ctx* c, double* k_out, double* P_out, long long* count_out) {
  const auto& pp = c->power_pending;
  const int Nk = pp.Nk, NV = pp.NV, NPs = pp.NPs, ls = pp.ls;
  char* pbuf = (char*)c->buf[BUF_PART];
  // the counts follow the sums: one copy
  const size_t o_hc = pp.o_cnt - pp.o_sum, hbytes = o_hc + (size_t)Nk * 8;
  char* h = (char*)ctx_pinned(c, hbytes);
  EXH_CHECK_HIP(hipMemcpyAsync(h, pbuf + pp.o_sum, hbytes, hipMemcpyDeviceToHost, c->stream));
  EXH_CHECK_HIP(hipStreamSynchronize(c->stream));
  const double* hs = (const double*)h;
  const unsigned long long* hc = (const unsigned long long*)(h + o_hc);
  for (int b = 0; b < Nk; b++) {
    long long n = (long long)hc[b];
    if (count_out) count_out[b] = n;
    if (k_out) k_out[b] = n > 0 ? hs[(size_t)b * NV + NV - 1] / n : 0.0;
    for (int p = 0; p < NPs; p++)
      for (int l = 0; l < ls; l++) {
        double s = hs[(size_t)b * NV + p * ls + l];
        if (P_out) P_out[((size_t)p * ls + l) * Nk + b] = n > 0 ? (4.0 * l + 1.0) * s / n : 0.0;
      }
  }
}

// ---------------------------------------------------------------------------
// adjoints of the monopole P(k) and of the mass assignment
// ---------------------------------------------------------------------------
// In place over the modes F = r2c(delta) of one grid (no interlacing):
// G = (dL/dF) / w with dL/dF = gPn[b] wk^2 F for every mode the forward
// pass bins (same mask and bin index), 0 elsewhere.  With
// P_b = sum_b |F wk|^2 / N_b, gPn[b] = 2 dL/dP_b / N_b.  w is the weight
// of a stored mode in the c2r (2 for 0 < kz < nd/2, 1 in the kz = 0, nd/2
// planes), so that c2r(G) is the gradient with respect to the real grid:
// the transpose of the r2c.
template <typename T>
__global__ void k_power_adjoint(PowerArgs a, const double* gPn, typename cplx<T>::type* gk) {
  using C2 = typename cplx<T>::type;
  const int nd = a.nd, nz = a.nz;
  const size_t nh = (size_t)nd * nd * nz;
  for (size_t id = blockIdx.x * (size_t)blockDim.x + threadIdx.x; id < nh;
       id += (size_t)gridDim.x * blockDim.x) {
    int i, j, k;
    if (nh < (1ull << 31)) {
      const unsigned r = fdiv((unsigned)id, a.dz);
      k = (int)((unsigned)id - r * (unsigned)nz);
      i = (int)fdiv(r, a.dnd);
      j = (int)(r - (unsigned)i * (unsigned)nd);
    } else {
      k = (int)(id % nz);
      const size_t r = id / nz;
      j = (int)(r % nd);
      i = (int)(r / nd);
    }
    double kmod, mu;
    const int b = mode_bin(a, i, j, k, kmod, mu);
    C2 out{(T)0, (T)0};
    if (b >= 0) {
      const int fi = (2 * i < nd) ? i : i - nd, fj = (2 * j < nd) ? j : j - nd;
      const double wk = a.rwin ? a.Normk / (double)window_r<T>(a, fi, fj, (2 * k < nd) ? k : k - nd)
                               : a.wx[i] * a.wx[j] * a.wz[k] * a.Normk;
      const double w = (k == 0 || 2 * k == nd) ? 1.0 : 2.0;
      const double f = gPn[b] * wk * wk / w;
      const C2 F = gk[id];
      out = C2{(T)(f * (double)F.x), (T)(f * (double)F.y)};
    }
    gk[id] = out;
  }
}

// CIC weights of one axis and their derivatives with respect to the
// coordinate, for the cell xt and its neighbour o toward the particle
// (dep_cic's arithmetic).
template <typename T>
__device__ inline void cic_axis(T x, T Ld, int nd, int& xt, int& o, T& t, T& d, double& dt) {
  T q = x / Ld;
  xt = (int)floor(q);
  if (xt == nd) xt -= 1;
  T dx = (T)((double)q - ((double)xt + 0.5));
  double sgn = 1.0;
  if (dx >= (T)0) {
    o = xt + 1 == nd ? 0 : xt + 1;
  } else {
    o = xt == 0 ? nd - 1 : xt - 1;
    dx = -dx;
    sgn = -1.0;
  }
  t = (T)(1.0 - (double)dx);
  d = dx;
  dt = -sgn / (double)Ld;  // d t / dx; d d / dx = -dt
}

// dL/dS of every particle of the nL^3 lattice (the LPT particles, lattice
// order) from g = dL/drho on the grid: the transpose of the deposit, the
// weights' derivatives at the particle times g at the cells it feeds, times
// `scale` (1 / rho_bar for normalised grids).  The positions are recomputed
// from the displacements, q + S with q = (i + 1/2) Lc, in double: for a
// float field this places each particle relative to the weights' kinks (the
// cell centres) to the precision of S rather than to that of a float
// coordinate up to L, so the gradient is that of the exact positions.
template <typename T, int WIN>
__global__ void k_deposit_adjoint(const T* S, int nL, double Lc, int nd, double L, const T* g,
                                  double scale, T* gpos) {
  using D = double;
  const D Ld = L / (D)nd;
  const size_t n2 = (size_t)nd * nd;
  const long long np = (long long)nL * nL * nL;
  for (long long p = blockIdx.x * (long long)blockDim.x + threadIdx.x; p < np;
       p += (long long)gridDim.x * blockDim.x) {
    const long long r = p / nL;
    const int q[3] = {(int)(r / nL), (int)(r % nL), (int)(p % nL)};
    D x[3];
    bool ok = true;
    for (int a = 0; a < 3; a++) {
      D v = ((D)q[a] * Lc + Lc / 2.0) + (D)S[3 * p + a];
      x[a] = wrap_while<D>(v, L);
      ok = ok && isfinite(x[a]);
    }
    double gx[3] = {0.0, 0.0, 0.0};
    if (ok && WIN == 2) {
      int xt[3], o[3];
      D t[3], d[3];
      double dt[3];
      for (int a = 0; a < 3; a++) cic_axis<D>(x[a], Ld, nd, xt[a], o[a], t[a], d[a], dt[a]);
      // the eight cells: c[ax] selects xt (0) or o (1) per axis
      for (int c = 0; c < 8; c++) {
        const int s0 = c & 1, s1 = (c >> 1) & 1, s2 = (c >> 2) & 1;
        const size_t id = (size_t)(s0 ? o[0] : xt[0]) * n2 + (size_t)(s1 ? o[1] : xt[1]) * nd +
                          (size_t)(s2 ? o[2] : xt[2]);
        const double gv = (double)g[id];
        const double w0 = s0 ? d[0] : t[0], w1 = s1 ? d[1] : t[1], w2 = s2 ? d[2] : t[2];
        const double e0 = s0 ? -dt[0] : dt[0], e1 = s1 ? -dt[1] : dt[1], e2 = s2 ? -dt[2] : dt[2];
        gx[0] += gv * e0 * w1 * w2;
        gx[1] += gv * w0 * e1 * w2;
        gx[2] += gv * w0 * w1 * e2;
      }
    } else if (ok && WIN == 5) {
      int cc[3];
      double w[3][3], dw[3][3];
      for (int a = 0; a < 3; a++) {
        const double u = x[a] / Ld - 0.5;
        const double cf = floor(u + 0.5);
        const double dd = u - cf;
        cc[a] = (int)cf;
        w[a][0] = 0.5 * (0.5 - dd) * (0.5 - dd);
        w[a][1] = 0.75 - dd * dd;
        w[a][2] = 0.5 * (0.5 + dd) * (0.5 + dd);
        const double du = 1.0 / (double)Ld;
        dw[a][0] = -(0.5 - dd) * du;
        dw[a][1] = -2.0 * dd * du;
        dw[a][2] = (0.5 + dd) * du;
      }
      for (int ia = 0; ia < 3; ia++) {
        int ix = cc[0] + ia - 1;
        ix = ix < 0 ? ix + nd : (ix >= nd ? ix - nd : ix);
        for (int ib = 0; ib < 3; ib++) {
          int iy = cc[1] + ib - 1;
          iy = iy < 0 ? iy + nd : (iy >= nd ? iy - nd : iy);
          for (int ie = 0; ie < 3; ie++) {
            int iz = cc[2] + ie - 1;
            iz = iz < 0 ? iz + nd : (iz >= nd ? iz - nd : iz);
            const double gv = (double)g[(size_t)ix * n2 + (size_t)iy * nd + iz];
            gx[0] += gv * dw[0][ia] * w[1][ib] * w[2][ie];
            gx[1] += gv * w[0][ia] * dw[1][ib] * w[2][ie];
            gx[2] += gv * w[0][ia] * w[1][ib] * dw[2][ie];
          }
        }
      }
    }
    for (int a = 0; a < 3; a++) gpos[3 * p + a] = (T)(gx[a] * scale);
  }
}

// Gradient of the monopole P(k) of `grid` with respect to the grid values:
// g = c2r(G) with G from k_power_adjoint; gP: host [Nk] dL/dP_b.  Runs
// the forward binning first (the counts N_b, and P_out / count_out when
// given).  The modes are left in the context's BUF_GRIDK and overwritten.
template <typename T>
void run_power_adjoint(exh_ctx* c, const T* grid, int nd, double L, int window, double R,
                       int Nk, double k_min, double k_max, int kbin_precision, const double* gP,
                       T* g, double* P_out, long long* count_out) {
  using C2 = typename cplx<T>::type;
  std::vector<long long> cnt(Nk);
  std::vector<double> Pk(Nk);
  run_power<T>(c, grid, 1, nd, L, window, R, 0, Nk, k_min, k_max, 0, -1, kbin_precision, nullptr,
               Pk.data(), cnt.data(), false);
  if (P_out) std::copy(Pk.begin(), Pk.end(), P_out);
  if (count_out) std::copy(cnt.begin(), cnt.end(), count_out);
  std::vector<double> gPn(Nk);
  for (int b = 0; b < Nk; b++) gPn[b] = cnt[b] > 0 ? 2.0 * gP[b] / (double)cnt[b] : 0.0;
  PowerArgs a = make_power_args<T>(c, 1, nd, L, window, R, 0, Nk, k_min, k_max, 0, -1,
                                   kbin_precision);
  double* dg = (double*)ctx_pinned(c, (size_t)Nk * sizeof(double));
  std::copy(gPn.begin(), gPn.end(), dg);
  double* dgd = (double*)ctx_buf(c, BUF_ADJ_TAB, (size_t)Nk * sizeof(double));
  EXH_CHECK_HIP(hipMemcpyAsync(dgd, dg, (size_t)Nk * sizeof(double), hipMemcpyHostToDevice,
                               c->stream));
  const size_t nh = (size_t)nd * nd * (nd / 2 + 1);
  C2* gk = (C2*)c->buf[BUF_GRIDK];
  {
    TimedScope ts(c, "power_adjoint");
    hipLaunchKernelGGL(k_power_adjoint<T>, dim3(std::min<size_t>((nh + 255) / 256, 65536)),
                       dim3(256), 0, c->stream, a, dgd, gk);
    EXH_LAUNCH_CHECK();
  }
  fft_c2r(c, nd, nd, nd, sizeof(T) == 4 ? 4 : 8, 1, gk, g);
  EXH_CHECK_HIP(hipStreamSynchronize(c->stream));  // dg is pinned host staging
}

// dL/dS (gS [nL^3][3]) of the LPT particles from dL/ddelta (g) of their
// unweighted, normalised grid: delta = rho ng / np - 1.  Lc: the lattice
// spacing (the box's cell), L the box side.
template <typename T>
void run_deposit_adjoint(exh_ctx* c, const T* S, int nL, double Lc, int nd, double L, int window,
                         const T* g, T* gS) {
  EXH_REQUIRE(window == EXH_WINDOW_CIC || window == EXH_WINDOW_TSC, EXH_ERR_UNSUPPORTED,
              "the adjoint supports the CIC (2) and TSC (5) windows");
  const long long np = (long long)nL * nL * nL;
  const double scale = (double)nd * nd * nd / (double)np;
  const unsigned gs = (unsigned)std::min<long long>((np + 255) / 256, 65536);
  TimedScope ts(c, "deposit_adjoint");
  if (window == EXH_WINDOW_CIC)
    hipLaunchKernelGGL((k_deposit_adjoint<T, 2>), dim3(gs), dim3(256), 0, c->stream, S, nL, Lc,
                       nd, L, g, scale, gS);
  else
    hipLaunchKernelGGL((k_deposit_adjoint<T, 5>), dim3(gs), dim3(256), 0, c->stream, S, nL, Lc,
                       nd, L, g, scale, gS);
  EXH_LAUNCH_CHECK();
}

template void run_power_adjoint<float>(exh_ctx*, const float*, int, double, int, double, int,
                                       double, double, int, const double*, float*, double*,
                                       long long*);
template void run_power_adjoint<double>(exh_ctx*, const double*, int, double, int, double, int,
                                        double, double, int, const double*, double*, double*,
                                        long long*);
template void run_deposit_adjoint<float>(exh_ctx*, const float*, int, double, int, double, int,
                                         const float*, float*);
template void run_deposit_adjoint<double>(exh_ctx*, const double*, int, double, int, double, int,
                                          const double*, double*);

// ---------------------------------------------------------------------------
// halo abundance: abundance_compute (spectrum.c:535-600) and
// Measure_Abundance (abundance.c:4-36)
// ---------------------------------------------------------------------------
// Per-block smallest and largest mass (at most 1024 blocks, reduced on the
// host).
template <typename T>
__global__ void k_mass_range(const T* Mh, long long n, T* bmin, T* bmax) {
  __shared__ T smin[256], smax[256];
  T lo = (T)1e30, hi = (T)-1e30;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    const T m = Mh[i];
    lo = m < lo ? m : lo;
    hi = m > hi ? m : hi;
  }
  smin[threadIdx.x] = lo;
  smax[threadIdx.x] = hi;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) {
      smin[threadIdx.x] = smin[threadIdx.x + w] < smin[threadIdx.x] ? smin[threadIdx.x + w]
                                                                    : smin[threadIdx.x];
      smax[threadIdx.x] = smax[threadIdx.x + w] > smax[threadIdx.x] ? smax[threadIdx.x + w]
                                                                    : smax[threadIdx.x];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    bmin[blockIdx.x] = smin[0];
    bmax[blockIdx.x] = smax[0];
  }
}

// Counts and mass sums per bin floor((ln M - ln Mmin) / dlnM), kept for
// 0 < bin < Nm as the reference does; LDS histograms, one atomic per block
// and bin.
template <typename T>
__global__ void k_abundance(const T* Mh, long long n, double lnMmin, float dlnM, int Nm,
                            unsigned long long* cnt, double* msum) {
  extern __shared__ double ab_lds[];
  double* ssum = ab_lds;
  unsigned* scnt = (unsigned*)(ab_lds + Nm);
  for (int b = threadIdx.x; b < Nm; b += blockDim.x) {
    ssum[b] = 0.0;
    scnt[b] = 0;
  }
  __syncthreads();
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    const double f = floor((log((double)Mh[i]) - lnMmin) / (double)dlnM);
    if (f > 0.0 && f < (double)Nm) {
      const int b = (int)f;
      atomicAdd(&scnt[b], 1u);
      atomicAdd(&ssum[b], (double)Mh[i]);
    }
  }
  __syncthreads();
  for (int b = threadIdx.x; b < Nm; b += blockDim.x)
    if (scnt[b]) {
      atomicAdd(&cnt[b], (unsigned long long)scnt[b]);
      atomicAdd(&msum[b], ssum[b]);
    }
}

template <typename T>
void run_abundance(exh_ctx* c, const T* Mh, long long nh, double Mmin_in, double Mmax_in, int Nm,
                   double Lc_in, int ndx, int ndy, int ndz, double* Mmean_out, double* dn_out,
                   double* dn_err_out) {
  EXH_REQUIRE(Nm >= 1 && Nm <= 4096, EXH_ERR_ARG, "Nm must lie in [1, 4096]");
  EXH_REQUIRE(nh >= 0 && (nh == 0 || Mh != nullptr), EXH_ERR_ARG, "null masses");
  T Mmin = (T)Mmin_in, Mmax = (T)Mmax_in;
  const T Lc = (T)Lc_in;
  const T Lx = Lc * (T)ndx, Ly = Lc * (T)ndy, Lz = Lc * (T)ndz;
  const unsigned nb = std::max(1u, std::min(grid_for(nh, 256), 1024u));
  char* buf = (char*)ctx_buf(c, BUF_MISC, 256 + 2 * 1024 * sizeof(T) + (size_t)Nm * 16);
  if (Mmin < (T)0 || Mmax < (T)0) {
    // abundance_compute's defaults: 0.9999 x the smallest, 1.0001 x the largest
    T* bmin = (T*)(buf + 256);
    T* bmax = bmin + 1024;
    hipLaunchKernelGGL(k_mass_range<T>, dim3(nb), dim3(256), 0, c->stream, Mh, nh, bmin, bmax);
    EXH_LAUNCH_CHECK();
    std::vector<T> hmin(nb), hmax(nb);
    EXH_CHECK_HIP(hipMemcpyAsync(hmin.data(), bmin, nb * sizeof(T), hipMemcpyDeviceToHost,
                                 c->stream));
    EXH_CHECK_HIP(hipMemcpyAsync(hmax.data(), bmax, nb * sizeof(T), hipMemcpyDeviceToHost,
                                 c->stream));
    EXH_CHECK_HIP(hipStreamSynchronize(c->stream));
    if (Mmin < (T)0) {
      T lo = (T)1e+20;
      for (long long b = 0; b < (long long)nb && nh > 0; b++) lo = hmin[b] < lo ? hmin[b] : lo;
      Mmin = (T)((double)lo * 0.9999);
    }
    if (Mmax < (T)0) {
      for (long long b = 0; b < (long long)nb && nh > 0; b++) Mmax = hmax[b] > Mmax ? hmax[b] : Mmax;
      Mmax = (T)((double)Mmax * 1.0001);
    }
  }
  const float dlnM = (float)((std::log((double)Mmax) - std::log((double)Mmin)) / Nm);
  unsigned long long* cnt = (unsigned long long*)(buf + 256 + 2 * 1024 * sizeof(T));
  double* msum = (double*)(cnt + Nm);
  hipLaunchKernelGGL(k_zero<unsigned long long>, dim3(grid_for(Nm, 256)), dim3(256), 0, c->stream,
                     cnt, (size_t)Nm);
  hipLaunchKernelGGL(k_zero<double>, dim3(grid_for(Nm, 256)), dim3(256), 0, c->stream, msum,
                     (size_t)Nm);
  if (nh > 0)
    hipLaunchKernelGGL(k_abundance<T>, dim3(nb), dim3(256), (size_t)Nm * 12, c->stream, Mh, nh,
                       std::log((double)Mmin), dlnM, Nm, cnt, msum);
  EXH_LAUNCH_CHECK();
  std::vector<unsigned long long> hc(Nm);
  std::vector<double> hs(Nm);
  EXH_CHECK_HIP(hipMemcpyAsync(hc.data(), cnt, Nm * 8, hipMemcpyDeviceToHost, c->stream));
  EXH_CHECK_HIP(hipMemcpyAsync(hs.data(), msum, Nm * 8, hipMemcpyDeviceToHost, c->stream));
  EXH_CHECK_HIP(hipStreamSynchronize(c->stream));
  // the reference's arithmetic: T sums and quotients, float dlnM
  const T V = Lx * Ly * Lz;
  for (int b = 0; b < Nm; b++) {
    const int N = (int)hc[b];
    const T mean = N > 0 ? (T)((T)hs[b] / (T)N) : (T)0;
    if (Mmean_out) Mmean_out[b] = (double)mean;
    if (dn_out) dn_out[b] = (double)(T)((T)N / V / (T)dlnM);
    if (dn_err_out) dn_err_out[b] = (double)(T)(std::sqrt((double)N) / (double)V / (double)dlnM);
  }
}

template void run_abundance<float>(exh_ctx*, const float*, long long, double, double, int,
                                   double, int, int, int, double*, double*, double*);
template void run_abundance<double>(exh_ctx*, const double*, long long, double, double, int,
                                    double, int, int, int, double*, double*, double*);

// ---------------------------------------------------------------------------
// bispectrum: bi_compute (spectrum.c:291-406) / Bi_Spectrum (bimodule.c)
// ---------------------------------------------------------------------------
// Combined, deconvolved modes of every tracer (Compute_gridk,
// spectrum_h.c:83-167, in the grid's precision as the reference evaluates
// it) and the shell of every mode, Indice(|k|, k_min, dk) (bimodule.c:72-75);
// per-shell sums of |k| and mode counts.
struct ShellArgs {
  int nd, nz, ntype, nsub, Nk, window;
  double kn, Lb, Normk, R, kmin, dk;  // kn, Lb, Normk, R, kmin, dk hold values of T
  FastDiv dz, dnd;
};

template <typename T>
__device__ inline T sinc_dev(T x) {
  return x != (T)0 ? (T)(sin((double)x) / (double)x) : (T)1;
}

template <typename T>
__global__ void k_shell_modes(ShellArgs a, const typename cplx<T>::type* raw,
                              typename cplx<T>::type* gk, short* shell, double* ksum,
                              unsigned long long* kcnt) {
  using C2 = typename cplx<T>::type;
  extern __shared__ double sm_lds[];
  double* sks = sm_lds;
  unsigned* scs = (unsigned*)(sm_lds + a.Nk);
  for (int q = threadIdx.x; q < a.Nk; q += blockDim.x) {
    sks[q] = 0.0;
    scs[q] = 0;
  }
  __syncthreads();
  const size_t nh = (size_t)a.nd * a.nd * a.nz;
  const T kn = (T)a.kn, Lb = (T)a.Lb, Normk = (T)a.Normk, kmin = (T)a.kmin, dk = (T)a.dk;
  for (size_t id = blockIdx.x * (size_t)blockDim.x + threadIdx.x; id < nh;
       id += (size_t)gridDim.x * blockDim.x) {
    const unsigned r = fdiv((unsigned)id, a.dz);
    const int k = (int)((unsigned)id - r * (unsigned)a.nz);
    const int i = (int)fdiv(r, a.dnd);
    const int j = (int)(r - (unsigned)i * (unsigned)a.nd);
    const T kx = (T)((2 * i < a.nd) ? i : i - a.nd) * kn;
    const T ky = (T)((2 * j < a.nd) ? j : j - a.nd) * kn;
    const T kz = (T)((2 * k < a.nd) ? k : k - a.nd) * kn;
    // W (spectrum_h.c:51-70)
    T W = (T)1;
    if (a.window == 1 || a.window == 2 || a.window == 5) {
      const T s3 = sinc_dev<T>((T)((double)kx * (double)Lb / 2.0)) *
                   sinc_dev<T>((T)((double)ky * (double)Lb / 2.0)) *
                   sinc_dev<T>((T)((double)kz * (double)Lb / 2.0));
      W = a.window == 1 ? s3 : (T)pow((double)s3, a.window == 2 ? 2.0 : 3.0);
    } else if (a.window == 3) {
      const T km = (T)sqrt((double)(kx * kx + ky * ky + kz * kz));
      const T kR = km * (T)a.R;
      W = (T)(3.0 / km / km / (T)a.R / (T)a.R * ((double)sinc_dev<T>(kR) - cos((double)kR)));
    } else if (a.window == 4) {
      const T km = kx * kx + ky * ky + kz * kz;
      W = (T)exp((double)(-km * (T)a.R * (T)a.R) / 2.0);
    }
    for (int t = 0; t < a.ntype; t++) {
      const C2 f1 = raw[(size_t)(t * a.nsub) * nh + id];
      C2 o;
      if (a.nsub == 2) {
        const C2 f2 = raw[(size_t)(t * a.nsub + 1) * nh + id];
        const double th = (double)((kx + ky + kz) * Lb) / 2.0;
        const double c = cos(th), sn = sin(th);
        o.x = (T)(((double)f1.x + (double)f2.x * c + (double)f2.y * sn) / 2.0 * (double)Normk /
                  (double)W);
        o.y = (T)(((double)f1.y + (double)f2.y * c - (double)f2.x * sn) / 2.0 * (double)Normk /
                  (double)W);
      } else {
        o.x = f1.x * Normk / W;
        o.y = f1.y * Normk / W;
      }
      gk[(size_t)t * nh + id] = o;
    }
    const T km = (T)sqrt((double)(kx * kx + ky * ky + kz * kz));
    const double f = floor((double)((km - kmin) / dk));
    const int b = (f >= 0.0 && f < (double)a.Nk) ? (int)f : -1;
    shell[id] = (short)b;
    if (b >= 0) {
      atomicAdd(&sks[b], (double)km);
      atomicAdd(&scs[b], 1u);
    }
  }
  __syncthreads();
  for (int q = threadIdx.x; q < a.Nk; q += blockDim.x)
    if (scs[q]) {
      atomicAdd(&ksum[q], sks[q]);
      atomicAdd(&kcnt[q], (unsigned long long)scs[q]);
    }
}

// The modes of shell s of every tracer and the shell's indicator (1 + 0i),
// zero elsewhere: ntype + 1 half-complex grids for one batched c2r.
template <typename T>
__global__ void k_shell_fill(const typename cplx<T>::type* gk, const short* shell, size_t nh,
                             int ntype, int s, typename cplx<T>::type* out) {
  using C2 = typename cplx<T>::type;
  for (size_t id = blockIdx.x * (size_t)blockDim.x + threadIdx.x; id < nh;
       id += (size_t)gridDim.x * blockDim.x) {
    const bool in = shell[id] == s;
    for (int t = 0; t < ntype; t++) {
      C2 v = gk[(size_t)t * nh + id];
      if (!in) v.x = v.y = (T)0;
      out[(size_t)t * nh + id] = v;
    }
    C2 one;
    one.x = in ? (T)1 : (T)0;
    one.y = (T)0;
    out[(size_t)ntype * nh + id] = one;
  }
}

// Sums over the cells of products of two or three shell fields, as a matrix
// product on the FP64 matrix cores: row r of the left factor holds the
// products A_r B_r of two fields, a column of the right factor a third field,
// and the sum over the cells is the contraction.  A job is one 16 x 16 tile
// of (rows, columns); the columns a row needs are a range, so only the tiles
// that hold a wanted triple are listed.  The pair sums are the sums of a row
// (a job with y set adds up its rows).
//
// A workgroup stages `ch` cells of every field in LDS; each wave runs its
// jobs over them, four cells a lane (one 16-byte LDS read per operand) and
// four v_mfma_f64_16x16x4 per job and 16 cells.  Lane l holds row (and
// column) l % 16 and cells 4 (l / 16) .. + 3; the result's row 4 v + l / 16,
// column l % 16 stands in accumulator v.  The products of two fields are
// exact to double's rounding, the third factor enters by a fused
// multiply-add.  What bounds it is the matrix cores' rate (128 flop per clock
// and CU; 0.31 ms of it) and the conversions and products beside: 20 shells
// of a 128^3 grid take 0.64 ms, and took 7.29 ms with one thread per product
// reading all its factors from LDS.
static constexpr int BS_JPW = 8;  // jobs per wave
typedef double bs_d4 __attribute__((ext_vector_type(4)));

template <typename T>
struct BsVec;
template <>
struct BsVec<float> {
  static constexpr int PAD = 4;
  using V = float4;
  static constexpr int W = 4;  // values per 16 bytes
};
template <>
struct BsVec<double> {
  static constexpr int PAD = 2;
  using V = double2;
  static constexpr int W = 2;
};

__device__ __forceinline__ void bs_read(const float* p, double (&v)[4]) {
  const float4 x = *reinterpret_cast<const float4*>(p);
  v[0] = x.x;
  v[1] = x.y;
  v[2] = x.z;
  v[3] = x.w;
}
__device__ __forceinline__ void bs_read(const double* p, double (&v)[4]) {
  const double2 x = reinterpret_cast<const double2*>(p)[0];
  const double2 y = reinterpret_cast<const double2*>(p)[1];
  v[0] = x.x;
  v[1] = x.y;
  v[2] = y.x;
  v[3] = y.y;
}

// rows: the two fields of each row, cols: each column's field, jobs: first
// row, first column, row sums wanted.  `split` waves share a job (few jobs).
template <typename T>
__global__ __launch_bounds__(256) void k_shell_products(const T* fields, int nfield, size_t ng,
                                                        int chs, const short2* rows,
                                                        const short* cols, const int4* jobs,
                                                        int njob, int per_wave, int split,
                                                        double* out, double* rowsum) {
  extern __shared__ __align__(16) unsigned char bs_raw[];
  T* lf = (T*)bs_raw;  // [nfield][ch + PAD]
  using V = typename BsVec<T>::V;
  constexpr int W = BsVec<T>::W;
  const int ch = 1 << chs, pitch = ch + BsVec<T>::PAD;
  const int lane = threadIdx.x & 63, l16 = lane & 15, kk = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j0 = ((int)blockIdx.y * 4 + w) / split * per_wave;
  const int nj = max(0, min(per_wave, njob - j0)), phase = w % split;
  int oa[BS_JPW], ob[BS_JPW], oc[BS_JPW];
  bool rsum[BS_JPW];
  bs_d4 acc[BS_JPW];
  double rs[BS_JPW];
#pragma unroll
  for (int q = 0; q < BS_JPW; q++) {
    const int4 job = jobs[q < nj ? j0 + q : 0];
    const short2 r = rows[job.x + l16];
    oa[q] = r.x * pitch + 4 * kk;
    ob[q] = r.y * pitch + 4 * kk;
    oc[q] = cols[job.y + l16] * pitch + 4 * kk;
    rsum[q] = job.z != 0;
    acc[q] = bs_d4{0.0, 0.0, 0.0, 0.0};
    rs[q] = 0.0;
  }
  const size_t nch = (ng + ch - 1) >> chs;
  const int vsh = chs - (W == 4 ? 2 : 1);  // log2 of the 16-byte vectors per field
  for (size_t chunk = blockIdx.x; chunk < nch; chunk += gridDim.x) {
    const size_t x0 = chunk << chs;
    const int nv = (int)(min((size_t)ch, ng - x0) / W);  // ng is a multiple of 8
    __syncthreads();
    for (int e = threadIdx.x; e < nfield << vsh; e += 256) {
      const int f = e >> vsh, v = e & ((1 << vsh) - 1);
      V x = {};
      if (v < nv) x = reinterpret_cast<const V*>(fields + (size_t)f * ng + x0)[v];
      *reinterpret_cast<V*>(lf + f * pitch + v * W) = x;
    }
    __syncthreads();
    for (int x = 16 * phase; x < ch; x += 16 * split) {
#pragma unroll
      for (int q = 0; q < BS_JPW; q++) {
        if (q >= nj) break;
        double va[4], vb[4], vc[4];
        bs_read(lf + oa[q] + x, va);
        bs_read(lf + ob[q] + x, vb);
        bs_read(lf + oc[q] + x, vc);
#pragma unroll
        for (int e = 0; e < 4; e++) va[e] *= vb[e];
        if (rsum[q]) rs[q] += (va[0] + va[1]) + (va[2] + va[3]);
#pragma unroll
        for (int e = 0; e < 4; e++)
          acc[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(va[e], vc[e], acc[q], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int q = 0; q < BS_JPW; q++) {
    if (q >= nj) break;
    double* o = out + (size_t)(j0 + q) * 256;
#pragma unroll
    for (int v = 0; v < 4; v++) atomicAdd(&o[(4 * v + kk) * 16 + l16], acc[q][v]);
    if (rsum[q]) {
      double t = rs[q];
      t += __shfl_xor(t, 16, 64);
      t += __shfl_xor(t, 32, 64);
      if (kk == 0) atomicAdd(&rowsum[jobs[j0 + q].x + l16], t);
    }
  }
}

// Configuration order of bimodule.c:49-317.
void bispectrum_configs(int Nk, std::vector<std::array<int, 3>>& tri) {
  tri.clear();
  for (int a = 0; a < Nk; a++) {
    for (int b = 0; b < a; b++) {
      if (b < a / 2) {
        tri.push_back({a, a, b});
        continue;
      }
      for (int c = std::max(a - b - 1, 0); c < b; c++) tri.push_back({a, b, c});
      tri.push_back({a, b, b});
      tri.push_back({a, a, b});
    }
    tri.push_back({a, a, a});
  }
}

template <typename T>
int run_bispectrum(exh_ctx* c, const T* grid, int ntype, int nd, double L, int window, double R,
                   int interlacing, int Nk, double k_min, double k_max, long long cap,
                   double* kP, double* Pk, double* Nk_out, double* kB, double* Bk,
                   double* Ntri_out) {
  using C2 = typename cplx<T>::type;
  EXH_REQUIRE(nd >= 2 && nd % 2 == 0, EXH_ERR_ARG, "nd must be even");
  EXH_REQUIRE(ntype >= 1 && ntype <= 4, EXH_ERR_UNSUPPORTED, "1 to 4 tracer types supported");
  EXH_REQUIRE(Nk >= 1 && Nk <= 4096, EXH_ERR_ARG, "Nk must lie in [1, 4096]");
  EXH_REQUIRE(window >= 0 && window <= 5, EXH_ERR_UNSUPPORTED, "window %d", window);
  EXH_REQUIRE(k_max > k_min, EXH_ERR_ARG, "k_max must exceed k_min");
  std::vector<std::array<int, 3>> tri;
  bispectrum_configs(Nk, tri);
  const long long ntri = (long long)tri.size();
  EXH_REQUIRE(cap >= ntri, EXH_ERR_ARG, "output capacity %lld below %lld configurations", cap,
              ntri);
  const int nsub = interlacing ? 2 : 1;
  const int nz = nd / 2 + 1;
  const size_t nh = (size_t)nd * nd * nz, ng = (size_t)nd * nd * nd;
  const int nf = ntype + 1;  // fields per shell: tracers and the indicator
  const size_t shells_bytes = (size_t)Nk * nf * ng * sizeof(T);
  EXH_REQUIRE(shells_bytes <= (size_t)96 << 30, EXH_ERR_UNSUPPORTED,
              "bispectrum: %zu bytes of shell fields exceed the 96 GiB budget", shells_bytes);
  // 1. r2c of every grid, combined modes and shells
  C2* raw = (C2*)ctx_buf(c, BUF_GRIDK, nh * ntype * nsub * sizeof(C2));
  fft_r2c(c, nd, nd, nd, sizeof(T) == 4 ? 4 : 8, ntype * nsub, grid, raw);
  size_t off = 0;
  auto take = [&](size_t b) {
    size_t r = off;
    off += (b + 255) & ~(size_t)255;
    return r;
  };
  const size_t o_gk = take(nh * ntype * sizeof(C2)), o_sh = take(nh * sizeof(short)),
               o_w = take(nh * nf * sizeof(C2)), o_ks = take((size_t)Nk * 8),
               o_kc = take((size_t)Nk * 8);
  char* kb = (char*)ctx_buf(c, BUF_SHELLK, off);
  C2* gk = (C2*)(kb + o_gk);
  short* shell = (short*)(kb + o_sh);
  C2* work = (C2*)(kb + o_w);
  double* ksum = (double*)(kb + o_ks);
  unsigned long long* kcnt = (unsigned long long*)(kb + o_kc);
  hipLaunchKernelGGL(k_zero<double>, dim3(grid_for(Nk, 256)), dim3(256), 0, c->stream, ksum,
                     (size_t)Nk);
  hipLaunchKernelGGL(k_zero<unsigned long long>, dim3(grid_for(Nk, 256)), dim3(256), 0,
                     c->stream, kcnt, (size_t)Nk);
  ShellArgs sa{};
  const T Lr = (T)L;
  sa.nd = nd;
  sa.nz = nz;
  sa.ntype = ntype;
  sa.nsub = nsub;
  sa.Nk = Nk;
  sa.window = window;
  sa.kn = (double)(T)(2 * M_PI / (double)Lr);
  sa.Lb = (double)(T)(Lr / (T)nd);
  sa.Normk = (double)(T)std::pow((double)(Lr / (T)(nd * nd)), 3.0 / 2.0);
  sa.R = (double)(T)R;
  sa.kmin = (double)(T)k_min;
  sa.dk = (double)(T)(((T)k_max - (T)k_min) / (T)Nk);
  sa.dz = fast_div((unsigned)nz);
  sa.dnd = fast_div((unsigned)nd);
  EXH_REQUIRE(nh < (1ull << 31), EXH_ERR_UNSUPPORTED, "grid too large for the shell kernels");
  {
    TimedScope ts(c, "bispec_shells");
    hipLaunchKernelGGL(k_shell_modes<T>, dim3(std::min(grid_for(nh, 256), 4096u)), dim3(256),
                       (size_t)Nk * 12, c->stream, sa, raw, gk, shell, ksum, kcnt);
    EXH_LAUNCH_CHECK();
    // 2. the real field of every shell and tracer, and of its indicator
    T* fields = (T*)ctx_buf(c, BUF_SHELLS, shells_bytes);
    for (int s = 0; s < Nk; s++) {
      hipLaunchKernelGGL(k_shell_fill<T>, dim3(std::min(grid_for(nh, 256), 8192u)), dim3(256), 0,
                         c->stream, gk, shell, nh, ntype, s, work);
      EXH_LAUNCH_CHECK();
      fft_c2r(c, nd, nd, nd, sizeof(T) == 4 ? 4 : 8, nf, work, fields + (size_t)s * nf * ng);
    }
  }
  // 3. the products: per configuration ntype^3 triples and the indicator's,
  // per shell the ntype (ntype+1)/2 pairs and the indicator's square.  Rows:
  // the pairs of shells (a, b) of the configurations, times ntype^2 for the
  // tracers, then once for the indicators; columns: the tracers' shells, then
  // the indicators'.
  const int NBs = ntype * ntype * ntype, NPs = ntype * (ntype + 1) / 2, nt2 = ntype * ntype;
  std::vector<int> pid((size_t)Nk * Nk, -1);
  std::vector<std::array<int, 2>> pairs;
  for (const auto& t : tri) {
    int& id = pid[(size_t)t[0] * Nk + t[1]];
    if (id < 0) {
      id = (int)pairs.size();
      pairs.push_back({t[0], t[1]});
    }
  }
  auto up16 = [](int n) { return (n + 15) & ~15; };
  const int np = (int)pairs.size();
  const int irow = up16(np * nt2), nrow = irow + up16(np);
  const int icol = up16(Nk * ntype), ncol = icol + up16(Nk);
  std::vector<short2> rows(nrow, make_short2(0, 0));
  std::vector<short> cols(ncol, 0);
  for (int p = 0; p < np; p++) {
    for (int f = 0; f < nt2; f++)
      rows[p * nt2 + f] = make_short2((short)(pairs[p][0] * nf + f / ntype),
                                      (short)(pairs[p][1] * nf + f % ntype));
    rows[irow + p] =
        make_short2((short)(pairs[p][0] * nf + ntype), (short)(pairs[p][1] * nf + ntype));
  }
  for (int s = 0; s < Nk; s++) {
    for (int f = 0; f < ntype; f++) cols[f * Nk + s] = (short)(s * nf + f);
    cols[icol + s] = (short)(s * nf + ntype);
  }
  // the tiles that hold a wanted triple
  const int ntr = nrow / 16, ntc = ncol / 16;
  std::vector<int> tile((size_t)ntr * ntc, -1);
  auto want = [&](int r, int c) { tile[(size_t)(r / 16) * ntc + c / 16] = 0; };
  for (const auto& t : tri) {
    const int p = pid[(size_t)t[0] * Nk + t[1]];
    for (int f = 0; f < nt2; f++)
      for (int f3 = 0; f3 < ntype; f3++) want(p * nt2 + f, f3 * Nk + t[2]);
    want(irow + p, icol + t[2]);
  }
  std::vector<int4> jobs;
  for (int r = 0; r < ntr; r++) {
    bool first = true;
    for (int q = 0; q < ntc; q++) {
      int& id = tile[(size_t)r * ntc + q];
      if (id < 0) continue;
      id = (int)jobs.size();
      jobs.push_back(make_int4(r * 16, q * 16, first ? 1 : 0, 0));
      first = false;
    }
  }
  const int njob = (int)jobs.size();
  size_t toff = 0;
  auto ttake = [&](size_t b) {
    size_t r = toff;
    toff += (b + 255) & ~(size_t)255;
    return r;
  };
  // one upload: jobs, rows, columns; then the sums
  const size_t o_jobs = ttake((size_t)njob * sizeof(int4)),
               o_rows = ttake((size_t)nrow * sizeof(short2)),
               o_cols = ttake((size_t)ncol * sizeof(short)), up_bytes = toff,
               o_out = ttake(((size_t)njob * 256 + nrow) * 8);
  std::vector<char> up(up_bytes);
  std::memcpy(up.data() + o_jobs, jobs.data(), (size_t)njob * sizeof(int4));
  std::memcpy(up.data() + o_rows, rows.data(), (size_t)nrow * sizeof(short2));
  std::memcpy(up.data() + o_cols, cols.data(), (size_t)ncol * sizeof(short));
  char* tb = (char*)ctx_buf(c, BUF_PART, toff);
  double* dout = (double*)(tb + o_out);
  double* drow = dout + (size_t)njob * 256;
  const size_t nout = (size_t)njob * 256 + nrow;
  EXH_CHECK_HIP(hipMemcpyAsync(tb, up.data(), up_bytes, hipMemcpyHostToDevice, c->stream));
  hipLaunchKernelGGL(k_zero<double>, dim3(grid_for(nout, 256)), dim3(256), 0, c->stream, dout,
                     nout);
  const int nfield = Nk * nf;
  // cells per chunk: the most that let two workgroups share a CU's LDS, at
  // least 16
  int chs = 8;
  auto lds_of = [&](int sh) {
    return (size_t)nfield * ((1 << sh) + BsVec<T>::PAD) * sizeof(T);
  };
  while (chs > 4 && lds_of(chs) > 72 * 1024) chs--;
  EXH_REQUIRE((size_t)nfield * 16 * sizeof(T) <= 96 * 1024, EXH_ERR_UNSUPPORTED,
              "bispectrum: %d shell fields exceed the LDS staging", nfield);
  {
    TimedScope ts(c, "bispec_products");
    const T* fields = (const T*)c->buf[BUF_SHELLS];
    const int lds = (int)lds_of(chs);
    EXH_CHECK_HIP(hipFuncSetAttribute((const void*)k_shell_products<T>,
                                      hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    const int ty = (njob + 4 * BS_JPW - 1) / (4 * BS_JPW);
    const int split = njob <= 1 ? 4 : (njob == 2 ? 2 : 1);
    const int per_wave = split > 1 ? 1 : (njob + 4 * ty - 1) / (4 * ty);
    const size_t nch = (ng + (1 << chs) - 1) >> chs;
    // three workgroups a CU, all resident (two: 0.68 ms; 513 workgroups, one
    // more than two a CU: 0.87 ms)
    const unsigned tx = (unsigned)std::max<size_t>(1, std::min<size_t>(nch, 768 / ty));
    hipLaunchKernelGGL(k_shell_products<T>, dim3(tx, ty), dim3(256), lds, c->stream, fields,
                       nfield, ng, chs, (const short2*)(tb + o_rows), (const short*)(tb + o_cols),
                       (const int4*)(tb + o_jobs), njob, per_wave, split, dout, drow);
    EXH_LAUNCH_CHECK();
  }
  std::vector<double> hs(nout), hks(Nk);
  std::vector<unsigned long long> hkc(Nk);
  EXH_CHECK_HIP(hipMemcpyAsync(hs.data(), dout, nout * 8, hipMemcpyDeviceToHost, c->stream));
  EXH_CHECK_HIP(hipMemcpyAsync(hks.data(), ksum, (size_t)Nk * 8, hipMemcpyDeviceToHost,
                               c->stream));
  EXH_CHECK_HIP(hipMemcpyAsync(hkc.data(), kcnt, (size_t)Nk * 8, hipMemcpyDeviceToHost,
                               c->stream));
  EXH_CHECK_HIP(hipStreamSynchronize(c->stream));
  const double* hrow = hs.data() + (size_t)njob * 256;
  auto triple = [&](int r, int q) {
    return hs[(size_t)tile[(size_t)(r / 16) * ntc + q / 16] * 256 + (r % 16) * 16 + q % 16];
  };
  // 4. normalisation (bimodule.c:356-370) and outputs in T (spectrum.c:368-383)
  std::vector<double> km(Nk);
  for (int s = 0; s < Nk; s++) km[s] = (double)(T)(hkc[s] ? hks[s] / (double)hkc[s] : NAN);
  const double L15 = std::pow((double)Lr, 1.5);
  for (long long n = 0; n < ntri; n++) {
    const auto& t = tri[n];
    const int p = pid[(size_t)t[0] * Nk + t[1]];
    const double IB = triple(irow + p, icol + t[2]);
    for (int j = 0; j < NBs; j++) {
      const double v = triple(p * nt2 + j / ntype, (j % ntype) * Nk + t[2]);
      Bk[(size_t)j * ntri + n] = (double)(T)(v / IB * L15);
    }
    Ntri_out[n] = (double)(T)(IB / (double)ng);
    for (int q = 0; q < 3; q++) kB[(size_t)q * ntri + n] = km[t[q]];
  }
  for (int s = 0; s < Nk; s++) {
    const int p = pid[(size_t)s * Nk + s];
    const double IP = hrow[irow + p];
    int j = 0;
    for (int f1 = 0; f1 < ntype; f1++)
      for (int f2 = 0; f2 <= f1; f2++, j++)
        Pk[(size_t)j * Nk + s] = (double)(T)(hrow[p * nt2 + f1 * ntype + f2] / IP);
    Nk_out[s] = (double)(T)(IP / (double)ng);
    kP[s] = km[s];
  }
  return (int)ntri;
}

template int run_bispectrum<float>(exh_ctx*, const float*, int, int, double, int, double, int,
                                   int, double, double, long long, double*, double*, double*,
                                   double*, double*, double*);
template int run_bispectrum<double>(exh_ctx*, const double*, int, int, double, int, double, int,
                                    int, double, double, long long, double*, double*, double*,
                                    double*, double*, double*);

template void run_grid<float>(exh_ctx*, const float*, const float*, const float*, const int*,
                              long long, int, int, double, double, double, int, int, double,
                              double, int, int, float*, void*);
template void run_grid<double>(exh_ctx*, const double*, const double*, const double*, const int*,
                               long long, int, int, double, double, double, int, int, double,
                               double, int, int, double*, void*);
template void run_power<float>(exh_ctx*, const float*, int, int, double, int, double, int, int,
                               double, double, int, int, int, double*, double*, long long*, bool);
template void run_power<double>(exh_ctx*, const double*, int, int, double, int, double, int, int,
                                double, double, int, int, int, double*, double*, long long*,
                                bool);

}  // namespace exh
