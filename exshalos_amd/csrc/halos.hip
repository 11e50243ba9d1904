// Excursion-set halo finder on the GPU (find_halos.c:96-476).
//
// 1. peaks: strict 6-neighbour periodic maxima, compacted in lexicographic
//    cell order (find_halos.c:96-156);
// 2. Lomuto quicksort emulation (sort.hip), exact tie order;
// 3. greedy spherical growth in deterministic rounds.  The reference visits
//    peaks from the densest down and each growth sees the flags of all
//    denser halos (find_halos.c:226-379).  Every round, each pending
//    candidate grows speculatively against the flags committed so far
//    (thread per candidate, the reference's exact double-precision sum
//    order) and claims the cells it could write (r^2 < G, G = first failing
//    shell; more flags can only stop the growth earlier, so the final halo
//    lies inside that ball).  A candidate of one cell (G = 1) claims nothing:
//    its centre's flag names its rank.  A candidate whose read ball
//    (r^2 <= G) holds no claim and no centre of a denser pending candidate
//    has seen its final flags: it commits.  The densest pending candidate
//    always commits, so the rounds terminate; the result equals the
//    sequential loop.
// 4. masses: taus uniforms by GF(2) jump-ahead, Tinker-integral splines
//    (find_halos.c:442-476);
// 5. halo positions from the displacement field (lpt.c:70-74, 245-255).
#include "common.hpp"
#include "kernels.hpp"
#include "util.hpp"

#include <algorithm>

namespace exh {

// Flags of the cells during the rounds: free, inside a rejected sphere, the
// free centre of the pending candidate of rank r (FLAG_PENDING - r), or >= 0
// in a halo.
static constexpr int FLAG_FREE = -1;
static constexpr int FLAG_REJECTED = -2;
static constexpr int FLAG_PENDING = -3;
static constexpr int S_TAB_MAX = 1024;  // largest r^2 a halo may reach
static constexpr int BALL_MAX = 65;     // largest ball whose cells are tabled in memory order

// x in [-n, 2n) wrapped into [0, n): of x, x + n and x - n the one that is
// in range is the smallest as unsigned.
__device__ __forceinline__ unsigned wrap_u(int x, int n) {
  return min(min((unsigned)x, (unsigned)(x + n)), (unsigned)(x - n));
}

// Cell at packed offset p from (ci, cj, ck), periodic; cells are below 2^30.
__device__ __forceinline__ unsigned cell_off(int ci, int cj, int ck, unsigned p, int n0, int n1,
                                             int n2) {
  const int di = (int)(p & 255u) - 128, dj = (int)((p >> 8) & 255u) - 128,
            dk = (int)((p >> 16) & 255u) - 128;
  return (wrap_u(ci + di, n0) * (unsigned)n1 + wrap_u(cj + dj, n1)) * (unsigned)n2 +
         wrap_u(ck + dk, n2);
}

// ---------------------------------------------------------------------------
// peaks
// ---------------------------------------------------------------------------
// Cells are below 2^30 here, so indices and offsets are 32-bit.  A thread
// tests the cells c0 + q * 256 (q < PK_ITEMS) of its block's tile: the
// coordinates of the first come from two multiply-high divisions, the
// others by stepping, and the six neighbours from offsets with the
// periodic wrap as a select.  Every neighbour is loaded (no short-circuit),
// so the loads of a thread's cells are all in flight together.
static constexpr int PK_ITEMS = 8;
static constexpr int PK_TILE = 256 * PK_ITEMS;

struct PeakGeom {
  int n0, n1, n2;
  unsigned sx, sy;  // plane and row strides
  FastDiv dz, dy;
};

template <typename T>
__device__ inline bool is_peak_at(const T* d, unsigned c, T v, int i, int j, int k,
                                  const PeakGeom& g) {
  const unsigned xp = i == g.n0 - 1 ? c - (unsigned)(g.n0 - 1) * g.sx : c + g.sx;
  const unsigned xm = i == 0 ? c + (unsigned)(g.n0 - 1) * g.sx : c - g.sx;
  const unsigned yp = j == g.n1 - 1 ? c - (unsigned)(g.n1 - 1) * g.sy : c + g.sy;
  const unsigned ym = j == 0 ? c + (unsigned)(g.n1 - 1) * g.sy : c - g.sy;
  const unsigned zp = k == g.n2 - 1 ? c - (unsigned)(g.n2 - 1) : c + 1;
  const unsigned zm = k == 0 ? c + (unsigned)(g.n2 - 1) : c - 1;
  const T a = d[xp], b = d[xm], e = d[yp], f = d[ym], h = d[zp], l = d[zm];
  return (v > a) & (v > b) & (v > e) & (v > f) & (v > h) & (v > l);
}

// Peak flags of the thread's PK_ITEMS cells (cells past the grid: false), and
// in the second byte those of its peaks below Bmin.  The pass also copies
// those cells of delta to eff, the growth rounds' effective density.
template <typename T>
__device__ inline unsigned peak_bits(const T* d, unsigned c0, unsigned ng, const PeakGeom& g,
                                     T Bmin, T* eff) {
  unsigned r = fdiv(c0, g.dz);
  int k = (int)(c0 - r * (unsigned)g.n2);
  int i = (int)fdiv(r, g.dy);
  int j = (int)(r - (unsigned)i * (unsigned)g.n1);
  unsigned bits = 0;
  T cv[PK_ITEMS];
#pragma unroll
  for (int q = 0; q < PK_ITEMS; q++) {
    const unsigned c = c0 + (unsigned)q * 256u;
    cv[q] = 0;
    if (c < ng) {
      cv[q] = d[c];
      if (is_peak_at(d, c, cv[q], i, j, k, g)) bits |= (cv[q] < Bmin ? 0x101u : 1u) << q;
    }
    k += 256;
    while (k >= g.n2) {
      k -= g.n2;
      if (++j == g.n1) {
        j = 0;
        ++i;
      }
    }
  }
  // stores after every load, so that no load waits behind a store
#pragma unroll
  for (int q = 0; q < PK_ITEMS; q++) {
    const unsigned c = c0 + (unsigned)q * 256u;
    if (c < ng) eff[c] = cv[q];
  }
  return bits;
}

// Peaks are found over tiles of PK_TILE consecutive cells; thread x of a
// block tests cells tile + q * 256 + x (q < PK_ITEMS), so every load row is
// coalesced.  The write pass ranks peaks in cell order from per-row wave
// ballots, which keeps the reference's lexicographic peak order.
// The count pass keeps each thread's PK_ITEMS peak flags as one byte
// (ng / 8 bytes), so the write pass reads them instead of testing the
// neighbours again.  A block's count of peaks and, above bit 32, of those
// below the smallest barrier, which are never visited (their number is the
// first visited sorted position), go through one scan; added up with one
// atomic per block of the write pass, all at one address, the latter took it
// from 265 to 809 us at 512^3.
static constexpr int LOW_SHIFT = 32;
template <typename T>
__global__ __launch_bounds__(256) void k_peak_count(const T* d, PeakGeom g, T Bmin,
                                                    long long* bcnt, T* eff,
                                                    unsigned char* pbits) {
  static_assert(PK_ITEMS == 8, "one byte of peak flags per thread");
  __shared__ long long sh[4];
  const unsigned ng = (unsigned)g.n0 * g.sx;
  const unsigned base = blockIdx.x * (unsigned)PK_TILE + threadIdx.x;
  const unsigned bits = peak_bits(d, base, ng, g, Bmin, eff);
  pbits[blockIdx.x * 256u + threadIdx.x] = (unsigned char)bits;
  // both counts of a wave in one int (at most 512 each)
  int cnt = __popc(bits & 0xffu) + (__popc(bits >> 8) << 16);
  for (int o = 32; o > 0; o >>= 1) cnt += __shfl_xor(cnt, o, 64);
  if ((threadIdx.x & 63) == 0)
    sh[threadIdx.x >> 6] = (long long)(cnt & 0xffff) | ((long long)(cnt >> 16) << LOW_SHIFT);
  __syncthreads();
  if (threadIdx.x == 0) bcnt[blockIdx.x] = sh[0] + sh[1] + sh[2] + sh[3];
}

template <typename T>
__global__ __launch_bounds__(256) void k_peak_write(const T* d, PeakGeom g, const long long* boff,
                                                    const unsigned char* pbits, T* key, int* cell,
                                                    int* flag) {
  __shared__ int wcnt[PK_ITEMS][4];
  const unsigned ng = (unsigned)g.n0 * g.sx;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const unsigned base = blockIdx.x * (unsigned)PK_TILE + threadIdx.x;
  const unsigned bits = pbits[blockIdx.x * 256u + threadIdx.x];
  // the peaks' densities, loaded before the first store (which could alias
  // them for the compiler)
  T dv[PK_ITEMS];
#pragma unroll
  for (int q = 0; q < PK_ITEMS; q++)
    dv[q] = (bits >> q) & 1u ? d[base + (unsigned)q * 256u] : (T)0;
#pragma unroll
  for (int q = 0; q < PK_ITEMS; q++) {
    const unsigned c = base + (unsigned)q * 256u;
    if (c < ng) flag[c] = FLAG_FREE;
  }
  unsigned long long bal[PK_ITEMS];
#pragma unroll
  for (int q = 0; q < PK_ITEMS; q++) {
    bal[q] = __ballot((bits >> q) & 1u);
    if (lane == 0) wcnt[q][w] = __popcll(bal[q]);
  }
  __syncthreads();
  long long o = boff[blockIdx.x] & ((1LL << LOW_SHIFT) - 1);
  const unsigned long long below = lanemask_lt();
  for (int q = 0; q < PK_ITEMS; q++) {
    long long ow = o;
    for (int u = 0; u < w; u++) ow += wcnt[q][u];
    if ((bal[q] >> lane) & 1ull) {
      const long long at = ow + __popcll(bal[q] & below);
      const unsigned c = base + (unsigned)q * 256u;
      key[at] = dv[q];
      cell[at] = (int)c;
    }
    o += wcnt[q][0] + wcnt[q][1] + wcnt[q][2] + wcnt[q][3];
  }
}

// Candidates: the peaks with density >= the smallest barrier, except the one
// at sorted position 0, which the reference does not visit.  Rank r (0 =
// densest) is sorted position np - 1 - r; perm gives each position's peak.
// Writes each candidate's rank by peak.
static constexpr int RT_RING = 16;   // device ring of per-round pending counts
static constexpr int RT_BATCH = 4;   // rounds per host read after the first
static constexpr int NXCD = 8;       // accelerator dies: lists of pending candidates

__global__ __launch_bounds__(256) void k_cand_ranks(const int* perm, int np, int below, int* rank,
                                                    int* rt) {
  if (blockIdx.x == 0 && threadIdx.x <= 2 * NXCD)  // the first two rounds' counts, the error flag
    rt[threadIdx.x < 2 * NXCD ? threadIdx.x : RT_RING * NXCD] = 0;
  const int l0 = below + (int)blockIdx.x * 1024 + (int)threadIdx.x;
  int p[4];
#pragma unroll
  for (int q = 0; q < 4; q++) p[q] = l0 + 256 * q < np ? perm[l0 + 256 * q] : -1;
#pragma unroll
  for (int q = 0; q < 4; q++)
    if (p[q] >= 0) rank[p[q]] = np - 1 - (l0 + 256 * q);
}

// The first round's lists: the candidates in the order of their cells, list
// x the x-th eighth of the blocks of PK_TILE peaks.  Neighbours in the list
// are neighbours in memory, and dense candidates (long growths) are spread
// over the workgroups.  (Lists by bricks of 16 x 16 columns and density gave
// a wave growths of similar length, but workgroups of long ones only: the
// first round of a 256^3 grid of 2 Mpc/h cells took 2.3 ms with them.)
// Clears the results by peak and flags the candidates' centres as pending.
template <typename T>
__global__ __launch_bounds__(256) void k_list_build(const T* key, const int* cell,
                                                    const int* rank, int np, int nc, T Bmin,
                                                    int cap, int* rt, int* prank, int* ppeak,
                                                    unsigned short* res, int* flag) {
  __shared__ int wcnt[PK_ITEMS][4];
  __shared__ int s_base;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int p0 = (int)blockIdx.x * PK_TILE + (int)threadIdx.x;
  int r[PK_ITEMS], c[PK_ITEMS];
#pragma unroll
  for (int q = 0; q < PK_ITEMS; q++) {
    const int p = p0 + 256 * q;
    c[q] = p < np ? cell[p] : 0;
    r[q] = p < np && key[p] >= Bmin ? rank[p] : nc;
  }
#pragma unroll
  for (int q = 0; q < PK_ITEMS; q++) {
    if (p0 + 256 * q < np) res[p0 + 256 * q] = 0;
    if (r[q] < nc) flag[c[q]] = FLAG_PENDING - r[q];
  }
  unsigned long long bal[PK_ITEMS];
#pragma unroll
  for (int q = 0; q < PK_ITEMS; q++) {
    bal[q] = __ballot(r[q] < nc);
    if (lane == 0) wcnt[q][w] = __popcll(bal[q]);
  }
  __syncthreads();
  const int x = (int)((long long)blockIdx.x * NXCD / gridDim.x);
  if (threadIdx.x == 0) {
    int tot = 0;
    for (int q = 0; q < PK_ITEMS; q++) tot += wcnt[q][0] + wcnt[q][1] + wcnt[q][2] + wcnt[q][3];
    s_base = atomicAdd(&rt[x], tot);
  }
  __syncthreads();
  int o = x * cap + s_base;
#pragma unroll
  for (int q = 0; q < PK_ITEMS; q++) {
    int ow = o;
    for (int u = 0; u < w; u++) ow += wcnt[q][u];
    if (r[q] < nc) {
      const int at = ow + __popcll(bal[q] & lanemask_lt());
      prank[at] = r[q];
      ppeak[at] = p0 + 256 * q;
    }
    o += wcnt[q][0] + wcnt[q][1] + wcnt[q][2] + wcnt[q][3];
  }
}

__global__ void k_fill_u64(unsigned long long* p, long long n, unsigned long long v) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x)
    p[i] = v;
}

// ---------------------------------------------------------------------------
// growth rounds
// ---------------------------------------------------------------------------
static constexpr int PRES_BLOCKED = 1 << 30;

template <typename T>
struct GrowArgs {
  int n0, n1, n2;
  const T* delta;
  T* eff;          // delta, or -Mtot where a halo (or a rejected sphere) has flagged the cell
  int* flag;
  unsigned long long* claim;
  ShellTab sh;
  const T* Bt;
  int nB;
  T Bmin;
  T negMtot;
  int Nmin;
  // cell and density by peak
  const int* pcell;
  const T* pkey;
  // the round's candidates by list position: rank (0 = densest), peak, and
  // the growth result handed from k_grow to k_commit: (G << 16 | R2), G the
  // first failing shell (read radius^2) and R2 the final halo's shells (its
  // cells are those of r^2 < R2, start[R2] of them), PRES_BLOCKED where the
  // centre of a denser pending candidate lies in the read ball; -1 = skipped
  const int* prank;
  const int* ppeak;
  int* pres;
  unsigned short* res;  // final result by peak: R2, or 0 (no halo)
  int* err;
};

template <typename T>
__device__ inline void decode_cell(int cell, int n1, int n2, int& i, int& j, int& k) {
  k = cell % n2;
  int r = cell / n2;
  j = r % n1;
  i = r / n1;
}

// A round's pending candidates stand in NXCD lists, list x at positions
// [x cap, x cap + n_x) of the arrays by list position, with its count n_x on
// the device.  Workgroup w, which runs on XCD w mod 8, takes CPB consecutive
// candidates of list w mod 8: consecutive candidates (neighbours in space)
// share one L2, and a candidate that must retry stays in its XCD's list, so
// the next round keeps that.  The grid may be larger than the lists (sized by
// an earlier round's counts); its extra blocks return.
struct RoundLists {
  const int* n;   // [NXCD] this round's counts
  int* next;      // [NXCD] the next round's (zero on entry; k_commit adds)
  int* clear;     // [NXCD] the round's after that, zeroed by k_grow
  int cap;
  int *rank_out, *peak_out;  // the next round's lists
};

// A table that no kernel of the rounds writes, read through the scalar cache
// where the index is uniform.
__device__ __forceinline__ int table_at(const int* p, int i) {
  return ((const int __attribute__((address_space(4)))*)(uintptr_t)p)[i];
}

// Value of lane E of the lane's row of 16 (row_newbcast).
template <int E>
__device__ __forceinline__ float row_lane(float v) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + E, 0xf, 0xf, true));
}
template <int E>
__device__ __forceinline__ double row_lane(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x150 + E, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x150 + E, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// s += v of lanes 0 .. nb - 1 of the row, in lane order (nb the same in the
// whole wave).  The lanes past nb hold zeros, which leave s unchanged, so
// four lanes are added at a time: one branch per four cells.
template <int E, typename T>
__device__ __forceinline__ void row_add(double& s, T v, int nb) {
  if constexpr (E < 16) {
    if (nb > E) {
      s += (double)row_lane<E>(v);
      s += (double)row_lane<E + 1>(v);
      s += (double)row_lane<E + 2>(v);
      s += (double)row_lane<E + 3>(v);
      row_add<E + 4>(s, v, nb);
    }
  }
}
// s -= v of the row's lanes, in lane order, zeros past the last cell.
template <int E, typename T>
__device__ __forceinline__ void row_sub(double& s, T v) {
  if constexpr (E < 16) {
    s -= (double)row_lane<E>(v);
    row_sub<E + 1>(s, v);
  }
}

// A row's centre and where its ball may wrap: with FLAT, cells within
// sqrt(flat) of the centre need no wrap in i and j.
struct Centre {
  int i, j, k, ij;  // ij: the cell (i, j, 0)
  int flat;
};

template <typename T>
__device__ __forceinline__ Centre centre_of(const GrowArgs<T>& a, int i, int j, int k) {
  Centre c;
  c.i = i;
  c.j = j;
  c.k = k;
  c.ij = (i * a.n1 + j) * a.n2;
  const int d = min(min(i, a.n0 - 1 - i), min(j, a.n1 - 1 - j));
  c.flat = d * d;
  return c;
}

// The offsets of the first SH_LDS cells of the shell table, in LDS (a load
// of theirs from memory would wait behind the loads of values in flight):
// x = di n1 n2 + dj n2, y = the packed offset.
static constexpr unsigned CENTRE_OFF = 0x808080u;  // packed offset (0, 0, 0)
static constexpr int SH_LDS = 1024;
static constexpr int ST_LDS = 256;  // shells whose starts are in LDS

__device__ __forceinline__ unsigned table_cell(const int2& t, bool flat, const Centre& c, int n0,
                                               int n1, int n2) {
  if (flat)
    return (unsigned)(c.ij + t.x) + wrap_u(c.k + (int)(((unsigned)t.y >> 16) & 255u) - 128, n2);
  return cell_off(c.i, c.j, c.k, (unsigned)t.y, n0, n1, n2);
}

// The row's values of f at cells [o, min(o + 64, o1)) of the shell table,
// 16 cells in each v[k], in lane order and zeros past o1.
static constexpr int ROW_K = 4;
template <typename T>
__device__ __forceinline__ void row_load(T (&v)[ROW_K], const T* f, const int2* tab,
                                         const GrowArgs<T>& a, int o, int o1, int lane, bool flat,
                                         const Centre& c) {
#pragma unroll
  for (int k = 0; k < ROW_K; k++) {
    if (o + 16 * k >= o1) break;
    const int e = o + 16 * k + lane;
    v[k] = 0;
    if (e < o1) {
      unsigned id;
      if (o1 <= SH_LDS)
        id = table_cell(tab[e], flat, c, a.n0, a.n1, a.n2);
      else
        id = cell_off(c.i, c.j, c.k, a.sh.offs[e], a.n0, a.n1, a.n2);
      v[k] = f[id];
    }
  }
}

// Claims are 64-bit (round tag << 32 | ~rank) or, with fewer than 2^24
// candidates, 32-bit (round tag << 24 | (2^24 - 1 - rank)): atomicMax keeps
// the densest claim of the current round, and any claim of the round beats
// those of earlier rounds.
template <bool C32>
__device__ __forceinline__ void claim_cell(unsigned long long* claim, unsigned id,
                                           unsigned long long tag_hi, int rank) {
  if constexpr (C32)
    atomicMax(reinterpret_cast<unsigned*>(claim) + id,
              (unsigned)tag_hi | (0xffffffu - (unsigned)rank));
  else
    atomicMax(claim + id, tag_hi | (unsigned long long)(0xffffffffu - (unsigned)rank));
}

// Whether a denser candidate has claimed cell id in this round.
template <bool C32>
__device__ __forceinline__ bool claimed(const unsigned long long* claim, unsigned id,
                                        unsigned long long tag_hi, int rank) {
  if constexpr (C32) {
    const unsigned v = reinterpret_cast<const unsigned*>(claim)[id];
    return (v & 0xff000000u) == (unsigned)tag_hi && (v & 0xffffffu) > 0xffffffu - (unsigned)rank;
  } else {
    const unsigned long long v = claim[id];
    return (v & 0xffffffff00000000ull) == tag_hi &&
           (unsigned)(v & 0xffffffffu) > 0xffffffffu - (unsigned)rank;
  }
}

// Growth of the round's candidates (find_halos.c:226-379), in two phases.
//
// One thread per candidate tests the flag and the first shell (6 cells).
// Most candidates end there (81% of a 512^3 box's halos of 4 Mpc/h cells are
// one cell); they claim nothing.  With 256 candidates a workgroup the
// threads go on to the next shells while at least GROW_MIN of them grow: a
// shell of n cells costs a wave about 20 n vector instructions for all of its
// candidates, and a row (below) about 4 n for one.
//
// The others go to a list in LDS, from which each wave takes four at a time,
// one per row of 16 lanes: the row loads a shell's cells in parallel, two
// shells ahead of the sum, and every lane forms the reference's ordered
// double sum from the row's values (row_newbcast moves).  A growth of n cells
// then waits for about one load per shell and not for one per 8 cells, and a
// wave is held by the longest of four growths and not of 64.  What bounds
// the kernel is vector issue in large boxes and that chain of loads and
// ordered additions in small ones.
static constexpr int GROW_MIN = 56;
// Last shell of the threads.  The smallest table (sides of at least 4: 14
// shells) holds their starts and those that the rows read ahead.
static constexpr int GROW_SHELLS = 9;

template <typename T, bool C32, int CPB>
__global__ __launch_bounds__(256) void k_grow(GrowArgs<T> a, RoundLists rl,
                                              unsigned long long tag_hi) {
  __shared__ double s_mean[CPB];
  __shared__ int s_i[CPB], s_j[CPB], s_k[CPB], s_rank[CPB];
  __shared__ short s_at[CPB], s_G[CPB];
  __shared__ int2 s_tab[SH_LDS];
  __shared__ int s_start[ST_LDS];
  __shared__ int nlist, taken;
  const int x = blockIdx.x % NXCD, t0 = (int)(blockIdx.x / NXCD) * CPB;
  if (blockIdx.x < NXCD && threadIdx.x == 0) rl.clear[blockIdx.x] = 0;
  const int n = rl.n[x];
  if (t0 >= n) return;
  const int base = x * rl.cap + t0, m = min(CPB, n - t0);
  const int* start = a.sh.start;
  if (threadIdx.x == 0) {
    nlist = 0;
    taken = 0;
  }
  const int noffs = table_at(start, a.sh.stab);
#pragma unroll
  for (int q = 0; q < SH_LDS / 256; q++) {
    const int e = (int)threadIdx.x + 256 * q;
    const unsigned p = e < noffs ? a.sh.offs[e] : 0u;
    const int di = (int)(p & 255u) - 128, dj = (int)((p >> 8) & 255u) - 128;
    s_tab[e] = make_int2((di * a.n1 + dj) * a.n2, (int)p);
  }
  s_start[threadIdx.x] = start[min((int)threadIdx.x, a.sh.stab)];
  __syncthreads();
  const double Bmin = (double)a.Bmin;
  const int lane = threadIdx.x & 63;
  int s = 1;
  if (threadIdx.x < CPB) {
    const int t = base + threadIdx.x;
    bool mine = false, more;
    double den = 0, mean = 0;
    int rank = 0, cell = 0, G = 0;
    Centre c = {0, 0, 0, 0, 0};
    if ((int)threadIdx.x < m) {
      rank = a.prank[t];
      const int p = a.ppeak[t];
      cell = a.pcell[p];
      mean = (double)a.pkey[p];
      mine = a.flag[cell] <= FLAG_PENDING;
      if (!mine) a.pres[t] = -1;  // already inside a denser halo
      int i, j, k;
      decode_cell<T>(cell, a.n1, a.n2, i, j, k);
      c = centre_of(a, i, j, k);
    }
    more = mine;
    const bool flat = __ballot(mine && c.flat < GROW_SHELLS) == 0;
    // cell e of the table around the thread's candidate
    auto at = [&](int e) {
      const unsigned p = (unsigned)table_at((const int*)a.sh.offs, e);
      if (!flat) return cell_off(c.i, c.j, c.k, p, a.n0, a.n1, a.n2);
      const int di = (int)(p & 255u) - 128, dj = (int)((p >> 8) & 255u) - 128;
      return (unsigned)(c.ij + (di * a.n1 + dj) * a.n2) +
             wrap_u(c.k + (int)((p >> 16) & 255u) - 128, a.n2);
    };
    for (;;) {
      const int o0 = table_at(start, s), o1 = table_at(start, s + 1);
      if (more) {
        // the shell's cells in cube order; loads issued in batches, summed
        // in order (flagged cells hold -Mtot in eff, as the reference adds)
        double sum = mean * (double)o0;
        for (int ob = o0; ob < o1; ob += 6) {
          T v[6];
#pragma unroll
          for (int e = 0; e < 6; e++)
            if (ob + e < o1) v[e] = a.eff[at(ob + e)];
#pragma unroll
          for (int e = 0; e < 6; e++)
            if (ob + e < o1) sum += (double)v[e];
        }
        sum = sum / (double)o1;
        den = mean;
        mean = sum;
        if (!(mean >= Bmin)) {
          more = false;
          G = s;
        }
      }
      s++;
      if (CPB < 256 || s > GROW_SHELLS) break;
      if (__builtin_amdgcn_readfirstlane(__syncthreads_count(more)) < GROW_MIN) break;
    }
    // grown out at one cell, which shrinks to none below its barrier; the
    // others are left to a row
    const bool row = more || G > 1;
    if (G == 1) a.pres[t] = 1 << 16 | (den < (double)a.Bt[1] ? 0 : 1);
    const unsigned long long bal = __ballot(row);
    int o = 0;
    if (bal && lane == 0) o = atomicAdd(&nlist, __popcll(bal));
    o = __shfl(o, 0, 64) + __popcll(bal & lanemask_lt());
    if (row) {
      s_mean[o] = more ? mean : den;
      s_G[o] = (short)G;
      s_i[o] = c.i;
      s_j[o] = c.j;
      s_k[o] = c.k;
      s_rank[o] = rank;
      s_at[o] = (short)threadIdx.x;
    }
  }
  __syncthreads();
  s = CPB < 256 ? 2 : __builtin_amdgcn_readfirstlane(s);  // the first shell of the rows
  const int nl = nlist, l16 = lane & 15, row = lane >> 4;
  for (;;) {
    int q = 0;
    if (lane == 0) q = atomicAdd(&taken, 4);
    q = __builtin_amdgcn_readfirstlane(q);
    if (q >= nl) break;
    const bool has = q + row < nl;
    const int it = has ? q + row : q;  // an idle row follows the first one
    const int rank = s_rank[it];
    const Centre c = centre_of(a, s_i[it], s_j[it], s_k[it]);
    // the rows that are to grow, from shell s on; count = start[sh] cells lie
    // inside shell sh
    int G = s_G[it];
    double den = s_mean[it], mean = den;
    bool act = has && G == 0;
    if (G == 0) G = -1;
    T va[ROW_K], vb[ROW_K], vc[ROW_K];
    if (__ballot(act)) {
      int fl = min(c.flat, __shfl_xor(c.flat, 16, 64));
      fl = __builtin_amdgcn_readfirstlane(min(fl, __shfl_xor(fl, 32, 64)));
      int o0 = table_at(start, s), o1 = table_at(start, s + 1), o2 = table_at(start, s + 2),
          o3 = table_at(start, s + 3);
      row_load(va, a.eff, s_tab, a, o0, o1, l16, s <= fl, c);
      row_load(vb, a.eff, s_tab, a, o1, o2, l16, s + 1 <= fl, c);
      for (int sh = s;; sh++) {
        if (sh >= a.sh.stab) {  // rows still growing leave the table
          if (act) atomicOr(a.err, 1);
          break;
        }
        const int o4 = sh + 3 < a.sh.stab ? table_at(start, sh + 4) : o3;
        row_load(vc, a.eff, s_tab, a, o2, o3, l16, sh + 2 <= fl, c);
        double sum = mean * (double)o0;
#pragma unroll
        for (int k = 0; k < ROW_K; k++)
          if (o0 + 16 * k < o1) row_add<0>(sum, va[k], o1 - o0 - 16 * k);
        for (int o = o0 + 16 * ROW_K; o < o1; o += 16 * ROW_K) {
          row_load(va, a.eff, s_tab, a, o, o1, l16, sh <= fl, c);
#pragma unroll
          for (int k = 0; k < ROW_K; k++)
            if (o + 16 * k < o1) row_add<0>(sum, va[k], o1 - o - 16 * k);
        }
        sum = sum / (double)o1;
        if (act) {
          den = mean;
          mean = sum;
          if (!(mean >= Bmin)) {
            act = false;
            G = sh;
          }
        }
        if (!__ballot(act)) break;
#pragma unroll
        for (int k = 0; k < ROW_K; k++) {
          va[k] = vb[k];
          vb[k] = vc[k];
        }
        o0 = o1;
        o1 = o2;
        o2 = o3;
        o3 = o4;
      }
    }
    const int t = base + s_at[it];
    if (has && G >= 0) {  // a row with a result: shrink it below the barrier
      auto start_of = [&](int sh) { return sh < ST_LDS ? s_start[sh] : start[sh]; };
      int grows = G - 1, grows_tmp = G, count = start_of(G);
      while (start_of(grows + 1) == start_of(grows)) grows--;  // the last shell with cells
      if (count >= a.nB) {
        if (l16 == 0) atomicOr(a.err, 2);
        G = -1;
      } else if (den < (double)a.Bt[count]) {
        // shells come off from the outside in; each one's values and the
        // barrier of the cells left are loaded one shell ahead
        int c1 = start_of(grows + 1), c0 = start_of(grows);
        T bt = a.Bt[c0];
        row_load(va, a.delta, s_tab, a, c0, c1, l16, grows <= c.flat, c);
        for (;;) {
          const int cn = grows > 0 ? start_of(grows - 1) : 0;
          T btn = 0;
          if (grows > 0) {
            btn = a.Bt[cn];
            row_load(vb, a.delta, s_tab, a, cn, c0, l16, grows <= c.flat, c);
          }
          den = den * (double)count;
#pragma unroll
          for (int k = 0; k < ROW_K; k++)
            if (c0 + 16 * k < c1) row_sub<0>(den, va[k]);
          for (int o = c0 + 16 * ROW_K; o < c1; o += 16 * ROW_K) {
            row_load(va, a.delta, s_tab, a, o, c1, l16, grows <= c.flat, c);
#pragma unroll
            for (int k = 0; k < ROW_K; k++)
              if (o + 16 * k < c1) row_sub<0>(den, va[k]);
          }
          count -= c1 - c0;
          if (count > 0) den = den / (double)count;
          if (c1 > c0) grows_tmp = grows;
          grows--;
          if (!(den < (double)bt && count > 0)) break;
          if (grows < 0) {  // cannot happen while count > 0 on an unclamped table
            if (l16 == 0) atomicOr(a.err, 32);
            G = -1;
            break;
          }
          bt = btn;
          c1 = c0;
          c0 = cn;
#pragma unroll
          for (int k = 0; k < ROW_K; k++) va[k] = vb[k];
        }
      }
      if (G >= 0) {
        // the read ball r^2 <= G: claim its cells of r^2 < G and look for the
        // centre of a denser pending candidate (flags change in k_commit
        // only, so every candidate sees those of the round's start).  In
        // memory order the atomics of a run along k share requests: global
        // atomics run at 26 G requests of 64 bytes a second, whatever they
        // touch.
        const bool tabled = G < a.sh.ball_max;
        const unsigned* offs = tabled ? a.sh.balls + a.sh.ball[G + 1] : a.sh.offs;
        const int rend = start_of(G + 1);
        bool hit = false;
        for (int ob = l16; ob < rend; ob += 64) {
          unsigned p[4];
          int f[4];
#pragma unroll
          for (int k = 0; k < 4; k++) p[k] = ob + 16 * k < rend ? offs[ob + 16 * k] : CENTRE_OFF;
#pragma unroll
          for (int k = 0; k < 4; k++) {
            const unsigned id = cell_off(c.i, c.j, c.k, p[k], a.n0, a.n1, a.n2);
            f[k] = a.flag[id];
            const int di = (int)(p[k] & 255u) - 128, dj = (int)((p[k] >> 8) & 255u) - 128,
                      dk = (int)((p[k] >> 16) & 255u) - 128;
            if (ob + 16 * k < rend && di * di + dj * dj + dk * dk < G)
              claim_cell<C32>(a.claim, id, tag_hi, rank);
          }
#pragma unroll
          for (int k = 0; k < 4; k++) hit |= f[k] <= FLAG_PENDING && FLAG_PENDING - f[k] < rank;
        }
        const bool blocked = ((__ballot(hit) >> (row * 16)) & 0xffffull) != 0;
        if (l16 == 0) a.pres[t] = G << 16 | grows_tmp | (blocked ? PRES_BLOCKED : 0);
      }
    }
    if (has && G < 0 && l16 == 0) a.pres[t] = -1;
  }
}

// Commit of the candidates that have seen their final flags: no denser
// pending candidate claims a cell of their read ball (r^2 <= G) or has its
// centre there (k_grow has looked for those; no two centres are neighbours,
// so a candidate of one cell has no other in its ball).  As in
// k_grow, one thread handles a candidate of one cell and a row of 16 lanes a
// larger one.  The others are appended to their XCD's list of the next round
// (in the order of the workgroups' atomics: the order of a list does not
// change the result), in place of a count, a scan and a write pass (12 us a
// round).  All rounds, against one thread per candidate and those passes: a
// 64^3 mock 283 -> 51 us, a 256^3 grid of 2 Mpc/h cells with an ellipsoidal
// barrier 2640 -> 430 us.
template <typename T, bool C32, int CPB>
__global__ __launch_bounds__(256) void k_commit(GrowArgs<T> a, RoundLists rl,
                                                unsigned long long tag_hi, int tmax) {
  __shared__ short s_at[CPB];
  __shared__ unsigned char s_retry[CPB];
  __shared__ int nlist, taken, s_wave[4], s_base;
  const int x = blockIdx.x % NXCD, t0 = (int)(blockIdx.x / NXCD) * CPB;
  const int n = rl.n[x];
  if (t0 >= n) return;
  const int base = x * rl.cap + t0, m = min(CPB, n - t0);
  if (threadIdx.x == 0) {
    nlist = 0;
    taken = 0;
  }
  __syncthreads();
  const int lane = threadIdx.x & 63;
  if (threadIdx.x < CPB) {
    const int t = base + threadIdx.x;
    bool more = false, retry = false;
    if ((int)threadIdx.x < m) {
      const int pr = a.pres[t], G = pr >> 16;  // -1: skipped or failed
      retry = pr > 0 && (pr & PRES_BLOCKED);
      more = G > 1 && !retry;
      if (G == 1) {
        const int rank = a.prank[t], p = a.ppeak[t], cell = a.pcell[p];
        int ci, cj, ck;
        decode_cell<T>(cell, a.n1, a.n2, ci, cj, ck);
#pragma unroll
        for (int e = 0; e < 7; e++)
          retry |= claimed<C32>(
              a.claim,
              cell_off(ci, cj, ck, (unsigned)table_at((const int*)a.sh.offs, e), a.n0, a.n1, a.n2),
              tag_hi, rank);
        if (!retry && (pr & 0xffff) == 0) a.flag[cell] = FLAG_FREE;  // no halo, pending no more
        if (!retry && (pr & 0xffff)) {
          const bool keep = 1 >= a.Nmin;
          a.flag[cell] = keep ? (rank << 1) | 1 : FLAG_REJECTED;
          a.eff[cell] = a.negMtot;
          if (keep) a.res[p] = 1;
        }
      }
    }
    const unsigned long long bal = __ballot(more);
    int at = 0;
    if (bal && lane == 0) at = atomicAdd(&nlist, __popcll(bal));
    at = __shfl(at, 0, 64) + __popcll(bal & lanemask_lt());
    if (more) s_at[at] = (short)threadIdx.x;
    s_retry[threadIdx.x] = retry;
  }
  __syncthreads();
  const int nl = nlist, l16 = lane & 15, row = lane >> 4;
  for (;;) {
    int q = 0;
    if (lane == 0) q = atomicAdd(&taken, 4);
    q = __builtin_amdgcn_readfirstlane(q);
    if (q >= nl) break;
    if (q + row >= nl) continue;
    const int at = s_at[q + row], t = base + at;
    const int rank = a.prank[t], p = a.ppeak[t], cell = a.pcell[p], pr = a.pres[t], G = pr >> 16;
    int ci, cj, ck;
    decode_cell<T>(cell, a.n1, a.n2, ci, cj, ck);
    const int oend = a.sh.start[G + 1];
    const unsigned* offs = G < a.sh.ball_max ? a.sh.balls + a.sh.ball[G + 1] : a.sh.offs;
    bool blocked = false;
    for (int ob = 0; ob < oend && !blocked; ob += 64) {
      unsigned off[4];
#pragma unroll
      for (int k = 0; k < 4; k++)
        off[k] = ob + 16 * k + l16 < oend ? offs[ob + 16 * k + l16] : CENTRE_OFF;
      bool hit = false;
#pragma unroll
      for (int k = 0; k < 4; k++)
        hit |= claimed<C32>(a.claim, cell_off(ci, cj, ck, off[k], a.n0, a.n1, a.n2), tag_hi, rank);
      blocked = ((__ballot(hit) >> (row * 16)) & 0xffffull) != 0;
    }
    if (blocked) {
      if (l16 == 0) s_retry[at] = 1;
      continue;
    }
    const int R2 = pr & 0xffff;
    if (R2 == 0) {  // shrunk to no cell: no halo, pending no more
      if (l16 == 0) a.flag[cell] = FLAG_FREE;
      continue;
    }
    if (isqrt_floor(R2 - 1) > tmax) {  // flag sphere would wrap (reference writes past its cube)
      if (l16 == 0) atomicOr(a.err, 4);
      continue;
    }
    const int fend = a.sh.start[R2];
    const bool keep = fend >= a.Nmin;
    const int v = keep ? (rank << 1) : FLAG_REJECTED;
    const unsigned* fo = R2 <= a.sh.ball_max ? a.sh.balls + a.sh.ball[R2] : a.sh.offs;
    for (int ob = l16; ob < fend; ob += 64) {
      unsigned off[4];
#pragma unroll
      for (int k = 0; k < 4; k++) off[k] = ob + 16 * k < fend ? fo[ob + 16 * k] : 0u;
#pragma unroll
      for (int k = 0; k < 4; k++)
        if (ob + 16 * k < fend) {
          const unsigned id = cell_off(ci, cj, ck, off[k], a.n0, a.n1, a.n2);
          a.flag[id] = keep && off[k] == CENTRE_OFF ? (rank << 1) | 1 : v;
          a.eff[id] = a.negMtot;
        }
    }
    if (keep && l16 == 0) a.res[p] = (unsigned short)R2;
  }
  __syncthreads();
  // the candidates to retry, in this block's order
  const bool retry = (int)threadIdx.x < m && s_retry[threadIdx.x % CPB] != 0;
  const unsigned long long bal = __ballot(retry);
  const int w = threadIdx.x >> 6;
  if (lane == 0) s_wave[w] = __popcll(bal);
  __syncthreads();
  if (threadIdx.x == 0) {
    const int tot = s_wave[0] + s_wave[1] + s_wave[2] + s_wave[3];
    s_base = tot ? atomicAdd(&rl.next[x], tot) : 0;
  }
  __syncthreads();
  if (retry) {
    int o = x * rl.cap + s_base + __popcll(bal & lanemask_lt());
    for (int u = 0; u < w; u++) o += s_wave[u];
    const int t = base + threadIdx.x;
    const int rank = a.prank[t], p = a.ppeak[t];
    rl.rank_out[o] = rank;
    rl.peak_out[o] = p;
  }
}

// ---------------------------------------------------------------------------
// catalogue, masses, flags, positions
// ---------------------------------------------------------------------------
// Halos in rank order: the results by rank and their counts per block of
// PK_TILE ranks, then (after the counts' scan) the halos and each rank's halo
// number.
__global__ __launch_bounds__(256) void k_halo_count(const unsigned short* res, const int* perm,
                                                    int np, int nc, unsigned short* rres,
                                                    long long* bcnt) {
  __shared__ int sh[4];
  const int r0 = (int)blockIdx.x * PK_TILE + (int)threadIdx.x;
  int p[PK_ITEMS], v[PK_ITEMS], cnt = 0;
#pragma unroll
  for (int q = 0; q < PK_ITEMS; q++) p[q] = r0 + 256 * q < nc ? perm[np - 1 - (r0 + 256 * q)] : -1;
#pragma unroll
  for (int q = 0; q < PK_ITEMS; q++) v[q] = p[q] >= 0 ? res[p[q]] : 0;
#pragma unroll
  for (int q = 0; q < PK_ITEMS; q++) {
    if (p[q] >= 0) rres[r0 + 256 * q] = (unsigned short)v[q];
    cnt += __popcll(__ballot(v[q] != 0));
  }
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = cnt;
  __syncthreads();
  if (threadIdx.x == 0) bcnt[blockIdx.x] = (long long)sh[0] + sh[1] + sh[2] + sh[3];
}

template <typename T>
__global__ __launch_bounds__(256) void k_gather_halos(const unsigned short* res,
                                                      const long long* boff, int nc,
                                                      const int* perm, const int* pcell, int np,
                                                      const int* start, int n1, int n2, int* hx,
                                                      int* hcount, int* hr2, int* hidx) {
  __shared__ int wcnt[PK_ITEMS][4];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int r0 = (int)blockIdx.x * PK_TILE + (int)threadIdx.x;
  int R2[PK_ITEMS], cell[PK_ITEMS];
  unsigned long long bal[PK_ITEMS];
#pragma unroll
  for (int q = 0; q < PK_ITEMS; q++) {
    const int r = r0 + 256 * q;
    R2[q] = r < nc ? res[r] : 0;
    cell[q] = R2[q] ? perm[np - 1 - r] : 0;
    bal[q] = __ballot(R2[q] != 0);
    if (lane == 0) wcnt[q][w] = __popcll(bal[q]);
  }
#pragma unroll
  for (int q = 0; q < PK_ITEMS; q++)
    if (R2[q]) cell[q] = pcell[cell[q]];
  __syncthreads();
  int o = (int)boff[blockIdx.x];
#pragma unroll
  for (int q = 0; q < PK_ITEMS; q++) {
    int ow = o;
    for (int u = 0; u < w; u++) ow += wcnt[q][u];
    const int h = ow + __popcll(bal[q] & lanemask_lt()), r = r0 + 256 * q;
    if (r < nc) hidx[r] = h;
    if (R2[q]) {
      int i, j, k;
      decode_cell<T>(cell[q], n1, n2, i, j, k);
      hx[3 * (size_t)h] = i;
      hx[3 * (size_t)h + 1] = j;
      hx[3 * (size_t)h + 2] = k;
      hcount[h] = start[R2[q]];
      hr2[h] = R2[q];
    }
    o += wcnt[q][0] + wcnt[q][1] + wcnt[q][2] + wcnt[q][3];
  }
}

// taus uniforms: thread b produces draws [b*64, b*64+64)
__global__ void k_taus(const unsigned* mats, unsigned s1, unsigned s2, unsigned s3, long long n,
                       double* u) {
  long long b = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  long long first = b * 64;
  if (first >= n) return;
  unsigned st[3] = {s1, s2, s3};
  for (int comp = 0; comp < 3; comp++) {
    const unsigned* M = mats + comp * 40 * 32;
    unsigned v = st[comp];
    for (int bit = 0; bit < 40; bit++) {
      if (!((first >> bit) & 1)) continue;
      unsigned r = 0;
      for (int col = 0; col < 32; col++)
        if ((v >> col) & 1u) r ^= M[bit * 32 + col];
      v = r;
    }
    st[comp] = v;
  }
  for (int q = 0; q < 64 && first + q < n; q++) {
    unsigned b1 = ((st[0] << 13) ^ st[0]) >> 19;
    st[0] = ((st[0] & 4294967294u) << 12) ^ b1;
    unsigned b2 = ((st[1] << 2) ^ st[1]) >> 25;
    st[1] = ((st[1] & 4294967288u) << 4) ^ b2;
    unsigned b3 = ((st[2] << 3) ^ st[2]) >> 11;
    st[2] = ((st[2] & 4294967280u) << 17) ^ b3;
    u[first + q] = (double)(st[0] ^ st[1] ^ st[2]) / 4294967296.0;
  }
}

__device__ inline double spline_eval_d(const double* x, const double* y, const double* m, int n,
                                       double xv, int* bad) {
  if (xv < x[0] || xv > x[n - 1]) {
    *bad = 1;
    xv = xv < x[0] ? x[0] : x[n - 1];
  }
  int lo = 0, hi = n - 1;
  while (hi - lo > 1) {
    int mid = (lo + hi) >> 1;
    if (x[mid] > xv)
      hi = mid;
    else
      lo = mid;
  }
  double h = x[hi] - x[lo];
  double t = xv - x[lo];
  double b = (y[hi] - y[lo]) / h - h * (2.0 * m[lo] + m[hi]) / 6.0;
  double c = m[lo] / 2.0;
  double d = (m[hi] - m[lo]) / (6.0 * h);
  return y[lo] + t * (b + t * (c + t * d));
}

// Mh = InvI(I(M_count) + (I(M_next) - I(M_count)) u)   (find_halos.c:455-476)
template <typename T>
__global__ void k_masses(const int* hcount, long long nh, const int* sphere, int nsph,
                         int Ncells, const double* itab, const int* ibad, const double* Mk,
                         const double* Int, const double* mInv, int Nr, const double* u, T* Mh,
                         int* err) {
  for (long long h = blockIdx.x * (long long)blockDim.x + threadIdx.x; h < nh;
       h += (long long)gridDim.x * blockDim.x) {
    int cnt = hcount[h];
    // first index with sphere[i] == cnt among the first Ncells entries
    int lo = 0, hi = (Ncells < nsph ? Ncells : nsph);
    while (lo < hi) {
      int mid = (lo + hi) >> 1;
      if (sphere[mid] < cnt)
        lo = mid + 1;
      else
        hi = mid;
    }
    int bad = 0;
    if (lo >= (Ncells < nsph ? Ncells : nsph) || sphere[lo] != cnt || lo + 1 >= nsph) {
      atomicOr(err, 8);
      Mh[h] = (T)0;
      continue;
    }
    // I of the masses of spheres lo and lo + 1, from the table
    const double I0 = itab[lo];
    T v = (T)(I0 + (itab[lo + 1] - I0) * u[h]);
    bad = ibad[lo] | ibad[lo + 1];
    Mh[h] = (T)spline_eval_d(Int, Mk, mInv, Nr, (double)v, &bad);
    if (bad) atomicOr(err, 16);
  }
}

// I(M) at the mass (T)sphere[q] * Mcell of every sphere size q < nt, as
// k_masses would evaluate it for a halo of that size (a table, since most
// halos share a few sizes); ibad[q] flags a mass outside the spline's range.
template <typename T>
__global__ void k_mass_table(const int* sphere, int nt, T Mcell, const double* Mk,
                             const double* Int, const double* mI, int Nr, double* itab,
                             int* ibad) {
  for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < nt; q += gridDim.x * blockDim.x) {
    int bad = 0;
    const T m = (T)sphere[q] * Mcell;
    itab[q] = spline_eval_d(Mk, Int, mI, Nr, (double)m, &bad);
    ibad[q] = bad;
  }
}

__global__ void k_flag_out(const int* flag, long long ng, const int* hidx, long long* out) {
  for (long long c = blockIdx.x * (long long)blockDim.x + threadIdx.x; c < ng;
       c += (long long)gridDim.x * blockDim.x) {
    int v = flag[c];
    long long o;
    if (v == FLAG_FREE || v <= FLAG_PENDING)
      o = ng;
    else if (v == FLAG_REJECTED)
      o = ng + 1;
    else {
      long long h = hidx[v >> 1];
      o = (v & 1) ? -h : h;
    }
    out[c] = o;
  }
}

// Halo displacements: the mean over the member sphere, summed in double.  A
// halo of one cell (81% of a 512^3 box's at 4 Mpc/h) takes one thread, a
// larger one a row of 16 lanes that share its cells, so that no wave waits
// for one thread's chain of loads through hundreds of cells.  The halos stand
// in order of density, so a workgroup's are of similar size: HPB = 16 of them
// (one a row) where there are few halos, else 256.  A row adds 16 partial sums
// (cells l, l + 16, ..) in a tree, not the cells in order: FP64 positions and
// velocities of halos of several cells differ from a sum in order in the last
// bits, like any two orders of a double sum.
template <typename T, bool VEL>
__device__ __forceinline__ void posh_store(const double* s, const double* v, int hc, int ci,
                                           int cj, int ck, T Lc, T L0, T L1, T L2, T* posh,
                                           T* velh, size_t h) {
  const int q[3] = {ci, cj, ck};
  const T L[3] = {L0, L1, L2};
#pragma unroll
  for (int a = 0; a < 3; a++) {
    const T base = (T)((double)((T)q[a] * Lc) + (double)Lc / 2.0);
    T r = base + (T)(s[a] / hc);
    if (r >= L[a]) r -= L[a];
    if (r < (T)0) r += L[a];
    posh[3 * h + a] = r;
    if constexpr (VEL) velh[3 * h + a] = (T)(v[a] / hc);
  }
}

template <typename T, bool VEL, int HPB>
__global__ __launch_bounds__(256) void k_halo_posh(const int* hx, const int* hcount,
                                                   const int* hr2, long long nh, ShellTab sh,
                                                   int n0, int n1, int n2, const T* S, const T* V,
                                                   T Lc, T L0, T L1, T L2, int lagrangian,
                                                   T* posh, T* velh) {
  __shared__ short s_at[HPB];
  __shared__ int s_end[HPB];
  __shared__ int nlist, taken;
  using V3 = typename vec3<T>::type;
  const long long h0 = blockIdx.x * (long long)HPB, h = h0 + threadIdx.x;
  const int lane = threadIdx.x & 63;
  if (threadIdx.x == 0) {
    nlist = 0;
    taken = 0;
  }
  __syncthreads();
  int end = 0;
  bool more = false;
  if ((int)threadIdx.x < HPB && h < nh) {
    const int ci = hx[3 * h], cj = hx[3 * h + 1], ck = hx[3 * h + 2], hc = hcount[h];
    end = lagrangian ? 0 : table_at(sh.start, hr2[h]);
    more = end > 1;
    if (!more) {
      double s[3] = {0, 0, 0}, v[3] = {0, 0, 0};
      if (end == 1) {
        const size_t id = ((size_t)ci * n1 + cj) * n2 + ck;
        const V3 a = *reinterpret_cast<const V3*>(S + 3 * id);
        s[0] += (double)a.x;
        s[1] += (double)a.y;
        s[2] += (double)a.z;
        if constexpr (VEL) {
          const V3 u = *reinterpret_cast<const V3*>(V + 3 * id);
          v[0] += (double)u.x;
          v[1] += (double)u.y;
          v[2] += (double)u.z;
        }
      }
      posh_store<T, VEL>(s, v, hc, ci, cj, ck, Lc, L0, L1, L2, posh, velh, h);
    }
  }
  const unsigned long long bal = __ballot(more);
  int at = 0;
  if (bal && lane == 0) at = atomicAdd(&nlist, __popcll(bal));
  at = __shfl(at, 0, 64) + __popcll(bal & lanemask_lt());
  if (more) {
    s_at[at] = (short)threadIdx.x;
    s_end[at] = end;
  }
  __syncthreads();
  const int nl = nlist, l16 = lane & 15, row = lane >> 4;
  for (;;) {
    int q = 0;
    if (lane == 0) q = atomicAdd(&taken, 4);
    q = __builtin_amdgcn_readfirstlane(q);
    if (q >= nl) break;
    if (q + row >= nl) continue;
    const size_t g = (size_t)h0 + s_at[q + row];
    const int cells = s_end[q + row];
    const int ci = hx[3 * g], cj = hx[3 * g + 1], ck = hx[3 * g + 2], hc = hcount[g];
    double s[3] = {0, 0, 0}, v[3] = {0, 0, 0};
    for (int ob = l16; ob < cells; ob += 64) {
      V3 sv[4], vv[4];
#pragma unroll
      for (int k = 0; k < 4; k++)
        if (ob + 16 * k < cells) {
          const size_t id = cell_off(ci, cj, ck, sh.offs[ob + 16 * k], n0, n1, n2);
          sv[k] = *reinterpret_cast<const V3*>(S + 3 * id);
          if constexpr (VEL) vv[k] = *reinterpret_cast<const V3*>(V + 3 * id);
        }
#pragma unroll
      for (int k = 0; k < 4; k++)
        if (ob + 16 * k < cells) {
          s[0] += (double)sv[k].x;
          s[1] += (double)sv[k].y;
          s[2] += (double)sv[k].z;
          if constexpr (VEL) {
            v[0] += (double)vv[k].x;
            v[1] += (double)vv[k].y;
            v[2] += (double)vv[k].z;
          }
        }
    }
#pragma unroll
    for (int a = 0; a < 3; a++) {
#pragma unroll
      for (int o = 8; o > 0; o >>= 1) {
        s[a] += __shfl_xor(s[a], o, 16);
        if constexpr (VEL) v[a] += __shfl_xor(v[a], o, 16);
      }
    }
    if (l16 == 0) posh_store<T, VEL>(s, v, hc, ci, cj, ck, Lc, L0, L1, L2, posh, velh, g);
  }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
// Shell starts, ball starts, shell offsets and ball offsets of (stab, tmax) in
// one array.
struct ShellArrays {
  std::vector<unsigned> all;
  size_t ns, nb, no;
  int ball_max;
};

static ShellArrays build_shells(int stab, int tmax) {
  std::vector<int> start, ball(BALL_MAX + 1, 0);
  std::vector<unsigned> packed, balls;
  shell_offsets(stab, tmax, start, packed);
  const int bmax = std::min(BALL_MAX, stab);
  // the largest ball is sorted once; the smaller ones are parts of it, in its
  // order (each sorted by itself, the balls took 3.3 ms, now 0.4)
  struct Off {
    unsigned order, p;
    int r2;
  };
  std::vector<Off> largest;
  for (int r2 = 0; r2 < bmax; r2++)
    for (int e = start[r2]; e < start[r2 + 1]; e++) {
      const unsigned p = packed[e];
      largest.push_back({(p & 255u) << 16 | (p & 0xff00u) | p >> 16, p, r2});
    }
  std::sort(largest.begin(), largest.end(),
            [](const Off& a, const Off& b) { return a.order < b.order; });
  for (int G = 1; G <= bmax; G++) {
    ball[G] = (int)balls.size();
    for (const Off& o : largest)
      if (o.r2 < G) balls.push_back(o.p);
  }
  ShellArrays t{{start.begin(), start.end()}, start.size(), ball.size(), packed.size(), bmax};
  t.all.insert(t.all.end(), ball.begin(), ball.end());
  t.all.insert(t.all.end(), packed.begin(), packed.end());
  t.all.insert(t.all.end(), balls.begin(), balls.end());
  return t;
}

// Those of every grid whose sides are 62 or more, built once per process (2 ms).
static constexpr int FULL_TMAX = 31;  // floor(sqrt(S_TAB_MAX - 1))
static const ShellArrays& full_shells() {
  static const ShellArrays t = build_shells(S_TAB_MAX, FULL_TMAX);
  return t;
}

// Upload the shell and ball tables for (stab, tmax) unless the context already
// holds them; returns the number of offsets.  Offsets of r^2 < stab lie within
// sqrt(stab - 1), so a larger tmax gives the same tables.
static long long ensure_shells(exh_ctx* c, int stab, int tmax) {
  HaloState& S = c->halo;
  tmax = std::min(tmax, isqrt_floor(stab - 1));
  if (S.sh.stab == stab && S.sh_tmax == tmax) return c->shell_noffs;
  const bool full = stab == S_TAB_MAX && tmax == FULL_TMAX;
  const ShellArrays own = full ? ShellArrays{} : build_shells(stab, tmax);
  const ShellArrays& t = full ? full_shells() : own;
  int* d = (int*)ctx_buf(c, BUF_SHELL, t.all.size() * 4);
  EXH_CHECK_HIP(
      hipMemcpyAsync(d, t.all.data(), t.all.size() * 4, hipMemcpyHostToDevice, c->stream));
  EXH_CHECK_HIP(hipStreamSynchronize(c->stream));
  S.sh.start = d;
  S.sh.ball = d + t.ns;
  S.sh.offs = (const unsigned*)(d + t.ns + t.nb);
  S.sh.balls = (const unsigned*)(d + t.ns + t.nb + t.no);
  S.sh.stab = stab;
  S.sh.ball_max = t.ball_max;
  S.sh_tmax = tmax;
  c->shell_noffs = (long long)t.no;
  return c->shell_noffs;
}

// Constant tables, built once per process.
static const std::vector<int>& sphere_table() {
  static const std::vector<int> t = cells_in_spheres(10000);
  return t;
}

static const std::vector<unsigned>& taus_table() {
  static const std::vector<unsigned> t = [] {
    std::vector<unsigned> m(3 * 40 * 32);
    taus_jump_tables(m.data());
    return m;
  }();
  return t;
}

template <typename T>
// phase(p), when given, is called as the finder reaches p: 0 = start,
// 1 = after the peak sort, 2 = before the growth rounds (launches of other
// streams can be placed there).
long long run_find_halos(exh_ctx* c, const exh_box* b, const T* delta, const exh_halo_opts* o,
                         const std::function<void(int)>& phase) {
  if (phase) phase(0);
  const int n0 = b->nd[0], n1 = b->nd[1], n2 = b->nd[2];
  const long long ng = b->ng;
  EXH_REQUIRE(ng < (1LL << 30), EXH_ERR_ARG, "grid too large for int32 cell indices");
  HaloState& S = c->halo;
  S.ng = ng;
  S.have_posh = S.have_velh = false;
  const int tmax = b->nmin / 2;
  const int stab = std::min(S_TAB_MAX, 3 * tmax * tmax + 2);
  const long long noffs = ensure_shells(c, stab, tmax);

  // tables (built on the host, kept on the device while their inputs are
  // unchanged): barrier per count, mass-function knots and their splines,
  // sphere counts, taus jump matrices
  const int nBt = (int)noffs + 2;
  const std::vector<int>& sph = sphere_table();
  const std::vector<unsigned>& mats = taus_table();
  size_t toff = 0;
  auto ttake = [&](size_t bytes) {
    size_t r = toff;
    toff += (bytes + 255) & ~(size_t)255;
    return r;
  };
  const int Nr = halo_table_radii(o);  // knots of the sigma(M) and Tinker tables
  const size_t o_bt = ttake(nBt * sizeof(T)), o_mk = ttake(Nr * 8), o_int = ttake(Nr * 8),
               o_mi = ttake(Nr * 8), o_minv = ttake(Nr * 8), o_sph = ttake(sph.size() * 4),
               o_mats = ttake(mats.size() * 4);
  std::vector<unsigned char> key;
  const double oscal[3] = {o->a, o->beta, o->alpha};
  const int sizes[3] = {o->Nk, nBt, o->sigma_radii};
  key_append(key, b, 1);
  key_append(key, oscal, 3);
  key_append(key, sizes, 3);
  key_append(key, o->k, o->Nk);
  key_append(key, o->P, o->Nk);
  const size_t cap0 = c->cap[BUF_HALOTAB];
  char* tabs = (char*)ctx_buf(c, BUF_HALOTAB, toff);
  if (c->cap[BUF_HALOTAB] != cap0) c->halotab_key.clear();  // reallocated
  if (key != c->halotab_key) {
    std::vector<T> sig(std::max(1, (int)std::floor(1e16 / (T)b->Mcell)) + 1), Bt(nBt);
    std::vector<double> Mk(Nr), Int(Nr);
    int Ncells = halo_tables(b, o, sig.data(), Bt.data(), nBt, Mk.data(), Int.data());
    EXH_REQUIRE(Ncells >= 1, Ncells < 0 ? EXH_ERR_RANGE : EXH_ERR_ARG,
                "sigma(M) table: cell mass %g gives %d cells below M_max", (double)b->Mcell,
                Ncells);
    std::vector<double> mI(Nr), mInv(Nr);
    spline_second_derivs(Mk.data(), Int.data(), Nr, mI.data());
    spline_second_derivs(Int.data(), Mk.data(), Nr, mInv.data());
    auto up = [&](size_t o2, const void* src, size_t bytes) {
      EXH_CHECK_HIP(hipMemcpyAsync(tabs + o2, src, bytes, hipMemcpyHostToDevice, c->stream));
    };
    up(o_bt, Bt.data(), nBt * sizeof(T));
    up(o_mk, Mk.data(), Nr * 8);
    up(o_int, Int.data(), Nr * 8);
    up(o_mi, mI.data(), Nr * 8);
    up(o_minv, mInv.data(), Nr * 8);
    up(o_sph, sph.data(), sph.size() * 4);
    up(o_mats, mats.data(), mats.size() * 4);
    EXH_CHECK_HIP(hipStreamSynchronize(c->stream));  // the host tables are temporaries
    c->halotab_key = key;
    c->halotab_ncells = Ncells;
    c->halotab_bmin = (double)Bt[Ncells - 1];
  }
  const int Ncells = c->halotab_ncells;
  const T Bmin = (T)c->halotab_bmin;
  // 1. peaks
  long long nblk = (ng + PK_TILE - 1) / PK_TILE;
  const PeakGeom pg{n0, n1, n2, (unsigned)((long long)n1 * n2), (unsigned)n2, fast_div(n2),
                    fast_div(n1)};
  // block counts and offsets, then the peak flag bytes
  const size_t o_pb = ((size_t)(2 * nblk + 2) * 8 + 255) & ~(size_t)255;
  char* hb = (char*)ctx_buf(c, BUF_HALO, o_pb + (size_t)nblk * 256);
  long long* bc = (long long*)hb;
  unsigned char* pbits = (unsigned char*)(hb + o_pb);
  int* flag = (int*)ctx_buf(c, BUF_FLAG, (size_t)ng * 4);
  T* eff = (T*)ctx_buf(c, BUF_EFF, (size_t)ng * sizeof(T));
  unsigned long long* claim = (unsigned long long*)ctx_buf(c, BUF_CLAIM, (size_t)ng * 8);
  {
    TimedScope ts(c, "peaks");
    hipLaunchKernelGGL(k_peak_count<T>, dim3((unsigned)nblk), dim3(256), 0, c->stream, delta, pg,
                       Bmin, bc, eff, pbits);
    EXH_LAUNCH_CHECK();
    exclusive_scan<long long>(c, bc, bc + nblk + 1, nblk);
  }
  long long* hbuf = (long long*)ctx_pinned(c, 1024);
  EXH_CHECK_HIP(hipMemcpyAsync(hbuf, bc + nblk + 1 + nblk, 8, hipMemcpyDeviceToHost, c->stream));
  EXH_CHECK_HIP(hipStreamSynchronize(c->stream));
  const long long np = hbuf[0] & ((1LL << LOW_SHIFT) - 1), below = hbuf[0] >> LOW_SHIFT;
  c->stat_peaks = np;
  T* pkey = (T*)ctx_buf(c, BUF_PEAK_KEY, (size_t)std::max(np, 1LL) * sizeof(T));
  int* pcell = (int*)ctx_buf(c, BUF_PEAK_CELL, (size_t)std::max(np, 1LL) * sizeof(int));
  {
    TimedScope ts(c, "peaks_write");
    hipLaunchKernelGGL(k_peak_write<T>, dim3((unsigned)nblk), dim3(256), 0, c->stream, delta, pg,
                       bc + nblk + 1, pbits, pkey, pcell, flag);
    EXH_LAUNCH_CHECK();
  }
  // 2. sort (densities in lexicographic peak order).  Peaks below the smallest
  // barrier are never visited: their count is the first visited sorted
  // position, and the sort leaves their order open.
  int* perm = (int*)ctx_buf(c, BUF_PEAK_IDX, (size_t)std::max(np, 1LL) * sizeof(int));
  lomuto_sort<T>(c, pkey, perm, np, (double)Bmin);
  if (phase) phase(1);

  // 3. candidates
  const long long nc = std::max(np - std::max(below, 1LL), 0LL);
  c->stat_candidates = nc;

  // candidate state in BUF_CAND: by rank, by list position, lists' counts
  size_t coff = 0;
  auto ctake = [&](size_t bytes) {
    size_t r = coff;
    coff += (bytes + 255) & ~(size_t)255;
    return r;
  };
  const size_t ncs = (size_t)std::max(nc, 1LL);
  // list x may hold every peak of its blocks
  const long long nblk_p = std::max((np + PK_TILE - 1) / PK_TILE, 1LL);
  const long long lcap = (nblk_p + NXCD - 1) / NXCD * PK_TILE;
  const size_t nls = (size_t)lcap * NXCD;
  const long long nblk_c = (nc + PK_TILE - 1) / PK_TILE;
  const size_t nps = (size_t)std::max(np, 1LL);
  const size_t o_res = ctake(nps * 2), o_rres = ctake(ncs * 2), o_p0 = ctake(nls * 4),
               o_p1 = ctake(nls * 4), o_rk = ctake(nps * 4), o_hid = ctake(ncs * 4),
               o_pk0 = ctake(nls * 4), o_pk1 = ctake(nls * 4), o_pg = ctake(nls * 4),
               o_hb = ctake((size_t)(2 * std::max(nblk_c, 1LL) + 2) * 8),
               o_rt = ctake((RT_RING * NXCD + 1) * 4);
  char* cand = (char*)ctx_buf(c, BUF_CAND, coff);
  // eff (delta) and the free flags were written by the peak passes
  S.flag = flag;
  int* rt = (int*)(cand + o_rt);
  int* derr = rt + RT_RING * NXCD;

  GrowArgs<T> ga{};
  ga.n0 = n0;
  ga.n1 = n1;
  ga.n2 = n2;
  ga.delta = delta;
  ga.eff = eff;
  ga.flag = flag;
  ga.claim = claim;
  ga.sh = S.sh;
  ga.Bt = (const T*)(tabs + o_bt);
  ga.nB = nBt;
  ga.Bmin = Bmin;
  ga.negMtot = -(T)b->Mtot;
  ga.Nmin = o->Nmin;
  ga.pcell = pcell;
  ga.pkey = pkey;
  ga.pres = (int*)(cand + o_pg);
  ga.res = (unsigned short*)(cand + o_res);
  ga.err = derr;
  int* pend = (int*)(cand + o_p0);
  int* pnext = (int*)(cand + o_p1);
  int* qpeak = (int*)(cand + o_pk0);
  int* qpeak_next = (int*)(cand + o_pk1);
  {
    TimedScope ts(c, "halo_candidates");
    int* rank = (int*)(cand + o_rk);
    const long long nrk = std::max(np - below, 1LL);
    hipLaunchKernelGGL(k_cand_ranks, dim3(grid_for(nrk, 1024)), dim3(256), 0, c->stream, perm,
                       (int)np, (int)below, rank, rt);
    hipLaunchKernelGGL(k_list_build<T>, dim3((unsigned)nblk_p), dim3(256), 0, c->stream, pkey,
                       pcell, rank, (int)np, (int)nc, Bmin, (int)lcap, rt, pend, qpeak, ga.res,
                       flag);
    EXH_LAUNCH_CHECK();
  }
  if (phase) phase(2);
  // Rounds run in batches without a host read between them: each round's
  // pending count stays on the device (a ring of RT_RING counts), grids are
  // sized by the last count the host read (counts only shrink), and the
  // host reads the counts and the error flag once per batch.  A round with
  // no pending candidate launches blocks that return at once.
  // Claims carry their round's tag (an epoch counted over the context's
  // calls) above the inverted rank, so the claims of earlier rounds and
  // calls never match a later round: the array is cleared only when it is
  // newly allocated, when the claim width changes, or before the epoch
  // wraps (every 255 rounds with 32-bit claims).
  const bool c32 = nc < (1LL << 24) && c->tune_halo_claims != 64;
  const int cmode = c32 ? 32 : 64;
  auto clear_claims = [&]() {
    const long long ncap = (long long)(c->cap[BUF_CLAIM] / 8);
    hipLaunchKernelGGL(k_fill_u64, dim3(grid_for(ncap, 256 * 8)), dim3(256), 0, c->stream, claim,
                       ncap, 0ull);
    EXH_LAUNCH_CHECK();
    c->claim_epoch = 0;
  };
  if (c->claim_gen != c->buf_gen[BUF_CLAIM] || c->claim_mode != cmode ||
      c->claim_epoch > 0xffffffffu - 2000000u) {
    clear_claims();
    c->claim_gen = c->buf_gen[BUF_CLAIM];
    c->claim_mode = cmode;
  }
  // candidates per workgroup: 256, or 64 (16 rows for their long growths)
  // where 256 would leave most CUs idle
  long long ub = nc > 0 ? std::min(lcap, nc) : 0;  // bounds the longest list
  int round = 0, launched = 0;
  {
    TimedScope ts(c, "halo_rounds");
    while (ub > 0) {
      const int batch = launched == 0 ? 1 : RT_BATCH;
      const int first = launched;
      const int cpb = ub * NXCD > 256 * 512 ? 256 : 64;
      const dim3 grid((unsigned)((ub + cpb - 1) / cpb) * NXCD);
      for (int q = 0; q < batch; q++) {
        RoundLists rl;
        rl.n = rt + launched % RT_RING * NXCD;
        rl.next = rt + (launched + 1) % RT_RING * NXCD;
        rl.clear = rt + (launched + 2) % RT_RING * NXCD;
        rl.cap = (int)lcap;
        rl.rank_out = pnext;
        rl.peak_out = qpeak_next;
        launched++;
        if (c32 && c->claim_epoch >= 255) clear_claims();
        const unsigned long long ep = ++c->claim_epoch;
        const unsigned long long tag_hi = c32 ? ep << 24 : ep << 32;
        ga.prank = pend;
        ga.ppeak = qpeak;
        auto go = [&](auto kg, auto kc) {
          hipLaunchKernelGGL(kg, grid, dim3(256), 0, c->stream, ga, rl, tag_hi);
          hipLaunchKernelGGL(kc, grid, dim3(256), 0, c->stream, ga, rl, tag_hi, tmax);
        };
        if (c32 && cpb == 256)
          go(k_grow<T, true, 256>, k_commit<T, true, 256>);
        else if (c32)
          go(k_grow<T, true, 64>, k_commit<T, true, 64>);
        else if (cpb == 256)
          go(k_grow<T, false, 256>, k_commit<T, false, 256>);
        else
          go(k_grow<T, false, 64>, k_commit<T, false, 64>);
        EXH_LAUNCH_CHECK();
        std::swap(pend, pnext);
        std::swap(qpeak, qpeak_next);
      }
      int* hr = (int*)hbuf;  // the ring and the error flag
      EXH_CHECK_HIP(hipMemcpyAsync(hr, rt, (RT_RING * NXCD + 1) * 4, hipMemcpyDeviceToHost,
                                   c->stream));
      EXH_CHECK_HIP(hipStreamSynchronize(c->stream));
      const int e = hr[RT_RING * NXCD];
      EXH_REQUIRE(e == 0, EXH_ERR_RANGE,
                  "halo growth left the supported range (code %d): radius^2 beyond %d, count "
                  "beyond the barrier table, or a sphere wider than half the box",
                  e, stab - 1);
      auto longest = [&](int r) {
        const int* h = hr + r % RT_RING * NXCD;
        return (long long)*std::max_element(h, h + NXCD);
      };
      for (int r = first; r < launched; r++)
        if (longest(r) > 0) round++;
      ub = longest(launched);
      EXH_REQUIRE(launched < 1000000, EXH_ERR_INTERNAL, "halo rounds did not converge");
    }
  }
  c->stat_rounds = round;

  // 4. catalogue
  long long* hb2 = (long long*)(cand + o_hb);
  int* hidx = (int*)(cand + o_hid);
  unsigned short* rres = (unsigned short*)(cand + o_rres);
  long long nh = 0;
  if (nc > 0) {
    hipLaunchKernelGGL(k_halo_count, dim3((unsigned)nblk_c), dim3(256), 0, c->stream, ga.res,
                       perm, (int)np, (int)nc, rres, hb2);
    EXH_LAUNCH_CHECK();
    exclusive_scan<long long>(c, hb2, hb2 + nblk_c + 1, nblk_c);
    EXH_CHECK_HIP(hipMemcpyAsync(hbuf, hb2 + 2 * nblk_c + 1, 8, hipMemcpyDeviceToHost, c->stream));
    EXH_CHECK_HIP(hipStreamSynchronize(c->stream));
    nh = hbuf[0];
  }
  S.hidx = hidx;
  size_t hs = (size_t)std::max(nh, 1LL);
  size_t hoff = 0;
  auto htake = [&](size_t bytes) {
    size_t r = hoff;
    hoff += (bytes + 255) & ~(size_t)255;
    return r;
  };
  size_t o_hx = htake(hs * 12), o_hc = htake(hs * 4), o_hr = htake(hs * 4),
         o_mh = htake(hs * sizeof(T)), o_u = htake(hs * 8), o_ph = htake(hs * 3 * sizeof(T)),
         o_vh = htake(hs * 3 * sizeof(T));
  // I(M) per sphere size for the masses: every index k_masses can read
  const int nsph = (int)sph.size();
  const int ntab = std::max(1, std::min(std::min(Ncells, nsph) + 1, nsph));
  const size_t o_itab = htake((size_t)ntab * 8), o_ibad = htake((size_t)ntab * 4);
  char* hal = (char*)ctx_buf(c, BUF_HALO, hoff);
  S.hx = (int*)(hal + o_hx);
  S.hcount = (int*)(hal + o_hc);
  S.hr2 = (int*)(hal + o_hr);
  S.Mh = hal + o_mh;
  S.posh = hal + o_ph;
  S.velh = hal + o_vh;
  if (nh > 0)
    hipLaunchKernelGGL(k_gather_halos<T>, dim3((unsigned)nblk_c), dim3(256), 0, c->stream, rres,
                       hb2 + nblk_c + 1, (int)nc, perm, pcell, (int)np, S.sh.start, n1, n2, S.hx,
                       S.hcount, S.hr2, hidx);
  EXH_LAUNCH_CHECK();
  // 5. masses
  if (nh > 0) {
    TimedScope ts(c, "halo_masses");
    uint32_t st[3];
    taus_seed_state(o->seed, st);
    double* u = (double*)(hal + o_u);
    hipLaunchKernelGGL(k_taus, dim3(grid_for((nh + 63) / 64, 256)), dim3(256), 0, c->stream,
                       (const unsigned*)(tabs + o_mats), st[0], st[1], st[2], nh, u);
    EXH_LAUNCH_CHECK();
    double* itab = (double*)(hal + o_itab);
    int* ibad = (int*)(hal + o_ibad);
    hipLaunchKernelGGL(k_mass_table<T>, dim3(grid_for(ntab, 256)), dim3(256), 0, c->stream,
                       (const int*)(tabs + o_sph), ntab, (T)b->Mcell,
                       (const double*)(tabs + o_mk), (const double*)(tabs + o_int),
                       (const double*)(tabs + o_mi), Nr, itab, ibad);
    hipLaunchKernelGGL(k_masses<T>, dim3(grid_for(nh, 256)), dim3(256), 0, c->stream, S.hcount, nh,
                       (const int*)(tabs + o_sph), nsph, Ncells, itab, ibad,
                       (const double*)(tabs + o_mk), (const double*)(tabs + o_int),
                       (const double*)(tabs + o_minv), Nr, u, (T*)S.Mh, derr);
    EXH_LAUNCH_CHECK();
    EXH_CHECK_HIP(hipMemcpyAsync(hbuf, derr, 4, hipMemcpyDeviceToHost, c->stream));
    EXH_CHECK_HIP(hipStreamSynchronize(c->stream));
    int e = ((int*)hbuf)[0];
    EXH_REQUIRE(e == 0, EXH_ERR_RANGE,
                "halo mass draw left the tabulated mass function (code %d): a halo's next "
                "sphere exceeds M_max = 1e16 Msun/h",
                e);
  }
  c->nh = nh;
  c->last_prec = b->precision;
  return nh;
}

template <typename T>
void run_halo_posh(exh_ctx* c, const exh_box* b, const T* S, const T* V, int lagrangian) {
  HaloState& st = c->halo;
  if (c->nh <= 0) return;
  TimedScope ts(c, "halo_posh");
  const bool few = c->nh < 256 * 1024;
  auto kern = few ? (V ? k_halo_posh<T, true, 16> : k_halo_posh<T, false, 16>)
                  : (V ? k_halo_posh<T, true, 256> : k_halo_posh<T, false, 256>);
  hipLaunchKernelGGL(kern, dim3(grid_for(c->nh, few ? 16 : 256)), dim3(256), 0, c->stream, st.hx,
                     st.hcount, st.hr2, c->nh, st.sh, b->nd[0], b->nd[1], b->nd[2], S, V,
                     (T)b->Lc, (T)b->L[0], (T)b->L[1], (T)b->L[2], lagrangian, (T*)st.posh,
                     V ? (T*)st.velh : nullptr);
  EXH_LAUNCH_CHECK();
}

void run_halo_flag(exh_ctx* c, const exh_box* b, long long* flag_dev) {
  HaloState& st = c->halo;
  hipLaunchKernelGGL(k_flag_out, dim3(grid_for(b->ng, 256 * 8)), dim3(256), 0, c->stream, st.flag,
                     b->ng, st.hidx, flag_dev);
  EXH_LAUNCH_CHECK();
}

template long long run_find_halos<float>(exh_ctx*, const exh_box*, const float*,
                                        const exh_halo_opts*, const std::function<void(int)>&);
template long long run_find_halos<double>(exh_ctx*, const exh_box*, const double*,
                                         const exh_halo_opts*, const std::function<void(int)>&);
template void run_halo_posh<float>(exh_ctx*, const exh_box*, const float*, const float*, int);
template void run_halo_posh<double>(exh_ctx*, const exh_box*, const double*, const double*, int);

}  // namespace exh
