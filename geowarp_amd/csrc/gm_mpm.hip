// cpGIMP implicit MPM kernels for gfx950 (FP64 state, FP64 or FP32 Jacobian).
//
// Design (one load step, weights fixed because particles do not move inside
// the Newton loop):
//   1. gm_bin_particles   sort particle ids by their stencil base node (counting
//                         sort + per-bucket id sort => deterministic order)
//   2. gm_bsr_pattern     per node row, OR the support boxes of the particles
//                         touching it into a 5^d window mask -> block-CSR pattern
//   3. per Newton iteration:
//      gm_particle_stage  one particle per lane: gather du, p; kinematics;
//                         constitutive update; particle stress vector Y and
//                         tangent D = dY/dz (z = grad(du), p, pbar, grad p ...)
//      gm_node_residual   one node per lane: r_I = sum_p L(geom_I) Y_p
//                         (deterministic gather instead of the reference's atomics)
//      gm_node_jacobian   one wavefront per node row: K_IJ = -sum_p L_I D_p M_J
//                         into the block-CSR slots, masked + identity rows
//   The reference builds the same matrix with 5^d x nb coloured reverse sweeps
//   (solvers/sparse_differentiation.py:213-401, qc3d:285-321); here it is
//   assembled analytically in one pass.
#include <hip/hip_runtime.h>
#include <stdarg.h>
#include <stdlib.h>
#include <string.h>

#include <type_traits>
#include <utility>

#include "gm_common.h"
#include "gm_device.h"
#include "gm_types.h"

namespace gm {
static thread_local char g_err[1024] = "";
void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
}
}  // namespace gm

extern "C" const char* gm_last_error(void) { return gm::g_err; }
extern "C" int gm_version(void) { return 1; }

using namespace gm;

// ------------------------------------------------------------------ layouts
template <int DIM, bool COUPLED>
struct Lay {
  static constexpr int NB = DIM + (COUPLED ? 1 : 0);
  static constexpr int NH = DIM * DIM;
  static constexpr int Z_DU = NH;  // 3D u-p only: z-displacement for the indenter penalty
  static constexpr int Z_P = NH + ((DIM == 3 && COUPLED) ? 1 : 0);
  static constexpr int Z_PB = Z_P + 1;
  static constexpr int Z_G = Z_P + 2;
  static constexpr int NZ = COUPLED ? Z_G + DIM : NH;
  static constexpr int Y_T = NH;
  static constexpr int Y_Q = NH + DIM;
  static constexpr int Y_M = Y_Q + 1;
  static constexpr int Y_S = Y_M + DIM;
  static constexpr int NY = COUPLED ? Y_S + 1 : NH + DIM;
};

template <int DIM>
__device__ __forceinline__ void load_axes(const gm_grid& g, const double* x, const double* lp, int p, Axis* ax) {
#pragma unroll
  for (int a = 0; a < DIM; ++a) ax[a] = gimp_axis(x[p * DIM + a], lp[p * DIM + a], g.h[a], g.inv_h[a]);
}

template <int DIM>
__device__ __forceinline__ int node_index(const gm_grid& g, const int* c) {
  if (DIM == 2) return c[0] + c[1] * (g.nx + 1);
  return c[0] + c[1] * (g.nx + 1) + c[2] * (g.nx + 1) * (g.ny + 1);
}

template <int DIM>
__device__ __forceinline__ void node_coords(const gm_grid& g, int n, int* c) {
  c[0] = n % (g.nx + 1);
  if (DIM == 2) {
    c[1] = n / (g.nx + 1);
  } else {
    c[1] = (n / (g.nx + 1)) % (g.ny + 1);
    c[2] = n / ((g.nx + 1) * (g.ny + 1));
  }
}

// ================================================================== binning
// Particles by base node, then id: a count (whose atomics hand every particle its place among the
// bin's, in no particular order), a scan, the ids to their places, and each id's rank within its
// bin.  The ids pass through x_s, which is written last.
__global__ void k_bin_count(gm_grid g, const double* x, const double* lp, int n, int* pbase, uint8_t* ext,
                            int* count, int* slot, int* err) {
  int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  int ncell[3] = {g.nx, g.ny, g.nz};
  int lo[3] = {0, 0, 0};
  uint8_t e = 0;
  bool ok = true;
  for (int a = 0; a < g.dim; ++a) {
    Axis ax = gimp_axis(x[p * g.dim + a], lp[p * g.dim + a], g.h[a], g.inv_h[a]);
    lo[a] = ax.lo;
    if (ax.ext == 3) e |= (uint8_t)(1u << a);
    if (ax.lo < 0 || ax.lo + ax.ext - 1 > ncell[a]) ok = false;
    double xv = x[p * g.dim + a];
    if (!(xv == xv)) ok = false;
  }
  if (!ok) {
    atomicAdd(err, 1);
    pbase[p] = -1;
    ext[p] = 0;
    return;
  }
  int b = (g.dim == 2) ? lo[0] + lo[1] * (g.nx + 1) : lo[0] + lo[1] * (g.nx + 1) + lo[2] * (g.nx + 1) * (g.ny + 1);
  pbase[p] = b;
  ext[p] = e;
  slot[p] = atomicAdd(&count[b], 1);
}

__global__ void k_bin_scatter(int n, const int* pbase, const int* start, const int* slot, int* ids) {
  int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  int b = pbase[p];
  if (b >= 0) ids[start[b] + slot[p]] = p;
}

// A thread per id counts the smaller ones of its bin, where a thread per bin sorting its ids in
// place waited for every swap: 28 -> 5 us for 102,080 particles.
__global__ void k_bin_rank(int n_nodes, const int* pbase, const int* start, const int* ids, int* sorted) {
  int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= start[n_nodes]) return;  // (particles off the grid have no place)
  const int p = ids[k], b = pbase[p], s = start[b], e = start[b + 1];
  int r = s;
  for (int i = s; i < e; ++i) r += ids[i] < p;
  sorted[r] = p;
}

// bin-sorted copies of the per-particle geometry (index k = position in `sorted`)
__global__ void k_bin_finalize(int n, int dim, const int* sorted, const double* x, const double* lp,
                               const uint8_t* ext, uint8_t* ext_s, double* x_s, double* lp_s) {
  int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  int p = sorted[k];
  ext_s[k] = ext[p];
  for (int a = 0; a < dim; ++a) {
    x_s[k * dim + a] = x[p * dim + a];
    lp_s[k * dim + a] = lp[p * dim + a];
  }
}

// ---- exclusive scan of n ints (n <= 4M), three phases
#define SCAN_T 1024
#define SCAN_ITEMS 4
__global__ void k_scan_blocks(const int* in, int* out, int n, int* sums) {
  __shared__ int sh[SCAN_T];
  int base = blockIdx.x * SCAN_T * SCAN_ITEMS + threadIdx.x * SCAN_ITEMS;
  int v[SCAN_ITEMS];
  int loc = 0;
#pragma unroll
  for (int i = 0; i < SCAN_ITEMS; ++i) {
    v[i] = (base + i < n) ? in[base + i] : 0;
    loc += v[i];
  }
  sh[threadIdx.x] = loc;
  __syncthreads();
  for (int off = 1; off < SCAN_T; off <<= 1) {
    int t = (threadIdx.x >= off) ? sh[threadIdx.x - off] : 0;
    __syncthreads();
    sh[threadIdx.x] += t;
    __syncthreads();
  }
  int excl = sh[threadIdx.x] - loc;
  int run = excl;
#pragma unroll
  for (int i = 0; i < SCAN_ITEMS; ++i) {
    if (base + i < n) out[base + i] = run;
    run += v[i];
  }
  if (threadIdx.x == SCAN_T - 1) sums[blockIdx.x] = sh[SCAN_T - 1];
}

__global__ void k_scan_sums(int* sums, int nb) {
  __shared__ int sh[SCAN_T];
  int v = (threadIdx.x < nb) ? sums[threadIdx.x] : 0;
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int off = 1; off < SCAN_T; off <<= 1) {
    int t = (threadIdx.x >= off) ? sh[threadIdx.x - off] : 0;
    __syncthreads();
    sh[threadIdx.x] += t;
    __syncthreads();
  }
  if (threadIdx.x < nb) sums[threadIdx.x] = sh[threadIdx.x] - v;
  if (threadIdx.x == SCAN_T - 1) sums[SCAN_T] = sh[SCAN_T - 1];
}

__global__ void k_scan_add(int* out, int n, const int* sums) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  out[i] += sums[i / (SCAN_T * SCAN_ITEMS)];
}

// exclusive scan of in[0..n) into out[0..n]; out[n] = total.  tmp >= SCAN_T+1 ints.
static int exclusive_scan(const int* in, int* out, int n, int* tmp, hipStream_t s) {
  int nblk = gm_blocks(n, SCAN_T * SCAN_ITEMS);
  GM_REQUIRE(nblk <= SCAN_T, "scan: array too large");
  k_scan_blocks<<<nblk, SCAN_T, 0, s>>>(in, out, n, tmp);
  k_scan_sums<<<1, SCAN_T, 0, s>>>(tmp, nblk);
  k_scan_add<<<gm_blocks(n, 256), 256, 0, s>>>(out, n, tmp);
  GM_HIP(hipMemcpyAsync(out + n, tmp + SCAN_T, sizeof(int), hipMemcpyDeviceToDevice, s));
  GM_LAUNCH_CHECK();
  return 0;
}

extern "C" int gm_exclusive_scan(const int* in, int* out, int n, int* tmp, hipStream_t s) {
  return exclusive_scan(in, out, n, tmp, s);
}

// pbase: n_particles ints of scratch; err: one device int (count of particles off the grid)
extern "C" int gm_bin_particles(const gm_grid* g, const double* x, const double* lp, gm_bins* b, int* pbase,
                                int* err, hipStream_t s) {
  GM_REQUIRE(g && b && x && lp, "gm_bin_particles: null argument");
  int n = b->n_particles;
  GM_HIP(hipMemsetAsync(b->cell_count, 0, sizeof(int) * (g->n_nodes + 1), s));
  GM_HIP(hipMemsetAsync(err, 0, sizeof(int), s));
  if (n > 0) {
    k_bin_count<<<gm_blocks(n, 256), 256, 0, s>>>(*g, x, lp, n, pbase, b->ext, b->cell_count, b->sorted, err);
    GM_LAUNCH_CHECK();
  }
  int rc = exclusive_scan(b->cell_count, b->cell_start, g->n_nodes, b->scan_tmp, s);
  if (rc) return rc;
  if (n > 0) {
    int* ids = (int*)b->x_s;
    k_bin_scatter<<<gm_blocks(n, 256), 256, 0, s>>>(n, pbase, b->cell_start, b->sorted, ids);
    k_bin_rank<<<gm_blocks(n, 256), 256, 0, s>>>(g->n_nodes, pbase, b->cell_start, ids, b->sorted);
    k_bin_finalize<<<gm_blocks(n, 256), 256, 0, s>>>(n, g->dim, b->sorted, x, lp, b->ext, b->ext_s, b->x_s,
                                                     b->lp_s);
  }
  GM_LAUNCH_CHECK();
  return 0;
}

// ================================================================== candidate walk
// Visit every particle whose 3^d stencil contains node I (base cell I - o,
// o in {0,1,2}^d), in a fixed order.  f(k, o, b, in_support) with k the
// particle's bin-sorted position (ext_s is bin-sorted).
template <int DIM, typename F>
__device__ __forceinline__ void for_candidates(const gm_grid& g, const int* ci, const int* cell_start,
                                               const uint8_t* ext_s, F&& f) {
  int ncell[3] = {g.nx, g.ny, g.nz};
  const int oz_n = (DIM == 3) ? 3 : 1;
  for (int oz = 0; oz < oz_n; ++oz) {
    for (int oy = 0; oy < 3; ++oy) {
      for (int ox = 0; ox < 3; ++ox) {
        int o[3] = {ox, oy, oz};
        int b[3];
        bool ok = true;
#pragma unroll
        for (int a = 0; a < DIM; ++a) {
          b[a] = ci[a] - o[a];
          if (b[a] < 0 || b[a] > ncell[a]) ok = false;
        }
        if (!ok) continue;
        int bn = node_index<DIM>(g, b);
        int s = cell_start[bn], e = cell_start[bn + 1];
        for (int k = s; k < e; ++k) {
          uint8_t ex = ext_s[k];
          bool in = true;
#pragma unroll
          for (int a = 0; a < DIM; ++a) in = in && (o[a] < (((ex >> a) & 1) ? 3 : 2));
          f(k, o, b, in);
        }
      }
    }
  }
}

// ================================================================== pattern
template <int DIM>
__global__ void k_pattern_count(gm_grid g, const int* cell_start, const uint8_t* ext_s, uint64_t* mask,
                                int* row_nnzb) {
  int I = blockIdx.x * blockDim.x + threadIdx.x;
  if (I >= g.n_nodes) return;
  int ci[3] = {0, 0, 0};
  node_coords<DIM>(g, I, ci);
  uint64_t m0 = 0, m1 = 0;
  // centre bit
  int cb = (DIM == 2) ? (2 + 5 * 2) : (2 + 5 * 2 + 25 * 2);
  if (cb < 64) m0 |= (1ull << cb); else m1 |= (1ull << (cb - 64));
  for_candidates<DIM>(g, ci, cell_start, ext_s, [&](int k, const int* o, const int* b, bool in) {
    if (!in) return;
    uint8_t ex = ext_s[k];
    int e[3];
#pragma unroll
    for (int a = 0; a < DIM; ++a) e[a] = ((ex >> a) & 1) ? 3 : 2;
    const int kz_n = (DIM == 3) ? e[2] : 1;
    for (int kz = 0; kz < kz_n; ++kz)
      for (int ky = 0; ky < e[1]; ++ky)
        for (int kx = 0; kx < e[0]; ++kx) {
          int rx = kx - o[0] + 2, ry = ky - o[1] + 2, rz = (DIM == 3) ? (kz - o[2] + 2) : 0;
          int bit = rx + 5 * ry + 25 * rz;
          if (bit < 64) m0 |= (1ull << bit); else m1 |= (1ull << (bit - 64));
        }
  });
  mask[2 * I] = m0;
  mask[2 * I + 1] = m1;
  row_nnzb[I] = __popcll(m0) + __popcll(m1);
}

// The same row masks from each bin's set of support shapes: bit e of extset[b] is set
// when a particle of bin b has ext value e.  A particle's contribution to a row depends
// only on its bin (base node) and its ext value, so the union over the bin's particles
// is the union over the shapes present, at most 2^DIM per bin instead of one per particle.
__global__ void k_bin_extset(int n_bins, const int* cell_start, const uint8_t* ext_s, int* extset) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= n_bins) return;
  int s = 0;
  for (int k = cell_start[b]; k < cell_start[b + 1]; ++k) s |= 1 << ext_s[k];
  extset[b] = s;
}

// A support of shape ex seen from its node at offset o sets the window bits (k - o + 2) of its box:
// the box at o = (2, 2, 2) shifted, so a shape costs two shifts and not a loop over its nodes (139,425
// nodes: 218 -> 9 us).
template <int DIM>
__global__ void k_pattern_count_sets(gm_grid g, const int* extset, uint64_t* mask, int* row_nnzb) {
  constexpr int M = DIM == 3 ? 27 : 9;
  int I = blockIdx.x * blockDim.x + threadIdx.x;
  if (I >= g.n_nodes) return;
  int ci[3] = {0, 0, 0};
  node_coords<DIM>(g, I, ci);
  const int nx1 = g.nx + 1, nxy = nx1 * (g.ny + 1);
  int es[M];
#pragma unroll
  for (int o = 0; o < M; ++o) {
    const bool ok = ci[0] >= o % 3 && ci[1] >= o / 3 % 3 && ci[2] >= o / 9;
    es[o] = ok ? extset[I - o % 3 - o / 3 % 3 * nx1 - o / 9 * nxy] : 0;
  }
  const int cb = (DIM == 2) ? (2 + 5 * 2) : (2 + 5 * 2 + 25 * 2);  // centre bit
  uint64_t m0 = cb < 64 ? 1ull << cb : 0ull, m1 = cb < 64 ? 0ull : 1ull << (cb - 64);
#pragma unroll
  for (int o = 0; o < M; ++o) {
    const int ox = o % 3, oy = o / 3 % 3, oz = o / 9;
    uint64_t box = 0;  // the union of the shapes present that hold the node, at offset (2, 2, 2)
#pragma unroll
    for (int ex = 0; ex < (1 << DIM); ++ex) {
      if ((ox == 2 && !(ex & 1)) || (oy == 2 && !(ex & 2)) || (oz == 2 && !(ex & 4))) continue;
      uint64_t bits = (ex & 1) ? 7ull : 3ull;
      bits |= bits << 5 | ((ex & 2) ? bits << 10 : 0ull);
      if (DIM == 3) bits |= bits << 25 | ((ex & 4) ? bits << 50 : 0ull);
      if ((es[o] >> ex) & 1) box |= bits;
    }
    const int sh = 2 - ox + 5 * (2 - oy) + (DIM == 3 ? 25 * (2 - oz) : 0);
    m0 |= box << sh;
    if (DIM == 3 && sh) m1 |= box >> (64 - sh);
  }
  mask[2 * I] = m0;
  mask[2 * I + 1] = m1;
  row_nnzb[I] = __popcll(m0) + __popcll(m1);
}

// A lane per window bit of a row (128 a row in 3D, 32 in 2D): consecutive lanes write consecutive
// columns (139,425 rows: 101 -> 44 us; a thread per row before).
template <int DIM>
__global__ void __launch_bounds__(256) k_pattern_fill(gm_grid g, const uint64_t* mask, const int* row_ptr,
                                                      int* col_idx) {
  constexpr int LANES = DIM == 3 ? 128 : 32, W = DIM == 3 ? 125 : 25;
  const int I = blockIdx.x * (256 / LANES) + threadIdx.x / LANES, bit = threadIdx.x % LANES;
  if (I >= g.n_nodes || bit >= W) return;
  const uint64_t m0 = mask[2 * I], m1 = mask[2 * I + 1];
  if (!(((bit < 64 ? m0 : m1) >> (bit & 63)) & 1ull)) return;
  const uint64_t low = (1ull << (bit & 63)) - 1ull;
  const int below = bit < 64 ? __popcll(m0 & low) : __popcll(m0) + __popcll(m1 & low);
  const int nx1 = g.nx + 1, nxy = nx1 * (g.ny + 1);
  col_idx[row_ptr[I] + below] = I + bit % 5 - 2 + (bit / 5 % 5 - 2) * nx1 + (DIM == 3 ? (bit / 25 - 2) * nxy : 0);
}

// Row masks from the bins' support-shape sets (1, the default) or particle by particle (0).
static int g_pattern_by_sets = 1;

extern "C" int gm_pattern_kernel(int by_sets) {
  g_pattern_by_sets = by_sets ? 1 : 0;
  return 0;
}

// row_nnzb: n_nodes + 1 ints of scratch.  On return pat->nnzb holds the block count
// (one host synchronisation, once per load step).
extern "C" int gm_bsr_pattern(const gm_grid* g, const gm_bins* b, gm_pattern* pat, int* row_nnzb,
                              int max_nnzb, hipStream_t s) {
  GM_REQUIRE(g && b && pat, "gm_bsr_pattern: null argument");
  int n = g->n_nodes;
  if (g_pattern_by_sets) {
    // the bins' support-shape sets in the binning's scratch counts (free once the particles are sorted)
    k_bin_extset<<<gm_blocks(n, 256), 256, 0, s>>>(n, b->cell_start, b->ext_s, b->cell_count);
    if (g->dim == 2)
      k_pattern_count_sets<2><<<gm_blocks(n, 128), 128, 0, s>>>(*g, b->cell_count, pat->row_mask, row_nnzb);
    else
      k_pattern_count_sets<3><<<gm_blocks(n, 128), 128, 0, s>>>(*g, b->cell_count, pat->row_mask, row_nnzb);
  } else if (g->dim == 2) {
    k_pattern_count<2><<<gm_blocks(n, 128), 128, 0, s>>>(*g, b->cell_start, b->ext_s, pat->row_mask, row_nnzb);
  } else {
    k_pattern_count<3><<<gm_blocks(n, 128), 128, 0, s>>>(*g, b->cell_start, b->ext_s, pat->row_mask, row_nnzb);
  }
  GM_LAUNCH_CHECK();
  int rc = exclusive_scan(row_nnzb, pat->row_ptr, n, b->scan_tmp, s);
  if (rc) return rc;
  int nnzb = 0;
  GM_HIP(hipMemcpyAsync(&nnzb, pat->row_ptr + n, sizeof(int), hipMemcpyDeviceToHost, s));
  GM_HIP(hipStreamSynchronize(s));
  pat->nnzb = nnzb;
  if (nnzb > max_nnzb) {
    gm::set_error("gm_bsr_pattern: pattern needs %d blocks, capacity %d", nnzb, max_nnzb);
    return -4;
  }
  if (g->dim == 2)
    k_pattern_fill<2><<<gm_blocks(n, 8), 256, 0, s>>>(*g, pat->row_mask, pat->row_ptr, pat->col_idx);
  else
    k_pattern_fill<3><<<gm_blocks(n, 2), 256, 0, s>>>(*g, pat->row_mask, pat->row_ptr, pat->col_idx);
  GM_LAUNCH_CHECK();
  return 0;
}

// ================================================================== particle stage
// Rows of W values, one a lane, to and from memory through the wave's LDS tile, so that
// consecutive lanes touch consecutive values (a lane writing its own row of 9 to 17 doubles
// touches a cache line a lane and store).  Every lane of the wave takes part; the first `n` lanes
// have a row.
template <typename T>
struct WaveRows {
  T* tile;
  int lane, n;
  static __device__ __forceinline__ void sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  template <int W>
  __device__ __forceinline__ void put(const double* v) {
    sync();
#pragma unroll
    for (int i = 0; i < W; ++i) tile[lane * (W | 1) + i] = (T)v[i];
    sync();
  }
  // lane l's row to row index(l) of an array of W values a row
  template <int W>
  __device__ __forceinline__ void store(T* base, int row, const double* v) {
    put<W>(v);
#pragma unroll
    for (int i = 0; i < W; ++i) {
      const int q = i * 64 + lane, l = q / W, e = q % W;
      const long r = __shfl(row, l, 64);
      if (l < n) base[r * W + e] = tile[l * (W | 1) + e];
    }
  }
  // the first w of the tile's W values a lane (at stride W | 1) to base + lane * stride
  template <int W>
  __device__ __forceinline__ void flush(T* base, int stride, int w) {
#pragma unroll
    for (int i = 0; i < W; ++i) {
      const int q = i * 64 + lane, l = q / W, e = q % W;
      if (l < n && e < w) base[l * stride + e] = tile[l * (W | 1) + e];
    }
  }
  // the same with P >= W lanes a row, a power of two: the steps differ by constants, where flush has a
  // place of its own for every step, W registers that the tangent's terms need
  template <int W, int P, int STRIDE>
  __device__ __forceinline__ void flush_padded(T* base, int w) {
    const int l0 = lane / P, e = lane % P;
    const T* t = tile + l0 * (W | 1) + e;
    const int at = l0 * STRIDE + e;
#pragma unroll
    for (int i = 0; i < P; ++i)
      if (l0 + i * (64 / P) < n && e < w) (base + i * (64 / P) * STRIDE)[at] = t[i * (64 / P) * (W | 1)];
  }
  // rows by index: the loads, then the exchange
  template <int W>
  __device__ __forceinline__ void load(const T* base, int row, T* t) {
#pragma unroll
    for (int i = 0; i < W; ++i) {
      const int q = i * 64 + lane, l = min(q / W, n - 1), e = q % W;
      t[i] = base[(long)__shfl(row, l, 64) * W + e];
    }
  }
  template <int W>
  __device__ __forceinline__ void take(const T* t, double* v) {
    sync();
#pragma unroll
    for (int i = 0; i < W; ++i) {
      const int q = i * 64 + lane;
      tile[q / W * (W | 1) + q % W] = t[i];
    }
    sync();
#pragma unroll
    for (int i = 0; i < W; ++i) v[i] = (double)tile[lane * (W | 1) + i];
  }
};

// f(0), f(1), ...: the rows of the tangent, unrolled whatever their size
template <typename F, int... I>
__device__ __forceinline__ void each(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}

// One particle a lane, an instance a material (MAT): the return maps of the others would cost it
// registers.  The per-particle arrays and the rows of Y and D pass through LDS (WaveRows); D is
// formed row by row, R rows a pass of the tile (1 and 4 FP32 rows a pass: 658 and 763 us where 2
// take 672).  Bound by the memory traffic of those rows.  1,048,576 particles, a lane writing its
// own rows and D by columns before: 3D u-p Neo-Hookean 334 -> 265 us without the tangent, 1282 ->
// 672 with FP32 and 2404 -> 1024 with FP64 rows of D; 2D J2 220 -> 149 and 340 -> 229 us; 37,128
// particles of 3D Drucker-Prager 151 -> 73 us.  6,048 particles take the latency of one wavefront,
// 29 us (30).  Neo-Hookean rows sum the terms of the full product that are not zero, in its order and
// with its roundings (see k_update_lp).  Two waves a SIMD: with the register or two more that the
// compiler takes otherwise, one fits, and the stage without the tangent takes 352 us.
template <int DIM, bool COUPLED, typename TD, int MAT>
__global__ void __launch_bounds__(128, MAT == MAT_NEOHOOKEAN || (DIM == 2 && !COUPLED) ? 2 : 1) k_particle_stage(gm_grid g, gm_stage_args a) {
  typedef Lay<DIM, COUPLED> L;
  constexpr bool neo_hookean = MAT == MAT_NEOHOOKEAN;
  constexpr int NY = L::NY, NZ = L::NZ;
  constexpr int R = sizeof(TD) == 4 ? 2 : 1;  // rows of D a pass
  constexpr int CMAX = NY > 9 ? NY : 9;
  constexpr int TILE = 64 * (CMAX | 1) * 8 > 64 * (R * NZ | 1) * (int)sizeof(TD) ? 64 * (CMAX | 1) * 8
                                                                                 : 64 * (R * NZ | 1) * (int)sizeof(TD);
  __shared__ double tiles[2][TILE / 8];
  const int lane = threadIdx.x & 63, k0 = blockIdx.x * 128 + (threadIdx.x & 64);
  const int n = min(64, a.n_particles - k0);
  if (n <= 0) return;  // the whole wave
  const bool on = lane < n;
  const int kq = k0 + min(lane, n - 1);  // bin-sorted position: Y/D row
  const int p = a.sorted ? a.sorted[kq] : kq;  // particle id: state arrays
  WaveRows<double> rows{tiles[threadIdx.x >> 6], lane, n};
  double Ft[9], bt[9];
  rows.template load<9>(a.F_old, p, Ft);
  rows.template load<9>(a.b_old, p, bt);
  Axis ax[DIM];
  load_axes<DIM>(g, a.x, a.lp, p, ax);
  double H[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
  double dup[3] = {0, 0, 0};
  double pp = 0, ppo = 0, ppa = 0, ppoa = 0;
  double graw[3] = {0, 0, 0};
  const int NB = L::NB;
  // gather over the support, reference loop order (i outer ... k inner); the first two nodes of
  // the last axis, which every particle has, are loaded together
  auto load = [&](int i, int j, int k, double* un, double* uo) {
    const int c[3] = {ax[0].lo + i, ax[1].lo + j, DIM == 3 ? ax[2].lo + k : 0};
    const int node = node_index<DIM>(g, c);
#pragma unroll
    for (int cc = 0; cc < NB; ++cc) {
      un[cc] = a.u_new[node * NB + cc];
      uo[cc] = COUPLED ? a.u_old[node * NB + cc] : 0.0;
    }
  };
  auto add = [&](int i, int j, int k, const double* un, const double* uo) {
    const int o[3] = {i, j, k};
    double w, G[3], wa, du[3];
    node_geom<DIM>(ax, o, w, G, wa);
#pragma unroll
    for (int cc = 0; cc < DIM; ++cc) du[cc] = COUPLED ? un[cc] - uo[cc] : un[cc];
#pragma unroll
    for (int aa = 0; aa < DIM; ++aa)
#pragma unroll
      for (int cc = 0; cc < DIM; ++cc) H[aa][cc] += G[aa] * du[cc];
    if (COUPLED) {
#pragma unroll
      for (int cc = 0; cc < DIM; ++cc) dup[cc] += w * du[cc];
      const double pn = un[NB - 1], po = uo[NB - 1];
      pp += w * pn;
      ppo += w * po;
      ppa += wa * pn;
      ppoa += wa * po;
#pragma unroll
      for (int aa = 0; aa < DIM; ++aa) graw[aa] += G[aa] * pn;
    }
  };
  const int el = ax[DIM - 1].ext;
  for (int i = 0; i < ax[0].ext; ++i)
    for (int j = 0; j < (DIM == 3 ? ax[1].ext : 1); ++j) {
      auto at = [&](int k) { return DIM == 3 ? k : 0; };
      auto jt = [&](int k) { return DIM == 3 ? j : k; };
      double n0[NB], o0[NB], n1[NB], o1[NB];
      load(i, jt(0), at(0), n0, o0);
      load(i, jt(1), at(1), n1, o1);
      add(i, jt(0), at(0), n0, o0);
      add(i, jt(1), at(1), n1, o1);
      if (el == 3) {
        load(i, jt(2), at(2), n0, o0);
        add(i, jt(2), at(2), n0, o0);
      }
    }
  // kinematics: incr_F = I + delta_u_GRAD (mpm_utils.py:510-517, 1199-1206)
  M3 f = m3_eye();
#pragma unroll
  for (int aa = 0; aa < DIM; ++aa)
#pragma unroll
    for (int cc = 0; cc < DIM; ++cc) f.a[aa][cc] += H[aa][cc];
  M3 A;
  if (DIM == 2) {
    double d = f.a[0][0] * f.a[1][1] - f.a[0][1] * f.a[1][0];
    A = m3_eye();
    A.a[0][0] = f.a[1][1] / d;
    A.a[0][1] = -f.a[0][1] / d;
    A.a[1][0] = -f.a[1][0] / d;
    A.a[1][1] = f.a[0][0] / d;
  } else {
    A = m3_inv(f);
  }
  M3 Fo, bo;
  rows.template take<9>(Ft, &Fo.a[0][0]);
  rows.template take<9>(bt, &bo.a[0][0]);
  M3 Fn = m3_mul(f, Fo);
  double J = m3_det(Fn);
  double Jo = m3_det(Fo);
  M3 btr = m3_mul(f, m3_mul(bo, m3_T(f)));
  MatParams mp;
  mp.kind = MAT;
  mp.dp_apex = a.dp_apex;
  mp.lam = a.lam;
  mp.mu = a.mu;
  mp.E = a.E;
  mp.kappa = a.kappa;
  mp.H = a.H;
  mp.phi = a.p_phi ? a.p_phi[p] : a.phi;
  mp.psi = a.psi;
  mp.coh = a.p_coh ? a.p_coh[p] : a.coh;
  mp.shape = a.shape;
  mp.ns = a.ns;
  mp.lnJ = log(J);
  M3 tau, bn;
  SpectralState ss;
  double alpha_o = a.alpha_old ? a.alpha_old[p] : 0.0;
  double alpha_n = alpha_o;
  M3 sig;
  if constexpr (neo_hookean) {
    // sigma = mu/J (F F^T - I) + lambda/J ln J I (mpm_utils.py:915)
    M3 FFt = m3_mul(Fn, m3_T(Fn));
    double lnJ = log(J);
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        double id = (i == j) ? 1.0 : 0.0;
        sig.a[i][j] = a.mu / J * (FFt.a[i][j] - id) + a.lam / J * lnJ * id;
        tau.a[i][j] = sig.a[i][j] * J;
      }
    bn = btr;
  } else {
    hencky_family(btr, mp, alpha_o, ss, tau, bn, alpha_n);
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j) sig.a[i][j] = tau.a[i][j] / J;
  }
  rows.template store<9>(a.F_new, p, &Fn.a[0][0]);
  rows.template store<9>(a.b_new, p, &bn.a[0][0]);
  rows.template store<9>(a.sigma, p, &sig.a[0][0]);
  if (a.alpha_new && on) a.alpha_new[p] = alpha_n;

  // ---- particle stress vector Y
  double V = a.p_vol * J;
  double Y[L::NY];
  // P[b][c] = -V sum_a A[a][b] (sigma - p I)[a][c]    (rhs_value, mpm_utils.py:588, 994, 1271)
#pragma unroll
  for (int bb = 0; bb < DIM; ++bb)
#pragma unroll
    for (int cc = 0; cc < DIM; ++cc) {
      double s = 0.0;
#pragma unroll
      for (int aa = 0; aa < DIM; ++aa) s += A.a[aa][bb] * (sig.a[aa][cc] - ((COUPLED && aa == cc) ? pp : 0.0));
      Y[bb * DIM + cc] = -s * V;
    }
  double pen_z = 0.0;
  bool pen_in = false;
  if (!COUPLED) {
    // single phase: rho_new V_new g + f_ext (mpm_utils.py:564-571)
    double rho = a.p_rho / J;
    bool ef = a.ext_flag && a.ext_flag[p];
#pragma unroll
    for (int cc = 0; cc < DIM; ++cc) Y[L::Y_T + cc] = rho * a.gravity[cc] * V + (ef ? a.point_load[cc] : 0.0);
  } else {
    double npor = 1.0 - (1.0 - a.phi0) / J;
    double rho_mix = npor * 1.0 + (1.0 - npor) * a.p_rho;
#pragma unroll
    for (int cc = 0; cc < DIM; ++cc) Y[L::Y_T + cc] = rho_mix * a.gravity[cc] * V;
    if (DIM == 2) {
      bool ef = a.ext_flag && a.ext_flag[p];
      bool tf = a.trac_flag && a.trac_flag[p];
#pragma unroll
      for (int cc = 0; cc < DIM; ++cc)
        Y[L::Y_T + cc] += (ef ? a.point_load[cc] : 0.0) + (tf ? a.traction[cc] : 0.0);
    } else if (a.penalty) {
      // penalty indenter (mpm_utils.py:1235-1248)
      double xz = a.x[p * 3 + 2], xx = a.x[p * 3], xy = a.x[p * 3 + 1];
      if (xz >= a.footing_height && xx > a.footing[0] && xx < a.footing[1] && xy > a.footing[2] &&
          xy < a.footing[3]) {
        pen_in = true;
        double pen = a.footing_height - (xz + dup[2]);
        pen_z = -pen * a.pen_par;
        Y[L::Y_T + 2] += pen_z;
      }
    }
    if (a.pen_force && on) a.pen_force[p] = pen_in ? -pen_z : 0.0;
    // mass balance and PPP (mpm_utils.py:1006-1015, 1284-1294)
    double lnJ = log(J), lnJo = log(Jo);
    Y[L::Y_Q] = (lnJ - lnJo) * V;
    double gsp[3];
#pragma unroll
    for (int aa = 0; aa < DIM; ++aa) {
      if (DIM == 2) {
        double s = 0.0;
#pragma unroll
        for (int bb = 0; bb < DIM; ++bb) s += A.a[aa][bb] * graw[bb];
        gsp[aa] = s;  // spatial gradient in 2D (mpm_utils.py:933, 950)
      } else {
        gsp[aa] = graw[aa];  // material gradient in 3D (mpm_utils.py:1169, 1194)
      }
    }
#pragma unroll
    for (int bb = 0; bb < DIM; ++bb) {
      double s = 0.0;
#pragma unroll
      for (int aa = 0; aa < DIM; ++aa) s += A.a[aa][bb] * (a.mobility * gsp[aa]);
      Y[L::Y_M + bb] = s * a.dt * V;
    }
    double tau_s = 0.5 / a.mu;
    double cpp = (pp - ppa) - (ppo - ppoa);
    Y[L::Y_S] = tau_s * cpp * V;
  }
  rows.template put<NY>(Y);
  rows.template flush<NY>(a.Y + (long)k0 * NY, NY, NY);
  if (!a.want_tangent) return;

  // ---- tangent D = dY/dz, row by row (every entry exactly once)
  WaveRows<TD> drows{(TD*)tiles[threadIdx.x >> 6], lane, n};
  // M = tau - p J I; P = -V0 A^T M
  M3 Mm = tau;
  if (COUPLED)
#pragma unroll
    for (int i = 0; i < 3; ++i) Mm.a[i][i] -= pp * J;
  M3 AtM;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      double s = 0.0;
#pragma unroll
      for (int k = 0; k < DIM; ++k) s += A.a[k][i] * Mm.a[k][j];
      AtM.a[i][j] = s;
    }
  // d b = dH B + B^T dH^T: B = F_old F^T for Neo-Hookean (b = F F^T), b_old f^T for the Hencky family
  const M3 B = neo_hookean ? m3_mul(Fo, m3_T(Fn)) : m3_mul(bo, m3_T(f));
  // Hencky family: d tau of the symmetric unit tensors E_aj + E_ja (E_aa), pairs (0,0) (0,1) (0,2)
  // (1,1) (1,2) (2,2); S = d tau / d ln J (NorSand's return depends on the specific volume)
  constexpr int NP = DIM == 3 ? 6 : 5;
  M3 K[NP], S;
  if constexpr (!neo_hookean) {
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      const int pa = q < 3 ? 0 : (q < 5 ? 1 : 2), pj = q < 3 ? q : (q < 5 ? q - 2 : 2);
      M3 db = m3_zero();
      db.a[pa][pj] = db.a[pj][pa] = 1.0;
      K[q] = spectral_dtau(ss, db);
    }
    if constexpr (MAT == MAT_NORSAND)
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          double s = 0.0;
#pragma unroll
          for (int k = 0; k < 3; ++k) s += ss.V.a[i][k] * ss.TJ[k] * ss.V.a[j][k];
          S.a[i][j] = s;
        }
  }
  double lnJ = log(J), lnJo = log(Jo);
  // A^T A, A g, A^T g, A^T A g (mass-balance terms)
  double AtA[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
  double Ag[3] = {0, 0, 0}, Atg[3] = {0, 0, 0}, AtAg[3] = {0, 0, 0};
  if (COUPLED) {
#pragma unroll
    for (int i = 0; i < DIM; ++i) {
#pragma unroll
      for (int j = 0; j < DIM; ++j) {
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < DIM; ++k) s += A.a[k][i] * A.a[k][j];
        AtA[i][j] = s;
        Ag[i] += A.a[i][j] * graw[j];
        Atg[i] += A.a[j][i] * graw[j];
      }
    }
#pragma unroll
    for (int i = 0; i < DIM; ++i)
#pragma unroll
      for (int k = 0; k < DIM; ++k) AtAg[i] += A.a[k][i] * Ag[k];
  }
  // Neo-Hookean: the terms of d tau - p dJ I by column dH_ab that are not zero, d tau = mu (dH B + B^T
  // dH^T) + lambda tr(A dH) I: mu B off the diagonal, and on it with and without a term of mu B
  double mB[3][3], diag[3][3], both[3][3];
  if constexpr (neo_hookean) {
#pragma unroll
    for (int bb = 0; bb < DIM; ++bb)
#pragma unroll
      for (int aa = 0; aa < DIM; ++aa) {
        const double t = a.lam * A.a[bb][aa], u = fma(a.mu, B.a[bb][aa] + B.a[bb][aa], t), dJ = J * A.a[bb][aa];
        mB[bb][aa] = a.mu * B.a[bb][aa];
        diag[bb][aa] = COUPLED ? fma(-pp, dJ, t) : t;
        both[bb][aa] = COUPLED ? fma(-pp, dJ, u) : u;
      }
  }
  const double kdt = a.mobility * a.dt * a.p_vol, kdtJ = kdt * J, ts = 0.5 / a.mu * a.p_vol * J;
  TD* D = (TD*)a.D + (long)k0 * NY * NZ;
  each([&](auto index) {
    constexpr int y = decltype(index)::value;
    double row[NZ];
#pragma unroll
    for (int z = 0; z < NZ; ++z) row[z] = 0.0;
    if (y < L::NH) {
      // dP = -V0 [ dA^T M + A^T (dtau - p dJ I) ],  (dA^T X)[i][c] = -A[b][i] (A^T X)[a][c]
      const int i = y / DIM, c = y % DIM;
      double T[DIM][3], ab = 0.0;  // Hencky family: A^T d tau by (a, j)
      if constexpr (!neo_hookean) {
#pragma unroll
        for (int aa = 0; aa < DIM; ++aa)
#pragma unroll
          for (int j = 0; j < 3; ++j) {
            const int lo = aa < j ? aa : j, hi = aa < j ? j : aa, q = lo == 0 ? hi : (lo == 1 ? hi + 2 : 5);
            double s = 0.0;
#pragma unroll
            for (int k = 0; k < DIM; ++k) s += A.a[k][i] * K[q].a[k][c];
            T[aa][j] = aa == j ? 2.0 * s : s;
          }
        if constexpr (MAT == MAT_NORSAND)
#pragma unroll
          for (int k = 0; k < DIM; ++k) ab += A.a[k][i] * S.a[k][c];
      }
#pragma unroll
      for (int aa = 0; aa < DIM; ++aa)
#pragma unroll
        for (int bb = 0; bb < DIM; ++bb) {  // column dH_ab
          const double dJ = J * A.a[bb][aa];
          double t2 = 0.0;
          if constexpr (neo_hookean) {
            // in the order and with the roundings of the full product (see k_update_lp)
#pragma unroll
            for (int k = 0; k < DIM; ++k) {
              if (k != aa && c != aa && k != c) continue;
              t2 = fma(A.a[k][i], k != c ? mB[bb][k == aa ? c : k] : (c == aa ? both[bb][aa] : diag[bb][aa]), t2);
            }
          } else {
            t2 = ab * A.a[bb][aa];
#pragma unroll
            for (int j = 0; j < 3; ++j) t2 += T[aa][j] * B.a[bb][j];
            if (COUPLED) t2 -= A.a[c][i] * pp * dJ;
          }
          row[aa * DIM + bb] = -a.p_vol * fma(-A.a[bb][i], AtM.a[aa][c], t2);
        }
      if constexpr (COUPLED) row[L::Z_P] = a.p_vol * J * A.a[c][i];  // dP/dp = V0 J A^T
    } else if constexpr (COUPLED) {
#pragma unroll
      for (int aa = 0; aa < DIM; ++aa)
#pragma unroll
        for (int bb = 0; bb < DIM; ++bb) {
          const double dJ = J * A.a[bb][aa];
          double v = 0.0;
          if (y < L::Y_Q) {
            v = a.gravity[y - L::Y_T] * a.p_vol * dJ;
          } else if (y == L::Y_Q) {
            v = a.p_vol * (1.0 + lnJ - lnJo) * dJ;
          } else if (y < L::Y_S) {
            const int i = y - L::Y_M;
            if (DIM == 3) {
              // m = kdt J A^T g
              v = kdt * (J * (-A.a[bb][i] * Atg[aa]) + dJ * Atg[i]);
            } else {
              // m = kdt J A^T A g ; d(A^T A g) = dA^T (A g) + A^T (dA g), (dA g)[k] = -A[k][a] (A g)[b]
              double dAtAg = -A.a[bb][i] * AtAg[aa];
              double AtdAg = 0.0;
#pragma unroll
              for (int k = 0; k < DIM; ++k) AtdAg += A.a[k][i] * (-A.a[k][aa] * Ag[bb]);
              v = kdt * (dJ * AtAg[i] + J * (dAtAg + AtdAg));
            }
          } else {
            v = Y[L::Y_S] * A.a[bb][aa];
          }
          row[aa * DIM + bb] = v;
        }
      if (DIM == 3 && y == L::Y_T + 2 && pen_in) row[L::Z_DU] = a.pen_par;  // 3D indenter penalty
      if (y == L::Y_S) {
        row[L::Z_P] = ts;
        row[L::Z_PB] = -ts;
      }
      // dm/dg = kdt J A^T (3D) or kdt J A^T A (2D)
      if (y >= L::Y_M && y < L::Y_S)
#pragma unroll
        for (int k = 0; k < DIM; ++k) row[L::Z_G + k] = kdtJ * (DIM == 3 ? A.a[k][y - L::Y_M] : AtA[y - L::Y_M][k]);
    }
    constexpr int W = R * NZ, TS = W | 1, P = W <= 4 ? 4 : W <= 8 ? 8 : W <= 16 ? 16 : 32;
    static_assert(W <= P, "a row fits its lanes");
    const int slot = y % R;
    if (slot == 0) drows.sync();
#pragma unroll
    for (int z = 0; z < NZ; ++z) drows.tile[lane * TS + slot * NZ + z] = (TD)row[z];
    if (slot == R - 1 || y == NY - 1) {
      drows.sync();
      drows.template flush_padded<W, P, NY * NZ>(D + (y - slot) * NZ, (slot + 1) * NZ);
    }
  }, std::make_integer_sequence<int, NY>{});
}

extern "C" int gm_particle_stage(const gm_grid* g, const gm_stage_args* a, hipStream_t s) {
  GM_REQUIRE(g && a, "gm_particle_stage: null argument");
  int n = a->n_particles;
  if (n == 0) return 0;
  GM_REQUIRE(!a->want_tangent || a->D, "gm_particle_stage: tangent requested without D");
  int blk = gm_blocks(n, 128);
#define GM_STAGE_M(D, C, M)                                                                       \
  do {                                                                                           \
    if (a->tangent_fp32) k_particle_stage<D, C, float, M><<<blk, 128, 0, s>>>(*g, *a);            \
    else k_particle_stage<D, C, double, M><<<blk, 128, 0, s>>>(*g, *a);                           \
  } while (0)
#define GM_STAGE(D, C)                                                  \
  do {                                                                 \
    switch (a->mat_kind) {                                             \
      case MAT_NEOHOOKEAN: GM_STAGE_M(D, C, MAT_NEOHOOKEAN); break;    \
      case MAT_J2: GM_STAGE_M(D, C, MAT_J2); break;                    \
      case MAT_DP: GM_STAGE_M(D, C, MAT_DP); break;                    \
      case MAT_NORSAND: GM_STAGE_M(D, C, MAT_NORSAND); break;          \
      default: GM_STAGE_M(D, C, MAT_HENCKY);                           \
    }                                                                  \
  } while (0)
  if (g->dim == 2 && !a->coupled) {
    GM_STAGE(2, false);
  } else if (g->dim == 2 && a->coupled) {
    GM_STAGE(2, true);
  } else if (g->dim == 3 && a->coupled) {
    GM_STAGE(3, true);
  } else {
    gm::set_error("gm_particle_stage: 3D single-phase is not a supported form");
    return -1;
  }
#undef GM_STAGE
#undef GM_STAGE_M
  GM_LAUNCH_CHECK();
  return 0;
}

// ================================================================== 2D strips
// Residual and Jacobian of the 2D forms, gathered by strips of consecutive node rows.  A
// workgroup has a wave per stencil line oy: the bins that hold the strip's candidates in line
// y - oy are consecutive, and so are their particles in bin order.  The wave stages that range
// a piece of C particles at a time in LDS (per-axis tables and particle rows, loaded once for
// the strip; odd strides, so that particles a few apart lie on different banks), every lane
// walks the particles of its row's three bins, and the lines' sums are added in the order
// oy = 0, 1, 2.  Workgroups of one XCD take consecutive strips: the three lines that read a
// particle find it in that XCD's L2.
template <bool COUPLED, typename TY, int ROWS, int NR, int C>
struct Strip2d {
  typedef Lay<2, COUPLED> L;
  static constexpr int NT = COUPLED ? 9 : 6;  // per axis: w, g (, wa)
  static constexpr int TS = 2 * NT | 1, RS = NR | 1;
  struct Piece {
    double t[C * TS];
    TY r[C * RS];
    uint8_t ext[C];
  };

  static __device__ __forceinline__ int first_row() {
    const int n = gridDim.x, b = blockIdx.x, q = n / 8, r = n % 8, x = b % 8;
    return (x * q + min(x, r) + b / 8) * ROWS;
  }
  // particles of the bins of line oy that strip rows [I0, I0 + ROWS) reach
  static __device__ __forceinline__ void range(const gm_grid& g, int I0, int oy, const int* cell_start, int* lo,
                                               int* hi) {
    const int o = oy * (g.nx + 1);
    const int b0 = max(I0 - 2 - o, 0), b1 = min(I0 + ROWS, g.n_nodes) - 1 - o;
    *lo = b1 >= b0 ? cell_start[b0] : 0;
    *hi = b1 >= b0 ? cell_start[b1 + 1] : 0;
  }
  // a row's candidates in line oy: the particles of bins (x - ox, y - oy), none where the row
  // or the bin is off the grid
  static __device__ __forceinline__ void bins(const gm_grid& g, int I, bool on, int oy, const int* cell_start, int* ks,
                                              int* ke) {
    const int nx1 = g.nx + 1, cx = I % nx1, cy = I / nx1;
#pragma unroll
    for (int ox = 0; ox < 3; ++ox) {
      const bool ok = on && cx >= ox && cy >= oy;
      const int b = I - ox - oy * nx1;
      ks[ox] = ok ? cell_start[b] : 0;
      ke[ox] = ok ? cell_start[b + 1] : 0;
    }
  }
  // a split's first particle of a bin that starts at ks, in the piece that starts at k0
  static __device__ __forceinline__ int first(int ks, int k0, int split, int n) {
    const int k = ks + split;  // then every n-th
    return k >= k0 ? k - k0 : (n - (k0 - k) % n) % n;
  }
  // particles [k0, k0 + n) into the wave's piece
  static __device__ __forceinline__ void stage(const gm_grid& g, const double* x_s, const double* lp_s,
                                               const uint8_t* ext_s, const TY* rows, int k0, int n, Piece& p) {
    const int lane = threadIdx.x & 63, last = n * NR - 1;
    const TY* src = rows + (long)k0 * NR;
    for (int q0 = 0; q0 <= last; q0 += 64 * 6) {
      TY v[6];
#pragma unroll
      for (int j = 0; j < 6; ++j) v[j] = src[min(q0 + j * 64 + lane, last)];
#pragma unroll
      for (int j = 0; j < 6; ++j) {
        const int q = q0 + j * 64 + lane;
        if (q <= last) p.r[q / NR * RS + q % NR] = v[j];
      }
    }
    for (int q = lane; q < 2 * n; q += 64) {
      const int a = q & 1;
      const long i = 2 * (long)k0 + q;
      const Axis ax = gimp_axis(x_s[i], lp_s[i], a ? g.h[1] : g.h[0], a ? g.inv_h[1] : g.inv_h[0]);
      double* t = p.t + (q >> 1) * TS + a * NT;
#pragma unroll
      for (int i3 = 0; i3 < 3; ++i3) {
        t[i3] = ax.w[i3];
        t[3 + i3] = ax.g[i3];
        if (COUPLED) t[6 + i3] = ax.wa[i3];
      }
    }
    if (lane < n) p.ext[lane] = ext_s[k0 + lane];
  }
  // orders the wave's LDS traffic between the stages (the piece belongs to one wave)
  static __device__ __forceinline__ void sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
};

// A lane per (row, dof, every fourth particle).  Bound by the staging of the particles' rows: a
// thread per row walked the nine bins in global memory and evaluated every particle's axis data
// nine times.  Strips of 8 rows (5 u-p), so that a piece of 40 particles holds a line's range and
// no lane waits for its bins: 32 (21) rows with pieces of 56 (40) and a lane for all of a bin's
// particles take 98 and 20 us where this takes 94 and 10, 16 rows with two lanes 109 and 12, 4
// with seven 130 and 12.  1,048,576 particles, 264,000 rows, single phase: 281 -> 94 us; 45,000
// particles u-p: 32 -> 10 us.  (The Jacobian gains nothing from it: see below.)
constexpr int RES_ROWS = 8, RES_ROWS_UP = 5, RES_SPLIT = 4, RES_C = 40;

template <bool COUPLED>
__global__ void __launch_bounds__(192) k_strip_residual(gm_grid g, const double* x_s, const double* lp_s,
                                                        const int* cell_start, const uint8_t* ext_s, const double* Y,
                                                        const uint8_t* freem, double* rhs) {
  typedef Lay<2, COUPLED> L;
  constexpr int NB = L::NB, NY = L::NY, ROWS = COUPLED ? RES_ROWS_UP : RES_ROWS, SPLIT = RES_SPLIT, C = RES_C;
  typedef Strip2d<COUPLED, double, ROWS, NY, C> S;
  constexpr int NT = S::NT;
  __shared__ typename S::Piece piece[3];
  __shared__ double OUT[3][ROWS * NB];
  constexpr int PART = ROWS * NB;  // lanes of a split
  const int lane = threadIdx.x & 63, split = lane / PART, row = lane % PART / NB, c = lane % PART % NB;
  const int I0 = S::first_row(), I = I0 + row;
  const int oy = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  typename S::Piece& p = piece[oy];
  int lo, hi, ks[3], ke[3];
  S::range(g, I0, oy, cell_start, &lo, &hi);
  S::bins(g, I, split < SPLIT && I < g.n_nodes, oy, cell_start, ks, ke);
  // the dof's rows of Y
  const int y0 = c < 2 ? c : L::Y_M, y1 = c < 2 ? 2 + c : L::Y_M + 1, y2 = c < 2 ? L::Y_T + c : L::Y_Q;
  double acc = 0.0;
  for (int k0 = lo; k0 < hi; k0 += C) {
    S::sync();
    S::stage(g, x_s, lp_s, ext_s, Y, k0, min(C, hi - k0), p);
    S::sync();
#pragma unroll
    for (int ox = 0; ox < 3; ++ox)
      for (int k = S::first(ks[ox], k0, split, SPLIT); k < min(ke[ox] - k0, C); k += SPLIT) {
        const uint8_t ex = p.ext[k];
        if ((ox == 2 && !(ex & 1)) || (oy == 2 && !(ex & 2))) continue;  // outside the particle's support
        const double *tx = p.t + k * S::TS, *ty = tx + NT, *yp = p.r + k * S::RS;
        const double wx = tx[ox], wy = ty[oy], w = wx * wy;
        acc += tx[3 + ox] * wy * yp[y0] + wx * ty[3 + oy] * yp[y1] + w * yp[y2];
        if constexpr (COUPLED)
          if (c == 2) acc += (w - tx[6 + ox] * ty[6 + oy]) * yp[L::Y_S];
      }
  }
  double sum = acc;
#pragma unroll
  for (int k = 1; k < SPLIT; ++k) sum += __shfl(acc, (lane + k * PART) & 63, 64);
  if (split == 0) OUT[oy][lane] = sum;
  __syncthreads();
  if (oy == 0 && split == 0 && I < g.n_nodes) {
    const long d = (long)I * NB + c;
    rhs[d] = freem[d] ? OUT[0][lane] + OUT[1][lane] + OUT[2][lane] : 0.0;
  }
}

// A lane per (row, row dof, column dof): its two E entries come from the lane's own two columns
// of D, and the 15 sums a line fit in registers.  Bound by the LDS reads of the 36 candidates
// (18 values a candidate and lane) and by the 15 wavefronts a CU that the pieces' LDS leaves:
// pieces of 24, 40 and 56 FP64 rows took 407, 407 and 497 us against 378 with 32; 40 FP32 rows
// 298 us.  8 rows with two lanes for a bin's particles and a line's whole range in one piece: 439
// and 276 us (an eighth more particles staged, and twice the workgroups' start and output).  One
// wavefront per row, lanes over its 25 blocks and one particle after the other,
// took 2750 us FP64 and 2709 us FP32 (1,048,576 particles, 264,000 rows; 210 MB of matrix and
// 201 MB of D); u-p with 11,628 rows 135 -> 69 us.
template <bool COUPLED, typename TD, typename TV>
__global__ void __launch_bounds__(192) k_strip_jacobian(gm_grid g, const double* x_s, const double* lp_s,
                                                        const int* cell_start, const uint8_t* ext_s, const TD* D,
                                                        const uint8_t* freem, const int* row_ptr,
                                                        const uint64_t* row_mask, TV* vals) {
  typedef Lay<2, COUPLED> L;
  constexpr int NB = L::NB, NB2 = NB * NB, NY = L::NY, NZ = L::NZ, ROWS = 64 / NB2, C = COUPLED ? 16 : sizeof(TD) == 4 ? 40 : 32;
  typedef Strip2d<COUPLED, TD, ROWS, NY * NZ, C> S;
  constexpr int NT = S::NT, RV = 25 * NB2, OS = RV | 1;
  union Shared {
    typename S::Piece piece[3];
    double out[ROWS * OS];
  };
  __shared__ Shared sh;
  const int lane = threadIdx.x & 63, row = lane / NB2, r = lane % NB2 / NB, c = lane % NB;
  const int I0 = S::first_row(), I = I0 + row;
  const int oy = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  typename S::Piece& p = sh.piece[oy];
  int lo, hi, ks[3], ke[3];
  S::range(g, I0, oy, cell_start, &lo, &hi);
  S::bins(g, I, row < ROWS && I < g.n_nodes, oy, cell_start, ks, ke);
  // the dof's rows of L_I and columns of D
  const int y0 = (r < 2 ? r : L::Y_M) * NZ, y1 = (r < 2 ? 2 + r : L::Y_M + 1) * NZ,
            y2 = (r < 2 ? L::Y_T + r : L::Y_Q) * NZ;
  const int z0 = c < 2 ? c : L::Z_G, z1 = c < 2 ? 2 + c : L::Z_G + 1;
  double acc[3][5];  // [jy][dx + 2]
#pragma unroll
  for (int j = 0; j < 3; ++j)
#pragma unroll
    for (int d = 0; d < 5; ++d) acc[j][d] = 0.0;
  for (int k0 = lo; k0 < hi; k0 += C) {
    S::sync();
    S::stage(g, x_s, lp_s, ext_s, D, k0, min(C, hi - k0), p);
    S::sync();
#pragma unroll
    for (int ox = 0; ox < 3; ++ox)
      for (int k = max(ks[ox], k0) - k0; k < min(ke[ox] - k0, C); ++k) {
        const uint8_t ex = p.ext[k];
        if ((ox == 2 && !(ex & 1)) || (oy == 2 && !(ex & 2))) continue;  // outside the particle's support
        const double *tx = p.t + k * S::TS, *ty = tx + NT;
        const TD* Dp = p.r + k * S::RS;
        const double wx = tx[ox], wy = ty[oy], w = wx * wy, g0 = tx[3 + ox] * wy, g1 = wx * ty[3 + oy];
        double wd = 0.0;
        if constexpr (COUPLED) wd = w - tx[6 + ox] * ty[6 + oy];
        // entries (r, z) of E = L_I D_p, then times M_J of the nine columns, one axis after the other
        auto E = [&](int z) {
          double e = g0 * (double)Dp[y0 + z] + g1 * (double)Dp[y1 + z] + w * (double)Dp[y2 + z];
          if constexpr (COUPLED)
            if (r == 2) e += wd * (double)Dp[L::Y_S * NZ + z];
          return e;
        };
        const double e0 = E(z0), e1 = E(z1);
#pragma unroll
        for (int jx = 0; jx < 3; ++jx) {
          const double u = e0 * tx[3 + jx], v = e1 * tx[jx];
#pragma unroll
          for (int jy = 0; jy < 3; ++jy) acc[jy][jx - ox + 2] += u * ty[jy] + v * ty[3 + jy];
        }
        if constexpr (COUPLED)
          if (c == 2) {
            const double ep = E(L::Z_P), eb = E(L::Z_PB);
#pragma unroll
            for (int jx = 0; jx < 3; ++jx) {
              const double u = ep * tx[jx], v = eb * tx[6 + jx];
#pragma unroll
              for (int jy = 0; jy < 3; ++jy) acc[jy][jx - ox + 2] += u * ty[jy] + v * ty[6 + jy];
            }
          }
      }
  }
  // the lines' sums, then masks, sign (the system matrix is -dR/du) and identity on fixed or
  // inactive dofs; consecutive threads write consecutive values of a row
  __syncthreads();
  for (int q = threadIdx.x; q < ROWS * OS; q += 192) sh.out[q] = 0.0;
  for (int o = 0; o < 3; ++o) {
    __syncthreads();
    if (oy == o && row < ROWS) {
      double* out = sh.out + row * OS + r * NB + c;
#pragma unroll
      for (int jy = 0; jy < 3; ++jy)
#pragma unroll
        for (int d = 0; d < 5; ++d) out[((jy - o + 2) * 5 + d) * NB2] += acc[jy][d];
    }
  }
  __syncthreads();
  const int nx1 = g.nx + 1;
  for (int q = threadIdx.x; q < ROWS * RV; q += 192) {
    const int rw = q / RV, e = q % RV, bit = e / NB2, rr = e % NB2 / NB, cc = e % NB, Ir = I0 + rw;
    if (Ir >= g.n_nodes) break;
    const uint64_t m = row_mask[2 * Ir];
    if (!((m >> bit) & 1ull)) continue;
    const int Jn = Ir + bit % 5 - 2 + (bit / 5 - 2) * nx1;
    const bool fr = freem[Ir * NB + rr], fc = freem[Jn * NB + cc];
    double v = (fr && fc) ? -sh.out[rw * OS + e] : 0.0;
    if (Jn == Ir && rr == cc && !fr) v = 1.0;
    vals[((long)row_ptr[Ir] + __popcll(m & ((1ull << bit) - 1ull))) * NB2 + rr * NB + cc] = (TV)v;
  }
}

// ================================================================== node residual
// 3D u-p, a thread per node (gm_node_residual_binned sums per bin)
__global__ void __launch_bounds__(128) k_node_residual(gm_grid g, const double* x_s, const double* lp_s,
                                                       const int* cell_start, const uint8_t* ext_s, const double* Y,
                                                       const uint8_t* freem, double* rhs) {
  typedef Lay<3, true> L;
  int I = blockIdx.x * blockDim.x + threadIdx.x;
  if (I >= g.n_nodes) return;
  int ci[3] = {0, 0, 0};
  node_coords<3>(g, I, ci);
  double r[L::NB];
#pragma unroll
  for (int k = 0; k < L::NB; ++k) r[k] = 0.0;
  for_candidates<3>(g, ci, cell_start, ext_s, [&](int k, const int* o, const int* b, bool in) {
    if (!in) return;
    Axis ax[3];
    load_axes<3>(g, x_s, lp_s, k, ax);
    double w, G[3], wa;
    node_geom<3>(ax, o, w, G, wa);
    const double* yp = Y + (long)k * L::NY;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      double s = 0.0;
#pragma unroll
      for (int bb = 0; bb < 3; ++bb) s += G[bb] * yp[bb * 3 + c];
      r[c] += s + w * yp[L::Y_T + c];
    }
    double s = w * yp[L::Y_Q];
#pragma unroll
    for (int bb = 0; bb < 3; ++bb) s += G[bb] * yp[L::Y_M + bb];
    s += (w - wa) * yp[L::Y_S];
    r[3] += s;
  });
#pragma unroll
  for (int k = 0; k < L::NB; ++k) rhs[I * L::NB + k] = freem[I * L::NB + k] ? r[k] : 0.0;
}

extern "C" int gm_node_residual(const gm_grid* g, const gm_bins* b, const double* Y, const uint8_t* freem,
                                double* rhs, int coupled, hipStream_t s) {
  GM_REQUIRE(g && b, "gm_node_residual: null argument");
  int n = g->n_nodes;
  int blk = gm_blocks(n, 128);
  if (g->dim == 2 && !coupled)
    k_strip_residual<false><<<gm_blocks(n, RES_ROWS), 192, 0, s>>>(*g, b->x_s, b->lp_s, b->cell_start, b->ext_s, Y, freem, rhs);
  else if (g->dim == 2)
    k_strip_residual<true><<<gm_blocks(n, RES_ROWS_UP), 192, 0, s>>>(*g, b->x_s, b->lp_s, b->cell_start, b->ext_s, Y, freem, rhs);
  else if (coupled)
    k_node_residual<<<blk, 128, 0, s>>>(*g, b->x_s, b->lp_s, b->cell_start, b->ext_s, Y, freem, rhs);
  else {
    gm::set_error("gm_node_residual: 3D single-phase is not a supported form");
    return -1;
  }
  GM_LAUNCH_CHECK();
  return 0;
}

// ================================================================== node Jacobian
// 3D u-p: one 64-lane wavefront per block row.  Lane l owns compressed slots l and l+64.
template <typename TD, typename TV>
__global__ void __launch_bounds__(64, 3) k_node_jacobian(gm_grid g, const double* x_s, const double* lp_s,
                                                      const int* cell_start, const uint8_t* ext_s, const TD* D,
                                                      const uint8_t* freem, const int* row_ptr,
                                                      const uint64_t* row_mask, TV* vals) {
  typedef Lay<3, true> L;
  const int NB = L::NB, NZ = L::NZ, NY = L::NY;
  // the particles of a bin are taken JB at a time: their axis data, support flags and
  // E = L_I D_p rows are formed in parallel, then every slot lane accumulates them in
  // bin order (the order and arithmetic of one-particle-at-a-time processing)
  constexpr int JB = 8;
  __shared__ double E[JB][NB * NZ];
  __shared__ Axis AX[JB][3];
  __shared__ int INS[JB];
  __shared__ uint8_t EXS[JB];
  int I = blockIdx.x;
  if (I >= g.n_nodes) return;
  int lane = threadIdx.x;
  int ci[3] = {0, 0, 0};
  node_coords<3>(g, I, ci);
  uint64_t m0 = row_mask[2 * I], m1 = row_mask[2 * I + 1];
  int nnz = __popcll(m0) + __popcll(m1);
  int rp = row_ptr[I];
  // window offsets of my two slots
  int myoff[2][3];
  bool has[2];
#pragma unroll
  for (int s2 = 0; s2 < 2; ++s2) {
    int slot = lane + 64 * s2;
    has[s2] = slot < nnz;
    myoff[s2][0] = myoff[s2][1] = myoff[s2][2] = 0;
    if (has[s2]) {
      int cnt = 0, bit = 0;
      for (bit = 0; bit < 125; ++bit) {
        uint64_t w = (bit < 64) ? m0 : m1;
        if ((w >> (bit & 63)) & 1ull) {
          if (cnt == slot) break;
          ++cnt;
        }
      }
      myoff[s2][0] = bit % 5 - 2;
      myoff[s2][1] = (bit / 5) % 5 - 2;
      myoff[s2][2] = bit / 25 - 2;
    }
  }
  double acc[2][NB * NB];
#pragma unroll
  for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
    for (int k = 0; k < NB * NB; ++k) acc[s2][k] = 0.0;

  int ncell[3] = {g.nx, g.ny, g.nz};
  for (int oz = 0; oz < 3; ++oz)
    for (int oy = 0; oy < 3; ++oy)
      for (int ox = 0; ox < 3; ++ox) {
        // base cell I - o: its particles have node I at stencil offset o (candidate walk order)
        int o[3] = {ox, oy, oz};
        int bc[3];
        bool ok = true;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          bc[a] = ci[a] - o[a];
          if (bc[a] < 0 || bc[a] > ncell[a]) ok = false;
        }
        if (!ok) continue;
        int bn = node_index<3>(g, bc);
        int ks = cell_start[bn], ke = cell_start[bn + 1];
        for (int k0 = ks; k0 < ke; k0 += JB) {
          const int nj = min(JB, ke - k0);
          if (lane < nj) {
            int k = k0 + lane;
            uint8_t ex = ext_s[k];
            bool in = true;
#pragma unroll
            for (int a = 0; a < 3; ++a) in = in && (o[a] < (((ex >> a) & 1) ? 3 : 2));
            INS[lane] = in ? 1 : 0;
            EXS[lane] = ex;
            Axis ax[3];
            load_axes<3>(g, x_s, lp_s, k, ax);
#pragma unroll
            for (int a = 0; a < 3; ++a) AX[lane][a] = ax[a];
          }
          __syncthreads();
          // E = L_I D_p  (NB x NZ) for each particle of the batch
          for (int q = lane; q < nj * NB * NZ; q += 64) {
            int pj = q / (NB * NZ), qq = q % (NB * NZ);
            if (!INS[pj]) continue;
            double wI, GI[3], waI;
            node_geom<3>(AX[pj], o, wI, GI, waI);
            const TD* Dp = D + (long)(k0 + pj) * NY * NZ;
            int r = qq / NZ, z = qq % NZ;
            double sE = 0.0;
            if (r < 3) {
#pragma unroll
              for (int bb = 0; bb < 3; ++bb) sE += GI[bb] * (double)Dp[(bb * 3 + r) * NZ + z];
              sE += wI * (double)Dp[(L::Y_T + r) * NZ + z];
            } else {
              sE = wI * (double)Dp[L::Y_Q * NZ + z];
#pragma unroll
              for (int bb = 0; bb < 3; ++bb) sE += GI[bb] * (double)Dp[(L::Y_M + bb) * NZ + z];
              sE += (wI - waI) * (double)Dp[L::Y_S * NZ + z];
            }
            E[pj][qq] = sE;
          }
          __syncthreads();
          for (int pj = 0; pj < nj; ++pj) {
            if (!INS[pj]) continue;  // uniform across the workgroup
#pragma unroll
            for (int s2 = 0; s2 < 2; ++s2) {
              if (!has[s2]) continue;
              int oJ[3];
              bool inJ = true;
#pragma unroll
              for (int aa = 0; aa < 3; ++aa) {
                oJ[aa] = o[aa] + myoff[s2][aa];  // offset of J inside this particle's stencil
                int e = ((EXS[pj] >> aa) & 1) ? 3 : 2;
                inJ = inJ && (oJ[aa] >= 0) && (oJ[aa] < e);
              }
              if (!inJ) continue;
              double wJ, GJ[3], waJ;
              node_geom<3>(AX[pj], oJ, wJ, GJ, waJ);
#pragma unroll
              for (int r = 0; r < NB; ++r) {
#pragma unroll
                for (int e = 0; e < 3; ++e) {
                  double sv = 0.0;
#pragma unroll
                  for (int aa = 0; aa < 3; ++aa) sv += E[pj][r * NZ + aa * 3 + e] * GJ[aa];
                  if (e == 2) sv += E[pj][r * NZ + L::Z_DU] * wJ;
                  acc[s2][r * NB + e] += sv;
                }
                double sv = E[pj][r * NZ + L::Z_P] * wJ + E[pj][r * NZ + L::Z_PB] * waJ;
#pragma unroll
                for (int aa = 0; aa < 3; ++aa) sv += E[pj][r * NZ + L::Z_G + aa] * GJ[aa];
                acc[s2][r * NB + 3] += sv;
              }
            }
          }
          __syncthreads();
        }
      }
  // masks, sign (the system matrix is -dR/du) and identity on fixed/inactive dofs
#pragma unroll
  for (int s2 = 0; s2 < 2; ++s2) {
    if (!has[s2]) continue;
    int cj[3] = {ci[0] + myoff[s2][0], ci[1] + myoff[s2][1], ci[2] + myoff[s2][2]};
    int Jn = node_index<3>(g, cj);
    bool diag = (Jn == I);
    TV* out = vals + (long)(rp + lane + 64 * s2) * NB * NB;
#pragma unroll
    for (int r = 0; r < NB; ++r) {
      bool fr = freem[I * NB + r];
#pragma unroll
      for (int c = 0; c < NB; ++c) {
        bool fc = freem[Jn * NB + c];
        double v = (fr && fc) ? -acc[s2][r * NB + c] : 0.0;
        if (diag && r == c && !fr) v = 1.0;
        out[r * NB + c] = (TV)v;
      }
    }
  }
}

// 3D u-p node Jacobian: one 128-lane workgroup per block row I.  The candidate
// particles of row I come in 27 base bins b = I - o; every particle of bin o
// reaches the same 3x3x3 box of columns J = b + k, so lane (k, c) (108 of 128
// lanes: 27 columns x 4 column dofs) owns entry column c of block (I, b + k) for
// the whole bin and adds the bin's particles to it in bin order.  The row's 125
// window blocks are accumulated in LDS (window-bit order), loaded into registers
// per bin and stored back, so every entry receives the same sums in the same
// order as in the one-wavefront-per-row form (k_node_jacobian) -- bit for bit the
// same matrix -- while no lane waits on columns outside the particle's support.
template <typename TD, typename TV>
__global__ void __launch_bounds__(128) k_node_jacobian_up3(gm_grid g, const double* x_s, const double* lp_s,
                                                           const int* cell_start, const uint8_t* ext_s,
                                                           const TD* D, const uint8_t* freem, const int* row_ptr,
                                                           const uint64_t* row_mask, TV* vals) {
  typedef Lay<3, true> L;
  constexpr int NB = 4, NZ = L::NZ, NY = L::NY, T = 128, JB = 8;
  __shared__ double ACC[125 * NB * NB];
  __shared__ double E[JB][NB * NZ];
  __shared__ Axis AX[JB][3];
  __shared__ int INS[JB];
  __shared__ uint8_t EXS[JB];
  const int I = blockIdx.x;
  if (I >= g.n_nodes) return;
  const int t = threadIdx.x;
  for (int q = t; q < 125 * NB * NB; q += T) ACC[q] = 0.0;
  int ci[3];
  node_coords<3>(g, I, ci);
  const int kk = t >> 2, c = t & 3;
  const int kx = kk % 3, ky = (kk / 3) % 3, kz = kk / 9;
  const bool lane_on = t < 27 * NB;
  const int ncell[3] = {g.nx, g.ny, g.nz};
  __syncthreads();
  for (int oz = 0; oz < 3; ++oz)
    for (int oy = 0; oy < 3; ++oy)
      for (int ox = 0; ox < 3; ++ox) {
        const int o[3] = {ox, oy, oz};
        int bc[3];
        bool ok = true;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          bc[a] = ci[a] - o[a];
          if (bc[a] < 0 || bc[a] > ncell[a]) ok = false;
        }
        if (!ok) continue;  // uniform across the workgroup
        const int bn = node_index<3>(g, bc);
        const int ks = cell_start[bn], ke = cell_start[bn + 1];
        // window bit of column J = b + k in row I (offset k - o per axis)
        const int bit = (kx - ox + 2) + 5 * (ky - oy + 2) + 25 * (kz - oz + 2);
        for (int k0 = ks; k0 < ke; k0 += JB) {
          const int nj = min(JB, ke - k0);
          if (t < nj) {
            const int k = k0 + t;
            const uint8_t ex = ext_s[k];
            bool in = true;
#pragma unroll
            for (int a = 0; a < 3; ++a) in = in && (o[a] < (((ex >> a) & 1) ? 3 : 2));
            INS[t] = in ? 1 : 0;
            EXS[t] = ex;
            Axis ax[3];
            load_axes<3>(g, x_s, lp_s, k, ax);
#pragma unroll
            for (int a = 0; a < 3; ++a) AX[t][a] = ax[a];
          }
          __syncthreads();
          // E = L_I D_p (NB x NZ) of each particle of the batch (same expressions as k_node_jacobian)
          for (int q = t; q < nj * NB * NZ; q += T) {
            const int pj = q / (NB * NZ), qq = q % (NB * NZ);
            if (!INS[pj]) continue;
            double wI, GI[3], waI;
            node_geom<3>(AX[pj], o, wI, GI, waI);
            const TD* Dp = D + (long)(k0 + pj) * NY * NZ;
            const int r = qq / NZ, z = qq % NZ;
            double sE = 0.0;
            if (r < 3) {
#pragma unroll
              for (int bb = 0; bb < 3; ++bb) sE += GI[bb] * (double)Dp[(bb * 3 + r) * NZ + z];
              sE += wI * (double)Dp[(L::Y_T + r) * NZ + z];
            } else {
              sE = wI * (double)Dp[L::Y_Q * NZ + z];
#pragma unroll
              for (int bb = 0; bb < 3; ++bb) sE += GI[bb] * (double)Dp[(L::Y_M + bb) * NZ + z];
              sE += (wI - waI) * (double)Dp[L::Y_S * NZ + z];
            }
            E[pj][qq] = sE;
          }
          __syncthreads();
          if (lane_on) {
            double acc[NB];
#pragma unroll
            for (int r = 0; r < NB; ++r) acc[r] = ACC[bit * NB * NB + r * NB + c];
            const int kJ[3] = {kx, ky, kz};
            for (int pj = 0; pj < nj; ++pj) {
              if (!INS[pj]) continue;
              bool inJ = true;
#pragma unroll
              for (int a = 0; a < 3; ++a) inJ = inJ && (kJ[a] < (((EXS[pj] >> a) & 1) ? 3 : 2));
              if (!inJ) continue;
              double wJ, GJ[3], waJ;
              node_geom<3>(AX[pj], kJ, wJ, GJ, waJ);
#pragma unroll
              for (int r = 0; r < NB; ++r) {
                double sv;
                if (c < 3) {
                  sv = 0.0;
#pragma unroll
                  for (int aa = 0; aa < 3; ++aa) sv += E[pj][r * NZ + aa * 3 + c] * GJ[aa];
                  if (c == 2) sv += E[pj][r * NZ + L::Z_DU] * wJ;
                } else {
                  sv = E[pj][r * NZ + L::Z_P] * wJ + E[pj][r * NZ + L::Z_PB] * waJ;
#pragma unroll
                  for (int aa = 0; aa < 3; ++aa) sv += E[pj][r * NZ + L::Z_G + aa] * GJ[aa];
                }
                acc[r] += sv;
              }
            }
#pragma unroll
            for (int r = 0; r < NB; ++r) ACC[bit * NB * NB + r * NB + c] = acc[r];
          }
          __syncthreads();
        }
      }
  // flush the window blocks present in the row pattern: masks, sign (-dR/du), identity rows
  const uint64_t m0 = row_mask[2 * I], m1 = row_mask[2 * I + 1];
  const int rp = row_ptr[I];
  for (int b = t; b < 125; b += T) {
    const uint64_t w = (b < 64) ? m0 : m1;
    const int sh = b & 63;
    if (!((w >> sh) & 1ull)) continue;
    const int below = (b < 64) ? __popcll(sh ? (m0 & ((1ull << sh) - 1ull)) : 0ull)
                               : __popcll(m0) + __popcll(sh ? (m1 & ((1ull << sh) - 1ull)) : 0ull);
    const int cj[3] = {ci[0] + b % 5 - 2, ci[1] + (b / 5) % 5 - 2, ci[2] + b / 25 - 2};
    const int Jn = node_index<3>(g, cj);
    const bool diag = (Jn == I);
    TV* out = vals + (long)(rp + below) * NB * NB;
#pragma unroll
    for (int r = 0; r < NB; ++r) {
      const bool fr = freem[I * NB + r];
#pragma unroll
      for (int cc = 0; cc < NB; ++cc) {
        const bool fc = freem[Jn * NB + cc];
        double v = (fr && fc) ? -ACC[b * NB * NB + r * NB + cc] : 0.0;
        if (diag && r == cc && !fr) v = 1.0;
        out[r * NB + cc] = (TV)v;
      }
    }
  }
}

extern "C" int gm_node_jacobian(const gm_grid* g, const gm_bins* b, const gm_pattern* pat, const void* D,
                                int tangent_fp32, const uint8_t* freem, void* vals, int vals_fp32, int coupled,
                                hipStream_t s) {
  GM_REQUIRE(g && b && pat, "gm_node_jacobian: null argument");
  int n = g->n_nodes;
  if (g->dim != 2 && !coupled) {
    gm::set_error("gm_node_jacobian: 3D single-phase is not a supported form");
    return -1;
  }
  // 3D u-p: lanes per (column, column dof) of a bin (k_node_jacobian_up3); GM_JACOBIAN_ROW_WAVE=1
  // selects the one-wavefront-per-row form, which assembles the same matrix
  const bool row_wave = getenv("GM_JACOBIAN_ROW_WAVE");
#define GM_JAC(TD, TV)                                                                                           \
  do {                                                                                                           \
    if (g->dim == 2 && !coupled)                                                                                 \
      k_strip_jacobian<false, TD, TV><<<gm_blocks(n, 16), 192, 0, s>>>(                                          \
          *g, b->x_s, b->lp_s, b->cell_start, b->ext_s, (const TD*)D, freem, pat->row_ptr, pat->row_mask, (TV*)vals); \
    else if (g->dim == 2)                                                                                        \
      k_strip_jacobian<true, TD, TV><<<gm_blocks(n, 7), 192, 0, s>>>(                                            \
          *g, b->x_s, b->lp_s, b->cell_start, b->ext_s, (const TD*)D, freem, pat->row_ptr, pat->row_mask, (TV*)vals); \
    else if (row_wave)                                                                                           \
      k_node_jacobian<TD, TV><<<n, 64, 0, s>>>(*g, b->x_s, b->lp_s, b->cell_start, b->ext_s, (const TD*)D, freem, \
                                               pat->row_ptr, pat->row_mask, (TV*)vals);                          \
    else                                                                                                         \
      k_node_jacobian_up3<TD, TV><<<n, 128, 0, s>>>(*g, b->x_s, b->lp_s, b->cell_start, b->ext_s, (const TD*)D,  \
                                                    freem, pat->row_ptr, pat->row_mask, (TV*)vals);              \
  } while (0)
  if (tangent_fp32 && vals_fp32) GM_JAC(float, float);
  else if (tangent_fp32) GM_JAC(float, double);
  else if (vals_fp32) GM_JAC(double, float);
  else GM_JAC(double, double);
#undef GM_JAC
  GM_LAUNCH_CHECK();
  return 0;
}

// ================================================================== indenter penalty, preconditioner copy
// The reference's indenter term r_z += -(h - (z + du_z)) pen_par w_I (mpm_utils.py:1240-1246)
// enters the Newton matrix K = -dR/du as -pen_par w_I w_J on the z-dofs of every
// penetrating particle's support: a negative stiffness that outweighs the soil's
// under the indenter and makes K indefinite there.  The multigrid hierarchy is
// built from a copy of K with that term's sign reversed (coef = 2 adds
// 2 pen_par w_I w_J), which is positive definite under the indenter; the Krylov
// operator keeps the exact K.  One thread per node row of the box
// [lo, lo + cnt) that holds every support node of the penetrating particles;
// the particles and the predicate are those of the particle stage
// (x_s is the bin-sorted copy of x), and only free z-dofs are touched.
template <typename TV>
__global__ void __launch_bounds__(128) k_penalty_pc(gm_grid g, const double* x_s, const double* lp_s,
                                                    const int* cell_start, const uint8_t* ext_s,
                                                    const uint8_t* freem, const int* row_ptr,
                                                    const uint64_t* row_mask, TV* vals, int lo0, int lo1, int lo2,
                                                    int c0, int c1, int c2, double fx0, double fx1, double fy0,
                                                    double fy1, double height, double coef) {
  const int NB = 4;
  int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= c0 * c1 * c2) return;
  int ci[3] = {lo0 + t % c0, lo1 + (t / c0) % c1, lo2 + t / (c0 * c1)};
  if (ci[0] > g.nx || ci[1] > g.ny || ci[2] > g.nz) return;
  int I = node_index<3>(g, ci);
  if (!freem[I * NB + 2]) return;
  const int rs = row_ptr[I];
  const uint64_t m0 = row_mask[2 * I], m1 = row_mask[2 * I + 1];
  for_candidates<3>(g, ci, cell_start, ext_s, [&](int k, const int* o, const int* b, bool in) {
    if (!in) return;
    double xx = x_s[3 * k], xy = x_s[3 * k + 1], xz = x_s[3 * k + 2];
    if (!(xz >= height && xx > fx0 && xx < fx1 && xy > fy0 && xy < fy1)) return;
    Axis ax[3];
    load_axes<3>(g, x_s, lp_s, k, ax);
    double wI = sel3(ax[0].w, o[0]) * sel3(ax[1].w, o[1]) * sel3(ax[2].w, o[2]);
    for (int kz = 0; kz < ax[2].ext; ++kz)
      for (int ky = 0; ky < ax[1].ext; ++ky)
        for (int kx = 0; kx < ax[0].ext; ++kx) {
          int cj[3] = {b[0] + kx, b[1] + ky, b[2] + kz};
          int Jn = node_index<3>(g, cj);
          if (!freem[Jn * NB + 2]) continue;
          double wJ = sel3(ax[0].w, kx) * sel3(ax[1].w, ky) * sel3(ax[2].w, kz);
          int bit = (kx - o[0] + 2) + 5 * (ky - o[1] + 2) + 25 * (kz - o[2] + 2);
          // compressed slot: set window bits below `bit`
          int below;
          if (bit < 64) {
            below = __popcll(bit ? (m0 & ((1ull << bit) - 1ull)) : 0ull);
          } else {
            int hb = bit - 64;
            below = __popcll(m0) + __popcll(hb ? (m1 & ((1ull << hb) - 1ull)) : 0ull);
          }
          long slot = (long)(rs + below) * (NB * NB) + 2 * NB + 2;
          vals[slot] = (TV)((double)vals[slot] + coef * wI * wJ);
        }
  });
}

extern "C" int gm_penalty_pc(const gm_grid* g, const gm_bins* b, const gm_pattern* pat, const uint8_t* freem,
                             void* vals, int vals_fp32, const int* box_lo, const int* box_cnt,
                             const double* footing, double height, double coef, hipStream_t s) {
  GM_REQUIRE(g && b && pat && freem && vals && box_lo && box_cnt && footing, "gm_penalty_pc: null argument");
  GM_REQUIRE(g->dim == 3 && g->nb == 4, "gm_penalty_pc: the indenter term exists in the 3D u-p form only");
  long cnt = (long)box_cnt[0] * box_cnt[1] * box_cnt[2];
  GM_REQUIRE(box_lo[0] >= 0 && box_lo[1] >= 0 && box_lo[2] >= 0 && box_cnt[0] >= 0 && box_cnt[1] >= 0 &&
                 box_cnt[2] >= 0 && cnt < (1L << 30),
             "gm_penalty_pc: bad node box");
  if (cnt == 0) return 0;
  int blk = gm_blocks(cnt, 128);
  if (vals_fp32)
    k_penalty_pc<float><<<blk, 128, 0, s>>>(*g, b->x_s, b->lp_s, b->cell_start, b->ext_s, freem, pat->row_ptr,
                                            pat->row_mask, (float*)vals, box_lo[0], box_lo[1], box_lo[2],
                                            box_cnt[0], box_cnt[1], box_cnt[2], footing[0], footing[1],
                                            footing[2], footing[3], height, coef);
  else
    k_penalty_pc<double><<<blk, 128, 0, s>>>(*g, b->x_s, b->lp_s, b->cell_start, b->ext_s, freem, pat->row_ptr,
                                             pat->row_mask, (double*)vals, box_lo[0], box_lo[1], box_lo[2],
                                             box_cnt[0], box_cnt[1], box_cnt[2], footing[0], footing[1],
                                             footing[2], footing[3], height, coef);
  GM_LAUNCH_CHECK();
  return 0;
}

// ================================================================== P2G
// Node-gather form of P2G_2d / P2G_coupled_2d / P2G_coupled_3d (mpm_utils.py:83-383).
//  act:     activation (threshold < 0: every support node, as P2G_2d; else w > threshold)
//  bflag:   pressure-Dirichlet flags are OR-ed into the p dof (coupled)
//  mrhs:    consistent-mass rhs, may be null
// Four lanes a node take every fourth particle of each of its bins: a lane alone is a chain of
// dependent loads (ids, pressures) and axis data over some 36 (2D) or 216 particles (11,628 2D nodes:
// 53 -> 26 us).
template <int DIM>
__global__ void __launch_bounds__(128) k_p2g(gm_grid g, int nb, const double* x_s, const double* lp_s,
                                             const int* cell_start, const int* sorted, const uint8_t* ext_s,
                                             double threshold, const uint8_t* pbc_flag, double node_h_last,
                                             double p_mass, const double* p_part, uint8_t* act, uint8_t* bflag,
                                             double* mrhs) {
  const int I = blockIdx.x * 32 + threadIdx.x / 4, sub = threadIdx.x % 4;
  int ci[3] = {0, 0, 0};
  node_coords<DIM>(g, I, ci);
  const int ncell[3] = {g.nx, g.ny, g.nz};
  int on = 0;  // 1: active, 2: pressure boundary
  double rhs = 0.0;
  const double nc = (double)ci[DIM - 1] * node_h_last;
  for (int q = 0; q < (DIM == 3 ? 27 : 9) && I < g.n_nodes; ++q) {
    const int o[3] = {q % 3, q / 3 % 3, q / 9};
    int bc[3] = {0, 0, 0};
    bool ok = true;
#pragma unroll
    for (int a = 0; a < DIM; ++a) {
      bc[a] = ci[a] - o[a];
      if (bc[a] < 0 || bc[a] > ncell[a]) ok = false;
    }
    if (!ok) continue;
    const int b = node_index<DIM>(g, bc);
    for (int k = cell_start[b] + sub; k < cell_start[b + 1]; k += 4) {
      const int p = sorted[k];
      const uint8_t ex = ext_s[k];
      bool in = true;
#pragma unroll
      for (int a = 0; a < DIM; ++a) in = in && o[a] < (((ex >> a) & 1) ? 3 : 2);
      // pressure boundary: 2D loops over the support, 3D over all 27 nodes (mpm_utils.py:225-235, 349-352)
      if (pbc_flag && pbc_flag[p] && (in || DIM == 3) && nc >= x_s[k * DIM + DIM - 1]) on |= 2;
      if (!in) continue;
      const double pp = mrhs ? p_part[p] : 0.0;
      Axis ax[DIM];
      load_axes<DIM>(g, x_s, lp_s, k, ax);
      double w, G[3], wa;
      node_geom<DIM>(ax, o, w, G, wa);
      if (threshold < 0.0 || w > threshold) on |= 1;
      if (mrhs) {
        // sum of the particle's weights over its support, one axis at a time
        double wsum = 1.0;
#pragma unroll
        for (int aa = 0; aa < DIM; ++aa) wsum *= ax[aa].w[0] + ax[aa].w[1] + ax[aa].w[2];
        rhs += w * wsum * p_mass * pp;
      }
    }
  }
#pragma unroll
  for (int s = 1; s < 4; s <<= 1) {
    rhs += __shfl_xor(rhs, s, 64);
    on |= __shfl_xor(on, s, 64);
  }
  if (sub || I >= g.n_nodes) return;
  if (on & 1)
    for (int k = 0; k < nb; ++k) act[I * nb + k] = 1;
  if ((on & 2) && bflag) bflag[I * nb + DIM] = 1;
  if (mrhs) mrhs[I] = rhs;
}

extern "C" int gm_p2g(const gm_grid* g, const gm_bins* b, const gm_pattern* pat, double threshold,
                      const uint8_t* pbc_flag, double node_h_last, double p_mass, const double* p_part, uint8_t* act,
                      uint8_t* bflag, double* mvals, double* mrhs, hipStream_t s) {
  GM_REQUIRE(g && b, "gm_p2g: null argument");
  int n = g->n_nodes;
  if (mvals) {
    GM_REQUIRE(pat, "gm_p2g: mass matrix needs the pattern");
    gm::launch_mass(*g, *b, *pat, p_mass, mvals, s);
    GM_LAUNCH_CHECK();
  }
  if (g->dim == 2)
    k_p2g<2><<<gm_blocks(n, 32), 128, 0, s>>>(*g, g->nb, b->x_s, b->lp_s, b->cell_start, b->sorted, b->ext_s, threshold,
                                               pbc_flag, node_h_last, p_mass, p_part, act, bflag, mrhs);
  else
    k_p2g<3><<<gm_blocks(n, 32), 128, 0, s>>>(*g, g->nb, b->x_s, b->lp_s, b->cell_start, b->sorted, b->ext_s, threshold,
                                               pbc_flag, node_h_last, p_mass, p_part, act, bflag, mrhs);
  GM_LAUNCH_CHECK();
  return 0;
}

// free mask = !boundary && active, node-interleaved
__global__ void k_free_mask(int n, const uint8_t* bflag, const uint8_t* act, uint8_t* freem) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  freem[i] = (!bflag[i] && act[i]) ? 1 : 0;
}

extern "C" int gm_free_mask(int n, const uint8_t* bflag, const uint8_t* act, uint8_t* freem, hipStream_t s) {
  if (n == 0) return 0;
  k_free_mask<<<gm_blocks(n, 256), 256, 0, s>>>(n, bflag, act, freem);
  GM_LAUNCH_CHECK();
  return 0;
}

// P2G_set_nodal_solution(_3d) (mpm_utils.py:387-414)
__global__ void k_set_nodal_p(int n_nodes, int nb, int pdof, const uint8_t* bflag, const uint8_t* act,
                              int require_active, const double* xp, double* old_s, double* new_s) {
  int I = blockIdx.x * blockDim.x + threadIdx.x;
  if (I >= n_nodes) return;
  int d = I * nb + pdof;
  if (!bflag[d] && (!require_active || act[d])) {
    old_s[d] = xp[I];
    new_s[d] = xp[I];
  }
}

extern "C" int gm_set_nodal_pressure(int n_nodes, int nb, const uint8_t* bflag, const uint8_t* act,
                                     int require_active, const double* xp, double* old_s, double* new_s,
                                     hipStream_t s) {
  k_set_nodal_p<<<gm_blocks(n_nodes, 256), 256, 0, s>>>(n_nodes, nb, nb - 1, bflag, act, require_active, xp, old_s,
                                                        new_s);
  GM_LAUNCH_CHECK();
  return 0;
}

// ================================================================== G2P + lp update
// G2P_2d / G2P_coupled_2d / G2P_coupled_3d (mpm_utils.py:1351-1590).  A particle a lane; a
// block's rows of F and b are one run of values each, copied with consecutive lanes on
// consecutive values (loaded first, so that they arrive during the gather).  Bound by HBM: 354
// bytes a particle and the nodes.  1,048,576 particles in 3D: 326 us with 9 strided values a
// lane, 139 us now.
template <int DIM, bool COUPLED>
__global__ void __launch_bounds__(128) k_g2p(gm_grid g, int n, double* x, const double* lp, const double* u_new,
                                             const double* u_old, double* F_old, const double* F_new, double* b_old,
                                             const double* b_new, double* alpha_old, const double* alpha_new,
                                             double* p_part) {
  constexpr int NB = DIM + (COUPLED ? 1 : 0);
  const int t = threadIdx.x, p0 = blockIdx.x * 128, n9 = 9 * min(128, n - p0);
  double Ft[9], bt[9];
#pragma unroll
  for (int i = 0; i < 9; ++i) {
    const long q = 9L * p0 + min(i * 128 + t, n9 - 1);
    Ft[i] = F_new[q];
    bt[i] = b_new[q];
  }
  const int p = p0 + t;
  if (p < n) {
    Axis ax[DIM];
    load_axes<DIM>(g, x, lp, p, ax);
    double du[3] = {0, 0, 0};
    double pn = 0.0;
    auto load = [&](int i, int j, int k, double* un, double* uo) {
      const int c[3] = {ax[0].lo + i, ax[1].lo + j, DIM == 3 ? ax[2].lo + k : 0};
      const int node = node_index<DIM>(g, c);
#pragma unroll
      for (int cc = 0; cc < NB; ++cc) un[cc] = u_new[node * NB + cc];
#pragma unroll
      for (int cc = 0; cc < DIM; ++cc) uo[cc] = COUPLED ? u_old[node * NB + cc] : 0.0;
    };
    auto add = [&](int i, int j, int k, const double* un, const double* uo) {
      const int o[3] = {i, j, k};
      double w, G[3], wa;
      node_geom<DIM>(ax, o, w, G, wa);
#pragma unroll
      for (int cc = 0; cc < DIM; ++cc) du[cc] += w * (COUPLED ? un[cc] - uo[cc] : un[cc]);
      if (COUPLED) pn += w * un[NB - 1];
    };
    // the first two nodes of the last axis, which every particle has, are loaded together
    const int el = ax[DIM - 1].ext;
    for (int i = 0; i < ax[0].ext; ++i)
      for (int j = 0; j < (DIM == 3 ? ax[1].ext : 1); ++j) {
        auto at = [&](int k) { return DIM == 3 ? k : 0; };
        auto jt = [&](int k) { return DIM == 3 ? j : k; };
        double n0[NB], o0[DIM], n1[NB], o1[DIM];
        load(i, jt(0), at(0), n0, o0);
        load(i, jt(1), at(1), n1, o1);
        add(i, jt(0), at(0), n0, o0);
        add(i, jt(1), at(1), n1, o1);
        if (el == 3) {
          load(i, jt(2), at(2), n0, o0);
          add(i, jt(2), at(2), n0, o0);
        }
      }
    if (alpha_old && alpha_new) alpha_old[p] = alpha_new[p];
#pragma unroll
    for (int cc = 0; cc < DIM; ++cc) x[p * DIM + cc] += du[cc];
    if (COUPLED && p_part) p_part[p] = pn;
  }
#pragma unroll
  for (int i = 0; i < 9; ++i) {
    const int q = i * 128 + t;
    if (q < n9) {
      F_old[9L * p0 + q] = Ft[i];
      b_old[9L * p0 + q] = bt[i];
    }
  }
}

extern "C" int gm_g2p(const gm_grid* g, int n, double* x, const double* lp, const double* u_new, const double* u_old,
                      double* F_old, const double* F_new, double* b_old, const double* b_new, double* alpha_old,
                      const double* alpha_new, double* p_part, int coupled, hipStream_t s) {
  if (n == 0) return 0;
  int blk = gm_blocks(n, 128);
  if (g->dim == 2 && !coupled)
    k_g2p<2, false><<<blk, 128, 0, s>>>(*g, n, x, lp, u_new, u_old, F_old, F_new, b_old, b_new, alpha_old, alpha_new,
                                        p_part);
  else if (g->dim == 2)
    k_g2p<2, true><<<blk, 128, 0, s>>>(*g, n, x, lp, u_new, u_old, F_old, F_new, b_old, b_new, alpha_old, alpha_new,
                                       p_part);
  else if (coupled)
    k_g2p<3, true><<<blk, 128, 0, s>>>(*g, n, x, lp, u_new, u_old, F_old, F_new, b_old, b_new, alpha_old, alpha_new,
                                       p_part);
  else {
    gm::set_error("gm_g2p: 3D single-phase is not a supported form");
    return -1;
  }
  GM_LAUNCH_CHECK();
  return 0;
}

// update_GIMP_lp_2d/3d (gimp.py:428-507).  A domain that sticks out of the box is cut 1e-6 inside it,
// a jump that a comparison decides.  In a wall cell x - min and lp0 |F col| are equal but for products
// of shears, so far from the load the comparison hangs on the last digits of x and F, and a change of
// rounding anywhere in the load step flips entries (64 x 64 x 32 cells, mixed form: the order of the
// sums of any one kernel of the step, in one to five of 24 load paths).  Hence the kernels of the 3D
// u-p step keep the order and the rounding of their sums.
__global__ void k_update_lp(int n, int dim, const double* F_new, double* lp, double lp0, const double* x,
                            double mnx, double mxx, double mny, double mxy, double mnz, double mxz) {
  int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  double mn[3] = {mnx, mny, mnz}, mx[3] = {mxx, mxy, mxz};
  const double* F = F_new + 9 * p;
  for (int a = 0; a < dim; ++a) {
    double U = sqrt(F[0 * 3 + a] * F[0 * 3 + a] + F[1 * 3 + a] * F[1 * 3 + a] + F[2 * 3 + a] * F[2 * 3 + a]);
    double l = lp0 * U;
    double xa = x[p * dim + a];
    if (xa - l < mn[a]) l = xa - mn[a] - 1e-6;
    if (xa + l > mx[a]) l = mx[a] - xa - 1e-6;
    lp[p * dim + a] = l;
  }
}

extern "C" int gm_update_lp(int n, int dim, const double* F_new, double* lp, double lp0, const double* x,
                            const double* dmin, const double* dmax, hipStream_t s) {
  if (n == 0) return 0;
  k_update_lp<<<gm_blocks(n, 256), 256, 0, s>>>(n, dim, F_new, lp, lp0, x, dmin[0], dmax[0], dmin[1], dmax[1],
                                                dim == 3 ? dmin[2] : 0.0, dim == 3 ? dmax[2] : 0.0);
  GM_LAUNCH_CHECK();
  return 0;
}

// ================================================================== standalone entry points
// Per-particle cpGIMP data in the reference's output layout
// (get_GIMP_shape_function_and_gradient_2d/3d, gimp.py:25-112, 197-315, and the
// _avg_ variants :115-193, :318-425): out[p] = (w0_x, w0_y[, w0_z], w1_..., w2_...,
// g0_..., g1_..., g2_...) and avg[p] likewise (weights then gradients), base[p*dim+a] = lo.
__global__ void k_gimp_weights(int n, int dim, const double* x, const double* lp, double h0, double h1, double h2,
                               double* out, double* avg, int* base) {
  int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  double hs[3] = {h0, h1, h2};
  for (int a = 0; a < dim; ++a) {
    Axis ax = gimp_axis(x[p * dim + a], lp[p * dim + a], hs[a], 1.0 / hs[a]);
    for (int k = 0; k < 3; ++k) {
      out[(long)p * 6 * dim + k * dim + a] = ax.w[k];
      out[(long)p * 6 * dim + 3 * dim + k * dim + a] = ax.g[k];
      if (avg) {
        avg[(long)p * 6 * dim + k * dim + a] = ax.wa[k];
        // the reference's average gradients: -sign(x - x_k)/(4 lp) at k = 0, 2 in the cpGIMP branch,
        // with sign(0) = +1 as Warp's wp.sign defines it
        double gk = 0.0;
        double xa = x[p * dim + a], la = lp[p * dim + a], ih = 1.0 / hs[a];
        bool cp = (int)((xa - la) * ih + 1e-8) != (int)((xa + la) * ih + 1e-8);  // cpGIMP branch
        if (cp && k != 1) {
          double d = xa - (ax.lo + k) * hs[a];
          gk = -1.0 / (4.0 * la) * (d < 0.0 ? -1.0 : 1.0);
        }
        avg[(long)p * 6 * dim + 3 * dim + k * dim + a] = gk;
      }
    }
    if (base) base[p * dim + a] = ax.lo;
  }
}

extern "C" int gm_gimp_weights(int n, int dim, const double* x, const double* lp, const double* h, double* out,
                               double* avg, int* base, hipStream_t s) {
  GM_REQUIRE(h && x && lp && out, "gm_gimp_weights: null argument");
  if (n == 0) return 0;
  k_gimp_weights<<<gm_blocks(n, 256), 256, 0, s>>>(n, dim, x, lp, h[0], h[1], dim == 3 ? h[2] : h[0], out, avg,
                                                   base);
  GM_LAUNCH_CHECK();
  return 0;
}

// Standalone principal return mapping (plasticity.py:8-37 J2; triaxial_DruckerPrager.py:308-412 DP):
// eps_tr, eps (n x 3 principal log strains), dE (n x 9 consistent tangent d eps/d eps_tr, may be null),
// alpha_old/new (J2 hardening, may be null).
__global__ void k_return_map(int n, MatParams m, const double* etr, double* eps, double* dE, const double* ao,
                             double* an) {
  int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  double e[3], d[9], a_new = 0.0;
  double et[3] = {etr[3 * p], etr[3 * p + 1], etr[3 * p + 2]};
  if (m.kind == MAT_J2) {
    return_j2(et, m, ao ? ao[p] : 0.0, e, d, a_new);
  } else if (m.kind == MAT_DP) {
    return_dp(et, m, e, d);
  } else {
    for (int i = 0; i < 3; ++i) e[i] = et[i];
    for (int i = 0; i < 9; ++i) d[i] = (i % 4 == 0) ? 1.0 : 0.0;
  }
  for (int i = 0; i < 3; ++i) eps[3 * p + i] = e[i];
  if (dE)
    for (int i = 0; i < 9; ++i) dE[9 * p + i] = d[i];
  if (an) an[p] = a_new;
}

extern "C" int gm_return_map(int n, int mat_kind, int dp_apex, double lam, double mu, double kappa, double H,
                             double phi, double psi, double coh, double shape, const double* eps_tr, double* eps,
                             double* dE, const double* alpha_old, double* alpha_new, hipStream_t s) {
  if (n == 0) return 0;
  MatParams m;
  m.kind = mat_kind;
  m.dp_apex = dp_apex;
  m.lam = lam;
  m.mu = mu;
  m.E = 0.0;
  m.kappa = kappa;
  m.H = H;
  m.phi = phi;
  m.psi = psi;
  m.coh = coh;
  m.shape = shape;
  k_return_map<<<gm_blocks(n, 256), 256, 0, s>>>(n, m, eps_tr, eps, dE, alpha_old, alpha_new);
  GM_LAUNCH_CHECK();
  return 0;
}

// ---------------------------------------------------------------------------------------------
// NorSand return mapping (triaxial_NorSand.py:155-400), one particle per lane (gm_device.h
// return_norsand: pressure-dependent hyperelasticity P = p0 exp(-(eps_v - ev0)/kappa), Q = 3 mu
// eps_s; yield Q + eta(P, pi) P; fixed 15-iteration local Newton on (eps_v, eps_s, dlambda, pi_i)
// with hardening h (pi_i - pi*); tension (eps_v > tol) returns zero strain).
// ---------------------------------------------------------------------------------------------
namespace {
__global__ void k_return_map_norsand(int n, gm_norsand_params q, const double* etr, const double* ev_total,
                                     const double* pi_old, double* eps, double* pi_new, double* res_last) {
  int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const double et[3] = {etr[3 * p], etr[3 * p + 1], etr[3 * p + 2]};
  double e[3], pn, r[4];
  return_norsand(et, ev_total[p], pi_old[p], q, e, pn, r, nullptr, nullptr);
  for (int i = 0; i < 3; ++i) eps[3 * p + i] = e[i];
  pi_new[p] = pn;
  if (res_last)
    for (int i = 0; i < 4; ++i) res_last[4 * p + i] = r[i];
}
}  // namespace

extern "C" int gm_return_map_norsand(int n, const gm_norsand_params* prm, const double* eps_tr,
                                     const double* eps_total_trace, const double* pi_old, double* eps, double* pi_new,
                                     double* res_last, hipStream_t s) {
  GM_REQUIRE(prm, "gm_return_map_norsand: null parameters");
  if (n == 0) return 0;
  GM_REQUIRE(eps_tr && eps_total_trace && pi_old && eps && pi_new, "gm_return_map_norsand: null argument");
  k_return_map_norsand<<<gm_blocks(n, 128), 128, 0, s>>>(n, *prm, eps_tr, eps_total_trace, pi_old, eps, pi_new,
                                                         res_last);
  GM_LAUNCH_CHECK();
  return 0;
}
