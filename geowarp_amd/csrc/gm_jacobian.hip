// Node Jacobian of the 3D u-p form, assembled per particle bin on the matrix cores.
//
// K_IJ = -sum_p L_I(p) D_p M_J(p) (block 4x4; I, J nodes; p particles).  L_I and
// M_J are linear in the particle's shape-function values at the node,
// g = (w, dw/dx, dw/dy, dw/dz, w_avg), so with E_I = L_I D_p (4 x 15) a bin's
// contribution is
//     C_b[(I,r),(J,c)] = sum_{p in b} sum_beta X_p[(I,r),(c,beta)] g_p[J,beta],
// X_p[(I,r),(c,beta)] an entry of E_I (or zero).  All particles of a bin (same
// stencil base node b) reach the same 3x3x3 nodes, so for every column dof c this
// is a dense product (108 rows (I,r)) x (5 n_p) x (27 columns J): the matrix
// cores take it 16x16x4 at a time, FP32 when the tangent is FP32 (mixed form),
// FP64 otherwise.  Two forms, each a product kernel and a gather:
//   k_jac_bin     a 256-lane workgroup per bin (or a persistent sweep over bins):
//                 E_I for a group of particles in LDS, 14 output tiles of 16x16
//                 over the 4 waves, the bin's 27 x 27 blocks written contiguously
//                 to a workspace (n_nodes x 11664 values).
//   k_jac_gather  one workgroup per block row I: every block (I, J) of the
//                 pattern sums the <= 27 bins b = I - o holding both nodes in the
//                 fixed order (oz, oy, ox); masks, sign and identity rows as in
//                 the node-row kernels (k_jac_gather_staged: the same sums from
//                 chunks staged in LDS).
//   k_jac_line    (FP64) a workgroup per segment of a bin line (fixed y, z): the products of
//                 its bins one after another, summed over the line while they stay in the
//                 accumulators; every pair of nodes a line reaches is written once (405
//                 blocks a bin where the bin itself has 729; n_nodes x 6480 values).
//   k_jac_line_gather  one workgroup per block row I: every block sums the <= 9 lines holding
//                 both nodes in the fixed order (oz, oy).
// Both forms are deterministic (fixed accumulation order), and bound by HBM on the workspace,
// written and read once, and the matrix itself.
//   FP32 takes bins at every size: a sum over a line would add up to three bin sums in FP32
//   where the gather adds all of them in FP64, which moves the mixed form's Newton iterates
//   (load steps are held to the last bit, see k_update_lp).  It would be faster on large grids:
//   2.23 + 1.05 ms against 2.84 + 1.56 with 64 x 64 x 32 cells, 1,048,576 particles (MI355X).
//   FP64 takes lines where they are the faster form (line_sums): 4.0 + 1.83 ms against 5.6 +
//   2.9 on that grid.  k_jac_line: the products take 1.3 ms, the stores of the line sums 1.95
//   (7.2 GB), and one follows the other in the product waves; the operand waves' arithmetic
//   adds 0.2.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "gm_common.h"
#include "gm_device.h"
#include "gm_types.h"

using namespace gm;

namespace {

// 3D u-p layout of the particle stress vector Y (17) and unknowns z (15): P (9),
// body/penalty force T (3), mass balance Q, Darcy flux m (3), PPP term S; z =
// grad du (9), du_z, p, pbar, grad p (3).
constexpr int NY = 17, NZ = 15;
constexpr int Y_T = 9, Y_Q = 12, Y_M = 13, Y_S = 16;
constexpr int Z_DU = 9, Z_P = 10, Z_PB = 11, Z_G = 12;
constexpr long CB_BIN = 27L * 27L * 16L;  // values per bin: 27 x 27 blocks of 4 x 4
// chunk of bin `bin`'s blocks (I_loc = o, J_loc = 0..26) in the workspace: bins one
// after another, each its 27 chunks in I_loc order
constexpr long CHUNK = 27L * 16L;
__device__ __forceinline__ long chunk_at(int o, int bin) { return (long)bin * CB_BIN + o * CHUNK; }
// Workspace of the line sums, per bin line (y, z) and node x of it (a grid node's share):
// the pairs of a row node and a column node of the line whose smaller x is that node's, which
// one step of k_jac_line completes together.  Parts: nine chunks A (row node (x, y + oy,
// z + oz), column nodes x .. x + 2), then nine chunks B for row nodes x + 1 and nine for
// x + 2 (column nodes x).  In a chunk: column dof c, column node ([dx] [jy + 3 jz]), row dof
// r.  A matrix-core lane ends with the four rows r of one (row node, column node, c), so
// that a store instruction writes whole runs of neighbouring 16-byte vectors.
constexpr long CHUNK_A = 4L * 27 * 4, CHUNK_B = 4L * 9 * 4;  // values
constexpr long LINE_NODE = 9L * (CHUNK_A + 2 * CHUNK_B);     // values per grid node
__device__ __forceinline__ long chunk_a(int o9, int node) { return (long)node * LINE_NODE + o9 * CHUNK_A; }
// d = 1, 2: the distance of the row node
__device__ __forceinline__ long chunk_b(int o9, int node, int d) {
  return (long)node * LINE_NODE + 9 * CHUNK_A + ((d - 1) * 9 + o9) * CHUNK_B;
}

typedef float f4v __attribute__((ext_vector_type(4)));
typedef double d4v __attribute__((ext_vector_type(4)));

template <typename T>
struct Mfma;
// A (16 x 4): lane l holds A[l % 16][l / 16]; B (4 x 16): B[l / 16][l % 16]; the
// 16 x 16 result: item v of lane l is row 4 (l / 16) + v (FP32) or l / 16 + 4 v
// (FP64) of column l % 16.  An M tile orders its 16 rows (I, r) I-major for FP32
// and r-major for FP64, so that either way lane l ends with the four rows r of
// one node I = l / 16 of the tile.
template <>
struct Mfma<float> {
  typedef f4v acc;
  static constexpr bool r_major = false;
  static __device__ __forceinline__ acc step(float a, float b, acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
};
template <>
struct Mfma<double> {
  typedef d4v acc;
  static constexpr bool r_major = true;
  static __device__ __forceinline__ acc step(double a, double b, acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
};

// z index of E feeding column dof c through shape-function component beta
// (0: w, 1-3: dw/dx_a, 4: w_avg), or ZERO (a column of E that holds zeros) where
// that product vanishes.
constexpr int ZERO = NZ;
__device__ __forceinline__ int zsel(int c, int beta) {
  if (c < 3) {
    if (beta == 0) return c == 2 ? Z_DU : ZERO;
    if (beta == 4) return ZERO;
    return (beta - 1) * 3 + c;
  }
  if (beta == 0) return Z_P;
  if (beta == 4) return Z_PB;
  return Z_G + beta - 1;
}

// shape-function component beta of stencil node J (x fastest) from the axis tables
template <typename TC>
__device__ __forceinline__ TC gcomp(const TC (*ax)[9], int J, int beta) {
  const int jx = J % 3, jy = (J / 3) % 3, jz = J / 9;
  if (beta == 4) return ax[0][6 + jx] * ax[1][6 + jy] * ax[2][6 + jz];
  const TC wx = ax[0][jx], wy = ax[1][jy], wz = ax[2][jz];
  if (beta == 0) return wx * wy * wz;
  if (beta == 1) return ax[0][3 + jx] * wy * wz;
  if (beta == 2) return wx * ax[1][3 + jy] * wz;
  return wx * wy * ax[2][3 + jz];
}

constexpr int MAX_SEG = 61;  // bins of a line segment (with two before it and the end, one a lane)

}  // namespace

// Per-bin products.  Workspace cb[b] = 27 x 27 blocks (I_loc, J_loc), I_loc = o_x +
// 3 o_y + 9 o_z with node = b + o.  A workgroup takes bins b = blockIdx.x, +gridDim.x,
// ... (one bin when the grid has one workgroup per bin, a persistent sweep when it is
// smaller) and each bin's particles PG at a time: the E table of a group in LDS, its
// products accumulated in the matrix-core registers, the bin's 27 x 27 blocks stored
// after its last group.  The global loads of the next group (of this bin or of the
// next one) are issued before the products of the current group when PF is set, so
// their latency hides behind the matrix cores (at the cost of the registers that hold
// them), else at the top of the group.
// K order: a K step of the MFMA is one shape-function component beta and four
// particles (lane group l / 16 = particle): the five components of a quad of
// particles, then the next quad, whatever PG is.  After the
// K loop unrolls, every A and B operand address is a per-lane base plus an immediate,
// and the (c, beta) products that vanish (u columns: no w term except the penalty
// on u_z, no w_avg term) are not issued.  Every (PG, OCC, PF, grid) variant adds the
// same products in the same order, so all of them write the same bits.
template <typename TD, typename TC, int PG, int OCC, bool PF>
__global__ void __launch_bounds__(256, OCC) k_jac_bin(gm_grid g, const double* x_s, const double* lp_s,
                                                      const int* cell_start, int n_bins, const TD* D, TC* cb) {
  static_assert(PG % 4 == 0, "particle groups are whole K steps");
  constexpr int KST = 5 * PG / 4;  // K steps of 4 per group
  constexpr int NI = 4 * NZ;       // (z, r) entries of a node row of E_p
  // shape-function tables of a group, two buffers: with PF the next group's are
  // computed (by wave 3, whose last row tile is empty) while the products run
  __shared__ TC AXT_[2][PG][3][9];
  // E_p[I][z][r] (r fastest), node rows 68 entries apart and particles 28 x 68 apart:
  // the 32 (particle, I, r) entries half a wave reads at once fall in 32 distinct banks.
  // Node row I = 27 is zero (the padding rows of the last row tile read it).
  constexpr int EI = 68, EP = 28 * EI;
  __shared__ TC E_[PG * EP];
#define E(p, I, z, r) E_[(p) * EP + (I) * EI + (z) * 4 + (r)]
  // B operand g_p[J][beta], J padded to 32 with zeros, particles 176 entries apart
  constexpr int BB = 32, BP = 5 * BB + 16;
  __shared__ TC BT_[PG * BP];
#define BT(p, beta, J) BT_[(p) * BP + (beta) * BB + (J)]
  int b = blockIdx.x, ks = 0, ke = 0;
  for (; b < n_bins; b += gridDim.x) {  // first non-empty bin (uniform across the workgroup)
    ks = cell_start[b];
    ke = cell_start[b + 1];
    if (ke > ks) break;
  }
  if (b >= n_bins) return;
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);  // uniform across the wave
  for (int q = t; q < PG * NI; q += 256) E(q / NI, 27, (q % NI) >> 2, q & 3) = 0;  // never written again
  typedef typename Mfma<TC>::acc ACC;
  ACC acc[4][4];
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[s][c] = ACC{0, 0, 0, 0};
  // output tiles tt = wave + 4 s: row tile mt = tt / 2 = wave / 2 + 2 s (16 rows (I, r)),
  // column tile nt = tt % 2 = wave % 2 (16 columns J); waves 2 and 3 have no fourth
  // tile (rows I >= 28)
  const int lg = lane >> 4, rt = lane & 15;
  const int r_l = Mfma<TC>::r_major ? (rt >> 2) : (rt & 3);
  const int i_l = Mfma<TC>::r_major ? (rt & 3) : (rt >> 2);
  int abase[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) abase[s] = lg * EP + min((wave >> 1) * 4 + 8 * s + i_l, 27) * EI + r_l;
  const int bbase = lg * BP + (wave & 1) * 16 + rt;
  constexpr int NQ = (PG * NI + 255) / 256;  // (p, z, r) items per thread
  constexpr int GT0 = PF ? 192 : 0;           // first thread of the shape-function tables
  static_assert(PG * 3 <= 64, "the tables of a group are one wave's work");
  TC dv[NQ][5];
  double xa = 0.0, la = 0.0;
  // tangent entries of this thread's (p, z, r) items, position and domain size of
  // particle (t - GT0) / 3 (axis (t - GT0) % 3) of the group starting at p0 (np particles)
  auto load_group = [&](int p0, int np) {
#pragma unroll
    for (int j = 0; j < NQ; ++j) {
      const int q = t + 256 * j;
      const int p = q / NI, zr = q % NI, z = zr >> 2, r = zr & 3;
#pragma unroll
      for (int i = 0; i < 5; ++i) dv[j][i] = (TC)0;
      if (q < PG * NI && p < np) {
        const TD* Dp = D + (long)(p0 + p) * NY * NZ;
        if (r < 3) {
          dv[j][0] = (TC)Dp[(0 * 3 + r) * NZ + z];
          dv[j][1] = (TC)Dp[(1 * 3 + r) * NZ + z];
          dv[j][2] = (TC)Dp[(2 * 3 + r) * NZ + z];
          dv[j][3] = (TC)Dp[(Y_T + r) * NZ + z];
        } else {
          const TC dS = (TC)Dp[Y_S * NZ + z];
          dv[j][0] = (TC)Dp[(Y_M + 0) * NZ + z];
          dv[j][1] = (TC)Dp[(Y_M + 1) * NZ + z];
          dv[j][2] = (TC)Dp[(Y_M + 2) * NZ + z];
          dv[j][3] = (TC)Dp[Y_Q * NZ + z] + dS;
          dv[j][4] = -dS;
        }
      }
    }
    xa = 0.0;
    la = 0.0;
    if (t >= GT0 && t < GT0 + PG * 3 && (t - GT0) / 3 < np) {
      xa = x_s[(long)(p0 + (t - GT0) / 3) * 3 + (t - GT0) % 3];
      la = lp_s[(long)(p0 + (t - GT0) / 3) * 3 + (t - GT0) % 3];
    }
  };
  // shape-function tables of the group whose positions are in xa / la (np particles)
  auto axis_tables = [&](int buf, int np) {
    if (t >= GT0 && t < GT0 + PG * 3) {
      const int p = (t - GT0) / 3, a = (t - GT0) % 3;
      if (p < np) {
        const Axis ax = gimp_axis(xa, la, g.h[a], g.inv_h[a]);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          AXT_[buf][p][a][i] = (TC)ax.w[i];
          AXT_[buf][p][a][3 + i] = (TC)ax.g[i];
          AXT_[buf][p][a][6 + i] = (TC)ax.wa[i];
        }
      } else {
#pragma unroll
        for (int i = 0; i < 9; ++i) AXT_[buf][p][a][i] = (TC)0;
      }
    }
  };
  int p0 = ks, cur = 0;
  if (PF) {
    load_group(p0, min(PG, ke - p0));
    axis_tables(0, min(PG, ke - p0));
  }
  while (true) {
    const int np = min(PG, ke - p0);
    if (!PF) load_group(p0, np);
    __syncthreads();  // the previous group's LDS reads are done (and, with PF, this one's tables written)
    if (!PF) {
      axis_tables(cur, np);
      __syncthreads();
    }
    const TC(*AXT)[3][9] = AXT_[cur];
    for (int q = t; q < PG * 5 * BB; q += 256) {
      const int p = q / (5 * BB), beta = (q / BB) % 5, J = q % BB;
      BT(p, beta, J) = (J < 27) ? gcomp<TC>(AXT[p], J, beta) : (TC)0;
    }
    // E_p[I][z][r] = (L_I D_p)[r][z]: u rows sum_b dw/dx_b D[(b,r)] + w D[T_r];
    // the pressure row w D[Q] + sum_b dw/dx_b D[M_b] + (w - w_avg) D[S]
#pragma unroll
    for (int j = 0; j < NQ; ++j) {
      const int q = t + 256 * j;
      if (q >= PG * NI) break;
      const int p = q / NI, zr = q % NI, z = zr >> 2, r = zr & 3;
      const TC d0 = dv[j][0], d1 = dv[j][1], d2 = dv[j][2], dw = dv[j][3], dwa = dv[j][4];
      // sum-factorised over the tensor-product axes: with u = gx d0 + wx dw, v = wx d1,
      // q = wx d2, a = wax dwa per x node, E = wz (wy u + gy v) + gz (wy q) + waz (way a)
      TC wx[3], gx[3], ax[3], wy[3], gy[3], ay[3], wz[3], gz[3], az[3];
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        wx[i] = AXT[p][0][i];
        gx[i] = AXT[p][0][3 + i];
        ax[i] = AXT[p][0][6 + i];
        wy[i] = AXT[p][1][i];
        gy[i] = AXT[p][1][3 + i];
        ay[i] = AXT[p][1][6 + i];
        wz[i] = AXT[p][2][i];
        gz[i] = AXT[p][2][3 + i];
        az[i] = AXT[p][2][6 + i];
      }
#pragma unroll
      for (int ix = 0; ix < 3; ++ix) {
        const TC u = gx[ix] * d0 + wx[ix] * dw, v = wx[ix] * d1, qx = wx[ix] * d2, a = ax[ix] * dwa;
#pragma unroll
        for (int iy = 0; iy < 3; ++iy) {
          const TC U = wy[iy] * u + gy[iy] * v, Q = wy[iy] * qx, A2 = ay[iy] * a;
#pragma unroll
          for (int iz = 0; iz < 3; ++iz) E(p, ix + 3 * iy + 9 * iz, z, r) = wz[iz] * U + gz[iz] * Q + az[iz] * A2;
        }
      }
    }
    // the next group: the rest of this bin, else the first of the next non-empty bin
    int nb = b, nks = ks, nke = ke, np0 = p0 + PG;
    const bool bin_done = np0 >= ke;
    if (bin_done) {
      for (nb = b + gridDim.x; nb < n_bins; nb += gridDim.x) {
        nks = cell_start[nb];
        nke = cell_start[nb + 1];
        if (nke > nks) break;
      }
      np0 = nks;
    }
    const bool more = nb < n_bins;
    if (PF && more) load_group(np0, min(PG, nke - np0));
    __syncthreads();  // E and B tables complete
    // particles past np have all-zero axis tables, hence zero B
#pragma unroll
    for (int kst = 0; kst < KST; ++kst) {
      const int beta = kst % 5, pb = (kst / 5) * 4;  // constants once unrolled
      const TC bk = BT_[bbase + pb * BP + beta * BB];
      // the step's A operands are read before its products are issued
      TC av[4][4];
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const int z = zsel(c, beta);
          av[s][c] = (z == ZERO) ? (TC)0 : E_[abase[s] + pb * EP + z * 4];  // z resolved at compile time
        }
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        if (s == 3 && wave >= 2) break;  // wave-uniform: no fourth tile
#pragma unroll
        for (int c = 0; c < 4; ++c)
          if (zsel(c, beta) != ZERO) acc[s][c] = Mfma<TC>::step(av[s][c], bk, acc[s][c]);
      }
    }
    if (bin_done) {
      // lane holds rows r = 0..3 of node I_loc = 4 mt + lane / 16 in column J_loc =
      // 16 nt + lane % 16: one whole 4 x 4 block
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int mt = (wave >> 1) + 2 * s, nt = wave & 1;
        const int I = mt * 4 + (lane >> 4), J = nt * 16 + (lane & 15);
        if (I < 27 && J < 27) {
          TC* o = cb + chunk_at(I, b) + J * 16;
#pragma unroll
          for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int c = 0; c < 4; ++c) o[r * 4 + c] = acc[s][c][r];
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[s][c] = ACC{0, 0, 0, 0};
      }
    }
    if (!more) break;
    if (PF) {
      cur ^= 1;
      axis_tables(cur, min(PG, nke - np0));  // read after the next barrier
    }
    b = nb;
    ks = nks;
    ke = nke;
    p0 = np0;
  }
}

#undef E
#undef BT

// One workgroup per block row I, four lanes per block (one per block row r).  The
// row's 27 candidate bins (b = I - o, -1 when outside the grid or empty) are read
// once into LDS.
template <typename TC, typename TV>
__global__ void __launch_bounds__(512) k_jac_gather(gm_grid g, const int* cell_start, const TC* cb,
                                                    const uint8_t* freem, const int* row_ptr,
                                                    const uint64_t* row_mask, TV* vals) {
  __shared__ int SLOT_BIT[125];
  __shared__ int BIN[27];
  const int I = blockIdx.x, t = threadIdx.x;
  const uint64_t m0 = row_mask[2 * I], m1 = row_mask[2 * I + 1];
  const int nx1 = g.nx + 1, nxy = (g.nx + 1) * (g.ny + 1);
  const int ci[3] = {I % nx1, (I / nx1) % (g.ny + 1), I / nxy};
  if (t < 125) {
    const uint64_t w = (t < 64) ? m0 : m1;
    const int sh = t & 63;
    if ((w >> sh) & 1ull) {
      const int below = (t < 64) ? __popcll(m0 & ((1ull << sh) - 1ull))
                                 : __popcll(m0) + __popcll(m1 & ((1ull << sh) - 1ull));
      SLOT_BIT[below] = t;
    }
  } else if (t >= 128 && t < 128 + 27) {
    const int o = t - 128, ox = o % 3, oy = (o / 3) % 3, oz = o / 9;
    const int bc[3] = {ci[0] - ox, ci[1] - oy, ci[2] - oz};
    int bn = -1;
    if (bc[0] >= 0 && bc[0] <= g.nx && bc[1] >= 0 && bc[1] <= g.ny && bc[2] >= 0 && bc[2] <= g.nz) {
      bn = bc[0] + bc[1] * nx1 + bc[2] * nxy;
      if (cell_start[bn + 1] == cell_start[bn]) bn = -1;
    }
    BIN[o] = bn;
  }
  __syncthreads();
  const int nnz = __popcll(m0) + __popcll(m1);
  const int slot = t >> 2, r = t & 3;
  if (slot >= nnz) return;
  const int bit = SLOT_BIT[slot];
  const int d[3] = {bit % 5 - 2, (bit / 5) % 5 - 2, bit / 25 - 2};
  double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int o = 0; o < 27; ++o) {
    const int kx = d[0] + o % 3, ky = d[1] + (o / 3) % 3, kz = d[2] + o / 9;
    const int bn = BIN[o];
    if (bn >= 0 && kx >= 0 && kx < 3 && ky >= 0 && ky < 3 && kz >= 0 && kz < 3) {
      const TC* src = cb + chunk_at(o, bn) + (kx + 3 * ky + 9 * kz) * 16 + r * 4;
#pragma unroll
      for (int c = 0; c < 4; ++c) s[c] += (double)src[c];
    }
  }
  const int Jn = I + d[0] + d[1] * nx1 + d[2] * nxy;
  const bool diag = (Jn == I);
  const bool fr = freem[I * 4 + r];
  TV* out = vals + (long)(row_ptr[I] + slot) * 16 + r * 4;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const bool fc = freem[Jn * 4 + c];
    double v = (fr && fc) ? -s[c] : 0.0;
    if (diag && r == c && !fr) v = 1.0;
    out[c] = (TV)v;
  }
}

// The same sums with coalesced reads: one workgroup per block row I stages the row's
// <= 27 bin chunks (bin I - o, I_loc = o: 27 blocks, contiguous) in LDS
// with whole 16-byte vector loads, OB chunks at a time, and every (block, row r) item
// then adds its <= 27 contributions from LDS in the same order (o = 0..26) as
// k_jac_gather: both write the same bits.
template <typename TC, typename TV, int OB>
__global__ void __launch_bounds__(256, 3) k_jac_gather_staged(gm_grid g, const int* cell_start, const TC* cb,
                                                           const uint8_t* freem, const int* row_ptr,
                                                           const uint64_t* row_mask, TV* vals) {
  static_assert(27 % OB == 0, "chunk rounds cover o = 0..26");
  constexpr int CH = 27 * 16;          // values per chunk
  constexpr int CV = CH * sizeof(TC) / 16;  // 16-byte vectors per chunk
  typedef uint32_t u4 __attribute__((ext_vector_type(4)));
  __shared__ int SLOT_BIT[125];
  __shared__ int BIN[27];
  __shared__ u4 ST[OB][CV];
  const int I = blockIdx.x, t = threadIdx.x;
  const uint64_t m0 = row_mask[2 * I], m1 = row_mask[2 * I + 1];
  const int nx1 = g.nx + 1, nxy = (g.nx + 1) * (g.ny + 1);
  const int ci[3] = {I % nx1, (I / nx1) % (g.ny + 1), I / nxy};
  if (t < 125) {
    const uint64_t w = (t < 64) ? m0 : m1;
    const int sh = t & 63;
    if ((w >> sh) & 1ull) {
      const int below = (t < 64) ? __popcll(m0 & ((1ull << sh) - 1ull))
                                 : __popcll(m0) + __popcll(m1 & ((1ull << sh) - 1ull));
      SLOT_BIT[below] = t;
    }
  } else if (t >= 128 && t < 128 + 27) {
    const int o = t - 128, ox = o % 3, oy = (o / 3) % 3, oz = o / 9;
    const int bc[3] = {ci[0] - ox, ci[1] - oy, ci[2] - oz};
    int bn = -1;
    if (bc[0] >= 0 && bc[0] <= g.nx && bc[1] >= 0 && bc[1] <= g.ny && bc[2] >= 0 && bc[2] <= g.nz) {
      bn = bc[0] + bc[1] * nx1 + bc[2] * nxy;
      if (cell_start[bn + 1] == cell_start[bn]) bn = -1;
    }
    BIN[o] = bn;
  }
  __syncthreads();
  const int nnz = __popcll(m0) + __popcll(m1);
  // items (slot, r) = (it / 4, it % 4), it = t and t + 256
  int dd[2][3];
  bool live[2];
  double s[2][4];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int it = t + 256 * h;
    live[h] = it < 4 * nnz;
    const int bit = live[h] ? SLOT_BIT[it >> 2] : 62;
    dd[h][0] = bit % 5 - 2;
    dd[h][1] = (bit / 5) % 5 - 2;
    dd[h][2] = bit / 25 - 2;
#pragma unroll
    for (int c = 0; c < 4; ++c) s[h][c] = 0.0;
  }
#pragma unroll 1
  for (int o0 = 0; o0 < 27; o0 += OB) {
    if (o0) __syncthreads();  // the previous round's LDS reads are done
    // all of a thread's loads are issued before its first LDS store
    constexpr int NJ = (OB * CV + 255) / 256;
    u4 tmp[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int q = t + 256 * j;
      tmp[j] = u4{0u, 0u, 0u, 0u};
      if (q < OB * CV) {
        const int oo = q / CV, f = q % CV;
        const int bn = BIN[o0 + oo];
        if (bn >= 0) tmp[j] = reinterpret_cast<const u4*>(cb + chunk_at(o0 + oo, bn))[f];
      }
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int q = t + 256 * j;
      if (q < OB * CV) ST[q / CV][q % CV] = tmp[j];
    }
    __syncthreads();
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (!live[h]) continue;
      const int r = (t + 256 * h) & 3;
#pragma unroll 3
      for (int oo = 0; oo < OB; ++oo) {
        const int o = o0 + oo;
        const int kx = dd[h][0] + o % 3, ky = dd[h][1] + (o / 3) % 3, kz = dd[h][2] + o / 9;
        if (BIN[o] >= 0 && kx >= 0 && kx < 3 && ky >= 0 && ky < 3 && kz >= 0 && kz < 3) {
          const TC* src = reinterpret_cast<const TC*>(&ST[oo][0]) + (kx + 3 * ky + 9 * kz) * 16 + r * 4;
#pragma unroll
          for (int c = 0; c < 4; ++c) s[h][c] += (double)src[c];
        }
      }
    }
  }
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    if (!live[h]) continue;
    const int it = t + 256 * h, slot = it >> 2, r = it & 3;
    const int Jn = I + dd[h][0] + dd[h][1] * nx1 + dd[h][2] * nxy;
    const bool diag = (Jn == I);
    const bool fr = freem[I * 4 + r];
    TV* out = vals + (long)(row_ptr[I] + slot) * 16 + r * 4;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const bool fc = freem[Jn * 4 + c];
      double v = (fr && fc) ? -s[h][c] : 0.0;
      if (diag && r == c && !fr) v = 1.0;
      out[c] = (TV)v;
    }
  }
}

// Line sums.  A workgroup takes the bins of one segment [xs, xe) of a bin line (fixed y, z)
// in ascending x.  The nodes x, x + 1, x + 2 that a bin reaches lie in the three slots
// node_x mod 3, so that from one bin to the next two of the three node planes stay where
// they are: the accumulators of the matrix cores (27 row nodes x 27 column nodes x 4 x 4)
// keep summing, and only the pairs that the next bin does not reach (the row or the column
// node is x: 405 of 729 blocks) are stored and cleared.  Pairs that bins before xs reach as
// well belong to this segment when min(row x, column x) >= xs; the sweep starts two bins
// early to have their whole sum.
// A bin's particles are taken four at a time (a group).  The first four waves hold the
// accumulators (four tiles each) and do nothing but products and stores.  The other four
// prepare E_p and the B operand of the coming group in the other half of the LDS buffers,
// stage the tangent rows and shape-function tables of the group after it and load the rows of
// the next ones: one barrier a group, and neither the tables nor the loads are in the matrix
// cores' way.
// K order: a K step of the MFMA is one shape-function component beta and the four
// particles (lane group l / 16 = particle).  After the
// K loop unrolls, every A and B operand address is a per-lane base plus an immediate,
// and the (c, beta) products that vanish (u columns: no w term except the penalty
// on u_z, no w_avg term) are not issued.  Every segment length adds the same products in
// the same order, so all of them write the same bits.
__global__ void __launch_bounds__(512, 2) k_jac_line(gm_grid g, const double* x_s, const double* lp_s,
                                                     const int* cell_start, int n_p, int seg_len, int n_seg,
                                                     const double* D, double* cb) {
  constexpr int CW = 4;             // product waves
  constexpr int TILES = 16 / CW;
  constexpr int PG = 4;             // particles of a group: one quad of K steps
  constexpr int NI = 4 * NZ;        // (z, r) entries of a node row of E_p
  // shape-function tables of the sweep's particles, a ring filled a batch at a time
  constexpr int RING = 32, BATCH = 16;
  __shared__ double AXT_[RING][3][9];
  // tangent rows of a group (particles are in bin order, so a group's rows are contiguous)
  constexpr int DROW = NY * NZ;
  __shared__ double DR_[2][PG * DROW];
  // E_p[I][z][r] (r fastest), node rows 68 entries apart and particles 1840: the 64
  // (particle, I, r) entries a wave reads at once fall in 64 distinct banks.  (The padding
  // rows of the last row tile read row 26; they are never stored.)
  constexpr int EI = 68, EP = 27 * EI + 4;
  __shared__ double E_[2][PG * EP];
  // B operand g_p[J][beta], J padded to 32 with zeros, particles 176 entries apart
  constexpr int BB = 32, BP = 5 * BB + 16;
  __shared__ double BT_[2][PG * BP];
  const int line = blockIdx.x / n_seg;  // y + (ny + 1) z
  const int lb = line * (g.nx + 1);     // the line's first bin (and node)
  const int xs = (blockIdx.x % n_seg) * seg_len, xe = min(xs + seg_len, g.nx + 1);
  const int x0 = max(xs - 2, 0);
  if (xs >= xe || cell_start[lb + x0] == cell_start[lb + xe]) return;  // uniform across the workgroup
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform across the wave
  // cell_start of the segment's bins, one a lane
  const int starts = cell_start[lb + min(x0 + lane, xe)];
  // the groups of the sweep, in order: bin x, first particle p0, end of the bin ke
  struct Group {
    int x, p0, ke;
  };
  auto cs = [&](int x) { return __builtin_amdgcn_readlane(starts, x - x0); };
  auto seek = [&](Group& q) {  // the first non-empty bin from q.x on (q.x = xe: none)
    if (q.x >= xe) return;
    int first = cs(q.x), end = cs(q.x + 1);
    while (first == end && ++q.x < xe) end = cs(q.x + 1);
    q.p0 = first;
    q.ke = end;
  };
  auto next = [&](Group q) {
    if (q.x >= xe) return q;
    q.p0 += PG;
    if (q.p0 >= q.ke) {
      ++q.x;
      seek(q);
    }
    return q;
  };
  Group cur{x0, 0, 0};
  seek(cur);
  // shape-function tables of particles [tabs, tabs + BATCH) of the sweep: 48 lanes of the last
  // product wave, which has a row tile less than the first ones, from positions loaded one batch
  // ahead (one wave's FP64 chain a batch rather than a group)
  const int ps = cs(x0), n_sweep = cs(xe) - ps;
  const int tl = wave == CW - 1 ? lane : -1;
  const int tp = tl >= 0 && tl < 3 * BATCH ? tl / 3 : 0, ta = tl >= 0 ? tl % 3 : 0;
  int tabs = 0;
  double xa, la;
  auto load_tables = [&](int e) {
    const long at = (long)(ps + min(e + tp, n_sweep - 1)) * 3 + ta;
    xa = x_s[at];
    la = lp_s[at];
  };
  // the tables of group q (none: the sweep ends before it)
  auto tables_for = [&](const Group& q) {
    if ((q.x < xe ? min(q.p0 + PG, q.ke) - ps : n_sweep) <= tabs) return;  // uniform
    if (tl >= 0 && tl < 3 * BATCH) {
      const Axis ax = gimp_axis(xa, la, g.h[ta], g.inv_h[ta]);
      double* T = AXT_[(tabs + tp) % RING][ta];
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        T[i] = ax.w[i];
        T[3 + i] = ax.g[i];
        T[6 + i] = ax.wa[i];
      }
    }
    tabs += BATCH;
    load_tables(tabs);
  };
  if (wave < CW) {
    // ---------------------------------------------------------------- products
    d4v acc[TILES][4];
#pragma unroll
    for (int s = 0; s < TILES; ++s)
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[s][c] = d4v{0, 0, 0, 0};
    // output tiles w + CW s: row tile mt = w / 2 + CW / 2 s (16 rows (I, r)), column tile
    // nt = w % 2 (16 columns J); the last waves have no last tile (rows I >= 28).  Node index
    // I = 9 slot + oy + 3 oz, J likewise.
    const int w = wave;
    const bool last = (w >> 1) + (CW >> 1) * (TILES - 1) < 7;
    const int lg = lane >> 4, rt = lane & 15;
    const int r_l = rt >> 2, i_l = rt & 3;  // r-major tiles
    int abase[TILES];
#pragma unroll
    for (int s = 0; s < TILES; ++s)
      abase[s] = lg * EP + min(((w >> 1) + (CW >> 1) * s) * 4 + i_l, 26) * EI + r_l;
    const int bbase = lg * BP + (w & 1) * 16 + rt;
    // the pairs whose first node in x is B leave: stored when the segment owns them, cleared
    auto flush = [&](int B) {
      const int q = B % 3;
      // (the lane's nodes are worked out here, behind the compiler's back, rather than kept in
      // registers that the accumulators need)
      int l = lane;
      asm volatile("" : "+v"(l));
      const int J = (w & 1) * 16 + (l & 15), jslot = J / 9, jyz = J % 9;
#pragma unroll
      for (int s = 0; s < TILES; ++s) {
        const int I = ((w >> 1) + (CW >> 1) * s) * 4 + (l >> 4), islot = I / 9, iyz = I - 9 * islot;
        if (I < 27 && J < 27 && (islot == q || jslot == q)) {
          const int di = islot >= q ? islot - q : islot - q + 3, dj = jslot >= q ? jslot - q : jslot - q + 3;
          if (B >= xs && B + di <= g.nx) {
            double* o = cb + (di == 0 ? chunk_a(iyz, lb + B) + (dj * 9 + jyz) * 4 : chunk_b(iyz, lb + B, di) + jyz * 4);
            const int plane = di == 0 ? 27 * 4 : 9 * 4;
#pragma unroll
            for (int c = 0; c < 4; ++c) *reinterpret_cast<d4v*>(o + c * plane) = acc[s][c];
          }
#pragma unroll
          for (int c = 0; c < 4; ++c) acc[s][c] = d4v{0, 0, 0, 0};
        }
      }
    };
    Group gt = cur;  // the group whose tables come next
    if (wave == CW - 1) {
      load_tables(0);
      tables_for(gt);
      gt = next(gt);
      tables_for(gt);
    }
    __syncthreads();
    __syncthreads();
    for (int buf = 0; cur.x < xe; buf ^= 1) {
      if (wave == CW - 1) {
        gt = next(gt);
        tables_for(gt);
      }
      // particles past the bin's last have zero B; a tile's operands are read before its products
      const double *E = E_[buf], *BT = BT_[buf];
      double b[5];
#pragma unroll
      for (int beta = 0; beta < 5; ++beta) b[beta] = BT[bbase + beta * BB];
#pragma unroll
      for (int s = 0; s < TILES; ++s) {
        if (s == TILES - 1 && !last) break;  // wave-uniform
        double a[4][5];
#pragma unroll
        for (int beta = 0; beta < 5; ++beta)
#pragma unroll
          for (int c = 0; c < 4; ++c)
            if (zsel(c, beta) != ZERO) a[c][beta] = E[abase[s] + zsel(c, beta) * 4];
#pragma unroll
        for (int beta = 0; beta < 5; ++beta)
#pragma unroll
          for (int c = 0; c < 4; ++c)  // (c, beta) resolved at compile time
            if (zsel(c, beta) != ZERO) acc[s][c] = Mfma<double>::step(a[c][beta], b[beta], acc[s][c]);
      }
      const Group nxt = next(cur);
      // after the bin's last group; up to three steps clear every pair the sweep has touched
      if (nxt.x != cur.x)
        for (int B = cur.x; B < min(min(nxt.x, cur.x + 3), xe); ++B) flush(B);
      cur = nxt;
      __syncthreads();
    }
    return;
  }
  // ------------------------------------------------------------------ operands
  const int t = threadIdx.x - 64 * CW;
  constexpr int VD = 2;  // tangent values per load
  constexpr int ND = (PG * DROW + 256 * VD - 1) / (256 * VD);
  typedef double dvec __attribute__((ext_vector_type(2), aligned(8)));
  // tangent rows of a group: addresses clamped rather than loads skipped, so that the loads
  // of two groups stay in flight (a skipped load leaves the count of those in flight unknown)
  dvec even[ND], odd[ND];
  auto load_group = [&](const Group& q, dvec* to) {
#pragma unroll
    for (int j = 0; j < ND; ++j)
      to[j] = *reinterpret_cast<const dvec*>(
          D + min((long)q.p0 * DROW + (t + 256 * j) * VD, (long)n_p * DROW - VD));
  };
  auto stage_group = [&](const Group& q, int buf, const dvec* from) {
    const long lim = min((long)q.p0 + PG, (long)q.ke) * DROW, k0 = (long)q.p0 * DROW;
#pragma unroll
    for (int j = 0; j < ND; ++j) {
      const int k = (t + 256 * j) * VD;
      // (at the array's end the loaded vector starts before k0 + k)
      const int back = (int)max(k0 + k - ((long)n_p * DROW - VD), 0L);
#pragma unroll
      for (int i = 0; i < VD; ++i) {
        double v = from[j][i];
        if (back > 0) v = i + back < VD ? from[j][min(i + back, VD - 1)] : 0.0;
        if (k + i < PG * DROW) DR_[buf][k + i] = k0 + k + i < lim ? v : 0.0;
      }
    }
  };
  auto operands = [&](const Group& q, int buf) {
    const int np = min(PG, q.ke - q.p0), rot = q.x % 3;  // node ox of the bin lies in slot (ox + rot) % 3
    // B operand: threads (J, particle)
    if (t < PG * 32) {
      const int p = t >> 5, Jb = t & 31;
      double* B = BT_[buf] + p * BP + Jb;
      const double(*AX)[9] = AXT_[(q.p0 - ps + p) % RING];
      if (Jb < 27 && p < np) {
        const int js = Jb / 9, sx = js >= rot ? js - rot : js - rot + 3, jy = Jb % 3, jz = (Jb / 3) % 3;
        const double wx = AX[0][sx], wy = AX[1][jy], wz = AX[2][jz];
        B[0] = (wx * wy * wz);
        B[BB] = (AX[0][3 + sx] * wy * wz);
        B[2 * BB] = (wx * AX[1][3 + jy] * wz);
        B[3 * BB] = (wx * wy * AX[2][3 + jz]);
        B[4 * BB] = (AX[0][6 + sx] * AX[1][6 + jy] * AX[2][6 + jz]);
      } else {
#pragma unroll
        for (int beta = 0; beta < 5; ++beta) B[beta * BB] = 0;
      }
    }
    // E_p[I][z][r] = (L_I D_p)[r][z]: u rows sum_b dw/dx_b D[(b,r)] + w D[T_r];
    // the pressure row w D[Q] + sum_b dw/dx_b D[M_b] + (w - w_avg) D[S]
    if (t < PG * NI) {
      const int p = t / NI, zr = t % NI, z = zr >> 2, r = zr & 3;
      const double* Dp = DR_[buf] + p * DROW + z;
      const int k0 = r < 3 ? r : Y_M, dk = r < 3 ? 3 : 1;
      const double d0 = Dp[k0 * NZ], d1 = Dp[(k0 + dk) * NZ], d2 = Dp[(k0 + 2 * dk) * NZ];
      const double dS = r < 3 ? 0.0 : Dp[Y_S * NZ];
      const double dw = Dp[(r < 3 ? Y_T + r : Y_Q) * NZ] + dS, dwa = -dS;
      // sum-factorised over the tensor-product axes: with u = gx d0 + wx dw, v = wx d1,
      // q = wx d2, a = wax dwa per x node, E = wz (wy u + gy v) + gz (wy q) + waz (way a)
      double wy[3], gy[3], ay[3], wz[3], gz[3], az[3];
      const double(*AX)[9] = AXT_[(q.p0 - ps + min(p, np - 1)) % RING];  // past the bin's last: zero tangent
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        wy[i] = AX[1][i];
        gy[i] = AX[1][3 + i];
        ay[i] = AX[1][6 + i];
        wz[i] = AX[2][i];
        gz[i] = AX[2][3 + i];
        az[i] = AX[2][6 + i];
      }
#pragma unroll
      for (int ix = 0; ix < 3; ++ix) {
        double* Eo = E_[buf] + p * EP + zr + 9 * EI * (ix + rot >= 3 ? ix + rot - 3 : ix + rot);
        const double wx = AX[0][ix], u = AX[0][3 + ix] * d0 + wx * dw, v = wx * d1, qx = wx * d2, a = AX[0][6 + ix] * dwa;
#pragma unroll
        for (int iy = 0; iy < 3; ++iy) {
          const double U = wy[iy] * u + gy[iy] * v, Q = wy[iy] * qx, A2 = ay[iy] * a;
#pragma unroll
          for (int iz = 0; iz < 3; ++iz) Eo[(iy + 3 * iz) * EI] = (wz[iz] * U + gz[iz] * Q + az[iz] * A2);
        }
      }
    }
  };
  Group g0 = cur, g1 = next(g0), g2 = next(g1), g3 = next(g2);
  load_group(g0, even);
  load_group(g1, odd);
  stage_group(g0, 0, even);
  load_group(g2, even);
  __syncthreads();
  operands(g0, 0);
  stage_group(g1, 1, odd);
  load_group(g3, odd);
  __syncthreads();
  // while the products of group i run: the operands of i + 1, the rows and tables of i + 2,
  // and the loads of i + 3 and i + 4 on their way
  while (cur.x < xe) {
    if (g1.x < xe) operands(g1, 1);
    stage_group(g2, 0, even);
    const Group g4 = next(g3);
    load_group(g4, even);
    __syncthreads();
    cur = next(cur);
    if (cur.x >= xe) break;
    if (g2.x < xe) operands(g2, 0);
    stage_group(g3, 1, odd);
    g1 = g3;
    g2 = g4;
    g3 = next(g4);
    load_group(g3, odd);
    __syncthreads();
    cur = next(cur);
  }
}

// One workgroup per block row I, one thread per window position and 128 / T column dofs:
// the <= 9 line sums of its four rows, all loads issued before the first is added.  Both
// the reads (runs of 16-byte vectors) and the writes (the row's blocks, through LDS) are
// coalesced; bound by HBM on the workspace and the matrix.
template <typename TV, int T>
__global__ void __launch_bounds__(T) k_jac_line_gather(gm_grid g, const int* cell_start, const double* cb,
                                                       const uint8_t* freem, const int* row_ptr,
                                                       const uint64_t* row_mask, TV* vals) {
  __shared__ int NODE[9], MASK[9];
  __shared__ __align__(16) TV OUT[125 * 16];
  const int I = blockIdx.x, t = threadIdx.x;
  const int nx1 = g.nx + 1, nxy = nx1 * (g.ny + 1);
  if (t < 9) {
    // the nine lines (y - oy, z - oz) holding the row: the row node's node there, and the
    // dx (bit dx + 2) that a non-empty bin reaches
    const int oy = t % 3, oz = t / 3;
    const int cx = I % nx1, cy = (I / nx1) % (g.ny + 1) - oy, cz = I / nxy - oz;
    int node = 0, mask = 0;
    if (cy >= 0 && cz >= 0) {
      node = cx + cy * nx1 + cz * nxy;
#pragma unroll
      for (int k = 0; k < 3; ++k)  // bin cx - k reaches the nodes cx - k .. cx - k + 2
        if (cx - k >= 0 && cell_start[node - k + 1] > cell_start[node - k]) mask |= 7 << (2 - k);
    }
    NODE[t] = node;
    MASK[t] = mask;
  }
  const uint64_t m0 = row_mask[2 * I], m1 = row_mask[2 * I + 1];
  const int nnz = __popcll(m0) + __popcll(m1);
  // thread order (dx, dz, dy): neighbouring threads read neighbouring vectors of a chunk
  const int u = t & 127;
  const int dy = u % 5 - 2, dz = (u / 5) % 5 - 2, dx = u / 25;  // dx: offset + 2
  const int bit = dx + 5 * (dy + 2) + 25 * (dz + 2);
  const bool live = u < 125 && (((bit < 64 ? m0 : m1) >> (bit & 63)) & 1ull);
  const int slot = bit < 64 ? __popcll(m0 & ((1ull << (bit & 63)) - 1ull))
                            : __popcll(m0) + __popcll(m1 & ((1ull << (bit & 63)) - 1ull));
  __syncthreads();
  // all column dofs of a thread in flight (1.95 -> 1.83 ms)
#pragma unroll
  for (int c0 = 0; c0 < 4 * 128 / T; ++c0) {
    const int c = (t >> 7) + c0 * (T / 128);
    d4v v[9];
    bool on[9];
#pragma unroll
    for (int o = 0; o < 9; ++o) {
      const int ky = dy + o % 3, kz = dz + o / 3, k = ky + 3 * kz, n = NODE[o];
      on[o] = live && ky >= 0 && ky < 3 && kz >= 0 && kz < 3 && ((MASK[o] >> dx) & 1);
      const long at = dx >= 2 ? chunk_a(o, n) + (c * 27 + (dx - 2) * 9 + k) * 4
                              : chunk_b(o, n + dx - 2, 2 - dx) + (c * 9 + k) * 4;
      v[o] = *reinterpret_cast<const d4v*>(cb + (on[o] ? at : 0L));
    }
    double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int o = 0; o < 9; ++o)
#pragma unroll
      for (int r = 0; r < 4; ++r) s[r] += on[o] ? v[o][r] : 0.0;
    if (live) {  // masks, sign, identity rows
      const int Jn = I + (dx - 2) + dy * nx1 + dz * nxy;
      const bool diag = (Jn == I), fc = freem[Jn * 4 + c];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bool fr = freem[I * 4 + r];
        double w = (fr && fc) ? -s[r] : 0.0;
        if (diag && r == c && !fr) w = 1.0;
        OUT[slot * 16 + r * 4 + c] = (TV)w;
      }
    }
  }
  __syncthreads();
  constexpr int PER = 16 / sizeof(TV);  // values per store
  typedef TV vec __attribute__((ext_vector_type(16 / sizeof(TV))));
  vec* row = reinterpret_cast<vec*>(vals + (long)row_ptr[I] * 16);
  for (int q = t; q < nnz * 16 / PER; q += T) row[q] = reinterpret_cast<const vec*>(OUT)[q];
}

// ================================================================== residual (3D u-p)
// r_I = sum_p L_I Y_p per bin (node I_loc of the bin's 3x3x3 box, its particles in bin order), then
// per node the fixed-order sum over the <= 27 bins holding it.
// A wave per bin: tables and rows of Y staged in its LDS together; two lanes a node take two dofs
// each and walk the particles one after the other (a load step depends on the order, see
// k_update_lp).  A bin without particles writes zeros, so that the gather has nothing to look up
// before its 27 loads.  Bound by the LDS reads (18 and 22 a lane and particle).  With the gather,
// 64 x 64 x 32 cells 222 us, 33 x 29 x 15 33, 12 x 9 x 7 12; with a lane per node reading Y from
// memory, and a gather that looked at every bin first, 233, 43 and 27; with the particles shared
// out to five groups of lanes, whose sums are added at the end, 194, 28 and 12, in another order.
constexpr int RES_PB = 10;
__global__ void __launch_bounds__(256) k_res_bin(gm_grid g, const double* x_s, const double* lp_s,
                                                 const int* cell_start, const double* Y, double* cb) {
  __shared__ struct {
    double ax[RES_PB][3][9], y[RES_PB * NY];
  } sh[4];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int b = blockIdx.x * 4 + wave;
  if (b >= g.n_nodes) return;  // the whole wave
  auto& S_ = sh[wave];
  const int ks = cell_start[b], ke = cell_start[b + 1];
  auto sync = [] {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  const int node = min(lane >> 1, 26), ix = node % 3, iy = node / 3 % 3, iz = node / 9;
  const bool odd = lane & 1;  // dofs 0 and 1, or 2 and 3 (the pressure's)
  const int c = odd ? 2 : 0;
  // the second dof's terms, in their order: three gradients and the body force, or a gradient, the
  // mass balance, two gradients and the PPP term
  const int q0 = odd ? Y_M : 1, q1 = odd ? Y_Q : 4, q2 = odd ? Y_M + 1 : 7, q3 = odd ? Y_M + 2 : Y_T + 1;
  double r0 = 0.0, r1 = 0.0;
  for (int p0 = ks; p0 < ke; p0 += RES_PB) {
    const int np = min(RES_PB, ke - p0);
    sync();
#pragma unroll
    for (int q = 0; q < (RES_PB * NY + 63) / 64; ++q) {
      const int k = q * 64 + lane;
      if (k < np * NY) S_.y[k] = Y[(long)p0 * NY + k];
    }
    if (lane < 3 * np) {
      const int a = lane % 3;
      const Axis ax = gimp_axis(x_s[(long)p0 * 3 + lane], lp_s[(long)p0 * 3 + lane], g.h[a], g.inv_h[a]);
      double* T = S_.ax[lane / 3][a];
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        T[i] = ax.w[i];
        T[3 + i] = ax.g[i];
        T[6 + i] = ax.wa[i];
      }
    }
    sync();
    for (int p = 0; p < np; ++p) {
      const double *X = S_.ax[p][0], *V = S_.ax[p][1], *W = S_.ax[p][2], *yp = S_.y + p * NY;
      const double wx = X[ix], wy = V[iy], wz = W[iz], w = wx * wy * wz;
      const double G0 = X[3 + ix] * wy * wz, G1 = wx * V[3 + iy] * wz, G2 = wx * wy * W[3 + iz];
      const double wa = X[6 + ix] * V[6 + iy] * W[6 + iz];
      r0 += fma(w, yp[Y_T + c], fma(G2, yp[6 + c], fma(G1, yp[3 + c], G0 * yp[c])));
      const double t = fma(odd ? G2 : w, yp[q3], fma(odd ? G1 : G2, yp[q2], fma(odd ? w : G1, yp[q1], G0 * yp[q0])));
      r1 += odd ? fma(w - wa, yp[Y_S], t) : t;
    }
  }
  if (lane < 54) {
    cb[((long)b * 27 + node) * 4 + c] = r0;
    cb[((long)b * 27 + node) * 4 + c + 1] = r1;
  }
}

__global__ void __launch_bounds__(256) k_res_gather(gm_grid g, const double* cb, const uint8_t* freem, double* rhs) {
  const int I = blockIdx.x * 64 + threadIdx.x / 4, c = threadIdx.x % 4;
  if (I >= g.n_nodes) return;
  const int nx1 = g.nx + 1, nxy = (g.nx + 1) * (g.ny + 1);
  const int cx = I % nx1, cy = (I / nx1) % (g.ny + 1), cz = I / nxy;
  double v[27];
#pragma unroll
  for (int o = 0; o < 27; ++o) {
    const bool on = cx >= o % 3 && cy >= o / 3 % 3 && cz >= o / 9;
    const int bn = on ? I - o % 3 - o / 3 % 3 * nx1 - o / 9 * nxy : I;
    v[o] = cb[((long)bn * 27 + o) * 4 + c];
  }
  const bool fr = freem[I * 4 + c];
  double s = 0.0;
#pragma unroll
  for (int o = 0; o < 27; ++o) s += cx >= o % 3 && cy >= o / 3 % 3 && cz >= o / 9 ? v[o] : 0.0;
  rhs[I * 4 + c] = fr ? s : 0.0;
}

extern "C" size_t gm_residual_work_bytes(const gm_grid* g) {
  return g ? (size_t)g->n_nodes * 27 * 4 * sizeof(double) : 0;
}

extern "C" int gm_node_residual_binned(const gm_grid* g, const gm_bins* b, const double* Y, const uint8_t* freem,
                                       double* rhs, void* work, size_t work_bytes, hipStream_t s) {
  GM_REQUIRE(g && b && Y && freem && rhs && work, "gm_node_residual_binned: null argument");
  GM_REQUIRE(g->dim == 3 && g->nb == 4, "gm_node_residual_binned: the 3D u-p form only");
  GM_REQUIRE(work_bytes >= gm_residual_work_bytes(g),
             "gm_node_residual_binned: workspace smaller than gm_residual_work_bytes");
  const int n = g->n_nodes;
  if (n == 0) return 0;
  k_res_bin<<<gm_blocks(n, 4), 256, 0, s>>>(*g, b->x_s, b->lp_s, b->cell_start, Y, (double*)work);
  GM_LAUNCH_CHECK();
  k_res_gather<<<gm_blocks(n, 64), 256, 0, s>>>(*g, (const double*)work, freem, rhs);
  GM_LAUNCH_CHECK();
  return 0;
}

// ================================================================== consistent mass
// M_IJ = sum_p m_p w_I w_J in the node pattern (one value per block slot), gathered by strips of
// 21 consecutive node rows.  A workgroup has a wave per stencil offset of the last axis (oz; oy in
// 2D); in it a lane per row and column offset of that axis sums the row's 5 (x 5 in 3D) entries in
// registers.  A stencil line's candidates lie in consecutive bins, so their weights are one range
// of particles, staged C at a time: weight-major, and particles eight apart next to each other, so
// that the rows of a wave read different banks.  The waves' sums are added in LDS in order.
// Bound by those LDS reads (8 a particle and lane in 3D).  1,048,576 particles, 139,425 rows: 414 us;
// 11,628 2D rows: 12 us, against 110 for a thread a row adding to its entries in memory.  Pieces of
// 64, 128 and 192 particles: 510, 478 and 493 us (what a lane waits for its bins in longer ranges
// against the wavefronts their LDS leaves); strips of 10 rows with two lanes for a bin's particles: 403.
constexpr int MASS_ROWS = 21;

template <int DIM>
__global__ void __launch_bounds__(192) k_mass_strip(gm_grid g, const double* x_s, const double* lp_s,
                                                    const int* cell_start, double p_mass, const int* row_ptr,
                                                    const uint64_t* row_mask, double* mvals) {
  constexpr int C = 96, W = DIM == 3 ? 125 : 25, NL = DIM == 3 ? 3 : 1, ND = DIM == 3 ? 5 : 1;
  constexpr int OS = W;  // odd
  __shared__ union {
    double w[3][3 * DIM][C];
    double out[MASS_ROWS * OS];
  } sh;
  const int lane = threadIdx.x & 63, row = lane / 3, jl = lane % 3;
  const int ol = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  double(*T)[C] = sh.w[ol];
  // consecutive strips on one XCD: the lines of one are read again by its neighbours
  const int nw = gridDim.x, x8 = blockIdx.x % 8, I0 = (x8 * (nw / 8) + min(x8, nw % 8) + blockIdx.x / 8) * MASS_ROWS;
  const int nx1 = g.nx + 1, nxy = nx1 * (g.ny + 1), I = I0 + row;
  const bool on = row < MASS_ROWS && I < g.n_nodes;
  const int cx = I % nx1, cy = DIM == 3 ? (I / nx1) % (g.ny + 1) : I / nx1, cz = DIM == 3 ? I / nxy : 0;
  double acc[ND][5];  // [dy + 2][dx + 2]
#pragma unroll
  for (int j = 0; j < ND; ++j)
#pragma unroll
    for (int d = 0; d < 5; ++d) acc[j][d] = 0.0;
  auto sync = [] {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  auto at = [](int k) { return (k & 7) * (C / 8) + (k >> 3); };
#pragma unroll
  for (int oy = 0; oy < NL; ++oy) {
    // the line's bins: those of the strip's rows at offset (., oy, ol) (2D: (., ol))
    const int o = DIM == 3 ? oy * nx1 + ol * nxy : ol * nx1;
    const int b0 = max(I0 - 2 - o, 0), b1 = min(I0 + MASS_ROWS, g.n_nodes) - 1 - o;
    const int lo = b1 >= b0 ? cell_start[b0] : 0, hi = b1 >= b0 ? cell_start[b1 + 1] : 0;
    int ks[3], ke[3];
#pragma unroll
    for (int ox = 0; ox < 3; ++ox) {
      const bool ok = on && cx >= ox && (DIM == 3 ? cy >= oy && cz >= ol : cy >= ol);
      const int b = I - ox - o;
      ks[ox] = ok ? cell_start[b] : 0;
      ke[ox] = ok ? cell_start[b + 1] : 0;
    }
    for (int k0 = lo; k0 < hi; k0 += C) {
      sync();
      for (int q = lane; q < DIM * min(C, hi - k0); q += 64) {
        const int k = q / DIM, a = q % DIM;
        const Axis ax = gimp_axis(x_s[(long)k0 * DIM + q], lp_s[(long)k0 * DIM + q], g.h[a], g.inv_h[a]);
#pragma unroll
        for (int i = 0; i < 3; ++i) T[3 * a + i][at(k)] = ax.w[i];
      }
      sync();
#pragma unroll
      for (int ox = 0; ox < 3; ++ox)
        for (int k = max(ks[ox], k0) - k0; k < min(ke[ox] - k0, C); ++k) {
          const int p = at(k);
          const double w[3] = {T[0][p], T[1][p], T[2][p]};
          double c = p_mass * w[ox] * T[3 * (DIM - 1) + ol][p] * T[3 * (DIM - 1) + jl][p];
          if constexpr (DIM == 3) {
            const double v[3] = {T[3][p], T[4][p], T[5][p]};
            c *= v[oy];
#pragma unroll
            for (int jy = 0; jy < 3; ++jy) {
              const double e = c * v[jy];
#pragma unroll
              for (int jx = 0; jx < 3; ++jx) acc[jy - oy + 2][jx - ox + 2] += e * w[jx];
            }
          } else {
#pragma unroll
            for (int jx = 0; jx < 3; ++jx) acc[0][jx - ox + 2] += c * w[jx];
          }
        }
    }
  }
  __syncthreads();
  for (int q = threadIdx.x; q < MASS_ROWS * OS; q += 192) sh.out[q] = 0.0;
  for (int w = 0; w < 3; ++w) {
    __syncthreads();
    if (ol == w && row < MASS_ROWS) {
      double* out = sh.out + row * OS + (jl - w + 2) * (DIM == 3 ? 25 : 5);
#pragma unroll
      for (int j = 0; j < ND; ++j)
#pragma unroll
        for (int d = 0; d < 5; ++d) out[j * 5 + d] += acc[j][d];
    }
  }
  __syncthreads();
  for (int q = threadIdx.x; q < MASS_ROWS * W; q += 192) {
    const int r = I0 + q / W, bit = q % W;
    if (r >= g.n_nodes) break;
    const uint64_t m0 = row_mask[2 * r], m1 = row_mask[2 * r + 1];
    if (!(((bit < 64 ? m0 : m1) >> (bit & 63)) & 1ull)) continue;
    const uint64_t low = (1ull << (bit & 63)) - 1ull;
    mvals[row_ptr[r] + (bit < 64 ? __popcll(m0 & low) : __popcll(m0) + __popcll(m1 & low))] = sh.out[q];
  }
}

// the consistent mass of a grid's pattern (declared in gm_common.h; for gm_p2g)
void gm::launch_mass(const gm_grid& g, const gm_bins& b, const gm_pattern& pat, double p_mass, double* mvals,
                     hipStream_t s) {
  const int blocks = gm_blocks(g.n_nodes, MASS_ROWS);
  if (g.dim == 3)
    k_mass_strip<3><<<blocks, 192, 0, s>>>(g, b.x_s, b.lp_s, b.cell_start, p_mass, pat.row_ptr, pat.row_mask, mvals);
  else
    k_mass_strip<2><<<blocks, 192, 0, s>>>(g, b.x_s, b.lp_s, b.cell_start, p_mass, pat.row_ptr, pat.row_mask, mvals);
}

// ------------------------------------------------------------------ consistent mass per bin (3D)
// The same matrix in the order that the 3D u-p step depends on (see k_update_lp): per bin the 27 x 27
// products of its particles, in bin order, then per row the fixed-order sum over the bins holding
// both nodes.  The products are formed from a table of the particles' 27 node weights.  With the
// right-hand side, 64 x 64 x 32 cells 890 us, 33 x 29 x 15 82, 12 x 9 x 7 20; the strips 410, 101 and
// 59; products from the axis weights 1140, 122 and 28.
__global__ void __launch_bounds__(256) k_mass_bin(gm_grid g, const double* x_s, const double* lp_s,
                                                  const int* cell_start, double p_mass, double* cb) {
  constexpr int PB = 32;
  __shared__ double A[PB][3][3], W[PB][27];
  const int b = blockIdx.x;
  const int ks = cell_start[b], ke = cell_start[b + 1];
  if (ks == ke) return;  // uniform across the workgroup
  const int t = threadIdx.x;
  double acc[3] = {0.0, 0.0, 0.0};
  for (int p0 = ks; p0 < ke; p0 += PB) {
    const int np = min(PB, ke - p0);
    __syncthreads();
    if (t < 3 * np) {
      const int a = t % 3;
      const Axis ax = gimp_axis(x_s[(long)p0 * 3 + t], lp_s[(long)p0 * 3 + t], g.h[a], g.inv_h[a]);
#pragma unroll
      for (int i = 0; i < 3; ++i) A[t / 3][a][i] = ax.w[i];
    }
    __syncthreads();
    for (int q = t; q < 27 * np; q += 256) {
      const int p = q / 27, i = q % 27;
      W[p][i] = A[p][0][i % 3] * A[p][1][i / 3 % 3] * A[p][2][i / 9];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const int q = min(t + 256 * j, 728), I = q / 27, J = q % 27;
      for (int p = 0; p < np; ++p) acc[j] = fma(W[p][I] * W[p][J], p_mass, acc[j]);
    }
  }
#pragma unroll
  for (int j = 0; j < 3; ++j)
    if (t + 256 * j < 729) cb[(long)b * 729 + t + 256 * j] = acc[j];
}

__global__ void __launch_bounds__(128) k_mass_gather(gm_grid g, const int* cell_start, const double* cb,
                                                     const int* row_ptr, const uint64_t* row_mask, double* mvals) {
  __shared__ int SLOT_BIT[125];
  __shared__ int BIN[27];
  const int I = blockIdx.x, t = threadIdx.x;
  const uint64_t m0 = row_mask[2 * I], m1 = row_mask[2 * I + 1];
  const int nx1 = g.nx + 1, nxy = (g.nx + 1) * (g.ny + 1);
  const int ci[3] = {I % nx1, (I / nx1) % (g.ny + 1), I / nxy};
  if (t < 125) {
    const uint64_t w = (t < 64) ? m0 : m1;
    const int sh = t & 63;
    if ((w >> sh) & 1ull) {
      const int below = (t < 64) ? __popcll(m0 & ((1ull << sh) - 1ull))
                                 : __popcll(m0) + __popcll(m1 & ((1ull << sh) - 1ull));
      SLOT_BIT[below] = t;
    }
  }
  if (t < 27) {
    const int ox = t % 3, oy = (t / 3) % 3, oz = t / 9;
    const int bc[3] = {ci[0] - ox, ci[1] - oy, ci[2] - oz};
    int bn = -1;
    if (bc[0] >= 0 && bc[0] <= g.nx && bc[1] >= 0 && bc[1] <= g.ny && bc[2] >= 0 && bc[2] <= g.nz) {
      bn = bc[0] + bc[1] * nx1 + bc[2] * nxy;
      if (cell_start[bn + 1] == cell_start[bn]) bn = -1;
    }
    BIN[t] = bn;
  }
  __syncthreads();
  const int nnz = __popcll(m0) + __popcll(m1);
  if (t >= nnz) return;
  const int bit = SLOT_BIT[t];
  const int d[3] = {bit % 5 - 2, (bit / 5) % 5 - 2, bit / 25 - 2};
  double s = 0.0;
#pragma unroll
  for (int o = 0; o < 27; ++o) {
    const int kx = d[0] + o % 3, ky = d[1] + (o / 3) % 3, kz = d[2] + o / 9;
    const int bn = BIN[o];
    if (bn >= 0 && kx >= 0 && kx < 3 && ky >= 0 && ky < 3 && kz >= 0 && kz < 3)
      s += cb[(long)bn * 729 + o * 27 + (kx + 3 * ky + 9 * kz)];
  }
  mvals[row_ptr[I] + t] = s;
}

extern "C" size_t gm_mass_work_bytes(const gm_grid* g) { return g ? (size_t)g->n_nodes * 729 * sizeof(double) : 0; }

extern "C" int gm_mass_binned(const gm_grid* g, const gm_bins* b, const gm_pattern* pat, double p_mass,
                              double* mvals, void* work, size_t work_bytes, hipStream_t s) {
  GM_REQUIRE(g && b && pat && mvals && work, "gm_mass_binned: null argument");
  GM_REQUIRE(g->dim == 3, "gm_mass_binned: 3D grids only");
  GM_REQUIRE(work_bytes >= gm_mass_work_bytes(g), "gm_mass_binned: workspace smaller than gm_mass_work_bytes");
  const int n = g->n_nodes;
  if (n == 0) return 0;
  k_mass_bin<<<n, 256, 0, s>>>(*g, b->x_s, b->lp_s, b->cell_start, p_mass, (double*)work);
  GM_LAUNCH_CHECK();
  k_mass_gather<<<n, 128, 0, s>>>(*g, b->cell_start, (const double*)work, pat->row_ptr, pat->row_mask, mvals);
  GM_LAUNCH_CHECK();
  return 0;
}

// ================================================================== P2G (3D)
// The activation flags, pressure-boundary flags and consistent-mass right-hand side of
// P2G_coupled_3d (mpm_utils.py:260-386) in two passes: per bin, each of the 27 nodes of
// its 3x3x3 box accumulates its particles' terms in bin order (the right-hand side
// w_I m_p p_p sum_J w_J, activation when w_I > threshold inside the particle's support,
// pressure boundary over all 27 nodes when the node lies at or above a flagged
// particle); per node, a fixed-order pass over the <= 27 bins holding it.
// Half a wave per bin, its particles' weights, pressures and flags staged in LDS together; a lane a
// node walks the particles one after the other (a load step depends on the order, see k_update_lp).
// Bins without particles write zeros, so that the gather has nothing to look up.  P2G with the
// active mask, 64 x 64 x 32 cells: 92 us; a wave per bin whose halves take every other particle
// 112, in another order; a wave per bin reading ids, flags and pressures one after the other, and a
// gather that looked at every bin, 183.
__global__ void __launch_bounds__(256) k_p2g_bin(gm_grid g, const double* x_s, const double* lp_s,
                                                 const int* cell_start, const int* sorted, const uint8_t* ext_s,
                                                 double threshold, const uint8_t* pbc_flag, double node_h_last,
                                                 double p_mass, const double* p_part, double* cb, uint8_t* cf) {
  constexpr int PB = 10;
  __shared__ struct {
    double w[PB][3][3], sum[PB], pr[PB], z[PB];
    uint8_t ext[PB];
  } sh[8];
  const int t = threadIdx.x & 31, half = threadIdx.x >> 5;
  const int b = blockIdx.x * 8 + half;
  auto& S = sh[half];
  const int ks = b < g.n_nodes ? cell_start[b] : 0, n = b < g.n_nodes ? cell_start[b + 1] - ks : 0;
  auto sync = [] {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  const int ox = t % 3, oy = (t / 3) % 3, oz = min(t / 9, 2);  // lanes 27 to 31 of a half: not stored
  const int nxy = (g.nx + 1) * (g.ny + 1);
  const double node_z = (double)(b / nxy + oz) * node_h_last;
  double rhs = 0.0;
  int on = 0;  // 1: active, 2: pressure boundary
  const int most = max(n, __shfl_xor(n, 32, 64));  // the same rounds for both halves
  for (int i0 = 0; i0 < most; i0 += PB) {
    const int np = min(PB, n - i0), p0 = ks + i0;  // (np <= 0: this half is through)
    sync();
    if (t < np) {
      const int k = p0 + t, pid = sorted[k];
      S.z[t] = pbc_flag && pbc_flag[pid] ? x_s[(long)k * 3 + 2] : INFINITY;  // height of a flagged particle
      S.pr[t] = p_part ? p_part[pid] : 0.0;
      S.ext[t] = ext_s[k];
    }
    if (t < 3 * np) {
      const int a = t % 3;
      const Axis ax = gimp_axis(x_s[(long)p0 * 3 + t], lp_s[(long)p0 * 3 + t], g.h[a], g.inv_h[a]);
#pragma unroll
      for (int i = 0; i < 3; ++i) S.w[t / 3][a][i] = ax.w[i];
    }
    sync();
    if (t < np) {
      double sum = 1.0;
#pragma unroll
      for (int a = 0; a < 3; ++a) sum *= S.w[t][a][0] + S.w[t][a][1] + S.w[t][a][2];
      S.sum[t] = sum;
    }
    sync();
    for (int p = 0; p < np; ++p) {
      if (node_z >= S.z[p]) on |= 2;
      const uint8_t ex = S.ext[p];
      const bool in = ox < ((ex & 1) ? 3 : 2) && oy < ((ex & 2) ? 3 : 2) && oz < ((ex & 4) ? 3 : 2);
      if (!in) continue;
      const double w = S.w[p][0][ox] * S.w[p][1][oy] * S.w[p][2][oz];
      if (threshold < 0.0 || w > threshold) on |= 1;
      if (p_part) rhs = fma(w * S.sum[p] * p_mass, S.pr[p], rhs);
    }
  }
  if (t < 27 && b < g.n_nodes) {
    cb[(long)b * 27 + t] = rhs;
    cf[(long)b * 27 + t] = (uint8_t)on;
  }
}

__global__ void __launch_bounds__(256) k_p2g_gather(gm_grid g, const double* cb, const uint8_t* cf, uint8_t* act,
                                                    uint8_t* bflag, double* mrhs) {
  const int I = blockIdx.x * blockDim.x + threadIdx.x;
  if (I >= g.n_nodes) return;
  const int nx1 = g.nx + 1, nxy = (g.nx + 1) * (g.ny + 1);
  const int cx = I % nx1, cy = (I / nx1) % (g.ny + 1), cz = I / nxy;
  double v[27];
  uint8_t f[27];
#pragma unroll
  for (int o = 0; o < 27; ++o) {
    const bool on = cx >= o % 3 && cy >= o / 3 % 3 && cz >= o / 9;
    const long at = (long)(on ? I - o % 3 - o / 3 % 3 * nx1 - o / 9 * nxy : I) * 27 + o;
    v[o] = cb[at];
    f[o] = cf[at];
  }
  double s = 0.0;
  int flags = 0;
#pragma unroll
  for (int o = 0; o < 27; ++o)
    if (cx >= o % 3 && cy >= o / 3 % 3 && cz >= o / 9) {
      s += v[o];
      flags |= f[o];
    }
  if (flags & 1)
#pragma unroll
    for (int k = 0; k < 4; ++k) act[I * 4 + k] = 1;
  if ((flags & 2) && bflag) bflag[I * 4 + 3] = 1;
  if (mrhs) mrhs[I] = s;
}

extern "C" size_t gm_p2g_work_bytes(const gm_grid* g) {
  return g ? (size_t)g->n_nodes * 27 * (sizeof(double) + 1) : 0;
}

extern "C" int gm_p2g_binned(const gm_grid* g, const gm_bins* b, double threshold, const uint8_t* pbc_flag,
                             double node_h_last, double p_mass, const double* p_part, uint8_t* act, uint8_t* bflag,
                             double* mrhs, void* work, size_t work_bytes, hipStream_t s) {
  GM_REQUIRE(g && b && act && work, "gm_p2g_binned: null argument");
  GM_REQUIRE(g->dim == 3 && g->nb == 4, "gm_p2g_binned: the 3D u-p form only");
  GM_REQUIRE(!mrhs || p_part, "gm_p2g_binned: the right-hand side needs the particle pressures");
  GM_REQUIRE(work_bytes >= gm_p2g_work_bytes(g), "gm_p2g_binned: workspace smaller than gm_p2g_work_bytes");
  const int n = g->n_nodes;
  if (n == 0) return 0;
  double* cb = (double*)work;
  uint8_t* cf = (uint8_t*)(cb + (size_t)n * 27);
  k_p2g_bin<<<gm_blocks(n, 8), 256, 0, s>>>(*g, b->x_s, b->lp_s, b->cell_start, b->sorted, b->ext_s, threshold, pbc_flag,
                             node_h_last, p_mass, mrhs ? p_part : nullptr, cb, cf);
  GM_LAUNCH_CHECK();
  k_p2g_gather<<<gm_blocks(n, 256), 256, 0, s>>>(*g, cb, cf, act, bflag, mrhs);
  GM_LAUNCH_CHECK();
  return 0;
}

extern "C" size_t gm_node_jacobian_work_bytes(const gm_grid* g, int tangent_fp32) {
  if (!g) return 0;
  return (size_t)g->n_nodes * (size_t)CB_BIN * (tangent_fp32 ? sizeof(float) : sizeof(double));
}

// ------------------------------------------------------------ variants and their tuner
// Product variants of the per-bin form (particles per group, workgroups per CU, grid):
//   FP32 tangent: 0 (8, 2, one per bin), 1 (8, 2, persistent), 2 (4, 4, persistent), 3 (4, 3, persistent)
//   FP64 tangent: 0 (4, 2, one per bin), 1 (4, 2, persistent), 2 (8, 1, one per bin), 3 (8, 1, persistent)
// "persistent": one workgroup per resident slot (CUs x workgroups per CU), each
// sweeping bins blockIdx.x + k gridDim.x, with the next group's loads issued before
// the current group's products; "one per bin": loads at the top of each group.  Gather
// variants: 0 (per-lane reads from the workspace), 1 (all 27 chunks of a row staged in
// LDS at once; 9 at a time in FP64), 2 (9 at a time; 3 in FP64).
// Variants of the line sums: 0 the number of segments of a line that best_segments picks,
// 1 twice and 2 three times as many, 3 one segment (as few as MAX_SEG allows); their gather's:
// 128, 256 or 512 threads a row.  Every variant of a form writes the same bits.
namespace {
constexpr int N_BIN_VARIANTS = 4, N_GATHER_VARIANTS = 3;
int g_bin_variant[2] = {0, 0};     // [tangent_fp32]
int g_gather_variant[2] = {0, 0};  // [tangent_fp32]

int cu_count() {
  static int n = 0;
  if (n == 0) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    hipDeviceProp_t pr;
    if (hipGetDeviceProperties(&pr, dev) != hipSuccess) return 0;
    n = pr.multiProcessorCount;
  }
  return n;
}

// Segments of a bin line: every segment after the first repeats the products of two bins, and
// the workgroups do not come out even over the CUs: the number of segments with the least
// (rounds + 1/2) x (bins of a segment + 2), at least one round.  The half round is what the
// lines without particles (which end at once) and the XCDs' shares make of the last one: whole
// rounds instead pick 1 segment for 21 x 17 x 13 cells, 249 us where 2 take 212.  (Some six
// particles a bin are taken for granted.)
int best_segments(int nbx, int lines, int n_p, int slots) {
  const double busy = std::max(1.0, std::min<double>(lines, n_p / (6.0 * nbx)));
  int best = 1;
  double cost = 0.0;
  for (int k = (nbx + MAX_SEG - 1) / MAX_SEG; k <= (nbx + 1) / 2; ++k) {
    const int len = (nbx + k - 1) / k;
    const double c = std::max(1.0, busy * k / slots + 0.5) * (len + (k > 1 ? 2 : 0));
    if (cost == 0.0 || c < cost) {
      cost = c;
      best = k;
    }
  }
  return best;
}

// FP64 assemblies take the line sums when there are lines enough for the CUs: from 24,000
// particles (at some eight a cell) on more than 7000 nodes.  Products and gather against the
// per-bin form's: 16 x 16 x 8 cells 167 and 146 us, 56 x 6 x 5 161 and 118, 24 x 12 x 8 (18,432
// particles) 178 and 175, 48 x 9 x 7 (24,192) 238 and 237, 20 x 16 x 10 231 and 255, 9 x 48 x 7 202
// and 252, 33 x 29 x 15 776 and 1034.
bool line_sums(const gm_grid* g, const gm_bins* b, int fp32) {
  return !fp32 && g->n_nodes > 7000 && b->n_particles >= 24000;
}

int launch_bins(const gm_grid* g, const gm_bins* b, const void* D, int fp32, int variant, void* work,
                hipStream_t s) {
  const int n = g->n_nodes;
  const int cus = cu_count();
  GM_REQUIRE(cus > 0, "gm_jacobian_bins: no device properties");
  if (line_sums(g, b, fp32)) {
    const int nbx = g->nx + 1, lines = n / nbx;
    int n_seg = best_segments(nbx, lines, b->n_particles, cus);  // one workgroup per CU (the operand buffers in LDS)
    if (variant == 1) n_seg *= 2;
    if (variant == 2) n_seg *= 3;
    if (variant == 3) n_seg = 1;
    n_seg = std::min(std::max(n_seg, (nbx + MAX_SEG - 1) / MAX_SEG), nbx);
    const int len = (nbx + n_seg - 1) / n_seg;
    k_jac_line<<<(unsigned)lines * n_seg, 512, 0, s>>>(*g, b->x_s, b->lp_s, b->cell_start, b->n_particles, len, n_seg,
                                                       (const double*)D, (double*)work);
    GM_LAUNCH_CHECK();
    return 0;
  }
#define GM_BIN(TT, PG, OCC, PERSIST)                                                                     \
  if (PERSIST)                                                                                           \
    k_jac_bin<TT, TT, PG, OCC, true><<<std::min(n, cus * OCC), 256, 0, s>>>(*g, b->x_s, b->lp_s,          \
                                                                        b->cell_start, n, (const TT*)D, \
                                                                        (TT*)work);                     \
  else                                                                                                   \
    k_jac_bin<TT, TT, PG, OCC, false><<<n, 256, 0, s>>>(*g, b->x_s, b->lp_s, b->cell_start, n, (const TT*)D, \
                                                      (TT*)work)
  if (fp32) {
    switch (variant) {
      case 0: GM_BIN(float, 8, 2, false); break;
      case 1: GM_BIN(float, 8, 2, true); break;
      case 2: GM_BIN(float, 4, 4, true); break;
      default: GM_BIN(float, 4, 3, true); break;
    }
  } else {
    switch (variant) {
      case 0: GM_BIN(double, 4, 2, false); break;
      case 1: GM_BIN(double, 4, 2, true); break;
      case 2: GM_BIN(double, 8, 1, false); break;
      default: GM_BIN(double, 8, 1, true); break;
    }
  }
#undef GM_BIN
  GM_LAUNCH_CHECK();
  return 0;
}

int launch_gather(const gm_grid* g, const gm_bins* b, const gm_pattern* pat, int fp32, int variant,
                  const void* work, const uint8_t* freem, void* vals, int vals_fp32, hipStream_t s) {
  const int n = g->n_nodes;
#define GM_LINES(TVV, T)                                                                                        \
  k_jac_line_gather<TVV, T><<<n, T, 0, s>>>(*g, b->cell_start, (const double*)work, freem, pat->row_ptr,        \
                                            pat->row_mask, (TVV*)vals)
#define GM_GATHER(TCC, TVV)                                                                                      \
  if (variant == 0)                                                                                              \
    k_jac_gather<TCC, TVV><<<n, 512, 0, s>>>(*g, b->cell_start, (const TCC*)work, freem, pat->row_ptr,         \
                                             pat->row_mask, (TVV*)vals);                                       \
  else if (variant == 1)                                                                                         \
    k_jac_gather_staged<TCC, TVV, sizeof(TCC) == 4 ? 27 : 9><<<n, 256, 0, s>>>(                                 \
        *g, b->cell_start, (const TCC*)work, freem, pat->row_ptr, pat->row_mask, (TVV*)vals);                  \
  else                                                                                                           \
    k_jac_gather_staged<TCC, TVV, sizeof(TCC) == 4 ? 9 : 3><<<n, 256, 0, s>>>(                                  \
        *g, b->cell_start, (const TCC*)work, freem, pat->row_ptr, pat->row_mask, (TVV*)vals)
  if (line_sums(g, b, fp32)) {
    if (variant == 0) {
      if (vals_fp32) GM_LINES(float, 128);
      else GM_LINES(double, 128);
    } else if (variant == 1) {
      if (vals_fp32) GM_LINES(float, 256);
      else GM_LINES(double, 256);
    } else {
      if (vals_fp32) GM_LINES(float, 512);
      else GM_LINES(double, 512);
    }
  } else if (fp32) {
    if (vals_fp32) GM_GATHER(float, float);
    else GM_GATHER(float, double);
  } else {
    if (vals_fp32) GM_GATHER(double, float);
    else GM_GATHER(double, double);
  }
#undef GM_GATHER
#undef GM_LINES
  GM_LAUNCH_CHECK();
  return 0;
}
}  // namespace

extern "C" int gm_jacobian_bins_variant(const gm_grid* g, const gm_bins* b, const void* D, int tangent_fp32,
                                        int variant, void* work, size_t work_bytes, hipStream_t s) {
  GM_REQUIRE(g && b && D && work, "gm_jacobian_bins: null argument");
  GM_REQUIRE(g->dim == 3 && g->nb == 4, "gm_jacobian_bins: the 3D u-p form only");
  GM_REQUIRE(variant >= 0 && variant < N_BIN_VARIANTS, "gm_jacobian_bins: variant out of range");
  GM_REQUIRE(work_bytes >= gm_node_jacobian_work_bytes(g, tangent_fp32),
             "gm_jacobian_bins: workspace smaller than gm_node_jacobian_work_bytes");
  if (g->n_nodes == 0) return 0;
  return launch_bins(g, b, D, tangent_fp32 ? 1 : 0, variant, work, s);
}

extern "C" int gm_jacobian_bins(const gm_grid* g, const gm_bins* b, const void* D, int tangent_fp32, void* work,
                                size_t work_bytes, hipStream_t s) {
  return gm_jacobian_bins_variant(g, b, D, tangent_fp32, g_bin_variant[tangent_fp32 ? 1 : 0], work, work_bytes, s);
}

extern "C" int gm_jacobian_gather_variant(const gm_grid* g, const gm_bins* b, const gm_pattern* pat,
                                          int tangent_fp32, int variant, const void* work, const uint8_t* freem,
                                          void* vals, int vals_fp32, hipStream_t s) {
  GM_REQUIRE(g && b && pat && work && freem && vals, "gm_jacobian_gather: null argument");
  GM_REQUIRE(g->dim == 3 && g->nb == 4, "gm_jacobian_gather: the 3D u-p form only");
  GM_REQUIRE(variant >= 0 && variant < N_GATHER_VARIANTS, "gm_jacobian_gather: variant out of range");
  if (g->n_nodes == 0) return 0;
  return launch_gather(g, b, pat, tangent_fp32 ? 1 : 0, variant, work, freem, vals, vals_fp32, s);
}

extern "C" int gm_jacobian_gather(const gm_grid* g, const gm_bins* b, const gm_pattern* pat, int tangent_fp32,
                                  const void* work, const uint8_t* freem, void* vals, int vals_fp32, hipStream_t s) {
  return gm_jacobian_gather_variant(g, b, pat, tangent_fp32, g_gather_variant[tangent_fp32 ? 1 : 0], work, freem,
                                    vals, vals_fp32, s);
}

// Times every per-bin and gather variant on the given tangent (`reps` launches each
// after one warm-up, HIP events on the stream), keeps the fastest of each for later
// assemblies in this precision and returns them with the average times (ms[0..3]
// per-bin variants, ms[4..6] gather variants).  The matrix and the workspace are
// overwritten with the assembly.
extern "C" int gm_jacobian_autotune(const gm_grid* g, const gm_bins* b, const gm_pattern* pat, const void* D,
                                    int tangent_fp32, const uint8_t* freem, void* vals, int vals_fp32, void* work,
                                    size_t work_bytes, int reps, int* best_bins, int* best_gather, float* ms,
                                    hipStream_t s) {
  GM_REQUIRE(g && b && pat && D && freem && vals && work && best_bins && best_gather && ms && reps >= 1,
             "gm_jacobian_autotune: bad argument");
  GM_REQUIRE(g->dim == 3 && g->nb == 4, "gm_jacobian_autotune: the 3D u-p form only");
  GM_REQUIRE(work_bytes >= gm_node_jacobian_work_bytes(g, tangent_fp32),
             "gm_jacobian_autotune: workspace smaller than gm_node_jacobian_work_bytes");
  const int fp = tangent_fp32 ? 1 : 0;
  if (g->n_nodes == 0) {
    *best_bins = g_bin_variant[fp];
    *best_gather = g_gather_variant[fp];
    return 0;
  }
  hipEvent_t e0, e1;
  GM_HIP(hipEventCreate(&e0));
  GM_HIP(hipEventCreate(&e1));
  int rc = 0;
  auto time = [&](auto&& launch, float* out) -> int {
    int r = launch();
    if (r) return r;
    GM_HIP(hipEventRecord(e0, s));
    for (int k = 0; k < reps; ++k)
      if ((r = launch())) return r;
    GM_HIP(hipEventRecord(e1, s));
    GM_HIP(hipEventSynchronize(e1));
    float t = 0.0f;
    GM_HIP(hipEventElapsedTime(&t, e0, e1));
    *out = t / reps;
    return 0;
  };
  int bb = 0, bg = 0;
  for (int v = 0; v < N_BIN_VARIANTS && !rc; ++v) {
    rc = time([&]() { return launch_bins(g, b, D, fp, v, work, s); }, &ms[v]);
    if (!rc && ms[v] < ms[bb]) bb = v;
  }
  if (!rc) rc = launch_bins(g, b, D, fp, bb, work, s);
  for (int v = 0; v < N_GATHER_VARIANTS && !rc; ++v) {
    rc = time([&]() { return launch_gather(g, b, pat, fp, v, work, freem, vals, vals_fp32, s); },
              &ms[N_BIN_VARIANTS + v]);
    if (!rc && ms[N_BIN_VARIANTS + v] < ms[N_BIN_VARIANTS + bg]) bg = v;
  }
  hipEventDestroy(e0);
  hipEventDestroy(e1);
  if (rc) return rc;
  g_bin_variant[fp] = bb;
  g_gather_variant[fp] = bg;
  *best_bins = bb;
  *best_gather = bg;
  return 0;
}

extern "C" int gm_node_jacobian_binned(const gm_grid* g, const gm_bins* b, const gm_pattern* pat, const void* D,
                                       int tangent_fp32, const uint8_t* freem, void* vals, int vals_fp32,
                                       void* work, size_t work_bytes, hipStream_t s) {
  GM_REQUIRE(g && b && pat && D && freem && vals && work, "gm_node_jacobian_binned: null argument");
  int rc = gm_jacobian_bins(g, b, D, tangent_fp32, work, work_bytes, s);
  if (rc) return rc;
  return gm_jacobian_gather(g, b, pat, tangent_fp32, work, freem, vals, vals_fp32, s);
}
