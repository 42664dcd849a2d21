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
// FP64 otherwise.
//   k_jac_line    a workgroup per segment of a bin line (fixed y, z): the products of its
//                 bins one after another, summed over the line while they stay in the
//                 accumulators; every pair of nodes a line reaches is written once (405
//                 blocks a bin where the bin itself has 729).
//   k_jac_gather  one workgroup per block row I: every block (I, J) of the pattern sums
//                 the <= 9 lines holding both nodes in the fixed order (oz, oy); masks,
//                 sign and identity rows as in the node-row kernels.
// Both steps are deterministic (fixed accumulation order).  The workspace holds n_nodes x
// 6480 values, written once and read once per assembly.
//   64 x 64 x 32 cells, 1,048,576 particles (MI355X), per assembly: FP32 2.23 + 1.05 ms
//   (one workgroup per bin, 11664 values per node in the workspace: 2.84 + 1.56 ms), FP64
//   4.0 + 1.83 ms (5.6 + 2.9).  k_jac_line: the products take 0.95 (FP32) and 1.3 ms (FP64),
//   the stores of the line sums 0.7 and 1.95 (3.6 and 7.2 GB), and one follows the other in the
//   product waves; the operand waves' FP64 arithmetic adds 0.4 and 0.2.  With the shape-function
//   tables made by an operand wave rather than the last product wave FP32 took 2.60.
//   k_jac_gather moves 4.7 GB (FP32) at 4.5 TB/s.
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
// Workspace of the line sums, per bin line (y, z) and node x of it (a grid node's share):
// the pairs of a row node and a column node of the line whose smaller x is that node's, which
// one step of k_jac_line completes together.  Parts: nine chunks A (row node (x, y + oy,
// z + oz), column nodes x .. x + 2), then nine chunks B for row nodes x + 1 and nine for
// x + 2 (column nodes x).  In a chunk: column dof c, column node ([dx] [jy + 3 jz]), row dof
// r.  A matrix-core lane ends with the four rows r of one (row node, column node, c), so
// that a store instruction writes whole runs of neighbouring 16-byte vectors.
constexpr long CHUNK_A = 4L * 27 * 4, CHUNK_B = 4L * 9 * 4;  // values
constexpr int CHUNK = CHUNK_A + 2 * CHUNK_B;                 // a row node's values of a line
constexpr long CB_NODE = 9L * CHUNK;                         // values per grid node
__device__ __forceinline__ long chunk_a(int o9, int node) { return (long)node * CB_NODE + o9 * CHUNK_A; }
// d = 1, 2: the distance of the row node
__device__ __forceinline__ long chunk_b(int o9, int node, int d) {
  return (long)node * CB_NODE + 9 * CHUNK_A + ((d - 1) * 9 + o9) * CHUNK_B;
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

template <int V>
struct Int {
  static constexpr int value = V;
};

constexpr int MAX_SEG = 61;  // bins of a line segment (with two before it and the end, one a lane)

}  // namespace

// Line sums.  A workgroup takes the bins of one segment [xs, xe) of a bin line (fixed y, z)
// in ascending x.  The nodes x, x + 1, x + 2 that a bin reaches lie in the three slots
// node_x mod 3, so that from one bin to the next two of the three node planes stay where
// they are: the accumulators of the matrix cores (27 row nodes x 27 column nodes x 4 x 4)
// keep summing, and only the pairs that the next bin does not reach (the row or the column
// node is x: 405 of 729 blocks) are stored and cleared.  Pairs that bins before xs reach as
// well belong to this segment when min(row x, column x) >= xs; the sweep starts two bins
// early to have their whole sum.
// A bin's particles are taken four at a time (a group).  The first CW waves hold the
// accumulators and do nothing but products and stores.  The others, in teams of four waves,
// prepare E_p and the B operand of one coming group each in the other half of the LDS
// buffers, stage the tangent rows and shape-function tables of the groups after those and
// load the rows of the next ones: one barrier for CW / 4 groups, and neither the tables nor
// the loads are in the matrix cores' way.
//   FP32: 8 product waves (two tiles each) and two teams.  A bin's products are summed from
//     zero in one set of accumulators and added to the line's sums in another, so that the
//     line's longer sum has one rounding a bin more and no longer chains (the matrix stays
//     as near the 64-bit one as with bin sums added in FP64).
//   FP64: 4 product waves (four tiles each) and one team, for the operands' size in LDS.
// The operands are formed in FP64 and rounded once.
// K order: a K step of the MFMA is one shape-function component beta and the four
// particles (lane group l / 16 = particle).  After the
// K loop unrolls, every A and B operand address is a per-lane base plus an immediate,
// and the (c, beta) products that vanish (u columns: no w term except the penalty
// on u_z, no w_avg term) are not issued.  Every segment length adds the same products in
// the same order, so all of them write the same bits.
template <typename TD, typename TC, int CW>
__global__ void __launch_bounds__(128 * CW, CW / 2) k_jac_line(gm_grid g, const double* x_s, const double* lp_s,
                                                               const int* cell_start, int n_p, int seg_len,
                                                               int n_seg, const TD* D, TC* cb) {
  constexpr int TEAMS = CW / 4, TILES = 16 / CW;
  constexpr bool BIN_SUMS = sizeof(TC) == 4;
  constexpr int PG = 4;             // particles of a group: one quad of K steps
  constexpr int NI = 4 * NZ;        // (z, r) entries of a node row of E_p
  // shape-function tables of the sweep's particles, a ring filled a batch at a time
  constexpr int RING = 32, BATCH = 16;
  __shared__ double AXT_[RING][3][9];
  // tangent rows of a group (particles are in bin order, so a group's rows are contiguous)
  constexpr int DROW = NY * NZ;
  __shared__ TD DR_[TEAMS][2][PG * DROW];
  // E_p[I][z][r] (r fastest), node rows 68 entries apart and particles 1840: the 64
  // (particle, I, r) entries a wave reads at once fall in 64 distinct banks.  (The padding
  // rows of the last row tile read row 26; they are never stored.)
  constexpr int EI = 68, EP = 27 * EI + 4;
  __shared__ TC E_[TEAMS][2][PG * EP];
  // B operand g_p[J][beta], J padded to 32 with zeros, particles 176 entries apart
  constexpr int BB = 32, BP = 5 * BB + 16;
  __shared__ TC BT_[TEAMS][2][PG * BP];
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
  auto next_round = [&](Group q) {
#pragma unroll
    for (int k = 0; k < TEAMS; ++k) q = next(q);
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
  // q: the last group of a round (none: the sweep ends in that round)
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
    typedef typename Mfma<TC>::acc ACC;
    ACC acc[TILES][4], sum[TILES][4];  // (sum: BIN_SUMS only)
#pragma unroll
    for (int s = 0; s < TILES; ++s)
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[s][c] = sum[s][c] = ACC{0, 0, 0, 0};
    // output tiles w + CW s: row tile mt = w / 2 + CW / 2 s (16 rows (I, r)), column tile
    // nt = w % 2 (16 columns J); the last waves have no last tile (rows I >= 28).  Node index
    // I = 9 slot + oy + 3 oz, J likewise.
    const int w = wave;
    const bool last = (w >> 1) + (CW >> 1) * (TILES - 1) < 7;
    const int lg = lane >> 4, rt = lane & 15;
    const int r_l = Mfma<TC>::r_major ? (rt >> 2) : (rt & 3);
    const int i_l = Mfma<TC>::r_major ? (rt & 3) : (rt >> 2);
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
        ACC* leave = BIN_SUMS ? sum[s] : acc[s];
        const int I = ((w >> 1) + (CW >> 1) * s) * 4 + (l >> 4), islot = I / 9, iyz = I - 9 * islot;
        if (I < 27 && J < 27 && (islot == q || jslot == q)) {
          const int di = islot >= q ? islot - q : islot - q + 3, dj = jslot >= q ? jslot - q : jslot - q + 3;
          if (B >= xs && B + di <= g.nx) {
            TC* o = cb + (di == 0 ? chunk_a(iyz, lb + B) + (dj * 9 + jyz) * 4 : chunk_b(iyz, lb + B, di) + jyz * 4);
            const int plane = di == 0 ? 27 * 4 : 9 * 4;
#pragma unroll
            for (int c = 0; c < 4; ++c) *reinterpret_cast<ACC*>(o + c * plane) = leave[c];
          }
#pragma unroll
          for (int c = 0; c < 4; ++c) leave[c] = ACC{0, 0, 0, 0};
        }
      }
    };
    Group gt = cur;  // the last group of the round whose tables come next
    if (wave == CW - 1) {
#pragma unroll
      for (int k = 1; k < TEAMS; ++k) gt = next(gt);
      load_tables(0);
      tables_for(gt);
      gt = next_round(gt);
      tables_for(gt);
    }
    __syncthreads();
    __syncthreads();
    for (int buf = 0; cur.x < xe; buf ^= 1) {
      if (wave == CW - 1) {
        gt = next_round(gt);
        tables_for(gt);
      }
#pragma unroll 1
      for (int k = 0; k < TEAMS && cur.x < xe; ++k) {
        // particles past the bin's last have zero B; a tile's operands are read before its products
        const TC *E = E_[k][buf], *BT = BT_[k][buf];
        TC b[5];
#pragma unroll
        for (int beta = 0; beta < 5; ++beta) b[beta] = BT[bbase + beta * BB];
        auto products = [&](auto tile) {
          constexpr int s = decltype(tile)::value;
          TC a[4][5];
#pragma unroll
          for (int beta = 0; beta < 5; ++beta)
#pragma unroll
            for (int c = 0; c < 4; ++c)
              if (zsel(c, beta) != ZERO) a[c][beta] = E[abase[s] + zsel(c, beta) * 4];
#pragma unroll
          for (int beta = 0; beta < 5; ++beta)
#pragma unroll
            for (int c = 0; c < 4; ++c)  // (c, beta) resolved at compile time
              if (zsel(c, beta) != ZERO) acc[s][c] = Mfma<TC>::step(a[c][beta], b[beta], acc[s][c]);
        };
        if constexpr (TILES == 4) {
          products(Int<0>{});
          products(Int<1>{});
        }
        products(Int<TILES - 2>{});
        if (last) products(Int<TILES - 1>{});  // wave-uniform
        const Group nxt = next(cur);
        if (nxt.x != cur.x) {  // the bin's last group
          if (BIN_SUMS) {
#pragma unroll
            for (int s = 0; s < TILES; ++s)
#pragma unroll
              for (int c = 0; c < 4; ++c) {
                sum[s][c] += acc[s][c];
                acc[s][c] = ACC{0, 0, 0, 0};
              }
          }
          // up to three steps clear every pair the sweep has touched
          for (int B = cur.x; B < min(min(nxt.x, cur.x + 3), xe); ++B) flush(B);
        }
        cur = nxt;
      }
      __syncthreads();
    }
    return;
  }
  // ------------------------------------------------------------------ operands
  const int team = (wave - CW) >> 2, t = (threadIdx.x - 64 * CW) & 255;
  constexpr int VD = 16 / sizeof(TD);  // tangent values per load
  constexpr int ND = (PG * DROW + 256 * VD - 1) / (256 * VD);
  typedef TD dvec __attribute__((ext_vector_type(16 / sizeof(TD)), aligned(sizeof(TD))));
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
        TD v = from[j][i];
        if (back > 0) v = i + back < VD ? from[j][min(i + back, VD - 1)] : (TD)0;
        if (k + i < PG * DROW) DR_[team][buf][k + i] = k0 + k + i < lim ? v : (TD)0;
      }
    }
  };
  auto operands = [&](const Group& q, int buf) {
    const int np = min(PG, q.ke - q.p0), rot = q.x % 3;  // node ox of the bin lies in slot (ox + rot) % 3
    // B operand: threads (J, particle)
    if (t < PG * 32) {
      const int p = t >> 5, Jb = t & 31;
      TC* B = BT_[team][buf] + p * BP + Jb;
      const double(*AX)[9] = AXT_[(q.p0 - ps + p) % RING];
      if (Jb < 27 && p < np) {
        const int js = Jb / 9, sx = js >= rot ? js - rot : js - rot + 3, jy = Jb % 3, jz = (Jb / 3) % 3;
        const double wx = AX[0][sx], wy = AX[1][jy], wz = AX[2][jz];
        B[0] = (TC)(wx * wy * wz);
        B[BB] = (TC)(AX[0][3 + sx] * wy * wz);
        B[2 * BB] = (TC)(wx * AX[1][3 + jy] * wz);
        B[3 * BB] = (TC)(wx * wy * AX[2][3 + jz]);
        B[4 * BB] = (TC)(AX[0][6 + sx] * AX[1][6 + jy] * AX[2][6 + jz]);
      } else {
#pragma unroll
        for (int beta = 0; beta < 5; ++beta) B[beta * BB] = 0;
      }
    }
    // E_p[I][z][r] = (L_I D_p)[r][z]: u rows sum_b dw/dx_b D[(b,r)] + w D[T_r];
    // the pressure row w D[Q] + sum_b dw/dx_b D[M_b] + (w - w_avg) D[S]
    if (t < PG * NI) {
      const int p = t / NI, zr = t % NI, z = zr >> 2, r = zr & 3;
      const TD* Dp = DR_[team][buf] + p * DROW + z;
      const int k0 = r < 3 ? r : Y_M, dk = r < 3 ? 3 : 1;
      const double d0 = Dp[k0 * NZ], d1 = Dp[(k0 + dk) * NZ], d2 = Dp[(k0 + 2 * dk) * NZ];
      const double dS = r < 3 ? 0.0 : (double)Dp[Y_S * NZ];
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
        TC* Eo = E_[team][buf] + p * EP + zr + 9 * EI * (ix + rot >= 3 ? ix + rot - 3 : ix + rot);
        const double wx = AX[0][ix], u = AX[0][3 + ix] * d0 + wx * dw, v = wx * d1, qx = wx * d2, a = AX[0][6 + ix] * dwa;
#pragma unroll
        for (int iy = 0; iy < 3; ++iy) {
          const double U = wy[iy] * u + gy[iy] * v, Q = wy[iy] * qx, A2 = ay[iy] * a;
#pragma unroll
          for (int iz = 0; iz < 3; ++iz) Eo[(iy + 3 * iz) * EI] = (TC)(wz[iz] * U + gz[iz] * Q + az[iz] * A2);
        }
      }
    }
  };
  // round i: the groups TEAMS i + team; `cur` stays the round's first group
  Group g0 = cur;
  for (int k = 0; k < team; ++k) g0 = next(g0);
  Group g1 = next_round(g0), g2 = next_round(g1), g3 = next_round(g2);
  load_group(g0, even);
  load_group(g1, odd);
  stage_group(g0, 0, even);
  load_group(g2, even);
  __syncthreads();
  if (g0.x < xe) operands(g0, 0);
  stage_group(g1, 1, odd);
  load_group(g3, odd);
  __syncthreads();
  // while the products of round i run: the operands of i + 1, the rows and tables of i + 2,
  // and the loads of i + 3 and i + 4 on their way
  while (cur.x < xe) {
    if (g1.x < xe) operands(g1, 1);
    stage_group(g2, 0, even);
    const Group g4 = next_round(g3);
    load_group(g4, even);
    __syncthreads();
    cur = next_round(cur);
    if (cur.x >= xe) break;
    if (g2.x < xe) operands(g2, 0);
    stage_group(g3, 1, odd);
    g1 = g3;
    g2 = g4;
    g3 = next_round(g4);
    load_group(g3, odd);
    __syncthreads();
    cur = next_round(cur);
  }
}

// One workgroup per block row I, one thread per window position and 128 / T column dofs:
// the <= 9 line sums of its four rows, all loads issued before the first is added.  Both
// the reads (runs of 16-byte vectors) and the writes (the row's blocks, through LDS) are
// coalesced; bound by HBM on the workspace and the matrix.
template <typename TC, typename TV, int T>
__global__ void __launch_bounds__(T) k_jac_gather(gm_grid g, const int* cell_start, const TC* cb,
                                                  const uint8_t* freem, const int* row_ptr,
                                                  const uint64_t* row_mask, TV* vals) {
  typedef typename Mfma<TC>::acc V4;
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
  // column dofs a thread has in flight: all of them in FP64 (1.95 -> 1.83 ms), one in FP32 (1.06; all 1.09)
  constexpr int UC = sizeof(TC) == 8 ? 4 * 128 / T : 1;
#pragma unroll UC
  for (int c0 = 0; c0 < 4 * 128 / T; ++c0) {
    const int c = (t >> 7) + c0 * (T / 128);
    V4 v[9];
    bool on[9];
#pragma unroll
    for (int o = 0; o < 9; ++o) {
      const int ky = dy + o % 3, kz = dz + o / 3, k = ky + 3 * kz, n = NODE[o];
      on[o] = live && ky >= 0 && ky < 3 && kz >= 0 && kz < 3 && ((MASK[o] >> dx) & 1);
      const long at = dx >= 2 ? chunk_a(o, n) + (c * 27 + (dx - 2) * 9 + k) * 4
                              : chunk_b(o, n + dx - 2, 2 - dx) + (c * 9 + k) * 4;
      v[o] = *reinterpret_cast<const V4*>(cb + (on[o] ? at : 0L));
    }
    double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int o = 0; o < 9; ++o)
#pragma unroll
      for (int r = 0; r < 4; ++r) s[r] += on[o] ? (double)v[o][r] : 0.0;
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
// r_I = sum_p L_I Y_p per bin (node I_loc of the bin's 3x3x3 box), then per node the fixed-order sum over the <= 27 bins holding it.
// A wave per bin: tables and rows of Y staged in its LDS together, five particles at a time, twelve
// lanes each: one per (iz, dof) with the sums of its nine (ix, iy) in registers, added over the
// five at the end.  A bin without particles writes zeros, so that the gather has nothing to look
// up before its 27 loads.  Bound by the LDS reads (26 a lane for nine sums; a lane per (iy, iz,
// dof) takes 20 for three and 227 us) and by HBM in the gather.  1,048,576 particles, 139,425
// nodes: 150 + 45 us (224 + 60 with a lane per node reading Y from memory, and a gather that
// looked at every bin before its load); 756 bins: 10 us (26).
constexpr int RES_PB = 10, RES_G = 5;
__global__ void __launch_bounds__(256) k_res_bin(gm_grid g, const double* x_s, const double* lp_s,
                                                 const int* cell_start, const double* Y, double* cb) {
  __shared__ union {
    struct {
      double ax[RES_PB][3][9], y[RES_PB * NY];
    };
    double red[RES_G][108];
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
  const int grp = lane / 12, c = lane % 12 & 3, iz = lane % 12 >> 2;
  // the dof's rows of Y: (b = 0, 1, 2) of P or m, body force or mass balance
  const int y0 = c < 3 ? c : Y_M, dy = c < 3 ? 3 : 1, yt = c < 3 ? Y_T + c : Y_Q;
  double r[9];
#pragma unroll
  for (int i = 0; i < 9; ++i) r[i] = 0.0;
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
    for (int p = grp; p < np && grp < RES_G; p += RES_G) {
      const double *X = S_.ax[p][0], *V = S_.ax[p][1], *W = S_.ax[p][2], *yp = S_.y + p * NY;
      const double wz = W[iz], S = c < 3 ? 0.0 : yp[Y_S];
      // r = gx (P0 wy wz) + wx (P1 gy wz + wy (P2 gz + T wz)) - wax way (waz S)
      const double u = yp[y0] * wz, v = yp[y0 + dy] * wz, t = yp[y0 + 2 * dy] * W[3 + iz] + (yp[yt] + S) * wz;
      const double a = W[6 + iz] * S;
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        const double uj = V[j] * u, vj = V[3 + j] * v + V[j] * t, aj = V[6 + j] * a;
#pragma unroll
        for (int i = 0; i < 3; ++i) r[3 * j + i] += X[3 + i] * uj + X[i] * vj - X[6 + i] * aj;
      }
    }
  }
  sync();
  if (grp < RES_G)
#pragma unroll
    for (int i = 0; i < 9; ++i) S_.red[grp][(iz * 9 + i) * 4 + c] = r[i];
  sync();
#pragma unroll
  for (int q = lane; q < 108; q += 64) {
    double s = S_.red[0][q];
#pragma unroll
    for (int k = 1; k < RES_G; ++k) s += S_.red[k][q];
    cb[(long)b * 108 + q] = s;
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
// Bound by those LDS reads (8 a particle and lane in 3D).  1,048,576 particles, 139,425 rows:
// 414 us, against 1110 for products per bin, stored (764 MB) and summed over 27 bins;
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

// the consistent mass of a grid's pattern (declared in gm_common.h; gm_p2g uses it as well)
void gm::launch_mass(const gm_grid& g, const gm_bins& b, const gm_pattern& pat, double p_mass, double* mvals,
                     hipStream_t s) {
  const int blocks = gm_blocks(g.n_nodes, MASS_ROWS);
  if (g.dim == 3)
    k_mass_strip<3><<<blocks, 192, 0, s>>>(g, b.x_s, b.lp_s, b.cell_start, p_mass, pat.row_ptr, pat.row_mask, mvals);
  else
    k_mass_strip<2><<<blocks, 192, 0, s>>>(g, b.x_s, b.lp_s, b.cell_start, p_mass, pat.row_ptr, pat.row_mask, mvals);
}

// (the workspace is not used any more; callers keep passing the bytes asked for)
extern "C" size_t gm_mass_work_bytes(const gm_grid* g) { return g ? sizeof(double) : 0; }

extern "C" int gm_mass_binned(const gm_grid* g, const gm_bins* b, const gm_pattern* pat, double p_mass,
                              double* mvals, void* work, size_t work_bytes, hipStream_t s) {
  GM_REQUIRE(g && b && pat && mvals && work, "gm_mass_binned: null argument");
  GM_REQUIRE(g->dim == 3, "gm_mass_binned: 3D grids only");
  GM_REQUIRE(work_bytes >= gm_mass_work_bytes(g), "gm_mass_binned: workspace smaller than gm_mass_work_bytes");
  const int n = g->n_nodes;
  if (n == 0) return 0;
  gm::launch_mass(*g, *b, *pat, p_mass, mvals, s);
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
// A wave per bin, its particles' weights, right-hand-side factors and flags staged in LDS together;
// two half waves take every other particle.  Bins without particles write zeros, so that the gather
// has nothing to look up.  1,048,576 particles, 139,425 nodes: 85 + 35 us (164 + 41 with each lane
// reading ids, flags and pressures one after the other, and a gather that looked at every bin).
__global__ void __launch_bounds__(256) k_p2g_bin(gm_grid g, const double* x_s, const double* lp_s,
                                                 const int* cell_start, const int* sorted, const uint8_t* ext_s,
                                                 double threshold, const uint8_t* pbc_flag, double node_h_last,
                                                 double p_mass, const double* p_part, double* cb, uint8_t* cf) {
  constexpr int PB = 16;
  __shared__ struct {
    double w[PB][3][3], m[PB], z[PB];
    uint8_t ext[PB];
  } sh[4];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int b = blockIdx.x * 4 + wave;
  if (b >= g.n_nodes) return;  // the whole wave
  auto& S = sh[wave];
  const int ks = cell_start[b], ke = cell_start[b + 1];
  auto sync = [] {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  const int t = lane & 31, half = lane >> 5;
  const int ox = t % 3, oy = (t / 3) % 3, oz = min(t / 9, 2);  // lanes 27 to 31 of a half: not stored
  const int nxy = (g.nx + 1) * (g.ny + 1);
  const double node_z = (double)(b / nxy + oz) * node_h_last;
  double rhs = 0.0;
  int on = 0;  // 1: active, 2: pressure boundary
  for (int p0 = ks; p0 < ke; p0 += PB) {
    const int np = min(PB, ke - p0);
    sync();
    double z = INFINITY, pm = 0.0;  // height of a flagged particle, m_p p_p
    if (lane < np) {
      const int k = p0 + lane, pid = sorted[k];
      if (pbc_flag && pbc_flag[pid]) z = x_s[(long)k * 3 + 2];
      if (p_part) pm = p_mass * p_part[pid];
      S.ext[lane] = ext_s[k];
      S.z[lane] = z;
    }
    if (lane < 3 * np) {
      const int a = lane % 3;
      const Axis ax = gimp_axis(x_s[(long)p0 * 3 + lane], lp_s[(long)p0 * 3 + lane], g.h[a], g.inv_h[a]);
#pragma unroll
      for (int i = 0; i < 3; ++i) S.w[lane / 3][a][i] = ax.w[i];
    }
    sync();
    if (lane < np) {
      double wsum = 1.0;
#pragma unroll
      for (int a = 0; a < 3; ++a) wsum *= S.w[lane][a][0] + S.w[lane][a][1] + S.w[lane][a][2];
      S.m[lane] = wsum * pm;
    }
    sync();
    for (int p = half; p < np; p += 2) {
      if (node_z >= S.z[p]) on |= 2;
      const uint8_t ex = S.ext[p];
      const bool in = ox < ((ex & 1) ? 3 : 2) && oy < ((ex & 2) ? 3 : 2) && oz < ((ex & 4) ? 3 : 2);
      if (!in) continue;
      const double w = S.w[p][0][ox] * S.w[p][1][oy] * S.w[p][2][oz];
      if (threshold < 0.0 || w > threshold) on |= 1;
      if (p_part) rhs += w * S.m[p];
    }
  }
  rhs += __shfl_xor(rhs, 32, 64);
  on |= __shfl_xor(on, 32, 64);
  if (lane < 27) {
    cb[(long)b * 27 + lane] = rhs;
    cf[(long)b * 27 + lane] = (uint8_t)on;
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
  k_p2g_bin<<<gm_blocks(n, 4), 256, 0, s>>>(*g, b->x_s, b->lp_s, b->cell_start, b->sorted, b->ext_s, threshold, pbc_flag,
                             node_h_last, p_mass, mrhs ? p_part : nullptr, cb, cf);
  GM_LAUNCH_CHECK();
  k_p2g_gather<<<gm_blocks(n, 256), 256, 0, s>>>(*g, cb, cf, act, bflag, mrhs);
  GM_LAUNCH_CHECK();
  return 0;
}

extern "C" size_t gm_node_jacobian_work_bytes(const gm_grid* g, int tangent_fp32) {
  if (!g) return 0;
  return (size_t)g->n_nodes * (size_t)CB_NODE * (tangent_fp32 ? sizeof(float) : sizeof(double));
}

// ------------------------------------------------------------ variants and their tuner
// Variants of the line sums: 0 the number of segments of a line that best_segments picks,
// 1 twice and 2 three times as many, 3 one segment (as few as MAX_SEG allows).  Gather
// variants: 128, 256 or 512 threads a row.  Every variant writes the same bits.
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
// rounds instead pick 1 and 3 segments for 21 x 17 x 13 (FP64) and 48 x 9 x 7 cells (FP32), 249 and
// 149 us where 2 and 6 take 212 and 117.  (Some six particles a bin are taken for granted.)
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

int launch_bins(const gm_grid* g, const gm_bins* b, const void* D, int fp32, int variant, void* work,
                hipStream_t s) {
  const int n = g->n_nodes;
  const int cus = cu_count();
  GM_REQUIRE(cus > 0, "gm_jacobian_bins: no device properties");
  const int nbx = g->nx + 1, lines = n / nbx;
  const int slots = cus;  // one workgroup per CU (the operand buffers in LDS)
  int n_seg = best_segments(nbx, lines, b->n_particles, slots);
  if (variant == 1) n_seg *= 2;
  if (variant == 2) n_seg *= 3;
  if (variant == 3) n_seg = 1;
  n_seg = std::min(std::max(n_seg, (nbx + MAX_SEG - 1) / MAX_SEG), nbx);
  const int len = (nbx + n_seg - 1) / n_seg;
  const unsigned wgs = (unsigned)lines * n_seg;
  if (fp32)
    k_jac_line<float, float, 8><<<wgs, 1024, 0, s>>>(*g, b->x_s, b->lp_s, b->cell_start, b->n_particles, len, n_seg,
                                                  (const float*)D, (float*)work);
  else
    k_jac_line<double, double, 4><<<wgs, 512, 0, s>>>(*g, b->x_s, b->lp_s, b->cell_start, b->n_particles, len,
                                                   n_seg, (const double*)D, (double*)work);
  GM_LAUNCH_CHECK();
  return 0;
}

int launch_gather(const gm_grid* g, const gm_bins* b, const gm_pattern* pat, int fp32, int variant,
                  const void* work, const uint8_t* freem, void* vals, int vals_fp32, hipStream_t s) {
  const int n = g->n_nodes;
#define GM_GATHER_T(TCC, TVV, T)                                                                               \
  k_jac_gather<TCC, TVV, T><<<n, T, 0, s>>>(*g, b->cell_start, (const TCC*)work, freem, pat->row_ptr,          \
                                            pat->row_mask, (TVV*)vals)
#define GM_GATHER(TCC, TVV)                          \
  do {                                               \
    if (variant == 0) GM_GATHER_T(TCC, TVV, 128);    \
    else if (variant == 1) GM_GATHER_T(TCC, TVV, 256); \
    else GM_GATHER_T(TCC, TVV, 512);                 \
  } while (0)
  if (fp32) {
    if (vals_fp32) GM_GATHER(float, float);
    else GM_GATHER(float, double);
  } else {
    if (vals_fp32) GM_GATHER(double, float);
    else GM_GATHER(double, double);
  }
#undef GM_GATHER
#undef GM_GATHER_T
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
