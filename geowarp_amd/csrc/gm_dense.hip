// Inverse of the multigrid hierarchy's coarsest operator (a few hundred to a few thousand dofs,
// block-CSR, FP64) as a dense matrix on the device.
//
// In-place Gauss-Jordan by blocks of 32, one launch a block: with D the inverse of the pivot block,
//   A_ij -= A_ik D A_kj,  A_kj = D A_kj,  A_ik = -A_ik D,  A_kk = D  (i, j != k),
// from one buffer into another, so every 32x32 tile is a workgroup of its own that needs nothing
// of the others.  Products on the FP64 matrix cores (16x16x4), a quarter tile a wave; operands
// come straight from global memory, all loads up front, and only A_ik D passes through LDS.  The
// workgroup of the next pivot tile inverts it as soon as it has it (rows pivoted inside the block)
// and starts first.  Rows and columns are scaled by powers of two to a unit diagonal, so that the
// pivots of dofs of different units (displacement, pressure) compare.  What bounds it is the chain of ceil(n / 32) launches, each about the 32
// dependent columns of one pivot block.  Blocks are not pivoted against each other: a probe of
// A A^-1 measures the result, and the caller falls back to a pivoted factorisation when it is off.
#include <hip/hip_runtime.h>

#include "gm_common.h"
#include "gm_types.h"

namespace {

constexpr int DB = 32;
typedef double d4v __attribute__((ext_vector_type(4)));

// scale_i: the power of two next to sqrt|a_ii| (1 where it is zero), and the probe v_i = +-scale_i
__global__ void k_scale(int n, int nb, const int* row_ptr, const int* col_idx, const double* vals, double* scale,
                        double* v, double* err) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) *err = 0.0;
  if (i >= n) return;
  const int I = i / nb, c = i % nb;
  double d = 0.0;
  for (int s = row_ptr[I]; s < row_ptr[I + 1]; ++s)
    if (col_idx[s] == I) d = fabs(vals[(long)s * nb * nb + c * nb + c]);
  int e = 0;
  if (d > 0.0 && d < INFINITY) frexp(sqrt(d), &e);
  d = ldexp(1.0, e);
  scale[i] = d;
  v[i] = ((unsigned)i * 2654435761u) >> 31 ? d : -d;
}

// dense copy of a block-CSR matrix, row i and column i divided by scale_i: a workgroup per block row
__global__ void __launch_bounds__(256) k_dense_fill(int n_nodes, int nb, const int* row_ptr, const int* col_idx,
                                                    const double* vals, const double* scale, double* A) {
  const int I = blockIdx.x, n = n_nodes * nb, nb2 = nb * nb;
  double* row = A + (long)I * nb * n;
  for (int q = threadIdx.x; q < nb * n; q += 256) row[q] = 0.0;
  __syncthreads();
  const int s0 = row_ptr[I], s1 = row_ptr[I + 1];
  for (int q = threadIdx.x; q < (s1 - s0) * nb2; q += 256) {
    const int s = s0 + q / nb2, r = q % nb2 / nb, c = q % nb;
    const int j = col_idx[s] * nb + c;
    row[(long)r * n + j] = vals[(long)s * nb2 + r * nb + c] / scale[I * nb + r] / scale[j];
  }
}

struct Pivot {
  double m[DB][DB + 1];
  int row[DB];  // pivot row of each column
};

__device__ __forceinline__ double lane_of(double v, int l) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                          __builtin_amdgcn_readlane(__double2loint(v), l));
}

// Gauss-Jordan inverse of s.m by one wave, in registers: lane l holds half l / 32 of row l % 32, 16
// columns.  The columns rotate, so that the current one is always the first of the lower half and
// no register is indexed by the loop; the largest remaining entry of the column is its pivot.  A
// singular block gives infinities or NaN.  (256 threads with the block in LDS and a barrier a
// column: 21.4 us a block step of 602 dofs, 19.5 so.)
__device__ void invert_block(Pivot& s, double* out) {
  __syncthreads();
  if (threadIdx.x >= 64) return;
  const int lane = threadIdx.x, r = lane & 31, h = lane >> 5;
  double a[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) a[k] = s.m[r][16 * h + k];
  bool used = false;
  int mine = 0;  // the column that the row is the pivot of
#pragma unroll 1
  for (int c = 0; c < DB; ++c) {
    const double cur = a[0];  // lower half: column c
    // order by the high word of |a| (5 low mantissa bits of it give way to the row)
    unsigned key = used ? 0u : ((unsigned)__double2hiint(cur) & 0x7fffffe0u) | (31u - r) | 0x80000000u;
    key = max(key, (unsigned)__builtin_amdgcn_update_dpp(0, (int)key, 0x121, 0xf, 0xf, false));
    key = max(key, (unsigned)__builtin_amdgcn_update_dpp(0, (int)key, 0x122, 0xf, 0xf, false));
    key = max(key, (unsigned)__builtin_amdgcn_update_dpp(0, (int)key, 0x124, 0xf, 0xf, false));
    key = max(key, (unsigned)__builtin_amdgcn_update_dpp(0, (int)key, 0x128, 0xf, 0xf, false));
    key = max((unsigned)__builtin_amdgcn_readlane((int)key, 0), (unsigned)__builtin_amdgcn_readlane((int)key, 16));
    const int p = 31 - (int)(key & 31u);
    double raw[16];  // the pivot row
#pragma unroll
    for (int k = 0; k < 16; ++k) raw[k] = __shfl(a[k], p + 32 * h, 64);
    const double inv = 1.0 / lane_of(cur, p), f = __shfl(cur, r, 64) * inv;
    if (r == p) {
      used = true;
      mine = c;
    }
    // the rest of the row, one register down; column c itself: -f, inv in the pivot row
    const double col = r == p ? inv : -f, first = r == p ? a[0] * inv : a[0] - f * raw[0];
    const double out0 = __shfl_xor(h == 0 ? col : first, 32, 64);
#pragma unroll
    for (int k = 0; k < 15; ++k) a[k] = a[k + 1] - f * raw[k + 1];
    if (r == p)
#pragma unroll
      for (int k = 0; k < 15; ++k) a[k] = raw[k + 1] * inv;
    a[15] = out0;
    if (lane == 0) s.row[c] = p;
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int k = 0; k < 16; ++k) out[mine * DB + s.row[16 * h + k]] = a[k];
}

// entry of A, continued by the identity outside
__device__ __forceinline__ double entry(int n, const double* A, int i, int j) {
  return (i < n && j < n) ? A[(long)i * n + j] : (i == j ? 1.0 : 0.0);
}

__global__ void __launch_bounds__(256) k_pivot_first(int n, const double* A, double* D) {
  __shared__ Pivot s;
  for (int q = threadIdx.x; q < DB * DB; q += 256) s.m[q / DB][q % DB] = entry(n, A, q / DB, q % DB);
  invert_block(s, D);
}

// step k of nt: A -> B; the pivot block's inverse is D[k & 1], the next one goes to D[(k + 1) & 1];
// the last step takes the scale off
__global__ void __launch_bounds__(256) k_gauss_jordan(int n, int nt, int k, const double* A, double* B, double* D,
                                                     const double* scale) {
  __shared__ union {
    double w[DB][DB + 2];
    Pivot s;
  } sh;
  int tile = blockIdx.x;
  const int next = (k + 1) * (nt + 1);  // tile (k + 1, k + 1), taken by the first workgroup
  if (k + 1 < nt) tile = tile == 0 ? next : (tile == next ? 0 : tile);
  const int ti = tile / nt, tj = tile % nt;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l = lane & 15, g = lane >> 4;
  const int r0 = (wave >> 1) * 16, c0 = (wave & 1) * 16;  // the wave's quarter
  const double* Dk = D + (k & 1) * DB * DB;
  double left[8], mid[8], right[8];
  d4v acc;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    // first product: A_ik D (or, in the pivot row, D A_kj); second: (A_ik D) A_kj
    left[q] = ti == k ? Dk[(r0 + l) * DB + 4 * q + g] : entry(n, A, ti * DB + r0 + l, k * DB + 4 * q + g);
    mid[q] = Dk[(4 * q + g) * DB + c0 + l];
    right[q] = entry(n, A, k * DB + 4 * q + g, tj * DB + c0 + l);
  }
#pragma unroll
  for (int q = 0; q < 4; ++q)
    acc[q] = (ti == k || tj == k) ? 0.0 : entry(n, A, ti * DB + r0 + 4 * q + g, tj * DB + c0 + l);
  if (ti == k && tj == k) {
#pragma unroll
    for (int q = 0; q < 4; ++q) acc[q] = Dk[(r0 + 4 * q + g) * DB + c0 + l];
  } else {
    d4v w = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < 8; ++q)
      w = __builtin_amdgcn_mfma_f64_16x16x4f64(left[q], ti == k ? right[q] : mid[q], w, 0, 0, 0);
    if (ti == k) {
      acc = w;
    } else if (tj == k) {
      acc = -w;
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) sh.w[r0 + 4 * q + g][c0 + l] = -w[q];
      __syncthreads();
#pragma unroll
      for (int q = 0; q < 8; ++q)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(sh.w[r0 + l][4 * q + g], right[q], acc, 0, 0, 0);
    }
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int i = ti * DB + r0 + 4 * q + g, j = tj * DB + c0 + l;
    if (i < n && j < n) B[(long)i * n + j] = k + 1 < nt ? acc[q] : acc[q] / scale[i] / scale[j];
  }
  if (ti == k + 1 && tj == k + 1) {
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int i = r0 + 4 * q + g, j = c0 + l;
      // outside the matrix the tile continues as the identity
      sh.s.m[i][j] = max(ti * DB + i, tj * DB + j) < n ? acc[q] : (i == j ? 1.0 : 0.0);
    }
    invert_block(sh.s, D + ((k + 1) & 1) * DB * DB);
  }
}

// y = X v, a wave per row
__global__ void __launch_bounds__(256) k_probe_mv(int n, const double* X, const double* v, double* y) {
  const int i = blockIdx.x * 4 + threadIdx.x / 64, lane = threadIdx.x & 63;
  double s = 0.0;
  if (i < n)
    for (int j = lane; j < n; j += 64) s += X[(long)i * n + j] * v[j];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  if (i < n && lane == 0) y[i] = s;
}

// err = max_i |(A y - v)_i| / scale_i; a NaN counts as the largest (bits of |r| as an integer)
__global__ void k_probe_error(int n, int nb, const int* row_ptr, const int* col_idx, const double* vals,
                              const double* y, const double* v, const double* scale, double* err) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int I = i / nb, r = i % nb;
  double s = -v[i];
  for (int q = row_ptr[I]; q < row_ptr[I + 1]; ++q)
    for (int c = 0; c < nb; ++c) s += vals[(long)q * nb * nb + r * nb + c] * y[col_idx[q] * nb + c];
  atomicMax((unsigned long long*)err, (unsigned long long)__double_as_longlong(fabs(s) / scale[i]));
}

}  // namespace

extern "C" size_t gm_dense_inverse_work_bytes(int n) {
  if (n <= 0) return 0;
  return sizeof(double) * ((size_t)n * n + 2 * DB * DB + 3 * (size_t)n);
}

extern "C" int gm_dense_inverse(int nb, int n_nodes, const int* row_ptr, const int* col_idx, const double* vals,
                                double* inv, void* work, size_t work_bytes, double* err, hipStream_t s) {
  GM_REQUIRE(row_ptr && col_idx && vals && inv && work && err, "gm_dense_inverse: null argument");
  GM_REQUIRE(nb >= 1 && n_nodes >= 1 && (long)nb * n_nodes <= 65536, "gm_dense_inverse: bad size");
  const int n = nb * n_nodes, nt = (n + DB - 1) / DB;
  GM_REQUIRE(work_bytes >= gm_dense_inverse_work_bytes(n), "gm_dense_inverse: workspace too small");
  double* other = (double*)work;
  double *D = other + (size_t)n * n, *v = D + 2 * DB * DB, *y = v + n, *scale = y + n;
  // an even number of steps ends in the buffer it starts from
  double *a = nt % 2 ? other : inv, *b = nt % 2 ? inv : other;
  k_scale<<<gm_blocks(n, 256), 256, 0, s>>>(n, nb, row_ptr, col_idx, vals, scale, v, err);
  k_dense_fill<<<n_nodes, 256, 0, s>>>(n_nodes, nb, row_ptr, col_idx, vals, scale, a);
  k_pivot_first<<<1, 256, 0, s>>>(n, a, D);
  for (int k = 0; k < nt; ++k) {
    k_gauss_jordan<<<nt * nt, 256, 0, s>>>(n, nt, k, a, b, D, scale);
    double* c = a;
    a = b;
    b = c;
  }
  k_probe_mv<<<gm_blocks(n, 4), 256, 0, s>>>(n, inv, v, y);
  k_probe_error<<<gm_blocks(n, 256), 256, 0, s>>>(n, nb, row_ptr, col_idx, vals, y, v, scale, err);
  GM_LAUNCH_CHECK();
  return 0;
}
