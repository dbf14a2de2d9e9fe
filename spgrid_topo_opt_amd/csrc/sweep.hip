// sweep.hip -- batched block sweep (see sweep.hpp).
//
// Sweeping pivot block K of a symmetric matrix: D = A_KK, W_i = A_iK D^-1,
// A_ij -= W_i A_jK^T for all other i, j, A_iK = W_i, A_KK = -D^-1.  After all
// pivots of an SPD matrix it holds -A^-1; after the pivots of a front it holds
// the front's inverse, its multipliers A21 A11^-1 and its update matrix, which
// is all that the bottom solve needs.  The pivots met on the way are those of
// the Cholesky factorization, so the matrix is positive definite exactly when
// all are positive.
//
// D^-1 is never applied as one matrix: with D = L L^T and M = L^-1, the panel is
// Y_i = A_iK M^T, the update A_ij -= Y_i Y_j^T and W_i = Y_i M.  An update
// through W_i = A_iK D^-1 loses the soft parts of a design behind a solid pivot
// (moduli 1 and 9e-9, 3 K to 7 K unknowns, residual of a solve: 6e6 to 6e7 of
// the right-hand side, this form and LAPACK's Cholesky 2e-7 to 1.5e-6).
//
// Every step is two launches over the whole batch: the panels Y, then the
// trailing tiles; the workgroup of the next diagonal tile also factors it, so
// that serial part runs beside the others, and so do W and -D^-1, which nothing
// in the step waits for.  The products are 64x64x64 FP64
// tiles on the matrix cores (v_mfma_f64_16x16x4), both operands staged in LDS,
// the result tile in registers.  Small batches are bound by the serial
// factorization of the diagonal tiles (64 dependent pivots each).  A density
// update, against one tile inverse applied as a matrix: dense 2.8 -> 2.6 ms at
// 3,072 unknowns, nested dissection 1.3 -> 1.3 ms there and 2.9 -> 2.7 ms at
// 15,120 (partial Cholesky front by front through rocSOLVER: 12.6, 12.6 and 62
// ms); with W and -D^-1 in the chain of the panel and of the factorization 3.2,
// 1.6 and 3.2 ms.
// The residual of a solve is 0.4 to 1.3 times rocSOLVER's over 3 K to 15 K
// unknowns, ordinary and high-contrast designs.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "sweep.hpp"

namespace spg {

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
// row stride of a staged tile: 16 rows x 4 columns of an operand fall on
// distinct banks in two passes, and rows stay 16-byte aligned
constexpr int LD = 68;

// trailing tiles take their operands in halves of 32 columns
constexpr int HLD = 36;
// stage columns 32h .. 32h + 31 of a row-major 64x64 tile, times sgn
__device__ __forceinline__ void load_half(const double* __restrict__ t, int h, double2 (&v)[4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int e = threadIdx.x + 256 * i;
    v[i] = *reinterpret_cast<const double2*>(t + (e >> 4) * 64 + 32 * h + (e & 15) * 2);
  }
}
__device__ __forceinline__ void put_half(const double2 (&v)[4], double (*s)[HLD], double sgn) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int e = threadIdx.x + 256 * i, r = e >> 4, c = (e & 15) * 2;
    s[r][c] = sgn * v[i].x;
    s[r][c + 1] = sgn * v[i].y;
  }
}
// stage rows 32h .. 32h + 31
__device__ __forceinline__ void stage_rows(const double* __restrict__ t, int h, double (*s)[LD]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int e = threadIdx.x + 256 * i, r = e >> 5, c = (e & 31) * 2;
    const double2 v = *reinterpret_cast<const double2*>(t + (32 * h + r) * 64 + c);
    s[r][c] = v.x;
    s[r][c + 1] = v.y;
  }
}
// stage a row-major 64x64 tile, times sgn
__device__ __forceinline__ void stage(const double* __restrict__ t, double (*s)[LD], double sgn) {
  for (int e = threadIdx.x; e < 2048; e += 256) {
    const double2 v = reinterpret_cast<const double2*>(t)[e];
    const int r = e >> 5, c = (e & 31) * 2;
    s[r][c] = sgn * v.x;
    s[r][c + 1] = sgn * v.y;
  }
}

// acc += A B^T over K = 64; wave w owns rows (w>>1)*32.. and columns
// (w&1)*32..; lane l of a 16x16 result holds rows 4q + (l>>4), column l & 15
template <int K = 64, int S = LD>
__device__ __forceinline__ void mm64(const double (*A)[S], const double (*B)[S], d4 (&acc)[2][2]) {
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  const int ra = (w >> 1) * 32 + (l & 15), rb = (w & 1) * 32 + (l & 15), k0 = l >> 4;
#pragma unroll
  for (int k = 0; k < K; k += 4) {
    const double a0 = A[ra][k + k0], a1 = A[ra + 16][k + k0];
    const double b0 = B[rb][k + k0], b1 = B[rb + 16][k + k0];
    acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, acc[0][0], 0, 0, 0);
    acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b1, acc[0][1], 0, 0, 0);
    acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, acc[1][0], 0, 0, 0);
    acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, acc[1][1], 0, 0, 0);
  }
}
// acc += A B and acc += B^T B over 32 rows of B (A: the matching columns),
// results placed as above
__device__ __forceinline__ void mm32n(const double (*A)[HLD], const double (*B)[LD], d4 (&acc)[2][2]) {
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  const int ra = (w >> 1) * 32 + (l & 15), rb = (w & 1) * 32 + (l & 15), k0 = l >> 4;
#pragma unroll
  for (int k = 0; k < 32; k += 4) {
    const double a0 = A[ra][k + k0], a1 = A[ra + 16][k + k0];
    const double b0 = B[k + k0][rb], b1 = B[k + k0][rb + 16];
    acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, acc[0][0], 0, 0, 0);
    acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b1, acc[0][1], 0, 0, 0);
    acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, acc[1][0], 0, 0, 0);
    acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, acc[1][1], 0, 0, 0);
  }
}
__device__ __forceinline__ void mm32sq(const double (*B)[LD], d4 (&acc)[2][2]) {
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  const int ra = (w >> 1) * 32 + (l & 15), rb = (w & 1) * 32 + (l & 15), k0 = l >> 4;
#pragma unroll
  for (int k = 0; k < 32; k += 4) {
    const double a0 = B[k + k0][ra], a1 = B[k + k0][ra + 16];
    const double b0 = B[k + k0][rb], b1 = B[k + k0][rb + 16];
    acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, acc[0][0], 0, 0, 0);
    acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b1, acc[0][1], 0, 0, 0);
    acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, acc[1][0], 0, 0, 0);
    acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, acc[1][1], 0, 0, 0);
  }
}
// position of element q of sub-tile (i, j) of the caller's accumulators
__device__ __forceinline__ void acc_pos(int i, int j, int q, int& row, int& col) {
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  row = (w >> 1) * 32 + i * 16 + 4 * q + (l >> 4);
  col = (w & 1) * 32 + j * 16 + (l & 15);
}

template <int CTRL>
__device__ __forceinline__ double dpp_d(double x) {
  const long long v = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(v & 0xffffffffll), CTRL, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(v >> 32), CTRL, 0xF, 0xF, true);
  return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}
// value of one lane, the same for all, in scalar registers
__device__ __forceinline__ double lane_d(double x, int lane) {
  const long long v = __double_as_longlong(x);
  const unsigned lo = __builtin_amdgcn_readlane((int)(v & 0xffffffffll), lane);
  const unsigned hi = __builtin_amdgcn_readlane((int)(v >> 32), lane);
  return __longlong_as_double(((long long)hi << 32) | (long long)lo);
}
// P = L L^T of a 16x16 SPD block held by a wave (lane l: rows 4 (l>>4) + i,
// column l & 15), pivot KK and the following ones.  Elimination by columns: at
// the end column c holds, above the diagonal, row c of the inverse of the unit
// triangular factor, and `dc` the pivot L_cc^2 (its root is taken once, not in
// the chain of pivots).
template <int KK>
__device__ __forceinline__ void chol16(double (&a)[4], double& dc, int& bad, int pivot0) {
  if constexpr (KK < 16) {
    const int l = threadIdx.x & 63, g = l >> 4, c = l & 15;
    constexpr int gk = KK >> 2, ik = KK & 3;
    const double d = lane_d(a[ik], 16 * gk + KK);
    const double row = __shfl(a[ik], 16 * gk + c, 64);
    double ci[4];  // the pivot column: lane KK of each 16 (row_newbcast)
#pragma unroll
    for (int i = 0; i < 4; ++i) ci[i] = dpp_d<0x150 + KK>(a[i]);
    if (!(d > 0.0) && bad == 0) bad = pivot0 + KK + 1;
    const double pr = row * (1.0 / d);
    dc = c == KK ? d : dc;
    if (c > KK) {
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = (g == gk && i == ik) ? -pr : __builtin_fma(-ci[i], pr, a[i]);
    }
    chol16<KK + 1>(a, dc, bad, pivot0);
  }
}

// The 64x64 SPD tile in LDS (lower blocks and whole diagonal blocks are read)
// -> M = L^-1 in minv, by blocks of 16.  Every wave factors the pivot block (no
// barrier between its 16 dependent pivots); wave r below it takes row block r:
// Y_r^T = M_KK A_rK^T, whose result registers are the left operand of A_rj -= Y_r
// Y_j^T and of the rows of M, T_rc -= Y_r M_Kc, when the sum over k runs in the
// order that they hold; the pivot's own wave finishes M_Kc = M_KK T_Kc.  Y_j^T
// waits in the block above the diagonal, which holds nothing else.  Two barriers
// per block.  Inlined: as a call it takes the caller 4 registers too many for
// four workgroups a CU.
__device__ __forceinline__ void factor_tile(double (*s)[LD], double (*mk)[17], double* __restrict__ minv,
                                            int* __restrict__ info, int pivot0) {
  const int r = threadIdx.x >> 6, l = threadIdx.x & 63, g = l >> 4, c = l & 15;
  int bad = 0;
  for (int K = 0; K < 4; ++K) {
    const int o = 16 * K;
    double a[4], dc = 1.0;
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] = s[o + 4 * g + i][o + c];
    chol16<0>(a, dc, bad, pivot0 + o);
    const double rs = 1.0 / sqrt(dc);
    double m[4];  // M_KK[c][4 g + i]
#pragma unroll
    for (int i = 0; i < 4; ++i) m[i] = 4 * g + i < c ? a[i] * rs : (4 * g + i == c ? rs : 0.0);
    d4 y = {};
    if (r > K) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        y = __builtin_amdgcn_mfma_f64_16x16x4f64(m[i], s[16 * r + c][o + 4 * g + i], y, 0, 0, 0);
#pragma unroll
      for (int q = 0; q < 4; ++q) s[o + 4 * q + g][16 * r + c] = y[q];
    } else if (r == K) {
      for (int j = 0; j < K; ++j) {
        d4 acc = {};
#pragma unroll
        for (int i = 0; i < 4; ++i)
          acc = __builtin_amdgcn_mfma_f64_16x16x4f64(m[i], s[o + 4 * g + i][16 * j + c], acc, 0, 0, 0);
#pragma unroll
        for (int q = 0; q < 4; ++q) s[o + 4 * q + g][16 * j + c] = acc[q];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) mk[c][4 * g + i] = m[i];
    }
    __syncthreads();  // the pivot block has been read, Y and row K of M are there
    if (r > K) {
      for (int j = 0; j <= r; ++j) {
        d4 acc = {};
#pragma unroll
        for (int q = 0; q < 4; ++q)
          acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-y[q], j == K ? mk[4 * q + g][c] : s[o + 4 * q + g][16 * j + c],
                                                     acc, 0, 0, 0);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          double* p = &s[16 * r + 4 * q + g][16 * j + c];
          *p = j == K ? acc[q] : *p + acc[q];
        }
      }
    } else if (r == K) {
#pragma unroll
      for (int i = 0; i < 4; ++i) s[o + c][o + 4 * g + i] = m[i];
    }
    __syncthreads();
  }
  for (int e = threadIdx.x; e < 4096; e += 256) {
    const int i = e >> 6, j = e & 63;
    minv[e] = (j >> 4) > (i >> 4) ? 0.0 : s[i][j];
  }
  if (threadIdx.x == 0 && bad && *info == 0) *info = bad;
}

// the first diagonal tile of every matrix
__global__ void __launch_bounds__(256) k_sw_first(const SweepMat* __restrict__ mats, const double* tiles,
                                                  double* minv,
                                                  int* info) {
  __shared__ __align__(16) double s[64][LD];
  __shared__ double mk[16][17];
  const SweepMat M = mats[blockIdx.x];
  stage(tiles + M.off * 4096, s, 1.0);
  __syncthreads();
  factor_tile(s, mk, minv + (int64_t)M.id * 8192, info + M.id, 0);
}

// panels of step k: Y_i = A_iK M^T
__global__ void __launch_bounds__(256) k_sw_panel(const SweepMat* __restrict__ mats, int k,
                                                  const double* __restrict__ tiles, double* __restrict__ pan,
                                                  const double* __restrict__ minv) {
  __shared__ __align__(16) double sx[64][LD], sm[64][LD];
  const SweepMat M = mats[blockIdx.y];
  const int i = blockIdx.x;
  if (i >= M.nt || i == k) return;
  const bool below = i > k;
  const double* t = tiles + (M.off + (below ? tile_at(i, k) : tile_at(k, i))) * 4096;
  double* Y = pan + (int64_t)(M.pan + i) * 4096;
  stage(minv + ((int64_t)M.id * 2 + (k & 1)) * 4096, sm, 1.0);
  if (below) {
    stage(t, sx, 1.0);
  } else {
    for (int e = threadIdx.x; e < 4096; e += 256) sx[e & 63][e >> 6] = t[e];
  }
  __syncthreads();
  d4 acc[2][2] = {};
  mm64(sx, sm, acc);
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        int r, c;
        acc_pos(a, b, q, r, c);
        Y[r * 64 + c] = acc[a][b][q];
      }
}

// trailing tiles of step k: A_ij -= Y_i Y_j^T, i >= j, both != k; A_iK = Y_i M and
// A_KK = -M^T M.  Workgroup 0 takes the next diagonal tile and factors it into
// the other of its two places in minv, as the others still read this one.
// Large matrices are bound by the loads and stores of the tiles: operands staged
// in halves (37 KB of LDS, the second half's loads under the first product) and
// 125 registers leave room for four workgroups a CU (whole tiles: two).  Density
// update of a dense bottom 150 -> 96 ms at 15,120 unknowns, 1180 -> 767 ms at
// 30,720 (rocSOLVER 187 and 1094 ms), no difference at 3,072.
__global__ void __launch_bounds__(256, 4) k_sw_trail(const SweepMat* __restrict__ mats, int k, double* tiles,
                                                  const double* __restrict__ pan, double* minv, int* info) {
  __shared__ __align__(16) double sm[2 * 64 * HLD];
  __shared__ double mk[16][17];
  static_assert(2 * HLD >= LD, "the factored tile takes the place of the operands");
  double(*sy)[HLD] = reinterpret_cast<double(*)[HLD]>(sm);
  double(*sx)[HLD] = reinterpret_cast<double(*)[HLD]>(sm + 64 * HLD);
  double(*sw)[LD] = reinterpret_cast<double(*)[LD]>(sm);
  double(*sr)[LD] = reinterpret_cast<double(*)[LD]>(sm + 64 * HLD);
  static_assert(64 * HLD >= 32 * LD, "32 rows take the place of an operand");
  const SweepMat M = mats[blockIdx.y];
  const bool more = k + 1 < M.np;
  int i, j;
  if (blockIdx.x == 0) {
    if (!more) return;
    i = j = k + 1;
  } else {
    const int64_t e = (int64_t)blockIdx.x - 1;
    if (e >= tile_at(M.nt, 0)) return;
    i = (int)((sqrt(8.0 * (double)e + 1.0) - 1.0) * 0.5);
    while (tile_at(i + 1, 0) <= e) ++i;
    while (tile_at(i, 0) > e) --i;
    j = (int)(e - tile_at(i, 0));
    if (more && i == k + 1 && j == k + 1) return;
  }
  double* t = tiles + (M.off + tile_at(i, j)) * 4096;
  if (i == k || j == k) {
    const double* Mk = minv + ((int64_t)M.id * 2 + (k & 1)) * 4096;
    const double* Yp = pan + (int64_t)(M.pan + (i == k ? j : i)) * 4096;
    const bool diag = i == j;
    d4 acc[2][2] = {};
    for (int h = 0; h < 2; ++h) {
      if (h) __syncthreads();
      stage_rows(Mk, h, sr);
      if (!diag) {
        double2 v[4];
        load_half(Yp, h, v);
        put_half(v, sy, 1.0);
      }
      __syncthreads();
      if (diag) mm32sq(sr, acc);
      else mm32n(sy, sr, acc);
    }
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          int r, c;
          acc_pos(a, b, q, r, c);
          if (diag) t[r * 64 + c] = -acc[a][b][q];
          else t[i > k ? r * 64 + c : c * 64 + r] = acc[a][b][q];
        }
    return;
  }
  // the product is summed by itself and added once: 64 terms added to a tile
  // that holds the sums of the steps before would each round at its size
  d4 acc[2][2] = {}, old[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        int r, c;
        acc_pos(a, b, q, r, c);
        old[a][b][q] = t[r * 64 + c];
      }
  const double *Yi = pan + (int64_t)(M.pan + i) * 4096, *Yj = pan + (int64_t)(M.pan + j) * 4096;
  double2 vi[4], vj[4];
  load_half(Yi, 0, vi);
  load_half(Yj, 0, vj);
  put_half(vi, sy, -1.0);
  put_half(vj, sx, 1.0);
  __syncthreads();
  load_half(Yi, 1, vi);
  load_half(Yj, 1, vj);
  mm64<32, HLD>(sy, sx, acc);
  __syncthreads();
  put_half(vi, sy, -1.0);
  put_half(vj, sx, 1.0);
  __syncthreads();
  mm64<32, HLD>(sy, sx, acc);
  const bool next = blockIdx.x == 0;
  if (next) __syncthreads();  // sm is reused
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        int r, c;
        acc_pos(a, b, q, r, c);
        const double v = old[a][b][q] + acc[a][b][q];
        if (next) sw[r][c] = v;
        else t[r * 64 + c] = v;
      }
  if (next) {
    __syncthreads();
    factor_tile(sw, mk, minv + ((int64_t)M.id * 2 + ((k + 1) & 1)) * 4096, info + M.id, 64 * (k + 1));
  }
}

}  // namespace

void sweep_run(hipStream_t st, const SweepBatch& b, double* tiles) {
  constexpr int kMaxY = 32768;  // matrices per launch
  for (size_t m0 = 0; m0 < b.h.size(); m0 += kMaxY) {
    const int n = (int)std::min<size_t>(kMaxY, b.h.size() - m0);
    const SweepMat* h = b.h.data() + m0;
    const SweepMat* d = b.d + m0;
    if (h[0].np == 0) break;  // sorted by decreasing np
    int live = n;
    while (live > 0 && h[live - 1].np == 0) --live;
    k_sw_first<<<live, 256, 0, st>>>(d, tiles, b.minv, b.info);
    for (int k = 0; k < h[0].np; ++k) {
      while (live > 0 && h[live - 1].np <= k) --live;
      int nt = 0;
      for (int i = 0; i < live; ++i) nt = std::max(nt, h[i].nt);
      if (nt > 1) k_sw_panel<<<dim3(nt, live), 256, 0, st>>>(d, k, tiles, b.pan, b.minv);
      k_sw_trail<<<dim3((unsigned)(tile_at(nt, 0) + 1), live), 256, 0, st>>>(d, k, tiles, b.pan, b.minv, b.info);
    }
  }
}

}  // namespace spg
