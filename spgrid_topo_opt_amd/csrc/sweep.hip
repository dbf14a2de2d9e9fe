// sweep.hip -- batched block sweep (see sweep.hpp).
//
// Sweeping pivot block K of a symmetric matrix: D = A_KK, W_i = A_iK D^-1,
// A_ij -= W_i A_jK^T for all other i, j, A_iK = W_i, A_KK = -D^-1.  After all
// pivots of an SPD matrix it holds -A^-1; after the pivots of a front it holds
// the front's inverse, its multipliers A21 A11^-1 and its update matrix, which
// is all that the bottom solve needs.  The pivots met on the way are those of
// the Cholesky factorization, so the matrix is positive definite exactly when
// all are positive, and the inverse is as accurate as the one from the
// Cholesky factors.
//
// Every step is two launches over the whole batch: the panels, then the
// trailing tiles; the workgroup of the next diagonal tile also inverts it, so
// that serial part runs beside the others.  The products are 64x64x64 FP64
// tiles on the matrix cores (v_mfma_f64_16x16x4), both operands staged in LDS,
// the result tile in registers.  Small batches are bound by the serial
// inversion of the diagonal tiles (64 dependent pivots each).  Per density update,
// against partial Cholesky front by front through rocSOLVER and rocBLAS, at the
// scalar inversion: 37 -> 2.0 ms (9,006 unknowns, nested dissection), 16 -> 1.1
// ms (4,131, nested dissection), 9 -> 1.9 ms (2,016, dense); the 16x16 blocks
// take another 0.3 ms from the last two.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "sweep.hpp"

namespace spg {

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
// row stride of a staged tile: 16 rows x 4 columns of an operand fall on
// distinct banks in two passes, and rows stay 16-byte aligned
constexpr int LD = 68;

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
__device__ __forceinline__ void mm64(const double (*A)[LD], const double (*B)[LD], d4 (&acc)[2][2]) {
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  const int ra = (w >> 1) * 32 + (l & 15), rb = (w & 1) * 32 + (l & 15), k0 = l >> 4;
#pragma unroll
  for (int k = 0; k < 64; k += 4) {
    const double a0 = A[ra][k + k0], a1 = A[ra + 16][k + k0];
    const double b0 = B[rb][k + k0], b1 = B[rb + 16][k + k0];
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
// one scalar sweep of a 16x16 SPD block held by a wave (lane l: rows
// 4 (l>>4) + i, column l & 15), pivot KK and the following ones; the block
// becomes minus its inverse
template <int KK>
__device__ __forceinline__ void sweep16(double (&a)[4], int& bad, int pivot0) {
  if constexpr (KK < 16) {
    const int l = threadIdx.x & 63, g = l >> 4, c = l & 15;
    constexpr int gk = KK >> 2, ik = KK & 3;
    const double d = lane_d(a[ik], 16 * gk + KK);
    const double row = __shfl(a[ik], 16 * gk + c, 64);
    double ci[4];  // the pivot column: lane KK of each 16 (row_newbcast)
#pragma unroll
    for (int i = 0; i < 4; ++i) ci[i] = dpp_d<0x150 + KK>(a[i]);
    if (!(d > 0.0) && bad == 0) bad = pivot0 + KK + 1;
    const double inv = 1.0 / d, pr = row * inv;
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] = c == KK ? ci[i] * inv : __builtin_fma(-ci[i], pr, a[i]);
    if (g == gk) a[ik] = c == KK ? -inv : pr;
    sweep16<KK + 1>(a, bad, pivot0);
  }
}

// The 64x64 SPD tile in LDS -> minus its inverse in the tile store, the
// inverse in dinv, by the block sweep above with 16x16 blocks.  Every wave
// inverts the pivot block D (no barrier between its 16 dependent pivots), then
// wave r takes row block r: W_r^T = D^-1 X_r^T, whose result registers are the
// left operand of A_rj -= W_r X_j^T when the sum over k runs in the order that
// they hold.  Two barriers per block.  Against a scalar sweep with a barrier
// for each of the 64 pivots, a thread holding 16 rows of a column: first tile
// 33.5 -> 19.1 us, a trailing step with its next diagonal tile 38.0 -> 25.7 us.
__device__ void invert_tile(double (*s)[LD], double* __restrict__ tile, double* __restrict__ dinv,
                            int* __restrict__ info, int pivot0) {
  const int r = threadIdx.x >> 6, l = threadIdx.x & 63, g = l >> 4, c = l & 15;
  int bad = 0;
  for (int K = 0; K < 4; ++K) {
    const int o = 16 * K;
    double a[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] = s[o + 4 * g + i][o + c];
    sweep16<0>(a, bad, pivot0 + o);
    d4 wt = {};
    if (r != K) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        wt = __builtin_amdgcn_mfma_f64_16x16x4f64(-a[i], s[16 * r + c][o + 4 * g + i], wt, 0, 0, 0);
      for (int j = 0; j < 4; ++j) {
        if (j == K) continue;
        d4 acc;
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[q] = s[16 * r + 4 * q + g][16 * j + c];
#pragma unroll
        for (int q = 0; q < 4; ++q)
          acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-wt[q], s[16 * j + c][o + 4 * q + g], acc, 0, 0, 0);
#pragma unroll
        for (int q = 0; q < 4; ++q) s[16 * r + 4 * q + g][16 * j + c] = acc[q];
      }
    }
    __syncthreads();  // the panel has been read
    if (r != K) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        s[16 * r + c][o + 4 * q + g] = wt[q];
        s[o + 4 * q + g][16 * r + c] = wt[q];
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) s[o + 4 * g + i][o + c] = a[i];
    }
    __syncthreads();
  }
  for (int e = threadIdx.x; e < 4096; e += 256) {
    const double v = s[e >> 6][e & 63];
    tile[e] = v;
    dinv[e] = -v;
  }
  if (threadIdx.x == 0 && bad && *info == 0) *info = bad;
}

// the first diagonal tile of every matrix
__global__ void __launch_bounds__(256) k_sw_first(const SweepMat* __restrict__ mats, double* tiles, double* dinv,
                                                  int* info) {
  __shared__ __align__(16) double s[64][LD];
  const SweepMat M = mats[blockIdx.x];
  double* t = tiles + M.off * 4096;
  stage(t, s, 1.0);
  __syncthreads();
  invert_tile(s, t, dinv + (int64_t)M.id * 4096, info + M.id, 0);
}

// panels of step k: X_i = A_iK (kept for the trailing tiles), W_i = X_i D^-1,
// A_iK = W_i
__global__ void __launch_bounds__(256) k_sw_panel(const SweepMat* __restrict__ mats, int k, double* tiles,
                                                  double* __restrict__ panw, double* __restrict__ panx,
                                                  const double* __restrict__ dinv) {
  __shared__ __align__(16) double sx[64][LD], sd[64][LD];
  const SweepMat M = mats[blockIdx.y];
  const int i = blockIdx.x;
  if (i >= M.nt || i == k) return;
  const bool below = i > k;
  double* t = tiles + (M.off + (below ? tile_at(i, k) : tile_at(k, i))) * 4096;
  double* X = panx + (int64_t)(M.pan + i) * 4096;
  double* W = panw + (int64_t)(M.pan + i) * 4096;
  stage(dinv + (int64_t)M.id * 4096, sd, 1.0);
  if (below) {
    stage(t, sx, 1.0);
  } else {
    for (int e = threadIdx.x; e < 4096; e += 256) sx[e & 63][e >> 6] = t[e];
  }
  __syncthreads();
  for (int e = threadIdx.x; e < 4096; e += 256) X[e] = sx[e >> 6][e & 63];
  d4 acc[2][2] = {};
  mm64(sx, sd, acc);
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        int r, c;
        acc_pos(a, b, q, r, c);
        W[r * 64 + c] = acc[a][b][q];
        t[below ? r * 64 + c : c * 64 + r] = acc[a][b][q];
      }
}

// trailing tiles of step k: A_ij -= W_i X_j^T, i >= j, both != k.  Workgroup 0
// takes the next diagonal tile and inverts it.
__global__ void __launch_bounds__(256) k_sw_trail(const SweepMat* __restrict__ mats, int k, double* tiles,
                                                  const double* __restrict__ panw, const double* __restrict__ panx,
                                                  double* dinv, int* info) {
  __shared__ __align__(16) double sw[64][LD], sx[64][LD];
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
    if (i == k || j == k || (more && i == k + 1 && j == k + 1)) return;
  }
  double* t = tiles + (M.off + tile_at(i, j)) * 4096;
  d4 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        int r, c;
        acc_pos(a, b, q, r, c);
        acc[a][b][q] = t[r * 64 + c];
      }
  stage(panw + (int64_t)(M.pan + i) * 4096, sw, -1.0);
  stage(panx + (int64_t)(M.pan + j) * 4096, sx, 1.0);
  __syncthreads();
  mm64(sw, sx, acc);
  const bool next = blockIdx.x == 0;
  if (next) __syncthreads();  // sw is reused
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        int r, c;
        acc_pos(a, b, q, r, c);
        if (next) sw[r][c] = acc[a][b][q];
        else t[r * 64 + c] = acc[a][b][q];
      }
  if (next) {
    __syncthreads();
    invert_tile(sw, t, dinv + (int64_t)M.id * 4096, info + M.id, 64 * (k + 1));
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
    k_sw_first<<<live, 256, 0, st>>>(d, tiles, b.dinv, b.info);
    for (int k = 0; k < h[0].np; ++k) {
      while (live > 0 && h[live - 1].np <= k) --live;
      int nt = 0;
      for (int i = 0; i < live; ++i) nt = std::max(nt, h[i].nt);
      if (nt == 1) break;  // a single tile is done
      k_sw_panel<<<dim3(nt, live), 256, 0, st>>>(d, k, tiles, b.panw, b.panx, b.dinv);
      k_sw_trail<<<dim3((unsigned)(tile_at(nt, 0) + 1), live), 256, 0, st>>>(d, k, tiles, b.panw, b.panx, b.dinv,
                                                                             b.info);
    }
  }
}

}  // namespace spg
