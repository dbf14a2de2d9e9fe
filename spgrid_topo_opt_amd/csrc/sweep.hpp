// sweep.hpp -- batched block sweep of symmetric positive definite FP64
// matrices in packed 64x64 tiles (sweep.hip): the numeric kernels of the
// bottom factorization.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

namespace spg {

// A symmetric matrix of nt x nt tiles as its lower triangle: tile (I, J),
// I >= J, row-major at (off + I(I+1)/2 + J) * 4096 of the tile store, diagonal
// tiles whole.  The first np tile rows are pivots.
struct SweepMat {
  int64_t off;
  int32_t np, nt;
  int32_t pan;  // first tile of its panels
  int32_t id;   // slot of its diagonal factor and of its error word
};

__host__ __device__ inline int64_t tile_at(int I, int J) { return (int64_t)I * (I + 1) / 2 + J; }

// A batch of matrices swept together, kept on the device with its workspace.
struct SweepBatch {
  std::vector<SweepMat> h;  // by decreasing np
  SweepMat* d = nullptr;    // device copy of h
  double *pan = nullptr, *minv = nullptr;  // panels; two inverse factors of diagonal tiles per id
  int* info = nullptr;      // per id: 0, or 1 + the first pivot that is not positive
};

// Sweeps the pivots of every matrix of the batch in place:
//   [A11 .; A21 A22] -> [-A11^-1 .; A21 A11^-1, A22 - A21 A11^-1 A12].
void sweep_run(hipStream_t st, const SweepBatch& b, double* tiles);

}  // namespace spg
