// bottom_nd.hip -- exact FP64 bottom solve by a nested-dissection
// multifrontal Cholesky factorization on the GPU.
//
// The reference factorizes the bottom level's Dirichlet-deleted stencil
// matrix with MKL PARDISO (nested-dissection ordering, sparse supernodal
// Cholesky; solver/MG/Elasticity_Matrix.cpp:15-269, called from
// MG/Multigrid_Hierarchy.h:332-372) and solves it once per V-cycle.  This
// file does the same job for bottoms too large for a dense inverse:
//
//   ordering   geometric nested dissection of the bottom nodes: the node box
//              is cut by the median plane normal to its longest axis; a plane
//              of nodes separates the two halves of a 27-point stencil.
//   symbolic   one front per separator (and per leaf box): its pivots are
//              eliminated together, its boundary is the set of later nodes
//              coupled to its subtree (host, once per topology).
//   numeric    all fronts of a tree depth together, deepest first: the stencil
//              entries and the children's update matrices in packed 64x64
//              tiles (pivots padded to whole tiles with ones on the diagonal),
//              then the block sweep of the pivots (sweep.hip), which leaves
//              -A11^-1, G = A21 A11^-1 and the update matrix in place.
//   solve      forward (deepest fronts first): u = w_B - G w_P, with w the
//              front's right-hand side plus its children's update vectors;
//              backward (root first): x_P = A11^-1 w_P - G^T x_B.  One launch
//              per tree depth and direction, a workgroup per tile row; each
//              gathers the vectors it needs, and sums run in a fixed order, so
//              a solve is deterministic.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstdint>
#include <functional>
#include <cstdio>
#include <numeric>
#include <stdexcept>
#include <string>
#include <vector>

#include "bottom_nd.hpp"
#include "kernels.hpp"

namespace spg {

namespace {

// a box of at most this many nodes is one front: fewer tree depths and launches
// per solve against larger pivot blocks.  Solve with 64 / 192 / 400: 56 / 49 /
// 46 us at 4,131 unknowns, 100 / 80 / 75 us at 9,006; density update 1.5 / 1.6 /
// 2.0 and 8.5 / 8.5 / 9.2 ms.
constexpr int kLeafNodes = 192;

#define NDCHK(x)                                                                              \
  do {                                                                                        \
    hipError_t e_ = (x);                                                                      \
    if (e_ != hipSuccess) throw std::runtime_error(std::string(#x) + ": " + hipGetErrorString(e_)); \
  } while (0)

// ------------------------------------------------------------------ kernels
// a front's local dof (pivots, then boundary) in its padded tile matrix
__device__ __forceinline__ int padded(int f, int p, int tp) { return f < p ? f : tp * 64 + (f - p); }

// add (or set) an entry of the lower triangle, r >= c; diagonal tiles are whole
__device__ __forceinline__ void add_entry(double* __restrict__ m, int r, int c, double v) {
  const int R = r >> 6, C = c >> 6;
  double* t = m + tile_at(R, C) * 4096;
  t[(r & 63) * 64 + (c & 63)] += v;
  if (R == C && r != c) t[(c & 63) * 64 + (r & 63)] += v;
}

// ones on the diagonal of the padded pivots
__global__ void k_nd_pad(const NdFrontDev* __restrict__ fr, double* __restrict__ tiles) {
  const NdFrontDev F = fr[blockIdx.x];
  const int r = F.p + threadIdx.x;
  if (r < F.tp * 64) tiles[(F.t_off + tile_at(r >> 6, r >> 6)) * 4096 + (r & 63) * 65] = 1.0;
}

// Stencil entries of all fronts: entry e = (slot of pivot node i, spoke s,
// local dof of i, local dof of neighbour j) of front of[e]; F(j*, i*) =
// st(i, s) (the transpose of row i's block, by symmetry).
__global__ void k_nd_assemble(int64_t n, const int4* __restrict__ ent, const int* __restrict__ of,
                              const NdFrontDev* __restrict__ fr, const double* __restrict__ ST,
                              double* __restrict__ tiles) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= n * 9) return;
  const int4 e = ent[g / 9];
  const NdFrontDev F = fr[of[g / 9]];
  const int v = (int)(g % 9) / 3, w = (int)(g % 9) % 3;
  if (e.w + w < e.z + v) return;  // above the diagonal of a node's own block
  add_entry(tiles + F.t_off * 4096, padded(e.w + w, F.p, F.tp), e.z + v, ST[st_index(e.x >> 6, e.x & 63, e.y * 9 + v * 3 + w)]);
}

// a child's update matrix added to its parent's entries; blockIdx.y: child of
// the list, blockIdx.x: tile of its update matrix (children of one parent run
// in separate launches)
__global__ void __launch_bounds__(256) k_nd_extend_add(const int* __restrict__ child, const NdFrontDev* __restrict__ fr,
                                                       const int* __restrict__ emap, double* __restrict__ tiles) {
  const NdFrontDev C = fr[child[blockIdx.y]];
  const int64_t e = blockIdx.x;
  if (e >= tile_at(C.tb, 0)) return;
  int R = (int)((sqrt(8.0 * (double)e + 1.0) - 1.0) * 0.5);
  while (tile_at(R + 1, 0) <= e) ++R;
  while (tile_at(R, 0) > e) --R;
  const int S = (int)(e - tile_at(R, 0));
  const NdFrontDev P = fr[C.parent];
  const double* u = tiles + (C.t_off + tile_at(C.tp + R, C.tp + S)) * 4096;
  const int* map = emap + C.emap_off;
  double* m = tiles + P.t_off * 4096;
  for (int q = threadIdx.x; q < 4096; q += 256) {
    const int a = R * 64 + (q >> 6), c = S * 64 + (q & 63);
    if (a >= C.b || c > a) continue;
    add_entry(m, padded(map[a], P.p, P.tp), padded(map[c], P.p, P.tp), u[q]);
  }
}

// The solve reads every tile with the output along the lanes: output c of a
// tile row adds T[r][c] v[r].  The multipliers of the forward pass and the
// tiles above the diagonal of A11^-1 are kept transposed for that.
__global__ void __launch_bounds__(256) k_nd_transpose(const NdFrontDev* __restrict__ fr,
                                                      const double* __restrict__ tiles, double* __restrict__ tr) {
  __shared__ double s[64][65];
  const NdFrontDev F = fr[blockIdx.y];
  const int64_t e = blockIdx.x, nsq = (int64_t)F.tp * (F.tp - 1) / 2;
  if (e >= nsq + (int64_t)F.tb * F.tp) return;
  int I, J;
  if (e < nsq) {  // strictly lower tiles of the pivot block
    I = (int)((sqrt(8.0 * (double)e + 1.0) + 1.0) * 0.5);
    while ((int64_t)I * (I - 1) / 2 > e) --I;
    while ((int64_t)(I + 1) * I / 2 <= e) ++I;
    J = (int)(e - (int64_t)I * (I - 1) / 2);
  } else {
    I = F.tp + (int)((e - nsq) / F.tp);
    J = (int)((e - nsq) % F.tp);
  }
  const double* t = tiles + (F.t_off + tile_at(I, J)) * 4096;
  double* o = tr + (F.tr_off + e) * 4096;
  for (int q = threadIdx.x; q < 4096; q += 256) s[q & 63][q >> 6] = t[q];
  __syncthreads();
  for (int q = threadIdx.x; q < 4096; q += 256) o[q] = s[q >> 6][q & 63];
}

constexpr int kWaves = 8;       // waves of a solve workgroup, a tile each at a time
constexpr int kChunk = 2048;    // vector entries staged at a time
static_assert(kChunk % (64 * kWaves) == 0, "a wave's tiles of a chunk start at its own number");

// acc + sum_r T[r][lane] v[r]
__device__ __forceinline__ double tile_dot(const double* __restrict__ T, const double* v, int lane, double acc) {
  double a0 = acc, a1 = 0.0, a2 = 0.0, a3 = 0.0;
#pragma unroll 8
  for (int r = 0; r < 64; r += 4) {
    a0 = __builtin_fma(T[r * 64 + lane], v[r], a0);
    a1 = __builtin_fma(T[(r + 1) * 64 + lane], v[r + 1], a1);
    a2 = __builtin_fma(T[(r + 2) * 64 + lane], v[r + 2], a2);
    a3 = __builtin_fma(T[(r + 3) * 64 + lane], v[r + 3], a3);
  }
  return (a0 + a1) + (a2 + a3);
}
// sum of the waves' partial results of one output tile row, in wave order
__device__ __forceinline__ double tile_sum(double acc, double (*ys)[64]) {
  const int t = threadIdx.x;
  ys[t >> 6][t & 63] = acc;
  __syncthreads();
  double v = 0.0;
  if (t < 64)
#pragma unroll
    for (int w = 0; w < kWaves; ++w) v += ys[w][t];
  return v;
}
// a front's own right-hand side at local dof f: its row of b (pivots) plus the
// children's update entries
template <class T>
__device__ __forceinline__ double front_rhs(const NdFrontDev& F, int f, const int2* __restrict__ kid,
                                            const int* __restrict__ vmap, const T* __restrict__ b,
                                            const double* ustore) {
  const int2 k = kid[F.k_off + f];
  double v = f < F.p ? (double)b[vmap[F.dof0 + f]] : 0.0;
  if (k.x >= 0) v += ustore[k.x];
  if (k.y >= 0) v += ustore[k.y];
  return v;
}

// Forward, one workgroup per (front, boundary tile row): the front's
// right-hand side w_P (kept for the backward pass by tile row 0) and u = w_B -
// G w_P for the tile's rows.  Bound by the chain item, front, child map, update
// entry, then the tiles; a wave per tile with one accumulator per lane keeps
// its 64 rows in flight.  A solve of 9,006 unknowns takes 80 us in 15 launches
// (150 us with a workgroup's waves splitting the rows of each tile).
template <class T>
__global__ void __launch_bounds__(64 * kWaves) k_nd_forward(const int2* __restrict__ item,
                                                            const NdFrontDev* __restrict__ fr,
                                                            const int2* __restrict__ kid, const int* __restrict__ vmap,
                                                            const T* __restrict__ b, const double* __restrict__ tr,
                                                            double* __restrict__ w, double* ustore) {
  __shared__ __align__(16) double xs[kChunk];
  __shared__ double ys[kWaves][64];
  const int2 it = item[blockIdx.x];
  const NdFrontDev F = fr[it.x];
  const int rt = it.y, t = threadIdx.x, wv = t >> 6, lane = t & 63, P = F.tp * 64;
  const bool rows = rt < F.tb;
  const int r = rt * 64 + t;
  double wb = 0.0;
  if (rows && t < 64 && r < F.b) wb = front_rhs<T>(F, F.p + r, kid, vmap, b, ustore);
  const double* G = tr + (F.tr_off + (int64_t)F.tp * (F.tp - 1) / 2 + (int64_t)rt * F.tp) * 4096;
  double acc = 0.0;
  for (int c0 = 0; c0 < P; c0 += kChunk) {
    const int c1 = min(P, c0 + kChunk);
    __syncthreads();
    for (int f = c0 + t; f < c1; f += 64 * kWaves) {
      const double v = f < F.p ? front_rhs<T>(F, f, kid, vmap, b, ustore) : 0.0;
      xs[f - c0] = v;
      if (rt == 0) w[F.w_off + f] = v;
    }
    __syncthreads();
    if (!rows) continue;
    for (int J = (c0 >> 6) + wv; J < (c1 >> 6); J += kWaves)
      acc = tile_dot(G + (int64_t)J * 4096, xs + (J * 64 - c0), lane, acc);
  }
  if (!rows) return;
  const double s = tile_sum(acc, ys);
  if (t < 64 && r < F.b) ustore[F.u_off + r] = wb - s;
}

// Backward, one workgroup per (front, pivot tile I): x_I = -((-A11^-1) w_P +
// G^T x_B) over the tile rows of the front, to x and to the level vector.
template <class T>
__global__ void __launch_bounds__(64 * kWaves) k_nd_backward(const int2* __restrict__ item,
                                                             const NdFrontDev* __restrict__ fr,
                                                             const int* __restrict__ bidx, const int* __restrict__ vmap,
                                                             const double* __restrict__ tiles,
                                                             const double* __restrict__ tr,
                                                             const double* __restrict__ w, double* x,
                                                             T* __restrict__ u) {
  __shared__ __align__(16) double xs[kChunk];
  __shared__ double ys[kWaves][64];
  const int2 it = item[blockIdx.x];
  const NdFrontDev F = fr[it.x];
  const int I = it.y, t = threadIdx.x, wv = t >> 6, lane = t & 63, P = F.tp * 64, m = P + F.tb * 64;
  double acc = 0.0;
  for (int c0 = 0; c0 < m; c0 += kChunk) {
    const int c1 = min(m, c0 + kChunk);
    __syncthreads();
    for (int f = c0 + t; f < c1; f += 64 * kWaves)
      xs[f - c0] = f < P ? w[F.w_off + f] : (f - P < F.b ? x[bidx[F.bidx_off + (f - P)]] : 0.0);
    __syncthreads();
    for (int J = (c0 >> 6) + wv; J < (c1 >> 6); J += kWaves) {
      const double* A = J >= I ? tiles + (F.t_off + tile_at(J, I)) * 4096
                               : tr + (F.tr_off + (int64_t)I * (I - 1) / 2 + J) * 4096;
      acc = tile_dot(A, xs + (J * 64 - c0), lane, acc);
    }
  }
  const double s = tile_sum(acc, ys);
  const int f = I * 64 + t;
  if (t < 64 && f < F.p) {
    x[F.dof0 + f] = -s;
    u[vmap[F.dof0 + f]] = (T)-s;
  }
}

// u = b at the inactive nodes
template <class T>
__global__ void k_nd_rest(int n, const int* __restrict__ rest, const T* __restrict__ b, T* __restrict__ u) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) u[rest[i]] = b[rest[i]];
}

unsigned grid(int64_t n, int t = 256) { return (unsigned)((n + t - 1) / t); }

template <class V>
void upload_vec(DevMem& d, const std::vector<V>& h, hipStream_t st) {
  d.alloc(h.size() * sizeof(V));
  if (!h.empty()) NDCHK(hipMemcpyAsync(d.p, h.data(), h.size() * sizeof(V), hipMemcpyHostToDevice, st));
}

}  // namespace

DevMem::~DevMem() {
  if (p) (void)hipFree(p);
}
void DevMem::alloc(size_t n) {
  if (p) (void)hipFree(p);
  p = nullptr;
  bytes = n;
  if (n) NDCHK(hipMalloc(&p, n));
}

// ------------------------------------------------------------------ symbolic
NdBottom::NdBottom(int64_t nb, const int32_t* base, const int32_t* nbr, const uint8_t* flags, uint8_t active_bit) {
  // active nodes, their coordinates and 27 neighbours
  std::vector<int32_t> id_of(nb * 64, -1);
  std::vector<int32_t> slot;
  for (int64_t s = 0; s < nb * 64; ++s)
    if (flags[s] & active_bit) {
      id_of[s] = (int32_t)slot.size();
      slot.push_back((int32_t)s);
    }
  const int64_t n = (int64_t)slot.size();
  nnode_ = n;
  std::vector<int32_t> xyz(n * 3), adj(n * 27, -1);
  for (int64_t i = 0; i < n; ++i) {
    const int64_t blk = slot[i] >> 6;
    const int l = slot[i] & 63, li = l >> 4, lj = (l >> 2) & 3, lk = l & 3;
    xyz[i * 3 + 0] = base[blk * 3 + 0] + li;
    xyz[i * 3 + 1] = base[blk * 3 + 1] + lj;
    xyz[i * 3 + 2] = base[blk * 3 + 2] + lk;
    for (int s = 0; s < 27; ++s) {
      const int a = li + s / 9 - 1, b = lj + (s / 3) % 3 - 1, c = lk + s % 3 - 1;
      const int sx = a < 0 ? 0 : (a > 3 ? 2 : 1), sy = b < 0 ? 0 : (b > 3 ? 2 : 1), sz = c < 0 ? 0 : (c > 3 ? 2 : 1);
      const int sp = sx * 9 + sy * 3 + sz;
      const int64_t bb = sp == 13 ? blk : nbr[blk * 27 + sp];
      if (bb < 0) continue;
      adj[i * 27 + s] = id_of[bb * 64 + (((a & 3) << 4) | ((b & 3) << 2) | (c & 3))];
    }
  }
  // nested dissection: fronts in postorder, each front's pivots take the
  // next consecutive positions
  std::vector<int64_t> pos(n, -1);
  int64_t next = 0;
  std::vector<int32_t> work(n);
  std::iota(work.begin(), work.end(), 0);
  std::vector<int32_t> piv_nodes;  // all fronts' pivots, in position order
  // recursive helper (depth stays below ~64: each cut halves the box)
  std::function<int(int64_t, int64_t, int)> nd = [&](int64_t lo, int64_t hi, int depth) -> int {
    const int64_t cnt = hi - lo;
    std::vector<int> kids;
    int64_t slo = lo, shi = hi;  // the separator's range after the split
    if (cnt > kLeafNodes) {
      int32_t mn[3] = {INT32_MAX, INT32_MAX, INT32_MAX}, mx[3] = {INT32_MIN, INT32_MIN, INT32_MIN};
      for (int64_t k = lo; k < hi; ++k)
        for (int d = 0; d < 3; ++d) {
          mn[d] = std::min(mn[d], xyz[work[k] * 3 + d]);
          mx[d] = std::max(mx[d], xyz[work[k] * 3 + d]);
        }
      int ax = 0;
      for (int d = 1; d < 3; ++d)
        if (mx[d] - mn[d] > mx[ax] - mn[ax]) ax = d;
      if (mx[ax] > mn[ax]) {
        const int64_t mid = lo + cnt / 2;
        std::nth_element(work.begin() + lo, work.begin() + mid, work.begin() + hi,
                         [&](int32_t a, int32_t b) { return xyz[a * 3 + ax] < xyz[b * 3 + ax]; });
        const int32_t p = xyz[work[mid] * 3 + ax];
        // three-way partition: < p | > p | == p
        auto it1 = std::stable_partition(work.begin() + lo, work.begin() + hi,
                                         [&](int32_t a) { return xyz[a * 3 + ax] < p; });
        auto it2 = std::stable_partition(it1, work.begin() + hi, [&](int32_t a) { return xyz[a * 3 + ax] > p; });
        const int64_t a1 = it1 - work.begin(), a2 = it2 - work.begin();
        if (a1 > lo) kids.push_back(nd(lo, a1, depth + 1));
        if (a2 > a1) kids.push_back(nd(a1, a2, depth + 1));
        slo = a2;
        shi = hi;
      }
    }
    // this front: the separator (or the whole leaf box)
    std::sort(work.begin() + slo, work.begin() + shi, [&](int32_t a, int32_t b) {
      for (int d = 0; d < 3; ++d)
        if (xyz[a * 3 + d] != xyz[b * 3 + d]) return xyz[a * 3 + d] < xyz[b * 3 + d];
      return false;
    });
    Front F;
    F.pos0 = next;
    F.np = (int)(shi - slo);
    F.depth = depth;
    F.kids = kids;
    for (int64_t k = slo; k < shi; ++k) {
      pos[work[k]] = next++;
      piv_nodes.push_back(work[k]);
    }
    const int id = (int)fr_.size();
    for (int c : kids) fr_[c].parent = id;
    fr_.push_back(std::move(F));
    return id;
  };
  if (n > 0) nd(0, n, 0);
  // the nd() recursion hands out depths from the root; levels of the solve
  // are the depths
  maxdepth_ = 0;
  for (const Front& F : fr_) maxdepth_ = std::max(maxdepth_, F.depth);
  // boundary sets, postorder
  for (size_t t = 0; t < fr_.size(); ++t) {
    Front& F = fr_[t];
    const int64_t last = F.pos0 + F.np;
    std::vector<int64_t> B;
    for (int c : F.kids)
      for (int64_t q : fr_[c].bnd)
        if (q >= last) B.push_back(q);
    for (int64_t k = F.pos0; k < last; ++k) {
      const int32_t i = piv_nodes[k];
      for (int s = 0; s < 27; ++s) {
        const int32_t j = adj[i * 27 + s];
        if (j >= 0 && pos[j] >= last) B.push_back(pos[j]);
      }
    }
    std::sort(B.begin(), B.end());
    B.erase(std::unique(B.begin(), B.end()), B.end());
    F.bnd = std::move(B);
  }
  // var_of: slot -> first dof (3 * position)
  var_of_.assign(nb * 64, -1);
  for (int64_t i = 0; i < n; ++i) var_of_[slot[i]] = (int32_t)(3 * pos[i]);
  ndof_ = 3 * n;
  // local index of a position inside a front: pivots first, then boundary
  auto local = [&](const Front& F, int64_t q) -> int {
    if (q >= F.pos0 && q < F.pos0 + F.np) return (int)(q - F.pos0);
    const auto it = std::lower_bound(F.bnd.begin(), F.bnd.end(), q);
    if (it == F.bnd.end() || *it != q) return -1;
    return F.np + (int)(it - F.bnd.begin());
  };
  // device-side front table, work lists per depth, gather lists, maps
  std::vector<NdFrontDev> fd(fr_.size());
  int64_t toff = 0, wofs = 0, uofs = 0, bofs = 0, gofs = 0;
  std::vector<int32_t> ent_of;
  std::vector<int2> kid;
  std::vector<int32_t> bidx;
  int64_t trofs = 0;
  std::vector<int32_t> emap;
  for (size_t t = 0; t < fr_.size(); ++t) {
    Front& F = fr_[t];
    NdFrontDev& D = fd[t];
    D.p = 3 * F.np;
    D.b = 3 * (int)F.bnd.size();
    const int m = D.p + D.b;
    D.dof0 = 3 * F.pos0;
    D.tp = (D.p + 63) / 64;
    D.tb = (D.b + 63) / 64;
    D.parent = F.parent;
    D.t_off = toff;
    toff += tile_at(D.tp + D.tb, 0);
    D.w_off = wofs;
    wofs += D.tp * 64;
    D.u_off = uofs;
    uofs += D.b;
    D.bidx_off = bofs;
    for (int64_t q : F.bnd)
      for (int c = 0; c < 3; ++c) bidx.push_back((int32_t)(3 * q + c));
    bofs += D.b;
    D.k_off = gofs;
    D.tr_off = trofs;
    trofs += (int64_t)D.tp * (D.tp - 1) / 2 + (int64_t)D.tb * D.tp;
    // children's update entries mapped into this front, at most two per dof
    kid.resize(kid.size() + m, make_int2(-1, -1));
    int2* km = kid.data() + gofs;
    for (size_t o = 0; o < F.kids.size(); ++o) {
      const int c = F.kids[o];
      const Front& C = fr_[c];
      fd[c].emap_off = (int64_t)emap.size();
      for (size_t k = 0; k < C.bnd.size(); ++k) {
        const int lq = local(F, C.bnd[k]);
        if (lq < 0) throw std::runtime_error("nested dissection: a child's boundary node is missing from its parent");
        for (int cc = 0; cc < 3; ++cc) {
          emap.push_back(3 * lq + cc);
          (o == 0 ? km[3 * lq + cc].x : km[3 * lq + cc].y) = (int)(fd[c].u_off + 3 * (int64_t)k + cc);
        }
      }
    }
    gofs += m;
    // stencil entries: pivot i, spoke s, neighbour j later in the front
    for (int64_t k = F.pos0; k < F.pos0 + F.np; ++k) {
      const int32_t i = piv_nodes[k];
      const int li = (int)(k - F.pos0);
      for (int s = 0; s < 27; ++s) {
        const int32_t j = adj[i * 27 + s];
        if (j < 0) continue;
        const int lj = local(F, pos[j]);
        if (lj < 0 || lj < li) continue;  // eliminated earlier, or an earlier pivot's entry
        ent_.push_back(make_int4(slot[i], s, 3 * li, 3 * lj));
        ent_of.push_back((int32_t)t);
      }
    }
  }
  ntile_ = toff;
  wlen_ = wofs;
  ulen_ = uofs;
  ent_of_ = std::move(ent_of);
  fdev_ = std::move(fd);
  kid_ = std::move(kid);
  ntr_ = trofs;
  if (uofs > INT32_MAX || ndof_ > INT32_MAX)
    throw std::runtime_error("nested dissection: more than 2^31 - 1 solve entries");
  vmap_.resize(ndof_);
  for (int64_t s = 0; s < nb * 64; ++s)
    for (int c = 0; c < 3; ++c) {
      const int32_t k = (int32_t)((s >> 6) * 192 + c * 64 + (s & 63));
      if (var_of_[s] >= 0) vmap_[var_of_[s] + c] = k;
      else rest_.push_back(k);
    }
  bidx_ = std::move(bidx);
  emap_ = std::move(emap);
  // per depth: the solve's work items (front, boundary tile row; front, pivot
  // tile), the children to add (first and second ones) and the sweep batch
  depth_.resize(maxdepth_ + 1);
  int64_t maxpan = 0, maxid = 0;
  for (int d = 0; d <= maxdepth_; ++d) {
    Depth& D = depth_[d];
    D.fwd0 = (int64_t)items_.size();
    for (size_t t = 0; t < fr_.size(); ++t)
      if (fr_[t].depth == d)
        for (int r = 0; r < std::max(1, fdev_[t].tb); ++r) items_.push_back(make_int2((int)t, r));
    D.bwd0 = (int64_t)items_.size();
    for (size_t t = 0; t < fr_.size(); ++t)
      if (fr_[t].depth == d)
        for (int r = 0; r < fdev_[t].tp; ++r) items_.push_back(make_int2((int)t, r));
    D.end = (int64_t)items_.size();
    std::vector<SweepMat> mats;
    for (size_t t = 0; t < fr_.size(); ++t) {
      if (fr_[t].depth != d) continue;
      mats.push_back(SweepMat{fdev_[t].t_off, fdev_[t].tp, fdev_[t].tp + fdev_[t].tb, 0, (int32_t)t});
    }
    std::stable_sort(mats.begin(), mats.end(), [](const SweepMat& a, const SweepMat& b) { return a.np > b.np; });
    int64_t pan = 0;
    for (SweepMat& m : mats) {
      m.pan = (int32_t)pan;
      pan += m.nt;
    }
    maxpan = std::max(maxpan, pan);
    D.mat0 = (int64_t)mats_.size();
    mats_.insert(mats_.end(), mats.begin(), mats.end());
    D.batch.h = std::move(mats);
    for (int o = 0; o < 2; ++o) {
      D.kid0[o] = (int64_t)kids_.size();
      D.kid_tiles[o] = 0;
      for (size_t t = 0; t < fr_.size(); ++t) {
        if (fr_[t].depth != d || (int)fr_[t].kids.size() <= o) continue;
        const int c = fr_[t].kids[o];
        if (fdev_[c].b == 0) continue;
        kids_.push_back(c);
        D.kid_tiles[o] = std::max(D.kid_tiles[o], tile_at(fdev_[c].tb, 0));
      }
      D.nkid[o] = (int64_t)kids_.size() - D.kid0[o];
    }
  }
  maxid = (int64_t)fr_.size();
  npan_ = maxpan;
  nid_ = maxid;
}

void NdBottom::upload(hipStream_t st) {
  upload_vec(d_fr_, fdev_, st);
  upload_vec(d_kid_, kid_, st);
  upload_vec(d_vmap_, vmap_, st);
  upload_vec(d_rest_, rest_, st);
  upload_vec(d_bidx_, bidx_, st);
  upload_vec(d_emap_, emap_, st);
  upload_vec(d_ent_, ent_, st);
  upload_vec(d_items_, items_, st);
  upload_vec(d_ent_of_, ent_of_, st);
  upload_vec(d_mats_, mats_, st);
  upload_vec(d_kids_, kids_, st);
  const size_t tile = 4096 * 8;
  tiles_.alloc((size_t)std::max<int64_t>(ntile_, 1) * tile);
  tr_.alloc((size_t)std::max<int64_t>(ntr_, 1) * tile);
  pan_.alloc((size_t)std::max<int64_t>(npan_, 1) * tile);
  minv_.alloc((size_t)std::max<int64_t>(nid_, 1) * 2 * tile);
  info_.alloc((size_t)std::max<int64_t>(nid_, 1) * sizeof(int));
  for (Depth& D : depth_) {
    D.batch.d = static_cast<SweepMat*>(d_mats_.p) + D.mat0;
    D.batch.pan = static_cast<double*>(pan_.p);
    D.batch.minv = static_cast<double*>(minv_.p);
    D.batch.info = static_cast<int*>(info_.p);
  }
  w_.alloc((size_t)std::max<int64_t>(wlen_, 1) * 8);
  u_.alloc((size_t)std::max<int64_t>(ulen_, 1) * 8);
  x_.alloc((size_t)std::max<int64_t>(ndof_, 1) * 8);
  NDCHK(hipStreamSynchronize(st));
}

size_t NdBottom::device_bytes() const {
  size_t s = 0;
  for (const DevMem* d : {&d_fr_, &d_kid_, &d_vmap_, &d_rest_, &d_bidx_, &d_emap_, &d_ent_, &d_ent_of_, &d_items_,
                          &d_mats_, &d_kids_, &tiles_, &tr_, &pan_, &minv_, &info_, &w_, &u_, &x_})
    s += d->bytes;
  return s;
}

// ------------------------------------------------------------------ numeric
void NdBottom::factor(const double* ST, hipStream_t st) {
  if (fr_.empty()) return;
  const NdFrontDev* fr = static_cast<const NdFrontDev*>(d_fr_.p);
  double* tiles = static_cast<double*>(tiles_.p);
  NDCHK(hipMemsetAsync(tiles_.p, 0, tiles_.bytes, st));
  NDCHK(hipMemsetAsync(info_.p, 0, info_.bytes, st));
  k_nd_pad<<<(unsigned)fr_.size(), 64, 0, st>>>(fr, tiles);
  const int64_t n = (int64_t)ent_.size();
  if (n > 0)
    k_nd_assemble<<<grid(n * 9), 256, 0, st>>>(n, static_cast<const int4*>(d_ent_.p),
                                               static_cast<const int*>(d_ent_of_.p), fr, ST, tiles);
  for (int d = maxdepth_; d >= 0; --d) {
    const Depth& D = depth_[d];
    for (int o = 0; o < 2; ++o)
      for (int64_t k = 0; k < D.nkid[o]; k += 32768)
        k_nd_extend_add<<<dim3((unsigned)D.kid_tiles[o], (unsigned)std::min<int64_t>(32768, D.nkid[o] - k)), 256, 0,
                          st>>>(static_cast<const int*>(d_kids_.p) + D.kid0[o] + k, fr,
                                static_cast<const int*>(d_emap_.p), tiles);
    sweep_run(st, D.batch, tiles);
  }
  int64_t most = 0;
  for (const NdFrontDev& D : fdev_)
    most = std::max(most, (int64_t)D.tp * (D.tp - 1) / 2 + (int64_t)D.tb * D.tp);
  if (most > 0)
    for (size_t f = 0; f < fr_.size(); f += 32768)
      k_nd_transpose<<<dim3((unsigned)most, (unsigned)std::min<size_t>(32768, fr_.size() - f)), 256, 0, st>>>(
          fr + f, tiles, static_cast<double*>(tr_.p));
  std::vector<int> h(fr_.size());
  NDCHK(hipMemcpyAsync(h.data(), info_.p, h.size() * sizeof(int), hipMemcpyDeviceToHost, st));
  NDCHK(hipStreamSynchronize(st));
  for (size_t t = 0; t < fr_.size(); ++t)
    if (h[t] != 0)
      throw NdNotSpd("bottom Cholesky failed: front " + std::to_string(t) + " (" + std::to_string(fdev_[t].p) +
                     " pivots) is not positive definite at its pivot " + std::to_string(h[t]));
}

// ------------------------------------------------------------------ solve
template <class T>
void NdBottom::solve(const T* b, T* u, hipStream_t st) {
  const NdFrontDev* fr = static_cast<const NdFrontDev*>(d_fr_.p);
  const int2* items = static_cast<const int2*>(d_items_.p);
  const int* vmap = static_cast<const int*>(d_vmap_.p);
  const double* tiles = static_cast<const double*>(tiles_.p);
  const double* tr = static_cast<const double*>(tr_.p);
  double* w = static_cast<double*>(w_.p);
  double* us = static_cast<double*>(u_.p);
  double* x = static_cast<double*>(x_.p);
  for (int d = (int)depth_.size() - 1; d >= 0; --d) {
    const Depth& D = depth_[d];
    if (D.bwd0 > D.fwd0)
      k_nd_forward<T><<<(unsigned)(D.bwd0 - D.fwd0), 64 * kWaves, 0, st>>>(
          items + D.fwd0, fr, static_cast<const int2*>(d_kid_.p), vmap, b, tr, w, us);
  }
  for (const Depth& D : depth_)
    if (D.end > D.bwd0)
      k_nd_backward<T><<<(unsigned)(D.end - D.bwd0), 64 * kWaves, 0, st>>>(
          items + D.bwd0, fr, static_cast<const int*>(d_bidx_.p), vmap, tiles, tr, w, x, u);
  const int n = (int)rest_.size();
  if (n > 0) k_nd_rest<T><<<grid(n), 256, 0, st>>>(n, static_cast<const int*>(d_rest_.p), b, u);
}

template void NdBottom::solve<float>(const float*, float*, hipStream_t);
template void NdBottom::solve<double>(const double*, double*, hipStream_t);

NdStats NdBottom::stats() const {
  NdStats s;
  s.fronts = (int64_t)fr_.size();
  s.depth = maxdepth_ + 1;
  s.factor_entries = (ntile_ + ntr_) * 4096;
  for (const NdFrontDev& D : fdev_) s.max_front = std::max<int64_t>(s.max_front, D.p + D.b);
  return s;
}

}  // namespace spg
