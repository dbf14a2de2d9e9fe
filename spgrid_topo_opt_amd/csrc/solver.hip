// solver.hip -- see solver.hpp.
#include <hip/hip_runtime.h>
#include <rocblas/rocblas.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <limits>
#include <mutex>

#include "solver.hpp"

namespace spg {

#define HIPCHK(x)                                                                                   \
  do {                                                                                              \
    hipError_t e_ = (x);                                                                            \
    if (e_ != hipSuccess) throw SpgError(SPG_E_HIP, std::string(#x) + ": " + hipGetErrorString(e_)); \
  } while (0)
#define RBCHK(x)                                                                                           \
  do {                                                                                                     \
    rocblas_status s_ = (x);                                                                               \
    if (s_ != rocblas_status_success)                                                                      \
      throw SpgError(SPG_E_HIP, std::string(#x) + ": rocblas status " + std::to_string((int)s_));          \
  } while (0)

static double now_s() {
  return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count();
}

// Boundary phases over at most this many nodes run as one dense map (2 maps x
// 3n x 3n entries in FP64 and FP32).  Level-0 phase by map / by data flow, FP32
// and FP64, and what both maps add to a density update:
//   405 nodes    7.1 / 36 us    8.2 / 41 us   0.36 ms
//   1425         9.8 / 38       16 / 43       1.2
//   2400         17 / 39        29 / 44       2.6
//   3000         23 / 38        41 / 43       6.0
// At four phases a V-cycle the maps are earned back after 3, 11, 30 and 99
// FP32 V-cycles, and 3, 11, 43 and over 500 FP64 ones.  The line is drawn for
// solves on kept operators and for FP32.  One FP64 solve of 25 V-cycles after
// each update earns them back up to about 1,900 nodes and loses about 1 ms of
// 10 at 2,400: there the data flow would be the faster way.
static constexpr int kMaxDenseBoundary = 2560;
// levels of at most this many blocks get the entries of the data-flow sweep
// (FlowBlocks in kernels.hip has each kernel's own limit)
static constexpr int kMaxFlowSweep = 4096;
// pcg() result: a data-flow kernel reported a wait that timed out; the pass is
// repeated with per-colour launches
static constexpr int kFlowRetry = -100;
// byte offset of the PCG report in the pinned scalar buffer
static constexpr int kReportOffset = 128;
// relative residual reduction one FP32 MG-PCG pass is asked for at most
static constexpr double kFp32PassReduction = 1e-6;
// bottom solve: the dense FP64 inverse up to this many unknowns (one
// bandwidth-bound GEMV per V-cycle), the nested-dissection Cholesky
// (bottom_nd.hip) above it, unless spg_config.bottom_dense_max sets another
// limit; SPG_BOTTOM=dense|nd overrides both (dense stays limited to
// kMaxDenseBottomDofs: its inverse is O(n^2)).A whole density update takes 3.8
// / 4.4 / 46 ms with the dense inverse and 3.0 / 1.8 / 3.3 ms with the nested
// dissection at 2.0 K / 4.1 K / 11.6 K unknowns (other levels' work included);
// the bottom solve of an FP32 V-cycle 6.5 / 15 / 76 us against 33 / 49 / 101 us:
// the dense inverse pays when many solves share a factorization.
static constexpr int64_t kDenseBottomDofs = 16384;
static constexpr int64_t kMaxDenseBottomDofs = 60000;

DBuf::~DBuf() {
  if (p) (void)hipFree(p);
}
void DBuf::alloc(size_t n) {
  if (p) {
    (void)hipFree(p);
    p = nullptr;
  }
  bytes = n;
  if (n) HIPCHK(hipMalloc(&p, n));
}

template <class V>
static void upload(DBuf& b, const V& v) {
  using T = typename V::value_type;
  b.alloc(v.size() * sizeof(T));
  if (!v.empty()) HIPCHK(hipMemcpy(b.p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
}

// the size rule of the colour-major copy of b (Solver::colour_major_b): u,
// b, E and the neighbour table of level 0 in FP32 above 256 MiB
static bool colour_major_by_size(int64_t nb) {
  return nb * (int64_t)(2 * 192 * 4 + 64 * 4 + 27 * 4 + 64) > ((int64_t)256 << 20);
}

template <> float* LevelRT::u<float>() const { return u32.as<float>(); }
template <> double* LevelRT::u<double>() const { return u64.as<double>(); }
template <> float* LevelRT::b<float>() const { return b32.as<float>(); }
template <> double* LevelRT::b<double>() const { return b64.as<double>(); }
template <> float* LevelRT::r<float>() const { return r32.as<float>(); }
template <> double* LevelRT::r<double>() const { return r64.as<double>(); }
template <> const float* LevelRT::st<float>() const { return st32.as<float>(); }
template <> const double* LevelRT::st<double>() const { return st64.as<double>(); }
template <> const float* Solver::E<float>() const { return E32_.as<float>(); }
template <> const double* Solver::E<double>() const { return E64_.as<double>(); }

Solver::Solver(const spg_config& cfg, const ProblemDesc& pd) : cfg_(cfg) {
  const double t0 = now_s();
  if (const char* e = std::getenv("SPG_BOTTOM_FP64")) bottom64_ = std::atoi(e) != 0;
  if (const char* e = std::getenv("SPG_COARSE_FP64")) coarse64_ = std::atoi(e) != 0;
  // flags, hierarchy and the index-range check on the host, before any
  // device call or allocation
  lay_ = build_layout(pd);
  const double t_layout = now_s();
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) throw SpgError(SPG_E_HIP, "no HIP device available");
  if (cfg.device < 0 || cfg.device >= ndev) throw SpgError(SPG_E_INVALID, "device ordinal out of range");
  HIPCHK(hipSetDevice(cfg.device));
  size_t free0 = 0, total0 = 0;
  HIPCHK(hipMemGetInfo(&free0, &total0));
  HIPCHK(hipStreamCreateWithFlags(&st_, hipStreamNonBlocking));
  HIPCHK(hipStreamCreateWithFlags(&st2_, hipStreamNonBlocking));
  HIPCHK(hipEventCreateWithFlags(&ev_a_, hipEventDisableTiming));
  HIPCHK(hipEventCreateWithFlags(&ev_b_, hipEventDisableTiming));
  if (const char* e = std::getenv("SPG_OVERLAP")) overlap_ = std::atoi(e) != 0;
  if (const char* e = std::getenv("SPG_GS_CMB")) cmb_mode_ = std::atoi(e) != 0 ? 1 : 0;
  RBCHK(rocblas_create_handle(&rb_));
  RBCHK(rocblas_set_stream(rb_, st_));
  double kmu[576], kla[576];
  element_tables(kmu, kla);
  for (int e = 0; e < 576; ++e) K0_[e] = cfg.mu * kmu[e] + cfg.lambda * kla[e];
  activate();
  const double t_init = now_s();
  upload_layout();
  sync();
  const double t_upload = now_s();
  build_operators();
  setup_colour_major();
  sync();
  size_t free1 = 0;
  HIPCHK(hipMemGetInfo(&free1, &total0));
  dev_bytes_ = (double)free0 - (double)free1;
  setup_s_ = now_s() - t0;
  if (const char* e = std::getenv("SPG_SETUP_TRACE"); e && std::atoi(e) > 0)
    std::fprintf(stderr, "[spg] setup %.3f s: host layout %.3f, device init %.3f, upload %.3f, operators %.3f\n",
                 setup_s_, t_layout - t0, t_init - t_layout, t_upload - t_init, now_s() - t_upload);
}

Solver::~Solver() {
  if (rb_) rocblas_destroy_handle(rb_);
  if (hscal_) (void)hipHostFree(hscal_);
  if (stage_) (void)hipHostFree(stage_);
  if (ev_a_) (void)hipEventDestroy(ev_a_);
  if (ev_b_) (void)hipEventDestroy(ev_b_);
  if (st2_) (void)hipStreamDestroy(st2_);
  if (st_) (void)hipStreamDestroy(st_);
}

void Solver::sync() { HIPCHK(hipStreamSynchronize(st_)); }

// The element constants live in device constant memory, one set per device,
// shared by every solver on it.  The last material uploaded is recorded per
// device; a solver whose material differs waits for the device (work of the
// other solver may still read the constants) and uploads its own.  Calls
// into solvers of different materials on one device from several threads
// at once are not supported.
void Solver::activate() {
  struct Key {
    bool set = false;
    double mu = 0, lambda = 0;
  };
  static std::mutex mu;
  static std::vector<Key> keys;
  std::lock_guard<std::mutex> lock(mu);
  if ((int)keys.size() <= cfg_.device) keys.resize(cfg_.device + 1);
  Key& k = keys[cfg_.device];
  if (k.set && k.mu == cfg_.mu && k.lambda == cfg_.lambda) return;
  int prev = 0;
  HIPCHK(hipGetDevice(&prev));
  HIPCHK(hipSetDevice(cfg_.device));
  HIPCHK(hipDeviceSynchronize());
  const hipError_t e = upload_k0(K0_);
  HIPCHK(hipSetDevice(prev));
  if (e != hipSuccess) throw SpgError(SPG_E_HIP, std::string("element constants: ") + hipGetErrorString(e));
  k.set = true;
  k.mu = cfg_.mu;
  k.lambda = cfg_.lambda;
}

// names of the FlowWho bits
static std::string flow_names(unsigned who) {
  static const std::pair<unsigned, const char*> kNames[] = {{kFlowBnd0, "level-0 boundary phase"},
                                                            {kFlowBndSt, "boundary phase of an explicit level"},
                                                            {kFlowGs0, "level-0 sweep"},
                                                            {kFlowSt, "sweep of an explicit level"}};
  std::string s;
  for (const auto& [bit, name] : kNames)
    if (who & bit) s += (s.empty() ? "" : ", ") + std::string(name);
  return s;
}

void Solver::check_flow() {
  if (lv_.empty() || !lv_[0].coop.p) return;
  unsigned w[2] = {0, 0};
  HIPCHK(hipMemcpyAsync(w, lv_[0].coop.p, sizeof(w), hipMemcpyDeviceToHost, st_));
  HIPCHK(hipStreamSynchronize(st_));
  if (w[1]) {
    // reported once: the next kernel starts from a clear word
    HIPCHK(hipMemsetAsync(static_cast<unsigned*>(lv_[0].coop.p) + 1, 0, sizeof(unsigned), st_));
    HIPCHK(hipStreamSynchronize(st_));
    throw SpgError(SPG_E_HIP, flow_names(w[1]) +
                                  ": a wait timed out (workgroups not resident together; SPG_COOP_LAUNCH=1 uses the "
                                  "cooperative launch API, SPG_DATA_FLOW=0 per-colour launches on every level)");
  }
}

// waves of data-flow kernels that the solvers of this process have on each device
static FlowBudget& flow_budget() {
  static FlowBudget* b = new FlowBudget();  // outlives every solver
  return *b;
}

void Solver::set_flow(FlowUse use) {
  for (LevelRT& R : lv_) R.d.flow = use;
}

// All data-flow kernels if their waves fit beside those that other solvers have
// on the device; else boundary phases by few waves; else none.  A cooperative
// launch makes its own room.  SPG_DATA_FLOW=0: none.
Solver::FlowLease::FlowLease(Solver& s, int precision, bool any) : s_(s) {
  const char* sw = std::getenv("SPG_DATA_FLOW");
  const char* coop = std::getenv("SPG_COOP_LAUNCH");
  FlowUse use = kFlowNone;
  if (s.flow_dead_ || (sw && std::atoi(sw) == 0)) {
  } else if (coop && std::atoi(coop) == 1) {
    use = kFlowAll;
  } else {
    int cus = 0;
    HIPCHK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, s.cfg_.device));
    for (const FlowUse u : {kFlowAll, kFlowFew}) {
      need_ = FlowNeed();
      for (size_t l = 0; l < s.lv_.size(); ++l) {
        if (precision != 1) add_flow_need(need_, s.lv_[l].d, l == 0, false, u, any);
        if (precision == 1 || s.coarse64_) add_flow_need(need_, s.lv_[l].d, l == 0, true, u, any);
      }
      held_ = need_.cus == 0.0 || flow_budget().take(s.cfg_.device, cus, need_);
      if (!held_) continue;
      held_ = need_.cus > 0.0;
      use = u;
      break;
    }
  }
  s_.set_flow(use);
}

Solver::FlowLease::~FlowLease() {
  s_.set_flow(kFlowNone);
  if (held_) flow_budget().give(s_.cfg_.device, need_);
}

void Solver::upload_layout() {
  const int L = lay_.nlev;
  lv_.clear();
  lv_.resize(L);
  for (int l = 0; l < L; ++l) {
    const LevelDesc& D = lay_.lv[l];
    LevelRT& R = lv_[l];
    R.d.nb = (int)D.nb;
    R.d.cell = cell_consts(cfg_.mu, cfg_.lambda);
    R.n3 = D.nb * 192;
    upload(R.nbr, D.nbr);
    upload(R.flags, D.flags);
    upload(R.base, D.base);
    if (!D.restrict_src.empty()) upload(R.rsrc, D.restrict_src);
    if (!D.prolong_src.empty()) upload(R.psrc, D.prolong_src);
    std::vector<int32_t> bnd;
    R.d.bnd_max = 0;
    for (int c = 0; c < 8; ++c) {
      R.d.bnd_off[c] = (int)bnd.size();
      bnd.insert(bnd.end(), D.bnd_list[c].begin(), D.bnd_list[c].end());
      R.d.bnd_max = std::max(R.d.bnd_max, (int)D.bnd_list[c].size());
    }
    R.d.bnd_off[8] = (int)bnd.size();
    if (!bnd.empty()) upload(R.bnd, bnd);
    R.d.bnd = R.bnd.as<int>();
    if (!bnd.empty()) {
      upload(R.bci, D.bnd_ci);
      upload(R.bslot, D.bnd_slot);
      R.bA64.alloc(bnd.size() * 288 * 8);
      R.bA32.alloc(bnd.size() * 288 * 4);
      R.bt64.alloc(bnd.size() * 4 * 8);
      R.bt32.alloc(bnd.size() * 4 * 4);
      if (l == 0) {
        R.coop.alloc(2 * sizeof(unsigned));
        HIPCHK(hipMemset(R.coop.p, 0, 2 * sizeof(unsigned)));
      }
      if (l == 0 || bnd.size() > (size_t)kMaxDenseBoundary) {
        R.btag.alloc(bnd.size() * 6 * 8);
        R.d.btag = R.btag.p;
        R.d.coop = lv_[0].coop.as<unsigned>();  // one error word for every level
      }
    }
    if (l == 0 && !bnd.empty()) {
      // the blocks that hold boundary nodes
      std::vector<int32_t> id((size_t)D.nb, -1), blk;
      for (const int32_t s : bnd) id[(size_t)(s >> 6)] = 0;
      for (int64_t i = 0; i < D.nb; ++i)
        if (id[(size_t)i] == 0) {
          id[(size_t)i] = (int32_t)blk.size();
          blk.push_back((int32_t)i);
        }
      if (blk.size() <= (size_t)kMaxFlowSweep) {
        std::vector<unsigned long long> own(blk.size(), 0), mask(blk.size() * 27, 0);
        for (const int32_t s : bnd) own[(size_t)id[(size_t)(s >> 6)]] |= 1ull << (s & 63);
        std::vector<int32_t> nb27(blk.size() * 27), id27(blk.size() * 27, -1);
        for (size_t i = 0; i < blk.size(); ++i)
          for (int k = 0; k < 27; ++k) {
            const int32_t q = k == 13 ? blk[i] : D.nbr[(size_t)blk[i] * 27 + k];
            nb27[i * 27 + k] = q;
            if (q < 0 || id[(size_t)q] < 0) continue;
            id27[i * 27 + k] = id[(size_t)q];
            mask[i * 27 + k] = own[(size_t)id[(size_t)q]];
          }
        upload(R.fb_blk, blk);
        upload(R.fb_nbr, nb27);
        upload(R.fb_id, id27);
        upload(R.fb_mask, mask);
        R.fb_tag.alloc(blk.size() * 64 * 6 * 8);
        HIPCHK(hipMemset(R.fb_tag.p, 0, R.fb_tag.bytes));
        R.d.fb_n = (int)blk.size();
        R.d.fb_blk = R.fb_blk.as<int>();
        R.d.fb_nbr = R.fb_nbr.as<int>();
        R.d.fb_id = R.fb_id.as<int>();
        R.d.fb_mask = R.fb_mask.as<unsigned long long>();
        R.d.fb_tag = R.fb_tag.p;
        R.d.fb_last = &R.fb_last;
      }
    }
    if (!D.bnd_cslot.empty()) {
      upload(R.b0cslot, D.bnd_cslot);
      upload(R.b0node, D.bnd_cnode);
      R.b0E64.alloc(D.bnd_cslot.size() * 8);
      R.b0E32.alloc(D.bnd_cslot.size() * 4);
      R.b0D64.alloc(bnd.size() * 8 * 8);
      R.b0D32.alloc(bnd.size() * 8 * 4);
      R.d.b0node = R.b0node.as<int16_t>();
      R.d.b0E64 = R.b0E64.as<double>();
      R.d.b0E32 = R.b0E32.as<float>();
      R.d.b0D64 = R.b0D64.as<double>();
      R.d.b0D32 = R.b0D32.as<float>();
    }
    R.d.bci = R.bci.as<int>();
    R.d.bslot = R.bslot.as<int>();
    R.d.bA64 = R.bA64.as<double>();
    R.d.bA32 = R.bA32.as<float>();
    R.d.bt64 = R.bt64.as<double>();
    R.d.bt32 = R.bt32.as<float>();
    R.d.nbr = R.nbr.as<int>();
    if (l == 0 && !bnd.empty()) {
      R.bnslot.alloc(bnd.size() * 27 * 4);
      launch_bnd_nslot(st_, R.d, R.bnslot.as<int>());
      R.d.bnslot = R.bnslot.as<int>();
    }
    if (l == 0 && !bnd.empty() && !D.gs_dist.empty()) {
      // near-band step lists of both sweep directions, and their neighbour slots
      std::vector<int32_t> all;
      for (int i = 0; i < 16; ++i) {
        const std::vector<int32_t>& L = D.gs_near[i / 8][i % 8];
        R.gsnear_off[i] = (int64_t)all.size();
        if (!L.empty()) {
          // the layout's step colours must be the sweep's
          const int32_t s0 = L[0] & 63;
          const int colour = (((s0 >> 4) & 1) << 2) | (((s0 >> 2) & 1) << 1) | (s0 & 1);
          if (colour != sweep_colour(true, i < 8, i % 8))
            throw SpgError(SPG_E_INVALID, "near-band step list in the wrong colour order");
        }
        all.insert(all.end(), L.begin(), L.end());
      }
      R.gsnear_off[16] = (int64_t)all.size();
      upload(R.gsdist, D.gs_dist);
      upload(R.gsnear, all);
      R.gsnslot.alloc(std::max<size_t>(all.size(), 1) * 27 * 4);
      launch_list_nslot(st_, R.d, (int)all.size(), R.gsnear.as<int>(), R.gsnslot.as<int>());
    }
    // SPG_GS_CMB compares the per-colour launches' reads of b: it keeps them
    if (D.nb <= kMaxFlowSweep && (l > 0 ? D.is_explicit : cmb_mode_ < 0) && lv_[0].coop.p) {
      R.stag.alloc((size_t)D.nb * 64 * 6 * 8);
      HIPCHK(hipMemset(R.stag.p, 0, R.stag.bytes));
      R.d.stag = R.stag.p;
      R.d.epoch = &R.epoch;
      R.d.coop = lv_[0].coop.as<unsigned>();
    }
    R.d.flags = R.flags.as<uint8_t>();
    R.d.base = R.base.as<int>();
    R.d.rsrc = R.rsrc.as<int>();
    R.d.psrc = R.psrc.as<int>();
    if (R.psrc.p) {
      R.psrc27.alloc((size_t)D.nb * 27 * 4);
      launch_prolong_table(st_, R.d, R.psrc27.as<int>());
      R.d.psrc27 = R.psrc27.as<int>();
    }
    R.u32.alloc(R.n3 * 4);
    R.b32.alloc(R.n3 * 4);
    R.r32.alloc(R.n3 * 4);
    R.u64.alloc(R.n3 * 8);
    R.b64.alloc(R.n3 * 8);
    R.r64.alloc(R.n3 * 8);
  }
  // level-0 cell data
  upload(E64_, lay_.E);
  E32_.alloc(lay_.E.size() * 4);  // rounded on the device (round to nearest, as a host cast)
  launch_cast_d2f(st_, E64_.as<double>(), E32_.as<float>(), (int64_t)lay_.E.size());
  upload(rho_, lay_.rho);
  upload(in_slot_, lay_.in_node_slot);
  upload(ud_idx_, lay_.ud_slot);
  upload(ud_val_, lay_.ud_value);
  n_ud_ = (int64_t)lay_.ud_slot.size();
  const int64_t n3 = lv_[0].n3;
  for (DBuf* b : {&x32_, &rr32_, &s32_, &q32_, &z32_}) b->alloc(n3 * 4);
  for (DBuf* b : {&x64_, &rr64_, &s64_, &q64_, &z64_, &u_, &f_, &res_, &tmp_}) b->alloc(n3 * 8);
  scal_.alloc(sizeof(CgScalars) + reduce_partials(0) * sizeof(double));
  part_.alloc((reduce_partials(0) + 16) * sizeof(double));
  apart_.alloc(apply_dot_partials(lv_[0].d.nb) * sizeof(double));
  HIPCHK(hipHostMalloc((void**)&hscal_, 256, hipHostMallocCoherent));
  std::memset(hscal_, 0, 256);
}

// Galerkin position matrices of one depth for this solver's K0, on its
// device: built and uploaded once per process and kept until it ends (the
// deepest usual one, depth 5, is 576 x 8^5 doubles = 151 MB), so solvers
// rebuilt for new block sets or densities with the same material reuse them
const double* Solver::posmat_device(int depth) {
  struct Entry {
    int dev, depth;
    std::vector<double> k0;
    double* ptr;
  };
  static std::mutex mu;
  static std::vector<Entry>* cache = new std::vector<Entry>();  // never freed: device memory held to the end
  const std::vector<double> k0(K0_, K0_ + 576);
  std::lock_guard<std::mutex> lock(mu);
  for (const Entry& e : *cache)
    if (e.dev == cfg_.device && e.depth == depth && e.k0 == k0) return e.ptr;
  const std::vector<double> M = galerkin_position_matrices(depth, K0_);
  double* p = nullptr;
  HIPCHK(hipMalloc((void**)&p, M.size() * sizeof(double)));
  HIPCHK(hipMemcpy(p, M.data(), M.size() * sizeof(double), hipMemcpyHostToDevice));
  cache->push_back(Entry{cfg_.device, depth, k0, p});
  return p;
}

void Solver::build_operators() {
  const int L = lay_.nlev;
  if (!lay_.use_mg) return;
  const char* tr = std::getenv("SPG_SETUP_TRACE");
  const bool trace = tr && std::atoi(tr) >= 2;
  double tm = now_s();
  auto mark = [&](const char* what) {
    if (!trace) return;
    sync();
    const double t = now_s();
    std::fprintf(stderr, "[spg] operators %-22s %.3f s\n", what, t - tm);
    tm = t;
  };
  const double one = 1.0, zero = 0.0;
  for (int l = 0; l < L; ++l) {
    const LevelDesc& D = lay_.lv[l];
    if (!D.is_explicit) continue;
    LevelRT& R = lv_[l];
    const int depth = (L == 1) ? 0 : l;
    const int64_t npos = (int64_t)1 << (3 * depth);
    upload(R.cell_row, D.cell_row);
    if (!D.cell_fine_blocks.empty()) upload(R.cfb, D.cell_fine_blocks);
    upload(R.cgi, D.cell_gpu_index);
    const double* dM = posmat_device(depth);
    DBuf G, Cm;
    const int64_t ncell = D.ncell;
    R.st64.alloc((size_t)D.nb * 243 * 64 * 8);
    R.st32.alloc((size_t)D.nb * 243 * 64 * 4);
    if (ncell > 0) {
      G.alloc((size_t)(ncell * npos) * 8);
      Cm.alloc((size_t)ncell * 576 * 8);
      launch_galerkin_gather(st_, ncell, depth, R.cfb.as<int>(), R.cgi.as<int>(), E64_.as<double>(), G.as<double>());
      // Cm^T (576 x ncell) = M^T (576 x npos) * G^T (npos x ncell), column-major views
      RBCHK(rocblas_dgemm(rb_, rocblas_operation_none, rocblas_operation_none, 576, (rocblas_int)ncell,
                          (rocblas_int)npos, &one, dM, 576, G.as<double>(), (rocblas_int)npos, &zero,
                          Cm.as<double>(), 576));
    }
    mark("  gather + product");
    launch_galerkin_assemble(st_, R.d, R.cell_row.as<int>(), Cm.as<double>(), cfg_.dx, R.st64.as<double>());
    launch_stencil_to_float(st_, R.st64.as<double>(), R.st32.as<float>(), (int64_t)D.nb * 243 * 64);
    sync();
    mark("  assemble");
  }
  mark("Galerkin levels");
  build_boundary_rows();
  mark("boundary rows");
  // bottom: FP64 inverse or factorization of the Dirichlet-deleted stencil matrix
  // (Multigrid_Hierarchy.h:332-341; Elasticity_Matrix.cpp:15-233 factorizes with PARDISO)
  const int B = L - 1;
  const LevelDesc& D = lay_.lv[B];
  std::vector<int32_t> var(D.nb * 64, -1);
  int64_t nv = 0;
  for (int64_t s = 0; s < D.nb * 64; ++s)
    if (D.flags[s] & D_ACTIVE) {
      var[s] = (int32_t)nv;
      nv += 3;
    }
  nvar_ = nv;
  if (trace) std::fprintf(stderr, "[spg] operators bottom unknowns        %lld\n", (long long)nv);
  const char* bsel = std::getenv("SPG_BOTTOM");
  const int64_t dense_max =
      std::min(cfg_.bottom_dense_max > 0 ? (int64_t)cfg_.bottom_dense_max : kDenseBottomDofs, kMaxDenseBottomDofs);
  const bool want_nd = bsel ? std::string(bsel) == "nd" : nv > dense_max;
  if (!want_nd && nv > kMaxDenseBottomDofs)
    throw SpgError(SPG_E_INVALID, "bottom level has " + std::to_string(nv) + " unknowns, more than the dense "
                                      "inverse takes (" + std::to_string(kMaxDenseBottomDofs) + "); SPG_BOTTOM=dense "
                                      "asked for it");
  if (want_nd) {
    // nested-dissection Cholesky: symbolic once per topology, numeric for
    // every new set of stencils
    try {
      if (!nd_) {
        nd_ = std::make_unique<NdBottom>(D.nb, D.base.data(), D.nbr.data(), D.flags.data(), D_ACTIVE);
        nd_->upload(st_);
      }
      nd_->factor(lv_[B].st64.as<double>(), st_);
      mark("bottom (nested dissection)");
    } catch (const NdNotSpd& e) {
      throw SpgError(SPG_E_SINGULAR, e.what());
    } catch (const SpgError&) {
      throw;
    } catch (const std::exception& e) {
      throw SpgError(SPG_E_HIP, std::string("nested-dissection bottom: ") + e.what());
    }
    build_boundary_maps();
    mark("boundary maps");
    return;
  }
  nd_.reset();
  // the matrix in packed lower-triangle 64x64 tiles (padding rows are
  // identity), its inverse by the block sweep in place, and the FP32 copy for
  // the FP32 cycle
  nT_ = (int)((nv + 63) / 64);
  const size_t ntile = (size_t)nT_ * (nT_ + 1) / 2;
  const size_t npad = (size_t)nT_ * 64;
  if (!tiles64_.p) {
    upload(var_of_, var);
    tiles64_.alloc(ntile * 4096 * 8);
    tiles32_.alloc(ntile * 4096 * 4);
    pan_.alloc((size_t)nT_ * 4096 * 8);
    minv_.alloc(2 * 4096 * 8);
    info_.alloc(sizeof(int));
    const std::vector<SweepMat> one_mat{SweepMat{0, nT_, nT_, 0, 0}};
    upload(smat_, one_mat);
    sweep_.h = one_mat;
    sweep_.d = smat_.as<SweepMat>();
    sweep_.pan = pan_.as<double>();
    sweep_.minv = minv_.as<double>();
    sweep_.info = info_.as<int>();
    std::vector<int32_t> vslot(npad, -1);
    for (size_t i = 0; i < var.size(); ++i)
      if (var[i] >= 0)
        for (int c = 0; c < 3; ++c) vslot[(size_t)var[i] + c] = (int32_t)((i >> 6) * 192 + c * 64 + (i & 63));
    upload(vslot_, vslot);
    pb64_.alloc((size_t)bottom_splits(nT_) * npad * 8);
    pb32_.alloc((size_t)bottom_splits(nT_) * npad * 4);
  }
  HIPCHK(hipMemsetAsync(tiles64_.p, 0, tiles64_.bytes, st_));
  HIPCHK(hipMemsetAsync(info_.p, 0, sizeof(int), st_));
  launch_tile_assemble(st_, lv_[B].d, lv_[B].st64.as<double>(), var_of_.as<int>(), nv, nT_, tiles64_.as<double>());
  sweep_run(st_, sweep_, tiles64_.as<double>());
  launch_tile_negate(st_, tiles64_.as<double>(), tiles32_.as<float>(), (int64_t)ntile * 4096);
  int hinfo = 0;
  HIPCHK(hipMemcpyAsync(&hinfo, info_.p, sizeof(int), hipMemcpyDeviceToHost, st_));
  sync();
  if (hinfo != 0)
    throw SpgError(SPG_E_SINGULAR, "bottom Cholesky failed: leading minor " + std::to_string(hinfo) +
                                       " not positive definite");
  mark("bottom (dense inverse)");
  build_boundary_maps();
  mark("boundary maps");
}

// coefficient rows of the boundary system of every smoothed level
void Solver::build_boundary_rows() {
  for (int l = 0; l < lay_.nlev; ++l) {
    LevelRT& R = lv_[l];
    const int n = R.d.bnd_off[8];
    if (n == 0 || !R.bA64.p) continue;
    if (l == 0 && R.b0cslot.p) {
      launch_bnd0_setup(st_, R.d, R.b0cslot.as<int>(), E64_.as<double>(), cfg_.dx, R.b0E64.as<double>(),
                        R.b0D64.as<double>());
      launch_cast_d2f(st_, R.b0E64.as<double>(), R.b0E32.as<float>(), (int64_t)n * 8);
      launch_cast_d2f(st_, R.b0D64.as<double>(), R.b0D32.as<float>(), (int64_t)n * 8);
    }
    if (l == 0) launch_bnd_coef0(st_, R.d, E64_.as<double>(), cfg_.dx, R.bA64.as<double>());
    else if (lay_.lv[l].is_explicit) launch_bnd_coef_st(st_, R.d, R.st64.as<double>(), R.bA64.as<double>());
    else continue;
    launch_cast_d2f(st_, R.bA64.as<double>(), R.bA32.as<float>(), (int64_t)n * 288);
  }
  sync();
}

// Small boundary sets: each phase becomes one dense map.  The maps are optional
// (up to 1.4 GB a level), so they come after everything the solve needs, and a
// level for which there is no memory runs its phases by data flow instead.
void Solver::build_boundary_maps() {
  if (cfg_.boundary_iters <= 0) return;
  for (int l = 0; l < lay_.nlev; ++l) {
    LevelRT& R = lv_[l];
    const int n = R.d.bnd_off[8];
    if (n == 0 || !R.bA64.p || n > kMaxDenseBoundary || R.no_maps) continue;
    if (l > 0 && !lay_.lv[l].is_explicit) continue;
    if (!R.d.bmap_sweeps && !alloc_boundary_maps(l)) {
      R.no_maps = true;
      continue;
    }
    double* const M[2] = {R.bmap64[0].as<double>(), R.bmap64[1].as<double>()};
    float* const F[2] = {R.bmap32[0].as<float>(), R.bmap32[1].as<float>()};
    launch_bmap_build(st_, R.d, cfg_.boundary_iters, l == 0, M, F);
  }
  sync();
}

bool Solver::alloc_boundary_maps(int l) {
  LevelRT& R = lv_[l];
  const int n = R.d.bnd_off[8];
  const size_t entries = (size_t)3 * n * bmap_stride(n), nx = (size_t)bmap_stride(n);
  try {
    // SPG_MAP_MAX_MB: what the maps of a level may take
    const char* e = std::getenv("SPG_MAP_MAX_MB");
    if (e && (double)entries * 24.0 > std::atof(e) * 1048576.0) throw SpgError(SPG_E_HIP, "SPG_MAP_MAX_MB");
    for (int d = 0; d < 2; ++d) {
      R.bmap64[d].alloc(entries * 8);
      R.bmap32[d].alloc(entries * 4);
    }
    const LevelDesc& D = lay_.lv[l];
    std::vector<int32_t> list, all(D.bnd_ci.size());
    for (int c = 0; c < 8; ++c) list.insert(list.end(), D.bnd_list[c].begin(), D.bnd_list[c].end());
    for (size_t k = 0; k < all.size(); ++k) all[k] = D.bnd_ci[k] >= 0 ? list[D.bnd_ci[k]] : D.bnd_slot[k];
    upload(R.ball, all);
    R.bmx64.alloc(nx * 8);
    R.bmx32.alloc(nx * 4);
  } catch (const SpgError&) {
    (void)hipGetLastError();
    for (DBuf* b : {&R.bmap64[0], &R.bmap64[1], &R.bmap32[0], &R.bmap32[1], &R.ball, &R.bmx64, &R.bmx32}) b->alloc(0);
    if (!R.btag.p && lv_[0].coop.p) {  // an explicit level of this size has none yet
      try {
        R.btag.alloc((size_t)n * 6 * 8);
        R.d.btag = R.btag.p;
        R.d.coop = lv_[0].coop.as<unsigned>();
      } catch (const SpgError&) {
        (void)hipGetLastError();  // its phases run in one workgroup
      }
    }
    return false;
  }
  for (int d = 0; d < 2; ++d) {
    // padding columns stay zero: the build writes columns < 3n only
    HIPCHK(hipMemsetAsync(R.bmap64[d].p, 0, entries * 8, st_));
    HIPCHK(hipMemsetAsync(R.bmap32[d].p, 0, entries * 4, st_));
    R.d.bmap64[d] = R.bmap64[d].as<double>();
    R.d.bmap32[d] = R.bmap32[d].as<float>();
  }
  HIPCHK(hipMemsetAsync(R.bmx64.p, 0, nx * 8, st_));
  HIPCHK(hipMemsetAsync(R.bmx32.p, 0, nx * 4, st_));
  R.d.ball = R.ball.as<int>();
  R.d.bmx64 = R.bmx64.as<double>();
  R.d.bmx32 = R.bmx32.as<float>();
  R.d.bmap_sweeps = cfg_.boundary_iters;
  return true;
}

// The lowest i in [0, n) with ev(i) != 0, and ev there (n and 0 if none):
// the answer of one pass in order, found on up to 16 threads
template <class F>
static std::pair<int64_t, int> first_event(int64_t n, F&& ev) {
  std::mutex m;
  int64_t at = n;
  int kind = 0;
  parallel_ranges(
      n,
      [&](int64_t a, int64_t b) {
        for (int64_t i = a; i < b; ++i)
          if (const int k = ev(i)) {
            std::lock_guard<std::mutex> g(m);
            if (i < at) {
              at = i;
              kind = k;
            }
            return;
          }
      },
      1 << 15);
  return {at, kind};
}

bool Solver::active_set_matches(const double* density) const {
  const Layout& Lc = lay_;
  // 1: NaN (throws), 2: a cell would switch on or off
  const int kind = first_event(Lc.nin_blocks * 64, [&](int64_t i) {
    const int32_t s = Lc.in_node_slot[i];
    const double d = density[i];
    if (std::isnan(d)) return 1;
    // a cell whose min corner has no GPU slot is inactive; it may not turn on
    if (s < 0) return d > 0 ? 2 : 0;
    return (Lc.E[s] != 0.0) != (d > 0) ? 2 : 0;
  }).second;
  if (kind == 1) throw SpgError(SPG_E_NAN, "density contains NaN");
  return kind == 0;
}

void Solver::update_density(const double* density) {
  activate();
  // recompute E (SIMP) for the existing cells, then the coarse operators;
  // nothing changes when the check fails
  const int64_t nin = lay_.nin_blocks * 64;
  const int kind = first_event(nin, [&](int64_t i) {
    const int32_t s = lay_.in_node_slot[i];
    if (s < 0) return 0;
    const double d = density[i];
    if (std::isnan(d)) return 1;
    if (lay_.E[s] != 0.0) return d > 0 ? 0 : 2;
    return d > 0 ? 3 : 0;
  }).second;
  if (kind == 1) throw SpgError(SPG_E_NAN, "density contains NaN");
  if (kind == 2) throw SpgError(SPG_E_INVALID, "density update would deactivate a cell (topology change)");
  if (kind == 3) throw SpgError(SPG_E_INVALID, "density update would activate a cell (topology change)");
  // input nodes have distinct slots: the ranges write disjoint entries
  parallel_ranges(
      nin,
      [&](int64_t a, int64_t b) {
        for (int64_t i = a; i < b; ++i) {
          const int32_t s = lay_.in_node_slot[i];
          if (s < 0) continue;
          const double d = density[i];
          lay_.rho[s] = d;
          if (lay_.E[s] != 0.0) lay_.E[s] = stiffness_mapping(cfg_.penalty, cfg_.min_stiffness, cfg_.min_density, d);
        }
      },
      1 << 15);
  // both arrays through the kept pinned buffer, filled on host threads: a
  // pageable copy runs at a few GB/s on one thread
  const size_t ne = lay_.E.size() * 8, nr = lay_.rho.size() * 8;
  HIPCHK(hipStreamSynchronize(st_));  // the buffer may still feed an earlier copy
  if (stage_bytes_ < ne + nr) {
    if (stage_) (void)hipHostFree(stage_);
    stage_ = nullptr;
    stage_bytes_ = 0;
    HIPCHK(hipHostMalloc(&stage_, ne + nr));
    stage_bytes_ = ne + nr;
  }
  uint8_t* hs = static_cast<uint8_t*>(stage_);
  const uint8_t* srcE = reinterpret_cast<const uint8_t*>(lay_.E.data());
  const uint8_t* srcR = reinterpret_cast<const uint8_t*>(lay_.rho.data());
  parallel_ranges(
      (int64_t)(ne + nr),
      [&](int64_t a, int64_t b) {
        for (int64_t i = a; i < b;) {
          const int64_t end = i < (int64_t)ne ? std::min<int64_t>(b, ne) : b;
          std::memcpy(hs + i, i < (int64_t)ne ? srcE + i : srcR + (i - ne), (size_t)(end - i));
          i = end;
        }
      },
      1 << 22);
  HIPCHK(hipMemcpyAsync(E64_.p, hs, ne, hipMemcpyHostToDevice, st_));
  HIPCHK(hipMemcpyAsync(rho_.p, hs + ne, nr, hipMemcpyHostToDevice, st_));
  launch_cast_d2f(st_, E64_.as<double>(), E32_.as<float>(), (int64_t)lay_.E.size());
  build_operators();
  // the pinned buffer must not change before the copies have read it
  HIPCHK(hipStreamSynchronize(st_));
}

void Solver::update_density_device(const double* density_dev) {
  activate();
  // same checks and SIMP map as update_density, on the device; nothing
  // changes when the check fails
  const int64_t nin = lay_.nin_blocks * 64;
  if (!derr_.p) derr_.alloc(16);
  int* err = derr_.as<int>();
  HIPCHK(hipMemsetAsync(err, 0, sizeof(int), st_));
  launch_density_check(st_, nin, in_slot_.as<int>(), density_dev, E64_.as<double>(), err);
  int herr = 0;
  HIPCHK(hipMemcpyAsync(&herr, err, sizeof(int), hipMemcpyDeviceToHost, st_));
  sync();
  if (herr & 1) throw SpgError(SPG_E_NAN, "density contains NaN");
  if (herr & 2) throw SpgError(SPG_E_INVALID, "density update would deactivate a cell (topology change)");
  if (herr & 4) throw SpgError(SPG_E_INVALID, "density update would activate a cell (topology change)");
  launch_density_update(st_, nin, in_slot_.as<int>(), density_dev, cfg_.penalty, cfg_.min_stiffness,
                        cfg_.min_density, E64_.as<double>(), E32_.as<float>(), rho_.as<double>());
  build_operators();
}

void Solver::set_forces(int64_t n, const int32_t* coord, const double* value) {
  // ForceOnNode assignment (SPGrid_CPU_Solver.cpp:289-296): later entries win
  if (gmap0_.empty()) {
    const LevelDesc& D = lay_.lv[0];
    gmap0_.reserve(D.nb * 2);
    for (int64_t b = 0; b < D.nb; ++b)
      gmap0_.emplace(bkey(D.base[3 * b] >> 2, D.base[3 * b + 1] >> 2, D.base[3 * b + 2] >> 2), (int32_t)b);
  }
  std::vector<int32_t> idx;
  std::vector<double> val;
  std::unordered_map<int32_t, size_t> at;  // node slot -> its entry: a repeated node keeps the last value
  for (int64_t i = 0; i < n; ++i) {
    const int x = coord[3 * i], y = coord[3 * i + 1], z = coord[3 * i + 2];
    auto it = gmap0_.find(bkey(x >> 2, y >> 2, z >> 2));
    if (it == gmap0_.end()) continue;  // forces outside the solved blocks are ignored
    const int32_t g = it->second;
    const int q = ((x & 3) << 4) | ((y & 3) << 2) | (z & 3);
    const int32_t slot = g * 64 + q;
    auto [pos, fresh] = at.emplace(slot, idx.size());
    if (!fresh) {
      for (int c = 0; c < 3; ++c) val[pos->second + c] = value[3 * i + c];
      continue;
    }
    for (int c = 0; c < 3; ++c) {
      idx.push_back(slot * 3 + c);
      val.push_back(value[3 * i + c]);
    }
  }
  upload(f_idx_, idx);
  upload(f_val_, val);
  n_f_ = (int64_t)idx.size();
}

double Solver::read_scalar(const double* dev) {
  HIPCHK(hipMemcpyAsync(hscal_, dev, sizeof(double), hipMemcpyDeviceToHost, st_));
  sync();
  return hscal_[0];
}

// ------------------------------------------------------------------ V-cycle
// Per block, a colour launch reads the 5^3 halo of u and E (mostly shared
// with the neighbouring blocks' halos) but, in node-major order, whole cache
// lines of b and the flags for the 8 nodes of its colour.  A colour-major
// copy of b, made once per V-cycle, saves 7/8 of those bytes in each of the
// 16 colour launches.  Measured per V-cycle (FP32 / FP64): the 256^3 shell
// (82,765 blocks) 1.605 / 2.405 ms node-major against 1.675 / 2.426 ms with
// the copy; the 512x256x256 band (245,910 blocks) 4.254 / 5.937 ms against
// 4.100 / 5.809 ms.  By default the copy is used above 256 MiB of u, b, E and
// neighbour table in FP32, i.e. above about 137 K blocks.
// The level-0 flags in colour-major order and room for b in that order,
// allocated after everything the solve needs: without the memory for them
// the colour sweeps keep reading node-major.
void Solver::setup_colour_major() {
  if (!(cmb_mode_ == 1 || (cmb_mode_ < 0 && colour_major_by_size(lv_[0].d.nb)))) return;
  const LevelRT& R0 = lv_[0];
  try {
    fcm_.alloc((size_t)R0.d.nb * 64);
    bcm_.alloc((size_t)R0.n3 * 8);
  } catch (const SpgError&) {
    (void)hipGetLastError();
    fcm_.alloc(0);
    bcm_.alloc(0);
    return;
  }
  launch_colour_major_flags(st_, R0.d.nb, R0.d.flags, fcm_.as<uint8_t>());
  lv_[0].d.flags_cm = fcm_.as<uint8_t>();
}

template <class T>
const T* Solver::colour_major_b(const T* b0) {
  if (!lv_[0].d.flags_cm) return nullptr;
  if (cmb_mode_ < 0 && !colour_major_by_size(lv_[0].d.nb)) return nullptr;
  T* bcm = reinterpret_cast<T*>(bcm_.p);
  launch_colour_major<T>(st_, lv_[0].d, b0, bcm);
  return bcm;
}

template <class T>
void Solver::smooth(int l, T* u, const T* b, bool forward, const T* bcm, Part part) {
  const LevelRT& R = lv_[l];
  // Multigrid_Hierarchy.h:577-586 / 605-617: boundary sweeps, full sweeps, boundary sweeps
  auto boundary = [&] {
    if (l == 0) launch_gs0_boundary<T>(st_, R.d, E<T>(), dxT<T>(), u, b, cfg_.boundary_iters, forward);
    else launch_st_boundary<T>(st_, R.d, R.st<T>(), u, b, cfg_.boundary_iters, forward);
  };
  int first = 0;
  if (part == Part::kFirst) {
    boundary();
    return;
  }
  if (l == 0 && overlap_ && R.gsdist.p && cfg_.smooth_iters > 0 && cfg_.boundary_iters > 0) {
    // The boundary phase writes only band nodes.  The first sweep's step-c
    // update of a node farther than c + 1 from the band reads nothing that
    // phase writes, directly or through earlier steps (Layout::gs_near), so
    // those updates run on st2_ beside the phase; the near ones follow on
    // st_ once both are done, step by step as the sequential sweep orders
    // them.  The result is the sequential sweep's.  256^3 shell, FP32
    // V-cycle: 1.71 ms against 1.62 ms sequential (the near-band list
    // launches cost what the overlap saves), hence off by default.
    HIPCHK(hipEventRecord(ev_a_, st_));
    boundary();
    HIPCHK(hipStreamWaitEvent(st2_, ev_a_, 0));
    for (int c = 0; c < 8; ++c)
      launch_gs0<T>(st2_, R.d, E<T>(), dxT<T>(), u, b, sweep_colour(true, forward, c), R.gsdist.as<uint8_t>(), c + 2);
    HIPCHK(hipEventRecord(ev_b_, st2_));
    HIPCHK(hipStreamWaitEvent(st_, ev_b_, 0));
    const int dir = forward ? 0 : 1;
    for (int c = 0; c < 8; ++c) {
      const int64_t o = R.gsnear_off[dir * 8 + c], n = R.gsnear_off[dir * 8 + c + 1] - o;
      launch_gs0_list<T>(st_, R.d, R.gsnear.as<int>() + o, R.gsnslot.as<int>() + o * 27, (int)n, E<T>(), dxT<T>(), u,
                         b);
    }
    first = 1;
  } else if (part == Part::kAll) {
    boundary();
  }
  for (int i = first; i < cfg_.smooth_iters; ++i) {
    if (l == 0) launch_gs0_sweep<T>(st_, R.d, E<T>(), dxT<T>(), u, b, forward, bcm);
    else launch_st_sweep<T>(st_, R.d, R.st<T>(), u, b, forward);
  }
  boundary();
}

template <class T>
void Solver::level_residual(int l, const T* u, const T* b, T* r) {
  if (l == 0) launch_apply<T>(st_, lv_[0].d, E<T>(), dxT<T>(), u, b, r, 1);
  else launch_st_residual<T>(st_, lv_[l].d, lv_[l].st<T>(), u, b, r);
}

template <class T>
void Solver::bottom(const T* b, T* u) {
  const LevelRT& R = lv_[lay_.nlev - 1];
  if (nd_) {
    // FP64 factors in both cycles: the FP32 cycle's right-hand side is
    // widened and the solution rounded, as the reference casts the PARDISO
    // result to float (Multigrid_Hierarchy.h:346-372, 439-451)
    nd_->solve<T>(b, u, st_);
    return;
  }
  const int *vs = vslot_.as<int>(), *vo = var_of_.as<int>();
  // FP32 cycle with the FP64 inverse: widened, applied and rounded back
  if (sizeof(T) == 8 || bottom64_)
    launch_bottom_dense<T, double>(st_, R.d, nT_, tiles64_.as<double>(), vs, vo, b, pb64_.as<double>(), u);
  else
    launch_bottom_dense<T, float>(st_, R.d, nT_, tiles32_.as<float>(), vs, vo, b, pb32_.as<float>(), u);
}

// FP32 cycle whose explicit levels (and bottom) run in FP64: the level
// handed over is restricted in FP32 and widened, and widened corrections are
// rounded back before the FP32 prolongation
void Solver::vcycle_coarse64(const float* b0, float* z, bool z_is_zero, Part part) {
  const int L = lay_.nlev;
  const int ex = lay_.explicit_level;
  if (!z_is_zero) launch_zero<float>(st_, z, lv_[0].n3);
  const float* bcm = colour_major_b<float>(b0);
  for (int l = 0; l < L - 1; ++l) {
    const bool d = l >= ex, dn = l + 1 >= ex;
    const bool sm = (l == 0 || l >= ex);
    if (d) {
      double* u = lv_[l].u<double>();
      const double* b = lv_[l].b<double>();
      smooth<double>(l, u, b, true);
      launch_zero<double>(st_, lv_[l + 1].u<double>(), lv_[l + 1].n3);
      level_residual<double>(l, u, b, lv_[l].r<double>());
      launch_restrict<double>(st_, lv_[l + 1].d, lv_[l].r<double>(), lv_[l + 1].b<double>());
    } else {
      float* u = l == 0 ? z : lv_[l].u<float>();
      const float* b = l == 0 ? b0 : lv_[l].b<float>();
      if (sm) smooth<float>(l, u, b, true, l == 0 ? bcm : nullptr, l == 0 ? part : Part::kAll);
      if (dn) launch_zero<double>(st_, lv_[l + 1].u<double>(), lv_[l + 1].n3);
      else launch_zero<float>(st_, lv_[l + 1].u<float>(), lv_[l + 1].n3);
      if (sm) {
        level_residual<float>(l, u, b, lv_[l].r<float>());
        launch_restrict<float>(st_, lv_[l + 1].d, lv_[l].r<float>(), lv_[l + 1].b<float>());
      } else {
        launch_restrict<float>(st_, lv_[l + 1].d, b, lv_[l + 1].b<float>());
      }
      if (dn) launch_cast_f2d(st_, lv_[l + 1].b<float>(), lv_[l + 1].b<double>(), lv_[l + 1].n3);
    }
  }
  if (L - 1 >= ex) bottom<double>(lv_[L - 1].b<double>(), lv_[L - 1].u<double>());
  else bottom<float>(lv_[L - 1].b<float>(), lv_[L - 1].u<float>());
  for (int l = L - 2; l >= 0; --l) {
    const bool d = l >= ex, dn = l + 1 >= ex;
    if (d) {
      launch_prolongate<double>(st_, lv_[l].d, lv_[l + 1].u<double>(), lv_[l].u<double>());
      smooth<double>(l, lv_[l].u<double>(), lv_[l].b<double>(), false);
    } else {
      float* u = l == 0 ? z : lv_[l].u<float>();
      const float* b = l == 0 ? b0 : lv_[l].b<float>();
      if (dn) launch_cast_d2f(st_, lv_[l + 1].u<double>(), lv_[l + 1].u<float>(), lv_[l + 1].n3);
      launch_prolongate<float>(st_, lv_[l].d, lv_[l + 1].u<float>(), u);
      if (l == 0 || l >= ex) smooth<float>(l, u, b, false, l == 0 ? bcm : nullptr);
    }
  }
}

bool Solver::has_first_part() const {
  return lay_.use_mg && lay_.nlev > 1 && lay_.explicit_level > 0 && !overlap_ && cfg_.boundary_iters > 0;
}

template <class T>
void Solver::vcycle(const T* b0, T* z, bool z_is_zero, Part part) {
  if (part == Part::kFirst) {
    smooth<T>(0, z, b0, true, nullptr, part);
    return;
  }
  const int L = lay_.nlev;
  const int ex = lay_.explicit_level;
  if (sizeof(T) == 4 && coarse64_ && lay_.use_mg && L > ex) {
    vcycle_coarse64(reinterpret_cast<const float*>(b0), reinterpret_cast<float*>(z), z_is_zero, part);
    return;
  }
  if (!lay_.use_mg) {
    launch_copy<T>(st_, b0, z, lv_[0].n3);
    return;
  }
  if (L == 1) {
    bottom<T>(b0, z);
    return;
  }
  if (!z_is_zero) launch_zero<T>(st_, z, lv_[0].n3);
  const T* bcm = colour_major_b<T>(b0);
  for (int l = 0; l < L - 1; ++l) {
    T* u = l == 0 ? z : lv_[l].u<T>();
    const T* b = l == 0 ? b0 : lv_[l].b<T>();
    const bool sm = (l == 0 || l >= ex);
    if (sm) smooth<T>(l, u, b, true, l == 0 ? bcm : nullptr, l == 0 ? part : Part::kAll);
    // the restriction also clears the coarse iterate
    if (sm) {
      level_residual<T>(l, u, b, lv_[l].r<T>());
      launch_restrict<T>(st_, lv_[l + 1].d, lv_[l].r<T>(), lv_[l + 1].b<T>(), lv_[l + 1].u<T>());
    } else {
      launch_restrict<T>(st_, lv_[l + 1].d, b, lv_[l + 1].b<T>(), lv_[l + 1].u<T>());
    }
  }
  bottom<T>(lv_[L - 1].b<T>(), lv_[L - 1].u<T>());
  for (int l = L - 2; l >= 0; --l) {
    T* u = l == 0 ? z : lv_[l].u<T>();
    const T* b = l == 0 ? b0 : lv_[l].b<T>();
    launch_prolongate<T>(st_, lv_[l].d, lv_[l + 1].u<T>(), u);
    if (l == 0 || l >= ex) smooth<T>(l, u, b, false, l == 0 ? bcm : nullptr);
  }
}

// ---------------------------------------------------------------------- PCG
// CONJUGATE_GRADIENT_4Ch::Solve (CG/CONJUGATE_GRADIENT.cpp:21-61): projected
// PCG on x (starting at 0) with the L_inf stop test; scalars stay FP64 on the
// device, the host reads ||r||_inf once per iteration.
CgReport Solver::report() {
  CgReport r;
  r.host = reinterpret_cast<unsigned long long*>(reinterpret_cast<char*>(hscal_) + kReportOffset);
  r.seq = ++report_seq_;
  if (lv_[0].coop.p && lv_[0].d.flow) r.err = lv_[0].coop.as<int>() + 1;
  return r;
}

// Each word carries the report's number, so the values are complete once all
// words do; the stream's state is looked at now and then so that a failed
// kernel ends the wait.
void Solver::wait_report(double* nrm, unsigned* bits) {
  const unsigned long long* w =
      reinterpret_cast<const unsigned long long*>(reinterpret_cast<const char*>(hscal_) + kReportOffset);
  unsigned long long v[kReportWords];
  auto arrived = [&] {
    bool ok = true;
    for (int i = 0; i < kReportWords; ++i) {
      v[i] = __atomic_load_n(w + i, __ATOMIC_ACQUIRE);
      ok = ok && (unsigned)(v[i] >> 32) == report_seq_;
    }
    return ok;
  };
  for (unsigned spin = 1; !arrived(); ++spin) {
    if (spin % 65536 == 0) {
      const hipError_t e = hipStreamQuery(st_);
      if (e == hipErrorNotReady) continue;
      HIPCHK(e);
      if (!arrived()) throw SpgError(SPG_E_HIP, "PCG: the stream is idle and the residual has not arrived");
      break;
    }
    __builtin_ia32_pause();
  }
  const unsigned long long b = (v[0] & 0xffffffffull) | (v[1] << 32);
  std::memcpy(nrm, &b, sizeof(b));
  *bits = (unsigned)v[2];
}

template <class T>
int Solver::pcg(T* x, T* r, double tol, int maxit, int* iters, double* last_nrm) {
  const LevelRT& R0 = lv_[0];
  const int64_t n = R0.n3;
  T* s = sizeof(T) == 4 ? (T*)s32_.p : (T*)s64_.p;
  T* q = sizeof(T) == 4 ? (T*)q32_.p : (T*)q64_.p;
  T* z = sizeof(T) == 4 ? (T*)z32_.p : (T*)z64_.p;
  CgScalars* sc = scal_.as<CgScalars>();
  double* part = part_.as<double>();
  launch_zero<T>(st_, x, n);
  launch_zero<T>(st_, s, n);
  launch_zero<T>(st_, z, n);
  launch_project<T>(st_, R0.d, r, true);
  launch_cg_scalars(st_, sc, 3);
  launch_linf<T>(st_, r, n, part, &sc->nrm, report(), sc);
  int it = 0;
  int rc = SPG_E_NOT_CONVERGED;
  const bool flows = lv_[0].coop.p && lv_[0].d.flow;
  // The next V-cycle's first boundary phase, which changes nothing but z, is
  // launched before the host reads the residual: the device has work while the
  // host decides and launches the rest.  With that, and the report written by
  // the iteration's last kernel instead of two copies and a synchronisation,
  // the device no longer idles between iterations.
  const bool split = has_first_part();
  bool ahead = false;
  for (;; ++it) {
    ahead = split && it < maxit;
    if (ahead) vcycle<T>(r, z, true, Part::kFirst);
    double nrm;
    unsigned bits;
    wait_report(&nrm, &bits);
    if (bits >> 1) {
      // a kernel of the last V-cycle ended early: its result is not a
      // Gauss-Seidel sweep.  Use none of them any more and let the caller
      // repeat the pass.
      HIPCHK(hipMemsetAsync(lv_[0].coop.as<unsigned>() + 1, 0, sizeof(unsigned), st_));
      sync();
      flow_dead_ = true;
      set_flow(kFlowNone);
      std::fprintf(stderr,
                   "spgrid_topo_opt_amd: %s: a wait timed out (workgroups not resident together); continuing with "
                   "per-colour launches\n",
                   flow_names(bits >> 1).c_str());
      *iters = it;
      return kFlowRetry;
    }
    *last_nrm = nrm;
    if (print_residuals_) {
      FILE* o = print_residuals_ == 2 ? stderr : stdout;
      std::fprintf(o, "%.9g\n", nrm);
      std::fflush(o);
    }
    if (bits & 1) {
      rc = SPG_E_SINGULAR;
      break;
    }
    if (std::isnan(nrm)) {
      rc = SPG_E_NAN;
      break;
    }
    if (nrm <= tol) {
      rc = SPG_OK;
      break;
    }
    if (it == maxit) break;
    vcycle<T>(r, z, true, ahead ? Part::kRest : Part::kAll);  // z was cleared before the loop / by the last update
    // the scalar stages (beta, alpha, rho_old) run in the last kernel of
    // the reduction they follow
    const int nr = launch_project_dot<T>(st_, R0.d, z, r, part, &sc->rho, sc, 0);
    launch_cg_direction<T>(st_, s, z, sc, n, part, nr);
    const int nq = launch_apply_dot<T>(st_, R0.d, E<T>(), dxT<T>(), s, q, apart_.as<double>(), part, &sc->sq, sc, 1);
    launch_cg_update<T>(st_, x, r, s, q, sc, n, 2, z, report(), apart_.as<double>(), nq);
  }
  // a time-out in a phase whose result nobody uses is nobody's error
  if (ahead && flows) HIPCHK(hipMemsetAsync(lv_[0].coop.as<unsigned>() + 1, 0, sizeof(unsigned), st_));
  *iters = it;
  return rc;
}

void Solver::reset_to_ud(double* u) {
  launch_zero<double>(st_, u, lv_[0].n3);
  launch_set_entries(st_, u, ud_idx_.as<int>(), ud_val_.as<double>(), n_ud_);
}

int Solver::solve_rhs(const spg_solve_params& prm, double* u, const double* f, spg_info* info, bool warm) {
  const FlowLease lease(*this, prm.precision);
  const LevelRT& R0 = lv_[0];
  const int64_t n = R0.n3;
  const double t0 = now_s();
  double* part = part_.as<double>();
  double* red = part + reduce_partials(0);
  auto residual_linf = [&](const double* x) {
    launch_apply<double>(st_, R0.d, E<double>(), cfg_.dx, x, f, res_.as<double>(), 1);
    launch_linf<double>(st_, res_.as<double>(), n, part, red);
    return read_scalar(red);
  };
  // The target is relative to the zero-guess residual: this problem's own,
  // or under a warm start the one stored from the first solve.  A warm
  // guess is kept when forced or when its residual is below that reference
  // (SPGrid_CPU_Solver.cpp:247-285, 318-326).
  double r0 = 0.0, rstart = 0.0;
  bool reused = false;
  if (warm) {
    r0 = prm.reference_linf;
    if (!(r0 > 0)) {
      reset_to_ud(tmp_.as<double>());
      r0 = residual_linf(tmp_.as<double>());
    }
    rstart = residual_linf(u);
    reused = prm.warm_start == 2 || r0 > rstart;
    if (!reused) {
      reset_to_ud(u);
      rstart = residual_linf(u);
    }
  } else {
    r0 = rstart = residual_linf(u);
  }
  const double target = prm.tolerance * r0;
  print_residuals_ = prm.print_residuals;
  int total = 0, passes = 0, rc = SPG_OK;
  double rn = rstart;
  bool conv = (rstart <= target);
  if (std::isnan(rstart) || std::isnan(r0)) rc = SPG_E_NAN;
  const int maxp = prm.max_passes < 1 ? 1 : prm.max_passes;
  for (int pass = 0; pass < maxp && !conv && rc == SPG_OK; ++pass) {
    // per-pass target: an explicit inner reduction, or (inner_tolerance <= 0)
    // the final target itself, but never asking an FP32 pass for more than
    // kFp32PassReduction of its starting residual
    double tolp = target;
    if (prm.inner_tolerance > 0) tolp = std::max(prm.inner_tolerance * rn, 0.7 * target);
    else if (prm.precision == 0) tolp = std::max(target, kFp32PassReduction * rn);
    int it = 0;
    double last = 0;
    int prc;
    for (int attempt = 0;; ++attempt) {
      if (prm.precision == 1) {
        launch_copy<double>(st_, res_.as<double>(), rr64_.as<double>(), n);
        prc = pcg<double>(x64_.as<double>(), rr64_.as<double>(), tolp, prm.max_iterations, &it, &last);
      } else {
        launch_cast_d2f(st_, res_.as<double>(), rr32_.as<float>(), n);
        prc = pcg<float>(x32_.as<float>(), rr32_.as<float>(), tolp, prm.max_iterations, &it, &last);
      }
      if (prc != kFlowRetry) break;
      total += it;
      if (attempt > 0) throw SpgError(SPG_E_HIP, "a data-flow wait timed out after the switch to per-colour launches");
    }
    if (prm.precision == 1) launch_axpy_d<double>(st_, u, x64_.as<double>(), n);
    else launch_axpy_d<float>(st_, u, x32_.as<float>(), n);
    total += it;
    passes++;
    launch_apply<double>(st_, R0.d, E<double>(), cfg_.dx, u, f, res_.as<double>(), 1);
    launch_linf<double>(st_, res_.as<double>(), n, part, red);
    rn = read_scalar(red);
    if (prc == SPG_E_SINGULAR || prc == SPG_E_NAN) rc = prc;
    if (std::isnan(rn)) rc = SPG_E_NAN;
    if (rn <= target) conv = true;
  }
  launch_sumsq(st_, res_.as<double>(), n, part, red);
  const double l2 = std::sqrt(read_scalar(red));
  if (info) {
    static_info(info);
    info->iterations = total;
    info->passes = passes;
    info->converged = conv ? 1 : 0;
    info->r0_linf = r0;
    info->r_linf = rn;
    info->r_l2 = l2;
    info->solve_seconds = now_s() - t0;
    info->r_start_linf = rstart;
    info->warm_reused = reused ? 1 : 0;
  }
  check_flow();
  if (rc == SPG_OK && !conv) rc = SPG_E_NOT_CONVERGED;
  return rc;
}

void Solver::static_info(spg_info* info) const {
  info->levels = lay_.nlev;
  info->setup_seconds = setup_s_;
  info->active_nodes = lay_.lv[0].n_active;
  info->active_cells = lay_.n_active_cells;
  info->gpu_blocks = lay_.lv[0].nb;
  info->bottom_dofs = nvar_;
  info->hbm_bytes = dev_bytes_;
  info->bottom_kind = nd_ ? 1 : 0;
  info->bottom_bytes = nd_ ? (double)nd_->device_bytes()
                           : (double)(tiles64_.bytes + tiles32_.bytes + pb64_.bytes + pb32_.bytes);
}

int Solver::solve(const spg_solve_params& prm, spg_info* info) {
  activate();
  const LevelRT& R0 = lv_[0];
  const int64_t n = R0.n3;
  if (prm.warm_start < 0 || prm.warm_start > 2) throw SpgError(SPG_E_INVALID, "warm_start must be 0, 1 or 2");
  // a warm start begins at the previous solution (or the given guess) with
  // u_D written over it; otherwise at u_D (SPGrid_CPU_Solver.cpp:241-285)
  const bool warm = prm.warm_start != 0 && (have_solution_ || have_guess_);
  if (warm) launch_set_entries(st_, u_.as<double>(), ud_idx_.as<int>(), ud_val_.as<double>(), n_ud_);
  else reset_to_ud(u_.as<double>());
  // f = P P_null forces (SPGrid_CPU_Solver.cpp:289-299)
  launch_zero<double>(st_, f_.as<double>(), n);
  launch_set_entries(st_, f_.as<double>(), f_idx_.as<int>(), f_val_.as<double>(), n_f_);
  launch_project<double>(st_, R0.d, f_.as<double>(), true);
  have_guess_ = false;
  have_solution_ = false;
  const int rc = solve_rhs(prm, u_.as<double>(), f_.as<double>(), info, warm);
  // a failed solve leaves nothing to warm-start from
  have_solution_ = rc == SPG_OK || rc == SPG_E_NOT_CONVERGED;
  return rc;
}

void Solver::set_initial_guess_in3(const double* dev) {
  const LevelRT& R0 = lv_[0];
  launch_zero<double>(st_, u_.as<double>(), R0.n3);
  launch_scatter_input_vec(st_, in_slot_.as<int>(), lay_.nin_blocks * 64, dev, u_.as<double>());
  launch_project<double>(st_, R0.d, u_.as<double>(), true);
  sync();
  have_guess_ = true;
}

int Solver::solve_adjoint(const spg_solve_params& prm, const double* g_in3, double* lam_in3, spg_info* info) {
  activate();
  const LevelRT& R0 = lv_[0];
  const int64_t n = R0.n3;
  const int64_t nin = lay_.nin_blocks * 64;
  launch_zero<double>(st_, tmp_.as<double>(), n);
  launch_scatter_input_vec(st_, in_slot_.as<int>(), nin, g_in3, tmp_.as<double>());
  launch_project<double>(st_, R0.d, tmp_.as<double>(), true);
  // lambda with homogeneous Dirichlet data
  if (!lam_.p) lam_.alloc(n * 8);
  launch_zero<double>(st_, lam_.as<double>(), n);
  const int rc = solve_rhs(prm, lam_.as<double>(), tmp_.as<double>(), info, false);
  launch_gather_input_vec(st_, in_slot_.as<int>(), nin, lam_.as<double>(), lam_in3);
  sync();
  return rc;
}

void Solver::pack_records(const int32_t* base, int hdr, uint8_t* dst) const {
  const int64_t nb = lay_.nin_blocks, nin = nb * 64;
  const size_t rec = (size_t)hdr * 4 + 64 * 32;
  if (nb > 0) {
    DBuf out, bdev;
    out.alloc((size_t)nb * rec);
    if (hdr > 0) {
      bdev.alloc((size_t)nb * 3 * sizeof(int32_t));
      HIPCHK(hipMemcpyAsync(bdev.p, base, (size_t)nb * 3 * sizeof(int32_t), hipMemcpyHostToDevice, st_));
    }
    launch_pack_out4(st_, in_slot_.as<int>(), nin, u_.as<double>(), res_.as<double>(), bdev.as<int32_t>(), hdr,
                     out.as<uint32_t>());
    // through a kept pinned buffer, copied out on host threads: a pageable
    // copy of this size runs at a few GB/s on one thread
    const size_t bytes = (size_t)nb * rec;
    if (stage_bytes_ < bytes) {
      if (stage_) (void)hipHostFree(stage_);
      stage_ = nullptr;
      stage_bytes_ = 0;
      HIPCHK(hipHostMalloc(&stage_, bytes));
      stage_bytes_ = bytes;
    }
    HIPCHK(hipMemcpyAsync(stage_, out.p, bytes, hipMemcpyDeviceToHost, st_));
    HIPCHK(hipStreamSynchronize(st_));
    const uint8_t* src = static_cast<const uint8_t*>(stage_);
    parallel_ranges(
        (int64_t)bytes, [&](int64_t a, int64_t b) { std::memcpy(dst + a, src + a, (size_t)(b - a)); }, 1 << 22);
  }
  // Dirichlet entries of nodes without a slot keep their prescribed value
  for (size_t k = 0; k < lay_.ud_extra.size(); ++k) {
    const int64_t e = lay_.ud_extra[k], n = e / 3;
    std::memcpy(dst + (n >> 6) * rec + hdr * 4 + ((n & 63) * 4 + e % 3) * 8, &lay_.ud_extra_value[k], 8);
  }
}

void Solver::pack_output(double* out4) const { pack_records(nullptr, 0, reinterpret_cast<uint8_t*>(out4)); }

void Solver::pack_output_records(const int32_t* base, uint8_t* dst) const { pack_records(base, 3, dst); }

void Solver::displacement_in3(double* dev) const {
  launch_gather_input_vec(st_, in_slot_.as<int>(), lay_.nin_blocks * 64, u_.as<double>(), dev);
  HIPCHK(hipStreamSynchronize(st_));
}

double Solver::sensitivity(const double* u_in3_dev, const double* lam_in3_dev, double* dc_in_dev) {
  activate();
  const LevelRT& R0 = lv_[0];
  const int64_t nin = lay_.nin_blocks * 64;
  // the FP64 PCG vectors are free between solves: x64 takes the scattered u,
  // q64 the sensitivities
  double* dc = q64_.as<double>();
  const double* u = u_.as<double>();
  if (u_in3_dev) {
    launch_zero<double>(st_, x64_.as<double>(), R0.n3);
    launch_scatter_input_vec(st_, in_slot_.as<int>(), nin, u_in3_dev, x64_.as<double>());
    u = x64_.as<double>();
  }
  const double* a = u;
  if (lam_in3_dev) {
    launch_zero<double>(st_, tmp_.as<double>(), R0.n3);
    launch_scatter_input_vec(st_, in_slot_.as<int>(), nin, lam_in3_dev, tmp_.as<double>());
    a = tmp_.as<double>();
  }
  double* part = part_.as<double>();
  double* obj = lam_in3_dev ? nullptr : part + reduce_partials(0);
  launch_sensitivity(st_, R0.d, rho_.as<double>(), u, a, cfg_.penalty, cfg_.min_stiffness, dc, apart_.as<double>(),
                     part, obj);
  launch_gather_input_scalar(st_, in_slot_.as<int>(), nin, dc, dc_in_dev);
  if (obj) return read_scalar(obj);
  sync();
  return 0.0;
}

// ----------------------------------------------------------- kernel hooks
template <class T>
static std::vector<T> to_dev_layout(const double* in, int64_t nb) {
  std::vector<T> v(nb * 192);
  for (int64_t b = 0; b < nb; ++b)
    for (int l = 0; l < 64; ++l)
      for (int c = 0; c < 3; ++c) v[(b * 3 + c) * 64 + l] = (T)in[(b * 64 + l) * 3 + c];
  return v;
}
template <class T>
static void from_dev_layout(const std::vector<T>& v, int64_t nb, double* out) {
  for (int64_t b = 0; b < nb; ++b)
    for (int l = 0; l < 64; ++l)
      for (int c = 0; c < 3; ++c) out[(b * 64 + l) * 3 + c] = (double)v[(b * 3 + c) * 64 + l];
}

void Solver::run_kernel(int op, int level, int precision, int forward, const double* in, const double* b,
                        double* out) {
  activate();
  if (level < 0 || level >= lay_.nlev) throw SpgError(SPG_E_INVALID, "level out of range");
  const FlowLease lease(*this, precision, true);
  auto body = [&](auto tag) {
    using T = decltype(tag);
    auto put = [&](DBuf& d, const double* h, int64_t nb) {
      std::vector<T> v = to_dev_layout<T>(h, nb);
      d.alloc(v.size() * sizeof(T));
      HIPCHK(hipMemcpy(d.p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
    };
    auto get = [&](const T* d, int64_t nb) {
      std::vector<T> v(nb * 192);
      sync();
      HIPCHK(hipMemcpy(v.data(), d, v.size() * sizeof(T), hipMemcpyDeviceToHost));
      from_dev_layout<T>(v, nb, out);
    };
    const int64_t nb = lv_[level].d.nb;
    DBuf A, Bv, O;
    switch (op) {
      case SPG_OP_APPLY:
      case SPG_OP_RESIDUAL:
      case SPG_OP_OPERATOR: {
        if (level != 0) throw SpgError(SPG_E_INVALID, "apply is a level-0 operator");
        put(A, in, nb);
        if (op == SPG_OP_RESIDUAL) put(Bv, b, nb);
        O.alloc(nb * 192 * sizeof(T));
        launch_apply<T>(st_, lv_[0].d, E<T>(), dxT<T>(), A.as<T>(), Bv.as<T>(), O.as<T>(),
                        op == SPG_OP_APPLY ? 0 : (op == SPG_OP_RESIDUAL ? 1 : 2));
        get(O.as<T>(), nb);
        break;
      }
      case SPG_OP_GS_SWEEP:
      case SPG_OP_GS_BOUNDARY: {
        if (level != 0 && !lay_.lv[level].is_explicit) throw SpgError(SPG_E_INVALID, "level has no smoother");
        put(A, in, nb);
        put(Bv, b, nb);
        const LevelDev& Ld = lv_[level].d;
        const bool fwd = (forward & 1) != 0;
        const int sweeps = std::max(1, forward >> 8);
        if (op == SPG_OP_GS_BOUNDARY) {
          if (level == 0) launch_gs0_boundary<T>(st_, Ld, E<T>(), dxT<T>(), A.as<T>(), Bv.as<T>(), sweeps, fwd);
          else launch_st_boundary<T>(st_, Ld, lv_[level].st<T>(), A.as<T>(), Bv.as<T>(), sweeps, fwd);
        } else {
          const T* bcm = level == 0 ? colour_major_b<T>(Bv.as<T>()) : nullptr;
          if (level == 0) launch_gs0_sweep<T>(st_, Ld, E<T>(), dxT<T>(), A.as<T>(), Bv.as<T>(), fwd, bcm);
          else launch_st_sweep<T>(st_, Ld, lv_[level].st<T>(), A.as<T>(), Bv.as<T>(), fwd);
        }
        get(A.as<T>(), nb);
        break;
      }
      case SPG_OP_RESTRICT: {
        if (level < 1) throw SpgError(SPG_E_INVALID, "restriction targets level >= 1");
        put(A, in, lv_[level - 1].d.nb);
        O.alloc(nb * 192 * sizeof(T));
        launch_restrict<T>(st_, lv_[level].d, A.as<T>(), O.as<T>());
        get(O.as<T>(), nb);
        break;
      }
      case SPG_OP_PROLONGATE: {
        if (level + 1 >= lay_.nlev) throw SpgError(SPG_E_INVALID, "prolongation needs a coarser level");
        put(A, in, lv_[level + 1].d.nb);
        put(Bv, b, nb);
        launch_prolongate<T>(st_, lv_[level].d, A.as<T>(), Bv.as<T>());
        get(Bv.as<T>(), nb);
        break;
      }
      case SPG_OP_STENCIL_RES: {
        if (!lay_.lv[level].is_explicit) throw SpgError(SPG_E_INVALID, "level has no stencils");
        put(A, in, nb);
        put(Bv, b, nb);
        O.alloc(nb * 192 * sizeof(T));
        launch_st_residual<T>(st_, lv_[level].d, lv_[level].st<T>(), A.as<T>(), Bv.as<T>(), O.as<T>());
        get(O.as<T>(), nb);
        break;
      }
      case SPG_OP_VCYCLE: {
        put(Bv, b, lv_[0].d.nb);
        O.alloc(lv_[0].n3 * sizeof(T));
        vcycle<T>(Bv.as<T>(), O.as<T>());
        get(O.as<T>(), lv_[0].d.nb);
        break;
      }
      case SPG_OP_BOTTOM: {
        const int B = lay_.nlev - 1;
        if (level != B) throw SpgError(SPG_E_INVALID, "bottom solve lives on the last level");
        put(Bv, b, nb);
        O.alloc(nb * 192 * sizeof(T));
        bottom<T>(Bv.as<T>(), O.as<T>());
        get(O.as<T>(), nb);
        break;
      }
      default:
        throw SpgError(SPG_E_INVALID, "unknown op");
    }
  };
  if (precision == 1) body(double());
  else body(float());
  check_flow();
}

void Solver::level_stencils(int level, double* out) {
  if (level < 0 || level >= lay_.nlev || !lay_.lv[level].is_explicit)
    throw SpgError(SPG_E_INVALID, "level has no stencils");
  const int64_t nb = lv_[level].d.nb;
  std::vector<double> v(nb * 243 * 64);
  sync();
  HIPCHK(hipMemcpy(v.data(), lv_[level].st64.p, v.size() * 8, hipMemcpyDeviceToHost));
  for (int64_t b = 0; b < nb; ++b)
    for (int e = 0; e < 243; ++e)
      for (int l = 0; l < 64; ++l) out[(b * 64 + l) * 243 + e] = v[st_index(b, l, e)];
}

double Solver::bench_apply(int precision, int reps) {
  activate();
  const LevelRT& R0 = lv_[0];
  hipEvent_t a, b;
  HIPCHK(hipEventCreate(&a));
  HIPCHK(hipEventCreate(&b));
  float ms = 0.f;
  if (precision == 1) {
    launch_copy<double>(st_, u_.as<double>(), x64_.as<double>(), R0.n3);
    launch_apply<double>(st_, R0.d, E<double>(), cfg_.dx, x64_.as<double>(), nullptr, q64_.as<double>(), 2);
    HIPCHK(hipEventRecord(a, st_));
    for (int i = 0; i < reps; ++i)
      launch_apply<double>(st_, R0.d, E<double>(), cfg_.dx, x64_.as<double>(), nullptr, q64_.as<double>(), 2);
    HIPCHK(hipEventRecord(b, st_));
  } else {
    launch_cast_d2f(st_, u_.as<double>(), x32_.as<float>(), R0.n3);
    launch_apply<float>(st_, R0.d, E<float>(), (float)cfg_.dx, x32_.as<float>(), nullptr, q32_.as<float>(), 2);
    HIPCHK(hipEventRecord(a, st_));
    for (int i = 0; i < reps; ++i)
      launch_apply<float>(st_, R0.d, E<float>(), (float)cfg_.dx, x32_.as<float>(), nullptr, q32_.as<float>(), 2);
    HIPCHK(hipEventRecord(b, st_));
  }
  HIPCHK(hipEventSynchronize(b));
  HIPCHK(hipEventElapsedTime(&ms, a, b));
  (void)hipEventDestroy(a);
  (void)hipEventDestroy(b);
  return (double)ms * 1e-3 / reps;
}

double Solver::bench_kernel(int op, int level, int precision, int arg, int reps) {
  activate();
  if (level < 0 || level >= lay_.nlev) throw SpgError(SPG_E_INVALID, "level out of range");
  const int B = lay_.nlev - 1;
  const FlowLease lease(*this, precision, true);
  hipEvent_t e0, e1;
  HIPCHK(hipEventCreate(&e0));
  HIPCHK(hipEventCreate(&e1));
  float ms = 0.f;
  auto body = [&](auto tag) {
    using T = decltype(tag);
    const LevelRT& R = lv_[level];
    T* u = R.u<T>();
    T* b = R.b<T>();
    T* r = R.r<T>();
    launch_zero<T>(st_, u, R.n3);
    launch_zero<T>(st_, b, R.n3);
    auto run = [&] {
      switch (op) {
        case SPG_OP_APPLY:
        case SPG_OP_RESIDUAL:
          if (level != 0) throw SpgError(SPG_E_INVALID, "apply is a level-0 operator");
          launch_apply<T>(st_, R.d, E<T>(), dxT<T>(), u, b, r, op == SPG_OP_APPLY ? 2 : 1);
          break;
        case SPG_OP_GS_SWEEP: {
          if (level != 0 && !lay_.lv[level].is_explicit) throw SpgError(SPG_E_INVALID, "level has no smoother");
          const T* bcm = level == 0 ? colour_major_b<T>(b) : nullptr;
          if (level == 0) launch_gs0_sweep<T>(st_, R.d, E<T>(), dxT<T>(), u, b, true, bcm);
          else launch_st_sweep<T>(st_, R.d, R.st<T>(), u, b, true);
          break;
        }
        case SPG_OP_GS_BOUNDARY:
          if (level == 0) launch_gs0_boundary<T>(st_, R.d, E<T>(), dxT<T>(), u, b, arg, true);
          else if (lay_.lv[level].is_explicit) launch_st_boundary<T>(st_, R.d, R.st<T>(), u, b, arg, true);
          else throw SpgError(SPG_E_INVALID, "level has no smoother");
          break;
        case SPG_OP_RESTRICT:
          if (level < 1) throw SpgError(SPG_E_INVALID, "restriction targets level >= 1");
          launch_restrict<T>(st_, R.d, lv_[level - 1].r<T>(), b);
          break;
        case SPG_OP_PROLONGATE:
          if (level >= B) throw SpgError(SPG_E_INVALID, "prolongation needs a coarser level");
          launch_prolongate<T>(st_, R.d, lv_[level + 1].u<T>(), u);
          break;
        case SPG_OP_STENCIL_RES:
          if (!lay_.lv[level].is_explicit) throw SpgError(SPG_E_INVALID, "level has no stencils");
          launch_st_residual<T>(st_, R.d, R.st<T>(), u, b, r);
          break;
        case SPG_OP_VCYCLE:
          vcycle<T>(lv_[0].b<T>(), lv_[0].r<T>());
          break;
        case SPG_OP_BOTTOM:
          if (level != B) throw SpgError(SPG_E_INVALID, "bottom solve lives on the last level");
          bottom<T>(b, u);
          break;
        default:
          throw SpgError(SPG_E_INVALID, "unknown op");
      }
    };
    run();  // warm
    HIPCHK(hipEventRecord(e0, st_));
    for (int i = 0; i < reps; ++i) run();
    HIPCHK(hipEventRecord(e1, st_));
  };
  if (precision == 1) body(double());
  else body(float());
  HIPCHK(hipEventSynchronize(e1));
  HIPCHK(hipEventElapsedTime(&ms, e0, e1));
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  check_flow();
  return (double)ms * 1e-3 / reps;
}

template void Solver::vcycle<float>(const float*, float*, bool, Part);
template void Solver::vcycle<double>(const double*, double*, bool, Part);

}  // namespace spg
