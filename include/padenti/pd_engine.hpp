// Engine of the gfx950 random-forest hot path: trainer (level loop,
// slicing, node update, routing) and forest predictor, templated on the
// feature functor.  Included by the library's C ABI (pd_capi.hip) for the
// built-in hooks and by a user's hipcc-compiled translation unit for a
// custom hook (pd_plugin.hpp).
//
// Reference: src/padenti/cl_tree_trainer_impl.hpp:203-255 (level loop),
// cl_tree_trainer_impl_init.hpp:24-365 (init, frontier),
// cl_tree_trainer_impl_traverse_ts.hpp:59-704 (traversal + accumulation),
// cl_tree_trainer_impl_learn_best_featthr.hpp:25-283 (split + node update),
// cl_classifier_impl.hpp:41-557 (classifier).
#pragma once
#include "../padenti_hip.h"
#include "pd_placement.hpp"
#include "pd_kernels.hpp"
#include "pd_runtime.hpp"

#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <chrono>
#include <cfloat>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <future>
#include <map>
#include <memory>
#include <new>
#include <stdexcept>
#include <string>
#include <system_error>
#include <vector>

#pragma clang fp contract(off)

// A translation unit may define PD_KERNEL_SET_LIGHT to 1 before including
// this header (feature plugins that instantiate many hooks): the histogram
// kernel is then compiled for two threshold buckets (16 and 64; a larger
// bucket pads with thresholds no finite response exceeds) and one block size
// (8 waves, launch tuning is ignored), and prediction for two class buckets.
#ifndef PD_KERNEL_SET_LIGHT
#define PD_KERNEL_SET_LIGHT 0
#endif

namespace pd {
namespace engine {

// FP64 gain of a split (the FP64 host oracle of the chosen split's gain).
inline double gain_f64(const uint32_t *left, const uint32_t *tot, uint32_t nC)
{
  double nL = 0, nR = 0;
  for (uint32_t l = 0; l < nC; l++) {
    nL += left[l];
    nR += (double)(tot[l] - left[l]);
  }
  const double N = nL + nR;
  double h = 0, hL = 0, hR = 0;
  for (uint32_t l = 0; l < nC; l++) {
    double p = tot[l] / N;
    if (p > 1e-6) h -= p * std::log2(p);
    p = nL > 0 ? left[l] / nL : 0.0;
    if (p > 1e-6) hL -= p * std::log2(p);
    p = nR > 0 ? (tot[l] - left[l]) / nR : 0.0;
    if (p > 1e-6) hR -= p * std::log2(p);
  }
  return h - (nL / N * hL + nR / N * hR);
}

// compiled threshold-count buckets of the histogram kernel (exact for the
// common 10 / 20 / 32; a larger bucket pads with thresholds no finite
// response exceeds)
inline int n_thr_bucket(uint32_t nT)
{
  static const int buckets[] = {1, 8, 10, 16, 20, 24, 32, 48, 64};
  for (int b : buckets)
    if (nT <= (uint32_t)b) return b;
  return 64;
}

template <class F>
Bounds<F> make_bounds(const pd_train_params &P)
{
  using T = typename F::FeatType;
  Bounds<F> b;
  for (int j = 0; j < F::FeatDim; j++) {
    b.lo[j] = (T)P.feat_low[j];
    b.hi[j] = (T)P.feat_up[j];
  }
  b.tlo = (T)P.thr_low;
  b.thi = (T)P.thr_up;
  return b;
}

// Zeros to host memory that usually holds them already (a new tree's arrays):
// pages that were never written are only read, which maps no memory to them.
inline void zero_fill(void *p, size_t bytes)
{
  static const char zeros[4096] = {};
  for (char *c = (char *)p, *e = c + bytes; c < e; c += sizeof(zeros)) {
    const size_t n = std::min<size_t>(sizeof(zeros), e - c);
    if (std::memcmp(c, zeros, n)) std::memset(c, 0, n);
  }
}

// Every candidate drawn from the bounds may take the hook's fast form: its
// offset parameters (the first four) lie in [lo, hi], so within RECIP_MAX.
template <class F>
bool fast_bounds(const Bounds<F> &b)
{
  if constexpr (has_fast<F>::value) {
    for (int j = 0; j < 4; j++)
      if (!(std::fabs((float)b.lo[j]) <= RECIP_MAX && std::fabs((float)b.hi[j]) <= RECIP_MAX)) return false;
    return true;
  } else {
    return false;
  }
}

inline void check_params(const pd_train_params &P, int fd, bool is_short)
{
  require(P.n_features >= 1, "n_features must be >= 1");
  require(P.n_thresholds >= 1 && P.n_thresholds <= 64, "n_thresholds must be in [1, 64]");
  if (is_short) {
    for (int j = 0; j < fd; j++)
      require(P.feat_low[j] >= -32768 && P.feat_up[j] <= 32767 && P.feat_up[j] - P.feat_low[j] <= 32767,
              "short feature bounds out of range");
    require(P.thr_low >= -32768 && P.thr_up <= 32767 && P.thr_up - P.thr_low <= 32767,
            "short threshold bounds out of range");
  }
}

// ---------------------------------------------------------------------------
// Split-proposal network (host side of pd_mlp.hpp)
// ---------------------------------------------------------------------------
struct SplitMix {
  uint64_t s;
  explicit SplitMix(uint64_t seed) : s(seed) {}
  uint64_t next()
  {
    uint64_t z = (s += 0x9e3779b97f4a7c15ull);
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
  }
  double uni() { return (double)(next() >> 11) * 0x1p-53; }
};

struct MlpNet {
  int device = 0;
  hipStream_t stream = nullptr;
  DevBuf theta, m, v, part, gbuf, lbuf;
  DevBuf W1, W2, W2T, W3, W3T, w4;
  DevBuf Xb, tb, yb, G, HT, DZT, dy, lossp, lsteps, perm, Xs, ys;   // G: saved BF16 GELU derivatives
  uint32_t ldb = 0;   // batch stride of the training buffers (multiple of SPLIT)
  uint64_t t_step = 0;
  uint32_t n_xcc = 1;   // XCDs of the device (weight-gradient tiles are grouped per XCD)
  PinnedStage stage;    // parameter transfers

  MlpNet(int dev, uint64_t seed)
  {
    device = dev;
    set_device(device);
    HIPCHK(hipStreamCreate(&stream));
    int xcc = 1;
    if (hipDeviceGetAttribute(&xcc, hipDeviceAttributeNumberOfXccs, device) != hipSuccess || xcc < 1) {
      (void)hipGetLastError();
      xcc = 1;
    }
    n_xcc = (uint32_t)xcc;
    theta.ensure(mlp::NPARAM * sizeof(float));
    m.ensure(mlp::NPARAM * sizeof(float));
    v.ensure(mlp::NPARAM * sizeof(float));
    gbuf.ensure(mlp::NPARAM * sizeof(float));
    lbuf.ensure(sizeof(float));
    W1.ensure(mlp::HID * mlp::INP * 2);
    W2.ensure(mlp::HID * mlp::HID * 2);
    W2T.ensure(mlp::HID * mlp::HID * 2);
    W3.ensure(mlp::HID * mlp::HID * 2);
    W3T.ensure(mlp::HID * mlp::HID * 2);
    w4.ensure(mlp::HID * 2);
    init(seed);
  }
  ~MlpNet()
  {
    if (stream) (void)hipStreamDestroy(stream);
  }
  mlp::Weights weights() const
  {
    return mlp::Weights{W1.as<uint16_t>(), W2.as<uint16_t>(),  W3.as<uint16_t>(), W2T.as<uint16_t>(),
                        W3T.as<uint16_t>(), w4.as<uint16_t>(), theta.as<float>()};
  }
  // weights U(-1/sqrt(fan_in), 1/sqrt(fan_in)), biases 0
  void init(uint64_t seed)
  {
    std::vector<float> h(mlp::NPARAM, 0.0f);
    SplitMix r(seed ^ 0x6d6c7001ull);
    auto fill = [&](int off, int n, int fan_in) {
      const double a = 1.0 / std::sqrt((double)fan_in);
      for (int i = 0; i < n; i++) h[off + i] = (float)((2.0 * r.uni() - 1.0) * a);
    };
    fill(mlp::OFF_W1, mlp::HID * mlp::IN, mlp::IN);
    fill(mlp::OFF_W2, mlp::HID * mlp::HID, mlp::HID);
    fill(mlp::OFF_W3, mlp::HID * mlp::HID, mlp::HID);
    fill(mlp::OFF_W4, mlp::HID, mlp::HID);
    set_params(h.data());
  }
  void pack()
  {
    hipLaunchKernelGGL(mlp::k_mlp_pack, dim3(mlp::HID * mlp::HID / 256), dim3(256), 0, stream, theta.as<float>(),
                       W1.as<uint16_t>(), W2.as<uint16_t>(), W2T.as<uint16_t>(), W3.as<uint16_t>(),
                       W3T.as<uint16_t>(), w4.as<uint16_t>(), m.as<float>(), v.as<float>());
    HIPCHK(hipGetLastError());
  }
  // new parameters; the Adam state restarts (through pinned memory)
  void set_params(const float *h)
  {
    set_device(device);
    const size_t bytes = mlp::NPARAM * sizeof(float);
    HIPCHK(hipMemcpyAsync(theta.p, stage.put(h, bytes), bytes, hipMemcpyHostToDevice, stream));
    t_step = 0;
    pack();
    HIPCHK(hipStreamSynchronize(stream));
    stage.reset();
  }
  void get_params(float *h)
  {
    set_device(device);
    const size_t bytes = mlp::NPARAM * sizeof(float);
    const char *pin = (const char *)stage.alloc(bytes);
    HIPCHK(hipMemcpyAsync((void *)pin, theta.p, bytes, hipMemcpyDeviceToHost, stream));
    HIPCHK(hipStreamSynchronize(stream));
    std::copy(pin, pin + bytes, (char *)h);
    stage.reset();
  }
  void ensure_batch(uint32_t B)
  {
    require(B <= (1u << 20), "batch of more than 1048576 rows");   // the weight gradient's buffer loads assume it
    const uint32_t l = (std::max<uint32_t>(B, 1u) + mlp::SPLIT - 1) / mlp::SPLIT * mlp::SPLIT;
    if (l <= ldb) return;
    ldb = l;
    Xb.ensure((size_t)ldb * mlp::INP * 2);
    tb.ensure((size_t)ldb * 4);
    yb.ensure((size_t)ldb * 4);
    G.ensure((size_t)3 * ldb * mlp::HID * 2);
    HT.ensure((size_t)4 * mlp::HID * ldb * 2);
    DZT.ensure((size_t)3 * mlp::HID * ldb * 2);
    dy.ensure((size_t)ldb * 4);
    lossp.ensure((size_t)(ldb / mlp::ROWS_SMALL) * 4);
    part.ensure((size_t)(ldb / mlp::SPLIT) * mlp::NPARAM * 4);
  }
  // inference on device rows (bf16 [n][32]) on stream s
  void forward(const uint16_t *X, uint64_t n, float *y, hipStream_t s)
  {
    const uint64_t blocks = (n + mlp::FWD_ROWS - 1) / mlp::FWD_ROWS;
    require(blocks < (1ull << 31), "too many rows");
    if (!blocks) return;
    hipLaunchKernelGGL((mlp::k_mlp_fwd<mlp::RowsMem, false>), dim3((uint32_t)blocks), dim3(mlp::THREADS), 0, s,
                       mlp::RowsMem{X, (uint32_t)n}, (uint32_t)n, weights(), y, (uint16_t *)nullptr,
                       (uint16_t *)nullptr, 0u);
    HIPCHK(hipGetLastError());
  }
  // one step on the n rows staged in Xb / tb: forward, backward, gradient
  // partials; then Adam (update) and/or the summed gradient into grad_out;
  // the step's mean squared error into loss_out (device pointers, may be null)
  void step(uint32_t n, bool update, const pd_adam &opt, float *grad_out, float *loss_out)
  {
    step(Xb.as<uint16_t>(), tb.as<float>(), nullptr, n, update, opt, grad_out, loss_out);
  }
  // the same on the rows perm[0 .. n) of X / t
  void step(const uint16_t *X, const float *t, const uint32_t *rows, uint32_t n, bool update, const pd_adam &opt,
            float *grad_out, float *loss_out)
  {
    require(n >= 1 && n <= ldb, "batch larger than the staged buffers");
    const uint32_t lrow = (n + mlp::SPLIT - 1) / mlp::SPLIT * mlp::SPLIT;
    // rows per weight-gradient partial: SPLIT doubled while it divides the
    // batch, leaves at least 32 partials (blocks enough for the chip) and
    // stays at most 4096 rows -- fewer partials to write and sum in Adam
    uint32_t split = mlp::SPLIT;
    while (split < 4096u && lrow % (2u * split) == 0 && lrow / (2u * split) >= 32u) split *= 2u;
    // 128-row backward tiles and 64 x 64 weight-gradient tiles halve the L2
    // re-reads of the weights and activations, once the batch gives both
    // grids blocks enough for the chip
    const bool big = lrow >= mlp::BIG_BATCH;
    const bool mid = lrow >= mlp::MID_BATCH;
    const uint32_t nblk = lrow / (big ? mlp::ROWS_BIG : (mid ? mlp::ROWS : mlp::ROWS_SMALL)), ns = lrow / split;
    const mlp::Weights w = weights();
    uint16_t *ht = HT.as<uint16_t>(), *dz = DZT.as<uint16_t>();
    const size_t hl = (size_t)mlp::HID * ldb;   // one layer of HT / DZT
    // forward row tile: 128 rows (half the weight re-reads of 64) once the
    // batch fills the chip with them, else 64 or 32 rows for more blocks
    const uint32_t fr = big ? 128u : (mid ? 64u : 32u);
    const mlp::RowsPerm src{X, rows, n};
    if (fr == 128u)
      hipLaunchKernelGGL((mlp::k_mlp_fwd<mlp::RowsPerm, true, 128>), dim3(lrow / 128u), dim3(mlp::THREADS), 0, stream,
                         src, n, w, yb.as<float>(), G.as<uint16_t>(), ht, ldb);
    else if (fr == 64u)
      hipLaunchKernelGGL((mlp::k_mlp_fwd<mlp::RowsPerm, true, 64>), dim3(lrow / 64u), dim3(mlp::THREADS), 0, stream,
                         src, n, w, yb.as<float>(), G.as<uint16_t>(), ht, ldb);
    else
      hipLaunchKernelGGL((mlp::k_mlp_fwd<mlp::RowsPerm, true, 32>), dim3(lrow / 32u), dim3(mlp::THREADS), 0, stream,
                         src, n, w, yb.as<float>(), G.as<uint16_t>(), ht, ldb);
    HIPCHK(hipGetLastError());
    if (big)
      hipLaunchKernelGGL(mlp::k_mlp_bwd<mlp::ROWS_BIG>, dim3(nblk), dim3(mlp::THREADS), 0, stream, yb.as<float>(),
                         t, rows, n, 1.0f / (float)n, G.as<uint16_t>(), w, dz, dy.as<float>(),
                         lossp.as<float>(), ldb);
    else if (mid)
      hipLaunchKernelGGL(mlp::k_mlp_bwd<mlp::ROWS>, dim3(nblk), dim3(mlp::THREADS), 0, stream, yb.as<float>(),
                         t, rows, n, 1.0f / (float)n, G.as<uint16_t>(), w, dz, dy.as<float>(),
                         lossp.as<float>(), ldb);
    else
      hipLaunchKernelGGL(mlp::k_mlp_bwd<mlp::ROWS_SMALL>, dim3(nblk), dim3(mlp::THREADS), 0, stream, yb.as<float>(),
                         t, rows, n, 1.0f / (float)n, G.as<uint16_t>(), w, dz, dy.as<float>(),
                         lossp.as<float>(), ldb);
    HIPCHK(hipGetLastError());
    float *pt = part.as<float>();
    if (big) {
      // layer 1's 64 x 32 tiles (grid row 0) and the output layer's partials
      // (rows 1 .. 5: 17 groups of 4 blocks per row)
      hipLaunchKernelGGL(mlp::k_mlp_wgrad, dim3(4, 1 + 5, ns), dim3(mlp::THREADS), 0, stream, dz, ht, ldb,
                         (uint32_t)mlp::IN, split, pt, (size_t)mlp::NPARAM, (size_t)0, (uint32_t)mlp::OFF_W1,
                         (uint32_t)mlp::OFF_B1, ht + 3 * hl, dy.as<float>(), 1u);
      HIPCHK(hipGetLastError());
      for (int l = 1; l <= 2; l++) {
        hipLaunchKernelGGL(mlp::k_mlp_wgrad64, dim3((mlp::HID / 64) * (mlp::HID / 64) * ns), dim3(mlp::THREADS), 0,
                           stream, dz + l * hl, ht + l * hl, ldb, (uint32_t)mlp::HID, split, ns, n_xcc, pt,
                           (size_t)mlp::NPARAM, (uint32_t)(l == 1 ? mlp::OFF_W2 : mlp::OFF_W3),
                           (uint32_t)(l == 1 ? mlp::OFF_B2 : mlp::OFF_B3));
        HIPCHK(hipGetLastError());
      }
    } else {
      // the three layers' 64 x 32 tiles (grid rows 0 .. 16) and the output
      // layer's partials (rows 17 .. 21) in one launch
      const uint32_t wy = 1 + 2 * mlp::HID / 32;
      hipLaunchKernelGGL(mlp::k_mlp_wgrad, dim3(4, wy + 5, ns), dim3(mlp::THREADS), 0, stream, dz, ht, ldb, 0u, split,
                         pt, (size_t)mlp::NPARAM, hl, 0u, 0u, ht + 3 * hl, dy.as<float>(), wy);
      HIPCHK(hipGetLastError());
    }
    float c1 = 1.0f, c2 = 1.0f;
    if (update) {
      t_step++;
      c1 = (float)(1.0 / (1.0 - std::pow((double)opt.beta1, (double)t_step)));
      c2 = (float)(1.0 / (1.0 - std::pow((double)opt.beta2, (double)t_step)));
    }
    // Adam, the BF16 weight copies and the step's loss in one launch
    const mlp::Packed pk{W1.as<uint16_t>(), W2.as<uint16_t>(), W2T.as<uint16_t>(),
                         W3.as<uint16_t>(), W3T.as<uint16_t>(), w4.as<uint16_t>()};
    hipLaunchKernelGGL(mlp::k_mlp_adam, dim3((mlp::NPARAM + 255) / 256), dim3(256), 0, stream, theta.as<float>(),
                       m.as<float>(), v.as<float>(), pt, ns, (size_t)mlp::NPARAM, grad_out, update ? 1 : 0, opt.lr,
                       opt.beta1, opt.beta2, opt.eps, c1, c2, pk, lossp.as<float>(), nblk, 1.0f / (float)n,
                       loss_out);
    HIPCHK(hipGetLastError());
  }
  // host rows (FP32 [n][32]) -> bf16 rows [n][32]
  static void encode(const float *x, uint64_t n, uint16_t *out)
  {
    for (uint64_t r = 0; r < n; r++)
      for (int k = 0; k < mlp::INP; k++) out[r * mlp::INP + k] = k < mlp::IN ? mlp::f2bf(x[r * mlp::IN + k]) : 0;
  }
  void stage_host(const float *x, const float *t, uint32_t n)
  {
    ensure_batch(n);
    std::vector<uint16_t> xb((size_t)ldb * mlp::INP, 0);
    std::vector<float> tv(ldb, 0.0f);
    encode(x, n, xb.data());
    if (t) std::copy(t, t + n, tv.begin());
    HIPCHK(hipMemcpyAsync(Xb.p, xb.data(), xb.size() * 2, hipMemcpyHostToDevice, stream));
    HIPCHK(hipMemcpyAsync(tb.p, tv.data(), tv.size() * 4, hipMemcpyHostToDevice, stream));
  }
  // training loop over device records X (bf16 [N][32]) / t (FP32 [N]):
  // `epochs` passes, each over a fresh permutation (SplitMix64 Fisher-Yates
  // of seed, epoch), batches of B rows (the last one shorter)
  void train(const uint16_t *X, const float *t, uint64_t N, uint32_t B, uint32_t epochs, const pd_adam &opt,
             uint64_t seed, float *epoch_loss, float *ms)
  {
    require(X && t && N >= 1 && N < (1ull << 32) && B >= 1 && B <= (1u << 20) && epochs >= 1,
            "bad training arguments");
    set_device(device);
    ensure_batch(B);
    const uint64_t steps = (N + B - 1) / B;
    perm.ensure(N * sizeof(uint32_t));
    lsteps.ensure(steps * sizeof(float));
    std::vector<uint32_t> p(N);
    std::vector<float> ls(steps);
    Event e0, e1;
    double total_ms = 0.0;
    for (uint32_t ep = 0; ep < epochs; ep++) {
      for (uint64_t i = 0; i < N; i++) p[i] = (uint32_t)i;
      SplitMix r(seed * 0x9e3779b97f4a7c15ull + ep + 1);
      for (uint64_t i = N - 1; i > 0; i--) std::swap(p[i], p[r.next() % (i + 1)]);
      HIPCHK(hipMemcpyAsync(perm.p, p.data(), N * sizeof(uint32_t), hipMemcpyHostToDevice, stream));
      HIPCHK(hipEventRecord(e0.e, stream));
      for (uint64_t sidx = 0; sidx < steps; sidx++) {
        const uint64_t base = sidx * B;
        const uint32_t cnt = (uint32_t)std::min<uint64_t>(B, N - base);
        step(X, t, perm.as<uint32_t>() + base, cnt, true, opt, nullptr, lsteps.as<float>() + sidx);
      }
      HIPCHK(hipEventRecord(e1.e, stream));
      HIPCHK(hipMemcpyAsync(ls.data(), lsteps.p, steps * sizeof(float), hipMemcpyDeviceToHost, stream));
      HIPCHK(hipStreamSynchronize(stream));
      total_ms += elapsed_ms(e0, e1);
      double acc = 0.0;
      for (uint64_t sidx = 0; sidx < steps; sidx++)
        acc += (double)ls[sidx] * (double)std::min<uint64_t>(B, N - sidx * B);
      if (epoch_loss) epoch_loss[ep] = (float)(acc / (double)N);
    }
    if (ms) *ms = (float)total_ms;
  }
};

// ---------------------------------------------------------------------------
// Trainer
// ---------------------------------------------------------------------------
struct TrainerBase {
  int device = 0;
  uint32_t nC = 0;
  uint64_t hist_budget = 8ull << 30;
  uint32_t chunk = 0;
  bool probe_order = true;   // probe-coherent candidate tiles (functors with kProbeRowA/B)
  bool wide_bins = true;     // one 32-bit histogram bin per rank where it fits (WIDE_LDS_MAX)
  // candidate table per histogram slice (k_cand_table), where it fits the budget
  bool cand_table = true;
  uint64_t cand_table_budget = 16ull << 30;
  pd_tuning tune{8u, 16u, 1u, 0u};   // waves per histogram block, target blocks per CU, samples per wave step, bins
  std::vector<pd_tuning_rule> tune_rules;   // per level, by samples per node (decreasing)
  pd_tuning level_tuning(uint64_t active, uint32_t trainable) const
  {
    const uint64_t spn = trainable ? active / trainable : active;
    for (const pd_tuning_rule &r : tune_rules)
      if (spn >= r.min_samples_per_node) return r.tuning;
    return tune;
  }
  hipStream_t stream = nullptr;
  // record sink of the plain trainer (device rows bf16 [cap][32], gains [cap])
  uint16_t *sink_x = nullptr;
  float *sink_t = nullptr;
  float *sink_rel = nullptr;
  uint64_t sink_cap = 0, sink_n = 0;
  uint32_t sink_R = 0;
  // split proposal (PD_MODE_PROPOSAL)
  MlpNet *prop_mlp = nullptr;
  uint32_t prop_keep = 0, prop_screen = 0, prop_min = 0;
  uint32_t prop_refine = 0, prop_refine_min = 0;   // subsample stride (0: off), smallest subsample
  // refinement subsample: 0 every stride-th record (exact subsample gains),
  // 1 class-stratified (estimated node gains), 2 class-stratified ranked by
  // the estimate plus the network's correction from the subsample statistics
  int prop_strata = 0;
  uint32_t prop_corr_rows = 0;   // mode 2: candidates per node the network corrects (0: every screened one)
  int xcd_by_position = 0;   // XCD placement of histogram work items (see xcd_order)
  int prop_judge = 0;
  virtual ~TrainerBase()
  {
    if (stream) (void)hipStreamDestroy(stream);
  }
  virtual void set_data(uint32_t n_images, const void *pixels, const uint64_t *img_off, const uint32_t *widths,
                        const uint32_t *heights, const uint8_t *labels, const uint64_t *lab_off,
                        const uint32_t *samples, const uint64_t *samp_off, const uint32_t *n_samples) = 0;
  virtual void train(const pd_train_params &P, uint32_t tree_id, uint32_t depth, uint32_t end_depth, int mode,
                     const float *prior, int32_t *left, void *feats, void *thrs, float *post, uint32_t *node_k,
                     float *node_gain, double *node_gain64, pd_level_stats *ls) = 0;
  virtual void hist_nodes(const pd_train_params &P, uint32_t tree_id, uint32_t n_nodes, const int32_t *nodes,
                          const int32_t *sample_node, uint32_t *H_out) = 0;
  virtual double time_level(const pd_train_params &P, uint32_t tree_id, uint32_t n_nodes, int reps) = 0;
};

struct SlotInfo {
  int32_t node;
  uint32_t begin, count;
  bool trainable;  // count > perLeafSamplesThr (the consumer gate)
};

template <class F>
struct Trainer final : TrainerBase {
  using T = typename F::FeatType;
  using I = typename F::ImgType;
  static constexpr int FD = F::FeatDim;

  // training set
  uint32_t n_images = 0;
  uint64_t S = 0;
  std::vector<uint4> h_recs;
  std::vector<uint32_t> root_tot;
  DevBuf d_pixels, d_imgs, d_recs;
  // level state
  DevBuf d_actA, d_actB, d_slotA, d_slotB;
  DevBuf d_H, d_out;
  DevBuf d_cand_key, d_cand_left;
  // a histogram slice's host tables on the device (one upload, see hist_slice)
  struct SliceTables {
    HistItem *items;              // work items in launch order
    int32_t *slot_node;           // [ns]
    int32_t *slot_hidx;           // [ns] H block of the slot, -1: searched in the kernel
    uint8_t *slot_mode;           // [ns]
    uint32_t *tot;                // [ns][nC]
    float *slot_h;                // [ns] node entropy
    uint32_t *zero;               // H blocks that several items add into
    uint32_t *hlist;              // slot of each H block
    unsigned long long *best;     // [ns] split keys, uploaded as zeros
  } sl{};
  DevBuf d_slice, d_route;
  DevBuf d_tleft, d_tfeat, d_tthr, d_ccount;
  DevBuf d_flags, d_rank, d_scan_tmp;
  // auto-context hooks: node-id maps of every image (two buffers), the
  // pixels that are routed (labelled), map offsets, the tree's posteriors
  DevBuf d_acmapA, d_acmapB, d_acsel, d_acoff, d_acblk, d_tpost;
  uint64_t ac_px = 0;
  uint32_t ac_blocks = 0;
  AcArgs ac{};
  uint32_t cu_count = 256;
  uint32_t n_xcc = 1;
  size_t lds_limit = 65536;
  // candidate map of the histogram launch in flight (proposal slices)
  const uint32_t *d_map_cur = nullptr;
  DevBuf d_perm;
  const uint16_t *d_perm_cur = nullptr;   // [slice slot][nF] candidate order of the current launch
  DevBuf d_ctab;
  const T *d_ctab_cur = nullptr;   // candidate table of the current launch (k_cand_table), or none
  PinnedStage stage;   // per-level transfers; reset after every stream synchronization

  void h2d(void *dst, const void *src, size_t bytes)
  {
    if (!bytes) return;
    HIPCHK(hipMemcpyAsync(dst, stage.put(src, bytes), bytes, hipMemcpyHostToDevice, stream));
  }
  // device -> host, synchronizing the stream (which also retires the staging)
  void d2h_sync(void *dst, const void *src, size_t bytes)
  {
    void *pin = bytes ? stage.alloc(bytes) : nullptr;
    if (bytes) HIPCHK(hipMemcpyAsync(pin, src, bytes, hipMemcpyDeviceToHost, stream));
    HIPCHK(hipStreamSynchronize(stream));
    if (bytes) std::copy((const char *)pin, (const char *)pin + bytes, (char *)dst);
    stage.reset();
  }
  // Several host arrays uploaded as one: each add() reserves a 16-byte aligned
  // piece, commit() copies the whole staging to the device buffer and at()
  // gives a piece's device address (a small copy costs about 3 us of the GPU's
  // time and as much of the host's).
  struct Upload {
    Trainer &t;
    DevBuf &dst;
    std::vector<std::pair<const void *, size_t>> src;   // source (null: left to the caller), bytes
    std::vector<size_t> off;
    size_t bytes = 0;
    char *pin = nullptr;
    size_t add(const void *p, size_t n)
    {
      src.push_back({p, n});
      off.push_back(bytes);
      bytes += (n + 15) & ~(size_t)15;
      return off.size() - 1;
    }
    // pinned staging with the sources copied in (pieces without one: host())
    void stage()
    {
      dst.grow(std::max<size_t>(bytes, 16));
      pin = (char *)t.stage.alloc(std::max<size_t>(bytes, 16));
      for (size_t i = 0; i < src.size(); i++)
        if (src[i].first && src[i].second) std::memcpy(pin + off[i], src[i].first, src[i].second);
    }
    void commit()
    {
      if (bytes) HIPCHK(hipMemcpyAsync(dst.p, pin, bytes, hipMemcpyHostToDevice, t.stream));
    }
    template <class T2>
    T2 *host(size_t i) const
    {
      return (T2 *)(pin + off[i]);
    }
    template <class T2>
    T2 *at(size_t i) const
    {
      return (T2 *)((char *)dst.p + off[i]);
    }
  };

  DevBuf d_sub_act, d_sub_idx, d_sub_cls, d_sub_sel, d_map2;
  DevBuf d_st_flags, d_st_pos, d_st_tmp, d_st_meta, d_st_rate, d_st_tot;
  DevBuf d_frac, d_gmax, d_ynet, d_score, d_score2, d_net_sel, d_full, d_gbest, d_top, d_ebase, d_eslots;
  DevBuf d_gains, d_emit_slots, d_emit_base, d_emit_best, d_emit_in, d_emit_node, d_pslot_in, d_pslot_node, d_scores,
      d_map;

  Trainer(int dev, uint32_t ncl)
  {
    device = dev;
    nC = ncl;
    set_device(device);
    HIPCHK(hipStreamCreate(&stream));
    hipDeviceProp_t prop;
    HIPCHK(hipGetDeviceProperties(&prop, device));
    cu_count = (uint32_t)prop.multiProcessorCount;
    lds_limit = prop.sharedMemPerBlock;
    int xcc = 1;
    if (hipDeviceGetAttribute(&xcc, hipDeviceAttributeNumberOfXccs, device) != hipSuccess || xcc < 1) {
      (void)hipGetLastError();
      xcc = 1;
    }
    n_xcc = (uint32_t)xcc;
  }

  // XCD-aware launch order.  Workgroup b of a launch runs on XCD b % n_xcc,
  // and each XCD has its own L2.  The items of one (slot, chunk) group (its
  // candidate tiles, which walk the same samples and so the same images)
  // are all placed on one XCD: group g -> XCD g % n_xcc, and the position
  // within that XCD's sequence is b / n_xcc.  Shorter sequences are padded
  // with NULL_SLOT items.  `group` gives the group id of every item (items
  // of a group are contiguous).
  //
  // With xcd_by_position, a group of a node cut into at least n_xcc chunks
  // instead goes to the XCD of its position in the node's sample sequence
  // (pos = (chunk + 1/2) / chunks; a node's samples run through the images
  // in order, so pos stands for an image range), and each XCD's groups run
  // in order of pos: chunks of different nodes over the same images run on
  // one XCD at about the same time and share its L2.  Other groups are
  // dealt round robin after them.
  void xcd_order(std::vector<HistItem> &items, const std::vector<uint32_t> &group_start,
                 const std::vector<float> &group_pos) const
  {
    const uint32_t X = n_xcc;
    if (X <= 1 || items.empty()) return;
    std::vector<std::vector<HistItem>> lanes(X);
    const size_t ng = group_start.size() - 1;
    if (xcd_by_position) {
      std::vector<std::pair<float, uint32_t>> placed;
      for (size_t g = 0; g < ng; g++)
        if (group_pos[g] >= 0.0f) placed.push_back({group_pos[g], (uint32_t)g});
      std::stable_sort(placed.begin(), placed.end(),
                       [](const std::pair<float, uint32_t> &a, const std::pair<float, uint32_t> &b) {
                         return a.first < b.first;
                       });
      for (const auto &pg : placed) {
        const uint32_t x = std::min<uint32_t>(X - 1, (uint32_t)(pg.first * (float)X));
        for (uint32_t i = group_start[pg.second]; i < group_start[pg.second + 1]; i++) lanes[x].push_back(items[i]);
      }
      uint32_t rr = 0;
      for (size_t g = 0; g < ng; g++) {
        if (group_pos[g] >= 0.0f) continue;
        for (uint32_t i = group_start[g]; i < group_start[g + 1]; i++) lanes[rr % X].push_back(items[i]);
        rr++;
      }
    } else {
      for (size_t g = 0; g < ng; g++)
        for (uint32_t i = group_start[g]; i < group_start[g + 1]; i++) lanes[g % X].push_back(items[i]);
    }
    size_t len = 0;
    for (auto &l : lanes) len = std::max(len, l.size());
    items.assign(len * X, HistItem{NULL_SLOT, 0u, 0u, 0u});
    for (uint32_t x = 0; x < X; x++)
      for (size_t j = 0; j < lanes[x].size(); j++) items[j * X + x] = lanes[x][j];
  }

  void set_data(uint32_t ni, const void *pixels, const uint64_t *img_off, const uint32_t *widths,
                const uint32_t *heights, const uint8_t *labels, const uint64_t *lab_off, const uint32_t *samples,
                const uint64_t *samp_off, const uint32_t *n_samples) override
  {
    require(ni >= 1 && ni < (1u << 24), "n_images must be in [1, 2^24)");
    require(pixels && img_off && widths && heights && labels && lab_off && samples && samp_off && n_samples,
            "null pointer in set_data");
    set_device(device);
    std::vector<ImgDesc> imgs(ni);
    uint64_t total_px = 0;
    for (uint32_t i = 0; i < ni; i++) {
      require(widths[i] >= 1 && widths[i] < 65536 && heights[i] >= 1 && heights[i] < 65536,
              "image size must be in [1, 65535]");
      require((uint64_t)widths[i] * heights[i] * F::nChannels * sizeof(I) < (1ull << 32),
              "an image must be smaller than 4 GiB");
      imgs[i].off = img_off[i];
      imgs[i].w = widths[i];
      imgs[i].h = heights[i];
      total_px = std::max(total_px, img_off[i] + (uint64_t)widths[i] * heights[i] * F::nChannels);
    }
    uint64_t s_total = 0;
    for (uint32_t i = 0; i < ni; i++) s_total += n_samples[i];
    require(s_total < (1ull << 32), "too many samples");
    h_recs.resize(s_total);
    root_tot.assign(nC, 0u);
    uint64_t g = 0;
    for (uint32_t i = 0; i < ni; i++) {
      const uint8_t *lab = labels + lab_off[i];
      const uint32_t *smp = samples + samp_off[i];
      const uint32_t w = widths[i], npx = widths[i] * heights[i];
      for (uint32_t s = 0; s < n_samples[i]; s++, g++) {
        const uint32_t px = smp[s];
        require(px < npx, "sample index outside its image");
        const uint32_t l = lab[px];
        require(l >= 1 && l <= nC, "sampled pixel is unlabelled or its label exceeds n_classes");
        const uint32_t c = l - 1u;
        root_tot[c]++;  // perClassTotSamples at depth 1, _traverse_ts.hpp:526
        h_recs[g] = make_uint4(i | (c << 24), (px % w) | ((px / w) << 16), 0u, 0u);
      }
    }
    d_pixels.ensure(total_px * sizeof(I));
    HIPCHK(hipMemcpy(d_pixels.p, pixels, total_px * sizeof(I), hipMemcpyHostToDevice));
    d_imgs.ensure(ni * sizeof(ImgDesc));
    HIPCHK(hipMemcpy(d_imgs.p, imgs.data(), ni * sizeof(ImgDesc), hipMemcpyHostToDevice));
    d_recs.ensure(std::max<uint64_t>(s_total, 1) * sizeof(uint4));
    if (s_total) {
      HIPCHK(hipMemcpy(d_recs.p, h_recs.data(), s_total * sizeof(uint4), hipMemcpyHostToDevice));
      // per-sample prepared state (the functor's shared per-pixel part)
      hipLaunchKernelGGL((k_prepare<F>), dim3((uint32_t)((s_total + 255) / 256)), dim3(256), 0, stream,
                         d_pixels.as<I>(), d_imgs.as<ImgDesc>(), d_recs.as<uint4>(), (uint32_t)s_total);
      HIPCHK(hipGetLastError());
      HIPCHK(hipStreamSynchronize(stream));
      HIPCHK(hipMemcpy(h_recs.data(), d_recs.p, s_total * sizeof(uint4), hipMemcpyDeviceToHost));
    }
    if constexpr (uses_context<F>::value) {
      // node maps packed back to back; routed pixels = labelled ones
      std::vector<uint64_t> moff(ni);
      std::vector<uint32_t> blk0(ni);
      uint64_t t = 0, b = 0;
      for (uint32_t i = 0; i < ni; i++) {
        moff[i] = t;
        blk0[i] = (uint32_t)b;
        const uint64_t npx = (uint64_t)widths[i] * heights[i];
        t += npx;
        b += (npx + 255) / 256;
      }
      require(b < (1ull << 31), "too many pixels for the node maps");
      std::vector<uint8_t> sel(t);
      for (uint32_t i = 0; i < ni; i++)
        std::memcpy(sel.data() + moff[i], labels + lab_off[i], (size_t)widths[i] * heights[i]);
      d_acsel.ensure(std::max<uint64_t>(t, 1));
      HIPCHK(hipMemcpy(d_acsel.p, sel.data(), t, hipMemcpyHostToDevice));
      d_acoff.ensure(ni * sizeof(uint64_t));
      HIPCHK(hipMemcpy(d_acoff.p, moff.data(), ni * sizeof(uint64_t), hipMemcpyHostToDevice));
      d_acblk.ensure(ni * sizeof(uint32_t));
      HIPCHK(hipMemcpy(d_acblk.p, blk0.data(), ni * sizeof(uint32_t), hipMemcpyHostToDevice));
      d_acmapA.ensure(std::max<uint64_t>(t, 1) * sizeof(int32_t));
      d_acmapB.ensure(std::max<uint64_t>(t, 1) * sizeof(int32_t));
      ac_px = t;
      ac_blocks = (uint32_t)b;
    }
    n_images = ni;
    S = s_total;
  }

  // Samples per wave step of the histogram launch for nT thresholds under
  // the current tuning: the requested 2 or 4 where that kernel is compiled
  // (thresholds 1, 10, 20, 32; 8 or 16 waves), else 1.
  uint32_t hist_spw(uint32_t nT) const
  {
#if PD_KERNEL_SET_LIGHT
    (void)nT;
    return 1u;
#else
    const uint32_t want = tune.samples_per_wave;
    if (want != 2u && want != 4u) return 1u;
    if (tune.waves != 8u && tune.waves != 16u) return 1u;
    const int b = n_thr_bucket(nT);
    return (b == 1 || b == 10 || b == 20 || b == 32) ? want : 1u;
#endif
  }
  // candidates per histogram tile
  uint32_t hist_fpw(uint32_t nT) const { return 64u / hist_spw(nT); }

  uint32_t pick_chunk(uint64_t level_samples, uint32_t nF, uint32_t nT, uint32_t launches = 1) const
  {
    if (chunk) return std::max<uint32_t>(64u, std::min<uint32_t>(chunk, 32768u));
    const uint32_t fpw = hist_fpw(nT);
    return item_chunk(level_samples, nF, (nF + fpw - 1) / fpw, nT, nC, (uint32_t)cu_count, tune.blocks_per_cu,
                      launches);
  }

  template <int NTP>
  void launch_hist_t(uint32_t n_items, uint32_t item_base, const uint4 *act, const Bounds<F> &bnd, uint32_t tree,
                     uint32_t nF, uint32_t nT)
  {
#if PD_KERNEL_SET_LIGHT
    launch_hist_w<NTP, 8, 1>(n_items, item_base, act, bnd, tree, nF, nT);
#else
    const uint32_t spw = hist_spw(nT);
    if constexpr (NTP == 1 || NTP == 10 || NTP == 20 || NTP == 32) {
      if (spw == 2u) {
        if (tune.waves == 16) launch_hist_w<NTP, 16, 2>(n_items, item_base, act, bnd, tree, nF, nT);
        else launch_hist_w<NTP, 8, 2>(n_items, item_base, act, bnd, tree, nF, nT);
        return;
      }
      if (spw == 4u) {
        if (tune.waves == 16) launch_hist_w<NTP, 16, 4>(n_items, item_base, act, bnd, tree, nF, nT);
        else launch_hist_w<NTP, 8, 4>(n_items, item_base, act, bnd, tree, nF, nT);
        return;
      }
    }
    if (tune.waves == 4) launch_hist_w<NTP, 4, 1>(n_items, item_base, act, bnd, tree, nF, nT);
    else if (tune.waves == 16) launch_hist_w<NTP, 16, 1>(n_items, item_base, act, bnd, tree, nF, nT);
    else launch_hist_w<NTP, 8, 1>(n_items, item_base, act, bnd, tree, nF, nT);
#endif
  }

  template <int NTP, int NW, int SPW>
  void launch_hist_w(uint32_t n_items, uint32_t item_base, const uint4 *act, const Bounds<F> &bnd, uint32_t tree,
                     uint32_t nF, uint32_t nT)
  {
#if !PD_KERNEL_SET_LIGHT
    // one 32-bit bin per rank where the tile still fits two blocks per CU
    // (tune.bins 0), or wherever it fits one block (2); 16-bit bins (1)
    if constexpr (sizeof(typename F::FeatType) == 4 && NW >= 8 && NTP <= 32) {
      const size_t wl = hist_lds_bytes<F, NTP, true, 64 / SPW>(nC);
      // (1 KiB of the block's LDS is left for the kernel's static reduction array)
      if (wide_bins && tune.bins != 1u && wl <= (tune.bins == 2u ? lds_limit - 1024u : WIDE_LDS_MAX)) {
        launch_hist_k<NTP, NW, true, SPW>(n_items, item_base, act, bnd, tree, nF, nT);
        return;
      }
    }
#endif
    launch_hist_k<NTP, NW, false, SPW>(n_items, item_base, act, bnd, tree, nF, nT);
  }

  template <int NTP, int NW, bool WIDE, int SPW>
  void launch_hist_k(uint32_t n_items, uint32_t item_base, const uint4 *act, const Bounds<F> &bnd, uint32_t tree,
                     uint32_t nF, uint32_t nT)
  {
    const size_t lds = hist_lds_bytes<F, NTP, WIDE, 64 / SPW>(nC);
    if (lds > lds_limit) throw ArgError("histogram tile needs " + std::to_string(lds) + " B of LDS");
    if (lds > 65536)
      HIPCHK(hipFuncSetAttribute((const void *)k_hist<F, NTP, NW, WIDE, SPW>,
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL((k_hist<F, NTP, NW, WIDE, SPW>), dim3(n_items), dim3(NW * 64), lds, stream, d_pixels.as<I>(),
                       d_imgs.as<ImgDesc>(), act, sl.items, item_base, sl.slot_node, sl.slot_mode, sl.slot_hidx, sl.tot,
                       sl.slot_h, bnd, tree, nF,
                       nT, nC, d_H.as<uint32_t>(), d_cand_key.as<unsigned long long>(), d_cand_left.as<uint32_t>(),
                       d_map_cur, d_perm_cur, d_ctab_cur, fast_bounds(bnd) ? 1u : 0u, ac);
    HIPCHK(hipGetLastError());
  }

  void launch_hist(uint32_t n_items, uint32_t item_base, const uint4 *act, const Bounds<F> &bnd, uint32_t tree,
                   uint32_t nF, uint32_t nT)
  {
    if (!n_items) return;
#if PD_KERNEL_SET_LIGHT
    if (nT <= 16) launch_hist_t<16>(n_items, item_base, act, bnd, tree, nF, nT);
    else launch_hist_t<64>(n_items, item_base, act, bnd, tree, nF, nT);
    return;
#endif
    switch (n_thr_bucket(nT)) {
      case 1: launch_hist_t<1>(n_items, item_base, act, bnd, tree, nF, nT); break;
      case 8: launch_hist_t<8>(n_items, item_base, act, bnd, tree, nF, nT); break;
      case 10: launch_hist_t<10>(n_items, item_base, act, bnd, tree, nF, nT); break;
      case 16: launch_hist_t<16>(n_items, item_base, act, bnd, tree, nF, nT); break;
      case 20: launch_hist_t<20>(n_items, item_base, act, bnd, tree, nF, nT); break;
      case 24: launch_hist_t<24>(n_items, item_base, act, bnd, tree, nF, nT); break;
      case 32: launch_hist_t<32>(n_items, item_base, act, bnd, tree, nF, nT); break;
      case 48: launch_hist_t<48>(n_items, item_base, act, bnd, tree, nF, nT); break;
      default: launch_hist_t<64>(n_items, item_base, act, bnd, tree, nF, nT); break;
    }
  }

  // Histogram launch(es) of the slots [s0, s1) (slice-local index q = slot -
  // s0).  With want_h every slot gets its H block (block q).  Otherwise a
  // slot whose samples fit one chunk is searched inside the kernel (fused)
  // and needs no H; a slot with several chunks adds into H block hslots-index.
  // tot: the slice's per-class node totals [q][nC].  Returns the number of
  // kernel launches; hslots receives the slots that have an H block, in
  // block order.
  uint32_t hist_slice(const std::vector<SlotInfo> &slots, size_t s0, size_t s1, const uint4 *act,
                      const pd_train_params &P, const Bounds<F> &bnd, uint32_t tree, int mode, uint32_t ch,
                      const std::vector<uint32_t> &tot, bool want_h, std::vector<uint32_t> &hslots,
                      const Event *ev_begin = nullptr, const Event *ev_end = nullptr)
  {
    const uint32_t nF = P.n_features, nT = P.n_thresholds;
    const uint32_t fpw = hist_fpw(nT);
    const uint32_t ftiles = (nF + fpw - 1) / fpw;
    const size_t per = (size_t)nC * nT * nF;
    const uint32_t ns = (uint32_t)(s1 - s0);
    std::vector<HistItem> items;
    std::vector<uint32_t> item_start(ns + 1, 0);
    std::vector<int32_t> snode(ns), shidx(ns, -1);
    std::vector<uint8_t> smode(ns, 0);
    std::vector<uint32_t> zero, group_start;
    std::vector<float> group_pos;
    // level-batched launches with balanced XCD placement: the (node, chunk)
    // groups are collected first and their items written straight into the
    // interleaved order of the launch (below; ftiles items a group in tile
    // order, NULL_SLOT padding), so the host does not build, copy and
    // re-interleave the item list per level
    const bool direct = mode == PD_MODE_LEVEL_BATCHED && n_xcc > 1 && !xcd_by_position;
    std::vector<uint4> groups;   // (slot, begin, count) of each group, in order
    hslots.clear();
    for (uint32_t q = 0; q < ns; q++) {
      const SlotInfo &si = slots[s0 + q];
      snode[q] = si.node;
      item_start[q] = (uint32_t)items.size();
      const uint32_t cnt = si.trainable ? si.count : 0u;
      const uint32_t chunks = std::max<uint32_t>(1u, (cnt + ch - 1) / ch);
      if (want_h) {
        shidx[q] = (int32_t)q;
        hslots.push_back(q);
        if (chunks > 1) {
          smode[q] = SLOT_ATOMIC;
          zero.push_back(q);
        }
      } else if (chunks == 1) {
        smode[q] = SLOT_FUSED;
      } else {
        smode[q] = SLOT_ATOMIC;
        shidx[q] = (int32_t)hslots.size();
        zero.push_back((uint32_t)hslots.size());
        hslots.push_back(q);
      }
      for (uint32_t k = 0; k < chunks; k++) {
        const uint32_t b = chunk_begin(si.begin, cnt, chunks, k);
        const uint32_t c = chunk_begin(si.begin, cnt, chunks, k + 1) - b;
        if (direct) {
          groups.push_back(uint4{q, b, c, 0u});
          continue;
        }
        group_start.push_back((uint32_t)items.size());
        group_pos.push_back(chunks >= n_xcc ? ((float)k + 0.5f) / (float)chunks : -1.0f);
        for (uint32_t ft = 0; ft < ftiles; ft++) items.push_back(HistItem{q, b, c, ft});
      }
    }
    // direct: the items are written into pinned staging and copied from there
    size_t n_items = 0;
    GroupOrder deal;   // (direct)
    if (direct) {
      std::vector<uint32_t> sizes(groups.size());
      for (size_t g = 0; g < groups.size(); g++) sizes[g] = groups[g].z;
      deal = deal_groups(sizes, n_xcc);
      n_items = deal.rows * ftiles * n_xcc;
    } else {
      item_start[ns] = (uint32_t)items.size();
      group_start.push_back((uint32_t)items.size());
      if (mode == PD_MODE_LEVEL_BATCHED) xcd_order(items, group_start, group_pos);
      n_items = items.size();
    }
    d_H.grow(per * std::max<size_t>(hslots.size(), 1) * sizeof(uint32_t), hist_budget);
    d_cand_key.grow((size_t)ns * ftiles * sizeof(unsigned long long));
    d_cand_left.grow((size_t)ns * ftiles * nC * sizeof(uint32_t));
    std::vector<float> sh(ns);
    for (uint32_t q = 0; q < ns; q++) sh[q] = slot_entropy(&tot[(size_t)q * nC], nC);
    Upload up{*this, d_slice};
    const size_t u_items = up.add(direct ? nullptr : items.data(), n_items * sizeof(HistItem));
    const size_t u_node = up.add(snode.data(), ns * sizeof(int32_t));
    const size_t u_hidx = up.add(shidx.data(), ns * sizeof(int32_t));
    const size_t u_mode = up.add(smode.data(), ns);
    const size_t u_tot = up.add(tot.data(), (size_t)ns * nC * sizeof(uint32_t));
    const size_t u_h = up.add(sh.data(), ns * sizeof(float));
    const size_t u_zero = up.add(zero.data(), zero.size() * sizeof(uint32_t));
    const size_t u_list = up.add(hslots.data(), hslots.size() * sizeof(uint32_t));
    const std::vector<uint64_t> no_key(ns, 0ull);
    const size_t u_best = up.add(no_key.data(), ns * sizeof(uint64_t));
    up.stage();
    if (direct) {
      HistItem *it = up.template host<HistItem>(u_items);
      std::fill(it, it + n_items, HistItem{NULL_SLOT, 0u, 0u, 0u});
      std::vector<uint64_t> len(n_xcc, 0);
      for (uint32_t g : deal.order) {
        const uint4 gr = groups[g];
        const uint32_t x = deal.xcd[g];
        HistItem *dst = it + len[x] * n_xcc + x;
        for (uint32_t ft = 0; ft < ftiles; ft++) dst[(size_t)ft * n_xcc] = HistItem{gr.x, gr.y, gr.z, ft};
        len[x] += ftiles;
      }
    }
    up.commit();
    sl = SliceTables{up.template at<HistItem>(u_items), up.template at<int32_t>(u_node),
                     up.template at<int32_t>(u_hidx),   up.template at<uint8_t>(u_mode),
                     up.template at<uint32_t>(u_tot),   up.template at<float>(u_h),
                     up.template at<uint32_t>(u_zero),  up.template at<uint32_t>(u_list),
                     up.template at<unsigned long long>(u_best)};
    d_perm_cur = nullptr;
    if constexpr (probe_rows<F>::on) {
      if (probe_order && nF > 64 && nF <= 65536u) {
        d_perm.grow((size_t)ns * nF * sizeof(uint16_t));
        const uint32_t segs = (nF + ORDER_MAX - 1) / ORDER_MAX;
        hipLaunchKernelGGL((k_cand_order<F>), dim3(ns, segs), dim3(ORDER_THREADS), 0, stream, tree,
                           sl.slot_node, nF, bnd, d_map_cur, d_perm.as<uint16_t>());
        HIPCHK(hipGetLastError());
        d_perm_cur = d_perm.as<uint16_t>();
      }
    }
    d_ctab_cur = nullptr;
    const size_t ctab_elems = (size_t)ns * ftiles * fpw * (F::FeatDim + nT);
    if (cand_table && ns && ctab_elems * sizeof(T) <= cand_table_budget) {
      // device memory short: the kernel derives the candidates itself
      try {
        d_ctab.grow(ctab_elems * sizeof(T), cand_table_budget);
      } catch (const NoMem &) {
        d_ctab.release();
      }
    }
    if (d_ctab.p && d_ctab.cap >= ctab_elems * sizeof(T) && cand_table && ns &&
        ctab_elems * sizeof(T) <= cand_table_budget) {
      const uint64_t n_thr = (uint64_t)ns * ftiles * fpw;
      hipLaunchKernelGGL((k_cand_table<F>), dim3((uint32_t)((n_thr + 255) / 256)), dim3(256), 0, stream, tree,
                         sl.slot_node, ns, nF, nT, fpw, ftiles, bnd, d_map_cur, d_perm_cur,
                         d_ctab.as<T>());
      HIPCHK(hipGetLastError());
      d_ctab_cur = d_ctab.as<T>();
    }
    if (!zero.empty()) {
      const size_t total = zero.size() * per;
      const uint32_t blocks = (uint32_t)std::min<size_t>((total + 255) / 256, (size_t)cu_count * 64);
      hipLaunchKernelGGL(k_zero_slots, dim3(blocks), dim3(256), 0, stream, d_H.as<uint32_t>(),
                         sl.zero, (uint32_t)zero.size(), per);
      HIPCHK(hipGetLastError());
    }
    uint32_t launches = 0;
    // the events bracket the histogram launches alone (the candidate order,
    // table and H zeroing before them are not the kernel being timed)
    if (ev_begin) HIPCHK(hipEventRecord(ev_begin->e, stream));
    if (mode == PD_MODE_LEVEL_BATCHED) {
      // (a launch holds fewer than 2^32 threads, 1024 an item at most; the padding
      // counts too)
      const size_t most = ((size_t)4000000 / n_xcc) * n_xcc;
      for (size_t b = 0; b < n_items; b += most, launches++)
        launch_hist((uint32_t)std::min(most, n_items - b), (uint32_t)b, act, bnd, tree, nF, nT);
    } else {
      for (uint32_t q = 0; q < ns; q++) {
        const uint32_t n = item_start[q + 1] - item_start[q];
        if (!n) continue;
        launch_hist(n, item_start[q], act, bnd, tree, nF, nT);
        launches++;
      }
    }
    d_perm_cur = nullptr;
    d_ctab_cur = nullptr;
    if (ev_end) HIPCHK(hipEventRecord(ev_end->e, stream));
    return launches;
  }

  // Split search over the nh H blocks of the current slice (block i belongs to
  // slot sl.hlist[i]).
  void launch_split(uint32_t nh, uint32_t nT, uint32_t nF, int mode, float *all_gains)
  {
    if (nC <= 8) launch_split_t<8>(nh, nT, nF, mode, all_gains);
    else if (nC <= 16) launch_split_t<16>(nh, nT, nF, mode, all_gains);
    else if (nC <= 32) launch_split_t<32>(nh, nT, nF, mode, all_gains);
    else launch_split_t<64>(nh, nT, nF, mode, all_gains);
  }
  template <int NCM>
  void launch_split_t(uint32_t nh, uint32_t nT, uint32_t nF, int mode, float *all_gains)
  {
    const uint32_t npairs = nT * nF;
    const uint32_t ppb = SPLIT_THREADS * 8;
    const uint32_t bps = (npairs + ppb - 1) / ppb;
    const size_t per = (size_t)nC * npairs;
    if (mode == PD_MODE_LEVEL_BATCHED) {
      hipLaunchKernelGGL((k_split<NCM>), dim3(nh * bps), dim3(SPLIT_THREADS), 0, stream, d_H.as<uint32_t>(),
                         sl.tot, nC, nT, nF, bps, ppb, sl.best, all_gains, sl.hlist);
      HIPCHK(hipGetLastError());
    } else {
      for (uint32_t i = 0; i < nh; i++) {
        hipLaunchKernelGGL((k_split<NCM>), dim3(bps), dim3(SPLIT_THREADS), 0, stream, d_H.as<uint32_t>() + i * per,
                           sl.tot, nC, nT, nF, bps, ppb, sl.best, all_gains, sl.hlist + i);
        HIPCHK(hipGetLastError());
      }
    }
  }

  // Split search + finalize of a slice of ns slots whose H blocks are
  // hslots (the fused slots were searched by the histogram kernel);
  // res_out[q*(nC+2) + {0: k, 1: gain bits, 2..: left counts}].
  // winners' parameters and thresholds of the slots of a level, filled by
  // split_slice through evaluate when set (train() sets them per level)
  std::vector<T> *lvl_par = nullptr, *lvl_thr = nullptr;

  // With `win` (the slice's candidate map, tree and bounds) the winners'
  // parameters and thresholds come back too (wpar [ns][FD], wthr [ns]).
  struct WinnerArgs {
    const uint32_t *d_map;
    uint32_t tree;
    const Bounds<F> *bnd;
    std::vector<T> *wpar, *wthr;
  };
  void split_slice(uint32_t ns, const std::vector<uint32_t> &hslots, uint32_t nT, uint32_t nF, int mode,
                   std::vector<uint32_t> &res_out, float *all_gains = nullptr, const WinnerArgs *win = nullptr)
  {
    const uint32_t nh = (uint32_t)hslots.size();
    if (nh) launch_split(nh, nT, nF, mode, all_gains);
    // one device buffer, one copy back: res [ns][nC + 2], then (with win) the
    // winners' parameters [ns][FD] and thresholds [ns]
    const size_t br = (size_t)ns * (nC + 2) * sizeof(uint32_t), o_par = (br + 15) & ~(size_t)15;
    const size_t bp = (size_t)ns * FD * sizeof(T), o_thr = (o_par + bp + 15) & ~(size_t)15;
    const size_t bt = ns * sizeof(T), bytes = win ? o_thr + bt : br;
    d_out.grow(std::max<size_t>(bytes, 16));
    char *dev = d_out.as<char>();
    const uint32_t threads = ns * (nC + 2);
    hipLaunchKernelGGL((k_finalize<F>), dim3((threads + 255) / 256), dim3(256), 0, stream, d_H.as<uint32_t>(), sl.best,
                       sl.slot_mode, sl.slot_hidx, d_cand_key.as<unsigned long long>(), d_cand_left.as<uint32_t>(), ns,
                       nC, nT, nF, hist_fpw(nT), (uint32_t *)dev, win ? win->tree : 0u, sl.slot_node,
                       win ? win->d_map : nullptr, win ? *win->bnd : Bounds<F>{}, win ? (T *)(dev + o_par) : nullptr,
                       win ? (T *)(dev + o_thr) : nullptr);
    HIPCHK(hipGetLastError());
    char *pin = (char *)stage.alloc(std::max<size_t>(bytes, 16));
    if (bytes) HIPCHK(hipMemcpyAsync(pin, dev, bytes, hipMemcpyDeviceToHost, stream));
    HIPCHK(hipStreamSynchronize(stream));
    res_out.resize((size_t)ns * (nC + 2));
    std::copy(pin, pin + br, (char *)res_out.data());
    if (win) {
      win->wpar->resize((size_t)ns * FD);
      win->wthr->resize(ns);
      std::copy(pin + o_par, pin + o_par + bp, (char *)win->wpar->data());
      std::copy(pin + o_thr, pin + o_thr + bt, (char *)win->wthr->data());
    }
    stage.reset();
  }

  // network input of a node: class histogram n_c / n (16) and depth / 16
  void slot_features(uint32_t node, uint32_t level, const uint32_t *classTot, float *out) const
  {
    uint32_t N = 0;
    for (uint32_t c = 0; c < nC; c++) N += classTot[(size_t)node * nC + c];
    for (uint32_t c = 0; c < (uint32_t)mlp::HIST_IN; c++)
      out[c] = (c < nC && N) ? (float)classTot[(size_t)node * nC + c] / (float)N : 0.0f;
    out[16] = (float)level / 16.0f;
  }
  static mlp::RowNorm make_norm(const Bounds<F> &bnd)
  {
    mlp::RowNorm nm{};
    for (int j = 0; j < 4; j++) {
      float b = 0.0f;
      if (j < FD) b = std::max(std::fabs((float)bnd.lo[j]), std::fabs((float)bnd.hi[j]));
      nm.inv_p[j] = b > 0.0f ? 1.0f / b : 0.0f;
    }
    const float range = (float)bnd.thi - (float)bnd.tlo;
    nm.thr_lo = (float)bnd.tlo;
    nm.thr_scale = range > 0.0f ? 2.0f / range : 0.0f;
    return nm;
  }

  // Records of the slots [s0, s0 + ns) of `sub` whose H blocks and all pair
  // gains (gains[q][t * nFe + f]) were just computed.
  void emit_records(const std::vector<SlotInfo> &sub, size_t s0, uint32_t ns, uint32_t nFe, uint32_t nT,
                    const Bounds<F> &bnd, uint32_t tree, const uint32_t *classTot, uint32_t level,
                    const float *gains, const std::vector<uint32_t> &res)
  {
    const uint32_t R = std::min<uint32_t>(sink_R, nT * nFe);
    if (!R) return;
    std::vector<uint32_t> es;
    std::vector<uint64_t> eb;
    std::vector<float> ebest;
    std::vector<float> sin((size_t)ns * 17, 0.0f);
    std::vector<int32_t> snode(ns);
    for (uint32_t q = 0; q < ns; q++) {
      const SlotInfo &si = sub[s0 + q];
      snode[q] = si.node;
      slot_features((uint32_t)si.node, level, classTot, &sin[(size_t)q * 17]);
      if (si.trainable && si.count > 0 && sink_n + R <= sink_cap) {
        es.push_back(q);
        eb.push_back(sink_n);
        float g;
        std::memcpy(&g, &res[(size_t)q * (nC + 2) + 1], 4);
        ebest.push_back(g);
        sink_n += R;
      }
    }
    if (es.empty()) return;
    d_emit_in.ensure(sin.size() * sizeof(float));
    d_emit_node.ensure(ns * sizeof(int32_t));
    d_emit_slots.ensure(es.size() * sizeof(uint32_t));
    d_emit_base.ensure(eb.size() * sizeof(uint64_t));
    d_emit_best.ensure(ebest.size() * sizeof(float));
    HIPCHK(hipMemcpyAsync(d_emit_best.p, ebest.data(), ebest.size() * sizeof(float), hipMemcpyHostToDevice, stream));
    HIPCHK(hipMemcpyAsync(d_emit_in.p, sin.data(), sin.size() * sizeof(float), hipMemcpyHostToDevice, stream));
    HIPCHK(hipMemcpyAsync(d_emit_node.p, snode.data(), ns * sizeof(int32_t), hipMemcpyHostToDevice, stream));
    HIPCHK(hipMemcpyAsync(d_emit_slots.p, es.data(), es.size() * sizeof(uint32_t), hipMemcpyHostToDevice, stream));
    HIPCHK(hipMemcpyAsync(d_emit_base.p, eb.data(), eb.size() * sizeof(uint64_t), hipMemcpyHostToDevice, stream));
    const uint64_t threads = (uint64_t)es.size() * R;
    hipLaunchKernelGGL((k_emit<F>), dim3((uint32_t)((threads + 255) / 256)), dim3(256), 0, stream, gains,
                       d_emit_slots.as<uint32_t>(), d_emit_base.as<uint64_t>(), d_emit_best.as<float>(),
                       (uint32_t)es.size(), R, d_emit_in.as<float>(), d_emit_node.as<int32_t>(), nFe, nT, tree, bnd,
                       make_norm(bnd), sink_x, sink_t, sink_rel);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(stream));
  }

  // Histogram + split search of the frontier slots `idx` (indices into
  // `slots`) with nFe candidates each: the sampler's candidates 0..nFe-1, or,
  // with a candidate map (d_map [idx.size()][nFe] on the device, h_map its
  // host copy), the listed sampler indices.  Results go to res_all at each
  // slot's index with k in sampler terms (t * P.n_features + f).  With
  // `emit`, every slot gets its H block and the FP32 gains of all pairs, and
  // the record sink receives samples of them.
  void evaluate(const std::vector<SlotInfo> &slots, const std::vector<uint32_t> &idx, const uint4 *act,
                const pd_train_params &P, uint32_t nFe, const uint32_t *d_map_all,
                const std::vector<uint32_t> *h_map, const Bounds<F> &bnd, uint32_t tree, int mode, uint32_t ch,
                const uint32_t *classTot, uint32_t level, bool emit, std::vector<uint32_t> &res_all,
                pd_level_stats &st)
  {
    if (idx.empty()) return;
    const uint32_t nT = P.n_thresholds, nFp = P.n_features;
    pd_train_params Pe = P;
    Pe.n_features = nFe;
    std::vector<SlotInfo> sub(idx.size());
    for (size_t i = 0; i < idx.size(); i++) sub[i] = slots[idx[i]];
    const size_t per_bytes = (size_t)nC * nT * nFe * sizeof(uint32_t);
    size_t h_per_slice = std::max<size_t>(1, hist_budget / per_bytes);   // H blocks per slice
    if (emit)   // the all-pair gains of a slice stay within 1 GiB
      h_per_slice = std::min<size_t>(h_per_slice, std::max<size_t>(1, (1ull << 30) / ((size_t)nT * nFe * 4)));
    Event e0, e1, e2;
    for (size_t s0 = 0; s0 < sub.size();) {
      // a slice holds at most h_per_slice slots that need an H block
      size_t s1 = s0, nh = 0;
      while (s1 < sub.size()) {
        const uint32_t cnt = sub[s1].trainable ? sub[s1].count : 0u;
        const bool needs_h = emit || cnt > ch;
        if (needs_h && nh == h_per_slice) break;
        nh += needs_h ? 1 : 0;
        s1++;
      }
      const uint32_t ns = (uint32_t)(s1 - s0);
      st.slices++;
      std::vector<uint32_t> tot((size_t)ns * nC);
      for (uint32_t q = 0; q < ns; q++)
        std::copy(&classTot[(size_t)sub[s0 + q].node * nC], &classTot[(size_t)sub[s0 + q].node * nC] + nC,
                  &tot[(size_t)q * nC]);
      std::vector<uint32_t> hslots, res;
      d_map_cur = d_map_all ? d_map_all + s0 * nFe : nullptr;
      st.hist_launches += hist_slice(sub, s0, s1, act, Pe, bnd, tree, mode, ch, tot, emit, hslots, &e0, &e1);
      d_map_cur = nullptr;
      float *gains = nullptr;
      if (emit) {
        d_gains.ensure((size_t)ns * nT * nFe * sizeof(float));
        gains = d_gains.as<float>();
      }
      std::vector<T> wpar, wthr;
      const WinnerArgs win{d_map_all ? d_map_all + s0 * nFe : nullptr, tree, &bnd, &wpar, &wthr};
      split_slice(ns, hslots, nT, nFe, mode, res, gains, lvl_par ? &win : nullptr);
      HIPCHK(hipEventRecord(e2.e, stream));
      HIPCHK(hipEventSynchronize(e2.e));
      stage.reset();
      st.hist_ms += elapsed_ms(e0, e1);
      st.split_ms += elapsed_ms(e1, e2);
      if (emit) emit_records(sub, s0, ns, nFe, nT, bnd, tree, classTot, level, gains, res);
      for (uint32_t q = 0; q < ns; q++) {
        const uint32_t *r = &res[(size_t)q * (nC + 2)];
        const uint32_t t = r[0] / nFe, f = r[0] % nFe;
        const uint32_t fs = h_map ? (*h_map)[(s0 + q) * nFe + f] : f;
        uint32_t *o = &res_all[(size_t)idx[s0 + q] * (nC + 2)];
        o[0] = t * nFp + fs;
        std::copy(r + 1, r + nC + 2, o + 1);
        if (lvl_par) {
          std::copy(&wpar[(size_t)q * FD], &wpar[(size_t)q * FD] + FD, &(*lvl_par)[(size_t)idx[s0 + q] * FD]);
          (*lvl_thr)[idx[s0 + q]] = wthr[q];
        }
      }
      s0 = s1;
    }
  }

  // Records of the learned refinement for the slice [s0, s0 + ns) of the
  // ranked slots gidx (rows: their screened candidates with the subsample
  // statistics): the exact gain of every screened candidate over all of its
  // node's samples, then sink_R records per slot (half of them its best
  // estimates), target = exact relative gain minus estimated relative gain.
  void emit_sub_records(const SubRows<F> &rows, const std::vector<SlotInfo> &slots,
                        const std::vector<uint32_t> &gidx, size_t s0, uint32_t ns, const uint4 *act,
                        const pd_train_params &P, uint32_t screen, const Bounds<F> &bnd, uint32_t tree,
                        const uint32_t *classTot)
  {
    const uint32_t R = sink_R & ~1u, half = R / 2;
    std::vector<uint32_t> eslots;
    std::vector<uint64_t> ebase;
    for (uint32_t q = 0; q < ns; q++) {
      if (sink_n + R > sink_cap) break;
      eslots.push_back(q);
      ebase.push_back(sink_n);
      sink_n += R;
    }
    if (eslots.empty()) return;
    // exact gains of the screened candidates on all samples (every slot gets
    // its H block; the subsample's H is no longer needed)
    std::vector<SlotInfo> full(ns);
    std::vector<uint32_t> T((size_t)ns * nC), hslots;
    uint64_t cnt = 0;
    for (uint32_t q = 0; q < ns; q++) {
      full[q] = slots[gidx[s0 + q]];
      cnt += full[q].count;
      std::copy(&classTot[(size_t)full[q].node * nC], &classTot[(size_t)full[q].node * nC] + nC, &T[(size_t)q * nC]);
    }
    pd_train_params Pe = P;
    Pe.n_features = screen;
    Pe.n_thresholds = 1;
    d_map_cur = rows.map;
    hist_slice(full, 0, ns, act, Pe, bnd, tree, PD_MODE_LEVEL_BATCHED,
               pick_chunk(cnt, screen, 1), T, true, hslots);
    d_map_cur = nullptr;
    const uint32_t nh = (uint32_t)hslots.size();
    d_full.ensure((size_t)ns * screen * sizeof(float));
    launch_split(nh, 1, screen, PD_MODE_LEVEL_BATCHED, d_full.as<float>());
    d_gbest.ensure((size_t)ns * sizeof(float));
    hipLaunchKernelGGL(k_slot_max, dim3(ns), dim3(256), 0, stream, d_full.as<float>(), screen, d_gbest.as<float>());
    // the best half-R estimates of every emitting slot
    d_top.ensure((size_t)ns * std::max<uint32_t>(half, 1) * sizeof(uint32_t));
    hipLaunchKernelGGL(mlp::k_topk, dim3(ns), dim3(256), 0, stream, rows.est, screen, half, half,
                       d_top.as<uint32_t>());
    HIPCHK(hipGetLastError());
    const uint32_t ne = (uint32_t)eslots.size();
    d_eslots.ensure(ne * sizeof(uint32_t));
    d_ebase.ensure(ne * sizeof(uint64_t));
    h2d(d_eslots.p, eslots.data(), ne * sizeof(uint32_t));
    h2d(d_ebase.p, ebase.data(), ne * sizeof(uint64_t));
    const uint64_t threads = (uint64_t)ne * R;
    hipLaunchKernelGGL((k_emit_sub<F>), dim3((uint32_t)((threads + 255) / 256)), dim3(256), 0, stream, rows,
                       d_full.as<float>(), d_gbest.as<float>(), d_top.as<uint32_t>(), d_eslots.as<uint32_t>(),
                       d_ebase.as<uint64_t>(), ne, R, sink_x, sink_t, sink_rel);
    HIPCHK(hipGetLastError());
  }

  // Class-stratified subsample of the slots gidx for the refinement: a slot
  // of n samples gets m = max(prop_refine_min, n / stride) of them, class c
  // (T_c samples) at the rate q_c / T_c with q_c = min(T_c, max(m T_c / n,
  // m / (2 nC))), so that every class the node holds is represented even
  // when it is rare (the best split often isolates a rare class).  Which
  // records are kept is a hash of (image, pixel, node) against the rate, so
  // it does not depend on record order; the kept records keep the node's
  // order.  Fills d_sub_act / d_sub_cls, db (G + 1 subsample offsets) and dc
  // (sizes); returns the subsample's size.
  uint64_t strat_subsample(const std::vector<SlotInfo> &slots, const std::vector<uint32_t> &gidx, const uint4 *act,
                           uint32_t stride, const uint32_t *classTot, std::vector<uint32_t> &db,
                           std::vector<uint32_t> &dc)
  {
    const uint32_t G = (uint32_t)gidx.size();
    std::vector<uint32_t> meta(3 * (size_t)G + 1), rate((size_t)G * nC);   // src_begin | cat_begin[G+1] | node
    uint64_t tot = 0;
    for (uint32_t g = 0; g < G; g++) {
      const SlotInfo &si = slots[gidx[g]];
      meta[g] = si.begin;
      meta[G + g] = (uint32_t)tot;
      meta[2 * G + 1 + g] = (uint32_t)si.node;
      tot += si.count;
      const double n = (double)std::max<uint32_t>(si.count, 1u);
      const double m = (double)std::max<uint32_t>(prop_refine_min, (si.count + stride - 1) / stride);
      const double mmin = std::max(1.0, std::floor(m / (2.0 * nC)));
      for (uint32_t c = 0; c < nC; c++) {
        const double Tc = (double)classTot[(size_t)si.node * nC + c];
        const double q = std::min(Tc, std::max(std::ceil(m * Tc / n), mmin));
        const double p = Tc > 0.0 ? q / Tc : 1.0;
        rate[(size_t)g * nC + c] = p >= 1.0 ? 0xffffffffu : (uint32_t)std::min(p * 4294967296.0, 4294967294.0);
      }
    }
    meta[2 * G] = (uint32_t)tot;
    require(tot < (1ull << 31), "refinement input too large");
    d_st_meta.ensure(meta.size() * sizeof(uint32_t));
    d_st_rate.ensure(std::max<size_t>(rate.size(), 1) * sizeof(uint32_t));
    h2d(d_st_meta.p, meta.data(), meta.size() * sizeof(uint32_t));
    h2d(d_st_rate.p, rate.data(), rate.size() * sizeof(uint32_t));
    const uint32_t *src_begin = d_st_meta.as<uint32_t>(), *cat = src_begin + G;
    const int32_t *node = (const int32_t *)(src_begin + 2 * G + 1);
    d_st_flags.ensure((tot + 1) * sizeof(unsigned long long));
    d_st_pos.ensure((tot + 1) * sizeof(unsigned long long));
    hipLaunchKernelGGL(k_strat_flags, dim3((uint32_t)((tot + 1 + 255) / 256)), dim3(256), 0, stream, act, src_begin,
                       cat, G, (uint32_t)tot, nC, node, d_st_rate.as<uint32_t>(),
                       d_st_flags.as<unsigned long long>(), d_sub_cls.as<uint32_t>());
    HIPCHK(hipGetLastError());
    size_t tmp_bytes = 0;
    HIPCHK(hipcub::DeviceScan::ExclusiveSum(nullptr, tmp_bytes, d_st_flags.as<unsigned long long>(),
                                            d_st_pos.as<unsigned long long>(), (int)(tot + 1), stream));
    d_st_tmp.ensure(tmp_bytes);
    HIPCHK(hipcub::DeviceScan::ExclusiveSum(d_st_tmp.p, tmp_bytes, d_st_flags.as<unsigned long long>(),
                                            d_st_pos.as<unsigned long long>(), (int)(tot + 1), stream));
    // subsample offsets of the slots: the scan at each slot's first record
    std::vector<unsigned long long> pos(G + 1);
    for (uint32_t g = 0; g <= G; g++)
      HIPCHK(hipMemcpyAsync(&pos[g], d_st_pos.as<unsigned long long>() + meta[G + g], sizeof(unsigned long long),
                            hipMemcpyDeviceToHost, stream));
    HIPCHK(hipStreamSynchronize(stream));
    const uint64_t total = pos[G];
    db.assign(G + 1, 0u);
    dc.assign(G, 0u);
    for (uint32_t g = 0; g < G; g++) {
      db[g] = (uint32_t)pos[g];
      dc[g] = (uint32_t)(pos[g + 1] - pos[g]);
    }
    db[G] = (uint32_t)total;
    d_sub_act.ensure(std::max<uint64_t>(total, 1) * sizeof(uint4));
    if (tot)
      hipLaunchKernelGGL(k_strat_scatter, dim3((uint32_t)((tot + 255) / 256)), dim3(256), 0, stream, act, src_begin,
                         cat, G, (uint32_t)tot, d_st_flags.as<unsigned long long>(),
                         d_st_pos.as<unsigned long long>(), d_sub_act.as<uint4>());
    HIPCHK(hipGetLastError());
    return total;
  }

  // Refinement stage of the split proposal for the slots gidx: each slot's
  // `screen` candidates (d_map1 [G][screen] / h_map1, sampler indices) are
  // evaluated exactly on an evenly spaced subsample of its samples (every
  // prop_refine-th, at least prop_refine_min, all samples of a smaller
  // node), and the `keep` with the largest subsample gains (ties to the
  // lower position, written in position order) form h_map2 / d_map2.
  void refine(const std::vector<SlotInfo> &slots, const std::vector<uint32_t> &gidx, const uint4 *act,
              const pd_train_params &P, uint32_t screen, uint32_t keep, const uint32_t *d_map1,
              const std::vector<uint32_t> &h_map1, const Bounds<F> &bnd, uint32_t tree,
              const uint32_t *classTot, std::vector<uint32_t> &h_map2, pd_level_stats &st)
  {
    const uint32_t G = (uint32_t)gidx.size();
    std::vector<uint32_t> sb(G), sc(G), db(G + 1), dc(G);
    uint64_t total = 0;
    Event ea, eb;
    HIPCHK(hipEventRecord(ea.e, stream));
    d_sub_cls.ensure((size_t)G * nC * sizeof(uint32_t));
    HIPCHK(hipMemsetAsync(d_sub_cls.p, 0, (size_t)G * nC * sizeof(uint32_t), stream));
    const uint32_t stride = std::max<uint32_t>(prop_refine, 1u);
    if (!prop_strata) {
      for (uint32_t g = 0; g < G; g++) {
        const SlotInfo &si = slots[gidx[g]];
        sb[g] = si.begin;
        sc[g] = si.count;
        const uint32_t want = std::max<uint32_t>(prop_refine_min, (si.count + stride - 1) / stride);
        dc[g] = std::min<uint32_t>(si.count, want);
        db[g] = (uint32_t)total;
        total += dc[g];
      }
      db[G] = (uint32_t)total;
      require(total < (1ull << 32), "refinement subsample too large");
      d_sub_idx.ensure((size_t)(4 * G + 1) * sizeof(uint32_t));
      uint32_t *di = d_sub_idx.as<uint32_t>();
      h2d(di, sb.data(), G * sizeof(uint32_t));
      h2d(di + G, sc.data(), G * sizeof(uint32_t));
      h2d(di + 2 * G, db.data(), (G + 1) * sizeof(uint32_t));
      h2d(di + 3 * G + 1, dc.data(), G * sizeof(uint32_t));
      d_sub_act.ensure(std::max<uint64_t>(total, 1) * sizeof(uint4));
      if (total) {
        hipLaunchKernelGGL(k_subsample, dim3((uint32_t)((total + 255) / 256)), dim3(256), 0, stream, act, di,
                           di + G, di + 2 * G, di + 3 * G + 1, G, (uint32_t)total, nC, d_sub_act.as<uint4>(),
                           d_sub_cls.as<uint32_t>());
        HIPCHK(hipGetLastError());
      }
    } else {
      total = strat_subsample(slots, gidx, act, stride, classTot, db, dc);
    }
    std::vector<uint32_t> cls((size_t)G * nC);
    d2h_sync(cls.data(), d_sub_cls.p, cls.size() * sizeof(uint32_t));
    // the subsample as frontier slots with their own class totals, searched
    // with every slot's H block and the gains of all its pairs
    std::vector<SlotInfo> sub(G);
    for (uint32_t g = 0; g < G; g++) sub[g] = SlotInfo{slots[gidx[g]].node, db[g], dc[g], true};
    pd_train_params Pe = P;
    Pe.n_features = screen;
    Pe.n_thresholds = 1;
    const uint32_t ch = pick_chunk(total, screen, 1);
    const size_t per_bytes = (size_t)nC * screen * sizeof(uint32_t);
    const size_t h_per_slice = std::max<size_t>(
        1, std::min<size_t>(hist_budget / per_bytes, (1ull << 30) / ((size_t)screen * 4)));
    h_map2.assign((size_t)G * keep, 0u);
    for (size_t s0 = 0; s0 < G; s0 += h_per_slice) {
      const size_t s1 = std::min<size_t>(G, s0 + h_per_slice);
      const uint32_t ns = (uint32_t)(s1 - s0);
      std::vector<uint32_t> tot(cls.begin() + s0 * nC, cls.begin() + s1 * nC), hslots, res;
      d_map_cur = d_map1 + s0 * screen;
      hist_slice(sub, s0, s1, d_sub_act.as<uint4>(), Pe, bnd, tree, PD_MODE_LEVEL_BATCHED, ch, tot, true, hslots);
      d_map_cur = nullptr;
      d_gains.ensure((size_t)ns * screen * sizeof(float));
      // the ranking scores: the exact gains on the subsample, or (stratified)
      // the estimate of the node's gain, optionally corrected by the network
      float *rank = d_gains.as<float>();
      if (prop_strata) {
        std::vector<uint32_t> T((size_t)ns * nC);
        for (uint32_t q = 0; q < ns; q++)
          std::copy(&classTot[(size_t)slots[gidx[s0 + q]].node * nC],
                    &classTot[(size_t)slots[gidx[s0 + q]].node * nC] + nC, &T[(size_t)q * nC]);
        d_st_tot.ensure(T.size() * sizeof(uint32_t));
        h2d(d_st_tot.p, T.data(), T.size() * sizeof(uint32_t));
        const uint64_t n_pairs = (uint64_t)ns * screen;
        const dim3 grid((uint32_t)((n_pairs + 255) / 256));
        const uint32_t *Sd = d_sub_cls.as<uint32_t>() + s0 * nC;
        // the network's inputs are needed to rank (mode 2) or to emit records
        const bool recs = sink_x != nullptr && sink_R >= 2 && sink_n < sink_cap;
        const bool stats = prop_strata == 2 || recs;
        if (stats) d_frac.ensure(n_pairs * 9 * sizeof(float));
        float *fr = stats ? d_frac.as<float>() : nullptr;
        if (nC <= 8)
          hipLaunchKernelGGL(k_est_gain<8>, grid, dim3(256), 0, stream, d_H.as<uint32_t>(), ns, screen, nC,
                             d_st_tot.as<uint32_t>(), Sd, d_gains.as<float>(), fr);
        else if (nC <= 16)
          hipLaunchKernelGGL(k_est_gain<16>, grid, dim3(256), 0, stream, d_H.as<uint32_t>(), ns, screen, nC,
                             d_st_tot.as<uint32_t>(), Sd, d_gains.as<float>(), fr);
        else
          hipLaunchKernelGGL(k_est_gain<64>, grid, dim3(256), 0, stream, d_H.as<uint32_t>(), ns, screen, nC,
                             d_st_tot.as<uint32_t>(), Sd, d_gains.as<float>(), fr);
        HIPCHK(hipGetLastError());
        // the score: the estimate relative to the slot's best estimate (the
        // same order as the estimate), plus the network's correction in mode 2
        d_gmax.ensure((size_t)ns * sizeof(float));
        hipLaunchKernelGGL(k_slot_max, dim3(ns), dim3(256), 0, stream, d_gains.as<float>(), screen,
                           d_gmax.as<float>());
        HIPCHK(hipGetLastError());
        if (recs) {
          const SubRows<F> rows{d_pslot_in.as<float>() + s0 * 17, d_pslot_node.as<int32_t>() + s0, d_map1 + s0 * screen,
                                d_frac.as<float>(), d_gains.as<float>(), d_gmax.as<float>(), screen, tree,
                                (uint32_t)n_pairs, bnd, make_norm(bnd)};
          emit_sub_records(rows, slots, gidx, s0, ns, act, P, screen, bnd, tree, classTot);
        }
        // rows the correction network scores per slot (mode 2): every
        // screened candidate, or the slot's best prop_corr_rows (at least
        // keep) by the estimate
        const uint32_t M = prop_corr_rows ? std::min<uint32_t>(screen, std::max<uint32_t>(prop_corr_rows, keep))
                                          : screen;
        const SubRows<F> rows{d_pslot_in.as<float>() + s0 * 17, d_pslot_node.as<int32_t>() + s0, d_map1 + s0 * screen,
                              d_frac.as<float>(), d_gains.as<float>(), d_gmax.as<float>(), screen, tree,
                              (uint32_t)n_pairs, bnd, make_norm(bnd)};
        const float *ynet = nullptr;
        if (prop_strata == 2) require(prop_mlp != nullptr, "the learned refinement needs a network");
        if (prop_strata == 2 && M == screen) {
          d_ynet.ensure(n_pairs * sizeof(float));
          hipLaunchKernelGGL((mlp::k_mlp_fwd<SubRows<F>, false>),
                             dim3((uint32_t)((n_pairs + mlp::FWD_ROWS - 1) / mlp::FWD_ROWS)), dim3(mlp::THREADS), 0,
                             stream, rows, (uint32_t)n_pairs, prop_mlp->weights(), d_ynet.as<float>(), (uint16_t *)nullptr,
                             (uint16_t *)nullptr, 0u);
          HIPCHK(hipGetLastError());
          ynet = d_ynet.as<float>();
        }
        d_score.ensure(n_pairs * sizeof(float));
        hipLaunchKernelGGL(k_residual_score, grid, dim3(256), 0, stream, d_gains.as<float>(), d_gmax.as<float>(), ynet,
                           screen, n_pairs, d_score.as<float>());
        HIPCHK(hipGetLastError());
        rank = d_score.as<float>();
        if (prop_strata == 2 && M < screen) {
          // the network corrects each slot's best M by the estimate (the
          // order of the final ranking's estimate term, ties to the lower
          // index); the others rank below them, so with a zero correction the
          // kept set is the estimate's own
          const uint64_t n_sel = (uint64_t)ns * M;
          d_net_sel.ensure(n_sel * sizeof(uint32_t));
          hipLaunchKernelGGL(mlp::k_topk, dim3(ns), dim3(256), 0, stream, d_score.as<float>(), screen, M, M,
                             d_net_sel.as<uint32_t>());
          HIPCHK(hipGetLastError());
          const SubRowsSel<F> srows{rows, d_net_sel.as<uint32_t>(), M, (uint32_t)n_sel};
          d_ynet.ensure(n_sel * sizeof(float));
          hipLaunchKernelGGL((mlp::k_mlp_fwd<SubRowsSel<F>, false>),
                             dim3((uint32_t)((n_sel + mlp::FWD_ROWS - 1) / mlp::FWD_ROWS)), dim3(mlp::THREADS), 0,
                             stream, srows, (uint32_t)n_sel, prop_mlp->weights(), d_ynet.as<float>(), (uint16_t *)nullptr,
                             (uint16_t *)nullptr, 0u);
          HIPCHK(hipGetLastError());
          d_score2.ensure(n_pairs * sizeof(float));
          hipLaunchKernelGGL(k_fill_f32, grid, dim3(256), 0, stream, d_score2.as<float>(), n_pairs, -FLT_MAX);
          hipLaunchKernelGGL(k_sel_score, dim3((uint32_t)((n_sel + 255) / 256)), dim3(256), 0, stream,
                             d_score.as<float>(), d_net_sel.as<uint32_t>(), d_ynet.as<float>(), screen, M, n_sel,
                             d_score2.as<float>());
          HIPCHK(hipGetLastError());
          rank = d_score2.as<float>();
        }
      } else {
        const uint32_t nh = (uint32_t)hslots.size();
        launch_split(nh, 1, screen, PD_MODE_LEVEL_BATCHED, d_gains.as<float>());
      }
      d_sub_sel.ensure((size_t)ns * keep * sizeof(uint32_t));
      hipLaunchKernelGGL(mlp::k_topk, dim3(ns), dim3(256), 0, stream, rank, screen, keep, keep,
                         d_sub_sel.as<uint32_t>());
      HIPCHK(hipGetLastError());
      std::vector<uint32_t> sel((size_t)ns * keep);
      d2h_sync(sel.data(), d_sub_sel.p, sel.size() * sizeof(uint32_t));
      for (uint32_t q = 0; q < ns; q++)
        for (uint32_t j = 0; j < keep; j++)
          h_map2[(s0 + q) * keep + j] = h_map1[(s0 + q) * screen + sel[(size_t)q * keep + j]];
    }
    d_map2.ensure(h_map2.size() * sizeof(uint32_t));
    h2d(d_map2.p, h_map2.data(), h_map2.size() * sizeof(uint32_t));
    HIPCHK(hipEventRecord(eb.e, stream));
    HIPCHK(hipEventSynchronize(eb.e));
    stage.reset();
    st.refine_ms += elapsed_ms(ea, eb);
  }

  // Split proposal of the slots idx: the network scores the pool of
  // K = P.n_features candidates of every node (one threshold each), the
  // best `prop_keep` are histogrammed exactly; optionally the exhaustive
  // evaluation of the whole pool is run beside it as the judge.
  void propose(const std::vector<SlotInfo> &slots, const std::vector<uint32_t> &idx, const uint4 *act,
               const pd_train_params &P, const Bounds<F> &bnd, uint32_t tree, const uint32_t *classTot,
               uint32_t level, std::vector<uint32_t> &res_all, pd_level_stats &st)
  {
    const uint32_t K = P.n_features, keep = prop_keep;
    const mlp::RowNorm nm = make_norm(bnd);
    const size_t g_max = std::max<size_t>(1, std::min<size_t>(idx.size(), (512ull << 20) / ((size_t)K * 4)));
    Event ea, eb, ec;
    for (size_t g0 = 0; g0 < idx.size(); g0 += g_max) {
      const size_t G = std::min(g_max, idx.size() - g0);
      const std::vector<uint32_t> gidx(idx.begin() + g0, idx.begin() + g0 + G);
      std::vector<float> sin(G * 17);
      std::vector<int32_t> snode(G);
      uint64_t gact = 0;
      for (size_t i = 0; i < G; i++) {
        const SlotInfo &si = slots[gidx[i]];
        snode[i] = si.node;
        slot_features((uint32_t)si.node, level, classTot, &sin[i * 17]);
        gact += si.count;
      }
      const uint64_t rows = (uint64_t)G * K;
      require(rows < (1ull << 32), "proposal pool too large");
      d_pslot_in.ensure(sin.size() * sizeof(float));
      d_pslot_node.ensure(G * sizeof(int32_t));
      d_scores.ensure(rows * sizeof(float));
      HIPCHK(hipMemcpyAsync(d_pslot_in.p, sin.data(), sin.size() * sizeof(float), hipMemcpyHostToDevice, stream));
      HIPCHK(hipMemcpyAsync(d_pslot_node.p, snode.data(), G * sizeof(int32_t), hipMemcpyHostToDevice, stream));
      const PoolRows<F> src{d_pslot_in.as<float>(), d_pslot_node.as<int32_t>(), K, tree, (uint32_t)rows, bnd, nm};
      const uint32_t screen = std::min<uint32_t>(K, std::max<uint32_t>(keep, prop_screen));
      // with refinement the whole screened set is kept for the subsample stage
      const uint32_t first = prop_refine ? screen : keep;
      // refinement of the whole pool needs no scores: the screened set is the
      // pool in sampler order
      const bool scored = !(prop_refine && screen >= K);
      d_map.ensure(G * first * sizeof(uint32_t));
      std::vector<uint32_t> hmap(G * first);
      HIPCHK(hipEventRecord(ea.e, stream));
      if (scored)
        hipLaunchKernelGGL((mlp::k_mlp_fwd<PoolRows<F>, false>),
                           dim3((uint32_t)((rows + mlp::FWD_ROWS - 1) / mlp::FWD_ROWS)),
                           dim3(mlp::THREADS), 0, stream, src, (uint32_t)rows, prop_mlp->weights(),
                           d_scores.as<float>(), (uint16_t *)nullptr, (uint16_t *)nullptr, 0u);
      HIPCHK(hipGetLastError());
      HIPCHK(hipEventRecord(eb.e, stream));
      if (scored) {
        hipLaunchKernelGGL(mlp::k_topk, dim3((uint32_t)G), dim3(256), 0, stream, d_scores.as<float>(), K, screen,
                           first, d_map.as<uint32_t>());
        HIPCHK(hipGetLastError());
        HIPCHK(hipEventRecord(ec.e, stream));
        HIPCHK(hipMemcpyAsync(hmap.data(), d_map.p, hmap.size() * sizeof(uint32_t), hipMemcpyDeviceToHost, stream));
      } else {
        for (size_t g = 0; g < G; g++)
          for (uint32_t j = 0; j < first; j++) hmap[g * first + j] = j;
        HIPCHK(hipMemcpyAsync(d_map.p, hmap.data(), hmap.size() * sizeof(uint32_t), hipMemcpyHostToDevice, stream));
        HIPCHK(hipEventRecord(ec.e, stream));
      }
      HIPCHK(hipStreamSynchronize(stream));
      st.mlp_ms += elapsed_ms(ea, eb);
      st.select_ms += elapsed_ms(eb, ec);
      const uint32_t *dmap = d_map.as<uint32_t>();
      if (prop_refine && keep < screen) {
        std::vector<uint32_t> hmap2;
        refine(slots, gidx, act, P, screen, keep, d_map.as<uint32_t>(), hmap, bnd, tree, classTot, hmap2, st);
        hmap.swap(hmap2);
        dmap = d_map2.as<uint32_t>();
      }
      evaluate(slots, gidx, act, P, keep, dmap, &hmap, bnd, tree, PD_MODE_LEVEL_BATCHED,
               pick_chunk(gact, keep, 1), classTot, level, false, res_all, st);
      if (prop_judge) {
        std::vector<uint32_t> res_j(slots.size() * (nC + 2), 0u);
        pd_level_stats js{};
        std::vector<T> *keep_par = lvl_par, *keep_thr = lvl_thr;
        lvl_par = lvl_thr = nullptr;   // the judge's winners are not the tree's
        evaluate(slots, gidx, act, P, K, nullptr, nullptr, bnd, tree, PD_MODE_LEVEL_BATCHED,
                 pick_chunk(gact, K, 1), classTot, level, false, res_j, js);
        lvl_par = keep_par;
        lvl_thr = keep_thr;
        st.judge_ms += js.hist_ms + js.split_ms;
        for (uint32_t q : gidx) {
          float ge, gp;
          std::memcpy(&ge, &res_j[(size_t)q * (nC + 2) + 1], 4);
          std::memcpy(&gp, &res_all[(size_t)q * (nC + 2) + 1], 4);
          st.judged_nodes++;
          st.gain_exhaustive += ge;
          st.gain_proposal += gp;
          if (ge > 0.0f) st.gain_loss_rel += ((double)ge - (double)gp) / (double)ge;
        }
      }
    }
  }

  void train(const pd_train_params &P, uint32_t tree_id, uint32_t depth, uint32_t end_depth, int mode,
             const float *prior, int32_t *left, void *feats_v, void *thrs_v, float *post, uint32_t *node_k,
             float *node_gain, double *node_gain64, pd_level_stats *ls) override
  {
    if (!S) throw StateError("pd_trainer_train before pd_trainer_set_data");
    check_params(P, FD, sizeof(T) == 2);
    require(depth >= 1 && depth <= 24, "tree depth must be in [1, 24]");
    require(end_depth >= 1 && end_depth <= depth, "end_depth must be in [1, tree depth]");
    require(mode == PD_MODE_PER_NODE || mode == PD_MODE_LEVEL_BATCHED || mode == PD_MODE_PROPOSAL,
            "unknown training mode");
    if (mode == PD_MODE_PROPOSAL) {
      require(prop_mlp != nullptr, "PD_MODE_PROPOSAL needs pd_trainer_set_proposal first");
      require(prop_keep >= 1 && prop_keep <= P.n_features, "proposal keep must be in [1, n_features]");
      require(nC <= (uint32_t)mlp::HIST_IN, "the proposal network takes at most 16 classes");
      require(prop_mlp->device == device, "proposal network on another device");
    }
    require(nC <= 64, "at most 64 classes");
    require(prior && left && feats_v && thrs_v && post, "null tree array");
    set_device(device);
    T *feats = (T *)feats_v;
    T *thrs = (T *)thrs_v;
    const Bounds<F> bnd = make_bounds<F>(P);
    const uint32_t nF = P.n_features, nT = P.n_thresholds, thr = P.per_leaf_samples_thr;
    const size_t N = ((size_t)1 << depth) - 1;
    // Tree::_init (tree_impl.hpp:239-273), root posterior = priors: the nodes of
    // the first INIT_LEVELS levels here, the others on a second host thread
    // while the GPU works on those levels (`init` is waited for before a deeper
    // level's results are written, and by its destructor).  A depth-20 tree's
    // arrays and totals took 15..20 ms of the call, before any GPU work (4000 x
    // 32 candidates: 142.5 ms a tree with it, 127.5 now; RGBD, 21 classes: 43.3 -> 23.3).
    auto init_nodes = [&](size_t b, size_t e) {
      std::fill(left + b, left + e, -2);
      zero_fill(feats + b * FD, (e - b) * FD * sizeof(T));
      zero_fill(thrs + b, (e - b) * sizeof(T));
      zero_fill(post + b * nC, (e - b) * nC * sizeof(float));
    };
    constexpr uint32_t INIT_LEVELS = 12;
    const size_t n_init = std::min(N, ((size_t)1 << INIT_LEVELS) - 1);
    std::future<void> init;
    size_t n_here = n_init;
    if (n_init < N) {
      try {
        init = std::async(std::launch::async, init_nodes, n_init, N);
      } catch (const std::system_error &) {
        n_here = N;   // no thread to be had
      }
    }
    init_nodes(0, n_here);
    std::copy(prior, prior + nC, post);
    // totals of the nodes reached, in storage that is zero without being written
    struct Free {
      void operator()(uint32_t *q) const { std::free(q); }
    };
    const std::unique_ptr<uint32_t[], Free> totals((uint32_t *)std::calloc(N * (1 + (size_t)nC), sizeof(uint32_t)));
    if (!totals) throw std::bad_alloc();
    uint32_t *const nodeTot = totals.get(), *const classTot = totals.get() + N;
    nodeTot[0] = (uint32_t)S;
    std::copy(root_tot.begin(), root_tot.end(), classTot);

    d_actA.ensure(S * sizeof(uint4));
    d_actB.ensure(S * sizeof(uint4));
    d_slotA.ensure(S * sizeof(uint32_t));
    d_slotB.ensure(S * sizeof(uint32_t));
    HIPCHK(hipMemcpyAsync(d_actA.p, d_recs.p, S * sizeof(uint4), hipMemcpyDeviceToDevice, stream));
    HIPCHK(hipMemsetAsync(d_slotA.p, 0, S * sizeof(uint32_t), stream));
    uint4 *act = d_actA.as<uint4>(), *act_next = d_actB.as<uint4>();
    uint32_t *aslot = d_slotA.as<uint32_t>(), *aslot_next = d_slotB.as<uint32_t>();
    uint64_t n_act = S;
    int32_t *acmap = nullptr, *acmap_next = nullptr;
    if constexpr (uses_context<F>::value) {
      // the device tree mirrors the host one: all -2, root posterior = priors;
      // every labelled pixel starts at the root
      d_tleft.ensure(N * sizeof(int32_t));
      d_tfeat.ensure(N * FD * sizeof(T));
      d_tthr.ensure(N * sizeof(T));
      d_tpost.ensure(N * nC * sizeof(float));
      hipLaunchKernelGGL(k_fill_i32, dim3((uint32_t)std::min<size_t>((N + 255) / 256, 65535)), dim3(256), 0, stream,
                         d_tleft.as<int32_t>(), (uint64_t)N, -2);
      HIPCHK(hipMemsetAsync(d_tpost.p, 0, N * nC * sizeof(float), stream));
      HIPCHK(hipMemcpyAsync(d_tpost.p, prior, nC * sizeof(float), hipMemcpyHostToDevice, stream));
      acmap = d_acmapA.as<int32_t>();
      acmap_next = d_acmapB.as<int32_t>();
      hipLaunchKernelGGL(k_ac_map_init, dim3((uint32_t)std::min<uint64_t>((ac_px + 255) / 256, 65535)), dim3(256), 0,
                         stream, d_acsel.as<uint8_t>(), ac_px, acmap);
      HIPCHK(hipGetLastError());
      ac = AcArgs{d_tleft.as<int32_t>(), d_tpost.as<float>(), nC, acmap, d_acoff.as<uint64_t>()};
    }

    std::vector<SlotInfo> slots{SlotInfo{0, 0u, (uint32_t)S, S > thr}};
    Event e3, e4;
    // The routed child populations of a level come back with the next
    // synchronization (the next level's split search, or the end of
    // training): the host goes on queueing the next level behind the
    // routing instead of waiting for it.  Every split node's children must
    // hold the populations of its chosen split.
    struct RouteCheck {
      bool pending = false;
      uint32_t level = 0;
      const uint32_t *counts = nullptr;   // pinned [2][nq], filled by an async copy
      std::vector<std::pair<int32_t, std::pair<uint32_t, uint32_t>>> want;   // (node, (left, right)) per slot
    } rc;
    PinnedStage route_stage;
    auto check_route = [&]() {
      if (!rc.pending) return;
      rc.pending = false;
      for (size_t q = 0; q < rc.want.size(); q++) {
        if (rc.want[q].first < 0) continue;
        if (rc.counts[2 * q] != rc.want[q].second.first || rc.counts[2 * q + 1] != rc.want[q].second.second)
          throw ParityError("routing of node " + std::to_string(rc.want[q].first) +
                            " disagrees with its histogram split");
      }
      if (ls) ls[rc.level - 1].route_ms = elapsed_ms(e3, e4);
      route_stage.reset();
    };

    for (uint32_t d = 1; d < end_depth; d++) {
      const auto t_start = std::chrono::steady_clock::now();
      pd_level_stats st{};
      st.level = d;
      st.frontier_nodes = (uint32_t)slots.size();
      if (slots.empty()) {
        if (ls) ls[d - 1] = st;
        continue;
      }
      uint64_t active = 0;
      for (const SlotInfo &s : slots)
        if (s.trainable) active += s.count;
      st.active_samples = active;
      st.evals = (double)active * nF * nT;
      uint32_t n_trainable = 0;
      for (const SlotInfo &s : slots) n_trainable += s.trainable ? 1u : 0u;
      const pd_tuning keep_tune = tune;
      tune = level_tuning(active, n_trainable);
      uint32_t ch = pick_chunk(active, nF, nT,
                               mode == PD_MODE_PER_NODE ? std::max<uint32_t>(n_trainable, 1u) : 1u);
      std::vector<uint8_t> split_flag(slots.size(), 0);
      // per-slot result: k = t * nF + f (sampler index f), FP32 gain bits, left counts
      std::vector<uint32_t> res_all(slots.size() * (nC + 2), 0u);
      std::vector<uint32_t> plain_idx, prop_idx;
      for (uint32_t q = 0; q < (uint32_t)slots.size(); q++) {
        const bool pr = mode == PD_MODE_PROPOSAL && slots[q].trainable && slots[q].count >= prop_min;
        (pr ? prop_idx : plain_idx).push_back(q);
      }
      const int lmode = mode == PD_MODE_PER_NODE ? PD_MODE_PER_NODE : PD_MODE_LEVEL_BATCHED;
      // the winners' parameters and thresholds, re-derived on the device
      std::vector<T> win_par(slots.size() * FD), win_thr(slots.size());
      {
        struct Reset {   // the pointers never outlive this level, exceptions included
          Trainer *tr;
          ~Reset() { tr->lvl_par = tr->lvl_thr = nullptr; }
        } reset{this};
        lvl_par = &win_par;
        lvl_thr = &win_thr;
        evaluate(slots, plain_idx, act, P, nF, nullptr, nullptr, bnd, tree_id, lmode, ch, classTot, d,
                 sink_x != nullptr && mode != PD_MODE_PROPOSAL, res_all, st);
        if (!prop_idx.empty()) propose(slots, prop_idx, act, P, bnd, tree_id, classTot, d, res_all, st);
      }
      check_route();   // the split search synchronized the stream
      if (d >= INIT_LEVELS && init.valid()) init.get();   // (children up to node 2^(d+1) - 2)
      if (mode == PD_MODE_PROPOSAL) {
        for (uint32_t q : plain_idx)
          if (slots[q].trainable) st.fallback_nodes++;
        st.proposal_nodes += (uint32_t)prop_idx.size();
      }
      // node update, cl_tree_trainer_impl_learn_best_featthr.hpp:101-233
      for (uint32_t q = 0; q < (uint32_t)slots.size(); q++) {
        const uint32_t n = (uint32_t)slots[q].node;
        const uint32_t *r = &res_all[(size_t)q * (nC + 2)];
        const uint32_t k = r[0];
        float g;
        std::memcpy(&g, &r[1], 4);
        const uint32_t *lh = r + 2;
        const uint32_t *tt = &classTot[(size_t)n * nC];
        if (node_k) node_k[n] = k;
        if (node_gain) node_gain[n] = g;
        if (node_gain64) node_gain64[n] = gain_f64(lh, tt, nC);
        uint32_t lS = 0, rS = 0;
        for (uint32_t c = 0; c < nC; c++) {
          lS += lh[c];
          rS += tt[c] - lh[c];
        }
        if (!lS || !rS) continue;
        const size_t L = 2 * (size_t)n + 1, R = L + 1;
        nodeTot[L] = lS;
        nodeTot[R] = rS;
        for (uint32_t c = 0; c < nC; c++) {
          classTot[L * nC + c] = lh[c];
          classTot[R * nC + c] = tt[c] - lh[c];
          post[L * nC + c] = (float)lh[c] / (float)lS;
          post[R * nC + c] = (float)(tt[c] - lh[c]) / (float)rS;
        }
        left[L] = -1;
        left[R] = -1;
        std::copy(&win_par[(size_t)q * FD], &win_par[(size_t)q * FD] + FD, &feats[(size_t)n * FD]);
        thrs[n] = win_thr[q];
        left[n] = (int32_t)L;
        split_flag[q] = 1;
        st.split_nodes++;
      }
      tune = keep_tune;
      if (d + 1 >= end_depth) {
        st.wall_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t_start).count();
        if (ls) ls[d - 1] = st;
        break;
      }
      if constexpr (uses_context<F>::value) {
        // the device tree a hook reads: this level's nodes and the children
        // (next level) as the hook will read them: leftChild -1 and their
        // posteriors (the reference's device copy reads the posteriors from
        // the wrong offset, _learn_best_featthr.hpp:270-274)
        const size_t lv0 = ((size_t)1 << (d - 1)) - 1, lvn = (size_t)1 << (d - 1);
        h2d(d_tleft.as<int32_t>() + lv0, left + lv0, lvn * sizeof(int32_t));
        h2d(d_tfeat.as<T>() + lv0 * FD, feats + lv0 * FD, lvn * FD * sizeof(T));
        h2d(d_tthr.as<T>() + lv0, thrs + lv0, lvn * sizeof(T));
        const size_t c0 = lv0 + lvn, cn = std::min(2 * lvn, N - c0);
        h2d(d_tleft.as<int32_t>() + c0, left + c0, cn * sizeof(int32_t));
        h2d(d_tpost.as<float>() + c0 * nC, post + c0 * nC, cn * nC * sizeof(float));
        // every routed pixel one level down (context: the map before the step)
        hipLaunchKernelGGL((k_ac_route_map<F>), dim3(ac_blocks), dim3(256), 0, stream, d_pixels.as<I>(),
                           d_imgs.as<ImgDesc>(), n_images, d_acblk.as<uint32_t>(), d_tfeat.as<T>(), d_tthr.as<T>(),
                           ac, acmap_next);
        HIPCHK(hipGetLastError());
      }
      // next frontier (children with more than perLeafSamplesThr samples,
      // _impl_init.hpp:343-355), in node order
      std::vector<SlotInfo> next;
      std::vector<int32_t> snext(2 * slots.size(), -1);
      std::vector<uint32_t> nbegin;   // first entry of each next slot
      uint32_t run = 0;
      for (size_t q = 0; q < slots.size(); q++) {
        if (!split_flag[q]) continue;
        for (int side = 0; side < 2; side++) {
          const int32_t ch_node = 2 * slots[q].node + 1 + side;
          const uint32_t cnt = nodeTot[ch_node];
          if (cnt > thr) {
            snext[2 * q + side] = (int32_t)next.size();
            next.push_back(SlotInfo{ch_node, run, cnt, true});
            nbegin.push_back(run);
            run += cnt;
          }
        }
      }
      const uint32_t nq = (uint32_t)slots.size();
      std::vector<uint32_t> sbegin(nq + 1);
      for (uint32_t q = 0; q < nq; q++) sbegin[q] = slots[q].begin;
      sbegin[nq] = (uint32_t)n_act;
      d_ccount.grow(2 * (size_t)nq * sizeof(uint32_t));
      d_flags.ensure((n_act + 1) * sizeof(unsigned long long));
      d_rank.ensure((n_act + 1) * sizeof(unsigned long long));
      // the level's splits by slot, in one upload
      Upload up{*this, d_route};
      const size_t u_split = up.add(split_flag.data(), nq), u_par = up.add(win_par.data(), (size_t)nq * FD * sizeof(T));
      const size_t u_thr = up.add(win_thr.data(), nq * sizeof(T));
      const size_t u_next = up.add(snext.data(), 2 * (size_t)nq * sizeof(int32_t));
      const size_t u_begin = up.add(sbegin.data(), (nq + 1) * sizeof(uint32_t));
      const size_t u_cursor = up.add(nbegin.data(), nbegin.size() * sizeof(uint32_t));
      up.stage();
      up.commit();
      size_t tmp_bytes = 0;
      HIPCHK(hipcub::DeviceScan::ExclusiveSum(nullptr, tmp_bytes, d_flags.as<unsigned long long>(),
                                              d_rank.as<unsigned long long>(), (int)(n_act + 1), stream));
      d_scan_tmp.ensure(tmp_bytes);
      HIPCHK(hipEventRecord(e3.e, stream));
      const uint32_t nb = (uint32_t)((n_act + 1 + 255) / 256);
      hipLaunchKernelGGL((k_route_flags<F>), dim3(nb), dim3(256), 0, stream, d_pixels.as<I>(), d_imgs.as<ImgDesc>(),
                         act, aslot, (uint32_t)n_act, up.template at<uint8_t>(u_split), up.template at<T>(u_par),
                         up.template at<T>(u_thr), d_flags.as<unsigned long long>(), ac);
      HIPCHK(hipGetLastError());
      HIPCHK(hipcub::DeviceScan::ExclusiveSum(d_scan_tmp.p, tmp_bytes, d_flags.as<unsigned long long>(),
                                              d_rank.as<unsigned long long>(), (int)(n_act + 1), stream));
      const uint64_t ts = std::max<uint64_t>(n_act, nq);
      hipLaunchKernelGGL(k_route_scatter, dim3((uint32_t)((ts + 255) / 256)), dim3(256), 0, stream, act, aslot,
                         (uint32_t)n_act, d_flags.as<unsigned long long>(), d_rank.as<unsigned long long>(),
                         up.template at<uint32_t>(u_begin), up.template at<int32_t>(u_next),
                         up.template at<uint32_t>(u_cursor), act_next, aslot_next, (uint32_t)S, nq,
                         d_ccount.as<uint32_t>());
      HIPCHK(hipGetLastError());
      HIPCHK(hipEventRecord(e4.e, stream));
      {
        uint32_t *cc = (uint32_t *)route_stage.alloc(2 * (size_t)nq * sizeof(uint32_t));
        HIPCHK(hipMemcpyAsync(cc, d_ccount.p, 2 * (size_t)nq * sizeof(uint32_t), hipMemcpyDeviceToHost, stream));
        rc.pending = true;
        rc.level = d;
        rc.counts = cc;
        rc.want.assign(nq, {-1, {0u, 0u}});
        for (size_t q = 0; q < slots.size(); q++) {
          if (!split_flag[q]) continue;
          const int32_t n = slots[q].node;
          rc.want[q] = {n, {nodeTot[2 * n + 1], nodeTot[2 * n + 2]}};
        }
      }
      std::swap(act, act_next);
      std::swap(aslot, aslot_next);
      if constexpr (uses_context<F>::value) {
        std::swap(acmap, acmap_next);
        ac.maps = acmap;
      }
      n_act = run;
      slots.swap(next);
      st.wall_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t_start).count();
      if (ls) ls[d - 1] = st;
    }
    if (rc.pending) {
      HIPCHK(hipStreamSynchronize(stream));
      check_route();
    }
    if (init.valid()) init.get();
  }

  // Device time (ms, mean of reps) of one level-batched histogram + split
  // pass over the training set cut into n_nodes equal consecutive shares
  // (node ids 0..n_nodes-1), with the current tuning: the autotuner's probe.
  double time_level(const pd_train_params &P, uint32_t tree_id, uint32_t n_nodes, int reps) override
  {
    if (!S) throw StateError("pd_trainer_time_level before pd_trainer_set_data");
    if constexpr (uses_context<F>::value)
      throw ArgError("this single-step entry point has no tree state for an auto-context hook");
    check_params(P, FD, sizeof(T) == 2);
    require(n_nodes >= 1 && n_nodes <= S && reps >= 1, "bad level shape");
    set_device(device);
    std::vector<SlotInfo> slots(n_nodes);
    std::vector<uint32_t> classTot((size_t)n_nodes * nC, 0u);
    for (uint32_t q = 0; q < n_nodes; q++) {
      const uint64_t b = S * q / n_nodes, e = S * (q + 1) / n_nodes;
      slots[q] = SlotInfo{(int32_t)q, (uint32_t)b, (uint32_t)(e - b), e > b};
      for (uint64_t i = b; i < e; i++) classTot[(size_t)q * nC + rec_class_host(h_recs[i])]++;
    }
    d_actA.ensure(S * sizeof(uint4));
    HIPCHK(hipMemcpyAsync(d_actA.p, d_recs.p, S * sizeof(uint4), hipMemcpyDeviceToDevice, stream));
    const Bounds<F> bnd = make_bounds<F>(P);
    std::vector<uint32_t> idx(n_nodes), res_all((size_t)n_nodes * (nC + 2));
    for (uint32_t q = 0; q < n_nodes; q++) idx[q] = q;
    const uint32_t ch = pick_chunk(S, P.n_features, P.n_thresholds);
    pd_level_stats st{};
    evaluate(slots, idx, d_actA.as<uint4>(), P, P.n_features, nullptr, nullptr, bnd, tree_id, PD_MODE_LEVEL_BATCHED,
             ch, classTot.data(), 1, false, res_all, st);   // warm-up (module load, buffers)
    st = pd_level_stats{};
    for (int r = 0; r < reps; r++)
      evaluate(slots, idx, d_actA.as<uint4>(), P, P.n_features, nullptr, nullptr, bnd, tree_id,
               PD_MODE_LEVEL_BATCHED, ch, classTot.data(), 1, false, res_all, st);
    return (st.hist_ms + st.split_ms) / reps;
  }
  static uint32_t rec_class_host(const uint4 &r) { return r.x >> 24; }

  void hist_nodes(const pd_train_params &P, uint32_t tree_id, uint32_t n_nodes, const int32_t *nodes,
                  const int32_t *sample_node, uint32_t *H_out) override
  {
    if (!S) throw StateError("pd_trainer_hist_nodes before pd_trainer_set_data");
    if constexpr (uses_context<F>::value)
      throw ArgError("this single-step entry point has no tree state for an auto-context hook");
    check_params(P, FD, sizeof(T) == 2);
    require(n_nodes >= 1 && nodes && sample_node && H_out, "bad hist_nodes arguments");
    set_device(device);
    std::map<int32_t, uint32_t> slot_of;
    for (uint32_t q = 0; q < n_nodes; q++) {
      require(slot_of.count(nodes[q]) == 0, "duplicate node id");
      slot_of[nodes[q]] = q;
    }
    std::vector<std::vector<uint4>> per(n_nodes);
    for (uint64_t s = 0; s < S; s++) {
      auto itn = slot_of.find(sample_node[s]);
      if (itn != slot_of.end()) per[itn->second].push_back(h_recs[s]);
    }
    std::vector<uint4> act;
    std::vector<SlotInfo> slots;
    for (uint32_t q = 0; q < n_nodes; q++) {
      slots.push_back(SlotInfo{nodes[q], (uint32_t)act.size(), (uint32_t)per[q].size(), true});
      act.insert(act.end(), per[q].begin(), per[q].end());
    }
    d_actA.ensure(std::max<size_t>(act.size(), 1) * sizeof(uint4));
    if (!act.empty())
      HIPCHK(hipMemcpyAsync(d_actA.p, act.data(), act.size() * sizeof(uint4), hipMemcpyHostToDevice, stream));
    const Bounds<F> bnd = make_bounds<F>(P);
    const uint32_t ch = pick_chunk(act.size(), P.n_features, P.n_thresholds);
    std::vector<uint32_t> tot((size_t)n_nodes * nC, 0u), hslots;
    hist_slice(slots, 0, slots.size(), d_actA.as<uint4>(), P, bnd, tree_id, PD_MODE_LEVEL_BATCHED, ch, tot, true,
               hslots);
    const size_t per_n = (size_t)nC * P.n_thresholds * P.n_features;
    HIPCHK(hipMemcpyAsync(H_out, d_H.p, per_n * n_nodes * sizeof(uint32_t), hipMemcpyDeviceToHost, stream));
    HIPCHK(hipStreamSynchronize(stream));
    stage.reset();
  }
};

inline TrainerBase *make_trainer(int kind, int device, uint32_t nC)
{
  switch (kind) {
    case PD_FEAT_DEPTH_F32: return new Trainer<DepthF32Feature>(device, nC);
    case PD_FEAT_DEPTH_U16: return new Trainer<DepthU16Feature>(device, nC);
    case PD_FEAT_RGBD_U16X4: return new Trainer<RGBDFeature>(device, nC);
    case PD_FEAT_DEMO_S16: return new Trainer<DemoS16Feature>(device, nC);
  }
  throw ArgError("unknown feature kind");
}

// ---------------------------------------------------------------------------
// Forest
// ---------------------------------------------------------------------------
// Device buffers of a multi-frame prediction and their sizes in bytes.
struct FrameBuffers {
  const void *pixels;
  uint64_t pixels_size;
  const uint8_t *masks;
  uint64_t masks_size;
  float *post;
  uint64_t post_size;
  int32_t *leaves;
  uint64_t leaves_size;
};

// [off, off + count) elements of elem_size bytes lie inside a buffer of
// size bytes (no wrap-around in the arithmetic).
inline bool range_inside(uint64_t off, uint64_t count, uint64_t elem_size, uint64_t size)
{
  uint64_t end, bytes;
  if (__builtin_add_overflow(off, count, &end)) return false;
  if (__builtin_mul_overflow(end, elem_size, &bytes)) return false;
  return bytes <= size;
}

struct ForestBase {
  int device = 0;
  uint32_t nC = 0;
  uint32_t n_xcc = 1;   // XCDs of the device (prediction blocks are ordered per XCD)
  hipStream_t stream = nullptr;
  virtual ~ForestBase()
  {
    if (stream) (void)hipStreamDestroy(stream);
  }
  virtual void add_tree(uint32_t depth, const int32_t *left, const void *feats, const void *thrs,
                        const float *posts) = 0;
  virtual int n_trees() const = 0;
  virtual void predict_host(int tree_index, const void *image, uint32_t w, uint32_t h, const uint8_t *mask,
                            int32_t *leaves, float *post) = 0;
  virtual void predict_frames(uint32_t n_frames, const FrameBuffers &fb, const uint64_t *img_off,
                              const uint32_t *widths, const uint32_t *heights, const uint64_t *mask_off,
                              const uint64_t *post_off, const uint64_t *leaf_off, int use_graph,
                              float *kernel_ms) = 0;
  // The same launch with the frame table in caller-provided device memory
  // (table_cap entries): allocates no device memory.
  virtual void predict_frames_table(uint32_t n_frames, const FrameBuffers &fb, const uint64_t *img_off,
                                    const uint32_t *widths, const uint32_t *heights, const uint64_t *mask_off,
                                    const uint64_t *post_off, const uint64_t *leaf_off, FrameDesc *d_table,
                                    uint32_t table_cap) = 0;
};

template <class F>
struct Forest final : ForestBase {
  using T = typename F::FeatType;
  using I = typename F::ImgType;
  using Rec = NodeRec<T, F::FeatDim>;
  // compact forest: existing nodes only (breadth first, children adjacent)
  // and one leaf table per tree (original node id, posterior row)
  std::vector<Rec> h_nodes;
  std::vector<float> h_leaf_post;
  std::vector<int32_t> h_leaf_id;
  std::vector<uint32_t> h_tree_off, h_leaf_off;
  std::vector<uint32_t> depths;
  uint32_t max_depth = 1;
  bool fast_nodes = true;   // every node's offset parameters are within RECIP_MAX
  DevBuf d_nodes, d_leaf_post, d_leaf_id, d_tree_off, d_leaf_off;
  DevBuf d_img, d_mask, d_out, d_leaf, d_frames;
  // auto-context hooks: the trees' breadth-first arrays (the hook reads them)
  std::vector<int32_t> h_ac_left;
  std::vector<T> h_ac_feat, h_ac_thr;
  std::vector<float> h_ac_post;
  std::vector<uint64_t> h_ac_off;   // first node of each tree
  DevBuf d_ac_left, d_ac_feat, d_ac_thr, d_ac_post, d_ac_mapA, d_ac_mapB, d_ac_img, d_ac_off0, d_ac_blk0;
  bool ac_dirty = false;
  // captured graph for predict_frames (keyed by the launch arguments)
  hipGraphExec_t gexec = nullptr;
  hipGraph_t graph = nullptr;
  std::vector<uint64_t> gkey;

  Forest(int dev, uint32_t ncl)
  {
    device = dev;
    nC = ncl;
    set_device(device);
    HIPCHK(hipStreamCreate(&stream));
    int xcc = 1;
    if (hipDeviceGetAttribute(&xcc, hipDeviceAttributeNumberOfXccs, device) != hipSuccess || xcc < 1) {
      (void)hipGetLastError();
      xcc = 1;
    }
    n_xcc = (uint32_t)xcc;
  }
  ~Forest() override
  {
    if (gexec) (void)hipGraphExecDestroy(gexec);
    if (graph) (void)hipGraphDestroy(graph);
  }
  int n_trees() const override { return (int)depths.size(); }

  void add_tree(uint32_t depth, const int32_t *left, const void *feats_v, const void *thrs_v,
                const float *posts) override
  {
    require(depth >= 1 && depth <= 24, "tree depth must be in [1, 24]");
    require(left && feats_v && thrs_v && posts, "null tree array");
    const T *feats = (const T *)feats_v;
    const T *thrs = (const T *)thrs_v;
    const size_t N = ((size_t)1 << depth) - 1;
    // every split node must point at its own children (2i+1, 2i+2 < N)
    for (size_t i = 0; i < N; i++)
      if (left[i] >= 0) require((size_t)left[i] == 2 * i + 1 && 2 * i + 2 < N, "malformed tree: bad leftChild");
    set_device(device);
    // compact the heap layout (cl_classifier_impl.hpp:153-168 uploads the
    // whole 2^D - 1 arrays): breadth-first walk of the existing nodes, a
    // split node's children placed side by side
    if constexpr (uses_context<F>::value) {
      h_ac_off.push_back(h_ac_left.size());
      h_ac_left.insert(h_ac_left.end(), left, left + N);
      h_ac_feat.insert(h_ac_feat.end(), feats, feats + N * F::FeatDim);
      h_ac_thr.insert(h_ac_thr.end(), thrs, thrs + N);
      h_ac_post.insert(h_ac_post.end(), posts, posts + N * nC);
      ac_dirty = true;
    }
    const uint32_t base = (uint32_t)h_nodes.size(), leaf_base = (uint32_t)h_leaf_id.size();
    require((uint64_t)h_nodes.size() + N < (1ull << 31), "forest too large");
    std::vector<int64_t> order{0};   // original ids in compact order
    for (size_t k = 0; k < order.size(); k++) {
      const int64_t i = order[k];
      Rec r{};
      if (left[i] >= 0) {
        r.left = (int32_t)order.size();
        order.push_back(2 * i + 1);
        order.push_back(2 * i + 2);
        r.thr = thrs[i];
        for (int j = 0; j < F::FeatDim; j++) r.p[j] = feats[i * F::FeatDim + j];
        if constexpr (has_fast<F>::value)
          for (int j = 0; j < 4; j++) fast_nodes = fast_nodes && std::fabs((float)r.p[j]) <= RECIP_MAX;
      } else {
        const uint32_t leaf = (uint32_t)h_leaf_id.size() - leaf_base;
        r.left = -1 - (int32_t)leaf;
        h_leaf_id.push_back((int32_t)i);
        h_leaf_post.insert(h_leaf_post.end(), posts + (size_t)i * nC, posts + (size_t)(i + 1) * nC);
        h_leaf_post.resize(h_leaf_post.size() + (((nC + 3u) & ~3u) - nC), 0.0f);   // row padding
      }
      h_nodes.push_back(r);
    }
    h_tree_off.push_back(base);
    h_leaf_off.push_back(leaf_base);
    depths.push_back(depth);
    max_depth = std::max(max_depth, depth);
    d_nodes.ensure(h_nodes.size() * sizeof(Rec));
    d_leaf_post.ensure(h_leaf_post.size() * sizeof(float));
    d_leaf_id.ensure(h_leaf_id.size() * sizeof(int32_t));
    d_tree_off.ensure(h_tree_off.size() * sizeof(uint32_t));
    d_leaf_off.ensure(h_leaf_off.size() * sizeof(uint32_t));
    HIPCHK(hipMemcpy(d_nodes.p, h_nodes.data(), h_nodes.size() * sizeof(Rec), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(d_leaf_post.p, h_leaf_post.data(), h_leaf_post.size() * sizeof(float), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(d_leaf_id.p, h_leaf_id.data(), h_leaf_id.size() * sizeof(int32_t), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(d_tree_off.p, h_tree_off.data(), h_tree_off.size() * sizeof(uint32_t), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(d_leaf_off.p, h_leaf_off.data(), h_leaf_off.size() * sizeof(uint32_t), hipMemcpyHostToDevice));
    if (gexec) {
      (void)hipGraphExecDestroy(gexec);
      gexec = nullptr;
    }
    if (graph) {
      (void)hipGraphDestroy(graph);
      graph = nullptr;
    }
    gkey.clear();
  }

  template <int NCM>
  void launch(uint32_t blocks, const I *pix, const FrameDesc *frames, uint32_t n_frames, const uint8_t *masks,
              uint32_t tree0, uint32_t ntr, uint32_t steps, float *out_post, int32_t *out_leaf)
  {
    if constexpr (has_fast<F>::value) {
      if (fast_nodes) return launch_k<NCM, true>(blocks, pix, frames, n_frames, masks, tree0, ntr, steps, out_post, out_leaf);
    }
    launch_k<NCM, false>(blocks, pix, frames, n_frames, masks, tree0, ntr, steps, out_post, out_leaf);
  }
  template <int NCM, bool FAST>
  void launch_k(uint32_t blocks, const I *pix, const FrameDesc *frames, uint32_t n_frames, const uint8_t *masks,
                uint32_t tree0, uint32_t ntr, uint32_t steps, float *out_post, int32_t *out_leaf)
  {
    const uint32_t per_xcc = (blocks + n_xcc - 1) / n_xcc;
    hipLaunchKernelGGL((k_predict<F, NCM, FAST>), dim3(per_xcc * n_xcc), dim3(256), 0, stream, pix, frames, n_frames, blocks,
                       n_xcc, per_xcc, masks, d_nodes.as<Rec>(), d_tree_off.as<uint32_t>() + tree0, ntr, steps,
                       d_leaf_post.as<float>(), d_leaf_id.as<int32_t>(), d_leaf_off.as<uint32_t>() + tree0, nC,
                       out_post, out_leaf);
    HIPCHK(hipGetLastError());
  }
  void launch_any(uint32_t blocks, const I *pix, const FrameDesc *frames, uint32_t n_frames, const uint8_t *masks,
                  uint32_t tree0, uint32_t ntr, uint32_t steps, float *out_post, int32_t *out_leaf)
  {
#if PD_KERNEL_SET_LIGHT
    if (nC <= 16) launch<16>(blocks, pix, frames, n_frames, masks, tree0, ntr, steps, out_post, out_leaf);
#else
    if (nC <= 8) launch<8>(blocks, pix, frames, n_frames, masks, tree0, ntr, steps, out_post, out_leaf);
    else if (nC <= 16) launch<16>(blocks, pix, frames, n_frames, masks, tree0, ntr, steps, out_post, out_leaf);
#endif
#if !PD_KERNEL_SET_LIGHT
    else if (nC <= 32) launch<32>(blocks, pix, frames, n_frames, masks, tree0, ntr, steps, out_post, out_leaf);
#endif
    else launch<64>(blocks, pix, frames, n_frames, masks, tree0, ntr, steps, out_post, out_leaf);
  }

  // Auto-context prediction of one frame resident on the device: per tree,
  // depth - 1 passes over the frame's routed pixels (a node-id map, the hook
  // reading the map of the pass before), then the leaf ids / the posterior
  // sum in tree order (cl_classifier_impl.hpp:356-557 runs the same passes).
  void predict_ac_frame(const I *d_pix, uint32_t w, uint32_t h, const uint8_t *d_mask, int tree_index,
                        int32_t *d_leaves, float *d_post)
  {
    if (ac_dirty) {
      auto up = [&](DevBuf &b, const void *src, size_t bytes) {
        b.ensure(std::max<size_t>(bytes, 16));
        HIPCHK(hipMemcpyAsync(b.p, src, bytes, hipMemcpyHostToDevice, stream));
      };
      up(d_ac_left, h_ac_left.data(), h_ac_left.size() * sizeof(int32_t));
      up(d_ac_feat, h_ac_feat.data(), h_ac_feat.size() * sizeof(T));
      up(d_ac_thr, h_ac_thr.data(), h_ac_thr.size() * sizeof(T));
      up(d_ac_post, h_ac_post.data(), h_ac_post.size() * sizeof(float));
      ac_dirty = false;
    }
    const uint32_t npx = w * h;
    const uint32_t blocks = (npx + 255) / 256;
    d_ac_mapA.ensure((size_t)npx * sizeof(int32_t));
    d_ac_mapB.ensure((size_t)npx * sizeof(int32_t));
    const ImgDesc idsc{0, w, h};
    const uint64_t zero64 = 0;
    const uint32_t zero32 = 0;
    d_ac_img.ensure(sizeof(ImgDesc));
    d_ac_off0.ensure(sizeof(uint64_t));
    d_ac_blk0.ensure(sizeof(uint32_t));
    HIPCHK(hipMemcpyAsync(d_ac_img.p, &idsc, sizeof(ImgDesc), hipMemcpyHostToDevice, stream));
    HIPCHK(hipMemcpyAsync(d_ac_off0.p, &zero64, sizeof(uint64_t), hipMemcpyHostToDevice, stream));
    HIPCHK(hipMemcpyAsync(d_ac_blk0.p, &zero32, sizeof(uint32_t), hipMemcpyHostToDevice, stream));
    const int t0 = tree_index >= 0 ? tree_index : 0;
    const int t1 = tree_index >= 0 ? tree_index + 1 : (int)depths.size();
    for (int t = t0; t < t1; t++) {
      int32_t *a = d_ac_mapA.as<int32_t>(), *b = d_ac_mapB.as<int32_t>();
      hipLaunchKernelGGL(k_ac_map_init, dim3(std::max<uint32_t>(1, std::min<uint32_t>(blocks, 65535))), dim3(256), 0,
                         stream, d_mask, (uint64_t)npx, a);
      const uint64_t o = h_ac_off[t];
      for (uint32_t s = 0; s + 1 < depths[t]; s++) {
        const AcArgs acx{d_ac_left.as<int32_t>() + o, d_ac_post.as<float>() + o * nC, nC, a, d_ac_off0.as<uint64_t>()};
        hipLaunchKernelGGL((k_ac_route_map<F>), dim3(blocks), dim3(256), 0, stream, d_pix, d_ac_img.as<ImgDesc>(), 1u,
                           d_ac_blk0.as<uint32_t>(), d_ac_feat.as<T>() + o * F::FeatDim, d_ac_thr.as<T>() + o, acx, b);
        std::swap(a, b);
      }
      HIPCHK(hipGetLastError());
      if (d_leaves && tree_index >= 0)
        HIPCHK(hipMemcpyAsync(d_leaves, a, (size_t)npx * sizeof(int32_t), hipMemcpyDeviceToDevice, stream));
      if (d_post)
        hipLaunchKernelGGL(k_ac_post_add, dim3(blocks), dim3(256), 0, stream, a, npx, d_ac_post.as<float>() + o * nC,
                           nC, t == t0 ? 1 : 0, d_post);
      if (d_post && t + 1 == t1)
        hipLaunchKernelGGL(k_ac_post_finish, dim3(blocks), dim3(256), 0, stream, a, npx, nC,
                           (float)depths.size(), d_post);
    }
    HIPCHK(hipGetLastError());
  }

  void predict_host(int tree_index, const void *image, uint32_t w, uint32_t h, const uint8_t *mask,
                    int32_t *leaves, float *post) override
  {
    if constexpr (uses_context<F>::value) {
      require(!depths.empty(), "forest has no trees");
      require(image && w >= 1 && h >= 1 && w < 65536 && h < 65536, "bad image");
      set_device(device);
      const size_t npx = (size_t)w * h;
      d_img.ensure(npx * F::nChannels * sizeof(I));
      HIPCHK(hipMemcpyAsync(d_img.p, image, npx * F::nChannels * sizeof(I), hipMemcpyHostToDevice, stream));
      if (mask) {
        d_mask.ensure(npx);
        HIPCHK(hipMemcpyAsync(d_mask.p, mask, npx, hipMemcpyHostToDevice, stream));
      }
      if (leaves) {
        require(tree_index >= 0 && tree_index < (int)depths.size(), "tree index out of range");
        d_leaf.ensure(npx * sizeof(int32_t));
        predict_ac_frame(d_img.as<I>(), w, h, mask ? d_mask.as<uint8_t>() : nullptr, tree_index,
                         d_leaf.as<int32_t>(), nullptr);
        HIPCHK(hipMemcpyAsync(leaves, d_leaf.p, npx * sizeof(int32_t), hipMemcpyDeviceToHost, stream));
      }
      if (post) {
        d_out.ensure(npx * nC * sizeof(float));
        predict_ac_frame(d_img.as<I>(), w, h, mask ? d_mask.as<uint8_t>() : nullptr, -1, nullptr,
                         d_out.as<float>());
        HIPCHK(hipMemcpyAsync(post, d_out.p, npx * nC * sizeof(float), hipMemcpyDeviceToHost, stream));
      }
      HIPCHK(hipStreamSynchronize(stream));
      return;
    }
    predict_host_plain(tree_index, image, w, h, mask, leaves, post);
  }

  void predict_host_plain(int tree_index, const void *image, uint32_t w, uint32_t h, const uint8_t *mask,
                          int32_t *leaves, float *post)
  {
    require(!depths.empty(), "forest has no trees");
    require(image && w >= 1 && h >= 1 && w < 65536 && h < 65536, "bad image");
    require((uint64_t)w * h * F::nChannels * sizeof(I) < (1ull << 32), "an image must be smaller than 4 GiB");
    set_device(device);
    const size_t npx = (size_t)w * h;
    d_img.ensure(npx * F::nChannels * sizeof(I));
    HIPCHK(hipMemcpyAsync(d_img.p, image, npx * F::nChannels * sizeof(I), hipMemcpyHostToDevice, stream));
    if (mask) {
      d_mask.ensure(npx);
      HIPCHK(hipMemcpyAsync(d_mask.p, mask, npx, hipMemcpyHostToDevice, stream));
    }
    FrameDesc fdsc{};
    fdsc.w = w;
    fdsc.h = h;
    d_frames.ensure(sizeof(FrameDesc));
    HIPCHK(hipMemcpyAsync(d_frames.p, &fdsc, sizeof(FrameDesc), hipMemcpyHostToDevice, stream));
    const uint32_t blocks = (uint32_t)((npx + 255) / 256);
    if (leaves) {
      require(tree_index >= 0 && tree_index < (int)depths.size(), "tree index out of range");
      d_leaf.ensure(npx * sizeof(int32_t));
      launch_any(blocks, d_img.as<I>(), d_frames.as<FrameDesc>(), 1, mask ? d_mask.as<uint8_t>() : nullptr,
                 (uint32_t)tree_index, 1, depths[tree_index] - 1, nullptr, d_leaf.as<int32_t>());
      HIPCHK(hipMemcpyAsync(leaves, d_leaf.p, npx * sizeof(int32_t), hipMemcpyDeviceToHost, stream));
    }
    if (post) {
      d_out.ensure(npx * nC * sizeof(float));
      launch_any(blocks, d_img.as<I>(), d_frames.as<FrameDesc>(), 1, mask ? d_mask.as<uint8_t>() : nullptr, 0,
                 (uint32_t)depths.size(), max_depth - 1, d_out.as<float>(), nullptr);
      HIPCHK(hipMemcpyAsync(post, d_out.p, npx * nC * sizeof(float), hipMemcpyDeviceToHost, stream));
    }
    HIPCHK(hipStreamSynchronize(stream));
  }

  // Every frame's range in every given buffer lies inside that buffer.
  void check_frames(uint32_t n_frames, const FrameBuffers &fb, const uint64_t *img_off, const uint32_t *widths,
                    const uint32_t *heights, const uint64_t *mask_off, const uint64_t *post_off,
                    const uint64_t *leaf_off) const
  {
    for (uint32_t i = 0; i < n_frames; i++) {
      require(widths[i] >= 1 && heights[i] >= 1 && widths[i] < 65536 && heights[i] < 65536, "bad frame size");
      const uint64_t npx = (uint64_t)widths[i] * heights[i];
      require(range_inside(img_off[i], npx * F::nChannels, sizeof(I), fb.pixels_size),
              "frame " + std::to_string(i) + ": pixel range outside d_pixels");
      if (fb.masks)
        require(range_inside(mask_off[i], npx, 1, fb.masks_size),
                "frame " + std::to_string(i) + ": mask range outside d_masks");
      if (fb.post)
        require(range_inside(post_off[i], npx * nC, sizeof(float), fb.post_size),
                "frame " + std::to_string(i) + ": posterior range outside d_post");
      if (fb.leaves)
        require(range_inside(leaf_off[i], npx * depths.size(), sizeof(int32_t), fb.leaves_size),
                "frame " + std::to_string(i) + ": leaf range outside d_leaves");
    }
  }

  // Host-side frame table of a multi-frame launch (frame ranges already
  // checked against the buffers); returns the launch's block count.
  uint32_t frame_table(uint32_t n_frames, const FrameBuffers &fb, const uint64_t *img_off, const uint32_t *widths,
                       const uint32_t *heights, const uint64_t *mask_off, const uint64_t *post_off,
                       const uint64_t *leaf_off, std::vector<FrameDesc> &fr) const
  {
    fr.assign(n_frames, FrameDesc{});
    uint64_t blocks = 0;
    for (uint32_t i = 0; i < n_frames; i++) {
      require(widths[i] >= 1 && heights[i] >= 1 && widths[i] < 65536 && heights[i] < 65536, "bad frame size");
      require((uint64_t)widths[i] * heights[i] * F::nChannels * sizeof(I) < (1ull << 32),
              "a frame must be smaller than 4 GiB");
      fr[i].img_off = img_off[i];
      fr[i].post_off = fb.post ? post_off[i] : 0;
      fr[i].leaf_off = fb.leaves ? leaf_off[i] : 0;
      fr[i].mask_off = fb.masks ? mask_off[i] : 0;
      fr[i].w = widths[i];
      fr[i].h = heights[i];
      fr[i].block0 = (uint32_t)blocks;
      blocks += ((uint64_t)widths[i] * heights[i] + 255) / 256;
      require(blocks < (1ull << 31) - 64, "too many pixels in one launch");
    }
    return (uint32_t)blocks;
  }

  void predict_frames_table(uint32_t n_frames, const FrameBuffers &fb, const uint64_t *img_off,
                            const uint32_t *widths, const uint32_t *heights, const uint64_t *mask_off,
                            const uint64_t *post_off, const uint64_t *leaf_off, FrameDesc *d_table,
                            uint32_t table_cap) override
  {
    require(!depths.empty(), "forest has no trees");
    require(n_frames >= 1 && fb.pixels && img_off && widths && heights, "bad frame arguments");
    require(n_frames <= table_cap, "at most " + std::to_string(table_cap) + " frames per call");
    require(fb.post || fb.leaves, "no output requested");
    require(!fb.post || post_off, "post_offsets missing");
    require(!fb.leaves || leaf_off, "leaf_offsets missing");
    require(!fb.masks || mask_off, "mask_offsets missing");
    require(!uses_context<F>::value, "auto-context hooks need node maps: use pd_forest_predict_frames_dev");
    check_frames(n_frames, fb, img_off, widths, heights, mask_off, post_off, leaf_off);
    set_device(device);
    std::vector<FrameDesc> fr;
    const uint32_t blocks = frame_table(n_frames, fb, img_off, widths, heights, mask_off, post_off, leaf_off, fr);
    HIPCHK(hipMemcpyAsync(d_table, fr.data(), n_frames * sizeof(FrameDesc), hipMemcpyHostToDevice, stream));
    launch_any(blocks, (const I *)fb.pixels, d_table, n_frames, fb.masks, 0, (uint32_t)depths.size(),
               max_depth - 1, fb.post, fb.leaves);
    HIPCHK(hipStreamSynchronize(stream));
  }

  void predict_frames(uint32_t n_frames, const FrameBuffers &fb, const uint64_t *img_off, const uint32_t *widths,
                      const uint32_t *heights, const uint64_t *mask_off, const uint64_t *post_off,
                      const uint64_t *leaf_off, int use_graph, float *kernel_ms) override
  {
    const void *d_pixels = fb.pixels;
    const uint8_t *d_masks = fb.masks;
    float *d_post = fb.post;
    int32_t *d_leaves = fb.leaves;
    require(!depths.empty(), "forest has no trees");
    require(n_frames >= 1 && d_pixels && img_off && widths && heights, "bad frame arguments");
    require(d_post || d_leaves, "no output requested");
    require(!d_post || post_off, "post_offsets missing");
    require(!d_leaves || leaf_off, "leaf_offsets missing");
    require(!d_masks || mask_off, "mask_offsets missing");
    check_frames(n_frames, fb, img_off, widths, heights, mask_off, post_off, leaf_off);
    set_device(device);
    if constexpr (uses_context<F>::value) {
      require(!use_graph, "auto-context hooks predict frame by frame (no graph capture)");
      require(!d_leaves, "auto-context hooks: leaf ids per tree through pd_forest_predict_leaves");
      Event a, b;
      HIPCHK(hipEventRecord(a.e, stream));
      for (uint32_t i = 0; i < n_frames; i++) {
        require(widths[i] >= 1 && heights[i] >= 1 && widths[i] < 65536 && heights[i] < 65536, "bad frame size");
        predict_ac_frame((const I *)d_pixels + img_off[i], widths[i], heights[i], d_masks ? d_masks + mask_off[i] : nullptr,
                         -1, nullptr, d_post + post_off[i]);
      }
      HIPCHK(hipEventRecord(b.e, stream));
      HIPCHK(hipEventSynchronize(b.e));
      if (kernel_ms) *kernel_ms = (float)elapsed_ms(a, b);
      return;
    }
    std::vector<FrameDesc> fr;
    const uint32_t blocks = frame_table(n_frames, fb, img_off, widths, heights, mask_off, post_off, leaf_off, fr);
    std::vector<uint64_t> key;
    key.push_back((uint64_t)(uintptr_t)d_pixels);
    key.push_back((uint64_t)(uintptr_t)d_masks);
    key.push_back((uint64_t)(uintptr_t)d_post);
    key.push_back((uint64_t)(uintptr_t)d_leaves);
    for (const FrameDesc &f : fr) {
      key.push_back(f.img_off);
      key.push_back(f.post_off);
      key.push_back(f.leaf_off);
      key.push_back(f.mask_off);
      key.push_back(((uint64_t)f.w << 32) | f.h);
    }
    const bool same = use_graph && gexec && key == gkey;
    if (!same) {
      d_frames.ensure(n_frames * sizeof(FrameDesc));
      HIPCHK(hipMemcpyAsync(d_frames.p, fr.data(), n_frames * sizeof(FrameDesc), hipMemcpyHostToDevice, stream));
      HIPCHK(hipStreamSynchronize(stream));
    }
    Event a, b;
    HIPCHK(hipEventRecord(a.e, stream));
    if (!use_graph) {
      launch_any(blocks, (const I *)d_pixels, d_frames.as<FrameDesc>(), n_frames, d_masks, 0,
                 (uint32_t)depths.size(), max_depth - 1, d_post, d_leaves);
    } else {
      if (!same) {
        if (gexec) (void)hipGraphExecDestroy(gexec);
        if (graph) (void)hipGraphDestroy(graph);
        gexec = nullptr;
        graph = nullptr;
        hipStream_t cs;
        HIPCHK(hipStreamCreate(&cs));
        HIPCHK(hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal));
        hipStream_t keep = stream;
        stream = cs;
        try {
          launch_any(blocks, (const I *)d_pixels, d_frames.as<FrameDesc>(), n_frames, d_masks, 0,
                     (uint32_t)depths.size(), max_depth - 1, d_post, d_leaves);
        } catch (...) {
          stream = keep;
          hipGraph_t g;
          (void)hipStreamEndCapture(cs, &g);
          (void)hipStreamDestroy(cs);
          throw;
        }
        stream = keep;
        HIPCHK(hipStreamEndCapture(cs, &graph));
        HIPCHK(hipStreamDestroy(cs));
        HIPCHK(hipGraphInstantiate(&gexec, graph, nullptr, nullptr, 0));
        gkey = key;
      }
      HIPCHK(hipGraphLaunch(gexec, stream));
    }
    HIPCHK(hipEventRecord(b.e, stream));
    HIPCHK(hipEventSynchronize(b.e));
    if (kernel_ms) *kernel_ms = (float)elapsed_ms(a, b);
  }
};

inline ForestBase *make_forest(int kind, int device, uint32_t nC)
{
  switch (kind) {
    case PD_FEAT_DEPTH_F32: return new Forest<DepthF32Feature>(device, nC);
    case PD_FEAT_DEPTH_U16: return new Forest<DepthU16Feature>(device, nC);
    case PD_FEAT_RGBD_U16X4: return new Forest<RGBDFeature>(device, nC);
    case PD_FEAT_DEMO_S16: return new Forest<DemoS16Feature>(device, nC);
  }
  throw ArgError("unknown feature kind");
}

template <class F>
void candidate_tables_t(const pd_train_params &P, uint32_t tree, uint32_t n_nodes, const int32_t *nodes,
                        void *params_out, void *thr_out)
{
  using T = typename F::FeatType;
  check_params(P, F::FeatDim, sizeof(T) == 2);
  const size_t nfe = (size_t)n_nodes * P.n_features;
  DevBuf dn, dp, dt;
  dn.ensure(n_nodes * sizeof(int32_t));
  dp.ensure(nfe * F::FeatDim * sizeof(T));
  dt.ensure(nfe * P.n_thresholds * sizeof(T));
  HIPCHK(hipMemcpy(dn.p, nodes, n_nodes * sizeof(int32_t), hipMemcpyHostToDevice));
  hipLaunchKernelGGL((k_candidates<F>), dim3((uint32_t)((nfe + 255) / 256)), dim3(256), 0, nullptr,
                     tree, dn.as<int32_t>(), n_nodes, P.n_features, P.n_thresholds, make_bounds<F>(P), dp.as<T>(),
                     dt.as<T>());
  HIPCHK(hipGetLastError());
  HIPCHK(hipMemcpy(params_out, dp.p, nfe * F::FeatDim * sizeof(T), hipMemcpyDeviceToHost));
  HIPCHK(hipMemcpy(thr_out, dt.p, nfe * P.n_thresholds * sizeof(T), hipMemcpyDeviceToHost));
}

template <class F>
void feature_eval_t(const void *image, uint32_t w, uint32_t h, uint32_t n, const int32_t *xy, const void *params,
                    void *out)
{
  using T = typename F::FeatType;
  using I = typename F::ImgType;
  DevBuf di, dx, dp, dout;
  const size_t npx = (size_t)w * h * F::nChannels;
  di.ensure(npx * sizeof(I));
  dx.ensure((size_t)n * 2 * sizeof(int32_t));
  dp.ensure((size_t)n * F::FeatDim * sizeof(T));
  dout.ensure((size_t)n * sizeof(T));
  for (uint32_t i = 0; i < n; i++)
    require(xy[2 * i] >= 0 && (uint32_t)xy[2 * i] < w && xy[2 * i + 1] >= 0 && (uint32_t)xy[2 * i + 1] < h,
            "evaluation pixel outside the image");
  HIPCHK(hipMemcpy(di.p, image, npx * sizeof(I), hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(dx.p, xy, (size_t)n * 2 * sizeof(int32_t), hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(dp.p, params, (size_t)n * F::FeatDim * sizeof(T), hipMemcpyHostToDevice));
  hipLaunchKernelGGL((k_feature_eval<F>), dim3((n + 255) / 256), dim3(256), 0, nullptr, di.as<I>(), w, h,
                     dx.as<int32_t>(), dp.as<T>(), n, dout.as<T>());
  HIPCHK(hipGetLastError());
  HIPCHK(hipMemcpy(out, dout.p, (size_t)n * sizeof(T), hipMemcpyDeviceToHost));
}

}  // namespace engine
}  // namespace pd

// Opaque handles of the C ABI.
struct pd_trainer {
  std::unique_ptr<pd::engine::TrainerBase> impl;
};
struct pd_mlp {
  std::unique_ptr<pd::engine::MlpNet> impl;
};
struct pd_forest {
  std::unique_ptr<pd::engine::ForestBase> impl;
};
