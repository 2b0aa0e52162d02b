// C ABI of the gfx950 random-forest hot path (include/padenti_hip.h) for the
// built-in feature hooks; the engine itself is pd_engine.hpp.
#include "padenti/pd_engine.hpp"

#include <map>
#include <mutex>

using namespace pd;
using namespace pd::engine;


extern "C" {

const char *pd_last_error(void) { return g_err.c_str(); }
int pd_version(void) { return 100; }

int pd_device_count(void)
{
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return n;
}

int pd_trainer_create(pd_trainer **out, int device, int feature_kind, uint32_t n_classes)
{
  return guarded([&] {
    require(out != nullptr, "null output handle");
    require(n_classes >= 1 && n_classes <= 64, "n_classes must be in [1, 64]");
    std::unique_ptr<pd_trainer> t(new pd_trainer);
    t->impl.reset(make_trainer(feature_kind, device, n_classes));
    *out = t.release();
  });
}

int pd_trainer_destroy(pd_trainer *tr)
{
  return guarded([&] { delete tr; });
}

int pd_trainer_set_data(pd_trainer *tr, uint32_t n_images, const void *pixels, const uint64_t *img_offsets,
                        const uint32_t *widths, const uint32_t *heights, const uint8_t *labels,
                        const uint64_t *label_offsets, const uint32_t *samples, const uint64_t *sample_offsets,
                        const uint32_t *n_samples)
{
  return guarded([&] {
    require(tr != nullptr, "null trainer");
    tr->impl->set_data(n_images, pixels, img_offsets, widths, heights, labels, label_offsets, samples, sample_offsets,
                       n_samples);
  });
}

int pd_trainer_set_hist_budget(pd_trainer *tr, uint64_t bytes)
{
  return guarded([&] {
    require(tr != nullptr && bytes >= 4096, "bad histogram budget");
    tr->impl->hist_budget = bytes;
  });
}

int pd_trainer_set_chunk(pd_trainer *tr, uint32_t samples_per_chunk)
{
  return guarded([&] {
    require(tr != nullptr && samples_per_chunk <= 32768, "chunk must be <= 32768 samples");
    tr->impl->chunk = samples_per_chunk;
  });
}

int pd_trainer_set_probe_order(pd_trainer *tr, int enable)
{
  return guarded([&] {
    require(tr != nullptr, "null trainer");
    tr->impl->probe_order = enable != 0;
  });
}

int pd_trainer_set_wide_bins(pd_trainer *tr, int enable)
{
  return guarded([&] {
    require(tr != nullptr, "null trainer");
    tr->impl->wide_bins = enable != 0;
  });
}

int pd_trainer_set_tuning(pd_trainer *tr, const pd_tuning *tuning)
{
  return guarded([&] {
    require(tr && tuning, "null argument");
    require(tuning->waves == 4 || tuning->waves == 8 || tuning->waves == 16, "waves must be 4, 8 or 16");
    require(tuning->blocks_per_cu >= 1 && tuning->blocks_per_cu <= 256, "blocks_per_cu must be in [1, 256]");
    require(tuning->samples_per_wave <= 2 || tuning->samples_per_wave == 4, "samples_per_wave must be 1, 2 or 4");
    require(tuning->bins <= 2, "bins must be 0, 1 or 2");
    tr->impl->tune = *tuning;
    if (tr->impl->tune.samples_per_wave == 0) tr->impl->tune.samples_per_wave = 1;
  });
}

int pd_trainer_set_tuning_rules(pd_trainer *tr, uint32_t n_rules, const pd_tuning_rule *rules)
{
  return guarded([&] {
    require(tr != nullptr && (n_rules == 0 || rules != nullptr), "null argument");
    require(n_rules <= 64, "at most 64 tuning rules");
    std::vector<pd_tuning_rule> v(rules, rules + n_rules);
    for (size_t i = 0; i < v.size(); i++) {
      const pd_tuning &t = v[i].tuning;
      require(t.waves == 4 || t.waves == 8 || t.waves == 16, "waves must be 4, 8 or 16");
      require(t.blocks_per_cu >= 1 && t.blocks_per_cu <= 256, "blocks_per_cu must be in [1, 256]");
      require(t.samples_per_wave <= 2 || t.samples_per_wave == 4, "samples_per_wave must be 1, 2 or 4");
      require(t.bins <= 2, "bins must be 0, 1 or 2");
      require(i == 0 || v[i].min_samples_per_node < v[i - 1].min_samples_per_node,
              "rules must have decreasing min_samples_per_node");
      if (v[i].tuning.samples_per_wave == 0) v[i].tuning.samples_per_wave = 1;
    }
    tr->impl->tune_rules = v;
  });
}

int pd_trainer_get_tuning(pd_trainer *tr, pd_tuning *tuning)
{
  return guarded([&] {
    require(tr && tuning, "null argument");
    *tuning = tr->impl->tune;
  });
}

int pd_trainer_time_level(pd_trainer *tr, const pd_train_params *params, uint32_t tree_id, uint32_t n_nodes, int reps,
                          double *ms)
{
  return guarded([&] {
    require(tr && params && ms, "null argument");
    *ms = tr->impl->time_level(*params, tree_id, n_nodes, reps);
  });
}

int pd_trainer_train(pd_trainer *tr, const pd_train_params *params, uint32_t tree_id, uint32_t tree_depth,
                     uint32_t end_depth, int mode, const float *root_prior, int32_t *left_children, void *features,
                     void *thresholds, float *posteriors, uint32_t *node_k, float *node_gain, double *node_gain64,
                     pd_level_stats *level_stats)
{
  return guarded([&] {
    require(tr != nullptr && params != nullptr, "null trainer or params");
    tr->impl->train(*params, tree_id, tree_depth, end_depth, mode, root_prior, left_children, features, thresholds,
                    posteriors, node_k, node_gain, node_gain64, level_stats);
  });
}

int pd_trainer_hist_nodes(pd_trainer *tr, const pd_train_params *params, uint32_t tree_id, uint32_t n_nodes,
                          const int32_t *node_ids, const int32_t *sample_node, uint32_t *H_out)
{
  return guarded([&] {
    require(tr != nullptr && params != nullptr, "null trainer or params");
    tr->impl->hist_nodes(*params, tree_id, n_nodes, node_ids, sample_node, H_out);
  });
}

int pd_split_search(int device, uint32_t n_nodes, uint32_t n_classes, uint32_t n_thresholds, uint32_t n_features,
                    const uint32_t *H, const uint32_t *tot, uint32_t *best_k, float *best_gain, float *all_gains)
{
  return guarded([&] {
    require(n_nodes >= 1 && n_classes >= 1 && n_classes <= 64 && n_thresholds >= 1 && n_features >= 1,
            "bad split-search shape");
    require(H && tot && best_k, "null split-search buffer");
    set_device(device);
    // the trainer's split path on a throw-away trainer: every node has an H block
    Trainer<DepthU16Feature> t(device, n_classes);
    const size_t per = (size_t)n_classes * n_thresholds * n_features;
    const uint32_t ftiles = (n_features + 63) / 64;
    t.d_H.ensure(per * n_nodes * sizeof(uint32_t));
    t.d_cand_key.ensure((size_t)n_nodes * ftiles * sizeof(unsigned long long));
    t.d_cand_left.ensure((size_t)n_nodes * ftiles * n_classes * sizeof(uint32_t));
    std::vector<uint8_t> mode(n_nodes, 0);
    std::vector<int32_t> hidx(n_nodes);
    std::vector<uint32_t> hslots(n_nodes), res;
    for (uint32_t q = 0; q < n_nodes; q++) hidx[q] = (int32_t)(hslots[q] = q);
    HIPCHK(hipMemcpy(t.d_H.p, H, per * n_nodes * sizeof(uint32_t), hipMemcpyHostToDevice));
    const std::vector<uint64_t> no_key(n_nodes, 0ull);
    Trainer<DepthU16Feature>::Upload up{t, t.d_slice};
    const size_t u_tot = up.add(tot, (size_t)n_nodes * n_classes * sizeof(uint32_t));
    const size_t u_mode = up.add(mode.data(), n_nodes);
    const size_t u_hidx = up.add(hidx.data(), n_nodes * sizeof(int32_t));
    const size_t u_list = up.add(hslots.data(), n_nodes * sizeof(uint32_t));
    const size_t u_best = up.add(no_key.data(), n_nodes * sizeof(uint64_t));
    up.stage();
    up.commit();
    t.sl.tot = up.at<uint32_t>(u_tot);
    t.sl.slot_mode = up.at<uint8_t>(u_mode);
    t.sl.slot_hidx = up.at<int32_t>(u_hidx);
    t.sl.hlist = up.at<uint32_t>(u_list);
    t.sl.best = up.at<unsigned long long>(u_best);
    DevBuf dg;
    if (all_gains) dg.ensure((size_t)n_nodes * n_thresholds * n_features * sizeof(float));
    t.split_slice(n_nodes, hslots, n_thresholds, n_features, PD_MODE_LEVEL_BATCHED, res,
                  all_gains ? dg.as<float>() : nullptr);
    if (all_gains)
      HIPCHK(hipMemcpy(all_gains, dg.p, (size_t)n_nodes * n_thresholds * n_features * sizeof(float),
                       hipMemcpyDeviceToHost));
    for (uint32_t q = 0; q < n_nodes; q++) {
      best_k[q] = res[(size_t)q * (n_classes + 2)];
      if (best_gain) std::memcpy(&best_gain[q], &res[(size_t)q * (n_classes + 2) + 1], 4);
    }
  });
}

int pd_candidate_tables(int device, int feature_kind, const pd_train_params *params, uint32_t tree_id,
                        uint32_t n_nodes, const int32_t *node_ids, void *params_out, void *thr_out)
{
  return guarded([&] {
    require(params && node_ids && params_out && thr_out && n_nodes >= 1, "bad candidate-table arguments");
    set_device(device);
    switch (feature_kind) {
      case PD_FEAT_DEPTH_F32: candidate_tables_t<DepthF32Feature>(*params, tree_id, n_nodes, node_ids, params_out, thr_out); break;
      case PD_FEAT_DEPTH_U16: candidate_tables_t<DepthU16Feature>(*params, tree_id, n_nodes, node_ids, params_out, thr_out); break;
      case PD_FEAT_RGBD_U16X4: candidate_tables_t<RGBDFeature>(*params, tree_id, n_nodes, node_ids, params_out, thr_out); break;
      case PD_FEAT_DEMO_S16: candidate_tables_t<DemoS16Feature>(*params, tree_id, n_nodes, node_ids, params_out, thr_out); break;
      default: throw ArgError("unknown feature kind");
    }
  });
}

int pd_md5rand(int device, uint32_t n, const uint32_t *seeds, uint32_t *out)
{
  return guarded([&] {
    require(n >= 1 && seeds && out, "bad md5 arguments");
    set_device(device);
    DevBuf di, dout;
    di.ensure((size_t)n * 16);
    dout.ensure((size_t)n * 16);
    HIPCHK(hipMemcpy(di.p, seeds, (size_t)n * 16, hipMemcpyHostToDevice));
    hipLaunchKernelGGL(k_md5, dim3((n + 255) / 256), dim3(256), 0, nullptr, di.as<uint4>(), dout.as<uint4>(), n);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpy(out, dout.p, (size_t)n * 16, hipMemcpyDeviceToHost));
  });
}

int pd_fast_div(int device, uint32_t n, const float *p, const float *d, float *q)
{
  return guarded([&] {
    require(n >= 1 && p && d && q, "bad division arguments");
    set_device(device);
    DevBuf dp, dd, dq;
    dp.ensure((size_t)n * 4);
    dd.ensure((size_t)n * 4);
    dq.ensure((size_t)n * 4);
    HIPCHK(hipMemcpy(dp.p, p, (size_t)n * 4, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(dd.p, d, (size_t)n * 4, hipMemcpyHostToDevice));
    hipLaunchKernelGGL(k_div, dim3((n + 255) / 256), dim3(256), 0, nullptr, dp.as<float>(), dd.as<float>(),
                       dq.as<float>(), n);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpy(q, dq.p, (size_t)n * 4, hipMemcpyDeviceToHost));
  });
}

int pd_int_div(int device, uint32_t n, const float *p, const float *d, float *q)
{
  return guarded([&] {
    require(n >= 1 && p && d && q, "bad division arguments");
    set_device(device);
    DevBuf dp, dd, dq;
    dp.ensure((size_t)n * 4);
    dd.ensure((size_t)n * 4);
    dq.ensure((size_t)n * 4);
    HIPCHK(hipMemcpy(dp.p, p, (size_t)n * 4, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(dd.p, d, (size_t)n * 4, hipMemcpyHostToDevice));
    hipLaunchKernelGGL(k_div_int, dim3((n + 255) / 256), dim3(256), 0, nullptr, dp.as<float>(), dd.as<float>(),
                       dq.as<float>(), n);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpy(q, dq.p, (size_t)n * 4, hipMemcpyDeviceToHost));
  });
}

int pd_count_klogk(int device, uint32_t n, const uint32_t *k, float *out)
{
  return guarded([&] {
    require(n >= 1 && k && out, "bad arguments");
    set_device(device);
    DevBuf dk, dout;
    dk.ensure((size_t)n * 4);
    dout.ensure((size_t)n * 4);
    HIPCHK(hipMemcpy(dk.p, k, (size_t)n * 4, hipMemcpyHostToDevice));
    hipLaunchKernelGGL(k_count_klogk, dim3((n + 255) / 256), dim3(256), 0, nullptr, dk.as<uint32_t>(),
                       dout.as<float>(), n);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpy(out, dout.p, (size_t)n * 4, hipMemcpyDeviceToHost));
  });
}

int pd_log2_det(int device, uint32_t n, const float *x, float *y)
{
  return guarded([&] {
    require(n >= 1 && x && y, "bad log2 arguments");
    set_device(device);
    DevBuf di, dout;
    di.ensure((size_t)n * 4);
    dout.ensure((size_t)n * 4);
    HIPCHK(hipMemcpy(di.p, x, (size_t)n * 4, hipMemcpyHostToDevice));
    hipLaunchKernelGGL(k_log2_det, dim3((n + 255) / 256), dim3(256), 0, nullptr, di.as<float>(), dout.as<float>(), n);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpy(y, dout.p, (size_t)n * 4, hipMemcpyDeviceToHost));
  });
}

int pd_feature_eval(int device, int feature_kind, const void *image, uint32_t w, uint32_t h, uint32_t n,
                    const int32_t *xy, const void *params, void *out)
{
  return guarded([&] {
    require(image && xy && params && out && n >= 1 && w >= 1 && h >= 1, "bad feature-eval arguments");
    set_device(device);
    switch (feature_kind) {
      case PD_FEAT_DEPTH_F32: feature_eval_t<DepthF32Feature>(image, w, h, n, xy, params, out); break;
      case PD_FEAT_DEPTH_U16: feature_eval_t<DepthU16Feature>(image, w, h, n, xy, params, out); break;
      case PD_FEAT_RGBD_U16X4: feature_eval_t<RGBDFeature>(image, w, h, n, xy, params, out); break;
      case PD_FEAT_DEMO_S16: feature_eval_t<DemoS16Feature>(image, w, h, n, xy, params, out); break;
      default: throw ArgError("unknown feature kind");
    }
  });
}

int pd_forest_create(pd_forest **out, int device, int feature_kind, uint32_t n_classes)
{
  return guarded([&] {
    require(out != nullptr, "null output handle");
    require(n_classes >= 1 && n_classes <= 64, "n_classes must be in [1, 64]");
    std::unique_ptr<pd_forest> f(new pd_forest);
    f->impl.reset(make_forest(feature_kind, device, n_classes));
    *out = f.release();
  });
}

int pd_forest_destroy(pd_forest *fo)
{
  return guarded([&] { delete fo; });
}

int pd_forest_add_tree(pd_forest *fo, uint32_t depth, const int32_t *left_children, const void *features,
                       const void *thresholds, const float *posteriors)
{
  return guarded([&] {
    require(fo != nullptr, "null forest");
    fo->impl->add_tree(depth, left_children, features, thresholds, posteriors);
  });
}

int pd_forest_n_trees(pd_forest *fo) { return fo ? fo->impl->n_trees() : -1; }

int pd_forest_predict_leaves(pd_forest *fo, uint32_t tree_index, const void *image, uint32_t w, uint32_t h,
                             const uint8_t *mask, int32_t *out)
{
  return guarded([&] {
    require(fo != nullptr && out != nullptr, "null forest or output");
    fo->impl->predict_host((int)tree_index, image, w, h, mask, out, nullptr);
  });
}

int pd_forest_predict_posterior(pd_forest *fo, const void *image, uint32_t w, uint32_t h, const uint8_t *mask,
                                float *out)
{
  return guarded([&] {
    require(fo != nullptr && out != nullptr, "null forest or output");
    fo->impl->predict_host(0, image, w, h, mask, nullptr, out);
  });
}

int pd_forest_predict_frames_dev(pd_forest *fo, uint32_t n_frames, const void *d_pixels, uint64_t pixels_size,
                                 const uint64_t *img_offsets, const uint32_t *widths, const uint32_t *heights,
                                 const uint8_t *d_masks, uint64_t masks_size, const uint64_t *mask_offsets,
                                 float *d_post, uint64_t post_size, const uint64_t *post_offsets, int32_t *d_leaves,
                                 uint64_t leaves_size, const uint64_t *leaf_offsets, int use_graph, float *kernel_ms)
{
  return guarded([&] {
    require(fo != nullptr, "null forest");
    FrameBuffers fb{d_pixels, pixels_size, d_masks, masks_size, d_post, post_size, d_leaves, leaves_size};
    fo->impl->predict_frames(n_frames, fb, img_offsets, widths, heights, mask_offsets, post_offsets, leaf_offsets,
                             use_graph, kernel_ms);
  });
}

}  // extern "C"

namespace {

// Frame table of pd_forest_predict_frames_noalloc.  One copy per GPU (each
// device holds its own instance of the module's globals, at its own
// address), held until the process ends.  Host code never passes this name
// to a kernel or a copy: it uses the per-device address that
// hipGetSymbolAddress returns (scratch_on).
static __device__ __align__(256) FrameDesc scratch[PD_NOALLOC_MAX_FRAMES];

std::mutex g_scratch_mu;             // one no-alloc call at a time per process
std::map<int, FrameDesc *> g_scratch_ptr;

// The device address of `scratch` on `device` (current), looked up once.
FrameDesc *scratch_on(int device)
{
  auto it = g_scratch_ptr.find(device);
  if (it != g_scratch_ptr.end()) return it->second;
  void *p = nullptr;
  const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess || p == nullptr)
    throw HipError(std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
  g_scratch_ptr[device] = (FrameDesc *)p;
  return (FrameDesc *)p;
}

}  // namespace

extern "C" {

int pd_forest_predict_frames_noalloc(pd_forest *fo, uint32_t n_frames, const void *d_pixels, uint64_t pixels_size,
                                     const uint64_t *img_offsets, const uint32_t *widths, const uint32_t *heights,
                                     const uint8_t *d_masks, uint64_t masks_size, const uint64_t *mask_offsets,
                                     float *d_post, uint64_t post_size, const uint64_t *post_offsets,
                                     int32_t *d_leaves, uint64_t leaves_size, const uint64_t *leaf_offsets)
{
  return guarded([&] {
    require(fo != nullptr, "null forest");
    require(n_frames <= PD_NOALLOC_MAX_FRAMES,
            "pd_forest_predict_frames_noalloc: at most PD_NOALLOC_MAX_FRAMES (" +
                std::to_string(PD_NOALLOC_MAX_FRAMES) + ") frames per call, got " + std::to_string(n_frames));
    std::lock_guard<std::mutex> g(g_scratch_mu);
    set_device(fo->impl->device);
    FrameDesc *table = scratch_on(fo->impl->device);
    FrameBuffers fb{d_pixels, pixels_size, d_masks, masks_size, d_post, post_size, d_leaves, leaves_size};
    fo->impl->predict_frames_table(n_frames, fb, img_offsets, widths, heights, mask_offsets, post_offsets,
                                   leaf_offsets, table, PD_NOALLOC_MAX_FRAMES);
  });
}

int pd_copy_bench(int device, uint64_t bytes, int reps, float *ms_per_copy)
{
  return guarded([&] {
    require(bytes >= 4096 && reps >= 1 && ms_per_copy, "bad copy-bench arguments");
    set_device(device);
    DevBuf a, b;
    a.ensure(bytes);
    b.ensure(bytes);
    HIPCHK(hipMemset(a.p, 1, bytes));
    const size_t n = bytes / 16;
    hipDeviceProp_t prop;
    HIPCHK(hipGetDeviceProperties(&prop, device));
    const uint32_t blocks = (uint32_t)prop.multiProcessorCount * 8;
    hipLaunchKernelGGL(k_copy, dim3(blocks), dim3(256), 0, nullptr, a.as<uint4>(), b.as<uint4>(), n);
    HIPCHK(hipDeviceSynchronize());
    Event e0, e1;
    HIPCHK(hipEventRecord(e0.e, nullptr));
    for (int r = 0; r < reps; r++)
      hipLaunchKernelGGL(k_copy, dim3(blocks), dim3(256), 0, nullptr, a.as<uint4>(), b.as<uint4>(), n);
    HIPCHK(hipEventRecord(e1.e, nullptr));
    HIPCHK(hipEventSynchronize(e1.e));
    *ms_per_copy = (float)(elapsed_ms(e0, e1) / reps);
  });
}

int pd_lds_atomic_bench(int device, uint32_t iters, int reps, float *ms_per_launch, double *adds_per_s)
{
  return guarded([&] {
    require(iters >= 1 && iters <= (1u << 20) && reps >= 1 && ms_per_launch && adds_per_s,
            "bad LDS-bench arguments");
    set_device(device);
    hipDeviceProp_t prop;
    HIPCHK(hipGetDeviceProperties(&prop, device));
    const uint32_t blocks = (uint32_t)prop.multiProcessorCount * 16;
    DevBuf out;
    out.ensure((size_t)blocks * 512 * sizeof(uint32_t));
    hipLaunchKernelGGL(k_lds_add, dim3(blocks), dim3(512), 0, nullptr, iters, out.as<uint32_t>());
    HIPCHK(hipGetLastError());
    HIPCHK(hipDeviceSynchronize());
    Event e0, e1;
    HIPCHK(hipEventRecord(e0.e, nullptr));
    for (int r = 0; r < reps; r++)
      hipLaunchKernelGGL(k_lds_add, dim3(blocks), dim3(512), 0, nullptr, iters, out.as<uint32_t>());
    HIPCHK(hipEventRecord(e1.e, nullptr));
    HIPCHK(hipEventSynchronize(e1.e));
    *ms_per_launch = (float)(elapsed_ms(e0, e1) / reps);
    *adds_per_s = (double)blocks * 512.0 * 8.0 * (double)iters / (*ms_per_launch * 1e-3);
  });
}

int pd_gather_bench(int device, uint64_t window_bytes, uint32_t lines_per_load, uint32_t iters, int reps,
                    float *ms_per_launch, double *cycles_per_load)
{
  return guarded([&] {
    require(window_bytes >= 128 && window_bytes <= (1ull << 30) && window_bytes % 128 == 0,
            "window must be a multiple of 128 bytes in [128 B, 1 GiB]");
    require(lines_per_load >= 1 && lines_per_load <= 64 && 64 % lines_per_load == 0,
            "lines_per_load must divide 64");
    require(iters >= 1 && iters <= (1u << 16) && reps >= 1 && ms_per_launch && cycles_per_load,
            "bad gather-bench arguments");
    set_device(device);
    hipDeviceProp_t prop;
    HIPCHK(hipGetDeviceProperties(&prop, device));
    const uint32_t cus = (uint32_t)prop.multiProcessorCount;
    const uint32_t blocks = cus * 8;   // 32 waves per CU
    const uint32_t lines = (uint32_t)(window_bytes / 128);
    DevBuf buf, out;
    buf.ensure(window_bytes);
    HIPCHK(hipMemset(buf.p, 1, window_bytes));
    out.ensure((size_t)blocks * 256 * sizeof(uint32_t));
    const uint32_t g = 64u / lines_per_load;
    hipLaunchKernelGGL(k_gather_probe, dim3(blocks), dim3(256), 0, nullptr, buf.as<uint16_t>(), lines, g, 64u,
                       out.as<uint32_t>());
    HIPCHK(hipGetLastError());
    HIPCHK(hipDeviceSynchronize());
    Event e0, e1;
    HIPCHK(hipEventRecord(e0.e, nullptr));
    for (int r = 0; r < reps; r++)
      hipLaunchKernelGGL(k_gather_probe, dim3(blocks), dim3(256), 0, nullptr, buf.as<uint16_t>(), lines, g, iters,
                         out.as<uint32_t>());
    HIPCHK(hipEventRecord(e1.e, nullptr));
    HIPCHK(hipEventSynchronize(e1.e));
    *ms_per_launch = (float)(elapsed_ms(e0, e1) / reps);
    const double loads_per_cu = (double)blocks * 4.0 * (double)iters / (double)cus;
    *cycles_per_load = (double)*ms_per_launch * 1e-3 * (double)prop.clockRate * 1e3 / loads_per_cu;
  });
}

int pd_dev_alloc(int device, uint64_t bytes, void **out)
{
  return guarded([&] {
    require(out != nullptr && bytes > 0, "bad allocation request");
    set_device(device);
    if (hipMalloc(out, bytes) != hipSuccess) {
      (void)hipGetLastError();
      throw NoMem("hipMalloc of " + std::to_string(bytes) + " bytes failed");
    }
  });
}

int pd_dev_free(void *p)
{
  return guarded([&] { HIPCHK(hipFree(p)); });
}

int pd_memcpy_h2d(void *dst, const void *src, uint64_t bytes)
{
  return guarded([&] { HIPCHK(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice)); });
}

int pd_memcpy_d2h(void *dst, const void *src, uint64_t bytes)
{
  return guarded([&] { HIPCHK(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost)); });
}

int pd_dev_sync(int device)
{
  return guarded([&] {
    set_device(device);
    HIPCHK(hipDeviceSynchronize());
  });
}

// ---- learned split proposal ------------------------------------------------

int pd_mlp_create(pd_mlp **out, int device, uint64_t seed)
{
  return guarded([&] {
    require(out != nullptr, "null output handle");
    *out = nullptr;
    auto m = std::make_unique<pd_mlp>();
    m->impl = std::make_unique<MlpNet>(device, seed);
    *out = m.release();
  });
}

int pd_mlp_destroy(pd_mlp *m)
{
  return guarded([&] { delete m; });
}

int pd_mlp_n_params(void) { return mlp::NPARAM; }

int pd_mlp_get_params(pd_mlp *m, float *theta)
{
  return guarded([&] {
    require(m && theta, "null argument");
    m->impl->get_params(theta);
  });
}

int pd_mlp_set_params(pd_mlp *m, const float *theta)
{
  return guarded([&] {
    require(m && theta, "null argument");
    // (one verdict for all: a message string per parameter took 870 us)
    bool finite = true;
    for (int i = 0; i < mlp::NPARAM; i++) finite = finite && std::isfinite(theta[i]);
    require(finite, "non-finite parameter");
    m->impl->set_params(theta);
  });
}

int pd_mlp_forward_host(pd_mlp *m, const float *x, uint32_t n, float *y)
{
  return guarded([&] {
    require(m && x && y && n >= 1, "bad forward arguments");
    MlpNet &net = *m->impl;
    set_device(net.device);
    std::vector<uint16_t> xb((size_t)n * mlp::INP);
    MlpNet::encode(x, n, xb.data());
    net.Xs.ensure(xb.size() * 2);
    net.ys.ensure((size_t)n * 4);
    HIPCHK(hipMemcpyAsync(net.Xs.p, xb.data(), xb.size() * 2, hipMemcpyHostToDevice, net.stream));
    net.forward(net.Xs.as<uint16_t>(), n, net.ys.as<float>(), net.stream);
    HIPCHK(hipMemcpyAsync(y, net.ys.p, (size_t)n * 4, hipMemcpyDeviceToHost, net.stream));
    HIPCHK(hipStreamSynchronize(net.stream));
  });
}

int pd_mlp_forward_dev(pd_mlp *m, const uint16_t *d_x, uint64_t n, float *d_y, float *kernel_ms)
{
  return guarded([&] {
    require(m && d_x && d_y && n >= 1, "bad forward arguments");
    MlpNet &net = *m->impl;
    set_device(net.device);
    Event a, b;
    HIPCHK(hipEventRecord(a.e, net.stream));
    net.forward(d_x, n, d_y, net.stream);
    HIPCHK(hipEventRecord(b.e, net.stream));
    HIPCHK(hipEventSynchronize(b.e));
    if (kernel_ms) *kernel_ms = (float)elapsed_ms(a, b);
  });
}

int pd_mlp_grad_host(pd_mlp *m, const float *x, const float *t, uint32_t n, float *grad, float *loss)
{
  return guarded([&] {
    require(m && x && t && grad && n >= 1 && n <= (1u << 20), "bad gradient arguments");
    MlpNet &net = *m->impl;
    set_device(net.device);
    net.stage_host(x, t, n);
    const pd_adam none{0.0f, 0.9f, 0.999f, 1e-8f};
    net.step(n, false, none, net.gbuf.as<float>(), net.lbuf.as<float>());
    HIPCHK(hipMemcpyAsync(grad, net.gbuf.p, mlp::NPARAM * 4, hipMemcpyDeviceToHost, net.stream));
    float l = 0.0f;
    HIPCHK(hipMemcpyAsync(&l, net.lbuf.p, 4, hipMemcpyDeviceToHost, net.stream));
    HIPCHK(hipStreamSynchronize(net.stream));
    if (loss) *loss = l;
  });
}

int pd_mlp_step_host(pd_mlp *m, const float *x, const float *t, uint32_t n, const pd_adam *opt, float *loss)
{
  return guarded([&] {
    require(m && x && t && opt && n >= 1 && n <= (1u << 20), "bad step arguments");
    require(opt->lr >= 0.0f && opt->beta1 >= 0.0f && opt->beta1 < 1.0f && opt->beta2 >= 0.0f &&
                opt->beta2 < 1.0f && opt->eps > 0.0f,
            "bad Adam settings");
    MlpNet &net = *m->impl;
    set_device(net.device);
    net.stage_host(x, t, n);
    net.step(n, true, *opt, nullptr, net.lbuf.as<float>());
    float l = 0.0f;
    HIPCHK(hipMemcpyAsync(&l, net.lbuf.p, 4, hipMemcpyDeviceToHost, net.stream));
    HIPCHK(hipStreamSynchronize(net.stream));
    if (loss) *loss = l;
  });
}

int pd_mlp_train_dev(pd_mlp *m, const uint16_t *d_x, const float *d_t, uint64_t n, uint32_t batch, uint32_t epochs,
                     const pd_adam *opt, uint64_t seed, float *epoch_loss, float *ms)
{
  return guarded([&] {
    require(m && opt, "null argument");
    require(opt->lr >= 0.0f && opt->beta1 >= 0.0f && opt->beta1 < 1.0f && opt->beta2 >= 0.0f &&
                opt->beta2 < 1.0f && opt->eps > 0.0f,
            "bad Adam settings");
    m->impl->train(d_x, d_t, n, batch, epochs, *opt, seed, epoch_loss, ms);
  });
}

int pd_mlp_encode_rows(const float *x, uint64_t n, uint16_t *out)
{
  return guarded([&] {
    require(x && out, "null argument");
    MlpNet::encode(x, n, out);
  });
}

int pd_mma_probe(int device, const uint16_t *A, const uint16_t *Bt, float *C)
{
  return guarded([&] {
    require(A && Bt && C, "null argument");
    set_device(device);
    DevBuf a, b, c;
    a.ensure(16 * 32 * 2);
    b.ensure(16 * 32 * 2);
    c.ensure(16 * 16 * 4);
    HIPCHK(hipMemcpy(a.p, A, 16 * 32 * 2, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(b.p, Bt, 16 * 32 * 2, hipMemcpyHostToDevice));
    hipLaunchKernelGGL(mlp::k_mma_probe, dim3(1), dim3(64), 0, nullptr, a.as<uint16_t>(), b.as<uint16_t>(),
                       c.as<float>());
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpy(C, c.p, 16 * 16 * 4, hipMemcpyDeviceToHost));
  });
}

int pd_topk_select(int device, const float *scores, uint32_t n_slots, uint32_t K, uint32_t screen, uint32_t keep,
                   uint32_t *sel)
{
  return guarded([&] {
    require(scores && sel && n_slots >= 1 && K >= 1 && keep >= 1 && keep <= screen && screen <= K,
            "bad top-k arguments");
    require((uint64_t)n_slots * K < (1ull << 32), "too many scores");
    set_device(device);
    DevBuf s, o;
    s.ensure((size_t)n_slots * K * 4);
    o.ensure((size_t)n_slots * keep * 4);
    HIPCHK(hipMemcpy(s.p, scores, (size_t)n_slots * K * 4, hipMemcpyHostToDevice));
    hipLaunchKernelGGL(mlp::k_topk, dim3(n_slots), dim3(256), 0, nullptr, s.as<float>(), K, screen, keep,
                       o.as<uint32_t>());
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpy(sel, o.p, (size_t)n_slots * keep * 4, hipMemcpyDeviceToHost));
  });
}

int pd_trainer_set_record_sink(pd_trainer *tr, uint16_t *d_x, float *d_gain, float *d_rel, uint64_t capacity,
                               uint32_t per_node)
{
  return guarded([&] {
    require(tr != nullptr, "null trainer");
    if (!d_x) {
      tr->impl->sink_x = nullptr;
      tr->impl->sink_t = nullptr;
      tr->impl->sink_rel = nullptr;
      tr->impl->sink_cap = tr->impl->sink_n = 0;
      tr->impl->sink_R = 0;
      return;
    }
    require(d_gain != nullptr && capacity >= 1 && per_node >= 1, "bad record sink");
    tr->impl->sink_x = d_x;
    tr->impl->sink_t = d_gain;
    tr->impl->sink_rel = d_rel;
    tr->impl->sink_cap = capacity;
    tr->impl->sink_n = 0;
    tr->impl->sink_R = per_node;
  });
}

int pd_trainer_records_written(pd_trainer *tr, uint64_t *n)
{
  return guarded([&] {
    require(tr && n, "null argument");
    *n = tr->impl->sink_n;
  });
}

int pd_trainer_set_proposal_refine(pd_trainer *tr, uint32_t stride, uint32_t min_samples)
{
  return guarded([&] {
    require(tr != nullptr, "null trainer");
    tr->impl->prop_refine = stride;
    tr->impl->prop_refine_min = min_samples;
  });
}

int pd_trainer_set_xcd_order(pd_trainer *tr, int by_position)
{
  return guarded([&] {
    require(tr != nullptr, "null trainer");
    tr->impl->xcd_by_position = by_position ? 1 : 0;
  });
}

int pd_trainer_set_candidate_table(pd_trainer *tr, int enable)
{
  return guarded([&] {
    require(tr != nullptr, "null trainer");
    tr->impl->cand_table = enable != 0;
  });
}

int pd_trainer_set_proposal_strata(pd_trainer *tr, int mode)
{
  return guarded([&] {
    require(tr != nullptr, "null trainer");
    require(mode >= 0 && mode <= 2, "refinement mode must be 0, 1 or 2");
    tr->impl->prop_strata = mode;
  });
}

int pd_trainer_set_correction_rows(pd_trainer *tr, uint32_t rows)
{
  return guarded([&] {
    require(tr != nullptr, "null trainer");
    tr->impl->prop_corr_rows = rows;
  });
}

int pd_trainer_set_proposal(pd_trainer *tr, pd_mlp *m, uint32_t keep, uint32_t screen, uint32_t min_samples,
                            int judge)
{
  return guarded([&] {
    require(tr != nullptr, "null trainer");
    require(m == nullptr || (keep >= 1 && (screen == 0 || screen >= keep)), "need keep >= 1 and screen >= keep");
    tr->impl->prop_mlp = m ? m->impl.get() : nullptr;
    tr->impl->prop_keep = keep;
    tr->impl->prop_screen = screen;
    tr->impl->prop_min = min_samples;
    tr->impl->prop_judge = judge;
  });
}

}  // extern "C"
