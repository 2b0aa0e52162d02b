/*
 * padenti_hip.h -- C ABI of the MI355X (gfx950) random-forest hot path.
 *
 * Plain pointers and sizes only.  Every entry point returns PD_OK (0) or a
 * negative PD_ERR_* code; pd_last_error() gives a thread-local message.
 * The C++ drop-in API (include/padenti/hip_tree_trainer.hpp,
 * include/padenti/hip_classifier.hpp) is a thin layer over this header.
 *
 * Reference interfaces replaced (paths relative to the reference root):
 *   CLTreeTrainer ctor       src/padenti/cl_tree_trainer_impl.hpp:73-198
 *   CLTreeTrainer::train     src/padenti/cl_tree_trainer_impl.hpp:203-255
 *                            (+ _initTrain, _traverseTrainingSet,
 *                               _learnBestFeatThr)
 *   computePerImageHistogram src/padenti/kernels/hist_update.cl:36-187
 *                            + host accumulation
 *                            src/padenti/cl_tree_trainer_impl_traverse_ts.hpp:462-704
 *   learnBestFeature         src/padenti/kernels/learn_best_feature.cl:22-111
 *                            + first max cl_tree_trainer_impl_learn_best_featthr.hpp:101-112
 *   CLClassifier ctor / <<   src/padenti/cl_classifier_impl.hpp:41-195
 *   CLClassifier::predict    src/padenti/cl_classifier_impl.hpp:198-557
 *                            (predict.cl:36-117)
 */
#ifndef PADENTI_HIP_H
#define PADENTI_HIP_H

#include <stddef.h>
#include <stdint.h>

/* Exported symbols; the library is built with hidden default visibility so
 * that separately compiled feature plugins never interpose each other. */
#define PD_API __attribute__((visibility("default")))

#ifdef __cplusplus
extern "C" {
#endif

#define PD_OK 0
#define PD_ERR_ARG -1      /* invalid argument / shape */
#define PD_ERR_HIP -2      /* HIP runtime error */
#define PD_ERR_STATE -3    /* call out of order (e.g. train before set_data) */
#define PD_ERR_NOMEM -4    /* device allocation failed */
#define PD_ERR_PARITY -5   /* internal consistency check failed */

/* Feature hooks compiled into the library (HIP functors standing in for
 * the reference's feature.cl plugin, test/feature.cl:29-34). */
#define PD_FEAT_DEPTH_F32 0  /* ImgType float x1, FeatType float, FeatDim 4 */
#define PD_FEAT_DEPTH_U16 1  /* ImgType uint16 x1, FeatType float, FeatDim 4 */
#define PD_FEAT_RGBD_U16X4 2 /* ImgType uint16 x4, FeatType float, FeatDim 6 */
#define PD_FEAT_DEMO_S16 3   /* ImgType uint16 x1, FeatType short, FeatDim 2 */

#define PD_MODE_PER_NODE 0      /* one histogram + one split launch per node */
#define PD_MODE_LEVEL_BATCHED 1 /* one launch per tree level (per slice) */
#define PD_MODE_PROPOSAL 2      /* level-batched; the split-proposal network picks
                                   the candidates histogrammed exactly */

/* Mirrors TreeTrainerParameters<FeatType, FeatDim> (src/padenti/tree_trainer.hpp:35-51).
 * Bounds are carried as double and converted to FeatType (exact for float
 * and short).  computeFRange / randomThrSampling are unused in the
 * reference and omitted. */
typedef struct {
  uint32_t n_features;
  uint32_t n_thresholds;
  double feat_low[8];
  double feat_up[8];
  double thr_low;
  double thr_up;
  uint32_t per_leaf_samples_thr;
  uint32_t reserved;
} pd_train_params;

/* Per-level record filled by pd_trainer_train (the reference logs the same
 * quantities with BOOST_LOG_TRIVIAL, cl_tree_trainer_impl.hpp:249-250 and
 * cl_tree_trainer_impl_traverse_ts.hpp:437-454). */
typedef struct {
  uint32_t level;
  uint32_t frontier_nodes;
  uint32_t slices;
  uint32_t hist_launches;
  uint64_t active_samples;  /* samples in trainable frontier nodes */
  double evals;             /* active_samples * nF * nT */
  double hist_ms;           /* device time of the histogram kernel(s) */
  double split_ms;          /* device time of split + finalize */
  double route_ms;          /* device time of routing */
  double wall_ms;           /* host wall clock of the level */
  uint32_t split_nodes;
  uint32_t proposal_nodes;  /* PD_MODE_PROPOSAL: nodes whose pool the network ranked */
  uint32_t fallback_nodes;  /* PD_MODE_PROPOSAL: trainable nodes evaluated exhaustively */
  uint32_t judged_nodes;    /* proposal nodes also evaluated exhaustively (judge on) */
  double mlp_ms;            /* device time of the candidate scoring */
  double select_ms;         /* device time of the top-k selection */
  double judge_ms;          /* device time of the exhaustive judge (not training work) */
  double gain_exhaustive;   /* sum over judged nodes of the exhaustive best FP32 gain */
  double gain_proposal;     /* sum over judged nodes of the chosen split's FP32 gain */
  double gain_loss_rel;     /* sum over judged nodes of (g_exh - g_prop) / g_exh, g_exh > 0 */
  uint32_t reserved;
  double refine_ms;         /* PD_MODE_PROPOSAL with refinement: device time of the subsample ranking */
} pd_level_stats;

/* Launch tuning of the histogram kernel (chosen by the autotuner). */
typedef struct {
  uint32_t waves;             /* wave64s per histogram block: 4, 8 or 16 */
  uint32_t blocks_per_cu;     /* target work items per CU when a level's samples are cut into chunks */
  uint32_t samples_per_wave;  /* samples per wave step: 1, 2 or 4, i.e. 64, 32 or 16 candidates per
                                 tile (0 reads as 1; 2 and 4 exist for 1, 10, 20 and 32 thresholds and
                                 8 or 16 waves, other shapes run with 1) */
  uint32_t bins;              /* LDS bin layout of the tile: 0 automatic (one 32-bit count per (rank,
                                 candidate) where the tile still leaves two blocks per CU, else 16-bit
                                 counts shared by neighbouring candidates), 1 always 16-bit, 2 32-bit
                                 wherever the tile fits one block's LDS (32-bit counts exist for
                                 4-byte responses, 8 or 16 waves and up to 32 thresholds) */
} pd_tuning;

/* Adam settings of the split-proposal network. */
typedef struct {
  float lr;
  float beta1;
  float beta2;
  float eps;
} pd_adam;

typedef struct pd_trainer pd_trainer;
typedef struct pd_forest pd_forest;
typedef struct pd_mlp pd_mlp;

PD_API const char *pd_last_error(void);
PD_API int pd_version(void);
/* Number of visible HIP devices (0 without a GPU; never fails). */
PD_API int pd_device_count(void);

/* ---- training (replaces CLTreeTrainer, cl_tree_trainer.hpp:115) ----- */
PD_API int pd_trainer_create(pd_trainer **out, int device, int feature_kind, uint32_t n_classes);
PD_API int pd_trainer_destroy(pd_trainer *tr);

/* Upload the training set (TrainingSetImage list, training_set_image.hpp:64-66).
 * pixels: all images packed, img_offsets[i] = element offset of image i;
 * labels: packed label images (uint8, 0 = unlabelled, 1..nC), label_offsets
 * in bytes; samples: packed pixel indices y*w+x, sample_offsets in elements.
 * Every sample must be labelled (the reference indexes label-1). */
PD_API int pd_trainer_set_data(pd_trainer *tr, uint32_t n_images, const void *pixels, const uint64_t *img_offsets,
                        const uint32_t *widths, const uint32_t *heights, const uint8_t *labels,
                        const uint64_t *label_offsets, const uint32_t *samples, const uint64_t *sample_offsets,
                        const uint32_t *n_samples);

/* Device memory budget for histograms (bytes); frontier levels whose
 * histograms exceed it are processed in slices (the reference slices at
 * GLOBAL_HISTOGRAM_MAX_SIZE of host RAM, cl_tree_trainer_impl.hpp:50). */
PD_API int pd_trainer_set_hist_budget(pd_trainer *tr, uint64_t bytes);
/* Samples per histogram work item (0 = automatic; an item may hold up to three
 * more, its node's chunks beginning on 64-byte lines of the sample records). */
PD_API int pd_trainer_set_chunk(pd_trainer *tr, uint32_t samples_per_chunk);
/* Probe-coherent candidate tiles (default on): for feature hooks that name
 * the row offset parameters of their probes, each node's candidates are
 * handed to the 64-lane histogram tiles along a Hilbert curve of those
 * offsets, so the gathers of a tile touch few cache lines and the samples
 * that follow reuse them.  Results are identical either way.  No
 * counterpart in the reference (hist_update.cl assigns candidate f to work
 * item f). */
PD_API int pd_trainer_set_probe_order(pd_trainer *tr, int enable);
/* Histogram bin layout (default on = one 32-bit bin per threshold rank
 * wherever that tile still fits two blocks per CU and the hook's responses
 * are 4-byte values; off = 16-bit bins, two lanes per word, everywhere).  Results
 * are identical either way.  No counterpart in the reference (its
 * histograms are per-sample global-memory increments, hist_update.cl). */
PD_API int pd_trainer_set_wide_bins(pd_trainer *tr, int enable);

/* Train one tree: TreeTrainer::train(tree, ts, params, 1, end_depth)
 * (tree_trainer.hpp:82-85).  Tree arrays are the reference SoA layout of a
 * tree of depth `tree_depth` (N = 2^tree_depth - 1 nodes): left_children[N],
 * features[N*FeatDim], thresholds[N] (FeatType), posteriors[N*nC]; they are
 * overwritten.  root_prior[nC] is TrainingSet::getPriors().  Optional
 * per-node outputs (size N, may be NULL): chosen k = t*nF + f, FP32 gain,
 * FP64 gain of the chosen split.  level_stats (may be NULL) receives
 * end_depth-1 records. */
PD_API int pd_trainer_train(pd_trainer *tr, const pd_train_params *params, uint32_t tree_id, uint32_t tree_depth,
                     uint32_t end_depth, int mode, const float *root_prior, int32_t *left_children,
                     void *features, void *thresholds, float *posteriors, uint32_t *node_k, float *node_gain,
                     double *node_gain64, pd_level_stats *level_stats);

/* Histogram launch tuning (default {8, 16}); pd_trainer_time_level gives the
 * device time (ms, mean of reps) of one level-batched histogram + split pass
 * over the training set cut into n_nodes equal shares with the current
 * tuning: the autotuner's probe (padenti_amd/autotune.py).  The reference
 * fixes its work split at compile time (hist_update.cl, local size 16x16). */
PD_API int pd_trainer_set_tuning(pd_trainer *tr, const pd_tuning *tuning);
PD_API int pd_trainer_get_tuning(pd_trainer *tr, pd_tuning *tuning);
/* Per-level tuning: rules sorted by decreasing min_samples_per_node; a level
 * uses the first rule whose min_samples_per_node <= its active samples per
 * trainable node (none matching, or n_rules = 0: the single tuning above). */
typedef struct {
  uint32_t min_samples_per_node;
  pd_tuning tuning;
} pd_tuning_rule;
PD_API int pd_trainer_set_tuning_rules(pd_trainer *tr, uint32_t n_rules, const pd_tuning_rule *rules);
/* Placement of the level-batched histogram's work items on the XCDs (each
 * XCD has its own L2): 0 deals the (node, chunk) groups evenly by samples; 1 places
 * a chunk of a node cut into at least as many chunks as there are XCDs on
 * the XCD of its position in the node's (image-ordered) samples, so chunks
 * of different nodes over the same images share one L2.  Timing only: trees
 * are identical either way. */
PD_API int pd_trainer_set_xcd_order(pd_trainer *tr, int by_position);
/* Candidate table: 1 (default) computes every histogram slice's candidate
 * parameters and thresholds in a separate kernel beforehand (at most 16 GiB
 * per slice; larger slices derive them inside the histogram kernel), 0
 * always derives them inside the histogram kernel.  Timing only: trees are
 * identical either way. */
PD_API int pd_trainer_set_candidate_table(pd_trainer *tr, int enable);
PD_API int pd_trainer_time_level(pd_trainer *tr, const pd_train_params *params, uint32_t tree_id, uint32_t n_nodes,
                                 int reps, double *ms);

/* (a) alone: histograms H[n][c][t][f] (uint32) of the listed nodes, with
 * sample_node[s] giving the node of every packed sample (-1 = none). */
PD_API int pd_trainer_hist_nodes(pd_trainer *tr, const pd_train_params *params, uint32_t tree_id, uint32_t n_nodes,
                          const int32_t *node_ids, const int32_t *sample_node, uint32_t *H_out);

/* (b) alone: for each node, the first maximum over k = t*nF + f of the FP32
 * gain, from host H[n][c][t][f] and per-class totals tot[n][c]. */
PD_API int pd_split_search(int device, uint32_t n_nodes, uint32_t n_classes, uint32_t n_thresholds,
                    uint32_t n_features, const uint32_t *H, const uint32_t *tot, uint32_t *best_k,
                    float *best_gain, float *all_gains);

/* Candidate tables on the device: params[n][f][FeatDim], thresholds[n][f][nT]. */
PD_API int pd_candidate_tables(int device, int feature_kind, const pd_train_params *params, uint32_t tree_id,
                        uint32_t n_nodes, const int32_t *node_ids, void *params_out, void *thr_out);

/* Unit entry points (device evaluation of single steps). */
PD_API int pd_md5rand(int device, uint32_t n, const uint32_t *seeds, uint32_t *out);
PD_API int pd_log2_det(int device, uint32_t n, const float *x, float *y);
/* q[i] = p[i] / d[i] through the feature hooks' per-pixel division path. */
PD_API int pd_fast_div(int device, uint32_t n, const float *p, const float *d, float *q);
/* q[i] = p[i] / d[i] through the one-correction quotient of the integer-depth
 * hooks (d[i] an integer, 1 <= |d[i]| <= 65535, any p[i]) and of the split
 * search's class fractions (p[i] <= d[i] < 2^21, both integers). */
PD_API int pd_int_div(int device, uint32_t n, const float *p, const float *d, float *q);
/* out[i] = k[i] log2 k[i] (0 for 0) as the fused split search approximates it. */
PD_API int pd_count_klogk(int device, uint32_t n, const uint32_t *k, float *out);
PD_API int pd_feature_eval(int device, int feature_kind, const void *image, uint32_t w, uint32_t h, uint32_t n,
                    const int32_t *xy, const void *params, void *out);

/* ---- prediction (replaces CLClassifier, cl_classifier.hpp:81-94) ----- */
PD_API int pd_forest_create(pd_forest **out, int device, int feature_kind, uint32_t n_classes);
PD_API int pd_forest_destroy(pd_forest *fo);
/* CLClassifier::operator<<(const Tree&): copies the tree to the device. */
PD_API int pd_forest_add_tree(pd_forest *fo, uint32_t depth, const int32_t *left_children, const void *features,
                       const void *thresholds, const float *posteriors);
PD_API int pd_forest_n_trees(pd_forest *fo);
/* predict(id, image, leafIdx[, mask]): out[h*w] leaf ids, -1 where mask==0. */
PD_API int pd_forest_predict_leaves(pd_forest *fo, uint32_t tree_index, const void *image, uint32_t w, uint32_t h,
                             const uint8_t *mask, int32_t *out);
/* predict(image, posterior[, mask]): out[nC][h][w] planar FP32. */
PD_API int pd_forest_predict_posterior(pd_forest *fo, const void *image, uint32_t w, uint32_t h, const uint8_t *mask,
                                float *out);

/* Batched multi-frame prediction on device-resident buffers (one launch,
 * optionally replayed from a captured hipGraph); the multi-frame form of
 * Classifier::predict (cl_classifier_impl.hpp:356-557, one frame per call
 * there).  d_pixels (pixels_size bytes): frames packed, img_offsets[i]
 * element offsets of interleaved pixels; d_masks (masks_size bytes) may be
 * NULL, else frame i's mask starts at byte mask_offsets[i].  Outputs (either
 * may be NULL): d_post (post_size bytes), frame i at float element
 * post_offsets[i] as [nC][h][w]; d_leaves (leaves_size bytes), frame i at
 * int32 element leaf_offsets[i] as [tree][h][w].  Every frame's range in
 * every given buffer is checked against the buffer's size on the host before
 * anything is launched (PD_ERR_ARG otherwise).  use_graph != 0 captures the
 * launch once per shape set and replays it.  *kernel_ms (may be NULL)
 * receives the device time. */
PD_API int pd_forest_predict_frames_dev(pd_forest *fo, uint32_t n_frames, const void *d_pixels,
                                 uint64_t pixels_size, const uint64_t *img_offsets, const uint32_t *widths,
                                 const uint32_t *heights, const uint8_t *d_masks, uint64_t masks_size,
                                 const uint64_t *mask_offsets, float *d_post, uint64_t post_size,
                                 const uint64_t *post_offsets, int32_t *d_leaves, uint64_t leaves_size,
                                 const uint64_t *leaf_offsets, int use_graph, float *kernel_ms);

/* The same multi-frame prediction for callers that cannot allocate device
 * memory (code under hipGraph capture, tight serving loops, harnesses that
 * forbid hipMalloc).  No counterpart in the reference.  It calls no hipMalloc,
 * hipFree or allocating library routine: the frame table lives in a
 * file-scope device array of PD_NOALLOC_MAX_FRAMES entries (48 B each, one
 * copy per GPU, held until the process ends), and the forest's own arrays
 * were allocated when its trees were added.  Arguments and checks as
 * pd_forest_predict_frames_dev (no graph replay, no timing); more than
 * PD_NOALLOC_MAX_FRAMES frames, or an auto-context hook, is PD_ERR_ARG.
 * Calls are serialised within the process (each returns after its launch has
 * finished); overlapping calls from several processes on one GPU each use
 * their own process's array. */
#define PD_NOALLOC_MAX_FRAMES 4096u
PD_API int pd_forest_predict_frames_noalloc(pd_forest *fo, uint32_t n_frames, const void *d_pixels,
                                            uint64_t pixels_size, const uint64_t *img_offsets,
                                            const uint32_t *widths, const uint32_t *heights,
                                            const uint8_t *d_masks, uint64_t masks_size,
                                            const uint64_t *mask_offsets, float *d_post, uint64_t post_size,
                                            const uint64_t *post_offsets, int32_t *d_leaves,
                                            uint64_t leaves_size, const uint64_t *leaf_offsets);

/* HBM probe: average time of a plain device-to-device copy kernel moving
 * `bytes` (read) + `bytes` (write), over `reps` launches. */
PD_API int pd_copy_bench(int device, uint64_t bytes, int reps, float *ms_per_copy);
/* Texel-gather probe: 32 waves per CU each issue `iters` 64-lane uint16
 * loads touching `lines_per_load` distinct 128-byte lines, drawn at random
 * from a window of `window_bytes` (inside the vector L1: the L1-hit rate;
 * a few MiB: the L1-miss rate).  Reports ms per launch and CU cycles per
 * wave load (at the device's reported clock). */
PD_API int pd_gather_bench(int device, uint64_t window_bytes, uint32_t lines_per_load, uint32_t iters, int reps,
                           float *ms_per_launch, double *cycles_per_load);

/* LDS-atomic probe: 16 blocks of 512 threads per CU, each lane doing
 * 8 * iters conflict-free 32-bit LDS adds into its own table column (the
 * histogram kernel's access pattern).  *adds_per_s = chip-wide rate. */
PD_API int pd_lds_atomic_bench(int device, uint32_t iters, int reps, float *ms_per_launch, double *adds_per_s);

/* ---- learned split proposal (no counterpart in the reference) ----------
 * Network: 22 inputs (node class histogram n_c/n [16, zero padded], depth/16,
 * candidate u, v scaled by the feature bounds, threshold mapped to [-1, 1])
 * -> 3 x 256 GELU -> predicted FP32 gain.  BF16 weights / activations, FP32
 * accumulation (MFMA), FP32 master weights and Adam state.  Flat FP32
 * parameter order: W1[256][22], b1[256], W2[256][256], b2, W3[256][256], b3,
 * w4[256], b4 (pd_mlp_n_params() values). */
PD_API int pd_mlp_create(pd_mlp **out, int device, uint64_t seed);
PD_API int pd_mlp_destroy(pd_mlp *m);
PD_API int pd_mlp_n_params(void);
PD_API int pd_mlp_get_params(pd_mlp *m, float *theta);
/* replaces the parameters and restarts the Adam state */
PD_API int pd_mlp_set_params(pd_mlp *m, const float *theta);
/* host rows x[n][22] (rounded to BF16) -> y[n] */
PD_API int pd_mlp_forward_host(pd_mlp *m, const float *x, uint32_t n, float *y);
/* device rows (BF16 [n][32], as pd_mlp_encode_rows writes) -> device y[n] */
PD_API int pd_mlp_forward_dev(pd_mlp *m, const uint16_t *d_x, uint64_t n, float *d_y, float *kernel_ms);
/* gradient of L = mean_r (y_r - t_r)^2 over one batch of host rows (n <= 2^20) */
PD_API int pd_mlp_grad_host(pd_mlp *m, const float *x, const float *t, uint32_t n, float *grad, float *loss);
/* one Adam step on one batch of host rows (n <= 2^20); *loss = the batch loss before the step */
PD_API int pd_mlp_step_host(pd_mlp *m, const float *x, const float *t, uint32_t n, const pd_adam *opt,
                            float *loss);
/* `epochs` passes over device records (BF16 rows [n][32], FP32 targets [n])
 * in shuffled batches of `batch` <= 2^20 rows; epoch_loss[e] = mean batch
 * loss of epoch e */
PD_API int pd_mlp_train_dev(pd_mlp *m, const uint16_t *d_x, const float *d_t, uint64_t n, uint32_t batch,
                            uint32_t epochs, const pd_adam *opt, uint64_t seed, float *epoch_loss, float *ms);
/* host FP32 rows [n][22] -> BF16 rows [n][32] (the device row format) */
PD_API int pd_mlp_encode_rows(const float *x, uint64_t n, uint16_t *out);
/* The proposal's selection alone: for each of n_slots rows of K scores, the
 * `screen` largest (ties: lower index first) are screened, and the first
 * `keep` of them in increasing index are listed (screen == keep: top keep). */
PD_API int pd_topk_select(int device, const float *scores, uint32_t n_slots, uint32_t K, uint32_t screen,
                          uint32_t keep, uint32_t *sel);
/* MFMA fragment probe: C[16][16] = A[16][32] . B, B given as Bt[16][32] (BF16) */
PD_API int pd_mma_probe(int device, const uint16_t *A, const uint16_t *Bt, float *C);

/* Record sink of the plain trainer: while set, every trainable node of a
 * PD_MODE_LEVEL_BATCHED / PD_MODE_PER_NODE training writes per_node records
 * (network input row, FP32 gain of that (feature, threshold) pair, sampled
 * with MD5 of (tree, node, j, 7)) to d_x / d_gain, and, if d_rel is not
 * NULL, the gain divided by the node's best gain over all its pairs (0 when
 * that is not positive), up to `capacity` records.  d_x = NULL removes the
 * sink. */
PD_API int pd_trainer_set_record_sink(pd_trainer *tr, uint16_t *d_x, float *d_gain, float *d_rel, uint64_t capacity,
                                      uint32_t per_node);
PD_API int pd_trainer_records_written(pd_trainer *tr, uint64_t *n);
/* PD_MODE_PROPOSAL settings: the network (kept alive by the caller); the
 * number of pool candidates histogrammed exactly (`keep`), taken in sampler
 * order from the `screen` best-scored (screen = keep or 0: the top keep;
 * screen = pool size: no use of the scores); the smallest node (samples)
 * that is ranked (smaller nodes evaluate the whole pool); judge != 0 to
 * evaluate the whole pool beside every ranked node and report the gain lost
 * (pd_level_stats). */
PD_API int pd_trainer_set_proposal(pd_trainer *tr, pd_mlp *mlp, uint32_t keep, uint32_t screen, uint32_t min_samples,
                                   int judge);
/* Refinement of the proposal (no counterpart in the reference): the
 * `screen` best-scored candidates of a node (screen from
 * pd_trainer_set_proposal, or all of them) are evaluated exactly on an evenly
 * spaced subsample of the node's samples (every `stride`-th, at least
 * `min_samples`, all samples of a smaller node), and the `keep` with the
 * largest subsample gains (ties to the lower sampler index) are histogrammed
 * on all samples.  stride 0 turns it off. */
PD_API int pd_trainer_set_proposal_refine(pd_trainer *tr, uint32_t stride, uint32_t min_samples);
/* Refinement subsample (mode): 0 (default) every stride-th sample of the
 * node and its exact gains; 1 a class-stratified subsample of the same size
 * (every class the node holds at a rate of at least size / (2 nC) samples,
 * the rest in proportion) whose counts, scaled back by class, estimate each
 * candidate's gain over the whole node; 2 the same estimate relative to the
 * node's best, plus the network's correction computed from the candidate's
 * subsample statistics (input columns 22..31; a network with every weight
 * zero ranks as mode 1).  A ranking only: the kept candidates are still
 * histogrammed exactly.  With the whole pool screened (screen = n_features)
 * no pool scores are computed.  With a record sink set, PD_MODE_PROPOSAL in
 * modes 1 and 2 emits per_node records per ranked node from these rows, with
 * the exact gain of the candidate over the whole node as target and, in the
 * relative-gain buffer, the exact relative gain minus the estimated one (the
 * correction the network learns). */
PD_API int pd_trainer_set_proposal_strata(pd_trainer *tr, int mode);
/* Refinement mode 2: the network corrects each ranked node's best `rows`
 * candidates by the estimate (at least keep of them; the others rank below
 * them), or every screened candidate with rows = 0 (the default).  A zero
 * correction keeps the estimate's own ranking either way. */
PD_API int pd_trainer_set_correction_rows(pd_trainer *tr, uint32_t rows);

/* ---- dataset ingestion ---------------------------------------------------
 * Replaces (paths relative to the reference root):
 *   UniformImageSampler::sample       src/padenti/uniform_image_sampler_impl.hpp:34-63
 *   ClassWeightedImageSampler ctors    src/padenti/classweighted_image_sampler_impl.hpp:26-44
 *   ClassWeightedImageSampler::sample  src/padenti/classweighted_image_sampler_impl.hpp:57-123
 *   CVRGBLabelsLoader::load / _rgb2label  src/padenti/cv_image_loader_impl.hpp:78-133, 235-267
 *   CVImageLoader::load (cv::imread)   src/padenti/cv_image_loader_impl.hpp:36-72
 *   TrainingSet directory constructor  src/padenti/training_set_impl.hpp:43-133
 * Sampling runs on the device, one workgroup per image, and reproduces the
 * reference's draws: MT19937 seeded with crc32(image bytes) ^ seed. */
#define PD_SAMPLER_UNIFORM 0        /* with replacement among labelled pixels */
#define PD_SAMPLER_CLASS_WEIGHTED 1 /* per-class reservoir of ceilf(w_c * n_samples) */

typedef struct {
  uint32_t kind;         /* PD_SAMPLER_* */
  uint32_t n_samples;    /* nSamples of the sampler constructor */
  uint32_t seed;         /* seed of the sampler constructor (default 0) */
  uint32_t n_classes;    /* class-weighted: nClasses (labels 1..n_classes) */
  const float *weights;  /* class-weighted: n_classes weights, NULL = 1.f / n_classes each */
} pd_sampler;

typedef struct {
  float crc_ms;    /* CRC-32 of the image bytes */
  float index_ms;  /* uniform: labelled-pixel rank index (mask + prefix) */
  float sample_ms; /* MT19937 draws and the reservoir / rank selection */
  float sort_ms;   /* per-image ascending sort */
  float total_ms;
  uint64_t crc_bytes;   /* image bytes hashed */
  uint64_t label_bytes; /* label bytes scanned */
} pd_ingest_stats;

/* Per-image output capacity (slots): n_samples (uniform) or sum_c
 * ceilf(w_c * n_samples) (class-weighted; can exceed n_samples). */
PD_API int pd_sampler_capacity(const pd_sampler *s, uint32_t *capacity);

/* Sample a batch of images.  data: the image bytes (any layout; image i is
 * the data_bytes[i] bytes at data_offsets[i], hashed as the reference's
 * sizeof(type) * w * h * nChannels bytes); labels: uint8 label images
 * (0 = unlabelled), image i at label_offsets[i], widths[i] * heights[i]
 * bytes.  Output: samples[i * capacity + k], k < n_out[i], pixel indices
 * y * w + x in ascending order; crc[i] (optional) = crc32 of image i.
 * An image without labelled pixels gets n_out = 0 (the reference's draw
 * range would be empty).  Class-weighted: a label above n_classes is an
 * error (the reference indexes out of bounds). */
PD_API int pd_sample_images(int device, const pd_sampler *s, uint32_t n_images, const void *data,
                            const uint64_t *data_offsets, const uint64_t *data_bytes, const uint8_t *labels,
                            const uint64_t *label_offsets, const uint32_t *widths, const uint32_t *heights,
                            uint32_t *samples, uint32_t *n_out, uint32_t *crc);
/* Device form: d_data (data_size bytes), d_labels (labels_size bytes),
 * d_samples (n_images * capacity slots), d_n_out, d_crc (optional, n_images)
 * are device pointers; offsets, sizes and stats are host memory.  Every
 * range must lie inside its buffer and every label image must start at a
 * 16-byte aligned device address (both checked).  Synchronous. */
PD_API int pd_sample_images_dev(int device, const pd_sampler *s, uint32_t n_images, const void *d_data,
                                uint64_t data_size, const uint64_t *data_offsets, const uint64_t *data_bytes,
                                const uint8_t *d_labels, uint64_t labels_size, const uint64_t *label_offsets,
                                const uint32_t *widths, const uint32_t *heights, uint32_t *d_samples,
                                uint32_t *d_n_out, uint32_t *d_crc, pd_ingest_stats *stats);
/* The same with at most scratch_bytes (rounded up to one step of a stream, 1816
 * bytes; pd_sample_images_dev: 256 MiB) of device memory for the random streams
 * of the class-weighted sampler.  Longer streams are generated in parts, larger
 * batches in groups of images; without any (0, or where the allocation fails)
 * every image is walked by one wave.  The samples do not depend on it.  What is
 * held beyond the bound from earlier calls on the device is freed. */
PD_API int pd_sample_images_dev_scratch(int device, const pd_sampler *s, uint32_t n_images, const void *d_data,
                                        uint64_t data_size, const uint64_t *data_offsets, const uint64_t *data_bytes,
                                        const uint8_t *d_labels, uint64_t labels_size, const uint64_t *label_offsets,
                                        const uint32_t *widths, const uint32_t *heights, uint32_t *d_samples,
                                        uint32_t *d_n_out, uint32_t *d_crc, pd_ingest_stats *stats,
                                        uint64_t scratch_bytes);
/* crc32 (zlib's) of n byte ranges of device memory d_data (data_size bytes;
 * every range is checked against it); kernel_ms optional */
PD_API int pd_crc32_images_dev(int device, uint32_t n, const void *d_data, uint64_t data_size,
                               const uint64_t *offsets, const uint64_t *bytes, uint32_t *d_crc, float *kernel_ms);
/* labels[i] = 1 + first class c with rgb2label[c] == pixel i's (R, G, B),
 * else 0; pixels are `channels` (3 or 4, the 4th ignored) bytes in R, G, B
 * order (the reference converts OpenCV's BGR to RGB before matching). */
PD_API int pd_rgb_to_labels(int device, uint64_t n_pixels, uint32_t channels, const uint8_t *rgb,
                            const uint8_t *rgb2label, uint32_t n_classes, uint8_t *labels);
PD_API int pd_rgb_to_labels_dev(int device, uint64_t n_pixels, uint32_t channels, const uint8_t *d_rgb,
                                const uint8_t *rgb2label, uint32_t n_classes, uint8_t *d_labels, float *kernel_ms);

/* PNG codec (host), standing in for cv::imread(path, -1) / cv::imwrite.
 * Read: gray 1/2/4/8/16-bit -> 1 channel (low depths scaled to 8 bit);
 * RGB, palette -> 3 channels B, G, R (4 with a tRNS chunk: B, G, R, A);
 * gray + alpha, RGBA -> 4 channels B, G, R, A; 16-bit samples in host
 * order.  pixels = NULL: header only.  capacity in bytes. */
typedef struct {
  uint32_t width, height, channels, bit_depth; /* bit_depth of the output: 8 or 16 */
} pd_png_info;
PD_API int pd_png_read(const char *path, pd_png_info *info, void *pixels, uint64_t capacity);
/* channels 1 (gray), 3 (B, G, R) or 4 (B, G, R, A); bit_depth 8 or 16 */
PD_API int pd_png_write(const char *path, uint32_t width, uint32_t height, uint32_t channels, uint32_t bit_depth,
                        const void *pixels);
/* Pairs of (dir/<p><data_suffix>, dir/<p><labels_suffix>) for every regular
 * file of dir whose name ends with data_suffix and whose labels file
 * exists, ordered by file name (the reference keeps the directory's own
 * iteration order).  Written to buf as 2 * n_pairs NUL-terminated paths;
 * *needed = bytes required (call with cap 0 to size buf). */
PD_API int pd_list_pairs(const char *dir, const char *data_suffix, const char *labels_suffix, char *buf,
                         uint64_t cap, uint32_t *n_pairs, uint64_t *needed);

/* ---- device memory helpers (for callers without another allocator) ---- */
PD_API int pd_dev_alloc(int device, uint64_t bytes, void **out);
PD_API int pd_dev_free(void *p);
PD_API int pd_memcpy_h2d(void *dst, const void *src, uint64_t bytes);
PD_API int pd_memcpy_d2h(void *dst, const void *src, uint64_t bytes);
PD_API int pd_dev_sync(int device);

#ifdef __cplusplus
}
#endif
#endif /* PADENTI_HIP_H */
