"""Padenti per-pixel random-forest hot path on MI355X (gfx950).

Host-side mirror of the reference C++ API (src/padenti/*.hpp) over the C ABI
of ``libpadenti_hip.so``:

  TrainingSetImage / TrainingSet   training_set_image.hpp:38-110, training_set.hpp:39-112
  Tree                             tree.hpp:72-173 (SoA, breadth-first heap)
  TreeTrainerParameters            tree_trainer.hpp:35-51
  HIPTreeTrainer                   CLTreeTrainer (cl_tree_trainer.hpp:115, train :203-255)
  HIPClassifier                    CLClassifier (cl_classifier.hpp:81-94, predict x4)

The C++ drop-in headers with the same names live in include/padenti/.
Everything computes on the GPU; nothing here falls back to the CPU.
"""
import numpy as np

from . import _lib as L
from ._lib import (PD_FEAT_DEMO_S16, PD_FEAT_DEPTH_F32, PD_FEAT_DEPTH_U16, PD_FEAT_RGBD_U16X4,
                   PD_MODE_LEVEL_BATCHED, PD_MODE_PER_NODE, PD_MODE_PROPOSAL, FEATURES, PdError, check, lib, ptr)

__all__ = [
    "TrainingSetImage", "TrainingSet", "Tree", "TreeTrainerParameters", "HIPTreeTrainer",
    "HIPClassifier", "PdError", "PD_FEAT_DEPTH_F32", "PD_FEAT_DEPTH_U16", "PD_FEAT_RGBD_U16X4",
    "PD_FEAT_DEMO_S16", "PD_MODE_PER_NODE", "PD_MODE_LEVEL_BATCHED", "FEATURES", "device_count",
    "Plugin", "example_plugin",
]


def device_count():
    return lib().pd_device_count()


class Plugin:
    """A separately compiled feature hook (include/padenti/pd_plugin.hpp):
    ``Plugin(path, name, img_dtype, channels, feat_dtype, feat_dim)`` loads
    the shared library and its pd_trainer_create_<name> /
    pd_forest_create_<name> entry points."""

    def __init__(self, path, name, img_dtype, channels, feat_dtype, feat_dim):
        import ctypes
        self.lib = ctypes.CDLL(path)
        self.name = name
        self.info = (img_dtype, channels, feat_dtype, feat_dim)
        for kind in ("trainer", "forest"):
            fn = getattr(self.lib, "pd_%s_create_%s" % (kind, name))
            fn.restype = ctypes.c_int
            fn.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_int, ctypes.c_uint32]
            setattr(self, "create_" + kind, fn)
        self.last_error = getattr(self.lib, "pd_last_error_" + name)
        self.last_error.restype = ctypes.c_char_p

    def check(self, rc):
        if rc < 0:
            raise PdError(rc, self.last_error().decode())


def example_plugin():
    """The example plugin built next to the library (float depth hook)."""
    import os
    path = os.path.join(os.path.dirname(os.path.abspath(__file__)), "libpd_example_plugin.so")
    return Plugin(path, "user_depth", np.float32, 1, np.float32, 4)


class TrainingSetImage:
    """Image + labels (uint8, 0 = unlabelled) + sampled pixel indices.

    Per-image priors follow training_set_image_impl.hpp:35-52: class
    frequencies over the labelled sampled pixels, as float32.
    """

    def __init__(self, data, width, height, labels, n_classes, samples):
        self.data = np.ascontiguousarray(data)
        self.width, self.height = int(width), int(height)
        self.labels = np.ascontiguousarray(labels, dtype=np.uint8).reshape(-1)
        self.samples = np.ascontiguousarray(samples, dtype=np.uint32).reshape(-1)
        self.n_classes = int(n_classes)
        lab = self.labels[self.samples]
        lab = lab[lab > 0]
        cnt = np.bincount(lab.astype(np.int64) - 1, minlength=n_classes)[:n_classes].astype(np.float32)
        with np.errstate(invalid="ignore", divide="ignore"):   # no samples: 0/0 as the reference
            self.priors = (cnt / np.float32(len(lab))).astype(np.float32)


class TrainingSet:
    """Ordered image list with the running-mean priors of
    training_set_impl.hpp:157-170 (p <- (float)(p*n/(n+1) + p_img/(n+1)) in FP64)."""

    def __init__(self, n_classes):
        self.n_classes = int(n_classes)
        self.images = []
        self.priors = np.zeros(n_classes, dtype=np.float32)

    def __lshift__(self, img):
        n = len(self.images)
        self.images.append(img)
        pc = self.priors.astype(np.float64)
        pi = img.priors.astype(np.float64)
        self.priors = (pc * n / (n + 1) + pi / (n + 1)).astype(np.float32)
        return self

    def packed(self):
        """(pixels, img_off, widths, heights, labels, lab_off, samples, samp_off, n_samples)."""
        imgs = self.images
        pix = np.concatenate([im.data.reshape(-1) for im in imgs])
        sizes = np.array([im.data.size for im in imgs], dtype=np.uint64)
        img_off = np.concatenate([[0], np.cumsum(sizes)[:-1]]).astype(np.uint64)
        labels = np.concatenate([im.labels for im in imgs])
        lsz = np.array([im.labels.size for im in imgs], dtype=np.uint64)
        lab_off = np.concatenate([[0], np.cumsum(lsz)[:-1]]).astype(np.uint64)
        samples = np.concatenate([im.samples for im in imgs]).astype(np.uint32)
        ns = np.array([im.samples.size for im in imgs], dtype=np.uint32)
        samp_off = np.concatenate([[0], np.cumsum(ns.astype(np.uint64))[:-1]]).astype(np.uint64)
        w = np.array([im.width for im in imgs], dtype=np.uint32)
        h = np.array([im.height for im in imgs], dtype=np.uint32)
        return pix, img_off, w, h, labels, lab_off, samples, samp_off, ns


class Tree:
    """Breadth-first SoA tree of depth D: 2^D - 1 nodes (tree_impl.hpp:239-273).
    left_children: -2 nonexistent, -1 leaf, 2i+1 split."""

    def __init__(self, tree_id, depth, feature_kind, n_classes):
        # feature_kind: a built-in PD_FEAT_* or a Plugin (its FeatType and FeatDim)
        _, _, fdt, fd = feature_kind.info if hasattr(feature_kind, "info") else FEATURES[feature_kind]
        self.id, self.depth, self.n_classes, self.kind = int(tree_id), int(depth), int(n_classes), feature_kind
        n = (1 << depth) - 1
        self.left_children = np.full(n, -2, dtype=np.int32)
        self.features = np.zeros((n, fd), dtype=fdt)
        self.thresholds = np.zeros(n, dtype=fdt)
        self.posteriors = np.zeros((n, n_classes), dtype=np.float32)

    @property
    def n_nodes(self):
        return self.left_children.size


class TreeTrainerParameters:
    """tree_trainer.hpp:35-51 (computeFRange / randomThrSampling unused there too)."""

    def __init__(self, n_features, n_thresholds, feat_low_bounds, feat_up_bounds, thr_low_bound,
                 thr_up_bound, per_leaf_samples_thr):
        self.n_features = int(n_features)
        self.n_thresholds = int(n_thresholds)
        self.feat_low_bounds = list(feat_low_bounds)
        self.feat_up_bounds = list(feat_up_bounds)
        self.thr_low_bound = thr_low_bound
        self.thr_up_bound = thr_up_bound
        self.per_leaf_samples_thr = int(per_leaf_samples_thr)

    def c(self):
        return L.make_params(self.n_features, self.n_thresholds, self.feat_low_bounds, self.feat_up_bounds,
                             self.thr_low_bound, self.thr_up_bound, self.per_leaf_samples_thr)


class HIPTreeTrainer:
    """Replaces CLTreeTrainer(featurePath, useCPU): the feature is one of the
    compiled HIP hooks, selected by ``feature_kind``."""

    def __init__(self, feature_kind, n_classes, device=0, plugin=None, tuned=True):
        import ctypes
        self.kind, self.n_classes, self.device = feature_kind, int(n_classes), device
        self.info = plugin.info if plugin is not None else FEATURES[feature_kind]
        h = ctypes.c_void_p()
        if plugin is not None:
            plugin.check(plugin.create_trainer(ctypes.byref(h), device, n_classes))
        else:
            check(lib().pd_trainer_create(ctypes.byref(h), device, feature_kind, n_classes))
        self._h = h
        self._ts = None
        self.last_level_stats = []
        # launch tuning from the autotuner's table (built-in hooks only)
        self._tuning = None
        if tuned and plugin is None:
            from .autotune import load_table
            self._tuning = load_table()

    def _apply_tuning(self, params):
        if not self._tuning:
            return
        from .autotune import DEFAULT_TUNING, key, set_tuning
        e = self._tuning.get(key(self.kind, params.n_thresholds, self.n_classes))
        if e:
            rules = [(r["min_samples_per_node"], r["waves"], r["blocks_per_cu"], r.get("samples_per_wave", 1),
                      r.get("bins", 0)) for r in e.get("rules", [])]
            set_tuning(self, e["waves"], e["blocks_per_cu"], rules, e.get("samples_per_wave", 1), e.get("bins", 0))
        else:
            # a shape the table does not hold runs with the engine's defaults,
            # not with whatever an earlier train() of another shape applied
            set_tuning(self, *DEFAULT_TUNING[:2], (), *DEFAULT_TUNING[2:])

    def close(self):
        if getattr(self, "_h", None):
            lib().pd_trainer_destroy(self._h)
            self._h = None

    def __del__(self):
        self.close()

    def set_training_set(self, ts):
        """Upload the training set once; later train() calls reuse it."""
        pix, img_off, w, h, labels, lab_off, samples, samp_off, ns = ts.packed()
        want = self.info[0]
        pix = np.ascontiguousarray(pix, dtype=want)
        check(lib().pd_trainer_set_data(self._h, len(ts.images), ptr(pix), ptr(img_off), ptr(w), ptr(h),
                                        ptr(labels), ptr(lab_off), ptr(samples), ptr(samp_off), ptr(ns)))
        self._ts = ts

    def set_hist_budget(self, nbytes):
        check(lib().pd_trainer_set_hist_budget(self._h, int(nbytes)))

    def set_chunk(self, samples_per_chunk):
        check(lib().pd_trainer_set_chunk(self._h, int(samples_per_chunk)))

    def set_probe_order(self, enable):
        """Probe-coherent candidate tiles on/off (results are identical)."""
        check(lib().pd_trainer_set_probe_order(self._h, 1 if enable else 0))

    def set_wide_bins(self, enable):
        """32-bit histogram bins per threshold rank where they fit (default) or
        16-bit bins everywhere (results are identical)."""
        check(lib().pd_trainer_set_wide_bins(self._h, 1 if enable else 0))

    def set_record_sink(self, buf, per_node):
        """Plain trainings emit per_node records per trainable node into the
        RecordBuffer `buf` (appending after its current count); None removes it."""
        if buf is None:
            check(lib().pd_trainer_set_record_sink(self._h, None, None, None, 0, 0))
            self._sink = None
            return
        self._sink = (buf, buf.count)
        check(lib().pd_trainer_set_record_sink(self._h, buf.x_at(buf.count), buf.t_at(buf.count),
                                               buf.rel_at(buf.count), buf.capacity - buf.count, int(per_node)))

    def records_written(self):
        import ctypes
        n = ctypes.c_uint64()
        check(lib().pd_trainer_records_written(self._h, ctypes.byref(n)))
        if getattr(self, "_sink", None):
            buf, base = self._sink
            buf.count = base + n.value
        return n.value

    def set_proposal(self, net, keep, min_samples=0, judge=False, screen=None):
        """PD_MODE_PROPOSAL: `net` scores the pool of params.n_features
        candidates (one threshold each) of every node with at least
        min_samples samples; `keep` of them are histogrammed exactly: the
        first (in sampler order) of the `screen` best-scored (default: the
        top keep)."""
        self._net = net
        check(lib().pd_trainer_set_proposal(self._h, net._h if net is not None else None, int(keep),
                                            int(screen or keep), int(min_samples), 1 if judge else 0))

    def set_proposal_refine(self, stride, min_samples=0):
        """Refinement of PD_MODE_PROPOSAL: the `screen` best-scored candidates
        of a node are ranked by their exact gain on every stride-th sample (at
        least min_samples) and the best `keep` are histogrammed; stride 0
        turns it off."""
        check(lib().pd_trainer_set_proposal_refine(self._h, int(stride), int(min_samples)))

    def set_xcd_order(self, by_position):
        """XCD placement of the level-batched histogram's work items: (node,
        chunk) groups dealt evenly by samples (False) or by the chunk's position in
        its node's image-ordered samples (True).  Trees are identical either way."""
        check(lib().pd_trainer_set_xcd_order(self._h, 1 if by_position else 0))

    def set_candidate_table(self, enable):
        """Candidate parameters and thresholds computed per slice beforehand
        (True, default) or inside the histogram kernel; timing only."""
        check(lib().pd_trainer_set_candidate_table(self._h, 1 if enable else 0))

    def set_proposal_strata(self, mode):
        """Refinement ranking: 0 (False) exact gains on every stride-th
        sample; 1 (True) the gain over the node estimated from a
        class-stratified subsample; 2 that estimate plus the network's
        correction from the candidate's subsample statistics."""
        check(lib().pd_trainer_set_proposal_strata(self._h, int(mode)))

    def set_correction_rows(self, rows):
        """Mode 2: the network corrects each ranked node's best `rows`
        candidates by the estimate (at least keep), every one with 0."""
        check(lib().pd_trainer_set_correction_rows(self._h, int(rows)))

    def train(self, tree, ts, params, start_depth, end_depth, mode=PD_MODE_LEVEL_BATCHED, diagnostics=False):
        """TreeTrainer::train(tree, ts, params, startDepth=1, endDepth)."""
        if start_depth != 1:
            raise ValueError("Starting depth must be equal to 1")   # cl_tree_trainer_impl.hpp:210
        if ts is not self._ts:
            self.set_training_set(ts)
        n = tree.n_nodes
        nk = np.zeros(n, dtype=np.uint32) if diagnostics else None
        ng = np.zeros(n, dtype=np.float32) if diagnostics else None
        ng64 = np.zeros(n, dtype=np.float64) if diagnostics else None
        stats = (L.LevelStats * max(end_depth - 1, 1))()
        prior = np.ascontiguousarray(ts.priors, dtype=np.float32)
        self._apply_tuning(params)
        p = params.c()
        check(lib().pd_trainer_train(self._h, p, tree.id, tree.depth, end_depth, mode, ptr(prior),
                                     ptr(tree.left_children), ptr(tree.features), ptr(tree.thresholds),
                                     ptr(tree.posteriors), ptr(nk), ptr(ng), ptr(ng64), stats))
        self.last_level_stats = [stats[i].as_dict() for i in range(max(end_depth - 1, 0))]
        if diagnostics:
            return {"node_k": nk, "node_gain": ng, "node_gain64": ng64}
        return None

    def hist_nodes(self, params, tree_id, nodes, sample_node):
        nodes = np.ascontiguousarray(nodes, dtype=np.int32)
        sample_node = np.ascontiguousarray(sample_node, dtype=np.int32)
        H = np.zeros((len(nodes), self.n_classes, params.n_thresholds, params.n_features), dtype=np.uint32)
        check(lib().pd_trainer_hist_nodes(self._h, params.c(), tree_id, len(nodes), ptr(nodes), ptr(sample_node),
                                          ptr(H)))
        return H


class HIPClassifier:
    """Replaces CLClassifier: ``clf << tree`` uploads a tree; predict_leaves /
    predict_posterior are the reference's four predict overloads
    (classifier.hpp:52-94; mask=None means every pixel)."""

    def __init__(self, feature_kind, n_classes, device=0, plugin=None):
        import ctypes
        self.kind, self.n_classes, self.device = feature_kind, int(n_classes), device
        self.info = plugin.info if plugin is not None else FEATURES[feature_kind]
        h = ctypes.c_void_p()
        if plugin is not None:
            plugin.check(plugin.create_forest(ctypes.byref(h), device, n_classes))
        else:
            check(lib().pd_forest_create(ctypes.byref(h), device, feature_kind, n_classes))
        self._h = h

    def close(self):
        if getattr(self, "_h", None):
            lib().pd_forest_destroy(self._h)
            self._h = None

    def __del__(self):
        self.close()

    def __lshift__(self, tree):
        check(lib().pd_forest_add_tree(self._h, tree.depth, ptr(tree.left_children), ptr(tree.features),
                                       ptr(tree.thresholds), ptr(tree.posteriors)))
        return self

    @property
    def n_trees(self):
        return lib().pd_forest_n_trees(self._h)

    def _img(self, image):
        return np.ascontiguousarray(image, dtype=self.info[0])

    def predict_leaves(self, tree_index, image, width, height, mask=None):
        img = self._img(image)
        out = np.empty(width * height, dtype=np.int32)
        m = None if mask is None else np.ascontiguousarray(mask, dtype=np.uint8).reshape(-1)
        check(lib().pd_forest_predict_leaves(self._h, tree_index, ptr(img), width, height, ptr(m), ptr(out)))
        return out.reshape(height, width)

    def predict_posterior(self, image, width, height, mask=None):
        img = self._img(image)
        out = np.empty(self.n_classes * width * height, dtype=np.float32)
        m = None if mask is None else np.ascontiguousarray(mask, dtype=np.uint8).reshape(-1)
        check(lib().pd_forest_predict_posterior(self._h, ptr(img), width, height, ptr(m), ptr(out)))
        return out.reshape(self.n_classes, height, width)
