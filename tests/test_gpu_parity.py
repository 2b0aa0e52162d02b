"""GPU parity tests: every step of the hot path through the C ABI against the
CPU oracle on the same seeded inputs.  Integer / index results and FP32
values are compared bit for bit; FP64 gains within 1e-12; posteriors within
1e-6 relative of an FP64 average."""
import ctypes

import numpy as np
import pytest

import padenti_amd as pa
from padenti_amd import _lib as L
from padenti_amd import synth
from oracle import oracle as orc
from tests import helpers as hp

pytestmark = pytest.mark.gpu

KINDS = [pa.PD_FEAT_DEPTH_F32, pa.PD_FEAT_DEPTH_U16, pa.PD_FEAT_RGBD_U16X4, pa.PD_FEAT_DEMO_S16]


def test_md5rand_device(gpu):
    rng = np.random.default_rng(1)
    seeds = rng.integers(0, 2 ** 32, size=(4096, 4), dtype=np.uint64).astype(np.uint32)
    seeds[0] = 0
    seeds[1] = 0xffffffff
    out = np.zeros_like(seeds)
    L.check(L.lib().pd_md5rand(0, len(seeds), L.ptr(seeds), L.ptr(out)))
    for i in range(0, len(seeds), 97):
        assert out[i].tolist() == hp.md5rand(seeds[i])
    want = np.stack([orc.md5rand(s) for s in seeds])
    assert np.array_equal(out, want)


def test_log2_det_device_bit_exact(gpu):
    rng = np.random.default_rng(2)
    x = np.concatenate([rng.uniform(1e-6, 1.0, 100000), np.float32(1.0) / np.arange(1, 5000)]).astype(np.float32)
    y = np.zeros_like(x)
    L.check(L.lib().pd_log2_det(0, len(x), L.ptr(x), L.ptr(y)))
    want = np.array([orc.log2_det(v) for v in x], dtype=np.float32)
    assert y.tobytes() == want.tobytes()


def test_fast_division_device(gpu):
    """The hooks' per-pixel division equals IEEE float32 division."""
    rng = np.random.default_rng(11)
    n = 2_000_000
    d = np.concatenate([rng.integers(1, 65536, n // 2).astype(np.float32),
                        np.exp2(rng.uniform(-16, 16, n // 2)).astype(np.float32)])
    mag = np.exp2(rng.uniform(-60, 60, n)).astype(np.float32)
    p = (mag * rng.choice([-1.0, 1.0], n)).astype(np.float32)
    p[:1000] = 0.0
    p[1000:200000] = rng.integers(-200000, 200000, 199000).astype(np.float32)  # integral numerators
    q = np.zeros(n, np.float32)
    L.check(L.lib().pd_fast_div(0, n, L.ptr(p), L.ptr(d), L.ptr(q)))
    want = (p / d).astype(np.float32)
    assert np.array_equal(q, want)
    # outside the fast range the hooks use the plain division
    d2 = np.array([1e-30, 1e30, 2.0 ** 17, 2.0 ** -17, 3.0], np.float32)
    p2 = np.array([1.0, 5.0, 7.0, 1e-3, 1e-40], np.float32)
    q2 = np.zeros(5, np.float32)
    L.check(L.lib().pd_fast_div(0, 5, L.ptr(p2), L.ptr(d2), L.ptr(q2)))
    assert np.array_equal(q2[:4], (p2 / d2)[:4].astype(np.float32))


def _midpoint_numerators(d, rng):
    """Numerators p whose quotient p/d lies next to a rounding midpoint of
    float32 (the cases a one-step quotient could round the wrong way): for
    a random quotient q, the midpoint m between q and its successor, and
    p = RN(m * d) and its float neighbours."""
    q = rng.uniform(0.5, 200.0, d.size).astype(np.float32) * rng.choice([-1, 1], d.size).astype(np.float32)
    q = q.astype(np.float32)
    m = (q.astype(np.float64) + np.nextafter(q, np.float32(np.inf) * np.sign(q)).astype(np.float64)) / 2
    p0 = (m * d.astype(np.float64)).astype(np.float32)
    return [p0, np.nextafter(p0, np.float32(np.inf)), np.nextafter(p0, np.float32(-np.inf))]


def test_int_division_device(gpu):
    """The integer-depth hooks' one-correction quotient equals IEEE float32
    division for every integer depth 1..65535 and -32768..-1: random
    numerators over the offset range, integral ones, half-integer
    quotients, and numerators next to rounding midpoints."""
    rng = np.random.default_rng(12)
    dd = np.concatenate([np.arange(1, 65536), -np.arange(1, 32769)]).astype(np.float32)
    ps, ds = [], []
    for _ in range(3):
        ps.append(rng.uniform(-2.0e5, 2.0e5, dd.size).astype(np.float32))
        ds.append(dd)
    ps.append(rng.integers(-200000, 200000, dd.size).astype(np.float32))
    ds.append(dd)
    ps.append(((rng.integers(-300, 300, dd.size) + 0.5) * dd).astype(np.float32))   # p/d = k + 0.5
    ds.append(dd)
    for pm in _midpoint_numerators(dd, rng):
        ps.append(pm)
        ds.append(dd)
    mag = np.exp2(rng.uniform(-60, 60, dd.size)).astype(np.float32)
    ps.append((mag * rng.choice([-1.0, 1.0], dd.size)).astype(np.float32))
    ds.append(dd)
    p = np.concatenate(ps)
    d = np.concatenate(ds)
    q = np.zeros_like(p)
    L.check(L.lib().pd_int_div(0, p.size, L.ptr(p), L.ptr(d), L.ptr(q)))
    want = (p / d).astype(np.float32)
    normal = np.abs(want) >= np.float32(2.0 ** -126)
    assert np.array_equal(q[normal], want[normal])
    # subnormal quotients are below 0.5 and only ever round to offset 0
    assert np.all(np.abs(q[~normal]) < 0.5)


def test_count_ratio_division_device(gpu):
    """Class fractions p / d of a split (integer counts, p <= d < 2^21) through
    the one-correction quotient equal IEEE float32 division: random pairs
    over the whole range, every d up to 4096 with all p, p in {1, d-1, d}
    and numerators next to the midpoints of half-integer-free quotients."""
    rng = np.random.default_rng(13)
    ds, ps = [], []
    d = rng.integers(1, 1 << 21, 3_000_000)
    ds.append(d)
    ps.append((rng.random(d.size) * (d + 1)).astype(np.int64).clip(0, d))
    for k in range(1, 4097):
        ds.append(np.full(k + 1, k))
        ps.append(np.arange(k + 1))
    d2 = rng.integers(2, 1 << 21, 500_000)
    for pp in (np.ones_like(d2), d2 - 1, d2):
        ds.append(d2)
        ps.append(pp)
    d = np.concatenate(ds).astype(np.float32)
    p = np.concatenate(ps).astype(np.float32)
    assert np.all(d < 2 ** 21) and np.all(p <= d)
    q = np.zeros_like(p)
    L.check(L.lib().pd_int_div(0, p.size, L.ptr(p), L.ptr(d), L.ptr(q)))
    assert np.array_equal(q, (p / d).astype(np.float32))


def _rand_image(kind, rng, w, h):
    if kind == pa.PD_FEAT_DEPTH_F32:
        im = rng.uniform(0.5, 6.0, (h, w)).astype(np.float32)
        im[rng.integers(0, h, 5), rng.integers(0, w, 5)] = 0.0
        return im
    if kind == pa.PD_FEAT_RGBD_U16X4:
        im = rng.integers(0, 256, (h, w, 4)).astype(np.uint16)
        im[..., 3] = rng.integers(400, 5000, (h, w))
        im[rng.integers(0, h, 5), rng.integers(0, w, 5), 3] = 0
        return im
    im = rng.integers(400, 5000, (h, w)).astype(np.uint16)
    im[rng.integers(0, h, 5), rng.integers(0, w, 5)] = 0
    return im


@pytest.mark.parametrize("kind", KINDS)
def test_feature_eval_device(gpu, kind):
    rng = np.random.default_rng(3 + kind)
    w, h = 61, 47
    img = _rand_image(kind, rng, w, h)
    n = 20000
    xy = np.stack([rng.integers(0, w, n), rng.integers(0, h, n)], axis=1).astype(np.int32)
    fd = L.FEATURES[kind][3]
    scale = {0: 60.0, 1: 100000.0, 2: 100000.0, 3: 60.0}[kind]
    prm = rng.uniform(-scale, scale, (n, fd))
    if kind == pa.PD_FEAT_RGBD_U16X4:
        prm[:, 4:] = rng.uniform(-0.5, 4.5, (n, 2))
    if kind in (pa.PD_FEAT_DEPTH_U16, pa.PD_FEAT_RGBD_U16X4):
        # offsets far outside any image, up to quotients beyond the int range
        big = 10.0 ** rng.uniform(5, 38, (200, 4)) * rng.choice([-1.0, 1.0], (200, 4))
        prm[50:250, :4] = big
    prm = prm.astype(L.FEATURES[kind][2])
    prm[:50] = np.round(prm[:50])       # exact .5 quotients occur with integral offsets
    out = np.zeros(n, dtype=L.FEATURES[kind][2])
    L.check(L.lib().pd_feature_eval(0, kind, L.ptr(img), w, h, n, L.ptr(xy), L.ptr(prm), L.ptr(out)))
    want = np.array([orc.feature_at(kind, img, int(xy[i, 0]), int(xy[i, 1]), prm[i]) for i in range(n)])
    assert np.array_equal(out.astype(np.float64), want)


@pytest.mark.parametrize("kind", KINDS)
def test_candidate_tables_device(gpu, kind):
    fd = L.FEATURES[kind][3]
    lo = [-60.0, -60.0, -100.0, -100.0, 0.0, 0.0][:fd]
    hi = [60.0, 60.0, 100.0, 100.0, 4.0, 4.0][:fd]
    tb = (-200.0, 200.0) if kind == pa.PD_FEAT_DEMO_S16 else (-0.5, 0.5)
    p = pa.TreeTrainerParameters(37, 13, lo, hi, tb[0], tb[1], 0)
    nodes = np.array([0, 1, 2, 77, 65534, 524287], dtype=np.int32)
    fdt = L.FEATURES[kind][2]
    P = np.zeros((len(nodes), 37, fd), dtype=fdt)
    T = np.zeros((len(nodes), 37, 13), dtype=fdt)
    L.check(L.lib().pd_candidate_tables(0, kind, p.c(), 5, len(nodes), L.ptr(nodes), L.ptr(P), L.ptr(T)))
    for i, n in enumerate(nodes):
        for f in range(37):
            assert P[i, f].tobytes() == orc.feature_params(kind, 5, int(n), f, lo, hi).tobytes()
            assert T[i, f].tobytes() == orc.thresholds(kind, 5, int(n), f, 13, tb[0], tb[1]).tobytes()


def _tiny_ts(kind, rng, n_img=3, w=40, h=30, nC=5, ns=300):
    ts = pa.TrainingSet(nC)
    for _ in range(n_img):
        px = _rand_image(kind, rng, w, h)
        lab = rng.integers(1, nC + 1, (h, w)).astype(np.uint8)
        smp = np.sort(rng.integers(0, w * h, ns)).astype(np.uint32)
        ts << pa.TrainingSetImage(px, w, h, lab, nC, smp)
    return ts


@pytest.mark.parametrize("kind,nF,nT,chunk", [
    (pa.PD_FEAT_DEPTH_F32, 100, 10, 0),      # nF not a multiple of 64
    (pa.PD_FEAT_DEPTH_U16, 130, 20, 64),     # several chunks per node -> atomic flush
    (pa.PD_FEAT_DEPTH_U16, 64, 32, 0),
    (pa.PD_FEAT_RGBD_U16X4, 70, 7, 100),
    (pa.PD_FEAT_DEMO_S16, 40, 33, 0),        # 33 thresholds -> 48-slot rank bins
    (pa.PD_FEAT_DEPTH_F32, 5, 1, 0),
    (pa.PD_FEAT_DEPTH_F32, 3, 64, 0),
])
def test_hist_nodes_device(gpu, kind, nF, nT, chunk):
    rng = np.random.default_rng(100 + nF + nT)
    ts = _tiny_ts(kind, rng)
    fd = L.FEATURES[kind][3]
    if kind == pa.PD_FEAT_DEMO_S16:
        lo, hi, tb = [-60] * fd, [60] * fd, (-300, 300)
    elif kind == pa.PD_FEAT_DEPTH_F32:
        lo, hi, tb = [-60.0] * fd, [60.0] * fd, (-0.8, 0.8)
    else:
        lo, hi, tb = [-100000.0] * fd, [100000.0] * fd, (-800.0, 800.0)
        if kind == pa.PD_FEAT_RGBD_U16X4:
            lo[4:], hi[4:] = [0.0, 0.0], [4.0, 4.0]
    p = pa.TreeTrainerParameters(nF, nT, lo, hi, tb[0], tb[1], 0)
    tr = pa.HIPTreeTrainer(kind, ts.n_classes)
    tr.set_training_set(ts)
    if chunk:
        tr.set_chunk(chunk)
    S = sum(im.samples.size for im in ts.images)
    nodes = np.array([4, 0, 11, 12], dtype=np.int32)
    sample_node = rng.choice([0, 4, 11, 12, -1, 3], S).astype(np.int32)
    sample_node[:S // 3] = 0     # one big node
    H = tr.hist_nodes(p, 2, nodes, sample_node)
    want = orc.hist_nodes(orc.Tset(kind, ts), p, 2, nodes, sample_node)
    assert np.array_equal(H, want)
    tr.close()


@pytest.mark.parametrize("kind,nF,nT", [
    (pa.PD_FEAT_DEPTH_U16, 200, 20),      # 4 tiles, the last one partial
    (pa.PD_FEAT_DEMO_S16, 129, 6),        # the single-probe demo hook, 1-lane last tile
    (pa.PD_FEAT_RGBD_U16X4, 300, 9),
    (pa.PD_FEAT_DEPTH_U16, 4200, 3),      # two order segments (4096 + 104 candidates)
])
def test_probe_order_histograms_identical(gpu, kind, nF, nT):
    """Probe-coherent candidate tiles change which lane evaluates which
    candidate, never a count: hist_nodes with the order on and off both
    equal the oracle, in fused (single-chunk) and chunked nodes."""
    rng = np.random.default_rng(300 + nF)
    ts = _tiny_ts(kind, rng)
    fd = L.FEATURES[kind][3]
    if kind == pa.PD_FEAT_DEMO_S16:
        lo, hi, tb = [-60] * fd, [60] * fd, (-300, 300)
    else:
        lo, hi, tb = [-100000.0] * fd, [100000.0] * fd, (-800.0, 800.0)
        if kind == pa.PD_FEAT_RGBD_U16X4:
            lo[4:], hi[4:] = [0.0, 0.0], [4.0, 4.0]
    p = pa.TreeTrainerParameters(nF, nT, lo, hi, tb[0], tb[1], 0)
    S = sum(im.samples.size for im in ts.images)
    nodes = np.array([0, 5, 6], dtype=np.int32)
    sample_node = rng.choice([0, 5, 6, -1], S).astype(np.int32)
    want = orc.hist_nodes(orc.Tset(kind, ts), p, 1, nodes, sample_node)
    for order in (True, False):
        for chunk in (0, 50):
            tr = pa.HIPTreeTrainer(kind, ts.n_classes)
            tr.set_training_set(ts)
            tr.set_probe_order(order)
            if chunk:
                tr.set_chunk(chunk)
            H = tr.hist_nodes(p, 1, nodes, sample_node)
            tr.close()
            assert np.array_equal(H, want), (order, chunk)


def test_probe_order_tree_identical(gpu):
    """A C2-shaped tree with fused in-kernel split search (the winning lane
    is found through the candidate order) is the same with the order off."""
    ts = synth.training_set("c2", n_images=6, samples=300)
    p = synth.params_for("c2", n_features=500)
    trees = []
    for order in (True, False):
        tree = pa.Tree(0, 8, pa.PD_FEAT_DEPTH_U16, 8)
        tr = pa.HIPTreeTrainer(pa.PD_FEAT_DEPTH_U16, 8)
        tr.set_training_set(ts)
        tr.set_probe_order(order)
        tr.train(tree, ts, p, 1, 8)
        tr.close()
        trees.append(tree)
    a, b = trees
    assert np.array_equal(a.left_children, b.left_children)
    assert np.array_equal(a.features, b.features) and np.array_equal(a.thresholds, b.thresholds)
    assert np.array_equal(a.posteriors, b.posteriors)


@pytest.mark.parametrize("kind,nF,nT,nC", [
    (pa.PD_FEAT_DEPTH_F32, 150, 20, 5),   # NaN and +inf pixels: NaN responses rank above every threshold
    (pa.PD_FEAT_DEPTH_U16, 200, 32, 8),   # widest tile that keeps 32-bit bins (8 x 33 ranks)
    (pa.PD_FEAT_RGBD_U16X4, 100, 10, 3),
    (pa.PD_FEAT_DEPTH_U16, 90, 20, 21),   # too many classes for 32-bit bins: 16-bit either way
])
def test_bin_layouts_identical(gpu, kind, nF, nT, nC):
    """32-bit and 16-bit rank bins give the oracle's histograms, in fused
    (single-chunk) and chunked nodes."""
    rng = np.random.default_rng(500 + nF + nC)
    ts = _tiny_ts(kind, rng, nC=nC)
    if kind == pa.PD_FEAT_DEPTH_F32:
        for im in ts.images:
            px = im.data.reshape(im.height, im.width)
            px[rng.integers(0, im.height, 12), rng.integers(0, im.width, 12)] = np.nan
            px[rng.integers(0, im.height, 6), rng.integers(0, im.width, 6)] = np.inf
    fd = L.FEATURES[kind][3]
    if kind == pa.PD_FEAT_DEPTH_F32:
        lo, hi, tb = [-3.0] * fd, [3.0] * fd, (-2.0, 2.0)
    else:
        lo, hi, tb = [-100000.0] * fd, [100000.0] * fd, (-800.0, 800.0)
        if kind == pa.PD_FEAT_RGBD_U16X4:
            lo[4:], hi[4:] = [0.0, 0.0], [4.0, 4.0]
    p = pa.TreeTrainerParameters(nF, nT, lo, hi, tb[0], tb[1], 0)
    S = sum(im.samples.size for im in ts.images)
    nodes = np.array([0, 1, 2], dtype=np.int32)
    sample_node = rng.choice([0, 1, 2, -1], S).astype(np.int32)
    want = orc.hist_nodes(orc.Tset(kind, ts), p, 3, nodes, sample_node)
    for wide in (True, False):
        for chunk in (0, 50):
            tr = pa.HIPTreeTrainer(kind, nC)
            tr.set_training_set(ts)
            tr.set_wide_bins(wide)
            if chunk:
                tr.set_chunk(chunk)
            H = tr.hist_nodes(p, 3, nodes, sample_node)
            tr.close()
            assert np.array_equal(H, want), (wide, chunk)


def test_bin_layouts_tree_identical(gpu):
    """A C2-shaped tree (fused in-kernel split search reading the prefix
    counts, chunked nodes through H) is the same with 32-bit and 16-bit
    rank bins."""
    ts = synth.training_set("c2", n_images=6, samples=300)
    p = synth.params_for("c2", n_features=300)
    trees = []
    for wide in (True, False):
        tree = pa.Tree(2, 9, pa.PD_FEAT_DEPTH_U16, 8)
        tr = pa.HIPTreeTrainer(pa.PD_FEAT_DEPTH_U16, 8, tuned=False)
        tr.set_training_set(ts)
        tr.set_wide_bins(wide)
        tr.set_chunk(256)
        tr.train(tree, ts, p, 1, 9)
        tr.close()
        trees.append(tree)
    a, b = trees
    assert np.array_equal(a.left_children, b.left_children)
    assert np.array_equal(a.features, b.features) and a.thresholds.tobytes() == b.thresholds.tobytes()
    assert a.posteriors.tobytes() == b.posteriors.tobytes()


def test_split_search_device(gpu):
    rng = np.random.default_rng(7)
    for nC, nT, nF in [(4, 10, 100), (8, 20, 2000), (16, 32, 70), (21, 5, 9), (3, 2, 3)]:
        nodes = 3
        tot = rng.integers(1, 400, (nodes, nC)).astype(np.uint32)
        H = np.stack([np.stack([rng.integers(0, t + 1, (nT, nF)) for t in tot[q]]) for q in range(nodes)])
        H = H.astype(np.uint32)
        # node 0: every pair sends all samples right (gain 0) except two
        # identical informative pairs -> an exact tie between them
        H[0] = 0
        H[0, 0, nT - 1, 0] = tot[0, 0]
        H[0, :, 0, nF - 1] = H[0, :, nT - 1, 0]
        bk = np.zeros(nodes, dtype=np.uint32)
        bg = np.zeros(nodes, dtype=np.float32)
        allg = np.zeros((nodes, nT * nF), dtype=np.float32)
        L.check(L.lib().pd_split_search(0, nodes, nC, nT, nF, L.ptr(H), L.ptr(tot), L.ptr(bk), L.ptr(bg),
                                        L.ptr(allg)))
        for q in range(nodes):
            k, g = orc.best_split(H[q], tot[q])
            assert bk[q] == k and bg[q].tobytes() == np.float32(g).tobytes(), (nC, nT, nF, q)
            for kk in range(0, nT * nF, max(1, nT * nF // 50)):
                t, f = divmod(kk, nF)
                assert allg[q, kk].tobytes() == orc.gain_f32(H[q, :, t, f], tot[q]).tobytes()
        assert bk[0] == nF - 1    # (t=0, f=nF-1) precedes (t=nT-1, f=0) in threshold-major order


def _check_tree_equal(tree, out, diag):
    assert np.array_equal(tree.left_children, out["left_children"])
    assert tree.features.tobytes() == out["features"].tobytes()
    assert tree.thresholds.tobytes() == out["thresholds"].tobytes()
    assert tree.posteriors.tobytes() == out["posteriors"].tobytes()
    split = out["left_children"] >= 0
    assert np.array_equal(diag["node_k"][split], out["node_k"][split])
    assert diag["node_gain"][split].tobytes() == out["node_gain"][split].tobytes()
    assert np.allclose(diag["node_gain64"][split], out["node_gain64"][split], rtol=0, atol=1e-12)


@pytest.mark.parametrize("mode", [pa.PD_MODE_LEVEL_BATCHED, pa.PD_MODE_PER_NODE])
def test_train_c1_bit_exact(gpu, mode):
    """Config C1 in full: 32 images 160x120, 100 x 10, depth 8."""
    ts = synth.training_set("c1")
    p = synth.params_for("c1")
    c = synth.CONFIGS["c1"]
    tree = pa.Tree(0, c["depth"], c["kind"], c["n_classes"])
    tr = pa.HIPTreeTrainer(c["kind"], c["n_classes"])
    diag = tr.train(tree, ts, p, 1, c["depth"], mode=mode, diagnostics=True)
    out = orc.train_tree(orc.Tset(c["kind"], ts), p, ts.priors, 0, c["depth"])
    _check_tree_equal(tree, out, diag)
    assert (tree.left_children >= 0).sum() > 20
    st = tr.last_level_stats
    assert st[0]["active_samples"] == 32 * 256 and st[0]["evals"] == 32 * 256 * 100 * 10
    tr.close()


@pytest.mark.parametrize("chunk", [0, 64])
def test_train_c2_shape_bit_exact(gpu, chunk):
    """C2 shapes (320x240 uint16 capsules, 8 classes, 2000 x 20) on 12 images,
    depth 10.  chunk 0: automatic work items (nodes below one chunk are
    searched inside the histogram kernel); chunk 64: every node above 64
    samples is split over several work items adding into H, and a small
    histogram budget forces several slices per level."""
    ts = synth.training_set("c2", n_images=12, samples=400)
    p = synth.params_for("c2")
    tree = pa.Tree(1, 10, pa.PD_FEAT_DEPTH_U16, 8)
    tr = pa.HIPTreeTrainer(pa.PD_FEAT_DEPTH_U16, 8)
    tr.set_training_set(ts)
    if chunk:
        tr.set_chunk(chunk)
        tr.set_hist_budget(3 * 8 * 20 * 2000 * 4)
    diag = tr.train(tree, ts, p, 1, 10, diagnostics=True)
    if chunk:
        assert max(s["slices"] for s in tr.last_level_stats) > 1
    out = orc.train_tree(orc.Tset(pa.PD_FEAT_DEPTH_U16, ts), p, ts.priors, 1, 10)
    _check_tree_equal(tree, out, diag)
    tr.close()


def test_train_c3_shape_bit_exact(gpu):
    """C3 shapes (640x480 uint16 blob scenes, 16 classes, 32 thresholds:
    the largest LDS footprint) on 6 images x 1500 samples, 256 candidates,
    depth 12, with multi-item nodes (chunk 512) at the top levels."""
    ts = synth.training_set("c3", n_images=6, samples=1500)
    p = synth.params_for("c3", n_features=256)
    tree = pa.Tree(0, 12, pa.PD_FEAT_DEPTH_U16, 16)
    tr = pa.HIPTreeTrainer(pa.PD_FEAT_DEPTH_U16, 16)
    tr.set_training_set(ts)
    tr.set_chunk(512)
    diag = tr.train(tree, ts, p, 1, 12, diagnostics=True)
    out = orc.train_tree(orc.Tset(pa.PD_FEAT_DEPTH_U16, ts), p, ts.priors, 0, 12)
    _check_tree_equal(tree, out, diag)
    assert int((tree.left_children >= 0).sum()) > 20
    tr.close()


@pytest.mark.parametrize("waves,bpc,rules,spw", [(4, 4, (), 1), (16, 64, (), 1), (8, 1, (), 1),
                                                 (8, 16, ((2000, 16, 64), (300, 4, 8), (0, 8, 1)), 1),
                                                 (8, 16, (), 2), (16, 4, (), 4), (16, 64, (), 2),
                                                 (8, 32, ((2000, 16, 64, 4), (300, 8, 8, 2), (0, 4, 16, 1)), 2)])
def test_tuning_does_not_change_the_tree(gpu, waves, bpc, rules, spw):
    """Launch tuning (waves per block, work items per CU -> chunking, fused
    vs multi-chunk nodes, samples per wave step -> candidate tile width and
    bin layout) changes timing only: the tree is bit-identical."""
    from padenti_amd import autotune
    ts = synth.training_set("c2", n_images=10, samples=600)
    p = synth.params_for("c2", n_features=300)
    tr = pa.HIPTreeTrainer(pa.PD_FEAT_DEPTH_U16, 8, tuned=False)
    ref = pa.Tree(1, 10, pa.PD_FEAT_DEPTH_U16, 8)
    tr.train(ref, ts, p, 1, 10)
    autotune.set_tuning(tr, waves, bpc, rules, spw)
    got = pa.Tree(1, 10, pa.PD_FEAT_DEPTH_U16, 8)
    tr.train(got, ts, p, 1, 10)
    assert np.array_equal(got.left_children, ref.left_children)
    assert got.thresholds.tobytes() == ref.thresholds.tobytes()
    assert got.posteriors.tobytes() == ref.posteriors.tobytes()
    ms = ctypes.c_double()
    L.check(L.lib().pd_trainer_time_level(tr._h, p.c(), 0, 16, 1, ctypes.byref(ms)))
    assert ms.value > 0
    with pytest.raises(pa.PdError):
        autotune.set_tuning(tr, 5, 16)
    tr.close()


@pytest.mark.parametrize("cfg", ["c2", "c3", "spw2", "pool"])
def test_candidate_table_does_not_change_the_tree(gpu, cfg):
    """Candidate parameters and thresholds from the per-slice table or derived
    inside the histogram kernel: the same tree bit for bit (20 and 32
    thresholds, 16 classes with multi-item nodes, 32-candidate tiles, and a
    proposal run whose kept candidates go through a candidate map)."""
    from padenti_amd import autotune
    from padenti_amd import proposal as pp
    kind, nC, depth, mode = pa.PD_FEAT_DEPTH_U16, 8, 10, pa.PD_MODE_LEVEL_BATCHED
    if cfg == "c3":
        ts = synth.training_set("c3", n_images=4, samples=1500)
        p, nC = synth.params_for("c3", n_features=300), 16
    elif cfg == "pool":
        ts = synth.training_set("c2", n_images=10, samples=500)
        p, mode = synth.params_for("c2", n_features=2000, n_thresholds=1), pa.PD_MODE_PROPOSAL
    else:
        ts = synth.training_set("c2", n_images=10, samples=600)
        p = synth.params_for("c2", n_features=300)
    trees = []
    net = pp.SplitProposalNet(seed=3) if cfg == "pool" else None
    for on in (True, False):
        tr = pa.HIPTreeTrainer(kind, nC, tuned=False)
        tr.set_training_set(ts)
        if cfg == "spw2":
            autotune.set_tuning(tr, 8, 16, (), 2)
        if cfg == "c3":
            tr.set_chunk(512)
        if net is not None:
            tr.set_proposal(net, keep=200, min_samples=64, judge=False, screen=2000)
        tr.set_candidate_table(on)
        tree = pa.Tree(0, depth, kind, nC)
        tr.train(tree, ts, p, 1, depth, mode=mode)
        trees.append(tree)
        tr.close()
    if net is not None:
        net.close()
    a, b = trees
    assert (a.left_children >= 0).sum() > 10
    assert np.array_equal(a.left_children, b.left_children)
    assert a.thresholds.tobytes() == b.thresholds.tobytes()
    assert a.features.tobytes() == b.features.tobytes()
    assert a.posteriors.tobytes() == b.posteriors.tobytes()


@pytest.mark.parametrize("bins", [1, 2])
@pytest.mark.parametrize("cfg", ["c1", "c3"])
def test_bin_layout_tuning_trees_bit_exact(gpu, cfg, bins):
    """The tuning's bin layout against the oracle: 16-bit counts where the
    automatic layout would take 32-bit ones (c1: float responses, 4 classes x
    10 thresholds), and 32-bit counts for 16 classes x 32 thresholds, a tile
    that leaves one block per CU (c3 shapes, multi-item nodes)."""
    from padenti_amd import autotune
    if cfg == "c1":
        ts, p, kind, nC, depth = synth.training_set("c1"), synth.params_for("c1"), pa.PD_FEAT_DEPTH_F32, 4, 8
    else:
        ts = synth.training_set("c3", n_images=4, samples=1500)
        p, kind, nC, depth = synth.params_for("c3", n_features=200), pa.PD_FEAT_DEPTH_U16, 16, 10
    tr = pa.HIPTreeTrainer(kind, nC, tuned=False)
    tr.set_training_set(ts)
    autotune.set_tuning(tr, 16, 16, (), 1, bins)
    if cfg == "c3":
        tr.set_chunk(512)
    tree = pa.Tree(0, depth, kind, nC)
    diag = tr.train(tree, ts, p, 1, depth, diagnostics=True)
    out = orc.train_tree(orc.Tset(kind, ts), p, ts.priors, 0, depth)
    _check_tree_equal(tree, out, diag)
    assert (tree.left_children >= 0).sum() > 10
    with pytest.raises(pa.PdError):
        autotune.set_tuning(tr, 16, 16, (), 1, 3)
    tr.close()


@pytest.mark.parametrize("spw", [2, 4])
@pytest.mark.parametrize("cfg", ["c1", "c3", "pool"])
def test_samples_per_wave_trees_bit_exact(gpu, cfg, spw):
    """Tiles of 32 or 16 candidates with 2 or 4 samples per wave step, against
    the oracle: float responses with 32-bit bins (c1, 10 thresholds), 16
    classes x 32 thresholds with 16-bit bins and multi-item nodes (c3 shapes),
    and one threshold per candidate (the proposal pool's shape)."""
    from padenti_amd import autotune
    if cfg == "c1":
        ts, p, kind, nC, depth = synth.training_set("c1"), synth.params_for("c1"), pa.PD_FEAT_DEPTH_F32, 4, 8
    elif cfg == "c3":
        ts = synth.training_set("c3", n_images=4, samples=1500)
        p, kind, nC, depth = synth.params_for("c3", n_features=200), pa.PD_FEAT_DEPTH_U16, 16, 10
    else:
        ts = synth.training_set("c2", n_images=6, samples=500)
        p, kind, nC, depth = synth.params_for("c2", n_features=700, n_thresholds=1), pa.PD_FEAT_DEPTH_U16, 8, 9
    tr = pa.HIPTreeTrainer(kind, nC, tuned=False)
    tr.set_training_set(ts)
    autotune.set_tuning(tr, 16 if spw == 4 else 8, 16, (), spw)
    if cfg == "c3":
        tr.set_chunk(512)
    tree = pa.Tree(0, depth, kind, nC)
    diag = tr.train(tree, ts, p, 1, depth, diagnostics=True)
    out = orc.train_tree(orc.Tset(kind, ts), p, ts.priors, 0, depth)
    _check_tree_equal(tree, out, diag)
    assert (tree.left_children >= 0).sum() > 10
    tr.close()


def test_xcd_order_does_not_change_the_tree(gpu):
    """Placing multi-chunk work items on the XCDs by their position in the
    node's samples changes timing only (C3 shapes, chunks forced)."""
    ts = synth.training_set("c3", n_images=6, samples=1500)
    p = synth.params_for("c3", n_features=200)
    tr = pa.HIPTreeTrainer(pa.PD_FEAT_DEPTH_U16, 16, tuned=False)
    tr.set_training_set(ts)
    tr.set_chunk(256)
    trees = []
    for by_pos in (0, 1):
        tr.set_xcd_order(by_pos)
        t = pa.Tree(0, 10, pa.PD_FEAT_DEPTH_U16, 16)
        tr.train(t, ts, p, 1, 10)
        trees.append(t)
    assert np.array_equal(trees[0].left_children, trees[1].left_children)
    assert trees[0].thresholds.tobytes() == trees[1].thresholds.tobytes()
    assert trees[0].posteriors.tobytes() == trees[1].posteriors.tobytes()
    assert (trees[0].left_children >= 0).sum() > 20
    tr.close()


def test_lds_atomic_probe(gpu):
    ms, rate = ctypes.c_float(), ctypes.c_double()
    pa.check(pa.lib().pd_lds_atomic_bench(0, 64, 2, ctypes.byref(ms), ctypes.byref(rate)))
    assert ms.value > 0 and rate.value > 1e11
    with pytest.raises(pa.PdError):
        pa.check(pa.lib().pd_lds_atomic_bench(0, 0, 1, ctypes.byref(ms), ctypes.byref(rate)))


@pytest.mark.parametrize("kind", [pa.PD_FEAT_DEMO_S16, pa.PD_FEAT_RGBD_U16X4])
def test_train_other_hooks_bit_exact(gpu, kind):
    if kind == pa.PD_FEAT_DEMO_S16:
        ts = synth.training_set("c2", n_images=6, samples=300)
        p = pa.TreeTrainerParameters(128, 10, [-60, -60], [60, 60], -200, 200, 20)
        nC = 8
    else:
        ts = synth.training_set("c4", n_images=6, samples=300, w=160, h=120)
        p = synth.params_for("c4", n_features=150, n_thresholds=12)
        nC = 21
    tree = pa.Tree(3, 9, kind, nC)
    tr = pa.HIPTreeTrainer(kind, nC)
    diag = tr.train(tree, ts, p, 1, 9, diagnostics=True)
    out = orc.train_tree(orc.Tset(kind, ts), p, ts.priors, 3, 9)
    _check_tree_equal(tree, out, diag)
    tr.close()


def test_train_end_depth_and_root_gate(gpu):
    ts = synth.training_set("c1", n_images=4, samples=64)
    p = synth.params_for("c1", n_features=20, n_thresholds=4)
    tree = pa.Tree(0, 8, pa.PD_FEAT_DEPTH_F32, 4)
    tr = pa.HIPTreeTrainer(pa.PD_FEAT_DEPTH_F32, 4)
    tr.train(tree, ts, p, 1, 4)            # train only 3 levels of a depth-8 tree
    out = orc.train_tree(orc.Tset(0, ts), p, ts.priors, 0, 8, end_depth=4)
    assert np.array_equal(tree.left_children, out["left_children"])
    assert (tree.left_children[15:] == -2).all()   # levels 5.. do not exist
    p.per_leaf_samples_thr = 10000         # root holds fewer samples: empty histogram, no split
    tr.train(tree, ts, p, 1, 8)
    assert (tree.left_children == -2).all()
    with pytest.raises(ValueError):
        tr.train(tree, ts, p, 2, 8)
    tr.close()


def _c1_forest(n_trees=3, depth=8):
    ts = synth.training_set("c1")
    p = synth.params_for("c1")
    tr = pa.HIPTreeTrainer(pa.PD_FEAT_DEPTH_F32, 4)
    trees = []
    for t in range(n_trees):
        tree = pa.Tree(t, depth, pa.PD_FEAT_DEPTH_F32, 4)
        tr.train(tree, ts, p, 1, depth)
        trees.append(tree)
    tr.close()
    return trees


def test_predict_leaves_and_posterior(gpu):
    trees = _c1_forest()
    clf = pa.HIPClassifier(pa.PD_FEAT_DEPTH_F32, 4)
    for t in trees:
        clf << t
    rng = np.random.default_rng(9)
    for img, lab in synth.heldout("c1", n=4):
        h, w = img.shape
        mask = (rng.uniform(size=(h, w)) > 0.3).astype(np.uint8)
        for m in (None, mask):
            for ti, t in enumerate(trees):
                got = clf.predict_leaves(ti, img, w, h, m)
                assert np.array_equal(got, orc.predict_leaves(0, img, m, t))
            post = clf.predict_posterior(img, w, h, m)
            want = orc.predict_posterior(0, img, m, trees, 4)
            assert post.tobytes() == want.tobytes()
            p64 = np.zeros(post.shape)
            for t in trees:
                lv = orc.predict_leaves(0, img, m, t)
                p64 += t.posteriors[np.maximum(lv, 0)].transpose(2, 0, 1)
            on = (m if m is not None else np.ones((h, w), np.uint8))[None] > 0
            p64 = np.where(on, p64 / len(trees), 0.0)
            assert np.allclose(post, p64, rtol=1e-6, atol=1e-7)
    clf.close()


def test_predict_frames_graph(gpu):
    """Mixed-size frames in one launch, eager and replayed from a hipGraph."""
    trees = _c1_forest(n_trees=2, depth=7)
    clf = pa.HIPClassifier(pa.PD_FEAT_DEPTH_F32, 4)
    for t in trees:
        clf << t
    sizes = [(160, 120), (64, 48), (200, 90), (33, 17)]
    frames = [synth.gen_image(0, 0, 5000 + i, w, h, 4)[0] for i, (w, h) in enumerate(sizes)]
    npx = [w * h for w, h in sizes]
    img_off = np.concatenate([[0], np.cumsum(npx)[:-1]]).astype(np.uint64)
    post_off = (img_off * 4).astype(np.uint64)
    leaf_off = (img_off * 2).astype(np.uint64)
    masks = [np.ones(n, np.uint8) for n in npx]
    masks[1][::3] = 0
    host_pix = np.concatenate([f.reshape(-1) for f in frames]).astype(np.float32)
    host_mask = np.concatenate(masks)
    lib = L.lib()

    def dalloc(nbytes):
        p = ctypes.c_void_p()
        L.check(lib.pd_dev_alloc(0, nbytes, ctypes.byref(p)))
        return p

    d_pix, d_mask = dalloc(host_pix.nbytes), dalloc(host_mask.nbytes)
    d_post, d_leaf = dalloc(sum(npx) * 4 * 4), dalloc(sum(npx) * 2 * 4)
    L.check(lib.pd_memcpy_h2d(d_pix, L.ptr(host_pix), host_pix.nbytes))
    L.check(lib.pd_memcpy_h2d(d_mask, L.ptr(host_mask), host_mask.nbytes))
    w = np.array([s[0] for s in sizes], np.uint32)
    h = np.array([s[1] for s in sizes], np.uint32)
    mask_off = img_off.copy()
    ms = ctypes.c_float()
    outs = []
    for use_graph in (0, 1, 1, 1):
        L.check(lib.pd_forest_predict_frames_dev(clf._h, len(sizes), d_pix, host_pix.nbytes, L.ptr(img_off),
                                                 L.ptr(w), L.ptr(h), d_mask, host_mask.nbytes, L.ptr(mask_off),
                                                 d_post, sum(npx) * 4 * 4, L.ptr(post_off), d_leaf,
                                                 sum(npx) * 2 * 4, L.ptr(leaf_off), use_graph, ctypes.byref(ms)))
        post = np.zeros(sum(npx) * 4, np.float32)
        leaf = np.zeros(sum(npx) * 2, np.int32)
        L.check(lib.pd_memcpy_d2h(L.ptr(post), d_post, post.nbytes))
        L.check(lib.pd_memcpy_d2h(L.ptr(leaf), d_leaf, leaf.nbytes))
        outs.append((post, leaf))
        # eager work between replays
        clf.predict_posterior(frames[0], 160, 120)
    for post, leaf in outs[1:]:
        assert post.tobytes() == outs[0][0].tobytes() and np.array_equal(leaf, outs[0][1])
    post, leaf = outs[0]
    for i, (fw, fh) in enumerate(sizes):
        m = masks[i].reshape(fh, fw)
        want = orc.predict_posterior(0, frames[i], m, trees, 4).reshape(-1)
        got = post[post_off[i]:post_off[i] + 4 * npx[i]]
        assert got.tobytes() == want.tobytes(), i
        for t in range(2):
            wl = orc.predict_leaves(0, frames[i], m, trees[t]).reshape(-1)
            gl = leaf[leaf_off[i] + t * npx[i]:leaf_off[i] + (t + 1) * npx[i]]
            assert np.array_equal(gl, wl)
    for p in (d_pix, d_mask, d_post, d_leaf):
        lib.pd_dev_free(p)
    clf.close()


def _ragged_set(n_classes=4, seed=3):
    """Images of very different sizes (1x1 up to 97x61), samples on borders
    and corners (probes leave the image), duplicated samples, and one image
    without samples."""
    rng = np.random.default_rng(seed)
    ts = pa.TrainingSet(n_classes)
    sizes = [(97, 61), (1, 1), (5, 40), (64, 2), (33, 17), (12, 12)]
    for i, (w, h) in enumerate(sizes):
        img = synth.gen_image(0, seed, 9000 + i, max(w, 8), max(h, 8), n_classes)[0][:h, :w].copy()
        lab = rng.integers(1, n_classes + 1, size=(h, w)).astype(np.uint8)
        n = 0 if i == 4 else int(rng.integers(5, 60))
        smp = rng.integers(0, w * h, size=n).astype(np.uint32)
        if n:
            corners = np.array([0, w - 1, (h - 1) * w, h * w - 1], np.uint32)
            smp = np.sort(np.concatenate([smp, corners, smp[:3]]))   # corners + duplicates
        ts << pa.TrainingSetImage(img, w, h, lab, n_classes, smp)
    ts.priors = np.full(n_classes, 1.0 / n_classes, np.float32)   # the empty image has no priors of its own
    return ts


@pytest.mark.parametrize("nF,nT", [(1, 1), (65, 2), (100, 3)])
def test_train_ragged_and_degenerate_shapes(gpu, nF, nT):
    ts = _ragged_set()
    p = synth.params_for("c1", n_features=nF, n_thresholds=nT)
    p.per_leaf_samples_thr = 3
    tr = pa.HIPTreeTrainer(pa.PD_FEAT_DEPTH_F32, 4)
    tree = pa.Tree(2, 7, pa.PD_FEAT_DEPTH_F32, 4)
    diag = tr.train(tree, ts, p, 1, 7, diagnostics=True)
    out = orc.train_tree(orc.Tset(pa.PD_FEAT_DEPTH_F32, ts), p, ts.priors, 2, 7)
    _check_tree_equal(tree, out, diag)
    tr.close()


def test_train_pure_root_is_a_leaf(gpu):
    """Every sample of one class: every split has gain 0 and the oracle and
    the device agree on what the reference does with it."""
    ts = synth.training_set("c1", n_images=4, samples=64)
    for im in ts.images:
        im.labels[:] = 2
        im.priors = np.array([0, 1, 0, 0], np.float32)
    ts.priors = np.array([0, 1, 0, 0], np.float32)
    p = synth.params_for("c1", n_features=30, n_thresholds=5)
    tr = pa.HIPTreeTrainer(pa.PD_FEAT_DEPTH_F32, 4)
    tree = pa.Tree(0, 6, pa.PD_FEAT_DEPTH_F32, 4)
    diag = tr.train(tree, ts, p, 1, 6, diagnostics=True)
    out = orc.train_tree(orc.Tset(pa.PD_FEAT_DEPTH_F32, ts), p, ts.priors, 0, 6)
    _check_tree_equal(tree, out, diag)
    assert diag["node_gain"][0] == 0.0
    tr.close()


def test_predict_tiny_and_masked_frames(gpu):
    trees = _c1_forest(n_trees=2, depth=6)
    clf = pa.HIPClassifier(pa.PD_FEAT_DEPTH_F32, 4)
    for t in trees:
        clf << t
    img = synth.gen_image(0, 0, 7777, 8, 8, 4)[0]
    for w, h in ((1, 1), (1, 7), (8, 1)):
        sub = img[:h, :w].copy()
        post = clf.predict_posterior(sub, w, h)
        assert post.tobytes() == orc.predict_posterior(0, sub, None, trees, 4).tobytes()
        for ti, t in enumerate(trees):
            assert np.array_equal(clf.predict_leaves(ti, sub, w, h), orc.predict_leaves(0, sub, None, t))
    zero = np.zeros((8, 8), np.uint8)
    assert not clf.predict_posterior(img, 8, 8, zero).any()
    assert (clf.predict_leaves(0, img, 8, 8, zero) == -1).all()
    clf.close()


def test_predict_frames_rgbd_21_classes(gpu):
    """The batched-prediction workload's path: RGB-D hook, 21 classes (padded
    leaf rows), mixed frame sizes in one launch replayed from a hipGraph,
    against the oracle bit for bit."""
    nC = 21
    ts = synth.training_set("c4", n_images=12, samples=400, w=96, h=72)
    p = synth.params_for("c4", n_features=120, n_thresholds=10)
    tr = pa.HIPTreeTrainer(pa.PD_FEAT_RGBD_U16X4, nC)
    trees = []
    for t in range(3):
        tree = pa.Tree(t, 10, pa.PD_FEAT_RGBD_U16X4, nC)
        tr.train(tree, ts, p, 1, 10)
        trees.append(tree)
    tr.close()
    assert all((t.left_children >= 0).sum() > 20 for t in trees)
    clf = pa.HIPClassifier(pa.PD_FEAT_RGBD_U16X4, nC)
    for t in trees:
        clf << t
    sizes = [(120, 90), (33, 21), (64, 48), (1, 1), (200, 30), (400, 300)]
    frames = [synth.gen_image(synth.CONFIGS["c4"]["scene"], 7, 6000 + i, w, h, nC)[0] for i, (w, h) in enumerate(sizes)]
    npx = np.array([w * h for w, h in sizes], np.uint64)
    first = np.concatenate([[0], np.cumsum(npx)[:-1]]).astype(np.uint64)
    img_off, post_off, leaf_off = first * 4, first * nC, first * 3
    host = np.concatenate([f.reshape(-1) for f in frames]).astype(np.uint16)
    lib = L.lib()

    def dalloc(nbytes):
        q = ctypes.c_void_p()
        L.check(lib.pd_dev_alloc(0, int(nbytes), ctypes.byref(q)))
        return q

    total = int(npx.sum())
    d_pix, d_post, d_leaf = dalloc(host.nbytes), dalloc(total * nC * 4), dalloc(total * 3 * 4)
    L.check(lib.pd_memcpy_h2d(d_pix, L.ptr(host), host.nbytes))
    w = np.array([s[0] for s in sizes], np.uint32)
    h = np.array([s[1] for s in sizes], np.uint32)
    ms = ctypes.c_float()
    outs = []
    for use_graph in (1, 1, 0):
        L.check(lib.pd_forest_predict_frames_dev(clf._h, len(sizes), d_pix, host.nbytes, L.ptr(img_off),
                                                 L.ptr(w), L.ptr(h), None, 0, None, d_post, total * nC * 4,
                                                 L.ptr(post_off), d_leaf, total * 3 * 4, L.ptr(leaf_off),
                                                 use_graph, ctypes.byref(ms)))
        post = np.zeros(total * nC, np.float32)
        leaf = np.zeros(total * 3, np.int32)
        L.check(lib.pd_memcpy_d2h(L.ptr(post), d_post, post.nbytes))
        L.check(lib.pd_memcpy_d2h(L.ptr(leaf), d_leaf, leaf.nbytes))
        outs.append((post, leaf))
    for post, leaf in outs[1:]:
        assert post.tobytes() == outs[0][0].tobytes() and np.array_equal(leaf, outs[0][1])
    post, leaf = outs[0]
    for i, (fw, fh) in enumerate(sizes):
        n = int(npx[i])
        want = orc.predict_posterior(pa.PD_FEAT_RGBD_U16X4, frames[i], None, trees, nC).reshape(-1)
        assert post[int(post_off[i]):int(post_off[i]) + nC * n].tobytes() == want.tobytes(), i
        for t in range(3):
            wl = orc.predict_leaves(pa.PD_FEAT_RGBD_U16X4, frames[i], None, trees[t]).reshape(-1)
            assert np.array_equal(leaf[int(leaf_off[i]) + t * n:int(leaf_off[i]) + (t + 1) * n], wl)
    for q in (d_pix, d_post, d_leaf):
        lib.pd_dev_free(q)
    clf.close()


def test_error_paths(gpu):
    tr = pa.HIPTreeTrainer(pa.PD_FEAT_DEPTH_F32, 4)
    tree = pa.Tree(0, 5, pa.PD_FEAT_DEPTH_F32, 4)
    ts = synth.training_set("c1", n_images=2, samples=16)
    p = synth.params_for("c1", n_features=8, n_thresholds=65)
    with pytest.raises(pa.PdError) as e:
        tr.train(tree, ts, p, 1, 5)
    assert e.value.code == -1 and "n_thresholds" in str(e.value)
    bad = pa.TrainingSet(4)
    img = np.ones((8, 8), np.float32)
    lab = np.zeros((8, 8), np.uint8)
    lab[0, 0] = 1
    bad << pa.TrainingSetImage(img, 8, 8, lab, 4, np.array([0, 5], np.uint32))   # pixel 5 is unlabelled
    with pytest.raises(pa.PdError) as e:
        tr.set_training_set(bad)
    assert e.value.code == -1 and "unlabelled" in str(e.value)
    clf = pa.HIPClassifier(pa.PD_FEAT_DEPTH_F32, 4)
    t = pa.Tree(0, 3, pa.PD_FEAT_DEPTH_F32, 4)
    t.left_children[0] = 5    # not 2*0+1
    with pytest.raises(pa.PdError):
        clf << t
    with pytest.raises(pa.PdError):
        clf.predict_posterior(img, 8, 8)    # no trees
    clf.close()
    tr.close()


def test_predict_frames_rejects_out_of_range(gpu):
    """Every frame range is checked against the buffer sizes on the host
    before a launch: a frame reaching past d_pixels, d_post, d_leaves or
    d_masks, a height larger than the packing assumed, or an offset that
    wraps around is an argument error, and nothing is launched."""
    trees = _c1_forest(n_trees=1, depth=4)
    clf = pa.HIPClassifier(pa.PD_FEAT_DEPTH_F32, 4)
    clf << trees[0]
    lib = L.lib()
    w0, h0 = 32, 16
    npx = w0 * h0
    ptrs = []

    def dalloc(nbytes):
        q = ctypes.c_void_p()
        L.check(lib.pd_dev_alloc(0, int(nbytes), ctypes.byref(q)))
        ptrs.append(q)
        return q

    d_pix, d_post, d_leaf, d_mask = dalloc(npx * 4), dalloc(npx * 4 * 4), dalloc(npx * 4), dalloc(npx)
    host = np.full(npx, 3.0, np.float32)
    L.check(lib.pd_memcpy_h2d(d_pix, L.ptr(host), host.nbytes))
    zero = np.zeros(1, np.uint64)
    ms = ctypes.c_float()

    def call(img_off=zero, w=w0, h=h0, post_size=npx * 16, leaf_size=npx * 4, mask=False, mask_off=zero,
             post_off=zero, leaf_off=zero, pix_size=npx * 4):
        wa, ha = np.array([w], np.uint32), np.array([h], np.uint32)
        return lib.pd_forest_predict_frames_dev(clf._h, 1, d_pix, pix_size, L.ptr(img_off), L.ptr(wa), L.ptr(ha),
                                                d_mask if mask else None, npx, L.ptr(mask_off) if mask else None,
                                                d_post, post_size, L.ptr(post_off), d_leaf, leaf_size,
                                                L.ptr(leaf_off), 0, ctypes.byref(ms))

    assert call() == 0                       # the frame that fits
    assert call(mask=True) == 0
    bad = [
        dict(h=h0 + 1),                                   # taller than the buffers
        dict(w=h0, h=w0 + 1),                             # width and height swapped, one more row
        dict(img_off=np.array([1], np.uint64)),          # pixels end past d_pixels
        dict(post_off=np.array([1], np.uint64)),         # posteriors end past d_post
        dict(leaf_off=np.array([1], np.uint64)),         # leaf ids end past d_leaves
        dict(mask=True, mask_off=np.array([npx], np.uint64)),
        dict(img_off=np.array([2 ** 64 - 8], np.uint64)),  # wraps around
        dict(post_size=npx * 16 - 4),
        dict(pix_size=0),
    ]
    for kw in bad:
        code = call(**kw)
        assert code == L.PD_ERR_ARG, kw
        assert "outside" in lib.pd_last_error().decode(), kw
    L.check(lib.pd_dev_sync(0))
    for q in ptrs:
        lib.pd_dev_free(q)
    clf.close()



def _tie_ts(kind, rng, n_classes, n_samples, levels):
    """Images of a few distinct depths (many candidates with equal responses,
    so many (threshold, candidate) pairs with equal or nearly equal gains)."""
    ts = pa.TrainingSet(n_classes)
    for _ in range(3):
        w, h = 64, 48
        im = rng.choice(np.linspace(1000, 4000, levels).astype(np.uint16), (h, w))
        if kind == pa.PD_FEAT_DEPTH_F32:
            im = (im / 1000.0).astype(np.float32)
        lab = (1 + rng.integers(0, n_classes, (h, w))).astype(np.uint8)
        smp = np.sort(rng.integers(0, w * h, n_samples)).astype(np.uint32)
        ts << pa.TrainingSetImage(im, w, h, lab, n_classes, smp)
    return ts


@pytest.mark.parametrize("kind,n_classes,nF,nT,levels,samples", [
    (pa.PD_FEAT_DEPTH_U16, 8, 70, 20, 1, 300),     # one depth: every pair one-sided, all gains equal
    (pa.PD_FEAT_DEPTH_U16, 8, 70, 20, 2, 300),     # three responses: large groups of equal gains
    (pa.PD_FEAT_DEPTH_U16, 16, 130, 32, 3, 700),
    (pa.PD_FEAT_DEPTH_U16, 64, 65, 16, 3, 900),    # most classes
    (pa.PD_FEAT_DEPTH_U16, 4, 65, 64, 3, 900),     # most thresholds
    (pa.PD_FEAT_DEPTH_U16, 2, 64, 2, 4, 5000),     # two pairs per column, larger counts
    (pa.PD_FEAT_DEPTH_F32, 5, 100, 9, 2, 40),      # small nodes, bucket padding
    (pa.PD_FEAT_DEPTH_U16, 1, 64, 10, 3, 100),     # one class: every gain 0
])
def test_pruned_split_search_equals_exhaustive(gpu, kind, n_classes, nF, nT, levels, samples):
    """The fused split search evaluates exactly only the pairs whose
    approximate gain is within the error bound of the tile's largest: with
    groups of equal and nearly equal gains the winner (lowest pair index), its
    FP32 gain and the whole tree stay the oracle's."""
    rng = np.random.default_rng(1000 + n_classes + nT)
    ts = _tie_ts(kind, rng, n_classes, samples, levels)
    b, t = (60.0, 0.8) if kind == pa.PD_FEAT_DEPTH_F32 else (60000.0, 800.0)
    p = pa.TreeTrainerParameters(nF, nT, [-b] * 4, [b] * 4, -t, t, 5)
    tr = pa.HIPTreeTrainer(kind, n_classes)
    tr.set_training_set(ts)
    tree = pa.Tree(3, 7, kind, n_classes)
    diag = tr.train(tree, ts, p, 1, 7, diagnostics=True)
    ref = orc.train_tree(orc.Tset(kind, ts), p, ts.priors, 3, 7)
    assert np.array_equal(tree.left_children, ref["left_children"])
    assert tree.features.tobytes() == ref["features"].tobytes()
    assert tree.thresholds.tobytes() == ref["thresholds"].tobytes()
    assert tree.posteriors.tobytes() == ref["posteriors"].tobytes()
    trained = ref["left_children"] >= 0
    assert np.array_equal(diag["node_k"][trained], ref["node_k"][trained])
    assert diag["node_gain"][trained].tobytes() == ref["node_gain"][trained].tobytes()
    tr.close()


def test_count_logarithm_bound(gpu):
    """The bound of the approximate gain (gain_slack) takes the hardware
    logarithm of a count as within 2^-20 and its product with the count as
    rounded once (2^-24 of at most 16 k): k log2 k is within k 2^-19 for every
    count of a fused node."""
    k = np.arange(65536, dtype=np.uint32)
    out = np.full(k.size, np.nan, np.float32)
    L.check(L.lib().pd_count_klogk(0, k.size, L.ptr(k), L.ptr(out)))
    assert out[0] == 0.0 and out[1] == 0.0
    want = k[1:].astype(np.float64) * np.log2(k[1:].astype(np.float64))
    err = np.abs(out[1:].astype(np.float64) - want) / k[1:]
    assert err.max() <= 2.0 ** -19, (int(err.argmax()) + 1, err.max())


@pytest.mark.parametrize("kind", [pa.PD_FEAT_DEPTH_U16, pa.PD_FEAT_RGBD_U16X4])
@pytest.mark.parametrize("bound", [1000.0, 4194304.0, 4194308.0, 3e9])
def test_fast_offset_form_equals_oracle(gpu, kind, bound):
    """Offsets through one double FMA (feature bounds up to 2^22) and through
    the general form (above): histograms, trees and leaf ids are the oracle's,
    with depths for which half-integer quotients and offsets just inside and
    outside the image occur (1, powers of two, small and the largest depths)."""
    rng = np.random.default_rng(77)
    w, h, n_classes = 45, 33, 3
    ch = 4 if kind == pa.PD_FEAT_RGBD_U16X4 else 1
    ts = pa.TrainingSet(n_classes)
    for _ in range(2):
        d = rng.choice(np.array([0, 1, 2, 3, 64, 128, 1000, 4096, 40000, 65535], np.uint16), (h, w))
        im = d if ch == 1 else np.stack([rng.integers(0, 256, (h, w)).astype(np.uint16)] * 3 + [d], axis=-1)
        lab = (1 + rng.integers(0, n_classes, (h, w))).astype(np.uint8)
        smp = np.sort(rng.integers(0, w * h, 400)).astype(np.uint32)
        ts << pa.TrainingSetImage(im, w, h, lab, n_classes, smp)
    fd = L.FEATURES[kind][3]
    lo, hi = [-bound] * fd, [bound] * fd
    if ch == 4:
        lo[4:], hi[4:] = [0.0, 0.0], [4.0, 4.0]
    p = pa.TreeTrainerParameters(150, 6, lo, hi, -3000.0, 3000.0, 5)
    tr = pa.HIPTreeTrainer(kind, n_classes)
    tr.set_training_set(ts)
    o = orc.Tset(kind, ts)
    nodes = np.array([0, 4], dtype=np.int32)
    sample_node = rng.choice([0, 4, -1], 800).astype(np.int32)
    H = tr.hist_nodes(p, 2, nodes, sample_node)
    assert np.array_equal(H, orc.hist_nodes(o, p, 2, nodes, sample_node))
    tree = pa.Tree(2, 6, kind, n_classes)
    tr.train(tree, ts, p, 1, 6)
    ref = orc.train_tree(o, p, ts.priors, 2, 6)
    assert np.array_equal(tree.left_children, ref["left_children"])
    assert tree.features.tobytes() == ref["features"].tobytes()
    assert tree.posteriors.tobytes() == ref["posteriors"].tobytes()
    tr.close()
    clf = pa.HIPClassifier(kind, n_classes)
    clf << tree
    im = ts.images[0]
    got = clf.predict_leaves(0, im.data, w, h)
    assert np.array_equal(got, orc.predict_leaves(kind, im.data.reshape(h, w, ch) if ch > 1 else im.data.reshape(h, w),
                                                  None, tree).reshape(h, w))
    clf.close()
