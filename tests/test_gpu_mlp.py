"""GPU tests of the learned split proposal: the MFMA network against the FP64
oracle (forward, gradients, Adam), the top-k selection, the record emitter
of the plain trainer against the oracle's gains, proposal-mode trees
against plain training, and what the trained network gains over ranking
without it."""
import ctypes

import numpy as np
import pytest

import padenti_amd as pa
from padenti_amd import _lib as L
from padenti_amd import proposal as pp
from padenti_amd import synth
from oracle import mlp as om
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _rows(n, seed):
    """Inputs shaped like real records: a histogram summing to 1, depth,
    u, v, threshold in [-1, 1], then subsample statistics (fractions in
    [0, 1], a relative gain in [-0.2, 1])."""
    rng = np.random.default_rng(seed)
    h = rng.dirichlet(np.ones(8), size=n)
    x = np.zeros((n, om.IN))
    x[:, :8] = h
    x[:, 16] = rng.integers(1, 16, size=n) / 16.0
    x[:, 17:22] = rng.uniform(-1, 1, size=(n, 5))
    x[:, 22:30] = rng.uniform(0, 1, size=(n, 8))
    x[:, 30] = rng.uniform(-0.2, 1, size=n)
    x[:, 31] = rng.uniform(0, 1, size=n)
    return x.astype(np.float32)


def test_mfma_fragment_layout(gpu):
    rng = np.random.default_rng(0)
    A = rng.integers(-8, 9, size=(16, 32)).astype(np.float32)
    B = rng.integers(-8, 9, size=(32, 16)).astype(np.float32)
    a16 = pp.encode_rows(np.zeros((1, om.IN)))   # warm the encoder path
    assert a16.shape == (1, 32)
    Ab = (A.view(np.uint32) >> 16).astype(np.uint16)
    Bt = (np.ascontiguousarray(B.T).view(np.uint32) >> 16).astype(np.uint16)
    C = np.zeros((16, 16), dtype=np.float32)
    L.check(L.lib().pd_mma_probe(0, L.ptr(Ab), L.ptr(Bt), L.ptr(C)))
    np.testing.assert_array_equal(C, A @ B)   # small integers: exact


def test_forward_matches_oracle(gpu):
    net = pp.SplitProposalNet(seed=11)
    theta = net.params
    x = _rows(1000, 1)   # not a multiple of the 64-row tile
    y = net.forward(x)
    yb = om.forward(theta, x, bf16_mode=True)[0]
    y64 = om.forward(theta, x)[0]
    scale = np.max(np.abs(yb))
    assert np.max(np.abs(y - yb)) <= 2e-3 * scale + 1e-5
    assert np.max(np.abs(y - y64)) <= 3e-2 * scale
    net.close()


@pytest.mark.parametrize("n", [700, 9000, 33000])
def test_gradients_match_oracle(gpu, n):
    # 700 rows: two 512-row splits, the second partial, 32-row forward and
    # backward tiles, 64 x 32 weight-gradient tiles; 9000 rows: 64-row tiles;
    # 33000 rows: the large-batch kernels (128-row tiles, 64 x 64
    # weight-gradient tiles), 65 splits
    net = pp.SplitProposalNet(seed=12)
    theta = om.init_params(4, scale=2.0)
    net.params = theta
    theta = net.params   # as FP32
    x = _rows(n, 2)
    t = np.random.default_rng(3).uniform(0, 1, size=n).astype(np.float32)
    g, loss = net.grad(x, t)
    lref, gref = om.loss_and_grad(theta, x, t, bf16_mode=True)
    assert abs(loss - lref) <= 1e-4 * lref
    p, q = om.unpack(g), om.unpack(gref)
    for name, _ in om.SIZES:
        err = np.linalg.norm(p[name] - q[name]) / np.linalg.norm(q[name])
        assert err < 2e-2, (name, err)
    # the BF16 gradient is still a gradient of the exact loss
    g64 = om.loss_and_grad(theta, x, t)[1]
    assert np.dot(g, g64) / (np.linalg.norm(g) * np.linalg.norm(g64)) > 0.999
    net.close()


@pytest.mark.parametrize("n", [700, 9000, 33000])
@pytest.mark.parametrize("z", [3e5, 1e19, 3e19])   # z^2 in FP32: finite, finite, infinite
def test_gradients_with_saturated_units(gpu, n, z):
    """Units far out on either side of the GELU (gelu' is 1 and 0 there) leave
    every gradient finite and the oracle's."""
    theta = om.init_params(6, scale=2.0)
    q = om.unpack(theta)
    q["W1"][:2], q["b1"][:2], q["W2"][:, :2] = 0.0, (z, -z), 0.0   # (views of theta's own values)
    theta = om.pack(q)
    net = pp.SplitProposalNet(seed=12)
    net.params = theta
    theta = net.params
    x = _rows(n, 7)
    t = np.random.default_rng(8).uniform(0, 1, size=n).astype(np.float32)
    g, loss = net.grad(x, t)
    lref, gref = om.loss_and_grad(theta, x, t, bf16_mode=True)
    assert np.all(np.isfinite(g)) and abs(loss - lref) <= 1e-4 * lref
    p, q = om.unpack(g), om.unpack(gref)
    big_p, big_q = p["W2"][:, :2].copy(), q["W2"][:, :2].copy()
    assert np.linalg.norm(big_p - big_q) <= 2e-2 * np.linalg.norm(big_q)
    p["W2"][:, :2] = q["W2"][:, :2] = 0.0
    for name, _ in om.SIZES:
        err = np.linalg.norm(p[name] - q[name]) / np.linalg.norm(q[name])
        assert err < 2e-2, (name, err)
    net.close()


def test_adam_steps_match_oracle(gpu):
    net = pp.SplitProposalNet(seed=13)
    x = _rows(512, 4)
    t = np.random.default_rng(5).uniform(0, 1, size=512).astype(np.float32)
    opt = pp.adam(lr=2e-3, beta1=0.9, beta2=0.99, eps=1e-7)
    th = net.params.astype(np.float64)
    m = np.zeros_like(th)
    v = np.zeros_like(th)
    for k in (1, 2):
        g, _ = net.grad(x, t)   # the gradient the step uses (deterministic kernels)
        net.step(x, t, opt)
        th, m, v = om.adam_step(th, m, v, g.astype(np.float64), k, lr=2e-3, beta1=0.9, beta2=0.99, eps=1e-7)
        np.testing.assert_allclose(net.params, th, rtol=2e-6, atol=2e-8)
    net.close()


def test_training_reduces_loss(gpu):
    x = _rows(65536, 6)
    # a smooth target of the candidate inputs and the histogram
    t = (0.3 * np.tanh(2 * x[:, 17] * x[:, 19]) + 0.2 * x[:, 21] ** 2 + 0.5 * x[:, 0]).astype(np.float32)
    buf = pp.RecordBuffer(len(t))
    buf.upload(pp.encode_rows(x), t)
    net = pp.SplitProposalNet(seed=14)
    y0 = net.forward(x[:4096])
    l0 = float(np.mean((y0 - t[:4096]) ** 2))
    loss, ms = net.train_records(buf, batch=1024, epochs=3, opt=pp.adam(lr=1e-3), target="gain")
    y1 = net.forward(x[:4096])
    l1 = float(np.mean((y1 - t[:4096]) ** 2))
    assert loss[-1] < loss[0] and l1 < 0.2 * l0, (l0, l1, loss)
    buf.close()
    net.close()


def test_topk_selection(gpu):
    rng = np.random.default_rng(7)
    K, keep, ns = 3000, 300, 5
    s = rng.normal(size=(ns, K)).astype(np.float32)
    s[1] = np.round(s[1] * 4) / 4          # many ties
    s[2] = 1.0                             # all tied: the first keep
    s[3, ::2] = -np.inf
    sel = np.zeros((ns, keep), dtype=np.uint32)
    L.check(L.lib().pd_topk_select(0, L.ptr(s), ns, K, keep, keep, L.ptr(sel)))
    for q in range(ns):
        want = np.sort(np.argsort(-s[q], kind="stable")[:keep])
        np.testing.assert_array_equal(sel[q], want)
    # screened selection: the first `keep` (by index) of the best 1000
    L.check(L.lib().pd_topk_select(0, L.ptr(s), ns, K, 1000, keep, L.ptr(sel)))
    for q in range(ns):
        want = np.sort(np.argsort(-s[q], kind="stable")[:1000])[:keep]
        np.testing.assert_array_equal(sel[q], want)


def test_record_emitter_matches_oracle(gpu):
    """Root level only, records of every pair in order: row j is pair
    (t, f) = (j / nF, j % nF) of node 0."""
    ts = synth.training_set("c2", n_images=4, samples=300)
    p = synth.params_for("c2", n_features=70, n_thresholds=6)
    nC, nF, nT = 8, 70, 6
    tr = pa.HIPTreeTrainer(pa.PD_FEAT_DEPTH_U16, nC)
    buf = pp.RecordBuffer(nF * nT)
    tr.set_record_sink(buf, per_node=nF * nT)
    tree = pa.Tree(2, 4, pa.PD_FEAT_DEPTH_U16, nC)
    tr.train(tree, ts, p, 1, 2)
    assert tr.records_written() == nF * nT
    rows, gains, rel = buf.download(rel=True)
    o = orc.Tset(pa.PD_FEAT_DEPTH_U16, ts)
    H = orc.hist_nodes(o, p, 2, [0], np.zeros(o.total, dtype=np.int32))[0]   # [c][t][f]
    cnt = np.bincount(np.concatenate([im.labels[im.samples] for im in ts.images]).astype(np.int64) - 1,
                      minlength=nC)[:nC].astype(np.uint32)
    want_g = np.zeros(nT * nF, dtype=np.float32)
    for j in range(nT * nF):
        t_, f_ = divmod(j, nF)
        want_g[j] = orc.gain_f32(H[:, t_, f_], cnt)
    assert gains.tobytes() == want_g.tobytes()
    best = want_g.max()
    assert rel.tobytes() == (want_g / best).astype(np.float32).tobytes()
    x = pp.bf16_to_f32(rows[:, :om.IN])
    hist = cnt / cnt.sum()
    lo = np.array(p.feat_low_bounds, dtype=np.float32)
    hi = np.array(p.feat_up_bounds, dtype=np.float32)
    for j in range(0, nT * nF, 37):
        t_, f_ = divmod(j, nF)
        par = orc.feature_params(pa.PD_FEAT_DEPTH_U16, 2, 0, f_, lo, hi)
        thr = orc.thresholds(pa.PD_FEAT_DEPTH_U16, 2, 0, f_, nT, p.thr_low_bound, p.thr_up_bound)[t_]
        want = np.zeros(om.IN, dtype=np.float32)
        want[:nC] = (cnt.astype(np.float32) / np.float32(cnt.sum()))
        want[16] = np.float32(1) / np.float32(16)
        want[17:21] = np.asarray(par, dtype=np.float32)[:4] * (np.float32(1) / np.maximum(np.abs(lo), np.abs(hi)))
        want[21] = (np.float32(thr) - np.float32(p.thr_low_bound)) * (
            np.float32(2) / (np.float32(p.thr_up_bound) - np.float32(p.thr_low_bound))) - np.float32(1)
        np.testing.assert_array_equal(x[j], om.bf16(want).astype(np.float32))
    assert np.allclose(x[0, :nC], hist, atol=4e-3)
    tr.close()
    buf.close()


def _pool_params(K):
    return synth.params_for("c2", n_features=K, n_thresholds=1)


def test_proposal_keep_all_equals_plain(gpu):
    """keep == K selects every candidate: the tree is the plain tree, and the
    plain tree with nT = 1 is the oracle's."""
    ts = synth.training_set("c2", n_images=10, samples=400)
    K = 200
    p = _pool_params(K)
    tr = pa.HIPTreeTrainer(pa.PD_FEAT_DEPTH_U16, 8)
    plain = pa.Tree(0, 9, pa.PD_FEAT_DEPTH_U16, 8)
    tr.train(plain, ts, p, 1, 9)
    out = orc.train_tree(orc.Tset(pa.PD_FEAT_DEPTH_U16, ts), p, ts.priors, 0, 9)
    assert np.array_equal(plain.left_children, out["left_children"])
    assert plain.thresholds.tobytes() == out["thresholds"].tobytes()
    net = pp.SplitProposalNet(seed=21)
    tr.set_proposal(net, keep=K, min_samples=0, judge=True)
    prop = pa.Tree(0, 9, pa.PD_FEAT_DEPTH_U16, 8)
    tr.train(prop, ts, p, 1, 9, mode=pa.PD_MODE_PROPOSAL)
    assert np.array_equal(prop.left_children, plain.left_children)
    assert prop.features.tobytes() == plain.features.tobytes()
    assert prop.thresholds.tobytes() == plain.thresholds.tobytes()
    assert prop.posteriors.tobytes() == plain.posteriors.tobytes()
    st = tr.last_level_stats
    assert sum(s["proposal_nodes"] for s in st) > 10
    assert sum(s["judged_nodes"] for s in st) == sum(s["proposal_nodes"] for s in st)
    assert all(s["gain_loss_rel"] == 0.0 for s in st)
    tr.close()
    net.close()


def test_proposal_refine_full_sample_equals_plain(gpu):
    """Refinement over every sample (stride 1) of the whole pool ranks the
    candidates by their exact gains, so the kept quarter holds each node's
    best split and the tree is the plain tree over the whole pool (also
    with the minimum subsample covering small nodes, stride 4)."""
    ts = synth.training_set("c2", n_images=10, samples=400)
    K = 256
    p = _pool_params(K)
    tr = pa.HIPTreeTrainer(pa.PD_FEAT_DEPTH_U16, 8)
    plain = pa.Tree(0, 9, pa.PD_FEAT_DEPTH_U16, 8)
    tr.train(plain, ts, p, 1, 9)
    net = pp.SplitProposalNet(seed=21)
    for stride, min_sub in ((1, 0), (4, 1 << 20)):
        tr.set_proposal(net, keep=K // 4, min_samples=0, judge=True, screen=K)
        tr.set_proposal_refine(stride, min_sub)
        prop = pa.Tree(0, 9, pa.PD_FEAT_DEPTH_U16, 8)
        tr.train(prop, ts, p, 1, 9, mode=pa.PD_MODE_PROPOSAL)
        assert np.array_equal(prop.left_children, plain.left_children), stride
        assert prop.features.tobytes() == plain.features.tobytes()
        assert prop.thresholds.tobytes() == plain.thresholds.tobytes()
        st = tr.last_level_stats
        assert sum(s["proposal_nodes"] for s in st) > 10
        assert all(s["gain_loss_rel"] == 0.0 for s in st)
        assert sum(s["refine_ms"] for s in st) > 0.0
    # a real subsample (every 4th sample of nodes above 64) keeps most of the gain
    tr.set_proposal_refine(4, 64)
    prop = pa.Tree(0, 9, pa.PD_FEAT_DEPTH_U16, 8)
    tr.train(prop, ts, p, 1, 9, mode=pa.PD_MODE_PROPOSAL)
    assert _mean_gain_loss(tr.last_level_stats) < 0.05
    tr.set_proposal_refine(0, 0)
    tr.close()
    net.close()


def _mean_gain_loss(st):
    n = sum(s["judged_nodes"] for s in st)
    return sum(s["gain_loss_rel"] for s in st) / max(n, 1)


def _spearman(a, b):
    ra = np.argsort(np.argsort(a)).astype(np.float64)
    rb = np.argsort(np.argsort(b)).astype(np.float64)
    return float(np.corrcoef(ra, rb)[0, 1])


@pytest.mark.xfail(reason="the 22-input network ranks a node's pool no better than the pool's own order "
                          "(mean gain loss of its top 10% above the network-free ranking's)", strict=False)
def test_trained_network_ranks_the_pool(gpu):
    """What the trained network gains over ranking without it.  Records from
    plain runs with the mid-size settings (2000 x 20) on other data (seeds 1,
    2) train the network on the relative gain.  On seed-0 data every
    candidate of the pool (K = 4000, one threshold each) of the first tree
    levels is emitted with its exhaustive gain: the network's scores must
    rank them better than chance within each node (mean Spearman > 0.05; a
    network-free ranking has no correlation).  The judge's mean gain loss of
    the top 10% against the whole pool is reported for the trained network
    and for ranking without it (the first 10% of the pool)."""
    nC = 8
    tr = pa.HIPTreeTrainer(pa.PD_FEAT_DEPTH_U16, nC)
    buf = pp.RecordBuffer(6_000_000)
    tr.set_record_sink(buf, per_node=500)
    for seed in (1, 2):
        train_ts = synth.training_set("c2", seed=seed, n_images=150, samples=1000)
        for tid in range(2):
            tr.train(pa.Tree(tid, 13, pa.PD_FEAT_DEPTH_U16, nC), train_ts, synth.params_for("c2"), 1, 13)
    assert tr.records_written() > 1_000_000
    tr.set_record_sink(None, 0)
    net = pp.SplitProposalNet(seed=3)
    loss, _ = net.train_records(buf, batch=4096, epochs=3, opt=pp.adam(lr=1e-3))
    assert loss[-1] < loss[0]
    buf.close()
    K = 4000
    ts = synth.training_set("c2", seed=0, n_images=60, samples=1000)
    pool = _pool_params(K)
    pbuf = pp.RecordBuffer(16 * K)
    tr.set_record_sink(pbuf, per_node=K)
    tr.train(pa.Tree(0, 5, pa.PD_FEAT_DEPTH_U16, nC), ts, pool, 1, 5)
    n = tr.records_written()
    tr.set_record_sink(None, 0)
    x, g = pbuf.download()
    pbuf.close()
    y = net.forward(pp.bf16_to_f32(x[:, :om.IN]))
    cors = [_spearman(y[a:a + K], g[a:a + K]) for a in range(0, n, K) if g[a:a + K].max() > 0]
    assert len(cors) >= 8
    mean_cor = float(np.mean(cors))

    def judged(theta):
        net.params = theta
        tr.set_proposal(net, keep=K // 10, min_samples=100, judge=True)
        tr.train(pa.Tree(0, 9, pa.PD_FEAT_DEPTH_U16, nC), ts, pool, 1, 9, mode=pa.PD_MODE_PROPOSAL)
        return _mean_gain_loss(tr.last_level_stats)

    trained = net.params
    loss_trained = judged(trained)
    loss_const = judged(np.zeros_like(trained))
    print(f"within-node Spearman {mean_cor:.3f} over {len(cors)} nodes; mean relative gain loss of the "
          f"top 10%: trained {loss_trained:.4f}, without the network {loss_const:.4f}")
    assert mean_cor > 0.05, cors
    assert 0.0 <= loss_trained <= 1.0 and 0.0 <= loss_const <= 1.0
    # the network must beat ranking without it by a clear margin
    assert loss_trained < 0.8 * loss_const, (loss_trained, loss_const)
    tr.close()
    net.close()


def test_stratified_refinement_whole_node_equals_plain(gpu):
    """The class-stratified refinement over a subsample that is the whole
    node (stride 1) estimates every candidate's gain from complete counts:
    the kept quarter holds each node's best split and the tree is the plain
    tree over the whole pool; with the learned correction of a zero-weight
    network (mode 2) it ranks exactly as the estimate (mode 1)."""
    ts = synth.training_set("c2", n_images=10, samples=400)
    K = 256
    p = _pool_params(K)
    tr = pa.HIPTreeTrainer(pa.PD_FEAT_DEPTH_U16, 8)
    plain = pa.Tree(0, 9, pa.PD_FEAT_DEPTH_U16, 8)
    tr.train(plain, ts, p, 1, 9)
    net = pp.SplitProposalNet(seed=21)
    net.params = np.zeros(pp.NPARAM, np.float32)
    trees = {}
    for mode in (1, 2):
        tr.set_proposal(net, keep=K // 4, min_samples=0, judge=True, screen=K)
        tr.set_proposal_refine(1, 0)
        tr.set_proposal_strata(mode)
        prop = pa.Tree(0, 9, pa.PD_FEAT_DEPTH_U16, 8)
        tr.train(prop, ts, p, 1, 9, mode=pa.PD_MODE_PROPOSAL)
        st = tr.last_level_stats
        assert sum(s["proposal_nodes"] for s in st) > 10
        assert all(s["gain_loss_rel"] == 0.0 for s in st), mode
        assert np.array_equal(prop.left_children, plain.left_children), mode
        assert prop.thresholds.tobytes() == plain.thresholds.tobytes()
        trees[mode] = prop
    # a real stratified subsample (1/8 of each node, at least 64) keeps most of
    # the gain, and a zero-weight correction changes nothing
    diag = {}
    for mode in (1, 2):
        tr.set_proposal_refine(8, 64)
        tr.set_proposal_strata(mode)
        prop = pa.Tree(0, 9, pa.PD_FEAT_DEPTH_U16, 8)
        diag[mode] = tr.train(prop, ts, p, 1, 9, mode=pa.PD_MODE_PROPOSAL, diagnostics=True)
        trees[10 + mode] = prop
        assert _mean_gain_loss(tr.last_level_stats) < 0.05
    assert np.array_equal(trees[11].left_children, trees[12].left_children)
    assert trees[11].thresholds.tobytes() == trees[12].thresholds.tobytes()
    # the kept candidates are histogrammed exactly: at every split node of the
    # proposal tree the chosen candidate's gain is its exact FP32 gain over the
    # node's samples (CPU: route through the tree, gains of the whole pool),
    # and no larger than the pool's best
    from oracle import cpu_ref as cr
    o = orc.Tset(pa.PD_FEAT_DEPTH_U16, ts)
    tree = trees[11]
    d = {"left_children": tree.left_children, "features": tree.features, "thresholds": tree.thresholds}
    checked = 0
    for level in range(1, 9):
        at = cr.route_samples(o, d, level - 1)
        for n in range((1 << (level - 1)) - 1, (1 << level) - 1):
            if tree.left_children[n] < 0:
                continue
            idx = np.nonzero(at == n)[0].astype(np.uint32)
            g = cr.pool_gains(o, p, 0, n, idx)
            k = int(diag[1]["node_k"][n])
            assert g[k].tobytes() == diag[1]["node_gain"][n].tobytes(), n
            assert g[k] <= g.max()
            checked += 1
    assert checked > 20
    tr.set_proposal_refine(0, 0)
    tr.set_proposal_strata(0)
    tr.close()
    net.close()


def test_refinement_records_match_oracle(gpu):
    """Records of the learned refinement at the root: every target is the
    exact FP32 gain of one of the pool's candidates over all of the node's
    samples (the oracle's histogram), the statistics columns are fractions
    and a relative gain, and the relative target is the exact relative gain
    minus the estimated one (column 30)."""
    ts = synth.training_set("c2", n_images=6, samples=400)
    K, R, nC = 300, 64, 8
    p = _pool_params(K)
    tr = pa.HIPTreeTrainer(pa.PD_FEAT_DEPTH_U16, nC)
    net = pp.SplitProposalNet(seed=3)
    buf = pp.RecordBuffer(4 * R)
    tr.set_record_sink(buf, per_node=R)
    tr.set_proposal(net, keep=K // 4, min_samples=0, judge=False, screen=K)
    tr.set_proposal_refine(4, 64)
    tr.set_proposal_strata(1)
    tr.train(pa.Tree(2, 4, pa.PD_FEAT_DEPTH_U16, nC), ts, p, 1, 2, mode=pa.PD_MODE_PROPOSAL)
    assert tr.records_written() == R
    rows, gains, rel = buf.download(rel=True)
    tr.set_record_sink(None, 0)
    o = orc.Tset(pa.PD_FEAT_DEPTH_U16, ts)
    H = orc.hist_nodes(o, p, 2, [0], np.zeros(o.total, dtype=np.int32))[0]   # [c][0][f]
    cnt = np.bincount(np.concatenate([im.labels[im.samples] for im in ts.images]).astype(np.int64) - 1,
                      minlength=nC)[:nC].astype(np.uint32)
    want = np.array([orc.gain_f32(H[:, 0, f], cnt) for f in range(K)], dtype=np.float32)
    assert set(gains.view(np.uint32).tolist()) <= set(want.view(np.uint32).tolist())
    x = pp.bf16_to_f32(rows[:, :om.IN])
    assert (x[:, 22:30] >= 0).all() and (x[:, 22:30] <= 1.0001).all()
    assert (x[:, 31] >= 0).all() and (x[:, 31] <= 1.0001).all()
    assert (x[:, 30] <= 1.0001).all() and x[:R // 2, 30].max() > 0.99   # the best estimate is among the first half
    assert np.allclose(rel, gains / want.max() - x[:, 30], atol=1e-2)
    tr.set_proposal_refine(0, 0)
    tr.set_proposal_strata(0)
    buf.close()
    tr.close()
    net.close()


def test_proposal_tree_is_exact_given_its_choices(gpu):
    """A proposal tree that histograms only part of the pool (the stratified
    estimate keeps 40 of K = 300 candidates per ranked node), checked node by
    node against the oracle.  The samples are routed through the tree with
    the oracle's feature; then every split is a pool candidate -- its
    parameters and threshold are the sampler's for the reported index --
    whose exact FP32 gain over the node's samples (the oracle's histogram)
    is the gain the trainer reports; a node below min_samples (evaluated on
    the whole pool) takes the oracle's exhaustive first maximum; a ranked
    node's choice is never better than that maximum; and a leaf's posterior
    is its samples' class frequency."""
    kind, nC, K, keep, depth, ranked = pa.PD_FEAT_DEPTH_U16, 8, 300, 40, 7, 300
    ts = synth.training_set("c2", n_images=8, samples=400)
    p = _pool_params(K)
    net = pp.SplitProposalNet(seed=3)
    tr = pa.HIPTreeTrainer(pa.PD_FEAT_DEPTH_U16, nC)
    tr.set_proposal(net, keep=keep, min_samples=ranked, judge=False, screen=K)
    tr.set_proposal_refine(4, 64)
    tr.set_proposal_strata(1)
    tree = pa.Tree(4, depth, kind, nC)
    diag = tr.train(tree, ts, p, 1, depth, mode=pa.PD_MODE_PROPOSAL, diagnostics=True)
    tr.set_proposal_refine(0, 0)
    tr.set_proposal_strata(0)
    tr.close()
    net.close()
    # route every sample through the tree (oracle feature evaluation)
    lab, node_of = [], []
    for im in ts.images:
        img = im.data.reshape(im.height, im.width)
        for s in im.samples.tolist():
            x, y, n, path = s % im.width, s // im.width, 0, [0]
            while tree.left_children[n] >= 0:
                v = np.float32(orc.feature_at(kind, img, x, y, tree.features[n]))
                n = 2 * n + 1 if v <= tree.thresholds[n] else 2 * n + 2
                path.append(n)
            path += [-1] * (depth - len(path))
            node_of.append(path)
            lab.append(int(im.labels[s]) - 1)
    node_of = np.array(node_of, dtype=np.int32)   # [sample][level]
    lab = np.array(lab)
    o = orc.Tset(kind, ts)
    n_ranked = n_fallback = 0
    for d in range(depth - 1):
        level = node_of[:, d]
        nodes = [int(q) for q in np.unique(level[level >= 0]) if tree.left_children[q] >= 0]
        if not nodes:
            continue
        H = orc.hist_nodes(o, p, tree.id, nodes, level)
        for i, q in enumerate(nodes):
            tot = np.bincount(lab[level == q], minlength=nC).astype(np.uint32)
            f = int(diag["node_k"][q]) % K
            assert tree.features[q].tobytes() == orc.feature_params(kind, tree.id, q, f, p.feat_low_bounds,
                                                                     p.feat_up_bounds).tobytes()
            assert tree.thresholds[q] == orc.thresholds(kind, tree.id, q, f, 1, p.thr_low_bound, p.thr_up_bound)[0]
            g = orc.gain_f32(H[i, :, 0, f], tot)
            assert g.tobytes() == diag["node_gain"][q].tobytes(), (q, g, diag["node_gain"][q])
            k_ex, g_ex = orc.best_split(H[i], tot)
            if tot.sum() == ranked:
                continue   # at the boundary: either treatment is allowed
            if tot.sum() < ranked:
                assert int(diag["node_k"][q]) == k_ex, (q, tot.sum())
                n_fallback += 1
            else:
                assert g <= g_ex
                n_ranked += 1
    assert n_ranked >= 3 and n_fallback >= 3, (n_ranked, n_fallback)
    # leaves: class frequencies of the samples that reach them
    leaf = np.array([path[np.nonzero(path >= 0)[0].max()] for path in node_of])
    for q in np.unique(leaf)[:40]:
        cnt = np.bincount(lab[leaf == q], minlength=nC).astype(np.float32)
        assert tree.posteriors[q].tobytes() == (cnt / np.float32(cnt.sum())).astype(np.float32).tobytes()


def test_learned_correction_beats_the_estimate(gpu):
    """What the network adds to the stratified refinement, at the proposal
    workload's shape (pool K = 20000 candidates with one threshold, keep
    2000, depth 16, each ranked node of >= 512 samples ranked on a stratified
    subsample of 1/64 of it, at least 256 samples).  Pool runs on other data
    (seeds 1..3) emit refinement records; the network learns the correction
    of the estimated relative gain from the candidates' subsample statistics.
    On seed-0 data, ranking by estimate + correction must lose less gain
    against the whole pool (the exhaustive judge) than the estimate alone,
    which is what the same network with every weight zero ranks by (and then
    the tree is the estimate's own)."""
    nC, K, keep, depth = 8, 20000, 2000, 16
    p = _pool_params(K)
    tr = pa.HIPTreeTrainer(pa.PD_FEAT_DEPTH_U16, nC)
    net = pp.SplitProposalNet(seed=11)
    buf = pp.RecordBuffer(6_000_000)
    tr.set_record_sink(buf, per_node=1000)
    tr.set_proposal_refine(64, 256)
    tr.set_proposal_strata(1)
    tr.set_proposal(net, keep=keep, min_samples=512, judge=False, screen=K)
    for seed in (1, 2, 3):
        ts_r = synth.training_set("c2", seed=seed, n_images=250)
        for tid in range(2):
            tr.train(pa.Tree(tid, depth, pa.PD_FEAT_DEPTH_U16, nC), ts_r, p, 1, depth, mode=pa.PD_MODE_PROPOSAL)
    n = tr.records_written()
    tr.set_record_sink(None, 0)
    assert n > 1_000_000
    loss, _ = net.train_records(buf, batch=4096, epochs=4, opt=pp.adam(lr=1e-3))
    assert loss[-1] < loss[0]
    buf.close()
    trained = net.params
    ts = synth.training_set("c2", seed=0, n_images=250)

    def judged(theta):
        net.params = theta
        tr.set_proposal_strata(2)
        tr.set_proposal(net, keep=keep, min_samples=512, judge=True, screen=K)
        tree = pa.Tree(0, depth, pa.PD_FEAT_DEPTH_U16, nC)
        tr.train(tree, ts, p, 1, depth, mode=pa.PD_MODE_PROPOSAL)
        return _mean_gain_loss(tr.last_level_stats), tree

    loss_learned, _ = judged(trained)
    loss_estimate, zero_tree = judged(np.zeros_like(trained))
    print(f"mean relative gain loss against the whole pool: estimate + correction {loss_learned:.4f}, "
          f"estimate alone {loss_estimate:.4f} ({n} records)")
    assert loss_learned < loss_estimate, (loss_learned, loss_estimate)
    # the zero-weight correction ranks as the estimate alone (mode 1)
    tr.set_proposal_strata(1)
    tr.set_proposal(net, keep=keep, min_samples=512, judge=False, screen=K)
    est_tree = pa.Tree(0, depth, pa.PD_FEAT_DEPTH_U16, nC)
    tr.train(est_tree, ts, p, 1, depth, mode=pa.PD_MODE_PROPOSAL)
    assert np.array_equal(zero_tree.left_children, est_tree.left_children)
    assert zero_tree.thresholds.tobytes() == est_tree.thresholds.tobytes()
    # ... also when the network corrects only each node's best 3000
    net.params = np.zeros_like(trained)
    tr.set_proposal_strata(2)
    tr.set_correction_rows(3000)
    part_tree = pa.Tree(0, depth, pa.PD_FEAT_DEPTH_U16, nC)
    tr.train(part_tree, ts, p, 1, depth, mode=pa.PD_MODE_PROPOSAL)
    tr.set_correction_rows(0)
    assert np.array_equal(part_tree.left_children, est_tree.left_children)
    assert part_tree.thresholds.tobytes() == est_tree.thresholds.tobytes()
    tr.set_proposal_refine(0, 0)
    tr.set_proposal_strata(0)
    tr.close()
    net.close()
