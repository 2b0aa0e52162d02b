"""Performance cases of the random-forest hot path.

What a program built on this package has the GPU do, each through the public
entry points: training a tree (HIPTreeTrainer.train, plain and with the
learned split proposal), predicting frames (HIPClassifier.predict_* on host
images, pd_forest_predict_frames_dev on frames resident in device memory),
the split-proposal network (SplitProposalNet.forward_dev / train_records) and
sampling a data set (the two samplers' device form).

  listed()            the cases
  draw(rng)           one more case of the same ranges
  prepare(case, seed) the data and handles a program holds before the call
  run(state)          one pass; returns every output whole
  work(case)          bytes and operations a pass cannot do without
  exact(case, seed)   the outputs in 64-bit arithmetic by plain torch

A case is a dict of plain values; "op" names the kind of call.
"""
import ctypes
import math

import numpy as np
import torch

import padenti_amd as pa
from padenti_amd import _lib as L
from padenti_amd import dataset, proposal, synth

KINDS = {"depth_f32": pa.PD_FEAT_DEPTH_F32, "depth_u16": pa.PD_FEAT_DEPTH_U16, "rgbd_u16": pa.PD_FEAT_RGBD_U16X4,
         "demo_s16": pa.PD_FEAT_DEMO_S16}
SCENES = {"blobs_f32": L.PD_SYN_BLOBS_F32, "capsules_u16": L.PD_SYN_CAPSULES_U16, "blobs_u16": L.PD_SYN_BLOBS_U16,
          "capsules_rgbd": L.PD_SYN_CAPSULES_RGBD}
DEVICE = "cuda:0"


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _train(kind, scene, images, w, h, classes, samples, features, thresholds, bound, thr, leaf, depth, **more):
    c = dict(op="train", kind=kind, scene=scene, images=images, w=w, h=h, classes=classes, samples=samples,
             features=features, thresholds=thresholds, bound=bound, thr=thr, leaf=leaf, depth=depth)
    c.update(more)
    return c


def listed():
    return [
        # a first tree on a handful of metric depth images: the smallest
        # configuration, all launches and host steps
        dict(name="train_small_f32", **_train("depth_f32", "blobs_f32", 32, 160, 120, 4, 256, 100, 10, 60.0, 0.5, 10,
                                              8)),
        # body-part style training, the mid-size configuration as stated
        # (one million samples): the framework's headline work
        dict(name="train_mid_u16", **_train("depth_u16", "capsules_u16", 500, 320, 240, 8, 2000, 2000, 20, 100000.0,
                                            500.0, 10, 16)),
        # the large configuration's shape (16 classes, 4000 x 32 candidates,
        # VGA frames, depth 20) on a twentieth of its images
        dict(name="train_wide_u16", **_train("depth_u16", "blobs_u16", 250, 640, 480, 16, 2000, 4000, 32, 100000.0,
                                             500.0, 10, 20)),
        # RGB-D frames, 21 classes: the training side of the prediction
        # configuration
        dict(name="train_rgbd", **_train("rgbd_u16", "capsules_rgbd", 60, 320, 240, 21, 2000, 2000, 20, 100000.0,
                                         500.0, 10, 20)),
        # integer responses (the reference's demo feature), odd image sizes
        # and candidate counts
        dict(name="train_odd_s16", **_train("demo_s16", "capsules_u16", 41, 157, 121, 6, 777, 333, 7, 60.0, 200.0, 20,
                                            11)),
        # the learned split proposal: a large single-threshold pool ranked on
        # subsamples with a network's correction, the best kept
        dict(name="train_proposal", **_train("depth_u16", "capsules_u16", 60, 320, 240, 8, 2000, 20000, 1, 100000.0,
                                             500.0, 10, 14, op="propose", keep=2000, stride=64, sub_min=256,
                                             ranked=512)),
        # one camera frame from and to host memory with a mask (an
        # interactive program's call)
        dict(name="predict_frame", op="predict_host", kind="depth_u16", scene="capsules_u16", w=317, h=239, classes=8,
             trees=3, depth=16, masked=True),
        # a batch of mixed frames resident on the GPU, posteriors and leaf
        # ids of five depth-20 trees (an eighth of the batch configuration)
        dict(name="predict_batch", op="predict_dev", kind="rgbd_u16", scene="capsules_rgbd", small=12, vga=16, hd=4,
             classes=21, trees=5, depth=20, leaves=True, graph=False),
        # the network scoring a candidate pool (the proposal's ranking)
        dict(name="net_score", op="score", rows=1 << 20),
        # the network learning from records at the proposal's batch size,
        # the last batch a partial one
        dict(name="net_train", op="fit", rows=30001, batch=4096, epochs=1),
        # drawing training pixels from a resident data set
        dict(name="sample_uniform", op="sample", sampler="uniform", images=400, w=640, h=480, classes=16, samples=2000),
        # the class-balanced reservoir on an odd-sized smaller set
        dict(name="sample_weighted", op="sample", sampler="weighted", images=150, w=321, h=243, classes=16,
             samples=2000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["train", "train", "train", "propose", "predict_host", "predict_dev", "predict_dev", "score",
                     "fit", "fit", "sample"])
    if op in ("train", "propose"):
        kind, scene = rng.choice([("depth_f32", "blobs_f32"), ("depth_u16", "capsules_u16"),
                                  ("depth_u16", "blobs_u16"), ("rgbd_u16", "capsules_rgbd"),
                                  ("demo_s16", "capsules_u16")])
        if op == "propose":
            kind, scene = "depth_u16", rng.choice(["capsules_u16", "blobs_u16"])
        w = rng.randint(100, 640)
        h = rng.randint(80, 480)
        images = _log_int(rng, 8, 250)
        if kind == "rgbd_u16":
            images = min(images, max(8, 4000000 // (w * h)))
        samples = _log_int(rng, 200, 2000)
        classes = rng.choice([2, 4, 6, 8, 13, 16, 21])
        features = _log_int(rng, 50, 4000)
        features = max(50, min(features, 800000000 // (images * samples)))   # below the largest listed case
        thresholds = rng.randint(5, 32)
        bound, thr = {"depth_f32": (60.0, 0.5), "demo_s16": (60.0, 200.0)}.get(kind, (100000.0, 500.0))
        c = _train(kind, scene, images, w, h, classes, samples, features, thresholds, bound, thr, rng.choice([5, 10, 20]),
                   rng.randint(8, 18))
        if op == "propose":
            pool = _log_int(rng, 2000, 20000)
            c.update(op="propose", classes=min(classes, 16), features=pool, thresholds=1, images=min(images, 60),
                     keep=max(100, pool // 10), stride=64, sub_min=256, ranked=512, depth=min(c["depth"], 14))
        return c
    if op == "predict_host":
        kind, scene = rng.choice([("depth_f32", "blobs_f32"), ("depth_u16", "capsules_u16"),
                                  ("rgbd_u16", "capsules_rgbd")])
        return dict(op=op, kind=kind, scene=scene, w=rng.randint(80, 640), h=rng.randint(60, 480),
                    classes=rng.choice([4, 8, 16, 21]), trees=rng.randint(1, 5), depth=rng.randint(8, 18),
                    masked=rng.random() < 0.5)
    if op == "predict_dev":
        kind, scene = rng.choice([("depth_u16", "capsules_u16"), ("rgbd_u16", "capsules_rgbd")])
        return dict(op=op, kind=kind, scene=scene, small=rng.randint(1, 12), vga=rng.randint(0, 12),
                    hd=rng.randint(0, 3), classes=rng.choice([4, 8, 16, 21]), trees=rng.randint(1, 5),
                    depth=rng.randint(8, 20), leaves=rng.random() < 0.5, graph=rng.random() < 0.3)
    if op == "score":
        return dict(op=op, rows=_log_int(rng, 1000, 1 << 20))
    if op == "fit":
        batch = _log_int(rng, 512, 65536)
        return dict(op=op, rows=int(batch * rng.uniform(1.0, 4.0)), batch=batch, epochs=1)
    return dict(op=op, sampler=rng.choice(["uniform", "weighted"]), images=_log_int(rng, 10, 200),
                w=rng.randint(100, 640), h=rng.randint(80, 480), classes=rng.choice([4, 8, 16]),
                samples=_log_int(rng, 200, 2000))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _images(scene, seed, n, w, h, classes, base=0):
    """n (pixels, labels) pairs of a synthetic scene."""
    from concurrent.futures import ThreadPoolExecutor
    with ThreadPoolExecutor(max_workers=8) as ex:
        return list(ex.map(lambda i: synth.gen_image(SCENES[scene], seed, base + i, w, h, classes), range(n)))


def _training_set(c, seed):
    ts = pa.TrainingSet(c["classes"])
    for i, (px, lab) in enumerate(_images(c["scene"], seed, c["images"], c["w"], c["h"], c["classes"])):
        smp = synth.gen_samples(seed, i, lab, c["samples"])
        ts << pa.TrainingSetImage(px, c["w"], c["h"], lab, c["classes"], smp)
    return ts


def _params(c):
    fd = L.FEATURES[KINDS[c["kind"]]][3]
    low, up = [-c["bound"]] * fd, [c["bound"]] * fd
    if fd == 6:   # the two channel parameters of the RGB-D feature
        low[4:], up[4:] = [0.0, 0.0], [4.0, 4.0]
    return pa.TreeTrainerParameters(c["features"], c["thresholds"], low, up, -c["thr"], c["thr"], c["leaf"])


def _probe(img, x, y, px, py, d, ch, bg):
    """I(x + round(px / d), y + round(py / d)), bg outside; img [n, h, w, c] by
    flat pixel row b, every argument a vector.  The quotients are the
    feature's own float32 ones, rounded half away from zero."""
    b, h, w, nch, flat = img
    qx, qy = (px / d.float()).double(), (py / d.float()).double()
    ox = x + (torch.sign(qx) * torch.floor(qx.abs() + 0.5)).clamp(-1e6, 1e6).long()
    oy = y + (torch.sign(qy) * torch.floor(qy.abs() + 0.5)).clamp(-1e6, 1e6).long()
    ok = (ox >= 0) & (ox < w) & (oy >= 0) & (oy < h)
    idx = ((b * h + oy) * w + ox) * nch + ch
    v = flat[torch.where(ok, idx, torch.zeros_like(idx))].double()
    return torch.where(ok, v, torch.full_like(v, bg))


def _response(kind, img, x, y, p):
    """The depth / RGB-D feature of pixels (x, y) with per-pixel parameters p."""
    b, h, w, nch, flat = img
    dch = 3 if nch == 4 else 0
    d = flat[((b * h + y) * w + x) * nch + dch].double()
    ok = d > 0
    ds = torch.where(ok, d, torch.ones_like(d))
    if nch == 4:
        ca, cb = p[:, 4].long().clamp(0, 3), p[:, 5].long().clamp(0, 3)
    else:
        ca = cb = torch.zeros_like(x)
    bg = 10.0 if kind == "depth_f32" else 10000.0
    a = _probe(img, x, y, p[:, 0], p[:, 1], ds, ca, bg)
    r = a - _probe(img, x, y, p[:, 2], p[:, 3], ds, cb, bg)
    if kind == "depth_f32":   # the response of a float feature is a float32
        r = r.float().double()
    return torch.where(ok, r, torch.zeros_like(r))


def _flat(pxs):
    """[n, h, w(, c)] images as (batch index placeholder, h, w, channels, flat device tensor)."""
    a = np.stack(pxs)
    n, h, w = a.shape[:3]
    nch = a.shape[3] if a.ndim == 4 else 1
    t = torch.from_numpy(a.astype(np.float32).reshape(-1)).to(DEVICE)
    return n, h, w, nch, t


def _forest(c, seed):
    """Trees as a trained forest holds them: random features with thresholds
    at a random quantile of the node's own pixels, grown on labelled pixels of
    synthetic scenes until 10 pixels or the last level, leaves holding class
    frequencies.  Returns a list of (left, features, thresholds, posteriors)."""
    fd = L.FEATURES[KINDS[c["kind"]]][3]
    nC, depth = c["classes"], c["depth"]
    pairs = _images(c["scene"], seed, 12, 160, 120, nC, base=500)
    n, h, w, nch, flat = _flat([p[0] for p in pairs])
    lab = torch.from_numpy(np.stack([p[1] for p in pairs]).reshape(-1).astype(np.int64)).to(DEVICE) - 1
    bound = 60.0 if c["kind"] == "depth_f32" else 100000.0
    trees = []
    for t in range(c["trees"]):
        g = torch.Generator().manual_seed(seed * 1000003 + t)
        S = 150000
        pix = torch.randint(n * h * w, (S,), generator=g).to(DEVICE)
        b, y, x = pix // (h * w), (pix // w) % h, pix % w
        img = (b, h, w, nch, flat)
        cls = lab[pix]
        N = (1 << depth) - 1
        left = np.full(N, -2, np.int32)
        feats = np.zeros((N, fd), np.float32)
        thrs = np.zeros(N, np.float32)
        posts = np.zeros((N, nC), np.float32)
        node = torch.zeros(S, dtype=torch.long, device=DEVICE)
        left[0] = -1
        for lv in range(depth):
            n0, cnt = (1 << lv) - 1, 1 << lv
            live = node >= n0
            if not bool(live.any()):
                break
            loc = torch.where(live, node - n0, torch.full_like(node, cnt))
            tab = torch.bincount(loc * nC + cls, minlength=(cnt + 1) * nC)[:cnt * nC].reshape(cnt, nC)
            tot = tab.sum(1)
            have = (tot > 0).nonzero().reshape(-1).cpu().numpy()
            posts[n0 + have] = (tab.double() / tot.clamp(min=1)[:, None]).float().cpu().numpy()[have]
            left[n0 + have] = -1
            if lv == depth - 1:
                break
            # one candidate per node, drawn for the nodes that exist
            u = torch.rand(len(have), 7, generator=g)
            p = torch.zeros(cnt, 6, dtype=torch.float32, device=DEVICE)
            hv = torch.from_numpy(have).to(DEVICE)
            p[hv, :4] = ((u[:, :4] * 2 - 1) * bound).to(DEVICE)
            p[hv, 4:] = (u[:, 4:6] * 4).to(DEVICE)
            quant = torch.full((cnt,), 0.5, device=DEVICE)
            quant[hv] = (0.15 + 0.7 * u[:, 6]).to(DEVICE)
            safe = loc.clamp(max=cnt - 1)
            r = _response(c["kind"], img, x, y, p[safe])
            # threshold: the node's response at its quantile
            order = torch.argsort(r, stable=True)
            order = order[torch.argsort(loc[order], stable=True)]
            start = torch.cumsum(tot, 0) - tot
            at = (start + (quant * tot).long().clamp(min=0)).clamp(max=S - 1)
            thr = r[order[torch.minimum(at, (start + tot - 1).clamp(min=0))]].float()
            go = r <= thr.double()[safe]
            nl = torch.bincount(torch.where(live & go, loc, torch.full_like(loc, cnt)), minlength=cnt + 1)[:cnt]
            split = (tot > 10) & (nl > 0) & (nl < tot)
            sp = split.nonzero().reshape(-1).cpu().numpy()
            left[n0 + sp] = 2 * (n0 + sp) + 1
            feats[n0 + sp] = p[:, :fd].cpu().numpy()[sp]
            thrs[n0 + sp] = thr.cpu().numpy()[sp]
            child = 2 * node + 1 + (~go).long()
            node = torch.where(live & split[safe], child, torch.zeros_like(node) - 1)
        trees.append((left, feats, thrs, posts))
    return trees


def _classifier(c, trees):
    clf = pa.HIPClassifier(KINDS[c["kind"]], c["classes"])
    for i, (left, feats, thrs, posts) in enumerate(trees):
        t = pa.Tree(i, c["depth"], KINDS[c["kind"]], c["classes"])
        t.left_children[:], t.features[:], t.thresholds[:], t.posteriors[:] = left, feats, thrs, posts
        clf << t
    return clf


def _host_frame(c, seed):
    px, _ = synth.gen_image(SCENES[c["scene"]], seed, 9000, c["w"], c["h"], c["classes"])
    mask = None
    if c["masked"]:
        mask = (np.random.default_rng(seed).random((c["h"], c["w"])) < 0.8).astype(np.uint8)
    return px, mask


def _frames(c, seed):
    sizes = [(320, 240)] * c["small"] + [(640, 480)] * c["vga"] + [(1280, 720)] * c["hd"]
    from concurrent.futures import ThreadPoolExecutor
    with ThreadPoolExecutor(max_workers=8) as ex:
        pxs = list(ex.map(lambda iw: synth.gen_image(SCENES[c["scene"]], seed, 9000 + iw[0], iw[1][0], iw[1][1],
                                                     c["classes"])[0], enumerate(sizes)))
    return sizes, pxs


def _records(c, seed):
    """Network rows (BF16 as uint16) and targets with the statistics of real
    records: class frequencies, depth, scaled parameters, subsample
    statistics; targets around zero."""
    rng = np.random.default_rng(seed)
    n = c["rows"]
    x = rng.uniform(-1, 1, size=(n, proposal.IN)).astype(np.float32)
    hist = rng.exponential(1.0, size=(n, 16)).astype(np.float32)
    x[:, :16] = hist / hist.sum(1, keepdims=True)
    x[:, 16] = rng.integers(1, 20, size=n) / 16.0
    x[:, 22:32] = rng.uniform(0, 1, size=(n, 10))
    t = (0.3 * x[:, 17] * x[:, 21] + 0.2 * x[:, 30] - 0.1 + rng.normal(0, 0.05, n)).astype(np.float32)
    return x, t


def _net_params(seed):
    """Parameters of a trained network's size: U(+-1/sqrt(fan in)) weights,
    small biases."""
    rng = np.random.default_rng(seed + 77)
    th = np.zeros(proposal.NPARAM, np.float32)
    for off, n, fan in ((proposal.OFF_W1, 256 * 32, 32), (proposal.OFF_W2, 65536, 256), (proposal.OFF_W3, 65536, 256),
                        (proposal.OFF_W4, 256, 256)):
        th[off:off + n] = rng.uniform(-1, 1, n) / math.sqrt(fan)
    for off in (proposal.OFF_B1, proposal.OFF_B2, proposal.OFF_B3):
        th[off:off + 256] = rng.uniform(-0.05, 0.05, 256)
    return th


# ---------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------
def prepare(case, seed):
    c, op = case, case["op"]
    s = {"case": c}
    if op in ("train", "propose"):
        s["ts"] = _training_set(c, seed)
        s["params"] = _params(c)
        s["trainer"] = pa.HIPTreeTrainer(KINDS[c["kind"]], c["classes"])
        s["trainer"].set_training_set(s["ts"])
        s["mode"] = pa.PD_MODE_LEVEL_BATCHED
        if op == "propose":
            net = proposal.SplitProposalNet(seed=1)
            th = _net_params(seed)
            th[proposal.OFF_W4:proposal.OFF_W4 + 256] *= 0.1   # corrections of a few hundredths
            net.params = th
            s["net"] = net
            s["trainer"].set_proposal_refine(c["stride"], c["sub_min"])
            s["trainer"].set_proposal_strata(2)
            s["trainer"].set_proposal(net, keep=c["keep"], min_samples=c["ranked"], screen=c["features"])
            s["mode"] = pa.PD_MODE_PROPOSAL
    elif op == "predict_host":
        s["clf"] = _classifier(c, _forest(c, seed))
        s["image"], s["mask"] = _host_frame(c, seed)
    elif op == "predict_dev":
        s["clf"] = _classifier(c, _forest(c, seed))
        sizes, pxs = _frames(c, seed)
        host = np.concatenate([p.reshape(-1) for p in pxs])
        s["pix"] = torch.from_numpy(host.view(np.int16)).to(DEVICE)
        npx = np.array([w * h for w, h in sizes], np.uint64)
        before = np.concatenate([[0], np.cumsum(npx)[:-1]]).astype(np.uint64)
        nch = 4 if c["kind"] == "rgbd_u16" else 1
        s["img_off"], s["post_off"] = before * np.uint64(nch), before * np.uint64(c["classes"])
        s["leaf_off"] = before * np.uint64(c["trees"])
        s["w"] = np.array([z[0] for z in sizes], np.uint32)
        s["h"] = np.array([z[1] for z in sizes], np.uint32)
        total = int(npx.sum())
        s["post"] = torch.empty(total * c["classes"], dtype=torch.float32, device=DEVICE)
        s["leaf"] = torch.empty(total * c["trees"], dtype=torch.int32, device=DEVICE) if c["leaves"] else None
    elif op == "score":
        net = proposal.SplitProposalNet(seed=1)
        net.params = _net_params(seed)
        x, _ = _records(c, seed)
        s["net"] = net
        s["x"] = torch.from_numpy(proposal.encode_rows(x).view(np.int16)).to(DEVICE)
        s["y"] = torch.empty(c["rows"], dtype=torch.float32, device=DEVICE)
    elif op == "fit":
        x, t = _records(c, seed)
        buf = proposal.RecordBuffer(c["rows"])
        buf.upload(proposal.encode_rows(x), t)
        s["buf"], s["net"], s["theta"] = buf, proposal.SplitProposalNet(seed=1), _net_params(seed)
    elif op == "sample":
        n, px = c["images"], c["w"] * c["h"]
        pairs = _images("blobs_u16", seed, n, c["w"], c["h"], c["classes"])
        lab_stride = (px + 15) // 16 * 16   # label images start at 16-byte boundaries
        labs = np.zeros((n, lab_stride), np.uint8)
        labs[:, :px] = np.stack([p[1].reshape(-1) for p in pairs])
        s["data"] = torch.from_numpy(np.stack([p[0] for p in pairs]).reshape(-1).view(np.int16)).to(DEVICE)
        s["labels"] = torch.from_numpy(labs.reshape(-1)).to(DEVICE)
        s["doff"] = np.arange(n, dtype=np.uint64) * np.uint64(px * 2)
        s["dbytes"] = np.full(n, px * 2, np.uint64)
        s["loff"] = np.arange(n, dtype=np.uint64) * np.uint64(lab_stride)
        s["w"], s["h"] = np.full(n, c["w"], np.uint32), np.full(n, c["h"], np.uint32)
        if c["sampler"] == "uniform":
            s["sampler"] = dataset.UniformImageSampler(c["samples"], seed=seed + 7)
        else:
            s["sampler"] = dataset.ClassWeightedImageSampler(c["samples"], c["classes"], seed=seed + 7)
        cap = s["sampler"].capacity()
        s["samples"] = torch.zeros(n * cap, dtype=torch.int32, device=DEVICE)
        s["n_out"] = torch.zeros(n, dtype=torch.int32, device=DEVICE)
        s["crc"] = torch.zeros(n, dtype=torch.int32, device=DEVICE)
    else:
        raise ValueError(op)
    torch.cuda.synchronize()
    return s


def _ptr(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def run(state):
    s, c = state, state["case"]
    op = c["op"]
    if op in ("train", "propose"):
        tree = pa.Tree(0, c["depth"], KINDS[c["kind"]], c["classes"])
        s["trainer"].train(tree, s["ts"], s["params"], 1, c["depth"], mode=s["mode"])
        return {"left": tree.left_children, "features": tree.features, "thresholds": tree.thresholds,
                "posteriors": tree.posteriors}
    if op == "predict_host":
        post = s["clf"].predict_posterior(s["image"], c["w"], c["h"], s["mask"])
        leaves = s["clf"].predict_leaves(0, s["image"], c["w"], c["h"], s["mask"])
        return {"posterior": post, "leaves": leaves}
    if op == "predict_dev":
        leaf = s["leaf"]
        L.check(L.lib().pd_forest_predict_frames_dev(
            s["clf"]._h, len(s["w"]), _ptr(s["pix"]), s["pix"].numel() * 2, L.ptr(s["img_off"]), L.ptr(s["w"]),
            L.ptr(s["h"]), None, 0, None, _ptr(s["post"]), s["post"].numel() * 4, L.ptr(s["post_off"]), _ptr(leaf),
            leaf.numel() * 4 if leaf is not None else 0, L.ptr(s["leaf_off"]), 1 if c["graph"] else 0, None))
        out = {"posterior": s["post"]}
        if leaf is not None:
            out["leaves"] = leaf
        return out
    if op == "score":
        s["net"].forward_dev(_ptr(s["x"]), c["rows"], _ptr(s["y"]))
        return {"score": s["y"]}
    if op == "fit":
        s["net"].params = s["theta"]   # every pass trains the same network
        loss, _ = s["net"].train_records(s["buf"], n=c["rows"], batch=c["batch"], epochs=c["epochs"], target="gain",
                                         seed=3)
        return {"params": s["net"].params, "loss": loss}
    s["sampler"].sample_dev(c["images"], _ptr(s["data"]), s["data"].numel() * 2, s["doff"], s["dbytes"],
                            _ptr(s["labels"]), s["labels"].numel(), s["loff"], s["w"], s["h"], _ptr(s["samples"]),
                            _ptr(s["n_out"]), _ptr(s["crc"]))
    return {"samples": s["samples"], "n_out": s["n_out"], "crc": s["crc"]}


# ---------------------------------------------------------------------------
# work
# ---------------------------------------------------------------------------
MLP_FLOP = 2 * (32 * 256 + 2 * 256 * 256 + 256)   # forward, per row


def work(case):
    c, op = case, case["op"]
    if op in ("train", "propose"):
        info = L.FEATURES[KINDS[c["kind"]]]
        px_bytes = np.dtype(info[0]).itemsize * info[1]
        S = c["images"] * c["samples"]
        nodes = (1 << c["depth"]) - 1
        tree = nodes * (4 + np.dtype(info[2]).itemsize * (info[3] + 1) + 4 * c["classes"])
        nodes = min(nodes, 2 * S)
        tree = min(tree, nodes * (4 + np.dtype(info[2]).itemsize * (info[3] + 1) + 4 * c["classes"]))
        # the levels a balanced tree of these samples has
        levels = min(c["depth"] - 1, max(1, int(math.log2(max(2, S / (c["leaf"] + 1)))) + 1))
        # per (sample, candidate) and level: two probes of two quotients, two
        # roundings and two border tests each, the difference, a search
        # among the thresholds and a count
        per = 2 * 6 + 1 + math.ceil(math.log2(c["thresholds"] + 1)) + 1
        cand = c["features"] if op == "train" else c["features"] / c["stride"] + c["keep"]
        return {"bytes": c["images"] * c["w"] * c["h"] * px_bytes + S * 5 + tree, "flops": S * levels * cand * per}
    if op in ("predict_host", "predict_dev"):
        info = L.FEATURES[KINDS[c["kind"]]]
        px_bytes = np.dtype(info[0]).itemsize * info[1]
        if op == "predict_host":
            px, leaves = c["w"] * c["h"], 1
        else:
            px, leaves = c["small"] * 76800 + c["vga"] * 307200 + c["hd"] * 921600, c["trees"] if c["leaves"] else 0
        steps = min(c["depth"] - 1, 14)
        return {"bytes": px * (px_bytes + 4 * c["classes"] + 4 * leaves),
                "flops": px * c["trees"] * (steps * 14 + c["classes"])}
    if op == "score":
        return {"bytes": c["rows"] * (64 + 4), "flops": c["rows"] * MLP_FLOP}
    if op == "fit":
        return {"bytes": c["rows"] * c["epochs"] * 68 + proposal.NPARAM * 4 * 6,
                "flops": c["rows"] * c["epochs"] * 3 * MLP_FLOP}
    px = c["images"] * c["w"] * c["h"]
    return {"bytes": px * 3 + c["images"] * c["samples"] * 4, "flops": px * 4}


# ---------------------------------------------------------------------------
# the outputs in 64-bit arithmetic
# ---------------------------------------------------------------------------
def _traverse(c, trees, pxs):
    """(posteriors [nC][pixels], leaf ids [tree][pixels]) of one frame."""
    n, h, w, nch, flat = _flat([pxs])
    y, x = torch.meshgrid(torch.arange(h, device=DEVICE), torch.arange(w, device=DEVICE), indexing="ij")
    y, x = y.reshape(-1), x.reshape(-1)
    img = (torch.zeros_like(x), h, w, nch, flat)
    post, ids = 0, []
    for left, feats, thrs, posts in trees:
        node = torch.zeros_like(x)
        for _ in range(c["depth"] - 1):
            lc = left[node]
            go = lc >= 0
            if not bool(go.any()):
                break
            r = _response(c["kind"], img, x, y, feats[node])
            node = torch.where(go, lc + (~(r <= thrs[node].double())).long(), node)
        ids.append(node)
        post = post + posts[node].double()
    return (post / len(trees)).T.contiguous(), torch.stack(ids)


def _dev_trees(trees):
    return [(torch.from_numpy(a).to(DEVICE).long(), torch.from_numpy(b).to(DEVICE), torch.from_numpy(t).to(DEVICE),
             torch.from_numpy(p).to(DEVICE)) for a, b, t, p in trees]


def _layers(th):
    p = proposal
    return [(th[p.OFF_W1:p.OFF_B1].reshape(256, 32), th[p.OFF_B1:p.OFF_W2]),
            (th[p.OFF_W2:p.OFF_B2].reshape(256, 256), th[p.OFF_B2:p.OFF_W3]),
            (th[p.OFF_W3:p.OFF_B3].reshape(256, 256), th[p.OFF_B3:p.OFF_W4]),
            (th[p.OFF_W4:p.OFF_B4].reshape(1, 256), th[p.OFF_B4:])]


def _net(th, x):
    for i, (w, b) in enumerate(_layers(th)):
        x = torch.addmm(b, x, w.T)
        if i < 3:
            x = torch.nn.functional.gelu(x, approximate="tanh")
    return x[:, 0]


def _bf16_rows(x):
    return torch.from_numpy(x).to(DEVICE).to(torch.bfloat16).double()


def _permutation(n, seed, epoch):
    """The documented batch order: Fisher-Yates of SplitMix64(seed, epoch)."""
    m = (1 << 64) - 1
    s = (seed * 0x9e3779b97f4a7c15 + epoch + 1) & m
    p = list(range(n))
    for i in range(n - 1, 0, -1):
        s = (s + 0x9e3779b97f4a7c15) & m
        z = ((s ^ (s >> 30)) * 0xbf58476d1ce4e5b9) & m
        z = ((z ^ (z >> 27)) * 0x94d049bb133111eb) & m
        j = (z ^ (z >> 31)) % (i + 1)
        p[i], p[j] = p[j], p[i]
    return torch.tensor(p, device=DEVICE)


def _fit(c, seed):
    x, t = _records(c, seed)
    x, t = _bf16_rows(x), torch.from_numpy(t).to(DEVICE).double()
    th = torch.from_numpy(_net_params(seed)).to(DEVICE).double()
    m, v, step = torch.zeros_like(th), torch.zeros_like(th), 0
    losses = []
    for ep in range(c["epochs"]):
        order = _permutation(c["rows"], 3, ep)
        acc = 0.0
        for at in range(0, c["rows"], c["batch"]):
            i = order[at:at + c["batch"]]
            p = th.clone().requires_grad_(True)
            loss = ((_net(p, x[i]) - t[i]) ** 2).mean()
            g, = torch.autograd.grad(loss, p)
            step += 1
            m = 0.9 * m + 0.1 * g
            v = 0.999 * v + 0.001 * g * g
            th = th - 1e-3 * (m / (1 - 0.9 ** step)) / (torch.sqrt(v / (1 - 0.999 ** step)) + 1e-8)
            acc += float(loss.detach()) * len(i)
        losses.append(acc / c["rows"])
    return {"params": th.cpu().numpy(), "loss": np.array(losses)}


def exact(case, seed):
    c, op = case, case["op"]
    if op in ("train", "propose", "sample"):
        # a tree is the first maximum of float32 gains node after node, a
        # sample list a stream of random draws: neither has a 64-bit value
        return None
    if op == "predict_host":
        px, mask = _host_frame(c, seed)
        post, _ = _traverse(c, _dev_trees(_forest(c, seed)), px)
        if mask is not None:
            post = post * torch.from_numpy(mask.reshape(-1).astype(np.float64)).to(DEVICE)
        return {"posterior": post.reshape(c["classes"], c["h"], c["w"]).cpu().numpy(), "leaves": None}
    if op == "predict_dev":
        trees = _dev_trees(_forest(c, seed))
        _, pxs = _frames(c, seed)
        post = torch.cat([_traverse(c, trees, p)[0].reshape(-1) for p in pxs])
        out = {"posterior": post}
        if c["leaves"]:
            out["leaves"] = None
        return out
    if op == "score":
        x, _ = _records(c, seed)
        th = torch.from_numpy(_net_params(seed)).to(DEVICE).double()
        x = _bf16_rows(x)
        return {"score": torch.cat([_net(th, x[i:i + 131072]) for i in range(0, len(x), 131072)])}
    return _fit(c, seed)
