"""Performance cases of the engine: what a user of this package has it do.

Twelve listed cases cover the public entry points over their real range: the
no-allocation scoring call, one image pair per call with the API's default
options, batches of pairs (uniform and ragged, host rows and rows resident in
HBM), the learned-guidance batch, and inference and training of its network.
``draw`` spreads more cases over the same ranges.

Scenes are made on the GPU from the seed alone (the generators of
``pygcransac.synthetic``, for a whole batch at once).  Every run's sampler
seeds are fixed by the case's seed, so a pass is reproducible.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "graph-cut-ransac_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import pygcransac  # noqa: E402
from pygcransac import _native, guided  # noqa: E402

KINDS = {"homography": 0, "fundamental": 1, "essential": 2}
SAMPLE = {"homography": 4, "fundamental": 7, "essential": 5}
IMAGE = {"homography": (640, 480), "fundamental": (640, 480), "essential": (1024, 768)}
FOCAL = {"homography": 800.0, "fundamental": 800.0, "essential": 1000.0}
NOISE = {"homography": 0.5, "fundamental": 0.5, "essential": 0.75}
THRESHOLD = {"homography": 3.0, "fundamental": 1.0, "essential": 0.75}


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # Scoring a handful of hypotheses from a serving loop that owns its
        # device buffers, masks included: launch latency.
        {"name": "score_small", "path": "score", "kind": "homography", "n": 1000, "models": 64, "masks": True},
        # Scoring a full chunk of fundamental-matrix hypotheses (the call's
        # largest model count) on the benchmark's 5,000 points: FP64 throughput.
        {"name": "score_large", "path": "score", "kind": "fundamental", "n": 5000, "models": 65536, "masks": False},
        # One image pair per call with the API's default options (PROSAC rows,
        # SPRT, space partitioning on the grid): an interactive caller.
        {"name": "h_single", "path": "single", "kind": "homography", "n": 2000, "inliers": 0.5, "defaults": True,
         "max_iters": 10000},
        # The same for a fundamental matrix (PROSAC, SPRT, radius graph).
        {"name": "f_single", "path": "single", "kind": "fundamental", "n": 3001, "inliers": 0.5, "defaults": True,
         "max_iters": 10000},
        # One essential matrix with the settings of the benchmark (uniform
        # sampler, grid, every model scored in full).
        {"name": "e_single", "path": "single", "kind": "essential", "n": 1500, "inliers": 0.4, "defaults": False,
         "max_iters": 10000},
        # A photo collection's homographies in one call, host rows through the
        # Python API (benchmark configuration: 2,000 points at 50 %).
        {"name": "h_batch", "path": "batch", "kind": "homography", "pairs": 1024, "n": 2000, "n_low": 2000,
         "inliers": 0.5, "max_iters": 1000000, "resident": False},
        # The benchmark's fundamental batch (5,000 points at 30 %), rows
        # resident in HBM, through the C interface.
        {"name": "f_batch", "path": "batch", "kind": "fundamental", "pairs": 1024, "n": 5000, "n_low": 5000,
         "inliers": 0.3, "max_iters": 1000000, "resident": True},
        # A ragged batch as feature matching gives it: half homographies, half
        # fundamental matrices, 200 to 4,000 points, odd sizes throughout.
        {"name": "mixed_batch", "path": "batch", "kind": "mixed", "pairs": 333, "n": 4000, "n_low": 200,
         "inliers": 0.5, "max_iters": 10000, "resident": False},
        # The benchmark's essential batch (10,000 points at 10 %): the
        # five-point solver over millions of samples.
        {"name": "e_batch", "path": "batch", "kind": "essential", "pairs": 32, "n": 10000, "n_low": 10000,
         "inliers": 0.1, "max_iters": 1000000, "resident": True},
        # The headline: learned guidance over 1,024 pairs of 4,000 points at
        # 5 % inliers, inputs resident in HBM.
        {"name": "guided_batch", "path": "guided", "pairs": 1024, "n": 4000, "inliers": 0.05, "max_iters": 10000},
        # The network alone over the rows of 128 pairs, host arrays in and out.
        {"name": "predict", "path": "predict", "n": 500003},
        # Training the network: steps of the training recipe (8,192 rows).
        {"name": "train", "path": "train", "n": 200000, "batch": 8192, "steps": 20},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["score", "score", "single", "single", "single", "batch", "batch", "batch", "guided",
                       "predict", "train"])
    if path == "score":
        n, k = _log(rng, 100, 20000), _log(rng, 16, 65536)
        return {"path": path, "kind": rng.choice(["homography", "fundamental"]), "n": n, "models": k,
                "masks": n * k < 20000000 and rng.random() < 0.5}
    if path == "single":
        kind = rng.choice(["homography", "fundamental", "essential"])
        return {"path": path, "kind": kind, "n": _log(rng, 150, 8000), "inliers": round(rng.uniform(0.35, 0.8), 3),
                "defaults": rng.random() < 0.5, "max_iters": 10000}
    if path == "batch":
        kind = rng.choice(["homography", "fundamental", "mixed", "essential"])
        if kind == "essential":
            pairs, n = _log(rng, 4, 48), _log(rng, 300, 6000)
            return {"path": path, "kind": kind, "pairs": pairs, "n": n, "n_low": n,
                    "inliers": round(rng.uniform(0.15, 0.6), 3), "max_iters": 100000,
                    "resident": rng.random() < 0.5}
        pairs, n = _log(rng, 8, 700), _log(rng, 300, 5000)
        return {"path": path, "kind": kind, "pairs": pairs, "n": n,
                "n_low": n if rng.random() < 0.5 else max(100, n // 8), "inliers": round(rng.uniform(0.35, 0.8), 3),
                "max_iters": 100000, "resident": rng.random() < 0.5}
    if path == "guided":
        return {"path": path, "pairs": _log(rng, 8, 700), "n": _log(rng, 300, 5000),
                "inliers": round(rng.uniform(0.05, 0.5), 3), "max_iters": 10000}
    if path == "predict":
        return {"path": path, "n": _log(rng, 500, 1500000)}
    return {"path": path, "n": _log(rng, 2000, 400000), "batch": _log(rng, 256, 16384), "steps": rng.randint(3, 30)}


# ---------------------------------------------------------------------------
# Scenes, a whole batch at once on the GPU
# ---------------------------------------------------------------------------

def _rotations(axis, angle):
    axis = axis / axis.norm(dim=1, keepdim=True)
    z = torch.zeros_like(angle)
    K = torch.stack([z, -axis[:, 2], axis[:, 1], axis[:, 2], z, -axis[:, 0], -axis[:, 1], axis[:, 0], z], 1)
    K = K.reshape(-1, 3, 3)
    eye = torch.eye(3, dtype=angle.dtype, device=angle.device)
    return eye + torch.sin(angle)[:, None, None] * K + (1 - torch.cos(angle))[:, None, None] * (K @ K)


class _Scenes:
    """Correspondences of many pairs, back to back: ``corr`` (rows x 4,
    float64, on the GPU), ``ratio`` (descriptor ratio per row), ``offsets``
    and per pair its kind and true model (x2^T F x1 = 0 or x2 ~ H x1, pixel
    coordinates)."""

    def __init__(self, kinds, counts, inliers, seed, sort_rows):
        self.kinds = kinds
        g = torch.Generator(device="cuda")
        g.manual_seed(seed)
        self.g = g
        dev = torch.device("cuda")
        B = len(kinds)
        n = np.asarray(counts, np.int64)
        n_in = np.round(n * inliers).astype(np.int64)
        self.offsets = np.concatenate([[0], np.cumsum(n)])
        kind = torch.tensor([KINDS[k] for k in kinds], device=dev)
        w = torch.tensor([float(IMAGE[k][0]) for k in kinds], dtype=torch.float64, device=dev)
        h = torch.tensor([float(IMAGE[k][1]) for k in kinds], dtype=torch.float64, device=dev)
        f = torch.tensor([FOCAL[k] for k in kinds], dtype=torch.float64, device=dev)
        noise = torch.tensor([NOISE[k] for k in kinds], dtype=torch.float64, device=dev)
        uni = self._uni
        # homographies: rotation +-30 deg, scale 0.7..1.4, perspective ~1e-4, translation +-40 px
        th, s = (uni(B) * 60 - 30) * (math.pi / 180), 0.7 + 0.7 * uni(B)
        p, tr = self._normal(B, 2) * 1e-4, uni(B, 2) * 80 - 40
        one, zero = torch.ones_like(s), torch.zeros_like(s)
        A = torch.stack([s * torch.cos(th), -s * torch.sin(th), tr[:, 0], s * torch.sin(th), s * torch.cos(th),
                         tr[:, 1], p[:, 0], p[:, 1], one], 1).reshape(B, 3, 3)
        Tc = torch.stack([one, zero, w / 2, zero, one, h / 2, zero, zero, one], 1).reshape(B, 3, 3)
        Ti = torch.stack([one, zero, -w / 2, zero, one, -h / 2, zero, zero, one], 1).reshape(B, 3, 3)
        H = Tc @ A @ Ti
        # two views: rotation up to 20 deg, baseline 0.5..2 m, depth 2..20 m
        R = _rotations(self._normal(B, 3), uni(B) * (20 * math.pi / 180))
        t = self._normal(B, 3)
        t = t / t.norm(dim=1, keepdim=True) * (0.5 + 1.5 * uni(B))[:, None]
        tx = torch.stack([zero, -t[:, 2], t[:, 1], t[:, 2], zero, -t[:, 0], -t[:, 1], t[:, 0], zero], 1)
        Ki = torch.stack([1 / f, zero, -w / 2 / f, zero, 1 / f, -h / 2 / f, zero, zero, one], 1).reshape(B, 3, 3)
        F = Ki.transpose(1, 2).contiguous() @ (tx.reshape(B, 3, 3) @ R) @ Ki
        F = F / F.flatten(1).norm(dim=1)[:, None, None]
        self.models = torch.where((kind == 0)[:, None, None], H, F)
        # rows: the inliers (redrawn until both views see them), then the outliers
        pid_in = torch.repeat_interleave(torch.arange(B, device=dev), torch.tensor(n_in, device=dev))
        rows_in = torch.empty((len(pid_in), 4), dtype=torch.float64, device=dev)
        todo = torch.arange(len(pid_in), device=dev)
        for _ in range(2000):
            if not len(todo):
                break
            q = pid_in[todo]
            m = len(q)
            u1 = uni(m, 2) * torch.stack([w[q], h[q]], 1)
            z = 2.0 + 18.0 * uni(m)
            c = torch.stack([w[q], h[q]], 1) / 2
            X = torch.cat([(u1 - c) / f[q, None] * z[:, None], z[:, None]], 1)
            X2 = (R[q] * X[:, None, :]).sum(2) + t[q]
            u2 = X2[:, :2] / X2[:, 2:3] * f[q, None] + c
            hx = (H[q] * torch.cat([u1, torch.ones_like(z)[:, None]], 1)[:, None, :]).sum(2)
            is_h = (kind[q] == 0)[:, None]
            ok = torch.where(is_h[:, 0], hx[:, 2] > 0, X2[:, 2] > 0.1)
            u2 = torch.where(is_h, hx[:, :2] / hx[:, 2:3], u2) + self._normal(m, 2) * noise[q, None]
            v1 = torch.where(is_h, u1, u1 + self._normal(m, 2) * noise[q, None])
            for v in (v1, u2):
                ok &= (v[:, 0] >= 0) & (v[:, 0] < w[q]) & (v[:, 1] >= 0) & (v[:, 1] < h[q])
            rows_in[todo[ok]] = torch.cat([v1, u2], 1)[ok]
            todo = todo[~ok]
        else:
            raise RuntimeError("a scene without overlap between its views")
        pid_out = torch.repeat_interleave(torch.arange(B, device=dev), torch.tensor(n - n_in, device=dev))
        wh = torch.stack([w[pid_out], h[pid_out]], 1)
        rows_out = torch.cat([uni(len(pid_out), 2) * wh, uni(len(pid_out), 2) * wh], 1)
        rows, pid = torch.cat([rows_in, rows_out]), torch.cat([pid_in, pid_out])
        # descriptor ratio: Beta(2, 5) for inliers, Beta(5, 2) for outliers
        # (the second and the fifth of six uniform draws in order)
        six = self._uni(len(pid), 6).sort(dim=1).values
        ratio = torch.cat([six[:len(pid_in), 1], six[len(pid_in):, 4]])
        # rows in random order, or by rising ratio (what a PROSAC caller passes)
        key = pid.double() + (ratio if sort_rows else uni(len(pid)))
        order = key.argsort()
        self.corr, self.ratio = rows[order].contiguous(), ratio[order].contiguous()

    def _uni(self, *shape):
        return torch.rand(shape, dtype=torch.float64, device="cuda", generator=self.g)

    def _normal(self, *shape):
        return torch.randn(shape, dtype=torch.float64, device="cuda", generator=self.g)


def _intrinsics(kind):
    (w, h), f = IMAGE[kind], FOCAL[kind]
    return np.array([[f, 0, w / 2], [0, f, h / 2], [0, 0, 1.0]])


def _batch_kinds_counts(case, seed):
    """Kinds and correspondence counts of a batch; the counts of a ragged one
    are log-uniform between n_low and n and the same for every seed."""
    B = case["pairs"]
    kinds = [("homography", "fundamental")[i % 2] for i in range(B)] if case["kind"] == "mixed" else [case["kind"]] * B
    lo, hi = case["n_low"], case["n"]
    if lo == hi:
        return kinds, [hi] * B
    r = np.random.default_rng(1234)
    return kinds, [int(v) for v in np.floor(np.exp(r.uniform(math.log(lo), math.log(hi + 1), B)))]


def _options(kind, case, seed):
    return dict(threshold=THRESHOLD[kind], conf=0.99, spatial_coherence_weight=0.975, max_iters=case["max_iters"],
                min_iters=50, use_sprt=False, sampler=0, neighborhood=0, neighborhood_size=8.0, lo_number=50,
                seed=seed)


# ---------------------------------------------------------------------------
# prepare: what the program holds before the call
# ---------------------------------------------------------------------------

def prepare(case, seed):
    state = {"score": _prepare_score, "single": _prepare_single, "batch": _prepare_batch,
             "guided": _prepare_guided, "predict": _prepare_predict, "train": _prepare_train}[case["path"]](case, seed)
    state["case"] = case
    torch.cuda.synchronize()
    return state


def _prepare_score(case, seed):
    """Points of one scene; models as a run scores them: a third near the true
    model, the others wrong."""
    sc = _Scenes([case["kind"]], [case["n"]], 0.4, seed, False)
    k = case["models"]
    m = sc.models[0].reshape(1, 9).repeat(k, 1)
    spread = 10.0 ** (-6.0 + 5.5 * sc._uni(k, 1))
    spread[::3] = 10.0 ** (-7.0 + 2.5 * sc._uni(len(spread[::3]), 1))
    m = m * (1.0 + spread * sc._normal(k, 9))
    masks = torch.empty((k, case["n"]), dtype=torch.uint8, device="cuda") if case["masks"] else None
    return {"pts": sc.corr, "models": m.contiguous(), "masks": masks,
            "counts": torch.empty(k, dtype=torch.int64, device="cuda"),
            "values": torch.empty(k, dtype=torch.float64, device="cuda"),
            "sq_thr": (1.5 * THRESHOLD[case["kind"]]) ** 2}


def _prepare_single(case, seed):
    kind = case["kind"]
    sc = _Scenes([kind], [case["n"]], case["inliers"], seed, case["defaults"])
    w, h = IMAGE[kind]
    args = [h, w, h, w, None]
    opts = {"seed": seed, "threshold": THRESHOLD[kind], "max_iters": case["max_iters"]} if case["defaults"] else \
        _options(kind, case, seed)
    if kind == "essential":
        args = [_intrinsics(kind), _intrinsics(kind)] + args
    elif kind == "homography" and not case["defaults"]:
        opts["use_space_partitioning"] = False
    return {"args": [sc.corr.cpu().numpy()] + args, "opts": opts}


def _prepare_batch(case, seed):
    kinds, counts = _batch_kinds_counts(case, seed)
    sc = _Scenes(kinds, counts, case["inliers"], seed, False)
    problems = []
    for i, kind in enumerate(kinds):
        w, h = IMAGE[kind]
        p = dict(_options(kind, case, (seed * 1000003 + i) & 0x7FFFFFFF), kind=kind, h1=h, w1=w, h2=h, w2=w)
        if kind == "essential":
            p.update(K1=_intrinsics(kind), K2=_intrinsics(kind))
        problems.append(p)
    if not case["resident"]:
        rows = sc.corr.cpu().numpy()
        for i, p in enumerate(problems):
            p["correspondences"] = rows[sc.offsets[i]:sc.offsets[i + 1]]
        return {"problems": problems}
    return _c_batch(problems, sc)


def _c_batch(problems, sc):
    """Arguments of the C batch entry points, rows resident in HBM."""
    B = len(problems)
    kinds, Ks, params = guided._batch_params(problems)
    sizes = np.array([[p["h1"], p["w1"], p["h2"], p["w2"]] for p in problems], np.int32).ravel()
    return {"kinds": kinds, "K": Ks if (kinds == 2).any() else None, "params": params, "sizes": sizes,
            "offsets": np.ascontiguousarray(sc.offsets, np.int64), "corr": sc.corr, "ratio": sc.ratio,
            "models": np.zeros((B, 9)), "masks": np.zeros(int(sc.offsets[-1]), np.uint8),
            "inliers": np.zeros(B, np.int32), "stats": (_native.GcrStats * B)()}


def _prepare_guided(case, seed):
    kinds, counts = ["fundamental"] * case["pairs"], [case["n"]] * case["pairs"]
    sc = _Scenes(kinds, counts, case["inliers"], seed, False)
    w, h = IMAGE["fundamental"]
    problems = [dict(_options("fundamental", case, (seed * 1000003 + i) & 0x7FFFFFFF), kind="fundamental", h1=h, w1=w,
                     h2=h, w2=w) for i in range(case["pairs"])]
    state = _c_batch(problems, sc)
    state["net"] = guided.load()
    return state


def _rows(n, seed):
    """Feature rows and labels with the distributions that the feature kernels
    give on two-view scenes: coordinates in [-1, 1], the descriptor ratio, the
    displacement against the neighbours'."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    label = (torch.rand(n, device="cuda", generator=g) < 0.3).float()
    six = torch.rand((n, 6), device="cuda", generator=g).sort(dim=1).values
    feat = torch.zeros((n, 8), device="cuda")
    feat[:, :4] = torch.rand((n, 4), device="cuda", generator=g) * 2 - 1
    feat[:, 4] = torch.where(label > 0, six[:, 1], six[:, 4])
    spread = torch.where(label > 0, 0.35, 0.9)[:, None]
    feat[:, 5:7] = torch.randn((n, 2), device="cuda", generator=g) * spread
    return feat.cpu().numpy(), label.cpu().numpy()


def _prepare_predict(case, seed):
    return {"net": guided.load(), "feat": _rows(case["n"], seed)[0]}


def _prepare_train(case, seed):
    feat, label = _rows(case["n"], seed)
    return {"net": guided.init_params(seed), "feat": feat, "labels": label, "seed": seed}


# ---------------------------------------------------------------------------
# run: one pass through the public entry points
# ---------------------------------------------------------------------------

def run(state):
    return {"score": _run_score, "single": _run_single, "batch": _run_batch, "guided": _run_guided,
            "predict": _run_predict, "train": _run_train}[state["case"]["path"]](state)


def _run_score(s):
    pts, m, masks = s["pts"], s["models"], s["masks"]
    rc = _native.lib().gcr_score_models_noalloc(
        KINDS[s["case"]["kind"]], pts.data_ptr(), len(pts), m.data_ptr(), len(m), s["sq_thr"], s["counts"].data_ptr(),
        s["values"].data_ptr(), None if masks is None else masks.data_ptr(), torch.cuda.current_stream().cuda_stream)
    _native.raise_for(rc)
    out = {"counts": s["counts"], "values": s["values"]}
    if masks is not None:
        out["masks"] = masks
    return out


def _run_single(s):
    find = {"homography": pygcransac.findHomography, "fundamental": pygcransac.findFundamentalMatrix,
            "essential": pygcransac.findEssentialMatrix}[s["case"]["kind"]]
    model, mask = find(*s["args"], **s["opts"])
    return {"model": np.zeros((3, 3)) if model is None else model, "mask": mask,
            "iterations": pygcransac.last_stats()["iteration_number"]}


def _run_batch(s):
    if "problems" in s:
        res = pygcransac.findBatch(s["problems"])
        return {"models": np.stack([np.zeros((3, 3)) if m is None else m for m, _ in res]),
                "masks": np.concatenate([k for _, k in res])}
    vp = lambda a: None if a is None else a.ctypes.data_as(ctypes.c_void_p)  # noqa: E731
    rc = _native.lib().gcr_find_batch(len(s["kinds"]), vp(s["kinds"]), vp(s["offsets"]), s["corr"].data_ptr(), 1,
                                      vp(s["sizes"]), vp(s["K"]), s["params"], vp(s["models"]), vp(s["masks"]),
                                      vp(s["inliers"]), s["stats"])
    _native.raise_for(rc)
    return {"models": s["models"], "masks": s["masks"], "inliers": s["inliers"]}


def _run_guided(s):
    vp = lambda a: None if a is None else a.ctypes.data_as(ctypes.c_void_p)  # noqa: E731
    rc = _native.lib().gcr_find_batch_guided(len(s["kinds"]), vp(s["kinds"]), vp(s["offsets"]), s["corr"].data_ptr(),
                                             1, vp(s["sizes"]), vp(s["K"]), s["ratio"].data_ptr(), vp(s["net"]),
                                             s["params"], vp(s["models"]), vp(s["masks"]), vp(s["inliers"]),
                                             s["stats"], None)
    _native.raise_for(rc)
    return {"models": s["models"], "masks": s["masks"], "inliers": s["inliers"]}


def _run_predict(s):
    logit, prob = guided.predict(s["net"], s["feat"])
    return {"logit": logit, "prob": prob}


def _run_train(s):
    tr = guided.Trainer(params=s["net"])
    losses = tr.train(s["feat"], s["labels"], steps=s["case"]["steps"], batch=s["case"]["batch"], lr=1e-3,
                      seed=s["seed"])
    return {"params": tr.params, "m": tr.m, "v": tr.v, "losses": losses}


# ---------------------------------------------------------------------------
# work, tolerance, exact
# ---------------------------------------------------------------------------

FLOPS_PER_RESIDUAL = {"homography": 18.0, "fundamental": 42.0, "essential": 42.0}
FLOPS_PER_SOLVE = {"homography": 700.0, "fundamental": 1500.0, "essential": 12000.0}
MODELS_PER_SOLVE = {"homography": 1.0, "fundamental": 2.0, "essential": 4.0}
FORWARD_FLOPS = 2.0 * (8 * 128 + 128 * 128 + 128 * 128 + 128)
TRAIN_FLOPS = FORWARD_FLOPS + 2.0 * (2 * 128 * 128 + 128) + 2.0 * (8 * 128 + 2 * 128 * 128 + 128)
NUM_PARAMS = guided.NUM_PARAMS


def _pair_work(kind, n, inliers, max_iters):
    """Rows in, mask out; the samples that the 0.99-confidence rule asks for,
    solved and scored on every point."""
    p = inliers ** SAMPLE[kind]
    iters = min(max_iters, max(50.0, math.log(0.01) / math.log1p(-p)))
    return 32.0 * n + n + 72, iters * (FLOPS_PER_SOLVE[kind] + MODELS_PER_SOLVE[kind] * n * FLOPS_PER_RESIDUAL[kind])


def work(case):
    path = case["path"]
    if path == "score":
        n, k = case["n"], case["models"]
        return {"bytes": 32.0 * n + 72.0 * k + 16.0 * k + (n * k if case["masks"] else 0),
                "flops": FLOPS_PER_RESIDUAL[case["kind"]] * n * k}
    if path == "predict":
        return {"bytes": case["n"] * (32.0 + 8.0) + 4.0 * NUM_PARAMS, "flops": FORWARD_FLOPS * case["n"]}
    if path == "train":
        rows = float(case["batch"] * case["steps"])
        return {"bytes": 36.0 * case["n"] + 24.0 * NUM_PARAMS, "flops": TRAIN_FLOPS * rows}
    if path == "single":
        b, f = _pair_work(case["kind"], case["n"], case["inliers"], case["max_iters"])
        return {"bytes": b, "flops": f}
    if path == "guided":
        kinds, counts = ["fundamental"] * case["pairs"], [case["n"]] * case["pairs"]
    else:
        kinds, counts = _batch_kinds_counts(case, 0)
    both = [_pair_work(k, n, case["inliers"], case["max_iters"]) for k, n in zip(kinds, counts)]
    extra = FORWARD_FLOPS * sum(counts) if path == "guided" else 0.0
    return {"bytes": sum(b for b, _ in both), "flops": sum(f for _, f in both) + extra}


def tolerance(case):
    path = case["path"]
    if path == "score":
        # FP64 sums of up to n residuals; counts and masks are whole values
        return {"rel": 1e-12}
    if path == "predict":
        # BF16 weights and activations: 0.24 % (logits) and 0.32 %
        # (probabilities) off the 64-bit network, four times that
        return {"rel": 1.2e-2}
    if path == "train":
        # BF16 passes: 0.16 % (second moments) off 64-bit training, four times
        # that; Adam's normalised steps carry a rounding on
        return {"rel": 7e-3}
    # whole runs are reproducible: the same masks, and models from the same
    # FP64 operations (another order of the same sums moves a model by ~1e-11)
    return {"rel": 1e-10}


def exact(case, seed):
    if case["path"] == "score":
        return _exact_score(case, seed)
    if case["path"] == "predict":
        return _exact_predict(case, seed)
    if case["path"] == "train":
        return _exact_train(case, seed)
    return None  # a whole RANSAC run has no closed form


def _exact_score(case, seed):
    s = _prepare_score(case, seed)
    x1, y1, x2, y2 = s["pts"].unbind(1)
    out = []
    step = max(1, 40000000 // case["n"])
    for a in range(0, case["models"], step):
        m = s["models"][a:a + step, :, None]
        e0 = m[:, 0] * x1 + m[:, 1] * y1 + m[:, 2]
        e1 = m[:, 3] * x1 + m[:, 4] * y1 + m[:, 5]
        e2 = m[:, 6] * x1 + m[:, 7] * y1 + m[:, 8]
        if case["kind"] == "homography":
            r2 = (x2 - e0 / e2) ** 2 + (y2 - e1 / e2) ** 2
        else:
            g0 = m[:, 0] * x2 + m[:, 3] * y2 + m[:, 6]
            g1 = m[:, 1] * x2 + m[:, 4] * y2 + m[:, 7]
            r2 = (x2 * e0 + y2 * e1 + e2) ** 2 / (e0 * e0 + e1 * e1 + g0 * g0 + g1 * g1)
        gain = 1.0 - r2 / s["sq_thr"]
        out.append(torch.where(gain > 0, gain, 0.0).sum(1))
    return {"counts": None, "values": torch.cat(out), **({"masks": None} if case["masks"] else {})}


def _split(net):
    p = torch.as_tensor(net, device="cuda").double()
    o = guided.OFF
    return [p[o["W1"]:o["b1"]].reshape(128, 8), p[o["b1"]:o["W2"]], p[o["W2"]:o["b2"]].reshape(128, 128),
            p[o["b2"]:o["W3"]], p[o["W3"]:o["b3"]].reshape(128, 128), p[o["b3"]:o["w4"]], p[o["w4"]:o["b4"]],
            p[o["b4"]:]]


def _forward(ws, x):
    act = lambda z: torch.nn.functional.gelu(z, approximate="tanh")  # noqa: E731
    x = act(x @ ws[0].T + ws[1])
    x = act(x @ ws[2].T + ws[3])
    x = act(x @ ws[4].T + ws[5])
    return x @ ws[6] + ws[7]


def _exact_predict(case, seed):
    s = _prepare_predict(case, seed)
    ws = _split(s["net"])
    logit = torch.cat([_forward(ws, torch.as_tensor(f, device="cuda").double())
                       for f in np.array_split(s["feat"], max(1, case["n"] // 100000))])
    return {"logit": logit, "prob": torch.sigmoid(logit)}


def _mix(x):
    """The row hash of the training step's mini-batches (splitmix64), on uint64 arrays."""
    x = x + np.uint64(0x9E3779B97F4A7C15)
    x = (x ^ (x >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    x = (x ^ (x >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return x ^ (x >> np.uint64(31))


def _exact_train(case, seed):
    s = _prepare_train(case, seed)
    feat, label = torch.as_tensor(s["feat"], device="cuda").double(), torch.as_tensor(s["labels"], device="cuda").double()
    ws = [w.clone().requires_grad_(True) for w in _split(s["net"])]
    m = [torch.zeros_like(w) for w in ws]
    v = [torch.zeros_like(w) for w in ws]
    losses = []
    for t in range(1, case["steps"] + 1):
        with np.errstate(over="ignore"):
            slot = np.uint64(t) * np.uint64(0x100000001B3) + np.arange(case["batch"], dtype=np.uint64)
            row = _mix(np.uint64(s["seed"]) ^ _mix(slot)) % np.uint64(case["n"])
        idx = torch.as_tensor(row.astype(np.int64), device="cuda")
        loss = torch.nn.functional.binary_cross_entropy_with_logits(_forward(ws, feat[idx]), label[idx])
        losses.append(loss.detach())
        grads = torch.autograd.grad(loss, ws)
        with torch.no_grad():
            for w, gr, mm, vv in zip(ws, grads, m, v):
                mm.mul_(0.9).add_(gr, alpha=0.1)
                vv.mul_(0.999).addcmul_(gr, gr, value=0.001)
                w -= 1e-3 * (mm / (1 - 0.9 ** t)) / ((vv / (1 - 0.999 ** t)).sqrt() + 1e-8)
    flat = lambda a: torch.cat([x.detach().reshape(-1) for x in a])  # noqa: E731
    return {"params": flat(ws), "m": flat(m), "v": flat(v), "losses": torch.stack(losses)}
