"""The error bounds of the matrix-core scoring pass, checked on the CPU.

The kernel (csrc/k_score_mx.hip) drops a point for a model only when the
low-precision quantities prove it an outlier: c^2 > d + slack, c from the
quantities C (Sampson) or P and Q (transfer) times sigma, d from a quarter D of
the denominator times kappa, the slack the accumulator's first term.  The models'
coefficients, the points' terms, sigma, kappa and the slack come from the header
that the kernel is built from (csrc/mx_rules.hpp); this test splits them as the
kernel does -- terms rounded to FP32, FP16 hi = fp16(v), lo = fp16(v - hi), the
coefficients split from FP64 -- forms the products hi*hi, hi*lo, lo*hi (exact in
FP32) and accumulates them in FP32 in several orders (the matrix unit's internal
order is not specified), then compares with FP64 from the unsplit numbers.
Inputs include near-threshold points, tiny and subnormal-range operands, and
coordinates at the scale limit |x'| = 1.
"""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
F32 = np.float32


class Rules:
    """csrc/mx_rules.hpp through ctypes."""

    def __init__(self, path):
        self.lib = ctypes.CDLL(path)

    @staticmethod
    def _p(a):
        return a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))

    def scales(self, s, sq_thr):
        out = np.zeros(3)
        self.lib.mx_scales(ctypes.c_double(s), ctypes.c_double(sq_thr), self._p(out))
        return bool(out[0]), out[1], out[2]

    def models(self, kind, M, s, sq_thr):
        """Normalised models (m, 9), quantities (m, 1 or 2, 9), denominators (m, 11)."""
        M = np.ascontiguousarray(M, np.float64)
        out = np.zeros((len(M), 38))
        self.lib.mx_models(ctypes.c_int32(kind), ctypes.c_int64(len(M)), self._p(M), ctypes.c_double(s),
                           ctypes.c_double(sq_thr), self._p(out))
        return out[:, :9], out[:, 9:27].reshape(-1, 2, 9)[:, :1 if kind == 1 else 2], out[:, 27:]

    def points(self, P, s, sq_thr):
        """Terms z (n, 9), squared terms (n, 11), slack (n,)."""
        P = np.ascontiguousarray(P, np.float64)
        out = np.zeros((len(P), 21))
        self.lib.mx_points(ctypes.c_int64(len(P)), self._p(P), ctypes.c_double(s), ctypes.c_double(sq_thr),
                           self._p(out))
        return out[:, :9], out[:, 9:20], out[:, 20]


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("g++ not available")
    so = str(tmp_path_factory.mktemp("mx") / "mx_rules_check.so")
    subprocess.check_call([gxx, "-std=c++17", "-O2", "-ffp-contract=off", "-Wno-unknown-pragmas", "-shared", "-fPIC",
                           "-o", so, "-I", os.path.join(ROOT, "graph-cut-ransac_amd", "csrc"),
                           os.path.join(ROOT, "tests", "cpp", "mx_rules_check.cpp")])
    return Rules(so)


def _split16(v):
    hi = v.astype(np.float16)
    lo = (v - hi.astype(v.dtype)).astype(np.float16)
    return hi.astype(F32), lo.astype(F32)


def _products(coefs, terms, last_is_one):
    """The products of one quantity, (m, n, 27 or 32): hi hi, hi lo (not of a
    last term that is 1, whose lo is 0) and lo hi."""
    ch, cl = _split16(coefs)
    zh, zl = _split16(terms.astype(F32))
    t = terms.shape[1] - 1 if last_is_one else terms.shape[1]
    if last_is_one:
        assert (zl[:, t] == 0).all()
    return np.concatenate([ch[:, None] * zh[None], ch[:, None, :t] * zl[None, :, :t], cl[:, None] * zh[None]], axis=-1)


def _accumulate(prods, rng, first=0.0):
    acc = np.broadcast_to(np.asarray(first, F32), prods.shape[:2]).astype(F32)
    for k in rng.permutation(prods.shape[-1]):
        acc = (acc + prods[..., k]).astype(F32)
    return acc


def _random_models(rng, trial, count=64):
    F = rng.uniform(-1, 1, (count, 9)) * 10.0 ** rng.uniform(-7, 0, (count, 9))
    F[rng.uniform(size=F.shape) < 0.05] = 0.0
    F[(F == 0).all(axis=1), 0] = 1.0
    return np.sign(F) + (F == 0) if trial % 4 == 0 else F  # every coefficient at its limit


def _random_points(rng, count=256):
    P = rng.uniform(-1, 1, (count, 4)) * (10.0 ** rng.uniform(-6, 0, (count, 4)))
    P[: count // 8] = np.sign(P[: count // 8])
    return P


def _sums(P):
    """The S of the bounds: of z and of the squared terms."""
    ax, ay, bx, by = np.abs(P).T
    sa, sb = 1 + ax + ay, 1 + bx + by
    return sa * sb, 1 + ax * sa + ay * (1 + ay) + bx * sb + by * (1 + by)


@pytest.mark.parametrize("kind", [1, 0])
def test_low_precision_error_within_kernel_bound(rules, kind):
    """C, P and Q within 2^-17 S + 2^-20 of their exact values at every sigma (the
    transfer test needs sqrt(2) times the error of each below it)."""
    rng = np.random.default_rng(17 + kind)
    worst = 0.0
    for trial in range(40):
        sq_thr = 10.0 ** rng.uniform(-12, -1)
        on, sigma, _ = rules.scales(1.0, sq_thr)
        assert on
        F, cq, _ = rules.models(kind, _random_models(rng, trial), 1.0, sq_thr)
        assert np.abs(F).max() <= 1.0 and np.abs(cq).max() <= 1.0
        P = _random_points(rng)
        z, _, _ = rules.points(P, 1.0, sq_thr)
        S, _ = _sums(P)
        delta = 2.0 ** -17 * S + 2.0 ** -20
        for q in range(cq.shape[1]):
            read = np.abs(z) @ (np.abs(cq[:, q]) > 0).T  # the terms that the quantity reads
            assert (read <= S[:, None] * (1 + 1e-12)).all()
            exact = cq[:, q] @ z.T
            prods = _products(cq[:, q] * sigma, z, False)
            for _ in range(3):
                err = np.abs(_accumulate(prods, rng).astype(np.float64) / sigma - exact)
                worst = max(worst, float((err / delta[None]).max()))
    print("worst low-precision error: %.3f of the kernel's bound" % worst)
    assert worst < 0.5


@pytest.mark.parametrize("kind", [1, 0])
def test_denominator_form_within_kernel_bound(rules, kind):
    """The denominator as one linear form of 32 products: kappa D within
    max(kappa, 1) (2^-17 S + 2^-20) of kappa / 4 times the sum of squares."""
    rng = np.random.default_rng(29 + kind)
    worst = 0.0
    for trial in range(40):
        sq_thr = 10.0 ** rng.uniform(-12, -1)
        _, _, kappa = rules.scales(1.0, sq_thr)
        F, _, g = rules.models(kind, _random_models(rng, trial), 1.0, sq_thr)
        assert np.abs(g).max() <= 1.0
        P = _random_points(rng)
        _, d, _ = rules.points(P, 1.0, sq_thr)
        _, S = _sums(P)
        assert (np.abs(d).sum(-1) <= S * (1 + 1e-12)).all()
        M = F.reshape(-1, 3, 3)
        p1, p2 = np.c_[P[:, :2], np.ones(len(P))], np.c_[P[:, 2:], np.ones(len(P))]
        l1 = np.einsum("mij,pj->mpi", M, p1)
        if kind == 1:
            l2 = np.einsum("mji,pj->mpi", M, p2)
            exact = 0.25 * ((l1[..., :2] ** 2).sum(-1) + (l2[..., :2] ** 2).sum(-1))
        else:
            exact = 0.25 * l1[..., 2] ** 2
        np.testing.assert_allclose(g @ d.T, exact, rtol=0, atol=1e-13)
        prods = _products(g * kappa, d, True)
        assert prods.shape[-1] == 32
        bound = max(kappa, 1.0) * (2.0 ** -17 * S + 2.0 ** -20)
        for _ in range(3):
            err = np.abs(_accumulate(prods, rng).astype(np.float64) - kappa * exact)
            worst = max(worst, float((err / bound[None]).max()))
    print("worst denominator error: %.3f of the kernel's bound" % worst)
    assert worst < 0.5


def _dropped(rules, kind, M, P, s, sq_thr, rng):
    """The kernel's test of the models M and the points P (scale s): (m, n)."""
    on, sigma, kappa = rules.scales(s, sq_thr)
    F, cq, g = rules.models(kind, M, s, sq_thr)
    z, d, slack = rules.points(P, s, sq_thr)
    t = _accumulate(_products(g * kappa, d, True), rng, slack)
    for q in range(cq.shape[1]):
        c = _accumulate(_products(cq[:, q] * sigma, z, False), rng).astype(np.float64)
        # one fused multiply-add: exact product and sum, one rounding
        t = (t.astype(np.float64) - c * c).astype(F32)
    return np.signbit(t) & on


def _distance(kind, M, P):
    """Exact squared distances (m, n)."""
    out = []
    p1, p2 = np.c_[P[:, :2], np.ones(len(P))], np.c_[P[:, 2:], np.ones(len(P))]
    for m in M.reshape(-1, 3, 3):
        a = p1 @ m.T
        if kind == 1:
            b = p2 @ m
            out.append((p2 * a).sum(1) ** 2 / np.maximum((a[:, :2] ** 2).sum(1) + (b[:, :2] ** 2).sum(1), 1e-300))
        else:
            out.append(((P[:, 2:] - a[:, :2] / a[:, 2:3]) ** 2).sum(1))
    return np.array(out)


def test_rejection_never_drops_an_inlier(rules):
    """Rank-2 models on pixel coordinates (a scale that is not 1), points on
    their epipolar lines and off them: no point below the threshold is dropped,
    and nearly all beyond twice the threshold are."""
    rng = np.random.default_rng(23)
    rejected_far = total_far = 0
    for trial in range(30):
        U, _, Vt = np.linalg.svd(rng.normal(size=(3, 3)))
        F = (U @ np.diag([1.0, rng.uniform(0.2, 1.0), 0.0]) @ Vt).ravel()
        n = 2000
        x1 = rng.uniform(-1, 1, (n, 2))
        line = np.c_[x1, np.ones(n)] @ F.reshape(3, 3).T
        # x2 on its epipolar line, then moved off it by d
        t = rng.uniform(-1, 1, n)
        nrm = line[:, :2] / np.linalg.norm(line[:, :2], axis=1, keepdims=True)
        foot = -line[:, 2:3] * nrm / np.linalg.norm(line[:, :2], axis=1, keepdims=True)
        x2 = foot + t[:, None] * nrm[:, ::-1] * [1, -1]
        d = 10.0 ** rng.uniform(-5, -1, n) * rng.choice([-1, 1], n)
        x2 = x2 + d[:, None] * nrm
        s = 1024.0
        keep = (np.abs(x2) <= 1).all(axis=1)
        P = s * np.c_[x1, x2][keep]
        S = np.diag([1 / s, 1 / s, 1.0])
        M = (S @ F.reshape(3, 3) @ S).ravel()[None]
        tau2 = (2e-3 * s) ** 2
        dist = _distance(1, M, P)
        rej = _dropped(rules, 1, M, P, s, tau2, rng)
        assert not (rej & (dist < tau2)).any(), trial
        far = dist > 4 * tau2
        rejected_far += int((rej & far).sum())
        total_far += int(far.sum())
    assert rejected_far > 0.95 * total_far


def test_scaled_test_never_drops_an_inlier(rules):
    """Both distances, thresholds over the whole range, points near the
    threshold of some model from both sides: no point below the threshold is
    dropped, and most far ones are."""
    rng = np.random.default_rng(31)
    far_n = far_rej = 0
    for trial in range(60):
        tau = 10.0 ** rng.uniform(-6, -0.4)
        kind = 0 if trial % 3 == 2 else 1
        on, sigma, kappa = rules.scales(1.0, tau * tau)
        assert on and kappa < 4 and 1 <= sigma <= 4096
        F = rng.uniform(-1, 1, (32, 9)) * 10.0 ** rng.uniform(-3, 0, (32, 9))
        n = 2048
        P = rng.uniform(-1, 1, (n, 4))
        for m in range(32):
            i = np.arange(m, n, 32)
            p1 = np.c_[P[i, :2], np.ones(len(i))]
            a = p1 @ F[m].reshape(3, 3).T
            if kind == 0:
                ang = rng.uniform(0, 2 * np.pi, len(i))
                off = tau * (1 + 10.0 ** rng.uniform(-6, -1, len(i)) * rng.choice([-1, 1], len(i)))
                P[i, 2:] = a[:, :2] / a[:, 2:3] + off[:, None] * np.c_[np.cos(ang), np.sin(ang)]
            else:
                nn = np.maximum(np.linalg.norm(a[:, :2], axis=1), 1e-30)
                d = (a[:, 0] * P[i, 2] + a[:, 1] * P[i, 3] + a[:, 2]) / nn
                off = tau * (1 + 10.0 ** rng.uniform(-6, 0, len(i)) * rng.choice([-1, 1], len(i)))
                P[i, 2:] -= ((d - off) / nn)[:, None] * a[:, :2]
        P = P[(np.abs(P) <= 1).all(1)]
        dist = _distance(kind, F, P)
        rej = _dropped(rules, kind, F, P, 1.0, tau * tau, rng)
        assert not (rej & (dist < tau * tau)).any(), (trial, tau, kind)
        if tau > 5e-4:
            far = dist > 4 * tau * tau
            far_n += int(far.sum())
            far_rej += int((rej & far).sum())
    print("far points dropped: %.3f" % (far_rej / far_n))
    assert far_rej > 0.9 * far_n


@pytest.mark.parametrize("kind", [1, 0])
def test_operands_of_any_model_are_numbers(rules, kind):
    """Models with inf, NaN, huge and subnormal entries: operands of magnitude at
    most 1, or all zero, with which nothing is dropped.  (The test's answer is
    the sign of a multiply-add: a NaN would be one.)"""
    rng = np.random.default_rng(5 + kind)
    odd = np.array([np.inf, -np.inf, np.nan, -np.nan, 1e306, -1.7e308, 5e-324, 1e-310, -1e-301, 0.0, 1e300, 1e-300])
    P = _random_points(rng, 64)
    untested = 0
    for trial in range(300):
        M = rng.uniform(-1, 1, (64, 9)) * 10.0 ** rng.uniform(-6, 6, (64, 1))
        for _ in range(trial % 4):
            M[np.arange(64), rng.integers(0, 9, 64)] = odd[rng.integers(0, len(odd), 64)]
        M[::16] = odd[rng.integers(0, len(odd), (4, 9))]
        s = 2.0 ** rng.integers(-20, 20)
        sq_thr = [1e-4, 1e-4, 1e9, np.nan, -1.0][trial % 5] * s * s
        F, cq, g = rules.models(kind, M, s, sq_thr)
        for v in (F, cq, g):
            assert (np.abs(v) <= 1 + 1e-15).all(), trial  # (false for NaN)
        off = (F == 0).all(axis=1)
        assert off[~np.isfinite(M).all(axis=1)].all()
        if not rules.scales(s, sq_thr)[0]:
            assert off.all()
        else:
            assert (np.abs(F[~off]).max(axis=1) >= 1 - 1e-15).all()
            assert not _dropped(rules, kind, M, P * s, s, sq_thr, rng)[off].any()
        untested += int(off.sum())
    assert 1000 < untested < 300 * 64
