"""The error bound of the matrix-core scoring pass, checked on the CPU.

The kernel (csrc/k_score_mx.hip) drops a point for a model only when the
low-precision quantities prove it an outlier, using
delta = 2^-17 S + 2^-20 for a quantity c . z with |c_t| <= 1, S = sum of |z_t|
over the terms it reads.  This test rebuilds the kernel's operands exactly as
it does -- z in FP64 then rounded to FP32, FP16 hi = fp16(z), lo = fp16(z - hi)
(the coefficients split from FP64) -- forms the 27 products hi*hi, hi*lo,
lo*hi (exact in FP32) and accumulates them in FP32 in several orders (the
MFMA's internal order is not specified), then compares with the exact value
(FP64 from the unsplit operands, whose own error is ~1e-16).  Inputs include
near-threshold cases, tiny and subnormal-range operands, and coordinates at
the scale limit |x'| = 1.  The measured worst case is reported as a fraction
of the bound; the bound must hold everywhere.
"""
import os
import shutil
import subprocess

import numpy as np
import pytest


def _split16(v):
    hi = v.astype(np.float16)
    lo = (v - hi.astype(v.dtype)).astype(np.float16)
    return hi, lo


def _z(x1, y1, x2, y2):
    return np.stack([x2 * x1, x2 * y1, x2, y2 * x1, y2 * y1, y2, x1, y1, np.ones_like(x1)], axis=-1)


def _quantities(F):
    """Coefficient vectors of C, (F x1)_0, (F x1)_1, (F^T x2)_0, (F^T x2)_1
    and of the transfer quantities P, Q, W (as the kernel builds them)."""
    n = F.shape[0]
    c = np.zeros((n, 8, 9))
    c[:, 0] = F
    c[:, 1, 6:9] = F[:, 0:3]
    c[:, 2, 6:9] = F[:, 3:6]
    c[:, 3, [2, 5, 8]] = F[:, [0, 3, 6]]
    c[:, 4, [2, 5, 8]] = F[:, [1, 4, 7]]
    c[:, 5, [0, 1, 2]] = F[:, 6:9]
    c[:, 5, [6, 7, 8]] = -F[:, 0:3]
    c[:, 6, [3, 4, 5]] = F[:, 6:9]
    c[:, 6, [6, 7, 8]] = -F[:, 3:6]
    c[:, 7, [6, 7, 8]] = F[:, 6:9]
    return c


def _sum_terms(q):
    """Which z terms each quantity reads -> the S of its bound."""
    return [[0, 1, 2, 3, 4, 5, 6, 7, 8], [6, 7, 8], [6, 7, 8], [2, 5, 8], [2, 5, 8],
            [0, 1, 2, 6, 7, 8], [3, 4, 5, 6, 7, 8], [6, 7, 8]][q]


def _bound_sets():
    # the kernel's three bounds: d[0] uses (1+|x1|+|y1|)(1+|x2|+|y2|) (C, P, Q),
    # d[1] 1+|x1|+|y1| ((F x1), W), d[2] 1+|x2|+|y2| ((F^T x2))
    return [0, 1, 1, 2, 2, 0, 0, 1]


def test_low_precision_error_within_kernel_bound():
    rng = np.random.default_rng(17)
    worst = 0.0
    for trial in range(40):
        nm, npts = 64, 256
        # models with |F''| <= 1: random, scaled, with tiny and zero entries
        F = rng.uniform(-1, 1, (nm, 9))
        F *= 10.0 ** rng.uniform(-7, 0, (nm, 9))
        F[rng.uniform(size=F.shape) < 0.05] = 0.0
        F /= np.abs(F).max(axis=1, keepdims=True)
        # scaled points |x'| <= 1, some at the limit, some tiny
        P = rng.uniform(-1, 1, (npts, 4)) * (10.0 ** rng.uniform(-6, 0, (npts, 4)))
        P[: npts // 8] = np.sign(P[: npts // 8]) * 1.0
        x1, y1, x2, y2 = P.T
        zd = _z(x1, y1, x2, y2)                      # FP64
        z32 = zd.astype(np.float32)
        zh, zl = _split16(z32)
        c = _quantities(F)                           # (nm, 8, 9) FP64
        ch, cl = _split16(c)
        exact = np.einsum("mqt,pt->mqp", c, zd)      # FP64 reference
        # the 27 products, exact in FP32 (11-bit x 11-bit significands)
        prods = np.concatenate([
            np.einsum("mqt,pt->mqpt", ch.astype(np.float32), zh.astype(np.float32)),
            np.einsum("mqt,pt->mqpt", ch.astype(np.float32), zl.astype(np.float32)),
            np.einsum("mqt,pt->mqpt", cl.astype(np.float32), zh.astype(np.float32))], axis=-1)
        sa = 1 + np.abs(x1) + np.abs(y1)
        sb = 1 + np.abs(x2) + np.abs(y2)
        S = np.stack([sa * sb, sa, sb])              # (3, npts)
        delta = 2.0 ** -17 * S + 2.0 ** -20
        bsel = _bound_sets()
        for order in range(3):
            perm = rng.permutation(27) if order else np.arange(27)
            acc = np.zeros(prods.shape[:3], np.float32)
            for k in perm:
                acc = (acc + prods[..., k]).astype(np.float32)
            err = np.abs(acc.astype(np.float64) - exact)
            for q in range(8):
                ratio = err[:, q, :] / delta[bsel[q]][None, :]
                worst = max(worst, float(ratio.max()))
                assert (ratio <= 1.0).all(), (trial, order, q, float(ratio.max()))
                # the S the kernel uses covers the terms the quantity reads
                Sq = np.abs(zd[:, _sum_terms(q)]).sum(axis=1)
                assert (Sq <= S[bsel[q]] * (1 + 1e-12)).all()
    print("worst low-precision error: %.3f of the kernel's bound" % worst)
    assert worst < 0.5


def test_rejection_never_drops_an_inlier():
    """End-to-end on scaled Sampson quantities: the kernel's rejection test,
    evaluated on the emulated low-precision values, never fires for a point
    whose exact squared Sampson distance is below the threshold; and it does
    fire for most far points (the pass is useful)."""
    rng = np.random.default_rng(23)
    rejected_far = total_far = 0
    for trial in range(30):
        # a rank-2 F'' and points near and far from its epipolar geometry
        U, _, Vt = np.linalg.svd(rng.normal(size=(3, 3)))
        F = (U @ np.diag([1.0, rng.uniform(0.2, 1.0), 0.0]) @ Vt).ravel()
        F /= np.abs(F).max()
        n = 2000
        x1 = rng.uniform(-1, 1, (n, 2))
        l2 = np.c_[x1, np.ones(n)] @ F.reshape(3, 3).T
        # x2 on its epipolar line, then moved off it by d (normalised units)
        t = rng.uniform(-1, 1, n)
        nrm = l2[:, :2] / np.linalg.norm(l2[:, :2], axis=1, keepdims=True)
        foot = -l2[:, 2:3] * nrm / np.linalg.norm(l2[:, :2], axis=1, keepdims=True)
        x2 = foot + t[:, None] * nrm[:, ::-1] * [1, -1]
        d = 10.0 ** rng.uniform(-5, -1, n) * rng.choice([-1, 1], n)
        x2 = x2 + d[:, None] * nrm
        keep = (np.abs(x2) <= 1).all(axis=1)
        x1, x2 = x1[keep], x2[keep]
        zd = _z(x1[:, 0], x1[:, 1], x2[:, 0], x2[:, 1])
        zh, zl = _split16(zd.astype(np.float32))
        c = _quantities(F[None])[0, :5]
        ch, cl = _split16(c)
        q = (ch.astype(np.float32) @ zh.astype(np.float32).T + ch.astype(np.float32) @ zl.astype(np.float32).T +
             cl.astype(np.float32) @ zh.astype(np.float32).T).astype(np.float32)
        ex = c @ zd.T
        sampson = ex[0] ** 2 / (ex[1] ** 2 + ex[2] ** 2 + ex[3] ** 2 + ex[4] ** 2)
        tau2 = (2e-3) ** 2
        sa = (1 + np.abs(x1).sum(1)).astype(np.float32)
        sb = (1 + np.abs(x2).sum(1)).astype(np.float32)
        dC = np.float32(2.0 ** -17) * sa * sb + np.float32(2.0 ** -20)
        da = np.float32(2.0 ** -17) * sa + np.float32(2.0 ** -20)
        db = np.float32(2.0 ** -17) * sb + np.float32(2.0 ** -20)
        den = ((np.abs(q[1]) + da) ** 2 + (np.abs(q[2]) + da) ** 2 + (np.abs(q[3]) + db) ** 2 +
               (np.abs(q[4]) + db) ** 2).astype(np.float32)
        cl_ = (np.abs(q[0]) - dC).astype(np.float32)
        tau2m = np.float32(tau2 * (1 + 2.0 ** -16))
        rej = (cl_ > 0) & (cl_ * cl_ > den * tau2m)
        assert not (rej & (sampson < tau2)).any(), trial
        far = sampson > 4 * tau2
        rejected_far += int((rej & far).sum())
        total_far += int(far.sum())
    assert rejected_far > 0.95 * total_far


def _denominator_coefs(F):
    """A quarter of |(F x1)_01|^2 + |(F^T x2)_01|^2 over the squared terms."""
    g = np.zeros((F.shape[0], 11))
    for h, rows in enumerate((([0, 1, 2], [3, 4, 5]), ([0, 3, 6], [1, 4, 7]))):
        a, b = F[:, rows[0]], F[:, rows[1]]
        g[:, 5 * h] = 0.25 * (a[:, 0] ** 2 + b[:, 0] ** 2)
        g[:, 5 * h + 1] = 0.5 * (a[:, 0] * a[:, 1] + b[:, 0] * b[:, 1])
        g[:, 5 * h + 2] = 0.25 * (a[:, 1] ** 2 + b[:, 1] ** 2)
        g[:, 5 * h + 3] = 0.5 * (a[:, 0] * a[:, 2] + b[:, 0] * b[:, 2])
        g[:, 5 * h + 4] = 0.5 * (a[:, 1] * a[:, 2] + b[:, 1] * b[:, 2])
        g[:, 10] += 0.25 * (a[:, 2] ** 2 + b[:, 2] ** 2)
    return g


def test_denominator_form_within_kernel_bound():
    """The Sampson denominator as one linear form of 32 products: within
    2^-17 S + 2^-20 of a quarter of the sum of squares in every order of
    accumulation, and the rejection test with it never drops an inlier."""
    rng = np.random.default_rng(29)
    worst = 0.0
    for trial in range(40):
        nm, npts = 64, 256
        F = rng.uniform(-1, 1, (nm, 9)) * 10.0 ** rng.uniform(-7, 0, (nm, 9))
        F[rng.uniform(size=F.shape) < 0.05] = 0.0
        F /= np.abs(F).max(axis=1, keepdims=True)
        if trial % 4 == 0:
            F = np.sign(F)  # every coefficient at its limit
        P = rng.uniform(-1, 1, (npts, 4)) * (10.0 ** rng.uniform(-6, 0, (npts, 4)))
        P[: npts // 8] = np.sign(P[: npts // 8]) * 1.0
        x1, y1, x2, y2 = P.T
        d = np.stack([x1 * x1, x1 * y1, y1 * y1, x1, y1, x2 * x2, x2 * y2, y2 * y2, x2, y2, np.ones(npts)], -1)
        g = _denominator_coefs(F)
        assert np.abs(g).max() <= 1.0
        z1, z2 = np.c_[P[:, :2], np.ones(npts)], np.c_[P[:, 2:], np.ones(npts)]
        M = F.reshape(nm, 3, 3)
        l1 = np.einsum("mij,pj->mpi", M, z1)[..., :2]
        l2 = np.einsum("mji,pj->mpi", M, z2)[..., :2]
        exact = 0.25 * ((l1 ** 2).sum(-1) + (l2 ** 2).sum(-1))
        dh, dl = _split16(d.astype(np.float32))
        gh, gl = _split16(g)
        assert (dl[:, 10] == 0).all()
        f = np.float32
        prods = np.concatenate([gh.astype(f)[:, None] * dh.astype(f)[None],
                                gh.astype(f)[:, None, :10] * dl.astype(f)[None, :, :10],
                                gl.astype(f)[:, None] * dh.astype(f)[None]], axis=-1)
        assert prods.shape[-1] == 32
        ax, ay, bx, by = np.abs(P).astype(f).T
        sa, sb = 1 + ax + ay, 1 + bx + by
        S = 1 + ax * sa + ay * (1 + ay) + bx * sb + by * (1 + by)
        assert (np.abs(d).sum(-1) <= S * (1 + 1e-6)).all()
        dD = f(2.0 ** -17) * S + f(2.0 ** -20)
        dC = f(2.0 ** -17) * (sa * sb) + f(2.0 ** -20)
        zh, zl = _split16(_z(x1, y1, x2, y2).astype(f))
        ch, cl = _split16(F)
        c32 = (ch.astype(f) @ zh.astype(f).T + ch.astype(f) @ zl.astype(f).T + cl.astype(f) @ zh.astype(f).T).astype(f)
        C = F @ _z(x1, y1, x2, y2).T
        for order in range(3):
            perm = rng.permutation(32) if order else np.arange(32)
            acc = np.zeros(prods.shape[:2], f)
            for k in perm:
                acc = (acc + prods[..., k]).astype(f)
            worst = max(worst, float((np.abs(acc - exact) / dD[None]).max()))
            for tau in (1e-4, 2e-3, 0.1):
                k1 = f(4) * f(tau ** 2 * (1 + 2.0 ** -16))
                low = np.abs(c32) - dC[None]
                rej = low * np.abs(low) > acc * k1 + k1 * dD[None]
                assert not (rej & (C ** 2 < tau ** 2 * 4 * exact)).any(), (trial, order, tau)
    print("worst denominator error: %.3f of the kernel's bound" % worst)
    assert worst < 0.5


def test_scaled_test_never_drops_an_inlier():
    """The kernel's whole test -- operands scaled by sigma and kappa, the slack
    as the accumulator's first term, the sign of den - c^2 -- on thresholds over
    the whole range: no point below the threshold is dropped, and most far ones
    are."""
    rng = np.random.default_rng(31)
    f = np.float32
    h, margin = 2.0 ** -4, 1 + 2.0 ** -14
    far_n = far_rej = 0
    for trial in range(60):
        tau = 10.0 ** rng.uniform(-6, -0.4)
        transfer = trial % 3 == 2
        kappa = 4 * tau * tau * margin * (1 + h)
        assert kappa < 1
        sigma = 1.0
        for _ in range(12):
            if kappa < 1:
                sigma, kappa = 2 * sigma, 4 * kappa
        assert kappa < 4 and sigma <= 4096
        F = rng.uniform(-1, 1, (32, 9)) * 10.0 ** rng.uniform(-3, 0, (32, 9))
        F /= np.abs(F).max(axis=1, keepdims=True)
        n = 2048
        P = rng.uniform(-1, 1, (n, 4))
        zero = np.zeros(n)
        for m in range(32):  # near the threshold of some model, from both sides
            i = np.arange(m, n, 32)
            p1 = np.c_[P[i, :2], np.ones(len(i))]
            l = p1 @ F[m].reshape(3, 3).T
            if transfer:
                ang = rng.uniform(0, 2 * np.pi, len(i))
                off = tau * (1 + 10.0 ** rng.uniform(-6, -1, len(i)) * rng.choice([-1, 1], len(i)))
                P[i, 2:] = l[:, :2] / l[:, 2:3] + off[:, None] * np.c_[np.cos(ang), np.sin(ang)]
            else:
                nn = np.maximum(np.linalg.norm(l[:, :2], axis=1), 1e-30)
                d = (l[:, 0] * P[i, 2] + l[:, 1] * P[i, 3] + l[:, 2]) / nn
                off = tau * (1 + 10.0 ** rng.uniform(-6, 0, len(i)) * rng.choice([-1, 1], len(i)))
                P[i, 2:] -= ((d - off) / nn)[:, None] * l[:, :2]
        P = P[(np.abs(P) <= 1).all(1)]
        x1, y1, x2, y2 = P.T
        z, one = _z(x1, y1, x2, y2), np.ones(len(P))
        d = np.stack([x1 * x1, x1 * y1, y1 * y1, x1, y1, x2 * x2, x2 * y2, y2 * y2, x2, y2, one], -1)
        if transfer:
            num_c = _quantities(F)[:, 5:7]
            g = np.zeros((32, 11))
            a = F[:, 6:9]
            g[:, 0], g[:, 1], g[:, 2] = a[:, 0] ** 2 / 4, a[:, 0] * a[:, 1] / 2, a[:, 1] ** 2 / 4
            g[:, 3], g[:, 4], g[:, 10] = a[:, 0] * a[:, 2] / 2, a[:, 1] * a[:, 2] / 2, a[:, 2] ** 2 / 4
        else:
            num_c = F[:, None, :]
            g = _denominator_coefs(F)
        exact = ((num_c @ z.T) ** 2).sum(1) / (4 * np.maximum(g @ d.T, 1e-300))
        sa, sb = 1 + np.abs(x1) + np.abs(y1), 1 + np.abs(x2) + np.abs(y2)
        sd = 1 + np.abs(x1) * sa + np.abs(y1) * (1 + np.abs(y1)) + np.abs(x2) * sb + np.abs(y2) * (1 + np.abs(y2))
        dc = sigma * (2.0 ** -17 * sa * sb + 2.0 ** -20)
        slack = (margin * (max(kappa, 1) * (2.0 ** -17 * sd + 2.0 ** -20) + (1 + 1 / h) * dc * dc)).astype(f)
        dh, dl = _split16(d.astype(f))
        zh, zl = _split16(z.astype(f))
        gh, gl = _split16(g * kappa)
        prods = np.concatenate([gh.astype(f)[:, None] * dh.astype(f)[None],
                                gh.astype(f)[:, None, :10] * dl.astype(f)[None, :, :10],
                                gl.astype(f)[:, None] * dh.astype(f)[None]], axis=-1)
        t = np.broadcast_to(slack, prods.shape[:2]).astype(f)
        for k in rng.permutation(32):
            t = (t + prods[..., k]).astype(f)
        t = t.astype(np.float64)
        for q in range(num_c.shape[1]):
            ch, cl = _split16(num_c[:, q] * sigma)
            pr = np.concatenate([ch.astype(f)[:, None] * zh.astype(f)[None], ch.astype(f)[:, None] * zl.astype(f)[None],
                                 cl.astype(f)[:, None] * zh.astype(f)[None]], axis=-1)
            c = np.zeros(pr.shape[:2], f)
            for k in rng.permutation(27):
                c = (c + pr[..., k]).astype(f)
            t = (t - c.astype(np.float64) ** 2).astype(f).astype(np.float64)
        rej = t < 0
        assert not (rej & (exact < tau * tau)).any(), (trial, tau, transfer)
        if tau > 5e-4:
            far = exact > 4 * tau * tau
            far_n += int(far.sum())
            far_rej += int((rej & far).sum())
    print("far points dropped: %.3f" % (far_rej / far_n))
    assert far_rej > 0.9 * far_n


def test_operands_of_any_model_are_numbers(tmp_path):
    """The kernel's own normalisation (csrc/mx_rules.hpp) on models with inf,
    NaN, huge and subnormal entries: operands of magnitude at most 1, or all
    zero, with which nothing is dropped."""
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("g++ not available")
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    exe = str(tmp_path / "mx_check")
    subprocess.check_call([gxx, "-std=c++17", "-O2", "-ffp-contract=off", "-Wno-unknown-pragmas", "-o", exe, "-I",
                           os.path.join(root, "graph-cut-ransac_amd", "csrc"),
                           os.path.join(root, "tests", "cpp", "mx_check.cpp")])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
