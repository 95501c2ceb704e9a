"""The deformation fit (emida_fit_deformation) of exact displacements where the ROIs span a
small part of the view: the normal matrix's blocks then differ by 1e6 and more, and a solver
that compares pivots with the whole trace loses digits that the data hold.

The fitted map is compared with the smallest eigenvector of the same normal matrix from
cyclic Jacobi rotations in extended precision (63-bit mantissa or more).  The tolerance is
32 times what the same rotations give in double, at the worst pattern of the layout, at least
1e-13: no digit that plain double arithmetic finds is lost to the method, and the factor
covers another order of the sums.
"""
import functools

import numpy as np
import pytest

from emida_amd import post as G

pytestmark = pytest.mark.gpu
P, MIN_ROIS = 5, 10
# ROIs, view size, detector distance in view sizes, spread of the ROIs about the centre, map
CASES = [(50, 1e4, 1.0, 1e-3, "small"), (100, 1.0, 1.0, 1e-3, "small"), (50, 800.0, 0.75, 1e-3, "stretch"),
         (300, 1e4, 1.0, 1e-3, "stretch"), (500, 800.0, 12.5, 1e-2, "small"), (600, 800.0, 1.0, 3e-3, "small")]


def _data(n, size, dist, spread, kind):
    rng = np.random.default_rng(n)
    cal = np.array([size / 2, size / 2, size * dist])
    mids = size / 2 + rng.normal(0, spread * size, (n, 2))
    offs = []
    for _ in range(P):
        F = np.diag([1.3, 0.7, 1.0]) if kind == "stretch" else np.eye(3)
        v = np.column_stack([mids - cal[:2], np.full(n, cal[2])]) @ (F + rng.normal(0, 2e-3, (3, 3))).T
        offs.append(v[:, :2] / v[:, 2:] * cal[2] + cal[:2] - mids)
    return mids, np.array(offs), cal


def _jacobi_null(mids, offs, cal, t):
    """The unit eigenvector of the smallest eigenvalue of A^T A, formed and rotated in type t."""
    z = t(cal[2])
    old = mids.astype(t) - cal[:2].astype(t)
    new = old + offs.astype(t)
    v = np.column_stack([old, np.full(len(old), z, t)])
    o = np.zeros_like(v)
    A = np.concatenate([np.concatenate([-v * z, o, v * new[:, :1]], 1), np.concatenate([o, -v * z, v * new[:, 1:]], 1)])
    a, e = A.T @ A, np.eye(9, dtype=t)
    eps = np.finfo(t).eps
    for _ in range(60):
        if not ((a - np.diag(np.diag(a))) ** 2).sum() > (eps * eps * 1e-2) * (np.diag(a) ** 2).sum():
            break
        for p in range(8):
            for q in range(p + 1, 9):
                if a[p, q] == 0:
                    continue
                th = (a[q, q] - a[p, p]) / (2 * a[p, q])
                s = (t(1) if th >= 0 else t(-1)) / (abs(th) + np.sqrt(th * th + 1))
                c = 1 / np.sqrt(s * s + 1)
                s = s * c
                for m in (a.T, a, e.T):
                    mp, mq = m[p].copy(), m[q].copy()
                    m[p], m[q] = c * mp - s * mq, s * mp + c * mq
    x = e[:, np.argmin(np.diag(a))]
    return x / np.sqrt((x * x).sum())


def _off(x, ref):
    x = np.asarray(x).reshape(9).astype(np.longdouble)
    x = x / np.sqrt((x * x).sum())
    return float(min(np.abs(x - ref).max(), np.abs(x + ref).max()))


@functools.lru_cache(None)
@np.errstate(over="ignore")  # a vanishing off-diagonal element: no rotation
def _expected(case):
    mids, offs, cal = _data(*case)
    ref = [_jacobi_null(mids, o, cal, np.longdouble) for o in offs]
    tol = 32 * max(_off(_jacobi_null(mids, o, cal, np.float64), r) for o, r in zip(offs, ref))
    return mids, offs, cal, ref, max(tol, 1e-13)


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"n{c[0]}_s{c[1]:g}_z{c[2]:g}_w{c[3]:g}_{c[4]}")
def test_exact_displacements_of_close_rois(case):
    mids, offs, cal, ref, tol = _expected(case)
    res = G.fit_deformation(mids, offs, None, cal, min_rois=MIN_ROIS)
    assert res["mask"].all()
    assert np.isfinite(res["F"]).all()
    errors = [_off(f, r) for f, r in zip(res["F"], ref)]
    assert max(errors) <= tol, (errors, tol)
