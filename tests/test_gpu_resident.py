"""Resident CG and BiCGStab loops: a sequence in one launch, on systems of at
most 262 144 rows whose gathered vector fits the LDS.

A solve gives the launched loops' bits: profile_every, which samples
launches, keeps a solve on the launched loops, so the two are compared
directly -- iteration counts, residual histories and solutions -- in every
layout the loops read, at sizes around the 1024 rows of a workgroup and the
256 of a partial sum, and for every exit (convergence, iteration limit, a
tightened unscaled test).
"""
import hashlib
import json
import os

import numpy as np
import pytest

from elmerfem_amd import _lib, workloads as W
from elmerfem_amd.system import System

pytestmark = pytest.mark.gpu

FORMS = [(_lib.FP64, _lib.FAITHFUL), (_lib.FP64, _lib.FAST), (_lib.MIXED_IR, _lib.FAST)]


def _same(s, kw, **how):
    vals, rhs = s.values()
    out = []
    for every in (0, 1 << 30):
        s.set_values(vals, rhs)  # scaling and back leaves them an ulp off
        out.append(s.solve(kw, history=True, profile_every=every, **how))
    s.set_values(vals, rhs)
    (x0, r0), (x1, r1) = out
    for k in ("info", "iters", "outer_iters", "res_scaled", "res_true"):
        assert r0[k] == r1[k], (k, r0[k], r1[k])
    assert np.array_equal(r0["history"], r1["history"])
    assert np.array_equal(x0, x1)
    return r0


def _tridiagonal(n):
    i = np.arange(n)
    rows, cols, vals, diag = [1], [], [], []
    for r in range(n):
        for c in (r - 1, r, r + 1):
            if 0 <= c < n:
                if c == r:
                    diag.append(len(cols) + 1)
                cols.append(c + 1)
                vals.append(2.5 + 0.1 * np.sin(r) if c == r else -1.0)
        rows.append(len(cols) + 1)
    return (np.array(rows, np.int32), np.array(cols, np.int32), np.array(diag, np.int32), np.array(vals),
            1.0 + 0.5 * np.cos(i))


# one row, one slice, the edges of a partial sum's 256 and a workgroup's 1024
# rows, and one workgroup more
@pytest.mark.parametrize("n", [1, 2, 63, 65, 255, 257, 1023, 1024, 1025, 2049, 3100])
@pytest.mark.parametrize("precision,mode", FORMS)
def test_row_counts(ehip, n, precision, mode):
    rows, cols, diag, vals, b = _tridiagonal(n)
    s = System.from_csr(rows, cols, diag)
    s.set_values(vals, b)
    r = _same(s, W._kw("cg", "diagonal", 1e-10, 500), precision=precision, mode=mode)
    assert r["info"] == 1
    s.free()


@pytest.mark.parametrize("fmt", [_lib.SPMV_SELL_SHARED, _lib.SPMV_SELL])
@pytest.mark.parametrize("precision,mode", FORMS)
@pytest.mark.parametrize("name", ["hex8_17", "tet4_21", "hex8_40"])
def test_meshes(ehip, name, precision, mode, fmt):
    kind, n = name.split("_")
    w = W.poisson_hex8(int(n), sigma=1.0) if kind == "hex8" else W.heat_tet4(int(n))
    s, _ = W.build_system(w)
    s.spmv_set_format(fmt, 0)
    s.spmv_set_format(fmt, 1)
    for stop in (False, True):
        r = _same(s, w["kw"], precision=precision, mode=mode, true_residual_stop=stop)
        assert r["info"] == 1
    s.free()


@pytest.mark.parametrize("precision,mode", FORMS)
@pytest.mark.parametrize("maxit", [1, 2, 7])
def test_iteration_limit(ehip, precision, mode, maxit):
    w = W.poisson_hex8(13, sigma=1.0)
    s, _ = W.build_system(w)
    w["kw"].maxit = maxit
    r = _same(s, w["kw"], precision=precision, mode=mode)
    assert r["info"] == 2
    s.free()


# ... and the 2048, 4096 and 8192 rows of one, two and four tiles to each of
# the first eight workgroups, and one workgroup row more
@pytest.mark.parametrize("n", [1, 65, 257, 1025, 2048, 2049, 3100, 4097, 8192, 8193])
@pytest.mark.parametrize("mode", [_lib.FAITHFUL, _lib.FAST])
def test_bicgstab_row_counts(ehip, n, mode):
    rows, cols, diag, vals, b = _tridiagonal(n)
    vals = vals.copy()
    vals[cols == np.repeat(np.arange(n), np.diff(rows))] = -1.3  # lower entries: not symmetric
    s = System.from_csr(rows, cols, diag)
    s.set_values(vals, b)
    _same(s, W._kw("bicgstab", "diagonal", 1e-10, 500), mode=mode)
    s.free()


@pytest.mark.parametrize("fmt", [_lib.SPMV_SELL_SHARED, _lib.SPMV_SELL])
@pytest.mark.parametrize("precision,mode", FORMS)
@pytest.mark.parametrize("n", [20, 71])
def test_bicgstab_convdiff(ehip, n, precision, mode, fmt):
    w = W.convdiff_quad4(n, index=3)
    s, _ = W.build_system(w)
    s.spmv_set_format(fmt, 0)
    s.spmv_set_format(fmt, 1)
    for stop in (False, True):
        _same(s, w["kw"], precision=precision, mode=mode, true_residual_stop=stop)
    w["kw"].maxit = 3
    assert _same(s, w["kw"], precision=precision, mode=mode)["info"] == 2
    s.free()


with open(os.path.join(os.path.dirname(__file__), "golden", "bicgstab_convdiff.json")) as _f:
    BICGSTAB = json.load(_f)


@pytest.mark.parametrize("case", sorted(BICGSTAB))
@pytest.mark.parametrize("form", ["faithful", "fast", "mixed"])
def test_bicgstab_recorded_bits(ehip, case, form):
    """BiCGStab's answers are those of the launched loops before there were
    resident ones, recorded then: iterations, exit, residual and solution
    bits.  Near the s-norm exit (info 36: the true residual stalls above the
    tolerance) the solution follows the order of the partial sums by 1e-12
    to 1e-7, so comparing the two loops alone cannot tell that both moved.
    Both loops, Peclet numbers 45 and 89."""
    _, n, index = case.split("_")
    want = BICGSTAB[case]
    w = W.convdiff_quad4(int(n), index=int(index))
    s, _ = W.build_system(w)
    vals, rhs = s.values()
    assert hashlib.sha256(vals.tobytes()).hexdigest() == want["values"]
    precision, mode = dict(zip(("faithful", "fast", "mixed"), FORMS))[form]
    for every in (0, 1 << 30):
        s.set_values(vals, rhs)
        x, r = s.solve(w["kw"], precision=precision, mode=mode, profile_every=every)
        got = {"iters": r["iters"], "info": r["info"], "res_true": r["res_true"].hex(),
               "x": hashlib.sha256(x.tobytes()).hexdigest()}
        assert got == want[form], every
    s.free()


def test_largest_and_too_wide(ehip):
    """262 144 rows fill the grid; a bandwidth beyond the LDS keeps the
    launched loops (the same solve either way)."""
    for n in (262144, 262145):
        m = 512
        i = np.arange(n)
        near = [(-m, -1.0), (-1, -1.0), (0, 4.3), (1, -1.0), (m, -1.0)]
        c = np.stack([i + o for o, _ in near], 1)
        ok = (c >= 0) & (c < n)
        v = np.broadcast_to([x for _, x in near], c.shape)
        rows = np.concatenate([[1], 1 + np.cumsum(ok.sum(1))]).astype(np.int32)
        diag = (rows[:-1] + ok[:, :2].sum(1)).astype(np.int32)
        s = System.from_csr(rows, (c[ok] + 1).astype(np.int32), diag)
        s.set_values(v[ok].copy(), np.ones(n))
        r = _same(s, W._kw("cg", "diagonal", 1e-10, 500), mode=_lib.FAST)
        assert r["info"] == 1
        s.free()
