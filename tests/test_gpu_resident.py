"""Resident CG and BiCGStab loops: a sequence in one launch, on systems of at
most 262 144 rows whose gathered vector fits the LDS.

A solve gives the launched loops' bits: profile_every, which samples
launches, keeps a solve on the launched loops, so the two are compared
directly -- iteration counts, residual histories and solutions -- in every
layout the loops read, at sizes around the 1024 rows of a workgroup and the
256 of a partial sum, and for every exit (convergence, iteration limit, a
tightened unscaled test).
"""
import ctypes as C
import hashlib
import json
import os
import threading
import time

import numpy as np
import pytest

from elmerfem_amd import _lib, workloads as W
from elmerfem_amd.batch import Server
from elmerfem_amd.system import System

pytestmark = pytest.mark.gpu

FORMS = [(_lib.FP64, _lib.FAITHFUL), (_lib.FP64, _lib.FAST), (_lib.MIXED_IR, _lib.FAST)]


def _same(s, kw, loops=_lib.LOOP_RESIDENT, **how):
    vals, rhs = s.values()
    out = []
    for every in (0, 1 << 30):
        s.set_values(vals, rhs)  # scaling and back leaves them an ulp off
        out.append(s.solve(kw, history=True, profile_every=every, **how))
        assert s.solve_route()["loops"] == (_lib.LOOP_LAUNCHED if every else loops)
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
    loops = _lib.LOOP_RESIDENT
    if n in (2, 65):  # padded to whole slices by too much for a layout that they read
        loops = _lib.LOOP_RECORDED if precision == _lib.MIXED_IR else _lib.LOOP_LAUNCHED
    r = _same(s, W._kw("cg", "diagonal", 1e-10, 500), precision=precision, mode=mode, loops=loops)
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
# the first eight workgroups, and one row more
@pytest.mark.parametrize("n", [1, 65, 257, 1025, 2048, 2049, 3100, 4097, 8192, 8193])
@pytest.mark.parametrize("mode", [_lib.FAITHFUL, _lib.FAST])
def test_bicgstab_row_counts(ehip, n, mode):
    rows, cols, diag, vals, b = _tridiagonal(n)
    vals = vals.copy()
    vals[cols == np.repeat(np.arange(n), np.diff(rows))] = -1.3  # lower entries: not symmetric
    s = System.from_csr(rows, cols, diag)
    s.set_values(vals, b)
    _same(s, W._kw("bicgstab", "diagonal", 1e-10, 500), mode=mode,
          loops=_lib.LOOP_LAUNCHED if n == 65 else _lib.LOOP_RESIDENT)
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


def test_largest(ehip):
    """262 144 rows fill the grid; one more keeps the launched loops (the same
    solve either way)."""
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
        r = _same(s, W._kw("cg", "diagonal", 1e-10, 500), mode=_lib.FAST,
                  loops=_lib.LOOP_RESIDENT if n == 262144 else _lib.LOOP_LAUNCHED)
        assert r["info"] == 1
        s.free()


# FP64: two windows of 1024 rows and the bandwidth on both sides, or one, in
# what the 156 KB leave beside 25 KB of sums; BiCGStab's windows are of 256
# rows, four of them
@pytest.mark.parametrize("method,mode,fits,too_wide", [("cg", _lib.FAITHFUL, 3640, 3720), ("cg", _lib.FAST, 7840, 7920),
                                                       ("bicgstab", _lib.FAITHFUL, 900, 940),
                                                       ("bicgstab", _lib.FAST, 1950, 1990)])
def test_bandwidth_beyond_the_lds(ehip, method, mode, fits, too_wide):
    for h, loops in ((fits, _lib.LOOP_RESIDENT), (too_wide, _lib.LOOP_LAUNCHED)):
        n = 20000
        i = np.arange(n)
        near = [(-h, -1.0), (-1, -1.0), (0, 4.3), (1, -1.0), (h, -1.0)]
        c = np.stack([i + o for o, _ in near], 1)
        ok = (c >= 0) & (c < n)
        v = np.broadcast_to([x for _, x in near], c.shape)
        rows = np.concatenate([[1], 1 + np.cumsum(ok.sum(1))]).astype(np.int32)
        diag = (rows[:-1] + ok[:, :2].sum(1)).astype(np.int32)
        s = System.from_csr(rows, (c[ok] + 1).astype(np.int32), diag)
        s.set_values(v[ok].copy(), np.ones(n))
        assert _same(s, W._kw(method, "diagonal", 1e-10, 500), loops=loops, mode=mode)["info"] == 1
        s.free()


def _resident(s, mode):
    assert _lib.load().ehip_internal_resident(s._h, C.c_int(mode)) == 0


@pytest.mark.parametrize("precision,mode", FORMS)
@pytest.mark.parametrize("method", ["cg", "bicgstab"])
def test_a_grid_that_gave_up(ehip, method, precision, mode):
    """A grid told that one of its threads gave up commits nothing: the
    launched loop (in the mixed CG, recorded blocks) goes on from unchanged
    vectors to the same bits.  The device's next solves do not try again,
    until the rest is over (here: ended by the test)."""
    w = W.poisson_hex8(14, sigma=1.0) if method == "cg" else W.convdiff_quad4(60, index=3)
    s, _ = W.build_system(w)
    vals, rhs = s.values()
    plain = _lib.LOOP_RECORDED if (method, precision) == ("cg", _lib.MIXED_IR) else _lib.LOOP_LAUNCHED
    out = []
    for test, loops in ((0, _lib.LOOP_RESIDENT), (2, _lib.LOOP_GAVE_UP | plain), (None, plain),
                        (0, _lib.LOOP_RESIDENT), (1, plain), (0, _lib.LOOP_RESIDENT)):
        if test is not None:
            _resident(s, test)
        s.set_values(vals, rhs)
        x, r = s.solve(w["kw"], precision=precision, mode=mode, history=True)
        assert s.solve_route()["loops"] == loops
        out.append((x, r))
    for x, r in out[1:]:
        assert (r["info"], r["iters"], r["outer_iters"]) == tuple(out[0][1][k] for k in ("info", "iters", "outer_iters"))
        assert np.array_equal(r["history"], out[0][1]["history"]) and np.array_equal(x, out[0][0])
    s.free()


@pytest.mark.parametrize("precision,mode", FORMS)
@pytest.mark.parametrize("method", ["cg", "bicgstab"])
def test_launches_that_stop_between_iterations(ehip, method, precision, mode):
    """A launch runs a number of iterations at most and the next goes on from
    the state it left: with launches of one iteration each a solve gives the
    same history and bits, whether it converges or meets its limit."""
    w = W.poisson_hex8(14, sigma=1.0) if method == "cg" else W.convdiff_quad4(60, index=3)
    s, _ = W.build_system(w)
    vals, rhs = s.values()
    for maxit in (10000, 5):
        w["kw"].maxit = maxit
        out = []
        for test in (0, 3):
            _resident(s, test)
            s.set_values(vals, rhs)
            out.append(s.solve(w["kw"], precision=precision, mode=mode, history=True, true_residual_stop=True))
            assert s.solve_route()["loops"] == _lib.LOOP_RESIDENT
        (x0, r0), (x1, r1) = out
        for k in ("info", "iters", "outer_iters", "res_scaled", "res_true"):
            assert r0[k] == r1[k], (k, r0[k], r1[k])
        assert np.array_equal(r0["history"], r1["history"]) and np.array_equal(x0, x1)
    s.free()


def test_none_beside_launched_work(ehip):
    """While a server holds a request, a direct solve takes turns with it launch
    by launch, to the same bits; before and after, it runs resident."""
    w = W.poisson_hex8(14, sigma=1.0)
    s, _ = W.build_system(w)
    vals, rhs = s.values()
    t, _ = W.build_system(W.heat_tet4(9))
    srv = Server(w["kw"], precision=_lib.MIXED_IR, max_slots=4)
    got = []
    for loops in (_lib.LOOP_RESIDENT, _lib.LOOP_LAUNCHED, _lib.LOOP_RESIDENT):
        if loops == _lib.LOOP_LAUNCHED:
            assert srv.submit(t)
        s.set_values(vals, rhs)
        got.append(s.solve(w["kw"], mode=_lib.FAST)[0])
        assert s.solve_route()["loops"] == loops
        if loops == _lib.LOOP_LAUNCHED:
            done = []
            while not done:
                done = srv.step()
            assert done[0][1]["info"] == 1
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])
    srv.free()
    s.free()
    t.free()


def test_several_threads(ehip):
    """Solves of four host threads: resident loops of small systems run side by
    side, not one after another, and larger ones (201 workgroups) leave the
    chip to everyone; each solve gives the bits it gives alone."""
    for n, share in ((17, 0.75), (58, None)):
        ws = [W.poisson_hex8(n, sigma=1.0, seed=11 + i) for i in range(4)]
        ss = [W.build_system(w)[0] for w in ws]
        kw, how = ws[0]["kw"], dict(precision=_lib.FP64, mode=_lib.FAITHFUL)
        start = [s.values() for s in ss]
        got = {}

        def work(i, rounds):
            for k in range(rounds):
                x, r = ss[i].solve(kw, **how)
                got.setdefault(i, []).append((k, r["iters"], x.tobytes(), ss[i].solve_route()["loops"]))

        def together(threads):
            th = [threading.Thread(target=work, args=(i, 6)) for i in range(4)]
            t0 = time.perf_counter()
            for t in th:
                t.start()
                if not threads:
                    t.join()
            for t in th:
                t.join()
            return time.perf_counter() - t0

        times, runs = {True: [], False: []}, []
        for threads in (False, True, True, False):
            got.clear()
            for s, (v, b) in zip(ss, start):
                s.set_values(v, b)
            times[threads].append(together(threads))
            runs.append({i: [g[:3] for g in got[i]] for i in got})
            if n == 17 or not threads:
                assert all(g[3] == _lib.LOOP_RESIDENT for i in got for g in got[i])
        assert all(r == runs[0] for r in runs[1:])
        if share:
            assert min(times[True]) < share * min(times[False]), times
        for s in ss:
            s.free()
