"""Half storage of symmetric stencil matrices in CG solves.

A launched CG solve of a large system on a slice-shared-offset pattern reads
only the values at offsets >= 0.  Row sums keep the CRS
order and the launches (of FP32 steps up to 1024 workgroups) their grid, so
whole solves give the bits of the SELL-64 layout: for assembled matrices with Dirichlet rows (zero rows whose
columns stay), for symmetric Dirichlet elimination, for 3-DOF node blocks,
and for values that are not symmetric, which keep the full copy.
"""
import ctypes as C

import numpy as np
import pytest

from elmerfem_amd import _lib, workloads as W
from elmerfem_amd.batch import Server
from elmerfem_amd.system import System
from conftest import launched_only

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _from_8_mb(monkeypatch):
    """By default the half storage takes the place of large copies only, which
    these tests need not have."""
    monkeypatch.setenv("EHIP_HALF_MIN_MB", "8")


FORMS = [(_lib.FP64, _lib.FAITHFUL), (_lib.FP64, _lib.FAST), (_lib.MIXED_IR, _lib.FAST)]


def _solves_equal(s, kw, half, **how):
    """half: which copies the solve on the shared-offset layout halves."""
    out = []
    vals, rhs = s.values()
    launched_only(s)  # resident loops read the full copy
    mixed = how.get("precision") == _lib.MIXED_IR
    for fmt in (_lib.SPMV_SELL_SHARED, _lib.SPMV_SELL):
        s.set_values(vals, rhs)  # scaling and back leaves them an ulp off
        s.spmv_set_format(fmt, 0)
        s.spmv_set_format(fmt, 1)
        out.append(s.solve(kw, **how))
        route = s.solve_route()
        assert route["half_storage"] & 3 == (half if fmt == _lib.SPMV_SELL_SHARED else 0)
        assert route["loops"] == (_lib.LOOP_RECORDED if mixed else _lib.LOOP_LAUNCHED)
    (x0, r0), (x1, r1) = out
    assert r0["info"] == r1["info"] == 1 and r0["iters"] == r1["iters"]
    assert r0["res_true"] == r1["res_true"]
    assert np.array_equal(x0, x1)
    return x0


# 45: a ragged last slice; 48: a multiple of 16;
# 64: more rows than the resident loops take, another ragged slice (not in
# mixed precision: more than 1024 workgroups group FP32 sums otherwise there)
@pytest.mark.parametrize("n,precision,mode", [(n, *f) for n in (45, 48, 64) for f in FORMS
                                              if n < 64 or f[0] == _lib.FP64])
def test_poisson_equals_sell(ehip, n, precision, mode):
    w = W.poisson_hex8(n, sigma=1.0)
    s, _ = W.build_system(w)
    _solves_equal(s, w["kw"], 3 if precision == _lib.MIXED_IR else 1, precision=precision, mode=mode)
    s.free()


@pytest.mark.parametrize("precision,mode", FORMS)
def test_tet4_symmetric_dirichlet_equals_sell(ehip, precision, mode):
    w = W.heat_tet4(53)
    w["kw"].symmetric = True
    s, _ = W.build_system(w)
    _solves_equal(s, w["kw"], 3 if precision == _lib.MIXED_IR else 1, precision=precision, mode=mode)
    s.free()


@pytest.mark.parametrize("precision,mode", FORMS)
def test_elasticity_equals_sell(ehip, precision, mode):
    w = W.elasticity_hex(22)
    s, _ = W.build_system(w)
    assert s.spmv_shared_layout()["node_block"] == 3
    _solves_equal(s, w["kw"], 0 if precision == _lib.MIXED_IR else 1, precision=precision, mode=mode, inner_tol=0.1)
    s.free()


def test_unsymmetric_values_keep_the_full_copy(ehip):
    """A convergent but not symmetric matrix (one off-diagonal entry changed
    by a relative 1e-9): the same bits in both layouts again, then the
    symmetric values once more."""
    w = W.poisson_hex8(45)
    s, _ = W.build_system(w)
    _, rows, _, _ = s.pattern()
    vals, rhs = s.values()
    r = (23 * 46 + 23) * 46 + 23  # an inner node; its first entry is not the diagonal
    changed = vals.copy()
    j = rows[r] - 1
    changed[j] *= 1.0 + 1e-9
    assert changed[j] != vals[j]
    s.set_values(changed, rhs)
    a = _solves_equal(s, w["kw"], 0, mode=_lib.FAST)
    s.set_values(vals, rhs)
    b = _solves_equal(s, w["kw"], 1, mode=_lib.FAST)
    assert not np.array_equal(a, b) and np.allclose(a, b, rtol=1e-6, atol=1e-12)
    s.free()


def _box27(nx, ny, nz):
    """27-point pattern of an nx x ny x nz node grid (1-based CRS), and
    values(seed): symmetric to the bit, diagonally dominant."""
    n = nx * ny * nz
    k, j, i = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    k, j, i = k.ravel(), j.ravel(), i.ravel()
    r = np.arange(n)
    off = [(c, b, a) for c in (-1, 0, 1) for b in (-1, 0, 1) for a in (-1, 0, 1)]
    ok = np.stack([(k + c >= 0) & (k + c < nz) & (j + b >= 0) & (j + b < ny) & (i + a >= 0) & (i + a < nx)
                   for c, b, a in off], 1)
    col = np.stack([r + (c * ny + b) * nx + a for c, b, a in off], 1)
    rows = np.concatenate([[1], 1 + np.cumsum(ok.sum(1))]).astype(np.int32)
    diag = (rows[:-1] + ok[:, :13].sum(1)).astype(np.int32)

    def values(seed):
        g = np.random.default_rng(seed).random(n)
        v = np.zeros(ok.shape)
        for q in range(27):
            if q != 13:
                lo, hi = np.minimum(r, col[:, q]) % n, np.maximum(r, col[:, q]) % n
                v[:, q] = np.where(ok[:, q], -(0.2 + g[lo] * g[hi]), 0.0)
        v[:, 13] = 0.02 + np.abs(v).sum(1)
        return v[ok]
    return rows, (col[ok] + 1).astype(np.int32), diag, values


@pytest.mark.parametrize("first", ["direct", "lane"])
def test_recorded_blocks_follow_the_copy_in_use(ehip, first):
    """A direct mixed solve reads the half storage, the same system's solve on
    a server's lane (at most 262 144 rows) the full copy; the bandwidth is
    beyond the resident loops', so both replay recorded blocks.  New values
    before every solve, the two kinds in turn: each is that of a system that
    was never solved before."""
    rows, cols, diag, values = _box27(136, 136, 14)
    n = len(rows) - 1
    kw = W._kw("cg", "diagonal", 1e-10, 2000)
    rhs = 1.0 + 0.5 * np.cos(np.arange(n))

    def solve(s, seed, how):
        s.set_values(values(seed), rhs)
        if how == "direct":
            x, rep = s.solve(kw, precision=_lib.MIXED_IR, mode=_lib.FAST)
            return x, rep
        srv = Server(kw, precision=_lib.MIXED_IR, max_slots=4)
        srv.set_lane(100000, 1)
        assert srv.submit(s)
        done = []
        while not done:
            done = srv.step()
        x = s.solution()
        srv.free()
        return x, done[0][1]

    kinds = ["direct", "lane"] if first == "direct" else ["lane", "direct"]
    s = System.from_csr(rows, cols, diag)
    for seed in range(4):
        x, rep = solve(s, seed, kinds[seed % 2])
        fresh = System.from_csr(rows, cols, diag)
        y, want = solve(fresh, seed, kinds[seed % 2])
        fresh.free()
        assert want["info"] == 1
        assert (rep["info"], rep["iters"], rep["outer_iters"]) == (1, want["iters"], want["outer_iters"]), seed
        assert np.array_equal(x, y), seed
    s.free()


def test_route_names_what_ran(ehip):
    """ehip_solve_route: 25^3 fits the resident loops (full copy); sampled
    solves launch; 274 625 rows replay recorded blocks of the half storage,
    or launch, in FP64, in HUTI's order; a zero right-hand side runs nothing."""
    small, large = W.poisson_hex8(25, sigma=1.0), W.poisson_hex8(64, sigma=1.0)
    s, _ = W.build_system(small)
    vals, rhs = s.values()
    for precision, mode in FORMS:
        for every, loops in ((0, _lib.LOOP_RESIDENT), (1 << 30, _lib.LOOP_LAUNCHED)):
            s.solve(small["kw"], precision=precision, mode=mode, profile_every=every)
            assert s.solve_route()["loops"] == loops and s.solve_route()["half_storage"] == 0
    s.solve(W._kw("cg", "ilu0", 1e-10, 500))
    assert s.solve_route()["loops"] == _lib.LOOP_LAUNCHED
    s.set_values(vals, 0.0 * rhs)
    s.solve(small["kw"])
    assert s.solve_route() == {"loops": 0, "half_storage": 0, "spmv_grid32": 0}
    s.free()
    s, _ = W.build_system(large)
    for precision, mode in FORMS:
        s.solve(large["kw"], precision=precision, mode=mode)
        mixed = precision == _lib.MIXED_IR
        assert s.solve_route()["loops"] == (_lib.LOOP_RECORDED if mixed else _lib.LOOP_LAUNCHED)
        assert s.solve_route()["half_storage"] == (3 if mixed else 1)
    s.free()


def test_fp32_workgroups_follow_the_copy_in_use(ehip):
    """The half storage's FP32 steps run on up to 2048 workgroups; values that
    are not symmetric and a pinned SELL-64 layout keep the 1024 those kernels
    are fastest with, and so the sums they always had.  274 625 rows make
    1080 workgroups."""
    w = W.poisson_hex8(64, sigma=1.0)
    s, _ = W.build_system(w)
    vals, rhs = s.values()
    unsym = vals.copy()
    unsym[s.pattern()[1][s.n // 2] - 1] *= 1.0 + 1e-6  # its first entry is not the diagonal
    got = []
    for v, fmt, half, grid in ((vals, _lib.SPMV_SELL_SHARED, 3, 1080), (unsym, _lib.SPMV_SELL_SHARED, 0, 1024),
                               (vals, _lib.SPMV_SELL, 0, 1024), (unsym, _lib.SPMV_SELL, 0, 1024),
                               (vals, _lib.SPMV_SELL_SHARED, 3, 1080)):
        s.spmv_set_format(fmt, 0)
        s.spmv_set_format(fmt, 1)
        for every in (0, 1 << 30):
            s.set_values(v, rhs)
            x, rep = s.solve(w["kw"], precision=_lib.MIXED_IR, mode=_lib.FAST, profile_every=every)
            assert rep["info"] == 1
            route = s.solve_route()
            assert (route["half_storage"] & 3, route["spmv_grid32"]) == (half, grid)
            got.append((x, rep["iters"]))
    for i, j in ((0, 1), (2, 3), (2, 6), (2, 7), (4, 5), (0, 8), (0, 9)):  # SELL-64 gives the full copy's bits
        assert got[i][1] == got[j][1] and np.array_equal(got[i][0], got[j][0]), (i, j)
    s.free()


@pytest.mark.parametrize("precision,mode", [(_lib.FP64, _lib.FAST), (_lib.MIXED_IR, _lib.FAST)])
@pytest.mark.parametrize("kind", ["scalar", "elastic"])
def test_unsymmetric_values_are_told_from_a_sample(ehip, kind, precision, mode):
    """Values that are symmetric to rounding only are told from a sample of the
    slices, never compared whole; a single unequal pair, wherever it lies,
    keeps the full copy, compared whole once and told from that slice's
    sample after.  Symmetric values in between take the half storage again:
    what happened before never decides."""
    w = W.poisson_hex8(64, sigma=1.0) if kind == "scalar" else W.elasticity_hex(22)
    how = dict(precision=precision, mode=mode, inner_tol=0.1)
    half = {("scalar", _lib.FP64): 1, ("scalar", _lib.MIXED_IR): 3, ("elastic", _lib.FP64): 1,
            ("elastic", _lib.MIXED_IR): 0}[kind, precision]
    s, _ = W.build_system(w)
    vals, rhs = s.values()
    _, rows, cols, _ = s.pattern()
    row = np.repeat(np.arange(s.n), np.diff(rows))
    off = (cols - 1 != row) & (np.abs(vals) > 1e-6)
    inner = np.bincount(row, off, s.n) > 0  # not a Dirichlet row
    pairs = np.nonzero(off & inner[row] & inner[cols - 1])[0]

    def halves(v, info=1):
        s.set_values(v, rhs)
        _, rep = s.solve(w["kw"], return_x=False, **how)
        assert rep["info"] == info
        return s.solve_route()["half_storage"]

    rounding = vals * (1.0 + 1e-7 * np.random.default_rng(4).random(len(vals)))
    assert halves(vals) == half
    for _ in range(2):
        assert halves(rounding) == 0
    assert halves(vals) == half
    for at in (0.013, 0.5, 0.77, 0.991):
        one = vals.copy()
        one[pairs[int(at * len(pairs))]] *= 1.0 + 1e-6
        assert halves(one) in ((0, 4) if half else (0,))
        assert halves(one) == 0
        assert halves(vals) == half
    # an entry without its mirror image (a zero there) shows only to the whole
    # comparison, or in the slice where that failed
    w["kw"].maxit = 2
    for at in (0.25, 0.6):
        one = vals.copy()
        one[pairs[int(at * len(pairs))]] = 0.0
        assert halves(one, 2) == (4 if half else 0)
        assert halves(one, 2) == 0
    assert halves(vals, 2) == half
    s.free()


def _fail_allocs(lo, hi, count):
    assert _lib.load().ehip_internal_fail_allocs(C.c_int64(lo), C.c_int64(hi), count) == 0


def test_solves_do_without_the_memory_of_a_faster_path(ehip):
    """Where there is no memory for the resident loops' buffers, the half
    storage's masks (system creation) or values, a solve runs as it would
    without them, to the same FP64 bits; and a half copy that the solve does
    not read gives way to the full copy it needs."""
    w = W.poisson_hex8(25, sigma=1.0)
    s, _ = W.build_system(w)
    vals, rhs = s.values()
    how = dict(precision=_lib.FP64, mode=_lib.FAST)
    x, _ = s.solve(w["kw"], profile_every=1 << 30, **how)  # all buffers but the resident loops'
    try:
        for expect in (_lib.LOOP_LAUNCHED, _lib.LOOP_RESIDENT):
            if expect == _lib.LOOP_LAUNCHED:
                _fail_allocs(72 * s.n, 1 << 40, 1)
            s.set_values(vals, rhs)
            y, rep = s.solve(w["kw"], **how)
            assert rep["info"] == 1 and s.solve_route()["loops"] == expect
            assert np.array_equal(x, y)
        s.free()

        w = W.poisson_hex8(64, sigma=1.0)
        masks = 8 * 27 * ((65 ** 3 + 63) // 64)
        _fail_allocs(masks, masks, 1)
        got = []
        for half in (0, 1):
            s, _ = W.build_system(w)
            _fail_allocs(0, 0, 0)
            vals, rhs = s.values()
            got.append(s.solve(w["kw"], **how)[0])
            assert s.solve_route()["half_storage"] == half
            if not half:
                s.free()
        assert np.array_equal(*got)
        # the full FP64 copy, wanted by BiCGStab, takes the place of the half one
        full = 8 * s.spmv_shared_layout()["entries"]
        before = s.device_bytes()
        _fail_allocs(full, full, 1)
        s.set_values(vals, rhs)
        _, rep = s.solve(W._kw("bicgstab", "diagonal", 1e-10, 3000), **how)
        assert rep["info"] == 1
        assert s.device_bytes() < before + full
        # and CG goes on with the full copy when the half one finds no memory
        _fail_allocs(full // 4, full, 1)
        s.set_values(vals, rhs)
        y, _ = s.solve(w["kw"], **how)
        assert s.solve_route()["half_storage"] == 0 and np.array_equal(y, got[0])
        s.set_values(vals, rhs)
        y, _ = s.solve(w["kw"], **how)
        assert s.solve_route()["half_storage"] == 1 and np.array_equal(y, got[0])
        s.free()
    finally:
        _fail_allocs(0, 0, 0)


def test_half_storage_ends_with_the_solve(ehip):
    """The engine reports on its full copies, whatever a direct solve before
    allowed: after one that left early (zero right-hand side) a batched solve
    of a system over the size limit allocates no half copy."""
    from elmerfem_amd.batch import solve_batch
    w = W.poisson_hex8(64, sigma=1.0)
    held = []
    for before in (False, True):
        s, _ = W.build_system(w)
        vals, rhs = s.values()
        s.set_values(vals, 0.0 * rhs)
        s.solve(w["kw"] if before else W._kw("bicgstab"))
        s.set_values(vals, rhs)
        _, reps, _ = solve_batch([s], w["kw"], mode=_lib.FAST)
        assert reps[0]["info"] == 1
        held.append(s.device_bytes())
        s.free()
    assert held[0] == held[1]


@pytest.mark.parametrize("kind,n,half64,half_mixed", [("hex8", 64, 0, 0), ("hex8", 80, 0, 2), ("hex8", 92, 1, 3),
                                                      ("elastic", 40, 0, 0), ("elastic", 50, 1, 0)])
def test_sizes_that_take_the_half_storage(ehip, monkeypatch, kind, n, half64, half_mixed):
    """FP64 copies from 150 MB on (224 MB with node blocks), FP32 copies from
    48 MB on: 64^3 Hex8 has 59 and 30 MB, 80^3 114 and 57, 92^3 172 and 86;
    40^3 elasticity 131 MB in FP64, 50^3 253."""
    monkeypatch.delenv("EHIP_HALF_MIN_MB")
    w = W.poisson_hex8(n) if kind == "hex8" else W.elasticity_hex(n)
    w["kw"].maxit = 2
    s, _ = W.build_system(w)
    for precision, half in ((_lib.FP64, half64), (_lib.MIXED_IR, half_mixed)):
        s.solve(w["kw"], precision=precision, mode=_lib.FAST, return_x=False)
        assert s.solve_route()["half_storage"] == half
    s.free()
