"""Half storage of symmetric stencil matrices in CG solves.

A CG solve of a system over 16 MB of FP64 values on a slice-shared-offset
pattern reads only the values at offsets >= 0.  Row sums keep the CRS order
and the launches their workgroups, so whole solves give the bits of the
SELL-64 layout: for assembled matrices with Dirichlet rows (zero rows whose
columns stay), for symmetric Dirichlet elimination, for 3-DOF node blocks,
and for values that are not symmetric, which keep the full copy.
"""
import numpy as np
import pytest

from elmerfem_amd import _lib, workloads as W

pytestmark = pytest.mark.gpu

FORMS = [(_lib.FP64, _lib.FAITHFUL), (_lib.FP64, _lib.FAST), (_lib.MIXED_IR, _lib.FAST)]


def _solves_equal(s, kw, **how):
    out = []
    vals, rhs = s.values()
    for fmt in (_lib.SPMV_SELL_SHARED, _lib.SPMV_SELL):
        s.set_values(vals, rhs)  # scaling and back leaves them an ulp off
        s.spmv_set_format(fmt, 0)
        s.spmv_set_format(fmt, 1)
        out.append(s.solve(kw, **how))
    (x0, r0), (x1, r1) = out
    assert r0["info"] == r1["info"] == 1 and r0["iters"] == r1["iters"]
    assert r0["res_true"] == r1["res_true"]
    assert np.array_equal(x0, x1)
    return x0


# 45: just over the size limit and a ragged last slice; 48: a multiple of 16
@pytest.mark.parametrize("n", [45, 48])
@pytest.mark.parametrize("precision,mode", FORMS)
def test_poisson_equals_sell(ehip, n, precision, mode):
    w = W.poisson_hex8(n, sigma=1.0)
    s, _ = W.build_system(w)
    assert 8 * s.spmv_shared_layout()["entries"] >= 16 << 20
    _solves_equal(s, w["kw"], precision=precision, mode=mode)
    s.free()


@pytest.mark.parametrize("precision,mode", FORMS)
def test_tet4_symmetric_dirichlet_equals_sell(ehip, precision, mode):
    w = W.heat_tet4(53)
    w["kw"].symmetric = True
    s, _ = W.build_system(w)
    _solves_equal(s, w["kw"], precision=precision, mode=mode)
    s.free()


@pytest.mark.parametrize("precision,mode", FORMS)
def test_elasticity_equals_sell(ehip, precision, mode):
    w = W.elasticity_hex(22)
    s, _ = W.build_system(w)
    assert s.spmv_shared_layout()["node_block"] == 3
    _solves_equal(s, w["kw"], precision=precision, mode=mode, inner_tol=0.1)
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
    a = _solves_equal(s, w["kw"], mode=_lib.FAST)
    s.set_values(vals, rhs)
    b = _solves_equal(s, w["kw"], mode=_lib.FAST)
    assert not np.array_equal(a, b) and np.allclose(a, b, rtol=1e-6, atol=1e-12)
    s.free()
