"""GPU: the treecode walk that a workgroup of 64 points shares, at the edges of its blocks and of the
sorted path, and at every order against the truncation bound of the direct sum."""
import ctypes

import numpy as np
import pytest

from conftest import rel_l2, shell_sources

pytestmark = pytest.mark.gpu


def _solver(order, src, w, J=None, cap=16, precision="fp64"):
    import bachelors_amd as fm
    F = fm.FMM(order=order, source_leaf_capacity=cap, target_leaf_capacity=64, precision=precision)
    F.set_sources(src, w, J)
    F.set_targets(np.zeros((1, 3)))
    F.build_trees()
    F.upward()
    return F


@pytest.mark.parametrize("m", [1, 63, 64, 65, 1024, 1025, 3001])
def test_points_do_not_depend_on_their_company(m):
    """Points among and around the sources in one call (above 1,024: served in sorted order) equal the same
    points served one by one or in tens: each point meets the same nodes in the same order, with the same
    operations, whatever its workgroup opens (only the rounding of nothing: equal bits)."""
    rng = np.random.default_rng(m)
    src = shell_sources(rng, 3000)
    F = _solver(8, src, np.full(3000, 1.0 / 3000))
    x = rng.uniform(-2.5, 2.5, (m, 3))
    B, A = F.treecode(x, 3.0)
    step = 1 if m <= 65 else 10
    pick = range(0, m, step) if m <= 1025 else range(0, m, 97)
    for i in pick:
        b, a = F.treecode(x[i:i + step], 3.0)
        assert np.array_equal(b, B[i:i + step]) and np.array_equal(a, A[i:i + step])
    F.close()


@pytest.mark.parametrize("order", range(1, 21))
def test_every_order_within_the_truncation_bound(orc, order):
    """Currents along x (no cancellation in A_x): a box of radius R seen from d > 2 R has a relative
    truncation error of at most (R/d)^(p+1) d / (d - R) < 2 * 2^-(p+1) in A; 1e-12 for the rounding."""
    rng = np.random.default_rng(200 + order)
    src = shell_sources(rng, 400)
    w = rng.uniform(0.5, 1.5, 400)
    J = np.tile([1.0, 0.0, 0.0], (400, 1))
    d = rng.normal(size=(100, 3))
    x = d / np.linalg.norm(d, axis=1)[:, None] * rng.uniform(6, 40, (100, 1))
    F = _solver(order, src, w, J)
    B, A = F.treecode(x, 2.0)
    F.close()
    direct = orc.direct_A(src, w, x, J=J, current=2.0)
    assert rel_l2(A, direct) < 2 * 0.5 ** (order + 1) + 1e-12
    assert np.isfinite(B).all()
    if order == 20:
        assert rel_l2(B, orc.direct_B(src, w, x, J=J, current=2.0)) < 40 * 2 * 0.5 ** 21
