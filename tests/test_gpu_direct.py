"""GPU: the FP64 direct sums at the edges of their blocks (64 targets, 4 sources, 1,024 sources per
range) and of their reciprocal powers (a target on a source, distances whose square leaves the range
of the fast path) against the oracle and the closed form of one source.

Tolerance: a pair term carries a few ulp and a sum of n <= 5,000 terms of one sign pattern at most
n ulp of its largest partial, 5,000 * 1.1e-16 = 5.5e-13; 1e-12 covers both."""
import ctypes

import numpy as np
import pytest

from conftest import rel_l2, shell_sources

pytestmark = pytest.mark.gpu


def _direct(fm, src, w, tgt, current=1.0):
    import torch
    F = fm.FMM(order=2, source_leaf_capacity=64, target_leaf_capacity=64)
    F.set_sources(src, w)
    F.set_targets(np.zeros((1, 3)))
    F.build_trees()
    x = torch.from_numpy(np.ascontiguousarray(tgt)).cuda()
    out = [torch.full_like(x, np.nan) for _ in range(2)]
    F.direct_B_dev(current, len(tgt), ctypes.c_void_p(x.data_ptr()), ctypes.c_void_p(out[0].data_ptr()))
    F.direct_A_dev(current, len(tgt), ctypes.c_void_p(x.data_ptr()), ctypes.c_void_p(out[1].data_ptr()))
    F.close()
    return [o.cpu().numpy() for o in out]


@pytest.mark.parametrize("ns,nt", [(1, 1), (3, 64), (4, 65), (5, 63), (1023, 7), (2047, 129), (2049, 1), (5000, 300)])
def test_direct_sums_at_block_edges(orc, ns, nt):
    import bachelors_amd as fm
    rng = np.random.default_rng(7000 + ns + nt)
    src = shell_sources(rng, ns)
    w = rng.uniform(0.5, 1.5, ns)
    tgt = rng.uniform(-2, 2, (nt, 3))
    tgt[nt // 2] = src[ns // 2]          # a target on a source: that pair adds nothing
    B, A = _direct(fm, src, w, tgt, current=2.0)
    if ns > 1:
        assert rel_l2(B, orc.direct_B(src, w, tgt, current=2.0)) < 1e-12
        assert rel_l2(A, orc.direct_A(src, w, tgt, current=2.0)) < 1e-12
    else:
        assert np.isfinite(B).all() and np.isfinite(A).all()
        if nt == 1:
            assert not B.any() and not A.any()


@pytest.mark.parametrize("d", [1e-101, 1e-99, 1e-3, 1e99, 1e101, 1e130])
def test_direct_sums_at_extreme_distances(d):
    """One source at (0, 1, 0) with current along -x; targets at distance d along z.  B = w d (1 / d^3)
    along the cross product, A = w / d, down to distances whose square or cube leaves the range of
    the fast reciprocal (2^-335 and 2^335 = 7e100); at 1e130 the cube is past the largest double and
    the formula in doubles gives 0."""
    import bachelors_amd as fm
    src, w = np.array([[0.0, 1.0, 0.0]]), np.array([1.0])
    B, A = _direct(fm, src, w, np.array([[0.0, 1.0, d]]), current=4 * 3.14159265359)
    assert abs(A[0, 0] + 1.0 / d) <= 1e-14 / d and A[0, 1] == 0 and A[0, 2] == 0
    # J x d = (-1, 0, 0) x (0, 0, d) = (0, d, 0)
    with np.errstate(over="ignore"):
        expect = 1.2566370614e-6 * d * (1.0 / (np.float64(d) * d * d))
    assert B[0, 0] == 0 and B[0, 2] == 0 and abs(B[0, 1] - expect) <= 1e-14 * abs(expect)
