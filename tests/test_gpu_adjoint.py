"""GPU: the hand-written adjoint FMM (dL/dw for L = sum_i |B_i - B*_i|^2) through the C ABI
and the torch.autograd harness."""
import numpy as np
import pytest

from conftest import rel_l2, shell_sources

pytestmark = pytest.mark.gpu


def _case(seed=21, ns=6000, nt=1500):
    rng = np.random.default_rng(seed)
    src = shell_sources(rng, ns)
    w = rng.uniform(0.5, 1.5, ns)
    tgt = rng.uniform(-2, 2, (nt, 3))
    return rng, src, w, tgt


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-11), ("fp32", 2e-6), ("f16x3", 2e-6)])
def test_adjoint_is_the_transpose(precision, tol):
    """B is linear in w, so g.B(w) == w.(adjoint g) for every g and w (exact up to rounding,
    independent of the FMM truncation error)."""
    import torch
    from bachelors_amd.torch_fmm import FMMBiotSavart
    rng, src, w, tgt = _case()
    F = FMMBiotSavart(src, tgt, order=8, cap=32, precision=precision)
    wt = torch.tensor(w, dtype=torch.float64, device="cuda", requires_grad=True)
    B = F(wt)
    g = torch.tensor(rng.normal(size=(len(tgt), 3)), dtype=torch.float64, device="cuda")
    (B * g).sum().backward()
    lhs = float((B * g).sum())
    rhs = float((wt.detach() * wt.grad).sum())
    assert abs(lhs - rhs) <= tol * abs(lhs)


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-11), ("fp32", 2e-6), ("f16x3", 2e-6)])
def test_adjoint_is_the_transpose_p16(precision, tol):
    """The same identity at p = 16 (the order of the 4M workload; in F16X3 the forward runs the
    persistent M2L GEMM with the near field beside it), with g = B(w) (1 + U[-1/2, 1/2]) so that
    g.B(w) >= |B(w)|^2 / 2 and the quotient is not a random-sign cancellation."""
    import torch
    from bachelors_amd.torch_fmm import FMMBiotSavart
    rng, src, w, tgt = _case(23, ns=8000, nt=2000)
    F = FMMBiotSavart(src, tgt, order=16, cap=64, precision=precision)
    wt = torch.tensor(w, dtype=torch.float64, device="cuda", requires_grad=True)
    B = F(wt)
    g = B.detach() * (1 + torch.tensor(rng.uniform(-0.5, 0.5, (len(tgt), 3)), device="cuda"))
    (B * g).sum().backward()
    lhs = float((B * g).sum())
    rhs = float((wt.detach() * wt.grad).sum())
    assert abs(lhs - rhs) <= tol * abs(lhs)


def test_adjoint_gradient_vs_finite_differences_and_direct():
    import torch
    from bachelors_amd.torch_fmm import FMMBiotSavart
    from oracle import oracle as O
    rng, src, w, tgt = _case(22)
    wstar = w * (1 + 0.1 * (2 * rng.random(len(w)) - 1))
    F = FMMBiotSavart(src, tgt, order=10, cap=32, precision="fp64")
    with torch.no_grad():
        Bstar = F(torch.tensor(wstar, device="cuda"))
    wt = torch.tensor(w, dtype=torch.float64, device="cuda", requires_grad=True)
    loss = ((F(wt) - Bstar) ** 2).sum()
    loss.backward()
    grad = wt.grad.cpu().numpy()
    # central finite differences, h = 1e-3, on 64 seeded weights
    idx = rng.choice(len(w), 64, replace=False)
    fd = []
    with torch.no_grad():
        for j in idx:
            wp = w.copy(); wp[j] += 1e-3
            wm = w.copy(); wm[j] -= 1e-3
            lp = float(((F(torch.tensor(wp, device="cuda")) - Bstar) ** 2).sum())
            lm = float(((F(torch.tensor(wm, device="cuda")) - Bstar) ** 2).sum())
            fd.append((lp - lm) / 2e-3)
    fd = np.array(fd)
    assert rel_l2(grad[idx], fd) < 1e-5
    # the adjoint operator alone: the FMM residual r = B(w) - B* pulled back through the exact
    # transposed kernel, dL/dw_j = 2 sum_i r_i . (MU0/4pi) (J_j x (x_i - y_j)) / |x_i - y_j|^3
    with torch.no_grad():
        r = (F(torch.tensor(w, device="cuda")) - Bstar).cpu().numpy()
    J = np.stack([-src[:, 1], src[:, 0], np.zeros(len(src))], 1) / np.hypot(src[:, 0], src[:, 1])[:, None]
    gk = np.zeros(len(src))
    for j0 in range(0, len(src), 500):
        d = tgt[None, :, :] - src[j0:j0 + 500, None, :]                        # (j, i, 3)
        k = np.cross(np.broadcast_to(J[j0:j0 + 500, None, :], d.shape), d) / (np.linalg.norm(d, axis=2) ** 3)[..., None]
        gk[j0:j0 + 500] = 2 * np.einsum("jic,ic->j", k, r) * (1.2566370614e-6 / (4 * 3.14159265359))
    assert rel_l2(grad, gk) < 1e-5      # p = 10 truncation of the transposed FMM
    # against the FP64 direct-sum gradient of the same loss (direct-sum B and B*): the FMM error of
    # the residual (a tenth of B) enters here too
    Bs = O.direct_B(src, wstar, tgt)
    gd = O.direct_grad_w(src, w, tgt, Bs)
    assert rel_l2(grad, gd) < 1e-4


@pytest.mark.parametrize("ns,nt,cap_s,cap_t", [(2, 1, 2, 1), (700, 300, 4, 200), (700, 300, 300, 3), (65, 64, 64, 64),
                                               (5000, 129, 8, 128)])
def test_transposed_near_field_is_the_transpose(ns, nt, cap_s, cap_t):
    """The near field summed at the source leaves through their ancestors' close pairs: leaf
    capacities far apart (close source nodes are then internal, or targets' leaves much larger), single
    points, and one point per 64-lane block, by g.B(w) = w.B^T g with g = B(w) (1 + U[-1/2, 1/2])
    (FP64 rounding, as above)."""
    import ctypes

    import torch
    import bachelors_amd as fm
    rng = np.random.default_rng(31 + ns + nt)
    src = shell_sources(rng, ns)
    w = rng.uniform(0.5, 1.5, ns)
    tgt = rng.uniform(-1.2, 1.2, (nt, 3))
    F = fm.FMM(order=6, source_leaf_capacity=cap_s, target_leaf_capacity=cap_t, precision="fp64", frame=1)
    F.set_sources(src, w)
    F.set_targets(tgt)
    B = F.run(1.0)
    g = torch.from_numpy(B * (1 + rng.uniform(-0.5, 0.5, B.shape))).cuda()
    gw = torch.empty(ns, dtype=torch.float64, device="cuda")
    F.adjoint_weights_dev(1.0, ctypes.c_void_p(g.data_ptr()), ctypes.c_void_p(gw.data_ptr()))
    F.synchronize()
    lhs, rhs = float((B * g.cpu().numpy()).sum()), float((w * gw.cpu().numpy()).sum())
    assert F.stats()["close_pairs"] > 0
    F.close()
    assert abs(lhs - rhs) <= 1e-11 * abs(lhs)


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-11), ("fp32", 2e-6)])
@pytest.mark.parametrize("order", [1, 2, 4, 5, 6, 8, 9, 11, 13, 15, 17, 18, 20])
def test_transposed_m2l_at_every_row_padding(order, precision, tol):
    """The transposed M2L with rows padded to multiples of 16 (one kernel instance per block count) at
    orders of each count, with classes of a few to a few hundred columns, by the same identity."""
    import torch
    from bachelors_amd.torch_fmm import FMMBiotSavart
    rng, src, w, tgt = _case(40 + order, ns=1500, nt=900)
    F = FMMBiotSavart(src, tgt, order=order, cap=24, precision=precision)
    wt = torch.tensor(w, dtype=torch.float64, device="cuda", requires_grad=True)
    B = F(wt)
    g = B.detach() * (1 + torch.tensor(rng.uniform(-0.5, 0.5, (len(tgt), 3)), device="cuda"))
    (B * g).sum().backward()
    lhs = float((B.detach() * g).sum())
    rhs = float((wt.detach() * wt.grad).sum())
    assert F._fmm.stats()["far_pairs"] > 0
    assert abs(lhs - rhs) <= tol * abs(lhs)


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-11), ("fp32", 2e-6)])
def test_transposed_near_field_out_of_rows(precision, tol):
    """40,000 sources in some 64 leaves, each with 65,000 close targets in one leaf, ask for more rows of partial
    sums than there are: equal bits in every run (no far pairs), and the transpose as above."""
    import ctypes

    import torch
    import bachelors_amd as fm
    rng = np.random.default_rng(97)
    ns, nt = 40000, 65000
    F = fm.FMM(order=4, source_leaf_capacity=1000, target_leaf_capacity=nt + 2, precision=precision, frame=1)
    w = rng.uniform(0.5, 1.5, ns)
    F.set_sources(rng.uniform(-2.9, 2.9, (ns, 3)), w)
    F.set_targets(rng.uniform(-2.9, 2.9, (nt, 3)))
    B = F.run(1.0)
    st = F.stats()
    assert st["far_pairs"] == 0 and st["source_leaves"] > 32
    g = torch.from_numpy(B * (1 + rng.uniform(-0.5, 0.5, B.shape))).cuda()
    runs = []
    for _ in range(4):
        gw = torch.empty(ns, dtype=torch.float64, device="cuda")
        F.adjoint_weights_dev(1.0, ctypes.c_void_p(g.data_ptr()), ctypes.c_void_p(gw.data_ptr()))
        F.synchronize()
        runs.append(gw)
    F.close()
    assert all(torch.equal(runs[0], r) for r in runs)
    lhs, rhs = float((B * g.cpu().numpy()).sum()), float((w * runs[0].cpu().numpy()).sum())
    assert abs(lhs - rhs) <= tol * abs(lhs)
