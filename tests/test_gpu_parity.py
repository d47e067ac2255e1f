"""GPU parity: the HIP library (through its C ABI) against the CPU oracle on the same
seeded inputs.  Integer work (trees, lists) must match bit for bit; floating point to
the tolerance written in each test."""
import numpy as np
import pytest

from conftest import gap_overlap_targets, rel_l2, shell_sources

pytestmark = pytest.mark.gpu

SHARED_ROOT = (np.zeros(3), np.full(3, 3.0))


@pytest.fixture(scope="module")
def fm():
    import bachelors_amd
    bachelors_amd.lib()
    return bachelors_amd


def _inputs(seed, ns, nt, kind="shell"):
    rng = np.random.default_rng(seed)
    src = shell_sources(rng, ns)
    w = np.full(ns, 1.0 / ns)
    if kind == "uniform":
        tgt = rng.uniform(-2, 2, (nt, 3))
    else:
        tgt = np.concatenate([rng.uniform(-2, 2, (nt // 2, 3)), shell_sources(rng, nt - nt // 2)])
    return src, w, tgt


def _boundary_targets(orc, tgt, cap, rng, nadd=400):
    """Targets placed exactly on child-box faces of the reference (bounding-box) target
    tree: exercises half-open containment and the float-rounded one-ulp gaps/overlaps."""
    T = orc.target_tree(tgt, cap)
    sub = np.nonzero(T.first_child >= 0)[0]
    pts = []
    for _ in range(nadd):
        b = sub[rng.integers(len(sub))]
        ch = T.first_child[b] + rng.integers(8)
        c, h = T.center[ch], T.half[ch]
        p = c + rng.uniform(-1, 1, 3) * h
        ax = rng.integers(3)
        p[ax] = c[ax] + (h[ax] if rng.random() < 0.5 else -h[ax])
        pts.append(p)
    return np.concatenate([tgt, np.array(pts)])


def _cmp_tree(g, o):
    assert len(g["level"]) == len(o.level)
    for k in ("level", "parent", "first_child", "begin", "end", "npts"):
        assert np.array_equal(g[k], getattr(o, k)), k
    assert np.array_equal(g["center"], o.center)
    assert np.array_equal(g["slots"], o.slots)


@pytest.mark.parametrize("frame", [0, 1])
def test_trees_bit_exact(fm, orc, frame):
    rng = np.random.default_rng(7)
    src, w, tgt = _inputs(3, 20000, 6000)
    if frame == 0:
        tgt = _boundary_targets(orc, tgt, 24, rng)
    F = fm.FMM(order=4, source_leaf_capacity=20, target_leaf_capacity=24, frame=frame)
    F.set_sources(src, w)
    F.set_targets(tgt)
    F.build_trees()
    _cmp_tree(F.tree(0), orc.source_tree(src, 20))
    _cmp_tree(F.tree(1), orc.target_tree(tgt, 24, root=SHARED_ROOT if frame == 1 else None))
    assert F.stats()["source_tree_sorted"] == 1


def test_trees_bit_exact_float_gaps_and_overlaps(fm, orc):
    """Reference frame: targets inside one-ulp gaps/overlaps of float-rounded sibling boxes are
    dropped or inserted twice, as by the reference's pointer insertion (level-by-level build)."""
    rng = np.random.default_rng(23)
    src, w, tgt = _inputs(3, 8000, 6000)
    tgt, nadd = gap_overlap_targets(orc, tgt, 24, rng)
    F = fm.FMM(order=4, source_leaf_capacity=20, target_leaf_capacity=24, frame=0)
    F.set_sources(src, w)
    F.set_targets(tgt)
    F.build_trees()
    _cmp_tree(F.tree(1), orc.target_tree(tgt, 24))
    assert F.stats()["target_tree_sorted"] == 0


def test_trees_bit_exact_lattice_faces_and_deep_cluster(fm, orc):
    """Shared frame: targets exactly on child faces (the half-open lattice boxes tile exactly,
    so the one-sort build applies) and a source cluster deeper than 10 levels (63-bit paths)."""
    rng = np.random.default_rng(17)
    src, w, tgt = _inputs(5, 12000, 3000)
    src = np.concatenate([src, 0.3 + rng.uniform(-1e-5, 1e-5, (3000, 3))])
    w = np.full(len(src), 1.0 / len(src))
    h = 3.0 / 2 ** rng.integers(1, 7, 500)            # faces of the shared lattice, levels 1..6
    faces = rng.uniform(-2, 2, (500, 3))
    ax = rng.integers(3, size=500)
    faces[np.arange(500), ax] = np.round(faces[np.arange(500), ax] / h) * h
    tgt = np.concatenate([tgt, faces])
    F = fm.FMM(order=4, source_leaf_capacity=20, target_leaf_capacity=24, frame=1)
    F.set_sources(src, w)
    F.set_targets(tgt)
    F.build_trees()
    S = orc.source_tree(src, 20)
    assert S.level.max() > 10
    _cmp_tree(F.tree(0), S)
    _cmp_tree(F.tree(1), orc.target_tree(tgt, 24, root=SHARED_ROOT))
    st = F.stats()
    assert st["source_tree_sorted"] == 1 and st["target_tree_sorted"] == 1


@pytest.mark.parametrize("max_depth", [1, 3, 5])
def test_trees_bit_exact_depth_capped(fm, orc, max_depth):
    """A depth cap leaves nodes above the leaf capacity unsplit."""
    src, w, tgt = _inputs(11, 20000, 6000)
    F = fm.FMM(order=4, source_leaf_capacity=20, target_leaf_capacity=24, frame=1, max_depth=max_depth)
    F.set_sources(src, w)
    F.set_targets(tgt)
    F.build_trees()
    S = orc.source_tree(src, 20, max_depth=max_depth)
    assert S.level.max() == max_depth
    _cmp_tree(F.tree(0), S)
    _cmp_tree(F.tree(1), orc.target_tree(tgt, 24, root=SHARED_ROOT, max_depth=max_depth))


def _grown_root(tgt):
    """The shared frame's target root: the source root doubled along its lattice until it holds the targets."""
    sc = 1.0
    while True:
        j = np.maximum(np.ceil((-3.0 - tgt.min(0)) / 6.0), 0.0)
        lo = -3.0 - 6.0 * j
        if np.all(j <= sc - 1) and np.all(tgt.max(0) < lo + 6.0 * sc):
            return lo + 3.0 * sc, np.full(3, 3.0 * sc)
        sc *= 2


@pytest.mark.parametrize("ns,nt,cap", [(1, 1, 20), (2, 255, 2), (256, 257, 2), (300, 121, 20), (1025, 1023, 3),
                                       (2048, 2049, 5000), (4095, 4096, 20), (4096, 4095, 64), (4096, 4097, 2)])
def test_small_trees_bit_exact(fm, orc, ns, nt, cap):
    """Trees of up to 4,096 points take one launch; at the edges of its sorts (powers of 2 from 256), of
    the mirror it returns (2,048 nodes) and of the range itself the tree is the oracle's."""
    src, w, tgt = _inputs(40 + ns, ns, nt)
    tgt[::7] *= 1.6   # some of them outside the source root
    F = fm.FMM(order=4, source_leaf_capacity=cap, target_leaf_capacity=cap, frame=1)
    F.set_sources(src, w)
    F.set_targets(tgt)
    F.build_trees()
    print(F.stats()["source_nodes"], F.stats()["target_nodes"], flush=True)
    _cmp_tree(F.tree(0), orc.source_tree(src, cap))
    _cmp_tree(F.tree(1), orc.target_tree(tgt, cap, root=_grown_root(tgt)))


def test_small_trees_what_the_one_launch_build_leaves(fm, orc):
    """Points in gaps and overlaps of the float-rounded boxes, a cluster deeper than 10 levels, a depth
    cap, targets far from the sources and sources that are all or in part outside the root give the
    oracle's tree at these sizes too."""
    rng = np.random.default_rng(29)
    src, w, tgt = _inputs(6, 2000, 1500)
    gap, _ = gap_overlap_targets(orc, tgt, 24, rng)
    deep = np.concatenate([src, 0.3 + rng.uniform(-1e-5, 1e-5, (600, 3))])
    assert len(gap) <= 4096
    for frame, s, t, depth in ((0, src, gap, None), (1, deep, tgt, None), (1, src, tgt, 2), (1, src, tgt + 50.0, None),
                               (1, src + 50.0, tgt, None), (1, 3.2 * src, tgt, None)):
        kw = {} if depth is None else dict(max_depth=depth)
        F = fm.FMM(order=4, source_leaf_capacity=20, target_leaf_capacity=24, frame=frame, **kw)
        F.set_sources(s, np.full(len(s), 1.0 / len(s)))
        F.set_targets(t)
        F.build_trees()
        _cmp_tree(F.tree(0), orc.source_tree(s, 20, **kw))
        _cmp_tree(F.tree(1), orc.target_tree(t, 24, root=_grown_root(t) if frame == 1 else None, **kw))
        assert F.stats()["target_tree_sorted"] == (0 if t is gap else 1)


@pytest.mark.parametrize("frame", [0, 1])
def test_interaction_lists_bit_exact(fm, orc, frame):
    src, w, tgt = _inputs(4, 12000, 4000)
    F = fm.FMM(order=4, source_leaf_capacity=24, target_leaf_capacity=24, frame=frame)
    F.set_sources(src, w)
    F.set_targets(tgt)
    F.build_trees()
    S = orc.source_tree(src, 24)
    T = orc.target_tree(tgt, 24, root=SHARED_ROOT if frame == 1 else None)
    (oft, ofs), (oct_, ocs) = orc.interaction_lists(S, T)
    F.leaf_expansions()
    F.upward()
    F.downward()
    (ft, fs), (ct, cs), ncls = F.lists()
    assert (ncls > 0) == (frame == 1)
    assert set(zip(ft.tolist(), fs.tolist())) == set(zip(oft.tolist(), ofs.tolist()))
    assert set(zip(ct.tolist(), cs.tolist())) == set(zip(oct_.tolist(), ocs.tolist()))
    assert len(ft) == len(oft) and len(ct) == len(oct_)


def _class_codes(S, T, ft, fs):
    """(level difference, centre offset in units of the finer box half size) of each far pair,
    from the oracle's trees, as one sortable integer."""
    hf = np.minimum(S.half[fs, 0], T.half[ft, 0])
    off = np.rint((S.center[fs] - T.center[ft]) / hf[:, None]).astype(np.int64) + 128
    d = (S.level[fs] - T.level[ft]).astype(np.int64) + 32
    return (d << 24) | (off[:, 0] << 16) | (off[:, 1] << 8) | off[:, 2]


@pytest.mark.parametrize("near_uniform", [True, False])
def test_far_pairs_class_order(fm, orc, near_uniform):
    """Shared frame: far pairs come sorted by (class, target) and the class count matches the
    distinct (level difference, offset) codes.  Uniform targets as dense as the sources give
    level differences up to 2 and offsets up to 15 finer half sizes; few targets around a
    thin shell give level differences up to 4 and offsets up to 51."""
    if near_uniform:
        src, w, tgt = _inputs(6, 16000, 16000, kind="uniform")
        caps = capt = 32
    else:
        src, w, tgt = _inputs(6, 12000, 4000)
        caps, capt = 20, 24
    F = fm.FMM(order=4, source_leaf_capacity=caps, target_leaf_capacity=capt, frame=1)
    F.set_sources(src, w)
    F.set_targets(tgt)
    F.build_trees()
    S = orc.source_tree(src, caps)
    T = orc.target_tree(tgt, capt, root=SHARED_ROOT)
    (oft, ofs), _ = orc.interaction_lists(S, T)
    F.leaf_expansions()
    F.upward()
    F.downward()
    (ft, fs), _, ncls = F.lists()
    code = _class_codes(S, T, oft, ofs)
    order = np.lexsort((oft, code))
    assert np.array_equal(ft, oft[order]) and np.array_equal(fs, ofs[order])
    assert ncls == len(np.unique(code))
    d = (code >> 24) - 32
    o = np.stack([(code >> 16) & 255, (code >> 8) & 255, code & 255], 1) - 128
    assert (d.max(), np.abs(o).max()) == ((2, 15) if near_uniform else (4, 51))


@pytest.mark.parametrize("kind", [0, 1, 2])
@pytest.mark.parametrize("p", [4, 12])
def test_operator_tables_fp64(fm, orc, kind, p):
    rng = np.random.default_rng(kind * 10 + p)
    deg = np.array([int(np.sqrt(i)) for i in range((p + 1) ** 2)])
    for _ in range(3):
        if kind == 1:
            t = rng.uniform(-3, 3, 3) + np.array([4.0, 0, 0])
            si, so = 0.5, 1.0
        else:
            t = rng.uniform(-0.5, 0.5, 3)
            si, so = (0.25, 0.5) if kind == 0 else (0.5, 0.25)
        G = fm.make_operator(kind, p, t, si, so, 1)
        T = orc.operator(kind, p, t, orc.CORRECTED)
        if kind == 0:
            E = T * (si ** deg[None, :]) / (so ** deg[:, None])
        elif kind == 2:
            E = T * (so ** (deg[:, None] + 1.0)) / (si ** (deg[None, :] + 1.0))
        else:
            E = T * (so ** (deg[:, None] + 1.0)) * (si ** deg[None, :])
        # 1e-10: the oracle keeps the reference's truncated 1/sqrt2 (math.hpp:16)
        assert np.abs(G - E).max() <= 1e-10 * np.abs(E).max()


def _oracle_run(orc, src, w, tgt, p, caps, cap_t, flags=None):
    return orc.FMMRun(src, w, tgt, p=p, cap_s=caps, cap_t=cap_t, flags=orc.CORRECTED if flags is None else flags,
                      target_root=SHARED_ROOT)


def _gpu_run(fm, src, w, tgt, p, caps, cap_t, precision):
    F = fm.FMM(order=p, source_leaf_capacity=caps, target_leaf_capacity=cap_t, precision=precision, frame=1)
    F.set_sources(src, w)
    F.set_targets(tgt)
    B = F.run(1.0)
    return F, B


@pytest.fixture(scope="module")
def small_case(orc):
    src, w, tgt = _inputs(11, 4096, 1500)
    R = _oracle_run(orc, src, w, tgt, 8, 32, 32)
    return src, w, tgt, R


def test_expansions_fp64(fm, orc, small_case):
    src, w, tgt, R = small_case
    F, _ = _gpu_run(fm, src, w, tgt, 8, 32, 32, "fp64")
    S = orc.source_tree(src, 32)
    T = orc.target_tree(tgt, 32, root=SHARED_ROOT)
    checked = 0
    for b in range(0, len(S.level), max(1, len(S.level) // 40)):
        if S.first_child[b] < 0 and S.npts[b] == 0:
            continue
        Mo = R.multipole(b)
        Mg = F.expansion(0, b)
        assert np.abs(Mg - Mo).max() <= 1e-9 * max(np.abs(Mo).max(), 1e-300)
        checked += 1
    for b in range(0, len(T.level), max(1, len(T.level) // 40)):
        if T.first_child[b] < 0 and T.npts[b] == 0:
            continue
        Lo = R.local(b)
        Lg = F.expansion(1, b)
        if np.abs(Lo).max() == 0:
            assert np.abs(Lg).max() == 0
        else:
            assert np.abs(Lg - Lo).max() <= 1e-9 * np.abs(Lo).max()
        checked += 1
    assert checked > 20


@pytest.mark.parametrize("p", [1, 2, 9, 20])
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-9), ("fp32", 1e-5), ("bf16x3", 1e-4)])
def test_local_expansions_of_the_short_m2l(fm, orc, p, precision, tol):
    """M2L tables with l + lambda <= p (m2l_full = 0), whole rows and padding, at the smallest and largest
    orders: a node's largest coefficient to 1e-9 in FP64 (as test_expansions_fp64), 100 units of the last
    place in FP32 and as much above it with bf16 splits (2^-16 a factor) as in the tests of B."""
    src, w, tgt = _inputs(31, 3000, 800)
    R = orc.FMMRun(src, w, tgt, p=p, cap_s=32, cap_t=32, flags=orc.SECTORAL_FIX | orc.FACT_FIX, target_root=SHARED_ROOT)
    F = fm.FMM(order=p, source_leaf_capacity=32, target_leaf_capacity=32, precision=precision, frame=1, m2l_full=0)
    F.set_sources(src, w)
    F.set_targets(tgt)
    F.run(1.0)
    T = orc.target_tree(tgt, 32, root=SHARED_ROOT)
    checked = 0
    for b in range(0, len(T.level), max(1, len(T.level) // 40)):
        if T.first_child[b] < 0 and T.npts[b] == 0:
            continue
        Lo = R.local(b)
        assert np.abs(F.expansion(1, b) - Lo).max() <= tol * np.abs(Lo).max()
        checked += 1
    assert checked > 10


# measured: fp32 2.2e-7, bf16x3 9.6e-7, f16x3 2.1e-7
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-10), ("fp32", 1e-6), ("bf16x3", 1e-5), ("f16x3", 1e-6)])
def test_B_matches_oracle(fm, orc, small_case, precision, tol):
    src, w, tgt, R = small_case
    F, B = _gpu_run(fm, src, w, tgt, 8, 32, 32, precision)
    Bo = R.B_input_order(len(tgt))
    assert np.all(np.isfinite(B))
    assert rel_l2(B, Bo) < tol
    Bf, Bn = F.B_parts()
    assert rel_l2(Bn, R.Bnear) < (1e-12 if precision == "fp64" else 1e-6)
    assert rel_l2(Bf, R.Bfar) < tol * 10


@pytest.mark.parametrize("ns,nt,cap", [(511, 3, 8), (1023, 130, 100), (2500, 65, 64), (9000, 65, 100), (9000, 1, 500)])
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("fp32", 1e-6)])
def test_near_field_of_few_leaves(fm, orc, ns, nt, cap, precision, tol):
    """Few target leaves: their close lists are shared by 1 to 16 workgroups, some without a chunk."""
    rng = np.random.default_rng(ns + nt)
    src = shell_sources(rng, ns)
    w = rng.uniform(0.5, 1.5, ns) / ns
    tgt = shell_sources(rng, nt)
    R = _oracle_run(orc, src, w, tgt, 3, cap, cap)
    F = fm.FMM(order=3, source_leaf_capacity=cap, target_leaf_capacity=cap, precision=precision, frame=1)
    F.set_sources(src, w)
    F.set_targets(tgt)
    F.run(1.0)
    assert np.abs(R.Bnear).max() > 0
    assert rel_l2(F.B_parts()[1], R.Bnear) < tol


@pytest.mark.parametrize("p", [1, 8, 12, 13, 14, 16, 18, 20])
def test_f16x3_with_and_without_groups(fm, p):
    """The F16X3 M2L over groups of far pairs (uniform points: many pairs per class) and over single pairs
    (few per class) against FP64 on the same trees: 1e-6, as against the oracle."""
    rng = np.random.default_rng(p)
    for n, grouped in ((30000, True), (1500, False)):
        src, tgt = rng.uniform(-2.9, 2.9, (n, 3)), rng.uniform(-2.9, 2.9, (n, 3))
        w = rng.uniform(0.5, 1.5, n) / n
        B = {}
        for precision in ("fp64", "f16x3"):
            F = fm.FMM(order=p, source_leaf_capacity=32, target_leaf_capacity=32, precision=precision, frame=1)
            F.set_sources(src, w)
            F.set_targets(tgt)
            F.run(1.0)
            B[precision] = F.B_parts()[0]
            st = F.stats()
            F.close()
        assert (st["far_pairs"] >= (128 if 14 <= p <= 18 else 1024) * st["m2l_classes"]) == grouped
        assert rel_l2(B["f16x3"], B["fp64"]) < 1e-6


def test_direct_sum_gpu_vs_oracle(fm, orc):
    import ctypes
    src, w, tgt = _inputs(12, 3000, 500)
    F = fm.FMM(order=4, source_leaf_capacity=32, target_leaf_capacity=32)
    F.set_sources(src, w)
    F.set_targets(tgt)
    F.build_trees()
    Bo = orc.direct_B(src, w, tgt, current=2.0)
    import torch
    t = torch.from_numpy(tgt).cuda()
    out = torch.zeros_like(t)
    F.direct_B_dev(2.0, len(tgt), ctypes.c_void_p(t.data_ptr()), ctypes.c_void_p(out.data_ptr()))
    assert rel_l2(out.cpu().numpy(), Bo) < 1e-13


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-10), ("fp32", 3e-6)])
def test_reference_frame_fmm_matches_oracle(fm, orc, precision, tol):
    """The whole FMM on the reference's own trees (bounding-box target root, float-rounded
    centres, per-pair M2L/L2L operators) against the oracle on the same trees."""
    src, w, tgt = _inputs(13, 3000, 800)
    F = fm.FMM(order=8, source_leaf_capacity=32, target_leaf_capacity=32, precision=precision, frame=0)
    F.set_sources(src, w)
    F.set_targets(tgt)
    B = F.run(1.0)
    R = orc.FMMRun(src, w, tgt, p=8, cap_s=32, cap_t=32, flags=orc.CORRECTED)
    Bf, Bn = F.B_parts()
    assert rel_l2(Bf + Bn, R.Bfar + R.Bnear) < tol
    Bo = R.B_input_order(len(tgt))
    ok = np.isfinite(Bo[:, 0])
    assert np.array_equal(np.isfinite(B[:, 0]), ok)
    assert rel_l2(B[ok], Bo[ok]) < tol


@pytest.mark.parametrize("p", [1, 2, 11, 20])
def test_reference_frame_orders_match_oracle(fm, orc, p):
    """The per-pair translations at the smallest and largest orders (3 and 231 outputs (l, m >= 0) over
    256 threads) and at a padded row length; M2L workgroups take 4 pairs, destinations end anywhere.  FP64
    to 1e-10 (the oracle's 10-digit 1/sqrt 2), the 32-bit expansions to 3e-6."""
    src, w, tgt = _inputs(14, 2000, 601)
    R = orc.FMMRun(src, w, tgt, p=p, cap_s=32, cap_t=32, flags=orc.CORRECTED)
    Bo = R.B_input_order(len(tgt))
    ok = np.isfinite(Bo[:, 0])
    for precision, tol in (("fp64", 1e-10), ("fp32", 3e-6), ("f16x3", 3e-6)):
        print("order", p, precision, flush=True)
        F = fm.FMM(order=p, source_leaf_capacity=32, target_leaf_capacity=32, precision=precision, frame=0)
        F.set_sources(src, w)
        F.set_targets(tgt)
        B = F.run(1.0)
        assert F.stats()["far_pairs"] > 100
        assert np.array_equal(np.isfinite(B[:, 0]), ok)
        assert rel_l2(B[ok], Bo[ok]) < tol
        F.close()


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-13), ("fp32", 1e-6), ("f16x3", 1e-6)])
def test_fused_run_matches_staged_run(fm, precision, tol):
    """fmm_run_B_dev (lists and near field on a side stream) equals the stage-by-stage calls; the
    only difference allowed is the order of the atomic M2M additions on narrow levels."""
    import torch
    src, w, tgt = _inputs(21, 20000, 6000)
    F = fm.FMM(order=8, source_leaf_capacity=32, target_leaf_capacity=32, precision=precision, frame=1)
    F.set_sources(src, w)
    F.set_targets(tgt)
    B_staged = F.run(1.0)
    out = torch.empty((len(tgt), 3), dtype=torch.float64, device="cuda")
    for _ in range(2):
        F.run_B_dev(1.0, out.data_ptr())
        F.synchronize()
        assert rel_l2(out.cpu().numpy(), B_staged) < tol


@pytest.mark.parametrize("ns,nt,cap", [(700, 1, 8), (1023, 130, 100), (9000, 1, 500), (60000, 273, 100), (100003, 40, 8),
                                       (60000, 30000, 8)])
def test_fused_near_field_takes_every_item(fm, ns, nt, cap):
    """The fused near field at p = 14 (two grids on one counter) sums every item: from one item to more than the
    grids' workgroups, its results are those of the stage-by-stage near field, bit for bit (parts of a leaf and
    the order of their sums follow from the lists), in every call."""
    import torch
    src, w, tgt = _inputs(ns + nt, ns, nt)
    F = fm.FMM(order=14, source_leaf_capacity=cap, target_leaf_capacity=cap, precision="f16x3", frame=1)
    F.set_sources(src, w)
    F.set_targets(tgt)
    F.run(1.0)
    near = F.B_parts()[1]
    assert np.abs(near).max() > 0
    out = torch.empty((nt, 3), dtype=torch.float64, device="cuda")
    for _ in range(3):
        F.run_B_dev(1.0, out.data_ptr())
        F.synchronize()
        assert np.array_equal(F.B_parts()[1], near)


@pytest.mark.parametrize("nt", [1, 255, 257, 32767, 32768, 70001])
def test_target_extent_on_device_equals_host(fm, nt):
    """The target tree of the reference frame (root = the targets' bounding box) is the same from a host
    array (extent by the host loop below 32,768 points) and from a device pointer (extent by a kernel),
    bit for bit, with NaN coordinates and coordinates of one sign among the targets."""
    import ctypes

    import torch
    rng = np.random.default_rng(nt)
    tgt = rng.uniform(0.5, 2, (nt, 3)) * [1, -1, 1]
    if nt > 300:
        tgt[rng.integers(1, nt, 5), rng.integers(0, 3, 5)] = np.nan
    trees = []
    d = torch.from_numpy(tgt).cuda()
    for dev in (False, True):
        F = fm.FMM(order=2, source_leaf_capacity=8, target_leaf_capacity=50)
        F.set_sources(np.array([[1.0, 0.0, 0.0]]), np.array([1.0]))
        if dev:
            F.set_targets_dev(nt, ctypes.c_void_p(d.data_ptr()))
        else:
            F.set_targets(tgt)
        F.build_trees()
        trees.append(F.tree(1))
        F.close()
    for k in trees[0]:
        assert np.array_equal(trees[0][k], trees[1][k]), k


def _far_part(fm, precision, p, src, w, tgt, **kw):
    F = fm.FMM(order=p, source_leaf_capacity=32, target_leaf_capacity=32, precision=precision, frame=1, **kw)
    F.set_sources(src, w)
    F.set_targets(tgt)
    F.run(1.0)
    far, st = F.B_parts()[0], F.stats()
    F.close()
    return far, st


@pytest.mark.parametrize("p", [8, 12, 14, 16, 17, 18])
def test_f16x3_groups_beside_a_strong_leaf(fm, p):
    """One source leaf of 2^20 times the weight: where it is no far pair, its siblings' groups keep the
    accuracy of their own columns.  Targets whose far field of the strong leaf alone is exactly zero, against
    FP64 on the same trees: 1e-6, as against the oracle."""
    rng = np.random.default_rng(50 + p)
    n = 30000
    src, tgt = rng.uniform(-2.9, 2.9, (n, 3)), rng.uniform(-2.9, 2.9, (n, 3))
    strong = np.all((src > 0) & (src < 0.375), axis=1)   # a box of the tree's fourth level, around 8 points
    assert strong.sum() > 3
    w = rng.uniform(0.5, 1.5, n) / n
    w[strong] *= 2.0 ** 20
    only, _ = _far_part(fm, "fp64", p, src, np.where(strong, w, 0.0), tgt)
    sel = np.all(only == 0, axis=1)
    assert sel.sum() > 20
    exact, st = _far_part(fm, "fp64", p, src, w, tgt)
    far, _ = _far_part(fm, "f16x3", p, src, w, tgt)
    assert st["far_pairs"] >= 1024 * st["m2l_classes"]   # groups at every order
    assert rel_l2(far[sel], exact[sel]) < 1e-6


@pytest.mark.parametrize("p", [1, 2, 4, 9, 12, 14, 16, 17, 18])
def test_f16x3_groups_of_the_short_m2l(fm, p):
    """M2L with l + lambda <= p over groups: the operators of some children have rows of zeros (an offset in a
    lattice plane) where their siblings' have none.  Local expansions against FP64 on the same trees: 1e-6, as B
    against the oracle."""
    rng = np.random.default_rng(70 + p)
    n = 30000
    src, tgt = rng.uniform(-2.9, 2.9, (n, 3)), rng.uniform(-2.9, 2.9, (n, 3))
    local = {}
    for precision in ("fp64", "f16x3"):
        F = fm.FMM(order=p, source_leaf_capacity=32, target_leaf_capacity=32, precision=precision, frame=1, m2l_full=0)
        F.set_sources(src, np.full(n, 1.0 / n))
        F.set_targets(tgt)
        F.run(1.0)
        st = F.stats()
        local[precision] = np.array([F.expansion(1, b) for b in range(0, st["target_nodes"], st["target_nodes"] // 300)])
        F.close()
    assert st["far_pairs"] >= 1024 * st["m2l_classes"]
    assert rel_l2(local["f16x3"], local["fp64"]) < 1e-6


def test_near_field_sums_few_terms_in_fp32(fm):
    """One leaf of 64 targets and sources of which one in 64 is 2^25 times the others: a weak term after a strong one
    is below half a unit of the sum's last place.  Runs of 8 FP32 terms lose 4 2^-25 of a strong term each on
    average, 1.2e-7, runs of 64 about 32 2^-25, 9.5e-7; the pairs' own roundings (some 5 units of 2^-24 each, of both
    signs) average out to less than 2e-7 over the 64 strong sources.  5e-7 against FP64."""
    rng = np.random.default_rng(90)
    n = 4096
    src = rng.uniform(0.4, 0.6, (n, 3))
    w = np.where(np.arange(n) % 64 == 0, 1.0, 2.0 ** -25)[rng.permutation(n)]
    J = np.tile([1.0, 0.0, 0.0], (n, 1))
    tgt = rng.uniform(-0.6, -0.4, (64, 3))
    near = {}
    for precision in ("fp64", "fp32"):
        F = fm.FMM(order=4, source_leaf_capacity=5000, target_leaf_capacity=64, precision=precision, frame=1)
        F.set_sources(src, w, J)
        F.set_targets(tgt)
        F.run(1.0)
        near[precision] = F.B_parts()[1]
        F.close()
    assert rel_l2(near["fp32"], near["fp64"]) < 5e-7


@pytest.mark.parametrize("order,precision,tol", [(4, "fp64", 1e-12), (4, "fp32", 1e-6), (14, "f16x3", 1e-6)])
@pytest.mark.parametrize("cap_t", [50000, 1000])
def test_near_field_out_of_rows(fm, order, precision, tol, cap_t):
    """40,000 targets, each with 65,000 close sources in one leaf, ask for 31 rows of partial sums a target, more
    than there are: the lists are cut into fewer parts, the same in every run (equal bits), for one leaf and for
    some 64 (in F16X3 taken from a queue).  Against the direct sum in FP64: no far pairs, so rounding alone."""
    import ctypes

    import torch
    rng = np.random.default_rng(95)
    ns, nt = 65000, 40000
    F = fm.FMM(order=order, source_leaf_capacity=ns + 2, target_leaf_capacity=cap_t, precision=precision, frame=1)
    src = torch.from_numpy(shell_sources(rng, ns)).cuda()
    w = torch.from_numpy(rng.uniform(0.5, 1.5, ns)).cuda()
    tgt = torch.from_numpy(rng.uniform(-2.9, 2.9, (nt, 3))).cuda()
    B, exact = torch.empty_like(tgt), torch.empty_like(tgt)
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    torch.cuda.synchronize()
    F.set_sources_dev(ns, ptr(src), ptr(w), None)
    F.set_targets_dev(nt, ptr(tgt))
    runs = []
    for _ in range(4):
        F.run_B_dev(1.0, ptr(B))
        F.synchronize()
        runs.append(B.clone())
    st = F.stats()
    assert st["far_pairs"] == 0 and (st["target_leaves"] == 1) == (cap_t == 50000)
    F.direct_B_dev(1.0, nt, ptr(tgt), ptr(exact))
    F.synchronize()
    F.close()
    assert all(torch.equal(runs[0], r) for r in runs)
    assert rel_l2(runs[0].cpu().numpy(), exact.cpu().numpy()) < tol


def test_evaluation_replayed_from_a_graph(fm):
    """fmm_evaluate_B_dev captured into a graph on the caller's stream (nothing allocated, no wait): every
    replay equals the eager evaluation, with eager evaluations in between."""
    import ctypes

    import torch
    rng = np.random.default_rng(96)
    src, tgt = shell_sources(rng, 20000), rng.uniform(-2, 2, (3001, 3))
    out = torch.empty((3001, 3), dtype=torch.float64, device="cuda")
    ref = torch.empty_like(out)
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    s = torch.cuda.Stream()
    F = fm.FMM(order=4, source_leaf_capacity=64, target_leaf_capacity=64, frame=1)
    F.set_stream(ctypes.c_void_p(s.cuda_stream))
    F.set_sources(src, np.full(20000, 1.0 / 20000))
    F.set_targets(tgt)
    F.build_trees()
    F.leaf_expansions()
    F.upward()
    F.downward()
    F.evaluate_B_dev(1.0, ptr(ref))
    F.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        F.evaluate_B_dev(1.0, ptr(out))
    for _ in range(4):
        out.zero_()
        ref.zero_()
        torch.cuda.synchronize()
        F.evaluate_B_dev(1.0, ptr(ref))
        F.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref) and float(out.abs().max()) > 0
    F.close()


@pytest.mark.parametrize("p", [1, 2, 7, 20])
@pytest.mark.parametrize("full", [0, 1])
def test_m2l_operator_tables(fm, orc, p, full):
    """The M2L tables that the evaluations use, at orders of one and of many slices of rows, with
    l + lambda <= p and <= 2 p, off and in the lattice planes (rows of zeros): 1e-10, as above."""
    flags = orc.CORRECTED if full else orc.SECTORAL_FIX | orc.FACT_FIX
    deg = np.array([int(np.sqrt(i)) for i in range((p + 1) ** 2)])
    for t in ([3.5, -1.5, 2.5], [4.0, 0.0, -2.0], [0.0, 0.0, 5.0]):
        si, so = 0.5, 1.0
        G = fm.make_operator(1, p, np.array(t), si, so, full)
        E = orc.operator(1, p, np.array(t), flags) * (so ** (deg[:, None] + 1.0)) * (si ** deg[None, :])
        assert np.abs(G - E).max() <= 1e-10 * np.abs(E).max()


@pytest.mark.parametrize("p", [8, 13, 14, 16, 18])
def test_f16x3_groups_with_wide_keys(fm, orc, p):
    """A tight cluster whose boxes of levels 11 and 12 are far pairs of target leaves of level 4 (its place and
    the boxes that hold it lie just outside twice the radius of the leaf at (0.1875, 0.1875, 0.1875)): offsets beyond
    the compact class code, so all pairs and groups are keyed by the wide codes.  The far field of all targets and
    of that leaf's against FP64 on the same trees: 1e-6, as above."""
    rng = np.random.default_rng(99)
    n, m = 30000, 2000
    box = np.array([-0.37792969, -0.07910156, -0.00292969])
    src = np.concatenate([rng.uniform(-2.9, 2.9, (n, 3)), box + rng.uniform(-2, 2, (m, 3)) * 3 / 1024])
    tgt = rng.uniform(-2.9, 2.9, (n, 3))
    tgt[:20] = 0.1875 + 0.18 * rng.uniform(-1, 1, (20, 3))
    S, T = orc.source_tree(src, 32), orc.target_tree(tgt, 32, root=SHARED_ROOT)
    ft, fs = orc.interaction_lists(S, T)[0]
    unit = 3.0 / 2.0 ** np.maximum(S.level[fs], T.level[ft])
    wide = (np.abs(S.center[fs] - T.center[ft]).max(axis=1) / unit > 127.5)
    families = len(np.unique(np.column_stack([ft, S.parent[fs]])[wide], axis=0))
    assert families > 20 and wide.sum() > 2 * families   # groups of several wide pairs
    w = np.full(n + m, 1.0 / n)
    exact, st = _far_part(fm, "fp64", p, src, w, tgt)
    far, _ = _far_part(fm, "f16x3", p, src, w, tgt)
    assert st["far_pairs"] == len(ft) and st["far_pairs"] >= 300 * st["m2l_classes"]
    assert rel_l2(far, exact) < 1e-6
    hit = np.unique(ft[wide])
    sel = np.concatenate([np.arange(T.begin[t], T.end[t]) for t in hit if T.first_child[t] < 0])
    assert len(sel) > 10 and rel_l2(far[sel], exact[sel]) < 1e-6


@pytest.mark.parametrize("ns,nt,cap_t", [(1024, 60, 64), (1025, 60, 64), (16385, 33, 16), (20000, 129, 200)])
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("fp32", 1e-6)])
def test_near_field_at_the_limits_of_parts(fm, orc, ns, nt, cap_t, precision, tol):
    """The largest problem without parts and the smallest with them, and lists longer than 32 parts of 512
    sources (few leaves): near field against the oracle."""
    rng = np.random.default_rng(ns + nt)
    src = shell_sources(rng, ns)
    w = rng.uniform(0.5, 1.5, ns) / ns
    tgt = shell_sources(rng, nt)
    R = _oracle_run(orc, src, w, tgt, 3, ns + 2, cap_t)
    F = fm.FMM(order=3, source_leaf_capacity=ns + 2, target_leaf_capacity=cap_t, precision=precision, frame=1)
    F.set_sources(src, w)
    F.set_targets(tgt)
    F.run(1.0)
    assert F.stats()["source_leaves"] == 1 and F.stats()["target_leaves"] < 20
    assert rel_l2(F.B_parts()[1], R.Bnear) < tol


def test_m2l_blocks(fm):
    """The slab blocks of the M2L: the far pairs, in F16X3 the (target, source parent) families where pairs are
    grouped and the pairs where they are not; none in the reference frame."""
    rng = np.random.default_rng(120)
    for n, grouped in ((30000, True), (1500, False)):
        src, tgt = rng.uniform(-2.9, 2.9, (n, 3)), rng.uniform(-2.9, 2.9, (n, 3))
        for precision, frame in (("fp64", 1), ("f16x3", 1), ("fp64", 0)):
            F = fm.FMM(order=8, source_leaf_capacity=32, target_leaf_capacity=32, precision=precision, frame=frame)
            F.set_sources(src, np.full(n, 1.0 / n))
            F.set_targets(tgt)
            with pytest.raises(fm.FMMError):
                F.m2l_blocks()
            F.run(1.0)
            (ft, fs), _, _ = F.lists()
            families = len(np.unique(np.column_stack([ft, F.tree(0)["parent"][fs]]), axis=0))
            expect = 0 if frame == 0 else families if precision == "f16x3" and grouped else len(ft)
            assert F.m2l_blocks() == expect
            F.close()


@pytest.mark.parametrize("p", [8, 14])
def test_f16x3_groups_add_no_rounding(fm, p):
    """Clusters with currents of any direction (nothing cancels by symmetry), enough pairs a class for groups: a
    child's own accumulator takes 3 roundings per 32 products, the FP32 mode's M2L 8, and every other stage of the
    far field is the same FP32 one, so F16X3 is the closer of the two to FP64.  Its error is 0.85 to 0.90 of the
    FP32 mode's pair by pair; one accumulator through up to 8 children brings it to 0.98 at p = 14."""
    rng = np.random.default_rng(140 + p)
    ns, nt = 500000, 400000
    centre, sigma = rng.uniform(-1, 1, (64, 3)), rng.uniform(0.01, 0.1, (64, 3))
    k, kt = rng.integers(0, 64, ns), rng.integers(0, 64, nt)
    src, tgt = centre[k] + sigma[k] * rng.normal(size=(ns, 3)), centre[kt] + sigma[kt] * rng.normal(size=(nt, 3))
    J = rng.normal(size=(ns, 3))
    J /= np.linalg.norm(J, axis=1)[:, None]
    w = rng.uniform(0.5, 1.5, ns) / ns
    far = {}
    for precision in ("fp64", "fp32", "f16x3"):
        F = fm.FMM(order=p, source_leaf_capacity=48, target_leaf_capacity=48, precision=precision, frame=1, max_depth=10)
        F.set_sources(src, w, J)
        F.set_targets(tgt)
        F.run(1.0)
        far[precision] = F.B_parts()[0]
        st, blocks = F.stats(), F.m2l_blocks()
        F.close()
    assert blocks < st["far_pairs"] / 3
    ratio = rel_l2(far["f16x3"], far["fp64"]) / rel_l2(far["fp32"], far["fp64"])
    print("p", p, "error against the FP32 mode's", ratio, flush=True)
    assert ratio < 0.93
