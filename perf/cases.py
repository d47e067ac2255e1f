"""The work that programs have this library do, as cases that a benchmark can run.

Every case goes through the public Python entry points (bachelors_amd.FMM, FastMultipoleSolver,
torch_fmm.FMMBiotSavart).  Kinds:

  field      the fused evaluation of B at the targets from device tensors (run_B_dev)
  moving     the same for a program whose sources and targets move: new positions, then B
  training   B(w) and dL/dw of a squared-error loss through the torch harness
  potential  the stage-by-stage calls, then B and the vector potential A on the same expansions
  dropin     FastMultipoleSolver as a caller of the reference uses it: host arrays in, the whole
             sequence of its methods with its default frame and FP64, host array out
  bem        the same for Problem.BEM
  treecode   the single-point treecode B and A of a coil at many points
  direct     the FP64 direct sum at some of the targets of a large problem

The mixed mode (f16x3) and FP32 carry about seven digits through FP32 expansions, so programs that
choose them keep the field in float32; FP64 results stay float64.
"""
import ctypes
import math

import torch

import bachelors_amd as fm

MU0 = 1.2566370614e-6      # the constants that scale B and A in the reference (math.hpp:12-13)
PI = 3.14159265359
PROBE = 4096               # targets of the large cases that the direct sum in 64 bits is taken at
EXACT_PAIRS = 1.2e11       # direct sums in 64 bits up to here take some seconds


def listed():
    return [
        # the headline workload: four coaxial coils of opposite currents, as many targets as sources
        dict(name="field_4m_p16_mixed", kind="field", geometry="shells", ns=4194304, nt=4194304, order=16, cap=64,
             depth=21, precision="f16x3"),
        # one coil at the size and order of the benchmark's second workload
        dict(name="field_1m_p12_mixed", kind="field", geometry="shell", ns=1048576, nt=1048576, order=12, cap=64,
             depth=21, precision="f16x3"),
        # the same coil in the plain FP64 mode, the accuracy baseline that users check against
        dict(name="field_1m_p12_fp64", kind="field", geometry="shell", ns=1048576, nt=1048576, order=12, cap=64,
             depth=21, precision="fp64"),
        # time stepping: clustered particles with currents of any direction, new positions in each
        # step, ragged counts, deep trees
        dict(name="moving_clusters_p14_mixed", kind="moving", geometry="clusters", ns=999983, nt=750019, order=14,
             cap=48, depth=10, precision="f16x3"),
        # fitting current weights to a measured field: forward, loss, backward
        dict(name="training_clusters_p14_mixed", kind="training", geometry="clusters", ns=262147, nt=131101,
             order=14, cap=48, depth=10, precision="f16x3"),
        # the vector potential and the field of one set of expansions, in FP32
        dict(name="potential_250k_p10_fp32", kind="potential", geometry="shells", ns=250000, nt=250007, order=10,
             cap=48, depth=21, precision="fp32"),
        # the CPU reference's own case (32,768 coil points, 4,096 targets, p = 10, leaf capacity 32)
        dict(name="field_32k_p10_fp64", kind="field", geometry="shell", ns=32768, nt=4096, order=10, cap=32,
             depth=21, precision="fp64"),
        # the smallest call: a few hundred points, where launches and waits are all there is
        dict(name="field_300_p10_fp64", kind="field", geometry="shell", ns=300, nt=121, order=10, cap=32,
             depth=21, precision="fp64"),
        # the reference's torus coil (38,400 quadrature points) with the reference's default leaf capacities
        dict(name="dropin_coil_p10_fp64", kind="dropin", ns=38400, nt=4096, order=10, cap=1000, cap_t=100),
        # the reference's boundary-element problem on a cylinder
        dict(name="bem_cylinder_p10_fp64", kind="bem", ns=6000, nt=1999, order=10, cap=32, cap_t=32),
        # the stray field of the torus coil at many points, by the treecode
        dict(name="treecode_coil_p10_fp64", kind="treecode", ns=38400, nt=65536, order=10, cap=1000),
        # the direct sum that an FMM result is checked against
        dict(name="direct_1m_16k_fp64", kind="direct", geometry="shell", ns=1048576, nt=16384),
    ]


def _log(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["field"] * 5 + ["moving", "training", "potential", "dropin", "bem", "treecode", "direct"])
    if kind == "field":
        precision = rng.choice(["f16x3", "f16x3", "fp64", "fp32"])
        big = {"f16x3": 4000000, "fp32": 1000000, "fp64": 1000000}[precision]
        order = rng.choice([8, 10, 12, 13, 14, 16] if precision == "f16x3" else [6, 8, 10, 11, 12])
        return dict(kind=kind, geometry=rng.choice(["shells", "shell", "clusters"]), ns=_log(rng, 300, big),
                    nt=_log(rng, 100, big), order=order, cap=rng.choice([32, 48, 64, 100]),
                    depth=rng.choice([10, 21]), precision=precision)
    if kind == "moving":
        return dict(kind=kind, geometry=rng.choice(["clusters", "shells"]), ns=_log(rng, 2000, 1000000),
                    nt=_log(rng, 2000, 1000000), order=rng.choice([10, 12, 14]), cap=rng.choice([48, 64]),
                    depth=10, precision="f16x3")
    if kind == "training":
        return dict(kind=kind, geometry=rng.choice(["clusters", "shell"]), ns=_log(rng, 4000, 262000),
                    nt=_log(rng, 1000, 131000), order=rng.choice([8, 10, 12, 14]), cap=rng.choice([32, 48, 64]),
                    depth=10, precision=rng.choice(["f16x3", "fp64"]))
    if kind == "potential":
        return dict(kind=kind, geometry=rng.choice(["shells", "shell"]), ns=_log(rng, 4000, 250000),
                    nt=_log(rng, 4000, 250000), order=rng.choice([8, 10, 12]), cap=rng.choice([32, 48]), depth=21,
                    precision=rng.choice(["fp32", "fp64"]))
    if kind == "dropin":
        return dict(kind=kind, ns=_log(rng, 4000, 38400), nt=_log(rng, 300, 4096), order=rng.choice([6, 8, 10]),
                    cap=rng.choice([500, 1000]), cap_t=rng.choice([100, 128]))
    if kind == "bem":
        return dict(kind=kind, ns=_log(rng, 1000, 6000), nt=_log(rng, 200, 1999), order=rng.choice([6, 8, 10]),
                    cap=rng.choice([32, 64]), cap_t=rng.choice([32, 128]))
    if kind == "treecode":
        return dict(kind=kind, ns=_log(rng, 5000, 38400), nt=_log(rng, 1, 65536), order=rng.choice([8, 10, 12]),
                    cap=rng.choice([500, 1000]))
    return dict(kind=kind, geometry=rng.choice(["shell", "clusters"]), ns=_log(rng, 10000, 1000000),
                nt=_log(rng, 100, 16384))


# ---------------------------------------------------------------- inputs
def _uniform(g, *shape):
    return torch.rand(shape, generator=g, device="cuda", dtype=torch.float64)


def _normal(g, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float64)


def _cylinders(g, n, radii, half):
    """n points uniform in hollow cylinders of the given radii and half thickness, |z| <= 0.5."""
    u = _uniform(g, n, 3)
    k = torch.arange(n, device="cuda") % len(radii)
    mid = torch.tensor(radii, device="cuda", dtype=torch.float64)[k]
    r0, r1 = mid - half, mid + half
    r = torch.sqrt(r0 * r0 + (r1 * r1 - r0 * r0) * u[:, 0])
    ph = 2 * math.pi * u[:, 1]
    return torch.stack([r * torch.cos(ph), r * torch.sin(ph), u[:, 2] - 0.5], 1).contiguous(), k


def _clusters(g, n, centres, sigma):
    k = torch.randint(len(centres), (n,), generator=g, device="cuda")
    return (centres[k] + _normal(g, n, 3) * sigma[k]).contiguous()


def _points(case, seed):
    """Sources, weights, current directions (None: along phi-hat) and targets on the GPU."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    ns, nt = case["ns"], case["nt"]
    if case["geometry"] == "clusters":
        # 64 anisotropic Gaussian clusters with currents of any direction; targets in the same clusters
        centres, sigma = 2 * _uniform(g, 64, 3) - 1, 0.01 + 0.09 * _uniform(g, 64, 3)
        src = _clusters(g, ns, centres, sigma)
        J = _normal(g, ns, 3)
        J = (J / J.norm(dim=1, keepdim=True)).contiguous()
        return src, (0.5 + _uniform(g, ns)) / ns, J, _clusters(g, nt, centres, sigma)
    if case["geometry"] == "shells":
        # four coaxial coils, a current sign each
        src, k = _cylinders(g, ns, (0.5, 0.8, 1.1, 1.4), 0.05)
        sign = 2.0 * torch.randint(2, (4,), generator=g, device="cuda").double() - 1
        w = sign[k] / ns
    else:
        src, _ = _cylinders(g, ns, (0.9,), 0.1)
        w = torch.full((ns,), 1.0 / ns, device="cuda", dtype=torch.float64)
    return src, w, None, 4 * _uniform(g, nt, 3) - 2


def _coil(case, seed):
    """Quadrature points of a torus coil (R = 2, section 0.2 x 0.2), equal weights."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    u = _uniform(g, case["ns"], 3)
    r, ph = 1.9 + 0.2 * u[:, 0], 2 * math.pi * u[:, 1]
    src = torch.stack([r * torch.cos(ph), r * torch.sin(ph), 0.2 * u[:, 2] - 0.1], 1).contiguous()
    w = torch.full((case["ns"],), 2 * math.pi * 2 * 0.04 / case["ns"], device="cuda", dtype=torch.float64)
    if case["kind"] == "treecode":   # the stray field, far enough out that the treecode drops no leaf of the coil
        d = _normal(g, case["nt"], 3)
        tgt = d / d.norm(dim=1, keepdim=True) * (6 + 3 * _uniform(g, case["nt"], 1))
    else:
        tgt = 5 * _uniform(g, case["nt"], 3) - 2.5
    return src, w, tgt.contiguous()


def _cylinder_surface(case, seed):
    """Points on the side of a cylinder with outward normals, a smooth field there, and targets."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    n = case["ns"]
    ph, z = 2 * math.pi * _uniform(g, n), 3 * _uniform(g, n) - 1.5
    src = torch.stack([torch.cos(ph), torch.sin(ph), z], 1)
    nrm = torch.stack([torch.cos(ph), torch.sin(ph), torch.zeros_like(z)], 1)
    B = torch.stack([0.3 * torch.sin(ph), 1.0 + 0.2 * z, torch.cos(2 * ph)], 1)
    w = torch.full((n,), 2 * math.pi * 3.0 / n, device="cuda", dtype=torch.float64)
    box = torch.tensor([1.6, 1.6, 2.4], device="cuda", dtype=torch.float64)
    tgt = (_uniform(g, case["nt"], 3) - 0.5) * box
    return src, w, B, nrm, tgt


def _ptr(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def _mixed(case):
    return case.get("precision", "fp64") != "fp64"


def _config(case):
    return dict(order=case["order"], source_leaf_capacity=case["cap"], target_leaf_capacity=case["cap"],
                precision=case["precision"], frame=fm.FRAME_SHARED, max_depth=case["depth"])


# ---------------------------------------------------------------- what a program has in hand
class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.case, kind = case, case["kind"]
    if kind in ("field", "moving", "potential"):
        s.src, s.w, s.J, s.tgt = _points(case, seed)
        s.fmm = fm.FMM(**_config(case))
        s.B = torch.empty((case["nt"], 3), dtype=torch.float64, device="cuda")
        s.A = torch.empty_like(s.B) if kind == "potential" else None
        torch.cuda.synchronize()
        if kind != "moving":
            s.fmm.set_sources_dev(case["ns"], _ptr(s.src), _ptr(s.w), _ptr(s.J))
            s.fmm.set_targets_dev(case["nt"], _ptr(s.tgt))
    elif kind == "training":
        from bachelors_amd.torch_fmm import FMMBiotSavart
        src, w, J, tgt = _points(case, seed)
        g = torch.Generator(device="cuda").manual_seed(int(seed) + 1)
        s.w = (w * (0.9 + 0.2 * _uniform(g, case["ns"]))).requires_grad_(True)
        s.measured = 0.2 * _normal(g, case["nt"], 3)
        torch.cuda.synchronize()
        # a current of 1e7 A makes the field of the unit total weight order one
        s.model = FMMBiotSavart(src, tgt, J=J, order=case["order"], cap=case["cap"], precision=case["precision"],
                                current=1e7, max_depth=case["depth"])
    elif kind == "dropin":
        src, w, tgt = _coil(case, seed)
        s.quadratures = torch.cat([src, w[:, None]], 1).cpu().numpy()
        s.points = tgt.cpu().numpy()
    elif kind == "bem":
        src, w, B, nrm, tgt = _cylinder_surface(case, seed)
        s.quadratures = torch.cat([src, w[:, None]], 1).cpu().numpy()
        s.field, s.normal, s.points = (t.cpu().numpy() for t in (B, nrm, tgt))
    elif kind == "treecode":
        src, w, s.tgt = _coil(case, seed)
        s.B, s.A = torch.empty_like(s.tgt), torch.empty_like(s.tgt)
        s.fmm = fm.FMM(order=case["order"], source_leaf_capacity=case["cap"], precision="fp64")
        torch.cuda.synchronize()
        s.fmm.set_sources_dev(case["ns"], _ptr(src), _ptr(w))
        s.fmm.set_targets_dev(case["nt"], _ptr(s.tgt))
        s.fmm.build_trees()
        s.fmm.upward()
        s.fmm.synchronize()
    else:
        s.src, s.w, s.J, s.tgt = _points(case, seed)
        s.B = torch.empty_like(s.tgt)
        s.fmm = fm.FMM(order=2, source_leaf_capacity=64, target_leaf_capacity=64)
        torch.cuda.synchronize()
        s.fmm.set_sources_dev(case["ns"], _ptr(s.src), _ptr(s.w), _ptr(s.J))
        s.fmm.set_targets_dev(case["nt"], _ptr(s.tgt))
        s.fmm.build_trees()
        s.fmm.synchronize()
    return s


def _solver_steps(solver):
    solver.calcMultipoleExpansionsAtLeaves()
    solver.calclMultipoleExpansions(fm.M2MAlg.Matrices, fm.Device.GPU)
    solver.calcLocalMultipoleExpansions(fm.M2LAlg.ComplexTranslation, fm.Device.GPU)


def run(s):
    case, kind = s.case, s.case["kind"]
    if kind in ("field", "moving"):
        if kind == "moving":
            s.fmm.set_sources_dev(case["ns"], _ptr(s.src), _ptr(s.w), _ptr(s.J))
            s.fmm.set_targets_dev(case["nt"], _ptr(s.tgt))
        s.fmm.run_B_dev(1.0, _ptr(s.B))
        s.fmm.synchronize()   # torch reads B on a stream of its own
        B = s.B.float() if _mixed(case) else s.B
        return {"B": B, "B_probe": B[:PROBE]}
    if kind == "training":
        s.w.grad = None
        B = s.model(s.w)
        ((B - s.measured) ** 2).sum().backward()
        B, g = B.detach(), s.w.grad
        return {"B": B.float(), "grad": g.float()} if _mixed(case) else {"B": B, "grad": g}
    if kind == "potential":
        F = s.fmm
        F.build_trees()
        F.leaf_expansions()
        F.upward()
        F.downward()
        F.evaluate_B_dev(1.0, _ptr(s.B))
        F.evaluate_A_dev(1.0, _ptr(s.A))
        F.synchronize()
        return {"B": s.B.float(), "A": s.A.float()} if _mixed(case) else {"B": s.B, "A": s.A}
    if kind == "dropin":
        solver = fm.FastMultipoleSolver(s.quadratures, s.points, quadratureOctreeLeafCapacity=case["cap"],
                                        calculationPointOctreeLeafCapacity=case["cap_t"], order=case["order"])
        _solver_steps(solver)
        return solver.calcB_array(5.0)
    if kind == "bem":
        solver = fm.FastMultipoleSolver(s.quadratures, s.points, problem=fm.Problem.BEM,
                                        quadratureOctreeLeafCapacity=case["cap"],
                                        calculationPointOctreeLeafCapacity=case["cap_t"], order=case["order"],
                                        bem_B=s.field, bem_normal=s.normal)
        _solver_steps(solver)
        return solver.calcBEM_array(5.0)
    if kind == "treecode":
        s.fmm.treecode_dev(5.0, case["nt"], _ptr(s.tgt), _ptr(s.B), _ptr(s.A))
        s.fmm.synchronize()
        return {"B": s.B, "A": s.A}
    s.fmm.direct_B_dev(1.0, case["nt"], _ptr(s.tgt), _ptr(s.B))
    s.fmm.synchronize()
    return s.B


# ---------------------------------------------------------------- the least work, and the exact values
def work(case):
    """Inputs read and outputs written once; flops of the near pairs (20 each, about 10 leaf
    capacities of sources per target, as measured on the coils), the translations of about 45 far
    pairs per target box by dense operators, and the expansions of every point (10 per coefficient)."""
    ns, nt, kind = case["ns"], case["nt"], case["kind"]
    bytes_ = 56.0 * ns + 48.0 * nt
    if kind == "direct":
        return {"bytes": bytes_, "flops": 20.0 * ns * nt}
    L = (case["order"] + 1) ** 2
    if kind == "treecode":   # some 20 boxes of the coil per point, B and A from each
        return {"bytes": bytes_ + 24.0 * nt, "flops": nt * 20.0 * 40.0 * L}
    cap_t = case.get("cap_t", case["cap"])
    flops = nt * min(10.0 * case["cap"], ns) * 20.0 + (nt / (0.5 * cap_t) + 1) * 45.0 * 6.0 * L * L + 10.0 * L * (ns + nt)
    if kind == "training":
        bytes_, flops = 2 * bytes_, 2 * flops
    if kind == "potential":
        bytes_ += 24.0 * nt
    return {"bytes": bytes_, "flops": flops}


def _phi_hat(src):
    J = torch.stack([-src[:, 1], src[:, 0], torch.zeros_like(src[:, 0])], 1)
    return J / J.norm(dim=1, keepdim=True)


def _inverse_powers(x, y, power):
    """|x_i - y_j|^power, 0 for coincident points."""
    r2 = torch.zeros((len(x), len(y)), device=x.device, dtype=torch.float64)
    for a in range(3):
        d = x[:, a, None] - y[None, :, a]
        r2.addcmul_(d, d)
    f = r2.pow(power / 2)
    return f.masked_fill_(r2 == 0, 0.0)


def _sums(x, y, columns, power):
    """sum_j |x_i - y_j|^power columns_j for every i, in blocks of y."""
    out = torch.zeros((len(x), columns.shape[1]), device=x.device, dtype=torch.float64)
    step = 8192
    for i in range(0, len(x), step):
        for j in range(0, len(y), step):
            out[i:i + step] += _inverse_powers(x[i:i + step], y[j:j + step], power) @ columns[j:j + step]
    return out


def _cross(a, b):
    return torch.linalg.cross(a, b, dim=1)


def _biot_savart(src, q, x):
    """sum_j q_j x (x_i - y_j) / |x_i - y_j|^3"""
    f = _sums(x, src, torch.cat([q, _cross(q, src)], 1), -3)
    return _cross(f[:, :3], x) - f[:, 3:]


def exact(case, seed):
    kind, ns, nt = case["kind"], case["ns"], case["nt"]
    m = min(nt, PROBE) if kind in ("field", "moving") else nt
    if float(ns) * m > EXACT_PAIRS:
        return None
    if kind in ("dropin", "treecode"):
        src, w, tgt = _coil(case, seed)
        q = w[:, None] * _phi_hat(src)
        B = 5.0 * MU0 / (4 * PI) * _biot_savart(src, q, tgt)
        if kind == "dropin":
            return B
        return {"B": B, "A": 5.0 / (4 * PI) * _sums(tgt, src, q, -1)}
    if kind == "bem":
        src, w, Bf, nrm, tgt = _cylinder_surface(case, seed)
        d, v = w * (Bf * nrm).sum(1), w[:, None] * _cross(Bf, nrm)
        f = _sums(tgt, src, torch.cat([src * d[:, None] + _cross(src, v), d[:, None], v], 1), -3)
        return (f[:, :3] - tgt * f[:, 3:4] - _cross(tgt, f[:, 4:])) / (4 * PI)
    src, w, J, tgt = _points(case, seed)
    J = _phi_hat(src) if J is None else J
    scale = MU0 / (4 * PI)
    if kind == "training":
        g = torch.Generator(device="cuda").manual_seed(int(seed) + 1)
        w = w * (0.9 + 0.2 * _uniform(g, ns))
        measured = 0.2 * _normal(g, nt, 3)
        B = 1e7 * scale * _biot_savart(src, w[:, None] * J, tgt)
        dB = 2 * (B - measured)
        f = _sums(src, tgt, torch.cat([_cross(tgt, dB), dB], 1), -3)
        return {"B": B, "grad": 1e7 * scale * (J * (f[:, :3] - _cross(src, f[:, 3:]))).sum(1)}
    q = w[:, None] * J
    B = scale * _biot_savart(src, q, tgt[:m])
    if kind == "direct":
        return B
    if kind == "potential":
        return {"B": B, "A": _sums(tgt, src, q, -1) / (4 * PI)}
    return {"B": B if m == nt else None, "B_probe": B}
