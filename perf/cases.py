"""Performance cases: the work a program that uses ikarus_amd has it do, called as such a program calls it, with
vectors in device memory.

    assemble  one Newton state: bind (u, lambda), residual and tangent (FULL Dirichlet treatment)
    vector    the residual alone at a bound state (a convergence check)
    eas       one Newton state of the EAS-21 element and the update of its internal variables by a correction
    solve     one linear solve with the assembled tangent
    path      LoadControl on a 3D block, mixed form (two-level preconditioner) with the learned predictor
    plane     LoadControl on the 2D plane-strain cantilever, plain FP64 form
    train     one training step of the learned predictor (forward, backward, Adam)

Meshes are seeded: +-5 % interior node jitter, a smooth deformed state, nodes and elements in grid order or (as for
a mesh from a generator that does not sort) in random order.
"""
import ctypes as C
import functools
import os

import numpy as np
import torch

import ikarus_amd as ia
from ikarus_amd import _capi as capi
from ikarus_amd import problems as pb
from ikarus_amd.learned import MLP, N_IN, N_OUT

WEIGHTS = os.path.join(os.path.dirname(os.path.abspath(ia.__file__)), "data", "predictor_mlp_32cubed.f32")
E_MOD, NU = 1000.0, 0.3
LAM, MU = E_MOD * NU / ((1 + NU) * (1 - 2 * NU)), E_MOD / (2 * (1 + NU))
HIDDEN = 128
DLAM = 1.0 / 40.0  # the load step the predictor was trained with
MLP_SHAPES = ((HIDDEN, N_IN), (HIDDEN,), (HIDDEN, HIDDEN), (HIDDEN,), (HIDDEN, HIDDEN), (HIDDEN,), (N_OUT, HIDDEN),
              (N_OUT,))


def listed():
    return [
        # the 64^3 Neo-Hooke block of the benchmark: every Newton iteration of the plain FP64 form starts with this
        dict(name="assemble_nh_fp64_64", op="assemble", nx=64, ny=64, nz=64, material="nh", precision="fp64",
             order="grid"),
        # a few hundred elements, as in parameter studies and tests: launches and round trips
        dict(name="assemble_nh_fp64_8", op="assemble", nx=8, ny=8, nz=8, material="nh", precision="fp64",
             order="grid"),
        # the FP32 tangent of the mixed form, St.Venant-Kirchhoff, odd extents, unsorted numbering
        dict(name="assemble_svk_fp32_odd", op="assemble", nx=53, ny=37, nz=29, material="svk", precision="fp32",
             order="random"),
        # the residual after a correction on the 3.2 M DOF mesh of the precision study
        dict(name="vector_nh_128x128x64", op="vector", nx=128, ny=128, nz=64, material="nh", order="grid"),
        # the EAS bending block of the benchmark: one Newton state and the update of its internal variables
        dict(name="eas_nh_96x96x48", op="eas", nx=96, ny=96, nz=48, material="nh", order="grid"),
        # the same on a small odd mesh
        dict(name="eas_nh_odd", op="eas", nx=23, ny=17, nz=11, material="nh", order="grid"),
        # the linear solve of the plain form: Jacobi-PCG in FP64
        dict(name="solve_jacobi_fp64_64", op="solve", nx=64, ny=64, nz=64, material="nh", solver="jacobi",
             order="grid"),
        # the linear solve of the mixed form, two-level preconditioner
        dict(name="solve_twolevel_64", op="solve", nx=64, ny=64, nz=64, material="nh", solver="twolevel",
             order="grid"),
        # the same with the block-Jacobi preconditioner, odd extents, unsorted numbering
        dict(name="solve_bjacobi_odd", op="solve", nx=41, ny=33, nz=57, material="svk", solver="bjacobi",
             order="random"),
        # the first load steps of a 40-step path, mixed form with the learned predictor: the headline method whole
        dict(name="path_learned_64", op="path", nx=64, ny=64, nz=64, material="nh", steps=4, order="grid"),
        # the 2D cantilever of the benchmark, ten load steps: small linear systems, thousands of short kernels
        dict(name="plane_64x16", op="plane", nx=64, ny=16, steps=10),
        # one step on the batch size the training program uses
        dict(name="train_8192", op="train", rows=8192),
    ]


def _log_int(rng, lo, hi):
    return int(round(float(np.exp(rng.uniform(np.log(lo), np.log(hi))))))


def _extents(rng, lo, hi):
    """Three extents whose product is spread over [lo, hi] on a logarithmic scale, odd ones among them."""
    n = np.exp(rng.uniform(np.log(lo), np.log(hi))) ** (1.0 / 3.0)
    a, b = rng.uniform(0.75, 1.33), rng.uniform(0.75, 1.33)
    e = [max(2, int(n * a)), max(2, int(n * b)), max(2, int(n / (a * b)))]
    return dict(nx=e[0], ny=e[1], nz=e[2])


def draw(rng):
    op = rng.choice(["assemble", "assemble", "vector", "eas", "solve", "solve", "path", "plane", "train"])
    order = rng.choice(["grid", "grid", "random"])
    material = rng.choice(["nh", "nh", "svk"])
    if op == "assemble":
        return dict(op=op, **_extents(rng, 200, 250000), material=material, precision=rng.choice(["fp64", "fp32"]),
                    order=order)
    if op == "vector":
        return dict(op=op, **_extents(rng, 1000, 800000), material=material, order=order)
    if op == "eas":
        return dict(op=op, **_extents(rng, 200, 250000), material=material, order=order)
    if op == "solve":
        solver = rng.choice(["jacobi", "twolevel", "bjacobi"])
        return dict(op=op, **_extents(rng, 2000, 100000), material=material, solver=solver, order=order)
    if op == "path":
        return dict(op=op, **_extents(rng, 2000, 60000), material="nh", steps=rng.randint(2, 4), order="grid")
    if op == "plane":
        ny = _log_int(rng, 4, 14)
        return dict(op=op, nx=4 * ny + rng.randint(0, 3), ny=ny, steps=rng.randint(2, 6))
    return dict(op=op, rows=_log_int(rng, 200, 8000))


# ---- inputs (numpy, made from the seed alone) -------------------------------------------------------------------
@functools.lru_cache(maxsize=2)
def _grid(n, order_seed):
    """Connectivity, lattice indices of the nodes and the grid's node numbers, for extents n."""
    nv = [k + 1 for k in n]
    idx = np.indices(nv[::-1]).reshape(3, -1)[::-1].T
    e = np.indices(n[::-1]).reshape(3, -1)[::-1]
    base = e[0] + nv[0] * (e[1] + nv[1] * e[2])
    off = [(a & 1) + nv[0] * ((a >> 1 & 1) + nv[1] * (a >> 2)) for a in range(8)]
    conn = (base[:, None] + np.array(off)[None, :]).astype(np.int32)
    if order_seed is not None:
        g = np.random.default_rng(order_seed)
        new = g.permutation(idx.shape[0])
        conn = new[conn][g.permutation(conn.shape[0])].astype(np.int32)
        old = np.empty_like(new)
        old[new] = np.arange(new.size)
        idx = idx[old]
    return np.ascontiguousarray(conn), np.ascontiguousarray(idx)


def _mesh(case, seed):
    """X, conn, fixed flags, loaded elements with their face axis and the traction of a 3D case."""
    n = (case["nx"], case["ny"], case["nz"])
    conn, idx = _grid(n, 7 + seed % 5 if case["order"] == "random" else None)
    bending = case["op"] == "eas"
    size = np.array((2.0, 2.0, 1.0) if bending else (1.0, 1.0, 1.0))
    h = size / np.array(n)
    g = np.random.default_rng([seed, 1])
    inner = ((idx > 0) & (idx < np.array(n))).all(1)
    X = idx * h + (g.random(idx.shape) * 2 - 1) * 0.05 * h * inner[:, None]
    axis = 0 if bending else 2  # clamped at 0, loaded at the other end
    fixed = np.repeat((idx[:, axis] == 0).astype(np.uint8), 3)
    faces = np.nonzero(idx[conn[:, 7], axis] == n[axis])[0].astype(np.int32)
    if bending:
        t = np.array([0.0, 0.0, -g.uniform(2.0, 8.0)])
    else:
        d = g.standard_normal(3)
        t = g.uniform(10.0, 40.0) * d / np.linalg.norm(d)
    return dict(X=X, conn=conn, fixed=fixed, faces=faces, axis=axis, t=t, size=size)


def _smooth(m, seed, scale, k):
    """A smooth nodal field of at most `scale` that vanishes on the clamped face (0.02: strains of a few per cent,
    where the tangent is positive definite)."""
    g = np.random.default_rng([seed, k])
    x = m["X"] / m["size"]
    f = sum(g.uniform(-1, 1, 3)[None, :] * np.sin(x @ g.uniform(0.5, 2.5, 3) + g.uniform(0, 6))[:, None]
            for _ in range(3)) / 3
    return np.ascontiguousarray((scale * x[:, m["axis"]:m["axis"] + 1] * f).reshape(-1) * (1 - m["fixed"]))


def _alpha(m, seed):
    """Internal variables whose enhanced strains are about 1e-3 (the modes scale with the element extent to the -8)."""
    ne = m["conn"].shape[0]
    return np.random.default_rng([seed, 5]).standard_normal((ne, 21)) * 1e-3 * (np.prod(m["size"]) / ne) ** (8 / 3)


def _rhs(m, seed):
    """A load vector: a smooth body force on the free DOFs."""
    return _smooth(m, seed, 1.0, 4) * np.prod(m["size"]) / m["conn"].shape[0]


def _batch(case, seed):
    g = np.random.default_rng([seed, 6])
    n = case["rows"]
    x = np.empty((n, N_IN), np.float32)
    x[:, 0:3] = g.random((n, 3))                               # coordinates
    t = g.standard_normal((n, 3))
    x[:, 3:6] = t / np.linalg.norm(t, axis=1, keepdims=True) * g.uniform(0.25, 1.0, (n, 1))  # traction
    x[:, 6] = g.integers(1, 41, n) * DLAM                       # load factor
    x[:, 7] = 1.0                                               # scaled load increment
    x[:, 8:11] = 0.5 * g.standard_normal((n, 3))                # the two previous velocities
    x[:, 11:14] = x[:, 8:11] + 0.05 * g.standard_normal((n, 3))
    y = (x[:, 8:11] - x[:, 11:14] + 0.02 * g.standard_normal((n, 3))).astype(np.float32)
    return x, y


# ---- the calls --------------------------------------------------------------------------------------------------
class _DeviceArray:
    """Library-owned device memory for torch; keeps its owner alive."""

    def __init__(self, owner, addr, count, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=(count,), typestr=typestr, data=(addr, False), version=2)


def _dev(a):
    return torch.from_numpy(a).cuda()


def _ptr(t):
    return C.c_void_p(t.data_ptr())


def _precision(case):
    if case["op"] == "solve":
        return capi.FP64 if case["solver"] == "jacobi" else capi.FP32
    return capi.FP32 if case.get("precision") == "fp32" else capi.FP64


def _problem3d(case, m):
    p = pb.Problem(m["X"], m["conn"], capi.NEOHOOKE if case["material"] == "nh" else capi.SVK, LAM, MU,
                   eas=21 if case["op"] == "eas" else 0, fixed=m["fixed"], traction=tuple(m["t"]))
    p.set_faces(m["faces"], m["axis"], 1)
    return p


def _matrix_view(dev):
    """The assembled blocks where the library holds them: the 3x3 blocks in sliced-ELL slots (ik_matrix_bsr)."""
    lib = capi.lib()
    nbr, nnzb, val, prec = C.c_int64(), C.c_int64(), C.c_void_p(), C.c_int()
    pos, rowptr = C.c_void_p(), C.c_void_p()
    dev.check(lib.ik_matrix_bsr(dev.h, C.byref(nbr), C.byref(nnzb), C.byref(rowptr), None, C.byref(pos),
                                C.byref(val), C.byref(prec)))
    rp = torch.as_tensor(_DeviceArray(dev, rowptr.value, nbr.value + 1, "<i4"), device="cuda").long()
    width = rp[1:] - rp[:-1]
    pad = (-width.numel()) % 64
    slots = int(torch.nn.functional.pad(width, (0, pad)).view(-1, 64).max(1).values.sum()) * 64
    return torch.as_tensor(_DeviceArray(dev, val.value, slots * 9, "<f4" if prec.value == capi.FP32 else "<f8"),
                           device="cuda")


def prepare(case, seed):
    op = case["op"]
    if op == "train":
        x, y = _batch(case, seed)
        mlp = MLP(seed)
        mlp.load(np.fromfile(WEIGHTS, dtype=np.float32))
        return dict(case=case, mlp=mlp, x=_dev(x), y=_dev(y), loss=C.c_double(),
                    params=torch.empty(capi.lib().ik_mlp_num_params(), device="cuda"))
    if op == "plane":
        p = pb.cantilever2d((case["nx"], case["ny"]), seed=seed)
        cfg = capi.LCConfig()
        cfg.load_steps, cfg.tbegin, cfg.tend, cfg.predictor = case["steps"], 0.0, 1.0, capi.PRED_CONSTANT
        settings = ia.nr_settings(tol=1e-8, linear=ia.solver_opts(rtol=1e-12))
        return dict(case=case, dev=ia.Device(p), cfg=cfg, settings=settings,
                    zero=torch.zeros(p.ndof, dtype=torch.float64, device="cuda"),
                    u=torch.empty(p.ndof, dtype=torch.float64, device="cuda"))
    m = _mesh(case, seed)
    p = _problem3d(case, m)
    dev = ia.Device(p)
    s = dict(case=case, dev=dev, R=torch.empty(p.ndof, dtype=torch.float64, device="cuda"))
    lib = capi.lib()
    if op == "path":
        dev.check(lib.ik_mlp_set_params(dev.h, capi.ptr(np.fromfile(WEIGHTS, dtype=np.float32)), capi.HOST))
        cfg = capi.LCConfig()
        cfg.load_steps, cfg.tbegin, cfg.tend, cfg.predictor = case["steps"], 0.0, case["steps"] * DLAM, capi.PRED_MLP
        lin = ia.solver_opts(capi.PCG_TWOLEVEL_FP32_IR, rtol=1e-10, inner_rtol=1e-3, max_refine=30)
        s |= dict(cfg=cfg, zero=torch.zeros(p.ndof, dtype=torch.float64, device="cuda"), u=torch.empty_like(s["R"]),
                  settings=ia.nr_settings(tol=1e-10, precision=capi.FP32, linear=lin, forcing=0.9, eta_max=1e-3))
        return s
    s["u"] = _dev(_smooth(m, seed, 0.02, 3))
    if op == "eas":
        s |= dict(alpha=_dev(_alpha(m, seed)), alpha1=torch.empty(p.ne, 21, dtype=torch.float64, device="cuda"),
                  du=_dev(_smooth(m, seed, 2e-3, 8)))
    # the pattern is built with the first assembly, once per mesh
    dev.check(lib.ik_set_requirement(dev.h, _ptr(s["u"]), 1.0, capi.DEVICE))
    if op == "vector":
        dev.check(lib.ik_vector(dev.h, capi.DBC_FULL, None, capi.DEVICE))
        return s
    if op == "solve":
        dev.check(lib.ik_matrix(dev.h, capi.DBC_FULL, _precision(case)))
        kind = dict(jacobi=capi.PCG_JACOBI_FP64, twolevel=capi.PCG_TWOLEVEL_FP32_IR,
                    bjacobi=capi.PCG_BJACOBI_FP32_IR)[case["solver"]]
        opts = ia.solver_opts(kind, rtol=1e-11, max_iter=5000, inner_rtol=1e-3, max_refine=20)
        s |= dict(opts=opts, info=capi.SolverInfo(), rhs=_dev(_rhs(m, seed)), x=torch.empty_like(s["R"]))
        return s
    dev.check(lib.ik_assemble(dev.h, capi.DBC_FULL, _precision(case), None, capi.DEVICE))
    s["K"] = _matrix_view(dev)
    return s


def run(state):
    lib, op = capi.lib(), state["case"]["op"]
    if op == "train":
        mlp = state["mlp"]
        mlp._check(lib.ik_mlp_train_step(mlp.h, _ptr(state["x"]), _ptr(state["y"]), state["case"]["rows"],
                                         C.c_float(2e-3), C.byref(state["loss"]), capi.DEVICE))
        mlp._check(lib.ik_mlp_params(mlp.h, _ptr(state["params"]), capi.DEVICE))
        return dict(loss=state["loss"].value, params=state["params"])
    dev = state["dev"]
    if op in ("path", "plane"):
        dev.check(lib.ik_set_requirement(dev.h, _ptr(state["zero"]), 0.0, capi.DEVICE))
        info, _, _ = dev.load_control(state["cfg"], state["settings"])
        dev.check(lib.ik_get_requirement(dev.h, _ptr(state["u"]), None, capi.DEVICE))
        return dict(success=int(info.success), u=state["u"])
    if op == "solve":
        dev.check(lib.ik_solve(dev.h, _ptr(state["rhs"]), _ptr(state["x"]), capi.DEVICE, C.byref(state["opts"]),
                               C.byref(state["info"])))
        return dict(converged=int(state["info"].converged), x=state["x"])
    dev.check(lib.ik_set_requirement(dev.h, _ptr(state["u"]), 1.0, capi.DEVICE))
    if op == "vector":
        dev.check(lib.ik_vector(dev.h, capi.DBC_FULL, _ptr(state["R"]), capi.DEVICE))
        return dict(R=state["R"])
    if op == "eas":
        dev.check(lib.ik_set_alpha(dev.h, _ptr(state["alpha"]), capi.DEVICE))
    dev.check(lib.ik_assemble(dev.h, capi.DBC_FULL, _precision(state["case"]), _ptr(state["R"]), capi.DEVICE))
    if op == "assemble":
        return dict(R=state["R"], K=state["K"])
    dev.check(lib.ik_update_state(dev.h, _ptr(state["du"]), capi.DEVICE))
    dev.check(lib.ik_get_alpha(dev.h, _ptr(state["alpha1"]), capi.DEVICE))
    return dict(R=state["R"], K=state["K"], alpha=state["alpha1"])


def work(case):
    """Inputs and outputs once; operations in the cheapest form known (the inverse-C form of the tangent: 27 kflop per
    element with the residual, 7 kflop for the residual alone, 87 kflop for the condensed EAS element). A solve reads
    its matrix once here; each of its iterations does so again."""
    op = case["op"]
    if op == "train":
        params = sum(int(np.prod(s)) for s in MLP_SHAPES)
        return dict(bytes=case["rows"] * (N_IN + N_OUT) * 4 + params * 24, flops=6.0 * case["rows"] * params)
    if op == "plane":
        ne, nn = case["nx"] * case["ny"], (case["nx"] + 1) * (case["ny"] + 1)
        return dict(bytes=16 * ne + 48 * nn, flops=case["steps"] * 2 * 3000.0 * ne)
    n = (case["nx"], case["ny"], case["nz"])
    ne, nn = int(np.prod(n)), int(np.prod([k + 1 for k in n]))
    nnzb = int(np.prod([3 * k + 1 for k in n]))
    mesh = 32 * ne + 48 * nn
    mat = nnzb * 9 * (8 if _precision(case) == capi.FP64 else 4)
    if op == "vector":
        return dict(bytes=mesh + 24 * nn, flops=7e3 * ne)
    if op == "assemble":
        return dict(bytes=mesh + mat + 24 * nn, flops=27e3 * ne)
    if op == "eas":
        return dict(bytes=mesh + mat + 48 * nn + 336 * ne, flops=87e3 * ne)
    if op == "solve":
        return dict(bytes=mat + 4 * nnzb + 48 * nn, flops=18.0 * nnzb)
    return dict(bytes=mesh + 24 * nn, flops=case["steps"] * 2 * 27e3 * ne)


# ---- the same in 64 bits with plain torch -----------------------------------------------------------------------
VOIGT = ((0, 0), (1, 1), (2, 2), (1, 2), (0, 2), (0, 1))
EAS_ROW = (0, 1, 2, 3, 3, 4, 4, 5, 5, 3, 3, 4, 4, 5, 5, 0, 0, 1, 1, 2, 2)
EAS_MONOMIAL = ("x", "y", "z", "y", "z", "x", "z", "x", "y", "xy", "xz", "xy", "yz", "xz", "yz", "xy", "xz", "xy", "yz",
                "xz", "yz")
CHUNK = 8192


def _f64(a):
    return torch.as_tensor(np.asarray(a), dtype=torch.float64, device="cuda")


def _d_shape(xi):
    f = np.array([[1 - xi[k], xi[k]] for k in range(3)])
    out = np.empty((8, 3))
    for a in range(8):
        b = [(a >> k) & 1 for k in range(3)]
        for k in range(3):
            out[a, k] = (1 if b[k] else -1) * f[(k + 1) % 3, b[(k + 1) % 3]] * f[(k + 2) % 3, b[(k + 2) % 3]]
    return out


GAUSS = np.array([[0.5 + (1 if (q >> k) & 1 else -1) / (2 * np.sqrt(3.0)) for k in range(3)] for q in range(8)])


def _law(material, Ev):
    """S (Voigt) and the tangent CC (6x6) at the Green-Lagrange strain Ev (engineering shear), [n, 6]."""
    n = Ev.shape[0]
    half = _f64([1, 1, 1, 0.5, 0.5, 0.5])
    one = _f64([1, 1, 1, 0, 0, 0])
    if material == "svk":
        CC = torch.zeros(6, 6, dtype=torch.float64, device="cuda")
        CC[:3, :3] = LAM
        CC += torch.diag(_f64([2 * MU] * 3 + [MU] * 3))
        return Ev @ CC, CC.expand(n, 6, 6)
    Cm = torch.empty(n, 3, 3, dtype=torch.float64, device="cuda")
    v = 2 * Ev * half + one
    for q, (i, j) in enumerate(VOIGT):
        Cm[:, i, j] = Cm[:, j, i] = v[:, q]
    Ci = torch.linalg.inv_ex(Cm).inverse
    ln = 0.5 * torch.log(torch.linalg.det(Cm))[:, None]
    cv = torch.stack([Ci[:, i, j] for i, j in VOIGT], 1)
    S = MU * (one - cv) + LAM * ln * cv
    CC = torch.empty(n, 6, 6, dtype=torch.float64, device="cuda")
    c2 = (MU - LAM * ln)[:, 0]
    for p, (i, j) in enumerate(VOIGT):
        for q, (k, l) in enumerate(VOIGT):
            CC[:, p, q] = LAM * cv[:, p] * cv[:, q] + c2 * (Ci[:, i, k] * Ci[:, j, l] + Ci[:, i, l] * Ci[:, j, k])
    return S, CC


def _transform(J):
    """Voigt strain transformation T(J) times det J, [n, 6, 6]."""
    T = torch.empty(J.shape[0], 6, 6, dtype=torch.float64, device="cuda")
    for r, (a, b) in enumerate(VOIGT):
        for c, (k, l) in enumerate(VOIGT):
            v = J[:, k, a] * J[:, l, b] + J[:, l, a] * J[:, k, b]
            T[:, r, c] = 0.5 * v if a == b else v
    return T * torch.linalg.det(J)[:, None, None].abs()


def _elements(material, x, u, alpha=None, want_k=True):
    """K_e [n, 24, 24], R_e [n, 24] (local order 3a + k) of n elements and, with alpha, D^-1 [L | Rt] [n, 21, 25]."""
    n = x.shape[0]
    K = torch.zeros(n, 24, 24, dtype=torch.float64, device="cuda") if want_k else None
    R = torch.zeros(n, 24, dtype=torch.float64, device="cuda")
    if alpha is not None:
        A = torch.zeros(n, 21, 46, dtype=torch.float64, device="cuda")
        T0i = torch.linalg.inv(_transform(x.transpose(1, 2) @ _f64(_d_shape([0.5] * 3))))
    for xi in GAUSS:
        dN = _f64(_d_shape(xi))
        J = x.transpose(1, 2) @ dN
        det = torch.linalg.det(J).abs()
        g = dN @ torch.linalg.inv_ex(J).inverse
        F = torch.eye(3, dtype=torch.float64, device="cuda") + u.transpose(1, 2) @ g
        B = torch.empty(n, 6, 8, 3, dtype=torch.float64, device="cuda")
        for q, (i, j) in enumerate(VOIGT):
            B[:, q] = F[:, None, :, i] * g[:, :, j, None]
            if i != j:
                B[:, q] += F[:, None, :, j] * g[:, :, i, None]
        B = B.reshape(n, 6, 24)
        Cm = F.transpose(1, 2) @ F
        Ev = torch.stack([0.5 * (Cm[:, i, j] - 1) if i == j else Cm[:, i, j] for i, j in VOIGT], 1)
        if alpha is not None:
            c = dict(zip("xyz", 2 * xi - 1))
            f = [np.prod([c[s] for s in m]) for m in EAS_MONOMIAL]
            M = T0i[:, :, list(EAS_ROW)] * _f64(f) / det[:, None, None]
            Ev = Ev + (M @ alpha[:, :, None])[:, :, 0]
        S, CC = _law(material, Ev)
        dV = det / 8
        R += ((S * dV[:, None])[:, None, :] @ B)[:, 0]
        CB = (CC @ B) * dV[:, None, None]
        if alpha is not None:
            Mt = M.transpose(1, 2)
            A[:, :, :21] += Mt @ ((CC @ M) * dV[:, None, None])
            A[:, :, 21:45] += Mt @ CB
            A[:, :, 45] += (Mt @ (S * dV[:, None])[:, :, None])[:, :, 0]
        if want_k:
            Sm = torch.empty(n, 3, 3, dtype=torch.float64, device="cuda")
            for q, (i, j) in enumerate(VOIGT):
                Sm[:, i, j] = Sm[:, j, i] = S[:, q] * dV
            G = g @ Sm @ g.transpose(1, 2)
            K += B.transpose(1, 2) @ CB
            K.view(n, 8, 3, 8, 3).diagonal(dim1=2, dim2=4).add_(G[..., None])
    if alpha is None:
        return K, R, None
    L = A[:, :, 21:45].clone()
    for j in range(21):  # Gauss-Jordan elimination (D is positive definite)
        A[:, j] /= A[:, j, j, None].clone()
        rest = torch.cat([torch.arange(0, j), torch.arange(j + 1, 21)])
        A[:, rest] -= A[:, rest, j, None] * A[:, j, None, :]
    Y = A[:, :, 21:]
    KR = L.transpose(1, 2) @ Y
    return K - KR[:, :, :24] if want_k else None, R - KR[:, :, 24], Y


def _assembled(case, m, u, lam=1.0, alpha=None, du=None, want_k=True):
    """R and K (block pattern rows, columns, [nnzb, 3, 3] values), FULL; with alpha its updated values."""
    conn, X = torch.from_numpy(m["conn"]).long().cuda(), _f64(m["X"])
    nn, ne = X.shape[0], conn.shape[0]
    u = u.view(nn, 3)
    R = torch.zeros(nn, 3, dtype=torch.float64, device="cuda")
    rows = cols = val = None
    if want_k:
        keys = torch.unique((conn[:, :, None] * nn + conn[:, None, :]).view(-1))
        rows, cols = keys // nn, keys % nn
        val = torch.zeros(keys.numel(), 3, 3, dtype=torch.float64, device="cuda")
    new = []
    for e0 in range(0, ne, CHUNK):
        c = conn[e0:e0 + CHUNK]
        Ke, Re, Y = _elements(case["material"], X[c], u[c], None if alpha is None else alpha[e0:e0 + CHUNK], want_k)
        R.index_add_(0, c.view(-1), Re.view(-1, 3))
        if want_k:
            at = torch.searchsorted(keys, (c[:, :, None] * nn + c[:, None, :]).reshape(-1))
            val.index_add_(0, at, Ke.view(-1, 8, 3, 8, 3).permute(0, 1, 3, 2, 4).reshape(-1, 3, 3))
        if du is not None:
            d = torch.cat([du.view(nn, 3)[c].view(-1, 24), torch.ones(c.shape[0], 1, device="cuda")], 1)
            new.append(alpha[e0:e0 + CHUNK] - (Y @ d[:, :, None])[:, :, 0])
    f = conn[torch.from_numpy(m["faces"]).long().cuda()]
    a = [a for a in range(8) if a >> m["axis"] & 1]  # the four corners of the loaded face
    p = X[f][:, a]
    t1 = (p[:, 1] - p[:, 0] + p[:, 3] - p[:, 2]) / 2
    t2 = (p[:, 2] - p[:, 0] + p[:, 3] - p[:, 1]) / 2
    area = torch.linalg.cross(t1, t2).norm(dim=1)
    load = (-0.25 * lam * area[:, None, None] * _f64(m["t"])).expand(-1, 4, 3)
    R.index_add_(0, f[:, a].reshape(-1), load.reshape(-1, 3))
    fx = torch.from_numpy(m["fixed"]).bool().cuda().view(nn, 3)
    R[fx] = 0.0
    if want_k:
        val[fx[rows][:, :, None] | fx[cols][:, None, :]] = 0.0
        dg = torch.nonzero(rows == cols)[:, 0]
        val[dg] += torch.diag_embed(fx.double())[rows[dg]]
    return R.view(-1), (rows, cols, val), torch.cat(new) if new else None


def _slots(rows, val, nn):
    """The blocks in sliced-ELL order: 64-row slices as wide as their longest row, block j of row r of a slice at
    64 j + r, zeros between."""
    cnt = torch.bincount(rows, minlength=nn)
    first = torch.cumsum(cnt, 0) - cnt
    width = torch.nn.functional.pad(cnt, (0, (-nn) % 64)).view(-1, 64).max(1).values
    start = 64 * (torch.cumsum(width, 0) - width)
    j = torch.arange(rows.numel(), device="cuda") - first[rows]
    out = torch.zeros(64 * int(width.sum()), 9, dtype=torch.float64, device="cuda")
    out[start[rows // 64] + 64 * j + rows % 64] = val.reshape(-1, 9)
    return out.view(-1)


def _cg(K, b, rtol):
    """Conjugate gradients with 3x3 block Jacobi."""
    rows, cols, val = K
    nn = b.numel() // 3
    dg = torch.nonzero(rows == cols)[:, 0]
    Mi = torch.linalg.inv(val[dg])

    def mul(v):
        out = torch.zeros(nn, 3, dtype=torch.float64, device="cuda")
        return out.index_add_(0, rows, (val * v.view(nn, 3)[cols][:, None, :]).sum(2)).view(-1)

    def pre(v):
        return (Mi * v.view(nn, 1, 3)).sum(2).view(-1)

    x, r = torch.zeros_like(b), b.clone()
    z = pre(r)
    p, rz = z, r @ z
    stop = rtol * float(b.norm())
    for k in range(6000):
        q = mul(p)
        a = rz / (p @ q)
        x = x + a * p
        r = r - a * q
        if k % 32 == 31 and float(r.norm()) <= stop:
            break
        z = pre(r)
        new = r @ z
        p, rz = z + (new / rz) * p, new
    return x


def _exact_train(case, seed):
    x, y = (_f64(a) for a in _batch(case, seed))
    flat, at = np.fromfile(WEIGHTS, dtype=np.float32), 0
    par = []
    for s in MLP_SHAPES:
        k = int(np.prod(s))
        par.append(_f64(flat[at:at + k].reshape(s)).requires_grad_())
        at += k
    h = x
    for l in range(4):
        h = h @ par[2 * l].T + par[2 * l + 1]
        h = torch.nn.functional.silu(h) if l < 3 else h
    loss = ((h - y) ** 2).mean()
    loss.backward()
    new = [p.detach() - 2e-3 * p.grad / (p.grad.abs() + 1e-8) for p in par]  # Adam's first step
    return dict(loss=float(loss.detach()), params=torch.cat([p.reshape(-1) for p in new]))


def _exact_plane(case, seed):
    """Equilibrium at lambda = 1 by load steps, dense, on the one-layer hexahedral extrusion of unit thickness with the
    displacement independent of z."""
    p = pb.cantilever2d((case["nx"], case["ny"]), seed=seed)
    nn, ne = p.X.shape[0], p.conn.shape[0]
    X = np.concatenate([np.c_[p.X, np.zeros(nn)], np.c_[p.X, np.ones(nn)]])
    conn = torch.from_numpy(np.concatenate([p.conn, p.conn + nn], 1)).long().cuda()
    x = _f64(X)[conn]
    fixed = torch.from_numpy(p.fixed.astype(bool)).cuda()
    dof = (2 * torch.from_numpy(p.conn).long().cuda()[:, :, None] + torch.arange(2, device="cuda")).view(ne, 8)
    f = torch.zeros(2 * nn, dtype=torch.float64, device="cuda")
    h = 1.0 / case["ny"]
    edge = torch.from_numpy(p.conn[p.face_elem][:, [1, 3]]).long().cuda()
    for k in range(2):
        f.index_add_(0, (2 * edge + k).reshape(-1), torch.full((edge.numel(),), 0.5 * h * p.traction[k],
                                                            dtype=torch.float64, device="cuda"))
    v = torch.zeros(2 * nn, dtype=torch.float64, device="cuda")
    for step in range(10):
        for _ in range(12):
            u3 = torch.cat([v.view(nn, 2), torch.zeros(nn, 1, dtype=torch.float64, device="cuda")], 1).repeat(2, 1)
            Ke, Re, _ = _elements("nh", x, u3[conn])
            Ke = Ke.view(ne, 2, 4, 3, 2, 4, 3).sum((1, 4))[:, :, :2, :, :2].reshape(ne, 8, 8)
            Re = Re.view(ne, 2, 4, 3).sum(1)[:, :, :2].reshape(ne, 8)
            R = -f * (step + 1) / 10
            R = R.index_add(0, dof.view(-1), Re.reshape(-1)).masked_fill(fixed, 0.0)
            if float(R.norm()) <= 1e-12:
                break
            K = torch.zeros(2 * nn, 2 * nn, dtype=torch.float64, device="cuda")
            K.view(-1).index_add_(0, (dof[:, :, None] * 2 * nn + dof[:, None, :]).view(-1), Ke.reshape(-1))
            K[fixed] = 0.0
            K[:, fixed] = 0.0
            K[fixed, fixed] = 1.0
            v = v - torch.linalg.solve(K, R)
    return dict(success=None, u=v)


def exact(case, seed):
    op = case["op"]
    if op == "train":
        return _exact_train(case, seed)
    if op == "plane":
        return _exact_plane(case, seed)
    m = _mesh(case, seed)
    if op == "path":
        lam = case["steps"] * DLAM
        u = torch.zeros(m["X"].size, dtype=torch.float64, device="cuda")
        for _ in range(12):
            R, K, _ = _assembled(case, m, u, lam)
            if float(R.norm()) <= 1e-11:
                break
            u = u - _cg(K, R, max(1e-8, 1e-12 / float(R.norm())))
        return dict(success=None, u=u)
    u = _f64(_smooth(m, seed, 0.02, 3))
    if op == "vector":
        return dict(R=_assembled(case, m, u, want_k=False)[0])
    if op == "solve":
        K = _assembled(case, m, u)[1]
        return dict(converged=None, x=_cg(K, _f64(_rhs(m, seed)), 1e-14))
    alpha = du = None
    if op == "eas":
        alpha, du = _f64(_alpha(m, seed)), _f64(_smooth(m, seed, 2e-3, 8))
    R, (rows, _, val), new = _assembled(case, m, u, alpha=alpha, du=du)
    out = dict(R=R, K=_slots(rows, val, m["X"].shape[0]))
    return out if new is None else dict(alpha=new, **out)
