"""Performance cases of the mixed-FEM framework: what its users have it do,
through its public entry points (`mfem_amd.native`), over the range of sizes,
precisions, solvers and element kinds that its scenes, tests and benchmark use.

Kinds of case:
  newton    one Newton iteration through the phase entry points
            (mfem_sim_update_system, _solve, _energy at 0 and 1) on a deformed
            start, with the step read back: every solver and element kind;
  step      one whole time step (mfem_sim_step) with the positions read back;
  batch     one time step of many independent beams (mfem_batch_step);
  pcg       the linear solver on a caller's own 3x3-block matrix on the device
            (mfem_pcg_bsr3);
  elements  the batched polar fit and material evaluation on device arrays
            (mfem_polar_batch, mfem_material_s6_batch).
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from mfem_amd import native, scenes

# element kinds of newton / step cases: dimension, mixed stretch or plain
# displacement, and the materials
KINDS = {
    "tet": (3, True, "snh"),         # mixed stretch, stable Neo-Hookean
    "tet_stiff": (3, True, "arap"),  # ARAP next to stable Neo-Hookean, E in [1e4, 1e8], nu 0.49
    "tet_plain": (3, False, "snh"),  # displacement-only
    "tri": (2, True, "snh"),
    "tri_plain": (2, False, "snh"),
}


def _newton(name, element, nx, ny, nz, precision, solver="eigen-pcg-diag", tol=1e-4, cap=500):
    return dict(name=name, kind="newton", element=element, nx=nx, ny=ny, nz=nz,
                precision=precision, solver=solver, tol=tol, cap=cap)


def _step(name, element, nx, ny, nz, precision, tol=1e-4, cap=500):
    return dict(_newton(name, element, nx, ny, nz, precision, tol=tol, cap=cap), kind="step")


def listed():
    return [
        # The smallest scene: the 2D displacement-only rectangle with a dense
        # direct solve, the solver that the reference's own scenes name.
        _newton("rect_direct", "tri_plain", 40, 10, 0, "fp64", solver="eigen-llt"),
        # A small interactive beam, as in the tests and the reference's small
        # meshes: latency and launches decide.
        _newton("beam_small_fp64", "tet", 13, 5, 5, "fp64"),
        # A 2D mixed-stretch sheet of ordinary size.
        _newton("sheet_fp64", "tri", 150, 61, 0, "fp64"),
        # The 24k-tet displacement-only benchmark beam, CG to 1e-10: a whole
        # time step whose solves are thousands of short iterations.
        _step("plain_24k_step", "tet_plain", 40, 10, 10, "fp64", tol=1e-10, cap=20000),
        # An ordinary production mesh at full precision (the default).
        _newton("beam_200k_fp64", "tet", 60, 24, 24, "fp64"),
        # The stiff, ill-conditioned two-material scene: CG runs into its cap.
        _newton("stiff_300k_mixed", "tet_stiff", 81, 25, 25, "mixed"),
        # The indefinite (KKT) solver of the reference, iteration cap 500.
        _newton("minres_23k_fp64", "tet", 27, 12, 12, "fp64", solver="minres-indefinite-block"),
        # CG with the incomplete-Cholesky preconditioner.
        _newton("ic_150k_mixed", "tet", 55, 21, 21, "mixed", solver="eigen-pcg-IC"),
        # Many independent beams of 2k to 60k tets advanced together.
        dict(name="batch_48_mixed", kind="batch", count=48, precision="mixed"),
        # The benchmark's own scene and the largest: 960k tets, mixed
        # precision, one whole time step.
        _step("beam_960k_step", "tet", 100, 40, 40, "mixed"),
        # Another program's system through the linear-solver entry point.
        dict(name="pcg_21k_rows", kind="pcg", nx=41, ny=27, nz=19, tol=1e-8, cap=2000),
        # Element evaluation for a caller's own assembly.
        dict(name="elements_300k", kind="elements", n=300_001),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["newton"] * 6 + ["step", "batch", "pcg", "elements"])
    precision = rng.choice(["fp64", "mixed"])
    if kind == "batch":
        return dict(kind=kind, count=_log(rng, 3, 32), precision=precision)
    if kind == "pcg":
        n = _log(rng, 8, 36)
        return dict(kind=kind, nx=n + rng.randrange(9), ny=n, nz=max(5, n - rng.randrange(9)),
                    tol=rng.choice([1e-4, 1e-6, 1e-8]), cap=2000)
    if kind == "elements":
        return dict(kind=kind, n=_log(rng, 1000, 290_000))
    element = rng.choice(["tet", "tet", "tet", "tet_stiff", "tet_plain", "tri"])
    solver = "eigen-pcg-diag"
    if element == "tri":
        ny = _log(rng, 8, 90)
        nx, nz = int(ny * rng.uniform(1.5, 4.0)), 0
    else:
        ny = _log(rng, 3, 20 if kind == "step" else 32)
        nx, nz = int(ny * rng.uniform(2.0, 3.5)) + rng.randrange(3), ny + rng.randrange(3)
        if kind == "newton" and element == "tet":
            solver = rng.choice(["eigen-pcg-diag"] * 3 + ["eigen-pcg-IC", "minres-indefinite-block"])
            if solver == "minres-indefinite-block":
                precision = "fp64"
                ny = _log(rng, 3, 12)
                nx, nz = int(ny * rng.uniform(1.5, 2.5)) + rng.randrange(3), ny + rng.randrange(2)
    c = dict(kind=kind, element=element, nx=nx, ny=ny, nz=nz, precision=precision, tol=1e-4,
             cap=500)
    return dict(c, solver=solver if kind == "newton" else "eigen-pcg-diag")


# --- inputs -------------------------------------------------------------------

def _scene(case, seed):
    """The scene of a newton or step case. A newton case starts from a smooth
    deformation of the rest shape (the pinned end stays), a step from rest;
    both with a smooth initial velocity."""
    dim, mixed, material = KINDS[case["element"]]
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    kw = dict(itr_tol=case["tol"], max_iters=case["cap"], solver=case["solver"])
    if dim == 2:
        sc = scenes.rect2d_scene(nx, ny, E=1e5, **kw)
        sc.mixed = mixed
    elif material == "arap":
        kw.pop("solver")
        sc = scenes.config_c5(nx, ny, nz, seed, **kw)
    elif mixed:
        sc = scenes.beam_scene(nx, ny, nz, seed=seed, E_range=(1e5, 1e6), **kw)
    else:
        sc = scenes.beam_scene(nx, ny, nz, seed=seed, mixed=False, **kw)
    rng = np.random.RandomState(seed % (1 << 31))
    top = sc.V.max(axis=0)
    u = sc.V / top  # unit box; the pinned end is u[:, 0] = 1
    free = (1.0 - u[:, :1])

    def smooth():
        a, b, p = rng.uniform(-1, 1, (3, dim, dim))
        return np.sin(math.pi * (u @ a.T) + p[0]) + 0.5 * u @ b

    if case["kind"] == "newton":
        sc.x0 = sc.V + 0.05 * top[1] * free * smooth()
    sc.v0 = 0.2 * free * smooth()
    sc.v0[sc.fixed != 0] = 0.0
    return sc


def _beams(case, seed):
    """The benchmark's independent beams: 2k to 60k tets (the same sizes for
    every seed), each with its own stiffness and jitter."""
    rng = np.random.RandomState(seed % (1 << 31))
    out = []
    for k, (nx, ny, nz) in enumerate(scenes.c4_beam_sizes(case["count"], 0)):
        out.append(scenes.beam_scene(nx, ny, nz, seed=seed + k, E=math.exp(rng.uniform(
            math.log(1e4), math.log(1e7))), nu=rng.uniform(0.3, 0.48), itr_tol=1e-4,
            max_iters=500, solver="eigen-pcg-diag"))
    return out


def _pcg_system(case, seed):
    """An elastic-network matrix on a grid with the 15-point couplings of a
    tetrahedral mesh: K_ij = -W_ij (random symmetric positive definite 3x3),
    K_ii the sum of its W plus a small mass. On the GPU, CSR order."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    n = nx * ny * nz
    ids = torch.arange(n, device="cuda").reshape(nx, ny, nz)
    eye = torch.eye(3, device="cuda", dtype=torch.float64)
    D = 1e-3 * eye.repeat(nx, ny, nz, 1, 1)
    ii, jj, ww = [], [], []
    for dx, dy, dz in [(1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 1, 0), (1, 0, 1), (0, 1, 1), (1, 1, 1)]:
        lo = (slice(0, nx - dx), slice(0, ny - dy), slice(0, nz - dz))
        hi = (slice(dx, nx), slice(dy, ny), slice(dz, nz))
        A = torch.randn(nx - dx, ny - dy, nz - dz, 3, 3, generator=g, device="cuda",
                        dtype=torch.float64)
        W = (A[..., :, None, :] * A[..., None, :, :]).sum(-1) + 0.3 * eye  # A A^T + 0.3 I
        D[lo] += W
        D[hi] += W
        ii.append(ids[lo].reshape(-1))
        jj.append(ids[hi].reshape(-1))
        ww.append(W.reshape(-1, 3, 3))
    i, j, W, D = torch.cat(ii), torch.cat(jj), torch.cat(ww), D.reshape(n, 3, 3)
    rows = torch.cat([i, j, ids.reshape(-1)])
    cols = torch.cat([j, i, ids.reshape(-1)])
    vals = torch.cat([-W, -W, D])
    order = torch.argsort(rows * n + cols)
    rowptr = torch.zeros(n + 1, dtype=torch.int32, device="cuda")
    rowptr[1:] = torch.cumsum(torch.bincount(rows, minlength=n), 0)
    b = torch.randn(3 * n, generator=g, device="cuda", dtype=torch.float64)
    return rowptr, cols[order].to(torch.int32), vals[order].reshape(-1).contiguous(), b


def _element_inputs(case, seed):
    """Deformation gradients of a moderately deformed mesh with rotations, and
    the stretches, materials and moduli of its elements."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    n = case["n"]

    def rand(*shape):
        return torch.rand(*shape, generator=g, device="cuda", dtype=torch.float64)

    F = torch.eye(3, device="cuda", dtype=torch.float64) + 0.5 * (rand(n, 3, 3) - 0.5)
    s = torch.cat([1.0 + 0.4 * (rand(n, 3) - 0.5), 0.3 * (rand(n, 3) - 0.5)], 1)
    mu, la = scenes.enu_to_lame(1e5, 0.45)
    scale = torch.exp(math.log(10.0) * rand(n))
    mat = torch.tensor([scenes.MATERIALS[m] for m in
                        ("Stable-Neohookean", "ARAP", "Corot", "FixedCorot")],
                       dtype=torch.int32, device="cuda")
    which = torch.randint(0, 4, (n,), generator=g, device="cuda") * (rand(n) < 0.3)
    return dict(F=F.transpose(1, 2).reshape(n, 9).contiguous(), s=s, mu=mu * scale, la=la * scale,
                mat=mat[which].contiguous())


def prepare(case, seed):
    kind = case["kind"]
    if kind == "pcg":
        return dict(case=case, system=_pcg_system(case, seed))
    if kind == "elements":
        st = dict(case=case, **_element_inputs(case, seed))
        n, new = case["n"], lambda *shape: torch.empty(*shape, dtype=torch.float64, device="cuda")
        st.update(eye=torch.eye(3, dtype=torch.float64, device="cuda").reshape(1, 9).repeat(n, 1),
                  R=new(n, 9), S=new(n, 6), dsdF=new(n, 54), E=new(n), g=new(n, 6), H=new(n, 36),
                  it=torch.empty(n, dtype=torch.int32, device="cuda"))
        return st
    if kind == "batch":
        return dict(case=case, count=case["count"],
                    batch=native.Batch(_beams(case, seed), case["precision"]))
    return dict(case=case, sim=native.Sim(_scene(case, seed), case["precision"]))


def run(state):
    kind = state["case"]["kind"]
    if kind == "newton":
        sim = state["sim"]
        sim.update_system()
        dec = sim.solve()
        e0, e1 = sim.energy(0.0), sim.energy(1.0)
        if state["case"]["element"] == "tet_stiff":
            # the solve ends at its cap, unconverged: the largest entry of the
            # step and E(1) of single hard elements are rounding there (they
            # move by 9% and 60% under a change of one last place in x)
            return dict(dx=sim.get("dx"), e0=e0)
        return dict(dx=sim.get("dx"), decrement=dec, e0=e0, e1=e1)
    if kind == "step":
        state["sim"].step()
        return state["sim"].positions()
    if kind == "batch":
        b = state["batch"]
        b.step()
        return np.concatenate([b.positions(k) for k in range(state["count"])])
    if kind == "pcg":
        c = state["case"]
        rowptr, col, vals, b = state["system"]
        x, _, _ = native.pcg_bsr3(rowptr, col, vals, b, c["tol"], c["cap"])
        return x
    p = {k: C.c_void_p(v.data_ptr()) for k, v in state.items() if torch.is_tensor(v)}
    n, stream = state["case"]["n"], C.c_void_p(torch.cuda.current_stream().cuda_stream)
    state["R"].copy_(state["eye"])  # the warm start, replaced by the fit
    lib = native.lib()
    native.check(lib.mfem_polar_batch(n, p["F"], p["R"], p["S"], p["dsdF"], p["it"], stream))
    native.check(lib.mfem_material_s6_batch(n, p["mat"], p["mu"], p["la"], p["s"], 1, p["E"],
                                            p["g"], p["H"], stream))
    return {k: state[k] for k in ("R", "S", "dsdF", "E", "g", "H")}


# --- work and tolerance ---------------------------------------------------------

def _counts(nx, ny, nz):
    """(vertices, elements, nonzero blocks per row) of a grid beam or sheet."""
    if nz == 0:
        return (nx + 1) * (ny + 1), 2 * nx * ny, 7
    return (nx + 1) * (ny + 1) * (nz + 1), 6 * nx * ny * nz, 15


def _iterations(case):
    """Linear-solver iterations of one Newton iteration (rounded, as counted
    with the present solvers on these scenes)."""
    size = max(case["nx"], case["ny"], case["nz"])
    solver = case["solver"]
    if solver == "eigen-llt":
        return 0
    if solver == "minres-indefinite-block":
        return case["cap"]
    if solver == "eigen-pcg-IC":
        return min(case["cap"], 8 + size // 2)
    if case["element"] == "tet_stiff":
        return case["cap"]
    return min(case["cap"], int((2 * size + 20) * max(1.0, math.log10(1 / case["tol"]) / 4)))


def work(case):
    kind = case["kind"]
    if kind == "elements":
        n = case["n"]
        return dict(bytes=n * 8.0 * (9 + 9 + 9 + 6 + 54 + 0.5 + 6 + 2.5 + 1 + 6 + 36), flops=n * 3000.0)
    if kind == "pcg":
        n = case["nx"] * case["ny"] * case["nz"]
        it = 25 * math.log10(1 / case["tol"])
        return dict(bytes=it * n * (15 * 76.0 + 3 * 8 * 8), flops=it * n * (15 * 18 + 30.0))
    if kind == "batch":
        r = 4 if case["precision"] == "mixed" else 8
        total = dict(bytes=0.0, flops=0.0)
        for nx, ny, nz in scenes.c4_beam_sizes(case["count"], 0):
            w = _newton_work(nx, ny, nz, r, 1.5 * nx + 30, True)
            total = {k: total[k] + 5 * w[k] for k in total}
        return total
    r = 4 if case["precision"] == "mixed" else 8
    w = _newton_work(case["nx"], case["ny"], case["nz"], r, _iterations(case),
                     KINDS[case["element"]][1])
    k = 5 if kind == "step" else 1
    if case["solver"] == "eigen-llt":
        n = 3 * _counts(case["nx"], case["ny"], case["nz"])[0]
        w = dict(bytes=w["bytes"] + 8.0 * n * n, flops=w["flops"] + n ** 3 / 3)
    return {q: k * v for q, v in w.items()}


def _newton_work(nx, ny, nz, r, iterations, mixed):
    """One Newton iteration: the mesh and the element state once, K written
    once, and per linear-solver iteration K and its columns and the solver's
    vectors once."""
    nv, nt, row = _counts(nx, ny, nz)
    element = 16 + 96 + 28 + (2 * (9 + 4 * 6) * 8 if mixed else 0)
    matrix = row * (9 * r + 4)
    return dict(bytes=nt * element + nv * (72.0 + matrix + iterations * (matrix + 3 * 6 * r)),
                flops=nt * 6000.0 + nv * iterations * (row * 18 + 36.0))


def tolerance(case):
    """About four times what the outputs move by when the CG dot products are
    summed in another order (other kernel shapes) or the start positions
    change in the last place, over the listed sizes and forty drawn ones."""
    kind = case["kind"]
    if kind == "elements":
        return {"rel": 2e-7}  # the fit stops at |gradient| < 1e-6: R is 5e-8 off the exact rotation
    if kind == "pcg":
        return {"rel": 20 * case["tol"]}  # x is 5 tol off the solution when CG stops
    if kind == "batch":
        return {"rel": 1e-9}  # positions of a converged step: 6e-12, 1e-10 on small beams
    stiff = case["element"] == "tet_stiff"
    if kind == "step":
        return {"rel": 1e-8 if stiff else 1e-9}  # 2e-9 and 1e-10
    if stiff:
        return {"rel": 4e-3, "max": 0.2}  # 1e-3, 5e-2: the 500th iterate of an unconverged CG
    return {"eigen-llt": {"rel": 1e-11},                # 2e-13
            "minres-indefinite-block": {"rel": 1e-4},   # 2e-5
            "eigen-pcg-IC": {"rel": 1e-5},              # 1e-7, and Jacobi CG's spread in dx
            "eigen-pcg-diag": {"rel": 4e-4},            # 1e-5 in dx, 1e-4 in the largest entry
            }[case["solver"]]


# --- the same in 64 bits with plain torch ----------------------------------------

_VOIGT3 = ((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2))
_VOIGT2 = ((0, 0), (1, 1), (0, 1))


def _f64(a):
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda").double()


def _polar(F):
    """Rotation R and symmetric stretch S of F = R S with det R = 1."""
    U, _, Vh = torch.linalg.svd(F.cpu())
    U, Vh = U.to(F.device), Vh.to(F.device)
    sign = torch.sign(torch.linalg.det(U) * torch.linalg.det(Vh))
    U = torch.cat([U[:, :, :-1], U[:, :, -1:] * sign[:, None, None]], 2)
    R = _mm(U, Vh)
    S = _mm(R.transpose(1, 2), F)
    return R, 0.5 * (S + S.transpose(1, 2))


def _mm(A, B):
    return (A[:, :, :, None] * B[:, None, :, :]).sum(2)


def _dsdF(R, F, S):
    """ds/dF (n, voigt, d, d): S + dS symmetric, F + dF = (R + dR)(S + dS), so
    with R^T dR = W skew, W S + S W = R^T dF - dF^T R and dS = R^T dF - W S."""
    n, d = F.shape[0], F.shape[1]
    voigt = _VOIGT3 if d == 3 else _VOIGT2
    out = torch.zeros(n, len(voigt), d, d, dtype=F.dtype, device=F.device)
    pairs = ((1, 2), (2, 0), (0, 1)) if d == 3 else ((1, 0),)
    tr = S.diagonal(dim1=1, dim2=2).sum(1)
    A = tr[:, None, None] * torch.eye(d, dtype=F.dtype, device=F.device) - S
    Ainv = torch.linalg.inv(A.cpu()).to(F.device) if d == 3 else None
    for i in range(d):
        for j in range(d):
            G = torch.zeros_like(F)
            G[:, :, j] = R[:, i, :]  # R^T E_ij
            Q = G - G.transpose(1, 2)
            W = torch.zeros_like(F)
            if d == 3:
                # skew matrices as vectors q_a = Q(c, b) for (b, c) = pairs[a]
                q = torch.stack([Q[:, c, b] for b, c in pairs], 1)
                w = (Ainv * q[:, None, :]).sum(2)
                for a, (b, c) in enumerate(pairs):
                    W[:, c, b] = w[:, a]
                    W[:, b, c] = -w[:, a]
            else:
                W[:, 1, 0] = Q[:, 1, 0] / tr
                W[:, 0, 1] = -W[:, 1, 0]
            dS = G - _mm(W, S)
            dS = 0.5 * (dS + dS.transpose(1, 2))
            for a, (p, q_) in enumerate(voigt):
                out[:, a, i, j] = dS[:, p, q_]
    return out


def _energy_of_s(mat, mu, la, s):
    """Psi(s) of symmetric stretch s in Voigt order, stable Neo-Hookean (0),
    Corot (2), FixedCorot (3) and ARAP (4)."""
    d = 3 if s.shape[1] == 6 else 2
    diag, off = s[:, :d], s[:, d:]
    if d == 3:
        a, b, c, f, e, g = s.unbind(1)
        J = a * b * c + 2 * f * e * g - a * g * g - b * e * e - c * f * f
    else:
        J = s[:, 0] * s[:, 1] - s[:, 2] ** 2
    n2 = (diag ** 2).sum(1) + 2 * (off ** 2).sum(1)
    dev = ((diag - 1) ** 2).sum(1) + 2 * (off ** 2).sum(1)
    tr = diag.sum(1) - d
    snh = 0.5 * mu * (n2 - d) - mu * (J - 1) + 0.5 * la * (J - 1) ** 2
    corot = 0.5 * la * tr ** 2 + mu * dev
    fixed = 0.5 * la * (J - 1) ** 2 + mu * dev
    return torch.where(mat == 0, snh, torch.where(mat == 2, corot,
                       torch.where(mat == 3, fixed, 0.5 * mu * dev)))


def _derivatives(psi, q):
    """Gradient and Hessian of psi (per element) at q (n, k)."""
    q = q.detach().requires_grad_(True)
    g = torch.autograd.grad(psi(q).sum(), q, create_graph=True)[0]
    rows = []
    for a in range(q.shape[1]):
        r = torch.autograd.grad(g[:, a].sum(), q, retain_graph=True, allow_unused=True)[0]
        rows.append(torch.zeros_like(q) if r is None else r)
    return g.detach(), torch.stack(rows, 1).detach()


def _project(H, floor, only=None):
    w, Q = torch.linalg.eigh(H.cpu())
    w, Q = w.to(H.device), Q.to(H.device)
    low = w[:, 0] < floor if only is None else (w[:, 0] < floor) & only
    P = _mm(Q * w.clamp(min=floor)[:, None, :], Q.transpose(1, 2))
    return torch.where(low[:, None, None], P, H)


class _Model:
    """One scene in plain torch: K and the residual of a Newton iteration at
    positions x (s on the constraint), and the energies along a step."""

    def __init__(self, sc):
        d = self.d = sc.V.shape[1]
        self.sc, self.mixed = sc, sc.mixed
        X, self.T = _f64(sc.V), torch.as_tensor(sc.T, device="cuda").long()
        self.mu, self.la = _f64(sc.mu), _f64(sc.la)
        self.mat = torch.as_tensor(sc.mat, device="cuda")
        Xc = X[self.T]
        Dm = (Xc[:, 1:] - Xc[:, :1]).transpose(1, 2)
        inv = torch.linalg.inv(Dm.cpu()).to(X.device)
        self.dphi = torch.cat([-inv.sum(1, keepdim=True), inv], 1)  # (n, d + 1, d)
        det = torch.linalg.det(Dm.cpu()).abs().to(X.device)
        self.vol = det / 6 if d == 3 else det
        self.mass = sc.density * self.vol / (20 if d == 3 else 12)
        self.h = sc.dt
        self.grav = _f64(np.asarray(sc.gravity[:d], dtype=np.float32))
        self.free = torch.as_tensor(sc.fixed == 0, device="cuda")
        self.dofs = self.free[:, None].expand(-1, d).reshape(-1)

    def F(self, x):
        return (x[self.T][:, :, :, None] * self.dphi[:, :, None, :]).sum(1)

    def inertia(self, x, xt):
        r = (x - xt - self.h ** 2 * self.grav)[self.T]
        return r, self.mass[:, None, None] * (r + r.sum(1, keepdim=True))

    def system(self, x, xt):
        n, d, k = self.T.shape[0], self.d, self.d + 1
        F = self.F(x)
        h2 = self.h ** 2
        if self.mixed:
            R, S = _polar(F)
            voigt = _VOIGT3 if d == 3 else _VOIGT2
            s = torch.stack([S[:, a, b] for a, b in voigt], 1)
            g, H = _derivatives(lambda q: _energy_of_s(self.mat, self.mu, self.la, q), s)
            H = _project(H, 1e-6, self.mat == 0)
            D = _dsdF(R, F, S)  # (n, m, d, d)
            self.s, self.D = s, D
        else:
            g, H = _derivatives(lambda q: self.psi_F(q.reshape(n, d, d)), F.reshape(n, d * d))
            H = _project(H, 0.0) if d == 3 else H
            D = torch.eye(d * d, dtype=F.dtype, device=F.device).reshape(1, d * d, d, d).expand(n, -1, -1, -1)
        self.g, self.H = h2 * g, h2 * H
        # B (n, m, k, d) = D : dF/dx
        B = (D[:, :, None, :, :] * self.dphi[:, None, :, None, :]).sum(-1)
        m = B.shape[1]
        B = B.reshape(n, m, k * d)
        HB = torch.zeros_like(B)
        for a in range(m):
            HB += self.H[:, :, a, None] * B[:, a, None, :]
        Ke = torch.zeros(n, k * d, k * d, dtype=F.dtype, device=F.device)
        for a in range(m):
            Ke += B[:, a, :, None] * HB[:, a, None, :]
        Ke *= self.vol[:, None, None]
        Me = (torch.ones(k, k) + torch.eye(k)).to(F)
        Ke += self.mass[:, None, None] * torch.kron(Me.cpu(), torch.eye(d).double()).to(F)
        f = -self.vol[:, None] * (B * self.g[:, :, None]).sum(1)
        f = f.reshape(n, k, d) - self.inertia(x, xt)[1]
        rhs = torch.zeros_like(x).index_add_(0, self.T.reshape(-1), f.reshape(-1, d))
        ids = (self.T[:, :, None] * d + torch.arange(d, device=x.device)).reshape(n, k * d)
        N = x.numel()
        keep = self.dofs[ids]
        Ke = torch.where(keep[:, :, None] & keep[:, None, :], Ke, torch.zeros_like(Ke))
        rows = ids[:, :, None].expand(-1, -1, k * d).reshape(-1)
        cols = ids[:, None, :].expand(-1, k * d, -1).reshape(-1)
        key, order = torch.sort(rows * N + cols)
        uniq, inverse = torch.unique_consecutive(key, return_inverse=True)
        vals = torch.zeros(uniq.numel(), dtype=x.dtype, device=x.device)
        vals.index_add_(0, inverse, Ke.reshape(-1)[order])
        crow = torch.zeros(N + 1, dtype=torch.int64, device=x.device)
        crow[1:] = torch.cumsum(torch.bincount(uniq // N, minlength=N), 0)
        return (crow, uniq % N, vals), (rhs * self.free[:, None]).reshape(-1)

    def psi_F(self, F):
        J = torch.linalg.det(F) if self.d == 3 else F[:, 0, 0] * F[:, 1, 1] - F[:, 0, 1] * F[:, 1, 0]
        if self.d == 3:
            J = (F[:, 0, 0] * (F[:, 1, 1] * F[:, 2, 2] - F[:, 1, 2] * F[:, 2, 1])
                 - F[:, 0, 1] * (F[:, 1, 0] * F[:, 2, 2] - F[:, 1, 2] * F[:, 2, 0])
                 + F[:, 0, 2] * (F[:, 1, 0] * F[:, 2, 1] - F[:, 1, 1] * F[:, 2, 0]))
        n2 = (F ** 2).sum((1, 2))
        return 0.5 * self.mu * (n2 - self.d) - self.mu * (J - 1) + 0.5 * self.la * (J - 1) ** 2

    def energy(self, x, xt, dx, alpha):
        """E(alpha) along dx after system(x): for the mixed method with ds and
        the multipliers of the eliminated step (ds = dS since s = S(x))."""
        xa = x + alpha * dx
        r, Mr = self.inertia(xa, xt)
        e = 0.5 * (r * Mr).sum()
        F = self.F(xa)
        if not self.mixed:
            return e + self.h ** 2 * (self.vol * self.psi_F(F)).sum()
        y = (self.D * self.F(dx)[:, None]).sum((2, 3))
        sa = self.s + alpha * y
        lam = -(self.g + (self.H * y[:, None, :]).sum(2))  # with the shear weights in
        S = _polar(F)[1]
        voigt = _VOIGT3 if self.d == 3 else _VOIGT2
        c = torch.stack([S[:, a, b] for a, b in voigt], 1) - sa
        e = e + self.h ** 2 * (self.vol * _energy_of_s(self.mat, self.mu, self.la, sa)).sum()
        return e - (self.vol * (lam * c).sum(1)).sum()


def _cg(A, b, tol, cap):
    """Jacobi CG in 64 bits on CSR arrays."""
    crow, col, vals = A
    K = torch.sparse_csr_tensor(crow, col, vals, size=(b.numel(), b.numel()))
    rows = torch.repeat_interleave(torch.arange(b.numel(), device=b.device), crow[1:] - crow[:-1])
    diag = torch.zeros_like(b)
    on = rows == col
    diag[rows[on]] = vals[on]
    dinv = torch.where(diag != 0, 1.0 / diag, torch.ones_like(diag))
    x, r = torch.zeros_like(b), b.clone()
    z = dinv * r
    p, rz, stop = z.clone(), torch.dot(r, z), tol ** 2 * torch.dot(b, b)
    for it in range(cap):
        q = torch.mv(K, p)
        a = rz / torch.dot(p, q)
        x += a * p
        r -= a * q
        if it % 16 == 15 and bool(torch.dot(r, r) < stop):
            break
        z = dinv * r
        rz, old = torch.dot(r, z), rz
        p = z + (rz / old) * p
    return x


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        return None  # every beam by itself takes longer than the others together
    if kind == "pcg":
        rowptr, col, vals, b = _pcg_system(case, seed)
        n = rowptr.numel() - 1
        cnt = (rowptr[1:] - rowptr[:-1]).long()
        ri = torch.repeat_interleave(torch.arange(n, device=b.device), cnt)
        k = torch.arange(3, device=b.device)
        rows = (3 * ri[:, None, None] + k[None, :, None]).expand(-1, 3, 3).reshape(-1)
        cols = (3 * col.long()[:, None, None] + k[None, None, :]).expand(-1, 3, 3).reshape(-1)
        order = torch.argsort(rows * (3 * n) + cols)
        crow = torch.zeros(3 * n + 1, dtype=torch.int64, device=b.device)
        crow[1:] = torch.cumsum(torch.bincount(rows, minlength=3 * n), 0)
        return _cg((crow, cols[order], vals[order]), b, 1e-14, 4000)
    if kind == "elements":
        e = _element_inputs(case, seed)
        n = case["n"]
        F = e["F"].reshape(n, 3, 3).transpose(1, 2)
        R, S = _polar(F)
        D = _dsdF(R, F, S)
        g, H = _derivatives(lambda q: _energy_of_s(e["mat"], e["mu"], e["la"], q), e["s"])
        H = _project(H, 1e-6, e["mat"] == 0)
        s = torch.stack([S[:, a, b] for a, b in _VOIGT3], 1)
        # column-major layouts of the entry points
        return dict(R=R.transpose(1, 2).reshape(n, 9), S=s,
                    dsdF=D.permute(0, 3, 2, 1).reshape(n, 54),
                    E=_energy_of_s(e["mat"], e["mu"], e["la"], e["s"]), g=g,
                    H=H.transpose(1, 2).reshape(n, 36))
    elements = _counts(case["nx"], case["ny"], case["nz"])[1]
    if elements > 450_000:
        return None  # over 20 s
    sc = _scene(case, seed)
    M = _Model(sc)
    x = _f64(sc.x0 if sc.x0 is not None else sc.V)
    xt = x + sc.dt * _f64(sc.v0)
    if kind == "newton":
        A, rhs = M.system(x, xt)
        if case["element"] == "tet_stiff":
            # the solver ends at its iteration cap, far from the solution
            return dict(dx=None, e0=float(M.energy(x, xt, torch.zeros_like(x), 0.0)))
        dx = _cg(A, rhs, 1e-13, 60000).reshape(x.shape)
        e0, e1 = float(M.energy(x, xt, dx, 0.0)), float(M.energy(x, xt, dx, 1.0))
        full = torch.zeros(x.shape[0], 3, dtype=x.dtype, device=x.device)
        full[:, :M.d] = dx
        # the decrement is the largest entry of dx and of the stretch step
        big = float(dx.abs().max())
        if M.mixed:
            big = max(big, float((M.D * M.F(dx)[:, None]).sum((2, 3)).abs().max()))
        return dict(dx=full[M.free].reshape(-1), decrement=big, e0=e0, e1=e1)
    for _ in range(12):
        A, rhs = M.system(x, xt)
        dx = _cg(A, rhs, 1e-8, 5000).reshape(x.shape)
        x = x + dx
        if float(dx.abs().max()) < 1e-9:
            break
    return x
