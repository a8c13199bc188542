"""GPU parity of "minres-indefinite-block" against the FP64 oracle (needs an
MI355X).

The device KKT product, right-hand side and block preconditioner are compared
with the oracle's on the same state (relative 1e-11 at the shared initial
state, where both sides hold the same data); MINRES by its iterates over a
fixed number of iterations (1e-9), by its iteration count at the default
tolerance (within 5%: see the test) and by whole timesteps. Positions after
timesteps agree to 1e-7 relative to the displacement: both loops stop at the
same Newton tolerance with solves converged to 1e-10.
"""
import numpy as np
import pytest

from mfem_amd import scenes

pytestmark = pytest.mark.gpu

SOLVER = "minres-indefinite-block"


@pytest.fixture(scope="module")
def native():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a visible MI355X"
    from mfem_amd import native as N
    N.lib()
    return N


def relerr(a, b):
    a, b = np.asarray(a), np.asarray(b)
    return float(np.abs(a - b).max() / max(np.abs(b).max(), 1e-300))


def _scene(material="Stable-Neohookean", **kw):
    base = dict(seed=4, mixed=True, solver=SOLVER, max_newton=5, material=material)
    base.update(kw)
    return scenes.beam_scene(3, 2, 2, **base)


@pytest.mark.parametrize("material", ["Stable-Neohookean", "Fung"])
def test_kkt_operator_matches_oracle(native, oracle, material):
    sc = _scene(material, v0=None)
    print(f"kkt operator: {material}, nT={sc.nT}", flush=True)
    dev = native.Sim(sc, precision="fp64")
    ref = oracle.Sim(sc)
    dev.update_system()
    ref.update_system()
    N = ref.kkt_size()
    assert dev.kkt_size() == N
    rng = np.random.default_rng(0)
    for _ in range(3):
        w = rng.standard_normal(N)
        assert relerr(dev.kkt_apply(0, w), ref.kkt_product(w)) < 1e-11
        assert relerr(dev.kkt_apply(1, w), ref.kkt_precond(w, False)) < 1e-11
    b_dev, b_ref = dev.kkt_apply(2), ref.kkt_rhs()
    assert np.abs(b_ref).max() > 0
    assert relerr(b_dev, b_ref) < 1e-11


def test_kkt_operator_after_motion(native, oracle):
    """After two tightly solved timesteps (lambda, ds and S - s nonzero)."""
    sc = _scene(itr_tol=1e-10, max_iters=20000)
    dev = native.Sim(sc, precision="fp64")
    ref = oracle.Sim(sc, solver=2)
    for _ in range(2):
        dev.step()
        ref.step()
    disp = np.abs(ref.positions() - sc.V).max()
    assert np.abs(dev.positions() - ref.positions()).max() < 1e-7 * disp
    dev.update_system()
    ref.update_system()
    b_ref = ref.kkt_rhs()
    N = ref.kkt_size()
    n = N - 12 * sc.nT
    assert np.abs(b_ref[n + 6 * sc.nT:]).max() > 0  # constraint residual present
    assert relerr(dev.kkt_apply(2), b_ref) < 1e-5
    w = np.random.default_rng(1).standard_normal(N)
    assert relerr(dev.kkt_apply(0, w), ref.kkt_product(w)) < 1e-6


@pytest.mark.parametrize("material", ["Stable-Neohookean", "ARAP"])
def test_minres_fixed_iterations_match_oracle(native, oracle, material):
    """30 iterations of the recurrence (tolerance 0): the iterates agree to
    rounding. Further on, Lanczos loses orthogonality and the two summation
    orders drift apart (the oracle against a numpy restatement of the same
    recurrence on the same matrices: 3e-13 at 40 iterations, 1e-2 at 80)."""
    sc = _scene(material, max_newton=1, itr_tol=1e-300, max_iters=30)
    dev = native.Sim(sc, precision="fp64")
    ref = oracle.Sim(sc)
    dev.update_system()
    ref.update_system()
    dev.solve()
    ref.solve()
    assert dev.get_int("pcg_iters")[0] == ref.get_int("pcg_iters", 1)[0] == 30
    for name in ("dx", "ds", "lambda"):
        assert relerr(dev.get(name), ref.get(name)) < 1e-9, name


@pytest.mark.parametrize("material", ["Stable-Neohookean", "ARAP"])
def test_minres_converged_solve_matches_oracle(native, oracle, material):
    """A solve to the default tolerance 1e-4. The iteration count depends on
    rounding once orthogonality is lost (the oracle's C loops and a numpy
    restatement of the same recurrence on the same matrices stop at 539 and
    528 iterations on this beam; eight shuffled summation orders give
    526-528), so counts agree to 5%, and the solutions to the accuracy the
    tolerance gives (dx within 2e-3 of the exact KKT solution here)."""
    sc = _scene(material, max_newton=1, itr_tol=1e-4, max_iters=5000)
    dev = native.Sim(sc, precision="fp64")
    ref = oracle.Sim(sc)
    dev.update_system()
    ref.update_system()
    dev.solve()
    ref.solve()
    it_dev = dev.get_int("pcg_iters")[0]
    it_ref = ref.get_int("pcg_iters", 1)[0]
    print(f"minres iterations {material}: device {it_dev}, oracle {it_ref}", flush=True)
    assert it_ref > 10
    assert abs(it_dev - it_ref) <= max(3, 0.05 * it_ref)
    for name in ("dx", "ds", "lambda"):
        assert relerr(dev.get(name), ref.get(name)) < 1e-2, name


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-7), ("mixed", 1e-6)])
def test_minres_timesteps_match_oracle(native, oracle, precision, tol):
    sc = _scene(itr_tol=1e-10, max_iters=20000)
    dev = native.Sim(sc, precision=precision)
    ref = oracle.Sim(sc, solver=2)
    for k in range(3):
        print(f"minres timestep {k} ({precision})", flush=True)
        dev.step()
        ref.step()
        disp = np.abs(ref.positions() - sc.V).max()
        assert disp > 1e-4
        assert np.abs(dev.positions() - ref.positions()).max() < tol * disp


def test_minres_matches_schur_path(native):
    """Both device solvers, solved tightly, give the same timesteps."""
    kw = dict(itr_tol=1e-10, max_iters=20000)
    a = native.Sim(_scene(**kw), precision="fp64")
    b = native.Sim(_scene(solver="eigen-pcg-diag", **kw), precision="fp64")
    for _ in range(3):
        a.step()
        b.step()
    disp = np.abs(b.positions() - b.scene.V).max()
    assert disp > 1e-4
    assert np.abs(a.positions() - b.positions()).max() < 1e-7 * disp


def test_minres_errors(native):
    with pytest.raises(native.MfemError):
        native.Sim(_scene(mixed=False), precision="fp64")
    cg = native.Sim(_scene(solver="eigen-pcg-diag"), precision="fp64")
    with pytest.raises(native.MfemError):
        cg.kkt_size()


# ---- 2D (triangles, 3-vector s): the DIM = 2 instance of the same solver
def _scene2d(material="Stable-Neohookean", **kw):
    base = dict(solver=SOLVER, max_newton=5)
    base.update(kw)
    sc = scenes.rect2d_scene(6, 3, 0.1, **base)
    sc.mixed = True
    if material != "Stable-Neohookean":
        sc.mat[:] = scenes.MATERIALS[material]
    return sc


def _dx2(dev):
    """Device dx (3 per free vertex, z rows zero) in the reference's 2D layout."""
    d = dev.get("dx").reshape(-1, 3)
    assert not d[:, 2].any()
    return d[:, :2].reshape(-1)


@pytest.mark.parametrize("moved", [False, True])
def test_kkt_operator_2d_matches_oracle(native, oracle, moved):
    sc = _scene2d(itr_tol=1e-10, max_iters=20000)
    print(f"kkt operator 2d: moved={moved}, nT={sc.nT}", flush=True)
    dev = native.Sim(sc, precision="fp64")
    ref = oracle.Sim(sc)
    if moved:
        for _ in range(2):
            dev.step()
            ref.step()
    dev.update_system()
    ref.update_system()
    N = ref.kkt_size()
    assert dev.kkt_size() == N == 2 * int((ref.get_int("free_map", sc.nV) >= 0).sum()) + 6 * sc.nT
    tol = 1e-6 if moved else 1e-11  # after motion the states differ by the solves' rounding
    rng = np.random.default_rng(2)
    for _ in range(3):
        w = rng.standard_normal(N)
        assert relerr(dev.kkt_apply(0, w), ref.kkt_product(w)) < tol
        assert relerr(dev.kkt_apply(1, w), ref.kkt_precond(w, False)) < tol
    b_ref = ref.kkt_rhs()
    assert np.abs(b_ref).max() > 0
    assert relerr(dev.kkt_apply(2), b_ref) < (1e-5 if moved else 1e-11)


@pytest.mark.parametrize("material", ["Stable-Neohookean", "ARAP"])
def test_minres_2d_fixed_iterations_match_oracle(native, oracle, material):
    sc = _scene2d(material, max_newton=1, itr_tol=1e-300, max_iters=30)
    print(f"minres 2d fixed iterations: {material}", flush=True)
    dev = native.Sim(sc, precision="fp64")
    ref = oracle.Sim(sc)
    dev.update_system()
    ref.update_system()
    dev.solve()
    ref.solve()
    assert dev.get_int("pcg_iters")[0] == ref.get_int("pcg_iters", 1)[0] == 30
    assert relerr(_dx2(dev), ref.get("dx")) < 1e-9
    for name in ("ds", "lambda"):
        assert relerr(dev.get(name), ref.get(name)) < 1e-9, name


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-7), ("mixed", 1e-6)])
def test_minres_2d_timesteps_match_oracle(native, oracle, precision, tol):
    sc = _scene2d(itr_tol=1e-10, max_iters=20000)
    dev = native.Sim(sc, precision=precision)
    ref = oracle.Sim(sc, solver=2)
    for k in range(3):
        print(f"minres 2d timestep {k} ({precision})", flush=True)
        dev.step()
        ref.step()
        disp = np.abs(ref.positions() - sc.V[:, :2]).max()
        assert disp > 1e-4
        assert np.abs(dev.positions()[:, :2] - ref.positions()).max() < tol * disp


@pytest.mark.parametrize("nx,ny,nz", [(5, 3, 3), (50, 17, 17), (60, 19, 19)])
def test_minres_alpha_sum_on_both_sides_of_its_line(native, oracle, nx, ny, nz):
    """alpha is summed inside the preconditioner kernel up to 1024 partials
    (270 tets: 1 chunk of 64; 87k tets: 12), by a kernel of its own above (130k).
    Four iterations against the oracle: each sum of n = 3e5..1e6 terms rounds to
    sqrt(n) 1e-16 < 1e-12 of its terms' size, and few iterations amplify that by
    less than the 1e3 left to the bar."""
    sc = scenes.beam_scene(nx, ny, nz, seed=4, mixed=True, solver=SOLVER, max_newton=1,
                           itr_tol=1e-300, max_iters=4)
    print(f"minres alpha: nT={sc.nT}", flush=True)
    dev = native.Sim(sc, precision="fp64")
    ref = oracle.Sim(sc)
    for sim in (dev, ref):
        sim.update_system()
        sim.solve()
    for name in ("dx", "ds", "lambda"):
        assert relerr(dev.get(name), ref.get(name)) < 1e-9, name
