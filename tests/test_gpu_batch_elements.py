"""Batched element entry points at the edges of a wave and of the half wave in
which their records pass through LDS, and the rotation fit's shared trials (the
lanes of a wave evaluate the trials of the elements that need many). Needs an
MI355X.

Records against the oracle with the bounds of the element-level parity tests.
Shared trials against the same elements one to a launch, where a lane has no
helpers: both form the same trials (w shrunk by one product after the other, as the
lane itself would) and accept by one rule, so iteration counts are equal; different
contractions of the two loops leave R equal to 100 applied rotations of a rounding
of 1e-16 each, 1e-12."""
import numpy as np
import pytest

from mfem_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 31, 32, 33, 63, 64, 65])
def test_records_at_wave_edges(n, oracle):
    from mfem_amd import native
    check_records(native, oracle, n, range(n), range(n))


# the lines from which records pass through LDS: 128 (material) and 65536 (fit)
@pytest.mark.parametrize("n", [127, 128, 129, 160, 65535, 65536, 65537, 65567, 65568, 65569])
def test_records_at_the_staging_lines(n, oracle):
    from mfem_amd import native
    tail = range(max(0, n - 130), n)
    check_records(native, oracle, n, tail if n > 1000 else range(n), tail)


def check_records(native, oracle, n, fits, materials):
    rng = np.random.RandomState(n)
    F = np.eye(3) + 0.15 * rng.uniform(-1, 1, (n, 3, 3))
    mu, la = scenes.enu_to_lame(1e6, 0.45)
    S = np.array([1, 1, 1, 0, 0, 0.0]) + 0.2 * rng.uniform(-1, 1, (n, 6))
    R, s, dsdF, it = native.polar_batch(F)
    E, g, H = native.material_s6_batch(0, mu, la, S)
    for i in fits:
        Ro, so, do, _, ito = oracle.polar_svd3(F[i])
        assert it[i] == ito
        assert np.abs(R[i] - Ro).max() < 1e-12 and np.abs(s[i] - so).max() < 1e-12
        assert np.abs(dsdF[i] - do).max() < 1e-10 * np.abs(do).max()
    for i in materials:
        Eo, go, Ho = oracle.material_s6(0, mu, la, S[i], True)
        assert abs(E[i] - Eo) <= 1e-12 * max(abs(Eo), mu)
        assert np.abs(g[i] - go).max() <= 1e-12 * max(np.abs(go).max(), mu)
        assert np.abs(H[i] - Ho).max() <= 1e-9 * np.abs(Ho).max(), i


@pytest.mark.parametrize("n,wild", [(1, 1), (64, 1), (64, 64), (65, 13), (190, 40)])
def test_shared_trials_equal_single_launches(n, wild):
    from mfem_amd import native
    rng = np.random.RandomState(n + wild)
    F = np.eye(3) + 0.1 * rng.randn(n, 3, 3)
    Q, _ = np.linalg.qr(rng.randn(n, 3, 3))
    Q *= np.sign(np.linalg.det(Q))[:, None, None]
    R0 = np.tile(np.eye(3), (n, 1, 1))
    far = rng.choice(n, wild, replace=False)
    # stretched elements whose fit is far from their warm start
    F[far] = Q[far] @ np.diag([5.0, 2.0, 0.7]) @ np.swapaxes(np.roll(Q, 1, 0)[far], 1, 2)
    R, s, _, it = native.polar_batch(F, R0)
    assert np.isfinite(R).all() and (wild < 13 or it.max() > 5)
    for e in range(n) if n <= 65 else far:
        R1, s1, _, it1 = native.polar_batch(F[e:e + 1], R0[e:e + 1])
        assert it1[0] == it[e], e
        assert np.abs(R1[0] - R[e]).max() < 1e-12 and np.abs(s1[0] - s[e]).max() < 1e-11, e


@pytest.mark.parametrize("n", [(6, 3, 3), (20, 8, 8)])
def test_energy_of_torn_elements(n, oracle):
    """The energy of trials 30 to 1000 steps out, where elements are torn and
    inverted and their rotation fits far from the warm start: the lanes of a wave
    share the trials there. Against the oracle, to the fit's own tolerance (R to
    1e-6)."""
    from mfem_amd import native
    sc = scenes.beam_scene(*n, seed=1, mixed=True, E=1e4, itr_tol=1e-12, max_iters=5000)
    g, o = native.Sim(sc, precision="fp64"), oracle.Sim(sc)
    for sim in (g, o):
        sim.update_system()
        sim.solve()
    dx, free = g.get("dx").reshape(-1, 3), sc.fixed == 0
    x = sc.V.copy()
    x[free] += 1000 * dx
    D = np.stack([x[sc.T[:, j]] - x[sc.T[:, 0]] for j in (1, 2, 3)], 1)
    assert (np.linalg.det(D) < 0).mean() > 0.01  # inverted
    for alpha in (30.0, 100.0, 300.0, 1000.0):
        want = o.energy(alpha)
        assert abs(g.energy(alpha) - want) < 1e-6 * abs(want), alpha
