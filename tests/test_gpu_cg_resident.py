"""The CG with the system resident in registers (one cooperative launch per
solve) against the one-kernel-per-iteration CG, which set_cg_shape selects, on
the same system: every kernel of its dispatch (row lengths up to 8, 16, 32 and
64 blocks, passes of rows, both precisions) at sizes around the edges of the
workgroup rule. Needs an MI355X.

Bars: both run Eigen's iteration from the same data and differ in the order of
their sums only. Converged to 1e-12 (FP64; defect-corrected to 1e-10 in mixed
precision), dx agrees to 1e-8, about the tolerance times the condition of
these systems; iteration counts may differ by the few steps that rounding
moves a residual of 1e-12 |b| by (2%; in mixed precision a different
rounding also changes where the defect-correction sweeps end, so the total is
not compared).
"""
import json
import os

import numpy as np
import pytest

from mfem_amd import meshio, scenes

pytestmark = pytest.mark.gpu
GOLDEN = os.path.join(os.path.dirname(__file__), "golden")


@pytest.fixture(scope="module")
def native():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a visible MI355X"
    from mfem_amd import native as N
    N.lib()
    return N


def solve(native, sc, precision, shape=None):
    g = native.Sim(sc, precision=precision)
    if shape is not None:
        g.set_cg_shape(shape)
    g.update_system()
    g.solve()
    return g.get("dx"), int(g.get_int("pcg_iters")[0]), g


def paths(g):
    """How this simulation's CG solves ran (a refused, unfitting or expired
    resident launch counts as one by launches too)."""
    return dict(zip(("resident", "refused", "no_fit", "expired", "launches"),
                    map(int, g.get_int("cg_paths"))))


def compare(native, sc, precision, path="resident"):
    """The default path, which has to be `path`, against the launches."""
    sc.itr_tol = 1e-12 if precision == "fp64" else 1e-10
    sc.max_iters = 20000
    a, ia, g = solve(native, sc, precision)
    b, ib, h = solve(native, sc, precision, 0)
    got, other = paths(g), paths(h)
    assert got.pop(path) > 0 and other.pop("launches") > 0
    if path == "no_fit":  # found at the first sweep, which launches took over
        assert got.pop("launches") > 0
    assert not any(got.values()) and not any(other.values()), (got, other)
    assert np.isfinite(a).all() and np.abs(b).max() > 0
    assert np.abs(a - b).max() / np.abs(b).max() < 1e-8
    if precision == "fp64":
        assert abs(ia - ib) <= max(3, 0.02 * ib), (ia, ib)
    return g


# 1 row per workgroup .. the last size on one XCD, the first over all of them,
# then 1, 2, 3 and 5 (FP64) or 2, 4 and 6 (mixed) passes of rows
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [(1, 1, 1), (2, 1, 2), (7, 3, 3), (32, 7, 7), (33, 7, 7), (41, 19, 20),
                               (61, 22, 22), (60, 24, 24), (81, 25, 25), (90, 30, 30)])
def test_beams(native, n, precision):
    compare(native, scenes.beam_scene(*n, seed=5, mixed=n[0] % 2 == 0), precision,
            # 86k rows are past the FP64 kernels
            "resident" if precision == "mixed" or n[0] < 90 else "launches")


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [(9, 4), (270, 60), (270, 61), (400, 120), (500, 160), (700, 150),
                               (900, 170), (900, 220)])
def test_sheets(native, n, precision):
    # 154k and 199k rows are past the FP64 kernels
    compare(native, scenes.rect2d_scene(*n), precision,
            "resident" if precision == "mixed" or n[0] < 900 else "launches")


def cloud_scene(points, seed, hub=0):
    """Delaunay mesh of jittered grid points: rows of up to ~30 blocks; with
    `hub`, points on a sphere around one vertex instead: a row of hub + 1."""
    from scipy.spatial import Delaunay
    rng = np.random.RandomState(seed)
    if hub:
        k = np.arange(hub) + 0.5
        phi, th = np.arccos(1 - 2 * k / hub), np.pi * (1 + 5 ** 0.5) * k
        P = np.vstack([[0.01, 0.02, 0.0], np.stack([np.cos(th) * np.sin(phi),
                                                    np.sin(th) * np.sin(phi), np.cos(phi)], 1)])
    else:
        P = np.stack(np.meshgrid(*[np.arange(points)] * 3, indexing="ij"), -1).reshape(-1, 3)
        P = P + rng.uniform(-0.35, 0.35, P.shape)
    T = Delaunay(P).simplices.astype(np.int32)
    D = np.stack([P[T[:, j]] - P[T[:, 0]] for j in (1, 2, 3)], 1)
    v = np.linalg.det(D)
    T = T[np.abs(v) > 1e-3]
    v = v[np.abs(v) > 1e-3]
    T[v < 0] = T[v < 0][:, [0, 2, 1, 3]]
    used = np.unique(T)
    renum = np.full(P.shape[0], -1, dtype=np.int32)
    renum[used] = np.arange(used.size)
    V, T = P[used] * 0.1, renum[T]
    mu, la = scenes.enu_to_lame(np.full(T.shape[0], 1e6), 0.45)
    fixed = scenes.bc_fixed("hangends", V, axis=0, ratio=0.2)
    return scenes.Scene(V=V, T=T, mu=mu, la=la, mat=np.zeros(T.shape[0], dtype=np.int32),
                        fixed=fixed, mixed=False)


# rows longer than 16 (any Delaunay mesh), than 32 (a hub of 50) and than 64
# (no kernel: the iteration falls back); 16^3 points pass 16 rows per workgroup
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("points,hub", [(6, 0), (16, 0), (27, 0), (0, 50), (0, 90)])
def test_long_rows(native, points, hub, precision):
    sc = cloud_scene(points, 3, hub)
    rows = np.diff(native.Sim(sc).get_int("bsr_rowptr"))
    assert rows.max() > (hub * 0.6 if hub else 16)
    # 64 or 32 rows a pass on 248 workgroups, 2 (FP64) or 4 passes
    room = 248 * (64 if rows.max() <= 32 else 32) * (2 if precision == "fp64" else 4)
    compare(native, sc, precision,
            "resident" if rows.max() <= 64 and rows.size <= room else "launches")


def shuffled(sc, seed):
    """The same mesh with its vertices in random order: rows of a workgroup then
    touch columns all over the mesh."""
    perm = np.random.RandomState(seed).permutation(sc.nV)
    inv = np.empty_like(perm)
    inv[perm] = np.arange(sc.nV)
    sc.V, sc.fixed, sc.T = sc.V[perm], sc.fixed[perm], inv[sc.T].astype(np.int32)
    return sc


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_columns_that_do_not_fit(native, precision):
    """37.5k rows, 152 a workgroup, in random order: some 2000 columns a workgroup,
    and 1365 have room. Every workgroup leaves at the start."""
    g = compare(native, shuffled(scenes.beam_scene(60, 24, 24, seed=5), 1), precision, "no_fit")
    g.update_system()
    g.solve()  # known now: not tried again
    assert paths(g)["no_fit"] == 1 and paths(g)["resident"] == 0


def test_caller_columns_that_do_not_fit(native):
    """The same through mfem_pcg_bsr3: 40k rows of 13 blocks at random distances.
    The residual of x itself, to the rounding of K x (about 1e-14)."""
    import torch
    rng = np.random.RandomState(2)
    n, i = 40000, np.arange(40000)
    A = 0.2 * rng.randn(6, n, 3, 3)
    W = A @ A.transpose(0, 1, 3, 2) + 0.3 * np.eye(3)
    far = rng.choice(np.arange(100, n // 2 - 100), 6, replace=False)
    to = [(i + o) % n for o in far]
    diag = np.tile(1e-2 * np.eye(3), (n, 1, 1))
    for w, j in zip(W, to):
        diag += w
        diag[j] += w
    rows = np.concatenate([i] + [i] * 6 + to)
    cols = np.concatenate([i] + to + [i] * 6)
    vals = np.concatenate([diag] + [-w for w in W] * 2)
    order = np.lexsort((cols, rows))
    rows, cols, vals = rows[order], cols[order], vals[order]
    rowptr = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))]).astype(np.int32)
    b = rng.randn(n, 3)
    dev = [torch.as_tensor(np.ascontiguousarray(a), device="cuda")
           for a in (rowptr, cols.astype(np.int32), vals.reshape(-1), b.reshape(-1))]
    x, it, rr = native.pcg_bsr3(*dev, 1e-9, 5000)
    x = x.cpu().numpy().reshape(-1, 3)
    r = b.copy()
    np.subtract.at(r, rows, (vals @ x[cols][:, :, None])[:, :, 0])
    assert 0 < it < 5000 and rr < 1e-9
    true = np.linalg.norm(r) / np.linalg.norm(b)
    assert abs(true - rr) < 1e-14 * np.abs(vals).sum((1, 2)).max() * np.linalg.norm(x) / np.linalg.norm(b) * it


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_matches_the_oracle(native, oracle, precision):
    sc = scenes.beam_scene(8, 3, 3, seed=7, mixed=True, E_range=(1e5, 1e6), itr_tol=1e-12,
                           max_iters=20000)
    o = oracle.Sim(sc)
    o.update_system()
    o.solve()
    dx, it, g = solve(native, sc, precision)
    assert paths(g)["resident"] > 0 and paths(g)["launches"] == 0
    ref = o.get("dx")
    # mixed: K itself is stored in FP32 (2^-24 = 6e-8 an entry), and a solve
    # amplifies that by at most the scaled condition, about 1e2 here
    bar = 1e-9 if precision == "fp64" else 1e2 * 2.0 ** -24
    assert np.abs(dx - ref).max() / np.abs(ref).max() < bar


def test_stopping_rule(native):
    """The iteration cap, and zero iterations for |b|^2 below tol^2 |b|^2."""
    for kw, want in ((dict(max_iters=3), 3), (dict(max_iters=1), 1), (dict(itr_tol=2.0), 0)):
        sc = scenes.beam_scene(8, 3, 3, seed=7, mixed=True, **kw)
        a, ia, g = solve(native, sc, "fp64")
        b, ib, _ = solve(native, sc, "fp64", 0)
        assert paths(g)["resident"] == 1
        assert ia == ib == want
        assert np.allclose(a, b, rtol=0, atol=1e-12 * max(1.0, np.abs(b).max()))


def test_expired_wait_falls_back(native, tmp_path):
    """With no time to wait for each other the workgroups leave, and the solve
    runs as one kernel per iteration: the same step."""
    scene = json.load(open(os.path.join(GOLDEN, "beam_scene.json")))
    scene["objects"][0]["path"] = os.path.join(GOLDEN, scene["objects"][0]["path"])
    scene["linear_solver"] = "eigen-pcg-diag"
    out = []
    for wait in (2000, 0):
        scene["resident_wait_ms"] = wait
        path = tmp_path / f"scene{wait}.json"
        path.write_text(json.dumps(scene))
        g = native.Sim(json_path=str(path))
        for _ in range(2):
            g.step()
        out.append((g.positions(), g.stats()["newton_iters"]))
        p = paths(g)
        assert (p["expired"] > 0) == (p["launches"] > 0) == (wait == 0), p
    assert out[0][1] == out[1][1]
    assert np.abs(out[0][0] - out[1][0]).max() < 1e-8


def test_expired_waits_are_not_tried_every_solve(native, tmp_path):
    """64 solves by launches after the first expiry, 128 after the second."""
    g = native.Sim(json_path=scene_file(tmp_path, (40, 13, 13), resident_wait_ms=0,
                                        max_iterative_solver_iters=3))
    g.update_system()
    expired = []
    for k in range(200):
        g.solve()
        expired.append(paths(g)["expired"])
    assert paths(g)["launches"] == 200
    assert [k for k in range(200) if expired[k] > (expired[k - 1] if k else 0)] == [0, 65, 194]


def scene_file(tmp_path, n, **kw):
    """A beam of n cells as a scene file: what resident_wait_ms can be set in."""
    scene = json.load(open(os.path.join(GOLDEN, "beam_scene.json")))
    V, T = scenes.kuhn_beam(*n, 0.1, 0.1, 3)
    meshio.write_mesh(str(tmp_path / "beam.mesh"), V, T)
    scene["objects"][0]["path"] = str(tmp_path / "beam.mesh")
    scene.update(kw)
    path = tmp_path / "scene.json"
    path.write_text(json.dumps(scene))
    return str(path)


@pytest.mark.parametrize("cap", [1, 2, 3])
@pytest.mark.parametrize("n", [(3, 1, 1), (20, 6, 6), (40, 13, 13)])
def test_a_solve_is_whole_whoever_gives_up(native, tmp_path, n, cap):
    """Short solves in which a workgroup's wait may run out at any point, the
    last sums included: every row of the step is the iterate of a whole solve
    (1, 31 and 157 workgroups). Few iterations from the same data round alike:
    1e-12."""
    path = scene_file(tmp_path, n, resident_wait_ms=0, max_iterative_solver_iters=cap,
                      iterative_solver_tolerance=1e-30)

    def dx(shape):
        g = native.Sim(json_path=path)
        if shape is not None:
            g.set_cg_shape(shape)
        g.update_system()
        g.solve()
        expired.append(paths(g)["expired"])
        return g.get("dx"), int(g.get_int("pcg_iters")[0])

    expired = []
    want, iters = dx(0)
    assert np.abs(want).max() > 0 and iters == cap
    for _ in range(6):
        got, it = dx(None)
        assert it == cap
        assert n[0] < 40 or expired[-1] == 1  # over all XCDs the first one has to wait
        assert np.abs(got - want).max() < 1e-12 * np.abs(want).max()


@pytest.mark.parametrize("nb", [1, 40, 2000, 6000])
def test_solves_that_stop_at_once(native, nb):
    """b = 0, no iterations allowed, and a tolerance that b itself meets: x is 0
    in every row, whatever it held."""
    import torch
    rp = torch.arange(nb + 1, dtype=torch.int32, device="cuda")
    col = torch.arange(nb, dtype=torch.int32, device="cuda")
    K = (2.0 * torch.eye(3, dtype=torch.float64, device="cuda")).repeat(nb, 1, 1).reshape(-1)
    b = torch.ones(3 * nb, dtype=torch.float64, device="cuda")
    for rhs, tol, cap in ((0 * b, 1e-6, 10), (b, 1e-6, 0), (b, 2.0, 10)):
        x = torch.full_like(b, float("nan"))
        x, it, rr = native.pcg_bsr3(rp, col, K, rhs, tol, cap, x=x)
        assert it == 0 and rr == (1.0 if rhs is b else 0.0)
        assert not torch.any(x != 0)
    x, it, rr = native.pcg_bsr3(rp, col, K, b, 1e-12, 10)
    assert torch.equal(x, 0.5 * b)
    x, it, rr = native.pcg_bsr3(rp, col, K, b, 1e-12, 10, x=b)  # in place
    assert torch.equal(x, 0.5 * torch.ones_like(b))


@pytest.mark.parametrize("n", [(1, 1, 1), (4, 3, 2), (9, 7, 5), (20, 16, 13), (40, 40, 32)])
def test_caller_matrices(native, n):
    """mfem_pcg_bsr3 with the forms it accepts: columns in any order, a column
    twice in a row, rows without a diagonal block (a zero right-hand side
    there). The last size is past the resident CG's, and goes the other way.
    Against K x = b itself: the residual is what the call says it is, in the
    2-norm to the rounding of K x (1e-14 of |K||x| per product), and below
    tol."""
    import torch
    rng = np.random.RandomState(n[0])
    ids = np.arange(np.prod(n)).reshape(n)
    rows, cols, vals = [], [], []
    diag = np.tile(1e-2 * np.eye(3), (ids.size, 1, 1))
    for ax in range(3):
        i = ids.take(range(n[ax] - 1), axis=ax).ravel()
        j = ids.take(range(1, n[ax]), axis=ax).ravel()
        A = rng.randn(i.size, 3, 3)
        W = A @ A.transpose(0, 2, 1) + 0.3 * np.eye(3)
        np.add.at(diag, i, W)
        np.add.at(diag, j, W)
        rows += [i, j]
        cols += [j, i]
        vals += [-W, -W]
    bare = ids.ravel()[::17][1:]  # rows and columns without any block
    keep = np.ones(ids.size, dtype=bool)
    keep[bare] = False
    part = rng.rand(ids.size, 1, 1)  # the diagonal block in two pieces
    rows += [ids.ravel()[keep]] * 2
    cols += [ids.ravel()[keep]] * 2
    vals += [(part * diag)[keep], ((1 - part) * diag)[keep]]
    rows, cols, vals = np.concatenate(rows), np.concatenate(cols), np.concatenate(vals)
    on = keep[rows] & keep[cols]
    rows, cols, vals = rows[on], cols[on], vals[on]
    order = np.lexsort((rng.rand(rows.size), rows))
    rows, cols, vals = rows[order], cols[order], vals[order]
    rowptr = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=ids.size))]).astype(np.int32)
    b = rng.randn(ids.size, 3)
    b[bare] = 0.0
    dev = [torch.as_tensor(np.ascontiguousarray(a), device="cuda")
           for a in (rowptr, cols.astype(np.int32), vals.reshape(-1), b.reshape(-1))]
    tol = 1e-9
    x, it, rr = native.pcg_bsr3(*dev, tol, 20000)
    x = x.cpu().numpy().reshape(-1, 3)
    r = b.copy()
    np.subtract.at(r, rows, (vals @ x[cols][:, :, None])[:, :, 0])
    true = np.linalg.norm(r) / np.linalg.norm(b)
    assert np.isfinite(x).all() and it < 20000 and rr < tol
    assert abs(true - rr) < 1e-14 * np.abs(vals).sum((1, 2)).max() * np.linalg.norm(x) / np.linalg.norm(b) * max(it, 1)
    assert not np.any(x[bare])


# with up to 8 beams each takes the 32 workgroups of an XCD, with more the
# small ones (up to 1024 rows) share it in teams of 8; (60, 13, 13) is past the
# FP64 kernels' rows and sends that batch to the lockstep CG
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("sizes", [[(2, 1, 1)], [(20, 6, 6), (5, 2, 3), (33, 9, 8)],
                                   [(4 + k, 2 + k % 5, 2 + k % 7) for k in range(21)] +
                                   [(32, 5, 4), (31, 5, 4), (40, 11, 12), (50, 13, 12)],
                                   [(60, 13, 13), (12, 3, 3)]])
def test_batches(native, sizes, precision):
    kw = dict(itr_tol=1e-12 if precision == "fp64" else 1e-10, max_iters=20000, max_newton=3)
    scs = [scenes.beam_scene(*n, seed=k, E=10.0 ** (4 + k % 4), nu=0.3 + 0.02 * (k % 8), mixed=True,
                             **kw) for k, n in enumerate(sizes)]
    a, b = native.Batch(scs, precision=precision), native.Batch(scs, precision=precision)
    b.set_cg_shape(0, 64)
    for step in range(2):
        a.step()
        b.step()
        for k in range(a.count):
            xa, xb = a.positions(k), b.positions(k)
            # both converge to the same dx (1e-8 of it, see the bars above);
            # positions are of the order of the beam
            assert np.abs(xa - xb).max() < 1e-8 * np.abs(xb).max(), (step, k)
    # a resident solve is one submission, an iteration of the lockstep CG one each
    (_, ca, na), (_, cb, _) = a.launch_counts(), b.launch_counts()
    if precision == "fp64" and (60, 13, 13) in sizes:
        assert ca > 4 * na
    else:
        assert 4 * ca < cb and (ca == na or precision == "mixed")


@pytest.mark.parametrize("precision,n,count,resident", [
    ("fp64", (6, 3, 3), 32, True), ("fp64", (6, 3, 3), 1024, False),
    ("mixed", (6, 3, 3), 1024, False), ("mixed", (20, 7, 7), 16, True),
    ("mixed", (20, 7, 7), 320, False), ("fp64", (20, 6, 6), 128, True)])
def test_batch_takes_the_shorter_way(native, precision, n, count, resident):
    """Many small beams are few iterations in lockstep and many solves one after
    another for a team: from the second solve on, when the iterations are known, the
    batch goes the way that is shorter by a factor of two or so either way."""
    kw = dict(itr_tol=1e-8, max_iters=2000, max_newton=2, mixed=True)
    base = [scenes.beam_scene(*n, seed=k, E=10.0 ** (4 + k % 4), **kw) for k in range(8)]
    a, b = (native.Batch(base * (count // 8), precision=precision) for _ in range(2))
    b.set_cg_shape(0, 64)
    a.step()
    b.step()
    before = a.launch_counts()
    a.step()
    b.step()
    cg, newton = (x - y for x, y in zip(a.launch_counts()[1:], before[1:]))
    assert (cg <= 8 * newton) if resident else (cg > 20 * newton), (cg, newton)
    for k in (0, 7, count - 1):
        assert np.abs(a.positions(k) - b.positions(k)).max() < 1e-6 * np.abs(b.positions(k)).max()


def test_batch_of_many_beams_is_resident(native):
    """A beam's place on its team depends on its own rows, not on the batch's: 640
    beams of 980 rows, 627k in all. The first and last against the lockstep CG."""
    scs = [scenes.beam_scene(20, 6, 6, seed=k, E=10.0 ** (4 + k % 4), itr_tol=1e-12,
                             max_iters=20000, max_newton=1, mixed=True) for k in range(8)] * 80
    a, b = native.Batch(scs, precision="fp64"), native.Batch(scs, precision="fp64")
    b.set_cg_shape(0, 256)
    a.step()
    b.step()
    assert a.launch_counts()[1] == a.launch_counts()[2] == 1
    for k in (0, 7, 632, 639):
        assert np.abs(a.positions(k) - b.positions(k)).max() < 1e-8 * np.abs(b.positions(k)).max()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("sequence", ["fresh", "restored", "used"])
def test_batch_falls_back_in_any_state(native, precision, sequence):
    """A resident launch that gives up while the lockstep CG is not set up: nothing
    done before, a shape forced and released, and solves of the other kind in
    between. Its buffers are made then, and the step is the forced batch's."""
    kw = dict(itr_tol=1e-12 if precision == "fp64" else 1e-10, max_iters=20000, max_newton=3,
              mixed=True)
    scs = [scenes.beam_scene(*n, seed=k, **kw)
           for k, n in enumerate([(20, 6, 6), (5, 2, 3), (33, 9, 8)])]
    a, b = native.Batch(scs, precision=precision), native.Batch(scs, precision=precision)
    b.set_cg_shape(0, 256)
    if sequence != "fresh":
        a.set_cg_shape(0, 64)
        if sequence == "used":
            a.step()
            b.step()
        a.set_cg_shape(-1)
    for wait in (0, 2000, 0):
        a.set_resident_wait(wait)
        before = a.launch_counts()
        a.step()
        b.step()
        cg, newton = (x - y for x, y in zip(a.launch_counts()[1:], before[1:]))
        assert (cg > 20 * newton) == (wait == 0), (wait, cg, newton)
        for k in range(a.count):
            xa, xb = a.positions(k), b.positions(k)
            assert np.abs(xa - xb).max() < 1e-8 * np.abs(xb).max(), k
    with pytest.raises(native.MfemError, match="wait"):
        a.set_resident_wait(-1.0)


def test_batch_tunes_ahead_of_a_solve_only(native):
    """21k rows, enough for the tuner, whose trials overwrite the solution: the
    solve that falls back has one in progress (the sum of its sweeps) and takes the
    default shape; the tuner runs ahead of a solve by launches."""
    scs = [scenes.beam_scene(50, 14, 13 + k, seed=k, itr_tol=1e-10, max_iters=20000, max_newton=1,
                             mixed=True) for k in range(2)]
    a, b = native.Batch(scs, precision="mixed"), native.Batch(scs, precision="mixed")
    b.set_cg_shape(0, 256)
    a.set_resident_wait(0)
    a.step()
    b.step()
    assert a.launch_counts()[1] > 20 and a.cg_shape() == (-1, 0)
    for k in range(2):
        assert np.abs(a.positions(k) - b.positions(k)).max() < 1e-8 * np.abs(b.positions(k)).max()
    a.step()  # the resident kernel is not tried: a solve by launches from its start
    assert a.cg_shape()[0] >= 0


def test_batch_columns_that_do_not_fit(native):
    """One beam whose columns do not fit its workgroups (9.4k rows, 293 a workgroup,
    in random order): the whole batch moves to the lockstep CG."""
    def batch():
        return native.Batch([scenes.beam_scene(20, 6, 6, seed=1, itr_tol=1e-12, max_iters=20000),
                             shuffled(scenes.beam_scene(48, 13, 13, seed=2, itr_tol=1e-12,
                                                        max_iters=20000), 3)], precision="fp64")
    a, b = batch(), batch()
    b.set_cg_shape(0, 64)
    a.step()
    b.step()
    for k in range(2):
        assert np.abs(a.positions(k) - b.positions(k)).max() < 1e-8
    assert a.launch_counts()[1] > 4 * a.launch_counts()[2]
