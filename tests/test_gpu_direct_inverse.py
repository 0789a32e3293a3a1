"""The direct global solve by the product with the explicit inverse: sizes at
the edges of its tiles (8 rows per workgroup, 4-value loads, 1,024 columns per
pass, one ticket or a tree of them) and scenes of several systems; and by the
triangular solves where the inverse has no room: one block of 64 rows, several
with remainders, a band of several hundred rows.  Both against a dense FP64
solve of the exported matrix."""
import numpy as np
import pytest
import scipy.sparse as sp
from scipy.linalg import solve_triangular
from scipy.sparse.csgraph import reverse_cuthill_mckee

from sbs_amd import capi, mesh
from sbs_amd.pd import PdSolver, SolverData, SolverParams, SolverType

pytestmark = pytest.mark.gpu

# vertices: up to 64 workgroups (8 .. 126, several systems), more; remainders of
# 8 rows and 4 columns (27, 125, 126, 729, 1,089), a pass of columns less 24 and
# with 32 and 65 more (1,000, 1,056, 1,089)
SCENES = {"8": [(1, 1, 1)], "12": [(2, 1, 1)], "27": [(2, 2, 2)], "120": [(3, 4, 5)], "125": [(4, 4, 4)],
          "126": [(2, 5, 6)], "729": [(8, 8, 8)], "1000": [(9, 9, 9)], "1056": [(10, 11, 7)], "1089": [(10, 10, 8)],
          "three": [(2, 2, 2), (4, 3, 1), (1, 2, 1)], "mixed": [(4, 4, 4), (1, 1, 1), (4, 5, 6), (3, 4, 4), (2, 2, 2)]}


def scene_of(dims):
    return mesh.make_scene([dict(nx=d[0], ny=d[1], nz=d[2], seed=3 + i, pin_top=True, origin=(3.0 * i, 0.0, 0.0))
                            for i, d in enumerate(dims)])


def solved(scene, precision, memory):
    """(matrix, b, x, direct_info) of one solve with a random right-hand side."""
    data = SolverData(scene, precision)
    pd = PdSolver(128, data)
    pd.SetGlobalSolver(SolverType.CuSolverCholesky)
    pd.set_direct_memory(memory)
    p = SolverParams(numIterations=2, dt=1.0 / 60.0, tol=0.0)
    pd.Update(data, p)
    ex = pd.export_system()
    n = scene.nv
    A = np.zeros((n, n))
    for v in range(n):
        A[v, ex["col"][ex["rowptr"][v]:ex["rowptr"][v + 1]]] = ex["val"][ex["rowptr"][v]:ex["rowptr"][v + 1]]
    rng = np.random.default_rng(1)
    b = (rng.normal(size=(n, 3)) * np.diag(A)[:, None]).astype(data.dtype)
    db, dx = capi.DeviceArray.from_numpy(b), capi.DeviceArray(b.nbytes)
    pd.solve(db.ptr, dx.ptr, p)
    x = dx.download(data.dtype, (n, 3)).astype(np.float64)
    info = pd.direct_info()
    pd.close()
    data.free()
    return A, b.astype(np.float64), x, info


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("name", list(SCENES))
def test_solve_against_dense(name, precision):
    scene = scene_of(SCENES[name])
    n = scene.nv
    A, b, x, info = solved(scene, precision, 4 << 30)
    assert info["inverse_bytes"] > 0 and info["systems"] == len(SCENES[name])
    inv = np.linalg.inv(A)
    ref = inv @ b
    # each entry of the inverse and each product is rounded once, and at most
    # n / 1024 + 24 sums stand between a product and the result; in FP64 the
    # factor's own error (condition number times the unit roundoff) adds to it
    u = np.finfo(np.float32 if precision == 32 else np.float64).eps / 2
    bound = (3 + n / 1024 + 24) * u * (np.abs(inv) @ np.abs(b))
    if precision == 64:
        bound = bound + 1e-12 * np.abs(ref).max()
    assert np.all(np.abs(x - ref) <= bound)


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("name", ["8", "27", "120", "125", "729", "1056", "1089", "three", "mixed"])
def test_triangular_solves_against_dense(name, precision):
    """Without memory for the inverse.  FP64: to the condition number (at most 1e6
    with the pins) times the roundoff.  FP32: the same solves in NumPy, the FP64
    factor (reverse Cuthill-McKee order) rounded to FP32 and its triangles
    solved in FP32, are off by as much; another order of the sums and of the
    elimination may double that twice."""
    scene = scene_of(SCENES[name])
    A, b, x, info = solved(scene, precision, 0)
    assert info["inverse_bytes"] == 0 and info["systems"] == len(SCENES[name])
    ref = np.linalg.solve(A, b)
    err = np.linalg.norm(x - ref) / np.linalg.norm(ref)
    if precision == 64:
        assert err <= 1e6 * np.finfo(np.float64).eps
        return
    q = reverse_cuthill_mckee(sp.csr_matrix(A), symmetric_mode=True)
    L = np.linalg.cholesky(A[np.ix_(q, q)]).astype(np.float32)
    own = np.zeros_like(b, dtype=np.float32)
    y = solve_triangular(L, b[q].astype(np.float32), lower=True)
    own[q] = solve_triangular(L, y, lower=True, trans="T")
    assert err <= 4 * np.linalg.norm(own - ref) / np.linalg.norm(ref)


def test_triangular_solves_of_a_wide_band(gpu):
    """27^3 hexes (21,952 rows, half bandwidth about 800), FP64: a step with the
    triangular solves and one with the product.  kappa(A) is about 1.1e6, so
    the solves are 1e-9 of each other at most."""
    scene = mesh.cube_scene(27)
    out = []
    for memory in (0, 8 << 30):
        data = SolverData(scene, 64)
        pd = PdSolver(128, data)
        pd.SetGlobalSolver(SolverType.CuSolverCholesky)
        pd.set_direct_memory(memory)
        pd.Update(data, SolverParams(numIterations=3, dt=1.0 / 60.0, tol=0.0))
        pd.synchronize()
        info = pd.direct_info()
        assert (info["inverse_bytes"] > 0) == (memory > 0) and info["bandwidth"] > 700
        out.append(data.get("X"))
        pd.close()
        data.free()
    assert np.abs(out[0] - out[1]).max() <= 1e-9 * np.abs(out[1]).max()


def test_memory_bound(gpu):
    """The bound on the inverse's memory: below the inverse's size the factor is
    solved by triangular solves, a changed bound takes effect with the next
    update, and both forms give the same step to FP64 rounding (the matrix's
    condition number, about 1e6 with the pins, times 1e-16, over 2 iterations)."""
    scene = mesh.make_scene([dict(nx=7, ny=8, nz=6, seed=3, pin_top=True)])
    n = scene.nv
    size = 8 * n * ((n + 3) // 4 * 4)
    data = SolverData(scene, 64)
    pd = PdSolver(128, data)
    pd.SetGlobalSolver(SolverType.CuSolverCholesky)
    p = SolverParams(numIterations=2, dt=1.0 / 60.0, tol=0.0)
    rest = {k: data.get(k) for k in ("X", "V", "XTilde")}
    out = {}
    for bound, held in ((None, size), (size - 1, 0), (size, size), (0, 0)):
        if bound is not None:
            before = pd.direct_info()
            pd.set_direct_memory(bound)
            assert pd.direct_info() == before  # until the next update
        for k, a in rest.items():
            data._bufs[k].upload(a)
        pd.Update(data, p)
        pd.synchronize()
        assert pd.direct_info()["inverse_bytes"] == held
        out[bound] = data.get("X")
        assert np.abs(out[bound] - out[None]).max() <= 1e-9 * np.abs(out[None]).max()
    assert np.array_equal(out[size], out[None]) and np.array_equal(out[size - 1], out[0])
    pd.close()
    data.free()


def test_error_and_early_exit_of_many_bodies(gpu):
    """The outer loop's error and decision from 1,300 workgroups' sums: the step
    ends after the same iteration as with the triangular solves (whose error
    and decision are launches of their own), FP64."""
    scene = mesh.make_scene([dict(nx=2, ny=2, nz=2, seed=i, pin_top=True, origin=(1.0 * (i % 20), 0.0, 1.0 * (i // 20)))
                             for i in range(320)] + [dict(nx=4, ny=5, nz=6, seed=7, origin=(0.0, 3.0, 0.0))])
    out = {}
    for tol in (0.0, 2e-5):
        for bound in (4 << 30, 0):
            data = SolverData(scene, 64)
            pd = PdSolver(128, data)
            pd.SetGlobalSolver(SolverType.CuSolverCholesky)
            pd.set_direct_memory(bound)
            for _ in range(2):
                pd.Update(data, SolverParams(numIterations=12, dt=1.0 / 60.0, tol=tol))
            pd.synchronize()
            info = pd.direct_info()
            assert info["systems"] == 321 and (info["inverse_bytes"] > 0) == (bound > 0)
            out[tol, bound > 0] = data.get("X")
            pd.close()
            data.free()
    scale = np.abs(out[0.0, True]).max()
    for tol in (0.0, 2e-5):
        assert np.abs(out[tol, True] - out[tol, False]).max() <= 1e-9 * scale
    # the exit was taken: an iteration more moves some vertex by more than that
    assert np.abs(out[0.0, True] - out[2e-5, True]).max() > 1e-7 * scale
