"""The batched solve's instances by rows per thread: bodies whose vertex counts
lie on both sides of each limit (the search direction in LDS or in memory, one,
two, four, six and ten rows of 1,024 threads in registers, 16- or 32-bit
columns) and a body whose widest row exceeds the rows kept in registers,
against one PCG solver per body (the general path of a single body).

Bounds: in FP64 both sides stop at ||D^-1 r|| <= 1e-13 of its start, so the
bar of the batched tests holds (1e-10 relative).  In FP32 both sides stop by
the same test after the same arithmetic in another order, each with its own
rounding, so neither is the reference: the distance to the FP64 solver may be
at most twice the single-body solver's (the batched vectors are relative to the
body, the other's to the world) plus 1e-6 (8 units of FP32 rounding of
positions that are handed back)."""
import numpy as np
import pytest

from conftest import rel_err
from sbs_amd import mesh
from sbs_amd.pd import PdSolver, SolverData, SolverParams, SolverType

pytestmark = pytest.mark.gpu

# hexes per axis; vertices (nx + 1)(ny + 1)(nz + 1)
SIZES = [(7, 7, 15), (4, 4, 40),        # 1,024  1,025
         (7, 15, 15), (4, 9, 40),       # 2,048  2,050
         (15, 15, 15), (9, 9, 40),      # 4,096  4,100
         (15, 15, 23), (9, 14, 40),     # 6,144  6,150
         (15, 19, 31), (9, 24, 40),     # 10,240 10,250
         (19, 24, 27), (19, 24, 43)]    # 14,000 (direction in memory) 22,000 (32-bit columns)


def solve(s, precision, solver, **kw):
    p = SolverParams(**dict(dict(numIterations=10, dt=1.0 / 60.0, gravity=9.8, tol=1e-6, rho=0.9992,
                                 pcg_chebyshev=True, pcg_max_iter=400, pcg_adaptive=False,
                                 pcg_tol=1e-6 if precision == 32 else 1e-13,
                                 pcg_floor=1e-8 if precision == 32 else 0.0), **kw))
    data = SolverData(s, precision)
    pd = PdSolver(128, data)
    pd.SetGlobalSolver(solver)
    try:
        for _ in range(2):
            pd.Update(data, p)
        pd.synchronize()
        return data.get("X"), pd.batch_info() if solver == SolverType.BatchedPCG else None
    finally:
        pd.close()
        data.free()


def check(bodies, scene, precision, tune):
    X, info = solve(scene, precision, SolverType.BatchedPCG, batch_autotune=tune)
    assert info["bodies"] == len(bodies) and (info["body_stats"][:, 5] == 0).all()
    for i, sb in enumerate(bodies):
        xb = X[scene.body_vert_start[i]:scene.body_vert_start[i + 1]]
        ref, _ = solve(sb, 64, SolverType.PCG, pcg_tol=1e-13, pcg_floor=0.0)
        err = rel_err(xb, ref)
        if precision == 64:
            assert err < 1e-10, (i, sb.nv, err)
        else:
            single, _ = solve(sb, 32, SolverType.PCG)
            assert err <= 2 * rel_err(single, ref) + 1e-6, (i, sb.nv, err, rel_err(single, ref))


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("largest", [1, *range(2, len(SIZES) + 1, 2)])
def test_row_limits(gpu, precision, largest):
    specs = [dict(nx=a, ny=b, nz=c, spacing=0.1, origin=(3.0 * i, 0.0, 0.0), jitter=1e-3, nu=0.3, E=2e5, seed=i,
                  density=1000.0, pin_top=True) for i, (a, b, c) in enumerate(SIZES[max(0, largest - 2):largest])]
    specs.append(dict(specs[0], nx=1, ny=1, nz=1, origin=(-3.0, 0.0, 0.0)))
    check([mesh.make_scene([b]) for b in specs], mesh.make_scene(specs), precision, tune=largest <= 2)


@pytest.mark.parametrize("precision", [32, 64])
def test_rows_wider_than_the_registers(gpu, precision):
    """Tets around an edge: its two vertices have 24 neighbours."""
    m = 23
    ang = 2 * np.pi * np.arange(m) / m
    X = np.vstack([[[0, 0, 0], [0, 0.3, 0]], np.stack([0.3 * np.cos(ang), 0.15 + 0 * ang, 0.3 * np.sin(ang)], 1)])
    ring = np.arange(m)
    tet = np.stack([0 * ring, 0 * ring + 1, 2 + (ring + 1) % m, 2 + ring], 1).astype(np.uint32)
    vol = np.linalg.det((X[tet[:, 1:]] - X[tet[:, :1]]).astype(np.float64))
    assert (vol > 0).all() or (vol < 0).all()
    if vol[0] < 0:
        tet = tet[:, [0, 2, 1, 3]]
    base = mesh.cube_scene(2)
    tri = np.array([[0, 1, 2]], dtype=base.tri.dtype)
    s = mesh.Scene(X=X, tet=tet.astype(base.tet.dtype), tri=tri, tri_fathers=np.zeros(1, base.tri_fathers.dtype),
                   mass=np.full(len(X), base.mass[0]), mu=np.full(m, base.mu[0]), lam=np.full(m, base.lam[0]),
                   dbc=np.zeros(len(X)), body_vert_start=np.array([0, len(X)]), body_tet_start=np.array([0, m]))
    check([s], s, precision, tune=False)


@pytest.mark.parametrize("precision", [32, 64])
def test_result_does_not_depend_on_the_other_bodies(gpu, precision):
    """A body's step is the same to the bit whatever bodies are beside it: bodies
    of less than a tet chunk, of several and of several whole ones.  Two bodies
    are in every scene at the corners of its box (the matrix is assembled in the
    order of a Morton curve over that box) and one is the largest (the workgroup
    size follows it)."""
    def spec(i, n, origin):
        return dict(nx=n[0], ny=n[1], nz=n[2], spacing=0.1, origin=origin, jitter=1e-3, nu=0.3, E=2e5,
                    seed=i, density=1000.0, pin_top=True)
    dims = [(1, 1, 1), (7, 7, 7), (2, 2, 2), (5, 4, 4), (8, 4, 8), (3, 4, 5), (1, 1, 1), (6, 7, 5)]
    assert 6 * 8 * 4 * 8 % 256 == 0  # whole chunks only
    specs = [spec(i, n, (3.0 * i, 0.0, 0.0)) for i, n in enumerate(dims)]
    specs[0] = spec(0, dims[0], (-5.0, -5.0, -5.0))
    specs.append(spec(8, (1, 1, 1), (30.0, 5.0, 5.0)))
    full = mesh.make_scene(specs)
    X, _ = solve(full, precision, SolverType.BatchedPCG, batch_autotune=False)
    ref = [X[full.body_vert_start[i]:full.body_vert_start[i + 1]] for i in range(len(specs))]
    for keep in ([0, 1, 8], [3, 0, 1, 8], [5, 0, 8, 1, 2], [0, 1, 7, 6, 4, 8]):
        s = mesh.make_scene([specs[i] for i in keep])
        x, _ = solve(s, precision, SolverType.BatchedPCG, batch_autotune=False)
        for j, i in enumerate(keep):
            assert np.array_equal(x[s.body_vert_start[j]:s.body_vert_start[j + 1]], ref[i]), (keep, i)
