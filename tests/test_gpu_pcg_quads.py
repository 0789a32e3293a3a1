"""The PCG kernels with four lanes per row (FP64 systems of up to 32,768 rows)
against the row-gather kernels, and the 256-row kernels (FP32, and FP64 just
above that limit):
one body of 8 vertices, exactly one workgroup (64 rows), remainders, the last
size of the rule and one past it, and rows of more entries than are loaded at
once.

Bounds: in FP64 both sides stop at ||D^-1 r|| <= 1e-13 of its start (1e-10
relative, the bar of the PCG tests).  In FP32 both stop by the same test and
differ in the order of a row's products, so the distance to the FP64 solution
may be at most twice the row-gather kernels' plus 1e-6 (8 units of FP32
rounding of the positions that are handed back)."""
import numpy as np
import pytest

from conftest import rel_err
from sbs_amd import mesh
from sbs_amd.pd import PdSolver, SolverData, SolverParams, SolverType

pytestmark = pytest.mark.gpu


def solve(s, precision, **kw):
    p = SolverParams(**dict(dict(numIterations=6, dt=1.0 / 60.0, gravity=9.8, tol=0.0, rho=0.9992, pcg_max_iter=400,
                                 pcg_tol=1e-6 if precision == 32 else 1e-13,
                                 pcg_floor=1e-8 if precision == 32 else 0.0), **kw))
    data = SolverData(s, precision)
    pd = PdSolver(128, data)
    pd.SetGlobalSolver(SolverType.PCG)
    try:
        for _ in range(2):
            pd.Update(data, p)
        pd.synchronize()
        return data.get("X")
    finally:
        pd.close()
        data.free()


def fan(m):
    """m tets around one edge, whose two vertices have m + 1 neighbours."""
    ang = 2 * np.pi * np.arange(m) / m
    X = np.vstack([[[0, 0, 0], [0, 0.3, 0]], np.stack([0.3 * np.cos(ang), 0.15 + 0 * ang, 0.3 * np.sin(ang)], 1)])
    ring = np.arange(m)
    tet = np.stack([0 * ring, 0 * ring + 1, 2 + (ring + 1) % m, 2 + ring], 1)
    assert (np.linalg.det(X[tet[:, 1:]] - X[tet[:, :1]]) > 0).all()
    base = mesh.cube_scene(2)
    return mesh.Scene(X=X, tet=tet.astype(base.tet.dtype), tri=np.array([[0, 1, 2]], dtype=base.tri.dtype),
                      tri_fathers=np.zeros(1, base.tri_fathers.dtype), mass=np.full(len(X), base.mass[0]),
                      mu=np.full(m, base.mu[0]), lam=np.full(m, base.lam[0]), dbc=np.zeros(len(X)),
                      body_vert_start=np.array([0, len(X)]), body_tet_start=np.array([0, m]))


def body(*n):
    return mesh.make_scene([dict(nx=n[0], ny=n[1], nz=n[2], spacing=0.1, origin=(0.0, 0.0, 0.0), jitter=1e-3, nu=0.3,
                                 E=2e5, seed=1, density=1000.0, pin_top=True)])


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("chebyshev", [True, False])
@pytest.mark.parametrize("size", [(1, 1, 1), (3, 3, 3), (1, 4, 12), (31, 31, 31), (30, 32, 32), "fan 14", "fan 60"])
def test_matches_the_row_gather_kernels(gpu, size, chebyshev, precision):
    s = fan(int(size.split()[1])) if isinstance(size, str) else body(*size)
    kw = dict(pcg_chebyshev=chebyshev)
    x = solve(s, precision, **kw)
    ref = solve(s, 64, pcg_halo=0, **kw)
    if precision == 64:
        assert rel_err(x, ref) < 1e-10, rel_err(x, ref)
    else:
        gather = rel_err(solve(s, 32, pcg_halo=0, **kw), ref)
        assert rel_err(x, ref) <= 2 * gather + 1e-6, (rel_err(x, ref), gather)
