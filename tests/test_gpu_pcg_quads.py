"""The PCG kernels with four lanes per row (FP64 systems of 1,025 to 32,768
rows) against the row-gather kernels, and the 256-row kernels (FP32, FP64 past
that limit, and FP64 where a row has more neighbours than a workgroup of the
others stages): the first size of the rule (a workgroup of one row at the end),
remainders, the last size and one past it, rows of exactly the entries that are
loaded at once (16) and of more, and a row that neither kind of tile takes.

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


def solve(s, precision, groups=None, **kw):
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
        if groups is not None:
            assert groups(pd.stats().halo_groups), pd.stats().halo_groups
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


def beside(a, b):
    """The bodies of two scenes in one, the second moved away."""
    cat = lambda f, off=0: np.concatenate([getattr(a, f), getattr(b, f) + np.asarray(off, getattr(b, f).dtype)])  # noqa: E731
    return mesh.Scene(X=np.concatenate([a.X, b.X + [20.0, 0.0, 0.0]]), tet=cat("tet", a.nv), tri=cat("tri", a.nv),
                      tri_fathers=cat("tri_fathers", 1), mass=cat("mass"), mu=cat("mu"), lam=cat("lam"), dbc=cat("dbc"),
                      body_vert_start=np.concatenate([a.body_vert_start, b.body_vert_start[1:] + a.nv]),
                      body_tet_start=np.concatenate([a.body_tet_start, b.body_tet_start[1:] + a.nt]))


# scene, rows per workgroup of the FP64 kernels (0: row-gather)
SCENES = {"1025": (lambda: body(4, 4, 40), 64), "1452": (lambda: body(10, 11, 10), 64),
          "32768": (lambda: body(31, 31, 31), 64), "33759": (lambda: body(30, 32, 32), 256),
          "rows of 16": (lambda: beside(body(9, 9, 10), fan(14)), 64),
          "rows of 17": (lambda: beside(body(9, 9, 10), fan(15)), 64),
          "rows of 62": (lambda: beside(body(9, 9, 10), fan(60)), 64),
          "rows of 602": (lambda: beside(body(9, 9, 10), fan(600)), 256),
          "rows of 902": (lambda: beside(body(9, 9, 10), fan(900)), 0)}


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("chebyshev", [True, False])
@pytest.mark.parametrize("name", list(SCENES))
def test_matches_the_row_gather_kernels(gpu, name, chebyshev, precision):
    make, rows = SCENES[name]
    s = make()
    assert s.nv > 1024  # smaller systems are solved in one workgroup
    rows = rows if precision == 64 or rows == 0 else 256
    kw = dict(pcg_chebyshev=chebyshev)
    # a workgroup ends early only where its halo is full: the count tells 64 rows from 256
    x = solve(s, precision, groups=lambda g: (rows == 0) == (g == 0) and (rows != 64 or g >= s.nv / 64)
              and (rows != 256 or g < s.nv / 64), **kw)
    ref = solve(s, 64, pcg_halo=0, **kw)
    if precision == 64:
        assert rel_err(x, ref) < 1e-10, rel_err(x, ref)
    else:
        gather = rel_err(solve(s, 32, pcg_halo=0, **kw), ref)
        assert rel_err(x, ref) <= 2 * gather + 1e-6, (rel_err(x, ref), gather)
