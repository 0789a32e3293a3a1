"""What this library is timed on: whole calls through its public entry points.

Each case is one call that a program makes over and over:

* ``pd``: one ``PdSolver.Update`` (a time step of projective dynamics) of a
  scene of hex-grid bodies, with one of the global solvers;
* ``collide``: the same step with collision handling, two cubes meeting, and
  a fixed sphere;
* ``ipc``: one ``IpcSolver.Update`` (FP64 Newton step with the contact
  barrier) of two stacked cubes in contact;
* ``coo``: one ``PCGJacobiSolver.Solve`` of an elasticity system handed over
  as unsorted triplets with repeated entries.

A step starts from a stored state (positions and velocities in the caller's
device arrays), as a rollout, a line search over controls or a rewind does,
so that every pass does the same work.  The stored states are deformed and
moving: a smooth displacement of a few percent strain and a smooth velocity
field, from the seed.  The solver of a state has run three steps from it
before it is handed out: a program that steps has its factor, its tuned
workgroups and its learned launch counts by then.
"""
import ctypes
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "soft-body-simulation-cuda_amd"))

from sbs_amd import capi, fixed, mesh  # noqa: E402
from sbs_amd.ipc import IpcData, IpcParams, IpcSolver  # noqa: E402
from sbs_amd.linear import PCGJacobiSolver  # noqa: E402
from sbs_amd.pd import PdSolver, SolverData, SolverParams, SolverType  # noqa: E402

SPACING = 0.1
DT = 1.0 / 60.0
DENSITY = 1000.0
DEVICE = "cuda"


def listed():
    return [
        # the headline body: 274,625 vertices, 1,572,864 tets, the benchmark's parameters
        dict(name="pcg_64x64x64_f32", kind="pd", solver="PCG", nx=64, ny=64, nz=64, bodies=1, precision=32,
             iterations=20, chebyshev=True, polar=True),
        # an interactive toy: 336 vertices, every default of SolverParams but the iteration count
        dict(name="pcg_5x7x6_f32", kind="pd", solver="PCG", nx=5, ny=7, nz=6, bodies=1, precision=32, iterations=10,
             chebyshev=False, polar=False),
        # a mid-size body in double precision
        dict(name="pcg_22x19x25_f64", kind="pd", solver="PCG", nx=22, ny=19, nz=25, bodies=1, precision=64,
             iterations=20, chebyshev=True, polar=False),
        # the default global solver (Jacobi + Chebyshev) and the default rotation (SVD) on a large ragged body
        dict(name="jacobi_47x40x33_f32", kind="pd", solver="Jacobi", nx=47, ny=40, nz=33, bodies=1, precision=32,
             iterations=20, chebyshev=False, polar=False),
        # the smallest workload of the benchmark: 729 vertices on the prefactored Cholesky
        dict(name="cholesky_8x8x8_f32", kind="pd", solver="CuSolverCholesky", nx=8, ny=8, nz=8, bodies=1,
             precision=32, iterations=10, chebyshev=False, polar=False),
        # a larger ragged body on the prefactored Cholesky
        dict(name="cholesky_13x15x14_f32", kind="pd", solver="CuSolverCholesky", nx=13, ny=15, nz=14, bodies=1,
             precision=32, iterations=20, chebyshev=False, polar=False),
        # many equal small bodies on the dense per-body solve (the benchmark's 256 bodies)
        dict(name="dense_256x6x6x6_f32", kind="pd", solver="DenseCholesky", nx=6, ny=6, nz=6, bodies=256,
             precision=32, iterations=10, chebyshev=False, polar=False),
        # many uneven bodies (3..20 hexes per axis), each its own solve; a quarter of the benchmark's 1,024
        dict(name="batched_256x3to20_f32", kind="pd", solver="BatchedPCG", nx=20, ny=20, nz=20, bodies=256,
             precision=32, iterations=10, chebyshev=True, polar=True),
        # two 24^3 cubes meeting, with collision handling (the benchmark's collision scene)
        dict(name="collide_24x24x24_f32", kind="collide", solver="PCG", nx=24, ny=24, nz=24, bodies=2, precision=32,
             iterations=20, chebyshev=True, polar=True),
        # the FP64 contact scene of the benchmark: two 16^3 Neo-Hookean cubes
        dict(name="ipc_16x16x16", kind="ipc", nx=16, ny=16, nz=16, elastic="neohookean"),
        # a small ragged contact scene with the default elasticity
        dict(name="ipc_6x4x5", kind="ipc", nx=6, ny=4, nz=5, elastic="corotated"),
        # a general linear solve with the contact solver's triplet layout (12 x 12 per tet)
        dict(name="coo_18x15x17_f64", kind="coo", nx=18, ny=15, nz=17, precision=64),
    ]


def _between(rng, lo, hi):
    """A whole number, spread evenly over the logarithm of its range."""
    return int(round(math.exp(rng.uniform(math.log(lo - 0.49), math.log(hi + 0.49)))))


def draw(rng):
    kind = rng.choice(("pcg", "pcg", "jacobi", "cholesky", "dense", "batched", "collide", "ipc", "coo"))

    def dims(lo, hi):
        return dict(nx=_between(rng, lo, hi), ny=_between(rng, lo, hi), nz=_between(rng, lo, hi))

    if kind in ("pcg", "jacobi"):
        precision = rng.choice((32, 32, 64))
        return dict(kind="pd", solver="PCG" if kind == "pcg" else "Jacobi", **dims(4, 60 if precision == 32 else 32),
                    bodies=1, precision=precision, iterations=rng.choice((10, 20)),
                    chebyshev=kind == "pcg" and rng.random() < 0.7, polar=rng.random() < 0.5)
    if kind == "cholesky":
        return dict(kind="pd", solver="CuSolverCholesky", **dims(3, 15), bodies=1, precision=rng.choice((32, 64)),
                    iterations=rng.choice((10, 20)), chebyshev=False, polar=rng.random() < 0.5)
    if kind == "dense":
        return dict(kind="pd", solver="DenseCholesky", **dims(2, 6), bodies=_between(rng, 8, 256), precision=32,
                    iterations=10, chebyshev=False, polar=False, dense_precision=rng.choice((0, 1)))
    if kind == "batched":
        return dict(kind="pd", solver="BatchedPCG", **dims(6, 20), bodies=_between(rng, 16, 256),
                    precision=rng.choice((32, 32, 64)), iterations=10, chebyshev=True, polar=rng.random() < 0.5)
    if kind == "collide":
        return dict(kind="collide", solver="PCG", **dims(5, 24), bodies=2, precision=32, iterations=20, chebyshev=True,
                    polar=rng.random() < 0.5)
    if kind == "ipc":
        return dict(kind="ipc", **dims(3, 15), elastic=rng.choice(("neohookean", "corotated")))
    return dict(kind="coo", **dims(4, 18), precision=rng.choice((32, 64)))


# ---------------------------------------------------------------- scenes --

@functools.lru_cache(maxsize=32)
def _body_dims(case_key):
    """Hexes per axis of each body: equal bodies, or (batched) uneven ones of 3 hexes up to the case's size."""
    c = dict(case_key)
    n, top = c["bodies"], np.array([c["nx"], c["ny"], c["nz"]])
    if c["solver"] != "BatchedPCG":
        return np.tile(top, (n, 1))
    u = mesh.uniform01(101, np.arange(3 * n, dtype=np.uint64)).reshape(n, 3)
    return 3 + np.floor(u * (top - 2)).astype(int)


@functools.lru_cache(maxsize=512)
def _grid_tets(nx, ny, nz):
    return mesh.hex_grid_tets(nx, ny, nz)


@functools.lru_cache(maxsize=8)
def _grid_tris(nx, ny, nz):
    return mesh.surface_triangles(_grid_tets(nx, ny, nz))


def _grid_points(nx, ny, nz):
    k, j, i = np.meshgrid(np.arange(nz + 1), np.arange(ny + 1), np.arange(nx + 1), indexing="ij")
    return np.stack([i.ravel(), j.ravel(), k.ravel()], axis=1).astype(np.float64)


def _scene(dims, origins, pins, seed, jitter, nu=0.3, surface=False):
    """Hex-grid bodies side by side: (mesh.Scene, per vertex its body, per vertex its distance below its body's top)."""
    rng = np.random.default_rng(seed)
    X, tet, tri, fathers, mass, mu, lam, dbc, body, below = [], [], [], [], [], [], [], [], [], []
    vs, ts = [0], [0]
    for b, (d, origin, pin) in enumerate(zip(dims, origins, pins)):
        d = tuple(int(v) for v in d)
        P, t = _grid_points(*d), _grid_tets(*d)
        n = len(P)
        m, la = mesh.lame(float(rng.uniform(8e4, 1.6e5)) if len(dims) > 2 else 1e5, nu)
        pinned = {"top": P[:, 1] == d[1], "bottom": P[:, 1] == 0, "": np.zeros(n, bool)}[pin]
        X.append(P * SPACING + origin + rng.uniform(-jitter, jitter, (n, 3)))
        tet.append(t.astype(np.int64) + vs[-1])
        mass.append(np.full(n, DENSITY * d[0] * d[1] * d[2] * SPACING ** 3 / n))
        mu.append(np.full(len(t), m))
        lam.append(np.full(len(t), la))
        dbc.append(pinned.astype(np.float64))
        body.append(np.full(n, b))
        below.append((d[1] - P[:, 1]) * SPACING if pin == "top" else P[:, 1] * SPACING)
        if surface:
            s = _grid_tris(*d)
            tri.append(s.astype(np.int64) + vs[-1])
            fathers.append(np.full(len(s), b, np.uint32))
        vs.append(vs[-1] + n)
        ts.append(ts[-1] + len(t))
    tri = np.concatenate(tri) if surface else np.zeros((0, 3))
    s = mesh.Scene(X=np.concatenate(X), tet=np.concatenate(tet).astype(np.uint32), tri=tri.astype(np.uint32),
                   tri_fathers=np.concatenate(fathers) if surface else np.zeros(0, np.uint32),
                   mass=np.concatenate(mass), mu=np.concatenate(mu), lam=np.concatenate(lam),
                   dbc=np.concatenate(dbc), body_vert_start=np.asarray(vs), body_tet_start=np.asarray(ts))
    return s, np.concatenate(body), np.concatenate(below)


def _field(X, weight, seed, size):
    """A smooth random vector field at X, about `size` per unit of `weight`."""
    rng = np.random.default_rng(seed)
    out = np.zeros_like(X)
    for k in range(3):
        for _ in range(3):
            freq = rng.normal(0.0, 1.5, 3)
            out[:, k] += np.sin(X @ freq + rng.uniform(0, 2 * np.pi)) / 3
    return size * out * weight[:, None]


def _state(case, seed):
    """(scene, body of each vertex, X, V): the rest scene and the moving state that a step starts from."""
    gap = 0.0
    if case["kind"] == "pd":
        dims = _body_dims(tuple(sorted((k, v) for k, v in case.items() if k != "name")))
        side = math.ceil(math.sqrt(len(dims)))
        pitch = (max(case["nx"], case["nz"]) + 5) * SPACING
        origins = [(pitch * (i % side), 0.0, pitch * (i // side)) for i in range(len(dims))]
        scene, body, below = _scene(dims, origins, ["top"] * len(dims), seed, 1e-3)
        weight = np.minimum(below, 1.0)
    else:
        d = (case["nx"], case["ny"], case["nz"])
        jitter = 5e-4
        gap = 2e-3 if case["kind"] == "collide" else 6e-4
        top = d[1] * SPACING + gap + 2 * jitter
        scene, body, below = _scene([d, d], [(0.0, 0.0, 0.0), (0.0, top, 0.0)], ["bottom", ""], seed, jitter,
                                    0.3 if case["kind"] == "collide" else 0.4, surface=True)
        # nothing at the pinned bottom, the same on both sides of the gap
        weight = np.minimum(np.where(body == 0, below, d[1] * SPACING), 1.0)
    strain = 0.0 if case["kind"] == "ipc" else 0.02
    speed = 0.05 if case["kind"] == "ipc" else 0.5
    X = scene.X + _field(scene.X, weight, seed + 1, strain)
    V = _field(scene.X, weight, seed + 2, speed)
    if gap:
        V[body == 1, 1] -= 0.4 if case["kind"] == "collide" else 0.1   # the upper cube comes down
    V[scene.dbc > 0] = 0.0
    return scene, body, X, V


# ------------------------------------------------------------- PD steps --

def _params(case):
    return SolverParams(numIterations=case["iterations"], dt=DT, gravity=9.8,
                        tol=0.0 if case["solver"] == "DenseCholesky" else 1e-6, rho=0.9992, pcg_tol=1e-6,
                        pcg_floor=1e-8 if case["precision"] == 32 else 0.0, pcg_max_iter=200,
                        pcg_chebyshev=case["chebyshev"], handleCollision=case["kind"] == "collide",
                        dense_precision=case.get("dense_precision", 0), dense_tol=1e-10, dense_max_iter=16,
                        polar_rotation=case["polar"])


def _sphere(case):
    """Beside the upper cube of the collision scene, reaching 5 mm or so into it."""
    r = 0.3
    return (case["nx"] * SPACING + r - 0.005, 1.5 * case["ny"] * SPACING, 0.5 * case["nz"] * SPACING), r


class _Pd:
    """A scene's solver, and the caller's arrays: the state and the stored state."""

    def __init__(self, case, seed):
        scene, _, X, V = _state(case, seed)
        dtype = torch.float32 if case["precision"] == 32 else torch.float64
        up = lambda a: torch.as_tensor(np.ascontiguousarray(a)).to(DEVICE, dtype)  # noqa: E731
        self.data = SolverData(scene, case["precision"])
        self.X0, self.V0 = up(X), up(V)
        self.X, self.V, self.XTilde = self.X0.clone(), self.V0.clone(), self.X0.clone()
        self.data.c.X, self.data.c.V = self.X.data_ptr(), self.V.data_ptr()
        self.data.c.XTilde = self.XTilde.data_ptr()
        self.sphere = None
        if case["kind"] == "collide":
            pos, r = _sphere(case)
            self.sphere = fixed.FixedBodyData([fixed.Sphere(pos=pos, radius=r)])
            self.data.set_fixed_bodies(self.sphere)
        self.params = _params(case)
        self.solver = PdSolver(128, self.data)
        self.solver.SetGlobalSolver(SolverType[case["solver"]])
        for _ in range(3):
            self.step()
        self.solver.synchronize()

    def step(self):
        self.X.copy_(self.X0)
        self.V.copy_(self.V0)
        self.XTilde.copy_(self.X0)
        self.solver.Update(self.data, self.params)
        return {"X": self.X, "V": self.V, "XTilde": self.XTilde}


class _Ipc:
    def __init__(self, case, seed):
        scene, _, X, V = _state(case, seed)
        self.data = IpcData(scene)
        self.params = IpcParams(dt=0.01, damp=0.999, dhat=1e-3, tol=5e-2, maxIterations=100, lin_tol=1e-10,
                                lin_max_iter=5000)
        up = lambda a: torch.as_tensor(np.ascontiguousarray(a)).to(DEVICE, torch.float64)  # noqa: E731
        self.X0, self.V0 = up(X), up(V)
        self.X, self.V = self.X0.clone(), self.V0.clone()
        for name, t in (("X", self.X), ("V", self.V)):  # the caller's own arrays
            self.data.arrays[name].free()
            self.data.arrays[name] = _Borrowed(t)
        self.solver = IpcSolver(self.data, elastic=case["elastic"])
        for _ in range(2):
            self.step()

    def step(self):
        self.X.copy_(self.X0)
        self.V.copy_(self.V0)
        if not self.solver.Update(self.data, self.params):
            raise RuntimeError("the IPC step failed: %r" % self.solver.stats())
        return {"X": self.X, "V": self.V}


class _Borrowed:
    """A torch tensor where IpcData keeps its device arrays."""

    def __init__(self, t):
        self.t, self.ptr = t, t.data_ptr()

    def free(self):
        self.t = None


# ----------------------------------------------------------- COO solves --

def _coo_system(case, seed, dtype):
    """Linear elasticity (12 x 12 per tet) plus mass on the diagonal: (n, values, rows, columns, right-hand side)."""
    scene, _, _, V = _state(dict(case, kind="pd", solver="PCG", bodies=1), seed)
    dev = dict(device=DEVICE, dtype=torch.float64)
    X = torch.as_tensor(scene.X).to(**dev)
    tet = torch.as_tensor(scene.tet.astype(np.int64)).to(DEVICE)
    mu, lam = (torch.as_tensor(a).to(**dev) for a in (scene.mu, scene.lam))
    P = X[tet]
    Dm = (P[:, 1:] - P[:, :1]).transpose(1, 2)
    inv, det = _inverse3(Dm)
    g = torch.cat([-inv.sum(1, keepdim=True), inv], 1)               # gradients of the 4 shape functions
    vol = det.abs() / 6
    gg = torch.einsum("tai,tbi->tab", g, g)
    eye = torch.eye(3, **dev)
    K = (mu[:, None, None, None, None] * (gg[..., None, None] * eye + torch.einsum("taj,tbi->tabij", g, g))
         + lam[:, None, None, None, None] * torch.einsum("tai,tbj->tabij", g, g)) * vol[:, None, None, None, None]
    dof = (3 * tet[:, :, None] + torch.arange(3, device=DEVICE)).reshape(-1, 12)
    K = K.permute(0, 1, 3, 2, 4).reshape(-1, 12, 12) * (10 * DT ** 2)  # h^2 K of a stiff rubber, E = 1 MPa
    n = 3 * scene.nv
    diag = torch.as_tensor(np.repeat(scene.mass + 1e3 * scene.dbc, 3)).to(**dev)
    at = torch.arange(n, device=DEVICE)
    rows = torch.cat([dof[:, :, None].expand(-1, 12, 12).reshape(-1), at])
    cols = torch.cat([dof[:, None, :].expand(-1, 12, 12).reshape(-1), at])
    vals = torch.cat([K.reshape(-1), diag])
    b = torch.as_tensor(V.reshape(-1)).to(**dev) * diag
    return n, vals.to(dtype).contiguous(), rows.int().contiguous(), cols.int().contiguous(), b.to(dtype).contiguous()


class _Coo:
    def __init__(self, case, seed):
        dtype = torch.float32 if case["precision"] == 32 else torch.float64
        self.n, self.vals, self.rows, self.cols, self.b = _coo_system(case, seed, dtype)
        self.x = torch.zeros_like(self.b)
        self.solver = PCGJacobiSolver(self.n, max_iter=2000, tolerance=_coo_tol(case), precision=case["precision"])
        self.step()

    def step(self):
        self.solver.Solve(self.n, self.b.data_ptr(), self.x.data_ptr(), self.vals.data_ptr(), self.vals.numel(),
                          self.rows.data_ptr(), self.cols.data_ptr())
        return {"x": self.x}


def _coo_tol(case):
    return 1e-3 if case["precision"] == 32 else 1e-8   # of a right-hand side of norm 10 to 30


# ---------------------------------------------------------- the interface --

def prepare(case, seed):
    return {"ipc": _Ipc, "coo": _Coo}.get(case["kind"], _Pd)(case, seed)


def run(state):
    return state.step()


def _sizes(case):
    if case["kind"] == "pd":
        dims = np.asarray(_body_dims(tuple(sorted((k, v) for k, v in case.items() if k != "name"))))
    else:
        dims = np.tile([case["nx"], case["ny"], case["nz"]], (1 if case["kind"] == "coo" else 2, 1))
    return int(np.prod(dims + 1, axis=1).sum()), int(6 * np.prod(dims, axis=1).sum())


def work(case):
    nv, nt = _sizes(case)
    s = 4 if case.get("precision") == 32 else 8
    if case["kind"] == "coo":
        n, nz = 3 * nv, 144 * nt + 3 * nv
        # the triplets once, the summed matrix (15 blocks of 9 a row, on the average) once an iteration
        its = 6 * nv ** (1 / 3)
        return {"bytes": (s + 8) * nz + 2 * s * n, "flops": 2 * 15 * 9 * nv * its}
    # positions, velocities, x~ in and out, mass and pins; tets, rest shapes and stiffness
    byte = nv * (5 * 3 * s + 2 * s) + nt * (16 + 10 * s)
    if case["kind"] == "ipc":
        its = 64 * nv ** (1 / 3)  # of a Jacobi-preconditioned solve; three solves a step
        return {"bytes": byte, "flops": 3 * (2 * 15 * 9 * nv * its + 6000 * nt)}
    # a deformation gradient, its rotation and the corner forces per tet, about 300 operations; a solve of
    # several sweeps over the scalar matrix (15 entries a row) for three right-hand sides
    sweeps = {"Jacobi": 1, "PCG": 6, "BatchedPCG": 12, "CuSolverCholesky": 6, "DenseCholesky": 6}[case["solver"]]
    return {"bytes": byte, "flops": case["iterations"] * (300 * nt + sweeps * nv * (6 * 15 + 30))}


def tolerance(case):
    """About four times what one path against another shows (both PCG kernel families, both rotations, a tighter
    inner tolerance); the velocity, a difference of positions over the time step, shows the most."""
    if case["kind"] == "ipc":
        return {"rel": 5e-8}    # inner solves stopped at 1e-9 instead of 1e-10: 3e-9
    if case["kind"] == "coo":
        return {"rel": 2e-4 if case["precision"] == 32 else 1e-8}
    if case["precision"] == 64:
        return {"rel": 2e-5}    # a solve may stop an iteration sooner or later: 4e-6 from the 64-bit reference
    return {"rel": 1e-3, "max": 0.02}    # 3e-4 and 3e-3 at 64^3 between the two PCG kernel families


# ------------------------------------------------------- 64-bit reference --

def _inverse3(D):
    """(inverse, determinant) of (..., 3, 3)."""
    r = [torch.linalg.cross(D[..., (i + 1) % 3], D[..., (i + 2) % 3], dim=-1) for i in range(3)]
    adj = torch.stack(r, dim=-2)
    det = (adj[..., 0, :] * D[..., :, 0]).sum(-1)
    return adj / det[..., None, None], det


def _rotation(F):
    """The rotation of the polar decomposition (Newton's iteration; the states hold no inverted element)."""
    R = F
    for _ in range(9):
        inv, _ = _inverse3(R)
        R = 0.5 * (R + inv.transpose(1, 2))
    return R


def _rounded(a, case):
    a = np.asarray(a)
    return torch.as_tensor(a.astype(np.float32) if case["precision"] == 32 else a).to(DEVICE, torch.float64)


def _exact_step(case, seed):
    """One PD step in 64 bits: the positions after the local/global iterations, and the state it started from."""
    scene, body_np, X_np, V_np = _state(case, seed)
    rest, X, V, mass, mu, dbc = (_rounded(a, case) for a in (scene.X, X_np, V_np, scene.mass, scene.mu, scene.dbc))
    tet = torch.as_tensor(scene.tet.astype(np.int64)).to(DEVICE)
    body = torch.as_tensor(body_np).to(DEVICE)
    nv, nb = scene.nv, int(body_np.max()) + 1 if case["solver"] == "BatchedPCG" else 1
    if nb == 1:
        body = torch.zeros_like(body)
    P = rest[tet]
    inv, det = _inverse3((P[:, 1:] - P[:, :1]).transpose(1, 2))
    w = det.abs() / 6 * mu
    g = torch.cat([-inv.sum(1, keepdim=True), inv], 1)
    K = w[:, None, None] * torch.einsum("tai,tbi->tab", g, g)
    rows = tet[:, :, None].expand(-1, 4, 4).reshape(-1)
    cols = tet[:, None, :].expand(-1, 4, 4).reshape(-1)
    key, at = torch.unique(rows * nv + cols, return_inverse=True)
    val = torch.zeros(len(key), device=DEVICE, dtype=torch.float64).index_add_(0, at, K.reshape(-1))
    rows, cols = key // nv, key % nv
    del key, at, K
    pin = dbc > 0
    c = (mass + 1e6 * dbc) / DT ** 2
    val = val + torch.where(rows == cols, c[rows], torch.zeros_like(val))
    diag = torch.zeros(nv, device=DEVICE, dtype=torch.float64).index_add_(0, rows[rows == cols], val[rows == cols])
    A = torch.sparse_coo_tensor(torch.stack([rows, cols]), val, (nv, nv)).to_sparse_csr()

    def per_body(q):
        return torch.zeros((nb, 3), device=DEVICE, dtype=torch.float64).index_add_(0, body, q) if nb > 1 else q.sum(0)[None]

    def spread(a):
        return a[body] if nb > 1 else a

    def pcg(b, x, tol, floor, most):
        r = b - A @ x
        z = r / diag[:, None]
        p, rz, zz = z, per_body(r * z), per_body(z * z)
        # the batched solver measures b from each body's first vertex
        b0 = b - c[:, None] * spread(origin) if nb > 1 else b
        thr = torch.maximum(tol ** 2 * zz, floor ** 2 * per_body((b0 / diag[:, None]) ** 2))
        act = zz > thr
        for _ in range(most):
            if not bool(act.any()):
                break
            q = A @ p
            pq = per_body(p * q)
            alpha = torch.where(act & (pq != 0), rz / pq, torch.zeros_like(rz))
            x = x + spread(alpha) * p
            r = r - spread(alpha) * q
            z = r / diag[:, None]
            new, zz = per_body(r * z), per_body(z * z)
            beta = torch.where(act & (rz != 0), new / rz, torch.zeros_like(rz))
            p, rz = z + spread(beta) * p, new
            act = act & (zz > thr)
        return x

    first = torch.full((nb,), nv, device=DEVICE, dtype=torch.long).scatter_reduce_(
        0, body, torch.arange(nv, device=DEVICE), "amin")
    origin = rest[first]
    sn = X + DT * V
    sn[:, 1] -= 9.8 * mass / c
    jacobi, pcg_solver = case["solver"] == "Jacobi", case["solver"] in ("PCG", "BatchedPCG")
    cheb = jacobi or case["solver"] == "BatchedPCG" or (case["solver"] == "PCG" and case["chebyshev"])
    base = c[:, None] * sn
    s, prev, omega, rho = sn, sn if cheb else torch.zeros_like(sn), 1.0, 0.9992
    for i in range(case["iterations"]):
        Q = s[tet]
        F = (Q[:, 1:] - Q[:, :1]).transpose(1, 2) @ inv
        R = _rotation(F)
        f = w[:, None, None] * torch.einsum("tij,taj->tai", R - F if jacobi else R, g)
        b = base.clone().index_add_(0, tet.reshape(-1), f.reshape(-1, 3))
        b = torch.where(pin[:, None], rest * 1e6 / DT ** 2, b)
        if jacobi:
            x = (b - c[:, None] * s) / diag[:, None] + s
        elif pcg_solver:
            x = pcg(b, s, 1e-6, 1e-8 if case["precision"] == 32 else 0.0, 200)
        else:
            x = pcg(b, s, 1e-13, 1e-15, 4000)
        if cheb:
            if i > 10:
                omega = 2 / (2 - rho ** 2) if i == 11 else 4 / (4 - rho ** 2 * omega)
            damped = 0.9 * (x - s) + s
            s, prev = (damped - prev) * omega + prev, s
        else:
            err = float(((prev - x) ** 2).mean())
            s = prev = x
            if math.sqrt(err) < _params(case).tol:
                break
    return X, s


def exact(case, seed):
    if case["kind"] == "ipc":
        return None  # the step works in 64 bits itself: its outputs at the start are the reference
    if case["kind"] == "coo":
        n, vals, rows, cols, b = _coo_system(case, seed, torch.float32 if case["precision"] == 32 else torch.float64)
        A = torch.sparse_coo_tensor(torch.stack([rows.long(), cols.long()]), vals.double(), (n, n))
        A = A.coalesce().to_sparse_csr()
        at = torch.arange(n, device=DEVICE)
        same = rows == cols
        diag = torch.zeros(n, device=DEVICE, dtype=torch.float64).index_add_(0, rows[same].long(), vals[same].double())
        del at
        x, r = torch.zeros_like(diag), b.double()
        z = r / diag
        p, rz = z, r @ z
        for _ in range(2000):
            if float(r.norm()) < _coo_tol(case) or abs(float(rz)) < 1e-15:
                break
            q = A @ p
            alpha = rz / (p @ q)
            x, r = x + alpha * p, r - alpha * q
            z = r / diag
            new = r @ z
            p, rz = z + new / rz * p, new
        return {"x": x}
    X, s = _exact_step(case, seed)
    if case["kind"] == "collide":
        # the sphere pushes x~ out; what the contact response makes of X and V has no 64-bit value here
        pos, radius = _sphere(case)
        centre = torch.as_tensor(np.float32(pos)).to(DEVICE, torch.float64)
        to = s - centre
        d = to.norm(dim=1, keepdim=True)
        return {"X": None, "V": None, "XTilde": torch.where(d < radius, centre + to / d * radius, s)}
    return {"X": s, "V": (s - X) / DT, "XTilde": s}
