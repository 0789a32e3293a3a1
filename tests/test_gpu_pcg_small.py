"""A PCG solve in one workgroup (systems of up to 1,024 rows) against the
row-gather kernels: one wavefront, a part of one, the largest size of the rule
and one past it, rows of exactly the entries held in registers and of more,
the Chebyshev form, the early exit of the local/global loop and solves cut by
the iteration limit.

Bounds: in FP64 both sides stop at ||D^-1 r|| <= 1e-13 of its start (1e-10
relative, the bar of the PCG tests).  In FP32 both stop by the same test and
differ in the sums' order, so the distance to the FP64 solution may be at most
twice the row-gather kernels' plus 1e-6 (8 units of FP32 rounding of the
positions that are handed back)."""
import numpy as np
import pytest

from conftest import rel_err
from test_gpu_pcg_quads import body, fan
from test_gpu_pd import graph_pair
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
        for _ in range(3):
            pd.Update(data, p)
        pd.synchronize()
        return data.get("X"), pd.stats()
    finally:
        pd.close()
        data.free()


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("mode", ["chebyshev", "all iterations", "early exit"])
@pytest.mark.parametrize("size", [(1, 1, 1), (3, 3, 3), (1, 4, 12), (7, 7, 15), (4, 4, 40), "fan 15", "fan 16", "fan 60"])
def test_matches_the_row_gather_kernels(gpu, size, mode, precision):
    s = fan(int(size.split()[1])) if isinstance(size, str) else body(*size)
    kw = dict(pcg_chebyshev=mode == "chebyshev", tol=1e-4 if mode == "early exit" else 0.0)
    x, st = solve(s, precision, **kw)
    ref, sr = solve(s, 64, pcg_halo=0, **kw)
    assert st.pcg_cap_hits == 0 and st.pcg_iterations_total > 0
    if mode != "early exit":
        assert st.pcg_solves_total == 18
    if precision == 64:
        assert st.pcg_solves_total == sr.pcg_solves_total
        assert rel_err(x, ref) < 1e-10, rel_err(x, ref)
    else:
        gather, sg = solve(s, 32, pcg_halo=0, **kw)
        assert st.pcg_solves_total == sg.pcg_solves_total
        assert rel_err(x, ref) <= 2 * rel_err(gather, ref) + 1e-6, (rel_err(x, ref), rel_err(gather, ref))


@pytest.mark.parametrize("precision", [32, 64])
def test_iteration_limit(gpu, precision):
    """Solves cut at 3 iterations: the same iterates as the row-gather kernels
    (three iterations' rounding apart) and every solve counted as cut."""
    s = body(4, 5, 6)
    kw = dict(pcg_chebyshev=True, pcg_max_iter=3, pcg_adaptive=False)
    x, st = solve(s, precision, **kw)
    ref, sr = solve(s, precision, pcg_halo=0, **kw)
    assert st.pcg_iterations_total == sr.pcg_iterations_total == 3 * 18
    assert st.pcg_cap_hits == sr.pcg_cap_hits == 18
    assert rel_err(x, ref) < (1e-5 if precision == 32 else 1e-12)


@pytest.mark.parametrize("mode", ["chebyshev", "early exit", "more solves than the log"])
def test_graph_is_captured_once(gpu, mode):
    """The launches of a step do not depend on the iteration counts, so the first
    step is captured and replayed from then on, solves that the early exit skips
    and solves past the 64 that the step's log holds among them."""
    p = SolverParams(numIterations=70 if mode == "more solves than the log" else 8, dt=1.0 / 60.0, rho=0.9992,
                     tol=1e-4 if mode == "early exit" else 0.0, pcg_tol=1e-6, pcg_floor=1e-8, pcg_max_iter=400,
                     pcg_chebyshev=mode == "chebyshev", pcg_adaptive=True)

    def check(k, xg, xe):
        np.testing.assert_array_equal(xg, xe, err_msg=f"step {k}")  # every sum has a fixed order

    sg, se = graph_pair(body(4, 5, 6), SolverType.PCG, p, 8, check)
    assert sg.graph_captures == 1 and sg.graph_replays == 8
    assert sg.pcg_solves_total == se.pcg_solves_total
    if mode == "early exit":
        assert se.pcg_solves_total < 8 * 8
    assert se.graph_captures == 0 and se.graph_replays == 0


def test_kernel_timing_counts_solves(gpu):
    """A solve is one launch: the timer has whole solves and no iteration launches."""
    data = SolverData(body(4, 5, 6), 32)
    pd = PdSolver(128, data)
    pd.SetGlobalSolver(SolverType.PCG)
    pd.set_kernel_timing(("local_step", "pcg_iteration", "pcg_solve"))
    try:
        for _ in range(2):
            pd.Update(data, SolverParams(numIterations=5, dt=1.0 / 60.0, tol=0.0, pcg_chebyshev=True))
        assert pd.kernel_time("local_step")[0] == 10
        launches, ms = pd.kernel_time("pcg_solve")
        assert launches == 10 and ms > 0
        assert pd.kernel_time("pcg_iteration") == (0, 0.0)
    finally:
        pd.close()
        data.free()
