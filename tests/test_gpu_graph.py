"""GPU: GMRES Arnoldi steps replayed from captured HIP graphs give the same
bits as the same kernels launched one by one, on every replay (each solve
replays a graph once per iteration, with eager refinement work and host
synchronisation in between), for the direct and the FMM far field; solves
that alternate precisions reuse their cached graphs."""
import numpy as np
import pytest

from beep3_amd import configs
from beep3_amd.device import Device
from beep3_amd.scene import Scene

pytestmark = pytest.mark.gpu


def _device(b, Dp, far, precs):
    sc = Scene(b.Dsolvent, b.kappa, b.quad, b.qual, b.nbsize)
    sc.add_instance(b.library[0], Dp)
    sc.build()
    a = sc.arrays()
    d = Device(0)
    d.set_far_field(far, 5, 40)
    d.set_geometry(a)
    d.set_tree(a)
    for p in precs:
        d.precompute(b.kappa, p)
    return d, sc, a


# born_auto: one leaf, no far field in FP64; off_centre_direct: above the
# symmetric far field's sizes
@pytest.mark.parametrize("case", ["born_direct", "born_auto", "off_centre_fmm", "off_centre_direct"])
def test_graph_replay_matches_eager(case):
    far = case.split("_")[-1]
    if case.startswith("born"):
        b, Dp = configs.born_ion(), 2.0
    else:
        b, Dp = configs.off_centre(), 4.0
    d, sc, a = _device(b, Dp, far, ("fp64", "fp32"))
    rhs = d.rhs(a["charges"], b.Dsolvent)
    out = {}
    for mode in ("fp64", "mixed"):
        d.set_graphs(False)
        x0, st0 = d.solve(rhs, tol=1e-6, max_iter=100, mode=mode)
        d.set_graphs(True)
        x1, st1 = d.solve(rhs, tol=1e-6, max_iter=100, mode=mode)
        x2, st2 = d.solve(rhs, tol=1e-6, max_iter=100, mode=mode)
        out[mode] = (st0["iterations"], st1["iterations"])
        assert st0["converged"] and st1["converged"]
        assert st0["iterations"] == st1["iterations"] == st2["iterations"]
        assert np.array_equal(x0, x1), mode
        assert np.array_equal(x1, x2), mode
    print(case, "iterations (eager, graph):", out)
    d.close()


def test_cached_graphs_across_alternating_solves():
    """FP64 and mixed solves in turn keep one cached step graph per precision;
    every solve matches the eager solve of its mode bit for bit."""
    b = configs.off_centre()
    d, sc, a = _device(b, 4.0, "fmm", ("fp64", "fp32"))
    rhs = d.rhs(a["charges"], b.Dsolvent)
    d.set_graphs(False)
    eager = {m: d.solve(rhs, tol=1e-6, max_iter=100, mode=m)[0] for m in ("fp64", "mixed", "fp32")}
    d.set_graphs(True)
    for m in ("fp64", "mixed", "fp64", "fp32", "mixed", "fp64", "fp32"):
        x, st = d.solve(rhs, tol=1e-6, max_iter=100, mode=m)
        assert st["converged"], m
        assert np.array_equal(x, eager[m]), m
    d.close()


def test_device_resident_solves_match_host_solve():
    """RHS and solve on device vectors give the bits of the host-vector calls."""
    b = configs.born_ion()
    d, sc, a = _device(b, 2.0, "direct", ("fp64", "fp32"))
    rhs = d.rhs(a["charges"], b.Dsolvent)
    n = rhs.shape[0]
    db, dx = d.alloc(8 * n), d.alloc(8 * n)
    d.rhs_device(a["charges"], b.Dsolvent, db)
    assert np.array_equal(d.download(np.empty(n), db), rhs)
    for mode in ("fp64", "mixed"):
        x0, st0 = d.solve(rhs, tol=1e-6, max_iter=100, mode=mode)
        d.upload(dx, np.zeros(n))
        st1 = d.solve_device(db, dx, tol=1e-6, max_iter=100, mode=mode)
        assert st1["iterations"] == st0["iterations"], mode
        assert np.array_equal(d.download(np.empty(n), dx), x0), mode
    d.free(db)
    d.free(dx)
    d.close()
