"""Points in planar runs (one plane per triangle of a patch) against the FP64
CPU oracle: every rule, runs of several lengths, and sets that are not such
runs, in near coefficients (stored and on the fly) and energy coefficients."""
import numpy as np
import pytest

import oracle
from beep3_amd.device import Device
from beep3_amd.scene import Mesh, Scene

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def renormalise(ef, a):
    """The oracle's f coefficients are Gauss-renormalised: the gap between the
    net charge and -sum(ef) is spread by area (one instance)."""
    return ef - a["area"] / a["area"].sum() * (a["charges"][:, 3].sum() + ef.sum())


def charges(n, seed, radius):
    r = np.random.default_rng(seed)
    d = r.normal(size=(n, 3))
    d *= (0.6 * radius * r.uniform(size=n) ** (1 / 3) / np.linalg.norm(d, axis=1))[:, None]
    return np.concatenate([d, r.normal(size=(n, 1))], axis=1)


def arrays(quad, qual, kappa, nbsize=60, nc=37):
    sc = Scene(80.0, kappa, quad, qual, nbsize)
    m = Mesh.star(2, 8.0, 8, 0.08, 3)
    sc.add_instance(m.set_charges(charges(nc, 4, 8.0)), 2.0)
    sc.build()
    return sc.arrays()


def check(a, kappa):
    n = a["area"].shape[0]
    x = np.random.default_rng(n).normal(size=2 * n)
    orc = oracle.Oracle(a, kappa, 80.0)
    ref = orc.matvec(x)
    # first-order rounding of the FP32 set: 16 roundings to form a coefficient,
    # twice that with FP32 products and sums
    u = 2.0 ** -24 * np.linalg.norm(np.abs(orc.assemble()) @ np.abs(x)) / np.linalg.norm(ref)
    for near in ("precompute", "on_the_fly"):
        d = Device(0)
        d.set_far_field("direct", 5, 40)
        d.set_geometry(a)
        d.set_tree(a)
        d.set_near_mode(near)
        for p, tol in (("fp64", 1e-12), ("fp32", 32 * u)):
            d.precompute(kappa, p)
            err = rel(d.matvec(x, p), ref)
            print(n, near, p, err, tol, flush=True)
            assert err < tol
        ef, eh = d.energy_coefficients(a["inst_patch_ptr"], a["inst_charge_ptr"], a["charges"])
        ef = renormalise(ef, a)
        rf, rh = orc.energy_coeffs()
        assert rel(ef, rf) < 1e-12 and rel(eh, rh) < 1e-12
        d.close()


# runs of 2 (kept as points), 8, 12, 14 and 32; one and many row points
@pytest.mark.parametrize("quad,qual", [(1, 0), (4, 0), (6, 0), (7, 1), (16, 0), (6, 4), (0, 0)])
@pytest.mark.parametrize("kappa", [0.125, 0.0])
def test_rules(quad, qual, kappa):
    check(arrays(quad, qual, kappa), kappa)


@pytest.mark.parametrize("case", ["bent", "shifted", "coplanar", "ragged"])
def test_points_that_are_not_runs(case):
    """One patch whose points have another normal, one whose points leave the
    plane, a first patch with several triangles in one plane, and a last patch
    one point short: all against the oracle on the same points."""
    a = {k: (v.copy() if isinstance(v, np.ndarray) else v) for k, v in arrays(6, 0, 0.125).items()}
    q = a["quad"]
    k = a["quad_ptr"][70] + 5
    if case == "bent":
        q[k, 3:6] = q[k + 12, 3:6]
    elif case == "shifted":
        q[k, :3] += 1e-3 * q[k, 3:6]
    elif case == "coplanar":
        e = a["quad_ptr"][1]
        q[:e, 2] = q[0, 2]
        q[:e, 3:6] = (0.0, 0.0, 1.0)
    else:
        a["quad_ptr"][-1] -= 1
        a["quad"] = q[:-1].copy()
    check(a, 0.125)


# one charge, odd numbers, and charges on and near the surface
@pytest.mark.parametrize("nc", [1, 2, 129, 300])
def test_energy_charges(nc):
    a = arrays(4, 0, 0.1, nc=nc)
    c = a["charges"]
    g = a["gal"]
    c[0, :3] = g[11, :3]          # on a point: contributes nothing there
    if nc > 2:
        c[2, :3] = g[40, :3] + 0.02 * g[40, 3:6]
        c[nc - 1, :3] = a["centroid"][9]
    d = Device(0)
    d.set_far_field("direct", 5, 40)
    d.set_geometry(a)
    d.set_tree(a)
    ef, eh = d.energy_coefficients(a["inst_patch_ptr"], a["inst_charge_ptr"], a["charges"])
    ef = renormalise(ef, a)
    rf, rh = oracle.Oracle(a, 0.1, 80.0).energy_coeffs()
    print(nc, rel(ef, rf), rel(eh, rh), flush=True)
    assert rel(ef, rf) < 1e-12 and rel(eh, rh) < 1e-12
    d.close()


def test_planar_beside_curved_and_far_from_the_origin():
    """Scenes that keep a normal per point: a planar mesh beside a curved one,
    and a mesh so far from the origin that the rounding of its coordinates
    takes its points off their planes; against the oracle."""
    mixed = Scene(80.0, 0.125, 6, 0, 60)
    mixed.add_instance(Mesh.star(2, 8.0, 8, 0.08, 3).set_charges(charges(5, 4, 8.0)), 2.0)
    bent = Mesh.star(2, 8.0, 8, 0.08, 7).set_charges(charges(5, 6, 8.0))
    bent.set_curved(True)
    mixed.add_instance(bent, 3.0, offset=[20.0, 0.0, 0.0])
    away = Scene(80.0, 0.125, 6, 0, 60)
    away.add_instance(Mesh.star(2, 8.0, 8, 0.08, 3).set_charges(charges(5, 4, 8.0)), 2.0,
                      offset=[30000.0, -20000.0, 10000.0])
    for sc in (mixed, away):
        a = sc.build().arrays()
        n = a["area"].shape[0]
        x = np.random.default_rng(n).normal(size=2 * n)
        orc = oracle.Oracle(a, 0.125, 80.0)
        ref = orc.matvec(x)
        u = 2.0 ** -24 * np.linalg.norm(np.abs(orc.assemble()) @ np.abs(x)) / np.linalg.norm(ref)
        # differences of coordinates c carry their rounding, 2^-53 c over a
        # distance of at least a third of a patch (0.5 A), cubed in the kernels
        far = 2.0 ** -53 * np.abs(a["centroid"]).max() / 0.5 * 3 * 8
        for near in ("precompute", "on_the_fly"):
            d = Device(0)
            d.set_far_field("direct", 5, 40)
            d.set_geometry(a)
            d.set_tree(a)
            d.set_near_mode(near)
            for p, tol in (("fp64", 1e-12 + far), ("fp32", 32 * u + far)):
                d.precompute(0.125, p)
                err = rel(d.matvec(x, p), ref)
                print(n, near, p, err, tol, flush=True)
                assert err < tol
            d.close()


def test_energy_without_charges():
    a = arrays(4, 0, 0.1, nc=3)
    d = Device(0)
    d.set_geometry(a)
    ef, eh = d.energy_coefficients(a["inst_patch_ptr"], np.zeros(2, np.int32), np.zeros((0, 4)))
    assert np.all(ef == 0) and np.all(eh == 0)
    d.close()


# two runs a patch, shorter and longer than the 64 points staged at a time
@pytest.mark.parametrize("gs", [3, 4, 20, 64, 65, 100])
def test_energy_run_lengths(gs):
    a = dict(arrays(4, 0, 0.1, nc=150))
    n = a["area"].shape[0]
    r = np.random.default_rng(gs)
    nrm = a["normal"][:, None] + 0.1 * r.normal(size=(n, 2, 3))
    nrm /= np.linalg.norm(nrm, axis=2)[..., None]
    t = r.normal(size=(n, 2, gs, 3)) * 0.3
    t -= np.sum(t * nrm[:, :, None], axis=3)[..., None] * nrm[:, :, None]
    g = np.empty((n, 2, gs, 7))
    g[..., :3] = a["centroid"][:, None, None] + t
    g[..., 3:6] = nrm[:, :, None]
    g[..., 6] = a["area"][:, None, None] / (2 * gs) * r.uniform(0.5, 1.5, size=(n, 2, gs))
    a["gal"] = np.ascontiguousarray(g.reshape(-1, 7))
    a["gal_ptr"] = np.arange(n + 1, dtype=np.int32) * (2 * gs)
    d = Device(0)
    d.set_geometry(a)
    ef, eh = d.energy_coefficients(a["inst_patch_ptr"], a["inst_charge_ptr"], a["charges"])
    rf, rh = oracle.Oracle(a, 0.1, 80.0).energy_coeffs()
    print(gs, rel(renormalise(ef, a), rf), rel(eh, rh), flush=True)
    assert rel(renormalise(ef, a), rf) < 1e-12 and rel(eh, rh) < 1e-12
    d.close()


def test_one_context_over_point_sets_of_both_forms():
    """Whether a set is in planar runs is found again for every geometry."""
    planar = arrays(6, 0, 0.125)
    bent = {k: (v.copy() if isinstance(v, np.ndarray) else v) for k, v in planar.items()}
    for s in ("quad", "gal"):
        k = bent[f"{s}_ptr"][70] + 1
        bent[s][k, 3:6] = bent[s][k + 12, 3:6]
    point = arrays(0, 0, 0.125)
    d = Device(0)
    d.set_far_field("direct", 5, 40)
    x = np.random.default_rng(2).normal(size=2 * planar["area"].shape[0])
    for a in (planar, bent, bent, planar, point, planar):
        d.set_geometry(a)
        d.set_tree(a)
        d.precompute(0.125, "fp64")
        orc = oracle.Oracle(a, 0.125, 80.0)
        assert rel(d.matvec(x, "fp64"), orc.matvec(x)) < 1e-12
        ef, eh = d.energy_coefficients(a["inst_patch_ptr"], a["inst_charge_ptr"], a["charges"])
        rf, rh = orc.energy_coeffs()
        assert rel(renormalise(ef, a), rf) < 1e-12 and rel(eh, rh) < 1e-12
    d.close()
