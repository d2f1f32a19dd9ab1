"""The direct far field as symmetric tile pairs and the FP64 set without a far
field, against the FP64 CPU oracle, at the edges of the 256- and 64-patch
tiles and of the SpMV's work items, over the routes to them (without
allocations: test_zz_no_alloc.py)."""
import threading

import numpy as np
import pytest

import oracle
from beep3_amd._lib import BeepError
from beep3_amd.device import Device
from beep3_amd.scene import Mesh, Scene

pytestmark = pytest.mark.gpu



def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def bounds(orc, x, ref):
    """Relative error bounds of a mat-vec: FP64 rounding, and for the FP32 set
    first-order rounding of the products, c u ||K||x|| / |K x| with u = 2^-24:
    c = 16 roundings to form a coefficient (about ten on its longest chain,
    more where terms nearly cancel), twice that with FP32 products and sums
    (at most 16 partial sums deep in blocks)."""
    u = 2.0 ** -24 * np.linalg.norm(np.abs(orc.assemble()) @ np.abs(x)) / np.linalg.norm(ref)
    return {"fp64": 1e-12, "fp32": 32 * u, "fp32_resid": 16 * u}


def scene(levels, nbsize, kappa=0.125):
    sc = Scene(80.0, kappa, 6, 0, nbsize)
    for k, lv in enumerate(levels):
        sc.add_instance(Mesh.star(lv, 25.0, 8, 0.04, 5 + k), 2.0 + k, offset=[70.0 * k, 3.0 * k, 0.0])
    return sc.build().arrays()


def device(a, far="auto", kappa=0.125, near="precompute", precs=("fp64", "fp32")):
    d = Device(0)
    d.set_far_field(far, 5, 40)
    d.set_geometry(a)
    d.set_tree(a)
    d.set_near_mode(near)
    for p in precs:
        d.precompute(kappa, p)
    return d


# 42 .. 3,204 patches: one to thirteen super-tiles, odd and even rings, last
# tiles of 2 .. 42 patches, one leaf and many
@pytest.mark.parametrize("levels,nbsize", [((1,), 1500), ((2,), 30), ((1, 2, 1), 1500), ((2, 2, 2, 1), 50),
                                           ((3,), 1500), ((3, 2), 100), ((3, 3, 2), 60), ((4, 3), 200),
                                           ((4,), 1500)])
@pytest.mark.parametrize("kappa", [0.125, 0.0])
def test_direct_matvec_against_oracle(levels, nbsize, kappa):
    a = scene(levels, nbsize, kappa)
    n = a["area"].shape[0]
    x = np.random.default_rng(n).normal(size=2 * n)
    orc = oracle.Oracle(a, kappa, 80.0)
    ref = orc.matvec(x)
    d = device(a, kappa=kappa)
    for p, tol in bounds(orc, x, ref).items():
        y = d.matvec(x, p)
        print(n, nbsize, kappa, p, rel(y, ref), tol, flush=True)
        assert rel(y, ref) < tol
        d.set_overlap(False)
        for cap in (0, 1):  # one block per work item; blocks that take the next free one
            d.set_spmv_residency(cap)
            assert np.array_equal(d.matvec(x, p), y)
        d.set_overlap(True)
    # sets made for either form of the direct far field serve both modes
    d.set_far_field("direct", 5, 40)
    assert rel(d.matvec(x, "fp64"), ref) < 1e-12
    d.close()


@pytest.mark.parametrize("levels,nbsize", [((3,), 1500), ((3, 2), 100), ((4,), 60)])
def test_spmv_settings_of_the_one_launch(levels, nbsize):
    """Near and far field in one launch: the load depth applies and changes no
    bits, and can be tuned; no residency cap applies, so its tuner gives every
    candidate one time and keeps the setting."""
    a = scene(levels, nbsize)
    n = a["area"].shape[0]
    x = np.random.default_rng(n).normal(size=2 * n)
    d = device(a, far="direct")
    for p in ("fp64", "fp32", "fp32_resid"):
        d.set_spmv_depth(1)
        d.set_spmv_residency(1)  # not among the candidates below
        y = d.matvec(x, p)
        for depth in (2, 4):
            d.set_spmv_depth(depth)
            assert np.array_equal(d.matvec(x, p), y), (depth, p)
        best, table = d.autotune_spmv_depth(p, (1, 2, 4), reps=2)
        assert table[best] == min(table.values())
        best, table = d.autotune_spmv(p, (3, 0, 2), reps=2)
        assert best == 3 and len(set(table.values())) == 1
        d.set_spmv_residency(2)
        assert d.autotune_spmv(p, (3, 0, 2), reps=2)[0] == 2
        assert np.array_equal(d.matvec(x, p), y)
    d.close()


@pytest.mark.parametrize("levels,nbsize", [((3,), 1500), ((3, 2), 100)])
def test_direct_matvec_on_the_fly(levels, nbsize):
    a = scene(levels, nbsize)
    n = a["area"].shape[0]
    x = np.random.default_rng(n).normal(size=2 * n)
    orc = oracle.Oracle(a, 0.125, 80.0)
    ref = orc.matvec(x)
    d = device(a, near="on_the_fly")
    for p, tol in bounds(orc, x, ref).items():
        assert rel(d.matvec(x, p), ref) < tol
    d.close()


def test_shared_near_field_of_a_one_leaf_mesh():
    """A context whose FP64 set has no far field, then shared: the pose over
    two copies of it matches the oracle of the scene with the same pairs."""
    one = scene((3,), 1500)
    n = one["area"].shape[0]
    src = device(one)
    x1 = np.random.default_rng(1).normal(size=2 * n)
    y1 = src.matvec(x1, "fp64")
    sc = Scene(80.0, 0.125, 6, 0, 1500)
    m = Mesh.star(3, 25.0, 8, 0.04, 5)
    two = sc.add_instance(m, 2.0).add_instance(m, 2.0, offset=[80.0, 0.0, 0.0]).build().arrays()
    x = np.random.default_rng(2).normal(size=4 * n)
    pose = Device(0)
    pose.set_far_field("direct", 5, 40)
    pose.set_geometry(two)
    pose.share_near(src, [0, n])
    lists = dict(two)
    lists["leaf_ptr"] = np.array([0, n, 2 * n], np.int32)
    lists["leaf_idx"] = np.arange(2 * n, dtype=np.int32)
    lists["nb_ptr"] = lists["leaf_ptr"]
    lists["nb_idx"] = lists["leaf_idx"]
    orc = oracle.Oracle(lists, 0.125, 80.0)
    ref = orc.matvec(x)
    for p, tol in bounds(orc, x, ref).items():
        pose.precompute(0.125, p)
        assert rel(pose.matvec(x, p), ref) < tol
    assert rel(src.matvec(x1, "fp64"), y1) < 1e-12
    pose.close()
    src.close()


def test_sharing_leaves_the_source_as_it_is():
    """Sharing only reads the source: its FP64 product keeps its bits, also
    while another thread shares it; a refused share costs it nothing; and the
    contexts that share it follow a new precompute of it."""
    one = scene((3,), 1500)
    n = one["area"].shape[0]
    src = device(one)
    x1 = np.random.default_rng(1).normal(size=2 * n)
    y1 = src.matvec(x1, "fp64")
    held = src.memory_held()
    two = Scene(80.0, 0.125, 6, 0, 1500)
    m = Mesh.star(3, 25.0, 8, 0.04, 5)
    two = two.add_instance(m, 2.0).add_instance(m, 2.0, offset=[80.0, 0.0, 0.0]).build().arrays()
    x = np.random.default_rng(2).normal(size=4 * n)
    poses = [Device(0) for _ in range(3)]
    for d in poses:
        d.set_far_field("direct", 5, 40)
        d.set_geometry(two)
    with pytest.raises(BeepError, match="overlap"):
        poses[0].share_near(src, [0, 0])
    assert src.memory_held() == held and np.array_equal(src.matvec(x1, "fp64"), y1)
    out = [None] * 3

    def share(k):
        poses[k].share_near(src, [0, n])
        poses[k].precompute(0.125, "fp64")
        out[k] = poses[k].matvec(x, "fp64")

    threads = [threading.Thread(target=share, args=(k,)) for k in range(3)]
    for t in threads:
        t.start()
    same = [np.array_equal(src.matvec(x1, "fp64"), y1) for _ in range(50)]
    for t in threads:
        t.join()
    assert all(same) and np.array_equal(src.matvec(x1, "fp64"), y1)
    assert all(np.array_equal(o, out[0]) for o in out)
    assert src.sanity_check() == 0
    # a new precompute of a shared source (the set in another form), then of
    # a new tree (folded again)
    src.precompute(0.125, "fp64")
    poses[0].precompute(0.125, "fp64")
    assert rel(poses[0].matvec(x, "fp64"), out[0]) < 1e-13
    src.set_tree(one)
    src.precompute(0.125, "fp64")
    poses[0].precompute(0.125, "fp64")
    assert rel(poses[0].matvec(x, "fp64"), out[0]) < 1e-13
    for d in poses:
        d.close()
    src.close()


@pytest.mark.parametrize("near", ["precompute", "on_the_fly"])
@pytest.mark.parametrize("kappa", [0.125, 0.0])
def test_bad_entries_keep_the_one_point_interaction(near, kappa):
    """A pair whose integral is not a number counts as one entry repaired and
    contributes its 1-point interaction, also in the FP64 set that has no far
    field: quadrature points with NaN normals against the oracle with one
    point at the centroid in their place."""
    a = scene((3,), 1500, kappa)
    n = a["area"].shape[0]
    p = 3
    k0, k1 = a["quad_ptr"][p], a["quad_ptr"][p + 1]
    one = np.concatenate([a["centroid"][p], a["normal"][p], a["area"][p:p + 1]])
    b = dict(a)
    b["quad"] = np.concatenate([a["quad"][:k0], one[None], a["quad"][k1:]])
    b["quad_ptr"] = a["quad_ptr"].copy()
    b["quad_ptr"][p + 1:] -= k1 - k0 - 1
    orc = oracle.Oracle(b, kappa, 80.0)
    x = np.random.default_rng(n).normal(size=2 * n)
    ref = orc.matvec(x)
    a["quad"] = a["quad"].copy()
    a["quad"][k0:k1, 3:6] = np.nan
    for far in ("auto", "direct"):
        d = device(a, far=far, kappa=kappa, near=near)
        for prec, tol in bounds(orc, x, ref).items():
            assert rel(d.matvec(x, prec), ref) < tol, (far, prec)
        if near == "precompute":
            assert d.guard_stats()["fp64"] == n - 1
            assert d.sanity_check() == 0
        d.close()


def test_guard_bound_without_far_field():
    """The entries over a low guard bound are the same with the direct far
    field chosen by size (no far field in FP64) and asked for."""
    a = scene((3,), 1500)
    n = a["area"].shape[0]
    x = np.random.default_rng(n).normal(size=2 * n)
    out = []
    for far in ("auto", "direct"):
        d = device(a, far=far, precs=("fp64",))
        d.set_guard(1e-3)
        d.precompute(0.125, "fp64")
        y = d.matvec(x, "fp64")
        out.append((d.guard_stats(), d.sanity_check(), y, d.matvec(x, "fp64")))
        d.close()
    (sa, ca, ya, za), (sd, cd, yd, zd) = out
    print(sa, sd, ca, cd, rel(ya, yd), flush=True)
    assert 0 < sd["fp64"] < n * (n - 1) and sa == sd and ca == cd
    assert rel(ya, yd) < 1e-12 and rel(za, zd) < 1e-12
