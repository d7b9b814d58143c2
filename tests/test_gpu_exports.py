"""The exports and monitors read the state directly, in every layout, storage
form and addressing: fields and stresses against the oracle's formulas on the
exported distributions (bitwise, as the formulas are binary64 in one order),
the exported distributions against the oracle's run, the reductions against
numpy over the exported fields."""
import ctypes as C

import numpy as np
import pytest

from hemelb_amd import _native as N
from hemelb_amd import lb as L
from hemelb_amd import workloads as WL
from hemelb_amd.geometry import Domain
from tests import cases as K

pytestmark = pytest.mark.gpu

# 11 x 11 x 19 and 9 x 9 x 13 sites: blocks cut on every side, partly filled
# planes, more than one block per axis
CASES = [("d3q19-bfl-ladd", lambda: K.cylinder_case(5.0, 19, 19, "LBGK", "BFL", "womersley",
                                                    tau=0.7)),
         ("d3q15-sbb-nash", lambda: K.cylinder_case(4.0, 13, 15, "MRT", "SBB", "cosine"))]
FORMS = [("blocks", "fp64", 0), ("blocks", "fp64", 1), ("blocks", "fp32", 0),
         ("blocks", "fp16", 0), ("blocks", "fp16", 1), ("pull_table", "fp64", 0),
         ("pull_table", "fp16", 0), ("compact_blocks", "fp64", 0), ("compact_blocks", "fp32", 0)]


@pytest.mark.parametrize("layout,storage,wide", FORMS)
@pytest.mark.parametrize("label,make", CASES, ids=[c[0] for c in CASES])
@pytest.mark.parametrize("steps", [0, 1, 8])
def test_exports_match_the_oracle(label, make, layout, storage, wide, steps):
    case = make()
    print(f"[exports] {label} {layout} {storage} wide={wide} steps={steps}", flush=True)
    gpu, orc = case.product(storage=storage, layout=layout), case.oracle()
    if wide:
        gpu.set_launch_shape(threads=128, wide=1)
    orc.set_equilibrium(1.0)
    gpu.SetInitialConditions(1.0)
    gpu.snapshot_velocity()
    _, u0 = gpu.macroscopic()
    gpu.step(steps)
    orc.step(steps)
    f = gpu.get_distributions()
    if storage == "fp64":
        np.testing.assert_array_equal(f, orc.get_f())
    orc.set_f(f)
    rho, u = gpu.macroscopic()
    want_rho, want_u = orc.macro()
    np.testing.assert_array_equal(rho, want_rho)
    np.testing.assert_array_equal(u, want_u)
    normal = case.domain.normal
    np.testing.assert_array_equal(gpu.wall_shear_stress(), orc.wall_shear_stress(normal))
    want, got = orc.stress(normal), gpu.stress()
    for name in want:
        np.testing.assert_array_equal(got[name], want[name], err_msg=name)
    # sums of at most 2500 positive values in two orders: 2500 ulp at most
    m = gpu.monitor()
    np.testing.assert_allclose(m["mass"], rho.sum(), rtol=2500 * 2.3e-16)
    assert (m["density_min"], m["density_max"]) == (rho.min(), rho.max()) and m["stable"]
    speed = lambda v: np.sqrt(((0.0 + v[:, 0] ** 2) + v[:, 1] ** 2) + v[:, 2] ** 2)  # noqa: E731
    assert m["velocity_max"] == speed(u).max()
    assert gpu.velocity_change(0.03) == (speed(u - u0) * (1.0 / 0.03)).max()
    one, = gpu.monitor_instances()
    assert one["sites"] == case.domain.n and one["velocity_max"] == m["velocity_max"]
    assert gpu.velocity_change_instances(0.03)[0] == gpu.velocity_change(0.03)


def test_instances_keep_their_own_tau_and_chunks():
    e = WL.stenosed_ensemble(3, seed=5, radius_range=(3.0, 9.0), period=200.0)
    ens = e.solver("fp32")
    ens.snapshot_velocity()
    ens.step(9)
    stress, wss = ens.stress(), ens.wall_shear_stress()
    mons, change = ens.monitor_instances(), ens.velocity_change_instances(0.02)
    for k, inst in enumerate(e.instances):
        print(f"[exports] instance {k} tau {inst.tau:.3f}", flush=True)
        one = L.LBM(e.traits, e.instance_domain(k), L.LbmParameters(tau=inst.tau),
                    e.inlets[inst.inlets], e.outlets[inst.outlets], storage="fp32", rho0=1.0)
        one.SetInitialConditions(1.0)
        one.snapshot_velocity()
        one.step(9)
        alone = one.stress()
        for name in alone:
            np.testing.assert_array_equal(stress[name][inst.sites], alone[name], err_msg=name)
        np.testing.assert_array_equal(wss[inst.sites], one.wall_shear_stress())
        m = one.monitor()
        assert (mons[k]["density_min"], mons[k]["density_max"], mons[k]["velocity_max"]) == (
            m["density_min"], m["density_max"], m["velocity_max"])
        np.testing.assert_allclose(mons[k]["mass"], m["mass"], rtol=1e-12)
        assert change[k] == one.velocity_change(0.02)


# 152 bytes a site: below and just above the 4 MiB from which copies go
# through the staging chunks, and past the 16 chunks of its ring, none a
# multiple of the 1 MiB chunk
@pytest.mark.parametrize("radius,length", [(10.0, 80), (10.0, 91), (20.0, 121)])
def test_large_exports_return_what_was_set(radius, length):
    from concurrent.futures import ThreadPoolExecutor

    case = K.cylinder_case(radius, length, 19, "LBGK", "SBB", "cosine")
    n = case.domain.n
    print(f"[exports] {n} sites, {n * 152 / 2 ** 20:.2f} MiB of distributions", flush=True)

    def one(seed):
        f = np.random.default_rng(seed).uniform(0.01, 0.1, (n, 19))
        lbm = case.product()
        lbm.set_distributions(f)
        for _ in range(3):
            np.testing.assert_array_equal(lbm.get_distributions(), f)
        rho, _ = lbm.macroscopic()
        np.testing.assert_allclose(rho, f.sum(1), rtol=19 * 2.3e-16)

    one(0)
    with ThreadPoolExecutor(3) as pool:   # concurrent copies: one stages, the others do not
        list(pool.map(one, (1, 2, 3)))


def slab(side, depth, rng):
    """side x side x depth sites between walls."""
    shape = np.array([side, side, depth])
    coords = np.indices(shape).reshape(3, -1).T.astype(np.int32)
    n = len(coords)
    mask = np.zeros(n, np.uint32)
    for d in range(1, 19):
        to = coords + L.LATTICES[19].VECTORS[d]
        inside = ((to >= 0) & (to < shape)).all(1)
        mask |= np.where(inside, 0, 1 << (d - 1)).astype(np.uint32)
    normal = rng.standard_normal((n, 3)).astype(np.float32)
    normal /= np.linalg.norm(normal, axis=1, keepdims=True)
    return K.Case(Domain(19, np.ascontiguousarray(coords), np.ones(n, np.uint32), mask,
                         np.zeros(n, np.uint32), np.full(n, -1, np.int32),
                         np.full((n, 18), 0.5, np.float32), normal, [], []))


# the outputs of the wall sites alone, which come by boundary record, also where
# the two tractions are more than 2^20 values and do not go through pinned memory
# (191 k of 990 k sites at a wall); or as whole fields, where most sites are at a
# wall or the arrays are large (traction, then the wall shear stress as well)
@pytest.mark.parametrize("side,depth,storage,layout", [
    (40, 1, "fp64", "blocks"), (300, 11, "fp64", "blocks"), (300, 11, "fp32", "compact_blocks"),
    (1025, 1, "fp64", "blocks"), (300, 14, "fp32", "blocks"), (300, 41, "fp16", "pull_table")])
def test_wall_outputs(side, depth, storage, layout):
    rng = np.random.default_rng(side + depth)
    case = slab(side, depth, rng)
    n, normal, wall = case.domain.n, case.domain.normal, case.domain.wall_mask != 0
    print(f"[exports] {n} sites, {wall.sum()} at a wall, {storage} {layout}", flush=True)
    gpu = case.product(storage=storage, layout=layout)
    gpu.set_distributions(rng.random((n, 19), np.float32).astype(np.float64) * 0.1 + 0.01)
    f = gpu.get_distributions()
    wss, stress = gpu.wall_shear_stress(), gpu.stress()
    traction, tangential = np.full((n, 3), np.nan), np.full((n, 3), np.nan)
    ptr = lambda a: a.ctypes.data_as(C.c_void_p)  # noqa: E731
    N.check(N.lib().hlb_get_stress(gpu._h, None, None, None, ptr(traction), ptr(tangential)))
    np.testing.assert_array_equal(traction, stress["traction"])
    np.testing.assert_array_equal(tangential, stress["tangential_traction"])
    assert (wss[~wall] == np.finfo(np.float64).max).all()
    assert not traction[~wall].any() and not tangential[~wall].any()
    # they are of a site's own values: a small sheet with the same rows
    rows = np.sort(rng.choice(np.flatnonzero(wall), 1600, replace=False))
    small = slab(40, 1, rng)
    small.domain.normal = np.ascontiguousarray(normal[rows])
    orc = small.oracle()
    orc.set_f(f[rows])
    np.testing.assert_array_equal(wss[rows], orc.wall_shear_stress(small.domain.normal))
    want = orc.stress(small.domain.normal)
    for name in ("traction", "tangential_traction"):
        np.testing.assert_array_equal(stress[name][rows], want[name])
