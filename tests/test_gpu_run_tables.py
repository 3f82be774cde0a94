"""The tables of the updates over runs of sorted slots on meshes of many tiles:
more than one workgroup of work items, tiles that hold most of the particles and
are shared, tiles that are empty, plasma too thin for them.  FP64 against the oracle bit for bit; mixed
against a context that is given the sorted particles and never sorts."""
import numpy as np
import pytest

import aperture3_amd as apt
from cases import Case
from logsph_cases import LogSphCase
from test_gpu_f64_runs import assert_same_fields
from test_gpu_parity_cart import assert_same_particles, run_both

pytestmark = pytest.mark.gpu

# 1D: 563 tiles of 16 cells; 2D: 325; 3D: 8 x 4 x 4 FP64, 8^3 mixed: 780, 120.
# 40,000 cells, 18,000 particles: thin on 2500 tiles, so not taken by tile
MESHES = [(9000,), (200, 390), (43, 41, 50), (40000,)]


def clustered(c, n, seed=3):
    """n particles: two thirds in a few cells, the others anywhere."""
    rng = np.random.default_rng(seed)
    p = {k: v[:n].copy() for k, v in c.oracle().particles().items()}
    at = [rng.integers(0, c.N[q], n) for q in range(3)]
    near = np.arange(n) % 3 > 0
    for q in range(3):
        at[q][near] = np.minimum(c.N[q] - 1, c.N[q] // 2 + at[q][near] % 3)
    g, d = c.guard, c.dims
    p["cell"] = ((at[0] + g[0]) + d[0] * ((at[1] + g[1]) + d[1] * (at[2] + g[2]))).astype(np.uint32)
    return p


@pytest.mark.parametrize("n", [300, 18000])
@pytest.mark.parametrize("N", MESHES)
def test_fp64_bit_exact(N, n):
    c = Case(N, 1, theta=(0.1, 0.1), drift=(0.2, -0.2), Bbg=(0.3, 0.0, 1.0), data_interval=4)
    p = clustered(c, n)
    o = c.oracle(load=False)
    o.set_particles(p)
    env, d = c.gpu(precision=apt.APT_PREC_FP64, load=False)
    d.set_particles(p)
    o.sort()
    d.sort_particles()
    run_both(c, o, env, d, 6, sort_every=3)
    assert_same_particles(d.get_particles(), o.particles())
    assert_same_fields(d, o)


@pytest.mark.parametrize("n", [300, 18000])
@pytest.mark.parametrize("N", MESHES)
def test_mixed_equals_unsorted_slots(N, n):
    c = Case(N, 1, theta=(0.2, 0.2), drift=(0.3, -0.3), Bbg=(0.3, 0.0, 1.0), data_interval=3)
    sims = []
    for _ in range(2):
        env = apt.sim_environment(apt.SimParams(
            N=c.N, guard=c.guard, periodic_boundary=[False] * 3, max_ptc_number=n + 64,
            precision=apt.APT_PREC_MIXED, data_interval=3))
        sims.append((env, apt.sim_data(env)))
    (env, a), (_, b) = sims
    a.set_particles(clustered(c, n))
    a.sort_particles()
    b.set_particles(a.get_particles())
    pu = apt.ptc_updater(env)
    for step in range(3):
        for d in (a, b):
            pu.update_particles(d, c.dt, step)
        for which in (apt.FIELD_J, apt.FIELD_RHO):
            for comp in range(2):
                assert np.array_equal(a.get_field(which, comp), b.get_field(which, comp)), step


@pytest.mark.parametrize("precision", [apt.APT_PREC_FP64, apt.APT_PREC_MIXED])
def test_log_spherical_mesh_with_guard_planes(precision):
    """Guard cells along the axis that a 2D mesh does not have: the step lives in
    the first plane, sorted or not."""
    c = LogSphCase(N=(40, 33), nptc=4000, damping_length=6, data_interval=1)
    out = []
    for planes in (0, 1):
        env = apt.sim_environment(apt.SimParams(
            N=[40, 33, 1], guard=c.guard[:2] + [planes], size=c.size, num_species=3,
            max_ptc_number=c.cap, precision=precision, data_interval=1,
            coord_system="LogSpherical", omega=0.1, B0=c.mu, damping_length=6))
        d = apt.sim_data(env)
        n = c.ncell
        for q, f in enumerate(c.dipole()):
            full = np.zeros(env.ncell())
            full[:n] = f
            d.set_field(apt.FIELD_BBG, q, full)
            d.set_field(apt.FIELD_B, q, full)
        d.set_particles(c.particles())
        d.sort_particles()
        pu = apt.ptc_updater_logsph(env)
        for step in range(2):
            pu.update_particles(d, c.dt, step)
        out.append([d.get_field(apt.FIELD_J, q)[:n] for q in range(3)] +
                   [d.get_particles()["x1"]])
    assert np.abs(out[0][0]).max() > 0
    for a, b in zip(*out):
        assert np.array_equal(a, b, equal_nan=True)


@pytest.mark.parametrize("precision", [apt.APT_PREC_FP64, apt.APT_PREC_MIXED])
@pytest.mark.parametrize("N,guard", [((50,), [2, 2, 0]), ((50,), [2, 0, 1]), ((21, 18), [2, 2, 1])])
def test_cartesian_mesh_with_idle_guards(N, guard, precision):
    """Guard cells along axes that the mesh does not have: a sort changes nothing
    but the order of the slots."""
    c = Case(N, 5, theta=(0.1, 0.1), drift=(0.2, -0.2), Bbg=(0.3, 0.0, 1.0), data_interval=1)
    dims = [c.N[q] + 2 * guard[q] for q in range(3)]
    p = c.oracle().particles()
    at = [p["cell"] % c.dims[0], p["cell"] // c.dims[0], np.full(c.nptc, guard[2])]
    if len(N) == 1:
        at[1] = at[1] + guard[1]
    p["cell"] = (at[0] + dims[0] * (at[1] + dims[1] * at[2])).astype(np.uint32)
    out = []
    for sort in (False, True):
        env = apt.sim_environment(apt.SimParams(
            N=c.N, guard=guard, periodic_boundary=[True] * 3, max_ptc_number=c.nptc,
            precision=precision, data_interval=1))
        d = apt.sim_data(env)
        rng = np.random.default_rng(4)
        for which in (apt.FIELD_E, apt.FIELD_B):
            for q in range(3):
                d.set_field(which, q, rng.normal(size=env.ncell()))
        d.set_particles(p)
        if sort:
            d.sort_particles()
        pu = apt.ptc_updater(env)
        for step in range(2):
            pu.update_particles(d, 0.3 * c.dt, step)
        out.append([d.get_field(apt.FIELD_J, q) for q in range(3)] +
                   [np.sort(d.get_particles()["x1"])])
    for a, b in zip(*out):
        assert np.array_equal(a, b, equal_nan=True)
