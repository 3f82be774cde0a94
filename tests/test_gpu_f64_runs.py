"""GPU tests of the FP64 update over runs of cell-sorted slots (LDS windows by
tile): bit-exact against the oracle on meshes that are no multiples of the
tile, smaller than a tile or than its window, open and periodic, with charge
output, a load after the sort, particles in guard cells, and fields
that are not finite."""
import ctypes as C

import numpy as np
import pytest

import aperture3_amd as apt
import oracle_ctypes as oc
from cases import Case
from test_gpu_parity_cart import PTC_KEYS, assert_same_particles, run_both

pytestmark = pytest.mark.gpu


def _two(v):
    return (C.c_double * 2)(v, v)


def assert_same_fields(d, o, rho=True):
    for comp in range(3):
        for which, key in ((apt.FIELD_E, "E"), (apt.FIELD_B, "B"), (apt.FIELD_J, "J")):
            assert np.array_equal(d.get_field(which, comp), o.f[key][comp], equal_nan=True), \
                (key, comp)
    for s in range(2 if rho else 0):
        assert np.array_equal(d.get_field(apt.FIELD_RHO, s), o.rho[s], equal_nan=True), s


@pytest.mark.parametrize("N,ppc", [
    ((300,), 30), ((5,), 50), ((1000,), 1), ((37, 29), 6), ((12, 5), 20), ((100, 16), 2),
    ((23, 9, 14), 3), ((6, 5, 4), 6), ((9, 9, 33), 1)])
def test_runs_bit_exact(N, ppc):
    """12 steps with sorts before the first and the 9th step and Rho on every
    4th: particles, E, B, J and Rho equal to the oracle's bits."""
    c = Case(sorted(N, reverse=True) if len(N) > 1 else N, ppc, theta=(0.1, 0.1),
             drift=(0.2, -0.2), Bbg=(0.3, 0.0, 1.0), data_interval=4)
    o = c.oracle()
    env, d = c.gpu(precision=apt.APT_PREC_FP64, load=False)
    d.set_particles(o.particles())
    o.sort()
    d.sort_particles()
    run_both(c, o, env, d, 12, sort_every=8)
    assert_same_particles(d.get_particles(), o.particles())
    assert_same_fields(d, o)


@pytest.mark.parametrize("N,periodic", [((64,), (False,)), ((40, 24), (False, True)),
                                        ((20, 20), (False, False)), ((10, 9, 8), (True, False, True))])
def test_runs_on_open_axes(N, periodic):
    """Open axes: particles that leave the bulk are erased by the next push;
    nothing is folded across an open edge."""
    dim = len(N)
    c = Case(N, 4, theta=(0.1, 0.1), drift=(0.3, -0.3), Bbg=(0.3, 0.0, 1.0), data_interval=3)
    per = list(periodic) + [True] * (3 - dim)
    o = oc.OracleSim(list(N), [2] * dim, size=c.size, periodic=tuple(per), q_e=1.0,
                     capacity=c.nptc, data_interval=3)
    p = apt.SimParams(N=c.N, guard=c.guard, periodic_boundary=per, max_ptc_number=c.nptc + 64,
                      precision=apt.APT_PREC_FP64, data_interval=3)
    env = apt.sim_environment(p)
    d = apt.sim_data(env)
    E, B = c.fields()
    for comp in range(3):
        o.f["E"][comp][:] = E[comp]
        o.f["B"][comp][:] = B[comp]
        o.f["Bbg"][comp][:] = B[comp]
        d.set_field(apt.FIELD_E, comp, E[comp])
        d.set_field(apt.FIELD_B, comp, B[comp])
        d.set_field(apt.FIELD_BBG, comp, B[comp])
    o.load_uniform(4, (0.1, 0.1), (0.3, -0.3), 1.0, 43210)
    d.set_particles(o.particles())
    o.sort()
    d.sort_particles()
    run_both(c, o, env, d, 9, sort_every=4)
    pg, po = d.get_particles(), o.particles()
    live = po["cell"] != apt.MAX_CELL
    assert np.array_equal(pg["cell"], po["cell"])
    for k in PTC_KEYS:
        assert np.array_equal(pg[k][live], po[k][live]), k
    assert_same_fields(d, o)


@pytest.mark.parametrize("N,value", [((64,), np.nan), ((24, 20), np.inf), ((10, 9, 8), -np.inf)])
def test_runs_with_fields_that_are_not_finite(N, value):
    """A field value that is not finite reaches every particle whose stencil of
    three taps per axis holds it, also with weight zero."""
    c = Case(N, 4, theta=(0.1, 0.1), Bbg=(0.3, 0.0, 1.0))
    o = c.oracle()
    env, d = c.gpu(precision=apt.APT_PREC_FP64, load=False)
    mid = sum((c.dims[k] // 2) * int(np.prod(c.dims[:k])) for k in range(3))
    for comp, at in ((0, mid), (2, mid + 3)):
        o.f["E"][comp][at] = value
        d.set_field(apt.FIELD_E, comp, o.f["E"][comp])
    d.set_particles(o.particles())
    o.sort()
    d.sort_particles()
    o.ptc_update(c.dt, 0)
    apt.ptc_updater(env).update_particles(d, c.dt, 0)
    pg, po = d.get_particles(), o.particles()
    bad = np.isnan(po["p1"]) | np.isnan(po["p2"]) | np.isnan(po["p3"])
    assert 0 < bad.sum() < len(bad)
    for k in ("p1", "p2", "p3", "E"):
        assert np.array_equal(pg[k], po[k], equal_nan=True), k
    for k in ("cell", "x1", "x2", "x3"):  # a NaN move has no defined cell
        assert np.array_equal(pg[k][~bad], po[k][~bad]), k


def test_runs_with_guard_cells_and_an_unsorted_tail():
    """Particles in guard cells are sorted with the others and erased by the
    next push; a second load after a sort leaves every slot to the update of
    consecutive slots (slots behind sorted ones: test_gpu_run_tails)."""
    for N in ((20,), (18, 10), (8, 7, 6)):
        c = Case(N, 2, theta=(0.1, 0.1), drift=(0.2, -0.2), Bbg=(0.3, 0.0, 1.0))
        o = c.oracle()
        po = o.particles()
        guard = np.arange(0, c.nptc, 7)
        po["cell"][guard[::2]] = 1                # the first row's guard cell
        po["cell"][guard[1::2]] = c.ncell - 1     # the last cell of all
        o.set_particles(po)
        env, d = c.gpu(precision=apt.APT_PREC_FP64, load=False, capacity=2 * c.nptc + 64)
        d.set_particles(po)
        o.sort()
        d.sort_particles()
        run_both(c, o, env, d, 2)
        pg, ps = d.get_particles(), o.particles()
        assert np.array_equal(pg["cell"], ps["cell"])
        assert (ps["cell"] == apt.MAX_CELL).sum() == len(guard)
        assert_same_fields(d, o, rho=False)
        # a second load: no slot is taken by tile any more
        before = d.get_particles()
        live = before["cell"] != apt.MAX_CELL
        d.sort_particles()
        d.lib.apt_ptc_load_uniform(d.ctx, 1, _two(0.1), _two(0.0), 1.0)
        both = d.get_particles()
        assert len(both["cell"]) >= live.sum() + 2 * c.nptc // 4
        o2 = c.oracle(load=False)
        o2.set_particles(both)
        for comp in range(3):
            for which, key in ((apt.FIELD_E, "E"), (apt.FIELD_B, "B")):
                o2.f[key][comp][:] = d.get_field(which, comp)
        o2.ptc_update(c.dt, 2)
        apt.ptc_updater(env).update_particles(d, c.dt, 2)
        pg, ps = d.get_particles(), o2.particles()
        on = ps["cell"] != apt.MAX_CELL
        for k in PTC_KEYS:
            assert np.array_equal(pg[k][on], ps[k][on]), k
        assert_same_fields(d, o2, rho=False)
