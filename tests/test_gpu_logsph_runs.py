"""The log-spherical update over tiles of cell-sorted slots: ragged tiles,
sorted slots with appended ones behind them, a corner of the mesh so dense that
its tile is shared by several workgroups, charge steps, and more rows than a
workgroup of the surface density keeps sums for."""
import numpy as np
import pytest

import aperture3_amd as apt
from logsph_cases import LogSphCase
from test_gpu_logsph import FIELDS, PTC_KEYS, run_steps

pytestmark = pytest.mark.gpu


class Dense(LogSphCase):
    """Half of the particles in 3 x 3 cells next to the star."""

    def particles(self):
        p = super().particles()
        n, (g0, g1, _) = self.nptc // 2, self.guard
        rng = np.random.default_rng(self.seed + 7)
        c1 = rng.integers(g0 + 2, g0 + 5, n)
        c2 = rng.integers(g1 + 20, g1 + 23, n)
        p["cell"][:n] = (c1 + c2 * self.dims[0]).astype(np.uint32)
        return p


CASES = [(LogSphCase, (64, 64), 20000), (LogSphCase, (35, 50), 3000), (Dense, (48, 33), 30000),
         (LogSphCase, (24, 301), 5000), (LogSphCase, (17, 16), 40)]


@pytest.mark.parametrize("kind,N,nptc", CASES)
def test_fp64_sorted_bit_exact(kind, N, nptc):
    c = kind(N=N, nptc=nptc, damping_length=6)
    o = c.oracle()
    env, d = c.gpu(precision=apt.APT_PREC_FP64)
    run_steps(c, o, env, d, 8, sort_every=2)
    pg, po = d.get_particles(), o.particles()
    for k in PTC_KEYS:
        assert np.array_equal(pg[k], po[k]), k
    for which, key in FIELDS:
        for comp in range(3):
            assert np.array_equal(d.get_field(which, comp), o.f[key][comp]), (key, comp)
    for s in range(3):
        assert np.array_equal(d.get_field(apt.FIELD_RHO, s), o.rho[s]), ("rho", s)
    d.close()


@pytest.mark.parametrize("kind,N,nptc", CASES)
def test_mixed_sorted_equals_unsorted(kind, N, nptc):
    """The current is an integer sum of the same contributions in any slot
    order, so a sort changes no field: no tolerance."""
    c = kind(N=N, nptc=nptc, damping_length=6)
    out = []
    for sort in (False, True):
        env, d = c.gpu(precision=apt.APT_PREC_MIXED)
        pu, fs = apt.ptc_updater_logsph(env), apt.field_solver_logsph(env)
        for step in range(6):
            if sort and step in (0, 2, 3):
                d.sort_particles()
            pu.update_particles(d, c.dt, step)
            fs.update_fields(d, c.dt, step * c.dt)
            fs.apply_boundary(d, 0.1, step * c.dt)
        out.append([d.get_field(w, k) for w, _ in FIELDS for k in range(3)] +
                   [d.get_field(apt.FIELD_RHO, s) for s in range(3)])
        d.close()
    for k, (a, b) in enumerate(zip(*out)):
        assert np.array_equal(a, b, equal_nan=True), k


def test_device_counts_more_slots_than_the_grid():
    """Slots never sorted, 512 to a cell, two a thread: the same integer sums
    under a device count as with host counts (behind sorted slots, where a device
    count caps the workgroups: test_gpu_run_tails)."""
    c = LogSphCase(N=(64, 64), nptc=4096 * 512 + 70001, damping_length=6)
    out = []
    for device in (False, True):
        env, d = c.gpu(precision=apt.APT_PREC_MIXED)
        if device:
            d.device_counts()
        pu = apt.ptc_updater_logsph(env)
        for step in range(3):
            pu.update_particles(d, c.dt, step)
        out.append([d.get_field(apt.FIELD_J, k) for k in range(3)] +
                   [d.get_field(apt.FIELD_RHO, s) for s in range(3)])
        d.close()
    for k, (a, b) in enumerate(zip(*out)):
        assert np.array_equal(a, b, equal_nan=True), k
