"""Slots appended behind the sorted ones by calls that keep the run table (pairs
from converting photons, injection): the sorted slots go by tile and the others
from their own slots, in one push, as a context does that is given the same
slots and never sorts.  Bit for bit: FP64 by construction, the mixed sums are of
integers."""
import numpy as np
import pytest

import aperture3_amd as apt
from cases import Case
from logsph_cases import LogSphCase

pytestmark = pytest.mark.gpu

KEYS = ("cell", "x1", "x2", "x3", "p1", "p2", "p3", "w", "flag")


@pytest.mark.parametrize("N,periodic,precision", [
    ((60,), (True,), apt.APT_PREC_FP64), ((20, 17), (False, True), apt.APT_PREC_FP64),
    ((10, 9, 8), (True, True, True), apt.APT_PREC_FP64),
    ((60,), (True,), apt.APT_PREC_MIXED), ((20, 17), (False, False), apt.APT_PREC_MIXED),
    ((10, 9, 8), (True, False, True), apt.APT_PREC_MIXED)])
def test_pairs_behind_sorted_slots(N, periodic, precision):
    c = Case(N, 4, theta=(0.1, 0.1), drift=(0.2, -0.2), Bbg=(0.3, 0.0, 1.0), data_interval=1)
    state = c.oracle().particles()
    n = 333  # photons, each a pair
    rng = np.random.default_rng(2)
    at = [rng.integers(0, c.N[q], n) + c.guard[q] for q in range(3)]
    ph = {"cell": (at[0] + c.dims[0] * (at[1] + c.dims[1] * at[2])).astype(np.uint32),
          "x1": rng.random(n), "x2": rng.random(n), "x3": rng.random(n), "w": np.ones(n),
          "p1": rng.normal(0, 20, n), "p2": np.full(n, 5.0), "p3": rng.normal(0, 20, n),
          "path": np.zeros(n), "flag": np.zeros(n, np.uint32)}
    ph["E"] = np.sqrt(ph["p1"] ** 2 + ph["p2"] ** 2 + ph["p3"] ** 2)
    sims = []
    for _ in range(2):
        env = apt.sim_environment(apt.SimParams(
            N=c.N, guard=c.guard, periodic_boundary=list(periodic) + [True] * (3 - len(N)),
            max_ptc_number=c.nptc + 2 * n + 64, max_photon_number=n + 64, precision=precision,
            data_interval=1))
        d = apt.sim_data(env)
        E, B = c.fields()
        for q in range(3):
            d.set_field(apt.FIELD_E, q, E[q])
            d.set_field(apt.FIELD_B, q, B[q])
        sims.append((env, d))
    (env, a), (_, b) = sims
    a.set_particles(state)
    a.sort_particles()
    a.set_photons(ph)
    assert apt.radiative_transfer(env).produce_pairs(a) == n
    assert a.num_particles() == c.nptc + 2 * n
    b.set_particles(a.get_particles())
    pu = apt.ptc_updater(env)
    for step in range(3):
        for d in (a, b):
            pu.update_particles(d, c.dt, step)
        for which in (apt.FIELD_J, apt.FIELD_RHO):
            for q in range(2):
                assert np.array_equal(a.get_field(which, q), b.get_field(which, q)), (step, q)
    pa, pb = a.get_particles(), b.get_particles()
    live = pb["cell"] != apt.MAX_CELL
    assert np.array_equal(pa["cell"], pb["cell"]) and live[c.nptc:].sum() > n
    for k in KEYS:
        assert np.array_equal(pa[k][live], pb[k][live]), k


@pytest.mark.parametrize("inj", [40, 17500])
@pytest.mark.parametrize("precision", [apt.APT_PREC_FP64, apt.APT_PREC_MIXED])
def test_device_counts_with_injected_slots(precision, inj):
    """17500 pairs a row: more slots behind the sorted ones than one a thread of
    the workgroups that a device count's bound gets (4096 of 512 threads)."""
    c = LogSphCase(N=(64, 64), nptc=5000, damping_length=6, cap=5000 + 62 * 2 * inj + 2000)
    out = []
    for device in (False, True):
        env, d = c.gpu(precision=precision)
        if device:
            d.device_counts()
        pu = apt.ptc_updater_logsph(env)
        d.sort_particles()
        pu.inject_ptc(d, inj, 0.05, 0.02, 0.0, 1e-3, 0.1)
        for step in range(2, 4):
            pu.update_particles(d, c.dt, step)
        out.append([d.get_field(apt.FIELD_J, k) for k in range(3)] +
                   [d.get_field(apt.FIELD_RHO, s) for s in range(3)] +
                   [d.get_particles()["x1"], np.array(d.num_particles())])
        d.close()
    assert out[0][-1] == 5000 + 62 * 2 * inj
    for k, (x, y) in enumerate(zip(*out)):
        assert np.array_equal(x, y, equal_nan=True), k
