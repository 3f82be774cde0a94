"""A step recorded while the sorted slots go by tile, replayed on particles that
were set after the recording: every slot is judged by its own cell, whatever row
of the mesh the sort had put its former particle in."""
import numpy as np
import pytest

import aperture3_amd as apt
from cases import Case
from logsph_cases import LogSphCase

pytestmark = pytest.mark.gpu

KEYS = ("cell", "x1", "x2", "x3", "p1", "p2", "p3", "w", "flag")


def in_guards(ptc, ncell):
    """Every 7th particle in the first row's guard cells, every 11th in the
    last row's."""
    out = {k: v.copy() for k, v in ptc.items()}
    out["cell"][::7] = 1
    out["cell"][::11] = ncell - 1
    return out


def check(recorded, eager):
    pr, pe = recorded.get_particles(), eager.get_particles()
    live = pe["cell"] != apt.MAX_CELL
    assert live.sum() > 0.9 * len(live)
    assert np.array_equal(pr["cell"], pe["cell"])
    for k in KEYS:
        assert np.array_equal(pr[k][live], pe[k][live]), k
    for which in (apt.FIELD_J, apt.FIELD_RHO):
        for c in range(2):
            assert np.array_equal(recorded.get_field(which, c), eager.get_field(which, c),
                                  equal_nan=True), (which, c)


@pytest.mark.parametrize("precision", [apt.APT_PREC_FP64, apt.APT_PREC_MIXED])
@pytest.mark.parametrize("N,periodic", [((60,), (False,)), ((40, 24), (True, False)),
                                        ((20, 17), (False, False)),
                                        ((10, 9, 8), (True, False, False))])
def test_replay_on_particles_set_after_a_sort(N, periodic, precision):
    c = Case(N, 4, theta=(0.1, 0.1), drift=(0.2, -0.2), Bbg=(0.3, 0.0, 1.0), data_interval=1)
    per = list(periodic) + [True] * (3 - len(N))
    state = c.oracle().particles()
    out = []
    for graph in (True, False):
        env = apt.sim_environment(apt.SimParams(
            N=c.N, guard=c.guard, periodic_boundary=per, max_ptc_number=c.nptc + 64,
            precision=precision, data_interval=1))
        d = apt.sim_data(env)
        E, B = c.fields()
        for q in range(3):
            d.set_field(apt.FIELD_E, q, E[q])
            d.set_field(apt.FIELD_B, q, B[q])
        pu = apt.ptc_updater(env)
        if graph:
            d.set_particles(in_guards(state, c.ncell))
            d.sort_particles()
            d.graph_begin()
            pu.update_particles(d, c.dt, 0)
            d.graph_end()
        d.set_particles(state)
        for _ in range(3):
            if graph:
                d.graph_launch(1)
            else:
                pu.update_particles(d, c.dt, 0)
        out.append(d)
    check(*out)


@pytest.mark.parametrize("precision", [apt.APT_PREC_FP64, apt.APT_PREC_MIXED])
@pytest.mark.parametrize("device", [False, True])
def test_replay_of_a_log_spherical_step(precision, device):
    c = LogSphCase(N=(40, 33), nptc=6000, damping_length=6, data_interval=1)
    state = c.particles()
    out = []
    for graph in (True, False):
        env, d = c.gpu(precision=precision)
        if device:
            d.device_counts()
        pu = apt.ptc_updater_logsph(env)
        if graph:
            d.set_particles(in_guards(state, c.ncell))
            d.sort_particles()
            d.graph_begin()
            pu.update_particles(d, c.dt, 0)
            d.graph_end()
        d.set_particles(state)
        for _ in range(3):
            if graph:
                d.graph_launch(1)
            else:
                pu.update_particles(d, c.dt, 0)
        out.append(d)
    check(*out)


def test_recording_outlives_eager_pushes_on_a_ragged_3d_mesh():
    """More eager pushes than a re-layout interval between recording and replay:
    the recording is still there, and fields equal those of eager pushes alone."""
    c = Case((12, 11, 9), 3, theta=(0.1, 0.1), drift=(0.2, -0.2), Bbg=(0.3, 0.0, 1.0))
    state = c.oracle().particles()
    out = []
    for graph in (True, False):
        env, d = c.gpu(precision=apt.APT_PREC_MIXED, load=False)
        d.set_particles(state)
        d.sort_particles()
        pu, fs = apt.ptc_updater(env), apt.field_solver(env)

        def step():
            pu.update_particles(d, c.dt, 0)
            fs.update_fields(d, c.dt, 1)

        if graph:
            d.graph_begin()
            step()
            d.graph_end()
        for k in range(12):
            if graph and k >= 8:
                d.graph_launch(1)
            else:
                step()
        out.append([d.get_field(w, q) for w in (apt.FIELD_E, apt.FIELD_B, apt.FIELD_J)
                    for q in range(3)])
    for a, b in zip(*out):
        assert np.array_equal(a, b)
