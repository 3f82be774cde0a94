"""The tiled 3D push where the library chooses the shape: a small halo for the
first pushes after a sort and for thin plasma, a large one later.  Particles past
the halo take another kernel's rounding, so the two runs differ as either does
from the FP64 oracle in test_gpu_ragged_tiles: twice its bounds."""
import numpy as np
import pytest

import aperture3_amd as apt
from cases import Case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,n", [((57, 60, 64), 60000), ((64, 64, 64), 200000)])
def test_chosen_shape_equals_the_large_halo(N, n):
    c = Case(N, 1, theta=(0.3, 0.3), drift=(0.5, -0.5), Bbg=(0.3, 0.0, 1.0), data_interval=3)
    state = {k: v[:n] for k, v in c.oracle().particles().items()}
    out = []
    for shape in (dict(), dict(tile=[8, 8, 8], tile_halo=5, tile_threads=1024)):
        env = apt.sim_environment(apt.SimParams(
            N=c.N, guard=c.guard, periodic_boundary=[True] * 3, max_ptc_number=n + 64,
            precision=apt.APT_PREC_MIXED, data_interval=3, **shape))
        d = apt.sim_data(env)
        E, B = c.fields()
        for q in range(3):
            d.set_field(apt.FIELD_E, q, E[q])
            d.set_field(apt.FIELD_B, q, B[q])
        d.set_particles(state)
        d.sort_particles()
        pu, fs = apt.ptc_updater(env), apt.field_solver(env)
        got = []
        for step in range(12):
            pu.update_particles(d, c.dt, step)
            fs.update_fields(d, c.dt, step)
            if step == 8:
                d.sort_particles()
            if step % 3 == 2:
                got += [(2e-5, 1e-6, d.get_field(apt.FIELD_E, q)) for q in range(3)]
                got += [(1e-4, 0.0, d.get_field(apt.FIELD_J, q)) for q in range(3)]
                got += [(1e-4, 0.0, d.get_field(apt.FIELD_RHO, s)) for s in range(2)]
        out.append((got, d.counters()["outside_tile"]))
    for (rel, floor, a), (_, _, b) in zip(out[0][0], out[1][0]):
        assert np.abs(b).max() > 0
        assert np.abs(a - b).max() <= 2 * (rel * np.abs(b).max() + floor)
    assert out[0][1] > out[1][1]
