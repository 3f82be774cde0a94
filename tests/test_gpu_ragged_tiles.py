"""GPU tests of the tiled mixed form on meshes whose sides are no multiples of
the tile extent (each axis split evenly over its tiles), on meshes smaller
than a tile or than its window, and with a tile's slots shared by several
workgroups; and of the charge of the tiled 3D push."""
import numpy as np
import pytest

import aperture3_amd as apt
from cases import Case
from test_gpu_mixed_tiled import by_tag, tagged

pytestmark = pytest.mark.gpu


def even_split(N, T):
    """Tile of every bulk coordinate: ceil(N / T) tiles, the first N % nt of
    them one cell longer."""
    nt = -(-N // T)
    w, r = divmod(N, nt)
    return np.repeat(np.arange(nt), [w + (t < r) for t in range(nt)]), nt


def check_binning(env, d, dim):
    off, T = d.tile_offsets()
    assert off is not None
    p = d.get_particles()
    assert off[-1] == d.num_particles()
    N, g, dims = env.params().N, env.params().guard, env.dims
    c = p["cell"].astype(np.int64)
    idx = [c % dims[0], c // dims[0] % dims[1], c // (dims[0] * dims[1])]
    t, mul = 0, 1
    for k in range(dim):
        lut, nt = even_split(N[k], T[k])
        t = t + mul * lut[idx[k] - g[k]]
        mul *= nt
    assert mul == len(off) - 1
    assert np.array_equal(t, np.repeat(np.arange(mul), np.diff(off.astype(np.int64))))


@pytest.mark.parametrize("N,ppc,tile,halo,threads", [
    ((50, 37), 4, (0, 0), 0, 0), ((100, 17), 3, (16, 16), 6, 256), ((65, 9), 6, (0, 0), 0, 0),
    ((8, 8), 40, (0, 0), 0, 0), ((33, 33), 4, (16, 8), 8, 512), ((31, 20), 4, (32, 16), 8, 512),
    ((23, 17, 10), 2, (0, 0, 0), 0, 0), ((31, 9, 8), 2, (8, 8, 8), 5, 1024),
    ((15, 8, 7), 6, (8, 8, 8), 4, 512)])
def test_ragged_step_vs_oracle(N, ppc, tile, halo, threads):
    """The bounds of test_tiled_step_vs_oracle for the particles: same cells
    but for rare FP32 ties, offsets to 1e-4, momenta to 1e-5.  Fields: each of
    16 steps adds dt/dx <= 1/2 times four values of a B of order 1 that FP32
    holds to 2^-25, 16 * 0.5 * 4 * 2^-25 = 1e-6 in all, and rounds the sum of
    the current's terms, 2e-5 of a field's scale.  The charge of the last step
    (node weights of positions known to 1e-4) to 1e-4 of its scale."""
    c = Case(N, ppc, theta=(0.1, 0.1), drift=(0.2, -0.2), Bbg=(0, 0, 1.0), data_interval=16)
    o = c.oracle()
    po0 = tagged(o.particles())
    o.set_particles(po0)
    p = apt.SimParams(N=c.N, guard=c.guard, periodic_boundary=[True] * 3,
                      max_ptc_number=c.nptc + 64, precision=apt.APT_PREC_MIXED,
                      tile=list(tile) + [0] * (3 - len(tile)), tile_halo=halo,
                      tile_threads=threads, data_interval=16)
    env = apt.sim_environment(p)
    d = apt.sim_data(env)
    E, B = c.fields()
    for comp in range(3):
        d.set_field(apt.FIELD_E, comp, E[comp])
        d.set_field(apt.FIELD_B, comp, B[comp])
        d.set_field(apt.FIELD_BBG, comp, B[comp])
    d.set_particles(po0)
    d.sort_particles()  # radix sort by tile
    check_binning(env, d, len(N))
    pu, fs = apt.ptc_updater(env), apt.field_solver(env)
    for step in range(16):
        o.ptc_update(c.dt, step)
        o.field_update(c.dt, step)
        pu.update_particles(d, c.dt, step)
        fs.update_fields(d, c.dt, step)
        if step in (5, 11):
            o.sort()
            d.sort_particles()  # tile-binning sort
            check_binning(env, d, len(N))
    pg, tg = by_tag(d.get_particles())
    ps, ts = by_tag(o.particles())
    assert np.array_equal(tg, ts)
    same = pg["cell"] == ps["cell"]
    assert np.mean(same) > 0.999
    for k in ("x1", "x2", "x3")[:max(2, len(N))]:
        assert np.abs(pg[k][same] - ps[k][same]).max() < 1e-4, k
    for k in ("p1", "p2", "p3"):
        assert np.abs(pg[k] - ps[k]).max() <= 1e-5 * np.abs(ps[k]).max(), k
    for comp in range(3):
        for which, key in ((apt.FIELD_E, "E"), (apt.FIELD_B, "B")):
            x, y = d.get_field(which, comp), o.f[key][comp]
            assert np.abs(x - y).max() <= 2e-5 * np.abs(y).max() + 1e-6, (key, comp)
    for s in range(2):
        x, y = d.get_field(apt.FIELD_RHO, s), o.rho[s]
        assert np.abs(y).max() > 0
        assert np.abs(x - y).max() <= 1e-4 * np.abs(y).max(), s
    assert d.counters()["nan_momenta"] == 0


def test_tiled_push_counts_nan_momenta():
    for N in ((32, 32), (16, 16, 16)):
        c = Case(N, 1, theta=(0.1, 0.1), Bbg=(0, 0, 1.0))
        ptc = c.oracle().particles()
        ptc["p2"][[3, 40]] = np.nan
        env, d = c.gpu(precision=apt.APT_PREC_MIXED, load=False)
        d.set_particles(ptc)
        d.sort_particles()
        apt.ptc_updater(env).update_particles(d, c.dt, 0)
        assert d.tile_offsets()[0] is not None
        assert d.counters()["nan_momenta"] == 2
