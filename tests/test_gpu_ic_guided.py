"""GPU tests of the guided inverse-Compton sampling against the oracle's plain
binary searches: smallest grids, the largest with a guide and the first without,
rows of NaN (a mono-energetic spectrum), and draws enough to hit every bucket."""
import numpy as np
import pytest

from test_gpu_ic import pair, same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,ng,nep", [
    ("soft_pl", 3, 3), ("mono", 3, 3), ("soft_pl", 3, 2048), ("mono", 3, 2049),
    ("soft_pl", 40, 257), ("mono", 40, 257)])
def test_guided_samples_bit_exact(name, ng, nep):
    ic, o = pair(name, ng=ng, nep=nep)
    rng = np.random.default_rng(ng + nep)
    g = np.concatenate([np.exp(rng.uniform(np.log(0.5), np.log(1e16), 20000)),
                        ic.gammas(), [1.01, 2.0, 1e15, 2e15, 1.0, np.inf]])
    same(ic.gen_photon_e(g, seed=7, epoch=2), o.gen_photon_e(g, seed=7, epoch=2), "eph")


def test_few_samples_of_large_tables_equal_many():
    """Tables of 2048 x 2048 are sampled with the guide from 2^19 samples on; a
    sample depends on its index alone, so fewer of them are the same bits."""
    import aperture3_amd as apt
    ic = apt.inverse_compton(apt.SimParams(n_gamma=2048, n_ep=2048))
    ne = apt.Spectra.power_law_soft(2.0, 1e-5, 0.1)
    ic.init(ne, ne.emin(), ne.emax())
    g = np.exp(np.random.default_rng(3).uniform(0.1, np.log(1e15), 1 << 19))
    many = ic.gen_photon_e(g, seed=7, epoch=2)
    few = ic.gen_photon_e(g[:30000], seed=7, epoch=2)
    assert np.array_equal(many[:30000], few) and np.unique(few).size > 1000
