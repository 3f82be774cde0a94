"""Device memory that a sort of a full particle set takes: the second particle
buffer and the sort's own arrays for the slots there are, no room beyond the
capacity."""
import pytest
import torch

import aperture3_amd as apt

pytestmark = pytest.mark.gpu


def context(n):
    env = apt.sim_environment(apt.SimParams(
        N=[n // 8, 1, 1], guard=[2, 0, 0], periodic_boundary=[True] * 3, max_ptc_number=n,
        precision=apt.APT_PREC_MIXED))
    d = apt.sim_data(env)
    d.fill_multiplicity(1.0, 4, (0.1, 0.1), (0.0, 0.0), sort=False)
    assert d.num_particles() == n
    d.sync()
    return d


def test_sort_of_a_full_set_takes_no_room_beyond_it():
    first = context(8000)
    first.sort_particles()  # the library's kernels are loaded
    n = 16000000
    d = context(n)
    before = torch.cuda.mem_get_info()[0]
    d.sort_particles()
    d.sync()
    taken = before - torch.cuda.mem_get_info()[0]
    # nine arrays of four bytes; two of keys and two of slots, and the library's
    # own pair of these; a quarter of them for its counters, the run table and the
    # last pages of some twenty arrays (half as much room again would be a half)
    arrays, scratch = 36 * n, 24 * n
    assert arrays + 16 * n <= taken <= arrays + scratch * 5 // 4, taken / n
    d.close()
