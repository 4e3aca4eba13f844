"""E read between bursts of replayed steps belongs to the last of them."""
import numpy as np
import pytest

import cpic_amd as ca

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flags", [0, ca.F_IDS, ca.F_IDS | ca.F_PARTICLE_E])
@pytest.mark.parametrize("edge", [32, 128])
def test_E_after_every_burst_is_the_gradient_of_phi(edge, flags):
    n = 4000
    r = np.random.default_rng(1)
    d = ca.Device(edge, edge, (edge, edge), 0.1, [-1.0], [n / edge ** 2], flags=flags, tile=(8, 8))
    ids = np.arange(n if flags & ca.F_IDS else 0, dtype=np.int64)
    d.upload(0, ids, r.random(n) * edge, r.random(n) * edge, r.normal(0, 0.1, n),
             r.normal(0, 0.1, n))
    d.pre_step()
    it = 0
    for burst in (1, 4, 4, 5, 4):
        d.run(it, burst)
        it += burst
        d.sync()
        phi = d.field("phi")
        assert np.array_equal(d.field("Ex"), (np.roll(phi, 1, 1) - np.roll(phi, -1, 1)) / 2)
        assert np.array_equal(d.field("Ey"), (np.roll(phi, 1, 0) - np.roll(phi, -1, 0)) / 2)
