"""Unsorted particle downloads are in storage order: the same state gives the
same rows in every call, whichever arrays a call asks for."""
import ctypes as C

import numpy as np
import pytest

import cpic_amd as ca

pytestmark = pytest.mark.gpu

GRID, TILE = 32, (16, 16)


def device(n, ids, flags, precision, steps=12, slack=0.0):
    """Fast particles in a few large buckets: every step leaves holes."""
    rng = np.random.default_rng(n)
    d = ca.Device(GRID, GRID, (float(GRID), float(GRID)), 0.1, [-1.0], [n / GRID ** 2],
                  precision=precision, flags=flags, tile=TILE, slack=slack)
    d.upload(0, ids, rng.random(n) * GRID, rng.random(n) * GRID, rng.normal(0, 3.0, n),
             rng.normal(0, 3.0, n))
    d.pre_step()
    for it in range(steps):
        d.step(it)
    assert n < 1000 or d.stats()["leavers"] > 0
    return d


def one_array(d, name):
    n = d.count(0)
    out = np.empty(n, np.int64 if name in ("id", "cell") else np.float64)
    p = ca.Particles()
    p.n = n
    setattr(p, name, (ca._ip if out.dtype == np.int64 else ca._dp)(out))
    ca.check(ca.lib().cpic_dev_download_particles(d._h, 0, C.byref(p)))
    return out


@pytest.mark.parametrize("slack", [0.0, -1.0])
@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("flags", [0, ca.F_IDS | ca.F_PARTICLE_E])
@pytest.mark.parametrize("n", [1, 257, 5003, 200003])
def test_every_call_gives_the_same_rows(n, flags, precision, slack):
    ids = np.arange(n) if flags else np.empty(0, np.int64)
    d = device(n, ids.astype(np.int64), flags, precision, slack=slack)
    whole, again = d.particles(0, sort=False), d.particles(0, sort=False)
    for k in whole:
        assert np.array_equal(whole[k], again[k]), k
        assert np.array_equal(whole[k], one_array(d, k)), k
    d.close()


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("ties", [1, 3])
def test_equal_indices_stay_in_storage_order(ties, precision):
    n = 100003
    d = device(n, np.arange(n, dtype=np.int64) % ties, ca.F_IDS, precision)
    stored, by_id = d.particles(0, sort=False), d.particles(0)
    order = np.argsort(stored["id"], kind="stable")
    for k in stored:
        assert np.array_equal(by_id[k], stored[k][order]), k
    d.close()
