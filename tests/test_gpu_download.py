"""Particle and field downloads: order by index, and every size of the copy
(one bounce buffer, several, the calling thread alone, several threads)."""
import numpy as np
import pytest

import cpic_amd as ca

pytestmark = pytest.mark.gpu


def device(n, ids, flags, precision=64, seed=3, steps=3):
    rng = np.random.default_rng(seed)
    nx, ny, L = 64, 32, (64.0, 32.0)
    d = ca.Device(nx, ny, L, 0.1, [-1.0], [max(n, 1) / (nx * ny)], precision=precision,
                  flags=flags, tile=(8, 8))
    d.upload(0, ids, rng.random(n) * L[0], rng.random(n) * L[1], rng.normal(0, 0.1, n),
             rng.normal(0, 0.1, n))
    d.pre_step()
    d.run(0, steps)
    d.sync()
    return d


def rows(p):
    """The particles as sorted tuples: order among equal indices aside."""
    keys = sorted(p)
    a = np.stack([p[k].view(np.int64) for k in keys])
    return a[:, np.lexsort(a)]


INDEX_SETS = {
    "arange": lambda n, r: np.arange(n),
    "shuffled_offset": lambda n, r: r.permutation(n) - 7,
    "gaps": lambda n, r: r.permutation(n) * 3 + 11,
    "dense_range_with_a_duplicate": lambda n, r: np.where(np.arange(n) == n // 2, 0, np.arange(n)),
    "extremes": lambda n, r: np.where(np.arange(n) == 0, np.iinfo(np.int64).min,
                                      np.where(np.arange(n) == 1, np.iinfo(np.int64).max,
                                               np.arange(n))),
    "all_equal": lambda n, r: np.zeros(n, np.int64),
}


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("n", [1, 2, 65, 3001])
@pytest.mark.parametrize("kind", sorted(INDEX_SETS))
def test_sorted_download_is_the_unsorted_one_in_order(kind, n, precision):
    ids = INDEX_SETS[kind](n, np.random.default_rng(n)).astype(np.int64)
    d = device(n, ids, ca.F_IDS | ca.F_PARTICLE_E, precision)
    got, ref = d.particles(0), d.particles(0, sort=False)
    assert np.array_equal(got["id"], np.sort(ids))
    assert np.array_equal(rows(got), rows(ref))


@pytest.mark.parametrize("n", [16385, 140000, 600001])
def test_large_downloads_arrive_whole(n):
    """1.0 MB, 9.0 MB and 38 MB: below and above one buffer, odd ends."""
    ids = np.random.default_rng(1).permutation(n).astype(np.int64)
    d = device(n, ids, ca.F_IDS | ca.F_PARTICLE_E)
    got, ref = d.particles(0), d.particles(0, sort=False)
    order = np.argsort(ref["id"])
    for k in ref:
        assert np.array_equal(got[k], ref[k][order]), k


def test_stages_one_by_one_gather_what_the_step_stores():
    n = 5000
    a = device(n, np.arange(n), ca.F_IDS | ca.F_PARTICLE_E, steps=0)
    b = device(n, np.arange(n), ca.F_IDS | ca.F_PARTICLE_E, steps=0)
    a.step(0)
    b.stage("field_E", 0)
    b.stage("plasma_E", 0)
    pa, pb = None, b.particles(0)
    b.stage("plasma_r", 0)
    b.stage("field_rho", 0)
    a.sync()
    b.sync()
    pa, pc = a.particles(0), b.particles(0)
    # two deposits of the same particles differ by the order of their sums
    for k in ("Ex", "Ey"):
        scale = np.abs(pb[k]).max()
        assert np.abs(pa[k] - pb[k]).max() <= 1e-12 * scale
        assert np.abs(pc[k] - pb[k]).max() == 0.0


@pytest.mark.parametrize("edge", [16, 256, 512, 2048])
def test_field_roundtrip(edge):
    d = ca.Device(edge, edge, (edge, edge), 0.1, [-1.0], [1.0])
    f = np.random.default_rng(edge).random((edge, edge))
    d.set_field("rho", f)
    assert np.array_equal(d.field("rho"), f)


def test_needs_indices():
    d = device(10, np.zeros(0, np.int64), 0)
    assert ca.lib().cpic_batch_download_particles_by_id(d._h, 0, 0, ca.Particles()) != 0
