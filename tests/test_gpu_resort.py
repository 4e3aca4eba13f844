"""Re-sorts of few buckets and of many (8,192 is the line between two forms of
their kernels), with holes, full buckets and replaced species: every particle
is kept, in the bucket of its cell, and the run goes on as the oracle's."""
import numpy as np
import pytest

import cpic_amd as ca
import pyoracle as po
from common import rel_l2

pytestmark = pytest.mark.gpu


# 8x8 tiles and two species: 8,192 buckets at 512x512, 4,096 at 512x256
@pytest.mark.parametrize("nx,ny", [(512, 256), (512, 512)])
@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("flags", [0, ca.F_IDS, ca.F_IDS | ca.F_PARTICLE_E])
@pytest.mark.parametrize("slack", [0.0, -1.0])
def test_resort_keeps_every_particle(nx, ny, precision, flags, slack):
    n = (60_011, 40_013)
    rng = np.random.default_rng(nx + ny)
    d = ca.Device(nx, ny, (float(nx), float(ny)), 0.1, [-1.0, 1.0], [1.0, 100.0],
                  precision=precision, tile=(8, 8), flags=flags, slack=slack)
    for s, k in enumerate(n):
        ids = np.arange(k) if flags else np.empty(0)
        d.upload(s, ids.astype(np.int64), rng.random(k) * nx, rng.random(k) * ny,
                 rng.normal(0, 5.0, k), rng.normal(0, 5.0, k))
    d.pre_step()
    for it in range(6):
        d.step(it)
    assert d.stats()["leavers"] > 0

    def rows(s):
        p = d.particles(s, sort=False)
        a = np.stack([p[k].view(np.int64) for k in sorted(p)])
        return a[:, np.lexsort(a)]

    before = [rows(s) for s in range(2)]
    cells = [d.cell_counts(s) for s in range(2)]
    d.rebuild()
    for s in range(2):
        after = rows(s)
        assert after.shape == before[s].shape
        if precision == 64:
            assert np.array_equal(after, before[s])
        assert np.array_equal(d.cell_counts(s), cells[s])
        assert int(cells[s].sum()) == n[s]
    # one species replaced, the other kept
    d.upload(1, np.arange(7 if flags else 0), *(rng.random(7) for _ in range(4)))
    assert d.particles(1)["x"].shape == (7,) and np.array_equal(d.cell_counts(0), cells[0])
    d.close()


@pytest.mark.parametrize("nx,ny", [(512, 256), (512, 512)])
def test_run_across_a_resort_follows_the_oracle(nx, ny):
    n, L = 50_021, (float(nx), float(ny))
    rng = np.random.default_rng(5)
    o = po.Oracle(nx, ny, L, 0.1, [-1.0, -1.0], [1.0, 1.0])
    d = ca.Device(nx, ny, L, 0.1, [-1.0, -1.0], [1.0, 1.0], tile=(8, 8), flags=ca.F_IDS)
    for s in range(2):
        a = (np.arange(n), rng.random(n) * nx, rng.random(n) * ny, rng.normal(0, 1.0, n),
             rng.normal(0, 1.0, n))
        o.add(s, *a)
        d.upload(s, *a)
    o.pre_step()
    d.pre_step()
    for it in range(8):
        o.step()
        d.step(it)
        if it % 3 == 1:
            d.rebuild()
    d.sync()
    assert rel_l2(d.field("rho"), o.field("rho")) < 1e-12
    for s in range(2):
        a, b = o.particles(s), d.particles(s)
        assert np.array_equal(a["id"], b["id"])
        for k in ("x", "y", "ux", "uy"):
            assert rel_l2(b[k], a[k]) < 1e-12, (s, k)
    d.close()
