"""The push's work units and slots against the oracle: buckets shared by
several workgroups, chunk remainders, holes left by leavers and filled by
arrivals, and the compacting push of large states (FP32 above 0.8 GB, FP64
above 1.25 GB).  FP64 within 1e-12
relative L2 of the oracle (rounding of the deposit's order only), FP32 within
1e-5."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import cpic_amd as ca                        # noqa: E402
import pyoracle as po                        # noqa: E402
from common import rel_l2, two_stream        # noqa: E402

BAR = {64: 1e-12, 32: 1e-5}


def run_both(n, grid, tile, precision, ppt, steps, v0, ids=True, seed=3):
    L = (float(grid), float(grid))
    m = max(1.0, 2 * n / (L[0] * L[1]))
    parts = two_stream(n, L, v0, 0.01, seed)
    o = po.Oracle(grid, grid, L, 0.1, [-1.0, -1.0], [m, m])
    d = ca.Device(grid, grid, L, 0.1, [-1.0, -1.0], [m, m], precision=precision, tile=tile,
                  ppt=ppt, flags=ca.F_IDS if ids else 0)
    for s, (i, x, y, ux, uy) in enumerate(parts):
        o.add(s, i, x, y, ux, uy)
        d.upload(s, i if ids else np.empty(0, np.int64), x, y, ux, uy)
    del parts
    o.pre_step()
    d.pre_step()
    for _ in range(steps):
        o.step()
    d.run(0, steps)
    d.sync()
    return o, d


# one bucket per species: particle counts around a chunk (U * 256), a part
# (2048) and several parts
@pytest.mark.parametrize("precision,ppt", [(64, 2), (64, 4), (32, 2), (32, 4)])
@pytest.mark.parametrize("n", [1, 63, 65, 511, 1025, 2049, 20003])
def test_bucket_remainders_and_parts(n, precision, ppt):
    o, d = run_both(n, 8, (8, 8), precision, ppt, 6, 0.1)
    for f in ("rho", "phi"):
        assert rel_l2(d.field(f), o.field(f)) < BAR[precision], f
    for s in range(2):
        a, b = o.particles(s), d.particles(s)
        assert np.array_equal(a["id"], b["id"])
        for k in ("x", "y", "ux", "uy"):
            assert rel_l2(b[k], a[k]) < BAR[precision], (s, k)
    d.close()


@pytest.mark.parametrize("precision", [64, 32])
def test_holes_are_reused_and_nothing_is_lost(precision):
    """Beams of 0.5 cells per step: each particle crosses 60 * 0.5 / 8 = 3.75
    tile edges in 60 steps, so slots become holes and are taken again."""
    o, d = run_both(30011, 32, (8, 8), precision, 4, 60, 5.0)
    st = d.stats()
    assert st["leavers"] > 3 * 2 * 30011 and st["nparticles"] == 2 * 30011, st
    assert rel_l2(d.field("rho"), o.field("rho")) < 100 * BAR[precision]
    for s in range(2):
        b = d.particles(s)
        assert np.array_equal(b["id"], np.arange(30011))
        # every particle is counted once, in the cell of its position
        cell = b["y"].astype(np.int64) * 32 + b["x"].astype(np.int64)
        assert np.array_equal(cell, b["cell"])
        assert np.array_equal(np.bincount(b["cell"], minlength=1024), d.cell_counts(s).ravel())
    d.rebuild()
    for s in range(2):
        assert np.array_equal(d.particles(s)["id"], np.arange(30011))
    d.close()


@pytest.mark.parametrize("precision,n,ppt", [(64, 20_500_003, 4), (32, 26_500_003, 4),
                                             (32, 26_500_003, 2)])
def test_compacting_push_of_a_large_state(precision, n, ppt):
    """2 n particles: just above the limit of the in-place push, and sized
    again below it."""
    o, d = run_both(n, 256, (16, 16), precision, ppt, 3, 0.1, ids=False)
    for f in ("rho", "phi", "Ex", "Ey"):
        assert rel_l2(d.field(f), o.field(f)) < BAR[precision], f
    for s in range(2):
        assert int(d.cell_counts(s).sum()) == n
    x = np.linspace(0.0, 255.0, 1000)
    d.upload(0, np.empty(0, np.int64), x, x, 0 * x, 0 * x)    # in place from here on
    d.rebuild()
    d.run(3, 4)
    d.sync()
    assert int(d.cell_counts(0).sum()) == 1000 and int(d.cell_counts(1).sum()) == n
    d.close()


def test_compact_buckets_that_overflow():
    """Buckets filled to the last slot (slack < 0): arrivals that find no room
    go back to their source, behind a gap, in the compacting push too (67 M
    FP32 particles in 64 x 64 cells); every particle stays counted."""
    n, grid = 33_554_432, 64
    rng = np.random.default_rng(5)
    L = (float(grid), float(grid))
    d = ca.Device(grid, grid, L, 0.1, [-1.0, -1.0], [2.0 * n / grid ** 2] * 2, precision=32,
                  tile=(16, 16), slack=-1.0)
    e = np.empty(0, np.int64)
    x, y = rng.uniform(0.0, grid, n), rng.uniform(0.0, grid, n)
    ux, uy = rng.normal(0.0, 1.0, n), rng.normal(0.0, 1.0, n)
    d.upload(0, e, x, y, ux, uy)
    d.upload(1, e, x, y, -ux, -uy)
    d.pre_step()
    total = float(d.field("rho").sum())
    d.run(0, 4)                     # no sync in between: no re-sort
    for s in range(2):
        assert int(d.cell_counts(s).sum()) == n
    # the charge is that of all particles (FP32 weights sum to 1 within 2^-22)
    assert abs(float(d.field("rho").sum()) - total) < 2.0 ** -22 * total
    assert d.stats()["fallbacks"] > 0
    px = [d.energy()[k] for k in ("px", "py")]
    assert np.all(np.isfinite(px))
    d.sync()                        # re-sorts
    d.run(4, 3)
    for s in range(2):
        assert int(d.cell_counts(s).sum()) == n
    d.close()
