"""Downloads of every size that is copied in a way of its own (through small
bounce buffers, by the runtime, through full ones), by one handle, in both
orders."""
import numpy as np
import pytest

import cpic_amd as ca

pytestmark = pytest.mark.gpu

# 32 B, 2 KB, 8 KB, 16 KB, 64 KB, 512 KB, 1 MB, 8 MB, 16 MB
SHAPES = [(2, 2), (16, 16), (32, 32), (64, 32), (128, 64), (256, 256), (512, 256), (1024, 1024),
          (2048, 1024)]


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("order", [1, -1])
def test_fields_of_a_batch(order, precision):
    b = ca.Batch([ca.make_desc(nx, ny, (nx, ny), 0.1, [-1.0], [1.0], precision=precision)
                  for nx, ny in SHAPES])
    rho = [np.random.default_rng(k).normal(0, 1, (ny, nx)) for k, (nx, ny) in enumerate(SHAPES)]
    for k, a in enumerate(rho):
        b.set_field("rho", a, plasma=k)
    b.stage("field_E", 0)
    for k in list(range(len(SHAPES)))[::order] * 2:
        assert np.array_equal(b.field("rho", plasma=k), rho[k])
        phi = b.field("phi", plasma=k)
        ex = (np.roll(phi, 1, 1) - np.roll(phi, -1, 1)) / 2
        got = b.field("Ex", plasma=k)
        assert np.array_equal(got, ex if precision == 64 else ex.astype(np.float32)), SHAPES[k]
    b.close()


@pytest.mark.parametrize("n", [1, 250, 1030, 2050, 8200, 16400, 70000])
def test_particles_through_each_buffer(n):
    rng = np.random.default_rng(n)
    x, y, ux, uy = rng.random(n) * 32, rng.random(n) * 32, rng.normal(0, 1, n), rng.normal(0, 1, n)
    d = ca.Device(32, 32, (32.0, 32.0), 0.1, [-1.0], [max(n / 1024, 1.0)], flags=ca.F_IDS)
    d.upload(0, np.arange(n), x, y, ux, uy)
    for _ in range(2):
        p = d.particles(0)
        assert np.array_equal(p["id"], np.arange(n))
        for k, v in (("x", x), ("y", y), ("ux", ux), ("uy", uy)):
            assert np.array_equal(p[k], v), k
        assert np.array_equal(p["cell"], y.astype(np.int64) * 32 + x.astype(np.int64))
        assert d.field("rho").shape == (32, 32)
    d.close()
