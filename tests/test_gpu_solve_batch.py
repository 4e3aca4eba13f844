"""Batches of small grids on either side of the number of plasmas up to which
each is one workgroup's solve, against the spectral solve in 64 bits."""
import numpy as np
import pytest

import cpic_amd as ca
from test_gpu_solve_small import reference

pytestmark = pytest.mark.gpu

# grid of most plasmas, its limit (0: none)
LIMITS = [((8, 8), 1280), ((16, 8), 1024), ((16, 16), 768), ((32, 16), 1536), ((32, 32), 1536),
          ((64, 32), 2304), ((64, 64), 0)]


def solve(shapes):
    tile = (8, 8)
    b = ca.Batch([ca.make_desc(nx, ny, (nx, ny), 0.1, [-1.0], [1.0], tile=tile, flags=ca.F_PROFILE)
                  for nx, ny in shapes])
    some = sorted({0, 1, len(shapes) // 2, len(shapes) - 1})
    rhos = {}
    for p in some:
        nx, ny = shapes[p]
        rhos[p] = np.random.default_rng(p).normal(0, 1, (ny, nx))
        b.set_field("rho", rhos[p], plasma=p)
    b.stage("field_E", 0)
    b.sync()
    for p, rho in rhos.items():
        ref = reference(rho)
        # of the largest value: the lowest mode's condition, as in the single solves
        tol = 1e-15 * max(rho.shape) ** 2 + 1e-13
        assert np.abs(b.field("phi", plasma=p) - ref).max() <= tol * np.abs(ref).max()
    names = set(b.kernel_times())
    b.close()
    return names


@pytest.mark.parametrize("grid,limit", LIMITS)
@pytest.mark.parametrize("beyond", [0, 1])
def test_either_side_of_the_limit(grid, limit, beyond):
    names = solve([grid] * ((limit or 2500) + beyond))
    assert ("solve_small" in names) == (not beyond or not limit), names
    assert ("fft_rows_r2c" in names) == (bool(limit) and bool(beyond)), names


def test_mixed_shapes_share_the_limit():
    """384 of 768 and 768 of 1536 are the whole of it; 64x64 takes no share."""
    mix = [(16, 16), (32, 32), (64, 64), (32, 32)] * 384
    assert "solve_small" in solve(mix)
    assert "fft_rows_r2c" in solve(mix + [(8, 8)])
    assert "fft_rows_r2c" in solve([(64, 64), (128, 64)])
