"""Differentiable run: the device's particle order (cells, round-robin in
chunks of 1,024) leaves every particle in the caller's place."""
import numpy as np
import pytest
import torch

import cpic_amd as ca
from common import rel_l2

pytestmark = pytest.mark.gpu

PLACES = {
    "uniform": lambda n, nx, ny, r: (r.random(n) * nx, r.random(n) * ny),
    "one_cell": lambda n, nx, ny, r: (r.random(n), r.random(n)),
    "far_edge": lambda n, nx, ny, r: (np.full(n, float(nx)), np.full(n, float(ny))),
    "one_row": lambda n, nx, ny, r: (r.random(n) * nx, np.full(n, ny - 0.5)),
    "two_cells": lambda n, nx, ny, r: (np.where(np.arange(n) % 5 == 0, 0.5, nx - 0.5),
                                       r.random(n)),
}


def run_of(n, nx, ny, ns=2):
    from cpic_amd import diff
    return diff.AdjointRun(nx, ny, (float(nx), float(ny)), 0.1, [-1.0] * ns,
                           [n / (nx * ny)] * ns, (np.arange(n) % ns).astype(np.int32))


@pytest.mark.parametrize("nx,ny", [(2, 2), (64, 32), (512, 256)])
@pytest.mark.parametrize("n", [1, 64, 1024, 1025, 5000])
@pytest.mark.parametrize("place", sorted(PLACES))
def test_state_comes_back_in_the_callers_order(place, n, nx, ny):
    r = np.random.default_rng(n)
    x, y = PLACES[place](n, nx, ny, r)
    # iteration 0 leaves positions where they are; one cell of 2x2 has E = 0
    run = run_of(n, nx, ny)
    run.forward(x, y, np.arange(n) * 1e-9, np.zeros(n), 1, 1)
    gx, gy, gux, _ = run.state()
    assert np.array_equal(gx, x) and np.array_equal(gy, y)
    run.close()


@pytest.mark.parametrize("n", [1, 1025, 3000])
def test_gradients_match_the_torch_reference(n):
    """Bounds as in the 64x64 gradient test: 1e-10 on the loss, 1e-7 on gradients."""
    from torch_pic import TorchPIC
    r = np.random.default_rng(n)
    nx, ny = 32, 32
    st = [r.random(n) * nx, r.random(n) * ny, r.normal(0, 0.1, n), r.normal(0, 0.1, n)]
    sp = (np.arange(n) % 2).astype(np.int32)
    run = run_of(n, nx, ny)
    loss, _ = run.forward(*st, 6, 4)
    g = run.backward(1.0)
    ref = TorchPIC(nx, ny, (float(nx), float(ny)), 0.1, [-1.0] * 2, [n / (nx * ny)] * 2)
    t = [torch.tensor(a, requires_grad=True) for a in st]
    lref, _ = ref.run(*t, sp, 6)
    lref.backward()
    assert abs(loss - float(lref)) < 1e-10 * abs(float(lref))
    for a, b in zip(g, t):
        assert rel_l2(a, b.grad.numpy()) < 1e-7
    run.close()


@pytest.mark.parametrize("array", range(4))
@pytest.mark.parametrize("value", [np.nan, np.inf, -1e-9, 33.0])
def test_refused_input_leaves_the_last_forward_usable(array, value):
    n = 1500
    r = np.random.default_rng(2)
    st = [r.random(n) * 32, r.random(n) * 32, r.normal(0, 0.1, n), r.normal(0, 0.1, n)]
    run = run_of(n, 32, 32)
    run.forward(*st, 5, 2)
    state, g = run.state(), run.backward(1.0)
    bad = [a.copy() for a in st]
    bad[array][n - 1] = value
    if array < 2 or not np.isfinite(value):
        with pytest.raises(ca.CpicError):
            run.forward(*bad, 5, 2)
        for a, b in zip(state, run.state()):
            assert np.array_equal(a, b)
        for a, b in zip(g, run.backward(1.0)):
            assert rel_l2(b, a) < 1e-9
    run.close()
