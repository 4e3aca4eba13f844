"""Differentiable run: particle by particle against the references on both
sides of 262,144 particles, where the kernels go over from one particle per
thread to several (odd counts: the last block is partly filled), and with
checkpoints in place of the position history."""
import numpy as np
import pytest

import pyoracle as po
from common import rel_l2

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

FEW = 262_144


def state_of(n, nx, v0, sigma, seed):
    """Two beams, the first with the odd particle."""
    rng = np.random.default_rng(seed)
    sp = (np.arange(n) >= n - n // 2).astype(np.int32)
    x, y = rng.random(n) * nx, rng.random(n) * nx
    ux = np.where(sp == 0, v0, -v0) + rng.normal(0, sigma, n)
    return sp, [x, y, ux, rng.normal(0, sigma, n)]


def run_of(n, nx, sp):
    from cpic_amd import diff
    m = n / nx ** 2
    return diff.AdjointRun(nx, nx, (float(nx), float(nx)), 0.1, [-1.0, -1.0], [m, m], sp)


def torch_gradient(n, nx, sp, st, steps):
    from torch_pic import TorchPIC
    m = n / nx ** 2
    ref = TorchPIC(nx, nx, (float(nx), float(nx)), 0.1, [-1.0, -1.0], [m, m])
    t = [torch.tensor(a, requires_grad=True) for a in st]
    loss, _ = ref.run(*t, sp, steps)
    loss.backward()
    return float(loss.detach()), [a.grad.numpy() for a in t]


@pytest.mark.parametrize("history", [True, False])
@pytest.mark.parametrize("n", [FEW, FEW + 1, FEW + 1025])
def test_either_side_of_several_particles_per_thread(n, history):
    """64x64, fast beams that cross x = 0, 10 steps; bounds of the other
    differentiable tests: 1e-12 on states and energies against the oracle,
    1e-10 on the loss and 1e-7 on gradients against torch."""
    nx, steps = 64, 10
    sp, st = state_of(n, nx, 0.5, 0.05, 37)
    run = run_of(n, nx, sp)
    run.set_position_history(history)
    loss, W = run.forward(*st, steps, 4)
    out, grad = run.state(), run.backward(1.0)
    run.close()

    m = n / nx ** 2
    o = po.Oracle(nx, nx, (float(nx), float(nx)), 0.1, [-1.0, -1.0], [m, m])
    for s in range(2):
        k = sp == s
        o.add(s, np.arange(int(k.sum())), *(a[k] for a in st))
    o.pre_step()
    Wo = []
    for it in range(steps):
        o.stage("field_E")
        Wo.append(o.field_energy())
        o.stage("plasma_E")
        o.stage("plasma_r")
        o.stage("field_rho")
        o.iter = it + 1
    assert rel_l2(W, Wo) < 1e-12
    for s in range(2):
        a = o.particles(s)
        for name, v in zip(("x", "y", "ux", "uy"), out):
            assert rel_l2(v[sp == s], a[name]) < 1e-12, (s, name)

    lref, gref = torch_gradient(n, nx, sp, st, steps)
    assert abs(loss - lref) < 1e-10 * abs(lref)
    for a, b in zip(grad, gref):
        assert rel_l2(a, b) < 1e-7


@pytest.mark.parametrize("n", [10_240, 10_241])
def test_checkpoints_without_the_position_history(n):
    """60 steps: every interval from a checkpoint per step to one for the whole
    run, a partial last segment and an interval beyond the run, with the field
    history and without."""
    nx, steps = 64, 60
    sp, st = state_of(n, nx, 0.1, 0.01, 31)
    lref, gref = torch_gradient(n, nx, sp, st, steps)
    run = run_of(n, nx, sp)
    run.set_position_history(False)
    for fields in (True, False):
        run.set_field_history(fields)
        for every in (1, 7, 20, steps, 500):
            loss, _ = run.forward(*st, steps, every)
            assert abs(loss - lref) < 1e-10 * abs(lref), (fields, every)
            for a, b in zip(run.backward(1.0), gref):
                assert rel_l2(a, b) < 1e-7, (fields, every)
    run.close()


@pytest.mark.parametrize("array,value", [(0, 0.0), (0, 32.0), (1, 0.0), (1, 32.0), (2, -1e-9),
                                         (3, -1e-9), (2, 3.0), (3, -3.0)])
def test_inputs_at_the_edges_of_what_is_accepted(array, value):
    """Positions on the box's edges and velocities of either sign: iteration 0
    leaves the positions as they came."""
    n = 1500
    sp, st = state_of(n, 32, 0.1, 0.01, 2)
    st[array][n - 1] = value
    run = run_of(n, 32, sp)
    run.forward(*st, 1, 1)
    x, y, ux, uy = run.state()
    assert np.array_equal(x, st[0]) and np.array_equal(y, st[1])
    assert np.all(np.isfinite(ux)) and np.all(np.isfinite(uy))
    for g in run.backward(1.0):
        assert np.all(np.isfinite(g))
    run.close()
