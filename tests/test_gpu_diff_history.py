"""Differentiable run: the position history against the checkpoints it
replaces, and its recompute paths."""
import numpy as np
import pytest

from common import rel_l2

pytestmark = pytest.mark.gpu


def make(n, nx=32, ny=16, seed=5):
    from cpic_amd import diff
    rng = np.random.default_rng(seed)
    sp = (np.arange(n) % 3).astype(np.int32)
    m = max(n, 1) / (nx * ny)
    run = diff.AdjointRun(nx, ny, (float(nx), float(ny)), 0.1, [-1.0, -1.0, 1.0],
                          [m, m, 1836 * m], sp, B=(0.0, 0.0, 0.2 * m))
    st = [rng.random(n) * nx, rng.random(n) * ny, rng.normal(0, 0.2, n), rng.normal(0, 0.2, n)]
    return run, st


@pytest.mark.parametrize("n", [1, 1023, 1025, 4097])
@pytest.mark.parametrize("steps,every", [(1, 1), (2, 1), (13, 5), (13, 50)])
def test_history_and_checkpoints_give_the_same_gradients(n, steps, every):
    run, st = make(n)
    loss, energy = run.forward(*st, steps, every)
    state, grad = run.state(), run.backward(1.0)
    again = run.backward(1.0)
    run.set_position_history(False)
    loss2, energy2 = run.forward(*st, steps, every)
    state2, grad2 = run.state(), run.backward(1.0)
    # same arithmetic, sums in another order
    assert abs(loss - loss2) <= 1e-12 * abs(loss)
    assert rel_l2(energy, energy2) < 1e-12
    for a, b, c in zip(grad, again, grad2):
        assert rel_l2(a, b) < 1e-9 and rel_l2(a, c) < 1e-9
    for a, b in zip(state, state2):
        assert rel_l2(a, b) < 1e-12
    run.close()


def test_history_can_be_switched_between_runs_of_different_length():
    run, st = make(2000)
    grads = {}
    for on, steps in ((True, 4), (False, 9), (True, 9), (True, 3), (False, 4)):
        run.set_position_history(on)
        run.forward(*st, steps, 4)
        g = run.backward(1.0)
        for a, b in zip(grads.setdefault(steps, g), g):
            assert rel_l2(b, a) < 1e-9
    run.close()
