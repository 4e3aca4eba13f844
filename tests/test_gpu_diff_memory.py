"""Differentiable run: a forward gives back the history or the checkpoints of
the mode that it does not use."""
import ctypes as C

import numpy as np
import pytest

from test_zz_no_alloc import hip_runtime, ok

pytestmark = pytest.mark.gpu

N, NX, STEPS, EVERY = 200_001, 32, 60, 10
HISTORY = 16 * N * STEPS
# every sixth iteration's state, and the positions of a segment's others
CHECKPOINTS = 32 * N * (STEPS // EVERY) + 16 * N * (EVERY - 1)
MARGIN = 16 << 20           # allocation granularity of nine buffers, 2 MB each


def used():
    free, total = C.c_size_t(), C.c_size_t()
    ok(hip_runtime().hipMemGetInfo(C.byref(free), C.byref(total)))
    return total.value - free.value


def run_of():
    from cpic_amd import diff
    return diff.AdjointRun(NX, NX, (float(NX), float(NX)), 0.1, [-1.0], [N / NX ** 2],
                           np.zeros(N, np.int32))


def gradients(run, steps=STEPS):
    r = np.random.default_rng(1)
    run.forward(r.random(N) * NX, r.random(N) * NX, r.normal(0, 0.1, N), r.normal(0, 0.1, N),
                steps, EVERY)
    return run.backward(1.0)


def held(modes):
    """Device memory that a run holds after a pass in each mode."""
    run = run_of()
    run.set_position_history(False)
    gradients(run, 1)                   # the buffers that both modes share
    base, out = used(), []
    for on in modes:
        run.set_position_history(on)
        gradients(run)
        out.append(used() - base)
    run.close()
    return out


def test_switching_gives_the_other_modes_memory_back():
    assert HISTORY > CHECKPOINTS + 4 * MARGIN
    held([True])                        # code objects and pinned buffers
    on, off, on_again, off_again = held([True, False, True, False])
    assert abs(on - HISTORY) < MARGIN, on
    assert abs(off - CHECKPOINTS) < MARGIN, off
    assert abs(on_again - on) < MARGIN and abs(off_again - off) < MARGIN


def test_a_backward_after_switching_still_has_its_history():
    """The switch is for later forwards."""
    run = run_of()
    r = np.random.default_rng(1)
    st = [r.random(N) * NX, r.random(N) * NX, r.normal(0, 0.1, N), r.normal(0, 0.1, N)]
    run.forward(*st, 6, 4)
    a = run.backward(1.0)
    run.set_position_history(False)
    b = run.backward(1.0)
    run.forward(*st, 6, 4)
    run.set_position_history(True)
    c = run.backward(1.0)
    for u, v, w in zip(a, b, c):
        assert np.linalg.norm(u - v) <= 1e-9 * np.linalg.norm(u)
        assert np.linalg.norm(u - w) <= 1e-9 * np.linalg.norm(u)
    run.close()
