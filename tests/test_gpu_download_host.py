"""What a download costs the host: threads that copy do not spin while the
device works, and destinations in pinned memory are written by the device."""
import ctypes as C
import time

import numpy as np
import pytest

import cpic_amd as ca
from test_zz_no_alloc import hip_runtime, ok

pytestmark = pytest.mark.gpu


def cpu_and_wall(f):
    c, w = time.process_time(), time.perf_counter()
    f()
    return time.process_time() - c, time.perf_counter() - w


def test_a_download_behind_a_long_queue_sleeps():
    """CPU time of the whole process while a field download waits for about
    half a second of queued steps: the calling thread and one of the runtime's
    may poll (2x the wall time); sixteen copying threads would add 16x."""
    g, n = 2048, 16_000_000
    rng = np.random.default_rng(1)
    d = ca.Device(g, g, (float(g), float(g)), 0.05, [-1.0], [n / g ** 2], precision=32)
    d.upload(0, np.empty(0, np.int64), rng.random(n) * g, rng.random(n) * g,
             rng.normal(0, 0.1, n), rng.normal(0, 0.1, n))
    d.pre_step()
    d.run(0, 21)
    d.sync()
    d.field("rho")
    steps = 21
    _, wall = cpu_and_wall(lambda: (d.run(steps, 20), d.sync()))
    steps += 20
    more = 20 * int(0.5 / wall + 1)
    queue, _ = cpu_and_wall(lambda: d.run(steps, more))
    cpu, wall = cpu_and_wall(lambda: d.field("rho"))
    print(f"queueing {queue:.3f} s of CPU time; download {cpu:.3f} s in {wall:.3f} s")
    assert wall > 0.1
    assert cpu < 4.0 * wall
    d.close()


class Pinned:
    """n doubles of host memory allocated by the HIP runtime."""

    def __init__(self, n):
        self.h, self.p = hip_runtime(), C.c_void_p()
        ok(self.h.hipSetDevice(0))
        self.h.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
        self.h.hipHostFree.argtypes = [C.c_void_p]
        ok(self.h.hipHostMalloc(C.byref(self.p), 8 * n, 0))
        self.a = np.ctypeslib.as_array(C.cast(self.p, C.POINTER(C.c_double)), (n,))

    def free(self):
        self.a = None
        ok(self.h.hipHostFree(self.p))


@pytest.mark.parametrize("which", ["rho", "phi"])
def test_a_pinned_destination_is_copied_to_directly(which):
    """128 MB: the host's own copy out of a bounce buffer takes several
    milliseconds of CPU time, a copy by the device next to none."""
    g = 4096
    d = ca.Device(g, g, (float(g), float(g)), 0.1, [-1.0], [1.0])
    f = np.random.default_rng(2).random((g, g))
    d.set_field(which, f)
    pinned = Pinned(g * g)
    cpu = {}
    for kind, a in (("pageable", np.zeros(g * g)), ("pinned", pinned.a)):
        def read():
            ca.check(ca.lib().cpic_dev_download_field(d._h, ca.FIELDS[which], ca._dp(a)))
        read()
        assert np.array_equal(a, f.ravel())
        a[:] = 0.0
        cpu[kind] = sum(cpu_and_wall(read)[0] for _ in range(10))
        assert np.array_equal(a, f.ravel())
    del a
    print(cpu)
    assert cpu["pinned"] < 0.5 * cpu["pageable"]
    d.close()
    pinned.free()


@pytest.mark.parametrize("n", [1, 301, 300001])
def test_pinned_and_ordinary_arrays_in_one_call(n):
    """Two arrays that share one pinned allocation, two ordinary ones."""
    rng = np.random.default_rng(3)
    x, y = rng.random(n) * 64, rng.random(n) * 64
    ux, uy = rng.normal(0, 0.1, n), rng.normal(0, 0.1, n)
    d = ca.Device(64, 64, (64.0, 64.0), 0.1, [-1.0], [max(n / 64 ** 2, 1.0)])
    d.upload(0, np.empty(0, np.int64), x, y, ux, uy)
    pinned = Pinned(2 * n)
    out = {"x": pinned.a[:n], "y": np.full(n, np.nan), "ux": pinned.a[n:], "uy": np.full(n, np.nan)}
    p = ca.Particles()
    p.n = n
    for k, a in out.items():
        setattr(p, k, ca._dp(a))
    ca.check(ca.lib().cpic_dev_download_particles(d._h, 0, C.byref(p)))
    ref = d.particles(0)
    for k, a in out.items():
        assert np.array_equal(a, ref[k]), k
    assert np.array_equal(np.sort(ref["x"]), np.sort(x))
    del out, a
    d.close()
    pinned.free()


@pytest.mark.parametrize("n", [1, 4097, 300001])
def test_gradients_of_pinned_inputs_into_pinned_outputs(n):
    from cpic_amd import diff
    nx = 32
    r = np.random.default_rng(4)
    st = [r.random(n) * nx, r.random(n) * nx, r.normal(0, 0.1, n), r.normal(0, 0.1, n)]
    run = diff.AdjointRun(nx, nx, (float(nx), float(nx)), 0.1, [-1.0], [max(n / nx ** 2, 1.0)],
                          np.zeros(n, np.int32))
    run.forward(*st, 3, 2)
    ref = run.backward(1.0)
    pinned = Pinned(8 * n)
    ins, outs = np.split(pinned.a, 8)[:4], np.split(pinned.a, 8)[4:]
    for a, b in zip(ins, st):
        a[:] = b
    run.forward(*ins, 3, 2)
    for a, b in zip(run.state(), st):
        assert a.shape == b.shape
    ca.check(ca.lib().cpic_adj_backward(run._h, 1.0, *(ca._dp(a) for a in outs)))
    for a, b in zip(outs, ref):
        assert np.linalg.norm(a - b) <= 1e-9 * np.linalg.norm(b)
    del ins, outs, a, b
    run.close()
    pinned.free()
