"""What a download costs the host: threads that copy do not spin while the
device works."""
import time

import numpy as np
import pytest

import cpic_amd as ca

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
