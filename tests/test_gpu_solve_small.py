"""The one-workgroup solve (half-spectra up to 2,048 values) and the sizes on
either side of its edge, against the spectral solve in 64 bits."""
import numpy as np
import pytest
import torch

import cpic_amd as ca
from test_zz_no_alloc import DeviceGrid, hip_runtime, ok

pytestmark = pytest.mark.gpu

SHAPES = [(2, 2), (2, 4), (4, 2), (8, 8), (16, 16), (16, 256), (32, 64), (64, 32), (64, 64),
          (128, 32), (2048, 2), (2, 2048), (1024, 4), (4, 1024), (128, 64), (64, 128), (4096, 2),
          (2, 4096)]


def green(nx, ny):
    kx, ky = np.arange(nx // 2 + 1), np.arange(ny)
    den = 2.0 * (np.cos(2 * np.pi / nx * kx)[None, :] + np.cos(2 * np.pi / ny * ky)[:, None]) - 4.0
    den[0, 0] = np.inf
    return 1.0 / den


def reference(rho):
    ny, nx = rho.shape
    return np.fft.irfft2(np.fft.rfft2(rho) * green(nx, ny), s=(ny, nx))


def noalloc(rho):
    ny, nx = rho.shape
    h = hip_runtime()
    ok(h.hipSetDevice(0))
    g = DeviceGrid(h, rho)
    try:
        ok(ca.lib().cpic_solve_xy_noalloc(nx, ny, g.rho, g.phi, None))
        ok(h.hipStreamSynchronize(None))
        return g.read("phi")
    finally:
        g.free()


@pytest.mark.parametrize("nx,ny", SHAPES)
def test_solve_matches_the_spectral_reference(nx, ny):
    """1e-13 of the largest value, times the condition of the lowest mode: the
    Green's function cancels to about (pi / n)^2 of its terms."""
    rho = np.random.default_rng(nx + ny).normal(0, 1, (ny, nx))
    ref = reference(rho)
    tol = 1e-15 * max(nx, ny) ** 2 + 1e-13
    assert np.abs(noalloc(rho) - ref).max() <= tol * np.abs(ref).max()
    # the handle's solve, and the E array made from its phi
    d = ca.Device(nx, ny, (nx, ny), 0.1, [-1.0], [1.0])
    d.set_field("rho", rho)
    d.stage("field_E", 0)
    d.sync()
    phi = d.field("phi")
    assert np.abs(phi - ref).max() <= tol * np.abs(ref).max()
    ex = (np.roll(phi, 1, 1) - np.roll(phi, -1, 1)) / 2
    ey = (np.roll(phi, 1, 0) - np.roll(phi, -1, 0)) / 2
    assert np.array_equal(d.field("Ex"), ex) and np.array_equal(d.field("Ey"), ey)


@pytest.mark.parametrize("nx,ny", [(4, 8), (64, 64), (16, 256), (128, 64)])
@pytest.mark.parametrize("n", [1, 257, 6000])
def test_gradient_matches_the_torch_reference(nx, ny, n):
    """The transposed solve, and few particles per thread; bounds as in the
    64x64 gradient test: 1e-10 on the loss, 1e-7 on gradients."""
    from cpic_amd import diff
    from common import rel_l2
    from torch_pic import TorchPIC
    r = np.random.default_rng(n)
    st = [r.random(n) * nx, r.random(n) * ny, r.normal(0, 0.1, n), r.normal(0, 0.1, n)]
    sp = (np.arange(n) % 2).astype(np.int32)
    q, m, L = [-1.0] * 2, [max(n / (nx * ny), 1.0)] * 2, (float(nx), float(ny))
    run = diff.AdjointRun(nx, ny, L, 0.1, q, m, sp)
    loss, _ = run.forward(*st, 5, 3)
    g = run.backward(1.0)
    ref = TorchPIC(nx, ny, L, 0.1, q, m)
    t = [torch.tensor(a, requires_grad=True) for a in st]
    lref, _ = ref.run(*t, sp, 5)
    lref.backward()
    assert abs(loss - float(lref)) <= 1e-10 * abs(float(lref))
    scale = max(np.linalg.norm(b.grad.numpy()) for b in t)
    for a, b in zip(g, t):
        assert np.linalg.norm(a - b.grad.numpy()) <= 1e-7 * max(np.linalg.norm(b.grad.numpy()),
                                                                 1e-6 * scale)
    run.close()


@pytest.mark.parametrize("dx,dy", [(1.0, 1.0), (0.25, 0.25), (0.3, 0.3), (0.3, 0.25), (0.25, 0.3)])
def test_gradient_with_cells_of_other_sizes(dx, dy):
    """Cell sizes whose E stencil divides and whose multiplies; bounds as above."""
    from cpic_amd import diff
    from common import rel_l2
    from torch_pic import TorchPIC
    n, nx, ny = 700, 32, 16
    L = (nx * dx, ny * dy)
    r = np.random.default_rng(9)
    st = [r.random(n) * L[0], r.random(n) * L[1], r.normal(0, 0.02 * dx, n),
          r.normal(0, 0.02 * dy, n)]
    sp = np.zeros(n, np.int32)
    run = diff.AdjointRun(nx, ny, L, 0.1, [-1.0], [n / (nx * ny)], sp)
    ref = TorchPIC(nx, ny, L, 0.1, [-1.0], [n / (nx * ny)])
    loss, _ = run.forward(*st, 4, 2)
    g = run.backward(1.0)
    t = [torch.tensor(a, requires_grad=True) for a in st]
    lref, _ = ref.run(*t, sp, 4)
    lref.backward()
    assert abs(loss - float(lref.detach())) <= 1e-10 * abs(float(lref.detach()))
    for a, b in zip(g, t):
        assert rel_l2(a, b.grad.numpy()) < 1e-7
    run.close()


def test_batch_of_small_grids_of_different_shapes():
    shapes = [(64, 64), (16, 32), (128, 32), (8, 8)]
    b = ca.Batch([ca.make_desc(nx, ny, (nx, ny), 0.1, [-1.0], [1.0]) for nx, ny in shapes])
    rhos = [np.random.default_rng(k).normal(0, 1, (ny, nx)) for k, (nx, ny) in enumerate(shapes)]
    for k, rho in enumerate(rhos):
        b.set_field("rho", rho, plasma=k)
    b.stage("field_E", 0)
    b.sync()
    for k, rho in enumerate(rhos):
        ref = reference(rho)
        assert np.abs(b.field("phi", plasma=k) - ref).max() <= 1e-11 * np.abs(ref).max()
