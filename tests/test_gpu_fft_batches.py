"""Batches of idgx_fft2d on both sides of the size above which they are read and written past the caches (128 MB), and of
the launch groups (256 MB): the planes of a large batch have the bits of the same planes transformed in small ones."""
import pytest

torch = pytest.importorskip("torch")

import idgx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx, ny, fp64", [(512, 512, False), (256, 128, True), (1024, 16, False), (128, 64, False),
                                          (32, 16, True), (16, 512, False), (64, 64, False), (256, 256, False)])
@pytest.mark.parametrize("inplace", [False, True])
def test_large_batches_have_the_bits_of_small_ones(nx, ny, fp64, inplace):
    real = torch.float64 if fp64 else torch.float32
    plane_bytes = nx * ny * (16 if fp64 else 8)
    batch = (300 << 20) // plane_bytes + 1  # past the caches, and two launch groups
    few = (16 << 20) // plane_bytes  # through them
    g = torch.Generator(device="cuda")
    g.manual_seed(nx + ny)
    x = torch.randn((batch, ny, nx, 2), generator=g, device="cuda", dtype=real)
    picks = [(0, few), (batch // 2, few), (batch - few, few)]
    precision = idgx.FFT_FP64 if fp64 else idgx.FFT_FP32
    small = []
    for first, n in picks:
        y = torch.empty_like(x[:n])
        idgx.fft2d(x[first:first + n].clone(), y, nx, ny, n, -1, precision)
        small.append(y)
    out = x if inplace else torch.full_like(x, 3.0)
    idgx.fft2d(x, out, nx, ny, batch, -1, precision)
    for (first, n), y in zip(picks, small):
        assert torch.equal(out[first:first + n], y)
