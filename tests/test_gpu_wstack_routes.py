"""The image side of a cycle where its route depends on the call: one layer at w = 0 takes the boxed transform's own row
pass (from the image only for boxes of at least three quarters of the columns), the box decides between the boxed and
the full transform to uv, and n(l, m) is a series up to a field of 0.2 rad and a square root beyond it.

Against FP64 (numpy FFTs), for one correlation.  Tolerance: an FP32 transform of a side of G <= 2048 points rounds about
12 times per axis, 24 roundings of 6e-8 whose root mean square grows with the square root (3e-7); the screens add 1e-7
absolute and the sum over layers less.  1e-6 holds these."""
import numpy as np
import pytest

from helpers import rel_l2
from idgx import FFT_FORWARD, METADATA_DTYPE, grid_fft_box, grid_to_image, image_to_grid, observation
from idgx.device import DeviceWorkload, download, upload

pytestmark = pytest.mark.gpu

TOL = 1e-6


def _device_workload(G, image_size, w_step, S=16):
    md = np.zeros(1, METADATA_DTYPE)
    md["nr_timesteps"] = 1
    md["station2"] = 1
    return DeviceWorkload(dict(
        metadata=md, channels=None, subgrid_size=S, grid_size=G, nr_stations=2, nr_aterm_slots=1,
        image_size=np.float32(image_size), w_step=w_step, wavenumbers=np.full(1, 3.0, np.float32),
        uvw=np.zeros((1, 3), np.float32), visibilities=np.zeros((1, 1, 4), np.complex64),
        spheroidal=np.ones((S, S), np.float32), aterms=observation.identity_aterms(1, 2, S), max_nr_timesteps=1,
        nr_subgrids=1))


def _centred(x, sign):
    G = x.shape[-1]
    c = (-1.0) ** np.arange(G)
    cc = c[:, None] * c[None, :]
    return (np.fft.ifft2(x * cc) * (G * G) if sign > 0 else np.fft.fft2(x * cc)) * cc


def _screens(G, image_size, w_step, z_min, nl):
    lm = (np.arange(G) - G / 2) * float(np.float32(image_size)) / G
    r2 = lm[None, :] ** 2 + lm[:, None] ** 2
    n = r2 / (1 + np.sqrt(1 - r2))
    return [np.exp(-2j * np.pi * (z_min + k + 0.5) * w_step * n) for k in range(nl)]


# One layer at w = 0 (0.0), one layer with a screen, three layers; fields on both sides of the series' 0.2 rad (w_step
# such that the outermost layer turns about 8 times in the corner).
@pytest.mark.parametrize("nl, field, w_step", [(1, 0.1, 0.0), (1, 0.1, 1600.0), (3, 0.19, 440.0), (3, 0.5, 64.0)])
@pytest.mark.parametrize("G, box", [
    (1024, (0, 1024, 0, 1024)),     # every cell: the full transform to uv
    (1024, (100, 869, 3, 1021)),    # 13 of 16 column tiles: the boxed passes, and the plain row pass at w = 0
    (1024, (130, 760, 100, 523)),   # 10 of 16: the w-stacked row pass from the image
    (2048, (1000, 1001, 2047, 2048)),
])
def test_grid_to_image_and_back_match_fp64(G, box, nl, field, w_step):
    rng = np.random.default_rng(17)
    z_min = -1
    dw = _device_workload(G, field, w_step)
    plan = dw.plan()
    screens = _screens(G, field, w_step, z_min, nl)
    x0, x1, y0, y1 = box
    x = np.zeros((nl, 4, G, G), np.complex64)
    x[..., y0:y1, x0:x1] = (rng.standard_normal((nl, 4, y1 - y0, x1 - x0)) +
                            1j * rng.standard_normal((nl, 4, y1 - y0, x1 - x0)))
    junk = x.copy()  # rows outside the box are not read
    junk[..., :y0, :] = 5 + 5j
    junk[..., y1:, :] = -3 + 1j
    d_img = dw.layer_buffer(1)
    d_img.fill_(3)
    grid_to_image(plan, upload(junk), z_min, nl, box, d_img)
    img = download(d_img, np.complex64, (4, G, G))
    ref = sum(screens[k] * _centred(x[k, 2].astype(np.complex128), -1) for k in range(nl))
    e_to = rel_l2(img[2], ref)

    X = (rng.standard_normal((4, G, G)) + 1j * rng.standard_normal((4, G, G))).astype(np.complex64)
    d_X, d_lay = upload(X), dw.layer_buffer(nl)
    image_to_grid(plan, d_X, z_min, nl, box, d_lay)
    got = download(d_lay, np.complex64, (nl, 4, G, G))
    e_from = 0.0
    for k in range(nl):
        ref = _centred(X[1].astype(np.complex128) * np.conj(screens[k]), +1)
        e_from = max(e_from, rel_l2(got[k, 1, y0:y1, x0:x1], ref[y0:y1, x0:x1]))
    assert download(d_X, np.complex64, X.shape).tobytes() == X.tobytes()  # the image is only read

    d_box = upload(X)
    grid_fft_box(plan, d_box, 1, FFT_FORWARD, box)
    ref = _centred(X[3].astype(np.complex128), +1)
    e_box = rel_l2(download(d_box, np.complex64, X.shape)[3, y0:y1, x0:x1], ref[y0:y1, x0:x1])
    print(f"G={G} box {box}, {nl} layers, field {field}: to image {e_to:.2e}, to grid {e_from:.2e}, box {e_box:.2e}")
    assert e_to < TOL and e_from < TOL and e_box < TOL
