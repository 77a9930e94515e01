"""Calls whose scratch buffers are separate run on two streams at once: grid_to_image beside a master-grid transform of the
same size.  Every result equals the one of the same call by itself, bit for bit."""
import numpy as np
import pytest

from idgx import FFT_BACKWARD, grid_fft, grid_to_image, make_plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nr_layers, w_step", [(1, 0.0), (2, 300.0)])
def test_grid_to_image_beside_a_transform_on_another_stream(nr_layers, w_step):
    import torch

    G, box = 1024, (100, 900, 30, 1000)
    plan = make_plan(nr_subgrids=0, subgrid_size=32, grid_size=G, nr_channels=1, nr_stations=2, nr_aterm_slots=1,
                     nr_rows=1, max_nr_timesteps=1, image_size=0.1, w_step=w_step)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(1)

    def planes(n):
        return torch.randn(n * 4 * G * G * 2, device="cuda", generator=gen).view(torch.complex64).reshape(n, 4, G, G)

    grids, fields = planes(nr_layers), planes(1)
    x0, x1, y0, y1 = box
    outside = torch.ones(G, G, dtype=torch.bool, device="cuda")
    outside[y0:y1, x0:x1] = False
    grids[..., outside] = 0

    image, field = torch.empty((4, G, G), dtype=torch.complex64, device="cuda"), fields.clone()
    grid_to_image(plan, grids.clone(), 0, nr_layers, box, image)
    grid_fft(plan, field, 1, FFT_BACKWARD)
    torch.cuda.synchronize()

    repeats = 20
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    sources = [grids.clone() for _ in range(repeats)]
    images = [torch.empty_like(image) for _ in range(repeats)]
    work = [fields.clone() for _ in range(repeats)]
    torch.cuda.synchronize()
    for i in range(repeats):
        grid_to_image(plan, sources[i], 0, nr_layers, box, images[i], a)
        grid_fft(plan, work[i], 1, FFT_BACKWARD, b)
    torch.cuda.synchronize()
    for i in range(repeats):
        assert np.array_equal(images[i].cpu().numpy().view(np.uint64), image.cpu().numpy().view(np.uint64)), i
        assert np.array_equal(work[i].cpu().numpy().view(np.uint64), field.cpu().numpy().view(np.uint64)), i
