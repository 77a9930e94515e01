"""Adder, splitter and subgrid FFT at the edges of their work split: residues that do not fill a workgroup, tile lists
around the adder's steps of 8, 4 and 2 and its staging of 256, tiles larger than the subgrid, subgrids inside, across and
outside the grid's edges, and subgrid counts on both sides of the splitter's runs of 8 x 64.  Integer-valued data: exact."""
import numpy as np
import pytest

import oracle
from idgx import METADATA_DTYPE, AdderPlan, add_subgrids, observation
from idgx.device import DeviceWorkload, download, upload

pytestmark = pytest.mark.gpu


def _device_workload(S, G, md):
    return DeviceWorkload(dict(
        metadata=md, channels=None, subgrid_size=S, grid_size=G, nr_stations=2, nr_aterm_slots=1,
        image_size=np.float32(0.1), w_step=0.0, wavenumbers=np.full(1, 3.0, np.float32),
        uvw=np.zeros((1, 3), np.float32), visibilities=np.zeros((1, 1, 4), np.complex64),
        spheroidal=np.ones((S, S), np.float32), aterms=observation.identity_aterms(1, 2, S), max_nr_timesteps=1,
        nr_subgrids=md.size))


def _metadata(rng, n, S, G, pile):
    md = np.zeros(n, METADATA_DTYPE)
    md["nr_timesteps"] = 1
    md["station2"] = 1
    md["x"] = rng.integers(-S - 2, G + 2, n)
    md["y"] = rng.integers(-S - 2, G + 2, n)
    # One tile with `pile` subgrids at different places of it, spread over the plan.
    at = rng.permutation(n)[:pile]
    md["x"][at] = S + rng.integers(0, S, pile)
    md["y"][at] = S + rng.integers(0, S, pile)
    return md


def _plan_of_tiles(md, T, G):
    """An adder plan with tiles of T cells: (plan, order, tile_start) as the library's own builder lays them out."""
    n_axis = G // T + 3
    tx, ty = np.floor_divide(md["x"], T) + 1, np.floor_divide(md["y"], T) + 1
    colour = ((tx - 1) & 1) + 2 * ((ty - 1) & 1)
    key = (colour * n_axis + np.clip(ty, 0, n_axis - 1)) * n_axis + np.clip(tx, 0, n_axis - 1)
    order = np.argsort(key, kind="stable").astype(np.int32)
    first = np.flatnonzero(np.r_[True, np.diff(key[order]) != 0])
    tile_start = np.r_[first, md.size].astype(np.int32)
    ap = AdderPlan()
    ap.tile_size, ap.nr_tiles, ap.nr_layers = T, first.size, 1
    ap.color_begin[:] = [int(np.searchsorted(colour[order][first], c)) for c in range(5)]
    return ap, order, tile_start


@pytest.mark.parametrize("S, G, n, pile", [(8, 64, 40, 3), (20, 128, 100, 9), (24, 128, 300, 257), (32, 256, 511, 8),
                                           (32, 256, 1100, 600), (48, 128, 64, 21), (128, 256, 20, 6)])
def test_adder_and_splitter_are_exact_at_the_edges_of_their_split(S, G, n, pile):
    rng = np.random.default_rng(S + n)
    md = _metadata(rng, n, S, G, pile)
    sub = (rng.integers(-8, 9, (n, 4, S, S)) + 1j * rng.integers(-8, 9, (n, 4, S, S))).astype(np.complex64)
    start = (rng.integers(-8, 9, (4, G, G)) + 1j * rng.integers(-8, 9, (4, G, G))).astype(np.complex64)
    want = start + oracle.adder_fp64(md, sub, G).astype(np.complex64)
    dw = _device_workload(S, G, md)
    plan = dw.plan()
    d_sub, d_md = upload(sub), upload(md)
    dw.d_subgrids.copy_(d_sub)
    d_grid = upload(start)
    dw.add(plan, d_grid)
    np.testing.assert_array_equal(download(d_grid, np.complex64, start.shape), want)
    for T in (S + 6, 2 * S):  # a caller's own plan, with tiles larger than the subgrid
        ap, order, tile_start = _plan_of_tiles(md, T, G)
        d_grid = upload(start)
        add_subgrids(plan, ap, d_md, upload(order), upload(tile_start), d_sub, d_grid)
        np.testing.assert_array_equal(download(d_grid, np.complex64, start.shape), want)
    dw.split(plan, upload(start))
    np.testing.assert_array_equal(dw.subgrids(), oracle.splitter_fp64(md, start, S).astype(np.complex64))
