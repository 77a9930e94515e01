"""The separable forms of the fp16x3 / bf16x3 gridder and degridder against the FP64 oracle, at the edges of their
dispatch: every row and column tile of the subgrid sizes, plans with fewer and more subgrids than CUs, visibility counts
around the chunk sizes, and spreads of w that take them without the product term, with it, and to the per-pair kernels.

Bars: an FP32 phase of up to 16 turns per axis is off by at most 2 x 4.8e-7 turns and the sine and cosine by 1.1e-7, 7e-6
rad together; the FP16 halves add 2^-21, so 1e-5 for fp16x3.  The BF16 halves hold 16 bits of each factor: 2^-16 each on
top, so 4e-5."""
import numpy as np
import pytest

from helpers import oracle_degrid, oracle_grid, rel_l2
from idgx import CHANNELS_DTYPE, METADATA_DTYPE, observation
from idgx.device import DeviceBatch, DeviceWorkload, selection_lists, upload

pytestmark = pytest.mark.gpu

BAR = {"fp16x3": 1e-5, "bf16x3": 4e-5}
IMAGE = 0.1


def corner_remainder(S, image=IMAGE):
    """n(l, m) minus its additive part at the subgrid's corner pixel."""
    lm = (0.5 - 0.5 / S) * image
    l0 = lm * np.sqrt(0.5)

    def n(l, m):
        return (l * l + m * m) / (1 + np.sqrt(1 - l * l - m * m))

    return n(lm, lm) - 2 * (n(lm, l0) - n(l0, l0) / 2)


def make(S, counts, eps, seed=0, C=9, w_step=0.0):
    """Subgrids of counts[i] timesteps x a channel window each, their uv samples within the subgrid and w spread so that
    the product term's largest phase at the corner is about eps[i] radians."""
    rng = np.random.default_rng(seed)
    n, G, K = len(counts), 2048, 4
    md, ch = np.zeros(n, METADATA_DTYPE), np.zeros(n, CHANNELS_DTYPE)
    k = np.linspace(3.1, 3.4, C).astype(np.float32)
    rows = int(sum(counts))
    uvw = np.zeros((rows, 3), np.float32)
    r = 0
    for i, T in enumerate(counts):
        md[i] = (0, r, T, i % 2, i % K, (i + 1) % K, *rng.integers(0, G - S, 2), int(rng.integers(-2, 3)))
        c0 = int(rng.integers(0, C - 1))
        ch[i] = (c0, int(rng.integers(1, C - c0 + 1)))
        centre = (np.array([md["x"][i], md["y"][i]]) + S / 2 - G / 2) / IMAGE
        half = max(1, S // 2 - 4) / IMAGE
        kc = float(k[c0]) / (2 * np.pi)
        uvw[r:r + T, :2] = (centre + rng.uniform(-half, half, (T, 2))) / kc
        # The channels spread w by their own ratio; the rows add the rest.
        spread = eps[i] / (2 * np.pi * corner_remainder(S))
        mid = (md["z"][i] + 0.5) * w_step + (spread if eps[i] else 0.0)
        uvw[r:r + T, 2] = (mid + rng.uniform(-spread, spread, T)) / kc
        r += T
    return dict(uvw=uvw, wavenumbers=k, metadata=md, channels=ch, nr_subgrids=n, subgrid_size=S, grid_size=G,
                spheroidal=observation.prolate_spheroidal_taper(S),
                aterms=observation.jones_aterms(rng, 2, K, S), nr_stations=K, nr_aterm_slots=2, nr_rows=rows,
                image_size=np.float32(IMAGE), w_step=w_step, max_nr_timesteps=int(max(counts)),
                visibilities=observation.random_visibilities(rows, C, seed))


def model(w, seed=5):
    rng = np.random.default_rng(seed)
    S, n = w["subgrid_size"], w["nr_subgrids"]
    return (rng.standard_normal((n, 4, S, S)) + 1j * rng.standard_normal((n, 4, S, S))).astype(np.complex64)


def windows(w):
    md, ch = w["metadata"], w["channels"]
    for s in range(md.size):
        r, c = int(md["time_offset"][s]), int(ch["channel_begin"][s])
        yield slice(r, r + int(md["nr_timesteps"][s])), slice(c, c + int(ch["nr_channels"][s]))


def check(w, form, sub_in, grids, vis, mask=None):
    """Every subgrid and every subgrid's visibilities against FP64; uncovered visibilities untouched."""
    w64 = w if mask is None else dict(w, visibilities=np.where(mask[..., None], 0, w["visibilities"]))
    g64, v64 = oracle_grid(w64, fp64=True), oracle_degrid(w, sub_in, fp64=True)
    worst = [0.0, 0.0]
    for s, (r, c) in enumerate(windows(w)):
        worst[0] = max(worst[0], rel_l2(grids[s], g64[s]))
        keep = np.ones(v64[r, c].shape[:2], bool) if mask is None else ~mask[r, c]
        if keep.any():
            worst[1] = max(worst[1], rel_l2(vis[r, c][keep], v64[r, c][keep]))
    covered = np.zeros(vis.shape[:2], bool)
    for r, c in windows(w):
        covered[r, c] = True
    if mask is not None:
        covered &= ~mask
    assert not np.any(vis[~covered])
    print(f"S={w['subgrid_size']} {form}: gridder worst {worst[0]:.2e}, degridder worst {worst[1]:.2e}")
    assert worst[0] <= BAR[form] and worst[1] <= BAR[form]


def run_oneshot(w, form, sub_in):
    d = DeviceWorkload(w)
    plan = d.plan(precision=form)
    d.grid(plan)
    got = d.subgrids()
    d.degrid(plan, d_subgrids=upload(sub_in))
    return got, d.visibilities_out()


def run_batch(w, form, sub_in):
    d = DeviceBatch([w], precision=form)
    d.grid()
    got = d.subgrids()
    d.classes[0]["d_subgrids"].copy_(upload(sub_in))
    d = _rebind(d)
    d.degrid()
    return got, d.visibilities_out()


def _rebind(d):
    from idgx import Batch

    d.data = Batch.data(d.d_uvw, d.d_wavenumbers, d.d_visibilities, d.d_vis_out, d.classes)
    return d


EDGES = (1, 2, 7, 8, 9, 15, 29, 40)


@pytest.mark.parametrize("form", ["fp16x3", "bf16x3"])
@pytest.mark.parametrize("S", [8, 10, 16, 18, 24, 26, 32, 34, 40, 48, 50, 64])
def test_every_tile_with_few_subgrids_vs_fp64(S, form):
    """Without and with the product term, one-shot and batch (the same bits)."""
    w = make(S, EDGES, [0.0, 1e-4, 5e-4, 1e-6, 0.0, 2e-4, 8e-4, 3e-4], w_step=40.0)
    sub = model(w)
    got, vis = run_oneshot(w, form, sub)
    check(w, form, sub, got, vis)
    bgot, bvis = run_batch(w, form, sub)
    assert np.array_equal(got, bgot) and np.array_equal(vis, bvis)


@pytest.mark.parametrize("S", [12, 24, 32, 40, 64])
def test_more_subgrids_than_cus_vs_fp64(S):
    """The wide column tiles of plans that fill the chip, with flagged data and empty subgrids."""
    rng = np.random.default_rng(S)
    counts = [int(t) for t in rng.integers(1, 12, 270)]
    w = make(S, counts, list(rng.uniform(0.0, 8e-4, 270)), seed=S)
    w["channels"]["nr_channels"][7] = 0
    flags = rng.random((w["nr_rows"], w["wavenumbers"].size)) < 0.3
    w["vis_index"], w["vis_offset"] = selection_lists(w, flags)
    sub = model(w)
    got, vis = run_batch(w, "fp16x3", sub)
    check(w, "fp16x3", sub, got, vis, flags)


@pytest.mark.parametrize("S", [16, 32, 48, 64])
@pytest.mark.parametrize("form", ["fp16x3", "bf16x3"])
def test_subgrids_outside_the_product_term_take_the_per_pair_kernels(S, form):
    """Spreads of w past the term's range beside ones inside it: the per-pair item inside the one-shot call, the
    per-pair launch of a batch; three replays of a batch on fresh outputs give the same bits."""
    w = make(S, (60, 33, 5, 40, 12), [5e-3, 3e-4, 8e-3, 0.0, 2e-3], seed=3)
    sub = model(w)
    check(w, form, sub, *run_oneshot(w, form, sub))
    first = run_batch(w, form, sub)
    check(w, form, sub, *first)
    for _ in range(2):
        again = run_batch(w, form, sub)
        assert np.array_equal(first[0], again[0]) and np.array_equal(first[1], again[1])


@pytest.mark.parametrize("S", [14, 24, 32])
def test_plans_between_eight_wave_workgroups_and_full_chips_vs_fp64(S):
    """150 subgrids: a workgroup of four waves per 8 columns, where 8 subgrids take eight waves and 270 all columns."""
    rng = np.random.default_rng(100 + S)
    w = make(S, [int(t) for t in rng.integers(1, 30, 150)], list(rng.uniform(0.0, 8e-4, 150)), seed=S)
    sub = model(w)
    got, vis = run_oneshot(w, "fp16x3", sub)
    check(w, "fp16x3", sub, got, vis)
