"""Subgrids that the separable kernels leave to the per-pair ones, because their w spreads too far, on every route of the
latter: inside a one-shot launch, behind it, in a batch's launch per class and in its merged launch, with every compiled
tile shape, with each class's own tiles, and in a captured graph.

Every workload holds subgrids of both kinds; that is asserted on the host from w and the product term's limits.

Bars: an FP32 phase of up to 16 turns per axis is off by at most 2 x 4.8e-7 turns and the sine and cosine by 1.1e-7, 7e-6
rad together; the FP16 halves add 2^-21, so 1e-5 for fp16x3.  The BF16 halves hold 16 bits of each factor: 2^-16 each on
top, so 4e-5."""
import numpy as np
import pytest

from helpers import oracle_degrid, oracle_grid, rel_l2
from idgx import CHANNELS_DTYPE, METADATA_DTYPE, observation
from idgx.device import DeviceWorkload, upload
from test_gpu_separable import corner_remainder

pytestmark = pytest.mark.gpu

BAR = {"fp16x3": 1e-5, "bf16x3": 4e-5}
PAST = 4e-3  # eps of the subgrids to be left: past every limit (1e-5 S, 2.5e-5 S, 1e-3, 4e-4)
WITHIN = 5e-5


def make(S, counts, left, image, C=9, seed=0, K=4, first_row=0):
    """Subgrids of counts[i] timesteps x a channel window each; w of those in `left` spreads to an eps of PAST, of the
    others to one of WITHIN."""
    rng = np.random.default_rng(seed)
    n, G = len(counts), 2048
    md, ch = np.zeros(n, METADATA_DTYPE), np.zeros(n, CHANNELS_DTYPE)
    k = np.linspace(3.39, 3.4, C).astype(np.float32)
    rows = int(sum(counts))
    uvw = np.zeros((rows, 3), np.float32)
    r = 0
    for i, T in enumerate(counts):
        md[i] = (0, first_row + r, T, 0, i % K, (i + 1) % K, *rng.integers(0, G - S, 2), 0)
        c0 = int(rng.integers(0, C - 1))
        ch[i] = (c0, int(rng.integers(1, C - c0 + 1)))
        centre = (np.array([md["x"][i], md["y"][i]]) + S / 2 - G / 2) / image
        half = max(1, S // 2 - 4) / image
        kc = float(k[c0]) / (2 * np.pi)
        uvw[r:r + T, :2] = (centre + rng.uniform(-half, half, (T, 2))) / kc
        spread = (PAST if i in left else WITHIN) / (2 * np.pi * corner_remainder(S, image))
        w = rng.uniform(-spread, spread, T)
        w[0], w[-1] = -spread, spread
        uvw[r:r + T, 2] = w / kc
        r += T
    return dict(uvw=uvw, wavenumbers=k, metadata=md, channels=ch, nr_subgrids=n, subgrid_size=S, grid_size=G,
                spheroidal=observation.prolate_spheroidal_taper(S), aterms=observation.jones_aterms(rng, 1, K, S),
                nr_stations=K, nr_aterm_slots=1, nr_rows=rows, image_size=np.float32(image), w_step=0.0,
                max_nr_timesteps=int(max(counts)), visibilities=observation.random_visibilities(rows, C, seed))


def largest_eps(w, first_row=0):
    """eps of every subgrid: the product term's phase at the corner for half its spread of w."""
    md, ch, k = w["metadata"], w["channels"], w["wavenumbers"].astype(np.float64) / (2 * np.pi)
    c = corner_remainder(w["subgrid_size"], float(w["image_size"]))
    out = []
    for s in range(md.size):
        r, c0 = int(md["time_offset"][s]) - first_row, int(ch["channel_begin"][s])
        x = w["uvw"][r:r + int(md["nr_timesteps"][s]), 2].astype(np.float64)
        p = np.outer([x.min(), x.max()], [k[c0], k[c0 + int(ch["nr_channels"][s]) - 1]])
        out.append(np.pi * (p.max() - p.min()) * c)
    return np.array(out)


def assert_both_kinds(w, left, first_row=0):
    eps = largest_eps(w, first_row)
    rest = [s for s in range(w["nr_subgrids"]) if s not in left]
    # Limits of a size: the gridder's 1e-5 S and 4e-4, the degridder's 1e-3 at most.
    assert left and (eps[list(left)] > 1e-3).all() and rest and (eps[rest] < 8e-5).all()


def model(w, seed=5):
    rng = np.random.default_rng(seed)
    S, n = w["subgrid_size"], w["nr_subgrids"]
    return (rng.standard_normal((n, 4, S, S)) + 1j * rng.standard_normal((n, 4, S, S))).astype(np.complex64)


def check(w, form, sub, grids, vis, first_row=0):
    """Every subgrid and its visibilities against FP64 (vis: the rows from first_row on)."""
    w = dict(w, metadata=w["metadata"].copy())
    w["metadata"]["time_offset"] -= first_row
    g64, v64 = oracle_grid(w, fp64=True), oracle_degrid(w, sub, fp64=True)
    md, ch = w["metadata"], w["channels"]
    worst = [0.0, 0.0]
    for s in range(md.size):
        r, c = int(md["time_offset"][s]), int(ch["channel_begin"][s])
        at = slice(r, r + int(md["nr_timesteps"][s])), slice(c, c + int(ch["nr_channels"][s]))
        worst[0] = max(worst[0], rel_l2(grids[s], g64[s]))
        worst[1] = max(worst[1], rel_l2(vis[at], v64[at]))
    print(f"S={w['subgrid_size']} {form}: gridder worst {worst[0]:.2e}, degridder worst {worst[1]:.2e}")
    assert worst[0] <= BAR[form] and worst[1] <= BAR[form]


@pytest.mark.parametrize("form", ["fp16x3", "bf16x3"])
@pytest.mark.parametrize("S, image", [(16, 0.05), (16, 0.12), (24, 0.1), (32, 0.06), (32, 0.16), (40, 0.1), (64, 0.06),
                                      (64, 0.12)])
@pytest.mark.parametrize("n", [6, 262])
def test_one_shot(S, image, n, form):
    """Fields whose one-shot calls take one launch (0.05, 0.06) and two; workgroups of 8 columns and of whole subgrids;
    subgrids of few and many visibilities of both kinds."""
    rng = np.random.default_rng(S + n)
    counts = [int(t) for t in rng.integers(2, 40, n)]
    left = set(range(1, n, 3))
    w = make(S, counts, left, image, seed=S)
    assert_both_kinds(w, left)
    sub = model(w)
    d = DeviceWorkload(w)
    plan = d.plan(precision=form)
    d.grid(plan)
    got = d.subgrids()
    d.degrid(plan, d_subgrids=upload(sub))
    check(w, form, sub, got, d.visibilities_out())


# ---- batches of three classes over one set of rows -----------------------------------------------------------------

SIZES = (24, 32, 48)


def make_classes(lefts, seed=0):
    """Classes of SIZES, lefts[k] the subgrids to be left in class k; every class carries the shared rows."""
    classes, first = [], 0
    rng = np.random.default_rng(seed)
    for k, S in enumerate(SIZES):
        w = make(S, [int(t) for t in rng.integers(2, 60, 12)], lefts[k], 0.1, seed=seed + k, first_row=first)
        if lefts[k]:
            assert_both_kinds(w, lefts[k], first)
        else:
            assert (largest_eps(w, first) < 8e-5).all()
        classes.append(dict(w, first_row=first, own_rows=w["nr_rows"]))
        first += w["nr_rows"]
    uvw = np.concatenate([w["uvw"] for w in classes])
    vis = np.concatenate([w["visibilities"] for w in classes])
    for w in classes:
        w["own_uvw"], w["own_vis"] = w["uvw"], w["visibilities"]
        w.update(uvw=uvw, visibilities=vis, nr_rows=first)
    return classes


def own(w):
    """A class with its own rows only, for the oracle."""
    return dict(w, uvw=w["own_uvw"], visibilities=w["own_vis"], nr_rows=w["own_rows"])


def three_classes(form, lefts=({1, 4, 7}, {0, 2, 9, 11}, {3, 5})):
    from idgx import Batch
    from idgx.device import DeviceBatch

    classes = make_classes(lefts)
    d = DeviceBatch(classes, precision=form)
    models = [model(w, seed=k) for k, w in enumerate(classes)]
    # The model subgrids are buffers of their own: the gridder writes the classes'.
    d.models = [upload(m) for m in models]
    d.predict = Batch.data(d.d_uvw, d.d_wavenumbers, d.d_visibilities, d.d_vis_out,
                           [dict(c, d_subgrids=m) for c, m in zip(d.classes, d.models)])
    return d, classes, models


def run(d):
    for c in d.classes:
        c["d_subgrids"].zero_()
    d.d_vis_out.zero_()
    d.grid()
    d.batch.degrid(d.predict)
    return [d.subgrids(k) for k in range(len(d.classes))], d.visibilities_out()


def check_classes(classes, models, form, grids, vis):
    for k, w in enumerate(classes):
        rows = slice(w["first_row"], w["first_row"] + w["own_rows"])
        check(own(w), form, models[k], grids[k], vis[rows], w["first_row"])


def test_autotuner_leaves_the_shapes_of_classes_without_leftovers():
    """Their persistent launch finds no work, so its time says nothing about a shape."""
    for lefts, kept in ((({1, 4}, set(), {3}), (1,)), ((set(), set(), set()), (0, 1, 2))):
        d, classes, models = three_classes("fp16x3", lefts)
        shape = len(d.batch.shapes()) - 3
        d.batch.set_single_launch(-1, -1)
        d.batch.set_shape(shape, shape)
        tg, td = d.batch.autotune(d.data, repeats=1)
        assert tg > 0 and td > 0 and d.batch.single_launch() == (-1, -1)
        for k in kept:
            assert d.batch.class_shape(k) == (shape, shape)
        if len(kept) == 3:
            d.batch.set_single_launch(shape, shape)
            tg, td = d.batch.autotune(d.data, repeats=1)
            assert tg > 0 and td > 0 and d.batch.single_launch() == (shape, shape)
        check_classes(classes, models, "fp16x3", *run(d))


def assert_same_bits(a, b):
    assert all(x.tobytes() == y.tobytes() for x, y in zip(a[0], b[0])) and a[1].tobytes() == b[1].tobytes()


@pytest.mark.parametrize("form", ["fp16x3", "bf16x3"])
def test_every_tile_shape_per_class_and_merged(form):
    """Each compiled shape as a launch per class and as the merged launch, whose items write the same bits."""
    d, classes, models = three_classes(form)
    for shape in range(len(d.batch.shapes())):
        d.batch.set_single_launch(-1, -1)
        d.batch.set_shape(shape, shape)
        per_class = run(d)
        assert d.batch.last_launches() == (3, 3)
        check_classes(classes, models, form, *per_class)
        d.batch.set_single_launch(shape, shape)
        merged = run(d)
        assert d.batch.last_launches() == (1, 1)
        assert_same_bits(per_class, merged)


@pytest.mark.parametrize("form", ["fp16x3", "bf16x3"])
def test_tiles_per_class(form):
    """Every compiled count of tiles per wave for each class in turn, merged with each class's own against launches per
    class."""
    from idgx import SHAPE_TILES_PER_CLASS

    d, classes, models = three_classes(form)
    shapes = d.batch.shapes()
    tiles = [shapes.index((t, 256, 0)) for t in (2, 3, 4, 6, 8)]
    degrid = shapes.index((4, 256, 0))
    for i in range(len(tiles)):
        for k in range(3):
            d.batch.set_class_shape(k, tiles[(i + k) % len(tiles)], degrid)
        d.batch.set_single_launch(-1, -1)
        per_class = run(d)
        d.batch.set_single_launch(SHAPE_TILES_PER_CLASS, degrid)
        merged = run(d)
        assert_same_bits(per_class, merged)
        check_classes(classes, models, form, *merged)


@pytest.mark.parametrize("merged", [False, True])
@pytest.mark.parametrize("lefts", [({1, 4, 7}, {0, 2, 9, 11}, {3, 5}), (set(), {0, 2, 9, 11}, set())])
def test_graph_replays(lefts, merged):
    """Capture with leftovers in every class and in one; replays on fresh outputs, with eager work between them."""
    import torch

    from idgx import SHAPE_TILES_PER_CLASS, STAGE_DEGRID, STAGE_GRID

    d, classes, models = three_classes("fp16x3", lefts)
    if merged:
        d.batch.set_single_launch(SHAPE_TILES_PER_CLASS, d.batch.shapes().index((4, 256, 0)))
    else:
        d.batch.set_single_launch(-1, -1)
    eager = run(d)
    check_classes(classes, models, "fp16x3", *eager)
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    for stage, data, read in ((STAGE_GRID, d.data, lambda: [d.subgrids(k) for k in range(3)]),
                              (STAGE_DEGRID, d.predict, d.visibilities_out)):
        d.batch.capture(data, stage, stream)
        for r in range(3):
            for c in d.classes:
                c["d_subgrids"].zero_()
            d.d_vis_out.zero_()
            torch.cuda.synchronize()
            d.batch.launch(stream)
            stream.synchronize()
            got = read()
            if stage == STAGE_GRID:
                assert all(x.tobytes() == y.tobytes() for x, y in zip(got, eager[0])), f"replay {r}"
            else:
                assert got.tobytes() == eager[1].tobytes(), f"replay {r}"
            assert float(torch.ones(1000, device="cuda").sum()) == 1000.0


def test_leftovers_come_and_go_with_the_data():
    """The same batch on data with other leftovers: nothing of the previous pass's marks remains."""
    d, classes, models = three_classes("fp16x3")
    first = run(d)
    calm = [dict(c) for c in make_classes((set(), {2}, set()), seed=0)]
    # Same counts, windows and rows: only uvw changes.
    assert all((a["metadata"] == b["metadata"]).all() for a, b in zip(calm, classes))
    keep = d.d_uvw.clone()
    d.d_uvw.copy_(upload(calm[0]["uvw"]))
    check_classes([dict(c, own_vis=w["own_vis"]) for c, w in zip(calm, classes)], models, "fp16x3", *run(d))
    d.d_uvw.copy_(keep)
    assert_same_bits(first, run(d))
