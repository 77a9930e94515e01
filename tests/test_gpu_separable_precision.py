"""The separable kernels' distance from 64 bits against the per-pair kernels' on the same data (IDGX_FLAG_PHASE_MFMA runs a
one-shot plan with those).  No larger, in the root mean square over the subgrids of a plan.

The bar on the ratio of the two is 1.02 for fp16x3: 1 and the noise of a root mean square over 48 subgrids, whose
distances differ among each other by less than a tenth.  The BF16 halves round independently in the two kernels, and with
few visibilities the ratio scatters by 3 %: 1.02 holds for its mean over all plans of the test."""
import numpy as np
import pytest

from helpers import oracle_degrid, oracle_grid, per_subgrid_rel_l2
from idgx import CHANNELS_DTYPE, FLAG_PHASE_MFMA, METADATA_DTYPE, observation
from idgx.device import DeviceWorkload, upload
from test_gpu_separable import corner_remainder

pytestmark = pytest.mark.gpu

IMAGE = 0.1
BAR = 1.02


def make(S, T, C, eps, spread_uv, n=48, seed=0):
    """n subgrids of T x C visibilities whose uv samples cover spread_uv of the subgrid, w spread so that the product
    term's phase at the corner goes up to eps."""
    rng = np.random.default_rng(seed)
    G, K = 2048, 4
    md, ch = np.zeros(n, METADATA_DTYPE), np.zeros(n, CHANNELS_DTYPE)
    ch["nr_channels"] = C
    md["time_offset"], md["nr_timesteps"] = np.arange(n) * T, T
    md["station1"], md["station2"] = np.arange(n) % K, (np.arange(n) + 1) % K
    md["x"], md["y"], md["z"] = rng.integers(0, G - S, n), rng.integers(0, G - S, n), rng.integers(-2, 3, n)
    k = np.linspace(3.3999, 3.4, C).astype(np.float32)
    half = (S // 2 - 4) / IMAGE * spread_uv
    centre = (np.stack([md["x"], md["y"]], 1) + S / 2 - G / 2) / IMAGE
    uvw = np.zeros((n, T, 3))
    uvw[..., :2] = centre[:, None] + rng.uniform(-half, half, (n, T, 2))
    spread = eps / (2 * np.pi * corner_remainder(S, IMAGE))
    uvw[..., 2] = rng.uniform(-spread, spread, (n, T))
    uvw[:, 0, 2], uvw[:, 1, 2] = -spread, spread
    uvw[..., 2] += rng.uniform(-500, 500, (n, 1))
    uvw = (uvw / (float(k[0]) / (2 * np.pi))).reshape(n * T, 3).astype(np.float32)
    return dict(uvw=uvw, wavenumbers=k, metadata=md, channels=ch, nr_subgrids=n, subgrid_size=S, grid_size=G,
                spheroidal=observation.prolate_spheroidal_taper(S), aterms=observation.jones_aterms(rng, 1, K, S),
                nr_stations=K, nr_aterm_slots=1, nr_rows=n * T, image_size=np.float32(IMAGE), w_step=0.0,
                max_nr_timesteps=T, visibilities=observation.random_visibilities(n * T, C, seed))


def ratios(w, form):
    """(gridder, degridder): the separable kernels' root-mean-square distance from 64 bits over the per-pair kernels'."""
    n, S = w["nr_subgrids"], w["subgrid_size"]
    rng = np.random.default_rng(5)
    sub = (rng.standard_normal((n, 4, S, S)) + 1j * rng.standard_normal((n, 4, S, S))).astype(np.complex64)
    g64, v64 = oracle_grid(w, fp64=True), oracle_degrid(w, sub, fp64=True)
    d, d_sub = DeviceWorkload(w), upload(sub)
    rms = []
    for flags in (0, FLAG_PHASE_MFMA):
        plan = d.plan(precision=form, flags=flags)
        d.grid(plan)
        d.degrid(plan, d_subgrids=d_sub)
        eg = per_subgrid_rel_l2(d.subgrids(), g64)
        ev = per_subgrid_rel_l2(d.visibilities_out().reshape(n, -1), v64.reshape(n, -1))
        rms.append([np.sqrt(np.mean(e.astype(np.float64) ** 2)) for e in (eg, ev)])
    r = np.array(rms[0]) / np.array(rms[1])
    print(f"S={S} {form}: gridder {rms[0][0]:.2e} / {rms[1][0]:.2e} = {r[0]:.3f}, "
          f"degridder {rms[0][1]:.2e} / {rms[1][1]:.2e} = {r[1]:.3f}")
    return r


@pytest.mark.parametrize("S", [16, 24, 32, 48])
@pytest.mark.parametrize("T, C", [(2, 2), (2, 4), (4, 4), (8, 4), (18, 4), (19, 4), (32, 4)])
@pytest.mark.parametrize("spread_uv", [0.05, 1.0])
def test_few_visibilities(S, T, C, spread_uv):
    """Subgrids of 4 to 128 visibilities, on both sides of the gridder's series phasors (72)."""
    w = make(S, T, C, 0.0, spread_uv, seed=S + T)
    assert (ratios(w, "fp16x3") <= BAR).all()


SIZES, SHAPES = (16, 24, 32, 40, 48, 64), ((2, 2), (4, 4), (64, 4))


def eps_values(S):
    """Without the product term (up to 1e-7) and just above that; in the middle of its range; at the limits of the gridder
    and of the degridder; past both, where the per-pair kernels run inside the call."""
    return dict(none=0.9e-7, some=3e-7, mid=1e-5, grid=0.97e-5 * S, degrid=0.97 * min(2.5e-5 * S, 1e-3),
                past=1.1e-3) | (dict(most=0.95e-3) if S < 40 else {})


@pytest.mark.parametrize("S", SIZES)
@pytest.mark.parametrize("T, C", SHAPES)
def test_product_term(S, T, C):
    for name, eps in eps_values(S).items():
        assert (ratios(make(S, T, C, eps, 1.0, seed=S + T), "fp16x3") <= BAR).all(), name


def test_product_term_bf16():
    r = [ratios(make(S, T, C, eps, 1.0, seed=S + T), "bf16x3")
         for S in SIZES for T, C in SHAPES for eps in eps_values(S).values()]
    mean = np.mean(r, axis=0)
    print(f"{len(r)} plans, mean ratio: gridder {mean[0]:.4f}, degridder {mean[1]:.4f}")
    assert (mean <= BAR).all()
