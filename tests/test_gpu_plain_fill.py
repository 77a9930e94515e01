"""The plain FP32 kernels on plans that leave CUs idle (one pixel, channel or visibility per thread) and on plans that do
not, at subgrid sizes whose last waves have fewer pixels than the others: batch and one-shot give the CPU restatement of the
reference to its FP32 rounding (the summation order is the same, the sine and cosine differ by 1.1e-7: 1e-5, the bar of every
plain form), and the gridders the same bits (the degridders fuse the A-term products of their pixels differently)."""
import numpy as np
import pytest

from helpers import oracle_degrid, oracle_grid, per_subgrid_rel_l2, rel_l2
from idgx import CHANNELS_DTYPE, METADATA_DTYPE, observation
from idgx.device import DeviceBatch, DeviceWorkload, upload

pytestmark = pytest.mark.gpu

PARITY = 1e-5


def make(S, n, T, C, seed):
    rng = np.random.default_rng(seed)
    G, K, image = 1024, 3, 0.05
    md, ch = np.zeros(n, METADATA_DTYPE), np.zeros(n, CHANNELS_DTYPE)
    md["time_offset"], md["nr_timesteps"] = np.arange(n) * T, rng.integers(0, T + 1, n)
    md["station1"], md["station2"] = rng.integers(0, K, n), rng.integers(0, K, n)
    md["x"], md["y"] = rng.integers(G // 2 - 40, G // 2 + 8, n), rng.integers(G // 2 - 40, G // 2 + 8, n)
    ch["channel_begin"] = rng.integers(0, C, n)
    ch["nr_channels"] = [int(rng.integers(1, C - c + 1)) for c in ch["channel_begin"]]
    uvw = rng.uniform(-150.0, 150.0, (n * T, 3)).astype(np.float32)
    uvw[:, 2] *= 0.1
    return dict(uvw=uvw, wavenumbers=np.linspace(3.1, 3.4, C).astype(np.float32), metadata=md, channels=ch, nr_subgrids=n,
                subgrid_size=S, grid_size=G, spheroidal=observation.prolate_spheroidal_taper(S),
                aterms=observation.jones_aterms(rng, 1, K, S), nr_stations=K, nr_aterm_slots=1, nr_rows=n * T,
                image_size=np.float32(image), w_step=0.0, max_nr_timesteps=T,
                visibilities=observation.random_visibilities(n * T, C, seed))


@pytest.mark.parametrize("S,n,T,C", [(8, 5, 9, 5), (20, 6, 40, 16), (24, 3, 90, 70), (28, 4, 33, 3), (40, 3, 21, 13),
                                     (64, 2, 17, 9), (20, 2100, 2, 3), (24, 2050, 2, 2), (40, 1040, 3, 2)])
def test_batch_equals_oneshot_and_the_cpu_restatement(S, n, T, C):
    w = make(S, n, T, C, S + n)
    rng = np.random.default_rng(1)
    sub = (rng.standard_normal((n, 4, S, S)) + 1j * rng.standard_normal((n, 4, S, S))).astype(np.complex64)
    d = DeviceWorkload(w)
    plan = d.plan()
    d.grid(plan)
    got = d.subgrids()
    d.degrid(plan, d_subgrids=upload(sub))
    vis = d.visibilities_out()
    eg, ev = per_subgrid_rel_l2(got, oracle_grid(w)).max(), rel_l2(vis, oracle_degrid(w, sub))
    print(f"S={S} n={n}: gridder worst {eg:.2e}, degridder {ev:.2e}")
    assert eg <= PARITY and ev <= PARITY
    b = DeviceBatch([w], precision="fp32")
    b.grid()
    same = np.array_equal(b.subgrids(), got) if C <= 64 else per_subgrid_rel_l2(b.subgrids(), got).max() <= PARITY
    b.classes[0]["d_subgrids"].copy_(upload(sub))
    b.degrid()
    eb = rel_l2(b.visibilities_out(), oracle_degrid(w, sub))
    assert same and eb <= PARITY and np.array_equal(b.visibilities_out() == 0, vis == 0)


@pytest.mark.parametrize("S,n,T,C", [(128, 1, 3, 1), (10, 2, 7, 2), (24, 2, 5, 64), (34, 2, 130, 4), (32, 64, 9, 3),
                                     (32, 65, 9, 3), (16, 2, 300, 6)])
def test_matrix_tiles_of_the_smallest_plans_give_the_bits_of_the_vector_form(S, n, T, C):
    """One-shot plans of at most a wave of 64 pixels per SIMD (two of 64 visibilities) run on the matrix cores, batches on
    the vector units: the same sums in the same order, also where channels, pixels or visibilities do not fill a step of
    four or a tile of 16.  Identity A-terms (Jones terms are fused differently in the degridders)."""
    w = make(S, n, T, C, 7 * S + n)
    w["aterms"] = observation.identity_aterms(1, 3, S)
    rng = np.random.default_rng(2)
    sub = (rng.standard_normal((n, 4, S, S)) + 1j * rng.standard_normal((n, 4, S, S))).astype(np.complex64)
    d = DeviceWorkload(w)
    plan = d.plan()
    d.grid(plan)
    got = d.subgrids()
    d.degrid(plan, d_subgrids=upload(sub))
    vis = d.visibilities_out()
    b = DeviceBatch([w], precision="fp32")
    b.grid()
    assert np.array_equal(b.subgrids(), got)
    b.classes[0]["d_subgrids"].copy_(upload(sub))
    b.degrid()
    assert np.array_equal(b.visibilities_out(), vis)
    assert per_subgrid_rel_l2(got, oracle_grid(w)).max() <= PARITY and rel_l2(vis, oracle_degrid(w, sub)) <= PARITY
