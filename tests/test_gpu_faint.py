"""The FP16 forms on data whose power-of-two scale would leave the range of a float: models and visibilities around 1e-36
(2^-120), whose scale of 2^-134 has no finite inverse.  One-shot and batch, in the separable kernels (S <= 64; 20 leaves
padded rows and columns) and the per-pair ones (S = 66).

Tolerance: the separable kernels' 1e-5 for FP16 halves at a normal scale.  Here the largest value is scaled to 2^6 or more
instead of 2^14; the low halves then end at FP16's 2^-25, 2^-31 of it, and the outputs at float's 2^-150, which add
nothing to 1e-5."""
import numpy as np
import pytest

from helpers import oracle_degrid, oracle_grid, rel_l2
from idgx import Batch, observation
from idgx.device import DeviceBatch, DeviceWorkload, upload

pytestmark = pytest.mark.gpu

SCALE = 2.0 ** -120


def _workload(S):
    w = observation.subset(observation.make_observation("small"), np.arange(6))
    w.update(subgrid_size=S, spheroidal=observation.prolate_spheroidal_taper(S),
             aterms=observation.identity_aterms(1, w["nr_stations"], S))
    w["visibilities"] = observation.random_visibilities(w["nr_rows"], w["wavenumbers"].size, 7)
    rng = np.random.default_rng(8)
    sub = rng.standard_normal((6, 4, S, S)) + 1j * rng.standard_normal((6, 4, S, S))
    return w, sub.astype(np.complex64)


@pytest.mark.parametrize("S", [20, 32, 66])
@pytest.mark.parametrize("api", ["oneshot", "batch"])
def test_faint_data_in_fp16_vs_fp64(api, S):
    w, sub = _workload(S)
    g64, v64 = oracle_grid(w, fp64=True), oracle_degrid(w, sub, fp64=True)
    faint = dict(w, visibilities=w["visibilities"] * np.float32(SCALE))
    d_sub = upload(sub * np.float32(SCALE))
    if api == "oneshot":
        d = DeviceWorkload(faint)
        plan = d.plan(precision="fp16x3")
        d.grid(plan)
        got = d.subgrids()
        d.degrid(plan, d_subgrids=d_sub)
    else:
        d = DeviceBatch([faint], precision="fp16x3")
        d.grid()
        got = d.subgrids()
        d.batch.degrid(Batch.data(d.d_uvw, d.d_wavenumbers, d.d_visibilities, d.d_vis_out,
                                  [dict(d.classes[0], d_subgrids=d_sub)]))
    vis = d.visibilities_out()
    assert np.isfinite(got).all() and np.isfinite(vis).all()
    eg, ev = rel_l2(got.astype(np.complex128) / SCALE, g64), rel_l2(vis.astype(np.complex128) / SCALE, v64)
    print(f"{api} S={S} at 2^-120: gridder {eg:.2e}, degridder {ev:.2e}")
    assert eg <= 1e-5 and ev <= 1e-5
