"""The plain FP32 kernels on plans that fill the chip: three and four pixels per thread in the one-shot gridder (large
subgrids, and the accurate sine and cosine from 32^2), batches whose gridder items all have their pixels and batches whose
last items do not, and batches of few visibilities a subgrid (one visibility per thread, and default gridder items where
finer ones would only lengthen the queue).  Bars as for the smaller plans: 1e-5 of the CPU restatement, and the gridders
the same bits."""
import numpy as np
import pytest

from helpers import oracle_degrid, oracle_grid, per_subgrid_rel_l2, rel_l2
from idgx import FLAG_ACCURATE_SINCOS
from idgx.device import DeviceBatch, DeviceWorkload, upload
from test_gpu_plain_fill import PARITY, make

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,n,T,C", [
    (72, 300, 3, 2),    # three pixels per thread, the last block's last waves without any
    (88, 270, 2, 3),    # the same with a ragged last wave
    (96, 230, 3, 2),    # three, whole
    (128, 140, 2, 2),   # four, whole
    (32, 2100, 2, 2),   # whole items of four in the batch
    (48, 1100, 2, 2),   # whole items of three
    (26, 2200, 2, 3),   # ragged items
    (32, 700, 4, 3),    # few visibilities: default items although they do not fill the chip
    (16, 1300, 9, 40),  # more than 256 visibilities in some subgrids, fewer in most
])
def test_batch_equals_oneshot_and_the_cpu_restatement(S, n, T, C):
    w = make(S, n, T, C, S + n)
    rng = np.random.default_rng(1)
    sub = (rng.standard_normal((n, 4, S, S)) + 1j * rng.standard_normal((n, 4, S, S))).astype(np.complex64)
    g32, v32 = oracle_grid(w), oracle_degrid(w, sub)
    d = DeviceWorkload(w)
    d_sub = upload(sub)
    for flags in (0, FLAG_ACCURATE_SINCOS):
        plan = d.plan(flags=flags)
        d.grid(plan)
        d.degrid(plan, d_subgrids=d_sub)
        got, vis = d.subgrids(), d.visibilities_out()
        eg, ev = per_subgrid_rel_l2(got, g32).max(), rel_l2(vis, v32)
        print(f"S={S} n={n} flags {flags}: gridder worst {eg:.2e}, degridder {ev:.2e}")
        assert eg <= PARITY and ev <= PARITY
        if not flags:
            hw = got
    b = DeviceBatch([w], precision="fp32")
    b.grid()
    assert np.array_equal(b.subgrids(), hw)
    b.classes[0]["d_subgrids"].copy_(d_sub)
    b.degrid()
    assert rel_l2(b.visibilities_out(), v32) <= PARITY and np.array_equal(b.visibilities_out() == 0, v32 == 0)
