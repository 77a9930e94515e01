"""The kernels that bench.py names for a pass are the ones the library launches: the committed profiles have their rows."""
import importlib.util
import os

import numpy as np
import pytest

from idgx import make_plan, observation, oneshot_plain_shape, plain_kernel_shape, separable_shape

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def bench():
    spec = importlib.util.spec_from_file_location("bench_module", os.path.join(ROOT, "bench.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def _plan(S, n, precision="fp16x3", image=0.1, T=128, C=64, flags=0):
    return make_plan(nr_subgrids=n, subgrid_size=S, grid_size=4096, nr_channels=C, nr_stations=8, nr_aterm_slots=1,
                     nr_rows=T, max_nr_timesteps=T, image_size=image, precision=precision, flags=flags)


@pytest.mark.parametrize("config", ["ska_low", "full_cycle"])
def test_pass_kernels_of_the_configurations_are_profiled(bench, config):
    c = observation.CONFIGS[config]
    plan = _plan(c["subgrid_size"], 70000, image=c["image_size"], T=c["timesteps_per_subgrid"], C=c["n_channels"])
    plain = _plan(c["subgrid_size"], 70000, "fp32", c["image_size"], c["timesteps_per_subgrid"], c["n_channels"])
    for direction in ("gridder", "degridder"):
        for path in ("one-shot", "batched"):
            key = bench.pass_kernel("fp16x3", path, direction, (4, 256, 0), [plan], [1000])
            assert "separable" in key
            assert bench.measured_traffic(config, key)["bytes"] > 1e9, key
            pipes = bench.pipe_profile(config, key)
            assert pipes is not None and pipes["SQ_INSTS_MFMA"] > 1e8, key
        key = bench.pass_kernel("fp32", "one-shot", direction, None, [plain], [1000],
                                oneshot_plain_shape(plain, True))
        assert bench.measured_traffic(config, key) is not None, key
        key = bench.pass_kernel("fp32", "batched", direction, [(4, 2, True)], [plain], [1000])
        assert bench.measured_traffic(config, key) is not None, key


def test_several_classes_sum_their_kernels(bench):
    plans = [_plan(S, 400000, image=0.1) for S in (24, 32, 48)]
    for direction in ("gridder", "degridder"):
        key = bench.pass_kernel("fp16x3", "batched", direction, "tiles per class", plans, [1000] * 3)
        parts = key.split(" + ")
        assert len(parts) == 3
        one = [bench.measured_traffic("batched_uneven", k)["bytes"] for k in parts]
        assert bench.measured_traffic("batched_uneven", key)["bytes"] == pytest.approx(sum(one))
        busy = [bench.pipe_profile("batched_uneven", k)["MfmaUtil"] for k in parts]
        assert min(busy) <= bench.pipe_profile("batched_uneven", key)["MfmaUtil"] <= max(busy)


def test_separable_shape_follows_the_limits():
    assert separable_shape(_plan(32, 1000), True, 1000) == (1, 2, 4, 1, 4, 1)
    assert separable_shape(_plan(32, 1000), True, 60) == (1, 2, 4, 1, 4, 2)  # FP16, few visibilities
    assert separable_shape(_plan(32, 1000, "bf16x3"), True, 60) == (0, 2, 4, 1, 4, 0)
    assert separable_shape(_plan(32, 10), True, 1000) == (1, 2, 1, 1, 8, 0)
    assert separable_shape(_plan(64, 1000), False, 1000) == (1, 4, 2, 8)
    for plan in (_plan(66, 1000), _plan(32, 1000, "fp32"), _plan(32, 1000, "fp16"), _plan(32, 1000, image=0.3),
                 _plan(32, 0), _plan(32, 1000, flags=2)):
        assert separable_shape(plan, True, 1000) == () and separable_shape(plan, False, 1000) == ()


def test_oneshot_plain_shape_of_small_and_large_plans():
    assert oneshot_plain_shape(_plan(32, 4, "fp32", T=8, C=4), False) == (0, 0)
    assert oneshot_plain_shape(_plan(32, 70000, "fp32"), True) == (1, 2)
    for S, n in ((96, 4000), (72, 4000), (24, 70000)):
        px, nch = oneshot_plain_shape(_plan(S, n, "fp32"), False)
        assert px in (1, plain_kernel_shape(_plan(S, n, "fp32"), False)[0]) and nch == 4


def _batch(idgx, S, n, V, precision):
    md = np.zeros(n, idgx.METADATA_DTYPE)
    md["nr_timesteps"] = 1
    md["station2"] = 1
    plan = make_plan(nr_subgrids=n, subgrid_size=S, grid_size=1024, nr_channels=V, nr_stations=2, nr_aterm_slots=1,
                     nr_rows=1, max_nr_timesteps=1, image_size=0.05, precision=precision)
    return idgx.Batch([(plan, md, None, None)])


@pytest.mark.gpu
def test_batch_plain_work():
    import idgx

    b = _batch(idgx, 32, 8, 16, "fp32")  # too few items for the chip
    assert b.plain_work(0) == (1, False, 1)
    with pytest.raises(idgx.IdgxError):
        b.plain_work(1)
    b.close()
    b = _batch(idgx, 32, 8000, 1024, "fp32")
    b.set_shape(b.shape_table().index(next(s for s in b.shape_table() if s[0] == 4)), 0)
    px, whole, nv = b.plain_work(0)
    assert (px, whole) == (4, True) and nv == b.shape_table()[0][1]
    b.close()
    b = _batch(idgx, 32, 8, 16, "fp16x3")
    with pytest.raises(idgx.IdgxError):
        b.plain_work(0)
    b.close()
