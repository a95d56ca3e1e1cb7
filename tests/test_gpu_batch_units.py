"""Units of the batched queue: the launch that is reported and tuned is the one that renders, and units of several
samples trace the same paths as units of one."""
import pytest

pytestmark = pytest.mark.gpu


def _batch(vpt, mode, side, spp):
    """Two requests, a dense and a NanoVDB volume."""
    import torch

    vpt.batch_clear()
    for sparse in (False, True):
        vpt.generate_fbm_cloud(40, 36, 44, seed=2)
        vpt.set_use_sparse_grid(sparse)
        vpt.set_vpt_mode(mode)
        vpt.set_grid_interpolation_type("stochastic")
        vpt.set_extinction_base([1.0, 0.8, 0.6] if mode in (1, 6) else [1.0, 1.0, 1.0])
        vpt.set_extinction_scale(96.0)
        vpt.set_scattering_albedo([0.9, 0.9, 0.9])
        vpt.set_phase_g(0.3)
        vpt.set_max_bounces(32)
        vpt.set_use_builtin_environment_map("Default")
        vpt.set_use_lights(False)
        vpt.set_camera_position([0.1, 0.2, 0.7])
        vpt.set_camera_target([0.0, 0.0, 0.0])
        vpt.set_seed_offset(5)
        vpt.batch_add_request(torch.zeros((3, side, side), dtype=torch.float32, device="cuda"), spp)


def test_reported_launch_is_the_one_that_renders(vpt):
    print("case: batch launch reports", flush=True)
    _batch(vpt, 0, 48, 8)  # 36 864 paths: fewer than the lanes of a launch by occupancy
    vpt.batch_set_launch_config(0, 128, 4, 16)
    got = vpt.batch_get_launch_config()
    assert (got["block_size"], got["steps_per_refill"], got["samples_per_unit"]) == (128, 4, 1)
    assert got["blocks"] > 36864 // 128
    # 64 lanes: 576 paths each, nine samples per unit
    vpt.batch_set_launch_config(1, 64, 4, 16)
    assert vpt.batch_get_launch_config() == {"blocks": 1, "block_size": 64, "steps_per_refill": 4,
                                             "samples_per_unit": 9}
    vpt.batch_set_launch_config(1, 64, 4, 3)
    assert vpt.batch_get_launch_config()["samples_per_unit"] == 3
    vpt.batch_clear()


def test_autotune_keeps_a_launch_that_renders(vpt):
    print("case: batch autotune of a small batch", flush=True)
    _batch(vpt, 5, 48, 8)
    vpt.batch_set_launch_config(0, 256, 16, 16)
    cfg = vpt.batch_autotune(2)
    # every setting of the samples per unit comes to one sample with so few paths
    assert cfg["samples_per_unit"] == 1
    assert vpt.batch_get_launch_config() == cfg
    tuned = [o.clone() for o in vpt.batch_render()]
    vpt.batch_set_launch_config(cfg["blocks"], cfg["block_size"], cfg["steps_per_refill"], cfg["samples_per_unit"])
    assert vpt.batch_get_launch_config() == cfg
    for a, b in zip(tuned, vpt.batch_render()):
        assert bool((a == b).all())
    vpt.batch_clear()


@pytest.mark.parametrize("samples", [2, 3, 16])
@pytest.mark.parametrize("mode", [0, 1, 2, 3, 4, 5, 6])
def test_units_of_several_samples_trace_the_same_paths(vpt, mode, samples):
    """One workgroup of 64 lanes keeps `samples` per unit (17 samples per pixel: the last unit of a pixel is a part);
    units of one sample leave their last paths to the drain. Equal up to the float sum within a unit: non-negative
    samples, so samples - 1 roundings of 2^-24 and one more of each result."""
    import numpy as np

    print(f"case: batch units mode={mode} samples={samples}", flush=True)
    _batch(vpt, mode, 48, 17)
    vpt.batch_set_launch_config(0, 256, 16, 1)
    want = [o.cpu().numpy().astype(np.float64) for o in vpt.batch_render()]
    vpt.batch_set_launch_config(1, 64, 16, samples)
    assert vpt.batch_get_launch_config()["samples_per_unit"] == samples
    for k, (a, b) in enumerate(zip(vpt.batch_render(), want)):
        a = a.cpu().numpy().astype(np.float64)
        off = np.abs(a - b) > (samples + 1) * 2.0 ** -24 * b
        assert not off.any(), f"request {k}: {int(off.sum())} of {off.size} values differ"
    vpt.batch_clear()
