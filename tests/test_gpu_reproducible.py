"""Images are a function of the scene and the seed alone: a path may be traced in the pool, in the path start or in the
drain, and which of them makes a given step depends on the order in which waves claim work, so all of them have to make
the same bits. The instrumented kernels (set_collect_stats) trace every path in the pool."""
import pytest

pytestmark = pytest.mark.gpu

MAPS = ["First X", "Depth", "Density", "Normal"]


def _scene(vpt, sparse, mode, interpolation, light, g):
    n = 128 if sparse else 48
    e0, e1 = (0.645, 0.795) if sparse else (0.45, 0.6)
    vpt.generate_fbm_cloud(n, n, n, seed=3, edge0=e0, edge1=e1)
    vpt.set_use_sparse_grid(sparse)
    vpt.set_vpt_mode(mode)
    vpt.set_grid_interpolation_type(interpolation)
    vpt.set_extinction_base([1.0, 1.0, 1.0])
    vpt.set_extinction_scale(900.0)
    vpt.set_scattering_albedo([0.93, 0.93, 0.93])
    vpt.set_phase_g(g)
    vpt.set_max_bounces(0)
    vpt.clear_lights()
    vpt.set_use_lights(light is not None)
    vpt.set_use_builtin_environment_map("Default")
    if light is not None:
        vpt.add_light()
        vpt.set_light_property(0, "type", light)
    vpt.set_camera_position([0.1, 0.2, 0.75])
    vpt.set_camera_target([0.0, 0.0, 0.0])
    vpt.set_seed_offset(9)


def _render(vpt, w, h, spp, stats=False):
    import torch

    vpt.set_collect_stats(stats)
    vpt.set_use_feature_maps(MAPS)
    probe = torch.zeros((4, h, w), dtype=torch.float32, device="cuda")
    out = [vpt.render_frame(probe, spp).clone()]
    out += [vpt.get_feature_map_from_string(probe, m).clone() for m in MAPS]
    vpt.set_collect_stats(False)
    vpt.set_use_feature_maps([])
    return [o.view(torch.int32) for o in out]  # bits: the maps hold NaN where no path met the medium


# Sizes on both sides of the most paths that skip the pool, and one with several hundred thousand paths handed over.
@pytest.mark.parametrize("sparse", [False, True])
@pytest.mark.parametrize("interpolation", [0, 1, 2])
@pytest.mark.parametrize("mode,light,g", [(0, None, 0.0), (2, None, 0.3), (3, None, 0.3), (4, None, 0.3),
                                          (5, None, 0.0), (5, "Spot Light", -0.4)])
def test_frames_do_not_depend_on_the_kernel(vpt, mode, light, g, interpolation, sparse):
    import torch

    print(f"case: reproducible frames mode={mode} {light} interpolation={interpolation} sparse={sparse}", flush=True)
    _scene(vpt, sparse, mode, interpolation, light, g)
    for w, h, spp in ((7, 5, 1), (131, 77, 3), (256, 257, 2), (640, 480, 2), (900, 700, 4)):
        want = _render(vpt, w, h, spp, stats=True)
        for _ in range(2):
            for k, (a, b) in enumerate(zip(_render(vpt, w, h, spp), want)):
                assert torch.equal(a, b), f"{w}x{h}x{spp} output {k}: {int((a != b).sum())} of {a.numel()} values differ"
    vpt.clear_lights()
    vpt.set_use_lights(False)


@pytest.mark.parametrize("mode", [0, 2, 3, 4, 5])
def test_batches_repeat(vpt, mode):
    import torch

    print(f"case: reproducible batch mode={mode}", flush=True)
    vpt.batch_clear()
    for sparse in (False, True):
        _scene(vpt, sparse, mode, 1, None, 0.5)
        vpt.batch_add_request(torch.zeros((3, 420, 400), dtype=torch.float32, device="cuda"), 7)
    first = [o.clone() for o in vpt.batch_render()]
    for _ in range(3):
        for k, (a, b) in enumerate(zip(first, vpt.batch_render())):
            assert torch.equal(a, b), f"request {k}: {int((a != b).sum())} of {a.numel()} values differ"
    vpt.batch_clear()
