"""The main pass's form that a context picks by itself: the same bits as every
form set by hand, on each side of its rule (moving and static scenes of
patches, a moving scene without, object rays shorter than and as long as a
stream that continues)."""
import pytest
import torch

from psychopath_cpp_amd import configs, gpu

pytestmark = pytest.mark.gpu

SCENES = {
    "moving patches": lambda: configs.bicubic_sphere_scene(seed=3, grid=6, dice_rate=1.0),
    "static patches": lambda: configs.heightfield_scene(seed=3, grid=6),
    "spheres": lambda: configs.sphere_scene(seed=3, n_spheres=24),
}


def _equal(a, b):
    return all(torch.equal(getattr(a, k), getattr(b, k)) for k in ("t", "inst", "u", "v", "aux"))


@pytest.mark.parametrize("name", SCENES)
@pytest.mark.parametrize("size", [(1, 1, 1), (9, 7, 1), (13, 5, 1), (64, 63, 3)])
def test_gpu_default_form_same_bits(name, size):
    auto, ctx = gpu.Context(0), gpu.Context(0)
    try:
        sc = SCENES[name]()
        ga, g = gpu.GpuScene(auto, sc), gpu.GpuScene(ctx, sc)
        w, _ = gpu.camera_rays(auto, ga, *size, 11)
        rays = gpu.world_to_rays(auto, w)
        got = gpu.trace_world(auto, ga, w)
        # (instances of patches with transforms take world rays only)
        got_o = None if name == "moving patches" else gpu.trace_rays(auto, ga, rays)
        for persistent, coherent in ((False, False), (False, True), (True, False), (True, True)):
            ctx.set_trace_mode(persistent=persistent, coherent=coherent)
            for below in (0, 24):
                ctx.set_continuation(below)
                assert _equal(got, gpu.trace_world(ctx, g, w)), (persistent, coherent, below)
                assert got_o is None or _equal(got_o, gpu.trace_rays(ctx, g, rays)), (persistent, coherent, below)
        auto.set_continuation(24)  # world rays that continue take the plain form
        assert _equal(got, gpu.trace_world(auto, ga, w))
        ga.close()
        g.close()
    finally:
        auto.close()
        ctx.close()


@pytest.mark.parametrize("n", [(1 << 21) - 1, 1 << 21])
def test_gpu_default_continuation_same_bits(n):
    auto, ctx = gpu.Context(0), gpu.Context(0)
    try:
        sc = SCENES["static patches"]()
        ga, g = gpu.GpuScene(auto, sc), gpu.GpuScene(ctx, sc)
        w, _ = gpu.camera_rays(auto, ga, 1024, 1024, 2, 11)
        rays = gpu.world_to_rays(auto, w)[:, :n].contiguous()
        got = gpu.trace_rays(auto, ga, rays)
        for below in (0, 24):
            ctx.set_continuation(below)
            assert _equal(got, gpu.trace_rays(ctx, g, rays)), below
        ga.close()
        g.close()
    finally:
        auto.close()
        ctx.close()
