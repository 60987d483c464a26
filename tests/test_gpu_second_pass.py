"""The second pass's forms: a wave per ray (short queues), a lane per ray
(queues of wide_min rays or more), and the third pass behind it, over rays
with a few and with many listed cache nodes, of bilinear and bicubic patches,
untransformed and transformed."""
import pytest
import torch

from psychopath_cpp_amd import configs, gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,depth", [("subdivision", 15), ("subdivision", 6), ("heightfield", 5), ("heightfield", 0)])
def test_gpu_second_pass_forms_agree(name, depth):
    sc = configs.subdivision_scene(grid=12, dice_rate=0.25) if name == "subdivision" else \
        configs.heightfield_scene(grid=12, dice_rate=0.25)
    ctx = gpu.Context(0)
    try:
        g = gpu.GpuScene(ctx, sc, dice_depth=depth)
        w, _ = gpu.camera_rays(ctx, g, 97, 61, 1, 2)
        bounce, valid = gpu.bounce_rays(ctx, g, w, gpu.trace_world(ctx, g, w), 97, 1, 2)
        w = torch.cat([w, bounce[:, valid.bool()]], 1).contiguous()
        ref = gpu.trace_world(ctx, g, w)
        queued = ctx.pass_counts()[0]
        assert queued > 0
        for wide_min in (0, 1, queued, queued + 1, 0xFFFFFFFF):
            for budget in (1, 7, 512):
                ctx.set_second_pass(wide_min, budget)
                print(name, depth, "queued", queued, "wide_min", wide_min, "budget", budget, flush=True)
                h = gpu.trace_world(ctx, g, w)
                second, third = ctx.pass_counts()
                assert second == queued
                assert third == 0 or wide_min <= queued
                # a lane's ray that needs more than one node expansion is handed over
                assert third > 0 or wide_min > queued or budget > 1
                # exactly tied micropolygons may resolve differently; distances do not depend on the form
                assert torch.equal(h.t, ref.t)
                same = h.inst == ref.inst
                for k in ("u", "v", "aux"):
                    same &= getattr(h, k) == getattr(ref, k)
                assert float(same.float().mean()) >= 0.9999
                occ = gpu.trace_world(ctx, g, w, occlusion_only=True)
                assert torch.equal(occ.inst != -1, ref.inst != -1)
        g.close()
    finally:
        ctx.close()
