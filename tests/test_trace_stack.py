"""Traversal stacks that outgrow the main pass's LDS entries in a scene with
patches: the bottom of the stack goes to the trace's scratch pool and comes
back, so the ray is finished in the main pass, with the hits of the second
pass's 64-entry stack.  With the pool exhausted the ray is retraced."""
import numpy as np
import pytest

from psychopath_cpp_amd import abi
from psychopath_cpp_amd.scene import Bilinear
from tests import test_gpu_parity as G


def _nested_with_patch(n):
    """Spheres around one centre (every ray through it hits every BVH box)
    over a ground patch."""
    sc = G._nested_spheres(n=n)
    sc.dice_rate = 4.0  # coarse: no ray dices the ground below the cache
    sc.root.add_object("ground", Bilinear([(-4, -4, -0.2), (4, -4, -0.3), (-4, 4, -0.25), (4, 4, -0.1)]))
    sc.root.create_object_instance("ground", [], "s")
    return sc


@pytest.mark.parametrize("n", [24, 1024])
def test_cpu_build_stack_kept_in_pool(n):
    from oracle import ora
    from tests.cpu_build import hostbuild
    from tests.test_cpu_build_parity import compare
    sc = _nested_with_patch(n)
    rc, need = hostbuild.scene_stack_need(sc)
    assert rc == 0 and (need > 16) == (n == 1024)
    o = ora.OracleScene(sc)
    w, _ = o.camera_rays(48, 32, 1, 4)
    hb = hostbuild.trace(sc, ora.planes_from_wrays(w), world=True, dice_depth=14)
    agree, t_ok, hits = compare(hb, o.trace(w, threads=8, chunk=8192))
    assert hb["retraced"] == 0  # 1024: handed on before the pool took the stack
    assert hits > 100 and agree >= 0.9999 and t_ok >= 0.9999


@pytest.mark.gpu
@pytest.mark.parametrize("size", [2, 48, 200])
def test_gpu_stack_kept_in_pool(size):
    """The same hits whatever the stack: 16 entries and the pool (2x2 rays:
    no room for one chunk; 48, 200: for a sixth of the rays), 32 entries, and
    world and object rays alike."""
    import torch
    from psychopath_cpp_amd import gpu
    ctx = gpu.Context(0)
    try:
        g = gpu.GpuScene(ctx, _nested_with_patch(4096))
        assert g.info.bvh_stack_need > 16
        w, _ = gpu.camera_rays(ctx, g, size, size, 1, 4)
        rays = gpu.world_to_rays(ctx, w)
        ref = None
        for stack in (32, 16):
            ctx.set_trace_stack(stack)
            for persistent in (True, False):
                ctx.set_trace_mode(persistent=persistent)
                print("rays", size * size, "stack", stack, "persistent", persistent, flush=True)
                for h in (gpu.trace_world(ctx, g, w), gpu.trace_rays(ctx, g, rays)):
                    got = [x.clone() for x in (h.t, h.inst, h.u, h.v, h.aux)]
                    ref = ref or got
                    assert all(torch.equal(a, b) for a, b in zip(got, ref))
        assert int((ref[1] != -1).sum()) > 0
        ctx.set_continuation(24)
        h = gpu.trace_world(ctx, g, w)
        assert all(torch.equal(a, b) for a, b in zip((h.t, h.inst, h.u, h.v, h.aux), ref))
        g.close()
    finally:
        ctx.close()
