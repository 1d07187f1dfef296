"""The wide walk on a deep, narrow tree, where the traversal stacks go far past
their LDS part (test_wide_walk_cpu.py's nested quads: over 48 entries)."""
import numpy as np
import pytest

from test_wide_walk_cpu import centre_camera, centre_rays, nested_scene, walk  # noqa: F401 (walk is a fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("stack", [4, 10, 24])
def test_trace_spills_on_a_deep_tree(rt, oracle, ctx, stack):
    hs = nested_scene(60)
    sc, rays = oracle.Scene(hs.arrays()), centre_rays(20001, 9)
    ctx.load_scene(hs)
    ctx.set_wide_config(1, stack)
    try:
        print("case: deep tree, %d LDS entries" % stack, flush=True)
        r = rays.view(rt.RAY_DTYPE).reshape(-1)
        got = ctx.trace(r, rt.CLOSEST_HIT, rt.KERNEL_WIDE).view(np.int32).reshape(-1, 4)
        assert np.array_equal(got, oracle.bruteforce(sc, rays))
        got = ctx.trace(r, rt.ANY_HIT, rt.KERNEL_WIDE)["slot"]
        want = oracle.bruteforce(sc, rays, any_hit=True)[:, 0]
        assert 0 < want.sum() < len(want) and np.array_equal(got, want)
    finally:
        ctx.set_wide_config(2, 10)


def test_max_stack_is_the_walks_bound(rt, walk, ctx):  # noqa: F811
    """gpugi_get_wide_config's max_stack: the stack entries the walk is given, not the children in them."""
    for hs, leaf in ((nested_scene(60), 1), (rt.HostScene.heightfield(64, 5), 2), (rt.HostScene.cornell(), 8)):
        ctx.load_scene(hs)
        ctx.set_wide_config(leaf, 10)
        try:
            _, n = walk(hs, centre_rays(1, 1), leaf)
            assert ctx.wide_config()["max_stack"] == n["stack"]
        finally:
            ctx.set_wide_config(2, 10)


def test_path_tracer_spills_on_a_deep_tree(rt, ctx):
    """The path tracer's 16 entries and the batch's 16, 24 and 32 give one image: where the stack lives
    does not change it."""
    hs = nested_scene(60)
    hs.add_point_light((0.9, 0.8, 1.1), (1.0, 1.0, 1.0))
    cam = centre_camera(64)
    lights = rt.LightSampler(hs, 3).generate(128)
    ctx.load_scene(hs)
    ctx.set_screen(64, 64)
    ctx.set_camera(cam)
    ctx.set_light_samples(lights)
    ctx.set_max_path_length(4)
    ctx.set_integrator_kernel(rt.KERNEL_WIDE)
    print("case: deep tree, path tracer", flush=True)
    ctx.draw(rt.PT, rt.wanghash(0))
    image = ctx.readback(64, 64)[0]
    ctx.set_integrator_kernel(rt.KERNEL_AUTO)
    assert image.max() > 0
    b = rt.Batch(0)
    try:
        b.add(hs, cam, 64, 64, lights, 4)
        b.finalize()
        for stack in (16, 24, 32):
            print("case: deep tree, batch, %d LDS entries" % stack, flush=True)
            b.config(rt.KERNEL_WIDE, 2, 2, stack)
            b.reset(0)
            b.draw(True)
            assert np.array_equal(b.readback(0).view(np.uint32), image.view(np.uint32)), stack
    finally:
        b.close()
