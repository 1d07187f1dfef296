"""The integrators in phases over the wide BVH (phased_paths) against the same
integrators over the reference walk, whose kernel traces each ray where it is
needed.  Every path computes the same terms in the same order, so an image can
differ only where the two walks do (an edge or a tie; at most 1e-3 of the
pixels here) and, for the light tracer's camera splats, in the order of float
atomics (each of a pixel's at most 2^12 sums rounds to 2^-24 of it: 2.5e-4).
A bidirectional image draws its connections from the whole light cache, so one
differing light path would change it everywhere: none of these has one.

The sizes: 16 and 32 lanes a wave (images of at most one wave per SIMD), sizes
that are no multiple of the 8 x 8 tiles, and more pixels than the resident waves
have lanes, so that lanes take second pixels.  The scene has more nodes than
the small-tree rule keeps in step."""
import numpy as np
import pytest

from gpugi_amd import workloads

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def phased_scene(rt):
    return rt.HostScene.clutter(24, 5)


def draw(rt, ctx, scene, integrator, kernel, w, h, frames=2, cam=None):
    ctx.set_screen(w, h)
    ctx.set_camera(cam or workloads.clutter_camera(w, h))
    ctx.set_max_path_length(4)
    ctx.set_integrator_kernel(kernel)
    sampler = rt.LightSampler(scene, 7)
    if integrator == rt.BPT:
        ctx.set_light_samples(sampler.generate(128))
        entries, _ = ctx.bpt_warmup(5)
        ctx.bpt_set_light_cache(entries + entries // 4)
    for k in range(frames):
        ctx.set_light_samples(sampler.generate(128))
        ctx.draw(integrator, rt.wanghash(k))
    img = ctx.readback(w, h)[0]
    ctx.set_integrator_kernel(rt.KERNEL_AUTO)
    return img


@pytest.mark.parametrize("size", [(64, 48), (203, 157), (330, 250), (1030, 530)])
@pytest.mark.parametrize("integrator", ["PT", "LT", "BPT"])
def test_phased_image_equals_the_reference_walk(rt, ctx, phased_scene, integrator, size):
    ctx.load_scene(phased_scene)
    w, h = size
    images = []
    for kernel in (rt.KERNEL_REFERENCE, rt.KERNEL_WIDE):
        print("case: phased %s %dx%d kernel %d" % (integrator, w, h, kernel), flush=True)
        images.append(draw(rt, ctx, phased_scene, getattr(rt, integrator), kernel, w, h))
    want, got = images
    assert want[..., :3].max() > 0 and np.isfinite(want).all() == np.isfinite(got).all()
    if integrator == "PT":
        same = (want.view(np.uint32) == got.view(np.uint32)).all(-1)
    else:
        same = np.isclose(got, want, rtol=2.5e-4, atol=1e-7, equal_nan=True).all(-1)
    assert same.mean() >= 0.999, same.mean()


@pytest.mark.parametrize("size", [(672, 680), (680, 680)])
@pytest.mark.parametrize("scene", ["cornell", "hf24", "hf96"])
@pytest.mark.parametrize("integrator", ["PT", "LT"])
def test_image_at_the_edge_of_staying_in_step(rt, ctx, integrator, scene, size):
    """Seven waves per SIMD are 458,752 paths on an undivided MI355X.  A small closed tree, a small open one, and
    an open one above the small-tree limit, whose light paths alone stay in step."""
    hs = rt.HostScene.cornell()
    if scene != "cornell":  # the heightfield with its triangles turned over: light paths light their front only
        a = rt.HostScene.heightfield(int(scene[2:]), 5).arrays()
        tri = a["triangles"][a["triangles"][:, 0] != a["triangles"][:, 1]]
        hs = rt.HostScene.build(a["positions"], tri[:, 2::-1].astype(np.uint32))
        for p in workloads.heightfield_lights():
            hs.add_point_light(p, (0.5, 0.5, 0.5))
    ctx.load_scene(hs)
    w, h = size
    cam = rt.camera((0.0, 1.0, 3.7), (0.0, 1.0, 0.0), (0.0, 1.0, 0.0), 40.0, w, h) if scene == "cornell" else \
        workloads.heightfield_camera(w, h)
    images = []
    for kernel in (rt.KERNEL_REFERENCE, rt.KERNEL_WIDE):
        print("case: in step %s %s %dx%d kernel %d" % (integrator, scene, w, h, kernel), flush=True)
        images.append(draw(rt, ctx, hs, getattr(rt, integrator), kernel, w, h, 2, cam))
    want, got = images
    assert want[..., :3].max() > 0
    if integrator == "PT":
        same = (want.view(np.uint32) == got.view(np.uint32)).all(-1)
    else:
        same = np.isclose(got, want, rtol=2.5e-4, atol=1e-7, equal_nan=True).all(-1)
    assert same.mean() >= 0.999, same.mean()


@pytest.mark.parametrize("integrator", ["PT", "LT", "BPT"])
def test_phased_watertight_image(rt, ctx, phased_scene, integrator):
    """The watertight kernels.  The wide walk's records hold b_y and b_z and b_x is rebuilt as 1 - (b_y + b_z),
    so hit attributes differ in their last bits from the reference walk's: a path may part at a roulette
    or lobe decision.  One parted pixel of 32,000 changes the mean by up to 1e-5 of it per frame (its share of
    the sum, for values up to a third of the image's mean apart)."""
    ctx.set_triangle_test(rt.TRIANGLE_WATERTIGHT)
    try:
        ctx.load_scene(phased_scene)
        want, got = (draw(rt, ctx, phased_scene, getattr(rt, integrator), k, 203, 157, 4)[..., :3].astype(np.float64)
                     for k in (rt.KERNEL_REFERENCE, rt.KERNEL_WIDE))
        print("case: phased watertight", integrator, want.mean(), got.mean(), flush=True)
        assert want.mean() > 0 and abs(got.mean() / want.mean() - 1) < 4e-5
    finally:
        ctx.set_triangle_test(rt.TRIANGLE_REFERENCE)
