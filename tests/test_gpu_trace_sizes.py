"""Ray counts at the edges of the trace kernel's launch: one ray, a batch of 64
and its neighbours, one batch per XCD, and the counts around which the launch
goes over from a wave for every batch to waves that take batches from the
per-XCD counters (7 resident blocks of 4 waves on each of 256 CUs, 458,752
rays, on an undivided MI355X), or, with the reference walk, from several
batches a wave (8 resident blocks, 1,048,513 rays) and from four on a tree
larger than an L2.  A ray's record does not depend on the launch,
so every prefix of one set must give the records of the whole set, and the
record behind it must stay as it was."""
import numpy as np
import pytest

from gpugi_amd import workloads

pytestmark = pytest.mark.gpu

RESIDENT = 256 * 7 * 4 * 64
MOST = 2 * RESIDENT + 77


@pytest.fixture(scope="module")
def ray_set(rt):
    c = rt.Context(0)
    c.load_scene(rt.HostScene.heightfield(64, workloads.MASTER_SEED))
    sets = workloads.HeightfieldRays(c, n=MOST)
    yield c, sets
    sets.free()
    c.close()


@pytest.mark.parametrize("n", [1, 63, 64, 65, 511, 512, 513, 2049, RESIDENT - 64, RESIDENT, RESIDENT + 1, MOST])
@pytest.mark.parametrize("query", ["closest", "any"])
@pytest.mark.parametrize("kernel", ["wide", "reference"])
def test_prefixes_of_a_ray_set(rt, ray_set, kernel, query, n):
    c, sets = ray_set
    print("case: %s, %s, %d rays" % (kernel, query, n), flush=True)
    rays, q = (sets.incoherent, rt.CLOSEST_HIT) if query == "closest" else (sets.shadow, rt.ANY_HIT)
    cols = slice(0, 4) if query == "closest" else slice(0, 1)
    c.trace_device(rays, sets.hits, MOST, q, rt.KERNEL_REFERENCE)
    want = sets.hits.download(np.int32, 4 * MOST).reshape(-1, 4)
    mark = np.full((MOST, 4), -77, np.int32)
    sets.hits.upload(mark)
    c.trace_device(rays, sets.hits, n, q, rt.KERNEL_WIDE if kernel == "wide" else rt.KERNEL_REFERENCE)
    got = sets.hits.download(np.int32, 4 * MOST).reshape(-1, 4)
    assert (got[n:] == -77).all()
    # an edge or a tie may differ between the walks
    most = n // 100000 if kernel == "wide" else 0
    assert (got[:n, cols] != want[:n, cols]).any(1).sum() <= most


class Part:
    """Records [first, ...) of a device buffer."""

    def __init__(self, buf, first, nbytes):
        self.ptr = buf.ptr + first * nbytes


REF_RESIDENT = 256 * 8 * 4 * 64


@pytest.mark.parametrize("scene,counts", [("cornell", (2 * REF_RESIDENT - 64, 2 * REF_RESIDENT - 63, 4 * REF_RESIDENT + 77)),
                                          ("hf64", (2 * REF_RESIDENT - 64, 2 * REF_RESIDENT - 63, 3000001)),
                                          ("hf512", (4 * REF_RESIDENT - 64, 4 * REF_RESIDENT + 4097))])
@pytest.mark.parametrize("mode", ["plain", "watertight", "obox"])
def test_reference_walk_of_several_batches_a_wave(rt, scene, counts, mode):
    """A ray's record is that of a launch of at most 65,536 rays, where every wave has one batch: on a tree whose
    waves have one always, and on trees below and above the L2's size; camera rays, whose waves wait for all of
    theirs, and diffuse ones."""
    c = rt.Context(0)
    sets = None
    try:
        if mode == "watertight":
            c.set_triangle_test(rt.TRIANGLE_WATERTIGHT)
        if mode == "obox":
            c.set_bvh_type(rt.BVH_OBOX)
        c.load_scene(rt.HostScene.cornell() if scene == "cornell" else
                     rt.HostScene.heightfield(int(scene[2:]), workloads.MASTER_SEED))
        n = max(counts)
        cam = workloads.cornell_camera(1024) if scene == "cornell" else workloads.heightfield_camera()
        w, h = (1024, 1024) if scene == "cornell" else (1920, 1080)
        lights = np.array([[0.0, 1.9, 0.0], [0.3, 1.8, -0.2]], np.float32) if scene == "cornell" else \
            workloads.heightfield_lights()
        sets = workloads.SceneRays(c, cam, lights, n, workloads.MASTER_SEED, w, h)
        for rays, query in ((sets.primary, rt.CLOSEST_HIT), (sets.incoherent, rt.CLOSEST_HIT), (sets.shadow, rt.ANY_HIT)):
            cols = slice(0, 4) if query == rt.CLOSEST_HIT else slice(0, 1)
            for at in range(0, n, 65536):
                c.trace_device(Part(rays, at, 32), Part(sets.hits, at, 16), min(65536, n - at), query, rt.KERNEL_REFERENCE)
            want = sets.hits.download(np.int32, 4 * n).reshape(-1, 4)
            assert (want[:, 0] > 0).any()
            for m in counts:
                print("case: %s %s, query %d, %d rays" % (scene, mode, query, m), flush=True)
                sets.hits.upload(np.full((n, 4), -77, np.int32))
                c.trace_device(rays, sets.hits, m, query, rt.KERNEL_REFERENCE)
                got = sets.hits.download(np.int32, 4 * n).reshape(-1, 4)
                assert (got[m:] == -77).all() and np.array_equal(got[:m, cols], want[:m, cols])
    finally:
        if sets is not None:
            sets.free()
        c.close()
