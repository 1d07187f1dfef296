"""Ray counts at the edges of the trace kernel's launch: one ray, a batch of 64
and its neighbours, one batch per XCD, and the counts around which the launch
goes over from a wave for every batch to waves that take batches from the
per-XCD counters (7 resident blocks of 4 waves on each of 256 CUs, 458,752
rays, on an undivided MI355X).  A ray's record does not depend on the launch,
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
