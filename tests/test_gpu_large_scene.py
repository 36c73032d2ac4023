"""GPU tests of scenes with more instances than a pool's entries can name
(trace.hip, kPoolWorld): their waves traverse one ray per lane to the end, in
small equal shares or refilled from the queues on a grid of their own."""
import numpy as np
import pytest
import torch

from radeonrays_sdk_amd import api, autotune, rr, scenes
from tests.gpu_util import say, to_dev

pytestmark = pytest.mark.gpu

INSTANCES = (1 << 19) - 1  # the smallest scene that cannot pool
SHARED = 256 * 24 * 64     # rays that 24 waves per CU hold on 256 CUs
LONE = 256 * 24 * 8        # ... in equal shares of eight
EXTENT = 40.0


@pytest.fixture(scope="module")
def scene(ctx, dev):
    geometries = []
    for k in range(4):
        v, i = scenes.triangle_soup(12, scenes.rng_for(90, k), sigma=0.2)
        geometries.append(ctx.build_geometry(to_dev(v, dev), to_dev(i, dev)))
    xf = scenes.random_transforms(np.random.default_rng(91), INSTANCES, trans=EXTENT)
    built = ctx.build_scene([geometries[k % 4] for k in range(INSTANCES)], xf)
    return api.Accel(built.buffer, "tlas", INSTANCES, tuple(geometries))


def _rays(n, seed):
    rng = np.random.default_rng(seed)
    return scenes.make_rays(rng.uniform(-EXTENT, EXTENT, size=(n, 3)).astype(np.float32), scenes.unit_sphere(n, rng))


@pytest.fixture(scope="module")
def rays(dev):
    return to_dev(_rays(LONE + 1, 92), dev)


@pytest.fixture(scope="module")
def plain(ctx, scene, rays):
    with autotune.plain_traversal(ctx.lib):
        hits = {q: ctx.intersect(scene, rays, q, "full_t") for q in ("closest", "any")}
        torch.cuda.synchronize()
        return hits


@pytest.mark.parametrize("depth", [8, 16])
@pytest.mark.parametrize("n", [1, 65, 5000, LONE, LONE + 1])
def test_hits_equal_plain(ctx, dev, scene, rays, plain, n, depth):
    """Few rays a wave, more than a wave has, the last equal share and the first query that goes to the queues; eight
    LDS entries a lane make the stacks spill, into the rays' slots or the lanes'."""
    say(f"scene of {INSTANCES} instances, {n} rays, LDS stack {depth}")
    saved = autotune.current(ctx.lib)
    try:
        autotune.set_(ctx.lib, rr.RRX_TUNING_TRACE_LDS_STACK, depth)
        for query, want in plain.items():
            got = ctx.intersect(scene, rays[:n], query, "full_t")
            torch.cuda.synchronize()
            assert torch.equal(got, want[:32 * n]), query
    finally:
        autotune.apply(ctx.lib, saved)


@pytest.mark.parametrize("limit", [0, 100, LONE])
def test_device_count_below_the_recorded_one(ctx, dev, scene, rays, plain, limit):
    say(f"scene of {INSTANCES} instances, indirect count {limit}")
    count = torch.tensor([limit], dtype=torch.int32, device=dev)
    hits = torch.full((rays.shape[0] * 32,), 0xAB, dtype=torch.uint8, device=dev)
    ctx.intersect(scene, rays, "closest", "full_t", indirect=count, hits=hits)
    torch.cuda.synchronize()
    assert torch.equal(hits[:32 * limit], plain["closest"][:32 * limit])
    assert bool((hits[32 * limit:] == 0xAB).all())


def test_last_equal_share_is_no_slower_than_the_queues(ctx, dev, scene):
    """A full share of 64 rays for each of 24 waves per CU needs the pool; without one, one ray more (which goes to the
    queues in any scene) may not make the query faster.  Equal shares took 1.17 to 1.54 times as long."""
    say(f"scene of {INSTANCES} instances, {SHARED} rays timed")
    r = to_dev(scenes.camera_rays(640, SHARED // 640 + 1, (0.0, 0.0, -3 * EXTENT)), dev)
    hits, scratch = ctx.empty(r.shape[0] * 16), ctx.trace_scratch(r.shape[0])
    times = {}
    for _ in range(5):
        for n in (SHARED, SHARED + 1):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            ctx.intersect(scene, r[:n], "closest", "full", hits=hits, scratch=scratch)
            a.record()
            for _ in range(3):
                ctx.intersect(scene, r[:n], "closest", "full", hits=hits, scratch=scratch)
            b.record()
            torch.cuda.synchronize()
            times.setdefault(n, []).append(a.elapsed_time(b))
    shared, queued = (sorted(times[n])[2] for n in (SHARED, SHARED + 1))
    assert shared < 1.15 * queued, (shared, queued)
