"""GPU tests of what bounds the pooled traversal's node reads (trace.hip): the
node count and the node offset of the buffer's own header, as in the loops
that traverse one ray per lane."""
import numpy as np
import pytest
import torch

from radeonrays_sdk_amd import api, autotune, rr, scenes
from tests.gpu_util import say, to_dev

pytestmark = pytest.mark.gpu

NODE_COUNT = slice(12, 16)  # AccelHeader.node_count
NODES_OFFSET = slice(16, 24)  # AccelHeader.nodes_offset
HEADER = 128


def _rays(n, seed, lo=0.0, hi=1.0):
    rng = np.random.default_rng(seed)
    return scenes.make_rays(rng.uniform(lo, hi, size=(n, 3)).astype(np.float32), scenes.unit_sphere(n, rng))


@pytest.mark.parametrize("query", ["closest", "any"])
@pytest.mark.parametrize("rays", [1, 65, 3000])
def test_batch_reads_no_node_past_the_header_count(ctx, dev, query, rays):
    """A buffer whose header counts its inner nodes alone has no leaf that may be read: every ray misses.  (The
    nodes past the count are there, so a read of one would show as a hit.)"""
    say(f"batched request, {rays} rays, {query}, leaves past the node count")
    v, i = scenes.triangle_soup(5000, scenes.rng_for(80))
    accel = ctx.build_geometry(to_dev(v, dev), to_dev(i, dev))
    r = to_dev(_rays(rays, 81), dev)
    whole = api.decode_hits(ctx.intersect_batch([(accel, r, query, "full")])[0])
    assert rays < 3000 or (whole["prim_id"] != rr.RR_INVALID).any()
    accel.buffer[NODE_COUNT].view(torch.int32)[0] = i.shape[0] - 1
    hits = api.decode_hits(ctx.intersect_batch([(accel, r, query, "full")])[0])
    assert (hits["prim_id"] == rr.RR_INVALID).all()


@pytest.mark.parametrize("query", ["closest", "any"])
@pytest.mark.parametrize("rays", [1, 65, 5000])
def test_scene_finds_geometry_nodes_where_the_header_says(ctx, dev, query, rays):
    """An instance of a geometry whose nodes lie further behind its header than the builders put them; what is there
    instead would read as leaves."""
    say(f"scene of a geometry with moved nodes, {rays} rays, {query}")
    v, i = scenes.triangle_soup(4000, scenes.rng_for(82))
    plain = ctx.build_geometry(to_dev(v, dev), to_dev(i, dev))
    gap = 4096
    moved = torch.full((plain.buffer.numel() + gap,), 0xFF, dtype=torch.uint8, device=dev)
    moved[:HEADER] = plain.buffer[:HEADER]
    moved[HEADER + gap:] = plain.buffer[HEADER:]
    moved[NODES_OFFSET].view(torch.int64)[0] = HEADER + gap
    geometries = (plain, api.Accel(moved, "blas", plain.prim_count))
    n = 20
    xf = scenes.random_transforms(np.random.default_rng(83), n, trans=1.0)
    r = to_dev(_rays(rays, 84, -1.5, 1.5), dev)
    want = ctx.intersect(ctx.build_scene([plain] * n, xf), r, query, "full_t")
    scene = ctx.build_scene([geometries[k % 2] for k in range(n)], xf)
    got = ctx.intersect(scene, r, query, "full_t")
    torch.cuda.synchronize()
    assert rays < 5000 or len(set(api.decode_hits(want, "full_t")["inst_id"].tolist()) - {rr.RR_INVALID}) == n
    assert torch.equal(got, want)
    with autotune.plain_traversal(ctx.lib):
        assert torch.equal(ctx.intersect(scene, r, query, "full_t"), want)


def _median_times(ctx, accel, r, depths):
    """Milliseconds of ten closest-hit queries at each LDS stack depth, measured in turn."""
    hits, scratch = ctx.empty(r.shape[0] * 16), ctx.trace_scratch(r.shape[0])
    saved = autotune.current(ctx.lib)
    times = {d: [] for d in depths}
    try:
        for _ in range(6):
            for depth in depths:
                autotune.set_(ctx.lib, rr.RRX_TUNING_TRACE_LDS_STACK, depth)
                a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                ctx.intersect(accel, r, "closest", "full", hits=hits, scratch=scratch)
                a.record()
                for _ in range(10):  # behind the first: the GPU does not wait for the host
                    ctx.intersect(accel, r, "closest", "full", hits=hits, scratch=scratch)
                b.record()
                torch.cuda.synchronize()
                times[depth].append(a.elapsed_time(b))
    finally:
        autotune.apply(ctx.lib, saved)
    return [sorted(times[d])[2] for d in depths]


@pytest.mark.parametrize("which", ["soup", "scene"])
def test_pool_of_short_stacks_has_room_to_work(ctx, dev, which):
    """Long rays, 64 for every wave that pools at once: with eight-entry stacks, whose pool was half reserve, they took
    4.7 times (a geometry) and 5.2 times (a scene) as long as with 16 entries; the stacks alone make no such
    difference (a factor of 1.2 for queries that do not pool)."""
    say(f"pool on eight-entry stacks timed, {which}")
    if which == "soup":
        v, i = scenes.triangle_soup(65536, scenes.rng_for(85))
        accel, n, eye = ctx.build_geometry(to_dev(v, dev), to_dev(i, dev), restructure=True), 260000, (0.5, 0.5, -1.5)
    else:
        geometries = []
        for k in range(8):
            v, i = scenes.triangle_soup(2000, scenes.rng_for(86, k))
            geometries.append(ctx.build_geometry(to_dev(v, dev), to_dev(i, dev), restructure=True))
        xf = scenes.random_transforms(np.random.default_rng(87), 1000, trans=12.0)
        accel, n, eye = ctx.build_scene([geometries[k % 8] for k in range(1000)], xf), 390000, (0.0, 0.0, -36.0)
    r = to_dev(scenes.camera_rays(500, n // 500, eye), dev)
    short, usual = _median_times(ctx, accel, r, (8, 16))
    assert short < 2 * usual, (short, usual)


@pytest.fixture(scope="module")
def terrain(ctx, dev):
    v, i = scenes.heightfield_mesh(724)
    return ctx.build_geometry(to_dev(v, dev), to_dev(i, dev), restructure=True)


@pytest.mark.parametrize("query", ["closest", "any"])
def test_spilled_entries_go_into_the_pool(ctx, dev, terrain, query):
    """More rays than equal shares hold, in a tree deeper than the stacks' eight LDS entries: waves form their pool
    while lanes have spilled."""
    say(f"pool of spilled stacks, {query}")
    r = to_dev(_rays(330001, 88), dev)
    saved = autotune.current(ctx.lib)
    try:
        autotune.set_(ctx.lib, rr.RRX_TUNING_TRACE_LDS_STACK, 8)
        got = ctx.intersect(terrain, r, query, "full_t")
        torch.cuda.synchronize()
    finally:
        autotune.apply(ctx.lib, saved)
    with autotune.plain_traversal(ctx.lib):
        assert torch.equal(got, ctx.intersect(terrain, r, query, "full_t"))


def test_spilled_stacks_pool_as_soon_as_others(ctx, dev, terrain):
    """Waves whose lanes had spilled did not pool, and went on one ray per lane: 1.9 times as long as with 16 entries,
    of which none spill here."""
    say("pool of spilled stacks timed")
    short, usual = _median_times(ctx, terrain, to_dev(_rays(300000, 88), dev), (8, 16))
    assert short < 1.4 * usual, (short, usual)
