"""GPU tests of the pooled traversal against the plain kernels, bit for bit,
each side on its own kernels (autotune.plain_traversal): geometries of
triangles and of boxes, scenes of both, every LDS stack depth, indirect
counts, pieces, batches, and pools that fill up to their reserve."""
import numpy as np
import pytest
import torch

from radeonrays_sdk_amd import autotune, rr, scenes
from tests.gpu_util import say, to_dev

pytestmark = pytest.mark.gpu

SHARED = 256 * 16 * 64     # rays that 16 waves per CU hold on 256 CUs
SHARED_SCENE = 256 * 24 * 64
SIZES = {"full": 16, "full_t": 32, "instance": 4}


def _plain(ctx, accel, rays, query, output):
    with autotune.plain_traversal(ctx.lib):
        hits = ctx.intersect(accel, rays, query, output)
        torch.cuda.synchronize()
    assert autotune.get(ctx.lib, rr.RRX_TUNING_TRACE_PLAIN) == 0
    return hits


def _rays(n, seed, tmax=1e30):
    rng = np.random.default_rng(seed)
    o = rng.uniform(-0.2, 1.2, size=(n, 3)).astype(np.float32)
    return scenes.make_rays(o, scenes.unit_sphere(n, rng), 0.0, tmax)


@pytest.fixture(scope="module")
def world(ctx, dev):
    rng = np.random.default_rng(5)
    v, i = scenes.triangle_soup(9000, rng, sigma=0.03)
    soup = ctx.build_geometry(to_dev(v, dev), to_dev(i, dev), restructure=True)
    v, i = scenes.triangle_soup(40, rng, sigma=0.2)
    dup = ctx.build_geometry(to_dev(v, dev), to_dev(np.tile(i, (30, 1)), dev))
    one = ctx.build_geometry(to_dev(v[:3], dev), to_dev(i[:1], dev))
    c, h = rng.uniform(size=(6000, 3)), 0.02 * rng.uniform(size=(6000, 3))
    boxes = ctx.build_aabbs(to_dev(np.concatenate([c - h, c + h], axis=1).astype(np.float32), dev), restructure=True)
    parts = (soup, dup, one, boxes)
    scene = ctx.build_scene([parts[k % 4] for k in range(60)], scenes.random_transforms(rng, 60, trans=0.8))
    return {"soup": soup, "dup": dup, "one": one, "boxes": boxes, "scene": scene}


@pytest.mark.parametrize("query", ["closest", "any"])
@pytest.mark.parametrize("which", ["soup", "dup", "one", "boxes", "scene"])
def test_hits_equal_plain(ctx, dev, world, which, query):
    """One ray, parts of a wave, full waves, the last equal share and more rays than the shares hold."""
    say(f"pooled hits, {which}, {query}")
    shared = SHARED_SCENE if which == "scene" else SHARED
    counts = [1, 2, 63, 64, 65, 1000, 4097, shared // 64 * 3 + 1, shared, shared + 1, shared + 70001]
    rays = to_dev(_rays(max(counts), 11, 1e30 if query == "closest" else 0.7), dev)
    for output in ("full_t", "instance"):
        want = _plain(ctx, world[which], rays, query, output)
        for n in counts:
            got = ctx.intersect(world[which], rays[:n], query, output)
            torch.cuda.synchronize()
            assert torch.equal(got, want[:n * SIZES[output]]), (output, n)


@pytest.mark.parametrize("depth", [8, 16, 32])
@pytest.mark.parametrize("which", ["soup", "boxes", "scene"])
def test_every_stack_depth(ctx, dev, world, which, depth):
    say(f"pooled hits, {which}, LDS stack {depth}")
    rays = to_dev(_rays(SHARED_SCENE + 50001, 12), dev)
    saved = autotune.current(ctx.lib)
    got = {}
    try:
        autotune.set_(ctx.lib, rr.RRX_TUNING_TRACE_LDS_STACK, depth)
        for query in ("closest", "any"):
            for n in (70001, rays.shape[0]):
                got[query, n] = ctx.intersect(world[which], rays[:n], query, "full")
        torch.cuda.synchronize()
    finally:
        autotune.apply(ctx.lib, saved)
    for query in ("closest", "any"):
        want = _plain(ctx, world[which], rays, query, "full")
        for n in (70001, rays.shape[0]):
            assert torch.equal(got[query, n], want[:16 * n]), (query, n)


@pytest.mark.parametrize("depth", [8, 16, 32])
@pytest.mark.parametrize("two_level", [False, True])
def test_pool_at_its_reserve(ctx, dev, depth, two_level):
    """Equal triangles across their box, and rays of which half cross the box beside them: such a ray visits every
    node, so 64 of them double the list with each step until only its reserve is left and a step takes one entry."""
    say(f"pool at its reserve, LDS stack {depth}, {'scene' if two_level else 'geometry'}")
    rng = np.random.default_rng(17)
    tri = np.array([[0, 0, 0.1], [1, 0, 0.5], [0, 1, 0.9]], np.float32)
    n_tri, n = (40, SHARED_SCENE) if two_level else (300, SHARED)
    accel = ctx.build_geometry(to_dev(tri, dev), to_dev(np.tile(np.arange(3, dtype=np.int32), (n_tri, 1)), dev))
    if two_level:
        accel = ctx.build_scene([accel] * 8, np.tile(np.eye(3, 4, dtype=np.float32), (8, 1, 1)))
    o = np.concatenate([rng.uniform(0.02, 0.98, size=(n, 2)), np.full((n, 1), -1.0)], axis=1).astype(np.float32)
    rays = to_dev(scenes.make_rays(o, np.tile(np.float32([0, 0, 1]), (n, 1))), dev)
    beside = (o[:, :2].sum(axis=1) > 1).mean()
    assert 0.4 < beside < 0.6
    saved = autotune.current(ctx.lib)
    got = {}
    try:
        autotune.set_(ctx.lib, rr.RRX_TUNING_TRACE_LDS_STACK, depth)
        for query in ("closest", "any"):
            got[query] = ctx.intersect(accel, rays, query, "full_t")
        torch.cuda.synchronize()
    finally:
        autotune.apply(ctx.lib, saved)
    for query, hits in got.items():
        assert torch.equal(hits, _plain(ctx, accel, rays, query, "full_t")), query


@pytest.mark.parametrize("limit", [0, 1, 777, 100000])
@pytest.mark.parametrize("which", ["soup", "boxes", "scene"])
def test_device_count(ctx, dev, world, which, limit):
    say(f"pooled hits, {which}, indirect count {limit}")
    n = 5000
    rays = to_dev(_rays(n, 14), dev)
    count = torch.tensor([limit], dtype=torch.int32, device=dev)
    hits = torch.full((n * 16,), 0xAB, dtype=torch.uint8, device=dev)
    ctx.intersect(world[which], rays, "closest", "full", indirect=count, hits=hits)
    torch.cuda.synchronize()
    live = min(n, limit)
    assert torch.equal(hits[:live * 16], _plain(ctx, world[which], rays, "closest", "full")[:live * 16])
    assert bool((hits[live * 16:] == 0xAB).all())


@pytest.mark.parametrize("fetch", [32, 64, 128])
@pytest.mark.parametrize("which,extra", [("soup", 1), ("soup", 8 * 64 * 128 + 5), ("scene", 37)])
def test_pieces_hand_out_every_ray_once(ctx, dev, world, which, extra, fetch):
    n = (SHARED_SCENE if which == "scene" else SHARED) + extra
    say(f"queue pieces, {which}, {n} rays, {fetch} a piece")
    key = rr.RRX_TUNING_TRACE_2L_RAYS_PER_FETCH if which == "scene" else rr.RRX_TUNING_TRACE_RAYS_PER_FETCH
    saved = autotune.get(ctx.lib, key)
    rays = to_dev(_rays(n, 15), dev)
    want = _plain(ctx, world[which], rays, "closest", "full")
    for live in (n, SHARED + 1):
        count = torch.tensor([live], dtype=torch.int32, device=dev)
        hits = torch.full((n * 16,), 0xAB, dtype=torch.uint8, device=dev)
        try:
            autotune.set_(ctx.lib, key, fetch)
            ctx.intersect(world[which], rays, "closest", "full", indirect=count, hits=hits)
            torch.cuda.synchronize()
        finally:
            autotune.set_(ctx.lib, key, saved)
        assert torch.equal(hits[:live * 16], want[:live * 16]), live
        assert bool((hits[live * 16:] == 0xAB).all()), live


@pytest.mark.parametrize("sizes", [(1,), (64, 65, 1), (0, 3, 0, 130) * 30, (97,) * 700, (3000, 5000, 4097) * 9])
def test_batches(ctx, dev, world, sizes):
    """Lanes of one pool with their own geometry, query and output; scenes among the requests."""
    say(f"batched requests, {len(sizes)} of {max(sizes)} rays")
    rays = to_dev(_rays(max(sizes), 16), dev)
    picks = [(("soup", "dup", "boxes", "one", "scene")[k % 5], ("closest", "any")[k // 5 % 2],
              ("full", "full_t", "instance")[k % 3]) for k in range(len(sizes))]
    want = {p: _plain(ctx, world[p[0]], rays, p[1], p[2]) for p in set(picks)}
    got = ctx.intersect_batch([(world[w], rays[:n], q, out) for n, (w, q, out) in zip(sizes, picks)])
    torch.cuda.synchronize()
    for k, (hits, n, pick) in enumerate(zip(got, sizes, picks)):
        assert n == 0 or torch.equal(hits[:SIZES[pick[2]] * n], want[pick][:SIZES[pick[2]] * n]), (k, pick)
