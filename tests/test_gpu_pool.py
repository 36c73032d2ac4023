"""GPU tests of the pooled traversal (trace.hip): a wave's last rays are
traversed together from one list in LDS.  Hits must be those of the plain
kernels, which walk one ray per lane in depth-first order, bit for bit: same
arithmetic, closest hits independent of the order, any hit the first in
depth-first order.  Ray counts sit at the edges of a wave's share (one ray,
a part of a wave, a full wave, one ray more than every wave can hold)."""
import numpy as np
import pytest
import torch

from radeonrays_sdk_amd import autotune, rr, scenes
from tests.gpu_util import say, to_dev

pytestmark = pytest.mark.gpu

SHARED = 256 * 16 * 64  # rays that 16 waves per CU hold on 256 CUs


def _plain(ctx, accel, rays, query, output):
    saved = autotune.current(ctx.lib)
    try:
        autotune.set_(ctx.lib, rr.RRX_TUNING_TRACE_PLAIN, 1)
        hits = ctx.intersect(accel, rays, query, output)
        torch.cuda.synchronize()
        return hits
    finally:
        autotune.apply(ctx.lib, saved)


def _soup_rays(n, seed, tmax=1e30):
    rng = np.random.default_rng(seed)
    o = rng.uniform(-0.2, 1.2, size=(n, 3)).astype(np.float32)
    return scenes.make_rays(o, scenes.unit_sphere(n, rng), 0.0, tmax)


@pytest.fixture(scope="module")
def world(ctx, dev):
    """A restructured soup, a coarse duplicate-heavy mesh (equal boxes and
    equal distances), a one-triangle mesh, and a scene of all three."""
    rng = np.random.default_rng(5)
    v, i = scenes.triangle_soup(9000, rng, sigma=0.03)
    soup = ctx.build_geometry(to_dev(v, dev), to_dev(i, dev), restructure=True)
    v, i = scenes.triangle_soup(40, rng, sigma=0.2)
    dup = ctx.build_geometry(to_dev(v, dev), to_dev(np.tile(i, (30, 1)), dev))
    one = ctx.build_geometry(to_dev(v[:3], dev), to_dev(i[:1], dev))
    n = 50
    xf = scenes.random_transforms(rng, n, trans=0.8)
    scene = ctx.build_scene([(soup, dup, one)[k % 3] for k in range(n)], xf)
    return {"soup": soup, "dup": dup, "one": one, "scene": scene}


@pytest.mark.parametrize("query", ["closest", "any"])
@pytest.mark.parametrize("which", ["soup", "dup", "one", "scene"])
def test_pooled_hits_equal_plain(ctx, dev, world, which, query):
    say(f"pooled traversal, {which}, {query}")
    accel = world[which]
    counts = [1, 2, 5, 64, 65, 1000, 4097, SHARED // 64 * 3 + 1]
    if which == "soup":
        counts += [SHARED - 1, SHARED, SHARED + 1]
    rays = to_dev(_soup_rays(max(counts), 11, 1e30 if query == "closest" else 0.7), dev)
    output = "full_t"
    for n in counts:
        got = ctx.intersect(accel, rays[:n], query, output)
        torch.cuda.synchronize()
        assert torch.equal(got, _plain(ctx, accel, rays[:n], query, output)), n


@pytest.mark.parametrize("depth", [8, 16, 32])
@pytest.mark.parametrize("which", ["soup", "scene"])
def test_pooled_hits_at_every_stack_depth(ctx, dev, world, which, depth):
    """The pool lies in the stacks' LDS, so its room follows their depth."""
    say(f"pooled traversal, {which}, LDS stack {depth}")
    rays = to_dev(_soup_rays(70001, 12), dev)
    saved = autotune.current(ctx.lib)
    try:
        autotune.set_(ctx.lib, rr.RRX_TUNING_TRACE_LDS_STACK, depth)
        got = {q: ctx.intersect(world[which], rays, q, "full") for q in ("closest", "any")}
        torch.cuda.synchronize()
    finally:
        autotune.apply(ctx.lib, saved)
    for q, hits in got.items():
        assert torch.equal(hits, _plain(ctx, world[which], rays, q, "full")), q


def test_pooled_batch_mixes_queries(ctx, dev, world):
    """Batched requests: lanes of one pool with their own geometry, query and output."""
    say("pooled traversal, batched requests")
    rng = np.random.default_rng(13)
    requests = []
    for k in range(60):
        n = int(rng.integers(0, 700))
        accel = world[("soup", "dup", "one")[k % 3]]
        requests.append((accel, to_dev(_soup_rays(n, 100 + k), dev), ("closest", "any")[k % 2],
                         ("full", "full_t", "instance")[k % 3]))
    got = ctx.intersect_batch(requests)
    torch.cuda.synchronize()
    for hits, (accel, rays, query, output) in zip(got, requests):
        if rays.shape[0]:
            assert torch.equal(hits, _plain(ctx, accel, rays, query, output)), (query, output)


@pytest.mark.parametrize("limit", [0, 1, 777, 100000])
def test_pooled_shares_follow_the_device_count(ctx, dev, world, limit):
    """An indirect ray count smaller than the recorded one: rays past it are not touched."""
    say(f"pooled traversal, indirect count {limit}")
    n = 5000
    rays = to_dev(_soup_rays(n, 14), dev)
    count = torch.tensor([limit], dtype=torch.int32, device=dev)
    hits = torch.full((n * 16,), 0xAB, dtype=torch.uint8, device=dev)
    ctx.intersect(world["soup"], rays, "closest", "full", indirect=count, hits=hits)
    torch.cuda.synchronize()
    live = min(n, limit)
    if live:
        assert torch.equal(hits[:live * 16], _plain(ctx, world["soup"], rays[:live], "closest", "full"))
    assert bool((hits[live * 16:] == 0xAB).all())


@pytest.mark.parametrize("fetch", [32, 64, 128])
@pytest.mark.parametrize("which,extra", [("soup", 1), ("soup", 8 * 64 * 128 + 5), ("scene", 37)])
def test_pieces_hand_out_every_ray_once(ctx, dev, world, which, extra, fetch):
    """More rays than equal shares hold: a first piece per wave, the rest from the queues; an indirect count cuts the
    queues shorter than the pieces were sized for."""
    n = SHARED + extra
    say(f"queue pieces, {which}, {n} rays, {fetch} a piece")
    key = rr.RRX_TUNING_TRACE_2L_RAYS_PER_FETCH if which == "scene" else rr.RRX_TUNING_TRACE_RAYS_PER_FETCH
    saved = autotune.get(ctx.lib, key)
    rays = to_dev(_soup_rays(n, 15), dev)
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


@pytest.mark.parametrize("sizes", [(1,), (64, 65, 1), (0, 3, 0, 130) * 30, (97,) * 700, (256,) * 1700])
def test_batch_chunks_are_found_among_any_number_of_requests(ctx, dev, world, sizes):
    """One chunk to more chunks than the grid has waves; the request of a chunk is searched 64 at a time."""
    say(f"batched requests, {len(sizes)} of {max(sizes)} rays")
    rays = to_dev(_soup_rays(max(sizes), 16), dev)
    want = {(w, q): _plain(ctx, world[w], rays, q, "full") for w in ("soup", "dup") for q in ("closest", "any")}
    picks = [(("soup", "dup")[k % 2], ("closest", "any")[k // 2 % 2]) for k in range(len(sizes))]
    got = ctx.intersect_batch([(world[w], rays[:n], q, "full") for n, (w, q) in zip(sizes, picks)])
    torch.cuda.synchronize()
    for k, (hits, n, pick) in enumerate(zip(got, sizes, picks)):
        assert n == 0 or torch.equal(hits[:16 * n], want[pick][:16 * n]), (k, pick)
