"""GPU tests of the tree builder (tree_device.h) at the edges of its windows
(512 leaves per workgroup), of its groups (48 windows) and of what a group can
take at a time (512 published subtrees): nodes must equal the oracle's
restated build, whose hierarchy is emitted top-down and refitted, node for
node, also into a result buffer full of stale bytes."""
import numpy as np
import pytest
import torch

import oracle
from radeonrays_sdk_amd import autotune, rr, scenes
from tests.gpu_util import nodes_equal, say, to_dev

pytestmark = pytest.mark.gpu

WINDOW, GROUP = 512, 48


def _check(ctx, dev, v, i):
    req = ctx.geometry_requirements(i.shape[0], v.shape[0], False)
    result = torch.full((req.result_buffer_size,), 0xA5, dtype=torch.uint8, device=dev)
    scratch = torch.full((req.temporary_build_buffer_size,), 0x5A, dtype=torch.uint8, device=dev)
    accel = ctx.build_geometry(to_dev(v, dev), to_dev(i, dev), result=result, scratch=scratch)
    torch.cuda.synchronize()
    ok, msg = nodes_equal(accel.buffer.cpu().numpy(), oracle.build_blas(v, i, False))
    assert ok, msg


@pytest.mark.parametrize("n", [WINDOW - 1, WINDOW, WINDOW + 1, 2 * WINDOW, 2 * WINDOW + 1, GROUP * WINDOW - 1,
                               GROUP * WINDOW, GROUP * WINDOW + 1, 2 * GROUP * WINDOW + 300])
def test_tree_at_window_and_group_edges(ctx, dev, n):
    say(f"tree of {n} soup triangles")
    _check(ctx, dev, *scenes.triangle_soup(n, scenes.rng_for(70, n)))


@pytest.mark.parametrize("kind", ["equal", "pairs", "line", "chain"])
def test_tree_of_skewed_codes(ctx, dev, kind):
    """Equal codes (prefixes continue into the key position), codes along one
    axis, and geometrically spaced ones (deep chains of merges)."""
    n = 20 * WINDOW + 77
    say(f"tree of {n} {kind} codes")
    k = np.arange(n)
    x = {"equal": np.zeros(n), "pairs": (k // 2) / n, "line": k / n, "chain": 2.0 ** -(k % 40)}[kind]
    c = np.stack([x, np.zeros(n), np.zeros(n)], axis=1)
    c[0, :], c[1, :] = 0.0, 1.0
    tri = np.array([[-1, 0, 0], [1, 0, 0], [0, 1, 0]]) * 1e-4
    v = (c[:, None, :] + tri).astype(np.float32).reshape(-1, 3)
    _check(ctx, dev, v, np.arange(3 * n, dtype=np.int32).reshape(n, 3))


def test_tree_whose_groups_publish_more_than_a_window(ctx, dev):
    """A terrain's windows publish about twelve subtrees each, so a group's
    are merged in two parts."""
    v, i = scenes.heightfield_mesh(360)
    say(f"tree of a terrain of {i.shape[0]} triangles")
    _check(ctx, dev, v, i)


def test_batched_trees_share_windows(ctx, dev):
    """Meshes of a batch that share a workgroup, fill one exactly, or start one of their own."""
    sizes = [1, 2, 63, 64, 65, 448, 449, 511, 512, 513, 1024, 1025, 3000, 16384] + [100] * 40
    say(f"batched trees of {len(sizes)} meshes")
    meshes = [scenes.triangle_soup(n, scenes.rng_for(71, k)) for k, n in enumerate(sizes)]
    accels = ctx.build_geometry_batch([(to_dev(v, dev), to_dev(i, dev)) for v, i in meshes])
    torch.cuda.synchronize()
    for k, ((v, i), a) in enumerate(zip(meshes, accels)):
        ok, msg = nodes_equal(a.buffer.cpu().numpy(), oracle.build_blas(v, i, False))
        assert ok, f"mesh {k} (n={sizes[k]}): {msg}"


@pytest.mark.parametrize("leaves", [5, 7, 9])
@pytest.mark.parametrize("kind", ["soup", "growing"])
def test_treelets_opened_deeper_than_the_fetched_levels(ctx, dev, kind, leaves):
    """Restructured nodes equal the oracle's; triangles whose sizes grow along their order make treelets that open
    one side again and again, below the three levels fetched with a treelet's root."""
    n = 3000
    say(f"treelets of {leaves} leaves, {kind}")
    v, i = scenes.triangle_soup(n, scenes.rng_for(71, leaves))
    if kind == "growing":
        c = np.stack([np.arange(n) / n] * 3, axis=1)
        size = 1e-5 * 1.5 ** (np.arange(n) % 29)
        tri = np.array([[-1, 0, 0.3], [1, 0.2, 0], [0, 1, -0.3]])
        v = (c[:, None, :] + size[:, None, None] * tri).astype(np.float32).reshape(-1, 3)
        i = np.arange(3 * n, dtype=np.int32).reshape(n, 3)
    saved = autotune.get(ctx.lib, rr.RRX_TUNING_TREELET_LEAVES)
    try:
        autotune.set_(ctx.lib, rr.RRX_TUNING_TREELET_LEAVES, leaves)
        accel = ctx.build_geometry(to_dev(v, dev), to_dev(i, dev), restructure=True)
        torch.cuda.synchronize()
    finally:
        autotune.set_(ctx.lib, rr.RRX_TUNING_TREELET_LEAVES, saved)
    ok, msg = nodes_equal(accel.buffer.cpu().numpy(), oracle.build_blas(v, i, True, leaves))
    assert ok, msg
