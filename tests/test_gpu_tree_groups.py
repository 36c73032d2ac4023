"""GPU tests of tree groups that publish more subtrees than a workgroup takes
at a time (tree_device.h, FinishTree), the root's group among them.  How many
a group publishes is counted from the oracle's tree, so that the tests cannot
stop covering the merge in parts unnoticed."""
import numpy as np
import pytest
import torch

import oracle
from radeonrays_sdk_amd import scenes
from tests.gpu_util import nodes_equal, say, to_dev

pytestmark = pytest.mark.gpu

WINDOW, GROUP = 512, 48


def _published(buf, n):
    """Per window of leaves, its subtrees whose parents reach beyond it."""
    nodes = oracle.nodes_of(buf)
    child = nodes[:n - 1][:, [3, 7]].astype(np.int64)
    first = np.concatenate([np.full(n - 1, -1), np.arange(n)])
    last = first.copy()
    order = [0]  # parents before children
    for k in order:
        order += [c for c in child[k] if c < n - 1]
    for k in reversed(order):
        first[k], last[k] = first[child[k]].min(), last[child[k]].max()
    inside = first // WINDOW == last // WINDOW
    whole = inside[child] & ~inside[:n - 1, None]
    return np.bincount((first[child] // WINDOW)[whole], minlength=(n + WINDOW - 1) // WINDOW)


@pytest.mark.parametrize("res,seed,root", [(111, 2, True), (360, scenes.SEED_BASE + 1, False)])
def test_group_of_more_subtrees_than_a_window(ctx, dev, res, seed, root):
    """24,200 triangles: the only group, whose last part holds the tree's root; 257,762: groups below the root's."""
    v, i = scenes.heightfield_mesh(res, seed=seed)
    n = i.shape[0]
    ref = oracle.build_blas(v, i, False)
    published = _published(ref, n)
    groups = [int(published[k:k + GROUP].sum()) for k in range(0, len(published), GROUP)]
    say(f"tree of {n} terrain triangles, {len(groups)} groups of up to {max(groups)} subtrees")
    assert max(groups) > WINDOW and (len(groups) == 1) == root
    result = torch.full((ctx.geometry_requirements(n, v.shape[0], False).result_buffer_size,), 0xA5, dtype=torch.uint8,
                        device=dev)
    accel = ctx.build_geometry(to_dev(v, dev), to_dev(i, dev), result=result)
    torch.cuda.synchronize()
    ok, msg = nodes_equal(accel.buffer.cpu().numpy(), ref)
    assert ok, msg


def test_batched_group_of_more_subtrees_than_a_window(ctx, dev):
    """The same in a batch, between meshes that share workgroups."""
    meshes = [scenes.heightfield_mesh(111, seed=2), scenes.triangle_soup(300, scenes.rng_for(95)),
              scenes.heightfield_mesh(111, seed=2), scenes.triangle_soup(40, scenes.rng_for(96))]
    say("batched trees whose root group is merged in parts")
    accels = ctx.build_geometry_batch([(to_dev(v, dev), to_dev(i, dev)) for v, i in meshes])
    torch.cuda.synchronize()
    for k, ((v, i), a) in enumerate(zip(meshes, accels)):
        ok, msg = nodes_equal(a.buffer.cpu().numpy(), oracle.build_blas(v, i, False))
        assert ok, f"mesh {k}: {msg}"
