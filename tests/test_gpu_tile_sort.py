"""The per-tile sort (csrc/tile_sort.h) at the edges of its paths: one-tile frames whose run length sits on either side of
a register network's size, of the LDS slab (512 keys) and of a merge pass (256 2^k), with equal depths among the keys. The
sorted order is exactly (depth key, primitive)."""
import dataclasses

import numpy as np
import pytest

from helpers import configure, read_device, settings, small_case, torch_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n', [1, 64, 65, 128, 129, 192, 193, 256, 257, 320, 511, 512, 513, 767, 768, 769, 1024, 1025, 1300, 2048, 2049, 5000])
def test_run_lengths(n):
    import torch
    from efgs.rasterization import forward_with_frame, frame_views
    print(f'one tile, {n} instances', flush=True)
    scene, app, cam = small_case(model='sh', n=n, width=16, height=12, seed=n)
    rng = np.random.default_rng(n)
    means = np.zeros((n, 3), np.float32)
    means[:, :2] = rng.uniform(-0.2, 0.2, (n, 2))
    means[:, 2] = rng.integers(0, max(2, n // 3), n) / np.float32(n)  # (about three primitives per depth)
    scene = dataclasses.replace(scene, means=means, opacities=np.full((n, 1), -1.0, np.float32))
    dev = torch.device('cuda:0')
    configure(app)
    inp = torch_inputs(scene, dev)
    _, frame, bufs = forward_with_frame(inp['means'], inp['scales'], inp['rotations'], inp['opacities'], settings(cam, dev),
                                        base_colors=inp['base_colors'], residual_params=inp['residual_params'])
    torch.cuda.synchronize()
    assert frame.n_instances == n
    v = frame_views(frame)
    depth = read_device(bufs, v.depth_keys, n, np.uint32)
    order = np.lexsort((np.arange(n), depth))
    slots = read_device(bufs, v.tile_sorted_instances, n, np.uint32)
    prims = read_device(bufs, v.instance_primitive, n, np.uint32)
    np.testing.assert_array_equal(prims[slots], order)
    assert not read_device(bufs, v.tile_sorted_keys, n, np.uint16).any()


@pytest.mark.parametrize('n', [16128, 16129, 16385, 40000])
def test_long_runs(n):
    """Runs past one batch of 63 merge blocks (16,128 outputs), with a last block of one key."""
    test_run_lengths(n)
