"""Tile ranges and the blends' tile order (csrc/raster.hip, tile_ranges_block; past 16,384 tiles order_runs_block and
tile_ranges_kernel): grids on either side of a 64-tile block, of a block's 256 tiles and of the line between the two. The
order, read back, is the tiles sorted by their size class (the instance count's leading bit and the two below it), heaviest
first, stable; the ranges equal the oracle's; frames without instances too ((0, 0) for every tile)."""
import numpy as np
import pytest

import oracle as O
from helpers import configure, read_device, settings, small_case, torch_inputs

pytestmark = pytest.mark.gpu


def size_class(n: np.ndarray) -> np.ndarray:
    """0 for an empty tile, else 1 + 4 e + the two bits of n below its leading bit e."""
    e = np.floor(np.log2(np.maximum(n, 1))).astype(np.int64)
    return np.where(n > 0, 1 + 4 * e + (np.left_shift(n, 2) >> e) - 4, 0)


@pytest.mark.parametrize('empty', [False, True])
@pytest.mark.parametrize('gw,gh', [(1, 1), (63, 1), (64, 1), (65, 1), (16, 16), (257, 1), (67, 77), (128, 128), (129, 128)])
def test_tile_order(gw, gh, empty):
    import torch
    from efgs.rasterization import forward_with_frame, frame_tile_views, frame_views
    print(f'grid {gw} x {gh}{", no instances" if empty else ""}', flush=True)
    n = 600
    scene, app, cam = small_case(model='sh', n=n, width=16 * gw - 3, height=12 * gh - 1, seed=gw, scale_shift=0.0)
    if empty:
        scene.opacities = np.full_like(scene.opacities, -20.0)
    fw = O.render(scene, app, cam)
    dev = torch.device('cuda:0')
    configure(app)
    inp = torch_inputs(scene, dev)
    for _ in range(2):  # (the second frame is launched on the first one's counts)
        image, frame, bufs = forward_with_frame(inp['means'], inp['scales'], inp['rotations'], inp['opacities'], settings(cam, dev),
                                                base_colors=inp['base_colors'], residual_params=inp['residual_params'])
        torch.cuda.synchronize()
        v = frame_views(frame)
        assert float(np.abs(image.cpu().numpy() - fw.image).max()) <= 1e-4
        ranges = read_device(bufs, v.tile_ranges, 2 * gw * gh, np.uint32).reshape(-1, 2)
        np.testing.assert_array_equal(ranges, np.zeros_like(ranges) if empty else fw.ranges)
        counts = np.diff(ranges.astype(np.int64), axis=1)[:, 0]
        np.testing.assert_array_equal(read_device(bufs, frame_tile_views(frame)[1], gw * gh, np.uint32), np.argsort(-size_class(counts), kind='stable'))
    assert empty or gw * gh == 1 or len(set(size_class(counts).tolist())) > 1
