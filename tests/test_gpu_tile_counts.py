"""The preprocess's tile tests (csrc/rtc/preprocess_forward.hip, count_touched_tiles) and the emission from their masks
(csrc/raster.hip, emit_wave; the last two frames: the largest grid that the fused kernel takes, and one past it): waves whose rectangles fill less than
one window of 64 tests, straddle windows, or are tested by the wave alone (more than 64 tiles; one of 2^15 tile-width products), with last waves that are partly or wholly invisible. Counts, rectangles, tile masks and the emitted
instances exactly equal the oracle's."""
import numpy as np
import pytest

import oracle as O
from helpers import check_emission, check_first_tiles, check_tile_rects, configure, read_device, settings, small_case, torch_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('model', ['precomputed', 'sh', 'neural'])
@pytest.mark.parametrize('n,width,height,shift', [(1, 16, 12, 0.0), (63, 64, 48, 0.0), (64, 130, 77, 1.0), (65, 130, 77, 3.0), (257, 333, 222, 2.0),
                                                  (700, 1600, 1200, 3.0), (130, 3000, 2400, 5.0),
                                                  (2000, 2048, 1536, 2.0), (1500, 4160, 3180, 2.0)])
def test_tile_counts(model, n, width, height, shift):
    import torch
    from efgs.rasterization import forward_with_frame, frame_tile_views, frame_views
    print(f'{model}: {n} primitives at {width}x{height}, scales x e^{shift}', flush=True)
    scene, app, cam = small_case(model=model, n=n, width=width, height=height, seed=n, scale_shift=shift)
    fw = O.render(scene, app, cam)
    dev = torch.device('cuda:0')
    configure(app)
    inp = torch_inputs(scene, dev)
    _, frame, bufs = forward_with_frame(inp['means'], inp['scales'], inp['rotations'], inp['opacities'], settings(cam, dev),
                                        **{k: inp[k] for k in ('base_colors', 'residual_params', 'mlp_weights', 'precomputed_colors')
                                           if inp.get(k) is not None})
    torch.cuda.synchronize()
    v = frame_views(frame)
    np.testing.assert_array_equal(read_device(bufs, v.n_touched, n, np.uint32), fw.n_touched)
    vis = fw.n_touched > 0
    rec = read_device(bufs, v.records, 12 * n, np.float32).reshape(n, 12)[vis]
    if vis.any():
        check_first_tiles(rec, fw, vis, *cam.grid())
        check_tile_rects(read_device(bufs, frame_tile_views(frame)[0], 2 * n, np.uint32).reshape(n, 2)[vis], fw, vis, cam.grid()[0])
        check_emission(bufs, v, frame, fw, n)
    if shift == 5.0:  # (a rectangle far past the shared windows' line)
        b = fw.bounds[vis].astype(np.int64)
        bw = (b[:, 1] + 15) // 16 - b[:, 0] // 16
        assert (bw * bw * ((b[:, 3] + 11) // 12 - b[:, 2] // 12)).max() >= 32768


@pytest.mark.parametrize('width,height,shift', [(800, 600, 2.5), (4160, 3180, 1.0)])
def test_rectangle_limits(width, height, shift):
    """Rectangles of 32 tiles (the most that emission's mask holds) and 33, of 64 (the most that are tested in the shared
    windows) and 65, in waves that hold all of these, on a grid of the fused emission and one past it."""
    import torch
    from efgs.rasterization import forward_with_frame, frame_tile_views, frame_views
    n = 3000
    scene, app, cam = small_case(model='sh', n=n, width=width, height=height, seed=n, scale_shift=shift)
    fw = O.render(scene, app, cam)
    vis = fw.n_touched > 0
    b = fw.bounds[vis].astype(np.int64)
    tiles = ((b[:, 1] + 15) // 16 - b[:, 0] // 16) * ((b[:, 3] + 11) // 12 - b[:, 2] // 12)
    assert {32, 33, 64, 65} <= set(tiles.tolist())
    dev = torch.device('cuda:0')
    configure(app)
    inp = torch_inputs(scene, dev)
    _, frame, bufs = forward_with_frame(inp['means'], inp['scales'], inp['rotations'], inp['opacities'], settings(cam, dev),
                                        base_colors=inp['base_colors'], residual_params=inp['residual_params'])
    torch.cuda.synchronize()
    v = frame_views(frame)
    np.testing.assert_array_equal(read_device(bufs, v.n_touched, n, np.uint32), fw.n_touched)
    check_first_tiles(read_device(bufs, v.records, 12 * n, np.float32).reshape(n, 12)[vis], fw, vis, *cam.grid())
    check_tile_rects(read_device(bufs, frame_tile_views(frame)[0], 2 * n, np.uint32).reshape(n, 2)[vis], fw, vis, cam.grid()[0])
    check_emission(bufs, v, frame, fw, n)
