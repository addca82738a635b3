"""The blend backward in segments (csrc/blend.hip, instances_per_segment): lists that end on either side of a segment, one
tile far deeper than the frame's average (its last wave walks many segments), tiles that saturate before a segment starts,
with and without the absolute-gradient variant. Image within 1e-4 and gradients within 1e-3 rel-L2 of the oracle (the bars of
test_gpu_parity); repeated backwards bit-identical."""
import dataclasses

import numpy as np
import pytest

import oracle as O
from helpers import configure, rel_l2, settings, small_case, torch_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('rows', [0, 3])
@pytest.mark.parametrize('n,logit', [(31, 0.0), (32, 0.0), (33, -1.0), (64, -2.0), (65, -2.0), (97, 3.0), (700, -3.0), (700, 2.0)])
def test_segments(n, logit, rows):
    import torch
    import efgs
    print(f'{n} instances in one tile, opacity logit {logit}, {rows} densification rows', flush=True)
    scene, app, cam = small_case(model='sh', n=n + 20, width=64, height=48, seed=n, scale_shift=1.0)
    means = scene.means.copy()
    rng = np.random.default_rng(n)
    means[:n, 0] = rng.uniform(0.15, 0.45, n)  # (tile (2, 2) of the 4 x 4 grid; the other 20 are anywhere)
    means[:n, 1] = rng.uniform(0.15, 0.45, n)
    scene = dataclasses.replace(scene, means=means, opacities=np.full((n + 20, 1), logit, np.float32))
    dev = torch.device('cuda:0')
    configure(app)
    inp = torch_inputs(scene, dev, requires_grad=True)
    info = torch.zeros((rows, n + 20) if rows else (0,), device=dev)
    image = efgs.diff_rasterize(inp['means'], inp['scales'], inp['rotations'], inp['opacities'], info, settings(cam, dev),
                                base_colors=inp['base_colors'], residual_params=inp['residual_params'])
    g = rng.normal(size=(3, cam.height, cam.width)).astype(np.float32)
    names = ('means', 'scales', 'rotations', 'opacities', 'base_colors', 'residual_params')
    up = torch.tensor(g, device=dev)
    grads = torch.autograd.grad(image, [inp[k] for k in names], up, retain_graph=True)
    first = info.clone()
    again = torch.autograd.grad(image, [inp[k] for k in names], up)
    assert all(bool((a == b).all()) for a, b in zip(grads, again))
    fw = O.render(scene, app, cam)
    ref = O.backward(scene, app, cam, fw, g, densify_rows=rows)
    assert float(np.abs(image.detach().cpu().numpy() - fw.image).max()) <= 1e-4
    for k, got in zip(names, grads):
        assert rel_l2(got.cpu().numpy(), ref[k]) <= 1e-3, k
    if rows:
        assert rel_l2(first.cpu().numpy(), ref['densification_info']) <= 1e-3


@pytest.mark.parametrize('n,shift,logit,chunks', [(16000, 2.2, -2.5, 2), (2500, 3.6, -3.0, 3), (900, 4.5, -2.0, 4)])
def test_segments_of_several_chunks(n, shift, logit, chunks):
    """Frames whose segments hold several 32-instance chunks: the forward's window stays open inside a segment and closes
    before its end, lists end on either side of one and two segments, and pixels stop inside segments."""
    import torch
    import efgs
    scene, app, cam = small_case(model='sh', n=n, width=780, height=580, seed=2, scale_shift=shift)
    opacities = np.random.default_rng(2).normal(logit, 1.0, (n, 1)).astype(np.float32)
    scene = dataclasses.replace(scene, opacities=opacities)
    fw = O.render(scene, app, cam)
    instances, lengths = len(fw.inst_keys), np.diff(fw.ranges.astype(np.int64), axis=1)
    print(f'{n} primitives, {instances} instances, lists of {lengths.min()} to {lengths.max()}', flush=True)
    segment = 32 * chunks
    assert segment == 32 * (instances // 349525 + 1) and cam.grid()[0] * cam.grid()[1] < 3072
    assert (lengths > 2 * segment).any() and ((lengths < segment).any() or n < 16000)
    g = np.random.default_rng(n).normal(size=(3, cam.height, cam.width)).astype(np.float32)
    ref = O.backward(scene, app, cam, fw, g, densify_rows=3)
    dev = torch.device('cuda:0')
    configure(app)
    names = ('means', 'scales', 'rotations', 'opacities', 'base_colors', 'residual_params')
    for rows in (0, 3):
        inp = torch_inputs(scene, dev, requires_grad=True)
        info = torch.zeros((rows, n) if rows else (0,), device=dev)

        def render():
            return efgs.diff_rasterize(inp['means'], inp['scales'], inp['rotations'], inp['opacities'], info, settings(cam, dev),
                                       base_colors=inp['base_colors'], residual_params=inp['residual_params'])
        image = render()
        grads = torch.autograd.grad(image, [inp[k] for k in names], torch.tensor(g, device=dev))
        with torch.no_grad():
            assert bool((render() == image).all())  # (a frame without a backward: no segments)
        assert float(np.abs(image.detach().cpu().numpy() - fw.image).max()) <= 1e-4
        for k, got in zip(names, grads):
            assert rel_l2(got.cpu().numpy(), ref[k]) <= 1e-3, k
        if rows:
            assert rel_l2(info.cpu().numpy(), ref['densification_info']) <= 1e-3


def test_checkpoint_memory():
    """Only a frame that gets a backward reserves checkpoints, and at most 10,923 of them (3 KB each) however many instances
    it has: bytes asked for by efgs_forward against efgs_forward_no_backward, efgs_render and efgs_update_pruning_scores, on
    frames of 10^4 and of 3 10^6 instances."""
    import ctypes
    import torch
    import efgs
    from efgs import _lib
    from efgs import rasterization as R
    dev = torch.device('cuda:0')
    for n, shift in ((400, 1.0), (2500, 5.0)):
        scene, app, cam = small_case(model='sh', n=n, width=780, height=580, seed=2, scale_shift=shift)
        configure(app)
        inp = torch_inputs(scene, dev)
        image, scores = torch.empty((3, cam.height, cam.width), device=dev), torch.zeros(n, device=dev)
        prims = R._native_primitives(inp['means'], inp['scales'], inp['rotations'], inp['opacities'], None, inp['base_colors'], inp['residual_params'], None)
        cs, keep = R._native_settings(settings(cam, dev), dev)
        h, p, s = R._rasterizer.handle, ctypes.byref(prims), ctypes.byref(cs)
        frame, counts = _lib.Frame(), (ctypes.c_int64 * 4)()
        calls = dict(
            forward=lambda a: _lib.lib.efgs_forward(h, p, s, image.data_ptr(), a.fn, a.ctx, ctypes.byref(frame), R._stream(dev)),
            no_backward=lambda a: _lib.lib.efgs_forward_no_backward(h, p, s, image.data_ptr(), a.fn, a.ctx, counts, R._stream(dev)),
            render=lambda a: _lib.lib.efgs_render(h, p, s, image.data_ptr(), 1, 0, a.fn, a.ctx, R._stream(dev)),
            scores=lambda a: _lib.lib.efgs_update_pruning_scores(h, p, s, scores.data_ptr(), a.fn, a.ctx, R._stream(dev)))
        asked = {}
        for _ in range(2):  # (the second round is laid out from the first one's counts: the same capacity in every call)
            for name, call in calls.items():
                a = _lib.WorkspaceAllocator(dev, f'memory test {name}')
                _lib.check(call(a))
                a.done()
                asked[name] = int(a.ws.requested)
        torch.cuda.synchronize()
        instances, capacity = int(frame.n_instances), int(frame.instance_capacity)
        print(f'{instances} instances, {asked}', flush=True)
        assert list(counts) == [n, frame.n_visible, instances, frame.grid_width * frame.grid_height]
        checkpoints = (min(capacity, 349525) // 32 + 1) * 192 * 16
        assert 0 <= asked['forward'] - asked['render'] - checkpoints <= 512
        assert asked['no_backward'] == asked['render']
        assert asked['scores'] <= asked['render'] + 4 * instances + image.numel() * 4 + 1024
    assert instances > 2_000_000
