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
