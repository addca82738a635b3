"""Residual rows staged through the LDS (csrc/rtc/residual_rows.h) at the edges of their layout: unit counts that leave
a part of a pass, take exactly one, or are too many for the backward's staging, active degrees that end inside a pass,
and primitive counts that leave the last wave and the last block partly empty. Image within 1e-4 of the oracle, gradients
within 1e-3 rel-L2 (the bars of test_gpu_parity), gradients of inactive units and culled primitives exactly zero."""
import dataclasses

import numpy as np
import pytest

import oracle as O
from helpers import configure, rel_l2, settings, small_case, torch_inputs

pytestmark = pytest.mark.gpu

# model, units per primitive, active degree, primitives
CASES = [('sh', 15, 3, 193), ('sh', 15, 2, 64), ('sh', 15, 1, 65),
         ('sv', 1, 1, 65), ('sv', 3, 2, 257), ('sv', 4, 4, 127), ('sv', 5, 5, 129), ('sv', 9, 8, 320), ('sv', 12, 11, 191),
         ('nasg', 1, 1, 63), ('nasg', 4, 4, 130), ('nasg', 5, 5, 129), ('nasg', 7, 6, 257),
         ('nasgabor', 3, 3, 191), ('nasgabor', 5, 4, 65), ('nasgabor', 8, 7, 193)]


@pytest.mark.parametrize('model,units,degree,n', CASES, ids=lambda v: str(v))
def test_staged_rows(model, units, degree, n):
    import torch
    import efgs
    print(f'{model}: {units} units, degree {degree}, {n} primitives', flush=True)
    scene, app, cam = small_case(model=model, n=n, scale_shift=2.5, degree=degree, seed=units)
    if model != 'sh':
        wide = np.concatenate([scene.residual_params, scene.residual_params[::-1]], axis=1)  # (up to 16 units)
        scene = dataclasses.replace(scene, residual_params=np.ascontiguousarray(wide[:, :units]))
        app = dataclasses.replace(app, max_degree=units)
    dev = torch.device('cuda:0')
    configure(app)
    inp = torch_inputs(scene, dev, requires_grad=True)
    st = settings(cam, dev)
    image = efgs.diff_rasterize(inp['means'], inp['scales'], inp['rotations'], inp['opacities'], torch.empty(0, device=dev), st,
                                base_colors=inp['base_colors'], residual_params=inp['residual_params'])
    g = np.random.default_rng(3).normal(size=(3, cam.height, cam.width)).astype(np.float32)
    image.backward(torch.tensor(g, device=dev))
    fw = O.render(scene, app, cam)
    ref = O.backward(scene, app, cam, fw, g)
    assert float(np.abs(image.detach().cpu().numpy() - fw.image).max()) <= 1e-4
    for k in ('means', 'scales', 'rotations', 'opacities', 'base_colors', 'residual_params'):
        assert rel_l2(inp[k].grad.cpu().numpy(), ref[k]) <= 1e-3, k
    res = inp['residual_params'].grad.cpu().numpy().reshape(n, units, -1)
    active = degree if model != 'sh' else (degree + 1) ** 2 - 1
    assert not res[:, active:].any()
    assert not res[np.asarray(fw.n_touched) == 0].any()
