"""Lobe gradients near the antipole (csrc/rtc/appearance_lobes.h): lobes whose axis points delta away from the reversed view
direction, where 1 - vz^2 and 1 + vz cancel. The residual gradients of the frame angles against autograd of the lobe in 64
bits, with the device's own base-colour gradients upstream. Bound: the fp32 direction (two roundings, 1.2e-7) and the frame
axis (a tanh or sech of three, 2e-7) put a relative error of r = 3.2e-7 / delta on the components across the axis. The
gradients go as 1 / delta (r once), times E = K^Ke whose exponent Ke log K, with Ke <= 1 a ratio of those components and
log K = 2 log(delta / 2), follows them twice over: r (1 + 2 |log K|), and 1e-4 for the arithmetic behind. (1 + vz taken as a
difference is off by 1.2e-7 / (delta^2 / 2), a quarter at delta 1e-3.)"""
import dataclasses

import numpy as np
import pytest

from helpers import configure, settings, small_case, torch_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('model', ['nasg', 'nasgabor'])
@pytest.mark.parametrize('delta', [1e-3, 4e-3, 3e-2])
def test_lobe_antipole(model, delta):
    import torch
    import efgs
    import torch_ref
    print(f'{model}, delta {delta}', flush=True)
    n, stride = 200, 8 if model == 'nasg' else 9
    scene, app, cam = small_case(model=model, n=n, seed=3)
    d = torch.nn.functional.normalize(torch.tensor(scene.means, dtype=torch.float64) - torch.tensor(np.asarray(cam.position), dtype=torch.float64), dim=-1)
    z = -d.numpy()
    aimed = z[:, 1] > 0.02  # (a frame's axis has a positive y)
    theta = np.arctan2(z[:, 1], z[:, 0]) + delta / np.sqrt(1.0 - z[:, 2] ** 2)
    aimed &= (theta > 0.02) & (theta < np.pi - 0.02) & (np.abs(z[:, 2]) < 0.999)
    raw = scene.residual_params.reshape(n, -1, stride).copy()
    raw[aimed, 0, 0] = np.arctanh(np.cos(theta[aimed]))
    raw[aimed, 0, 1] = np.arctanh(z[aimed, 2])
    raw[aimed, 0, 3:5] = 0.0
    if model == 'nasgabor':
        raw[aimed, 0, 5] = -0.5
    raw[aimed, 0, -3:] = 1.0
    scene = dataclasses.replace(scene, residual_params=raw.reshape(scene.residual_params.shape).astype(np.float32))
    dev = torch.device('cuda:0')
    configure(app)
    inp = torch_inputs(scene, dev, requires_grad=True)
    image = efgs.diff_rasterize(inp['means'], inp['scales'], inp['rotations'], inp['opacities'], torch.zeros((0,), device=dev), settings(cam, dev),
                                base_colors=inp['base_colors'], residual_params=inp['residual_params'])
    g = torch.tensor(np.random.default_rng(0).normal(size=(3, cam.height, cam.width)).astype(np.float32), device=dev)
    g_base, g_res = torch.autograd.grad(image, [inp['base_colors'], inp['residual_params']], g)
    p = torch.tensor(scene.residual_params.reshape(n, -1, stride), dtype=torch.float64, requires_grad=True)
    want, = torch.autograd.grad(torch_ref.lobe_residual(p, d, cam.degree, app.res_act, model == 'nasgabor'), p, g_base.cpu().double().reshape(n, 3))
    got, want = g_res.cpu().double().reshape(p.shape).numpy()[aimed, 0, :3], want.numpy()[aimed, 0, :3]
    size = np.abs(want).max(1)
    assert (size > 0).sum() >= 10
    worst = (np.abs(got - want).max(1)[size > 0] / size[size > 0]).max()
    print(f'{int(aimed.sum())} lobes, worst relative error {worst:.2e}', flush=True)
    assert worst <= 3.2e-7 / delta * (1.0 + 4.0 * np.log(2.0 / delta)) + 1e-4
