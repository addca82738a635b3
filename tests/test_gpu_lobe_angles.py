"""Lobe angles near zero (csrc/rtc/appearance_lobes.h, lobe_tanh) on both sides of the line between its two forms: Gaussians
on the camera's axis, whose view direction is (0, 0, 1), so that vx = -sin(phi) cos(tau) and the gradient of the raw tau is
proportional to cos(tau) = tanh(raw): its relative error is the tanh's, and that of about 40 operations and hardware
functions behind it (at most 1.2e-7 each), of which log K amplifies its argument's by up to 1 / 0.1 (K in [0.1, 0.9]):
1e-5. (A tanh that is off by 6e-8 in absolute terms: 6e-4 at a raw angle of 1e-4.) Against autograd of the lobe in 64 bits,
with the device's own base-colour gradients upstream."""
import dataclasses

import numpy as np
import pytest

from helpers import configure, settings, small_case, torch_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('model', ['nasg', 'nasgabor'])
def test_small_lobe_angles(model):
    import torch
    import efgs
    import torch_ref
    print(model, flush=True)
    n, stride = 48, 8 if model == 'nasg' else 9
    scene, app, cam = small_case(model=model, n=n, seed=5, scale_shift=4.0)
    rng = np.random.default_rng(5)
    means = np.zeros((n, 3), np.float32)
    means[:, 2] = np.linspace(-5.0, 5.0, n)
    raw = scene.residual_params.reshape(n, 8, stride).copy()
    raw[..., 1] = np.arctanh(rng.uniform(0.1, 0.8, (n, 8)) * rng.choice([-1.0, 1.0], (n, 8)))
    raw[..., 2] = np.exp(rng.uniform(np.log(1e-4), np.log(1.5), (n, 8))) * rng.choice([-1.0, 1.0], (n, 8))
    raw[0, :, 2] = [0.69999, 0.7, 0.70001, -0.69999, -0.7, -0.70001, 1e-6, -1e-6]
    raw[..., 3:5] = 0.0
    if model == 'nasgabor':
        raw[..., 5] = -2.0  # (a factor near 1 that does not pass through 0)
    raw[..., -3:] = 1.0
    scene = dataclasses.replace(scene, means=means, opacities=np.full((n, 1), -3.0, np.float32),
                                base_colors=np.full((n, 3), 1.0, np.float32), residual_params=raw.reshape(scene.residual_params.shape).astype(np.float32))
    dev = torch.device('cuda:0')
    configure(app)
    inp = torch_inputs(scene, dev, requires_grad=True)
    image = efgs.diff_rasterize(inp['means'], inp['scales'], inp['rotations'], inp['opacities'], torch.zeros((0,), device=dev), settings(cam, dev),
                                base_colors=inp['base_colors'], residual_params=inp['residual_params'])
    g = torch.tensor(np.random.default_rng(0).uniform(0.5, 1.0, size=(3, cam.height, cam.width)).astype(np.float32), device=dev)
    g_base, g_res = torch.autograd.grad(image, [inp['base_colors'], inp['residual_params']], g)
    p = torch.tensor(scene.residual_params.reshape(n, 8, stride), dtype=torch.float64, requires_grad=True)
    d = torch.tensor([[0.0, 0.0, 1.0]], dtype=torch.float64).expand(n, 3)
    want, = torch.autograd.grad(torch_ref.lobe_residual(p, d, 8, app.res_act, model == 'nasgabor'), p, g_base.cpu().double().reshape(n, 3))
    got, want = g_res.cpu().double().reshape(p.shape).numpy()[..., 2], want.numpy()[..., 2]
    seen = np.abs(want) > 0
    assert seen.mean() > 0.9
    worst = (np.abs(got - want)[seen] / np.abs(want[seen])).max()
    print(f'{int(seen.sum())} lobes, worst relative error {worst:.2e}', flush=True)
    assert worst <= 1e-5
