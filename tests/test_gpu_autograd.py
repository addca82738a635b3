"""The C++ autograd functions behind diff_rasterize and neural_decode (csrc/torch_binding.cpp): what autograd does around
them. Repeated backwards and backwards through saved-tensor hooks or on another stream give bit-identical gradients (the
kernels are deterministic); in-place changes of saved inputs, freed graphs, second derivatives, forward mode and vmap are
refused."""
import numpy as np
import pytest

from helpers import configure, settings, small_case, torch_inputs

pytestmark = pytest.mark.gpu

NAMES = ('means', 'scales', 'rotations', 'opacities', 'base_colors', 'residual_params')


@pytest.fixture
def case():
    import torch
    import efgs
    scene, app, cam = small_case(model='sh', n=300)
    dev = torch.device('cuda:0')
    configure(app)
    inp = torch_inputs(scene, dev, requires_grad=True)
    st = settings(cam, dev)
    grad = torch.tensor(np.random.default_rng(1).normal(size=(3, cam.height, cam.width)).astype(np.float32), device=dev)

    def render(**over):
        t = dict(inp, **over)
        return efgs.diff_rasterize(t['means'], t['scales'], t['rotations'], t['opacities'], torch.empty(0, device=dev), st,
                                   base_colors=t['base_colors'], residual_params=t['residual_params'])
    return torch, render, inp, grad


def _grads(torch, image, inp, grad, **kw):
    return [g.clone() for g in torch.autograd.grad(image, [inp[k] for k in NAMES], grad, **kw)]


def _same(a, b):
    return all(bool((x == y).all()) for x, y in zip(a, b))


def test_repeated_and_freed_backward(case):
    torch, render, inp, grad = case
    image = render()
    first = _grads(torch, image, inp, grad, retain_graph=True)
    assert _same(first, _grads(torch, image, inp, grad))
    with pytest.raises(RuntimeError, match='second time'):
        _grads(torch, image, inp, grad)


def test_saved_tensor_hooks_and_streams(case):
    torch, render, inp, grad = case
    want = _grads(torch, render(), inp, grad)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t.cuda()):
        image = render()
    assert _same(want, _grads(torch, image, inp, grad))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = _grads(torch, render(), inp, grad)
    torch.cuda.current_stream().wait_stream(side)
    assert _same(want, got)


def test_inputs_without_gradient(case):
    torch, render, inp, grad = case
    want = _grads(torch, render(), inp, grad)
    image = render(means=inp['means'].detach(), residual_params=inp['residual_params'].detach())
    got = torch.autograd.grad(image, [inp['scales'], inp['base_colors']], grad)
    assert _same([want[1], want[4]], got)
    with torch.no_grad():
        assert not render().requires_grad
    assert not render(**{k: inp[k].detach() for k in NAMES}).requires_grad


def test_refusals(case):
    torch, render, inp, grad = case
    for over, error in ((dict(means=inp['means'].double()), ValueError), (dict(scales=inp['scales'].detach().t().contiguous().t()), ValueError),
                        (dict(base_colors=inp['base_colors'].cpu()), ValueError), (dict(base_colors=torch.empty(0, device='cuda')), RuntimeError)):
        with pytest.raises(error, match='efgs'):
            render(**over)
    image = render()
    with torch.no_grad():
        inp['scales'].add_(0.0)
    with pytest.raises(RuntimeError, match='inplace'):
        _grads(torch, image, inp, grad)
    up = grad.clone().requires_grad_(True)
    (g,) = torch.autograd.grad(render(), [inp['means']], up, create_graph=True)
    with pytest.raises(RuntimeError, match='once_differentiable'):
        g.sum().backward()
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda m: render(means=m))(inp['means'].detach()[None])
    with pytest.raises((RuntimeError, NotImplementedError)):
        with torch.autograd.forward_ad.dual_level():
            render(means=torch.autograd.forward_ad.make_dual(inp['means'].detach(), torch.ones_like(inp['means'])))
    with pytest.raises(ValueError, match='image gradient'):
        image = render()
        image.grad_fn(grad[:, 1:])


def test_gradients_of_gradients(case):
    """With an upstream that requires a gradient, the gradients hold the same values, may be changed in place, and raise when
    they are differentiated; with one that does not, they require no gradient."""
    torch, render, inp, grad = case
    want = _grads(torch, render(), inp, grad)
    up = grad.clone().requires_grad_(True)
    got = torch.autograd.grad(render(), [inp[k] for k in NAMES], up, create_graph=True)
    assert _same(want, got) and all(g.requires_grad for g in got)
    got[0].mul_(2.0)
    assert bool((got[0] == 2.0 * want[0]).all())
    for g in got:
        with pytest.raises(RuntimeError, match='differentiate twice'):
            g.sum().backward(retain_graph=True)
    assert not any(g.requires_grad for g in torch.autograd.grad(render(), [inp[k] for k in NAMES], grad, create_graph=True))
