"""The pruning-score walk (csrc/blend.hip, blend_scores_kernel): lists that end on either side of a 32-Gaussian chunk, of the
two-chunk window and of a four-step group, tiles that saturate before their list ends (the rest scores 0) and tiles cut by
the image's edge. The bars of test_gpu_pruning."""
import dataclasses

import numpy as np
import pytest

import oracle as O
from helpers import small_case
from test_gpu_pruning import _check, _scores

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('logit', [-2.0, 4.0])
@pytest.mark.parametrize('n,width,height', [(1, 16, 12), (4, 16, 12), (31, 16, 12), (32, 16, 12), (33, 19, 17), (64, 19, 17), (65, 16, 12), (96, 16, 12),
                                            (97, 33, 13), (300, 16, 12)])
def test_score_walk(n, width, height, logit):
    print(f'{n} Gaussians at {width}x{height}, opacity logit {logit}', flush=True)
    scene, app, cam = small_case(model='sh', n=n, width=width, height=height, seed=n)
    rng = np.random.default_rng(n)
    means = rng.uniform(-0.3, 0.3, (n, 3)).astype(np.float32)
    scene = dataclasses.replace(scene, means=means, opacities=np.full((n, 1), logit, np.float32))
    fw = O.render(scene, app, cam)
    _check(_scores(scene, app, cam), O.pruning_scores(cam, fw), f'{n}')
