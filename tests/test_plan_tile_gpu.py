"""A plan and the eager calls work on the same tiles by default, whatever the
number of lines: images and gradients of the two are identical, also when
the plan was made for more lines than are drawn."""
import numpy as np
import pytest
import torch

from cbclib_v2_amd import autograd, batch, ndimage
from tests.lines_gen import random_segments

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('made_for', [1, 40])
@pytest.mark.parametrize('per_tile', [1, 5, 11, 12, 13])
def test_plan_and_eager_defaults(cuda, per_tile, made_for):
    shape = (2, 128, 200)                       # 16 tiles of 64 pixels
    rng = np.random.default_rng(per_tile)
    n = 16 * per_tile
    lines = random_segments(rng, n * made_for, *shape[1:], 2.0, 150.0, 1.0, 6.0, pad=5.0).astype(np.float32)
    idxs = rng.integers(0, 2, n * made_for).astype(np.int32)
    t_lines, t_idxs = torch.from_numpy(lines).cuda(), torch.from_numpy(idxs).cuda()
    g = torch.from_numpy(rng.standard_normal(shape).astype(np.float32)).cuda()
    plan = batch.Plan(shape, t_lines, t_idxs, kernel='biweight')
    t_lines, t_idxs = t_lines[:n].contiguous(), t_idxs[:n].contiguous()
    out, ref = torch.zeros(shape, device='cuda'), torch.zeros(shape, device='cuda')
    plan.draw(out, t_lines, t_idxs)
    got = plan.adjoint(g, t_lines, t_idxs)
    plan.check()
    plan.close()
    ndimage.draw_lines(ref, t_lines, t_idxs, 1.0, 'biweight')
    assert torch.equal(out, ref)
    assert torch.equal(got, autograd.adjoint(g, t_lines, t_idxs, 1.0, 'biweight'))
