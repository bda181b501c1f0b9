"""Stacks of many small frames with a few lines each (the tile kernels that keep less
of a tile, frames that fill part of a tile, 32-pixel tiles of frames up to 32
pixels), against the oracle: the tile path's tolerances, support bit-exact.
One frame holds several fixed-point rounds of items.  A plan made with room for
many more items (the other kernel) draws the same bits."""
import numpy as np
import pytest
import torch

from cbclib_v2_amd import autograd, batch, ndimage
from tests.lines_gen import random_segments

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('shape,per_frame', [((1100, 16, 16), 2), ((1100, 32, 32), 1), ((1100, 33, 40), 2), ((1030, 64, 64), 2),
                                             ((300, 70, 66), 3), ((1100, 8, 100), 2), ((1100, 1, 48), 2), ((1024, 20, 20), 2)])
@pytest.mark.parametrize('kernel', ['gaussian', 'triangular', 'rectangular'])
def test_small_frames(cuda, oracle, shape, per_frame, kernel):
    F, H, W = shape
    rng = np.random.default_rng(H * W)
    lines = random_segments(rng, F * per_frame, H, W, 1.0, 30.0, 0.5, 4.0, pad=3.0)
    idxs = np.repeat(np.arange(F), per_frame)
    dense = random_segments(rng, 2500, H, W, 2.0, 6.0, 0.6, 1.5)
    lines = np.concatenate([lines, dense]).astype(np.float32)
    idxs = np.concatenate([idxs, np.full(2500, F // 2)]).astype(np.int32)
    t_lines, t_idxs = torch.from_numpy(lines).cuda(), torch.from_numpy(idxs).cuda()
    for overlap, start in (('sum', 0.0), ('max', -0.25)):
        ref = oracle.draw_lines(np.full(shape, start, np.float32), lines, idxs, 1.3, kernel, overlap)
        out = torch.full(shape, start, device='cuda')
        ndimage.draw_lines(out, t_lines, t_idxs, 1.3, kernel, overlap)
        got = out.cpu().numpy()
        assert np.array_equal(got != np.float32(start), ref != np.float32(start)), overlap
        np.testing.assert_allclose(got, ref, rtol=1e-5, atol=1.3e-6, err_msg=overlap)
        plan = batch.Plan(shape, t_lines, t_idxs, kernel=kernel, headroom=64.0)
        again = torch.full(shape, start, device='cuda')
        plan.draw(again, t_lines, t_idxs, None, 1.3, kernel, overlap)
        plan.check()
        plan.close()
        assert overlap == 'sum' or torch.equal(out, again)
        # (rounds of 1023 items are cut from lists in no fixed order: sums of the dense frame may differ)
        few = torch.arange(F, device='cuda') != F // 2
        assert torch.equal(out[few], again[few])
    if kernel == 'gaussian':
        g = rng.standard_normal(shape).astype(np.float32)
        got = autograd.adjoint(torch.from_numpy(g).cuda(), t_lines, t_idxs, 1.3, kernel).cpu().numpy()
        ref = oracle.adjoint_f64(g.astype(np.float64), lines, idxs, 1.3, kernel, walk='f32')
        np.testing.assert_allclose(got, ref, rtol=1e-6, atol=1e-8 * np.abs(ref).max())
