"""Draws and gradients on both sides of the default tile size's rule (256 tiles of
64 pixels; a dozen lines per tile for float draws), against the oracle: the tile
path's tolerances, support bit-exact."""
import numpy as np
import pytest
import torch

from cbclib_v2_amd import autograd, ndimage
from tests.lines_gen import random_segments

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dtype', [np.float32, np.float64])
@pytest.mark.parametrize('shape', [(1, 1024, 1024), (1, 1025, 960), (257, 20, 30), (256, 20, 30), (1, 64, 64)])
@pytest.mark.parametrize('per_tile', [2, 13])
def test_tile_rule(cuda, oracle, shape, per_tile, dtype):
    F, H, W = shape
    n = per_tile * F * -(-H // 64) * -(-W // 64)
    rng = np.random.default_rng(n + H)
    lines = random_segments(rng, n, H, W, 2.0, 25.0, 1.0, 3.0, pad=2.0).astype(dtype)
    idxs = rng.integers(0, F, n).astype(np.int32 if dtype == np.float32 else np.int64)
    f32 = dtype == np.float32
    ref = oracle.draw_lines(np.zeros(shape, dtype), lines, idxs, 1.3, 'biweight', 'sum')
    out = torch.zeros(shape, dtype=torch.float32 if f32 else torch.float64, device='cuda')
    ndimage.draw_lines(out, torch.from_numpy(lines).cuda(), torch.from_numpy(idxs).cuda(), 1.3, 'biweight', 'sum')
    got = out.cpu().numpy()
    assert np.array_equal(got != 0, ref != 0)
    np.testing.assert_allclose(got, ref, rtol=1e-5 if f32 else 1e-12, atol=1.3e-6 if f32 else 1e-12)
    if f32:
        g = rng.standard_normal(shape).astype(np.float32)
        got = autograd.adjoint(torch.from_numpy(g).cuda(), torch.from_numpy(lines).cuda(),
                               torch.from_numpy(idxs).cuda(), 1.3, 'biweight').cpu().numpy()
        ref = oracle.adjoint_f64(g.astype(np.float64), lines, idxs, 1.3, 'biweight', walk='f32')
        np.testing.assert_allclose(got, ref, rtol=1e-6, atol=1e-8 * np.abs(ref).max())
