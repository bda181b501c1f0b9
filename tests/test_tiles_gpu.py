"""The tile kernel of float images at the edges of its cases, against the
oracle: support bit-exact, values within the tile path's tolerance (rtol 1e-5,
atol 1e-6 * max_val: float profile values and the fixed-point step).

* line ends: lines shorter than their width (every column within the width of
  an end), and long ones (hardly any);
* bands: widths below half a pixel, and bands of 60 to 70 short-axis pixels
  around the limit of the counted loop (64 long-axis units);
* exactly axis-parallel and diagonal lines on grid and half-grid points, whose
  pixels fall on the band's edge;
* item counts around the waves' turns (1, 4 x 32 +- 1) and above several
  fixed-point rounds (4300);
* frames of one pixel more or less than a tile, rows of no multiple of four.
"""
import numpy as np
import pytest
import torch

from cbclib_v2_amd import ndimage
from tests.lines_gen import random_segments

pytestmark = pytest.mark.gpu

KERNELS = ['biweight', 'gaussian', 'parabolic', 'rectangular', 'triangular']


def lines_for(kind, rng, H, W):
    if kind == 'short':
        return random_segments(rng, 300, H, W, 0.0, 6.0, 1.0, 8.0, pad=8.0)
    if kind == 'thin':
        return random_segments(rng, 200, H, W, 1.0, 90.0, 0.05, 0.6, pad=4.0)
    if kind == 'wide':
        return random_segments(rng, 12, H, W, 30.0, 160.0, 28.0, 70.0, pad=20.0)
    if kind == 'grid':
        ln = random_segments(rng, 200, H, W, 4.0, 80.0, 1.0, 5.0, pad=4.0)
        ln = np.round(ln * 2) / 2
        ln[::3, 3] = ln[::3, 1]                                        # along x
        ln[1::3, 2] = ln[1::3, 0]                                      # along y
        d = ln[2::3, 2] - ln[2::3, 0]
        ln[2::3, 3] = ln[2::3, 1] + d                                  # diagonal
        return ln
    n = {'one': 1, 'turn-': 127, 'turn': 128, 'turn+': 129, 'round+': 4300}[kind]
    ln = random_segments(rng, n, 40, 40, 3.0, 7.0, 0.5, 3.0)
    ln[:, :4] += 4.0
    return ln


@pytest.mark.parametrize('overlap', ['sum', 'max'])
@pytest.mark.parametrize('kind', ['short', 'thin', 'wide', 'grid', 'one', 'turn-', 'turn', 'turn+', 'round+'])
@pytest.mark.parametrize('shape,opts', [((1, 63, 65), {}), ((2, 128, 64), {}), ((1, 65, 130), dict(tile=32, seg=16)),
                                        ((1, 96, 64), dict(threads=64)), ((1, 70, 68), dict(seg=16))])
def test_tile_edges(cuda, oracle, kind, shape, opts, overlap):
    rng = np.random.default_rng(len(kind) + 17 * shape[1])
    lines = lines_for(kind, rng, shape[1], shape[2]).astype(np.float32)
    idxs = rng.integers(0, shape[0], len(lines)).astype(np.int32)
    for kernel in KERNELS:
        ref = oracle.draw_lines(np.full(shape, -0.25 if overlap == 'max' else 0.0, np.float32), lines, idxs, 1.3, kernel,
                                overlap)
        out = torch.full(shape, -0.25 if overlap == 'max' else 0.0, dtype=torch.float32, device='cuda')
        ndimage.draw_lines(out, torch.from_numpy(lines).cuda(), torch.from_numpy(idxs).cuda(), 1.3, kernel, overlap,
                           **opts)
        got = out.cpu().numpy()
        init = np.float32(-0.25 if overlap == 'max' else 0.0)
        assert np.array_equal(got != init, ref != init), kernel
        np.testing.assert_allclose(got, ref, rtol=1e-5, atol=1.3e-6, err_msg=kernel)
