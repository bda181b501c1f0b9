"""The float adjoint at the edges of its cases, against the oracle's FP64
gradient over the same pixel set.  The kernel's terms and sums are FP64, so what
remains is the gradient's rounding to float (2^-24) and FP64 sums: rtol 1e-6,
atol 1e-8 of the gradient scale.

* line ends: lines shorter than their width (every column within the width of
  an end), and long ones (hardly any);
* thin lines, and bands around the limit of the counted loop (64 long-axis units);
* axis-parallel and diagonal lines on grid and half-grid points;
* item counts around a wave's and a workgroup's chunks, and many chunks;
* frames of one pixel more or less than a tile, both tile and segment sizes.
"""
import numpy as np
import pytest
import torch

from cbclib_v2_amd import autograd
from tests.test_tiles_gpu import lines_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('kernel', ['biweight', 'gaussian', 'parabolic', 'triangular'])
@pytest.mark.parametrize('kind', ['short', 'thin', 'wide', 'grid', 'one', 'turn-', 'turn+', 'round+'])
@pytest.mark.parametrize('shape,opts', [((1, 63, 65), {}), ((2, 128, 64), dict(seg=16)),
                                        ((1, 65, 130), dict(tile=32, seg=16)), ((1, 70, 68), dict(tile=32))])
def test_adjoint_edges(cuda, oracle, shape, opts, kind, kernel):
    if kernel == 'triangular' and kind == 'grid':
        pytest.skip('pixels exactly on a line, where the profile has no derivative')
    rng = np.random.default_rng(len(kind) + 17 * shape[1])
    lines = lines_for(kind, rng, shape[1], shape[2]).astype(np.float32)
    idxs = rng.integers(0, shape[0], len(lines)).astype(np.int32)
    g = rng.standard_normal(shape).astype(np.float32)
    got = autograd.adjoint(torch.from_numpy(g).cuda(), torch.from_numpy(lines).cuda(), torch.from_numpy(idxs).cuda(),
                           1.3, kernel, **opts).cpu().numpy()
    ref = oracle.adjoint_f64(g.astype(np.float64), lines, idxs, 1.3, kernel, walk='f32')
    np.testing.assert_allclose(got, ref, rtol=1e-6, atol=1e-8 * np.abs(ref).max())
