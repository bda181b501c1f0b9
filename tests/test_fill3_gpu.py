"""The plane fills of 3D lines at the edges of their cases, against the oracle:
max bit-exact; sums within the rounding of at most 64 float additions
(64 * 2^-24 < 5e-6, 64 * 2^-53 < 1e-14), support bit-exact.

* planes per wave (16) and per workgroup (64): line counts whose planes end a
  wave anywhere, a single short line among them;
* patches in LDS: widths whose planes need 1 x 1 up to more than the whole
  patch, so that planes with, without and partly outside of one are mixed;
* volumes one voxel thick along an axis, lines that reach outside;
* lines along one axis, and on the diagonals of two and three axes, between grid
  points, whose voxels fall on the limit of the width (the reference's walk does
  not end for lines between some half-grid points).
"""
import numpy as np
import pytest
import torch

from cbclib_v2_amd import ndimage
from tests.lines_gen import segments3

pytestmark = pytest.mark.gpu


def lines_for(kind, rng, shape):
    if kind == 'one':
        return segments3(rng, 1, shape, 2.0, 0.7, 0.7, 0.0)
    if kind == 'thin':
        return segments3(rng, 37, shape, 12.0, 0.05, 0.9, 2.0)
    if kind == 'wide':
        return segments3(rng, 13, shape, 9.0, 3.0, 12.0, 4.0)
    if kind == 'mixed':
        return segments3(rng, 64, shape, 15.0, 0.3, 6.0, 3.0)
    ln = segments3(rng, 60, shape, 12.0, 0.5, 4.0, 1.0)
    ln = np.round(ln)
    for k, keep in enumerate(((0,), (1,), (2,), (0, 1), (1, 2), (0, 1, 2))):
        for row in ln[k::6]:
            d = max(1.0, np.abs(row[3:6] - row[:3]).max())
            row[3:6] = row[:3] + [(d if j % 2 else -d) * (j in keep) for j in range(3)]
    return np.maximum(ln, [-99.0] * 6 + [0.5])


@pytest.mark.parametrize('dtype', [np.float32, np.float64])
@pytest.mark.parametrize('kind', ['one', 'thin', 'wide', 'mixed', 'grid'])
@pytest.mark.parametrize('shape', [(1, 17, 19, 23), (3, 1, 33, 40), (2, 40, 1, 18), (2, 24, 30, 1)])
def test_fill_edges(cuda, oracle, shape, kind, dtype):
    rng = np.random.default_rng(len(kind) + 31 * shape[2])
    lines = lines_for(kind, rng, shape).astype(dtype)
    idxs = rng.integers(0, shape[0], len(lines)).astype(np.int32 if dtype == np.float32 else np.int64)
    for kernel in ('biweight', 'rectangular', 'triangular'):
        for overlap in ('sum', 'max'):
            ref = oracle.draw_lines3(np.zeros(shape, dtype), lines, idxs, 1.3, kernel, overlap)
            out = torch.zeros(shape, dtype=torch.from_numpy(ref).dtype, device='cuda')
            ndimage.draw_lines(out, torch.from_numpy(lines).cuda(), torch.from_numpy(idxs).cuda(), max_val=1.3,
                               kernel=kernel, overlap=overlap)
            got = out.cpu().numpy()
            assert np.array_equal(got != 0, ref != 0), (kernel, overlap)
            if overlap == 'max':
                assert np.array_equal(got, ref), kernel
            else:
                np.testing.assert_allclose(got, ref, rtol=5e-6 if dtype == np.float32 else 1e-14, err_msg=kernel)
