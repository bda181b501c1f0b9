"""3D draws of line counts on both sides of the plane fills' split (8192, 32 768 and
131 072 planes: 1, 4, 8 and 16 planes a wave, and the instance of few planes),
thin and wide lines together, against the oracle: max bit-exact; sums within
the rounding of their additions (k voxel values of at most 1.3: 2 k 2^-24, k
counted with the oracle), support bit-exact."""
import numpy as np
import pytest
import torch

from cbclib_v2_amd import ndimage
from tests.lines_gen import segments3

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dtype', [np.float32, np.float64])
@pytest.mark.parametrize('n', [3, 250, 420, 1000, 2400, 5500, 9000])
def test_plane_counts(cuda, oracle, n, dtype):
    shape = (3, 24, 40, 50)
    rng = np.random.default_rng(n)
    lines = segments3(rng, n, shape, 24.0, 0.2, 4.0, 2.0)
    lines[::7, 6] *= 0.1
    lines[::50, 6] += 5.0
    lines = lines.astype(dtype)
    idxs = rng.integers(0, shape[0], n).astype(np.int32 if dtype == np.float32 else np.int64)
    t_lines, t_idxs = torch.from_numpy(lines).cuda(), torch.from_numpy(idxs).cuda()
    count = oracle.draw_lines3(np.zeros(shape, dtype), lines, idxs, 1.0, 'rectangular', 'sum')
    eps = 2.0 ** -24 if dtype == np.float32 else 2.0 ** -53
    for kernel in ('rectangular', 'parabolic', 'triangular', 'biweight'):
        for overlap in ('sum', 'max'):
            ref = oracle.draw_lines3(np.zeros(shape, dtype), lines, idxs, 1.3, kernel, overlap)
            out = torch.zeros(shape, dtype=torch.from_numpy(ref).dtype, device='cuda')
            ndimage.draw_lines(out, t_lines, t_idxs, max_val=1.3, kernel=kernel, overlap=overlap)
            got = out.cpu().numpy()
            assert np.array_equal(got != 0, ref != 0), (kernel, overlap)
            if overlap == 'max':
                assert np.array_equal(got, ref), kernel
            else:
                assert (np.abs(got.astype(np.float64) - ref) <= 2.0 * count * eps * ref).all(), kernel
