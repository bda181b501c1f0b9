"""3D lines whose squared length lies near or below the smallest normal number
(they start in the volume's corner at the origin), a frame each, against the
oracle: the same voxels, max bit-exact."""
import numpy as np
import pytest
import torch

from cbclib_v2_amd import ndimage

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dtype,exponents', [(np.float32, (-75, -72)), (np.float32, (-66, -58)), (np.float32, (-30, -10)),
                                             (np.float64, (-537, -534)), (np.float64, (-515, -505))])
def test_tiny_lines(cuda, oracle, dtype, exponents):
    n = 500
    rng = np.random.default_rng(-exponents[0])
    lines = np.zeros((n, 7), dtype)
    lines[:, 3:6] = (rng.normal(size=(n, 3)) * 2.0 ** rng.integers(*exponents, (n, 1), endpoint=True)).astype(dtype)
    lines[:, 6] = rng.uniform(0.5, 6.0, n)
    shape = (n, 9, 10, 11)
    for kernel in ('rectangular', 'parabolic'):
        ref = oracle.draw_lines3(np.zeros(shape, dtype), lines, None, 1.3, kernel, 'max')
        out = torch.zeros(shape, dtype=torch.from_numpy(ref).dtype, device='cuda')
        ndimage.draw_lines(out, torch.from_numpy(lines).cuda(), None, max_val=1.3, kernel=kernel, overlap='max')
        differ = np.flatnonzero((out.cpu().numpy() != ref).any((1, 2, 3)))
        assert differ.size == 0, (kernel, len(differ), differ[:5])
