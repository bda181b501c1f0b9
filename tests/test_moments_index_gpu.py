"""Region sums around the number of regions whose largest label one workgroup
finds (8192 = 32 x 256): every region is one pixel, so the total mass of label l is
its pixel's value, exactly; labels in reverse order, and with an entry that no
pixel has."""
import numpy as np
import pytest
import torch

from cbclib_v2_amd import label as cl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n', [1, 255, 256, 257, 8191, 8192, 8193, 20000])
def test_index_sizes(cuda, n):
    W = 150
    rows = (n + W) // W + 1
    lab = np.zeros(rows * W, np.int32)
    lab[:n] = np.arange(1, n + 1)
    data = np.random.default_rng(n).random(rows * W).astype(np.float32)
    index = np.concatenate([np.arange(1, n + 1)[::-1], [n + 7]])
    res = cl.CPLabelResult(labels=torch.from_numpy(lab.reshape(rows, W)).cuda(), index=torch.from_numpy(index).cuda())
    got = cl.total_mass(res, torch.from_numpy(data.reshape(rows, W)).cuda()).cpu().numpy()
    assert np.array_equal(got, np.concatenate([data[:n][::-1], [np.float32(0)]]))
