"""The ordered mode sorts up to 8192 segments of a tile (32 pixels).  A line next
to a tile whose pixels come no nearer than the walk's own positions and errors
say is not among the tile's segments: full tiles beside such lines are drawn."""
import numpy as np
import pytest
import torch

from cbclib_v2_amd import ndimage

pytestmark = pytest.mark.gpu

# lines below the tile's last row (31) whose segments reach up to row 32 and, by a
# bound of the whole line, to row 31
BESIDE = np.array([[15.24687385559082, 36.8828010559082, 16.630733489990234, 36.55535888671875, 2.4533655643463135],
                   [9.200050354003906, 35.86571502685547, 11.259428977966309, 35.75332260131836, 2.5186240673065186],
                   [11.972413063049316, 36.411685943603516, 12.648722648620605, 35.8814697265625, 0.42470407485961914]],
                  np.float32)


@pytest.mark.parametrize('beside', [0, 1, 2])
def test_full_tile(cuda, oracle, beside):
    # 8192 lines of one segment each in rows 8 to 12, columns 4 to 9
    rng = np.random.default_rng(0)
    full = np.zeros((8192, 5), np.float32)
    full[:, 0] = rng.uniform(6.0, 6.4, 8192)
    full[:, 1] = rng.uniform(9.5, 10.5, 8192)
    full[:, 2] = full[:, 0] + 1.0
    full[:, 3] = full[:, 1]
    full[:, 4] = 0.75
    lines = np.concatenate([full, BESIDE[beside:beside + 1]])
    ref = oracle.draw_lines(np.zeros((64, 64), np.float32), lines, None, 1.0, 'parabolic', 'sum')
    out = torch.zeros(64, 64, device='cuda')
    ndimage.draw_lines(out, torch.from_numpy(lines).cuda(), None, 1.0, 'parabolic', 'sum', deterministic=True)
    assert np.array_equal(out.cpu().numpy(), ref)


def test_overfull_tile_is_refused(cuda):
    lines = np.tile(np.array([[6.0, 10.0, 7.0, 10.0, 0.75]], np.float32), (8193, 1))
    out = torch.zeros(64, 64, device='cuda')
    with pytest.raises(RuntimeError):
        ndimage.draw_lines(out, torch.from_numpy(lines).cuda(), None, 1.0, 'parabolic', 'sum', deterministic=True)
    assert float(out.abs().max()) == 0.0
