"""Dilation of rows of no whole number of words, at any byte alignment of the
input, the mask and the output, against the oracle (bit-exact): rows shorter
than a 16-byte piece, around one piece and one word, pieces that hold several
rows, single elements; structures whose tables travel with the kernel's
arguments and larger ones."""
import numpy as np
import pytest
import torch

from cbclib_v2_amd import _native
from cbclib_v2_amd.label import Structure

pytestmark = pytest.mark.gpu


def at(a, off):
    """A copy of `a` on the device, `off` bytes after a 256-byte boundary, with exactly its bytes behind it."""
    buf = torch.empty(a.size + off, dtype=torch.uint8, device='cuda')
    t = buf[off:]
    t.copy_(torch.from_numpy(a.reshape(-1).view(np.uint8)))
    return buf, t


@pytest.mark.parametrize('shape', [(1,), (15,), (7, 1), (9, 5), (3, 4, 15), (5, 16), (6, 17), (4, 63), (3, 64), (4, 65),
                                   (2, 3, 129), (3, 200)])
@pytest.mark.parametrize('offs', [(0, 0, 0), (1, 2, 3), (4, 8, 15), (7, 0, 12)])
def test_rows(cuda, oracle, shape, offs):
    rng = np.random.default_rng(sum(shape) + 7 * sum(offs))
    nd = len(shape)
    for radii, conn, it in (([1] * nd, 1, 2), ([0] * (nd - 1) + [3], 3, 1), ([9] * nd if nd < 3 else [3] * nd, 27, 1)):
        st = Structure(radii, conn)
        shifts = np.ascontiguousarray(st.shifts(), dtype=np.int64)
        inp, mask = rng.random(shape) < 0.2, rng.random(shape) < 0.7
        ref = oracle.binary_dilation(inp, shifts, it, mask)
        keep_i, ti = at(inp, offs[0])
        keep_m, tm = at(mask, offs[1])
        guard = torch.full((inp.size + offs[2] + 16,), 7, dtype=torch.uint8, device='cuda')
        dims = np.asarray(shape, np.int64)
        torch.cuda.synchronize()
        _native.check(_native.lib().cbx_binary_dilation(
            ti.data_ptr(), tm.data_ptr(), nd, dims.ctypes.data, shifts.ctypes.data, len(shifts), it,
            guard.data_ptr() + offs[2], None))
        torch.cuda.synchronize()
        got = guard.cpu().numpy()
        assert np.array_equal(got[offs[2]:offs[2] + inp.size].reshape(shape), ref.astype(np.uint8)), (radii, conn, it)
        assert (got[:offs[2]] == 7).all() and (got[offs[2] + inp.size:] == 7).all()
