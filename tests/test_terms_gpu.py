"""accumulate_lines with different overlaps by frame tiles, against the oracle,
where its rules change: terms of one line (nothing to reduce), terms whose
lines all cross in one tile (more items than one pass of the term kernel
holds), the largest term that goes this way and one line more (the other
way), frames of a ragged size, negative max_val.

Tolerance: every drawn value is within a few ulp plus 2^-23 max_val of the
oracle's, and a pixel adds up at most a few hundred of them: rtol 1e-5, atol
1e-6 (as in test_accumulate); support exact.
"""
import numpy as np
import pytest
import torch

from cbclib_v2_amd import ndimage
from tests.lines_gen import random_segments

pytestmark = pytest.mark.gpu


def make(kind, rng):
    if kind == 'alone':
        n, T, H, W, lmax = 500, 500, 130, 190, 40.0
    elif kind == 'crossing':
        n, T, H, W, lmax = 6000, 200, 64, 60, 20.0
    elif kind == 'few':
        n, T, H, W, lmax = 900, 60, 131, 97, 60.0
    else:
        n, T, H, W, lmax = {'256': 256, '257': 257}[kind], 1, 150, 140, 50.0
    lines = random_segments(rng, n, H, W, 1.0, lmax, 0.4, 3.0, pad=5.0).astype(np.float32)
    terms = np.arange(n) % T if kind != 'few' else rng.integers(0, T, n)
    F = 1 if kind == 'crossing' else 3
    return (F, H, W), lines, terms.astype(np.int32), rng.integers(0, F, T).astype(np.int32)


@pytest.mark.parametrize('modes', [('max', 'sum'), ('sum', 'max')])
@pytest.mark.parametrize('kind', ['alone', 'crossing', 'few', '256', '257'])
@pytest.mark.parametrize('kernel', ['gaussian', 'triangular', 'rectangular'])
def test_terms_by_tile(cuda, oracle, kind, modes, kernel):
    rng = np.random.default_rng(len(kind) * 5 + len(kernel))
    shape, lines, terms, frames = make(kind, rng)
    for max_val in (0.9, -0.6):
        base = rng.uniform(-0.4, 0.4, shape).astype(np.float32)
        ref = oracle.accumulate_lines(base.copy(), lines, terms, frames, max_val, kernel, *modes)
        out = torch.from_numpy(base.copy()).cuda()
        ndimage.accumulate_lines(out, *(torch.from_numpy(v).cuda() for v in (lines, terms, frames)), max_val, kernel,
                                 *modes)
        np.testing.assert_allclose(out.cpu().numpy(), ref, rtol=1e-5, atol=1e-6, err_msg=str(max_val))
    zero = np.zeros(shape, np.float32)
    ref = oracle.accumulate_lines(zero.copy(), lines, terms, frames, 0.9, kernel, *modes)
    out = torch.zeros(shape, dtype=torch.float32, device='cuda')
    ndimage.accumulate_lines(out, *(torch.from_numpy(v).cuda() for v in (lines, terms, frames)), 0.9, kernel, *modes)
    assert np.array_equal(out.cpu().numpy() != 0, ref != 0)
