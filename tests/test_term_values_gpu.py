"""Values of accumulate_lines with different overlaps in float images: the
reference's own values and, within a term, its order of additions.

* A term's sum into a maximum: bit-equal to the oracle (single-threaded
  reference); gaussian profiles within 3e-7 (the device's double exp against
  glibc's, rounded to float).
* A term's maximum into a sum: the terms of a pixel reach it in no fixed order, so
  k terms of positive values differ by at most 2 k 2^-24 of their sum (k 2^-24
  each for this and for the oracle's); k is counted with the oracle.

The value range covers faint pixels (profiles near zero at the edge of a line),
where an absolute error would show.
"""
import numpy as np
import pytest
import torch

from cbclib_v2_amd import ndimage
from tests.lines_gen import random_segments

pytestmark = pytest.mark.gpu


def case(kind):
    rng = np.random.default_rng(len(kind))
    # lines that touch no other line of their term are drawn apart from the rest: from
    # 4096 such lines in 128 tiles of 32 pixels on (a frame of 360 x 390 has 156)
    shape, n, n_terms, lmax = {
        'spread': ((2, 360, 390), 9000, 1500, 40.0),      # some lines of a term touch another one of it
        'crossing': ((1, 360, 390), 9000, 80, 60.0),      # most of them do
        'alone': ((1, 360, 390), 4500, 4500, 60.0),       # one line a term
        'fewer': ((1, 360, 390), 4095, 2000, 60.0),       # too few lines
        'large': ((1, 360, 390), 5140, 20, 30.0),         # terms of 257 lines
        'small frame': ((1, 90, 70), 9000, 1500, 30.0),   # too few tiles
        'at most': ((1, 360, 390), 5376, 40, 12.0),       # terms of up to 256 lines, in no order
        'one more': ((1, 360, 390), 5377, 40, 12.0),      # a term of 257
    }[kind]
    lines = random_segments(rng, n, *shape[1:], 1.0, lmax, 0.4, 4.0, pad=5.0).astype(np.float32)
    terms = (np.arange(n) % n_terms).astype(np.int32)
    if kind in ('at most', 'one more'):
        terms = np.minimum(np.arange(n) // 256, 20).astype(np.int32)
        rng.shuffle(terms)
    return shape, lines, terms, rng.integers(0, shape[0], n_terms).astype(np.int32)


def accumulated(shape, lines, terms, frames, kernel, modes):
    out = torch.zeros(shape, dtype=torch.float32, device='cuda')
    ndimage.accumulate_lines(out, *(torch.from_numpy(v).cuda() for v in (lines, terms, frames)), 0.9, kernel, *modes)
    return out.cpu().numpy()


@pytest.mark.parametrize('kernel', ['biweight', 'gaussian', 'parabolic', 'rectangular', 'triangular'])
@pytest.mark.parametrize('kind', ['spread', 'crossing', 'alone', 'fewer', 'large', 'small frame', 'at most', 'one more'])
def test_term_values(cuda, oracle, kind, kernel):
    shape, lines, terms, frames = case(kind)
    rtol = 3e-7 if kernel == 'gaussian' else 0.0
    zero = np.zeros(shape, np.float32)
    ref = oracle.accumulate_lines(zero.copy(), lines, terms, frames, 0.9, kernel, 'sum', 'max')
    got = accumulated(shape, lines, terms, frames, kernel, ('sum', 'max'))
    np.testing.assert_allclose(got, ref, rtol=rtol, atol=0.0)
    ref = oracle.accumulate_lines(zero.copy(), lines, terms, frames, 0.9, kernel, 'max', 'sum').astype(np.float64)
    count = oracle.accumulate_lines(zero.copy(), lines, terms, frames, 1.0, 'rectangular', 'max', 'sum')
    got = accumulated(shape, lines, terms, frames, kernel, ('max', 'sum'))
    assert np.array_equal(got != 0, ref != 0)
    assert (np.abs(got - ref) <= (2.0 * count * 2.0 ** -24 + rtol) * ref).all()
