"""accumulate_lines with different overlaps: lines of 12 000 pixels, whose pixels the
float walk draws some pixels beyond their ends, meet another line of their term
there.  The term's maximum counts such a pixel once."""
import numpy as np
import pytest
import torch

from cbclib_v2_amd import ndimage
from tests.lines_gen import random_segments

pytestmark = pytest.mark.gpu


def test_ends_of_long_lines(cuda, oracle):
    shape = (1, 16, 26880)
    pair = np.array([[4.0, 8.0, 12199.9072265625, 8.0, 2.02], [26855.453125, 8.0, 12207.970703125, 8.0, 2.02]], np.float32)
    alone = [oracle.draw_lines(np.zeros(shape, np.float32), pair[k:k + 1], None, 1.0, 'rectangular', 'max') for k in (0, 1)]
    assert (alone[0] * alone[1]).any()          # both draw column 12204
    # lines of terms of their own: enough lines for those alone in their pixels to go by frame tiles
    rng = np.random.default_rng(3)
    lines = np.concatenate([pair, random_segments(rng, 4200, 16, 26880, 2.0, 9.0, 0.5, 1.5)]).astype(np.float32)
    terms = np.maximum(np.arange(len(lines)) - 1, 0).astype(np.int32)
    frames = np.zeros(len(lines) - 1, np.int32)
    for modes in (('max', 'sum'), ('sum', 'max')):
        ref = oracle.accumulate_lines(np.zeros(shape, np.float32), lines, terms, frames, 1.0, 'rectangular', *modes)
        out = torch.zeros(shape, dtype=torch.float32, device='cuda')
        ndimage.accumulate_lines(out, *(torch.from_numpy(v).cuda() for v in (lines, terms, frames)), 1.0, 'rectangular',
                                 *modes)
        np.testing.assert_array_equal(out.cpu().numpy(), ref, err_msg=str(modes))   # whole numbers: exact sums
