"""Layout copies on either side of each rule that picks their kernel: tiles with
a fifth or three eighths of their elements inside the array, long and very short
axes of 16-byte elements, rows that widen and rows that do not, odd lengths, and
buffers that start one element past an aligned address. Copies are bit-exact."""
import numpy as np
import pytest
import torch

import pencil_fft_hip as pf

pytestmark = pytest.mark.gpu

# (shape, destination order): the last axis is the source's fastest
TILES = [(9, 64, 12), (9, 64, 13), (7, 24, 40), (3, 33, 48), (5, 32, 48), (5, 31, 48), (3, 256, 16), (3, 257, 7),
         (2, 767, 33), (2, 768, 33), (11, 6, 32), (11, 7, 32), (11, 6, 31), (301, 2, 2), (40, 3, 64)]
ROWS = [(6, 17, 3), (6, 17, 4), (6, 17, 5), (6, 17, 7), (6, 17, 14), (6, 17, 16), (6, 17, 17), (6, 17, 24), (6, 17, 32),
        (6, 17, 33), (6, 17, 63), (6, 17, 64), (6, 17, 65), (6, 17, 95), (6, 17, 96), (6, 17, 129), (6, 17, 300)]


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("element", [1, 2, 4, 8, 16])
def test_both_sides_of_the_copy_rules(gpu, element, shift):
    rng = np.random.default_rng(element)
    for shapes, dst in ((TILES, (0, 2, 1)), (TILES, (2, 0, 1)), (ROWS, (1, 0, 2))):
        for shape in shapes:
            n = int(np.prod(shape))
            raw = rng.integers(0, 256, size=((n + shift), element), dtype=np.uint8)
            x = torch.from_numpy(raw.reshape(-1)).cuda()[shift * element:]
            y = torch.zeros((n + shift) * element, dtype=torch.uint8, device="cuda")
            pf.LocalTransposePlan(shape, (0, 1, 2), dst, element).execute(x, y[shift * element:])
            ref = raw[shift:].reshape(*shape, element).transpose(*dst, 3)
            got = y.cpu().numpy()
            assert np.array_equal(got[shift * element:], np.ascontiguousarray(ref).reshape(-1)), (shape, dst)
            assert not got[:shift * element].any()
