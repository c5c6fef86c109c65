"""The contiguous adjoint on either side of the lines (65536 chunks of 8 rows,
systems of 2048 rows) up to which it runs the shortest chunks in one-wave
work-groups: systems that share a wave, fill one and span several, the batch's
last wave short."""
from __future__ import annotations

import numpy as np
import pytest

from tests import test_gpu_adjoint_layouts as layouts

pytestmark = pytest.mark.gpu

# 1, 4, 16, 64, 128, 512 chunks per system
CASES = [([n, q + extra], None, 0)
         for n, q in ((5, 65536), (20, 16384), (100, 4096), (420, 1024), (600, 512), (4090, 128))
         for extra in (-1, 0, 1)]
CASES += [([n, 6], None, 0) for n in (1023, 1100, 2047, 2048, 2049)]
CASES += [([20, 127, 129], [20, 127, 130], 0), ([600, 127, 4], [603, 127, 5], 0)]


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("dims,pads,sd", CASES)
def test_either_side_of_the_line(dims, pads, sd, dtype, offset):
    layouts.test_adjoint_layouts(dims, pads, sd, dtype, offset)
