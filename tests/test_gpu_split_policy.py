"""Split-line solves under the autotuner: their layout and cache policy are
rules, not tuned choices, so both are the same with tuning on and off, at the
first call of a shape and at later ones."""
from __future__ import annotations

import numpy as np
import pytest

import tridsolver_amd as ta
from tests.test_gpu_scalar import run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("dims,sd", [([51, 2048], 1), ([51, 2100, 3], 1), ([7, 5, 9001], 2),
                                     ([9001, 3], 0)])
def test_tuning_leaves_split_solves_alone(dims, sd, dtype):
    run_case(dims, sd, dtype, False, seed=sd)
    untuned = ta.last_config()
    assert untuned.startswith("split<") and (",cached" in untuned) == (sd != 0)
    ta.set_autotune(1)
    try:
        for _ in range(2):
            run_case(dims, sd, dtype, False, seed=sd)
            assert ta.last_config() == untuned
    finally:
        ta.set_autotune(0)
