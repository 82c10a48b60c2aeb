"""FP32 CG on many right-hand sides with a preconditioner on the two sides of the
line between separate and fused steps (31 and 33 columns of 66,049 rows)."""
import numpy as np
import pytest

from test_gpu_multi_steps import test_fused_steps_equal_separate_ones as equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R", [31, 33])
def test_both_sides(hip, R):
    equal(hip, 8, R, True, np.float32)
