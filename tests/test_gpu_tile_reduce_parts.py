"""The smallest tile shape's optimizer workgroup (a wavefront per parameter instead of four parameters a lane) over rows that
come in the parts of their blocks: the comparisons of test_gpu_batch_parts.py."""
import pytest

import test_gpu_batch_parts as parts


@pytest.mark.gpu
@pytest.mark.parametrize("cap", [2, 3])
def test_parts_of_the_smallest_shape(cap):
    parts.test_parts_do_not_depend_on_the_grid_or_the_other_problems((1, 1, 1, 1), cap)
