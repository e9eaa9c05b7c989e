"""The 3D momentum steps at the edges of their level counts: the instances that hold a column
on chip take up to 16, 24, 32, 40, 48 and 64 levels, deeper grids the scratch form.  Same
checks as the small-grid tests (FP64, bit for bit against the oracle)."""
from __future__ import annotations

import pytest

from tests.test_gpu_coupled import test_coupled_fp64_bitwise_against_oracle as coupled_case
from tests.test_gpu_step3d import test_main3d_bitwise as main3d_case

pytestmark = pytest.mark.gpu

LEVELS = [16, 24, 25, 32, 33, 40, 41, 48, 49, 64, 65]


@pytest.mark.parametrize("N", LEVELS)
def test_step3d_uv_levels(N):
    main3d_case(19, 13, N, True)


@pytest.mark.parametrize("N", LEVELS)
def test_step3d_uv_coupled_levels(N):
    coupled_case(19, 13, N)
