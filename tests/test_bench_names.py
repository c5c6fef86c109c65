"""The benchmark's kernel names for the ADI's first kernel."""
from __future__ import annotations

import pytest

import bench


@pytest.mark.parametrize("desc,dtype,nx,name", [
    ("rhs+x(fused,R8,xcd,cached)<double> x:part<double> y:cc<R16,cps16,cached> z:cc<R16,cps16>",
     "f64", 256, "k_adi_rhs_x<double, 8, 1, 0, 2>"),
    ("rhs+x(fused,R4,cached)<float> x:part<float> y:p z:q step:rhs+x(lines,R13,cached)",
     "f32", 256, "k_adi_rhs_xl<float, 13, 3, 1>"),
    ("rhs+x(lines,R7)<double> x:part<double> y:p z:q", "f64", 201, "k_adi_rhs_xl<double, 7, 4, 0>"),
])
def test_first_kernel(desc, dtype, nx, name):
    assert bench.kernel_of_config(bench.stage_config(desc, "rhs_x_fused"), dtype, 0, "CoefConst",
                                  nx) == name
