"""CPU check that the benchmark's patterns find the kernels under the names that
a profiler prints, of every form of the FP64 kernels and of no other."""
import os
import re
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402

C = "msod::ConvecArgs<double, double, double, double, double>"
D = "msod::DiffuArgs<double, double, double, double>"


@pytest.mark.parametrize("kernel,name", [
    ("full_convec_ijk", f"void msod::k_convec_col<4, false, {C} >({C})"),
    ("full_convec_ijk", f"void msod::k_convec_wide<7, false, {C} >({C})"),
    ("full_convec_ijk", f"void msod::k_convec<3, {C}, double>({C})"),
    ("full_diffusion_ijk", f"void msod::k_diffu_col<4, false, {D}, false>({D}, float const*)"),
    ("full_diffusion_ijk", f"void msod::k_diffu_wide<6, {D}, false>({D}, float const*)"),
    ("full_diffusion_ijk", f"void msod::k_diffu_split<7, 2, {D}, false>({D}, float const*)"),
    ("full_diffusion_ijk", f"void msod::k_diffu<4, {D}, false, double>({D}, float const*)"),
])
def test_fp64_kernels(kernel, name):
    assert re.search(bench.KERNEL_RE[kernel], name)
    assert [k for k, pat in bench.KERNEL_RE.items() if re.search(pat, name)] == [kernel]


@pytest.mark.parametrize("name", [
    f"void msod::k_diffu_col<3, false, {D}, true>({D}, float const*)",
    "void msod::k_convec_col<4, false, msod::ConvecArgs<float, float, double, double, double> >(...)",
    f"void msod::k_convec_col<4, true, {C} >({C})",
])
def test_other_forms(name):
    assert not any(re.search(pat, name) for pat in bench.KERNEL_RE.values())
