"""The NFOR regression's weights (device/nfor_weight.hpp, IEEE operations alone, so the host
computes what the device does) against 64-bit-mantissa exponentials: exp(-x), and exp(-4x)
from its rounded value and correction, each rounded once and a little more, over the
arguments of weights from 1 down to the smallest normal ones."""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "device/nfor_weight.hpp"
#include <algorithm>
#include <cstdio>
#include <random>

static long double	ulps(double got, long double want)
{
	int e;
	std::frexp(want, &e);
	return std::fabs(static_cast<long double>(got) - want) / std::ldexp(1.0L, e - 53);
}

int	main()
{
	std::mt19937_64 g(7);
	long double worst1 = 0.0L, worst4 = 0.0L;
	auto check = [&](double x) {
		const luzgpu::NforExp e = luzgpu::nforExpNegative(x);
		const double w = luzgpu::nforWeight1(e);
		worst1 = std::max(worst1, ulps(w, std::exp(-static_cast<long double>(x))));
		if (x <= 176.0) worst4 = std::max(worst4, ulps(luzgpu::nforWeight4(w, luzgpu::nforWeight4Correction(e)), std::exp(-4.0L * x)));
	};
	for (double range : {1e-3, 0.3, 2.0, 20.0, 176.0, 708.0})
	{
		std::uniform_real_distribution<double> u(0.0, range);
		for (int i = 0; i < 300000; i++) check(u(g));
	}
	check(0.0);
	for (int k = 1; k < 250; k++)	// where the reduction changes to the next power of two
	{
		const double x = (k - 0.5) * 0.69314718055994531;
		for (double y : {std::nextafter(x, 0.0), x, std::nextafter(x, 1e3)}) check(y);
	}
	for (double x = 170.0; x < 800.0; x += 0.01)	// down to zero: to the fourth within the smallest double's few
	{
		const luzgpu::NforExp e = luzgpu::nforExpNegative(x);
		const double w4 = luzgpu::nforWeight4(luzgpu::nforWeight1(e), luzgpu::nforWeight4Correction(e));
		if (!(std::fabs(w4 - std::exp(-4.0L * x)) <= std::max(1e-300L * 1e-15L, 1e-15L * std::exp(-4.0L * x)))) worst4 = 1e9L;
	}
	const bool zero = luzgpu::nforWeight1(luzgpu::nforExpNegative(1e300)) == 0.0 && luzgpu::nforWeight1(luzgpu::nforExpNegative(HUGE_VAL)) == 0.0;
	volatile double none = std::nan("");
	const luzgpu::NforExp n = luzgpu::nforExpNegative(none);
	const bool nan = std::isnan(luzgpu::nforWeight1(n)) && std::isnan(luzgpu::nforWeight4(luzgpu::nforWeight1(n), luzgpu::nforWeight4Correction(n)));
	std::printf("%.4Lf %.4Lf %d %d\n", worst1, worst4, zero, nan);
	return 0;
}
"""


def test_weights_are_rounded_once(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not installed")
    source, program = tmp_path / "weights.cpp", tmp_path / "weights"
    source.write_text(PROGRAM)
    subprocess.run([hipcc, "-std=c++20", "-O2", "-x", "hip", "--cuda-host-only", "-I", os.path.join(ROOT, "luz_amd", "csrc"), str(source),
                    "-o", str(program)], check=True)
    worst1, worst4, zero, nan = subprocess.run([str(program)], check=True, capture_output=True, text=True).stdout.split()
    # half an ulp is the final rounding; the sum's 2^-57 (2^-55 in the fourth power) comes to
    # under 0.04 and 0.1 ulp
    assert float(worst1) <= 0.54 and float(worst4) <= 0.61, (worst1, worst4)
    assert zero == "1" and nan == "1"
