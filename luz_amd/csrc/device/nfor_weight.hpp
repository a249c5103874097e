// The weights of the NFOR regression (colorWeightFromDistance, NFOR.cpp:313-318): exp(-x), and
// exp(-4x) from it, for the two bandwidths that share a pass.
#pragma once

#include <hip/hip_runtime.h>

#include <bit>
#include <cmath>
#include <cstdint>

namespace luzgpu
{
	// (hi + lo) * 2^exponent, hi in [0.7, 1.42] and |lo| at most half an ulp of it
	struct	NforExp
	{
		double	hi, lo;
		int	exponent;
	};

	// exp(-x) for x >= 0 (NaN stays NaN): 2^k e^r with k the nearest integer to -x log2 e, r the
	// rest (ln 2 in two parts), e^r its Taylor sum to r^14 (|r| <= ln 2 / 2: the first term left
	// out is 1e-19 of it). 1, r, its rounding and r^2 / 2 are added with their errors kept, so
	// the sum's own error is below 2^-57 and hi within 0.53 ulp (the device's exp, over the same
	// arguments: 0.87). Rounded sums throughout would be within 1.02 and save 0.35 ms of the
	// 5.9 that one bandwidth takes at 1280 x 720, radius 9.
	__host__ __device__ __forceinline__ NforExp	nforExpNegative(double x)
	{
		#pragma clang fp contract(off)
		x = x > 1000.0 ? 1000.0 : x;	// 2^-1443: zero already
		const double k = rint(x * -1.4426950408889634);
		const double t = fma(k, -0.69314718055994529, -x);	// exact
		const double r = fma(k, -2.3190468138462996e-17, t);
		const double rLow = fma(k, -2.3190468138462996e-17, t - r);
		// two half sums of the even and odd powers from r^3 on: two chains in flight
		const double r2 = r * r;
		double even = fma(r2, 1.1470745597729725e-11, 2.0876756987868099e-09);	// 1/14!, 1/12!
		double odd = fma(r2, 1.6059043836821613e-10, 2.5052108385441720e-08);		// 1/13!, 1/11!
		even = fma(r2, even, 2.7557319223985893e-07);
		odd = fma(r2, odd, 2.7557319223985893e-06);
		even = fma(r2, even, 2.4801587301587302e-05);
		odd = fma(r2, odd, 1.9841269841269841e-04);
		even = fma(r2, even, 1.3888888888888889e-03);
		odd = fma(r2, odd, 8.3333333333333332e-03);
		even = fma(r2, even, 4.1666666666666664e-02);
		odd = fma(r2, odd, 1.6666666666666666e-01);
		const double half = 0.5 * r2, halfLow = 0.5 * fma(r, r, -r2);
		const double rest = fma(r2, fma(r2, even, r * odd), fma(rLow, r, rLow) + halfLow);
		const double a = 1.0 + r, aLow = r - (a - 1.0);
		const double b = a + half, bLow = half - (b - a);
		const double low = rest + (aLow + bLow);
		NforExp e;
		e.hi = b + low;
		e.lo = low - (e.hi - b);
		e.exponent = static_cast<int>(k);
		return e;
	}

	__host__ __device__ __forceinline__ double	nforWeight1(const NforExp& e) { return ldexp(e.hi, e.exponent); }

	// How many doubles nforWeight4's product of rounded values lies from the fourth power of the
	// sum, rounded (up to 6). Weights that are not normal to the fourth, or above 1, go without.
	__host__ __device__ __forceinline__ std::int8_t	nforWeight4Correction(const NforExp& e)
	{
		#pragma clang fp contract(off)
		const double square = e.hi * e.hi, squareLow = fma(e.hi, e.hi, -square);
		const double fourth = square * square, fourthLow = fma(square, square, -fourth);
		const double exact = fourth + fma(square + square, fma(e.hi + e.hi, e.lo, squareLow), fourthLow);
		const bool normal = e.exponent > -255 && e.exponent <= 0;
		return static_cast<std::int8_t>(normal ? std::bit_cast<std::int64_t>(exact) - std::bit_cast<std::int64_t>(fourth) : 0);
	}

	// exp(-4x) from exp(-x): 0.6 ulp, against 5.8 without the correction (which takes 0.5 ms of
	// the 8.6 of two bandwidths).
	__host__ __device__ __forceinline__ double	nforWeight4(double weight, std::int8_t correction)
	{
		#pragma clang fp contract(off)
		const double square = weight * weight, fourth = square * square;
		return std::bit_cast<double>(std::bit_cast<std::int64_t>(fourth) + correction);
	}
}
