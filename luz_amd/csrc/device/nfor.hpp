// NFOR denoiser on the device (Denoise::applyNFOR, src/core/Denoise/NFOR.cpp:977-1102), in
// FP64 like the reference.
//
// Inputs are the half-buffer statistics the integrator accumulates with denoising on
// (Threads.cpp:274-372): mean colours of the even and odd samples (A / B), the per-pixel
// colour variance, the mean primary features of each half (11 per pixel) and their variance.
// Stages, one kernel each:
//   firefly suppression of A, B and of their average (NFOR.cpp:145-211);
//   feature prefiltering, each half guided by the other (NL-means weights, :403-464);
//   first-order feature regression of A with B's features and of B with A's, at two
//   bandwidths (k = 0.5, 1) (:739-832);
//   MSE estimation, its and the bandwidth selection's cross-bilateral filtering (:834-936);
//   per-pixel blend, then a final regression of the blend (:1074-1101).
//
// The regression solves a 12 x 12 weighted least-squares system per pixel. The systems are
// accumulated on the FP64 matrix unit, four window samples (in the reference's raster
// order) to an instruction, and a second kernel solves each by the reference's
// Gauss-Jordan elimination with partial pivoting.
#pragma once

#include "median.hpp"
#include "nfor_weight.hpp"

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

namespace luzgpu
{
	constexpr int	kNforFeatures = 11;
	constexpr int	kNforBasis = kNforFeatures + 1;			// REGRESSION_SIZE
	constexpr int	kNforUpper = kNforBasis * (kNforBasis + 1) / 2;	// 78 upper-triangle entries
	constexpr int	kNforSystem = kNforUpper + kNforBasis * 3;		// + the RGB right-hand side

	// Per-pixel FP64 statistics of a denoised render, in sample order (_threadRender with
	// denoise buffers, Threads.cpp:585-627): [0,3) half A colour sum, [3,6) half B, [6,9) all
	// colours, [9,12) colour squares, then kNforFeatures each of half A, half B, all features
	// and feature squares.
	constexpr int	kDenoiseStats = 12 + 4 * kNforFeatures;

	// Adds one sample (cleaned colour, primary features) to a pixel's statistics `a`;
	// `odd`: the sample index is odd (half B, sampler stream 2).
	__device__ __forceinline__ void	denoiseAddSample(double* a, const float* color, const float* feat, bool odd)
	{
		#pragma clang fp contract(off)
		const int half = odd ? 3 : 0;
		for (int j = 0; j < 3; j++)
		{
			const double c = color[j];
			a[half + j] += c;
			a[6 + j] += c;
			a[9 + j] += c * c;
		}
		const int fh = odd ? 12 + kNforFeatures : 12;
		for (int j = 0; j < kNforFeatures; j++)
		{
			const double f = feat[j];
			a[fh + j] += f;
			a[12 + 2 * kNforFeatures + j] += f;
			a[12 + 3 * kNforFeatures + j] += f * f;
		}
	}

#ifndef LUZ_FEATURES	// the denoiser's kernels are compiled once, in luzgpu.hip
	struct	NforParams
	{
		std::uint32_t	width, height;
		std::uint32_t	prefilterRadius, regressionRadius, patchRadius;
		double	minVariance;
	};

	__device__ __forceinline__ std::uint32_t	nforClamp(long long v, std::uint32_t limit)
	{
		return v < 0 ? 0u : (v >= static_cast<long long>(limit) ? limit - 1u : static_cast<std::uint32_t>(v));
	}

	__device__ __forceinline__ int	nforClampInt(int v, int limit)
	{
		return v < 0 ? 0 : (v >= limit ? limit - 1 : v);
	}

	// colorDistanceSquared, colorLuminance (NFOR.cpp:84-103)
	__device__ __forceinline__ double	nforDist2(const double* a, const double* b)
	{
		const double r = a[0] - b[0], g = a[1] - b[1], bl = a[2] - b[2];
		return ((r * r) + (g * g) + (bl * bl)) / 3.0;
	}

	__device__ __forceinline__ double	nforLuminance(const double* c)
	{
		const double l = c[0] * 0.2722287168 + c[1] * 0.6740817658 + c[2] * 0.0536895174;
		return (!isfinite(l) || l <= 0.0) ? 0.0 : l;
	}

	// patchDistance (NFOR.cpp:236-311); border patches clamp their coordinates
	__device__ inline double	nforPatchDistance(const double* guide, const double* variance, const NforParams& P, std::uint32_t x1,
		std::uint32_t y1, std::uint32_t x2, std::uint32_t y2, std::uint32_t patchRadius)
	{
		if (x1 == x2 && y1 == y2) return 0.0;
		const long long r = patchRadius;
		double distance = 0.0;
		unsigned samples = 0;
		for (long long oy = -r; oy <= r; oy++)
		{
			for (long long ox = -r; ox <= r; ox++)
			{
				const std::uint32_t ia = nforClamp(static_cast<long long>(y1) + oy, P.height) * P.width + nforClamp(static_cast<long long>(x1) + ox, P.width);
				const std::uint32_t ib = nforClamp(static_cast<long long>(y2) + oy, P.height) * P.width + nforClamp(static_cast<long long>(x2) + ox, P.width);
				const double lv = variance[ia] + variance[ib] + P.minVariance;
				distance += nforDist2(guide + 3 * ia, guide + 3 * ib) / lv;
				samples++;
			}
		}
		return distance / static_cast<double>(samples);
	}

	// colorWeightFromDistance (NFOR.cpp:313-318)
	__device__ __forceinline__ double	nforWeight(double distance, double bandwidth, double minVariance)
	{
		return exp(-distance / fmax(minVariance, bandwidth * bandwidth));
	}

	// suppressDenoiseFireflies (NFOR.cpp:145-211): a bright pixel with fewer than two similar
	// neighbours in its 5 x 5 window that stands 2.5x and 0.18 above the window's median
	// luminance takes the luminance-median of its darker neighbours. `average` != 0: the
	// input is the mean of a and b (averageColorBuffers) instead of a.
	static __global__ __launch_bounds__(256) void	nfor_fireflies(const double* __restrict__ a, const double* __restrict__ b, double* __restrict__ out,
		NforParams P, int average)
	{
		const std::uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
		if (i >= P.width * P.height) return;
		auto colorAt = [&](std::uint32_t k, double* c) {
			if (average)
			{
				for (int j = 0; j < 3; j++) c[j] = (a[3 * k + j] + b[3 * k + j]) * 0.5;
			}
			else
			{
				for (int j = 0; j < 3; j++) c[j] = a[3 * k + j];
			}
		};
		double center[3];
		colorAt(i, center);
		for (int j = 0; j < 3; j++) out[3 * i + j] = center[j];
		if (P.width < 3 || P.height < 3) return;
		const std::uint32_t x = i % P.width, y = i / P.width;
		const double lum = nforLuminance(center);
		if (lum < 0.30) return;
		const double none = __builtin_nan("");
		double key[24];	// neighbours' luminances, row by row
		std::uint32_t inside = 0, candidates = 0;
		auto neighbor = [&](int k) {
			const int at = k + (k >= 12 ? 1 : 0);
			return (y + static_cast<std::uint32_t>(at / 5) - 2u) * P.width + x + static_cast<std::uint32_t>(at % 5) - 2u;
		};
		#pragma unroll
		for (int k = 0; k < 24; k++)
		{
			const int at = k + (k >= 12 ? 1 : 0);
			const long long sx = static_cast<long long>(x) + at % 5 - 2, sy = static_cast<long long>(y) + at / 5 - 2;
			key[k] = none;
			if (sx < 0 || sy < 0 || sx >= P.width || sy >= P.height) continue;
			double c[3];
			colorAt(neighbor(k), c);
			key[k] = nforLuminance(c);
			inside |= 1u << k;
			if (!(key[k] >= lum * 0.65)) candidates |= 1u << k;
		}
		// isDenoiseFirefly (NFOR.cpp:115-143)
		if (candidates == 0u || __popc(inside & ~candidates) >= 2) return;
		const int middle = medianIndex(key, inside);
		double median = 0.0;
		#pragma unroll
		for (int k = 0; k < 24; k++) median = k == middle ? key[k] : median;
		if (!(lum >= median * 2.5 && lum >= median + 0.18)) return;
		// medianColorByLuminance (NFOR.cpp:105-113)
		#pragma unroll
		for (int k = 0; k < 24; k++)
		{
			if ((candidates >> k & 1u) == 0u) key[k] = none;
		}
		double c[3];
		colorAt(neighbor(medianIndex(key, candidates)), c);
		for (int j = 0; j < 3; j++) out[3 * i + j] = c[j];
	}

	// doubledVariance and averageFeatureVarianceMap (NFOR.cpp:331-353)
	static __global__ void	nfor_variances(const double* __restrict__ colorVariance, const double* __restrict__ featureVariance,
		double* __restrict__ regressionVariance, double* __restrict__ featureVarianceAverage, std::uint32_t n)
	{
		const std::uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
		if (i >= n) return;
		regressionVariance[i] = colorVariance[i] * 2.0;
		double v = 0.0;
		for (int k = 0; k < kNforFeatures; k++) v += featureVariance[kNforFeatures * i + k];
		featureVarianceAverage[i] = v / static_cast<double>(kNforFeatures);
	}

	// prefilterFeatures (NFOR.cpp:403-464): `image`'s features averaged with weights from
	// `guide`'s feature distances and a spatial Gaussian.
	static __global__ void	nfor_prefilter(const double* __restrict__ image, const double* __restrict__ guide,
		const double* __restrict__ varianceAverage, double* __restrict__ out, NforParams P)
	{
		const std::uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
		if (i >= P.width * P.height) return;
		const std::uint32_t x = i % P.width, y = i / P.width;
		const long long r = P.prefilterRadius;
		const double sigma = fmax(1.0, static_cast<double>(P.prefilterRadius));
		double sum[kNforFeatures] = {};
		double total = 0.0;
		for (long long oy = -r; oy <= r; oy++)
		{
			for (long long ox = -r; ox <= r; ox++)
			{
				const std::uint32_t k = nforClamp(static_cast<long long>(y) + oy, P.height) * P.width + nforClamp(static_cast<long long>(x) + ox, P.width);
				const double lv = varianceAverage[i] + varianceAverage[k] + P.minVariance;
				double d = 0.0;
				for (int f = 0; f < kNforFeatures; f++)
				{
					const double diff = guide[kNforFeatures * i + f] - guide[kNforFeatures * k + f];
					d += diff * diff;
				}
				const double distance = (d / static_cast<double>(kNforFeatures)) / lv;
				const double spatial = static_cast<double>(ox * ox + oy * oy);
				const double w = exp(-distance / 0.25) * exp(-spatial / (2.0 * sigma * sigma));
				for (int f = 0; f < kNforFeatures; f++) sum[f] += image[kNforFeatures * k + f] * w;
				total += w;
			}
		}
		for (int f = 0; f < kNforFeatures; f++)
		{
			out[kNforFeatures * i + f] = total <= 2.220446049250313e-16 ? image[kNforFeatures * i + f] : sum[f] / total;
		}
	}

	// weightedAverageFallback (NFOR.cpp:518-553), when a system is singular
	__device__ inline void	nforFallback(const double* image, const double* variance, const NforParams& P, std::uint32_t x, std::uint32_t y,
		double* out)
	{
		const long long r = P.regressionRadius;
		double acc[3] = {0.0, 0.0, 0.0}, total = 0.0;
		for (long long oy = -r; oy <= r; oy++)
		{
			for (long long ox = -r; ox <= r; ox++)
			{
				const std::uint32_t k = nforClamp(static_cast<long long>(y) + oy, P.height) * P.width + nforClamp(static_cast<long long>(x) + ox, P.width);
				const double spatial = static_cast<double>(ox * ox + oy * oy);
				const double w = (1.0 / (variance[k] + P.minVariance)) * exp(-spatial / 8.0);
				for (int j = 0; j < 3; j++) acc[j] += image[3 * k + j] * w;
				total += w;
			}
		}
		const std::uint32_t c = y * P.width + x;
		for (int j = 0; j < 3; j++) out[j] = total <= 2.220446049250313e-16 ? image[3 * c + j] : acc[j] / total;
	}

	constexpr int	kNforTileX = 16, kNforTileY = 8;	// pixels of a regression tile
	constexpr int	kNforTilePixels = kNforTileX * kNforTileY;
	constexpr int	kNforBlock = 512;					// 8 waves, one per tile row
	constexpr int	kNforMaxPatchRadius = 8;
	constexpr int	kNforDepth = 4;						// window samples (k) of one matrix instruction
	constexpr int	kNforChunk = 8;						// window displacements per step, two per lane
	constexpr int	kNforQuads = kNforTileX / 4;		// a wave's row in groups of 4 pixels
	constexpr int	kNforWeightStride = kNforTilePixels + 4;	// doubles between a step's displacements: disjoint LDS banks
	static_assert(kNforBlock == 64 * kNforTileY && 2 * kNforBlock == kNforTilePixels * kNforChunk, "a wave per row, two weights per lane");

	// index of upper-triangle entry (row, col >= row) in the row-major packing
	__host__ __device__ constexpr int	nforUpperIndex(int row, int col)
	{
		return row * kNforBasis - row * (row - 1) / 2 + (col - row);
	}

	// Dynamic LDS of nfor_accumulate, in doubles. Staged: the colours (three planes) and
	// variances of the tile grown by the window and patch radii, and the 11 feature planes of
	// the tile grown by the window radius, each slot holding the pixel of its clamped
	// coordinate. Both forms: the patch terms, the weights and the weights' corrections (a byte
	// each) of two steps each. Strides keep
	// the doubles that lanes read together on disjoint banks: an operand reads four planes at
	// once, up to 7 neighbours of each (planes 8 doubles apart modulo the LDS's 32), and half a
	// wave reads the patch terms of two rows four apart (rows 4 doubles apart modulo 8).
	struct	NforLdsLayout
	{
		int	colorWidth, colorHeight, featureWidth, featureHeight, apronX, apronY, apronStride;
		std::uint32_t	colorStride, featureStride;	// doubles between planes
		std::uint32_t	colors, variances, features, pairs, weights, corrections, doubles;
	};

	__host__ __device__ inline NforLdsLayout	nforLdsLayout(std::uint32_t regressionRadius, std::uint32_t patchRadius, bool staged)
	{
		NforLdsLayout L;
		const int cr = 2 * static_cast<int>(regressionRadius + patchRadius), fr = 2 * static_cast<int>(regressionRadius);
		L.colorWidth = staged ? kNforTileX + cr : 0;
		L.colorHeight = staged ? kNforTileY + cr : 0;
		L.featureWidth = staged ? kNforTileX + fr : 0;
		L.featureHeight = staged ? kNforTileY + fr : 0;
		L.apronX = kNforTileX + 2 * static_cast<int>(patchRadius);
		L.apronY = kNforTileY + 2 * static_cast<int>(patchRadius);
		L.apronStride = L.apronX + (12 - L.apronX % 8) % 8;
		const std::uint32_t cc = static_cast<std::uint32_t>(L.colorWidth * L.colorHeight);
		const std::uint32_t ff = static_cast<std::uint32_t>(L.featureWidth * L.featureHeight);
		L.colorStride = staged ? cc + (40u - cc % 32u) % 32u : 0u;
		L.featureStride = staged ? ff + (40u - ff % 32u) % 32u : 0u;
		L.colors = 0;
		L.variances = 3 * L.colorStride;
		L.features = L.variances + cc;
		L.pairs = L.features + kNforFeatures * L.featureStride;
		L.weights = L.pairs + 2 * kNforChunk * static_cast<std::uint32_t>(L.apronStride * L.apronY);
		L.corrections = L.weights + 2 * kNforChunk * kNforWeightStride;
		L.doubles = L.corrections + 2 * kNforChunk * kNforWeightStride / 8;
		return L;
	}

	// regressionPass (NFOR.cpp:679-737), accumulation: each pixel's 12 x 12 weighted normal
	// matrix and its three right-hand sides, over the samples of its window, at one bandwidth
	// or at two (the systems then differ by the weights only). nfor_solve solves the systems.
	//
	// The sums are a contraction over the window: basis^T (w * [basis | colour]). It runs on
	// the FP64 matrix instruction of four independent 4 x 4 x 4 products: a block is one
	// pixel, k four window samples, and the 12 x 15 system is nine 4 x 4 products (the upper
	// triangle's six and the colours' three), accumulated in two VGPRs each. Lane l holds row
	// or column l % 4 of block (l / 4) % 4 for sample l / 16, so an operand is one feature
	// difference per lane, and a wave's row of 16 pixels at two bandwidths takes 144
	// accumulator VGPRs.
	//
	// A 16 x 8 tile per block of 8 waves. Patch distances: for a window displacement d, the
	// term of patch offset o between pixel p and its sample p + d is D(p + o, p + o + d)
	// (patchDistance, NFOR.cpp:240-311), which depends on p + o only, so a step's terms are
	// evaluated once for every pixel of the tile and its apron into LDS. The stages of a step
	// of 8 displacements (terms, then weights, then products) run on three consecutive steps
	// at once, with one barrier a step; the two waves of a SIMD take them in opposite order.
	// Lanes whose sample would lie off the image take the border sample's own terms. `Two`:
	// bandwidth 1 and half of it; the second weight is the first's fourth power, from the first
	// and a correction that keeps it within 0.6 ulp (a byte beside the weight: eight more would
	// not fit; the host takes two passes where the variance floor breaks that ratio).
	//
	// Staged: the block first copies every colour, variance and feature its window reads into
	// LDS (radius 9, patch radius 1: 153 KiB); the unstaged form reads them from global
	// memory, for windows too wide for LDS.
	//
	// Bound by FP64 issue, which matrix and vector instructions share: at 1280 x 720, radius 9,
	// 5.9 ms for one bandwidth and 8.6 for two, of which the products take 2.4 and 3.8 (1.2 and
	// 2.4 at the matrix unit's rate), the weights 2.0, their corrections 0.5, the terms 1.5,
	// staging and stores 0.6 and 0.9 (each stage's time on its own; they overlap in part). With each lane owning half a pixel's system in vector FMAs, 14 LDS reads a sample and
	// three barriers per 4 displacements, one bandwidth took 8.8 ms. Border lanes that read
	// their patches from global memory cost 1.8 ms of the weights; 16 waves of half the pixels
	// each were slower (spills).
	template <bool Staged, bool Two>
	static __global__ __launch_bounds__(kNforBlock, 2) void	nfor_accumulate(const double* __restrict__ image,
		const double* __restrict__ features, const double* __restrict__ variance, double* __restrict__ system, NforParams P,
		double bandwidth, std::uint32_t firstRow, std::uint32_t rows)
	{
		#pragma clang fp contract(off)
		extern __shared__ double lds[];
		constexpr int Bandwidths = Two ? 2 : 1;
		const NforLdsLayout L = nforLdsLayout(P.regressionRadius, P.patchRadius, Staged);
		double* const colors = lds + L.colors;
		double* const vars = lds + L.variances;
		double* const feats = lds + L.features;
		double* const pairs = lds + L.pairs;
		double* const weights = lds + L.weights;
		std::int8_t* const corrections = reinterpret_cast<std::int8_t*>(lds + L.corrections);
		const int cw = L.colorWidth, fw = L.featureWidth, ax = L.apronX, as = L.apronStride;
		const int cells = cw * L.colorHeight, ff = fw * L.featureHeight, aa = ax * L.apronY, termsSize = as * L.apronY;
		const int cc = static_cast<int>(L.colorStride), fs = static_cast<int>(L.featureStride);
		const int iw = static_cast<int>(P.width), ih = static_cast<int>(P.height);
		const int ir = static_cast<int>(P.regressionRadius), ipr = static_cast<int>(P.patchRadius);
		const int tilesX = (iw + kNforTileX - 1) / kNforTileX;
		const int x0 = static_cast<int>(blockIdx.x % static_cast<unsigned>(tilesX)) * kNforTileX;
		const int y0 = static_cast<int>(firstRow) + static_cast<int>(blockIdx.x / static_cast<unsigned>(tilesX)) * kNforTileY;
		const int thread = static_cast<int>(threadIdx.x);
		auto pixelAt = [&](int x, int y) { return static_cast<size_t>(nforClampInt(y, ih)) * P.width + static_cast<size_t>(nforClampInt(x, iw)); };
		if constexpr (Staged)
		{
			for (int i = thread; i < cells; i += kNforBlock)
			{
				const size_t g = pixelAt(x0 - ir - ipr + i % cw, y0 - ir - ipr + i / cw);
				colors[i] = image[3 * g];
				colors[cc + i] = image[3 * g + 1];
				colors[2 * cc + i] = image[3 * g + 2];
				vars[i] = variance[g];
			}
			for (int i = thread; i < ff; i += kNforBlock)
			{
				const size_t g = pixelAt(x0 - ir + i % fw, y0 - ir + i / fw);
				#pragma unroll
				for (int j = 0; j < kNforFeatures; j++) feats[j * fs + i] = features[kNforFeatures * g + j];
			}
			__syncthreads();
		}
		const int side = 2 * ir + 1;
		const int samples = side * side;
		const int steps = (samples + kNforChunk - 1) / kNforChunk;
		// a window sample's displacement, walked in raster order; past the last sample it is the
		// pixel itself (with weight 0)
		struct	Walk
		{
			int	s, x, y;
		};
		auto walkFrom = [&](int s0) { return Walk{s0, s0 % side - ir, s0 / side - ir}; };
		auto advance = [&](Walk& w) {
			w.s += kNforDepth;
			w.x += kNforDepth % side;
			w.y += kNforDepth / side;
			const bool wrap = w.x > ir;
			w.x -= wrap ? side : 0;
			w.y += wrap ? 1 : 0;
		};

		// Stages that form terms and weights: two waves have displacements kk and kk + 4 of the
		// step, one pixel per lane
		const int kk = __builtin_amdgcn_readfirstlane(thread / kNforTilePixels);
		const int kLane = thread % kNforTilePixels;
		// a patch term of two pixels: slots of the staged colours, or pixels
		auto term = [&](auto a, auto b) {
			double dr, dg, db, lv;
			if constexpr (Staged)
			{
				dr = colors[a] - colors[b];
				dg = colors[cc + a] - colors[cc + b];
				db = colors[2 * cc + a] - colors[2 * cc + b];
				lv = vars[a] + vars[b] + P.minVariance;
			}
			else
			{
				dr = image[3 * a] - image[3 * b];
				dg = image[3 * a + 1] - image[3 * b + 1];
				db = image[3 * a + 2] - image[3 * b + 2];
				lv = variance[a] + variance[b] + P.minVariance;
			}
			return ((dr * dr) + (dg * dg) + (db * db)) / (3.0 * lv);
		};
		// patch terms D(q, q + d) of a step over the tile and its apron, coordinates clamped
		auto pairTerm = [&](int j, const Walk& w, int slot) {
			const int ox = w.s < samples ? w.x : 0, oy = w.s < samples ? w.y : 0;
			const int jy = j / ax, jx = j - jy * ax;
			if constexpr (Staged)
			{
				const int a = (jy + ir) * cw + (jx + ir);	// q = tile origin - patch radius + (jx, jy)
				pairs[slot + jy * as + jx] = term(a, a + oy * cw + ox);
			}
			else pairs[slot + jy * as + jx] = term(pixelAt(x0 - ipr + jx, y0 - ipr + jy), pixelAt(x0 - ipr + jx + ox, y0 - ipr + jy + oy));
		};
		auto formPairs = [&](int t, const Walk& w0, const Walk& w1) {
			const int slot = ((t & 1) * kNforChunk + kk) * termsSize;
			for (int j = kLane; j < aa; j += kNforTilePixels)
			{
				pairTerm(j, w0, slot);
				pairTerm(j, w1, slot + kNforDepth * termsSize);
			}
		};

		// weights of a step (colorWeightFromDistance, NFOR.cpp:313-318), at bandwidth 1
		const int wtx = kLane % kNforTileX, wty = (kLane / kNforTileX % 2) * 4 + kLane / (2 * kNforTileX);
		const int wPixel = wty * kNforTileX + wtx;
		const int wx = x0 + wtx, wy = y0 + wty;
		const bool wActive = wx < iw && wy < ih;
		const double patchTerms = static_cast<double>((2 * ipr + 1) * (2 * ipr + 1));
		const double scale = patchTerms * fmax(P.minVariance, bandwidth * bandwidth);
		const double inverseScale = 1.0 / scale, farthest = 1000.0 * scale;
		auto patchSum = [&](int t, int k, const Walk& at) {
			const int ux = at.s < samples ? wx + at.x : wx, uy = at.s < samples ? wy + at.y : wy;
			const int sx = nforClampInt(ux, iw), sy = nforClampInt(uy, ih);
			double distance = 0.0;
			if (!wActive || (sx == wx && sy == wy))
			{
				distance = 0.0;
			}
			else if (ux == sx && uy == sy)
			{
				// patches may overhang the image: a term's two pixels are clamped one by one, as here
				const double* terms = pairs + ((t & 1) * kNforChunk + k) * termsSize;
				if (ipr == 1)
				{
					// the common 3 x 3 patch: the nine reads issued together, then summed in order
					double v[9];
					#pragma unroll
					for (int i = 0; i < 9; i++) v[i] = terms[(wty + i / 3) * as + (wtx + i % 3)];
					#pragma unroll
					for (int i = 0; i < 9; i++) distance += v[i];
				}
				else
				{
					for (int py = 0; py <= 2 * ipr; py++)
					{
						for (int px = 0; px <= 2 * ipr; px++) distance += terms[(wty + py) * as + (wtx + px)];
					}
				}
			}
			else
			{
				// the window overhangs: the sample is a pixel of the border, with its own patch
				for (int py = -ipr; py <= ipr; py++)
				{
					for (int px = -ipr; px <= ipr; px++)
					{
						if constexpr (Staged)
						{
							const int left = x0 - ir - ipr, top = y0 - ir - ipr;
							distance += term((nforClampInt(wy + py, ih) - top) * cw + nforClampInt(wx + px, iw) - left,
								(nforClampInt(sy + py, ih) - top) * cw + nforClampInt(sx + px, iw) - left);
						}
						else distance += term(pixelAt(wx + px, wy + py), pixelAt(sx + px, sy + py));
					}
				}
			}
			return distance;
		};
		// exp(-distance / scale); the quotient by the reciprocal and one correction (the nearest
		// double, as a division gives it)
		auto weightOf = [&](double distance) {
			distance = distance > farthest ? farthest : distance;
			const double q = distance * inverseScale;
			return nforExpNegative(fma(fma(-q, scale, distance), inverseScale, q));
		};
		auto storeWeight = [&](int at, const NforExp& e, bool sample) {
			weights[at] = sample ? nforWeight1(e) : 0.0;
			if (Two) corrections[at] = sample ? nforWeight4Correction(e) : std::int8_t(0);
		};
		auto formWeights = [&](int t, const Walk& at0, const Walk& at1) {
			const double d0 = patchSum(t, kk, at0), d1 = patchSum(t, kk + kNforDepth, at1);
			const NforExp e0 = weightOf(d0), e1 = weightOf(d1);
			const int at = ((t & 1) * kNforChunk + kk) * kNforWeightStride + wPixel;
			storeWeight(at, e0, wActive && at0.s < samples);
			storeWeight(at + kNforDepth * kNforWeightStride, e1, wActive && at1.s < samples);
		};

		// products of step t
		const int wave = __builtin_amdgcn_readfirstlane(thread / 64);
		const int lane = thread % 64;
		const int li = lane % 4, lb = (lane / 4) % 4, lk = lane / 16;
		// basis entry 4 m + li is 1 for entry 0, else feature 4 m + li - 1 less the pixel's own
		const int plane0 = li > 0 ? li - 1 : 0, plane1 = 3 + li, colorPlane = li < 3 ? li : 2;
		const int fBase = (wave + ir) * fw + (lb + ir);
		const int cBase = (wave + ir + ipr) * cw + (lb + ir + ipr);
		double own[kNforQuads][3];
		#pragma unroll
		for (int q = 0; q < kNforQuads; q++)
		{
			if constexpr (Staged)
			{
				own[q][0] = feats[plane0 * fs + fBase + 4 * q];
				own[q][1] = feats[plane1 * fs + fBase + 4 * q];
				own[q][2] = feats[(plane1 + 4) * fs + fBase + 4 * q];
			}
			else
			{
				const double* f = features + kNforFeatures * pixelAt(x0 + 4 * q + lb, y0 + wave);
				own[q][0] = f[plane0];
				own[q][1] = f[plane1];
				own[q][2] = f[plane1 + 4];
			}
		}
		// [bandwidth][quad]: products 00 01 02 11 12 22 of basis quarters, then 0 1 2 by colour;
		// a fresh system has the ridge 1e-4 on its diagonal
		double acc[Bandwidths][kNforQuads][9];
		#pragma unroll
		for (int b = 0; b < Bandwidths; b++)
		{
			#pragma unroll
			for (int q = 0; q < kNforQuads; q++)
			{
				#pragma unroll
				for (int e = 0; e < 9; e++) acc[b][q][e] = (e == 0 || e == 3 || e == 5) && lk == li ? 1e-4 : 0.0;
			}
		}
		auto multiply = [&](int t, int g, const Walk& at) {
			const int ox = at.s < samples ? at.x : 0, oy = at.s < samples ? at.y : 0;
			const int fOff = oy * fw + ox, cOff = oy * cw + ox;
			const double* f0 = feats + plane0 * fs + fBase + fOff;
			const double* f1 = feats + plane1 * fs + fBase + fOff;
			const double* col = colors + colorPlane * cc + cBase + cOff;
			const int wAt = ((t & 1) * kNforChunk + g * kNforDepth + lk) * kNforWeightStride + wave * kNforTileX + lb;
			#pragma unroll
			for (int q = 0; q < kNforQuads; q++)
			{
				double v0, v1, v2, c;
				if constexpr (Staged)
				{
					v0 = f0[4 * q];
					v1 = f1[4 * q];
					v2 = f1[4 * fs + 4 * q];
					c = col[4 * q];
				}
				else
				{
					const size_t at0 = pixelAt(x0 + 4 * q + lb + ox, y0 + wave + oy);
					const double* f = features + kNforFeatures * at0;
					v0 = f[plane0];
					v1 = f[plane1];
					v2 = f[plane1 + 4];
					c = image[3 * at0 + colorPlane];
				}
				const double d0 = v0 - own[q][0], b1 = v1 - own[q][1], b2 = v2 - own[q][2];
				const double b0 = li == 0 ? 1.0 : d0;
				double wk = weights[wAt + 4 * q];
				const double w4 = Two ? nforWeight4(wk, corrections[wAt + 4 * q]) : 0.0;
				#pragma unroll
				for (int k = 0; k < Bandwidths; k++)
				{
					if (k == 1) wk = w4;
					const double a0 = wk * b0, a1 = wk * b1, a2 = wk * b2;
					double (&d)[9] = acc[k][q];
					d[0] = __builtin_amdgcn_mfma_f64_4x4x4f64(a0, b0, d[0], 0, 0, 0);
					d[1] = __builtin_amdgcn_mfma_f64_4x4x4f64(a0, b1, d[1], 0, 0, 0);
					d[2] = __builtin_amdgcn_mfma_f64_4x4x4f64(a0, b2, d[2], 0, 0, 0);
					d[3] = __builtin_amdgcn_mfma_f64_4x4x4f64(a1, b1, d[3], 0, 0, 0);
					d[4] = __builtin_amdgcn_mfma_f64_4x4x4f64(a1, b2, d[4], 0, 0, 0);
					d[5] = __builtin_amdgcn_mfma_f64_4x4x4f64(a2, b2, d[5], 0, 0, 0);
					d[6] = __builtin_amdgcn_mfma_f64_4x4x4f64(a0, c, d[6], 0, 0, 0);
					d[7] = __builtin_amdgcn_mfma_f64_4x4x4f64(a1, c, d[7], 0, 0, 0);
					d[8] = __builtin_amdgcn_mfma_f64_4x4x4f64(a2, c, d[8], 0, 0, 0);
				}
			}
		};

		Walk walk0 = walkFrom(kk), walk1 = walkFrom(kk + kNforDepth), productWalk = walkFrom(lk);
		auto nextStep = [&]() {
			advance(walk0);
			advance(walk0);
			advance(walk1);
			advance(walk1);
		};
		auto products = [&](int t) {
			#pragma unroll
			for (int g = 0; g < kNforChunk / kNforDepth; g++)
			{
				multiply(t, g, productWalk);
				advance(productWalk);
			}
		};
		formPairs(0, walk0, walk1);
		__syncthreads();
		formWeights(0, walk0, walk1);
		nextStep();
		if (steps > 1) formPairs(1, walk0, walk1);
		__syncthreads();
		const bool first = wave < 4;
		for (int t = 0; t < steps; t++)
		{
			if (first) products(t);
			if (t + 1 < steps) formWeights(t + 1, walk0, walk1);
			nextStep();
			if (t + 2 < steps) formPairs(t + 2, walk0, walk1);
			if (!first) products(t);
			__syncthreads();
		}

		// the systems, slot-major: entry k of pixel p of the band at k * n + p; entries 0..77 the
		// upper triangle, 78 + 3 * row + channel the right-hand sides. A product's row is held
		// by lane / 16, its column by lane % 4.
		const int y = y0 + wave;
		if (y >= ih || y >= static_cast<int>(firstRow + rows)) return;
		const size_t n = static_cast<size_t>(P.width) * rows;
		#pragma unroll
		for (int b = 0; b < Bandwidths; b++)
		{
			#pragma unroll
			for (int q = 0; q < kNforQuads; q++)
			{
				const int x = x0 + 4 * q + lb;
				if (x >= iw) continue;
				double* out = system + static_cast<size_t>(b) * kNforSystem * n + static_cast<size_t>(y - static_cast<int>(firstRow)) * P.width + x;
				int e = 0;
				#pragma unroll
				for (int m = 0; m < 3; m++)
				{
					#pragma unroll
					for (int c = m; c < 3; c++)
					{
						const int row = 4 * m + lk, col = 4 * c + li;
						if (row <= col) out[static_cast<size_t>(nforUpperIndex(row, col)) * n] = acc[b][q][e];
						e++;
					}
				}
				#pragma unroll
				for (int m = 0; m < 3; m++)
				{
					if (li < 3) out[static_cast<size_t>(kNforUpper + 3 * (4 * m + lk) + li) * n] = acc[b][q][6 + m];
				}
			}
		}
	}

	// completeRegressionMatrix (NFOR.cpp:628-637), then solveLinearSystemRGB (:466-516): the
	// reference's Gauss-Jordan elimination with partial pivoting on each system from
	// nfor_accumulate (the pixels of `rows` image rows from firstRow); a singular system takes
	// weightedAverageFallback.
	static __global__ __launch_bounds__(256) void	nfor_solve(const double* __restrict__ system, const double* __restrict__ image,
		const double* __restrict__ variance, double* __restrict__ out, NforParams P, std::uint32_t firstRow, std::uint32_t rows)
	{
		#pragma clang fp contract(off)
		const size_t n = static_cast<size_t>(P.width) * rows;
		const size_t c = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
		if (c >= n) return;
		const std::uint32_t x = static_cast<std::uint32_t>(c % P.width), y = firstRow + static_cast<std::uint32_t>(c / P.width);
		double upper[kNforUpper];
		double rhs[kNforBasis][3];
		#pragma unroll
		for (int k = 0; k < kNforUpper; k++) upper[k] = system[static_cast<size_t>(k) * n + c];
		#pragma unroll
		for (int row = 0; row < kNforBasis; row++)
		{
			#pragma unroll
			for (int j = 0; j < 3; j++) rhs[row][j] = system[static_cast<size_t>(kNforUpper + 3 * row + j) * n + c];
		}
		double m[kNforBasis][kNforBasis];
		{
			int k = 0;
			#pragma unroll
			for (int row = 0; row < kNforBasis; row++)
			{
				#pragma unroll
				for (int col = row; col < kNforBasis; col++)
				{
					m[row][col] = upper[k];
					m[col][row] = upper[k];
					k++;
				}
			}
		}
		bool solved = true;
		#pragma unroll
		for (int pivot = 0; pivot < kNforBasis; pivot++)
		{
			int best = pivot;
			double bestValue = fabs(m[pivot][pivot]);
			#pragma unroll
			for (int row = pivot + 1; row < kNforBasis; row++)
			{
				const double v = fabs(m[row][pivot]);
				if (v > bestValue)
				{
					bestValue = v;
					best = row;
				}
			}
			if (bestValue < 1e-10)
			{
				solved = false;
				break;
			}
			// row swap (columns below the pivot are zero in every row already)
			#pragma unroll
			for (int row = pivot + 1; row < kNforBasis; row++)
			{
				if (row == best)
				{
					#pragma unroll
					for (int col = pivot; col < kNforBasis; col++)
					{
						const double t = m[pivot][col];
						m[pivot][col] = m[row][col];
						m[row][col] = t;
					}
					#pragma unroll
					for (int j = 0; j < 3; j++)
					{
						const double t = rhs[pivot][j];
						rhs[pivot][j] = rhs[row][j];
						rhs[row][j] = t;
					}
				}
			}
			const double pivotValue = m[pivot][pivot];
			#pragma unroll
			for (int col = pivot; col < kNforBasis; col++) m[pivot][col] /= pivotValue;
			#pragma unroll
			for (int j = 0; j < 3; j++) rhs[pivot][j] /= pivotValue;
			#pragma unroll
			for (int row = 0; row < kNforBasis; row++)
			{
				if (row == pivot) continue;
				const double factor = m[row][pivot];
				#pragma unroll
				for (int col = pivot; col < kNforBasis; col++) m[row][col] -= factor * m[pivot][col];
				#pragma unroll
				for (int j = 0; j < 3; j++) rhs[row][j] -= factor * rhs[pivot][j];
			}
		}
		double* o = out + 3 * (static_cast<size_t>(y) * P.width + x);
		if (solved)
		{
			o[0] = rhs[0][0];
			o[1] = rhs[0][1];
			o[2] = rhs[0][2];
		}
		else
		{
			nforFallback(image, variance, P, x, y, o);
		}
	}

	// estimateMSE (NFOR.cpp:875-893) of the first and the second bandwidth
	static __global__ void	nfor_mse(const double* __restrict__ colorA, const double* __restrict__ colorB, const double* __restrict__ a0,
		const double* __restrict__ b0, const double* __restrict__ a1, const double* __restrict__ b1,
		const double* __restrict__ variance, double* __restrict__ mse0, double* __restrict__ mse1, std::uint32_t n)
	{
		const std::uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
		if (i >= n) return;
		auto mse = [&](const double* fa, const double* fb) {
			const double mseA = nforDist2(colorB + 3 * i, fa + 3 * i) - 2.0 * variance[i];
			const double mseB = nforDist2(colorA + 3 * i, fb + 3 * i) - 2.0 * variance[i];
			const double residual = nforDist2(fa + 3 * i, fb + 3 * i) * 0.25;
			return fmax(0.0, ((mseA + mseB) * 0.5) - residual);
		};
		mse0[i] = mse(a0, b0);
		mse1[i] = mse(a1, b1);
	}

	// filterScalarMapPair (NFOR.cpp:834-873): radius-3 cross-bilateral filter of two maps,
	// weights from 3 x 3 colour patches of `guide` (bandwidth 1). `select` != 0: the maps are
	// first turned into bandwidthSelectionMap(first, second) and (second, first) (:907-919).
	static __global__ void	nfor_filter_pair(const double* __restrict__ first, const double* __restrict__ second,
		const double* __restrict__ guide, const double* __restrict__ guideVariance, double* __restrict__ out0,
		double* __restrict__ out1, NforParams P, int select)
	{
		const std::uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
		if (i >= P.width * P.height) return;
		const std::uint32_t x = i % P.width, y = i / P.width;
		auto value = [&](std::uint32_t k, double& v0, double& v1) {
			if (select)
			{
				v0 = first[k] <= second[k] ? 1.0 : 0.0;
				v1 = second[k] <= first[k] ? 1.0 : 0.0;
			}
			else
			{
				v0 = first[k];
				v1 = second[k];
			}
		};
		double f0 = 0.0, f1 = 0.0, total = 0.0;
		for (long long oy = -3; oy <= 3; oy++)
		{
			for (long long ox = -3; ox <= 3; ox++)
			{
				const std::uint32_t sx = nforClamp(static_cast<long long>(x) + ox, P.width);
				const std::uint32_t sy = nforClamp(static_cast<long long>(y) + oy, P.height);
				const std::uint32_t k = sy * P.width + sx;
				const double w = nforWeight(nforPatchDistance(guide, guideVariance, P, x, y, sx, sy, 1u), 1.0, P.minVariance);
				double v0, v1;
				value(k, v0, v1);
				f0 += v0 * w;
				f1 += v1 * w;
				total += w;
			}
		}
		if (total > 2.220446049250313e-16)
		{
			out0[i] = f0 / total;
			out1[i] = f1 / total;
		}
		else
		{
			value(i, out0[i], out1[i]);
		}
	}

	// The per-pixel blend of applyNFOR (NFOR.cpp:1072-1087) and combinedResultVariance
	// (:895-905): combined colour, blended features and the final regression's variance.
	static __global__ void	nfor_combine(const double* __restrict__ sel0, const double* __restrict__ sel1, const double* __restrict__ mse0,
		const double* __restrict__ mse1, const double* __restrict__ a0, const double* __restrict__ a1, const double* __restrict__ b0,
		const double* __restrict__ b1, const double* __restrict__ featA, const double* __restrict__ featB,
		double* __restrict__ combined, double* __restrict__ features, double* __restrict__ variance, NforParams P)
	{
		const std::uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
		if (i >= P.width * P.height) return;
		const double total = sel0[i] + sel1[i];
		const double w0 = total > P.minVariance ? sel0[i] / total : (mse0[i] <= mse1[i] ? 1.0 : 0.0);
		for (int j = 0; j < 3; j++)
		{
			const double ra = a0[3 * i + j] * w0 + a1[3 * i + j] * (1.0 - w0);
			const double rb = b0[3 * i + j] * w0 + b1[3 * i + j] * (1.0 - w0);
			combined[3 * i + j] = (ra + rb) * 0.5;
		}
		for (int f = 0; f < kNforFeatures; f++)
		{
			features[kNforFeatures * i + f] = featA[kNforFeatures * i + f] * 0.5 + featB[kNforFeatures * i + f] * (1.0 - 0.5);
		}
		variance[i] = nforDist2(a1 + 3 * i, b1 + 3 * i) * 0.25;
	}
#endif
}
