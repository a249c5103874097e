// The plain (megakernel) integrator's kernels, one thread per (pixel, sample) with the whole
// path in registers: single scene, several scenes in one launch, with denoising features, and
// the path-replay adjoint. Each launch function is instantiated per scene feature class in its
// own translation unit (features.hip).
#pragma once

#include "adjoint.hpp"
#include "integrator.hpp"
#include "nfor.hpp"

#include <hip/hip_runtime.h>

namespace luzgpu
{
	constexpr int	kMegaBlock = 128;
	constexpr int	kStackDepth = 48;

	// counters: [0] closest-hit rays, [1] shadow rays, [2] nodes visited, [3] primitives tested.
	// Renders samples [sampleBegin, sampleBegin + sampleCount) of `pixels` pixels: entries of
	// `list` (adaptive rounds), or the whole image when `list` is nullptr.
	template <bool Count, int Feat>
	static __global__ __launch_bounds__(kMegaBlock) void	render_mega(SceneView s, GpuParams p, const std::uint32_t* __restrict__ list,
		std::uint32_t pixels, float* __restrict__ sampleColors, unsigned long long* __restrict__ counters)
	{
		__shared__ std::uint32_t stackMem[kStackDepth * kMegaBlock];
		const std::uint64_t gid = static_cast<std::uint64_t>(blockIdx.x) * kMegaBlock + threadIdx.x;
		std::uint32_t closest = 0, shadow = 0;
		VisitCounter visits{0u, 0u};
		if (gid < static_cast<std::uint64_t>(pixels) * p.sampleCount)
		{
			const std::uint32_t slot = static_cast<std::uint32_t>(gid / pixels);
			const std::uint32_t entry = static_cast<std::uint32_t>(gid % pixels);
			const std::uint32_t pixel = list ? list[entry] : entry;
			LdsStack<kStackDepth, kMegaBlock> stack{stackMem + threadIdx.x, 0};
			const f3 c = cleanColor(tracePath<Count, Feat>(s, p, pixel % p.width, pixel / p.width, p.sampleBegin + slot, stack, closest, shadow, visits));
			float* out = sampleColors + (static_cast<size_t>(slot) * pixels + entry) * 3;
			out[0] = c.x;
			out[1] = c.y;
			out[2] = c.z;
		}
		// one atomic per wave for the ray counters
		for (int off = 32; off > 0; off >>= 1)
		{
			closest += __shfl_down(closest, off);
			shadow += __shfl_down(shadow, off);
			if (Count)
			{
				visits.nodes += __shfl_down(visits.nodes, off);
				visits.prims += __shfl_down(visits.prims, off);
			}
		}
		if ((threadIdx.x & 63) == 0)
		{
			atomicAdd(counters + 0, static_cast<unsigned long long>(closest));
			atomicAdd(counters + 1, static_cast<unsigned long long>(shadow));
			if (Count)
			{
				atomicAdd(counters + 2, static_cast<unsigned long long>(visits.nodes));
				atomicAdd(counters + 3, static_cast<unsigned long long>(visits.prims));
			}
		}
	}

	template <int Feat>
	void	launchMegaF(bool count, size_t grid, hipStream_t st, const SceneView& s, const GpuParams& p, const std::uint32_t* list,
		std::uint32_t pixels, float* colors, unsigned long long* counters)
	{
		if (count) render_mega<true, Feat><<<grid, kMegaBlock, 0, st>>>(s, p, list, pixels, colors, counters);
		else render_mega<false, Feat><<<grid, kMegaBlock, 0, st>>>(s, p, list, pixels, colors, counters);
	}

	// One scene of a batched plain-kernel launch. Its (pixel, sample) threads start on a wave
	// boundary, so every wave renders one scene and reads that scene's parameters with
	// scalar loads.
	struct	MegaJob
	{
		GpuParams	params;			// sampleBegin / sampleCount: this launch's slice
		std::uint32_t	firstWave;	// first wave of the slice in the launch
		std::uint32_t	pixels;
		std::uint32_t	count;		// pixels * sampleCount
		std::uint32_t	pixelBase;	// first pixel of the scene in the launch's pixel numbering
		std::uint64_t	colorBase;	// first sample colour of the slice
		double*	sums;			// the scene's FP64 pixel sums
	};

	// Several scenes in one launch (render_batch on the plain kernel): small scenes that
	// cannot fill the GPU alone run side by side, each path still in one thread.
	template <bool Count, int Feat>
	static __global__ __launch_bounds__(kMegaBlock) void	render_mega_batch(SceneView s, const MegaJob* __restrict__ jobs, std::uint32_t jobCount,
		float* __restrict__ sampleColors, unsigned long long* __restrict__ counters)
	{
		__shared__ std::uint32_t stackMem[kStackDepth * kMegaBlock];
		const std::uint32_t wave = __builtin_amdgcn_readfirstlane((blockIdx.x * kMegaBlock + threadIdx.x) >> 6);
		std::uint32_t lo = 0, hi = jobCount;
		while (hi - lo > 1u)
		{
			const std::uint32_t mid = (lo + hi) >> 1;
			if (jobs[mid].firstWave <= wave) lo = mid;
			else hi = mid;
		}
		const MegaJob& J = jobs[__builtin_amdgcn_readfirstlane(lo)];
		const std::uint32_t local = (wave - J.firstWave) * 64u + (threadIdx.x & 63u);
		std::uint32_t closest = 0, shadow = 0;
		VisitCounter visits{0u, 0u};
		if (wave >= J.firstWave && local < J.count)
		{
			const GpuParams& p = J.params;
			const std::uint32_t slot = local / J.pixels, pixel = local % J.pixels;
			LdsStack<kStackDepth, kMegaBlock> stack{stackMem + threadIdx.x, 0};
			const f3 c = cleanColor(tracePath<Count, Feat>(s, p, pixel % p.width, pixel / p.width, p.sampleBegin + slot, stack, closest,
				shadow, visits));
			float* out = sampleColors + (J.colorBase + local) * 3;
			out[0] = c.x;
			out[1] = c.y;
			out[2] = c.z;
		}
		for (int off = 32; off > 0; off >>= 1)
		{
			closest += __shfl_down(closest, off);
			shadow += __shfl_down(shadow, off);
			if (Count)
			{
				visits.nodes += __shfl_down(visits.nodes, off);
				visits.prims += __shfl_down(visits.prims, off);
			}
		}
		if ((threadIdx.x & 63) == 0)
		{
			atomicAdd(counters + 0, static_cast<unsigned long long>(closest));
			atomicAdd(counters + 1, static_cast<unsigned long long>(shadow));
			if (Count)
			{
				atomicAdd(counters + 2, static_cast<unsigned long long>(visits.nodes));
				atomicAdd(counters + 3, static_cast<unsigned long long>(visits.prims));
			}
		}
	}

	template <int Feat>
	void	launchMegaBatchF(bool count, size_t grid, hipStream_t st, const SceneView& s, const MegaJob* jobs, std::uint32_t n, float* colors,
		unsigned long long* counters)
	{
		if (count) render_mega_batch<true, Feat><<<grid, kMegaBlock, 0, st>>>(s, jobs, n, colors, counters);
		else render_mega_batch<false, Feat><<<grid, kMegaBlock, 0, st>>>(s, jobs, n, colors, counters);
	}

	// The plain kernel with denoising on: each (pixel, sample) also writes its primary
	// features (kNforFeatures floats, RenderSample of _calculatePixelSample, ColorHelper.cpp:1119-1126).
	template <int Feat>
	static __global__ __launch_bounds__(kMegaBlock) void	render_mega_denoise(SceneView s, GpuParams p, const std::uint32_t* __restrict__ list,
		std::uint32_t pixels, float* __restrict__ sampleColors, float* __restrict__ sampleFeatures, unsigned long long* __restrict__ counters)
	{
		__shared__ std::uint32_t stackMem[kStackDepth * kMegaBlock];
		const std::uint64_t gid = static_cast<std::uint64_t>(blockIdx.x) * kMegaBlock + threadIdx.x;
		std::uint32_t closest = 0, shadow = 0;
		VisitCounter visits{0u, 0u};
		if (gid < static_cast<std::uint64_t>(pixels) * p.sampleCount)
		{
			const std::uint32_t slot = static_cast<std::uint32_t>(gid / pixels);
			const std::uint32_t entry = static_cast<std::uint32_t>(gid % pixels);
			const std::uint32_t pixel = list ? list[entry] : entry;
			LdsStack<kStackDepth, kMegaBlock> stack{stackMem + threadIdx.x, 0};
			float f[kNforFeatures];
			const f3 c = cleanColor(tracePath<false, Feat>(s, p, pixel % p.width, pixel / p.width, p.sampleBegin + slot, stack, closest,
				shadow, visits, static_cast<NoAdjoint*>(nullptr), f));
			const size_t k = static_cast<size_t>(slot) * pixels + entry;
			sampleColors[3 * k] = c.x;
			sampleColors[3 * k + 1] = c.y;
			sampleColors[3 * k + 2] = c.z;
			for (int j = 0; j < kNforFeatures; j++) sampleFeatures[kNforFeatures * k + j] = f[j];
		}
		for (int off = 32; off > 0; off >>= 1)
		{
			closest += __shfl_down(closest, off);
			shadow += __shfl_down(shadow, off);
		}
		if ((threadIdx.x & 63) == 0)
		{
			if (closest) atomicAdd(counters + 0, static_cast<unsigned long long>(closest));
			if (shadow) atomicAdd(counters + 1, static_cast<unsigned long long>(shadow));
		}
	}

	template <int Feat>
	void	launchMegaDenoiseF(size_t grid, hipStream_t st, const SceneView& s, const GpuParams& p, const std::uint32_t* list,
		std::uint32_t pixels, float* colors, float* feats, unsigned long long* counters)
	{
		render_mega_denoise<Feat><<<grid, kMegaBlock, 0, st>>>(s, p, list, pixels, colors, feats, counters);
	}

	// Path-replay adjoint, one thread per (pixel, sample): dLdI is dLoss/dImage (W*H*3),
	// grads receives kGradPerMaterial FP64 sums per material.
	template <int Feat>
	static __global__ __launch_bounds__(kMegaBlock) void	adjoint_mega(SceneView s, GpuParams p, const float* __restrict__ dLdI,
		double* __restrict__ grads, std::uint32_t materialCount)
	{
		__shared__ std::uint32_t stackMem[kStackDepth * kMegaBlock];
		extern __shared__ float ldsGrads[];
		const std::uint32_t n = materialCount * kGradPerMaterial;
		for (std::uint32_t i = threadIdx.x; i < n; i += kMegaBlock) ldsGrads[i] = 0.0f;
		__syncthreads();
		const std::uint32_t pixels = p.width * p.height;
		const size_t id = static_cast<size_t>(blockIdx.x) * kMegaBlock + threadIdx.x;
		if (id < static_cast<size_t>(pixels) * p.sampleCount)
		{
			const std::uint32_t pixel = static_cast<std::uint32_t>(id % pixels), slot = static_cast<std::uint32_t>(id / pixels);
			LdsStack<kStackDepth, kMegaBlock> stack{stackMem + threadIdx.x, 0};
			AdjointRecorder rec;
			rec.grads = ldsGrads;
			rec.count = 0;
			rec.pendingMaterial = -1;
			rec.pendingScale = 0.0f;
			rec.materials = s.materials;
			const float inv = 1.0f / static_cast<float>(p.sampleCount);
			rec.weight = mk(dLdI[3 * static_cast<size_t>(pixel)] * inv, dLdI[3 * static_cast<size_t>(pixel) + 1] * inv,
				dLdI[3 * static_cast<size_t>(pixel) + 2] * inv);
			std::uint32_t closest = 0, shadow = 0;
			VisitCounter visits{0u, 0u};
			const f3 L = tracePath<false, Feat>(s, p, pixel % p.width, pixel / p.width, p.sampleBegin + slot, stack, closest, shadow,
				visits, &rec);
			rec.finish(L);
		}
		__syncthreads();
		for (std::uint32_t i = threadIdx.x; i < n; i += kMegaBlock)
		{
			if (ldsGrads[i] != 0.0f) atomicAdd(grads + i, static_cast<double>(ldsGrads[i]));
		}
	}

	template <int Feat>
	void	launchAdjointF(size_t grid, size_t shmem, hipStream_t st, const SceneView& s, const GpuParams& p, const float* dLdI, double* grads,
		std::uint32_t materialCount)
	{
		// the adjoint refuses Burley subsurface scenes
		constexpr int F = Feat & ~kFeatSubsurface;
		adjoint_mega<F><<<grid, kMegaBlock, shmem, st>>>(s, p, dLdI, grads, materialCount);
	}
}
