// The middle element of a small set by rank, without sorting it.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace luzgpu
{
	// Index of the element that a stable ascending sort of the valid ones (bits of `valid`, not
	// empty) puts at popc(valid) / 2. Keys of valid elements are no NaN; those of the others are.
	//
	// Sorting at run-time indexes would keep the arrays in scratch memory, which bounded both
	// firefly filters (1080p display 0.58 -> 0.10 ms, the denoiser's three passes at 720p 0.49 ->
	// 0.21 ms). Unrolled, the keys and ranks stay in registers: one compare a pair. An
	// invalid element compares false with everything, so it counts as before each valid one
	// that follows it (taken off at the end) and never moves one that precedes it.
	template <int N>
	__device__ __forceinline__ int	medianIndex(const double (&key)[N], std::uint32_t valid)
	{
		int rank[N] = {};
		#pragma unroll
		for (int i = 1; i < N; i++)
		{
			#pragma unroll
			for (int j = 0; j < i; j++)
			{
				const int after = key[j] > key[i] ? 1 : 0;
				rank[j] += after;
				rank[i] += 1 - after;
			}
		}
		const int middle = __popc(valid) / 2;
		int at = 0;
		#pragma unroll
		for (int i = 0; i < N; i++)
		{
			if ((valid >> i & 1u) != 0u && rank[i] - __popc(~valid & ((1u << i) - 1u)) == middle) at = i;
		}
		return at;
	}
}
