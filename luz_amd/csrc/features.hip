// The kernels that are compiled per scene feature class (LUZ_FEATURES, layout.h kFeat*): the
// wavefront stages, the plain kernels and the adjoint. One translation unit per class, so the
// classes compile side by side.
#include <hip/hip_runtime.h>

#include "device/mega.hpp"
#include "device/wavefront.hpp"

namespace luzgpu
{
	template void	enqueuePassF<LUZ_FEATURES>(WavefrontState&, const SceneView&, std::uint32_t, int, bool, unsigned long long*, hipStream_t,
		bool, WaveTuning, std::vector<hipEvent_t>*);
	template void	launchMegaF<LUZ_FEATURES>(bool, size_t, hipStream_t, const SceneView&, const GpuParams&, const std::uint32_t*,
		std::uint32_t, float*, unsigned long long*);
	template void	launchMegaBatchF<LUZ_FEATURES>(bool, size_t, hipStream_t, const SceneView&, const MegaJob*, std::uint32_t, float*,
		unsigned long long*);
	template void	launchMegaDenoiseF<LUZ_FEATURES>(size_t, hipStream_t, const SceneView&, const GpuParams&, const std::uint32_t*,
		std::uint32_t, float*, float*, unsigned long long*);
	template void	launchAdjointF<LUZ_FEATURES>(size_t, size_t, hipStream_t, const SceneView&, const GpuParams&, const float*, double*,
		std::uint32_t);
}
