// Wavefront integrator: the bounce loop of calculateLightRaysColor (ColorHelper.cpp:1136-1326)
// split into stages over SoA path state in HBM, so the traversal kernels carry only a ray,
// a stack and a hit record (low VGPR count, high occupancy) and the shading kernel carries
// no traversal state.
//
// It is multi-scene by construction: a launch renders a batch of scenes whose device
// arrays were merged into one SceneView (per-scene bases in GpuParams), and one render of
// one scene is a batch of one. A pass renders a slice of samples of every scene of the
// batch; its paths are numbered globally (scene job j owns [pathBase_j, pathBase_j +
// pixels_j * samples_j), sample slot major), and every queued ray carries its scene id.
//
// Per pass:
//   raygen            camera rays (FP64, bit-exact sampler) -> queue 0, path state init
//   for b = 0..maxBounces:
//     extend          closest hit for every ray of queue b (persistent, lane refill)
//     shade           first adds the visible connections of the path's previous vertex in the
//                     reference's order (light, then environment); then miss / emission /
//                     scatter / NEE and environment connections, in batches one scene per
//                     wave iteration (waterfall over the wave's scene ids); the next ray and
//                     up to two shadow rays are appended with one atomic per block and queue;
//                     a path that ended writes its colour
//     shadow          any-hit test of the appended shadow rays -> visibility bytes
//   accumulate        adds the pass's sample colours into each scene's FP64 pixel sums; a path
//                     that ended with connections to test gets them added here
// Queue lengths and the pass's job table live in device memory and every stage is a
// grid-stride or work-claiming loop over them, so a pass is a fixed launch sequence that
// the host captures once as a hipGraph and replays for every pass.
#pragma once

#include "adaptive.hpp"
#include "integrator.hpp"
#include "nfor.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <stdexcept>
#include <string>
#include <vector>

namespace luzgpu
{
	// path flags
	constexpr std::uint32_t	PF_PREV_SPECULAR = 1u;
	constexpr std::uint32_t	PF_PREV_INFINITE = 2u;
	constexpr std::uint32_t	PF_CONN_LIGHT = 8u;	// a light connection is pending
	constexpr std::uint32_t	PF_CONN_ENV = 16u;	// an environment connection is pending

	// A value that all lanes of the wave hold, as a scalar.
	__device__ __forceinline__ std::uint32_t	uniform(std::uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

	constexpr int	kMaxBounceSlots = 64;
	// A queue is eight parts, each with its own counters: the camera rays go to the parts tile by
	// tile, a path stays in its part, and blocks k, k + 8, ... work on part k. Appends and claims
	// on one counter queue up behind each other at about 12 ns each however many waves there
	// are, which bounded every launch of short rays. Eight also follow the eight XCDs that blocks
	// are dealt to in turn, so a part stays within one XCD's L2. One part -> eight: traversal of
	// the material test scene at 641x479, 17 samples 2.0 -> 0.8 ms, of the 300x300 box at 50
	// samples 4.6 -> 2.7 ms, of an uneven 16-scene batch 10.1 -> 7.7 ms (its shade 6.9 -> 6.1 ms).
	// Tiles are 512 paths: with 64, a shade block's paths lie in four places of the image and
	// spheres at 1080p shades in 10.1 instead of 8.6 ms; from 512 to 4096 the times are level,
	// and small passes spread best over the smallest.
	constexpr std::uint32_t	kQueueParts = 8;
	constexpr std::uint32_t	kPartTile = 512;	// paths, a multiple of 64
	constexpr std::uint32_t	kCounterStride = 64;	// words between counters: lines of their own
	enum : int { COUNT_RAYS = 0, COUNT_SHADOW = 1, CLAIM_EXTEND = 2, CLAIM_SHADOW = 3, kCounterKinds = 4 };
	constexpr std::uint32_t	kCounterWords = kCounterKinds * kMaxBounceSlots * kQueueParts * kCounterStride;

	// The part of tile t: each row of kQueueParts tiles gives every part one, turned by a hash of
	// the row so that no part follows a column of the image.
	__host__ __device__ __forceinline__ std::uint32_t	partOfTile(std::uint32_t t)
	{
		return (t + ((t / kQueueParts * 0x9e3779b1u) >> 29)) % kQueueParts;
	}

	struct	WaveBuffers
	{
		// queue-ordered (double-buffered by bounce parity)
		float4*	qOrigin[2];
		float4*	qDir[2];		// xyz, w = hittable the ray leaves from (bits)
		std::int32_t*	qFrom[2];	// its triangle slot / cube face (RayOrigin::tri)
		std::uint32_t*	qPath[2];
		float4*	qHit;		// t, u, v, hittable (bits)
		std::int32_t*	qTri;
		// path-ordered
		float4*	throughput;	// xyz, w = previous scatter pdf
		float4*	radiance;	// xyz, w = flags (bits)
		float4*	prevOrigin;
		float4*	connection;	// [2 * path + slot]: contribution xyz
		std::uint8_t*	visible;	// [2 * path + slot]
		// shadow queue (rebuilt every bounce)
		float4*	sOrigin;	// xyz, w = tMax
		float4*	sDir;		// xyz, w = scene << 25 | (2 * path + slot) (bits)
		float*	sLogU;		// volume free-flight sample of the shadow ray (batches with volumes)
		int2*	sFrom;		// RayOrigin of the shadow ray (hittable bits, tri)
		std::uint32_t*	counts;		// see counter(); then the pass's path count and the part stride
		std::uint32_t	capacity;
		std::uint32_t*	spill;		// traversal stack spill, [entry][grid thread]
		// Queued extension rays carry their scene above the global path id in qPath
		// (scene << pathBits | path), shadow rays above the connection slot in their tag
		// (scene << (pathBits + 1) | 2 * path + slot). pathBits = 31 - the bits of the largest
		// scene index of the render: 31 for one scene, 24 for 127.
		std::uint32_t	pathBits;

		// Counter `kind` of bounce b and queue part `part` (see kQueueParts).
		__device__ __forceinline__ std::uint32_t*	counter(int kind, int b, std::uint32_t part) const
		{
			return counts + ((static_cast<std::uint32_t>(kind) * kMaxBounceSlots + static_cast<std::uint32_t>(b)) * kQueueParts + part) * kCounterStride;
		}
		__device__ __forceinline__ std::uint32_t	pathCount() const { return counts[kCounterWords]; }
		// queue entries of a part: [part * partStride(), + its count); shadow rays at twice that
		__device__ __forceinline__ std::uint32_t	partStride() const { return counts[kCounterWords + 1]; }

		__device__ __forceinline__ std::uint32_t	sceneOfPath(std::uint32_t qp) const { return qp >> pathBits; }
		__device__ __forceinline__ std::uint32_t	pathOf(std::uint32_t qp) const { return qp & ((1u << pathBits) - 1u); }
		__device__ __forceinline__ std::uint32_t	queuedPath(std::uint32_t scene, std::uint32_t path) const { return (scene << pathBits) | path; }
		__device__ __forceinline__ std::uint32_t	shadowTag(std::uint32_t scene, std::uint32_t slot) const
		{
			return pathBits < 31u ? (scene << (pathBits + 1u)) | slot : slot;
		}
		__device__ __forceinline__ std::uint32_t	sceneOfTag(std::uint32_t tag) const { return pathBits < 31u ? tag >> (pathBits + 1u) : 0u; }
		__device__ __forceinline__ std::uint32_t	slotOfTag(std::uint32_t tag) const
		{
			return pathBits < 31u ? tag & ((2u << pathBits) - 1u) : tag;
		}
	};

	// Queued extension rays carry their volume sample in qOrigin.w.
	constexpr std::uint32_t	kMaxBatchScenes = 127;
	// Paths per pass: 2^27 (~39 GB of path state, 1920 x 1080 x 64 samples in one pass), fewer
	// when a batch's scene bits leave less room in the 32-bit queue entries (2^24 at 127 scenes).
	constexpr std::uint32_t	kMaxPassPaths = 1u << 27;

	// pathBits of a render of n scenes (see WaveBuffers).
	inline std::uint32_t	pathBitsFor(std::uint32_t n)
	{
		std::uint32_t sceneBits = 0;
		while ((1u << sceneBits) < n) sceneBits++;
		return 31u - sceneBits;
	}

	// One scene of a pass. The table lives in device memory: a pass is replayed with a new
	// table and the same launches.
	struct	PassJob
	{
		GpuParams	params;		// sampleBegin / sampleCount: this pass's slice
		std::uint32_t	pathBase;	// first global path id of the slice
		std::uint32_t	pixels;		// pixels rendered: the image, or the entries of pixelList
		double*	sums;			// the scene's FP64 pixel sums
		std::uint32_t	pixelsInverse;	// floor(2^32 / pixels) and floor(2^32 / width) for divide()
		std::uint32_t	widthInverse;
		const std::uint32_t*	pixelList;	// adaptive rounds: the active pixels (nullptr: every pixel)
		double*	moments;		// adaptive rounds: per-pixel AdaptiveAccumulator (or nullptr)
		float*	features;		// denoising: primary features per global path id (or nullptr)
		double*	denoise;		// denoising: per-pixel statistics (kDenoiseStats) instead of sums
	};

	// n / d and n % d for inverse = floor(2^32 / d) (0xffffffff for d = 1): the estimate is at
	// most one short.
	__host__ __device__ __forceinline__ std::uint32_t	divide(std::uint32_t n, std::uint32_t d, std::uint32_t inverse, std::uint32_t& rest)
	{
		std::uint32_t q = static_cast<std::uint32_t>((static_cast<std::uint64_t>(n) * inverse) >> 32);
		rest = n - q * d;
		const bool more = rest >= d;
		q += more ? 1u : 0u;
		rest -= more ? d : 0u;
		return q;
	}

	inline std::uint32_t	inverseOf(std::uint32_t d)
	{
		return d <= 1u ? 0xffffffffu : static_cast<std::uint32_t>((1ull << 32) / d);
	}

	// A colour that no sample has (cleanColor leaves finite values only): the path ended with
	// connections that had yet to be tested, and accumulation adds them (pathColor).
	constexpr std::uint32_t	kPendingColor = 0x7fc0beefu;

	// Adds the visible ones of a path's connections to its radiance (light, then environment).
	__device__ __forceinline__ f3	addConnections(const WaveBuffers& w, std::uint32_t path, std::uint32_t flags, f3 acc)
	{
		if ((flags & PF_CONN_LIGHT) && w.visible[2 * path])
		{
			const float4 c = w.connection[2 * path];
			acc = acc + clampRay(mk(c.x, c.y, c.z));
		}
		if ((flags & PF_CONN_ENV) && w.visible[2 * path + 1])
		{
			const float4 c = w.connection[2 * path + 1];
			acc = acc + clampRay(mk(c.x, c.y, c.z));
		}
		return acc;
	}

	// The cleaned colour of sample (path) `g` of a pass.
	__device__ __forceinline__ void	pathColor(const WaveBuffers& w, const float* __restrict__ colors, size_t g, float (&out)[3])
	{
		const float* c = colors + 3 * g;
		out[0] = c[0];
		out[1] = c[1];
		out[2] = c[2];
		if (__float_as_uint(out[0]) == kPendingColor)
		{
			const std::uint32_t path = static_cast<std::uint32_t>(g);
			const float4 r4 = w.radiance[path];
			const f3 v = cleanColor(addConnections(w, path, __float_as_uint(r4.w), mk(r4.x, r4.y, r4.z)));
			out[0] = v.x;
			out[1] = v.y;
			out[2] = v.z;
		}
	}

	// Image pixel of entry i of a pass's pixel range.
	__device__ __forceinline__ std::uint32_t	passPixel(const PassJob& J, std::uint32_t i)
	{
		return J.pixelList ? J.pixelList[i] : i;
	}

	constexpr int	kWaveBlock = 256;
	constexpr int	kWaveLdsStack = 16;		// default LDS stack entries per lane (tunable: 8, 16, 24)
	constexpr int	kWaveLdsStackMin = 8;
	constexpr int	kWaveStackCapacity = 64;
	constexpr unsigned	kWaveGrid = 2048;	// 256 CUs x 8 waves per SIMD x 4 SIMDs / 4 waves per block
	// default traversal launch shape: as many persistent waves as the traversal kernels'
	// registers let every SIMD hold (256 CUs x 4 SIMDs x 5 waves / 4 waves per block). 1080p
	// spheres: 32.0 ms a frame, against 34.3 with 1024 blocks and 32.2 with 1536 and 2048; 720p
	// hazy terrain 71.5 to 72.7 with any of them.
	constexpr unsigned	kDefaultGrid = 1280;
	// Idle lanes at which a wave takes new rays when the caller names no number: 48 in
	// triangle-only scenes (1080p spheres: 32.0 ms a frame, against 34.3 at 64, 33.0 at 32 and
	// 33.9 at 16), 16 in scenes with analytic primitives or volumes, whose rays differ more in
	// length (720p hazy terrain: 71.8 ms, against 72.8 at 8, 76.4 at 32, 83.8 at 48 and 106 at 64).
	constexpr int	kRefillTriangles = 48;
	constexpr int	kRefillAnalytic = 16;
	// Lanes whose next entry is a leaf (primitive tests, an instance entry) wait while other
	// lanes of the wave still have internal nodes to open, until this many are waiting or no
	// lane has a node left; then every live lane takes one step. Each lane's entries are
	// processed in the same order as without the wait, so results do not depend on it; it
	// only lets the wave run the node code and the leaf code less often side by side. The
	// triangle-only kernels wait for 16 lanes (1080p spheres: 31.9 ms a frame, against 32.8 at 8,
	// 32.4 at 24 and 32.8 at 32); the others for 32 on closest-hit rays and 48 on shadow rays (720p
	// hazy terrain: 72.3 ms, against 72.6 at 32 / 32, 73.5 at 24 / 24 and 75.6 at 16 / 16).
	template <int Feat, bool AnyHit>
	constexpr int	kLeafBatch = Feat == 0 ? 16 : (AnyHit ? 48 : 32);

	__device__ __forceinline__ std::uint32_t	laneId() { return threadIdx.x & 63u; }

	// Clears the pass's counters and sets its path count, the part stride and the parts' shares
	// of queue 0, which holds every path: tile t of kPartTile paths is in part partOfTile(t).
	static __global__ void	wf_zero_counts(WaveBuffers w, const PassJob* jobs, std::uint32_t jobCount)
	{
		const std::uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
		if (i >= kCounterWords / kCounterStride) return;
		std::uint32_t first = 0;
		if (i < kQueueParts)	// the parts of (COUNT_RAYS, bounce 0)
		{
			std::uint32_t total = 0;
			for (std::uint32_t j = 0; j < jobCount; j++) total += jobs[j].pixels * jobs[j].params.sampleCount;
			const std::uint32_t tiles = (total + kPartTile - 1u) / kPartTile, rows = tiles / kQueueParts;
			first = kPartTile * rows;
			for (std::uint32_t t = rows * kQueueParts; t < tiles; t++) first += partOfTile(t) == i ? kPartTile : 0u;
			if (tiles > 0u && partOfTile(tiles - 1u) == i) first -= kPartTile * tiles - total;
			if (i == 0)
			{
				w.counts[kCounterWords] = total;
				w.counts[kCounterWords + 1] = kPartTile * ((tiles + kQueueParts - 1u) / kQueueParts);
			}
		}
		w.counts[i * kCounterStride] = first;
	}

	// Adds a pass's traced rays (its queues' lengths) to the render's counters.
	static __global__ void	wf_count_rays(WaveBuffers w, unsigned long long* counters)
	{
		unsigned long long rays = 0, shadow = 0;
		for (std::uint32_t i = threadIdx.x; i < kMaxBounceSlots * kQueueParts; i += 64u)
		{
			rays += w.counts[i * kCounterStride];
			shadow += w.counts[(kMaxBounceSlots * kQueueParts + i) * kCounterStride];
		}
		for (int off = 32; off > 0; off >>= 1)
		{
			rays += __shfl_down(rays, off);
			shadow += __shfl_down(shadow, off);
		}
		if (threadIdx.x == 0)
		{
			counters[0] += rays;
			counters[1] += shadow;
		}
	}

	// log(max(u, 1e-12)) of DIM_VOLUME_DISTANCE for (pixel, sample) at bounce b.
	__device__ __forceinline__ float	pathVolumeLogU(const GpuParams& p, std::uint32_t x, std::uint32_t y, std::uint32_t sample, int b)
	{
		PixelSampler ps;
		ps.begin(p.renderSeed, x, y, sample, sampleStream(p, sample));
		ps.bounce = static_cast<std::uint32_t>(b);
		return volumeLogU(p, ps);
	}

	// Camera rays of every job of the pass in one launch (the pass's paths in job order, tile by
	// tile to the parts of queue 0).
	static __global__ __launch_bounds__(kWaveBlock) void	wf_raygen(const PassJob* jobs, std::uint32_t jobCount, WaveBuffers w)
	{
		const std::uint32_t total = w.pathCount(), partStride = w.partStride();
		for (std::uint32_t g = blockIdx.x * kWaveBlock + threadIdx.x; g < total; g += gridDim.x * kWaveBlock)
		{
			std::uint32_t lo = 0, hi = jobCount;	// the last job whose slice starts at or before g
			while (hi - lo > 1u)
			{
				const std::uint32_t mid = (lo + hi) >> 1;
				if (jobs[mid].pathBase <= g) lo = mid;
				else hi = mid;
			}
			const std::uint32_t job = lo;
			const PassJob& J = jobs[job];
			const GpuParams& p = J.params;
			const std::uint32_t pixels = J.pixels;
			// entry g is the job's id-th camera ray; the queue visits the image in
			// bands of 8 rows, column by column, so a wave's 64 rays cover an 8 x 8 block
			// (coherent first traversals). The path keeps its row-major id, which the later
			// stages and the accumulation decode.
			const std::uint32_t id = g - J.pathBase;
			std::uint32_t order;
			const std::uint32_t slot = divide(id, pixels, J.pixelsInverse, order);
			std::uint32_t pixel;
			if (J.pixelList)
			{
				pixel = J.pixelList[order];
			}
			else
			{
				std::uint32_t inRow;
				const std::uint32_t row = divide(order, p.width, J.widthInverse, inRow);
				const std::uint32_t band = row / 8u;
				const std::uint32_t bandRows = min(8u, p.height - band * 8u);
				const std::uint32_t within = order - band * 8u * p.width;
				const std::uint32_t column = bandRows == 8u ? within / 8u : within / bandRows;
				pixel = (band * 8u + within - column * bandRows) * p.width + column;
			}
			const std::uint32_t path = J.pathBase + slot * pixels + (J.pixelList ? order : pixel);
			std::uint32_t x;
			const std::uint32_t y = divide(pixel, p.width, J.widthInverse, x);
			PixelSampler ps;
			ps.begin(p.renderSeed, x, y, p.sampleBegin + slot, sampleStream(p, p.sampleBegin + slot));
			const Ray r = cameraRay(p, x, y, ps);
			const float logU = p.hasVolumes ? volumeLogU(p, ps) : 0.0f;
			const std::uint32_t tile = g / kPartTile;
			const std::uint32_t at = partOfTile(tile) * partStride + (tile / kQueueParts) * kPartTile + g % kPartTile;
			w.qOrigin[0][at] = make_float4(r.o.x, r.o.y, r.o.z, logU);
			w.qDir[0][at] = make_float4(r.d.x, r.d.y, r.d.z, __uint_as_float(kNoOrigin.hittable));
			w.qFrom[0][at] = kNoOrigin.tri;
			w.qPath[0][at] = w.queuedPath(job, path);
			// the path's throughput and radiance start as constants the first shade stage
			// supplies itself
		}
	}

	// Queue slots handed to the lanes of one wave, claimed from the queue's fetch counter in
	// chunks of `chunk` rays (one atomic per chunk; tunable 64..1024). All fields are
	// wave-uniform.
	constexpr std::uint32_t	kFetchChunk = 256;	// the most rays a wave claims per atomic

	struct	WaveFeed
	{
		std::uint32_t	next;
		std::uint32_t	end;
		bool	drained;
		std::uint32_t	first;	// the slots before this one were dealt without a claim

		__device__ __forceinline__ bool	any() const { return !drained || next < end; }

		// Gives every lane in `idle` (ballot mask) the next queue slot, in lane order; lanes
		// left without one (queue exhausted) get 0xffffffff.
		__device__ __forceinline__ std::uint32_t	hand(unsigned long long idle, std::uint32_t n, std::uint32_t* fetch, std::uint32_t chunk)
		{
			const std::uint32_t want = static_cast<std::uint32_t>(__popcll(idle));
			const std::uint32_t rank = static_cast<std::uint32_t>(__popcll(idle & ((1ull << laneId()) - 1ull)));
			const std::uint32_t avail = end - next;
			std::uint32_t slot;
			if (want <= avail)
			{
				slot = next + rank;
				next += want;
				return slot;
			}
			if (drained)	// what is left of the last claim
			{
				slot = rank < avail ? next + rank : 0xffffffffu;
				next = end;
				return slot;
			}
			std::uint32_t c = 0;
			if (laneId() == static_cast<std::uint32_t>(__ffsll(static_cast<long long>(idle)) - 1))
			{
				c = atomicAdd(fetch, chunk);
			}
			c = first + __builtin_amdgcn_readfirstlane(__shfl(c, __ffsll(static_cast<long long>(idle)) - 1));
			const std::uint32_t cEnd = c >= n ? c : min(c + chunk, n);
			if (rank < avail) slot = next + rank;
			else
			{
				const std::uint32_t k = c + (rank - avail);
				slot = k < cEnd ? k : 0xffffffffu;
			}
			if (c >= n)
			{
				next = end;
				drained = true;
			}
			else
			{
				next = min(c + (want - avail), cEnd);
				end = cEnd;
			}
			return slot;
		}
	};

	// counters: [0] closest rays, [1] shadow rays (wf_count_rays), [2]/[3] closest
	// nodes/primitives, [4]/[5] shadow nodes/primitives
	__device__ __forceinline__ void	flushVisits(unsigned long long* counters, int slot, VisitCounter visits)
	{
		for (int off = 32; off > 0; off >>= 1)
		{
			visits.nodes += __shfl_down(visits.nodes, off);
			visits.prims += __shfl_down(visits.prims, off);
		}
		if (laneId() == 0 && visits.nodes + visits.prims)
		{
			atomicAdd(counters + 2 + 2 * slot, static_cast<unsigned long long>(visits.nodes));
			atomicAdd(counters + 3 + 2 * slot, static_cast<unsigned long long>(visits.prims));
		}
	}

	// Persistent traversal over one ray queue with lane refill: a lane whose traversal has
	// ended takes the next ray of the queue once at least `refillAt` lanes of its wave are
	// idle (refillAt = 64: the wave claims 64 rays at a time and every lane traverses its
	// ray to the end before the next claim). Each turn of the loop runs the leaf code, if its
	// turn has come, then the node code, then the pop they share, each once per wave.
	// VALU-bound before the node test became a straight line (nodeStep): 1080p spheres extend
	// 27.7 -> 18.9 ms, shadow 5.8 -> 3.5; 720p hazy terrain 50.9 -> 25.6 and 53.7 -> 26.7.
	// Source supplies a queue part: load(slot, ray, tMax) and store(slot, state), `n` rays and the
	// claim counter `fetch`.
	template <bool AnyHit, bool Count, int Feat, int LdsDepth, typename Source>
	__device__ __forceinline__ void	traceQueue(const SceneView& s, const PassJob* jobs, Source& src, std::uint32_t n, std::uint32_t* fetch,
		std::uint32_t wave, std::uint32_t waves, int refillAt, std::uint32_t maxChunk, unsigned long long* counters, int counterSlot,
		std::uint32_t* stackMem)
	{
		const std::uint32_t gtid = blockIdx.x * kWaveBlock + threadIdx.x;
		SpillStack<LdsDepth, kWaveBlock> stack{stackMem + threadIdx.x, src.spill + gtid, gridDim.x * kWaveBlock, 0,
			kWaveStackCapacity};
		// Rays a wave claims per atomic on the part's counter: about an eighth of an even share
		// of the part, a multiple of 64 between 64 and maxChunk, so a long queue is claimed with
		// few atomics and a short one still spreads over the waves. Its first chunk a wave has
		// without a claim.
		const std::uint32_t share = ((n / (8u * waves)) + 63u) & ~63u;
		const std::uint32_t chunk = min(max(share, 64u), maxChunk);
		// Waves beyond what the part can feed leave. The waves that stay claim until it is
		// exhausted, so every ray is still traced.
		const std::uint64_t mine = static_cast<std::uint64_t>(wave) * chunk;
		if (mine >= n)
		{
			return;
		}
		const std::uint64_t dealt = static_cast<std::uint64_t>(waves) * chunk;
		const std::uint32_t begin = static_cast<std::uint32_t>(mine);
		WaveFeed feed{begin, min(begin + chunk, n), dealt >= n, static_cast<std::uint32_t>(min(dealt, static_cast<std::uint64_t>(n)))};
		VisitCounter visits{0u, 0u};
		TraceState st;
		std::uint32_t slot = 0xffffffffu;
		bool active = false;
		// the last job's root and unbounded list: a single-scene pass loads them once per lane
		std::uint32_t lastJob = 0xffffffffu, lastUnbounded = 0u;
		std::int32_t lastRoot = -1;
		while (true)
		{
			const unsigned long long idle = __ballot(!active);
			if (feed.any() && (__popcll(idle) >= refillAt || idle == ~0ull))
			{
				const std::uint32_t k = feed.hand(idle, n, fetch, chunk);
				if (!active && k != 0xffffffffu)
				{
					slot = k;
					Ray r;
					float tMax, logU;
					RayOrigin from;
					const std::uint32_t job = src.load(slot, r, tMax, logU, from);
					if (job != lastJob)
					{
						const GpuParams& jp = jobs[job].params;
						lastJob = job;
						lastRoot = jp.tlasRoot;
						lastUnbounded = unboundedOf(jp);
					}
					active = traceBegin(st, lastRoot, lastUnbounded, r, tMax, logU, from, stack);
					if (!active) src.store(slot, st);
				}
			}
			if (__ballot(active) == 0ull && !feed.any())
			{
				break;
			}
			const bool wantNode = active && (st.entry & kLeafBit) == 0u;
			const unsigned long long nodes = __ballot(wantNode);
			const bool leafTurn = nodes == 0ull || __popcll(__ballot(active) & ~nodes) >= kLeafBatch<Feat, AnyHit>;
			bool pop = false, ended = false;
			if (leafTurn && active && !wantNode)
			{
				const int step = leafStep<AnyHit, Count, Feat>(s, st, stack.sp, kTMinF, &visits);
				pop = step == STEP_POP;
				ended = step == STEP_END;
			}
			if (wantNode)
			{
				pop = !nodeStep<Count>(s, st, stack, &visits);
			}
			if (pop)
			{
				ended = popEntry<AnyHit, Feat>(s, st, kTMinF, stack);
			}
			if (ended)
			{
				src.store(slot, st);
				active = false;
			}
		}
		if (Count) flushVisits(counters, counterSlot, visits);
	}

	// Runs `trace(part, wave, waves)` for the queue parts of this block: wave `wave` of the
	// `waves` that share the part (a grid of fewer than kQueueParts blocks gives a block several).
	template <typename Trace>
	__device__ __forceinline__ void	forQueueParts(Trace&& trace)
	{
		const std::uint32_t groups = min(gridDim.x, kQueueParts), group = blockIdx.x % groups;
		const std::uint32_t wave = (blockIdx.x / groups) * (kWaveBlock / 64) + threadIdx.x / 64u;
		const std::uint32_t waves = ((gridDim.x - group + groups - 1u) / groups) * (kWaveBlock / 64);
		for (std::uint32_t part = group; part < kQueueParts; part += groups)
		{
			trace(part, uniform(wave), waves);
		}
	}

	struct	ExtendQueue
	{
		const WaveBuffers&	w;
		int	b;
		std::uint32_t*	spill;
		std::uint32_t	base;	// of the queue part
		// returns the ray's scene job
		__device__ __forceinline__ std::uint32_t	load(std::uint32_t slot, Ray& r, float& tMax, float& logU, RayOrigin& from) const
		{
			const std::uint32_t i = base + slot;
			const float4 o = w.qOrigin[b & 1][i], d = w.qDir[b & 1][i];
			r = makeRay(mk(o.x, o.y, o.z), mk(d.x, d.y, d.z));
			tMax = INFINITY;
			logU = o.w;
			from = RayOrigin{__float_as_uint(d.w), w.qFrom[b & 1][i]};
			return w.sceneOfPath(w.qPath[b & 1][i]);
		}
		__device__ __forceinline__ void	store(std::uint32_t slot, const TraceState& st) const
		{
			const std::uint32_t i = base + slot;
			w.qHit[i] = make_float4(st.found ? st.hit.t : -1.0f, st.hit.u, st.hit.v, __uint_as_float(st.hit.hittable));
			w.qTri[i] = st.hit.tri;
		}
	};

	struct	ShadowQueue
	{
		const WaveBuffers&	w;
		int	b;
		std::uint32_t*	spill;
		std::uint32_t	volumes;	// the batch has volumes: shadow rays carry a sample
		std::uint32_t	base;	// of the queue part
		std::uint32_t	target;	// connection slot of the ray being traced
		__device__ __forceinline__ std::uint32_t	load(std::uint32_t slot, Ray& r, float& tMax, float& logU, RayOrigin& from)
		{
			const std::uint32_t i = base + slot;
			const float4 o = w.sOrigin[i], d = w.sDir[i];
			r = makeRay(mk(o.x, o.y, o.z), mk(d.x, d.y, d.z));
			tMax = o.w;
			const std::uint32_t tag = __float_as_uint(d.w);
			target = w.slotOfTag(tag);
			logU = volumes ? w.sLogU[i] : 0.0f;
			const int2 f = w.sFrom[i];
			from = RayOrigin{static_cast<std::uint32_t>(f.x), f.y};
			return w.sceneOfTag(tag);
		}
		__device__ __forceinline__ void	store(std::uint32_t, const TraceState& st) const
		{
			w.visible[target] = st.found ? 0 : 1;
		}
	};

	// closest hit of every ray of queue b
	template <bool Count, int Feat, int LdsDepth>
	// The traversal kernels are asked for at least 4 waves per SIMD (at most 128 VGPRs), which they
	// keep to by themselves (86 and 82 VGPRs in triangle-only scenes, 109 and 103 with analytic
	// primitives): the request holds them to it. At 3 waves the terrain's extend took 41.4 ms
	// instead of 36.8, on a longer node test.
	static __global__ __launch_bounds__(kWaveBlock, 4) void	wf_extend(SceneView s, const PassJob* jobs, WaveBuffers w, int b,
		unsigned long long* counters, int refillAt, std::uint32_t chunk)
	{
		__shared__ std::uint32_t stackMem[LdsDepth * kWaveBlock];
		forQueueParts([&](std::uint32_t part, std::uint32_t wave, std::uint32_t waves) {
			ExtendQueue src{w, b, w.spill, uniform(part * w.partStride())};
			traceQueue<false, Count, Feat, LdsDepth>(s, jobs, src, uniform(*w.counter(COUNT_RAYS, b, part)), w.counter(CLAIM_EXTEND, b, part), wave, waves,
				refillAt, chunk, counters, 0, stackMem);
		});
	}

	// Waves per SIMD asked of the shade kernels, whose chains of dependent loads (queue, hit,
	// primitive, material, light tables) are latency-bound: what their registers allow with
	// next to no spills. 1080p spheres: shade 12.1 -> 8.8 ms (180 -> 16 bytes spilled at 4 waves);
	// 720p hazy terrain 35.8 -> 21.4 (1 -> 3 waves); 641 x 479 principled scene 2.7 -> 1.8.
	template <int Feat>
	constexpr int	kShadeWaves = Feat == 0 ? 4 : (Feat & kFeatRich) ? 2 : 3;

	// Batch: the pass holds several scenes. What a path appends to the queues is staged in LDS
	// until the block's ranges are known, and its connections' contributions are stored at
	// once: held in registers they would live across the whole body (in a batch across the
	// bodies of the wave's other scenes too) and spill.
	template <int Feat, bool Batch>
	static __global__ __launch_bounds__(kWaveBlock, kShadeWaves<Feat>) void	wf_shade(SceneView s, const PassJob* jobs, WaveBuffers w, int b,
		std::uint32_t volumes, float* __restrict__ sampleColors)
	{
		// this block's queue part (the grid is a multiple of the parts)
		const std::uint32_t part = blockIdx.x % kQueueParts;
		const std::uint32_t n = uniform(*w.counter(COUNT_RAYS, b, part)), partBase = uniform(part * w.partStride());
		const int q = b & 1;
		std::uint32_t* nextCount = w.counter(COUNT_RAYS, b + 1, part);
		std::uint32_t* shadowCount = w.counter(COUNT_SHADOW, b, part);
		// Queue appends: each wave counts its continuing paths and its shadow rays (light
		// connections, then environment ones) in LDS, and one thread claims the block's
		// ranges of the next queue and the shadow queue with one atomic each.
		constexpr int kWaves = kWaveBlock / 64;
		__shared__ std::uint32_t waveNext[kWaves], waveShadow[kWaves], blockNext, blockShadow;
		// staged per lane: the vertex, the next direction, its origin's identity, the light
		// connection's direction and distance, the environment's direction, the volume samples
		// of the next ray and of the shadow rays
		constexpr int kStageFrom = 6, kStageLight = 8, kStageEnv = 12, kStageLogU = 15, kStageFields = 17;
		__shared__ float stageMem[kStageFields * kWaveBlock];
		float* const stage = stageMem + threadIdx.x;
		auto put = [&](int field, float v) { stage[field * kWaveBlock] = v; };
		auto put3 = [&](int field, f3 v) {
			put(field, v.x);
			put(field + 1, v.y);
			put(field + 2, v.z);
		};
		auto get = [&](int field) { return stage[field * kWaveBlock]; };
		const int wave = static_cast<int>(threadIdx.x >> 6);
		// grid-stride loop with a block-uniform trip count so every lane reaches the ballots
		// and every wave the barriers
		const std::uint32_t stride = gridDim.x / kQueueParts * kWaveBlock;
		for (std::uint32_t blockBase = blockIdx.x / kQueueParts * kWaveBlock; blockBase < n; blockBase += stride)
		{
			const bool valid = blockBase + threadIdx.x < n;
			const std::uint32_t i = partBase + blockBase + threadIdx.x;
			bool cont = false, wantLight = false, wantEnv = false;
			const std::uint32_t qp = valid ? w.qPath[q][i] : 0u;
			const std::uint32_t job = Batch ? w.sceneOfPath(qp) : 0u;
			const std::uint32_t path = Batch ? w.pathOf(qp) : qp;
			auto shadePath = [&](const PassJob& J) {
				const GpuParams& p = J.params;
				std::uint32_t entry, px;
				const std::uint32_t slot = divide(path - J.pathBase, J.pixels, J.pixelsInverse, entry);
				const std::uint32_t py = divide(passPixel(J, entry), p.width, J.widthInverse, px);
				PixelSampler ps;
				ps.begin(p.renderSeed, px, py, p.sampleBegin + slot, sampleStream(p, p.sampleBegin + slot));
				ps.bounce = static_cast<std::uint32_t>(b);
				const float4 hv = w.qHit[i];
				const float4 o = w.qOrigin[q][i], d = w.qDir[q][i];
				const Ray ray = makeRay(mk(o.x, o.y, o.z), mk(d.x, d.y, d.z));
				// a camera path starts with throughput 1, no radiance, and counts as leaving a
				// specular vertex (the camera): those are not stored by ray generation
				const float4 t4 = b == 0 ? make_float4(1.0f, 1.0f, 1.0f, 0.0f) : w.throughput[path];
				const float4 r4 = b == 0 ? make_float4(0.0f, 0.0f, 0.0f, __uint_as_float(PF_PREV_SPECULAR)) : w.radiance[path];
				f3 thr = mk(t4.x, t4.y, t4.z), acc = mk(r4.x, r4.y, r4.z);
				const std::uint32_t before = __float_as_uint(r4.w);
				acc = addConnections(w, path, before, acc);
				const bool prevSpecular = before & PF_PREV_SPECULAR;
				const bool prevInfinite = before & PF_PREV_INFINITE;
				const float prevPdf = t4.w;
				std::uint32_t flags = 0u;	// of this vertex
				float nextPdf = 0.0f;
				if (hv.x < 0.0f)
				{
					float wgt = 1.0f;
					if (b > 0 && !prevSpecular && prevInfinite)
					{
						wgt = powerHeuristic(prevPdf, infiniteLightPdf(s, p, ray.d));
					}
					f3 c = thr * missRadiance<Feat>(s, p, ray, ps, wgt);
					if (b > 0 && hasConstantBackgroundLight(p)) c = clampConstantBackground(p, c);
					acc = acc + clampRay(c);
					if (b == 0 && J.features)
					{
						primaryFeatures(J.features + static_cast<size_t>(kNforFeatures) * path, p, px, py, false, 0.0f, mk(0, 0, 0),
							missRadiance<Feat>(s, p, ray, ps, 1.0f), 0u);
					}
				}
				else
				{
					HitInfo h;
					h.t = hv.x;
					h.u = hv.y;
					h.v = hv.z;
					h.hittable = __float_as_uint(hv.w);
					h.tri = w.qTri[i];
					Surface sf = surfaceAt<Feat>(s, ray, h);
					RayOrigin from = originOf(s, h);
					const GpuMaterial& m = s.materials[sf.material];
					if (b == 0 && J.features)
					{
						primaryFeatures(J.features + static_cast<size_t>(kNforFeatures) * path, p, px, py, true, h.t, sf.normal,
							ld3(m.color), m.kind);
					}
					bool alive = true;
					if constexpr ((Feat & kFeatRich) != 0)
					{
						if (b == 0 && p.sky == GPU_SKY_ATMOSPHERE)
						{
							atmospherePrimary(p.atmosphere, ray.o, ray.d, h.t, acc, thr);
							alive = !terminated(thr);
						}
					}
					const f3 emitted = m.kind == GPU_MAT_EMISSIVE ? ld3(m.color) : mk(0, 0, 0);
					Scatter sc;
					if (!alive)
					{
					}
					else if (!scatter<Feat>(m, sf, ray.d, ps, sc))
					{
						float lp = 0.0f;
						if (!prevSpecular && p.lightCount > 0)
						{
							const float4 po = w.prevOrigin[path];
							lp = lightsPdf<Feat>(s, p, mk(po.x, po.y, po.z), ray.d);
						}
						const float wgt = prevSpecular ? 1.0f : powerHeuristic(prevPdf, lp);
						acc = acc + clampRay((thr * emitted) * wgt);
					}
					else
					{
						if constexpr ((Feat & kFeatSubsurface) != 0)
						{
							if (sc.subsurfaceExit)
							{
								LocalStack probeStack;
								probeStack.reset();
								std::uint32_t probes = 0;
								relocateSubsurface<Feat>(s, p, m, h, sf, sc, ps, probeStack, o.w, probes);
								from = originOf(s, h);
							}
						}
						f3 att = sc.attenuation;
						if (!sf.frontFace && sc.absorbing)
						{
							const float dm = h.t * p.metersPerUnit;
							if (isfinite(dm) && dm > 0.0f)
							{
								att = att * mk(expf(-m.absorption[0] * dm), expf(-m.absorption[1] * dm), expf(-m.absorption[2] * dm));
							}
						}
						put3(0, sf.position);
						put(kStageFrom, __uint_as_float(from.hittable));
						put(kStageFrom + 1, __int_as_float(from.tri));
						put(kStageLogU + 1, o.w);
						if (sc.specular)
						{
							if (leavesOpaque(sf, m, sc.direction))
							{
								thr = clampRay(thr * att);
								if (!terminated(thr) && russianRoulette(thr, b, ps))
								{
									put3(3, sc.direction);
									flags = PF_PREV_SPECULAR;
									cont = b < p.maxBounces;
								}
							}
						}
						else
						{
							acc = acc + thr * emitted;
							if (!terminated(thr * att))
							{
								// a connection's clampRay is applied when it is added
								auto connect = [&](std::uint32_t slotOf, const Connection& c, bool test) {
									const f3 v = thr * c.contribution;
									w.connection[2 * path + slotOf] = make_float4(v.x, v.y, v.z, 0.0f);
									w.visible[2 * path + slotOf] = test ? 0 : 1;
								};
								if (p.lightCount > 0)
								{
									const Connection c = connectLight<Feat>(s, p, sf, m, sc, b, ps);
									if (c.active)
									{
										wantLight = c.tMax > 0.0f;
										flags |= PF_CONN_LIGHT;
										connect(0u, c, wantLight);
										put3(kStageLight, c.direction);
										put(kStageLight + 3, c.tMax);
									}
								}
								if (hasEnvLight(p) || hasConstantBackgroundLight(p))
								{
									const Connection c = connectInfinite<Feat>(s, p, sf, m, sc, b, ps);
									if (c.active)
									{
										wantEnv = true;
										flags |= PF_CONN_ENV;
										connect(1u, c, true);
										put3(kStageEnv, c.direction);
									}
								}
								const f3 dir = scatterDirection<Feat>(sf, sc, ps);
								if (leavesOpaque(sf, m, dir))
								{
									const float pdf = scatterPdf<Feat>(m, sf, sc, dir);
									if (pdf > 0.0f && isfinite(pdf))
									{
										thr = clampRay(thr * att);
										if (!terminated(thr) && russianRoulette(thr, b, ps))
										{
											put3(3, dir);
											flags |= samplesVisibleInfinite(p, sc) ? PF_PREV_INFINITE : 0u;
											nextPdf = pdf;
											cont = b < p.maxBounces;
											// read back only for an emitter's MIS weight
											if (cont && p.lightCount > 0)
											{
												w.prevOrigin[path] = make_float4(sf.position.x, sf.position.y, sf.position.z, 0.0f);
											}
										}
									}
								}
							}
						}
					}
				}
				if (cont)
				{
					w.throughput[path] = make_float4(thr.x, thr.y, thr.z, nextPdf);
					if (p.hasVolumes) put(kStageLogU, pathVolumeLogU(p, px, py, p.sampleBegin + slot, b + 1));
				}
				const bool pending = (flags & (PF_CONN_LIGHT | PF_CONN_ENV)) != 0u;
				if (cont || pending) w.radiance[path] = make_float4(acc.x, acc.y, acc.z, __uint_as_float(flags));
				if (!cont)
				{
					const f3 c = cleanColor(acc);
					float* out = sampleColors + static_cast<size_t>(path) * 3;
					out[0] = pending ? __uint_as_float(kPendingColor) : c.x;
					out[1] = c.y;
					out[2] = c.z;
				}
			};
			if constexpr (Batch)
			{
				// one scene per iteration, so the scene's parameters are wave-uniform (scalar loads)
				unsigned long long left = __ballot(valid);
				while (left)
				{
					const int leader = __ffsll(static_cast<long long>(left)) - 1;
					const std::uint32_t cur = __builtin_amdgcn_readfirstlane(__shfl(job, leader));
					const bool mine = valid && job == cur;
					if (mine) shadePath(jobs[cur]);
					left &= ~__ballot(mine);
				}
			}
			else if (valid)
			{
				shadePath(jobs[0]);
			}
			const unsigned long long mNext = __ballot(cont), mLight = __ballot(wantLight), mEnv = __ballot(wantEnv);
			const std::uint32_t nLight = static_cast<std::uint32_t>(__popcll(mLight));
			if (laneId() == 0)
			{
				waveNext[wave] = static_cast<std::uint32_t>(__popcll(mNext));
				waveShadow[wave] = nLight + static_cast<std::uint32_t>(__popcll(mEnv));
			}
			__syncthreads();
			if (threadIdx.x == 0)
			{
				std::uint32_t tNext = 0, tShadow = 0;
				for (int k = 0; k < kWaves; k++)
				{
					tNext += waveNext[k];
					tShadow += waveShadow[k];
				}
				blockNext = tNext > 0 ? atomicAdd(nextCount, tNext) : 0u;
				blockShadow = tShadow > 0 ? atomicAdd(shadowCount, tShadow) : 0u;
			}
			__syncthreads();
			std::uint32_t nextBase = partBase + blockNext, shadowBase = 2u * partBase + blockShadow;
			for (int k = 0; k < wave; k++)
			{
				nextBase += waveNext[k];
				shadowBase += waveShadow[k];
			}
			const unsigned long long below = (1ull << laneId()) - 1ull;
			if (cont || wantLight || wantEnv)
			{
				const float x = get(0), y = get(1), z = get(2);
				const float fromHittable = get(kStageFrom);
				const std::int32_t fromTri = __float_as_int(get(kStageFrom + 1));
				if (cont)
				{
					const std::uint32_t pos = nextBase + static_cast<std::uint32_t>(__popcll(mNext & below));
					const int nq = (b + 1) & 1;
					w.qOrigin[nq][pos] = make_float4(x, y, z, volumes ? get(kStageLogU) : 0.0f);
					w.qDir[nq][pos] = make_float4(get(3), get(4), get(5), fromHittable);
					w.qFrom[nq][pos] = fromTri;
					w.qPath[nq][pos] = qp;
				}
				auto appendShadow = [&](std::uint32_t at, int field, float tMax, std::uint32_t slotOf) {
					w.sOrigin[at] = make_float4(x, y, z, tMax);
					w.sDir[at] = make_float4(get(field), get(field + 1), get(field + 2), __uint_as_float(w.shadowTag(job, 2u * path + slotOf)));
					w.sFrom[at] = make_int2(__float_as_int(fromHittable), fromTri);
					if (volumes) w.sLogU[at] = get(kStageLogU + 1);
				};
				if (wantLight)
				{
					appendShadow(shadowBase + static_cast<std::uint32_t>(__popcll(mLight & below)), kStageLight, get(kStageLight + 3), 0u);
				}
				if (wantEnv)
				{
					appendShadow(shadowBase + nLight + static_cast<std::uint32_t>(__popcll(mEnv & below)), kStageEnv, INFINITY, 1u);
				}
			}
			// the next iteration rewrites the per-wave counts
			__syncthreads();
		}
	}

	// any-hit test of the shadow rays appended in bounce b
	template <bool Count, int Feat, int LdsDepth>
	static __global__ __launch_bounds__(kWaveBlock, 4) void	wf_shadow(SceneView s, const PassJob* jobs, WaveBuffers w, int b,
		unsigned long long* counters, int refillAt, std::uint32_t chunk, std::uint32_t volumes)
	{
		__shared__ std::uint32_t stackMem[LdsDepth * kWaveBlock];
		forQueueParts([&](std::uint32_t part, std::uint32_t wave, std::uint32_t waves) {
			ShadowQueue src{w, b, w.spill, volumes, uniform(2u * part * w.partStride()), 0u};
			traceQueue<true, Count, Feat, LdsDepth>(s, jobs, src, uniform(*w.counter(COUNT_SHADOW, b, part)), w.counter(CLAIM_SHADOW, b, part), wave,
				waves, refillAt, chunk, counters, 1, stackMem);
		});
	}

	// Adds a pass's sample colours of one scene into its FP64 pixel sums, in sample order
	// (the per-pixel sum of _threadRender, Threads.cpp:551-583), and in adaptive rounds into
	// the pixel's AdaptiveAccumulator (Threads.cpp:571-576).
	static __global__ void	wf_accumulate(WaveBuffers w, const float* __restrict__ colors, const PassJob* jobs, std::uint32_t job)
	{
		const PassJob& J = jobs[job];
		const std::uint32_t count = J.params.sampleCount;
		if (J.denoise)
		{
			// denoising: half-buffer and feature statistics (Threads.cpp:585-627)
			for (std::uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < J.pixels; i += gridDim.x * blockDim.x)
			{
				const size_t px = passPixel(J, i);
				double a[kDenoiseStats];
				for (int j = 0; j < kDenoiseStats; j++) a[j] = J.denoise[kDenoiseStats * px + j];
				double m[kAdaptiveMoments];
				if (J.moments)
				{
					for (int k = 0; k < kAdaptiveMoments; k++) m[k] = J.moments[kAdaptiveMoments * px + k];
				}
				for (std::uint32_t k = 0; k < count; k++)
				{
					const size_t g = static_cast<size_t>(J.pathBase) + static_cast<size_t>(k) * J.pixels + i;
					float c[3];
					pathColor(w, colors, g, c);
					denoiseAddSample(a, c, J.features + kNforFeatures * g, ((J.params.sampleBegin + k) & 1u) != 0u);
					if (J.moments) adaptiveAdd(m, c[0], c[1], c[2]);
				}
				for (int j = 0; j < kDenoiseStats; j++) J.denoise[kDenoiseStats * px + j] = a[j];
				if (J.moments)
				{
					for (int k = 0; k < kAdaptiveMoments; k++) J.moments[kAdaptiveMoments * px + k] = m[k];
				}
			}
			return;
		}
		for (std::uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < J.pixels; i += gridDim.x * blockDim.x)
		{
			const size_t px = passPixel(J, i);
			double r = J.sums[3 * px], g = J.sums[3 * px + 1], b = J.sums[3 * px + 2];
			double m[kAdaptiveMoments];
			if (J.moments)
			{
				for (int k = 0; k < kAdaptiveMoments; k++) m[k] = J.moments[kAdaptiveMoments * px + k];
			}
			for (std::uint32_t k = 0; k < count; k++)
			{
				float c[3];
				pathColor(w, colors, static_cast<size_t>(J.pathBase) + static_cast<size_t>(k) * J.pixels + i, c);
				const double cr = c[0], cg = c[1], cb = c[2];
				r += cr;
				g += cg;
				b += cb;
				if (J.moments) adaptiveAdd(m, cr, cg, cb);
			}
			J.sums[3 * px] = r;
			J.sums[3 * px + 1] = g;
			J.sums[3 * px + 2] = b;
			if (J.moments)
			{
				for (int k = 0; k < kAdaptiveMoments; k++) J.moments[kAdaptiveMoments * px + k] = m[k];
			}
		}
	}

	// Launch shape of the traversal stages: persistent blocks per launch and the number of
	// idle lanes at which a wave takes new rays (1..64).
	// Launch shape of the traversal kernels; 0 = default. None of it changes results: every
	// ray is traversed in the same order whichever lane, chunk or stack level holds it.
	struct	WaveTuning
	{
		unsigned	grid = 0;			// persistent blocks per traversal launch
		int	extendRefill = 0;		// idle lanes at which a wave takes new closest-hit rays
		int	shadowRefill = 0;		// idle lanes at which a wave takes new shadow rays
		unsigned	chunk = 0;			// most rays a wave claims per queue atomic
		int	ldsStack = 0;			// LDS stack entries per lane (the rest spill to HBM)

		// `features`: the scene's kFeat* classes
		WaveTuning	resolved(int features) const
		{
			WaveTuning t = *this;
			if (t.grid == 0) t.grid = kDefaultGrid;
			const int refill = (features & kFeatAnalytic) ? kRefillAnalytic : kRefillTriangles;
			if (t.extendRefill == 0) t.extendRefill = refill;
			if (t.shadowRefill == 0) t.shadowRefill = refill;
			if (t.chunk == 0) t.chunk = kFetchChunk;
			if (t.ldsStack == 0) t.ldsStack = kWaveLdsStack;
			if (t.grid > kWaveGrid || t.extendRefill < 1 || t.extendRefill > 64 || t.shadowRefill < 1 || t.shadowRefill > 64
				|| t.chunk < 64 || t.chunk > 1024 || (t.ldsStack != 8 && t.ldsStack != 16 && t.ldsStack != 24))
			{
				throw std::invalid_argument("wavefront tuning out of range: grid 1.." + std::to_string(kWaveGrid)
					+ ", refill 1..64, chunk 64..1024, LDS stack 8, 16 or 24");
			}
			return t;
		}
		bool	operator==(const WaveTuning& o) const
		{
			return grid == o.grid && extendRefill == o.extendRefill && shadowRefill == o.shadowRefill && chunk == o.chunk
				&& ldsStack == o.ldsStack;
		}
	};

	struct	StageTimes
	{
		double	extendMs = 0.0, shadeMs = 0.0, shadowMs = 0.0;
		std::uint32_t	extendLaunches = 0;
		std::uint32_t	passes = 0;
		std::uint32_t	graphReplays = 0;
	};

	// One scene of a render call: its parameters (sampleBegin / sampleCount: the whole
	// range of this call) and its FP64 pixel sums.
	struct	BatchJob
	{
		GpuParams	params;
		double*	sums;
		const std::uint32_t*	pixelList = nullptr;	// adaptive round: the active pixels
		std::uint32_t	listCount = 0;				// ... and how many
		double*	moments = nullptr;				// adaptive round: per-pixel accumulators
		double*	denoise = nullptr;				// denoising: per-pixel statistics (sums unused)
	};

	inline std::uint32_t	jobPixels(const BatchJob& j)
	{
		return j.pixelList ? j.listCount : j.params.width * j.params.height;
	}

	// Device state of one context (grown on demand, kept between renders), and the
	// captured pass graph with what it was captured for.
	struct	WavefrontState
	{
		void*	mem = nullptr;
		size_t	bytes = 0;
		WaveBuffers	buf{};
		float*	colors = nullptr;		// [global path][3]
		float*	features = nullptr;		// denoising: [global path][kNforFeatures], on demand
		std::uint32_t	featureCapacity = 0;
		PassJob*	jobs = nullptr;		// the current pass's table
		PassJob*	plans = nullptr;	// every pass's table of a render
		size_t	planCapacity = 0;
		hipGraphExec_t	graph = nullptr;
		std::vector<unsigned char>	graphKey;

		void	dropGraph()
		{
			if (graph) (void)hipGraphExecDestroy(graph);
			graph = nullptr;
			graphKey.clear();
		}

		void	release()
		{
			dropGraph();
			if (mem) (void)hipFree(mem);
			if (plans) (void)hipFree(plans);
			if (features) (void)hipFree(features);
			features = nullptr;
			featureCapacity = 0;
			mem = nullptr;
			plans = nullptr;
			planCapacity = 0;
			bytes = 0;
		}

		// Carves the state arrays for `capacity` paths out of `base` (each 256-byte aligned)
		// and returns the bytes used; with base == nullptr it only measures.
		size_t	carve(char* base, std::uint32_t capacity)
		{
			const size_t n = capacity;
			const size_t nq = n + kPartTile * (kQueueParts + 1);	// the parts' strides are whole tiles
			const size_t spillBytes = static_cast<size_t>(kWaveStackCapacity - kWaveLdsStackMin) * kWaveGrid * kWaveBlock * 4;
			size_t off = 0;
			auto take = [&](size_t b) { char* r = base ? base + off : nullptr; off += (b + 255) & ~size_t(255); return r; };
			WaveBuffers nb;
			std::memset(&nb, 0, sizeof(nb));	// padding too: graph keys compare the raw bytes
			for (int k = 0; k < 2; k++)
			{
				nb.qOrigin[k] = reinterpret_cast<float4*>(take(16 * nq));
				nb.qDir[k] = reinterpret_cast<float4*>(take(16 * nq));
				nb.qFrom[k] = reinterpret_cast<std::int32_t*>(take(4 * nq));
				nb.qPath[k] = reinterpret_cast<std::uint32_t*>(take(4 * nq));
			}
			nb.qHit = reinterpret_cast<float4*>(take(16 * nq));
			nb.qTri = reinterpret_cast<std::int32_t*>(take(4 * nq));
			nb.throughput = reinterpret_cast<float4*>(take(16 * n));
			nb.radiance = reinterpret_cast<float4*>(take(16 * n));
			nb.prevOrigin = reinterpret_cast<float4*>(take(16 * n));
			nb.connection = reinterpret_cast<float4*>(take(32 * n));
			nb.visible = reinterpret_cast<std::uint8_t*>(take(2 * n));
			nb.sOrigin = reinterpret_cast<float4*>(take(32 * nq));
			nb.sDir = reinterpret_cast<float4*>(take(32 * nq));
			nb.sLogU = reinterpret_cast<float*>(take(8 * nq));
			nb.sFrom = reinterpret_cast<int2*>(take(16 * nq));
			float* nc = reinterpret_cast<float*>(take(12 * n));
			nb.counts = reinterpret_cast<std::uint32_t*>(take((kCounterWords + 2) * 4));
			PassJob* nj = reinterpret_cast<PassJob*>(take(sizeof(PassJob) * kMaxBatchScenes));
			nb.spill = reinterpret_cast<std::uint32_t*>(take(spillBytes));
			nb.capacity = capacity;
			if (base)
			{
				buf = nb;
				colors = nc;
				jobs = nj;
			}
			return off;
		}

		// The layout is fixed between reallocations (captured graphs hold its pointers):
		// a smaller request keeps the larger layout.
		void	ensure(std::uint32_t capacity)
		{
			if (mem && capacity <= buf.capacity)
			{
				return;
			}
			const size_t need = carve(nullptr, capacity);
			if (need > bytes)
			{
				dropGraph();
				if (mem) (void)hipFree(mem);
				mem = nullptr;
				bytes = 0;
				if (hipMalloc(&mem, need) != hipSuccess)
				{
					mem = nullptr;
					throw std::runtime_error("wavefront state allocation failed");
				}
				bytes = need;
			}
			carve(static_cast<char*>(mem), capacity);
		}

		// The per-path feature buffer of denoising passes (not part of the captured layout:
		// passes find it through their job table).
		void	ensureFeatures(std::uint32_t capacity)
		{
			if (features && capacity <= featureCapacity) return;
			if (features) (void)hipFree(features);
			features = nullptr;
			featureCapacity = 0;
			if (hipMalloc(reinterpret_cast<void**>(&features), static_cast<size_t>(capacity) * kNforFeatures * sizeof(float)) != hipSuccess)
			{
				features = nullptr;
				throw std::runtime_error("wavefront feature buffer allocation failed");
			}
			featureCapacity = capacity;
		}

		void	ensurePlans(size_t entries)
		{
			if (entries <= planCapacity) return;
			if (plans) (void)hipFree(plans);
			plans = nullptr;
			planCapacity = 0;
			if (hipMalloc(reinterpret_cast<void**>(&plans), entries * sizeof(PassJob)) != hipSuccess)
			{
				plans = nullptr;
				throw std::runtime_error("wavefront pass-table allocation failed");
			}
			planCapacity = entries;
		}
	};

	inline void	checkHip(hipError_t e, const char* what)
	{
		if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
	}

	// Calls f with the scene's feature class as a compile-time constant.
	template <typename F>
	inline void	withFeatures(int features, F&& f)
	{
		switch (featureClass(features))
		{
			case 0: f.template operator()<0>(); break;
			case kFeatAnalytic: f.template operator()<kFeatAnalytic>(); break;
			case kFeatMedia: f.template operator()<kFeatMedia>(); break;
			case kFeatRich: f.template operator()<kFeatRich>(); break;
			case kFeatAll: f.template operator()<kFeatAll>(); break;
			default: f.template operator()<kFeatEvery>(); break;
		}
	}

	// Enqueues the launches of one pass (the table is already in st.jobs).
	template <int Feat>
	void	enqueuePassF(WavefrontState& st, const SceneView& s, std::uint32_t jobCount, int maxBounces, bool volumes,
		unsigned long long* counters, hipStream_t stream, bool count, WaveTuning tune, std::vector<hipEvent_t>* marks)
	{
		const WaveBuffers& w = st.buf;
		auto mark = [&]() {
			if (!marks) return;
			hipEvent_t e;
			checkHip(hipEventCreate(&e), "hipEventCreate");
			marks->push_back(e);
			checkHip(hipEventRecord(e, stream), "hipEventRecord");
		};
		const std::uint32_t vol = volumes ? 1u : 0u;
		constexpr int T = Feat & kFeatAll;	// extend and shadow differ only by primitive / material class
		wf_zero_counts<<<kCounterWords / kCounterStride / 256, 256, 0, stream>>>(w, st.jobs, jobCount);
		wf_raygen<<<kWaveGrid, kWaveBlock, 0, stream>>>(st.jobs, jobCount, w);
		for (int b = 0; b <= maxBounces; b++)
		{
			mark();
			const unsigned ch = tune.chunk;
			if (count) wf_extend<true, T, kWaveLdsStack><<<tune.grid, kWaveBlock, 0, stream>>>(s, st.jobs, w, b, counters, tune.extendRefill, ch);
			else if (tune.ldsStack == 8) wf_extend<false, T, 8><<<tune.grid, kWaveBlock, 0, stream>>>(s, st.jobs, w, b, counters, tune.extendRefill, ch);
			else if (tune.ldsStack == 24) wf_extend<false, T, 24><<<tune.grid, kWaveBlock, 0, stream>>>(s, st.jobs, w, b, counters, tune.extendRefill, ch);
			else wf_extend<false, T, 16><<<tune.grid, kWaveBlock, 0, stream>>>(s, st.jobs, w, b, counters, tune.extendRefill, ch);
			mark();
			if (jobCount > 1u) wf_shade<Feat, true><<<kWaveGrid, kWaveBlock, 0, stream>>>(s, st.jobs, w, b, vol, st.colors);
			else wf_shade<Feat, false><<<kWaveGrid, kWaveBlock, 0, stream>>>(s, st.jobs, w, b, vol, st.colors);
			mark();
			if (count) wf_shadow<true, T, kWaveLdsStack><<<tune.grid, kWaveBlock, 0, stream>>>(s, st.jobs, w, b, counters, tune.shadowRefill, ch, vol);
			else if (tune.ldsStack == 8) wf_shadow<false, T, 8><<<tune.grid, kWaveBlock, 0, stream>>>(s, st.jobs, w, b, counters, tune.shadowRefill, ch, vol);
			else if (tune.ldsStack == 24) wf_shadow<false, T, 24><<<tune.grid, kWaveBlock, 0, stream>>>(s, st.jobs, w, b, counters, tune.shadowRefill, ch, vol);
			else wf_shadow<false, T, 16><<<tune.grid, kWaveBlock, 0, stream>>>(s, st.jobs, w, b, counters, tune.shadowRefill, ch, vol);
			mark();
		}
		wf_count_rays<<<1, 64, 0, stream>>>(w, counters);
		for (std::uint32_t j = 0; j < jobCount; j++)
		{
			wf_accumulate<<<1024, 256, 0, stream>>>(w, st.colors, st.jobs, j);
		}
	}

#ifndef LUZ_FEATURES
	// enqueuePassF is instantiated per scene feature class in features.hip
	#define LUZ_PASS(F) extern template void enqueuePassF<F>(WavefrontState&, const SceneView&, std::uint32_t, int, bool, \
		unsigned long long*, hipStream_t, bool, WaveTuning, std::vector<hipEvent_t>*);
	LUZ_PASS(0)
	LUZ_PASS(kFeatAnalytic)
	LUZ_PASS(kFeatMedia)
	LUZ_PASS(kFeatRich)
	LUZ_PASS(kFeatAll)
	LUZ_PASS(kFeatEvery)
	#undef LUZ_PASS

	inline void	enqueuePass(int features, WavefrontState& st, const SceneView& s, std::uint32_t jobCount, int maxBounces, bool volumes,
		unsigned long long* counters, hipStream_t stream, bool count, WaveTuning tune, std::vector<hipEvent_t>* marks)
	{
		withFeatures(features, [&]<int F>() { enqueuePassF<F>(st, s, jobCount, maxBounces, volumes, counters, stream, count, tune, marks); });
	}

	// Renders every job's sample range into its sums: passes of at most kMaxPassPaths paths
	// over all scenes at once. Without stage timing or visit counting, one pass is captured
	// as a hipGraph (its varying inputs are all in device memory) and replayed for every pass
	// and every later render with the same shape.
	inline void	renderWavefront(WavefrontState& st, const SceneView& s, int features, const std::vector<BatchJob>& jobs,
		unsigned long long* counters, hipStream_t stream, bool count, StageTimes* times, WaveTuning tune)
	{
		tune = tune.resolved(features);
		if (jobs.empty() || jobs.size() > kMaxBatchScenes)
		{
			throw std::invalid_argument("wavefront: 1.." + std::to_string(kMaxBatchScenes) + " scenes per launch");
		}
		int maxBounces = 0;
		bool volumes = false;
		std::uint64_t total = 0;
		for (const BatchJob& j : jobs)
		{
			if (j.params.maxBounces + 2 > kMaxBounceSlots)
			{
				throw std::runtime_error("Unsupported: more than 62 bounces in the wavefront integrator");
			}
			const std::uint64_t pixels = j.pixelList ? j.listCount : static_cast<std::uint64_t>(j.params.width) * j.params.height;
			if (pixels == 0 || pixels > std::min<std::uint64_t>(kMaxPassPaths, 1ull << pathBitsFor(static_cast<std::uint32_t>(jobs.size()))))
			{
				throw std::runtime_error("Unsupported: image of more pixels than a wavefront pass holds (2^27, fewer in large batches)");
			}
			maxBounces = std::max(maxBounces, j.params.maxBounces);
			volumes = volumes || j.params.hasVolumes;
			total += pixels * j.params.sampleCount;
		}
		const std::uint32_t n = static_cast<std::uint32_t>(jobs.size());
		const std::uint32_t pathBits = pathBitsFor(n);
		const std::uint32_t capacity = static_cast<std::uint32_t>(std::min<std::uint64_t>(std::min<std::uint64_t>(kMaxPassPaths, 1ull << pathBits),
			std::max<std::uint64_t>(total, 1)));
		// pass plan: each pass gives every scene with samples left as many as the budget holds
		std::vector<PassJob> plan;
		std::vector<std::uint32_t> done(n, 0);
		for (;;)
		{
			bool any = false;
			for (std::uint32_t j = 0; j < n; j++) any = any || done[j] < jobs[j].params.sampleCount;
			if (!any) break;
			std::uint32_t budget = capacity, base = 0;
			for (std::uint32_t j = 0; j < n; j++)
			{
				const GpuParams& p = jobs[j].params;
				const std::uint32_t pixels = jobPixels(jobs[j]);
				const std::uint32_t c = std::min(p.sampleCount - done[j], budget / pixels);
				PassJob pj{};
				pj.params = p;
				pj.params.sampleBegin = p.sampleBegin + done[j];
				pj.params.sampleCount = c;
				pj.pathBase = base;
				pj.pixels = pixels;
				pj.pixelsInverse = inverseOf(pixels);
				pj.widthInverse = inverseOf(p.width);
				pj.sums = jobs[j].sums;
				pj.pixelList = jobs[j].pixelList;
				pj.moments = jobs[j].moments;
				pj.denoise = jobs[j].denoise;
				plan.push_back(pj);
				done[j] += c;
				base += pixels * c;
				budget -= pixels * c;
			}
		}
		const std::uint32_t passes = static_cast<std::uint32_t>(plan.size() / n);
		st.ensure(capacity);
		st.buf.pathBits = pathBits;
		bool denoising = false;
		for (const BatchJob& j : jobs) denoising = denoising || j.denoise != nullptr;
		if (denoising)
		{
			st.ensureFeatures(st.buf.capacity);
			for (PassJob& pj : plan) pj.features = pj.denoise ? st.features : nullptr;
		}
		st.ensurePlans(plan.size());
		// the host table dies with this call: copy it before returning (ordered on the stream)
		checkHip(hipMemcpyAsync(st.plans, plan.data(), plan.size() * sizeof(PassJob), hipMemcpyHostToDevice, stream), "pass tables");
		checkHip(hipStreamSynchronize(stream), "pass tables");
		const bool useGraph = !count && !times;
		if (useGraph)
		{
			// what the captured launches depend on besides device memory
			std::vector<unsigned char> key(sizeof(SceneView) + sizeof(WaveTuning) + 4 * sizeof(std::uint32_t) + sizeof(void*) * 2);
			unsigned char* k = key.data();
			std::memcpy(k, &s, sizeof(SceneView)); k += sizeof(SceneView);
			std::memcpy(k, &tune, sizeof(WaveTuning)); k += sizeof(WaveTuning);
			const std::uint32_t shape[4] = {n, static_cast<std::uint32_t>(maxBounces), volumes ? 1u : 0u,
				static_cast<std::uint32_t>(features)};
			std::memcpy(k, shape, sizeof(shape)); k += sizeof(shape);
			void* ptrs[2] = {st.mem, counters};
			std::memcpy(k, ptrs, sizeof(ptrs));
			// the buffer layout the launches were captured with
			const unsigned char* lb = reinterpret_cast<const unsigned char*>(&st.buf);
			key.insert(key.end(), lb, lb + sizeof(WaveBuffers));
			const void* more[2] = {st.jobs, st.colors};
			const unsigned char* mb = reinterpret_cast<const unsigned char*>(more);
			key.insert(key.end(), mb, mb + sizeof(more));
			if (!st.graph || st.graphKey != key)
			{
				st.dropGraph();
				hipGraph_t g = nullptr;
				checkHip(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal), "hipStreamBeginCapture");
				enqueuePass(features, st, s, n, maxBounces, volumes, counters, stream, false, tune, nullptr);
				checkHip(hipStreamEndCapture(stream, &g), "hipStreamEndCapture");
				const hipError_t e = hipGraphInstantiate(&st.graph, g, nullptr, nullptr, 0);
				(void)hipGraphDestroy(g);
				checkHip(e, "hipGraphInstantiate");
				st.graphKey = key;
			}
		}
		// stage-timing events, destroyed on every exit (an error thrown mid-pass included)
		struct Marks
		{
			std::vector<hipEvent_t>	v;
			~Marks() { for (hipEvent_t e : v) (void)hipEventDestroy(e); }
		} held;
		std::vector<hipEvent_t>& marks = held.v;
		for (std::uint32_t k = 0; k < passes; k++)
		{
			checkHip(hipMemcpyAsync(st.jobs, st.plans + static_cast<size_t>(k) * n, n * sizeof(PassJob), hipMemcpyDeviceToDevice,
				stream), "pass table");
			if (useGraph)
			{
				checkHip(hipGraphLaunch(st.graph, stream), "hipGraphLaunch");
				if (times) times->graphReplays++;
			}
			else
			{
				enqueuePass(features, st, s, n, maxBounces, volumes, counters, stream, count, tune, times ? &marks : nullptr);
			}
		}
		if (times)
		{
			times->passes += passes;
			checkHip(hipStreamSynchronize(stream), "wavefront stage timing");
			for (size_t k = 0; k + 3 < marks.size(); k += 4)
			{
				float a = 0, b2 = 0, c = 0;
				(void)hipEventElapsedTime(&a, marks[k], marks[k + 1]);
				(void)hipEventElapsedTime(&b2, marks[k + 1], marks[k + 2]);
				(void)hipEventElapsedTime(&c, marks[k + 2], marks[k + 3]);
				times->extendMs += a;
				times->shadeMs += b2;
				times->shadowMs += c;
				times->extendLaunches++;
			}
		}
	}
#endif
}
