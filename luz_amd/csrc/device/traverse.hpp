// Two-level BVH traversal (closest hit and any hit) over the 64-byte node layout.
//
// One stack serves both levels: entering a mesh instance notes the stack's height, and a pop
// at that height leaves the instance (the world-space ray is restored). The instance's ray
// keeps the world parameterisation (its direction is the affine image of the world
// direction, not renormalised), so a hit distance needs no rescaling between levels.
//
// Semantics follow the reference's intersection routines:
//   slab test from T_MIN, zero direction components tested against the slab,
//   tMax <= tMin -> miss                          BVHNode.cpp:20-61, Mesh.cpp:99-140
//   Möller–Trumbore, |det| < 1e-12, inclusive edges, t in [tMin, tMax]
//                                                  Triangle.cpp:196-240,272-305
//   rectangle plane test and half-extent check      Rectangle.cpp:212-293
// A later equal-distance hit replaces an earlier one, as with the reference's
// `t > t_max` rejection.
#pragma once

#include "vec.hpp"
#include "../common/layout.h"

namespace luzgpu
{
	constexpr float	kTMinF = 0.001f;

	struct	SceneView
	{
		const Bvh4Node*	nodes;	// top level, then the mesh BVHs
		const GpuTri*	topTris;
		const GpuTri*	meshTris;
		const float*	meshNormals;
		const uint2*	tlasLeaf;	// top-level leaf items: (hittable index, kind << 28 | index)
		const GpuHittable*	hittables;
		const GpuRect*	rects;
		const GpuInstance*	instances;
		const GpuMaterial*	materials;
		const GpuLight*	lights;
		const double*	lightCdf;
		const double*	lightTriCdf;		// emissive mesh instances: triangle-area prefix sums
		const std::uint32_t*	lightTriSlot;	// ... and the mesh-triangle slot of each entry
		const float4*	envPixels;
		const float*	envPdf;
		const double*	envCdf;
		const std::uint32_t*	envGuide;	// texel-aligned with envCdf
		const double*	iesData;	// IES profiles of sphere lights (GpuLight::ies)
		const std::uint32_t*	unbounded;	// hittable ids of the planes, tested after the BVH
		const GpuSphere*	spheres;
		const GpuRect*	cubeFaces;
		const GpuVolume*	volumes;
		const GpuPlane*	planes;
	};

	struct	Ray
	{
		f3	o, d;
	};

	__device__ __forceinline__ Ray	makeRay(f3 o, f3 d) { return Ray{o, d}; }

	// The 48-byte triangle is fetched as three 16-byte loads issued together (one memory
	// round trip), not field by field, and tested without branches. `id`: GpuTri::prim.
	__device__ __forceinline__ bool	triHit(const GpuTri& tri, const Ray& r, float tMin, float tMax, float& t, float& u, float& v,
		std::int32_t& id)
	{
		const float4* tp = reinterpret_cast<const float4*>(&tri);
		const float4 A = tp[0], B = tp[1], C = tp[2];
		id = __float_as_int(A.w);
		const f3 v0 = mk(A.x, A.y, A.z), e1 = mk(B.x, B.y, B.z), e2 = mk(C.x, C.y, C.z);
		const f3 p = cross(r.d, e2);
		const float det = dot(e1, p);
		const f3 tv = r.o - v0;
		const float inv = __builtin_amdgcn_rcpf(det);	// 1 ulp, against the FP64 reference's 1 / det
		u = dot(tv, p) * inv;
		const f3 q = cross(tv, e1);
		v = dot(r.d, q) * inv;
		t = dot(e2, q) * inv;
		return !((fabsf(det) < 1e-12f) | (u < 0.0f) | (u > 1.0f) | (v < 0.0f) | (u + v > 1.0f) | (t > tMax) | (t < tMin));
	}

	__device__ __forceinline__ bool	rectHit(const GpuRect& rc, const Ray& r, float tMin, float tMax, float& t)
	{
		const f3 n = ld3(rc.normal);
		const f3 pos = ld3(rc.position);
		const float a = dot(r.o - pos, n);
		const float b = dot(r.d, n);
		if (b == 0.0f || (a < 0.0f && b < 0.0f) || (a > 0.0f && b > 0.0f))
		{
			return false;
		}
		t = -a / b;
		if (t > tMax || t < tMin)
		{
			return false;
		}
		const f3 d = (r.o + r.d * t) - pos;
		return !(fabsf(dot(d, ld3(rc.widthAxis))) > rc.halfWidth || fabsf(dot(d, ld3(rc.heightAxis))) > rc.halfHeight);
	}

	__device__ __forceinline__ bool	zeroDir(const Ray& r)
	{
		return r.d.x == 0.0f && r.d.y == 0.0f && r.d.z == 0.0f;
	}

	// Sphere::hit / hitAny (Sphere.cpp:226-301), in FP64 from the fp32 ray: the reference
	// solves the quadratic for a unit direction (a = 1).
	__device__ __forceinline__ bool	sphereHit(const GpuSphere& sp, const Ray& r, float tMin, float tMax, float& t)
	{
		if (zeroDir(r)) return false;
		const double ox = static_cast<double>(r.o.x) - sp.center[0], oy = static_cast<double>(r.o.y) - sp.center[1],
			oz = static_cast<double>(r.o.z) - sp.center[2];
		const double dx = r.d.x, dy = r.d.y, dz = r.d.z;
		const double b = ox * dx + oy * dy + oz * dz;
		const double rr = static_cast<double>(sp.radius) * sp.radius;
		const double c = (ox * ox + oy * oy + oz * oz) - rr;
		const double disc = b * b - c;
		if (disc < 0.0) return false;
		const double sq = sqrt(disc);
		double root = -b - sq;
		if (root < tMin || root > tMax)
		{
			root = -b + sq;
			if (root < tMin || root > tMax) return false;
		}
		t = static_cast<float>(root);
		return true;
	}

	// ConstantVolume::sampleScatteringDistance (ConstantVolume.cpp:62-101) with the boundary's
	// hitInterval over (-T_MAX, T_MAX) (Sphere.cpp:303-339, Cube.cpp:120-164). `logU` is
	// log(max(u, 1e-12)) of the path's DIM_VOLUME_DISTANCE sample at this bounce.
	__device__ __forceinline__ bool	volumeHit(const GpuVolume& v, const Ray& r, float tMin, float tMax, float logU, float& t)
	{
		if (zeroDir(r)) return false;
		double entry, exit;
		const double o[3] = {r.o.x, r.o.y, r.o.z}, d[3] = {r.d.x, r.d.y, r.d.z};
		if (v.sphere)
		{
			const double ox = o[0] - v.center[0], oy = o[1] - v.center[1], oz = o[2] - v.center[2];
			const double b = ox * d[0] + oy * d[1] + oz * d[2];
			const double c = (ox * ox + oy * oy + oz * oz) - static_cast<double>(v.radius) * v.radius;
			const double disc = b * b - c;
			if (disc < 0.0) return false;
			const double sq = sqrt(disc);
			entry = fmin(-b - sq, -b + sq);
			exit = fmax(-b - sq, -b + sq);
			if (entry >= exit) return false;
		}
		else
		{
			entry = -1.7976931348623157e308;
			exit = 1.7976931348623157e308;
			const float lo[3] = {v.lo[0], v.lo[1], v.lo[2]}, hi[3] = {v.hi[0], v.hi[1], v.hi[2]};
			for (int a = 0; a < 3; a++)
			{
				if (d[a] == 0.0)
				{
					if (o[a] < lo[a] || o[a] > hi[a]) return false;
					continue;
				}
				const double inv = 1.0 / d[a];
				double t0 = (lo[a] - o[a]) * inv, t1 = (hi[a] - o[a]) * inv;
				if (t0 > t1)
				{
					const double x = t0; t0 = t1; t1 = x;
				}
				entry = fmax(entry, t0);
				exit = fmin(exit, t1);
				if (entry >= exit) return false;
			}
		}
		if (entry < tMin) entry = tMin;
		if (exit > tMax) exit = tMax;
		if (entry >= exit) return false;
		if (entry < 0.0) entry = 0.0;
		const double len = sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
		if (!(len > 0.0) || !isfinite(len)) return false;
		const double inside = (exit - entry) * len;
		const double dist = static_cast<double>(v.negInvDensity) * logU;
		if (dist > inside) return false;
		t = static_cast<float>(entry + dist / len);
		return true;
	}

	// Plane::hit / hitAny (Plane.cpp:51-87)
	__device__ __forceinline__ bool	planeHit(const GpuPlane& pl, const Ray& r, float tMin, float tMax, float& t)
	{
		const f3 o = ld3(pl.orientation);
		const float d = dot(r.d, o);
		if (d == 0.0f) return false;
		t = dot(ld3(pl.point) - r.o, o) / d;
		return !(t > tMax || t < tMin);
	}

	__device__ __forceinline__ Ray	toLocal(const float4 r0, const float4 r1, const float4 r2, const Ray& w)
	{
		const float m[12] = {r0.x, r0.y, r0.z, r0.w, r1.x, r1.y, r1.z, r1.w, r2.x, r2.y, r2.z, r2.w};
		const f3 o = mk(m[0] * w.o.x + m[1] * w.o.y + m[2] * w.o.z + m[3],
			m[4] * w.o.x + m[5] * w.o.y + m[6] * w.o.z + m[7],
			m[8] * w.o.x + m[9] * w.o.y + m[10] * w.o.z + m[11]);
		const f3 d = mk(m[0] * w.d.x + m[1] * w.d.y + m[2] * w.d.z,
			m[4] * w.d.x + m[5] * w.d.y + m[6] * w.d.z,
			m[8] * w.d.x + m[9] * w.d.y + m[10] * w.d.z);
		return makeRay(o, d);
	}

	__device__ __forceinline__ Ray	toLocal(const GpuInstance& in, const Ray& w)
	{
		const float4* mp = reinterpret_cast<const float4*>(in.worldToLocal);
		return toLocal(mp[0], mp[1], mp[2], w);
	}

	struct	HitInfo
	{
		float	t;
		float	u, v;
		std::uint32_t	hittable;	// top-level hittable index, 0xffffffff: none
		std::int32_t	tri;		// mesh triangle slot (global) for instances, -1 otherwise
	};

	// The primitive a ray leaves from. A planar one (triangle, rectangle, cube face, plane) is
	// left out of the ray's traversal: a ray cannot meet the plane it starts on again, and
	// the FP64 reference never does, but an fp32 hit position may sit a little behind that
	// plane, so a grazing ray would meet it again beyond T_MIN. Curved and volume hits, and
	// camera rays, exclude nothing (hittable 0xffffffff).
	struct	RayOrigin
	{
		std::uint32_t	hittable;
		std::int32_t	tri;		// instance: mesh triangle slot; cube: face; else -1
	};
	constexpr RayOrigin	kNoOrigin{0xffffffffu, -1};

	// What a stack holds beyond the bound that a scene is admitted by (its deferred entries,
	// PackedScene::tlasStackBound + blasStackBound): one entry where a leaf of two kinds was split
	// into nodes, and the slot above the top entry that push3 writes in vain: with less, the
	// clamp would put that write on the top entry itself.
	constexpr int	kStackReserve = 2;

	// Per-thread traversal stack in LDS, laid out [depth][thread] so the 64 lanes of a
	// wave touch 64 consecutive banks.
	template <int Depth, int Block>
	struct	LdsStack
	{
		std::uint32_t*	base;
		int	sp;

		// The host refuses scenes whose bound and kStackReserve exceed Depth; the clamp only keeps
		// every LDS access inside this thread's column whatever happens.
		__device__ __forceinline__ void	push(std::uint32_t v) { base[min(sp, Depth - 1) * Block] = v; sp++; }
		// pushes a if wanted, then b, then c: a slot written in vain is the next push's
		__device__ __forceinline__ void	push3(std::uint32_t a, bool wa, std::uint32_t b, bool wb, std::uint32_t c, bool wc)
		{
			base[min(sp, Depth - 1) * Block] = a;
			sp += wa ? 1 : 0;
			base[min(sp, Depth - 1) * Block] = b;
			sp += wb ? 1 : 0;
			base[min(sp, Depth - 1) * Block] = c;
			sp += wc ? 1 : 0;
		}
		__device__ __forceinline__ std::uint32_t	pop() { sp--; return base[min(sp, Depth - 1) * Block]; }
		__device__ __forceinline__ void	reset() { sp = 0; }
	};

	// A private traversal stack (scratch memory) for the rare traversals made outside the
	// traversal kernels, such as re-intersecting one emissive mesh instance for its light pdf.
	// Scenes are admitted only when a BLAS traversal fits (their bound is checked on load).
	constexpr int	kLocalStackDepth = 48;
	struct	LocalStack
	{
		std::uint32_t	v[kLocalStackDepth];
		int	sp;

		__device__ __forceinline__ void	push(std::uint32_t x) { v[min(sp, kLocalStackDepth - 1)] = x; sp++; }
		__device__ __forceinline__ void	push3(std::uint32_t a, bool wa, std::uint32_t b, bool wb, std::uint32_t c, bool wc)
		{
			if (wa) push(a);
			if (wb) push(b);
			if (wc) push(c);
		}
		__device__ __forceinline__ std::uint32_t	pop() { sp--; return v[min(sp, kLocalStackDepth - 1)]; }
		__device__ __forceinline__ void	reset() { sp = 0; }
	};

	// Node / primitive visit counts (only maintained when Count is true).
	struct	VisitCounter
	{
		std::uint32_t	nodes;
		std::uint32_t	prims;
	};

	// LDS stack of LdsDepth entries per thread, continued in a per-thread column of global
	// memory (`spill`, stride = threads in the grid) for deeper entries. Keeping the LDS
	// part short lets 8 waves per SIMD share a CU's LDS.
	template <int LdsDepth, int Block>
	struct	SpillStack
	{
		std::uint32_t*	base;
		std::uint32_t*	spill;
		std::uint32_t	stride;
		int	sp;
		int	capacity;

		__device__ __forceinline__ void	push(std::uint32_t v)
		{
			if (sp < LdsDepth) base[sp * Block] = v;
			else spill[static_cast<size_t>(min(sp, capacity - 1) - LdsDepth) * stride] = v;
			sp++;
		}
		// As three pushes. While no lane of the wave is near the end of its LDS column (nearly
		// always) the three slots are written without branches: one that was not wanted is the
		// next push's slot.
		__device__ __forceinline__ void	push3(std::uint32_t a, bool wa, std::uint32_t b, bool wb, std::uint32_t c, bool wc)
		{
			if (__ballot(sp > LdsDepth - 3) == 0ull)
			{
				base[sp * Block] = a;
				sp += wa ? 1 : 0;
				base[sp * Block] = b;
				sp += wb ? 1 : 0;
				base[sp * Block] = c;
				sp += wc ? 1 : 0;
				return;
			}
			if (wa) push(a);
			if (wb) push(b);
			if (wc) push(c);
		}
		__device__ __forceinline__ std::uint32_t	pop()
		{
			sp--;
			if (__ballot(sp >= LdsDepth) == 0ull || sp < LdsDepth) return base[sp * Block];
			return spill[static_cast<size_t>(min(sp, capacity - 1) - LdsDepth) * stride];
		}
		__device__ __forceinline__ void	reset() { sp = 0; }
	};

	// Resumable per-lane traversal state. A persistent kernel advances it one entry at a time
	// (nodeStep for an internal node, leafStep for a leaf, then popEntry when neither named the
	// next entry), so it can hand a lane a new ray as soon as its traversal ends.
	//
	// Node tests run on the ray in slab form, set once per level: on each axis a plane at
	// origin + q * scale is met at t = fma(q, scale * inv, fma(origin, inv, -o * inv)). The
	// reciprocal is the hardware's (1 ulp); an axis the ray is parallel to takes a huge one, so
	// its planes lie far behind or ahead, as AABB::hit's test of the origin against the slab
	// has it (AABB.cpp:37-80). `nearC` / `farC` are -o * inv moved outward by 2^-21 of
	// itself, which covers the rounding of that product, and the far distance is compared with a
	// relative margin of 2^-19 for the reciprocals' and the last sums'. The sum with
	// origin * inv rounds by up to 2^-24 of the distance to the node's origin, which neither
	// covers where that is large against |o| and the plane is near: there a box can be missed by
	// rays that pass within 2^-24 of that distance of its border (scene units; 6e-5 at 1000),
	// as vertices that far away are rounded in FP32. Box tests only decide which primitives are
	// tested; the primitive tests alone decide the hit.
	struct	TraceState
	{
		f3	world_o, world_d;	// world-space ray, restored when an instance is left
		f3	o, d;				// ray of the current level
		f3	inv, nearC, farC;	// its slab form
		HitInfo	hit;	// hit.t is the current closest distance
		float	logU;	// log(max(u, 1e-12)) of the volume free-flight sample (scenes with volumes)
		std::uint32_t	unbounded;	// this ray's scene: unbounded list base << 16 | count
		std::uint32_t	entry;
		std::uint32_t	instHittable;
		RayOrigin	from;	// planar primitive the ray leaves from
		int	instBase;		// inside an instance: the stack height it was entered at; else -1
		bool	found;

		__device__ __forceinline__ Ray	ray() const { return Ray{o, d}; }
		__device__ __forceinline__ Ray	world() const { return Ray{world_o, world_d}; }

		__device__ __forceinline__ static void	slabAxis(float o, float d, float& inv, float& n, float& f)
		{
			float r = __builtin_amdgcn_rcpf(d);
			// zero, denormal, infinite and NaN components: parallel
			r = __builtin_amdgcn_classf(r, 0x198) ? r : 0x1p80f;	// +-normal, +-denormal
			const float c = -o * r;
			const float slack = fmaxf(fabsf(c) * 0x1p-21f, fabsf(r) * 0x1p-41f);
			inv = r;
			n = c - slack;
			f = c + slack;
		}

		__device__ __forceinline__ void	setLevel(f3 origin, f3 dir)
		{
			o = origin;
			d = dir;
			slabAxis(o.x, d.x, inv.x, nearC.x, farC.x);
			slabAxis(o.y, d.y, inv.y, nearC.y, farC.y);
			slabAxis(o.z, d.z, inv.z, nearC.z, farC.z);
		}
	};

	// Not a node: popped first when a scene has only unbounded hittables.
	constexpr std::uint32_t	kNoEntry = kEmptyChild;

	// Starts a traversal; returns false when there is nothing to traverse.
	template <typename Stack>
	__device__ __forceinline__ bool	traceBegin(TraceState& st, std::int32_t tlasRoot, std::uint32_t unbounded,
		const Ray& worldRay, float tMax, float logU, RayOrigin from, Stack& stack)
	{
		st.logU = logU;
		st.from = from;
		st.unbounded = unbounded;
		st.world_o = worldRay.o;
		st.world_d = worldRay.d;
		st.setLevel(worldRay.o, worldRay.d);
		st.hit.t = tMax;
		st.hit.hittable = 0xffffffffu;
		st.hit.tri = -1;
		// without bounded hittables only the unbounded ones are tested: start from the
		// empty entry, which leads straight to the end of the traversal
		st.entry = tlasRoot >= 0 ? static_cast<std::uint32_t>(tlasRoot) : kNoEntry;
		st.instHittable = 0;
		st.instBase = -1;
		st.found = false;
		// an any-hit query ends with entries still on the stack: every traversal starts
		// from an empty stack
		stack.reset();
		return tlasRoot >= 0 || (unbounded & 0xffffu) != 0u;
	}

	// Opens the internal node st.entry: the nearest hit child becomes the entry, the others are
	// pushed, farthest first. Returns false when no child is hit (the next entry is popped).
	//
	// Bound by VALU issue: the whole node is one straight line (about 130 instructions against
	// the 330 of a form that branched per child, per push and for axis-parallel rays, and
	// decoded exponents and leaf counts), so it keeps to four 16-byte loads issued together, a
	// ready scale and ready stack entries in the node, one six-comparator sort, and stack
	// writes that need no branch.
	template <bool Count, typename Stack>
	__device__ __forceinline__ bool	nodeStep(const SceneView& s, TraceState& st, Stack& stack, VisitCounter* counter)
	{
		//   n0 = origin xyz | scale x      n1 = scale yz | q_lo x, y
		//   n2 = q_lo z | q_hi xyz         n3 = children
		const uint4* np = reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(s.nodes) + (st.entry << 6));
		const uint4 n0 = np[0], n1 = np[1], n2 = np[2], n3 = np[3];
		if (Count) counter->nodes++;
		const float s0 = __uint_as_float(n0.w) * st.inv.x, s1 = __uint_as_float(n1.x) * st.inv.y, s2 = __uint_as_float(n1.y) * st.inv.z;
		const float o0 = __uint_as_float(n0.x), o1 = __uint_as_float(n0.y), o2 = __uint_as_float(n0.z);
		const float nb0 = fmaf(o0, st.inv.x, st.nearC.x), nb1 = fmaf(o1, st.inv.y, st.nearC.y), nb2 = fmaf(o2, st.inv.z, st.nearC.z);
		const float fb0 = fmaf(o0, st.inv.x, st.farC.x), fb1 = fmaf(o1, st.inv.y, st.farC.y), fb2 = fmaf(o2, st.inv.z, st.farC.z);
		// fma(q, s, b) is monotone in q (increasing for s >= 0), so on each axis the q_lo plane
		// is the near one when the direction is positive and the q_hi plane otherwise: the words
		// are chosen once per node
		const bool p0 = st.inv.x > 0.0f, p1 = st.inv.y > 0.0f, p2 = st.inv.z > 0.0f;
		const std::uint32_t near0 = p0 ? n1.z : n2.y, far0 = p0 ? n2.y : n1.z;
		const std::uint32_t near1 = p1 ? n1.w : n2.z, far1 = p1 ? n2.z : n1.w;
		const std::uint32_t near2 = p2 ? n2.x : n2.w, far2 = p2 ? n2.w : n2.x;
		std::uint32_t e[4] = {n3.x, n3.y, n3.z, n3.w};
		float key[4];	// entry distance; a miss sorts last
		#pragma unroll
		for (int k = 0; k < 4; k++)
		{
			const float l0 = fmaf(static_cast<float>((near0 >> (8 * k)) & 0xffu), s0, nb0);
			const float h0 = fmaf(static_cast<float>((far0 >> (8 * k)) & 0xffu), s0, fb0);
			const float l1 = fmaf(static_cast<float>((near1 >> (8 * k)) & 0xffu), s1, nb1);
			const float h1 = fmaf(static_cast<float>((far1 >> (8 * k)) & 0xffu), s1, fb1);
			const float l2 = fmaf(static_cast<float>((near2 >> (8 * k)) & 0xffu), s2, nb2);
			const float h2 = fmaf(static_cast<float>((far2 >> (8 * k)) & 0xffu), s2, fb2);
			const float near = fmaxf(fmaxf(fmaxf(l0, l1), l2), kTMinF);
			const float far = fminf(fminf(fminf(h0, h1), h2), st.hit.t) * (1.0f + 0x1p-19f);
			const bool in = (far >= near) & (k == 0 || e[k] != kEmptyChild);
			key[k] = in ? near : INFINITY;
		}
		// Exchanges of neighbours alone keep equal distances in child order: of primitives hit at
		// the same distance the last one visited is the hit, and boxes entered at the same
		// distance (primitives of one plane, boxes around the ray's origin) are common. Five
		// exchanges would sort without keeping it, at most 1 % faster (a 1080p spheres frame
		// 31.7 against 32.0 ms, 720p hazy terrain 71.5 against 71.9).
		auto exchange = [&](int i) {
			const bool swap = key[i + 1] < key[i];
			const float ki = key[i];
			const std::uint32_t ei = e[i];
			key[i] = fminf(key[i + 1], ki);
			key[i + 1] = fmaxf(key[i + 1], ki);
			e[i] = swap ? e[i + 1] : ei;
			e[i + 1] = swap ? ei : e[i + 1];
		};
		exchange(0);
		exchange(2);
		exchange(1);
		exchange(0);
		exchange(2);
		exchange(1);
		stack.push3(e[3], key[3] < INFINITY, e[2], key[2] < INFINITY, e[1], key[1] < INFINITY);
		st.entry = e[0];
		return key[0] < INFINITY;
	}

	// What a leaf step leaves: the next entry is on the stack, is st.entry already, or the
	// any-hit query has ended.
	enum : int { STEP_POP = 0, STEP_ENTRY = 1, STEP_END = 2 };

	// Processes the leaf (or empty) st.entry: a run of triangles, a mesh instance (whose root
	// becomes the entry), or a list of other primitives.
	template <bool AnyHit, bool Count, int Feat>
	__device__ __forceinline__ int	leafStep(const SceneView& s, TraceState& st, int stackHeight, float tMin, VisitCounter* counter)
	{
		const std::uint32_t entry = st.entry;
		const bool mesh = st.instBase >= 0;
		if (entry == kNoEntry) return STEP_POP;
		const std::uint32_t start = entry & kLeafStartMask;
		const std::uint32_t kind = mesh ? kTopTriangles : (entry >> kTopKindShift) & 3u;
		const std::uint32_t last = (entry >> kLeafCountShift) & (mesh ? 15u : 3u);	// count - 1
		if (kind == kTopTriangles)
		{
			const GpuTri* tris = mesh ? s.meshTris : s.topTris;
			// the triangle the ray leaves from: a mesh triangle by its slot, a top-level one by
			// its hittable
			const std::int32_t skip = mesh ? (st.instHittable == st.from.hittable ? st.from.tri : -1)
				: static_cast<std::int32_t>(st.from.hittable);
			for (std::uint32_t i = 0; i <= last; i++)
			{
				if (Count) counter->prims++;
				const std::int32_t slot = static_cast<std::int32_t>(start + i);
				float t, u, v;
				std::int32_t id;
				const bool hit = triHit(tris[slot], st.ray(), tMin, st.hit.t, t, u, v, id);
				if (hit && (mesh ? slot : id) != skip)
				{
					st.found = true;
					st.hit.t = t; st.hit.u = u; st.hit.v = v;
					st.hit.hittable = mesh ? st.instHittable : static_cast<std::uint32_t>(id);
					st.hit.tri = mesh ? slot : -1;
					if (AnyHit) return STEP_END;
				}
			}
			return STEP_POP;
		}
		if (kind == kTopInstance)
		{
			if (Count) counter->prims++;
			// 3x4 map and mesh links: one group of four 16-byte loads
			const float4* ip = reinterpret_cast<const float4*>(s.instances + start);
			const float4 r0 = ip[0], r1 = ip[1], r2 = ip[2];
			const int4 links = reinterpret_cast<const int4*>(ip)[3];
			const Ray local = toLocal(r0, r1, r2, st.world());
			st.setLevel(local.o, local.d);
			st.instBase = stackHeight;
			st.instHittable = static_cast<std::uint32_t>(links.w);
			st.entry = static_cast<std::uint32_t>(links.x);
			return STEP_ENTRY;
		}
		const Ray ray = st.ray();
		for (std::uint32_t i = 0; i <= last; i++)
		{
			if (Count) counter->prims++;
			const uint2 item = s.tlasLeaf[start + i];
			const std::uint32_t h = item.x;
			const std::uint32_t hk = item.y >> kKindShift;
			const std::uint32_t idx = item.y & kIndexMask;
			float t = 0.0f;
			bool hit = false;
			std::int32_t part = -1;
			if (hk == GPU_HIT_RECTANGLE)
			{
				hit = h != st.from.hittable && rectHit(s.rects[idx], ray, tMin, st.hit.t, t);
			}
			else if ((Feat & kFeatAnalytic) && hk == GPU_HIT_SPHERE)
			{
				hit = sphereHit(s.spheres[idx], ray, tMin, st.hit.t, t);
			}
			else if ((Feat & kFeatAnalytic) && hk == GPU_HIT_CUBE)
			{
				// Cube::hit (Cube.cpp:97-111): its six faces, closest first-found
				float closest = st.hit.t;
				for (int f = 0; f < 6; f++)
				{
					float ft;
					if ((h != st.from.hittable || f != st.from.tri) && rectHit(s.cubeFaces[6 * idx + f], ray, tMin, closest, ft))
					{
						hit = true;
						t = closest = ft;
						part = f;
						if (AnyHit) break;
					}
				}
			}
			else if ((Feat & kFeatAnalytic) && hk == GPU_HIT_VOLUME)
			{
				hit = volumeHit(s.volumes[idx], ray, tMin, st.hit.t, st.logU, t);
			}
			// GPU_HIT_HIDDEN_SPHERE, an invisible sphere (Sphere.cpp:227-233, 271-277): never hit
			if (hit)
			{
				st.found = true;
				st.hit.t = t;
				st.hit.hittable = h;
				st.hit.tri = part;
				if (AnyHit) return STEP_END;
			}
		}
		return STEP_POP;
	}

	// Takes the next entry off the stack, leaving an instance whose entries are used up; returns
	// true when the traversal has ended (st.found and st.hit hold the result).
	template <bool AnyHit, int Feat, typename Stack>
	__device__ __forceinline__ bool	popEntry(const SceneView& s, TraceState& st, float tMin, Stack& stack)
	{
		if (stack.sp == st.instBase)
		{
			st.setLevel(st.world_o, st.world_d);
			st.instBase = -1;
		}
		if (stack.sp != 0)
		{
			st.entry = stack.pop();
			return false;
		}
		// the unbounded hittables after the acceleration structure (HitHelper.cpp:5-32)
		const std::uint32_t ubBase = st.unbounded >> 16, ubCount = (Feat & kFeatAnalytic) ? (st.unbounded & 0xffffu) : 0u;
		for (std::uint32_t i = 0; i < ubCount; i++)
		{
			const std::uint32_t h = s.unbounded[ubBase + i];
			const GpuPlane& pl = s.planes[s.hittables[h].kindIndex & kIndexMask];
			float t;
			if (h != st.from.hittable && planeHit(pl, st.world(), tMin, st.hit.t, t))
			{
				st.found = true;
				st.hit.t = t;
				st.hit.hittable = h;
				st.hit.tri = -1;
				if (AnyHit) return true;
			}
		}
		return true;
	}

	// Runs a traversal to its end: a lane opens nodes until it holds a leaf.
	template <bool AnyHit, bool Count, int Feat, typename Stack>
	__device__ __forceinline__ void	traceToEnd(const SceneView& s, TraceState& st, float tMin, Stack& stack, VisitCounter* counter)
	{
		for (;;)
		{
			while ((st.entry & kLeafBit) == 0u)
			{
				if (!nodeStep<Count>(s, st, stack, counter) && popEntry<AnyHit, Feat>(s, st, tMin, stack)) return;
			}
			const int r = leafStep<AnyHit, Count, Feat>(s, st, stack.sp, tMin, counter);
			if (r == STEP_END || (r == STEP_POP && popEntry<AnyHit, Feat>(s, st, tMin, stack))) return;
		}
	}

	__device__ __forceinline__ std::uint32_t	unboundedOf(const GpuParams& p)
	{
		return (p.unboundedBase << 16) | p.unboundedCount;
	}

	// Closest hit of a world ray against one mesh instance alone (MeshInstance::hit,
	// MeshInstance.cpp:303-327): its BLAS traversed in local space, t shared with the world
	// ray (the local direction is not renormalised).
	__device__ inline bool	instanceClosest(const SceneView& s, std::uint32_t instance, std::uint32_t hittable, const Ray& world,
		float tMax, HitInfo& hit)
	{
		const GpuInstance& in = s.instances[instance];
		const Ray local = toLocal(in, world);
		LocalStack stack;
		TraceState st;
		// entered at the bottom of the stack: popEntry ends the traversal there
		traceBegin(st, in.blasRoot, 0u, local, tMax, 0.0f, kNoOrigin, stack);
		st.instBase = 0;
		st.instHittable = hittable;
		traceToEnd<false, false, 0>(s, st, kTMinF, stack, nullptr);
		hit = st.hit;
		return st.found;
	}

	// The exclusion identity of a hit (see RayOrigin).
	__device__ __forceinline__ RayOrigin	originOf(const SceneView& s, const HitInfo& h)
	{
		const std::uint32_t kind = s.hittables[h.hittable].kindIndex >> kKindShift;
		const bool planar = kind == GPU_HIT_TRIANGLE || kind == GPU_HIT_RECTANGLE || kind == GPU_HIT_INSTANCE || kind == GPU_HIT_CUBE
			|| kind == GPU_HIT_PLANE;
		return planar ? RayOrigin{h.hittable, h.tri} : kNoOrigin;
	}

	template <bool AnyHit, bool Count = false, int Feat = kFeatAll, typename Stack>
	__device__ __forceinline__ bool	traverse(const SceneView& s, const GpuParams& p, const Ray& worldRay, float tMin, float tMax,
		HitInfo& hit, Stack& stack, VisitCounter* counter = nullptr, float logU = 0.0f, RayOrigin from = kNoOrigin)
	{
		TraceState st;
		if (traceBegin(st, p.tlasRoot, unboundedOf(p), worldRay, tMax, logU, from, stack))
		{
			traceToEnd<AnyHit, Count, Feat>(s, st, tMin, stack, counter);
		}
		hit = st.hit;
		return st.found;
	}
}
