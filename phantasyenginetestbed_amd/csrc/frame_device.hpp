// Device functions shared by the frame kernels: record indices, random streams, and a light's
// contribution and shadow ray at a hit record.
#pragma once

#include <hip/hip_runtime.h>

#include "kernels.hpp"
#include "rng.hpp"
#include "shading.hpp"

namespace phx {
namespace frame {

using namespace shading;

__device__ __forceinline__ uint32_t pixel_id(uint32_t x, uint32_t y, uint32_t w, uint32_t h)
{
	if ((w % 8u) == 0u && (h % 8u) == 0u) {
		const uint32_t tile = (y / 8u) * (w / 8u) + (x / 8u);
		return tile * 64u + (y % 8u) * 8u + (x % 8u);
	}
	return y * w + x;
}

// The pixel of a record: pixel_id's inverse.
__device__ __forceinline__ uint2 pixel_of(uint32_t id, uint32_t w, uint32_t h)
{
	if ((w % 8u) == 0u && (h % 8u) == 0u) {
		const uint32_t tile = id / 64u, in = id % 64u;
		return make_uint2(tile % (w / 8u) * 8u + in % 8u, tile / (w / 8u) * 8u + in / 8u);
	}
	return make_uint2(id % w, id / w);
}

__device__ __forceinline__ Pcg32 frame_rng(uint64_t seed, uint32_t frame, uint32_t purpose,
                                           uint32_t id)
{
	return Pcg32::seeded(seed ^ (uint64_t(frame) << 32), (uint64_t(purpose) << 32) | id);
}

__device__ __forceinline__ V3 xyz(float4 a) { return v3(a.x, a.y, a.z); }

// What a light gives a record (shadeHit, MaterialKernel.cu:49-114): the contribution
// mask * falloff * shade and, if `ray`, a shadow ray from the record's point towards a point on the
// light's disc (soft shadows, radius 0 = point light). No ray when the light has no static shadows or
// contributes nothing (every channel <= 1e-4).
struct LightSample {
	V3 c;
	bool ray;
	V3 dir;
	float len;
};

__device__ __forceinline__ LightSample sample_light(const PhxSphereLight& L, V3 p, V3 n, V3 view,
                                                    V3 albedo, float rough, float metal, V3 mask,
                                                    Pcg32& rng)
{
	LightSample s;
	const V3 lp = v3(L.pos[0], L.pos[1], L.pos[2]);
	const V3 toL = sub(lp, p);
	const float dist = length(toL);
	const V3 l = divs(toL, dist);
	const float fo = falloff(dist, L.range);
	const V3 sh = shade(n, view, albedo, rough, metal, l, dist,
	                    v3(L.strength[0], L.strength[1], L.strength[2]), L.range);
	s.c = mul(scale(mask, fo), sh);
	const float eps = 0.0001f;
	const bool lit = s.c.x > eps || s.c.y > eps || s.c.z > eps;
	s.ray = L.staticShadows && lit;
	s.dir = v3(0.0f, 1.0f, 0.0f);
	s.len = 0.001f;
	if (s.ray) {
		const V3 cu = fabsf(n.z) > 0.01f ? normalize(v3(0.0f, -n.z, n.y))
		                                 : normalize(v3(-n.y, n.x, 0.0f));
		const V3 cv = cross(cu, l);
		const float r1 = rng.uniform();
		const float r2 = rng.uniform();
		const float cd = L.radius * (2.0f * r2 - 1.0f);
		float sn, cs;
		turn_sincos(r1, sn, cs);
		const V3 off = add(scale(scale(cu, cs), cd), scale(scale(cv, sn), cd));
		const V3 diff = sub(add(lp, off), p);
		s.dir = normalize(diff);
		s.len = length(diff);
	}
	return s;
}

}  // namespace frame
}  // namespace phx
