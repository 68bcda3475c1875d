// SBVH traversal kernels for gfx950 (wave64).
//
// Node layout (64 B, BVHNode.hpp:23-149): four 16-B words read as four 128-bit loads
//   w0 = lc.min.xyz, lc.max.x   w1 = lc.max.yz, rc.min.xy   w2 = rc.min.z, rc.max.xyz
//   w3 = (lcIndex, rcIndex, lcNumTriangles, rcNumTriangles)
// Triangles are the pre-transformed copy made at upload: (p0, e1 = p1 - p0, e2 = p2 - p0), three
// 128-bit loads per triangle.
//
// Visiting order of every closest-hit kernel here is castRay's (BVHTraversal.hpp:37-128): pop a
// node, decide both children against min(tMax, closest.t) taken before either is processed,
// handle the left child (push if inner, test its triangles if a leaf), then the right child; the
// stack is LIFO. The persistent kernels keep the node castRay would pop next in a register
// ("next") and the rest of castRay's stack in LDS, so the order -- and every hit -- is unchanged.
#include <hip/hip_runtime.h>

#include <mutex>

#include "frame_device.hpp"
#include "kernels.hpp"
#include "trace_device.hpp"
#include "wide_nodes.hpp"

namespace phx {
namespace {

constexpr uint32_t kInvalid = 0xFFFFFFFFu;
constexpr int kBlock = 256;

// Address-space views: records are loaded through pointers the compiler knows to be global (or
// LDS), so the loads are global_load / ds_read rather than flat loads, whose latency is higher
// and which wait on both the vector-memory and LDS counters.
typedef uint32_t U32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t U32x4 __attribute__((ext_vector_type(4)));
typedef float F32x4 __attribute__((ext_vector_type(4)));
#if defined(__HIP_DEVICE_COMPILE__)
typedef const float4 __attribute__((address_space(1))) GlobalF4;
typedef const F32x4 __attribute__((address_space(1))) GlobalV4;
typedef F32x4 __attribute__((address_space(3))) LdsF4;
typedef U32x2 __attribute__((address_space(1))) GlobalU2;
typedef U32x4 __attribute__((address_space(1))) GlobalU4;
typedef uint8_t __attribute__((address_space(1))) GlobalU8;
typedef U32x2 __attribute__((address_space(3))) LdsU2;
typedef uint32_t __attribute__((address_space(3))) LdsU1;
#else  // the host pass only needs the declarations to parse
typedef const float4 GlobalF4;
typedef const F32x4 GlobalV4;
typedef F32x4 LdsF4;
typedef U32x2 GlobalU2;
typedef U32x4 GlobalU4;
typedef uint8_t GlobalU8;
typedef U32x2 LdsU2;
typedef uint32_t LdsU1;
#endif
__device__ __forceinline__ GlobalF4* as_global(const float4* p) { return (GlobalF4*)(p); }

struct NodeWords {
	float4 w0, w1, w2;
	int4 w3;
};

__device__ __forceinline__ NodeWords load_node(const float4* __restrict__ nodes, uint32_t i)
{
	NodeWords n;
	const float4* p = nodes + 4u * i;
	n.w0 = p[0];
	n.w1 = p[1];
	n.w2 = p[2];
	n.w3 = reinterpret_cast<const int4*>(p)[3];
	return n;
}

struct Closest {
	uint32_t tri;
	float t, u, v;
};

struct Counts {
	uint32_t nodes = 0, accepted = 0, triTests = 0, boxHits = 0;
};

// Tests the `count` triangles of a leaf starting at `first` (BVHTraversal.hpp:78-93).
template <bool kCount>
__device__ __forceinline__ void closest_leaf(const dev::Ray& r, const float4* __restrict__ tris,
                                             uint32_t first, int32_t count, Closest& c, Counts& k)
{
	for (int32_t j = 0; j < count; j++) {
		const float4* p = tris + 3u * (first + uint32_t(j));
		const float4 p0 = p[0], e1 = p[1], e2 = p[2];
		float t, u, v;
		if (dev::triangle_pre(r, p0, e1, e2, t, u, v) && t < c.t && r.tMin <= t && t <= r.tMax) {
			c.tri = first + uint32_t(j);
			c.t = t;
			c.u = u;
			c.v = v;
			if (kCount) k.accepted++;
		}
	}
	if (kCount) k.triTests += uint32_t(count);
}

// Any-hit leaf: true iff a triangle has tMin <= t < tMax (RayCastKernel.cu:759-765).
__device__ __forceinline__ bool anyhit_leaf(const dev::Ray& r, const float4* __restrict__ tris,
                                            uint32_t first, int32_t count)
{
	for (int32_t j = 0; j < count; j++) {
		const float4* p = tris + 3u * (first + uint32_t(j));
		float t, u, v;
		if (dev::triangle_pre(r, p[0], p[1], p[2], t, u, v) && r.tMin <= t && t < r.tMax)
			return true;
	}
	return false;
}

__device__ __forceinline__ uint32_t child_index(int32_t raw)
{
	return uint32_t(raw < 0 ? ~raw : raw);
}

// To the block's stripe of the counters (an address takes an addition every 10 ns).
__device__ __forceinline__ void add_counts(unsigned long long* counters, const Counts& k)
{
	counters += blockIdx.x % kCountStripes * kCountStride;
	atomicAdd(&counters[0], (unsigned long long)k.nodes);
	atomicAdd(&counters[1], (unsigned long long)k.accepted);
	atomicAdd(&counters[2], (unsigned long long)k.triTests);
	atomicAdd(&counters[3], 2ull * k.nodes);
	atomicAdd(&counters[4], (unsigned long long)k.boxHits);
}

// ---- one ray per lane -------------------------------------------------------------------------

// Deepest castRay stack for a tree of depth <= 64 (enforced at upload): one pending entry per
// level plus the two children of the node being expanded.
constexpr int kSimpleStack = 72;
// Words that hold such a stack, or 8-B entries of either walk.
constexpr int kMaxPending = 66;  // children of a binary walk (64 levels), or slots of a wide one
static_assert(int(kWideMaxPending) <= kMaxPending, "pending slots of a wide walk");
constexpr int kStackWords = 2 * kMaxPending;
static_assert(kStackWords >= kSimpleStack, "4-B entries");

// castRay<144> of one ray (BVHTraversal.hpp:37-128) into `c` (which holds the miss result on
// entry): pop, decide both children, left first; a visited leaf is tested at once, a visited
// inner node pushed.
// Pending stack of one lane: its first words in the lane's LDS column (word e at col[e * kBlock], one
// 4-B word per lane per row, so a wave's accesses are conflict-free), the rest in private memory. A
// pop is on the path to the next node's load, and an LDS pop returns sooner than a private (scratch)
// one. Binary traversals keep 4-B entries (put / get), wide ones 8-B entries of a reference and its
// entry distance (put2 / get2).
template <int kLds>
struct ColumnStack {
	static_assert(kLds % 2 == 0, "an 8-B entry is in one place");
	uint32_t* col;
	uint32_t deep[kStackWords - kLds];
	__device__ __forceinline__ void put(int e, uint32_t v)
	{
		if (e < kLds)
			col[e * kBlock] = v;
		else
			deep[e - kLds] = v;
	}
	__device__ __forceinline__ uint32_t get(int e) const
	{
		return e < kLds ? col[e * kBlock] : deep[e - kLds];
	}
	__device__ __forceinline__ void put2(int e, uint32_t ref, float tIn)
	{
		if (2 * e < kLds) {
			col[2 * e * kBlock] = ref;
			col[(2 * e + 1) * kBlock] = __float_as_uint(tIn);
		} else {
			deep[2 * e - kLds] = ref;
			deep[2 * e + 1 - kLds] = __float_as_uint(tIn);
		}
	}
	__device__ __forceinline__ void get2(int e, uint32_t& ref, float& tIn) const
	{
		if (2 * e < kLds) {
			ref = col[2 * e * kBlock];
			tIn = __uint_as_float(col[(2 * e + 1) * kBlock]);
		} else {
			ref = deep[2 * e - kLds];
			tIn = __uint_as_float(deep[2 * e + 1 - kLds]);
		}
	}
};

// LDS stack words per lane of the one-ray-per-lane casts (24 KB per 256-thread block). Larger splits
// lower the blocks a CU holds and measured slower.
constexpr int kSimpleLds = 24;

template <bool kCount, class Stack>
__device__ __forceinline__ void closest_one(const float4* __restrict__ nodes,
                                            const float4* __restrict__ tris, const dev::Ray& r,
                                            Closest& c, Counts& k, Stack& stack)
{
	stack.put(0, 0u);
	int sp = 1;
	while (sp > 0) {
		sp--;
		const NodeWords nd = load_node(nodes, stack.get(sp));
		if (kCount) k.nodes++;
		float inL, outL, inR, outR;
		dev::slab(r, nd.w0.x, nd.w0.y, nd.w0.z, nd.w0.w, nd.w1.x, nd.w1.y, inL, outL);
		dev::slab(r, nd.w1.z, nd.w1.w, nd.w2.x, nd.w2.y, nd.w2.z, nd.w2.w, inR, outR);
		const float tCurrMax = dev::min_first(r.tMax, c.t);
		const bool visitL = (outL >= inL) && outL > r.tMin && inL < tCurrMax;
		const bool visitR = (outR >= inR) && outR > r.tMin && inR < tCurrMax;
		if (visitL) {
			if (kCount) k.boxHits++;
			if (nd.w3.z == 0) {
				if (sp < kSimpleStack) stack.put(sp++, child_index(nd.w3.x));
			} else {
				closest_leaf<kCount>(r, tris, child_index(nd.w3.x), nd.w3.z, c, k);
			}
		}
		if (visitR) {
			if (kCount) k.boxHits++;
			if (nd.w3.w == 0) {
				if (sp < kSimpleStack) stack.put(sp++, child_index(nd.w3.y));
			} else {
				closest_leaf<kCount>(r, tris, child_index(nd.w3.y), nd.w3.w, c, k);
			}
		}
	}
}

// Any-hit leaf that counts its triangle tests (up to and including the first hit).
__device__ __forceinline__ bool anyhit_leaf_counted(const dev::Ray& r,
                                                    const float4* __restrict__ tris,
                                                    uint32_t first, int32_t count, Counts& k)
{
	for (int32_t j = 0; j < count; j++) {
		const float4* p = tris + 3u * (first + uint32_t(j));
		float t, u, v;
		k.triTests++;
		if (dev::triangle_pre(r, p[0], p[1], p[2], t, u, v) && r.tMin <= t && t < r.tMax) {
			k.accepted++;
			return true;
		}
	}
	return false;
}

// Any hit of one ray: castRay's traversal with tCurrMax = tMax, stopping at the first triangle
// with tMin <= t < tMax. kCount adds castDebugRay-style counters of that traversal to k.
template <bool kCount, class Stack>
__device__ __forceinline__ bool anyhit_one(const float4* __restrict__ nodes,
                                           const float4* __restrict__ tris, const dev::Ray& r,
                                           Counts& k, Stack& stack)
{
	stack.put(0, 0u);
	int sp = 1;
	bool occluded = false;
	while (sp > 0 && !occluded) {
		sp--;
		const NodeWords nd = load_node(nodes, stack.get(sp));
		if (kCount) k.nodes++;
		float inL, outL, inR, outR;
		dev::slab(r, nd.w0.x, nd.w0.y, nd.w0.z, nd.w0.w, nd.w1.x, nd.w1.y, inL, outL);
		dev::slab(r, nd.w1.z, nd.w1.w, nd.w2.x, nd.w2.y, nd.w2.z, nd.w2.w, inR, outR);
		const bool visitL = (outL >= inL) && outL > r.tMin && inL < r.tMax;
		const bool visitR = (outR >= inR) && outR > r.tMin && inR < r.tMax;
		if (visitL) {
			if (kCount) k.boxHits++;
			if (nd.w3.z == 0) {
				if (sp < kSimpleStack) stack.put(sp++, child_index(nd.w3.x));
			} else {
				occluded = kCount ? anyhit_leaf_counted(r, tris, child_index(nd.w3.x), nd.w3.z, k)
				                  : anyhit_leaf(r, tris, child_index(nd.w3.x), nd.w3.z);
			}
		}
		if (visitR && !occluded) {
			if (kCount) k.boxHits++;
			if (nd.w3.w == 0) {
				if (sp < kSimpleStack) stack.put(sp++, child_index(nd.w3.y));
			} else {
				occluded = kCount ? anyhit_leaf_counted(r, tris, child_index(nd.w3.y), nd.w3.w, k)
				                  : anyhit_leaf(r, tris, child_index(nd.w3.y), nd.w3.w);
			}
		}
	}
	return occluded;
}

// ---- four-wide nodes ---------------------------------------------------------------------------
//
// wide_nodes.hpp says what they are and why taking their slots in order, with each slot's entry
// distance compared again when it is taken, gives castRay's hits bit for bit for every ray with an origin
// within 2^126. Rays whose slab values may be NaN are decided with castRay's own min and max (dev::slab)
// by the kernels that trace four lanes per ray or one ray per lane in persistent waves; the others trace
// such rays on the binary nodes (dev::Ray::nanFree).
// A traversal is bound by its chain of dependent steps; on 1,004,000 triangles a bounce ray takes
// 9.8 wide node visits where it takes 21.6 binary ones (random triangles: 32 for 65).

struct WideWords {
	float4 w[8];  // slot i: (min.xyz, reference) in word 2i, (max.xyz, lastMax) in word 2i + 1
};

__device__ __forceinline__ WideWords load_wide(const float4* __restrict__ wide, uint32_t i)
{
	WideWords n;
	const float4* p = wide + 8u * size_t(i);
#pragma unroll
	for (int k = 0; k < 8; k++) n.w[k] = p[k];
	return n;
}

// Entry distance and box predicate of the four slots against tCurrMax (BVHTraversal.hpp:59-64;
// any-hit: tMax).
struct WideVisit {
	float tIn[4];
	bool pass[4];
};

__device__ __forceinline__ bool decide_slot(const dev::Ray& r, const float4 lo, const float4 hi,
                                            float tCurrMax, float& tIn)
{
	float tOut;
	dev::slab_fast(r, lo.x, lo.y, lo.z, hi.x, hi.y, hi.z, tIn, tOut);
	return (tOut >= tIn) && tOut > r.tMin && tIn < tCurrMax;
}

__device__ __forceinline__ WideVisit decide_wide(const dev::Ray& r, const WideWords& n, float tCurrMax)
{
	WideVisit v;
#pragma unroll
	for (int i = 0; i < 4; i++)
		v.pass[i] = decide_slot(r, n.w[2 * i], n.w[2 * i + 1], tCurrMax, v.tIn[i]);
	return v;
}

// The same of rays whose slab values may be NaN.
__device__ __forceinline__ WideVisit decide_wide_nan(const dev::Ray& r, const WideWords& n, float tCurrMax)
{
	WideVisit v;
#pragma unroll
	for (int i = 0; i < 4; i++) {
		const float4 lo = n.w[2 * i], hi = n.w[2 * i + 1];
		float tOut;
		dev::slab(r, lo.x, lo.y, lo.z, hi.x, hi.y, hi.z, v.tIn[i], tOut);
		v.pass[i] = (tOut >= v.tIn[i]) && tOut > r.tMin && v.tIn[i] < tCurrMax;
	}
	return v;
}

// One triangle, with the fast reciprocal: true iff castRay's test passes; t, u, v are its outputs.
__device__ __forceinline__ bool triangle_fast(const dev::Ray& r, const float4 p0, const float4 e1,
                                              const float4 e2, float& t, float& u, float& v)
{
	const dev::TriDet d = dev::tri_det(r, e1, e2);
	float f = dev::recip_newton(d.a);
	if (!dev::recip_newton_ok(d.a)) f = 1.0f / d.a;
	return dev::tri_finish(r, d, f, p0, e1, e2, t, u, v);
}

// The triangles of a leaf from `first` to its end marker (p0.w < 0, BVHTraversal.hpp:78-93).
__device__ __forceinline__ void closest_leaf_marked(const dev::Ray& r, const float4* __restrict__ tris,
                                                    uint32_t first, Closest& c)
{
	for (uint32_t j = first;; j++) {
		const float4* p = tris + 3u * size_t(j);
		const float4 p0 = p[0], e1 = p[1], e2 = p[2];
		float t, u, v;
		const bool acc = triangle_fast(r, p0, e1, e2, t, u, v) && t < c.t && r.tMin <= t && t <= r.tMax;
		c.tri = acc ? j : c.tri;
		c.t = acc ? t : c.t;
		c.u = acc ? u : c.u;
		c.v = acc ? v : c.v;
		if (p0.w < 0.0f) break;
	}
}

__device__ __forceinline__ bool anyhit_leaf_marked(const dev::Ray& r, const float4* __restrict__ tris,
                                                   uint32_t first)
{
	for (uint32_t j = first;; j++) {
		const float4* p = tris + 3u * size_t(j);
		const float4 p0 = p[0];
		float t, u, v;
		if (triangle_fast(r, p0, p[1], p[2], t, u, v) && r.tMin <= t && t < r.tMax) return true;
		if (p0.w < 0.0f) return false;
	}
}

// castRay of one NaN-free ray over the wide nodes into `c` (the miss result on entry); any hit:
// returns whether a triangle was hit, in any order, and leaves `c` alone. A leaf that a node leaves
// as its next slot is tested in the same iteration.
template <bool kAnyHit, class Stack>
__device__ __forceinline__ bool wide_one(const float4* __restrict__ wide,
                                         const float4* __restrict__ tris, const dev::Ray& r,
                                         Closest& c, Stack& st)
{
	uint32_t ref = 0u;
	float tIn = -INFINITY;
	int sp = 0;
	while (true) {
		bool have = true;
		float lim = kAnyHit ? r.tMax : dev::min_first(r.tMax, c.t);
		if (!(ref & kWideLeaf)) {
			const WideWords n = load_wide(wide, ref);
			const WideVisit v = decide_wide(r, n, lim);
			const uint32_t refs[4] = {__float_as_uint(n.w[0].w), __float_as_uint(n.w[2].w),
			                          __float_as_uint(n.w[4].w), __float_as_uint(n.w[6].w)};
			// Last slot first, so that the first passing slot is what remains to be taken. A leaf
			// pair stays one only if both leaves pass.
			have = false;
#pragma unroll
			for (int i = 3; i >= 0; i--) {
				if (v.pass[i]) {
					if (have) st.put2(sp++, ref, tIn);
					ref = refs[i];
					if (!kAnyHit && i < 3 && !v.pass[i + 1]) ref &= ~kWidePair;
					tIn = v.tIn[i];
					have = true;
				}
			}
		}
		if (have && (ref & kWideLeaf)) {
			have = false;
			const uint32_t first = ref & kWideIndex;
			if (kAnyHit) {
				if (anyhit_leaf_marked(r, tris, first)) return true;
			} else if (tIn < lim) {
				if (ref & kWidePair) {
					// The sibling leaf (the top entry) is decided now too.
					uint32_t sib;
					float sIn;
					st.get2(sp - 1, sib, sIn);
					st.put2(sp - 1, sib, sIn < lim ? -INFINITY : INFINITY);
				}
				closest_leaf_marked(r, tris, first, c);
				lim = dev::min_first(r.tMax, c.t);
			}
		}
		while (!have) {
			if (sp == 0) return false;
			st.get2(--sp, ref, tIn);
			have = kAnyHit || tIn < lim;
		}
	}
}

// castRay of any ray: over the wide nodes where the scene has them (wide != nullptr) and the ray
// is NaN-free, else over the binary ones.
template <class Stack>
__device__ __forceinline__ void closest_any(const float4* __restrict__ wide,
                                            const float4* __restrict__ nodes,
                                            const float4* __restrict__ tris, const dev::Ray& r,
                                            Closest& c, Stack& st)
{
	Counts none;
	if (wide && r.nanFree)
		wide_one<false>(wide, tris, r, c, st);
	else
		closest_one<false>(nodes, tris, r, c, none, st);
}
template <class Stack>
__device__ __forceinline__ bool anyhit_any(const float4* __restrict__ wide,
                                           const float4* __restrict__ nodes,
                                           const float4* __restrict__ tris, const dev::Ray& r,
                                           Stack& st)
{
	Counts none;
	Closest c;
	if (wide && r.nanFree) return wide_one<true>(wide, tris, r, c, st);
	return anyhit_one<false>(nodes, tris, r, none, st);
}

// The ray of this lane; false if it has none. Counting casts give a wave `perWave` rays (<= 64): a wave takes
// as long as its rays' different steps together, and callers count few rays (1,000 camera rays on 1,004,000
// triangles, the whole call: 580 us with 64 rays a wave, 180 with one).
template <bool kCount>
__device__ __forceinline__ bool simple_ray(uint32_t n, uint32_t perWave, uint32_t& i)
{
	i = blockIdx.x * blockDim.x + threadIdx.x;
	if (kCount) {
		const uint32_t lane = i & 63u;
		i = (i >> 6) * perWave + lane;
		if (lane >= perWave) return false;
	}
	return i < n;
}

// kCount: castDebugRay's counters, which count binary nodes, so every ray walks those.
template <bool kCount>
__global__ __launch_bounds__(kBlock) void k_closest_simple(
	const float4* __restrict__ wide, const float4* __restrict__ nodes,
	const float4* __restrict__ tris, const float4* __restrict__ rays, uint4* __restrict__ hits,
	uint32_t n, uint32_t perWave, unsigned long long* __restrict__ counters)
{
	__shared__ uint32_t stackLds[kSimpleLds * kBlock];
	uint32_t i;
	if (!simple_ray<kCount>(n, perWave, i)) return;
	const dev::Ray r = dev::make_ray(rays[2 * size_t(i)], rays[2 * size_t(i) + 1]);
	Closest c = {kInvalid, FLT_MAX, FLT_MAX, FLT_MAX};
	Counts k;
	ColumnStack<kSimpleLds> st;
	st.col = stackLds + threadIdx.x;
	if (kCount)
		closest_one<true>(nodes, tris, r, c, k, st);
	else
		closest_any(wide, nodes, tris, r, c, st);
	hits[i] = make_uint4(c.tri, __float_as_uint(c.t), __float_as_uint(c.u), __float_as_uint(c.v));
	if (kCount) add_counts(counters, k);
}

template <bool kCount>
__global__ __launch_bounds__(kBlock) void k_anyhit_simple(
	const float4* __restrict__ wide, const float4* __restrict__ nodes,
	const float4* __restrict__ tris, const float4* __restrict__ rays,
	uint8_t* __restrict__ inLight, uint32_t n, uint32_t perWave,
	unsigned long long* __restrict__ counters)
{
	__shared__ uint32_t stackLds[kSimpleLds * kBlock];
	uint32_t i;
	if (!simple_ray<kCount>(n, perWave, i)) return;
	const dev::Ray r = dev::make_ray(rays[2 * size_t(i)], rays[2 * size_t(i) + 1]);
	Counts k;
	ColumnStack<kSimpleLds> st;
	st.col = stackLds + threadIdx.x;
	const bool occluded =
		kCount ? anyhit_one<true>(nodes, tris, r, k, st) : anyhit_any(wide, nodes, tris, r, st);
	inLight[i] = occluded ? 0 : 1;
	if (kCount) add_counts(counters, k);
}

// Visit decision of both children of a binary node (BVHTraversal.hpp:59-64; any-hit: tMax).
__device__ __forceinline__ void decide(const dev::Ray& r, const NodeWords& nd, float tCurrMax,
                                       bool& visitL, bool& visitR)
{
	float inL, outL, inR, outR;
	dev::slab(r, nd.w0.x, nd.w0.y, nd.w0.z, nd.w0.w, nd.w1.x, nd.w1.y, inL, outL);
	dev::slab(r, nd.w1.z, nd.w1.w, nd.w2.x, nd.w2.y, nd.w2.z, nd.w2.w, inR, outR);
	visitL = (outL >= inL) && outL > r.tMin && inL < tCurrMax;
	visitR = (outR >= inR) && outR > r.tMin && inR < tCurrMax;
}

// ---- packet traversal (coherent rays) ------------------------------------------------------------
//
// For coherent rays -- camera rays in 8x8-tile order, shadow rays towards one light -- a wave traces
// 64 consecutive rays together over one shared stack of (node, lane mask) entries. Each node is
// loaded once for the wave (every lane reads the same address, a scalar load); each lane decides the
// boxes with its own ray and closest hit, and tests a visited leaf's triangles only where it decided
// to. A lane takes part only in the entries it pushed, and per lane their order is castRay's
// (BVHTraversal.hpp:37-128), so its hits are too. The wave expands the union of its lanes' nodes,
// which for coherent rays is close to one ray's, and every step does the same kind of work. Stack
// entry e lives in lane e % 64 of a few registers.
//
// A step is bound by the instructions that one wave can issue (loading the next node before the leaves
// are tested gains nothing) and the launch by its longest packets (2 waves per SIMD in flight on
// average), so packets of NaN-free rays walk the four-wide nodes: half the steps, for twice the box
// tests each. 2,073,600 tiled camera rays on 1,004,000 triangles, generation included: 0.522 ms with
// binary nodes and IEEE divisions, 0.472 ms with wide nodes and the fast reciprocal. Packets whose rays
// part do not stay packets: see k_packet.

constexpr uint32_t kPacketBlock = 256;
// A packet ends after kPacketSteps steps that fewer than kPacketLanes of its rays take part in, and its
// rays go on one per lane (k_packet).
constexpr int kPacketSteps = 8, kPacketLanes = 24;

__device__ __forceinline__ uint32_t lane_get(uint32_t v, int l)
{
	return uint32_t(__builtin_amdgcn_readlane(int(v), l));
}
// v_writelane_b32 (clang has no builtin for this intrinsic).
extern "C" __device__ int amdgcn_writelane(int v, int l, int old) __asm("llvm.amdgcn.writelane.i32");
__device__ __forceinline__ uint32_t lane_set(uint32_t old, uint32_t v, int l)
{
	return uint32_t(amdgcn_writelane(int(v), l, int(old)));
}
__device__ __forceinline__ uint32_t uniform(uint32_t v)
{
	return uint32_t(__builtin_amdgcn_readfirstlane(int(v)));
}

// The binary nodes, for packets with a ray whose slab values may be NaN and for scenes without
// wide nodes. Both child boxes are decided before either child is used, a visited leaf's triangles
// are tested at once, left child first, and inner children are pushed left then right. The stack
// holds at most one pending left child per level (64, checked at upload).
template <bool kAnyHit>
__device__ __forceinline__ void packet_binary(const float4* __restrict__ nodes,
                                              const float4* __restrict__ tris, const dev::Ray& r,
                                              bool active, Closest& c, bool& occluded)
{
	const uint32_t lane = __lane_id();
	Counts none;
	uint32_t sN0 = 0u, sL0 = 0u, sH0 = 0u, sN1 = 0u, sL1 = 0u, sH1 = 0u;
	int sp = 0;
	auto push = [&](uint32_t node, uint64_t m) {
		const uint32_t lo = uint32_t(m), hi = uint32_t(m >> 32);
		const bool low = sp < 64;
		const bool mine = int(lane) == (low ? sp : sp - 64);
		sN0 = low && mine ? node : sN0;
		sL0 = low && mine ? lo : sL0;
		sH0 = low && mine ? hi : sH0;
		sN1 = !low && mine ? node : sN1;
		sL1 = !low && mine ? lo : sL1;
		sH1 = !low && mine ? hi : sH1;
		sp++;
	};
	uint32_t cur = 0u;
	uint64_t mask = __ballot(active);
	while (true) {
		const bool in = ((mask >> lane) & 1ull) != 0;
		NodeWords nd = load_node(nodes, cur);
		const int32_t lRaw = __builtin_amdgcn_readfirstlane(nd.w3.x);
		const int32_t rRaw = __builtin_amdgcn_readfirstlane(nd.w3.y);
		const int32_t lCnt = __builtin_amdgcn_readfirstlane(nd.w3.z);
		const int32_t rCnt = __builtin_amdgcn_readfirstlane(nd.w3.w);
		const float tCurrMax = kAnyHit ? r.tMax : dev::min_first(r.tMax, c.t);
		bool visitL, visitR;
		decide(r, nd, tCurrMax, visitL, visitR);
		visitL = visitL && in;
		visitR = visitR && in;
		uint64_t pushL = 0ull, pushR = 0ull;
		if (lCnt == 0)
			pushL = __ballot(visitL);
		else if (visitL)
			kAnyHit ? void(occluded = anyhit_leaf(r, tris, child_index(lRaw), lCnt))
			        : closest_leaf<false>(r, tris, child_index(lRaw), lCnt, c, none);
		if (rCnt == 0)
			pushR = __ballot(visitR && !(kAnyHit && occluded));
		else if (visitR && !(kAnyHit && occluded))
			kAnyHit ? void(occluded = anyhit_leaf(r, tris, child_index(rRaw), rCnt))
			        : closest_leaf<false>(r, tris, child_index(rRaw), rCnt, c, none);
		const uint64_t done = kAnyHit ? __ballot(occluded) : 0ull;
		pushL &= ~done;
		if (pushL != 0ull && sp < 128) push(child_index(lRaw), pushL);
		if (pushR != 0ull && sp < 128) push(child_index(rRaw), pushR);
		// Next: the top entry that still has lanes (any hit: lanes without an occluder).
		mask = 0ull;
		while (mask == 0ull && sp > 0) {
			sp--;
			const bool low = sp < 64;
			const int l = low ? sp : sp - 64;
			cur = lane_get(low ? sN0 : sN1, l);
			const uint32_t lo = lane_get(low ? sL0 : sL1, l);
			const uint32_t hi = lane_get(low ? sH0 : sH1, l);
			mask = ((uint64_t(hi) << 32) | lo) & ~done;
		}
		if (mask == 0ull) break;
	}
}

// A leaf's triangles (uniform addresses: scalar loads) for the lanes in `on`.
template <bool kAnyHit>
__device__ __forceinline__ void packet_leaf(const float4* __restrict__ tris, uint32_t first,
                                            const dev::Ray& r, bool on, Closest& c, bool& occluded)
{
	for (uint32_t j = first;; j++) {
		const float4* p = tris + 3u * size_t(j);
		const float4 p0 = p[0], e1 = p[1], e2 = p[2];
		const dev::TriDet d = dev::tri_det(r, e1, e2);
		float f = dev::recip_newton(d.a);
		if (__ballot(on && !dev::recip_newton_ok(d.a)) != 0ull) f = 1.0f / d.a;
		float t, u, v;
		const bool hit = dev::tri_finish(r, d, f, p0, e1, e2, t, u, v);
		if (kAnyHit) {
			occluded = occluded || (on && hit && r.tMin <= t && t < r.tMax);
		} else {
			const bool acc = on && hit && t < c.t && r.tMin <= t && t <= r.tMax;
			c.tri = acc ? j : c.tri;
			c.t = acc ? t : c.t;
			c.u = acc ? u : c.u;
			c.v = acc ? v : c.v;
		}
		if (p0.w < 0.0f) break;
	}
}

// The wide nodes. Slots are taken in order: leaf slots are tested at once as long as no inner slot
// comes before them; the first inner slot is the next node, and the slots after it are pushed. A
// leaf slot that was pushed is decided again when it is taken, from its box in the node (closest
// hit; entry word 1 names node and slot). Any hit does not depend on order: all its leaf slots are
// tested at once.
template <bool kAnyHit, bool kLoose, class Leave>
__device__ __forceinline__ void packet_wide(const float4* __restrict__ wide,
                                            const float4* __restrict__ tris, const dev::Ray& r,
                                            bool active, Closest& c, bool& occluded,
                                            Leave leave)
{
	const uint32_t lane = __lane_id();
	uint32_t sR = 0u, sB = 0u, sL = 0u, sH = 0u;  // reference, node and slot, mask
	int sp = 0, steps = 0;
	uint32_t cur = 0u;
	uint64_t mask = __ballot(active);
	while (true) {
		const bool in = ((mask >> lane) & 1ull) != 0;
		const WideWords n = load_wide(wide, kLoose ? cur & kWideIndex : cur);
		const float lim = kAnyHit ? r.tMax : dev::min_first(r.tMax, c.t);
		WideVisit v = decide_wide(r, n, lim);
		const uint32_t refs[4] = {
			uniform(__float_as_uint(n.w[0].w)), uniform(__float_as_uint(n.w[2].w)),
			uniform(__float_as_uint(n.w[4].w)), uniform(__float_as_uint(n.w[6].w))};
		uint64_t m[4];
#pragma unroll
		for (int i = 0; i < 4; i++) {
			v.pass[i] = v.pass[i] && in;
			m[i] = __ballot(v.pass[i]);
		}
		bool sibling[4] = {false, false, false, false};  // a pair's second leaf: decided with the first
		int next = -1;
#pragma unroll
		for (int i = 0; i < 4; i++) {
			if (m[i] == 0ull) continue;
			if (!(refs[i] & kWideLeaf)) {
				if (next < 0) next = i;
				continue;
			}
			if (!kAnyHit && next >= 0) continue;  // pushed below
			if (kAnyHit) {
				packet_leaf<true>(tris, refs[i] & kWideIndex, r, v.pass[i] && !occluded, c, occluded);
			} else {
				const float cm = dev::min_first(r.tMax, c.t);
				const bool on = v.pass[i] && (sibling[i] || v.tIn[i] < cm);
				if (i < 3 && (refs[i] & kWidePair)) {
					v.pass[i + 1] = v.pass[i + 1] && v.tIn[i + 1] < cm;
					sibling[i + 1] = true;
				}
				packet_leaf<false>(tris, refs[i] & kWideIndex, r, on, c, occluded);
			}
		}
		const uint64_t done = kAnyHit ? __ballot(occluded) : 0ull;
#pragma unroll
		for (int i = 3; i >= 1; i--) {
			const uint64_t mi = m[i] & ~done;
			if (i <= next || next < 0 || mi == 0ull) continue;
			if (kAnyHit && (refs[i] & kWideLeaf)) continue;
			uint32_t ref = refs[i];
			if (i == 3 || m[i < 3 ? i + 1 : 3] == 0ull) ref &= ~kWidePair;
			sR = lane_set(sR, ref, sp);
			sB = lane_set(sB, cur * 4u + uint32_t(i), sp);
			sL = lane_set(sL, uint32_t(mi), sp);
			sH = lane_set(sH, uint32_t(mi >> 32), sp);
			sp++;
		}
		mask = 0ull;
		if (next >= 0) {
#pragma unroll
			for (int i = 0; i < 4; i++)
				if (next == i) {
					mask = m[i] & ~done;
					cur = refs[i];
				}
		}
		while (mask == 0ull && sp > 0) {
			sp--;
			const uint32_t ref = lane_get(sR, sp);
			const uint64_t me = ((uint64_t(lane_get(sH, sp)) << 32) | lane_get(sL, sp)) & ~done;
			if (kAnyHit || !(ref & kWideLeaf)) {
				mask = me;
				cur = ref;
				continue;
			}
			auto decided = [&](int e, uint64_t who) {
				const uint32_t at = lane_get(sB, e);
				const float4* b = wide + 2u * size_t(at);
				float tIn;
				const bool pass = decide_slot(r, b[0], b[1], dev::min_first(r.tMax, c.t), tIn);
				return ((who >> lane) & 1ull) != 0 && pass;
			};
			const bool on = decided(sp, me);
			bool on2 = false;
			uint32_t ref2 = 0u;
			if (ref & kWidePair) {
				sp--;
				ref2 = lane_get(sR, sp);
				on2 = decided(sp, (uint64_t(lane_get(sH, sp)) << 32) | lane_get(sL, sp));
			}
			if (__ballot(on) != 0ull) packet_leaf<false>(tris, ref & kWideIndex, r, on, c, occluded);
			if (__ballot(on2) != 0ull) packet_leaf<false>(tris, ref2 & kWideIndex, r, on2, c, occluded);
		}
		if (mask == 0ull) break;
		// (In loose trees packets do not part: lanes by themselves would need the slow steps of LaneWalk.)
		if (!kLoose && __popcll(mask) < kPacketLanes && ++steps == kPacketSteps) {
			// Each lane goes on by itself with its part of the stack, bottom entry first, and the node.
			int n = 0;
			for (int e = 0; e < sp; e++) {
				const uint64_t who = (uint64_t(lane_get(sH, e)) << 32) | lane_get(sL, e);
				const uint64_t below = e > 0 ? (uint64_t(lane_get(sH, e - 1)) << 32) | lane_get(sL, e - 1) : 0ull;
				uint32_t ref = lane_get(sR, e);
				float tIn = -INFINITY;
				if (!kAnyHit && (ref & kWideLeaf)) {
					const float4* b = wide + 2u * size_t(lane_get(sB, e));
					decide_slot(r, b[0], b[1], 0.0f, tIn);
				}
				if (((below >> lane) & 1ull) == 0ull) ref &= ~kWidePair;
				if (((who & ~done) >> lane) & 1ull) leave.push(n++, ref, tIn);
			}
			leave(n, cur, ((mask >> lane) & 1ull) != 0);
			break;
		}
	}
}

__device__ __forceinline__ uint32_t find_batch(const uint32_t* offsets, uint32_t numBatches,
                                               uint32_t g)
{
	// largest b with offsets[b] <= g (offsets[0] = 0, offsets[numBatches] = total > g)
	uint32_t lo = 0, hi = numBatches;
	while (hi - lo > 1) {
		const uint32_t mid = (lo + hi) >> 1;
		if (offsets[mid] <= g)
			lo = mid;
		else
			hi = mid;
	}
	return lo;
}

// ---- four lanes per ray ---------------------------------------------------------------------------
//
// Single casts of incoherent rays (k_quad). Four lanes trace a ray: one box of a wide node each, or one
// triangle of a leaf each, combined across the four (DPP and 4 bits of a ballot). A wave holds 16
// rays, its stacks are in LDS, and seven of them run on a SIMD. An iteration loads and consumes a
// leaf and the node to be taken after it together: the node's slots are decided after the leaf's
// triangles, with its entry distance compared again, so the order is castRay's. See wide_nodes.hpp
// for why the hits are too.
//
// With one lane per ray and binary nodes (64 rays a wave, two or three waves per SIMD, a software
// pipeline and a one-ray-per-wave mode for a wave's last rays) a launch was bound by its chains of
// steps: 25 a bounce ray on 1,004,000 triangles, half of the time spent on the last 1% of the rays,
// and 15,600 fetches from and 2,048 retirements to one address at 10 ns each. Before and now:
//   998,029 bounce rays, closest hit   0.567 ms   0.428 ms
//   their 998,029 shadow rays, any hit  0.254 ms   0.119 ms
//   65,536 random rays, 100,000 random triangles  0.243 ms   0.120 ms
// Many rays at once are bound by VALU issue (a wave instruction serves 16 rays), the rest by the
// chain of the costliest rays: about 450 iterations of 0.9 us, the time a wave takes to issue one. So
// instructions count: flags between bytes, selects and compares to make a ballot, minima that first
// canonicalise, a multiplication by 48 and the binary walk's checks cost 5% (bounce 0.467 -> 0.442).
// Selects in place of the branches of what comes next cost more than they save (0.488).

constexpr uint32_t kQuadBlock = 512;  // largest block of the persistent kernels
constexpr uint32_t kLaneBlock = 1024;  // (of fused launches)
constexpr uint32_t kLdsBytes = 160u * 1024u;  // of a CU
constexpr uint32_t kStageWords = 512u + 64u;  // of a wave: a window's rays and their indices
constexpr uint32_t kQuadWavesPerSimd = 7;  // (72 registers)
static_assert(kCastRaysPerCu == kQuadWavesPerSimd * 4u * 16u, "rays in flight per CU of a single cast");

// Stacks of a wave: kCols columns of kRows entries (8 B) in LDS, with three rows below the bottom, so
// that the top three can be read at any depth. Deeper entries spill to memory, kSpillEntries a
// column, one after another.
constexpr int kQuadRows = 20;  // (pending stacks of 20 are rare)
constexpr int kLaneRows = 10;  // (8.5 KB a wave with 2 KB of rays: 16 waves per CU beside the batch tables)
constexpr uint32_t kSpillEntries = kSpillWordsPerRay / 2u;
static_assert(kLaneRows + int(kSpillEntries) >= kMaxPending, "stack entries of a ray");
static_assert(kQuadRows + int(kSpillEntries) >= kMaxPending, "stack entries of a ray");

template <int kRows, uint32_t kCols>
__host__ __device__ constexpr uint32_t wave_stack_entries() { return (uint32_t(kRows) + 3u) * kCols; }

// LDS entry of the bottom of column `col` of the block's wave `wave`.
template <int kRows, uint32_t kCols>
__device__ __forceinline__ uint32_t stack_base(uint32_t wave, uint32_t col)
{
	return wave * wave_stack_entries<kRows, kCols>() + 3u * kCols + col;
}
template <int kRows, uint32_t kCols>
__device__ __forceinline__ GlobalU2* spill_entry(U32x2* spill, uint32_t base, int at)
{
	const uint32_t b = base - 3u * kCols, wave = b / wave_stack_entries<kRows, kCols>();
	const uint32_t col = b - wave * wave_stack_entries<kRows, kCols>();
	const size_t column = size_t(blockIdx.x * (blockDim.x / 64u) + wave) * kCols + col;
	return (GlobalU2*)(spill) + column * kSpillEntries + uint32_t(at - kRows);
}

// Ray counters of a launch, one 128-B line each: 8 that hand out windows, 8 + 1 that count blocks
// as they end.
constexpr uint32_t kCounters = 8;
constexpr uint32_t kCounterStride = 32;

__host__ __device__ __forceinline__ uint32_t quad_lds_words(uint32_t waves)
{
	return waves * (2u * wave_stack_entries<kQuadRows, 16u>() + kStageWords);
}

// (__ballot takes an int: a select and a compare more.)
__device__ __forceinline__ uint64_t ballot(bool p) { return __builtin_amdgcn_ballot_w64(p); }

// v of another lane of the quad (DPP quad_perm).
template <int kCtrl>
__device__ __forceinline__ float quad_perm(float v)
{
	return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), kCtrl, 0xF, 0xF, true));
}

// 1/a: the fast reciprocal, or the division where a lane's value is out of its range.
__device__ __forceinline__ float recip_wave(float a)
{
	float f = dev::recip_newton(a);
	if (__builtin_expect(ballot(!dev::recip_newton_ok(a)) != 0ull, 0)) f = 1.0f / a;
	return f;
}

// Sets r up from its record. A direction component outside the fast reciprocal's range (zero among them)
// takes the division and slab, with which NaN slab values come out as castRay's; an origin beyond 2^126
// the binary nodes (wide_nodes.hpp). Rays with a zero component are ordinary ones (probes, a sun
// overhead): on the binary nodes 1,048,576 of them straight up took 0.91 ms, on the wide ones 0.52 ms.
__device__ __forceinline__ uint32_t quad_ray(const float4 a, const float4 b, uint32_t sceneWith, dev::Ray& r)
{
	r.ox = a.x, r.oy = a.y, r.oz = a.z, r.tMin = a.w;
	r.dx = b.x, r.dy = b.y, r.dz = b.z, r.tMax = b.w;
	r.ix = dev::recip_newton(b.x);
	r.iy = dev::recip_newton(b.y);
	r.iz = dev::recip_newton(b.z);
	auto within = [](float x) { return fabsf(x) >= 0x1p-126f && fabsf(x) < 0x1p126f; };
	const bool near = fabsf(a.x) <= 0x1p126f && fabsf(a.y) <= 0x1p126f && fabsf(a.z) <= 0x1p126f;
	const uint32_t with = !near ? kBinary : within(b.x) && within(b.y) && within(b.z) ? kFast : kSlab;
	return with > sceneWith ? with : sceneWith;
}
__device__ __forceinline__ void divide(const float4 b, dev::Ray& r)
{
	r.ix = 1.0f / b.x;
	r.iy = 1.0f / b.y;
	r.iz = 1.0f / b.z;
}

// What a launch traces. Single casts: one scene, ray array and output. Batches: per ray through its
// batch's descriptor (offsets in LDS).
struct QuadArgs {
	const float4* wide;         // (tris where the scene has no wide nodes)
	const float4* nodes;
	const float4* tris;
	const float4* rays;
	void* out;                  // uint4 hits or uint8_t inLight flags
	uint32_t n;                 // rays of the launch
	uint32_t with;              // what the scene's rays are decided with at least
	uint32_t window;            // rays a wave claims at a time (at most 64)
	uint32_t refill;            // idle rays of a wave before it takes new ones
	uint32_t* work;             // kCounters window counters, then the retirement counters
	U32x2* spill;
	unsigned long long* clock;  // completion clock per ray, and the earliest block start in word n
	const BatchDesc* descs;
	const uint32_t* offsets;    // LDS
	uint32_t numBatches;
	unsigned long long* blockFinish;  // LDS, per batch (completion tracking)
	uint32_t* blockDone;              // LDS, per batch
};

// One lane's state of its ray.
struct Quad {
	dev::Ray r;
	uint32_t ray = kInvalid;     // index in the launch
	uint32_t node = kInvalid;    // node to expand next, entered at nodeIn
	float nodeIn = 0.0f;
	uint32_t tri = 0u, triNext = 0u;  // triNext: lane 0's next one if the leaf goes on
	uint32_t skip = 0u;          // lanes whose end marker is the first leaf's of a pair
	int sp = 0;
	uint32_t base = 0u;          // its stack column: LDS entry of the bottom row
	float best = FLT_MAX, u = FLT_MAX, v = FLT_MAX;  // closest hit; u, v, hit in the lane it is `mine`
	uint32_t hit = kInvalid;
	// (4-byte flags: between the others' bytes, hit was kept in four registers.)
	uint32_t mine = 0u;          // holds the closest hit
	uint32_t with = kFast;       // kFast, kSlab or kBinary
	uint32_t any = 0u;
	bool leaf = false;           // triangles to test before node: this lane's is tri
	// batches
	const float4* wide = nullptr;
	const float4* tris = nullptr;
	uint32_t batch = 0u;
};

// Writes a ray's result: its closest hit, or 0 if occluded and 1 if not.
template <bool kBatch, bool kTrack, bool kClock>
__device__ __forceinline__ void quad_result(const QuadArgs& P, uint32_t ray, uint32_t batch,
                                            const Closest& c, bool any, bool occluded)
{
	void* out = P.out;
	uint32_t at = ray;
	if (kBatch) {
		out = P.descs[batch].out;
		at = ray - P.offsets[batch];
	}
	const U32x4 hit = {c.tri, __float_as_uint(c.t), __float_as_uint(c.u), __float_as_uint(c.v)};
	if (any)
		((GlobalU8*)(out))[at] = occluded ? 0 : 1;
	else
		((GlobalU4*)(out))[at] = hit;
	if (kClock) P.clock[ray] = wall_clock64();
	if (kTrack) {
		atomicAdd(&P.blockDone[batch], 1u);
		atomicMax(&P.blockFinish[batch], wall_clock64());
	}
}

// Rays [next, end) claimed by a wave (uniform). Its first window is its own, so that no launch starts
// with all waves at one counter; the others come from a counter shared by every eighth block,
// interleaved, so that costly regions of a ray array are spread over all of them.
struct RayWindows {
	uint32_t next = 0u, end = 0u;
	uint32_t* counter;

	__device__ __forceinline__ RayWindows(const QuadArgs& P, uint32_t waveInBlock)
		: counter(P.work + blockIdx.x % kCounters * kCounterStride)
	{
		set(P, uint64_t(blockIdx.x * (blockDim.x / 64u) + waveInBlock) * P.window);
	}
	__device__ __forceinline__ void set(const QuadArgs& P, uint64_t first)
	{
		if (first >= P.n) return;
		next = uint32_t(first);
		end = P.n - next < P.window ? P.n : next + P.window;
	}
	// The next window; false if there is none.
	__device__ __forceinline__ bool claim(const QuadArgs& P)
	{
		const uint32_t waves = gridDim.x * (blockDim.x / 64u);
		const uint32_t counters = gridDim.x < kCounters ? gridDim.x : kCounters;
		uint32_t b = 0u;
		if (__lane_id() == 0u) b = atomicAdd(counter, 1u);
		const uint64_t first =
			(uint64_t(waves) + uint64_t(uniform(b)) * counters + blockIdx.x % kCounters) * P.window;
		if (first >= P.n) return false;
		set(P, first);
		return true;
	}
};

// kAny: the launch's any-hit rays: 0 none, 1 all, 2 per batch. kBig: a scene's triangles or wide
// nodes take 4 GB or more, so 32-bit offsets into them do not do.
template <int kAny, bool kBatch, bool kTrack, bool kClock, bool kBig, int kRows, uint32_t kCols>
struct QuadTracer {
	const QuadArgs& P;
	LdsU2* stacks;       // the block's stack columns
	uint32_t lane, l;
	bool slow = false;  // (uniform) a ray of the wave may be decided with slab
	Quad q;

	__device__ __forceinline__ bool isAny() const { return kAny == 1 || (kAny == 2 && q.any); }
	// The quad's four bits of a ballot. (Ballots of single comparisons, combined as masks: of a
	// combined condition, a ballot takes a select and a compare more.)
	__device__ __forceinline__ uint32_t nibble(uint64_t b) const { return uint32_t(b >> (lane & 60u)) & 15u; }
	// Entry `at` of the stack column: in LDS, or spilled (at >= kRows).
	__device__ __forceinline__ LdsU2* row(int at) const { return stacks + (q.base + uint32_t(at) * kCols); }
	__device__ __forceinline__ GlobalU2* spilled(int at) const
	{
		return spill_entry<kRows, kCols>(P.spill, q.base, at);
	}
	__device__ __forceinline__ U32x2 entry(int at) const
	{
		U32x2 e = {0u, 0u};
		if (at < kRows) e = *row(at);
		else e = *spilled(at);
		return e;
	}

	// Sets this quad up for ray `ray` with the record (a, b).
	__device__ __forceinline__ void set(uint32_t ray, const float4 a, const float4 b, uint32_t sceneWith)
	{
		q.with = quad_ray(a, b, sceneWith, q.r);
		if (__builtin_expect(ballot(q.with != kFast) != 0ull, 0)) divide(b, q.r);
		q.ray = ray;
	}
	// Starts a ray of a single cast.
	__device__ __forceinline__ void start(uint32_t ray, const float4 a, const float4 b)
	{
		set(ray, a, b, P.with);
		q.node = 0u;
		q.nodeIn = -INFINITY;
		q.leaf = false;
		q.sp = 0;
		q.best = q.u = q.v = FLT_MAX;
		q.hit = kInvalid;
		q.mine = l == 0u;
	}
	// Takes over a ray of a batch that is being traced (its batch is set; its traversal is the caller's).
	__device__ __forceinline__ void take_over(uint32_t ray)
	{
		const uint32_t at = ray - P.offsets[q.batch];
		const BatchDesc d = P.descs[q.batch];
		q.wide = d.wide;
		q.tris = d.tris;
		q.any = d.kind & 1u;
		set(ray, as_global(d.rays)[2 * size_t(at)], as_global(d.rays)[2 * size_t(at) + 1], d.kind >> 1);
	}

	// Expands a binary node: lanes 0 and 1 decide its children as castRay does, and what is visited is
	// pushed in castRay's order (left leaf, right leaf, right subtree, left subtree; decided now).
	__device__ __forceinline__ void expand_binary(float lim)
	{
		const float4* nodes = kBatch ? P.descs[q.batch].nodes : P.nodes;
		const float* f = reinterpret_cast<const float*>(nodes + 4u * size_t(q.node));
		const float* box = f + 6u * (l & 1u);
		const int32_t child = __float_as_int(f[12u + (l & 1u)]);
		const bool isLeaf = __float_as_int(f[14u + (l & 1u)]) != 0;
		float tIn, tOut;
		dev::slab(q.r, box[0], box[1], box[2], box[3], box[4], box[5], tIn, tOut);
		const bool pass = l < 2u && (tOut >= tIn) && tOut > q.r.tMin && tIn < lim;
		const uint32_t m = nibble(ballot(pass));
		const bool leftFirst = (nibble(ballot(pass && isLeaf)) & 1u) != 0u;
		const int at = q.sp + (m == 3u && (l == 0u) == leftFirst ? 1 : 0);
		const U32x2 e = {child_index(child) | (isLeaf ? kWideLeaf : 0u), __float_as_uint(-INFINITY)};
		if (pass) {
			if (at < kRows) *row(at) = e;
			else *spilled(at) = e;
		}
		q.sp += __popc(m);
	}

	// One iteration of the wave's rays.
	__device__ __forceinline__ void step()
	{
		const bool active = q.ray != kInvalid;
		const bool any = isAny();
		const float4* wide = kBatch ? q.wide : P.wide;
		const float4* tris = kBatch ? q.tris : P.tris;
		// Straight-line loads, so that a leaf's and a node's are in flight together (in branches, the
		// compiler waits for the first to test its end marker); quads without one read the array's
		// first line. Offsets in bytes: 48 per triangle, 128 per wide node.
		const uint32_t tri = q.leaf ? q.tri : 0u;
		uint32_t node = q.node != kInvalid ? q.node : 0u;
		if (slow) node = q.with == kBinary ? 0u : node;
		const float4* pl;
		const float4* pn;
		if (kBig) {
			pl = tris + 3u * size_t(tri);
			pn = wide + 8u * size_t(node & kWideIndex) + 2u * l;
		} else {
			uint32_t tri3;
			asm("v_lshl_add_u32 %0, %1, 1, %1" : "=v"(tri3) : "v"(tri));  // (a 32-bit multiply takes four times as long)
			pl = reinterpret_cast<const float4*>(reinterpret_cast<const char*>(tris) + (tri3 << 4));
			// (a kWideLoose in the reference is shifted out)
			pn = reinterpret_cast<const float4*>(reinterpret_cast<const char*>(wide) + ((node << 7) + (l << 5)));
		}
		const float4 p0 = as_global(pl)[0], e1 = as_global(pl)[1], e2 = as_global(pl)[2];
		const float4 lo = as_global(pn)[0], hi = as_global(pn)[1];
		bool more = false, occluded = false;
		if (q.leaf) {
			// The leaf's triangles up to its end marker; candidates are accepted in lane order, which
			// is castRay's: the smallest t, the lowest lane on equal t.
			const uint32_t ends = nibble(ballot(p0.w < 0.0f)) & ~q.skip;
			const bool inLeaf = (ends & ((1u << l) - 1u)) == 0u;
			const dev::TriDet d = dev::tri_det(q.r, e1, e2);
			const float f = recip_wave(d.a);
			float t, u, v;
			const bool hit = dev::tri_finish(q.r, d, f, p0, e1, e2, t, u, v) && inLeaf && q.r.tMin <= t;
			if (kAny != 0) occluded = nibble(ballot(hit) & ballot(t < q.r.tMax)) != 0u && any;
			if (kAny != 1 && !any) {
				const bool cand = hit && t < q.best && t <= q.r.tMax;
				float tm = cand ? t : INFINITY;
				tm = dev::vmin(tm, quad_perm<0xB1>(tm));  // lanes 1 0 3 2
				tm = dev::vmin(tm, quad_perm<0x4E>(tm));  // lanes 2 3 0 1
				const bool least = cand && t == tm;
				const uint32_t win = nibble(ballot(cand) & ballot(t == tm));
				const bool me = least && (win & ((1u << l) - 1u)) == 0u;
				q.best = me ? t : dev::vmin(q.best, tm);  // (its own t: a zero's sign)
				q.mine = win != 0u ? uint32_t(me) : q.mine;
				q.u = me ? u : q.u;
				q.v = me ? v : q.v;
				q.hit = me ? q.tri : q.hit;
			}
			q.leaf = more = ends == 0u;
			q.tri = q.triNext + l;
			q.triNext += 4u;
			q.skip = 0u;
		}
		const float lim = any ? q.r.tMax : dev::min_first(q.r.tMax, q.best);
		float tIn, tOut;
		dev::slab_fast(q.r, lo.x, lo.y, lo.z, hi.x, hi.y, hi.z, tIn, tOut);
		if (__builtin_expect(slow, 0)) {  // (all of it in one branch that fast rays' waves do not take)
			dev::slab(q.r, lo.x, lo.y, lo.z, hi.x, hi.y, hi.z, tIn, tOut);
			if (int32_t(__float_as_uint(lo.w)) >= int32_t(kWideLoose))  // decided now, and not to be again
				tIn = tOut >= tIn && tIn < lim ? -INFINITY : INFINITY;
			if (q.with == kBinary && q.node != kInvalid && !more) {
				expand_binary(lim);
				q.node = kInvalid;
			}
		}
		if (q.node != kInvalid && !more) {
			// The passing slots are pushed, last slot first; a leaf pair stays one only if both pass.
			const bool enters = any || q.nodeIn < lim;
			const bool pass = (tOut >= tIn) && tOut > q.r.tMin && tIn < lim && enters;
			const uint32_t m = nibble(ballot(tOut >= tIn) & ballot(tOut > q.r.tMin) & ballot(tIn < lim) & ballot(enters));
			const uint32_t after = m >> (l + 1u);
			uint32_t ref = __float_as_uint(lo.w);
			ref = (after & 1u) ? ref : ref & ~kWidePair;
			const int at = q.sp + __popc(after);
			const U32x2 e = {ref, __float_as_uint(tIn)};
			if (pass && at < kRows) *row(at) = e;
			if (__builtin_expect(pass && at >= kRows, 0)) *spilled(at) = e;
			q.sp += __popc(m);
			q.node = kInvalid;
		}
		if (!active) return;
		bool end = occluded;
		if (!more && !occluded) {
			// What comes next: the top entry that the closest hit has not overtaken; if it is a leaf,
			// also its sibling (decided now, tested with it if the leaf has at most three
			// triangles) and the entry below, if that is a node.
			U32x2 x1, x2, x3;
			if (__builtin_expect(q.sp <= kRows, 1)) {
				const LdsU2* top = row(q.sp - 3);
				x3 = top[0];
				x2 = top[kCols];
				x1 = top[2u * kCols];
			} else {
				x1 = entry(q.sp - 1);
				x2 = entry(q.sp - 2);
				x3 = entry(q.sp - 3);
			}
			if (!any)
				while (q.sp > 0 && !(__uint_as_float(x1.y) < lim)) {
					q.sp--;
					x1 = x2;
					x2 = x3;
					x3 = entry(q.sp - 3);
				}
			if (q.sp == 0) {
				end = true;
			} else {
				q.sp--;
				if (!(x1.x & kWideLeaf)) {
					q.node = x1.x;
					q.nodeIn = __uint_as_float(x1.y);
				} else {
					const uint32_t first = x1.x & kWideIndex;
					const uint32_t count = (x1.x >> kWideCountShift) & 3u;
					q.leaf = true;
					q.tri = first + l;
					q.triNext = first + 4u;
					q.skip = 0u;
					U32x2 below = x2;
					if (x1.x & kWidePair) {
						const bool both = any || __uint_as_float(x2.y) < lim;
						if (count != 0u) {
							q.sp--;
							below = x3;
							if (both) {
								const uint32_t at = (x2.x & kWideIndex) - count;
								q.tri = l < count ? q.tri : at + l;
								q.triNext = at + 4u;
								q.skip = (1u << count) - 1u;
							}
						} else if (!any) {
							const U32x2 e = {x2.x, __float_as_uint(both ? -INFINITY : INFINITY)};
							if (q.sp <= kRows) *row(q.sp - 1) = e;
							else *spilled(q.sp - 1) = e;
						}
					}
					if (q.sp > 0 && !(below.x & kWideLeaf)) {
						q.node = below.x;
						q.nodeIn = __uint_as_float(below.y);
						q.sp--;
					}
				}
			}
		}
		if (end) {
			const Closest c = {q.hit, q.best, q.u, q.v};
			if (any ? l == 0u : q.mine)
				quad_result<kBatch, kTrack, kClock>(P, q.ray, q.batch, c, any, occluded);
			q.ray = kInvalid;
			q.node = kInvalid;
			q.leaf = false;
		}
	}
};

// A window's rays are loaded when it is claimed, one per lane, and handed out of LDS: a ray that started
// with loads of its own held up the wave's other 15 (with 2 of 16 rays taking new ones at a time, every
// other step). With it 998,029 any-hit shadow rays take 0.122 ms instead of 0.127, bounce rays 0.438
// instead of 0.449. An any-hit ray with an empty interval (what stands for none) is answered there.
template <int kAny, bool kClock, bool kBig>
__device__ __forceinline__ void quad_trace(const QuadArgs& P, uint32_t* lds)
{
	const uint32_t waveInBlock = uniform(threadIdx.x >> 6), blockWaves = blockDim.x / 64u;
	QuadTracer<kAny, false, false, kClock, kBig, kQuadRows, 16u> T{P};
	T.stacks = (LdsU2*)(reinterpret_cast<U32x2*>(lds));
	T.lane = __lane_id();
	T.l = T.lane & 3u;
	T.q.base = stack_base<kQuadRows, 16u>(waveInBlock, T.lane >> 2);
	LdsU1* const area = (LdsU1*)(lds) + blockWaves * 2u * wave_stack_entries<kQuadRows, 16u>() + waveInBlock * kStageWords;
	LdsF4* const staged = (LdsF4*)(area);  // ray records: first words, then second ones
	LdsU1* const index = area + 512u;      // any hit: the rays that they are of
	if (kClock && threadIdx.x == 0u) atomicMin(&P.clock[P.n], wall_clock64());
	RayWindows W(P, waveInBlock);
	uint32_t taken = 0u, count = 0u;  // of the staged rays
	auto stage = [&] {
		const uint32_t ray = W.next + T.lane;
		bool mine = W.next < W.end && ray < W.end;
		F32x4 a = {}, b = {};
		if (mine) {
			GlobalV4* p = (GlobalV4*)(P.rays) + 2u * size_t(ray);
			a = p[0];
			b = p[1];
			if (kAny == 1 && !(a.w < b.w)) {
				quad_result<false, false, kClock>(P, ray, 0u, Closest{}, true, false);
				mine = false;
			}
		}
		const uint64_t all = ballot(mine);
		const uint32_t at = uint32_t(__popcll(all & __lanemask_lt()));
		if (mine) {
			staged[at] = a;
			staged[64u + at] = b;
			if (kAny == 1) index[at] = ray;
		}
		taken = 0u;
		count = uint32_t(__popcll(all));
		__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
		__builtin_amdgcn_wave_barrier();
		__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
	};
	stage();
	while (true) {
		const uint64_t idle = ballot(T.q.ray == kInvalid);
		if (idle != 0ull) {
			if (taken >= count) {
				if (!W.claim(P)) break;
				stage();
				if (count == 0u) continue;
			}
			const uint32_t room = uint32_t(__popcll(idle)) / 4u;
			if (room >= P.refill) {
				const uint32_t at = taken + uint32_t(__popcll(idle & __lanemask_lt())) / 4u;
				if (T.q.ray == kInvalid && at < count) {
					const F32x4 a = staged[at], b = staged[64u + at];
					T.start(kAny == 1 ? index[at] : W.next + at, make_float4(a.x, a.y, a.z, a.w),
					        make_float4(b.x, b.y, b.z, b.w));
				}
				T.slow = ballot(T.q.with != kFast) != 0ull;
				taken += room;
			}
		}
		T.step();
	}

	// The rays are handed out (a loop of its own: its state is only what step() needs).
	while (ballot(T.q.ray != kInvalid) != 0ull) T.step();
	__syncthreads();
}

// ---- one ray per lane, then four lanes per ray -----------------------------------------------------
//
// Fused launches: a wave traces 64 rays, one a lane, and once no rays are left to take and at most 16
// are busy, those four lanes each, on the stack columns that they have. A step of one ray per lane issues fewer instructions a ray (a wave
// instruction serves 64 rays, not 16) but reads 64 lines with each load, takes a leaf and a node in
// steps of their own and is as slow as its costliest lane, so four lanes per ray are the faster way
// for a launch by itself (1,048,576 random rays, 4 waves per SIMD: 0.485 ms against 0.468 ms) and one
// lane is where the device is full: 64 batches of 4.4 million rays on two scenes take 1.48 ms (2.3 ms
// four lanes each; 1.79 ms with the binary nodes). There the texture data path is busy 83% of
// the time, the VALUs 70%. Handing the records over in LDS, four lanes to a line, took it from 1.65 to
// 1.60 ms and single casts from 0.106 to 0.123 ms, so each lane loads its own.

// One lane's castRay over the wide nodes, or the binary ones, one record at a time.
struct LaneWalk {
	dev::Ray r;
	uint32_t ref = 0u;  // what the ray takes next: a node, or kWideLeaf and a triangle
	int sp = 0;
	int floor = 0;      // the stack's bottom for this walk
	Closest c = {kInvalid, FLT_MAX, FLT_MAX, FLT_MAX};
	uint32_t with = kFast;  // kFast, kSlab or kBinary

	// Decides a binary node's children as castRay does and pushes what is visited in its order.
	template <class Stack>
	__device__ __forceinline__ void expand_binary(const float4* nodes, float lim, Stack& st)
	{
		const NodeWords nd = load_node(nodes, ref);
		bool visitL, visitR;
		decide(r, nd, lim, visitL, visitR);
		const uint32_t refL = child_index(nd.w3.x) | (nd.w3.z != 0 ? kWideLeaf : 0u);
		const uint32_t refR = child_index(nd.w3.y) | (nd.w3.w != 0 ? kWideLeaf : 0u);
		const bool leftFirst = visitL && nd.w3.z != 0;
		if (visitL && visitR) st.put2(sp++, leftFirst ? refR : refL, -INFINITY);
		if (visitL || visitR)
			st.put2(sp++, visitL && visitR ? (leftFirst ? refL : refR) : visitL ? refL : refR, -INFINITY);
	}

	__device__ __forceinline__ bool at_leaf() const { return (ref & kWideLeaf) != 0u; }
	// The record that advance() consumes: a wide node, or a leaf's next two triangles (the words past
	// a leaf's last one are the next triangle's or the array's padding). Binary nodes read the array's
	// first line. The loads are bound by the 16 B a lane that the texture data path returns a cycle, so
	//   - a node is read in seven words: slot 3's max.xyz is in the last components of words 1, 3 and 5
	//     too (with eight, 64 fused batches took 1.635 ms, with seven 1.563; 1,048,576 rays into 300
	//     instances 3.235 and 3.137 ms);
	//   - lanes without a record (`on` false) read nothing: 17 of 64 lanes are active on average in the
	//     instance kernel, which took 3.036 ms where they read the first line, and 2.977 so.
	__device__ __forceinline__ void load(bool on, const float4* wide, const float4* tris,
	                                     float4 w[7]) const
	{
		if (!on) return;
		const float4* rec = at_leaf() ? tris + 3u * size_t(ref & kWideIndex)
		                              : wide + 8u * size_t(with != kBinary ? ref : 0u);
#pragma unroll
		for (int i = 0; i < 7; i++) w[i] = as_global(rec)[i];
	}

	// Expands a node or tests up to two triangles of a leaf, and picks what the lane takes next. True
	// if the traversal has ended (`occluded`: with an any-hit ray's hit).
	template <int kAny, bool kSlow, class Stack>
	__device__ __forceinline__ bool advance(const float4 w[7], const float4* nodes, bool any, Stack& st,
	                                        bool& occluded)
	{
		const bool leaf = at_leaf(), node = !leaf && !(kSlow && with == kBinary);
		bool pop = true;
		occluded = false;
		if (leaf) {
			// Up to two triangles, accepted in order.
			const dev::TriDet d0 = dev::tri_det(r, w[1], w[2]);
			const dev::TriDet d1 = dev::tri_det(r, w[4], w[5]);
			const float f0 = recip_wave(d0.a), f1 = recip_wave(d1.a);
			float t0, u0, v0, t1, u1, v1;
			const bool last0 = w[0].w < 0.0f;
			const bool h0 = dev::tri_finish(r, d0, f0, w[0], w[1], w[2], t0, u0, v0) && r.tMin <= t0;
			const bool h1 = dev::tri_finish(r, d1, f1, w[3], w[4], w[5], t1, u1, v1) && !last0 && r.tMin <= t1;
			if (kAny != 0) occluded = any && ((h0 && t0 < r.tMax) || (h1 && t1 < r.tMax));
			if (kAny != 1) {
				const uint32_t first = ref & kWideIndex;
				const bool acc0 = h0 && t0 < c.t && t0 <= r.tMax;
				c.tri = acc0 ? first : c.tri;
				c.t = acc0 ? t0 : c.t;
				c.u = acc0 ? u0 : c.u;
				c.v = acc0 ? v0 : c.v;
				const bool acc1 = h1 && t1 < c.t && t1 <= r.tMax;
				c.tri = acc1 ? first + 1u : c.tri;
				c.t = acc1 ? t1 : c.t;
				c.u = acc1 ? u1 : c.u;
				c.v = acc1 ? v1 : c.v;
			}
			pop = last0 || w[3].w < 0.0f;
			ref = kWideLeaf | ((ref & kWideIndex) + 2u);
		}
		const float lim = any ? r.tMax : dev::min_first(r.tMax, c.t);
		if (node) {
			WideWords n;
#pragma unroll
			for (int i = 0; i < 7; i++) n.w[i] = w[i];
			n.w[7] = make_float4(w[1].w, w[3].w, w[5].w, 0.0f);
			WideVisit v;
			if (kSlow) v = decide_wide_nan(r, n, lim);
			else v = decide_wide(r, n, lim);
			const bool p0 = v.pass[0], p1 = v.pass[1], p2 = v.pass[2], p3 = v.pass[3];
			uint32_t r0 = __float_as_uint(w[0].w), r1 = __float_as_uint(w[2].w);
			uint32_t r2 = __float_as_uint(w[4].w);
			uint32_t r3 = __float_as_uint(w[6].w);
			if (kSlow) {
				auto inner = [](uint32_t& at, float& tIn) {
					if (int32_t(at) >= int32_t(kWideLoose)) at &= kWideIndex, tIn = -INFINITY;
				};
				inner(r0, v.tIn[0]);
				inner(r1, v.tIn[1]);
				inner(r2, v.tIn[2]);
				inner(r3, v.tIn[3]);
			}
			r0 = p1 ? r0 : r0 & ~kWidePair;
			r1 = p2 ? r1 : r1 & ~kWidePair;
			r2 = p3 ? r2 : r2 & ~kWidePair;
			const bool p01 = p0 || p1, p012 = p01 || p2;
			const int at2 = sp + (p3 ? 1 : 0), at1 = at2 + (p2 ? 1 : 0);
			if (p3 && p012) st.put2(sp, r3, v.tIn[3]);
			if (p2 && p01) st.put2(at2, r2, v.tIn[2]);
			if (p1 && p0) st.put2(at1, r1, v.tIn[1]);
			pop = !(p012 || p3);
			sp = pop ? sp : at1 + (p1 ? 1 : 0) + (p0 ? 1 : 0) - 1;
			ref = p0 ? r0 : p1 ? r1 : p2 ? r2 : r3;
		}
		if (kSlow && with == kBinary && !leaf) expand_binary(nodes, lim, st);
		if (occluded || (pop && !take(lim, any, st))) return true;
		if (!any && (pop || node)) decide_sibling(lim, st);
		return false;
	}
	// Takes the top entry that the closest hit has not overtaken; false if there is none.
	template <class Stack>
	__device__ __forceinline__ bool take(float lim, bool any, Stack& st)
	{
		while (sp > floor) {
			uint32_t at;
			float tIn;
			st.get2(--sp, at, tIn);
			if (any || tIn < lim) {
				ref = at;
				return true;
			}
		}
		return false;
	}
	// The sibling of a leaf that is taken is decided with it.
	template <class Stack>
	__device__ __forceinline__ void decide_sibling(float lim, Stack& st)
	{
		if ((ref & (kWideLeaf | kWidePair)) == (kWideLeaf | kWidePair)) {
			uint32_t at;
			float tIn;
			st.get2(sp - 1, at, tIn);
			st.put2(sp - 1, at, tIn < lim ? -INFINITY : INFINITY);
		}
	}
};

// A lane's stack column: kRows entries in LDS, the deeper ones in private memory. (The LDS part through
// an LDS pointer and read in any case: a choice between the two would be made of flat loads.)
template <int kRows, int kEntries>
struct PrivateStack {
	LdsU2* col;
	U32x2 (&deep)[kEntries - kRows];
	__device__ __forceinline__ void put2(int at, uint32_t ref, float tIn)
	{
		const U32x2 e = {ref, __float_as_uint(tIn)};
		if (__builtin_expect(at < kRows, 1)) col[at * kBlock] = e;
		else deep[at - kRows] = e;
	}
	__device__ __forceinline__ void get2(int at, uint32_t& ref, float& tIn) const
	{
		U32x2 e = col[(at < kRows ? at : 0) * kBlock];
		if (__builtin_expect(ballot(at >= kRows) != 0ull, 0))
			if (at >= kRows) e = deep[at - kRows];
		ref = e.x;
		tIn = __uint_as_float(e.y);
	}
};

// A lane's stack column: entries in LDS, the deeper ones spilled.
struct SpillStack {
	LdsU2* stacks;
	U32x2* spill;
	uint32_t base;
	__device__ __forceinline__ void put2(int at, uint32_t ref, float tIn)
	{
		const U32x2 e = {ref, __float_as_uint(tIn)};
		if (__builtin_expect(at < kLaneRows, 1)) stacks[base + uint32_t(at) * 64u] = e;
		else *spill_entry<kLaneRows, 64u>(spill, base, at) = e;
	}
	__device__ __forceinline__ void get2(int at, uint32_t& ref, float& tIn) const
	{
		U32x2 e = stacks[base + uint32_t(at < kLaneRows ? at : 0) * 64u];
		if (__builtin_expect(at >= kLaneRows, 0)) e = *spill_entry<kLaneRows, 64u>(spill, base, at);
		ref = e.x;
		tIn = __uint_as_float(e.y);
	}
};

template <bool kTrack>
struct LaneTracer {
	const QuadArgs& P;
	SpillStack stack;
	LaneWalk t;
	uint32_t ray = kInvalid;
	bool any = false;
	uint32_t batch = 0u;
	const float4* wide = nullptr;
	const float4* tris = nullptr;

	// A window whose rays are staged in LDS, a lane's each. Its batch and that one's scene, if it has
	// only one.
	LdsF4* staged;
	uint32_t first = 0u, windowBatch = 0u;
	bool single = true;
	BatchDesc desc = {};
	__device__ __forceinline__ void stage(const RayWindows& W)
	{
		const uint32_t lane = __lane_id();
		first = W.next;
		if (W.next < W.end) {
			windowBatch = uniform(find_batch(P.offsets, P.numBatches, first));
			single = uniform(P.offsets[windowBatch + 1u]) >= W.end;
			desc = P.descs[windowBatch];
			const uint32_t at = first + lane;
			if (at < W.end) {
				const uint32_t b = single ? windowBatch : find_batch(P.offsets, P.numBatches, at);
				const float4* rays = single ? desc.rays : P.descs[b].rays;
				GlobalV4* p = (GlobalV4*)(rays) + 2u * size_t(at - P.offsets[b]);
				staged[lane] = p[0];
				staged[64u + lane] = p[1];
			}
		}
		__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
		__builtin_amdgcn_wave_barrier();
		__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
	}
	__device__ __forceinline__ void start(uint32_t index)
	{
		batch = windowBatch;
		BatchDesc d = desc;
		if (!single) {
			batch = find_batch(P.offsets, P.numBatches, index);
			d = P.descs[batch];
		}
		wide = d.wide;
		tris = d.tris;
		any = (d.kind & 1u) != 0u;
		const F32x4 sa = staged[index - first], sb = staged[64u + index - first];
		const float4 a = make_float4(sa.x, sa.y, sa.z, sa.w), b = make_float4(sb.x, sb.y, sb.z, sb.w);
		t.with = quad_ray(a, b, d.kind >> 1, t.r);
		if (__builtin_expect(t.with != kFast, 0)) divide(b, t.r);
		ray = index;
		t.ref = 0u;
		t.sp = 0;
		t.c = {kInvalid, FLT_MAX, FLT_MAX, FLT_MAX};
	}

	__device__ __forceinline__ void step()
	{
		const bool active = ray != kInvalid;
		float4 w[7];
		t.load(active, wide, tris, w);
		if (!active) return;
		bool occluded;
		const float4* nodes = P.descs[batch].nodes;
		const bool ended = __builtin_expect(ballot(t.with != kFast) != 0ull, 0)
		                       ? t.template advance<2, true>(w, nodes, any, stack, occluded)
		                       : t.template advance<2, false>(w, nodes, any, stack, occluded);
		if (ended) {
			quad_result<true, kTrack, false>(P, ray, batch, t.c, any, occluded);
			ray = kInvalid;
		}
	}
};

template <bool kTrack>
__device__ __forceinline__ void lane_trace(const QuadArgs& P, uint32_t* lds)
{
	const uint32_t waveInBlock = uniform(threadIdx.x >> 6), lane = __lane_id();
	LdsU2* stacks = (LdsU2*)(reinterpret_cast<U32x2*>(lds));
	LaneTracer<kTrack> T{P, {stacks, P.spill, stack_base<kLaneRows, 64u>(waveInBlock, lane)}};
	T.t.r = {};
	T.staged = (LdsF4*)(lds + blockDim.x / 64u * 2u * wave_stack_entries<kLaneRows, 64u>()) + waveInBlock * 128u;
	RayWindows W(P, waveInBlock);
	T.stage(W);
	while (true) {
		const uint64_t idle = ballot(T.ray == kInvalid);
		if (idle != 0ull) {
			if (W.next >= W.end) {
				if (!W.claim(P)) break;
				T.stage(W);
			}
			const uint32_t room = uint32_t(__popcll(idle));
			if (room >= P.refill) {
				const uint32_t ray = W.next + uint32_t(__popcll(idle & __lanemask_lt()));
				if (T.ray == kInvalid && ray < W.end) T.start(ray);
				W.next = W.end - W.next < room ? W.end : W.next + room;
			}
		}
		T.step();
	}
	// No more rays: until at most 16 are left.
	uint64_t busy = ballot(T.ray != kInvalid);
	while (__popcll(busy) > 16) {
		T.step();
		busy = ballot(T.ray != kInvalid);
	}
	if (busy == 0ull) return;
	// The k-th busy lane's ray goes to lanes 4k to 4k + 3.
	QuadTracer<2, true, kTrack, false, true, kLaneRows, 64u> Q{P};
	Q.stacks = stacks;
	Q.lane = lane;
	Q.l = lane & 3u;
	const uint32_t rank = uint32_t(__popcll(busy & __lanemask_lt()));
	const bool on = T.ray != kInvalid;
	auto move = [&](uint32_t v) {
		// Lane 4k reads its source: the busy lanes push to it, all others to a lane that nobody reads.
		const int to = on ? int(rank * 16u) : 4;
		const uint32_t at4k = uint32_t(__builtin_amdgcn_ds_permute(to, int(v)));
		return uint32_t(__builtin_amdgcn_update_dpp(0, int(at4k), 0x00, 0xF, 0xF, true));
	};
	const uint32_t ray = move(T.ray), ref = move(T.t.ref);
	Q.q.sp = int(move(uint32_t(T.t.sp)));
	Q.q.base = move(T.stack.base);
	const float best = __uint_as_float(move(__float_as_uint(T.t.c.t)));
	const float u = __uint_as_float(move(__float_as_uint(T.t.c.u)));
	const float v = __uint_as_float(move(__float_as_uint(T.t.c.v)));
	const uint32_t hit = move(T.t.c.tri), batch = move(T.batch);
	if (lane / 4u < uint32_t(__popcll(busy))) {
		Q.q.batch = batch;
		Q.take_over(ray);
		Q.q.best = best;
		Q.q.u = u;
		Q.q.v = v;
		Q.q.hit = hit;
		Q.q.mine = Q.l == 0u;
		Q.q.leaf = (ref & kWideLeaf) != 0u;
		Q.q.tri = (ref & kWideIndex) + Q.l;
		Q.q.triNext = (ref & kWideIndex) + 4u;
		Q.q.node = Q.q.leaf ? kInvalid : ref;
		Q.q.nodeIn = -INFINITY;
	}
	if (Q.q.ray == kInvalid) {  // read by lanes without a ray
		Q.q.wide = P.descs[0].wide;
		Q.q.tris = P.descs[0].tris;
	}
	Q.slow = ballot(Q.q.with != kFast) != 0ull;
	while (ballot(Q.q.ray != kInvalid) != 0ull) Q.step();
}

// Called by every block as it ends: the last one resets the launch's counters. Counted per group of
// blocks first, so that no address sees more than an eighth of them.
__device__ __forceinline__ bool retire_block(uint32_t* work)
{
	const uint32_t group = blockIdx.x % kCounters;
	const uint32_t inGroup = (gridDim.x - group + kCounters - 1u) / kCounters;
	const uint32_t groups = gridDim.x < kCounters ? gridDim.x : kCounters;
	__threadfence();
	if (atomicAdd(&work[(kCounters + group) * kCounterStride], 1u) != inGroup - 1u) return false;
	if (atomicAdd(&work[2u * kCounters * kCounterStride], 1u) != groups - 1u) return false;
	for (uint32_t i = 0; i <= 2u * kCounters; i++) atomicExch(&work[i * kCounterStride], 0u);
	return true;
}

__host__ __device__ __forceinline__ uint32_t lane_lds_words(uint32_t waves)
{
	return waves * (2u * wave_stack_entries<kLaneRows, 64u>() + 512u);  // stacks, staged rays
}

// ---- packets, then one ray per lane ----------------------------------------------------------------
//
// A packet whose rays part (a tile of grazing rays expands hundreds of nodes, most of them for a few of
// its rays) takes as many steps as the union of its rays: of 32,400 tiles of a 1080p view of 1,004,000
// triangles, half were done after 12 us and 90% after 78 us, but the longest took 351 us and set the
// launch's 0.43 ms. Such a packet ends and its lanes go on by themselves, each with its part of the
// shared stack: the longest now takes 250 us. The cast with ray generation: 0.468 -> 0.36 ms; a 1080p
// frame with 8 lights, whose shadow rays are packets too: 1.77 -> 1.62 ms. (The limits matter little:
// 0.377 to 0.383 ms for 4 or 8 steps and 12 to 48 rays; 16 steps of 24 rays 0.390, any 64 steps 0.419.
// Four lanes per ray instead, 16 rays at a time: slower than not leaving, 0.59 ms.)

constexpr int kPacketRows = 10;  // stack entries of a lane in LDS (20 KB a block, 7 blocks a CU)

// Takes over a packet's lane: its stack entries, and whether the packet's next node is its own.
struct PacketLeave {
	PrivateStack<kPacketRows, kMaxPending>& stack;
	LaneWalk& t;
	bool& on;
	__device__ __forceinline__ void push(int at, uint32_t ref, float tIn) { stack.put2(at, ref, tIn); }
	__device__ __forceinline__ void operator()(int n, uint32_t node, bool at)
	{
		t.ref = node;
		t.sp = n;
		on = at;
	}
};

// Traces the wave's rays t.r of the `active` lanes: t.c, or for any hit whether one was hit.
template <bool kAnyHit, bool kLoose>
__device__ __forceinline__ bool packet_trace(const float4* __restrict__ wide,
                                             const float4* __restrict__ nodes,
                                             const float4* __restrict__ tris, LaneWalk& t, bool active,
                                             LdsU2* column)
{
	bool occluded = false;
	t.c = Closest{kInvalid, FLT_MAX, FLT_MAX, FLT_MAX};
	// The wide nodes only when every active lane may walk them (the decision is uniform).
	if (!wide || __ballot(active && !t.r.nanFree) != 0ull) {
		packet_binary<kAnyHit>(nodes, tris, t.r, active, t.c, occluded);
		return occluded;
	}
	U32x2 deep[kMaxPending - kPacketRows];
	PrivateStack<kPacketRows, kMaxPending> stack = {column, deep};
	bool on = false;
	t.sp = 0;
	packet_wide<kAnyHit, kLoose>(wide, tris, t.r, active, t.c, occluded, PacketLeave{stack, t, on});
	if (ballot(on || t.sp > 0) == 0ull) return occluded;
	if (!on && t.sp > 0) {
		const float lim = kAnyHit ? t.r.tMax : dev::min_first(t.r.tMax, t.c.t);
		on = t.take(lim, kAnyHit, stack);
		if (on && !kAnyHit) t.decide_sibling(lim, stack);
	}
	while (ballot(on) != 0ull) {
		float4 w[7];
		t.load(on, wide, tris, w);
		if (on) on = !t.template advance<kAnyHit ? 1 : 0, false>(w, nodes, kAnyHit, stack, occluded);
	}
	return occluded;
}

template <bool kAnyHit, bool kLoose>
__global__ __launch_bounds__(kPacketBlock) void k_packet(const float4* __restrict__ wide,
                                                         const float4* __restrict__ nodes,
                                                         const float4* __restrict__ tris,
                                                         const float4* __restrict__ rays,
                                                         void* __restrict__ out, uint32_t n)
{
	__shared__ U32x2 stackLds[kPacketRows * kPacketBlock];
	const uint32_t lane = __lane_id();
	const uint32_t first = blockIdx.x * kPacketBlock + (threadIdx.x & ~63u);
	if (first >= n) return;  // whole wave
	const uint32_t i = first + lane;
	const bool active = i < n;
	const uint32_t ri = active ? i : first;  // lanes past the end read a valid ray, never used
	LaneWalk t;
	t.r = dev::make_ray(rays[2 * size_t(ri)], rays[2 * size_t(ri) + 1]);
	// (An any-hit ray with an empty interval hits nothing; the one that stands for none would keep its
	// packet on the binary nodes.)
	const bool traced = active && (!kAnyHit || t.r.tMin < t.r.tMax);
	const bool occluded =
		packet_trace<kAnyHit, kLoose>(wide, nodes, tris, t, traced, (LdsU2*)(stackLds) + threadIdx.x);
	if (active) {
		if (kAnyHit)
			static_cast<uint8_t*>(out)[i] = occluded ? 0 : 1;
		else
			static_cast<uint4*>(out)[i] = make_uint4(t.c.tri, __float_as_uint(t.c.t),
			                                         __float_as_uint(t.c.u), __float_as_uint(t.c.v));
	}
}

// ---- primary shading with its shadow rays ---------------------------------------------------------
//
// What k_shade, an any-hit cast of its rays and k_shadow_logic do for the primary records, in one pass:
// a wave takes 64 records (an 8x8 tile, if the records are in tiles) and, light by light, samples it,
// traces the lanes' shadow rays as a packet and adds the contributions that arrive -- in the same order,
// so the image is the same bit for bit. The contributions and shadow rays of 8 lights took 48 B a record
// and light to write and to read again (0.8 GB of a 1080p frame: 0.165 ms in k_shade, 0.058 in
// k_shadow_logic), and a lane without a ray had a dummy one whose zero direction components kept its
// packet on the binary nodes. A 1080p frame with 8 lights, whose bounce cast runs beside this and now
// starts before the shading: 1.61 -> 1.43 ms; 333x251 with 2 lights, in row order: 0.33 -> 0.28 ms.
template <bool kLoose>
__global__ __launch_bounds__(kPacketBlock, 5) void k_shade_trace(
	const float4* __restrict__ wide, const float4* __restrict__ nodes,
	const float4* __restrict__ tris, const float4* __restrict__ info,
	const PhxSphereLight* __restrict__ lights, uint32_t numLights, uint32_t w, uint32_t h,
	const FrameParams* __restrict__ fp, uint32_t purpose, float4* __restrict__ img)
{
	using namespace frame;
	__shared__ U32x2 stackLds[kPacketRows * kPacketBlock];
	const uint32_t first = blockIdx.x * kPacketBlock + (threadIdx.x & ~63u), count = w * h;
	if (first >= count) return;  // whole wave
	const uint32_t i = first + __lane_id();
	const bool active = i < count;
	const uint32_t id = active ? i : first;
	const float4 d1 = info[3 * size_t(id)], d2 = info[3 * size_t(id) + 1], d3 = info[3 * size_t(id) + 2];
	const bool hit = active && d3.w >= 0.0f;
	const V3 p = xyz(d1);
	const V3 view = normalize(sub(v3(fp->cam.origin[0], fp->cam.origin[1], fp->cam.origin[2]), p));
	Pcg32 rng = frame_rng(fp->seed, fp->frame, purpose, id);
	float c0 = 0.0f, c1 = 0.0f, c2 = 0.0f;
	for (uint32_t k = 0; k < numLights; k++) {
		LightSample s = {v3(0.0f, 0.0f, 0.0f), false, v3(0.0f, 1.0f, 0.0f), 0.0f};
		if (hit)
			s = sample_light(lights[k], p, xyz(d2), view, xyz(d3), d1.w, d2.w, v3(1.0f, 1.0f, 1.0f), rng);
		bool occluded = false;
		if (ballot(s.ray) != 0ull) {
			LaneWalk t;
			t.r = dev::make_ray(make_float4(p.x, p.y, p.z, 0.001f),
			                    make_float4(s.dir.x, s.dir.y, s.dir.z, s.len));
			occluded = packet_trace<true, kLoose>(wide, nodes, tris, t, s.ray, (LdsU2*)(stackLds) + threadIdx.x);
		}
		if (hit && !occluded) {
			c0 = c0 + s.c.x;
			c1 = c1 + s.c.y;
			c2 = c2 + s.c.z;
		}
	}
	if (active) {
		const uint2 at = pixel_of(id, w, h);
		img[size_t(at.y) * w + at.x] = make_float4(c0, c1, c2, 1.0f);
	}
}

// ---- instances (two-level traversal) ------------------------------------------------------------
//
// A top tree over the instances' world boxes (one instance per leaf, PhxBVHNode layout) is walked
// in castRay's order. An instance is entered iff the ray's slab test on its world box hits with
// tOut > tMin and tIn <= min(tMax, best t) -- `<=`, so an instance that could tie the best hit is
// still traced. Each entered instance runs castRay on its own SBVH with the ray moved into object
// space (o' = A o + b, d' = A d, the same t range; t is the same parameter in both spaces), from a
// miss, so its result is the one castRay gives for that instance alone. The closest of those
// results wins, the lower instance index on equal t. With `hits` holding a static-scene result on
// entry (seeded), that result counts as instance -1: an instance must be strictly closer.

// Ray (a, b) in an instance's object space; what its boxes are decided with.
__device__ __forceinline__ uint32_t object_ray(const DevInstance& in, const float4 a, const float4 b,
                                               dev::Ray& r)
{
	const float* A = in.worldToObject;
	float o[3], d[3];
	for (int k = 0; k < 3; k++) {
		float p = A[4 * k] * a.x + A[4 * k + 1] * a.y;
		p = p + A[4 * k + 2] * a.z;
		o[k] = p + A[4 * k + 3];
		float q = A[4 * k] * b.x + A[4 * k + 1] * b.y;
		d[k] = q + A[4 * k + 2] * b.z;
	}
	const float4 dir = make_float4(d[0], d[1], d[2], b.w);
	const uint32_t with = quad_ray(make_float4(o[0], o[1], o[2], a.w), dir, in.with, r);
	if (with != kFast) divide(dir, r);
	return with;
}

// The kernel is a per-lane state machine over persistent waves. The top tree has wide nodes too, so a
// lane between instances and a lane inside one take the same kind of step (LaneWalk), each with its
// own ray; `tIn <= x` is taken as `tIn < next float above x`. A lane that enters or leaves an instance
// loads the ray of the top tree again (two words for nine registers) and does so at once: collecting
// such lanes until they are 8 or 16 makes the wave wait longer than their instructions take (3.18 and
// 3.6 ms instead of 3.0). Rays are handed out as in the other persistent kernels, so lanes do not wait
// for the wave's costliest ray.
//
// Bound by VALU issue (81% busy, with 18 of 64 lanes active on average) and by the texture data path,
// which returns a lane's 16 B a cycle (76%). On the binary nodes, with exact slabs and divisions, a
// top-tree step in every iteration and a fixed range of rays per wave, 1,048,576 rays into 300
// instances took 4.92 ms (closest) and 262,147 any-hit rays into 120 instances and a scene 0.71 ms;
// now 2.92 and 0.40 ms. (Wide nodes inside the instances alone: 4.14 and 0.49 ms.)

constexpr uint32_t kInstanceRefill = 8;  // idle lanes of a wave before it takes new rays
constexpr uint32_t kInstanceWaves = 20;  // per CU: 5 per SIMD (96 registers)
constexpr int kInstanceRows = 14;        // stack entries of a lane in LDS (28 KB a block, 5 blocks a CU)

// The next float above x, so that t < next_up(x) is t <= x.
__device__ __forceinline__ float next_up(float x)
{
	const float y = x + 0.0f;  // (-0 to 0)
	if (!(fabsf(y) < INFINITY)) return y;
	return __uint_as_float(y >= 0.0f ? __float_as_uint(y) + 1u : __float_as_uint(y) - 1u);
}

template <bool kAnyHit>
__global__ __launch_bounds__(kBlock, 5) void k_trace_instances(
	const float4* __restrict__ top, const float4* __restrict__ topWide,
	const DevInstance* __restrict__ inst, uint32_t numInst, const float4* __restrict__ rays,
	uint4* __restrict__ hits, uint32_t* __restrict__ instOut, uint8_t* __restrict__ inLight,
	uint32_t n, uint32_t seeded, uint32_t* __restrict__ work)
{
	__shared__ U32x2 stackLds[kInstanceRows * kBlock];
	U32x2 deep[2 * kMaxPending - kInstanceRows];
	// The top tree's entries, an instance's above.
	PrivateStack<kInstanceRows, 2 * kMaxPending> stack = {(LdsU2*)(stackLds) + threadIdx.x, deep};
	QuadArgs P = {};
	P.n = n;
	P.window = 64u;
	P.work = work;
	RayWindows W(P, uniform(threadIdx.x >> 6));

	LaneWalk t;  // in the top tree, or the entered instance's castRay
	t.r = {};
	Closest best = t.c;
	uint32_t ray = kInvalid, bestInst = kInvalid, id = 0u;
	bool inside = false;   // t walks an instance
	bool leave = false;    // that walk has ended (or the ray is new)
	bool seededHit = false, fresh = false, handedOut = false;
	const float4* wide = topWide;
	const float4* tris = nullptr;
	const float4* nodes = top;
	while (true) {
		const uint64_t idle = ballot(ray == kInvalid);
		if (!handedOut && uint32_t(__popcll(idle)) >= kInstanceRefill) {
			if (W.next >= W.end && !W.claim(P)) {
				handedOut = true;
			} else {
				const uint32_t mine = W.next + uint32_t(__popcll(idle & __lanemask_lt()));
				if (ray == kInvalid && mine < W.end) {
					ray = mine;
					best = t.c = Closest{kInvalid, FLT_MAX, FLT_MAX, FLT_MAX};
					bestInst = kInvalid;
					seededHit = false;
					leave = fresh = true;
					if (!kAnyHit && seeded) {
						const uint4 h = hits[ray];
						best = Closest{h.x, __uint_as_float(h.y), __uint_as_float(h.z), __uint_as_float(h.w)};
						seededHit = h.x != kInvalid;
					}
					if (kAnyHit && seeded && inLight[ray] == 0) ray = kInvalid;  // (stays 0)
				}
				const uint32_t taken = uint32_t(__popcll(idle));
				W.next = W.end - W.next < taken ? W.end : W.next + taken;
			}
		}
		const bool busy = ray != kInvalid;
		if (ballot(busy) == 0ull) {
			if (handedOut) break;
			continue;
		}
		if (busy && (leave || (!inside && t.at_leaf()))) {
			const float4 a = as_global(rays)[2 * size_t(ray)], b = as_global(rays)[2 * size_t(ray) + 1];
			if (leave) {
				leave = inside = false;
				// The closer result, the lower index on equal t.
				if (!kAnyHit && t.c.tri != kInvalid) {
					const bool tieWins = t.c.t == best.t && !seededHit && (bestInst == kInvalid || id < bestInst);
					if (t.c.t < best.t || tieWins) {
						best = t.c;
						bestInst = id;
						seededHit = false;
					}
				}
				t.with = quad_ray(a, b, topWide != top ? kFast : kBinary, t.r);
				if (__builtin_expect(t.with != kFast, 0)) divide(b, t.r);
				if (!kAnyHit) t.r.tMax = next_up(t.r.tMax);
				t.c = Closest{kInvalid, kAnyHit ? FLT_MAX : next_up(best.t), FLT_MAX, FLT_MAX};
				t.floor = 0;
				wide = topWide;
				nodes = top;
				const float lim = kAnyHit ? t.r.tMax : dev::min_first(t.r.tMax, t.c.t);
				if (fresh) {
					t.ref = 0u;
					t.sp = 0;
				}
				if (fresh ? numInst == 0u : !t.take(lim, kAnyHit, stack)) {
					if (kAnyHit) {
						inLight[ray] = 1;
					} else {
						if (bestInst != kInvalid || !seeded)
							hits[ray] = make_uint4(best.tri, __float_as_uint(best.t), __float_as_uint(best.u),
							                       __float_as_uint(best.v));
						if (instOut) instOut[ray] = bestInst;
					}
					ray = kInvalid;
				} else if (!kAnyHit && !fresh) {
					t.decide_sibling(lim, stack);
				}
				fresh = false;
			}
			if (ray != kInvalid && (t.ref & kWideLeaf)) {
				const DevInstance& in = inst[t.ref & kWideIndex];
				id = in.index;
				nodes = in.nodes;
				tris = in.tris;
				wide = in.wide;
				t.with = object_ray(in, a, b, t.r);
				t.ref = 0u;
				t.floor = t.sp;
				t.c = Closest{kInvalid, FLT_MAX, FLT_MAX, FLT_MAX};
				inside = true;
			}
		}
		const bool walks = ray != kInvalid && !leave && (inside || !t.at_leaf());
		if (ballot(walks) == 0ull) continue;
		float4 w[7];
		t.load(walks, wide, tris, w);
		bool occluded;
		bool ended = false;
		if (__builtin_expect(ballot(walks && t.with != kFast) != 0ull, 0)) {
			if (walks) ended = t.template advance<kAnyHit ? 1 : 0, true>(w, nodes, kAnyHit, stack, occluded);
		} else if (walks) {
			ended = t.template advance<kAnyHit ? 1 : 0, false>(w, nodes, kAnyHit, stack, occluded);
		}
		if (ended) {
			leave = true;
			if (kAnyHit && occluded) {
				inLight[ray] = 0;
				ray = kInvalid;
				leave = inside = false;
			}
		}
	}
	__syncthreads();
	if (threadIdx.x == 0u) retire_block(work);
}

template <bool kAnyHit, bool kClock, bool kBig>
__global__ __launch_bounds__(kQuadBlock, kQuadWavesPerSimd) void k_quad(
	const float4* __restrict__ wide, const float4* __restrict__ nodes,
	const float4* __restrict__ tris, const float4* __restrict__ rays, void* __restrict__ out,
	uint32_t n, uint32_t window, uint32_t refill, uint32_t* __restrict__ work,
	U32x2* __restrict__ spill, unsigned long long* __restrict__ clock, uint32_t with)
{
	extern __shared__ uint32_t lds[];
	const QuadArgs P = {wide, nodes, tris, rays, out, n, with, window, refill, work, spill, clock,
	                    nullptr, nullptr, 0u, nullptr, nullptr};
	quad_trace<kAnyHit ? 1 : 0, kClock, kBig>(P, lds);
	if (threadIdx.x == 0u) retire_block(work);
}

// ---- fused multi-batch launch ---------------------------------------------------------------------
//
// One persistent launch over many ray batches (closest-hit or any-hit, on one or several scenes):
// the batches' rays form one index space [0, total) handed out as above; a ray's index is mapped to
// (batch, local index) by binary search over the batch offsets held in LDS, when its lane starts it.
// With completion tracking on, the lanes completing rays in the block count completions and the
// latest completion time per batch in LDS, and every block adds them to the batch table with one
// global atomic per batch when it ends, so each batch's latency inside the launch is known (the
// clock only grows, so completion times need no reset between launches). The last block to end
// resets the counters for the next launch.
// Four waves per SIMD: a wave's stacks and rays take 8.5 KB of LDS, and four fill blocks of 1,024 threads.

__host__ __device__ __forceinline__ uint32_t batch_lds_words(uint32_t waves, uint32_t numBatches,
                                                             bool tracked)
{
	return lane_lds_words(waves) + (tracked ? 3u * numBatches : 0u) + numBatches + 1u;
}

template <bool kTrack>
__global__ __launch_bounds__(kLaneBlock, 4) void k_trace_batches(
	const BatchDesc* __restrict__ descs, const uint32_t* __restrict__ offsetsGlobal,
	uint32_t numBatches, uint32_t total, uint32_t window, uint32_t refill,
	uint32_t* __restrict__ work, U32x2* __restrict__ spill, BatchClock* __restrict__ clock)
{
	extern __shared__ uint32_t lds[];
	// (An even number of words precedes the 8-byte finish times.)
	unsigned long long* blockFinish =
		reinterpret_cast<unsigned long long*>(lds + lane_lds_words(blockDim.x / 64u));
	uint32_t* blockDone = reinterpret_cast<uint32_t*>(blockFinish + (kTrack ? numBatches : 0u));
	uint32_t* offsets = blockDone + (kTrack ? numBatches : 0u);
	if (kTrack && threadIdx.x == 0) atomicMin(&clock->start, wall_clock64());
	for (uint32_t i = threadIdx.x; i <= numBatches; i += blockDim.x) offsets[i] = offsetsGlobal[i];
	if (kTrack)
		for (uint32_t i = threadIdx.x; i < numBatches; i += blockDim.x) {
			blockFinish[i] = 0ull;
			blockDone[i] = 0u;
		}
	__syncthreads();
	const QuadArgs P = {nullptr, nullptr, nullptr, nullptr, nullptr, total, 0u, window, refill, work,
	                    spill, nullptr, descs, offsets, numBatches, blockFinish, blockDone};
	lane_trace<kTrack>(P, lds);
	__syncthreads();
	if (kTrack) {
		for (uint32_t b = threadIdx.x; b < numBatches; b += blockDim.x)
			if (blockDone[b]) {
				atomicAdd(&clock->done[b], blockDone[b]);
				atomicMax(&clock->finish[b], blockFinish[b]);
			}
		__threadfence();
		__syncthreads();
	}
	if (threadIdx.x == 0u && retire_block(work) && kTrack) {
		for (uint32_t b = 0; b < numBatches; b++) atomicExch(&clock->done[b], 0u);
		clock->lastStart = atomicExch(&clock->start, ~0ull);
	}
}

// ---- device self-check of the fast reciprocal -----------------------------------------------------

constexpr uint64_t kBinade = 1ull << 23;           // significands per exponent
constexpr uint64_t kNormalBinades = 252;            // exponent fields 1 .. 252: 2^-126 <= |a| < 2^126
constexpr uint32_t kSampleExponents[4] = {1u, 126u, 127u, 252u};

__global__ __launch_bounds__(kBlock) void k_check_reciprocal(bool exhaustive, uint64_t total,
                                                             unsigned long long* mismatches)
{
	const uint64_t perSign = total / 2u;
	unsigned long long bad = 0;
	for (uint64_t i = blockIdx.x * uint64_t(blockDim.x) + threadIdx.x; i < total;
	     i += uint64_t(gridDim.x) * blockDim.x) {
		const uint32_t sign = i >= perSign ? 0x80000000u : 0u;
		const uint64_t j = i % perSign;
		const uint32_t binade = uint32_t(j / kBinade), mant = uint32_t(j % kBinade);
		const uint32_t expField = exhaustive ? 1u + binade : kSampleExponents[binade];
		const float a = __uint_as_float(sign | (expField << 23) | mant);
		if (__float_as_uint(dev::recip_newton(a)) != __float_as_uint(1.0f / a)) bad++;
	}
	if (bad) atomicAdd(mismatches, bad);
}

uint32_t gridFor(uint32_t n, uint32_t block) { return n / block + (n % block != 0u); }

// Rays per wave of a counting cast: as few as the 24 waves that a CU holds need.
uint32_t countedRaysPerWave(const TraceLaunch& L, uint32_t n)
{
	return std::min(64u, std::max(1u, gridFor(n, L.cus * 24u)));
}

// Whether 32-bit byte offsets into the scene's triangles and wide nodes do not do (kBig).
bool bigScene(const SceneView& s)
{
	return size_t(s.numTris) * 48u >= (size_t(1) << 32) || size_t(s.numNodes) * 128u >= (size_t(1) << 32);
}

// Launch shapes of the persistent kernels for n rays. A launch keeps at most L.raysInFlight rays in
// flight, each on a column of the spill area, takes at most L.window of them at a time and new ones when
// a share of L.refillMin / 64 of a wave's places is idle.
using Shape = LaunchShape;

Shape shapeOf(uint32_t waves, uint32_t most, uint32_t block)
{
	while (block > 64u && block / 64u > most) block /= 2u;
	const uint32_t perBlock = block / 64u;
	return Shape{std::max(1u, std::min(gridFor(waves, perBlock), most / perBlock)), block, 0u, 0u};
}

// Four lanes per ray.
//   - A launch that fills the device takes windows of 16 rays, as many as a wave traces at a time: what
//     remains of a wider one is traced by the same wave, one after another, and rays beside costly rays
//     are costly ones. Any-hit rays end sooner, and those that stand for none are answered a window at a
//     time: up to 64, two windows a wave at least, so that the last ones even out what the waves have
//     left. In us with 16, 32 and 64 (a frame, whose bounce shadow rays are mostly none: 32 and 64):
//       2,073,600 camera rays on 1,004,000 triangles     470   493   602 (any hit 265   214   236)
//       1,048,576 that look along the ground             516   612   961 (any hit 166   140   161)
//       998,029 bounce rays                              407   407   421 (any hit 168   161   170)
//       998,029 shadow rays, any hit                     154   117   119
//       1080p frame, 8 lights; any hit                         1,331 1,207
//   - A launch that does not gives each wave as few rays as about 2,048 waves need (two per SIMD: a
//     wave's time per iteration grows with the kinds of step its rays are at), up to the 16 it has
//     lanes for.
Shape quadShape(const TraceLaunch& L, uint32_t n, bool anyHit)
{
	const uint32_t most = std::max(
		1u, std::min(std::min(L.raysInFlight, L.spillColumns) / 16u, L.cus * kQuadWavesPerSimd * 4u));
	const uint32_t window =
		std::min(std::min(anyHit ? 64u : 16u, L.window),
		         n / 16u >= most ? std::max(16u, n / (2u * most))
		                         : std::min(16u, std::max(gridFor(n, 2048u), gridFor(n, most))));
	const uint32_t waves = std::min(most, gridFor(n, window));
	Shape s = shapeOf(waves, most, 256u);  // (four waves: a CU holds seven such blocks)
	s.window = window;
	s.refill = std::min(16u, std::max(1u, L.refillMin / 4u));
	return s;
}

// One ray per lane: windows of 64 rays, or fewer by L. A launch whose waves need 16 rays at most takes 16,
// which they trace four lanes each from the start: 6,077 rays in 8 batches 160 us with 64 and 98 with 16,
// 46,460 in 8 238 and 228; 85,813 in 64 (which would take 21) 247 and 267.
// Blocks small enough that every CU has one, and of 1,024 threads where `tableWords` of LDS beside the waves'
// (the batch tables) would halve the waves of a CU in blocks of 512 (256 tracked batches of 29.6 million
// rays: 7.4 ms with 8 waves per CU, 4.7 with 16). No more waves than are resident: the others' first windows
// would wait for a block to end.
Shape laneShape(const TraceLaunch& L, uint32_t n, uint32_t tableWords)
{
	auto resident = [&](uint32_t block) {
		const uint32_t perBlock = block / 64u, lds = (lane_lds_words(perBlock) + tableWords) * 4u;
		return std::min(16u, kLdsBytes / lds * perBlock);
	};
	uint32_t block = resident(kLaneBlock) > resident(kQuadBlock) ? kLaneBlock : kQuadBlock;
	const uint32_t most = std::max(1u, std::min(std::min(L.raysInFlight, L.spillColumns) / 64u,
	                                            L.cus * std::max(1u, resident(block))));
	const uint32_t window = std::min(n <= 16u * most ? 16u : 64u, L.window), waves = std::min(most, gridFor(n, window));
	while (block > 64u && waves / (block / 64u) < L.cus) block /= 2u;
	Shape s = shapeOf(waves, most, block);
	s.window = window;
	s.refill = std::min(64u, std::max(1u, L.refillMin));
	return s;
}

}  // namespace

// Device scratch of the allocation-free closest-hit cast (phx_cast_closest_noalloc): the ray
// counter pair of its persistent launch in the first kNoAllocCounterBytes, then the stack spill
// area, kNoAllocSpillWords words. A file-scope device array: every GPU the library runs on holds
// its own copy from the module load until the process ends. Host code must not pass `scratch`
// itself to a kernel (on the host it is only a stand-in for the symbol); it uses the address
// hipGetSymbolAddress returns for the current device, looked up once per device.
static __device__ __align__(256) uint8_t
	scratch[kNoAllocCounterBytes + size_t(kNoAllocSpillWords) * 4u];

namespace {

std::mutex gScratchMu;
void* gScratchPtr[kNoAllocMaxDevices] = {};

// Zeroes `n` words (n <= 1024); a kernel rather than a memset, so a caller may capture it in a graph.
__global__ void k_zero_words(uint32_t* p, uint32_t n)
{
	if (threadIdx.x < n) p[threadIdx.x] = 0u;
}

}  // namespace

hipError_t noAllocScratchInit(int device)
{
	if (device < 0 || device >= kNoAllocMaxDevices) return hipErrorInvalidDevice;
	std::lock_guard<std::mutex> g(gScratchMu);
	if (gScratchPtr[device]) return hipSuccess;
	void* ptr = nullptr;
	const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
	if (e != hipSuccess) return e;
	gScratchPtr[device] = ptr;
	return hipSuccess;
}

void* noAllocScratch(int device)
{
	if (device < 0 || device >= kNoAllocMaxDevices) return nullptr;
	std::lock_guard<std::mutex> g(gScratchMu);
	return gScratchPtr[device];
}

hipError_t launchZeroWords(uint32_t* p, uint32_t n, hipStream_t stream)
{
	hipLaunchKernelGGL(k_zero_words, dim3(1), dim3(1024), 0, stream, p, n);
	return hipGetLastError();
}

static_assert(kRayCounterWords >= (2u * kCounters + 1u) * kCounterStride, "ray counters");

hipError_t launchCheckReciprocal(bool exhaustive, unsigned long long* mismatches, uint64_t* tested,
                                 hipStream_t stream)
{
	const uint64_t total = 2u * kBinade * (exhaustive ? kNormalBinades : 4u);
	*tested = total;
	hipLaunchKernelGGL(k_check_reciprocal, dim3(2048), dim3(kBlock), 0, stream, exhaustive, total,
	                   mismatches);
	return hipGetLastError();
}

hipError_t launchClosest(const SceneView& s, const PhxRayIn* rays, uint32_t n, PhxRayHit* hits,
                         const TraceLaunch& L, unsigned long long* counters, hipStream_t stream)
{
	if (n == 0) return hipSuccess;
	const float4* wide = reinterpret_cast<const float4*>(s.wide);
	const float4* nodes = reinterpret_cast<const float4*>(s.nodes);
	const float4* tris = reinterpret_cast<const float4*>(s.trisPre);
	const float4* r4 = reinterpret_cast<const float4*>(rays);
	uint4* h4 = reinterpret_cast<uint4*>(hits);
	if (L.kernel == TraceKernel::Packet && !counters) {
		hipLaunchKernelGGL((s.loose ? k_packet<false, true> : k_packet<false, false>), dim3(gridFor(n, kPacketBlock)),
		                   dim3(kPacketBlock), 0, stream, wide, nodes, tris, r4, static_cast<void*>(h4), n);
		return hipGetLastError();
	}
	// Counters count binary node visits, which the one-ray-per-lane kernel makes.
	if (counters) {
		const uint32_t perWave = countedRaysPerWave(L, n);
		hipLaunchKernelGGL(k_closest_simple<true>, dim3(gridFor(n, kBlock / 64u * perWave)), dim3(kBlock), 0, stream,
		                   wide, nodes, tris, r4, h4, n, perWave, counters);
		return hipGetLastError();
	}
	if (L.kernel != TraceKernel::Persistent || n > 0x7FFFFFFFu) {
		hipLaunchKernelGGL(k_closest_simple<false>, dim3(gridFor(n, kBlock)), dim3(kBlock), 0, stream,
		                   s.loose ? nullptr : wide, nodes, tris, r4, h4, n, 64u, nullptr);
		return hipGetLastError();
	}
	const Shape q = quadShape(L, n, false);
	auto kernel = bigScene(s) ? k_quad<false, false, true> : k_quad<false, false, false>;
	hipLaunchKernelGGL(kernel, dim3(q.grid), dim3(q.block), quad_lds_words(q.block / 64u) * 4u, stream,
	                   wide ? wide : tris, nodes, tris, r4, static_cast<void*>(h4), n, q.window, q.refill,
	                   L.work, reinterpret_cast<U32x2*>(L.spill), nullptr, sceneWith(s.wide, s.loose));
	return hipGetLastError();
}

hipError_t launchClosestClock(const SceneView& s, const PhxRayIn* rays, uint32_t n, PhxRayHit* hits,
                              const TraceLaunch& L, unsigned long long* clock, hipStream_t stream)
{
	if (n == 0) return hipSuccess;
	if (n > 0x7FFFFFFFu) return hipErrorInvalidValue;
	const float4* nodes = reinterpret_cast<const float4*>(s.nodes);
	const float4* tris = reinterpret_cast<const float4*>(s.trisPre);
	const float4* wide = s.wide ? reinterpret_cast<const float4*>(s.wide) : tris;
	const Shape q = quadShape(L, n, false);
	auto kernel = k_quad<false, true, true>;
	hipLaunchKernelGGL(kernel, dim3(q.grid), dim3(q.block), quad_lds_words(q.block / 64u) * 4u, stream,
	                   wide, nodes, tris, reinterpret_cast<const float4*>(rays),
	                   static_cast<void*>(hits), n, q.window,
	                   q.refill, L.work, reinterpret_cast<U32x2*>(L.spill), clock,
	                   sceneWith(s.wide, s.loose));
	return hipGetLastError();
}

hipError_t launchAnyHitCounted(const SceneView& s, const PhxRayIn* rays, uint32_t n,
                               uint8_t* inLight, const TraceLaunch& L, unsigned long long* counters,
                               hipStream_t stream)
{
	if (n == 0) return hipSuccess;
	const uint32_t perWave = countedRaysPerWave(L, n);
	hipLaunchKernelGGL(k_anyhit_simple<true>, dim3(gridFor(n, kBlock / 64u * perWave)), dim3(kBlock), 0, stream,
	                   nullptr, reinterpret_cast<const float4*>(s.nodes),
	                   reinterpret_cast<const float4*>(s.trisPre),
	                   reinterpret_cast<const float4*>(rays), inLight, n, perWave, counters);
	return hipGetLastError();
}

hipError_t launchInstances(const PhxBVHNode* top, const WideNode* topWide, const DevInstance* inst, uint32_t numInst,
                          const PhxRayIn* rays, uint32_t n, PhxRayHit* hits, uint32_t* instOut,
                          uint8_t* inLight, bool seeded, const TraceLaunch& L, hipStream_t stream)
{
	if (n == 0) return hipSuccess;
	const float4* t4 = reinterpret_cast<const float4*>(top);
	const float4* w4 = topWide ? reinterpret_cast<const float4*>(topWide) : t4;
	const float4* r4 = reinterpret_cast<const float4*>(rays);
	const uint32_t waves = std::min(L.cus * kInstanceWaves, gridFor(n, 64u));
	const dim3 grid(gridFor(waves, kBlock / 64u));
	if (inLight)
		hipLaunchKernelGGL(k_trace_instances<true>, grid, dim3(kBlock), 0, stream, t4, w4, inst,
		                   numInst, r4, nullptr, nullptr, inLight, n, uint32_t(seeded), L.work);
	else
		hipLaunchKernelGGL(k_trace_instances<false>, grid, dim3(kBlock), 0, stream, t4, w4, inst,
		                   numInst, r4, reinterpret_cast<uint4*>(hits), instOut, nullptr, n,
		                   uint32_t(seeded), L.work);
	return hipGetLastError();
}

hipError_t launchAnyHit(const SceneView& s, const PhxRayIn* rays, uint32_t n, uint8_t* inLight,
                        const TraceLaunch& L, hipStream_t stream)
{
	if (n == 0) return hipSuccess;
	const float4* wide = reinterpret_cast<const float4*>(s.wide);
	const float4* nodes = reinterpret_cast<const float4*>(s.nodes);
	const float4* tris = reinterpret_cast<const float4*>(s.trisPre);
	const float4* r4 = reinterpret_cast<const float4*>(rays);
	if (L.kernel == TraceKernel::Packet) {
		hipLaunchKernelGGL((s.loose ? k_packet<true, true> : k_packet<true, false>), dim3(gridFor(n, kPacketBlock)),
		                   dim3(kPacketBlock), 0, stream, wide, nodes, tris, r4, static_cast<void*>(inLight), n);
		return hipGetLastError();
	}
	if (L.kernel == TraceKernel::Simple || n > 0x7FFFFFFFu) {
		hipLaunchKernelGGL(k_anyhit_simple<false>, dim3(gridFor(n, kBlock)), dim3(kBlock), 0,
		                   stream, s.loose ? nullptr : wide, nodes, tris, r4, inLight, n, 64u, nullptr);
		return hipGetLastError();
	}
	const Shape q = quadShape(L, n, true);
	auto kernel = bigScene(s) ? k_quad<true, false, true> : k_quad<true, false, false>;
	hipLaunchKernelGGL(kernel, dim3(q.grid), dim3(q.block), quad_lds_words(q.block / 64u) * 4u, stream,
	                   wide ? wide : tris, nodes, tris, r4, static_cast<void*>(inLight), n, q.window, q.refill,
	                   L.work, reinterpret_cast<U32x2*>(L.spill), nullptr, sceneWith(s.wide, s.loose));
	return hipGetLastError();
}

hipError_t launchShadeTrace(const SceneView& s, const float4* info, const PhxSphereLight* lights,
                            uint32_t numLights, uint32_t w, uint32_t h, const FrameParams* fp,
                            uint32_t purpose, float4* img, hipStream_t stream)
{
	if (w == 0 || h == 0) return hipSuccess;
	hipLaunchKernelGGL((s.loose ? k_shade_trace<true> : k_shade_trace<false>), dim3(gridFor(w * h, kPacketBlock)),
	                   dim3(kPacketBlock), 0, stream,
	                   reinterpret_cast<const float4*>(s.wide), reinterpret_cast<const float4*>(s.nodes),
	                   reinterpret_cast<const float4*>(s.trisPre), info, lights, numLights, w, h, fp,
	                   purpose, img);
	return hipGetLastError();
}

LaunchShape castShape(const TraceLaunch& L, uint32_t n, bool anyHit) { return quadShape(L, n, anyHit); }

LaunchShape batchShape(const TraceLaunch& L, uint32_t total, uint32_t numBatches, bool tracked)
{
	return laneShape(L, total, batch_lds_words(0u, numBatches, tracked));
}

hipError_t launchBatches(const BatchDesc* descs, const uint32_t* offsets, uint32_t numBatches,
                         uint32_t total, const TraceLaunch& L, BatchClock* clock, hipStream_t stream)
{
	if (total == 0) return hipSuccess;
	const Shape q = batchShape(L, total, numBatches, clock != nullptr);
	hipLaunchKernelGGL(clock ? k_trace_batches<true> : k_trace_batches<false>, dim3(q.grid),
	                   dim3(q.block), batch_lds_words(q.block / 64u, numBatches, clock != nullptr) * 4u,
	                   stream, descs, offsets, numBatches, total, q.window, q.refill, L.work,
	                   reinterpret_cast<U32x2*>(L.spill), clock);
	return hipGetLastError();
}

}  // namespace phx
