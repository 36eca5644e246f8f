// Nearest-hit traversal for nearest_hits (replaces BVH2::nearest_tri, bvh.hpp:224-265, and
// the thread split of CPUBackend::nearest_hits, intersect_cpu.hpp:20-43).
//
// One lane per ray, persistent waves. A wave takes rays from a global counter in batches:
// lanes whose ray has finished are counted with a ballot, one lane reserves that many ray
// indices with a single atomic and the base is broadcast with readlane, so finished lanes are
// refilled while the others keep traversing. The traversal stack lives in an LDS ring per lane
// (spilling its oldest entries to global memory when deep). Entries carry the entry distance
// of their box so they are re-culled when popped.
//
// Node tests are conservative versions of the reference slab test on the child boxes (fp32 or
// 8-bit quantized boxes rounded outward), so a node is never rejected when the exact test of a
// triangle below it would pass. Every triangle reached gets the exact reference predicates
// (slab on its own box, then Moller-Trumbore, operation by operation). The answer is the
// minimum t over all candidates with equal t resolved to the lowest primitive id.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <mutex>
#include <type_traits>

#include "common.h"
#include "internal.h"

namespace prt {
namespace {

struct KArgs {
	const void *nodes;
	const NodeQ *nodes_q;   // quantized nodes: their byte 15 is the never-cull mask of either format
	int any_ncull;          // some triangle is flagged (or the count is unknown)
	int leaf_test;          // 0 Moller-Trumbore (the reference's), 1 watertight
	const TriRec *tris;
	const float *rays;
	uint8_t *out;
	unsigned long long *counter;  // kCounters words (C_*), all 0 at the start of the launch
	unsigned long long *left;     // rays left to kRest: ray index | scene << 40, kLeftMax entries
	unsigned long long *next;     // another set, cleared here for the launch that follows, or null
	uint2 *spill;           // spill_depth entries per launched thread
	uint64_t n_rays;
	uint32_t n_nodes;
	uint32_t n_tris;
	uint32_t max_entries;   // stack bound 7 * depth + 8
	uint32_t stride;
	uint32_t mask;
	uint32_t spill_depth;
	uint32_t chunk;         // rays a wave reserves per atomic
	uint32_t leaf_phase;    // triangle phase once parked lanes >= live lanes * leaf_phase / 64
	uint32_t wide_grid;     // workgroups of k_trace_wide for the first pass, 0: k_trace
	uint32_t wide_rest;     // of the second pass, 0: k_trace
	uint32_t refill;        // load new rays once at least this many lanes are idle (or all are)
	float margin_rel;
	float margin_abs;
	int cull;
	float reach;            // largest vertex coordinate of the scene in magnitude
	// learned seeding (null when off): 4 cluster ids per ray, cluster entries and fp32 boxes
	const uint32_t *seeds;
	const uint32_t *cl_entry;
	const float *cl_box;
	uint32_t n_clusters;
	int n_seeds;            // predicted clusters searched first (1..4, the best ones)
	// several scenes (null when off): ray tiles {first lo, first hi, count, scene} claimed one
	// per atomic, and per scene {margin_abs, reach}; BVH8 node s is the root of scene s
	const uint4 *tiles;
	uint32_t n_tiles;
	const float2 *scene_info;
};

// Words of a launch's counters.
enum : int {
	C_WORK = 0,       // next ray (or tile) of the main pass
	C_NODES = 1,      // statistics
	C_TRIS = 2,
	C_LEAVES = 3,
	C_ERR = 4,        // low 32 bits: error flags, high 32 bits: rays left to the second pass (see kLeftMax)
	C_NPHASE = 5,
	C_TPHASE = 6,
	C_CULLED = 7,
	C_WORK_REST = 8,  // next ray (or tile, or list entry) of the second pass
	kCounters = 9
};

// Quantized nodes are traversed in two launches: kFast takes the rays of the one-fma node test
// (one_fma_ray) and leaves the others (d_x = 0, a zero axis near coordinate 0, magnitudes out of its
// range) to kRest. Up to kLeftMax of them are
// listed; past that kRest goes through all rays again and takes those (a second look at 24 M
// rays in 382,000 tiles takes 4.8 ms, which a single such ray must not cost). With none its waves
// end at once. One kernel for both held
// the reference formula's registers against every ray: at the plain mode's 64 it spilled 10, and
// with the treatment of d_x = 0 (child_slab) 58. kAll: fp32 nodes, one node test for every ray.
enum Pass : int { kAll = 0, kFast = 1, kRest = 2 };

// kWatertight: the plain traversal with the watertight leaf test (wt_candidate), no culling.
// kSeeded searches the best predicted cluster first, kSeededMulti the best 2..4.
enum : int { kPlain = 0, kSeeded = 1, kBatch = 2, kWatertight = 3, kSeededMulti = 4 };

constexpr uint32_t kInvalid = 0xFFFFFFFFu;

// Per-lane ray state.
struct Ray {
	float o[3], d[3];
	float inv[3];      // 1/d, with +-kFlat in the place of +-inf where the one-fma node test is used
	float tb, ub, vb;
	uint32_t idb;
	float abs_margin;  // margin_abs / |d|; infinite: this ray is not culled by distance
	bool mine;         // this launch traces the ray (Pass)
	bool odd;          // some 1/d or o is not finite (child_slab)
	bool line;         // d_x = 0, and the leaf test's error is bounded (child_slab)
	bool never;        // no triangle can be hit: NaN in origin or direction, or no direction
};

template <int PASS, bool WT>
__device__ __forceinline__ void load_ray(const KArgs &a, uint64_t idx, float margin_abs, float reach, Ray &r) {
	const float *p = a.rays + 6 * idx;  // 4-byte aligned AoS records of 24 bytes
#pragma unroll
	for (int k = 0; k < 3; ++k) {
		r.o[k] = p[k];
		r.d[k] = p[3 + k];
	}
#pragma unroll
	for (int k = 0; k < 3; ++k) r.inv[k] = 1.0f / r.d[k];  // IEEE division, as the reference
	const bool zero[3] = {r.d[0] == 0.0f, r.d[1] == 0.0f, r.d[2] == 0.0f};
	bool nan = false;
#pragma unroll
	for (int k = 0; k < 3; ++k) nan |= __builtin_isnan(r.o[k]) || __builtin_isnan(r.d[k]);
	const bool in_range = ray_in_range(r.o, r.d, r.inv, reach);
	// With NaN in the origin or the direction every t is NaN, which never wins; without a
	// direction every determinant is 0 (Moller-Trumbore) or NaN (the watertight test).
	r.never = nan || (zero[0] && zero[1] && zero[2]);
	bool fast = in_range && !zero[0];
	const bool exact = !a.cull && !WT;
	if (fast && (exact || zero[1] || zero[2])) fast = one_fma_ray(r.o, r.d, r.inv, reach, exact);
	r.mine = PASS == kFast ? fast || r.never : !(fast || r.never);
	// margin_abs / |d|, rounded up (1 + 2^-20 covers the reciprocal square root's error). An
	// infinite margin turns distance culling off for this ray: culling is exact only for rays
	// with every direction component within [2^-30, 2^30] (|d|^2 <= 2^60 bounds them above)
	// and |o| < 2^60 (cull_unsafe in common.h); other rays (huge or tiny values, zero components)
	// traverse without it. Rays along an axis meet walls and edges that run along it, where the
	// determinant is a rounding error and t anything: 0.7% of 4 M such rays through vertices of the
	// room differed from the reference with culling.
	const float len2 = r.d[0] * r.d[0] + r.d[1] * r.d[1] + r.d[2] * r.d[2];
	const bool bounded = (a.cull || WT) && in_range && len2 <= 0x1p60f;
	r.abs_margin = bounded && !(zero[0] || zero[1] || zero[2])
	                   ? margin_abs * (__builtin_amdgcn_rsqf(len2) * (1.0f + 0x1p-20f))
	                   : __builtin_inff();
	r.line = bounded && zero[0];
	r.odd = !(__builtin_isfinite(r.inv[0]) && __builtin_isfinite(r.inv[1]) && __builtin_isfinite(r.inv[2]) &&
	          __builtin_isfinite(r.o[0]) && __builtin_isfinite(r.o[1]) && __builtin_isfinite(r.o[2]));
	if (PASS == kFast) {
#pragma unroll
		for (int k = 1; k < 3; ++k) r.inv[k] = zero[k] ? copysignf(kFlat, r.d[k]) : r.inv[k];
	}
	r.tb = __builtin_inff();
	r.ub = r.vb = 0.0f;
	r.idb = kInvalid;
}

// Distance beyond which no box can hold a better candidate (+inf: no culling).
__device__ __forceinline__ float cull_limit(const Ray &r, const KArgs &a) {
	if (!a.cull || !__builtin_isfinite(r.tb)) return __builtin_inff();
	return r.tb + fmaxf(fabsf(r.tb) * a.margin_rel, r.abs_margin);
}

// Conservative slab test of one child box [lo, hi]. Returns the entry distance (tmin), or NaN
// when the box is rejected. WIDE (the watertight mode): the interval is widened by 2^-20 of its
// end points, so that a ray through a box corner (a vertex shared by several triangles) is not
// rejected by the rounding of tmin and tmax. `flagged`: the subtree holds an ill-conditioned
// triangle (cull_unsafe).
//
// A ray with d_x = 0 whose origin lies exactly on the low x side of a triangle's own box meets
// 0 * inf on the x axis, and the exact slab test of that triangle then passes outright, wherever
// the box lies on the other axes and also behind the origin (bvh.hpp:210-217 with
// std::max/std::min argument order). Only the leaf test can reject it, so every box that holds
// o_x has to pass as far as the leaf test's error reaches: everywhere where that error is not
// bounded (without culling, values out of range, flagged subtrees), else where the ray's line, not
// only the part ahead, comes within 2^-8 of the coordinates' magnitude T = |lo| + |hi| + |o|.
// That holds at any angle. Let the triangle's vertices have x_i = 0 (vertex 1, at o_x), X0, X2 >= 0 above
// o_x and D_i the distances of the line from them in the yz plane times |d|. The leaf test's three
// weights times the determinant are N0 = -X2 D1, N1 = X2 D0 - X0 D2, N2 = X0 D1, computed within c 2^-24
// (X0 + X2) |d| T, c about 10, N2 within c 2^-24 X0 |d| T; a hit has all three of one sign within
// that. With X2 >= X0 it follows that |D1| <= c 2^-24 |d| T, the line meets the vertex. Else, r = X2 / X0,
// either the line crosses the edge from vertex 1 to 2 within c 2^-24 T, or D1 <= c 2^-24 |d| T / r and
// D2 <= r |d| T: the nearer of the two is within sqrt(c 2^-24) T = 2^-10.3 T at worst. (A search for
// the worst pair ends at 2^-11.0 T.) The T of a box around the triangle's is at least half of its own.
// The watertight test's sheared vertices are within 2^-21 of theirs.
struct SlabRay {
	float o[3], inv[3];
	bool odd;   // some 1/d or o is not finite
	bool line;  // d_x = 0, and the leaf test's error is bounded (not: cull off, values out of range)
};

__device__ __forceinline__ SlabRay slab_ray(const Ray &r) {
	return {{r.o[0], r.o[1], r.o[2]}, {r.inv[0], r.inv[1], r.inv[2]}, r.odd, r.line};
}

// ODD = false: no lane's ray is odd.
template <bool WIDE = false, bool ODD = true>
__device__ __forceinline__ float child_slab(const SlabRay &r, const float lo[3], const float hi[3], float limit,
                                            bool flagged = false) {
#pragma clang fp contract(off)
	float amin[3], amax[3];
	bool pass = false, line = false;
#pragma unroll
	for (int k = 0; k < 3; ++k) {
		const float t1 = (lo[k] - r.o[k]) * r.inv[k];
		const float t2 = (hi[k] - r.o[k]) * r.inv[k];
		amin[k] = fminf(t1, t2);
		amax[k] = fmaxf(t1, t2);
	}
	if (ODD && r.odd) {
		// 1/d infinite on an axis: a box side through the origin gives NaN in the exact test, and a
		// box containing the origin's coordinate on that axis is unbounded there.
		const bool x_in = !__builtin_isfinite(r.inv[0]) && lo[0] <= r.o[0] && r.o[0] <= hi[0];
		line = x_in && r.line;
		pass = (x_in && (!line || flagged)) ||  // an infinite origin: every node passes
		       !(__builtin_isfinite(r.o[0]) && __builtin_isfinite(r.o[1]) && __builtin_isfinite(r.o[2]));
		if (x_in) {
			amin[0] = -__builtin_inff();
			amax[0] = __builtin_inff();
		}
#pragma unroll
		for (int k = 1; k < 3; ++k) {
			const float tol = line ? 0x1p-8f * (fabsf(lo[k]) + fabsf(hi[k]) + fabsf(r.o[k])) : 0.0f;
			if (__builtin_isfinite(r.inv[k])) {
				amin[k] -= tol * fabsf(r.inv[k]);
				amax[k] += tol * fabsf(r.inv[k]);
			} else if (lo[k] - tol <= r.o[k] && r.o[k] <= hi[k] + tol) {
				amin[k] = -__builtin_inff();
				amax[k] = __builtin_inff();
			}
		}
	}
	const float tmin = fmaxf(fmaxf(amin[0], amin[1]), amin[2]);
	const float tmax = fminf(fminf(amax[0], amax[1]), amax[2]);
	if (pass) return -__builtin_inff();
	float slack = WIDE ? 0x1p-20f * (fabsf(tmin) + fabsf(tmax)) : 0.0f;
	if (WIDE && !__builtin_isfinite(slack)) slack = 0.0f;  // a zero axis: inside or outside, exactly
	const bool hit = (line || tmax >= -slack) && (tmin <= tmax + slack) && (tmin <= limit);
	return hit ? tmin : __builtin_nanf("");
}

// LDS ring stack: the newest `S` entries of each lane stay in LDS, older ones are moved to
// global memory (the entry at depth k of launched thread g lives at spill[(k - S) * threads + g]
// once evicted, so lanes spilling at equal depths write adjacent words). An entry is
// {work entry, sort key of its box entry distance}.
template <int S, int B>
struct Stack {
	uint2 *lds;        // [S][B]
	uint2 *spill;      // shared spill array
	uint32_t thread;   // launched thread index g
	uint32_t threads;  // launched threads
	uint32_t sp;
	__device__ __forceinline__ uint2 *spilled(uint32_t depth) const {
		return spill + (static_cast<uint64_t>(depth - S) * threads + thread);
	}
	__device__ __forceinline__ void push(uint32_t ref, uint32_t key) {
		uint2 *slot = lds + (sp & (S - 1)) * B;
		if (sp >= static_cast<uint32_t>(S)) *spilled(sp) = *slot;
		*slot = make_uint2(ref, key);
		++sp;
	}
	__device__ __forceinline__ uint2 pop() {
		--sp;
		uint2 *slot = lds + (sp & (S - 1)) * B;
		const uint2 e = *slot;
		if (sp >= static_cast<uint32_t>(S)) *slot = *spilled(sp);
		return e;
	}
};

// Sort key of a child hit: the order-preserving integer image of its entry distance with the
// low three bits replaced by the child slot. Clearing bits only lowers the distance the key
// stands for, so re-culling by key at pop stays conservative. -inf (a box that must pass) is
// clamped to -FLT_MAX, which every culling limit admits. Misses sort last.
constexpr uint32_t kMiss = 0xFFFFFFFFu;

// Key of a finite (or +inf) entry distance.
__device__ __forceinline__ uint32_t sort_key_finite(float tmin, int slot) {
	const uint32_t u = __float_as_uint(tmin);
	const uint32_t o = u ^ (static_cast<uint32_t>(static_cast<int32_t>(u) >> 31) | 0x80000000u);
	return (o & ~7u) | static_cast<uint32_t>(slot);
}

__device__ __forceinline__ uint32_t sort_key(float tmin, int slot) {
	return sort_key_finite(fmaxf(tmin, -3.402823466e38f), slot);
}

// Largest key whose decoded distance is within `limit` (not NaN): a key k passes iff
// k <= key_limit(limit). The decoded distance of k is at most the box's entry distance.
__device__ __forceinline__ uint32_t key_limit(float limit) {
	const uint32_t u = __float_as_uint(limit);
	return (u ^ (static_cast<uint32_t>(static_cast<int32_t>(u) >> 31) | 0x80000000u)) | 7u;
}

#define PRT_CE(i, j)                                                                               \
	{                                                                                              \
		const uint32_t lo_ = min(k[i], k[j]);                                                      \
		k[j] = max(k[i], k[j]);                                                                    \
		k[i] = lo_;                                                                                \
	}

// Sorting network for 8 keys (19 compare-exchanges).
__device__ __forceinline__ void sort8(uint32_t k[8]) {
	PRT_CE(0, 2) PRT_CE(1, 3) PRT_CE(4, 6) PRT_CE(5, 7) PRT_CE(0, 4) PRT_CE(1, 5) PRT_CE(2, 6) PRT_CE(3, 7)
	PRT_CE(0, 1) PRT_CE(2, 3) PRT_CE(4, 5) PRT_CE(6, 7) PRT_CE(2, 4) PRT_CE(3, 5) PRT_CE(1, 4) PRT_CE(3, 6)
	PRT_CE(1, 2) PRT_CE(3, 4) PRT_CE(5, 6)
}
#undef PRT_CE

// Children of one node that pass the box test, sorted by entry distance, plus what is needed
// to turn a key back into a stack entry.
struct NodeHits {
	uint32_t key[8];
	uint32_t child_base, lbase;
	uint64_t meta;  // the 8 meta bytes, slot k in bits 8k..8k+7
	__device__ __forceinline__ uint32_t entry(uint32_t key) const {
		const uint32_t m = static_cast<uint32_t>(meta >> ((key << 3) & 63u));
		return child_entry(m & 0xFFu, child_base, lbase);
	}
};

// Key of a child slot whose subtree holds a triangle the build flagged as ill-conditioned
// (cull_unsafe in common.h): the order-preserving image of -FLT_MAX, which no culling limit
// rejects, so such a box is never culled (and is visited before its siblings).
constexpr uint32_t kKeyNoCull = 0x00800000u;

// Tests the children of one node (PASS kFast: by the one-fma bound evaluation). Slots whose bit
// is set in the node's never-cull mask pass whenever the box is hit, at any distance, and take
// the key kKeyNoCull | slot; the other slots of such a node are tested without the limit and
// culled only when popped. `ncull_q` is the quantized node array, which holds the mask of
// both formats (byte 15 of node idx).
// Byte k of a little-endian dword pair, as a float (one v_cvt_f32_ubyteN when k is constant).
__device__ __forceinline__ float byte_f(const uint32_t w[2], int k) {
	return static_cast<float>((w[k >> 2] >> (8 * (k & 3))) & 0xFFu);
}

// Flagged slots that were hit take the never-cull key (their boxes were tested without the
// culling limit).
__device__ __forceinline__ void no_cull_keys(uint32_t key[8], uint32_t ncull) {
#pragma unroll
	for (int k = 0; k < 8; ++k)
		if (((ncull >> k) & 1u) && key[k] != kMiss) key[k] = kKeyNoCull | static_cast<uint32_t>(k);
}

// NC = false: the scene has no flagged triangle (every mask is 0) and the masks are not read.
// WIDE: widened reference-formula intervals (child_slab).
template <class Node, bool NC, bool WIDE, int PASS>
struct ChildTest;

template <bool NC, bool WIDE, int PASS>
struct ChildTest<NodeQ, NC, WIDE, PASS> {
static __device__ __forceinline__ void run(const NodeQ *nodes, const NodeQ * /*ncull_q*/, uint32_t idx, const Ray &r,
                                           float limit, NodeHits &h) {
	const uint4 *src = reinterpret_cast<const uint4 *>(nodes + idx);
	const uint4 w0 = src[0], w1 = src[1], w2 = src[2], w3 = src[3], w4 = src[4];
	const float p[3] = {__uint_as_float(w0.x), __uint_as_float(w0.y), __uint_as_float(w0.z)};
	const float s[3] = {exp2i(static_cast<int8_t>(w0.w & 0xFF)), exp2i(static_cast<int8_t>((w0.w >> 8) & 0xFF)),
	                    exp2i(static_cast<int8_t>((w0.w >> 16) & 0xFF))};
	const uint32_t ncull = NC ? (w0.w >> 24) : 0u;  // never-cull mask (the node's byte 15)
	h.child_base = w1.x;
	h.lbase = leaf_base(w1.y);
	const uint32_t meta_lo = w1.z, meta_hi = w1.w;
	h.meta = static_cast<uint64_t>(meta_lo) | (static_cast<uint64_t>(meta_hi) << 32);
	// qlo x: w2.x w2.y, qlo y: w2.z w2.w, qlo z: w3.x w3.y, qhi x: w3.z w3.w, qhi y: w4.x w4.y, qhi z: w4.z w4.w
	const uint32_t ql[3][2] = {{w2.x, w2.y}, {w2.z, w2.w}, {w3.x, w3.y}};
	const uint32_t qh[3][2] = {{w3.z, w3.w}, {w4.x, w4.y}, {w4.z, w4.w}};

	// Fast test: on axis a the child bound q lies at t = q * step_a + base_a in real arithmetic,
	// with step_a = 2^e_a / d_a and base_a = (p_a - o_a) / d_a. One fma per bound replaces the
	// dequantize / subtract / multiply of the reference formula. Both fp32 evaluations stay
	// within 8 * 2^-24 * |1/d_a| * (255 * 2^e_a + |p_a| + |o_a|) of the real value, so moving the
	// near plane in and the far plane out by 2^-18 times that amount keeps every fast interval
	// around the interval the reference formula gives for the same dequantized box (which the
	// builder already rounded outward). A fast ray guarantees |1/d|, |o| and the scene coordinates
	// are below 2^60, so none of these values overflows; other rays take the reference formula.
	if constexpr (PASS == kFast) {
		// a slot is used iff its meta byte is not 0xFF, i.e. its byte of the complement is not 0
		const uint32_t unused_lo = ~meta_lo, unused_hi = ~meta_hi;
		float step[3], bnear[3], bfar[3];
		uint32_t qn[3][2], qf[3][2];
#pragma unroll
		for (int ax = 0; ax < 3; ++ax) {
			step[ax] = s[ax] * r.inv[ax];
			const float base = (p[ax] - r.o[ax]) * r.inv[ax];
			const float margin = (0x1p-18f * fabsf(r.inv[ax])) * fmaf(255.0f, s[ax], fabsf(p[ax]) + fabsf(r.o[ax]));
			bnear[ax] = base - margin;
			bfar[ax] = base + margin;
			// the near plane is the low bound for 1/d >= 0, the high bound otherwise
			const bool pos = r.inv[ax] >= 0.0f;
			qn[ax][0] = pos ? ql[ax][0] : qh[ax][0];
			qn[ax][1] = pos ? ql[ax][1] : qh[ax][1];
			qf[ax][0] = pos ? qh[ax][0] : ql[ax][0];
			qf[ax][1] = pos ? qh[ax][1] : ql[ax][1];
		}
		// a node with a flagged slot tests every slot without the limit (its unflagged slots are
		// still culled when popped); the flagged slots' keys are replaced below
		const float lim = ncull != 0u ? __builtin_inff() : limit;
#pragma unroll
		for (int k = 0; k < 8; ++k) {
			const uint32_t used = ((k < 4 ? unused_lo : unused_hi) >> (8 * (k & 3))) & 0xFFu;
			float tn[3], tf[3];
#pragma unroll
			for (int ax = 0; ax < 3; ++ax) {
				tn[ax] = fmaf(byte_f(qn[ax], k), step[ax], bnear[ax]);
				tf[ax] = fmaf(byte_f(qf[ax], k), step[ax], bfar[ax]);
			}
			const float tmin = fmaxf(fmaxf(tn[0], tn[1]), tn[2]);
			const float tmax = fminf(fminf(tf[0], tf[1]), tf[2]);
			// the fast bounds are finite (no overflow below 2^60), so no clamp in the key
			const bool hit = used != 0u && tmax >= 0.0f && tmin <= tmax && tmin <= lim;
			h.key[k] = hit ? sort_key_finite(tmin, k) : kMiss;
		}
		if (ncull != 0u) no_cull_keys(h.key, ncull);
		sort8(h.key);
		return;
	}
	// Reference formula on the dequantized box.
	const SlabRay sr = slab_ray(r);
#pragma unroll
	for (int k = 0; k < 8; ++k) {
		const uint32_t meta = ((k < 4 ? meta_lo : meta_hi) >> (8 * (k & 3))) & 0xFFu;
		float lo[3], hi[3];
#pragma unroll
		for (int ax = 0; ax < 3; ++ax) {
			const uint32_t bl = (ql[ax][k >> 2] >> (8 * (k & 3))) & 0xFFu;
			const uint32_t bh = (qh[ax][k >> 2] >> (8 * (k & 3))) & 0xFFu;
			lo[ax] = fmaf(static_cast<float>(bl), s[ax], p[ax]);
			hi[ax] = fmaf(static_cast<float>(bh), s[ax], p[ax]);
		}
		const float tmin = child_slab<WIDE>(sr, lo, hi, ncull != 0u ? __builtin_inff() : limit, (ncull >> k) & 1u);
		const bool hit = meta != kMetaEmpty && !__builtin_isnan(tmin);
		h.key[k] = hit ? sort_key(tmin, k) : kMiss;
	}
	if (ncull != 0u) no_cull_keys(h.key, ncull);
	sort8(h.key);
}
};

template <bool NC, bool WIDE, int PASS>
struct ChildTest<NodeF, NC, WIDE, PASS> {
static __device__ __forceinline__ void run(const NodeF *nodes, const NodeQ *ncull_q, uint32_t idx, const Ray &r,
                                           float limit, NodeHits &hh) {
	const NodeF *n = nodes + idx;
	const uint4 h = *reinterpret_cast<const uint4 *>(n);
	const uint32_t ncull = NC ? reinterpret_cast<const uint32_t *>(ncull_q + idx)[3] >> 24 : 0u;
	hh.child_base = h.x;
	hh.lbase = leaf_base(h.y);
	hh.meta = static_cast<uint64_t>(h.z) | (static_cast<uint64_t>(h.w) << 32);
	float lo[3][8], hi[3][8];
#pragma unroll
	for (int ax = 0; ax < 3; ++ax) {
		const float4 *l4 = reinterpret_cast<const float4 *>(n->lo[ax]);
		const float4 *h4 = reinterpret_cast<const float4 *>(n->hi[ax]);
		const float4 a = l4[0], b = l4[1], c = h4[0], d = h4[1];
		lo[ax][0] = a.x; lo[ax][1] = a.y; lo[ax][2] = a.z; lo[ax][3] = a.w;
		lo[ax][4] = b.x; lo[ax][5] = b.y; lo[ax][6] = b.z; lo[ax][7] = b.w;
		hi[ax][0] = c.x; hi[ax][1] = c.y; hi[ax][2] = c.z; hi[ax][3] = c.w;
		hi[ax][4] = d.x; hi[ax][5] = d.y; hi[ax][6] = d.z; hi[ax][7] = d.w;
	}
	auto test = [&](auto odd) {
#pragma unroll
		for (int k = 0; k < 8; ++k) {
			const uint32_t meta = ((k < 4 ? h.z : h.w) >> (8 * (k & 3))) & 0xFFu;
			const float l[3] = {lo[0][k], lo[1][k], lo[2][k]};
			const float u[3] = {hi[0][k], hi[1][k], hi[2][k]};
			const float tmin = child_slab<WIDE, decltype(odd)::value>(slab_ray(r), l, u, ncull != 0u ? __builtin_inff() : limit,
			                                                          (ncull >> k) & 1u);
			const bool hit = meta != kMetaEmpty && !__builtin_isnan(tmin);
			hh.key[k] = hit ? sort_key(tmin, k) : kMiss;
		}
	};
	if (__ballot(r.odd) != 0ull) test(std::true_type());
	else test(std::false_type());
	if (ncull != 0u) no_cull_keys(hh.key, ncull);
	sort8(hh.key);
}
};

// Lane 0's value in every lane, as a wave-uniform (scalar) value; every lane of the wave must be
// active.
__device__ __forceinline__ uint64_t uniform64(uint64_t v) {
	const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
	const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32));
	return static_cast<uint64_t>(lo) | (static_cast<uint64_t>(hi) << 32);
}

// Writes the finished ray's record in the caller's layout.
__device__ __forceinline__ void write_record(const KArgs &a, uint64_t ray_idx, const Ray &r) {
	Hit h;
	h.t = r.tb;
	h.u = r.ub;
	h.v = r.vb;
	h.id = r.idb;
	write_any(a.mask, a.out + ray_idx * a.stride, h, r.o, r.d);
}

template <bool WT, int PASS>
__device__ __forceinline__ void test_leaf(const TriRec *tris, uint32_t entry, Ray &r) {
	const uint32_t first = leaf_first(entry);
	const uint32_t count = leaf_count(entry);
	float inv[3];  // 1/d as the reference has it (kFast: y and z may hold kFlat)
#pragma unroll
	for (int k = 0; k < 3; ++k)
		inv[k] = PASS == kFast && k > 0 && r.d[k] == 0.0f ? copysignf(__builtin_inff(), r.d[k]) : r.inv[k];
	for (uint32_t m = 0; m < count; ++m) {
		const uint4 *src = reinterpret_cast<const uint4 *>(tris + first + m);
		const uint4 a = src[0], b = src[1], c = src[2];
		const float v[9] = {__uint_as_float(a.x), __uint_as_float(a.y), __uint_as_float(a.z),
		                    __uint_as_float(a.w), __uint_as_float(b.x), __uint_as_float(b.y),
		                    __uint_as_float(b.z), __uint_as_float(b.w), __uint_as_float(c.x)};
		const uint32_t id = c.y;
		float t, u, vv;
		const bool cand = WT ? wt_candidate(v, r.o, r.d, inv, t, u, vv) : exact_candidate(v, r.o, r.d, inv, t, u, vv);
		if (cand && better(t, id, r.tb, r.idb)) {
			r.tb = t;
			r.ub = u;
			r.vb = vv;
			r.idb = id;
		}
	}
}

// The first workgroup of a launch clears the set of the launch that follows and, since the error flags
// of all sets are read together as those of the last launch, the flags of the captured launches' set
// (the last one, just before the list).
__device__ __forceinline__ void clear_next(const KArgs &a) {
	if (blockIdx.x != 0 || !a.next) return;
	if (threadIdx.x < kCounters) a.next[threadIdx.x] = 0ull;
	else if (threadIdx.x == kCounters) (a.left - TraceScratch::kSetWords)[C_ERR] = 0ull;
}

// Waves per SIMD the register allocation must allow. Quantized nodes with an 8-entry LDS stack
// (4 KB per wave): 8 for the plain mode, i.e. at most 64 VGPRs, which it keeps to without a spill;
// the traversal is partly latency-bound (dependent node fetches) and the extra waves hide more of
// it. The other modes carry more state per lane (seed clusters, scene tiles) and would spill
// 2 to 5 registers at 64: they run at 7 waves (72 VGPRs, no spill). Spills inside the loop cost far
// more than a wave of occupancy: the batch step took 8.92 ms at 64 VGPRs with 5 of them, 8.22 ms
// at 72. A 16-entry stack allows 5 waves by LDS alone. The fp32 node test needs 101 VGPRs; held to 96 with
// 2 spilled, 5 waves instead of 4, 8 M rays take 2.33 ms instead of 2.45 in the room and 1.62 instead of
// 1.70 over the icosphere (5.49 instead of 5.01 over a soup of 100,000). With never-cull masks, seeds or scenes
// it would spill more and is left to the compiler (1 = no constraint).
template <int S, int MODE, bool NC, int PASS>
constexpr int kWavesPerEu = PASS == kFast ? (S == 8 ? (MODE == kPlain ? 8 : 7) : 5)
                            : PASS == kAll && !NC && (MODE == kPlain || MODE == kWatertight) ? 5 : 1;

template <class Node, int S, int B, bool COUNT, int MODE, bool NC, int PASS>
__global__ __launch_bounds__(B) __attribute__((amdgpu_waves_per_eu(kWavesPerEu<S, MODE, NC, PASS>))) void k_trace(KArgs a) {
	static_assert(std::is_same<Node, NodeF>::value == (PASS == kAll), "fp32 nodes take one pass");
	unsigned long long *work = a.counter + (PASS == kRest ? C_WORK_REST : C_WORK);
	uint32_t *flags = reinterpret_cast<uint32_t *>(a.counter + C_ERR);  // [0] errors, [1] rays left to kRest
	const uint32_t n_left = PASS == kRest ? flags[1] : 0u;
	if (PASS == kRest && n_left == 0u) return;
	const bool listed = PASS == kRest && n_left <= kLeftMax;
	if (PASS != kRest) clear_next(a);
	bool told = false;  // the list is full: this wave adds nothing to it any more
	constexpr bool MULTI = MODE == kSeededMulti, SEEDED = MODE == kSeeded || MULTI, BATCH = MODE == kBatch;
	__shared__ uint2 lds[S * B];
	const Node *nodes = static_cast<const Node *>(a.nodes);
	const uint32_t lane = threadIdx.x & 63u;
	Stack<S, B> st;
	st.lds = lds + threadIdx.x;
	st.spill = a.spill;
	st.thread = blockIdx.x * B + threadIdx.x;
	st.threads = gridDim.x * B;
	st.sp = 0;

	Ray r;
	uint64_t ray_idx = ~0ull;
	bool active = false;       // lane holds a ray
	uint32_t cur = kInvalid;   // next entry to process (node or leaf)
	uint32_t pend = kInvalid;  // parked leaf, tested in the next triangle phase
	// learned seeding: the entries of the seed clusters (sd[0] the best) and, with several
	// seeds, which of sd[1..3] have been taken from the stack
	uint32_t sd[4] = {kInvalid, kInvalid, kInvalid, kInvalid};
	uint32_t seen = 0u;
	// wave-uniform ray chunk [chunk_next, chunk_end) reserved with one atomic
	uint64_t chunk_next = 0, chunk_end = 0;
	uint32_t chunk_scene = 0;
	bool exhausted = false;
	unsigned long long c_nodes = 0, c_tris = 0, c_leaves = 0, c_nphase = 0, c_tphase = 0, c_culled = 0;

	// Issue priority: 1 while the wave may still reserve rays, 0 once the work is used up. At the
	// end of a launch the waves that still hold reserved rays (the last to finish) then win the
	// issue slots over waves draining their last rays. The SIMD's arbiter otherwise favours the
	// older waves, and the younger ones, which trace about half as many rays, end the launch.
	__builtin_amdgcn_s_setprio(1);
	while (true) {
		// ---- refill finished lanes from the wave's chunk (one ballot when none is idle); the
		// ray loads are amortised over at least `refill` lanes unless the whole wave is idle
		const uint64_t need = __ballot(!active);
		const uint32_t n_need = __popcll(need);
		if (n_need != 0u && !exhausted && (n_need >= a.refill || n_need == __popcll(__ballot(true)))) {
			if (chunk_next >= chunk_end && BATCH && !listed) {
				uint64_t tix = 0;
				if (lane == 0) tix = atomicAdd(work, 1ull);
				tix = uniform64(tix);
				if (tix < a.n_tiles) {
					const uint4 tl = a.tiles[tix];
					chunk_next = static_cast<uint64_t>(tl.x) | (static_cast<uint64_t>(tl.y) << 32);
					chunk_end = chunk_next + tl.z;
					chunk_scene = tl.w;
				} else {
					exhausted = true;
					chunk_next = chunk_end = 0;
					__builtin_amdgcn_s_setprio(0);
				}
			} else if (chunk_next >= chunk_end) {
				uint64_t base = 0;
				if (lane == 0) base = atomicAdd(work, static_cast<unsigned long long>(a.chunk));
				base = uniform64(base);
				chunk_next = base;
				const uint64_t n_work = listed ? n_left : a.n_rays;
				chunk_end = base + a.chunk < n_work ? base + a.chunk : n_work;
				if (base >= n_work) {
					exhausted = true;
					__builtin_amdgcn_s_setprio(0);
				}
			}
			const uint64_t avail = chunk_end > chunk_next ? chunk_end - chunk_next : 0ull;
			// idle lanes below this one
			const uint32_t rank = __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(need >> 32),
			                                                __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(need), 0u));
			if (!active && rank < avail) {
				ray_idx = chunk_next + rank;
				uint32_t scene = chunk_scene;
				if (listed) {
					const unsigned long long e = a.left[ray_idx];
					ray_idx = e & ((1ull << 40) - 1ull);
					scene = static_cast<uint32_t>(e >> 40);
				}
				if (BATCH) {
					const float2 si = a.scene_info[scene];
					load_ray<PASS, MODE == kWatertight>(a, ray_idx, si.x, si.y, r);
					cur = scene;
				} else {
					load_ray<PASS, MODE == kWatertight>(a, ray_idx, a.margin_abs, a.reach, r);
					cur = 0u;
				}
				if (r.never || a.n_nodes == 0) cur = kInvalid;
				pend = kInvalid;
				st.sp = 0;
				active = PASS == kAll || r.mine;
				if (SEEDED && cur != kInvalid) {
					// The lane starts at the best predicted cluster's entry instead of the root,
					// which waits at the bottom of the stack; with several seeds the others sit
					// above the root (the better on top) with their box entry distances. The
					// clusters' subtrees are intersected exactly first and seed the culling
					// distance; the root traversal afterwards covers every triangle except those
					// of the clusters already searched. The best cluster's box is not tested:
					// the leaf test is exact, so a ray that misses it only visits its entry.
					uint4 s4 = make_uint4(0u, 0u, 0u, 0u);  // best first
					if (MULTI) s4 = reinterpret_cast<const uint4 *>(a.seeds)[ray_idx];
					else s4.x = a.seeds[ray_idx];
					sd[0] = s4.x < a.n_clusters ? a.cl_entry[s4.x] : 0u;
					if (sd[0] == 0u) sd[0] = kInvalid;  // no seed, or the cluster is the whole tree
					uint32_t key[4] = {};
					if (MULTI) {
						seen = 0u;
						const uint32_t sc[4] = {s4.x, s4.y, s4.z, s4.w};
#pragma unroll
						for (int q = 1; q < 4; ++q) {
							sd[q] = kInvalid;
							if (q < a.n_seeds && sc[q] < a.n_clusters) {
								const float *bx = a.cl_box + 6ull * sc[q];
								const float lo[3] = {bx[0], bx[1], bx[2]}, hi[3] = {bx[3], bx[4], bx[5]};
								const float tmin = child_slab(slab_ray(r), lo, hi, __builtin_inff());
								const uint32_t ce = a.cl_entry[sc[q]];
								if (ce != 0u && !__builtin_isnan(tmin)) {
									sd[q] = ce;
									key[q] = sort_key(tmin, 0);
								}
							}
						}
					}
					if (sd[0] != kInvalid || (MULTI && (sd[1] & sd[2] & sd[3]) != kInvalid)) {
						st.push(0u, sort_key(-3.402823466e38f, 0));
						if (MULTI) {
#pragma unroll
							for (int q = 3; q >= 1; --q)
								if (sd[q] != kInvalid) st.push(sd[q], key[q]);
						}
						cur = sd[0];  // kInvalid: the next pop takes the best pushed cluster
					}
				}
			}
			if (PASS == kFast && !told) {
				const uint64_t left = __ballot(!active && rank < avail);
				if (left != 0ull) {
					const uint32_t n = static_cast<uint32_t>(__popcll(left));
					uint32_t at = 0;
					if (lane == 0) at = atomicAdd(flags + 1, n);
					at = __builtin_amdgcn_readfirstlane(at);
					told = at + n > kLeftMax;
					if (!active && rank < avail) {
						const uint32_t k = at + __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(left >> 32),
						                                                  __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(left), 0u));
						if (k < kLeftMax) a.left[k] = ray_idx | static_cast<unsigned long long>(BATCH ? chunk_scene : 0u) << 40;
					}
				}
			}
			const uint64_t took = n_need < avail ? n_need : avail;
			chunk_next += took;
		}
		if (__ballot(active) == 0ull) {
			if (exhausted || chunk_next >= chunk_end) {
				if (exhausted) break;
				continue;  // chunk used up with every lane idle: reserve the next one
			}
		}
		if (!active) continue;

		// clusters searched in the seed phase are not searched again: their entries are dropped
		// when the root traversal takes them (from the stack or as a node's nearest child). The
		// clusters are disjoint subtrees, so a cluster's entry is never met inside another
		// cluster's search; the best one is never on the stack, so meeting its entry always
		// means the root traversal reached it. A pushed cluster counts once it has been taken
		// from the stack (one culled there is traversed if the root traversal reaches it).
		auto searched = [&](uint32_t e) {
			if (!SEEDED) return false;
			bool s = e == sd[0];
			if (MULTI) {
#pragma unroll
				for (int q = 1; q < 4; ++q) s |= ((seen >> q) & 1u) && e == sd[q];
			}
			return s;
		};

		// ---- fetch work: pop one entry (a culled one leaves the lane without work for this
		// iteration: no divergent loop over consecutive culled entries); park a leaf if the
		// parking slot is free
		if (cur == kInvalid && st.sp > 0) {
			const uint32_t klim = key_limit(cull_limit(r, a));
			{
				const uint2 e = st.pop();
				if (e.y <= klim) {
					cur = e.x;
					if (searched(cur)) {
						cur = kInvalid;
					} else if (MULTI) {
						// a pushed cluster taken here is searched before anything below it
#pragma unroll
						for (int q = 1; q < 4; ++q) seen |= cur == sd[q] ? (1u << q) : 0u;
					}
				} else if (COUNT) {
					++c_culled;
				}
			}
		}
		if (cur != kInvalid && (cur & kLeafBit) && pend == kInvalid) {
			pend = cur;
			cur = kInvalid;
		}
		if (cur == kInvalid && pend == kInvalid && st.sp == 0) {  // ray finished
			write_record(a, ray_idx, r);
			active = false;
			continue;
		}

		// ---- one phase per iteration for the whole wave: nodes, or the triangles of every
		// parked leaf. Lanes with a parked leaf keep traversing nodes meanwhile; the triangle
		// phase runs when no lane has a node to visit or enough lanes have parked a leaf.
		const uint64_t want_node = __ballot(cur != kInvalid && !(cur & kLeafBit));
		const uint64_t parked = __ballot(pend != kInvalid);
		const uint64_t live = __ballot(true);
		const bool tri_phase = want_node == 0ull || __popcll(parked) * 64u >= __popcll(live) * a.leaf_phase;
		if (COUNT && lane == static_cast<uint32_t>(__ffsll(static_cast<unsigned long long>(live)) - 1)) {
			if (tri_phase) ++c_tphase;
			else ++c_nphase;
		}
		if (tri_phase) {
			if (pend != kInvalid) {
				const uint32_t tri = leaf_first(pend);
				const uint32_t left = leaf_count(pend);
				if (tri + left > a.n_tris) {  // corrupt entry: report, never read
					atomicOr(flags, 1u);
					pend = kInvalid;
					continue;
				}
				test_leaf<MODE == kWatertight, PASS>(a.tris, pend, r);  // the whole leaf (1..4 triangles)
				if (COUNT) c_tris += left;
				pend = kInvalid;
			}
		} else if (cur != kInvalid && !(cur & kLeafBit)) {
			if (cur >= a.n_nodes || st.sp + 7u > a.max_entries) {  // corrupt node or stack bound
				atomicOr(flags, 2u);
				cur = kInvalid;
				continue;
			}
			NodeHits h;
			// the one-fma test's margins also cover the watertight mode's box corners
			ChildTest<Node, NC, MODE == kWatertight, PASS>::run(nodes, a.nodes_q, cur, r, cull_limit(r, a), h);
			if (COUNT) ++c_nodes;
			cur = h.key[0] != kMiss ? h.entry(h.key[0]) : kInvalid;
			if (searched(cur)) cur = kInvalid;
			// farthest first, so the nearest remaining child is on top
#pragma unroll
			for (int k = 7; k >= 1; --k) {
				if (h.key[k] != kMiss) {
					const uint32_t e = h.entry(h.key[k]);
					if (COUNT) c_leaves += (e & kLeafBit) ? 1u : 0u;
					st.push(e, h.key[k]);
				}
			}
		}
	}
	if (COUNT) {
		atomicAdd(a.counter + C_NODES, c_nodes);
		atomicAdd(a.counter + C_TRIS, c_tris);
		atomicAdd(a.counter + C_LEAVES, c_leaves);
		atomicAdd(a.counter + C_NPHASE, c_nphase);
		atomicAdd(a.counter + C_TPHASE, c_tphase);
		atomicAdd(a.counter + C_CULLED, c_culled);
	}
}

// -------------------------------------------------------------- eight lanes per ray, few rays
//
// A launch of few rays lasts as long as its slowest ray's chain of visits, and in k_trace a visit
// is some 300 instructions of one lane after the node's loads (65,536 room rays: 138 us at one wave
// per SIMD, most of it waiting). Here a group of 8 lanes traces a ray: a lane per child slot in the
// node test, per triangle in a leaf. The children's order is a rank (7 lane exchanges instead of
// the sorting network), all pushes are one LDS store, and near and far planes are picked by
// address. A wave holds 8 rays, each traversed at its own pace: pop, node test and leaf test in
// one iteration. Costs more issue slots per ray than k_trace, which takes larger launches. 65,536
// rays: room 137 -> 102 us, 1.5 M-triangle soup 510 -> 325, icosphere camera 153 -> 90. kRest, the second
// pass, tests its lane's child by the reference formula.
constexpr int kWideStack = 32;   // LDS stack entries per ray; deeper ones in the spill array
constexpr int kWidePad = 33;     // entry stride of a ray's stack (the groups' tops in different banks)
constexpr int kWideBlock = 128;

// Value of lane g ^ X of the group (X in 1..7).
template <int X>
__device__ __forceinline__ uint32_t xor_lane(uint32_t v) {
	constexpr int quad = (X & 3) == 1 ? 0xB1 : (X & 3) == 2 ? 0x4E : 0x1B;  // lane ^ 1, ^ 2, ^ 3
	if (X >= 4) v = __builtin_amdgcn_update_dpp(0, v, 0x141, 0xF, 0xF, false);  // row_half_mirror: ^ 7
	constexpr int rest = X >= 4 ? X ^ 7 : X;
	constexpr int q = (rest & 3) == 1 ? 0xB1 : (rest & 3) == 2 ? 0x4E : 0x1B;
	if (rest != 0) v = __builtin_amdgcn_update_dpp(0, v, X >= 4 ? q : quad, 0xF, 0xF, false);
	return v;
}

struct WideHit {
	float t, u, v;
	uint32_t id;
};

template <int X>
__device__ __forceinline__ void wide_best(WideHit &h) {
	const float t = __uint_as_float(xor_lane<X>(__float_as_uint(h.t)));
	const float u = __uint_as_float(xor_lane<X>(__float_as_uint(h.u)));
	const float v = __uint_as_float(xor_lane<X>(__float_as_uint(h.v)));
	const uint32_t id = xor_lane<X>(h.id);
	if (better(t, id, h.t, h.id)) h = {t, u, v, id};
}

template <int MODE, bool NC, int PASS>
__global__ __launch_bounds__(kWideBlock) __attribute__((amdgpu_waves_per_eu(PASS == kFast ? 8 : 6))) void k_trace_wide(KArgs a) {
	static_assert(MODE == kPlain || MODE == kWatertight, "one scene, no seeds");
	__shared__ uint2 lds[kWideBlock / 8][kWidePad];
	uint32_t *flags = reinterpret_cast<uint32_t *>(a.counter + C_ERR);  // [0] errors, [1] rays left to kRest
	const uint32_t n_left = PASS == kRest ? flags[1] : 0u;
	if (PASS == kRest && n_left == 0u) return;
	if (PASS == kFast) clear_next(a);
	const bool listed = PASS == kRest && n_left <= kLeftMax;
	const uint64_t n_work = listed ? n_left : a.n_rays;
	const uint8_t *nodes = static_cast<const uint8_t *>(a.nodes);
	const uint32_t g = threadIdx.x & 7u, group = (blockIdx.x * kWideBlock + threadIdx.x) >> 3;
	const uint32_t groups = gridDim.x * (kWideBlock / 8);
	uint2 *stack = lds[threadIdx.x >> 3];
	auto spilled = [&](uint32_t k) { return a.spill + (static_cast<uint64_t>(k - kWideStack) * groups + group); };
	bool told = false;  // the list of left rays is full
	Ray r;
	uint32_t near_at[3] = {0, 0, 0};  // byte of this lane's near bound on each axis, in the node
	uint64_t work = group;
	bool active = false;
	uint32_t cur = kInvalid, sp = 0;
	for (;;) {
		const bool full = PASS != kFast || __ballot(told) != 0ull;  // the same in every lane
		// ---- a group without a ray takes its next one
		if (!active && work < n_work) {
			load_ray<PASS, MODE == kWatertight>(a, listed ? a.left[work] : work, a.margin_abs, a.reach, r);
			active = r.mine;
			const uint64_t left = __ballot(!active && g == 0u);
			if (left != 0ull && !full) {  // to the second pass: one atomic for the wave's groups
				const uint32_t lane = threadIdx.x & 63u, n = static_cast<uint32_t>(__popcll(left));
				const uint32_t lead = static_cast<uint32_t>(__ffsll(static_cast<unsigned long long>(left))) - 1u;
				uint32_t at = 0;
				if (lane == lead) {
					at = __hip_atomic_load(flags + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
					if (at <= kLeftMax) at = atomicAdd(flags + 1, n);
				}
				at = __builtin_amdgcn_readlane(at, lead);
				told = at + n > kLeftMax;
				const uint32_t k = at + static_cast<uint32_t>(__popcll(left & ((1ull << lane) - 1ull)));
				if (!active && g == 0u && k < kLeftMax) a.left[k] = work;
			}
			if (!active) work += groups;
			cur = r.never || a.n_nodes == 0 ? kInvalid : 0u;
			sp = 0;
#pragma unroll
			for (int ax = 0; ax < 3; ++ax) near_at[ax] = 32u + 8u * ax + (PASS == kRest || r.inv[ax] >= 0.0f ? 0u : 24u) + g;
		}
		if (__ballot(active || work < n_work) == 0ull) break;
		if (!active) continue;
		const float limit = cull_limit(r, a);
		// ---- next entry: the nearest child of the last node, else the stack's top (culled again)
		if (cur == kInvalid) {
			const uint32_t klim = key_limit(limit);
			while (cur == kInvalid && sp > 0) {
				--sp;
				const uint2 e = sp < static_cast<uint32_t>(kWideStack) ? stack[sp] : *spilled(sp);
				if (e.y <= klim) cur = e.x;
			}
		}
		if (cur == kInvalid) {  // ray finished
			if (g == 0u) write_record(a, listed ? a.left[work] : work, r);
			active = false;
			work += groups;
			continue;
		}
		if (!(cur & kLeafBit)) {
			if (cur >= a.n_nodes || sp + 7u > a.max_entries) {  // corrupt node or stack bound
				if (g == 0u) atomicOr(flags, 2u);
				cur = kInvalid;
				continue;
			}
			const uint8_t *node = nodes + static_cast<uint64_t>(cur) * sizeof(NodeQ);
			const uint4 w0 = reinterpret_cast<const uint4 *>(node)[0], w1 = reinterpret_cast<const uint4 *>(node)[1];
			uint32_t qn[3], qf[3];  // near and far bounds (kRest: low and high)
#pragma unroll
			for (int ax = 0; ax < 3; ++ax) {
				qn[ax] = node[near_at[ax]];
				qf[ax] = node[PASS == kRest || r.inv[ax] >= 0.0f ? near_at[ax] + 24u : near_at[ax] - 24u];
			}
			const float p[3] = {__uint_as_float(w0.x), __uint_as_float(w0.y), __uint_as_float(w0.z)};
			const uint32_t ncull = NC ? w0.w >> 24 : 0u;
			const float lim = ncull != 0u ? __builtin_inff() : limit;
			const uint32_t meta = ((g < 4u ? w1.z : w1.w) >> (8u * (g & 3u))) & 0xFFu;
			float sc[3], tmin;
#pragma unroll
			for (int ax = 0; ax < 3; ++ax) sc[ax] = exp2i(static_cast<int8_t>((w0.w >> (8 * ax)) & 0xFF));
			bool hit = meta != kMetaEmpty;
			uint32_t key;
			if constexpr (PASS == kFast) {  // the one-fma bounds of ChildTest<NodeQ>, for this lane's child
				float tn[3], tf[3];
#pragma unroll
				for (int ax = 0; ax < 3; ++ax) {
					const float step = sc[ax] * r.inv[ax];
					const float base = (p[ax] - r.o[ax]) * r.inv[ax];
					const float margin = (0x1p-18f * fabsf(r.inv[ax])) * fmaf(255.0f, sc[ax], fabsf(p[ax]) + fabsf(r.o[ax]));
					tn[ax] = fmaf(static_cast<float>(qn[ax]), step, base - margin);
					tf[ax] = fmaf(static_cast<float>(qf[ax]), step, base + margin);
				}
				tmin = fmaxf(fmaxf(tn[0], tn[1]), tn[2]);
				const float tmax = fminf(fminf(tf[0], tf[1]), tf[2]);
				hit = hit && tmax >= 0.0f && tmin <= tmax && tmin <= lim;
				key = sort_key_finite(tmin, static_cast<int>(g));
			} else {  // its reference formula
				float lo[3], hi[3];
#pragma unroll
				for (int ax = 0; ax < 3; ++ax) {
					lo[ax] = fmaf(static_cast<float>(qn[ax]), sc[ax], p[ax]);
					hi[ax] = fmaf(static_cast<float>(qf[ax]), sc[ax], p[ax]);
				}
				tmin = child_slab<MODE == kWatertight>(slab_ray(r), lo, hi, lim, (ncull >> g) & 1u);
				hit = hit && !__builtin_isnan(tmin);
				key = sort_key(tmin, static_cast<int>(g));
			}
			if (NC && ((ncull >> g) & 1u)) key = kKeyNoCull | g;
			if (!hit) key = kMiss;
			// rank among the group's hits (keys differ in their slot bits)
			uint32_t rank = 0;
			rank += xor_lane<1>(key) < key;
			rank += xor_lane<2>(key) < key;
			rank += xor_lane<3>(key) < key;
			rank += xor_lane<4>(key) < key;
			rank += xor_lane<5>(key) < key;
			rank += xor_lane<6>(key) < key;
			rank += xor_lane<7>(key) < key;
			uint32_t first = min(key, xor_lane<1>(key));
			first = min(first, xor_lane<2>(first));
			first = min(first, xor_lane<7>(first));
			const uint32_t hits = static_cast<uint32_t>(__popcll((__ballot(hit) >> (threadIdx.x & 56u)) & 0xFFull));
			const uint32_t lbase = leaf_base(w1.y);
			// farthest lowest, so the nearest remaining child is on top
			if (hit && rank != 0u) {
				const uint32_t at = sp + hits - 1u - rank;
				const uint2 e = make_uint2(child_entry(meta, w1.x, lbase), key);
				if (at < static_cast<uint32_t>(kWideStack)) stack[at] = e;
				else *spilled(at) = e;
			}
			// the group's other lanes pop these entries
			__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
			__builtin_amdgcn_wave_barrier();
			__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
			sp += hits != 0u ? hits - 1u : 0u;
			const uint32_t fs = first & 7u;
			cur = first != kMiss ? child_entry(((fs < 4u ? w1.z : w1.w) >> (8u * (fs & 3u))) & 0xFFu, w1.x, lbase) : kInvalid;
		}
		if (cur != kInvalid && (cur & kLeafBit)) {
			const uint32_t tri = leaf_first(cur), count = leaf_count(cur);
			cur = kInvalid;
			if (tri + count > a.n_tris) {  // corrupt entry: report, never read
				if (g == 0u) atomicOr(flags, 1u);
				continue;
			}
			// a lane per triangle (1..4), the best of them in every lane
			WideHit h = {__builtin_inff(), 0.0f, 0.0f, kInvalid};
			if (g < count) {
				const uint4 *src = reinterpret_cast<const uint4 *>(a.tris + tri + g);
				const uint4 x = src[0], y = src[1], z = src[2];
				const float v[9] = {__uint_as_float(x.x), __uint_as_float(x.y), __uint_as_float(x.z),
				                    __uint_as_float(x.w), __uint_as_float(y.x), __uint_as_float(y.y),
				                    __uint_as_float(y.z), __uint_as_float(y.w), __uint_as_float(z.x)};
				float inv[3];
#pragma unroll
				for (int k = 0; k < 3; ++k)
					inv[k] = k > 0 && r.d[k] == 0.0f ? copysignf(__builtin_inff(), r.d[k]) : r.inv[k];
				float t, u, vv;
				const bool cand = MODE == kWatertight ? wt_candidate(v, r.o, r.d, inv, t, u, vv) : exact_candidate(v, r.o, r.d, inv, t, u, vv);
				if (cand && better(t, z.y, h.t, h.id)) h = {t, u, vv, z.y};
			}
			wide_best<1>(h);
			wide_best<2>(h);
			wide_best<7>(h);
			if (better(h.t, h.id, r.tb, r.idb)) {
				r.tb = h.t;
				r.ub = h.u;
				r.vb = h.v;
				r.idb = h.id;
			}
		}
	}
}

__global__ void k_zero(unsigned long long *p, int n) {
	if (static_cast<int>(threadIdx.x) < n) p[threadIdx.x] = 0ull;
}

// Before a captured launch, one wave: its set (the last one) and the error flags of the others.
__global__ void k_zero_captured(unsigned long long *sets) {
	constexpr int last = (TraceScratch::kSets - 1) * TraceScratch::kSetWords;
	const int t = threadIdx.x;
	if (t < kCounters) sets[last + t] = 0ull;
	else if (t - kCounters < TraceScratch::kSets - 1) sets[(t - kCounters) * TraceScratch::kSetWords + C_ERR] = 0ull;
}

template <class Node, int S, int B, int MODE, bool NC, int PASS>
void launch_pass(const KArgs &a, uint32_t grid, bool count, hipStream_t st) {
	if (count)
		hipLaunchKernelGGL((k_trace<Node, S, B, true, MODE, NC, PASS>), dim3(grid), dim3(B), 0, st, a);
	else
		hipLaunchKernelGGL((k_trace<Node, S, B, false, MODE, NC, PASS>), dim3(grid), dim3(B), 0, st, a);
}

template <class Node, int S, int B, int MODE, bool NC>
void launch_nc(const KArgs &a, uint32_t grid, bool count, hipStream_t st) {
	if constexpr (std::is_same<Node, NodeF>::value) {
		launch_pass<Node, S, B, MODE, NC, kAll>(a, grid, count, st);
	} else {
		if constexpr (MODE == kPlain || MODE == kWatertight) {
			if (a.wide_grid) hipLaunchKernelGGL((k_trace_wide<MODE, NC, kFast>), dim3(a.wide_grid), dim3(kWideBlock), 0, st, a);
			else launch_pass<Node, S, B, MODE, NC, kFast>(a, grid, count, st);
		} else {
			launch_pass<Node, S, B, MODE, NC, kFast>(a, grid, count, st);
		}
		// seeds do not change a record: the second pass of the learned modes is the plain one
		constexpr int REST = MODE == kSeeded || MODE == kSeededMulti ? kPlain : MODE;
		if constexpr (MODE == kPlain || MODE == kWatertight) {
			if (a.wide_rest) {
				hipLaunchKernelGGL((k_trace_wide<MODE, NC, kRest>), dim3(a.wide_rest), dim3(kWideBlock), 0, st, a);
				return;
			}
		}
		launch_pass<Node, S, B, REST, NC, kRest>(a, grid, count, st);
	}
}

// The batch always reads the never-cull masks (its builds are not read back); the other modes
// only when the scene has a flagged triangle.
template <class Node, int S, int B, int MODE>
void launch_m(const KArgs &a, uint32_t grid, bool count, hipStream_t st) {
	if constexpr (MODE == kBatch) {
		launch_nc<Node, S, B, MODE, true>(a, grid, count, st);
	} else if constexpr (MODE == kWatertight) {  // no distance culling: the masks are not read
		launch_nc<Node, S, B, MODE, false>(a, grid, count, st);
	} else {
		if (a.any_ncull) launch_nc<Node, S, B, MODE, true>(a, grid, count, st);
		else launch_nc<Node, S, B, MODE, false>(a, grid, count, st);
	}
}

template <class Node, int S, int B>
hipError_t launch(const KArgs &a, uint32_t grid, bool count, hipStream_t st) {
	if (a.tiles) launch_m<Node, S, B, kBatch>(a, grid, count, st);
	else if (a.seeds && a.n_seeds > 1) launch_m<Node, S, B, kSeededMulti>(a, grid, count, st);
	else if (a.seeds) launch_m<Node, S, B, kSeeded>(a, grid, count, st);
	else if (a.leaf_test == 1) launch_m<Node, S, B, kWatertight>(a, grid, count, st);
	else launch_m<Node, S, B, kPlain>(a, grid, count, st);
	return hipGetLastError();
}

template <class Node, int B>
hipError_t launch_s(const KArgs &a, uint32_t grid, int S, bool count, hipStream_t st) {
	switch (S) {
	case 8: return launch<Node, 8, B>(a, grid, count, st);
	case 16: return launch<Node, 16, B>(a, grid, count, st);
	default: return hipErrorInvalidValue;
	}
}

template <class Node>
hipError_t launch_b(const KArgs &a, uint32_t grid, int B, int S, bool count, hipStream_t st) {
	switch (B) {
	case 64: return launch_s<Node, 64>(a, grid, S, count, st);
	case 128: return launch_s<Node, 128>(a, grid, S, count, st);
	case 256: return launch_s<Node, 256>(a, grid, S, count, st);
	default: return hipErrorInvalidValue;
	}
}

}  // namespace

#define PRT_TRY(x)                                                                                 \
	do {                                                                                           \
		hipError_t e_ = (x);                                                                       \
		if (e_ != hipSuccess) return e_;                                                           \
	} while (0)

namespace {

// Launch shape and stack bound of one traversal.
struct TracePlan {
	uint32_t grid = 0;         // workgroups
	uint32_t max_entries = 0;  // stack bound 7 * depth + 8
	uint32_t spill_depth = 0;  // stack entries per thread kept in global memory
	uint32_t chunk = 64;       // rays a wave reserves at a time
	uint32_t wide_grid = 0;    // workgroups of k_trace_wide, 0: k_trace
	uint32_t wide_rest = 0;    // of the second pass
};

// several: seeds or scenes, which only k_trace takes.
hipError_t plan_trace(const Bvh8 &b, TraceScratch &s, const TraceParams &p, uint64_t n, bool several, TracePlan &pl) {
	if (s.n_cus == 0) {
		int dev = 0;
		PRT_TRY(hipGetDevice(&dev));
		PRT_TRY(hipDeviceGetAttribute(&s.n_cus, hipDeviceAttributeMultiprocessorCount, dev));
	}
	const int B = p.block, S = p.lds_stack;
	// Automatic: about 6 rays per lane, 16 to 32 waves per CU. A launch ends when each wave's
	// slowest last ray does; with few rays per lane that end weighs more than the latency the
	// extra waves hide (1 Mi rays of the random soup: 0.415 ms at 16 waves per CU against 0.459
	// at 32; 8 Mi room rays: 32 is fastest).
	int wpc = p.waves_per_cu;
	if (wpc <= 0) {
		const uint64_t rays_per_wave_per_cu = static_cast<uint64_t>(s.n_cus) * 64u * 6u;  // 6 rays a lane
		wpc = static_cast<int>(
		    std::min<uint64_t>(32, std::max<uint64_t>(16, (n + rays_per_wave_per_cu - 1) / rays_per_wave_per_cu)));
	}
	const uint64_t waves = static_cast<uint64_t>(s.n_cus) * static_cast<uint64_t>(wpc);
	uint64_t grid64 = (waves * 64 + B - 1) / B;
	// With at most one ray per launched lane a wave reserves a wave's worth: twice that leaves half of
	// the waves without work, which costs a ray's chain of visits, so by the tree's depth; the default of
	// 128 halves the reservations, which cost about 70 ps a ray. 128 against 64, in us: 12 triangles (2 levels)
	// 32,768 rays 30 / 27, 65,536 38 / 40, 262,144 94 / 114; 400 (5) 131,072 rays 92 / 88, 200,000 114 / 121;
	// 8,000 (6) 131,072 rays 179 / 158, 200,000 210 / 218; 20,000 (7) 200,000 rays 257 / 251; 100,000 (8)
	// 262,144 rays 443 / 420; the room (11) 208 / 167 and 263 / 246. Above one ray per lane 128 is the faster
	// (1 Mi icosphere rays 316 against 406 us).
	const uint64_t one_each = std::min<uint64_t>(waves * 64, 37500ull * (std::max(2u, b.depth) - 1u));
	pl.chunk = static_cast<uint32_t>(n <= one_each ? 64 : std::max(64, std::min(1 << 16, p.chunk)));
	const uint64_t need_threads = (n + 63) / 64 * 64;
	grid64 = std::max<uint64_t>(1, std::min<uint64_t>(grid64, (need_threads + B - 1) / B));
	pl.grid = static_cast<uint32_t>(grid64);
	// Eight lanes per ray while the rays take at most one and a half rounds of the chip's 65,536
	// groups (one for the watertight test, which culls nothing). One lane against eight, in us, for
	// room, 1.5 M-triangle soup and icosphere camera: 16,384 rays 121 / 63, 506 / 287, 127 / 76; 98,304
	// rays 160 / 135, 519 / 369, 169 / 96; 131,072 rays 171 / 178, 535 / 555, 178 / 91. Watertight,
	// 65,536 rays: 358 / 300, 1344 / 1211, 231 / 169; 131,072 rays 396 / 484, 1393 / 2021, 261 / 276.
	const uint64_t resident = static_cast<uint64_t>(s.n_cus) * 32 * 8;
	const bool wide = p.node_format != 0 && p.waves_per_cu <= 0 && !p.count_stats && !several;
	const uint32_t wide_groups = static_cast<uint32_t>((std::min(n, resident) * 8 + kWideBlock - 1) / kWideBlock);
	if (wide && n <= (p.leaf_test == 1 ? resident : resident + resident / 2)) pl.wide_grid = wide_groups;
	// The second pass's reference formula is a longer chain for one lane, and its rays are not culled: parallel
	// rays along y (z for the icosphere), one lane against eight, in us, for room, 1.5 M-triangle soup and icosphere:
	// 4,096 rays 591 / 267, 1,519 / 637, 311 / 163; 65,536 rays 693 / 472, 1,976 / 1,646, 405 / 333; 131,072 rays
	// 751 / 705, 2,054 / 2,504, 465 / 364; 262,144 rays 873 / 1,309, 2,465 / 5,210, 619 / 723. Watertight, the room:
	// 4,096 rays 625 / 269, 131,072 rays 790 / 750, 262,144 rays 948 / 1,442.
	if (wide && n <= 2 * resident) pl.wide_rest = wide_groups;
	// stack bound: each visited node pushes at most 7 entries, so 7 * depth + 1 suffice
	pl.max_entries = 7u * std::max(1u, b.depth) + 8u;
	pl.spill_depth = pl.max_entries > static_cast<uint32_t>(S) ? pl.max_entries - S : 1u;
	return hipSuccess;
}

// Spill entries of either kernel of the first pass (k_trace's also serve the second).
uint64_t spill_entries(const TracePlan &pl, const TraceParams &p) {
	const uint64_t one = static_cast<uint64_t>(pl.spill_depth) * pl.grid * p.block;
	const uint64_t deep = pl.max_entries > static_cast<uint32_t>(kWideStack) ? pl.max_entries - kWideStack : 0u;
	return std::max(one, deep * std::max(pl.wide_grid, pl.wide_rest) * (kWideBlock / 8));
}

// Launches the traversal with the given counters (clear: not all 0 yet, cleared here by a kernel)
// and spill array (spill_depth entries per launched thread). `next`, when given, is cleared for
// the launch that follows.
hipError_t run_trace(const Bvh8 &b, const TraceParams &p, const float *rays, uint64_t n, uint32_t mask, void *out,
                     hipStream_t st, unsigned long long *counter, bool clear, unsigned long long *next,
                     unsigned long long *left, uint2 *spill,
                     const TracePlan &pl, float *ms,
                     TraceStats *stats, const SeedArgs *seeds, const BatchArgs *batch) {
	const int B = p.block, S = p.lds_stack;
	KArgs a;
	a.nodes = p.node_format == 0 ? b.nodes_f.ptr : b.nodes_q.ptr;
	a.nodes_q = b.nodes_q.as<NodeQ>();
	a.any_ncull = b.n_ncull != 0u ? 1 : 0;
	a.tris = b.tris.as<TriRec>();
	a.rays = rays;
	a.out = static_cast<uint8_t *>(out);
	a.counter = counter;
	a.next = next;
	a.left = left;
	a.spill = spill;
	a.n_rays = n;
	a.n_nodes = b.n_nodes;
	a.n_tris = static_cast<uint32_t>(b.n_tris);
	a.max_entries = pl.max_entries;
	a.stride = static_cast<uint32_t>(layout_of(mask).size);
	a.mask = mask;
	a.spill_depth = pl.spill_depth;
	a.chunk = pl.chunk;
	a.wide_grid = pl.wide_grid;
	a.wide_rest = pl.wide_rest;
	a.leaf_phase = static_cast<uint32_t>(std::max(1, std::min(64, p.leaf_phase)));
	a.refill = static_cast<uint32_t>(std::max(1, std::min(64, p.refill)));
	a.margin_rel = p.margin_rel;
	a.margin_abs = p.margin_abs;
	a.leaf_test = p.leaf_test;
	// the watertight test's t is not covered by the culling guard (derived for Moller-Trumbore)
	a.cull = p.leaf_test == 1 ? 0 : p.cull;
	if (p.leaf_test == 1 && (seeds || batch)) return hipErrorInvalidValue;  // plain traversal only
	a.seeds = seeds ? seeds->seeds : nullptr;
	a.cl_entry = seeds ? seeds->entry : nullptr;
	a.cl_box = seeds ? seeds->box : nullptr;
	a.n_clusters = seeds ? seeds->count : 0u;
	a.n_seeds = std::max(1, std::min(4, p.n_seeds));
	a.tiles = batch ? batch->tiles : nullptr;
	a.n_tiles = batch ? batch->n_tiles : 0u;
	a.scene_info = batch ? batch->info : nullptr;
	if (batch && (seeds || b.n_nodes < batch->n_scenes || !batch->tiles || !batch->info)) return hipErrorInvalidValue;
	a.reach = 0.0f;
	for (int k = 0; k < 6; ++k) a.reach = std::max(a.reach, std::fabs(b.scene_box[k]));

	if (clear) hipLaunchKernelGGL(k_zero, dim3(1), dim3(64), 0, st, a.counter, static_cast<int>(kCounters));
	hipEvent_t e0 = nullptr, e1 = nullptr;
	if (ms) {
		PRT_TRY(hipEventCreate(&e0));
		PRT_TRY(hipEventCreate(&e1));
		PRT_TRY(hipEventRecord(e0, st));
	}
	const bool count = p.count_stats != 0;
	hipError_t e = p.node_format == 0 ? launch_b<NodeF>(a, pl.grid, B, S, count, st)
	                                  : launch_b<NodeQ>(a, pl.grid, B, S, count, st);
	PRT_TRY(e);
	if (ms) {
		PRT_TRY(hipEventRecord(e1, st));
		PRT_TRY(hipEventSynchronize(e1));
		PRT_TRY(hipEventElapsedTime(ms, e0, e1));
		(void)hipEventDestroy(e0);
		(void)hipEventDestroy(e1);
	}
	if (stats) {
		unsigned long long h[kCounters];
		PRT_TRY(hipMemcpyAsync(h, a.counter, sizeof(h), hipMemcpyDeviceToHost, st));
		PRT_TRY(hipStreamSynchronize(st));
		stats->node_visits = h[C_NODES];
		stats->tri_tests = h[C_TRIS];
		stats->leaf_visits = h[C_LEAVES];
		stats->errors = static_cast<uint32_t>(h[C_ERR]);
		stats->node_phases = h[C_NPHASE];
		stats->tri_phases = h[C_TPHASE];
		stats->culled_pops = h[C_CULLED];
	}
	return hipSuccess;
}

// Allocates the counter sets, all 0. Where `st` is being captured they are cleared on a stream of their own:
// a launch recorded with the graph clears nothing before its first replay, and uncaptured launches
// and reads of the error flags may come before that.
hipError_t new_counters(TraceScratch &s, hipStream_t st, bool captured) {
	constexpr int words = TraceScratch::kSets * TraceScratch::kSetWords;
	PRT_TRY(s.counter.ensure(sizeof(unsigned long long) * (words + kLeftMax)));
	hipStream_t own = nullptr;
	hipError_t e = captured ? hipStreamCreateWithFlags(&own, hipStreamNonBlocking) : hipSuccess;
	if (e == hipSuccess) {
		hipLaunchKernelGGL(k_zero, dim3(1), dim3(64), 0, own ? own : st, s.counter.as<unsigned long long>(), words);
		e = hipGetLastError();
	}
	if (own) {
		if (e == hipSuccess) e = hipStreamSynchronize(own);
		(void)hipStreamDestroy(own);
	}
	if (e != hipSuccess) s.counter.release();
	else s.clean = true;
	return e;
}

}  // namespace

static_assert(static_cast<int>(kCounters) <= TraceScratch::kSetWords, "counter set");

hipError_t trace_bvh8(const Bvh8 &b, TraceScratch &s, const TraceParams &p, const float *rays, uint64_t n,
                      uint32_t mask, void *out, hipStream_t st, float *ms, TraceStats *stats, const SeedArgs *seeds,
                      const BatchArgs *batch) {
	if (n == 0) return hipSuccess;
	TracePlan pl;
	PRT_TRY(plan_trace(b, s, p, n, seeds || batch, pl));
	hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
	PRT_TRY(hipStreamIsCapturing(st, &cap));
	const bool captured = cap != hipStreamCaptureStatusNone;
	if (!s.counter.ptr) PRT_TRY(new_counters(s, st, captured));
	PRT_TRY(s.spill.ensure(sizeof(uint2) * spill_entries(pl, p)));
	// Sets 0 and 1 alternate: a launch clears the set of the next one, which saves that one its
	// clearing kernel (1.3 to 4.3 us). A launch recorded into a graph may be
	// replayed at any time: it has a set of its own and clears it itself.
	const int set = captured ? TraceScratch::kSets - 1 : s.next_set;
	const bool clear = !captured && !s.clean;
	if (captured) hipLaunchKernelGGL(k_zero_captured, dim3(1), dim3(64), 0, st, s.set(0));
	else s.clean = false;
	s.last_set = set;
	PRT_TRY(run_trace(b, p, rays, n, mask, out, st, s.set(set), clear, captured ? nullptr : s.set(set ^ 1),
	                  s.set(TraceScratch::kSets), s.spill.as<uint2>(), pl, ms, stats, seeds, batch));
	if (!captured) {
		s.clean = true;
		s.next_set = set ^ 1;
	}
	return hipSuccess;
}

// ------------------------------------------------------------ traversal without allocation
//
// A device array of fixed size that the library never allocates or frees: the counter in its
// first 256 bytes, the stack spill after it, and the list of rays for the second pass. Every GPU holds its own copy for the life of the
// process; its address on each device is looked up once (hipGetSymbolAddress, with that device
// current) and only that address is passed to kernels or copies. All calls on one GPU share it:
// calls that overlap on one GPU (other streams, other contexts) race.
static __device__ __align__(256) uint8_t scratch[kNoAllocScratchBytes + sizeof(unsigned long long) * kLeftMax];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[kMaxDevices] = {};
}  // namespace

hipError_t noalloc_scratch_setup(int device) {
	if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
	std::lock_guard<std::mutex> g(g_scratch_mu);
	if (g_scratch_ptr[device]) return hipSuccess;
	int cur = -1;
	PRT_TRY(hipGetDevice(&cur));
	if (cur != device) return hipErrorInvalidDevice;  // the caller makes `device` current
	void *ptr = nullptr;
	PRT_TRY(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
	if (!ptr) return hipErrorInvalidSymbol;
	g_scratch_ptr[device] = ptr;
	return hipSuccess;
}

void *noalloc_scratch(int device) {
	if (device < 0 || device >= kMaxDevices) return nullptr;
	std::lock_guard<std::mutex> g(g_scratch_mu);
	return g_scratch_ptr[device];
}

hipError_t trace_bvh8_noalloc(const Bvh8 &b, TraceScratch &s, const TraceParams &p, const float *rays, uint64_t n,
                              uint32_t mask, void *out, hipStream_t st, void *scratch_ptr, uint64_t *need_bytes) {
	if (n == 0) return hipSuccess;
	if (!scratch_ptr) return hipErrorInvalidValue;
	TracePlan pl;
	PRT_TRY(plan_trace(b, s, p, n, false, pl));
	// as many workgroups as the spill part holds (the kernel is persistent: fewer waves trace
	// the same rays)
	const uint64_t per_group = sizeof(uint2) * static_cast<uint64_t>(pl.spill_depth) * p.block;
	const uint64_t fit = (kNoAllocScratchBytes - kNoAllocCounterBytes) / per_group;
	*need_bytes = kNoAllocCounterBytes + per_group;
	if (fit == 0) return hipErrorInvalidValue;
	pl.grid = static_cast<uint32_t>(std::min<uint64_t>(pl.grid, fit));
	if (sizeof(uint2) * spill_entries(pl, p) > kNoAllocScratchBytes - kNoAllocCounterBytes) pl.wide_grid = pl.wide_rest = 0;
	uint8_t *base = static_cast<uint8_t *>(scratch_ptr);
	return run_trace(b, p, rays, n, mask, out, st, reinterpret_cast<unsigned long long *>(base), true, nullptr,
	                 reinterpret_cast<unsigned long long *>(base + kNoAllocScratchBytes),
	                 reinterpret_cast<uint2 *>(base + kNoAllocCounterBytes), pl, nullptr, nullptr, nullptr, nullptr);
}

// ORs the error words of `sets` counter sets at `counter`.
static hipError_t read_errors(TraceScratch &s, const unsigned long long *counter, int sets, hipStream_t st, uint32_t *flags) {
	*flags = 0;
	if (!counter) return hipSuccess;
	const size_t bytes = sizeof(unsigned long long) * TraceScratch::kSetWords * sets;
	if (!s.host_err) {
		hipError_t e = hipHostMalloc(reinterpret_cast<void **>(&s.host_err),
		                             sizeof(unsigned long long) * TraceScratch::kSetWords * TraceScratch::kSets);
		if (e != hipSuccess) return e;
	}
	hipError_t e = hipMemcpyAsync(s.host_err, counter, bytes, hipMemcpyDeviceToHost, st);
	if (e == hipSuccess) e = hipStreamSynchronize(st);
	for (int k = 0; e == hipSuccess && k < sets; ++k)
		*flags |= static_cast<uint32_t>(s.host_err[k * TraceScratch::kSetWords + C_ERR]);
	return e;
}

hipError_t trace_errors_at(TraceScratch &s, const void *counter, hipStream_t st, uint32_t *flags) {
	return read_errors(s, static_cast<const unsigned long long *>(counter), 1, st, flags);
}

#undef PRT_TRY

hipError_t trace_errors(TraceScratch &s, hipStream_t st, uint32_t *flags) {
	return read_errors(s, s.counter.as<unsigned long long>(), TraceScratch::kSets, st, flags);
}

const uint32_t *trace_error_word(const TraceScratch &s) {
	return reinterpret_cast<const uint32_t *>(s.set(s.last_set) + C_ERR);
}

}  // namespace prt
