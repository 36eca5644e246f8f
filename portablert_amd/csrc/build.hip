// GPU BVH8 build for set_tris (replaces the reference's host binned-SAH BVH2,
// include/portableRT/bvh.hpp:58-193, whose result does not matter for the nearest hit except
// for tie order).
//
// Pipeline, all on one stream:
//   1. k_tri_prep     triangle boxes, per-scene centroid bounds, finiteness check
//   2. k_morton       30-bit Morton code of the box centre (Karras 2012) below the scene index
//   3. radix sort     stable LSD, 8-bit digits, hand-written (hist / scan / scatter)
//   4. set_tris: k_ploc_step, k_ploc_tail: clustering over the sorted order, boxes and collapse
//                     costs at each merge. Batches: k_karras, the binary radix tree over the
//                     sorted codes (index tiebreak; the node spanning exactly one scene's keys is
//                     that scene's root), and k_bottomup, boxes leaf to root
//   5. k_collapse     per BVH8 level, 8 lanes per node: children of least expected cost (or the
//                     child of largest area opened until there are `width`); writes fp32 and 8-bit
//                     quantized nodes (bounds rounded outward and verified in fp32)
//   6. k_emit_tris    leaf triangle records in the order the nodes address them
//
// Several scenes build together: the scene index sits above the Morton bits of each key, so
// every scene is one subtree of the radix tree and BVH8 node s is the root of scene s.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "common.h"
#include "internal.h"

namespace prt {
namespace {

constexpr int kBlock = 256;
// Keys per thread of a radix tile (256, 1,024 or 4,096 keys): a tile's rounds are a serial chain, so
// few keys take small tiles that use more CUs (262,144 keys in 64 tiles of 4,096 took 15.5 us a
// scatter), many keys large ones (fewer counts to scan).
inline int sort_items(uint64_t n) { return n <= 32768 ? 1 : n <= (2u << 20) ? 4 : 16; }
constexpr uint32_t kNone = 0xFFFFFFFFu;
constexpr int kMaxLevels = 128;                      // BVH8 levels of a build
constexpr int kSceneShift = 30;                      // key = scene << 30 | 30-bit Morton code

// misc buffer layout (uint32 words)
enum : int {
	M_ERR = 0,         // bit 0 non-finite input, 1 triangle not placed, 2 levels exhausted
	M_NCULL = 1,       // triangles flagged by cull_unsafe (never culled by distance)
	M_PTILES = 2,      // clustering: tiles of the cluster list a step reads, by parity of the step,
	M_PSTRIDE = 4,     // and how far apart they are
	M_PHELD = 6,       // clustering: the step that found at most kTailMax clusters (held_by), or 0
	M_PDONE = 7,       // clustering: finished
	M_LCNT = 8,        // per BVH8 level, 64 bits: its nodes, and the triangles of the level above's leaves
	M_LBASE = M_LCNT + 2 * (kMaxLevels + 2),  // first node of each BVH8 level
	M_TBASE = M_LBASE + kMaxLevels + 2,       // first leaf triangle of each level
	M_SCENE = M_TBASE + kMaxLevels + 2,  // per scene 12 words: ordered centroid min xyz, max xyz, box min, max
	M_PER_SCENE = 12
};
constexpr uint32_t misc_words(uint32_t scenes) { return M_SCENE + M_PER_SCENE * scenes; }

__device__ __forceinline__ uint32_t f2o(float f) {
	const uint32_t u = __float_as_uint(f);
	return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float o2f(uint32_t u) {
	return __uint_as_float((u & 0x80000000u) ? (u & 0x7FFFFFFFu) : ~u);
}

__global__ __launch_bounds__(kBlock) void k_init_misc(uint32_t *misc, uint32_t words) {
	const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
	if (i < words) {
		uint32_t v = 0;
		if (i >= M_SCENE) {
			const uint32_t k = (i - M_SCENE) % M_PER_SCENE;  // min words start +inf, max words -inf
			v = f2o(((k / 3) & 1u) ? -__builtin_inff() : __builtin_inff());
		}
		misc[i] = v;
	}
}

// Scene of input triangle i: last s with off[s] <= i (off has scenes + 1 entries).
__device__ __forceinline__ uint32_t scene_of(const uint32_t *off, uint32_t scenes, uint32_t i) {
	uint32_t lo = 0, hi = scenes;  // off[lo] <= i < off[hi]
	while (hi - lo > 1) {
		const uint32_t mid = (lo + hi) >> 1;
		if (off[mid] <= i) lo = mid;
		else hi = mid;
	}
	return lo;
}

__device__ __forceinline__ void scene_atomics(uint32_t *w, const float c[3], const float cmax[3], const float smn[3],
                                              const float smx[3]) {
#pragma unroll
	for (int k = 0; k < 3; ++k) {
		atomicMin(w + k, f2o(c[k]));
		atomicMax(w + 3 + k, f2o(cmax[k]));
		atomicMin(w + 6 + k, f2o(smn[k]));
		atomicMax(w + 9 + k, f2o(smx[k]));
	}
}

constexpr int kPrepBlock = 1024;

// Triangle boxes (the scene index in the w word of the lower corner, the never-cull flag in the
// w word of the upper corner) and per-scene centroid and
// vertex bounds. The bounds are reduced over the workgroup before the atomics when all of its
// triangles belong to one scene (one set of 12 atomics per 1024 triangles: same-address
// atomics serialise), else per lane.
__global__ __launch_bounds__(kPrepBlock) void k_tri_prep(const float *__restrict__ tris, uint32_t n,
                                                         const uint32_t *__restrict__ off, uint32_t scenes,
                                                         float4 *__restrict__ tbox, uint32_t *misc) {
	__shared__ float red[kPrepBlock / 64][12];
	__shared__ uint32_t mixed;
	const uint32_t i = blockIdx.x * kPrepBlock + threadIdx.x;
	const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
	if (threadIdx.x == 0) mixed = 0u;
	float c[3] = {__builtin_inff(), __builtin_inff(), __builtin_inff()};
	float cmax[3] = {-__builtin_inff(), -__builtin_inff(), -__builtin_inff()};
	float smn[3] = {__builtin_inff(), __builtin_inff(), __builtin_inff()};
	float smx[3] = {-__builtin_inff(), -__builtin_inff(), -__builtin_inff()};
	const uint32_t scene = (i < n && scenes > 1) ? scene_of(off, scenes, i) : 0u;
	if (i < n) {
		float v[9];
#pragma unroll
		for (int k = 0; k < 9; ++k) v[k] = tris[9ull * i + k];
		bool finite = true;
#pragma unroll
		for (int k = 0; k < 9; ++k) finite &= __builtin_isfinite(v[k]);
		if (!finite) atomicOr(misc + M_ERR, 1u);
		float lo[3], hi[3];
#pragma unroll
		for (int k = 0; k < 3; ++k) {
			lo[k] = fminf(v[k], fminf(v[3 + k], v[6 + k]));
			hi[k] = fmaxf(v[k], fmaxf(v[3 + k], v[6 + k]));
			c[k] = cmax[k] = 0.5f * lo[k] + 0.5f * hi[k];
			smn[k] = lo[k];
			smx[k] = hi[k];
		}
		tbox[2ull * i] = make_float4(lo[0], lo[1], lo[2], __uint_as_float(scene));
		// w of the upper corner: the distance-culling guard's flag (cull_unsafe, common.h)
		const bool unsafe = cull_unsafe(v);
		if (unsafe) atomicAdd(misc + M_NCULL, 1u);
		tbox[2ull * i + 1] = make_float4(hi[0], hi[1], hi[2], __uint_as_float(unsafe ? 1u : 0u));
	}
	// the block's first triangle decides the scene the block reduces for
	const uint32_t first = blockIdx.x * kPrepBlock;
	const uint32_t s0 = scenes > 1 ? scene_of(off, scenes, first) : 0u;
	__syncthreads();
	if (i < n && scene != s0) mixed = 1u;
	__syncthreads();
	const bool block_mixed = mixed != 0u;  // the block spans a scene boundary (rare)
	const uint32_t ws = __shfl(scene, 0);
	if (block_mixed && __ballot(i < n && scene != ws) != 0ull) {  // this wave spans it: per lane
		if (i < n) scene_atomics(misc + M_SCENE + M_PER_SCENE * scene, c, cmax, smn, smx);
		return;
	}
#pragma unroll
	for (int k = 0; k < 3; ++k) {
		for (int sh = 32; sh > 0; sh >>= 1) {
			c[k] = fminf(c[k], __shfl_xor(c[k], sh));
			cmax[k] = fmaxf(cmax[k], __shfl_xor(cmax[k], sh));
			smn[k] = fminf(smn[k], __shfl_xor(smn[k], sh));
			smx[k] = fmaxf(smx[k], __shfl_xor(smx[k], sh));
		}
	}
	if (block_mixed) {  // uniform wave in a mixed block: one set of atomics per wave
		if (lane == 0 && !__builtin_isnan(c[0])) scene_atomics(misc + M_SCENE + M_PER_SCENE * ws, c, cmax, smn, smx);
		return;
	}
	if (lane == 0) {
#pragma unroll
		for (int k = 0; k < 3; ++k) {
			red[wave][k] = c[k];
			red[wave][3 + k] = cmax[k];
			red[wave][6 + k] = smn[k];
			red[wave][9 + k] = smx[k];
		}
	}
	__syncthreads();
	if (threadIdx.x < 12) {
		const uint32_t k = threadIdx.x;
		const bool is_min = ((k / 3) & 1u) == 0u;  // centroid min, centroid max, box min, box max
		float r = red[0][k];
		for (int w = 1; w < kPrepBlock / 64; ++w) r = is_min ? fminf(r, red[w][k]) : fmaxf(r, red[w][k]);
		if (!__builtin_isnan(r)) {  // lanes past n contribute the identities +-inf
			uint32_t *dst = misc + M_SCENE + M_PER_SCENE * s0 + k;
			if (is_min) atomicMin(dst, f2o(r));
			else atomicMax(dst, f2o(r));
		}
	}
}

__device__ __forceinline__ uint32_t spread10(uint32_t x) {
	x &= 0x3FFu;
	x = (x | (x << 16)) & 0x030000FFu;
	x = (x | (x << 8)) & 0x0300F00Fu;
	x = (x | (x << 4)) & 0x030C30C3u;
	x = (x | (x << 2)) & 0x09249249u;
	return x;
}

// 1 / half-area of a scene's box (1 for an empty or flat scene).
__device__ __forceinline__ double scene_scale(const uint32_t *misc, uint32_t s) {
	const uint32_t *b = misc + M_SCENE + M_PER_SCENE * s + 6;
	const double dx = static_cast<double>(o2f(b[3])) - o2f(b[0]), dy = static_cast<double>(o2f(b[4])) - o2f(b[1]),
	             dz = static_cast<double>(o2f(b[5])) - o2f(b[2]);
	const double a = dx * dy + dx * dz + dy * dz;
	return (a > 0.0 && a < 1e300) ? 1.0 / a : 1.0;
}

__global__ __launch_bounds__(kBlock) void k_morton(const float4 *__restrict__ tbox, uint32_t n,
                                                   const uint32_t *misc, uint64_t *__restrict__ keys,
                                                   uint32_t *__restrict__ vals, uint32_t *__restrict__ tri_dest,
                                                   double *scale, uint32_t scenes) {
	const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
	if (i >= n) return;
	if (scale) {  // least-cost collapse: the scenes' area scales
		for (uint32_t s = i; s < scenes; s += n) scale[s] = scene_scale(misc, s);
	}
	const float4 lo = tbox[2ull * i], hi = tbox[2ull * i + 1];
	const uint32_t scene = __float_as_uint(lo.w);
	const uint32_t *cb = misc + M_SCENE + M_PER_SCENE * scene;
	const float c[3] = {0.5f * lo.x + 0.5f * hi.x, 0.5f * lo.y + 0.5f * hi.y, 0.5f * lo.z + 0.5f * hi.z};
	uint32_t q[3];
#pragma unroll
	for (int k = 0; k < 3; ++k) {
		const float mn = o2f(cb[k]), mx = o2f(cb[3 + k]);
		const float ext = mx - mn;
		float x = ext > 0.0f ? (c[k] - mn) / ext : 0.0f;
		x = fminf(fmaxf(x * 1024.0f, 0.0f), 1023.0f);
		q[k] = static_cast<uint32_t>(x);
	}
	keys[i] = (static_cast<uint64_t>(scene) << kSceneShift) | (spread10(q[0]) << 2) | (spread10(q[1]) << 1) |
	          spread10(q[2]);
	vals[i] = i;
	tri_dest[i] = kNone;  // not placed yet
}

// ------------------------------------------------------------------------- radix sort

template <int kSortItems>
__global__ __launch_bounds__(kBlock) void k_hist(const uint64_t *__restrict__ keys, uint32_t n, int shift,
                                                 uint32_t *__restrict__ hist, uint32_t tiles) {
	__shared__ uint32_t h[256];
	h[threadIdx.x] = 0;
	__syncthreads();
	const uint64_t base = static_cast<uint64_t>(blockIdx.x) * kBlock * kSortItems;
#pragma unroll 4
	for (int r = 0; r < kSortItems; ++r) {
		const uint64_t i = base + static_cast<uint64_t>(r) * kBlock + threadIdx.x;
		if (i < n) atomicAdd(&h[(keys[i] >> shift) & 0xFFu], 1u);
	}
	__syncthreads();
	hist[static_cast<uint64_t>(threadIdx.x) * tiles + blockIdx.x] = h[threadIdx.x];
}

constexpr int kScanItems = 16;                 // histogram entries per thread
constexpr int kScanSeg = kBlock * kScanItems;  // entries per segment

// Exclusive scan of hist (digit-major: entry d * tiles + t) in two levels: each segment of
// 4096 entries is scanned in place by one workgroup and its total goes to seg[]; the scatter scans
// up to kBlock totals itself (k_scan more) and adds that of segment entry / 4096.
__global__ __launch_bounds__(kBlock) void k_scan_seg(uint32_t *hist, uint32_t total, uint32_t *seg) {
	__shared__ uint32_t part[kBlock];
	const uint64_t base = static_cast<uint64_t>(blockIdx.x) * kScanSeg + static_cast<uint64_t>(threadIdx.x) * kScanItems;
	uint32_t v[kScanItems];
	uint32_t s = 0;
#pragma unroll
	for (int k = 0; k < kScanItems; ++k) {
		v[k] = base + k < total ? hist[base + k] : 0u;
		s += v[k];
	}
	part[threadIdx.x] = s;
	__syncthreads();
	for (int sh = 1; sh < kBlock; sh <<= 1) {
		const uint32_t a = threadIdx.x >= static_cast<uint32_t>(sh) ? part[threadIdx.x - sh] : 0u;
		__syncthreads();
		part[threadIdx.x] += a;
		__syncthreads();
	}
	uint32_t run = part[threadIdx.x] - s;
#pragma unroll
	for (int k = 0; k < kScanItems; ++k) {
		if (base + k < total) hist[base + k] = run;
		run += v[k];
	}
	if (threadIdx.x == kBlock - 1) seg[blockIdx.x] = part[threadIdx.x];
}

// Exclusive scan of a short array in place, one workgroup.
__global__ __launch_bounds__(1024) void k_scan(uint32_t *hist, uint32_t total) {
	__shared__ uint32_t part[1024];
	const uint32_t per = (total + 1023) / 1024;
	const uint32_t b = threadIdx.x * per;
	const uint32_t e = min(total, b + per);
	uint32_t s = 0;
	for (uint32_t i = b; i < e; ++i) s += hist[i];
	part[threadIdx.x] = s;
	__syncthreads();
	for (int off = 1; off < 1024; off <<= 1) {
		const uint32_t v = threadIdx.x >= static_cast<uint32_t>(off) ? part[threadIdx.x - off] : 0u;
		__syncthreads();
		part[threadIdx.x] += v;
		__syncthreads();
	}
	uint32_t run = part[threadIdx.x] - s;
	for (uint32_t i = b; i < e; ++i) {
		const uint32_t x = hist[i];
		hist[i] = run;
		run += x;
	}
}

// Stable scatter through LDS. A tile's keys are loaded at once (kSortItems per thread), ranked
// in index order (round-major, then wave, then lane; equal digits matched within a wave with
// eight ballots) and placed in LDS in digit order; the tile is then written out so that
// consecutive threads write consecutive positions of a digit's run. The tile's count of a digit
// is the difference of two consecutive entries of the scanned histogram: it is digit-major, so
// the entry after a digit's last tile is the next digit's first.
template <int kSortItems>
__global__ __launch_bounds__(kBlock) void k_scatter(const uint64_t *__restrict__ kin, const uint32_t *__restrict__ vin,
                                                    uint64_t *__restrict__ kout, uint32_t *__restrict__ vout,
                                                    uint32_t n, int shift, const uint32_t *__restrict__ hist,
                                                    const uint32_t *__restrict__ seg, uint32_t n_seg, uint32_t tiles) {
	constexpr int kSortTile = kBlock * kSortItems;
	__shared__ uint64_t skey[kSortTile];
	__shared__ uint32_t sval[kSortTile];
	__shared__ uint32_t run[256];                // next tile position of each digit
	__shared__ uint32_t delta[256];              // output position minus tile position, per digit
	__shared__ uint32_t wtot[kBlock / 64];
	__shared__ uint8_t wcnt[kBlock / 64][256];  // keys of each digit in each wave of a round (<= 64)
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	const uint32_t d = threadIdx.x;
	const uint64_t total = 256ull * tiles;
	const uint64_t e = static_cast<uint64_t>(d) * tiles + blockIdx.x;
	const uint32_t h0 = hist[e], h1 = e + 1 < total ? hist[e + 1] : n;
	const uint64_t base = static_cast<uint64_t>(blockIdx.x) * kSortTile;
	uint64_t kk[kSortItems];
	uint32_t vv[kSortItems];
#pragma unroll
	for (int r = 0; r < kSortItems; ++r) {
		const uint64_t i = base + static_cast<uint64_t>(r) * kBlock + threadIdx.x;
		kk[r] = i < n ? kin[i] : 0ull;
		vv[r] = i < n ? vin[i] : 0u;
	}
	// inclusive scan over the workgroup's 256 threads
	auto scan = [&](uint32_t v) {
		for (int sh = 1; sh < 64; sh <<= 1) {
			const uint32_t o = __shfl_up(v, sh);
			if (lane >= sh) v += o;
		}
		if (lane == 63) wtot[wave] = v;
		__syncthreads();
		for (int w = 0; w < wave; ++w) v += wtot[w];
		__syncthreads();
		return v;
	};
	uint32_t s0 = 0, s1 = 0;  // what the segments before add to h0 and h1
	if (n_seg <= static_cast<uint32_t>(kBlock)) {
		const uint32_t v = d < n_seg ? seg[d] : 0u;
		delta[d] = scan(v) - v;
		__syncthreads();
		s0 = delta[e / kScanSeg];
		s1 = e + 1 < total ? delta[(e + 1) / kScanSeg] : 0u;
	} else {
		s0 = seg[e / kScanSeg];
		s1 = e + 1 < total ? seg[(e + 1) / kScanSeg] : 0u;
	}
	const uint32_t g0 = h0 + s0, cnt = h1 + s1 - g0;
	// exclusive scan of the tile's digit counts: each digit's first tile position
	const uint32_t lofs = scan(cnt) - cnt;
	run[d] = lofs;
	delta[d] = g0 - lofs;
	const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
	for (int r = 0; r < kSortItems; ++r) {
#pragma unroll
		for (int w = 0; w < kBlock / 64; ++w) wcnt[w][threadIdx.x] = 0;
		__syncthreads();
		const uint64_t i = base + static_cast<uint64_t>(r) * kBlock + threadIdx.x;
		const bool act = i < n;
		const uint64_t k = kk[r];
		const uint32_t digit = static_cast<uint32_t>(k >> shift) & 0xFFu;
		uint64_t peers = __ballot(act);
#pragma unroll
		for (int b = 0; b < 8; ++b) {
			const bool bit = (digit >> b) & 1u;
			const uint64_t m = __ballot(bit);
			peers &= bit ? m : ~m;
		}
		const uint32_t rank = __popcll(peers & lt);
		if (act && rank == 0) wcnt[wave][digit] = static_cast<uint8_t>(__popcll(peers));
		__syncthreads();
		if (act) {
			uint32_t pos = run[digit] + rank;
			for (int w = 0; w < wave; ++w) pos += wcnt[w][digit];
			skey[pos] = k;
			sval[pos] = vv[r];
		}
		__syncthreads();
		uint32_t add = 0;
#pragma unroll
		for (int w = 0; w < kBlock / 64; ++w) add += wcnt[w][threadIdx.x];
		run[threadIdx.x] += add;
	}
	__syncthreads();
	const uint32_t m = static_cast<uint32_t>(min(static_cast<uint64_t>(kSortTile), n - base));
	for (uint32_t j = threadIdx.x; j < m; j += kBlock) {
		const uint64_t k = skey[j];
		const uint32_t g = delta[static_cast<uint32_t>(k >> shift) & 0xFFu] + j;
		kout[g] = k;
		vout[g] = sval[j];
	}
}

// ------------------------------------------------------------------------ Karras 2012

struct BinTree {
	uint4 *link;       // internal nodes: left, right, first sorted triangle, triangle count
	uint32_t *parent, *flag;  // radix tree: parent of every node, arrivals at an internal one
	uint32_t *plan;    // internal nodes: how the least-cost collapse splits them (make_plan), or null
	float4 *box;       // 2 per node: lo, hi
	uint32_t n;        // leaves; internal nodes 0..n-2, leaf j is node (n-1)+j
	__device__ __forceinline__ uint32_t first(uint32_t x) const { return x >= n - 1 ? x - (n - 1) : link[x].z; }
	__device__ __forceinline__ uint32_t count(uint32_t x) const { return x >= n - 1 ? 1u : link[x].w; }
};

__device__ __forceinline__ int delta(const uint64_t *keys, uint32_t n, int i, int j) {
	if (j < 0 || j >= static_cast<int>(n)) return -1;
	const uint64_t a = keys[i], b = keys[j];
	if (a != b) return __clzll(a ^ b);
	return 64 + __clz(static_cast<uint32_t>(i) ^ static_cast<uint32_t>(j));
}

__global__ __launch_bounds__(kBlock) void k_karras(const uint64_t *__restrict__ keys, BinTree t,
                                                   uint32_t *__restrict__ scene_root) {
	const int n = static_cast<int>(t.n);
	const int i = blockIdx.x * kBlock + threadIdx.x;
	if (i >= n - 1) return;
	const int d = (delta(keys, n, i, i + 1) - delta(keys, n, i, i - 1)) >= 0 ? 1 : -1;
	const int dmin = delta(keys, n, i, i - d);
	int lmax = 2;
	while (delta(keys, n, i, i + lmax * d) > dmin) lmax <<= 1;
	int l = 0;
	for (int s = lmax >> 1; s >= 1; s >>= 1)
		if (delta(keys, n, i, i + (l + s) * d) > dmin) l += s;
	const int j = i + l * d;
	const int dnode = delta(keys, n, i, j);
	int s = 0, div = 2, step;
	do {
		step = (l + div - 1) / div;
		if (delta(keys, n, i, i + (s + step) * d) > dnode) s += step;
		div <<= 1;
	} while (step > 1);
	const int gamma = i + s * d + min(d, 0);
	const uint32_t lc = (min(i, j) == gamma) ? static_cast<uint32_t>(n - 1 + gamma) : static_cast<uint32_t>(gamma);
	const uint32_t rc = (max(i, j) == gamma + 1) ? static_cast<uint32_t>(n - 1 + gamma + 1) : static_cast<uint32_t>(gamma + 1);
	t.parent[lc] = static_cast<uint32_t>(i);
	t.parent[rc] = static_cast<uint32_t>(i);
	const int lo = min(i, j), hi = max(i, j);
	t.link[i] = make_uint4(lc, rc, static_cast<uint32_t>(lo), static_cast<uint32_t>(hi - lo + 1));
	t.flag[i] = 0;
	if (i == 0) t.parent[0] = kNone;
	// the keys of one scene share the bits above the Morton code and no other key does, so
	// exactly one node spans them: the one whose range ends at both scene boundaries
	const uint64_t sc = keys[lo] >> kSceneShift;
	if ((keys[hi] >> kSceneShift) == sc && (lo == 0 || (keys[lo - 1] >> kSceneShift) != sc) &&
	    (hi == n - 1 || (keys[hi + 1] >> kSceneShift) != sc))
		scene_root[sc] = static_cast<uint32_t>(i);
}

// Scene roots before the radix tree: none for an empty scene, the leaf for a one-triangle
// scene; scenes of two or more triangles get their internal root from k_karras.
__global__ __launch_bounds__(kBlock) void k_scene_init(const uint32_t *__restrict__ off, uint32_t scenes, uint32_t n,
                                                       uint32_t *__restrict__ scene_root) {
	const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
	if (s >= scenes) return;
	const uint32_t b = scenes > 1 ? off[s] : 0u, e = scenes > 1 ? off[s + 1] : n;
	scene_root[s] = (e - b == 1u) ? (n - 1u + b) : kNone;
}

// Boxes that one thread writes and a thread of another workgroup reads in the same launch go
// through device-scope atomic 8-byte stores and loads, which are coherent across the XCDs'
// separate L2 caches without writing back a whole L2 as a device-scope fence does.
__device__ __forceinline__ uint64_t pack2(float a, float b) {
	return static_cast<uint64_t>(__float_as_uint(a)) | (static_cast<uint64_t>(__float_as_uint(b)) << 32);
}
__device__ __forceinline__ void st_box(float4 *box, uint32_t node, float4 lo, float4 hi) {
	uint64_t *p = reinterpret_cast<uint64_t *>(box + 2ull * node);
	__hip_atomic_store(p + 0, pack2(lo.x, lo.y), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
	__hip_atomic_store(p + 1, pack2(lo.z, 0.0f), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
	__hip_atomic_store(p + 2, pack2(hi.x, hi.y), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
	__hip_atomic_store(p + 3, pack2(hi.z, hi.w), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void ld_box(const float4 *box, uint32_t node, float4 &lo, float4 &hi) {
	const uint64_t *p = reinterpret_cast<const uint64_t *>(box + 2ull * node);
	uint64_t w[4];
#pragma unroll
	for (int k = 0; k < 4; ++k) w[k] = __hip_atomic_load(p + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
	lo = make_float4(__uint_as_float(static_cast<uint32_t>(w[0])), __uint_as_float(static_cast<uint32_t>(w[0] >> 32)),
	                 __uint_as_float(static_cast<uint32_t>(w[1])), 0.0f);
	hi = make_float4(__uint_as_float(static_cast<uint32_t>(w[2])), __uint_as_float(static_cast<uint32_t>(w[2] >> 32)),
	                 __uint_as_float(static_cast<uint32_t>(w[3])), __uint_as_float(static_cast<uint32_t>(w[3] >> 32)));
}
// Waits until this lane's earlier stores are complete (device-scope atomic stores are then
// visible to every CU), so the flag increment that follows publishes them.
__device__ __forceinline__ void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// ------------------------------------------- collapse costs (surface-area heuristic, SAH)
//
// Cost-optimal collapse of the binary tree into nodes of at most `width` children, by the
// dynamic program of Ylitie, Karras and Laine 2017 ("Efficient incoherent ray traversal on GPUs
// through compressed wide BVHs", section 3.1). For binary node x and i in 1..7 slots, C(x, i) is
// the least expected cost of x's subtree when it may fill i child slots of the node above it:
//   C(x, 1) = min(leaf(x), A(x) * kCostNode + split(x, width))
//   C(x, i) = min(C(x, i - 1), split(x, i))                               for i >= 2
//   split(x, i) = min over k in 1..i-1 of C(left(x), k) + C(right(x), i - k)
//   leaf(x) = A(x) * kCostTri * P(x) if x holds at most leaf_size triangles, else +inf
// with A the half surface area of x's box relative to its scene's box (computed in double, so
// coordinates near 1e19 or 1e-19 neither overflow nor vanish) and P the triangle count; a single
// triangle costs A * kCostTri in any number of slots. A row holds C(x, 1..7). Rows of internal nodes are computed where the tree is built (at the
// merge for the clustered tree, in the bottom-up box pass for the radix tree); rows of binary
// leaves are recomputed from their boxes wherever they are needed.
constexpr float kCostNode = 1.0f;
constexpr float kCostTri = 0.6f;  // swept 0.2-1.5 on the room: 0.6 traces fastest
constexpr int kCostRow = 8;

struct CostCtx {
	float *row;             // kCostRow floats per binary internal node, or null: greedy collapse
	uint32_t scenes;        // scenes of the build (one: no key is read for a node's scene)
	const double *scale;    // per scene: 1 / half-area of the scene box
	const uint64_t *keys;   // sorted keys: the scene of binary node b is keys[first[b]] >> 30
	const uint32_t *param;  // per scene leaf_size | width << 8, or null: leaf_size and width below
	int leaf_size;
	int width;
};

// Leaf size and node width of scene `scene` (per-scene parameters when given).
__device__ __forceinline__ void scene_shape(const CostCtx &c, uint32_t scene, int &ls, int &w) {
	int leaf_size = c.leaf_size, width = c.width;
	if (c.param) {
		const uint32_t pr = c.param[scene];
		leaf_size = static_cast<int>(pr & 0xFFu);
		width = static_cast<int>((pr >> 8) & 0xFFu);
	}
	ls = max(1, min(kMaxLeaf, leaf_size));
	w = max(2, min(8, width));
}

// Scene of binary node x (leaf j holds sorted key j; an internal node, its first key's).
__device__ __forceinline__ uint32_t scene_of(const BinTree &t, const CostCtx &c, uint32_t x) {
	return c.scenes == 1u ? 0u : static_cast<uint32_t>(c.keys[t.first(x)] >> kSceneShift);
}

// Half-area of [lo, hi] relative to the scene's.
__device__ __forceinline__ float rel_area(float4 lo, float4 hi, double scale) {
	const double dx = static_cast<double>(hi.x) - lo.x, dy = static_cast<double>(hi.y) - lo.y,
	             dz = static_cast<double>(hi.z) - lo.z;
	return static_cast<float>((dx * dy + dx * dz + dy * dz) * scale);
}

__device__ __forceinline__ void leaf_row(float area, float r[kCostRow]) {
#pragma unroll
	for (int k = 0; k < kCostRow - 1; ++k) r[k] = area * kCostTri;
	r[kCostRow - 1] = 0.0f;
}

// split(x, i) from the rows of x's children, and the k that attains it (the smallest on ties).
__device__ __forceinline__ float best_split(const float *cl, const float *cr, int i, int &kbest) {
	float best = cl[0] + cr[i - 2];
	kbest = 1;
#pragma unroll
	for (int k = 2; k < i; ++k) {
		const float v = cl[k - 1] + cr[i - k - 1];
		if (v < best) {
			best = v;
			kbest = k;
		}
	}
	return best;
}

// The collapse's decisions at a node, made with its row: for i = 2..8 slots the k that attains
// split(x, i) (3 bits at 3 (i - 2)), for i = 2..7 whether C(x, i) = C(x, i - 1) (bit 19 + i), and
// whether the node is best kept as one leaf (bit 27). The collapse then reads one word per binary
// node instead of its children's rows.
__device__ __forceinline__ int plan_split(uint32_t plan, int i) { return static_cast<int>((plan >> (3 * (i - 2))) & 7u); }
__device__ __forceinline__ bool plan_leaf(uint32_t plan) { return (plan >> 27) & 1u; }
// The fewest slots that cost as little as `slots` of them.
__device__ __forceinline__ int plan_slots(uint32_t plan, int slots) {
	while (slots > 1 && ((plan >> (19 + slots)) & 1u)) --slots;
	return slots;
}

// Row (and plan) of an internal node from its area, triangle count, shape and its children's rows.
__device__ __forceinline__ uint32_t node_row(float area, uint32_t count, int ls, int w, const float cl[kCostRow],
                                             const float cr[kCostRow], float c[kCostRow]) {
	float split[9];
	uint32_t plan = 0;
#pragma unroll
	for (int i = 2; i <= 8; ++i) {
		int kb;
		split[i] = best_split(cl, cr, i, kb);
		plan |= static_cast<uint32_t>(kb) << (3 * (i - 2));
	}
	const bool can_leaf = count <= static_cast<uint32_t>(ls);
	const float as_leaf = can_leaf ? area * kCostTri * static_cast<float>(count) : __builtin_inff();
	float whole = split[8];
#pragma unroll
	for (int i = 2; i < 8; ++i) whole = i == w ? split[i] : whole;
	const float as_node = area * kCostNode + whole;
	const bool leaf_best = can_leaf && as_leaf <= as_node;
	c[0] = leaf_best ? as_leaf : as_node;
#pragma unroll
	for (int i = 2; i < kCostRow; ++i) {
		c[i - 1] = fminf(c[i - 2], split[i]);
		plan |= (c[i - 1] == c[i - 2] ? 1u : 0u) << (19 + i);
	}
	c[kCostRow - 1] = 0.0f;
	return plan | (leaf_best ? 1u << 27 : 0u);
}

// Rows written by one thread and read by a thread of another workgroup in the same launch go
// through device-scope atomic 8-byte stores and loads, as the boxes do.
__device__ __forceinline__ void st_row(float *rows, uint32_t x, const float c[kCostRow]) {
	uint64_t *p = reinterpret_cast<uint64_t *>(rows + static_cast<uint64_t>(kCostRow) * x);
#pragma unroll
	for (int k = 0; k < kCostRow / 2; ++k)
		__hip_atomic_store(p + k, pack2(c[2 * k], c[2 * k + 1]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void ld_row(const float *rows, uint32_t x, float c[kCostRow]) {
	const uint64_t *p = reinterpret_cast<const uint64_t *>(rows + static_cast<uint64_t>(kCostRow) * x);
#pragma unroll
	for (int k = 0; k < kCostRow / 2; ++k) {
		const uint64_t v = __hip_atomic_load(p + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		c[2 * k] = __uint_as_float(static_cast<uint32_t>(v));
		c[2 * k + 1] = __uint_as_float(static_cast<uint32_t>(v >> 32));
	}
}

// Row of binary node x written in an earlier launch (plain loads), or computed for a leaf.
__device__ __forceinline__ void row_of(const BinTree &t, const CostCtx &c, uint32_t x, float r[kCostRow]) {
	if (x >= t.n - 1) {
		leaf_row(rel_area(t.box[2ull * x], t.box[2ull * x + 1], c.scale[scene_of(t, c, x)]), r);
		return;
	}
	const float4 *p = reinterpret_cast<const float4 *>(c.row + static_cast<uint64_t>(kCostRow) * x);
	const float4 a = p[0], b = p[1];
	r[0] = a.x; r[1] = a.y; r[2] = a.z; r[3] = a.w;
	r[4] = b.x; r[5] = b.y; r[6] = b.z; r[7] = b.w;
}

// The same with x's box at hand (one scene).
__device__ __forceinline__ void ploc_row(const BinTree &t, const CostCtx &c, uint32_t x, float4 lo, float4 hi,
                                         float r[kCostRow]) {
	if (x >= t.n - 1) leaf_row(rel_area(lo, hi, c.scale[0]), r);
	else row_of(t, c, x, r);
}

// Boxes (and collapse-cost rows) from the leaves to the roots: each leaf's thread climbs, and at
// every internal node the second of its two children to arrive continues. A node whose leaf range
// lies inside the workgroup's own leaves (most of them: a radix-tree node's range starts or ends
// at its own index) is met by two threads of this workgroup, so its arrival counter and its
// children's boxes and rows live in LDS; only nodes spanning two workgroups use the global
// counters, which every XCD reaches through device-coherent atomics. Every node's box and row is
// also written to global memory for the collapse. Compiled once per cost mode: without the rows
// a workgroup holds 17 KB of LDS instead of 25 KB, so eight fit on a CU instead of six.
template <bool COST>
__global__ __launch_bounds__(kBlock) void k_bottomup(const float4 *__restrict__ tbox,
                                                     const uint32_t *__restrict__ sorted, BinTree t, CostCtx cc) {
	// slots 0..kBlock-1: internal nodes b0 + s; kBlock..2 kBlock-1: leaves of sorted positions b0 + s
	__shared__ uint32_t lflag[kBlock];
	__shared__ float4 lbox[2 * kBlock][2];
	__shared__ float lrow[COST ? kBlock : 1][kCostRow];
	const uint32_t b0 = blockIdx.x * kBlock;
	const uint32_t b1 = min(b0 + kBlock, t.n) - 1;  // last leaf position of this workgroup
	lflag[threadIdx.x] = 0u;
	__syncthreads();
	const uint32_t j = b0 + threadIdx.x;
	if (j >= t.n) return;
	uint32_t node = t.n - 1 + j;
	const uint32_t tri = sorted[j];
	float4 lo = tbox[2ull * tri], hi = tbox[2ull * tri + 1];
	lo.w = 0.0f;  // hi.w: the never-cull flag, ORed up the tree with the boxes
	st_box(t.box, node, lo, hi);
	lbox[kBlock + threadIdx.x][0] = lo;
	lbox[kBlock + threadIdx.x][1] = hi;
	float c[kCostRow];  // this node's collapse row (when costs are on)
	if (COST) leaf_row(rel_area(lo, hi, cc.scale[scene_of(t, cc, node)]), c);
	uint32_t p = (t.n > 1) ? t.parent[node] : kNone;
	// the parent's links (range, children, its own parent); no thread of this kernel writes them,
	// so the next level's are fetched before this level's arrival counter and the climb waits
	// on the counters and the sibling boxes only
	uint4 pk = make_uint4(0, 0, 0, 0);
	uint32_t pp = kNone;
	if (p != kNone) {
		pk = t.link[p];
		pp = t.parent[p];
	}
	// a radix tree over at most 2^29 keys of at most 46 bits is at most 46 + 29 levels deep
	for (int guard = 0; p != kNone && guard < 128; ++guard) {
		const bool local = pk.z >= b0 && pk.z + pk.w - 1u <= b1;
		const bool left = pk.x == node;
		const uint32_t sib = left ? pk.y : pk.x;
		// this thread's box (and row) stores complete before the device-scope count (the wait
		// is for every load too, so it comes before the next level's links are fetched)
		if (!local) stores_done();
		uint4 qk = make_uint4(0, 0, 0, 0);
		uint32_t qp = kNone;
		if (pp != kNone) {
			qk = t.link[pp];
			qp = t.parent[pp];
		}
		float4 sl, sh;
		if (local) {
			// this thread's box (and row) are in LDS already; the release orders them before the
			// count, the acquire the sibling's before the reads below
			if (__hip_atomic_fetch_add(&lflag[p - b0], 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP) == 0u) return;
			const uint32_t ss = sib >= t.n - 1 ? kBlock + (sib - (t.n - 1) - b0) : sib - b0;
			sl = lbox[ss][0];
			sh = lbox[ss][1];
		} else {
			if (atomicAdd(&t.flag[p], 1u) == 0u) return;  // sibling not finished: it continues
			ld_box(t.box, sib, sl, sh);
		}
		lo.x = fminf(lo.x, sl.x);
		lo.y = fminf(lo.y, sl.y);
		lo.z = fminf(lo.z, sl.z);
		hi.x = fmaxf(hi.x, sh.x);
		hi.y = fmaxf(hi.y, sh.y);
		hi.z = fmaxf(hi.z, sh.z);
		hi.w = __uint_as_float(__float_as_uint(hi.w) | __float_as_uint(sh.w));
		st_box(t.box, p, lo, hi);
		if (COST) {
			float cs[kCostRow], cp[kCostRow];
			if (sib >= t.n - 1) leaf_row(rel_area(sl, sh, cc.scale[scene_of(t, cc, sib)]), cs);
			else if (local) {
#pragma unroll
				for (int k = 0; k < kCostRow; ++k) cs[k] = lrow[sib - b0][k];
			} else {
				ld_row(cc.row, sib, cs);
			}
			const uint32_t scene = scene_of(t, cc, p);
			int ls, w;
			scene_shape(cc, scene, ls, w);
			t.plan[p] = node_row(rel_area(lo, hi, cc.scale[scene]), pk.w, ls, w, left ? c : cs, left ? cs : c, cp);
#pragma unroll
			for (int k = 0; k < kCostRow; ++k) c[k] = cp[k];
			st_row(cc.row, p, c);
			if (local) {
#pragma unroll
				for (int k = 0; k < kCostRow; ++k) lrow[p - b0][k] = c[k];
			}
		}
		if (local) {
			lbox[p - b0][0] = lo;
			lbox[p - b0][1] = hi;
		}
		node = p;
		p = pp;
		pk = qk;
		pp = qp;
	}
}

// No level collapsed yet: level 0 holds the scenes' roots (threads 0..2 (kMaxLevels + 2) - 1 take part).
__device__ __forceinline__ void init_levels(uint32_t *misc, uint32_t tid, uint32_t scenes) {
	if (tid < 2u * (kMaxLevels + 2)) misc[M_LCNT + tid] = tid == 0u ? scenes : 0u;
	if (tid == 0u) {
		misc[M_LBASE] = 0u;
		misc[M_ERR] &= 1u;
	}
}

// ------------------------------------------------- clustered tree (PLOC), the other builder
//
// Bottom-up agglomerative clustering over the key order (Meister and Bittner 2018, "Parallel
// Locally-Ordered Clustering"): every cluster finds its nearest neighbour among the clusters
// within kPlocR positions by the surface area of their union; mutual nearest neighbours merge into
// a new internal node; an ordered compaction removes the merged partners; repeat until one cluster
// is left. One scene. Boxes, counts and cost rows are computed at the merge, so no bottom-up pass
// is needed. Leaf of sorted triangle j = node n-1+j; a merge's node is the dropped partner's first
// sorted triangle minus 1: every triangle but the 0th is the first one of a dropped cluster exactly
// once, so the numbers are 0..n-2 and need no counter.
//
// A step took six launches (search, merge, two scan levels, compaction, count) with a host
// synchronisation every eight steps; 41 of the 64 steps of a 262,144-triangle scene work on fewer
// than 4,096 clusters, where only launches and their gaps count (2.06 of 2.9 ms). Now a step is
// one launch: a tile finds the clusters of its positions from the counts the previous step's tiles
// left, and the last kTailMax clusters are finished by one workgroup in LDS.

constexpr int kPlocR = 16;
// Steps before a build is given up. A step merges at least one pair, and only one where all areas tie
// (thousands of equal triangles), which makes a chain deeper than the BVH8 levels allow anyway.
constexpr int kPlocMaxSteps = 4096;
constexpr int kStepBlock = 512;
constexpr int kStepTile = kStepBlock - 2 * kPlocR;  // positions a tile merges: 480 of 512 searched
constexpr int kStepLoad = kStepTile + 4 * kPlocR;   // positions whose boxes it needs: 544
// With few clusters, four threads share a position's search (96 of 128 positions merge): four times
// the workgroups, a quarter of the search's latency (11.5 -> 7 us per step at 2,000 to 40,000
// clusters). The line is where the small tiles fill the chip: 420 of them.
constexpr int kShare = 4;
constexpr int kSmallTile = kStepBlock / kShare - 2 * kPlocR;
constexpr uint32_t kSmallMax = 40000;
constexpr int kMaxTiles = 4096;                     // tile counts a step sums itself (LDS)
constexpr uint32_t kTailMax = 1024;                 // clusters the tail holds in LDS, one a thread

// Half-area of the union of two boxes; overflow (huge coordinates) and inf * 0 as +inf, so that
// the order (area, position) is total and symmetric and some pair is always mutual.
__device__ __forceinline__ float union_area(const float4 alo, const float2 ahi, const float4 blo, const float2 bhi) {
	const float dx = fmaxf(alo.w, blo.w) - fminf(alo.x, blo.x);
	const float dy = fmaxf(ahi.x, bhi.x) - fminf(alo.y, blo.y);
	const float dz = fmaxf(ahi.y, bhi.y) - fminf(alo.z, blo.z);
	const float ar = dx * dy + dx * dz + dy * dz;
	return ar < __builtin_inff() ? ar : __builtin_inff();
}

struct PlocArgs {
	BinTree t;
	CostCtx cc;               // cc.row null: greedy collapse, no rows
	const float4 *tbox;       // triangle boxes and the sorted triangle order (first step)
	const uint32_t *sorted;
	const uint32_t *list_in;  // tiles of clusters, misc[M_PSTRIDE + parity] apart
	const uint32_t *cnt_in;   // clusters in each of them
	const uint32_t *scan_in;  // more than kMaxTiles tiles: their exclusive scan within segments of
	const uint32_t *pre;      // kScanSeg tiles, and the segments' offsets; else null
	uint32_t *list_out;
	uint32_t *cnt_out;
	uint32_t *scan_out;       // a copy of cnt_out (0 past the last tile) to be scanned, or null
	uint32_t *misc;
	uint32_t step;            // from 0
	int parity;               // of the step: reads buffer `parity`, writes the other
	uint32_t tiles_max;       // tiles of the first step: the scan has one more entry
};

// Node id of the merge of l and r (r the later position), written with its box, row and plan.
__device__ __forceinline__ uint32_t write_merge(const PlocArgs &a, uint32_t l, uint32_t r, uint4 ll, uint4 rl, float4 lo,
                                                float4 hi, const float cl[kCostRow], const float cr[kCostRow],
                                                float cp[kCostRow]) {
	const uint32_t id = rl.z - 1u, count = ll.w + rl.w;
	a.t.box[2ull * id] = lo;
	a.t.box[2ull * id + 1] = hi;
	a.t.link[id] = make_uint4(l, r, ll.z, count);
	if (a.cc.row) {
		int ls, w;
		scene_shape(a.cc, 0u, ls, w);
		a.t.plan[id] = node_row(rel_area(lo, hi, a.cc.scale[0]), count, ls, w, cl, cr, cp);
	}
	return id;
}

// min over the lanes that share a search (PER = 1..16 neighbouring lanes) of (area, position).
template <int CTRL>
__device__ __forceinline__ void nn_min_dpp(float &best, int32_t &bj) {
	const float ob = __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(best), CTRL, 0xF, 0xF, false));
	const int32_t oj = __builtin_amdgcn_update_dpp(0, bj, CTRL, 0xF, 0xF, false);
	if (ob < best || (ob == best && oj < bj)) {
		best = ob;
		bj = oj;
	}
}
__device__ __forceinline__ void nn_min(float &best, int32_t &bj, uint32_t per) {
	if (per > 1u) nn_min_dpp<0xB1>(best, bj);   // quad_perm 1 0 3 2
	if (per > 2u) nn_min_dpp<0x4E>(best, bj);   // quad_perm 2 3 0 1
	if (per > 4u) nn_min_dpp<0x141>(best, bj);  // row_half_mirror: the other quad of 8
	if (per > 8u) nn_min_dpp<0x140>(best, bj);  // row_mirror: the other half of 16
}

// One step. FIRST: the clusters are the triangles in sorted order, whose boxes are also written
// to their leaves here.
template <bool FIRST>
__global__ __launch_bounds__(kStepBlock) __attribute__((amdgpu_waves_per_eu(6))) void k_ploc_step(PlocArgs a) {
	__shared__ float4 slo[kStepLoad];  // lo xyz, hi x
	__shared__ float2 shi[kStepLoad];  // hi yz
	__shared__ uint32_t sid[kStepLoad], sflag[kStepLoad];
	__shared__ int32_t snn[kStepBlock];  // LDS index of the nearest neighbour, or -1
	__shared__ uint32_t pre[FIRST ? 1 : kMaxTiles];
	__shared__ uint32_t wsum[kStepBlock / 64];
	const uint32_t n = a.t.n;
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	uint32_t m = n, tiles = 0, stride = 0;
	if (!FIRST) {
		tiles = a.misc[M_PTILES + a.parity];
		stride = a.misc[M_PSTRIDE + a.parity];
		if (held_before(a.misc[M_PHELD], a.step)) return;  // the tail's turn already
		if (a.pre) {
			m = a.scan_in[a.tiles_max] + a.pre[a.tiles_max / kScanSeg];
		} else {
			// exclusive scan of the tile counts, 8 a round of kStepBlock * 8
			constexpr int per = kMaxTiles / kStepBlock;
			uint32_t v[per], sum = 0;
#pragma unroll
			for (int k = 0; k < per; ++k) {
				const uint32_t i = tid * per + k;
				v[k] = i < tiles ? a.cnt_in[i] : 0u;
				sum += v[k];
			}
			uint32_t inc = sum;
			for (int sh = 1; sh < 64; sh <<= 1) {
				const uint32_t o = __shfl_up(inc, sh);
				if (lane >= sh) inc += o;
			}
			if (lane == 63) wsum[wave] = inc;
			__syncthreads();
			uint32_t before = 0;
			m = 0;
#pragma unroll
			for (int w = 0; w < kStepBlock / 64; ++w) {
				before += w < wave ? wsum[w] : 0u;
				m += wsum[w];
			}
			uint32_t run = before + inc - sum;
#pragma unroll
			for (int k = 0; k < per; ++k) {
				pre[tid * per + k] = run;
				run += v[k];
			}
			__syncthreads();
		}
		if (m <= kTailMax) {
			if (blockIdx.x == 0 && tid == 0) a.misc[M_PHELD] = held_by(a.step);
			return;
		}
	}
	const int per = m <= kSmallMax ? kShare : 1;  // threads a position
	const int searched = kStepBlock / per, tile = searched - 2 * kPlocR, load = tile + 4 * kPlocR;
	if (blockIdx.x == 0 && tid == 0) {
		a.misc[M_PTILES + (a.parity ^ 1)] = (m + tile - 1) / tile;
		a.misc[M_PSTRIDE + (a.parity ^ 1)] = tile;
	}
	// past the last tile the copy that is scanned is 0
	if (a.scan_out)
		for (uint32_t b = (m + tile - 1) / tile + blockIdx.x * kStepBlock + tid; b <= a.tiles_max; b += gridDim.x * kStepBlock)
			a.scan_out[b] = 0u;
	for (uint32_t b = blockIdx.x; static_cast<uint64_t>(b) * tile < m; b += gridDim.x) {
		const uint32_t base = b * tile;
		for (int k = tid; k < load; k += kStepBlock) {
			const int64_t g = static_cast<int64_t>(base) + k - 2 * kPlocR;
			if (g < 0 || g >= static_cast<int64_t>(m)) continue;
			uint32_t node;
			float4 lo, hi;
			if (FIRST) {
				node = n - 1 + static_cast<uint32_t>(g);
				const uint32_t tri = a.sorted[g];
				lo = a.tbox[2ull * tri];
				hi = a.tbox[2ull * tri + 1];
				if (k >= 2 * kPlocR && k < 2 * kPlocR + tile) {
					a.t.box[2ull * node] = lo;
					a.t.box[2ull * node + 1] = hi;
				}
			} else {
				// the tile that holds position g: the last one whose first position is not past it
				uint32_t x = 0, y = tiles;
				auto start = [&](uint32_t i) { return a.pre ? a.scan_in[i] + a.pre[i / kScanSeg] : pre[i]; };
				while (y - x > 1) {
					const uint32_t mid = (x + y) >> 1;
					if (start(mid) <= static_cast<uint32_t>(g)) x = mid;
					else y = mid;
				}
				node = a.list_in[static_cast<uint64_t>(x) * stride + (static_cast<uint32_t>(g) - start(x))];
				lo = a.t.box[2ull * node];
				hi = a.t.box[2ull * node + 1];
			}
			slo[k] = make_float4(lo.x, lo.y, lo.z, hi.x);
			shi[k] = make_float2(hi.y, hi.z);
			sid[k] = node;
			sflag[k] = __float_as_uint(hi.w);  // never-cull flag
		}
		__syncthreads();
		// nearest neighbour of position base - kPlocR + p (LDS index p + kPlocR)
		{
			const int p = tid / per, sub = tid & (per - 1), me = p + kPlocR;
			const int64_t gi = static_cast<int64_t>(base) + p - kPlocR;
			float best = __builtin_inff();
			int32_t bj = 0x7FFFFFFF;
			if (gi >= 0 && gi < static_cast<int64_t>(m)) {
				const float4 blo = slo[me];
				const float2 bhi = shi[me];
				const int d0 = static_cast<int>(max(static_cast<int64_t>(-kPlocR), -gi));
				const int d1 = static_cast<int>(min(static_cast<int64_t>(kPlocR), static_cast<int64_t>(m) - 1 - gi));
				// ascending positions, so the first of equal areas stays
#pragma unroll 4
				for (int d = d0 + sub; d <= d1; d += per) {
					if (d == 0) continue;
					const float ar = union_area(blo, bhi, slo[me + d], shi[me + d]);
					if (ar < best || bj == 0x7FFFFFFF) {
						best = ar;
						bj = me + d;
					}
				}
			}
			nn_min(best, bj, static_cast<uint32_t>(per));
			if (sub == 0) snn[p] = bj == 0x7FFFFFFF ? -1 : bj;
		}
		__syncthreads();
		const int me = tid + kPlocR;
		const bool mine = tid >= kPlocR && tid < kPlocR + tile && base + tid - kPlocR < m;
		const int32_t bj = mine ? snn[tid] : -1;
		bool keep = mine;
		uint32_t node = mine ? sid[me] : 0u;
		// the partner is mutual iff its own neighbour is this position (it is within the searched ones)
		if (bj >= 0 && snn[bj - kPlocR] == me) {
			if (bj > me) {
				const uint32_t r = sid[bj];
				const uint4 ll = node >= n - 1 ? make_uint4(0, 0, node - (n - 1), 1u) : a.t.link[node];
				const uint4 rl = r >= n - 1 ? make_uint4(0, 0, r - (n - 1), 1u) : a.t.link[r];
				const float4 al = slo[me], bl = slo[bj];
				const float2 ah = shi[me], bh = shi[bj];
				const float4 llo = make_float4(al.x, al.y, al.z, 0.0f), lhi = make_float4(al.w, ah.x, ah.y, 0.0f);
				const float4 rlo = make_float4(bl.x, bl.y, bl.z, 0.0f), rhi = make_float4(bl.w, bh.x, bh.y, 0.0f);
				const float4 lo = make_float4(fminf(al.x, bl.x), fminf(al.y, bl.y), fminf(al.z, bl.z), 0.0f);
				const float4 hi = make_float4(fmaxf(al.w, bl.w), fmaxf(ah.x, bh.x), fmaxf(ah.y, bh.y),
				                              __uint_as_float(sflag[me] | sflag[bj]));
				float cl[kCostRow], cr[kCostRow], cp[kCostRow];
				if (a.cc.row) {
					ploc_row(a.t, a.cc, node, llo, lhi, cl);
					ploc_row(a.t, a.cc, r, rlo, rhi, cr);
				}
				node = write_merge(a, node, r, ll, rl, lo, hi, cl, cr, cp);
				if (a.cc.row) {
					float4 *dst = reinterpret_cast<float4 *>(a.cc.row + static_cast<uint64_t>(kCostRow) * node);
					dst[0] = make_float4(cp[0], cp[1], cp[2], cp[3]);
					dst[1] = make_float4(cp[4], cp[5], cp[6], cp[7]);
				}
			} else {
				keep = false;
			}
		}
		// ordered compaction within the tile
		const uint64_t kept = __ballot(keep);
		if (lane == 0) wsum[wave] = static_cast<uint32_t>(__popcll(kept));
		__syncthreads();
		uint32_t pos = __popcll(kept & ((1ull << lane) - 1ull)), total = 0;
#pragma unroll
		for (int w = 0; w < kStepBlock / 64; ++w) {
			pos += w < wave ? wsum[w] : 0u;
			total += wsum[w];
		}
		if (keep) a.list_out[static_cast<uint64_t>(b) * tile + pos] = node;
		if (tid == 0) {
			a.cnt_out[b] = total;
			if (a.scan_out) a.scan_out[b] = total;
		}
		__syncthreads();  // the tile's LDS is free again
	}
}

// The last clusters, in one workgroup: boxes, rows, links and neighbours live in LDS, one cluster a
// thread, and a step is three barriers. Threads share a cluster's search where there are fewer
// clusters than threads (2 to 16 of them below 512 clusters). FIRST: no step ran (n <= kTailMax),
// the clusters are the triangles. Ends with the root as BVH8 level 0.
//
// What bounds it is the chain of one step: search, mutual test, cost row, compaction. The
// barriers wait for LDS only: __syncthreads would also wait for the merged nodes' global stores.
constexpr int kTailBlock = 1024;
static_assert(kTailMax == kTailBlock, "one cluster a thread");

struct TailLds {
	float4 lo[kTailMax];  // lo xyz, hi x
	float2 hi[kTailMax];  // hi yz
	float4 row[2][kTailMax];
	uint32_t id[kTailMax], first[kTailMax], count[kTailMax];  // count: bit 31 the never-cull flag
	int32_t nn[kTailMax];
	uint32_t wsum[kTailBlock / 64];
};

__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <bool FIRST>
__global__ __launch_bounds__(kTailBlock) void k_ploc_tail(PlocArgs a, uint32_t *bin_of) {
	__shared__ TailLds s;
	const uint32_t n = a.t.n;
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	const uint32_t i = tid;
	uint32_t m = n;
	const uint32_t held = FIRST ? 0u : a.misc[M_PHELD];
	if (!FIRST && held == 0u) {  // too many clusters left: the host runs more steps
		if (tid == 0) bin_of[0] = kNone;
		init_levels(a.misc, tid, 1u);
		return;
	}
	if (FIRST) {
		if (i < m) s.id[i] = n - 1 + i;
	} else {
		const uint32_t buf = held_buffer(held);
		const uint32_t *list = buf == 0u ? a.list_in : a.list_out;
		const uint32_t *cnt = buf == 0u ? a.cnt_in : a.cnt_out;
		const uint32_t tiles = a.misc[M_PTILES + buf], stride = a.misc[M_PSTRIDE + buf];
		// gather the tiles' clusters in order, a wave per tile in turn
		m = 0;
		for (uint32_t t = 0; t < tiles; t += kTailBlock / 64) {
			uint32_t at = m, c[kTailBlock / 64];
#pragma unroll
			for (uint32_t w = 0; w < kTailBlock / 64; ++w) c[w] = t + w < tiles ? cnt[t + w] : 0u;
#pragma unroll
			for (uint32_t w = 0; w < kTailBlock / 64; ++w) {
				if (static_cast<int>(w) == wave)
					for (uint32_t k = lane; k < c[w] && at + k < kTailMax; k += 64)
						s.id[at + k] = list[static_cast<uint64_t>(t + w) * stride + k];
				at += c[w];
			}
			m = at;
		}
		m = min(m, kTailMax);
	}
	__syncthreads();
	if (i < m) {
		const uint32_t x = s.id[i];
		float4 lo, hi;
		if (FIRST) {
			const uint32_t tri = a.sorted[i];
			lo = a.tbox[2ull * tri];
			hi = a.tbox[2ull * tri + 1];
			a.t.box[2ull * x] = lo;
			a.t.box[2ull * x + 1] = hi;
		} else {
			lo = a.t.box[2ull * x];
			hi = a.t.box[2ull * x + 1];
		}
		const uint4 link = x >= n - 1 ? make_uint4(0, 0, x - (n - 1), 1u) : a.t.link[x];
		s.lo[i] = make_float4(lo.x, lo.y, lo.z, hi.x);
		s.hi[i] = make_float2(hi.y, hi.z);
		s.first[i] = link.z;
		s.count[i] = link.w | (__float_as_uint(hi.w) != 0u ? 0x80000000u : 0u);
		if (a.cc.row) {
			float r[kCostRow];
			ploc_row(a.t, a.cc, x, lo, hi, r);
			s.row[0][i] = make_float4(r[0], r[1], r[2], r[3]);
			s.row[1][i] = make_float4(r[4], r[5], r[6], r[7]);
		}
	}
	lds_barrier();
	while (m > 1) {
		// neighbours: `per` threads (a power of two up to 16) share a cluster
		uint32_t per = 1;
		while (per < 16u && m * per * 2u <= static_cast<uint32_t>(kTailBlock)) per *= 2u;
		{
			const uint32_t c = tid / per, sub = tid & (per - 1u);
			float best = __builtin_inff();
			int32_t bj = 0x7FFFFFFF;
			if (c < m) {
				const float4 alo = s.lo[c];
				const float2 ahi = s.hi[c];
				for (uint32_t k = sub; k < 2u * kPlocR; k += per) {
					const int j = static_cast<int>(c) + static_cast<int>(k) - kPlocR + (k < kPlocR ? 0 : 1);
					if (j < 0 || j >= static_cast<int>(m)) continue;
					const float ar = union_area(alo, ahi, s.lo[j], s.hi[j]);
					if (ar < best || (ar == best && j < bj)) {
						best = ar;
						bj = j;
					}
				}
			}
			nn_min(best, bj, per);
			if (c < m && sub == 0) s.nn[c] = bj;
		}
		lds_barrier();
		bool keep = i < m;
		uint32_t id = 0, fi = 0, co = 0;
		float4 lo, r0, r1;
		float2 hi;
		if (keep) {
			const int32_t j = s.nn[i];
			lo = s.lo[i];
			hi = s.hi[i];
			id = s.id[i];
			fi = s.first[i];
			co = s.count[i];
			if (a.cc.row) {
				r0 = s.row[0][i];
				r1 = s.row[1][i];
			}
			if (s.nn[j] == tid) {
				if (j < tid) {
					keep = false;
				} else {
					const float4 bl = s.lo[j];
					const float2 bh = s.hi[j];
					lo = make_float4(fminf(lo.x, bl.x), fminf(lo.y, bl.y), fminf(lo.z, bl.z), fmaxf(lo.w, bl.w));
					hi = make_float2(fmaxf(hi.x, bh.x), fmaxf(hi.y, bh.y));
					const uint32_t cj = s.count[j], flag = (co | cj) & 0x80000000u;
					float cl[kCostRow], cr[kCostRow], cp[kCostRow];
					if (a.cc.row) {
						const float4 b0 = s.row[0][j], b1 = s.row[1][j];
						cl[0] = r0.x; cl[1] = r0.y; cl[2] = r0.z; cl[3] = r0.w;
						cl[4] = r1.x; cl[5] = r1.y; cl[6] = r1.z; cl[7] = r1.w;
						cr[0] = b0.x; cr[1] = b0.y; cr[2] = b0.z; cr[3] = b0.w;
						cr[4] = b1.x; cr[5] = b1.y; cr[6] = b1.z; cr[7] = b1.w;
					}
					id = write_merge(a, id, s.id[j], make_uint4(0, 0, fi, co & 0x7FFFFFFFu),
					                 make_uint4(0, 0, s.first[j], cj & 0x7FFFFFFFu), make_float4(lo.x, lo.y, lo.z, 0.0f),
					                 make_float4(lo.w, hi.x, hi.y, __uint_as_float(flag ? 1u : 0u)), cl, cr, cp);
					co = ((co & 0x7FFFFFFFu) + (cj & 0x7FFFFFFFu)) | flag;
					if (a.cc.row) {
						r0 = make_float4(cp[0], cp[1], cp[2], cp[3]);
						r1 = make_float4(cp[4], cp[5], cp[6], cp[7]);
					}
				}
			}
		}
		const uint64_t kept = __ballot(keep);
		if (lane == 0) s.wsum[wave] = static_cast<uint32_t>(__popcll(kept));
		lds_barrier();  // also: every thread has read what it needs of the old clusters
		uint32_t k = __popcll(kept & ((1ull << lane) - 1ull)), total = 0;
#pragma unroll
		for (int w = 0; w < kTailBlock / 64; ++w) {
			const uint32_t v = s.wsum[w];
			k += w < wave ? v : 0u;
			total += v;
		}
		if (keep) {
			s.lo[k] = lo;
			s.hi[k] = hi;
			s.id[k] = id;
			s.first[k] = fi;
			s.count[k] = co;
			if (a.cc.row) {
				s.row[0][k] = r0;
				s.row[1][k] = r1;
			}
		}
		m = total;
		lds_barrier();
	}
	if (tid == 0) {
		bin_of[0] = s.id[0];
		a.misc[M_PDONE] = 1u;
	}
	init_levels(a.misc, tid, 1u);
}

// ------------------------------------------------------------------------- BVH8 collapse

__device__ __forceinline__ float half_area(float4 lo, float4 hi) {
	const float dx = hi.x - lo.x, dy = hi.y - lo.y, dz = hi.z - lo.z;
	return dx * dy + dx * dz + dy * dz;
}

// Quantizes [clo, chi] against a grid at p with step s = 2^e; both bounds round outward,
// checked with the same fmaf the traversal evaluates.
__device__ __forceinline__ void quantize(float clo, float chi, float p, float s, uint8_t &qlo, uint8_t &qhi) {
	int lo = static_cast<int>(floorf((clo - p) / s));
	lo = max(0, min(255, lo));
	while (lo > 0 && fmaf(static_cast<float>(lo), s, p) > clo) --lo;
	int hi = static_cast<int>(ceilf((chi - p) / s));
	hi = max(0, min(255, hi));
	while (hi < 255 && fmaf(static_cast<float>(hi), s, p) < chi) ++hi;
	qlo = static_cast<uint8_t>(lo);
	qhi = static_cast<uint8_t>(hi);
}

// Smallest e in [-126, 127] with p + 255 * 2^e >= top in fp32.
__device__ __forceinline__ int grid_exp(float p, float top) {
	const float ext = top - p;
	int e = -126;
	if (ext > 0.0f) {
		int ex;
		(void)frexpf(ext / 255.0f, &ex);  // ext/255 in [2^(ex-1), 2^ex)
		e = max(-126, min(127, ex - 1));
	}
	while (e < 127 && fmaf(255.0f, exp2i(e), p) < top) ++e;
	return e;
}

struct CollapseArgs {
	BinTree t;
	uint32_t *misc;
	uint32_t *bin_of;
	uint32_t *tri_dest;
	NodeQ *nq;
	NodeF *nf;
	CostCtx cc;  // keys, per-scene shape; cc.row null: greedy collapse
};

// Value of lane `src` of this lane's group of 8.
__device__ __forceinline__ uint32_t group_get(uint32_t v, int src) {
	return static_cast<uint32_t>(__shfl(static_cast<int>(v), (static_cast<int>(threadIdx.x) & 56) | src));
}
__device__ __forceinline__ float group_min(float v) {
#pragma unroll
	for (int sh = 1; sh < 8; sh <<= 1) v = fminf(v, __shfl_xor(v, sh));
	return v;
}
__device__ __forceinline__ float group_max(float v) {
#pragma unroll
	for (int sh = 1; sh < 8; sh <<= 1) v = fmaxf(v, __shfl_xor(v, sh));
	return v;
}
// This group's 8 bits of a ballot.
__device__ __forceinline__ uint32_t group_ballot(bool p) {
	return static_cast<uint32_t>(__ballot(p) >> (threadIdx.x & 56u)) & 0xFFu;
}

constexpr int kGroups = kBlock / 8;  // BVH8 nodes a workgroup collapses at a time

struct CollapseLds {
	uint4 q[kGroups][sizeof(NodeQ) / 16];
	uint4 f[kGroups][sizeof(NodeF) / 16];
};

// A BVH8 node is collapsed by the 8 lanes of a group, one lane per child slot: pick_children finds
// the children, the caller allocates node numbers and triangle slots, write_node writes both node
// formats. Every lane of a wave takes part; groups with on = false only in the shuffles.
//
// One thread per node took 35 to 57 us for any level however small: a chain of some 20 dependent
// loads (links, child boxes, cost rows), 8 children quantized one after the other, and two
// same-address atomics per 64 nodes. With a lane per slot the loads of a round go out together (3
// to 5 rounds), the cost rows are one plan word per binary node, and each lane quantizes its own
// child.
struct Child {
	uint32_t x;    // binary node, or kNone
	uint32_t cnt;  // triangles of a leaf; 0: internal (or no child)
	__device__ __forceinline__ bool leaf() const { return cnt != 0u; }
	__device__ __forceinline__ bool inner() const { return x != kNone && cnt == 0u; }
};

// The child in this lane's slot of BVH8 node i (binary node bin_of[i]), in slot order but not
// necessarily in the lowest lanes.
template <bool COST>
__device__ __forceinline__ Child pick_children(const CollapseArgs &a, uint32_t i, bool on) {
	const BinTree &t = a.t;
	const uint32_t n_int = t.n - 1;  // binary internal nodes are ids < n_int
	const int g = static_cast<int>(threadIdx.x & 7u);
	const uint32_t b = on ? a.bin_of[i] : kNone;  // kNone: root of an empty scene, written as an empty node
	const bool inner_root = b < n_int;
	int leaf_size = 1, width = 8;
	uint4 link = make_uint4(0, 0, 0, 0);
	uint32_t plan = 0;
	if (inner_root) {
		link = t.link[b];
		if (COST) plan = t.plan[b];
	}
	if (b != kNone) scene_shape(a.cc, a.cc.scenes == 1u ? 0u : scene_of(t, a.cc, b), leaf_size, width);
	uint32_t x = kNone;  // this lane's child, when it is one
	bool child = false, is_leaf = false;
	uint32_t cnt = 0;
	if (COST) {
		// A subtree that may fill `slots` slots owns the lanes [head, head + slots); the lane `head`
		// stands for it. A split at k leaves the left part at head and starts the right one at
		// head + k, until every part is a leaf or one slot wide (fewer slots where they cost as
		// little).
		int head = -1, slots = 0;
		bool open = false;
		if (inner_root) {
			const int k = plan_split(plan, width);
			head = g < k ? 0 : k;
			if (g >= width) head = -1;
			slots = g < k ? k : width - k;
			if (head == g) {
				x = g < k ? link.x : link.y;
				child = open = true;
			}
		} else if (b != kNone && g == 0) {  // a one-triangle scene
			x = b;
			child = is_leaf = true;
			cnt = 1;
		}
		while (__ballot(open) != 0ull) {
			uint32_t k = 0;
			if (open) {
				if (x >= n_int) {  // one triangle: a leaf
					open = false;
					is_leaf = true;
					cnt = 1;
				} else {
					link = t.link[x];
					plan = t.plan[x];
					slots = plan_slots(plan, slots);
					if (slots == 1) {
						open = false;
						is_leaf = plan_leaf(plan);
						cnt = link.w;
					} else {
						k = static_cast<uint32_t>(plan_split(plan, slots));
					}
				}
			}
			const int h = head < 0 ? 0 : head;
			const uint32_t hk = group_get(k, h), hr = group_get(link.y, h);
			const int hs = static_cast<int>(group_get(static_cast<uint32_t>(slots), h));
			if (head >= 0 && hk != 0u) {
				const int split = head + static_cast<int>(hk), end = head + hs;
				if (g >= end) {
					head = -1;
				} else if (g >= split) {
					head = split;
					slots = end - split;
					if (g == split) {
						x = hr;
						child = open = true;
					}
				} else {
					slots = static_cast<int>(hk);
					if (g == head) x = link.x;
				}
			}
		}
	} else {
		// open the child of largest area until there are `width` (the opened one's left part stays
		// in its lane, the right part takes the next free one); subtrees of at most leaf_size
		// triangles become leaves
		float area = -1.0f;
		auto take = [&](uint32_t node) {
			x = node;
			child = true;
			const float4 lo = t.box[2ull * x], hi = t.box[2ull * x + 1];
			link = x < n_int ? t.link[x] : make_uint4(0, 0, 0, 1u);
			cnt = link.w;
			area = x < n_int ? half_area(lo, hi) : -1.0f;
		};
		int ne = 0;
		if (inner_root) {
			if (g < 2) take(g == 0 ? link.x : link.y);
			ne = 2;
		} else if (b != kNone) {
			if (g == 0) take(b);
			ne = 1;
		}
		bool more = inner_root;
		while (__ballot(more) != 0ull) {
			const float top = group_max(area);
			const uint32_t is_top = group_ballot(area == top);
			const int best = __ffs(static_cast<int>(is_top)) - 1;  // the first of equal areas
			more = more && ne < width && top > -1.0f;
			const uint32_t l = group_get(link.x, best < 0 ? 0 : best), r = group_get(link.y, best < 0 ? 0 : best);
			if (more) {
				if (g == best || g == ne) take(g == best ? l : r);
				++ne;
			}
		}
		is_leaf = child && (cnt <= static_cast<uint32_t>(leaf_size) || x >= n_int);
	}
	return {child ? x : kNone, is_leaf ? cnt : 0u};
}

// Internal children (low 32 bits) and leaf triangles (high 32 bits) of this lane's node.
__device__ __forceinline__ uint64_t node_needs(const Child &c) {
	uint32_t tris = c.cnt;
#pragma unroll
	for (int sh = 1; sh < 8; sh <<= 1) tris += __shfl_xor(tris, sh);
	return static_cast<uint64_t>(tris) << 32 | static_cast<uint32_t>(__popc(group_ballot(c.inner())));
}

// Sum over the wave's groups before this lane's, and over all of them in `total`.
__device__ __forceinline__ uint64_t wave_before(uint64_t needs, uint64_t &total) {
	uint64_t inc = needs;
#pragma unroll
	for (int sh = 8; sh < 64; sh <<= 1) {
		const uint64_t o = __shfl_up(inc, sh);
		if ((threadIdx.x & 63u) >= static_cast<uint32_t>(sh)) inc += o;
	}
	total = __shfl(inc, 63);
	return inc - needs;
}

// Writes node i: its internal children are child_base.. (their binary nodes go to bin_of), its
// leaves' triangles tri_base...
__device__ __forceinline__ void write_node(const CollapseArgs &a, uint32_t i, bool on, const Child &c, uint32_t child_base,
                                           uint32_t tri_base, CollapseLds &lds) {
	const BinTree &t = a.t;
	const uint32_t n_int = t.n - 1;
	const int g = static_cast<int>(threadIdx.x & 7u);
	const uint32_t x = c.x, cnt = c.cnt;
	const bool child = x != kNone, inner = c.inner();
	float4 lo = make_float4(0, 0, 0, 0), hi = make_float4(0, 0, 0, 0);
	if (child) {
		lo = t.box[2ull * x];
		hi = t.box[2ull * x + 1];
	}
	const uint32_t inner_mask = group_ballot(inner), child_mask = group_ballot(child);
	const uint32_t below = (1u << g) - 1u;
	const int ne = __popc(child_mask);
	if (inner_mask == 0u) child_base = 0u;
	uint32_t toff = cnt;  // leaf triangles before this lane
#pragma unroll
	for (int sh = 1; sh < 8; sh <<= 1) {
		const uint32_t o = __shfl_up(toff, sh, 8);
		if (g >= sh) toff += o;
	}
	if (group_get(toff, 7) == 0u) tri_base = 0u;
	toff -= cnt;
	// node box = union of the children's
	float np[3], nt[3], sc[3];
	int8_t ex[3];
	const float l3[3] = {lo.x, lo.y, lo.z}, h3[3] = {hi.x, hi.y, hi.z};
#pragma unroll
	for (int ax = 0; ax < 3; ++ax) {
		np[ax] = group_min(child ? l3[ax] : __builtin_inff());
		nt[ax] = group_max(child ? h3[ax] : -__builtin_inff());
		if (ne == 0) np[ax] = nt[ax] = 0.0f;
		const int e = grid_exp(np[ax], nt[ax]);
		ex[ax] = static_cast<int8_t>(e);
		sc[ax] = exp2i(e);
	}
	const uint32_t ncull = group_ballot(child && __float_as_uint(hi.w) != 0u);
	// slot of this lane: children first, in lane order
	const int slot = child ? __popc(child_mask & below) : ne + __popc(~child_mask & below);
	uint32_t slot_ncull = 0;  // ncull by slot
#pragma unroll
	for (int k = 0; k < 8; ++k)
		if ((ncull >> k) & 1u) slot_ncull |= 1u << __popc(child_mask & ((1u << k) - 1u));
	uint8_t meta = kMetaEmpty;
	if (inner) {
		const uint32_t at = static_cast<uint32_t>(__popc(inner_mask & below));
		meta = static_cast<uint8_t>(kMetaInternal | at);
		a.bin_of[child_base + at] = x;
	} else if (child) {
		meta = meta_leaf(toff, cnt);
		// the subtree's triangles in depth-first (left to right) order: a range of sorted positions
		// for the radix tree, any set of them for the clustered tree; s0 is the stack's top
		uint32_t s0 = x, s1 = kNone, s2 = kNone, s3 = kNone;
		for (uint32_t m = 0, step = 0; s0 != kNone && m < cnt && step < 2u * kMaxLeaf; ++step) {
			if (s0 >= n_int) {
				a.tri_dest[s0 - n_int] = tri_base + toff + m;
				++m;
				s0 = s1;
				s1 = s2;
				s2 = s3;
				s3 = kNone;
			} else {
				const uint4 k = t.link[s0];
				s3 = s2;
				s2 = s1;
				s1 = k.y;
				s0 = k.x;
			}
		}
	}
	// both formats through LDS (a wave's lanes only), then stored 16 bytes a lane
	const uint32_t grp = threadIdx.x >> 3;
	NodeQ *q = reinterpret_cast<NodeQ *>(lds.q[grp]);
	NodeF *f = reinterpret_cast<NodeF *>(lds.f[grp]);
	q->meta[slot] = f->meta[slot] = meta;
#pragma unroll
	for (int ax = 0; ax < 3; ++ax) {
		uint8_t ql = 255, qh = 0;
		if (child) quantize(l3[ax], h3[ax], np[ax], sc[ax], ql, qh);
		q->qlo[ax][slot] = ql;
		q->qhi[ax][slot] = qh;
		f->lo[ax][slot] = child ? l3[ax] : __builtin_inff();
		f->hi[ax][slot] = child ? h3[ax] : -__builtin_inff();
	}
	if (g == 0) {
#pragma unroll
		for (int ax = 0; ax < 3; ++ax) {
			q->p[ax] = np[ax];
			q->e[ax] = ex[ax];
		}
		q->ncull = static_cast<uint8_t>(slot_ncull);
		q->child_base = f->child_base = child_base;
		q->tri_base = f->tri_base = tri_base;
	}
	__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
	__builtin_amdgcn_wave_barrier();
	__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
	if (on) {
		uint4 *dq = reinterpret_cast<uint4 *>(a.nq + i), *df = reinterpret_cast<uint4 *>(a.nf + i);
		constexpr int cq = sizeof(NodeQ) / 16, cf = sizeof(NodeF) / 16;
		for (int k = g; k < cq + cf; k += 8) {
			if (k < cq) dq[k] = lds.q[grp][k];
			else df[k - cq] = lds.f[grp][k - cq];
		}
	}
	__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
	__builtin_amdgcn_wave_barrier();  // the slice is free again
}

__device__ __forceinline__ unsigned long long *level_counter(const CollapseArgs &a, int level) {
	return reinterpret_cast<unsigned long long *>(a.misc + M_LCNT) + level;
}

// First node, node count and first leaf triangle of a level, final when its launch starts; the
// first workgroup writes where the next level starts.
__device__ __forceinline__ void level_range(const CollapseArgs &a, int level, uint32_t &begin, uint32_t &count, uint32_t &tris) {
	const uint64_t c = *level_counter(a, level);
	begin = a.misc[M_LBASE + level];
	count = static_cast<uint32_t>(c);
	tris = level ? a.misc[M_TBASE + level - 1] + static_cast<uint32_t>(c >> 32) : 0u;
	if (blockIdx.x == 0 && threadIdx.x == 0) {
		a.misc[M_LBASE + level + 1] = begin + count;
		a.misc[M_TBASE + level] = tris;
	}
}

// One BVH8 level. A workgroup picks the children of up to kRounds * kGroups nodes, allocates for all
// of them with one 64-bit atomic, and writes them: an atomic on one address takes about 5 ns, and
// one for every wave's 8 nodes held a level of 350,000 nodes for 525 us.
constexpr int kRounds = 8;

template <bool COST>
__global__ __launch_bounds__(kBlock) void k_collapse(CollapseArgs a, int level) {
	__shared__ CollapseLds lds;
	__shared__ Child kids[kRounds][kBlock];
	__shared__ uint64_t before[kRounds][kGroups];  // needs of the wave's earlier groups and rounds
	__shared__ uint64_t wtotal[kBlock / 64];
	__shared__ uint64_t sbase;
	uint32_t begin, count, tris;
	level_range(a, level, begin, count, tris);
	const uint32_t grp = threadIdx.x >> 3, wave = threadIdx.x >> 6;
	// rounds: enough that the grid covers the level once, at most kRounds
	const uint32_t rounds = min(static_cast<uint32_t>(kRounds), max(1u, (count + gridDim.x * kGroups - 1) / (gridDim.x * kGroups)));
	for (uint32_t i0 = blockIdx.x * kGroups * rounds; i0 < count; i0 += gridDim.x * kGroups * rounds) {
		uint64_t run = 0;
		for (uint32_t r = 0; r < rounds; ++r) {
			const uint32_t k = i0 + r * kGroups + grp;
			const Child c = pick_children<COST>(a, begin + k, k < count);
			uint64_t total;
			const uint64_t b = wave_before(node_needs(c), total);
			kids[r][threadIdx.x] = c;
			if ((threadIdx.x & 7u) == 0u) before[r][grp] = run + b;
			run += total;
		}
		if ((threadIdx.x & 63u) == 0u) wtotal[wave] = run;
		__syncthreads();
		if (threadIdx.x == 0) {
			uint64_t all = 0;
			for (int w = 0; w < kBlock / 64; ++w) all += wtotal[w];
			sbase = all ? atomicAdd(level_counter(a, level + 1), static_cast<unsigned long long>(all)) : 0ull;
		}
		__syncthreads();
		uint64_t base = sbase;
		for (uint32_t w = 0; w < wave; ++w) base += wtotal[w];
		for (uint32_t r = 0; r < rounds; ++r) {
			const uint32_t k = i0 + r * kGroups + grp;
			const uint64_t at = base + before[r][grp];
			write_node(a, begin + k, k < count, kids[r][threadIdx.x], begin + count + static_cast<uint32_t>(at),
			           tris + static_cast<uint32_t>(at >> 32), lds);
		}
		__syncthreads();
	}
}

// The rest of the tree from `level` on, depth first, one frontier node per group of lanes: a
// fixed-length build (capturable) runs a few level launches for the wide top of the tree and
// then this one launch instead of a long tail of mostly empty level launches. The stack holds
// one {first node, nodes left} range per level; a deeper tree sets error bit 2.
//
// A frontier node of m triangles has at most m - 2 BVH8 nodes below it (one per binary node strictly
// inside its subtree) and its leaves hold m triangles, so that much is reserved for it at the start, in the
// next level's counts, by one atomic per 8 of them: all reservations together fit the build's node
// capacity, and the numbers that stay unused are referenced by nothing. With an atomic for every 8 nodes
// of the walk, 64 scenes (2.5 M triangles) in nodes of 4 children took 2.7 ms here, 4.05 ms a step; the step now
// takes 2.14 (2.63 with one thread per frontier node).
constexpr int kDfsStack = kFixedDfsDepth;

template <bool COST>
__global__ __launch_bounds__(kBlock) void k_collapse_dfs(CollapseArgs a, int level) {
	__shared__ CollapseLds lds;
	__shared__ uint2 stack[kGroups][kDfsStack];
	uint32_t begin, count, tris;
	level_range(a, level, begin, count, tris);
	const uint32_t grp = threadIdx.x >> 3;
	uint2 *st = stack[grp];
	for (uint32_t i0 = blockIdx.x * kGroups; i0 < count; i0 += gridDim.x * kGroups) {
		int sp = 0;
		uint2 top = make_uint2(begin + i0 + grp, i0 + grp < count ? 1u : 0u);
		const uint32_t x = top.y != 0u ? a.bin_of[top.x] : kNone;
		const uint32_t m = x == kNone ? 0u : a.t.count(x);
		uint64_t total, at = 0;
		const uint64_t before = wave_before(static_cast<uint64_t>(m) << 32 | (m > 2u ? m - 2u : 0u), total);
		if ((threadIdx.x & 63u) == 0u && total) at = atomicAdd(level_counter(a, level + 1), static_cast<unsigned long long>(total));
		at = __shfl(at, 0) + before;
		uint32_t node_at = begin + count + static_cast<uint32_t>(at), tri_at = tris + static_cast<uint32_t>(at >> 32);
		// top: the range being walked (the group's lanes hold the same values)
		while (__ballot(top.y != 0u) != 0ull) {
			const bool on = top.y != 0u;
			const uint32_t node = top.x;
			const Child c = pick_children<COST>(a, node, on);
			const uint64_t needs = node_needs(c);
			const uint2 ch = make_uint2(node_at, static_cast<uint32_t>(needs));
			write_node(a, node, on, c, ch.x, tri_at, lds);
			if (!on) continue;
			node_at += ch.y;
			tri_at += static_cast<uint32_t>(needs >> 32);
			++top.x;
			--top.y;
			if (ch.y != 0u) {
				if (top.y != 0u) {
					if (sp == kDfsStack) {
						atomicOr(a.misc + M_ERR, 4u);
						top.y = 0u;
						continue;
					}
					if ((threadIdx.x & 7u) == 0u) st[sp] = top;
					__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
					++sp;
				}
				top = ch;
			} else if (top.y == 0u && sp > 0) {
				--sp;
				__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
				top = st[sp];
			}
		}
	}
}

// Leaf triangle records; ids are scene-local (input index minus the scene's first index).
__global__ __launch_bounds__(kBlock) void k_emit_tris(const float *__restrict__ tris, const uint32_t *__restrict__ sorted,
                                                      const uint64_t *__restrict__ keys, const uint32_t *__restrict__ off,
                                                      const uint32_t *__restrict__ dest, uint32_t n,
                                                      TriRec *__restrict__ out, uint32_t *misc) {
	const uint32_t j = blockIdx.x * kBlock + threadIdx.x;
	if (j >= n) return;
	const uint32_t src = sorted[j];
	if (dest[j] >= n || src >= n) {  // a triangle not placed by the collapse: report, never write
		atomicOr(misc + M_ERR, 2u);
		return;
	}
	TriRec r;
#pragma unroll
	for (int k = 0; k < 9; ++k) r.v[k] = tris[9ull * src + k];
	r.id = off ? src - off[keys[j] >> kSceneShift] : src;
	r.pad[0] = r.pad[1] = 0;
	out[dest[j]] = r;
}

// BVH8 level 0: node s is the root of scene s.
__global__ __launch_bounds__(kBlock) void k_roots(uint32_t *misc, uint32_t *bin_of, const uint32_t *scene_root,
                                                  uint32_t scenes) {
	const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
	if (s < scenes) bin_of[s] = scene_root[s];
	init_levels(misc, s, scenes);
}

__global__ void k_clear_err(uint32_t *misc) {
	if (threadIdx.x == 0) misc[M_ERR] &= 1u;
}

// After a fixed-length build: a triangle the collapse did not place.
__global__ void k_check_done(uint32_t *misc, uint32_t n) {  // one wave
	uint32_t sum = 0;
	for (uint32_t l = threadIdx.x; l < kMaxLevels + 2; l += 64) sum += misc[M_LCNT + 2 * l + 1];
	for (int sh = 32; sh > 0; sh >>= 1) sum += __shfl_xor(sum, sh);
	if (threadIdx.x == 0 && sum != n) atomicOr(misc + M_ERR, 2u);
}

// Per-scene vertex bounds as floats: min xyz, max xyz.
__global__ __launch_bounds__(kBlock) void k_scene_boxes(const uint32_t *misc, uint32_t scenes, float *box) {
	const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
	if (i < 6 * scenes) box[i] = o2f(misc[M_SCENE + M_PER_SCENE * (i / 6) + 6 + i % 6]);
}

inline uint32_t blocks_for(uint64_t n, int per = kBlock) { return static_cast<uint32_t>((n + per - 1) / per); }

// ------------------------------------------------------------ refit: new vertices, same tree
//
// Every leaf record takes its primitive's new vertices; then every node's child boxes are
// recomputed from the deepest level up (children have larger indices than their parent, and
// a level's nodes are one contiguous index range), and the quantized boxes re-derived with the
// build's outward rounding. Topology, child order and leaf membership do not change.

__global__ __launch_bounds__(kBlock) void k_refit_tris(const float *__restrict__ tri_in, TriRec *__restrict__ tris,
                                                       uint32_t n, uint32_t *misc) {
	const uint32_t j = blockIdx.x * kBlock + threadIdx.x;
	if (j >= n) return;
	TriRec r = tris[j];
	if (r.id >= n) {  // not a record of this tree: report, never read
		atomicOr(misc + M_ERR, 2u);
		return;
	}
	bool finite = true;
#pragma unroll
	for (int k = 0; k < 9; ++k) {
		r.v[k] = tri_in[9ull * r.id + k];
		finite &= __builtin_isfinite(r.v[k]);
	}
	tris[j] = r;
	if (!finite) atomicOr(misc + M_ERR, 1u);
	if (cull_unsafe(r.v)) atomicAdd(misc + M_NCULL, 1u);
}

struct RefitArgs {
	const TriRec *tris;
	NodeQ *nq;
	NodeF *nf;
	float4 *box;  // [2 * n_nodes] node boxes (lo, hi), written here for the parent level
	uint32_t n_nodes;
	uint32_t n_tris;
	uint32_t *misc;
};

// Node i with the 8 lanes of a group, one child slot a lane (one thread per node held a level for
// 20 to 44 us: 8 children one after the other, each a dependent load, at two waves a SIMD). Every
// lane of the wave takes part.
__device__ __forceinline__ void refit_node(const RefitArgs &a, uint32_t i, bool on, CollapseLds &lds) {
	const int g = static_cast<int>(threadIdx.x & 7u);
	const uint32_t grp = (threadIdx.x >> 3) % kGroups;
	uint4 head = make_uint4(0u, 0u, 0xFFFFFFFFu, 0xFFFFFFFFu);  // child_base, tri_base, meta
	if (on) head = *reinterpret_cast<const uint4 *>(a.nf + i);
	const uint32_t m = ((g < 4 ? head.z : head.w) >> (8 * (g & 3))) & 0xFFu;
	float lo[3] = {__builtin_inff(), __builtin_inff(), __builtin_inff()};
	float hi[3] = {-__builtin_inff(), -__builtin_inff(), -__builtin_inff()};
	bool flagged = false;  // the slot's subtree holds a triangle that is never culled (cull_unsafe)
	if (meta_internal(m)) {
		const uint32_t c = head.x + meta_offset(m);
		if (c <= i || c >= a.n_nodes) {
			atomicOr(a.misc + M_ERR, 2u);
		} else {
			const float4 cl = a.box[2ull * c], ch = a.box[2ull * c + 1];
			lo[0] = cl.x; lo[1] = cl.y; lo[2] = cl.z;
			hi[0] = ch.x; hi[1] = ch.y; hi[2] = ch.z;
			flagged = __float_as_uint(ch.w) != 0u;
		}
	} else if (meta_used(m)) {
		const uint32_t first = head.y + meta_offset(m), cnt = meta_count(m);
		if (first + cnt > a.n_tris) {
			atomicOr(a.misc + M_ERR, 2u);
		} else {
			for (uint32_t t = first; t < first + cnt; ++t) {
				const uint4 *src = reinterpret_cast<const uint4 *>(a.tris + t);
				const uint4 r0 = src[0], r1 = src[1], r2 = src[2];
				const float v[9] = {__uint_as_float(r0.x), __uint_as_float(r0.y), __uint_as_float(r0.z),
				                    __uint_as_float(r0.w), __uint_as_float(r1.x), __uint_as_float(r1.y),
				                    __uint_as_float(r1.z), __uint_as_float(r1.w), __uint_as_float(r2.x)};
#pragma unroll
				for (int p = 0; p < 3; ++p)
#pragma unroll
					for (int ax = 0; ax < 3; ++ax) {
						lo[ax] = fminf(lo[ax], v[3 * p + ax]);
						hi[ax] = fmaxf(hi[ax], v[3 * p + ax]);
					}
				flagged |= cull_unsafe(v);
			}
		}
	}
	const uint32_t ncull = group_ballot(flagged);
	NodeQ *q = reinterpret_cast<NodeQ *>(lds.q[grp]);
	float *f = reinterpret_cast<float *>(lds.f[grp]);  // the node's boxes, lo then hi
	float nlo[3], nhi[3];
#pragma unroll
	for (int ax = 0; ax < 3; ++ax) {
		nlo[ax] = group_min(lo[ax]);
		nhi[ax] = group_max(hi[ax]);
		const int e = grid_exp(nlo[ax], nhi[ax]);
		uint8_t ql = 255, qh = 0;
		if (meta_used(m)) quantize(lo[ax], hi[ax], nlo[ax], exp2i(e), ql, qh);
		q->qlo[ax][g] = ql;
		q->qhi[ax][g] = qh;
		f[8 * ax + g] = lo[ax];
		f[24 + 8 * ax + g] = hi[ax];
		if (g == 0) {
			q->p[ax] = nlo[ax];
			q->e[ax] = static_cast<int8_t>(e);
		}
	}
	q->meta[g] = static_cast<uint8_t>(m);
	if (g == 0) {
		q->ncull = static_cast<uint8_t>(ncull);
		q->child_base = head.x;
		q->tri_base = head.y;
	}
	__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
	__builtin_amdgcn_wave_barrier();
	__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
	if (on) {
		if (g == 0) a.box[2ull * i] = make_float4(nlo[0], nlo[1], nlo[2], 0.0f);
		if (g == 1) a.box[2ull * i + 1] = make_float4(nhi[0], nhi[1], nhi[2], __uint_as_float(ncull != 0u ? 1u : 0u));
		uint4 *dq = reinterpret_cast<uint4 *>(a.nq + i), *df = reinterpret_cast<uint4 *>(a.nf + i) + 1;
		constexpr int cq = sizeof(NodeQ) / 16, cf = sizeof(NodeF) / 16 - 1;
		for (int k = g; k < cq + cf; k += 8) {
			if (k < cq) dq[k] = lds.q[grp][k];
			else df[k - cq] = lds.f[grp][k - cq];
		}
	}
	__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
	__builtin_amdgcn_wave_barrier();
}

__global__ __launch_bounds__(kBlock) void k_refit_level(RefitArgs a, uint32_t begin, uint32_t end) {
	__shared__ CollapseLds lds;
	for (uint32_t i0 = begin + blockIdx.x * kGroups; i0 < end; i0 += gridDim.x * kGroups) {
		const uint32_t i = i0 + (threadIdx.x >> 3);
		refit_node(a, i, i < end, lds);
	}
}

// Consecutive levels of at most kFewNodes nodes each, deepest first, by one workgroup: a launch for
// each would take longer than its nodes.
constexpr uint32_t kFewNodes = 256;
constexpr int kFewLevels = 32;
struct FewLevels {
	int count;
	uint32_t bound[kFewLevels + 1];  // level k of the run is [bound[k + 1], bound[k])
};

constexpr int kFewBlock = 1024;

__global__ __launch_bounds__(kFewBlock) void k_refit_few(RefitArgs a, FewLevels f) {
	__shared__ CollapseLds lds[kFewBlock / kBlock];
	for (int k = 0; k < f.count; ++k) {
		for (uint32_t i0 = f.bound[k + 1]; i0 < f.bound[k]; i0 += kFewBlock / 8) {
			const uint32_t i = i0 + (threadIdx.x >> 3);
			refit_node(a, i, i < f.bound[k], lds[threadIdx.x / kBlock]);
		}
		__syncthreads();  // the level's boxes are read by the next one
	}
	// the root's box goes back with the flags
	if (f.bound[f.count] == 0u && threadIdx.x < 6u)
		a.misc[M_SCENE + 6 + threadIdx.x] = f2o(reinterpret_cast<const float *>(a.box)[threadIdx.x + (threadIdx.x < 3u ? 0u : 1u)]);
}

}  // namespace

// Host form of o2f.
static float ordered_float(uint32_t u) {
	union {
		uint32_t u;
		float f;
	} c;
	c.u = (u & 0x80000000u) ? (u & 0x7FFFFFFFu) : ~u;
	return c.f;
}

// The scratch's pair of timing events, created at the first use.
static hipError_t time_events(BuildScratch &s, hipEvent_t ev[2]) {
	for (int k = 0; k < 2; ++k) {
		if (!s.ev[k]) {
			const hipError_t e = hipEventCreate(&s.ev[k]);
			if (e != hipSuccess) return e;
		}
		ev[k] = s.ev[k];
	}
	return hipSuccess;
}

hipError_t build_bvh8(BuildScratch &s, uint64_t n64, const BuildParams &p, Bvh8 &out, hipStream_t st,
                      bool *bad_input, double *build_ms, const SceneSet *scenes) {
#define PRT_TRY(x)                                                                                 \
	do {                                                                                           \
		hipError_t e_ = (x);                                                                       \
		if (e_ != hipSuccess) return e_;                                                           \
	} while (0)
	SceneSet one;
	const SceneSet &ss = scenes ? *scenes : one;
	const uint32_t S = ss.count;
	const bool fixed = ss.levels > 0;  // no host synchronisation: capturable in a graph
	*bad_input = false;
	out.levels.clear();
	out.n_tris = n64;
	out.n_nodes = 0;
	out.n_ncull = 0;
	out.depth = 0;
	out.leaf_size = static_cast<uint32_t>(p.leaf_size);
	if (S == 0 || S > kMaxScenes || (S > 1 && !ss.tri_off) || (fixed && build_ms)) return hipErrorInvalidValue;
	if (n64 == 0) return hipSuccess;
	if (n64 > static_cast<uint64_t>(kTriMask)) return hipErrorInvalidValue;
	const uint32_t n = static_cast<uint32_t>(n64);
	const uint32_t nb = 2 * n - 1;
	const uint32_t cap = n + S;  // BVH8 nodes: at most one per binary internal node, one per scene root
	const uint32_t words = misc_words(S);
	const uint32_t *off = S > 1 ? ss.tri_off : nullptr;

	PRT_TRY(s.tbox.ensure(sizeof(float4) * 2 * n));
	for (int k = 0; k < 2; ++k) {
		PRT_TRY(s.keys[k].ensure(sizeof(uint64_t) * n));
		PRT_TRY(s.vals[k].ensure(sizeof(uint32_t) * n));
	}
	const int items = sort_items(n);
	const uint32_t tiles = blocks_for(n, kBlock * items);
	const uint32_t hist_n = 256 * tiles, n_seg = blocks_for(hist_n, kScanSeg);
	PRT_TRY(s.hist.ensure(sizeof(uint32_t) * (static_cast<uint64_t>(hist_n) + n_seg)));
	PRT_TRY(s.bin.ensure(sizeof(uint4) * n + sizeof(uint32_t) * (nb + 2ull * n)));
	PRT_TRY(s.bbox.ensure(sizeof(float4) * 2ull * nb));
	PRT_TRY(s.bin_of.ensure(sizeof(uint32_t) * cap));
	PRT_TRY(s.tri_dest.ensure(sizeof(uint32_t) * n));
	const uint64_t scale_words = (S + 1ull) & ~1ull;  // doubles, keeps the rows 16-byte aligned
	if (p.collapse == 1) PRT_TRY(s.cost.ensure(sizeof(double) * scale_words + sizeof(float) * kCostRow * n));
	PRT_TRY(s.misc.ensure(sizeof(uint32_t) * words));
	PRT_TRY(s.scene_root.ensure(sizeof(uint32_t) * S));
	if (!s.host_misc) PRT_TRY(hipHostMalloc(&s.host_misc, sizeof(uint32_t) * misc_words(1)));
	PRT_TRY(out.nodes_q.ensure(sizeof(NodeQ) * cap));
	PRT_TRY(out.nodes_f.ensure(sizeof(NodeF) * cap));
	PRT_TRY(out.tris.ensure(sizeof(TriRec) * n));

	hipEvent_t ev[2] = {nullptr, nullptr};
	if (build_ms) {  // device time of the build kernels (allocations above are not counted)
		PRT_TRY(time_events(s, ev));
		PRT_TRY(hipEventRecord(ev[0], st));
	}
	uint32_t *misc = s.misc.as<uint32_t>();
	const float *tri_in = ss.tris ? ss.tris : s.tri_in.as<float>();
	hipLaunchKernelGGL(k_init_misc, dim3(blocks_for(words)), dim3(kBlock), 0, st, misc, words);
	hipLaunchKernelGGL(k_tri_prep, dim3(blocks_for(n, kPrepBlock)), dim3(kPrepBlock), 0, st, tri_in, n, off, S, s.tbox.as<float4>(),
	                   misc);
	hipLaunchKernelGGL(k_morton, dim3(blocks_for(n)), dim3(kBlock), 0, st, s.tbox.as<float4>(), n, misc,
	                   s.keys[0].as<uint64_t>(), s.vals[0].as<uint32_t>(), s.tri_dest.as<uint32_t>(),
	                   p.collapse == 1 ? s.cost.as<double>() : nullptr, S);
	int key_bits = kSceneShift;
	while (S > 1 && (1ull << (key_bits - kSceneShift)) < S) ++key_bits;
	int cur = 0;
	for (int shift = 0; shift < key_bits; shift += 8) {
		uint32_t *hist = s.hist.as<uint32_t>(), *seg = hist + hist_n;
		const uint64_t *kin = s.keys[cur].as<uint64_t>();
		uint64_t *kout = s.keys[cur ^ 1].as<uint64_t>();
		const uint32_t *vin = s.vals[cur].as<uint32_t>();
		uint32_t *vout = s.vals[cur ^ 1].as<uint32_t>();
		const dim3 tg(tiles), tb(kBlock);
		if (items == 1) hipLaunchKernelGGL(k_hist<1>, tg, tb, 0, st, kin, n, shift, hist, tiles);
		else if (items == 4) hipLaunchKernelGGL(k_hist<4>, tg, tb, 0, st, kin, n, shift, hist, tiles);
		else hipLaunchKernelGGL(k_hist<16>, tg, tb, 0, st, kin, n, shift, hist, tiles);
		hipLaunchKernelGGL(k_scan_seg, dim3(n_seg), tb, 0, st, hist, hist_n, seg);
		if (n_seg > static_cast<uint32_t>(kBlock)) hipLaunchKernelGGL(k_scan, dim3(1), dim3(1024), 0, st, seg, n_seg);
		if (items == 1) hipLaunchKernelGGL(k_scatter<1>, tg, tb, 0, st, kin, vin, kout, vout, n, shift, hist, seg, n_seg, tiles);
		else if (items == 4) hipLaunchKernelGGL(k_scatter<4>, tg, tb, 0, st, kin, vin, kout, vout, n, shift, hist, seg, n_seg, tiles);
		else hipLaunchKernelGGL(k_scatter<16>, tg, tb, 0, st, kin, vin, kout, vout, n, shift, hist, seg, n_seg, tiles);
		cur ^= 1;
	}
	const uint64_t *keys = s.keys[cur].as<uint64_t>();
	BinTree t;
	t.link = s.bin.as<uint4>();
	t.parent = reinterpret_cast<uint32_t *>(t.link + n);
	t.flag = t.parent + nb;
	t.plan = t.flag + n;
	t.box = s.bbox.as<float4>();
	t.n = n;
	uint32_t *scene_root = s.scene_root.as<uint32_t>();
	uint32_t *hm = static_cast<uint32_t *>(s.host_misc);
	const int leaf_size = std::max(1, std::min(kMaxLeaf, p.leaf_size)), width = std::max(2, std::min(8, p.width));
	CostCtx cc;
	cc.row = nullptr;
	cc.scale = nullptr;
	cc.scenes = S;
	cc.keys = keys;
	cc.param = ss.param;
	cc.leaf_size = leaf_size;
	cc.width = width;
	if (p.collapse == 1) {
		double *scale = s.cost.as<double>();
		cc.scale = scale;
		cc.row = reinterpret_cast<float *>(scale + scale_words);
	}
	// the clustering takes one scene (set_tris): several build together only with a fixed length
	const bool clustered = p.builder == 1 && !fixed && S == 1;
	PlocArgs pa;
	const uint32_t p_tiles = std::max(blocks_for(n, kStepTile), blocks_for(std::min(n, kSmallMax), kSmallTile));
	const uint32_t p_grid = p_tiles;  // a workgroup per tile of the first step and of the small ones
	int step = 0;
	uint32_t *lists = nullptr, *cnts = nullptr, *scans = nullptr, *segs = nullptr;
	const bool scanned = p_tiles > static_cast<uint32_t>(kMaxTiles);
	if (clustered) {
		const uint64_t list_n = static_cast<uint64_t>(p_tiles) * kStepTile;
		PRT_TRY(s.ploc.ensure(sizeof(uint32_t) * (2 * list_n + 4ull * (p_tiles + 1) + 2 * (p_tiles / kScanSeg + 2))));  // lists: at most n clusters in whole tiles
		static_assert(kSmallMax / kSmallTile + 1 < kMaxTiles, "small tiles fit the scan");
		lists = s.ploc.as<uint32_t>();
		cnts = lists + 2 * list_n;
		scans = cnts + 2 * (p_tiles + 1);
		segs = scans + 2 * (p_tiles + 1);
		pa.t = t;
		pa.cc = cc;
		pa.tbox = s.tbox.as<float4>();
		pa.sorted = s.vals[cur].as<uint32_t>();
		pa.misc = misc;
		pa.tiles_max = p_tiles;
	}
	// One step, in which buffer step & 1 is read and the other written.
	auto ploc_args = [&](int par) {
		const uint64_t list_n = static_cast<uint64_t>(p_tiles) * kStepTile;
		pa.step = static_cast<uint32_t>(step);
		pa.parity = par;
		pa.list_in = lists + par * list_n;
		pa.list_out = lists + (par ^ 1) * list_n;
		pa.cnt_in = cnts + par * (p_tiles + 1);
		pa.cnt_out = cnts + (par ^ 1) * (p_tiles + 1);
		pa.scan_in = scanned ? scans + par * (p_tiles + 1) : nullptr;
		pa.scan_out = scanned ? scans + (par ^ 1) * (p_tiles + 1) : nullptr;
		pa.pre = scanned ? segs : nullptr;
	};
	auto ploc_step = [&]() {
		ploc_args(step & 1);
		if (step == 0) {
			pa.pre = nullptr;
			hipLaunchKernelGGL(k_ploc_step<true>, dim3(p_grid), dim3(kStepBlock), 0, st, pa);
		} else {
			if (scanned) {
				const uint32_t ns = blocks_for(p_tiles + 1ull, kScanSeg);
				hipLaunchKernelGGL(k_scan_seg, dim3(ns), dim3(kBlock), 0, st, const_cast<uint32_t *>(pa.scan_in), p_tiles + 1, segs);
				hipLaunchKernelGGL(k_scan, dim3(1), dim3(1024), 0, st, segs, ns);
			}
			hipLaunchKernelGGL(k_ploc_step<false>, dim3(p_grid), dim3(kStepBlock), 0, st, pa);
		}
		++step;
	};
	auto ploc_tail = [&]() {
		ploc_args(0);
		uint32_t *bin_of = s.bin_of.as<uint32_t>();
		if (n <= kTailMax) hipLaunchKernelGGL(k_ploc_tail<true>, dim3(1), dim3(kTailBlock), 0, st, pa, bin_of);
		else hipLaunchKernelGGL(k_ploc_tail<false>, dim3(1), dim3(kTailBlock), 0, st, pa, bin_of);
	};
	if (clustered) {
		if (n > kTailMax) {
			// A step leaves about 0.8 of the clusters (0.79 to 0.81 measured on the room, the icosphere
			// and soups up to 1.5 M triangles): launch what that takes and two more without asking;
			// steps after the last needed one end at once.
			const int guess = 2 + static_cast<int>(std::ceil(std::log(static_cast<double>(n) / kTailMax) / std::log(1.22)));
			while (step < guess) ploc_step();
		}
		ploc_tail();
	} else {
		hipLaunchKernelGGL(k_scene_init, dim3(blocks_for(S)), dim3(kBlock), 0, st, off, S, n, scene_root);
		if (n > 1)
			hipLaunchKernelGGL(k_karras, dim3(blocks_for(n - 1)), dim3(kBlock), 0, st, keys, t, scene_root);
		if (cc.row)
			hipLaunchKernelGGL(k_bottomup<true>, dim3(blocks_for(n)), dim3(kBlock), 0, st, s.tbox.as<float4>(),
			                   s.vals[cur].as<uint32_t>(), t, cc);
		else
			hipLaunchKernelGGL(k_bottomup<false>, dim3(blocks_for(n)), dim3(kBlock), 0, st, s.tbox.as<float4>(),
			                   s.vals[cur].as<uint32_t>(), t, cc);
	}
	CollapseArgs ca;
	ca.t = t;
	ca.misc = misc;
	ca.bin_of = s.bin_of.as<uint32_t>();
	ca.tri_dest = s.tri_dest.as<uint32_t>();
	ca.nq = out.nodes_q.as<NodeQ>();
	ca.nf = out.nodes_f.as<NodeF>();
	ca.cc = cc;
	const uint32_t grid = std::min<uint32_t>(blocks_for(cap, kGroups), 2048);
	int level = 0;
	uint64_t level_nodes = S;  // most BVH8 nodes the next level can hold: the roots, then 8 children each
	auto roots = [&]() {
		hipLaunchKernelGGL(k_roots, dim3(std::max(blocks_for(S), blocks_for(2 * (kMaxLevels + 2)))), dim3(kBlock), 0, st, misc, ca.bin_of, scene_root, S);
		level = 0;
		level_nodes = S;
	};
	auto collapse = [&]() {
		// a grid for that many nodes (the kernel's loop covers any count), so that the small top
		// levels do not dispatch thousands of idle waves
		const uint32_t lgrid = std::min<uint32_t>(grid, blocks_for(level_nodes, kGroups));
		level_nodes = std::min<uint64_t>(level_nodes * 8u, cap);
		if (ca.cc.row) hipLaunchKernelGGL(k_collapse<true>, dim3(lgrid), dim3(kBlock), 0, st, ca, level);
		else hipLaunchKernelGGL(k_collapse<false>, dim3(lgrid), dim3(kBlock), 0, st, ca, level);
		++level;
	};
	auto emit = [&]() {
		hipLaunchKernelGGL(k_emit_tris, dim3(blocks_for(n)), dim3(kBlock), 0, st, tri_in, s.vals[cur].as<uint32_t>(), keys,
		                   off, s.tri_dest.as<uint32_t>(), n, out.tris.as<TriRec>(), misc);
	};
	auto read_back = [&]() -> hipError_t {
		PRT_TRY(hipGetLastError());
		PRT_TRY(hipMemcpyAsync(hm, misc, sizeof(uint32_t) * misc_words(1), hipMemcpyDeviceToHost, st));
		return hipSuccess;
	};
	if (!clustered) roots();
	if (fixed) {
		// a few level launches, then the rest of the tree depth first
		while (level < std::min(ss.levels, kFixedTopLevels)) collapse();
		if (ca.cc.row) hipLaunchKernelGGL(k_collapse_dfs<true>, dim3(grid), dim3(kBlock), 0, st, ca, level);
		else hipLaunchKernelGGL(k_collapse_dfs<false>, dim3(grid), dim3(kBlock), 0, st, ca, level);
		emit();
		if (ss.box) hipLaunchKernelGGL(k_scene_boxes, dim3(blocks_for(6ull * S)), dim3(kBlock), 0, st, misc, S, ss.box);
		hipLaunchKernelGGL(k_check_done, dim3(1), dim3(64), 0, st, misc, n);
		PRT_TRY(hipGetLastError());
		out.n_nodes = cap;  // an upper bound: the device holds the count
		out.depth = static_cast<uint32_t>(ss.levels);
		out.n_ncull = kNcullUnknown;  // not read back: traversals handle never-cull slots
		return hipSuccess;
	}
	// The whole build is enqueued on a guess of its steps and levels and read back once; what the
	// guess fell short of is run afterwards. The level guess: the room (262,144 triangles) has 10 or
	// 11 levels, the icosphere (81,920) 7, soups of 1.5 M triangles 10; a level too many costs an
	// empty launch (2 us), a synchronisation about 25 us.
	const int guess_levels = std::min(kMaxLevels, 3 + static_cast<int>(std::ceil(std::log2(static_cast<double>(n) + 1.0) / 2.0)));
	while (level < guess_levels) collapse();
	emit();
	if (ss.box) hipLaunchKernelGGL(k_scene_boxes, dim3(blocks_for(6ull * S)), dim3(kBlock), 0, st, misc, S, ss.box);
	PRT_TRY(read_back());
	if (build_ms) PRT_TRY(hipEventRecord(ev[1], st));
	PRT_TRY(hipStreamSynchronize(st));
	bool again = false;
	if (!(hm[M_ERR] & 1u)) {
		if (clustered && !hm[M_PDONE]) {
			while (!hm[M_PDONE]) {
				if (step >= kPlocMaxSteps) return hipErrorUnknown;
				for (int k = 0; k < 16; ++k) ploc_step();
				ploc_tail();
				PRT_TRY(read_back());
				PRT_TRY(hipStreamSynchronize(st));
			}
			level = 0;
			level_nodes = S;
			while (level < guess_levels) collapse();
			again = true;
		}
		while (again || hm[M_LCNT + 2 * level] != 0u) {
			if (!again) {  // the last launched level has left nodes for the next one
				if (level >= kMaxLevels) return hipErrorUnknown;
				for (int k = 0; k < 8 && level < kMaxLevels; ++k) collapse();
			}
			hipLaunchKernelGGL(k_clear_err, dim3(1), dim3(64), 0, st, misc);
			emit();
			PRT_TRY(read_back());
			if (build_ms) PRT_TRY(hipEventRecord(ev[1], st));
			PRT_TRY(hipStreamSynchronize(st));
			again = false;
		}
	}
	if (build_ms) {
		float ms = 0.0f;
		PRT_TRY(hipEventElapsedTime(&ms, ev[0], ev[1]));
		*build_ms = ms;
	}
	*bad_input = (hm[M_ERR] & 1u) != 0;
	if (*bad_input) return hipSuccess;  // the caller reports the input; the tree is not used
	if (hm[M_ERR] & 2u) return hipErrorUnknown;  // inconsistent build
	for (int k = 0; k < 6; ++k) out.scene_box[k] = ordered_float(hm[M_SCENE + 6 + k]);
	uint32_t nodes = 0, placed = 0;
	for (int l = 0; l < level && hm[M_LCNT + 2 * l]; ++l) {
		if (hm[M_LBASE + l] != nodes) return hipErrorUnknown;
		out.levels.push_back(nodes);
		nodes += hm[M_LCNT + 2 * l];
		placed += hm[M_LCNT + 2 * (l + 1) + 1];
	}
	out.n_nodes = nodes;
	out.depth = static_cast<uint32_t>(out.levels.size());
	out.n_ncull = hm[M_NCULL];
	if (placed != n || nodes > cap) return hipErrorUnknown;  // incomplete build
	return hipSuccess;
#undef PRT_TRY
}

hipError_t refit_bvh8(BuildScratch &s, Bvh8 &b, const float *tris, hipStream_t st, bool *bad_input, double *refit_ms) {
#define PRT_TRY(x)                                                                                 \
	do {                                                                                           \
		hipError_t e_ = (x);                                                                       \
		if (e_ != hipSuccess) return e_;                                                           \
	} while (0)
	*bad_input = false;
	const uint64_t n = b.n_tris;
	if (n == 0 || b.n_nodes == 0) return hipSuccess;
	if (b.levels.empty()) return hipErrorInvalidValue;  // the build leaves them
	PRT_TRY(s.refit_box.ensure(sizeof(float4) * 2ull * b.n_nodes));
	PRT_TRY(s.misc.ensure(sizeof(uint32_t) * misc_words(1)));
	if (!s.host_misc) PRT_TRY(hipHostMalloc(&s.host_misc, sizeof(uint32_t) * misc_words(1)));
	hipEvent_t ev[2] = {nullptr, nullptr};
	if (refit_ms) {
		PRT_TRY(time_events(s, ev));
		PRT_TRY(hipEventRecord(ev[0], st));
	}
	uint32_t *misc = s.misc.as<uint32_t>();
	hipLaunchKernelGGL(k_init_misc, dim3(blocks_for(misc_words(1))), dim3(kBlock), 0, st, misc, misc_words(1));
	hipLaunchKernelGGL(k_refit_tris, dim3(blocks_for(n)), dim3(kBlock), 0, st, tris, b.tris.as<TriRec>(),
	                   static_cast<uint32_t>(n), misc);
	RefitArgs ra;
	ra.tris = b.tris.as<TriRec>();
	ra.nq = b.nodes_q.as<NodeQ>();
	ra.nf = b.nodes_f.as<NodeF>();
	ra.box = s.refit_box.as<float4>();
	ra.n_nodes = b.n_nodes;
	ra.n_tris = static_cast<uint32_t>(n);
	ra.misc = misc;
	auto level_end = [&](size_t l) { return l + 1 < b.levels.size() ? b.levels[l + 1] : b.n_nodes; };
	for (size_t l = b.levels.size(); l > 0;) {  // levels l - 1, l - 2, ... are left
		FewLevels few;
		few.count = 0;
		few.bound[0] = level_end(l - 1);
		while (l > 0 && few.count < kFewLevels && level_end(l - 1) - b.levels[l - 1] <= kFewNodes) few.bound[++few.count] = b.levels[--l];
		if (few.count) hipLaunchKernelGGL(k_refit_few, dim3(1), dim3(kFewBlock), 0, st, ra, few);
		if (l == 0) break;
		if (few.count == kFewLevels) continue;
		--l;
		const uint32_t begin = b.levels[l], end = level_end(l);
		hipLaunchKernelGGL(k_refit_level, dim3(std::min<uint32_t>(blocks_for(end - begin, kGroups), 2048)), dim3(kBlock), 0, st, ra,
		                   begin, end);
	}
	PRT_TRY(hipGetLastError());
	if (refit_ms) PRT_TRY(hipEventRecord(ev[1], st));
	PRT_TRY(hipMemcpyAsync(s.host_misc, misc, sizeof(uint32_t) * misc_words(1), hipMemcpyDeviceToHost, st));
	PRT_TRY(hipStreamSynchronize(st));
	if (refit_ms) {
		float ms = 0.0f;
		PRT_TRY(hipEventElapsedTime(&ms, ev[0], ev[1]));
		*refit_ms = ms;
	}
	const uint32_t err = static_cast<const uint32_t *>(s.host_misc)[M_ERR];
	*bad_input = (err & 1u) != 0;
	if (*bad_input) return hipSuccess;  // the caller reports the input; the tree is not used
	if (err & 2u) return hipErrorUnknown;
	b.n_ncull = static_cast<const uint32_t *>(s.host_misc)[M_NCULL];
	for (int k = 0; k < 6; ++k) b.scene_box[k] = ordered_float(static_cast<const uint32_t *>(s.host_misc)[M_SCENE + 6 + k]);
	return hipSuccess;
#undef PRT_TRY
}

hipError_t build_errors(BuildScratch &s, hipStream_t st, uint32_t *flags) {
	*flags = 0;
	if (!s.misc.ptr || !s.host_misc) return hipSuccess;
	uint32_t *hm = static_cast<uint32_t *>(s.host_misc);
	hipError_t e = hipMemcpyAsync(hm, s.misc.ptr, sizeof(uint32_t) * misc_words(1), hipMemcpyDeviceToHost, st);
	if (e == hipSuccess) e = hipStreamSynchronize(st);
	if (e == hipSuccess) *flags = hm[M_ERR];
	return e;
}

}  // namespace prt
