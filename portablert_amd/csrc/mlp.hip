// The learned t_max seeding network: a 192 -> 256 -> 256 -> 256 -> 4097 MLP (ReLU hidden
// layers, BF16 weights and activations, FP32 accumulation) trained and run with hand-written
// MFMA kernels on gfx950. It predicts, per ray, the BVH8 cluster (subtree) that holds the hit
// triangle, or "miss" (logit 4096). No counterpart in the reference.
//
// Every matrix product is C[M,N] = A[M,K] * B[N,K]^T with both operands K-contiguous (bf16),
// computed by k_gemm with v_mfma_f32_16x16x32_bf16 (lane layout checked on the device:
// A[l%16][(l/16)*8+i], B[(l/16)*8+i][l%16], C[(l/16)*4+i][l%16]). Weights are kept as
// W^T [out, in] (forward) and W [in, out] (backward data gradient); weight gradients use
// transposed activations so that the batch is the contiguous reduction dimension.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "common.h"
#include "internal.h"
#include "mlp.h"

namespace prt {
namespace {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kBK = 32;             // K of one MFMA
constexpr int kThreads = 256;
constexpr int kSplits = 8;  // of the batch in a weight gradient
// split-K scratch: every layer's partial weight gradients
constexpr size_t kLayerWeights[4] = {static_cast<size_t>(kMlpHidden) * kMlpIn, static_cast<size_t>(kMlpHidden) * kMlpHidden,
                                     static_cast<size_t>(kMlpHidden) * kMlpHidden, static_cast<size_t>(kMlpOutPad) * kMlpHidden};
constexpr size_t kSplitFloats = kSplits * (kLayerWeights[0] + kLayerWeights[1] + kLayerWeights[2] + kLayerWeights[3]);

__device__ __forceinline__ uint16_t f2bf(float f) {
	// round to nearest even (inputs are finite here)
	const uint32_t u = __float_as_uint(f);
	const uint32_t r = u + 0x7FFFu + ((u >> 16) & 1u);
	return static_cast<uint16_t>(r >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float(static_cast<uint32_t>(h) << 16); }

// Place of weight (row, col) of a W^T [rows][cols] in its fragment order: 16 rows x 32 columns follow
// each other as the MFMA operand of 64 lanes x 8 values, so a wave loads a fragment as 1 KB in a row.
// Of 32 rows, tile 0 holds rows 0-3, 8-11, 16-19, 24-27 and tile 1 the others: a lane's results of the
// two tiles are then 8 consecutive rows, which is its operand in the next layer.
__device__ __forceinline__ size_t fragment_at(int row, int col, int cols) {
	const int tile = (row >> 5) * 2 + ((row >> 2) & 1), at = ((row >> 3) & 3) * 4 + (row & 3);
	return (static_cast<size_t>(tile) * (cols >> 5) + (col >> 5)) * 512 + ((((col >> 3) & 3) << 4) | at) * 8 + (col & 7);
}
// First of the 4 rows that a lane of group quad (lane / 16) holds of the results of a tile.
__device__ __forceinline__ int fragment_row(int tile, int quad) { return (tile >> 1) * 32 + quad * 8 + (tile & 1) * 4; }

enum Epi : int {
	E_BIAS_F32 = 0,   // out f32 = acc + bias[n]
	E_MASK_BF16 = 1,  // out bf16 = acc * (aux_bf16[m][n] > 0)
	E_F32 = 2         // out f32 = acc (split-K partial: out += split * M * N)
};

struct GemmArgs {
	const uint16_t *A;   // [M][lda] bf16
	const uint16_t *B;   // [N][ldb] bf16
	void *out;
	const float *bias;   // [N] (E_BIAS_*)
	const uint16_t *aux; // [M][ldo] bf16 (E_MASK_BF16)
	int M, N, K, lda, ldb, ldo;
	int k_split;         // K range per y-slice (split-K), multiple of kBK
};

// C tile (BM x BN) of one workgroup: 4 waves, each BM/2 x BN/2 as 16 x 16 MFMA tiles. K runs in
// tiles of TK through two LDS buffers: the next tile's loads are issued before this tile's MFMAs
// and stored after them, one barrier a tile. The MFMA's A operand holds the columns of C and its B
// operand the rows, so that a lane's four results are four consecutive columns of one row and go
// out as one 16-byte (fp32) or 8-byte (bf16) store; each result is the same chain of products
// over K in the same order. Workgroups that share rows of A follow each other on one XCD.
//
// With 32-wide K tiles loaded and multiplied in turn, and the results through LDS to stores of one
// element each, a batch of 8,192 took 298 us for the logits (138 MB of fp32 written: 27 us at the
// 5.1 TB/s of a large copy), 73 us for a data gradient and 56 us for a weight gradient.
template <int EPI, int BM, int BN, int TK>
__global__ __launch_bounds__(kThreads) void k_gemm(GemmArgs g) {
	constexpr int kTKPad = TK + 8;  // row stride of an LDS tile: 16-byte reads without bank conflicts
	constexpr int RC = TK / 8;      // 16-byte chunks a row
	constexpr int CA = BM * RC / kThreads, CB = BN * RC / kThreads;  // and a thread
	constexpr int TM = BM / 32, TN = BN / 32;                                   // MFMA tiles a wave
	__shared__ __align__(16) uint16_t As[2][BM * kTKPad], Bs[2][BN * kTKPad];
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	const int tiles_n = (g.N + BN - 1) / BN, tiles = tiles_n * ((g.M + BM - 1) / BM);
	const int per_xcd = gridDim.x / 8;  // workgroup b runs on XCD b % 8
	const int t = static_cast<int>(blockIdx.x % 8) * per_xcd + static_cast<int>(blockIdx.x / 8);
	if (t >= tiles) return;
	const int m0 = t / tiles_n * BM, n0 = t % tiles_n * BN;
	const int wr = (wave >> 1) * (BM / 2), wc = (wave & 1) * (BN / 2);
	const int kbeg = blockIdx.y * g.k_split, kend = min(g.K, kbeg + g.k_split);
	f32x4 acc[TM][TN];
#pragma unroll
	for (int i = 0; i < TM; ++i)
#pragma unroll
		for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
	u32x4 ra[CA], rb[CB];
	const u32x4 zero = {0u, 0u, 0u, 0u};
	auto load = [&](int k0) {
#pragma unroll
		for (int c = 0; c < CA; ++c) {
			const int q = tid + c * kThreads, row = m0 + (q / RC), k = k0 + (q % RC) * 8;
			ra[c] = row < g.M && k < kend ? *reinterpret_cast<const u32x4 *>(g.A + static_cast<size_t>(row) * g.lda + k) : zero;
		}
#pragma unroll
		for (int c = 0; c < CB; ++c) {
			const int q = tid + c * kThreads, row = n0 + (q / RC), k = k0 + (q % RC) * 8;
			rb[c] = row < g.N && k < kend ? *reinterpret_cast<const u32x4 *>(g.B + static_cast<size_t>(row) * g.ldb + k) : zero;
		}
	};
	auto store = [&](int buf) {
#pragma unroll
		for (int c = 0; c < CA; ++c) {
			const int q = tid + c * kThreads;
			*reinterpret_cast<u32x4 *>(As[buf] + (q / RC) * kTKPad + (q % RC) * 8) = ra[c];
		}
#pragma unroll
		for (int c = 0; c < CB; ++c) {
			const int q = tid + c * kThreads;
			*reinterpret_cast<u32x4 *>(Bs[buf] + (q / RC) * kTKPad + (q % RC) * 8) = rb[c];
		}
	};
	if (kbeg < kend) {
		load(kbeg);
		store(0);
	}
	int buf = 0;
	for (int k0 = kbeg; k0 < kend; k0 += TK, buf ^= 1) {
		__syncthreads();
		const bool more = k0 + TK < kend;
		if (more) load(k0 + TK);
#pragma unroll
		for (int kk = 0; kk < TK / kBK; ++kk) {
			if (k0 + kk * kBK >= kend) break;  // K is a multiple of 32
			bf16x8 af[TM], bfr[TN];
#pragma unroll
			for (int i = 0; i < TM; ++i)
				af[i] = *reinterpret_cast<const bf16x8 *>(As[buf] + (wr + i * 16 + (lane & 15)) * kTKPad + kk * kBK + (lane >> 4) * 8);
#pragma unroll
			for (int j = 0; j < TN; ++j)
				bfr[j] = *reinterpret_cast<const bf16x8 *>(Bs[buf] + (wc + j * 16 + (lane & 15)) * kTKPad + kk * kBK + (lane >> 4) * 8);
#pragma unroll
			for (int i = 0; i < TM; ++i)
#pragma unroll
				for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bfr[j], af[i], acc[i][j], 0, 0, 0);
		}
		if (more) store(buf ^ 1);  // read two tiles ago: the barrier above has passed since
	}
	// lane: row m = lane % 16 of a tile, columns n = (lane / 16) * 4 ..+3 (N is a multiple of 4)
#pragma unroll
	for (int i = 0; i < TM; ++i) {
		const int m = m0 + wr + i * 16 + (lane & 15);
		if (m >= g.M) continue;
#pragma unroll
		for (int j = 0; j < TN; ++j) {
			const int n = n0 + wc + j * 16 + (lane >> 4) * 4;
			if (n >= g.N) continue;
			f32x4 x = acc[i][j];
			const size_t o = static_cast<size_t>(m) * g.ldo + n;
			if constexpr (EPI == E_BIAS_F32) {
				const f32x4 b = *reinterpret_cast<const f32x4 *>(g.bias + n);
#pragma unroll
				for (int e = 0; e < 4; ++e) x[e] = x[e] + b[e];
			}
			if constexpr (EPI == E_MASK_BF16) {
				uint16_t h[4];
				const uint2 av = *reinterpret_cast<const uint2 *>(g.aux + o);
				const uint32_t aw[4] = {av.x & 0xFFFFu, av.x >> 16, av.y & 0xFFFFu, av.y >> 16};
#pragma unroll
				for (int e = 0; e < 4; ++e) h[e] = bf2f(static_cast<uint16_t>(aw[e])) > 0.0f ? f2bf(x[e]) : static_cast<uint16_t>(0);
				*reinterpret_cast<uint2 *>(reinterpret_cast<uint16_t *>(g.out) + o) =
				    make_uint2(h[0] | static_cast<uint32_t>(h[1]) << 16, h[2] | static_cast<uint32_t>(h[3]) << 16);
			} else {
				float *dst = reinterpret_cast<float *>(g.out) + (EPI == E_F32 ? static_cast<size_t>(blockIdx.y) * g.M * g.ldo : 0);
				*reinterpret_cast<f32x4 *>(dst + o) = x;
			}
		}
	}
}

// Positional encoding: 6 inputs (origin scaled to [-1,1] by the scene box, direction) times
// 16 frequencies 2^(j/2) * pi, sin and cos: 192 features, bf16, in the order (input, frequency,
// sin/cos).

__device__ __forceinline__ uint32_t encode_pair(float y) {
	return static_cast<uint32_t>(f2bf(__builtin_amdgcn_sinf(y))) | (static_cast<uint32_t>(f2bf(__builtin_amdgcn_cosf(y))) << 16);
}

// Inputs a0..a0+2, frequencies j0..j0+7 of one ray, each (sin, cos) pair as one 32-bit store: four
// threads per ray.
__device__ __forceinline__ void encode_quarter(const float *r, float4 lo, float4 inv_ext, int a0, int j0, uint16_t *o) {
	float in[3];
	if (a0 == 0) {
		in[0] = (r[0] - lo.x) * inv_ext.x * 2.0f - 1.0f;
		in[1] = (r[1] - lo.y) * inv_ext.y * 2.0f - 1.0f;
		in[2] = (r[2] - lo.z) * inv_ext.z * 2.0f - 1.0f;
	} else {
		in[0] = r[3];
		in[1] = r[4];
		in[2] = r[5];
	}
	uint32_t *o32 = reinterpret_cast<uint32_t *>(o);
#pragma unroll
	for (int q = 0; q < 3; ++q) {
#pragma unroll
		for (int jj = 0; jj < 8; ++jj) {
			const int j = j0 + jj;  // v_sin/v_cos take revolutions: sin(2 pi y), y = in * 2^(j/2) / 2
			const float y = in[q] * (0.5f * exp2f(0.5f * static_cast<float>(j)));
			o32[(a0 + q) * 16 + j] = encode_pair(y);
		}
	}
}

// ------------------------------------------------------------- fused inference with top-4
//
// One workgroup (4 waves) takes 64 rays through the whole network: encoding, the three hidden
// layers and the 4097 output logits, keeping the activations in LDS (X, 64 x 256 bf16) and
// streaming W^T tiles of 64 output neurons (prefetched into registers one tile ahead) from L2,
// with v_mfma_f32_16x16x32_bf16 over K in steps of 32. In every layer each wave loads all 64 rows
// of the layer's input into registers and owns 16 of each tile's 64 neurons, so each W fragment
// read from LDS serves 64 rows; a hidden layer writes its outputs to X as its tiles finish
// (two barriers per layer). In the output layer each wave fetches and stages only its own 16
// rows of W^T (in its slice of two tile buffers, one of them in X's space), and passes its
// 64 x 16 logits through the same slice to its 64 lanes, one ray
// each, which keep a running top-4 (value descending, index ascending). No wave reads another's
// slice, so the 65 output tiles run without a barrier; the four waves' lists of a ray are merged
// at the end, and no logit leaves the chip. The tiles are software-pipelined: a wave issues tile
// t + 1's MFMAs interleaved with the compares of tile t's logits against its running bound.
// The workgroup uses 66 KB of LDS, so two share a CU.
constexpr int kFRows = 64;     // rays per workgroup
constexpr int kFCols = 64;     // output neurons per W tile
constexpr int kFStride = 264;  // bf16 row stride of X and W (16-byte reads without bank conflicts)

struct FusedArgs {
	const float *rays;
	uint64_t first;
	int rows;
	float4 lo, inv_ext;
	const uint16_t *w[4];  // W^T bf16 [out][in]; in fragment order for k_mlp_top1
	const float *b[4];
	uint32_t *seeds;       // [rows][4] (k_mlp_top4) or [rows] (k_mlp_top1)
};

// One hidden layer computed per wave, without barriers between its tiles: every wave loads all 64
// rows of X[:, :K] into registers, then owns 16 of each 64-neuron tile's columns and stages only
// its own 16 rows of W^T in its slice of the W region (the next tile's rows prefetched into
// registers during the MFMAs), so each W fragment read from LDS serves 64 rows. Once every wave
// holds X, X's region takes the outputs as each tile finishes. Two barriers per layer; each
// output element is the same MFMA chain over K in the same order as before.
template <int K>
__device__ __forceinline__ void hidden_layer_pw(uint16_t *X, uint16_t *W, const uint16_t *wt, const float *bias,
                                                int lane, int wave) {
	constexpr int KS = K / kBK;       // MFMA K steps
	constexpr int RC = K / 8;         // 16-byte chunks per W^T row
	constexpr int CH = 16 * RC / 64;  // chunks per lane of a 16-row slice
	bf16x8 xr[4][KS];
#pragma unroll
	for (int i = 0; i < 4; ++i)
#pragma unroll
		for (int kk = 0; kk < KS; ++kk)
			xr[i][kk] = *reinterpret_cast<const bf16x8 *>(X + (i * 16 + (lane & 15)) * kFStride + kk * kBK + (lane >> 4) * 8);
	uint16_t *ws = W + wave * 16 * kFStride;  // this wave's slice
	auto fetch = [&](int t, u32x4 q[CH]) {
#pragma unroll
		for (int j = 0; j < CH; ++j) {
			const int c = lane + 64 * j;
			q[j] = *reinterpret_cast<const u32x4 *>(wt + static_cast<size_t>(t * kFCols + wave * 16 + c / RC) * K + (c % RC) * 8);
		}
	};
	auto store = [&](const u32x4 q[CH]) {
#pragma unroll
		for (int j = 0; j < CH; ++j) {
			const int c = lane + 64 * j;
			*reinterpret_cast<u32x4 *>(ws + (c / RC) * kFStride + (c % RC) * 8) = q[j];
		}
	};
	u32x4 pre[CH];
	fetch(0, pre);
	__syncthreads();  // every wave holds X in registers: X's region takes the outputs
	store(pre);
#pragma unroll
	for (int t = 0; t < 4; ++t) {
		if (t + 1 < 4) fetch(t + 1, pre);
		__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
		__builtin_amdgcn_wave_barrier();
		__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
		f32x4 acc[4];
#pragma unroll
		for (int i = 0; i < 4; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
		for (int kk = 0; kk < KS; ++kk) {
			const bf16x8 bfr = *reinterpret_cast<const bf16x8 *>(ws + (lane & 15) * kFStride + kk * kBK + (lane >> 4) * 8);
#pragma unroll
			for (int i = 0; i < 4; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xr[i][kk], bfr, acc[i], 0, 0, 0);
		}
		if (t + 1 < 4) store(pre);  // this wave's MFMAs have read the slice (LDS operations of one wave complete in order)
		const int col = t * kFCols + wave * 16 + (lane & 15);
		const float bj = bias[col];
#pragma unroll
		for (int i = 0; i < 4; ++i)
#pragma unroll
			for (int e = 0; e < 4; ++e)
				X[(i * 16 + (lane >> 4) * 4 + e) * kFStride + col] = f2bf(fmaxf(acc[i][e] + bj, 0.0f));
	}
	__syncthreads();
}

// The encodings of rays r0..r0+ROWS-1 in X; rows past the end are zero. A quarter of a ray at a time:
// inputs 0-2 or 3-5, frequencies 0-7 or 8-15.
template <int ROWS>
__device__ __forceinline__ void encode_rows(const FusedArgs &a, int r0, uint16_t *X) {
	for (int task = threadIdx.x; task < ROWS * 4; task += 256) {
		const int row = task >> 2, half = (task >> 1) & 1, fq = task & 1;
		uint16_t *o = X + row * kFStride;
		if (r0 + row < a.rows) {
			encode_quarter(a.rays + 6 * (a.first + r0 + row), a.lo, a.inv_ext, half * 3, fq * 8, o);
		} else {
			uint32_t *o32 = reinterpret_cast<uint32_t *>(o);
#pragma unroll
			for (int q = 0; q < 3; ++q)
#pragma unroll
				for (int jj = 0; jj < 8; ++jj) o32[(half * 3 + q) * 16 + fq * 8 + jj] = 0u;
		}
	}
}

// Encoding and hidden layers of 64 rays a workgroup, with every activation also written out for
// the backward pass: one launch instead of four (77 us for 8,192 rays).
struct HiddenOut {
	uint16_t *x0, *h[3];
};

__global__ __launch_bounds__(256, 2) void k_hidden(FusedArgs a, HiddenOut out) {
	__shared__ __align__(16) uint16_t X[kFRows * kFStride];
	__shared__ __align__(16) uint16_t W[kFCols * kFStride];
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	const int r0 = blockIdx.x * kFRows;
	auto write = [&](uint16_t *dst, int cols) {
		for (int q = tid; q < kFRows * cols / 8; q += 256) {
			const int r = q / (cols / 8), c = (q % (cols / 8)) * 8;
			if (r0 + r < a.rows)
				*reinterpret_cast<u32x4 *>(dst + static_cast<size_t>(r0 + r) * cols + c) = *reinterpret_cast<const u32x4 *>(X + r * kFStride + c);
		}
	};
	encode_rows<kFRows>(a, r0, X);
	__syncthreads();
	write(out.x0, kMlpIn);
	hidden_layer_pw<kMlpIn>(X, W, a.w[0], a.b[0], lane, wave);
	write(out.h[0], kMlpHidden);
	hidden_layer_pw<kMlpHidden>(X, W, a.w[1], a.b[1], lane, wave);
	write(out.h[1], kMlpHidden);
	hidden_layer_pw<kMlpHidden>(X, W, a.w[2], a.b[2], lane, wave);
	write(out.h[2], kMlpHidden);
}

__device__ __forceinline__ bool top_better(float va, uint32_t ia, float vb, uint32_t ib) {
	return va > vb || (va == vb && ia < ib);
}

// Inserts (x, n) into a list of 4 kept in (value descending, index ascending) order.
__device__ __forceinline__ void top_insert(float v[4], uint32_t ix[4], float x, uint32_t n) {
	if (!top_better(x, n, v[3], ix[3])) return;
	v[3] = x;
	ix[3] = n;
#pragma unroll
	for (int k = 3; k > 0; --k) {
		if (top_better(v[k], ix[k], v[k - 1], ix[k - 1])) {
			const float tv = v[k]; v[k] = v[k - 1]; v[k - 1] = tv;
			const uint32_t ti = ix[k]; ix[k] = ix[k - 1]; ix[k - 1] = ti;
		}
	}
}

// Merges the list of the lane `mask` away into this lane's list.
__device__ __forceinline__ void top_merge(float v[4], uint32_t ix[4], int mask) {
	float ov[4];
	uint32_t oi[4];
#pragma unroll
	for (int q = 0; q < 4; ++q) {
		ov[q] = __shfl_xor(v[q], mask);
		oi[q] = __shfl_xor(ix[q], mask);
	}
#pragma unroll
	for (int q = 0; q < 4; ++q) top_insert(v, ix, ov[q], oi[q]);
}

__global__ __launch_bounds__(256, 2) void k_mlp_top4(FusedArgs a) {
	__shared__ __align__(16) uint16_t X[kFRows * kFStride];
	__shared__ __align__(16) uint16_t W[kFCols * kFStride];
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	const int r0 = blockIdx.x * kFRows;
	encode_rows<kFRows>(a, r0, X);
	__syncthreads();
	hidden_layer_pw<kMlpIn>(X, W, a.w[0], a.b[0], lane, wave);
	hidden_layer_pw<kMlpHidden>(X, W, a.w[1], a.b[1], lane, wave);
	hidden_layer_pw<kMlpHidden>(X, W, a.w[2], a.b[2], lane, wave);
	// output layer: all 64 rows of the last hidden layer in every wave's registers; each wave
	// computes 16 of a tile's 64 columns, so each W fragment read from LDS serves 64 rows
	const int oc = wave * 16;
	bf16x8 ar[4][kMlpHidden / kBK];
#pragma unroll
	for (int i = 0; i < 4; ++i)
#pragma unroll
		for (int kk = 0; kk < kMlpHidden / kBK; ++kk)
			ar[i][kk] = *reinterpret_cast<const bf16x8 *>(X + (i * 16 + (lane & 15)) * kFStride + kk * kBK + (lane >> 4) * 8);
	// Output tiles without barriers: every wave fetches, stages and reads only its own 16 rows of
	// each W^T tile (columns oc .. oc + 15 of the 64 output neurons), in its own slice of the two
	// tile buffers, and passes its 64 x 16 block of logits through that slice (free once its
	// MFMAs have read it) to its 64 lanes, one row each: lane r keeps the running top-4 of row r
	// over this wave's columns. The four waves' lists of a row are merged at the end.
	constexpr int kSliceStride = 20;  // fp32 row stride of a wave's 64 x 16 logit block (16-byte rows, no bank conflicts)
	auto slice = [&](auto *buf) { return buf + oc * kFStride; };
	// this wave's 16 rows of tile t's W^T, 16 x 512 bytes: chunk c = lane + 64 j is row c / 32,
	// 16-byte column group c % 32
	auto w_chunk = [&](int t, int j) {
		const int c = lane + 64 * j;
		return *reinterpret_cast<const u32x4 *>(a.w[3] + static_cast<size_t>(t * kFCols + oc + c / 32) * kMlpHidden +
		                                        (c % 32) * 8);
	};
	auto fetch_own = [&](int t, u32x4 q[8]) {
#pragma unroll
		for (int j = 0; j < 8; ++j) q[j] = w_chunk(t, j);
	};
	auto store_own = [&](uint16_t *buf, const u32x4 q[8]) {
#pragma unroll
		for (int j = 0; j < 8; ++j) {
			const int c = lane + 64 * j;
			*reinterpret_cast<u32x4 *>(slice(buf) + (c / 32) * kFStride + (c % 32) * 8) = q[j];
		}
	};
	float v[4] = {-__builtin_inff(), -__builtin_inff(), -__builtin_inff(), -__builtin_inff()};
	uint32_t ix[4] = {0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu};
	constexpr int kOutTiles = (kMlpOut + kFCols - 1) / kFCols;  // the last one holds the miss logit
	// bias of this lane's column (padding columns: -inf, never taken)
	auto bias_of = [&](int t) {
		const int col = t * kFCols + oc + (lane & 15);
		const float b = a.b[3][col < kMlpOut ? col : kMlpOut - 1];  // no branch around the load
		return col < kMlpOut ? b : -__builtin_inff();
	};
	auto mma = [&](const uint16_t *buf, f32x4 acc[4]) {
#pragma unroll
		for (int i = 0; i < 4; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
		for (int kk = 0; kk < kMlpHidden / kBK; ++kk) {
			const bf16x8 bfr = *reinterpret_cast<const bf16x8 *>(slice(buf) + (lane & 15) * kFStride + kk * kBK + (lane >> 4) * 8);
#pragma unroll
			for (int i = 0; i < 4; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ar[i][kk], bfr, acc[i], 0, 0, 0);
		}
	};
	// this wave's logits into its slice of buf, whose W the MFMAs that made them have read (LDS
	// operations of one wave complete in order)
	auto put_logits = [&](uint16_t *buf, const f32x4 acc[4], float bias) {
		float *C = reinterpret_cast<float *>(slice(buf));
#pragma unroll
		for (int i = 0; i < 4; ++i)
#pragma unroll
			for (int e = 0; e < 4; ++e) C[(i * 16 + (lane >> 4) * 4 + e) * kSliceStride + (lane & 15)] = acc[i][e] + bias;
	};
	auto sync_wave = [&]() {
		__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
		__builtin_amdgcn_wave_barrier();
		__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
	};
	// lane r compares row r's 16 logits of tile t with its 4th best (a strict comparison keeps
	// the lower index first; held entries come from earlier tiles)
	auto scan_mask = [&](const uint16_t *buf) {
		const float *crow = reinterpret_cast<const float *>(slice(buf)) + lane * kSliceStride;
		uint32_t cand = 0;
#pragma unroll
		for (int c4 = 0; c4 < 4; ++c4) {
			const float4 q = *reinterpret_cast<const float4 *>(crow + c4 * 4);
			const float xs[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
			for (int e = 0; e < 4; ++e) cand |= xs[e] > v[3] ? (1u << (c4 * 4 + e)) : 0u;
		}
		return cand;
	};
	auto insert = [&](const uint16_t *buf, uint32_t cand, int t) {
		const float *crow = reinterpret_cast<const float *>(slice(buf)) + lane * kSliceStride;
		const int nbase = t * kFCols + oc;
		while (cand) {
			const int c = __builtin_ctz(cand);
			cand &= cand - 1u;
			const float x = crow[c];
			if (x > v[3]) {
				v[3] = x;
				ix[3] = static_cast<uint32_t>(nbase + c);
#pragma unroll
				for (int k = 3; k > 0; --k) {
					if (v[k] > v[k - 1]) {
						const float tv = v[k]; v[k] = v[k - 1]; v[k - 1] = tv;
						const uint32_t ti = ix[k]; ix[k] = ix[k - 1]; ix[k - 1] = ti;
					}
				}
			}
		}
	};
	// Software pipeline over the output tiles: while the matrix core computes tile t + 1, the
	// wave scans tile t's logits. Buffer roles alternate: at the top of iteration t, `cur` is
	// free (its W was read by tile t's MFMAs, whose results are in acc) and `nxt` holds tile
	// t + 1's W.
	f32x4 acc[4];
	uint16_t *cur = W, *nxt = X;
	{
		u32x4 p0[8];
		fetch_own(0, p0);
		__syncthreads();  // every wave has its rows of X in registers: X's space becomes a tile buffer
		store_own(cur, p0);
		fetch_own(1, p0);
		store_own(nxt, p0);
		sync_wave();
		mma(cur, acc);
	}
	float bias = bias_of(0);
	for (int t = 0; t < kOutTiles - 1; ++t) {
		put_logits(cur, acc, bias);
		bias = bias_of(t + 1);
		sync_wave();
		// Tile t + 1's MFMAs with tile t's scan in hand-ordered steps (a scheduling barrier after
		// each keeps the order): the four logit reads and the first two B fragment reads, then per
		// K step the B fragment read two steps ahead, four MFMAs, one W prefetch load and two of
		// the sixteen compares, which issue while the matrix core works.
		const float *crow = reinterpret_cast<const float *>(slice(cur)) + lane * kSliceStride;
		float lf[16];
#pragma unroll
		for (int c4 = 0; c4 < 4; ++c4) {
			const float4 q = *reinterpret_cast<const float4 *>(crow + c4 * 4);
			lf[c4 * 4] = q.x;
			lf[c4 * 4 + 1] = q.y;
			lf[c4 * 4 + 2] = q.z;
			lf[c4 * 4 + 3] = q.w;
		}
		const uint16_t *bsrc = slice(nxt) + (lane & 15) * kFStride + (lane >> 4) * 8;
		bf16x8 bq[kMlpHidden / kBK];
		bq[0] = *reinterpret_cast<const bf16x8 *>(bsrc);
		bq[1] = *reinterpret_cast<const bf16x8 *>(bsrc + kBK);
#pragma unroll
		for (int i = 0; i < 4; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
		__builtin_amdgcn_sched_barrier(0);
		u32x4 pre[8];
		// tile t + 2's W rows of this wave: chunk kk of w_chunk is 2 kk rows further
		const uint16_t *wsrc = a.w[3] + static_cast<size_t>(((t + 2) % kOutTiles) * kFCols + oc + (lane >> 5)) * kMlpHidden +
		                       (lane & 31) * 8;
		uint32_t cand = 0;
		const float thr = v[3];
#pragma unroll
		for (int kk = 0; kk < kMlpHidden / kBK; ++kk) {
			if (kk + 2 < kMlpHidden / kBK) bq[kk + 2] = *reinterpret_cast<const bf16x8 *>(bsrc + (kk + 2) * kBK);
			pre[kk] = *reinterpret_cast<const u32x4 *>(wsrc + 2 * kk * kMlpHidden);
#pragma unroll
			for (int i = 0; i < 4; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ar[i][kk], bq[kk], acc[i], 0, 0, 0);
			cand |= (lf[2 * kk] > thr ? (1u << (2 * kk)) : 0u) | (lf[2 * kk + 1] > thr ? (1u << (2 * kk + 1)) : 0u);
			__builtin_amdgcn_sched_barrier(0);
		}
		insert(cur, cand, t);
		sync_wave();
		store_own(cur, pre);  // tile t + 2's W into the buffer tile t's logits have left
		uint16_t *tmp = cur; cur = nxt; nxt = tmp;
	}
	put_logits(cur, acc, bias);
	sync_wave();
	insert(cur, scan_mask(cur), kOutTiles - 1);
	// merge the four waves' lists of each row (value descending, index ascending)
	__syncthreads();
	float *mv = reinterpret_cast<float *>(W);
	uint32_t *mi = reinterpret_cast<uint32_t *>(W) + 4 * 64 * 4;
#pragma unroll
	for (int k = 0; k < 4; ++k) {
		mv[(wave * 64 + lane) * 4 + k] = v[k];
		mi[(wave * 64 + lane) * 4 + k] = ix[k];
	}
	__syncthreads();
	const int orow = tid >> 2, opart = tid & 3;
#pragma unroll
	for (int k = 0; k < 4; ++k) {
		v[k] = mv[(opart * 64 + orow) * 4 + k];
		ix[k] = mi[(opart * 64 + orow) * 4 + k];
	}
	top_merge(v, ix, 1);
	top_merge(v, ix, 2);
	if (opart == 0 && r0 + orow < a.rows) {
		const uint32_t res[4] = {ix[0], ix[1], ix[2], ix[3]};
		reinterpret_cast<uint4 *>(a.seeds)[r0 + orow] = make_uint4(res[0], res[1], res[2], res[3]);
	}
}

// ------------------------------------------------------------- fused inference, the best cluster only
//
// One seed per ray is the traversal's default, and its argmax needs neither the logits' trip through
// LDS nor the insertions of k_mlp_top4. A workgroup takes 64 rays, all of them as MFMA B operands
// in every wave's registers; each wave owns 16 of a tile's 64 neurons and reads their weights from L2
// straight into its A operands, a tile ahead, without LDS and without barriers. The results are the
// transposed tile: a lane holds four neurons of one ray per 16 x 16 block and keeps that ray's best over
// its neurons, four instructions an element, issued between the next tile's MFMAs. Each logit is the
// same chain of products over K as in k_mlp_top4. 1 Mi rays: 1.93 ms (1.34 PFLOP/s) against 2.9 in
// k_mlp_top4; 16,384 rays take 38 us. Bound by the weights' way from L2 (2.4 MB per 64 rays, 20 TB/s).
constexpr int kRayTiles = 4, kTop1Rows = kRayTiles * 16;

template <int K>
__device__ __forceinline__ void load_rays(const uint16_t *X, int lane, bf16x8 (&xr)[kRayTiles][K / kBK]) {
#pragma unroll
	for (int i = 0; i < kRayTiles; ++i)
#pragma unroll
		for (int kk = 0; kk < K / kBK; ++kk)
			xr[i][kk] = *reinterpret_cast<const bf16x8 *>(X + (i * 16 + (lane & 15)) * kFStride + kk * kBK + (lane >> 4) * 8);
}

template <int K>
__device__ __forceinline__ void hidden_layer_t(uint16_t *X, const uint16_t *wt, const float *bias, int lane, int wave) {
	constexpr int RT = kRayTiles, KS = K / kBK;
	const uint16_t *wsrc = wt + static_cast<size_t>(wave * 4 * KS) * 512 + lane * 8;
	bf16x8 w[KS], xr[RT][KS];
#pragma unroll
	for (int kk = 0; kk < KS; ++kk) w[kk] = *reinterpret_cast<const bf16x8 *>(wsrc + kk * 512);
	load_rays<K>(X, lane, xr);
	__syncthreads();  // every wave holds X in registers: its space takes the outputs
#pragma unroll
	for (int t = 0; t < 4; ++t) {
		f32x4 acc[RT];
#pragma unroll
		for (int i = 0; i < RT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
		const int n = fragment_row(wave * 4 + t, lane >> 4);
		const f32x4 b = *reinterpret_cast<const f32x4 *>(bias + n);
#pragma unroll
		for (int kk = 0; kk < KS; ++kk) {
#pragma unroll
			for (int i = 0; i < RT; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[kk], xr[i][kk], acc[i], 0, 0, 0);
			if (t + 1 < 4) w[kk] = *reinterpret_cast<const bf16x8 *>(wsrc + ((t + 1) * KS + kk) * 512);
		}
#pragma unroll
		for (int i = 0; i < RT; ++i) {
			uint32_t h[4];
#pragma unroll
			for (int e = 0; e < 4; ++e) h[e] = f2bf(fmaxf(acc[i][e] + b[e], 0.0f));
			*reinterpret_cast<uint2 *>(X + (i * 16 + (lane & 15)) * kFStride + n) = make_uint2(h[0] | h[1] << 16, h[2] | h[3] << 16);
		}
	}
	__syncthreads();
}

__global__ __launch_bounds__(256, 2) void k_mlp_top1(FusedArgs a) {
	constexpr int kRows = kTop1Rows, RT = kRayTiles, KS = kMlpHidden / kBK;
	constexpr int kTiles = (kMlpOut + kFCols - 1) / kFCols;  // the last one holds the miss logit
	static_assert(kTiles * kFCols <= kMlpOutPad && kTiles % 2 == 1, "padding rows are read; tiles go in pairs after the first");
	__shared__ __align__(16) uint16_t X[kRows * kFStride];
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, quad = lane >> 4;
	const int r0 = blockIdx.x * kRows;
	encode_rows<kRows>(a, r0, X);
	__syncthreads();
	hidden_layer_t<kMlpIn>(X, a.w[0], a.b[0], lane, wave);
	hidden_layer_t<kMlpHidden>(X, a.w[1], a.b[1], lane, wave);
	hidden_layer_t<kMlpHidden>(X, a.w[2], a.b[2], lane, wave);
	const uint16_t *wsrc = a.w[3] + wave * KS * 512 + lane * 8;
	const float *bsrc = a.b[3] + fragment_row(wave, quad);
	bf16x8 w[KS], xr[RT][KS];
#pragma unroll
	for (int kk = 0; kk < KS; ++kk) w[kk] = *reinterpret_cast<const bf16x8 *>(wsrc + kk * 512);
	load_rays<kMlpHidden>(X, lane, xr);
	float best[RT];
	uint32_t code[RT];  // tile * 4 + element
#pragma unroll
	for (int i = 0; i < RT; ++i) {
		best[i] = -__builtin_inff();
		code[i] = 0xFFFFFFFFu;
	}
	// a strict comparison keeps the lower neuron at equal logits
	auto take = [&](int i, int e, float x, uint32_t c) {
		const bool more = x > best[i];
		best[i] = more ? x : best[i];
		code[i] = more ? c + e : code[i];
	};
	// tile t's MFMAs into acc with the comparisons of tile t - 1's results (old, its bias ob) between
	// them; each K step's weights of tile t + 1 are loaded once its own are used
	auto step = [&](int t, f32x4 (&acc)[RT], f32x4 &b, const f32x4 (&old)[RT], const f32x4 &ob, bool first) {
		const int next = t + 1 < kTiles ? t + 1 : t;
		const uint16_t *ws = wsrc + static_cast<size_t>(next) * 4 * KS * 512;
		b = *reinterpret_cast<const f32x4 *>(bsrc + t * kFCols);
		const uint32_t c = static_cast<uint32_t>(t - 1) * 4u;
#pragma unroll
		for (int kk = 0; kk < KS; ++kk) {
#pragma unroll
			for (int i = 0; i < RT; ++i)
				acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[kk], xr[i][kk], kk == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[i], 0, 0, 0);
			w[kk] = *reinterpret_cast<const bf16x8 *>(ws + kk * 512);
			if (!first) {
#pragma unroll
				for (int q = 0; q < RT / 2; ++q) {
					const int at = kk * (RT / 2) + q;
					take(at / 4, at % 4, old[at / 4][at % 4] + ob[at % 4], c);
				}
			}
			__builtin_amdgcn_sched_barrier(0);
		}
	};
	f32x4 acc0[RT], acc1[RT], b0, b1;
	step(0, acc0, b0, acc1, b0, true);
	for (int t = 1; t < kTiles; t += 2) {
		step(t, acc1, b1, acc0, b0, false);
		step(t + 1, acc0, b0, acc1, b1, false);
	}
#pragma unroll
	for (int e = 0; e < 4; ++e) {  // the last tile's padding neurons are never taken
		if ((kTiles - 1) * kFCols + fragment_row(wave, quad) + e < kMlpOut) {
#pragma unroll
			for (int i = 0; i < RT; ++i) take(i, e, acc0[i][e] + b0[e], (kTiles - 1) * 4);
		}
	}
	// the best of a ray's four lanes, then of the four waves
	__syncthreads();
	float *mv = reinterpret_cast<float *>(X);
	uint32_t *mi = reinterpret_cast<uint32_t *>(X) + 4 * kRows;
#pragma unroll
	for (int i = 0; i < RT; ++i) {
		float x = best[i];
		uint32_t n = code[i] == 0xFFFFFFFFu ? code[i] : (code[i] >> 2) * kFCols + fragment_row(wave, quad) + (code[i] & 3u);
#pragma unroll
		for (int m = 16; m < 64; m *= 2) {
			const float ox = __shfl_xor(x, m);
			const uint32_t on = __shfl_xor(n, m);
			if (top_better(ox, on, x, n)) {
				x = ox;
				n = on;
			}
		}
		if (quad == 0) {
			mv[wave * kRows + i * 16 + lane] = x;
			mi[wave * kRows + i * 16 + lane] = n;
		}
	}
	__syncthreads();
	if (tid < kRows && r0 + tid < a.rows) {
		float x = mv[tid];
		uint32_t n = mi[tid];
#pragma unroll
		for (int q = 1; q < 4; ++q) {
			const float ox = mv[q * kRows + tid];
			const uint32_t on = mi[q * kRows + tid];
			if (top_better(ox, on, x, n)) {
				x = ox;
				n = on;
			}
		}
		a.seeds[r0 + tid] = n;
	}
}

// Many rays: a wave takes 64 rays through the whole network by itself, and a workgroup's four waves
// share the weights, which pass through two LDS buffers of two 16-neuron tiles each (a barrier per
// pair of tiles), so 256 rays cost one stream of weights from L2 instead of four. Activations never
// leave the wave's registers: a lane computes its own operand of the encoding, and its results of a
// hidden layer's two tiles are its operand of the next layer (the order of the fragments). The
// hidden layers take 32 rays at a time, whose inputs and outputs fit the registers together. 1 Mi
// rays: 1.78 ms (1.45 PFLOP/s) against 1.93 in k_mlp_top1. The comparisons hide behind the products:
// with a quarter of them left out (the bias as the products' first addend) it took the same 1.78 ms.
constexpr int kManyRows = 256;
constexpr int kBiasAt[4] = {0, kMlpHidden, 2 * kMlpHidden, 3 * kMlpHidden};
constexpr int kPairs = (kMlpOut - 1) / 32;  // pairs of output tiles before the one that holds the miss logit
static_assert(kMlpOut == kPairs * 32 + 1 && kPairs % 2 == 0 && kMlpOutPad >= kPairs * 32 + 32, "output tiles");

__global__ __launch_bounds__(256, 2) void k_mlp_top1_many(FusedArgs a) {
	constexpr int KS = kMlpHidden / kBK, KS0 = kMlpIn / kBK;
	__shared__ __align__(16) uint16_t W[2][2 * KS * 512];
	__shared__ __align__(16) float bias[kBiasAt[3] + kPairs * 32 + 32];
	const uint32_t tid = threadIdx.x;
	const int lane = tid & 63, wave = tid >> 6, quad = lane >> 4;
	const int r0 = blockIdx.x * kManyRows + wave * 64 + (lane & 15);
	u32x4 pre[KS / 2];
	auto fetch = [&](const uint16_t *src, int ks) {  // the weights of two tiles, ks fragments each
		uint32_t zero = 0u;  // hidden from the compiler, which else keeps all layers' addresses across the loop below
		asm volatile("" : "+s"(zero));
		src += zero;
#pragma unroll
		for (int c = 0; c < KS / 2; ++c)
			if (c < ks / 2) pre[c] = *reinterpret_cast<const u32x4 *>(reinterpret_cast<const uint8_t *>(src + c * 2048) + tid * 16u);
	};
	auto store = [&](uint16_t *dst, int ks) {
#pragma unroll
		for (int c = 0; c < KS / 2; ++c)
			if (c < ks / 2) *reinterpret_cast<u32x4 *>(dst + (c * 256 + tid) * 8) = pre[c];
	};
	auto frag = [&](const uint16_t *w, int f) { return *reinterpret_cast<const bf16x8 *>(w + f * 512 + lane * 8); };
	fetch(a.w[0], KS0);
#pragma unroll
	for (int l = 0; l < 3; ++l) bias[kBiasAt[l] + tid] = a.b[l][tid];
	for (uint32_t k = tid; k < kPairs * 32 + 32; k += 256) bias[kBiasAt[3] + k] = a.b[3][k];
	store(W[0], KS0);
	__syncthreads();

	bf16x8 lo[2][KS], hi[2][KS];  // the last hidden layer of rays 0-31 and 32-63
	// one hidden layer; W[0] holds its first pair of tiles, and the next layer's at the end
	auto layer = [&](auto ks_, const auto &in, bf16x8 (&out)[2][KS], const uint16_t *w, const float *b, const uint16_t *next, int next_ks) {
		constexpr int ks = decltype(ks_)::value;
#pragma unroll
		for (int p = 0; p < KS; ++p) {
			if (p + 1 < KS) fetch(w + (p + 1) * 2 * ks * 512, ks);
			else fetch(next, next_ks);
			f32x4 acc[2][2];  // tile, ray tile
#pragma unroll
			for (int t = 0; t < 2; ++t)
#pragma unroll
				for (int i = 0; i < 2; ++i) acc[t][i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
			for (int kk = 0; kk < ks; ++kk)
#pragma unroll
				for (int t = 0; t < 2; ++t) {
					const bf16x8 f = frag(W[p & 1], t * ks + kk);
#pragma unroll
					for (int i = 0; i < 2; ++i) acc[t][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f, in[i][kk], acc[t][i], 0, 0, 0);
				}
			store(W[(p + 1) & 1], p + 1 < KS ? ks : next_ks);
			union {
				uint32_t u[4];
				bf16x8 v;
			} o[2];
#pragma unroll
			for (int t = 0; t < 2; ++t) {
				const f32x4 bt = *reinterpret_cast<const f32x4 *>(b + fragment_row(2 * p + t, quad));
#pragma unroll
				for (int i = 0; i < 2; ++i)
#pragma unroll
					for (int h = 0; h < 2; ++h)
						o[i].u[t * 2 + h] = f2bf(fmaxf(acc[t][i][2 * h] + bt[2 * h], 0.0f)) |
						                    static_cast<uint32_t>(f2bf(fmaxf(acc[t][i][2 * h + 1] + bt[2 * h + 1], 0.0f))) << 16;
			}
#pragma unroll
			for (int i = 0; i < 2; ++i) out[i][p] = o[i].v;
			__syncthreads();
		}
	};
#pragma unroll 1
	for (int half = 0; half < 2; ++half) {
#pragma unroll
		for (int i = 0; i < 2; ++i)
#pragma unroll
			for (int kk = 0; kk < KS; ++kk) lo[i][kk] = hi[i][kk];
		bf16x8 x[2][KS0], h[2][KS];
#pragma unroll
		for (int i = 0; i < 2; ++i) {
			const int row = min(r0 + (half * 2 + i) * 16, a.rows - 1);
			const float *r = a.rays + 6 * (a.first + row);
			float in[6];
			in[0] = (r[0] - a.lo.x) * a.inv_ext.x * 2.0f - 1.0f;
			in[1] = (r[1] - a.lo.y) * a.inv_ext.y * 2.0f - 1.0f;
			in[2] = (r[2] - a.lo.z) * a.inv_ext.z * 2.0f - 1.0f;
			in[3] = r[3];
			in[4] = r[4];
			in[5] = r[5];
#pragma unroll
			for (int kk = 0; kk < KS0; ++kk) {
				union {
					uint32_t u[4];
					bf16x8 v;
				} o;
#pragma unroll
				for (int q = 0; q < 4; ++q) {
					const float y = in[kk] * (0.5f * exp2f(0.5f * static_cast<float>(quad * 4 + q)));
					o.u[q] = encode_pair(y);
				}
				x[i][kk] = o.v;
			}
		}
		constexpr auto k0 = std::integral_constant<int, KS0>();
		constexpr auto k1 = std::integral_constant<int, KS>();
		layer(k0, x, hi, a.w[0], bias + kBiasAt[0], a.w[1], KS);
		layer(k1, hi, h, a.w[1], bias + kBiasAt[1], a.w[2], KS);
		layer(k1, h, hi, a.w[2], bias + kBiasAt[2], half == 0 ? a.w[0] : a.w[3], KS);
	}

	float best[4];
	uint32_t code[4];  // tile * 4 + element
#pragma unroll
	for (int i = 0; i < 4; ++i) {
		best[i] = -__builtin_inff();
		code[i] = 0xFFFFFFFFu;
	}
	auto take = [&](int i, int e, float x, uint32_t c) {  // strict: the lower neuron at equal logits
		const bool more = x > best[i];
		best[i] = more ? x : best[i];
		code[i] = more ? c + e : code[i];
	};
	bf16x8 f[4];
	// tile t's MFMAs from fragments w, w + 1, .. with the comparisons of tile t - 1's results between them
	auto tile = [&](const uint16_t *w, int first, int last, f32x4 (&acc)[4], const f32x4 (&old)[4], const f32x4 &ob, uint32_t c, bool compare) {
#pragma unroll
		for (int kk = 0; kk < KS; ++kk) {
			const int p = first + kk;
#pragma unroll
			for (int i = 0; i < 4; ++i)
				acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[p & 3], i < 2 ? lo[i & 1][kk] : hi[i & 1][kk],
				                                                 kk == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[i], 0, 0, 0);
			if (p + 4 < last) f[p & 3] = frag(w, p + 4);
			if (compare) {
#pragma unroll
				for (int q = 0; q < 2; ++q) {
					const int at = kk * 2 + q;
					take(at / 4, at % 4, old[at / 4][at % 4] + ob[at % 4], c);
				}
			}
			__builtin_amdgcn_sched_barrier(0);
		}
	};
	f32x4 acc0[4], acc1[4], b0, b1;
#pragma unroll
	for (int i = 0; i < 4; ++i) acc1[i] = f32x4{-__builtin_inff(), -__builtin_inff(), -__builtin_inff(), -__builtin_inff()};
	b1 = f32x4{0.f, 0.f, 0.f, 0.f};
	const float *bo = bias + kBiasAt[3] + quad * 8;
	for (int p = 0; p < kPairs; ++p) {
		const uint16_t *w = W[p & 1];
		fetch(a.w[3] + static_cast<size_t>(p + 1) * 2 * KS * 512, KS);
#pragma unroll
		for (int q = 0; q < 4; ++q) f[q] = frag(w, q);
		b0 = *reinterpret_cast<const f32x4 *>(bo + p * 32);
		__builtin_amdgcn_sched_barrier(0);
		tile(w, 0, 2 * KS, acc0, acc1, b1, static_cast<uint32_t>(2 * p - 1) * 4u, true);
		b1 = *reinterpret_cast<const f32x4 *>(bo + p * 32 + 4);
		tile(w, KS, 2 * KS, acc1, acc0, b0, static_cast<uint32_t>(2 * p) * 4u, true);
		store(W[(p + 1) & 1], KS);
		__syncthreads();
	}
#pragma unroll
	for (int q = 0; q < 4; ++q) f[q] = frag(W[0], q);
	tile(W[0], 0, KS, acc0, acc1, b1, static_cast<uint32_t>(2 * kPairs - 1) * 4u, true);
	if (quad == 0) {  // the miss logit; the rest of the tile is padding
#pragma unroll
		for (int i = 0; i < 4; ++i) take(i, 0, acc0[i][0] + bo[kPairs * 32], static_cast<uint32_t>(2 * kPairs) * 4u);
	}
#pragma unroll
	for (int i = 0; i < 4; ++i) {  // the best of a ray's four lanes
		float x = best[i];
		uint32_t n = code[i] == 0xFFFFFFFFu ? code[i] : fragment_row(static_cast<int>(code[i] >> 2), quad) + (code[i] & 3u);
#pragma unroll
		for (int m = 16; m < 64; m *= 2) {
			const float ox = __shfl_xor(x, m);
			const uint32_t on = __shfl_xor(n, m);
			if (top_better(ox, on, x, n)) {
				x = ox;
				n = on;
			}
		}
		if (quad == 0 && r0 + i * 16 < a.rows) a.seeds[r0 + i * 16] = n;
	}
}

// Softmax cross-entropy over the first n_valid logits of each row. Writes dlogits =
// (softmax - onehot) / batch as bf16 (0 in padding columns) and each row's share of the mean loss. One
// workgroup a row, whose logits stay in registers (17 a thread) between the maximum, the sum and the
// gradient: bound by memory (207 MB for 8,192 rows). Reading the row three times with block-wide
// LDS reductions it took 134 us, and 113 us with one atomic per row on the loss. The sum is each thread's columns in order, then the tree over
// the threads 128, 64, .. 1 apart.
constexpr int kRowCols = (kMlpOutPad + 255) / 256;

__global__ __launch_bounds__(256) void k_softmax_ce(const float *__restrict__ logits, const uint32_t *__restrict__ label,
                                                    int rows, int ld, int n_valid, float inv_batch,
                                                    uint16_t *__restrict__ dlog, float *__restrict__ loss_row) {
	const int row = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	if (row >= rows) return;
	__shared__ float red[256];
	const float *L = logits + static_cast<size_t>(row) * ld;
	float x[kRowCols];
	float mx = -__builtin_inff();
#pragma unroll
	for (int k = 0; k < kRowCols; ++k) {
		const int c = tid + 256 * k;
		x[k] = c < n_valid ? L[c] : -__builtin_inff();
		mx = fmaxf(mx, x[k]);
	}
	for (int sh = 32; sh > 0; sh >>= 1) mx = fmaxf(mx, __shfl_xor(mx, sh));
	if (lane == 0) red[wave] = mx;
	__syncthreads();
	mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
	__syncthreads();
	float sum = 0.0f;
#pragma unroll
	for (int k = 0; k < kRowCols; ++k) {
		x[k] = expf(x[k] - mx);
		if (tid + 256 * k < n_valid) sum += x[k];
	}
	red[tid] = sum;
	__syncthreads();
	sum = (red[lane] + red[lane + 128]) + (red[lane + 64] + red[lane + 192]);
	for (int sh = 32; sh > 0; sh >>= 1) sum += __shfl_down(sum, sh);
	sum = __shfl(sum, 0);
	const uint32_t y = label[row];
	const float inv = 1.0f / sum;
	uint16_t *D = dlog + static_cast<size_t>(row) * ld;
#pragma unroll
	for (int k = 0; k < kRowCols; ++k) {
		const int c = tid + 256 * k;
		float gval = 0.0f;
		if (c < n_valid) gval = (x[k] * inv - (static_cast<uint32_t>(c) == y ? 1.0f : 0.0f)) * inv_batch;
		if (c < ld) D[c] = f2bf(gval);
	}
	if (tid == 0) loss_row[row] = (logf(sum) + mx - L[y]) * inv_batch;
}

// out[c][r] = in[r][c] for a bf16 [rows][cols] matrix (rows a multiple of 32, cols of 64), in tiles
// of 128 rows x 64 columns through LDS with 16-byte loads and stores. SUM: the tile's column sums
// too, each over its 128 rows in order, to part[row tile][c] (the bias gradient's first stage:
// reading the matrix again for it took 32 us a layer).
constexpr int kTrRows = 128, kTrCols = 64, kTrPad = 66;

template <bool SUM>
__global__ __launch_bounds__(256) void k_transpose(const uint16_t *__restrict__ in, int rows, int cols, int ld_in,
                                                   uint16_t *__restrict__ out, int ld_out, float *__restrict__ part) {
	__shared__ uint16_t t[kTrRows][kTrPad];
	const int c0 = blockIdx.x * kTrCols, r0 = blockIdx.y * kTrRows, tid = threadIdx.x;
	const int n_rows = min(kTrRows, rows - r0);
#pragma unroll
	for (int q = 0; q < kTrRows * kTrCols / 8 / 256; ++q) {
		const int k = tid + q * 256, r = k >> 3, c = (k & 7) * 8;
		uint4 v = make_uint4(0u, 0u, 0u, 0u);
		if (r < n_rows) v = *reinterpret_cast<const uint4 *>(in + static_cast<size_t>(r0 + r) * ld_in + c0 + c);
		uint32_t *d = reinterpret_cast<uint32_t *>(&t[r][c]);  // 4-byte aligned rows
		d[0] = v.x;
		d[1] = v.y;
		d[2] = v.z;
		d[3] = v.w;
	}
	__syncthreads();
#pragma unroll
	for (int q = 0; q < kTrRows * kTrCols / 8 / 256; ++q) {
		const int k = tid + q * 256, c = k >> 4, r = (k & 15) * 8;
		if (r >= n_rows) continue;
		uint32_t w[4];
#pragma unroll
		for (int e = 0; e < 4; ++e) w[e] = t[r + 2 * e][c] | static_cast<uint32_t>(t[r + 2 * e + 1][c]) << 16;
		*reinterpret_cast<uint4 *>(out + static_cast<size_t>(c0 + c) * ld_out + r0 + r) = make_uint4(w[0], w[1], w[2], w[3]);
	}
	if (SUM && tid < kTrCols) {
		float s = 0.0f;
#pragma unroll 16
		for (int r = 0; r < n_rows; ++r) s += bf2f(t[r][tid]);
		part[static_cast<size_t>(blockIdx.y) * cols + c0 + tid] = s;
	}
}

// Sums partials: g[i] = sum_s part[s][i], in order (n a multiple of 4).
__device__ __forceinline__ f32x4 sum_parts(const float *__restrict__ part, int splits, size_t n, size_t i) {
	f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
	for (int k = 0; k < splits; ++k) {
		const f32x4 v = *reinterpret_cast<const f32x4 *>(part + k * n + i);
#pragma unroll
		for (int e = 0; e < 4; ++e) s[e] += v[e];
	}
	return s;
}

// One layer's weights or bias in the update launch.
struct AdamPart {
	float *p, *g, *m, *v;
	const float *part;   // partial gradients [splits][n]
	int splits;
	uint16_t *bf, *bft;  // weights: bf16 copies W^T [rows][cols] and W [cols][rows]
	uint16_t *frag;      // and W^T in fragment order
	int rows, cols;      // bias: rows entries, of which the first cols are updated
	unsigned first;      // first workgroup
};

struct AdamArgs {
	AdamPart w[4], b[4];
	unsigned loss_block;  // the workgroup that sums the rows' losses
	const float *loss_row;
	float *loss;
	int n_loss;
	float lr, b1, b2, eps, c1, c2;  // lr 0: the gradients only
};

// Partial gradients summed and stored and, with lr > 0, an Adam step on the fp32 master
// parameters: every layer's weights and biases in one launch (eight took 50 us a batch, mostly
// launches). Weights in tiles of 32 x 64, which also refresh both bf16 copies, the transposed one
// through LDS (element by element its stores were 8 KB apart).
__global__ __launch_bounds__(256) void k_update(AdamArgs a) {
	__shared__ uint16_t t[32][66];
	__shared__ float red[256];
	const int tid = threadIdx.x;
	const unsigned b = blockIdx.x;
	if (b == a.loss_block) {
		float s = 0.0f;
		for (int i = tid; i < a.n_loss; i += 256) s += a.loss_row[i];
		red[tid] = s;
		__syncthreads();
		for (int sh = 128; sh > 0; sh >>= 1) {
			if (tid < sh) red[tid] += red[tid + sh];
			__syncthreads();
		}
		if (tid == 0) *a.loss = red[0];
		return;
	}
	auto step = [&](float g, float &p, float &m, float &v) {
		m = a.b1 * m + (1.0f - a.b1) * g;
		v = a.b2 * v + (1.0f - a.b2) * g * g;
		p = p - a.lr * (m * a.c1) / (sqrtf(v * a.c2) + a.eps);
	};
#pragma unroll
	for (int l = 0; l < 4; ++l) {
		const AdamPart &q = a.b[l];
		if (b < q.first || b >= q.first + (q.rows + 255) / 256) continue;
		const int i = static_cast<int>(b - q.first) * 256 + tid;
		if (i >= q.rows) return;
		float s = 0.0f;
#pragma unroll 16
		for (int k = 0; k < q.splits; ++k) s += q.part[static_cast<size_t>(k) * q.rows + i];
		q.g[i] = s;
		if (i < q.cols && a.lr > 0.0f) step(s, q.p[i], q.m[i], q.v[i]);
		return;
	}
#pragma unroll
	for (int l = 0; l < 4; ++l) {
		const AdamPart &q = a.w[l];
		const unsigned tiles_c = q.cols / 64, tiles = tiles_c * (q.rows / 32);
		if (b < q.first || b >= q.first + tiles) continue;
		const int r0 = static_cast<int>((b - q.first) / tiles_c) * 32, c0 = static_cast<int>((b - q.first) % tiles_c) * 64;
		const size_t n = static_cast<size_t>(q.rows) * q.cols;
#pragma unroll
		for (int h = 0; h < 2; ++h) {
			const int k = tid + h * 256, r = k >> 4, c = (k & 15) * 4;
			const size_t i = static_cast<size_t>(r0 + r) * q.cols + c0 + c;
			const f32x4 g = sum_parts(q.part, q.splits, n, i);
			*reinterpret_cast<f32x4 *>(q.g + i) = g;
			if (!(a.lr > 0.0f)) continue;
			f32x4 m = *reinterpret_cast<f32x4 *>(q.m + i), v = *reinterpret_cast<f32x4 *>(q.v + i), p = *reinterpret_cast<f32x4 *>(q.p + i);
#pragma unroll
			for (int e = 0; e < 4; ++e) {
				float pe = p[e], me = m[e], ve = v[e];
				step(g[e], pe, me, ve);
				p[e] = pe;
				m[e] = me;
				v[e] = ve;
			}
			*reinterpret_cast<f32x4 *>(q.m + i) = m;
			*reinterpret_cast<f32x4 *>(q.v + i) = v;
			*reinterpret_cast<f32x4 *>(q.p + i) = p;
			const uint32_t w0 = f2bf(p[0]) | static_cast<uint32_t>(f2bf(p[1])) << 16, w1 = f2bf(p[2]) | static_cast<uint32_t>(f2bf(p[3])) << 16;
			*reinterpret_cast<uint2 *>(q.bf + i) = make_uint2(w0, w1);
			*reinterpret_cast<uint2 *>(q.frag + fragment_at(r0 + r, c0 + c, q.cols)) = make_uint2(w0, w1);
			reinterpret_cast<uint32_t *>(&t[r][c])[0] = w0;
			reinterpret_cast<uint32_t *>(&t[r][c])[1] = w1;
		}
		if (!(a.lr > 0.0f)) return;
		__syncthreads();
		const int c = tid >> 2, r = (tid & 3) * 8;
		uint32_t w[4];
#pragma unroll
		for (int e = 0; e < 4; ++e) w[e] = t[r + 2 * e][c] | static_cast<uint32_t>(t[r + 2 * e + 1][c]) << 16;
		*reinterpret_cast<uint4 *>(q.bft + static_cast<size_t>(c0 + c) * q.rows + r0 + r) = make_uint4(w[0], w[1], w[2], w[3]);
		return;
	}
}

// Deterministic initialisation (uniform +-sqrt(6/(fan_in+fan_out)) from a counter hash).
__global__ __launch_bounds__(256) void k_init(float *__restrict__ w, size_t n, int fan_in, int fan_out, uint64_t seed,
                                              int rows_valid, int cols) {
	const size_t i = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x;
	if (i >= n) return;
	uint64_t z = seed + i * 0x9E3779B97F4A7C15ull;
	z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
	z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
	z ^= z >> 31;
	const float u = static_cast<float>(z >> 40) * 0x1p-24f * 2.0f - 1.0f;
	const float a = sqrtf(6.0f / static_cast<float>(fan_in + fan_out));
	w[i] = (static_cast<int>(i / cols) < rows_valid) ? u * a : 0.0f;
}

__global__ __launch_bounds__(256) void k_fill_f32(float *p, size_t n, float v) {
	const size_t i = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x;
	if (i < n) p[i] = v;
}

__global__ __launch_bounds__(256) void k_to_bf16(const float *__restrict__ p, size_t n, uint16_t *__restrict__ bf,
                                                 uint16_t *__restrict__ bft, uint16_t *__restrict__ frag, int rows, int cols) {
	const size_t i = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x;
	if (i >= n) return;
	const uint16_t h = f2bf(p[i]);
	bf[i] = h;
	frag[fragment_at(static_cast<int>(i / cols), static_cast<int>(i % cols), cols)] = h;
	if (bft) bft[static_cast<size_t>(i % cols) * rows + i / cols] = h;
}

inline unsigned blocks(size_t n, int per = 256) { return static_cast<unsigned>((n + per - 1) / per); }

// 64 x 64 tiles take K 128 at a time: with one or two workgroups a CU the loads' latency counts,
// once per tile of K.
template <int EPI, int BM, int BN>
hipError_t gemm(const GemmArgs &g, int splits, hipStream_t st) {
	const unsigned tiles = blocks(g.N, BN) * blocks(g.M, BM);
	hipLaunchKernelGGL((k_gemm<EPI, BM, BN, BM == 64 ? 128 : 64>), dim3((tiles + 7) / 8 * 8, splits), dim3(kThreads), 0, st, g);
	return hipGetLastError();
}

}  // namespace

// ------------------------------------------------------------------------------ host side

// Rows below which k_mlp_top1 runs: its workgroups of 64 rays fill the chip earlier. It against
// k_mlp_top1_many, in us: 65,536 rays 125 / 149, 262,144 rays 485 / 455, 1 Mi rays 1,930 / 1,780.
constexpr int kManyFrom = 262144;

const int kLayerIn[4] = {kMlpIn, kMlpHidden, kMlpHidden, kMlpHidden};
const int kLayerOut[4] = {kMlpHidden, kMlpHidden, kMlpHidden, kMlpOutPad};

hipError_t mlp_init(Mlp &m, uint64_t seed, hipStream_t st) {
#define PRT_TRY(x)                                                                                 \
	do {                                                                                           \
		hipError_t e_ = (x);                                                                       \
		if (e_ != hipSuccess) return e_;                                                           \
	} while (0)
	for (int l = 0; l < 4; ++l) {
		const size_t n = static_cast<size_t>(kLayerOut[l]) * kLayerIn[l];
		PRT_TRY(m.w[l].ensure(n * 4));
		PRT_TRY(m.b[l].ensure(kLayerOut[l] * 4));
		PRT_TRY(m.wt_bf[l].ensure(n * 2));
		PRT_TRY(m.wt_frag[l].ensure(n * 2));
		PRT_TRY(m.w_bf[l].ensure(n * 2));
		PRT_TRY(m.mw[l].ensure(n * 4));
		PRT_TRY(m.vw[l].ensure(n * 4));
		PRT_TRY(m.mb[l].ensure(kLayerOut[l] * 4));
		PRT_TRY(m.vb[l].ensure(kLayerOut[l] * 4));
		PRT_TRY(m.gw[l].ensure(n * 4));
		PRT_TRY(m.gb[l].ensure(kLayerOut[l] * 4));
		const int valid = l == 3 ? kMlpOut : kLayerOut[l];
		hipLaunchKernelGGL(k_init, dim3(blocks(n)), dim3(256), 0, st, m.w[l].as<float>(), n, kLayerIn[l], valid,
		                   seed * 31 + l, valid, kLayerIn[l]);
		hipLaunchKernelGGL(k_fill_f32, dim3(blocks(kLayerOut[l])), dim3(256), 0, st, m.b[l].as<float>(),
		                   static_cast<size_t>(kLayerOut[l]), 0.0f);
		if (l == 3) {  // padding logits never win and get no probability mass
			hipLaunchKernelGGL(k_fill_f32, dim3(1), dim3(256), 0, st, m.b[l].as<float>() + kMlpOut,
			                   static_cast<size_t>(kMlpOutPad - kMlpOut), -1e30f);
		}
		hipLaunchKernelGGL(k_fill_f32, dim3(blocks(n)), dim3(256), 0, st, m.mw[l].as<float>(), n, 0.0f);
		hipLaunchKernelGGL(k_fill_f32, dim3(blocks(n)), dim3(256), 0, st, m.vw[l].as<float>(), n, 0.0f);
		hipLaunchKernelGGL(k_fill_f32, dim3(blocks(kLayerOut[l])), dim3(256), 0, st, m.mb[l].as<float>(),
		                   static_cast<size_t>(kLayerOut[l]), 0.0f);
		hipLaunchKernelGGL(k_fill_f32, dim3(blocks(kLayerOut[l])), dim3(256), 0, st, m.vb[l].as<float>(),
		                   static_cast<size_t>(kLayerOut[l]), 0.0f);
		hipLaunchKernelGGL(k_to_bf16, dim3(blocks(n)), dim3(256), 0, st, m.w[l].as<float>(), n, m.wt_bf[l].as<uint16_t>(),
		                   m.w_bf[l].as<uint16_t>(), m.wt_frag[l].as<uint16_t>(), kLayerOut[l], kLayerIn[l]);
	}
	m.step = 0;
	m.ready = true;
	return hipGetLastError();
}

hipError_t mlp_refresh_bf16(Mlp &m, hipStream_t st) {
	for (int l = 0; l < 4; ++l) {
		const size_t n = static_cast<size_t>(kLayerOut[l]) * kLayerIn[l];
		hipLaunchKernelGGL(k_to_bf16, dim3(blocks(n)), dim3(256), 0, st, m.w[l].as<float>(), n, m.wt_bf[l].as<uint16_t>(),
		                   m.w_bf[l].as<uint16_t>(), m.wt_frag[l].as<uint16_t>(), kLayerOut[l], kLayerIn[l]);
	}
	return hipGetLastError();
}

static hipError_t ensure_act(Mlp &m, int rows) {
	PRT_TRY(m.x0.ensure(static_cast<size_t>(rows) * kMlpIn * 2));
	for (int l = 0; l < 3; ++l) PRT_TRY(m.h[l].ensure(static_cast<size_t>(rows) * kMlpHidden * 2));
	PRT_TRY(m.logits.ensure(static_cast<size_t>(rows) * kMlpOutPad * 4));
	PRT_TRY(m.dlog.ensure(static_cast<size_t>(rows) * kMlpOutPad * 2));
	PRT_TRY(m.dlog_t.ensure(static_cast<size_t>(rows) * kMlpOutPad * 2));
	for (int l = 0; l < 3; ++l) PRT_TRY(m.dh[l].ensure(static_cast<size_t>(rows) * kMlpHidden * 2));
	PRT_TRY(m.act_t.ensure(static_cast<size_t>(rows) * kMlpHidden * 2));
	PRT_TRY(m.dact_t.ensure(static_cast<size_t>(rows) * kMlpHidden * 2));
	PRT_TRY(m.split.ensure(kSplitFloats * 4));
	PRT_TRY(m.colsum.ensure(sizeof(float) * (kMlpOutPad + 3 * kMlpHidden) * static_cast<size_t>((rows + kTrRows - 1) / kTrRows)));
	PRT_TRY(m.loss_row.ensure(sizeof(float) * rows));
	PRT_TRY(m.loss.ensure(4));
	return hipSuccess;
}

static FusedArgs fused_args(const Mlp &m, const float *rays, uint64_t first, int rows) {
	FusedArgs f;
	f.rays = rays;
	f.first = first;
	f.rows = rows;
	f.lo = make_float4(m.scene_lo[0], m.scene_lo[1], m.scene_lo[2], 0.f);
	f.inv_ext = make_float4(m.scene_inv_ext[0], m.scene_inv_ext[1], m.scene_inv_ext[2], 0.f);
	for (int l = 0; l < 4; ++l) {
		f.w[l] = m.wt_bf[l].as<uint16_t>();
		f.b[l] = m.b[l].as<float>();
	}
	f.seeds = nullptr;
	return f;
}

hipError_t mlp_forward_logits(Mlp &m, const float *rays, uint64_t first, int rows, hipStream_t st) {
	PRT_TRY(ensure_act(m, rows));
	HiddenOut out;
	out.x0 = m.x0.as<uint16_t>();
	for (int l = 0; l < 3; ++l) out.h[l] = m.h[l].as<uint16_t>();
	hipLaunchKernelGGL(k_hidden, dim3(blocks(rows, kFRows)), dim3(256), 0, st, fused_args(m, rays, first, rows), out);
	GemmArgs g{};
	g.A = m.h[2].as<uint16_t>();
	g.B = m.wt_bf[3].as<uint16_t>();
	g.out = m.logits.ptr;
	g.bias = m.b[3].as<float>();
	g.M = rows;
	g.N = kMlpOutPad;
	g.K = kMlpHidden;
	g.lda = g.ldb = kMlpHidden;
	g.ldo = kMlpOutPad;
	g.k_split = g.K;
	return gemm<E_BIAS_F32, 128, 128>(g, 1, st);
}

hipError_t mlp_infer_top4(Mlp &m, const float *rays, uint64_t first, int rows, uint32_t *top4, hipStream_t st) {
	if (rows <= 0) return hipSuccess;
	FusedArgs f = fused_args(m, rays, first, rows);
	f.seeds = top4;
	hipLaunchKernelGGL(k_mlp_top4, dim3((rows + kFRows - 1) / kFRows), dim3(256), 0, st, f);
	return hipGetLastError();
}

hipError_t mlp_infer_top1(Mlp &m, const float *rays, uint64_t first, int rows, uint32_t *top1, hipStream_t st) {
	if (rows <= 0) return hipSuccess;
	FusedArgs f = fused_args(m, rays, first, rows);
	for (int l = 0; l < 4; ++l) f.w[l] = m.wt_frag[l].as<uint16_t>();
	f.seeds = top1;
	if (rows < kManyFrom) hipLaunchKernelGGL(k_mlp_top1, dim3(blocks(rows, kTop1Rows)), dim3(256), 0, st, f);
	else hipLaunchKernelGGL(k_mlp_top1_many, dim3(blocks(rows, kManyRows)), dim3(256), 0, st, f);
	return hipGetLastError();
}

// Backward of one batch whose logits are in m.logits: gradients land in m.gw / m.gb and, with lr > 0,
// one Adam step is taken after them.
hipError_t mlp_backward(Mlp &m, const uint32_t *labels, int rows, float lr, hipStream_t st) {
	PRT_TRY(ensure_act(m, rows));
	AdamArgs a{};
	if (lr > 0.0f) {
		++m.step;
		a.lr = lr;
		a.b1 = 0.9f;
		a.b2 = 0.999f;
		a.eps = 1e-8f;
		a.c1 = 1.0f / (1.0f - std::pow(a.b1, static_cast<float>(m.step)));
		a.c2 = 1.0f / (1.0f - std::pow(a.b2, static_cast<float>(m.step)));
	}
	hipLaunchKernelGGL(k_softmax_ce, dim3(rows), dim3(256), 0, st, m.logits.as<float>(), labels, rows, kMlpOutPad, kMlpOut,
	                   1.0f / static_cast<float>(rows), m.dlog.as<uint16_t>(), m.loss_row.as<float>());
	const uint16_t *dy = m.dlog.as<uint16_t>();
	int dy_cols = kMlpOutPad;
	const unsigned row_tiles = blocks(rows, kTrRows);
	float *split = m.split.as<float>(), *colsum = m.colsum.as<float>();
	unsigned n_blocks = 0;
	for (int l = 3; l >= 0; --l) {
		const int in = kLayerIn[l], out = kLayerOut[l];
		const uint16_t *x = l == 0 ? m.x0.as<uint16_t>() : m.h[l - 1].as<uint16_t>();
		uint16_t *dyt = (l == 3) ? m.dlog_t.as<uint16_t>() : m.dact_t.as<uint16_t>();
		// dy transposed, with its column sums over tiles of 128 rows (the bias gradient)
		hipLaunchKernelGGL(k_transpose<true>, dim3(out / kTrCols, row_tiles), dim3(256), 0, st, dy, rows, out, dy_cols, dyt, rows,
		                   colsum);
		hipLaunchKernelGGL(k_transpose<false>, dim3(in / kTrCols, row_tiles), dim3(256), 0, st, x, rows, in, in,
		                   m.act_t.as<uint16_t>(), rows, nullptr);
		// weight gradient gW^T[out][in] = dy^T[out][rows] * x^T[in][rows]^T (split over the batch)
		GemmArgs g{};
		g.A = dyt;
		g.B = m.act_t.as<uint16_t>();
		g.out = split;
		g.M = out;
		g.N = in;
		g.K = rows;
		g.lda = g.ldb = rows;
		g.ldo = in;
		g.k_split = ((rows / kSplits + kBK - 1) / kBK) * kBK;
		if (l == 3) PRT_TRY((gemm<E_F32, 128, 128>(g, kSplits, st)));
		else PRT_TRY((gemm<E_F32, 64, 64>(g, kSplits, st)));  // 96 or 128 workgroups instead of 32
		if (l > 0) {
			// data gradient dh[l-1] = (dy * W) masked by relu'(h[l-1]); 64 x 64 tiles: two workgroups per
			// CU at a batch of 8,192
			GemmArgs d{};
			d.A = dy;
			d.B = m.w_bf[l].as<uint16_t>();
			d.out = m.dh[l - 1].ptr;
			d.aux = m.h[l - 1].as<uint16_t>();
			d.M = rows;
			d.N = in;
			d.K = out;
			d.lda = dy_cols;
			d.ldb = out;
			d.ldo = in;
			d.k_split = d.K;
			PRT_TRY((gemm<E_MASK_BF16, 64, 64>(d, 1, st)));
		}
		a.w[l] = {m.w[l].as<float>(), m.gw[l].as<float>(), m.mw[l].as<float>(), m.vw[l].as<float>(), split, kSplits,
		          m.wt_bf[l].as<uint16_t>(), m.w_bf[l].as<uint16_t>(), m.wt_frag[l].as<uint16_t>(), out, in, n_blocks};
		n_blocks += static_cast<unsigned>(in / 64) * (out / 32);
		a.b[l] = {m.b[l].as<float>(), m.gb[l].as<float>(), m.mb[l].as<float>(), m.vb[l].as<float>(), colsum, static_cast<int>(row_tiles),
		          nullptr, nullptr, nullptr, out, l == 3 ? kMlpOut : out, n_blocks};  // the padding logits' bias stays
		n_blocks += blocks(out);
		split += kSplits * kLayerWeights[l];
		colsum += static_cast<size_t>(row_tiles) * out;
		dy = l > 0 ? m.dh[l - 1].as<uint16_t>() : nullptr;
		dy_cols = in;
	}
	a.loss_block = n_blocks++;
	a.loss_row = m.loss_row.as<float>();
	a.loss = m.loss.as<float>();
	a.n_loss = rows;
	hipLaunchKernelGGL(k_update, dim3(n_blocks), dim3(256), 0, st, a);
	return hipGetLastError();
#undef PRT_TRY
}

}  // namespace prt
