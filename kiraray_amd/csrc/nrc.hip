// nrc.hip - neural radiance cache on gfx950 matrix cores (krr_nrc.h).
//
// Network: x0 = enc(vertex) (64), z_l = W_l^T x_l, x_{l+1} = relu(z_l) for
// l = 0..4, y = W_5^T x_5 (3 outputs, no activation, no biases; the encoding
// carries two constant 1 inputs).  W_l is stored [in][out].
//
// MFMA formulation.  Each wave owns a tile of 32 samples and computes the
// transposed products Z^T = W^T X^T in 8-deep k-steps: the A operand is a
// 32x8 slice of W^T (LDS), the B operand an 8x32 slice of X^T held by the
// lanes (lane m + 32g holds features 8s + 4g + j, j < 4, of sample m for
// k-step s), and the 32x32 accumulator tile leaves feature 8(r/4) + 4g + r%4
// of sample m in register r of lane m + 32g - exactly the B-operand layout of
// the next layer, so activations never leave the registers between layers.
// Pairs of k-steps run as one v_mfma_f32_32x32x16_bf16.  Backward uses the
// same layout with A = W (dX^T = W dZ^T).  Weight gradients
// dW_l = X_l dZ_l^T are summed over the batch in the same launch, on operands
// transposed through LDS; the blocks' sums are reduced in a fixed order
// (deterministic), then Adam updates the FP32 master weights and rewrites both
// BF16 copies.
//
// Encoding (64 features, lane half g = 0/1 computes slots q = 4s + j of
// feature 8s + 4g + j):
//   half 0: q = 10c + 2f + t: sin (t = 0) / cos (t = 1) of 2^f pi pos_c,
//           c < 3, f < 5 (hardware sine/cosine of pi pos_c, doubled f
//           times); q = 30, 31: 1.
//   half 1: q 0..2 pos; 3..6 / 7..10 one-blob(4) of dir theta / phi;
//           11..14 / 15..18 of normal theta / phi; 19..22 of roughness;
//           23..25 diffuse; 26..28 specular; 29..31: 0.
//   one-blob(4) of x in [0,1]: exp(-0.5 (4 (x - (i + 0.5) / 4))^2), i < 4.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <memory>
#include <vector>

#include "detmath.h"
#include "errors.h"
#include "json.h"
#include "krr_nrc.h"
#include "nrc_dev.h"

namespace krr {
namespace nrc {

// ---------------------------------------------------------------- device

// Round to nearest even (inf stays inf, a nan becomes a quiet nan): the
// hardware conversion, v_cvt_pk_bf16_f32 on gfx950, two values per
// instruction where the compiler pairs them.
__device__ __forceinline__ uint16_t toBf16(float f) { return __builtin_bit_cast(uint16_t, (__bf16) f); }
__device__ __forceinline__ float fromBf16(uint16_t h) { return __uint_as_float((uint32_t) h << 16); }

// Two values with one conversion (left to itself the compiler converts them one
// by one and joins the halves).
typedef float float2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack2(float a, float b) { return __builtin_bit_cast(uint32_t, __builtin_convertvector((float2v){a, b}, bf16x2v)); }
__device__ __forceinline__ short4v pack4(float a, float b, float c, float d) {
	return __builtin_bit_cast(short4v, (uint64_t) pack2(c, d) << 32 | pack2(a, b));
}

// The encoding uses the hardware exp2 / sine / cosine (a learned input needs
// no bit-exact agreement with the CPU; the checker compares to 2e-5).
__device__ __forceinline__ float oneBlob(float x, int i) {
	const float d = 4.0f * (x - ((float) i + 0.5f) * 0.25f);
	return __builtin_amdgcn_exp2f(-0.72134752044448170368f * d * d); // exp(-d^2 / 2)
}

// Encoding slot q (0..31) of lane half g for vertex record v (16 floats).
__device__ float encodeSlot(const float *v, int g, int q) {
	if (g == 0) {
		if (q >= 30) return 1.0f;
		const int c = q / 10, f = (q % 10) / 2, t = q & 1;
		float sn = __builtin_amdgcn_sinf(0.5f * v[c]), cs = __builtin_amdgcn_cosf(0.5f * v[c]);
		for (int k = 0; k < f; k++) {
			const float s2 = 2.0f * sn * cs, c2 = (cs - sn) * (cs + sn);
			sn = s2;
			cs = c2;
		}
		return t ? cs : sn;
	}
	if (q < 3) return v[q];						  // pos
	if (q < 7) return oneBlob(v[3], q - 3);		  // dir theta
	if (q < 11) return oneBlob(v[4], q - 7);	  // dir phi
	if (q < 15) return oneBlob(v[5], q - 11);	  // normal theta
	if (q < 19) return oneBlob(v[6], q - 15);	  // normal phi
	if (q < 23) return oneBlob(v[7], q - 19);	  // roughness
	if (q < 29) return v[8 + (q - 23)];			  // diffuse, specular
	return 0.0f;
}

// B operands of layer 0 for sample record v: b[s] = features 8s + 4g + j
// (slots q = 4s + j of half g).
__device__ void encodeB(const float *v, int g, short4v b[8]) {
	float e[32];
	if (g == 0) {
		// sin / cos of pi x from the hardware (argument in revolutions: x / 2),
		// higher frequencies by the double-angle recurrence
#pragma unroll
		for (int c = 0; c < 3; c++) {
			float sn = __builtin_amdgcn_sinf(0.5f * v[c]), cs = __builtin_amdgcn_cosf(0.5f * v[c]);
#pragma unroll
			for (int f = 0; f < 5; f++) {
				e[10 * c + 2 * f]	  = sn;
				e[10 * c + 2 * f + 1] = cs;
				const float s2 = 2.0f * sn * cs, c2 = (cs - sn) * (cs + sn);
				sn = s2;
				cs = c2;
			}
		}
		e[30] = e[31] = 1.0f;
	} else {
#pragma unroll
		for (int q = 0; q < 32; q++) e[q] = encodeSlot(v, 1, q);
	}
#pragma unroll
	for (int s = 0; s < 8; s++) b[s] = pack4(e[4 * s], e[4 * s + 1], e[4 * s + 2], e[4 * s + 3]);
}

__device__ __forceinline__ float16v zero16() {
	float16v z;
#pragma unroll
	for (int i = 0; i < 16; i++) z[i] = 0.f;
	return z;
}

// Two consecutive 8-deep K-steps (4 bf16 per lane half each) in one gfx950
// v_mfma_f32_32x32x16_bf16: lane half g passes the A row elements (a0, a1)
// and the B column elements (b0, b1) in the same order, so the 16 products
// summed are those of the two 32x32x8 steps (a0, b0) and (a1, b1); only the
// FP32 order of the additions inside the instruction differs.  Half the
// instructions of the 32x32x8 form, each at the same rate.
typedef __bf16 bf16x8v __attribute__((ext_vector_type(8)));
__device__ __forceinline__ short8v join(short4v a, short4v b) { return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7); }
__device__ __forceinline__ float16v mfma2(short8v a, short4v b0, short4v b1, float16v c) {
	const short8v b = join(b0, b1);
	return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8v, a), __builtin_bit_cast(bf16x8v, b), c, 0, 0, 0);
}

// A lane's operand pair `pair` of a weight copy (in LDS or in memory).
__device__ __forceinline__ short8v weightPair(const uint16_t *w, int pair, int lane) {
	return *reinterpret_cast<const short8v *>(w + pair * 512 + lane * 8);
}

// ReLU of both row halves' accumulators, rounded to bf16 (B layout).
__device__ __forceinline__ void reluPack(const float16v &a0, const float16v &a1, short4v out[8]) {
#pragma unroll
	for (int s = 0; s < 4; s++) {
		out[s]	   = pack4(fmaxf(a0[4 * s], 0.f), fmaxf(a0[4 * s + 1], 0.f), fmaxf(a0[4 * s + 2], 0.f), fmaxf(a0[4 * s + 3], 0.f));
		out[4 + s] = pack4(fmaxf(a1[4 * s], 0.f), fmaxf(a1[4 * s + 1], 0.f), fmaxf(a1[4 * s + 2], 0.f), fmaxf(a1[4 * s + 3], 0.f));
	}
}

// One hidden layer, forward: out (B layout, relu, bf16) = W^T x.
__device__ __forceinline__ void hiddenForward(const uint16_t *wt, int lane, const short4v x[8], short4v out[8]) {
	float16v acc0 = zero16(), acc1 = zero16();
#pragma unroll
	for (int s = 0; s < 4; s++) {
		acc0 = mfma2(weightPair(wt, s, lane), x[2 * s], x[2 * s + 1], acc0);
		acc1 = mfma2(weightPair(wt, 4 + s, lane), x[2 * s], x[2 * s + 1], acc1);
	}
	reluPack(acc0, acc1, out);
}

// Output layer forward: y_c (c < 3) lands in acc[c] of lanes with g == 0.
__device__ __forceinline__ float16v outputForward(const uint16_t *wt5, int lane, const short4v x[8]) {
	float16v acc = zero16();
#pragma unroll
	for (int s = 0; s < 4; s++) acc = mfma2(weightPair(wt5, s, lane), x[2 * s], x[2 * s + 1], acc);
	return acc;
}

// Forward weights into LDS as they are.  Each thread issues up to twelve
// 16-byte loads before it stores them, so a block of 256 threads fetches all
// layers' weights (44 KB) in one round trip; one load per store would put a
// memory round trip between consecutive loads.
__device__ void loadWeights(uint16_t *lds, const uint16_t *wtAll) {
	constexpr int batch = 12, total = kFwdElems / 8;
	const uint4 *src = reinterpret_cast<const uint4 *>(wtAll);
	const int stride = (int) blockDim.x;
	for (int base = (int) threadIdx.x; base < total; base += batch * stride) {
		uint4 v[batch];
#pragma unroll
		for (int k = 0; k < batch; k++) v[k] = src[min(base + k * stride, total - 1)];
#pragma unroll
		for (int k = 0; k < batch; k++)
			if (base + k * stride < total) reinterpret_cast<uint4 *>(lds)[base + k * stride] = v[k];
	}
}

// ----------------------------------------------------------------- kernels

__global__ void __launch_bounds__(256) k_encode(const float *vertices, int64_t n, float *out) {
	const int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n * 64) return;
	const int64_t row = i / 64;
	const int k		  = (int) (i % 64);
	const int s = k / 8, g = (k / 4) & 1, j = k & 3;
	out[i] = encodeSlot(vertices + row * 16, g, 4 * s + j);
}

// Vertex record i as 16 floats, zeros past the end.
__device__ __forceinline__ void loadVertex(const float *vertices, int64_t i, int64_t n, float v[16]) {
	if (i < n) {
		const float4 *p = reinterpret_cast<const float4 *>(vertices + i * 16);
#pragma unroll
		for (int q = 0; q < 4; q++) {
			const float4 f = p[q];
			v[4 * q]	   = f.x;
			v[4 * q + 1]   = f.y;
			v[4 * q + 2]   = f.z;
			v[4 * q + 3]   = f.w;
		}
	} else {
#pragma unroll
		for (int q = 0; q < 16; q++) v[q] = 0.f;
	}
}

// Inference: each wave evaluates T tiles of 32 samples at a time.  Reading a
// layer's weights from LDS takes as long as the matrix cores take for one tile
// (44 KB at 128 bytes a cycle, 350 cycles each), so with two tiles per wave the
// reads halve; 118 registers leave 4 waves per SIMD, in two blocks of 8 waves
// that share a copy of the weights each and stay resident.  1 M samples 51
// against 58 us, 4 M 197 against 228 us on one card; on another 53 against 61
// (one tile, 5 waves: 57; two tiles with the next ones prefetched, 3 waves: 55;
// four tiles: 59).  A wave's own vector work (encoding, rounding) is the larger
// part now.
template <int T, int THREADS, int WAVES>
__global__ void __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(WAVES, 8))) k_infer(const uint16_t *wtAll, const float *vertices, int64_t n, float *radiance) {
	extern __shared__ uint16_t ldsW[];
	loadWeights(ldsW, wtAll);
	__syncthreads();
	const int lane = threadIdx.x & 63, g = lane >> 5, m = lane & 31;
	const int64_t tiles = (n + 32 * T - 1) / (32 * T), stride = (int64_t) gridDim.x * (THREADS / 64);
	int64_t t = (int64_t) blockIdx.x * (THREADS / 64) + (threadIdx.x >> 6);
	for (; t < tiles; t += stride) {
		float v[T][16];
		short4v x[T][8];
#pragma unroll
		for (int k = 0; k < T; k++) loadVertex(vertices, (t * T + k) * 32 + m, n, v[k]);
#pragma unroll
		for (int k = 0; k < T; k++) encodeB(v[k], g, x[k]);
		// not unrolled: an unrolled loop hoists every layer's weight loads
#pragma unroll 1
		for (int l = 0; l < kHidden; l++) {
			const uint16_t *wt = ldsW + l * 4096;
			float16v a0[T], a1[T];
#pragma unroll
			for (int k = 0; k < T; k++) a0[k] = a1[k] = zero16();
#pragma unroll
			for (int s = 0; s < 4; s++) {
				const short8v w0 = weightPair(wt, s, lane), w1 = weightPair(wt, 4 + s, lane);
#pragma unroll
				for (int k = 0; k < T; k++) {
					a0[k] = mfma2(w0, x[k][2 * s], x[k][2 * s + 1], a0[k]);
					a1[k] = mfma2(w1, x[k][2 * s], x[k][2 * s + 1], a1[k]);
				}
			}
#pragma unroll
			for (int k = 0; k < T; k++) reluPack(a0[k], a1[k], x[k]);
		}
#pragma unroll
		for (int k = 0; k < T; k++) {
			const float16v o = outputForward(ldsW + kHidden * 4096, lane, x[k]);
			const int64_t i	 = (t * T + k) * 32 + m;
			if (g == 0 && i < n) {
				radiance[3 * i]		= o[0];
				radiance[3 * i + 1] = o[1];
				radiance[3 * i + 2] = o[2];
			}
		}
	}
}

// Threads per k_infer_queue block: the block's waves share one LDS copy of
// the weights (44 KB), which limits a CU to 3 copies; blocks of 8 waves,
// compiled for 5 waves per SIMD (96 VGPRs, 20 B of spills), run 5 waves per SIMD
// where blocks of 4 ran 3.  On the 1080p field (0.36 M queries per launch):
// 27.8 us per launch against 32.4 us; 6 waves per SIMD (80 VGPRs, 84 B of
// spills) 33.6 us, 512 threads without a wave target (97 VGPRs, 4 waves)
// 29.4 us.
constexpr int kInferBlock = 512;

// Inference on a query queue whose length lives on the device; adds
// thp * max(y, 0) to L[pixel].  A wave's next tile of queries is loaded while
// it evaluates the current one, and the pixel's radiance is read as soon as
// the query names the pixel: the network in between hides both loads.  A
// launch answers one sample's queries, at most one per pixel, so no other
// lane writes that pixel's radiance meanwhile.
__device__ __forceinline__ void loadQuery(const float4 *queries, int stride, int i, int n, float v[16], float4 &pay) {
	pay = make_float4(0.f, 0.f, 0.f, __int_as_float(-1));
	if (i < n) {
		const float4 *p = queries + (int64_t) i * stride;
#pragma unroll
		for (int q = 0; q < 4; q++) {
			const float4 f = p[q];
			v[4 * q]	   = f.x;
			v[4 * q + 1]   = f.y;
			v[4 * q + 2]   = f.z;
			v[4 * q + 3]   = f.w;
		}
		pay = p[4];
	} else {
#pragma unroll
		for (int q = 0; q < 16; q++) v[q] = 0.f;
	}
}

__global__ void __launch_bounds__(kInferBlock) __attribute__((amdgpu_waves_per_eu(5, 8))) k_infer_queue(const uint16_t *wtAll, const float4 *queries, int stride, const int *countPtr, int capacity,
													 float4 *L) {
	extern __shared__ uint16_t ldsW[];
	loadWeights(ldsW, wtAll);
	__syncthreads();
	const int n	   = min(max(*countPtr, 0), capacity);
	const int lane = threadIdx.x & 63, g = lane >> 5, m = lane & 31;
	const int wavesPerBlock = blockDim.x >> 6;
	const int tiles			= (n + 31) / 32;
	const int tStride		= gridDim.x * wavesPerBlock;
	int t					= blockIdx.x * wavesPerBlock + (threadIdx.x >> 6);
	float v[16];
	float4 pay;
	loadQuery(queries, stride, t * 32 + m, n, v, pay);
	for (; t < tiles; t += tStride) {
		const int i		= t * 32 + m;
		const int pixel = __float_as_int(pay.w);
		const bool mine = g == 0 && i < n;
		const float4 thp = pay;
		float4 acc		 = make_float4(0.f, 0.f, 0.f, 0.f);
		if (mine) acc = L[pixel];
		short4v x[8], y[8];
		encodeB(v, g, x);
		loadQuery(queries, stride, (t + tStride) * 32 + m, n, v, pay); // the next tile's queries
		// not unrolled: an unrolled loop hoists every layer's weight loads
#pragma unroll 1
		for (int l = 0; l < kHidden; l++) {
			hiddenForward(ldsW + l * 4096, lane, x, y);
#pragma unroll
			for (int s = 0; s < 8; s++) x[s] = y[s];
		}
		const float16v o = outputForward(ldsW + kHidden * 4096, lane, x);
		if (mine) {
			acc.x += thp.x * fmaxf(o[0], 0.f);
			acc.y += thp.y * fmaxf(o[1], 0.f);
			acc.z += thp.z * fmaxf(o[2], 0.f);
			L[pixel] = acc;
		}
	}
}

// Training works on groups of 128 samples: a block of four waves, one tile of
// 32 samples each.
constexpr int kTrainBlock = 256;
constexpr int kGroup	  = 128;
constexpr int kTileElems  = 32 * 64; // a tile's layer input or output gradient in LDS, sample-major

// A mini-batch: `n` samples, or with a device count, the step-th of `steps`
// equal slices of the first min(*nDev, capTotal) samples (at most n).
struct Batch {
	int64_t n;
	const int *nDev;
	int64_t capTotal;
	int step, steps;
	__device__ int64_t range(int64_t &off) const {
		off = 0;
		if (!nDev) return n;
		const int64_t cnt = min((int64_t) max(*nDev, 0), capTotal);
		off				  = (int64_t) step * cnt / steps;
		return min((int64_t) (step + 1) * cnt / steps - off, n);
	}
};

// A tile in LDS: row m = sample, sixteen 8-byte chunks of 4 features.  Rows
// are 128 bytes, so chunks are permuted by the row: the 64 lanes that write
// one chunk pair of 32 rows, and the 64 lanes that read 8 rows of 8 chunks, each
// spread evenly over the banks.
__device__ __forceinline__ int tileChunk(int m, int c) { return m * 64 + 4 * (c ^ ((((m >> 1) & 1) << 3) | (m >> 2))); }

// The tile transposed, as an operand whose rows are features f0 + (lane & 31)
// and whose K-step s holds samples 8s + 4g + j: of each 16 lanes, lane i reads
// the chunk of 4 features i % 4 of row i / 4 and receives feature i of the 4 rows.
__device__ __forceinline__ int tileRead(int lane, int f0, int s) {
	return tileChunk(8 * s + 4 * (lane >> 5) + ((lane & 15) >> 2), f0 / 4 + 4 * ((lane >> 4) & 1) + (lane & 3));
}
typedef __attribute__((address_space(3))) short4v *LdsShort4;
__device__ __forceinline__ short4v tileT(const uint16_t *p) { return __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsShort4) p); }

// The A operands of a layer's two 32-row halves (`pairs` pairs of K-steps
// each), read ahead of the products that use them.
struct Rows {
	short8v w[8];
	__device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t copy, int first, int pairs, int lane) {
#pragma unroll
		for (int k = 0; k < 2 * pairs; k++)
			w[k] = __builtin_bit_cast(short8v, __builtin_amdgcn_raw_buffer_load_b128(copy, lane * 16, (first + k * 512) * (int) sizeof(uint16_t), 0));
	}
	__device__ __forceinline__ void multiply(const short4v x[8], int pairs, float16v &a0, float16v &a1) const {
		a0 = zero16();
		a1 = zero16();
#pragma unroll
		for (int s = 0; s < pairs; s++) {
			a0 = mfma2(w[s], x[2 * s], x[2 * s + 1], a0);
			a1 = mfma2(w[pairs + s], x[2 * s], x[2 * s + 1], a1);
		}
	}
};

// The transposed X and dZ operands of one tile.
struct TileRead {
	short4v x[4], z[4];
	__device__ __forceinline__ void load(const uint16_t *const getX[4], const uint16_t *const getZ[4], int offset) {
#pragma unroll
		for (int s = 0; s < 4; s++) {
			x[s] = tileT(getX[s] + offset);
			z[s] = tileT(getZ[s] + offset);
		}
	}
	__device__ __forceinline__ void multiply(float16v &acc) const {
#pragma unroll
		for (int s = 0; s < 4; s += 2) acc = mfma2(join(x[s], x[s + 1]), z[s], z[s + 1], acc);
	}
};

// (a, b, c, d) where x > 0, else 0, as the next B operand's four features; x is
// a ReLU's output (zero of either sign, or positive), so a 16-bit half of it
// is zero but for the sign exactly where adding 0x7fff leaves the top bit clear.
__device__ __forceinline__ uint32_t positiveMask(uint32_t x) {
	const uint32_t top = ((x & 0x7fff7fffu) + 0x7fff7fffu) & 0x80008000u;
	return (top - (top >> 15)) | top;
}
__device__ __forceinline__ short4v maskedPack(const short4v x, float a, float b, float c, float d) {
	const uint64_t bits = __builtin_bit_cast(uint64_t, x);
	const uint32_t lo = pack2(a, b) & positiveMask((uint32_t) bits), hi = pack2(c, d) & positiveMask((uint32_t) (bits >> 32));
	return __builtin_bit_cast(short4v, (uint64_t) hi << 32 | lo);
}

// A lane's LDS offset the compiler takes as it is: the offsets of layers and
// tiles then stay immediates of the accesses (below 64 KB from this base),
// where folding the base in would take a register for each of them.
__device__ __forceinline__ int laneOffset(int elems) {
	asm("" : "+v"(elems));
	return elems;
}

// Forward, backward and weight gradients of one mini-batch; block b takes the
// groups b, b + gridDim.x, ... and writes its sum of every weight's gradient
// to partial[layer][b] (read by k_reduce; blocks without a group write
// nothing).  Samples i >= n contribute nothing.
//
// Bound by latency: a mini-batch of 16384 samples is half a block per CU, one
// wave per SIMD, a chain of 12 products and 6 barriers with vector work in
// between (about 720 cycles per layer forward and 1900 backward, of which the
// matrix cores are busy 512 and 768).  So every layer's input stays in
// registers, a layer's weight gradient is taken while its X and dZ are here
// (their transposed operands come from LDS by the transposing read), nothing
// but the partial sums goes to memory, and operands are read ahead of the
// products that use them.  16384 samples 16.3 us and k_reduce 6.1 us, where
// X^T and dZ^T stored for a split-K product in a launch of its own took
// 23 + 18 + 7 us; four training steps with weights set and read back 192
// against 350 us.  Weights through LDS: 18 us; without the reads ahead 22 us.
__global__ void __launch_bounds__(kTrainBlock) __attribute__((amdgpu_waves_per_eu(1, 1)))
k_train(const uint16_t *wtAll, const uint16_t *wAll, const float *vertices, const float *targets, Batch batch, float lossEps, float *partialAll,
		float *tileLoss, int *adamStep) {
	// a training step (not a bare gradient) counts Adam's step here: the
	// kernel after this one in the stream reads the new count
	if (adamStep && blockIdx.x == 0 && threadIdx.x == 0) *adamStep += 1;
	int64_t off;
	const int64_t n = batch.range(off), groups = (n + kGroup - 1) / kGroup;
	if (blockIdx.x >= groups) return;
	vertices += off * 16;
	targets += off * 3;
	__shared__ __attribute__((aligned(16))) uint16_t lds[2 * 8 * kTileElems];
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 5, m = lane & 31;
	const int kt = 32 * (wave >> 1), nt = 32 * (wave & 1); // this wave's 32x32 tile of each weight gradient
	const float invCount = 1.0f / (3.0f * (float) n);

	float v[16], tg[3];
	auto fetch = [&](int64_t group) {
		const int64_t i = group * kGroup + 32 * wave + m;
		loadVertex(vertices, i, n, v);
#pragma unroll
		for (int c = 0; c < 3; c++) tg[c] = g == 0 && i < n ? targets[3 * i + c] : 0.f;
	};
	fetch(blockIdx.x);
	// A layer's weights come straight from memory (the copies are in operand
	// order: each read is one kilobyte, and the block's waves share the lines)
	// two layers ahead of the products; LDS, which the transposition keeps busy,
	// would have to carry them twice more.
	// (Buffer loads: one register of address for all of them.)
	const __amdgpu_buffer_rsrc_t fwd = __builtin_amdgcn_make_buffer_rsrc((void *) wtAll, (short) 0, kFwdElems * (int) sizeof(uint16_t), 0x00020000);
	const __amdgpu_buffer_rsrc_t bwd = __builtin_amdgcn_make_buffer_rsrc((void *) wAll, (short) 0, kBwdElems * (int) sizeof(uint16_t), 0x00020000);
	Rows w[3];
	w[0].load(fwd, 0, 4, lane);
	w[1].load(fwd, 4096, 4, lane);

	// this lane's chunks of its wave's tile, its reads of the transposed tiles
	constexpr int buffer = 8 * kTileElems; // four X tiles, then four dZ tiles
	uint16_t *put[8];
	const uint16_t *getX[4], *getZ[4];
#pragma unroll
	for (int s = 0; s < 8; s++) put[s] = lds + laneOffset(wave * kTileElems + tileChunk(m, 2 * s + g));
#pragma unroll
	for (int s = 0; s < 4; s++) {
		getX[s] = lds + laneOffset(tileRead(lane, kt, s));
		getZ[s] = lds + laneOffset(4 * kTileElems + tileRead(lane, nt, s));
	}

	float16v dW[kHidden + 1];
#pragma unroll
	for (int l = 0; l <= kHidden; l++) dW[l] = zero16();
	for (int64_t group = blockIdx.x; group < groups; group += gridDim.x) {
		const int64_t i	 = group * kGroup + 32 * wave + m;
		const bool valid = i < n;
		short4v x[kHidden + 1][8];
		encodeB(v, g, x[0]);
		// (the barriers keep the scheduler from moving reads back to their use)
		float16v a0, a1;
#pragma unroll
		for (int l = 0; l < kHidden; l++) {
			if (l + 2 < kHidden) w[(l + 2) % 3].load(fwd, (l + 2) * 4096, 4, lane);
			if (l + 2 == kHidden) w[(l + 2) % 3].load(fwd, (l + 2) * 4096, 2, lane); // four pairs of one half
			if (l + 2 == kHidden + 1) w[(l + 2) % 3].load(bwd, kHidden * 4096, 2, lane);
			__builtin_amdgcn_sched_barrier(0);
			w[l % 3].multiply(x[l], 4, a0, a1);
			reluPack(a0, a1, x[l + 1]);
			__builtin_amdgcn_sched_barrier(0);
		}
		// from here layer l's backward weights are in w[(2 kHidden + 1 - l) % 3]
		w[(kHidden + 2) % 3].load(bwd, (kHidden - 1) * 4096, 4, lane);
		__builtin_amdgcn_sched_barrier(0);
		// output c < 3 lands in o[c] of lanes with g == 0
		float16v o = zero16();
#pragma unroll
		for (int s = 0; s < 4; s++) o = mfma2(w[kHidden % 3].w[s], x[kHidden][2 * s], x[kHidden][2 * s + 1], o);
		// relative L2 loss and its gradient (lanes g == 0 hold the 3 outputs)
		float d[3] = {0.f, 0.f, 0.f};
		float lsum = 0.f;
		if (g == 0 && valid) {
#pragma unroll
			for (int c = 0; c < 3; c++) {
				const float yv = o[c], r = yv - tg[c];
				const float den = yv * yv + lossEps;
				lsum += r * r / den;
				d[c] = 2.0f * r / den * invCount;
			}
		}
		if (group + gridDim.x < groups) fetch(group + gridDim.x);
		// dZ of the output layer as a B operand: outputs 8s + 4g + j, only the
		// first 3 nonzero, of 32 padded ones
		short4v dz[8];
#pragma unroll
		for (int s = 0; s < 4; s++) dz[s] = pack4(0.f, 0.f, 0.f, 0.f);
		if (g == 0) dz[0] = pack4(d[0], d[1], d[2], 0.f);
#pragma unroll
		for (int l = kHidden; l >= 0; l--) {
			// the other buffer was last read before the barrier of layer l + 1
			const int buf = (l & 1) * buffer;
#pragma unroll
			for (int s = 0; s < 8; s++) {
				*reinterpret_cast<short4v *>(put[s] + buf) = x[l][s];
				if (s < 4 || l < kHidden) *reinterpret_cast<short4v *>(put[s] + buf + 4 * kTileElems) = dz[s];
			}
			__syncthreads();
			// dX_l^T = W_l dZ_l^T, and dW_l = X_l^T dZ_l over the block's 128 samples
			// (a 32x32 tile per wave; of the output layer only 3 columns are kept)
			TileRead t[4];
			t[0].load(getX, getZ, buf);
			t[1].load(getX, getZ, buf + kTileElems);
			__builtin_amdgcn_sched_barrier(0);
			if (l > 0) w[(2 * kHidden + 1 - l) % 3].multiply(dz, l == kHidden ? 2 : 4, a0, a1);
			t[2].load(getX, getZ, buf + 2 * kTileElems);
			t[3].load(getX, getZ, buf + 3 * kTileElems);
			__builtin_amdgcn_sched_barrier(0);
			t[0].multiply(dW[l]);
			t[1].multiply(dW[l]);
			if (l > 2) w[(2 * kHidden + 3 - l) % 3].load(bwd, (l - 2) * 4096, 4, lane);
			if (l < 2) w[1 - l].load(fwd, (1 - l) * 4096, 4, lane); // the next group's first layers
			__builtin_amdgcn_sched_barrier(0);
			t[2].multiply(dW[l]);
			t[3].multiply(dW[l]);
			if (l == 0) { // the wave's sum of the loss, here where nothing waits for it
				for (int k = 32; k > 0; k >>= 1) lsum += __shfl_xor(lsum, k);
				if (lane == 0) tileLoss[group * (kGroup / 32) + wave] = lsum * invCount;
			}
			// masked by x_l > 0, the next dZ
			if (l > 0) {
#pragma unroll
				for (int s = 0; s < 4; s++) {
					dz[s]	  = maskedPack(x[l][s], a0[4 * s], a0[4 * s + 1], a0[4 * s + 2], a0[4 * s + 3]);
					dz[4 + s] = maskedPack(x[l][4 + s], a1[4 * s], a1[4 * s + 1], a1[4 * s + 2], a1[4 * s + 3]);
				}
			}
			__builtin_amdgcn_sched_barrier(0);
		}
	}
	// D[i = k][j = n]: lane holds column n = nt + m, rows k = kt + 8(r/4) + 4g + r%4
#pragma unroll
	for (int l = 0; l <= kHidden; l++) {
		const int nOut = l < kHidden ? 64 : 3;
		float *dst	   = partialAll + ((int64_t) l * gridDim.x) * 4096 + (int64_t) blockIdx.x * 64 * nOut;
		if (nt + m < nOut)
#pragma unroll
			for (int r = 0; r < 16; r++) dst[(kt + 8 * (r / 4) + 4 * g + (r % 4)) * nOut + nt + m] = dW[l][r];
	}
}

// Deterministic loss total over tiles (one block of 256 threads).
__device__ void reduceLoss(const float *tileLoss, int64_t nTiles, float *out) {
	__shared__ float part[256];
	float s = 0.f;
	for (int64_t t = threadIdx.x; t < nTiles; t += blockDim.x) s += tileLoss[t];
	part[threadIdx.x] = s;
	__syncthreads();
	for (int w = blockDim.x / 2; w > 0; w >>= 1) {
		if ((int) threadIdx.x < w) part[threadIdx.x] += part[threadIdx.x + w];
		__syncthreads();
	}
	if (threadIdx.x == 0) *out = part[0];
}

// Rewrites both bf16 copies from the fp32 master weights.
__device__ void writeCopies(const float *w, uint16_t *wt, uint16_t *wb, int p) {
	// p indexes the master array: layer l < 5 at 4096 l + 64 k + n; layer 5 at 20480 + 3 k + n.
	const int l = min(p / 4096, kHidden), q = p - l * 4096;
	const int k = l < kHidden ? q / 64 : q / 3, n = l < kHidden ? q % 64 : q % 3;
	const uint16_t b = toBf16(w[p]);
	wt[l * 4096 + operandIndex(n, k, 64)]					   = b;
	wb[l * 4096 + operandIndex(k, n, l < kHidden ? 64 : 32)] = b;
}

// New master weights: both copies, no moments, no steps.
__global__ void k_set_weights(const float *w, float *mo, float *ve, uint16_t *wt, uint16_t *wb, int *step) {
	const int p = blockIdx.x * blockDim.x + threadIdx.x;
	if (p == 0) *step = 0;
	if (p >= KRR_NRC_PARAMS) return;
	mo[p] = ve[p] = 0.f;
	writeCopies(w, wt, wb, p);
}

// Adam (Kingma & Ba 2015) with bias corrections c1 = 1 - beta1^t, c2 = 1 - beta2^t.
// Adam's step count lives in device memory, so that training steps recorded
// in a graph count up on every replay.
struct AdamState {
	float w, m, v, c1, c2;
};
__device__ __forceinline__ void adamUpdate(float *w, float *mo, float *ve, const AdamState &a, float gr, float lr, float b1, float b2, float eps,
										   uint16_t *wt, uint16_t *wb, int p) {
	const float m = b1 * a.m + (1.f - b1) * gr;
	const float v = b2 * a.v + (1.f - b2) * gr * gr;
	mo[p]		  = m;
	ve[p]		  = v;
	w[p]		  = a.w - lr * (m / a.c1) / (sqrtf(v / a.c2) + eps);
	writeCopies(w, wt, wb, p);
}

// The tail of a gradient or training step in one launch: per weight the
// fixed-order sum over the blocks of k_train that had samples, stored to `grad`
// or, with Adam, applied (the step count was raised by k_train) and copied to
// bf16; the last block also totals the loss.
//
// A block of 256 threads takes 32 weights: thread (group q, weight j) sums
// its eighth of the partials in order, and the eight group sums are added in
// group order (a fixed order: deterministic).  One thread per weight would
// leave most of the chip idle on a few hundred latency-bound sequential loads;
// with sixteen partials and Adam's state in flight at once 6.1 us for 128
// partials, 8.7 us with the loads as the compiler orders them.
constexpr int kReduceWeights = 32, kReduceGroups = 8;
constexpr int kReduceBatch = 16; // partials in flight per thread
struct Adam {
	float *w, *m, *v;
	uint16_t *wt, *wb;
	const int *step;
	float lr, b1, b2, eps;
};
template <bool ADAM>
__global__ void __launch_bounds__(256) k_reduce(const float *partialAll, int blocks, Batch batch, float *grad, Adam adam, const float *tileLoss,
												float *loss) {
	__shared__ float part[kReduceGroups][kReduceWeights];
	int64_t off;
	const int64_t groups = (batch.range(off) + kGroup - 1) / kGroup;
	const int chunks	 = (int) min((int64_t) blocks, groups);
	const int j = threadIdx.x % kReduceWeights, q = threadIdx.x / kReduceWeights;
	const int p = blockIdx.x * kReduceWeights + j;
	float s		= 0.f;
	AdamState a;
	if (ADAM && q == 0 && p < KRR_NRC_PARAMS) { // on their way while the partials are
		a.w	 = adam.w[p];
		a.m	 = adam.m[p];
		a.v	 = adam.v[p];
		a.c1 = 1.f - powf(adam.b1, (float) *adam.step); // bias corrections
		a.c2 = 1.f - powf(adam.b2, (float) *adam.step);
	}
	if (p < KRR_NRC_PARAMS) {
		const int layer	 = min(p / 4096, kHidden);
		const int count	 = layer < kHidden ? 4096 : 64 * 3;
		const float *src = partialAll + (int64_t) layer * blocks * 4096 + (p - layer * 4096);
		const int c0 = q * chunks / kReduceGroups, c1 = (q + 1) * chunks / kReduceGroups;
		for (int c = c0; c < c1; c += kReduceBatch) {
			float r[kReduceBatch];
#pragma unroll
			for (int k = 0; k < kReduceBatch; k++) r[k] = c + k < c1 ? src[(int64_t) (c + k) * count] : 0.f;
#pragma unroll
			for (int k = 0; k < kReduceBatch; k++) s += r[k];
		}
	}
	part[q][j] = s;
	__syncthreads();
	if (q == 0 && p < KRR_NRC_PARAMS) {
		float gr = part[0][j];
		for (int k = 1; k < kReduceGroups; k++) gr += part[k][j];
		if (ADAM)
			adamUpdate(adam.w, adam.m, adam.v, a, gr, adam.lr, adam.b1, adam.b2, adam.eps, adam.wt, adam.wb, p);
		else
			grad[p] = gr;
	}
	if (blockIdx.x == gridDim.x - 1) reduceLoss(tileLoss, groups * (kGroup / 32), loss);
}

} // namespace nrc
} // namespace krr

// ------------------------------------------------------------------- host

using namespace krr::nrc;

namespace {

struct Buf {
	void *p	  = nullptr;
	size_t sz = 0;
	~Buf() {
		if (p) (void) hipFree(p);
	}
	hipError_t alloc(size_t bytes) {
		if (p) (void) hipFree(p);
		p  = nullptr;
		sz = 0;
		hipError_t e = hipMalloc(&p, bytes ? bytes : 16);
		if (e == hipSuccess) sz = bytes;
		return e;
	}
	template <class T> T *as() const { return reinterpret_cast<T *>(p); }
};

// A float that kernels write into host memory: it is read after the stream's
// synchronisation without a copy in between.
struct HostFloat {
	float *p = nullptr, *dev = nullptr;
	~HostFloat() {
		if (p) (void) hipHostFree(p);
	}
	hipError_t alloc() {
		if (hipError_t e = hipHostMalloc((void **) &p, sizeof(float), hipHostMallocMapped)) return e;
		*p = 0.f;
		return hipHostGetDevicePointer((void **) &dev, p, 0);
	}
	float read() const { return *(const volatile float *) p; }
};

#define NRC_HIP(expr)                                                                                                  \
	do {                                                                                                               \
		hipError_t e_ = (expr);                                                                                        \
		if (e_ != hipSuccess) return krr::fail(KRR_ERR_HIP, "%s: %s", #expr, hipGetErrorString(e_));                  \
	} while (0)

constexpr int64_t kInferSmall = 1 << 17;
} // namespace

struct krr_nrc {
	float lr = 1e-3f, beta1 = 0.9f, beta2 = 0.99f, eps = 1e-8f, lossEps = 0.01f;
	uint64_t seed	= 1;
	int64_t maxBatch = 65536;
	int cus			 = 256;
	int inferBlocks	 = 1024;  // k_infer_queue blocks resident at once on the device (each loads the weights once)
	Buf w, m, v, wt, wb, partial, tileLoss, step;
	HostFloat loss;
};

namespace {

int uploadWeights(krr_nrc *h, const std::vector<float> &host) {
	NRC_HIP(hipMemcpy(h->w.p, host.data(), sizeof(float) * KRR_NRC_PARAMS, hipMemcpyHostToDevice));
	hipLaunchKernelGGL(k_set_weights, dim3((KRR_NRC_PARAMS + 255) / 256), dim3(256), 0, 0, h->w.as<float>(), h->m.as<float>(), h->v.as<float>(),
					   h->wt.as<uint16_t>(), h->wb.as<uint16_t>(), h->step.as<int>());
	NRC_HIP(hipGetLastError());
	NRC_HIP(hipDeviceSynchronize());
	return KRR_OK;
}

// Seeded Xavier-uniform initial weights (PCG32 stream of the seed).
std::vector<float> initialWeights(uint64_t seed) {
	std::vector<float> w(KRR_NRC_PARAMS);
	uint64_t state = 0, inc = (seed << 1u) | 1u;
	auto next = [&]() {
		uint64_t old = state;
		state		 = old * 6364136223846793005ULL + inc;
		uint32_t xs	 = (uint32_t) (((old >> 18u) ^ old) >> 27u);
		uint32_t rot = (uint32_t) (old >> 59u);
		return (xs >> rot) | (xs << ((-rot) & 31));
	};
	next();
	state += 0x853c49e6748fea9bULL;
	next();
	for (int p = 0; p < KRR_NRC_PARAMS; p++) {
		const int fanOut = p < kHidden * 4096 ? 64 : 3;
		const float a	 = std::sqrt(6.0f / (64.0f + (float) fanOut));
		const float u	 = (float) (next() >> 8) * (1.0f / 16777216.0f);
		w[p]			 = (2.0f * u - 1.0f) * a;
	}
	return w;
}

bool validN(int64_t n) { return n >= 0 && n <= ((int64_t) 1 << 31); }

// Gradient of one batch, stored to `grad`, or without `grad` the Adam step.
// One block per CU at most: each holds a CU's LDS and its share of the
// batch's groups, and leaves one partial sum however large the batch is.
int gradientImpl(krr_nrc *h, const krr_nrc_vertex *vert, const float *targets, int64_t n, hipStream_t st, float *grad, const int *nDev = nullptr,
				 int64_t capTotal = 0, int step = 0, int steps = 1) {
	const int blocks = (int) std::min<int64_t>(h->cus, (n + kGroup - 1) / kGroup);
	const Batch batch{n, nDev, capTotal, step, steps};
	hipLaunchKernelGGL(k_train, dim3(blocks), dim3(kTrainBlock), 0, st, h->wt.as<uint16_t>(), h->wb.as<uint16_t>(), (const float *) vert,
					   targets, batch, h->lossEps, h->partial.as<float>(), h->tileLoss.as<float>(), grad ? nullptr : h->step.as<int>());
	NRC_HIP(hipGetLastError());
	const Adam adam{h->w.as<float>(), h->m.as<float>(), h->v.as<float>(), h->wt.as<uint16_t>(), h->wb.as<uint16_t>(), h->step.as<int>(), h->lr, h->beta1, h->beta2, h->eps};
	hipLaunchKernelGGL(grad ? k_reduce<false> : k_reduce<true>, dim3((KRR_NRC_PARAMS + kReduceWeights - 1) / kReduceWeights),
					   dim3(kReduceWeights * kReduceGroups), 0, st, h->partial.as<float>(), blocks, batch, grad, adam, h->tileLoss.as<float>(),
					   h->loss.dev);
	NRC_HIP(hipGetLastError());
	return KRR_OK;
}

} // namespace

extern "C" {

int krr_nrc_create(const char *json, krr_nrc **out) {
	krr::clearError();
	if (!out) return krr::fail(KRR_ERR_INVALID_ARG, "krr_nrc_create: null out");
	*out   = nullptr;
	auto h = std::make_unique<krr_nrc>();
	if (json && *json) {
		try {
			krr::Json j = krr::Json::parse(json);
			if (!j.isObject()) return krr::fail(KRR_ERR_BAD_CONFIG, "nrc config must be a JSON object");
			h->lr		= (float) j.value("lr", 1e-3);
			h->beta1	= (float) j.value("beta1", 0.9);
			h->beta2	= (float) j.value("beta2", 0.99);
			h->eps		= (float) j.value("eps", 1e-8);
			h->lossEps	= (float) j.value("loss_eps", 0.01);
			h->seed		= (uint64_t) j.value("seed", 1.0);
			h->maxBatch = (int64_t) j.value("max_batch", 65536.0);
		} catch (const std::exception &e) {
			return krr::fail(KRR_ERR_BAD_CONFIG, "nrc config: %s", e.what());
		}
	}
	if (!(h->lr > 0) || !(h->beta1 >= 0 && h->beta1 < 1) || !(h->beta2 >= 0 && h->beta2 < 1) || !(h->eps > 0) || !(h->lossEps > 0))
		return krr::fail(KRR_ERR_BAD_CONFIG, "nrc config: lr, eps and loss_eps must be > 0 and betas in [0, 1)");
	if (h->maxBatch < 32 || h->maxBatch > (1 << 24)) return krr::fail(KRR_ERR_BAD_CONFIG, "nrc config: max_batch must be in [32, 2^24]");
	int nDev = 0;
	if (hipGetDeviceCount(&nDev) != hipSuccess || nDev < 1) return krr::fail(KRR_ERR_NO_DEVICE, "krr_nrc_create: no HIP device");
	NRC_HIP(h->w.alloc(sizeof(float) * KRR_NRC_PARAMS));
	NRC_HIP(h->m.alloc(sizeof(float) * KRR_NRC_PARAMS));
	NRC_HIP(h->v.alloc(sizeof(float) * KRR_NRC_PARAMS));
	{
		int dev = 0;
		NRC_HIP(hipGetDevice(&dev));
		int cus = 0, perCu = 0;
		NRC_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
		NRC_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCu, k_infer_queue, kInferBlock, kFwdElems * sizeof(uint16_t)));
		h->cus		   = std::max(cus, 1);
		h->inferBlocks = std::max(1, cus * std::max(perCu, 1));
	}
	NRC_HIP(h->wt.alloc(sizeof(uint16_t) * kFwdElems));
	NRC_HIP(h->wb.alloc(sizeof(uint16_t) * kBwdElems));
	const int64_t groups = (h->maxBatch + kGroup - 1) / kGroup;
	NRC_HIP(h->partial.alloc(sizeof(float) * 4096 * (kHidden + 1) * std::min<int64_t>(groups, h->cus)));
	NRC_HIP(h->tileLoss.alloc(sizeof(float) * groups * (kGroup / 32)));
	NRC_HIP(h->loss.alloc());
	NRC_HIP(h->step.alloc(sizeof(int)));
	// the padded rows and columns of the bf16 copies are never written
	NRC_HIP(hipMemset(h->wt.p, 0, h->wt.sz));
	NRC_HIP(hipMemset(h->wb.p, 0, h->wb.sz));
	if (int rc = uploadWeights(h.get(), initialWeights(h->seed))) return rc;
	*out = h.release();
	return KRR_OK;
}

int krr_nrc_destroy(krr_nrc *nrc) {
	delete nrc;
	return KRR_OK;
}

int krr_nrc_get_weights(const krr_nrc *nrc, float *host_out) {
	krr::clearError();
	if (!nrc || !host_out) return krr::fail(KRR_ERR_INVALID_ARG, "krr_nrc_get_weights: null argument");
	NRC_HIP(hipDeviceSynchronize());
	NRC_HIP(hipMemcpy(host_out, nrc->w.p, sizeof(float) * KRR_NRC_PARAMS, hipMemcpyDeviceToHost));
	return KRR_OK;
}

int krr_nrc_set_weights(krr_nrc *nrc, const float *host_in) {
	krr::clearError();
	if (!nrc || !host_in) return krr::fail(KRR_ERR_INVALID_ARG, "krr_nrc_set_weights: null argument");
	std::vector<float> w(host_in, host_in + KRR_NRC_PARAMS);
	for (float x : w)
		if (!std::isfinite(x)) return krr::fail(KRR_ERR_INVALID_ARG, "krr_nrc_set_weights: non-finite weight");
	return uploadWeights(nrc, w);
}

int krr_nrc_encode(const krr_nrc *nrc, const krr_nrc_vertex *vertices_dev, int64_t n, float *encoded_dev, void *hip_stream) {
	krr::clearError();
	if (!nrc || !validN(n) || (n > 0 && (!vertices_dev || !encoded_dev))) return krr::fail(KRR_ERR_INVALID_ARG, "krr_nrc_encode: bad argument");
	if (n == 0) return KRR_OK;
	const int64_t total = n * 64;
	hipLaunchKernelGGL(k_encode, dim3((unsigned) ((total + 255) / 256)), dim3(256), 0, (hipStream_t) hip_stream, (const float *) vertices_dev, n,
					   encoded_dev);
	NRC_HIP(hipGetLastError());
	return KRR_OK;
}

int krr_nrc_infer(krr_nrc *nrc, const krr_nrc_vertex *vertices_dev, int64_t n, float *radiance_dev, void *hip_stream) {
	krr::clearError();
	if (!nrc || !validN(n) || (n > 0 && (!vertices_dev || !radiance_dev))) return krr::fail(KRR_ERR_INVALID_ARG, "krr_nrc_infer: bad argument");
	if (n == 0) return KRR_OK;
	// up to kInferSmall samples, one tile per wave in small blocks: the chip is
	// not full and the launch is most of the time (60 K samples 6.8 us)
	const bool small  = n <= kInferSmall;
	const int threads = small ? 256 : 512, perBlock = 32 * (small ? 1 : 2) * (threads / 64);
	const int blocks  = (int) std::min<int64_t>(small ? 2048 : 2 * nrc->cus, (n + perBlock - 1) / perBlock);
	hipLaunchKernelGGL((small ? k_infer<1, 256, 3> : k_infer<2, 512, 4>), dim3(blocks), dim3(threads), kFwdElems * (int) sizeof(uint16_t), (hipStream_t) hip_stream,
					   nrc->wt.as<uint16_t>(), (const float *) vertices_dev, n, radiance_dev);
	NRC_HIP(hipGetLastError());
	return KRR_OK;
}

int krr_nrc_gradient(krr_nrc *nrc, const krr_nrc_vertex *vertices_dev, const float *targets_dev, int64_t n, float *grad_dev,
					 float *loss_out, void *hip_stream) {
	krr::clearError();
	if (!nrc || n < 1 || !vertices_dev || !targets_dev || !grad_dev) return krr::fail(KRR_ERR_INVALID_ARG, "krr_nrc_gradient: bad argument");
	if (n > nrc->maxBatch) return krr::fail(KRR_ERR_CAPACITY, "krr_nrc_gradient: batch %lld exceeds max_batch %lld", (long long) n, (long long) nrc->maxBatch);
	hipStream_t st = (hipStream_t) hip_stream;
	if (int rc = gradientImpl(nrc, vertices_dev, targets_dev, n, st, grad_dev)) return rc;
	if (loss_out) {
		NRC_HIP(hipStreamSynchronize(st));
		*loss_out = nrc->loss.read();
	}
	return KRR_OK;
}

} // extern "C"

int nrcInferAccumulate(krr_nrc *nrc, const float4 *queries, int strideF4, const int *count, int capacity, float4 *L, hipStream_t st) {
	if (capacity <= 0) return KRR_OK;
	// one resident wave of blocks: each block loads the weights into LDS once
	// and then takes query tiles until the queue is done
	const int tilesPerPass = kInferBlock / 64; // one 32-query tile per wave
	const int blocks	   = std::max(1, std::min(nrc->inferBlocks, (capacity + 32 * tilesPerPass - 1) / (32 * tilesPerPass)));
	hipLaunchKernelGGL(k_infer_queue, dim3(blocks), dim3(kInferBlock), kFwdElems * (int) sizeof(uint16_t), st, nrc->wt.as<uint16_t>(), queries, strideF4,
					   count, capacity, L);
	NRC_HIP(hipGetLastError());
	return KRR_OK;
}

int nrcTrainDevice(krr_nrc *nrc, const float *vertices, const float *targets, const int *count, int capacity, int steps, hipStream_t st) {
	const int64_t cap = std::min<int64_t>(capacity, nrc->maxBatch);
	if (cap <= 0 || steps <= 0) return KRR_OK;
	const int64_t m = (cap + steps - 1) / steps; // largest mini-batch
	for (int b = 0; b < steps; b++)
		if (int rc = gradientImpl(nrc, (const krr_nrc_vertex *) vertices, targets, m, st, nullptr, count, cap, b, steps)) return rc;
	return KRR_OK;
}

float nrcLastLoss(krr_nrc *nrc, hipStream_t st) {
	if (hipStreamSynchronize(st) != hipSuccess) return -1.f;
	return nrc->loss.read();
}

extern "C" {

int krr_nrc_train_step(krr_nrc *nrc, const krr_nrc_vertex *vertices_dev, const float *targets_dev, int64_t n, float *loss_out,
					   void *hip_stream) {
	krr::clearError();
	if (!nrc || n < 1 || !vertices_dev || !targets_dev) return krr::fail(KRR_ERR_INVALID_ARG, "krr_nrc_train_step: bad argument");
	if (n > nrc->maxBatch) return krr::fail(KRR_ERR_CAPACITY, "krr_nrc_train_step: batch %lld exceeds max_batch %lld", (long long) n, (long long) nrc->maxBatch);
	hipStream_t st = (hipStream_t) hip_stream;
	if (int rc = gradientImpl(nrc, vertices_dev, targets_dev, n, st, nullptr)) return rc;
	if (loss_out) {
		NRC_HIP(hipStreamSynchronize(st));
		*loss_out = nrc->loss.read();
	}
	return KRR_OK;
}

int64_t krr_nrc_steps(const krr_nrc *nrc) {
	if (!nrc) return -1;
	int t = 0;
	if (hipDeviceSynchronize() != hipSuccess || hipMemcpy(&t, nrc->step.p, sizeof(int), hipMemcpyDeviceToHost) != hipSuccess) return -1;
	return t;
}

} // extern "C"
