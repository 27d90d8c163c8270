// nrc_dev.h - network geometry and matrix-core operand types of the neural
// radiance cache (nrc.hip).
#pragma once

#include <stdint.h>

#include "krr_nrc.h"

namespace krr {
namespace nrc {

constexpr int kHidden = KRR_NRC_HIDDEN_LAYERS; // hidden layers of width 64 (= matrices before the output one)
// bf16 weight copies: forward A operands W^T [out][in] (output layer padded
// to 32 rows) and backward A operands W [in][out] (output layer padded to 32
// columns), each layer in the order in which the matrix cores' lanes take it:
// half of 32 rows, pair of 8-column K-steps, lane, 8 bf16.  A wave reads a pair
// as 64 consecutive 16-byte pieces, from LDS without bank conflicts or
// padding, from memory without partial lines.
constexpr int kFwdElems = kHidden * 64 * 64 + 32 * 64;
constexpr int kBwdElems = kHidden * 64 * 64 + 64 * 32;
// Place of element (row, col) of a layer with `cols` columns: lane half g of
// row r holds columns 8s + 4g + j of K-steps s and s + 1.
__host__ __device__ constexpr int operandIndex(int row, int col, int cols) {
	return ((row / 32 * (cols / 16) + col / 16) * 64 + (col / 4 % 2) * 32 + row % 32) * 8 + col / 8 % 2 * 4 + col % 4;
}

typedef short short4v __attribute__((ext_vector_type(4)));	// 4 x bf16 (bit patterns)
typedef short short8v __attribute__((ext_vector_type(8)));	// two of them: a pair of K-steps
typedef float float16v __attribute__((ext_vector_type(16))); // 32x32 accumulator slice of one lane

} // namespace nrc
} // namespace krr

#ifdef __HIPCC__
#include <hip/hip_runtime.h>

// Entry points for the path tracer, with counts read on the device (no host
// synchronisation inside a frame).
//
// Queries: `count` records of `strideF4` float4 each; float4 0..3 are the
// krr_nrc_vertex, float4 4 = {thp.xyz, pixel bits}.  Adds thp * max(cache, 0)
// to L[pixel] (one query per pixel per sample, so no atomics).
int nrcInferAccumulate(krr_nrc *nrc, const float4 *queries, int strideF4, const int *count, int capacity, float4 *L, hipStream_t st);
// `steps` Adam steps, one per equal consecutive slice of the first
// min(*count, capacity) vertices (16 floats each) and targets (3 floats
// each), the slices computed on the device; kernels sized for `capacity`.
int nrcTrainDevice(krr_nrc *nrc, const float *vertices, const float *targets, const int *count, int capacity, int steps, hipStream_t st);
// Loss of the last training step (synchronises the stream).
float nrcLastLoss(krr_nrc *nrc, hipStream_t st);
#endif
