// Host interface of the dequantize-once linears (dense_gemm.hip): the weight
// is decoded into scratch memory by one launch and multiplied by the dense
// MFMA GEMM (rq_dense_gemm.h).  For NF4 and INT8 weights, forward and dX,
// any activation dtype, sizes, block sizes and alignments.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include "rq_common.h"
#include "rq_generic.h"
#include "rq_linear.h"

namespace rq {

// Scratch bytes of a product of M activation rows with C output columns over
// a reduction of R, LoRA rank included; 0 when the product never runs here
// (operands past 32-bit offsets, more than 256 ranks).
size_t dense_scratch_bytes(int x_dtype, int64_t M, int64_t C, int64_t R, int64_t rank);

// The GEMM over the stored codes that a call runs on otherwise (the NF4 forward's
// splits K for its last round of tiles).
enum FusedKernel { kFusedNF4, kFusedNF4Dx, kFusedInt8 };
// Whether the dense path is the faster one for a call that kernel takes.
bool dense_beats_fused(int64_t M, int64_t C, int64_t R, FusedKernel kernel);

// The same for fp32 activations and the row-block GEMV kernels (forward).
bool dense_beats_f32_blocks(int64_t M, int64_t C, int64_t R, int64_t rank);

// Whether the operands' alignment suits the dense path (any, once the
// reduction is padded; else activation rows of 16-byte chunks).
bool dense_nf4_linear_ok(const LinearArgs& L);
bool dense_nf4_dx_ok(const DxArgs& D);
bool dense_int8_ok(const GenericInt8& A, bool dx);

int run_dense_nf4_linear(const LinearArgs& L, void* scratch, size_t bytes, hipStream_t stream);
int run_dense_nf4_dx(const DxArgs& D, void* scratch, size_t bytes, hipStream_t stream);
int run_dense_int8(const GenericInt8& A, bool dx, void* scratch, size_t bytes, hipStream_t stream);

}  // namespace rq
