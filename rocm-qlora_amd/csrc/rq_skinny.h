// Host interface of the skinny linear (skinny_linear.hip): NF4
// weights, 16-bit activations, a few tens of rows.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include "rq_linear.h"

namespace rq {

// Whether a call with M rows runs on the skinny kernel (its other operands
// being those the fused GEMMs take, LoRA rank at most 64).
bool skinny_takes(int64_t M, int64_t N, int64_t K, int64_t rank);

// Its workspace: the K splits' partial tiles and the LoRA operand's partials.
size_t skinny_workspace(int64_t M, int64_t N, int64_t K, int64_t rank);
// Tile counters it uses (zero before and after the call; 0: none).
size_t skinny_counters(int64_t M, int64_t N, int64_t K);

int run_skinny_nf4(const LinearArgs& L, void* workspace, size_t bytes, uint32_t* cnt, hipStream_t stream);

}  // namespace rq
