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

// Its scratch memory: the K splits' partial tiles and the LoRA operand's partials
// (contents ignored; 0: none needed).
// Up to kSkinnyHeldBytes of it are part of the workspace, which callers keep: a
// call that small is bound by its host time, and memory of its own for each call
// costs 1.6 of 15 us.  More is asked for per call and given back.
constexpr size_t kSkinnyHeldBytes = size_t(1536) << 10;
size_t skinny_scratch(int64_t M, int64_t N, int64_t K, int64_t rank);
// Tile counters it uses (zero before and after the call; 0: none).
size_t skinny_counters(int64_t M, int64_t N, int64_t K);

int run_skinny_nf4(const LinearArgs& L, void* scratch, size_t bytes, uint32_t* cnt, hipStream_t stream);

}  // namespace rq
