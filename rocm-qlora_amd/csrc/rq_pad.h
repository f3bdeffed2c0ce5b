// Copies of small operands into padded rows, as part of another launch or one of
// their own (device code shared by dense_gemm.hip and lora_grad.hip).
#pragma once
#include "rq_mfma.h"

namespace rq {

constexpr int kPadThreads = 256;

// Eight values in the operand type at p (16-byte aligned): 16 or 32 bytes.
template <int XT>
__device__ __forceinline__ void store8(void* p, const float (&v)[8]) {
  u32x4* o = static_cast<u32x4*>(p);
  if constexpr (XT == RQ_DTYPE_F32) {
    o[0] = u32x4{f2u(v[0]), f2u(v[1]), f2u(v[2]), f2u(v[3])};
    o[1] = u32x4{f2u(v[4]), f2u(v[5]), f2u(v[6]), f2u(v[7])};
  } else {
    o[0] = u32x4{cvt_pk<XT>(v[0], v[1]), cvt_pk<XT>(v[2], v[3]), cvt_pk<XT>(v[4], v[5]), cvt_pk<XT>(v[6], v[7])};
  }
}

// The small operands of a product: `cnt` words zeroed, and up to four copies out[r][c] = RND(in[r * sr + c * sc]) with zeros past the source's
// rows and columns -- the GEMM's second LoRA operand, and for reduction lengths
// that are not whole k steps the activations, the LoRA input and the first
// LoRA factor (fp32: always the first factor).
struct PadCopy {
  const void* in;
  int dt;
  int64_t sr, sc;
  int64_t rows, cols;          // live part
  int64_t out_rows, out_cols;  // out_cols a multiple of 8
  void* out;
  int64_t first;               // first workgroup
};
struct PadCopies {
  PadCopy c[4];
  int n;
  int64_t groups;  // workgroups of all copies
  uint32_t* cnt;
  int n_cnt;
  // appends a copy; returns its output
  void* add(const void* in, int dt, int64_t sr, int64_t sc, int64_t rows, int64_t cols, int64_t out_rows,
            int64_t out_cols, void* out) {
    c[n++] = PadCopy{in, dt, sr, sc, rows, cols, out_rows, out_cols, out, groups};
    groups += ceil_div(out_rows * (out_cols / 8), kPadThreads);
    return out;
  }
  int64_t blocks() const { return groups > 0 ? groups : (n_cnt > 0 ? 1 : 0); }
};

// Workgroup g of the copies (kPadThreads threads).
template <int XT>
__device__ __forceinline__ void pad_copy_block(const PadCopies& P, int64_t g) {
  if (g == 0)
    for (int i = threadIdx.x; i < P.n_cnt; i += kPadThreads) P.cnt[i] = 0u;
  for (int i = 0; i < P.n; ++i) {
    const PadCopy& c = P.c[i];
    const int64_t per = c.out_cols / 8, groups = c.out_rows * per;
    const int64_t idx = (g - c.first) * kPadThreads + threadIdx.x;
    if (g < c.first || idx >= groups) continue;
    // lanes run along the source's contiguous index
    int64_t r, c8;
    if (c.sc == 1) {
      r = idx / per;
      c8 = (idx - r * per) * 8;
    } else {
      const int64_t q = idx / c.out_rows;
      r = idx - q * c.out_rows;
      c8 = q * 8;
    }
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e)
      v[e] = r < c.rows && c8 + e < c.cols ? load_as_f32(c.in, r * c.sr + (c8 + e) * c.sc, c.dt) : 0.0f;
    store8<XT>(static_cast<uint8_t*>(c.out) + (r * c.out_cols + c8) * (XT == RQ_DTYPE_F32 ? 4 : 2), v);
  }
}

}  // namespace rq
