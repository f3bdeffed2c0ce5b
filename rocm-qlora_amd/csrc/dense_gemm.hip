// Linears over a weight decoded once per call, for many activation rows: one
// launch writes RND(W_deq) in the activation dtype into scratch memory -- as
// W rows [N][R] for the forward, as W^T rows [K][R] for dX, the reduction
// length padded with zeros to a multiple of 64 -- and the dense MFMA GEMM
// (rq_dense_gemm.h) multiplies by it.  The decoded weight is the reference's
// own intermediate, dequantize_int4 / dequantize_int8 (...).to(x.dtype)
// (quant_ops.py:55-78, :128-150, quant_linear.py:189-195), so only the order
// of fp32 sums can differ from the fused kernels.
//
// Decoding costs one pass of N K / 2 (NF4) bytes in and 2 N K out, whatever
// the row count; the fused GEMM decodes every weight tile again for each 256
// activation rows, in the same issue slots and LDS as its MFMAs.
#include "rq_dense_gemm.h"
#include "rq_dense.h"
#include "rq_pad.h"
#include "rq_launch.h"

#include <algorithm>

namespace rq {
namespace {

// ---------------------------------------------------------------------------
// Weight sources: the codes as stored.  load(f, n): raw words of n codes at
// flat index f; value(raw, i, lut): code i's fp32 value before its scale.
// ---------------------------------------------------------------------------
struct SrcNF4 {
  static constexpr int kBytesPer8 = 4;  // bytes of 8 codes
  const uint8_t* p;
  __device__ __forceinline__ float at(int64_t f, const float* lut) const {
    const uint32_t b = p[f >> 1];
    return lut[(f & 1) ? b >> 4 : b & 15u];
  }
  // the values of the 8 codes in `w` (low word) in k order
  __device__ static __forceinline__ void expand8(u32x2 w, const float* lut, float (&v)[8]) {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = lut[(w.x >> (4 * i)) & 15u];
  }
  __device__ static __forceinline__ u32x2 piece(const u32x4 (&r)[1], int i) { return u32x2{r[0][i], 0u}; }
};
struct SrcInt8 {
  static constexpr int kBytesPer8 = 8;
  const uint8_t* p;
  __device__ __forceinline__ float at(int64_t f, const float*) const { return float(int8_t(p[f])); }
  __device__ static __forceinline__ void expand8(u32x2 w, const float*, float (&v)[8]) {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = float(int8_t(uint8_t((i < 4 ? w.x : w.y) >> (8 * (i & 3)))));
  }
  __device__ static __forceinline__ u32x2 piece(const u32x4 (&r)[2], int i) {
    return u32x2{r[i >> 1][2 * (i & 1)], r[i >> 1][2 * (i & 1) + 1]};
  }
};

// The scale of flat element f of row n: blockwise over the flat weight
// (log2 >= 0: power-of-two block), or one per row (bs 0).
struct BlockOf {
  int64_t bs;
  int log2;
  __device__ __forceinline__ int64_t operator()(int64_t f, int64_t n) const {
    return bs == 0 ? n : (log2 >= 0 ? f >> log2 : f / bs);
  }
};

constexpr int kDecThreads = kPadThreads;

// one value in the operand type, as its storage word
template <int XT>
using Word = std::conditional_t<XT == RQ_DTYPE_F32, uint32_t, uint16_t>;
template <int XT>
__device__ __forceinline__ Word<XT> to_word(float v) {
  if constexpr (XT == RQ_DTYPE_F32) return f2u(v);
  else return uint16_t(to_x16<XT>(v));
}

// W rows, K % 64 == 0 and blocks of at least 8 inside a row: the output is
// the flat weight.  A lane takes 8 codes (one 16-byte store, consecutive
// lanes consecutive bytes), four such per thread, all loads first.  HBM and
// MALL writes bound it (4096 x 14336 to bf16: 32 us, 4.8 TB/s; 11008 x 4096 double
// quantized to fp16: 24 us).
template <int XT, class Src, class Scale>
__global__ __launch_bounds__(kDecThreads) void decode_rows_kernel(Src src, Scale scale, BlockOf blk, uint32_t n_chunks,
                                                                  uint32_t row_chunks, uint8_t* __restrict__ out,
                                                                  unsigned blocks, PadCopies pads) {
  __shared__ float lut[16];
  if (blockIdx.x >= blocks) return pad_copy_block<XT>(pads, blockIdx.x - blocks);
  if (threadIdx.x < 16) lut[threadIdx.x] = u2f(kNF4Bits[threadIdx.x]);
  __syncthreads();
  const uint32_t c0 = blockIdx.x * (4 * kDecThreads) + threadIdx.x;
  u32x2 w[4];
  float s[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    uint32_t c = c0 + kDecThreads * j;
    c = c < n_chunks ? c : n_chunks - 1;
    if constexpr (Src::kBytesPer8 == 4)
      w[j] = u32x2{__builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(src.p) + c), 0u};
    else
      w[j] = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(src.p) + c);
    s[j] = scale(blk(int64_t(c) * 8, c / row_chunks));
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t c = c0 + kDecThreads * j;
    if (c >= n_chunks) break;
    float v[8];
    Src::expand8(w[j], lut, v);
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = __fmul_rn(v[k], s[j]);
    store8<XT>(out + size_t(c) * (8 * DnEl<XT>::kSize), v);
  }
}

// W^T rows, N % 64 == 0, K % 64 == 0, blocks of at least 32 inside a row: a
// workgroup takes 64 weight rows x 256 columns, a thread rows 2p, 2p + 1 (p
// = thread % 32) and columns 32 (thread / 32) .. + 31.  It stores the pairs
// {n, n + 1} as one word at [k][2p] of an LDS tile (32 lanes fill one 128-byte
// row), which leaves as 128-byte runs of the output's rows (4096 x 14336 to bf16:
// 34 us, 4.5 TB/s).
template <int XT, class Src, class Scale>
__global__ __launch_bounds__(kDecThreads) void decode_cols_kernel(Src src, Scale scale, BlockOf blk, int64_t K,
                                                                  int64_t ldo, uint8_t* __restrict__ out, unsigned gx,
                                                                  unsigned blocks, PadCopies pads) {
  constexpr int ES = DnEl<XT>::kSize, kRow = 64 * ES;  // bytes of 64 rows' values of one column
  __shared__ float lut[16];
  __shared__ __attribute__((aligned(16))) uint8_t tile[256 * kRow];
  if (blockIdx.x >= blocks) return pad_copy_block<XT>(pads, blockIdx.x - blocks);
  const unsigned bx = blockIdx.x % gx, by = blockIdx.x / gx;
  const int t = threadIdx.x, p = t & 31;
  if (t < 16) lut[t] = u2f(kNF4Bits[t]);
  __syncthreads();
  const int64_t n0 = int64_t(by) * 64, k0 = int64_t(bx) * 256, kc = k0 + 32 * (t >> 5);
  constexpr int kPieces = Src::kBytesPer8 / 4;  // 16-byte loads of 32 codes
  if (kc < K) {  // K is a multiple of 32: the thread's columns are all live
    u32x4 w[2][kPieces];
    float s[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int64_t f = (n0 + 2 * p + i) * K + kc;
      const u32x4* src4 = reinterpret_cast<const u32x4*>(src.p + (f >> 3) * Src::kBytesPer8);
#pragma unroll
      for (int j = 0; j < kPieces; ++j) w[i][j] = src4[j];
      s[i] = scale(blk(f, n0 + 2 * p + i));
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float v[2][8];
#pragma unroll
      for (int i = 0; i < 2; ++i) Src::expand8(Src::piece(w[i], j), lut, v[i]);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        uint8_t* o = tile + (32 * (t >> 5) + 8 * j + e) * kRow + 2 * ES * p;
        const float a = __fmul_rn(v[0][e], s[0]), b = __fmul_rn(v[1][e], s[1]);
        if constexpr (XT == RQ_DTYPE_F32) *reinterpret_cast<u32x2*>(o) = u32x2{f2u(a), f2u(b)};
        else *reinterpret_cast<uint32_t*>(o) = cvt_pk<XT>(a, b);
      }
    }
  }
  __syncthreads();
  constexpr int kLanes = kRow / 16;  // 16-byte chunks per column
#pragma unroll
  for (int it = 0; it < kLanes; ++it) {
    const int r = (kDecThreads / kLanes) * it + t / kLanes, c = t % kLanes;
    if (k0 + r < K)
      *reinterpret_cast<u32x4*>(out + ((k0 + r) * ldo + n0) * ES + 16 * c) =
          *reinterpret_cast<const u32x4*>(tile + r * kRow + 16 * c);
  }
}

// Every other layout: 64 x 64 tiles decoded element by element (coalesced
// along k), written along either index; zeros past N and K up to the padded
// reduction length.  out has `rows` rows of ldo.
template <int XT, class Src, class Scale, bool TRANS>
__global__ __launch_bounds__(kDecThreads) void decode_any_kernel(Src src, Scale scale, BlockOf blk, int64_t N,
                                                                 int64_t K, int64_t rows, int64_t ldo,
                                                                 Word<XT>* __restrict__ out, unsigned gx,
                                                                 unsigned blocks, PadCopies pads) {
  __shared__ float lut[16];
  __shared__ Word<XT> tile[64][64 + 4 / sizeof(Word<XT>)];
  if (blockIdx.x >= blocks) return pad_copy_block<XT>(pads, blockIdx.x - blocks);
  const unsigned bx = blockIdx.x % gx, by = blockIdx.x / gx;
  const int t = threadIdx.x, c = t & 63;
  if (t < 16) lut[t] = u2f(kNF4Bits[t]);
  __syncthreads();
  const int64_t k0 = int64_t(bx) * 64, n0 = int64_t(by) * 64;
#pragma unroll 4
  for (int i = 0; i < 16; ++i) {
    const int r = 4 * i + (t >> 6);
    const int64_t n = n0 + r, k = k0 + c;
    float v = 0.0f;
    if (n < N && k < K) {
      const int64_t f = n * K + k;
      v = __fmul_rn(src.at(f, lut), scale(blk(f, n)));
    }
    tile[r][c] = to_word<XT>(v);
  }
  __syncthreads();
#pragma unroll 4
  for (int i = 0; i < 16; ++i) {
    const int r = 4 * i + (t >> 6);
    const int64_t row = (TRANS ? k0 : n0) + r, col = (TRANS ? n0 : k0) + c;
    if (row < rows && col < ldo) out[row * ldo + col] = TRANS ? tile[c][r] : tile[r][c];
  }
}

// u = RN(xl * pre) . S^T in fp32 on v_mfma_f32_16x16x4_f32, as K-split partials
// part[split][m][j] (the split's k steps of 32 in order): four waves of 16 rows
// per workgroup, up to 64 ranks; then their sum in split order into rows of
// rankp (zeros past the rank).  Lane (i, q) loads 16 bytes of row i at k = 16 t +
// 4 q in both operands, four MFMAs' k.  Latency bound: 16-64 ranks of a few
// hundred rows, so the splits spread it over the compute units.
template <int JB>
__global__ __launch_bounds__(256) void lora_rows_f32_kernel(const float* __restrict__ x, int64_t ldx, int64_t M,
                                                            const float* __restrict__ s, int64_t lds_, int rank,
                                                            float pre, int steps, int steps_per,
                                                            float* __restrict__ part) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i16 = lane & 15, q = lane >> 4;
  const int64_t m0 = int64_t(blockIdx.x) * 64 + 16 * wave;
  const int j0 = blockIdx.y * 16 * JB, b = blockIdx.z * steps_per;
  const int e = b + steps_per < steps ? b + steps_per : steps;
  int64_t m = m0 + i16;
  m = m < M ? m : M - 1;
  const float* xr = x + m * ldx + 4 * q;
  const float* sr[JB];
#pragma unroll
  for (int jb = 0; jb < JB; ++jb) {
    const int j = j0 + 16 * jb + i16;
    sr[jb] = s + int64_t(j < rank ? j : rank - 1) * lds_ + 4 * q;  // ranks past the end: never stored
  }
  f32x4 acc[JB];
#pragma unroll
  for (int jb = 0; jb < JB; ++jb) acc[jb] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int t = b; t < e; ++t) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int64_t k = 32 * int64_t(t) + 16 * h;
      const f32x4 xv = *reinterpret_cast<const f32x4*>(xr + k);
#pragma unroll
      for (int jb = 0; jb < JB; ++jb) {
        const f32x4 sv = *reinterpret_cast<const f32x4*>(sr[jb] + k);
#pragma unroll
        for (int c = 0; c < 4; ++c)
          acc[jb] = __builtin_amdgcn_mfma_f32_16x16x4f32(__fmul_rn(xv[c], pre), sv[c], acc[jb], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int jb = 0; jb < JB; ++jb) {
    const int j = j0 + 16 * jb + i16;
    if (j >= rank) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t mo = m0 + 4 * q + r;
      if (mo < M) part[(int64_t(blockIdx.z) * M + mo) * rank + j] = acc[jb][r];
    }
  }
}

__global__ __launch_bounds__(256) void lora_sum_f32_kernel(const float* __restrict__ part, int splits, int64_t M,
                                                           int rank, int rankp, float* __restrict__ u) {
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i >= M * rankp) return;
  const int64_t m = i / rankp;
  const int j = int(i - m * rankp);
  float v = 0.0f;
  if (j < rank) {
#pragma unroll 8
    for (int k = 0; k < splits; ++k) v = __fadd_rn(v, part[(int64_t(k) * M + m) * rank + j]);
  }
  u[i] = v;
}

// ---------------------------------------------------------------------------
// Plan
// ---------------------------------------------------------------------------
constexpr size_t kPad = 256;
size_t up(size_t b) { return (b + kPad - 1) / kPad * kPad; }
int el_size(int dt) { return dt == RQ_DTYPE_F32 ? 4 : 2; }
int64_t step_len(int dt) { return 128 / el_size(dt); }

struct DensePlan {
  int halves, tiles_m, tiles_n, whole, splits;
  int64_t Rp, rankp;
  bool pad;  // the reduction length is padded: activations and factors copied
  LoraRowsPlan lr;          // 16-bit
  int u_splits, u_steps;    // fp32: K splits of u and their k steps
  size_t w, cnt, b, u, lpart, x, xl, s, part, bytes;
};

// Microseconds of a tiling, from measurements with all 256 compute units busy:
// 1.45 us per 64-k step of a 256 x 256 tile and 8 us per round of tiles, 0.55 us
// per step of a 128 x 128 one (N(0, 1) operands; power bound), K splits adding
// 20 and 8 us for their partial tiles (2048 x 4096 x 4096: 128 tiles of 256 in
// two splits 77 us, 512 tiles of 128 unsplit 69 us; 1024 x 4096 x 4096: 55.6 and
// 35.5 us; 4096 x 4096 x 14336: 347 and 429 us).  fp32: 128 x 128 tiles, 2 us per
// 32-k step, up to 8 splits (fp32 MFMA bound).
double pick_tiles(DensePlan& p, int xt, int64_t M, int64_t C, int nk, int cus) {
  const bool f32 = xt == RQ_DTYPE_F32;
  double best = 1e300;
  for (int h = f32 ? 1 : 2; h >= 1; --h) {
    const int64_t B = 128 * h, tm = ceil_div(M, B), tn = ceil_div(C, B), T = tm * tn;
    const double step = f32 ? 2.0 : (h == 2 ? 1.45 : 0.55), round = h == 2 ? 8.0 : 0.0, extra = h == 2 ? 20.0 : 8.0;
    const int64_t lt = T % cus, lf = T - lt;
    for (int s = 1; s <= (f32 ? 8 : 4); s *= 2) {
      if (s > 1 && (lt == 0 || lt * s > cus || nk / s < 4)) break;
      const double t = double(lf / cus) * (step * nk + round) + (lt ? step * double(ceil_div(nk, s)) + round : 0.0) +
                       (s > 1 ? extra : 0.0);
      if (t < best) {
        best = t;
        p.halves = h;
        p.tiles_m = int(tm);
        p.tiles_n = int(tn);
        p.splits = s;
        p.whole = int(s > 1 ? lf : T);
      }
    }
  }
  return best;
}

DensePlan plan_dense(int xt, int64_t M, int64_t C, int64_t R, int64_t rank, int cus) {
  DensePlan p{};
  const int64_t sl = step_len(xt), rp = xt == RQ_DTYPE_F32 ? 8 : 16;
  const size_t es = size_t(el_size(xt));
  p.Rp = ceil_div(R, sl) * sl;
  p.pad = p.Rp != R;
  p.rankp = rank > 0 ? ceil_div(rank, rp) * rp : 0;
  pick_tiles(p, xt, M, C, int(p.Rp / sl), cus);
  size_t off = 0;
  auto take = [&](size_t b) {
    const size_t o = off;
    off += up(b);
    return o;
  };
  const size_t lt = size_t(p.tiles_m) * p.tiles_n - p.whole;
  p.w = take(size_t(C) * p.Rp * es);
  p.cnt = take(lt * 4 + 4);
  if (rank > 0) {
    p.b = take(size_t(C) * p.rankp * es);
    p.u = take(size_t(M) * p.rankp * es);
    if (xt == RQ_DTYPE_F32) {
      // about two workgroups per compute unit, at least two steps each
      const int64_t steps = p.Rp / sl, wgs = ceil_div(M, 64) * ceil_div(rank, 64);
      int64_t ks = std::min(std::max<int64_t>(2 * cus / wgs, 1), std::max<int64_t>(steps / 2, 1));
      ks = std::min<int64_t>(ks, 64);
      p.u_steps = int(ceil_div(steps, ks));
      p.u_splits = int(ceil_div(steps, p.u_steps));
      p.lpart = take(size_t(p.u_splits) * M * rank * 4);
    } else {
      p.lr = plan_lora_rows(M, p.Rp, rank, cus);
      p.lpart = take(p.lr.part_bytes);
    }
  }
  if (p.pad) {
    p.x = take(size_t(M) * p.Rp * es);
    if (rank > 0) p.xl = take(size_t(M) * p.Rp * es);
  }
  if (rank > 0 && (p.pad || xt == RQ_DTYPE_F32)) p.s = take(size_t(rank) * p.Rp * es);
  if (p.splits > 1) {
    const size_t B = 128 * p.halves;
    p.part = take(size_t(p.splits) * lt * B * B * 4);
  }
  p.bytes = off;
  return p;
}

// A product: activations x [M][R], the weight's columns C.
struct Product {
  int xt;
  const void* x;
  int64_t ldx, M, C, R;
  // LoRA: u = RND(RND(xl * pre) . RND(S)^T), S[j][r] at s[j s_j + r s_r];
  // second factor F[c][j] at f[c f_c + j f_j]
  int64_t rank;
  const void* xl;
  int64_t ldxl;
  const void* s;
  int64_t s_j, s_r;
  bool prescale;
  float pre = 1.0f;
  const void* f;
  int64_t f_c, f_j;
  int lora_dt;
  const void* u;  // u itself ([M][rankp]) when the caller has it
  DenseEpi e;
};

template <int XT, class Src, class Scale>
int launch_decode(Src src, Scale scale, int64_t N, int64_t K, int64_t bs, bool trans, int64_t Rp, void* w,
                  const PadCopies& pads, hipStream_t stream) {
  uint8_t* const out = static_cast<uint8_t*>(w);
  const BlockOf blk{bs, bs > 0 ? pow2_shift(bs) : -1};
  const bool blocks_ok = bs == 0 || (blk.log2 >= 5 && K % bs == 0);
  const int64_t chunks = N * (K / 8);
  // a linear grid: the decode's workgroups, then the copies'
  auto grid = [&](int64_t gx, int64_t gy, unsigned* blocks) {
    const int64_t n = gx * gy, all = n + pads.blocks();
    if (all > int64_t(INT32_MAX)) return 0u;
    *blocks = unsigned(n);
    return unsigned(all);
  };
  unsigned blocks = 0, all = 0;
  if (!trans && K % 64 == 0 && blocks_ok && aligned(src.p, 8) && chunks < int64_t(UINT32_MAX) - 4096) {
    if (!(all = grid(ceil_div(chunks, 4 * kDecThreads), 1, &blocks))) return RQ_ERR_UNSUPPORTED;
    decode_rows_kernel<XT, Src, Scale><<<all, kDecThreads, 0, stream>>>(src, scale, blk, uint32_t(chunks),
                                                                        uint32_t(K / 8), out, blocks, pads);
  } else if (trans && K % 64 == 0 && N % 64 == 0 && blocks_ok && aligned(src.p, 16)) {
    const int64_t gx = ceil_div(K, 256);
    if (!(all = grid(gx, N / 64, &blocks))) return RQ_ERR_UNSUPPORTED;
    decode_cols_kernel<XT, Src, Scale>
        <<<all, kDecThreads, 0, stream>>>(src, scale, blk, K, Rp, out, unsigned(gx), blocks, pads);
  } else {
    // tiles over the output: its padded reduction index and its rows
    const int64_t gx = ceil_div(trans ? K : Rp, 64), gy = ceil_div(trans ? Rp : N, 64);
    if (!(all = grid(gx, gy, &blocks))) return RQ_ERR_UNSUPPORTED;
    if (trans)
      decode_any_kernel<XT, Src, Scale, true><<<all, kDecThreads, 0, stream>>>(
          src, scale, blk, N, K, K, Rp, static_cast<Word<XT>*>(w), unsigned(gx), blocks, pads);
    else
      decode_any_kernel<XT, Src, Scale, false><<<all, kDecThreads, 0, stream>>>(
          src, scale, blk, N, K, N, Rp, static_cast<Word<XT>*>(w), unsigned(gx), blocks, pads);
  }
  return rq_check_launch();
}

// The launches of a product whose weight `decode` writes into w16.
template <int XT, class Decode>
int run_product(const Product& P, const Decode& decode, void* scratch, size_t bytes, hipStream_t stream) {
  constexpr bool kF32 = XT == RQ_DTYPE_F32;
  const DensePlan p = plan_dense(XT, P.M, P.C, P.R, P.rank, device_cus());
  if (!scratch || bytes < p.bytes) return RQ_ERR_WORKSPACE;
  if (!aligned(scratch, 256)) return RQ_ERR_BAD_ALIGNMENT;
  char* ws = static_cast<char*>(scratch);
  uint32_t* cnt = reinterpret_cast<uint32_t*>(ws + p.cnt);
  DenseEpi e = P.e;
  DenseGemmArgs a{};
  a.x = P.x;
  a.ldx = P.ldx;
  const void* xl = P.xl;
  int64_t ldxl = P.ldxl;
  const void* s = P.s;
  int64_t s_j = P.s_j, s_r = P.s_r;
  int s_dt = P.lora_dt;

  PadCopies pc{};
  auto copy = [&](const void* in, int dt, int64_t sr, int64_t sc, int64_t rows, int64_t cols, int64_t out_rows,
                  int64_t out_cols, size_t off) -> const void* {
    return pc.add(in, dt, sr, sc, rows, cols, out_rows, out_cols, ws + off);
  };
  if (P.rank > 0) {
    e.rankp = int(p.rankp);
    e.u = P.u ? P.u : ws + p.u;
    e.b = copy(P.f, P.lora_dt, P.f_c, P.f_j, P.C, P.rank, P.C, p.rankp, p.b);
  }
  if (p.pad) {
    const bool same = P.xl == P.x && P.ldxl == P.ldx;
    a.x = copy(P.x, XT, P.ldx, 1, P.M, P.R, P.M, p.Rp, p.x);
    a.ldx = p.Rp;
    if (P.rank > 0 && !P.u) {
      xl = same ? a.x : copy(P.xl, XT, P.ldxl, 1, P.M, P.R, P.M, p.Rp, p.xl);
      ldxl = p.Rp;
    }
  }
  if (P.rank > 0 && !P.u && (p.pad || kF32)) {
    s = copy(P.s, P.lora_dt, P.s_j, P.s_r, P.rank, P.R, P.rank, p.Rp, p.s);
    s_j = p.Rp;
    s_r = 1;
    s_dt = XT;
  }
  if (p.splits > 1) {
    pc.cnt = cnt;
    pc.n_cnt = p.tiles_m * p.tiles_n - p.whole;
  }
  // one launch decodes the weight and makes the copies
  int st = decode(static_cast<void*>(ws + p.w), p.Rp, pc);
  if (st != RQ_OK) return st;
  if (P.rank > 0 && !P.u) {
    float* lpart = reinterpret_cast<float*>(ws + p.lpart);
    if constexpr (kF32) {
      const int rank = int(P.rank), jb = rank <= 16 ? 1 : (rank <= 32 ? 2 : 4);
      const dim3 grid(unsigned(ceil_div(P.M, 64)), unsigned(ceil_div(rank, 16 * jb)), unsigned(p.u_splits));
      auto launch = [&](auto kernel) {
        kernel<<<grid, 256, 0, stream>>>(static_cast<const float*>(xl), ldxl, P.M, static_cast<const float*>(s), s_j,
                                         rank, P.pre, int(p.Rp / 32), p.u_steps, lpart);
      };
      if (jb == 1) launch(lora_rows_f32_kernel<1>);
      else if (jb == 2) launch(lora_rows_f32_kernel<2>);
      else launch(lora_rows_f32_kernel<4>);
      lora_sum_f32_kernel<<<unsigned(ceil_div(P.M * p.rankp, 256)), 256, 0, stream>>>(
          lpart, p.u_splits, P.M, rank, int(p.rankp), reinterpret_cast<float*>(ws + p.u));
      st = rq_check_launch();
    } else {
      st = run_lora_rows(XT, static_cast<const uint16_t*>(xl), ldxl, P.M, p.Rp, s, s_dt, s_j, s_r, int(P.rank),
                         P.prescale, P.pre, p.lr, lpart, reinterpret_cast<uint16_t*>(ws + p.u), int(p.rankp), stream);
    }
    if (st != RQ_OK) return st;
  }
  a.w = ws + p.w;
  a.ldw = p.Rp;
  a.M = P.M;
  a.N = P.C;
  a.nk = int(p.Rp / step_len(XT));
  a.tiles_m = p.tiles_m;
  a.tiles_n = p.tiles_n;
  a.whole = p.whole;
  a.splits = p.splits;
  a.part = reinterpret_cast<float*>(ws + p.part);
  a.tile_cnt = cnt;
  const int64_t T = int64_t(p.tiles_m) * p.tiles_n;
  const unsigned grid = unsigned(p.whole + (T - p.whole) * p.splits);
  if constexpr (kF32) {
    dense_gemm_kernel<XT, 1><<<grid, kDnThreads, 0, stream>>>(a, e);
  } else {
    if (p.halves == 2) dense_gemm_kernel<XT, 2><<<grid, kDnThreads, 0, stream>>>(a, e);
    else dense_gemm_kernel<XT, 1><<<grid, kDnThreads, 0, stream>>>(a, e);
  }
  return rq_check_launch();
}

// `fn(scale)` with the scale provider of an NF4 weight.
template <class Fn>
int with_nf4_scale(const void* absmax, int dt, const uint8_t* c2, int c2_format, int64_t block2, const Fn& fn) {
  if (c2) {
    const int sh = pow2_shift(block2);
    switch (dt) {
      case RQ_DTYPE_F32: return fn(ScaleDQ<RQ_DTYPE_F32>{c2, absmax, c2_format, sh, block2});
      case RQ_DTYPE_BF16: return fn(ScaleDQ<RQ_DTYPE_BF16>{c2, absmax, c2_format, sh, block2});
      default: return fn(ScaleDQ<RQ_DTYPE_F16>{c2, absmax, c2_format, sh, block2});
    }
  }
  switch (dt) {
    case RQ_DTYPE_F32: return fn(ScaleAbsmax<RQ_DTYPE_F32>{absmax});
    case RQ_DTYPE_BF16: return fn(ScaleAbsmax<RQ_DTYPE_BF16>{absmax});
    default: return fn(ScaleAbsmax<RQ_DTYPE_F16>{absmax});
  }
}

template <int XT, class Src, class WithScale>
int run_weight(const Product& P, const Src& src, const WithScale& with_scale, int64_t N, int64_t K, int64_t bs,
               bool trans, void* scratch, size_t bytes, hipStream_t stream) {
  return run_product<XT>(
      P,
      [&](void* w, int64_t Rp, const PadCopies& pads) {
        return with_scale([&](auto sc) { return launch_decode<XT>(src, sc, N, K, bs, trans, Rp, w, pads, stream); });
      },
      scratch, bytes, stream);
}

// run_weight for the activation dtype
template <class Src, class WithScale>
int run_any(const Product& P, const Src& src, const WithScale& ws, int64_t N, int64_t K, int64_t bs, bool trans,
            void* scratch, size_t bytes, hipStream_t stream) {
  switch (P.xt) {
    case RQ_DTYPE_F32: return run_weight<RQ_DTYPE_F32>(P, src, ws, N, K, bs, trans, scratch, bytes, stream);
    case RQ_DTYPE_BF16: return run_weight<RQ_DTYPE_BF16>(P, src, ws, N, K, bs, trans, scratch, bytes, stream);
    default: return run_weight<RQ_DTYPE_F16>(P, src, ws, N, K, bs, trans, scratch, bytes, stream);
  }
}

// 16-byte activation loads when the reduction is not copied into padded rows
bool act_ok(int dt, const void* x, int64_t ldx, int64_t M, int64_t R) {
  const int64_t es = el_size(dt);
  return R % step_len(dt) != 0 ||
         (aligned(x, 16) && ldx * es % 16 == 0 && double(M) * double(ldx) * double(es) < 4294967296.0);
}

}  // namespace

size_t dense_scratch_bytes(int x_dtype, int64_t M, int64_t C, int64_t R, int64_t rank) {
  const int64_t Rp = ceil_div(R, step_len(x_dtype)) * step_len(x_dtype);
  if (M < 1 || rank < 0 || rank > 256) return 0;
  // 32-bit byte offsets into both operands, tile counts in an int
  const double es = el_size(x_dtype);
  if (double(C) * double(Rp) * es >= 4294967296.0 || double(M) * double(Rp) * es >= 4294967296.0) return 0;
  if (ceil_div(M, 128) * ceil_div(C, 128) > int64_t(1) << 28) return 0;
  return plan_dense(x_dtype, M, C, R, rank > 0 ? rank : 0, device_cus()).bytes;
}

namespace {
// Microseconds of a tiled product, fitted to measurements (957 calls: 17 to 4096
// rows, 1024 to 14336 columns and reduction lengths, both routes timed in turn).
// A round of tiles costs `round` and, per 64-k step, `alone` while at most half
// of the compute units have a workgroup, growing to alone + shared when all do;
// splitting K costs `split`, the call `call`.
struct ProductCost {
  double alone, shared, round, split, call;
};
constexpr ProductCost kFusedCost[3] = {
    {0.73, 0.28, 6.6, 7.2, 1.5},  // kFusedNF4
    {0.92, 0.16, 4.8, 0.0, 5.7},  // kFusedNF4Dx
    {0.78, 0.26, 6.0, 0.0, 0.9},  // kFusedInt8
};
// by tile: 128 x 128, 256 x 256 (the call: its decode launch)
constexpr ProductCost kDenseCost[2] = {{0.20, 0.23, 5.3, 2.6, 9.0}, {0.84, 0.57, 9.2, 13.6, 9.0}};
constexpr double kDecodeUs = 0.48e-6;  // a weight's, written and read back

double product_us(const ProductCost& c, int64_t rounds, int64_t tail, int splits, int64_t nk, int cus) {
  auto step = [&](int64_t busy) { return c.alone + c.shared * std::max(0.0, 2.0 * std::min<int64_t>(busy, cus) / cus - 1.0); };
  return c.call + double(rounds) * (double(nk) * step(cus) + c.round) +
         (tail > 0 ? double(ceil_div(nk, splits)) * step(tail * splits) + c.round : 0.0) + (splits > 1 ? c.split : 0.0);
}
}  // namespace

// Both sides measured, us, fused against dense: NF4 forward 4096 -> 4096 M = 256
// 27.6 / 37.3, M = 1536 62.5 / 72.1, M = 3072 120 / 96.4; 14336 -> 4096 M = 256 58.3
// / 76.9, M = 1024 130 / 139, M = 2048 242 / 213; 4096 -> 14336 M = 640 106 / 111, M =
// 1024 135 / 120; dX from 4096 to 11008 columns M = 256 71.5 / 56.0; INT8 1024 ->
// 8192 M = 512 20.2 / 28.1.  The rule sends here four
// of the 957 calls, and eleven of 659 further ones of drawn sizes, that are more than
// 3 % faster fused (9 % at most); the 1.5 % that it asks for keeps calls that gain
// nothing from taking scratch memory.  fp16 and double-quantized scales cost both
// sides alike (3 and 5 %).
bool dense_beats_fused(int64_t M, int64_t C, int64_t R, FusedKernel kernel) {
  if (M <= kGemvMaxM) return false;
  const int cus = device_cus();
  const GemmPlan f = plan_gemm(M, C, R, 0, cus, kernel == kFusedNF4);
  const int64_t T = int64_t(f.tiles_m) * f.tiles_n;
  const int64_t rounds = f.splits > 1 ? f.lf * 8 / cus : T / cus;
  const double fused = product_us(kFusedCost[kernel], rounds, T - rounds * cus, f.splits, ceil_div(R, 64), cus);
  DensePlan p{};
  const int64_t nk = ceil_div(R, 64);
  pick_tiles(p, RQ_DTYPE_BF16, M, C, int(nk), cus);
  const int64_t D = int64_t(p.tiles_m) * p.tiles_n;
  const double dense = product_us(kDenseCost[p.halves - 1], D / cus, D % cus, p.splits, nk, cus);
  return dense + kDecodeUs * double(C) * double(R) < 0.985 * fused;
}

// fp32 forward against the GEMV kernels over blocks of 16 rows.  A block costs 3.9 +
// 0.0021 K us per round of 16-column tiles (one per compute unit), its LoRA operand
// 2.6 us plus, per rank, 0.14 us a round and 13 ps per k; the dense side the
// product's estimate, 0.9 us per million weights decoded, 8 us of launches and for
// LoRA 7 us + 0.16 us per rank.  Of 240 calls timed on both routes (512 to 14336
// columns and reduction lengths, 32 to 256 rows, ranks 0, 16, 64) two taken here are
// slower, by 4 %.  Blocks against dense, us: 4096 -> 4096 M = 64 49 / 65, M = 96 74 /
// 65, rank 16 M = 64 75 / 75; 1024 -> 1024 rank 16 M = 48 35 / 33, M = 256 186 / 34;
// 14336 -> 4096 M = 64 149 / 181.
bool dense_beats_f32_blocks(int64_t M, int64_t C, int64_t R, int64_t rank) {
  if (M <= kGemvMaxM) return false;
  const int cus = device_cus();
  const double rounds = double(ceil_div(ceil_div(C, 16), cus)), K = double(R), r = double(rank);
  const double block = rounds * (3.9 + 0.0021 * K) + (rank > 0 ? 2.6 + r * (0.14 * rounds + 1.3e-5 * K) : 0.0);
  DensePlan p{};
  const double dense = pick_tiles(p, RQ_DTYPE_F32, M, C, int(ceil_div(R, 32)), cus) + 8.0 +
                       0.9e-6 * double(C) * K + (rank > 0 ? 7.0 + 0.16 * r : 0.0);
  return dense < block * double(ceil_div(M, 16));
}

bool dense_nf4_linear_ok(const LinearArgs& L) {
  return act_ok(L.x_dtype, L.x, L.ldx, L.M, L.K) &&
         (L.rank == 0 || act_ok(L.x_dtype, L.lora_x, L.ld_lora_x, L.M, L.K));
}
bool dense_nf4_dx_ok(const DxArgs& D) { return act_ok(D.dy_dtype, D.dy, D.lddy, D.M, D.N); }
bool dense_int8_ok(const GenericInt8& A, bool dx) { return act_ok(A.x_dtype, A.x, A.ldx, A.M, dx ? A.N : A.K); }

int run_dense_nf4_linear(const LinearArgs& L, void* scratch, size_t bytes, hipStream_t stream) {
  Product P{};
  P.xt = L.x_dtype; P.x = L.x; P.ldx = L.ldx; P.M = L.M; P.C = L.N; P.R = L.K;
  if (L.rank > 0) {
    P.rank = L.rank; P.xl = L.lora_x; P.ldxl = L.ld_lora_x;
    P.s = L.lora_a; P.s_j = L.K; P.s_r = 1;
    P.f = L.lora_b; P.f_c = L.ld_lora_b; P.f_j = 1;
    P.lora_dt = L.lora_dtype;
  }
  P.e.bias = L.bias; P.e.bias_dt = L.bias_dtype; P.e.scaling = L.scaling;
  P.e.y = L.y; P.e.ldy = L.ldy;
  auto ws = [&](auto fn) { return with_nf4_scale(L.absmax, L.absmax_dtype, L.c2, L.c2_format, L.block2, fn); };
  const SrcNF4 src{L.w_packed};
  return run_any(P, src, ws, L.N, L.K, L.block_size, false, scratch, bytes, stream);
}

int run_dense_nf4_dx(const DxArgs& D, void* scratch, size_t bytes, hipStream_t stream) {
  Product P{};
  P.xt = D.dy_dtype; P.x = D.dy; P.ldx = D.lddy; P.M = D.M; P.C = D.K; P.R = D.N;
  if (D.rank > 0) {
    // g = RND(RND(dY * s) . RND(B)), then g . RND(A): S[j][n] = B[n][j], F[k][j] = A[j][k]
    P.rank = D.rank; P.xl = D.dy; P.ldxl = D.lddy;
    P.s = D.lora_b; P.s_j = 1; P.s_r = D.ld_lora_b; P.prescale = true; P.pre = D.scaling;
    P.f = D.lora_a; P.f_c = 1; P.f_j = D.K;
    P.lora_dt = D.lora_dtype;
    P.u = D.lora_g;
    P.e.mask = D.lora_mask; P.e.ldm = D.ld_lora_mask; P.e.mask_scale = D.mask_scale;
  }
  P.e.scaling = 1.0f;
  P.e.y = D.dx; P.e.ldy = D.lddx;
  auto ws = [&](auto fn) { return with_nf4_scale(D.absmax, D.absmax_dtype, D.c2, D.c2_format, D.block2, fn); };
  const SrcNF4 src{D.w_packed};
  return run_any(P, src, ws, D.N, D.K, D.block_size, true, scratch, bytes, stream);
}

int run_dense_int8(const GenericInt8& A, bool dx, void* scratch, size_t bytes, hipStream_t stream) {
  Product P{};
  P.xt = A.x_dtype; P.x = A.x; P.ldx = A.ldx; P.M = A.M; P.C = dx ? A.K : A.N; P.R = dx ? A.N : A.K;
  P.e.bias = dx ? nullptr : A.bias; P.e.bias_dt = A.bias_dtype; P.e.scaling = 1.0f;
  P.e.y = A.y; P.e.ldy = A.ldy;
  if (dx && A.rank > 0) {
    P.rank = A.rank; P.u = A.lora_g;
    P.f = A.lora_a; P.f_c = 1; P.f_j = A.K;
    P.lora_dt = A.lora_dtype;
    P.e.mask = A.lora_mask; P.e.ldm = A.ld_lora_mask; P.e.mask_scale = A.mask_scale;
  }
  auto ws = [&](auto fn) {
    return with_nf4_scale(A.scales, A.scales_dtype, nullptr, 0, 1, fn);
  };
  const SrcInt8 src{reinterpret_cast<const uint8_t*>(A.q)};
  return run_any(P, src, ws, A.N, A.K, A.block_size, dx, scratch, bytes, stream);
}

}  // namespace rq

extern "C" int rq_dense_tile_plan(int x_dtype, int64_t M, int64_t C, int64_t R, int32_t* out) {
  if (!out) return RQ_ERR_NULL_POINTER;
  if (!rq::valid_float_dtype(x_dtype)) return RQ_ERR_BAD_DTYPE;
  if (M < 1 || C < 1 || R < 1 || rq::dense_scratch_bytes(x_dtype, M, C, R, 0) == 0) return RQ_ERR_BAD_SHAPE;
  const rq::DensePlan p = rq::plan_dense(x_dtype, M, C, R, 0, rq::device_cus());
  out[0] = 128 * p.halves;
  out[1] = p.whole;
  out[2] = p.tiles_m * p.tiles_n - p.whole;
  out[3] = p.splits;
  return RQ_OK;
}
