// Gradients of the LoRA adapters (lora_layer.py:67 differentiated), 16-bit
// activations:
//   dv = RND(dY * s)                       [M, N]
//   u  = RND(x . RND(A)^T)                 [M, r]
//   g  = RND(dv . RND(B))                  [M, r]   (also dX's LoRA operand)
//   dB = RND(dv^T u)  [N, r],  dA = RND(g^T x)  [r, K], widened to the
//        adapters' dtype.
// u and g are split-K products of the rows (lora_rows_kernel, rq_lora.hip)
// whose finish writes them transposed, [r16][M], as MFMA operands; dB and dA
// are one launch that reads dY and x once.
//
// lora_grad_kernel is a contraction over the rows m, the slow index of dY and
// x: lane (i, g) = (lane % 16, lane / 16) loads 16 bytes (8 columns) of the 8
// rows 8 g .. 8 g + 7, so that 32 byte permutes give it, for each of its 8
// columns, the 8 consecutive m of a v_mfma_f32_16x16x32 operand row -- no LDS,
// whole 256-byte row pieces per instruction.  A wave covers 128 columns x 32
// rows per step with 8 x (r / 16) MFMAs.  Bound by reading dY and x: at M =
// 4096, K = 4096, N = 14336, r = 64 the library GEMMs, the dY * s pass and the
// casts it replaces took 182 us; now g 46 us, u 16 us, their finish 14 us and this
// kernel 69 us (2.2 TB/s with 64 ranks; 8 ranks at M = 1500, K = 11008: 12 us).
#include "rq_mfma.h"
#include "rq_launch.h"
#include "rq_linear.h"
#include "rq_linear_dev.h"
#include "rq_lora.h"
#include "rq_pad.h"

#include <algorithm>

namespace rq {
namespace {

constexpr int kLgThreads = 256;
constexpr int kLgWaves = 4;
// columns per lane, by 16-rank blocks (1, 2, 4): with 64 ranks, eight columns'
// accumulators and the rows of two steps would not fit two waves per SIMD
constexpr int lg_cw(int jb) { return jb == 4 ? 4 : 8; }

struct GradTask {
  const uint16_t* src;  // [M][ld], cols columns (a multiple of 8, rows 16-byte aligned)
  int64_t ld;
  int64_t cols;
  const uint16_t* small;  // [r16][Mp]
  bool prescale;
  bool trans;           // partials as [rank][cols] (dA) instead of [cols][rank] (dB)
  float* part;          // [splits][cols * rank]
  int tiles;            // ceil(cols / (16 lg_cw))
};

struct GradArgs {
  GradTask t[2];
  int n;
  int64_t M, Mp;
  int rank;
  float scale;
  int splits;
  int64_t rows_per_split;  // multiple of 32
};

template <int CW>
struct RowPiece {
  uint32_t d[CW / 2];
};
template <int CW>
__device__ __forceinline__ RowPiece<CW> load_piece(const uint16_t* p) {
  RowPiece<CW> r;
  if constexpr (CW == 8) {
    const u32x4 v = *reinterpret_cast<const u32x4*>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) r.d[i] = v[i];
  } else {
    const u32x2 v = *reinterpret_cast<const u32x2*>(p);
    r.d[0] = v.x;
    r.d[1] = v.y;
  }
  return r;
}

// 8 consecutive rows' dwords d (columns 2 d, 2 d + 1) -> column h (0 low, 1
// high) as an operand: pairs of rows.
template <int CW>
__device__ __forceinline__ u32x4 column_operand(const RowPiece<CW> (&row)[8], int d, int h) {
  const uint32_t sel = h ? 0x07060302u : 0x05040100u;  // {hi, lo} halves: row 2i + 1 above row 2i
  u32x4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i) o[i] = __builtin_amdgcn_perm(row[2 * i + 1].d[d], row[2 * i].d[d], sel);
  return o;
}

template <int XT, int JB>
__global__ __launch_bounds__(kLgThreads) __attribute__((amdgpu_waves_per_eu(2))) void lora_grad_kernel(GradArgs a) {
  constexpr int CW = lg_cw(JB), kLgCols = 16 * CW;
  constexpr int kPitch = 16 * JB + 1;
  __shared__ float red[2][kLgCols][kPitch];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i16 = lane & 15, g4 = lane >> 4;
  int g = blockIdx.x;
  const int per0 = a.t[0].tiles * a.splits;
  const int which = g >= per0 ? 1 : 0;
  g -= which ? per0 : 0;
  const GradTask& T = a.t[which];
  // workgroups of an XCD (workgroup id mod 8) take adjacent column tiles, so
  // that the row pieces they read at a time are adjacent too
  const int n = T.tiles * a.splits;
  if (n % 8 == 0 && per0 % 8 == 0) g = (g & 7) * (n / 8) + (g >> 3);
  const int tile = g % T.tiles, sp = g / T.tiles;
  const int64_t c0 = int64_t(tile) * kLgCols;
  const int64_t mb = sp * a.rows_per_split;
  const int64_t me = mb + a.rows_per_split < a.M ? mb + a.rows_per_split : a.M;
  const bool pre = T.prescale;
  const int64_t col = c0 + CW * i16;
  const bool clive = col < T.cols;

  f32x4 acc[CW][JB];
#pragma unroll
  for (int c = 0; c < CW; ++c)
#pragma unroll
    for (int jb = 0; jb < JB; ++jb) acc[c][jb] = f32x4{0.f, 0.f, 0.f, 0.f};

  const uint16_t* sp0 = T.src + (clive ? col : 0);
  const uint16_t* sm = T.small + int64_t(i16) * a.Mp + 8 * g4;
  // rows past M and columns past the end read a live address and count as zero
  auto load = [&](RowPiece<CW> (&row)[8], u32x4 (&b)[JB], int64_t m0) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int64_t m = m0 + 8 * g4 + e;
      row[e] = load_piece<CW>(sp0 + (m < me ? m : 0) * T.ld);
    }
#pragma unroll
    for (int jb = 0; jb < JB; ++jb) b[jb] = *reinterpret_cast<const u32x4*>(sm + int64_t(16 * jb) * a.Mp + m0);
  };
  auto compute = [&](RowPiece<CW> (&row)[8], const u32x4 (&b)[JB], int64_t m0) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const bool live = clive && m0 + 8 * g4 + e < me;
#pragma unroll
      for (int d = 0; d < CW / 2; ++d) {
        uint32_t& w = row[e].d[d];
        w = live ? w : 0u;
        if (pre)
          w = cvt_pk<XT>(__fmul_rn(from_x16<XT>(w & 0xFFFFu), a.scale), __fmul_rn(from_x16<XT>(w >> 16), a.scale));
      }
    }
#pragma unroll
    for (int c = 0; c < CW; ++c) {
      const u32x4 op = column_operand<CW>(row, c >> 1, c & 1);
#pragma unroll
      for (int jb = 0; jb < JB; ++jb) acc[c][jb] = mfma16x16x32<XT>(op, b[jb], acc[c][jb]);
    }
  };
  // this wave's steps: rows mb + 32 (wave + 4 k), two in flight
  RowPiece<CW> r0[8], r1[8];
  u32x4 b0[JB], b1[JB];
  int64_t m = mb + 32 * wave;
  if (m < me) {
    load(r0, b0, m);
    for (;;) {
      const int64_t m1 = m + 32 * kLgWaves, m2 = m1 + 32 * kLgWaves;
      if (m1 < me) load(r1, b1, m1);
      compute(r0, b0, m);
      if (m1 >= me) break;
      if (m2 < me) load(r0, b0, m2);
      compute(r1, b1, m1);
      if (m2 >= me) break;
      m = m2;
    }
  }
  // waves summed as (0 + 2) + (1 + 3): acc[c][jb][r] of lane (i, g) is column
  // CW (4 g + r) + c, rank 16 jb + i
#pragma unroll
  for (int ph = 0; ph < 2; ++ph) {
    if ((wave >> 1) == 1 - ph) {
#pragma unroll
      for (int c = 0; c < CW; ++c)
#pragma unroll
        for (int jb = 0; jb < JB; ++jb)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float& o = red[wave & 1][CW * (4 * g4 + r) + c][16 * jb + i16];
            o = ph == 0 ? acc[c][jb][r] : __fadd_rn(acc[c][jb][r], o);
          }
    }
    __syncthreads();
  }
  const int cols = int(T.cols - c0 < kLgCols ? T.cols - c0 : kLgCols);
  float* part = T.part + int64_t(sp) * T.cols * a.rank;
  for (int i = tid; i < cols * a.rank; i += kLgThreads) {
    const int c = T.trans ? i % cols : i / a.rank, j = T.trans ? i / cols : i % a.rank;
    part[T.trans ? int64_t(j) * T.cols + c0 + c : (c0 + c) * a.rank + j] = __fadd_rn(red[0][c][j], red[1][c][j]);
  }
}

// Sums of the row splits in order, rounded to the activation dtype and written
// in the adapters' dtype (fp32, or the activation dtype): out[o] over `n` values,
// the live columns of rows of `cols` when the columns were padded.
struct GradOut {
  const float* part;
  int64_t n;         // partial values per split
  int64_t row;       // values per row of the partials
  int64_t live;      // live values per row
  int64_t live_rows;
  void* out;
};

template <int XT>
__global__ __launch_bounds__(256) void lora_grad_finish_kernel(GradOut o0, GradOut o1, int splits, int dt,
                                                               unsigned first1) {
  const bool second = blockIdx.x >= first1;
  const GradOut& o = second ? o1 : o0;
  const int64_t i = int64_t(blockIdx.x - (second ? first1 : 0u)) * 256 + threadIdx.x;
  if (i >= o.n) return;
  const int64_t r = i / o.row, c = i - r * o.row;
  if (r >= o.live_rows || c >= o.live) return;
  float v = 0.0f;
#pragma unroll 8
  for (int s = 0; s < splits; ++s) v = __fadd_rn(v, o.part[int64_t(s) * o.n + i]);
  v = round_x<XT>(v);
  store_from_f32(o.out, r * o.live + c, dt, v);
}

// out[m][j] = RND(sum of the K splits' partials in order) (j < R, zeros to
// R16) when given, and outt[j][m], zeros for M <= m < Mp, for one or two operands
// in one launch.  A thread takes 8 rows of one rank, four splits in flight.
struct FinishT {
  const float* part;
  int splits;
  uint16_t* out;
  uint16_t* outt;
};

template <int XT>
__global__ __launch_bounds__(256) void lora_finish_t_kernel(FinishT f0, FinishT f1, unsigned first1, int64_t M, int R,
                                                            int R16, int64_t Mp) {
  const bool second = blockIdx.x >= first1;
  const FinishT& f = second ? f1 : f0;
  const int64_t i = int64_t(blockIdx.x - (second ? first1 : 0u)) * 256 + threadIdx.x;
  const int64_t m8 = i / R16;
  const int j = int(i - m8 * R16);
  if (8 * m8 >= Mp) return;
  float v[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = 0.0f;
  if (j < R) {
    for (int k0 = 0; k0 < f.splits; k0 += 4) {
      float p[4][8];
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int64_t m = 8 * m8 + e;
          p[k][e] = f.part[(int64_t(k0 + k < f.splits ? k0 + k : 0) * M + (m < M ? m : M - 1)) * R + j];
        }
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (k0 + k < f.splits) v[e] = __fadd_rn(v[e], p[k][e]);
    }
  }
  uint32_t w[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float a = 8 * m8 + 2 * e < M ? v[2 * e] : 0.0f, b = 8 * m8 + 2 * e + 1 < M ? v[2 * e + 1] : 0.0f;
    w[e] = cvt_pk<XT>(a, b);
  }
  *reinterpret_cast<u32x4*>(f.outt + int64_t(j) * Mp + 8 * m8) = u32x4{w[0], w[1], w[2], w[3]};
  if (f.out) {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (8 * m8 + e < M) f.out[(8 * m8 + e) * R16 + j] = uint16_t(w[e >> 1] >> (16 * (e & 1)));
  }
}

template <int XT>
__global__ __launch_bounds__(kPadThreads) void pad_copy_kernel(PadCopies P) {
  pad_copy_block<XT>(P, blockIdx.x);
}

size_t up(size_t b) { return (b + 255) & ~size_t(255); }

struct GradPlan {
  int64_t Kp, Np, Mp, r16;
  int jb;             // 16-rank blocks of lora_grad_kernel: 1, 2 or 4
  bool pad_x, pad_y;  // the rows are copied (length not a multiple of 64)
  LoraRowsPlan lu, lg;
  int splits;
  int64_t rows_per_split;
  size_t lu_part, lg_part, s, ut, gt, x, y, pa, pb, a, bytes;
};

GradPlan plan_grads(int64_t M, int64_t K, int64_t N, int64_t rank, int cus) {
  GradPlan p{};
  p.Kp = ceil_div(K, 64) * 64;
  p.Np = ceil_div(N, 64) * 64;
  p.Mp = ceil_div(M, 32) * 32;
  p.r16 = ceil_div(rank, 16) * 16;
  p.jb = p.r16 <= 16 ? 1 : (p.r16 <= 32 ? 2 : 4);
  p.pad_x = p.Kp != K;
  p.pad_y = p.Np != N;
  p.lu = plan_lora_rows(M, p.Kp, rank, cus);
  p.lg = plan_lora_rows(M, p.Np, rank, cus);
  // about two workgroups per compute unit, every wave of a workgroup with at
  // least one step of 32 rows
  const int64_t cols = 16 * lg_cw(p.jb), tiles = ceil_div(p.Kp, cols) + ceil_div(p.Np, cols);
  int64_t s = std::max<int64_t>(2 * cus / tiles, 1);
  s = std::min(s, std::max<int64_t>(M / (32 * kLgWaves), 1));
  s = std::min<int64_t>(s, 16);
  p.rows_per_split = ceil_div(ceil_div(M, s), 32) * 32;
  p.splits = int(ceil_div(M, p.rows_per_split));
  size_t off = 0;
  auto take = [&](size_t b) {
    const size_t o = off;
    off += up(b);
    return o;
  };
  p.lu_part = take(p.lu.part_bytes);
  p.lg_part = take(p.lg.part_bytes);
  p.s = take(size_t(rank) * p.Np * 2);   // RND(B)^T rows
  p.a = p.pad_x ? take(size_t(rank) * p.Kp * 2) : 0;
  // operand rows for every rank block, written up to r16
  p.ut = take(size_t(16 * p.jb) * p.Mp * 2);
  p.gt = take(size_t(16 * p.jb) * p.Mp * 2);
  if (p.pad_x) p.x = take(size_t(M) * p.Kp * 2);
  if (p.pad_y) p.y = take(size_t(M) * p.Np * 2);
  p.pa = take(size_t(p.splits) * p.Kp * rank * 4);
  p.pb = take(size_t(p.splits) * p.Np * rank * 4);
  p.bytes = off;
  return p;
}

struct GradCall {
  const void* x;
  int64_t M, K, ldx;
  const void* dy;
  int64_t N, lddy;
  const void* a;
  const void* b;
  int64_t ldb;
  int lora_dt;
  int rank;
  float scale;
  void* da;
  void* db;
  uint16_t* g;  // [M][r16], or nullptr
};

template <int XT>
int run_grads(const GradCall& C, void* scratch, size_t bytes, hipStream_t stream) {
  const GradPlan p = plan_grads(C.M, C.K, C.N, C.rank, device_cus());
  if (!scratch || bytes < p.bytes) return RQ_ERR_WORKSPACE;
  if (!aligned(scratch, 256)) return RQ_ERR_BAD_ALIGNMENT;
  char* ws = static_cast<char*>(scratch);
  auto at16 = [&](size_t o) { return reinterpret_cast<uint16_t*>(ws + o); };
  auto atf = [&](size_t o) { return reinterpret_cast<float*>(ws + o); };
  int st = RQ_OK;
  const uint16_t* x = static_cast<const uint16_t*>(C.x);
  const uint16_t* dy = static_cast<const uint16_t*>(C.dy);
  int64_t ldx = C.ldx, lddy = C.lddy;
  const bool need_g = C.da || C.g, need_u = C.db != nullptr;
  const void* sa = C.a;
  int sa_dt = C.lora_dt;
  int64_t sa_j = C.K;
  PadCopies pc{};
  if (p.pad_x) {
    x = static_cast<const uint16_t*>(pc.add(C.x, XT, C.ldx, 1, C.M, C.K, C.M, p.Kp, ws + p.x));
    ldx = p.Kp;
    if (need_u) {
      sa = pc.add(C.a, C.lora_dt, C.K, 1, C.rank, C.K, C.rank, p.Kp, ws + p.a);
      sa_dt = XT;
      sa_j = p.Kp;
    }
  }
  if (p.pad_y) {
    dy = static_cast<const uint16_t*>(pc.add(C.dy, XT, C.lddy, 1, C.M, C.N, C.M, p.Np, ws + p.y));
    lddy = p.Np;
  }
  // g's factor S[j][n] = B[n][j] as contiguous 16-bit rows
  if (need_g) pc.add(C.b, C.lora_dt, 1, C.ldb, C.rank, C.N, C.rank, p.Np, ws + p.s);
  if (pc.blocks() > int64_t(INT32_MAX)) return RQ_ERR_UNSUPPORTED;
  if (pc.n > 0) {
    pad_copy_kernel<XT><<<unsigned(pc.blocks()), kPadThreads, 0, stream>>>(pc);
    if ((st = rq_check_launch()) != RQ_OK) return st;
  }
  FinishT f[2] = {};
  int nf = 0;
  if (need_g) {
    st = run_lora_rows_parts(XT, dy, lddy, C.M, p.Np, at16(p.s), XT, p.Np, 1, C.rank, true, C.scale, p.lg,
                             atf(p.lg_part), stream);
    if (st != RQ_OK) return st;
    f[nf++] = FinishT{atf(p.lg_part), p.lg.splits, C.g, at16(p.gt)};
  }
  if (need_u) {
    st = run_lora_rows_parts(XT, x, ldx, C.M, p.Kp, sa, sa_dt, sa_j, 1, C.rank, false, 1.0f, p.lu, atf(p.lu_part),
                             stream);
    if (st != RQ_OK) return st;
    f[nf++] = FinishT{atf(p.lu_part), p.lu.splits, nullptr, at16(p.ut)};
  }
  const unsigned fb = unsigned(ceil_div((p.Mp / 8) * p.r16, 256));
  lora_finish_t_kernel<XT><<<fb * nf, 256, 0, stream>>>(f[0], f[1], fb, C.M, C.rank, int(p.r16), p.Mp);
  if ((st = rq_check_launch()) != RQ_OK) return st;
  if (!C.da && !C.db) return RQ_OK;
  GradArgs a{};
  a.M = C.M;
  a.Mp = p.Mp;
  a.rank = C.rank;
  a.scale = C.scale;
  a.splits = p.splits;
  a.rows_per_split = p.rows_per_split;
  GradOut o[2] = {};
  if (C.db) {
    a.t[a.n] = GradTask{dy, lddy, p.Np, at16(p.ut), C.scale != 1.0f, false, atf(p.pb), int(ceil_div(p.Np, 16 * lg_cw(p.jb)))};
    o[a.n++] = GradOut{atf(p.pb), p.Np * C.rank, C.rank, C.rank, C.N, C.db};
  }
  if (C.da) {
    a.t[a.n] = GradTask{x, ldx, p.Kp, at16(p.gt), false, true, atf(p.pa), int(ceil_div(p.Kp, 16 * lg_cw(p.jb)))};
    o[a.n++] = GradOut{atf(p.pa), p.Kp * C.rank, p.Kp, C.K, C.rank, C.da};
  }
  const unsigned grid = unsigned((a.t[0].tiles + (a.n > 1 ? a.t[1].tiles : 0)) * p.splits);
  if (p.jb == 1) lora_grad_kernel<XT, 1><<<grid, kLgThreads, 0, stream>>>(a);
  else if (p.jb == 2) lora_grad_kernel<XT, 2><<<grid, kLgThreads, 0, stream>>>(a);
  else lora_grad_kernel<XT, 4><<<grid, kLgThreads, 0, stream>>>(a);
  if ((st = rq_check_launch()) != RQ_OK) return st;
  const unsigned b0 = unsigned(ceil_div(o[0].n, 256)), b1 = unsigned(ceil_div(o[1].n, 256));
  lora_grad_finish_kernel<XT><<<b0 + b1, 256, 0, stream>>>(o[0], o[1], p.splits, C.lora_dt, b0);
  return rq_check_launch();
}

}  // namespace
}  // namespace rq

extern "C" int rq_lora_grads_scratch_size(int x_dtype, int64_t M, int64_t K, int64_t N, int64_t rank,
                                          int64_t* bytes) {
  if (!bytes) return RQ_ERR_NULL_POINTER;
  if (!rq::valid_float_dtype(x_dtype)) return RQ_ERR_BAD_DTYPE;
  if (M < 0 || K < 1 || N < 1 || rank < 1) return RQ_ERR_BAD_SHAPE;
  *bytes = 0;
  if (x_dtype == RQ_DTYPE_F32 || rank > 64 || M == 0) return RQ_OK;
  *bytes = int64_t(rq::plan_grads(M, K, N, rank, rq::device_cus()).bytes);
  return RQ_OK;
}

extern "C" int rq_lora_grads(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx, const void* dy, int64_t N,
                             int64_t lddy, const void* lora_a, const void* lora_b, int64_t ld_lora_b, int lora_dtype,
                             int64_t rank, float scaling, void* da, void* db, void* g, void* scratch,
                             int64_t scratch_bytes, hipStream_t stream) {
  if (x_dtype != RQ_DTYPE_BF16 && x_dtype != RQ_DTYPE_F16) return RQ_ERR_BAD_DTYPE;
  if (lora_dtype != RQ_DTYPE_F32 && lora_dtype != x_dtype) return RQ_ERR_BAD_DTYPE;
  if (M < 1 || K < 1 || N < 1 || rank < 1 || ldx < K || lddy < N || ld_lora_b < rank) return RQ_ERR_BAD_SHAPE;
  if (rank > 64) return RQ_ERR_UNSUPPORTED;
  if (!da && !db && !g) return RQ_OK;
  if (!x || !dy || !lora_a || !lora_b) return RQ_ERR_NULL_POINTER;
  if (!rq::aligned(x, 2) || !rq::aligned(dy, 2)) return RQ_ERR_BAD_ALIGNMENT;
  if ((K % 64 == 0 && (!rq::aligned(x, 16) || ldx % 8 != 0)) ||
      (N % 64 == 0 && (!rq::aligned(dy, 16) || lddy % 8 != 0)))
    return RQ_ERR_BAD_ALIGNMENT;
  if (scratch_bytes < 0) return RQ_ERR_BAD_SHAPE;
  const rq::GradCall c{x, M, K, ldx, dy, N, lddy, lora_a, lora_b, ld_lora_b, lora_dtype, int(rank), scaling, da, db,
                       static_cast<uint16_t*>(g)};
  return x_dtype == RQ_DTYPE_BF16 ? rq::run_grads<RQ_DTYPE_BF16>(c, scratch, size_t(scratch_bytes), stream)
                                  : rq::run_grads<RQ_DTYPE_F16>(c, scratch, size_t(scratch_bytes), stream);
}
