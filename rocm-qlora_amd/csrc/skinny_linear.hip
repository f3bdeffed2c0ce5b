// NF4 linears for a few tens of activation rows (batched decode, short prompts),
// 16-bit activations:
//   y = RND(RND(x W^T + RND(bias)) + RND(RND(RND(u) RND(B)^T) * scaling))
// with W = RND(T[code] * scale), as the decode GEMV and the GEMM compute it.
//
// A workgroup of sixteen waves takes 256 weight rows (16 per wave) and a K split
// of up to U segments of 256 k, for all of up to 64 activation rows.  The split's
// activations ([k / 64][row][128 bytes], swizzled) are brought into LDS whole by
// direct-to-LDS loads, the waves' weights into registers right behind them, the
// pair table is filled while they fly, and after one barrier every wave runs
// through its weights on its own: each weight is decoded once for all rows (the
// GEMM's 256 x 128 tiles pad 17-64 rows to 256 and give few workgroups).  MFMA
// 16x16x32 with the weights as the A operand, so a lane's four results run along
// an output row.
//
// Splits store their fp32 tiles with device-coherent stores; the last one of a
// workgroup column to count itself sums them in split order, adds bias and LoRA
// term and stores (the same bits whichever is last).
//
// Bound by latencies in a row (loads, decode, split exchange, epilogue; about 12 us
// with one segment per split) and the exact decode, about four VALU operations
// and one 8-byte LDS read per code byte as in the GEMV (4 us for 4 segments).
// Without LoRA, M = 48: 4096 -> 14336 24 us, 14336 -> 4096 31 us, 4096 -> 4096
// 18 us; the 256 x 128 GEMM takes 46, 65 and 29 us.
#include "rq_gemm_core.h"
#include "rq_skinny.h"

#include <algorithm>

namespace rq {
namespace {

constexpr int kSkThreads = 1024;
constexpr int kSkWaves = 16;
constexpr int kSkRows = 64;                 // activation rows, at most
constexpr int kSkSeg = 256;                 // k per segment
constexpr int kSkLds = 160 * 1024;
constexpr int kSkXBytes = kSkLds - kLutBytes;  // activations
constexpr int kSkUPitch = 72;               // LoRA operand row pitch (elements)

// segments per split: 4 (the activations of 48 rows in kSkXBytes; a wave's
// weights wait in registers), or 2
static_assert(4 * 4 * 48 * 128 <= kSkXBytes && 2 * 4 * 64 * 128 <= kSkXBytes, "LDS plan");

struct SkArgs {
  const uint16_t* x;
  int64_t ldx;
  const uint8_t* w;
  int64_t M, N, K;
  int64_t row_bytes;
  int64_t blocks_per_row;
  int bs_log2;
  int groups, splits, nseg;
  float* part;
  uint32_t* cnt;
  // the LoRA operand inside the launch (la set): this split's part of x . RND(A)^T,
  // summed over the workgroup's waves and stored to upart [groups][splits][rank
  // blocks of 16][16][16 MB rows]; A [rank][K], rows 16-byte aligned
  const void* la;
  int la_dt;
  float* upart;
};

struct SkEpi {
  const void* bias;
  int bias_dt;
  int rank;
  const float* u;  // [u_splits][M][rank]
  int u_splits;
  const void* b;   // [N][ldb]
  int64_t ldb;
  int b_dt;
  bool b_vec;
  float scaling;
  uint16_t* y;
  int64_t ldy;
};

// A unit is 16 rows x 256 k of a wave; lane (i, q) = (lane % 16, lane / 16) owns row
// i.  Its steps are MFMAs of 32 k, 8 consecutive k per
// lane; piece(s), chunk(s, q): where step s's k lie in the activations' 64-k
// pieces of 8 chunks.
template <int XT, class Scale>
struct UnitNF4 {
  static constexpr int kLoads = 2 + 2 * Scale::kLoads;
  u32x4 w[2];                    // k = 32 q + 128 h + [0, 32)
  typename Scale::Raw s[2];
  __device__ __forceinline__ void load(const SkArgs& a, const Scale& sc, __amdgpu_buffer_rsrc_t r, int64_t n, int q,
                                       int64_t k0) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      int64_t k = k0 + 128 * h + 32 * q;
      k = k < a.K ? k : a.K - 32;  // past K: a live address, its products are dropped
      w[h] = buf_load16(r, uint32_t(n * a.row_bytes + (k >> 1)));
      s[h] = sc.load(n * a.blocks_per_row + (k >> a.bs_log2));
      asm volatile("" ::: "memory");  // one load per scale, as kLoads counts
    }
  }
  __device__ __forceinline__ u32x4 operand(const Scale& sc, const u32x2* lut, uint32_t lane_off, int st) const {
    return expand8_scaled<XT>(lut, w[st >> 2][st & 3], lane_off, sc.value(s[st >> 2]));
  }
  __device__ static __forceinline__ int piece(int st, int q) { return 2 * (st >> 2) + (q >> 1); }
  __device__ static __forceinline__ int chunk(int st, int q) { return 4 * (q & 1) + (st & 3); }
};

template <int XT, class Scale, int MB, int U>
__global__ __launch_bounds__(kSkThreads) __attribute__((amdgpu_waves_per_eu(4, 4)))
void skinny_kernel(SkArgs a, Scale scale, SkEpi e) {
  using Unit = UnitNF4<XT, Scale>;
  constexpr int kXRows = 16 * MB, kPiece = kXRows * 128;
  __shared__ __attribute__((aligned(16))) uint8_t lds[kSkLds];
  u32x2* lut = reinterpret_cast<u32x2*>(lds);
  uint8_t* xs = lds + kLutBytes;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i16 = lane & 15, q = lane >> 4;
  const int group = blockIdx.x % a.groups, split = blockIdx.x / a.groups;
  const int64_t n0 = (int64_t(group) * kSkWaves + wave) * 16;
  const int seg0 = int(int64_t(a.nseg) * split / a.splits);
  const int nu = int(int64_t(a.nseg) * (split + 1) / a.splits) - seg0;  // <= U
  const int64_t kbeg = int64_t(seg0) * kSkSeg;

  // activations: piece p (64 k), rows 8 j + lane / 8, chunk swizzled
  {
    const int pieces = int((a.K - kbeg < int64_t(nu) * kSkSeg ? a.K - kbeg : int64_t(nu) * kSkSeg) / 64);
    for (int t = wave; t < 4 * U * 2 * MB; t += kSkWaves) {
      const int p = t / (2 * MB), j = t - p * (2 * MB);
      const int r = 8 * j + (lane >> 3);
      int64_t m = r;
      m = m < a.M ? m : a.M - 1;                // rows past M: a live row, never stored
      const int pl = p < pieces ? p : pieces - 1;  // pieces past K: a live piece, never used
      const uint32_t off =
          uint32_t(m * a.ldx + kbeg + 64 * pl) * 2u + uint32_t(16 * ((lane & 7) ^ ((r >> 1) & 7)));
      dma16(a.x, off, __builtin_amdgcn_readfirstlane(uint32_t(kLutBytes + p * kPiece + j * 1024)));
    }
  }
  // weights: all of this wave's units
  int64_t n = n0 + i16;
  n = n < a.N ? n : a.N - 1;
  const __amdgpu_buffer_rsrc_t wr = buffer_rsrc(a.w, uint32_t(a.N * a.row_bytes));
  Unit un[U];
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < U; ++u) un[u].load(a, scale, wr, n, q, kbeg + int64_t(u < nu ? u : nu - 1) * kSkSeg);
  __builtin_amdgcn_sched_barrier(0);
  fill_f32pair_lut<kSkThreads>(lut, tid);
  // the activation loads are older than the U * kLoads weight loads
  step_barrier<U * Unit::kLoads>();

  // LoRA operand: the split's 32-k steps t = wave, wave + 16, ...; the first rank
  // block's values of A are requested here, under the units
  constexpr int kUSteps = U / 2;
  const int rank = e.rank, nsteps = 8 * nu;
  u32x4 a_lo[kUSteps], a_hi[kUSteps];
  auto a_load = [&](int jb) {
#pragma unroll
    for (int t = 0; t < kUSteps; ++t) {
      const int j = 16 * jb + i16;
      int64_t k = kbeg + 32 * (wave + kSkWaves * t) + 8 * q;
      k = k < a.K ? k : a.K - 8;
      const int64_t off = int64_t(j < rank ? j : rank - 1) * a.K + k;
      const uint8_t* p = static_cast<const uint8_t*>(a.la) + off * (a.la_dt == RQ_DTYPE_F32 ? 4 : 2);
      a_lo[t] = *reinterpret_cast<const u32x4*>(p);
      a_hi[t] = *reinterpret_cast<const u32x4*>(p + (a.la_dt == RQ_DTYPE_F32 ? 16 : 0));
    }
  };
  if (a.la) a_load(0);

  f32x4 acc[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) acc[mb] = f32x4{0.f, 0.f, 0.f, 0.f};
  const uint32_t lane_off = uint32_t(lane & 31) * 8u;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (u < nu) {
      const int64_t k0 = kbeg + int64_t(u) * kSkSeg;
      const bool whole = k0 + kSkSeg <= a.K;
#pragma unroll
      for (int st = 0; st < 8; ++st) {
        u32x4 wv = un[u].operand(scale, lut, lane_off, st);
        const int pc = Unit::piece(st, q);
        const uint8_t* xp = xs + (4 * u + pc) * kPiece + i16 * 128 + ((Unit::chunk(st, q) ^ ((i16 >> 1) & 7)) << 4);
        u32x4 xv[MB];
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) xv[mb] = *reinterpret_cast<const u32x4*>(xp + mb * 2048);
        if (!whole) {  // lanes past K multiply zeros
          const bool live = k0 + 64 * pc < a.K;
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            wv[c] = live ? wv[c] : 0u;
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) xv[mb][c] = live ? xv[mb][c] : 0u;
          }
        }
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[mb] = mfma16x16x32<XT>(wv, xv[mb], acc[mb]);
      }
    }
  }

  // ---- this split's part of u: every workgroup of a column group needs all of u
  // at its end, so each computes it for its own K split beside its tiles, and the
  // split exchange below carries it (a launch of its own before this one took 4.5
  // us and a gap, and its partials 2 us of the epilogue)
  float* const up = a.upart + (int64_t(group) * a.splits + split) * (((rank + 15) / 16) * 16 * kXRows);
  if (a.la) {
    f32x4* red = reinterpret_cast<f32x4*>(lds);  // [16 waves][MB][64 lanes], over the table
    static_assert(kSkWaves * 4 * 64 * 16 <= kLutBytes, "u reduction");
    for (int jb = 0; 16 * jb < rank; ++jb) {
      if (jb > 0) a_load(jb);
      f32x4 ua[MB];
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) ua[mb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < kUSteps; ++t) {
        const int st = wave + kSkWaves * t;
        if (st < nsteps) {
          const bool live = kbeg + 32 * st + 8 * q < a.K;
          u32x4 av = raw8_to_x<XT>(a_lo[t], a_hi[t], a.la_dt);
          const uint8_t* xp = xs + (st >> 1) * kPiece + i16 * 128 + (((4 * (st & 1) + q) ^ ((i16 >> 1) & 7)) << 4);
#pragma unroll
          for (int c = 0; c < 4; ++c) av[c] = live ? av[c] : 0u;
#pragma unroll
          for (int mb = 0; mb < MB; ++mb) {
            u32x4 xv = *reinterpret_cast<const u32x4*>(xp + mb * 2048);
#pragma unroll
            for (int c = 0; c < 4; ++c) xv[c] = live ? xv[c] : 0u;
            ua[mb] = mfma16x16x32<XT>(av, xv, ua[mb]);
          }
        }
      }
      __syncthreads();  // the table (or the last block's sums) is no longer read
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) red[(wave * MB + mb) * 64 + lane] = ua[mb];
      __syncthreads();
      // value (rank 4 q + r, row 16 mb + i) of lane (i, q): summed in wave order
      for (int idx = tid; idx < 256 * MB; idx += kSkThreads) {
        const float* r = reinterpret_cast<const float*>(red) + idx;
        float v = 0.0f;
#pragma unroll
        for (int w = 0; w < kSkWaves; ++w) v = __fadd_rn(v, r[w * 256 * MB]);
        const int mb = idx >> 8, l = (idx >> 2) & 63, j = 16 * jb + 4 * (l >> 4) + (idx & 3);
        __hip_atomic_store(&up[j * kXRows + 16 * mb + (l & 15)], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }

  // The epilogue's first operands, requested before the splits' tiles so that the
  // round trips overlap: up to 16 parts of the thread's first u value and the
  // first 8 ranks of its column's B row, raw.  In-launch u: the splits' parts, rows
  // contiguous; else the row kernel's partials, ranks contiguous.
  const int r16 = (rank + 15) / 16 * 16, live = r16 * kXRows;
  const int64_t ustep = a.la ? int64_t(live) : a.M * rank;
  const int ns = a.la ? a.splits : e.u_splits;
  auto u_index = [&](int idx, int& j, int& m) {
    const bool rows = a.la || idx >= live;
    j = rows ? idx / kXRows : idx % r16;
    m = rows ? idx % kXRows : idx / r16;
    return j < rank && m < a.M;
  };
  auto u_load = [&](float (&t)[16], int idx, int j, int m, int s0) {
    const float* p = a.la ? a.upart + int64_t(group) * ns * live + idx : e.u + m * rank + j;
#pragma unroll
    for (int s = 0; s < 16; ++s)
      if (s0 + s < ns) t[s] = __hip_atomic_load(p + int64_t(s0 + s) * ustep, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  float ut[16];
  u32x4 b_lo = {0u, 0u, 0u, 0u}, b_hi = {0u, 0u, 0u, 0u};
  const bool b_pre = e.b_vec && 8 * q + 8 <= rank && (e.b_dt == RQ_DTYPE_F32 || e.ldb % 8 == 0);
  auto pre_load = [&]() {
    if (rank <= 0) return;
    int j, m;
    if (tid < kXRows * 64 && u_index(tid, j, m)) u_load(ut, tid, j, m, 0);
    if (b_pre) {
      const uint8_t* p = static_cast<const uint8_t*>(e.b) + (n * e.ldb + 8 * q) * (e.b_dt == RQ_DTYPE_F32 ? 4 : 2);
      b_lo = *reinterpret_cast<const u32x4*>(p);
      b_hi = *reinterpret_cast<const u32x4*>(p + (e.b_dt == RQ_DTYPE_F32 ? 16 : 0));
    }
  };

  if (a.splits > 1) {
    // tile (16 rows of this wave) x split: MB x 64 lanes x 16 bytes
    uint8_t* base = reinterpret_cast<uint8_t*>(a.part) + (int64_t(group) * kSkWaves + wave) * a.splits * (MB * 1024);
    const __amdgpu_buffer_rsrc_t part = buffer_rsrc(base, uint32_t(a.splits * MB * 1024));
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
      buf_store16_coherent(part, uint32_t(lane) * 16u, uint32_t((split * MB + mb) * 1024),
                           u32x4{f2u(acc[mb][0]), f2u(acc[mb][1]), f2u(acc[mb][2]), f2u(acc[mb][3])});
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    uint32_t* flag = reinterpret_cast<uint32_t*>(lds);
    if (tid == 0) {
      const uint32_t old = __hip_atomic_fetch_add(&a.cnt[group], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const bool last = old == uint32_t(a.splits - 1);
      if (last) __hip_atomic_store(&a.cnt[group], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *flag = last ? 1u : 0u;
    }
    __syncthreads();
    const uint32_t last = __builtin_amdgcn_readfirstlane(*flag);
    __syncthreads();
    if (!last) return;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[mb] = f32x4{0.f, 0.f, 0.f, 0.f};
    pre_load();
    constexpr int kFly = MB == 4 ? 4 : (MB == 3 ? 5 : 8);  // splits' tiles in flight
    for (int s0 = 0; s0 < a.splits; s0 += kFly) {
      u32x4 v[kFly][MB];
#pragma unroll
      for (int s = 0; s < kFly; ++s)
        if (s0 + s < a.splits)
#pragma unroll
          for (int mb = 0; mb < MB; ++mb)
            v[s][mb] = buf_load16_coherent(part, uint32_t(lane) * 16u, uint32_t(((s0 + s) * MB + mb) * 1024));
#pragma unroll
      for (int s = 0; s < kFly; ++s)
        if (s0 + s < a.splits)
#pragma unroll
          for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[mb][r] = __fadd_rn(acc[mb][r], u2f(v[s][mb][r]));
    }
  } else {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // u's stores, read below by other waves
    __syncthreads();  // the activations' and table's LDS is free
    pre_load();
  }

  // ---- epilogue: acc[mb][r] of lane (i, q) is row 16 mb + i, column n0 +
  // 4 q + r
  f32x4 lo[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) lo[mb] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (rank > 0) {
    uint16_t* us = reinterpret_cast<uint16_t*>(lds);  // RND(u) [16 MB][kSkUPitch], zero padded to 64 ranks
    for (int idx = tid; idx < kXRows * 64; idx += kSkThreads) {
      int j, m;
      float v = 0.0f;
      if (u_index(idx, j, m)) {
        for (int s0 = 0; s0 < ns; s0 += 16) {
          if (idx != tid || s0 > 0) u_load(ut, idx, j, m, s0);
#pragma unroll
          for (int s = 0; s < 16; ++s)
            if (s0 + s < ns) v = __fadd_rn(v, ut[s]);
        }
      }
      us[m * kSkUPitch + j] = uint16_t(to_x16<XT>(v));
    }
    __syncthreads();
    for (int j0 = 0; j0 < rank; j0 += 32) {
      const int left = rank - j0 - 8 * q;
      u32x4 bv = {0u, 0u, 0u, 0u};
      if (j0 == 0 && b_pre) bv = raw8_to_x<XT>(b_lo, b_hi, e.b_dt);
      else if (left > 0) bv = load_a8_masked<XT>(e.b, e.b_dt, n * e.ldb + j0 + 8 * q, left, e.b_vec);
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
        lo[mb] = mfma16x16x32<XT>(
            bv, *reinterpret_cast<const u32x4*>(us + (16 * mb + i16) * kSkUPitch + j0 + 8 * q), lo[mb]);
    }
  }
  const bool vec = (reinterpret_cast<uintptr_t>(e.y) & 7u) == 0 && (e.ldy & 3) == 0;
  const int64_t nn = n0 + 4 * q;
  float bias[4];
#pragma unroll
  for (int r = 0; r < 4; ++r)
    bias[r] = e.bias && nn + r < a.N ? round_x<XT>(load_as_f32(e.bias, nn + r, e.bias_dt)) : -0.0f;
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int64_t m = 16 * mb + i16;
    float v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      v[r] = round_x<XT>(__fadd_rn(acc[mb][r], bias[r]));
      if (rank > 0) v[r] = __fadd_rn(v[r], round_x<XT>(__fmul_rn(round_x<XT>(lo[mb][r]), e.scaling)));
    }
    const uint32_t p0 = cvt_pk<XT>(v[0], v[1]), p1 = cvt_pk<XT>(v[2], v[3]);
    if (m >= a.M) continue;
    uint16_t* yp = e.y + m * e.ldy + nn;
    if (vec && nn + 4 <= a.N) {
      *reinterpret_cast<u32x2*>(yp) = u32x2{p0, p1};
    } else {
      const uint16_t o[4] = {uint16_t(p0), uint16_t(p0 >> 16), uint16_t(p1), uint16_t(p1 >> 16)};
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (nn + r < a.N) yp[r] = o[r];
    }
  }
}

struct SkPlan {
  int mb, units, groups, nseg, splits;
  LoraRowsPlan lr;
  size_t part_off, u_off, bytes;
};

SkPlan plan_skinny(int64_t M, int64_t N, int64_t K, int64_t rank, int cus) {
  SkPlan p{};
  const int64_t mb = M > 48 ? 4 : (M > 32 ? 3 : 2);
  p.mb = int(mb);
  p.groups = int(ceil_div(N, 16 * kSkWaves));
  p.nseg = int(ceil_div(K, kSkSeg));
  // Four segments per split halve the exchange and the table fills, two double
  // the workgroups (M = 48, without LoRA: 4096 -> 4096 22.0 us with four, 17.9
  // with two; 4096 -> 14336 24.1 and 28.5; 14336 -> 4096 31.2 and 39.0); 64 rows
  // of four segments do not fit the LDS.
  p.units = mb < 4 && 2 * int64_t(p.groups) * ceil_div(p.nseg, 4) >= cus ? 4 : 2;
  p.splits = int(ceil_div(p.nseg, p.units));
  if (rank > 0) {
    p.lr = plan_lora_rows(M, K, rank, cus);
    p.part_off = p.lr.part_bytes;
  }
  p.u_off = p.part_off;
  if (p.splits > 1) p.u_off += size_t(p.groups) * kSkWaves * p.splits * p.mb * 1024;
  p.bytes = p.u_off;
  if (rank > 0) p.bytes += size_t(p.groups) * p.splits * (ceil_div(rank, 16) * 16) * (16 * p.mb) * 4;
  return p;
}

template <int XT, class Scale>
int launch_skinny(const SkArgs& a, Scale scale, const SkEpi& e, const SkPlan& p, hipStream_t stream) {
  const unsigned grid = unsigned(p.groups * p.splits);
  if (p.mb == 4) skinny_kernel<XT, Scale, 4, 2><<<grid, kSkThreads, 0, stream>>>(a, scale, e);
  else if (p.mb == 3 && p.units == 4)
    skinny_kernel<XT, Scale, 3, 4><<<grid, kSkThreads, 0, stream>>>(a, scale, e);
  else if (p.mb == 3) skinny_kernel<XT, Scale, 3, 2><<<grid, kSkThreads, 0, stream>>>(a, scale, e);
  else if (p.units == 4) skinny_kernel<XT, Scale, 2, 4><<<grid, kSkThreads, 0, stream>>>(a, scale, e);
  else skinny_kernel<XT, Scale, 2, 2><<<grid, kSkThreads, 0, stream>>>(a, scale, e);
  return rq_check_launch();
}

template <int XT>
int launch_scale(const SkArgs& a, const void* s, int sdt, const uint8_t* c2, int c2_format, int64_t block2,
                 const SkEpi& e, const SkPlan& p, hipStream_t stream) {
  if (c2) {
    const int sh = pow2_shift(block2);
    switch (sdt) {
      case RQ_DTYPE_F32:
        return launch_skinny<XT>(a, ScaleDQ<RQ_DTYPE_F32>{c2, s, c2_format, sh, block2}, e, p, stream);
      case RQ_DTYPE_BF16:
        return launch_skinny<XT>(a, ScaleDQ<RQ_DTYPE_BF16>{c2, s, c2_format, sh, block2}, e, p, stream);
      default:
        return launch_skinny<XT>(a, ScaleDQ<RQ_DTYPE_F16>{c2, s, c2_format, sh, block2}, e, p, stream);
    }
  }
  switch (sdt) {
    case RQ_DTYPE_F32: return launch_skinny<XT>(a, ScaleAbsmax<RQ_DTYPE_F32>{s}, e, p, stream);
    case RQ_DTYPE_BF16: return launch_skinny<XT>(a, ScaleAbsmax<RQ_DTYPE_BF16>{s}, e, p, stream);
    default: return launch_skinny<XT>(a, ScaleAbsmax<RQ_DTYPE_F16>{s}, e, p, stream);
  }
}

}  // namespace

// Bounded by the bytes the splits exchange: they are written and read once beside
// the weight, 0.19 N K of them at up to 48 rows and 0.5 N K at 64 (the packed weight
// is 0.5 N K).  Against the fused GEMM, us: 4096 -> 128256 48 rows 159 / 268 (100 MB),
// 64 rows 235 / 267 and with LoRA 281 / 287 (266 MB); 14336 -> 14336 64 rows 95 / 107
// and 113 / 117 (104 MB); 4096 -> 14336 31 / 41.
constexpr size_t kSkMaxScratch = size_t(128) << 20;

bool skinny_takes(int64_t M, int64_t N, int64_t K, int64_t rank) {
  // 32-bit offsets into weights and activations are the callers' fast-path checks
  return M > kGemvMaxM && M <= kSkRows && rank <= 64 && K % 64 == 0 && double(N) * double(K) < 8.58e9 &&
         plan_skinny(M, N, K, rank, device_cus()).bytes <= kSkMaxScratch;
}

size_t skinny_scratch(int64_t M, int64_t N, int64_t K, int64_t rank) {
  return plan_skinny(M, N, K, rank, device_cus()).bytes;
}

size_t skinny_counters(int64_t M, int64_t N, int64_t K) {
  const SkPlan p = plan_skinny(M, N, K, 0, device_cus());
  return p.splits > 1 ? size_t(p.groups) : 0;
}

int run_skinny_nf4(const LinearArgs& L, void* scratch, size_t bytes, uint32_t* cnt, hipStream_t stream) {
  const SkPlan p = plan_skinny(L.M, L.N, L.K, L.rank, device_cus());
  if (p.bytes > 0 && (!scratch || bytes < p.bytes || !aligned(scratch, 256))) return RQ_ERR_WORKSPACE;
  SkEpi e{};
  bool u_in = false;
  e.bias = L.bias;
  e.bias_dt = L.bias_dtype;
  e.y = static_cast<uint16_t*>(L.y);
  e.ldy = L.ldy;
  if (L.rank > 0) {
    float* u = static_cast<float*>(scratch);
    // the operand inside the launch when the adapter reads x itself
    u_in = L.lora_x == L.x && L.ld_lora_x == L.ldx && aligned(L.lora_a, 16);
    const int st = u_in ? RQ_OK
                        : run_lora_rows_parts(L.x_dtype, static_cast<const uint16_t*>(L.lora_x), L.ld_lora_x, L.M, L.K,
                                              L.lora_a, L.lora_dtype, L.K, 1, int(L.rank), false, 1.0f, p.lr, u, stream);
    if (st != RQ_OK) return st;
    e.rank = int(L.rank);
    e.u = u;
    e.u_splits = p.lr.splits;
    e.b = L.lora_b;
    e.ldb = L.ld_lora_b;
    e.b_dt = L.lora_dtype;
    e.b_vec = aligned(L.lora_b, 16) && (L.lora_dtype != RQ_DTYPE_F32 || L.ld_lora_b % 4 == 0);
    e.scaling = L.scaling;
  }
  SkArgs a{};
  a.x = static_cast<const uint16_t*>(L.x);
  a.ldx = L.ldx;
  a.w = L.w_packed;
  a.M = L.M;
  a.N = L.N;
  a.K = L.K;
  a.row_bytes = L.K / 2;
  a.blocks_per_row = L.K / L.block_size;
  a.bs_log2 = pow2_shift(L.block_size);
  a.groups = p.groups;
  a.splits = p.splits;
  a.nseg = p.nseg;
  a.part = reinterpret_cast<float*>(static_cast<char*>(scratch) + p.part_off);
  a.cnt = cnt;
  if (u_in) {
    a.la = L.lora_a;
    a.la_dt = L.lora_dtype;
    a.upart = reinterpret_cast<float*>(static_cast<char*>(scratch) + p.u_off);
  }
  auto launch = L.x_dtype == RQ_DTYPE_BF16 ? launch_scale<RQ_DTYPE_BF16> : launch_scale<RQ_DTYPE_F16>;
  return launch(a, L.absmax, L.absmax_dtype, L.c2, L.c2_format, L.block2, e, p, stream);
}

}  // namespace rq
