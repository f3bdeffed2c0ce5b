// Dense MFMA GEMM for gfx950: out[M, N] = X[M, K] . W[N, K]^T with the
// quantized linears' epilogue (bias, LoRA term, the reference's roundings),
// where W is the weight RND(W_deq) that a launch before it wrote into scratch
// memory (dense_gemm.hip), as W rows (forward) or W^T rows (dX).  bf16 and
// fp16 (v_mfma_f32_32x32x16), and fp32 (v_mfma_f32_32x32x2_f32, 128 x 128
// tiles only, everything in fp32).
//
// Tile 256 x 256 (HALVES = 2) or 128 x 128 (HALVES = 1), 64 k per step,
// eight waves, two per SIMD: wave (wr, wc) = (wave / 4, wave % 4) owns rows
// 64 wr .. + 63 and columns 32 wc .. + 31 of each 128 x 128 quadrant as two
// blocks of v_mfma_f32_32x32x16 (weights as the A operand, so a lane's
// results run along an output row).  A phase is one quadrant's eight MFMAs
// (256 cycles) behind that phase's LDS reads and direct-to-LDS loads; the two
// waves of a SIMD run one phase slot apart (an extra barrier delays waves 4-7
// once), so one issues MFMAs while the other reads.  Both operands come by
// global_load_lds in half tiles of 128 rows x 64 k (16 KiB, 128-byte rows,
// swizzled as the activation ring of rq_gemm8.h); a half tile is refilled as
// soon as every wave has read it, 1.5 to 2 steps ahead of its next use, and
// the waits leave the younger half tiles in flight (vmcnt 12 of 16).
//
// What bounds it: power first, then the loop.  4096 x 4096 x 14336, launches in a
// row: with N(0, 1) operands 367 to 517 us as the clock drops (1.31 to 0.93
// PFLOP/s), with zero operands (no toggling) 283 to 308 us throughout (1.70 to 1.56,
// two thirds of the dense peak).  The fused eight-wave kernel it replaces for many rows
// (nf4_gemm8_kernel), which dequantizes each weight tile again for every 256
// activation rows, reached 0.89 PFLOP/s.
#pragma once
#include "rq_gemm_core.h"

namespace rq {

constexpr int kDnThreads = 512;
constexpr int kDnHalf = 128 * 128;  // bytes of a half tile: 128 rows x 64 k

// Element bytes of an operand type, and the elements of one k step (128-byte
// rows).
template <int XT>
struct DnEl {
  static constexpr int kSize = XT == RQ_DTYPE_F32 ? 4 : 2;
  static constexpr int kStep = 128 / kSize;
  static constexpr int kRankPad = XT == RQ_DTYPE_F32 ? 8 : 16;  // one LoRA epilogue step
};

// LDS: two buffers of X0 X1 W0 W1 (256 x 256 tiles), or four of X W (128 x
// 128); the epilogue stages the output tile in it (16-byte padded rows).
template <int XT, int HALVES>
struct DnTile {
  static constexpr int kB = 128 * HALVES;           // tile rows and columns
  static constexpr int kBuf = 2 * HALVES * kDnHalf;  // one k step
  static constexpr int kBufs = 4 / HALVES;
  static constexpr int kOutPitch = kB * DnEl<XT>::kSize + 16;
  static constexpr int kLds = kB * kOutPitch > kBufs * kBuf ? kB * kOutPitch : kBufs * kBuf;
  static_assert(kLds <= 160 * 1024, "LDS plan");
};

struct DenseGemmArgs {
  const void* x;  // [M][ldx]
  const void* w;  // [N][ldw]
  int64_t ldx, ldw;
  int64_t M, N;
  int nk;             // k steps of 128 bytes (the operands are zero past K)
  int tiles_m, tiles_n;
  int whole;          // tiles run whole; the other tiles - whole run as `splits` workgroups
  int splits;
  float* part;         // [splits][split tiles][32 x 512 x 4]
  uint32_t* tile_cnt;  // [split tiles], zero before the launch and after it
};

struct DenseEpi {
  const void* bias;
  int bias_dt;
  int rankp;           // LoRA rank rounded up to kRankPad (0: none)
  const void* u;       // [M][rankp]
  const void* b;       // [N][rankp]
  float scaling;
  const uint8_t* mask;  // dX with LoRA dropout
  int64_t ldm;
  float mask_scale;
  void* y;
  int64_t ldy;
};

// RND: rounding to the result type (none for fp32)
template <int XT>
__device__ __forceinline__ void dn_round2(float& x, float& y) {
  if constexpr (XT != RQ_DTYPE_F32) round2<XT>(x, y);
}

// The products of one 16-byte operand chunk pair per lane: 8 16-bit values (one
// MFMA), or 4 fp32 values (four 32x32x2 MFMAs; lanes 0-31 and 32-63 hold
// different k in both operands alike, so any order of k serves).
template <int XT>
__device__ __forceinline__ f32x16 dn_mfma(const u32x4& w, const u32x4& x, f32x16 c) {
  if constexpr (XT == RQ_DTYPE_F32) {
#pragma unroll
    for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_32x32x2f32(u2f(w[j]), u2f(x[j]), c, 0, 0, 0);
    return c;
  } else {
    return mfma32x32x16<XT>(w, x, c);
  }
}

template <int XT, int HALVES>
__global__ __launch_bounds__(kDnThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void dense_gemm_kernel(DenseGemmArgs a, DenseEpi e) {
  using Tile = DnTile<XT, HALVES>;
  constexpr int ES = DnEl<XT>::kSize;
  constexpr int H = HALVES, kBuf = Tile::kBuf, kOutPitch = Tile::kOutPitch;
  __shared__ __attribute__((aligned(16))) uint8_t lds[Tile::kLds];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wave >> 2, wc = wave & 3;
  const int i32 = lane & 31, q = lane >> 5;

  // tile of this workgroup
  const int T = a.tiles_m * a.tiles_n;
  int g = blockIdx.x, split = 0, nsplit = 1, ti = 0;
  if (g >= a.whole) {
    const int lt = T - a.whole, r = g - a.whole;
    nsplit = a.splits;
    split = r / lt;
    ti = r - split * lt;
    g = a.whole + ti;
  }
  int mt, nt;
  {
    // XCD x = workgroup % 8 takes a contiguous run of tiles when the count
    // divides, in groups of 4 row tiles walked column by column
    int t = g;
    const int n8 = (g < a.whole ? a.whole : T - a.whole) / 8, base = g < a.whole ? 0 : a.whole;
    if (n8 * 8 == (g < a.whole ? a.whole : T - a.whole)) {
      const int l = g - base;
      t = base + (l & 7) * n8 + (l >> 3);
    }
    constexpr int GM = 4;
    const int per = GM * a.tiles_n, grp = t / per, r = t - grp * per;
    const int gm = a.tiles_m - grp * GM < GM ? a.tiles_m - grp * GM : GM;
    mt = grp * GM + r % gm;
    nt = r / gm;
  }
  const int64_t m0 = int64_t(mt) * Tile::kB, n0 = int64_t(nt) * Tile::kB;
  const int kbeg = int(int64_t(a.nk) * split / nsplit);
  const int nk = int(int64_t(a.nk) * (split + 1) / nsplit) - kbeg;

  // direct-to-LDS lanes: half tile h of X (W): rows 128 h + 16 wave + 8 i +
  // lane / 8, chunk swizzled
  uint32_t xo[H][2], wo[H][2];
#pragma unroll
  for (int h = 0; h < H; ++h)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = 16 * wave + 8 * i + (lane >> 3);
      const uint32_t c = uint32_t(16 * ((lane & 7) ^ ((r >> 1) & 7)));
      int64_t m = m0 + 128 * h + r, n = n0 + 128 * h + r;
      m = m < a.M ? m : a.M - 1;
      n = n < a.N ? n : a.N - 1;
      xo[h][i] = uint32_t(m * a.ldx) * uint32_t(ES) + c;
      wo[h][i] = uint32_t(n * a.ldw) * uint32_t(ES) + c;
    }
  const uint32_t dst0 = __builtin_amdgcn_readfirstlane(uint32_t(wave) * 2048u);
  auto load_half = [&](const void* base, const uint32_t (&off)[2], int step, uint32_t lds_off) {
    const int st = step < nk ? step : nk - 1;  // past the end: a live step again, never used
    const uint8_t* p = static_cast<const uint8_t*>(base) + int64_t(kbeg + st) * 128;
    dma16(p, off[0], dst0 + lds_off);
    dma16(p, off[1], dst0 + lds_off + 1024u);
  };
  // half tile byte offsets in buffer b: the X halves, then the W halves
  auto xoff = [](int b, int h) { return uint32_t(b * kBuf + h * kDnHalf); };
  auto woff = [](int b, int h) { return uint32_t(b * kBuf + (H + h) * kDnHalf); };

  // operand read offsets of sub-step s: chunk 2 s + q of the lane's row
  uint32_t xr[4], wrd[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    xr[s] = swz(uint32_t(64 * wr + i32), uint32_t(2 * s + q));
    wrd[s] = swz(uint32_t(32 * wc + i32), uint32_t(2 * s + q));
  }

  // acc[hm][hn][mb]: quadrant (hm, hn), 32-row block mb
  constexpr int kBlocks = 2 * H * H;
  f32x16 acc[H][H][2];
#pragma unroll
  for (int i = 0; i < kBlocks; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[i / (2 * H)][(i >> 1) % H][i & 1][r] = 0.0f;

  u32x4 xa[2][4], w[H][4];
  auto read_x = [&](int b, int h) {
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
        xa[mb][s] = *reinterpret_cast<const u32x4*>(lds + xoff(b, h) + mb * 4096 + xr[s]);
  };
  auto read_w = [&](u32x4 (&o)[4], int b, int h) {
#pragma unroll
    for (int s = 0; s < 4; ++s) o[s] = *reinterpret_cast<const u32x4*>(lds + woff(b, h) + wrd[s]);
  };
  // fp32: two steps' products are summed on their own (32 MFMAs of 2 k) and added to
  // the tile while the next step's operands are read.  In one chain over K the error
  // grows with its length; so it is no larger than with the short chains of the GEMV
  // blocks that take fewer rows (against float64, in the 2-norm: 4096 -> 4096 with 1000 rows 1.1e-6 in one chain,
  // 2.0e-7 so, 2.9e-7 in the blocks; 14336 -> 4096 2.1e-6, 3.0e-7 and 5.2e-7; 1024 ->
  // 4096 5.5e-7, 1.6e-7 and 2.0e-7).  The adds cost 2 % (1 % to 4 %).
  constexpr bool kF32 = XT == RQ_DTYPE_F32;
  f32x16 pair_sum[kF32 ? 2 : 1];
#pragma unroll
  for (int mb = 0; mb < (kF32 ? 2 : 1); ++mb)
#pragma unroll
    for (int r = 0; r < 16; ++r) pair_sum[mb][r] = 0.0f;
  auto fold = [&]() {
    if constexpr (kF32) {
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[0][0][mb][r] = __fadd_rn(acc[0][0][mb][r], pair_sum[mb][r]);
    }
  };
  auto mma = [&](f32x16 (&c)[2], const u32x4 (&wv)[4], bool fresh = true) {
    __builtin_amdgcn_s_setprio(1);
    if (kF32 && fresh) {
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int r = 0; r < 16; ++r) pair_sum[mb][r] = 0.0f;
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      if constexpr (kF32) {  // the two blocks in turn: no MFMA waits for the one before it
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int mb = 0; mb < 2; ++mb)
            pair_sum[mb] =
                __builtin_amdgcn_mfma_f32_32x32x2f32(u2f(wv[s][j]), u2f(xa[mb][s][j]), pair_sum[mb], 0, 0, 0);
      } else {
#pragma unroll
        for (int mb = 0; mb < 2; ++mb) c[mb] = mfma32x32x16<XT>(wv[s], xa[mb][s], c[mb]);
      }
    }
    __builtin_amdgcn_s_setprio(0);
  };
#define RQ_DN_MEM_END(N)                                                      \
  do {                                                                        \
    __builtin_amdgcn_sched_barrier(0);                                        \
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory"); \
    __builtin_amdgcn_sched_barrier(0);                                        \
  } while (0)
#define RQ_DN_MMA_END()                          \
  do {                                           \
    __builtin_amdgcn_sched_barrier(0);           \
    asm volatile("s_barrier" ::: "memory");      \
    __builtin_amdgcn_sched_barrier(0);           \
  } while (0)
  // 256 x 256, step t, F = t % 2: its buffer and the W half it starts with
  // (alternating, so that a step's first W half can be read while the step
  // before it still multiplies by the other).  A half tile read in one phase
  // is loaded again in the next (its reads end before the barrier that ends
  // the phase's slot, for both wave groups); each is waited for six half
  // tiles (12 loads) later, one phase before its reads.
#define RQ_DN_STEP(t, F)                                     \
  do {                                                       \
    read_x(F, 0);                                            \
    load_half(a.w, wo[F], (t) + 2, woff(F, F));              \
    RQ_DN_MEM_END(12);                                       \
    mma(acc[0][F], w[F]);                                    \
    RQ_DN_MMA_END();                                         \
    read_w(w[1 - (F)], F, 1 - (F));                          \
    load_half(a.x, xo[0], (t) + 2, xoff(F, 0));              \
    RQ_DN_MEM_END(12);                                       \
    mma(acc[0][1 - (F)], w[1 - (F)]);                        \
    RQ_DN_MMA_END();                                         \
    read_x(F, 1);                                            \
    load_half(a.w, wo[1 - (F)], (t) + 2, woff(F, 1 - (F)));  \
    RQ_DN_MEM_END(12);                                       \
    mma(acc[1][1 - (F)], w[1 - (F)]);                        \
    RQ_DN_MMA_END();                                         \
    read_w(w[1 - (F)], 1 - (F), 1 - (F));                    \
    load_half(a.x, xo[1], (t) + 2, xoff(F, 1));              \
    RQ_DN_MEM_END(12);                                       \
    mma(acc[1][F], w[F]);                                    \
    RQ_DN_MMA_END();                                         \
  } while (0)
  // 128 x 128, step t in buffer B: step t - 1's buffer is refilled with step
  // t + 3, and the next step's loads are waited for (two steps younger)
#define RQ_DN_STEP1(t, B)                                          \
  do {                                                             \
    read_x(B, 0);                                                  \
    read_w(w[0], B, 0);                                            \
    load_half(a.w, wo[0], (t) + 3, woff(((B) + 3) & 3, 0));        \
    load_half(a.x, xo[0], (t) + 3, xoff(((B) + 3) & 3, 0));        \
    if (((B) & 1) == 0) fold();                                    \
    RQ_DN_MEM_END(8);                                              \
    mma(acc[0][0], w[0], ((B) & 1) == 0);                          \
    RQ_DN_MMA_END();                                               \
  } while (0)
  int t = 0;
  if constexpr (H == 2) {
    load_half(a.w, wo[0], 0, woff(0, 0));
    load_half(a.x, xo[0], 0, xoff(0, 0));
    load_half(a.w, wo[1], 0, woff(0, 1));
    load_half(a.x, xo[1], 0, xoff(0, 1));
    load_half(a.w, wo[1], 1, woff(1, 1));
    load_half(a.x, xo[0], 1, xoff(1, 0));
    load_half(a.w, wo[0], 1, woff(1, 0));
    load_half(a.x, xo[1], 1, xoff(1, 1));
    RQ_DN_MEM_END(12);
    read_w(w[0], 0, 0);
    RQ_DN_MEM_END(12);
    if (wr == 1) RQ_DN_MMA_END();  // waves 4-7 run one slot behind
    for (; t + 2 <= nk; t += 2) {
      RQ_DN_STEP(t, 0);
      RQ_DN_STEP(t + 1, 1);
    }
    if (t < nk) RQ_DN_STEP(t, 0);
  } else {
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      load_half(a.w, wo[0], p, woff(p, 0));
      load_half(a.x, xo[0], p, xoff(p, 0));
    }
    RQ_DN_MEM_END(8);
    if (wr == 1) RQ_DN_MMA_END();
    for (; t + 4 <= nk; t += 4) {
      RQ_DN_STEP1(t, 0);
      RQ_DN_STEP1(t + 1, 1);
      RQ_DN_STEP1(t + 2, 2);
      RQ_DN_STEP1(t + 3, 3);
    }
    if (t < nk) RQ_DN_STEP1(t, 0);
    if (t + 1 < nk) RQ_DN_STEP1(t + 1, 1);
    if (t + 2 < nk) RQ_DN_STEP1(t + 2, 2);
    fold();
  }
  if (wr == 0) asm volatile("s_barrier" ::: "memory");
  step_barrier<0>();
#undef RQ_DN_STEP
#undef RQ_DN_STEP1
#undef RQ_DN_MEM_END
#undef RQ_DN_MMA_END

  // K splits, as nf4_gemm8_kernel's: every split stores its fp32 tile with
  // device-coherent stores, the last one to count itself sums them in split
  // order (the same bits whichever is last) and runs the epilogue.
  if (nsplit > 1) {
    constexpr uint32_t kTileBytes = Tile::kB * Tile::kB * 4;
    const int lt = T - a.whole;
    const uint32_t lane_off = uint32_t(tid) * 16u;
    auto tile_rsrc = [&](int sp) {
      return buffer_rsrc(reinterpret_cast<const uint8_t*>(a.part) + (int64_t(sp) * lt + ti) * kTileBytes, kTileBytes);
    };
    const __amdgpu_buffer_rsrc_t mine = tile_rsrc(split);
#pragma unroll
    for (int i = 0; i < kBlocks; ++i)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        const f32x16& c = acc[i / (2 * H)][(i >> 1) % H][i & 1];
        buf_store16_coherent(mine, lane_off, uint32_t((4 * i + r4) * kDnThreads * 16),
                             u32x4{f2u(c[4 * r4]), f2u(c[4 * r4 + 1]), f2u(c[4 * r4 + 2]), f2u(c[4 * r4 + 3])});
      }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    uint32_t* flag = reinterpret_cast<uint32_t*>(lds);
    if (tid == 0) {
      const uint32_t old = __hip_atomic_fetch_add(&a.tile_cnt[ti], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const bool last = old == uint32_t(nsplit - 1);
      if (last) __hip_atomic_store(&a.tile_cnt[ti], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *flag = last ? 1u : 0u;
    }
    __syncthreads();
    const uint32_t last = __builtin_amdgcn_readfirstlane(*flag);
    __syncthreads();
    if (!last) return;
#pragma unroll
    for (int i = 0; i < kBlocks; ++i) {
      f32x16& c = acc[i / (2 * H)][(i >> 1) % H][i & 1];
#pragma unroll
      for (int r = 0; r < 16; ++r) c[r] = 0.0f;
      for (int sp = 0; sp < nsplit; ++sp) {
        const __amdgpu_buffer_rsrc_t o = tile_rsrc(sp);
        u32x4 v[4];
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4)
          v[r4] = buf_load16_coherent(o, lane_off, uint32_t((4 * i + r4) * kDnThreads * 16));
#pragma unroll
        for (int r = 0; r < 16; ++r) c[r] = __fadd_rn(c[r], u2f(v[r >> 2][r & 3]));
      }
    }
  }

  // Epilogue, one 64 x 32 quadrant (hm, hn) of the wave at a time
#pragma unroll
  for (int hm = 0; hm < H; ++hm)
#pragma unroll
    for (int hn = 0; hn < H; ++hn) {
      const int64_t nq = n0 + 128 * hn + 32 * wc;
      const int64_t mq = m0 + 128 * hm + 64 * wr;
      f32x16 lo[2];
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int r = 0; r < 16; ++r) lo[mb][r] = 0.0f;
      if (e.rankp > 0) {
        int64_t n = nq + i32;
        n = n < a.N ? n : a.N - 1;
        const uint8_t* bp = static_cast<const uint8_t*>(e.b) + n * e.rankp * ES + 16 * q;
        const uint8_t* up[2];
#pragma unroll
        for (int mb = 0; mb < 2; ++mb) {
          int64_t m = mq + 32 * mb + i32;
          m = m < a.M ? m : a.M - 1;
          up[mb] = static_cast<const uint8_t*>(e.u) + m * e.rankp * ES + 16 * q;
        }
        for (int s = 0; s < e.rankp * ES; s += 32) {
          const u32x4 bv = *reinterpret_cast<const u32x4*>(bp + s);
#pragma unroll
          for (int mb = 0; mb < 2; ++mb)
            lo[mb] = dn_mfma<XT>(bv, *reinterpret_cast<const u32x4*>(up[mb] + s), lo[mb]);
        }
      }
      float bias[4][4];
#pragma unroll
      for (int h = 0; h < 4; ++h) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const int64_t n = nq + 8 * h + 4 * q + c;
          bias[h][c] = e.bias && n < a.N ? load_as_f32(e.bias, n, e.bias_dt) : -0.0f;
        }
        dn_round2<XT>(bias[h][0], bias[h][1]);
        dn_round2<XT>(bias[h][2], bias[h][3]);
      }
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          float v[4];
#pragma unroll
          for (int c = 0; c < 4; ++c) v[c] = __fadd_rn(acc[hm][hn][mb][4 * h + c], bias[h][c]);
          if (e.rankp > 0) {
            dn_round2<XT>(v[0], v[1]);
            dn_round2<XT>(v[2], v[3]);
            float l[4], s[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
              l[c] = lo[mb][4 * h + c];
              s[c] = e.scaling;
            }
            if (e.mask) {
              const int64_t m = mq + 32 * mb + i32, n = nq + 8 * h + 4 * q;
#pragma unroll
              for (int c = 0; c < 4; ++c)
                s[c] = m < a.M && n + c < a.N && e.mask[m * e.ldm + n + c] ? e.mask_scale : 0.0f;
            }
            dn_round2<XT>(l[0], l[1]);
            dn_round2<XT>(l[2], l[3]);
#pragma unroll
            for (int c = 0; c < 4; ++c) l[c] = __fmul_rn(l[c], s[c]);
            dn_round2<XT>(l[0], l[1]);
            dn_round2<XT>(l[2], l[3]);
#pragma unroll
            for (int c = 0; c < 4; ++c) v[c] = __fadd_rn(v[c], l[c]);
          }
          uint8_t* o = lds + (128 * hm + 64 * wr + 32 * mb + i32) * kOutPitch +
                       (128 * hn + 32 * wc + 8 * h + 4 * q) * ES;
          if constexpr (XT == RQ_DTYPE_F32)
            *reinterpret_cast<u32x4*>(o) = u32x4{f2u(v[0]), f2u(v[1]), f2u(v[2]), f2u(v[3])};
          else
            *reinterpret_cast<u32x2*>(o) = u32x2{cvt_pk<XT>(v[0], v[1]), cvt_pk<XT>(v[2], v[3])};
        }
    }
  __syncthreads();
  // 16 H rows per wave, whole rows of the tile per instruction
  constexpr int kPer = 16 / ES;            // outputs per 16-byte chunk
  constexpr int kLpr = Tile::kB / kPer;    // lanes per row
  constexpr int kRows = 64 / kLpr;         // rows per instruction
  const bool vec = (reinterpret_cast<uintptr_t>(e.y) & 15u) == 0 && e.ldy % kPer == 0;
  const int64_t nc = n0 + kPer * (lane & (kLpr - 1));
#pragma unroll 4
  for (int it = 0; it < Tile::kB / 8 / kRows; ++it) {
    const int r = (Tile::kB / 8) * wave + kRows * it + lane / kLpr;
    const int64_t m = m0 + r;
    if (m >= a.M) continue;
    const u32x4 v = *reinterpret_cast<const u32x4*>(lds + r * kOutPitch + 16 * (lane & (kLpr - 1)));
    uint8_t* yp = static_cast<uint8_t*>(e.y) + (m * e.ldy + nc) * ES;
    if (vec && nc + kPer <= a.N) {
      *reinterpret_cast<u32x4*>(yp) = v;
    } else {
#pragma unroll
      for (int c = 0; c < kPer; ++c) {
        if (nc + c >= a.N) break;
        if constexpr (ES == 4) reinterpret_cast<uint32_t*>(yp)[c] = v[c];
        else reinterpret_cast<uint16_t*>(yp)[c] = uint16_t(v[c >> 1] >> (16 * (c & 1)));
      }
    }
  }
}

}  // namespace rq
