// Projections of the indexer sidecar for batches of tokens (reference
// sidecar.py:55-58 wq / wk / weights_proj, used by encode_queries and
// encode_keys, sidecar.py:74-88): out[t][f] = sum_k hidden[t][k] * W[f][k].
// (A decode step of at most 16 tokens streams the weights in project.hip.)
//
// gemm_bf16_kernel: bf16 hidden and weights, fp32 accumulation, bf16 out
// rounded once (nearest even), as a bf16 Linear stores it.  A workgroup owns
// BF features x BT tokens; its waves split them WF x WT.  Each k-stage of 64 stages the
// weight rows and the hidden rows in LDS (rows padded to 144 B), loaded NPF
// stages ahead into registers, and every wave runs
// v_mfma_f32_16x16x32_bf16 with 16 weight rows as the A operand and 16
// tokens as B: the accumulator of a tile then holds, per lane, four
// consecutive features of one token, stored as one 8-byte bf16x4.
// With kRope the output stage also applies the non-interleaved RoPE of the
// query heads (sidecar.py:10-28, 78-88): every 128-feature head rotates its
// first 64 dims, dim d with dim d + 32.  A wave's 64 features are one head's
// rotated or unrotated half, and dims d and d + 32 sit in the same lane (tiles
// f and f + 2), so the rotation needs no data exchange.  cos / sin come from
// rope_table_kernel, in the bf16 precision and per-op rounding of the
// encoder epilogues (sidecar.hip).
//
// gemm_wide_kernel: the same product for whole 256-feature tiles and enough
// tokens to give every CU one (see there).
//
// gemm_f32_kernel: fp32 weights (weights_proj, which the reference runs on
// hidden.float(), and fp32 modules), hidden bf16 or fp32 widened exactly to
// fp32, v_mfma_f32_16x16x4_f32, fp32 out times an optional scale (the head
// weights' (heads * head_dim)^-0.5, one fp32 product as in the reference).
//
// gemm_narrow_kernel: wk and weights_proj of many tokens, k split over
// workgroups; finish_keys_kernel and finish_weights_kernel complete the rows.
#include "common.hpp"
#include "dsa_amd.h"
#include "status.hpp"

#include <algorithm>
#include <type_traits>

namespace dsa {
namespace {

constexpr int kGemmBK = 64;            // k per stage (bf16)
constexpr int kGemmRow = kGemmBK + 8;  // bf16 per LDS row: 144 B against bank conflicts
constexpr uint32_t kFar = 0x80000000u; // a buffer offset past every resource: loads read 0, stores drop
constexpr int kRopeHalf = 32;          // fused RoPE: 64 rotated dims of every 128-dim head

struct GemmArgs {
  const uint16_t* hidden;  // [tokens][hidden_stride] bf16, or fp32 (gemm_f32_kernel with hidden_f32)
  int64_t hidden_stride;   // elements between tokens
  const void* weight;      // [features][kdim] bf16 or fp32
  void* out;               // [tokens][out_stride] bf16 or fp32
  int64_t out_stride;
  int32_t tokens, features, kdim;
  float scale;             // gemm_f32_kernel: out = acc * scale
  const uint32_t* rope;    // kRope: [tokens][kRopeHalf] bf16 cos << 16 | bf16 sin
};

__device__ __forceinline__ uint32_t bf16_rne_bits(float x) {
  const uint32_t u = __float_as_uint(x);
  const uint32_t rounded = (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
  return (u & 0x7fffffffu) > 0x7f800000u ? (u >> 16) | 0x40u : rounded;  // NaN stays a (quiet) NaN
}
__device__ __forceinline__ float round_bf16f(float x) { return __uint_as_float(bf16_rne_bits(x) << 16); }

// cos / sin of position * theta^(-i / 32), i < 32, rounded to bf16: the
// rotation table of one token (the formula of the encoder epilogues).
__device__ __forceinline__ uint32_t rope_entry(int64_t position, int i, float theta) {
  const float angle = (float)position * powf(theta, -(float)i / (float)kRopeHalf);
  return (bf16_rne_bits(cosf(angle)) << 16) | bf16_rne_bits(sinf(angle));
}

struct RopeTableArgs {
  const int64_t* positions;  // [tokens]
  uint32_t* table;           // [tokens][kRopeHalf]
  int32_t tokens;
  float theta;
};

__device__ __forceinline__ void rope_table_block(const RopeTableArgs& a, int64_t block) {
  const int64_t e = block * 256 + threadIdx.x;
  if (e >= (int64_t)a.tokens * kRopeHalf) return;
  a.table[e] = rope_entry(a.positions[e / kRopeHalf], (int)(e % kRopeHalf), a.theta);
}

__global__ __launch_bounds__(256) void rope_table_kernel(RopeTableArgs a) { rope_table_block(a, blockIdx.x); }

int64_t rope_table_blocks(int64_t tokens) { return (tokens * kRopeHalf + 255) / 256; }

// Two fp32 values rounded to nearest-even bf16, the first in the low half
// (v_cvt_pk_bf16_f32).
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  const floatx2 v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}
__device__ __forceinline__ float bf16_low(uint32_t v) { return __uint_as_float(v << 16); }
__device__ __forceinline__ float bf16_high(uint32_t v) { return __uint_as_float(v & 0xffff0000u); }

// Rotates two dims (packed bf16 pairs x and, kRopeHalf dims on, y) by their
// table entries, every product and sum rounded to bf16.
__device__ __forceinline__ void rotate_pairs(uint32_t& x, uint32_t& y, uint32_t cs0, uint32_t cs1) {
  const float x0 = bf16_low(x), x1 = bf16_high(x), y0 = bf16_low(y), y1 = bf16_high(y);
  const float c0 = bf16_high(cs0), s0 = bf16_low(cs0), c1 = bf16_high(cs1), s1 = bf16_low(cs1);
  const uint32_t xc = pack_bf16(x0 * c0, x1 * c1), ys = pack_bf16(y0 * s0, y1 * s1);
  const uint32_t yc = pack_bf16(y0 * c0, y1 * c1), xs = pack_bf16(x0 * s0, x1 * s1);
  x = pack_bf16(bf16_low(xc) - bf16_low(ys), bf16_high(xc) - bf16_high(ys));
  y = pack_bf16(bf16_low(yc) + bf16_low(xs), bf16_high(yc) + bf16_high(xs));
}

template <int BF, int BT, int WF, int WT, bool kRope, int NPF>
__global__ __launch_bounds__(64 * WF * WT) void gemm_bf16_kernel(GemmArgs a) {
  constexpr int kThreads = 64 * WF * WT;
  constexpr int FW = BF / WF;  // features per wave
  constexpr int TW = BT / WT;  // tokens per wave
  constexpr int FT = FW / 16;
  constexpr int TT = TW / 16;
  constexpr int kRows = BF + BT;                  // LDS rows per stage: weights, then tokens
  // 16-byte chunks a thread stages: its first kPerW are weight rows, the
  // rest token rows, so that the buffer resource of a load is known at
  // compile time (a per-lane choice would cost a waterfall loop per load).
  constexpr int kPerW = BF * (kGemmBK / 8) / kThreads;
  constexpr int kPer = kPerW + BT * (kGemmBK / 8) / kThreads;
  static_assert(BF * (kGemmBK / 8) % kThreads == 0 && BT * (kGemmBK / 8) % kThreads == 0, "stage chunks per thread");
  static_assert(!kRope || FW == 64 || FW % 128 == 0, "a rotating wave owns half a 128-dim head or whole heads");
  __shared__ __align__(16) uint16_t lds[2][kRows][kGemmRow];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wf = wave % WF;
  const int wt = wave / WF;
  const int r = lane & 15;
  const int g = lane >> 4;
  const int feature_tiles = (a.features + BF - 1) / BF;
  const int f0 = (int)(blockIdx.x % (uint32_t)feature_tiles) * BF;
  const int t0 = (int)(blockIdx.x / (uint32_t)feature_tiles) * BT;
  const int kdim = a.kdim;

  const BufferRsrc wr = make_buffer(a.weight, (uint32_t)a.features * (uint32_t)kdim * 2u);
  const BufferRsrc hr = make_buffer(a.hidden, (uint32_t)(((int64_t)(a.tokens - 1) * a.hidden_stride + kdim) * 2));
  // This thread's chunks of a stage: row rows_[i] (weights below BF), k
  // offset 8 * part_[i] within the stage.
  int row_of[kPer];
  uint32_t base_of[kPer];  // byte offset of the row's k = 0, or kFar for rows past the matrix
  int part_of[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int c = tid + kThreads * (i < kPerW ? i : i - kPerW);
    const int row = c / (kGemmBK / 8) + (i < kPerW ? 0 : BF);
    row_of[i] = row;
    part_of[i] = c % (kGemmBK / 8);
    if (i < kPerW) {
      const int f = f0 + row;
      base_of[i] = f < a.features ? (uint32_t)f * (uint32_t)kdim * 2u : kFar;
    } else {
      const int t = t0 + row - BF;
      base_of[i] = t < a.tokens ? (uint32_t)((int64_t)t * a.hidden_stride * 2) : kFar;
    }
  }
  // NPF stages in flight in registers (a ring), two in LDS.
  uint4 stage[NPF][kPer];
  auto load_stage = [&](int kt, uint4 (&dst)[kPer]) {
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int k = kt * kGemmBK + 8 * part_of[i];
      const uint32_t off = (base_of[i] == kFar || k >= kdim) ? kFar : base_of[i] + (uint32_t)k * 2u;
      dst[i] = buffer_load_16(i < kPerW ? wr : hr, off);
    }
  };
  auto store_stage = [&](int s, const uint4 (&src)[kPer]) {
#pragma unroll
    for (int i = 0; i < kPer; ++i)
      *reinterpret_cast<uint4*>(&lds[s][row_of[i]][8 * part_of[i]]) = src[i];
  };

  floatx4 acc[FT][TT];
#pragma unroll
  for (int i = 0; i < FT; ++i)
#pragma unroll
    for (int j = 0; j < TT; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

  const int nk = (kdim + kGemmBK - 1) / kGemmBK;
  {
    uint4 first[kPer];
    load_stage(0, first);
#pragma unroll
    for (int p = 0; p < NPF; ++p) load_stage(min(1 + p, nk - 1), stage[p]);
    store_stage(0, first);
  }
  __syncthreads();
  // Iteration kt computes stage kt from LDS while stages kt + 1 .. kt + NPF
  // are in flight in registers; stage kt + 1 then goes to LDS and the loads
  // of stage kt + 1 + NPF take its registers.  Loads past the last stage
  // repeat it (unconditional, so that the compiler's waits cover exactly
  // the registers being stored).
  for (int kt0 = 0; kt0 < nk; kt0 += NPF) {
#pragma unroll
    for (int p = 0; p < NPF; ++p) {
    const int kt = kt0 + p;
    if (kt >= nk) break;
    const int cur = kt & 1;
#pragma unroll
    for (int ks = 0; ks < kGemmBK / 32; ++ks) {
      uint4 af[FT];
      uint4 bfrag[TT];
#pragma unroll
      for (int i = 0; i < FT; ++i)
        af[i] = *reinterpret_cast<const uint4*>(&lds[cur][wf * FW + 16 * i + r][32 * ks + 8 * g]);
#pragma unroll
      for (int j = 0; j < TT; ++j)
        bfrag[j] = *reinterpret_cast<const uint4*>(&lds[cur][BF + wt * TW + 16 * j + r][32 * ks + 8 * g]);
      // All of the k-step's fragment reads are issued before its MFMAs: left
      // to itself the scheduler reads one A fragment at a time, each behind
      // a wait for the previous one.
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < FT; ++i)
#pragma unroll
        for (int j = 0; j < TT; ++j) acc[i][j] = mfma_16x16x32(Bf16Tag{}, af[i], bfrag[j], acc[i][j]);
    }
    // Buffer cur ^ 1 was last read in the previous iteration, before the
    // barrier every thread has passed since.
    store_stage(cur ^ 1, stage[p]);
    load_stage(min(kt + 1 + NPF, nk - 1), stage[p]);
    __syncthreads();
    }
  }

  // Output: lane (r, g) of tile (i, j) holds features f0 + wf * FW + 16 i +
  // 4 g + e (e < 4) of token t0 + wt * TW + 16 j + r.
  const BufferRsrc outr = make_buffer(a.out, (uint32_t)(((int64_t)(a.tokens - 1) * a.out_stride + a.features) * 2));
  const int fw0 = f0 + wf * FW;
  // Tile i holds dims 16 (i % 8) .. of its head (FW = 64: the wave's first
  // tile starts at dim 0 or 64); tiles of dims 0..31 rotate with tile i + 2.
  auto rotates = [&](int i) { return (((fw0 + 16 * i) % 128) / 16) < 2; };
#pragma unroll
  for (int j = 0; j < TT; ++j) {
    const int t = t0 + wt * TW + 16 * j + r;
    float v[FT][4];
#pragma unroll
    for (int i = 0; i < FT; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) v[i][e] = round_bf16f(acc[i][j][e]);  // the projection, as bf16
    if constexpr (kRope) {
      const uint32_t* cs = a.rope + (size_t)min(t, a.tokens - 1) * kRopeHalf;
#pragma unroll
      for (int i = 0; i + 2 < FT; ++i) {
        if (!rotates(i)) continue;  // uniform across the wave
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t p = cs[16 * (i % 2) + 4 * g + e];
          const float c = __uint_as_float(p & 0xffff0000u);
          const float s = __uint_as_float(p << 16);
          const float x1 = v[i][e];
          const float x2 = v[i + 2][e];
          v[i][e] = round_bf16f(round_bf16f(x1 * c) - round_bf16f(x2 * s));
          v[i + 2][e] = round_bf16f(round_bf16f(x2 * c) + round_bf16f(x1 * s));
        }
      }
    }
#pragma unroll
    for (int i = 0; i < FT; ++i) {
      const int f = fw0 + 16 * i + 4 * g;
      const uint32_t lo = (__float_as_uint(v[i][0]) >> 16) | (__float_as_uint(v[i][1]) & 0xffff0000u);
      const uint32_t hi = (__float_as_uint(v[i][2]) >> 16) | (__float_as_uint(v[i][3]) & 0xffff0000u);
      const uint32_t off = (t < a.tokens && f < a.features) ? (uint32_t)(((int64_t)t * a.out_stride + f) * 2) : kFar;
      buffer_store_u64(outr, off, ((uint64_t)hi << 32) | lo);
    }
  }
}

// The product for whole tiles of 256 features (a 256-token tail is allowed)
// and kdim a multiple of 64, 256 features x 256 tokens per tile, tiles dealt
// round-robin to at most one workgroup per CU.  Bound: LDS and issue slots
// beside the MFMAs, then the chip's power (the clock falls from 2.3 to about
// 2.0 GHz while it runs).
//  - Four waves of 128 x 128 (one per SIMD, accumulators in the 256 AGPRs)
//    read 64 KB of fragments per 32 k, where eight waves of 128 x 64 read 96
//    KB and kept the LDS busy all the time.
//  - With one wave per SIMD nothing else fills a stall, so the k-loop is
//    scheduled by hand: every MFMA is followed by at most one memory
//    instruction, fragments are read four 16-row steps (512 cycles) ahead,
//    and a stage of 64 k is 260 instructions for its 128 MFMAs.
//  - LDS rows are 128 bytes, their 16-byte chunks permuted by the row so that
//    the 16 lanes of a read phase fall on 16 different bank groups (padded
//    rows of 144 bytes had conflicts in a third of the LDS cycles).
//  - Row 8 (m / 4) + 4 (i & 1) + m % 4 of the 32-feature group i / 2 is row m
//    of A tile i, so a lane's accumulators of tiles 2p and 2p + 1 are eight
//    consecutive features: one 16-byte store.
//  - The next tile's first stages are loaded while the previous tile ends, and
//    its stores drain under the next tile's products.
// wq at 4096 tokens, hidden 2048 with its RoPE: 146-158 us before, 118 us now
// (1.17 PFLOP/s; the platform's own matrix product reaches 1.18-1.26 on this
// card at 4096^3 and 8192^3).
constexpr int kWideTile = 256;
constexpr int kWideRow = kGemmBK;  // bf16 per LDS row
constexpr int64_t kWideGrid = 256;  // one workgroup per CU

template <bool kRope>
__global__ __launch_bounds__(256, 1) void gemm_wide_kernel(GemmArgs a, int tiles) {
  __shared__ __align__(16) uint16_t lds[2 * 2 * kWideTile * kWideRow];
  constexpr int kStage = 2 * kWideTile * kWideRow;  // weight rows, then token rows
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wf = wave & 1;
  const int wt = wave >> 1;
  const int r = lane & 15;
  const int g = lane >> 4;
  const int ftiles = a.features / kWideTile;
  const int kdim = a.kdim;
  const int nk = kdim / kGemmBK;
  const uint32_t wbytes = (uint32_t)a.features * (uint32_t)kdim * 2u;
  const uint32_t hbytes = (uint32_t)(((int64_t)(a.tokens - 1) * a.hidden_stride + kdim) * 2);
  const BufferRsrc outr = make_buffer(a.out, (uint32_t)(((int64_t)(a.tokens - 1) * a.out_stride + a.features) * 2));
  auto tile_f = [&](int tile) { return (int)((uint32_t)tile % (uint32_t)ftiles) * kWideTile; };
  auto tile_t = [&](int tile) { return (int)((uint32_t)tile / (uint32_t)ftiles) * kWideTile; };

  // Global loads: thread (row0, part) stages 16-byte chunk `part` of rows
  // row0 + 32 i, of the weights (i < 8) and the tokens.  The cursor (tile, k)
  // runs one stage ahead of the LDS; it moves through scalar base pointers, so
  // a load costs no address arithmetic.  Token rows past the last repeat it.
  const int row0 = tid >> 3;
  const int part = tid & 7;
  const int wstep = 32 * kdim * 2;
  const uint32_t woff = (uint32_t)row0 * (uint32_t)kdim * 2u + 16u * part;
  uint32_t hoff[8];
  const uint8_t* wp = nullptr;
  const uint8_t* hp = nullptr;
  uint32_t wleft = 0, hleft = 0;
  int load_tile = blockIdx.x;
  int load_k = 0;
  auto seek = [&](int tile) {
    const uint32_t skip = (uint32_t)tile_f(tile) * (uint32_t)kdim * 2u;
    wp = static_cast<const uint8_t*>(a.weight) + skip;
    wleft = wbytes - skip;
    hp = reinterpret_cast<const uint8_t*>(a.hidden);
    hleft = hbytes;
    const int t0 = tile_t(tile);
#pragma unroll
    for (int i = 0; i < 8; ++i)
      hoff[i] = (uint32_t)min(t0 + row0 + 32 * i, a.tokens - 1) * (uint32_t)a.hidden_stride * 2u + 16u * part;
  };
  auto advance = [&] {
    if (++load_k == nk) {  // past the last tile the cursor repeats it (loads nobody uses)
      load_k = 0;
      if (load_tile + (int)gridDim.x < tiles) load_tile += gridDim.x;
      seek(load_tile);
    } else {
      wp += kGemmBK * 2;
      hp += kGemmBK * 2;
      wleft -= kGemmBK * 2;
      hleft -= kGemmBK * 2;
    }
  };
  uint4 stage[16];
  auto load = [&](int i) {
    const u32x4 v = i < 8 ? __builtin_amdgcn_raw_buffer_load_b128(make_buffer(wp, wleft), (int)woff, i * wstep, 0)
                          : __builtin_amdgcn_raw_buffer_load_b128(make_buffer(hp, hleft), (int)hoff[i & 7], 0, 0);
    stage[i] = make_uint4(v.x, v.y, v.z, v.w);
  };
  // Chunk permutations.  A read phase takes 16 lanes of different r (and two
  // values of g): weight rows 8 (r / 4) + r % 4 differ in bits 0, 1, 3 and 4,
  // token rows in bits 0 to 3; bit 0 picks the 128-byte half of the banks.
  auto swizzle_w = [](int row) { return ((row >> 1) & 1) | (((row >> 3) & 3) << 1); };
  auto swizzle_t = [](int row) { return (row >> 1) & 7; };
  uint16_t* const put_w = lds + row0 * kWideRow + 8 * (part ^ swizzle_w(row0));
  uint16_t* const put_t = lds + row0 * kWideRow + 8 * (part ^ swizzle_t(row0));
  auto put = [&](int i, int buf) {
    *reinterpret_cast<uint4*>((i < 8 ? put_w : put_t) + buf * kStage + 32 * i * kWideRow) = stage[i];
  };
  const int arow = 8 * (r >> 2) + (r & 3);
  const uint16_t* const read_w = lds + (wf * 128 + arow) * kWideRow;
  const uint16_t* const read_t = lds + (kWideTile + wt * 128 + r) * kWideRow;
  const int wc[2] = {8 * (g ^ swizzle_w(arow)), 8 * ((4 + g) ^ swizzle_w(arow))};
  const int tc[2] = {8 * (g ^ swizzle_t(r)), 8 * ((4 + g) ^ swizzle_t(r))};
  // A fragments: a ring of eight; step n of a stage's 16 uses tile n & 7 of
  // k-step n >> 3.  B fragments: all eight of both k-steps.
  uint4 fa[8], fb[2][8];
  auto read_a = [&](int buf, int n) {
    fa[n & 7] = *reinterpret_cast<const uint4*>(read_w + buf * kStage +
                                                (32 * ((n & 7) >> 1) + 4 * (n & 1)) * kWideRow + wc[n >> 3]);
  };
  auto read_b = [&](int buf, int ks, int j) {
    fb[ks][j] = *reinterpret_cast<const uint4*>(read_t + buf * kStage + 16 * j * kWideRow + tc[ks]);
  };
  floatx4 acc[8][8];
  auto clear = [&] {
    // Opaque to the compiler, which otherwise shares the zeros and copies
    // accumulators between registers inside the k-loop.
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
        asm volatile("" : "+a"(acc[i][j]));
      }
  };
  int buf = 0;
  // One stage of 64 k from lds[buf].  The stage in registers goes to the other
  // buffer and the cursor's stage takes its registers (steps 0 to 7); all
  // reads of this buffer are issued by step 11, so the barrier before step 12
  // both publishes the next stage and frees this one.  kLast: no reads ahead
  // (the epilogue follows and needs their registers).
  auto stage_step = [&](auto last) {
    constexpr bool kLast = decltype(last)::value;
    const int next = buf ^ 1;
#pragma unroll
    for (int n = 0; n < 16; ++n) {
      if (n == 12) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if (j == 0 && n < 12) read_a(buf, n + 4);
        if (j == 0 && n >= 12 && !kLast) read_a(next, n - 12);
        if (j == 1 && n < 8) read_b(buf, 1, n);
        if (j == 1 && n >= 12 && !kLast) read_b(next, 0, 2 * (n - 12));
        if (j == 3 && n >= 12 && !kLast) read_b(next, 0, 2 * (n - 12) + 1);
        if (j == 2 && n < 8) put(2 * n, next);
        if (j == 3 && n < 8) load(2 * n);
        if (j == 5 && n < 8) put(2 * n + 1, next);
        if (j == 6 && n < 8) load(2 * n + 1);
        acc[n & 7][j] = mfma_16x16x32(Bf16Tag{}, fa[n & 7], fb[n >> 3][j], acc[n & 7][j]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    advance();
    buf = next;
  };

  seek(load_tile);
#pragma unroll
  for (int i = 0; i < 16; ++i) load(i);
  advance();
#pragma unroll
  for (int i = 0; i < 16; ++i) put(i, 0);
#pragma unroll
  for (int i = 0; i < 16; ++i) load(i);
  advance();
  __syncthreads();
  clear();
  for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
#pragma unroll
    for (int j = 0; j < 8; ++j) read_b(buf, 0, j);
#pragma unroll
    for (int n = 0; n < 4; ++n) read_a(buf, n);
    for (int kt = 0; kt < nk - 1; ++kt) stage_step(std::false_type{});
    stage_step(std::true_type{});
    // Lane (r, g) of tiles 2p, 2p + 1 holds features f0 + 128 wf + 32 p + 8 g
    // .. + 7 of token t0 + 128 wt + 16 j + r: the wave's 128 features are one
    // head, whose dims 0..31 (p = 0) rotate with dims 32..63 (p = 1).
    const int fw0 = tile_f(tile) + wf * 128;
    const int tw0 = tile_t(tile) + wt * 128 + r;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int t = tw0 + 16 * j;
      const uint32_t off = t < a.tokens ? (uint32_t)(((int64_t)t * a.out_stride + fw0 + 8 * g) * 2) : kFar;
      uint2 v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i)
        v[i] = make_uint2(pack_bf16(acc[i][j][0], acc[i][j][1]), pack_bf16(acc[i][j][2], acc[i][j][3]));
      if constexpr (kRope) {
        const uint4* cs = reinterpret_cast<const uint4*>(a.rope + (size_t)min(t, a.tokens - 1) * kRopeHalf);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const uint4 p = cs[2 * g + i];
          rotate_pairs(v[i].x, v[i + 2].x, p.x, p.y);
          rotate_pairs(v[i].y, v[i + 2].y, p.z, p.w);
        }
      }
#pragma unroll
      for (int p = 0; p < 4; ++p)
        buffer_store_16(outr, off + 64u * p, make_uint4(v[2 * p].x, v[2 * p].y, v[2 * p + 1].x, v[2 * p + 1].y));
      __builtin_amdgcn_sched_barrier(0);
    }
    clear();
  }
}

// Narrow products (wk: 128 bf16 features, weights_proj: 64 fp32 ones) of many
// tokens.  A CU takes in about 25-40 KB per us whatever the pattern (its L1
// tracks about 32 KB of misses at the L2's latency), so a workgroup that reads
// every weight row whole (576 KB with 16 tokens beside 128 rows) needs more
// than 20 us: 18.8 us for wk and 30 us for weights_proj at 4096 tokens, hidden
// 2048.  Here k is split over workgroups as well: a workgroup takes 64 tokens,
// all features of its tile and kNarrowK of k, 192 KB, and writes fp32 partial
// sums; the launch that finishes the rows adds them in a fixed order (8 MB of
// partial sums at 4096 tokens).  All of a workgroup's loads are issued at
// once, into registers, and go through two LDS buffers stage by stage.  4096 tokens, hidden 2048: wk
// 12.1 us and its rows 5 us (18.8 and 7.9 before), weights_proj 19.3 us with
// the rotation table beside it and its rows 5 us (30 and 5.1).
constexpr int kNarrowTok = 64;
constexpr int kNarrowStages = 8;                        // stages of 64 k in flight
constexpr int kNarrowK = kNarrowStages * kGemmBK;       // most k per workgroup

template <bool kF32>
constexpr int kNarrowFeat = kF32 ? 64 : 128;

struct NarrowArgs {
  const uint16_t* hidden;
  int64_t hidden_stride;
  const void* weight;  // [features][kdim] bf16 or fp32
  int32_t tokens, features, kdim;
  int32_t kper;    // k per workgroup, a multiple of 64 up to kNarrowK
  int32_t splits;  // ceil(kdim / kper)
  float* parts;    // [splits][tokens][features]
};

template <bool kF32>
__global__ __launch_bounds__(256, 1) void gemm_narrow_kernel(NarrowArgs a, RopeTableArgs rope, int product_blocks) {
  constexpr int kFeat = kNarrowFeat<kF32>;
  constexpr int kWBytes = kF32 ? 4 : 2;
  constexpr int kWRow = kGemmBK * kWBytes;     // weight row bytes per stage
  constexpr int kWLoads = kFeat * kWRow / 16 / 256;
  constexpr int kTRow = kGemmBK * 2;
  constexpr int kTLoads = kNarrowTok * kTRow / 16 / 256;
  constexpr int kLoads = kWLoads + kTLoads;
  __shared__ __align__(16) uint8_t lds[2][kFeat * kWRow + kNarrowTok * kTRow];
  if ((int)blockIdx.x >= product_blocks) {
    rope_table_block(rope, (int64_t)blockIdx.x - product_blocks);
    return;
  }
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15;
  const int g = lane >> 4;
  const int kdim = a.kdim;
  const int ftiles = (a.features + kFeat - 1) / kFeat;
  const int split = (int)(blockIdx.x % (uint32_t)a.splits);
  const int f0 = (int)(blockIdx.x / (uint32_t)a.splits % (uint32_t)ftiles) * kFeat;
  const int t0 = (int)(blockIdx.x / (uint32_t)a.splits / (uint32_t)ftiles) * kNarrowTok;
  const int k0 = split * a.kper;
  const int k1 = min(kdim, k0 + a.kper);
  const BufferRsrc wr = make_buffer(a.weight, (uint32_t)a.features * (uint32_t)kdim * kWBytes);
  const BufferRsrc hr = make_buffer(a.hidden, (uint32_t)(((int64_t)(a.tokens - 1) * a.hidden_stride + kdim) * 2));
  // Chunk c = tid + 256 i of a stage: 16 bytes of a weight row, or of a token
  // row.  The LDS slot of a row's chunk is permuted by the row, so that the 16
  // rows a read phase touches fall on different banks.
  uint4 stage[kNarrowStages][kLoads];
  uint32_t slot[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const bool weight = i < kWLoads;
    constexpr int kWChunks = kWRow / 16, kTChunks = kTRow / 16;
    const int c = tid + 256 * (weight ? i : i - kWLoads);
    const int row = c / (weight ? kWChunks : kTChunks);
    const int chunk = c % (weight ? kWChunks : kTChunks);
    const int swz = weight && kF32 ? row & 15 : (row >> 1) & 7;
    slot[i] = (weight ? (uint32_t)(row * kWRow) : (uint32_t)(kFeat * kWRow + row * kTRow)) + 16u * (chunk ^ swz);
    const int k = k0 + chunk * (weight ? 16 / kWBytes : 8);
    const int at = weight ? f0 + row : t0 + row;
    const bool live = at < (weight ? a.features : a.tokens);
    const uint32_t base = weight ? (uint32_t)at * (uint32_t)kdim * kWBytes : (uint32_t)((int64_t)at * a.hidden_stride * 2);
#pragma unroll
    for (int st = 0; st < kNarrowStages; ++st) {
      const int ks = k + st * kGemmBK;
      stage[st][i] = buffer_load_16(weight ? wr : hr, live && ks < k1 ? base + (uint32_t)ks * (weight ? kWBytes : 2) : kFar);
    }
  }
  auto put = [&](int st) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) *reinterpret_cast<uint4*>(&lds[st & 1][slot[i]]) = stage[st][i];
  };
  constexpr int FT = kF32 ? 2 : 4;  // feature tiles of a wave; two token tiles
  const int wf = (wave & 1) * 16 * FT;
  const int wt = (wave >> 1) * 32;
  floatx4 acc[FT][2];
#pragma unroll
  for (int i = 0; i < FT; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int st = 0; st < kNarrowStages; ++st) {
    if (st * kGemmBK >= a.kper) break;  // uniform
    // Buffer st & 1 was last read two stages ago, before the previous barrier.
    put(st);
    __syncthreads();
    const uint8_t* w = lds[st & 1];
    const uint8_t* t = w + kFeat * kWRow;
    if constexpr (kF32) {
#pragma unroll
      for (int q = 0; q < kGemmBK / 16; ++q) {
        // k = 16 q + 4 g + e feeds element e of both operands.
        float wv[2][4], hv[2][4];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int row = wf + 16 * i + r;
          const uint4 v = *reinterpret_cast<const uint4*>(w + row * kWRow + 16 * ((4 * q + g) ^ (row & 15)));
          wv[i][0] = __uint_as_float(v.x);
          wv[i][1] = __uint_as_float(v.y);
          wv[i][2] = __uint_as_float(v.z);
          wv[i][3] = __uint_as_float(v.w);
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int row = wt + 16 * j + r;
          const int u = 4 * q + g;  // 8-byte unit of the row
          const uint2 v =
              *reinterpret_cast<const uint2*>(t + row * kTRow + 16 * ((u >> 1) ^ ((row >> 1) & 7)) + 8 * (u & 1));
          hv[j][0] = bf16_low(v.x);
          hv[j][1] = bf16_high(v.x);
          hv[j][2] = bf16_low(v.y);
          hv[j][3] = bf16_high(v.y);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[i][e], hv[j][e], acc[i][j], 0, 0, 0);
      }
    } else {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        uint4 fw[FT], ft[2];
#pragma unroll
        for (int i = 0; i < FT; ++i) {
          const int row = wf + 16 * i + r;
          fw[i] = *reinterpret_cast<const uint4*>(w + row * kWRow + 16 * ((4 * ks + g) ^ ((row >> 1) & 7)));
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int row = wt + 16 * j + r;
          ft[j] = *reinterpret_cast<const uint4*>(t + row * kTRow + 16 * ((4 * ks + g) ^ ((row >> 1) & 7)));
        }
#pragma unroll
        for (int i = 0; i < FT; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) acc[i][j] = mfma_16x16x32(Bf16Tag{}, fw[i], ft[j], acc[i][j]);
      }
    }
  }
  // Lane (r, g) of tile (i, j) holds features f0 + wf + 16 i + 4 g .. + 3 of
  // token t0 + wt + 16 j + r (features % 4 == 0: all four in or out).
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int token = t0 + wt + 16 * j + r;
    if (token >= a.tokens) continue;
    float* out = a.parts + ((int64_t)split * a.tokens + token) * a.features;
#pragma unroll
    for (int i = 0; i < FT; ++i) {
      const int f = f0 + wf + 16 * i + 4 * g;
      if (f < a.features) *reinterpret_cast<floatx4*>(out + f) = acc[i][j];
    }
  }
}

// The sum of a row's partial sums at four consecutive features, in the order
// of k.
__device__ __forceinline__ floatx4 sum_parts(const float* parts, int64_t at, int64_t stride, int splits) {
  floatx4 sum = *reinterpret_cast<const floatx4*>(parts + at);
#pragma unroll 4
  for (int s = 1; s < splits; ++s) sum += *reinterpret_cast<const floatx4*>(parts + s * stride + at);
  return sum;
}

// weights_proj's rows from their partial sums: one fp32 product with the
// head-weight scale.
__global__ __launch_bounds__(256) void finish_weights_kernel(const float* parts, int splits, int64_t quads,
                                                             float scale, float* out) {
  const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (q >= quads) return;
  const floatx4 v = sum_parts(parts, 4 * q, 4 * quads, splits);
  *reinterpret_cast<float4*>(out + 4 * q) = make_float4(v[0] * scale, v[1] * scale, v[2] * scale, v[3] * scale);
}

// The keys' rows from wk's partial sums (sidecar.py:74-76): the projection
// rounded to bf16, LayerNorm in fp32 rounded to bf16, the rotation in bf16
// steps, as encode_rows_kernel rounds them.  32 threads per token, four
// features each.
struct KeysArgs {
  const float* parts;
  int32_t splits, tokens;
  const void* ln_weight;  // [128] fp32, or bf16 with ln_bf16
  const void* ln_bias;
  int32_t ln_bf16;
  float ln_eps;
  const int64_t* positions;
  float theta;
  uint16_t* out;
  int64_t out_stride;
  const int64_t* out_rows;  // nullable: output row of each token
  int64_t out_row_limit;
};

__global__ __launch_bounds__(256) void finish_keys_kernel(KeysArgs a) {
  const int c = threadIdx.x & 31;
  const int token = blockIdx.x * 8 + (threadIdx.x >> 5);
  const int t = min(token, a.tokens - 1);
  floatx4 sum = sum_parts(a.parts, (int64_t)t * kHeadDim + 4 * c, (int64_t)a.tokens * kHeadDim, a.splits);
  uint32_t cs[4];
  float ln_w[4], ln_b[4], y[4];
  // The token's 32 threads compute one rotation entry each and exchange them.
  const uint32_t entry = rope_entry(a.positions[t], c, a.theta);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    cs[e] = __shfl(entry, (threadIdx.x & 32) + 4 * (c & 7) + e, kWave);
    const int d = 4 * c + e;
    ln_w[e] = a.ln_bf16 ? __uint_as_float((uint32_t) static_cast<const uint16_t*>(a.ln_weight)[d] << 16)
                        : static_cast<const float*>(a.ln_weight)[d];
    ln_b[e] = a.ln_bf16 ? __uint_as_float((uint32_t) static_cast<const uint16_t*>(a.ln_bias)[d] << 16)
                        : static_cast<const float*>(a.ln_bias)[d];
    y[e] = round_bf16f(sum[e]);
  }
  float total = (y[0] + y[1]) + (y[2] + y[3]);
#pragma unroll
  for (int off = 16; off > 0; off >>= 1) total += __shfl_xor(total, off, kWave);
  const float mean = total / (float)kHeadDim;
  float sq = 0.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) sq = fmaf(y[e] - mean, y[e] - mean, sq);
#pragma unroll
  for (int off = 16; off > 0; off >>= 1) sq += __shfl_xor(sq, off, kWave);
  const float rstd = 1.f / sqrtf(sq / (float)kHeadDim + a.ln_eps);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    y[e] = round_bf16f(__fadd_rn(__fmul_rn(__fmul_rn(y[e] - mean, rstd), ln_w[e]), ln_b[e]));
    // Dims below 64 rotate: thread c < 8 with thread c + 8.
    const float other = __shfl_xor(y[e], 8, kWave);
    const float a0 = round_bf16f(y[e] * bf16_high(cs[e]));
    const float b0 = round_bf16f(other * bf16_low(cs[e]));
    if (c < 16) y[e] = c < 8 ? round_bf16f(a0 - b0) : round_bf16f(a0 + b0);
  }
  if (token >= a.tokens) return;
  const int64_t row = a.out_rows ? a.out_rows[t] : t;
  if (row < 0 || row >= a.out_row_limit) return;
  *reinterpret_cast<uint2*>(a.out + row * a.out_stride + 4 * c) =
      make_uint2(pack_bf16(y[0], y[1]), pack_bf16(y[2], y[3]));
}

// fp32 weights: a workgroup owns 64 features x 16 tokens and its four waves
// split k in four; each wave loads its MFMA operands straight from memory
// (both are read from L2 many times over, by the token tiles and the
// feature tiles).  For a chunk of 16 k, lane (r, g) loads weight row r and
// token r at k = 16 q + 4 g .. + 3 and feeds element j to k-step j of
// v_mfma_f32_16x16x4_f32: both operands use that same order of k, so the
// product is the plain sum.  (bf16 hidden: chunks of 32 k, 8 values a lane.)
// kF32Ahead chunks are in flight per wave.  The four partial sums are added in
// LDS in a fixed order.
constexpr int kF32Feat = 64;
constexpr int kF32Tok = 16;

// kHiddenF32 is a template parameter because a branch on it beside every load
// had split the pipelined loop into blocks that each waited for all loads.
template <bool kHiddenF32>
__global__ __launch_bounds__(256) void gemm_f32_kernel(GemmArgs a) {
  constexpr int kPer = kHiddenF32 ? 4 : 8;  // k of a chunk per lane
  constexpr int kF32Ahead = 32 / kPer;
  __shared__ float red[4][64][17];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int r = lane & 15;
  const int g = lane >> 4;
  const int feature_tiles = (a.features + kF32Feat - 1) / kF32Feat;
  const int f0 = (int)(blockIdx.x % (uint32_t)feature_tiles) * kF32Feat;
  const int t0 = (int)(blockIdx.x / (uint32_t)feature_tiles) * kF32Tok;
  const int kdim = a.kdim;
  const int chunks = (kdim + 4 * kPer - 1) / (4 * kPer);
  const int per = (chunks + 3) / 4;  // chunks of this wave: [wave * per, min(chunks, wave * per + per))
  const int q0 = wave * per;
  const int q1 = min(chunks, q0 + per);
  constexpr int hbytes = kHiddenF32 ? 4 : 2;
  const BufferRsrc wr = make_buffer(a.weight, (uint32_t)a.features * (uint32_t)kdim * 4u);
  const BufferRsrc hr =
      make_buffer(a.hidden, (uint32_t)(((int64_t)(a.tokens - 1) * a.hidden_stride + kdim) * hbytes));
  uint32_t wbase[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int f = f0 + 16 * i + r;
    wbase[i] = f < a.features ? (uint32_t)f * (uint32_t)kdim * 4u : kFar;
  }
  const int t = t0 + r;
  const uint32_t hbase = t < a.tokens ? (uint32_t)((int64_t)t * a.hidden_stride * hbytes) : kFar;
  auto load = [&](int q, uint4 (&wv)[4][kPer / 4], uint4& hv) {
    const int k = kPer * (4 * q + g);
    const bool in = q < q1 && k < kdim;  // kdim % 8 == 0: a lane's values are all in or all out
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int h = 0; h < kPer / 4; ++h)
        wv[i][h] = buffer_load_16(wr, in && wbase[i] != kFar ? wbase[i] + (uint32_t)(k + 4 * h) * 4u : kFar);
    hv = buffer_load_16(hr, in && hbase != kFar ? hbase + (uint32_t)k * (uint32_t)hbytes : kFar);
  };
  floatx4 acc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] = floatx4{0.f, 0.f, 0.f, 0.f};
  uint4 wv[kF32Ahead][4][kPer / 4];
  uint4 hv[kF32Ahead];  // as loaded: bf16 widened on use, or the widening waits for every chunk's loads
#pragma unroll
  for (int s = 0; s < kF32Ahead; ++s) {
    load(q0 + s, wv[s], hv[s]);
    __builtin_amdgcn_sched_barrier(0);
  }
  for (int q = q0; q < q1; q += kF32Ahead) {
#pragma unroll
    for (int s = 0; s < kF32Ahead; ++s) {
      // chunk q + s is in registers; chunks past q1 read zeros
      const uint32_t h[4] = {hv[s].x, hv[s].y, hv[s].z, hv[s].w};
#pragma unroll
      for (int j = 0; j < kPer; ++j) {
        const float b = kHiddenF32 ? __uint_as_float(h[j & 3]) : j & 1 ? bf16_high(h[j >> 1]) : bf16_low(h[j >> 1]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint4 w = wv[s][i][j >> 2];
          const uint32_t wbits = (j & 3) == 0 ? w.x : (j & 3) == 1 ? w.y : (j & 3) == 2 ? w.z : w.w;
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(wbits), b, acc[i], 0, 0, 0);
        }
      }
      load(q + s + kF32Ahead, wv[s], hv[s]);
      // Left to itself the scheduler moves every load behind the last product
      // of the iteration, and the next one waits for all of them: 2048 x 64 and
      // x 8192 from fp32 hidden of 2048, 28.1 and 1266 us against 22.9 and 1199.
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // Lane (r, g) of tile i holds features f0 + 16 i + 4 g + e of token t0 + r.
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) red[wave][lane][4 * i + e] = acc[i][e];
  __syncthreads();
  if (wave == 0 && t < a.tokens) {
    float* out = static_cast<float*>(a.out) + (int64_t)t * a.out_stride;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int f = f0 + 16 * i + 4 * g + e;
        const float sum = ((red[0][lane][4 * i + e] + red[1][lane][4 * i + e]) + red[2][lane][4 * i + e]) +
                          red[3][lane][4 * i + e];
        if (f < a.features) out[f] = sum * a.scale;
      }
  }
}

template <int BF, int BT, int WF, int WT, bool kRope, int NPF>
int launch_bf16(const GemmArgs& a, hipStream_t stream) {
  const int64_t grid = (int64_t)((a.features + BF - 1) / BF) * ((a.tokens + BT - 1) / BT);
  if (grid > 0x7fffffffLL) return fail(DSA_STATUS_INVALID_ARGUMENT, "problem too large");
  hipLaunchKernelGGL((gemm_bf16_kernel<BF, BT, WF, WT, kRope, NPF>), dim3((unsigned)grid), dim3(64 * WF * WT), 0,
                     stream, a);
  return check_launch("gemm_bf16_kernel");
}

template <bool kF32>
int64_t narrow_ftiles(int64_t features) {
  return (features + kNarrowFeat<kF32> - 1) / kNarrowFeat<kF32>;
}

// k per workgroup of the narrow products: as many workgroups as the CUs take at
// once (a workgroup's registers fill a CU).  At least 192 instead sent some
// counts into a half-empty second round: encode_keys at 3000 x 1000 (376
// workgroups against 188) 18.5 -> 13.6 us, 2304 x 2048 16.9 -> 13.9, 300 x 7168
// 19.4 -> 13.9.  Feature tiles count as well: without them 8192 fp32 features took
// 137 us at 200 x 2048 and 582 at 1000 x 2048, now 92 and 352.
int32_t narrow_k(int64_t tokens, int64_t kdim, int64_t ftiles) {
  const int64_t tiles = (tokens + kNarrowTok - 1) / kNarrowTok * ftiles;
  int64_t kper = kNarrowK;
  while (kper > 2 * kGemmBK && tiles * ((kdim + kper / 2 - 1) / (kper / 2)) <= 256) kper /= 2;
  return (int32_t)kper;
}

// Tokens whose partial sums one launch leaves: at most kNarrowParts bytes of
// them, so that the workspace does not grow with the batch (the fp32 wq of
// 4096 tokens, hidden 2048, would leave 512 MiB, of 65000 tokens 8 GiB); longer
// batches take a launch per slice.
constexpr int64_t kNarrowParts = int64_t(64) << 20;
int64_t narrow_slice(int64_t tokens, int64_t kdim, int64_t features, int64_t ftiles) {
  const int64_t kper = narrow_k(tokens, kdim, ftiles);
  const int64_t token_bytes = (kdim + kper - 1) / kper * features * (int64_t)sizeof(float);
  const int64_t most = std::max<int64_t>(kNarrowParts / token_bytes / kNarrowTok, 1) * kNarrowTok;
  return std::min(tokens, most);
}

int64_t narrow_parts_bytes(int64_t tokens, int64_t kdim, int64_t features, int64_t ftiles) {
  const int64_t kper = narrow_k(tokens, kdim, ftiles);
  return (kdim + kper - 1) / kper * narrow_slice(tokens, kdim, features, ftiles) * features * (int64_t)sizeof(float);
}

// Partial sums of a narrow product over the slice of a.tokens (of `batch`, from
// which k's split follows), with the rotation table of `rope` (its table
// nullable) beside it.
template <bool kF32>
int launch_narrow(NarrowArgs& a, int64_t batch, const RopeTableArgs& rope, hipStream_t stream) {
  const int64_t ftiles = narrow_ftiles<kF32>(a.features);
  a.kper = narrow_k(batch, a.kdim, ftiles);
  a.splits = (a.kdim + a.kper - 1) / a.kper;
  const int64_t blocks = a.splits * ftiles * ((a.tokens + kNarrowTok - 1) / kNarrowTok);
  const int64_t grid = blocks + (rope.table ? rope_table_blocks(rope.tokens) : 0);
  if (grid > 0x7fffffffLL) return fail(DSA_STATUS_INVALID_ARGUMENT, "problem too large");
  hipLaunchKernelGGL(gemm_narrow_kernel<kF32>, dim3((unsigned)grid), dim3(256), 0, stream, a, rope, (int)blocks);
  return check_launch("gemm_narrow_kernel");
}

// bf16 products of whole 256-feature tiles (kRope: 128-dim heads rotated from
// a.rope).  The wide tile wherever it gives kWideMin CUs one; below, the
// largest token tile that still gives that many workgroups.  encode_queries'
// wq at hidden 2048 (8192 features), us for the whole call: at 1280 tokens (160
// wide tiles) 84 against 97 with 128-token tiles, at 1000 (128 wide tiles) 82
// against 77; 256-token tiles of eight waves, the only ones before, took 95
// and 96 there, and 89 at 17 to 128 tokens, where 32-token tiles take 46;
// 64-token tiles take 51 at 200 against 58 with 128-token tiles and 55 with
// 32-token ones, 128-token tiles 59 at 400 against 61 and 72.  At hidden 512,
// 1024, 2048, 4096 and 7168 no count of 17 to 8192 tokens is slower than the
// 256-token tiles of eight waves alone (0.23 to 0.82 of their time).
//
// Hidden 1000, 256- against 128-token tiles: 2000 tokens (256 tiles of 256 x
// 256) 63 / 75 us, 4096 (512) 113 / 133, 3000 (384, three quarters of two
// rounds) 110 / 105; hidden 4040: 2048 tokens 165 / 208, 8192 567 / 742.
constexpr int64_t kWideMin = 160;
template <bool kRope>
int launch_bf16_features(const GemmArgs& a, hipStream_t stream) {
  auto groups = [&](int64_t features, int64_t tokens) {
    return (a.features + features - 1) / features * ((a.tokens + tokens - 1) / tokens);
  };
  const int64_t tiles = groups(kWideTile, kWideTile);
  if (tiles >= kWideMin && tiles <= 0x7fffffffLL && a.kdim % kGemmBK == 0 && a.kdim <= (1 << 16)) {
    hipLaunchKernelGGL(gemm_wide_kernel<kRope>, dim3((unsigned)std::min<int64_t>(tiles, kWideGrid)), dim3(256), 0,
                       stream, a, (int)tiles);
    return check_launch("gemm_wide_kernel");
  }
  // A kdim that is no multiple of 64: the same tiles on eight waves, one
  // workgroup per CU, where they fill their last round to seven eighths.
  const int64_t rounds = (tiles + kWideGrid - 1) / kWideGrid;
  if (8 * tiles >= 7 * rounds * kWideGrid) return launch_bf16<256, 256, 2, 4, kRope, 1>(a, stream);
  if (groups(128, 128) >= kWideMin) return launch_bf16<128, 128, 2, 4, kRope, 1>(a, stream);
  if (groups(128, 64) >= kWideMin) return launch_bf16<128, 64, 2, 2, kRope, 2>(a, stream);
  return launch_bf16<128, 32, 2, 2, kRope, 4>(a, stream);
}

}  // namespace
}  // namespace dsa

using namespace dsa;

extern "C" int64_t dsa_project_gemm_workspace_bytes(int64_t tokens) {
  return tokens > 0 ? tokens * kRopeHalf * (int64_t)sizeof(uint32_t) : 0;
}

extern "C" int dsa_project_gemm(const void* hidden, int32_t hidden_dtype, int64_t hidden_stride, int64_t tokens,
                                int64_t kdim, const void* weight, int32_t weight_dtype, int64_t features, void* out,
                                int64_t out_stride, float out_scale, const int64_t* positions, float theta,
                                void* workspace, int64_t workspace_bytes, void* stream) {
  DSA_REQUIRE(hidden && weight && out, "null pointer argument");
  DSA_REQUIRE(tokens > 0 && tokens <= 0x7fffffffLL, "tokens %lld out of range", (long long)tokens);
  DSA_REQUIRE(kdim > 0 && kdim % 8 == 0, "kdim %lld must be a positive multiple of 8", (long long)kdim);
  DSA_REQUIRE(features > 0 && features % 4 == 0, "features %lld must be a positive multiple of 4",
              (long long)features);
  DSA_REQUIRE(hidden_stride >= kdim && hidden_stride % 8 == 0, "hidden_stride must be >= kdim and a multiple of 8");
  DSA_REQUIRE(out_stride >= features && out_stride % 4 == 0, "out_stride must be >= features and a multiple of 4");
  DSA_REQUIRE(reinterpret_cast<uintptr_t>(hidden) % 16 == 0 && reinterpret_cast<uintptr_t>(weight) % 16 == 0 &&
                  reinterpret_cast<uintptr_t>(out) % 16 == 0,
              "hidden, weight and out must be 16-byte aligned");
  DSA_REQUIRE(hidden_dtype == kBF16 || (hidden_dtype == kF32 && weight_dtype == kF32),
              "hidden must be bf16 (or fp32 with fp32 weights)");
  DSA_REQUIRE(weight_dtype == kBF16 || weight_dtype == kF32, "weights must be bf16 or fp32");
  const int64_t hidden_bytes = ((tokens - 1) * hidden_stride + kdim) * (hidden_dtype == kF32 ? 4 : 2);
  const int64_t out_bytes = ((tokens - 1) * out_stride + features) * (weight_dtype == kF32 ? 4 : 2);
  DSA_REQUIRE(hidden_bytes < (int64_t(1) << 31) && out_bytes < (int64_t(1) << 31) &&
                  features * kdim * (weight_dtype == kF32 ? 4 : 2) < (int64_t(1) << 31),
              "hidden, weight and out must each be below 2 GiB");
  GemmArgs a = {};
  a.hidden = static_cast<const uint16_t*>(hidden);
  a.hidden_stride = hidden_stride;
  a.weight = weight;
  a.out = out;
  a.out_stride = out_stride;
  a.tokens = (int32_t)tokens;
  a.features = (int32_t)features;
  a.kdim = (int32_t)kdim;
  a.scale = out_scale;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (weight_dtype == kF32) {
    DSA_REQUIRE(!positions, "the fused RoPE takes bf16 weights");
    DSA_REQUIRE(kdim % 4 == 0 && hidden_stride % 4 == 0, "fp32 projections need kdim and hidden_stride divisible by 4");
    const int64_t grid = ((features + kF32Feat - 1) / kF32Feat) * ((tokens + kF32Tok - 1) / kF32Tok);
    DSA_REQUIRE(grid <= 0x7fffffffLL, "problem too large");
    if (hidden_dtype == kF32)
      hipLaunchKernelGGL(gemm_f32_kernel<true>, dim3((unsigned)grid), dim3(256), 0, s, a);
    else
      hipLaunchKernelGGL(gemm_f32_kernel<false>, dim3((unsigned)grid), dim3(256), 0, s, a);
    return check_launch("gemm_f32_kernel");
  }
  DSA_REQUIRE(out_scale == 1.f, "bf16 projections take no output scale");
  if (positions) {
    // Query projection with the fused RoPE of every 128-dim head.
    DSA_REQUIRE(features % 256 == 0, "the fused RoPE needs whole pairs of 128-dim heads (features a multiple of 256)");
    DSA_REQUIRE(workspace && workspace_bytes >= dsa_project_gemm_workspace_bytes(tokens) &&
                    reinterpret_cast<uintptr_t>(workspace) % 16 == 0,
                "the fused RoPE needs dsa_project_gemm_workspace_bytes(tokens) bytes of 16-byte aligned workspace");
    a.rope = static_cast<const uint32_t*>(workspace);
    hipLaunchKernelGGL(rope_table_kernel, dim3((unsigned)rope_table_blocks(tokens)), dim3(256), 0, s,
                       RopeTableArgs{positions, static_cast<uint32_t*>(workspace), (int32_t)tokens, theta});
    if (int st = check_launch("rope_table_kernel")) return st;
    return launch_bf16_features<true>(a, s);
  }
  if (features % 256 == 0) return launch_bf16_features<false>(a, s);
  return launch_bf16<128, 32, 2, 2, false, 4>(a, s);
}

extern "C" int64_t dsa_project_weights_workspace_bytes(int64_t tokens, int64_t kdim, int64_t features) {
  if (tokens <= 0 || kdim <= 0 || features <= 0) return 0;
  return narrow_parts_bytes(tokens, kdim, features, narrow_ftiles<true>(features));
}

// Shared by the two entry points below: weights_proj's partial sums (with the
// rotation table of `rope` beside them) and their sums.
static int project_weights(const GemmArgs& a, const float* weight, int64_t features, float scale, float* out,
                           void* parts, const RopeTableArgs& rope, hipStream_t s) {
  DSA_REQUIRE(features > 0 && features % 4 == 0, "features %lld must be a positive multiple of 4",
              (long long)features);
  DSA_REQUIRE(features * a.kdim * 4 < (int64_t(1) << 31), "the fp32 weights must be below 2 GiB");
  DSA_REQUIRE(reinterpret_cast<uintptr_t>(weight) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0,
              "the fp32 weights and their output must be 16-byte aligned");
  DSA_REQUIRE((int64_t)a.tokens * features * 4 < (int64_t(1) << 31), "the fp32 output must be below 2 GiB");
  const int64_t slice = narrow_slice(a.tokens, a.kdim, features, narrow_ftiles<true>(features));
  for (int64_t t0 = 0; t0 < a.tokens; t0 += slice) {
    NarrowArgs w = {};
    w.hidden = a.hidden + t0 * a.hidden_stride;
    w.hidden_stride = a.hidden_stride;
    w.weight = weight;
    w.tokens = (int32_t)std::min<int64_t>(slice, a.tokens - t0);
    w.features = (int32_t)features;
    w.kdim = a.kdim;
    w.parts = static_cast<float*>(parts);
    if (int st = launch_narrow<true>(w, a.tokens, t0 == 0 ? rope : RopeTableArgs{}, s)) return st;
    const int64_t quads = (int64_t)w.tokens * features / 4;
    hipLaunchKernelGGL(finish_weights_kernel, dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, s, w.parts, w.splits,
                       quads, scale, out + t0 * features);
    if (int st = check_launch("finish_weights_kernel")) return st;
  }
  return 0;
}

extern "C" int dsa_project_weights(const void* hidden, int64_t hidden_stride, int64_t tokens, int64_t kdim,
                                   const float* weight, int64_t features, float scale, float* out, void* workspace,
                                   int64_t workspace_bytes, void* stream) {
  DSA_REQUIRE(hidden && weight && out, "null pointer argument");
  DSA_REQUIRE(tokens > 0 && tokens <= 0x7fffffffLL, "tokens %lld out of range", (long long)tokens);
  DSA_REQUIRE(kdim > 0 && kdim % 8 == 0, "kdim %lld must be a positive multiple of 8", (long long)kdim);
  DSA_REQUIRE(hidden_stride >= kdim && hidden_stride % 8 == 0, "hidden_stride must be >= kdim and a multiple of 8");
  DSA_REQUIRE(reinterpret_cast<uintptr_t>(hidden) % 16 == 0, "hidden must be 16-byte aligned");
  DSA_REQUIRE(((tokens - 1) * hidden_stride + kdim) * 2 < (int64_t(1) << 31), "hidden must be below 2 GiB");
  if (!workspace || workspace_bytes < dsa_project_weights_workspace_bytes(tokens, kdim, features) ||
      reinterpret_cast<uintptr_t>(workspace) % 16 != 0)
    return fail(DSA_STATUS_WORKSPACE_TOO_SMALL,
                "needs dsa_project_weights_workspace_bytes(tokens, kdim, features) bytes of 16-byte aligned workspace");
  GemmArgs a = {};
  a.hidden = static_cast<const uint16_t*>(hidden);
  a.hidden_stride = hidden_stride;
  a.tokens = (int32_t)tokens;
  a.kdim = (int32_t)kdim;
  return project_weights(a, weight, features, scale, out, workspace, RopeTableArgs{},
                         static_cast<hipStream_t>(stream));
}

extern "C" int64_t dsa_encode_queries_workspace_bytes(int64_t tokens, int64_t kdim, int64_t heads) {
  if (tokens <= 0 || kdim <= 0 || heads <= 0) return 0;
  return dsa_project_gemm_workspace_bytes(tokens) +
         narrow_parts_bytes(tokens, kdim, heads, narrow_ftiles<true>(heads));
}

extern "C" int64_t dsa_encode_keys_workspace_bytes(int64_t tokens, int64_t kdim, int64_t dim) {
  if (tokens <= 0 || kdim <= 0 || dim <= 0) return 0;
  return std::max(tokens * dim * 2, tokens > 16 && dim == kHeadDim ? narrow_parts_bytes(tokens, kdim, dim, 1) : 0);
}

extern "C" int dsa_encode_queries_gemm(const void* hidden, int64_t hidden_stride, int64_t tokens, int64_t kdim,
                                       const void* wq, int32_t heads, const float* weights_proj,
                                       const int64_t* positions, float theta, float weight_scale, void* out_queries,
                                       float* out_weights, void* workspace, int64_t workspace_bytes, void* stream) {
  const int64_t features = (int64_t)heads * kHeadDim;
  DSA_REQUIRE(hidden && wq && weights_proj && positions && out_queries && out_weights, "null pointer argument");
  DSA_REQUIRE(tokens > 0 && tokens <= 0x7fffffffLL / kRopeHalf, "tokens %lld out of range", (long long)tokens);
  DSA_REQUIRE(kdim > 0 && kdim % 8 == 0, "kdim %lld must be a positive multiple of 8", (long long)kdim);
  DSA_REQUIRE(heads > 0 && heads % 4 == 0, "heads %d must be a positive multiple of 4", heads);
  DSA_REQUIRE(hidden_stride >= kdim && hidden_stride % 8 == 0, "hidden_stride must be >= kdim and a multiple of 8");
  DSA_REQUIRE(reinterpret_cast<uintptr_t>(hidden) % 16 == 0 && reinterpret_cast<uintptr_t>(wq) % 16 == 0 &&
                  reinterpret_cast<uintptr_t>(out_queries) % 16 == 0,
              "hidden, wq and out_queries must be 16-byte aligned");
  DSA_REQUIRE(((tokens - 1) * hidden_stride + kdim) * 2 < (int64_t(1) << 31) &&
                  tokens * features * 2 < (int64_t(1) << 31) && features * kdim * 2 < (int64_t(1) << 31),
              "hidden, wq and out_queries must each be below 2 GiB");
  DSA_REQUIRE(workspace && workspace_bytes >= dsa_encode_queries_workspace_bytes(tokens, kdim, heads) &&
                  reinterpret_cast<uintptr_t>(workspace) % 16 == 0,
              "needs dsa_encode_queries_workspace_bytes(tokens, kdim, heads) bytes of 16-byte aligned workspace");
  hipStream_t s = static_cast<hipStream_t>(stream);
  GemmArgs a = {};
  a.hidden = static_cast<const uint16_t*>(hidden);
  a.hidden_stride = hidden_stride;
  a.tokens = (int32_t)tokens;
  a.kdim = (int32_t)kdim;
  uint32_t* table = static_cast<uint32_t*>(workspace);
  if (int st = project_weights(a, weights_proj, heads, weight_scale, out_weights,
                               static_cast<uint8_t*>(workspace) + dsa_project_gemm_workspace_bytes(tokens),
                               RopeTableArgs{positions, table, (int32_t)tokens, theta}, s))
    return st;
  a.weight = wq;
  a.features = (int32_t)features;
  a.out = out_queries;
  a.out_stride = features;
  a.rope = table;
  return launch_bf16_features<true>(a, s);
}

namespace dsa {

// encode_keys of bf16 rows of 128 dims, 64 of them rotated: wk's partial sums
// into `parts`, then the rows (finish_keys_kernel).
int launch_encode_keys_gemm(const void* hidden, int64_t hidden_stride, int64_t tokens, int64_t kdim, const void* wk,
                            void* parts, const void* ln_weight, const void* ln_bias, bool ln_bf16, float ln_eps,
                            const int64_t* positions, float theta, void* out, int64_t out_stride,
                            const int64_t* out_rows, int64_t out_row_limit, hipStream_t stream) {
  DSA_REQUIRE(hidden_stride >= kdim && hidden_stride % 8 == 0, "hidden_stride must be >= kdim and a multiple of 8");
  DSA_REQUIRE(reinterpret_cast<uintptr_t>(hidden) % 16 == 0 && reinterpret_cast<uintptr_t>(wk) % 16 == 0,
              "hidden and wk must be 16-byte aligned");
  DSA_REQUIRE(((tokens - 1) * hidden_stride + kdim) * 2 < (int64_t(1) << 31) &&
                  kHeadDim * kdim * 2 < (int64_t(1) << 31),
              "hidden and wk must each be below 2 GiB");
  const int64_t slice = narrow_slice(tokens, kdim, kHeadDim, 1);
  for (int64_t t0 = 0; t0 < tokens; t0 += slice) {
    NarrowArgs w = {};
    w.hidden = static_cast<const uint16_t*>(hidden) + t0 * hidden_stride;
    w.hidden_stride = hidden_stride;
    w.weight = wk;
    w.tokens = (int32_t)std::min(slice, tokens - t0);
    w.features = kHeadDim;
    w.kdim = (int32_t)kdim;
    w.parts = static_cast<float*>(parts);
    if (int st = launch_narrow<false>(w, tokens, RopeTableArgs{}, stream)) return st;
    KeysArgs a = {};
    a.parts = w.parts;
    a.splits = w.splits;
    a.tokens = w.tokens;
    a.ln_weight = ln_weight;
    a.ln_bias = ln_bias;
    a.ln_bf16 = ln_bf16;
    a.ln_eps = ln_eps;
    a.positions = positions + t0;
    a.theta = theta;
    a.out = static_cast<uint16_t*>(out) + (out_rows ? 0 : t0 * out_stride);
    a.out_stride = out_stride;
    a.out_rows = out_rows ? out_rows + t0 : nullptr;
    a.out_row_limit = out_rows ? out_row_limit : w.tokens;
    hipLaunchKernelGGL(finish_keys_kernel, dim3((unsigned)((w.tokens + 7) / 8)), dim3(256), 0, stream, a);
    if (int st = check_launch("finish_keys_kernel")) return st;
  }
  return 0;
}

}  // namespace dsa
