// Grouped GEMM in fp32 on the bf16 matrix instruction: every value is split into three bf16 parts (24 bits, Chunk below), and the
// six products of parts that reach 2^-18 of a product are summed in fp32 (v_mfma_f32_16x16x32_bf16).
//
// What bounds it: the matrix cores and the power they draw.  The fp32 instruction (v_mfma_f32_16x16x4_f32) does 256 FLOP
// per cycle and compute unit, the bf16 one 4096, a sixth of which is 683.  Next to a product there is room for two vector-ALU
// instructions per SIMD (measured: 2 are free, 3 cost a fifth, 4 half of the rate), and a value takes six to become parts.  So a
// workgroup converts a value once, on its way to the LDS, and its waves multiply parts: 1.7 instructions per product.  When every
// wave converted what it read, 4 per product, the matrix cores were busy 45 - 50 % of the time, now 55 - 59 %, at 2.0 GHz instead
// of 2.1.  8 experts of 1024 +- 30 rows, [1024, 4096], normal values: 376 / 379 / 352 us NT / NN / TN (operands in the last-level cache or
// not) against 460 / 459 / 408 that way and 947 / 983 / 882 in the element-wise kernel of gmm.hip, which serves every alignment; 4096^3: 626 /
// 643 / 646 us, 220 - 213 TFLOP/s, against 799 / 802 / 783 (torch.mm: 1067 - 1071).  On the fp32 instruction the first three were some 40 %
// longer than here.  Reductions of a dozen K tiles or less in small launches, whose time is the latency of a K tile's way through registers and
// LDS, are 1 - 3 us longer than when operands went to the LDS directly (24 experts of 74, [128, 256], NT: 13.3 / 10.5).  Keeping the
// pipeline filled across a workgroup's tiles changed nothing; cutting the parts off instead of rounding them is 3 % faster and up to a third less exact.
//
// How exact: three parts hold all 24 bits of a value; the three products of parts not taken come to less than 2^-25 of a product,
// and an accumulator is rounded six times per 32 k instead of 32 times.  Relative error (2-norm) against fp64: 4.8e-7 over
// k = 1024, 9.8e-7 over 4096, where a chain of fp32 fused multiply-adds shows 5.7e-7 and 1.15e-6; 3.1e-8 over eight terms (5.4e-8).
// The small tile, which puts its sums aside every 256 terms: 2.3e-7 over 1024 terms of which a launch that is cut into four parts made
// 2.3e-7 too, 2.4e-7 over 4096 (3.5e-7 cut into eight).
// The error of a single product is larger than that chain's, up to 2.6 2^-24 of it instead of one: sums of one or two terms,
// and those that the parts do not serve (infinities, NaN, values next to the largest or the smallest), are formed on the fp32
// instruction: multiply().
// Why not two fp16 parts of a value times a power of two of its row, and three products (4096^3: 403 / 412 / 411 us): they hold 22 bits, fewer
// below 2^-13 of the row's largest value and none below 2^-35, and a sum whose large values meet zeros of the other operand is made of just those
// (off by up to 0.14 of the sum of its terms' magnitudes).  The result does not show it, and a check of the operands for such values finds
// them in every tile: of normal values one in 3000 is that far below the largest of its row.
//
// Tile: 128 x 256 per workgroup of eight waves, two to a SIMD, K tiles of 32 in two stages of 72 KiB; 256 x 128 for TN products
// whose edges it leaves less empty (12 experts of 500 rows, [2728, 1032]: 252 -> 212 us); 64 x 128, 36 KiB a stage and two
// workgroups to a compute unit, for short experts, launches of few tiles and columns that leave the wide one half empty (f32_small_rows()).  Values pass through registers, a
// K tile ahead: while K tile kt is multiplied, kt + 1 is converted and written to the other stage, and the loads of kt + 2 go
// out into the registers that frees.  One barrier per K tile.
//
// LDS layout: the three parts of an operand tile, each [row][32 k] bf16: 64-byte rows, the 16-byte chunk of k = 8 q .. 8 q + 7 of
// row r at position q ^ x(r) (chunk_at), which neither the reads (16 rows, one chunk) nor the writes (64 rows of one chunk, or
// 16 whole rows) find in the same banks; x = (r >> 2) & 3 alone costs 14 % of the cycles in conflicts.  An operand whose reduction
// dimension is contiguous (KC) is loaded in 16-byte pieces, two to a chunk; one whose reduction dimension is strided (MC) in
// dwords, 64 consecutive columns to a load and eight k to a chunk, so that both end up in the same layout.
#include "gmm_common.h"

namespace mbx {
namespace {

#include "gmm_dma.h"   // buffer descriptors, LDS reads, tile lists

namespace f32 {

using dma::clamp_row;
using dma::clip_bytes;
using dma::lds_ptr;
using dma::make_rsrc;
using dma::RowTiles;
using dma::tile_done;

constexpr int kBK = 32, kThreads = 512;
constexpr uint32_t kRowBytes = kBK * 2;                    // a part of a row's K tile
constexpr int kMaxKSplit = 8, kMinPartTiles = 8;           // parts of a reduction, K tiles per part

// A tile of BM x BN and how the eight waves share it.
template <int BM_, int BN_>
struct Shape {
  static constexpr int BM = BM_, BN = BN_;
  static constexpr int WN = BM == 256 ? 2 : 4, WM = 8 / WN;                      // waves along the columns, the rows
  static constexpr int TM = BM / WM / 16, TN = BN / WN / 16;                     // 16 x 16 accumulator tiles of a wave
  static constexpr uint32_t kPlaneBytes = (BM + BN) * kRowBytes, kStageBytes = 3 * kPlaneBytes;
  static constexpr size_t kLdsBytes = 2 * kStageBytes;
  static constexpr size_t kPartBytes = (size_t)BM * BN * 4;                      // one tile's accumulators in the workspace
  static constexpr int kPerUnit = kLdsBytes > 80 * 1024 ? 1 : 2;                 // workgroups that share a compute unit
  // K tiles after which the sums so far are put aside and new ones begun (0: never).  Launches of few tiles get the small tile
  // and with it are cut along the reduction less often; what that took off the error of a long sum this does.
  static constexpr int kBlock = BM == 64 ? kMinPartTiles : 0;
  // Accumulator tile (i, j), register r of lane l is row row(wave) + 16 i + l % 16, column column(wave) + 16 j + 4 (l / 16) + r
  // of the workgroup's tile (the operands are swapped, so a lane owns runs of four consecutive columns).
  typedef f32x4 Acc[TM][TN];
  static __device__ __forceinline__ int row(int wave) { return wave / WN * (TM * 16); }
  static __device__ __forceinline__ int column(int wave) { return wave % WN * (TN * 16); }
};
typedef Shape<128, 256> Wide;    // the main tile
typedef Shape<256, 128> Tall;    // TN, where it leaves less of the product's edges empty
typedef Shape<64, 128> Small;    // NN / NT launches of few rows per expert, and those that leave compute units idle

// The operands of a tile: buffers (out-of-range bytes read as zero), row pitches in bytes, tile origins, the first and
// one past the last K tile to multiply, the length of the whole reduction (pieces of a row past it read as zeros).
// Two operand pairs (DUAL): K tiles nk1 .. 2 nk1 - 1 come from the second.
struct Args {
  __amdgpu_buffer_rsrc_t rsrc_a, rsrc_b, rsrc_a2, rsrc_b2;
  uint32_t a_ld, b_ld;
  int a_r0, b_r0, kt0, kt1, k, nk1;
};

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef const __attribute__((address_space(3))) u32x4* lds_in;
typedef __attribute__((address_space(3))) u32x4* lds_out;
typedef __attribute__((address_space(3))) u32x2* lds_out_half;

__device__ __forceinline__ f32x4 mfma(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// V (8 or 4) consecutive k of one row (column) of an operand on their way from memory to the LDS: the chunk of one thread.
// step() forms the three bf16 parts, v = part 0 + part 1 + part 2 up to 2^-27 |v|: every part is the rest the parts before
// it leave (the differences are exact), rounded to nearest.  In kSteps steps of a few instructions, to be put between
// products: step V / 2 q + p forms part q of the values 2 p and 2 p + 1, the last of a part stores it.
template <int V, uint32_t PLANE>
struct Chunk {
  static constexpr int kPairs = V / 2, kSteps = 3 * kPairs;
  float v[V];
  uint32_t part[kPairs];

  template <int X>
  __device__ __forceinline__ void step(float& largest, lds_ptr to) {   // largest: magnitude seen
    constexpr int q = X / kPairs, p = X % kPairs;
    if constexpr (q == 0) asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(largest) : "v"(v[2 * p]), "v"(v[2 * p + 1]));
    const uint32_t both = pack2<MBX_BF16>(v[2 * p], v[2 * p + 1]);
    part[p] = both;
    if constexpr (q < 2) {
      v[2 * p] -= __uint_as_float(both << 16);
      v[2 * p + 1] -= __uint_as_float(both & 0xffff0000u);
    }
    if constexpr (p == kPairs - 1) {
      if constexpr (V == 8) *(lds_out)(to + q * PLANE) = u32x4{part[0], part[1], part[2], part[3]};
      else *(lds_out_half)(to + q * PLANE) = u32x2{part[0], part[1]};
    }
  }
  // for the fp32 instruction: the values as they are, k 0 .. 3 of eight to one plane, 4 .. 7 to the next
  __device__ __forceinline__ void store_as_is(lds_ptr to, int half) const {
    if constexpr (V == 8) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
        *(lds_out)(to + h * PLANE) = u32x4{__float_as_uint(v[4 * h]), __float_as_uint(v[4 * h + 1]), __float_as_uint(v[4 * h + 2]), __float_as_uint(v[4 * h + 3])};
    } else {
      *(lds_out)(to + half * ((int)PLANE - 8)) = u32x4{__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])};
    }
  }
};

template <typename S>
__device__ __forceinline__ void clear(typename S::Acc& acc) {
#pragma unroll
  for (int i = 0; i < S::TM; ++i)
#pragma unroll
    for (int j = 0; j < S::TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
}

// acc += A_tile * B_tile over K tiles [g.kt0, g.kt1); largest: the largest magnitude among the operands (unless FP32)
template <bool A_MC, bool B_MC, typename S, bool DUAL, bool FP32>
__device__ __forceinline__ void multiply_as(const Args& g, typename S::Acc& acc, char* lds_generic, float& largest) {
  constexpr int TM = S::TM, TN = S::TN, kA = S::BM == 256 ? 2 : 1, kB = S::BN / 128, kChunks = kA + kB;   // chunks of a thread
  constexpr int kAV = S::BM == 64 ? 4 : 8;
  if (g.kt0 >= g.kt1) return;
  const lds_ptr lds = (lds_ptr)lds_generic;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = lane_id();

  // This thread's chunks: k = 8 q .. 8 q + 7 of rows r and r + 128 of A and of B; BM = 64: one half of eight k of a row of A.
  auto chunk_at = [&](int row, int q) -> uint32_t {
    const int b = row >> 2 & 3, x = (((b << 1 ^ b) & 2) | b >> 1) ^ (row >> 1 & 1);
    return (uint32_t)row * kRowBytes + (uint32_t)((q ^ x) << 4);
  };
  const int kc_r = threadIdx.x >> 2, kc_q = threadIdx.x & 3;                    // four lanes a row: 128 bytes of it
  const int half_r = A_MC ? lane : threadIdx.x >> 3, half_k = 4 * (A_MC ? wave : threadIdx.x & 7);   // eight lanes a row; 64 columns per load
  const int mc_r = lane + 64 * (wave >> 2), mc_q = wave & 3;                    // 64 consecutive columns per load
  const uint32_t a_to = kAV == 4 ? chunk_at(half_r, half_k >> 3) + (half_k & 4 ? 8u : 0u) : A_MC ? chunk_at(mc_r, mc_q) : chunk_at(kc_r, kc_q);
  const uint32_t b_to = S::BM * kRowBytes + (B_MC ? chunk_at(mc_r, mc_q) : chunk_at(kc_r, kc_q));
  const uint32_t a_lane = kAV == 4 ? (A_MC ? (uint32_t)half_k * g.a_ld + (uint32_t)(g.a_r0 + half_r) * 4u : (uint32_t)(g.a_r0 + half_r) * g.a_ld + (uint32_t)half_k * 4u)
                          : A_MC ? (uint32_t)(8 * mc_q) * g.a_ld + (uint32_t)(g.a_r0 + mc_r) * 4u
                                 : (uint32_t)(g.a_r0 + kc_r) * g.a_ld + (uint32_t)kc_q * 32u;
  const uint32_t b_lane = B_MC ? (uint32_t)(8 * mc_q) * g.b_ld + (uint32_t)(g.b_r0 + mc_r) * 4u
                               : (uint32_t)(g.b_r0 + kc_r) * g.b_ld + (uint32_t)kc_q * 32u;
  const uint32_t a_step = A_MC ? kBK * g.a_ld : kBK * 4u, b_step = B_MC ? kBK * g.b_ld : kBK * 4u;   // per K tile

  typedef Chunk<kAV, S::kPlaneBytes> ChunkA;
  typedef Chunk<8, S::kPlaneBytes> ChunkB;
  ChunkA ca[kA];
  ChunkB cb[kB];
  uint32_t a_at = 0, b_at = 0, past_half = 0, past_low = 0, past_high = 0;
  __amdgpu_buffer_rsrc_t ra = g.rsrc_a, rb = g.rsrc_b;
  auto load_at = [&](int kt) {
    const bool second = DUAL && kt >= g.nk1;
    const int kk = second ? kt - g.nk1 : kt;
    // bit 31 puts a load out of its buffer's range, so that it reads zeros: a K tile past the last, and the pieces of a row
    // past the end of the reduction (k is a multiple of 4), where the next row's values could be infinite
    const uint32_t none = kt < g.kt1 ? 0u : 0x80000000u;
    const int left = g.k - kk * kBK;
    past_half = left > half_k ? 0u : 0x80000000u;
    past_low = left > 8 * kc_q ? 0u : 0x80000000u;
    past_high = left > 8 * kc_q + 4 ? 0u : 0x80000000u;
    if (DUAL) { ra = second ? g.rsrc_a2 : g.rsrc_a; rb = second ? g.rsrc_b2 : g.rsrc_b; }
    a_at = (a_lane + (uint32_t)kk * a_step) | none;
    b_at = (b_lane + (uint32_t)kk * b_step) | none;
  };
  auto load_whole = [&](auto mc, ChunkB& to, const __amdgpu_buffer_rsrc_t& rsrc, uint32_t at, uint32_t ld, uint32_t number) {
    if constexpr (decltype(mc)::value) {
      at += number * (128 * 4);
#pragma unroll
      for (int u = 0; u < 8; ++u) to.v[u] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)(at + u * ld), 0, 0));
    } else {
      at += number * (128 * ld);
      const u32x4 low = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)(at | past_low), 0, 0));
      const u32x4 high = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)((at + 16) | past_high), 0, 0));
#pragma unroll
      for (int u = 0; u < 4; ++u) { to.v[u] = __uint_as_float(low[u]); to.v[4 + u] = __uint_as_float(high[u]); }
    }
  };
  auto load_a = [&](int number, ChunkA& to) {
    if constexpr (kAV == 4 && A_MC) {
#pragma unroll
      for (int u = 0; u < 4; ++u) to.v[u] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(ra, (int)(a_at + u * g.a_ld), 0, 0));
    } else if constexpr (kAV == 4) {
      const u32x4 w = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ra, (int)(a_at | past_half), 0, 0));
#pragma unroll
      for (int u = 0; u < 4; ++u) to.v[u] = __uint_as_float(w[u]);
    } else {
      load_whole(std::integral_constant<bool, A_MC>{}, to, ra, a_at, g.a_ld, number);
    }
  };
  auto load_b = [&](int number, ChunkB& to) { load_whole(std::integral_constant<bool, B_MC>{}, to, rb, b_at, g.b_ld, number); };
  auto a_chunk_to = [&](int number, uint32_t stage) -> lds_ptr { return lds + (a_to + stage) + number * (128 * kRowBytes); };
  auto b_chunk_to = [&](int number, uint32_t stage) -> lds_ptr { return lds + (b_to + stage) + number * (128 * kRowBytes); };

  const uint32_t frag_lane = chunk_at(lane & 15, lane >> 4);
  const uint32_t fa_at = (uint32_t)S::row(wave) * kRowBytes + frag_lane;
  const uint32_t fb_at = (uint32_t)(S::BM + S::column(wave)) * kRowBytes + frag_lane;
  u32x4 fa[3][TM], fb[3][TN];
  auto read_a = [&](auto qi, auto ii, uint32_t stage) {
    constexpr int q = decltype(qi)::value, i = decltype(ii)::value;
    fa[q][i] = *(lds_in)(lds + (fa_at + stage) + (q * S::kPlaneBytes + i * 16 * kRowBytes));
  };
  auto read_b = [&](auto qi, auto ji, uint32_t stage) {
    constexpr int q = decltype(qi)::value, j = decltype(ji)::value;
    fb[q][j] = *(lds_in)(lds + (fb_at + stage) + (q * S::kPlaneBytes + j * 16 * kRowBytes));
  };
  auto barrier = [&] {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
  };
  constexpr std::integral_constant<int, 0> c0{};
  constexpr std::integral_constant<int, 1> c1{};
  constexpr std::integral_constant<int, 2> c2{};

  // K tile kt0 into stage 0, K tile kt0 + 1 under way
  {
    ChunkA first_a[kA];
    ChunkB first_b[kB];
    load_at(g.kt0);
#pragma unroll
    for (int c = 0; c < kA; ++c) load_a(c, first_a[c]);
#pragma unroll
    for (int c = 0; c < kB; ++c) load_b(c, first_b[c]);
    load_at(g.kt0 + 1);
#pragma unroll
    for (int c = 0; c < kA; ++c) load_a(c, ca[c]);
#pragma unroll
    for (int c = 0; c < kB; ++c) load_b(c, cb[c]);
    dma::static_for<kA>([&](auto ci) {
      constexpr int c = decltype(ci)::value;
      if constexpr (FP32) first_a[c].store_as_is(a_chunk_to(c, 0), (half_k & 4) != 0);
      else dma::static_for<ChunkA::kSteps>([&](auto xi) { first_a[c].template step<decltype(xi)::value>(largest, a_chunk_to(c, 0)); });
    });
    dma::static_for<kB>([&](auto ci) {
      constexpr int c = decltype(ci)::value;
      if constexpr (FP32) first_b[c].store_as_is(b_chunk_to(c, 0), 0);
      else dma::static_for<ChunkB::kSteps>([&](auto xi) { first_b[c].template step<decltype(xi)::value>(largest, b_chunk_to(c, 0)); });
    });
  }
  barrier();
  uint32_t stage = 0;
  typename S::Acc aside;
  if constexpr (S::kBlock != 0) clear<S>(aside);
  auto put_aside = [&](int kt) {   // behind K tile kt, and at the end
    if constexpr (S::kBlock != 0) {
      if ((kt + 1 - g.kt0) % S::kBlock != 0 && kt + 1 != g.kt1) return;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          aside[i][j] += acc[i][j];
          acc[i][j] = kt + 1 == g.kt1 ? aside[i][j] : f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
  };
  if constexpr (FP32) {
    for (int kt = g.kt0; kt < g.kt1; ++kt) {
      dma::static_for<TM>([&](auto ii) { read_a(c0, ii, stage); read_a(c1, ii, stage); });
      dma::static_for<TN>([&](auto ji) { read_b(c0, ji, stage); read_b(c1, ji, stage); });
      stage = S::kStageBytes - stage;
      load_at(kt + 2);
#pragma unroll
      for (int c = 0; c < kA; ++c) { ca[c].store_as_is(a_chunk_to(c, stage), (half_k & 4) != 0); load_a(c, ca[c]); }
#pragma unroll
      for (int c = 0; c < kB; ++c) { cb[c].store_as_is(b_chunk_to(c, stage), 0); load_b(c, cb[c]); }
#pragma unroll
      for (int t = 0; t < 8; ++t)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(fb[t / 4][j][t % 4]), __uint_as_float(fa[t / 4][i][t % 4]), acc[i][j], 0, 0, 0);
      put_aside(kt);
      barrier();
    }
    return;
  }

  // The products of a K tile go by pairs of parts, the small ones first.  Parts 1 are read ahead of the loop's head, the other
  // parts a pass before the products that take them; between the products of the first five passes stand the conversions
  // of K tile kt + 1 (and, when a chunk is converted, the loads of kt + 2 into its registers); the barrier stands where all
  // waves have read this stage and written the other, with the last pass still to be multiplied behind it.
  constexpr int kPass = TM * TN, kConvert = 5 * kPass - 2, kWorkA = kA * ChunkA::kSteps, kWork = kWorkA + kB * ChunkB::kSteps;
  constexpr int pa[6] = {1, 0, 2, 0, 1, 0}, pb[6] = {1, 2, 0, 1, 0, 0};
  dma::static_for<TM>([&](auto ii) { read_a(c1, ii, 0); });
  dma::static_for<TN>([&](auto ji) { read_b(c1, ji, 0); });
  for (int kt = g.kt0; kt < g.kt1; ++kt) {
    const uint32_t next = S::kStageBytes - stage;
    load_at(kt + 2);
    dma::static_for<6>([&](auto pi) {
      constexpr int pass = decltype(pi)::value;
      if constexpr (pass == 5) barrier();
      dma::static_for<kPass>([&](auto mi) {
        constexpr int m = decltype(mi)::value, i = m / TN, j = m % TN, at = pass * kPass + m;
        // the next pass's (pass 5: the next K tile's) operands: TM + TN reads over the pass
        constexpr int f0 = m * (TM + TN) / kPass, f1 = (m + 1) * (TM + TN) / kPass;
        if constexpr (pass < 2 || pass == 5)
          dma::static_for<f1 - f0>([&](auto oi) {
            constexpr int f = f0 + decltype(oi)::value;
            if constexpr (f < TM) {
              constexpr std::integral_constant<int, f> fi{};
              if constexpr (pass == 0) read_a(c0, fi, stage);
              if constexpr (pass == 1) read_a(c2, fi, stage);
              if constexpr (pass == 5) read_a(c1, fi, next);
            } else {
              constexpr std::integral_constant<int, f - TM> fi{};
              if constexpr (pass == 0) read_b(c2, fi, stage);
              if constexpr (pass == 1) read_b(c0, fi, stage);
              if constexpr (pass == 5) read_b(c1, fi, next);
            }
          });
        acc[i][j] = mfma(fb[pb[pass]][j], fa[pa[pass]][i], acc[i][j]);
        constexpr int x0 = at * kWork / kConvert, x1 = (at + 1) * kWork / kConvert < kWork ? (at + 1) * kWork / kConvert : kWork;
        dma::static_for<(x1 > x0 ? x1 - x0 : 0)>([&](auto oi) {
          constexpr int x = x0 + decltype(oi)::value;
          if constexpr (x < kWorkA) {
            constexpr int c = x / ChunkA::kSteps, y = x % ChunkA::kSteps;
            ca[c].template step<y>(largest, a_chunk_to(c, next));
            if constexpr (y == ChunkA::kSteps - 1) load_a(c, ca[c]);
          } else {
            constexpr int c = (x - kWorkA) / ChunkB::kSteps, y = (x - kWorkA) % ChunkB::kSteps;
            cb[c].template step<y>(largest, b_chunk_to(c, next));
            if constexpr (y == ChunkB::kSteps - 1) load_b(c, cb[c]);
          }
        });
        __builtin_amdgcn_sched_barrier(0);
      });
    });
    stage = next;
    put_aside(kt);
  }
}

// Whether one of the values a tile multiplies over K tiles [g.kt0, g.kt1) is so small that its parts lose some of it, zeros
// apart.  Values of the same operand beyond the tile's last column count along.
constexpr float kSmall = 0x1p-102f;

template <bool MC, int R, bool DUAL>   // R: rows (columns) of the tile
__device__ __forceinline__ bool any_small(const Args& g, const __amdgpu_buffer_rsrc_t& first, const __amdgpu_buffer_rsrc_t& second, int r0, uint32_t ld) {
  // KC: eight lanes a row of 32 k;  MC: R / 4 lanes a row of R columns
  constexpr int kLanes = MC ? R / 4 : 8, kStep = kThreads / kLanes, kRows = MC ? kBK : R;
  const int t = threadIdx.x, piece = t % kLanes, row = t / kLanes;
  constexpr int kLoads = kRows / kStep, kAhead = 16 / kLoads;   // loads per K tile, K tiles under way
  uint32_t smallest = 0xffffffffu;   // of the magnitudes as integers; less one, which leaves zeros out
  for (int kt0 = g.kt0; kt0 < g.kt1; kt0 += kAhead) {
    u32x4 v[kAhead][kLoads];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int kt = kt0 + u;
      const bool other = DUAL && kt >= g.nk1;
      const int kk = (other ? kt - g.nk1 : kt) * kBK;
      // a piece past the end of the reduction, a K tile past the last: zeros
      const uint32_t past = kt < g.kt1 && (MC || kk + 4 * piece < g.k) ? 0u : 0x80000000u;
#pragma unroll
      for (int q = 0; q < kLoads; ++q) {
        const uint32_t at = MC ? (uint32_t)(kk + row + q * kStep) * ld + (uint32_t)r0 * 4u + (uint32_t)piece * 16u
                               : (uint32_t)(r0 + row + q * kStep) * ld + (uint32_t)(kk + 4 * piece) * 4u;
        v[u][q] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(other ? second : first, (int)(at | past), 0, 0));
      }
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u)
#pragma unroll
      for (int q = 0; q < kLoads; ++q)
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const uint32_t m = (v[u][q][w] & 0x7fffffffu) - 1u;
          smallest = smallest < m ? smallest : m;
        }
  }
  return smallest < __float_as_uint(kSmall) - 1u;
}

// acc = A_tile * B_tile over K tiles [g.kt0, g.kt1), on the split operands (multiply()); a second time on the fp32 instruction,
// which takes every value as it is, where
//   * a sum comes out infinite, NaN or of a magnitude below kTiny, or an operand is kHuge or more.  The splitting of an
//     infinity, or of a value that rounds to one, leaves NaN parts, so no such sum stays unnoticed.  Parts of a value below
//     kSmall can fall below the normal range: next to operands below kHuge its products are below kTiny, and what they
//     lose (2^-134 of the value, 2^-96 of a product) is 2^-32 of any sum that stays;
//   * a sum comes out zero and the tile has such a value, whose parts may all have been zero.  Zero sums are common (rows that
//     pad an expert), so the values are looked at before the tile is repeated.
// Of the sums only those that are stored count: rows below m_lim, columns below n_lim.  A launch that is formed twice throughout
// (operands of 2^-60 and less next to others of order one, or of 2^40) takes 993 / 1013 / 954 us NT / NN / TN for 8 experts of 1024
// rows, [1024, 4096], instead of 376 / 379 / 352; the element-wise kernel takes 947 / 983 / 882 for any values.
constexpr float kTiny = 0x1p-64f, kHuge = 0x1p38f;

template <bool A_MC, bool B_MC, typename S, bool DUAL>
__device__ __forceinline__ bool sums_need_fp32(const Args& g, const typename S::Acc& acc, float operand, int m_lim, int n_lim) {
  const int wave = threadIdx.x / kWave, lane = lane_id();
  const int m0 = S::row(wave) + (lane & 15), n0 = S::column(wave) + 4 * (lane >> 4);
  // twice the bits less one: no sign, zeros at the top; whether there is anything to look at more closely
  uint32_t low = 0xffffffffu, high = 0;
#pragma unroll
  for (int i = 0; i < S::TM; ++i)
#pragma unroll
    for (int j = 0; j < S::TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const uint32_t t = __float_as_uint(acc[i][j][r]) * 2u - 1u;
        low = low < t ? low : t;
        high = high > t ? high : t;
      }
  bool again = operand >= kHuge, zero = false;
  if (low < 2u * __float_as_uint(kTiny) - 1u || high >= 2u * 0x7f800000u - 1u) {
#pragma unroll
    for (int i = 0; i < S::TM; ++i)
#pragma unroll
      for (int j = 0; j < S::TN; ++j) {
        const bool stored = m0 + 16 * i < m_lim && n0 + 16 * j < n_lim;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float v = fabsf(acc[i][j][r]);
          again |= stored && v != 0.f && !(v >= kTiny && v < INFINITY);
          zero |= stored && v == 0.f;
        }
      }
  }
  if (__syncthreads_or(again || zero)) {
    if (__syncthreads_or(zero))
      again |= any_small<A_MC, S::BM, DUAL>(g, g.rsrc_a, g.rsrc_a2, g.a_r0, g.a_ld) || any_small<B_MC, S::BN, DUAL>(g, g.rsrc_b, g.rsrc_b2, g.b_r0, g.b_ld);
    return __syncthreads_or(again);
  }
  return false;
}

// A reduction of one or two terms goes to the fp32 instruction at once: its result is rounded once or twice there, and the
// products of parts that are left out, and what the bf16 instruction drops of a sum, are more than that (largest error over the
// sum of the magnitudes, 2^-24: 1.0 / 2.6 over one term, 1.9 / 2.6 over two, 2.5 / 2.3 over three, 3.7 / 2.1 over eight).
constexpr int kFewTerms = 2;

template <bool A_MC, bool B_MC, typename S, bool DUAL>
__device__ __forceinline__ void multiply(const Args& g, typename S::Acc& acc, int m_lim, int n_lim, char* lds) {
  clear<S>(acc);
  float operand = 0.f;
  if (!A_MC || g.k > kFewTerms) {   // NN / NT: k is a multiple of 4
    multiply_as<A_MC, B_MC, S, DUAL, false>(g, acc, lds, operand);
    if (!sums_need_fp32<A_MC, B_MC, S, DUAL>(g, acc, operand, m_lim, n_lim)) return;
    clear<S>(acc);
  }
  multiply_as<A_MC, B_MC, S, DUAL, true>(g, acc, lds, operand);
}

// c[m][n] = acc for the tile's rows below m_lim and columns below n (n a multiple of 4, c 16-byte aligned)
template <typename S>
__device__ __forceinline__ void store(const typename S::Acc& acc, float* __restrict__ c, int64_t ldc, int m_lim, int n0, int n) {
  const int wave = threadIdx.x / kWave, lane = lane_id();
  const int wm = S::row(wave), wn = S::column(wave);
#pragma unroll
  for (int i = 0; i < S::TM; ++i) {
    const int m = wm + 16 * i + (lane & 15);
    if (m >= m_lim) continue;
    float* const row = c + (int64_t)m * ldc;
#pragma unroll
    for (int j = 0; j < S::TN; ++j) {
      const int col = n0 + wn + 16 * j + 4 * (lane >> 4);
      if (col < n) *(f32x4*)(row + col) = acc[i][j];
    }
  }
}

// Part `part` of tile `tile` (of `tiles`) of a reduction cut into ksplit parts: hands the accumulators over through
// the workspace and returns whether this workgroup was the tile's last, which then holds the sum of all parts in
// `acc`, added in part order whoever came last.  The parts go past the caches (workgroups of a tile sit on different
// XCDs), a part is counted in once its stores are acknowledged, and nobody waits for anybody: see gmm_dma.h.
template <typename S>
__device__ __forceinline__ bool join_parts(typename S::Acc& acc, int tile, int tiles, int part, int ksplit, int32_t* counters,
                                           float* parts, char* lds) {
  constexpr int kThroughCaches = 0x11, kPieces = S::TM * S::TN;   // sc0 | sc1; 16-byte pieces per lane
  const uint32_t lane_off = threadIdx.x * 16u;
  const __amdgpu_buffer_rsrc_t mine = make_rsrc((const char*)parts + ((size_t)part * tiles + tile) * S::kPartBytes, (uint32_t)S::kPartBytes);
#pragma unroll
  for (int p = 0; p < kPieces; ++p)
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[p / S::TN][p % S::TN]), mine, (int)lane_off, p * (kThreads * 16), kThroughCaches);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  int* const flag = (int*)lds;
  if (threadIdx.x == 0) *flag = __hip_atomic_fetch_add(counters + tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  const bool last = *flag == ksplit - 1;
  if (!last) return false;
#pragma unroll
  for (int p = 0; p < kPieces; p += 4) {
    f32x4 sum[4];
#pragma unroll 1
    for (int q = 0; q < ksplit; ++q) {
      const __amdgpu_buffer_rsrc_t theirs = make_rsrc((const char*)parts + ((size_t)q * tiles + tile) * S::kPartBytes, (uint32_t)S::kPartBytes);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const f32x4 w = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(theirs, (int)lane_off, (p + u) * (kThreads * 16), kThroughCaches));
        sum[u] = q == 0 ? w : sum[u] + w;
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) acc[(p + u) / S::TN][(p + u) % S::TN] = sum[u];
  }
  if (threadIdx.x == 0) counters[tile] = 0;   // as the launch found it
  return true;
}

// ---- NN / NT ----
// P = gridDim.x workgroups (one per compute unit, two of the small tile) walk the list of tiles as those of gmm_dma.h's kernel do.  The tiles of a
// last round that would leave at least half of the workgroups idle are cut along the reduction when there is a
// workspace: with four and a half rounds of long reductions (8 experts of 1024 rows: 4.4 rounds NT, 1.1 NN) the tail
// would otherwise take as long as a full round.
template <bool B_MC, typename S, bool DUAL>
__global__ void __launch_bounds__(kThreads, 2 * S::kPerUnit)
gmm_f32_rows_kernel(const float* __restrict__ a, const float* __restrict__ b, float* __restrict__ c, const int32_t* __restrict__ bins,
                    int num_groups, int64_t rows, int k, int n, int tiles_n, const float* __restrict__ a2, const float* __restrict__ b2,
                    int32_t* __restrict__ ws_counters, float* ws_parts, int ws_capacity) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int P = gridDim.x, run = P / kXcds, xcd = blockIdx.x % kXcds, member = blockIdx.x / kXcds;
  const RowTiles<S::BM> tiles(bins, num_groups, tiles_n, (int)rows, false, 8);
  const int total = tiles.total, full_rounds = total / P, rest = total - full_rounds * P;
  Args g;
  g.a_ld = (uint32_t)k * 4u;
  g.b_ld = (uint32_t)(B_MC ? n : k) * 4u;
  g.a_r0 = 0;
  g.k = k;
  g.nk1 = (k + kBK - 1) / kBK;
  const int nk = DUAL ? 2 * g.nk1 : g.nk1;
  int ksplit = 1;
  if (ws_parts != nullptr && rest > 0 && 2 * rest <= P) {
    int s = P / rest;
    s = s > kMaxKSplit ? kMaxKSplit : s;
    s = s > nk / kMinPartTiles ? nk / kMinPartTiles : s;
    s = (int64_t)s * rest > ws_capacity ? ws_capacity / rest : s;
    ksplit = s < 2 ? 1 : s;
  }
  const int rounds = full_rounds + (rest > 0 ? 1 : 0);
  for (int r = 0; r < rounds; ++r) {
    int id, part = 0;
    const bool cut = r == full_rounds && ksplit > 1;
    if (cut) {
      const int j = member * kXcds + xcd;
      if (j >= ksplit * rest) break;
      id = full_rounds * P + j % rest;
      part = j / rest;
    } else if (r == full_rounds) {
      // the tiles of a partly filled round in equal shares to the XCDs: dealt in runs they would leave some XCDs idle and
      // put two tiles on every compute unit of the others
      const int first = xcd * rest / kXcds;
      if (member >= (xcd + 1) * rest / kXcds - first) break;
      id = full_rounds * P + first + member;
    } else {
      id = (r * kXcds + xcd) * run + (member + r) % run;
    }
    int e, start, end, tm, tn;
    tiles.find(id, e, start, end, tm, tn);
    const int row0 = start + tm * S::BM;
    // up to the expert's last row: the next expert's rows, or rows behind the last bin that nobody may have written, must not
    // have a say in which instruction forms these sums
    const uint32_t a_bytes = clip_bytes((int64_t)(end - row0) * k * 4), b_bytes = (uint32_t)((int64_t)k * n * 4);
    g.rsrc_a = make_rsrc(a + (int64_t)row0 * k, a_bytes);
    g.rsrc_b = make_rsrc(b + (int64_t)e * k * n, b_bytes);
    g.rsrc_a2 = DUAL ? make_rsrc(a2 + (int64_t)row0 * k, a_bytes) : g.rsrc_a;
    g.rsrc_b2 = DUAL ? make_rsrc(b2 + (int64_t)e * k * n, b_bytes) : g.rsrc_b;
    g.b_r0 = tn * S::BN;
    g.kt0 = cut ? (int)((int64_t)part * nk / ksplit) : 0;
    g.kt1 = cut ? (int)((int64_t)(part + 1) * nk / ksplit) : nk;
    typename S::Acc acc;
    multiply<false, B_MC, S, DUAL>(g, acc, end - row0, n - g.b_r0, lds);
    if (!cut || join_parts<S>(acc, id - full_rounds * P, rest, part, ksplit, ws_counters, ws_parts, lds))
      store<S>(acc, c + (int64_t)row0 * n, n, end - row0, g.b_r0, n);
    tile_done();
  }
}

// ---- TN ----
// One workgroup per tile and part of its reduction; ksplit is the launch's (> 1: there are few tiles and a workspace).
// Experts are taken longest reduction first (every wave ranks up to 64 of them), so that the last tiles are short ones.
template <typename S>
__global__ void __launch_bounds__(kThreads, 2 * S::kPerUnit)
gmm_f32_tn_kernel(const float* __restrict__ a, const float* __restrict__ b, float* __restrict__ c, const int32_t* __restrict__ bins,
                  int num_groups, int rows, int k, int n, int tiles_m, int tiles_n, int ksplit, int32_t* __restrict__ ws_counters,
                  float* ws_parts) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int per_group = tiles_m * tiles_n, total = per_group * num_groups;
  const int id = xcd_tile_id(blockIdx.x, S::kPerUnit * kXcdRun);
  if (id >= total * ksplit) return;
  const int tile = id % total, part = id / total;
  int e = tile / per_group;
  if (num_groups <= kWave) {
    const int lane = lane_id();
    const int rank = rank_by_rows(lane < num_groups ? bins[lane] - (lane > 0 ? bins[lane - 1] : 0) : -1, num_groups);
    e = __builtin_amdgcn_readfirstlane((int)__builtin_ctzll(__ballot(rank == e)));
  }
  // tiles of an expert in bands of eight row tiles (the last band takes what is left), rows fastest
  const int t = tile % per_group;
  const int band = t / (8 * tiles_n), left = tiles_m - band * 8 < 8 ? tiles_m - band * 8 : 8;
  const int in = t - band * 8 * tiles_n;
  const int tm = band * 8 + in % left, tn = in / left;
  const int start = e > 0 ? clamp_row(bins[e - 1], rows) : 0;
  int end = clamp_row(bins[e], rows);
  end = end < start ? start : end;
  Args g;
  g.a_ld = (uint32_t)k * 4u;
  g.b_ld = (uint32_t)n * 4u;
  g.a_r0 = tm * S::BM;
  g.b_r0 = tn * S::BN;
  g.k = end - start;
  const int nk = (end - start + kBK - 1) / kBK;
  g.nk1 = nk;
  // the buffers cover exactly the expert's rows: later ones read as zeros
  g.rsrc_a = make_rsrc(a + (int64_t)start * k, (uint32_t)((int64_t)(end - start) * k * 4));
  g.rsrc_b = make_rsrc(b + (int64_t)start * n, (uint32_t)((int64_t)(end - start) * n * 4));
  g.rsrc_a2 = g.rsrc_a;
  g.rsrc_b2 = g.rsrc_b;
  g.kt0 = (int)((int64_t)part * nk / ksplit);
  g.kt1 = (int)((int64_t)(part + 1) * nk / ksplit);
  typename S::Acc acc;
  multiply<true, true, S, false>(g, acc, k - g.a_r0, n - g.b_r0, lds);
  if (ksplit > 1 && !join_parts<S>(acc, tile, total, part, ksplit, ws_counters, ws_parts, lds)) return;
  store<S>(acc, c + ((int64_t)e * k + g.a_r0) * n, n, k - g.a_r0, g.b_r0, n);
}

template <bool B_MC, typename S, bool DUAL>
int launch_rows(const float* a, const float* b, float* c, const int32_t* bins, int num_groups, int64_t rows, int k, int n, const float* a2,
                const float* b2, const Workspace& lent, int units, hipStream_t s) {
  WorkspaceParts ws(lent, S::kPartBytes);
  if (units > (int)kWorkspaceCounters) ws.parts = nullptr;   // at most half of the workgroups' tiles are cut
  auto kern = gmm_f32_rows_kernel<B_MC, S, DUAL>;
  const int rc = allow_lds(kern, S::kLdsBytes);
  if (rc) return rc;
  kern<<<(unsigned)(S::kPerUnit * units), kThreads, S::kLdsBytes, s>>>(a, b, c, bins, num_groups, rows, k, n, (int)ceil_div(n, S::BN), a2, b2,
                                                                      ws.counters, ws.parts, ws.capacity);
  return launch_status();
}

template <typename S>
int launch_tn(const float* a, const float* b, float* c, const int32_t* bins, int num_groups, int64_t rows, int k, int n,
              const Workspace& lent, int units, hipStream_t s) {
  WorkspaceParts ws(lent, S::kPartBytes);
  if (units > (int)kWorkspaceCounters) ws.parts = nullptr;
  const int tiles_m = (int)ceil_div(k, S::BM), tiles_n = (int)ceil_div(n, S::BN);
  const int64_t total = (int64_t)tiles_m * tiles_n * num_groups;
  if (total * kMaxKSplit > 0x7fffff00) return MBX_ERANGE;
  int64_t ksplit = 1;
  const int slots = S::kPerUnit * units;
  if (ws.parts && 2 * total <= slots) {
    const int64_t nk = rows / num_groups / kBK;
    ksplit = slots / total;
    ksplit = ksplit > kMaxKSplit ? kMaxKSplit : ksplit;
    ksplit = ksplit > nk / kMinPartTiles ? nk / kMinPartTiles : ksplit;
    ksplit = ksplit * total > ws.capacity ? ws.capacity / total : ksplit;
    ksplit = ksplit < 2 ? 1 : ksplit;
  }
  auto kern = gmm_f32_tn_kernel<S>;
  const int rc = allow_lds(kern, S::kLdsBytes);
  if (rc) return rc;
  kern<<<(unsigned)xcd_grid(total * ksplit, S::kPerUnit * kXcdRun), kThreads, S::kLdsBytes, s>>>(a, b, c, bins, num_groups, (int)rows, k, n, tiles_m, tiles_n,
                                                                         (int)ksplit, ws.counters, ws.parts);
  return launch_status();
}

}  // namespace f32

// Whether the fp32 kernels of this file take a product: whole 16-byte pieces, 32-bit byte offsets from the buffer of a
// tile's rows, of an expert's weights or (TN) of an expert's rows, which could be all of them.
static inline bool f32_ok(const void* a, const void* b, const void* c, int64_t rows, int k, int n, int layout) {
  const int64_t lim = (int64_t)1 << 31;
  if (((uintptr_t)a | (uintptr_t)b | (uintptr_t)c) & 15u || k <= 0 || k % 4 || n % 4) return false;
  if (layout == MBX_TN) return rows * (int64_t)(k > n ? k : n) * 4 < lim;
  return (int64_t)k * n * 4 < lim && (int64_t)k * 4 * 128 < lim;
}

// TN launches left to gmm.hip's element-wise kernel, a chain of fp32 multiply-adds per sum: up to 24 rows per expert on average.
// There is next to nothing to multiply, and three of its workgroups share a compute unit, which is what the stores want (us, that
// kernel / this one; 64 experts, [1024, 4096]: 32 rows 347 / 397, 64: 500 / 467;  8, [4096, 4096]: 170 / 187, 254 / 224;  128, [768,
// 2048]: 269 / 272, 379 / 323).  The size limits are that kernel's.  Up to some 190 rows the stores bound this kernel too, and one workgroup
// to a compute unit overlaps them with little: a third of the launches of 25 - 190 rows are 3 - 15 % longer than two of half the tile
// were (8 of 128, [4096, 4096]: 286 / 266; 128 of 128, [768, 2048]: 430 / 396), the others shorter (64 of 64, [1024, 4096]: 467 / 519), together 5 %.
static inline bool f32_short_tn(int num_groups, int64_t rows, int k) {
  return rows <= 24 * (int64_t)num_groups && ceil_div(k, 128) <= 65535 && num_groups <= 65535;
}

// TN: the small tile, two workgroups to a compute unit, where the main tile would leave three eighths of the compute units or more
// without one (us, main / small tile: 8 of 512, [1024, 512], 128 tiles: 41 / 31; 8 of 256, [1408, 512], 176 tiles: 29 / 34).
static inline bool f32_small(int64_t tiles, int units) { return 8 * tiles < 5 * (int64_t)units; }

// NN / NT: the small tile (us, main / small tile)
//   * up to 64 rows per expert on average, where main tiles would be half empty (64 experts of 64, [1408, 1024]: 140 / 118; of 100: 157 / 158);
//   * for few tiles as above (NT 8 of 256, [1408, 512]: 40 / 29; 4 of 1500, [704, 4096], 144 tiles: 240 / 218; 32 of 100, [1408, 1024], 192
//     tiles: 75 / 80).  Long reductions that only the main tile's launch has few enough tiles to be cut along are shorter there (NN 38 of
//     209, [3520, 192]: 105 / 157), but less exact: the small tile puts its sums aside;
//   * where it multiplies that much less padding: kShortArea in reductions of up to kShortTiles K tiles, which are mostly the first
//     loads and the stores, whose latency the second workgroup hides (28 of 726, [320, 320]: 57 / 45; 68 of 101, [288, 816]: 59 / 43; 22 of
//     109, [320, 4672]: 68 / 76), kLongArea in longer ones, where it multiplies at three quarters of the main tile's rate (45 of 165,
//     [8192, 320]: 533 / 365; 19 of 768, [2496, 320]: 175 / 188).  13 of 500 launches (2 - 128 experts of 20 - 2000 rows, [128 - 8192, 128 -
//     8192]) are 3 - 30 % shorter by this line, one 3 % longer.
constexpr int64_t kF32SmallRows = 64;
constexpr int kShortTiles = 12;
constexpr double kShortArea = 1.25, kLongArea = 1.45;
static bool f32_small_rows(int num_groups, int64_t rows, int n, int64_t nk, int units) {
  const int64_t average = ceil_div(rows, num_groups);
  if (average <= kF32SmallRows) return true;
  // an expert's rows in whole tiles
  const int64_t tiles = num_groups * ceil_div(average, f32::Wide::BM) * ceil_div(n, f32::Wide::BN);
  if (f32_small(tiles, units)) return true;
  const auto area = [&](int bm, int bn) { return ((double)average / bm + 0.5) * bm * (double)ceil_div(n, bn) * bn; };   // the row counts vary
  return area(f32::Wide::BM, f32::Wide::BN) > (nk <= kShortTiles ? kShortArea : kLongArea) * area(f32::Small::BM, f32::Small::BN);
}

}  // namespace

bool gmm_f32_rows_small(int num_groups, int64_t rows, int k, int n, bool dual) {
  return f32_small_rows(num_groups, rows, n, (dual ? 2 : 1) * ceil_div(k, f32::kBK), persistent_grid((int64_t)1 << 30));
}

int gmm_f32(const void* a, const void* b, const void* a2, const void* b2, void* c, const int32_t* bins, int num_groups,
                   int64_t rows, int k, int n, int layout, void* workspace, size_t workspace_bytes, hipStream_t s) {
  if (layout == MBX_TN && f32_short_tn(num_groups, rows, k)) return MBX_EUNSUPPORTED;
  if (!f32_ok(a, b, c, rows, k, n, layout) || (a2 && !f32_ok(a2, b2, c, rows, k, n, layout))) return MBX_EUNSUPPORTED;
  const float *ap = (const float*)a, *bp = (const float*)b, *ap2 = (const float*)a2, *bp2 = (const float*)b2;
  float* cp = (float*)c;
  const Workspace lent{workspace, workspace_bytes};
  const int units = persistent_grid((int64_t)1 << 30);
  if (layout == MBX_TN) {
    const int64_t wide = ceil_div(k, 128) * ceil_div(n, 256), tall = ceil_div(k, 256) * ceil_div(n, 128);
    if (f32_small(num_groups * (tall < wide ? tall : wide), units)) return f32::launch_tn<f32::Small>(ap, bp, cp, bins, num_groups, rows, k, n, lent, units, s);
    return tall < wide ? f32::launch_tn<f32::Tall>(ap, bp, cp, bins, num_groups, rows, k, n, lent, units, s)
                       : f32::launch_tn<f32::Wide>(ap, bp, cp, bins, num_groups, rows, k, n, lent, units, s);
  }
  if ((ceil_div(rows, 64) + num_groups) * ceil_div(n, 128) > 0x7fffffff) return MBX_ERANGE;
  const bool small = f32_small_rows(num_groups, rows, n, (a2 ? 2 : 1) * ceil_div(k, f32::kBK), units);
#define MBX_LAUNCH_F32(B_MC, S, DUAL) return f32::launch_rows<B_MC, S, DUAL>(ap, bp, cp, bins, num_groups, rows, k, n, ap2, bp2, lent, units, s)
#define MBX_LAUNCH_F32_BM(B_MC, DUAL) do { if (small) MBX_LAUNCH_F32(B_MC, f32::Small, DUAL); else MBX_LAUNCH_F32(B_MC, f32::Wide, DUAL); } while (0)
  if (layout == MBX_NT) {
    if (a2) MBX_LAUNCH_F32_BM(false, true); else MBX_LAUNCH_F32_BM(false, false);
  } else {
    if (a2) MBX_LAUNCH_F32_BM(true, true); else MBX_LAUNCH_F32_BM(true, false);
  }
#undef MBX_LAUNCH_F32_BM
#undef MBX_LAUNCH_F32
}

}  // namespace mbx
