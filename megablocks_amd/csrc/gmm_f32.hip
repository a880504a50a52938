// Grouped GEMM in fp32 on the bf16 matrix instruction: every value is split into three bf16 parts (24 bits, Split below), and the
// six products of parts that reach 2^-18 of a product are summed in fp32 (v_mfma_f32_16x16x32_bf16).
//
// What bounds it: the matrix cores and the power they draw.  The fp32 instruction (v_mfma_f32_16x16x4_f32) does 256 FLOP
// per cycle and compute unit, the bf16 one 4096, a sixth of which is 683.  Next to the 96 products of a K tile, 1536 cycles
// of a SIMD, a wave spends 384 vector-ALU instructions, 1536 cycles, on the splitting; two waves share a SIMD, and what
// one converts the other multiplies.  8 experts of 1024 +- 30 rows, hidden 1024, ffn 4096: 416 / 380 / 366 us NT / NN / TN
// against 533 / 545 / 522 on the fp32 instruction and 961 in the element-wise kernel of gmm.hip, which serves every
// alignment; 195 TFLOP/s on 4096^3 against 141.  Half the conversion instructions (v_dot2c_f32_bf16) changed nothing;
// cutting the parts off instead of rounding them is 3 % faster and up to a third less exact.
//
// How exact: three parts hold all 24 bits of a value; the three products of parts not taken come to less than 2^-25 of a product,
// and an accumulator is rounded six times per 32 k instead of 32 times.  Relative error (2-norm) against fp64: 4.8e-7 over
// k = 1024, 9.8e-7 over 4096, where a chain of fp32 fused multiply-adds shows 5.7e-7 and 1.15e-6; 3.4e-8 over eight terms (5.4e-8).
// The error of a single product is larger than that chain's, up to 2.6 2^-24 of it instead of one: sums of one or two terms,
// and those that the parts do not serve (infinities, NaN, values next to the largest or the smallest), are formed on the fp32
// instruction: multiply().
//
// Tile: 128 x 128 (64 x 128 for short experts) per workgroup of four waves (2 x 2), K tiles of 32, two stages of
// 32 KiB, so two workgroups share a compute unit and one multiplies while the other converts, waits at its barrier or
// stores.  Operands go global -> LDS without registers as whole 16-byte pieces (k and n multiples of 4, 16-byte aligned
// operands); the loads of a K tile are issued a K tile before they are needed, and one barrier per K tile is enough.
//
// LDS layouts: an operand whose reduction dimension is contiguous (KC) is [row][32 k], 128-byte rows, 16-byte chunk c of row r
// at position c ^ ((r >> 1) & 7) (gmm_dma.h's layout of 64 16-bit values, byte for byte); one ds_read_b128 gives a
// lane its row's operand of four instructions.  An operand whose reduction dimension is strided (MC) is [k][128 columns],
// the column XORed by 16 ((k >> 2) & 3), so that the four quarter waves, which read rows four apart, use different
// banks; a lane reads two rows per ds_read2st64_b32.  Step j (of 4) of group s (of 2) of a K tile multiplies
// k = 16 s + 4 (lane / 16) + j of both operands; the bf16 instruction takes both groups' four as a lane's eight.
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

constexpr int kBN = 128, kBK = 32, kThreads = 256;
constexpr uint32_t kOperandBytes = 128 * kBK * 4, kStageBytes = 2 * kOperandBytes;
constexpr size_t kLdsBytes = 2 * kStageBytes;
constexpr size_t kPartBytes = (size_t)128 * kBN * 4;       // one tile's accumulators in the workspace
constexpr int kMaxKSplit = 8, kMinPartTiles = 8;           // parts of a reduction, K tiles per part

// The operands of a tile: buffers (out-of-range bytes read as zero), row pitches in bytes, tile origins, the first and
// one past the last K tile to multiply, the length of the whole reduction (pieces of a row past it read as zeros).
// Two operand pairs (DUAL): K tiles nk1 .. 2 nk1 - 1 come from the second.
struct Args {
  __amdgpu_buffer_rsrc_t rsrc_a, rsrc_b, rsrc_a2, rsrc_b2;
  uint32_t a_ld, b_ld;
  int a_r0, b_r0, kt0, kt1, k, nk1;
};

template <int ROW>   // this lane's column in rows ROW and ROW + 1 of an MC tile
__device__ __forceinline__ u32x2 lds_read2_rows(uint32_t addr) {
  u32x2 v;
  asm volatile("ds_read2st64_b32 %0, %1 offset0:%2 offset1:%3" : "=v"(v) : "v"(addr), "n"(2 * ROW), "n"(2 * ROW + 2));
  return v;
}

// The operand of four matrix instructions of a 16-row (column) fragment, as the reads deliver it.  A read is under way from
// its statement to the wait for it: nothing may touch its registers in between, so they are taken apart (at) only where a
// product uses them, and every path from the reads to a loop's end or a use goes through the wait and tie().
template <bool MC> struct Frag;
template <> struct Frag<false> {
  u32x4 v;
  __device__ __forceinline__ float at(int t) const { return __uint_as_float(v[t]); }
  __device__ __forceinline__ void tie() { asm volatile("" : "+v"(v)); }
};
template <> struct Frag<true> {
  u32x2 v[2];
  __device__ __forceinline__ float at(int t) const { return __uint_as_float(v[t / 2][t % 2]); }
  __device__ __forceinline__ void tie() { asm volatile("" : "+v"(v[0]), "+v"(v[1])); }
};

// Eight fp32 values as three bf16 parts each, v = part 0 + part 1 + part 2 up to 2^-27 |v|: every part is the rest the parts
// before it leave (the differences are exact), rounded to nearest.  In kSteps steps of a few instructions, to be put between
// products: step 3 p + q forms part q of the values 2 p and 2 p + 1.
struct Split {
  static constexpr int kSteps = 12;
  u32x4 part[3];
  float rest[2];
  template <int X, bool MC>
  __device__ __forceinline__ void step(const Frag<MC>& low, const Frag<MC>& high, float& largest) {   // largest: magnitude seen
    constexpr int p = X / 3, q = X % 3, v = 2 * (p & 1);
    if constexpr (q == 0) {
      rest[0] = p < 2 ? low.at(v) : high.at(v);
      rest[1] = p < 2 ? low.at(v + 1) : high.at(v + 1);
      asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(largest) : "v"(rest[0]), "v"(rest[1]));
    }
    const uint32_t both = pack2<MBX_BF16>(rest[0], rest[1]);
    part[q][p] = both;
    if constexpr (q < 2) {
      rest[0] -= __uint_as_float(both << 16);
      rest[1] -= __uint_as_float(both & 0xffff0000u);
    }
  }
};

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ f32x4 mfma(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

template <int N>
__device__ __forceinline__ void wait_lgkm() {   // at most N LDS reads of this wave still in flight
  static_assert(N < 16, "lgkmcnt is a 4-bit counter");
  asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(N) : "memory");
}

// The accumulators of a wave: (BM / 32) x 4 tiles of 16 x 16 of its (BM / 2) x 64 part of the tile.  Tile (i, j), register r of
// lane l is
//   row wm + 16 i + l % 16, column wn + 16 j + 4 (l / 16) + r
// of the workgroup's tile (the operands are swapped, so a lane owns runs of four consecutive columns).
template <int BM> using Acc = f32x4[BM / 32][4];

// acc += A_tile * B_tile over K tiles [g.kt0, g.kt1); largest: the largest magnitude among the operands (unless FP32)
template <bool A_MC, bool B_MC, int BM, bool DUAL, bool FP32>
__device__ __forceinline__ void multiply_as(const Args& g, Acc<BM>& acc, char* lds_generic, float& largest) {
  constexpr int TM = BM / 32, TN = 4;
  static_assert(!A_MC || BM == 128, "a strided first operand: full tiles");
  const lds_ptr lds = (lds_ptr)lds_generic;
  const uint32_t lds_base = (uint32_t)(uintptr_t)lds;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = lane_id(), quarter = lane >> 4;
  const int wm = (wave / 2) * (BM / 2), wn = (wave % 2) * 64;
  constexpr int LA = BM / 32, LB = 4;   // wave-wide loads of a K tile per wave

  // KC: load j = wave + 4 q holds rows 8 j .. 8 j + 7; a lane's 16-byte piece is the same for all q.
  // MC: load j holds rows k = 2 j, 2 j + 1, whose (k >> 2) & 3 is (wave >> 1) + 2 (q & 1).
  auto mc_offset = [&](int r0, uint32_t ld, int odd) -> uint32_t {
    return (uint32_t)(lane >> 5) * ld + (uint32_t)r0 * 4u + (uint32_t)((lane & 31) ^ (4 * ((wave >> 1) + 2 * odd))) * 16u;
  };
  const uint32_t a_lane = A_MC ? mc_offset(g.a_r0, g.a_ld, 0) : dma::load_lane_offset<false, 64, 128>(wave, g.a_r0, g.a_ld);
  const uint32_t b_lane = B_MC ? mc_offset(g.b_r0, g.b_ld, 0) : dma::load_lane_offset<false, 64, 128>(wave, g.b_r0, g.b_ld);
  const uint32_t a_odd = A_MC ? mc_offset(g.a_r0, g.a_ld, 1) - a_lane : 0u, b_odd = B_MC ? mc_offset(g.b_r0, g.b_ld, 1) - b_lane : 0u;
  const uint32_t a_j = A_MC ? 2u * g.a_ld : 8u * g.a_ld, b_j = B_MC ? 2u * g.b_ld : 8u * g.b_ld;   // from load j to j + 1
  const uint32_t a_step = A_MC ? kBK * g.a_ld : kBK * 4u, b_step = B_MC ? kBK * g.b_ld : kBK * 4u;   // per K tile
  const int piece_k = 4 * ((lane & 7) ^ ((4 * (wave & 1) + ((lane >> 3) >> 1)) & 7));   // first k of a KC lane's piece
  // One of the LA + LB loads of a K tile: load_at() works out the K tile's addresses, load_one() issues number q.
  uint32_t a0 = 0, b0 = 0, dst = 0;
  __amdgpu_buffer_rsrc_t ra = g.rsrc_a, rb = g.rsrc_b;
  auto load_at = [&](int kt, uint32_t stage) {
    const bool second = DUAL && kt >= g.nk1;
    const int kk = second ? kt - g.nk1 : kt;
    // k is a multiple of 4: a piece of a row lies inside the reduction or past it, where it has to read as zeros (the
    // next row's values could be infinite); bit 31 puts it out of the buffer's range, as it does a K tile past the last
    const uint32_t past = kk * kBK + piece_k < g.k ? 0u : 0x80000000u, none = kt < g.kt1 ? 0u : 0x80000000u;
    if (DUAL) { ra = second ? g.rsrc_a2 : g.rsrc_a; rb = second ? g.rsrc_b2 : g.rsrc_b; }
    a0 = (a_lane + (uint32_t)kk * a_step + (uint32_t)wave * a_j) | (A_MC ? none : past | none);
    b0 = (b_lane + (uint32_t)kk * b_step + (uint32_t)wave * b_j) | (B_MC ? none : past | none);
    dst = stage + (uint32_t)wave * 1024u;
  };
  auto load_one = [&](auto qi) {
    constexpr uint32_t q = decltype(qi)::value;
    if constexpr (q < LA)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (__attribute__((address_space(3))) void*)(lds + dst + q * 4096u), 16, (int)(a0 + 4u * q * a_j + (q & 1 ? a_odd : 0u)), 0, 0, 0);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (__attribute__((address_space(3))) void*)(lds + dst + kOperandBytes + (q - LA) * 4096u), 16, (int)(b0 + 4u * (q - LA) * b_j + ((q - LA) & 1 ? b_odd : 0u)), 0, 0, 0);
  };

  // LDS addresses of this lane's operands of group 0 in stage 0
  auto mc_frag = [&](int r) -> uint32_t { return (uint32_t)(quarter * 4 * 512 + ((r + (lane & 15)) ^ (16 * quarter)) * 4); };
  uint32_t fa_off[A_MC ? TM : 1], fb_off[B_MC ? TN : 1];
#pragma unroll
  for (int i = 0; i < (A_MC ? TM : 1); ++i) fa_off[i] = A_MC ? mc_frag(wm + 16 * i) : dma::frag_lane_offset<false, 64, 128>(wm);
#pragma unroll
  for (int j = 0; j < (B_MC ? TN : 1); ++j) fb_off[j] = kOperandBytes + (B_MC ? mc_frag(wn + 16 * j) : dma::frag_lane_offset<false, 64, 128>(wn));

  Frag<A_MC> fa[2][TM];
  Frag<B_MC> fb[2][TN];
  // the read instructions of group s of one fragment: one of a KC fragment (four k), two of an MC fragment (two each)
  auto read_a = [&](auto ii, uint32_t base) {
    constexpr int i = decltype(ii)::value;
    dma::static_for<2>([&](auto si) {
      constexpr int s = decltype(si)::value;
      if constexpr (A_MC) { fa[s][i].v[0] = lds_read2_rows<16 * s>(base + fa_off[i]); fa[s][i].v[1] = lds_read2_rows<16 * s + 2>(base + fa_off[i]); }
      else fa[s][i].v = dma::read_frag_kc<s, i * 16 * 128>(base, fa_off[0]);
    });
  };
  auto read_b = [&](auto ji, uint32_t base) {
    constexpr int j = decltype(ji)::value;
    dma::static_for<2>([&](auto si) {
      constexpr int s = decltype(si)::value;
      if constexpr (B_MC) { fb[s][j].v[0] = lds_read2_rows<16 * s>(base + fb_off[j]); fb[s][j].v[1] = lds_read2_rows<16 * s + 2>(base + fb_off[j]); }
      else fb[s][j].v = dma::read_frag_kc<s, j * 16 * 128>(base, fb_off[0]);
    });
  };
  // the values of a K tile as registers written at this point: orders their users behind the wait in front of it
  auto tie = [&] {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int i = 0; i < TM; ++i) fa[s][i].tie();
#pragma unroll
      for (int j = 0; j < TN; ++j) fb[s][j].tie();
    }
  };
  // The products of a K tile on its split operands.  Fragments of A go in pairs, so that twelve products on two
  // accumulators stand between the conversions; what is converted behind the products of (pair, j) is the next fragment
  // of B, or the next pair of A.  The fragments of the next K tile are read behind the products of the last pair, when
  // the conversions are done (with one pair: as soon as a fragment is converted), so that their registers serve the
  // parts until then; one of the loads of K tile kt + 2 goes out behind every second product.
  Split sa[2][2], sb[TN];
  auto products = [&](uint32_t next_base) {
    constexpr int PAIRS = TM / 2;
    auto convert_a = [&](auto ii, auto xi) {
      constexpr int i = decltype(ii)::value, x = decltype(xi)::value;
      sa[i / 2 % 2][i % 2].template step<x>(fa[0][i], fa[1][i], largest);
      if constexpr (PAIRS == 1 && x == Split::kSteps - 1) { __builtin_amdgcn_sched_barrier(0); read_a(ii, next_base); }
    };
    auto convert_b = [&](auto ji, auto xi) {
      constexpr int j = decltype(ji)::value, x = decltype(xi)::value;
      sb[j].template step<x>(fb[0][j], fb[1][j], largest);
      if constexpr (PAIRS == 1 && x == Split::kSteps - 1) { __builtin_amdgcn_sched_barrier(0); read_b(ji, next_base); }
    };
    constexpr std::integral_constant<int, 0> c0{};
    constexpr std::integral_constant<int, 1> c1{};
    dma::static_for<Split::kSteps>([&](auto xi) { convert_a(c0, xi); convert_b(c0, xi); convert_a(c1, xi); });
    dma::static_for<PAIRS * TN>([&](auto pj) {
      constexpr int p = decltype(pj)::value / TN, j = decltype(pj)::value % TN;
      dma::static_for<12>([&](auto mi) {
        constexpr int m = decltype(mi)::value, t = m / 2, i = m % 2;
        constexpr int pa[6] = {0, 2, 1, 0, 1, 0}, pb[6] = {2, 0, 1, 1, 0, 0};   // the small products first
        acc[2 * p + i][j] = mfma(sb[j].part[pb[t]], sa[p % 2][i].part[pa[t]], acc[2 * p + i][j]);
        if constexpr (p == 0 && j + 1 < TN) convert_b(std::integral_constant<int, j + 1>{}, mi);
        if constexpr (p + 1 < PAIRS && j >= TN - 2) convert_a(std::integral_constant<int, 2 * p + 2 + j - (TN - 2)>{}, mi);
        if constexpr (p == 1 && m % 6 == 5) {
          if constexpr (j < 2) read_a(std::integral_constant<int, 2 * j + m / 6>{}, next_base);
          else { read_b(std::integral_constant<int, 2 * (j - 2) + m / 6>{}, next_base); }
        }
        constexpr int load = (decltype(pj)::value * 12 + m) / 2;
        if constexpr (m % 2 == 1 && load < LA + LB) load_one(std::integral_constant<uint32_t, load>{});
        __builtin_amdgcn_sched_barrier(0);
      });
    });
  };
  // The same products on the fp32 instruction.
  auto products_fp32 = [&](uint32_t next_base) {
    dma::static_for<2>([&](auto si) {
      dma::static_for<4>([&](auto ti) {
        constexpr int s = decltype(si)::value, t = decltype(ti)::value;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fb[s][j].at(t), fa[s][i].at(t), acc[i][j], 0, 0, 0);
      });
    });
    __builtin_amdgcn_sched_barrier(0);
    dma::static_for<LA + LB>(load_one);
    dma::static_for<TM>([&](auto ii) { read_a(ii, next_base); });
    dma::static_for<TN>([&](auto ji) { read_b(ji, next_base); });
  };
  // A K tile's values are in registers when its iteration begins.  The barrier stands where every wave has read its
  // stage, which takes K tile kt + 2 from then on, and where K tile kt + 1 has landed in the other, to be read during
  // the products.
  if (g.kt0 >= g.kt1) return;
  load_at(g.kt0, 0);
  dma::static_for<LA + LB>(load_one);
  load_at(g.kt0 + 1, kStageBytes);
  dma::static_for<LA + LB>(load_one);
  dma::wait_vmcnt<LA + LB>();
  __builtin_amdgcn_s_barrier();
  uint32_t stage = 0;
  dma::static_for<TM>([&](auto ii) { read_a(ii, lds_base); });
  dma::static_for<TN>([&](auto ji) { read_b(ji, lds_base); });
  wait_lgkm<0>();
  tie();
  for (int kt = g.kt0; kt < g.kt1; ++kt) {
    dma::wait_vmcnt<0>();
    __builtin_amdgcn_s_barrier();
    load_at(kt + 2, stage);
    stage ^= kStageBytes;
    if constexpr (FP32) products_fp32(lds_base + stage); else products(lds_base + stage);   // past the last K tile: reads of stale LDS into dead registers
    wait_lgkm<0>();
    tie();
  }
  dma::wait_vmcnt<0>();
}

template <int BM>
__device__ __forceinline__ void clear(Acc<BM>& acc) {
#pragma unroll
  for (int i = 0; i < BM / 32; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
}

// Whether one of the values a tile multiplies over K tiles [g.kt0, g.kt1) is so small that its parts lose some of it, zeros
// apart.  Values of the same operand beyond the tile's last column count along.
constexpr float kSmall = 0x1p-102f;

template <bool MC, int R, bool DUAL>   // R: rows (KC) of the tile
__device__ __forceinline__ bool any_small(const Args& g, const __amdgpu_buffer_rsrc_t& first, const __amdgpu_buffer_rsrc_t& second, int r0, uint32_t ld) {
  // KC: eight lanes a row of 32 k;  MC: 32 lanes a row of 128 columns
  const int t = threadIdx.x, piece = MC ? t % 32 : t % 8, row = MC ? t / 32 : t / 8;
  constexpr int kStep = MC ? kThreads / 32 : kThreads / 8, kRows = MC ? kBK : R;
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
// (operands of 2^-60 and less next to others of order one, or of 2^40) takes 920 / 911 / 838 us NT / NN / TN for 8 experts of 1024
// rows, [1024, 4096], instead of 403 / 406 / 371; the element-wise kernel takes 840 / 878 / 780 for any values.
constexpr float kTiny = 0x1p-64f, kHuge = 0x1p38f;

template <bool A_MC, bool B_MC, int BM, bool DUAL>
__device__ __forceinline__ bool sums_need_fp32(const Args& g, const Acc<BM>& acc, float operand, int m_lim, int n_lim) {
  const int wave = threadIdx.x / kWave, lane = lane_id();
  const int m0 = (wave / 2) * (BM / 2) + (lane & 15), n0 = (wave % 2) * 64 + 4 * (lane >> 4);
  // twice the bits less one: no sign, zeros at the top; whether there is anything to look at more closely
  uint32_t low = 0xffffffffu, high = 0;
#pragma unroll
  for (int i = 0; i < BM / 32; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const uint32_t t = __float_as_uint(acc[i][j][r]) * 2u - 1u;
        low = low < t ? low : t;
        high = high > t ? high : t;
      }
  bool again = operand >= kHuge, zero = false;
  if (low < 2u * __float_as_uint(kTiny) - 1u || high >= 2u * 0x7f800000u - 1u) {
#pragma unroll
    for (int i = 0; i < BM / 32; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
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
      again |= any_small<A_MC, BM, DUAL>(g, g.rsrc_a, g.rsrc_a2, g.a_r0, g.a_ld) || any_small<B_MC, 128, DUAL>(g, g.rsrc_b, g.rsrc_b2, g.b_r0, g.b_ld);
    return __syncthreads_or(again);
  }
  return false;
}

// A reduction of one or two terms goes to the fp32 instruction at once: its result is rounded once or twice there, and the
// products of parts that are left out, and what the bf16 instruction drops of a sum, are more than that (largest error over the
// sum of the magnitudes, 2^-24: 1.0 / 2.6 over one term, 1.9 / 2.6 over two, 2.5 / 2.3 over three, 3.7 / 2.1 over eight).
constexpr int kFewTerms = 2;

template <bool A_MC, bool B_MC, int BM, bool DUAL>
__device__ __forceinline__ void multiply(const Args& g, Acc<BM>& acc, int m_lim, int n_lim, char* lds) {
  clear<BM>(acc);
  float operand = 0.f;
  if (!A_MC || g.k > kFewTerms) {   // NN / NT: k is a multiple of 4
    multiply_as<A_MC, B_MC, BM, DUAL, false>(g, acc, lds, operand);
    if (!sums_need_fp32<A_MC, B_MC, BM, DUAL>(g, acc, operand, m_lim, n_lim)) return;
    clear<BM>(acc);
  }
  multiply_as<A_MC, B_MC, BM, DUAL, true>(g, acc, lds, operand);
}

// c[m][n] = acc for the tile's rows below m_lim and columns below n (n a multiple of 4, c 16-byte aligned)
template <int BM>
__device__ __forceinline__ void store(const Acc<BM>& acc, float* __restrict__ c, int64_t ldc, int m_lim, int n0, int n) {
  const int wave = threadIdx.x / kWave, lane = lane_id();
  const int wm = (wave / 2) * (BM / 2), wn = (wave % 2) * 64;
#pragma unroll
  for (int i = 0; i < BM / 32; ++i) {
    const int m = wm + 16 * i + (lane & 15);
    if (m >= m_lim) continue;
    float* const row = c + (int64_t)m * ldc;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int col = n0 + wn + 16 * j + 4 * (lane >> 4);
      if (col < n) *(f32x4*)(row + col) = acc[i][j];
    }
  }
}

// Part `part` of tile `tile` (of `tiles`) of a reduction cut into ksplit parts: hands the accumulators over through
// the workspace and returns whether this workgroup was the tile's last, which then holds the sum of all parts in
// `acc`, added in part order whoever came last.  The parts go past the caches (workgroups of a tile sit on different
// XCDs), a part is counted in once its stores are acknowledged, and nobody waits for anybody: see gmm_dma.h.
template <int BM>
__device__ __forceinline__ bool join_parts(Acc<BM>& acc, int tile, int tiles, int part, int ksplit, int32_t* counters,
                                           float* parts, char* lds) {
  constexpr int kThroughCaches = 0x11, kPieces = BM / 32 * 4;   // sc0 | sc1; 16-byte pieces per lane
  const uint32_t lane_off = threadIdx.x * 16u;
  const __amdgpu_buffer_rsrc_t mine = make_rsrc((const char*)parts + ((size_t)part * tiles + tile) * kPartBytes, (uint32_t)kPartBytes);
#pragma unroll
  for (int p = 0; p < kPieces; ++p)
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[p / 4][p % 4]), mine, (int)lane_off, p * (kThreads * 16), kThroughCaches);
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
      const __amdgpu_buffer_rsrc_t theirs = make_rsrc((const char*)parts + ((size_t)q * tiles + tile) * kPartBytes, (uint32_t)kPartBytes);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const f32x4 w = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(theirs, (int)lane_off, (p + u) * (kThreads * 16), kThroughCaches));
        sum[u] = q == 0 ? w : sum[u] + w;
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) acc[p / 4][u] = sum[u];
  }
  if (threadIdx.x == 0) counters[tile] = 0;   // as the launch found it
  return true;
}

// ---- NN / NT ----
// P = gridDim.x workgroups (two per compute unit) walk the list of tiles as those of gmm_dma.h's kernel do.  The tiles of a
// last round that would leave at least half of the workgroups idle are cut along the reduction when there is a
// workspace: with four and a half rounds of long reductions (8 experts of 1024 rows: 4.4 rounds NT, 1.1 NN) the tail
// would otherwise take as long as a full round.
template <bool B_MC, int BM, bool DUAL>
__global__ void __launch_bounds__(kThreads, 2)
gmm_f32_rows_kernel(const float* __restrict__ a, const float* __restrict__ b, float* __restrict__ c, const int32_t* __restrict__ bins,
                    int num_groups, int64_t rows, int k, int n, int tiles_n, const float* __restrict__ a2, const float* __restrict__ b2,
                    int32_t* __restrict__ ws_counters, float* ws_parts, int ws_capacity) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int P = gridDim.x, run = P / kXcds, xcd = blockIdx.x % kXcds, member = blockIdx.x / kXcds;
  const RowTiles<BM> tiles(bins, num_groups, tiles_n, (int)rows, false, 8);
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
    const int row0 = start + tm * BM;
    // up to the expert's last row: the next expert's rows, or rows behind the last bin that nobody may have written, must not
    // have a say in which instruction forms these sums
    const uint32_t a_bytes = clip_bytes((int64_t)(end - row0) * k * 4), b_bytes = (uint32_t)((int64_t)k * n * 4);
    g.rsrc_a = make_rsrc(a + (int64_t)row0 * k, a_bytes);
    g.rsrc_b = make_rsrc(b + (int64_t)e * k * n, b_bytes);
    g.rsrc_a2 = DUAL ? make_rsrc(a2 + (int64_t)row0 * k, a_bytes) : g.rsrc_a;
    g.rsrc_b2 = DUAL ? make_rsrc(b2 + (int64_t)e * k * n, b_bytes) : g.rsrc_b;
    g.b_r0 = tn * kBN;
    g.kt0 = cut ? (int)((int64_t)part * nk / ksplit) : 0;
    g.kt1 = cut ? (int)((int64_t)(part + 1) * nk / ksplit) : nk;
    Acc<BM> acc;
    multiply<false, B_MC, BM, DUAL>(g, acc, end - row0, n - g.b_r0, lds);
    if (!cut || join_parts<BM>(acc, id - full_rounds * P, rest, part, ksplit, ws_counters, ws_parts, lds))
      store<BM>(acc, c + (int64_t)row0 * n, n, end - row0, g.b_r0, n);
    tile_done();
  }
}

// ---- TN ----
// One workgroup per tile and part of its reduction; ksplit is the launch's (> 1: there are few tiles and a workspace).
// Experts are taken longest reduction first (every wave ranks up to 64 of them), so that the last tiles are short ones.
__global__ void __launch_bounds__(kThreads, 2)
gmm_f32_tn_kernel(const float* __restrict__ a, const float* __restrict__ b, float* __restrict__ c, const int32_t* __restrict__ bins,
                  int num_groups, int rows, int k, int n, int tiles_m, int tiles_n, int ksplit, int32_t* __restrict__ ws_counters,
                  float* ws_parts) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int per_group = tiles_m * tiles_n, total = per_group * num_groups;
  const int id = xcd_tile_id(blockIdx.x, 2 * kXcdRun);
  if (id >= total * ksplit) return;
  const int tile = id % total, part = id / total;
  int e = tile / per_group;
  if (num_groups <= kWave) {
    const int lane = lane_id();
    const int mine = lane < num_groups ? bins[lane] - (lane > 0 ? bins[lane - 1] : 0) : -1;
    int rank = 0;
    for (int o = 0; o < num_groups; ++o) {
      const int other = __shfl(mine, o, kWave);
      rank += (other > mine || (other == mine && o < lane)) ? 1 : 0;
    }
    if (lane >= num_groups) rank = -1;
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
  g.a_r0 = tm * 128;
  g.b_r0 = tn * kBN;
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
  Acc<128> acc;
  multiply<true, true, 128, false>(g, acc, k - g.a_r0, n - g.b_r0, lds);
  if (ksplit > 1 && !join_parts<128>(acc, tile, total, part, ksplit, ws_counters, ws_parts, lds)) return;
  store<128>(acc, c + ((int64_t)e * k + g.a_r0) * n, n, k - g.a_r0, g.b_r0, n);
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
// kernel / this one; 64 experts, [1024, 4096]: 1 row 214 / 393, 16: 270 / 405, 32: 347 / 418, 64: 500 / 490;  8, [4096,
// 4096]: 99 / 153, 123 / 153, 170 / 156, 254 / 197;  128, [768, 2048]: 162 / 211, 211 / 221, 269 / 217, 379 / 305).  The size limits are that kernel's.
static inline bool f32_short_tn(int num_groups, int64_t rows, int k) {
  return rows <= 24 * (int64_t)num_groups && ceil_div(k, 128) <= 65535 && num_groups <= 65535;
}

// Tiles of 64 rows up to 192 rows per expert on average: of full ones an expert of that many leaves a quarter and more of
// the multiplications to padding, which this kernel, bound by the matrix cores, pays in full (64 experts of 100 - 156 rows,
// 1024 x 1408: 228 us NT).
constexpr int64_t kF32ShortRows = 192;

}  // namespace

int gmm_f32(const void* a, const void* b, const void* a2, const void* b2, void* c, const int32_t* bins, int num_groups,
                   int64_t rows, int k, int n, int layout, void* workspace, size_t workspace_bytes, hipStream_t s) {
  if (layout == MBX_TN && f32_short_tn(num_groups, rows, k)) return MBX_EUNSUPPORTED;
  if (!f32_ok(a, b, c, rows, k, n, layout) || (a2 && !f32_ok(a2, b2, c, rows, k, n, layout))) return MBX_EUNSUPPORTED;
  const float *ap = (const float*)a, *bp = (const float*)b, *ap2 = (const float*)a2, *bp2 = (const float*)b2;
  float* cp = (float*)c;
  WorkspaceParts ws(Workspace{workspace, workspace_bytes}, f32::kPartBytes);
  const int slots = 2 * persistent_grid((int64_t)1 << 30);   // two workgroups per compute unit
  if (slots / 2 > (int)kWorkspaceCounters) ws.parts = nullptr;
  if (layout == MBX_TN) {
    const int tiles_m = (int)ceil_div(k, 128), tiles_n = (int)ceil_div(n, f32::kBN);
    const int64_t total = (int64_t)tiles_m * tiles_n * num_groups;
    if (total * f32::kMaxKSplit > 0x7fffff00) return MBX_ERANGE;
    int64_t ksplit = 1;
    if (ws.parts && 2 * total <= slots) {
      const int64_t nk = rows / num_groups / f32::kBK;
      ksplit = slots / total;
      ksplit = ksplit > f32::kMaxKSplit ? f32::kMaxKSplit : ksplit;
      ksplit = ksplit > nk / f32::kMinPartTiles ? nk / f32::kMinPartTiles : ksplit;
      ksplit = ksplit * total > ws.capacity ? ws.capacity / total : ksplit;
      ksplit = ksplit < 2 ? 1 : ksplit;
    }
    int rc = allow_lds(f32::gmm_f32_tn_kernel, f32::kLdsBytes);
    if (rc) return rc;
    f32::gmm_f32_tn_kernel<<<(unsigned)xcd_grid(total * ksplit, 2 * kXcdRun), f32::kThreads, f32::kLdsBytes, s>>>(
        ap, bp, cp, bins, num_groups, (int)rows, k, n, tiles_m, tiles_n, (int)ksplit, ws.counters, ws.parts);
    return launch_status();
  }
  const int tiles_n = (int)ceil_div(n, f32::kBN);
  const bool short_tiles = rows <= kF32ShortRows * num_groups;
  if ((ceil_div(rows, 64) + num_groups) * tiles_n > 0x7fffffff) return MBX_ERANGE;
#define MBX_LAUNCH_F32(B_MC, BM, DUAL)                                                                            \
  do {                                                                                                            \
    auto kern = f32::gmm_f32_rows_kernel<B_MC, BM, DUAL>;                                                         \
    int rc = allow_lds(kern, f32::kLdsBytes);                                                                     \
    if (rc) return rc;                                                                                            \
    kern<<<(unsigned)slots, f32::kThreads, f32::kLdsBytes, s>>>(ap, bp, cp, bins, num_groups, rows, k, n, tiles_n, ap2, bp2, \
                                                                ws.counters, ws.parts, ws.capacity);              \
  } while (0)
#define MBX_LAUNCH_F32_BM(B_MC, DUAL) do { if (short_tiles) MBX_LAUNCH_F32(B_MC, 64, DUAL); else MBX_LAUNCH_F32(B_MC, 128, DUAL); } while (0)
  if (layout == MBX_NT) {
    if (a2) MBX_LAUNCH_F32_BM(false, true); else MBX_LAUNCH_F32_BM(false, false);
  } else {
    if (a2) MBX_LAUNCH_F32_BM(true, true); else MBX_LAUNCH_F32_BM(true, false);
  }
#undef MBX_LAUNCH_F32_BM
#undef MBX_LAUNCH_F32
  return launch_status();
}

}  // namespace mbx
