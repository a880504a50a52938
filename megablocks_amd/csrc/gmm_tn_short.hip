// TN products of 16-bit operands (weight gradients) where an expert has few rows: c[e] = a[r_e]^T @ b[r_e] with reductions of a
// few K tiles.
//
// What bounds them: the stores of the products, once, and the latencies around them.  A 256 x 256 tile of gmm_dma.h has a
// compute unit to itself, so with one to four K tiles its first loads, its products and its 128 KiB of stores follow each
// other with nothing beside them: of 240 us for 64 experts of 256 rows, [1024, 4096], 90 are what storing the same
// tiles takes, 105 the products.  Here a workgroup of four waves computes one 128 x 128 tile out of one 32 KiB stage, with
// no pipeline of its own: four workgroups share a compute unit, and one stores while others load and multiply.
// Measured (us, gmm_dma.h's kernel / this one, rows per expert +- 6 %; z: Zipf-distributed, exponent 1.2):
//   64 experts, [1024, 4096]:   4 rows 141 / 87,  64: 156 / 112,  128: 179 / 135,  128z: 180 / 140,  256: 221 / 191
//   16 experts, [1408, 2048]:   28 / 20,  29 / 23,  35 / 27,  37 / 27,  48 / 37
//   8 experts, [4096, 14336]:   202 / 167,  222 / 192,  259 / 232,  265 / 228,  370 / 350
//   128 experts, [768, 2048]:   88 / 66,  100 / 81,  121 / 99,  154 / 139,  174 / 146
//   32 experts, [1032, 2728]:   62 / 60,  64 / 60,  70 / 62,  86 / 76,  92 / 81
// (4 rows of the first: 537 MB stored, 6.2 TB/s; operands in the last-level cache, without Prefetch.)  Neighbours that store to different rows cost that case 100 instead of 87 us.
//
// Layouts are gmm_dma.h's for strided operands of 128 columns: [k][128] rows, transposing reads.
#include "gmm_common.h"

#include <cmath>

namespace mbx {
namespace {

#include "gmm_dma.h"

namespace tn_short {

using dma::clamp_row;
using dma::clip_bytes;
using dma::lds_ptr;
using dma::make_rsrc;

typedef dma::Tile<128, 128, 2, 2, 64, 2> T;   // for its shape; the ring is not used
constexpr uint32_t kStageBytes = T::A_BYTES + T::B_BYTES;
constexpr size_t kLdsBytes = T::EPILOGUE_BYTES > kStageBytes ? T::EPILOGUE_BYTES : kStageBytes;
constexpr int kPerCu = 4;
static_assert(kPerCu * kLdsBytes <= 160 * 1024, "workgroups per compute unit");

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));

template <int DT>
__device__ __forceinline__ f32x4 mfma(const u32x4& a, const u32x4& b, const f32x4& c) {
  if (DT == MBX_BF16) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}

// Which tile the workgroups of an XCD take: at(member) for its `member`-th, in the order they start.
// Experts that are alike go to the XCDs in whole runs: an expert's panels are then fetched into one L2.  With one of more
// than twice the average every XCD takes a part of each, those experts first (up to 64 experts; more come as they are).
struct Tiles {
  struct Tile { int e, tm, tn; };
  int num_groups, rows, tiles_m, tiles_n, xcd, mine = 0, wide;
  bool alike;

  __device__ __forceinline__ Tiles(const int32_t* __restrict__ bins, int num_groups_, int rows_, int tiles_m_, int tiles_n_)
      : num_groups(num_groups_), rows(rows_), tiles_m(tiles_m_), tiles_n(tiles_n_), xcd(blockIdx.x % kXcds) {
    int most = 0;
    for (int e0 = 0; e0 < num_groups; e0 += kWave) {
      const int e = e0 + lane_id();
      mine = e < num_groups ? clamp_row(bins[e], rows) - (e > 0 ? clamp_row(bins[e - 1], rows) : 0) : -1;
      most = mine > most ? mine : most;
    }
    most = wave_max(most);
    alike = (int64_t)__builtin_amdgcn_readfirstlane(most) * num_groups <= 2 * (int64_t)rows;
    // bands of column tiles whose panel of b takes an L2 1.5 MiB; of few panels in a part of an expert
    const int average = (int)((int64_t)rows / num_groups) + 1, fits = 6144 / average;
    wide = alike && fits > 8 ? fits : 8;
    wide = wide < tiles_n ? wide : tiles_n;
  }
  // Tile t of an expert: in bands of column tiles, a band's columns fastest, so that neighbours store to the same rows.
  __device__ __forceinline__ void place(int t, Tile& tile) const {
    const int band = t / (wide * tiles_m), left = tiles_n - band * wide, w = left < wide ? left : wide, in = t - band * wide * tiles_m;
    tile.tm = in / w;
    tile.tn = band * wide + in % w;
  }
  __device__ __forceinline__ bool at(int member, Tile& tile) const {   // false: there is none
    const int per_group = tiles_m * tiles_n;
    if (alike) {
      const int64_t total = (int64_t)per_group * num_groups, share = (total + kXcds - 1) / kXcds, id = xcd * share + member;
      if (member >= share || id >= total) return false;
      tile.e = (int)(id / per_group);
      place((int)(id % per_group), tile);
    } else {
      const int share = (per_group + kXcds - 1) / kXcds;
      tile.e = member / share;
      const int t = xcd * share + member % share;
      if (tile.e >= num_groups || t >= per_group) return false;
      place(t, tile);
      if (num_groups <= kWave) {
        // a full ranking is a loop over the experts in every workgroup: 40 of 250 us for 64 experts of 256 rows
        const int lane = lane_id();
        const bool exists = lane < num_groups, large = exists && (int64_t)mine * num_groups > 2 * (int64_t)rows;
        const uint64_t larger = __ballot(large), others = __ballot(exists && !large), before = ((uint64_t)1 << lane) - 1;
        const int rank = !exists ? -1 : large ? __popcll(larger & before) : __popcll(larger) + __popcll(others & before);
        tile.e = __builtin_amdgcn_readfirstlane((int)__builtin_ctzll(__ballot(rank == tile.e)));
      }
    }
    return true;
  }
};

// An expert's rows, inside [0, rows] and in order whatever the table holds.
__device__ __forceinline__ void expert_rows(const int32_t* __restrict__ bins, int e, int rows, int& start, int& count) {
  start = e > 0 ? clamp_row(bins[e - 1], rows) : 0;
  const int end = clamp_row(bins[e], rows);
  count = end < start ? 0 : end - start;
}

// The operands of the tile a workgroup of this XCD will start with when the ones running now are done, fetched into the L2 by
// those: the rows of a (columns of its row tile) by the workgroups of the tiles beside it, a share each, and the rows of b likewise
// where an expert begins.  A workgroup's first loads otherwise wait for memory that is busy with the stores of the others, a
// few microseconds in each of its 10 to 20: 64 experts, [1024, 4096], operands and products not in the last-level cache: 128 rows
// 184 -> 165 us, 256 rows 238 -> 210.  One dword a lane, a lane a 128-byte line; out of range: no access.
template <int BM, int BN, int AHEAD>
struct Prefetch {
  __amdgpu_buffer_rsrc_t ra, rb;
  uint32_t a_at = 0x80000000u, b_at = 0x80000000u, a = 0, b = 0;
  // behind the workgroup's own first loads
  __device__ __forceinline__ Prefetch(const Tiles& tiles, int e, const uint16_t* __restrict__ pa, const uint16_t* __restrict__ pb,
                                      const int32_t* __restrict__ bins, int k, int n) {
    Tiles::Tile next;
    int start = 0, count = 0;
    if (tiles.at(blockIdx.x / kXcds + AHEAD, next)) {
      expert_rows(bins, next.e, tiles.rows, start, count);
      constexpr int kLinesA = BM * 2 / 128, kLinesB = BN * 2 / 128;   // of a row
      const int thread = threadIdx.x, line_a = next.tn % tiles.wide * 256 + thread;
      const int line_b = next.tm % (AHEAD / 8) * 256 + thread;        // eight column tiles or more at a time
      if (line_a / kLinesA < count) a_at = (uint32_t)(line_a / kLinesA) * (uint32_t)k * 2u + (uint32_t)(next.tm * kLinesA + line_a % kLinesA) * 128u;
      if (line_b / kLinesB < count && next.e != e) b_at = (uint32_t)(line_b / kLinesB) * (uint32_t)n * 2u + (uint32_t)(next.tn * kLinesB + line_b % kLinesB) * 128u;
    }
    ra = make_rsrc(pa + (int64_t)start * k, (uint32_t)((int64_t)count * k * 2));
    rb = make_rsrc(pb + (int64_t)start * n, (uint32_t)((int64_t)count * n * 2));
  }
  __device__ __forceinline__ void issue() {   // where no loads follow that are waited for
    a = __builtin_amdgcn_raw_buffer_load_b32(ra, (int)a_at, 0, 0);
    b = __builtin_amdgcn_raw_buffer_load_b32(rb, (int)b_at, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  }
  __device__ __forceinline__ void arrived() const { asm volatile("" ::"v"(a), "v"(b)); }   // behind the stores
};

// OUT32: c is fp32.  GATHER: the rows of b are picked through gmm_dma.h's row table (there: gmm_tn_kernel).
template <int DT, bool GATHER, bool OUT32, bool AHEAD>
__global__ void __launch_bounds__(T::THREADS, kPerCu)
gmm_tn_short_kernel(const uint16_t* __restrict__ a, const uint16_t* __restrict__ b, uint16_t* __restrict__ c,
                    const int32_t* __restrict__ bins, int num_groups, int rows, int k, int n, int tiles_m, int tiles_n,
                    const uint32_t* __restrict__ row_table, const int32_t* __restrict__ src_bins, int src_rows, int n_slots) {
  extern __shared__ __attribute__((aligned(1024))) char lds_generic[];
  const lds_ptr lds = (lds_ptr)lds_generic;
  const uint32_t lds_base = (uint32_t)(uintptr_t)lds;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = lane_id();
  const Tiles tiles(bins, num_groups, rows, tiles_m, tiles_n);
  Tiles::Tile tile;
  if (!tiles.at(blockIdx.x / kXcds, tile)) return;
  const int e = tile.e, tm = tile.tm, tn = tile.tn;
  int start, count;
  expert_rows(bins, e, rows, start, count);
  const int nk = (count + T::BK - 1) / T::BK;
  const uint32_t a_ld = (uint32_t)k * 2u, b_ld = (uint32_t)n * 2u;
  // the buffers cover exactly the expert's rows: later ones read as zeros
  const __amdgpu_buffer_rsrc_t ra = make_rsrc(a + (int64_t)start * k, (uint32_t)((int64_t)(count) * k * 2));
  const __amdgpu_buffer_rsrc_t rb = GATHER ? make_rsrc(b, clip_bytes((int64_t)src_rows * n * 2))
                                           : make_rsrc(b + (int64_t)start * n, (uint32_t)((int64_t)(count) * n * 2));
  // load j = wave + 4 q (q < 4) of an operand holds rows 4 j .. 4 j + 3 of the K tile, 16 lanes a row
  const uint32_t a_lane = dma::load_lane_offset<true, T::BK, 128>(wave, tm * T::BM, a_ld) + (uint32_t)(4 * wave) * a_ld;
  const uint32_t b_lane = dma::load_lane_offset<true, T::BK, 128>(wave, tn * T::BN, GATHER ? 0u : b_ld) + (GATHER ? 0u : (uint32_t)(4 * wave) * b_ld);
  // GATHER: the table entries of this lane's four rows (zero, past the expert's part: no row)
  __amdgpu_buffer_rsrc_t rt = ra;
  uint32_t entry[4] = {0u, 0u, 0u, 0u}, entry_at[4];
  if constexpr (GATHER) {
    int xs = e > 0 ? src_bins[e - 1] : 0, xe = src_bins[e];
    xs = xs < 0 ? 0 : (xs > n_slots ? n_slots : xs);
    xe = xe < xs ? xs : (xe > n_slots ? n_slots : xe);
    rt = make_rsrc(row_table + xs + (int64_t)dma::kRowTableTile * e, (uint32_t)((xe - xs + dma::kRowTableTile - 1) / dma::kRowTableTile * dma::kRowTableTile) * 4u);
#pragma unroll
    for (int q = 0; q < 4; ++q) entry_at[q] = (uint32_t)dma::row_entry_slot(4 * (wave + 4 * q) + (lane >> 4)) * 4u;
  }
  auto fetch_entries = [&](int kt) {
    if constexpr (GATHER) {
#pragma unroll
      for (int q = 0; q < 4; ++q) entry[q] = __builtin_amdgcn_raw_buffer_load_b32(rt, (int)(entry_at[q] + (uint32_t)kt * (dma::kRowTableTile * 4u)), 0, 0);
    }
  };
  // Of a last K tile of at most 32 rows (half of the experts, where their rows vary around whole K tiles) the second half, all
  // zeros, is neither loaded nor multiplied (64 experts of 256 +- 16 rows, [1024, 4096]: 187 -> 181 us).
  const int half_at = nk > 0 && count - (nk - 1) * T::BK <= 32 ? nk - 1 : -1;
  auto load = [&](int kt) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {   // rows 16 q .. of the K tile
      if (q >= 2 && kt == half_at) break;
      const uint32_t dst = (uint32_t)(wave + 4 * q) * 1024u, row = (uint32_t)(kt * T::BK + 16 * q);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (__attribute__((address_space(3))) void*)(lds + dst), 16, (int)(a_lane + row * a_ld), 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (__attribute__((address_space(3))) void*)(lds + T::A_BYTES + dst), 16,
                                               (int)(GATHER ? b_lane + (entry[q] ^ 0x80000000u) : b_lane + row * b_ld), 0, 0, 0);
    }
  };
  const int wm = (wave / T::WN) * T::WTM, wn = (wave % T::WN) * T::WTN;
  // the fragments of a wave are 32 bytes apart before the swizzle, which exchanges places among its eight: XOR moves from one to the next
  static_assert(T::WTM == 64 && T::WTN == 64, "four fragments");
  const uint32_t fa0 = lds_base + dma::frag_lane_offset<true, T::BK, 128>(wm), fb0 = lds_base + T::A_BYTES + dma::frag_lane_offset<true, T::BK, 128>(wn);
  u32x4 fa[T::TM], fb[T::TN];
  auto read = [&](auto si) {   // the operands of k-step si, all there when it returns
    constexpr int at = decltype(si)::value * 32 * 128 * 2, half = 4 * 128 * 2;
#pragma unroll
    for (int i = 0; i < T::TM; ++i) {
      const u32x2 lo = dma::lds_read_tr16_b64<at>(fa0 ^ (32u * i)), hi = dma::lds_read_tr16_b64<at + half>(fa0 ^ (32u * i));
      fa[i] = u32x4{lo[0], lo[1], hi[0], hi[1]};
    }
#pragma unroll
    for (int j = 0; j < T::TN; ++j) {
      const u32x2 lo = dma::lds_read_tr16_b64<at>(fb0 ^ (32u * j)), hi = dma::lds_read_tr16_b64<at + half>(fb0 ^ (32u * j));
      fb[j] = u32x4{lo[0], lo[1], hi[0], hi[1]};
    }
    dma::wait_frags(fa, fb);
  };
  typename T::Acc acc[T::TM][T::TN];
  auto multiply = [&] {
#pragma unroll
    for (int i = 0; i < T::TM; ++i)
#pragma unroll
      for (int j = 0; j < T::TN; ++j) acc[i][j] = mfma<DT>(fb[j], fa[i], acc[i][j]);
  };
  if (nk > 0) {
    fetch_entries(0);
    load(0);
    fetch_entries(1);
  }
#pragma unroll
  for (int i = 0; i < T::TM; ++i)
#pragma unroll
    for (int j = 0; j < T::TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  Prefetch<T::BM, T::BN, kPerCu * kXcdRun> prefetch(tiles, e, a, b, bins, k, n);
  for (int kt = 0; kt < nk; ++kt) {
    __builtin_amdgcn_sched_barrier(0);
    dma::wait_vmcnt<0>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (AHEAD && kt + 1 == nk) prefetch.issue();
    read(std::integral_constant<int, 0>{});
    multiply();
    __builtin_amdgcn_sched_barrier(0);
    if (kt != half_at) {
      read(std::integral_constant<int, 1>{});
      __builtin_amdgcn_s_barrier();   // every wave has the stage's operands: it can be refilled
      __builtin_amdgcn_sched_barrier(0);
      if (kt + 1 < nk) {
        load(kt + 1);
        fetch_entries(kt + 2);
      }
      multiply();
    }
  }
  if constexpr (OUT32) dma::block_store_f32<T>(acc, (float*)c + (int64_t)e * k * n, n, tm * T::BM, k, tn * T::BN, n);
  else dma::block_store<DT, T>(acc, c + (int64_t)e * k * n, n, tm * T::BM, k, tn * T::BN, n, lds_generic);
  if (AHEAD) prefetch.arrived();
}

// Products of up to kSplitRows rows per expert whose rows are no whole 64-byte pieces: tiles beside each other store parts of the same piece,
// which leave the L2 one by one (59 experts of 35, [2376, 1736]: 13 - 15 % more written than the product has, 154 us; [2376, 1728]: 79).
// From more than kSplitColumns columns on, what is fetched ahead next to such stores costs more than it saves, and so do 256 x 128 tiles, which
// fetch ahead (us, with / without, 256 x 128: 185 / 154, 59 experts of 35; 52 of 82, [1400, 1832]: 104 / 92; 50 launches 9 % on the geometric
// mean, 13 % above 24 column tiles; of up to kSplitColumns columns 5 % the other way, above kSplitRows rows 3 - 9 %, and with whole pieces 4 - 7 %).
constexpr int kSplitRows = 128, kSplitColumns = 1024;
static bool split_rows(const DmaCall& q) { return q.n % 32 != 0 && q.n > kSplitColumns && q.rows <= (int64_t)kSplitRows * q.num_groups; }

// ---- a few hundred rows per expert: choose() ----
// 256 x 128 tiles, two workgroups of four waves to a compute unit, each with three stages of 32 rows: two K tiles under way while one is
// multiplied, one barrier per K tile.
typedef dma::Tile<256, 128, 2, 2, 64, 2> TM;   // for its shape
constexpr int kMidK = 32, kMidStages = 3, kMidPerCu = 2;
constexpr uint32_t kMidA = TM::BM * kMidK * 2, kMidStage = kMidA + TM::BN * kMidK * 2;
constexpr size_t kMidLds = TM::EPILOGUE_BYTES > kMidStages * kMidStage ? TM::EPILOGUE_BYTES : kMidStages * kMidStage;
static_assert(kMidPerCu * kMidLds <= 160 * 1024, "workgroups per compute unit");

template <int N>
__device__ __forceinline__ void wait_lgkm() {
  asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(N) : "memory");
}

template <int DT, bool OUT32>
__global__ void __launch_bounds__(TM::THREADS, kMidPerCu)
gmm_tn_mid_kernel(const uint16_t* __restrict__ a, const uint16_t* __restrict__ b, uint16_t* __restrict__ c,
                  const int32_t* __restrict__ bins, int num_groups, int rows, int k, int n, int tiles_m, int tiles_n) {
  extern __shared__ __attribute__((aligned(1024))) char lds_generic[];
  const lds_ptr lds = (lds_ptr)lds_generic;
  const uint32_t lds_base = (uint32_t)(uintptr_t)lds;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const Tiles tiles(bins, num_groups, rows, tiles_m, tiles_n);
  Tiles::Tile tile;
  if (!tiles.at(blockIdx.x / kXcds, tile)) return;
  const int e = tile.e, tm = tile.tm, tn = tile.tn;
  int start, count;
  expert_rows(bins, e, rows, start, count);
  const int nk = (count + kMidK - 1) / kMidK;
  const uint32_t a_ld = (uint32_t)k * 2u, b_ld = (uint32_t)n * 2u;
  // the buffers cover exactly the expert's rows: later ones read as zeros
  const __amdgpu_buffer_rsrc_t ra = make_rsrc(a + (int64_t)start * k, (uint32_t)((int64_t)(count) * k * 2));
  const __amdgpu_buffer_rsrc_t rb = make_rsrc(b + (int64_t)start * n, (uint32_t)((int64_t)(count) * n * 2));
  // load j = wave + 4 q holds rows 2 j, 2 j + 1 of a (q < 4), rows 4 j .. 4 j + 3 of b (q < 2)
  uint32_t a_at[2];
#pragma unroll
  for (int odd = 0; odd < 2; ++odd) a_at[odd] = dma::load_lane_offset<true, 64, 256>(wave, tm * TM::BM, a_ld, odd != 0) + (uint32_t)(2 * wave + 8 * odd) * a_ld;
  uint32_t b_at = dma::load_lane_offset<true, 64, 128>(wave, tn * TM::BN, b_ld) + (uint32_t)(4 * wave) * b_ld;
  auto load = [&](uint32_t stage) {   // the next K tile
#pragma unroll
    for (int q = 0; q < 4; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (__attribute__((address_space(3))) void*)(lds + (stage + (uint32_t)(wave + 4 * q) * 1024u)), 16,
                                               (int)(a_at[q & 1] + (uint32_t)(q / 2) * 16u * a_ld), 0, 0, 0);
#pragma unroll
    for (int q = 0; q < 2; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (__attribute__((address_space(3))) void*)(lds + (stage + kMidA + (uint32_t)(wave + 4 * q) * 1024u)), 16,
                                               (int)(b_at + (uint32_t)q * 16u * b_ld), 0, 0, 0);
    a_at[0] += kMidK * a_ld;
    a_at[1] += kMidK * a_ld;
    b_at += kMidK * b_ld;
  };
  const int wm = (wave / TM::WN) * TM::WTM, wn = (wave % TM::WN) * TM::WTN;
  // XOR moves from one fragment of a wave to the next (its 128 / 64 columns start at a multiple of as many)
  const uint32_t fa0 = lds_base + dma::frag_lane_offset<true, 64, 256>(wm), fb0 = lds_base + kMidA + dma::frag_lane_offset<true, 64, 128>(wn);
  typename TM::Acc acc[TM::TM][TM::TN];
#pragma unroll
  for (int i = 0; i < TM::TM; ++i)
#pragma unroll
    for (int j = 0; j < TM::TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  uint32_t at = 0, to = 2 * kMidStage;
  if (nk > 0) load(0);
  if (nk > 1) load(kMidStage);
  Prefetch<TM::BM, TM::BN, kMidPerCu * kXcdRun> prefetch(tiles, e, a, b, bins, k, n);
  for (int kt = 0; kt < nk; ++kt) {
    __builtin_amdgcn_sched_barrier(0);
    if (kt + 1 < nk) dma::wait_vmcnt<6>(); else dma::wait_vmcnt<0>();   // K tile kt is there, kt + 1 under way
    __builtin_amdgcn_s_barrier();    // ... for every wave, and nobody reads the stage of K tile kt - 1 any more
    __builtin_amdgcn_sched_barrier(0);
    u32x2 pa[TM::TM][2], pb[TM::TN][2];
#pragma unroll
    for (int j = 0; j < TM::TN; ++j) {
      pb[j][0] = dma::lds_read_tr16_b64<0>((fb0 + at) ^ (32u * j));
      pb[j][1] = dma::lds_read_tr16_b64<4 * 128 * 2>((fb0 + at) ^ (32u * j));
    }
#pragma unroll
    for (int i = 0; i < TM::TM; ++i) {
      pa[i][0] = dma::lds_read_tr16_b64<0>((fa0 + at) ^ (32u * i));
      pa[i][1] = dma::lds_read_tr16_b64<4 * 256 * 2>((fa0 + at) ^ (32u * i));
    }
    if (kt + 2 < nk) load(to);
    if (kt + 1 == nk) prefetch.issue();
    u32x4 fb[TM::TN];
    dma::static_for<TM::TM>([&](auto ii) {
      constexpr int i = decltype(ii)::value, left = 2 * (TM::TM - 1 - i);
      wait_lgkm<left>();
      asm volatile("" : "+v"(pa[i][0]), "+v"(pa[i][1]));
      if constexpr (i == 0) {
#pragma unroll
        for (int j = 0; j < TM::TN; ++j) {
          asm volatile("" : "+v"(pb[j][0]), "+v"(pb[j][1]));
          fb[j] = u32x4{pb[j][0][0], pb[j][0][1], pb[j][1][0], pb[j][1][1]};
        }
      }
      const u32x4 fa = {pa[i][0][0], pa[i][0][1], pa[i][1][0], pa[i][1][1]};
#pragma unroll
      for (int j = 0; j < TM::TN; ++j) acc[i][j] = mfma<DT>(fb[j], fa, acc[i][j]);
      __builtin_amdgcn_sched_barrier(0);
    });
    at = at == (kMidStages - 1) * kMidStage ? 0 : at + kMidStage;
    to = to == (kMidStages - 1) * kMidStage ? 0 : to + kMidStage;
  }
  if constexpr (OUT32) dma::block_store_f32<TM>(acc, (float*)c + (int64_t)e * k * n, n, tm * TM::BM, k, tn * TM::BN, n);
  else dma::block_store<DT, TM>(acc, c + (int64_t)e * k * n, n, tm * TM::BM, k, tn * TM::BN, n, lds_generic);
  prefetch.arrived();
}

template <int DT, bool OUT32>
int launch_mid(const DmaCall& q) {
  const int tiles_m = (int)ceil_div(q.k, TM::BM), tiles_n = (int)ceil_div(q.n, TM::BN);
  const int64_t grid = ceil_div((int64_t)tiles_m * tiles_n, kXcds) * q.num_groups * kXcds;
  if (grid > 0x7fffffff) return MBX_ERANGE;
  auto kern = gmm_tn_mid_kernel<DT, OUT32>;
  const int rc = allow_lds(kern, kMidLds);
  if (rc) return rc;
  kern<<<(unsigned)grid, TM::THREADS, kMidLds, q.stream>>>((const uint16_t*)q.a, (const uint16_t*)q.b, (uint16_t*)q.c, q.bins, q.num_groups, (int)q.rows, q.k, q.n, tiles_m, tiles_n);
  return launch_status();
}

template <int DT, bool OUT32>
int launch(const DmaCall& q) {
  const int tiles_m = (int)ceil_div(q.k, T::BM), tiles_n = (int)ceil_div(q.n, T::BN);
  const int64_t grid = ceil_div((int64_t)tiles_m * tiles_n, kXcds) * q.num_groups * kXcds;
  if (grid > 0x7fffffff) return MBX_ERANGE;
  const uint16_t *a = (const uint16_t*)q.a, *b = (const uint16_t*)q.b;
  if (q.gather.slots) {
    if (!q.gather.src_bins || !q.gather.row_table || q.gather.top_k <= 0 || q.gather.n_slots > 0x7fffffff) return MBX_EINVAL;
    if (!q.gather.table_ready) dma::build_row_table(q);
    gmm_tn_short_kernel<DT, true, OUT32, false><<<(unsigned)grid, T::THREADS, kLdsBytes, q.stream>>>(a, b, (uint16_t*)q.c, q.bins, q.num_groups, (int)q.rows, q.k, q.n, tiles_m, tiles_n, q.gather.row_table, q.gather.src_bins, q.gather.src_rows, (int)q.gather.n_slots);
    return launch_status();
  }
  auto kern = split_rows(q) ? gmm_tn_short_kernel<DT, false, OUT32, false> : gmm_tn_short_kernel<DT, false, OUT32, true>;
  kern<<<(unsigned)grid, T::THREADS, kLdsBytes, q.stream>>>(a, b, (uint16_t*)q.c, q.bins, q.num_groups, (int)q.rows, q.k, q.n, tiles_m, tiles_n, nullptr, nullptr, 0, 0);
  return launch_status();
}

enum Kernel { kDma, kShort, kMid };   // gmm_dma.h's 256 x 256 tiles, 128 x 128 of 64 rows, 256 x 128 of 32 rows

// What the kernel's launch is estimated to take, us: rounds of tiles, each a start and so much per 64 rows, and no less than the
// operands and products at the rate it moves them.  A last round that is not full costs `part` of one with the compute units' first
// workgroups and grows from there to a whole one.  Fitted to 472 launches (4 - 128 experts of 280 - 1300 rows, [704 - 8192, 512 - 4096],
// memory that is not in the last-level cache); rms 11 %.
struct Cost {
  int height, width, per_cu;
  double start, tile, k_tile, part, rate;
  double operator()(const DmaCall& q, double units, double average) const {
    const double all = (double)ceil_div(q.k, height) * ceil_div(q.n, width) * q.num_groups / (per_cu * units), full = floor(all), rest = all - full;
    const double one = 1.0 / per_cu, grown = per_cu == 1 ? rest : rest > one ? (rest - one) / (1 - one) : 0.0;
    const double rounds = full + (rest > 0 ? part + (1 - part) * grown : 0.0);
    const double mb = ((double)q.rows * (q.k + q.n) + (double)q.num_groups * q.k * q.n) * 2e-6;
    return start + fmax(rounds * (tile + k_tile * average / 64), mb / rate);
  }
};
constexpr Cost kCosts[] = {{256, 256, 1, 5.0, 6.2, 1.59, 0.58, 2.96}, {128, 128, kPerCu, 4.8, 0.75, 2.35, 0.46, 3.62}, {256, 128, kMidPerCu, 4.9, 3.3, 2.01, 0.53, 3.61}};

// Up to 256 rows per expert on average 128 x 128 tiles: beyond, gmm_dma.h's tile hides its latencies behind its products, and its
// wider tile reads less.  Up to 1024 rows where all of them run at once: 256 x 256 tiles would leave most compute units idle (8
// experts, [576, 1024]: 18.6 against 12.8 us at 512 rows, 26.9 against 20.7 at 1024).
// 256 x 128 tiles out of three small stages where there are five rounds of them, up to 512 rows per expert on average, and of few rows
// where no half of a row of them is empty: they read a quarter less than 128 x 128 tiles and need a third fewer workgroups, but
// their last round is longer (us, this / 128 x 128, gmm_dma.h's above 256 rows; operands and products not in the last-level cache:
// 64 experts, [1024, 4096]: 64 rows 134 / 135, 128: 155 / 170, 256: 203 / 216, 512: 318 / 330;  8, [4096, 14336]: 250: 333 / 345, 500: 522 / 515,
// 600: 603 / 574;  64, [2048, 1408]: 100: 106 / 99, 200: 134 / 133, 300: 172 / 176;  16 of 300, [2048, 1408], three rounds: 53 / 46).
// From 256 to 768 rows another kernel than these lines say where its estimate is shorter by a sixteenth: half-empty last rounds and
// half-empty tiles decide there.  135 launches that the estimates were not fitted to (4 - 128 experts, [704 - 8192, 512 - 4096] at random): 256 - 320
// rows 15 % shorter on the geometric mean, to 400 8 %, to 512 6 %, to 768 3 %, four of them 3 - 9 % longer; above 768 rows they gain nothing.
// (From / to: 64 experts of 300, [1408, 512]: 59 / 43; 64 of 520, [2304, 576]: 148 / 108; 16 of 300, [3072, 768]: 44 / 36; 8 of 450, [1408, 2048]: 35 / 30;
// 12 of 500, [1472, 1344]: 41 / 42; 32 of 670, [1664, 832]: 88 / 96.)  128 x 128 tiles only up to 512 rows: beyond, narrow products take
// longer than estimated (54 of 755, [176, 6184]: 222 us against 170 with gmm_dma.h's; 93 of 648, [1392, 216]: 85 / 78).
// All of this against the lines on rows alone and no fetching ahead, 500 launches that none of it was fitted to (2 - 128 experts of 20 - 1100
// rows, [128 - 8192, 128 - 8192], half of them odd): 5 % shorter on the geometric mean, 35 by more than
// 3 % longer (few rows and few column tiles, 92 experts of 27, [3072, 448]: 61 / 73; half-empty tiles, 84 of 478, [328, 7368]: 351 / 387).
static Kernel choose(const DmaCall& q) {
  const double units = persistent_grid((int64_t)1 << 30);
  const int64_t average = q.rows / q.num_groups, tiles = ceil_div(q.k, 128) * ceil_div(q.n, 128) * q.num_groups;
  const int64_t mid_tiles = ceil_div(q.k, TM::BM) * ceil_div(q.n, TM::BN) * q.num_groups;
  Kernel kernel = q.rows <= (int64_t)((double)tiles <= kPerCu * units ? 1024 : 256) * q.num_groups ? kShort : kDma;
  if (q.gather.slots) return kernel;
  if (average > 64 && average <= 512 && !split_rows(q) && (double)mid_tiles >= 5 * kMidPerCu * units && (average > 256 || q.k % TM::BM == 0 || q.k % TM::BM > TM::BM / 2)) kernel = kMid;
  if (average < 256 || average > 768) return kernel;
  const double here = kCosts[kernel](q, units, (double)average);
  for (Kernel other : {kDma, kShort, kMid})
    if ((other != kShort || average <= 512) && kCosts[other](q, units, (double)average) < fmin(0.94 * here, kCosts[kernel](q, units, (double)average))) kernel = other;
  return kernel;
}

}  // namespace tn_short
}  // namespace

bool gmm_tn_short_takes(const DmaCall& q) {
  const int64_t widest = q.k > q.n ? q.k : q.n;
  if (q.layout != MBX_TN || q.rows * widest * 2 >= ((int64_t)1 << 31)) return false;   // one buffer per operand
  return tn_short::choose(q) != tn_short::kDma;
}

int gmm_tn_short_choice(const DmaCall& q) {
  const tn_short::Kernel kernel = gmm_tn_short_takes(q) ? tn_short::choose(q) : tn_short::kDma;
  return kernel == tn_short::kShort && !tn_short::split_rows(q) ? 3 : (int)kernel;
}

int gmm_tn_short(const DmaCall& q) {
  const bool mid = tn_short::choose(q) == tn_short::kMid;
  if (q.out32) {
    if (mid) return q.dtype == MBX_BF16 ? tn_short::launch_mid<MBX_BF16, true>(q) : tn_short::launch_mid<MBX_F16, true>(q);
    return q.dtype == MBX_BF16 ? tn_short::launch<MBX_BF16, true>(q) : tn_short::launch<MBX_F16, true>(q);
  }
  if (mid) return q.dtype == MBX_BF16 ? tn_short::launch_mid<MBX_BF16, false>(q) : tn_short::launch_mid<MBX_F16, false>(q);
  return q.dtype == MBX_BF16 ? tn_short::launch<MBX_BF16, false>(q) : tn_short::launch<MBX_F16, false>(q);
}

}  // namespace mbx
