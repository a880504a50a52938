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
// (4 rows of the first: 537 MB stored, 6.2 TB/s.)  Neighbours that store to different rows cost that case 100 instead of 87 us.
//
// Layouts are gmm_dma.h's for strided operands of 128 columns: [k][128] rows, transposing reads.
#include "gmm_common.h"

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

// OUT32: c is fp32.  GATHER: the rows of b are picked through gmm_dma.h's row table (there: gmm_tn_kernel).
template <int DT, bool GATHER, bool OUT32>
__global__ void __launch_bounds__(T::THREADS, kPerCu)
gmm_tn_short_kernel(const uint16_t* __restrict__ a, const uint16_t* __restrict__ b, uint16_t* __restrict__ c,
                    const int32_t* __restrict__ bins, int num_groups, int rows, int k, int n, int tiles_m, int tiles_n,
                    const uint32_t* __restrict__ row_table, const int32_t* __restrict__ src_bins, int src_rows, int n_slots) {
  extern __shared__ __attribute__((aligned(1024))) char lds_generic[];
  const lds_ptr lds = (lds_ptr)lds_generic;
  const uint32_t lds_base = (uint32_t)(uintptr_t)lds;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = lane_id();
  const int per_group = tiles_m * tiles_n, xcd = blockIdx.x % kXcds, member = blockIdx.x / kXcds;
  // Experts that are alike go to the XCDs in whole runs: an expert's panels are then fetched into one L2.  With one of more
  // than twice the average every XCD takes a part of each, those experts first (up to 64 experts; more come as they are).
  int mine = 0, most = 0;
  for (int e0 = 0; e0 < num_groups; e0 += kWave) {
    const int e = e0 + lane;
    mine = e < num_groups ? clamp_row(bins[e], rows) - (e > 0 ? clamp_row(bins[e - 1], rows) : 0) : -1;
    most = mine > most ? mine : most;
  }
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) {
    const int other = __shfl_xor(most, o, kWave);
    most = other > most ? other : most;
  }
  most = __builtin_amdgcn_readfirstlane(most);
  int e, tm, tn;
  // Tile t of an expert: in bands of column tiles whose panel of b takes an L2 1.5 MiB, a band's columns fastest, so that
  // neighbours store to the same rows.
  const int average = (int)((int64_t)rows / num_groups) + 1, fits = 6144 / average;
  int wide = fits > 8 ? fits : 8;
  auto place = [&](int t) {
    const int band = t / (wide * tiles_m), left = tiles_n - band * wide, w = left < wide ? left : wide, in = t - band * wide * tiles_m;
    tm = in / w;
    tn = band * wide + in % w;
  };
  if ((int64_t)most * num_groups <= 2 * (int64_t)rows) {
    const int64_t total = (int64_t)per_group * num_groups, share = (total + kXcds - 1) / kXcds, id = xcd * share + member;
    if (member >= share || id >= total) return;
    e = (int)(id / per_group);
    place((int)(id % per_group));
  } else {
    const int share = (per_group + kXcds - 1) / kXcds;
    wide = 8;   // a part of few panels
    e = member / share;
    const int t = xcd * share + member % share;
    if (e >= num_groups || t >= per_group) return;
    place(t);
    if (num_groups <= kWave) {
      // a full ranking is a loop over the experts in every workgroup: 40 of 250 us for 64 experts of 256 rows
      const bool exists = lane < num_groups, large = exists && (int64_t)mine * num_groups > 2 * (int64_t)rows;
      const uint64_t larger = __ballot(large), others = __ballot(exists && !large), before = ((uint64_t)1 << lane) - 1;
      const int rank = !exists ? -1 : large ? __popcll(larger & before) : __popcll(larger) + __popcll(others & before);
      e = __builtin_amdgcn_readfirstlane((int)__builtin_ctzll(__ballot(rank == e)));
    }
  }
  const int start = e > 0 ? clamp_row(bins[e - 1], rows) : 0;
  int end = clamp_row(bins[e], rows);
  end = end < start ? start : end;
  const int nk = (end - start + T::BK - 1) / T::BK;
  const uint32_t a_ld = (uint32_t)k * 2u, b_ld = (uint32_t)n * 2u;
  // the buffers cover exactly the expert's rows: later ones read as zeros
  const __amdgpu_buffer_rsrc_t ra = make_rsrc(a + (int64_t)start * k, (uint32_t)((int64_t)(end - start) * k * 2));
  const __amdgpu_buffer_rsrc_t rb = GATHER ? make_rsrc(b, clip_bytes((int64_t)src_rows * n * 2))
                                           : make_rsrc(b + (int64_t)start * n, (uint32_t)((int64_t)(end - start) * n * 2));
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
  const int half_at = nk > 0 && end - start - (nk - 1) * T::BK <= 32 ? nk - 1 : -1;
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
  for (int kt = 0; kt < nk; ++kt) {
    __builtin_amdgcn_sched_barrier(0);
    dma::wait_vmcnt<0>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
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
  dma::wait_vmcnt<0>();
  if constexpr (OUT32) dma::block_store_f32<T>(acc, (float*)c + (int64_t)e * k * n, n, tm * T::BM, k, tn * T::BN, n);
  else dma::block_store<DT, T>(acc, c + (int64_t)e * k * n, n, tm * T::BM, k, tn * T::BN, n, lds_generic);
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
    gmm_tn_short_kernel<DT, true, OUT32><<<(unsigned)grid, T::THREADS, kLdsBytes, q.stream>>>(a, b, (uint16_t*)q.c, q.bins, q.num_groups, (int)q.rows, q.k, q.n, tiles_m, tiles_n, q.gather.row_table, q.gather.src_bins, q.gather.src_rows, (int)q.gather.n_slots);
  } else {
    gmm_tn_short_kernel<DT, false, OUT32><<<(unsigned)grid, T::THREADS, kLdsBytes, q.stream>>>(a, b, (uint16_t*)q.c, q.bins, q.num_groups, (int)q.rows, q.k, q.n, tiles_m, tiles_n, nullptr, nullptr, 0, 0);
  }
  return launch_status();
}

}  // namespace tn_short
}  // namespace

// Up to 256 rows per expert on average: beyond, gmm_dma.h's tile hides its latencies behind its products, and its wider tile
// reads less (64 experts, [1024, 4096]: 344 against 366 us at 512 rows; 8 experts, [4096, 14336]: 443 against 447 at 384).
// Up to 1024 rows where all tiles run at once: 256 x 256 tiles would leave most compute units idle (8 experts, [576, 1024]:
// 18.6 against 12.8 us at 512 rows, 26.9 against 20.7 at 1024).
bool gmm_tn_short_takes(const DmaCall& q) {
  const int64_t widest = q.k > q.n ? q.k : q.n;
  if (q.layout != MBX_TN || q.rows * widest * 2 >= ((int64_t)1 << 31)) return false;   // one buffer per operand
  const int64_t tiles = ceil_div(q.k, 128) * ceil_div(q.n, 128) * q.num_groups, at_once = tn_short::kPerCu * (int64_t)persistent_grid((int64_t)1 << 30);
  return q.rows <= (int64_t)(tiles <= at_once ? 1024 : 256) * q.num_groups;
}

int gmm_tn_short(const DmaCall& q) {
  if (q.out32) return q.dtype == MBX_BF16 ? tn_short::launch<MBX_BF16, true>(q) : tn_short::launch<MBX_F16, true>(q);
  return q.dtype == MBX_BF16 ? tn_short::launch<MBX_BF16, false>(q) : tn_short::launch<MBX_F16, false>(q);
}

}  // namespace mbx
