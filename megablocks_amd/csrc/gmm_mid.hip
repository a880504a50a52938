// NT products of 16-bit operands where an expert has a few dozen rows: short prompts, decoding of larger batches, small
// training batches over many experts.
//
// What bounds them: the reading of the weights, as with a handful of rows (gmm_few.hip), but with products that want the
// operands in LDS.  gmm_dma.h's 128 x 256 tiles have a compute unit each: the first loads and the stores of a tile stand
// alone, and 350 tiles on 256 compute units take as long as 512.  Here a workgroup of four waves computes a 64 x 256 tile out of one
// 40 KiB stage, with no pipeline of its own: four workgroups share a compute unit, their loads under way in turn, and
// a launch of up to 1024 tiles is one round.
// Measured (us, gmm_dma.h's kernel / this one; gated first products, first product and activation, product and its gradient):
//   64 experts x 24 rows, [1408, 2048]: 154 / 136, 96 / 68, 89 / 70;  x 40: 174 / 137, 97 / 71, 102 / 71
//   32 x 24, [2816, 2048]: 174 / 135, 98 / 69, 90 / 69;  8 x 24, [14336, 4096]: 405 / 332, 216 / 161, 222 / 165
//   8 x 32, [11008, 4096]: 321 / 258, 181 / 129, 190 / 131;  64 x 32, [1408, 512]: 38 / 30, 24 / 18, 30 / 21
//   64 x 24, [4096, 1024]: 200 / 193, 105 / 99, 120 / 101;  128 x 24, [2048, 768]: 159 / 148, 86 / 77, 100 / 79
// (369 MB of weights in 68 us: 5.4 TB/s.)
//
// Layouts are gmm_dma.h's for operands whose reduction is contiguous: rows of 128 bytes.
#include "gmm_common.h"

#include <cmath>

namespace mbx {
namespace {

#include "gmm_dma.h"

namespace mid {

using dma::clip_bytes;
using dma::lds_ptr;
using dma::make_rsrc;

// What dma::block_store() wants to know of a tile.
struct T {
  static constexpr int BM = 64, BN = 256, BK = 64, WM = 1, WN = 4, WAVES = 4, THREADS = 256, MF = 16;
  static constexpr int WTM = 64, WTN = 64, TM = 4, TN = 4;
  typedef f32x4 Acc;
  static constexpr int A_BYTES = BM * BK * 2, B_BYTES = BN * BK * 2;
  static constexpr size_t EPILOGUE_BYTES = (size_t)BM * (BN * 2 + 16), LDS_BYTES = A_BYTES + B_BYTES;
};
static_assert(T::EPILOGUE_BYTES <= T::LDS_BYTES && 4 * T::LDS_BYTES <= 160 * 1024, "four workgroups per compute unit");

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));

template <int DT>
__device__ __forceinline__ f32x4 mfma(const u32x4& a, const u32x4& b, const f32x4& c) {
  if (DT == MBX_BF16) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}

// The epilogues that fetch inputs of their own hold more registers.
constexpr int per_cu(int epi) { return dma::epi_is_dglu(epi) ? 2 : epi == dma::kEpiDact ? 3 : 4; }

// Parameters as those of gmm_dma.h's gmm_rows_kernel.
template <int DT, int EPI, bool GATHER>
__global__ void __launch_bounds__(T::THREADS, per_cu(EPI))
gmm_mid_kernel(const uint16_t* __restrict__ a, const uint16_t* __restrict__ b, uint16_t* __restrict__ c, const int32_t* __restrict__ bins,
               int num_groups, int rows, int k, int n, int tiles_n, const uint16_t* __restrict__ a2, const uint16_t* __restrict__ b2,
               uint16_t* __restrict__ extra, uint16_t* __restrict__ out2, const int32_t* __restrict__ slots,
               const int32_t* __restrict__ src_bins, int top_k, int src_rows) {
  extern __shared__ __attribute__((aligned(1024))) char lds_generic[];
  constexpr bool kGlu = dma::epi_is_glu(EPI), kDglu = dma::epi_is_dglu(EPI);
  constexpr int kTileCols = kGlu ? T::BN / 2 : T::BN;
  const lds_ptr lds = (lds_ptr)lds_generic;
  const uint32_t lds_base = (uint32_t)(uintptr_t)lds;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = lane_id();
  // the tiles in equal consecutive shares to the XCDs: an expert's row tiles find its weights in one L2
  const dma::RowTiles<T::BM> tiles(bins, num_groups, tiles_n, rows, false, 8);
  const int share = (tiles.total + kXcds - 1) / kXcds, member = blockIdx.x / kXcds, id = (int)(blockIdx.x % kXcds) * share + member;
  if (member >= share || id >= tiles.total) return;
  int e, start, end, tm, tn;
  tiles.find(id, e, start, end, tm, tn);
  const int row0 = start + tm * T::BM, n0 = tn * kTileCols;

  const uint32_t ld = (uint32_t)k * 2u, b_bytes = (uint32_t)((int64_t)k * n * 2);
  const __amdgpu_buffer_rsrc_t ra = GATHER ? make_rsrc(a, clip_bytes((int64_t)src_rows * k * 2)) : make_rsrc(a + (int64_t)row0 * k, clip_bytes((int64_t)(end - row0) * k * 2));
  const __amdgpu_buffer_rsrc_t rb = make_rsrc(b + (int64_t)e * k * n, b_bytes), rb2 = kGlu ? make_rsrc(b2 + (int64_t)e * k * n, b_bytes) : rb;
  // A: load j = wave + 4 q (q < 2) holds rows 8 j .. 8 j + 7
  uint32_t a_off[2];
  if constexpr (GATHER) {
    const int src_start = e > 0 ? src_bins[e - 1] : 0;
    const int64_t slots_end = (int64_t)src_rows * top_k;
    const int limit = (int)(src_bins[e] < slots_end ? src_bins[e] : slots_end);
    const uint32_t piece = dma::load_lane_offset<false, T::BK, T::BM>(wave, 0, 0u);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int r = tm * T::BM + 8 * (wave + 4 * q) + (lane >> 3), j = (src_start < 0 ? 0 : src_start) + r;
      const int slot = start + r < end && j < limit ? slots[j] : -1, row = slot >= 0 ? slot / top_k : src_rows;
      a_off[q] = row < src_rows ? (uint32_t)row * ld + piece : 0x80000000u;
    }
  } else {
#pragma unroll
    for (int q = 0; q < 2; ++q) a_off[q] = dma::load_lane_offset<false, T::BK, T::BM>(wave, 0, ld) + (uint32_t)(8 * (wave + 4 * q)) * ld;
  }
  // B: load j = wave + 4 q (q < 8) holds rows 8 j ..; with the gate the upper half of them come from the second matrix
  const uint32_t b_lane = dma::load_lane_offset<false, T::BK, T::BN>(wave, n0, ld) + (uint32_t)(8 * wave) * ld;
  const int piece_k = 8 * ((lane & 7) ^ ((4 * (wave & 1) + (lane >> 4)) & 7));   // first k of this lane's pieces
  const int nk = (k + T::BK - 1) / T::BK;
  // The workgroups start at different places of the reduction and go round: started together, they would all read the first
  // bytes of rows that are often a power of two apart, from a few memory channels (32 experts of 24 rows, [2816, 2048]: 90
  // us, 69 this way).  A column's place does not depend on the epilogue: the product of a launch with one is the plain
  // launch's, bit for bit.
  const int turn = (int)(((uint32_t)(n0 / T::BN) * 5u + (uint32_t)e * 3u) % (uint32_t)nk);
  auto load = [&](int kt) {
    const int kk = kt + turn < nk ? kt + turn : kt + turn - nk;
    const uint32_t past = kk * T::BK + piece_k < k ? 0u : 0x80000000u, at = (uint32_t)kk * 128u;   // pieces past the end of the reduction read as zeros
#pragma unroll
    for (int q = 0; q < 2; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (__attribute__((address_space(3))) void*)(lds + (uint32_t)(wave + 4 * q) * 1024u), 16, (int)((a_off[q] + at) | past | (a_off[q] & 0x80000000u)), 0, 0, 0);
#pragma unroll
    for (int q = 0; q < 8; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(kGlu && q >= 4 ? rb2 : rb, (__attribute__((address_space(3))) void*)(lds + T::A_BYTES + (uint32_t)(wave + 4 * q) * 1024u), 16,
                                               (int)((b_lane + at + (uint32_t)(32 * (kGlu ? q % 4 : q)) * ld) | past), 0, 0, 0);
  };
  const int wn = wave * T::WTN;
  const uint32_t fa0 = dma::frag_lane_offset<false, T::BK, T::BM>(0), fb0 = dma::frag_lane_offset<false, T::BK, T::BN>(wn);
  u32x4 fa[T::TM], fb[T::TN];
  auto read = [&](auto si) {   // the operands of k-step si, all there when it returns
    constexpr int s = decltype(si)::value;
    dma::static_for<T::TM>([&](auto ii) { constexpr int i = decltype(ii)::value; fa[i] = dma::read_frag_kc<s, i * 16 * 128>(lds_base, fa0); });
    dma::static_for<T::TN>([&](auto ji) { constexpr int j = decltype(ji)::value; fb[j] = dma::read_frag_kc<s, j * 16 * 128>(lds_base + T::A_BYTES, fb0); });
    dma::wait_frags(fa, fb);
  };
  T::Acc acc[T::TM][T::TN];
  auto multiply = [&] {
#pragma unroll
    for (int i = 0; i < T::TM; ++i)
#pragma unroll
      for (int j = 0; j < T::TN; ++j) acc[i][j] = mfma<DT>(fb[j], fa[i], acc[i][j]);
  };
  load(0);
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
    read(std::integral_constant<int, 1>{});
    __builtin_amdgcn_s_barrier();   // every wave has the stage's operands: it can be refilled
    __builtin_amdgcn_sched_barrier(0);
    if (kt + 1 < nk) load(kt + 1);
    multiply();
  }
  uint16_t* const c_tile = dma::epi_c_optional(EPI) && c == nullptr ? nullptr : c + (int64_t)row0 * n;
  uint16_t* const e_tile = EPI != dma::kEpiNone ? extra + (int64_t)row0 * n : nullptr;
  const uint16_t* const p_tile = kDglu ? a2 + (int64_t)row0 * n : nullptr;
  uint16_t* const o_tile = kDglu || kGlu ? out2 + (int64_t)row0 * n : nullptr;
  dma::block_store<DT, T, EPI>(acc, c_tile, n, 0, end - row0, n0, n, lds_generic, e_tile, p_tile, o_tile);
}

template <int DT, int EPI, bool GATHER>
int launch(const DmaCall& q) {
  const int tiles_n = (int)ceil_div(q.n, dma::epi_is_glu(EPI) ? T::BN / 2 : T::BN);
  // an upper bound: the row counts are only known on the device
  const int64_t row_tiles = (q.rows < q.num_groups ? q.rows : q.num_groups) + q.rows / T::BM;
  const int64_t grid = ceil_div(row_tiles * tiles_n, kXcds) * kXcds;
  if (grid > 0x7fffffff) return MBX_ERANGE;
  gmm_mid_kernel<DT, EPI, GATHER><<<(unsigned)grid, T::THREADS, T::LDS_BYTES, q.stream>>>(
      (const uint16_t*)q.a, (const uint16_t*)q.b, (uint16_t*)q.c, q.bins, q.num_groups, (int)q.rows, q.k, q.n, tiles_n,
      (const uint16_t*)q.a2, (const uint16_t*)q.b2, (uint16_t*)q.extra, (uint16_t*)q.out2, q.gather.slots, q.gather.src_bins,
      q.gather.top_k, q.gather.src_rows);
  return launch_status();
}

template <int DT>
int dispatch(const DmaCall& q) {
#define MBX_MID(EPI) (q.gather.slots ? launch<DT, EPI, true>(q) : launch<DT, EPI, false>(q))
  switch (q.epi) {
    case dma::kEpiNone: return MBX_MID(dma::kEpiNone);
    case dma::kEpiAct: return MBX_MID(dma::kEpiAct);
    case dma::kEpiGluSilu: return MBX_MID(dma::kEpiGluSilu);
    case dma::kEpiGluGelu: return MBX_MID(dma::kEpiGluGelu);
    case dma::kEpiDact: return launch<DT, dma::kEpiDact, false>(q);
    case dma::kEpiDgluSilu: return launch<DT, dma::kEpiDgluSilu, false>(q);
    default: return launch<DT, dma::kEpiDgluGelu, false>(q);
  }
#undef MBX_MID
}

}  // namespace mid
}  // namespace

// Up to 40 rows per expert on average (from 64 on an expert's weights are read twice: 64 experts, [4096, 1024], 107 / 101 us at
// 40 rows, 108 / 111 at 52) and more tiles than compute units: with fewer a workgroup is alone on its compute unit and
// waits out every stage, where gmm_dma.h's ring has three under way (16 experts, [2816, 1024], 176 tiles: 19.5 / 21.4; 16,
// [1024, 3072], 64 tiles: 33 / 51).  The number of experts that get rows is an expectation: rows that choose evenly.  Skewed rows
// (gated, plain, gradient, 16 and 38 rows on average): Zipf-distributed, exponent 1.2, like even ones (64 experts top-6, [1408,
// 2048]: 172, 94, 101 / 135, 67, 69 and 194, 93, 99 / 153, 70, 73; 8 top-2, [14336, 4096]: 342, 205, 210 / 353, 160, 164
// and 363, 216, 223 / 352, 168, 172); where a few experts get everything there are too few tiles again, and the launch is short
// (all on top_k of them: 30, 28, 32 / 35, 33, 35 and 51, 29, 33 / 42, 34, 36; 86, 68, 72 / 98, 63, 66 and 126, 56, 63 / 136, 66, 82).
// The epilogues do not enter the rule: the product of a launch with one is the plain launch's, bit for bit.  NN launches stay
// with gmm_dma.h, which cuts their last round along the reduction (8 experts, [4096, 14336]: 210 / 314).
bool gmm_mid_takes(const DmaCall& q) {
  if (q.layout != MBX_NT || (q.a2 && !dma::epi_is_dglu(q.epi)) || q.rows > 40 * (int64_t)q.num_groups) return false;
  const double experts = q.num_groups * (1.0 - pow(1.0 - 1.0 / q.num_groups, (double)q.rows));
  return experts * (double)ceil_div(q.n, mid::T::BN) > persistent_grid((int64_t)1 << 30);
}

int gmm_mid(const DmaCall& q) { return q.dtype == MBX_BF16 ? mid::dispatch<MBX_BF16>(q) : mid::dispatch<MBX_F16>(q); }

}  // namespace mbx
