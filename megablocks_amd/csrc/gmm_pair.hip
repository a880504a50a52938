// NN / NT products of 16-bit operands in launches of few tiles: a few hundred rows per expert, small layers.
//
// What bounds them: with gmm_dma.h's 256 x 256 tiles, one workgroup to a compute unit, the rounds.  12 experts of 500 rows with a
// [2728, 1032] product are 264 tiles on 256 compute units, their other product is 130 tiles with reductions of 43 K tiles each, and
// within a round the first loads and the stores of all tiles come at the same time.  Here a workgroup of four waves computes a
// 128 x 128 tile, two workgroups share a compute unit, each with three 16 KiB stages of A and two of B (together all of the LDS), and
// one stores or waits while the other multiplies.
//
// Layouts and the order of the sums are gmm_dma.h's: the products are bit for bit those of its kernels.
#include "gmm_common.h"

#include <cmath>

namespace mbx {
namespace {

#include "gmm_dma.h"

namespace pair {

using dma::clip_bytes;
using dma::lds_ptr;
using dma::make_rsrc;

typedef dma::Tile<128, 128, 2, 2, 64, 2> T;   // for its shape
constexpr uint32_t kARing = 3 * T::A_BYTES, kRing = kARing + 2 * T::B_BYTES;   // three stages of A, two of B behind them
constexpr size_t kLdsBytes = kRing;
constexpr int kPerCu = 2;
static_assert(kPerCu * kLdsBytes <= 160 * 1024 && T::EPILOGUE_BYTES + T::BM * 8 <= kLdsBytes, "workgroups per compute unit");

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));

template <int DT>
__device__ __forceinline__ f32x4 mfma(const u32x4& a, const u32x4& b, const f32x4& c) {
  if (DT == MBX_BF16) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}

// Parameters as those of gmm_dma.h's gmm_rows_kernel.
template <int DT, bool B_MC, int EPI, bool GATHER, bool DUAL>
__global__ void __launch_bounds__(T::THREADS, kPerCu)
gmm_pair_kernel(const uint16_t* __restrict__ a, const uint16_t* __restrict__ b, uint16_t* __restrict__ c, const int32_t* __restrict__ bins,
                int num_groups, int rows, int k, int n, int tiles_n, const uint16_t* __restrict__ a2, const uint16_t* __restrict__ b2,
                uint16_t* __restrict__ extra, uint16_t* __restrict__ out2, const int32_t* __restrict__ slots,
                const int32_t* __restrict__ src_bins, int top_k, int src_rows, const void* __restrict__ combine_weights, int combine_w_dtype,
                int combine_tokens) {
  extern __shared__ __attribute__((aligned(1024))) char lds_generic[];
  constexpr bool kGlu = dma::epi_is_glu(EPI), kDglu = dma::epi_is_dglu(EPI);
  constexpr int kTileCols = kGlu ? T::BN / 2 : T::BN;   // the same columns of both first products side by side
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

  const uint32_t a_ld = (uint32_t)k * 2u, b_ld = (uint32_t)(B_MC ? n : k) * 2u, b_bytes = (uint32_t)((int64_t)k * n * 2);
  const uint32_t a_bytes = GATHER ? clip_bytes((int64_t)src_rows * k * 2) : clip_bytes((int64_t)(end - row0) * k * 2);
  const __amdgpu_buffer_rsrc_t ra1 = make_rsrc(GATHER ? a : a + (int64_t)row0 * k, a_bytes), ra2 = DUAL ? make_rsrc(a2 + (int64_t)row0 * k, a_bytes) : ra1;
  const __amdgpu_buffer_rsrc_t rb1 = make_rsrc(b + (int64_t)e * k * n, b_bytes), rb2 = DUAL || kGlu ? make_rsrc(b2 + (int64_t)e * k * n, b_bytes) : rb1;
  // A, and B of NT: load j = wave + 4 q holds rows 8 j .. 8 j + 7;  B of NN: rows k = 4 j .. 4 j + 3
  uint32_t a_off[GATHER ? 4 : 1];
  if constexpr (GATHER) {
    const int src_start = e > 0 ? src_bins[e - 1] : 0;
    const int64_t slots_end = (int64_t)src_rows * top_k;
    const int limit = (int)(src_bins[e] < slots_end ? src_bins[e] : slots_end);
    const uint32_t piece = dma::load_lane_offset<false, T::BK, T::BM>(wave, 0, 0u);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = tm * T::BM + 8 * (wave + 4 * q) + (lane >> 3), j = (src_start < 0 ? 0 : src_start) + r;
      const int slot = start + r < end && j < limit ? slots[j] : -1, row = slot >= 0 ? slot / top_k : src_rows;
      a_off[q] = row < src_rows ? (uint32_t)row * a_ld + piece : 0x80000000u;
    }
  } else {
    a_off[0] = dma::load_lane_offset<false, T::BK, T::BM>(wave, 0, a_ld) + (uint32_t)(8 * wave) * a_ld;
  }
  const uint32_t b_lane = B_MC ? dma::load_lane_offset<true, T::BK, T::BN>(wave, n0, b_ld) + (uint32_t)(4 * wave) * b_ld
                               : dma::load_lane_offset<false, T::BK, T::BN>(wave, n0, b_ld) + (uint32_t)(8 * wave) * b_ld;
  const uint32_t b_step = B_MC ? (uint32_t)T::BK * b_ld : 128u;
  const int piece_k = 8 * ((lane & 7) ^ ((4 * (wave & 1) + (lane >> 4)) & 7));   // first k of this lane's pieces
  const int nk1 = (k + T::BK - 1) / T::BK, nk = DUAL ? 2 * nk1 : nk1;
  auto load_a = [&](int kt, uint32_t stage) {
    const bool second = DUAL && kt >= nk1;
    const int kk = second ? kt - nk1 : kt;
    const __amdgpu_buffer_rsrc_t ra = second ? ra2 : ra1;
    // pieces past the end of the reduction read as zeros (NN: rows of b past it are past the buffer)
    const uint32_t past = kk * T::BK + piece_k < k ? 0u : 0x80000000u;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t off = GATHER ? a_off[GATHER ? q : 0] : a_off[0] + (uint32_t)(32 * q) * a_ld;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (__attribute__((address_space(3))) void*)(lds + (stage + (uint32_t)(wave + 4 * q) * 1024u)), 16,
                                               (int)((off + (uint32_t)kk * 128u) | past | (GATHER ? off & 0x80000000u : 0u)), 0, 0, 0);
    }
  };
  auto load_b = [&](int kt, uint32_t stage) {
    const bool second = DUAL && kt >= nk1;
    const int kk = second ? kt - nk1 : kt;
    const __amdgpu_buffer_rsrc_t rb = second ? rb2 : rb1;
    const uint32_t past = kk * T::BK + piece_k < k ? 0u : 0x80000000u;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(kGlu && q >= 2 ? rb2 : rb, (__attribute__((address_space(3))) void*)(lds + (stage + (uint32_t)(wave + 4 * q) * 1024u)), 16,
                                               (int)((b_lane + (uint32_t)kk * b_step + (uint32_t)((B_MC ? 16 : 32) * (kGlu ? q % 2 : q)) * b_ld) | (B_MC ? 0u : past)), 0, 0, 0);
  };
  const int wm = (wave / T::WN) * T::WTM, wn = (wave % T::WN) * T::WTN;
  const uint32_t fa0 = dma::frag_lane_offset<false, T::BK, T::BM>(wm), fb0 = dma::frag_lane_offset<B_MC, T::BK, T::BN>(wn);
  u32x4 fa[2][T::TM], fb[2][T::TN];
  auto read = [&](auto si, uint32_t a_stage, uint32_t b_stage) {   // the operands of k-step si
    constexpr int s = decltype(si)::value;
    dma::static_for<T::TM>([&](auto ii) { constexpr int i = decltype(ii)::value; fa[s][i] = dma::read_frag_kc<s, i * 16 * 128>(lds_base + a_stage, fa0); });
    dma::static_for<T::TN>([&](auto ji) {
      constexpr int j = decltype(ji)::value;
      if constexpr (B_MC) {
        // the fragments of a wave are 32 bytes apart before the swizzle, which exchanges places among its eight: XOR moves from one to the next
        const uint32_t at = (lds_base + b_stage + fb0) ^ (32u * j);
        const u32x2 lo = dma::lds_read_tr16_b64<s * 32 * 128 * 2>(at), hi = dma::lds_read_tr16_b64<s * 32 * 128 * 2 + 4 * 128 * 2>(at);
        fb[s][j] = u32x4{lo[0], lo[1], hi[0], hi[1]};
      } else {
        fb[s][j] = dma::read_frag_kc<s, j * 16 * 128>(lds_base + b_stage, fb0);
      }
    });
  };
  T::Acc acc[T::TM][T::TN];
  auto multiply = [&](auto si) {
    constexpr int s = decltype(si)::value;
#pragma unroll
    for (int i = 0; i < T::TM; ++i)
#pragma unroll
      for (int j = 0; j < T::TN; ++j) acc[i][j] = mfma<DT>(fb[s][j], fa[s][i], acc[i][j]);
  };
  dma::Combine combine;
  if constexpr (EPI == dma::kEpiCombine) {
    // the assignment of tile row threadIdx.x (top_k = 1: the token itself), on its way during the main loop
    combine.out = extra;
    combine.weights = combine_weights;
    combine.w_dtype = combine_w_dtype;
    combine.tokens = combine_tokens;
    const int row = row0 + (int)threadIdx.x;
    combine.row_exists = (int)threadIdx.x < T::BM && row < end;
    combine.token = slots[combine.row_exists ? row : end - 1];
  }
  constexpr std::integral_constant<int, 0> s0{};
  constexpr std::integral_constant<int, 1> s1{};
  load_a(0, 0);
  load_b(0, kARing);
  if (nk > 1) {
    load_a(1, T::A_BYTES);
    load_b(1, kARing + T::B_BYTES);
  }
#pragma unroll
  for (int i = 0; i < T::TM; ++i)
#pragma unroll
    for (int j = 0; j < T::TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  uint32_t a_at = 0, a_to = 2 * T::A_BYTES, b_at = kARing;
  for (int kt = 0; kt < nk; ++kt) {
    __builtin_amdgcn_sched_barrier(0);
    if (kt + 1 < nk) dma::wait_vmcnt<8>(); else dma::wait_vmcnt<0>();   // K tile kt is there, kt + 1 under way
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    read(s0, a_at, b_at);
    if (kt + 2 < nk) load_a(kt + 2, a_to);   // into the stage of K tile kt - 1
    dma::wait_frags(fa[0], fb[0]);
    __builtin_amdgcn_sched_barrier(0);
    read(s1, a_at, b_at);
    multiply(s0);
    __builtin_amdgcn_sched_barrier(0);
    dma::wait_frags(fa[1], fb[1]);
    __builtin_amdgcn_s_barrier();   // every wave has the stages' operands: that of B can be refilled
    __builtin_amdgcn_sched_barrier(0);
    if (kt + 2 < nk) load_b(kt + 2, b_at);
    multiply(s1);
    a_at = a_at == 2 * T::A_BYTES ? 0 : a_at + T::A_BYTES;
    a_to = a_to == 2 * T::A_BYTES ? 0 : a_to + T::A_BYTES;
    b_at = 2 * kARing + T::B_BYTES - b_at;
  }
  uint16_t* const c_tile = dma::epi_c_optional(EPI) && c == nullptr ? nullptr : c + (int64_t)row0 * n;
  uint16_t* const e_tile = EPI != dma::kEpiNone && EPI != dma::kEpiCombine ? extra + (int64_t)row0 * n : nullptr;
  const uint16_t* const p_tile = kDglu ? a2 + (int64_t)row0 * n : nullptr;
  uint16_t* const o_tile = kDglu || kGlu ? out2 + (int64_t)row0 * n : nullptr;
  dma::block_store<DT, T, EPI>(acc, c_tile, n, 0, end - row0, n0, n, lds_generic, e_tile, p_tile, o_tile, combine);
}

template <int DT, bool B_MC, int EPI, bool GATHER, bool DUAL>
int launch(const DmaCall& q) {
  const int tiles_n = (int)ceil_div(q.n, dma::epi_is_glu(EPI) ? T::BN / 2 : T::BN);
  // an upper bound: the row counts are only known on the device
  const int64_t row_tiles = (q.rows < q.num_groups ? q.rows : q.num_groups) + q.rows / T::BM;
  const int64_t grid = ceil_div(row_tiles * tiles_n, kXcds) * kXcds;
  if (grid > 0x7fffffff) return MBX_ERANGE;
  auto kern = gmm_pair_kernel<DT, B_MC, EPI, GATHER, DUAL>;
  const int rc = allow_lds(kern, kLdsBytes);
  if (rc) return rc;
  const int32_t* const slots = EPI == dma::kEpiCombine ? q.combine.indices : q.gather.slots;
  kern<<<(unsigned)grid, T::THREADS, kLdsBytes, q.stream>>>(
      (const uint16_t*)q.a, (const uint16_t*)q.b, (uint16_t*)q.c, q.bins, q.num_groups, (int)q.rows, q.k, q.n, tiles_n,
      (const uint16_t*)q.a2, (const uint16_t*)q.b2, (uint16_t*)q.extra, (uint16_t*)q.out2, slots, q.gather.src_bins,
      q.gather.top_k, q.gather.src_rows, q.combine.weights, q.combine.w_dtype, q.combine.tokens);
  return launch_status();
}

template <int DT>
int dispatch(const DmaCall& q) {
  const bool dual = q.a2 && !dma::epi_is_dglu(q.epi);   // else: x2 of the gate's gradient
  if (q.layout == MBX_NN) {
    if (dual) return launch<DT, true, dma::kEpiNone, false, true>(q);
    if (q.epi == dma::kEpiCombine) return launch<DT, true, dma::kEpiCombine, false, false>(q);
    if (q.epi == dma::kEpiAct) return launch<DT, true, dma::kEpiAct, false, false>(q);
    return launch<DT, true, dma::kEpiNone, false, false>(q);
  }
  if (dual) return launch<DT, false, dma::kEpiNone, false, true>(q);
  switch (q.epi) {
    case dma::kEpiNone: return q.gather.slots ? launch<DT, false, dma::kEpiNone, true, false>(q) : launch<DT, false, dma::kEpiNone, false, false>(q);
    case dma::kEpiAct: return q.gather.slots ? launch<DT, false, dma::kEpiAct, true, false>(q) : launch<DT, false, dma::kEpiAct, false, false>(q);
    case dma::kEpiGluSilu: return q.gather.slots ? launch<DT, false, dma::kEpiGluSilu, true, false>(q) : launch<DT, false, dma::kEpiGluSilu, false, false>(q);
    case dma::kEpiGluGelu: return q.gather.slots ? launch<DT, false, dma::kEpiGluGelu, true, false>(q) : launch<DT, false, dma::kEpiGluGelu, false, false>(q);
    case dma::kEpiDact: return launch<DT, false, dma::kEpiDact, false, false>(q);
    case dma::kEpiDgluSilu: return launch<DT, false, dma::kEpiDgluSilu, false, false>(q);
    default: return launch<DT, false, dma::kEpiDgluGelu, false, false>(q);
  }
}

}  // namespace pair
}  // namespace

// Gathered rows: whole K tiles.
bool gmm_pair_can(const DmaCall& q) { return q.layout != MBX_TN && !(q.gather.slots && q.k % pair::T::BK); }

// By which part the launch has to be estimated shorter here than with gmm_dma.h's tiles (0: never here), a sixteenth in general.  `rounds`: of
// tiles, here.  What the estimates leave out, from 5300 launches (2 - 4000 experts of 4 - 12000 rows on average, even or popular as r^-0.6 or r^-1.2, [64 - 4096,
// 64 - 12000], plain, two pairs and every epilogue but the combine; time here / gmm_dma.h's on the geometric mean):
//   * up to eight rounds the sixteenth holds, whatever the number of experts (above 64: 0.88, the activation's gradient 0.83).  The gain is the last
//     round and what overlaps across it.  Beyond, most launches are longer here (1.06; 8 experts of 13700, [128, 4328], with the gate: 1262 / 1824 us;
//     activation, 16 of 17200, [128, 2960]: 886 / 1109), but not those of up to kHalfHeightRows rows (0.91 to 24 rounds) and the activation's
//     gradient (0.95) that an eighth is expected from, nor where gmm_dma.h's tile is mostly padding (0.74);
//   * the gate's three outputs are not in the estimates: four rounds (two to four 0.93, four to eight 0.99, then 1.12); and of up to kHalfHeightRows rows,
//     where the half-height tiles are quicker than estimated (16 experts of 100, [4096, 1024]: 58 / 66 us), only what is shorter by a fifth;
//   * cutting products of kLongCutTiles K tiles and more gains gmm_dma.h's kernel more than estimated (1.09; 8 of 2037, [9536, 240]: 109 / 146 us; 4 of 1700,
//     [10880, 752]: 126 / 169), except where its tile is mostly padding (36 of 825, [7768, 64]: 218 / 144);
//   * every workgroup looks its expert up anew: with more than kManyExperts four rounds (0.63, beyond 1.06).
// As chosen, 1400 other launches of 2 - 256 experts are 11 % shorter than gmm_dma.h's (up to 64 experts 17 %, above 3 %); 2.6 % of them are by more than 3 %
// longer, none by more than 18 %.
constexpr double kFewRounds = 8, kLowRounds = 24, kMostRounds = 32, kGluRounds = 4, kManyRounds = 4, kManyExperts = 1024, kLongCutTiles = 96;

static double gain_line(const DmaCall& q, bool may_cut, double nk, double average, double rounds) {
  const bool glu = dma::epi_is_glu(q.epi), low = average <= kHalfHeightRows;
  if (rounds > kMostRounds || (glu && rounds > kGluRounds) || (q.num_groups > kManyExperts && rounds > kManyRounds)) return 0;
  if (may_cut && nk >= kLongCutTiles) return 0.55;
  if (glu && low) return 0.8;
  if (rounds <= kFewRounds) return 0.94;
  return q.epi == dma::kEpiDact || (low && rounds <= kLowRounds) ? 0.88 : 0.7;
}

// Whether the launch is estimated to be shorter here than with gmm_dma.h's tiles by enough (gain_line).  Both estimates are
// rounds of tiles times K tiles times what one takes, us, fitted to 206 NT and 206 NN launches (4 - 64 experts of 48 - 800 rows,
// [512 - 2048, 1408 - 4096], operands out of memory; rms 11 - 12 %), and no less than the operands at the rate the kernel reads them.
// gmm_dma.h's kernel / this one: NT 4 experts of 500, [1408, 2048]: 42 / 23; 8 of 300, [4096, 2048]: 66 / 58; 64 of 48, [4096, 2048]: 247 /
// 189; 12 of 500, [2728, 1032]: 62 / 65; 16 of 500, [4096, 2048]: 136 / 151.  NN 8 of 500, [1408, 512]: 32 / 16; 16 of 300, [1408, 2048]: 56 /
// 41; 8 of 300, [4096, 1024], cut: 49 / 41; 4 of 100: 30 / 40; 32 of 500, [3072, 768]: 79 / 110.
bool gmm_pair_takes(const DmaCall& q) {
  if (!gmm_pair_can(q)) return false;
  const bool nn = q.layout == MBX_NN, dual = q.a2 && !dma::epi_is_dglu(q.epi), glu = dma::epi_is_glu(q.epi);
  const double units = persistent_grid((int64_t)1 << 30), experts = q.num_groups, average = (double)q.rows / experts;
  const double nk = (dual ? 2.0 : 1.0) * (double)ceil_div(q.k, pair::T::BK), n = q.n * (glu ? 2.0 : 1.0);
  const double mb = ((experts * q.k * n + (double)q.rows * q.k) * (dual ? 2 : 1) + (double)q.rows * n) * 2e-6;
  auto row_tiles = [&](double height) { return experts * (average > 64 ? average / height + 0.5 : 1.0); };   // the row counts vary
  // here: a round is two tiles to a compute unit, which one by itself works off in little more than half the time
  const double tiles = row_tiles(128) * ceil(n / 128), rounds = floor(tiles / (2 * units)), rest = tiles / (2 * units) - rounds;
  // gmm_dma.h's kernel cuts the combine's tails as the plain product's (120 combines, 4 - 128 experts of 17 - 1500 rows, mostly where it matters, over the
  // shorter of the two: judged as cut 1.04, as never cut 1.13; 4 of 104, [13120, 512]: 58 us there, 130 here)
  const bool may_cut = nn && (q.epi == dma::kEpiNone || q.epi == dma::kEpiCombine) && q.ws.base;
  const double line = gain_line(q, may_cut, nk, average, tiles / (2 * units));
  double here = 4.8 + rounds * nk * 1.2;
  if (rest > 0) here += nk * (rest <= 0.5 ? 0.56 : 0.56 + 0.64 * (2 * rest - 1));
  here = fmax(here, 4.8 + mb / 5.5);
  // there: gmm_rows.h's choice of the half-height tile, and the cut of a last round that is at most half full
  const bool half = average <= kHalfHeightRows || (average <= kMixedRows && row_tiles(256) * ceil(n / 256) < kMixedRounds * units);
  const double tile = nk * (nn ? (half ? 1.03 : 1.57) : (half ? 0.9 : 1.4)) + (nn ? 0 : 5);
  const double all = row_tiles(half ? 128 : 256) * ceil(n / 256), full = floor(all / units), left = all - full * units;
  double there = (nn ? 1.3 : 0.5) + full * tile;
  if (left > 0) {
    const double parts = fmin(fmin((double)kMaxKSplit, floor(units / left)), floor(nk / kMinPartTiles));
    // half-height tiles only: estimated as if always cut, which is what the lines above were drawn on; two short parts are left whole since and gain 2 - 3 %
    // (64 experts of 227, [1216, 1344]: 94 there, 77 here)
    const bool cut = may_cut && 2 * left <= units && (full > 0 || nk >= kMinCutTiles) && (half ? parts >= 2 : cut_pays(false, (int)full, (int)parts, (int)nk));
    there += cut ? tile / parts + 21 : 2 * left <= units && full > 0 && !half ? 0.75 * tile : tile;
  }
  there = fmax(there, (nn ? 1.3 : 0.5) + mb / (nn ? 5.4 : 4.6));
  return here < line * there;
}

int gmm_pair(const DmaCall& q) { return q.dtype == MBX_BF16 ? pair::dispatch<MBX_BF16>(q) : pair::dispatch<MBX_F16>(q); }

}  // namespace mbx
