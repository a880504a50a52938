// NN / NT products of 16-bit operands where an expert has a handful of rows: decoding, short prompts, small batches
// over many experts.
//
// What bounds them: the reading of the weights, once.  A row of the output costs no arithmetic to speak of (a matrix
// instruction multiplies 16 rows whether they exist or not), so the tiles of gmm_dma.h, 256 columns by one workgroup per
// compute unit, only make the launch coarse: 26 experts with a [2816, 2048] first product are 286 tiles on 256 compute
// units, and their second product, 8 tiles of 22 K tiles each, is a chain of memory latencies on two thirds of the chip.
//
// Here a workgroup of four waves takes 64 output columns of one expert and 16 of its rows, and each wave a quarter of the
// reduction in chunks of 64.  The weights go from memory to registers as the matrix instruction wants them and are used
// once; no wave waits for another until the end, where the four partial sums meet in LDS (added in wave order: results do
// not depend on timing).  Two chunks per wave are in flight, and four workgroups share a compute unit: 256 KiB of weights
// under way.  (Eight waves per workgroup: 2 - 12 % slower where the reduction is short, no faster elsewhere.  Workgroups
// that walk a list of units with the next unit's loads under way: the registers for two units' addresses spill, 82
// against 71 us on 64 experts of 4 rows, [1408, 2048].  32 or 64 rows at a time: the registers of one workgroup leave
// too few loads in flight, 3.8 against 5.0 TB/s.)
//
// Measured (bf16, TB/s of the weights of the experts that got rows, gmm_dma.h's kernel / this one; a plain read reaches 5.8):
//   8 experts x 4 rows, [14336, 4096]: gated first products 4.8 - 5.4 (by placement) / 5.6, second product 5.17 / 5.52
//   64 x 4, [1408, 2048]: 5.21 / 5.32, 5.58 / 5.59;  25 of 64 experts with a row or two: 3.88 / 4.73, 4.66 / 4.76
//   64 x 4, [3840, 1024]: 5.29 / 5.37, 5.62 / 5.66;  6 of 64 experts: 4.19 / 5.07, 1.52 / 3.75
//   32 x 4, [2816, 3072]: 5.33 / 4.80, 4.85 / 5.12;  3 of 32 experts: 2.34 / 3.51, 1.66 / 4.29
//   16 x 4, [1408, 1024]: 4.32 / 3.91, 1.98 / 3.78
//
//   NT ([n][k] weights): lane (c = l % 16, g = l / 16) reads 32 contiguous bytes of row c of a 16-row fragment, two 16-byte
//   loads; 16 lines of 128 bytes per pair of loads.
//   NN ([k][n] weights): lane (c, g) reads four columns (8 bytes) of eight rows k, whole 128-byte lines again, and swaps
//   the 8 x 4 values into k order with byte permutes (32 of them per 8 KiB).
// In a chunk, lane group g holds k = 16 g + 8 s .. + 7 for instruction s, in both operands.
#include "gmm_common.h"

#include <cmath>
#include <type_traits>

namespace mbx {
namespace {

#include "gmm_dma.h"   // buffer descriptors, tile list, activations

namespace few {

using dma::clip_bytes;
using dma::make_rsrc;

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));

constexpr int kWaves = 4, kThreads = kWaves * kWave, kRows = 16, kCols = 64, kChunk = 64;
constexpr int kPitch = kCols + 4;                                   // floats per row of a partial sum in LDS
constexpr uint32_t kNone = 0x80000000u;   // an offset past every buffer: the load brings zeros

template <int DT>
__device__ __forceinline__ f32x4 mfma(const u32x4& a, const u32x4& b, const f32x4& c) {
  if (DT == MBX_BF16) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}

// One chunk's operands of a lane.
template <bool B_MC> struct Chunk;
template <> struct Chunk<false> { u32x4 a[2], b[2][4]; };
template <> struct Chunk<true> { u32x4 a[2]; u32x2 b[2][8]; };

// EPI: dma::kEpiNone, kEpiAct, kEpiGlu*, kEpiDact, kEpiDglu* (NT), kEpiCombine (NN).  GATHER (NT): as in gmm_dma.h's gmm_rows_kernel.
// c (with the gate: and out2) may be null where only the epilogue's output is wanted.  a2: x2 of kEpiDglu*.
template <int DT, bool B_MC, int EPI, bool GATHER>
__global__ void __launch_bounds__(kThreads, 4)
gmm_few_kernel(const uint16_t* __restrict__ a, const uint16_t* __restrict__ b, uint16_t* __restrict__ c,
               const int32_t* __restrict__ bins, int num_groups, int rows, int k, int n, int tiles_n,
               const uint16_t* __restrict__ a2, const uint16_t* __restrict__ b2, uint16_t* __restrict__ extra, uint16_t* __restrict__ out2,
               const int32_t* __restrict__ slots, const int32_t* __restrict__ src_bins, int top_k, int src_rows,
               const void* __restrict__ combine_weights, int combine_w_dtype, int combine_tokens) {
  __shared__ __attribute__((aligned(16))) float sums[kWaves * kRows * kPitch];
  constexpr bool kGlu = dma::epi_is_glu(EPI), kDglu = dma::epi_is_dglu(EPI);
  constexpr int kTileCols = kGlu ? kCols / 2 : kCols;
  const dma::RowTiles<kRows> tiles(bins, num_groups, tiles_n, rows, false, 8);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = lane_id(), col = lane & 15, g = lane >> 4;
  const uint32_t pitch = (uint32_t)k * 2u;
  const int chunks = (k + kChunk - 1) / kChunk;
  const int steps = (chunks + 2 * kWaves - 1) / (2 * kWaves) * 2;   // chunks per wave, an even number; those past the last chunk are not fetched

  struct Unit { int e, start, row0, end, n0; };
  auto locate = [&](int id) {
    Unit u;
    int tm, tn;
    tiles.find(id, u.e, u.start, u.end, tm, tn);
    const int mt = (u.end - u.start + kRows - 1) / kRows;
    if (mt > 1) {
      // Eight column tiles, then the same eight with the expert's next rows: those workgroups follow on the same XCDs and find
      // the weights in their L2s.
      const int t = tn * mt + tm, first = t / (8 * mt) * 8, in = t - first * mt, wide = tiles_n - first < 8 ? tiles_n - first : 8;
      tm = in / wide;
      tn = first + in % wide;
    }
    u.row0 = u.start + tm * kRows;
    u.n0 = tn * kTileCols;
    return u;
  };
  auto slot_of = [&](const Unit& u) -> int {   // GATHER: the assignment of this lane's row
    const int src_start = u.e > 0 ? src_bins[u.e - 1] : 0;
    const int64_t slots_end = (int64_t)src_rows * top_k;
    const int limit = (int)(src_bins[u.e] < slots_end ? src_bins[u.e] : slots_end);
    const int j = (src_start < 0 ? 0 : src_start) + (u.row0 - u.start) + col;
    return u.row0 + col < u.end && j < limit ? slots[j] : -1;
  };
  // where the loads issued now read from
  __amdgpu_buffer_rsrc_t rsrc_a = make_rsrc(a, GATHER ? clip_bytes((int64_t)src_rows * k * 2) : 0u), rsrc_b = rsrc_a, rsrc_b2 = rsrc_a;
  uint32_t a_off = kNone, b_off = 0;
  auto aim = [&](const Unit& u, int slot) {
    if constexpr (GATHER) {
      const int row = slot >= 0 ? slot / top_k : src_rows;
      a_off = row < src_rows ? (uint32_t)row * pitch + (uint32_t)g * 32u : kNone;
    } else {
      rsrc_a = make_rsrc(a + (int64_t)u.row0 * k, clip_bytes((int64_t)(u.end - u.row0) * k * 2));
      a_off = u.row0 + col < u.end ? (uint32_t)col * pitch + (uint32_t)g * 32u : kNone;
    }
    rsrc_b = make_rsrc(b + (int64_t)u.e * k * n, (uint32_t)((int64_t)k * n * 2));
    rsrc_b2 = kGlu ? make_rsrc(b2 + (int64_t)u.e * k * n, (uint32_t)((int64_t)k * n * 2)) : rsrc_b;
    b_off = B_MC ? (uint32_t)(16 * g) * (uint32_t)n * 2u + (uint32_t)(u.n0 + col * 4) * 2u : (uint32_t)(u.n0 + col) * pitch + (uint32_t)g * 32u;
  };
  // A wave's chunks are a quarter of the reduction, and the columns start at different places in it and go round: started
  // together at its beginning, the workgroups would all read the first bytes of rows that are a power of two apart, and
  // which memory channels those fall on is a matter of where the weights lie (the same launch took 341 to 456 us on
  // different copies of the same weights; now 335 to 336).
  int turn = 0;
  auto fetch = [&](Chunk<B_MC>& x, int step) {
    const int at = step + turn < steps ? step + turn : step + turn - steps;
    const int ch = wave * steps + at;
    const uint32_t byte0 = (uint32_t)ch * (kChunk * 2), none = step < steps && ch < chunks ? 0u : kNone;
    uint32_t b_at = B_MC ? (b_off + (uint32_t)ch * kChunk * (uint32_t)n * 2u) | none : b_off + byte0;
    asm volatile("" : "+v"(b_at));   // the loads' addresses are sums with scalars, not sixteen registers carried through the loop
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      // pieces past the end of the reduction read as zeros (k is a multiple of 8); NN: rows past k are past the buffer
      const uint32_t past = ch * kChunk + 16 * g + 8 * s < k ? none : kNone;
      x.a[s] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc_a, (int)((a_off + byte0 + 16u * s) | past | (a_off & kNone)), 0, 0));
      if constexpr (B_MC) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
          x.b[s][i] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rsrc_b, (int)(b_at + (8u * s + i) * (uint32_t)n * 2u), 0, 0));
      } else {
#pragma unroll
        for (int f = 0; f < 4; ++f) {
          const uint32_t rows_on = kGlu ? (uint32_t)(f & 1) * 16u : (uint32_t)f * 16u;
          x.b[s][f] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(kGlu && f >= 2 ? rsrc_b2 : rsrc_b, (int)((b_at + rows_on * pitch + 16u * s) | past), 0, 0));
        }
      }
    }
  };
  f32x4 acc[4];
  auto multiply = [&](const Chunk<B_MC>& x) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        u32x4 bf;
        if constexpr (B_MC) {   // fragment f: columns 4 (lane % 16) + f
          const uint32_t sel = f & 1 ? 0x07060302u : 0x05040100u;
#pragma unroll
          for (int w = 0; w < 4; ++w) bf[w] = __builtin_amdgcn_perm(x.b[s][2 * w + 1][f >> 1], x.b[s][2 * w][f >> 1], sel);
        } else {
          bf = x.b[s][f];
        }
        acc[f] = mfma<DT>(bf, x.a[s], acc[f]);
      }
  };
  // eight columns of a row of the finished unit
  auto total = [&](int m, int ch8, float (&f)[8]) {
#pragma unroll
    for (int t = 0; t < 8; ++t) f[t] = 0.f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const f32x4* p = (const f32x4*)(sums + (size_t)(w * kRows + m) * kPitch + ch8 * 8);
      const f32x4 lo = p[0], hi = p[1];
#pragma unroll
      for (int t = 0; t < 4; ++t) { f[t] += lo[t]; f[4 + t] += hi[t]; }
    }
  };

  if ((int)blockIdx.x >= tiles.total) return;
  const Unit cur = locate(blockIdx.x);
  aim(cur, GATHER ? slot_of(cur) : 0);
  turn = (int)(((uint32_t)(cur.n0 / kCols) * 5u + (uint32_t)cur.e * 3u) % (uint32_t)steps);
  Chunk<B_MC> x0, x1;
  fetch(x0, 0);
#pragma unroll
  for (int f = 0; f < 4; ++f) acc[f] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int step = 0; step < steps; step += 2) {
    fetch(x1, step + 1);
    __builtin_amdgcn_sched_barrier(0);   // a chunk's loads are all issued before the products of the one before it
    multiply(x0);
    __builtin_amdgcn_sched_barrier(0);
    fetch(x0, step + 2);
    __builtin_amdgcn_sched_barrier(0);
    multiply(x1);
    __builtin_amdgcn_sched_barrier(0);
  }
  constexpr int kItems = kTileCols / 8;
  const int m = threadIdx.x / kItems, ch8 = threadIdx.x % kItems, row = cur.row0 + m, cn = cur.n0 + ch8 * 8;
  const bool mine = m < kRows && row < cur.end && cn < n;   // n is a multiple of 8
  const int64_t at = (int64_t)row * n + cn;
  u32x4 in1 = {0u, 0u, 0u, 0u}, in2 = in1;   // the epilogue's inputs, under way while the sums meet
  if constexpr (EPI == dma::kEpiDact || kDglu)
    if (mine) in1 = *(const u32x4*)(extra + at);
  if constexpr (kDglu)
    if (mine) in2 = *(const u32x4*)(a2 + at);
  // partial sums: sums[wave][row][column]
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    // NT: fragment q, columns 16 q + 4 g + r.  NN: register q of the four fragments, columns 4 (4 g + q) + f.
    f32x4 v;
    if constexpr (B_MC) {
#pragma unroll
      for (int f = 0; f < 4; ++f) v[f] = acc[f][q];
    } else {
      v = acc[q];
    }
    *(f32x4*)(sums + (size_t)(wave * kRows + col) * kPitch + (B_MC ? 16 * g + 4 * q : 16 * q + 4 * g)) = v;
  }
  __syncthreads();
  if (!mine) return;
  float f[8];
  total(m, ch8, f);
  const u32x4 v = dma::pack8<DT>(f);
  if constexpr (kGlu) {
    total(m, ch8 + kItems, f);
    const u32x4 v2 = dma::pack8<DT>(f);
    if (c != nullptr) {
      *(u32x4*)(c + at) = v;
      *(u32x4*)(out2 + at) = v2;
    }
    *(u32x4*)(extra + at) = dma::glu_chunk<DT, EPI == dma::kEpiGluGelu>(v, v2);
  } else if constexpr (kDglu) {
    u32x4 d1, d2;
    dma::dglu_chunk<DT, EPI == dma::kEpiDgluGelu>(v, in1, in2, d1, d2);
    *(u32x4*)(c + at) = d1;
    *(u32x4*)(out2 + at) = d2;
  } else if constexpr (EPI == dma::kEpiDact) {
    *(u32x4*)(c + at) = dma::gelu_bwd_chunk<DT>(v, in1);
  } else {
    if (c != nullptr) *(u32x4*)(c + at) = v;
    if constexpr (EPI == dma::kEpiAct) *(u32x4*)(extra + at) = dma::gelu_fwd_chunk<DT>(v);
    if constexpr (EPI == dma::kEpiCombine) {
      dma::Combine cb;
      cb.weights = combine_weights;
      cb.w_dtype = combine_w_dtype;
      cb.tokens = combine_tokens;
      cb.token = slots[row];
      cb.row_exists = true;
      const int token = dma::combine_token(cb);
      if (token >= 0) *(u32x4*)(extra + (int64_t)token * n + cn) = dma::scale_chunk<DT>(v, dma::combine_weight(cb, token));
    }
  }
}

}  // namespace few

template <int DT, bool B_MC, int EPI, bool GATHER>
int launch_few(const DmaCall& q, const int32_t* slots) {
  const int cols = dma::epi_is_glu(EPI) ? few::kCols / 2 : few::kCols;
  const int tiles_n = (int)ceil_div(q.n, cols);
  // an upper bound: the row counts are only known on the device
  const int64_t row_tiles = (q.rows < q.num_groups ? q.rows : q.num_groups) + q.rows / few::kRows;
  if (row_tiles * tiles_n > 0x7fffffff) return MBX_ERANGE;
  few::gmm_few_kernel<DT, B_MC, EPI, GATHER><<<(unsigned)(row_tiles * tiles_n), few::kThreads, 0, q.stream>>>(
      (const uint16_t*)q.a, (const uint16_t*)q.b, (uint16_t*)q.c, q.bins, q.num_groups, (int)q.rows, q.k, q.n, tiles_n,
      (const uint16_t*)q.a2, (const uint16_t*)q.b2, (uint16_t*)q.extra, (uint16_t*)q.out2, slots, q.gather.src_bins, q.gather.top_k, q.gather.src_rows,
      q.combine.weights, q.combine.w_dtype, q.combine.tokens);
  return launch_status();
}

template <int DT>
int dispatch_few(const DmaCall& q) {
  if (q.layout == MBX_NN) {
    if (q.epi == dma::kEpiCombine) return launch_few<DT, true, dma::kEpiCombine, false>(q, q.combine.indices);
    if (q.epi == dma::kEpiAct) return launch_few<DT, true, dma::kEpiAct, false>(q, nullptr);
    return launch_few<DT, true, dma::kEpiNone, false>(q, nullptr);
  }
#define MBX_FEW_NT(EPI) (q.gather.slots ? launch_few<DT, false, EPI, true>(q, q.gather.slots) : launch_few<DT, false, EPI, false>(q, nullptr))
  switch (q.epi) {
    case dma::kEpiNone: return MBX_FEW_NT(dma::kEpiNone);
    case dma::kEpiAct: return MBX_FEW_NT(dma::kEpiAct);
    case dma::kEpiGluSilu: return MBX_FEW_NT(dma::kEpiGluSilu);
    case dma::kEpiGluGelu: return MBX_FEW_NT(dma::kEpiGluGelu);
    case dma::kEpiDact: return launch_few<DT, false, dma::kEpiDact, false>(q, nullptr);
    case dma::kEpiDgluSilu: return launch_few<DT, false, dma::kEpiDgluSilu, false>(q, nullptr);
    default: return launch_few<DT, false, dma::kEpiDgluGelu, false>(q, nullptr);
  }
#undef MBX_FEW_NT
}

}  // namespace

// Up to eight rows per expert on average (beyond, experts of more than 16 rows read their weights twice: 16 rows per expert
// cost 20 - 40 %).
// NN: wherever gmm_dma.h's tiles would leave the chip partly idle; with reductions of 3072 and more only up to half a round of
// them: there that kernel cuts its tiles along the reduction, and here a workgroup runs so long that a compute unit with one
// more than the others ends late (8 experts of [14336, 4096], two to a compute unit, 174 us, 9 experts 235).  (us, that
// kernel / this one, two rows per expert: [14336, 4096] 8 experts 178 / 173, 9: 185 / 231, 12: 227 / 258;  [8192, 4096] 8: 104 /
// 115, 12: 134 / 172, 28: 311 / 400;  [4096, 2048] 16: 45 / 43, 24: 71 / 78;  [2816, 3072] 16: 46 / 44, 32: 112 / 103).
// NT: that kernel keeps up as long as its rounds of tiles are about three quarters full (32 experts, [2816, 3072]: 195 against
// 216 us with 0.86 of them full, 124 against 134 with 0.77; 25 of 64 experts, [1408, 2048]: 74 against 61 with 0.54), with
// short reductions, sixteen chunks of which are four per wave here, longer still (16 experts, [1408, 1024]: 21 against 24 us
// with 0.69), and with long ones it depends on where the weights lie (8 experts, [14336, 4096]: 347 - 398 against 335 us).
// From four rows per expert on gmm_mid.hip's launches are its own: as fast with even rows, faster with skewed ones (us, this
// kernel / that one, gated and plain, 8 rows on average, even, Zipf-distributed (exponent 1.2) and all on top_k experts: 8 experts
// top-2, [14336, 4096]: 352, 173 / 343, 158;  376, 187 / 344, 158;  158, 81 / 94, 63;  64 top-6, [1408, 4096]: 282, 147 / 264,
// 129;  303, 159 / 254, 122;  141, 85 / 68, 64).
// Skewed rows where the launch stays here, against gmm_dma.h (Zipf and all on top_k, 8 rows): NN, 8 experts, [14336, 4096]: 192
// / 215, 52 / 52;  16 top-4, [4096, 2048]: 47 / 53, 26 / 16;  32 top-2, [2816, 1024]: 34 / 35, 25 / 12;  NT gated, 16 top-2,
// [4096, 4096]: 214 / 216, 58 / 79 (even: 227 / 203).
// The number of experts that get rows is an expectation: rows that choose evenly.  The epilogues do not enter the rule: the
// product of a launch with one is the plain launch's, bit for bit.
bool gmm_few_takes(const DmaCall& q) {
  const bool nn = q.layout == MBX_NN, nt = q.layout == MBX_NT;
  if (!(nn || nt) || (q.a2 && !dma::epi_is_dglu(q.epi)) || q.rows > 8 * (int64_t)q.num_groups) return false;
  if (nt && q.rows > 4 * (int64_t)q.num_groups && gmm_mid_takes(q)) return false;
  const double experts = q.num_groups * (1.0 - pow(1.0 - 1.0 / q.num_groups, (double)q.rows));
  const double rounds = experts * (double)ceil_div(q.n, nn ? 256 : 128) / persistent_grid((int64_t)1 << 30);
  const double filled = rounds / ceil(rounds);
  if (nn && q.k >= 3072) return rounds <= 0.5;
  return nn ? filled < 0.92 : q.k >= 4096 || filled < (q.k >= 2048 ? 0.7 : 0.5);
}

int gmm_few(const DmaCall& q) { return q.dtype == MBX_BF16 ? dispatch_few<MBX_BF16>(q) : dispatch_few<MBX_F16>(q); }

}  // namespace mbx
