// Launch of the NN / NT kernels of gmm_dma.h, instantiated for whole K tiles by gmm_rows.hip and for reductions that end
// inside one by gmm_rows_tail.hip.
#pragma once

#include "gmm_common.h"

#include <cstdlib>

namespace mbx {
namespace {

#include "gmm_dma.h"

// NN / NT: whether to tile a launch with the half-height tile only.  With about one such tile per expert
// (up to kHalfHeightRows rows on average) the full tile would mostly multiply padding.  Up to kMixedRows the mix of
// full tiles and a half-height last tile moves fewer weight bytes through the compute units (the
// weights are streamed once per row tile), but its tiles cost unequal time, and a launch of fewer than
// kMixedRounds rounds of them does not balance over the statically assigned workgroups.
static inline bool half_height_only(int64_t rows, int num_groups, int n) {
  const int64_t avg = rows / (num_groups > 0 ? num_groups : 1);
  if (avg <= kHalfHeightRows) return true;
  if (avg > kMixedRows) return false;
  const int64_t mixed_tiles = (ceil_div(rows, dma::TileMain::BM) + num_groups / 2) * ceil_div(n, dma::TileMain::BN);
  return mixed_tiles < kMixedRounds * (int64_t)persistent_grid((int64_t)1 << 30);
}

// TS is the tile the tail of a launch is cut into (TS = T: never cut).
template <int DT, typename T, typename TS, bool KTAIL>
int launch_rows(const DmaCall& call) {
  const int32_t* const bins = call.bins;
  const int num_groups = call.num_groups, k = call.k, n = call.n, layout = call.layout;
  const int64_t rows = call.rows;
  const hipStream_t s = call.stream;
  const int epi = call.epi;
  const uint16_t *ap = (const uint16_t*)call.a, *bp = (const uint16_t*)call.b, *ap2 = (const uint16_t*)call.a2, *bp2 = (const uint16_t*)call.b2;
  const void *a2 = call.a2, *b2 = call.b2;
  uint16_t* cp = (uint16_t*)call.c;
  void *const extra = call.extra, *const out2 = call.out2;
  const GatherRows& gather = call.gather;
  const CombineRows& combine = call.combine;
  const Workspace& ws = call.ws;
  const bool dual = a2 != nullptr && !dma::epi_is_dglu(epi) && !dma::epi_is_glu(epi);
  constexpr size_t lds = T::LDS_BYTES > TS::LDS_BYTES ? T::LDS_BYTES : TS::LDS_BYTES;
  // a [w1 | v1] tile covers half as many output columns
  const int tiles_n = (int)ceil_div(n, dma::epi_is_glu(epi) ? T::BN / 2 : T::BN);
  const int64_t tiles = (ceil_div(rows, T::BM) + num_groups) * tiles_n;   // the row counts are only known on the device
  if (tiles > 0x7fffffff) return MBX_ERANGE;
  // launches that may cut their tiles along the reduction want the compute units that have no tile for the parts
  const bool may_cut = layout == MBX_NN && (epi == dma::kEpiNone || epi == dma::kEpiCombine) && ws.base != nullptr && (dual ? 2 : 1) * ceil_div(k, T::BK) >= kMinCutTiles;
  const unsigned grid = (unsigned)persistent_grid(may_cut ? (int64_t)1 << 30 : tiles);
  // An expert's last row tile, when at most half full, is computed with the half-height tile -- unless a row of tiles is
  // longer than the run of tiles an XCD's workgroups take per round: the half-height tiles of such a row fill whole
  // rounds of some XCDs, those finish early, and from then on the XCD's workgroups are no longer within the few K tiles
  // of each other that the L2 holds (c3's NT launches, 112 and 56 column tiles against runs of 32: L2 misses 5.8 ->
  // 3.3 GB; the launches themselves take 1 % longer for the padding they multiply, the step is 0.7 % shorter, the
  // launches after them running at a higher clock).  With shorter rows of tiles the half-height tile wins (every
  // launch of c2, c4 and c5: 0.7 - 2.8 % per step), and with few row tiles per expert the padding would be a large
  // part of the work.  MBX_FULL_SHORT_FROM=N overrides the column-tile count from which
  // the full tile is used (measurements).
  static const int full_short_from = [] { const char* v = getenv("MBX_FULL_SHORT_FROM"); return v ? atoi(v) : -1; }();
  const int run_tiles = (int)grid / kXcds;
  // ... and only for experts of eight row tiles and more on average, where the padding is a few percent of the work
  const bool long_experts = rows >= (int64_t)num_groups * 8 * T::BM;
  const int half_limit = (full_short_from >= 0 ? tiles_n >= full_short_from : tiles_n > run_tiles && long_experts) ? 0 : TS::BM;
  uint32_t gather_magic = 0;
  int gather_shift = 0;
  if (!KTAIL && gather.slots) dma::gather_divisor(gather.top_k, gather_magic, gather_shift);
  const WorkspaceParts lent(ws, (size_t)T::BM * T::BN * sizeof(float));
  int32_t* const ws_counters = lent.counters;
  float* const ws_parts = (int)grid / 2 <= (int)kWorkspaceCounters ? lent.parts : nullptr;
  const int ws_capacity = lent.capacity;
#define MBX_LAUNCH_ROWS_G(B_MC, DUAL, EPI, GATHER)                                                    \
  do {                                                                                                \
    auto kern = dma::gmm_rows_kernel<DT, B_MC, T, TS, DUAL, EPI, GATHER, KTAIL>;                             \
    int rc = allow_lds(kern, lds);                                                                    \
    if (rc) return rc;                                                                                \
    kern<<<grid, T::THREADS, lds, s>>>(ap, bp, cp, bins, num_groups, rows, k, n, tiles_n, ap2, bp2, (uint16_t*)extra, (uint16_t*)out2,  \
                                       gather.slots, gather.src_bins, gather.top_k, gather.src_rows, gather_magic, gather_shift, half_limit,  \
                                       ws_counters, ws_parts, ws_capacity, combine.weights, combine.w_dtype, combine.tokens);  \
  } while (0)
#define MBX_LAUNCH_ROWS(B_MC, DUAL, EPI) MBX_LAUNCH_ROWS_G(B_MC, DUAL, EPI, false)
  // the combine epilogue takes the sorted assignments where the gathered launches take theirs
#define MBX_LAUNCH_ROWS_C(B_MC, DUAL, EPI)                                                            \
  do {                                                                                                \
    auto kern = dma::gmm_rows_kernel<DT, B_MC, T, TS, DUAL, EPI, false, KTAIL>;                              \
    int rc = allow_lds(kern, lds);                                                                    \
    if (rc) return rc;                                                                                \
    kern<<<grid, T::THREADS, lds, s>>>(ap, bp, cp, bins, num_groups, rows, k, n, tiles_n, ap2, bp2, (uint16_t*)extra, (uint16_t*)out2,  \
                                       combine.indices, nullptr, 1, 0, 0u, 0, half_limit, ws_counters, ws_parts, ws_capacity, \
                                       combine.weights, combine.w_dtype, combine.tokens);             \
  } while (0)
  if constexpr (KTAIL) {
    if (gather.slots) return MBX_EUNSUPPORTED;   // gathered rows: whole K tiles
  } else if (gather.slots) {
    if (layout != MBX_NT || a2 || !gather.src_bins || gather.top_k <= 0) return MBX_EINVAL;
    switch (epi) {
      case dma::kEpiNone: MBX_LAUNCH_ROWS_G(false, false, dma::kEpiNone, true); break;
      case dma::kEpiAct: if (!extra) return MBX_EINVAL; MBX_LAUNCH_ROWS_G(false, false, dma::kEpiAct, true); break;
      case dma::kEpiGluSilu: if (!extra || !b2 || (!out2 && cp)) return MBX_EINVAL; MBX_LAUNCH_ROWS_G(false, false, dma::kEpiGluSilu, true); break;
      case dma::kEpiGluGelu: if (!extra || !b2 || (!out2 && cp)) return MBX_EINVAL; MBX_LAUNCH_ROWS_G(false, false, dma::kEpiGluGelu, true); break;
      default: return MBX_EINVAL;
    }
    return launch_status();
  }
  if (dma::epi_is_glu(epi)) {
    // b2 is the second matrix of the [w1 | v1] tiles (not a second operand pair)
    if (layout != MBX_NT || !extra || !b2 || (!out2 && cp) || a2) return MBX_EINVAL;
    if (epi == dma::kEpiGluSilu) MBX_LAUNCH_ROWS(false, false, dma::kEpiGluSilu); else MBX_LAUNCH_ROWS(false, false, dma::kEpiGluGelu);
    return launch_status();
  }
  if (dma::epi_is_dglu(epi)) {
    // a2 carries x2 of the gated activation (not a second operand pair)
    if (layout != MBX_NT || !extra || !a2 || !out2) return MBX_EINVAL;
    if (epi == dma::kEpiDgluSilu) MBX_LAUNCH_ROWS(false, false, dma::kEpiDgluSilu); else MBX_LAUNCH_ROWS(false, false, dma::kEpiDgluGelu);
    return launch_status();
  }
  if (epi == dma::kEpiCombine) {
    // extra is the combined output [tokens, n]; c (the product itself) may be absent
    if (layout != MBX_NN || a2 || !extra || !combine.indices) return MBX_EINVAL;
    MBX_LAUNCH_ROWS_C(true, false, dma::kEpiCombine);
    return launch_status();
  }
  if (epi != dma::kEpiNone) {
    if (dual || !extra || (layout != MBX_NT && epi != dma::kEpiAct)) return MBX_EINVAL;
    if (epi == dma::kEpiDact) MBX_LAUNCH_ROWS(false, false, dma::kEpiDact);
    else if (layout == MBX_NN) MBX_LAUNCH_ROWS(true, false, dma::kEpiAct);
    else MBX_LAUNCH_ROWS(false, false, dma::kEpiAct);
    return launch_status();
  }
  if (layout == MBX_NT) {
    if (dual) MBX_LAUNCH_ROWS(false, true, dma::kEpiNone); else MBX_LAUNCH_ROWS(false, false, dma::kEpiNone);
  } else {
    if (dual) MBX_LAUNCH_ROWS(true, true, dma::kEpiNone); else MBX_LAUNCH_ROWS(true, false, dma::kEpiNone);
  }
#undef MBX_LAUNCH_ROWS
#undef MBX_LAUNCH_ROWS_C
#undef MBX_LAUNCH_ROWS_G
  return launch_status();
}

template <bool KTAIL>
int dispatch_rows(const DmaCall& call) {
  if (half_height_only(call.rows, call.num_groups, call.n)) {
    if (call.dtype == MBX_BF16) return launch_rows<MBX_BF16, dma::TileSmallM, dma::TileSmallM, KTAIL>(call);
    return launch_rows<MBX_F16, dma::TileSmallM, dma::TileSmallM, KTAIL>(call);
  }
  if (call.dtype == MBX_BF16) return launch_rows<MBX_BF16, dma::TileMain, dma::TileSmallM, KTAIL>(call);
  return launch_rows<MBX_F16, dma::TileMain, dma::TileSmallM, KTAIL>(call);
}

}  // namespace
}  // namespace mbx
