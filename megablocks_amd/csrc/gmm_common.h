// What the translation units of the grouped GEMM share: vector types, the mapping of tiles to XCDs, the workspace a
// caller lends, launch helpers.
#pragma once

#include "common.h"

namespace mbx {

// kWorkspaceCounters int32 counters, zero before the launch and zero again after it, then room for fp32 tiles.
constexpr size_t kWorkspaceCounters = 1024, kWorkspacePartBytes = (size_t)256 * 256 * 4, kWorkspaceParts = 320;
struct Workspace {
  void* base = nullptr;
  size_t bytes = 0;
};

// The weighted combine in the epilogue (kEpiCombine): the sorted assignments (top_k = 1: tokens) of the product's rows,
// the weights by token (or null) and their type, the row count of the combined output.
struct CombineRows {
  const int32_t* indices = nullptr;
  const void* weights = nullptr;
  int w_dtype = 0;
  int tokens = 0;
};

// Rows of an operand gathered on the fly.
struct GatherRows {
  const int32_t* slots = nullptr;      // non-null: a (NT) / b (TN) is [src_rows, .], read through the row map
  const int32_t* src_bins = nullptr;
  int top_k = 1, src_rows = 0;
  // TN only: the table of row offsets the kernel reads (4 bytes per sorted assignment, n_slots of them), and whether an
  // earlier call with the same slots, top_k, src_rows and n has already filled it
  uint32_t* row_table = nullptr;
  int64_t n_slots = 0;
  bool table_ready = false;
};

// A launch of the direct-to-LDS kernels on 16-bit operands (gmm_dma.h).
//   a2 / b2 non-null (no epilogue): c = a @ b[e] + a2 @ b2[e], the second pair shaped like the first;
//   epi / extra / out2: an epilogue (dma::kEpi*) and its second output / input, third output; kEpiDglu*: a2 is x2; kEpiGlu*: b2 is
//   the second matrix;
//   gather: rows of `a` (NT; no epilogue, kEpiAct or kEpiGlu*) or of `b` (TN) picked through the sorted assignments;
//   ws: device memory the launch may use for the parts of tiles it cuts along the reduction (NN without epilogue or with the combine).
struct DmaCall {
  const void *a, *b;
  void* c;
  int dtype;
  const int32_t* bins;
  int num_groups;
  int64_t rows;
  int k, n, layout;
  hipStream_t stream;
  const void *a2 = nullptr, *b2 = nullptr;
  int epi = 0;
  void *extra = nullptr, *out2 = nullptr;
  GatherRows gather{};
  Workspace ws{};
  CombineRows combine{};
  bool out32 = false;   // TN: c is fp32
};

// NN / NT launches with a handful of rows per expert (gmm_few.hip), and whether a launch is one of them.
bool gmm_few_takes(const DmaCall& call);
int gmm_few(const DmaCall& call);

// NT launches with a few dozen rows per expert (gmm_mid.hip), and whether a launch is one of them.
bool gmm_mid_takes(const DmaCall& call);
int gmm_mid(const DmaCall& call);

// NN launches with no full round of tiles are cut along the reduction from this many K tiles on: exchanging the parts takes some 20
// us.  8 experts of 48 rows, [4096, 1024]: 61 -> 36 us; 4 of 500, [2816, 1024]: 58 -> 45; 8 of 256, [1408, 512]: 18 -> 21.
constexpr int kMinCutTiles = 32;
// A cut tile has up to kMaxKSplit parts of at least kMinPartTiles K tiles.
constexpr int kMaxKSplit = 8, kMinPartTiles = 8;
// Behind full rounds the tail's tiles are cut along the reduction into three parts and more from kMinTailCutTiles K tiles on, into two from kMinTailHalvesTiles:
// below, half-height tiles, where a launch has them, take less (8 experts of 1024 rows, [k, 2304 / 2560 / 2816 / 3072], i.e. tails cut into 8 / 4 / 2 / 2 parts, operands out of
// memory, us cut and not: k = 1024 69 / 50 and 73 / 50 (2 parts); 2048 85 / 80, 95 / 85, 93 / 81, 101 / 84; 4096 160 / 143, 153 / 151, 153 / 145, 162 / 152; 5120 192 / 182,
// 183 / 193, 188 / 184, 195 / 192; 6144 199 / 213, 205 / 225, 224 / 215, 226 / 229; 8192 245 / 271, 254 / 293, 289 / 280, 302 / 294; 10240 305 / 344, 313 / 365, 354 / 352,
// 369 / 378; 14336 404 / 467, 436 / 501, 481 / 488, 508 / 544).
constexpr int kMinTailCutTiles = 80, kMinTailHalvesTiles = 160;
// Launches of half-height tiles only have nothing to take instead, but two parts pay from kMinHalfHeightHalvesTiles K tiles on (160 launches, 4 - 128
// experts of 30 - 320 rows, with the combine; cut / not: two parts of up to 23 K tiles 1.035, 24 - 31 1.015, 32 - 39 0.99, 40 - 47 0.96, beyond 0.93; three 0.96 - 0.86,
// more 0.92 - 0.72).
constexpr int kMinHalfHeightHalvesTiles = 40;
__host__ __device__ constexpr bool cut_pays(bool half_height_only, int full_rounds, int parts, int k_tiles) {
  if (parts < 2 || full_rounds == 0) return parts >= 2;
  if (half_height_only) return parts >= 3 || k_tiles >= kMinHalfHeightHalvesTiles;
  return k_tiles >= (parts >= 3 ? kMinTailCutTiles : kMinTailHalvesTiles);
}

// NN / NT launches of gmm_dma.h's kernel are tiled with the half-height tile only up to kHalfHeightRows rows per expert on average, and
// up to kMixedRows unless full tiles with a half-height last one make kMixedRounds rounds (gmm_rows.h).
constexpr int kHalfHeightRows = 144, kMixedRows = 320, kMixedRounds = 3;

// NN / NT launches of few tiles (gmm_pair.hip): whether a launch could run there, and whether it is one of them.
bool gmm_pair_can(const DmaCall& call);
bool gmm_pair_takes(const DmaCall& call);
int gmm_pair(const DmaCall& call);

// TN launches with few rows per expert (gmm_tn_short.hip), and whether a launch is one of them.
bool gmm_tn_short_takes(const DmaCall& call);
int gmm_tn_short(const DmaCall& call);
// For tests: 0 gmm_dma.h's kernel, 1 128 x 128 tiles, 2 256 x 128 tiles, 3 128 x 128 tiles that fetch ahead.
int gmm_tn_short_choice(const DmaCall& call);

// NN / NT launches, k a multiple of 64 (gmm_rows.hip) and of 8 only (gmm_rows_tail.hip).
int gmm_rows(const DmaCall& call);
int gmm_rows_tail(const DmaCall& call);
#ifdef MBX_TICKS
int gmm_rows_set_ticks(void* buffer);
int gmm_rows_tail_set_ticks(void* buffer);
#endif

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));

template <int DT>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  const f32x2_t v = {a, b};
  if (DT == MBX_BF16) return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));  // v_cvt_pk_bf16_f32, RNE
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2_t));
}

// Workgroups are dispatched to the 8 XCDs round-robin by workgroup id, and every XCD has its own
// L2.  The logical tile order is cut into runs of kXcdRun tiles and run r goes to XCD r % 8, so
// the workgroups resident on one XCD at a time form a compact block of tiles (same expert, a few
// row tiles x a few column tiles) whose operand panels are fetched into that L2 once.
constexpr int kXcds = 8;
constexpr int kXcdRun = 32;

__device__ __forceinline__ int xcd_tile_id(int block, int run = kXcdRun) {
  const int xcd = block % kXcds, l = block / kXcds;
  return ((l / run) * kXcds + xcd) * run + (l % run);
}

static inline int64_t xcd_grid(int64_t tiles, int run = kXcdRun) {
  const int64_t q = (int64_t)kXcds * run;
  return (tiles + q - 1) / q * q;
}

// This lane's expert's place (lane e: expert e, num_groups <= 64) in the order of decreasing row count, equal ones as they come; -1
// past the last expert.  Every workgroup of a TN launch works it out: lane by lane out of registers, 0.4 us for 64 experts where
// shuffles through the LDS take 2.
__device__ __forceinline__ int rank_by_rows(int rows_of_expert, int num_groups) {
  const int lane = __lane_id();
  const int limit = 0x7fffffff >> 6, rows = rows_of_expert < 0 ? 0 : rows_of_expert < limit ? rows_of_expert : limit;
  const int key = lane < num_groups ? rows << 6 | (kWave - 1 - lane) : -1;   // no two alike
  int rank = 0;
  for (int first = 0; first < num_groups; first += 8)   // up to seven lanes past the last expert, whose keys are below all
#pragma unroll
    for (int o = 0; o < 8; ++o) rank += __builtin_amdgcn_readlane(key, first + o) > key ? 1 : 0;
  return lane < num_groups ? rank : -1;
}

// A row bound read from the bins, kept inside [lo, rows]: a table that does not belong to the operands can make
// the result wrong but never an access out of range.
__device__ __forceinline__ int clamp_bound(int v, int lo, int rows) { return v < lo ? lo : (v > rows ? rows : v); }

// The workspace as the kernels take it: counters, then parts of `part_bytes` each, 16-byte aligned; parts null where it
// cannot hold two.
struct WorkspaceParts {
  int32_t* counters = nullptr;
  float* parts = nullptr;
  int capacity = 0;
  WorkspaceParts(const Workspace& ws, size_t part_bytes) {
    const size_t head = kWorkspaceCounters * sizeof(int32_t);
    if (!ws.base || ((uintptr_t)ws.base & 15u) != 0 || ws.bytes < head + 2 * part_bytes) return;
    const size_t fit = (ws.bytes - head) / part_bytes;
    counters = (int32_t*)ws.base;
    parts = (float*)((char*)ws.base + head);
    capacity = (int)(fit > 0x7fffffff ? 0x7fffffff : fit);
  }
};

static inline bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

template <typename K>
int allow_lds(K kernel, size_t bytes) {
  return (int)hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

// One persistent workgroup per compute unit (a multiple of 8, so that every XCD gets the same number),
// fewer when there are not that many tiles.
static inline int persistent_grid(int64_t tiles_upper_bound) {
  static int cus[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
  if (cus[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < kXcds) n = 256;
    cus[dev] = n / kXcds * kXcds;
  }
  const int64_t need = (tiles_upper_bound + kXcds - 1) / kXcds * kXcds;
  return (int)(need < cus[dev] ? need : cus[dev]);
}

}  // namespace

// gmm_f32.hip: fp32 products of whole 16-byte pieces; MBX_EUNSUPPORTED where the operands are not, and for TN launches with few
// rows per expert.  a2 / b2 non-null
// (NN / NT): c = a @ b[e] + a2 @ b2[e].
int gmm_f32(const void* a, const void* b, const void* a2, const void* b2, void* c, const int32_t* bins, int num_groups,
            int64_t rows, int k, int n, int layout, void* workspace, size_t workspace_bytes, hipStream_t s);
// For tests: whether an NN / NT launch takes the small tile.
bool gmm_f32_rows_small(int num_groups, int64_t rows, int k, int n, bool dual);

}  // namespace mbx
