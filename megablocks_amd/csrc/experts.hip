// The dropless layer's forward behind its router, for few assignments and without gradients: the launches of the separate entry
// points, enqueued by one call.
//
// What bounds such a pass is the host: a layer of a few tokens keeps the GPU busy for 20 - 100 us with five kernels, and four
// calls from Python, each with its checks and allocations, take longer than that.
#include "common.h"

using namespace mbx;

namespace {

// one buffer, in 256-byte pieces
struct Layout {
  size_t total = 0;
  size_t take(size_t bytes) {
    const size_t at = total;
    total += (bytes + 255) & ~(size_t)255;
    return at;
  }
};

struct Parts {
  Layout all;
  size_t indices, bin_ids, bins, slot_rows, sort, hidden, product, sort_bytes;
  Parts(int64_t slots, int num_experts, int end_bit, int hidden_size, int ffn, int dtype) {
    const size_t size = dtype == MBX_F32 ? 4 : 2, n = (size_t)slots;
    sort_bytes = mbx_sort_scratch_bytes(slots > 0 ? slots : 1, MBX_I32, end_bit);
    indices = all.take(n * 4);
    bin_ids = all.take(n * 4);
    slot_rows = all.take(n * 4);
    bins = all.take((size_t)num_experts * 4);
    sort = all.take(sort_bytes);
    hidden = all.take(n * (size_t)ffn * size);
    product = all.take(n * (size_t)hidden_size * size);
  }
};

bool sizes_ok(int64_t tokens, int top_k, int num_experts, int end_bit, int hidden_size, int ffn) {
  return tokens >= 0 && tokens <= 0x7fffffff && top_k > 0 && num_experts > 0 && end_bit > 0 && hidden_size >= 0 && ffn >= 0;
}

}  // namespace

extern "C" {

size_t mbx_experts_forward_scratch_bytes(int64_t tokens, int top_k, int num_experts, int end_bit, int hidden_size, int ffn, int dtype) {
  return sizes_ok(tokens, top_k, num_experts, end_bit, hidden_size, ffn) ? Parts(tokens * top_k, num_experts, end_bit, hidden_size, ffn, dtype).all.total : 0;
}

int mbx_experts_forward(const void* x, int64_t tokens, int hidden_size, int dtype, const int32_t* expert_ids, int top_k,
                        const void* weights, int w_dtype, int num_experts, int end_bit, const void* w1, const void* v1, const void* w2,
                        int ffn, int act, int fused_combine, void* out, int32_t* tokens_per_expert, void* scratch, size_t scratch_bytes,
                        void* workspace, size_t workspace_bytes, mbx_stream_t stream) {
  if (!sizes_ok(tokens, top_k, num_experts, end_bit, hidden_size, ffn)) return MBX_EINVAL;
  if (dtype != MBX_BF16 && dtype != MBX_F16) return MBX_EUNSUPPORTED;
  const int64_t slots = tokens * top_k;
  if (slots == 0 || hidden_size == 0 || ffn == 0) return MBX_EUNSUPPORTED;
  if (!x || !expert_ids || !w1 || !w2 || !out || !tokens_per_expert) return MBX_EINVAL;
  const Parts parts(slots, num_experts, end_bit, hidden_size, ffn, dtype);
  if (!scratch || scratch_bytes < parts.all.total || ((uintptr_t)scratch & 15)) return MBX_ESCRATCH;
  char* const base = (char*)scratch;
  int32_t *const indices = (int32_t*)(base + parts.indices), *const bin_ids = (int32_t*)(base + parts.bin_ids);
  int32_t *const slot_rows = (int32_t*)(base + parts.slot_rows), *const bins = (int32_t*)(base + parts.bins);
  void *const h = base + parts.hidden, *const y = base + parts.product;
  int rc = mbx_route(expert_ids, slots, num_experts, end_bit, 0, indices, bin_ids, tokens_per_expert, bins, nullptr, slot_rows, base + parts.sort, parts.sort_bytes, stream);
  if (rc) return rc;
  rc = mbx_gmm_hidden(x, tokens, indices, top_k, nullptr, w1, v1, h, dtype, bins, num_experts, slots, hidden_size, ffn, act, stream);
  if (rc == MBX_EUNSUPPORTED) {
    // rows that are no whole K tiles: gathered by a launch of their own, to where the second product will be
    rc = mbx_gather(x, dtype, tokens, hidden_size, top_k, indices, bins, nullptr, num_experts, nullptr, 0, y, slots, slot_rows, stream);
    if (!rc) rc = mbx_gmm_hidden(y, slots, nullptr, 1, nullptr, w1, v1, h, dtype, bins, num_experts, slots, hidden_size, ffn, act, stream);
  }
  if (rc) return rc;
  if (top_k == 1 && fused_combine) {
    rc = mbx_gmm_scatter(h, w2, nullptr, out, dtype, bins, num_experts, slots, ffn, hidden_size, indices, weights, w_dtype, tokens, stream);
    if (rc != MBX_EUNSUPPORTED) return rc;
  }
  rc = mbx_gmm_ws(h, w2, nullptr, nullptr, y, dtype, bins, num_experts, slots, ffn, hidden_size, MBX_NN, workspace, workspace_bytes, stream);
  if (rc) return rc;
  return mbx_scatter(y, dtype, tokens, hidden_size, top_k, indices, bin_ids, bins, nullptr, num_experts, weights, w_dtype, out, slot_rows, nullptr, 0, stream);
}

}  // extern "C"
