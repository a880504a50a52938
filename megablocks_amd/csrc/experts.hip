// The dropless layer behind its router, the launches of the separate entry points enqueued by one call: the forward of few
// assignments without gradients, and a training step's forward and backward.
//
// What bounds such passes is the host: a layer of a few tokens keeps the GPU busy for 20 - 100 us with five kernels, and four
// calls from Python, each with its checks and allocations, take longer than that.  A training step is some 15 launches, three autograd
// nodes and their views behind the router (us a step, separate nodes / one call each way: 572 tokens, top-2 of 4 experts of [696, 856],
// gated: 463 / 246;  1024, top-2 of 8 of [512, 1408], gated, fp32 parameters under autocast with both auxiliary losses: 985 / 770).
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

// A training step's three buffers: what the forward keeps for the backward, and what either needs for itself.
struct StepParts {
  Layout kept, forward, backward;
  size_t indices, bin_ids, bins, slot_rows, weights[3], rows, x1, x2, hidden;             // kept
  size_t product;                                                                        // kept with MBX_STEP_KEEP_PRODUCT, else the forward's own
  size_t sort, sort_bytes, hidden_forward;                                               // forward
  size_t grad_rows, d1, d2, table, table_bytes, hidden_again;                            // backward
  StepParts(int64_t tokens, int top_k, int num_experts, int end_bit, int hidden_size, int ffn, bool gate, int flags) {
    const size_t n = (size_t)(tokens * top_k), wide = n * (size_t)ffn * 2, narrow = n * (size_t)hidden_size * 2;
    const size_t weight = (size_t)num_experts * ffn * hidden_size * 2;
    indices = kept.take(n * 4);
    bin_ids = kept.take(n * 4);
    slot_rows = kept.take(n * 4);
    bins = kept.take((size_t)num_experts * 4);
    for (int w = 0; w < 3; ++w) weights[w] = flags & MBX_STEP_FP32_WEIGHTS && (w != 1 || gate) ? kept.take(weight) : 0;
    rows = flags & MBX_STEP_GATHER ? 0 : kept.take(narrow);
    x1 = kept.take(wide);
    x2 = gate ? kept.take(wide) : 0;
    const bool again = flags & MBX_STEP_RECOMPUTE;
    hidden = again ? 0 : kept.take(wide);
    if (flags & MBX_STEP_KEEP_PRODUCT) product = kept.take(narrow);
    sort_bytes = mbx_sort_scratch_bytes(n ? n : 1, MBX_I32, end_bit);
    sort = forward.take(sort_bytes);
    hidden_forward = again ? forward.take(wide) : 0;
    if (!(flags & MBX_STEP_KEEP_PRODUCT)) product = forward.take(narrow);
    grad_rows = backward.take(narrow);
    d1 = backward.take(wide);
    d2 = gate ? backward.take(wide) : 0;
    table_bytes = flags & MBX_STEP_GATHER ? mbx_gmm_tn_gather_table_bytes(tokens, top_k, num_experts) : 0;
    table = backward.take(table_bytes);
    hidden_again = again ? d1 : 0;   // before the gradient of the first product, and done with by then
  }
};

// count (a multiple of 8) fp32 values as 16-bit ones, of up to three arrays: a launch for all of them
template <int DT>
__global__ void __launch_bounds__(256) cast_kernel(const float* __restrict__ s0, const float* __restrict__ s1, const float* __restrict__ s2,
                                                   uint16_t* __restrict__ d0, uint16_t* __restrict__ d1, uint16_t* __restrict__ d2, int64_t count) {
  const float* const src = blockIdx.y == 0 ? s0 : blockIdx.y == 1 ? s1 : s2;
  uint16_t* const dst = blockIdx.y == 0 ? d0 : blockIdx.y == 1 ? d1 : d2;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < count / 8; i += (int64_t)gridDim.x * 256) {
    const float4 a = ((const float4*)src)[2 * i], b = ((const float4*)src)[2 * i + 1];
    typedef typename Elem<DT>::type T;
    T v[8] = {Elem<DT>::from_f32(a.x), Elem<DT>::from_f32(a.y), Elem<DT>::from_f32(a.z), Elem<DT>::from_f32(a.w),
              Elem<DT>::from_f32(b.x), Elem<DT>::from_f32(b.y), Elem<DT>::from_f32(b.z), Elem<DT>::from_f32(b.w)};
    uint4 out;
    __builtin_memcpy(&out, v, 16);
    ((uint4*)dst)[i] = out;
  }
}

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
    rc = mbx_gmm_scatter_ws(h, w2, nullptr, out, dtype, bins, num_experts, slots, ffn, hidden_size, indices, weights, w_dtype, tokens, workspace, workspace_bytes, stream);
    if (rc != MBX_EUNSUPPORTED) return rc;
  }
  rc = mbx_gmm_ws(h, w2, nullptr, nullptr, y, dtype, bins, num_experts, slots, ffn, hidden_size, MBX_NN, workspace, workspace_bytes, stream);
  if (rc) return rc;
  return mbx_scatter(y, dtype, tokens, hidden_size, top_k, indices, bin_ids, bins, nullptr, num_experts, weights, w_dtype, out, slot_rows, nullptr, 0, stream);
}

// which: 0 what the forward keeps for the backward, 1 / 2 the scratch of the forward / the backward
size_t mbx_experts_step_bytes(int64_t tokens, int top_k, int num_experts, int end_bit, int hidden_size, int ffn, int gate, int flags, int which) {
  if (!sizes_ok(tokens, top_k, num_experts, end_bit, hidden_size, ffn) || which < 0 || which > 2) return 0;
  const StepParts p(tokens, top_k, num_experts, end_bit, hidden_size, ffn, gate != 0, flags);
  return which == 0 ? p.kept.total : which == 1 ? p.forward.total : p.backward.total;
}

int mbx_experts_step_forward(const void* x, int64_t tokens, int hidden_size, int dtype, const int32_t* expert_ids, int top_k,
                             const void* weights, int w_dtype, int num_experts, int end_bit, const void* w1, const void* v1, const void* w2,
                             int ffn, int act, int flags, void* out, int32_t* tokens_per_expert, void* kept, size_t kept_bytes,
                             void* scratch, size_t scratch_bytes, void* workspace, size_t workspace_bytes, mbx_stream_t stream) {
  if (!sizes_ok(tokens, top_k, num_experts, end_bit, hidden_size, ffn)) return MBX_EINVAL;
  const int64_t slots = tokens * top_k;
  // what the launches of the backward take, which cannot go another way any more: 16-bit whole 16-byte pieces of rows, four K tiles to an
  // operand pair of the gate's input gradient, more than a half-height tile of the indexed weight gradient, up to eight experts a token, 256
  // rows of an operand below 2 GiB (the gate's two halves of a tile: half a tile more)
  if ((dtype != MBX_BF16 && dtype != MBX_F16) || slots == 0 || hidden_size == 0 || hidden_size % 8 || ffn % 8 || ffn <= 192 || top_k > 8 ||
      ffn >= (1 << 22) - 128 || hidden_size >= 1 << 22 ||
      slots * (int64_t)(hidden_size > ffn ? hidden_size : ffn) * 2 >= (int64_t)1 << 31 || (int64_t)hidden_size * ffn * 2 >= (int64_t)1 << 30)
    return MBX_EUNSUPPORTED;
  if (!x || !expert_ids || !weights || !w1 || !w2 || !out || !tokens_per_expert) return MBX_EINVAL;
  const StepParts p(tokens, top_k, num_experts, end_bit, hidden_size, ffn, v1 != nullptr, flags);
  if (!kept || !scratch || kept_bytes < p.kept.total || scratch_bytes < p.forward.total || (((uintptr_t)kept | (uintptr_t)scratch) & 15)) return MBX_ESCRATCH;
  if (((uintptr_t)x | (uintptr_t)w1 | (uintptr_t)v1 | (uintptr_t)w2 | (uintptr_t)out) & 15) return MBX_EUNSUPPORTED;
  char* const base = (char*)kept;
  int32_t *const indices = (int32_t*)(base + p.indices), *const bin_ids = (int32_t*)(base + p.bin_ids);
  int32_t *const slot_rows = (int32_t*)(base + p.slot_rows), *const bins = (int32_t*)(base + p.bins);
  void *const x1 = base + p.x1, *const x2 = v1 ? base + p.x2 : nullptr;
  void* const y = (flags & MBX_STEP_KEEP_PRODUCT ? base : (char*)scratch) + p.product;
  void* const h = flags & MBX_STEP_RECOMPUTE ? (char*)scratch + p.hidden_forward : base + p.hidden;
  int rc = mbx_route(expert_ids, slots, num_experts, end_bit, 0, indices, bin_ids, tokens_per_expert, bins, nullptr, slot_rows, (char*)scratch + p.sort, p.sort_bytes, stream);
  if (rc) return rc;
  if (flags & MBX_STEP_FP32_WEIGHTS) {
    const int64_t count = (int64_t)num_experts * ffn * hidden_size;
    const int64_t blocks = ceil_div(count / 8, 256);
    const dim3 grid((unsigned)(blocks > 2048 ? 2048 : blocks), v1 ? 3 : 2);
    const float *s1 = (const float*)w1, *s2 = (const float*)(v1 ? v1 : w2), *s3 = (const float*)w2;
    uint16_t *d1 = (uint16_t*)(base + p.weights[0]), *d2 = (uint16_t*)(base + p.weights[v1 ? 1 : 2]), *d3 = (uint16_t*)(base + p.weights[2]);
    if (dtype == MBX_BF16) cast_kernel<MBX_BF16><<<grid, 256, 0, as_stream(stream)>>>(s1, s2, s3, d1, d2, d3, count);
    else cast_kernel<MBX_F16><<<grid, 256, 0, as_stream(stream)>>>(s1, s2, s3, d1, d2, d3, count);
    if ((rc = launch_status())) return rc;
    w1 = base + p.weights[0];
    v1 = v1 ? base + p.weights[1] : nullptr;
    w2 = base + p.weights[2];
  }
  rc = MBX_EUNSUPPORTED;
  if (flags & MBX_STEP_GATHER)
    rc = mbx_gmm_gather(x, tokens, indices, top_k, nullptr, w1, v1, x1, x2, h, dtype, bins, num_experts, slots, hidden_size, ffn, act, stream);
  if (rc == MBX_EUNSUPPORTED) {
    // rows that are no whole K tiles go where the second product will be
    void* const rows = flags & MBX_STEP_GATHER ? y : base + p.rows;
    rc = mbx_gather(x, dtype, tokens, hidden_size, top_k, indices, bins, nullptr, num_experts, nullptr, 0, rows, slots, top_k > 1 ? slot_rows : nullptr, stream);
    if (!rc) rc = v1 ? mbx_gmm_glu(rows, w1, v1, x1, x2, h, dtype, bins, num_experts, slots, hidden_size, ffn, act, stream)
                     : mbx_gmm_act(rows, w1, x1, h, dtype, bins, num_experts, slots, hidden_size, ffn, act, stream);
  }
  if (rc) return rc;
  if (top_k == 1 && flags & MBX_STEP_COMBINE) {
    rc = mbx_gmm_scatter_ws(h, w2, flags & MBX_STEP_KEEP_PRODUCT ? y : nullptr, out, dtype, bins, num_experts, slots, ffn, hidden_size, indices, weights, w_dtype, tokens, workspace, workspace_bytes, stream);
    if (rc != MBX_EUNSUPPORTED) return rc;
  }
  rc = mbx_gmm_ws(h, w2, nullptr, nullptr, y, dtype, bins, num_experts, slots, ffn, hidden_size, MBX_NN, workspace, workspace_bytes, stream);
  if (rc) return rc;
  return mbx_scatter(y, dtype, tokens, hidden_size, top_k, indices, bin_ids, bins, nullptr, num_experts, weights, w_dtype, out, slot_rows, nullptr, 0, stream);
}

int mbx_experts_step_backward(const void* grad, const void* x, int64_t tokens, int hidden_size, int dtype, int top_k, const void* weights,
                              int w_dtype, int num_experts, int end_bit, const void* w1, const void* v1, const void* w2, int ffn, int act,
                              int flags, const void* kept, size_t kept_bytes, void* dx, void* dweights, void* dw1, void* dv1, void* dw2,
                              void* scratch, size_t scratch_bytes, void* workspace, size_t workspace_bytes, mbx_stream_t stream) {
  if (!sizes_ok(tokens, top_k, num_experts, end_bit, hidden_size, ffn) || tokens == 0 || !grad || !weights) return MBX_EINVAL;
  const bool gate = flags & MBX_STEP_GATE, gathered = flags & MBX_STEP_GATHER, fp32 = flags & MBX_STEP_FP32_WEIGHTS;
  if ((!fp32 && (!w1 || !w2 || (gate && !v1))) || (gathered && !x) || (dv1 && !gate) || (dweights && !(flags & MBX_STEP_KEEP_PRODUCT))) return MBX_EINVAL;
  const int64_t slots = tokens * top_k;
  const StepParts p(tokens, top_k, num_experts, end_bit, hidden_size, ffn, gate, flags);
  if (!kept || !scratch || kept_bytes < p.kept.total || scratch_bytes < p.backward.total || (((uintptr_t)kept | (uintptr_t)scratch) & 15)) return MBX_ESCRATCH;
  const char* const base = (const char*)kept;
  char* const own = (char*)scratch;
  const int32_t *const indices = (const int32_t*)(base + p.indices), *const bin_ids = (const int32_t*)(base + p.bin_ids);
  const int32_t *const slot_rows = (const int32_t*)(base + p.slot_rows), *const bins = (const int32_t*)(base + p.bins);
  const void *const x1 = base + p.x1, *const x2 = gate ? base + p.x2 : nullptr, *const y = base + p.product;   // y: with MBX_STEP_KEEP_PRODUCT only
  const bool again = flags & MBX_STEP_RECOMPUTE;
  const void* const h = again ? own + p.hidden_again : base + p.hidden;
  if (fp32) {
    w1 = base + p.weights[0];
    v1 = gate ? base + p.weights[1] : nullptr;
    w2 = base + p.weights[2];
  }
  void *const grad_rows = own + p.grad_rows, *const d1 = own + p.d1, *const d2 = gate ? own + p.d2 : nullptr;
  int rc = dweights ? mbx_scatter_backward(grad, y, dtype, tokens, hidden_size, top_k, indices, bins, nullptr, num_experts, weights, w_dtype, slot_rows, grad_rows, slots, dweights, stream)
                    : mbx_gather(grad, dtype, tokens, hidden_size, top_k, indices, bins, nullptr, num_experts, weights, w_dtype, grad_rows, slots, top_k > 1 ? slot_rows : nullptr, stream);
  if (rc) return rc;
  if (dw2) {
    if (again) {
      rc = gate ? mbx_glu_forward(x1, x2, (void*)h, dtype, act, slots * ffn, stream) : mbx_gelu_forward(x1, (void*)h, dtype, slots * ffn, stream);
      if (rc) return rc;
    }
    rc = fp32 ? mbx_gmm_tn_f32(h, grad_rows, 0, nullptr, 1, nullptr, (float*)dw2, dtype, bins, num_experts, slots, ffn, hidden_size, nullptr, 0, 0, stream)
              : mbx_gmm(h, grad_rows, dw2, dtype, bins, num_experts, slots, ffn, hidden_size, MBX_TN, stream);
    if (rc) return rc;
  }
  if (!dx && !dw1 && !dv1) return 0;
  rc = gate ? mbx_gmm_dglu(grad_rows, w2, x1, x2, d1, d2, dtype, bins, num_experts, slots, hidden_size, ffn, act, stream)
            : mbx_gmm_dact(grad_rows, w2, x1, d1, dtype, bins, num_experts, slots, hidden_size, ffn, act, stream);
  if (rc) return rc;
  int ready = 0;
  for (int w = 0; w < 2; ++w) {
    void* const dw = w ? dv1 : dw1;
    const void* const d = w ? d2 : d1;
    if (!dw) continue;
    void* const table = own + p.table;
    if (gathered)
      rc = fp32 ? mbx_gmm_tn_f32(d, x, tokens, indices, top_k, nullptr, (float*)dw, dtype, bins, num_experts, slots, ffn, hidden_size, table, p.table_bytes, ready, stream)
                : mbx_gmm_tn_gather(d, x, tokens, indices, top_k, nullptr, dw, dtype, bins, num_experts, slots, ffn, hidden_size, table, p.table_bytes, ready, stream);
    else
      rc = fp32 ? mbx_gmm_tn_f32(d, base + p.rows, 0, nullptr, 1, nullptr, (float*)dw, dtype, bins, num_experts, slots, ffn, hidden_size, nullptr, 0, 0, stream)
                : mbx_gmm(d, base + p.rows, dw, dtype, bins, num_experts, slots, ffn, hidden_size, MBX_TN, stream);
    if (rc) return rc;
    ready = 1;
  }
  if (!dx) return 0;
  // the rows' gradient goes where the incoming one was, which nothing reads any more
  rc = mbx_gmm_ws(d1, w1, d2, gate ? v1 : nullptr, grad_rows, dtype, bins, num_experts, slots, ffn, hidden_size, MBX_NN, workspace, workspace_bytes, stream);
  if (rc) return rc;
  return mbx_scatter(grad_rows, dtype, tokens, hidden_size, top_k, indices, bin_ids, bins, nullptr, num_experts, nullptr, 0, dx, slot_rows, nullptr, 0, stream);
}

}  // extern "C"
