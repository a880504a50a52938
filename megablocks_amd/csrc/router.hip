// Router post-processing: softmax over the experts, top-k selection and the optional p-norm
// renormalisation of the selected weights in one kernel, and their backward in another
// (megablocks/layers/router.py:87-106).  One wave per token; lane l holds experts l, l + 64, ...
#include "common.h"

namespace mbx {
namespace {

constexpr int kTokenThreads = 256;
constexpr int kTokenWaves = kTokenThreads / kWave;

// ||w||_p of the first top_k lanes' values (p > 0)
__device__ __forceinline__ float wave_pnorm(float w, bool live, float p) {
  const float a = fabsf(w);
  float term = 0.f;
  if (live) term = p == 1.f ? a : (p == 2.f ? a * a : powf(a, p));
  const float sum = wave_sum(term);
  return p == 1.f ? sum : (p == 2.f ? sqrtf(sum) : powf(sum, 1.f / p));
}

// One token's scores, choices and weights, by one wave: lane l has the logits of experts l, l + 64, ... in x (-inf past the
// last).  scores = softmax(logits) rounded to the storage type (computed in fp32: exp(x - max) / sum, as
// torch's softmax does for 16-bit inputs); the k largest rounded scores in descending order, ties to the
// lower expert index (NaN scores first); weights = those scores, divided by their rounded p-norm if p > 0
// (each of torch's two operations rounds to the storage type).
template <int DT, int R>
__device__ __forceinline__ void route_token(float (&x)[R], int64_t t, int num_experts, int top_k, float p,
                                            typename Elem<DT>::type* __restrict__ scores, typename Elem<DT>::type* __restrict__ weights,
                                            int64_t* __restrict__ indices, int32_t* __restrict__ indices32, float* __restrict__ lse) {
  typedef typename Elem<DT>::type E;
  const int lane = lane_id();
  float m = -INFINITY;
#pragma unroll
  for (int r = 0; r < R; ++r) m = fmaxf(m, x[r]);
  m = wave_max(m);
  float sum = 0.f;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    x[r] = lane + r * kWave < num_experts ? expf(x[r] - m) : 0.f;
    sum += x[r];
  }
  sum = wave_sum(sum);
  // logsumexp of the row, the term of the router z-loss (router.py:37): an infinite maximum is the result itself
  if (lse && lane == 0) lse[t] = (m == INFINITY || m == -INFINITY) ? m : m + logf(sum);
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int e = lane + r * kWave;
    const E s = Elem<DT>::from_f32(x[r] / sum);
    if (e < num_experts) scores[t * num_experts + e] = s;
    // The selection key: the rounded score; -1 marks "not a candidate" (scores are >= 0).  A NaN score (a NaN
    // or +inf logit makes the whole row NaN) ranks above every number, as torch.topk ranks it, so that the
    // indices written are always experts: +inf, which no score can be, stands for it.
    const float v = Elem<DT>::to_f32(s);
    x[r] = e < num_experts ? (v != v ? INFINITY : v) : -1.f;
  }
  float my_w = 0.f;
  int my_i = 0;
  for (int j = 0; j < top_k; ++j) {
    float best = -1.f;
    int best_e = 0x7fffffff;
#pragma unroll
    for (int r = 0; r < R; ++r)   // ascending expert index: a later equal value does not replace an earlier one
      if (x[r] > best) { best = x[r]; best_e = lane + r * kWave; }
    // the largest score, then the lowest expert that has it
    const float top = wave_butterfly(best, [](float a, float b) { return a > b ? a : b; });
    best_e = wave_butterfly(best == top ? best_e : 0x7fffffff, [](int a, int b) { return a < b ? a : b; });
    best = top;
    if (lane == j) { my_w = best == INFINITY ? NAN : best; my_i = best_e; }
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (lane + r * kWave == best_e) x[r] = -1.f;
  }
  const bool live = lane < top_k;
  if (p > 0.f) {
    const float norm = Elem<DT>::to_f32(Elem<DT>::from_f32(wave_pnorm(my_w, live, p)));
    my_w = my_w / norm;
  }
  if (live) {
    weights[t * top_k + lane] = Elem<DT>::from_f32(my_w);
    indices[t * top_k + lane] = my_i;
    if (indices32) indices32[t * top_k + lane] = my_i;   // what the routing kernels take, without a cast pass
  }
}

template <int DT, int R>
__global__ void __launch_bounds__(kTokenThreads)
router_forward_kernel(const void* __restrict__ logits_, int64_t tokens, int num_experts, int top_k, float p,
                      void* __restrict__ scores, void* __restrict__ weights, int64_t* __restrict__ indices,
                      int32_t* __restrict__ indices32, float* __restrict__ lse) {
  typedef typename Elem<DT>::type E;
  const E* logits = (const E*)logits_;
  const int lane = lane_id(), wave = threadIdx.x / kWave;
  for (int64_t t = (int64_t)blockIdx.x * kTokenWaves + wave; t < tokens; t += (int64_t)gridDim.x * kTokenWaves) {
    float x[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int e = lane + r * kWave;
      x[r] = e < num_experts ? Elem<DT>::to_f32(logits[t * num_experts + e]) : -INFINITY;
    }
    route_token<DT, R>(x, t, num_experts, top_k, p, (E*)scores, (E*)weights, indices, indices32, lse);
  }
}

// The router's linear layer and the above in one launch, for a few tokens: logits[t][e] = x[t] . weight[e], summed in fp32 and
// rounded to the storage type.  One workgroup of sixteen waves per token: wave w has experts w, w + 16, ..., a lane eight
// columns of every 512, so that a load of a wave is 1 KiB of one row.
//
// What bounds it: the latency of reading the weights (64 experts of 2048: 256 KiB) through one compute unit, and of the chain
// of waits behind it.  The vendor library's product and router_forward_kernel / this kernel, us, 5 tokens: 8 experts of 4096:
// 12.4 / 6.8, 12 of 1032: 10.8 / 7.8, 64 of 2048: 11.1 / 9.1, 64 of 4096: 13.6 / 11.1, 128 of 2048: 11.6 / 11.7, 128 of 4096:
// 14.0 / 16.1; 256 tokens (one per compute unit): 12.8 / 7.4, 11.7 / 8.4, 11.4 / 10.4, 14.0 / 12.7, 12.0 / 13.7.  (On the matrix
// instruction, 16 tokens per workgroup, whose loads take 16 rows at a stride of often a power of two: 64 of 2048 16 - 21.)
constexpr int kLinearWaves = 16;
constexpr int kLinearMaxExperts = 8 * kLinearWaves;

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// PER: experts per wave
template <int DT, int PER>
__global__ void __launch_bounds__(kLinearWaves * kWave)
router_linear_kernel(const uint16_t* __restrict__ x_, const uint16_t* __restrict__ weight, int hidden, int num_experts,
                     int top_k, float p, void* __restrict__ scores, void* __restrict__ weights, int64_t* __restrict__ indices,
                     int32_t* __restrict__ indices32) {
  typedef typename Elem<DT>::type E;
  constexpr int kAhead = PER >= 8 ? 2 : PER >= 4 ? 4 : 8;   // pieces of a row under way, next to those of the other experts
  constexpr int R = PER <= 4 ? 1 : 2;
  __shared__ float logits[PER * kLinearWaves < kWave ? kWave : PER * kLinearWaves];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = lane_id();
  const int64_t t = blockIdx.x;
  // pieces past the end of a row and experts past the last (bit 31: out of range) read as zeros
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void*)(x_ + t * hidden), 0, hidden * 2, 0x00020000);
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)weight, 0, num_experts * hidden * 2, 0x00020000);
  auto unpack = [](uint32_t v, float& lo, float& hi) {
    lo = Elem<DT>::to_f32(__builtin_bit_cast(E, (uint16_t)v));
    hi = Elem<DT>::to_f32(__builtin_bit_cast(E, (uint16_t)(v >> 16)));
  };
  float acc[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) acc[i] = 0.f;
  const uint32_t pitch = (uint32_t)hidden * 2u;
  for (int k0 = lane * 8; k0 - lane * 8 < hidden; k0 += 512 * kAhead) {
    u32x4_t xv[kAhead], wv[kAhead][PER];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const uint32_t at = 2u * (uint32_t)(k0 + 512 * u) | (k0 + 512 * u < hidden ? 0u : 0x80000000u);
      xv[u] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rx, (int)at, 0, 0));
#pragma unroll
      for (int i = 0; i < PER; ++i)
        wv[u][i] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rw, (int)(at + (uint32_t)(wave + kLinearWaves * i) * pitch), 0, 0));
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u)
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        float x0, x1;
        unpack(xv[u][w], x0, x1);
#pragma unroll
        for (int i = 0; i < PER; ++i) {
          float w0, w1;
          unpack(wv[u][i][w], w0, w1);
          acc[i] = fmaf(x0, w0, acc[i]);
          acc[i] = fmaf(x1, w1, acc[i]);
        }
      }
  }
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const float sum = wave_sum(acc[i]);
    if (lane == 0) logits[wave + kLinearWaves * i] = sum;
  }
  __syncthreads();
  if (wave != 0) return;
  float v[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int e = lane + r * kWave;
    v[r] = e < num_experts ? Elem<DT>::to_f32(Elem<DT>::from_f32(logits[e])) : -INFINITY;
  }
  route_token<DT, R>(v, t, num_experts, top_k, p, (E*)scores, (E*)weights, indices, indices32, nullptr);
}

// grad_logits = d(loss)/d(logits) given d/d(weights) (and optionally d/d(scores) from other users of the
// scores, e.g. a load-balancing loss): through the p-norm division, the selection (a scatter to the chosen
// experts) and the softmax, in fp32 from the rounded forward values.  grad_lse (optional): d/d(logsumexp of the
// row), whose gradient with respect to the logits is the softmax itself.
template <int DT, int R>
__global__ void __launch_bounds__(kTokenThreads)
router_backward_kernel(const void* __restrict__ grad_weights_, const void* __restrict__ grad_scores_,
                       const void* __restrict__ scores_, const int64_t* __restrict__ indices, int64_t tokens,
                       int num_experts, int top_k, float p, void* __restrict__ grad_logits_,
                       const float* __restrict__ grad_lse) {
  typedef typename Elem<DT>::type E;
  const E* grad_weights = (const E*)grad_weights_;
  const E* grad_scores = (const E*)grad_scores_;
  const E* scores = (const E*)scores_;
  E* grad_logits = (E*)grad_logits_;
  const int lane = lane_id(), wave = threadIdx.x / kWave;
  for (int64_t t = (int64_t)blockIdx.x * kTokenWaves + wave; t < tokens; t += (int64_t)gridDim.x * kTokenWaves) {
    float s[R], ds[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int e = lane + r * kWave;
      s[r] = e < num_experts ? Elem<DT>::to_f32(scores[t * num_experts + e]) : 0.f;
      ds[r] = (grad_scores && e < num_experts) ? Elem<DT>::to_f32(grad_scores[t * num_experts + e]) : 0.f;
    }
    if (grad_weights) {
      const bool live = lane < top_k;
      int my_i = live ? (int)indices[t * top_k + lane] : 0;
      if (my_i < 0 || my_i >= num_experts) my_i = 0;
      const float dy = live ? Elem<DT>::to_f32(grad_weights[t * top_k + lane]) : 0.f;
      const float w = live ? Elem<DT>::to_f32(scores[t * num_experts + my_i]) : 0.f;   // the weight before the division
      float dw = dy;
      if (p > 0.f) {
        // y = w / n, n = ||w||_p:  dw_j = dy_j / n - (sum_i dy_i w_i) / n^2 * (w_j / n)^(p - 1)
        const float n = Elem<DT>::to_f32(Elem<DT>::from_f32(wave_pnorm(w, live, p)));
        const float dot = wave_sum(dy * w);
        const float dn = p == 1.f ? 1.f : (p == 2.f ? w / n : powf(w / n, p - 1.f));
        dw = dy / n - dot / (n * n) * dn;
      }
      for (int j = 0; j < top_k; ++j) {
        const int e = lane_value(my_i, j);
        const float v = lane_value(dw, j);
#pragma unroll
        for (int r = 0; r < R; ++r)
          if (lane + r * kWave == e) ds[r] += v;
      }
    }
    float dot = 0.f;
#pragma unroll
    for (int r = 0; r < R; ++r) dot += ds[r] * s[r];
    dot = wave_sum(dot);
    const float gl = grad_lse ? grad_lse[t] : 0.f;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int e = lane + r * kWave;
      if (e < num_experts) grad_logits[t * num_experts + e] = Elem<DT>::from_f32(s[r] * (ds[r] - dot + gl));
    }
  }
}

// out[t] = add[t] + grad_logits[t] @ weight, the input's gradient of the router's linear layer on top of the experts': fp32 sums, rounded
// once.  What bounds it: one reading of `add` and one writing of `out` (a product of its own and the addition read and write 2 1/2 times as much):
// 16384 x 1024 and 64 experts 17 us (4.1 TB/s; two passes 17.5 + 17.5), 24576 x 2048 and 16 experts 41 (4.9 TB/s; 36 + 45), 16384 x 768, 32: 12 (18.3 + 12.5).
// A wave has 64 columns and keeps their weights, all experts', in registers as operands (KT 16-byte pieces for each 16 columns); it then goes
// through tokens, two sixteens at a time so that eight 16-byte loads are under way.  An operand of 16 columns has every eighth group of four
// of 32: a lane's results of two products are eight columns in a row then, a 16-byte piece of its token's row of `add` and `out`.
// ALIGNED: experts % 8 == 0, rows of grad_logits are whole 16-byte pieces.  Where they are not, the rows with zeros up to whole pieces, which the
// kernels have in registers, can be written to `padded` on the way: the weight's gradient wants them like that (a fill and a strided copy of
// 10 us otherwise, 3001 tokens, 12 experts).
constexpr int kInputGradColumns = 64, kInputGradTokens = 32, kInputGradMaxExperts = 128, kInputGradBlocks = 512;
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
template <int DT>
__device__ __forceinline__ f32x4_t mfma_16x16x32(const u32x4_t& a, const u32x4_t& b, const f32x4_t& c) {
  typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
  typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
  if constexpr (DT == MBX_BF16) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  else return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}
template <int DT, int KT, bool ALIGNED>
__global__ void __launch_bounds__(kTokenThreads)
router_input_gradient_kernel(const uint16_t* __restrict__ grad_logits, const uint16_t* __restrict__ weight, const uint16_t* __restrict__ add,
                             int64_t tokens, int hidden, int num_experts, uint16_t* __restrict__ out, uint16_t* __restrict__ padded) {
  typedef typename Elem<DT>::type E;
  const int lane = lane_id(), row = lane % 16, group = lane / 16;
  const int c0 = ((int)blockIdx.x * kTokenWaves + (int)(threadIdx.x / kWave)) * kInputGradColumns;
  if (c0 >= hidden) return;
  // eight experts from `first` on of a row of n, past the last one zero
  const auto pack = [&](const uint16_t* p, int64_t step, int first) {
    uint32_t v[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = p[(first + q < num_experts ? first + q : num_experts - 1) * step];   // one load after the other, no branches
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = first + q < num_experts ? v[q] : 0u;
    return u32x4_t{v[0] | v[1] << 16, v[2] | v[3] << 16, v[4] | v[5] << 16, v[6] | v[7] << 16};
  };
  struct Rows { u32x4_t g[2][KT], v[2][2]; };
  const auto fetch = [&](int64_t t0, Rows& r) {
    auto& g = r.g;
    auto& v = r.v;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int64_t t = t0 + 16 * u + row;
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) {
        const int first = 32 * kt + 8 * group;
        if constexpr (ALIGNED) g[u][kt] = t < tokens && first < num_experts ? *(const u32x4_t*)(grad_logits + t * num_experts + first) : u32x4_t{0, 0, 0, 0};
        else g[u][kt] = t < tokens ? pack(grad_logits + t * num_experts, 1, first) : u32x4_t{0, 0, 0, 0};
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int column = c0 + 32 * i + 8 * group;
        v[u][i] = t < tokens && column < hidden ? *(const u32x4_t*)(add + t * hidden + column) : u32x4_t{0, 0, 0, 0};
      }
    }
  };
  int64_t t0 = (int64_t)blockIdx.y * kInputGradTokens;
  const int64_t step = (int64_t)gridDim.y * kInputGradTokens;
  Rows next;
  fetch(t0, next);
  u32x4_t w[2][2][KT];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int column = c0 + 32 * i + 8 * (row / 4) + 4 * half + row % 4;
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) w[i][half][kt] = pack(weight + (column < hidden ? column : 0), hidden, 32 * kt + 8 * group);
    }
  for (; t0 < tokens; t0 += step) {
    const Rows now = next;
    fetch(t0 + step, next);
    const auto& g = now.g;
    const auto& v = now.v;
    if constexpr (!ALIGNED) {
      if (padded != nullptr && c0 == 0) {
        const int pitch = (num_experts + 7) & ~7;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int kt = 0; kt < KT; ++kt) {
            const int64_t t = t0 + 16 * u + row;
            const int first = 32 * kt + 8 * group;
            if (t < tokens && first < pitch) *(u32x4_t*)(padded + t * pitch + first) = g[u][kt];
          }
      }
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int64_t t = t0 + 16 * u + row;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        f32x4_t acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
          for (int half = 0; half < 2; ++half) acc[half] = mfma_16x16x32<DT>(w[i][half][kt], g[u][kt], acc[half]);
        const int column = c0 + 32 * i + 8 * group;
        if (t >= tokens || column >= hidden) continue;
        u32x4_t r;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint32_t pair = v[u][i][q];
          const float low = Elem<DT>::to_f32(__builtin_bit_cast(E, (uint16_t)pair)) + acc[q / 2][2 * q % 4];
          const float high = Elem<DT>::to_f32(__builtin_bit_cast(E, (uint16_t)(pair >> 16))) + acc[q / 2][2 * q % 4 + 1];
          r[q] = (uint32_t)__builtin_bit_cast(uint16_t, Elem<DT>::from_f32(low)) | (uint32_t)__builtin_bit_cast(uint16_t, Elem<DT>::from_f32(high)) << 16;
        }
        *(u32x4_t*)(out + t * hidden + column) = r;
      }
    }
  }
}

// out[i] = sum over the parts, in fp32, rounded once.  A block takes 64 runs of four values; each of its four waves adds up a
// quarter of the parts, eight loads under way, and the first puts the quarters together, in order.  What bounds it: one reading of the
// parts (64 of 64 x 1024, 16.8 MB: 5 us; torch's sum of as many 16-bit values 9.9, and the cast of its result 4.8).
template <int DT>
__global__ void __launch_bounds__(kTokenThreads)
sum_parts_kernel(const float* __restrict__ parts, int num_parts, int64_t pitch, void* __restrict__ out_, int64_t n) {
  typedef typename Elem<DT>::type E;
  __shared__ f32x4_t sums[kTokenWaves][kWave];
  constexpr int kAhead = 8;
  const int lane = lane_id(), wave = threadIdx.x / kWave;
  const int64_t i = ((int64_t)blockIdx.x * kWave + lane) * 4;
  const int first = (int)((int64_t)wave * num_parts / kTokenWaves), last = (int)((int64_t)(wave + 1) * num_parts / kTokenWaves);
  f32x4_t sum = {0.f, 0.f, 0.f, 0.f};
  if (i + 4 <= n && (pitch & 3) == 0) {
    const f32x4_t* p = (const f32x4_t*)(parts + i);
    for (int q = first; q < last; q += kAhead) {
      f32x4_t v[kAhead];
#pragma unroll
      for (int u = 0; u < kAhead; ++u)
        if (q + u < last) v[u] = p[(int64_t)(q + u) * (pitch / 4)];
#pragma unroll
      for (int u = 0; u < kAhead; ++u)
        if (q + u < last) sum += v[u];
    }
  } else {
    for (int q = first; q < last; ++q)
#pragma unroll
      for (int t = 0; t < 4; ++t)
        if (i + t < n) sum[t] += parts[(int64_t)q * pitch + i + t];
  }
  sums[wave][lane] = sum;
  __syncthreads();
  if (wave != 0) return;
#pragma unroll
  for (int w = 1; w < kTokenWaves; ++w) sum += sums[w][lane];
#pragma unroll
  for (int t = 0; t < 4; ++t)
    if (i + t < n) ((E*)out_)[i + t] = Elem<DT>::from_f32(sum[t]);
}

// The sums of the auxiliary losses: values[i] counts[i % period] (the load-balancing loss: scores and tokens per expert), or without
// counts values[i]^2 (the z-loss), for all saved layers by one launch, a row of workgroups each.  A layer's sum of up to kLossOneBlock values is one
// workgroup's, a longer one is cut into runs of kLossRun for a workgroup each, whose sums a second launch adds in order.  What bounds the losses is the
// number of launches and the calls behind them: as torch's operations the two are ten of 1 - 7 us forward and ten backward for a layer, each with a node of
// its own (a step of 1024 tokens, 8 experts, the host in its slower mode: 825 us with them, 695 with these four); with a launch and a call for every layer
// the z-loss of 32 took 1400 us of the host's time each way together, with one for all 1105, torch's operations 2166 (a faster host 487, torch's
// 1602 - 1966; of 2 layers 134, torch's 177).
constexpr int kLossThreads = 1024, kLossOneBlock = 32 * kLossThreads, kLossRun = 8 * kLossThreads, kLossParts = 256, kLossLayers = 64;

// Of one launch, in its arguments: MOST is 1 or kLossLayers.  One layer has arguments of its own: with the 2.3 KB of those for many every launch of its step took
// longer on the host (1024 tokens, 8 experts, medians of 12 processes: forward of the layer 280.0 -> 276.6 us, each loss 1.2 less).
template <int MOST>
struct LossLayers {
  const void* values[MOST];
  const int32_t* counts[MOST];
  void* out[MOST];   // the gradients
  int64_t n[MOST];
  float scale[MOST];
};

__host__ __device__ constexpr int loss_blocks(int64_t n) {
  return n <= kLossOneBlock ? 1 : n > (int64_t)kLossParts * kLossRun ? kLossParts : (int)((n + kLossRun - 1) / kLossRun);
}

__device__ __forceinline__ float block_sum(float v) {   // in thread 0
  __shared__ float sums[kLossThreads / kWave];
  v = wave_sum(v);
  if (lane_id() == 0) sums[threadIdx.x / kWave] = v;
  __syncthreads();
  if (threadIdx.x >= kWave) return 0.f;
  return wave_sum(threadIdx.x < kLossThreads / kWave ? sums[threadIdx.x] : 0.f);
}

template <int DT, int MOST>
__global__ void __launch_bounds__(kLossThreads) loss_sum_kernel(const LossLayers<MOST> layers, int period, float* __restrict__ out, float* __restrict__ parts) {
  typedef typename Elem<DT>::type E;
  const int layer = blockIdx.y;
  const int64_t n = layers.n[layer];
  const int blocks = loss_blocks(n);
  if ((int)blockIdx.x >= blocks) return;
  const E* __restrict__ const values = (const E*)layers.values[layer];
  const int32_t* __restrict__ const counts = layers.counts[layer];
  const int64_t stride = (int64_t)blocks * kLossThreads;
  int64_t i = (int64_t)blockIdx.x * kLossThreads + threadIdx.x;
  int e = (int)(i % period);
  const int step = (int)(stride % period);
  float sum = 0.f;
#pragma unroll 8
  for (; i < n; i += stride) {
    const float v = Elem<DT>::to_f32(values[i]);
    sum += v * (counts ? (float)counts[e] : v);
    e += step;
    e = e >= period ? e - period : e;
  }
  sum = block_sum(sum);
  if (threadIdx.x != 0) return;
  if (blocks == 1) out[layer] = layers.scale[layer] * sum;
  else parts[layer * kLossParts + blockIdx.x] = sum;
}

template <int MOST>
__global__ void __launch_bounds__(kLossThreads) loss_parts_kernel(const LossLayers<MOST> layers, const float* __restrict__ parts, float* __restrict__ out) {
  const int layer = blockIdx.x, blocks = loss_blocks(layers.n[layer]);
  if (blocks == 1) return;
  const float sum = block_sum((int)threadIdx.x < blocks ? parts[layer * kLossParts + threadIdx.x] : 0.f);
  if (threadIdx.x == 0) out[layer] = layers.scale[layer] * sum;
}

// The sums' gradients: grad scale counts[i % period], or without counts grad scale 2 values[i].
template <int DT, int MOST>
__global__ void __launch_bounds__(256) loss_gradient_kernel(const float* __restrict__ grad, const LossLayers<MOST> layers, int period) {
  typedef typename Elem<DT>::type E;
  const int layer = blockIdx.y;
  E* __restrict__ const out = (E*)layers.out[layer];
  if (out == nullptr) return;
  const E* __restrict__ const values = (const E*)layers.values[layer];
  const int32_t* __restrict__ const counts = layers.counts[layer];
  const int64_t n = layers.n[layer];
  const float g = grad[layer] * layers.scale[layer];
  const int64_t stride = (int64_t)gridDim.x * 256;
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  int e = (int)(i % period);
  const int step = (int)(stride % period);
  for (; i < n; i += stride) {
    out[i] = Elem<DT>::from_f32(counts ? g * (float)counts[e] : g * (2.f * Elem<DT>::to_f32(values[i])));
    e += step;
    e = e >= period ? e - period : e;
  }
}

// A launch of up to MOST layers (two for long sums); parts: kLossParts floats a layer
template <int MOST>
static void launch_loss_sums(const void* const* values, int dtype, const int32_t* const* counts, const int64_t* n, const float* scales, int count, int period,
                             float* out, float* parts, hipStream_t s) {
  LossLayers<MOST> of = {};
  int blocks = 1;
  for (int l = 0; l < count; ++l) {
    of.values[l] = values[l];
    of.counts[l] = counts ? counts[l] : nullptr;
    of.n[l] = n[l];
    of.scale[l] = scales[l];
    blocks = loss_blocks(n[l]) > blocks ? loss_blocks(n[l]) : blocks;
  }
  const dim3 grid((unsigned)blocks, (unsigned)count);
  switch (dtype) {
    case MBX_BF16: loss_sum_kernel<MBX_BF16, MOST><<<grid, kLossThreads, 0, s>>>(of, period, out, parts); break;
    case MBX_F16: loss_sum_kernel<MBX_F16, MOST><<<grid, kLossThreads, 0, s>>>(of, period, out, parts); break;
    default: loss_sum_kernel<MBX_F32, MOST><<<grid, kLossThreads, 0, s>>>(of, period, out, parts); break;
  }
  if (blocks > 1) loss_parts_kernel<MOST><<<(unsigned)count, kLossThreads, 0, s>>>(of, parts, out);
}

template <int MOST>
static void launch_loss_gradients(const float* grad, const void* const* values, int dtype, const int32_t* const* counts, const int64_t* n, const float* scales,
                                  int count, int period, void* const* out, hipStream_t s) {
  LossLayers<MOST> of = {};
  int64_t most = 0;
  for (int l = 0; l < count; ++l) {
    of.values[l] = counts ? nullptr : values[l];
    of.counts[l] = counts ? counts[l] : nullptr;
    of.out[l] = out[l];
    of.n[l] = n[l];
    of.scale[l] = scales[l];
    if (out[l] && n[l] > most) most = n[l];
  }
  if (most == 0) return;
  const int64_t wanted = ceil_div(most, 256);
  const dim3 grid((unsigned)(wanted < 2048 ? wanted : 2048), (unsigned)count);
  switch (dtype) {
    case MBX_BF16: loss_gradient_kernel<MBX_BF16, MOST><<<grid, 256, 0, s>>>(grad, of, period); break;
    case MBX_F16: loss_gradient_kernel<MBX_F16, MOST><<<grid, 256, 0, s>>>(grad, of, period); break;
    default: loss_gradient_kernel<MBX_F32, MOST><<<grid, 256, 0, s>>>(grad, of, period); break;
  }
}

static inline unsigned token_grid(int64_t tokens) {
  int64_t blocks = ceil_div(tokens, kTokenWaves);
  if (blocks > 256 * 8) blocks = 256 * 8;
  return (unsigned)(blocks < 1 ? 1 : blocks);
}

#define MBX_ROUTER_DISPATCH(KERNEL, ...)                                                              \
  do {                                                                                                \
    const unsigned grid = token_grid(tokens);                                                         \
    const int per_lane = (num_experts + kWave - 1) / kWave;                                           \
    switch (dtype) {                                                                                  \
      case MBX_BF16:                                                                                  \
        if (per_lane <= 1) KERNEL<MBX_BF16, 1><<<grid, kTokenThreads, 0, s>>>(__VA_ARGS__);           \
        else if (per_lane <= 2) KERNEL<MBX_BF16, 2><<<grid, kTokenThreads, 0, s>>>(__VA_ARGS__);      \
        else if (per_lane <= 4) KERNEL<MBX_BF16, 4><<<grid, kTokenThreads, 0, s>>>(__VA_ARGS__);      \
        else KERNEL<MBX_BF16, 8><<<grid, kTokenThreads, 0, s>>>(__VA_ARGS__);                         \
        break;                                                                                        \
      case MBX_F16:                                                                                   \
        if (per_lane <= 1) KERNEL<MBX_F16, 1><<<grid, kTokenThreads, 0, s>>>(__VA_ARGS__);            \
        else if (per_lane <= 2) KERNEL<MBX_F16, 2><<<grid, kTokenThreads, 0, s>>>(__VA_ARGS__);       \
        else if (per_lane <= 4) KERNEL<MBX_F16, 4><<<grid, kTokenThreads, 0, s>>>(__VA_ARGS__);       \
        else KERNEL<MBX_F16, 8><<<grid, kTokenThreads, 0, s>>>(__VA_ARGS__);                          \
        break;                                                                                        \
      default:                                                                                        \
        if (per_lane <= 1) KERNEL<MBX_F32, 1><<<grid, kTokenThreads, 0, s>>>(__VA_ARGS__);            \
        else if (per_lane <= 2) KERNEL<MBX_F32, 2><<<grid, kTokenThreads, 0, s>>>(__VA_ARGS__);       \
        else if (per_lane <= 4) KERNEL<MBX_F32, 4><<<grid, kTokenThreads, 0, s>>>(__VA_ARGS__);       \
        else KERNEL<MBX_F32, 8><<<grid, kTokenThreads, 0, s>>>(__VA_ARGS__);                          \
        break;                                                                                        \
    }                                                                                                 \
  } while (0)

constexpr int kMaxRouterExperts = 8 * kWave;

}  // namespace
}  // namespace mbx

using namespace mbx;

extern "C" {

int mbx_router_forward(const void* logits, int dtype, int64_t tokens, int num_experts, int top_k, float norm_p,
                       void* scores, void* weights, int64_t* indices, int32_t* indices32, float* lse,
                       mbx_stream_t stream) {
  if (tokens < 0 || num_experts <= 0 || top_k <= 0 || top_k > num_experts || !(norm_p >= 0.f)) return MBX_EINVAL;
  if (dtype != MBX_BF16 && dtype != MBX_F16 && dtype != MBX_F32) return MBX_EINVAL;
  if (num_experts > kMaxRouterExperts || top_k > kWave) return MBX_EUNSUPPORTED;
  if (tokens == 0) return 0;
  if (!logits || !scores || !weights || !indices) return MBX_EINVAL;
  hipStream_t s = as_stream(stream);
  MBX_ROUTER_DISPATCH(router_forward_kernel, logits, tokens, num_experts, top_k, norm_p, scores, weights, indices, indices32, lse);
  return launch_status();
}

int mbx_router_linear_forward(const void* x, const void* weight, int dtype, int64_t tokens, int hidden, int num_experts, int top_k,
                              float norm_p, void* scores, void* weights, int64_t* indices, int32_t* indices32, mbx_stream_t stream) {
  if (tokens < 0 || hidden <= 0 || num_experts <= 0 || top_k <= 0 || top_k > num_experts || !(norm_p >= 0.f)) return MBX_EINVAL;
  if (dtype != MBX_BF16 && dtype != MBX_F16 && dtype != MBX_F32) return MBX_EINVAL;
  if (dtype == MBX_F32 || hidden % 8 || num_experts > kLinearMaxExperts || top_k > kWave || (int64_t)num_experts * hidden * 2 >= ((int64_t)1 << 30) ||
      tokens > 0x7fffffff || (((uintptr_t)x | (uintptr_t)weight) & 15u)) return MBX_EUNSUPPORTED;
  if (tokens == 0) return 0;
  if (!x || !weight || !scores || !weights || !indices) return MBX_EINVAL;
  hipStream_t s = as_stream(stream);
#define MBX_ROUTER_LINEAR(PER)                                                                                              \
  do {                                                                                                                      \
    if (dtype == MBX_BF16)                                                                                                  \
      router_linear_kernel<MBX_BF16, PER><<<(unsigned)tokens, kLinearWaves * kWave, 0, s>>>(                                \
          (const uint16_t*)x, (const uint16_t*)weight, hidden, num_experts, top_k, norm_p, scores, weights, indices, indices32); \
    else                                                                                                                    \
      router_linear_kernel<MBX_F16, PER><<<(unsigned)tokens, kLinearWaves * kWave, 0, s>>>(                                 \
          (const uint16_t*)x, (const uint16_t*)weight, hidden, num_experts, top_k, norm_p, scores, weights, indices, indices32); \
  } while (0)
  if (num_experts <= kLinearWaves) MBX_ROUTER_LINEAR(1);
  else if (num_experts <= 2 * kLinearWaves) MBX_ROUTER_LINEAR(2);
  else if (num_experts <= 4 * kLinearWaves) MBX_ROUTER_LINEAR(4);
  else MBX_ROUTER_LINEAR(8);
#undef MBX_ROUTER_LINEAR
  return launch_status();
}

int mbx_router_backward(const void* grad_weights, const void* grad_scores, const void* scores, const int64_t* indices,
                        int dtype, int64_t tokens, int num_experts, int top_k, float norm_p, void* grad_logits,
                        const float* grad_lse, mbx_stream_t stream) {
  if (tokens < 0 || num_experts <= 0 || top_k <= 0 || top_k > num_experts || !(norm_p >= 0.f)) return MBX_EINVAL;
  if (dtype != MBX_BF16 && dtype != MBX_F16 && dtype != MBX_F32) return MBX_EINVAL;
  if (num_experts > kMaxRouterExperts || top_k > kWave) return MBX_EUNSUPPORTED;
  if (tokens == 0) return 0;
  if (!scores || !grad_logits || (grad_weights && !indices)) return MBX_EINVAL;
  hipStream_t s = as_stream(stream);
  MBX_ROUTER_DISPATCH(router_backward_kernel, grad_weights, grad_scores, scores, indices, tokens, num_experts, top_k,
                      norm_p, grad_logits, grad_lse);
  return launch_status();
}

int mbx_router_input_gradient(const void* grad_logits, const void* weight, const void* add, int dtype, int64_t tokens, int hidden,
                              int num_experts, void* out, void* padded, mbx_stream_t stream) {
  if (tokens < 0 || hidden <= 0 || num_experts <= 0 || (dtype != MBX_BF16 && dtype != MBX_F16 && dtype != MBX_F32)) return MBX_EINVAL;
  if (tokens == 0) return 0;
  if (!grad_logits || !weight || !add || !out) return MBX_EINVAL;
  if (dtype == MBX_F32 || hidden % 8 || num_experts > kInputGradMaxExperts || (((uintptr_t)add | (uintptr_t)out | (uintptr_t)padded) & 15u)) return MBX_EUNSUPPORTED;
  hipStream_t s = as_stream(stream);
  const bool aligned = num_experts % 8 == 0 && ((uintptr_t)grad_logits & 15u) == 0 && !padded;
  // two waves to a SIMD where there are tokens for as many: each reads all experts' weights of its columns first (us with 256 / 512 / 1024 / 2048
  // workgroups: 16384 x 1024, 64 experts 17.8 / 17.1 / 19.0 / 22.7; 16384 x 768, 32 experts 14.6 / 12.2 / 12.7 / 13.0)
  const int64_t columns = ceil_div(hidden, kTokenWaves * kInputGradColumns), pieces = ceil_div(tokens, kInputGradTokens), most = ceil_div(kInputGradBlocks, columns);
  const dim3 grid((unsigned)columns, (unsigned)(pieces < most ? pieces : most));
#define MBX_INPUT_GRAD(DT, KT)                                                                                                                    \
  do {                                                                                                                                            \
    if (aligned) router_input_gradient_kernel<DT, KT, true><<<grid, kTokenThreads, 0, s>>>((const uint16_t*)grad_logits, (const uint16_t*)weight, \
                                                                                          (const uint16_t*)add, tokens, hidden, num_experts, (uint16_t*)out, (uint16_t*)nullptr); \
    else router_input_gradient_kernel<DT, KT, false><<<grid, kTokenThreads, 0, s>>>((const uint16_t*)grad_logits, (const uint16_t*)weight,        \
                                                                                   (const uint16_t*)add, tokens, hidden, num_experts, (uint16_t*)out, (uint16_t*)padded); \
  } while (0)
#define MBX_INPUT_GRAD_DT(DT)                        \
  do {                                               \
    if (num_experts <= 32) MBX_INPUT_GRAD(DT, 1);    \
    else if (num_experts <= 64) MBX_INPUT_GRAD(DT, 2); \
    else MBX_INPUT_GRAD(DT, 4);                      \
  } while (0)
  if (dtype == MBX_BF16) MBX_INPUT_GRAD_DT(MBX_BF16);
  else MBX_INPUT_GRAD_DT(MBX_F16);
#undef MBX_INPUT_GRAD_DT
#undef MBX_INPUT_GRAD
  return launch_status();
}

int mbx_sum_parts(const float* parts, int num_parts, int64_t pitch, void* out, int dtype, int64_t n, mbx_stream_t stream) {
  if (num_parts <= 0 || n < 0 || pitch < n) return MBX_EINVAL;
  if (dtype != MBX_BF16 && dtype != MBX_F16 && dtype != MBX_F32) return MBX_EINVAL;
  if (n == 0) return 0;
  if (!parts || !out || ((uintptr_t)parts & 15u)) return MBX_EINVAL;
  const int64_t blocks = ceil_div(n, 4 * kWave);
  if (blocks > 0x7fffffff) return MBX_ERANGE;
  hipStream_t s = as_stream(stream);
  if (dtype == MBX_BF16) sum_parts_kernel<MBX_BF16><<<(unsigned)blocks, kTokenThreads, 0, s>>>(parts, num_parts, pitch, out, n);
  else if (dtype == MBX_F16) sum_parts_kernel<MBX_F16><<<(unsigned)blocks, kTokenThreads, 0, s>>>(parts, num_parts, pitch, out, n);
  else sum_parts_kernel<MBX_F32><<<(unsigned)blocks, kTokenThreads, 0, s>>>(parts, num_parts, pitch, out, n);
  return launch_status();
}

size_t mbx_loss_sums_scratch_bytes(int64_t n, int layers) { return n > kLossOneBlock && layers > 0 ? (size_t)layers * kLossParts * sizeof(float) : 0; }

int mbx_loss_sums(const void* const* values, int dtype, const int32_t* const* counts, const int64_t* n, const float* scales, int layers,
                  int period, float* out, float* scratch, mbx_stream_t stream) {
  if (layers < 0 || period <= 0 || (dtype != MBX_BF16 && dtype != MBX_F16 && dtype != MBX_F32)) return MBX_EINVAL;
  if (layers == 0) return 0;
  if (!out || !values || !n || !scales) return MBX_EINVAL;
  for (int l = 0; l < layers; ++l) {
    if (n[l] < 0 || (n[l] > 0 && !values[l]) || (counts && n[l] > 0 && !counts[l])) return MBX_EINVAL;
    if (n[l] > kLossOneBlock && !scratch) return MBX_ESCRATCH;
  }
  if (layers == 1) launch_loss_sums<1>(values, dtype, counts, n, scales, 1, period, out, scratch, as_stream(stream));
  else
    for (int first = 0; first < layers; first += kLossLayers)
      launch_loss_sums<kLossLayers>(values + first, dtype, counts ? counts + first : nullptr, n + first, scales + first, layers - first < kLossLayers ? layers - first : kLossLayers,
                                    period, out + first, scratch ? scratch + (int64_t)first * kLossParts : nullptr, as_stream(stream));
  return launch_status();
}

int mbx_loss_gradients(const float* grad, const void* const* values, int dtype, const int32_t* const* counts, const int64_t* n, const float* scales,
                       int layers, int period, void* const* out, mbx_stream_t stream) {
  if (layers < 0 || period <= 0 || (dtype != MBX_BF16 && dtype != MBX_F16 && dtype != MBX_F32)) return MBX_EINVAL;
  if (layers == 0) return 0;
  if (!grad || !out || !n || !scales || (!counts && !values)) return MBX_EINVAL;
  for (int l = 0; l < layers; ++l)
    if (n[l] < 0 || (out[l] && n[l] > 0 && !(counts ? (const void*)counts[l] : values[l]))) return MBX_EINVAL;
  if (layers == 1) launch_loss_gradients<1>(grad, values, dtype, counts, n, scales, 1, period, out, as_stream(stream));
  else
    for (int first = 0; first < layers; first += kLossLayers)
      launch_loss_gradients<kLossLayers>(grad + first, values ? values + first : nullptr, dtype, counts ? counts + first : nullptr, n + first, scales + first,
                                         layers - first < kLossLayers ? layers - first : kLossLayers, period, out + first, as_stream(stream));
  return launch_status();
}

size_t mbx_loss_scratch_bytes(int64_t n) { return mbx_loss_sums_scratch_bytes(n, 1); }

int mbx_loss_sum(const void* values, int dtype, const int32_t* counts, int64_t n, int period, float scale, float* out, float* scratch,
                 mbx_stream_t stream) {
  return mbx_loss_sums(&values, dtype, counts ? &counts : nullptr, &n, &scale, 1, period, out, scratch, stream);
}

int mbx_loss_gradient(const float* grad, const void* values, int dtype, const int32_t* counts, int64_t n, int period, float scale, void* out,
                      mbx_stream_t stream) {
  if (n > 0 && !out) return MBX_EINVAL;
  return mbx_loss_gradients(grad, &values, dtype, counts ? &counts : nullptr, &n, &scale, 1, period, &out, stream);
}

}  // extern "C"
