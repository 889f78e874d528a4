// Fused AdamW over flat fp32 spans: param, grad and both moments are read once and param and both moments written once
// (28 B per element with fp32 grads; amsgrad adds the running maximum of the second moment, 8 B more).
#include "mfsdp_common.h"

#include <algorithm>
#include <cmath>

namespace mfsdp {
namespace {

// Four elements as one access.  Parameters, gradients and moments start at any element of a flat shard: the accesses are
// aligned to an element only (global memory takes that at full vector width).
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef f32x4 f32x4_a4 __attribute__((aligned(4)));
typedef u32x2 u32x2_a2 __attribute__((aligned(2)));

struct AdamWArgs {
  float decay;       // 1 - lr * weight_decay
  float beta1;
  float one_minus_beta1;
  float beta2;
  float one_minus_beta2;
  float eps;
  float grad_sign;   // -1 with maximize, else +1
};

// One span of a launch; the step count, and with it the bias corrections, may differ from span to span.
struct Span {
  float* param;
  const void* grad;
  float* exp_avg;
  float* exp_avg_sq;
  float* max_exp_avg_sq;
  int64_t numel;
  float neg_step_size;  // -lr / (1 - beta1^t)
  float bc2_sqrt;       // sqrt(1 - beta2^t)
};

constexpr int kMaxSpans = 56;  // of one launch: its kernel arguments carry the table

// Kernel arguments of up to N spans: one, whose fields then need no lookup, a few or many, because 4 KiB of arguments make a
// launch 1.2 us longer than a few hundred bytes (3.7 against 2.5 us for an empty kernel), which is most of a small update.
template <int N>
struct SpanTable {
  uint32_t begin[N];  // first workgroup of a span; entries past the last span are beyond every workgroup
  AdamWArgs a;
  Span span[N];
};
static_assert(sizeof(SpanTable<kMaxSpans>) <= 4096, "kernel arguments are limited to 4 KiB");

// Tensor.lerp as ATen evaluates it.
__device__ __forceinline__ float lerp_aten(float start, float end, float weight) {
  // one fused multiply-add from the nearer end point, the form ATen's vectorised kernel spells out
  // (fmadd(weight, end - start, start) / fmadd(weight - 1, end - start, end)); written explicitly so that the
  // compiler's contraction choices cannot differ between code paths
  const float diff = end - start;
  return fabsf(weight) < 0.5f ? __builtin_fmaf(weight, diff, start) : __builtin_fmaf(weight - 1.0f, diff, end);
}

// The operation order of the single-tensor path of torch.optim.AdamW:
//   g = -g (maximize);  p *= 1 - lr*wd;  m += (g - m)*(1 - b1);  v = v*b2 + (1 - b2)*g*g;
//   vmax = max(vmax, v) (amsgrad);  p += (-step_size * m) / (sqrt(amsgrad ? vmax : v)/sqrt(bc2) + eps)
// No multiply-add contraction: every operation rounds on its own, so an element gets the same bits whether it is
// updated in the vector body or in the scalar tail, alone, as part of a merged span or beside others.
template <bool AMSGRAD>
__device__ __forceinline__ void adamw_one(float& p, float g, float& m, float& v, float& vmax, const AdamWArgs& a, float neg_step_size, float bc2_sqrt) {
#pragma clang fp contract(off)
  g = g * a.grad_sign;
  p = p * a.decay;
  m = lerp_aten(m, g, a.one_minus_beta1);
  v = v * a.beta2 + (a.one_minus_beta2 * g) * g;
  float second = v;
  if constexpr (AMSGRAD) {
    vmax = (vmax != vmax || v != v) ? __builtin_nanf("") : fmaxf(vmax, v);  // torch.maximum propagates NaN
    second = vmax;
  }
  const float denom = sqrtf(second) / bc2_sqrt + a.eps;  // sqrtf is correctly rounded; __fsqrt_rn is the fast native one here
  p = p + (neg_step_size * m) / denom;
}

constexpr int kThreads = 64;     // one wavefront per workgroup
constexpr int kVectors = 2;      // groups of four elements per thread, all of their loads issued before the first use
constexpr int64_t kPerBlock = kThreads * kVectors * 4;

template <typename T, typename P>
__device__ __forceinline__ T load_once(const P* p) { return __builtin_nontemporal_load(reinterpret_cast<const T*>(p)); }
template <typename T, typename P, typename V>
__device__ __forceinline__ void store_once(P* p, V v) { __builtin_nontemporal_store(v, reinterpret_cast<T*>(p)); }

// All spans of a step in one launch.  Bound by memory.  Non-temporal accesses (every byte is touched once) and one small
// workgroup per block of each stream rather than a persistent grid: workgroups are dispatched in order, so the ones running
// at any moment sweep neighbouring addresses of all seven streams, and the finer the workgroups the more evenly loads and
// stores mix.  One span of 41 M elements: one wavefront per workgroup with two vectors per thread 6.22 TB/s (one vector
// 5.55, four 6.01; 256 threads with four vectors 5.93, with two 5.94; 16 persistent workgroups per CU 5.71); 5.1-5.5 TB/s
// with cached loads or stores.  One launch
// for all spans of a step: 15 parameters of 1000 to 6.1 M elements (8.2 M in all) take 127 us of host and device time a
// step against 293 us with a launch each.
template <bool GRAD_BF16, bool AMSGRAD, int N>
__global__ void __launch_bounds__(kThreads)
adamw_kernel(SpanTable<N> table) {
  int index = 0;
  if constexpr (N > 1) {
    // the whole table of begins is one scalar load, then compares
#pragma unroll
    for (int i = 1; i < N; ++i) index += blockIdx.x >= table.begin[i] ? 1 : 0;
  }
  const Span& s = table.span[index];
  const AdamWArgs& a = table.a;
  const uint32_t block = N > 1 ? blockIdx.x - table.begin[index] : blockIdx.x;
  float* __restrict__ param = s.param;
  float* __restrict__ exp_avg = s.exp_avg;
  float* __restrict__ exp_avg_sq = s.exp_avg_sq;
  float* __restrict__ max_exp_avg_sq = s.max_exp_avg_sq;
  const uint16_t* __restrict__ grad16 = static_cast<const uint16_t*>(s.grad);
  const float* __restrict__ grad32 = static_cast<const float*>(s.grad);
  const int64_t first = static_cast<int64_t>(block) * kPerBlock + threadIdx.x * 4;
  f32x4 p[kVectors], m[kVectors], v[kVectors], g[kVectors], vmax[kVectors];
#pragma unroll
  for (int u = 0; u < kVectors; ++u) {
    const int64_t i = first + u * kThreads * 4;
    if (i + 4 <= s.numel) {
      p[u] = load_once<f32x4_a4>(param + i);
      m[u] = load_once<f32x4_a4>(exp_avg + i);
      v[u] = load_once<f32x4_a4>(exp_avg_sq + i);
      if constexpr (AMSGRAD) vmax[u] = load_once<f32x4_a4>(max_exp_avg_sq + i);
      if constexpr (GRAD_BF16) {
        const u32x2 raw = load_once<u32x2_a2>(grad16 + i);
        g[u].x = __uint_as_float(raw.x << 16);
        g[u].y = __uint_as_float(raw.x & 0xffff0000u);
        g[u].z = __uint_as_float(raw.y << 16);
        g[u].w = __uint_as_float(raw.y & 0xffff0000u);
      } else {
        g[u] = load_once<f32x4_a4>(grad32 + i);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  // Wait for all of them (vmcnt(0)): arithmetic that starts on the first group while the second is on its way, and its stores
  // between the loads of others, is slower (41 M elements: 184.2 to 185.7 us in any order tried, 182.6 us so).
  __builtin_amdgcn_s_waitcnt(0x0f70);
#pragma unroll
  for (int u = 0; u < kVectors; ++u) {
    const int64_t i = first + u * kThreads * 4;
    if (i + 4 <= s.numel) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        float pk = p[u][k], mk = m[u][k], vk = v[u][k], xk = 0.0f;
        if constexpr (AMSGRAD) xk = vmax[u][k];
        adamw_one<AMSGRAD>(pk, g[u][k], mk, vk, xk, a, s.neg_step_size, s.bc2_sqrt);
        p[u][k] = pk; m[u][k] = mk; v[u][k] = vk;
        if constexpr (AMSGRAD) vmax[u][k] = xk;
      }
      __builtin_amdgcn_sched_barrier(0);
      store_once<f32x4_a4>(param + i, p[u]);
      store_once<f32x4_a4>(exp_avg + i, m[u]);
      store_once<f32x4_a4>(exp_avg_sq + i, v[u]);
      if constexpr (AMSGRAD) store_once<f32x4_a4>(max_exp_avg_sq + i, vmax[u]);
    } else {
      for (int64_t j = i; j < s.numel; ++j) {  // the span's last group: one to three elements, at most one thread's
        float pk = param[j], mk = exp_avg[j], vk = exp_avg_sq[j], xk = 0.0f, gk;
        if constexpr (GRAD_BF16) gk = __uint_as_float(static_cast<uint32_t>(grad16[j]) << 16);
        else gk = grad32[j];
        if constexpr (AMSGRAD) xk = max_exp_avg_sq[j];
        adamw_one<AMSGRAD>(pk, gk, mk, vk, xk, a, s.neg_step_size, s.bc2_sqrt);
        param[j] = pk; exp_avg[j] = mk; exp_avg_sq[j] = vk;
        if constexpr (AMSGRAD) max_exp_avg_sq[j] = xk;
      }
    }
  }
}

int check_span(const mfsdp_adamw_span& s) {
  if (s.numel < 0) return fail(MFSDP_ERR_INVALID, "numel must be non-negative");
  if (s.step < 1) return fail(MFSDP_ERR_INVALID, "step must be >= 1, got %lld", static_cast<long long>(s.step));
  if (s.grad_dtype != MFSDP_F32 && s.grad_dtype != MFSDP_BF16) return fail(MFSDP_ERR_INVALID, "grad_dtype must be f32 or bf16");
  if (s.numel == 0) return MFSDP_OK;
  if (!s.param || !s.grad || !s.exp_avg || !s.exp_avg_sq) return fail(MFSDP_ERR_INVALID, "null tensor pointer");
  if (s.numel / kPerBlock >= INT32_MAX) return fail(MFSDP_ERR_UNSUPPORTED, "spans of more than 2^40 elements");
  return MFSDP_OK;
}

template <int N>
int launch(const mfsdp_adamw_span* const* spans, int n, const AdamWArgs& a, double lr, double beta1, double beta2, hipStream_t stream) {
  SpanTable<N> table;
  table.a = a;
  uint32_t blocks = 0;
  int64_t step = 0;
  float neg_step_size = 0.0f, bc2_sqrt = 0.0f;
  for (int i = 0; i < n; ++i) {
    const mfsdp_adamw_span& s = *spans[i];
    if (s.step != step) {
      // every scalar is computed in double from the hyper-parameters as given, as Python does, and rounded to fp32 once
      // (1 - beta2 formed from an fp32 beta2 = 0.999 would already be off by 1.3e-5)
      step = s.step;
      neg_step_size = static_cast<float>(-lr / (1.0 - std::pow(beta1, static_cast<double>(step))));
      bc2_sqrt = static_cast<float>(std::sqrt(1.0 - std::pow(beta2, static_cast<double>(step))));
    }
    table.begin[i] = blocks;
    table.span[i] = Span{s.param, s.grad, s.exp_avg, s.exp_avg_sq, s.max_exp_avg_sq, s.numel, neg_step_size, bc2_sqrt};
    blocks += static_cast<uint32_t>((s.numel + kPerBlock - 1) / kPerBlock);
  }
  for (int i = n; i < N; ++i) table.begin[i] = UINT32_MAX;
  const dim3 grid(blocks), threads(kThreads);
  const bool bf16 = spans[0]->grad_dtype == MFSDP_BF16;
  if (spans[0]->max_exp_avg_sq != nullptr) {
    if (bf16) hipLaunchKernelGGL((adamw_kernel<true, true, N>), grid, threads, 0, stream, table);
    else hipLaunchKernelGGL((adamw_kernel<false, true, N>), grid, threads, 0, stream, table);
  } else {
    if (bf16) hipLaunchKernelGGL((adamw_kernel<true, false, N>), grid, threads, 0, stream, table);
    else hipLaunchKernelGGL((adamw_kernel<false, false, N>), grid, threads, 0, stream, table);
  }
  MFSDP_CHECK_LAUNCH("adamw_kernel");
  return MFSDP_OK;
}

// Consecutive spans with one gradient type and one amsgrad setting share a launch; spans whose parameters overlap keep
// launches of their own, in the order given.
int run_spans(int64_t n, const mfsdp_adamw_span* spans, double lr, double beta1, double beta2, double eps, double weight_decay,
              int maximize, hipStream_t stream) {
  for (int64_t i = 0; i < n; ++i)  // everything that can be refused is refused before the first launch
    if (int rc = check_span(spans[i])) return rc;
  AdamWArgs a;
  a.decay = static_cast<float>(1.0 - lr * weight_decay);
  a.beta1 = static_cast<float>(beta1);
  a.one_minus_beta1 = static_cast<float>(1.0 - beta1);
  a.beta2 = static_cast<float>(beta2);
  a.one_minus_beta2 = static_cast<float>(1.0 - beta2);
  a.eps = static_cast<float>(eps);
  a.grad_sign = maximize ? -1.0f : 1.0f;
  for (int64_t next = 0; next < n;) {
    const mfsdp_adamw_span* batch[kMaxSpans];
    int count = 0;
    int64_t blocks = 0;
    uintptr_t low = 0, high = 0;  // the addresses the launch's parameters span, gaps included
    for (; next < n && count < kMaxSpans; ++next) {
      const mfsdp_adamw_span& s = spans[next];
      if (s.numel == 0) continue;
      const uintptr_t start = reinterpret_cast<uintptr_t>(s.param), stop = start + static_cast<uintptr_t>(s.numel) * 4;
      const int64_t more = (s.numel + kPerBlock - 1) / kPerBlock;
      if (count > 0 && (s.grad_dtype != batch[0]->grad_dtype || (s.max_exp_avg_sq != nullptr) != (batch[0]->max_exp_avg_sq != nullptr) ||
                        (start < high && stop > low) || blocks + more > INT32_MAX))
        break;
      low = count > 0 ? std::min(low, start) : start;
      high = std::max(high, stop);
      blocks += more;
      batch[count++] = &s;
    }
    if (count == 0) continue;
    const auto launch_for = count == 1 ? launch<1> : count <= 8 ? launch<8> : launch<kMaxSpans>;
    if (int rc = launch_for(batch, count, a, lr, beta1, beta2, stream)) return rc;
  }
  return MFSDP_OK;
}

}  // namespace
}  // namespace mfsdp

using namespace mfsdp;

extern "C" int mfsdp_adamw_step_many(int64_t n, const mfsdp_adamw_span* spans, double lr, double beta1, double beta2, double eps,
                                     double weight_decay, int maximize, void* stream) {
  if (n < 0 || (n > 0 && spans == nullptr)) return fail(MFSDP_ERR_INVALID, "spans is null or n negative");
  return run_spans(n, spans, lr, beta1, beta2, eps, weight_decay, maximize, as_stream(stream));
}

extern "C" int mfsdp_adamw_step_ex(float* param, const void* grad, int grad_dtype, float* exp_avg, float* exp_avg_sq,
                                   float* max_exp_avg_sq, int64_t numel, int64_t step, double lr, double beta1,
                                   double beta2, double eps, double weight_decay, int maximize, void* stream) {
  const mfsdp_adamw_span span{param, grad, exp_avg, exp_avg_sq, max_exp_avg_sq, numel, step, grad_dtype};
  return run_spans(1, &span, lr, beta1, beta2, eps, weight_decay, maximize, as_stream(stream));
}

extern "C" int mfsdp_adamw_step(float* param, const void* grad, int grad_dtype, float* exp_avg, float* exp_avg_sq,
                                int64_t numel, int64_t step, double lr, double beta1, double beta2, double eps,
                                double weight_decay, void* stream) {
  return mfsdp_adamw_step_ex(param, grad, grad_dtype, exp_avg, exp_avg_sq, nullptr, numel, step, lr, beta1, beta2, eps,
                             weight_decay, 0, stream);
}
