// Fused log-prob + PG/GRPO loss over the 152k vocab:
// forward emits per-token log p(target) + the row LSE in a
// single online-logsumexp streaming pass (never materializing a (B,T,V)
// log-prob tensor — the reference loops rows through log_softmax+gather,
// distributed_actor.py:253-260); backward emits dlogits directly:
// dlogits_v = w * (1[v=target] - softmax_v), w = mask*coef*dloss.
#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>
#include "common.h"

namespace {

template <typename T>
DEV_INLINE float ld(const T* p, int64_t i);
template <> DEV_INLINE float ld<__hip_bfloat16>(const __hip_bfloat16* p, int64_t i) { return bf2f(p[i]); }
template <> DEV_INLINE float ld<float>(const float* p, int64_t i) { return p[i]; }

// Eight values at any element: rows of an odd vocabulary, or of a matrix that
// starts inside another, lie on 2 bytes. One 16-byte access all the same, which
// needs no alignment in device memory.
DEV_INLINE bf16x8 load8(const __hip_bfloat16* p) {
  bf16x8 v;
  __builtin_memcpy(&v, p, sizeof v);
  return v;
}
// Past the caches: what is written here is of the size of the logits.
DEV_INLINE void store8(__hip_bfloat16* p, const bf16x8& v) {
  typedef int Four __attribute__((ext_vector_type(4)));
  typedef Four Anywhere __attribute__((aligned(2)));
  Four q;
  __builtin_memcpy(&q, &v, sizeof q);
  __builtin_nontemporal_store(q, (Anywhere*)p);
}

// One workgroup per (b, t) row; single streaming pass, online logsumexp: a
// thread takes 32 values at a time, the next 32 on their way, compares their
// maximum with its own once and then sums exponentials without branches (value
// by value, with two branches and an equality test for the target each, vector
// work held it to 3.4 TB/s: 215 us for 2408 rows of 152064, 171 now; 512 and 1024
// threads a row are a quarter and half slower).
template <typename T>
__global__ __launch_bounds__(256)
void logprob_lse_kernel(const T* __restrict__ logits,
                        const int64_t* __restrict__ targets,
                        float* __restrict__ token_logp,
                        float* __restrict__ lse_out, int V) {
  constexpr float LOG2E = 1.4426950408889634f;
  constexpr bool BF16 = std::is_same<T, __hip_bfloat16>::value;
  __shared__ float red[16];
  const int64_t row = blockIdx.x;
  const T* lr = logits + row * V;

  float m = -1e30f, s = 0.f;     // s: sum of 2^((x - m) log2 e)
  auto take = [&](const float* x, int n) {
    float top = m;
    #pragma unroll
    for (int j = 0; j < n; ++j) top = fmaxf(top, x[j]);
    if (top > m) {
      s *= __builtin_amdgcn_exp2f((m - top) * LOG2E);
      m = top;
    }
    const float c = m * LOG2E;
    #pragma unroll
    for (int j = 0; j < n; ++j) s += __builtin_amdgcn_exp2f(x[j] * LOG2E - c);
  };
  int done = 0;
  if constexpr (BF16) {
    const int nvec = V / 8;
    int i = threadIdx.x;
    if (i + 3 * 256 < nvec) {
      bf16x8 v[4], next[4];
      auto load = [&](int at) {
        #pragma unroll
        for (int k = 0; k < 4; ++k) next[k] = load8(lr + min(at + k * 256, nvec - 1) * 8);
      };
      load(i);
      for (; i + 3 * 256 < nvec; i += 1024) {
        #pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = next[k];
        load(i + 1024);                 // past the end the last again
        float x[32];
        #pragma unroll
        for (int k = 0; k < 4; ++k)
          #pragma unroll
          for (int j = 0; j < 8; ++j) x[8 * k + j] = bf2f(v[k].v[j]);
        take(x, 32);
      }
    }
    for (; i < nvec; i += 256) {
      const bf16x8 v = load8(lr + i * 8);
      float x[8];
      #pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = bf2f(v.v[j]);
      take(x, 8);
    }
    done = nvec * 8;
  }
  for (int i = done + threadIdx.x; i < V; i += 256) {
    const float x = ld(lr, i);
    take(&x, 1);
  }
  // combine per-thread (m, s): M = max m; S = sum s_i * exp(m_i - M)
  const float M = block_max(m, red);
  const float S = block_sum(s * __builtin_amdgcn_exp2f((m - M) * LOG2E), red);
  if (threadIdx.x == 0) {
    const float lse = M + __logf(S);
    const int64_t tgt = targets[row];
    lse_out[row] = lse;
    token_logp[row] = (tgt >= 0 && tgt < V ? ld(lr, tgt) : 0.f) - lse;
  }
}

// Row weights and the loss itself: w[b, t] = mask * coef_b with
// coef_b = -reward_b / max(sum mask, 1) / B * scale, loss = sum w * token_logp.
// One wave a sequence and turn.
template <typename M>
__global__ __launch_bounds__(1024)
void loss_reduce_kernel(const float* __restrict__ token_logp, const M* __restrict__ mask,
                        const float* __restrict__ rewards, float* __restrict__ w,
                        float* __restrict__ loss, int B, int T, float scale) {
  __shared__ float part[16];
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x & (WAVE - 1);
  float total = 0.f;
  for (int b = wave; b < B; b += 16) {
    const int64_t at = (int64_t)b * T;
    float n = 0.f, sum = 0.f;
    for (int t = lane; t < T; t += WAVE) {
      const float k = (float)mask[at + t];
      n += k;
      sum += token_logp[at + t] * k;
    }
    const float coef = -rewards[b] / fmaxf(wave_sum(n), 1.f) / B * scale;
    for (int t = lane; t < T; t += WAVE) w[at + t] = (float)mask[at + t] * coef;
    total += wave_sum(sum) * coef;
  }
  if (lane == 0) part[wave] = total;
  __syncthreads();
  if (threadIdx.x == 0) {
    float sum = 0.f;
    for (int i = 0; i < 16; ++i) sum += part[i];
    *loss = sum;
  }
}

// sum of w * token_logp over rows, in an order of its own for every row count
__global__ __launch_bounds__(1024)
void loss_rows_kernel(const float* __restrict__ token_logp, const float* __restrict__ w,
                      float* __restrict__ loss, int64_t rows) {
  __shared__ float red[16];
  float sum = 0.f;
  for (int64_t i = threadIdx.x; i < rows; i += 1024) sum += w[i] * token_logp[i];
  sum = block_sum(sum, red);
  if (threadIdx.x == 0) *loss = sum;
}

// Memory alone: rows are read and written once, four loads of a thread in flight. The
// gradient goes past the caches (written through them it drove out the logits before
// they were read, and waited for room: 2408 rows of 152064, a quarter of them of weight
// zero and only written, 440 -> 268 us, 600 rows 127 -> 55). The rows run from the last,
// whose logits the forward pass read last: both passes 401 -> 375 us, with THREADS 1024
// for rows that give each four loads at least (32768 values: 242 and 242 us for 8000
// rows) 345.
template <typename T, int THREADS>
__global__ __launch_bounds__(THREADS)
void loss_bwd_kernel(const T* __restrict__ logits,
                     const int64_t* __restrict__ targets,
                     const float* __restrict__ w,
                     const float* __restrict__ lse,
                     const float* __restrict__ dloss,   // scalar, or null: 1
                     T* __restrict__ dlogits, int V) {
  const int64_t row = gridDim.x - 1 - blockIdx.x;
  const T* lr = logits + row * V;
  T* dr = dlogits + row * V;
  const float wv = dloss ? w[row] * *dloss : w[row];
  const float l = lse[row];
  const int64_t tgt = targets[row];
  if constexpr (std::is_same<T, __hip_bfloat16>::value) {
    const int nvec = V / 8;
    auto put = [&](int i, const bf16x8& v) {
      bf16x8 o;
      #pragma unroll
      for (int j = 0; j < 8; ++j) {
        float p = __expf(bf2f(v.v[j]) - l);
        o.v[j] = f2bf(wv * ((i * 8 + j == (int)tgt ? 1.f : 0.f) - p));
      }
      store8(dr + i * 8, o);
    };
    if (wv == 0.f) {
      bf16x8 o;
      #pragma unroll
      for (int j = 0; j < 8; ++j) o.v[j] = f2bf(0.f);
      for (int i = threadIdx.x; i < nvec; i += THREADS) store8(dr + i * 8, o);
    } else {
      int i = threadIdx.x;
      for (; i + 3 * THREADS < nvec; i += 4 * THREADS) {
        bf16x8 v[4];
        #pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = load8(lr + (i + k * THREADS) * 8);
        #pragma unroll
        for (int k = 0; k < 4; ++k) put(i + k * THREADS, v[k]);
      }
      for (; i < nvec; i += THREADS) put(i, load8(lr + i * 8));
    }
    for (int i = nvec * 8 + threadIdx.x; i < V; i += blockDim.x) {
      float g = 0.f;
      if (wv != 0.f)
        g = wv * ((i == (int)tgt ? 1.f : 0.f) - __expf(ld(lr, i) - l));
      dr[i] = f2bf(g);
    }
    return;
  }
  if (wv == 0.f) {
    for (int i = threadIdx.x; i < V; i += blockDim.x)
      dr[i] = (T)(0.f);
    return;
  }
  for (int i = threadIdx.x; i < V; i += blockDim.x) {
    float p = __expf(ld(lr, i) - l);
    float g = wv * ((i == tgt ? 1.f : 0.f) - p);
    dr[i] = g;
  }
}

}  // namespace

std::vector<torch::Tensor> logprob_lse_fwd(torch::Tensor logits,
                                           torch::Tensor targets) {
  TORCH_CHECK(logits.is_cuda() && logits.is_contiguous());
  TORCH_CHECK(targets.scalar_type() == at::kLong);
  const int V = logits.size(-1);
  const int64_t rows = logits.numel() / V;
  auto sizes = logits.sizes().vec();
  sizes.pop_back();
  auto opts = logits.options().dtype(at::kFloat);
  auto token_logp = torch::empty(sizes, opts);
  auto lse = torch::empty(sizes, opts);
  if (rows == 0) return {token_logp, lse};
  dim3 grid(rows), block(256);
  auto stream = at::cuda::getCurrentCUDAStream();
  if (logits.scalar_type() == at::kBFloat16) {
    hipLaunchKernelGGL(logprob_lse_kernel<__hip_bfloat16>, grid, block, 0, stream,
                       reinterpret_cast<const __hip_bfloat16*>(logits.data_ptr()),
                       targets.contiguous().data_ptr<int64_t>(),
                       token_logp.data_ptr<float>(), lse.data_ptr<float>(), V);
  } else {
    TORCH_CHECK(logits.scalar_type() == at::kFloat);
    hipLaunchKernelGGL(logprob_lse_kernel<float>, grid, block, 0, stream,
                       logits.data_ptr<float>(),
                       targets.contiguous().data_ptr<int64_t>(),
                       token_logp.data_ptr<float>(), lse.data_ptr<float>(), V);
  }
  HIP_CHECK_LAST();
  return {token_logp, lse};
}

// The masked PG/GRPO loss of logits (B, T, V): {loss, row weights (B, T), lse}.
// mask int64 or fp32, rewards fp32.
static std::vector<torch::Tensor> logprob_loss_fwd(torch::Tensor logits, torch::Tensor targets,
                                                   torch::Tensor mask, torch::Tensor rewards,
                                                   double scale) {
  TORCH_CHECK(logits.dim() == 3 && mask.is_cuda() && rewards.is_cuda());
  const int B = logits.size(0), T = logits.size(1);
  TORCH_CHECK(mask.numel() == (int64_t)B * T && targets.numel() == (int64_t)B * T &&
              rewards.numel() == B, "logprob_loss: shape mismatch");
  TORCH_CHECK(mask.is_contiguous() && rewards.is_contiguous() &&
              rewards.scalar_type() == at::kFloat);
  auto lp = logprob_lse_fwd(logits, targets);
  auto w = torch::empty_like(lp[0]);
  auto loss = torch::empty({}, lp[0].options());
  auto stream = at::cuda::getCurrentCUDAStream();
  #define REDUCE(M)                                                                   \
    hipLaunchKernelGGL(loss_reduce_kernel<M>, dim3(1), dim3(1024), 0, stream,         \
                       lp[0].data_ptr<float>(), mask.data_ptr<M>(),                   \
                       rewards.data_ptr<float>(), w.data_ptr<float>(),                \
                       loss.data_ptr<float>(), B, T, (float)scale)
  if (mask.scalar_type() == at::kLong) REDUCE(int64_t);
  else { TORCH_CHECK(mask.scalar_type() == at::kFloat); REDUCE(float); }
  #undef REDUCE
  HIP_CHECK_LAST();
  return {loss, w, lp[1]};
}

torch::Tensor logprob_loss_bwd(torch::Tensor logits, torch::Tensor targets,
                               torch::Tensor w, torch::Tensor lse,
                               c10::optional<torch::Tensor> dloss) {
  TORCH_CHECK(logits.is_cuda() && logits.is_contiguous());
  const float* dl = nullptr;
  if (dloss) {
    TORCH_CHECK(dloss->is_cuda() && dloss->numel() == 1 && dloss->scalar_type() == at::kFloat);
    dl = dloss->data_ptr<float>();
  }
  const int V = logits.size(-1);
  const int64_t rows = logits.numel() / V;
  auto dlogits = torch::empty_like(logits);
  if (rows == 0) return dlogits;
  auto stream = at::cuda::getCurrentCUDAStream();
  auto wc = w.contiguous();
  auto lsec = lse.contiguous();
  auto tc = targets.contiguous();
  #define BWD(T, THREADS)                                                              \
    hipLaunchKernelGGL((loss_bwd_kernel<T, THREADS>), dim3(rows), dim3(THREADS), 0,    \
                       stream, reinterpret_cast<const T*>(logits.data_ptr()),          \
                       tc.data_ptr<int64_t>(), wc.data_ptr<float>(),                   \
                       lsec.data_ptr<float>(), dl,                                     \
                       reinterpret_cast<T*>(dlogits.data_ptr()), V)
  if (logits.scalar_type() != at::kBFloat16) BWD(float, 256);
  else if (V / 8 >= 4 * 1024) BWD(__hip_bfloat16, 1024);
  else BWD(__hip_bfloat16, 256);
  #undef BWD
  HIP_CHECK_LAST();
  return dlogits;
}

// The differentiable loss: a node of the C++ engine.
namespace {

struct LogprobLoss : public torch::autograd::Function<LogprobLoss> {
  static torch::Tensor forward(torch::autograd::AutogradContext* ctx, torch::Tensor logits,
                               torch::Tensor targets, torch::Tensor mask, torch::Tensor rewards,
                               double scale) {
    logits = logits.contiguous();
    targets = targets.contiguous();
    // int64 masks are read as they are
    auto m = mask.scalar_type() == at::kLong ? mask : mask.to(at::kFloat);
    auto r = logprob_loss_fwd(logits, targets, m.contiguous(),
                              rewards.to(at::kFloat).contiguous(), scale);
    ctx->save_for_backward({logits, targets, r[1], r[2]});
    return r[0];
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    const auto s = ctx->get_saved_variables();
    auto d = logprob_loss_bwd(s[0], s[1], s[2], s[3], grads[0].to(at::kFloat));
    return {d, torch::Tensor(), torch::Tensor(), torch::Tensor(), torch::Tensor()};
  }
};

}  // namespace

torch::Tensor logprob_loss(torch::Tensor logits, torch::Tensor targets, torch::Tensor mask,
                           torch::Tensor rewards, double scale) {
  return LogprobLoss::apply(logits, targets, mask, rewards, scale);
}

// The same sum for rows that carry weights of their own: sum_i w_i log p(target_i)
// of logits (rows, V); no gradient for the weights.
namespace {

struct LogprobRows : public torch::autograd::Function<LogprobRows> {
  static torch::Tensor forward(torch::autograd::AutogradContext* ctx, torch::Tensor logits,
                               torch::Tensor targets, torch::Tensor w) {
    TORCH_CHECK(logits.dim() == 2 && targets.is_cuda() && w.is_cuda() &&
                targets.numel() == logits.size(0) && w.numel() == logits.size(0) &&
                w.scalar_type() == at::kFloat, "logprob_rows: shape mismatch");
    logits = logits.contiguous();
    targets = targets.contiguous();
    w = w.contiguous();
    auto lp = logprob_lse_fwd(logits, targets);
    auto loss = torch::empty({}, lp[0].options());
    hipLaunchKernelGGL(loss_rows_kernel, dim3(1), dim3(1024), 0, at::cuda::getCurrentCUDAStream(),
                       lp[0].data_ptr<float>(), w.data_ptr<float>(), loss.data_ptr<float>(),
                       logits.size(0));
    HIP_CHECK_LAST();
    ctx->save_for_backward({logits, targets, w, lp[1]});
    return loss;
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    const auto s = ctx->get_saved_variables();
    auto d = logprob_loss_bwd(s[0], s[1], s[2], s[3], grads[0].to(at::kFloat));
    return {d, torch::Tensor(), torch::Tensor()};
  }
};

}  // namespace

torch::Tensor logprob_rows(torch::Tensor logits, torch::Tensor targets, torch::Tensor w) {
  return LogprobRows::apply(logits, targets, w);
}
