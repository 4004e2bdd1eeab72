// RMSNorm forward + backward (dx only — norm weights are frozen in this
// framework: only LoRA trains). Replaces the fused RMSNorm the reference
// gets from vLLM/Unsloth.
//
// Memory-bound: explicit bf16x8 (16 B/lane) vector loads — hipcc does not
// auto-vectorize scalar bf16 loads (guide G13) — fp32 accumulation, one
// block per row, wave64 + LDS reduction.
#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>
#include "common.h"

namespace {

__global__ void rmsnorm_fwd_bf16(const __hip_bfloat16* __restrict__ x,
                                 const __hip_bfloat16* __restrict__ w,
                                 __hip_bfloat16* __restrict__ y,
                                 int hidden, int64_t ldy, float eps) {
  __shared__ float red[16];
  const int64_t row = blockIdx.x;
  const bf16x8* xr = reinterpret_cast<const bf16x8*>(x + row * hidden);
  const bf16x8* wr = reinterpret_cast<const bf16x8*>(w);
  bf16x8* yr = reinterpret_cast<bf16x8*>(y + row * ldy);
  const int nvec = hidden / 8;

  float ss = 0.f;
  for (int i = threadIdx.x; i < nvec; i += blockDim.x) {
    bf16x8 v = xr[i];
    #pragma unroll
    for (int j = 0; j < 8; ++j) { float f = bf2f(v.v[j]); ss += f * f; }
  }
  ss = block_sum(ss, red);
  const float r = rsqrtf(ss / hidden + eps);
  for (int i = threadIdx.x; i < nvec; i += blockDim.x) {
    bf16x8 v = xr[i], wv = wr[i], o;
    #pragma unroll
    for (int j = 0; j < 8; ++j) o.v[j] = f2bf(bf2f(v.v[j]) * r * bf2f(wv.v[j]));
    yr[i] = o;
  }
}

__global__ void rmsnorm_fwd_f32(const float* __restrict__ x,
                                const float* __restrict__ w,
                                float* __restrict__ y, int hidden, float eps) {
  __shared__ float red[16];
  const int64_t row = blockIdx.x;
  const float* xr = x + row * hidden;
  float* yr = y + row * hidden;
  float ss = 0.f;
  for (int i = threadIdx.x; i < hidden; i += blockDim.x) { float f = xr[i]; ss += f * f; }
  ss = block_sum(ss, red);
  const float r = rsqrtf(ss / hidden + eps);
  for (int i = threadIdx.x; i < hidden; i += blockDim.x) yr[i] = xr[i] * r * w[i];
}

// dx = r*(dy*w) - r^3/H * x * sum(dy*w*x), plus g where given: the gradient
// that reaches x past the norm (the residual's), which saves a pass of its own
__global__ void rmsnorm_bwd_bf16(const __hip_bfloat16* __restrict__ dy,
                                 const __hip_bfloat16* __restrict__ x,
                                 const __hip_bfloat16* __restrict__ w,
                                 const __hip_bfloat16* __restrict__ g,
                                 __hip_bfloat16* __restrict__ dx,
                                 int hidden, float eps) {
  __shared__ float red[16];
  const int64_t row = blockIdx.x;
  const bf16x8* gr = reinterpret_cast<const bf16x8*>(g + row * hidden);
  const bf16x8* dyr = reinterpret_cast<const bf16x8*>(dy + row * hidden);
  const bf16x8* xr = reinterpret_cast<const bf16x8*>(x + row * hidden);
  const bf16x8* wr = reinterpret_cast<const bf16x8*>(w);
  bf16x8* dxr = reinterpret_cast<bf16x8*>(dx + row * hidden);
  const int nvec = hidden / 8;

  float ss = 0.f, dot = 0.f;
  for (int i = threadIdx.x; i < nvec; i += blockDim.x) {
    bf16x8 xv = xr[i], dyv = dyr[i], wv = wr[i];
    #pragma unroll
    for (int j = 0; j < 8; ++j) {
      float xf = bf2f(xv.v[j]);
      float dyw = bf2f(dyv.v[j]) * bf2f(wv.v[j]);
      ss += xf * xf;
      dot += dyw * xf;
    }
  }
  ss = block_sum(ss, red);
  dot = block_sum(dot, red);
  const float r = rsqrtf(ss / hidden + eps);
  const float c = r * r * r * dot / hidden;
  for (int i = threadIdx.x; i < nvec; i += blockDim.x) {
    bf16x8 xv = xr[i], dyv = dyr[i], wv = wr[i], gv, o;
    if (g) gv = gr[i];
    #pragma unroll
    for (int j = 0; j < 8; ++j) {
      float dyw = bf2f(dyv.v[j]) * bf2f(wv.v[j]);
      float d = dyw * r - bf2f(xv.v[j]) * c;
      o.v[j] = f2bf(g ? d + bf2f(gv.v[j]) : d);
    }
    dxr[i] = o;
  }
}

__global__ void rmsnorm_bwd_f32(const float* __restrict__ dy,
                                const float* __restrict__ x,
                                const float* __restrict__ w,
                                float* __restrict__ dx, int hidden, float eps) {
  __shared__ float red[16];
  const int64_t row = blockIdx.x;
  const float* dyr = dy + row * hidden;
  const float* xr = x + row * hidden;
  float* dxr = dx + row * hidden;
  float ss = 0.f, dot = 0.f;
  for (int i = threadIdx.x; i < hidden; i += blockDim.x) {
    float dyw = dyr[i] * w[i];
    ss += xr[i] * xr[i];
    dot += dyw * xr[i];
  }
  ss = block_sum(ss, red);
  dot = block_sum(dot, red);
  const float r = rsqrtf(ss / hidden + eps);
  const float c = r * r * r * dot / hidden;
  for (int i = threadIdx.x; i < hidden; i += blockDim.x)
    dxr[i] = dyr[i] * w[i] * r - xr[i] * c;
}

}  // namespace

torch::Tensor rmsnorm_fwd(torch::Tensor x, torch::Tensor w, double eps) {
  TORCH_CHECK(x.is_cuda() && x.is_contiguous());
  const int hidden = x.size(-1);
  const int64_t rows = x.numel() / hidden;
  auto y = torch::empty_like(x);
  if (rows == 0) return y;
  dim3 grid(rows), block(256);
  auto stream = at::cuda::getCurrentCUDAStream();
  if (x.scalar_type() == at::kBFloat16) {
    TORCH_CHECK(hidden % 8 == 0, "rmsnorm bf16 needs hidden % 8 == 0");
    hipLaunchKernelGGL(rmsnorm_fwd_bf16, grid, block, 0, stream,
                       reinterpret_cast<const __hip_bfloat16*>(x.data_ptr()),
                       reinterpret_cast<const __hip_bfloat16*>(w.data_ptr()),
                       reinterpret_cast<__hip_bfloat16*>(y.data_ptr()),
                       hidden, (int64_t)hidden, (float)eps);
  } else {
    TORCH_CHECK(x.scalar_type() == at::kFloat, "rmsnorm: bf16 or fp32 only");
    hipLaunchKernelGGL(rmsnorm_fwd_f32, grid, block, 0, stream,
                       x.data_ptr<float>(), w.data_ptr<float>(),
                       y.data_ptr<float>(), hidden, (float)eps);
  }
  HIP_CHECK_LAST();
  return y;
}

// The same into rows of a wider matrix: out (rows, hidden), bf16
void rmsnorm_fwd_into(torch::Tensor x, torch::Tensor w, double eps, torch::Tensor out) {
  const int hidden = x.size(-1);
  TORCH_CHECK(x.is_cuda() && x.is_contiguous() && x.dim() == 2 && x.scalar_type() == at::kBFloat16);
  TORCH_CHECK(w.scalar_type() == at::kBFloat16 && w.numel() == hidden && w.is_contiguous());
  TORCH_CHECK(out.sizes() == x.sizes() && out.scalar_type() == at::kBFloat16 && out.is_cuda() &&
              out.stride(1) == 1 && out.stride(0) % 8 == 0 && hidden % 8 == 0 &&
              reinterpret_cast<uintptr_t>(out.data_ptr()) % 16 == 0, "rmsnorm_fwd_into: output");
  if (x.size(0) == 0) return;
  hipLaunchKernelGGL(rmsnorm_fwd_bf16, dim3(x.size(0)), dim3(256), 0,
                     at::cuda::getCurrentCUDAStream(),
                     reinterpret_cast<const __hip_bfloat16*>(x.data_ptr()),
                     reinterpret_cast<const __hip_bfloat16*>(w.data_ptr()),
                     reinterpret_cast<__hip_bfloat16*>(out.data_ptr()), hidden, out.stride(0),
                     (float)eps);
  HIP_CHECK_LAST();
}

torch::Tensor rmsnorm_bwd(torch::Tensor dy, torch::Tensor x, torch::Tensor w,
                          double eps) {
  TORCH_CHECK(dy.is_cuda() && dy.is_contiguous() && x.is_contiguous());
  const int hidden = x.size(-1);
  const int64_t rows = x.numel() / hidden;
  auto dx = torch::empty_like(x);
  if (rows == 0) return dx;
  dim3 grid(rows), block(256);
  auto stream = at::cuda::getCurrentCUDAStream();
  if (x.scalar_type() == at::kBFloat16) {
    TORCH_CHECK(hidden % 8 == 0);
    hipLaunchKernelGGL(rmsnorm_bwd_bf16, grid, block, 0, stream,
                       reinterpret_cast<const __hip_bfloat16*>(dy.data_ptr()),
                       reinterpret_cast<const __hip_bfloat16*>(x.data_ptr()),
                       reinterpret_cast<const __hip_bfloat16*>(w.data_ptr()),
                       (const __hip_bfloat16*)nullptr,
                       reinterpret_cast<__hip_bfloat16*>(dx.data_ptr()),
                       hidden, (float)eps);
  } else {
    TORCH_CHECK(x.scalar_type() == at::kFloat);
    hipLaunchKernelGGL(rmsnorm_bwd_f32, grid, block, 0, stream,
                       dy.data_ptr<float>(), x.data_ptr<float>(),
                       w.data_ptr<float>(), dx.data_ptr<float>(),
                       hidden, (float)eps);
  }
  HIP_CHECK_LAST();
  return dx;
}

// dx = g + rmsnorm's dx (bf16)
torch::Tensor rmsnorm_bwd_add(torch::Tensor dy, torch::Tensor x, torch::Tensor w,
                              torch::Tensor g, double eps) {
  TORCH_CHECK(dy.is_cuda() && dy.is_contiguous() && x.is_contiguous() && g.is_contiguous());
  TORCH_CHECK(dy.scalar_type() == at::kBFloat16 && x.scalar_type() == at::kBFloat16 &&
              w.scalar_type() == at::kBFloat16 && g.scalar_type() == at::kBFloat16);
  TORCH_CHECK(dy.sizes() == x.sizes() && g.sizes() == x.sizes() && w.numel() == x.size(-1));
  const int hidden = x.size(-1);
  TORCH_CHECK(hidden % 8 == 0);
  const int64_t rows = x.numel() / hidden;
  auto dx = torch::empty_like(x);
  if (rows == 0) return dx;
  hipLaunchKernelGGL(rmsnorm_bwd_bf16, dim3(rows), dim3(256), 0,
                     at::cuda::getCurrentCUDAStream(),
                     reinterpret_cast<const __hip_bfloat16*>(dy.data_ptr()),
                     reinterpret_cast<const __hip_bfloat16*>(x.data_ptr()),
                     reinterpret_cast<const __hip_bfloat16*>(w.data_ptr()),
                     reinterpret_cast<const __hip_bfloat16*>(g.data_ptr()),
                     reinterpret_cast<__hip_bfloat16*>(dx.data_ptr()), hidden, (float)eps);
  HIP_CHECK_LAST();
  return dx;
}

// ---- fused residual-add + RMSNorm (decode path): res = x + h;
// y = rmsnorm(res) * w. Saves one full elementwise pass per layer site.
namespace {

__global__ void add_rmsnorm_fwd_bf16(const __hip_bfloat16* __restrict__ x,
                                     const __hip_bfloat16* __restrict__ h,
                                     const __hip_bfloat16* __restrict__ w,
                                     __hip_bfloat16* __restrict__ y,
                                     __hip_bfloat16* __restrict__ res,
                                     int hidden, float eps) {
  __shared__ float red[16];
  const int64_t row = blockIdx.x;
  const bf16x8* xr = reinterpret_cast<const bf16x8*>(x + row * hidden);
  const bf16x8* hr = reinterpret_cast<const bf16x8*>(h + row * hidden);
  const bf16x8* wr = reinterpret_cast<const bf16x8*>(w);
  bf16x8* yr = reinterpret_cast<bf16x8*>(y + row * hidden);
  bf16x8* rr = reinterpret_cast<bf16x8*>(res + row * hidden);
  const int nvec = hidden / 8;

  float ss = 0.f;
  for (int i = threadIdx.x; i < nvec; i += blockDim.x) {
    bf16x8 xv = xr[i], hv = hr[i], s;
    #pragma unroll
    for (int j = 0; j < 8; ++j) {
      float f = bf2f(xv.v[j]) + bf2f(hv.v[j]);
      s.v[j] = f2bf(f);
      ss += f * f;
    }
    rr[i] = s;
  }
  ss = block_sum(ss, red);
  const float r = rsqrtf(ss / hidden + eps);
  for (int i = threadIdx.x; i < nvec; i += blockDim.x) {
    bf16x8 sv = rr[i], wv = wr[i], o;
    #pragma unroll
    for (int j = 0; j < 8; ++j) o.v[j] = f2bf(bf2f(sv.v[j]) * r * bf2f(wv.v[j]));
    yr[i] = o;
  }
}

}  // namespace

std::vector<torch::Tensor> add_rmsnorm_fwd(torch::Tensor x, torch::Tensor h,
                                           torch::Tensor w, double eps) {
  TORCH_CHECK(x.is_cuda() && x.is_contiguous() && h.is_contiguous());
  TORCH_CHECK(x.scalar_type() == at::kBFloat16);
  const int hidden = x.size(-1);
  TORCH_CHECK(hidden % 8 == 0);
  const int64_t rows = x.numel() / hidden;
  auto y = torch::empty_like(x);
  auto res = torch::empty_like(x);
  if (rows == 0) return {y, res};
  hipLaunchKernelGGL(add_rmsnorm_fwd_bf16, dim3(rows), dim3(256), 0,
                     at::cuda::getCurrentCUDAStream(),
                     reinterpret_cast<const __hip_bfloat16*>(x.data_ptr()),
                     reinterpret_cast<const __hip_bfloat16*>(h.data_ptr()),
                     reinterpret_cast<const __hip_bfloat16*>(w.data_ptr()),
                     reinterpret_cast<__hip_bfloat16*>(y.data_ptr()),
                     reinterpret_cast<__hip_bfloat16*>(res.data_ptr()),
                     hidden, (float)eps);
  HIP_CHECK_LAST();
  return {y, res};
}

// ---- the same behind a product that left partial sums (S, rows, hidden + r):
// res' = res + their sum (+ u bt, u the sum of the last r columns, bt (r, hidden)
// an adapter's output weights), y = rmsnorm(res') * w. One workgroup a row, 8
// columns a thread: all of a row's loads are in flight at once.
namespace {

template <int VPT>
__global__ __launch_bounds__(512)
void add_rmsnorm_join_kernel(const float* __restrict__ parts, const __hip_bfloat16* __restrict__ x,
                             const __hip_bfloat16* __restrict__ bt,
                             const __hip_bfloat16* __restrict__ w, __hip_bfloat16* __restrict__ y,
                             __hip_bfloat16* __restrict__ res, int rows, int hidden, int r, int S,
                             float eps) {
  __shared__ float red[16], us[128];
  const int64_t row = blockIdx.x, ld = hidden + r, step = rows * ld;
  const float* pr = parts + row * ld;
  for (int j = threadIdx.x; j < r; j += blockDim.x) {
    float u = 0.f;
    for (int z = 0; z < S; ++z) u += pr[z * step + hidden + j];
    us[j] = u;
  }
  float v[VPT][8];
  #pragma unroll
  for (int k = 0; k < VPT; ++k) {
    const int n = (k * blockDim.x + threadIdx.x) * 8;
    #pragma unroll
    for (int j = 0; j < 8; ++j) v[k][j] = 0.f;
    if (n >= hidden) continue;
    const bf16x8 xv = *reinterpret_cast<const bf16x8*>(x + row * hidden + n);
    add_parts8(v[k], pr + n, step, S);
    #pragma unroll
    for (int j = 0; j < 8; ++j) v[k][j] += bf2f(xv.v[j]);
  }
  if (r > 0) {
    __syncthreads();
    #pragma unroll
    for (int k = 0; k < VPT; ++k) {
      const int n = (k * blockDim.x + threadIdx.x) * 8;
      if (n >= hidden) continue;
      #pragma unroll 8
      for (int i = 0; i < r; ++i) {
        const bf16x8 b = *reinterpret_cast<const bf16x8*>(bt + (int64_t)i * hidden + n);
        #pragma unroll
        for (int j = 0; j < 8; ++j) v[k][j] += us[i] * bf2f(b.v[j]);
      }
    }
  }
  float ss = 0.f;
  #pragma unroll
  for (int k = 0; k < VPT; ++k)
    #pragma unroll
    for (int j = 0; j < 8; ++j) ss += v[k][j] * v[k][j];
  ss = block_sum(ss, red);
  const float rn = rsqrtf(ss / hidden + eps);
  #pragma unroll
  for (int k = 0; k < VPT; ++k) {
    const int n = (k * blockDim.x + threadIdx.x) * 8;
    if (n >= hidden) continue;
    const bf16x8 wv = *reinterpret_cast<const bf16x8*>(w + n);
    bf16x8 o, s;
    #pragma unroll
    for (int j = 0; j < 8; ++j) {
      s.v[j] = f2bf(v[k][j]);
      o.v[j] = f2bf(bf2f(s.v[j]) * rn * bf2f(wv.v[j]));
    }
    *reinterpret_cast<bf16x8*>(res + row * hidden + n) = s;
    *reinterpret_cast<bf16x8*>(y + row * hidden + n) = o;
  }
}

}  // namespace

// {rmsnorm(res') * w, res'}, res' = res + the parts' sum (+ the adapter)
std::vector<torch::Tensor> add_rmsnorm_join(torch::Tensor parts, torch::Tensor res, torch::Tensor w,
                                            double eps, c10::optional<torch::Tensor> bt) {
  TORCH_CHECK(res.is_cuda() && res.is_contiguous() && res.dim() == 2 &&
              res.scalar_type() == at::kBFloat16);
  TORCH_CHECK(parts.is_cuda() && parts.is_contiguous() && parts.dim() == 3 &&
              parts.scalar_type() == at::kFloat && parts.size(1) == res.size(0));
  const int rows = res.size(0), hidden = res.size(1), r = (int)parts.size(2) - hidden;
  TORCH_CHECK(w.is_cuda() && w.is_contiguous() && w.scalar_type() == at::kBFloat16 &&
              w.numel() == hidden);
  TORCH_CHECK(hidden % 8 == 0 && hidden <= 8192 && r >= 0 && r <= 128 && r % 8 == 0,
              "add_rmsnorm_join: unsupported shape");
  TORCH_CHECK((r > 0) == bt.has_value());
  if (bt)
    TORCH_CHECK(bt->is_cuda() && bt->is_contiguous() && bt->scalar_type() == at::kBFloat16 &&
                bt->dim() == 2 && bt->size(0) == r && bt->size(1) == hidden);
  for (const auto* t : {&res, &w})
    TORCH_CHECK(reinterpret_cast<uintptr_t>(t->data_ptr()) % 16 == 0, "add_rmsnorm_join: alignment");
  TORCH_CHECK(!bt || reinterpret_cast<uintptr_t>(bt->data_ptr()) % 16 == 0);
  auto y = torch::empty_like(res), out = torch::empty_like(res);
  if (rows == 0) return {y, out};
  const int threads = std::min(512, CDIV(hidden / 8, 64) * 64);
  auto bf = [](const torch::Tensor& t) { return reinterpret_cast<__hip_bfloat16*>(t.data_ptr()); };
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(rows), dim3(threads), 0, at::cuda::getCurrentCUDAStream(),
                       parts.data_ptr<float>(), bf(res), bt ? bf(*bt) : nullptr, bf(w), bf(y),
                       bf(out), rows, hidden, r, (int)parts.size(0), (float)eps);
  };
  if (hidden <= 4096) go(add_rmsnorm_join_kernel<1>);
  else go(add_rmsnorm_join_kernel<2>);
  HIP_CHECK_LAST();
  return {y, out};
}
