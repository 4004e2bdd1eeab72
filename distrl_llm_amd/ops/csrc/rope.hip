// Fused in-place RoPE for the generation path (rotate_half / neox
// convention, matching HF Qwen2/Llama). Replaces vLLM's pos_encoding
// kernels. cos/sin computed once per token into LDS and
// reused across all q + kv heads.
#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>
#include "common.h"

namespace {

__global__ void rope_inplace_kernel(__hip_bfloat16* __restrict__ q,
                                    __hip_bfloat16* __restrict__ k,
                                    const int* __restrict__ positions,
                                    const float* __restrict__ inv_freq,
                                    int H, int KV, int D) {
  extern __shared__ float smem[];  // [D/2 cos][D/2 sin]
  const int half = D / 2;
  float* cs = smem;
  float* sn = smem + half;
  const int t = blockIdx.x;
  const float pos = (float)positions[t];
  for (int i = threadIdx.x; i < half; i += blockDim.x) {
    float a = pos * inv_freq[i];
    sn[i] = __sinf(a);
    cs[i] = __cosf(a);
  }
  __syncthreads();

  const int total = (H + KV) * half;
  for (int idx = threadIdx.x; idx < total; idx += blockDim.x) {
    const int head = idx / half;
    const int i = idx % half;
    __hip_bfloat16* ptr = (head < H)
        ? q + ((int64_t)t * H + head) * D
        : k + ((int64_t)t * KV + (head - H)) * D;
    float x1 = bf2f(ptr[i]);
    float x2 = bf2f(ptr[i + half]);
    float c = cs[i], s = sn[i];
    ptr[i] = f2bf(x1 * c - x2 * s);
    ptr[i + half] = f2bf(x2 * c + x1 * s);
  }
}

// The same for half % 8 == 0 and rows on 16 bytes: a thread rotates 8 pairs,
// 16 B at each end (2-byte accesses held the one above to ~2 TB/s). One wave a
// token and 64 units of eight pairs; four tokens a workgroup.
__global__ __launch_bounds__(256)
void rope_inplace_vec_kernel(__hip_bfloat16* __restrict__ q, __hip_bfloat16* __restrict__ k,
                             const int* __restrict__ positions,
                             const float* __restrict__ inv_freq, int T, int H, int KV, int D,
                             int64_t ldq, int64_t ldk) {
  const int t = blockIdx.x * 4 + threadIdx.x / WAVE, lane = threadIdx.x & (WAVE - 1);
  if (t >= T) return;
  const int half = D / 2, per = half / 8;        // units of a head
  const float pos = (float)positions[t];
  int unit_c = -1;
  float cs[8], sn[8];
  for (int u = lane; u < (H + KV) * per; u += WAVE) {
    const int head = u / per, c = u % per * 8;
    if (c != unit_c) {                           // 64 % per == 0: once a lane
      unit_c = c;
      #pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float a = pos * inv_freq[c + j];
        sn[j] = __sinf(a);
        cs[j] = __cosf(a);
      }
    }
    __hip_bfloat16* p = (head < H ? q + t * ldq + head * D : k + t * ldk + (head - H) * D) + c;
    const bf16x8 a = *reinterpret_cast<const bf16x8*>(p);
    const bf16x8 b = *reinterpret_cast<const bf16x8*>(p + half);
    bf16x8 x, y;
    #pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float x1 = bf2f(a.v[j]), x2 = bf2f(b.v[j]);
      x.v[j] = f2bf(x1 * cs[j] - x2 * sn[j]);
      y.v[j] = f2bf(x2 * cs[j] + x1 * sn[j]);
    }
    *reinterpret_cast<bf16x8*>(p) = x;
    *reinterpret_cast<bf16x8*>(p + half) = y;
  }
}

// ---- fused packed-QKV RoPE + paged KV scatter (decode fast path) ----
// qkv: (T, H*D + 2*KV*D) packed rows straight out of the fused qkv GEMM.
// Rotates q and k in place, then scatters the (rotated) k and v rows into
// the paged pool — one kernel replaces rope + 2 contiguous-copies +
// kv_cache_scatter.
__global__ void rope_scatter_qkv_kernel(__hip_bfloat16* __restrict__ qkv,
                                        const int* __restrict__ positions,
                                        const int64_t* __restrict__ slots,
                                        const float* __restrict__ inv_freq,
                                        __hip_bfloat16* __restrict__ key_cache,
                                        __hip_bfloat16* __restrict__ value_cache,
                                        int H, int KV, int D) {
  extern __shared__ float smem[];  // [D/2 cos][D/2 sin]
  const int half = D / 2;
  float* cs = smem;
  float* sn = smem + half;
  const int t = blockIdx.x;
  const int row_stride = (H + 2 * KV) * D;
  const float pos = (float)positions[t];
  for (int i = threadIdx.x; i < half; i += blockDim.x) {
    float a = pos * inv_freq[i];
    sn[i] = __sinf(a);
    cs[i] = __cosf(a);
  }
  __syncthreads();

  __hip_bfloat16* base = qkv + (int64_t)t * row_stride;
  const int total = (H + KV) * half;  // rotate q heads then k heads
  for (int idx = threadIdx.x; idx < total; idx += blockDim.x) {
    const int head = idx / half;
    const int i = idx % half;
    __hip_bfloat16* ptr = base + head * D;  // q heads then k heads: packed
    float x1 = bf2f(ptr[i]);
    float x2 = bf2f(ptr[i + half]);
    float c = cs[i], s = sn[i];
    ptr[i] = f2bf(x1 * c - x2 * s);
    ptr[i + half] = f2bf(x2 * c + x1 * s);
  }
  __syncthreads();

  // scatter rotated k and raw v into the pool
  const int64_t slot = slots[t];
  if (slot < 0) return;
  const int row_vecs = KV * D / 8;
  const bf16x8* ks = reinterpret_cast<const bf16x8*>(base + H * D);
  const bf16x8* vs = reinterpret_cast<const bf16x8*>(base + (H + KV) * D);
  bf16x8* kd = reinterpret_cast<bf16x8*>(key_cache) + slot * row_vecs;
  bf16x8* vd = reinterpret_cast<bf16x8*>(value_cache) + slot * row_vecs;
  for (int i = threadIdx.x; i < row_vecs; i += blockDim.x) {
    kd[i] = ks[i];
    vd[i] = vs[i];
  }
}

// The same for D 64 and 128 with 16 B accesses: 8 pairs a thread, so a head
// takes D/16 neighbouring lanes, which also norm it (q_norm, k_norm: RMS norm
// of each head before the rotation, rounded to bf16 in between as a separate
// norm's output is; as torch operations it cost fourteen launches a layer).
__global__ __launch_bounds__(256)
void rope_scatter_vec_kernel(__hip_bfloat16* __restrict__ qkv, const int* __restrict__ positions,
                             const int64_t* __restrict__ slots,
                             const float* __restrict__ inv_freq,
                             __hip_bfloat16* __restrict__ key_cache,
                             __hip_bfloat16* __restrict__ value_cache,
                             const __hip_bfloat16* __restrict__ q_norm,
                             const __hip_bfloat16* __restrict__ k_norm, float eps, int H, int KV,
                             int D) {
  const int t = blockIdx.x, half = D / 2, per = half / 8;
  const int64_t slot = slots[t];
  const float pos = (float)positions[t];
  __hip_bfloat16* base = qkv + (int64_t)t * (H + 2 * KV) * D;
  const int c = threadIdx.x % per * 8;          // 256 % per == 0: fixed
  float cs[8], sn[8];
  #pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float a = pos * inv_freq[c + j];
    sn[j] = __sinf(a);
    cs[j] = __cosf(a);
  }
  const int rot = (H + KV) * per, all = rot + KV * D / 8;
  // whole heads stay together: rot and the step are multiples of per
  for (int u = threadIdx.x; u < all; u += 256) {
    if (u >= rot) {                             // a value unit
      const int i = u - rot;
      if (slot >= 0)
        reinterpret_cast<bf16x8*>(value_cache)[slot * (KV * D / 8) + i] =
            reinterpret_cast<const bf16x8*>(base + (H + KV) * D)[i];
      continue;
    }
    const int head = u / per;
    __hip_bfloat16* p = base + head * D + c;
    const bf16x8 a = *reinterpret_cast<const bf16x8*>(p);
    const bf16x8 b = *reinterpret_cast<const bf16x8*>(p + half);
    float x1[8], x2[8];
    #pragma unroll
    for (int j = 0; j < 8; ++j) { x1[j] = bf2f(a.v[j]); x2[j] = bf2f(b.v[j]); }
    const __hip_bfloat16* nw = head < H ? q_norm : k_norm;
    if (nw) {
      float ss = 0.f;
      #pragma unroll
      for (int j = 0; j < 8; ++j) ss += x1[j] * x1[j] + x2[j] * x2[j];
      for (int off = per / 2; off > 0; off >>= 1) ss += __shfl_xor(ss, off, WAVE);
      const float r = rsqrtf(ss / D + eps);
      #pragma unroll
      for (int j = 0; j < 8; ++j) {
        x1[j] = bf2f(f2bf(x1[j] * r * bf2f(nw[c + j])));
        x2[j] = bf2f(f2bf(x2[j] * r * bf2f(nw[c + half + j])));
      }
    }
    bf16x8 x, y;
    #pragma unroll
    for (int j = 0; j < 8; ++j) {
      x.v[j] = f2bf(x1[j] * cs[j] - x2[j] * sn[j]);
      y.v[j] = f2bf(x2[j] * cs[j] + x1[j] * sn[j]);
    }
    *reinterpret_cast<bf16x8*>(p) = x;
    *reinterpret_cast<bf16x8*>(p + half) = y;
    if (head >= H && slot >= 0) {
      __hip_bfloat16* kd = key_cache + (slot * KV + head - H) * D + c;
      *reinterpret_cast<bf16x8*>(kd) = x;
      *reinterpret_cast<bf16x8*>(kd + half) = y;
    }
  }
}

}  // namespace

void rope_scatter_qkv(torch::Tensor qkv, torch::Tensor positions,
                      torch::Tensor slots, torch::Tensor inv_freq,
                      torch::Tensor key_cache, torch::Tensor value_cache,
                      int64_t H, int64_t KV, int64_t D,
                      c10::optional<torch::Tensor> q_norm,
                      c10::optional<torch::Tensor> k_norm, double eps) {
  TORCH_CHECK(qkv.is_cuda() && qkv.is_contiguous());
  TORCH_CHECK(qkv.scalar_type() == at::kBFloat16);
  TORCH_CHECK(positions.scalar_type() == at::kInt);
  TORCH_CHECK(slots.scalar_type() == at::kLong);
  const int T = qkv.size(0);
  TORCH_CHECK(qkv.size(1) == (H + 2 * KV) * D);
  TORCH_CHECK((KV * D) % 8 == 0);
  auto norm = [&](const c10::optional<torch::Tensor>& w) {
    if (!w) return (const __hip_bfloat16*)nullptr;
    TORCH_CHECK(w->is_cuda() && w->is_contiguous() && w->scalar_type() == at::kBFloat16 &&
                w->numel() == D, "rope_scatter_qkv: head norm weight");
    return reinterpret_cast<const __hip_bfloat16*>(w->data_ptr());
  };
  const auto *qn = norm(q_norm), *kn = norm(k_norm);
  const bool vec = (D == 64 || D == 128) && reinterpret_cast<uintptr_t>(qkv.data_ptr()) % 16 == 0;
  TORCH_CHECK(vec || (!qn && !kn), "rope_scatter_qkv: head norms need head_dim 64 or 128");
  if (T == 0) return;
  if (vec) {
    hipLaunchKernelGGL(rope_scatter_vec_kernel, dim3(T), dim3(256), 0,
                       at::cuda::getCurrentCUDAStream(),
                       reinterpret_cast<__hip_bfloat16*>(qkv.data_ptr()),
                       positions.data_ptr<int>(), slots.data_ptr<int64_t>(),
                       inv_freq.data_ptr<float>(),
                       reinterpret_cast<__hip_bfloat16*>(key_cache.data_ptr()),
                       reinterpret_cast<__hip_bfloat16*>(value_cache.data_ptr()), qn, kn,
                       (float)eps, (int)H, (int)KV, (int)D);
    HIP_CHECK_LAST();
    return;
  }
  const int smem = D * sizeof(float);
  hipLaunchKernelGGL(rope_scatter_qkv_kernel, dim3(T), dim3(256), smem,
                     at::cuda::getCurrentCUDAStream(),
                     reinterpret_cast<__hip_bfloat16*>(qkv.data_ptr()),
                     positions.data_ptr<int>(), slots.data_ptr<int64_t>(),
                     inv_freq.data_ptr<float>(),
                     reinterpret_cast<__hip_bfloat16*>(key_cache.data_ptr()),
                     reinterpret_cast<__hip_bfloat16*>(value_cache.data_ptr()),
                     (int)H, (int)KV, (int)D);
  HIP_CHECK_LAST();
}

// q (T, H, D), k (T, KV, D), whose rows may lie apart
void rope_rows(torch::Tensor q, torch::Tensor k, torch::Tensor positions,
               torch::Tensor inv_freq) {
  // heads of a row follow one another
  auto rows = [](const torch::Tensor& x) {
    return x.dim() == 3 && (x.size(2) <= 1 || x.stride(2) == 1) &&
           (x.size(1) <= 1 || x.stride(1) == x.size(2));
  };
  TORCH_CHECK(q.is_cuda() && rows(q) && rows(k));
  TORCH_CHECK(q.scalar_type() == at::kBFloat16 && k.scalar_type() == at::kBFloat16);
  TORCH_CHECK(positions.scalar_type() == at::kInt);
  const int T = q.size(0), H = q.size(1), D = q.size(2);
  const int KV = k.size(1);
  TORCH_CHECK(k.size(0) == T && k.size(2) == D);
  if (T == 0) return;
  auto aligned = [](const torch::Tensor& x) {
    return reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 && x.stride(0) % 8 == 0;
  };
  if (D % 16 == 0 && aligned(q) && aligned(k)) {
    hipLaunchKernelGGL(rope_inplace_vec_kernel, dim3((T + 3) / 4), dim3(256), 0,
                       at::cuda::getCurrentCUDAStream(),
                       reinterpret_cast<__hip_bfloat16*>(q.data_ptr()),
                       reinterpret_cast<__hip_bfloat16*>(k.data_ptr()),
                       positions.data_ptr<int>(), inv_freq.data_ptr<float>(), T, H, KV, D,
                       q.stride(0), k.stride(0));
    HIP_CHECK_LAST();
    return;
  }
  TORCH_CHECK(q.is_contiguous() && k.is_contiguous());
  const int smem = D * sizeof(float);
  hipLaunchKernelGGL(rope_inplace_kernel, dim3(T), dim3(256), smem,
                     at::cuda::getCurrentCUDAStream(),
                     reinterpret_cast<__hip_bfloat16*>(q.data_ptr()),
                     reinterpret_cast<__hip_bfloat16*>(k.data_ptr()),
                     positions.data_ptr<int>(), inv_freq.data_ptr<float>(),
                     H, KV, D);
  HIP_CHECK_LAST();
}

void rope_inplace(torch::Tensor q, torch::Tensor k, torch::Tensor positions,
                  torch::Tensor inv_freq) {
  TORCH_CHECK(q.is_contiguous() && k.is_contiguous());
  rope_rows(q, k, positions, inv_freq);
}
