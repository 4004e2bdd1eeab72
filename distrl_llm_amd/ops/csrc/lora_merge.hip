// Decode weights of an adapted projection: out = W + scale * B A, (N, K) bf16,
// B (N, r), A (r, K), the sum in fp32 and rounded once. Refreshed once per
// generation, for every projection of the model.
//
// One read of W and one write of out, 16 B a lane; B A comes from MFMA
// 16x16x32 on the way (one product per 16 x 16 x 32 of r): A's tile lies in
// LDS and is read transposed, with the columns of two products interleaved so
// that a lane ends up with 8 consecutive k of one row. Bound: memory.
// As torch operations (fp32 product, two conversions, scale, sum, concatenation
// and copy into the captured storage) the 7B model's refresh took 44 ms,
// 13 ms now for 2 x 13 GB (with the 4-bit site's adapter packs).
#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>
#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16v8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16v4;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((address_space(3))) bf16v4 lds_bf16v4;

namespace {

constexpr int KC = 256;            // columns of a workgroup
constexpr int ROWS = 128;          // rows of a workgroup, 16 a wave and turn

__global__ __launch_bounds__(256)
void lora_merge_kernel(const __hip_bfloat16* __restrict__ w, const __hip_bfloat16* __restrict__ a,
                       const __hip_bfloat16* __restrict__ b, __hip_bfloat16* __restrict__ out,
                       int N, int K, int r, float scale) {
  extern __shared__ __attribute__((aligned(16))) char smem[];   // A: [r32][KC], rows 16 B apart
  constexpr int RS = KC * 2 + 16;
  const int k0 = blockIdx.x * KC, r32 = (r + 31) / 32 * 32;
  for (int i = threadIdx.x; i < r32 * (KC / 8); i += 256) {
    const int row = i / (KC / 8), c = i % (KC / 8);
    bf16v8 v;
    #pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = (__bf16)0.f;
    if (row < r && k0 + c * 8 < K)
      v = *reinterpret_cast<const bf16v8*>(a + (int64_t)row * K + k0 + c * 8);
    *reinterpret_cast<bf16v8*>(smem + row * RS + c * 16) = v;
  }
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = threadIdx.x & 63, g = l >> 4, lr = l & 15;
  for (int n0 = blockIdx.y * ROWS + wave * 16; n0 < min(N, (int)(blockIdx.y + 1) * ROWS); n0 += 64) {
    const int n = min(n0 + lr, N - 1);
    #pragma unroll 2
    for (int kk = 0; kk < KC; kk += 32) {
      if (k0 + kk >= K) break;                          // K % 32 == 0
      const int64_t at = (int64_t)n * K + k0 + kk + g * 8;
      const bf16v8 wv = *reinterpret_cast<const bf16v8*>(w + at);
      f32x4 d[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
      for (int s = 0; s < r32; s += 32) {
        bf16v8 bv;
        #pragma unroll
        for (int j = 0; j < 8; ++j) bv[j] = (__bf16)0.f;
        if (s + g * 8 < r)                              // r % 8 == 0
          bv = *reinterpret_cast<const bf16v8*>(b + (int64_t)n * r + s + g * 8);
        #pragma unroll
        for (int t = 0; t < 2; ++t) {
          // rows s + 8 g + 0..7 of A; lane i gets column 8 (i/4) + i%4 + 4 t
          char* p = smem + (s + g * 8 + (lr >> 2)) * RS + (kk + (lr & 3) * 8 + t * 4) * 2;
          const bf16v4 x = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16v4*)p);
          const bf16v4 y = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16v4*)(p + 4 * RS));
          const bf16v8 av = __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7);
          d[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv, d[t], 0, 0, 0);
        }
      }
      bf16v8 o;
      #pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = (__bf16)((float)wv[j] + scale * d[j >> 2][j & 3]);
      if (n0 + lr < N) *reinterpret_cast<bf16v8*>(out + at) = o;
    }
  }
}

}  // namespace

bool lora_merge_takes(int64_t K, int64_t r) { return K % 32 == 0 && r % 8 == 0 && r >= 8 && r <= 128; }

void lora_merge(torch::Tensor w, torch::Tensor a, torch::Tensor b, torch::Tensor out, double scale) {
  TORCH_CHECK(w.dim() == 2 && a.dim() == 2 && b.dim() == 2);
  const int N = w.size(0), K = w.size(1), r = a.size(0);
  TORCH_CHECK(a.size(1) == K && b.size(0) == N && b.size(1) == r && out.sizes() == w.sizes());
  TORCH_CHECK(lora_merge_takes(K, r), "lora_merge: unsupported K ", K, " or rank ", r);
  for (const auto& t : {w, a, b, out})
    TORCH_CHECK(t.is_cuda() && t.is_contiguous() && t.scalar_type() == at::kBFloat16 &&
                reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0, "lora_merge: operand");
  if (N == 0) return;
  auto p = [](const torch::Tensor& t) { return reinterpret_cast<const __hip_bfloat16*>(t.data_ptr()); };
  hipLaunchKernelGGL(lora_merge_kernel, dim3(CDIV(K, KC), CDIV(N, ROWS)), dim3(256),
                     (r + 31) / 32 * 32 * (KC * 2 + 16), at::cuda::getCurrentCUDAStream(), p(w),
                     p(a), p(b), reinterpret_cast<__hip_bfloat16*>(out.data_ptr()), N, K, r,
                     (float)scale);
  HIP_CHECK_LAST();
}
