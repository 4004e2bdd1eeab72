// Paged KV-cache scatter (the reference's vLLM reshape_and_cache): write the
// step's new K/V rows into their pool slots; and copies of a page, where a prompt's
// last one is shared out.
#include <algorithm>
#include <climits>
#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>
#include "common.h"

namespace {

// k,v: (T, KV, D) bf16; caches: (num_blocks, block_size, KV, D);
// slot_mapping: (T,) int32 flat slot = block*block_size + offset, -1 skips.
__global__ void kv_scatter_kernel(const bf16x8* __restrict__ k,
                                  const bf16x8* __restrict__ v,
                                  bf16x8* __restrict__ key_cache,
                                  bf16x8* __restrict__ value_cache,
                                  const int* __restrict__ slot_mapping,
                                  int row_vecs /* KV*D/8 */) {
  const int t = blockIdx.x;
  const int slot = slot_mapping[t];
  if (slot < 0) return;
  const bf16x8* ks = k + (int64_t)t * row_vecs;
  const bf16x8* vs = v + (int64_t)t * row_vecs;
  bf16x8* kd = key_cache + (int64_t)slot * row_vecs;
  bf16x8* vd = value_cache + (int64_t)slot * row_vecs;
  for (int i = threadIdx.x; i < row_vecs; i += blockDim.x) {
    kd[i] = ks[i];
    vd[i] = vs[i];
  }
}

constexpr int PAGES = 60;               // a launch copies a page to, by its arguments

struct Copies {
  int src, n;
  int dst[PAGES];
};

// Caches (layers, num_blocks, vecs): page src of every layer, key and value, to n others.
// A page is read once; a copy a launch (torch's, key and value apart) was 32 launches for
// the 16 candidates of a prompt, and between prompt phase and first step the GPU waits for
// the host: 10 prompts x 16 candidates of the 7B model 168.3 -> 167.0 ms, 2 x 16 of the 4B
// 104.7 -> 103.9, of the 1.5B 67.8 -> 67.2. grid (16 B of a page / 256, layers, 2)
__global__ __launch_bounds__(256)
void kv_copy_kernel(uint4* __restrict__ key, uint4* __restrict__ value, Copies to, int64_t num_blocks,
                    int64_t vecs) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= vecs) return;
  uint4* layer = (blockIdx.z ? value : key) + blockIdx.y * num_blocks * vecs + i;
  const uint4 x = layer[to.src * vecs];
  for (int j = 0; j < to.n; ++j) layer[to.dst[j] * vecs] = x;
}

}  // namespace

// Page src of all layers to pages dst; key, value (layers, num_blocks, page sizes...).
// False, and nothing done, for caches that 16 B accesses can't walk.
bool kv_copy_page(torch::Tensor key, torch::Tensor value, int64_t src, std::vector<int64_t> dst) {
  TORCH_CHECK(key.is_cuda() && key.dim() >= 2 && value.sizes() == key.sizes() &&
              value.scalar_type() == key.scalar_type() && value.device() == key.device());
  const int64_t layers = key.size(0), blocks = key.size(1);
  if (!key.is_contiguous() || !value.is_contiguous() || layers > 65535) return false;
  if (key.numel() == 0) return true;
  const int64_t bytes = key.numel() / layers / blocks * key.element_size();
  auto at16 = [](const torch::Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; };
  if (bytes % 16 || bytes > ((int64_t)1 << 30) || blocks > INT_MAX || !at16(key) || !at16(value)) return false;
  auto inside = [&](int64_t page) { return page >= 0 && page < blocks; };
  TORCH_CHECK(inside(src) && std::all_of(dst.begin(), dst.end(), inside), "kv_copy_page: no such page");
  for (size_t first = 0; first < dst.size(); first += PAGES) {
    Copies to;
    to.src = (int)src;
    to.n = (int)std::min<size_t>(PAGES, dst.size() - first);
    for (int j = 0; j < to.n; ++j) to.dst[j] = (int)dst[first + j];
    hipLaunchKernelGGL(kv_copy_kernel, dim3(CDIV(bytes / 16, 256), layers, 2), dim3(256), 0,
                       at::cuda::getCurrentCUDAStream(), reinterpret_cast<uint4*>(key.data_ptr()),
                       reinterpret_cast<uint4*>(value.data_ptr()), to, blocks, bytes / 16);
    HIP_CHECK_LAST();
  }
  return true;
}

void kv_cache_scatter(torch::Tensor k, torch::Tensor v,
                      torch::Tensor key_cache, torch::Tensor value_cache,
                      torch::Tensor slot_mapping) {
  TORCH_CHECK(k.is_cuda() && k.is_contiguous() && v.is_contiguous());
  TORCH_CHECK(key_cache.is_contiguous() && value_cache.is_contiguous());
  TORCH_CHECK(k.scalar_type() == at::kBFloat16);
  TORCH_CHECK(slot_mapping.scalar_type() == at::kInt);
  const int T = k.size(0);
  if (T == 0) return;
  const int KV = k.size(1), D = k.size(2);
  TORCH_CHECK((KV * D) % 8 == 0);
  const int row_vecs = KV * D / 8;
  hipLaunchKernelGGL(kv_scatter_kernel, dim3(T), dim3(128), 0,
                     at::cuda::getCurrentCUDAStream(),
                     reinterpret_cast<const bf16x8*>(k.data_ptr()),
                     reinterpret_cast<const bf16x8*>(v.data_ptr()),
                     reinterpret_cast<bf16x8*>(key_cache.data_ptr()),
                     reinterpret_cast<bf16x8*>(value_cache.data_ptr()),
                     slot_mapping.data_ptr<int>(), row_vecs);
  HIP_CHECK_LAST();
}
