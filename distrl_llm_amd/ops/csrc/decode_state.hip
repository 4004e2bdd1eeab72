// State of a decode session's sequences between steps: where the next token's key
// and value go, and what a sampled token does to its sequence.
//
// As torch operations this was some twenty launches a step over a few hundred
// bytes, one behind the other: 90 us of a step's 980 for one sequence of the 0.5B
// model. Bound: the two launches that are left, ~4 us each.
#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>
#include "common.h"

namespace {

__global__ __launch_bounds__(256)
void decode_slots_kernel(const int64_t* __restrict__ positions, const int* __restrict__ tables,
                         int64_t* __restrict__ slots, int* __restrict__ pos32, int N, int max_nb,
                         int block_size) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= N) return;
  const int pos = (int)positions[i];
  // no further than the table reaches
  const int b = min(max(pos / block_size, 0), max_nb - 1);
  slots[i] = (int64_t)tables[(int64_t)i * max_nb + b] * block_size + pos % block_size;
  pos32[i] = pos;
}

// One workgroup: every sequence reads the step before it is counted up.
__global__ __launch_bounds__(256)
void decode_advance_kernel(const int64_t* __restrict__ sampled, int64_t* __restrict__ tokens,
                           int64_t* __restrict__ positions, int* __restrict__ ctx_lens,
                           const int64_t* __restrict__ limits, bool* __restrict__ finished,
                           int64_t* __restrict__ step, int64_t* __restrict__ out, int64_t rows,
                           int N, int64_t eos, int has_eos) {
  const int64_t s = *step;
  for (int i = threadIdx.x; i < N; i += 256) {
    const int64_t t = sampled[i], p = positions[i];
    const bool was = finished[i];
    if (s >= 0 && s < rows) out[s * N + i] = t;
    finished[i] = was || p + 1 >= limits[i] || (has_eos && t == eos);
    if (!was) {
      tokens[i] = t;
      positions[i] = p + 1;
      ctx_lens[i] += 1;
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) *step = s + 1;
}

void check_state(const torch::Tensor& t, at::ScalarType type, int64_t n) {
  TORCH_CHECK(t.is_cuda() && t.is_contiguous() && t.scalar_type() == type && t.numel() == n,
              "decode state: type, size or layout");
}

}  // namespace

// Cache rows of the tokens at positions (N,), from block tables (N, pages), and
// the positions as int32.
std::vector<torch::Tensor> decode_slots(torch::Tensor positions, torch::Tensor tables,
                                        int64_t block_size) {
  const int64_t N = positions.numel();
  check_state(positions, at::kLong, N);
  TORCH_CHECK(tables.dim() == 2 && tables.size(0) == N && tables.size(1) > 0 && block_size > 0);
  check_state(tables, at::kInt, N * tables.size(1));
  auto slots = torch::empty({N}, positions.options());
  auto pos32 = torch::empty({N}, tables.options());
  if (N > 0)
    hipLaunchKernelGGL(decode_slots_kernel, dim3(CDIV(N, 256)), dim3(256), 0,
                       at::cuda::getCurrentCUDAStream(), positions.data_ptr<int64_t>(),
                       tables.data_ptr<int>(), slots.data_ptr<int64_t>(), pos32.data_ptr<int>(),
                       (int)N, (int)tables.size(1), (int)block_size);
  HIP_CHECK_LAST();
  return {slots, pos32};
}

// What the tokens sampled in a step do to the session, in place: they are row
// `step` of out; a sequence that goes on moves to its token; it ends at its limit
// or with eos.
void decode_advance(torch::Tensor sampled, torch::Tensor tokens, torch::Tensor positions,
                    torch::Tensor ctx_lens, torch::Tensor limits, torch::Tensor finished,
                    torch::Tensor step, torch::Tensor out, c10::optional<int64_t> eos) {
  const int64_t N = tokens.numel();
  for (const auto& t : {sampled, tokens, positions, limits}) check_state(t, at::kLong, N);
  check_state(ctx_lens, at::kInt, N);
  check_state(finished, at::kBool, N);
  check_state(step, at::kLong, 1);
  TORCH_CHECK(out.dim() == 2 && out.size(1) == N);
  check_state(out, at::kLong, out.numel());
  hipLaunchKernelGGL(decode_advance_kernel, dim3(1), dim3(256), 0,
                     at::cuda::getCurrentCUDAStream(), sampled.data_ptr<int64_t>(),
                     tokens.data_ptr<int64_t>(), positions.data_ptr<int64_t>(),
                     ctx_lens.data_ptr<int>(), limits.data_ptr<int64_t>(),
                     finished.data_ptr<bool>(), step.data_ptr<int64_t>(), out.data_ptr<int64_t>(),
                     out.size(0), (int)N, eos.value_or(0), (int)eos.has_value());
  HIP_CHECK_LAST();
}
