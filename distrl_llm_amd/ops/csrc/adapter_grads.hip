// Gradients of LoRA adapters over a micro-batch: C = P^T Y for some (rows, N)
// operands Y with their (rows, r) operands P, r <= 128: dB^T = u^T dY for every
// adapted projection, dA = du^T x for every input.
//
// These products sum over the rows, have next to no output, and only read Y. The
// library ran them as products of a few tiles with little of K split: 18800 rows,
// 1536 columns, r 32 70 us, r 96 101, where reading Y takes 12; 8960 columns
// 117 and 160 us where it takes 69. Here one launch does all of a layer half's
// (six or five): a workgroup owns 128 columns of one Y and a share of the rows,
// 64 rows a step through LDS, both operands read transposed (LDS transpose
// reads); shares of the rows give fp32 partial sums, added up in a fixed order
// by a second launch, so results do not depend on the order of workgroups.
// Bound: HBM, Y read once.
#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>
#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16v8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16v4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((address_space(3))) bf16v4 lds_bf16v4;

namespace {

constexpr int JOBS = 6, COLS = 128, ROWS = 64;

struct Job {
  const __hip_bfloat16 *y, *p;
  __hip_bfloat16* out;      // (r, N), or (N, r) if by_col
  int64_t ldy, ldp, at;     // at: first element of its partial sums in a share
  int N, r, by_col, block;  // block: its first workgroup (of the sum: thread / 256)
};

struct Jobs { Job j[JOBS]; int n; };

// 16 B chunk c of a tile's row, rows of 256 B: 8 rows read at one chunk and 4
// rows over 64 B (transpose reads) fall into different banks
DEV_INLINE int chunk(int row, int c) {
  return row * 256 + ((c ^ (((row & 3) << 2) | ((row >> 2) & 3))) << 4);
}

// element column dt * 32 + (l & 31), rows k0 + {4h.., 8 + 4h..}, h = l / 32
DEV_INLINE bf16v8 column(char* lds, int k0, int dt) {
  const int l = threadIdx.x & 63, h = l >> 5;
  const int x = dt * 4 + ((l >> 4) & 1) * 2 + ((l & 3) >> 1);
  const int r0 = k0 + 4 * h + ((l & 15) >> 2), e = (l & 1) * 8;
  const bf16v4 a = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16v4*)(lds + chunk(r0, x) + e));
  const bf16v4 b = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16v4*)(lds + chunk(r0 + 8, x) + e));
  return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
}

template <int RT>       // 32 columns of P each
DEV_INLINE void share_sum(const Job& job, float* part, char* ty, char* tp, int n0, int64_t r0,
                          int64_t r1) {
  const int tid = threadIdx.x, l = tid & 63, h = l >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  f32x16 acc[RT];
  #pragma unroll
  for (int t = 0; t < RT; ++t)
    #pragma unroll
    for (int i = 0; i < 16; ++i) acc[t][i] = 0.f;
  u32x4 yv[4], pv[RT];
  bool live = false;
  const u32x4 zero = {0, 0, 0, 0};
  // rows past the end repeat the last one with weight zero. The next step's rows
  // are fetched before this one's products and only looked at when they are stored:
  // cleared where they were fetched, and sunk behind the products by the compiler,
  // they were waited for in every step (18793 rows, feed-forward half of 1536 and
  // 8960 columns: 283 us, 263 now)
  const int yc = tid & 15, ycol = min(n0 + yc * 8, job.N - 8);
  auto fetch = [&](int64_t row) {
    #pragma unroll
    for (int i = 0; i < 4; ++i)
      yv[i] = *reinterpret_cast<const u32x4*>(job.y + min(row + (tid >> 4) + i * 16, r1 - 1) * job.ldy +
                                              ycol);
    #pragma unroll
    for (int i = 0; i < RT; ++i) {
      const int c = i * 32 + (tid & 3) * 8;
      pv[i] = *reinterpret_cast<const u32x4*>(job.p + min(row + (tid >> 2), r1 - 1) * job.ldp +
                                              min(c, job.r - 8));
    }
    live = row + (tid >> 2) < r1;
  };
  fetch(r0);
  for (int64_t row = r0; row < r1; row += ROWS) {
    __syncthreads();
    #pragma unroll
    for (int i = 0; i < 4; ++i)
      *reinterpret_cast<u32x4*>(ty + chunk((tid >> 4) + i * 16, yc)) = yv[i];
    #pragma unroll
    for (int i = 0; i < RT; ++i)
      *reinterpret_cast<u32x4*>(tp + chunk(tid >> 2, i * 4 + (tid & 3))) =
          live && i * 32 + (tid & 3) * 8 < job.r ? pv[i] : zero;
    __syncthreads();
    if (row + ROWS < r1) fetch(row + ROWS);
    __builtin_amdgcn_sched_barrier(0);
    #pragma unroll
    for (int k = 0; k < ROWS; k += 16) {
      const bf16v8 y = column(ty, k, wave);
      #pragma unroll
      for (int t = 0; t < RT; ++t)
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(column(tp, k, t), y, acc[t], 0, 0, 0);
    }
  }
  // column n of Y, rows 8 (i / 4) + 4 h + i % 4 of C
  const int n = n0 + wave * 32 + (l & 31);
  if (n >= job.N) return;
  #pragma unroll
  for (int t = 0; t < RT; ++t)
    #pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int r = t * 32 + 8 * (i >> 2) + 4 * h + (i & 3);
      if (r < job.r) part[(int64_t)r * job.N + n] = acc[t][i];
    }
}

// grid (workgroups of all jobs' columns, shares of the rows)
__global__ __launch_bounds__(256, 2)
void adapter_grads_kernel(Jobs jobs, float* __restrict__ part, int64_t rows, int64_t share) {
  __shared__ __attribute__((aligned(16))) char tiles[2 * ROWS * 256];
  int i = 0;
  while (i + 1 < jobs.n && (int)blockIdx.x >= jobs.j[i + 1].block) ++i;
  const Job job = jobs.j[i];
  const int steps = (int)((rows + ROWS - 1) / ROWS), S = gridDim.y, s = blockIdx.y;
  const int64_t r0 = (int64_t)s * steps / S * ROWS;
  const int64_t r1 = min((int64_t)(s + 1) * steps / S * ROWS, rows);
  float* p = part + s * share + job.at;
  const int n0 = ((int)blockIdx.x - job.block) * COLS;
  char* tp = tiles + ROWS * 256;
  if (job.r <= 32) share_sum<1>(job, p, tiles, tp, n0, r0, r1);
  else if (job.r <= 64) share_sum<2>(job, p, tiles, tp, n0, r0, r1);
  else if (job.r <= 96) share_sum<3>(job, p, tiles, tp, n0, r0, r1);
  else share_sum<4>(job, p, tiles, tp, n0, r0, r1);
}

// Adds the shares up: eight neighbours of the output a thread.
__global__ __launch_bounds__(256)
void adapter_sum_kernel(Jobs jobs, const float* __restrict__ part, int64_t share, int S) {
  int i = 0;
  while (i + 1 < jobs.n && (int)blockIdx.x >= jobs.j[i + 1].block) ++i;
  const Job job = jobs.j[i];
  const int id = ((int)blockIdx.x - job.block) * 256 + threadIdx.x;
  if (id >= job.N * (job.r / 8)) return;
  float v[8];
  #pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = 0.f;
  const float* p = part + job.at;
  __hip_bfloat16* o;
  if (job.by_col) {
    const int n = id % job.N, r = id / job.N * 8;     // neighbouring threads, neighbouring n
    for (int s = 0; s < S; ++s)
      #pragma unroll
      for (int j = 0; j < 8; ++j) v[j] += p[s * share + (int64_t)(r + j) * job.N + n];
    o = job.out + (int64_t)n * job.r + r;
  } else {
    add_parts8(v, p + (int64_t)id * 8, share, S);
    o = job.out + (int64_t)id * 8;
  }
  bf16x8 x;
  #pragma unroll
  for (int j = 0; j < 8; ++j) x.v[j] = f2bf(v[j]);
  *reinterpret_cast<bf16x8*>(o) = x;
}

// rows of a (rows, columns) operand that 16 B accesses can walk
torch::Tensor walkable(const torch::Tensor& t) {
  TORCH_CHECK(t.is_cuda() && t.dim() == 2 && t.scalar_type() == at::kBFloat16);
  const bool ok = t.stride(1) == 1 && t.stride(0) % 8 == 0 &&
                  reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  return ok ? t : t.clone(at::MemoryFormat::Contiguous);
}

}  // namespace

// p[i]^T y[i] (r, N), or with by_col its transpose (N, r), of y (rows, N) and p
// (rows, r), N and r multiples of 8, r <= 128; the sums over the rows in fp32.
std::vector<torch::Tensor> adapter_grads(std::vector<torch::Tensor> y, std::vector<torch::Tensor> p,
                                         std::vector<int64_t> by_col) {
  const int n = (int)y.size();
  TORCH_CHECK(n >= 1 && n <= JOBS && p.size() == y.size() && by_col.size() == y.size());
  const int64_t rows = y[0].size(0);
  Jobs jobs{};
  jobs.n = n;
  std::vector<torch::Tensor> out;
  int cols = 0, sums = 0;
  int64_t share = 0;
  Jobs sum{};
  for (int i = 0; i < n; ++i) {
    y[i] = walkable(y[i]);
    p[i] = walkable(p[i]);
    const int N = y[i].size(1), r = p[i].size(1);
    TORCH_CHECK(y[i].size(0) == rows && p[i].size(0) == rows && N >= 8 && N % 8 == 0 && r >= 8 &&
                r % 8 == 0 && r <= 128, "adapter_grads: unsupported shape");
    out.push_back(by_col[i] ? torch::empty({N, r}, y[i].options())
                            : torch::empty({r, N}, y[i].options()));
    jobs.j[i] = {reinterpret_cast<const __hip_bfloat16*>(y[i].data_ptr()),
                 reinterpret_cast<const __hip_bfloat16*>(p[i].data_ptr()),
                 reinterpret_cast<__hip_bfloat16*>(out[i].data_ptr()), y[i].stride(0),
                 p[i].stride(0), share, N, r, (int)by_col[i], cols};
    sum.j[i] = jobs.j[i];
    sum.j[i].block = sums;
    cols += CDIV(N, COLS);
    sums += CDIV(N * (r / 8), 256);
    share += (int64_t)N * r;
  }
  sum.n = n;
  if (rows == 0) {
    for (auto& t : out) t.zero_();
    return out;
  }
  // four workgroups a CU, none under two steps
  const int64_t steps = CDIV(rows, ROWS);
  const int S = (int)std::max<int64_t>(1, std::min<int64_t>(1024 / cols, steps / 2));
  auto part = torch::empty({S * share}, y[0].options().dtype(at::kFloat));
  auto stream = at::cuda::getCurrentCUDAStream();
  hipLaunchKernelGGL(adapter_grads_kernel, dim3(cols, S), dim3(256), 0, stream, jobs,
                     part.data_ptr<float>(), rows, share);
  hipLaunchKernelGGL(adapter_sum_kernel, dim3(sums), dim3(256), 0, stream, sum,
                     part.data_ptr<float>(), share, S);
  HIP_CHECK_LAST();
  return out;
}
