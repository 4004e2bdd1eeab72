// Decode weights of an adapted projection: out = W + scale * B A, (N, K) bf16,
// B (N, r), A (r, K), the sum in fp32 and rounded once. Refreshed once per
// generation, for every projection of the model.
//
// One read of W and one write of out, 16 B a lane; B A comes from MFMA
// 16x16x32 on the way (one product per 16 x 16 x 32 of r): A's tile lies in
// LDS and is read transposed, with the columns of two products interleaved so
// that a lane ends up with 8 consecutive k of one row. Bound: memory; the
// eight loads of a row's 256 columns are all in flight before the products
// (two at a time: 8.6 us where this takes 5.0, a chain of waits).
// As torch operations (fp32 product, two conversions, scale, sum, concatenation
// and copy into the captured storage) the 7B model's refresh took 44 ms,
// 13 ms with two loads in flight; 61 us for a projection of 18944 x 3584, of
// which a copy of that size takes 55.
//
// The same kernel adds an adapter's output to the rows of a product, in place (the
// prompt phase): y += scale * u B^T (TA: A given as (K, r), staged as it lies) and
// y += scale * u A. r 32, rows x columns, the library's addmm against this, us:
// 128 x 896 3.9 and 5.3, 2408 x 3584 10 and 12, 2408 x 18944 41 and 40, 4816 x 3584
// 160 and 19; the library's call costs 19 us of host time and this one 4.
// And it joins adapter, bias and residual to an fp32 product of large weights, rounded
// once (the learner's short micro-batches): 308 x 18944 11.8 us, 2008 x 18944 54 us,
// 4.2 TB/s.
#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>
#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16v8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16v4;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((address_space(3))) bf16v4 lds_bf16v4;

namespace {

constexpr int KC = 256;            // columns of a workgroup
constexpr int STEPS = KC / 32;     // loads of W in flight

// w (bf16, or fp32 sums) and out may be one; res (or none) is added to the same
// sum. Rows of w are ldw elements apart, of out ldo, of b ldb, of res ldr (zero: one
// for all). TA: a is (K, r). TILES: out in tiles of 32 rows x 16 of K, [K half][row][8
// elements], row n of w at row + n of out, or (glu) at row + n in blocks of 16 of
// every 32; r may be 0.
template <bool TA, bool TILES, typename W>
DEV_INLINE void merge(const W* w, const __hip_bfloat16* __restrict__ a,
                      const __hip_bfloat16* __restrict__ b, const __hip_bfloat16* __restrict__ res,
                      __hip_bfloat16* out, int N, int K, int r, int rows, int64_t ldw, int64_t ldo,
                      int ldb, int64_t ldr, float scale, int row0, int glu, int bx, int by) {
  typedef __attribute__((ext_vector_type(8))) float f32x8;
  typedef std::conditional_t<std::is_same_v<W, float>, f32x8, bf16v8> WV;
  // A: [r32][KC], TA: [KC][r32], rows 16 B apart
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int RS = KC * 2 + 16;
  const int k0 = bx * KC, r32 = (r + 31) / 32 * 32;
  const int ts = r32 * 2 + 16;
  for (int i = threadIdx.x; i < r32 * (KC / 8); i += 256) {
    const int row = TA ? i / (r32 / 8) : i / (KC / 8), c = TA ? i % (r32 / 8) : i % (KC / 8);
    bf16v8 v;
    #pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = (__bf16)0.f;
    if (TA ? k0 + row < K && c * 8 < r : row < r && k0 + c * 8 < K)
      v = *reinterpret_cast<const bf16v8*>(TA ? a + (int64_t)(k0 + row) * r + c * 8
                                              : a + (int64_t)row * K + k0 + c * 8);
    *reinterpret_cast<bf16v8*>(smem + row * (TA ? ts : RS) + c * 16) = v;
  }
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = threadIdx.x & 63, g = l >> 4, lr = l & 15;
  const int end = min(N, (by + 1) * rows);
  for (int n0 = by * rows + wave * 16; n0 < end; n0 += 64) {
    const W* wrow = w + min(n0 + lr, N - 1) * ldw + g * 8;
    const __hip_bfloat16* brow = b + (int64_t)min(n0 + lr, N - 1) * ldb;
    WV wv[STEPS];
    #pragma unroll
    for (int i = 0; i < STEPS; ++i)                     // K % 32 == 0
      wv[i] = *reinterpret_cast<const WV*>(wrow + min(k0 + i * 32, K - 32));
    bf16v8 rv[STEPS];
    if (res) {
      #pragma unroll
      for (int i = 0; i < STEPS; ++i)
        rv[i] = *reinterpret_cast<const bf16v8*>(res + min(n0 + lr, N - 1) * ldr + g * 8 +
                                                 min(k0 + i * 32, K - 32));
    }
    f32x4 d[STEPS][2];
    #pragma unroll
    for (int i = 0; i < STEPS; ++i)
      d[i][0] = d[i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < r32; s += 32) {
      bf16v8 bv = *reinterpret_cast<const bf16v8*>(brow + min(s + g * 8, r - 8));
      if (s + g * 8 >= r) {                             // r % 8 == 0
        #pragma unroll
        for (int j = 0; j < 8; ++j) bv[j] = (__bf16)0.f;
      }
      #pragma unroll
      for (int i = 0; i < STEPS; ++i) {
        #pragma unroll
        for (int t = 0; t < 2; ++t) {
          // rows s + 8 g + 0..7 of A; lane i gets column 8 (i/4) + i%4 + 4 t
          bf16v8 av;
          if (TA) {
            const int k = i * 32 + (lr >> 2) * 8 + (lr & 3) + t * 4;
            av = *reinterpret_cast<const bf16v8*>(smem + k * ts + (s + g * 8) * 2);
          } else {
            char* p = smem + (s + g * 8 + (lr >> 2)) * RS + (i * 32 + (lr & 3) * 8 + t * 4) * 2;
            const bf16v4 x = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16v4*)p);
            const bf16v4 y = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16v4*)(p + 4 * RS));
            av = __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7);
          }
          d[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv, d[i][t], 0, 0, 0);
        }
      }
    }
    #pragma unroll
    for (int i = 0; i < STEPS; ++i) {
      bf16v8 o;
      #pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float t = (float)wv[i][j] + scale * d[i][j >> 2][j & 3];
        o[j] = (__bf16)(res ? t + (float)rv[i][j] : t);
      }
      if (n0 + lr < N && k0 + i * 32 < K) {
        const int n = n0 + lr, k = k0 + i * 32 + g * 8, row = row0 + (glu ? n + (n & ~15) : n);
        const int64_t at = TILES ? (int64_t)(row >> 5) * K * 32 + (k >> 4) * 512 + (k & 8) * 32 +
                                       (row & 31) * 8
                                 : n * ldo + k;
        *reinterpret_cast<bf16v8*>(out + at) = o;
      }
    }
  }
}

template <bool TA, typename W = __hip_bfloat16>
__global__ __launch_bounds__(256)
void lora_merge_kernel(const W* w, const __hip_bfloat16* __restrict__ a,
                       const __hip_bfloat16* __restrict__ b, const __hip_bfloat16* __restrict__ res,
                       __hip_bfloat16* out, int N, int K, int r, int rows, int64_t ldw, int64_t ldo,
                       int ldb, int64_t ldr, float scale) {
  merge<TA, false, W>(w, a, b, res, out, N, K, r, rows, ldw, ldo, ldb, ldr, scale, 0, 0, blockIdx.x,
                      blockIdx.y);
}

// Weights into tiles, several of them a launch: a layer's seven. A launch each left the
// chip idle in between, where the host was the slower (0.5B, 168 of 6 us), and behind
// the small ones (7B, of 7 to 70 us). Whole calls, their fan-out in one launch a prompt
// in both: 160 candidates of the 7B model 167.0 -> 162.7 ms, 32 of the 4B 79.3 -> 78.3,
// one of the 0.5B 35.7 -> 35.3.
constexpr int JOBS = 8;

struct Job {
  const __hip_bfloat16 *w, *a, *b;
  __hip_bfloat16* out;
  int64_t ldw;
  int N, K, r, rows, ldb, row0, glu, first;    // first: of the launch's workgroups
  float scale;
};
struct Jobs {
  Job job[JOBS];
  int n;
};

__global__ __launch_bounds__(256)
void weight_tiles_kernel(const Jobs jobs) {
  int i = 0;
  while (i + 1 < jobs.n && (int)blockIdx.x >= jobs.job[i + 1].first) ++i;
  const Job& j = jobs.job[i];
  const int at = blockIdx.x - j.first, wide = CDIV(j.K, KC);
  merge<false, true, __hip_bfloat16>(j.w, j.a, j.b, nullptr, j.out, j.N, j.K, j.r, j.rows, j.ldw, j.K,
                                     j.ldb, 0, j.scale, j.row0, j.glu, at % wide, at / wide);
}

}  // namespace

static bool lora_merge_takes(int64_t K, int64_t r) { return K % 32 == 0 && r % 8 == 0 && r >= 8 && r <= 128; }

namespace {

const __hip_bfloat16* lptr(const torch::Tensor& t) {
  return reinterpret_cast<const __hip_bfloat16*>(t.data_ptr());
}

// rows of a (rows, columns) operand that 16 B accesses can walk
bool lrows(const torch::Tensor& t, at::ScalarType type = at::kBFloat16) {
  return t.is_cuda() && t.scalar_type() == type && t.dim() == 2 && t.stride(1) == 1 &&
         t.stride(0) % 8 == 0 && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
}

// out = w + scale * b a, or b a^T (ta), then + res; w bf16 or fp32; false: not these
// operands
bool launch_merge(const torch::Tensor& w, const torch::Tensor& a, const torch::Tensor& b,
                  const torch::Tensor& out, bool ta, double scale,
                  const c10::optional<torch::Tensor>& res = c10::nullopt) {
  if (w.dim() != 2 || a.dim() != 2 || b.dim() != 2) return false;
  const int N = w.size(0), K = w.size(1), r = b.size(1);
  const bool sums = w.scalar_type() == at::kFloat;
  if (!lora_merge_takes(K, r) || (ta ? a.size(0) : a.size(1)) != K ||
      (ta ? a.size(1) : a.size(0)) != r || b.size(0) != N || out.sizes() != w.sizes() ||
      !lrows(w, sums ? at::kFloat : at::kBFloat16) || !lrows(b) || !lrows(out) || !lrows(a) ||
      !a.is_contiguous() || (!sums && w.stride(0) != out.stride(0)))
    return false;
  if (N > 1 && out.stride(0) < K) return false;         // rows over one another
  if (res && (!lrows(*res) || res->sizes() != w.sizes())) return false;
  if (N == 0) return true;
  // 4096 tiles fill the chip eight deep: then a staged A serves four turns,
  // below that every 64 rows get a workgroup of their own.
  const int rows = (int64_t)CDIV(K, KC) * CDIV(N, 64) >= 4096 ? 256 : 64;
  const dim3 grid(CDIV(K, KC), CDIV(N, rows)), block(256);
  auto stream = at::cuda::getCurrentCUDAStream();
  const int r32 = (r + 31) / 32 * 32, smem = ta ? KC * (r32 * 2 + 16) : r32 * (KC * 2 + 16);
  auto go = [&](auto kernel, auto* from) {
    hipLaunchKernelGGL(kernel, grid, block, smem, stream, from, lptr(a), lptr(b),
                       res ? lptr(*res) : nullptr,
                       reinterpret_cast<__hip_bfloat16*>(out.data_ptr()), N, K, r, rows,
                       w.stride(0), out.stride(0), (int)b.stride(0), res ? res->stride(0) : 0,
                       (float)scale);
  };
  if (sums) {
    const float* p = w.data_ptr<float>();
    if (ta) go(lora_merge_kernel<true, float>, p);
    else go(lora_merge_kernel<false, float>, p);
  } else if (ta) {
    go(lora_merge_kernel<true>, lptr(w));
  } else {
    go(lora_merge_kernel<false>, lptr(w));
  }
  HIP_CHECK_LAST();
  return true;
}

}  // namespace

// out = w + scale * b a. False, and nothing done, for operands that 16 B
// accesses or the tiles can't take.
bool lora_merge(torch::Tensor w, torch::Tensor a, torch::Tensor b, torch::Tensor out, double scale) {
  return launch_merge(w, a, b, out, false, scale);
}

namespace {

// Job into `to`; false for operands that 16 B accesses can't take.
bool tiles_job(Job& to, const torch::Tensor& w, const torch::Tensor& out, int64_t row, bool glu,
               const c10::optional<torch::Tensor>& a, const c10::optional<torch::Tensor>& b,
               double scale) {
  TORCH_CHECK(out.is_cuda() && out.is_contiguous() && out.dim() == 2 &&
              out.scalar_type() == at::kBFloat16 && out.size(0) % 32 == 0);
  if (w.dim() != 2 || !lrows(w) || w.size(1) != out.size(1) || w.size(1) % 32 != 0) return false;
  const int N = w.size(0), K = w.size(1);
  TORCH_CHECK(row >= 0 && (glu ? (row == 0 || row == 16) && N % 16 == 0 && 2 * N == out.size(0)
                               : row + N <= out.size(0)),
              "weight_tiles: rows past the end");
  TORCH_CHECK(reinterpret_cast<uintptr_t>(out.data_ptr()) % 16 == 0);
  int r = 0;
  if (a) {
    TORCH_CHECK(b.has_value());
    if (a->dim() != 2 || b->dim() != 2 || !lrows(*a) || !a->is_contiguous() || !lrows(*b))
      return false;
    r = a->size(0);
    TORCH_CHECK(a->size(1) == K && b->size(0) == N && b->size(1) == r, "weight_tiles: adapter");
    if (!lora_merge_takes(K, r)) return false;
  }
  const int rows = (int64_t)CDIV(K, KC) * CDIV(N, 64) >= 4096 ? 256 : 64;
  to = {lptr(w), r ? lptr(*a) : nullptr, r ? lptr(*b) : nullptr,
        reinterpret_cast<__hip_bfloat16*>(out.data_ptr()), w.stride(0), N, K, r, rows,
        r ? (int)b->stride(0) : 0, (int)row, (int)glu, 0, (float)scale};
  return true;
}

void launch_tiles(Jobs& jobs) {
  int64_t blocks = 0;
  int r32 = 0;
  for (int i = 0; i < jobs.n; ++i) {
    Job& j = jobs.job[i];
    j.first = (int)blocks;
    blocks += (int64_t)CDIV(j.K, KC) * CDIV(j.N, j.rows);
    r32 = std::max(r32, CDIV(j.r, 32) * 32);
  }
  if (blocks == 0) return;
  TORCH_CHECK(blocks < (1 << 30), "weight_tiles: size");
  hipLaunchKernelGGL(weight_tiles_kernel, dim3(blocks), dim3(256), r32 * (KC * 2 + 16),
                     at::cuda::getCurrentCUDAStream(), jobs);
  HIP_CHECK_LAST();
}

}  // namespace

// Of each weight: rows row .. of out, a weight in tiles ((rows, K), K % 32 == 0, see the
// kernel) <- w, or w + scale * b a. glu: w is gate (row 0) or up (row 16) of a SiLU*mul
// pair. False, and nothing done, where 16 B accesses can't take an operand.
bool weights_tiles(std::vector<torch::Tensor> w, std::vector<torch::Tensor> out,
                   std::vector<int64_t> row, std::vector<bool> glu,
                   std::vector<c10::optional<torch::Tensor>> a,
                   std::vector<c10::optional<torch::Tensor>> b, std::vector<double> scale) {
  const size_t n = w.size();
  TORCH_CHECK(out.size() == n && row.size() == n && glu.size() == n && a.size() == n &&
              b.size() == n && scale.size() == n, "weight_tiles: lists");
  std::vector<Jobs> all(CDIV(n, JOBS));
  for (size_t i = 0; i < n; ++i) {
    Jobs& to = all[i / JOBS];
    to.n = (int)(i % JOBS) + 1;
    if (!tiles_job(to.job[i % JOBS], w[i], out[i], row[i], glu[i], a[i], b[i], scale[i])) return false;
  }
  for (auto& jobs : all) launch_tiles(jobs);
  return true;
}

// y (M, N) += scale * u (M, r) m (r, N), then + res if given: one rounding for
// all of it. m as it lies or a transposed view, rows of y, u and res in any
// strides of whole 16 bytes. False, and nothing done, for other operands: the
// caller takes the library's product.
bool lora_add(torch::Tensor y, torch::Tensor u, torch::Tensor m, double scale,
              c10::optional<torch::Tensor> res) {
  if (m.dim() != 2) return false;
  const bool ta = m.stride(1) != 1;
  return launch_merge(y, ta ? m.t() : m, u, y, ta, scale, res);
}

// out (M, N) bf16 = y (M, N) fp32 + u m + res if given (rows that may be one), rounded
// once; otherwise as lora_add.
bool lora_join(torch::Tensor y, torch::Tensor u, torch::Tensor m, torch::Tensor out,
               c10::optional<torch::Tensor> res) {
  const bool ta = m.stride(1) != 1;
  return y.scalar_type() == at::kFloat && launch_merge(y, ta ? m.t() : m, u, out, ta, 1., res);
}

// ---- base and adapter weights as one matrix, so that one product does both:
// [x | u] [W | B]^T and [dY | du] [W; A], the adapter's sum in the product's fp32.
// The second is laid out transposed, (K, rows): the library's products of two
// row-major operands with K innermost are its faster ones (18793 rows, GPU time as
// it lies -> transposed: 1568 x 8960 585 -> 476 us, 2144 x 1536 133 -> 100,
// 3616 x 18944 2185 -> 1906).
namespace {

struct Parts {
  const __hip_bfloat16 *w[3], *b[3];
  int row[4], col[4];                   // first row and adapter column of each, and the ends
  int n;
};

// 16 B a thread: (rows, K + pad), zeros where a row has another projection's columns
__global__ __launch_bounds__(256)
void adapted_weight_kernel(Parts q, __hip_bfloat16* __restrict__ out, int K, int pad) {
  const int cpr = (K + pad) / 8;
  const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x, row = id / cpr;
  const int c = (int)(id % cpr) * 8;
  if (row >= q.row[q.n]) return;
  int i = 0;
  while (i + 1 < q.n && row >= q.row[i + 1]) ++i;
  bf16x8 v;
  if (c < K) {
    v = *reinterpret_cast<const bf16x8*>(q.w[i] + (row - q.row[i]) * K + c);
  } else {
    const int r = q.col[i + 1] - q.col[i];
    #pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int k = c - K + j - q.col[i];
      v.v[j] = k >= 0 && k < r ? q.b[i][(row - q.row[i]) * r + k] : f2bf(0.f);
    }
  }
  *reinterpret_cast<bf16x8*>(out + id * 8) = v;
}

constexpr int STACK = 6, TT = 64;

struct Stack {
  const __hip_bfloat16* w[STACK];
  int at[STACK], rows[STACK];
  int n;
};

// A 64 x 64 tile through LDS, 16 B a thread on both sides. grid (columns / 64, K / 64)
__global__ __launch_bounds__(256)
void stack_transposed_kernel(Stack q, __hip_bfloat16* __restrict__ out, int K, int cols) {
  __shared__ __hip_bfloat16 tile[TT][TT + 2];
  const int n0 = blockIdx.x * TT, k0 = blockIdx.y * TT;
  #pragma unroll
  for (int u = threadIdx.x; u < TT * (TT / 8); u += 256) {
    const int n = n0 + u / 8, k = k0 + u % 8 * 8;
    bf16x8 v;
    #pragma unroll
    for (int j = 0; j < 8; ++j) v.v[j] = f2bf(0.f);
    if (k < K)
      for (int i = 0; i < q.n; ++i)
        if (n >= q.at[i] && n < q.at[i] + q.rows[i])
          v = *reinterpret_cast<const bf16x8*>(q.w[i] + (int64_t)(n - q.at[i]) * K + k);
    #pragma unroll
    for (int j = 0; j < 8; ++j) tile[u / 8][u % 8 * 8 + j] = v.v[j];
  }
  __syncthreads();
  #pragma unroll
  for (int u = threadIdx.x; u < TT * (TT / 8); u += 256) {
    // neighbouring threads, neighbouring k: their columns of the tile lie in
    // different banks
    const int k = u % TT, c = u / TT * 8;
    bf16x8 v;
    #pragma unroll
    for (int j = 0; j < 8; ++j) v.v[j] = tile[c + j][k];
    if (k0 + k < K && n0 + c < cols)
      *reinterpret_cast<bf16x8*>(out + (int64_t)(k0 + k) * cols + n0 + c) = v;
  }
}

torch::Tensor dense16(const torch::Tensor& t) {
  TORCH_CHECK(t.is_cuda() && t.dim() == 2 && t.scalar_type() == at::kBFloat16);
  auto c = t.contiguous();
  return reinterpret_cast<uintptr_t>(c.data_ptr()) % 16 == 0 ? c : c.clone();
}

}  // namespace

// [W | B] of up to three projections of one input, one below the other: w[i] (N_i,
// K), b[i] (N_i, r_i) from the column where the last one's ended; pad columns
// beside K, at least the ranks' sum; K and pad multiples of 8.
torch::Tensor adapted_weight(std::vector<torch::Tensor> w, std::vector<torch::Tensor> b,
                             int64_t pad) {
  const int n = (int)w.size(), K = (int)w.at(0).size(1);
  TORCH_CHECK(n <= 3 && b.size() == w.size() && K % 8 == 0 && pad % 8 == 0);
  Parts q{};
  q.n = n;
  for (int i = 0; i < n; ++i) {
    w[i] = dense16(w[i]);
    b[i] = dense16(b[i]);
    TORCH_CHECK(w[i].size(1) == K && b[i].size(0) == w[i].size(0), "adapted_weight: shape mismatch");
    q.w[i] = lptr(w[i]);
    q.b[i] = lptr(b[i]);
    q.row[i + 1] = q.row[i] + w[i].size(0);
    q.col[i + 1] = q.col[i] + b[i].size(1);
  }
  TORCH_CHECK(q.col[n] <= pad);
  auto out = torch::empty({q.row[n], K + pad}, w[0].options());
  if (out.numel() == 0) return out;
  hipLaunchKernelGGL(adapted_weight_kernel, dim3(CDIV(out.numel() / 8, 256)), dim3(256), 0,
                     at::cuda::getCurrentCUDAStream(), q,
                     reinterpret_cast<__hip_bfloat16*>(out.data_ptr()), K, (int)pad);
  HIP_CHECK_LAST();
  return out;
}

// (K, cols): w[i]^T, (rows_i, K) each, from column at[i] on, zeros elsewhere; K and
// cols multiples of 8.
torch::Tensor stack_transposed(std::vector<torch::Tensor> w, std::vector<int64_t> at,
                               int64_t cols) {
  const int n = (int)w.size(), K = (int)w.at(0).size(1);
  TORCH_CHECK(n <= STACK && at.size() == w.size() && K % 8 == 0 && cols % 8 == 0);
  Stack q{};
  q.n = n;
  for (int i = 0; i < n; ++i) {
    w[i] = dense16(w[i]);
    TORCH_CHECK(w[i].size(1) == K && at[i] >= 0 && at[i] + w[i].size(0) <= cols,
                "stack_transposed: shape mismatch");
    q.w[i] = lptr(w[i]);
    q.at[i] = (int)at[i];
    q.rows[i] = w[i].size(0);
  }
  auto out = torch::empty({K, cols}, w[0].options());
  if (out.numel() == 0) return out;
  hipLaunchKernelGGL(stack_transposed_kernel, dim3(CDIV(cols, TT), CDIV(K, TT)), dim3(256), 0,
                     at::cuda::getCurrentCUDAStream(), q,
                     reinterpret_cast<__hip_bfloat16*>(out.data_ptr()), K, (int)cols);
  HIP_CHECK_LAST();
  return out;
}
