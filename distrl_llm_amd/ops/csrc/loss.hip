// Fused log-prob + PG/GRPO loss over the 152k vocab:
// forward emits per-token log p(target) + the row LSE in a
// single online-logsumexp streaming pass (never materializing a (B,T,V)
// log-prob tensor — the reference loops rows through log_softmax+gather,
// distributed_actor.py:253-260); backward emits dlogits directly:
// dlogits_v = w * (1[v=target] - softmax_v), w = mask*coef*dloss.
// Where a gradient is wanted, both are one pass over logits that a workgroup's registers
// hold (loss_both_kernel).
#include <torch/extension.h>
#include <ATen/SavedTensorHooks.h>
#include <ATen/cuda/CUDAContext.h>
#include "common.h"

typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16v2;

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

// A target as an element of its row, -1 where it is none
DEV_INLINE int word_of(int64_t target, int V) { return target >= 0 && target < V ? (int)target : -1; }

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

// Workgroups that count themselves: in groups on cache lines of their own, then the groups.
// 2048 of them that end at once on one word took 17 us (8 x 600 x 4096 46 us, so 31).
constexpr int GROUPS = 32, LINE = 32, COUNTS = (GROUPS + 1) * LINE;

// Whether this one is the last; counts cleared, one thread of each
DEV_INLINE bool last_to_end(uint32_t* counts) {
  const uint32_t n = gridDim.x, groups = min((uint32_t)GROUPS, n), g = blockIdx.x % groups;
  return atomicAdd(counts + (g + 1) * LINE, 1u) == (n - g - 1) / groups &&
         atomicAdd(counts, 1u) == groups - 1;
}

// The row weights alone, ahead of a pass over logits that makes the gradient at once,
// whose every row would else read its sequence's whole mask. A workgroup a sequence.
// counts <- 0, for the workgroups of that pass.
template <typename M>
__global__ __launch_bounds__(1024)
void loss_weights_kernel(const M* __restrict__ mask, const float* __restrict__ rewards,
                         float* __restrict__ w, uint32_t* __restrict__ counts, int B, int T,
                         float scale) {
  __shared__ float red[16];
  const int64_t at = (int64_t)blockIdx.x * T;
  if (blockIdx.x == 0)
    for (int i = threadIdx.x; i < COUNTS; i += 1024) counts[i] = 0;
  float n = 0.f;
  for (int t = threadIdx.x; t < T; t += 1024) n += (float)mask[at + t];
  const float coef = -rewards[blockIdx.x] / fmaxf(block_sum(n, red), 1.f) / B * scale;
  for (int t = threadIdx.x; t < T; t += 1024) w[at + t] = (float)mask[at + t] * coef;
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
DEV_INLINE void loss_bwd_row(const T* __restrict__ logits,
                     const int64_t* __restrict__ targets,
                     const float* __restrict__ w,
                     const float* __restrict__ lse,
                     const float* __restrict__ dloss,   // scalar, or null: 1
                     T* __restrict__ dlogits, int V, int64_t row) {
  const T* lr = logits + row * V;
  T* dr = dlogits + row * V;
  const float wv = dloss ? w[row] * *dloss : w[row];
  const float l = lse[row];
  const int tgt = word_of(targets[row], V);
  if constexpr (std::is_same<T, __hip_bfloat16>::value) {
    const int nvec = V / 8;
    auto put = [&](int i, const bf16x8& v) {
      bf16x8 o;
      #pragma unroll
      for (int j = 0; j < 8; ++j) {
        float p = __expf(bf2f(v.v[j]) - l);
        o.v[j] = f2bf(wv * ((i * 8 + j == tgt ? 1.f : 0.f) - p));
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
        g = wv * ((i == tgt ? 1.f : 0.f) - __expf(ld(lr, i) - l));
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

template <typename T, int THREADS>
__global__ __launch_bounds__(THREADS)
void loss_bwd_kernel(const T* __restrict__ logits, const int64_t* __restrict__ targets,
                     const float* __restrict__ w, const float* __restrict__ lse,
                     const float* __restrict__ dloss, T* __restrict__ dlogits, int V) {
  loss_bwd_row<T, THREADS>(logits, targets, w, lse, dloss, dlogits, V,
                           (int64_t)gridDim.x - 1 - blockIdx.x);
}

// The same where dlogits holds the gradient for a dloss of 1 already: a few workgroups
// look whether it is that. What it costs where it is not, with the pass before it, us:
// 2400 rows of 152064 592 with rows from the first, 567 from the last (389 in two passes);
// 8000 of 32003 486, 440 (312). The gradient at hand can't be scaled instead: it is rounded.
template <typename T, int THREADS>
__global__ __launch_bounds__(THREADS)
void loss_anew_kernel(const T* __restrict__ logits, const int64_t* __restrict__ targets,
                      const float* __restrict__ w, const float* __restrict__ lse,
                      const float* __restrict__ dloss, T* __restrict__ dlogits, int V,
                      int64_t rows) {
  if (*dloss == 1.f) return;
  for (int64_t row = blockIdx.x; row < rows; row += gridDim.x)
    loss_bwd_row<T, THREADS>(logits, targets, w, lse, dloss, dlogits, V, rows - 1 - row);
}

// Rows' weights, or what they are made of and where they go
struct RowWeights {
  float* w;
  const void* mask;           // (B, T), int64 or fp32, or null: w is there
  bool mask64;
  const float* rewards;
  int B, T;
  float scale;
};

// Both passes at once, where the gradient will be asked for: a workgroup holds a row in
// registers, KEEP pieces of 8 values a thread, makes its log-sum-exp and writes the
// gradient for a dloss of 1, so that logits are read once. As a piece is written the
// next row's takes its registers: a workgroup walks rows, and reads and writes are on
// their way all the time. Bound by memory: 2408 rows of 152064, a quarter of weight zero,
// 308 us (4.75 TB/s read and written), 133 and 222 in two passes; with the sum over rows
// and the look at dloss 356 -> 315. Loads or stores through or past the caches are even.
// With loss and counts the rows' weighted sum is made here too: a workgroup's part of it goes
// through token_logp (an element a workgroup) to the last to end, which adds them up in
// their order.
template <int THREADS, int KEEP>
__global__ __launch_bounds__(THREADS)
void loss_both_kernel(const __hip_bfloat16* __restrict__ logits, const int64_t* __restrict__ targets,
                      RowWeights weights, float* __restrict__ token_logp,
                      float* __restrict__ lse_out, __hip_bfloat16* __restrict__ dlogits,
                      float* __restrict__ loss, uint32_t* __restrict__ counts, int rows, int V) {
  constexpr float LOG2E = 1.4426950408889634f;
  constexpr int NW = THREADS / WAVE;
  __shared__ float part[2][3][NW], ends[NW];
  __shared__ bool last;
  const int tid = threadIdx.x, lane = tid & (WAVE - 1), nvec = V / 8;
  u32x4 v[KEEP];
  // One offset that walks a row, as 19 addresses would take the registers: what lies past
  // the row's end reads as zero, is left out of the sums and not written.
  const int bytes = nvec * 16;
  auto row_at = [&](const __hip_bfloat16* p) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<__hip_bfloat16*>(p), 0, bytes, 0x00027000);
  };
  auto next = [&](int& off) {
    off += THREADS * 16;
    asm volatile("" : "+v"(off));
  };
  auto value = [&](int c, int j) {
    return __uint_as_float(j & 1 ? v[c][j / 2] & 0xffff0000u : v[c][j / 2] << 16);
  };
  float mine = 0.f;             // of the loss
  int64_t row = blockIdx.x;
  {
    const auto from = row_at(logits + row * V);
    int off = tid * 16;
    #pragma unroll
    for (int c = 0; c < KEEP; ++c, next(off)) v[c] = __builtin_amdgcn_raw_buffer_load_b128(from, off, 0, 0);
  }
  for (int turn = 0; row < rows; row += gridDim.x, turn ^= 1) {
    const __hip_bfloat16* lr = logits + row * V;
    __hip_bfloat16* dr = dlogits + row * V;
    const int tgt = word_of(targets[row], V);
    // the sequence's mask, summed beside the logits
    float share = 0.f;
    const int64_t seq = weights.mask ? row / weights.T : 0;
    auto mask = [&](int64_t i) {
      return weights.mask64 ? (float)reinterpret_cast<const int64_t*>(weights.mask)[i]
                            : reinterpret_cast<const float*>(weights.mask)[i];
    };
    if (weights.mask)
      for (int t = tid; t < weights.T; t += THREADS) share += mask(seq * weights.T + t);
    const int at = nvec * 8 + tid;                        // of the last few
    const float tail = at < V ? ld(lr, at) : -__builtin_inff();

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
    #pragma unroll
    for (int c = 0; c < KEEP; ++c) {
      if (c * THREADS >= nvec) continue;
      if (c * THREADS + tid < nvec) {
        float x[8];
        #pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = value(c, j);
        take(x, 8);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (at < V) take(&tail, 1);
    // over the workgroup: one meeting a row, in turns of LDS
    const float M = wave_max(m);
    s = wave_sum(s * __builtin_amdgcn_exp2f((m - M) * LOG2E));
    if (weights.mask) share = wave_sum(share);
    if (lane == 0) {
      part[turn][0][tid / WAVE] = M;
      part[turn][1][tid / WAVE] = s;
      part[turn][2][tid / WAVE] = share;
    }
    __syncthreads();
    // a wave's lanes take a wave each, in every wave
    const int of = lane & (NW - 1);
    float top = part[turn][0][of], sum = part[turn][1][of];
    float high = top;
    #pragma unroll
    for (int off = NW / 2; off > 0; off >>= 1) high = fmaxf(high, __shfl_xor(high, off, WAVE));
    sum *= __builtin_amdgcn_exp2f((top - high) * LOG2E);
    #pragma unroll
    for (int off = NW / 2; off > 0; off >>= 1) sum += __shfl_xor(sum, off, WAVE);
    top = high;
    const float l = top + __logf(sum);
    float wv;
    if (weights.mask) {
      float n = part[turn][2][of];
      #pragma unroll
      for (int off = NW / 2; off > 0; off >>= 1) n += __shfl_xor(n, off, WAVE);
      wv = mask(row) * (-weights.rewards[seq] / fmaxf(n, 1.f) / weights.B * weights.scale);
      if (tid == 0) weights.w[row] = wv;
    } else {
      wv = weights.w[row];
    }
    if (tid == 0) lse_out[row] = l;
    auto put = [&](float logp) {
      if (loss) mine += wv * logp;
      else token_logp[row] = logp;
    };
    if (tid == 0 && tgt < 0) put(0.f - l);
    if (at < V) {
      if (at == tgt) put(tail - l);
      float g = 0.f;
      if (wv != 0.f) g = wv * ((at == tgt ? 1.f : 0.f) - __expf(tail - l));
      dr[at] = f2bf(g);
    }
    const auto to = row_at(dr), from = row_at(lr + (int64_t)gridDim.x * V);
    auto write = [&](auto more_) {
      int off = tid * 16;
      #pragma unroll
      for (int c = 0; c < KEEP; ++c, next(off)) {
        {
          if (off == (tgt >> 3) * 16 && off < bytes) {
            float x = value(c, 0);
            #pragma unroll
            for (int j = 1; j < 8; ++j) x = (tgt & 7) == j ? value(c, j) : x;
            put(x - l);
          }
          u32x4 o;
          #pragma unroll
          for (int j = 0; j < 4; ++j) {
            float g[2];
            #pragma unroll
            for (int h = 0; h < 2; ++h) {
              const float p = __expf(value(c, 2 * j + h) - l);
              g[h] = wv == 0.f ? 0.f : wv * ((off / 2 + 2 * j + h == tgt ? 1.f : 0.f) - p);
            }
            o[j] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{g[0], g[1]}, bf16v2));
          }
          __builtin_amdgcn_raw_buffer_store_b128(o, to, off, 0, 2);     // 2: past the caches
        }
        if (decltype(more_)::value) v[c] = __builtin_amdgcn_raw_buffer_load_b128(from, off, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    if (row + gridDim.x < rows) write(std::true_type{});
    else write(std::false_type{});
  }
  if (!loss) return;
  auto over_block = [&](float x) {      // thread 0 has the sum
    x = wave_sum(x);
    if (lane == 0) ends[tid / WAVE] = x;
    __syncthreads();
    if (tid == 0)
      for (int i = 1; i < NW; ++i) x += ends[i];
    return x;
  };
  mine = over_block(mine);
  if (tid == 0) {
    store_through(token_logp + blockIdx.x, mine);
    stores_done();
    last = last_to_end(counts);
  }
  __syncthreads();
  if (!last) return;
  float sum = 0.f;
  for (int i = tid; i < (int)gridDim.x; i += THREADS) sum += load_through(token_logp + i);
  sum = over_block(sum);
  if (tid == 0) *loss = sum;
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

// Whether loss_both_kernel takes the rows: longer ones don't fit its registers. Below 2 MB
// of logits two passes, which hold no gradient from forward to backward: their kernels
// take 11.4 us at 40 rows of 4096 and this one's 10.5, their launches' host 36 to 58 either
// way. From there on 13.0 and 11.2 (600 x 4096), 22.3 and 16.4 (3000 x 4096), 35.1 and 30.3
// (64 x 151936).
static bool takes_both(const torch::Tensor& logits) {
  const int64_t V = logits.size(-1);
  return logits.scalar_type() == at::kBFloat16 && logits.numel() >= 1 << 20 && V >= 8 &&
         V / 8 <= 19 * 1024 && logits.numel() / V < (1 << 30);
}

// f(threads, pieces) as constants, FIRST <= pieces <= LAST
template <int FIRST, int LAST, typename T, typename F>
static void by_pieces(int pieces, T threads, F&& f) {
  if constexpr (FIRST < LAST) {
    if (pieces > FIRST) return by_pieces<FIRST + 1, LAST>(pieces, threads, f);
  }
  f(threads, std::integral_constant<int, FIRST>{});
}

// Threads of a workgroup of loss_both_kernel for rows of nvec pieces of 8 values, and
// workgroups a CU by their registers.
static int threads_of(int nvec) { return nvec <= 8 * 256 ? 256 : nvec <= 8 * 512 ? 512 : 1024; }
static constexpr int per_cu(int threads, int pieces) {
  return std::max(1, (8 - (pieces > 5) - (pieces > 7)) * 256 / threads);
}

// lse; grad <- the gradient for a dloss of 1, token_logp <- its values, or, with counts, the
// workgroups' parts of loss <- the sum of w * token_logp
static torch::Tensor logprob_both(const torch::Tensor& logits, const torch::Tensor& targets,
                                  const RowWeights& weights, const torch::Tensor& grad,
                                  float* token_logp, float* loss, uint32_t* counts) {
  TORCH_CHECK(logits.is_cuda() && logits.is_contiguous() && takes_both(logits));
  TORCH_CHECK(targets.scalar_type() == at::kLong && targets.is_contiguous());
  const int V = logits.size(-1), nvec = V / 8;
  const int rows = (int)(logits.numel() / V);
  auto sizes = logits.sizes().vec();
  sizes.pop_back();
  auto lse = torch::empty(sizes, logits.options().dtype(at::kFloat));
  auto go = [&](auto threads_, auto keep_) {
    constexpr int THREADS = decltype(threads_)::value, KEEP = decltype(keep_)::value;
    hipLaunchKernelGGL((loss_both_kernel<THREADS, KEEP>),
                       dim3(std::min(rows, 256 * per_cu(THREADS, KEEP))),
                       dim3(THREADS), 0, at::cuda::getCurrentCUDAStream(),
                       reinterpret_cast<const __hip_bfloat16*>(logits.data_ptr()),
                       targets.data_ptr<int64_t>(), weights, token_logp,
                       lse.data_ptr<float>(), reinterpret_cast<__hip_bfloat16*>(grad.data_ptr()),
                       loss, counts, rows, V);
  };
  // As many pieces as the row has: a thread's work on pieces past its end is not free, nor
  // a look whether there are any. With 2, 8 pieces of 256 threads and 4, 8, 16, 19 of 1024,
  // with a branch a piece, so, and in two passes, us: 8000 x 8192 68, 55, 53, 69; 8000 x
  // 17000 153, 144, 105, 139; 2400 x 33000 89, 80, 70, 83; 2400 x 66000 185, 170, 146, 163;
  // 300 x 70000 43, 37, 33, 36; 2400 x 152064 320, 356, 317, 389.
  const int threads = threads_of(nvec), pieces = CDIV(nvec, threads);
  if (threads == 256) by_pieces<1, 8>(pieces, std::integral_constant<int, 256>{}, go);
  else if (threads == 512) by_pieces<5, 8>(pieces, std::integral_constant<int, 512>{}, go);
  else by_pieces<5, 19>(pieces, std::integral_constant<int, 1024>{}, go);
  HIP_CHECK_LAST();
  return lse;
}

// loss <- the sum of w * token_logp
static void sum_rows(const torch::Tensor& token_logp, const torch::Tensor& w,
                     const torch::Tensor& loss) {
  hipLaunchKernelGGL(loss_rows_kernel, dim3(1), dim3(1024), 0, at::cuda::getCurrentCUDAStream(),
                     token_logp.data_ptr<float>(), w.data_ptr<float>(), loss.data_ptr<float>(),
                     w.numel());
  HIP_CHECK_LAST();
}

// Whether a masked loss' row weights are made by a launch ahead, with the sum over rows
// then in loss_both_kernel, and not by each row from its sequence's whole mask. That launch
// and the workgroups' meeting cost 5 us more than the sum's own launch, a mask in the rows
// some 0.7 and 0.5 for each of a thread's loads of it, on every turn of a workgroup. Masks
// in the rows, ahead, two passes, us: 8 x 200 x 4096 17.0, 22.5, 18.1; 8 x 600 x 4096 31.7,
// 31.1, 33.8; 4 x 1500 x 4096 40, 33.5, 44; 1 x 16384 x 4096 249, 65, 174; 2000 x 100 x 64
// 507, 315, 513; 2 x 1200 x 32003 65, 64, 95; 8 x 100 x 152064 110, 111, 117; 8 x 301 x
// 152064 325, 323, 360; 1 x 2400 x 152064 339, 322, 371.
static bool weights_ahead(int rows, int T, int nvec) {
  const int threads = threads_of(nvec), grid = 256 * per_cu(threads, CDIV(nvec, threads));
  return std::max(1., (double)rows / grid) * (0.7 + 0.5 * T / threads) > 5.;
}

// The masked PG/GRPO loss of logits (B, T, V): {loss, row weights (B, T), lse}, and
// grad, if any, <- the gradient for a dloss of 1. mask int64 or fp32, rewards fp32.
static std::vector<torch::Tensor> logprob_loss_fwd(torch::Tensor logits, torch::Tensor targets,
                                                   torch::Tensor mask, torch::Tensor rewards,
                                                   double scale,
                                                   const c10::optional<torch::Tensor>& grad) {
  TORCH_CHECK(logits.dim() == 3 && mask.is_cuda() && rewards.is_cuda());
  const int B = logits.size(0), T = logits.size(1);
  TORCH_CHECK(mask.numel() == (int64_t)B * T && targets.numel() == (int64_t)B * T &&
              rewards.numel() == B, "logprob_loss: shape mismatch");
  TORCH_CHECK(mask.is_contiguous() && rewards.is_contiguous() &&
              rewards.scalar_type() == at::kFloat);
  const bool mask64 = mask.scalar_type() == at::kLong;
  TORCH_CHECK(mask64 || mask.scalar_type() == at::kFloat);
  auto stream = at::cuda::getCurrentCUDAStream();
  auto w = torch::empty({B, T}, logits.options().dtype(at::kFloat));
  auto loss = torch::empty({}, w.options());
  if (grad && weights_ahead(B * T, T, (int)(logits.size(2) / 8))) {
    // the workgroups' parts and their counts
    auto parts = torch::empty({(int64_t)B * T + COUNTS}, w.options());
    auto* counts = reinterpret_cast<uint32_t*>(parts.data_ptr<float>() + (int64_t)B * T);
    #define WEIGHTS(M)                                                                \
      hipLaunchKernelGGL(loss_weights_kernel<M>, dim3(B), dim3(1024), 0, stream,      \
                         mask.data_ptr<M>(), rewards.data_ptr<float>(),               \
                         w.data_ptr<float>(), counts, B, T, (float)scale)
    if (mask64) WEIGHTS(int64_t);
    else WEIGHTS(float);
    #undef WEIGHTS
    auto lse = logprob_both(logits, targets, {w.data_ptr<float>()}, *grad, parts.data_ptr<float>(),
                            loss.data_ptr<float>(), counts);
    return {loss, w, lse};
  }
  if (grad) {
    auto token_logp = torch::empty({B, T}, w.options());
    auto lse = logprob_both(logits, targets,
                            {w.data_ptr<float>(), mask.data_ptr(), mask64, rewards.data_ptr<float>(),
                             B, T, (float)scale},
                            *grad, token_logp.data_ptr<float>(), nullptr, nullptr);
    sum_rows(token_logp, w, loss);
    return {loss, w, lse};
  }
  auto lp = logprob_lse_fwd(logits, targets);
  #define REDUCE(M)                                                                   \
    hipLaunchKernelGGL(loss_reduce_kernel<M>, dim3(1), dim3(1024), 0, stream,         \
                       lp[0].data_ptr<float>(), mask.data_ptr<M>(),                   \
                       rewards.data_ptr<float>(), w.data_ptr<float>(),                \
                       loss.data_ptr<float>(), B, T, (float)scale)
  if (mask64) REDUCE(int64_t);
  else REDUCE(float);
  #undef REDUCE
  HIP_CHECK_LAST();
  return {loss, w, lp[1]};
}

// made: the gradient for a dloss of 1, which is kept where dloss is that
static torch::Tensor loss_bwd(torch::Tensor logits, torch::Tensor targets, torch::Tensor w,
                              torch::Tensor lse, c10::optional<torch::Tensor> dloss,
                              c10::optional<torch::Tensor> made) {
  TORCH_CHECK(logits.is_cuda() && logits.is_contiguous());
  const float* dl = nullptr;
  if (dloss) {
    TORCH_CHECK(dloss->is_cuda() && dloss->numel() == 1 && dloss->scalar_type() == at::kFloat);
    dl = dloss->data_ptr<float>();
  }
  const int V = logits.size(-1);
  const int64_t rows = logits.numel() / V;
  TORCH_CHECK(!made || (dl && made->is_contiguous() && made->sizes() == logits.sizes() &&
                        made->scalar_type() == logits.scalar_type()));
  auto dlogits = made ? *made : torch::empty_like(logits);
  if (rows == 0) return dlogits;
  auto stream = at::cuda::getCurrentCUDAStream();
  auto wc = w.contiguous();
  auto lsec = lse.contiguous();
  auto tc = targets.contiguous();
  const bool bf16 = logits.scalar_type() == at::kBFloat16;
  const bool many = bf16 && V / 8 >= 4 * 1024;
  #define BWD(KERNEL, T, THREADS, BLOCKS, ...)                                         \
    hipLaunchKernelGGL((KERNEL<T, THREADS>), dim3(BLOCKS), dim3(THREADS), 0, stream,   \
                       reinterpret_cast<const T*>(logits.data_ptr()),                  \
                       tc.data_ptr<int64_t>(), wc.data_ptr<float>(),                   \
                       lsec.data_ptr<float>(), dl,                                     \
                       reinterpret_cast<T*>(dlogits.data_ptr()), V, ##__VA_ARGS__)
  if (made) {
    const int64_t blocks = std::min<int64_t>(rows, 512);
    if (many) BWD(loss_anew_kernel, __hip_bfloat16, 1024, blocks, rows);
    else BWD(loss_anew_kernel, __hip_bfloat16, 256, blocks, rows);
  } else if (many) {
    BWD(loss_bwd_kernel, __hip_bfloat16, 1024, rows);
  } else if (bf16) {
    BWD(loss_bwd_kernel, __hip_bfloat16, 256, rows);
  } else {
    BWD(loss_bwd_kernel, float, 256, rows);
  }
  #undef BWD
  HIP_CHECK_LAST();
  return dlogits;
}

torch::Tensor logprob_loss_bwd(torch::Tensor logits, torch::Tensor targets, torch::Tensor w,
                               torch::Tensor lse, c10::optional<torch::Tensor> dloss) {
  return loss_bwd(logits, targets, w, lse, dloss, c10::nullopt);
}

// The differentiable loss: a node of the C++ engine. Where a gradient is wanted of rows
// that loss_both_kernel takes, forward makes it for a dloss of 1, which backward hands
// out; any other dloss makes it anew from the logits, and so does every further backward
// of a graph that is kept, as what was handed out is the caller's. So a loss that is
// scaled or only looked at costs more than in two passes, and one whose backward is still
// to come holds a gradient beside its logits: the price of the one pass, which callers
// that scale by weights and run backward at once, as the learner, do not pay.
namespace {

// Not under hooks on saved tensors (checkpoints, offloading): they would drop or move the
// logits, and the gradient, which they don't see, would stay.
bool wants_both(const torch::Tensor& logits) {
  return at::GradMode::is_enabled() && logits.requires_grad() && logits.is_cuda() &&
         takes_both(logits) && !at::SavedTensorDefaultHooks::get_hooks();
}

// Where the gradient goes; two passes where memory has no room for it yet.
c10::optional<torch::Tensor> gradient_room(const torch::Tensor& logits, bool both) {
  if (!both) return c10::nullopt;
  try {
    return torch::empty_like(logits);
  } catch (const c10::OutOfMemoryError&) {
    return c10::nullopt;
  }
}

torch::Tensor handed_out(torch::autograd::AutogradContext* ctx, const torch::Tensor& dloss) {
  const auto s = ctx->get_saved_variables();
  c10::optional<torch::Tensor> made;
  if (const auto it = ctx->saved_data.find("grad"); it != ctx->saved_data.end()) {
    made = it->second.toTensor();
    ctx->saved_data.erase(it);
  }
  return loss_bwd(s[0], s[1], s[2], s[3], dloss.to(at::kFloat), made);
}

struct LogprobLoss : public torch::autograd::Function<LogprobLoss> {
  static torch::Tensor forward(torch::autograd::AutogradContext* ctx, torch::Tensor logits,
                               torch::Tensor targets, torch::Tensor mask, torch::Tensor rewards,
                               double scale, bool both) {
    logits = logits.contiguous();
    targets = targets.contiguous();
    // int64 masks are read as they are
    auto m = mask.scalar_type() == at::kLong ? mask : mask.to(at::kFloat);
    const auto grad = gradient_room(logits, both);
    auto r = logprob_loss_fwd(logits, targets, m.contiguous(),
                              rewards.to(at::kFloat).contiguous(), scale, grad);
    ctx->save_for_backward({logits, targets, r[1], r[2]});
    if (grad) ctx->saved_data["grad"] = *grad;
    return r[0];
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    return {handed_out(ctx, grads[0]), torch::Tensor(), torch::Tensor(), torch::Tensor(),
            torch::Tensor(), torch::Tensor()};
  }
};

}  // namespace

torch::Tensor logprob_loss(torch::Tensor logits, torch::Tensor targets, torch::Tensor mask,
                           torch::Tensor rewards, double scale) {
  return LogprobLoss::apply(logits, targets, mask, rewards, scale, wants_both(logits));
}

// The same sum for rows that carry weights of their own: sum_i w_i log p(target_i)
// of logits (rows, V); no gradient for the weights.
namespace {

struct LogprobRows : public torch::autograd::Function<LogprobRows> {
  static torch::Tensor forward(torch::autograd::AutogradContext* ctx, torch::Tensor logits,
                               torch::Tensor targets, torch::Tensor w, bool both) {
    TORCH_CHECK(logits.dim() == 2 && targets.is_cuda() && w.is_cuda() &&
                targets.numel() == logits.size(0) && w.numel() == logits.size(0) &&
                w.scalar_type() == at::kFloat, "logprob_rows: shape mismatch");
    logits = logits.contiguous();
    targets = targets.contiguous();
    w = w.contiguous();
    const auto grad = gradient_room(logits, both);
    torch::Tensor token_logp, lse;
    if (grad) {
      token_logp = torch::empty({logits.size(0)}, w.options());
      lse = logprob_both(logits, targets, {w.data_ptr<float>()}, *grad, token_logp.data_ptr<float>(),
                         nullptr, nullptr);
    } else {
      auto lp = logprob_lse_fwd(logits, targets);
      token_logp = lp[0];
      lse = lp[1];
    }
    auto loss = torch::empty({}, lse.options());
    sum_rows(token_logp, w, loss);
    ctx->save_for_backward({logits, targets, w, lse});
    if (grad) ctx->saved_data["grad"] = *grad;
    return loss;
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    return {handed_out(ctx, grads[0]), torch::Tensor(), torch::Tensor(), torch::Tensor()};
  }
};

}  // namespace

torch::Tensor logprob_rows(torch::Tensor logits, torch::Tensor targets, torch::Tensor w) {
  return LogprobRows::apply(logits, targets, w, wants_both(logits));
}
