// Fused sampler: temperature, histogram top-k/top-p threshold and Gumbel-max
// draw, without sorting the vocabulary (reference counterpart: vLLM's sampler
// inside fast_generate).
//
// Semantics. z = (logit - row max) / temperature. 1024 bins of 1/32 cover
// z in (-32, 0]; the threshold keeps whole bins down to the one in which the
// cumulative probability reaches top_p (or the count top_k). The draw is the
// argmax of z - log(-log u) over the kept set, u a counter-based hash of
// (seed of the row, step, element): the step is read from device memory, so a
// replayed graph draws anew. Slices add their probabilities up as integers of
// 2^-32, whose sum does not hang on their order: a call repeats itself exactly.
// How a row was split over workgroups (by the number of rows) shows only where
// a cumulative probability lies within fp32 rounding of top_p.
//
// A row is cut into slices, so that any number of rows fills the chip: a
// maximum pass; with a threshold two histogram passes, first over 32 groups of
// 32 bins and then over the bins of the group in which the threshold falls;
// and the draw, whose last slice of a row writes the token. A thread adds into
// histogram columns of its own, so nothing collides and no atomics are needed:
// LDS float atomics into 1024 shared bins took ~3 clocks a lane (124 us for
// 160 rows of 152064), the two passes take 44 us.
// An element that is kept costs ~330 cycles of hashing a wave, so sparse ones
// are gathered into full waves first. 160 rows of 152064 at top_p 0.95: 284 us
// as eight launches with one serial thread a row for the threshold, 95 us now
// (draw 46, histograms 44, maximum 9), bound by the draw's integer products;
// one row of 151936 without a threshold 24.6 -> 11.3 us, bound by two launches.
#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>
#include "common.h"

typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

namespace {

constexpr int NBINS = 1024;
constexpr float ZRANGE = 32.f;        // z below -32 has no probability left
// u is at most 1 - 2^-24 and at least 2^-24: a draw adds between -2.82 and
// 16.64 to z. The row maximum (z = 0) reaches -2.82, nothing below -19.46 does.
constexpr float ZDRAW = -19.5f;

DEV_INLINE float bf_lo(uint32_t w) { return __uint_as_float(w << 16); }
DEV_INLINE float bf_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

DEV_INLINE uint64_t row_seed(const int64_t* seeds, const int64_t* step, int row) {
  return (uint64_t)seeds[row] ^ splitmix64(0x5D21u + (uint64_t)*step);
}

DEV_INLINE int bin_of(float z) { return min(NBINS - 1, (int)(-z * (NBINS / ZRANGE))); }

// The best key of a lane; equal keys go to the lower index.
struct Best {
  float key = -1e30f;
  int idx = 0x7fffffff;
  DEV_INLINE void offer(float k, int i) {
    if (k > key || (k == key && i < idx)) { key = k; idx = i; }
  }
  DEV_INLINE void over_wave() {
    #pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const float k = __shfl_xor(key, off, WAVE);
      const int i = __shfl_xor(idx, off, WAVE);
      offer(k, i);
    }
  }
};

// splitmix64(idx) for idx < 2^31: the first sum's upper half is a constant,
// which leaves two of the first product's three partial products.
DEV_INLINE uint64_t mix_index(uint32_t idx) {
  constexpr uint64_t C1 = 0xBF58476D1CE4E5B9ull;
  constexpr uint32_t H = 0x9E3779B9u;
  const uint32_t x0 = idx + 0x7F4A7C15u;
  const uint32_t lo = x0 ^ ((H << 2) | (x0 >> 30));
  uint64_t x = (uint64_t)lo * (uint32_t)C1;
  x += (uint64_t)(lo * (uint32_t)(C1 >> 32) + (H ^ (H >> 30)) * (uint32_t)C1) << 32;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}

// z - log(-log u), u = (the hash's upper 24 bits + 1) / 2^24, kept below 1: u = 1
// would make the key infinite and draw the element whatever its probability.
// Neither logarithm's argument is ever denormal.
DEV_INLINE float gumbel_key(uint64_t seed, int idx, float z) {
  constexpr float LN2 = 0.6931471805599453f;
  const uint64_t h = splitmix64(seed ^ mix_index((uint32_t)idx));
  const float u = (float)min((uint32_t)(h >> 40) + 1u, (1u << 24) - 1u) * 0x1p-24f;
  return z - LN2 * __builtin_amdgcn_logf(-LN2 * __builtin_amdgcn_logf(u));
}

// Gathers the elements that a wave keeps and draws 64 at a time.
struct DrawQueue {
  uint2* q;             // 128 entries of this wave: index, z
  uint64_t seed;
  int head = 0, count = 0;
  Best best;

  DEV_INLINE void draw(int n) {
    __builtin_amdgcn_wave_barrier();
    const int lane = threadIdx.x & (WAVE - 1);
    if (lane < n) {
      const uint2 e = q[(head + lane) & 127];
      best.offer(gumbel_key(seed, (int)e.x, __uint_as_float(e.y)), (int)e.x);
    }
    head += n;
    count -= n;
    __builtin_amdgcn_wave_barrier();
  }
  // Every lane of the wave calls it. Gathering costs a fifth of a draw: a wave
  // that is mostly kept draws at once.
  DEV_INLINE void push(bool keep, int idx, float z) {
    const uint64_t mask = __ballot(keep);
    if (mask == 0) return;
    if (__popcll(mask) >= 48) {
      if (keep) best.offer(gumbel_key(seed, idx, z), idx);
      return;
    }
    if (keep) {
      const int at = __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                               __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0));
      q[(head + count + at) & 127] = uint2{(uint32_t)idx, __float_as_uint(z)};
    }
    count += __popcll(mask);
    if (count >= WAVE) draw(WAVE);
  }
};

constexpr int GROUPS = 32, IN_GROUP = NBINS / GROUPS;

// Where a running sum over 32 bins (lanes 0..31 of every wave) reaches the
// limit: {bin, sum before it}; the last bin if it never does.
template <typename T>
struct Crossing { int bin; T before; };

template <typename T>
DEV_INLINE Crossing<T> crossing(T x, T start, T limit) {
  const int lane = threadIdx.x & (WAVE - 1);
  T cum = x;
  #pragma unroll
  for (int off = 1; off < 32; off <<= 1) {
    const T y = __shfl_up(cum, off, WAVE);
    if ((lane & 31) >= off) cum += y;
  }
  const uint64_t mask = __ballot(start + cum >= limit) & 0xffffffffull;
  const int bin = mask ? __ffsll((unsigned long long)mask) - 1 : 31;
  const T before = __shfl(cum, max(bin - 1, 0), WAVE);
  return {bin, start + (bin ? before : T(0))};
}

DEV_INLINE float wave_total(float x) {   // lanes 0..31, in their order
  #pragma unroll
  for (int off = 1; off < 32; off <<= 1) {
    const float y = __shfl_up(x, off, WAVE);
    if ((threadIdx.x & 31) >= off) x += y;
  }
  return __shfl(x, 31, WAVE);
}

// Sums of a row's groups and of the bins of the crossing groups, in global
// memory: probability in units of 2^-32 (a row's is below V < 2^31) and count.
struct Hist {
  unsigned long long *group_p, *bin_p;     // (B, 32) each
  int *group_c, *bin_c;
};

DEV_INLINE float prob(unsigned long long x) { return (float)x * 0x1p-32f; }

// The row's crossing groups, from the group sums: every wave computes them.
template <bool BY_P, bool BY_K>
DEV_INLINE void crossing_groups(const Hist& h, int row, float top_p, int top_k,
                                Crossing<float>& cp, Crossing<int>& ck, float& target) {
  const int at = row * GROUPS + (threadIdx.x & 31);
  if (BY_P) {
    const float x = prob(h.group_p[at]);
    target = top_p * wave_total(x);
    cp = crossing(x, 0.f, target);
  }
  if (BY_K) ck = crossing(h.group_c[at], 0, top_k);
}

// ----------------------------------------------------------------- slices
// Eight elements a thread of the block's next 2048: 16-byte loads where rows
// are aligned for them, else one element a lane. -inf past the end.
template <typename T, bool VEC>
DEV_INLINE void load8(const T* lr, int base, int i1, float (&x)[8], int (&id)[8]) {
  constexpr bool BF16 = std::is_same<T, __hip_bfloat16>::value;
  #pragma unroll
  for (int k = 0; k < 8; ++k) id[k] = VEC ? base + threadIdx.x * 8 + k : base + k * 256 + threadIdx.x;
  if constexpr (VEC) {
    const int at = min(id[0], i1 - 8);
    if constexpr (BF16) {
      const u32x4 d = *reinterpret_cast<const u32x4*>(lr + at);
      #pragma unroll
      for (int w = 0; w < 4; ++w) { x[2 * w] = bf_lo(d[w]); x[2 * w + 1] = bf_hi(d[w]); }
    } else {
      #pragma unroll
      for (int k = 0; k < 2; ++k) {
        const u32x4 d = *reinterpret_cast<const u32x4*>(lr + at + 4 * k);
        #pragma unroll
        for (int w = 0; w < 4; ++w) x[4 * k + w] = __uint_as_float(d[w]);
      }
    }
  } else {
    #pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int at = min(id[k], i1 - 1);
      if constexpr (BF16) x[k] = bf2f(lr[at]); else x[k] = lr[at];
    }
  }
  #pragma unroll
  for (int k = 0; k < 8; ++k)
    if (id[k] >= i1) x[k] = __uint_as_float(0xff800000u);
}

DEV_INLINE float row_max(const float* ms, int row, int S) {   // S <= 64
  return wave_max(ms[row * S + min((int)(threadIdx.x & (WAVE - 1)), S - 1)]);
}

// Slice maxima; a row's first slice also clears what the later passes add to.
template <typename T, bool VEC>
__global__ __launch_bounds__(256)
void slice_max_kernel(const T* __restrict__ logits, int V, int per, float* __restrict__ ms,
                      unsigned long long* __restrict__ top, int* __restrict__ done, Hist h) {
  __shared__ float red[16];
  const int row = blockIdx.x, sl = blockIdx.y;
  const T* lr = logits + (int64_t)row * V;
  const int i1 = min(V, (sl + 1) * per);
  float m = -1e30f, x[8];
  int id[8];
  for (int base = sl * per; base < i1; base += 2048) {
    load8<T, VEC>(lr, base, i1, x, id);
    #pragma unroll
    for (int k = 0; k < 8; ++k) m = fmaxf(m, x[k]);
  }
  m = block_max(m, red);
  if (threadIdx.x == 0) ms[row * gridDim.y + sl] = m;
  if (sl == 0) {
    if (threadIdx.x == 0) { top[row] = 0ull; done[row] = 0; }
    if (h.group_p && threadIdx.x < 32) {
      const int at = row * 32 + threadIdx.x;
      h.group_p[at] = h.bin_p[at] = 0ull;
      h.group_c[at] = h.bin_c[at] = 0;
    }
  }
}

// FINE false: sums of the 32 groups of bins. FINE true: sums of the bins of the
// group where the probability (count) crosses its limit.
template <typename T, bool VEC, bool BY_P, bool BY_K, bool FINE>
__global__ __launch_bounds__(256)
void slice_hist_kernel(const T* __restrict__ logits, int V, int per, float inv_temp, float top_p,
                       int top_k, const float* __restrict__ ms, Hist h) {
  __shared__ float hp[BY_P ? 32 * 256 : 1];     // [bin][thread]
  __shared__ int hc[BY_K ? 32 * 256 : 1];
  const int row = blockIdx.x, sl = blockIdx.y, tid = threadIdx.x;
  const T* lr = logits + (int64_t)row * V;
  const int i1 = min(V, (sl + 1) * per);
  const float m = row_max(ms, row, gridDim.y);
  int gp = 0, gc = 0;
  if (FINE) {
    Crossing<float> cp;
    Crossing<int> ck;
    float target;
    crossing_groups<BY_P, BY_K>(h, row, top_p, top_k, cp, ck, target);
    if (BY_P) gp = cp.bin;
    if (BY_K) gc = ck.bin;
  }
  for (int i = 0; i < 32; ++i) {
    if (BY_P) hp[i * 256 + tid] = 0.f;
    if (BY_K) hc[i * 256 + tid] = 0;
  }
  float x[8], next[8];
  int id[8], next_id[8];
  if (sl * per < i1) load8<T, VEC>(lr, sl * per, i1, next, next_id);
  for (int base = sl * per; base < i1; base += 2048) {
    #pragma unroll
    for (int k = 0; k < 8; ++k) { x[k] = next[k]; id[k] = next_id[k]; }
    load8<T, VEC>(lr, base + 2048, i1, next, next_id);   // past the end: the last eight again
    #pragma unroll
    for (int k = 0; k < 8; ++k) {
      // without branches: what does not count adds zero
      const float z = (x[k] - m) * inv_temp;
      const int b = bin_of(z), g = b / IN_GROUP, at = (FINE ? b % IN_GROUP : g) * 256 + tid;
      const bool in = z > -ZRANGE;
      if (BY_P) hp[at] += in && (!FINE || g == gp) ? __expf(z) : 0.f;
      if (BY_K) hc[at] += in && (!FINE || g == gc) ? 1 : 0;
    }
  }
  __syncthreads();
  const int wid = tid / WAVE, lane = tid & (WAVE - 1);
  for (int b = wid * 8; b < wid * 8 + 8; ++b) {
    if (BY_P) {
      float v = 0.f;
      #pragma unroll
      for (int i = 0; i < 4; ++i) v += hp[b * 256 + i * WAVE + lane];
      v = wave_sum(v);
      if (lane == 0 && v != 0.f)
        atomicAdd(&(FINE ? h.bin_p : h.group_p)[row * 32 + b],
                  (unsigned long long)(v * 0x1p32f + 0.5f));
    }
    if (BY_K) {
      int v = 0;
      #pragma unroll
      for (int i = 0; i < 4; ++i) v += hc[b * 256 + i * WAVE + lane];
      #pragma unroll
      for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, WAVE);
      if (lane == 0 && v != 0) atomicAdd(&(FINE ? h.bin_c : h.group_c)[row * 32 + b], v);
    }
  }
}

template <typename T, bool VEC, bool BY_P, bool BY_K>
__global__ __launch_bounds__(256)
void slice_draw_kernel(const T* __restrict__ logits, int V, int per, float inv_temp, float top_p,
                       int top_k, const float* __restrict__ ms, Hist h,
                       const int64_t* __restrict__ seeds, const int64_t* __restrict__ step, unsigned long long* __restrict__ top,
                       int* __restrict__ done, int64_t* __restrict__ out) {
  __shared__ uint2 queue[4 * 128];
  __shared__ float fpart[4];
  __shared__ int ipart[4];
  const int row = blockIdx.x, sl = blockIdx.y, S = gridDim.y, tid = threadIdx.x;
  const T* lr = logits + (int64_t)row * V;
  const int i1 = min(V, (sl + 1) * per);
  const float m = row_max(ms, row, S);
  float zlow = ZDRAW;
  if (BY_P || BY_K) {
    Crossing<float> cp;
    Crossing<int> ck;
    float target;
    crossing_groups<BY_P, BY_K>(h, row, top_p, top_k, cp, ck, target);
    const int at = row * 32 + (tid & 31);
    int thr = NBINS - 1;
    if (BY_P) thr = min(thr, cp.bin * IN_GROUP + crossing(prob(h.bin_p[at]), cp.before, target).bin);
    if (BY_K) thr = min(thr, ck.bin * IN_GROUP + crossing(h.bin_c[at], ck.before, top_k).bin);
    // the bins up to thr are z > -(thr + 1) / 32; the edge itself lies in the next
    zlow = fmaxf(-(thr + 1) * (ZRANGE / NBINS), ZDRAW);
  }
  DrawQueue dq{queue + (tid / WAVE) * 128, row_seed(seeds, step, row)};
  float x[8], next[8];
  int id[8], next_id[8];
  if (sl * per < i1) load8<T, VEC>(lr, sl * per, i1, next, next_id);
  for (int base = sl * per; base < i1; base += 2048) {
    #pragma unroll
    for (int k = 0; k < 8; ++k) { x[k] = next[k]; id[k] = next_id[k]; }
    load8<T, VEC>(lr, base + 2048, i1, next, next_id);   // past the end: the last eight again
    #pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float z = (x[k] - m) * inv_temp;
      dq.push(z > zlow, id[k], z);
    }
  }
  dq.draw(dq.count);
  dq.best.over_wave();
  __syncthreads();
  if ((tid & (WAVE - 1)) == 0) {
    fpart[tid / WAVE] = dq.best.key;
    ipart[tid / WAVE] = dq.best.idx;
  }
  __syncthreads();
  if (tid != 0) return;
  Best b;
  for (int w = 0; w < 4; ++w) b.offer(fpart[w], ipart[w]);
  // key and index in one word whose order is that of Best; 0: nothing kept
  uint32_t o = __float_as_uint(b.key);
  o = (o >> 31) ? ~o : o | 0x80000000u;
  unsigned long long mine = b.idx == 0x7fffffff ? 0ull
      : ((unsigned long long)o << 32) | (0xffffffffu - (uint32_t)b.idx);
  if (S > 1) {
    atomicMax(&top[row], mine);
    __threadfence();
    if (atomicAdd(&done[row], 1) != S - 1) return;
    __threadfence();
    mine = atomicMax(&top[row], 0ull);      // all slices have arrived
  }
  out[row] = mine == 0ull ? 0 : (int64_t)(0xffffffffu - (uint32_t)mine);
}

template <typename T, bool VEC>
void sample_slices(const T* logits, int B, int V, float inv_t, float top_p, int top_k,
                   const torch::Tensor& seeds, const torch::Tensor& step, torch::Tensor& out) {
  const bool by_p = top_p < 1.f, by_k = top_k > 0, filtering = by_p || by_k;
  // enough slices for four workgroups a CU, none under one load of a block
  int S = 1;
  while (S < 64 && (int64_t)B * S < 1024 && V / (2 * S) >= 2048) S *= 2;
  const int per = (CDIV(V, S) + 7) / 8 * 8;
  auto ws = torch::empty({B * (int64_t)(12 + 4 * S + (filtering ? (8 + 4) * 2 * 32 : 0))},
                         out.options().dtype(at::kByte));
  char* w = reinterpret_cast<char*>(ws.data_ptr());
  auto* top = reinterpret_cast<unsigned long long*>(w);
  w += 8ll * B;
  Hist h{};
  if (filtering) {
    h.group_p = reinterpret_cast<unsigned long long*>(w);
    h.bin_p = h.group_p + 32ll * B;
    h.group_c = reinterpret_cast<int*>(h.bin_p + 32ll * B);
    h.bin_c = h.group_c + 32ll * B;
    w = reinterpret_cast<char*>(h.bin_c + 32ll * B);
  }
  int* done = reinterpret_cast<int*>(w);
  float* ms = reinterpret_cast<float*>(w + 4ll * B);
  auto stream = at::cuda::getCurrentCUDAStream();
  const dim3 grid(B, S), block(256);
  hipLaunchKernelGGL((slice_max_kernel<T, VEC>), grid, block, 0, stream, logits, V, per, ms, top,
                     done, h);
  auto hist = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, block, 0, stream, logits, V, per, inv_t, top_p, top_k, ms, h);
  };
  auto draw = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, block, 0, stream, logits, V, per, inv_t, top_p, top_k, ms, h,
                       seeds.data_ptr<int64_t>(), step.data_ptr<int64_t>(), top, done,
                       out.data_ptr<int64_t>());
  };
  #define BY(P, K)                                        \
    do {                                                  \
      if (P || K) {                                       \
        hist(slice_hist_kernel<T, VEC, P, K, false>);     \
        hist(slice_hist_kernel<T, VEC, P, K, true>);      \
      }                                                   \
      draw(slice_draw_kernel<T, VEC, P, K>);              \
    } while (0)
  if (by_p && by_k) BY(true, true);
  else if (by_p) BY(true, false);
  else if (by_k) BY(false, true);
  else BY(false, false);
  #undef BY
}

}  // namespace

torch::Tensor sample_tokens(torch::Tensor logits, double temperature, double top_p, int64_t top_k,
                            torch::Tensor seeds, torch::Tensor step) {
  TORCH_CHECK(logits.is_cuda() && logits.is_contiguous() && logits.dim() == 2);
  TORCH_CHECK(temperature > 0.0, "temperature 0 is greedy: use argmax");
  TORCH_CHECK(seeds.scalar_type() == at::kLong);
  TORCH_CHECK(step.scalar_type() == at::kLong && step.is_cuda());
  const int B = logits.size(0), V = logits.size(1);
  const bool bf16 = logits.scalar_type() == at::kBFloat16;
  TORCH_CHECK(bf16 || logits.scalar_type() == at::kFloat);
  auto out = torch::empty({B}, logits.options().dtype(at::kLong));
  if (B == 0) return out;
  const float inv_t = 1.f / (float)temperature;
  const float p = top_p < 1.0 ? (float)top_p : 1.f;
  const int k = top_k > 0 && top_k < V ? (int)top_k : 0;
  const bool vec = V % 8 == 0 && reinterpret_cast<uintptr_t>(logits.data_ptr()) % 16 == 0;
  if (bf16) {
    auto* x = reinterpret_cast<const __hip_bfloat16*>(logits.data_ptr());
    if (vec) sample_slices<__hip_bfloat16, true>(x, B, V, inv_t, p, k, seeds, step, out);
    else sample_slices<__hip_bfloat16, false>(x, B, V, inv_t, p, k, seeds, step, out);
  } else {
    auto* x = logits.data_ptr<float>();
    if (vec) sample_slices<float, true>(x, B, V, inv_t, p, k, seeds, step, out);
    else sample_slices<float, false>(x, B, V, inv_t, p, k, seeds, step, out);
  }
  HIP_CHECK_LAST();
  return out;
}
