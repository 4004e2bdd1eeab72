// Fused sampler: temperature, histogram top-k/top-p threshold and Gumbel-max
// draw, without sorting the vocabulary (reference counterpart: vLLM's sampler
// inside fast_generate).
//
// Semantics. z = (logit - row max) / temperature. 1024 bins of 1/32 cover
// z in (-32, 0]; the threshold keeps whole bins down to the one in which the
// cumulative probability reaches top_p (or the count top_k). The draw is the
// argmax of z - log(-log u) over the kept set, u a counter-based hash of
// (seed of the row, step, element): the step is read from device memory, so a
// replayed graph draws anew. What workgroups add up meets as whole numbers of a small
// unit, whose sum does not hang on their order: a call repeats itself exactly. How a
// row was split over workgroups (by the number of rows) shows only where a
// cumulative probability lies within fp32 rounding of top_p.
//
// A row is cut into slices, so that any number of rows fills the chip, and a
// workgroup holds its slice in registers: all its loads are in flight at once
// and every further look at an element is free of memory.
//  * With a threshold, two launches. The first finds a slice's maximum and the
//    probability (count) in each of 23 steps below it. The second knows from
//    all slices of the row to within some steps where the threshold lies: it sums
//    and draws what lies above that window, keeps sum and best draw of
//    each of the window's bins apart, and the row's last slice to end finds the
//    threshold's bin and the best draw down to it.
//  * Without one, one launch, and keys that hang on no maximum: a slice leaves out
//    what the largest possible draw would not lift over the best of its threads'
//    own maxima.
// A step's probability is added up in an LDS column of the thread's own, so nothing
// collides (LDS float atomics took ten times as long); an element that is drawn costs
// ~330 cycles of hashing a wave, so sparse ones are gathered into full waves first.
// 160 rows of 151936, us, against four launches that each read all logits: top_p 0.95 of
// peaked logits 84 -> 47, of a language model's 79 -> 38, of flat ones, where most is
// drawn, 102 -> 102; top_k 50 75 -> 41; no threshold, a model's logits 40 -> 22. One row
// without a threshold 11.3 -> 8.8. Bound by vector work: ~14 instructions an element for
// the steps (20 us), then the hash of what lies above the window's end.
#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>
#include "common.h"

typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

namespace {

constexpr int NBINS = 1024;
constexpr float ZRANGE = 32.f;        // z below -32 has no probability left
// u is at most 1 - 2^-24 and at least 2^-24: a draw adds between -2.82 and
// 16.64 to z. The row maximum (z = 0) reaches -2.82, nothing below -19.46 does.
constexpr float ZDRAW = -19.5f, MOST = 16.7f;

DEV_INLINE float bf_lo(uint32_t w) { return __uint_as_float(w << 16); }
DEV_INLINE float bf_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

DEV_INLINE uint64_t row_seed(const int64_t* seeds, const int64_t* step, int row) {
  return (uint64_t)seeds[row] ^ splitmix64(0x5D21u + (uint64_t)*step);
}

DEV_INLINE int bin_of(float z) { return min(NBINS - 1, (int)(-z * (NBINS / ZRANGE))); }

// The best key of a lane; equal keys go to the lower index.
template <typename K>
struct BestOf {
  K key = std::is_same<K, double>::value ? (K)-1e300 : (K)-1e30f;    // below all
  int idx = 0x7fffffff;
  DEV_INLINE void offer(K k, int i) {
    if (k > key || (k == key && i < idx)) { key = k; idx = i; }
  }
  DEV_INLINE void over_wave() {
    #pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const K k = __shfl_xor(key, off, WAVE);
      const int i = __shfl_xor(idx, off, WAVE);
      offer(k, i);
    }
  }
};
using Best = BestOf<float>;

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

// -log(-log u), u = (the hash's upper 24 bits + 1) / 2^24, kept below 1: u = 1
// would make the key infinite and draw the element whatever its probability.
// Neither logarithm's argument is ever denormal.
DEV_INLINE float gumbel(uint64_t seed, int idx) {
  constexpr float LN2 = 0.6931471805599453f;
  const uint64_t h = splitmix64(seed ^ mix_index((uint32_t)idx));
  const float u = (float)min((uint32_t)(h >> 40) + 1u, (1u << 24) - 1u) * 0x1p-24f;
  return -LN2 * __builtin_amdgcn_logf(-LN2 * __builtin_amdgcn_logf(u));
}
DEV_INLINE float gumbel_key(uint64_t seed, int idx, float z) { return z + gumbel(seed, idx); }

// Sum over lanes 0..31 (and 32..63) up to this one.
template <typename T>
DEV_INLINE T upto32(T x) {
  #pragma unroll
  for (int off = 1; off < 32; off <<= 1) {
    const T y = __shfl_up(x, off, WAVE);
    if ((threadIdx.x & 31) >= off) x += y;
  }
  return x;
}

// key and index in one word whose order is that of Best; 0: nothing kept
DEV_INLINE unsigned long long word_of(const Best& b) {
  uint32_t o = __float_as_uint(b.key);
  o = (o >> 31) ? ~o : o | 0x80000000u;
  return b.idx == 0x7fffffff ? 0ull
                             : ((unsigned long long)o << 32) | (0xffffffffu - (uint32_t)b.idx);
}
DEV_INLINE int index_of(unsigned long long w) { return (int)(0xffffffffu - (uint32_t)w); }
// ----------------------------------------------------------------- slices
constexpr int CHUNKS = 10, CHUNK = 2048;       // of a slice: 80 elements a thread
constexpr int SLICE = CHUNKS * CHUNK;

// A slice of a row in a workgroup's registers, -inf past its end. 16-byte loads
// where rows are aligned for them (eight elements on end a thread), else one
// element a lane.
template <typename T, bool VEC>
struct Slice {
  static constexpr bool BF16 = std::is_same<T, __hip_bfloat16>::value;
  static constexpr uint32_t NONE = BF16 ? 0xff80ff80u : 0xff800000u;   // -inf
  uint32_t raw[CHUNKS][BF16 ? 4 : 8];

  static DEV_INLINE int at(int c, int k) {      // element of the slice
    return VEC ? c * CHUNK + (int)threadIdx.x * 8 + k : c * CHUNK + k * 256 + (int)threadIdx.x;
  }
  DEV_INLINE void load(const T* p, int n) {
    #pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      if (c * CHUNK >= n) continue;
      if constexpr (VEC) {
        const T* q = p + min(at(c, 0), n - 8);
        #pragma unroll
        for (int v = 0; v < (BF16 ? 1 : 2); ++v) {
          const u32x4 d = *reinterpret_cast<const u32x4*>(reinterpret_cast<const char*>(q) + 16 * v);
          #pragma unroll
          for (int w = 0; w < 4; ++w) raw[c][4 * v + w] = d[w];
        }
      } else {
        const uint16_t* h = reinterpret_cast<const uint16_t*>(p);
        const uint32_t* f = reinterpret_cast<const uint32_t*>(p);
        #pragma unroll
        for (int w = 0; w < (BF16 ? 4 : 8); ++w) {
          if constexpr (BF16) {
            const uint32_t lo = h[min(at(c, 2 * w), n - 1)], hi = h[min(at(c, 2 * w + 1), n - 1)];
            raw[c][w] = lo | (hi << 16);
          } else {
            raw[c][w] = f[min(at(c, w), n - 1)];
          }
        }
      }
    }
    #pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      if ((c + 1) * CHUNK <= n || c * CHUNK >= n) continue;   // a whole chunk, or none
      #pragma unroll
      for (int w = 0; w < (BF16 ? 4 : 8); ++w) {
        if constexpr (VEC) {
          if (at(c, 0) >= n) raw[c][w] = NONE;
        } else if constexpr (BF16) {
          if (at(c, 2 * w) >= n) raw[c][w] = NONE;
          else if (at(c, 2 * w + 1) >= n) raw[c][w] = (raw[c][w] & 0xffffu) | (NONE << 16);
        } else {
          if (at(c, w) >= n) raw[c][w] = NONE;
        }
      }
    }
  }
  DEV_INLINE float get(int c, int k) const {
    if constexpr (BF16) return k & 1 ? bf_hi(raw[c][k / 2]) : bf_lo(raw[c][k / 2]);
    else return __uint_as_float(raw[c][k]);
  }
  template <typename F>
  DEV_INLINE void each(int n, F f) const {      // f(element of the slice, value)
    #pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      if (c * CHUNK >= n) continue;
      #pragma unroll
      for (int k = 0; k < 8; ++k) f(at(c, k), get(c, k));
    }
  }
};

// Gathers what the lanes of a wave keep of their elements, two chunks at a time, and
// hands it on 64 at a time: f(element of the slice, value), a lane each. An element's
// ballot says where each lane's goes; a chunk of which none is kept costs its maximum
// alone. Against counts of each lane's, a prefix sum over the wave and a second look, us:
// 160 rows of 152064, top_p 0.95 47.3 -> 45.8, no threshold 55.1 -> 51.3, 135 fp32 rows
// 58.9 -> 51.6, 84 rows top_k 50 26.6 -> 24.5, one row 9.16 -> 8.81, 4 to 27 rows level.
// Which lane adds which probability hangs on the places, and a slice's sum above the window
// on that, in fp32: a threshold that lies within that rounding of a bin's edge may keep an
// element more or less than with other places.
template <typename T, bool VEC>
struct Gather {
  using Entry = std::conditional_t<Slice<T, VEC>::BF16, uint32_t, unsigned long long>;
  static constexpr int ROOM = 2 * 8 * WAVE + WAVE;
  Entry* q;                                     // ROOM entries of this wave
  int count = 0;

  template <typename F>
  DEV_INLINE void take(int at, F& f) {
    const Entry e = q[at];
    if constexpr (Slice<T, VEC>::BF16)
      f((int)(e & 0xffffu), __uint_as_float(e & 0xffff0000u));
    else
      f((int)(e >> 32), __uint_as_float((uint32_t)e));
  }
  // Every lane of the wave calls it; keep(value), which keeps what lies above some value.
  template <typename K, typename F>
  DEV_INLINE void run(const Slice<T, VEC>& s, int n, K keep, F f) {
    const int lane = threadIdx.x & (WAVE - 1);
    #pragma unroll
    for (int c0 = 0; c0 < CHUNKS; c0 += 2) {
      if (c0 * CHUNK >= n) continue;
      #pragma unroll
      for (int c = c0; c < c0 + 2; ++c) {
        if (c * CHUNK >= n) continue;
        float top = -1e30f;
        #pragma unroll
        for (int k = 0; k < 8; ++k) top = fmaxf(top, s.get(c, k));
        if (__ballot(keep(top)) == 0) continue;
        #pragma unroll
        for (int k = 0; k < 8; ++k) {
          const float x = s.get(c, k);
          const bool kept = keep(x);
          const unsigned long long who = __ballot(kept);
          if (kept) {
            const int to = count + __builtin_amdgcn_mbcnt_hi((uint32_t)(who >> 32),
                                       __builtin_amdgcn_mbcnt_lo((uint32_t)who, 0));
            const uint32_t id = s.at(c, k), bits = __float_as_uint(x);
            if constexpr (Slice<T, VEC>::BF16) q[to] = bits | id;       // SLICE < 2^16
            else q[to] = ((unsigned long long)id << 32) | bits;
          }
          count += __popcll(who);
        }
      }
      __builtin_amdgcn_wave_barrier();
      int done = 0;
      for (; done + WAVE <= count; done += WAVE) take(done + lane, f);
      count -= done;
      if (done > 0) {
        Entry e{};
        if (lane < count) e = q[done + lane];
        __builtin_amdgcn_wave_barrier();
        if (lane < count) q[lane] = e;
      }
      __builtin_amdgcn_wave_barrier();
    }
    if (lane < count) take(lane, f);
    count = 0;
  }
};

// The best of a workgroup's lanes, in thread 0.
template <typename K>
DEV_INLINE void over_block(BestOf<K>& b, K* fpart, int* ipart) {
  b.over_wave();
  if ((threadIdx.x & (WAVE - 1)) == 0) {
    fpart[threadIdx.x / WAVE] = b.key;
    ipart[threadIdx.x / WAVE] = b.idx;
  }
  __syncthreads();
  if (threadIdx.x == 0)
    for (int w = 1; w < 4; ++w) b.offer(fpart[w], ipart[w]);
}

// --------------------------------------------------------- no threshold
// What a slice passes on to the row's last slice to end, each word with the launch's
// mark above it: the halves of its best key, and that key's element. A mark's 32 bits
// might lie in old memory by chance, but not in all three.
// A key is logit / temperature + the variate, in 64 bits: of nothing but its element, so
// that a row draws the same token whatever slices it is cut into. In 32 bits, relative
// to a slice's maximum and then moved to the row's, it was rounded twice, and keys next
// to each other came out by how many rows were drawn together.
enum { KEY_LOW = 0, KEY_HIGH = 1, ELEMENT = 2, WORDS = 3 };

template <typename T, bool VEC>
__global__ __launch_bounds__(256)
void draw_kernel(const T* __restrict__ logits, int V, int per, float inv_temp,
                 const int64_t* __restrict__ seeds, const int64_t* __restrict__ step,
                 unsigned long long* __restrict__ found, uint32_t mark, int64_t* __restrict__ out) {
  __shared__ typename Gather<T, VEC>::Entry queue[4 * Gather<T, VEC>::ROOM];
  __shared__ float red[16];
  __shared__ double kpart[4];
  __shared__ int ipart[4];
  const int row = blockIdx.x, sl = blockIdx.y, S = gridDim.y, tid = threadIdx.x;
  const int i0 = sl * per, n = min(V - i0, per);
  Slice<T, VEC> s;
  s.load(logits + (int64_t)row * V + i0, n);
  const uint64_t seed = row_seed(seeds, step, row);
  float own = -1e30f;
  int own_at = 0;
  s.each(n, [&](int at, float x) {
    if (x > own) { own = x; own_at = at; }
  });
  const float m = block_max(own, red);
  // a key that is reached, relative to m and less its rounding: nothing MOST below it can be
  // the best, and no key below it is looked at in 64 bits (320 flat rows 103 us, all
  // of them 113)
  const float reached =
      block_max(gumbel_key(seed, i0 + own_at, (own - m) * inv_temp), red) - 1e-3f;
  BestOf<double> b;
  Gather<T, VEC> gather{queue + (tid / WAVE) * Gather<T, VEC>::ROOM};
  gather.run(s, n, [&](float x) { return (x - m) * inv_temp > reached - MOST; },
             [&](int at, float x) {
               const float g = gumbel(seed, i0 + at);
               if ((x - m) * inv_temp + g > reached) b.offer((double)x * inv_temp + g, i0 + at);
             });
  over_block(b, kpart, ipart);
  if (tid >= WAVE) return;
  // a maximum of infinity: nothing is finite beside it, and the row has no draw
  if (__float_as_uint(m) == 0x7f800000u) b = {1e300, 0x7fffffff};
  // Of the row's slices the last to come finds all of them here, as each looks only
  // when its own words have arrived. Another may, too, and writes the same token.
  // Nothing has to be cleared first; who has seen all clears them, because a replay of
  // a captured launch has the same mark.
  unsigned long long* const words = found + (int64_t)row * S * WORDS;
  const unsigned long long high = (unsigned long long)mark << 32;
  const unsigned long long key = (unsigned long long)__double_as_longlong(b.key);
  const uint32_t own_word[WORDS] = {(uint32_t)key, (uint32_t)(key >> 32), (uint32_t)b.idx};
  if (tid == 0) {
    #pragma unroll
    for (int i = 0; i < WORDS; ++i) store_through(words + sl * WORDS + i, high | own_word[i]);
  }
  stores_done();
  bool all_here = true;
  b = {};
  for (int i = tid; i < S; i += WAVE) {
    unsigned long long w[WORDS];
    #pragma unroll
    for (int j = 0; j < WORDS; ++j) w[j] = load_through(words + i * WORDS + j);
    #pragma unroll
    for (int j = 0; j < WORDS; ++j) all_here = all_here && (w[j] >> 32) == mark;
    b.offer(__longlong_as_double((long long)(w[KEY_HIGH] << 32 | (uint32_t)w[KEY_LOW])),
            (int)(uint32_t)w[ELEMENT]);
  }
  if (__ballot(!all_here) != 0) return;
  b.over_wave();
  if (tid == 0) out[row] = b.idx == 0x7fffffff ? 0 : b.idx;
  for (int i = tid; i < S * WORDS; i += WAVE) words[i] = 0ull;
}

// ------------------------------------------------------------- threshold
// Steps of -z, one wide from 0 to 20 and four wide from there to 32, where little is
// left that a window could hold. Steps of half an octave are eleven instead of 23, but
// with a threshold 11 below the maximum the window took in most of a row (72 us of
// drawing for 160 rows).
constexpr int STEPS = 23;
DEV_INLINE int step_of(float t) { return (int)fminf(t, 15.f + 0.25f * t); }
constexpr int LEVELS = 64;             // at which a row's steps are compared, z = 1/2 apart
constexpr int PER_LEVEL = NBINS / LEVELS;
// Bins in which the threshold may lie: up to a step, two levels and rounding.
constexpr int WINDOW = 16 * PER_LEVEL;
constexpr int POOL = 768;              // as often as they fit, in LDS

// Of a slice: its maximum, probability and count down to each step below it. Of a
// row: slices that are done; sum, count and best draw above the window (entry 0)
// and in its bins.
struct Sums {
  float *top, *p;                      // (B, S), (B, S, STEPS)
  int* c;                              // (B, S, STEPS)
  unsigned long long *mass, *best;     // (B, 1 + WINDOW)
  int *count, *done;                   // (B, 1 + WINDOW), (B)
  // What probability meets in: whole numbers of 1 / unit (back), 2^-44 for 152064
  // elements, so that the most there is, one of each, fits. Of 2^-32 100000 elements 14
  // below the maximum, rounded one by one, were up to 1e-5 of the row too much or little.
  float unit, back;
  DEV_INLINE unsigned long long whole(float p) const { return (unsigned long long)(p * unit + 0.5f); }
};

DEV_INLINE int64_t width_at(int row) { return (int64_t)row * (1 + WINDOW); }

template <typename T, bool VEC, bool BY_P, bool BY_K>
__global__ __launch_bounds__(256)
void steps_kernel(const T* __restrict__ logits, int V, int per, float inv_temp, Sums sums) {
  __shared__ float hp[BY_P ? STEPS * 256 : 1];          // [step][thread]
  __shared__ uint32_t hc[BY_K ? (STEPS + 3) / 4 * 256 : 1];   // four counts a word, 80 at most each
  __shared__ float red[4], tp[STEPS];
  __shared__ int tc[STEPS];
  const int row = blockIdx.x, sl = blockIdx.y, S = gridDim.y, tid = threadIdx.x;
  const int i0 = sl * per, n = min(V - i0, per);
  Slice<T, VEC> s;
  s.load(logits + (int64_t)row * V + i0, n);
  if (sl == 0) {
    for (int i = tid; i < 1 + WINDOW; i += 256) {
      sums.mass[width_at(row) + i] = sums.best[width_at(row) + i] = 0ull;
      sums.count[width_at(row) + i] = 0;
    }
    if (tid == 0) sums.done[row] = 0;
  }
  float m = -1e30f;
  s.each(n, [&](int, float x) { m = fmaxf(m, x); });
  if (BY_P)
    #pragma unroll
    for (int i = 0; i < STEPS; ++i) hp[i * 256 + tid] = 0.f;
  if (BY_K)
    #pragma unroll
    for (int i = 0; i < (STEPS + 3) / 4; ++i) hc[i * 256 + tid] = 0;
  m = block_max(m, red);
  s.each(n, [&](int, float x) {
    // without branches; what lies deeper adds e^-32, nothing beside the maximum's 1
    const float below = (m - x) * inv_temp, t = fminf(below, ZRANGE - 0.01f);
    const int g = step_of(t);
    if (BY_P) hp[g * 256 + tid] += __expf(-t);
    if (BY_K) hc[(g >> 2) * 256 + tid] += below < ZRANGE ? 1u << (g & 3) * 8 : 0u;
  });
  __syncthreads();
  const int wid = tid / WAVE, lane = tid & (WAVE - 1);
  for (int b = wid; b < STEPS; b += 4) {
    if (BY_P) {
      float v = 0.f;
      #pragma unroll
      for (int i = 0; i < 4; ++i) v += hp[b * 256 + i * WAVE + lane];
      v = wave_sum(v);
      if (lane == 0) tp[b] = v;
    }
    if (BY_K) {
      int v = 0;
      #pragma unroll
      for (int i = 0; i < 4; ++i) v += (hc[(b >> 2) * 256 + i * WAVE + lane] >> (b & 3) * 8) & 255;
      #pragma unroll
      for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, WAVE);
      if (lane == 0) tc[b] = v;
    }
  }
  __syncthreads();
  if (tid >= 32) return;
  const int64_t at = (int64_t)row * S + sl;
  if (tid == 0) sums.top[at] = m;
  const int b = min(tid, STEPS - 1);
  if (BY_P) {
    const float v = upto32(tid < STEPS ? tp[b] : 0.f);
    if (tid < STEPS) sums.p[at * STEPS + b] = v;
  }
  if (BY_K) {
    const int v = upto32(tid < STEPS ? tc[b] : 0);
    if (tid < STEPS) sums.c[at * STEPS + b] = v;
  }
}

// Bins [first, end) in which the threshold lies, from the steps of a row's slices; all
// threads get it. With a slice's maximum at z = d a level -L is L + d below it: down to
// there the slice holds at least the steps that end above it and at most those that
// begin above it.
struct Window { int first, end; float total; };

// LDS of the search: the steps of as many slices as a wave has lanes, then sums of its
// four shares.
struct Search {
  static constexpr int AT_ONCE = WAVE;
  unsigned long long total[AT_ONCE];
  float p[AT_ONCE * STEPS], d[AT_ONCE], w[AT_ONCE];
  int c[AT_ONCE * STEPS];
};
struct Shares {
  float f[4][LEVELS][2];
  unsigned long long total[4];
  int i[4][LEVELS][2];
};

template <bool BY_P, bool BY_K>
DEV_INLINE Window find_window(const Sums& sums, int row, int S, float m, float inv_temp, float top_p,
                              int top_k, char* lds) {
  auto& in = *reinterpret_cast<Search*>(lds);
  auto& out = *reinterpret_cast<Shares*>(lds);
  const int tid = threadIdx.x, L = tid & (LEVELS - 1), sub = tid / LEVELS;
  float least = 0.f, most = 0.f;
  // Slices meet in it as whole numbers, as in the masses; made of each once, not by every
  // level's lane (74 slices: 0.8 of 25 us).
  unsigned long long total = 0;
  int cleast = 0, cmost = 0;
  for (int s0 = 0; s0 < S; s0 += Search::AT_ONCE) {
    const int n = min(S - s0, Search::AT_ONCE);
    const int64_t at = (int64_t)row * S + s0;
    if (s0) __syncthreads();
    #pragma unroll
    for (int i = 0; i < CDIV(Search::AT_ONCE * STEPS, 256); ++i) {
      const int j = i * 256 + tid;
      if (BY_P && j < n * STEPS) in.p[j] = sums.p[at * STEPS + j];
      if (BY_K && j < n * STEPS) in.c[j] = sums.c[at * STEPS + j];
    }
    if (tid < n) {
      const float all = BY_P ? sums.p[(at + tid) * STEPS + STEPS - 1] : 0.f;
      const float d = fmaxf((sums.top[at + tid] - m) * inv_temp, -1000.f), w = __expf(d);
      in.d[tid] = d;
      in.w[tid] = w;
      if (BY_P) in.total[tid] = sums.whole(w * all);
    }
    __syncthreads();
    for (int s = sub; s < n; s += 4) {
      // what lies on a level's edge may have been rounded over it
      const float t = L * (ZRANGE / LEVELS) + in.d[s], w = in.w[s];
      const int ends = t > 2e-4f ? min(step_of(t - 1e-4f) - 1, STEPS - 1) : -1;
      const int begins = t > -1e-4f ? min(step_of(fmaxf(t, 0.f) + 1e-4f), STEPS - 1) : -1;
      if (BY_P) {
        const float* p = in.p + s * STEPS;
        least += ends >= 0 ? w * p[max(ends, 0)] : 0.f;
        most += begins >= 0 ? w * p[max(begins, 0)] : 0.f;
        total += in.total[s];
      }
      if (BY_K) {
        const int* c = in.c + s * STEPS;
        cleast += ends >= 0 ? c[max(ends, 0)] : 0;
        cmost += begins >= 0 ? c[max(begins, 0)] : 0;
      }
    }
  }
  __syncthreads();
  if (BY_P) { out.f[sub][L][0] = least; out.f[sub][L][1] = most; out.total[sub] = total; }
  if (BY_K) { out.i[sub][L][0] = cleast; out.i[sub][L][1] = cmost; }
  __syncthreads();
  least = most = 0.f;
  total = 0;
  cleast = cmost = 0;
  #pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (BY_P) { least += out.f[i][L][0]; most += out.f[i][L][1]; total += out.total[i]; }
    if (BY_K) { cleast += out.i[i][L][0]; cmost += out.i[i][L][1]; }
  }
  // a level a lane; reached at the end of z if nowhere before
  auto cut = [&](bool reached, bool short_of, int& first, int& end) {
    const unsigned long long r = __ballot(reached), o = __ballot(short_of);
    first = max(0, 63 - __clzll((long long)o));     // __clzll(0) = 64: none
    end = min(r ? __ffsll(r) - 1 : LEVELS, first + WINDOW / PER_LEVEL);
    end = max(end, first + 1);
  };
  Window w{0, LEVELS, (float)total * sums.back};
  if (BY_P) {
    const float target = top_p * w.total;
    cut(least >= target * (1.f + 2e-6f), most < target * (1.f - 2e-6f), w.first, w.end);
  }
  if (BY_K) {
    int first, end;
    cut(cleast >= top_k, cmost < top_k, first, end);
    w.first = BY_P ? min(w.first, first) : first;
    w.end = BY_P ? min(w.end, end) : end;
  }
  w.first *= PER_LEVEL;
  w.end *= PER_LEVEL;
  return w;
}

template <typename T, bool VEC, bool BY_P, bool BY_K>
__global__ __launch_bounds__(256)
void pick_kernel(const T* __restrict__ logits, int V, int per, float inv_temp, float top_p,
                 int top_k, Sums sums, const int64_t* __restrict__ seeds,
                 const int64_t* __restrict__ step, int64_t* __restrict__ out) {
  __shared__ typename Gather<T, VEC>::Entry queue[4 * Gather<T, VEC>::ROOM];
  __shared__ unsigned long long wmass[BY_P ? POOL : 1], wbest[POOL];   // [bin][copy]
  __shared__ int wcount[BY_K ? POOL : 1];
  __shared__ float red[4], fpart[4];
  __shared__ int ipart[4], last;
  // the search for the window comes before the gathering
  static_assert(sizeof(queue) >= sizeof(Search) && sizeof(queue) >= sizeof(Shares), "");
  const int row = blockIdx.x, sl = blockIdx.y, S = gridDim.y, tid = threadIdx.x;
  const int i0 = sl * per, n = min(V - i0, per);
  Slice<T, VEC> s;
  s.load(logits + (int64_t)row * V + i0, n);
  for (int i = tid; i < POOL; i += 256) {
    if (BY_P) wmass[i] = 0ull;
    if (BY_K) wcount[i] = 0;
    wbest[i] = 0ull;
  }
  float m = -1e30f;
  for (int i = tid & (WAVE - 1); i < S; i += WAVE) m = fmaxf(m, sums.top[(int64_t)row * S + i]);
  m = wave_max(m);
  const Window w = find_window<BY_P, BY_K>(sums, row, S, m, inv_temp, top_p, top_k,
                                            reinterpret_cast<char*>(queue));
  __syncthreads();
  const uint64_t seed = row_seed(seeds, step, row);
  const float zlow = -w.end * (ZRANGE / NBINS);
  const int bins = w.end - w.first;
  const int copies = 1 << (31 - __clz(min(POOL / bins, 16))), copy = tid & (copies - 1);
  Best b;
  float above = 0.f;
  int cabove = 0;
  Gather<T, VEC> gather{queue + (tid / WAVE) * Gather<T, VEC>::ROOM};
  gather.run(s, n, [&](float x) { return (x - m) * inv_temp > zlow; }, [&](int at, float x) {
    const float z = (x - m) * inv_temp;
    const int bin = bin_of(z);
    const float p = BY_P ? __expf(z) : 0.f;
    Best e;
    if (z > ZDRAW) e.offer(gumbel_key(seed, i0 + at, z), i0 + at);
    if (bin < w.first) {
      above += p;
      ++cabove;
      b.offer(e.key, e.idx);
    } else {
      const int to = min(bin - w.first, bins - 1) * copies + copy;
      if (BY_P) atomicAdd(wmass + to, sums.whole(p));
      if (BY_K) atomicAdd(wcount + to, 1);
      const unsigned long long o = word_of(e);
      if (o > wbest[to]) atomicMax(wbest + to, o);      // seldom
    }
  });
  over_block(b, fpart, ipart);                  // waits for the window too
  const int64_t at = width_at(row);
  above = block_sum(above, red);
  if (BY_K) {
    #pragma unroll
    for (int off = 32; off > 0; off >>= 1) cabove += __shfl_xor(cabove, off, WAVE);
    if ((tid & (WAVE - 1)) == 0 && cabove) atomicAdd(sums.count + at, cabove);
  }
  if (tid == 0) {
    if (BY_P && above != 0.f)
      atomicAdd(sums.mass + at, sums.whole(above));
    if (word_of(b)) atomicMax(sums.best + at, word_of(b));
  }
  for (int j = tid; j < bins; j += 256) {
    unsigned long long mass = 0, best = 0;
    int count = 0;
    for (int i = j * copies; i < (j + 1) * copies; ++i) {
      if (BY_P) mass += wmass[i];
      if (BY_K) count += wcount[i];
      best = wbest[i] > best ? wbest[i] : best;
    }
    if (BY_P && mass) atomicAdd(sums.mass + at + 1 + j, mass);
    if (BY_K && count) atomicAdd(sums.count + at + 1 + j, count);
    if (best) atomicMax(sums.best + at + 1 + j, best);
  }
  stores_done();
  __syncthreads();
  if (tid == 0) last = atomicAdd(&sums.done[row], 1) == S - 1;
  __syncthreads();
  if (!last) return;
  // all slices have arrived: their sums come into LDS, and the first wave walks them
  for (int j = tid; j < (bins + 31) / 32 * 32; j += 256) {
    if (BY_P) wmass[j] = load_through(sums.mass + at + 1 + j);
    if (BY_K) wcount[j] = load_through(sums.count + at + 1 + j);
    wbest[j] = load_through(sums.best + at + 1 + j);
  }
  __syncthreads();
  if (tid >= WAVE) return;
  const float target = top_p * w.total;
  unsigned long long best = load_through(sums.best + at);
  unsigned long long mass = BY_P ? load_through(sums.mass + at) : 0ull;
  int count = BY_K ? load_through(sums.count + at) : 0;
  for (int b0 = 0; b0 < bins; b0 += 32) {
    const int i = b0 + (tid & 31);            // POOL is a multiple of 32; zeros past the end
    const unsigned long long pm = BY_P ? mass + upto32(wmass[i]) : 0ull;
    const int pc = BY_K ? count + upto32(wcount[i]) : 0;
    const uint32_t hit = (uint32_t)__ballot((BY_P && (float)pm * sums.back >= target) ||
                                            (BY_K && pc >= top_k));
    const int kept = hit ? __ffs((int)hit) : 32;      // down to the threshold's bin
    unsigned long long o = (tid & 31) < kept ? wbest[i] : 0ull;
    #pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const unsigned long long y = __shfl_xor(o, off, WAVE);
      o = y > o ? y : o;
    }
    best = o > best ? o : best;
    if (hit) break;
    mass = __shfl(pm, 31, WAVE);
    count = __shfl(pc, 31, WAVE);
  }
  if (tid == 0) out[row] = best == 0ull ? 0 : (int64_t)index_of(best);
}

// Slices of a row: two or three workgroups a CU, none longer than a workgroup's
// registers hold or shorter than `least`. A workgroup of the threshold's launches takes
// ~8 us whatever its slice (32 rows of 151936 in 640, 1280, 1920 workgroups 21, 26, 41
// us; from 80 rows on the longest slices are more anyway).
int slices(int B, int V, int least) {
  return std::max(CDIV(V, SLICE), std::max(1, std::min(V / least, 640 / B)));
}

template <typename T, bool VEC>
void sample_slices(const T* logits, int B, int V, float inv_t, float top_p, int top_k,
                   const torch::Tensor& seeds, const torch::Tensor& step, torch::Tensor& out) {
  const bool by_p = top_p < 1.f, by_k = top_k > 0;
  int S = slices(B, V, by_p || by_k ? 2048 : 1024);
  const int per = CDIV(CDIV(V, S), 8) * 8;
  S = CDIV(V, per);
  TORCH_CHECK(per <= SLICE && (int64_t)per * S >= V && (int64_t)per * (S - 1) < V && S < 65536);
  const int64_t rows = B, cells = rows * S;
  auto stream = at::cuda::getCurrentCUDAStream();
  const dim3 grid(B, S), block(256);
  auto room = [&](int64_t bytes) {
    return torch::empty({bytes}, out.options().dtype(at::kByte));
  };
  if (!by_p && !by_k) {
    auto ws = room(cells * WORDS * 8);
    hipLaunchKernelGGL((draw_kernel<T, VEC>), grid, block, 0, stream, logits, V, per, inv_t,
                       seeds.data_ptr<int64_t>(), step.data_ptr<int64_t>(),
                       reinterpret_cast<unsigned long long*>(ws.data_ptr()),
                       (uint32_t)(arrival_tag() >> 32), out.data_ptr<int64_t>());
    return;
  }
  auto ws = room(rows * (1 + WINDOW) * 20 + rows * 4 + cells * 4 * (1 + 2 * STEPS));
  Sums sums;
  sums.mass = reinterpret_cast<unsigned long long*>(ws.data_ptr());
  sums.best = sums.mass + rows * (1 + WINDOW);
  sums.count = reinterpret_cast<int*>(sums.best + rows * (1 + WINDOW));
  sums.done = sums.count + rows * (1 + WINDOW);
  sums.top = reinterpret_cast<float*>(sums.done + rows);
  sums.p = sums.top + cells;
  sums.c = reinterpret_cast<int*>(sums.p + cells * STEPS);
  sums.unit = std::ldexp(1.f, 30 + __builtin_clz(V));   // V times it: 2^62 at most
  sums.back = 1.f / sums.unit;
  auto go = [&](auto p_, auto k_) {
    constexpr bool P = decltype(p_)::value, K = decltype(k_)::value;
    hipLaunchKernelGGL((steps_kernel<T, VEC, P, K>), grid, block, 0, stream, logits, V, per, inv_t,
                       sums);
    hipLaunchKernelGGL((pick_kernel<T, VEC, P, K>), grid, block, 0, stream, logits, V, per, inv_t,
                       top_p, top_k, sums, seeds.data_ptr<int64_t>(), step.data_ptr<int64_t>(),
                       out.data_ptr<int64_t>());
  };
  if (by_p && by_k) go(std::true_type{}, std::true_type{});
  else if (by_p) go(std::true_type{}, std::false_type{});
  else go(std::false_type{}, std::true_type{});
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
