// Paged-attention decode (GQA) over the block-paged KV pool — the decode
// hot loop of the generation engine (reference counterpart: vLLM
// paged_attention_v1/v2).
//
// One workgroup owns (sequence, kv head, slice of the context) with all query
// heads of the kv head; its waves take 32 tokens each in turn and keep a
// softmax of their own, joined once at the end. Per 32 tokens a wave
//  * loads whole K and V rows, neighbouring lanes neighbouring 16 B pieces, and
//    passes both through tiles of its own in LDS (K straight into MFMA operands,
//    a row a lane, touched a cache line a lane: the round below 74.7 us, 70.4
//    now, three long chats 11.3 and 10.6); no workgroup barrier in the loop;
//  * forms S^T[token][head] = K Q^T (16x16x32), q and K exact in bf16, sums in
//    fp32;
//  * keeps the weights in fp32 and feeds them to the second product as two
//    bf16 terms, p = hi + lo (error 2^-17 of p): the accumulator's token rows
//    serve as k-slots as they lie;
//  * reads V back transposed (LDS transpose reads).
// The next 32 tokens' rows are in flight meanwhile (page numbers two ahead).
//
// The engine's step fuses what stands before it: the workgroup of (sequence, kv
// head) takes its heads from the projections' packed rows, or from a product's
// partial sums and the bias, norms and rotates them, writes the new token's key
// and value into the cache and attends over them from LDS, while the first rows
// of the context are on their way. Slices of one sequence are joined by the last
// of them to end (as a launch of its own that took 3 us). As kernels of their own
// rotation and join took 7.7 and 4.6 us a layer at 160 sequences, 3.0 and 1.3 at eight.
// K and V are read once per sequence and kv head; bound by HBM.
// 160 sequences of 420..1550 tokens sharing prompts, 28/4 heads of 128
// (251 MB of distinct rows): 157 us with one lane a token on vector FMAs,
// 67 us now; 3 sequences of 911..3777, 14/2 heads of 64: 43 -> 8.4, a chain of
// length and pages, rows, products and the slices' join.
#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>
#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16v8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16v4;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((address_space(3))) bf16v4 lds_bf16v4;

namespace {

constexpr float LOG2E = 1.4426950408889634f;
constexpr int CHUNK = 32;        // tokens of a wave's step

// 16 B chunk c of row r in a wave's V tile: rows read at one chunk (writes)
// and 16 rows read over two chunks (transpose reads) spread over the banks.
template <int D>
DEV_INLINE int v_off(int r, int c) {
  return r * (2 * D) + ((c ^ (D == 128 ? r & 15 : (r >> 1) & 7)) << 4);
}

// What the fused kernel makes its queries, keys and values from: packed rows
// [q heads | k heads | v heads], as bf16 or as fp32 partial sums (splits, N, width)
struct Packed {
  const __hip_bfloat16* rows;
  const float* parts;
  int splits;
  const __hip_bfloat16* bias;                 // of the parts, or null
  const int* positions;
  const int64_t* slots;                       // cache rows; negative: none
  const float* inv_freq;
  const __hip_bfloat16 *q_norm, *k_norm;      // or null
  float eps;
  __hip_bfloat16 *kcache, *vcache;
  int* arrived;                               // (N, KV), zero before and after
};

enum { QUERIES = 0, ROWS = 1, PARTS = 2 };

template <int D, int NW, int SRC>
__global__ __launch_bounds__(NW * 64, 2)
void paged_decode_kernel(const __hip_bfloat16* __restrict__ q,      // rows of q_row_stride
                         const __hip_bfloat16* __restrict__ kcache, // (nb, bs, KV, D)
                         const __hip_bfloat16* __restrict__ vcache,
                         const int* __restrict__ block_tables,      // (N, max_nb)
                         const int* __restrict__ ctx_lens,          // (N,)
                         __hip_bfloat16* __restrict__ out,          // (N, H, D)
                         float* __restrict__ o_part,                // (cs, N, H, D)
                         float* __restrict__ ml_part,               // (cs, N, H, 2)
                         int H, int KV, int max_nb, int block_size, int bs_shift,
                         float scale_log2, int64_t q_row_stride, int slice_len,
                         unsigned long long* __restrict__ there,    // (N, KV, cs)
                         unsigned long long tag, Packed src) {
  constexpr int KS = D / 32, DT = D / 16;
  constexpr int LPR = D / 8, RPL = 64 / LPR, NL = CHUNK / RPL;   // lanes of a row, rows of a load
  const int seq = blockIdx.x, kv = blockIdx.y, z = blockIdx.z, N = gridDim.x;
  const int group = H / KV;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = threadIdx.x & 63, g = l >> 4, lr = l & 15;
  const int* bt = block_tables + (int64_t)seq * max_nb;
  const int c0 = z * slice_len;
  auto block_of = [&](int t) { return bs_shift >= 0 ? t >> bs_shift : t / block_size; };
  // What a workgroup needs first is on its way at once: the length, its pages, and
  // below what its queries are made of. One behind the other they are a microsecond each.
  int t0 = c0 + wave * CHUNK;
  // the page of this lane's token l % 32 of the first chunk, whether there is one or not
  int page = max_nb > 0 ? bt[min(block_of(t0 + (l & 31)), max_nb - 1)] : 0;
  const int len = ctx_lens[seq];
  // no further than the block table reaches
  const int c1 = min(len, min(c0 + slice_len, max_nb * block_size));
  if (z > 0 && c0 >= len) return;       // an empty slice is not read

  extern __shared__ __attribute__((aligned(16))) char smem[];
  char* ktile = smem + wave * (2 * CHUNK * D * 2);      // also 16 heads x D floats
  char* tile = ktile + CHUNK * D * 2;
  float* ml_lds = reinterpret_cast<float*>(smem + NW * (2 * CHUNK * D * 2));  // [NW][16][2]
  // fused: the heads' queries, then the new token's key and value
  __hip_bfloat16* fresh = reinterpret_cast<__hip_bfloat16*>(ml_lds + NW * 32);
  // only the slice that has the new token makes its key and value: another one's
  // rows past its end repeat the cache's row before (weight zero, but it must be a
  // number)
  const bool owner = z + 1 == (int)gridDim.z || c0 + slice_len >= len;
  const int last = SRC == QUERIES || !owner ? 0x7fffffff : len - 1;

  float m = -1e30f, lsum = 0.f;
  f32x4 acc[DT];
  #pragma unroll
  for (int dt = 0; dt < DT; ++dt) acc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int row_elems = KV * D;
  bf16v8 kf[NL], vf[NL];
  auto token = [&](int t0) { return min(t0 + (l & 31), c1 - 1); };     // past the end: weight zero
  auto load = [&](int page, int t0) {   // page: of this lane's token
    const int t = token(t0), row = page * block_size + (t - block_of(t) * block_size);
    #pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int64_t at = (int64_t)__shfl(row, i * RPL + l / LPR, WAVE) * row_elems + kv * D +
                         (l % LPR) * 8;
      kf[i] = *reinterpret_cast<const bf16v8*>(kcache + at);
      vf[i] = *reinterpret_cast<const bf16v8*>(vcache + at);
    }
  };

  auto begin = [&] {
    if (t0 < c1) {
      load(__shfl(page, token(t0) - t0, WAVE), t0);
      // With the length known a chunk's pages are looked up where its rows end: lanes
      // that trade them for every chunk stand in front of its rows (32 of 300..1500,
      // 40/8 heads 26.4 us, 26.05 so; 300 of 60..400, 14/2 heads 10.1 and 10.0).
      page = bt[block_of(token(t0 + NW * CHUNK))];
    }
  };
  bf16v8 qf[KS];
  if constexpr (SRC == QUERIES) {
    begin();
    #pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const __hip_bfloat16* qp = q + seq * q_row_stride + (kv * group + min(lr, group - 1)) * D;
      qf[ks] = *reinterpret_cast<const bf16v8*>(qp + ks * 32 + g * 8);   // spare columns repeat
    }
  } else {
    // eight rotation pairs a thread, so a head takes D / 16 neighbouring lanes;
    // then the value, eight elements a thread
    constexpr int PER = D / 16;
    const int width = (H + 2 * KV) * D;
    const int64_t slot = src.slots[seq];
    const int units = (group + (owner ? 1 : 0)) * PER, all = units + (owner ? D / 8 : 0);
    // eight elements at `at` and eight at `other` of this sequence: the rows, or the
    // first partial sums of them. Four hold 64 registers, 182 in all with rows of 64: two
    // workgroups of four waves a CU instead of three (160 sequences of 30..200, 16/4
    // heads 14.1 us, two 10.0; 96 of 100..600, 8/8 heads 22.8 and 18.8). Eight waves run
    // one workgroup a CU, rows of 128 two with either.
    constexpr int AHEAD = D == 64 && NW == 4 ? 2 : 4;
    struct Raw {
      bf16x8 x, y;
      f32x4v part[AHEAD][4];
    };
    auto fetch = [&](Raw& r, int at, int other) {
      if constexpr (SRC == ROWS) {
        const __hip_bfloat16* p = src.rows + (int64_t)seq * width;
        r.x = *reinterpret_cast<const bf16x8*>(p + at);
        r.y = *reinterpret_cast<const bf16x8*>(p + other);
      } else {
        #pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
          const float* p = src.parts + ((int64_t)min(i, src.splits - 1) * N + seq) * width;
          #pragma unroll
          for (int h = 0; h < 2; ++h) {
            r.part[i][h] = *reinterpret_cast<const f32x4v*>(p + at + 4 * h);
            r.part[i][2 + h] = *reinterpret_cast<const f32x4v*>(p + other + 4 * h);
          }
        }
      }
    };
    auto take = [&](const Raw& r, float (&x)[8], float (&y)[8], int at, int other) {
      if constexpr (SRC == ROWS) {
        #pragma unroll
        for (int j = 0; j < 8; ++j) { x[j] = bf2f(r.x.v[j]); y[j] = bf2f(r.y.v[j]); }
      } else {
        #pragma unroll
        for (int j = 0; j < 8; ++j) {
          x[j] = src.bias ? bf2f(src.bias[at + j]) : 0.f;
          y[j] = src.bias ? bf2f(src.bias[other + j]) : 0.f;
        }
        #pragma unroll
        for (int i = 0; i < AHEAD; ++i)
          if (i < src.splits) {
            #pragma unroll
            for (int j = 0; j < 8; ++j) {
              x[j] += r.part[i][j / 4].v[j % 4];
              y[j] += r.part[i][2 + j / 4].v[j % 4];
            }
          }
        if (src.splits > AHEAD)
          add_parts8x2(x, y, src.parts + ((int64_t)AHEAD * N + seq) * width + at, other - at,
                       (int64_t)N * width, src.splits - AHEAD);
      }
    };
    // where unit u's elements are: of the value eight, twice
    auto places = [&](int u, int& at, int& other) {
      if (u >= units) {
        at = other = (H + KV + kv) * D + (u - units) * 8;
      } else {
        const int head = u / PER;
        at = (head < group ? kv * group + head : H + kv) * D + u % PER * 8;
        other = at + D / 2;
      }
    };
    Raw raw;
    int at, other;
    if ((int)threadIdx.x < all) {
      places(threadIdx.x, at, other);
      fetch(raw, at, other);
    }
    begin();
    for (int u = threadIdx.x; u < all; u += NW * 64) {
      if (u >= NW * 64) {
        places(u, at, other);
        fetch(raw, at, other);
      }
      bf16x8 x, y;
      float x1[8], x2[8];
      take(raw, x1, x2, at, other);
      if (u >= units) {
        const int c = (u - units) * 8;
        #pragma unroll
        for (int j = 0; j < 8; ++j) x.v[j] = f2bf(x1[j]);
        *reinterpret_cast<bf16x8*>(fresh + (group + 1) * D + c) = x;
        if (slot >= 0)
          *reinterpret_cast<bf16x8*>(src.vcache + (slot * KV + kv) * D + c) = x;
        continue;
      }
      const int head = u / PER, c = u % PER * 8;        // head == group: the key
      const __hip_bfloat16* nw = head < group ? src.q_norm : src.k_norm;
      if (nw) {
        float ss = 0.f;
        #pragma unroll
        for (int j = 0; j < 8; ++j) ss += x1[j] * x1[j] + x2[j] * x2[j];
        #pragma unroll
        for (int off = PER / 2; off > 0; off >>= 1) ss += __shfl_xor(ss, off, WAVE);
        const float r = rsqrtf(ss / D + src.eps);
        #pragma unroll
        for (int j = 0; j < 8; ++j) {
          x1[j] *= r * bf2f(nw[c + j]);
          x2[j] *= r * bf2f(nw[c + D / 2 + j]);
        }
      }
      const float pos = (float)src.positions[seq];
      #pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float a = pos * src.inv_freq[c + j], sn = __sinf(a), cs = __cosf(a);
        x.v[j] = f2bf(x1[j] * cs - x2[j] * sn);
        y.v[j] = f2bf(x2[j] * cs + x1[j] * sn);
      }
      *reinterpret_cast<bf16x8*>(fresh + head * D + c) = x;
      *reinterpret_cast<bf16x8*>(fresh + head * D + c + D / 2) = y;
      if (head == group && slot >= 0) {
        __hip_bfloat16* kd = src.kcache + (slot * KV + kv) * D + c;
        *reinterpret_cast<bf16x8*>(kd) = x;
        *reinterpret_cast<bf16x8*>(kd + D / 2) = y;
      }
    }
    __syncthreads();
    #pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      qf[ks] = *reinterpret_cast<const bf16v8*>(fresh + min(lr, group - 1) * D + ks * 32 + g * 8);
  }
  for (; t0 < c1; t0 += NW * CHUNK) {
    const bool more = t0 + NW * CHUNK < c1;             // wave-uniform
    if (SRC != QUERIES && t0 + CHUNK > last) {
      // the new token, and what repeats it past the end: its row of the cache may
      // not be written yet
      #pragma unroll
      for (int i = 0; i < NL; ++i)
        if (t0 + i * RPL + l / LPR >= last) {
          kf[i] = *reinterpret_cast<const bf16v8*>(fresh + group * D + l % LPR * 8);
          vf[i] = *reinterpret_cast<const bf16v8*>(fresh + (group + 1) * D + l % LPR * 8);
        }
    }
    #pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int r = i * RPL + l / LPR, c = l % LPR;
      *reinterpret_cast<bf16v8*>(ktile + v_off<D>(r, c)) = kf[i];
      *reinterpret_cast<bf16v8*>(tile + v_off<D>(r, c)) = vf[i];
    }
    if (more) {
      load(page, t0 + NW * CHUNK);
      page = bt[block_of(token(t0 + 2 * NW * CHUNK))];
    }
    __builtin_amdgcn_wave_barrier();
    f32x4 st[2];
    #pragma unroll
    for (int s = 0; s < 2; ++s) {
      st[s] = f32x4{0.f, 0.f, 0.f, 0.f};
      #pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        st[s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            *reinterpret_cast<const bf16v8*>(ktile + v_off<D>(s * 16 + lr, ks * 4 + g)), qf[ks],
            st[s], 0, 0, 0);
    }

    // this lane: head lr, tokens t0 + 16 s + 4 g + r
    float mx = -1e30f;
    #pragma unroll
    for (int s = 0; s < 2; ++s)
      #pragma unroll
      for (int r = 0; r < 4; ++r) {
        st[s][r] = t0 + s * 16 + g * 4 + r < c1 ? st[s][r] * scale_log2 : -1e30f;
        mx = fmaxf(mx, st[s][r]);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, WAVE));
    mx = fmaxf(mx, __shfl_xor(mx, 32, WAVE));
    // The subtracted maximum may lag by 2^8: rescaling the sums at every chunk
    // would cost as much as weighing V. The weights' two terms carry 17 bits
    // whatever their size, so nothing is lost by it.
    if (__any(mx > m + 8.f)) {
      const float m_new = fmaxf(m, mx), alpha = __builtin_amdgcn_exp2f(m - m_new);
      lsum *= alpha;
      #pragma unroll
      for (int dt = 0; dt < DT; ++dt)
        #pragma unroll
        for (int r = 0; r < 4; ++r) acc[dt][r] *= alpha;
      m = m_new;
    }
    bf16v8 hi, lo;
    #pragma unroll
    for (int s = 0; s < 2; ++s)
      #pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float p = __builtin_amdgcn_exp2f(st[s][r] - m);
        lsum += p;
        hi[s * 4 + r] = (__bf16)p;
        lo[s * 4 + r] = (__bf16)(p - (float)hi[s * 4 + r]);
      }
    __builtin_amdgcn_wave_barrier();
    #pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      // V^T: rows d = 16 dt + lr, k-slots = tokens 4g.. and 16 + 4g..
      const int c = dt * 2 + ((l & 3) >> 1), r0 = 4 * g + (lr >> 2), e = (l & 1) * 8;
      const bf16v4 a = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16v4*)(tile + v_off<D>(r0, c) + e));
      const bf16v4 b = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16v4*)(tile + v_off<D>(r0 + 16, c) + e));
      const bf16v8 vt = __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
      acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vt, hi, acc[dt], 0, 0, 0);
      acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vt, lo, acc[dt], 0, 0, 0);
    }
    __builtin_amdgcn_wave_barrier();
  }

  // join the waves: m, l per head, then the weighted sums
  lsum += __shfl_xor(lsum, 16, WAVE);
  lsum += __shfl_xor(lsum, 32, WAVE);
  if (g == 0) {
    ml_lds[(wave * 16 + lr) * 2] = m;
    ml_lds[(wave * 16 + lr) * 2 + 1] = lsum;
  }
  float* o_tile = reinterpret_cast<float*>(ktile);      // [16 heads][D]
  #pragma unroll
  for (int dt = 0; dt < DT; ++dt)
    *reinterpret_cast<f32x4*>(o_tile + lr * D + dt * 16 + g * 4) = acc[dt];
  __syncthreads();
  const bool whole = len <= slice_len || gridDim.z == 1;  // nothing to join outside
  for (int i = threadIdx.x; i < group * (D / 4); i += NW * 64) {
    const int h = i / (D / 4), d = i % (D / 4) * 4;
    float top = -1e30f, total = 0.f;
    #pragma unroll
    for (int w = 0; w < NW; ++w) top = fmaxf(top, ml_lds[(w * 16 + h) * 2]);
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
    #pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float f = __builtin_amdgcn_exp2f(ml_lds[(w * 16 + h) * 2] - top);
      total += f * ml_lds[(w * 16 + h) * 2 + 1];
      const f32x4 x = *reinterpret_cast<const f32x4*>(smem + w * (2 * CHUNK * D * 2) + (h * D + d) * 4);
      #pragma unroll
      for (int r = 0; r < 4; ++r) o[r] += f * x[r];
    }
    const int64_t head = (int64_t)seq * H + kv * group + h;
    if (whole) {
      const float inv = total > 0.f ? 1.f / total : 0.f;
      bf16v4 y;
      #pragma unroll
      for (int r = 0; r < 4; ++r) y[r] = (__bf16)(o[r] * inv);
      *reinterpret_cast<bf16v4*>(out + head * D + d) = y;
    } else {
      const int64_t at = (int64_t)z * N * H + head;
      #pragma unroll
      for (int r = 0; r < 4; r += 2) store_pair(o_part + at * D + d + r, o[r], o[r + 1]);
      if (d == 0) store_pair(ml_part + at * 2, top, total);
    }
  }
  {
    if (whole) return;
    // the last slice of the sequence and kv head to end joins them
    __shared__ int last;
    stores_done();
    __syncthreads();
    const int n = min((len + slice_len - 1) / slice_len, (int)gridDim.z);
    if constexpr (SRC == QUERIES) {
      if (wave == 0) {
        const bool all = all_there(there + ((int64_t)seq * KV + kv) * gridDim.z, n, z, tag);
        if (l == 0) last = all;
      }
    } else {
      if (threadIdx.x == 0) last = atomicAdd(src.arrived + seq * KV + kv, 1) == n - 1;
    }
    __syncthreads();
    if (!last) return;
    if (SRC != QUERIES && threadIdx.x == 0) src.arrived[seq * KV + kv] = 0;
    for (int i = threadIdx.x; i < group * (D / 4); i += NW * 64) {
      const int h = i / (D / 4), d = i % (D / 4) * 4;
      const int64_t head = (int64_t)seq * H + kv * group + h, step = (int64_t)N * H;
      // with the maximum of those before: one look at each
      float top = -1e30f, total = 0.f;
      f32x4 o = {0.f, 0.f, 0.f, 0.f};
      for (int s0 = 0; s0 < n; s0 += 4) {
        float2 ml[4], lo[4], hi[4];
        #pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int64_t at = min(s0 + s, n - 1) * step + head;
          ml[s] = load_pair(ml_part + at * 2);
          lo[s] = load_pair(o_part + at * D + d);
          hi[s] = load_pair(o_part + at * D + d + 2);
        }
        float high = top;
        #pragma unroll
        for (int s = 0; s < 4; ++s) high = fmaxf(high, ml[s].x);
        const float old = __builtin_amdgcn_exp2f(top - high);
        total *= old;
        o *= old;
        top = high;
        #pragma unroll
        for (int s = 0; s < 4; ++s)
          if (s0 + s < n) {
            const float f = __builtin_amdgcn_exp2f(ml[s].x - top);
            total += f * ml[s].y;
            o += f32x4{lo[s].x, lo[s].y, hi[s].x, hi[s].y} * f;
          }
      }
      const float inv = total > 0.f ? 1.f / total : 0.f;
      bf16v4 y;
      #pragma unroll
      for (int r = 0; r < 4; ++r) y[r] = (__bf16)(o[r] * inv);
      *reinterpret_cast<bf16v4*>(out + head * D + d) = y;
    }
  }
}

template <int D, int NW, int SRC>
void launch_decode(const __hip_bfloat16* q, const torch::Tensor& kcache,
                   const torch::Tensor& vcache, const torch::Tensor& bt,
                   const torch::Tensor& ctx, torch::Tensor& out, int N, int H, int KV,
                   float scale, int64_t q_row_stride, int cs, int slice_len, const Packed& src) {
  const int block_size = kcache.size(1);
  const int shift = (block_size & (block_size - 1)) == 0 ? __builtin_ctz(block_size) : -1;
  auto stream = at::cuda::getCurrentCUDAStream();
  torch::Tensor part;
  float *o_p = nullptr, *ml_p = nullptr;
  unsigned long long* there = nullptr;
  if (cs > 1) {
    const int64_t heads = (int64_t)cs * N * H;
    part = torch::empty({heads * (D + 2) + 2ll * N * KV * cs}, out.options().dtype(at::kFloat));
    o_p = part.data_ptr<float>();
    ml_p = o_p + heads * D;
    there = reinterpret_cast<unsigned long long*>(ml_p + heads * 2);   // of QUERIES alone
  }
  auto* o = reinterpret_cast<__hip_bfloat16*>(out.data_ptr());
  const int smem = NW * (2 * CHUNK * D * 2 + 16 * 2 * 4) + (SRC == QUERIES ? 0 : (H / KV + 2) * D * 2);
  hipLaunchKernelGGL((paged_decode_kernel<D, NW, SRC>), dim3(N, KV, cs), dim3(NW * 64), smem,
                     stream, q, reinterpret_cast<const __hip_bfloat16*>(kcache.data_ptr()),
                     reinterpret_cast<const __hip_bfloat16*>(vcache.data_ptr()),
                     bt.data_ptr<int>(), ctx.data_ptr<int>(), o, o_p, ml_p, H, KV,
                     (int)bt.size(1), block_size, shift, scale * LOG2E, q_row_stride, slice_len,
                     there, cs > 1 ? arrival_tag() : 0, src);
}

// Slices of the context (known here: a table's width, not its sequence's
// length). A round of loads takes ~4 us from cold pages, joining as long: few
// sequences run with eight waves in slices of 512 tokens, up to one workgroup a
// CU (3 sequences of 911..3777, 2 kv heads: 1 slice 18 us, 2: 13.5, 4: 11.1, 8:
// 11.5; 16 of 1500, 4 kv heads: 18.4, 18.2, 4: 16.8, 6: 21; 8 of 4000, 8 kv heads:
// 37, 30, 29, 8: 35). From 129 workgroups on one slice is left of that, a fifth
// too slow at most (33 of 4000, 4 kv heads: 50, 2: 61, 3: 50, 4: 57). More
// sequences fill the chip by themselves (the round above: 60.2 us, 2: 59.8, 4:
// 62; 10 x 16 of 180..380: 21, 2: 27; 63 of 4000: 100, 2: 101).
int slices(int64_t blocks, int max_ctx) {
  int cs = blocks < 256 ? (int)std::max<int64_t>(1, std::min<int64_t>(256 / blocks, CDIV(max_ctx, 512)))
                        : 1;
  if (const char* e = getenv("DISTRL_PAGED_CS")) {
    cs = std::max(1, std::min(atoi(e), 16));
    while (cs > 1 && (max_ctx + cs - 1) / cs < 32) cs /= 2;
  }
  return cs;
}

// out (N, H, D) by the kernel for its sizes
template <int SRC>
void decode(const __hip_bfloat16* q, const torch::Tensor& kcache, const torch::Tensor& vcache,
            const torch::Tensor& bt, const torch::Tensor& ctx, torch::Tensor& out, int N, int H,
            int KV, int D, double scale, int64_t q_row_stride, const Packed& src) {
  const int group = H / KV, max_ctx = bt.size(1) * kcache.size(1);
  TORCH_CHECK(H % KV == 0 && group <= 16, "GQA group too large");
  if (N == 0) return;
  TORCH_CHECK((D == 128 && (group <= 2 || (group >= 4 && group <= 8))) ||
              (D == 64 && (group == 1 || group == 2 || group == 4 || group == 7)),
              "paged decode: unsupported (head_dim=", D, ", gqa group=", group, ")");
  const int64_t blocks = (int64_t)N * KV;
  const bool few = blocks < 256;
  const int cs = slices(blocks, max_ctx), slice_len = std::max(1, CDIV(max_ctx, cs));
  #define DECODE(DD, NN) launch_decode<DD, NN, SRC>(q, kcache, vcache, bt, ctx, out, N, H, KV, \
                                                    (float)scale, q_row_stride, cs, slice_len, src)
  // From 513 workgroups on those of four waves with rows of 128 no longer run at
  // once (two a CU by their LDS), those of two do: the round above 70.6 -> 67.7 us,
  // 10 x 16 of 180..380 20.5 -> 18.1 (from partial sums 29.1 -> 21.8), 16 x 16
  // 26.6 -> 24.0; 256 workgroups of
  // 500..1500 would take 49.4 for 35.5, and rows of 64 fit three or four a CU anyway
  // (two waves there: 160 of 300..1500, 32/8 heads from partial sums 73 for 62).
  if (D == 128) { if (few) DECODE(128, 8); else if (blocks > 512) DECODE(128, 2); else DECODE(128, 4); }
  else { if (few) DECODE(64, 8); else DECODE(64, 4); }
  #undef DECODE
  HIP_CHECK_LAST();
}

}  // namespace

torch::Tensor paged_attention_decode_strided(
    torch::Tensor q, int64_t n_heads, int64_t head_dim, int64_t q_row_stride,
    torch::Tensor kcache, torch::Tensor vcache, torch::Tensor block_tables,
    torch::Tensor ctx_lens, double scale) {
  // q: (N, q_row_stride) packed rows (e.g. the fused qkv GEMM output);
  // query heads occupy the first n_heads*head_dim elements of each row.
  TORCH_CHECK(q.is_cuda() && q.is_contiguous());
  TORCH_CHECK(q.scalar_type() == at::kBFloat16);
  TORCH_CHECK(block_tables.scalar_type() == at::kInt &&
              ctx_lens.scalar_type() == at::kInt);
  const int N = q.size(0), H = (int)n_heads, D = (int)head_dim;
  if (q_row_stride % 8 != 0 || reinterpret_cast<uintptr_t>(q.data_ptr()) % 16 != 0) {
    // rows that 16 B loads cannot read
    q = q.view({N, q_row_stride}).slice(1, 0, (int64_t)H * D).clone(at::MemoryFormat::Contiguous);
    q_row_stride = (int64_t)H * D;
  }
  auto out = torch::empty({N, (int64_t)H, (int64_t)D}, q.options());
  decode<QUERIES>(reinterpret_cast<const __hip_bfloat16*>(q.data_ptr()), kcache, vcache,
                  block_tables, ctx_lens, out, N, H, kcache.size(2), D, scale, q_row_stride, {});
  return out;
}

// One decode step's attention from the packed projections [q | k | v] of its N
// tokens, (N, (H + 2 KV) D) bf16 or (splits, N, ...) fp32 partial sums without
// their bias: head norms (if given), rotation, the new keys and values into the
// cache, attention over it. Returns (N, H D). arrived: int32, N KV zeros at least,
// which it leaves zero; calls that may overlap need one each.
torch::Tensor paged_decode_packed(torch::Tensor qkv, c10::optional<torch::Tensor> bias,
                                  torch::Tensor positions, torch::Tensor slots,
                                  torch::Tensor inv_freq, torch::Tensor kcache,
                                  torch::Tensor vcache, torch::Tensor block_tables,
                                  torch::Tensor ctx_lens, torch::Tensor arrived, int64_t n_heads,
                                  double scale, c10::optional<torch::Tensor> q_norm,
                                  c10::optional<torch::Tensor> k_norm, double eps) {
  const bool parts = qkv.dim() == 3;
  TORCH_CHECK(qkv.is_cuda() && qkv.is_contiguous() && (parts || qkv.dim() == 2) &&
              qkv.scalar_type() == (parts ? at::kFloat : at::kBFloat16));
  const int N = qkv.size(-2), H = (int)n_heads, KV = kcache.size(2), D = kcache.size(3);
  TORCH_CHECK(qkv.size(-1) == (int64_t)(H + 2 * KV) * D && (parts || !bias));
  TORCH_CHECK(vcache.sizes() == kcache.sizes() && kcache.scalar_type() == at::kBFloat16 &&
              vcache.scalar_type() == at::kBFloat16);
  // the kernel walks all of them as they lie on the GPU
  for (const auto* t : {&kcache, &vcache, &positions, &slots, &inv_freq, &block_tables, &ctx_lens})
    TORCH_CHECK(t->is_cuda() && t->is_contiguous(), "paged_decode_packed: device or layout");
  TORCH_CHECK(positions.scalar_type() == at::kInt && slots.scalar_type() == at::kLong &&
              positions.numel() == N && slots.numel() == N && inv_freq.numel() == D / 2 &&
              inv_freq.scalar_type() == at::kFloat);
  TORCH_CHECK(block_tables.scalar_type() == at::kInt && block_tables.dim() == 2 &&
              block_tables.size(0) == N && ctx_lens.scalar_type() == at::kInt &&
              ctx_lens.numel() == N);
  TORCH_CHECK(arrived.is_cuda() && arrived.scalar_type() == at::kInt && arrived.is_contiguous() &&
              arrived.numel() >= (int64_t)N * KV);
  auto vec = [&](const c10::optional<torch::Tensor>& w, int64_t n) {
    if (!w) return (const __hip_bfloat16*)nullptr;
    TORCH_CHECK(w->is_cuda() && w->is_contiguous() && w->scalar_type() == at::kBFloat16 &&
                w->numel() == n, "paged_decode_packed: norm weight or bias");
    return reinterpret_cast<const __hip_bfloat16*>(w->data_ptr());
  };
  Packed src{};
  src.bias = vec(bias, qkv.size(-1));
  src.q_norm = vec(q_norm, D);
  src.k_norm = vec(k_norm, D);
  for (const void* p : {(const void*)qkv.data_ptr(), (const void*)src.bias})
    TORCH_CHECK(reinterpret_cast<uintptr_t>(p) % 16 == 0, "paged_decode_packed: alignment");
  src.positions = positions.data_ptr<int>();
  src.slots = slots.data_ptr<int64_t>();
  src.inv_freq = inv_freq.data_ptr<float>();
  src.eps = (float)eps;
  src.kcache = reinterpret_cast<__hip_bfloat16*>(kcache.data_ptr());
  src.vcache = reinterpret_cast<__hip_bfloat16*>(vcache.data_ptr());
  src.arrived = arrived.data_ptr<int>();
  auto out = torch::empty({N, (int64_t)H * D}, qkv.options().dtype(at::kBFloat16));
  if (parts) {
    src.parts = qkv.data_ptr<float>();
    src.splits = qkv.size(0);
    decode<PARTS>(nullptr, kcache, vcache, block_tables, ctx_lens, out, N, H, KV, D, scale, 0, src);
  } else {
    src.rows = reinterpret_cast<const __hip_bfloat16*>(qkv.data_ptr());
    decode<ROWS>(nullptr, kcache, vcache, block_tables, ctx_lens, out, N, H, KV, D, scale, 0, src);
  }
  return out;
}


torch::Tensor paged_attention_decode(torch::Tensor q, torch::Tensor kcache,
                                     torch::Tensor vcache,
                                     torch::Tensor block_tables,
                                     torch::Tensor ctx_lens, double scale) {
  TORCH_CHECK(q.dim() == 3);
  return paged_attention_decode_strided(
      q.view({q.size(0), q.size(1) * q.size(2)}), q.size(1), q.size(2),
      q.size(1) * q.size(2), kcache, vcache, block_tables, ctx_lens, scale);
}

// ---- varlen causal prefill attention (prompt phase) ----
// One workgroup per (q-row-tile of 16, q-head): same three-phase structure
// as the decode kernel with the GQA group slot re-used for the 16 q rows
// of the tile — lane-per-kv-token scoring against the LDS-staged q tile
// (with causal masking), per-row softmax, PV through LDS V tiles.
// K/V are the flat pre-RoPE'd prefill tensors (no paging needed here).
// Replaces the torch-SDPA library call in the engine.
namespace {

// the legacy prefill kernel keeps the original 32-token V tile: the
// decode kernel's VTILE=64 retune doubled this kernel's LDS and cost it
// ~10x in occupancy (one reason the MFMA flash kernel is now the
// prefill default)
constexpr int PF_VTILE = 32;

template <int D>
__global__ __launch_bounds__(256)
void prefill_attn_kernel(const __hip_bfloat16* __restrict__ q,   // (T,H,D)
                         const __hip_bfloat16* __restrict__ k,   // (T,KV,D)
                         const __hip_bfloat16* __restrict__ v,   // (T,KV,D)
                         const int* __restrict__ tile_q0,    // global q row
                         const int* __restrict__ tile_rows,  // rows in tile
                         const int* __restrict__ tile_kv0,   // prompt start
                         __hip_bfloat16* __restrict__ out,       // (T,H,D)
                         int H, int KV, int Lpad, float scale) {
  constexpr int QT = 16;
  const int tile = blockIdx.x;
  const int h = blockIdx.y;
  const int kvh = h / (H / KV);
  const int q0 = tile_q0[tile];
  const int rows = tile_rows[tile];
  const int kv0 = tile_kv0[tile];
  // causal: tile rows attend to kv positions [kv0, q0 + rows)
  const int Lmax = q0 - kv0 + rows;
  const int tid = threadIdx.x;

  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  float* q_lds = reinterpret_cast<float*>(smem_raw);          // QT*D
  float* denom = q_lds + QT * D;                              // QT
  float* scores = denom + QT;                                 // QT*Lpad
  __hip_bfloat16* v_lds = reinterpret_cast<__hip_bfloat16*>(
      scores + (size_t)QT * Lpad);                            // PF_VTILE*D

  for (int i = tid; i < QT * D; i += blockDim.x) {
    const int r = i / D;
    q_lds[i] = (r < rows)
        ? bf2f(q[((int64_t)(q0 + r) * H + h) * D + i % D]) * scale
        : 0.f;
  }
  __syncthreads();

  // phase 1: lane-per-kv-token scoring with causal mask
  for (int t = tid; t < Lmax; t += blockDim.x) {
    const __hip_bfloat16* kp = k + ((int64_t)(kv0 + t) * KV + kvh) * D;
    float part[QT];
    #pragma unroll
    for (int r = 0; r < QT; ++r) part[r] = 0.f;
    #pragma unroll
    for (int c = 0; c < D / 8; ++c) {
      const bf16x8 kvec = *reinterpret_cast<const bf16x8*>(kp + c * 8);
      float kf[8];
      #pragma unroll
      for (int j = 0; j < 8; ++j) kf[j] = bf2f(kvec.v[j]);
      #pragma unroll
      for (int r = 0; r < QT; ++r) {
        const float* qr = q_lds + r * D + c * 8;
        #pragma unroll
        for (int j = 0; j < 8; ++j) part[r] += qr[j] * kf[j];
      }
    }
    #pragma unroll
    for (int r = 0; r < QT; ++r) {
      // causal: kv position kv0+t visible to q row q0+r iff kv0+t <= q0+r
      const bool vis = (kv0 + t) <= (q0 + r);
      scores[(size_t)r * Lpad + t] = vis ? part[r] : -1e30f;
    }
  }
  __syncthreads();

  // phase 2: per-row softmax
  const int wid = tid / WAVE;
  const int wlane = tid % WAVE;
  const int nw = blockDim.x / WAVE;
  for (int r = wid; r < QT; r += nw) {
    float* s = scores + (size_t)r * Lpad;
    float m = -1e30f;
    for (int t = wlane; t < Lmax; t += WAVE) m = fmaxf(m, s[t]);
    m = wave_max(m);
    float d = 0.f;
    for (int t = wlane; t < Lmax; t += WAVE) {
      float e = __expf(s[t] - m);
      s[t] = e;
      d += e;
    }
    d = wave_sum(d);
    if (wlane == 0) denom[r] = d;
  }
  __syncthreads();

  // phase 3: PV through LDS V tiles
  constexpr int DV = D / 8;
  constexpr int UNITS = QT * DV;  // 128 (D=64) or 256 (D=128)
  float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  const int u = tid;
  const int ur = u / DV, ud = u % DV;
  for (int base = 0; base < Lmax; base += PF_VTILE) {
    const int tl = min(PF_VTILE, Lmax - base);
    for (int i = tid; i < tl * DV; i += blockDim.x) {
      reinterpret_cast<bf16x8*>(v_lds)[i] =
          *reinterpret_cast<const bf16x8*>(
              v + ((int64_t)(kv0 + base + i / DV) * KV + kvh) * D
              + (i % DV) * 8);
    }
    __syncthreads();
    if (u < UNITS) {
      const float* ps = scores + (size_t)ur * Lpad + base;
      #pragma unroll 4
      for (int j = 0; j < tl; ++j) {
        const float p = ps[j];
        const bf16x8 vv = reinterpret_cast<const bf16x8*>(v_lds)[j * DV + ud];
        #pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] += p * bf2f(vv.v[e]);
      }
    }
    __syncthreads();
  }

  if (u < UNITS && ur < rows) {
    const float inv = 1.f / denom[ur];
    bf16x8 o;
    #pragma unroll
    for (int e = 0; e < 8; ++e) o.v[e] = f2bf(acc[e] * inv);
    *reinterpret_cast<bf16x8*>(
        out + ((int64_t)(q0 + ur) * H + h) * D + ud * 8) = o;
  }
}

}  // namespace

torch::Tensor prefill_attention(torch::Tensor q, torch::Tensor k,
                                torch::Tensor v, torch::Tensor tile_q0,
                                torch::Tensor tile_rows, torch::Tensor tile_kv0,
                                int64_t max_len, double scale) {
  TORCH_CHECK(q.is_cuda() && q.is_contiguous() && k.is_contiguous()
              && v.is_contiguous());
  TORCH_CHECK(q.scalar_type() == at::kBFloat16);
  TORCH_CHECK(tile_q0.scalar_type() == at::kInt);
  const int H = q.size(1), D = q.size(2), KV = k.size(1);
  const int n_tiles = tile_q0.size(0);
  auto out = torch::empty_like(q);
  if (n_tiles == 0) return out;
  const int Lpad = (int)max_len + 4;
  size_t smem = 16 * D * 4 + 16 * 4 + (size_t)16 * Lpad * 4
                + (size_t)PF_VTILE * D * 2;
  TORCH_CHECK(smem <= 160 * 1024, "prompt too long for prefill kernel: ",
              max_len);
  dim3 grid(n_tiles, H), block(256);
  auto stream = at::cuda::getCurrentCUDAStream();
  if (D == 128) {
    hipLaunchKernelGGL(prefill_attn_kernel<128>, grid, block, smem, stream,
        reinterpret_cast<const __hip_bfloat16*>(q.data_ptr()),
        reinterpret_cast<const __hip_bfloat16*>(k.data_ptr()),
        reinterpret_cast<const __hip_bfloat16*>(v.data_ptr()),
        tile_q0.data_ptr<int>(), tile_rows.data_ptr<int>(),
        tile_kv0.data_ptr<int>(),
        reinterpret_cast<__hip_bfloat16*>(out.data_ptr()),
        H, KV, Lpad, (float)scale);
  } else if (D == 64) {
    hipLaunchKernelGGL(prefill_attn_kernel<64>, grid, block, smem, stream,
        reinterpret_cast<const __hip_bfloat16*>(q.data_ptr()),
        reinterpret_cast<const __hip_bfloat16*>(k.data_ptr()),
        reinterpret_cast<const __hip_bfloat16*>(v.data_ptr()),
        tile_q0.data_ptr<int>(), tile_rows.data_ptr<int>(),
        tile_kv0.data_ptr<int>(),
        reinterpret_cast<__hip_bfloat16*>(out.data_ptr()),
        H, KV, Lpad, (float)scale);
  } else {
    TORCH_CHECK(false, "prefill attention: head_dim 64 or 128 only");
  }
  HIP_CHECK_LAST();
  return out;
}
