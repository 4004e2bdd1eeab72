// Causal GQA flash attention, forward and backward, for the learner's
// teacher-forced pass and the engine's prompt phase (reference
// distributed_actor.py:241-243 forward + loss.backward()).
//
// Layout. q, o, dout, dq are (B, Hq, T, D) and k, v, dk, dv (B, Hkv, T, D)
// with any strides whose innermost one is 1: the model's (B, T, H, D)
// projections go in and come out without a copy. The prompt phase passes
// one flat (tokens, H, D) batch with row offsets instead of padded rows.
//
// Products run on MFMA 32x32x16. A wave owns 32 rows (queries in the
// forward and the dQ pass, keys in the dK/dV pass) whose operands stay in
// registers; the other side streams through LDS in double-buffered tiles,
// fetched into registers one tile ahead. Scores are formed transposed,
// ST[key][query] = K Q^T (dK/dV: S[query][key] = Q K^T), so that
//  * a lane holds 16 scores of ONE query of each 32x32 block: the softmax
//    reduces in registers and over one lane swap, and rescaling the output
//    is a lane-local multiply;
//  * the accumulator's rows {4h..4h+3, 8+4h..8+4h+3} (h = lane / 32) of a
//    16-row step serve directly as the next product's k-slots: packing to
//    bf16 is the only conversion. The other operand is read with the same
//    k order, by LDS transpose reads from the row-major tile, so nothing is
//    ever transposed in memory.
// Bound: LDS reads (1 KB per MFMA and wave, 128 B/clk) run level with the
// matrix cores here; two workgroups a CU let one's softmax overlap the
// other's products.
//
// A tile row is XOR-swizzled in 16 B chunks by swz(row): 8 consecutive rows
// read at one chunk (row fragments) and 4 rows read over 64 B (transpose
// reads) both fall into different banks.
//
// The backward has two passes and no atomics: results do not depend on the
// order of workgroups. dQ (query rows) also forms delta = rowsum(dO * O);
// dK/dV (key rows) walks the query heads of its kv head and adds them up in
// fp32 registers; where key blocks alone leave the chip idle, the heads are
// split over workgroups that leave fp32 partials for a small sum kernel.
//
// Measured at B 16, 28/4 heads, T 1550, D 128 (275 GFLOP in the causal half,
// forward): forward 390 us = 705 TFLOP/s, backward 1177 us. It was 440 and 1845 with
// waits for the next tile's loads inside the dK/dV step (a row statistic used
// behind a branch, fragments spilled or not waited for before the loop, 64-bit
// addresses in registers) and pairs of heads one after the other; 16-row waves on
// 16x16x32 with single-buffered tiles and transposed copies of q, k, v, dout took
// 1161 and 5563 us + 1.9 ms of copies and sums. What bounds them now: LDS reads and
// vector work beside the products at two waves a SIMD.
#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>
#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16v8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16v4;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16v2;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((address_space(3))) bf16v4 lds_bf16v4;

namespace {

constexpr float LOG2E = 1.4426950408889634f;
constexpr float LN2 = 0.6931471805599453f;
constexpr int WROWS = 32;   // rows a wave owns

// Keys of a tile: two waves share the fetch of a smaller one, or their
// prefetch registers would spill.
template <int NW>
constexpr int tile_rows() { return NW == 4 ? 64 : 32; }

// element strides of a (B, H, T, D) operand
struct Strides { int64_t b, h; int t; };

// The sequences of a batch: T rows each, or rows cu[b] .. cu[b + 1] of a flat
// one. A (batch, heads, rows) array of numbers lies b * heads * T apart, or as
// (heads, rows of the flat batch).
struct Seqs {
  const int* cu;
  int T;            // rows of each, or of the longest
  int64_t b, h;     // of a query head's numbers
  DEV_INLINE int first(int i) const { return cu ? cu[i] : 0; }
  DEV_INLINE int len(int i) const { return cu ? cu[i + 1] - cu[i] : T; }
};

DEV_INLINE f32x16 mfma(bf16v8 a, bf16v8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

DEV_INLINE f32x16 zero16() {
  f32x16 z;
  #pragma unroll
  for (int i = 0; i < 16; ++i) z[i] = 0.f;
  return z;
}

// maximum and sum over the two half-waves
DEV_INLINE float halves_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
DEV_INLINE float halves_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// the wave's number as a scalar, so that branches on its rows are scalar too
DEV_INLINE int wave_id() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

template <int D>
DEV_INLINE int swz(int row) {
  return D == 128 ? ((row & 3) << 2) | ((row >> 2) & 3)
                  : (((row >> 1) & 1) << 2) | ((row >> 2) & 3);
}

// One ROWS x D tile: fetched into registers, then stored to LDS.
template <int D, int ROWS, int NT>
struct Tile {
  static constexpr int UN = D / 8, STEP = NT / UN;     // rows NT threads cover
  static constexpr int PER = ROWS / STEP;
  static_assert(NT % UN == 0 && ROWS % STEP == 0, "tile does not divide");
  u32x4 r[PER];

  // base is wave-uniform: a full tile's loads share one lane offset. Rows past
  // the end repeat the last one, their weights are zero. (A branch around
  // each load would make the loads wait for one another.)
  DEV_INLINE void fetch(const __hip_bfloat16* base, int stride_t, int valid) {
    const int row = threadIdx.x / UN, cu = threadIdx.x % UN;
    if (valid >= ROWS) {
      const int off = row * stride_t + cu * 8;
      #pragma unroll
      for (int i = 0; i < PER; ++i)
        r[i] = *reinterpret_cast<const u32x4*>(base + (int64_t)(i * STEP) * stride_t + off);
    } else {
      #pragma unroll
      for (int i = 0; i < PER; ++i)
        r[i] = *reinterpret_cast<const u32x4*>(base + min(i * STEP + row, valid - 1) * stride_t
                                               + cu * 8);
    }
  }
  DEV_INLINE void store(char* lds) const {
    #pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int row = i * STEP + threadIdx.x / UN, cu = threadIdx.x % UN;
      *reinterpret_cast<u32x4*>(lds + row * (2 * D) + ((cu ^ swz<D>(row)) << 4)) = r[i];
    }
  }
};

// A tile whose loads take one 32-bit offset a lane: rows past the end read as zero.
template <int D, int ROWS, int NT>
struct Rows : Tile<D, ROWS, NT> {
  using T = Tile<D, ROWS, NT>;
  int off;          // bytes, of this lane's first 16

  DEV_INLINE explicit Rows(int stride_t)
      : off(((int)threadIdx.x / T::UN * stride_t + (int)threadIdx.x % T::UN * 8) * 2) {}

  DEV_INLINE void fetch(const __hip_bfloat16* base, int stride_t, int valid) {
    // stride_t < 2^24: 64 rows stay within 2^31 bytes
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<__hip_bfloat16*>(base), 0, ((min(valid, ROWS) - 1) * stride_t + D) * 2, 0x00027000);
    #pragma unroll
    for (int i = 0; i < T::PER; ++i)
      this->r[i] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, off + i * T::STEP * stride_t * 2, 0, 0);
  }
};

// Lane offsets of the two kinds of fragment of a tile.
template <int D>
struct Frags {
  int row_off;         // row fragment: row l&31, chunk h
  int tr_lo, tr_hi;    // transpose reads: rows 4h + (l&15)/4 and 8 further

  DEV_INLINE Frags() {
    const int l = threadIdx.x & 63, h = l >> 5;
    const int row = l & 31;
    row_off = row * (2 * D) + ((h ^ swz<D>(row)) << 4);
    const int x = ((l >> 4) & 1) * 2 + ((l & 3) >> 1);
    const int r0 = 4 * h + ((l & 15) >> 2), r1 = r0 + 8;
    tr_lo = r0 * (2 * D) + ((x ^ swz<D>(r0)) << 4) + (l & 1) * 8;
    tr_hi = r1 * (2 * D) + ((x ^ swz<D>(r1)) << 4) + (l & 1) * 8;
  }
  // rows sub*32 + (l&31), elements ks*16 + h*8 ..
  DEV_INLINE bf16v8 row(const char* lds, int sub, int ks) const {
    return *reinterpret_cast<const bf16v8*>(lds + sub * (32 * 2 * D) + (row_off ^ (ks << 5)));
  }
  // element column dt*32 + (l&31), rows k0 + {4h.., 8+4h..}; k0 % 16 == 0
  DEV_INLINE bf16v8 col(char* lds, int k0, int dt) const {
    char* p = lds + k0 * (2 * D);
    const bf16v4 a = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
        (lds_bf16v4*)(p + (tr_lo ^ (dt << 6))));
    const bf16v4 b = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
        (lds_bf16v4*)(p + (tr_hi ^ (dt << 6))));
    return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
  }
};

// two floats rounded to nearest even (v_cvt_pk_bf16_f32)
DEV_INLINE bf16v2 round2(float a, float b) {
  return __builtin_convertvector(f32x2{a, b}, bf16v2);
}

// accumulator rows 8*k .. 8*k+7 of this lane as bf16 k-slots of a 16-row step
DEV_INLINE bf16v8 pack8(const f32x16& s, int k) {
  bf16v8 out;
  #pragma unroll
  for (int j = 0; j < 4; ++j) {
    const bf16v2 v = round2(s[8 * k + 2 * j], s[8 * k + 2 * j + 1]);
    out[2 * j] = v[0];
    out[2 * j + 1] = v[1];
  }
  return out;
}

// row index within a 32-row block of accumulator register r
DEV_INLINE int acc_row(int r, int h) { return 8 * (r >> 2) + 4 * h + (r & 3); }

// this lane's row of a (rows, D) operand as fragments
template <int D>
DEV_INLINE void load_row(bf16v8 (&f)[D / 16], const __hip_bfloat16* base, int stride_t, int row) {
  const int h = (threadIdx.x & 63) >> 5;
  #pragma unroll
  for (int ks = 0; ks < D / 16; ++ks)
    f[ks] = *reinterpret_cast<const bf16v8*>(base + (int64_t)row * stride_t + ks * 16 + h * 8);
}

// Waits for fragments here: left to their first use, in a loop, the wait would be
// for the loop's own loads as well, in every step.
template <int D>
DEV_INLINE void arrived(bf16v8 (&f)[D / 16]) {
  #pragma unroll
  for (int ks = 0; ks < D / 16; ++ks) {
    u32x4 x = __builtin_bit_cast(u32x4, f[ks]);
    asm volatile("" : "+v"(x));
    f[ks] = __builtin_bit_cast(bf16v8, x);
  }
}

// acc[dt] holds X^T (rows d, column = this lane's row): write the row times f.
// Two half-waves hold alternating groups of four d; one swap makes 16 B runs.
template <int D>
DEV_INLINE void store_rows(const f32x16 (&acc)[D / 32], float f, __hip_bfloat16* row, bool valid) {
  const int h = (threadIdx.x & 63) >> 5;
  #pragma unroll
  for (int dt = 0; dt < D / 32; ++dt) {
    #pragma unroll
    for (int g = 0; g < 2; ++g) {       // d 16g .. 16g+15 of the 32
      uint32_t w[4];
      #pragma unroll
      for (int j = 0; j < 4; ++j) {
        w[j] = __builtin_bit_cast(
            uint32_t, round2(acc[dt][8 * g + 2 * j] * f, acc[dt][8 * g + 2 * j + 1] * f));
      }
      const auto x = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
      const auto y = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
      if (valid)
        *reinterpret_cast<u32x4*>(row + dt * 32 + g * 16 + h * 8) = u32x4{x[0], y[0], x[1], y[1]};
    }
  }
}

// The same rows in fp32 (partial sums of a head split).
template <int D>
DEV_INLINE void store_rows_f32(const f32x16 (&acc)[D / 32], float* row, bool valid) {
  const int h = (threadIdx.x & 63) >> 5;
  if (!valid) return;
  #pragma unroll
  for (int dt = 0; dt < D / 32; ++dt)
    #pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<f32x4*>(row + dt * 32 + g * 8 + h * 4) =
          f32x4{acc[dt][4 * g], acc[dt][4 * g + 1], acc[dt][4 * g + 2], acc[dt][4 * g + 3]};
}

// What workgroup id works on: a kv head of a sequence (pair), a block of its rows
// (longest first) and a query head or share of them.
struct Place { int pair, block, part; };

// Longest blocks first over all pairs, so that short ones fill the end. Workgroups
// go to the 8 XCDs in turn; where they divide, each XCD gets pairs of its own, whose
// heads and row blocks meet in one L2. (Pair by pair, every pair's longest block
// first, the last pair's ended late: backward at (16, 28/4, 1550, 128) 1339 us for
// 1230, (8, 64/8, 1024, 128) 733 for 636.)
DEV_INLINE Place place(int id, int pairs, int blocks, int parts) {
  int x = 0, n = pairs * parts;
  if (pairs % 8 == 0) {
    x = id & 7;
    id >>= 3;
    n >>= 3;
  }
  const int r = id % n;
  return {(x * n + r) / parts, id / n, r % parts};
}

// ---------------------------------------------------------------- forward
template <int D, int NW>
__global__ __launch_bounds__(NW * 64, 2)
void flash_fwd_kernel(const __hip_bfloat16* __restrict__ q, const __hip_bfloat16* __restrict__ k,
                      const __hip_bfloat16* __restrict__ v, __hip_bfloat16* __restrict__ o,
                      float* __restrict__ lse, Seqs seqs, Strides sq, Strides sk, Strides sv,
                      Strides so, int Hq, int Hkv, int nq, float scale_log2) {
  constexpr int KV = tile_rows<NW>(), NS = KV / 32, NT = NW * 64;
  const int group = Hq / Hkv;
  const Place at = place(blockIdx.x, gridDim.x / (nq * group), nq, group);
  const int qb = nq - 1 - at.block, hg = at.part, kvh = at.pair % Hkv, b = at.pair / Hkv;
  const int h = kvh * group + hg;
  const int row0 = seqs.first(b), len = seqs.len(b);
  if (qb * (NW * WROWS) >= len) return;

  const int wave = wave_id(), l = threadIdx.x & 63, half = l >> 5;
  const int q0 = qb * (NW * WROWS) + wave * WROWS;
  const int qq = q0 + (l & 31);
  const __hip_bfloat16* qp = q + b * sq.b + h * sq.h + (int64_t)row0 * sq.t;
  const __hip_bfloat16* kp = k + b * sk.b + kvh * sk.h + (int64_t)row0 * sk.t;
  const __hip_bfloat16* vp = v + b * sv.b + kvh * sv.h + (int64_t)row0 * sv.t;

  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int TB = KV * D * 2;
  const Frags<D> fr;
  bf16v8 qf[D / 16];
  load_row<D>(qf, qp, sq.t, min(qq, len - 1));  // rows past the end are not stored

  float m = -1e30f, lsum = 0.f;
  f32x16 acc[D / 32];
  #pragma unroll
  for (int dt = 0; dt < D / 32; ++dt) acc[dt] = zero16();

  const int last = min((qb + 1) * (NW * WROWS), len);   // keys of this workgroup
  const int n = (last + KV - 1) / KV;
  Rows<D, KV, NT> tk(sk.t), tv(sv.t);
  tk.fetch(kp, sk.t, len);
  tv.fetch(vp, sv.t, len);
  tk.store(smem);
  tv.store(smem + TB);
  __syncthreads();

  for (int t = 0; t < n; ++t) {
    const int kv0 = t * KV;
    char* ks_ = smem + (t & 1) * (2 * TB);
    char* vs_ = ks_ + TB;
    if (t + 1 < n) {
      tk.fetch(kp + (int64_t)(kv0 + KV) * sk.t, sk.t, len - kv0 - KV);
      tv.fetch(vp + (int64_t)(kv0 + KV) * sv.t, sv.t, len - kv0 - KV);
    }
    if (kv0 <= q0 + WROWS - 1 && q0 < len) {            // wave-uniform
      f32x16 st[NS];
      #pragma unroll
      for (int s = 0; s < NS; ++s) {
        st[s] = zero16();
        #pragma unroll
        for (int ks = 0; ks < D / 16; ++ks) st[s] = mfma(fr.row(ks_, s, ks), qf[ks], st[s]);
      }
      if (kv0 + KV - 1 > q0) {                          // the diagonal
        #pragma unroll
        for (int s = 0; s < NS; ++s)
          #pragma unroll
          for (int r = 0; r < 16; ++r)
            if (kv0 + s * 32 + acc_row(r, half) > qq) st[s][r] = -1e30f;
      }
      float mx = st[0][0];
      #pragma unroll
      for (int s = 0; s < NS; ++s)
        #pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, st[s][r]);
      // The exact running maximum is subtracted, so that a row's leading weight
      // is 1 and rounds to bf16 exactly. (Letting it lag by up to 2^8 saves most
      // of the rescaling, but the leading weight's rounding is then not in lsum:
      // output error against 64 bits 0.00212 instead of 0.00186 at T 1550.)
      const float m_new = fmaxf(m, halves_max(mx) * scale_log2);
      if (__any(m_new > m)) {
        const float alpha = __builtin_amdgcn_exp2f(m - m_new);
        lsum *= alpha;
        #pragma unroll
        for (int dt = 0; dt < D / 32; ++dt)
          #pragma unroll
          for (int r = 0; r < 16; ++r) acc[dt][r] *= alpha;
        m = m_new;
      }
      #pragma unroll
      for (int s = 0; s < NS; ++s)
        #pragma unroll
        for (int r = 0; r < 16; ++r) {
          st[s][r] = __builtin_amdgcn_exp2f(st[s][r] * scale_log2 - m);
          lsum += st[s][r];
        }
      #pragma unroll
      for (int s = 0; s < NS; ++s)
        #pragma unroll
        for (int k2 = 0; k2 < 2; ++k2) {
          const bf16v8 p = pack8(st[s], k2);
          #pragma unroll
          for (int dt = 0; dt < D / 32; ++dt)
            acc[dt] = mfma(fr.col(vs_, s * 32 + k2 * 16, dt), p, acc[dt]);
        }
    }
    if (t + 1 < n) {
      char* nk = smem + ((t + 1) & 1) * (2 * TB);
      tk.store(nk);
      tv.store(nk + TB);
      __syncthreads();
    }
  }

  lsum = halves_sum(lsum);
  store_rows<D>(acc, 1.f / lsum, o + b * so.b + h * so.h + (int64_t)(row0 + qq) * so.t, qq < len);
  if (lse != nullptr && half == 0 && qq < len)
    lse[b * seqs.b + h * seqs.h + row0 + qq] = m * LN2 + __logf(lsum);
}

// ------------------------------------------------------------- backward
// dQ: P = exp(S*scale - lse), dS = P * (dP - delta), dQ = scale * dS K.
template <int D, int NW>
__global__ __launch_bounds__(NW * 64, 2)
void flash_bwd_dq_kernel(const __hip_bfloat16* __restrict__ q, const __hip_bfloat16* __restrict__ k,
                         const __hip_bfloat16* __restrict__ v, const __hip_bfloat16* __restrict__ o,
                         const __hip_bfloat16* __restrict__ dout, const float* __restrict__ lse,
                         float* __restrict__ delta, __hip_bfloat16* __restrict__ dq, Seqs seqs,
                         Strides sq, Strides sk, Strides sv, Strides so, Strides sdo, Strides sdq,
                         int Hq, int Hkv, int nq, float scale) {
  constexpr int KV = tile_rows<NW>(), NS = KV / 32, NT = NW * 64;
  const int group = Hq / Hkv;
  const Place pl = place(blockIdx.x, gridDim.x / (nq * group), nq, group);
  const int qb = nq - 1 - pl.block, hg = pl.part, kvh = pl.pair % Hkv, b = pl.pair / Hkv;
  const int h = kvh * group + hg;
  const int row0 = seqs.first(b), T = seqs.len(b);
  if (qb * (NW * WROWS) >= T) return;

  const int wave = wave_id(), l = threadIdx.x & 63, half = l >> 5;
  const int q0 = qb * (NW * WROWS) + wave * WROWS;
  const int qq = q0 + (l & 31);
  const bool live = qq < T;
  const __hip_bfloat16* kp = k + b * sk.b + kvh * sk.h + (int64_t)row0 * sk.t;
  const __hip_bfloat16* vp = v + b * sv.b + kvh * sv.h + (int64_t)row0 * sv.t;

  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int TB = KV * D * 2;
  const Frags<D> fr;
  bf16v8 qf[D / 16], dof[D / 16];
  const int qrow = row0 + min(qq, T - 1);
  load_row<D>(qf, q + b * sq.b + h * sq.h, sq.t, qrow);
  load_row<D>(dof, dout + b * sdo.b + h * sdo.h, sdo.t, qrow);
  float dl = 0.f;
  {
    bf16v8 of[D / 16];
    load_row<D>(of, o + b * so.b + h * so.h, so.t, qrow);
    #pragma unroll
    for (int ks = 0; ks < D / 16; ++ks)
      #pragma unroll
      for (int j = 0; j < 8; ++j) dl += (float)of[ks][j] * (float)dof[ks][j];
    dl = halves_sum(dl);
  }
  const int64_t at = b * seqs.b + h * seqs.h + row0 + qq;
  const float scale_log2 = scale * LOG2E;
  const float lse2 = live ? lse[at] * LOG2E : 1e30f;    // 1e30: weight zero
  if (live && half == 0) delta[at] = dl;

  f32x16 acc[D / 32];
  #pragma unroll
  for (int dt = 0; dt < D / 32; ++dt) acc[dt] = zero16();

  const int last = min((qb + 1) * (NW * WROWS), T);
  const int n = (last + KV - 1) / KV;
  Rows<D, KV, NT> tk(sk.t), tv(sv.t);
  tk.fetch(kp, sk.t, T);
  tv.fetch(vp, sv.t, T);
  tk.store(smem);
  tv.store(smem + TB);
  __syncthreads();

  for (int t = 0; t < n; ++t) {
    const int kv0 = t * KV;
    char* ks_ = smem + (t & 1) * (2 * TB);
    char* vs_ = ks_ + TB;
    if (t + 1 < n) {
      tk.fetch(kp + (int64_t)(kv0 + KV) * sk.t, sk.t, T - kv0 - KV);
      tv.fetch(vp + (int64_t)(kv0 + KV) * sv.t, sv.t, T - kv0 - KV);
    }
    #pragma unroll
    for (int s = 0; s < NS; ++s) {
      const int c0 = kv0 + s * 32;
      if (c0 > q0 + WROWS - 1 || q0 >= T) continue;     // wave-uniform
      f32x16 st = zero16(), dp = zero16();
      __builtin_amdgcn_s_setprio(1);
      #pragma unroll
      for (int ks = 0; ks < D / 16; ++ks) {
        st = mfma(fr.row(ks_, s, ks), qf[ks], st);
        dp = mfma(fr.row(vs_, s, ks), dof[ks], dp);
      }
      __builtin_amdgcn_s_setprio(0);
      #pragma unroll
      for (int r = 0; r < 16; ++r)
        st[r] = __builtin_amdgcn_exp2f(st[r] * scale_log2 - lse2) * (dp[r] - dl);
      if (c0 + 31 > q0) {                               // the diagonal
        #pragma unroll
        for (int r = 0; r < 16; ++r)
          if (c0 + acc_row(r, half) > qq) st[r] = 0.f;
      }
      #pragma unroll
      for (int k2 = 0; k2 < 2; ++k2) {
        const bf16v8 ds = pack8(st, k2);
        #pragma unroll
        for (int dt = 0; dt < D / 32; ++dt)
          acc[dt] = mfma(fr.col(ks_, s * 32 + k2 * 16, dt), ds, acc[dt]);
      }
    }
    if (t + 1 < n) {
      char* nk = smem + ((t + 1) & 1) * (2 * TB);
      tk.store(nk);
      tv.store(nk + TB);
      __syncthreads();
    }
  }
  store_rows<D>(acc, scale, dq + b * sdq.b + h * sdq.h + (int64_t)(row0 + qq) * sdq.t, live);
}

// dK, dV of one kv head's 32*NW keys, summed over query heads
// hs*part .. of its group. Partials (split > 1) go to fp32 (split, B, Hkv, T, D),
// part_rows rows a share.
template <int D, int NW>
__global__ // two waves' tiles take twice the registers to fetch: 23 would spill
__launch_bounds__(NW * 64, NW == 2 && D == 128 ? 1 : 2)
void flash_bwd_dkv_kernel(const __hip_bfloat16* __restrict__ q, const __hip_bfloat16* __restrict__ k,
                          const __hip_bfloat16* __restrict__ v,
                          const __hip_bfloat16* __restrict__ dout, const float* __restrict__ lse,
                          const float* __restrict__ delta, __hip_bfloat16* __restrict__ dk,
                          __hip_bfloat16* __restrict__ dv, float* __restrict__ pk,
                          float* __restrict__ pv, Seqs seqs, Strides sq, Strides sk, Strides sv,
                          Strides sdo, Strides sdk, Strides sdv, int Hq, int Hkv, int nkv, int split,
                          int64_t part_rows, float scale) {
  constexpr int QT = 32, NT = NW * 64;
  const int group = Hq / Hkv;
  const Place pl = place(blockIdx.x, gridDim.x / (nkv * split), nkv, split);
  const int kb = pl.block, hs = pl.part, kvh = pl.pair % Hkv, b = pl.pair / Hkv;
  const int row0 = seqs.first(b), T = seqs.len(b);
  if (kb * (NW * WROWS) >= T) return;
  const int h0 = hs * group / split, h1 = (hs + 1) * group / split;

  const int wave = wave_id(), l = threadIdx.x & 63, half = l >> 5;
  const int kv0 = kb * (NW * WROWS) + wave * WROWS;
  const int kk = kv0 + (l & 31);
  const bool live = kk < T;

  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int TB = QT * D * 2, SB = 2 * TB + QT * 8;  // Q, dO, lse, delta
  constexpr int KB = NW * WROWS * D * 2;
  const Frags<D> lane;
  // V rows stay in registers, K rows in LDS: both in registers would leave
  // 256 too few for the accumulators, one wave a SIMD, and copies to the
  // accumulation registers around every product
  {
    Tile<D, NW * WROWS, NT> tk;
    const int r0 = kb * (NW * WROWS);
    tk.fetch(k + b * sk.b + kvh * sk.h + (int64_t)(row0 + r0) * sk.t, sk.t, T - r0);
    tk.store(smem);
  }
  bf16v8 vf[D / 16];
  load_row<D>(vf, v + b * sv.b + kvh * sv.h, sv.t, row0 + min(kk, T - 1));
  const float scale_log2 = scale * LOG2E;

  f32x16 ak[D / 32], av[D / 32];
  #pragma unroll
  for (int dt = 0; dt < D / 32; ++dt) { ak[dt] = zero16(); av[dt] = zero16(); }

  const int first = kb * (NW * WROWS), n = (T - first + QT - 1) / QT * (h1 - h0);
  Rows<D, QT, NT> tq(sq.t), td(sdo.t);
  // threads 0..31: lse, 32..63: delta of the tile's rows. Loaded by every wave and
  // only looked at when it is stored: a use behind a branch made the loop wait for
  // all of the next tile's loads here, a third of its time.
  float stat = 0.f;
  bool stat_live = false;
  const float* sp = ((threadIdx.x & 32) == 0 ? lse : delta) + b * seqs.b + row0;
  int fh = kvh * group + h0, fr0 = first;              // the next tile to fetch
  auto fetch = [&] {
    tq.fetch(q + b * sq.b + fh * sq.h + (int64_t)(row0 + fr0) * sq.t, sq.t, T - fr0);
    td.fetch(dout + b * sdo.b + fh * sdo.h + (int64_t)(row0 + fr0) * sdo.t, sdo.t, T - fr0);
    const int r = fr0 + (threadIdx.x & 31);
    stat = sp[fh * seqs.h + min(r, T - 1)];
    stat_live = r < T;
    fr0 += QT;
    if (fr0 >= T) { fr0 = first; ++fh; }
  };
  auto store = [&](int i) {
    char* s = smem + KB + (i & 1) * SB;
    tq.store(s);
    td.store(s + TB);
    // rows past the end get weight exp(-huge) = 0
    if (threadIdx.x < 64)
      reinterpret_cast<float*>(s + 2 * TB)[threadIdx.x] =
          threadIdx.x >= 32 ? stat : stat_live ? stat * LOG2E : 1e30f;
  };
  fetch();
  store(0);
  arrived<D>(vf);
  __syncthreads();

  int r0 = first;
  for (int i = 0; i < n; ++i) {
    char* qs = smem + KB + (i & 1) * SB;
    char* ds_ = qs + TB;
    const float* st_lse = reinterpret_cast<const float*>(ds_ + TB);
    if (i + 1 < n) fetch();
    if (r0 + QT - 1 >= kv0 && kv0 < T) {                // wave-uniform
      // a tile's fragment offsets anew in every step: sixteen registers less
      Frags<D> fr = lane;
      asm volatile("" : "+v"(fr.row_off), "+v"(fr.tr_lo), "+v"(fr.tr_hi));
      f32x16 s = zero16(), dp = zero16();
      __builtin_amdgcn_s_setprio(1);
      #pragma unroll
      for (int ks = 0; ks < D / 16; ++ks) {
        s = mfma(fr.row(qs, 0, ks), fr.row(smem, wave, ks), s);
        dp = mfma(fr.row(ds_, 0, ks), vf[ks], dp);
      }
      __builtin_amdgcn_s_setprio(0);
      #pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 le = *reinterpret_cast<const f32x4*>(st_lse + 8 * g + 4 * half);
        const f32x4 de = *reinterpret_cast<const f32x4*>(st_lse + 32 + 8 * g + 4 * half);
        #pragma unroll
        for (int j = 0; j < 4; ++j) {
          s[4 * g + j] = __builtin_amdgcn_exp2f(s[4 * g + j] * scale_log2 - le[j]);
          dp[4 * g + j] = s[4 * g + j] * (dp[4 * g + j] - de[j]);
        }
      }
      if (r0 < kv0 + WROWS - 1) {                       // the diagonal
        #pragma unroll
        for (int r = 0; r < 16; ++r)
          if (r0 + acc_row(r, half) < kk) s[r] = dp[r] = 0.f;
      }
      #pragma unroll
      for (int k2 = 0; k2 < 2; ++k2) {
        const bf16v8 p = pack8(s, k2), ds = pack8(dp, k2);
        __builtin_amdgcn_s_setprio(1);
        #pragma unroll
        for (int dt = 0; dt < D / 32; ++dt) {
          av[dt] = mfma(fr.col(ds_, k2 * 16, dt), p, av[dt]);
          ak[dt] = mfma(fr.col(qs, k2 * 16, dt), ds, ak[dt]);
        }
        __builtin_amdgcn_s_setprio(0);
      }
    }
    r0 += QT;
    if (r0 >= T) r0 = first;
    if (i + 1 < n) {
      store(i + 1);
      __syncthreads();
    }
  }

  if (split == 1) {
    store_rows<D>(ak, scale, dk + b * sdk.b + kvh * sdk.h + (int64_t)(row0 + kk) * sdk.t, live);
    store_rows<D>(av, 1.f, dv + b * sdv.b + kvh * sdv.h + (int64_t)(row0 + kk) * sdv.t, live);
  } else {
    // rows as the query heads' numbers lie, of Hkv heads
    const int64_t at = (hs * part_rows + b * (seqs.b / Hq) * Hkv + kvh * seqs.h + row0 + kk) * D;
    store_rows_f32<D>(ak, pk + at, live);
    store_rows_f32<D>(av, pv + at, live);
  }
}

// dK = scale * sum of partials, dV = sum of partials; 8 elements a thread.
template <int D>
__global__ __launch_bounds__(256)
void flash_bwd_sum_kernel(const float* __restrict__ pk, const float* __restrict__ pv,
                          __hip_bfloat16* __restrict__ dk, __hip_bfloat16* __restrict__ dv,
                          Strides sdk, Strides sdv, int Hkv, int T, int64_t rows, int split,
                          float scale) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t row = i / (D / 8);
  const int c = (int)(i % (D / 8)) * 8;
  if (row >= rows) return;
  const int t = (int)(row % T);
  const int64_t bh = row / T;
  const int kvh = (int)(bh % Hkv);
  const int64_t b = bh / Hkv;
  float a[8] = {0, 0, 0, 0, 0, 0, 0, 0}, w[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int s = 0; s < split; ++s) {
    const int64_t at = (s * rows + row) * D + c;
    #pragma unroll
    for (int j = 0; j < 8; ++j) { a[j] += pk[at + j]; w[j] += pv[at + j]; }
  }
  bf16x8 x, y;
  #pragma unroll
  for (int j = 0; j < 8; ++j) { x.v[j] = f2bf(a[j] * scale); y.v[j] = f2bf(w[j]); }
  *reinterpret_cast<bf16x8*>(dk + b * sdk.b + kvh * sdk.h + t * sdk.t + c) = x;
  *reinterpret_cast<bf16x8*>(dv + b * sdv.b + kvh * sdv.h + t * sdv.t + c) = y;
}

// A (B, H, T, D) operand whose rows can be read 16 B at a time as it lies.
torch::Tensor rows16(const torch::Tensor& x) {
  bool ok = x.stride(3) == 1 && reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0;
  for (int d = 0; d < 3; ++d) ok = ok && (x.size(d) == 1 || x.stride(d) % 8 == 0);
  ok = ok && x.stride(2) < (1 << 24);     // 64 rows of a tile within 32-bit offsets
  return ok ? x : x.clone(at::MemoryFormat::Contiguous);
}

Strides strides(const torch::Tensor& x) {
  return {x.stride(0), x.stride(1), (int)x.stride(2)};
}

// A flat batch is one (1, H, tokens, D) operand for all sequences.
Strides strides(const torch::Tensor& x, bool flat) {
  return {flat ? 0 : x.stride(0), x.stride(1), (int)x.stride(2)};
}

// The forward's running maximum and mask are those of unscaled scores: they
// need scale > 0.
torch::Tensor positive_scale(const torch::Tensor& q, double& scale) {
  if (scale > 0) return q;
  const bool zero = scale == 0;
  scale = zero ? 1 : -scale;
  return zero ? torch::zeros_like(q) : -q;
}

// An output laid out like the operand it belongs to, if that is dense.
torch::Tensor like(const torch::Tensor& x) {
  return x.is_non_overlapping_and_dense() ? torch::empty_like(x)
                                          : torch::empty(x.sizes(), x.options());
}

const __hip_bfloat16* bf(const torch::Tensor& x) {
  return reinterpret_cast<const __hip_bfloat16*>(x.data_ptr());
}
__hip_bfloat16* bfm(torch::Tensor& x) { return reinterpret_cast<__hip_bfloat16*>(x.data_ptr()); }

void check_qkv(const torch::Tensor& q, const torch::Tensor& k, const torch::Tensor& v) {
  TORCH_CHECK(q.is_cuda() && q.scalar_type() == at::kBFloat16);
  TORCH_CHECK(k.is_cuda() && v.is_cuda() && k.scalar_type() == at::kBFloat16 &&
              v.scalar_type() == at::kBFloat16);
  TORCH_CHECK(q.dim() == 4 && k.dim() == 4 && v.dim() == 4);
  TORCH_CHECK(k.size(0) == q.size(0) && k.size(2) == q.size(2) && k.size(3) == q.size(3) &&
              v.sizes() == k.sizes(), "flash attention: k/v shape mismatch");
  TORCH_CHECK(k.size(1) > 0 && q.size(1) % k.size(1) == 0);
  TORCH_CHECK(q.size(3) == 64 || q.size(3) == 128, "flash attention: head_dim 64/128 only");
}

// 128-row workgroups (four waves share a tile) once they fill the chip
// twice over; below that 64-row ones, which spread short batches wider.
int waves_for(int64_t rows_of_heads, int T) { return rows_of_heads * ((T + 127) / 128) >= 512 ? 4 : 2; }

#define FLASH_DISPATCH(D_, NW_, ...)                                             \
  [&] {                                                                         \
    if ((D_) == 128 && (NW_) == 4) { constexpr int D = 128, NW = 4; __VA_ARGS__; } \
    else if ((D_) == 128) { constexpr int D = 128, NW = 2; __VA_ARGS__; }        \
    else if ((NW_) == 4) { constexpr int D = 64, NW = 4; __VA_ARGS__; }          \
    else { constexpr int D = 64, NW = 2; __VA_ARGS__; }                          \
  }()

// B sequences of T rows, or (cu) of up to T rows of one flat batch
Seqs sequences(const torch::Tensor& q, const int* cu, int T) {
  return {cu, T, cu ? 0 : q.size(1) * q.size(2), q.size(2)};
}

void launch_fwd(const torch::Tensor& q, const torch::Tensor& k, const torch::Tensor& v,
                torch::Tensor& o, float* lse, const int* cu, int B, int T, double scale) {
  const int Hq = q.size(1), Hkv = k.size(1);
  const int nw = waves_for((int64_t)B * Hq, T);
  const int nq = (T + nw * WROWS - 1) / (nw * WROWS);
  const int64_t blocks = (int64_t)B * Hq * nq;
  if (blocks == 0) return;
  TORCH_CHECK(blocks < (1ll << 31), "flash attention: batch too large");
  auto stream = at::cuda::getCurrentCUDAStream();
  FLASH_DISPATCH(q.size(3), nw, {
    const size_t smem = 4 * tile_rows<NW>() * D * 2;
    hipLaunchKernelGGL((flash_fwd_kernel<D, NW>), dim3(blocks), dim3(NW * 64), smem, stream, bf(q),
                       bf(k), bf(v), bfm(o), lse, sequences(q, cu, T), strides(q, cu),
                       strides(k, cu), strides(v, cu), strides(o, cu), Hq, Hkv, nq,
                       (float)scale * LOG2E);
  });
  HIP_CHECK_LAST();
}

std::vector<torch::Tensor> launch_bwd(const torch::Tensor& dout, const torch::Tensor& q,
                                      const torch::Tensor& k, const torch::Tensor& v,
                                      const torch::Tensor& o, const torch::Tensor& lse,
                                      const int* cu, int B, int T, double scale,
                                      std::vector<torch::Tensor> grads = {}) {
  check_qkv(q, k, v);
  TORCH_CHECK(dout.scalar_type() == at::kBFloat16 && o.scalar_type() == at::kBFloat16 &&
              lse.scalar_type() == at::kFloat);
  TORCH_CHECK(dout.sizes() == q.sizes() && o.sizes() == q.sizes(),
              "flash_attn_bwd: dout/o shape mismatch");
  const int Hq = q.size(1), Hkv = k.size(1);
  const int64_t rows_all = q.size(0) * q.size(2);
  TORCH_CHECK(lse.numel() == Hq * rows_all, "flash_attn_bwd: lse shape mismatch");
  auto qc = rows16(q), kc = rows16(k), vc = rows16(v), oc = rows16(o), doc = rows16(dout);
  auto lsec = lse.contiguous();
  auto delta = torch::empty_like(lsec);
  if (grads.empty()) grads = {like(qc), like(kc), like(vc)};
  auto &dq = grads[0], &dk = grads[1], &dv = grads[2];
  const int nw = waves_for((int64_t)B * Hq, T);
  const int rows = nw * WROWS, nq = (T + rows - 1) / rows;
  const int64_t blocks = (int64_t)B * Hq * nq, kv_blocks = (int64_t)B * Hkv * nq;
  if (blocks == 0) return grads;
  TORCH_CHECK(blocks < (1ll << 31), "flash attention: batch too large");
  const int group = Hq / Hkv;
  // 768 workgroups and more: below that shares of the heads, whole ones where the
  // fullest would have two anyway. Partial sums cost: 832 blocks of the round above
  // as they are 1140 us, in halves 1230.
  int split = (int)std::min<int64_t>(group, (768 + kv_blocks - 1) / kv_blocks);
  if (2 * split > group) split = group;
  torch::Tensor part;
  float *pk = nullptr, *pv = nullptr;
  if (split > 1) {
    part = torch::empty({2, split, Hkv * rows_all, q.size(3)}, lsec.options());
    pk = part.data_ptr<float>();
    pv = pk + part.numel() / 2;
  }
  const Seqs seqs = sequences(q, cu, T);
  auto st = [&](const torch::Tensor& x) { return strides(x, cu); };
  auto stream = at::cuda::getCurrentCUDAStream();
  FLASH_DISPATCH(q.size(3), nw, {
    hipLaunchKernelGGL((flash_bwd_dq_kernel<D, NW>), dim3(blocks), dim3(NW * 64), 4 * tile_rows<NW>() * D * 2,
                       stream, bf(qc), bf(kc), bf(vc), bf(oc), bf(doc), lsec.data_ptr<float>(),
                       delta.data_ptr<float>(), bfm(dq), seqs, st(qc), st(kc), st(vc), st(oc),
                       st(doc), st(dq), Hq, Hkv, nq, (float)scale);
    hipLaunchKernelGGL((flash_bwd_dkv_kernel<D, NW>), dim3(kv_blocks * split), dim3(NW * 64),
                       NW * WROWS * D * 2 + 2 * (2 * 32 * D * 2 + 32 * 8), stream, bf(qc), bf(kc), bf(vc), bf(doc),
                       lsec.data_ptr<float>(), delta.data_ptr<float>(), bfm(dk), bfm(dv), pk, pv,
                       seqs, st(qc), st(kc), st(vc), st(doc), st(dk), st(dv), Hq, Hkv, nq, split,
                       Hkv * rows_all, (float)scale);
    if (split > 1) {
      const int64_t n = Hkv * rows_all;
      hipLaunchKernelGGL((flash_bwd_sum_kernel<D>), dim3((n * (D / 8) + 255) / 256), dim3(256), 0,
                         stream, pk, pv, bfm(dk), bfm(dv), strides(dk), strides(dv), Hkv,
                         (int)q.size(2), n, split, (float)scale);
    }
  });
  HIP_CHECK_LAST();
  return grads;
}

// A flat (tokens, H, D) batch as one (1, H, tokens, D) operand
torch::Tensor flat4(const torch::Tensor& x) {
  TORCH_CHECK(x.dim() == 3);
  return x.transpose(0, 1).unsqueeze(0);
}

// an output that the kernels can write as it lies
void check_out(const torch::Tensor& out, const torch::Tensor& like) {
  TORCH_CHECK(out.is_cuda() && out.sizes() == like.sizes() && out.scalar_type() == at::kBFloat16);
  const auto o4 = flat4(out);
  TORCH_CHECK(rows16(o4).is_same(o4), "flash attention: output rows on 16 bytes");
}

void check_cu(const torch::Tensor& q, const torch::Tensor& cu, int64_t max_len) {
  TORCH_CHECK(cu.is_cuda() && cu.scalar_type() == at::kInt && cu.is_contiguous() && cu.dim() == 1 &&
              cu.numel() >= 1);
  TORCH_CHECK(max_len >= 0 && max_len <= q.size(0));
}

}  // namespace

std::vector<torch::Tensor> flash_attn_fwd(torch::Tensor q, torch::Tensor k, torch::Tensor v,
                                          double scale) {
  check_qkv(q, k, v);
  auto qc = rows16(positive_scale(q, scale)), kc = rows16(k), vc = rows16(v);
  auto o = like(qc);
  auto lse = torch::empty({q.size(0), q.size(1), q.size(2)}, q.options().dtype(at::kFloat));
  launch_fwd(qc, kc, vc, o, lse.data_ptr<float>(), nullptr, q.size(0), q.size(2), scale);
  return {o, lse};
}

// Causal attention inside each of the sequences cu[i] .. cu[i+1] of a flat
// batch: q (tokens, Hq, D), k/v (tokens, Hkv, D), cu int32 (n+1,) rising from
// 0 to tokens, max_len the longest of them. {output, log-sum-exp (Hq, tokens)};
// into: where the output goes, rows of a wider matrix.
std::vector<torch::Tensor> flash_varlen_fwd(torch::Tensor q, torch::Tensor k, torch::Tensor v,
                                            torch::Tensor cu, int64_t max_len, double scale,
                                            c10::optional<torch::Tensor> into) {
  auto q4 = flat4(q), k4 = flat4(k), v4 = flat4(v);
  check_cu(q, cu, max_len);
  check_qkv(q4, k4, v4);
  auto qc = rows16(positive_scale(q4, scale)), kc = rows16(k4), vc = rows16(v4);
  auto out = into ? *into : torch::empty(q.sizes(), q.options());
  check_out(out, q);
  auto lse = torch::empty({q.size(1), q.size(0)}, q.options().dtype(at::kFloat));
  auto o4 = flat4(out);
  launch_fwd(qc, kc, vc, o4, lse.data_ptr<float>(), cu.data_ptr<int>(), cu.numel() - 1, max_len,
             scale);
  return {out, lse};
}

torch::Tensor flash_attn_varlen(torch::Tensor q, torch::Tensor k, torch::Tensor v,
                                torch::Tensor cu, int64_t max_len, double scale) {
  return flash_varlen_fwd(q, k, v, cu, max_len, scale, c10::nullopt)[0];
}

std::vector<torch::Tensor> flash_attn_bwd(torch::Tensor dout, torch::Tensor q, torch::Tensor k,
                                          torch::Tensor v, torch::Tensor o, torch::Tensor lse,
                                          double scale) {
  return launch_bwd(dout, q, k, v, o, lse, nullptr, q.size(0), q.size(2), scale);
}

// dq, dk, dv of flash_varlen_fwd into (tokens, H, D) tensors, rows of wider ones
void flash_varlen_bwd(torch::Tensor dout, torch::Tensor q, torch::Tensor k, torch::Tensor v,
                      torch::Tensor o, torch::Tensor lse, torch::Tensor cu, int64_t max_len,
                      double scale, torch::Tensor dq, torch::Tensor dk, torch::Tensor dv) {
  check_cu(q, cu, max_len);
  check_out(dq, q);
  check_out(dk, k);
  check_out(dv, v);
  launch_bwd(flat4(dout), flat4(q), flat4(k), flat4(v), flat4(o), lse, cu.data_ptr<int>(),
             cu.numel() - 1, max_len, scale, {flat4(dq), flat4(dk), flat4(dv)});
}

// The differentiable call: a node of the C++ engine (from Python, node and
// dispatch of forward and backward took as long as the kernels of a short
// micro-batch: 90 us a pass at (2, 14/2, 333, 64), 73 now).
namespace {

struct FlashAttention : public torch::autograd::Function<FlashAttention> {
  static torch::Tensor forward(torch::autograd::AutogradContext* ctx, torch::Tensor q,
                               torch::Tensor k, torch::Tensor v, double scale) {
    auto r = flash_attn_fwd(q, k, v, scale);
    ctx->save_for_backward({q, k, v, r[0], r[1]});
    ctx->saved_data["scale"] = scale;
    return r[0];
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    const auto s = ctx->get_saved_variables();
    auto r = flash_attn_bwd(grads[0].to(s[0].scalar_type()), s[0], s[1], s[2], s[3], s[4],
                            ctx->saved_data["scale"].toDouble());
    return {r[0], r[1], r[2], torch::Tensor()};
  }
};

}  // namespace

torch::Tensor flash_attention(torch::Tensor q, torch::Tensor k, torch::Tensor v, double scale) {
  return FlashAttention::apply(q, k, v, scale);
}
