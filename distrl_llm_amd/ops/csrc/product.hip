// Products of many rows on matrix cores, y = sum of x[:, part] B, bf16 with fp32 sums:
// the projections of LoRA training and their input gradients, each with what stands
// around it in the layer (bias, residual sum, SiLU*mul forward and backward).
//
// A workgroup owns a tile of the output and walks K 32 at a time. Operands go from
// global memory straight into LDS, four tiles of K in a ring: what is read now, and
// three on their way. Rows of 64 B are XOR-swizzled in 16 B chunks by the address each
// lane loads from, as such a load writes its lanes one behind the other. B as it lies
// in backward, (K, N), is read back with LDS transpose reads.
//  * Tiles of up to 256 x 256: eight waves, two a SIMD, in two groups one phase apart:
//    while one group reads its operands, the other has the matrix cores. The rows of a
//    tile, 128 to 256 of them, are what makes the last round of workgroups fullest.
//  * Small outputs: tiles of 128 x 128 and 64 x 64 of four waves, several a CU, whose
//    waves read a step's operands during the one before; K in up to eight shares, which
//    the last workgroup of a tile to end adds up in their order.
// A sum may run over several matrices: an adapter is more of its projection's K, taken
// from where it lies, so that weights are not laid out beside adapters first.
//
// Large tiles are bound by LDS: 96 KB read and 32 KB written a step are 1024 clocks,
// as many as its products. 8192 x 8192 x 8192 790 us, 1390 TFLOP/s (library 680);
// 18793 x 2048 x 1568 121 (139); 4000 x 1536 x 8992 125 (109 and 20 for what it needs
// beside adapters); 924 x 896 x 4896 27 (28), 924 x 1152 x 928 9.5 (19, its launch).
// Sums over a vocabulary in shares of K, us (library's product): rows x 896 x 151936, 5 rows
// 51 (184), 130 rows 78 (320), 561 rows 180 (437), 4801 rows 1205 (1650); 14400 x 1536 x
// 151936 5540 (8397), 9000 x 3584 x 152064 7530 (11236).
// One wave a SIMD with tiles of 128 x 128 each, for less LDS, spilled registers: 1530
// us where this takes 930. Pairs of steps loaded together, for whole cache lines, were
// slower (8192^3 870 for 770).
#include <ATen/cuda/CUDAContext.h>
#include "common.h"
#include "product.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16v8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16v4;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((address_space(3))) bf16v4 lds_bf16v4;

namespace {

constexpr int BK = 32, RING = 4;
constexpr int TERMS = 6, BLOCKS = 3;

enum { PLAIN = 0, GLU = 1, GLU_BWD = 2 };

struct Term {
  const __hip_bfloat16 *a, *b;
  int lda, ldb, steps;
};

struct Args {
  int M, cols, steps;                   // cols: columns of tiles
  Term term[TERMS];
  int first[BLOCKS], terms[BLOCKS];     // of a block, or of gate and up
  int width[BLOCKS], tiles[BLOCKS];     // columns, and columns of tiles
  const __hip_bfloat16* bias[BLOCKS];
  __hip_bfloat16* c;                    // GLU: [gate | up], or null
  int ldc;
  const __hip_bfloat16* res;
  int ldr;
  __hip_bfloat16* act;
  int ldact;
  const __hip_bfloat16* gu;
  int ldgu;
  __hip_bfloat16 *dgate, *dup;
  int ldd;
  // shares of K a workgroup each, which the last of a tile to end adds up, or (large
  // tiles) a launch behind this one
  int splits;
  float* part;                          // (tiles, shares, floats of a tile), or (shares, M, N)
  unsigned long long *there, tag;       // (tiles, shares)
};

// what a term without b multiplies by: 32 columns, any number of times
__device__ const uint4 ZEROS[4] = {};

// 16 B a lane from base + off into LDS at lds + 16 * lane. m0 is lost to the compiler,
// which warns that nothing keeps it: nothing has to.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
DEV_INLINE void load_to_lds(uint32_t lds, const char* base, uint32_t off) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :: "s"(lds), "v"(off), "s"(base) : "memory", "m0");
}
#pragma clang diagnostic pop
// Until at most VM of this wave's loads are on their way and its LDS reads are done.
template <int VM>
DEV_INLINE void arrived() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"(VM) : "memory"); }
DEV_INLINE void meet() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

DEV_INLINE float silu(float g) { return g / (1.f + __expf(-g)); }

// Where 32 B of a row of B (K, N) lie among the row's, by its row in the tile: the 16
// rows of a transpose read spread over all banks.
template <int BN>
DEV_INLINE int row_swizzle(int k) {
  return BN >= 128 ? (k & 3) | ((k >> 3) & 1) << 2 : ((k >> 1) & 1) | ((k >> 3) & 1) << 1;
}

// WM x WN waves of TM x TN products of 16 x 16
template <int WM, int WN, int TM, int TN, bool ROWS, int MODE>
__global__ __launch_bounds__(WM * WN * 64, 2)
void product_kernel(const Args args) {
  constexpr int NW = WM * WN, BM = WM * TM * 16, BN = WN * TN * 16;
  // pieces of 1 KB a wave loads; of A some past a tile's rows where they don't divide
  constexpr int PA = CDIV(BM / 16, NW), PB = BN / 16 / NW, EACH = PA + PB;
  constexpr bool SPLITS = NW == 4, SHARES = NW == 8 && MODE == PLAIN;
  constexpr int ABYTES = PA * NW * 1024, RINGBYTES = ABYTES + BN * BK * 2;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = threadIdx.x & 63, g = l >> 4, lr = l & 15, wm = wave / WN, wn = wave % WN;
  const int M = args.M;

  // An XCD takes tiles one behind the other, four rows of tiles by turns of columns, so
  // that what runs on it at once shares its L2.
  // Of large tiles all of one share of K, then the next share's.
  int m_tile, n_tile, share = SPLITS ? blockIdx.y : 0;
  {
    const int rows = CDIV(M, BM), cols = args.cols, tiles = rows * cols;
    const int x = blockIdx.x & 7, total = SHARES ? tiles * args.splits : tiles;
    int t = x * (total >> 3) + min(x, total & 7) + (blockIdx.x >> 3);
    if (SHARES && args.splits > 1) {
      share = t / tiles;
      t -= share * tiles;
    }
    const int band = t / (4 * cols), in = t - band * 4 * cols, h = min(4, rows - band * 4);
    m_tile = band * 4 + in % h;
    n_tile = in / h;
  }
  int block = 0, c0 = 0;                // c0: the block's first column in the output
  if (MODE == PLAIN)
    while (n_tile >= args.tiles[block]) {
      n_tile -= args.tiles[block];
      c0 += args.width[block];
      ++block;
    }
  const int N = args.width[block], m0 = m_tile * BM, n0 = n_tile * (MODE == GLU ? BN / 2 : BN);
  // gate rows of B, then up rows: a wave loads of one of them
  const int half = MODE == GLU && wave >= NW / 2 ? 1 : 0;

  // what this lane loads: rows of A, and rows or columns of B
  int term = args.first[MODE == GLU ? half : block], left, ldb;
  const int end = term + args.terms[MODE == GLU ? half : block];
  const char *ap, *bp;
  uint32_t ao[PA], bo[PB];
  auto start = [&] {
    const Term& t = args.term[term];
    left = t.steps;
    ldb = t.ldb;
    ap = reinterpret_cast<const char*>(t.a + (int64_t)m0 * t.lda);
    #pragma unroll
    for (int i = 0; i < PA; ++i) {
      const int r = (wave * PA + i) * 16 + (l >> 2);
      // past the end the last again; pieces past the tile's rows, unread, one row
      const int row = (wave * PA + i) * 16 < BM ? min(r, M - 1 - m0) : 0;
      ao[i] = (uint32_t)row * t.lda * 2 + ((l & 3) ^ ((l >> 3) & 3)) * 16;
    }
    const auto* b = t.b ? t.b : reinterpret_cast<const __hip_bfloat16*>(ZEROS);
    bp = reinterpret_cast<const char*>(b + (t.b ? (ROWS ? n0 : (int64_t)n0 * ldb) : 0));
    #pragma unroll
    for (int i = 0; i < PB; ++i) {
      if constexpr (ROWS) {
        constexpr int CHUNKS = BN / 8, AT_ONCE = 64 / CHUNKS;
        const int k = (wave * PB + i) * AT_ONCE + l / CHUNKS, p = l % CHUNKS;
        const int c = min((((p >> 1) ^ row_swizzle<BN>(k)) << 1) | (p & 1), (N - n0) / 8 - 1);
        bo[i] = (uint32_t)k * ldb * 2 + c * 16;
      } else {
        const int r = (wave * PB + i) * 16 + (l >> 2) - half * (BN / 2);
        bo[i] = (uint32_t)min(r, N - 1 - n0) * ldb * 2 + ((l & 3) ^ ((l >> 3) & 3)) * 16;
      }
    }
  };
  start();
  int step0 = 0, steps = args.steps;
  if (SPLITS || (SHARES && args.splits > 1)) {
    step0 = (int)((int64_t)share * args.steps / args.splits);
    steps = (int)((int64_t)(share + 1) * args.steps / args.splits) - step0;
    int skip = step0;
    while (skip >= left) {
      skip -= left;
      ++term;
      start();
    }
    left -= skip;
    ap += skip * BK * 2;
    if (ROWS) bp += (int64_t)skip * ldb * BK * 2;
    else if (ldb) bp += skip * BK * 2;
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  auto load = [&](int s) {
    const uint32_t to = lds0 + (s % RING) * RINGBYTES;
    #pragma unroll
    for (int i = 0; i < PA; ++i) load_to_lds(to + (wave * PA + i) * 1024, ap, ao[i]);
    #pragma unroll
    for (int i = 0; i < PB; ++i) load_to_lds(to + ABYTES + (wave * PB + i) * 1024, bp, bo[i]);
    ap += BK * 2;
    if (ROWS) bp += (int64_t)ldb * BK * 2;
    else if (ldb) bp += BK * 2;         // zeros stay where they are
    if (--left == 0 && ++term < end) start();
  };

  const int fo = lr * 64 + ((g ^ ((lr >> 1) & 3)) << 4);
  int no[TN];
  #pragma unroll
  for (int j = 0; j < TN; ++j) {
    if constexpr (ROWS) {
      const int k = 8 * g + (lr >> 2);
      no[j] = ABYTES + k * BN * 2 + (((wn * TN + j) ^ row_swizzle<BN>(k)) << 5) + (l & 3) * 8;
    } else if constexpr (MODE == GLU) {
      const int tile = j < TN / 2 ? wn * (TN / 2) + j : (BN / 2) / 16 + wn * (TN / 2) + j - TN / 2;
      no[j] = ABYTES + tile * 1024 + fo;
    } else {
      no[j] = ABYTES + (wn * TN + j) * 1024 + fo;
    }
  }
  f32x4 acc[TM][TN];
  #pragma unroll
  for (int i = 0; i < TM; ++i)
    #pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  constexpr int SETS_OF = NW == 8 ? 1 : 2;
  bf16v8 fa[SETS_OF][TM], fb[SETS_OF][TN];
  auto read = [&](int f, int s) {
    const char* p = smem + (s % RING) * RINGBYTES;
    #pragma unroll
    for (int j = 0; j < TN; ++j) {
      if constexpr (ROWS) {
        const bf16v4 x = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16v4*)(p + no[j]));
        const bf16v4 y =
            __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16v4*)(p + no[j] + 4 * BN * 2));
        fb[f][j] = __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7);
      } else {
        fb[f][j] = *reinterpret_cast<const bf16v8*>(p + no[j]);
      }
    }
    #pragma unroll
    for (int i = 0; i < TM; ++i)
      fa[f][i] = *reinterpret_cast<const bf16v8*>(p + (wm * TM + i) * 1024 + fo);
  };
  auto multiply = [&](int f) {
    #pragma unroll
    for (int i = 0; i < TM; ++i)
      #pragma unroll
      for (int j = 0; j < TN; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[f][j], fa[f][i], acc[i][j], 0, 0, 0);
  };

  if constexpr (NW == 8) {
    // Phases: reads of a step, then its products; the second group of waves one phase
    // behind the first. A step's loads have arrived for both groups a phase before the
    // first reads it, and go where both have read, three steps back.
    for (int s = 0; s < min(RING - 1, steps); ++s) load(s);
    if (steps >= RING - 1) arrived<(RING - 2) * EACH>(); else arrived<0>();
    meet();
    if (wave >= 4) meet();
    for (int s = 0; s < steps; ++s) {
      if (s + RING - 1 < steps) {
        load(s + RING - 1);
        read(0, s);
        arrived<(RING - 2) * EACH>();
      } else {
        read(0, s);
        arrived<0>();
      }
      meet();
      __builtin_amdgcn_s_setprio(1);
      multiply(0);
      __builtin_amdgcn_s_setprio(0);
      meet();
    }
    if (wave < 4) meet();
  } else {
    // A step reads the next one's operands while it multiplies its own, and loads into
    // the place that was read a step before.
    for (int s = 0; s < min(RING, steps); ++s) load(s);
    if (steps >= RING) arrived<(RING - 1) * EACH>(); else arrived<0>();
    meet();
    read(0, 0);
    if (steps >= RING) arrived<(RING - 2) * EACH>(); else arrived<0>();
    meet();
    auto step = [&](int f, int s) {
      if (s + RING < steps) load(s + RING);
      if (s + 1 < steps) read(f ^ (SETS_OF - 1), s + 1);
      multiply(f);
      if (s + RING < steps) arrived<(RING - 2) * EACH>(); else arrived<0>();
      meet();
    };
    int s = 0;
    for (; s + 1 < steps; s += 2) {
      step(0, s);
      step(SETS_OF - 1, s + 1);
    }
    if (s < steps) step(0, s);
  }

  if constexpr (SPLITS) {
    if (args.splits > 1) {
      // every share's sums in turn, whoever adds them: [pair of floats][thread]
      __shared__ int last;
      const int64_t tile = blockIdx.x;
      constexpr int PAIRS = TM * TN * 2, THREADS = NW * 64;
      auto* part = reinterpret_cast<unsigned long long*>(args.part) +
                   tile * args.splits * PAIRS * THREADS + threadIdx.x;
      #pragma unroll
      for (int p = 0; p < PAIRS; ++p) {
        const f32x4& x = acc[p / 2 / TN][p / 2 % TN];
        store_through(part + ((int64_t)share * PAIRS + p) * THREADS,
                      (unsigned long long)__float_as_uint(x[p % 2 * 2 + 1]) << 32 |
                          __float_as_uint(x[p % 2 * 2]));
      }
      stores_done();
      __syncthreads();
      if (wave == 0) {
        const bool all = all_there(args.there + tile * args.splits, args.splits, share, args.tag);
        if (l == 0) last = all;
      }
      __syncthreads();
      if (!last) return;
      #pragma unroll
      for (int i = 0; i < TM; ++i)
        #pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      for (int z = 0; z < args.splits; ++z) {
        unsigned long long v[PAIRS];
        #pragma unroll
        for (int p = 0; p < PAIRS; ++p)
          v[p] = load_through(part + ((int64_t)z * PAIRS + p) * THREADS);
        #pragma unroll
        for (int p = 0; p < PAIRS; ++p) {
          f32x4& x = acc[p / 2 / TN][p / 2 % TN];
          x[p % 2 * 2] += __uint_as_float((uint32_t)v[p]);
          x[p % 2 * 2 + 1] += __uint_as_float((uint32_t)(v[p] >> 32));
        }
      }
    }
  }

  // acc[i][j]: row m = lr of tile i, columns 4 g + 0..3 of tile j. What the epilogue
  // reads is in flight two rows of tiles ahead, past the end the last again: behind a
  // branch each, 32 loads would wait one for the other.
  auto row_of = [&](int i) { return m0 + (wm * TM + i) * 16 + lr; };
  constexpr int HALF = MODE == GLU ? TN / 2 : TN;       // tiles of output columns
  int n[HALF], nc[HALF];
  #pragma unroll
  for (int j = 0; j < HALF; ++j) {
    n[j] = n0 + (wn * HALF + j) * 16 + g * 4;
    nc[j] = min(n[j], N - 4);
  }
  auto at4 = [](const __hip_bfloat16* p) { return *reinterpret_cast<const bf16v4*>(p); };
  if constexpr (SHARES) {
    if (args.splits > 1) {
      float* part = args.part + (int64_t)share * M * N;
      #pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int m = row_of(i);
        #pragma unroll
        for (int j = 0; j < TN; ++j)
          if (m < M && n[j] < N) *reinterpret_cast<f32x4*>(part + (int64_t)m * N + n[j]) = acc[i][j];
      }
      return;
    }
  }
  if constexpr (MODE != GLU_BWD) {
    #pragma unroll
    for (int h = 0; h < TN / HALF; ++h) {
      const __hip_bfloat16* bias = args.bias[MODE == GLU ? h : block];
      if (!bias) continue;
      #pragma unroll
      for (int j = 0; j < HALF; ++j) {
        const bf16v4 b = at4(bias + nc[j]);
        #pragma unroll
        for (int i = 0; i < TM; ++i)
          #pragma unroll
          for (int r = 0; r < 4; ++r) acc[i][h * HALF + j][r] += (float)b[r];
      }
    }
  }
  constexpr int SETS = MODE == GLU_BWD ? 2 : 1, AHEAD = 2;
  bf16v4 in[TM][SETS][HALF];
  auto fetch = [&](int i) {
    if constexpr (MODE != GLU) {
      const int64_t m = min(row_of(i), M - 1);
      #pragma unroll
      for (int j = 0; j < HALF; ++j) {
        if constexpr (MODE == GLU_BWD) {
          const __hip_bfloat16* p = args.gu + m * args.ldgu + nc[j];
          in[i][0][j] = at4(p);
          in[i][SETS - 1][j] = at4(p + N);
        } else {
          in[i][0][j] = at4(args.res + m * args.ldr + c0 + nc[j]);
        }
      }
    }
  };
  const bool fetches = MODE == GLU_BWD || (MODE == PLAIN && args.res);
  if (fetches) {
    #pragma unroll
    for (int i = 0; i < AHEAD; ++i) fetch(i);
  }
  #pragma unroll
  for (int i = 0; i < TM; ++i) {
    if (fetches && i + AHEAD < TM) fetch(i + AHEAD);
    const int m = row_of(i);
    #pragma unroll
    for (int j = 0; j < HALF; ++j) {
      const f32x4 x = acc[i][j];
      bf16v4 o, p, q;
      #pragma unroll
      for (int r = 0; r < 4; ++r) {
        if constexpr (MODE == GLU) {
          o[r] = (__bf16)x[r];
          p[r] = (__bf16)acc[i][j + TN / 2][r];
          q[r] = (__bf16)(silu((float)o[r]) * (float)p[r]);
        } else if constexpr (MODE == GLU_BWD) {
          const float v = (float)in[i][0][j][r], sig = 1.f / (1.f + __expf(-v));
          o[r] = (__bf16)(x[r] * (float)in[i][SETS - 1][j][r] * sig * (1.f + v * (1.f - sig)));
          p[r] = (__bf16)(x[r] * v * sig);
        } else {
          o[r] = (__bf16)(fetches ? x[r] + (float)in[i][0][j][r] : x[r]);
        }
      }
      if (m >= M || n[j] >= N) continue;
      auto put = [&](__hip_bfloat16* to, bf16v4 v) { *reinterpret_cast<bf16v4*>(to) = v; };
      if constexpr (MODE == GLU_BWD) {
        put(args.dgate + (int64_t)m * args.ldd + n[j], o);
        put(args.dup + (int64_t)m * args.ldd + n[j], p);
      } else {
        if (MODE == PLAIN || args.c) put(args.c + (int64_t)m * args.ldc + c0 + n[j], o);
        if constexpr (MODE == GLU) {
          if (args.c) put(args.c + (int64_t)m * args.ldc + N + n[j], p);
          put(args.act + (int64_t)m * args.ldact + n[j], q);
        }
      }
    }
  }
}

// out (rows of ld elements) <- the shares' sums in their order, (shares, M, N); four
// columns a thread. Bound: memory.
__global__ __launch_bounds__(256)
void share_sum_kernel(const float* __restrict__ part, __hip_bfloat16* __restrict__ out,
                      uint32_t cells, uint32_t N, int64_t ld, int shares) {
  const uint32_t at = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (at >= cells) return;
  f32x4 sum = *reinterpret_cast<const f32x4*>(part + at);
  #pragma unroll 4
  for (int z = 1; z < shares; ++z) sum += *reinterpret_cast<const f32x4*>(part + (int64_t)z * cells + at);
  bf16v4 o;
  #pragma unroll
  for (int r = 0; r < 4; ++r) o[r] = (__bf16)sum[r];
  *reinterpret_cast<bf16v4*>(out + at / N * ld + at % N) = o;
}

template <int WM, int WN, int TM, int TN, bool ROWS, int MODE>
void launch(Args& a, int blocks, int splits) {
  constexpr int NW = WM * WN, BM = WM * TM * 16, BN = WN * TN * 16;
  constexpr int smem = RING * (CDIV(BM / 16, NW) * NW * 1024 + BN * BK * 2);
  static const hipError_t raised = hipFuncSetAttribute(
      reinterpret_cast<const void*>(&product_kernel<WM, WN, TM, TN, ROWS, MODE>),
      hipFuncAttributeMaxDynamicSharedMemorySize, smem);
  TORCH_CHECK(raised == hipSuccess, "product: LDS");
  a.cols = 0;
  for (int i = 0; i < blocks; ++i) {
    a.tiles[i] = CDIV(a.width[i], MODE == GLU ? BN / 2 : BN);
    a.cols += a.tiles[i];
    if (MODE == GLU) break;             // gate and up side by side in every tile
  }
  const int64_t total = (int64_t)CDIV(a.M, BM) * a.cols;
  TORCH_CHECK(total < (1 << 30), "product: size");
  constexpr bool JOINS = NW == 4;       // in the kernel, in every mode
  const bool plain = MODE == PLAIN && blocks == 1 && !a.bias[0] && !a.res;
  a.splits = JOINS || plain ? std::max(1, std::min(splits, a.steps)) : 1;
  at::Tensor room;
  const int64_t cells = (int64_t)a.M * a.width[0];
  if (!JOINS && a.splits > 1) {
    TORCH_CHECK(a.splits * cells < (int64_t)1 << 31 && total * a.splits < (1 << 30), "product: shares");
    // where memory has no room for the partial sums, tiles take all of K
    try {
      room = at::empty({a.splits * cells}, at::TensorOptions().dtype(at::kFloat).device(
          at::kCUDA, at::cuda::current_device()));
      a.part = room.data_ptr<float>();
    } catch (const c10::OutOfMemoryError&) {
      a.splits = 1;
    }
  } else if (a.splits > 1) {
    const int64_t shares = total * a.splits;
    room = at::empty({shares * (BM * BN * 4 + 8)}, at::TensorOptions().dtype(at::kByte).device(
        at::kCUDA, at::cuda::current_device()));
    a.there = reinterpret_cast<unsigned long long*>(room.data_ptr());
    a.part = reinterpret_cast<float*>(a.there + shares);
    a.tag = arrival_tag();
  }
  const auto stream = at::cuda::getCurrentCUDAStream();
  hipLaunchKernelGGL((product_kernel<WM, WN, TM, TN, ROWS, MODE>),
                     JOINS ? dim3(total, a.splits) : dim3(total * a.splits), dim3(NW * 64), smem,
                     stream, a);
  HIP_CHECK_LAST();
  if (!JOINS && a.splits > 1) {
    hipLaunchKernelGGL(share_sum_kernel, dim3(CDIV(cells, 1024)), dim3(256), 0, stream, a.part, a.c,
                       cells, a.width[0], a.ldc, a.splits);
    HIP_CHECK_LAST();
  }
}

template <bool ROWS, int MODE>
void by_size(Args& a, int blocks, int tile) {
  auto columns = [&](int bn) {
    int n = 0;
    for (int i = 0; i < (MODE == GLU ? 1 : blocks); ++i)
      n += CDIV(a.width[i], MODE == GLU ? bn / 2 : bn);
    return n;
  };
  // Time a step of K, us, by workgroups (of n a CU) and tiles, fitted to a sweep of 60
  // shapes of 80 to 18793 rows and all tiles: within a tenth of the best for most.
  int pick = 64, splits = 1;
  double least = 1e30;
  auto offer = [&](int what, int z, double cost) {
    if (cost < least) { least = cost; pick = what; splits = z; }
  };
  // Sums over a vocabulary (the LM head's input gradient), in shares where tiles alone leave
  // workgroups idle or their last round half empty: 561 x 896 x 151936 is 12 tiles. Shorter
  // ones of few rows are the small tiles', whose shares meet without a launch. 1 GB of
  // partial sums at most, 6 us for the launch that adds them at 4.5 TB/s. Fitted apart, to 87
  // shapes of 5 to 19200 rows, 896 to 8192 wide, over 32768 to 152064 words: within 3 % of
  // the best for nearly all. With the costs below for them, library's product, so, us:
  // 2408 x 4096 x 128256 2390, 2141, 2158; 1200 x 8192 x 152064 2850, 2577, 2562; 1200 x
  // 4096 x 32768, without shares, 442, 395, 278; 6400 x 1536 x 151936 2834, 5093, 2394.
  const int64_t cells = (int64_t)a.M * a.width[0];
  const bool sums = MODE == PLAIN && blocks == 1 && !a.bias[0] && !a.res && a.steps >= 1024;
  for (int tm = 8; tm >= 4; --tm) {
    const int64_t tiles = (int64_t)CDIV(a.M, 32 * tm) * columns(256);
    if (!sums) {
      const int64_t rounds = CDIV(tiles, (int64_t)256);
      offer(tm, 1, a.steps * (rounds == 1 ? 0.29 + 0.043 * tm : rounds * (0.24 + 0.081 * tm)));
      continue;
    }
    for (int z = 1; z <= 64 && (z == 1 || (a.steps / z >= 64 && z * cells <= 1 << 28)); ++z) {
      const int64_t rounds = CDIV(tiles * z, (int64_t)256);
      const double full = 0.27 + 0.063 * tm, half = 0.26 + 0.045 * tm;
      const double step = rounds > 1 ? rounds * 1.02 * full
                                     : half + (full - half) * std::max(0., tiles * z / 128. - 1);
      offer(tm, z, CDIV(a.steps, z) * step + (z > 1 ? 6. + z * cells * 8 / 4.5e6 : 0.));
    }
  }
  for (int z = 1; z <= 8 && (z == 1 || a.steps / z >= 8); ++z) {
    const double n128 = CDIV(a.M, 128) * (double)columns(128) * z / 256;
    const double n64 = CDIV(a.M, 64) * (double)columns(64) * z / 256;
    const double join = z > 1 ? 4. + z * 0.5 : 0.;
    offer(128, z, a.steps / z * (n128 <= 1 ? 0.3 : 0.62 * std::ceil(n128 / 2)) + join);
    offer(64, z, a.steps / z * (n64 <= 5 ? 0.05 + 0.14 * std::ceil(n64) : 0.78 * std::ceil(n64 / 5)) + join);
  }
  if (tile) { pick = tile & 255; splits = std::max(1, tile >> 8); }
  switch (pick) {
    case 8: return launch<2, 4, 8, 4, ROWS, MODE>(a, blocks, splits);
    case 7: return launch<2, 4, 7, 4, ROWS, MODE>(a, blocks, splits);
    case 6: return launch<2, 4, 6, 4, ROWS, MODE>(a, blocks, splits);
    case 5: return launch<2, 4, 5, 4, ROWS, MODE>(a, blocks, splits);
    case 4: return launch<2, 4, 4, 4, ROWS, MODE>(a, blocks, splits);
    case 128: return launch<2, 2, 4, 4, ROWS, MODE>(a, blocks, splits);
    default: return launch<2, 2, 2, 2, ROWS, MODE>(a, blocks, splits);
  }
}

__hip_bfloat16* ptr(const at::Tensor& t) { return reinterpret_cast<__hip_bfloat16*>(t.data_ptr()); }

// a matrix whose rows loads and stores of `bytes` can walk
bool walks(const at::Tensor& t, int bytes) {
  return t.is_cuda() && t.dim() == 2 && t.scalar_type() == at::kBFloat16 && t.stride(1) == 1 &&
         t.stride(0) >= t.size(1) && t.stride(0) % (bytes / 2) == 0 && t.stride(0) < (1 << 21) &&
         reinterpret_cast<uintptr_t>(t.data_ptr()) % bytes == 0;
}

// The blocks into args; false for what the kernel does not take.
bool fill(Args& o, const std::vector<const ProductBlock*>& blocks, bool rows) {
  if (blocks.empty() || blocks.size() > BLOCKS || blocks[0]->terms.empty()) return false;
  const int64_t M = blocks[0]->terms[0].a.size(0);
  const auto device = blocks[0]->terms[0].a.device();
  if (M < 1 || M > (1 << 30)) return false;
  o.M = (int)M;
  int n = 0;
  o.steps = -1;
  for (size_t i = 0; i < blocks.size(); ++i) {
    const auto& block = *blocks[i];
    if (block.terms.empty() || block.width < 8 || block.width % 8 || block.width > (1 << 24))
      return false;
    o.width[i] = (int)block.width;
    o.first[i] = n;
    o.terms[i] = (int)block.terms.size();
    int64_t k = 0;
    for (const auto& t : block.terms) {
      if (n == TERMS || !walks(t.a, 16) || t.a.size(0) != M || t.a.device() != device) return false;
      const int64_t deep = t.a.size(1);
      if (deep < BK || deep % BK || deep > (1 << 24) || (!t.b && rows)) return false;
      Term& to = o.term[n++];
      to = {ptr(t.a), nullptr, (int)t.a.stride(0), 0, (int)(deep / BK)};
      if (t.b) {
        if (!walks(*t.b, 16) || t.b->size(rows ? 0 : 1) != deep ||
            t.b->size(rows ? 1 : 0) != block.width || t.b->device() != device)
          return false;
        to.b = ptr(*t.b);
        to.ldb = (int)t.b->stride(0);
      }
      k += deep / BK;
    }
    if (o.steps >= 0 && k != o.steps) return false;
    o.steps = (int)k;
    if (block.bias) {
      const auto& b = *block.bias;
      if (b.device() != device || b.scalar_type() != at::kBFloat16 || b.numel() != block.width ||
          !b.is_contiguous() || reinterpret_cast<uintptr_t>(b.data_ptr()) % 8)
        return false;
      o.bias[i] = ptr(b);
    }
  }
  return true;
}

std::vector<const ProductBlock*> each(const std::vector<ProductBlock>& blocks) {
  std::vector<const ProductBlock*> out;
  for (const auto& b : blocks) out.push_back(&b);
  return out;
}

bool shaped(const at::Tensor& t, int64_t rows, int64_t cols) {
  return walks(t, 8) && t.size(0) == rows && t.size(1) == cols;
}

// Whether what is read lies clear of what is written: a tile in shares of K may be
// joined and written by two workgroups, the second after the first has written.
bool clear_of(const at::Tensor& read, const at::Tensor& written) {
  auto from = [](const at::Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()); };
  auto to = [&](const at::Tensor& t) {
    return from(t) + ((t.size(0) - 1) * t.stride(0) + t.size(1)) * t.element_size();
  };
  return to(read) <= from(written) || to(written) <= from(read);
}

}  // namespace

bool product_takes(const std::vector<ProductBlock>& blocks, bool rows_of_b) {
  Args o{};
  return fill(o, each(blocks), rows_of_b);
}

bool product(const std::vector<ProductBlock>& blocks, bool rows_of_b, const at::Tensor& out,
             const c10::optional<at::Tensor>& res, int tile) {
  Args o{};
  int64_t width = 0;
  for (const auto& b : blocks) width += b.width;
  if (!fill(o, each(blocks), rows_of_b) || !shaped(out, o.M, width) ||
      (res && !(shaped(*res, o.M, width) && clear_of(*res, out))))
    return false;
  o.c = ptr(out);
  o.ldc = (int)out.stride(0);
  if (res) {
    o.res = ptr(*res);
    o.ldr = (int)res->stride(0);
  }
  if (rows_of_b) by_size<true, PLAIN>(o, (int)blocks.size(), tile);
  else by_size<false, PLAIN>(o, (int)blocks.size(), tile);
  return true;
}

bool product_glu(const ProductBlock& gate, const ProductBlock& up,
                 const c10::optional<at::Tensor>& gu, const at::Tensor& act, int tile) {
  Args o{};
  if (!fill(o, {&gate, &up}, false) || gate.width != up.width ||
      gate.terms.size() != up.terms.size() || (gu && !shaped(*gu, o.M, 2 * gate.width)) ||
      !shaped(act, o.M, gate.width))
    return false;
  for (size_t i = 0; i < gate.terms.size(); ++i)
    if (!gate.terms[i].a.is_same(up.terms[i].a)) return false;
  if (gu) {
    o.c = ptr(*gu);
    o.ldc = (int)gu->stride(0);
  }
  o.act = ptr(act);
  o.ldact = (int)act.stride(0);
  by_size<false, GLU>(o, 2, tile);
  return true;
}

bool product_glu_bwd(const ProductBlock& block, const at::Tensor& gu, const at::Tensor& dgate,
                     const at::Tensor& dup, int tile) {
  Args o{};
  if (!fill(o, {&block}, true) || block.bias || !shaped(gu, o.M, 2 * block.width) ||
      !shaped(dgate, o.M, block.width) || !shaped(dup, o.M, block.width) ||
      dgate.stride(0) != dup.stride(0) || !clear_of(gu, dgate) || !clear_of(gu, dup))
    return false;
  o.gu = ptr(gu);
  o.ldgu = (int)gu.stride(0);
  o.dgate = ptr(dgate);
  o.dup = ptr(dup);
  o.ldd = (int)dgate.stride(0);
  by_size<true, GLU_BWD>(o, 1, tile);
  return true;
}

// g w, g (M, V), w (V, N): own products for vocabularies of models in use, else the
// library's. From 32768 words on, 1 to 19200 rows, 896 to 8192 wide, own ones take what the
// library's do or less, within 4 % (2408 x 8192 x 32768 1160 us here, 1119 there; 1200 x 8192
// x 152064 2562, 2579; 19200 x 8192 x 152064 38.7 ms, 38.3; 300 x 4096 x 32768 103 us, 301);
// only 19200 rows of 512 are slower, 842 and 759. Below it either may be the faster: 9000 x
// 512 x 4096, 16384, 32000 79, 240, 417 us here, 44, 183, 372 there, 2400 x 4096 x 24576 437,
// 403, 300 x 1024 x 4096 25, 19; 37 x 512 x 4096, 32000 11, 30 here, 18, 116 there.
at::Tensor product_rows(const at::Tensor& g, const at::Tensor& w) {
  auto out = at::empty({g.size(0), w.size(1)}, g.options());
  if (g.size(0) > 0 && g.size(1) >= 32768 && product({{w.size(1), {{g, w}}, {}}}, true, out)) return out;
  return at::mm(g, w);
}

// The products above from Python, for tests. Whether they were taken.
bool product_py(std::vector<std::vector<at::Tensor>> a,
                std::vector<std::vector<c10::optional<at::Tensor>>> b,
                std::vector<c10::optional<at::Tensor>> bias, std::vector<int64_t> width,
                std::string what, std::vector<at::Tensor> out, c10::optional<at::Tensor> res,
                int64_t tile) {
  std::vector<ProductBlock> blocks;
  for (size_t i = 0; i < a.size(); ++i) {
    blocks.push_back({width.at(i), {}, bias.at(i)});
    for (size_t j = 0; j < a[i].size(); ++j) blocks[i].terms.push_back({a[i][j], b.at(i).at(j)});
  }
  if (what == "glu") return product_glu(blocks.at(0), blocks.at(1), out.at(0), out.at(1), (int)tile);
  if (what == "glu_bwd") {
    TORCH_CHECK(res, "product: [gate | up]");
    return product_glu_bwd(blocks.at(0), *res, out.at(0), out.at(1), (int)tile);
  }
  return product(blocks, what == "rows", out.at(0), res, (int)tile);
}
