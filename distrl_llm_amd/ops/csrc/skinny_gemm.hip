// Products of a decode step with few rows: y = x W^T for M <= 32 rows,
// W (N, K) bf16, fp32 sums, with what stands around the product in the same
// launch: the RMS norm of x before it; bias, residual sum or SiLU*mul after it.
//
// Such a product only streams W. A workgroup owns 16 rows of W (for SiLU*mul 16
// gate rows and their 16 up rows) and its waves split K, so that small matrices
// spread over the chip (few rows of W: 8 a workgroup); a wave has up to ten steps of its share of W and x in
// flight, straight into MFMA operands (16x16x32: lane = row, 16 B pieces).
// Partial sums meet in LDS. The norm needs no pass of its own: the waves
// multiply x by the norm weight as they read it and sum its squares on the way,
// 1/rms scales the finished row.
// Tiles of W are read past the caches where these (256 MB) hold no model's weights from
// one step to the next, which the caller knows. At one row, us: 19456 x 2560 22.3 ->
// 21.3, 2560 x 9728 13.6 -> 12.7; but 9728 x 896 from the caches 5.6, past them 6.3. From
// rows a load is half a cache line of each, whose other half has to stay: 35.9 past
// the caches, 29.3 through them.
// A step of a few sequences is bound by its launches' latency (~4 us each) as
// much as by bytes, hence the fusions: on the 0.5B model at 8 rows a layer took
// 67 us in 11 launches, 39 in 7 now (gate|up + SiLU 17 + 5 -> 11.6 us, down and
// output 8.3 and 6.8 -> 8.8 and 4.6 with the residual sum, qkv 6.8 -> 4.9; the two
// norms' 4.8 each are in them).
#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>
#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16v8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16v4;
typedef __attribute__((ext_vector_type(4))) float f32x4;

namespace {

enum { PLAIN = 0, RESIDUAL = 1, GLU = 2 };
enum { ROWS = 0, TILES = 1, KEPT = 2 };     // W, KEPT: tiles that the caches hold

// Steps of K a wave has in flight: what its registers hold.
template <int MT, int KW, int ACC, bool NORM>
constexpr int in_flight() {
  const int n = 96 / (4 * (ACC + MT + (NORM ? 1 : 0)));
  return n > 10 ? 10 : n;
}

template <int MT, int KW, int MODE, bool NORM, int W>
__global__ __launch_bounds__(KW * 64)
void skinny_gemm_kernel(const __hip_bfloat16* __restrict__ x, const __hip_bfloat16* __restrict__ w,
                        const __hip_bfloat16* __restrict__ bias,
                        const __hip_bfloat16* __restrict__ res,
                        const __hip_bfloat16* __restrict__ norm_w,
                        const __hip_bfloat16* __restrict__ u,    // (M, R): y += u ub^T
                        const __hip_bfloat16* __restrict__ ub,   // (N, R)
                        __hip_bfloat16* __restrict__ y, int M, int N, int K, int R, int tr, float eps) {
  constexpr int ACC = MODE == GLU ? 2 : 1, U = in_flight<MT, KW, ACC, NORM>();
  extern __shared__ __attribute__((aligned(16))) char smem[];
  f32x4* red = reinterpret_cast<f32x4*>(smem);            // [KW][ACC][MT][64]
  __shared__ float squares[NORM ? KW * MT * 16 : 1];      // of x, [KW][MT][16 rows]
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = threadIdx.x & 63, g = l >> 4, lr = l & 15;
  const int n0 = blockIdx.x * tr, wr = min(lr, tr - 1);   // spare rows repeat
  const int steps = K / 32, s0 = wave * steps / KW, s1 = (wave + 1) * steps / KW;

  const __hip_bfloat16* wp[ACC];
  #pragma unroll
  for (int a = 0; a < ACC; ++a) {
    if (W != ROWS) {
      // row of the tile; SiLU*mul: 16 gate and 16 up rows
      const int n = MODE == GLU ? (n0 + wr) / 16 * 32 + a * 16 + (n0 + wr) % 16 : n0 + wr;
      wp[a] = w + (int64_t)(n >> 5) * K * 32 + (g >> 1) * 512 + (g & 1) * 256 + (n & 31) * 8;
    } else {
      wp[a] = w + (int64_t)(n0 + a * N + wr) * K + g * 8;
    }
  }
  f32x4 acc[ACC][MT];
  #pragma unroll
  for (int a = 0; a < ACC; ++a)
    #pragma unroll
    for (int t = 0; t < MT; ++t) acc[a][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  int row[MT];
  float ss[MT];
  #pragma unroll
  for (int t = 0; t < MT; ++t) {
    row[t] = min(t * 16 + lr, M - 1);                     // spare rows repeat
    ss[t] = 0.f;
  }

  for (int s = s0; s < s1; s += U) {
    bf16v8 wf[U][ACC], xf[U][MT], nf[U];
    #pragma unroll
    for (int i = 0; i < U; ++i) {
      const int k = min(s + i, s1 - 1) * 32;              // past the end: the last again
      #pragma unroll
      for (int a = 0; a < ACC; ++a) {
        const bf16v8* from = reinterpret_cast<const bf16v8*>(wp[a] + k * (W == ROWS ? 1 : 32));
        wf[i][a] = W == TILES ? __builtin_nontemporal_load(from) : *from;
      }
      #pragma unroll
      for (int t = 0; t < MT; ++t)
        xf[i][t] = *reinterpret_cast<const bf16v8*>(x + (int64_t)row[t] * K + k + g * 8);
      if (NORM) nf[i] = *reinterpret_cast<const bf16v8*>(norm_w + k + g * 8);
    }
    #pragma unroll
    for (int i = 0; i < U; ++i)
      if (s + i < s1) {                                   // wave-uniform
        #pragma unroll
        for (int t = 0; t < MT; ++t) {
          if (NORM) {
            #pragma unroll
            for (int j = 0; j < 8; ++j) {
              const float v = (float)xf[i][t][j];
              ss[t] += v * v;
              xf[i][t][j] = (__bf16)(v * (float)nf[i][j]);
            }
          }
          #pragma unroll
          for (int a = 0; a < ACC; ++a)
            acc[a][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[i][a], xf[i][t], acc[a][t],
                                                                0, 0, 0);
        }
      }
  }
  if (NORM) {
    #pragma unroll
    for (int t = 0; t < MT; ++t) {
      ss[t] += __shfl_xor(ss[t], 16, WAVE);
      ss[t] += __shfl_xor(ss[t], 32, WAVE);
      if (g == 0) squares[(wave * MT + t) * 16 + lr] = ss[t];
    }
  }
  if (MODE == RESIDUAL && wave == 0) {      // an adapter: more of K, elsewhere
    for (int k = g * 8; k < R; k += 32) {
      const bf16v8 b = *reinterpret_cast<const bf16v8*>(ub + (int64_t)(n0 + wr) * R + k);
      #pragma unroll
      for (int t = 0; t < MT; ++t)
        acc[0][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            b, *reinterpret_cast<const bf16v8*>(u + (int64_t)row[t] * R + k), acc[0][t], 0, 0, 0);
    }
  }

  #pragma unroll
  for (int a = 0; a < ACC; ++a)
    #pragma unroll
    for (int t = 0; t < MT; ++t) red[((wave * ACC + a) * MT + t) * 64 + l] = acc[a][t];
  __syncthreads();
  // lane of tile t: row m = 16 t + lr of x, columns n0 + 4 g + 0..3
  for (int t = wave; t < MT; t += KW) {
    const int m = t * 16 + lr, n = n0 + g * 4;
    f32x4 sum[ACC];
    #pragma unroll
    for (int a = 0; a < ACC; ++a) {
      sum[a] = red[(a * MT + t) * 64 + l];
      #pragma unroll
      for (int v = 1; v < KW; ++v) sum[a] += red[((v * ACC + a) * MT + t) * 64 + l];
    }
    if (NORM) {
      float sq = 0.f;
      #pragma unroll
      for (int v = 0; v < KW; ++v) sq += squares[(v * MT + t) * 16 + lr];
      const float r = rsqrtf(sq / K + eps);
      #pragma unroll
      for (int a = 0; a < ACC; ++a) sum[a] *= r;
    }
    if (m >= M || g * 4 >= tr) continue;
    const int64_t at = (int64_t)m * N + n;
    bf16v4 o;
    if (MODE == GLU) {
      #pragma unroll
      for (int r = 0; r < 4; ++r) {
        // gate and up round as the separate product's output does
        const float gt = (float)(__bf16)sum[0][r], up = (float)(__bf16)sum[ACC - 1][r];
        o[r] = (__bf16)(gt / (1.f + __expf(-gt)) * up);
      }
    } else {
      bf16v4 add;
      if (MODE == RESIDUAL) add = *reinterpret_cast<const bf16v4*>(res + at);
      else if (bias) add = *reinterpret_cast<const bf16v4*>(bias + n);
      #pragma unroll
      for (int r = 0; r < 4; ++r)
        o[r] = (__bf16)(MODE == RESIDUAL || bias ? sum[0][r] + (float)add[r] : sum[0][r]);
    }
    *reinterpret_cast<bf16v4*>(y + at) = o;
  }
}

// The same for M <= 8 rows of x. Such an x fills half of a product's 16
// columns, and loads that repeat it (or 8 rows of W) cost as much of a CU's 64 B/clk as
// others do, which bound the small products. Here a product's rows are 8 of W at two
// steps of K, and its columns 8 of x at the same two: the blocks on the diagonal are the
// two steps' sums, the others are left. Every lane loads something of its own, whole
// cache lines of either, and the norm's work is halved; its squares are a product too.
// Bound by the launch (1.7 us of a captured chain), the way to memory and back, and W.
// 8 rows and cold weights in a captured chain, us, before -> now: 1152 x 896 with the norm
// 3.95 -> 3.4, 896 x 896 3.5 -> 3.1, gate and up of 4864 x 896 8.4 -> 6.6, 896 x 4864 7.1 ->
// 6.1; 2048 x 1536 5.2 -> 4.2, 1536 x 1536 4.6 -> 3.7, 8960 x 1536 13.5 -> 12.5, 1536 x 8960
// 13.2 -> 11.4; 6144 x 2560 12.9 -> 10.2, 2560 x 4096 9.5 -> 7.5, 9728 x 2560 23.1 -> 19.5,
// 2560 x 9728 17.9 -> 14.3; 3584 x 18944 32.7 -> 26.7, 18944 x 3584 55 -> 47.
struct PairArgs {
  const __hip_bfloat16 *x, *w, *bias, *res, *norm_w, *u, *ub;
  __hip_bfloat16* y;
  int M, N, K, R;
  float eps;
};

// NG groups of 8 rows of W a workgroup, U double steps of K a wave has in flight
template <int NG, int KW, int U, int MODE, int W>
__global__ __launch_bounds__(KW * 64)
void skinny_pair_kernel(const PairArgs p) {
  constexpr bool NORM = MODE != RESIDUAL;
  constexpr int ACC = MODE == GLU ? 2 : 1, OUT = NG / ACC, TR = OUT * 8;
  constexpr int QUADS = OUT * 16, PARTS = WAVE / QUADS;   // four columns of a row; lanes that share one
  __shared__ f32x4 red[KW][NG][32];
  __shared__ float squares[NORM ? KW * 16 : 1];
  const int M = p.M, N = p.N, K = p.K, R = p.R;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = threadIdx.x & 63, g = l >> 4, r8 = l & 7, second = (l >> 3) & 1;
  const int n0 = blockIdx.x * TR, ko = second * 32 + g * 8;
  const int steps = K / 64, s0 = wave * steps / KW, s1 = (wave + 1) * steps / KW;

  const __hip_bfloat16* wp[NG];
  #pragma unroll
  for (int a = 0; a < NG; ++a) {
    const int n = n0 + a % OUT * 8 + r8, t = MODE == GLU ? n / 16 * 32 + a / OUT * 16 + n % 16 : n;
    wp[a] = W == ROWS ? p.w + (int64_t)(a / OUT * N + n) * K + ko
                      : p.w + (int64_t)(t >> 5) * K * 32 + (ko >> 4) * 512 + ((ko >> 3) & 1) * 256 +
                            (t & 31) * 8;
  }
  const __hip_bfloat16* xp = p.x + (int64_t)min(r8, M - 1) * K + ko;    // spare rows repeat
  f32x4 acc[NG];
  #pragma unroll
  for (int a = 0; a < NG; ++a) acc[a] = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 sq = f32x4{0.f, 0.f, 0.f, 0.f};     // x x^T: rows' squares on its diagonal
  // of this lane's output, for the end
  const int m = l & 7, n = n0 + (l % QUADS) / 16 * 8 + ((l >> 3) & 1) * 4;
  const int64_t at = (int64_t)min(m, M - 1) * N + n;
  bf16v4 add = {};
  if (wave == 0) {
    if (MODE == RESIDUAL) add = *reinterpret_cast<const bf16v4*>(p.res + at);
    else if (MODE == PLAIN && p.bias) add = *reinterpret_cast<const bf16v4*>(p.bias + n);
  }

  for (int s = s0; s < s1; s += U) {
    bf16v8 wf[U][NG], xf[U], nf[U];
    #pragma unroll
    for (int i = 0; i < U; ++i) {
      const int k = min(s + i, s1 - 1) * 64;              // past the end: the last again
      #pragma unroll
      for (int a = 0; a < NG; ++a) {
        const bf16v8* from = reinterpret_cast<const bf16v8*>(wp[a] + k * (W == ROWS ? 1 : 32));
        wf[i][a] = W == TILES ? __builtin_nontemporal_load(from) : *from;
      }
      xf[i] = *reinterpret_cast<const bf16v8*>(xp + k);
      if (NORM) nf[i] = *reinterpret_cast<const bf16v8*>(p.norm_w + ko + k);
    }
    #pragma unroll
    for (int i = 0; i < U; ++i)
      if (s + i < s1) {                                   // wave-uniform
        if (NORM) {
          sq = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[i], xf[i], sq, 0, 0, 0);
          #pragma unroll
          for (int j = 0; j < 8; ++j) xf[i][j] = (__bf16)((float)xf[i][j] * (float)nf[i][j]);
        }
        #pragma unroll
        for (int a = 0; a < NG; ++a)
          acc[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[i][a], xf[i], acc[a], 0, 0, 0);
      }
  }
  if (NORM) {
    #pragma unroll
    for (int r = 0; r < 4; ++r)
      if ((l & 15) == 4 * g + r) squares[wave * 16 + (l & 15)] = sq[r];
  }
  if (MODE == RESIDUAL && wave == 0) {      // an adapter: more of K, elsewhere
    for (int k0 = 0; k0 < R; k0 += 64) {
      const int k = k0 + ko;
      const bool there = k < R;             // an odd number of steps: zeros
      const bf16v8 v = there ? *reinterpret_cast<const bf16v8*>(p.u + (int64_t)min(r8, M - 1) * R + k)
                             : bf16v8{};
      #pragma unroll
      for (int a = 0; a < NG; ++a) {
        const bf16v8 b = there ? *reinterpret_cast<const bf16v8*>(
                                     p.ub + (int64_t)(n0 + a * 8 + r8) * R + k)
                               : bf16v8{};
        acc[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, v, acc[a], 0, 0, 0);
      }
    }
  }
  // the diagonal: lanes whose four rows and whose column are of the same step
  if ((g >> 1) == second) {
    #pragma unroll
    for (int a = 0; a < NG; ++a) red[wave][a][second * 16 + (g & 1) * 8 + r8] = acc[a];
  }
  __syncthreads();
  if (wave != 0) return;
  f32x4 sum[ACC];
  const int quad = l % QUADS, part = l / QUADS;
  #pragma unroll
  for (int c = 0; c < ACC; ++c) {
    sum[c] = f32x4{0.f, 0.f, 0.f, 0.f};
    #pragma unroll
    for (int i = 0; i < 2 * KW / PARTS; ++i) {
      const int v = i * PARTS + part;
      sum[c] += red[v >> 1][c * OUT + quad / 16][(v & 1) * 16 + quad % 16];
    }
    #pragma unroll
    for (int off = QUADS; off < WAVE; off <<= 1)
      #pragma unroll
      for (int r = 0; r < 4; ++r) sum[c][r] += __shfl_xor(sum[c][r], off, WAVE);
  }
  if (NORM) {
    float ss = 0.f;
    #pragma unroll
    for (int v = 0; v < 2 * KW; ++v) ss += squares[v * 8 + m];
    const float r = rsqrtf(ss / K + p.eps);
    #pragma unroll
    for (int c = 0; c < ACC; ++c) sum[c] *= r;
  }
  if (m >= M || part) return;
  bf16v4 o;
  #pragma unroll
  for (int r = 0; r < 4; ++r) {
    if (MODE == GLU) {
      // gate and up round as the separate product's output does
      const float gt = (float)(__bf16)sum[0][r], up = (float)(__bf16)sum[ACC - 1][r];
      o[r] = (__bf16)(gt / (1.f + __expf(-gt)) * up);
    } else {
      o[r] = (__bf16)(MODE == RESIDUAL || p.bias ? sum[0][r] + (float)add[r] : sum[0][r]);
    }
  }
  *reinterpret_cast<bf16v4*>(p.y + at) = o;
}

template <int MODE, int NG, int KW, int U>
void launch_pair(const PairArgs& p, int kind) {
  const dim3 grid(p.N / (NG / (MODE == GLU ? 2 : 1) * 8));
  auto stream = at::cuda::getCurrentCUDAStream();
  auto go = [&](auto w_) {
    hipLaunchKernelGGL((skinny_pair_kernel<NG, KW, U, MODE, decltype(w_)::value>), grid, dim3(KW * 64),
                       0, stream, p);
  };
  if (kind == ROWS) go(std::integral_constant<int, ROWS>{});
  else if (kind == KEPT) go(std::integral_constant<int, KEPT>{});
  else go(std::integral_constant<int, TILES>{});
}

// Rows of W a workgroup, waves and double steps in flight, from a sweep of them at 8 rows
// and cold weights (us; rows, waves, in flight: their best). What is on its way passes
// a CU's 32 KB of cache: where workgroups are many fewer steps are faster, few ones need
// a wave's whole share at once. N 896 K 896 3.03 with 8/16/1 (8/8/2 3.38, 16/8/2 4.26);
// 896 x 4864 6.12 8/8/10 (8/8/5 6.41, 16/8/10 9.5); 1536 x 8960 11.4 8/8/9; 2560 x 9728
// 14.25 16/8/5 (16/8/10 14.84, 8/8/10 21.1); 3584 x 18944 26.7 16/8/5; 6144 x 2560 10.2
// 16/8/5 (8/8/5 12.6); SiLU*mul of N 4864 K 896 6.4 8/8/2 (16/8/2 7.95), 8960 x 1536 12.5
// 16/8/2 (16/8/3 14.8), 9728 x 2560 19.5 16/8/2 (16/8/5 22.1), 18944 x 3584 46.9 16/8/4.
template <int MODE>
void pair(const PairArgs& p, int kind) {
  constexpr int ACC = MODE == GLU ? 2 : 1;
  const int steps = p.K / 64, share = CDIV(steps, 8);
  const bool narrow = p.N <= 2048 || (MODE == GLU && steps <= 16);
  // a wave's share in even rounds of at most so many steps
  const int most = narrow ? 10 : MODE != GLU ? 5 : share <= 6 ? 2 : 4;
  const int u = CDIV(share, CDIV(share, most));
  if (!narrow) {
    if (u <= 2) launch_pair<MODE, 2 * ACC, 8, 2>(p, kind);
    else if (u == 3) launch_pair<MODE, 2 * ACC, 8, 3>(p, kind);
    else if (MODE == GLU || u == 4) launch_pair<MODE, 2 * ACC, 8, 4>(p, kind);
    else launch_pair<MODE, 2 * ACC, 8, MODE == GLU ? 4 : 5>(p, kind);
  } else if (MODE == GLU ? u <= 2 : steps <= 16) {
    launch_pair<MODE, ACC, MODE == GLU ? 8 : 16, MODE == GLU ? 2 : 1>(p, kind);
  } else if (u <= 3) {                      // 2 only where steps <= 16
    launch_pair<MODE, ACC, 8, 3>(p, kind);
  } else if (u <= 5) {
    launch_pair<MODE, ACC, 8, 5>(p, kind);
  } else if (u <= 7) {
    launch_pair<MODE, ACC, 8, 7>(p, kind);
  } else if (u <= 9) {
    launch_pair<MODE, ACC, 8, 9>(p, kind);
  } else {
    launch_pair<MODE, ACC, 8, 10>(p, kind);
  }
}

// An operand as 16 B loads can read it: a parameter cut out of a larger buffer
// may start anywhere.
torch::Tensor at16(const torch::Tensor& t) {
  return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0 ? t : t.clone();
}

const __hip_bfloat16* ptr(const torch::Tensor& t) {
  return reinterpret_cast<const __hip_bfloat16*>(t.data_ptr());
}

}  // namespace

// Whether skinny_gemm takes the shape: rows of x, columns of y (the activation's
// for SiLU*mul), K.
bool skinny_gemm_takes(int64_t M, int64_t N, int64_t K) {
  return M >= 1 && M <= 32 && N >= 16 && N % 16 == 0 && K >= 512 && K % 32 == 0;
}

// mode 0: x W^T (+ bias); 1: res + x W^T (+ u ub^T); 2: silu(x Wg^T) * (x Wu^T)
// with w = [Wg; Wu]. norm_w: x is RMS-normed first. tiles: w lies in tiles; kept: and
// stays in the caches from one call to the next.
torch::Tensor skinny_gemm(torch::Tensor x, torch::Tensor w, int64_t mode,
                          c10::optional<torch::Tensor> bias, c10::optional<torch::Tensor> res,
                          c10::optional<torch::Tensor> norm_w, double eps,
                          c10::optional<torch::Tensor> u, c10::optional<torch::Tensor> ub,
                          bool tiles, bool kept) {
  TORCH_CHECK(x.is_cuda() && x.dim() == 2 && x.is_contiguous());
  TORCH_CHECK(w.is_cuda() && w.dim() == 2 && w.is_contiguous());
  TORCH_CHECK(x.scalar_type() == at::kBFloat16 && w.scalar_type() == at::kBFloat16);
  TORCH_CHECK(mode >= PLAIN && mode <= GLU && w.size(1) == x.size(1));
  const int M = x.size(0), K = x.size(1), N = mode == GLU ? w.size(0) / 2 : w.size(0);
  TORCH_CHECK(mode != GLU || w.size(0) % 2 == 0);
  TORCH_CHECK(skinny_gemm_takes(M, N, K), "skinny_gemm: unsupported shape (", M, ", ", N, ", ", K, ")");
  TORCH_CHECK(!tiles || w.size(0) % 32 == 0, "skinny_gemm: rows of W in tiles");
  x = at16(x);
  w = at16(w);
  auto check = [&](c10::optional<torch::Tensor>& t, int64_t n, const char* what) {
    if (!t) return (const __hip_bfloat16*)nullptr;
    TORCH_CHECK(t->is_cuda() && t->is_contiguous() && t->scalar_type() == at::kBFloat16 &&
                t->numel() == n, "skinny_gemm: ", what);
    t = at16(*t);
    return ptr(*t);
  };
  const auto* b = check(bias, N, "bias");
  const auto* r = check(res, (int64_t)M * N, "residual");
  const auto* nw = check(norm_w, K, "norm weight");
  const int R = u ? (int)u->size(-1) : 0;
  TORCH_CHECK(u.has_value() == ub.has_value() && (!u || (mode == RESIDUAL && R % 32 == 0)),
              "skinny_gemm: adapter");
  const auto* up = check(u, (int64_t)M * R, "adapter input");
  const auto* ubp = check(ub, (int64_t)N * R, "adapter weight");
  TORCH_CHECK((mode == RESIDUAL) == (r != nullptr) && (b == nullptr || mode == PLAIN));
  auto y = torch::empty({M, N}, x.options());
  auto* o = reinterpret_cast<__hip_bfloat16*>(y.data_ptr());
  auto stream = at::cuda::getCurrentCUDAStream();
  TORCH_CHECK(mode != RESIDUAL || !nw, "skinny_gemm: norm with a residual sum");
  const int kind = !tiles ? ROWS : kept ? KEPT : TILES;
  // As a step of few sequences calls them; without a norm only adapters of 32 rows are
  // multiplied, which wait for the launch. A row's sums over K are of another order here
  // than below: its product is the same bits beside up to 7 other rows, and beside 8 to 15,
  // but not on either side of that line (as on either side of the lines to other kernels).
  if (M <= 8 && K % 64 == 0 && (nw != nullptr) == (mode != RESIDUAL)) {
    const PairArgs args{ptr(x), ptr(w), b, r, nw, up, ubp, o, M, N, K, R, (float)eps};
    if (mode == PLAIN) pair<PLAIN>(args, kind);
    else if (mode == RESIDUAL) pair<RESIDUAL>(args, kind);
    else pair<GLU>(args, kind);
    HIP_CHECK_LAST();
    return y;
  }
  // Rows of W a workgroup takes and waves that share its K, for 9 to 32 rows of x (and
  // fewer where K is no multiple of 64). The lines are those of sweeps at 8 rows and cold
  // weights, which this kernel took too then (us; rows/waves): N 896, K 4864: 16/4 11.8,
  // 16/16 10.6, 8/16 8.6, 4/16 7.8; N 1536, K 8960: 19.4, 19.6, 15.3, 24.0;
  // N 2560, K 9728: 22.7, 20.3, 28.0; N 1152, K 896: 4.6 (8/4 4.3, 8/16 8.0);
  // N 1536, K 1536: 7.1 (8/4 6.3, 8/8 5.7); SiLU*mul of N 8960, K 1536: 16/4
  // 20.6, 16/8 18.1; N 9728, K 2560: 36, 33; N 4864, K 896: 11.4, 11.5.
  // Fewer rows a workgroup reach more CUs but re-read x; more waves shorten
  // the chain of loads until joining them costs more.
  const int nt = N / 16, steps = K / 32, tr = nt <= 128 ? 8 : 16;
  const int kw = nt <= 256 ? (steps >= 64 ? 16 : steps >= 32 ? 8 : 4)
                        : (mode == GLU && steps >= 48 ? 8 : 4);
  auto launch = [&](auto mt_, auto kw_, auto mode_, auto norm_, auto w_) {
    constexpr int MT = decltype(mt_)::value, KW = decltype(kw_)::value,
                  MODE = decltype(mode_)::value;
    constexpr bool NORM = decltype(norm_)::value;
    const size_t smem = KW * (MODE == GLU ? 2 : 1) * MT * 64 * 16;
    hipLaunchKernelGGL((skinny_gemm_kernel<MT, KW, MODE, NORM, decltype(w_)::value>), dim3(N / tr),
                       dim3(KW * 64), smem, stream, ptr(x), ptr(w), b, r, nw, up, ubp, o, M, N, K, R, tr, (float)eps);
  };
  auto go = [&](auto mt_, auto kw_, auto mode_, auto norm_) {
    if (kind == ROWS) launch(mt_, kw_, mode_, norm_, std::integral_constant<int, ROWS>{});
    else if (kind == KEPT) launch(mt_, kw_, mode_, norm_, std::integral_constant<int, KEPT>{});
    else launch(mt_, kw_, mode_, norm_, std::integral_constant<int, TILES>{});
  };
  auto by_norm = [&](auto mt_, auto kw_, auto mode_) {
    if (nw) go(mt_, kw_, mode_, std::true_type{}); else go(mt_, kw_, mode_, std::false_type{});
  };
  auto by_mode = [&](auto mt_, auto kw_) {
    if (mode == PLAIN) by_norm(mt_, kw_, std::integral_constant<int, PLAIN>{});
    else if (mode == RESIDUAL) go(mt_, kw_, std::integral_constant<int, RESIDUAL>{}, std::false_type{});
    else by_norm(mt_, kw_, std::integral_constant<int, GLU>{});
  };
  auto by_kw = [&](auto mt_) {
    if (kw == 16) by_mode(mt_, std::integral_constant<int, 16>{});
    else if (kw == 8) by_mode(mt_, std::integral_constant<int, 8>{});
    else by_mode(mt_, std::integral_constant<int, 4>{});
  };
  if (M <= 16) by_kw(std::integral_constant<int, 1>{});
  else by_kw(std::integral_constant<int, 2>{});
  HIP_CHECK_LAST();
  return y;
}
