// Products of a decode step with some tens of rows: y = x W^T for M <= 160
// rows, W bf16 in tiles, fp32 sums.
//
// Tiles. A tile is 32 rows of W x 16 of K, 1 KB: [K half][row][8 elements], the
// operand of one MFMA 32x32x16 in the order of its lanes; a tile row's K follows
// on, then the next 32 rows. A wave's load of W is then 1 KB on end. From a
// row-major W the same load touches 32 rows 16 B at a time, one cache line a
// lane: gate and up of 18944 x 3584 at 160 rows took 80 us so, 59 from tiles
// (271 MB, 4.6 TB/s), at 32 rows 62 and 47; the library's product and the
// activation 83 and 61. For SiLU*mul a tile holds 16 gate rows and their 16 up
// rows.
//
// A workgroup owns 32 WN columns and all rows; WN waves split the columns and
// two halves of the waves split K. x passes through LDS in tiles of 64 of K,
// fetched into registers up to three steps ahead as W is (a step is ~1 us: what
// HBM needs), XOR-swizzled in 16 B chunks. Products with few columns split K
// over workgroups too: fp32 partial sums, which the kernel that reads the result
// adds up on its way (the residual sum with the norm, the rotation with the cache
// write), so the sums are rounded once. Bound: HBM where W is large, else the
// launch with its first loads.
// W is read past the caches, as no step finds a model's weights there (the last
// level holds 256 MB): 37888 x 3584 at 32 and 128 rows 48.5 and 58.0 -> 43.3 and 53.2
// us (6.3 and 5.1 TB/s), 3584 x 18944 26.8 and 33.7 -> 24.3 and 33.2; 160 rows even.
// 160 rows, GPU time before -> now: 4608 x 3584 24.6 -> 15 us, 3584 x 3584
// 24.6 -> 13, 3584 x 18944 (4-bit product, adapter and join) 70 -> 34.
#include <torch/extension.h>
#include <ATen/cuda/CUDAContext.h>
#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16v8;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

namespace {

enum { PARTS = 0, GLU = 1 };

constexpr int BK = 64;                 // K of a step

// floats of a row of joined sums in LDS: 16 B more than its columns
template <int WN>
constexpr int red_row() { return 32 * WN + 4; }

template <int MT, int WN, int MODE>
__global__ __launch_bounds__(WN * 128, 2)
void stream_gemm_kernel(const __hip_bfloat16* __restrict__ x, const __hip_bfloat16* __restrict__ w,
                        const __hip_bfloat16* __restrict__ w2, __hip_bfloat16* __restrict__ y,
                        float* __restrict__ ws, int M, int N, int N2, int K, int splits) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int RB = BK * 2, TB = 32 * MT * RB, NT = WN * 128, RS = red_row<WN>();
  constexpr int PIECES = MT * 256, PER = (PIECES + NT - 1) / NT;   // 16 B pieces of an x tile
  const int tid = threadIdx.x, l = tid & 63, lr = l & 31, h = l >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wn = wave % WN, wk = wave / WN;
  const int z = blockIdx.x % splits, nb = blockIdx.x / splits;
  const int steps = K / BK, s0 = (int)((int64_t)z * steps / splits),
            s1 = (int)((int64_t)(z + 1) * steps / splits);

  // this wave's tiles of W, past the end the last ones; its half of every step
  const int tile = nb * WN + wn, tiles = MODE == GLU ? N / 16 : N / 32, tiles2 = N2 / 32;
  const __hip_bfloat16* wp = tile < tiles ? w + (int64_t)tile * K * 32
                                          : tiles2 ? w2 + (int64_t)min(tile - tiles, tiles2 - 1) * K * 32
                                          : w + (int64_t)(tiles - 1) * K * 32;
  wp += wk * 2 * 512 + l * 8;
  const __hip_bfloat16* xp[PER];
  int xs[PER];
  #pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int p = min(tid + j * NT, PIECES - 1), row = p >> 3, c = p & 7;
    xp[j] = x + (int64_t)min(row, M - 1) * K + c * 8;
    xs[j] = row * RB + ((c ^ (row & 7)) << 4);
  }

  f32x16 acc[MT];
  #pragma unroll
  for (int t = 0; t < MT; ++t)
    #pragma unroll
    for (int r = 0; r < 16; ++r) acc[t][r] = 0.f;
  u32x4 xv[3][PER];
  bf16v8 wv[3][2];
  // Loads run without branches, so that each wait counts only what it must:
  // steps past the end repeat the last one.
  auto load = [&](int i, int s) {
    const int k = min(s, s1 - 1) * BK;
    #pragma unroll
    for (int j = 0; j < PER; ++j) xv[i][j] = *reinterpret_cast<const u32x4*>(xp[j] + k);
    #pragma unroll
    for (int ks = 0; ks < 2; ++ks)
      wv[i][ks] = __builtin_nontemporal_load(
          reinterpret_cast<const bf16v8*>(wp + (int64_t)k * 32 + ks * 512));
  };
  auto store_x = [&](int i, int buf) {
    #pragma unroll
    for (int j = 0; j < PER; ++j)
      if ((j + 1) * NT <= PIECES || tid + j * NT < PIECES)
        *reinterpret_cast<u32x4*>(smem + buf + xs[j]) = xv[i][j];
  };
  int buf = 0;
  auto step = [&](int i, int s) {
    #pragma unroll
    for (int ks = 0; ks < 2; ++ks)
      #pragma unroll
      for (int t = 0; t < MT; ++t) {
        const bf16v8 xf = *reinterpret_cast<const bf16v8*>(
            smem + buf + (t * 32 + lr) * RB + (((wk * 4 + h + ks * 2) ^ (lr & 7)) << 4));
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wv[i][ks], xf, acc[t], 0, 0, 0);
      }
    buf ^= TB;
    store_x((i + 1) % 3, buf);
    load(i, s + 3);
    __syncthreads();
  };
  load(0, s0);
  load(1, s0 + 1);
  load(2, s0 + 2);
  store_x(0, 0);
  __syncthreads();
  int s = s0;
  for (; s + 2 < s1; s += 3) {
    step(0, s);
    step(1, s + 1);
    step(2, s + 2);
  }
  if (s < s1) step(0, s);
  if (s + 1 < s1) step(1, s + 1);

  // the two halves of K meet in LDS; acc[t]: row m = 32 t + lr of x, columns
  // 8 q + 4 h + 0..3 of the wave's 32
  float* red = reinterpret_cast<float*>(smem);
  if (wk == 1) {
    #pragma unroll
    for (int t = 0; t < MT; ++t)
      #pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<f32x4*>(red + (t * 32 + lr) * RS + wn * 32 + q * 8 + h * 4) =
            f32x4{acc[t][4 * q], acc[t][4 * q + 1], acc[t][4 * q + 2], acc[t][4 * q + 3]};
  }
  __syncthreads();
  if (wk == 0) {
    #pragma unroll
    for (int t = 0; t < MT; ++t)
      #pragma unroll
      for (int q = 0; q < 4; ++q) {
        f32x4* p = reinterpret_cast<f32x4*>(red + (t * 32 + lr) * RS + wn * 32 + q * 8 + h * 4);
        *p += f32x4{acc[t][4 * q], acc[t][4 * q + 1], acc[t][4 * q + 2], acc[t][4 * q + 3]};
      }
  }
  __syncthreads();
  if (MODE == GLU) {
    for (int p = tid; p < M * WN * 2; p += NT) {
      const int m = p / (WN * 2), c = p % (WN * 2), at = m * RS + (c >> 1) * 32 + (c & 1) * 8;
      const int n = nb * WN * 16 + c * 8;
      if (n >= N) continue;
      bf16v8 o;
      #pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float g = red[at + j], u = red[at + 16 + j];
        o[j] = (__bf16)(g / (1.f + __expf(-g)) * u);
      }
      *reinterpret_cast<bf16v8*>(y + (int64_t)m * N + n) = o;
    }
  } else {
    const int ld = N + N2;
    for (int p = tid; p < M * WN * 8; p += NT) {
      const int m = p / (WN * 8), c = p % (WN * 8) * 4, n = nb * WN * 32 + c;
      if (n < ld)
        *reinterpret_cast<f32x4*>(ws + ((int64_t)z * M + m) * ld + n) =
            *reinterpret_cast<const f32x4*>(red + m * RS + c);
    }
  }
}

const __hip_bfloat16* sptr(const torch::Tensor& t) {
  return reinterpret_cast<const __hip_bfloat16*>(t.data_ptr());
}

void check_stream(const torch::Tensor& x, const torch::Tensor& w) {
  TORCH_CHECK(x.is_cuda() && x.dim() == 2 && x.is_contiguous() && x.scalar_type() == at::kBFloat16);
  TORCH_CHECK(w.is_cuda() && w.dim() == 2 && w.is_contiguous() && w.scalar_type() == at::kBFloat16);
  TORCH_CHECK(w.size(1) == x.size(1), "stream_gemm: shape mismatch");
  TORCH_CHECK(reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0, "stream_gemm: W on 16 bytes");
}

// x as 16 B loads can read it
torch::Tensor on16(const torch::Tensor& t) {
  return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0 ? t : t.clone();
}

// Tiles side by side in a workgroup and shares of K. A workgroup's traffic,
// steps x (rows of x and of W) x 128 B, times the workgroups a CU gets, plus
// the partial sums, written and read, at twice their bytes. Within 5 % of the best of
// a sweep at 32 and 160 rows (us): 4608 x 3584 2 tiles/3 shares 15.9, 4/7 14.7;
// 3584 x 3584 2/4 13.0, 4/9 13.4; 3584 x 18944 2/4 43, 3/6 39, 4/9 33.7, 5/11 34.2;
// 2560 x 9728 2/6 19.5, 4/12 17.7; 1536 x 8960 2/10 13.2, 4/21 14.2; gate and
// up of 18944 x 3584 2 tiles 93, 4 95, 5 59 (237 workgroups), of 8960 x 1536 2
// tiles 29.5, 3 21.3, 5 24.9.
struct Cut { int wn, splits; };

Cut cut(int M, int tiles, int K, bool split) {
  Cut best{2, 1};
  double least = 1e30;
  const int steps = K / BK, mt = CDIV(M, 32);
  for (int wn = 2; wn <= 5; ++wn) {
    const int nb = CDIV(tiles, wn);
    const int s = split ? std::max(1, std::min(256 / nb, steps / 3)) : 1;
    const double cost = (double)CDIV(nb * s, 256) * CDIV(steps, s) * (mt + wn) * 32 * 128 +
                        (split ? (double)s * M * tiles * 32 * 16 / 256 : 0.);
    if (cost < least) { least = cost; best = {wn, s}; }
  }
  return best;
}

template <int MODE>
void launch_stream(const torch::Tensor& x, const torch::Tensor& w, const __hip_bfloat16* w2,
                   __hip_bfloat16* y, float* ws, int M, int N, int N2, int K, int wn, int blocks,
                   int splits) {
  auto stream = at::cuda::getCurrentCUDAStream();
  auto go = [&](auto mt_, auto wn_) {
    constexpr int MT = decltype(mt_)::value, WN = decltype(wn_)::value;
    constexpr int smem = std::max(2 * 32 * MT * BK * 2, 32 * MT * red_row<WN>() * 4);
    if (smem > 64 * 1024) {
      static const hipError_t raised = hipFuncSetAttribute(
          reinterpret_cast<const void*>(&stream_gemm_kernel<MT, WN, MODE>),
          hipFuncAttributeMaxDynamicSharedMemorySize, smem);
      TORCH_CHECK(raised == hipSuccess, "stream_gemm: LDS");
    }
    hipLaunchKernelGGL((stream_gemm_kernel<MT, WN, MODE>), dim3(blocks), dim3(WN * 128), smem,
                       stream, sptr(x), sptr(w), w2, y, ws, M, N, N2, K, splits);
  };
  auto by_m = [&](auto wn_) {
    switch (CDIV(M, 32)) {
      case 1: go(std::integral_constant<int, 1>{}, wn_); break;
      case 2: go(std::integral_constant<int, 2>{}, wn_); break;
      case 3: go(std::integral_constant<int, 3>{}, wn_); break;
      case 4: go(std::integral_constant<int, 4>{}, wn_); break;
      default: go(std::integral_constant<int, 5>{}, wn_); break;
    }
  };
  if (wn == 2) by_m(std::integral_constant<int, 2>{});
  else if (wn == 3) by_m(std::integral_constant<int, 3>{});
  else if (wn == 4) by_m(std::integral_constant<int, 4>{});
  else by_m(std::integral_constant<int, 5>{});
  HIP_CHECK_LAST();
}

}  // namespace

// Whether the products below take rows of x, rows of W (for SiLU*mul both
// halves), K. Five row tiles are what fits: 154 of the 168 registers that ten waves
// of a workgroup have each. The library's product is not as fast from there on (7B, us:
// gate, up and activation of 161 rows 88 where 160 take 61 here, down with the sum and
// norm behind it 122 and 46).
bool stream_gemm_takes(int64_t M, int64_t N, int64_t K) {
  return M >= 1 && M <= 160 && N >= 32 && N % 32 == 0 && K >= 64 && K % 64 == 0;
}

// silu(x Wg^T) * (x Wu^T); w (2 F, K) in tiles of 16 gate and 16 up rows
torch::Tensor stream_glu(torch::Tensor x, torch::Tensor w) {
  check_stream(x, w);
  const int M = x.size(0), K = x.size(1), N = w.size(0);
  TORCH_CHECK(stream_gemm_takes(M, N, K), "stream_glu: unsupported shape (", M, ", ", N, ", ", K, ")");
  x = on16(x);
  auto y = torch::empty({M, N / 2}, x.options());
  const Cut c = cut(M, N / 32, K, false);
  launch_stream<GLU>(x, w, nullptr, reinterpret_cast<__hip_bfloat16*>(y.data_ptr()), nullptr, M,
                     N / 2, 0, K, c.wn, CDIV(N / 32, c.wn), 1);
  return y;
}

// x [w; w2]^T as partial sums (shares of K, M, rows of both) fp32; w, w2 in tiles
torch::Tensor stream_gemm(torch::Tensor x, torch::Tensor w, c10::optional<torch::Tensor> w2) {
  check_stream(x, w);
  const int M = x.size(0), K = x.size(1), N = w.size(0);
  TORCH_CHECK(stream_gemm_takes(M, N, K), "stream_gemm: unsupported shape (", M, ", ", N, ", ", K, ")");
  x = on16(x);
  const int N2 = w2 ? (int)w2->size(0) : 0;
  if (w2) {
    check_stream(x, *w2);
    TORCH_CHECK(N2 % 32 == 0, "stream_gemm: rows of w2");
  }
  const int tiles = (N + N2) / 32;
  const Cut c = cut(M, tiles, K, true);
  auto ws = torch::empty({c.splits, M, N + N2}, x.options().dtype(at::kFloat));
  launch_stream<PARTS>(x, w, N2 ? sptr(*w2) : nullptr, nullptr, ws.data_ptr<float>(), M, N, N2, K,
                       c.wn, CDIV(tiles, c.wn) * c.splits, c.splits);
  return ws;
}
