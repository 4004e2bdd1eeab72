// Inputs of LoRA adapters over a micro-batch: u = scale * x A^T beside its x, and
// backward du = scale * dY B, for adapters that share x (side by side) and for
// several dY in one launch.
//
// These products have 32 to 128 columns and only read x or dY. The library took one
// call for each, five forward and seven backward a layer, 17 us of the host's time
// apiece, with another for the concatenation of the A; short micro-batches wait for
// that: a pass of the 0.5B model over 3 x 308 tokens 20.7 -> 17.2 ms. A workgroup
// owns 32 rows and all columns; 128 of K a step pass through LDS, fetched into
// registers up to three steps ahead, and eight waves take 16 of K each, so that few
// workgroups have short chains. B lies with its columns innermost and is read
// transposed (LDS transpose reads). The waves' sums meet in LDS, two and two.
// Bound: HBM for many rows, else the chain of steps. rows x K, columns, the
// library's product against this, us: 900 x 896, 96 20.1 and 7.8; 900 x 4864, 32
// 19.6 and 11.1; 4816 x 8960, 32 20.3 and 19.1 (B 28.6 and 20.3); 18793 x 1536, 32
// 19.2 and 13.4; 18793 x 8960, 32 76.7 and 81.3; 18793 x 1536, 96 19.5 and 28.9.
#include <ATen/cuda/CUDAContext.h>
#include "adapted.h"
#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16v8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16v4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((address_space(3))) bf16v4 lds_bf16v4;

namespace {

constexpr int JOBS = 3, PIECES = 3, NW = 8, NT = NW * 64, BK = NW * 16, RB = BK * 2;

struct Input {
  const __hip_bfloat16 *x, *m[PIECES];
  __hip_bfloat16* out;
  int64_t ldx, ldo;
  float scale[PIECES];
  int first[PIECES + 1];    // columns of each adapter
  int n, K, cols, total;
};

struct Inputs { Input j[JOBS]; };

// The jobs' pointers come out of an array, so the compiler does not see that they
// are global: flat loads would wait on LDS too.
typedef __attribute__((address_space(1))) const u32x4 global_u32x4;
typedef __attribute__((address_space(1))) bf16v4 global_bf16v4;
DEV_INLINE u32x4 load16(const __hip_bfloat16* p) { return *(global_u32x4*)p; }

// 16 B chunk c of row k of a B tile of 32 RT columns: 4 rows over 64 B (transpose
// reads) fall into different banks
template <int RT>
DEV_INLINE int b_chunk(int k, int c) {
  constexpr int W = RT == 3 ? 4 : RT;
  const int swz = RT == 1 ? 0 : RT == 2 ? ((k >> 1) & 1) << 2 : (k & 3) << 2;
  return k * (W * 64) + ((c ^ swz) << 4);
}

// The adapter that column n belongs to. (By index, the job would lie in scratch.)
struct Piece { const __hip_bfloat16* m; float scale; int first, end; };
DEV_INLINE Piece piece(const Input& j, int n) {
  Piece p{j.m[0], j.scale[0], 0, j.first[1]};
  if (j.n > 1 && n >= j.first[1]) p = {j.m[1], j.scale[1], j.first[1], j.first[2]};
  if (j.n > 2 && n >= j.first[2]) p = {j.m[2], j.scale[2], j.first[2], j.first[3]};
  return p;
}

// the waves' sums meet in wave 0, two and two
template <int RT>
DEV_INLINE void join_waves(f32x16 (&acc)[RT], f32x4* red, int wave, int l) {
  #pragma unroll
  for (int half = NW / 2; half > 0; half >>= 1) {
    if (wave >= half && wave < 2 * half) {
      #pragma unroll
      for (int t = 0; t < RT; ++t)
        #pragma unroll
        for (int q = 0; q < 4; ++q)
          red[(((wave - half) * RT + t) * 4 + q) * 64 + l] =
              f32x4{acc[t][4 * q], acc[t][4 * q + 1], acc[t][4 * q + 2], acc[t][4 * q + 3]};
    }
    __syncthreads();
    if (wave < half) {
      #pragma unroll
      for (int t = 0; t < RT; ++t)
        #pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x4 v = red[((wave * RT + t) * 4 + q) * 64 + l];
          #pragma unroll
          for (int i = 0; i < 4; ++i) acc[t][4 * q + i] += v[i];
        }
    }
    __syncthreads();
  }
}

// element column 32 t + l % 32, rows 16 wave + 8 h + 0..7 of a B tile
template <int RT>
DEV_INLINE bf16v8 read_columns(char* p, int t, int wave, int l, int h) {
  const int x = t * 4 + ((l >> 4) & 1) * 2 + ((l & 3) >> 1);
  const int k = wave * 16 + 8 * h + ((l & 15) >> 2), e = (l & 1) * 8;
  const bf16v4 a = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16v4*)(p + b_chunk<RT>(k, x) + e));
  const bf16v4 b = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16v4*)(p + b_chunk<RT>(k + 4, x) + e));
  return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
}

// grid (rows / 32, jobs)
template <int RT, bool KM>
__global__ __launch_bounds__(NT)
void adapter_inputs_kernel(Inputs in, int rows) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int XB = 32 * RB, MB = (KM && RT == 3 ? 4 : RT) * 32 * RB, TB = XB + MB;
  const Input job = in.j[blockIdx.y];
  const int tid = threadIdx.x, l = tid & 63, lr = l & 31, h = l >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row0 = blockIdx.x * 32, K = job.K, steps = (K + BK - 1) / BK;
  const int total = job.total;
  const u32x4 zero = {0, 0, 0, 0};

  // rows of 16 chunks: chunk c of row r at r * 256 + ((c ^ r % 16) << 4)
  const int c = tid & 15, r0 = tid >> 4;
  const __hip_bfloat16* xp = job.x + min(row0 + r0, rows - 1) * job.ldx;
  const int xs = r0 * RB + ((c ^ (r0 & 15)) << 4);
  const __hip_bfloat16* mp[RT];
  int mk[RT], ms[RT];                     // KM: row of the tile; place in it
  bool mok[RT];
  #pragma unroll
  for (int j = 0; j < RT; ++j) {
    if (KM) {
      const int p = tid + j * NT, mc = p % (RT * 4);
      mk[j] = p / (RT * 4);
      mok[j] = mc * 8 < total;
      mp[j] = job.m[0] + min(mc * 8, total - 8);
      ms[j] = b_chunk<RT>(mk[j], mc);
    } else {
      const int n = r0 + j * 32;
      const Piece pc = piece(job, n);
      mok[j] = n < total;
      mp[j] = pc.m + (int64_t)min(n - pc.first, pc.end - pc.first - 1) * K;
      mk[j] = 0;
      ms[j] = n * RB + ((c ^ (n & 15)) << 4);
    }
  }

  f32x16 acc[RT];
  #pragma unroll
  for (int t = 0; t < RT; ++t)
    #pragma unroll
    for (int i = 0; i < 16; ++i) acc[t][i] = 0.f;
  u32x4 xv[3], mv[3][RT];
  // steps past the end repeat the last one; past K both operands are zero
  auto load = [&](int i, int s) {
    const int k0 = min(s, steps - 1) * BK, k = k0 + c * 8;
    xv[i] = load16(xp + min(k, K - 8));
    #pragma unroll
    for (int j = 0; j < RT; ++j)
      mv[i][j] = load16(
          mp[j] + (KM ? (int64_t)min(k0 + mk[j], K - 1) * total : (int64_t)min(k, K - 8)));
  };
  auto store = [&](int i, int s, int buf) {
    const int k0 = min(s, steps - 1) * BK, k = k0 + c * 8;
    *reinterpret_cast<u32x4*>(smem + buf + xs) = k < K ? xv[i] : zero;
    #pragma unroll
    for (int j = 0; j < RT; ++j)
      *reinterpret_cast<u32x4*>(smem + buf + XB + ms[j]) =
          mok[j] && (KM ? k0 + mk[j] : k) < K ? mv[i][j] : zero;
  };
  int buf = 0;
  auto step = [&](int i, int s) {
    load(i, s + 3);
    __builtin_amdgcn_sched_barrier(0);    // not behind the products
    const int at = lr * RB + (((wave * 2 + h) ^ (lr & 15)) << 4);
    const bf16v8 xf = *reinterpret_cast<const bf16v8*>(smem + buf + at);
    #pragma unroll
    for (int t = 0; t < RT; ++t) {
      bf16v8 mf;
      if (KM) {
        mf = read_columns<RT>(smem + buf + XB, t, wave, l, h);
      } else {
        mf = *reinterpret_cast<const bf16v8*>(smem + buf + XB + t * 32 * RB + at);
      }
      acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(mf, xf, acc[t], 0, 0, 0);
    }
    buf ^= TB;
    store((i + 1) % 3, s + 1, buf);
    __syncthreads();
  };
  load(0, 0);
  load(1, 1);
  load(2, 2);
  store(0, 0, 0);
  __syncthreads();
  int s = 0;
  for (; s + 2 < steps; s += 3) {
    step(0, s);
    step(1, s + 1);
    step(2, s + 2);
  }
  if (s < steps) step(0, s);
  if (s + 1 < steps) step(1, s + 1);

  join_waves<RT>(acc, reinterpret_cast<f32x4*>(smem), wave, l);
  // row l % 32 of x, columns 8 q + 4 h + 0..3 of the tile
  const int row = row0 + lr;
  if (wave > 0 || row >= rows) return;
  #pragma unroll
  for (int t = 0; t < RT; ++t)
    #pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int n = t * 32 + 8 * q + 4 * h;
      if (n >= job.cols) continue;
      const float scale = piece(job, n).scale;
      bf16v4 o;
      #pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = (__bf16)(acc[t][4 * q + r] * scale);
      *(global_bf16v4*)(job.out + row * job.ldo + n) = o;
    }
}

// ------------------------------------------------------------ activation
// The activation, or its gradients, with the adapter inputs of what it writes: from
// [gate | up] (and dact) 128 columns a step to x[0] (and x[1]) in memory and LDS. On its own
// the product reads again what the activation has just written. 18793 rows of 8960
// columns, us, forward 183 and 110 -> 222 (4.5 TB/s), backward 305 and 153 -> 384; bound
// by memory. A workgroup owns 32 rows: below some 8192 the chip is not full.
struct Activation {
  const __hip_bfloat16 *dact, *gu, *m[2];
  __hip_bfloat16 *x[2], *out;
  int64_t ldx, ldo;
  float scale[2];
  int F, r[2], cols;
};

typedef __attribute__((address_space(1))) u32x4 global_out16;

template <int RT, bool BWD>
__global__ __launch_bounds__(NT)
void activation_inputs_kernel(Activation job, int rows) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int P = BWD ? 2 : 1;          // products
  constexpr int XB = 32 * RB, MB = RT * 32 * RB, TB = P * (XB + MB);
  const int tid = threadIdx.x, l = tid & 63, lr = l & 31, h = l >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row0 = blockIdx.x * 32, F = job.F, steps = (F + BK - 1) / BK;
  const u32x4 zero = {0, 0, 0, 0};

  // rows of 16 chunks: chunk c of row r at r * 256 + ((c ^ r % 16) << 4)
  const int c = tid & 15, r0 = tid >> 4;
  const int64_t row = min(row0 + r0, rows - 1);
  const bool live = row0 + r0 < rows;
  const __hip_bfloat16 *gp = job.gu + row * 2 * F, *dp = BWD ? job.dact + row * F : nullptr;
  const int xs = r0 * RB + ((c ^ (r0 & 15)) << 4);
  const __hip_bfloat16* mp[P][RT];
  int mk[RT], ms[RT];
  bool mok[P][RT];
  #pragma unroll
  for (int j = 0; j < RT; ++j) {
    if (BWD) {
      const int p = tid + j * NT, mc = p % (RT * 4);
      mk[j] = p / (RT * 4);
      ms[j] = b_chunk<RT>(mk[j], mc);
      #pragma unroll
      for (int i = 0; i < P; ++i) {
        mok[i][j] = mc * 8 < job.r[i];
        mp[i][j] = job.m[i] + min(mc * 8, job.r[i] - 8);
      }
    } else {
      const int n = r0 + j * 32;
      mk[j] = 0;
      ms[j] = n * RB + ((c ^ (n & 15)) << 4);
      mok[0][j] = n < job.r[0];
      mp[0][j] = job.m[0] + (int64_t)min(n, job.r[0] - 1) * F;
    }
  }
  f32x16 acc[P][RT];
  #pragma unroll
  for (int i = 0; i < P; ++i)
    #pragma unroll
    for (int t = 0; t < RT; ++t)
      #pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][t][e] = 0.f;
  u32x4 gv[3], uv[3], dv[3], mv[3][P][RT];
  // steps past the end repeat the last one; past F both operands are zero
  auto load = [&](int i, int s) {
    const int k0 = min(s, steps - 1) * BK, k = min(k0 + c * 8, F - 8);
    gv[i] = load16(gp + k);
    uv[i] = load16(gp + F + k);
    if (BWD) dv[i] = load16(dp + k);
    #pragma unroll
    for (int p = 0; p < P; ++p)
      #pragma unroll
      for (int j = 0; j < RT; ++j)
        mv[i][p][j] = load16(mp[p][j] + (BWD ? (int64_t)min(k0 + mk[j], F - 1) * job.r[p] : (int64_t)k));
  };
  auto store = [&](int i, int s, int buf) {
    const int k0 = min(s, steps - 1) * BK, k = k0 + c * 8;
    const bf16v8 g = __builtin_bit_cast(bf16v8, gv[i]), u = __builtin_bit_cast(bf16v8, uv[i]);
    bf16v8 x[P];
    #pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float v = (float)g[e];
      if (BWD) {
        const float d = (float)__builtin_bit_cast(bf16v8, dv[i])[e], sig = 1.f / (1.f + __expf(-v));
        x[0][e] = (__bf16)(d * (float)u[e] * sig * (1.f + v * (1.f - sig)));
        x[P - 1][e] = (__bf16)(d * (v * sig));
      } else {
        x[0][e] = (__bf16)(v / (1.f + __expf(-v)) * (float)u[e]);
      }
    }
    #pragma unroll
    for (int p = 0; p < P; ++p) {
      const u32x4 w = __builtin_bit_cast(u32x4, x[p]);
      char* to = smem + buf + p * (XB + MB);
      *reinterpret_cast<u32x4*>(to + xs) = k < F ? w : zero;
      if (live && k < F && s < steps) *(global_out16*)(job.x[p] + row * job.ldx + k) = w;
      #pragma unroll
      for (int j = 0; j < RT; ++j)
        *reinterpret_cast<u32x4*>(to + XB + ms[j]) =
            mok[p][j] && (BWD ? k0 + mk[j] : k) < F ? mv[i][p][j] : zero;
    }
  };
  int buf = 0;
  auto step = [&](int i, int s) {
    load(i, s + 3);
    __builtin_amdgcn_sched_barrier(0);    // not behind the products
    const int at = lr * RB + (((wave * 2 + h) ^ (lr & 15)) << 4);
    #pragma unroll
    for (int p = 0; p < P; ++p) {
      char* from = smem + buf + p * (XB + MB);
      const bf16v8 xf = *reinterpret_cast<const bf16v8*>(from + at);
      #pragma unroll
      for (int t = 0; t < RT; ++t) {
        bf16v8 mf;
        if (BWD) mf = read_columns<RT>(from + XB, t, wave, l, h);
        else mf = *reinterpret_cast<const bf16v8*>(from + XB + t * 32 * RB + at);
        acc[p][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(mf, xf, acc[p][t], 0, 0, 0);
      }
    }
    buf ^= TB;
    store((i + 1) % 3, s + 1, buf);
    __syncthreads();
  };
  load(0, 0);
  load(1, 1);
  load(2, 2);
  store(0, 0, 0);
  __syncthreads();
  int s = 0;
  for (; s + 2 < steps; s += 3) {
    step(0, s);
    step(1, s + 1);
    step(2, s + 2);
  }
  if (s < steps) step(0, s);
  if (s + 1 < steps) step(1, s + 1);

  #pragma unroll
  for (int p = 0; p < P; ++p) {
    join_waves<RT>(acc[p], reinterpret_cast<f32x4*>(smem), wave, l);
    if (wave > 0 || row0 + lr >= rows) continue;
    // row l % 32 of x, columns 8 q + 4 h + 0..3 of the tile; the last product's with
    // the spare columns behind it
    const int first = p ? job.r[0] : 0, end = p + 1 < P ? job.r[0] : job.cols;
    #pragma unroll
    for (int t = 0; t < RT; ++t)
      #pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int n = first + t * 32 + 8 * q + 4 * h;
        if (n >= end) continue;
        bf16v4 o;
        #pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = (__bf16)(acc[p][t][4 * q + e] * job.scale[p]);
        *(global_bf16v4*)(job.out + (row0 + lr) * job.ldo + n) = o;
      }
  }
}

const __hip_bfloat16* iptr(const torch::Tensor& t) {
  return reinterpret_cast<const __hip_bfloat16*>(t.data_ptr());
}

// rows that accesses of so many bytes can walk
bool walks(const torch::Tensor& t, int bytes) {
  return t.is_cuda() && t.dim() == 2 && t.scalar_type() == at::kBFloat16 && t.stride(1) == 1 &&
         t.stride(0) * 2 % bytes == 0 && reinterpret_cast<uintptr_t>(t.data_ptr()) % bytes == 0;
}

template <int RT, bool KM>
void launch_inputs(const Inputs& in, int jobs, int rows) {
  constexpr int tiles = 2 * (1 + (KM && RT == 3 ? 4 : RT)) * 32 * RB;
  constexpr int smem = std::max(tiles, NW / 2 * RT * 4096);
  if (smem > 64 * 1024) {
    static const hipError_t raised = hipFuncSetAttribute(
        reinterpret_cast<const void*>(&adapter_inputs_kernel<RT, KM>),
        hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    TORCH_CHECK(raised == hipSuccess, "adapter_inputs: LDS");
  }
  hipLaunchKernelGGL((adapter_inputs_kernel<RT, KM>), dim3(CDIV(rows, 32), jobs), dim3(NT),
                     smem, at::cuda::getCurrentCUDAStream(), in, rows);
}

}  // namespace

bool adapter_inputs(const std::vector<AdapterInput>& jobs, bool k_major) {
  Inputs in{};
  if (jobs.empty() || jobs.size() > JOBS) return false;
  const int64_t rows = jobs[0].x.size(0);
  int most = 0;
  for (size_t i = 0; i < jobs.size(); ++i) {
    const auto& j = jobs[i];
    Input& o = in.j[i];
    if (!walks(j.x, 16) || !walks(j.out, 8) || j.m.empty() || j.m.size() > (k_major ? 1 : PIECES) ||
        j.scales.size() != j.m.size())
      return false;
    const int64_t K = j.x.size(1);
    if (K < 8 || K % 8 != 0 || K > INT32_MAX / 2 || j.x.size(0) != rows || j.out.size(0) != rows)
      return false;
    o.n = j.m.size();
    for (int p = 0; p < o.n; ++p) {
      const auto& m = j.m[p];
      if (!walks(m, 16) || !m.is_contiguous()) return false;
      const int64_t r = m.size(k_major ? 1 : 0);
      if (r < 8 || r % 8 != 0 || r > 128 || m.size(k_major ? 0 : 1) != K) return false;
      o.m[p] = iptr(m);
      o.first[p + 1] = o.first[p] + (int)r;
      o.scale[p] = (float)j.scales[p];
    }
    // columns are written by fours
    if (j.out.size(1) < o.first[o.n] || j.out.size(1) > 128 || j.out.size(1) % 4 != 0) return false;
    if (rows > 1 && j.out.stride(0) < j.out.size(1)) return false;   // rows over one another
    o.cols = (int)j.out.size(1);
    o.total = o.first[o.n];
    most = std::max(most, o.cols);
    o.x = iptr(j.x);
    o.out = reinterpret_cast<__hip_bfloat16*>(j.out.data_ptr());
    o.ldx = j.x.stride(0);
    o.ldo = j.out.stride(0);
    o.K = (int)K;
  }
  if (rows > INT32_MAX - 64) return false;
  if (rows == 0) return true;
  auto go = [&](auto rt, auto km) {
    constexpr int RT = decltype(rt)::value;
    constexpr bool KM = decltype(km)::value;
    launch_inputs<RT, KM>(in, jobs.size(), rows);
  };
  auto by_cols = [&](auto km) {
    if (most <= 32) go(std::integral_constant<int, 1>{}, km);
    else if (most <= 64) go(std::integral_constant<int, 2>{}, km);
    else if (most <= 96) go(std::integral_constant<int, 3>{}, km);
    else go(std::integral_constant<int, 4>{}, km);
  };
  if (k_major) by_cols(std::true_type{});
  else by_cols(std::false_type{});
  HIP_CHECK_LAST();
  return true;
}

namespace {

template <bool BWD>
bool activation_inputs(Activation& o, const torch::Tensor& gu, const torch::Tensor* dact,
                       const std::vector<torch::Tensor>& x, const std::vector<torch::Tensor>& m,
                       const std::vector<double>& scales, const torch::Tensor& out) {
  constexpr int P = BWD ? 2 : 1;
  const int64_t rows = gu.size(0), F = gu.size(1) / 2;
  if (!walks(gu, 16) || !gu.is_contiguous() || gu.size(1) != 2 * F || F < 8 || F % 8 != 0 ||
      F > INT32_MAX / 4 || rows < 1 || rows > INT32_MAX - 64 || !walks(out, 8) || out.size(0) != rows ||
      (rows > 1 && out.stride(0) < out.size(1)))
    return false;
  if (BWD && (!walks(*dact, 16) || !dact->is_contiguous() || dact->size(0) != rows || dact->size(1) != F))
    return false;
  int most = 0, sum = 0;
  for (int p = 0; p < P; ++p) {
    const int64_t r = m[p].size(BWD ? 1 : 0);
    if (!walks(m[p], 16) || !m[p].is_contiguous() || m[p].size(BWD ? 0 : 1) != F || r < 8 || r % 8 != 0 ||
        r > 64 || !walks(x[p], 16) || x[p].size(0) != rows || x[p].size(1) != F ||
        x[p].stride(0) != x[0].stride(0) || x[p].stride(0) < F)
      return false;
    o.m[p] = iptr(m[p]);
    o.x[p] = reinterpret_cast<__hip_bfloat16*>(x[p].data_ptr());
    o.scale[p] = (float)scales[p];
    o.r[p] = (int)r;
    most = std::max(most, (int)r);
    sum += (int)r;
  }
  o.cols = (int)out.size(1);
  // spare columns are the last product's, whose tiles must reach them
  most = std::max(most, o.cols - sum + o.r[P - 1]);
  if (o.cols < sum || o.cols % 4 != 0 || most > 64) return false;
  o.gu = iptr(gu);
  o.dact = BWD ? iptr(*dact) : nullptr;
  o.out = reinterpret_cast<__hip_bfloat16*>(out.data_ptr());
  o.ldx = x[0].stride(0);
  o.ldo = out.stride(0);
  o.F = (int)F;
  auto go = [&](auto rt) {
    constexpr int RT = decltype(rt)::value;
    constexpr int smem = std::max(2 * P * (1 + RT) * 32 * RB, NW / 2 * RT * 4096);
    if (smem > 64 * 1024) {
      static const hipError_t raised = hipFuncSetAttribute(
          reinterpret_cast<const void*>(&activation_inputs_kernel<RT, BWD>),
          hipFuncAttributeMaxDynamicSharedMemorySize, smem);
      TORCH_CHECK(raised == hipSuccess, "activation_inputs: LDS");
    }
    hipLaunchKernelGGL((activation_inputs_kernel<RT, BWD>), dim3(CDIV(rows, 32)), dim3(NT), smem,
                       at::cuda::getCurrentCUDAStream(), o, (int)rows);
  };
  if (most <= 32) go(std::integral_constant<int, 1>{});
  else go(std::integral_constant<int, 2>{});
  HIP_CHECK_LAST();
  return true;
}

}  // namespace

bool silu_mul_inputs(torch::Tensor gu, torch::Tensor act, torch::Tensor m, double scale,
                     torch::Tensor out) {
  Activation o{};
  return activation_inputs<false>(o, gu, nullptr, {act}, {m}, {scale}, out);
}

bool silu_mul_bwd_inputs(torch::Tensor dact, torch::Tensor gu, torch::Tensor dgate,
                         torch::Tensor dup, std::vector<torch::Tensor> m,
                         std::vector<double> scales, torch::Tensor out) {
  Activation o{};
  return m.size() == 2 && scales.size() == 2 &&
         activation_inputs<true>(o, gu, &dact, {dgate, dup}, m, scales, out);
}

// One job for tests and other callers: out <- x m scaled
bool adapter_input(torch::Tensor x, std::vector<torch::Tensor> m, std::vector<double> scales,
                   torch::Tensor out, bool k_major) {
  return adapter_inputs({{x, out, m, scales}}, k_major);
}
