// Common device helpers for the distrl_llm_amd gfx950 kernel library.
// CDNA4-native: wave64, bf16x8 vector loads, LDS + cross-lane reductions.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>
#include <atomic>
#include <cstdint>
#include <random>

#define WAVE 64
#define DEV_INLINE __device__ __forceinline__

// 16-byte vector of 8 bf16 values (coalescing sweet spot: 16 B/lane).
struct alignas(16) bf16x8 { __hip_bfloat16 v[8]; };
struct alignas(16) f32x4v { float v[4]; };

DEV_INLINE float bf2f(__hip_bfloat16 x) { return __bfloat162float(x); }
DEV_INLINE __hip_bfloat16 f2bf(float x) { return __float2bfloat16(x); }

// ---- cross-lane reductions (wave64) ----
DEV_INLINE float wave_sum(float x) {
  #pragma unroll
  for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, WAVE);
  return x;
}
DEV_INLINE float wave_max(float x) {
  #pragma unroll
  for (int off = 32; off > 0; off >>= 1) x = fmaxf(x, __shfl_xor(x, off, WAVE));
  return x;
}

// Block reduction through LDS; `red` must have >= blockDim.x/WAVE slots.
DEV_INLINE float block_sum(float x, float* red) {
  const int lane = threadIdx.x & (WAVE - 1);
  const int wid = threadIdx.x / WAVE;
  const int nw = blockDim.x / WAVE;
  x = wave_sum(x);
  if (lane == 0) red[wid] = x;
  __syncthreads();
  float r = (threadIdx.x < nw) ? red[threadIdx.x] : 0.f;
  if (wid == 0) {
    #pragma unroll
    for (int off = 32; off > 0; off >>= 1) r += __shfl_xor(r, off, WAVE);
    if (lane == 0) red[0] = r;
  }
  __syncthreads();
  float out = red[0];
  __syncthreads();
  return out;
}

DEV_INLINE float block_max(float x, float* red) {
  const int lane = threadIdx.x & (WAVE - 1);
  const int wid = threadIdx.x / WAVE;
  const int nw = blockDim.x / WAVE;
  x = wave_max(x);
  if (lane == 0) red[wid] = x;
  __syncthreads();
  float r = (threadIdx.x < nw) ? red[threadIdx.x] : -1e30f;
  if (wid == 0) {
    #pragma unroll
    for (int off = 32; off > 0; off >>= 1) r = fmaxf(r, __shfl_xor(r, off, WAVE));
    if (lane == 0) red[0] = r;
  }
  __syncthreads();
  float out = red[0];
  __syncthreads();
  return out;
}

// ---- partial sums ----
// v[0..7] += 8 elements of n arrays `step` elements apart, four of them in
// flight at a time
DEV_INLINE void add_parts8(float (&v)[8], const float* p, int64_t step, int n) {
  for (int z = 0; z < n; z += 4) {
    f32x4v a[4], b[4];
    #pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float* q = p + min(z + i, n - 1) * step;
      a[i] = *reinterpret_cast<const f32x4v*>(q);
      b[i] = *reinterpret_cast<const f32x4v*>(q + 4);
    }
    #pragma unroll
    for (int i = 0; i < 4; ++i)
      if (z + i < n) {
        #pragma unroll
        for (int j = 0; j < 4; ++j) { v[j] += a[i].v[j]; v[4 + j] += b[i].v[j]; }
      }
  }
}

// the same for two runs of eight, d elements apart
DEV_INLINE void add_parts8x2(float (&v)[8], float (&w)[8], const float* p, int64_t d, int64_t step,
                             int n) {
  for (int z = 0; z < n; z += 4) {
    f32x4v a[4][4];
    #pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float* q = p + min(z + i, n - 1) * step;
      a[i][0] = *reinterpret_cast<const f32x4v*>(q);
      a[i][1] = *reinterpret_cast<const f32x4v*>(q + 4);
      a[i][2] = *reinterpret_cast<const f32x4v*>(q + d);
      a[i][3] = *reinterpret_cast<const f32x4v*>(q + d + 4);
    }
    #pragma unroll
    for (int i = 0; i < 4; ++i)
      if (z + i < n) {
        #pragma unroll
        for (int j = 0; j < 4; ++j) {
          v[j] += a[i][0].v[j];
          v[4 + j] += a[i][1].v[j];
          w[j] += a[i][2].v[j];
          w[4 + j] += a[i][3].v[j];
        }
      }
  }
}

// ---- hash (counter-based random numbers) ----
DEV_INLINE uint64_t splitmix64(uint64_t x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}

// ---- arrival of workgroups ----
// A mark that no other launch of this process has; neither half is zero.
inline unsigned long long arrival_tag() {
  static std::atomic<unsigned long long> calls{(unsigned long long)std::random_device{}() << 32};
  unsigned long long x = ++calls * 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  return (x ^ (x >> 31)) | 0x100000001ull;
}

// What workgroups of one launch pass to each other goes past the caches of their XCDs,
// so that a wait is all it takes to order it: a fence, which writes a whole L2 back and
// empties it, took 50 us of 1184 workgroups that drew a token and 9 without.
template <typename T>
DEV_INLINE void store_through(T* p, T x) {
  __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
DEV_INLINE T load_through(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// two floats on 8 bytes
DEV_INLINE void store_pair(float* p, float x, float y) {
  store_through(reinterpret_cast<unsigned long long*>(p),
                (unsigned long long)__float_as_uint(y) << 32 | __float_as_uint(x));
}
DEV_INLINE float2 load_pair(const float* p) {
  const unsigned long long v = load_through(reinterpret_cast<const unsigned long long*>(p));
  return {__uint_as_float((uint32_t)v), __uint_as_float((uint32_t)(v >> 32))};
}
// Until this wave's stores and atomics have arrived.
DEV_INLINE void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// For one whole wave of workgroup `mine` of n, whose own stores_done are behind it:
// leaves the launch's mark in its place and says whether all n marks are there, so
// that what the n stored through before may be joined. Of the n workgroups the last to come sees all of them; another may too, and
// then does the same join. Nothing has to be cleared beforehand, as no place holds the
// mark by chance; a replay of a captured launch has the same mark, so those who saw
// all of them take them away.
DEV_INLINE bool all_there(unsigned long long* there, int n, int mine, unsigned long long tag) {
  const int lane = threadIdx.x & (WAVE - 1);
  if (lane == 0) atomicExch(there + mine, tag);
  stores_done();
  bool all = true;
  for (int i = lane; i < n; i += WAVE) all = all && atomicAdd(there + i, 0ull) == tag;
  if (__ballot(!all) != 0) return false;
  stores_done();
  for (int i = lane; i < n; i += WAVE) there[i] = 0ull;
  return true;
}

#define HIP_CHECK_LAST()                                                     \
  do {                                                                       \
    hipError_t e = hipGetLastError();                                        \
    TORCH_CHECK(e == hipSuccess, "HIP kernel launch failed: ",               \
                hipGetErrorString(e));                                       \
  } while (0)

#define CDIV(a, b) (((a) + (b) - 1) / (b))
