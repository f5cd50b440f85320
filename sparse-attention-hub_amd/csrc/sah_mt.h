// MT19937 (Matsumoto & Nishimura, ACM TOMACS 8, 1998), the generator behind torch's CPU random numbers, by one
// workgroup: what a seeded torch.Generator draws can be drawn where it is used, instead of on the host and copied over.
// The next 624 words depend on the 624 before them in three runs (227, 227, 170 words), each complete before the next
// starts: three barriers a block, 0.3 us.
#ifndef SAH_MT_H
#define SAH_MT_H
#include "sah_common.h"

#define MT_N 624
#define MT_M 397

struct mt_lds {
  uint32_t st[2][MT_N];
};

// state of a freshly seeded generator into S.st[0]; every thread of the workgroup calls, a barrier is passed
__device__ __forceinline__ void mt_seed(mt_lds& S, uint32_t seed) {
  if (threadIdx.x == 0) {
    uint32_t x = seed;
    S.st[0][0] = x;
    for (int i = 1; i < MT_N; ++i) {
      x = 1812433253u * (x ^ (x >> 30)) + (uint32_t)i;
      S.st[0][i] = x;
    }
  }
  __syncthreads();
}

// the block after S.st[from] into S.st[from ^ 1]: at least 227 threads, every thread of the workgroup calls; the new block
// is complete (a barrier passed) on return
__device__ __forceinline__ void mt_next(mt_lds& S, int from) {
  const uint32_t* o = S.st[from];
  uint32_t* w = S.st[from ^ 1];
  const int tid = threadIdx.x;
  constexpr int RUN = MT_N - MT_M;
  auto mix = [](uint32_t a, uint32_t b, uint32_t m) {
    const uint32_t y = (a & 0x80000000u) | (b & 0x7fffffffu);
    return m ^ (y >> 1) ^ ((y & 1u) ? 0x9908b0dfu : 0u);
  };
  if (tid < RUN) w[tid] = mix(o[tid], o[tid + 1], o[tid + MT_M]);
  __syncthreads();
  if (tid < RUN) w[tid + RUN] = mix(o[tid + RUN], o[tid + RUN + 1], w[tid]);
  __syncthreads();
  if (tid < MT_N - 2 * RUN) {
    const int i = tid + 2 * RUN;
    w[i] = mix(o[i], i + 1 < MT_N ? o[i + 1] : w[0], w[i - RUN]);
  }
  __syncthreads();
}

__device__ __forceinline__ uint32_t mt_temper(uint32_t y) {
  y ^= y >> 11;
  y ^= (y << 7) & 0x9d2c5680u;
  y ^= (y << 15) & 0xefc60000u;
  return y ^ (y >> 18);
}
#endif
