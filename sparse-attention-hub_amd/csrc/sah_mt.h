// MT19937 (Matsumoto & Nishimura, ACM TOMACS 8, 1998), the generator behind torch's CPU random numbers, by one
// workgroup: what a seeded torch.Generator draws can be drawn where it is used, instead of on the host and copied over.
// mt_next: the next 624 words depend on the 624 before them in three runs (227, 227, 170 words), each complete before the
// next starts: three barriers a block, 0.6 us. mt_stream: whole sequences, 454 words a barrier.
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

// one step of the recurrence's linear part: x[k + 624] = x[k + 397] ^ mt_mix(x[k], x[k + 1])
__device__ __forceinline__ uint32_t mt_mix(uint32_t a, uint32_t b) {
  const uint32_t y = (a & 0x80000000u) | (b & 0x7fffffffu);
  return (y >> 1) ^ ((0u - (y & 1u)) & 0x9908b0dfu);
}

// The generator's state after seeding, for a kernel argument: a serial chain of 624 steps, 1 us on the host, 10 on the device.
struct mt_state {
  uint32_t w[MT_N];
};
static inline mt_state mt_seeded(uint32_t seed) {
  mt_state s;
  s.w[0] = seed;
  for (uint32_t i = 1; i < MT_N; ++i) s.w[i] = 1812433253u * (s.w[i - 1] ^ (s.w[i - 1] >> 30)) + i;
  return s;
}

// The words 0 .. total - 1 (not yet tempered) that the generator yields, by one workgroup of MTS_NT threads. Applied to itself the
// recurrence reads x[k + 1248] = x[k + 794] ^ mix(mix(x[k], x[k + 1]), mix(x[k + 1], x[k + 2])) (mix is linear over bits, the
// terms that come twice cancel): 454 words depend on earlier ones alone, so that two words of the plain form's 227 come at
// each barrier. consume(word, first, count, t): word(i) is word `first + i`, i < count; called with t = 0 .. 255 by the four
// waves that do not generate, while the others make the next 454. 65536 words, a start vector drawn from every two: 54 us; 78
// with mt_next, the seeding on the device and the drawing in turn. What bounds it: the way from LDS to LDS through a barrier,
// 0.3 us of 144.
#define MTS_GEN 512                 // threads that generate
#define MTS_USE 256                 // threads that use
#define MTS_NT (MTS_GEN + MTS_USE)
#define MTS_RING 2048
#define MTS_STEP (2 * (MT_N - MT_M))  // words per barrier: 454
struct mts_lds {
  uint32_t x[MTS_RING];
};
template <typename F>
__device__ __forceinline__ void mt_stream(mts_lds& S, const mt_state& seeded, int64_t total, F&& consume) {
  const int tid = threadIdx.x;
  auto at = [&](uint32_t i) -> uint32_t& { return S.x[i & (MTS_RING - 1)]; };  // i: 624 more than the word's number
  if (tid < MT_N) S.x[tid] = seeded.w[tid];
  __syncthreads();
  for (int run = MT_N; run < 2 * MT_N; run += MT_N - MT_M) {
    if (tid < MT_N - MT_M && run + tid < 2 * MT_N) at(run + tid) = at(run + tid - (MT_N - MT_M)) ^ mt_mix(at(run + tid - MT_N), at(run + tid - MT_N + 1));
    __syncthreads();
  }
  int64_t done = 0, made = MT_N;  // words handed over; words there
  while (done < total) {          // uniform
    if (tid < MTS_GEN) {
      if (tid < MTS_STEP && made < total) {
        const uint32_t i = (uint32_t)made + MT_N + tid;
        const uint32_t a = at(i - 2 * MT_N), b = at(i - 2 * MT_N + 1), c = at(i - 2 * MT_N + 2);
        at(i) = at(i - MTS_STEP) ^ mt_mix(mt_mix(a, b), mt_mix(b, c));
      }
    } else {
      const int64_t count = (made < total ? made : total) - done;
      const uint32_t from = (uint32_t)done + MT_N;
      consume([&](int i) -> uint32_t { return at(from + i); }, done, (int)count, tid - MTS_GEN);
    }
    done = made;
    made += MTS_STEP;
    __syncthreads();
  }
}

__device__ __forceinline__ uint32_t mt_temper(uint32_t y) {
  y ^= y >> 11;
  y ^= (y << 7) & 0x9d2c5680u;
  y ^= (y << 15) & 0xefc60000u;
  return y ^ (y >> 18);
}
#endif
