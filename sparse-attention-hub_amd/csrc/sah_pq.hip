// PQCache kernels: batched Lloyd iteration (assignment + centre update) over
// the sub-vectors of the key cache, quantisation of newly appended keys, and
// asymmetric-distance (ADC) scoring through an LDS-resident lookup table.
//
// A group g = (b*Hkv + hk)*n_sub + s is one sub-space of one KV head. The
// assignment kernel keeps the group's centres (n_cent x d_sub fp32, <= 16 KB) in
// LDS, one thread per key, and accumulates the per-centre sums in LDS before a
// single flush of global atomics per workgroup, so no (b, n, k, d) tensor ever
// exists. Blocks are ordered sub-space-fastest so the n_sub workgroups that read
// different 16 B slices of the same key rows run next to each other and share
// the rows in L2.
#include "sah_common.h"
#include "sah_mt.h"

#define PQ_NT 256
#define PQ_MAX_D 17  // widest sub-vector of the kernels that keep a key in registers: 16 plus the extra coordinate of
                     // inner-product search done as L2 search; wider sub-vectors (up to PQM_MAX_D) take the matrix-core
                     // assignment and the one-centre-per-thread quantisation
#define PQ_MAX_CENT 256
#define PQ_TILES 8  // key tiles of PQ_NT per workgroup

// Per-centre sums of the Lloyd update are kept in 64-bit fixed point, so that their value does not depend on the
// order in which threads and workgroups add to them (floating-point atomics would make two runs on the same keys
// differ in a centroid's last bits). The scale is a power of two picked from the largest |key element|:
// |x| * scale < 2^41, which leaves room for 2^20 keys per centre and costs nothing in precision (a float has 24
// significant bits).
__device__ __forceinline__ float pq_sum_scale(uint32_t absmax_bits) {
  const float m = sah_bits_to_float(absmax_bits);
  if (!(m > 0.f) || !(m < INFINITY)) return 1.f;
  int e;
  frexpf(m, &e);  // m = f * 2^e, f in [0.5, 1)
  int sh = 40 - e;
  sh = sh < -100 ? -100 : (sh > 100 ? 100 : sh);
  return ldexpf(1.0f, sh);
}
__device__ __forceinline__ void pq_sum_add(long long* p, float x, float scale) {
  atomicAdd((unsigned long long*)p, (unsigned long long)__float2ll_rn(x * scale));
}
// The same for keys that are all finite, in three instructions: x * scale is exact in fp64 and below 2^51, so adding
// 1.5 * 2^52 rounds it to the nearest integer, ties to even, in the low bits of the sum.
__device__ __forceinline__ void pq_sum_add_finite(long long* p, float x, double scale) {
  const double m = 6755399441055744.0;
  atomicAdd((unsigned long long*)p, __builtin_bit_cast(unsigned long long, fma((double)x, scale, m)) - __builtin_bit_cast(unsigned long long, m));
}

struct pq_assign_params {
  const void* k; int64_t ks_b, ks_h, ks_l;
  int Hkv, n_sub, d_sub, n_cent;
  int key_offset, n_keys;
  const float* centres;
  uint8_t* codes; int64_t code_pitch, code_offset;
  long long* sums; int* counts;
  const uint32_t* absmax_bits;
  int round_dist;
  const int* skip_flag;
};

template <int DT>
__global__ __launch_bounds__(PQ_NT) void k_pq_assign(pq_assign_params P) {
  __shared__ float s_c[PQ_MAX_CENT * PQ_MAX_D];
  __shared__ long long s_sum[PQ_MAX_CENT * PQ_MAX_D];
  __shared__ int s_cnt[PQ_MAX_CENT];
  if (P.skip_flag && *P.skip_flag) return;
  const float sum_scale = P.sums ? pq_sum_scale(*P.absmax_bits) : 1.f;
  const int tid = threadIdx.x;
  const int s = blockIdx.x % P.n_sub;
  const int tg = blockIdx.x / P.n_sub;
  const int bh = blockIdx.y;  // b*Hkv + hk
  const int hk = bh % P.Hkv;
  const int b = bh / P.Hkv;
  const int g = bh * P.n_sub + s;
  const int d_sub = P.d_sub, n_cent = P.n_cent;
  const int cd = n_cent * d_sub;

  for (int i = tid; i < cd; i += PQ_NT) {
    s_c[i] = P.centres[(int64_t)g * cd + i];
    s_sum[i] = 0;
  }
  for (int i = tid; i < n_cent; i += PQ_NT) s_cnt[i] = 0;
  __syncthreads();

  const int64_t kbase = (int64_t)b * P.ks_b + (int64_t)hk * P.ks_h + (int64_t)s * d_sub;
  for (int t = 0; t < PQ_TILES; ++t) {
    const int n = (tg * PQ_TILES + t) * PQ_NT + tid;
    if (n >= P.n_keys) continue;
    float x[PQ_MAX_D];
    const int64_t off = kbase + (int64_t)(P.key_offset + n) * P.ks_l;
#pragma unroll
    for (int d = 0; d < PQ_MAX_D; ++d) x[d] = (d < d_sub) ? sah_load<DT>(P.k, off + d) : 0.f;
    int best = 0;
    float bd = INFINITY;
    for (int c = 0; c < n_cent; ++c) {
      const float* cc = s_c + c * d_sub;
      float dist = 0.f;
      if (P.round_dist) {
#pragma unroll
        for (int d = 0; d < PQ_MAX_D; ++d) {
          if (d < d_sub) {
            const float df = sah_round<DT>(x[d] - cc[d]);
            dist += sah_round<DT>(df * df);
          }
        }
        dist = sah_round<DT>(dist);
      } else {
#pragma unroll
        for (int d = 0; d < PQ_MAX_D; ++d) {
          if (d < d_sub) {
            const float df = x[d] - cc[d];
            dist = fmaf(df, df, dist);
          }
        }
      }
      if (dist < bd) {
        bd = dist;
        best = c;
      }
    }
    P.codes[(((int64_t)bh * P.code_pitch) + P.code_offset + n) * P.n_sub + s] = (uint8_t)best;
    if (P.sums) {
#pragma unroll
      for (int d = 0; d < PQ_MAX_D; ++d)
        if (d < d_sub) pq_sum_add(&s_sum[best * d_sub + d], x[d], sum_scale);
      atomicAdd(&s_cnt[best], 1);
    }
  }
  if (!P.sums) return;
  __syncthreads();
  for (int c = tid; c < n_cent; c += PQ_NT) {
    const int cn = s_cnt[c];
    if (cn) {
      atomicAdd(&P.counts[(int64_t)g * n_cent + c], cn);
      for (int d = 0; d < d_sub; ++d)
        atomicAdd((unsigned long long*)&P.sums[(int64_t)g * cd + c * d_sub + d], (unsigned long long)s_sum[c * d_sub + d]);
    }
  }
}

// Quantisation of a handful of keys (a decode step appends one): the work of one key and sub-space is a
// 256-way argmin, so the centres take the threads - one centre per thread, read straight from memory - and
// the keys take the grid. Same distances, same order of operations and the same lowest-index rule as the
// one-thread-per-key kernel above.
template <int DT>
__global__ __launch_bounds__(PQ_NT) void k_pq_assign_few(pq_assign_params P) {
  sah_touch_kernargs<sizeof(pq_assign_params)>();
  __shared__ float s_d[PQ_NT / SAH_WAVE];
  __shared__ int s_i[PQ_NT / SAH_WAVE];
  const int tid = threadIdx.x;
  const int lane = tid & (SAH_WAVE - 1);
  const int wave = sah_wave_id();
  const int s = blockIdx.x;
  const int bh = blockIdx.y;
  const int n = blockIdx.z;
  const int hk = bh % P.Hkv;
  const int b = bh / P.Hkv;
  const int g = bh * P.n_sub + s;
  const int d_sub = P.d_sub, n_cent = P.n_cent;
  const int64_t off = (int64_t)b * P.ks_b + (int64_t)hk * P.ks_h + (int64_t)s * d_sub + (int64_t)(P.key_offset + n) * P.ks_l;
  float dist = INFINITY;
  int best = 0x7fffffff;
  for (int c = tid; c < n_cent; c += PQ_NT) {
    const float* cc = P.centres + ((int64_t)g * n_cent + c) * d_sub;
    float dd = 0.f;
    if (P.round_dist) {
      for (int d = 0; d < d_sub; ++d) {
        const float df = sah_round<DT>(sah_load<DT>(P.k, off + d) - cc[d]);
        dd += sah_round<DT>(df * df);
      }
      dd = sah_round<DT>(dd);
    } else {
      for (int d = 0; d < d_sub; ++d) {
        const float df = sah_load<DT>(P.k, off + d) - cc[d];
        dd = fmaf(df, df, dd);
      }
    }
    if (dd < dist) {  // c ascends: the first minimum is kept
      dist = dd;
      best = c;
    }
  }
  // smallest distance, lowest centre among equals
#pragma unroll
  for (int o = 1; o < SAH_WAVE; o <<= 1) {
    const float od = __shfl_xor(dist, o);
    const int oi = __shfl_xor(best, o);
    if (od < dist || (od == dist && oi < best)) {
      dist = od;
      best = oi;
    }
  }
  if (lane == 0) {
    s_d[wave] = dist;
    s_i[wave] = best;
  }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < PQ_NT / SAH_WAVE; ++w) {
      if (s_d[w] < dist || (s_d[w] == dist && s_i[w] < best)) {
        dist = s_d[w];
        best = s_i[w];
      }
    }
    P.codes[(((int64_t)bh * P.code_pitch) + P.code_offset + n) * P.n_sub + s] = (uint8_t)best;
  }
}

// A block of new keys (up to a few hundred) against frozen centres: one workgroup per (sub-space, batch x KV head)
// stages the group's centres in LDS once; a wave takes every 4th key, its lanes share the centres out
// (lane, lane + 64, ...), and the argmin of a key is a wave reduction: no workgroup barrier per key. Same
// arithmetic per (key, centre) pair as k_pq_assign_few, same "first minimum" rule.
#define PQB_NT 1024
template <int DT>
__global__ __launch_bounds__(PQB_NT) void k_pq_assign_block(pq_assign_params P) {
  sah_touch_kernargs<sizeof(pq_assign_params)>();
  __shared__ float s_c[PQ_MAX_CENT * PQ_MAX_D];
  const int tid = threadIdx.x;
  const int lane = tid & (SAH_WAVE - 1);
  const int wave = tid / SAH_WAVE;
  const int s = blockIdx.x;
  const int bh = blockIdx.y;
  const int hk = bh % P.Hkv;
  const int b = bh / P.Hkv;
  const int g = bh * P.n_sub + s;
  const int d_sub = P.d_sub, n_cent = P.n_cent;
  // centres transposed, s_c[d][c]: the lanes of a wave (consecutive centres) read consecutive words
  for (int i = tid; i < n_cent * d_sub; i += PQB_NT) {
    const int c = i / d_sub, d = i - c * d_sub;
    s_c[d * n_cent + c] = P.centres[(int64_t)g * n_cent * d_sub + i];
  }
  // this wave's keys (every 16th), up to four of them requested before the first is used
  constexpr int NW = PQB_NT / SAH_WAVE;
  constexpr int KB = 4;
  const int64_t key0 = (int64_t)b * P.ks_b + (int64_t)hk * P.ks_h + (int64_t)s * d_sub;
  auto load_key = [&](int n, float (&x)[PQ_MAX_D]) {
    const int64_t off = key0 + (int64_t)(P.key_offset + n) * P.ks_l;
#pragma unroll
    for (int d = 0; d < PQ_MAX_D; ++d) x[d] = d < d_sub ? sah_load<DT>(P.k, off + d) : 0.f;
  };
  __syncthreads();
  for (int n0 = wave; n0 < P.n_keys; n0 += KB * NW) {
    float xs[KB][PQ_MAX_D];
#pragma unroll
    for (int u = 0; u < KB; ++u) {
      const int n = n0 + u * NW;
      load_key(n < P.n_keys ? n : n0, xs[u]);
    }
#pragma unroll
    for (int u = 0; u < KB; ++u) {
      const int n = n0 + u * NW;
      if (n >= P.n_keys) break;  // uniform across the wave
      const float (&x)[PQ_MAX_D] = xs[u];
      float dist = INFINITY;
      int best = 0x7fffffff;
      for (int c = lane; c < n_cent; c += SAH_WAVE) {
        float dd = 0.f;
        if (P.round_dist) {
#pragma unroll
          for (int d = 0; d < PQ_MAX_D; ++d) {
            if (d < d_sub) {
              const float df = sah_round<DT>(x[d] - s_c[d * n_cent + c]);
              dd += sah_round<DT>(df * df);
            }
          }
          dd = sah_round<DT>(dd);
        } else {
#pragma unroll
          for (int d = 0; d < PQ_MAX_D; ++d) {
            if (d < d_sub) {
              const float df = x[d] - s_c[d * n_cent + c];
              dd = fmaf(df, df, dd);
            }
          }
        }
        if (dd < dist) {  // c ascends: the first minimum is kept
          dist = dd;
          best = c;
        }
      }
#pragma unroll
      for (int o = 1; o < SAH_WAVE; o <<= 1) {
        const float od = __shfl_xor(dist, o);
        const int oi = __shfl_xor(best, o);
        if (od < dist || (od == dist && oi < best)) {
          dist = od;
          best = oi;
        }
      }
      if (lane == 0) P.codes[(((int64_t)bh * P.code_pitch) + P.code_offset + n) * P.n_sub + s] = (uint8_t)best;
    }
  }
}

struct pq_update_params {
  const void* k; int64_t ks_b, ks_h, ks_l;
  int Hkv, n_sub, d_sub, n_cent, key_offset;
  float* centres;
  long long* sums; int* counts;
  const uint32_t* absmax_bits;
  const int* reseed_idx;   // NULL: vector i of an empty centre is number reseed_first + g * n_cent + c of the generator
  uint32_t reseed_seed;    // seeded with reseed_seed, modulo n_keys (torch.randint of the whole run, drawn where needed)
  int64_t reseed_first;
  int n_keys;
  int clear;               // sums and counts are left zero for the next assignment
  float* shift2;
  float tol;
  int* state;
  int n_groups;
};

struct pq_update_lds {
  float red[PQ_MAX_CENT / SAH_WAVE];
  mt_lds mt;
};
// vector of the group that an empty centre takes (thread c: centre c; ridx of the others: any); all threads call
template <int NT>
__device__ __forceinline__ int pq_reseed_vector(const pq_update_params& P, int g, int cn, pq_update_lds& S) {
  static_assert(NT >= PQ_MAX_CENT, "a thread per centre");
  const int tid = threadIdx.x;
  int ridx = 0;
  if (P.reseed_idx) {
    if (tid < P.n_cent && cn == 0) ridx = P.reseed_idx[(int64_t)g * P.n_cent + tid];
  } else if (__syncthreads_or(tid < P.n_cent && cn == 0)) {  // rare: the generator runs only where a centre is empty
    const int64_t first = P.reseed_first + (int64_t)g * P.n_cent;
    const int64_t mine = first + (tid < P.n_cent ? tid : 0);
    const int last = (int)((first + P.n_cent - 1) / MT_N);
    mt_seed(S.mt, P.reseed_seed);
    for (int blk = 0; blk <= last; ++blk) {
      mt_next(S.mt, blk & 1);
      if (mine / MT_N == blk) ridx = (int)(mt_temper(S.mt.st[(blk & 1) ^ 1][mine % MT_N]) % (uint32_t)P.n_keys);
    }
  }
  return ridx;
}
// the group's share of the verdict: thread c < n_cent brings the distance centre c has moved
__device__ __forceinline__ void pq_update_verdict(const pq_update_params& P, int g, float move, pq_update_lds& S) {
  const int tid = threadIdx.x;
  move = sah_wave_sum(move);
  if ((tid & (SAH_WAVE - 1)) == 0 && tid < PQ_MAX_CENT) S.red[tid / SAH_WAVE] = move;
  __syncthreads();
  if (tid == 0) {
    float tot = 0.f;
    for (int i = 0; i < PQ_MAX_CENT / SAH_WAVE; ++i) tot += S.red[i];
    const float sh2 = tot * tot;
    P.shift2[g] = sh2;
    // the verdict's two counters only: the converged count is in before the ticket is taken, nothing else is handed over
    if (sh2 < P.tol) atomicAdd(&P.state[0], 1);
    sah_stores_done();
    const int ticket = atomicAdd(&P.state[1], 1);
    if (ticket == P.n_groups - 1) {
      // last group of this iteration, every other has read the done flag: publish the verdict, reset the counters
      const int conv = atomicAdd(&P.state[0], 0);
      if (conv == P.n_groups) P.state[2] = 1;
      P.state[0] = 0;
      P.state[1] = 0;
    }
  }
}
__device__ __forceinline__ int64_t pq_update_key(const pq_update_params& P, int g, int ridx) {
  const int s = g % P.n_sub, bh = g / P.n_sub;
  return (int64_t)(bh / P.Hkv) * P.ks_b + (int64_t)(bh % P.Hkv) * P.ks_h + (int64_t)(P.key_offset + ridx) * P.ks_l + (int64_t)s * P.d_sub;
}

// The update of a group by the workgroup (NT threads) of an assignment that ends last: sums and counts come with accesses that
// see what the others have added, requested together and at consecutive addresses, and are left zero; the new centres element
// by element, the distances by a thread per centre in ascending dimensions (as k_pq_update).
static __host__ __device__ size_t pq_update_here_bytes(int n_cent, int d_sub) {
  return (sizeof(pq_update_lds) + 15) / 16 * 16 + (size_t)n_cent * 16 + (size_t)n_cent * (d_sub + 1) * 4;
}
template <int DT, int NT>
__device__ __forceinline__ void pq_update_here(const pq_update_params& P, int g, unsigned char* lds) {
  const int tid = threadIdx.x;
  const int d_sub = P.d_sub, n_cent = P.n_cent, n_el = n_cent * d_sub;
  pq_update_lds& S = *(pq_update_lds*)lds;
  double* s_un = (double*)(lds + (sizeof(pq_update_lds) + 15) / 16 * 16);  // [n_cent] 1 / (scale * members)
  int* s_from = (int*)(s_un + n_cent);                                     // [n_cent] vector an empty centre takes, -1: none
  float* s_df = (float*)(s_from + 2 * n_cent);                             // [n_cent][d_sub + 1]
  float* cc = P.centres + (int64_t)g * n_el;
  long long* ss = P.sums + (int64_t)g * n_el;
  int* cp = P.counts + (int64_t)g * n_cent;
  constexpr int B = 4;  // elements a thread requests at a time
  long long sv[B];
  float ov[B];
  auto request = [&](int i0) {
#pragma unroll
    for (int u = 0; u < B; ++u) {
      const int i = i0 + u * NT < n_el ? i0 + u * NT : n_el - 1;
      sv[u] = sah_agent_load(&ss[i]);
      ov[u] = cc[i];
    }
  };
  const int cn = tid < n_cent ? sah_agent_load(&cp[tid]) : 1;
  request(tid);
  const int ridx = pq_reseed_vector<NT>(P, g, cn, S);
  if (tid < n_cent) {
    s_un[tid] = 1.0 / ((double)pq_sum_scale(*P.absmax_bits) * (double)(cn > 0 ? cn : 1));
    s_from[tid] = cn > 0 ? -1 : ridx;
    sah_agent_store(&cp[tid], 0);
  }
  __syncthreads();
  for (int i0 = tid; i0 < n_el; i0 += B * NT) {
    if (i0 != tid) request(i0);
#pragma unroll
    for (int u = 0; u < B; ++u) {
      const int i = i0 + u * NT;
      if (i < n_el) {
        const int c = i / d_sub, d = i - c * d_sub, from = s_from[c];
        const float nv = from < 0 ? (float)((double)sv[u] * s_un[c]) : sah_load<DT>(P.k, pq_update_key(P, g, from) + d);
        s_df[c * (d_sub + 1) + d] = nv - ov[u];
        cc[i] = nv;
        sah_agent_store(&ss[i], 0ll);
      }
    }
  }
  __syncthreads();
  float move = 0.f;
  if (tid < n_cent) {
    float acc = 0.f;
    for (int d = 0; d < d_sub; ++d) {
      const float df = s_df[tid * (d_sub + 1) + d];
      acc = fmaf(df, df, acc);
    }
    move = sqrtf(acc);
  }
  pq_update_verdict(P, g, move, S);
}

// The update in a launch of its own: one workgroup per group, a thread per centre. What bounds it is latency (a group's 18 KB):
// the sums of eight dimensions are requested together.
template <int DT>
__global__ __launch_bounds__(PQ_NT) void k_pq_update(pq_update_params P) {
  __shared__ pq_update_lds S;
  if (P.state[2]) return;
  const int tid = threadIdx.x, g = blockIdx.x;
  const int d_sub = P.d_sub, n_cent = P.n_cent;
  float move = 0.f;
  const int cn = tid < n_cent ? P.counts[(int64_t)g * n_cent + tid] : 1;
  const int ridx = pq_reseed_vector<PQ_NT>(P, g, cn, S);
  if (tid < n_cent) {
    const int c = tid;
    float* cc = P.centres + ((int64_t)g * n_cent + c) * d_sub;
    long long* ss = P.sums + ((int64_t)g * n_cent + c) * d_sub;
    const double unscale = 1.0 / ((double)pq_sum_scale(*P.absmax_bits) * (double)(cn > 0 ? cn : 1));
    float acc = 0.f;
    const int64_t roff = pq_update_key(P, g, ridx);
    for (int d0 = 0; d0 < d_sub; d0 += 8) {
      long long sv[8];
      float ov[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int d = d0 + u < d_sub ? d0 + u : d_sub - 1;
        sv[u] = ss[d];
        ov[u] = cc[d];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int d = d0 + u;
        if (d >= d_sub) break;
        const float nv = (cn > 0) ? (float)((double)sv[u] * unscale) : sah_load<DT>(P.k, roff + d);
        const float df = nv - ov[u];
        acc = fmaf(df, df, acc);
        cc[d] = nv;
        if (P.clear) ss[d] = 0;
      }
    }
    if (P.clear) P.counts[(int64_t)g * n_cent + c] = 0;
    move = sqrtf(acc);
  }
  pq_update_verdict(P, g, move, S);
}

// ---------------------------------------------------------------------------
// Lloyd assignment on the matrix cores. argmin_c ||x - c||^2 = argmin_c (||c||^2 - 2 x.c): the key x centre
// contraction is a 32 x 32 matrix product whose accumulator starts at ||c||^2 and whose A operand is -2 c, so the
// accumulator IS the quantity to minimise. A lane owns one key (column) and, per centre tile, 16 centres (rows) in
// ascending order: the running argmin needs no cross-lane work until the two lanes of a key are merged at the end.
// Centres (pre-scaled, in operand order) and their norms sit in LDS; per-centre sums for the update step are
// accumulated in LDS and flushed once.
// SPLIT (bf16 keys): -2 c is cut into three bf16 terms of 8 bits each, which together ARE the fp32 number, and the
// product runs on the bf16 instructions (32 cycles for 16 dimensions x 1 term; in fp32 64 cycles for 2 dimensions):
// every x * term is exact in fp32, the accumulation is fp32 as before.
// The split form's rounding is another one (and smaller), so where several centres come within both forms' rounding of the
// smallest value they are evaluated in the fp32 form's order of operations: the codes are those of the fp32 form, bit for
// bit, whichever form the alignment and shape of the keys allow (without: 1e-6 of the codes of an iteration, 5e-4 after ten).
// Measured (bf16, 8 heads x 16277 keys, 16 sub-vectors of 8, 256 centres, sums and update included, by events on a warm GPU): 66 us
// (a trace of a few passes, its clock still low, says 70 to 73); 85 with every tile's 16 values selected, not their minima over
// the tiles, the second look by matrix instruction, its test by ballots, the key
// operand in a structure (which went through scratch memory) and the centres read element by element. What bounds it: 20 vector
// and 2 matrix instructions a tile, in sum (5 us a centre tile: 40), 150 vector ones a key tile of eight (20), 6 before and
// after the loop. fp16 (no split: terms of small centres would leave its range): 121 at 16405 keys. 32768 keys, 2 sub-vectors of 64, 64
// centres: 218 -> 47 with the split. Sums in [centre][d] order and a flush of one centre a lane took 40 (8 dims) to 100 us
// (64 dims) of these.
// The expansion rounds differently from the difference form of the reference ((A - B)^2 summed,
// pq_utils.py:220-257): a key whose two nearest centres tie to the last bits may take the other one.
// ---------------------------------------------------------------------------
#define PQM_NT 512
#define PQM_NW (PQM_NT / SAH_WAVE)
#define PQM_MIN_TILES 64   // 32-key tiles a workgroup takes at least: 2048 keys
#define PQM_WGS 512        // and no more workgroups than this where the keys allow it (two per CU): every workgroup
                           // loads the centres and flushes n_cent * d_sub 64-bit sums with atomics
#define PQM_MAX_D 128      // widest sub-vector of the matrix-core assignment (64 k-steps)
#define PQM_FUSED_LDS (80 * 1024)  // operands + sums up to this much LDS: sums in the same kernel, two workgroups a CU
#define PQM_MAX_LDS (144 * 1024)  // operands at most (128 dimensions x 256 centres in fp32: 129 KB); the rest of a CU is static LDS
#define PQM_MIN(a, b) __builtin_elementwise_minimum(a, b)  // three-way minimum instruction, no quieting of its operands
// Slots of a lane whose centres are evaluated one by one; with more in some lane (repeated keys, whose centres are equal) the key
// tile goes to the matrix instructions again. Six iterations at 8 heads x 16277 keys, 16 sub-vectors of 8, 256 centres (in us):
// all keys equal 2178 (8656 one by one, however many), the first 60 % of them zeros 2206 (7139), random keys 508 (503). A slot
// costs 10 us a launch there, the tile again 43; 2 sub-vectors of 64 and 64 centres: 7 and 42. 1: random keys 2 to 8 % slower.
#define PQM_NEAR 3

// 16-byte operands per lane and centre tile of the split form: terms x dimensions in slots of 16 (sub-vectors of 8: two
// instructions; beyond: three per 16 dimensions)
__host__ __device__ constexpr int pqm_split_ops(int ks) { return ks <= 4 ? 2 : 3 * (ks / 8); }

// LDS of the assignment kernel: A operands, centre norms and, when the sums are fused, the fixed-point sums and counts
static size_t pqm_lds_bytes(int n_cent, int d_sub, int ks, bool sums, bool split) {
  const size_t n_tiles = (size_t)(n_cent + 31) / 32;
  size_t bytes = n_tiles * 64 * (split ? 16 * (size_t)pqm_split_ops(ks) : 4 * (size_t)ks) + n_tiles * 32 * 4;
  if (sums) bytes += (size_t)n_cent * d_sub * 8 + (size_t)n_cent * 4;
  const size_t update = sums ? pq_update_here_bytes(n_cent, d_sub) : 0;  // (runs in the same LDS)
  return bytes > update ? bytes : update;
}

// term 0, 1, 2 of a float as bf16 bits: eight significant bits each, their sum is the float (a float that is not finite
// stays in term 0)
__device__ __forceinline__ uint32_t pqm_term(float c, int term) {
  uint32_t hi = sah_float_to_bits(c) & 0xffff0000u;
  if ((hi & 0x7f800000u) == 0x7f800000u) return term ? 0u : (hi >> 16) | ((sah_float_to_bits(c) & 0xffffu) ? 1u : 0u);
  for (int i = 0; i < term; ++i) {
    c -= sah_bits_to_float(hi);
    hi = sah_float_to_bits(c) & 0xffff0000u;
  }
  return hi >> 16;
}

// bit v: a[v] <= b. Two instructions a value: a comparison into the carry, and the mask doubled with the carry in.
__device__ __forceinline__ uint32_t pqm_mask_le(const sah_f32x16& a, float b) {
#if defined(__HIP_DEVICE_COMPILE__)
  uint32_t m = 0;
#define PQM_LE4(x, y, z, w)                                                                                        \
  asm("v_cmp_le_f32 vcc, %1, %5\n\tv_addc_co_u32 %0, vcc, %0, %0, vcc\n\tv_cmp_le_f32 vcc, %2, %5\n\t"             \
      "v_addc_co_u32 %0, vcc, %0, %0, vcc\n\tv_cmp_le_f32 vcc, %3, %5\n\tv_addc_co_u32 %0, vcc, %0, %0, vcc\n\t"   \
      "v_cmp_le_f32 vcc, %4, %5\n\tv_addc_co_u32 %0, vcc, %0, %0, vcc"                                             \
      : "+&v"(m)                                                                                                   \
      : "v"(a[x]), "v"(a[y]), "v"(a[z]), "v"(a[w]), "v"(b)                                                         \
      : "vcc")
  PQM_LE4(15, 14, 13, 12);
  PQM_LE4(11, 10, 9, 8);
  PQM_LE4(7, 6, 5, 4);
  PQM_LE4(3, 2, 1, 0);
#undef PQM_LE4
  return m;
#else
  uint32_t m = 0;
  for (int v = 0; v < 16; ++v) m |= a[v] <= b ? 1u << v : 0u;
  return m;
#endif
}

// (two waves per SIMD at least: with at most 256 registers a wave the compiler keeps the accumulators in ordinary
// vector registers, which the minimum search reads directly)
// KS k-steps of two dimensions each: sub-vectors of up to 2 KS dimensions (the operands beyond d_sub are zero), of
// exactly 2 KS in the split form. SUMS: the per-centre sums of the update step are accumulated here (P.sums given and
// the LDS holds them). A workgroup takes wg_tiles tiles of 32 keys of one group.
// PIPE: the centre tiles go by in pairs, a multiple of four of them; a pair's products are under way while the minima of the
// pair before are taken, each matrix instruction between ten vector ones, and a key tile's last pair has the next key tile's
// first behind it, which so computes while the key tile is concluded. Sub-vectors of 8 alone: 8 heads x 16 of them, 256 centres:
// 4096 keys 30.4 -> 29.5 us, 16405 keys 66.8 -> 66.2, 32768 keys 114.8 -> 113.3 (32 heads x 8192 keys 113.3 -> 114.2, 128 centres x
// 16405 keys 46.6 -> 47.2); sub-vectors of 16 lost up to 2 % (8 of them, 128 centres, 16405 keys 38.9 -> 39.5).
template <int DT, int KS, bool SUMS, bool SPLIT, bool PIPE>
__global__ __launch_bounds__(PQM_NT, KS <= 16 ? 4 : 2) void k_pq_assign_mfma(pq_assign_params P, pq_update_params U, uint32_t* arrivals,
                                                                                           int wg_tiles, int ranges, int n_heads) {
  SAH_DYNAMIC_LDS(pqm_dyn)
  static_assert(!PIPE || (SPLIT && KS == 4), "the pipelined loop has two operands a tile and the norms among them");
  static_assert(!SPLIT || (DT == SAH_BF16 && KS >= 4), "the split form multiplies bf16 keys in sub-vectors of 8 and more");
  if (P.skip_flag && *P.skip_flag) return;
  const int tid = threadIdx.x;
  const int lane = tid & (SAH_WAVE - 1);
  const int wave = sah_wave_id();
  const int j = lane & 31, g = lane >> 5;
  // The workgroups of all sub-vectors of a range of keys read slices of the same rows and write bytes of the same code
  // words: they follow each other on one XCD (workgroups are dealt to the eight XCDs in turn) and meet in its L2
  // (with the next tile's keys requested ahead: 80 -> 71 us, 16 sub-vectors of 8, 8 heads x 16405 keys).
  const int s_idx = (blockIdx.x >> 3) % P.n_sub;
  const int unit = (int)((blockIdx.x >> 3) / P.n_sub) * 8 + (blockIdx.x & 7);  // (key range, head)
  const int bh = unit / ranges;
  const int tg = unit - bh * ranges;
  if (bh >= n_heads) return;
  const int hk = bh % P.Hkv;
  const int b = bh / P.Hkv;
  const int grp = bh * P.n_sub + s_idx;
  const int n_cent = P.n_cent, d_sub = SPLIT ? 2 * KS : P.d_sub;
  const int n_tiles = (n_cent + 31) >> 5;
  const float* cbase = P.centres + (int64_t)grp * n_cent * d_sub;
  constexpr int SQ = KS >= 4 ? 4 : KS;          // k-steps per 16-byte (8-byte) group of the fp32 form
  constexpr int OPS = pqm_split_ops(KS);        // 16-byte operands of the split form
  constexpr int TILE_A = SPLIT ? 64 * 4 * OPS : 64 * KS;  // 32-bit words of a tile's A operands
  // Sub-vectors of 8 leave slots of their first operand free: the norm's three terms stand there, against ones in the key
  // operand, instead of four 16-byte LDS reads per tile (16 x 8 dims x 256 centres, 8 heads x 16405 keys: 67 -> 64 us).
  constexpr bool NORM_IN_A = SPLIT && KS == 4;
  // -2 c as the A operand. fp32: element (k-step s, half g, centre row i of tile t); four k-steps of a row sit together
  // and consecutive rows follow each other, so that a wave's 16-byte reads are conflict-free whatever KS is.
  float* s_a = (float*)pqm_dyn;                                    // [tile][g][s / 4][i][s % 4]   (KS = 2: [tile][g][i][s])
                                                                   // SPLIT: [tile][op][g][i] of eight bf16
  float* s_cn = s_a + (size_t)n_tiles * TILE_A;                    // ||c||^2, [tile][g][v]
  long long* s_sum = (long long*)(s_cn + (size_t)n_tiles * 32);    // [d][centre] (SUMS only; 8-byte aligned: both sizes
  int* s_cnt = (int*)(s_sum + (size_t)n_cent * d_sub);             // [centre]     above are multiples of 8). A wave adds
                                                                   // one dimension at a time: the centres of its keys
                                                                   // spread over the banks
  const uint32_t absmax = SUMS ? *P.absmax_bits : 0u;
  const float sum_scale = SUMS ? pq_sum_scale(absmax) : 1.f;
  const double sum_scale_d = (double)sum_scale;
  const bool no_inf = absmax < 0x7f800000u;

  // The centres pass once through LDS (in the place of the sums, which fit them) on their way to operands and norms: one
  // round trip to memory instead of one per operand element of a thread.
  float* s_c = SUMS ? (float*)s_sum : nullptr;
  if (SUMS) {
    for (int i = tid; i < n_cent * d_sub; i += PQM_NT) s_c[i] = cbase[i];
    __syncthreads();
  }
  auto centre = [&](int c, int d) -> float { return SUMS ? s_c[c * d_sub + d] : cbase[c * d_sub + d]; };
  int odd = 0;  // a centre that is not finite
  for (int idx = tid; idx < n_tiles * 32; idx += PQM_NT) {
    const int v = idx & 15, gg = (idx >> 4) & 1, t = idx >> 5;
    const int c = t * 32 + 8 * (v >> 2) + 4 * gg + (v & 3);
    float nn = INFINITY;  // centres beyond n_cent never win
    if (c < n_cent) {
      nn = 0.f;
      for (int d = 0; d < d_sub; ++d) nn = fmaf(centre(c, d), centre(c, d), nn);
      if (!(nn < INFINITY)) odd = 1;
    }
    s_cn[idx] = nn;
  }
  if (NORM_IN_A) __syncthreads();
  if constexpr (SPLIT) {
    // a pair of dimensions each: its three terms, smallest in the first operands (they meet the accumulator while it holds the
    // norm alone)
    uint32_t* a32 = (uint32_t*)s_a;
    for (int idx = tid; idx < n_tiles * 32 * KS; idx += PQM_NT) {
      const int e = idx & 3, i = (idx >> 2) & 31, rest = idx >> 7, q8 = rest % (KS / 4), t = rest / (KS / 4);
      const int c = t * 32 + i, d = 8 * q8 + 2 * e;
      uint32_t w[3] = {0, 0, 0};
      if (c < n_cent) {
        const float lo = -2.0f * centre(c, d), hi = -2.0f * centre(c, d + 1);
#pragma unroll
        for (int term = 0; term < 3; ++term) w[term] = pqm_term(lo, term) | pqm_term(hi, term) << 16;
      }
      uint32_t* at = a32 + (size_t)t * TILE_A + i * 4 + e;  // + 256 * operand + 128 * half
      if constexpr (KS == 4) {
        at[0] = w[2];
        at[256] = w[0];
        at[384] = w[1];
        const float nn = s_cn[t * 32 + ((i >> 2) & 1) * 16 + 4 * (i >> 3) + (i & 3)];
        at[128] = e == 0 ? pqm_term(nn, 0) | pqm_term(nn, 1) << 16 : (e == 1 ? pqm_term(nn, 2) : 0u);
      } else {
#pragma unroll
        for (int term = 0; term < 3; ++term) at[256 * ((q8 >> 1) + (KS / 8) * (2 - term)) + 128 * (q8 & 1)] = w[term];
      }
    }
  } else {
    for (int idx = tid; idx < n_tiles * TILE_A; idx += PQM_NT) {
      const int s4 = idx % SQ, i = (idx / SQ) & 31, q = (idx / (SQ * 32)) % (KS / SQ), gg = (idx / (SQ * 32 * (KS / SQ))) & 1,
                t = idx / (64 * KS);
      const int c = t * 32 + i, d = 2 * (q * SQ + s4) + gg;
      s_a[idx] = (c < n_cent && d < d_sub) ? -2.0f * centre(c, d) : 0.f;
    }
  }
  odd = __syncthreads_or(odd);
  if (SUMS) {
    for (int i = tid; i < n_cent * d_sub; i += PQM_NT) s_sum[i] = 0;
    for (int i = tid; i < n_cent; i += PQM_NT) s_cnt[i] = 0;
    __syncthreads();
  }

  const int64_t kbase = (int64_t)b * P.ks_b + (int64_t)hk * P.ks_h + (int64_t)s_idx * d_sub;
  uint8_t* codes = P.codes + ((int64_t)bh * P.code_pitch + P.code_offset + (int64_t)tg * wg_tiles * 32) * P.n_sub + s_idx;  // of the workgroup's first key
  constexpr int NB = SPLIT ? (KS >= 8 ? KS / 8 : 1) : 1;  // key operands of 16 dimensions
  auto key_offset = [&](int n) { return kbase + (int64_t)(P.key_offset + (n < P.n_keys ? n : P.n_keys - 1)) * P.ks_l; };
  sah_u4 nb[NB];  // SPLIT: the next tile's keys, requested while this one is searched
  auto request = [&](int n) {
    const uint16_t* kp = (const uint16_t*)P.k + key_offset(n);
    if constexpr (KS == 4) {
      nb[0] = *(const sah_u4*)kp;
    } else {
#pragma unroll
      for (int q = 0; q < NB; ++q) nb[q] = *(const sah_u4*)(kp + 16 * q + 8 * g);
    }
  };
  if constexpr (SPLIT) request((tg * wg_tiles + wave) * 32 + j);
  // From a key tile's minima to its codes and sums. kept: every slot's minimum over the tiles (SPLIT) or the 16 values of the
  // tile of the smallest; xb / xs: its keys.
  auto conclude = [&](int kt, int n, const sah_u4 (&xb)[NB], const float (&xs)[SPLIT ? 1 : KS], const sah_f32x16& kept, float best,
                      float second, int bt, bool nan) __attribute__((always_inline)) {
    // (the lane is opaque here: what follows from it is computed again for every key tile, in a few instructions, instead of
    // being held in registers that the products need)
    int own = tid & (SAH_WAVE - 1);
#if defined(__HIP_DEVICE_COMPILE__)
    if (PIPE) asm volatile("" : "+v"(own));
#endif
    const int j = own & 31, g = own >> 5;
    const bool valid = n < P.n_keys;
    int slot = 0, bidx;
    bool again;  // uniform: the key tile is evaluated in fp32, centres or keys not finite
    if constexpr (SPLIT) {
      // The split form's values round differently from the fp32 form's, and the codes are the fp32 form's whichever form
      // ran. They agree where no other centre comes within twice the two forms' difference of the smallest value. With
      // u = 2^-24, fp32's value is off by at most d u of the mass ||c||^2 + 2 sum |x c| (one rounding per product), and the
      // two by up to 2.8 sqrt(d) u of it from each other (measured over 4e6 pairs each of 8 to 128 dimensions; the split
      // form is the closer one to fp64): min(2 d, 6 sqrt(d)) u is allowed. A centre that can win is no farther from 0
      // than |x| + r, r the distance to the nearest, so its mass is at most 3 (|x| + r)^2; 3.5 leaves room for those beyond.
      float x2 = 0.f;
#pragma unroll
      for (int q = 0; q < NB; ++q) {
#pragma unroll
        for (int e = 0; e < 4; ++e) x2 = sah_dot2<SAH_BF16>(xb[q][e], xb[q][e], x2);
      }
      if (KS != 4) x2 = sah_half_sum(x2);
      best = sah_half_min(best);
      float r2 = best + x2;
      r2 = r2 < 0.f ? 0.f : r2;
      const float reach = __builtin_amdgcn_sqrtf(x2) + __builtin_amdgcn_sqrtf(r2);
      constexpr float FORMS = KS == 4 ? 16.f : KS == 8 ? 24.f : KS == 16 ? 34.f : KS == 32 ? 48.f : 68.f;
      const float lim = best + 7.0f * 0x1p-24f * FORMS * reach * reach;  // (not finite where the key is not)
      // The centres within it, of the minima of this lane's 16 slots (bit v of `in`) and of the other tiles (bit 16): exactly
      // one wins. (In vector registers throughout: ballots combined by the scalar unit cost 10 us of a launch.)
      uint32_t in = pqm_mask_le(kept, lim);
      const uint32_t info = in | (second <= lim ? 1u << 16 : 0u) | (uint32_t)bt << 20;
      uint32_t lo_half, hi_half;  // of the lanes g = 0 and g = 1 of the key
      sah_half_both(info, lo_half, hi_half);
      const bool from_lo = (lo_half & 0xffffu) != 0;
      const uint32_t src = from_lo ? lo_half : hi_half;
      slot = __builtin_ctz(src | 0x10000u);
      bidx = (int)(src >> 20) * 32 + 8 * (slot >> 2) + (from_lo ? 0 : 4) + (slot & 3);  // tile, slot -> centre
      const bool open = __popc(lo_half & 0x1ffffu) + __popc(hi_half & 0x1ffffu) != 1;
      const bool any_open = __ballot(open) != 0;  // uniform
      again = odd || (any_open && __ballot(!(lim < INFINITY) || (open && __popc(in) > PQM_NEAR)) != 0);
      if (any_open && !again) {
        // The fp32 form's values, for the keys with several centres in reach, of every centre in a slot that holds one: the fp32
        // matrix instruction is a chain of fused multiply-adds in ascending dimensions (checked bit for bit on the hardware),
        // so a lane can evaluate one centre.
        if (!open) in = 0;
        float fb = INFINITY;
        int fi = 0x7fffffff;
        const int64_t koff = key_offset(n);
        while (in) {
          const int v = __builtin_ctz(in);
          in &= in - 1;
          const int c0 = 8 * (v >> 2) + 4 * g + (v & 3);
          for (int t = 0; t < n_tiles && t * 32 + c0 < n_cent; ++t) {
            const int c = t * 32 + c0;
            float val = s_cn[(t * 2 + g) * 16 + v];
#pragma unroll 8
            for (int d = 0; d < 2 * KS; ++d) val = fmaf(-2.0f * cbase[c * d_sub + d], sah_load<DT>(P.k, koff + d), val);
            if (val < fb || (val == fb && c < fi)) {  // the first minimum
              fb = val;
              fi = c;
            }
          }
        }
        const float ob = __shfl_xor(fb, 32);
        const int oi = __shfl_xor(fi, 32);
        if (ob < fb || (ob == fb && oi < fi)) fi = oi;
        if (open) bidx = fi;
      }
    } else {
#pragma unroll
      for (int v = 15; v >= 0; --v) slot = kept[v] == best ? v : slot;
      bidx = bt * 32 + 8 * (slot >> 2) + 4 * g + (slot & 3);
      const float ob = __shfl_xor(best, 32);
      const int oi = __shfl_xor(bidx, 32);
      if (ob < best || (ob == best && oi < bidx)) bidx = oi;
      again = odd || __ballot(nan) != 0;
    }
    if (again) {  // all centres in fp32, operands straight from memory; a value that is not a number loses to any other
      best = INFINITY;
      bidx = 0;
      const int64_t off = key_offset(n);
      for (int t2 = 0; t2 < n_tiles; ++t2) {
        sah_f32x16 acc;
        const float4* cn4 = (const float4*)(s_cn + (t2 * 2 + g) * 16);
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
          const float4 c4 = cn4[q4];
          acc[4 * q4] = c4.x; acc[4 * q4 + 1] = c4.y; acc[4 * q4 + 2] = c4.z; acc[4 * q4 + 3] = c4.w;
        }
        const bool there = t2 * 32 + j < n_cent;
        const float* cp = cbase + (there ? t2 * 32 + j : 0) * d_sub;
#pragma unroll 8
        for (int s = 0; s < KS; ++s) {
          const int d = 2 * s + g;
          const bool in = d < d_sub;
          const float a = in ? -2.0f * cp[d] : 0.f;
          acc = sah_mfma_32x32x2_f32(there ? a : 0.f, in ? sah_load<DT>(P.k, off + d) : 0.f, acc);
        }
        float m = INFINITY;
        int mv = 0;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          if (acc[v] < m) {
            m = acc[v];
            mv = v;
          }
        }
        if (m < best) {
          best = m;
          bidx = t2 * 16 + mv;
        }
      }
      bidx = (bidx >> 4) * 32 + 8 * ((bidx >> 2) & 3) + 4 * g + (bidx & 3);
      const float ob = __shfl_xor(best, 32);
      const int oi = __shfl_xor(bidx, 32);
      if (ob < best || (ob == best && oi < bidx)) bidx = oi;
    }
    if (valid) {
      if (g == 0) codes[(uint32_t)((kt * 32 + j) * P.n_sub)] = (uint8_t)bidx;
      if (SUMS) {
        if constexpr (SPLIT) {
          auto add_all = [&](auto&& add) {
            auto add2 = [&](uint32_t w, int d) {  // two dimensions of a packed word
              add(&s_sum[d * n_cent + bidx], sah_bits_to_float(w << 16));
              add(&s_sum[(d + 1) * n_cent + bidx], sah_bits_to_float(w & 0xffff0000u));
            };
            if constexpr (KS == 4) {
              const uint32_t upper = 0u - (uint32_t)g;  // (a choice between elements would become an index into scratch memory)
              add2((xb[0].z & upper) | (xb[0].x & ~upper), 4 * g);
              add2((xb[0].w & upper) | (xb[0].y & ~upper), 4 * g + 2);
            } else {
#pragma unroll
              for (int q = 0; q < NB; ++q) {
                add2(xb[q].x, 16 * q + 8 * g);
                add2(xb[q].y, 16 * q + 8 * g + 2);
                add2(xb[q].z, 16 * q + 8 * g + 4);
                add2(xb[q].w, 16 * q + 8 * g + 6);
              }
            }
          };
          // uniform; the largest |element| passes over NaN, but a key that holds one has had its tile evaluated again
          if (no_inf && !again) add_all([&](long long* p, float x) { pq_sum_add_finite(p, x, sum_scale_d); });
          else add_all([&](long long* p, float x) { pq_sum_add(p, x, sum_scale); });
        } else {
#pragma unroll
          for (int s = 0; s < KS; ++s)
            if (2 * s + g < d_sub) pq_sum_add(&s_sum[(2 * s + g) * n_cent + bidx], xs[s], sum_scale);
        }
        if (g == 0) atomicAdd(&s_cnt[bidx], 1);
      }
    }
  };
  if constexpr (PIPE) {
    auto first_op = [&](const sah_u4& x) { return g ? sah_u4{0x3f803f80u, 0x3f80u, 0u, 0u} : x; };
    auto in_range = [&](int kt) { return kt < wg_tiles && (tg * wg_tiles + kt) * 32 < P.n_keys; };  // uniform across the wave
    int kt = wave;
    if (in_range(kt)) {
      float best, second;
      int bt;
      sah_f32x16 kept;
      sah_u4 cur[NB];  // the keys in hand (nb: the next ones)
      cur[0] = nb[0];
      request((tg * wg_tiles + kt + PQM_NW) * 32 + j);
      // the products of a pair of centre tiles: for every operand its two loads and two matrix instructions
      auto load = [&](int t, int op, uint4 (&o)[2]) __attribute__((always_inline)) {
        const uint4* ap = (const uint4*)s_a + (size_t)t * 64 * OPS + g * 32 + j;
        o[0] = ap[op * 64];
        o[1] = ap[(OPS + op) * 64];
      };
      auto mm = [&](const sah_u4& x, const uint4& o, sah_f32x16& acc) __attribute__((always_inline)) {
        acc = sah_mfma_32x32x16<SAH_BF16>(o, __builtin_bit_cast(uint4, x), acc);
        __builtin_amdgcn_sched_barrier(0);
      };
      auto take = [&](float m, int t) __attribute__((always_inline)) {
        second = __builtin_amdgcn_fmed3f(best, second, m);
        const bool less = m < best;
        best = less ? m : best;
        bt = less ? t : bt;
      };
      // the minima of tiles t and t + 1 (c0, c1), the products of tiles t_next and t_next + 1 (n0, n1) with the keys x
      auto step = [&](auto first_c, const sah_f32x16& c0, const sah_f32x16& c1, int t, sah_f32x16& n0, sah_f32x16& n1, int t_next,
                      const sah_u4& x, const sah_u4& x0) __attribute__((always_inline)) {
        constexpr bool FIRST = decltype(first_c)::value;
        uint4 o[2];
        n0 = n1 = sah_f32x16{};
        load(t_next, 0, o);
        if (FIRST) {
          best = second = INFINITY;
          bt = 0;
        }
        float m = c0[0];
#pragma unroll
        for (int v = 1; v < 8; ++v) m = PQM_MIN(m, c0[v]);
        __builtin_amdgcn_sched_barrier(0);
        mm(x0, o[0], n0);
#pragma unroll
        for (int v = 8; v < 16; ++v) m = PQM_MIN(m, c0[v]);
        take(m, t);
        __builtin_amdgcn_sched_barrier(0);
        mm(x0, o[1], n1);
        load(t_next, 1, o);
#pragma unroll
        for (int v = 0; v < 16; ++v) kept[v] = FIRST ? PQM_MIN(c0[v], c1[v]) : PQM_MIN(PQM_MIN(kept[v], c0[v]), c1[v]);
        __builtin_amdgcn_sched_barrier(0);
        mm(x, o[0], n0);
        m = c1[0];
#pragma unroll
        for (int v = 1; v < 8; ++v) m = PQM_MIN(m, c1[v]);
        __builtin_amdgcn_sched_barrier(0);
        mm(x, o[1], n1);
#pragma unroll
        for (int v = 8; v < 16; ++v) m = PQM_MIN(m, c1[v]);
        take(m, t + 1);
      };
      sah_f32x16 a0, a1, b0, b1;
      {
        a0 = a1 = sah_f32x16{};
#pragma unroll
        for (int op = 0; op < OPS; ++op) {
          uint4 o[2];
          load(0, op, o);
          mm(op ? cur[0] : first_op(cur[0]), o[0], a0);
          mm(op ? cur[0] : first_op(cur[0]), o[1], a1);
        }
      }
      for (;;) {
        const int n = (tg * wg_tiles + kt) * 32 + j;
        const sah_u4 cur0 = first_op(cur[0]);
        step(std::true_type(), a0, a1, 0, b0, b1, 2, cur[0], cur0);
        int t = 2;  // tiles t, t + 1 in b0, b1
        for (; t + 2 < n_tiles; t += 4) {
          step(std::false_type(), b0, b1, t, a0, a1, t + 2, cur[0], cur0);
          step(std::false_type(), a0, a1, t + 2, b0, b1, t + 4, cur[0], cur0);
        }
        step(std::false_type(), b0, b1, t, a0, a1, 0, nb[0], first_op(nb[0]));
        conclude(kt, n, cur, {0.f}, kept, best, second, bt, false);
        kt += PQM_NW;
        if (!in_range(kt)) break;
        cur[0] = nb[0];
        request(n + 2 * 32 * PQM_NW);
      }
    }
  } else {
    for (int kt = wave; kt < wg_tiles; kt += PQM_NW) {
      const int n0 = (tg * wg_tiles + kt) * 32;
      if (n0 >= P.n_keys) break;  // uniform across the wave
      const int n = n0 + j;
      float xs[SPLIT ? 1 : KS];  // this lane's dims 2 s + g of its key
      sah_u4 xb[NB];             // SPLIT: dims 16 q + 8 g .. + 7 (sub-vectors of 8: both halves hold all)
      sah_u4 x0;                 // key operand of the first instruction: with the norm in A, ones against its terms
      if constexpr (SPLIT) {
  #pragma unroll
        for (int q = 0; q < NB; ++q) xb[q] = nb[q];
        request(n + 32 * PQM_NW);
        x0 = xb[0];
        if (KS == 4 && g) x0 = sah_u4{0x3f803f80u, 0x3f80u, 0u, 0u};
      } else {
        const int64_t off = key_offset(n);
  #pragma unroll
        for (int s = 0; s < KS; ++s) xs[s] = (2 * s + g < d_sub) ? sah_load<DT>(P.k, off + 2 * s + g) : 0.f;
      }
      // accumulator of centre tile t: seeded with the norms, then the matrix instructions
      auto product = [&](sah_f32x16& acc, int t) {
        if constexpr (NORM_IN_A) {
          acc = sah_f32x16{};
        } else {
          const float4* cn4 = (const float4*)(s_cn + (t * 2 + g) * 16);
  #pragma unroll
          for (int q4 = 0; q4 < 4; ++q4) {
            const float4 c4 = cn4[q4];
            acc[4 * q4] = c4.x; acc[4 * q4 + 1] = c4.y; acc[4 * q4 + 2] = c4.z; acc[4 * q4 + 3] = c4.w;
          }
        }
        if constexpr (SPLIT) {
          const uint4* ap = (const uint4*)s_a + (size_t)t * 64 * OPS + g * 32 + j;
  #pragma unroll
          for (int op = 0; op < OPS; ++op) acc = sah_mfma_32x32x16<SAH_BF16>(ap[op * 64], __builtin_bit_cast(uint4, op ? xb[op % NB] : x0), acc);
        } else if constexpr (KS >= 4) {
          const float4* ap = (const float4*)(s_a + (size_t)(t * 2 + g) * 32 * KS) + j;
  #pragma unroll
          for (int q = 0; q < KS / 4; ++q) {
            const float4 a4 = ap[q * 32];
            acc = sah_mfma_32x32x2_f32(a4.x, xs[4 * q], acc);
            acc = sah_mfma_32x32x2_f32(a4.y, xs[4 * q + 1], acc);
            acc = sah_mfma_32x32x2_f32(a4.z, xs[4 * q + 2], acc);
            acc = sah_mfma_32x32x2_f32(a4.w, xs[4 * q + 3], acc);
          }
        } else {
          const float* ap = s_a + ((t * 2 + g) * 32 + j) * KS;
  #pragma unroll
          for (int s = 0; s < KS; ++s) acc = sah_mfma_32x32x2_f32(ap[s], xs[s], acc);
        }
      };
      // The smallest value and its tile; a value that is not a number makes its tile's minimum one, and such key tiles are
      // evaluated again below. Without the split form also that tile's 16 values, from which the slot is found once at the end
      // (27 vector instructions a tile; a search for the slot takes 48): strictly smaller in ascending tiles, lowest slot, so
      // that the first minimum is kept. In the split form instead every slot's minimum over the tiles, two tiles to a three-way
      // minimum, and the second smallest of the tiles' minima (20 instructions a tile): together they tell whether any other
      // centre came near the smallest value, and with none near the smallest value's slot is the one whose minimum it is.
      float best = INFINITY, second = INFINITY;
      int bt = 0;
      bool nan = false;
      sah_f32x16 kept = {};
      auto tile_min = [&](const sah_f32x16& acc, int t) -> bool {
        float m = acc[0];
  #pragma unroll
        for (int v = 1; v < 16; ++v) m = PQM_MIN(m, acc[v]);
        if (SPLIT) second = __builtin_amdgcn_fmed3f(best, second, m);
        else nan |= m != m;
        const bool less = m < best;
        best = less ? m : best;
        bt = less ? t : bt;
        return less;
      };
      sah_f32x16 acc0, acc1;
      if constexpr (SPLIT) {
        product(acc0, 0);
        tile_min(acc0, 0);
        kept = acc0;
        int t = 1;
        for (; t + 1 < n_tiles; t += 2) {
          product(acc0, t);
          product(acc1, t + 1);
  #pragma unroll
          for (int v = 0; v < 16; ++v) kept[v] = PQM_MIN(PQM_MIN(kept[v], acc0[v]), acc1[v]);
          tile_min(acc0, t);
          tile_min(acc1, t + 1);
        }
        if (t < n_tiles) {
          product(acc0, t);
  #pragma unroll
          for (int v = 0; v < 16; ++v) kept[v] = PQM_MIN(kept[v], acc0[v]);
          tile_min(acc0, t);
        }
      } else {
        auto take_min = [&](const sah_f32x16& acc, int t) {
          const bool less = tile_min(acc, t);
  #pragma unroll
          for (int v = 0; v < 16; ++v) kept[v] = less ? acc[v] : kept[v];
        };
        // two accumulators: a tile's products are issued before the minimum of the tile before is taken, which so never waits
        // for a product just started
        product(acc0, 0);
        int t = 0;
        for (; t + 2 < n_tiles; t += 2) {
          product(acc1, t + 1);
          take_min(acc0, t);
          product(acc0, t + 2);
          take_min(acc1, t + 1);
        }
        if (t + 1 < n_tiles) {
          product(acc1, t + 1);
          take_min(acc0, t);
          take_min(acc1, t + 1);
        } else {
          take_min(acc0, t);
        }
      }
      conclude(kt, n, xb, xs, kept, best, second, bt, nan);
    }
  }
  if (!SUMS) return;
  __syncthreads();
  // the workgroup's sums, consecutive lanes at consecutive addresses
  for (int i = tid; i < n_cent * d_sub; i += PQM_NT) {
    const int c = i / d_sub, d = i - c * d_sub;
    if (s_cnt[c])
      atomicAdd((unsigned long long*)&P.sums[(int64_t)grp * n_cent * d_sub + i], (unsigned long long)s_sum[d * n_cent + c]);
  }
  for (int c = tid; c < n_cent; c += PQM_NT)
    if (s_cnt[c]) atomicAdd(&P.counts[(int64_t)grp * n_cent + c], s_cnt[c]);
  if (!arrivals) return;
  // The workgroup of the group that arrives last carries out the update: 7 us of this kernel, where a launch of its own takes
  // 8.7 and the way from kernel to kernel.
  sah_stores_done();  // (the atomics' too)
  __syncthreads();
  int* s_last = s_cnt;
  if (tid == 0) *s_last = sah_last_arrival(arrivals + (int64_t)grp * n_cent, (uint32_t)ranges) ? 1 : 0;
  __syncthreads();
  const bool last = *s_last != 0;
  __syncthreads();  // the LDS goes on to the update
  if (last) pq_update_here<DT, PQM_NT>(U, grp, pqm_dyn);
}

// Per-centre sums and counts from the codes an assignment wrote, for shapes whose sums do not fit beside the
// assignment's operands in LDS. One workgroup takes 2048 keys of a group; consecutive threads take consecutive
// dimensions of a key, so their LDS atomics fall into consecutive words of one centre's row.
#define PQS_NT 1024
#define PQS_KEYS 2048
#define PQS_MAX_SUMS 16384  // fixed-point sums a workgroup keeps in LDS (128 KB): wider groups are split by dimension
// grid.z splits the dimensions into slices of d_chunk; slice 0 also counts the members
template <int DT>
__global__ __launch_bounds__(PQS_NT) void k_pq_sums(pq_assign_params P, int d_chunk) {
  SAH_DYNAMIC_LDS(pqs_dyn)
  if (P.skip_flag && *P.skip_flag) return;
  const int tid = threadIdx.x;
  const int s_idx = blockIdx.x % P.n_sub;
  const int tg = blockIdx.x / P.n_sub;
  const int bh = blockIdx.y;
  const int hk = bh % P.Hkv;
  const int b = bh / P.Hkv;
  const int grp = bh * P.n_sub + s_idx;
  const int n_cent = P.n_cent, d_sub = P.d_sub;
  const int d0 = blockIdx.z * d_chunk;
  const int dn = d_sub - d0 < d_chunk ? d_sub - d0 : d_chunk;
  long long* s_sum = (long long*)pqs_dyn;                  // [centre][dn]
  int* s_cnt = (int*)(s_sum + (size_t)n_cent * d_chunk);
  const float sum_scale = pq_sum_scale(*P.absmax_bits);
  for (int i = tid; i < n_cent * dn; i += PQS_NT) s_sum[i] = 0;
  for (int i = tid; i < n_cent; i += PQS_NT) s_cnt[i] = 0;
  __syncthreads();
  const int first = tg * PQS_KEYS;
  const int count = P.n_keys - first < PQS_KEYS ? P.n_keys - first : PQS_KEYS;
  const int64_t kbase = (int64_t)b * P.ks_b + (int64_t)hk * P.ks_h + (int64_t)s_idx * d_sub + d0;
  for (int idx = tid; idx < count * dn; idx += PQS_NT) {
    const int n = first + idx / dn, d = idx % dn;
    const int code = P.codes[(((int64_t)bh * P.code_pitch) + P.code_offset + n) * P.n_sub + s_idx];
    pq_sum_add(&s_sum[code * dn + d], sah_load<DT>(P.k, kbase + (int64_t)(P.key_offset + n) * P.ks_l + d), sum_scale);
    if (d == 0) atomicAdd(&s_cnt[code], 1);
  }
  __syncthreads();
  for (int i = tid; i < n_cent * dn; i += PQS_NT) {
    const int c = i / dn, d = i % dn;
    if (s_cnt[c])
      atomicAdd((unsigned long long*)&P.sums[(int64_t)grp * n_cent * d_sub + c * d_sub + d0 + d], (unsigned long long)s_sum[i]);
  }
  if (blockIdx.z == 0)
    for (int c = tid; c < n_cent; c += PQS_NT)
      if (s_cnt[c]) atomicAdd(&P.counts[(int64_t)grp * n_cent + c], s_cnt[c]);
}

template <int DT, int KS, bool SPLIT, bool PIPE>
static int pq_launch_mfma_ks(const sah_pq_assign_args* a, const pq_assign_params& P, const pq_update_params& U, uint32_t* arrivals, bool fused,
                             size_t lds) {
  const int tiles = (a->n_keys + 31) / 32;
  const int64_t all = (int64_t)tiles * a->n_sub * a->B * a->Hkv;
  int64_t wg_tiles = (all + PQM_WGS - 1) / PQM_WGS;
  if (wg_tiles < PQM_MIN_TILES) wg_tiles = PQM_MIN_TILES;
  const int wgs = (int)((tiles + wg_tiles - 1) / wg_tiles);  // per group, of about the same size
  const int per = (tiles + wgs - 1) / wgs;
  const int ranges = (tiles + per - 1) / per, heads = a->B * a->Hkv;
  const int64_t n_wg = (((int64_t)ranges * heads + 7) / 8) * 8 * a->n_sub;
  if (n_wg > 0x7fffffff) return sah_fail(SAH_ESHAPE, "sah_pq_kmeans_assign: too many workgroups");
  dim3 g((unsigned)n_wg), blk(PQM_NT);
  hipStream_t st = (hipStream_t)a->stream;
  sah_timed timed("k_pq_assign_mfma", a->stream);
  if (fused) {
    if (int rc = sah_allow_lds((const void*)k_pq_assign_mfma<DT, KS, true, SPLIT, PIPE>, PQM_MAX_LDS, "sah_pq_kmeans_assign")) return rc;
    hipLaunchKernelGGL((k_pq_assign_mfma<DT, KS, true, SPLIT, PIPE>), g, blk, lds, st, P, U, arrivals, per, ranges, heads);
  } else {
    if (int rc = sah_allow_lds((const void*)k_pq_assign_mfma<DT, KS, false, SPLIT, PIPE>, PQM_MAX_LDS, "sah_pq_kmeans_assign")) return rc;
    hipLaunchKernelGGL((k_pq_assign_mfma<DT, KS, false, SPLIT, PIPE>), g, blk, lds, st, P, U, nullptr, per, ranges, heads);
  }
  return sah_launch_status("sah_pq_kmeans_assign");
}

template <int DT, int KS>
static int pq_launch_mfma_form(const sah_pq_assign_args* a, const pq_assign_params& P, const pq_update_params& U, uint32_t* arrivals, bool split,
                               bool fused, size_t lds) {
  if constexpr (DT == SAH_BF16 && KS >= 4) {
    if constexpr (KS == 4) {
      if (split && (a->n_cent + 31) / 32 % 4 == 0) return pq_launch_mfma_ks<DT, KS, true, true>(a, P, U, arrivals, fused, lds);
    }
    if (split) return pq_launch_mfma_ks<DT, KS, true, false>(a, P, U, arrivals, fused, lds);
  }
  return pq_launch_mfma_ks<DT, KS, false, false>(a, P, U, arrivals, fused, lds);
}

template <int DT>
static int pq_launch_mfma(const sah_pq_assign_args* a, const pq_assign_params& P, const pq_update_params* U, uint32_t* arrivals, bool* updated) {
  int ks = 2;
  while (2 * ks < a->d_sub) ks *= 2;  // 2, 4, 8, 16, 32, 64 k-steps: sub-vectors of up to 4 ... 128 dimensions
  const bool want_sums = a->sums != nullptr;
  // The split form: bf16 keys, sub-vectors that fill its operands, key rows whose slices can be read 16 bytes at a time,
  // and centres whose three terms fit LDS. Sub-vectors of 4 stay in fp32: their two matrix instructions take about the
  // time of the minimum search anyway.
  const uint64_t align = (uint64_t)(uintptr_t)a->k | 2 * (uint64_t)a->ks_b | 2 * (uint64_t)a->ks_h | 2 * (uint64_t)a->ks_l;
  const bool split = DT == SAH_BF16 && ks >= 4 && a->d_sub == 2 * ks && align % 16 == 0 &&
                     pqm_lds_bytes(a->n_cent, a->d_sub, ks, false, true) <= PQM_MAX_LDS;
  const bool fused = want_sums && pqm_lds_bytes(a->n_cent, a->d_sub, ks, true, split) <= PQM_FUSED_LDS;
  const size_t lds = pqm_lds_bytes(a->n_cent, a->d_sub, ks, fused, split);
  const pq_update_params u = U ? *U : pq_update_params{};
  if (!U || !fused) arrivals = nullptr;
  if (updated) *updated = arrivals != nullptr;
  int rc;
  switch (ks) {
    case 2: rc = pq_launch_mfma_form<DT, 2>(a, P, u, arrivals, split, fused, lds); break;
    case 4: rc = pq_launch_mfma_form<DT, 4>(a, P, u, arrivals, split, fused, lds); break;
    case 8: rc = pq_launch_mfma_form<DT, 8>(a, P, u, arrivals, split, fused, lds); break;
    case 16: rc = pq_launch_mfma_form<DT, 16>(a, P, u, arrivals, split, fused, lds); break;
    case 32: rc = pq_launch_mfma_form<DT, 32>(a, P, u, arrivals, split, fused, lds); break;
    default: rc = pq_launch_mfma_form<DT, 64>(a, P, u, arrivals, split, fused, lds); break;
  }
  if (rc || !want_sums || fused) return rc;
  // the sums from the codes just written, in a launch of their own
  int d_chunk = a->d_sub;
  while (a->n_cent * d_chunk > PQS_MAX_SUMS) d_chunk = (d_chunk + 1) / 2;
  const size_t lds_s = (size_t)a->n_cent * d_chunk * 8 + (size_t)a->n_cent * 4;
  if ((rc = sah_allow_lds((const void*)k_pq_sums<DT>, 160 * 1024, "sah_pq_kmeans_assign"))) return rc;
  dim3 g(((a->n_keys + PQS_KEYS - 1) / PQS_KEYS) * a->n_sub, a->B * a->Hkv, (a->d_sub + d_chunk - 1) / d_chunk), blk(PQS_NT);
  sah_timed timed("k_pq_sums", a->stream);
  hipLaunchKernelGGL(k_pq_sums<DT>, g, blk, lds_s, (hipStream_t)a->stream, P, d_chunk);
  return sah_launch_status("sah_pq_kmeans_assign(sums)");
}

// Start vectors of every group: number (g, c) of a seeded torch.rand in float64 picks one vector of stratum c of
// [0, n_keys) (n_cent equal strata). One workgroup draws the whole sequence, two words a number.
struct pq_start_params {
  int64_t total;  // n_groups * n_cent
  int n_cent, n_keys;
  double stratum;
  int* idx;
};
struct pq_start_lds {
  mts_lds mt;
  int2 stratum[PQ_MAX_CENT];  // first vector, width
};
__device__ __forceinline__ void pq_start_draw(pq_start_lds& S, const mt_state& seeded, const pq_start_params& P) {
  for (int c = threadIdx.x; c < P.n_cent; c += MTS_NT) {
    const int b = (int)floor((double)c * P.stratum);
    const double e_all = floor((double)(c + 1) * P.stratum);
    const int e = e_all > (double)P.n_keys ? P.n_keys : (int)e_all;
    S.stratum[c] = make_int2(b, e - b > 1 ? e - b : 1);
  }
  const int t_mod = (int)(threadIdx.x % MTS_USE) % P.n_cent, step_mod = MTS_USE % P.n_cent;
  const int first_mod = MT_N / 2 % P.n_cent, call_mod = MTS_STEP / 2 % P.n_cent;
  int c_first = 0;  // stratum of the first number of a call
  mt_stream(S.mt, seeded, 2 * P.total, [&](auto&& word, int64_t first, int count, int t) {
    int c = c_first + t_mod;
    if (c >= P.n_cent) c -= P.n_cent;
    for (int n = t; n < count / 2; n += MTS_USE) {
      const uint32_t hi = mt_temper(word(2 * n)), lo = mt_temper(word(2 * n + 1));
      const double u = fma((double)(hi & 0x1fffffu), 0x1p32, (double)lo) * 0x1p-53;  // exact: 53 bits
      const int2 st = S.stratum[c];
      const int v = st.x + (int)floor(u * (double)st.y);
      P.idx[first / 2 + n] = v < P.n_keys - 1 ? v : P.n_keys - 1;
      c += step_mod;
      if (c >= P.n_cent) c -= P.n_cent;
    }
    c_first += first ? call_mod : first_mod;  // (the last call's numbers need no successor)
    if (c_first >= P.n_cent) c_first -= P.n_cent;
  });
}

// Reseed vectors of a whole run: numbers 0 .. total - 1 of the sequence the update draws from, by one workgroup. For runs of
// so many numbers that the groups with an empty centre, each drawing the sequence again up to its own, would take longer.
__global__ __launch_bounds__(MTS_NT) void k_pq_reseed(mt_state seeded, int64_t total, int n_keys, int* idx) {
  __shared__ mts_lds S;
  mt_stream(S, seeded, total, [&](auto&& word, int64_t first, int count, int t) {
    for (int i = t; i < count; i += MTS_USE) idx[first + i] = (int)(mt_temper(word(i)) % (uint32_t)n_keys);
  });
}

// centres[g][c][:] = vector idx[g][c] of the group, as fp32. A workgroup per group; idx[g][0] becomes the group's arrival
// counter (zero) of the assignments that follow.
#define PQG_NT 1024
template <int DT>
__global__ __launch_bounds__(PQG_NT) void k_pq_gather(const void* k, int64_t ks_b, int64_t ks_h, int64_t ks_l, int Hkv, int n_sub,
                                                      int d_sub, int n_cent, int key_offset, int* idx, float* centres) {
  const int g = blockIdx.x, s = g % n_sub, bh = g / n_sub;
  const int64_t base = (int64_t)(bh / Hkv) * ks_b + (int64_t)(bh % Hkv) * ks_h + (int64_t)s * d_sub;
  int* mine = idx + (int64_t)g * n_cent;
  for (int i = threadIdx.x; i < n_cent * d_sub; i += PQG_NT) {
    const int c = i / d_sub, d = i - c * d_sub;
    centres[(int64_t)g * n_cent * d_sub + i] = sah_load<DT>(k, base + (int64_t)(key_offset + mine[c]) * ks_l + d);
  }
  __syncthreads();
  if (threadIdx.x == 0) mine[0] = 0;
}

struct pq_adc_params {
  const void* q; int64_t qs_b, qs_h, qs_l;
  int Hq, Hkv, Lq, n_sub, d_sub, n_cent;
  const float* centres;
  const void* centres_narrow;  // the same values in the storage type, or NULL
  const uint8_t* codes; int64_t code_pitch;
  int n_cand;
  void* keys_out; int64_t key_pitch;
};

#define ADC_MAX_LUT 4096  // n_sub * n_cent
#define ADC_NT 1024       // threads of the scoring kernel
#define ADC_KEYS 4096     // candidates per workgroup of the scoring kernel
#define ADC_MAX_HEAD_DIM 512  // widest query vector a workgroup stages in LDS when it builds its own table
#define ADC_OWN_LUT_WGS 16 // up to this many workgroups per KV head each build the lookup table themselves

// Lookup table of one decode step: lut[bh][vg][s][c][i] = round(q_v . centre[bh][s][c]) for the NQ query vectors
// v = vg * NQ + i of the KV head's group, in the storage type (fp32: NQ = 2, 16-bit: NQ = 4, i.e. 8 bytes per
// (s, c): one LDS read serves all the query vectors a workgroup scores).
// NQ dot products -> one 8-byte table entry, each rounded to the storage type
template <int DT, int NQ>
__device__ __forceinline__ uint2 pq_pack_entry(const float (&acc)[NQ]) {
  float val[NQ];
#pragma unroll
  for (int i = 0; i < NQ; ++i) val[i] = sah_round<DT>(acc[i]);
  uint2 pk;
  if (DT == SAH_F32) {
    pk.x = sah_float_to_bits(val[0]);
    pk.y = sah_float_to_bits(val[1]);
  } else if (DT == SAH_BF16) {
    pk.x = (uint32_t)sah_float_to_bf16(val[0]) | ((uint32_t)sah_float_to_bf16(val[1]) << 16);
    pk.y = (uint32_t)sah_float_to_bf16(val[NQ > 2 ? 2 : 0]) | ((uint32_t)sah_float_to_bf16(val[NQ > 2 ? 3 : 0]) << 16);
  } else {
    pk.x = (uint32_t)sah_float_to_f16(val[0]) | ((uint32_t)sah_float_to_f16(val[1]) << 16);
    pk.y = (uint32_t)sah_float_to_f16(val[NQ > 2 ? 2 : 0]) | ((uint32_t)sah_float_to_f16(val[NQ > 2 ? 3 : 0]) << 16);
  }
  return pk;
}

// One table entry: the NQ rounded dot products of sub-space s, centre c, packed into 8 bytes.
template <int DT>
__device__ __forceinline__ uint2 pq_lut_entry(const pq_adc_params& P, int b, int hk, int bh, int vg, int s, int c) {
  constexpr int NQ = (DT == SAH_F32) ? 2 : 4;
  const int G = P.Hq / P.Hkv;
  const int nvec = G * P.Lq;
  const int d_sub = P.d_sub;
  const float* cc = P.centres + (((int64_t)bh * P.n_sub + s) * P.n_cent + c) * d_sub;
  float val[NQ];
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    const int v = vg * NQ + i;
    val[i] = 0.f;
    if (v < nvec) {
      const int h = hk * G + v / P.Lq, qi = v % P.Lq;
      const int64_t qo = (int64_t)b * P.qs_b + (int64_t)h * P.qs_h + (int64_t)qi * P.qs_l + (int64_t)s * d_sub;
      float acc = 0.f;
      for (int d = 0; d < d_sub; ++d) acc = fmaf(sah_load<DT>(P.q, qo + d), cc[d], acc);
      val[i] = acc;
    }
  }
  return pq_pack_entry<DT>(val);
}

template <int DT>
__global__ __launch_bounds__(PQ_NT) void k_pq_lut(pq_adc_params P, void* lut) {
  constexpr int NQ = (DT == SAH_F32) ? 2 : 4;
  const int s = blockIdx.x;
  const int bh = blockIdx.y;
  const int vg = blockIdx.z;
  const int hk = bh % P.Hkv;
  const int b = bh / P.Hkv;
  const int nvec = (P.Hq / P.Hkv) * P.Lq;
  const int n_vg = (nvec + NQ - 1) / NQ;
  for (int c = threadIdx.x; c < P.n_cent; c += PQ_NT) {
    const int64_t e = (((int64_t)bh * n_vg + vg) * P.n_sub + s) * P.n_cent + c;
    ((uint2*)lut)[e] = pq_lut_entry<DT>(P, b, hk, bh, vg, s, c);
  }
}

// Scores of ADC_KEYS candidates for the NQ query vectors of one group: one 16-wave workgroup, the table in LDS
// as 8-byte entries per (s, c) (two floats for fp32, four packed 16-bit values otherwise: the entries are rounded to
// the storage type anyway, and the LDS reads are what bounds this kernel), one thread per candidate. A lookup is
// one LDS read, NQ widenings (a shift or a mask for bf16) and NQ additions. (The packed dot-product instruction
// against (1, 0) would widen and add in one operation, but its sum is not always the correctly rounded one: one
// addition in 800 differed in the last bit.) OWN_LUT: the workgroup computes its table itself
// (every workgroup of a KV head repeats that work, which is cheaper than a launch of its own as long as a head is
// covered by a few dozen workgroups); otherwise the entries k_pq_lut wrote are copied in.
template <int DT, bool OWN_LUT>
__global__ __launch_bounds__(ADC_NT) void k_pq_adc(pq_adc_params P, const void* lut) {
  sah_touch_kernargs<sizeof(pq_adc_params) + 8>();
  constexpr int NQ = (DT == SAH_F32) ? 2 : 4;
  typedef typename std::conditional<DT == SAH_F32, uint32_t, uint16_t>::type key_t;
  typedef uint2 entry_t;
  SAH_DYNAMIC_LDS(adc_dyn)
  const int tid = threadIdx.x;
  const int bh = blockIdx.y;
  const int vg = blockIdx.z;
  const int hk = bh % P.Hkv;
  const int b = bh / P.Hkv;
  const int G = P.Hq / P.Hkv;
  const int nvec = G * P.Lq;
  const int n_vg = (nvec + NQ - 1) / NQ;
  const int n_sub = P.n_sub, n_cent = P.n_cent;
  const int lut_n = n_sub * n_cent;
  entry_t* s_lut = (entry_t*)adc_dyn;                      // lut_n entries
  float* s_q = (float*)(adc_dyn + (size_t)lut_n * sizeof(entry_t));  // NQ x ADC_MAX_HEAD_DIM (OWN_LUT only)

  int row[NQ];
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    const int v = vg * NQ + i;
    row[i] = -1;
    if (v < nvec) row[i] = (b * P.Hq + hk * G + v / P.Lq) * P.Lq + v % P.Lq;
  }
  // rounded to the storage type by the hardware converters (round to nearest even, as the software rounding)
  auto store_entry = [&](int i, const float (&val)[NQ]) {
    if constexpr (NQ == 2) s_lut[i] = make_uint2(sah_float_to_bits(val[0]), sah_float_to_bits(val[1]));
    else s_lut[i] = make_uint2(sah_pack2_hw<DT>(val[0], val[1]), sah_pack2_hw<DT>(val[2], val[3]));
  };
  // 16 one-byte codes per candidate = one 16-byte load: all of the thread's candidates are requested before
  // anything else and arrive while the table is built
  constexpr int T = ADC_KEYS / ADC_NT;
  const bool wide = n_sub == 16 && ((uintptr_t)P.codes & 15) == 0;
  uint4 cw[T];
  if (wide) {
#pragma unroll
    for (int t = 0; t < T; ++t) {
      int n = blockIdx.x * ADC_KEYS + t * ADC_NT + tid;
      if (n >= P.n_cand) n = P.n_cand - 1;
      cw[t] = *(const uint4*)(P.codes + ((int64_t)bh * P.code_pitch + n) * 16);
    }
  }
  if (OWN_LUT) {
    // the group's query vectors once into LDS (as floats), then every thread builds lut_n / ADC_NT entries
    // from one centre each: the centre's d_sub floats from memory, the query elements as LDS broadcasts
    const int d_sub = P.d_sub;
    const int D = n_sub * d_sub;
    for (int i = tid; i < NQ * D; i += ADC_NT) {
      const int qn = i / D, e = i % D;
      const int v = vg * NQ + qn;
      float x = 0.f;
      if (v < nvec) {
        const int h = hk * G + v / P.Lq, qi = v % P.Lq;
        x = sah_load<DT>(P.q, (int64_t)b * P.qs_b + (int64_t)h * P.qs_h + (int64_t)qi * P.qs_l + e);
      }
      s_q[qn * ADC_MAX_HEAD_DIM + e] = x;
    }
    __syncthreads();
    const bool pow2 = (n_cent & (n_cent - 1)) == 0;  // the usual case (2^bits centres): no integer division per entry
    const int shift = 31 - __builtin_clz(n_cent);
    int first = tid;  // first entry the general loop below still has to build
    if (DT != SAH_F32 && P.centres_narrow && d_sub == 8 && pow2 && n_cent >= SAH_WAVE) {
      // Sub-vectors of 8 in 16-bit storage. A wave takes whole sub-spaces (wave w: s = w, w + 16, ...), so the
      // query elements of a sub-space are read from LDS once per wave and lane instead of once per entry (those
      // broadcast reads were most of the table's cost); a lane builds the entries of centres lane, lane + 64, ...:
      // one 16-byte load per centre, up to four of them requested together.
      const int lane = tid & (SAH_WAVE - 1);
      constexpr int LE = 4;
      for (int s = sah_wave_id(); s < n_sub; s += ADC_NT / SAH_WAVE) {
        float qv[NQ][8];
#pragma unroll
        for (int qn = 0; qn < NQ; ++qn) {
          const float4 q0 = *(const float4*)&s_q[qn * ADC_MAX_HEAD_DIM + s * 8];
          const float4 q1 = *(const float4*)&s_q[qn * ADC_MAX_HEAD_DIM + s * 8 + 4];
          qv[qn][0] = q0.x; qv[qn][1] = q0.y; qv[qn][2] = q0.z; qv[qn][3] = q0.w;
          qv[qn][4] = q1.x; qv[qn][5] = q1.y; qv[qn][6] = q1.z; qv[qn][7] = q1.w;
        }
        for (int c0 = lane; c0 < n_cent; c0 += LE * SAH_WAVE) {
          uint4 raw[LE];
#pragma unroll
          for (int u = 0; u < LE; ++u) {
            int c = c0 + u * SAH_WAVE;
            if (c >= n_cent) c = n_cent - 1;
            raw[u] = *(const uint4*)((const uint16_t*)P.centres_narrow + (((int64_t)bh * n_sub + s) * n_cent + c) * 8);
          }
#pragma unroll
          for (int u = 0; u < LE; ++u) {
            const int c = c0 + u * SAH_WAVE;
            if (c < n_cent) {
              const uint32_t w[4] = {raw[u].x, raw[u].y, raw[u].z, raw[u].w};
              float cv[8];
#pragma unroll
              for (int t = 0; t < 4; ++t) {
                if (DT == SAH_BF16) {
                  cv[2 * t] = sah_bits_to_float(w[t] << 16);
                  cv[2 * t + 1] = sah_bits_to_float(w[t] & 0xffff0000u);
                } else {
                  cv[2 * t] = sah_f16_to_float((uint16_t)(w[t] & 0xffffu));
                  cv[2 * t + 1] = sah_f16_to_float((uint16_t)(w[t] >> 16));
                }
              }
              float acc[NQ];
#pragma unroll
              for (int qn = 0; qn < NQ; ++qn) {
                float a = 0.f;
#pragma unroll
                for (int d = 0; d < 8; ++d) a = fmaf(qv[qn][d], cv[d], a);
                acc[qn] = a;
              }
              store_entry(s * n_cent + c, acc);
            }
          }
        }
      }
      first = lut_n;
    }
    for (int i = first; i < lut_n; i += ADC_NT) {
      const int s = pow2 ? i >> shift : i / n_cent;
      const int c = pow2 ? i & (n_cent - 1) : i % n_cent;
      const float* cc = P.centres + (((int64_t)bh * n_sub + s) * n_cent + c) * d_sub;
      float acc[NQ];
#pragma unroll
      for (int qn = 0; qn < NQ; ++qn) acc[qn] = 0.f;
      if (DT != SAH_F32 && P.centres_narrow) {
        // the centres in their 16-bit storage form: every workgroup of a KV head reads the whole codebook of the
        // head, so halving its bytes halves the larger part of this kernel's memory traffic
        for (int d = 0; d < d_sub; d += 8) {
          float cv[8];
          sah_load8<DT>(P.centres_narrow, (((int64_t)bh * n_sub + s) * n_cent + c) * d_sub + d, cv);
#pragma unroll
          for (int qn = 0; qn < NQ; ++qn) {
            const float4 q0 = *(const float4*)&s_q[qn * ADC_MAX_HEAD_DIM + s * d_sub + d];
            const float4 q1 = *(const float4*)&s_q[qn * ADC_MAX_HEAD_DIM + s * d_sub + d + 4];
            acc[qn] = fmaf(q0.x, cv[0], acc[qn]);
            acc[qn] = fmaf(q0.y, cv[1], acc[qn]);
            acc[qn] = fmaf(q0.z, cv[2], acc[qn]);
            acc[qn] = fmaf(q0.w, cv[3], acc[qn]);
            acc[qn] = fmaf(q1.x, cv[4], acc[qn]);
            acc[qn] = fmaf(q1.y, cv[5], acc[qn]);
            acc[qn] = fmaf(q1.z, cv[6], acc[qn]);
            acc[qn] = fmaf(q1.w, cv[7], acc[qn]);
          }
        }
      } else if ((d_sub & 3) == 0) {
        // 16-byte reads of the centre and of the staged queries (the same fused multiply-adds in the same order)
        for (int d = 0; d < d_sub; d += 4) {
          const float4 cv = *(const float4*)(cc + d);
#pragma unroll
          for (int qn = 0; qn < NQ; ++qn) {
            const float4 qv = *(const float4*)&s_q[qn * ADC_MAX_HEAD_DIM + s * d_sub + d];
            acc[qn] = fmaf(qv.x, cv.x, acc[qn]);
            acc[qn] = fmaf(qv.y, cv.y, acc[qn]);
            acc[qn] = fmaf(qv.z, cv.z, acc[qn]);
            acc[qn] = fmaf(qv.w, cv.w, acc[qn]);
          }
        }
      } else {
        for (int d = 0; d < d_sub; ++d) {
          const float cv = cc[d];
#pragma unroll
          for (int qn = 0; qn < NQ; ++qn) acc[qn] = fmaf(s_q[qn * ADC_MAX_HEAD_DIM + s * d_sub + d], cv, acc[qn]);
        }
      }
      store_entry(i, acc);
    }
  } else {
    const uint2* slab = (const uint2*)lut + ((int64_t)bh * n_vg + vg) * lut_n;
    for (int i = tid; i < lut_n; i += ADC_NT) s_lut[i] = slab[i];
  }
  __syncthreads();

  float acc[NQ];
  auto add = [&](int s, int c) {
    const entry_t e = s_lut[s * n_cent + c];
    if constexpr (NQ == 2) {
      acc[0] += sah_bits_to_float(e.x);
      acc[1] += sah_bits_to_float(e.y);
    } else if constexpr (DT == SAH_BF16) {
      acc[0] += sah_bits_to_float(e.x << 16);
      acc[1] += sah_bits_to_float(e.x & 0xffff0000u);
      acc[2] += sah_bits_to_float(e.y << 16);
      acc[3] += sah_bits_to_float(e.y & 0xffff0000u);
    } else {
      acc[0] += sah_f16_to_float((uint16_t)(e.x & 0xffffu));
      acc[1] += sah_f16_to_float((uint16_t)(e.x >> 16));
      acc[2] += sah_f16_to_float((uint16_t)(e.y & 0xffffu));
      acc[3] += sah_f16_to_float((uint16_t)(e.y >> 16));
    }
  };
  auto store = [&](int n) {
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      if (row[i] >= 0)
        ((key_t*)P.keys_out)[(int64_t)row[i] * P.key_pitch + n] = (key_t)sah_sort_key<DT>(sah_round<DT>(acc[i]));
    }
  };
  if (wide) {
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int n = blockIdx.x * ADC_KEYS + t * ADC_NT + tid;
      const uint32_t w4[4] = {cw[t].x, cw[t].y, cw[t].z, cw[t].w};
#pragma unroll
      for (int i = 0; i < NQ; ++i) acc[i] = 0.f;
#pragma unroll
      for (int s = 0; s < 16; ++s) add(s, (int)((w4[s >> 2] >> (8 * (s & 3))) & 0xffu));
      if (n < P.n_cand) store(n);
    }
    return;
  }
  const bool words = (n_sub & 3) == 0 && ((P.code_pitch * n_sub) & 3) == 0 && ((uintptr_t)P.codes & 3) == 0;
  for (int t = 0; t < T; ++t) {
    const int n = blockIdx.x * ADC_KEYS + t * ADC_NT + tid;
    if (n >= P.n_cand) continue;
    const uint8_t* code = P.codes + ((int64_t)bh * P.code_pitch + n) * n_sub;
#pragma unroll
    for (int i = 0; i < NQ; ++i) acc[i] = 0.f;
    if (words) {
      for (int s4 = 0; s4 < n_sub; s4 += 4) {
        const uint32_t w = *(const uint32_t*)(code + s4);
        add(s4, (int)(w & 0xffu));
        add(s4 + 1, (int)((w >> 8) & 0xffu));
        add(s4 + 2, (int)((w >> 16) & 0xffu));
        add(s4 + 3, (int)(w >> 24));
      }
    } else {
      for (int s = 0; s < n_sub; ++s) add(s, (int)code[s]);
    }
    store(n);
  }
}

// dynamic LDS of k_pq_adc: the table (8 bytes per entry) and, for OWN_LUT, the staged query vectors
template <int DT>
static size_t adc_lds_bytes(int lut_n) {
  constexpr int NQ = (DT == SAH_F32) ? 2 : 4;
  return (size_t)lut_n * 8 + (size_t)NQ * ADC_MAX_HEAD_DIM * 4;
}

template <int DT, bool OWN_LUT>
static int adc_launch(const pq_adc_params& P, const void* lut, dim3 g, hipStream_t st) {
  if (int rc = sah_allow_lds((const void*)k_pq_adc<DT, OWN_LUT>, 150 * 1024, "sah_pq_adc_scores")) return rc;
  hipLaunchKernelGGL((k_pq_adc<DT, OWN_LUT>), g, dim3(ADC_NT), adc_lds_bytes<DT>(P.n_sub * P.n_cent), st, P, lut);
  return SAH_OK;
}

static int pq_check_common(const char* what, int B, int Hkv, int n_sub, int d_sub, int n_cent) {
  if (B <= 0 || Hkv <= 0 || n_sub <= 0) return sah_fail(SAH_EINVAL, "%s: bad B/Hkv/n_sub", what);
  if (d_sub <= 0 || d_sub > PQM_MAX_D) return sah_fail(SAH_ESHAPE, "%s: d_sub %d not in [1, %d]", what, d_sub, PQM_MAX_D);
  if (n_cent <= 0 || n_cent > PQ_MAX_CENT) return sah_fail(SAH_ESHAPE, "%s: n_cent %d not in [1, %d]", what, n_cent, PQ_MAX_CENT);
  if ((int64_t)B * Hkv > 65535) return sah_fail(SAH_ESHAPE, "%s: B*Hkv > 65535", what);
  return SAH_OK;
}

// Largest |element| of the keys [key_offset, key_offset + n_keys) of every (b, kv head), as float bits (non-negative
// floats order like their bit patterns, so an integer atomic max does it). *out must be zero before the launch.
// VEC elements a load: 16 bytes where the rows allow it (an element at a time, with a 64-bit division each, a 33 MB
// cache took 72 us; its bytes take 7; with one atomic per wave 51, as here 17).
// share `part` of `parts` of head bh, by one workgroup of NT threads
template <int DT, int VEC, int NT>
__device__ __forceinline__ void pq_absmax_part(const void* k, int64_t ks_b, int64_t ks_h, int64_t ks_l, int Hkv, int D, int key_offset,
                                               int n_keys, uint32_t* out, int bh, int part, int parts, uint32_t* s_best) {
  const int64_t base = (int64_t)(bh / Hkv) * ks_b + (int64_t)(bh % Hkv) * ks_h + (int64_t)key_offset * ks_l;
  const int upr = D / VEC;  // loads per row
  const int64_t total = (int64_t)n_keys * upr;
  const int64_t step = (int64_t)parts * NT;
  uint32_t best = 0u;
  auto take = [&](uint32_t bits) {
    bits &= 0x7fffffffu;
    if (bits <= 0x7f800000u) best = bits > best ? bits : best;  // NaN is skipped
  };
  int64_t i = (int64_t)part * NT + threadIdx.x;
  int64_t n = i / upr;
  int c = (int)(i - n * upr);
  const int64_t dn = step / upr;
  const int dc = (int)(step - dn * upr);
#pragma unroll 4
  for (; i < total; i += step) {
    const int64_t off = base + n * ks_l + (int64_t)c * VEC;
    if constexpr (VEC == 1) {
      take(sah_float_to_bits(sah_load<DT>(k, off)));
    } else {
      const uint4 q = *(const uint4*)((const char*)k + off * (DT == SAH_F32 ? 4 : 2));
      const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if (DT == SAH_F32) {
          take(w[t]);
        } else if (DT == SAH_BF16) {
          take(w[t] << 16);
          take(w[t] & 0xffff0000u);
        } else {
          take(sah_float_to_bits(sah_f16_to_float((uint16_t)w[t])));
          take(sah_float_to_bits(sah_f16_to_float((uint16_t)(w[t] >> 16))));
        }
      }
    }
    n += dn;
    c += dc;
    if (c >= upr) {
      c -= upr;
      ++n;
    }
  }
#pragma unroll
  for (int o = 1; o < SAH_WAVE; o <<= 1) {
    const uint32_t other = (uint32_t)__shfl_xor((int)best, o);
    best = other > best ? other : best;
  }
  // one atomic per workgroup: all go to one address, 5 ns each (8192 of them, one per wave, took 41 us)
  if ((threadIdx.x & (SAH_WAVE - 1)) == 0) s_best[threadIdx.x / SAH_WAVE] = best;
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < NT / SAH_WAVE; ++w) best = s_best[w] > best ? s_best[w] : best;
    if (best) atomicMax(out, best);
  }
}

template <int DT, int VEC>
__global__ __launch_bounds__(PQ_NT) void k_pq_absmax(const void* k, int64_t ks_b, int64_t ks_h, int64_t ks_l, int Hkv, int D,
                                                     int key_offset, int n_keys, uint32_t* out) {
  __shared__ uint32_t s_best[PQ_NT / SAH_WAVE];
  pq_absmax_part<DT, VEC, PQ_NT>(k, ks_b, ks_h, ks_l, Hkv, D, key_offset, n_keys, out, blockIdx.y, blockIdx.x, gridDim.x, s_best);
}

// What a run needs before its first assignment and what does not need each other: workgroup 0 draws the start vectors, the
// others find the largest |element| (`parts` workgroups a head). 54 us (8 heads x 16277 keys of 128, 128 groups of 256 centres);
// one after the other 78 and 16.
template <int DT, int VEC>
__global__ __launch_bounds__(MTS_NT) void k_pq_prepare(mt_state seeded, pq_start_params S, const void* k, int64_t ks_b, int64_t ks_h,
                                                       int64_t ks_l, int Hkv, int D, int key_offset, int n_keys, uint32_t* out, int parts) {
  __shared__ pq_start_lds s_start;
  if (blockIdx.x == 0) {
    pq_start_draw(s_start, seeded, S);
    return;
  }
  const int w = (int)blockIdx.x - 1;
  pq_absmax_part<DT, VEC, MTS_NT>(k, ks_b, ks_h, ks_l, Hkv, D, key_offset, n_keys, out, w / parts, w % parts, parts, s_start.mt.x);
}

// workgroups of nt threads per head, and whether the keys can be read 16 bytes at a time
static int pq_absmax_parts(const sah_pq_absmax_args* a, int nt, bool* vec) {
  const int v = a->dtype == SAH_F32 ? 4 : 8;
  *vec = a->D % v == 0 && a->ks_b % v == 0 && a->ks_h % v == 0 && a->ks_l % v == 0 && (uintptr_t)a->k % 16 == 0;
  const int64_t total = (int64_t)a->n_keys * (*vec ? a->D / v : a->D), heads = (int64_t)a->B * a->Hkv;
  int64_t parts = (total + nt * 8 - 1) / (nt * 8);
  const int64_t most = ((int64_t)1024 * PQ_NT / nt + heads - 1) / heads;
  return (int)(parts < 1 ? 1 : (parts > most ? most : parts));
}
template <int DT>
static void pq_absmax_launch(const sah_pq_absmax_args* a) {
  constexpr int VEC = DT == SAH_F32 ? 4 : 8;
  bool vec;
  const int parts = pq_absmax_parts(a, PQ_NT, &vec);
  dim3 g((unsigned)parts, a->B * a->Hkv), blk(PQ_NT);
  hipStream_t st = (hipStream_t)a->stream;
  if (vec)
    hipLaunchKernelGGL((k_pq_absmax<DT, VEC>), g, blk, 0, st, a->k, a->ks_b, a->ks_h, a->ks_l, a->Hkv, a->D, a->key_offset, a->n_keys, a->absmax_bits);
  else
    hipLaunchKernelGGL((k_pq_absmax<DT, 1>), g, blk, 0, st, a->k, a->ks_b, a->ks_h, a->ks_l, a->Hkv, a->D, a->key_offset, a->n_keys, a->absmax_bits);
}
template <int DT>
static void pq_prepare_launch(const sah_pq_absmax_args* a, const pq_start_params& S, uint32_t seed) {
  constexpr int VEC = DT == SAH_F32 ? 4 : 8;
  bool vec;
  const int parts = pq_absmax_parts(a, MTS_NT, &vec);
  dim3 g((unsigned)(parts * a->B * a->Hkv + 1)), blk(MTS_NT);
  hipStream_t st = (hipStream_t)a->stream;
  if (vec)
    hipLaunchKernelGGL((k_pq_prepare<DT, VEC>), g, blk, 0, st, mt_seeded(seed), S, a->k, a->ks_b, a->ks_h, a->ks_l, a->Hkv, a->D, a->key_offset,
                       a->n_keys, a->absmax_bits, parts);
  else
    hipLaunchKernelGGL((k_pq_prepare<DT, 1>), g, blk, 0, st, mt_seeded(seed), S, a->k, a->ks_b, a->ks_h, a->ks_l, a->Hkv, a->D, a->key_offset,
                       a->n_keys, a->absmax_bits, parts);
}

extern "C" int sah_pq_keys_absmax(const sah_pq_absmax_args* a) {
  if (!a) return sah_fail(SAH_ENULL, "sah_pq_keys_absmax: args is NULL");
  if (!a->k || !a->absmax_bits) return sah_fail(SAH_ENULL, "sah_pq_keys_absmax: NULL tensor");
  if (a->B <= 0 || a->Hkv <= 0 || a->D <= 0 || a->key_offset < 0 || a->n_keys < 0 || (int64_t)a->B * a->Hkv > 65535)
    return sah_fail(SAH_EINVAL, "sah_pq_keys_absmax: bad B/Hkv/D/key range");
  if (a->n_keys == 0) return SAH_OK;
  sah_timed timed("k_pq_absmax", a->stream);
  switch (a->dtype) {
    case SAH_F32: pq_absmax_launch<SAH_F32>(a); break;
    case SAH_BF16: pq_absmax_launch<SAH_BF16>(a); break;
    case SAH_F16: pq_absmax_launch<SAH_F16>(a); break;
    default: return sah_fail(SAH_EDTYPE, "sah_pq_keys_absmax: dtype %d", a->dtype);
  }
  return sah_launch_status("sah_pq_keys_absmax");
}

// sah_pq_kmeans_assign; with U and the groups' arrival counters (arrivals[g * n_cent], zero) the kernel that sums also carries
// out the update where it can, and says so in *updated
static int pq_assign(const sah_pq_assign_args* a, const pq_update_params* U, uint32_t* arrivals, bool* updated) {
  if (updated) *updated = false;
  if (!a) return sah_fail(SAH_ENULL, "sah_pq_kmeans_assign: args is NULL");
  int rc = pq_check_common("sah_pq_kmeans_assign", a->B, a->Hkv, a->n_sub, a->d_sub, a->n_cent);
  if (rc) return rc;
  if (!a->k || !a->centres || !a->codes) return sah_fail(SAH_ENULL, "sah_pq_kmeans_assign: NULL tensor");
  if ((a->sums == nullptr) != (a->counts == nullptr)) return sah_fail(SAH_EINVAL, "sah_pq_kmeans_assign: sums and counts go together");
  if (a->sums && !a->absmax_bits) return sah_fail(SAH_ENULL, "sah_pq_kmeans_assign: sums need absmax_bits (sah_pq_keys_absmax)");
  if (a->n_keys <= 0) return SAH_OK;
  if (a->key_offset < 0 || a->code_offset < 0 || a->code_pitch < a->code_offset + a->n_keys)
    return sah_fail(SAH_ECAPACITY, "sah_pq_kmeans_assign: code_pitch %lld < code_offset %lld + n_keys %d",
                    (long long)a->code_pitch, (long long)a->code_offset, a->n_keys);
  pq_assign_params P;
  P.k = a->k; P.ks_b = a->ks_b; P.ks_h = a->ks_h; P.ks_l = a->ks_l;
  P.Hkv = a->Hkv; P.n_sub = a->n_sub; P.d_sub = a->d_sub; P.n_cent = a->n_cent;
  P.key_offset = a->key_offset; P.n_keys = a->n_keys;
  P.centres = a->centres;
  P.codes = a->codes; P.code_pitch = a->code_pitch; P.code_offset = a->code_offset;
  P.sums = (long long*)a->sums; P.counts = a->counts;
  P.absmax_bits = a->absmax_bits;
  P.round_dist = a->round_dist;
  P.skip_flag = a->skip_flag;
  hipStream_t st = (hipStream_t)a->stream;
  const bool wide = a->d_sub > PQ_MAX_D;  // no kernel keeps such a key in registers
  if (wide && a->round_dist && a->sums)
    return sah_fail(SAH_ESHAPE, "sah_pq_kmeans_assign: rounded distances with sums need d_sub <= %d", PQ_MAX_D);
  if ((!a->sums && !a->skip_flag && a->n_keys <= 32) || (wide && a->round_dist)) {
    // new keys of a decode step (or, for wide sub-vectors, any number of keys against frozen centres)
    for (int first = 0; first < a->n_keys; first += 32768) {
      pq_assign_params Q = P;
      Q.key_offset += first; Q.code_offset += first;
      Q.n_keys = a->n_keys - first < 32768 ? a->n_keys - first : 32768;
      dim3 gf(a->n_sub, a->B * a->Hkv, Q.n_keys), blk(PQ_NT);
      sah_timed timed("k_pq_assign_few", a->stream);
      switch (a->dtype) {
        case SAH_F32: hipLaunchKernelGGL(k_pq_assign_few<SAH_F32>, gf, blk, 0, st, Q); break;
        case SAH_BF16: hipLaunchKernelGGL(k_pq_assign_few<SAH_BF16>, gf, blk, 0, st, Q); break;
        case SAH_F16: hipLaunchKernelGGL(k_pq_assign_few<SAH_F16>, gf, blk, 0, st, Q); break;
        default: return sah_fail(SAH_EDTYPE, "sah_pq_kmeans_assign: dtype %d", a->dtype);
      }
      if (int rc2 = sah_launch_status("sah_pq_kmeans_assign")) return rc2;
    }
    return SAH_OK;
  }
  if (!wide && !a->sums && !a->skip_flag && a->n_keys <= 512) {  // a block of new keys of a decode plan
    dim3 gb(a->n_sub, a->B * a->Hkv), blk(PQB_NT);
    sah_timed timed("k_pq_assign_block", a->stream);
    switch (a->dtype) {
      case SAH_F32: hipLaunchKernelGGL(k_pq_assign_block<SAH_F32>, gb, blk, 0, st, P); break;
      case SAH_BF16: hipLaunchKernelGGL(k_pq_assign_block<SAH_BF16>, gb, blk, 0, st, P); break;
      case SAH_F16: hipLaunchKernelGGL(k_pq_assign_block<SAH_F16>, gb, blk, 0, st, P); break;
      default: return sah_fail(SAH_EDTYPE, "sah_pq_kmeans_assign: dtype %d", a->dtype);
    }
    return sah_launch_status("sah_pq_kmeans_assign");
  }
  if (!a->round_dist && (wide || (a->n_keys >= 1024 && (a->d_sub == 4 || a->d_sub == 8 || a->d_sub == 16)))) {
    // Lloyd iterations over a whole context: the contraction goes to the matrix cores
    switch (a->dtype) {
      case SAH_F32: return pq_launch_mfma<SAH_F32>(a, P, U, arrivals, updated);
      case SAH_BF16: return pq_launch_mfma<SAH_BF16>(a, P, U, arrivals, updated);
      case SAH_F16: return pq_launch_mfma<SAH_F16>(a, P, U, arrivals, updated);
      default: return sah_fail(SAH_EDTYPE, "sah_pq_kmeans_assign: dtype %d", a->dtype);
    }
  }
  const int per_wg = PQ_NT * PQ_TILES;
  dim3 g(((a->n_keys + per_wg - 1) / per_wg) * a->n_sub, a->B * a->Hkv), blk(PQ_NT);
  sah_timed timed("k_pq_assign", a->stream);
  switch (a->dtype) {
    case SAH_F32: hipLaunchKernelGGL(k_pq_assign<SAH_F32>, g, blk, 0, st, P); break;
    case SAH_BF16: hipLaunchKernelGGL(k_pq_assign<SAH_BF16>, g, blk, 0, st, P); break;
    case SAH_F16: hipLaunchKernelGGL(k_pq_assign<SAH_F16>, g, blk, 0, st, P); break;
    default: return sah_fail(SAH_EDTYPE, "sah_pq_kmeans_assign: dtype %d", a->dtype);
  }
  return sah_launch_status("sah_pq_kmeans_assign");
}

extern "C" int sah_pq_kmeans_assign(const sah_pq_assign_args* a) { return pq_assign(a, nullptr, nullptr, nullptr); }

static int pq_update_launch(const pq_update_params& P, int dtype, void* stream, const char* what) {
  dim3 g(P.n_groups), blk(PQ_NT);
  hipStream_t st = (hipStream_t)stream;
  sah_timed timed("k_pq_update", stream);
  switch (dtype) {
    case SAH_F32: hipLaunchKernelGGL(k_pq_update<SAH_F32>, g, blk, 0, st, P); break;
    case SAH_BF16: hipLaunchKernelGGL(k_pq_update<SAH_BF16>, g, blk, 0, st, P); break;
    case SAH_F16: hipLaunchKernelGGL(k_pq_update<SAH_F16>, g, blk, 0, st, P); break;
    default: return sah_fail(SAH_EDTYPE, "%s: dtype %d", what, dtype);
  }
  return sah_launch_status(what);
}

extern "C" int sah_pq_kmeans_update(const sah_pq_update_args* a) {
  if (!a) return sah_fail(SAH_ENULL, "sah_pq_kmeans_update: args is NULL");
  int rc = pq_check_common("sah_pq_kmeans_update", a->B, a->Hkv, a->n_sub, a->d_sub, a->n_cent);
  if (rc) return rc;
  if (!a->k || !a->centres || !a->sums || !a->counts || !a->reseed_idx || !a->shift2 || !a->state || !a->absmax_bits)
    return sah_fail(SAH_ENULL, "sah_pq_kmeans_update: NULL tensor");
  pq_update_params P = {};
  P.k = a->k; P.ks_b = a->ks_b; P.ks_h = a->ks_h; P.ks_l = a->ks_l;
  P.Hkv = a->Hkv; P.n_sub = a->n_sub; P.d_sub = a->d_sub; P.n_cent = a->n_cent; P.key_offset = a->key_offset;
  P.centres = a->centres; P.sums = (long long*)a->sums; P.counts = (int*)a->counts;  // read only: P.clear is 0
  P.reseed_idx = a->reseed_idx; P.n_keys = 1;
  P.absmax_bits = a->absmax_bits;
  P.shift2 = a->shift2; P.tol = a->tol; P.state = a->state;
  P.n_groups = a->B * a->Hkv * a->n_sub;
  return pq_update_launch(P, a->dtype, a->stream, "sah_pq_kmeans_update");
}

extern "C" int sah_pq_kmeans(const sah_pq_kmeans_args* a) {
  if (!a) return sah_fail(SAH_ENULL, "sah_pq_kmeans: args is NULL");
  int rc = pq_check_common("sah_pq_kmeans", a->B, a->Hkv, a->n_sub, a->d_sub, a->n_cent);
  if (rc) return rc;
  if (!a->k || !a->centres || !a->codes || !a->sums || !a->counts || !a->shift2 || !a->state || !a->absmax_bits ||
      (!a->given_start && !a->start_idx))
    return sah_fail(SAH_ENULL, "sah_pq_kmeans: NULL tensor");
  if (a->n_keys <= 0 || a->key_offset < 0 || a->max_iter < 0)
    return sah_fail(SAH_EINVAL, "sah_pq_kmeans: n_keys must be > 0, key_offset and max_iter >= 0");
  if (a->code_offset < 0 || a->code_pitch < a->code_offset + a->n_keys)
    return sah_fail(SAH_ECAPACITY, "sah_pq_kmeans: code_pitch %lld < code_offset %lld + n_keys %d", (long long)a->code_pitch,
                    (long long)a->code_offset, a->n_keys);
  const int n_groups = a->B * a->Hkv * a->n_sub;
  hipStream_t st = (hipStream_t)a->stream;
  sah_pq_absmax_args m = {a->k, a->ks_b, a->ks_h, a->ks_l, a->dtype, a->B, a->Hkv, a->n_sub * a->d_sub, a->key_offset, a->n_keys,
                          a->absmax_bits, a->stream};
  if (!a->given_start) {
    if (a->n_keys < a->n_cent) return sah_fail(SAH_EINVAL, "sah_pq_kmeans: fewer keys than centres");
    if ((int64_t)a->B * a->Hkv > 65535) return sah_fail(SAH_EINVAL, "sah_pq_kmeans: more than 65535 heads");
    const pq_start_params sp = {(int64_t)n_groups * a->n_cent, a->n_cent, a->n_keys, (double)a->n_keys / (double)a->n_cent, a->start_idx};
    sah_timed timed("k_pq_start", a->stream);
    dim3 g(n_groups), blk(PQG_NT);
#define SAH_PQG(DTC)                                                                                                          \
  do {                                                                                                                        \
    pq_prepare_launch<DTC>(&m, sp, (uint32_t)a->start_seed);                                                                  \
    hipLaunchKernelGGL(k_pq_gather<DTC>, g, blk, 0, st, a->k, a->ks_b, a->ks_h, a->ks_l, a->Hkv, a->n_sub, a->d_sub, a->n_cent, \
                       a->key_offset, a->start_idx, a->centres);                                                              \
  } while (0)
    switch (a->dtype) {
      case SAH_F32: SAH_PQG(SAH_F32); break;
      case SAH_BF16: SAH_PQG(SAH_BF16); break;
      case SAH_F16: SAH_PQG(SAH_F16); break;
      default: return sah_fail(SAH_EDTYPE, "sah_pq_kmeans: dtype %d", a->dtype);
    }
#undef SAH_PQG
    if ((rc = sah_launch_status("sah_pq_kmeans(start)"))) return rc;
  } else if ((rc = sah_pq_keys_absmax(&m))) {
    return rc;
  }
  sah_pq_assign_args as = {};
  as.k = a->k; as.ks_b = a->ks_b; as.ks_h = a->ks_h; as.ks_l = a->ks_l;
  as.dtype = a->dtype; as.B = a->B; as.Hkv = a->Hkv; as.n_sub = a->n_sub; as.d_sub = a->d_sub; as.n_cent = a->n_cent;
  as.key_offset = a->key_offset; as.n_keys = a->n_keys; as.centres = a->centres;
  as.codes = a->codes; as.code_pitch = a->code_pitch; as.code_offset = a->code_offset;
  as.sums = a->sums; as.counts = a->counts; as.skip_flag = a->state + 2; as.stream = a->stream; as.absmax_bits = a->absmax_bits;
  pq_update_params P = {};
  P.k = a->k; P.ks_b = a->ks_b; P.ks_h = a->ks_h; P.ks_l = a->ks_l;
  P.Hkv = a->Hkv; P.n_sub = a->n_sub; P.d_sub = a->d_sub; P.n_cent = a->n_cent; P.key_offset = a->key_offset;
  P.centres = a->centres; P.sums = (long long*)a->sums; P.counts = a->counts;
  P.reseed_seed = (uint32_t)a->reseed_seed; P.n_keys = a->n_keys; P.clear = 1;
  const int64_t n_all = (int64_t)n_groups * a->n_cent;
  if (a->reseed_idx && a->max_iter) {
    sah_timed timed("k_pq_reseed", a->stream);
    hipLaunchKernelGGL(k_pq_reseed, dim3(1), dim3(MTS_NT), 0, st, mt_seeded((uint32_t)a->reseed_seed), n_all * a->max_iter, a->n_keys,
                       a->reseed_idx);
    if ((rc = sah_launch_status("sah_pq_kmeans(reseed)"))) return rc;
  }
  P.absmax_bits = a->absmax_bits;
  P.shift2 = a->shift2; P.tol = a->tol; P.state = a->state; P.n_groups = n_groups;
  for (int it = 0; it < a->max_iter; ++it) {
    P.reseed_first = it * n_all;
    P.reseed_idx = a->reseed_idx ? a->reseed_idx + it * n_all : nullptr;
    bool updated;
    if ((rc = pq_assign(&as, &P, a->given_start ? nullptr : (uint32_t*)a->start_idx, &updated))) return rc;
    if (!updated && (rc = pq_update_launch(P, a->dtype, a->stream, "sah_pq_kmeans"))) return rc;
  }
  return SAH_OK;
}

extern "C" int64_t sah_pq_adc_lut_bytes(int32_t B, int32_t Hq, int32_t Hkv, int32_t Lq, int32_t n_sub, int32_t n_cent,
                                        int32_t dtype) {
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || Lq <= 0 || n_sub <= 0 || n_cent <= 0 || Hq % Hkv) return 0;
  const int nq = dtype == SAH_F32 ? 2 : 4;
  const int n_vg = ((Hq / Hkv) * Lq + nq - 1) / nq;
  return (int64_t)B * Hkv * n_vg * n_sub * n_cent * 8;
}

extern "C" int sah_pq_adc_scores(const sah_pq_adc_args* a) {
  if (!a) return sah_fail(SAH_ENULL, "sah_pq_adc_scores: args is NULL");
  int rc = pq_check_common("sah_pq_adc_scores", a->B, a->Hkv, a->n_sub, a->d_sub, a->n_cent);
  if (rc) return rc;
  if (!a->q || !a->centres || !a->codes || !a->keys_out) return sah_fail(SAH_ENULL, "sah_pq_adc_scores: NULL tensor");
  if (a->Hq <= 0 || a->Lq <= 0 || a->Hq % a->Hkv) return sah_fail(SAH_EINVAL, "sah_pq_adc_scores: bad Hq/Lq");
  if (a->n_sub * a->n_cent > ADC_MAX_LUT) return sah_fail(SAH_ESHAPE, "sah_pq_adc_scores: n_sub*n_cent > %d", ADC_MAX_LUT);
  if (a->n_cand <= 0) return SAH_OK;
  if (a->code_pitch < a->n_cand || a->key_pitch < a->n_cand) return sah_fail(SAH_ECAPACITY, "sah_pq_adc_scores: pitch < n_cand");
  pq_adc_params P;
  P.q = a->q; P.qs_b = a->qs_b; P.qs_h = a->qs_h; P.qs_l = a->qs_l;
  P.Hq = a->Hq; P.Hkv = a->Hkv; P.Lq = a->Lq; P.n_sub = a->n_sub; P.d_sub = a->d_sub; P.n_cent = a->n_cent;
  P.centres = a->centres; P.codes = a->codes; P.code_pitch = a->code_pitch; P.n_cand = a->n_cand;
  P.centres_narrow = (a->dtype != SAH_F32 && a->d_sub % 8 == 0 && ((uintptr_t)a->centres_narrow % 16) == 0) ? a->centres_narrow : nullptr;
  P.keys_out = a->keys_out; P.key_pitch = a->key_pitch;
  const int nvec = (a->Hq / a->Hkv) * a->Lq;
  const int nq = a->dtype == SAH_F32 ? 2 : 4;
  const int n_vg = (nvec + nq - 1) / nq;
  if (n_vg > 65535) return sah_fail(SAH_ESHAPE, "sah_pq_adc_scores: too many query vectors per KV head");
  hipStream_t st = (hipStream_t)a->stream;
  const int wgs_per_head = (a->n_cand + ADC_KEYS - 1) / ADC_KEYS;
  dim3 g(wgs_per_head, a->B * a->Hkv, n_vg), blk(PQ_NT);
  if (wgs_per_head <= ADC_OWN_LUT_WGS && a->n_sub * a->d_sub <= ADC_MAX_HEAD_DIM) {
    // short contexts: no table in memory, no second launch
    sah_timed timed("k_pq_adc", a->stream);
    switch (a->dtype) {
      case SAH_F32: rc = adc_launch<SAH_F32, true>(P, nullptr, g, st); break;
      case SAH_BF16: rc = adc_launch<SAH_BF16, true>(P, nullptr, g, st); break;
      case SAH_F16: rc = adc_launch<SAH_F16, true>(P, nullptr, g, st); break;
      default: return sah_fail(SAH_EDTYPE, "sah_pq_adc_scores: dtype %d", a->dtype);
    }
    if (rc) return rc;
    return sah_launch_status("sah_pq_adc_scores");
  }
  const int64_t need = (int64_t)a->B * a->Hkv * n_vg * a->n_sub * a->n_cent * 8;
  if (!a->lut || a->lut_bytes < need)
    return sah_fail(SAH_ECAPACITY, "sah_pq_adc_scores: lut holds %lld bytes, need %lld", (long long)(a->lut ? a->lut_bytes : 0),
                    (long long)need);
  {
    dim3 gl(a->n_sub, a->B * a->Hkv, n_vg);
    sah_timed timed("k_pq_lut", a->stream);
    switch (a->dtype) {
      case SAH_F32: hipLaunchKernelGGL(k_pq_lut<SAH_F32>, gl, blk, 0, st, P, a->lut); break;
      case SAH_BF16: hipLaunchKernelGGL(k_pq_lut<SAH_BF16>, gl, blk, 0, st, P, a->lut); break;
      case SAH_F16: hipLaunchKernelGGL(k_pq_lut<SAH_F16>, gl, blk, 0, st, P, a->lut); break;
      default: return sah_fail(SAH_EDTYPE, "sah_pq_adc_scores: dtype %d", a->dtype);
    }
    rc = sah_launch_status("sah_pq_adc_scores(lut)");
    if (rc) return rc;
  }
  sah_timed timed("k_pq_adc", a->stream);
  switch (a->dtype) {
    case SAH_F32: rc = adc_launch<SAH_F32, false>(P, a->lut, g, st); break;
    case SAH_BF16: rc = adc_launch<SAH_BF16, false>(P, a->lut, g, st); break;
    default: rc = adc_launch<SAH_F16, false>(P, a->lut, g, st); break;
  }
  if (rc) return rc;
  return sah_launch_status("sah_pq_adc_scores");
}
