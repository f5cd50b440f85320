// Masked-softmax attention of many query vectors per KV head on the matrix cores.
//
// In a question pass every KV head has G x Lq mask rows, each with its own columns. Gathering them row by row
// (k_sparse_attn) reads K and V once per entry: 1536 rows of 2278 entries, head_dim 128, are 1.8 GB through the caches,
// 195 us. Together the rows of a head touch nearly every key, so here the whole of K and V passes once per 128 (or 64)
// rows, the products run dense on the matrix cores and the rows' bitmaps decide which entries count: 63 us (64 with the
// causal mask) and 9 for the merge. Work grows with rows x keys instead of rows x entries: see members_attention_pays().
//
// A workgroup: 4 waves over stages of 64 keys, K and V staged in LDS by loads that write there themselves (two buffers,
// the next stage under way while the current one is worked on; through registers, with V transposed on the way, 87 us). A
// wave owns 32 mask rows: S^T = K Q^T puts row j in lane j (16 of a tile's 32 keys in lane j, 16 in lane j + 32), so
// maximum, weights and sums of a row need one exchange between two lanes, and the weights are where the second product,
// O^T = V^T P^T, wants its B operand, with the key slots of a 16-key step taken in the order [0-3][8-11] / [4-7][12-15]:
// the transposing LDS reads of V follow that order. The weights enter the second product as 16-bit terms that
// together are the fp32 weight (qa_weights), so that nothing but the output is rounded to the storage type. Before that
// rounding the result is off by 2.4e-7 (2-norm, 4096 keys, bf16; fp16 3.5e-7) where the gather's is by 1.6e-7 (1.8e-7): the
// order of the fp32 sums. With two terms for bf16 2.3e-6.
// What bounds it: per wave and 32-key tile 32 matrix instructions (fp16: 24; 1024 and 768 cycles) and about 190 vector ones
// with 17 exponentials (150; 960 and 800 cycles), which overlap little with two waves on a SIMD, each issuing one in eight cycles. The third term costs 3 us of a pass of 244
// with the causal mask.
// Keys are split over workgroups; the partial results (m, l, acc) are merged by a second kernel.
#include "sah_common.h"
#include "sah_attn.h"

#define QA_NT 256
#define QA_NW (QA_NT / SAH_WAVE)
#define QA_STAGE 64      // keys per LDS stage: two 32-key tiles
#define QA_MIN_WGS 512   // keys are split until there are this many workgroups (two per CU: one round) ...
#define QA_MIN_STAGES 8  // ... of at least this many stages (a partial result costs as much as half a stage to write and merge)
typedef uint32_t qa_u4 __attribute__((ext_vector_type(4)));
typedef uint32_t qa_u2 __attribute__((ext_vector_type(2)));
typedef qa_u2 qa_u2_any __attribute__((aligned(2)));  // 8 bytes at an address that is only element aligned
typedef qa_u4 qa_u4_any __attribute__((aligned(2)));
typedef qa_u2 qa_u2_word __attribute__((aligned(4)));

struct qa_params {
  int n_split;         // key splits (workgroups along the keys)
  int stages_per_split;
  int row_tiles;       // workgroups along the rows of a KV head
};

// 16 bytes per lane from memory straight into LDS: the wave's 64 units land one after the other at `lds` (wave-uniform)
__device__ __forceinline__ void qa_load_lds(const void* p, void* lds) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)p, (__attribute__((address_space(3))) void*)lds, 16, 0, 0);
#else
  (void)p; (void)lds;
#endif
}
// Transposing LDS read, one 4 x 16 block of 16-bit elements per 16 lanes (layout checked on the hardware): lane l hands in
// the address of row (l % 16) / 4, columns 4 (l % 4) .. + 3 and receives column l % 16, rows 0 .. 3.
__device__ __forceinline__ qa_u2 qa_read_tr(const uint16_t* lds) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef short v4s __attribute__((ext_vector_type(4)));
  const v4s r = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s*)lds);
  return __builtin_bit_cast(qa_u2, r);
#else
  return *(const qa_u2*)lds;
#endif
}

// How far a row's maximum may rise, in powers of two, before the row is rescaled: the weights are then at most 2^SLACK
// relative to the maximum in use, which costs a floating-point sum nothing. A row's maximum rises in most of the few
// tiles a workgroup sees; it rises by 2^8 in one or two of them.
// The weights enter the second product in 16-bit terms that together are the fp32 weight: three for bf16 (8 bits each),
// two for fp16 (11 bits and a sign each), whose range is used to its upper end, the weights scaled by 2^SCALE: what its
// smallest number, 2^-24, then cuts off is 2^-39 of the row's largest weight or less.
template <int DT> struct qa_weights {
  static constexpr int TERMS = DT == SAH_BF16 ? 3 : 2;
  static constexpr float SLACK = DT == SAH_BF16 ? 8.0f : 1.0f;
  static constexpr float SCALE = DT == SAH_BF16 ? 0.0f : 14.0f;     // SLACK + SCALE <= 15
  static constexpr float UNSCALE = DT == SAH_BF16 ? 1.0f : 0x1p-14f;
};

// RW: waves along the rows (4: 128 rows a workgroup; 2: 64 rows, and the two 32-key tiles of a stage go to two waves)
// AM: additive mask. DENSE: every key counts (no bitmap).
template <int DT, int D, int RW, bool AM, bool DENSE>
__global__ __launch_bounds__(QA_NT, 2) void k_members_attn_mfma(att_params P, qa_params Q) {
  sah_touch_kernargs<sizeof(att_params) + sizeof(qa_params)>();
  constexpr int KW = QA_NW / RW;      // waves along the keys of a stage
  constexpr int KS = D / 16;          // matrix steps of the first product
  constexpr int DTL = D / 32;         // 32-row tiles of the output
  // LDS: K and V as they lie in memory, a row per key, its 16-byte units permuted against bank conflicts. K: unit c of key
  // j at place c ^ (j % 16) (head_dim 64: c ^ (j / 2 % 8)), so that 16 rows read at one c meet every bank once; V: groups
  // of four units (32 dims) at place u ^ (j % 4) (head_dim 64: u ^ (j / 2 % 2)), so that the four rows of a transposing
  // read do. The permutation is applied to the addresses read from memory; the writes to LDS are the loads themselves.
  constexpr int SE = QA_STAGE * D;        // elements of a staged K or V
  constexpr int KPW = SAH_WAVE / (D / 8); // keys per load instruction of a wave
  constexpr int UW = QA_STAGE / KPW / QA_NW;  // load instructions per wave, matrix and stage
  constexpr int SH = D == 128 ? 0 : 1;
  // (an array each: the compiler then knows that what is read is not what the loads under way will write)
  __shared__ __align__(16) uint16_t s_k0[SE], s_k1[SE], s_v0[SE], s_v1[SE];
  __shared__ float4 s_seed[16];                    // bit t of the index: element t is 0 (else -inf)
  const int tid = threadIdx.x;
  const int lane = tid & (SAH_WAVE - 1);
  const int wave = sah_wave_id();
  const int i32 = lane & 31, g = lane >> 5;
  // workgroup -> (KV head, key split, row tile): the row tiles of a stream of K and V take adjacent slots of one XCD
  const int slot = blockIdx.x / ATT_XCDS;
  const int stream = (slot / Q.row_tiles) * ATT_XCDS + (int)(blockIdx.x % ATT_XCDS);
  const int G = P.Hq / P.Hkv;
  const int n_bhk = P.rows.n_rows / (G * P.Lq);
  if (stream >= n_bhk * Q.n_split) return;
  const int rt = slot % Q.row_tiles;
  const int split = stream % Q.n_split;
  const int bhk = stream / Q.n_split;
  const int hk = bhk % P.Hkv, b = bhk / P.Hkv;
  const int nvec = G * P.Lq;
  const int rw = wave % RW, kw = wave / RW;

  // this lane's mask row (vector v of the head); lanes beyond the last repeat it and store nothing
  const int v_own = (rt * RW + rw) * 32 + i32;
  const bool rows_live = (rt * RW + rw) * 32 < nvec;  // uniform across the wave
  const bool live = v_own < nvec;
  const int v = live ? v_own : nvec - 1;
  const int h = hk * G + v / P.Lq, qi = v % P.Lq;
  const int r = (b * P.Hq + h) * P.Lq + qi;
  uint4 qf[KS];
  {
    const uint16_t* qp = (const uint16_t*)P.q + (int64_t)b * P.qs_b + (int64_t)h * P.qs_h + (int64_t)qi * P.qs_l + 8 * g;
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[s] = *(const uint4*)(qp + 16 * s);
  }
  const uint32_t* bm = DENSE ? nullptr : P.rows.bitmap + (int64_t)r * P.rows.n_words;
  const uint16_t* am = AM ? (const uint16_t*)P.amask + (int64_t)b * P.ms_b + (int64_t)h * P.ms_h + (int64_t)qi * P.ms_l + 4 * g : nullptr;

  const int n_stages = (P.Lk + QA_STAGE - 1) / QA_STAGE;
  const int st0 = split * Q.stages_per_split;
  const int st1 = st0 + Q.stages_per_split < n_stages ? st0 + Q.stages_per_split : n_stages;

  // A stage's rows on their way to LDS: per load instruction a scalar base (the stage, the instruction's keys) and a
  // per-lane byte offset that stays the same, recomputed for the stage in which K ends: keys past it repeat the last one,
  // and no bitmap has them.
  const char* kbase = (const char*)P.k + ((int64_t)b * P.ks_b + (int64_t)hk * P.ks_h) * 2;
  const char* vbase = (const char*)P.v + ((int64_t)b * P.vs_b + (int64_t)hk * P.vs_h) * 2;
  const int lkey = lane / (D / 8), lpos = lane % (D / 8);  // this lane's key within an instruction, its 16-byte place in the row
  uint32_t ko[UW], vo[UW];
  auto offsets = [&](int keys_left) {
#pragma unroll
    for (int u = 0; u < UW; ++u) {
      const int key = (wave * UW + u) * KPW + lkey;
      const int src = key < keys_left ? key : keys_left - 1;
      ko[u] = (uint32_t)src * (uint32_t)P.ks_l * 2u + 16u * (lpos ^ ((key >> SH) & (D / 8 - 1)));
      vo[u] = (uint32_t)src * (uint32_t)P.vs_l * 2u + 16u * (lpos ^ (4 * ((key >> SH) & (D / 32 - 1))));
    }
  };
  // the bits and the mask of a stage's tiles (this wave's), requested before they are used
  constexpr int TW = KW == 1 ? 2 : 1;  // tiles of a stage per wave
  uint32_t bits[TW];
  auto fetch_bits = [&](int st) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < TW; ++t) {
      const int wi = 2 * st + (KW == 1 ? t : kw);
      bits[t] = DENSE ? sah_range_bits(wi, 0, P.Lk) : (wi < P.rows.n_words ? bm[wi] : 0u);
    }
  };
  // Whether a tile's mask is all zeros, as most are, is asked in whole lines: four lanes take the 64 bytes of a row, an
  // instruction 16 rows. A lane's own elements (16 bytes a row and instruction: four times the cache lines, 1536 rows x 32768
  // keys under the causal mask 72 us instead of 64) are fetched where that answer is no, and ahead of their use once it has
  // been no in the stage before (a bias on every key: 17 us more than the causal mask).
  qa_u4 mv[AM ? TW : 1][2];  // lines of rows lane / 4 and 16 + lane / 4, or (own, uniform) this lane's elements
  bool own = false;
  const uint16_t* az[2] = {nullptr, nullptr};
  if (AM) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int vz_own = (rt * RW + rw) * 32 + 16 * i + (lane >> 2);
      const int vz = vz_own < nvec ? vz_own : nvec - 1;
      az[i] = (const uint16_t*)P.amask + (int64_t)b * P.ms_b + (int64_t)(hk * G + vz / P.Lq) * P.ms_h + (int64_t)(vz % P.Lq) * P.ms_l + 8 * (lane & 3);
    }
  }
  auto fetch_own = [&](int wi, qa_u4 (&m4)[2]) __attribute__((always_inline)) {
    const int key0 = wi * 32;
    qa_u2 m[4];
    if (key0 + 32 <= P.Lk) {  // uniform
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) m[q4] = *(const qa_u2_any*)(am + key0 + 8 * q4);
    } else {
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        uint32_t two[2] = {0u, 0u};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int kk = key0 + 8 * q4 + e;
          if (kk + 4 * g < P.Lk) two[e >> 1] |= (uint32_t)am[kk] << (16 * (e & 1));
        }
        m[q4] = qa_u2{two[0], two[1]};
      }
    }
    m4[0] = qa_u4{m[0].x, m[0].y, m[1].x, m[1].y};
    m4[1] = qa_u4{m[2].x, m[2].y, m[3].x, m[3].y};
  };
  auto fetch_mask = [&](int st, int t) __attribute__((always_inline)) {
    const int wi = 2 * st + (KW == 1 ? t : kw);
    if (own) {
      fetch_own(wi, mv[t]);
    } else {
#pragma unroll
      for (int i = 0; i < 2; ++i) mv[t][i] = *(const qa_u4_any*)(az[i] + wi * 32);
    }
  };
  auto fetch = [&](int st, int buf) __attribute__((always_inline)) {
    if ((st + 1) * QA_STAGE > P.Lk) offsets(P.Lk - st * QA_STAGE);  // uniform: the last stage
    const char* ks = kbase + (int64_t)st * QA_STAGE * P.ks_l * 2;
    const char* vs = vbase + (int64_t)st * QA_STAGE * P.vs_l * 2;
#pragma unroll
    for (int u = 0; u < UW; ++u) qa_load_lds(ks + ko[u], (buf ? s_k1 : s_k0) + (wave * UW + u) * KPW * D);
#pragma unroll
    for (int u = 0; u < UW; ++u) qa_load_lds(vs + vo[u], (buf ? s_v1 : s_v0) + (wave * UW + u) * KPW * D);
  };
  // where this lane reads. K: key row i32 of a tile, unit 2 s + g. V (transposed): for the four keys from 4 g on of a
  // 16-key step, row (lane % 16) / 4 of them, dims 32 t + 16 (lane / 16 % 2) + 4 (lane % 4) .. + 3
  const int k_from = i32 * D + 8 * (g ^ ((i32 >> SH) & (D / 8 - 1)));
  int v_from[DTL];
  {
    const int row = 4 * g + ((lane & 15) >> 2);
#pragma unroll
    for (int t = 0; t < DTL; ++t) v_from[t] = row * D + 32 * (t ^ ((row >> SH) & (D / 32 - 1))) + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  }

  // running maximum of the logits, denominator, output tiles
  constexpr float LOG2E = 1.4426950408889634f;
  float m_run = -INFINITY, l_run = 0.f;
  sah_f32x16 acc[DTL];
#pragma unroll
  for (int t = 0; t < DTL; ++t)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[t][e] = 0.f;

  // biased: the tile's mask is not all zeros (uniform)
  auto tile = [&](int buf, int t32, uint32_t word, bool biased, const qa_u4 (&am16)[2]) __attribute__((always_inline)) {
    if (__ballot(word != 0u) == 0) return;  // no row of this wave has a column here
    // element e of the product is key 8 (e / 4) + 4 g + e % 4 of the tile; it starts at 0 or, where the row does not hold
    // the key, at -inf (four elements per table entry)
    const uint32_t mine = g ? word : word << 4;
    sah_f32x16 s;
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      const float4 c = *(const float4*)((const char*)s_seed + ((mine >> (8 * q4)) & 0xf0u));
      s[4 * q4] = c.x; s[4 * q4 + 1] = c.y; s[4 * q4 + 2] = c.z; s[4 * q4 + 3] = c.w;
    }
    const uint16_t* kp = (buf ? s_k1 : s_k0) + t32 * 32 * D;
#pragma unroll
    for (int st = 0; st < KS; ++st) s = sah_mfma_32x32x16<DT>(*(const uint4*)(kp + (k_from ^ (16 * st))), qf[st], s);
    // most tiles of a mask are zeros: the maximum is then kept in the mask's scale, the products stay as they are
    if (AM) {
      if (biased) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const uint32_t two = am16[e >> 3][(e >> 1) & 3];
          float a4;
          if (DT == SAH_BF16) a4 = sah_bits_to_float((e & 1) ? (two & 0xffff0000u) : (two << 16));
          else a4 = sah_f16_to_float((uint16_t)(two >> (16 * (e & 1))));
          s[e] = fmaf(s[e], P.scaling, a4);
        }
      }
    }
    float mx = s[0];
#pragma unroll
    for (int e = 1; e < 16; ++e) mx = fmaxf(mx, s[e]);
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    if (!biased) mx *= P.scaling;
    // (-inf - -inf is NaN: no rise)
    if (__ballot((mx - m_run) * LOG2E > qa_weights<DT>::SLACK) != 0) {  // uniform: some row's maximum has risen too far
      const float m_new = fmaxf(m_run, mx);
      const float up = m_run == -INFINITY ? 0.f : exp2f((m_run - m_new) * LOG2E);
      m_run = m_new;
      l_run *= up;
#pragma unroll
      for (int t = 0; t < DTL; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[t][e] *= up;
    }
    float z[16];
    if (biased) {
      const float m_use = m_run == -INFINITY ? 0.f : m_run;
#pragma unroll
      for (int e = 0; e < 16; ++e) z[e] = __builtin_amdgcn_exp2f(fmaf(s[e] - m_use, LOG2E, qa_weights<DT>::SCALE));
    } else {
      // a row whose every key so far is hidden has a maximum near the type's lowest value, and none here if it holds no
      // key of this tile: kept in range, so that -inf products come to 0
      const float mc = fmaxf(m_run, -1e37f) * LOG2E - qa_weights<DT>::SCALE;
      const float c_exp = P.scaling * LOG2E;
#pragma unroll
      for (int e = 0; e < 16; ++e) z[e] = __builtin_amdgcn_exp2f(fmaf(s[e], c_exp, -mc));
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) l_run += z[e];
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      uint4 va[DTL];
#pragma unroll
      for (int t = 0; t < DTL; ++t) {
        const uint16_t* vp = (buf ? s_v1 : s_v0) + (t32 * 32 + 16 * st) * D + v_from[t];
        const qa_u2 a0 = qa_read_tr(vp), a1 = qa_read_tr(vp + 8 * D);
        va[t] = make_uint4(a0.x, a0.y, a1.x, a1.y);
      }
      constexpr int TERMS = qa_weights<DT>::TERMS;
      uint32_t term[TERMS][4];
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        float p0 = z[8 * st + 2 * p], p1 = z[8 * st + 2 * p + 1];
#pragma unroll
        for (int i = 0; i < TERMS; ++i) {
          term[i][p] = sah_pack2_hw<DT>(p0, p1);
          if (i + 1 == TERMS) break;
          sah_keep(term[i][p]);  // taken apart as it is, instead of converted a second time
          if (DT == SAH_BF16) {
            p0 -= sah_bits_to_float(term[i][p] << 16);
            p1 -= sah_bits_to_float(term[i][p] & 0xffff0000u);
          } else {
            p0 -= sah_f16_to_float((uint16_t)term[i][p]);
            p1 -= sah_f16_to_float((uint16_t)(term[i][p] >> 16));
          }
        }
      }
#pragma unroll
      for (int i = 0; i < TERMS; ++i) {
        const uint4 pt = make_uint4(term[i][0], term[i][1], term[i][2], term[i][3]);
#pragma unroll
        for (int t = 0; t < DTL; ++t) acc[t] = sah_mfma_32x32x16<DT>(va[t], pt, acc[t]);
      }
    }
  };
  auto stage = [&](int buf, int st) __attribute__((always_inline)) {  // buf: a constant in the loop below, LDS offsets are immediates
    uint32_t w[TW];
    bool biased[TW];  // uniform: the tile's mask is not all zeros
    bool any_biased = false;
#pragma unroll
    for (int t = 0; t < TW; ++t) {
      w[t] = bits[t];
      biased[t] = false;
      if (AM) {
        uint32_t any = 0u;
#pragma unroll
        for (int i = 0; i < 2; ++i) any |= mv[t][i].x | mv[t][i].y | mv[t][i].z | mv[t][i].w;
        biased[t] = __ballot((any & 0x7fff7fffu) != 0u) != 0;
        any_biased = any_biased || biased[t];
      }
    }
    const bool was_own = own;
    const bool more = st + 1 < st1;
    if (more) {
      fetch_bits(st + 1);
      own = any_biased || (st + 2) * QA_STAGE > P.Lk;  // the stage in which the mask's rows end goes by elements
      fetch(st + 1, buf ^ 1);  // the other buffer: read for the last time before the previous barrier
    }
#pragma unroll
    for (int t = 0; t < TW; ++t) {
      qa_u4 am_now[2];
      if (AM) {
        am_now[0] = mv[t][0];
        am_now[1] = mv[t][1];
        if (biased[t] && !was_own) fetch_own(2 * st + (KW == 1 ? t : kw), am_now);
        if (more) fetch_mask(st + 1, t);
      }
      if (rows_live) tile(buf, KW == 1 ? t : kw, w[t], biased[t], am_now);
    }
    sah_stores_done();  // this wave's loads into LDS have landed
    __syncthreads();
  };

  if (tid < 16) s_seed[tid] = make_float4(tid & 1 ? 0.f : -INFINITY, tid & 2 ? 0.f : -INFINITY, tid & 4 ? 0.f : -INFINITY, tid & 8 ? 0.f : -INFINITY);
  offsets(QA_STAGE);
  fetch_bits(st0);
  if (AM) {
    own = (st0 + 1) * QA_STAGE > P.Lk;
#pragma unroll
    for (int t = 0; t < TW; ++t) fetch_mask(st0, t);
  }
  fetch(st0, 0);  // every split has at least one stage
  sah_stores_done();
  __syncthreads();
  for (int st = st0; st < st1; st += 2) {
    stage(0, st);
    if (st + 1 < st1) stage(1, st + 1);
  }

  l_run += __shfl_xor(l_run, 32);
  if (KW == 2) {
    // the second wave of a row hands its share over through LDS (free since the last barrier)
    static_assert(SE * 2 == 16 * DTL * SAH_WAVE * 4, "a wave's output tiles fill a staged K");
    float* s_f = (float*)(rw ? s_k1 : s_k0);
    float* s_ml = (float*)s_v0 + rw * 2 * SAH_WAVE;
    if (kw == 1) {
#pragma unroll
      for (int t = 0; t < DTL; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) s_f[(16 * t + e) * SAH_WAVE + lane] = acc[t][e];
      s_ml[lane] = m_run;
      s_ml[SAH_WAVE + lane] = l_run;
    }
    __syncthreads();
    if (kw == 1) return;
    const float m2 = s_ml[lane], l2 = s_ml[SAH_WAVE + lane];
    const float m_new = fmaxf(m_run, m2);
    const float up1 = m_run == -INFINITY ? 0.f : exp2f((m_run - m_new) * LOG2E);
    const float up2 = m2 == -INFINITY ? 0.f : exp2f((m2 - m_new) * LOG2E);
    m_run = m_new;
    l_run = l_run * up1 + l2 * up2;
#pragma unroll
    for (int t = 0; t < DTL; ++t)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[t][e] = acc[t][e] * up1 + s_f[(16 * t + e) * SAH_WAVE + lane] * up2;
  }
  if (!live) return;
  // every entry of unit weight carries the factor unit_inv_w, in numerator and denominator
  const float unit = P.unit_inv_w * qa_weights<DT>::UNSCALE;
  float* w = P.work + ((int64_t)r * Q.n_split + split) * (D + 2);
  if (g == 0) {
    w[0] = m_run;
    w[1] = l_run * unit;
  }
#pragma unroll
  for (int t = 0; t < DTL; ++t) {
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      float2* o = (float2*)(w + 2 + 32 * t + 8 * q4 + 4 * g);
      o[0] = make_float2(acc[t][4 * q4] * unit, acc[t][4 * q4 + 1] * unit);
      o[1] = make_float2(acc[t][4 * q4 + 2] * unit, acc[t][4 * q4 + 3] * unit);
    }
  }
}

// Merges a row's partial results. The products above meet every key of a stage, so a key that is not finite reaches rows
// that do not hold it (-inf plus a NaN product in the logits, 0 times it in the second product); what reaches a row is not
// finite either. Such a row, and one whose sums left the range of fp32, is done again entry by entry: its result is the
// gather's, from the keys it holds alone.
template <int DT, int D>
__global__ __launch_bounds__(D) void k_members_merge(att_params P, int n_split) {
  constexpr int NW = D / SAH_WAVE;
  __shared__ float s_sm[ATT_MAX_SPLIT];
  __shared__ float s_sl[ATT_MAX_SPLIT];
  __shared__ float s_m[NW];
  __shared__ float s_l[NW];
  __shared__ float s_acc[NW][D];
  const int r = blockIdx.x;
  const int qi = r % P.Lq;
  const int h = (r / P.Lq) % P.Hq;
  const int b = r / (P.Lq * P.Hq);
  float a, M, L;
  att_merge_splits<DT, D>(P.work, n_split, r, s_sm, s_sl, a, M, L);
  if (__syncthreads_or(!(fabsf(a) < INFINITY) || !(fabsf(L) < INFINITY))) {
    int cnt = P.dense ? P.Lk : P.rows.cnt[r];
    if (!P.dense && cnt > P.rows.cap) cnt = P.rows.cap;
    const int* cols = P.dense ? nullptr : P.rows.cols + (int64_t)r * P.rows.cap;
    att_wave_state st;
    st.clear();
    att_walk<DT, D>(P, r, b, h, h / (P.Hq / P.Hkv), qi, sah_wave_id() * SAH_WAVE, cnt, D, [&](int i) { return cols ? cols[i] : i; },
                    [&](int) { return P.unit_inv_w; }, st);
    att_park<D, NW>(st, sah_wave_id(), s_m, s_l, s_acc);
    __syncthreads();
    att_gather<DT, D, NW>(s_m, s_l, s_acc, a, M, L);
  }
  att_store_row<DT, D>(P, r, b, h, qi, a, M, L);
}

// ---------------------------------------------------------------------------
// host
// ---------------------------------------------------------------------------
// the shape of a launch: rows per workgroup, key splits. Rows go 128 to a workgroup, 64 where that pads less.
static void qa_plan(int B, int Hkv, int nvec, int Lk, int* rw, qa_params* Q) {
  const int w4 = (nvec + 127) / 128 * 128, w2 = (nvec + 63) / 64 * 64;
  *rw = w2 < w4 ? 2 : 4;
  Q->row_tiles = (nvec + 32 * *rw - 1) / (32 * *rw);
  const int n_stages = (Lk + QA_STAGE - 1) / QA_STAGE;
  const int64_t wgs = (int64_t)B * Hkv * Q->row_tiles;
  int64_t split = wgs >= QA_MIN_WGS ? 1 : QA_MIN_WGS / wgs;  // one round of workgroups that all fit at once
  if (split > n_stages / QA_MIN_STAGES) split = n_stages / QA_MIN_STAGES;
  if (split < 1) split = 1;
  if (split > ATT_MAX_SPLIT) split = ATT_MAX_SPLIT;
  Q->stages_per_split = (int)((n_stages + split - 1) / split);
  Q->n_split = (n_stages + Q->stages_per_split - 1) / Q->stages_per_split;
}

extern "C" int64_t sah_members_attention_work_floats(int32_t B, int32_t Hq, int32_t Hkv, int32_t Lq, int32_t Lk, int32_t D) {
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || Lq <= 0 || Lk <= 0 || D <= 0 || Hq % Hkv) return 0;
  int rw;
  qa_params Q;
  qa_plan(B, Hkv, Hq / Hkv * Lq, Lk, &rw, &Q);
  return (int64_t)B * Hq * Lq * Q.n_split * (D + 2);
}

// May the call run here, and does it pay? one_kernel: the other choice is not sah_sparse_attention's gather but the kernel
// that selects the rows' columns and gathers them (sah_select_topk_attention). The two sides' times in microseconds, up to
// what both have in common, fitted to 1800 measured pairs of layer-steps (head_dim 64 and 128, 1 to 128 KV heads, 2 to 270
// query vectors each, 1024 to 65536 keys, 1 to 20 % of them in a row or all, with and without a mask; bf16 and fp16). This form:
// its workgroups' stages one after the other (two workgroups a CU share its matrix units), the partial results merged.
// The gather: a workgroup per row in the whole-row and one-kernel forms, so rounds of 256 rows; half the bytes where score
// keys stand for K. Of 900 pairs of other shapes 12 are more than 4 % slower here than there where this says they pay (30 % at
// most), and the sum of the times is within 1 % of the best choice. 128 vectors x 2 heads x 32768 keys of which 1175 count:
// 48 us of a step there, 66 here; 48 queries x 32 heads x 32768 keys, 2278 of them, causal mask: 825 there, 245 here.
bool members_attention_pays(const sah_attention_args* a, const att_params& P, bool one_kernel) {
  if (a->dtype == SAH_F32 || (a->D != 64 && a->D != 128) || a->Lq < 2) return false;
  // (a row's running maximum lags behind its largest logit, see SLACK: statistics come from the gather)
  if (P.drop.thresh || a->logits_out || a->stats_out || a->rows.w || P.dense == 2 || !(a->scaling > 0.f)) return false;
  if (a->ks_l * QA_STAGE >= (1 << 30) || a->vs_l * QA_STAGE >= (1 << 30)) return false;  // 32-bit offsets inside a stage
  const int64_t need = sah_members_attention_work_floats(a->B, a->Hq, a->Hkv, a->Lq, a->Lk, a->D);
  if (!a->work || a->work_floats < need) return false;
  int rw;
  qa_params Q;
  qa_plan(a->B, a->Hkv, a->Hq / a->Hkv * a->Lq, a->Lk, &rw, &Q);
  const double d = a->D / 128.0, rows = a->rows.n_rows;
  const double wgs = (double)a->B * a->Hkv * Q.row_tiles * Q.n_split;
  double stage = (wgs <= 256 ? 1.3 * d : 2.8 * d) + 0.45 + (P.amask ? 0.6 : 0.0) + (a->dtype == SAH_BF16 ? 0.2 * d : 0.0);
  if (rw == 2) stage *= 0.5;         // one tile of a stage per wave
  if (wgs > 512) stage *= wgs / 512;
  const double here = Q.stages_per_split * stage + 0.1 * Q.n_split + rows * (5e-4 + 4.2e-5 * d * Q.n_split);
  const double cnt = 1e-3 * (a->dense ? a->Lk : a->max_cnt < a->rows.cap ? a->max_cnt : a->rows.cap), work = cnt * d;
  const double rounds = ceil(rows / 256);
  const bool keyed = P.score_keys != nullptr;
  double there;
  if (one_kernel)
    there = keyed ? rounds * (1.7 + 3.0 * work + 1.3e-4 * a->Lk) - 1.6 : rounds * (2.2 + 3.9 * work + 6e-5 * a->Lk) - 0.3;
  else if (P.n_split == 0)
    there = keyed ? rounds * (1.2 + 2.0 * work) - 1.0 : rounds * (3.6 + 6.5 * work + (P.amask ? 2.0 * cnt : 0.0)) - 5.5;
  else
    there = keyed ? rows / 256 * 6.6 * work + rounds * 0.3 + 0.3 : rows / 256 * 7.1 * work + rounds * (P.amask ? 0.8 * cnt : 0.0) + 3.3;
  return 1.03 * here + 1.0 < there;
}

template <int DT, int D, int RW>
static void qa_launch_rw(const att_params& P, const qa_params& Q, unsigned n_wg, hipStream_t st) {
  if (P.dense) {
    if (P.amask) hipLaunchKernelGGL((k_members_attn_mfma<DT, D, RW, true, true>), dim3(n_wg), dim3(QA_NT), 0, st, P, Q);
    else hipLaunchKernelGGL((k_members_attn_mfma<DT, D, RW, false, true>), dim3(n_wg), dim3(QA_NT), 0, st, P, Q);
  } else {
    if (P.amask) hipLaunchKernelGGL((k_members_attn_mfma<DT, D, RW, true, false>), dim3(n_wg), dim3(QA_NT), 0, st, P, Q);
    else hipLaunchKernelGGL((k_members_attn_mfma<DT, D, RW, false, false>), dim3(n_wg), dim3(QA_NT), 0, st, P, Q);
  }
}

template <int DT, int D>
static int qa_launch(const sah_attention_args* a, const att_params& P) {
  int rw;
  qa_params Q;
  qa_plan(a->B, a->Hkv, a->Hq / a->Hkv * a->Lq, a->Lk, &rw, &Q);
  const int64_t streams = (int64_t)a->B * a->Hkv * Q.n_split;
  const int64_t n_wg = (streams + ATT_XCDS - 1) / ATT_XCDS * ATT_XCDS * Q.row_tiles;
  if (n_wg > 0x7fffffff) return sah_fail(SAH_ESHAPE, "sah_members_attention: too many workgroups");
  {
    sah_timed timed("k_members_attn_mfma", a->stream);
    if (rw == 4) qa_launch_rw<DT, D, 4>(P, Q, (unsigned)n_wg, (hipStream_t)a->stream);
    else qa_launch_rw<DT, D, 2>(P, Q, (unsigned)n_wg, (hipStream_t)a->stream);
    if (int rc = sah_launch_status("sah_members_attention")) return rc;
  }
  sah_timed timed("k_members_merge", a->stream);
  hipLaunchKernelGGL((k_members_merge<DT, D>), dim3(a->rows.n_rows), dim3(D), 0, (hipStream_t)a->stream, P, Q.n_split);
  return sah_launch_status("sah_members_attention(merge)");
}

int members_attention(const sah_attention_args* a, const att_params& P) {
  if (a->dtype == SAH_BF16) return a->D == 128 ? qa_launch<SAH_BF16, 128>(a, P) : qa_launch<SAH_BF16, 64>(a, P);
  return a->D == 128 ? qa_launch<SAH_F16, 128>(a, P) : qa_launch<SAH_F16, 64>(a, P);
}

extern "C" int sah_members_attention(const sah_attention_args* a) {
  if (!a) return sah_fail(SAH_ENULL, "sah_members_attention: args is NULL");
  att_params P;
  const int rc = att_prepare(a, P);
  if (rc) return rc;
  return members_attention_pays(a, P, false) ? members_attention(a, P) : sah_sparse_attention(a);
}
