// Row-wise top-k over 16-bit sortable keys, stand-alone form: the row's list, count and bitmap in memory are extended.
//
// One workgroup of NW waves per mask row; a lane owns eight consecutive candidates of a 512-candidate chunk, a wave up to CPW
// consecutive chunks, whose keys stay in its registers until the winners are known. The k-th largest key T is found in two
// steps. A histogram of every eighth key over its upper 13 bits brackets T between two bins, 3.5 standard deviations of the
// sampled rank to either side. Every key is compared with the bracket's two ends, and the few per cent inside are looked at
// one by one: counted value by value, which gives T exactly or shows that the bracket missed it, and kept in LDS until they
// can be compared with T. Rows for which that does not work (active columns that rank among them, a bracket of more than
// SQ_FINE key values, a missed T, waves that hold little else than keys of the bracket) take the general way: the bracket's
// keys picked from the registers, the bracket taken from a histogram of all keys if need be. Then, and where a lane has more of
// the bracket's keys than slots, every key is compared with T.
// Winners above T are written by every wave independently; the ties taken are the lowest columns. The list is unordered
// inside a row; its order is a pure function of the inputs.
#pragma once
#include "sah_sel16.h"

#define SQ_SHIFT 3                     // key values per bin of the sample's histogram, log2 (16-bit counters, two to a word)
#define SQ_COARSE (65536 >> SQ_SHIFT)
#define SQ_ALL_SHIFT 4                 // ... of the histogram of all keys (32-bit counters, in the same place)
#define SQ_ALL_COARSE (65536 >> SQ_ALL_SHIFT)
#define SQ_COARSE_WORDS 4096
static_assert(SQ_COARSE == 2 * SQ_COARSE_WORDS && SQ_ALL_COARSE == SQ_COARSE_WORDS, "the two histograms share their LDS");
#define SQ_FINE 1024                   // key values a bracket may span
#define SQ_COPIES 4                    // counters per key value, by lane: rows of few distinct keys (signature scores)
#define SQ_GATHER 4                    // keys a lane requests at a time
// keys a lane can keep for their comparison with T (all of them where it owns no more)
#define SQ_SLOTS(CPW) ((CPW) >= 16 ? 32 : (CPW) >= 8 ? 24 : (CPW) >= 2 ? 16 : 8)

#define SQ_MAX_CHUNKS 256  // chunks of a row that fit the registers of a workgroup (16 waves of 16): 131072 candidates

struct sq_lds {
  int part[16];
  int eq[16];
  int out[16];
  int lo_bin, hi_bin, lo_above;  // bins of the two sample ranks; keys in the bins above lo_bin
  int above;                     // keys above the bracket
  int sel_bin, sel_need;
  int over;                      // 1: a lane ran out of slots; 2: and a wave left its keys to be counted from the registers
};

// words of the histograms' and the slots' common place
__host__ __device__ constexpr int sq_coarse_words(int nw, int cpw) {
  return SQ_SLOTS(cpw) * nw * SAH_WAVE / 2 > SQ_COARSE_WORDS ? SQ_SLOTS(cpw) * nw * SAH_WAVE / 2 : SQ_COARSE_WORDS;
}

__device__ __forceinline__ void sq_keep_scalar(int& v) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+s"(v));
#endif
}

// flag bits 2 p and 2 p + 1 -> the two 16-bit masks of word p
__device__ __forceinline__ uint32_t sq_mask2(uint32_t flags, int p) {
  return ((0u - ((flags >> (2 * p)) & 1u)) & 0xffffu) | ((0u - ((flags >> (2 * p + 1)) & 1u)) << 16);
}
// packed 0 / 1 results of the four words of a chunk -> one bit per candidate (bits 16 and up: garbage)
__device__ __forceinline__ uint32_t sq_join(const uint32_t (&g)[4]) {
  const uint32_t m = g[0] | (g[1] << 2) | (g[2] << 4) | (g[3] << 6);
  return m | (m >> 15);
}

// The threads of a workgroup take the bins of a histogram from the top down, a few consecutive ones each; `mine`: the sum
// of this thread's. Returns the number in all bins above them. One barrier inside.
template <int NW>
__device__ __forceinline__ int sq_above(int mine, sq_lds& S) {
  const int lane = threadIdx.x & (SAH_WAVE - 1), wave = threadIdx.x / SAH_WAVE;
  const int incl = sah_wave_incl_scan(mine);
  if (lane == SAH_WAVE - 1) S.part[wave] = incl;
  __syncthreads();
  int above = incl - mine;
#pragma unroll
  for (int w = 0; w < NW; ++w) above += w < wave ? S.part[w] : 0;
  return above;
}

template <int NW, int CPW>
__device__ __forceinline__ void sq_select_row(sq_lds& S, unsigned char* dyn, const sah_rows& R, int r, const uint16_t* keys,
                                              int n_cand, int col_offset, int k, uint32_t excluded_key, int fresh, int sink,
                                              int window) {
  constexpr int NT = NW * SAH_WAVE;
  constexpr int SLOTS = SQ_SLOTS(CPW);
  constexpr bool LONG = CPW >= 8;           // what rows of few different keys lose grows with their length
  constexpr int NWD = (CPW + 3) / 4;        // 32-bit words of a lane's candidate masks: word w holds chunks 4 w .. 4 w + 3
  const int tid = threadIdx.x;
  const int lane = tid & (SAH_WAVE - 1);
  const int wave = sah_wave_id();
  const int n_chunks = (n_cand + SF_CHUNK - 1) / SF_CHUNK;
  const int cpw = (n_chunks + NW - 1) / NW;  // <= CPW (the host picks CPW)
  const int c0 = wave * cpw;
  const int c1 = c0 + cpw < n_chunks ? c0 + cpw : n_chunks;

  uint32_t* s_bm = (uint32_t*)dyn;                          // n_words + 2
  uint32_t* s_co = s_bm + ((R.n_words + 2 + 3) & ~3);       // [SQ_COARSE_WORDS]
  uint16_t* s_slot = (uint16_t*)s_co;                       // [SLOTS][NT], in the place of the sample's histogram
  uint32_t* s_fi = s_co + sq_coarse_words(NW, CPW);         // [SQ_COPIES][SQ_FINE]
  uint32_t* s_any = s_fi + SQ_COPIES * SQ_FINE;             // [NW * CPW] chunk holds active columns
  uint32_t* bm = R.bitmap + (int64_t)r * R.n_words;
  const uint32_t ek = excluded_key & 0xffffu;

  // the lane's first candidate of chunk c; opaque, so that no pass keeps its addresses alive for the next
  auto first_cand = [&](int c) -> int {
    uint32_t l = (uint32_t)lane;
    sah_keep(l);
    return c * SF_CHUNK + (int)l * 8;
  };
  auto clear = [&](uint32_t* p, int words) {
    for (int i = tid; i < words / 4; i += NT) ((uint4*)p)[i] = make_uint4(0u, 0u, 0u, 0u);
  };

  // the key loads go out first and land while the bitmap row and the counters are set up
  uint4 kreg[CPW];
#pragma unroll
  for (int u = 0; u < CPW; ++u) {
    int cand = first_cand(c0 + u);
    if (cand >= n_cand) cand = 0;  // a group with no candidate: any valid address will do
    kreg[u] = *(const uint4*)(keys + cand);
  }
  clear(s_co, SQ_COARSE_WORDS);
  clear(s_fi, SQ_COPIES * SQ_FINE);
  if (tid < NW * CPW) s_any[tid] = 0u;
  if (tid == 0) {
    S.above = 0;
    S.lo_bin = -1;
    S.hi_bin = -1;
    S.sel_bin = -1;
    S.over = 0;
  }
  int* cols = R.cols + (int64_t)r * R.cap;
  float* wgt = R.w ? R.w + (int64_t)r * R.cap : nullptr;
  __syncthreads();
  // the bitmap row, and which chunks have active columns
  auto put_word = [&](int i, uint32_t w) {
    s_bm[i] = w;
    if (w) {
      const int a = i * 32 - col_offset, b = a + 31;  // its candidates
      if (a >= 0 && a < n_cand) s_any[a / SF_CHUNK] = 1u;
      if (b >= 0 && b < n_cand) s_any[b / SF_CHUNK] = 1u;
      else if (a < n_cand && b >= n_cand) s_any[n_chunks - 1] = 1u;
    }
  };
  int cnt0;
  if (fresh) {
    // rows still empty: the sink and local columns of one query per row in closed form, as
    // k_sink_local would have left them (basic_fixed.py:354-363, :48-67), without a launch of their own
    const int n = R.n_keys;
    const int s_hi = sink < n ? sink : n;
    int lo = 0, hi = 0;
    if (window > 0) {
      lo = n - window;
      hi = n;
      if (lo < 0) lo = 0;
    }
    const int lo2 = lo > s_hi ? lo : s_hi;
    const int fixed = s_hi + (hi > lo2 ? hi - lo2 : 0);
    for (int i = tid; i < fixed && i < R.cap; i += NT) {
      cols[i] = i < s_hi ? i : lo2 + (i - s_hi);
      if (wgt) wgt[i] = 1.0f;
    }
    cnt0 = fixed < R.cap ? fixed : R.cap;
    for (int i = tid; i < R.n_words + 2; i += NT)
      put_word(i, i < R.n_words ? (sah_range_bits(i, 0, s_hi) | sah_range_bits(i, lo, hi)) : 0u);
  } else {
    cnt0 = R.cnt[r];  // read before the first barrier: rewritten at the end
    if (cnt0 > R.cap) cnt0 = R.cap;
    for (int i = tid; i < R.n_words + 2; i += NT) put_word(i, i < R.n_words ? bm[i] : 0u);
  }
  __syncthreads();
  // active candidates take the excluded key, missing ones 0; most chunks have neither
  const uint64_t any = __ballot(lane < CPW && s_any[wave * cpw + (lane < cpw ? lane : 0)] != 0u);
  const uint32_t ek2 = ek * 0x00010001u;
#pragma unroll
  for (int u = 0; u < CPW; ++u) {
    if (((any >> u) & 1) || (c0 + u + 1) * SF_CHUNK > n_cand) {  // uniform across the wave
      uint32_t excl, valid;
      sf_flags(s_bm, R.n_words, first_cand(c0 + u), n_cand, col_offset, excl, valid);
      uint32_t w[4] = {kreg[u].x, kreg[u].y, kreg[u].z, kreg[u].w};
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const uint32_t me = sq_mask2(excl, p);
        w[p] = ((w[p] & ~me) | (ek2 & me)) & sq_mask2(valid, p);
      }
      kreg[u] = make_uint4(w[0], w[1], w[2], w[3]);
    }
  }

  // run f(chunk, keys, register slot) over this wave's chunks in ascending order
  auto for_chunks = [&](auto&& f) {
    int n_mine = c1 - c0;
    sq_keep_scalar(n_mine);  // the conditions are cheaper to evaluate again than to keep
#pragma unroll
    for (int u = 0; u < CPW; ++u)
      if (u < n_mine) {
        // opaque to the optimiser: values derived from the keys in one pass are not kept
        // alive for the next, they are cheaper to recompute than to hold in registers
        sah_keep(kreg[u].x), sah_keep(kreg[u].y), sah_keep(kreg[u].z), sah_keep(kreg[u].w);
        const uint32_t kk[4] = {kreg[u].x, kreg[u].y, kreg[u].z, kreg[u].w};
        f(c0 + u, kk, u);
      }
  };
  auto key_of = [](const uint32_t (&kk)[4], int t) -> uint32_t { return t & 1 ? kk[t >> 1] >> 16 : kk[t >> 1] & 0xffffu; };

  // ---- the bracket [lo, lo + span) of key values ------------------------------------------------------
  int lo = 0, span = 0;
  constexpr int CPT = SQ_COARSE_WORDS / NT;  // words of the first histogram per thread, from the top down
  // counts of a word of it: the upper bin's and the lower one's (all keys: one bin, in the first)
  auto bins_of = [&](int word, bool sample, int& c1st, int& c2nd) {
    const uint32_t v = s_co[word];
    c1st = sample ? (int)(v >> 16) : (int)v;
    c2nd = sample ? (int)(v & 0xffffu) : 0;
  };
  auto coarse_sum = [&](bool sample) -> int {
    int sum = 0;
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
      int a, b;
      bins_of(SQ_COARSE_WORDS - (tid + 1) * CPT + j, sample, a, b);
      sum += a + b;
    }
    return sum;
  };
  auto find_bin = [&](bool sample, int rank, int above, int mine, int& bin_out, int* above_out) {
    if (above < rank && rank <= above + mine) {  // one thread at most
      for (int word = SQ_COARSE_WORDS - tid * CPT - 1;; --word) {  // ends: the rank lies in one of this thread's words
        int a, b;
        bins_of(word, sample, a, b);
        if (rank <= above + a + b) {
          const bool first = rank <= above + a;
          bin_out = sample ? 2 * word + (first ? 1 : 0) : word;
          if (above_out) *above_out = above + (first ? 0 : a);
          break;
        }
        above += a + b;
      }
    }
  };
  // T's place in the bracket from the counts of its values: the value of rank k - above, from the top down
  auto pick = [&](int above) {
    constexpr int FPT = SQ_FINE / NT;
    int fc[FPT], mine = 0;
#pragma unroll
    for (int j = 0; j < FPT; ++j) {
      const int v = SQ_FINE - 1 - (tid * FPT + j);
      fc[j] = 0;
#pragma unroll
      for (int cp = 0; cp < SQ_COPIES; ++cp) fc[j] += (int)s_fi[cp * SQ_FINE + v];
      mine += fc[j];
    }
    int ab = above + sq_above<NW>(mine, S);
    if (ab < k && k <= ab + mine) {
#pragma unroll
      for (int j = 0; j < FPT; ++j) {
        if (ab < k && k <= ab + fc[j]) {
          S.sel_bin = SQ_FINE - 1 - (tid * FPT + j);
          S.sel_need = k - ab;
        }
        ab += fc[j];
      }
    }
    __syncthreads();
  };

  // Many of a wave's 64 lanes with one key (hidden columns, rows of few keys): their adds to one counter go one after the other,
  // 2.4 cycles each. crowd: whether an eighth of the lanes hold the same word as the first or the 32nd one, and its lower key;
  // the lanes with that index then add once, together (all lanes call). 1056 rows x 131000 candidates, k 6550, and how long
  // without: the first 90 % hidden 247 us (709), 97 % 242 (480), the same share hidden here and there 233 (682) and 235 (470),
  // one key throughout 272 (506); no two columns alike 148 (144).
  auto crowd = [&](uint32_t word, uint32_t& key) -> bool {
    uint32_t w = (uint32_t)__builtin_amdgcn_readlane((int)word, 0);
    uint64_t all = __ballot(word == w);
    if (__popcll(all) < SAH_WAVE / 8) {
      w = (uint32_t)__builtin_amdgcn_readlane((int)word, SAH_WAVE / 2);
      all = __ballot(word == w);
    }
    key = w & 0xffffu;
    return __popcll(all) >= SAH_WAVE / 8;
  };
  auto add_crowd = [&](uint32_t* counters, uint32_t index, uint32_t of_crowd, bool counted) {
    const bool same = counted && index == of_crowd;
    const uint64_t all = __ballot(same);
    if (counted && (!same || lane == __builtin_ctzll(all))) atomicAdd(&counters[index], same ? (uint32_t)__popcll(all) : 1u);
  };
  uint32_t* my_f = s_fi + (lane & (SQ_COPIES - 1)) * SQ_FINE;

  uint32_t of_crowd;
  const bool crowds = LONG && crowd(kreg[0].x, of_crowd);  // uniform across the wave
  for_chunks([&](int, const uint32_t (&kk)[4], int u) {
    const uint32_t key = key_of(kk, u & 7), bin = key >> SQ_SHIFT;
    const uint32_t n = bin & 1u ? 0x10000u : 1u;
    if (crowds) {
      const bool same = bin == of_crowd >> SQ_SHIFT;
      const uint64_t all = __ballot(same);
      if (!same || lane == __builtin_ctzll(all)) atomicAdd(&s_co[bin >> 1], same ? n * (uint32_t)__popcll(all) : n);
    } else {
      atomicAdd(&s_co[bin >> 1], n);
    }
  });
  __syncthreads();
  {
    const int mine = coarse_sum(true);
    const int above = sq_above<NW>(mine, S);
    const float rho = (float)k * 0.125f, dev = 3.5f * sqrtf(rho) + 1.0f;
    const int r_hi = (int)(rho - dev), r_lo = (int)(rho + dev) + 1;
    if (r_hi >= 1) find_bin(true, r_hi, above, mine, S.hi_bin, nullptr);
    find_bin(true, r_lo, above, mine, S.lo_bin, nullptr);
  }
  __syncthreads();
  bool exact = false;  // uniform: the next bracket comes from all keys
  lo = S.lo_bin < 0 ? 0 : S.lo_bin << SQ_SHIFT;
  span = (S.hi_bin < 0 ? 65536 : (S.hi_bin + 1) << SQ_SHIFT) - lo;
  if (span > SQ_FINE) {
    exact = S.hi_bin >= 0 || S.lo_bin < 0;
    span = SQ_FINE;  // nothing bounds the largest keys: as far up as the counters go
  }

  // Candidate masks of this lane: above T, equal to T, active (all zero unless active columns may rank)
  uint32_t gt[NWD], eq[NWD], act[NWD];
#pragma unroll
  for (int w = 0; w < NWD; ++w) gt[w] = eq[w] = act[w] = 0u;
  // candidate of bit b of mask word w
  auto bit_cand = [&](int w, int b) -> int { return first_cand(c0 + 4 * w) + ((b & 24) << 6) + (b & 7); };
  bool found = false, done = false;  // uniform: T is known, and the masks are
  bool tried = false;                // uniform: the short way's masks have been made, what lies above the bracket is counted
  bool counted = false;              // uniform across the wave: its keys of the bracket are
  if (!exact && (uint32_t)lo > ek) {
    // ---- the short way: keys above the bracket into gt, the bracket's keys one by one
    uint32_t in[NWD];
#pragma unroll
    for (int w = 0; w < NWD; ++w) in[w] = 0u;
    const uint32_t below2 = (uint32_t)(lo - 1) * 0x00010001u, last2 = (uint32_t)(lo + span - 1) * 0x00010001u;
    for_chunks([&](int, const uint32_t (&kk)[4], int u) {
      uint32_t a[4], b[4];
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        a[p] = sah_pk_gt01_u16(kk[p], below2);
        b[p] = sah_pk_gt01_u16(kk[p], last2);
        a[p] ^= b[p];
      }
      in[u >> 2] |= (sq_join(a) & 0xffu) << (8 * (u & 3));
      gt[u >> 2] |= (sq_join(b) & 0xffu) << (8 * (u & 3));
    });
    int n = 0, n_above = 0;
#pragma unroll
    for (int w = 0; w < NWD; ++w) {
      if (LONG) n += __popc(in[w]);
      n_above += __popc(gt[w]);
    }
    tried = true;
    // (requested one by one, 1056 rows x 131000 of one key: 507 us; at three eighths in place of three quarters, rows that rise
    // with the column lose more than rows of two keys gain)
    counted = !LONG || __ballot(n <= SLOTS || n <= 6 * (c1 - c0)) != 0;
    if (counted) {
      n = 0;
#pragma unroll
      for (int w = 0; w < NWD; ++w) {
        uint32_t m = in[w];
        while (m) {
          uint32_t kv[SQ_GATHER];
          uint32_t left = m;
#pragma unroll
          for (int i = 0; i < SQ_GATHER; ++i) {
            kv[i] = keys[left ? bit_cand(w, __builtin_ctz(left)) : 0];  // (not active: the key in memory is the key)
            left &= left - 1;
          }
#pragma unroll
          for (int i = 0; i < SQ_GATHER; ++i) {
            if (m) {
              atomicAdd(&my_f[kv[i] - (uint32_t)lo], 1u);
              if (n < SLOTS) s_slot[n * NT + tid] = (uint16_t)kv[i];
              ++n;
            }
            m &= m - 1;
          }
        }
      }
    }
    if (n > SLOTS) {  // (every lane of a wave that has not counted)
      if (LONG) atomicMax(&S.over, counted ? 1 : 2);
      else S.over = 1;
    }
    const int na = sah_wave_sum_i(n_above);
    if (lane == 0 && na) atomicAdd(&S.above, na);
    __syncthreads();
    if (!LONG || S.over < 2) {
      pick(S.above);
      found = S.sel_bin >= 0;
      exact = !found;
      done = found && !S.over;
    }
    if (done) {
      const uint32_t t = (uint32_t)(lo + S.sel_bin);
      n = 0;
#pragma unroll
      for (int w = 0; w < NWD; ++w) {
        uint32_t m = in[w];
        while (m) {
          const uint32_t kv = s_slot[n * NT + tid];
          const uint32_t bit = m & (0u - m);
          m ^= bit;
          ++n;
          gt[w] |= kv > t ? bit : 0u;
          eq[w] |= kv == t ? bit : 0u;
        }
      }
    } else {
#pragma unroll
      for (int w = 0; w < NWD; ++w) gt[w] = 0u;
    }
  }
  if (!found) {
    // ---- the general way to T
    uint32_t of_crowd;
    const bool crowds = crowd(kreg[0].x, of_crowd);
    for (;;) {  // at most twice, uniform
      if (exact) {
        counted = false;
        __syncthreads();  // the counts of the attempt before have been read
        clear(s_co, SQ_COARSE_WORDS);
        clear(s_fi, SQ_COPIES * SQ_FINE);
        if (tid == 0) {
          S.lo_bin = -1;
          S.sel_bin = -1;
        }
        __syncthreads();
        for_chunks([&](int, const uint32_t (&kk)[4], int) {
          const bool crowded = crowds && crowd(kk[0], of_crowd);  // uniform across the wave
#pragma unroll
          for (int t = 0; t < 8; ++t) {
            if (crowded) add_crowd(s_co, key_of(kk, t) >> SQ_ALL_SHIFT, of_crowd >> SQ_ALL_SHIFT, true);
            else atomicAdd(&s_co[key_of(kk, t) >> SQ_ALL_SHIFT], 1u);
          }
        });
        __syncthreads();
        const int mine = coarse_sum(false);
        const int ab = sq_above<NW>(mine, S);
        find_bin(false, k, ab, mine, S.lo_bin, &S.lo_above);
        __syncthreads();
        lo = S.lo_bin << SQ_ALL_SHIFT;  // found: k is at most the number of candidates
        span = 1 << SQ_ALL_SHIFT;
      }
      // what lies above the bracket, and the bracket's keys value by value
      const uint32_t lo2 = (uint32_t)lo * 0x00010001u, span2 = (uint32_t)span * 0x00010001u;
      const uint32_t last2 = (uint32_t)(lo + span - 1) * 0x00010001u;
      uint32_t n_above = 0;
      if (!counted) for_chunks([&](int, const uint32_t (&kk)[4], int) {
        uint32_t d[4], g[4];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          if (!exact) n_above += sah_pk_gt01_u16(kk[p], last2);
          d[p] = sah_pk_sub_u16(kk[p], lo2);
          g[p] = sah_pk_gt01_u16(span2, d[p]);
        }
        uint32_t in = sq_join(g) & 0xffu;
        if (crowds && crowd(d[0], of_crowd) && of_crowd < (uint32_t)span) {  // uniform across the wave
#pragma unroll
          for (int t = 0; t < 8; ++t) add_crowd(s_fi, key_of(d, t), of_crowd, key_of(g, t) != 0u);
          return;
        }
        while (in) {
          const int t = __builtin_ctz(in);
          in &= in - 1;
          const uint32_t a = t & 2 ? d[1] : d[0], b = t & 2 ? d[3] : d[2];
          const uint32_t two = t & 4 ? b : a;
          atomicAdd(&my_f[t & 1 ? two >> 16 : two & 0xffffu], 1u);
        }
      });
      if (!exact && !tried) {
        const int na = sah_wave_sum_i((int)((n_above & 0xffffu) + (n_above >> 16)));
        if (lane == 0 && na) atomicAdd(&S.above, na);
      }
      __syncthreads();
      pick(exact ? S.lo_above : S.above);
      if (S.sel_bin >= 0 || exact) break;
      exact = true;  // the bracket missed T
    }
  }
  const uint32_t T = (uint32_t)(lo + S.sel_bin);
  const int need = S.sel_need;
  if (!done) {
    // ---- every key compared with T
    // Active candidates carry the excluded key. While that ranks below T they are neither winners nor ties; otherwise (a
    // row with fewer than k better inactive candidates) they take rank but are never emitted.
    const bool slow = ek >= T;
    const uint32_t T2 = T * 0x00010001u;
    for_chunks([&](int c, const uint32_t (&kk)[4], int u) {
      uint32_t g[4], e[4];
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        g[p] = sah_pk_gt01_u16(kk[p], T2);
        e[p] = sah_pk_ne01_u16(kk[p], T2);
      }
      uint32_t cg = sq_join(g) & 0xffu, ce = ~sq_join(e) & 0xffu;
      if (slow) {
        uint32_t ex, valid;
        sf_flags(s_bm, R.n_words, first_cand(c), n_cand, col_offset, ex, valid);
        ce &= valid;  // a missing candidate has key 0, which ties when T is 0
        cg &= ~ex;
        act[u >> 2] |= ex << (8 * (u & 3));
      }
      gt[u >> 2] |= cg << (8 * (u & 3));
      eq[u >> 2] |= ce << (8 * (u & 3));
    });
  }

  // ---- ties: the lowest columns, `need` of them (active ones count, but are not emitted)
  int n_eq = 0;
#pragma unroll
  for (int w = 0; w < NWD; ++w) n_eq += __popc(eq[w]);
  const int wave_eq = sah_wave_sum_i(n_eq);
  if (lane == 0) S.eq[wave] = wave_eq;
  __syncthreads();
  int tie_base = 0;
#pragma unroll
  for (int w = 0; w < NW; ++w) tie_base += w < wave ? S.eq[w] : 0;
  if (tie_base >= need) {
#pragma unroll
    for (int w = 0; w < NWD; ++w) eq[w] = 0u;
  } else if (tie_base + wave_eq > need) {  // the boundary lies inside this wave
    int run = tie_base;
#pragma unroll
    for (int u = 0; u < CPW; ++u) {
      const uint32_t e = (eq[u >> 2] >> (8 * (u & 3))) & 0xffu;
      const int ne = __popc(e);
      const int incl = sah_wave_incl_scan(ne);
      const uint32_t take = sf_lowest(e, need - run - (incl - ne));
      run += __builtin_amdgcn_readlane(incl, SAH_WAVE - 1);
      eq[u >> 2] ^= (e ^ take) << (8 * (u & 3));
    }
  }
  int mine = 0;
#pragma unroll
  for (int w = 0; w < NWD; ++w) {
    gt[w] |= eq[w] & ~act[w];
    mine += __popc(gt[w]);
  }
  const int incl = sah_wave_incl_scan(mine);
  if (lane == SAH_WAVE - 1) S.out[wave] = incl;
  __syncthreads();
  int out_base = 0, total = 0;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    const int v = S.out[w];
    out_base += w < wave ? v : 0;
    total += v;
  }

  // ---- write
  int pos = cnt0 + out_base + incl - mine;
#pragma unroll
  for (int w = 0; w < NWD; ++w) {
    uint32_t m = gt[w];
    while (m) {
      const int col = bit_cand(w, __builtin_ctz(m)) + col_offset;
      m &= m - 1;
      atomicOr(&s_bm[col >> 5], 1u << (col & 31));
      if (pos < R.cap) {
        cols[pos] = col;
        if (wgt) wgt[pos] = 1.0f;
      }
      ++pos;
    }
  }
  __syncthreads();
  if (total > 0 || fresh)
    for (int i = tid; i < R.n_words; i += NT) bm[i] = s_bm[i];
  if (tid == 0) R.cnt[r] = cnt0 + total;
}

// dynamic LDS bytes of one launch
static inline size_t sq_lds_bytes(int n_words, int nw, int cpw) {
  return ((size_t)((n_words + 2 + 3) & ~3) + sq_coarse_words(nw, cpw) + SQ_COPIES * SQ_FINE + nw * cpw) * 4;
}
