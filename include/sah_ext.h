/* Entry points of libsah_mi355.so beyond those of sah.h: other forms of calls declared there, over the same argument
 * blocks. Conventions and error codes are sah.h's. */
#ifndef SAH_EXT_H
#define SAH_EXT_H
#include "sah.h"

#ifdef __cplusplus
extern "C" {
#endif

/* sah_sparse_attention for a caller whose rows.bitmap holds exactly the rows' entries (what every row builder and
 * selection of this library leaves unless asked to skip it): same arguments, same results. With several queries per row
 * (16-bit tensors, head_dim 64 / 128, unit weights, no dropout, no logits or statistics output, scaling > 0) and rows
 * that hold more than a small share of the keys the products run dense on the matrix cores and the bitmap decides which
 * entries count; the weights of the softmax then enter the second product as 16-bit terms that together are the fp32
 * weight, and rows that a key of another row could have reached (K or V not finite) are done again entry by entry. It
 * needs a->work to hold sah_members_attention_work_floats(...) floats; with less, or in any other case, the call is
 * sah_sparse_attention. */
int64_t sah_members_attention_work_floats(int32_t B, int32_t Hq, int32_t Hkv, int32_t Lq, int32_t Lk, int32_t D);
int sah_members_attention(const sah_attention_args* a);

/* A whole Lloyd run: sah_pq_keys_absmax, then max_iter times sah_pq_kmeans_assign and sah_pq_kmeans_update, in one call
 * and without host-made random numbers. given_start != 0: centres hold the start. Otherwise the start is vector
 * start_idx[g][c] (scratch of the caller, no output) of every group: one vector of each of n_cent equal strata of
 * [0, n_keys), chosen by number g * n_cent + c of torch.rand(float64) with a CPU generator seeded with start_seed. In
 * iteration i an empty centre takes vector number (i * n_groups + g) * n_cent + c of torch.randint(0, n_keys) with a CPU
 * generator seeded with reseed_seed (below 2^28 keys; beyond, where torch draws 64 bits, still the 32-bit number modulo
 * n_keys). reseed_idx, optional scratch: all these numbers are drawn into it first, in one pass; without it a group with an
 * empty centre draws the sequence up to its own numbers by itself, which is the cheaper way up to some millions of them. The seeds' low 32 bits count, as in torch. sums, counts, state and absmax_bits must
 * be zero before the call (sums and counts are zero again after it); the codes are the assignment to the centres that
 * entered the last iteration carried out. */
typedef struct sah_pq_kmeans_args {
  const void* k; int64_t ks_b, ks_h, ks_l;
  int32_t dtype;
  int32_t B, Hkv, n_sub, d_sub, n_cent;
  int32_t key_offset, n_keys;
  float* centres;                 /* [n_groups, n_cent, d_sub] */
  uint8_t* codes; int64_t code_pitch; int64_t code_offset;
  int64_t* sums; int32_t* counts; /* [n_groups, n_cent, d_sub], [n_groups, n_cent] */
  float* shift2;                  /* [n_groups] */
  int32_t* state;                 /* [4] */
  uint32_t* absmax_bits;          /* [1] */
  int32_t* start_idx;             /* [n_groups, n_cent], scratch; may be NULL with given_start */
  int32_t* reseed_idx;            /* [max_iter, n_groups, n_cent] or NULL */
  uint64_t start_seed, reseed_seed;
  float tol;
  int32_t max_iter, given_start;
  void* stream;
} sah_pq_kmeans_args;
int sah_pq_kmeans(const sah_pq_kmeans_args* a);

/* sah_amask_classify whose answer the host has when the call returns, without a cleared output, a copy and a wait for the
 * stream: the kernel writes the flags into host memory, and the call watches that word (after 2 ms, behind long work of the
 * stream, now and then). mask.flags is not used. scratch: two words of device memory, zero before the
 * first call and left zero; host_word: pinned host memory the device can write, zero before the first call. Both serve one
 * call at a time. Refused while the stream is being captured. */
typedef struct sah_amask_read_args {
  sah_amask_classify_args mask;
  uint32_t* scratch;
  uint64_t* host_word;
  int32_t flags;  /* out */
} sah_amask_read_args;
int sah_amask_read(sah_amask_read_args* a);

/* The same as two calls, for a caller that puts other work on its way between question and answer. scratch and host_word serve
 * one question at a time, from ask to answer, and stay allocated that long, as does the mask. */
typedef struct sah_amask_question {
  sah_amask_read_args read;
  uint32_t asked;  /* of the library */
} sah_amask_question;
int sah_amask_ask(sah_amask_question* q);
int sah_amask_answer(sah_amask_question* q);

/* sah_hash_decode_attention under an additive mask (attention.amask, of the queries' type) that holds nothing but 0, the
 * type's lowest value and -inf, in one kernel: the selection ranks a column at the lowest value below every other one (as the
 * sum of score and mask does) and leaves out one at -inf, whose weight is 0. fits says whether one kernel runs the step: fp32
 * or bf16, skip_bitmap set, no key_sig (the compact form may be given or not), and what else sah_hash_decode_attention needs for it;
 * with ask != 0 the call only says so, otherwise a step that does not fit is refused. */
typedef struct sah_hash_decode_masked_args {
  const sah_hash_decode_args* decode;
  const sah_attention_args* attention;
  uint32_t* tickets;
  int32_t ask;
  int32_t fits;  /* out */
} sah_hash_decode_masked_args;
int sah_hash_decode_masked(sah_hash_decode_masked_args* m);

#ifdef __cplusplus
}
#endif
#endif
