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
 * (16-bit tensors, head_dim 64 / 128, unit weights, no dropout, no logits output, scaling > 0) and rows that hold more
 * than a small share of the keys the products run dense on the matrix cores and the bitmap decides which entries count;
 * the weights of the softmax then enter the second product as two 16-bit terms. It needs a->work to hold
 * sah_members_attention_work_floats(...) floats; with less, or in any other case, the call is sah_sparse_attention. */
int64_t sah_members_attention_work_floats(int32_t B, int32_t Hq, int32_t Hkv, int32_t Lq, int32_t Lk, int32_t D);
int sah_members_attention(const sah_attention_args* a);

#ifdef __cplusplus
}
#endif
#endif
