/*
 * Entry points of libqfactory_hip.so that the package's own host code calls beside those of qfactory_hip.h; the same
 * conventions (device pointers, a hipStream_t, calls only enqueue; 0 success, 1 invalid arguments, 2 launch failed).
 */
#ifndef QFACTORY_HIP_EXT_H
#define QFACTORY_HIP_EXT_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/*
 * qf_pack_weight, qf_transpose_scale and qf_pack_zero of one layer in one launch (scale and zero may be null), with the
 * range check of the fields and zero-points in the same pass: *bad (device or pinned host memory, may be null) is set to a nonzero
 * value if any lies outside [0, 2^nbits) and left alone otherwise; the caller clears it first.
 */
int qf_pack_layer(const int32_t* weight, int8_t* w_out, const uint16_t* scale, uint16_t* s_out, const int32_t* zero, int8_t* z_out,
                  int64_t K, int64_t N, int64_t G, int nbits, uint32_t* bad, void* stream);

/*
 * Causal attention of `tokens` positions of every sequence over its cache: q and out (batch, tokens, heads, head_dim)
 * fp16, caches (batch, heads, max_len, head_dim) fp16, pos (tokens) int64 device values; token t sees cache rows
 * 0 .. pos[t].  head_dim 64 or 128; q, caches and out 16-byte aligned.  Scores and sums in fp32.
 */
int qf_prefill_attention(const uint16_t* q, const uint16_t* k_cache, const uint16_t* v_cache, const int64_t* pos, uint16_t* out,
                         int64_t batch, int64_t tokens, int64_t heads, int64_t head_dim, int64_t max_len, void* stream);

/*
 * qf_decode_attention and qf_rope_decode_attention with the number of launches of this shape, each on caches of its own, that lie between
 * one launch on these caches and the next: the layers of the model (0: not known).  Where the rows that they read together
 * are more than the 256 MB of the Infinity Cache, they are loaded past it.  The results are the same.
 */
int qf_decode_attention_layers(const uint16_t* q, const uint16_t* k_cache, const uint16_t* v_cache, const int64_t* pos,
                               uint16_t* out, int64_t batch, int64_t heads, int64_t head_dim, int64_t max_len, int64_t layers,
                               void* stream);
int qf_rope_decode_attention_layers(const uint16_t* qkv, const int64_t* pos, const float* cos_table, const float* sin_table,
                                    uint16_t* k_cache, uint16_t* v_cache, uint16_t* out, int64_t batch, int64_t heads,
                                    int64_t head_dim, int64_t max_len, int64_t layers, void* stream);

#ifdef __cplusplus
}
#endif
#endif
