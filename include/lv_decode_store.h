/* A layer's decode step in one call: lv_store_kvcache and lv_decode_attn (lv_attention.h). */
#ifndef LV_DECODE_STORE_H
#define LV_DECODE_STORE_H

#include "lv_attention.h"

#ifdef __cplusplus
extern "C" {
#endif

/* The results of
 *   lv_store_kvcache(key, value, key_stride0, value_stride0, k_cache, v_cache, slot_mapping, batch, num_kv_heads, head_dim,
 *                    num_slots, stream);
 *   lv_decode_attn(q, k_cache, v_cache, o, ..., stream);
 * for any slots: one elsewhere among the tokens that this or another sequence reads (tokens of one sequence as several rows of the
 * batch) is read as it was stored. Two rows with one slot leave either. Up to 64 sequences take one launch: the attention kernel
 * reads the step's rows from key and value and writes them to the caches on its way. num_splits 0 leaves the choice to the
 * library; a workspace for lv_decode_num_splits splits always serves. */
int lv_decode_attn_store(const void* q, const void* key, const void* value, int64_t key_stride0, int64_t value_stride0,
                         void* k_cache, void* v_cache, const int32_t* slot_mapping, int64_t num_slots, void* o, int64_t q_stride0,
                         int64_t o_stride0, const int32_t* context_lens, const int32_t* block_table, int block_table_stride, int batch,
                         int max_blocks_per_seq, int block_size, int num_heads, int num_kv_heads, int head_dim, float scale,
                         void* workspace, size_t workspace_bytes, int num_splits, const int32_t* seq_order, int kernel_hint,
                         lv_stream_t stream);

#ifdef __cplusplus
}
#endif
#endif
