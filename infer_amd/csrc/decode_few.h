// Paged decode attention of a few sequences (decode_few.hip), for the entry points of paged_decode.hip.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

struct FewDecode {
    const uint16_t* q; int64_t q_stride0;
    const uint16_t* k; const uint16_t* v;      // paged caches
    int64_t blk_stride, tok_stride;
    const int32_t* bt; int64_t bt_stride0;
    const int32_t* ctx;
    int max_ctx;                               // what the block table can address
    int batch, group, num_kv_heads, block_size, num_blocks;
    float scale_log2;
    int pieces;                                // workgroups per (sequence, KV head)
    float* rec;                                // [batch][KV head][pieces][few_record_floats(group)]
    uint16_t* out; int64_t out_stride0;
};

// What stands in front of the attention of new tokens: norms of their query and key heads, rotary positions, the append (as in
// qk_norm_rope_append.hip).
struct FewFront {
    const uint16_t* k; int64_t k_stride0;      // the new tokens' rows
    const uint16_t* v; int64_t v_stride0;
    const int64_t* positions;
    const uint16_t* q_weight; const uint16_t* k_weight;
    const uint16_t* cos_sin; int64_t max_position;
    uint16_t* k_cache; uint16_t* v_cache;      // those of FewDecode
    const int32_t* slots; int64_t num_slots;
    float eps;
};

// What a piece leaves: [group][128] unnormalised sums, then [group] (running maximum in the log2 domain, sum).
__host__ __device__ inline int few_record_floats(int group) { return 130 * group + (group & 1 ? 2 : 0); }

// Pieces per (sequence, KV head), or 0 where the batch is not small.
int few_decode_pieces(int64_t batch, int64_t num_kv_heads, int64_t max_tokens);
int launch_few_decode(const FewDecode& a, hipStream_t stream, const FewFront* front = nullptr);      // records, then their sum in `out`
