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

// Of the steps of 32 tokens that a sequence has, no more than `pieces` are somebody's first.
__device__ __forceinline__ int few_pieces_of(const FewDecode& a, int len) {
    len = len < a.max_ctx ? len : a.max_ctx;
    const int steps = len > 0 ? (len + 31) / 32 : 0;
    return steps < a.pieces ? steps : a.pieces;
}
typedef float few_f32x4 __attribute__((ext_vector_type(4)));
// Adds sums `x` with (maximum, sum of weights) `o` to `num` with `s`.  The products are fused as written, so that all callers get the same bits.
__device__ __forceinline__ void few_add(few_f32x4& num, float2& s, few_f32x4 x, float2 o) {
    const float top = fmaxf(s.x, o.x), f1 = s.x == top ? 1.f : __builtin_amdgcn_exp2f(s.x - top), f2 = o.x == top ? 1.f : __builtin_amdgcn_exp2f(o.x - top);
#pragma unroll
    for (int e = 0; e < 4; ++e) num[e] = __builtin_fmaf(num[e], f1, x[e] * f2);
    s = make_float2(top, __builtin_fmaf(s.y, f1, o.y * f2));
}
// The same, the other product rounded by itself.
__device__ __forceinline__ void few_append(few_f32x4& num, float2& s, few_f32x4 x, float2 o) {
    const float top = fmaxf(s.x, o.x), f1 = s.x == top ? 1.f : __builtin_amdgcn_exp2f(s.x - top), f2 = o.x == top ? 1.f : __builtin_amdgcn_exp2f(o.x - top);
#pragma unroll
    for (int e = 0; e < 4; ++e) num[e] = __builtin_fmaf(x[e], f2, num[e] * f1);
    s = make_float2(top, __builtin_fmaf(o.y, f2, s.y * f1));
}
// Pieces meet in pairs, and every fourth pair in one of four parts: piece e of pair i of a part, and the sum of a part's N pairs, if there are any.
__device__ __forceinline__ int few_piece(int part, int i, int e) { return 2 * (part + 4 * i) + e; }
template <int N>
__device__ __forceinline__ void few_part(few_f32x4& num, float2& s, int part, int pieces, const few_f32x4 (&v)[N][2], const float2 (&ml)[N][2]) {
    num = few_f32x4{0.f, 0.f, 0.f, 0.f};
    s = make_float2(-INFINITY, 0.f);
#pragma unroll
    for (int i = 0; i < N; ++i) {
        few_f32x4 x = v[i][0];
        float2 o = ml[i][0];
        if (few_piece(part, i, 1) < pieces) few_add(x, o, v[i][1], ml[i][1]);
        if (few_piece(part, i, 0) >= pieces) continue;
        if (i > 0) {
            few_append(num, s, x, o);
        } else {
            num = x;
            s = o;
        }
    }
}

// Pieces per (sequence, KV head), or 0 where the batch is not small.
int few_decode_pieces(int64_t batch, int64_t num_kv_heads, int64_t max_tokens);
int launch_few_decode(const FewDecode& a, hipStream_t stream, const FewFront* front = nullptr);      // records, then their sum in `out`, if there is one

// A product behind the pieces (skinny_gemm.hip): `hidden` rows of weights, float32 sums [splits][hidden].
int few_product_splits(int64_t batch, int64_t num_q_heads, int64_t pieces, int64_t hidden);
int launch_few_product(const FewDecode& f, const void* w, int64_t hidden, float* sums, int splits, hipStream_t stream);
