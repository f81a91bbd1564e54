// Paged decode attention of a few sequences for gfx950 (MI355X): one query token per sequence, bf16 in, float32 sums.
//
// With little to read, what counts is the chain of waits from the launch to the result.  paged_decode.hip lays all steps of a batch end to
// end and cuts them into equal spans, for which it first reads all lengths, adds them up and gathers block ids, and it gives a compute
// unit eight wavefronts of one span each: right for a full chip, but a few sequences wait for the plan, and for a compute unit that brings 40
// KB/us.  Here workgroup (p, h, b) takes the steps p, p + P, p + 2 P, ... of 32 tokens of sequence b, a wavefront every fourth of
// them: the length, the block id and the query are requested at once, keys and values behind them, and neighbouring steps lie on different compute
// units.  A second launch adds the pieces of a head up.
//
// Layouts of the two products are those of paged_decode.hip: S^T = K Q^T with keys as they lie in memory, O^T += V^T P^T with values
// through a tile of the wavefront's own in LDS.
#include "decode_few.h"

#include <type_traits>

#include "../../include/infer_kv.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef short i16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) i16x4 lds_i16x4;

constexpr int kD = 128, kStep = 32, kWaves = 4;
constexpr int kRow = 288;                          // bytes of a value row in LDS: four rows meet different banks
constexpr int kTile = kStep * kRow;                // of a wavefront; later its partial result
static_assert(kTile >= 16 * 130 * 4 && kTile >= 17 * 272, "a partial result of 16 heads; 16 queries and a key");

__device__ __forceinline__ u32x4 load16(const uint16_t* p) { return *reinterpret_cast<const u32x4*>(p); }
__device__ __forceinline__ u32x4 load16_stream(const uint16_t* p) { return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p)); }
__device__ __forceinline__ bf16x8 as_bf16x8(u32x4 x) { return __builtin_bit_cast(bf16x8, x); }
__device__ __forceinline__ void lds_order() { __asm__ volatile("" ::: "memory"); }

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float lo16(uint32_t x) { return __builtin_bit_cast(float, x << 16); }
__device__ __forceinline__ float hi16(uint32_t x) { return __builtin_bit_cast(float, x & 0xffff0000u); }
__device__ __forceinline__ uint32_t pack(float lo, float hi) { return __builtin_bit_cast(uint32_t, bf16x2{(__bf16)lo, (__bf16)hi}); }

// Norm and rotation of a head: 16 lanes hold eight elements each.  w: weights, c, s: cosines and sines of lanes 0 .. 7 and again of 8 .. 15, the
// sines of the lower half with the other sign.  Sums, order and roundings are those of qk_norm_rope_append.hip.
__device__ __forceinline__ u32x4 norm_and_rotate(u32x4 x, u32x4 w, u32x4 c, u32x4 s, float eps) {
    auto dot2 = [](uint32_t a, uint32_t b, float z) { return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, a), __builtin_bit_cast(bf16x2, b), z, false); };
    auto ror = [](uint32_t v, auto C) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x120 + decltype(C)::value, 0xf, 0xf, false); };
    auto plus = [&](float v, auto C) { return v + __builtin_bit_cast(float, ror(__builtin_bit_cast(uint32_t, v), C)); };
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) ss = dot2(x[i], x[i], ss);
    ss = plus(ss, std::integral_constant<int, 8>{});
    ss = plus(ss, std::integral_constant<int, 4>{});
    ss = plus(ss, std::integral_constant<int, 2>{});
    ss = plus(ss, std::integral_constant<int, 1>{});
    const float r = __builtin_amdgcn_rsqf(__builtin_fmaf(ss, 1.0f / kD, eps));
    u32x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t y = pack(lo16(x[i]) * r, hi16(x[i]) * r), z = pack(lo16(y) * lo16(w[i]), hi16(y) * hi16(w[i])), one = 0x3f803f80u;
        const uint32_t other = ror(z, std::integral_constant<int, 8>{});
        o[i] = pack(dot2(pack(lo16(z) * lo16(c[i]), lo16(other) * lo16(s[i])), one, 0.f), dot2(pack(hi16(z) * hi16(c[i]), hi16(other) * hi16(s[i])), one, 0.f));
    }
    return o;
}

// FRONT: queries and new keys are as projected, and nothing of the new tokens is in the caches yet.  Every wavefront with a step norms and
// rotates the queries that it uses, four heads at once, while its keys and values are on their way; the one with a sequence's last step does
// so with the new key, takes key and value from its registers, since what it has requested is older, and puts them into the caches at its
// end, where nothing waits for the stores.  Nobody waits for those stores either: a step that holds the slot of another new token (two rows of
// one sequence, say), or its own in the middle, takes that row's key and value from the row, normed and rotated on the spot, whatever the caches
// hold there by then.  us, 16 heads on 8, front and attention in launches of their own / this: 1 x 700 tokens 9.6 / 8.0,
// 4 x 700 11.4 / 10.2, 8 x 700 16.3 / 15.4; 32 heads 9.9 / 8.2, 12.0 / 11.0, 16.8 / 16.3; a step of a 0.6B model with one sequence 820 -> 778.
// (With the stores in front of the products, with front loads of wavefronts without a step, or with heads spread as operands are, it gained nothing.)
template <bool FRONT>
__global__ void __launch_bounds__(64 * kWaves) few_decode_kernel(FewDecode a, FewFront f) {
    __shared__ __attribute__((aligned(16))) unsigned char lds_all[kWaves * kTile];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, n = lane & 15;
    const int p = blockIdx.x, h = blockIdx.y, b = blockIdx.z, G = a.group, P = a.pieces;
    unsigned char* lds = lds_all + wave * kTile;
    const int32_t* bt = a.bt + (int64_t)b * a.bt_stride0;
    const int last_col = a.max_ctx / a.block_size - 1;
    const unsigned per_block = (unsigned)a.block_size / kStep;
    auto block_of = [&](int step) {                // read whether or not the sequence has the step
        const int col = (int)((unsigned)step / per_block);
        return bt[col < last_col ? col : last_col];
    };
    const int first = p + P * wave, stride = P * kWaves;
    int blk = block_of(first), next_blk = block_of(first + stride);
    int len = a.ctx[b];
    u32x4 q[4];
    if constexpr (!FRONT) {
        const uint16_t* qp = a.q + (int64_t)b * a.q_stride0 + (int64_t)(h * G + (n < G ? n : 0)) * kD + 8 * g;
#pragma unroll
        for (int j = 0; j < 4; ++j) q[j] = load16(qp + 32 * j);
    }
    int64_t slot = -1, pos = 0;
    int row_slot = -1;                             // lane r: that of row r (a batch has no more than 64)
    auto position_of = [&](int row) {
        const int64_t at = f.positions[row];
        return at < 0 ? 0 : at >= f.max_position ? f.max_position - 1 : at;
    };
    if constexpr (FRONT) {
        slot = f.slots[b];
        pos = position_of(b);
    }
    // Heads 4 i .. 4 i + 3 of the group's queries with the new key behind them, 16 lanes each
    u32x4 x[2], w[2], cs, sn, kn[4], vn;
    auto load_heads = [&](int i, u32x4& xi, u32x4& wi) {
        const int head = 4 * i + g;
        const bool query = head < G;
        xi = load16(query ? a.q + (int64_t)b * a.q_stride0 + (int64_t)(h * G + head) * kD + 8 * n : f.k + (int64_t)b * f.k_stride0 + h * kD + 8 * n);
        wi = load16((query ? f.q_weight : f.k_weight) + 8 * n);
    };
    auto load_front = [&](bool two) {
        row_slot = f.slots[lane < a.batch ? lane : b];
        cs = load16(f.cos_sin + pos * kD + 8 * (n & 7));
        sn = load16(f.cos_sin + pos * kD + 64 + 8 * (n & 7));
        vn = load16(f.v + (int64_t)b * f.v_stride0 + h * kD + 8 * n);
        load_heads(0, x[0], w[0]);
        if (two) load_heads(1, x[1], w[1]);
    };
    constexpr int kHead = 272;                     // bytes of a head in LDS, where they change to the layout of operands
    auto finish_front = [&](int heads) {
        if (n < 8) sn ^= u32x4{0x80008000u, 0x80008000u, 0x80008000u, 0x80008000u};
        for (int i = 0; 4 * i < heads; ++i) {
            u32x4 xi = x[0], wi = w[0];
            if (i == 1) { xi = x[1]; wi = w[1]; }
            if (i > 1) load_heads(i, xi, wi);
            xi = norm_and_rotate(xi, wi, cs, sn, f.eps);
            if (4 * i + g <= G) *reinterpret_cast<u32x4*>(lds + (4 * i + g) * kHead + 16 * n) = xi;
        }
        lds_order();
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            q[j] = *reinterpret_cast<const u32x4*>(lds + (n < G ? n : 0) * kHead + 64 * j + 16 * g);
            kn[j] = *reinterpret_cast<const u32x4*>(lds + G * kHead + 64 * j + 16 * g);      // of the wavefront that needs it
        }
        lds_order();
    };
    // Key and value of row r as its own wavefront appends them
    auto new_row = [&](int r, u32x4 (&kr)[4], u32x4& vr) {
        const uint16_t* turn = f.cos_sin + position_of(r) * kD + 8 * (n & 7);
        u32x4 s = load16(turn + 64);
        if (n < 8) s ^= u32x4{0x80008000u, 0x80008000u, 0x80008000u, 0x80008000u};
        const u32x4 xr = norm_and_rotate(load16(f.k + (int64_t)r * f.k_stride0 + h * kD + 8 * n), load16(f.k_weight + 8 * n), load16(turn), s, f.eps);
        vr = load16(f.v + (int64_t)r * f.v_stride0 + h * kD + 8 * n);
        if (g == 0) *reinterpret_cast<u32x4*>(lds + 16 * n) = xr;
        lds_order();
#pragma unroll
        for (int j = 0; j < 4; ++j) kr[j] = *reinterpret_cast<const u32x4*>(lds + 64 * j + 16 * g);
        lds_order();
    };
    auto append = [&] {
        if (slot < 0 || slot >= f.num_slots) return;
        const int64_t at = (slot * a.num_kv_heads + h) * kD;
        if (n == 0)
#pragma unroll
            for (int j = 0; j < 4; ++j) *reinterpret_cast<u32x4*>(f.k_cache + at + 32 * j + 8 * g) = kn[j];
        if (g == 0) *reinterpret_cast<u32x4*>(f.v_cache + at + 8 * n) = vn;
    };
    len = len < a.max_ctx ? len : a.max_ctx;
    const int steps = len > 0 ? (len + kStep - 1) / kStep : 0;
    if constexpr (FRONT)
        if (steps == 0 && p == 0 && wave == 0) {
            load_front(G >= 4);
            finish_front(G + 1);
            append();
        }
    if (p >= steps) return;                        // the whole workgroup
    const int waves = (steps - p + P - 1) / P < kWaves ? (steps - p + P - 1) / P : kWaves;

    f32x4 acc[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;

    // Row r of key tile t is token 8 (r / 4) + 4 t + r % 4 of the step, so that lane group g ends up with tokens 8 g .. 8 g + 7.
    const uint32_t tok = (uint32_t)a.tok_stride, k_lane = (8 * (n >> 2) + (n & 3)) * tok + 8 * g, v_lane = g * tok + 8 * n;
    u32x4 k[2][4], v[8];
    int64_t row0 = 0;                              // slot of the requested step's first token
    auto request = [&](int step, int id) {
        id = __builtin_amdgcn_readfirstlane(id < 0 ? 0 : id >= a.num_blocks ? a.num_blocks - 1 : id);
        const int in = (int)((unsigned)step % per_block) * kStep;
        const int64_t at = (int64_t)id * a.blk_stride + in * a.tok_stride + (int64_t)h * kD;
        const uint16_t *kb = a.k + at, *vb = a.v + at;       // one for the wavefront; lanes differ in 32 bits
        row0 = (int64_t)id * a.block_size + in;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j) k[t][j] = load16(kb + 4 * t * a.tok_stride + k_lane + 32 * j);
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = load16_stream(vb + 4 * i * a.tok_stride + v_lane);
    };
    bool newest = false;                           // this wavefront has the sequence's last step
    if (first < steps) {
        if constexpr (FRONT) {
            newest = (steps - 1 - first) % stride == 0;
            const int heads = G + newest;
            load_front(heads > 4);
            __builtin_amdgcn_sched_barrier(0);
            request(first, blk);
            __builtin_amdgcn_sched_barrier(0);     // the rest while keys and values are on their way
            finish_front(heads);
        } else {
            request(first, blk);
        }
    }
    if (n >= G)
#pragma unroll
        for (int j = 0; j < 4; ++j) q[j] = u32x4{0u, 0u, 0u, 0u};
    for (int step = first; step < steps; step += stride) {
        if constexpr (FRONT) {
            auto put_row = [&](int i, const u32x4 (&kr)[4], u32x4 vr) {      // as token i of the step
#pragma unroll
                for (int t = 0; t < 2; ++t)
                    if (8 * (n >> 2) + (n & 3) + 4 * t == i)
#pragma unroll
                        for (int j = 0; j < 4; ++j) k[t][j] = kr[j];
#pragma unroll
                for (int t = 0; t < 8; ++t)
                    if (4 * t + g == i) v[t] = vr;
            };
            const bool own = newest && (uint64_t)(slot - row0) < kStep;
            if (own) put_row((int)(slot - row0), kn, vn);
            uint64_t others = __ballot(lane < a.batch && (uint64_t)(row_slot - row0) < kStep && !(own && lane == b));
            while (__builtin_expect(others != 0, 0)) {
                const int r = __builtin_ctzll(others);
                others &= others - 1;
                u32x4 kr[4], vr;
                new_row(r, kr, vr);
                put_row((int)(__builtin_amdgcn_readlane(row_slot, r) - row0), kr, vr);
            }
        }
        f32x4 s[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            s[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < 4; ++j) s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(k[t][j]), as_bf16x8(q[j]), s[t], 0, 0, 0);
        }
        const int tok0 = step * kStep;
        const bool tail = tok0 + kStep > len;
        if (tail) {                                // rows behind the end: their weights are 0, and 0 * NaN must not leak
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (tok0 + 4 * i + g >= len) v[i] = u32x4{0u, 0u, 0u, 0u};
        }
        lds_order();
#pragma unroll
        for (int i = 0; i < 8; ++i) *reinterpret_cast<u32x4*>(lds + (4 * i + g) * kRow + n * 16) = v[i];
        lds_order();
        if (step + stride < steps) {
            blk = next_blk;
            next_blk = block_of(step + 2 * stride);
            request(step + stride, blk);
        }
        float x[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = s[i >> 2][i & 3] * a.scale_log2;
        if (tail) {
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (tok0 + 8 * g + i >= len) x[i] = -INFINITY;
        }
        float top = x[0];
#pragma unroll
        for (int i = 1; i < 8; ++i) top = fmaxf(top, x[i]);
        top = fmaxf(top, __shfl_xor(top, 16));
        top = fmaxf(top, __shfl_xor(top, 32));
        top = fmaxf(top, m);
        const float keep = __builtin_amdgcn_exp2f(m - top);
        m = top;
        float sum = 0.f;
        bf16x8 w;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float e = __builtin_amdgcn_exp2f(x[i] - top);
            sum += e;
            w[i] = (__bf16)e;
        }
        l = l * keep + sum;
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            acc[t] *= keep;
            // in each group of 16 lanes, lane i points at four elements of row i / 4 and lane c receives column c of those rows
            const unsigned char* src = lds + (8 * g + (n >> 2)) * kRow + (16 * t + 4 * (n & 3)) * 2;
            const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(src));
            const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(src + 4 * kRow));
            const i16x8 vt = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, vt), w, acc[t], 0, 0, 0);
        }
        lds_order();
    }
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);

    // lane (g, n) holds columns 16 t + 4 g .. + 3 of head n
    auto leave = [&](float* to) {
        if (n >= G) return;
#pragma unroll
        for (int t = 0; t < 8; ++t) *reinterpret_cast<f32x4*>(to + n * kD + 16 * t + 4 * g) = acc[t];
        if (g == 0) *reinterpret_cast<float2*>(to + G * kD + 2 * n) = make_float2(m, l);
    };
    if (waves > 1) {
        lds_order();
        if (wave > 0 && wave < waves) leave(reinterpret_cast<float*>(lds));
        __syncthreads();
        if constexpr (FRONT)
            if (newest) append();                  // nothing waits for the stores any more
        if (wave > 0) return;
        for (int w = 1; w < waves; ++w) {
            const float* from = reinterpret_cast<const float*>(lds_all + w * kTile);
            const int nn = n < G ? n : 0;
            const float2 o = *reinterpret_cast<const float2*>(from + G * kD + 2 * nn);
            const float top = fmaxf(m, o.x), f1 = __builtin_amdgcn_exp2f(m - top), f2 = __builtin_amdgcn_exp2f(o.x - top);
#pragma unroll
            for (int t = 0; t < 8; ++t) acc[t] = acc[t] * f1 + *reinterpret_cast<const f32x4*>(from + nn * kD + 16 * t + 4 * g) * f2;
            l = l * f1 + o.y * f2;
            m = top;
        }
    } else {
        if (wave > 0) return;
        if constexpr (FRONT)
            if (newest) append();
    }
    leave(a.rec + (((int64_t)b * a.num_kv_heads + h) * P + p) * few_record_floats(G));
}

constexpr int kMostPieces = 64;

// Up to 8 N pieces.  Grid (query heads, batch): 32 lanes hold the columns of the head, the four halves of wavefronts every fourth pair of pieces.  Pieces are requested
// before it is known how many there are; what lies behind the last is not looked at.  The order and the roundings are those of the general kernels where every
// step has a wavefront of its own: there, too, two steps meet first (in LDS), then every fourth record.  So a single sequence with no more steps than pieces has the
// bits of those kernels (KV heads in fours, up to two query heads each: as the compiler fuses their products).
template <int N>
__global__ void __launch_bounds__(128) few_decode_sum_kernel(FewDecode a) {
    __shared__ f32x4 sums[3][32];
    __shared__ float2 mls[3];
    const int head = blockIdx.x, b = blockIdx.y, G = a.group, h = head / G, n = head - h * G, c = threadIdx.x & 31, part = threadIdx.x >> 5;
    const int floats = few_record_floats(G);
    const float* rec = a.rec + ((int64_t)b * a.num_kv_heads + h) * a.pieces * floats;
    f32x4 v[N][2];
    float2 ml[N][2];
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int p = few_piece(part, i, e);
            const float* from = rec + (int64_t)(p < a.pieces ? p : 0) * floats;
            v[i][e] = *reinterpret_cast<const f32x4*>(from + n * kD + 4 * c);
            ml[i][e] = *reinterpret_cast<const float2*>(from + G * kD + 2 * n);
        }
    const int pieces = few_pieces_of(a, a.ctx[b]);
    f32x4 num;
    float2 s;
    few_part<N>(num, s, part, pieces, v, ml);
    if (part > 0) {
        sums[part - 1][c] = num;
        if (c == 0) mls[part - 1] = s;
    }
    __syncthreads();
    if (part > 0) return;
    for (int w = 1; w < 4 && 2 * w < pieces; ++w) few_add(num, s, sums[w - 1][c], mls[w - 1]);
    const float inv = s.y > 0.f ? 1.f / s.y : 0.f;
    bf16x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = (__bf16)(num[e] * inv);
    *reinterpret_cast<bf16x4*>(a.out + (int64_t)b * a.out_stride0 + (int64_t)head * kD + 4 * c) = o;
}

}  // namespace

// Pairs of a sequence and a KV head, against paged_decode.hip, us, both launches (32 heads on 8, tokens of each sequence or of the shortest and
// longest): 1 x 700 12.5 / 7.0, 1 x 4000 18.1 / 10.3, 1 x 30000 39 / 28, 4 x 700 13.1 / 9.0, 4 x 16000 54.6 / 52.3, 4 x 100 .. 16000 33 / 23,
// 6 x 2541 .. 7125 32.5 / 31.6, 8 x 700 13.7 / 12.9, 8 x 4000 31.2 / 30.2, 8 x 100 .. 16000 29.8 / 26.9, but 8 x 1420 .. 7184 35.8 / 36.7 and 8 x
// 16000 92 / 98; 16 x 372 .. 7560 54 / 63.  So 48 pairs, and up to 64 where the table holds no more than 4096 tokens.  As many pieces as make 1024
// workgroups, but no more than there is use for: 256 of them leave a compute unit's memory requests short (8 x 100 .. 16000 55), and more
// records cost their sum (8 x 700 11.8 with 256).  Up to seven pairs 64 pieces, so that a long sequence meets the whole chip (1 x 120000, 8 heads on
// 2, 50 / 32, against 55 with 32 pieces).
int few_decode_pieces(int64_t batch, int64_t num_kv_heads, int64_t max_tokens) {
    if (batch < 1 || num_kv_heads < 1 || batch > 64 || num_kv_heads > 64) return 0;
    const int64_t pairs = batch * num_kv_heads, p = 1024 / pairs, most = pairs < 8 ? kMostPieces : kMostPieces / 2;
    if (pairs > 64 || (pairs > 48 && max_tokens > 4096)) return 0;
    return (int)(p > most ? most : p);
}

int launch_few_decode(const FewDecode& a, hipStream_t stream, const FewFront* front) {
    const dim3 pieces((unsigned)a.pieces, (unsigned)a.num_kv_heads, (unsigned)a.batch);
    if (front) hipLaunchKernelGGL(few_decode_kernel<true>, pieces, dim3(64 * kWaves), 0, stream, a, *front);
    else hipLaunchKernelGGL(few_decode_kernel<false>, pieces, dim3(64 * kWaves), 0, stream, a, FewFront{});
    const int rc = (int)hipGetLastError();
    if (rc || !a.out) return rc;
    const dim3 grid((unsigned)(a.group * a.num_kv_heads), (unsigned)a.batch), block(128);
    if (a.pieces <= 32) hipLaunchKernelGGL(few_decode_sum_kernel<4>, grid, block, 0, stream, a);
    else hipLaunchKernelGGL(few_decode_sum_kernel<8>, grid, block, 0, stream, a);
    return (int)hipGetLastError();
}
