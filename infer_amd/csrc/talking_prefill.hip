// Attention whose heads mix their softmax weights (talking_attention.hip), for long prompt portions, for gfx950 (MI355X).  bf16 in, float32
// accumulate; keys and values go straight from their pages (tile_pages.h) into operands.
//
//     w_h(i, j) = e^{s_h(i, j)} / (1 + sum_j' e^{s_h(i, j')}) ,   o_h(i) = c sum_j (sum_g T[h][g] w_g(i, j)) v_j
//
// A running rescale does not commute with the mixture, so denominators come first, and the scores are computed twice instead of passing
// through memory:
//   talk_lse_kernel   log2 of every (head, query)'s denominator; a wavefront owns 16 U queries of a head
//   talk_mix_kernel   a workgroup of eight wavefronts owns 16 QT queries and ALL heads, UH heads per wavefront, and walks the keys in
//                     steps of 32:
//       S^T[key, query] = K[key, :] . q^T           per wavefront its heads; weights e^{S - lse} go to LDS as two bf16 pieces each
//                                                   (2^-17), one record [head][piece] per (query, key)
//       P'^T[key, h]    = W^T[key, g] . T^T[g, h]    per wavefront 2 QT queries, the pieces side by side along k; to LDS as bf16
//       O^T[v, query]  += V^T[v, key] . P'^T[key, query]      per wavefront its heads
//                     Nothing is rescaled: what is added up is final, and the keys of a few queries can be split over workgroups, whose
//                     sums talk_sum_kernel adds up.  Between the barriers that enclose the mixture a wavefront computes the scores
//                     of the next step and the sums of this one, the two wavefronts of a vector unit in opposite order.
// A lane's eight results of the first two products are those of eight consecutive keys (tile_row_token).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "elem.h"
#include "pieces.h"
#include "tile_pages.h"

namespace {

typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

constexpr int kStep = kTileTokens;
constexpr int kLseWaves = 4;
constexpr int kMixWaves = 8;
constexpr float kLow = -1e30f;            // a maximum before any key was seen; finite, since hidden scores are -inf
constexpr float kLazy = 8.f;              // log2 units by which a sum's terms may exceed one before it is rescaled
constexpr float kBound = 100.f;           // log2 units: powers of scores below it add up in a float as they are

// The order in which workgroups take blocks of queries.  A block sees as many keys as its place in its sequence says, so some take a hundred times as long as
// others, and a launch is done when its last workgroup is.  Sorted: units of `run` neighbouring blocks in falling order of the steps of their last one, over all
// sequences, dealt to the dies in turn, so that a unit's blocks share what the L2 of their die holds.  Walks of more than `most` steps are cut into parts of one
// length (at most `splits`), which are turns of their own.  Otherwise blocks by their place in their sequences.  The call, us, 16 heads, by place in their sequences
// with walks whole, or all cut alike where blocks are few / now (5 .. 7 of each by the order of loads and the rows at the end of talk_mix_kernel), in turn on one card, the
// shortest of five times ten: 8 sequences of 700 .. 2300 tokens 311 / 281, 6 of 1214 .. 2313 285 / 256, one of 6000 503 / 403, one of 600 49 / 36, 16 of 100 .. 1500 218 / 200, 4 of
// 500 .. 1500 behind 1500 cached 329 / 258, 64 of 61 .. 179 60 / 51.  Runs of 1, 2, 4, 8 blocks: 8 of 700 .. 2300 263, 261, 265, 272 (the same inputs again and again).
constexpr int kLanes = 64;
constexpr int kMostKeys = 1 << 30;      // of a sequence, so that numbers of steps can be doubled
struct Turns { int queries, run, most, splits; bool sorted; int units; };      // queries of a block; run, queries: powers of two; units of the longest sequence
struct Turn { int seq, q_beg, sq, shift, block, part, parts; };        // shift: keys in front of the sequence's first query
__device__ __forceinline__ int steps_of(int last_q, int shift) { return last_q + shift < 0 ? 1 : (last_q + shift) / kStep + 1; }
__device__ __forceinline__ int parts_of(const Turns& t, int steps) {
    const int n = (steps + t.most - 1) / t.most;
    return n < t.splits ? n : t.splits;
}
// parts of the walks of block `block` of a sequence
__device__ __forceinline__ int parts_of_block(const Turns& t, int sq, int shift, int block) {
    if (t.splits == 1) return 1;
    const int blocks = (sq + t.queries - 1) >> __builtin_ctz(t.queries), in_front = (blocks - 1 - block) & ~(t.run - 1), end = (blocks - in_front) * t.queries;
    return parts_of(t, steps_of((end < sq ? end : sq) - 1, shift));
}
__device__ __forceinline__ int wave_sum(int x) {
    auto ror = [](int v, auto C) { return __builtin_amdgcn_update_dpp(0, v, decltype(C)::value, 0xf, 0xf, false); };
    x += ror(x, std::integral_constant<int, 0x128>{});
    x += ror(x, std::integral_constant<int, 0x124>{});
    x += ror(x, std::integral_constant<int, 0x122>{});
    x += ror(x, std::integral_constant<int, 0x121>{});
    return __builtin_amdgcn_readlane(x, 0) + __builtin_amdgcn_readlane(x, 16) + __builtin_amdgcn_readlane(x, 32) + __builtin_amdgcn_readlane(x, 48);
}
// Without an order: turn `rest` of sequence s.  Few sequences begin with their last blocks; of many, that are not sorted whatever their walks, blocks go by their place in
// their sequences, so that the longest ones begin (80 of 100 .. 600 tokens, us, by their last blocks / by place: 8, 16, 32 heads 153 / 148, 248 / 247, 506 / 481, 32 ungrouped
// ones 1134 / 984; 64 of 61 .. 179, 32 ungrouped ones 147 / 156).
__device__ __forceinline__ Turn plain_turn(const Turns& t, int s, int rest, int nseq, const int32_t* cu_q, const int32_t* cu_k) {
    const int part = t.splits == 1 ? 0 : rest / t.units, unit = rest - part * t.units;
    const int q_beg = cu_q[s], sq = cu_q[s + 1] - q_beg, shift = cu_k[s + 1] - cu_k[s] - sq, blocks = (sq + t.queries - 1) >> __builtin_ctz(t.queries);
    const int at = (nseq > kLanes ? t.units : blocks) - 1 - unit, block = at < blocks ? at : -1;
    const int parts = block < 0 ? 1 : parts_of_block(t, sq, shift, block);
    return {s, q_beg, sq, shift, part < parts ? block : -1, part, parts};
}
// Block `inside` of the unit whose turn is number `turn`; block < 0: there is none.  Up to 64 sequences, a lane for each.
__device__ __forceinline__ Turn turn_of(const Turns& t, int turn, int inside, int nseq, const int32_t* cu_q, const int32_t* cu_k) {
    const int lane = threadIdx.x & 63;
    int q_beg = 0, sq = 0, shift = 0;
    if (lane < nseq) {
        q_beg = cu_q[lane];
        sq = cu_q[lane + 1] - q_beg;
        shift = cu_k[lane + 1] - cu_k[lane] - sq;
        if (sq > kMostKeys || sq + shift > kMostKeys) sq = 0;
    }
    const int q_bits = __builtin_ctz(t.queries), run_bits = __builtin_ctz(t.run), blocks = (sq + t.queries - 1) >> q_bits;
    // units of this lane's sequence with more than x steps
    auto longer = [&](int x) {
        const int need = x > 0 ? x * kStep + 1 - shift : 0, from = need > t.queries ? (need + t.queries - 1) >> q_bits : 1;      // blocks that end behind that
        if (sq <= 0 || (x > 0 && sq - 1 + shift < x * kStep)) return 0;
        return 1 + (blocks > from ? (blocks - from) >> run_bits : 0);
    };
    auto turns_before = [&](int x) {                             // of units with more than x steps, a turn for every part
        int n = 0;
        for (int m = 0; m < t.splits; ++m) n += longer(x > m * t.most ? x : m * t.most);
        return wave_sum(n);
    };
    int lo = 0, hi = 16;                                         // the unit has more than lo steps, and at most hi
    if (turns_before(0) <= turn) return {0, 0, 0, 0, -1, 0, 1};
    while (turns_before(hi) > turn) {                            // it ends: nobody has more than kMostKeys / kStep
        lo = hi;
        hi = 4 * hi < kMostKeys / kStep + 1 ? 4 * hi : kMostKeys / kStep + 1;
    }
    while (hi - lo > 1) {
        const int x = (lo + hi) / 2;
        if (turns_before(x) > turn) lo = x;
        else hi = x;
    }
    const int parts = parts_of(t, hi), rest = turn - turns_before(hi), mine = longer(hi), with = longer(lo) - mine;
    const int at = rest / parts;                                 // among the units of hi steps, of which a sequence has three at most
    const uint64_t one = __ballot(with & 1), two = __ballot(with & 2), below = (1ull << lane) - 1;
    const int in_front = __popcll(one & below) + 2 * __popcll(two & below);
    const int s = __builtin_ctzll(__ballot(in_front <= at && at < in_front + with));
    const int unit = __builtin_amdgcn_readlane(mine + at - in_front, s);
    auto of = [&](int x) { return __builtin_amdgcn_readlane(x, s); };
    return {s, of(q_beg), of(sq), of(shift), of(blocks) - 1 - unit * t.run - inside, rest - at * parts, parts};
}

struct TalkPrefillArgs {
    const __bf16* q; int64_t q_stride;    // [token][head * dim]
    const __bf16* keys; const __bf16* values;                 // tile_pages.h
    int key_pad, vdim_pad;
    const int32_t* bt; int64_t bt_stride; int table_cols, block_size, num_blocks;
    const int32_t* seqs; const int32_t* cu_q; const int32_t* cu_k;
    int heads, kv_heads, dim, vdim, nseq;
    float scale_log2;
    const __bf16* talk;                   // [heads][heads]
    float out_scale;
    __bf16* out; int64_t out_stride;      // [token][head * vdim]
    float* lse; int64_t tokens;           // [heads][tokens], or [sums.splits][heads][tokens] sums of powers of the BOUNDED form
    Turns turns, sums;                    // of the mixture and of the sums of exponentials
    bool bounded;
    float* part;                          // [turns.splits][tokens][heads * vdim], if turns.splits > 1
};

// The tiles of 32 keys of a sequence, one behind the other; a tile lies in one block, whose id is looked up one block ahead.
struct PageWalk {
    typedef const __attribute__((address_space(4))) int32_t* Table;       // nobody writes it meanwhile: scalar loads
    Table bt;
    int tiles_per_block, col, in_block, id, next_id;
    __device__ __forceinline__ int lookup(const TalkPrefillArgs& a, int c) const {
        const int b = bt[c < a.table_cols ? c : a.table_cols - 1];
        return b < 0 ? 0 : (b >= a.num_blocks ? a.num_blocks - 1 : b);
    }
    __device__ __forceinline__ PageWalk(const TalkPrefillArgs& a, int seq, int first = 0) {
        bt = (Table)(uintptr_t)(a.bt + (int64_t)a.seqs[seq] * a.bt_stride);
        tiles_per_block = a.block_size / kStep;
        col = first / tiles_per_block;
        in_block = first - col * tiles_per_block;
        id = lookup(a, col);
        next_id = lookup(a, col + 1);
    }
    // the tile's number among the tiles of all blocks of one head (of kv_heads), for key/value head 0; then moves on
    __device__ __forceinline__ int64_t next(const TalkPrefillArgs& a) {
        const int64_t at = (int64_t)id * a.kv_heads * tiles_per_block + in_block;
        if (++in_block == tiles_per_block) {
            in_block = 0;
            ++col;
            id = next_id;
            next_id = lookup(a, col + 1);
        }
        return at;
    }
};

// An operand at an address that all lanes share plus a byte offset of each
__device__ __forceinline__ bf16x8_t load_operand(const __bf16* base, unsigned lane_bytes) {
    return *reinterpret_cast<const bf16x8_t*>(reinterpret_cast<const char*>(base) + lane_bytes);
}

// Entries at .. at + 7 of a row of `size` (a multiple of eight), zero behind it; without a branch, behind which the compiler waits for the load
__device__ __forceinline__ bf16x8_t query_operand(const __bf16* row, int at, int size) {
    const u32x4_t x = *reinterpret_cast<const u32x4_t*>(row + (at < size ? at : 0)), zero = {0, 0, 0, 0};
    return __builtin_bit_cast(bf16x8_t, at < size ? x : zero);
}

// BOUNDED: all scores are below kBound, so that their powers need no maximum.
template <int KS, int U, bool BOUNDED>
__global__ void __launch_bounds__(64 * kLseWaves, 2) talk_lse_kernel(TalkPrefillArgs a) {
    constexpr int kLseQ = 16 * U;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, n = lane & 15;
    int h = blockIdx.x % a.heads;
    Turn turn;
    if (a.sums.sorted) turn = turn_of(a.sums, blockIdx.x / a.heads, 0, a.nseq, a.cu_q, a.cu_k);
    else {                                            // a share of the heads of all sequences for every die
        const int pairs = a.nseq * a.heads, share = (pairs + 7) / 8, i = blockIdx.x >> 3, rest = i / share, pair = (int)(blockIdx.x & 7u) * share + i - rest * share;
        if (pair >= pairs) return;
        h = pair % a.heads;
        turn = plain_turn(a.sums, pair / a.heads, rest, a.nseq, a.cu_q, a.cu_k);
    }
    const auto [b, q_beg, sq, shift, qblk, part, parts] = turn;
    if (qblk < 0) return;
    const int q0 = (qblk * kLseWaves + wave) * kLseQ;
    if (q0 >= sq) return;
    // sums of powers add up, whoever takes them; a maximum is of the whole walk (parts is 1)
    const int last_q = q0 + kLseQ < sq ? q0 + kLseQ - 1 : sq - 1, all_steps = steps_of(last_q, shift), each = (all_steps + parts - 1) / parts;
    const int s0 = part * each, steps = s0 + each < all_steps ? s0 + each : all_steps;
    float* const lse = a.lse + ((int64_t)part * a.heads + h) * a.tokens + q_beg + q0;
    if (s0 >= steps) {
        for (int i = lane; i <= last_q - q0; i += 64) lse[i] = 0.f;
        return;
    }
    bf16x8_t q[U][KS];
    float m[U], l[U];
    int limit[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int qi = q0 + 16 * u + n < sq ? q0 + 16 * u + n : sq - 1;
        limit[u] = qi + shift;
        m[u] = BOUNDED ? 0.f : kLow;
        l[u] = 0.f;
        const __bf16* qp = a.q + (int64_t)(q_beg + qi) * a.q_stride + (int64_t)h * a.dim;
#pragma unroll
        for (int j = 0; j < KS; ++j) q[u][j] = query_operand(qp, 32 * j + 8 * g, a.dim);
    }
    int k_step[KS];                                   // k-steps behind the size repeat the first one, which meets zeros
#pragma unroll
    for (int j = 0; j < KS; ++j) k_step[j] = tile_key_entry(0, 32 * j < a.key_pad ? 32 * j : 0);
    const int64_t head_at = (int64_t)(h / (a.heads / a.kv_heads)) * a.block_size * a.key_pad;
    const unsigned k_lane = 2u * (unsigned)tile_key_entry(tile_row_token(n, 0), 8 * g);
    PageWalk walk(a, b, s0);
    bf16x8_t kf[2][KS];
    auto fetch = [&]() {
        const __bf16* src = a.keys + walk.next(a) * kStep * a.key_pad + head_at;
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int j = 0; j < KS; ++j) kf[x][j] = load_operand(src + k_step[j] + tile_key_entry(tile_row_token(0, x), 0), k_lane);
    };
    fetch();
    for (int s = s0; s < steps; ++s) {
        f32x4_t sc[U][2];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int x = 0; x < 2; ++x) sc[u][x] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < KS; ++j)
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int u = 0; u < U; ++u) sc[u][x] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[x][j], q[u][j], sc[u][x], 0, 0, 0);
        if (s + 1 < steps) fetch();
        const int tok0 = s * kStep;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            float sv[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) sv[i] = sc[u][i >> 2][i & 3];
            if (tok0 + kStep - 1 > q0 + 16 * u + shift) {        // the earliest query of the tile does not see all of it
                const int rel = limit[u] - tok0 - 8 * g;
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    if (i > rel) sv[i] = -INFINITY;
            }
            if constexpr (BOUNDED) {
#pragma unroll
                for (int i = 0; i < 8; ++i) l[u] += __builtin_amdgcn_exp2f(sv[i] * a.scale_log2);
            } else {
                float mx = sv[0];
#pragma unroll
                for (int i = 1; i < 8; ++i) mx = fmaxf(mx, sv[i]);
                mx *= a.scale_log2;
                const bool grow = mx > m[u] + kLazy;
                if (__any(grow)) {
                    l[u] *= grow ? __builtin_amdgcn_exp2f(m[u] - mx) : 1.f;
                    m[u] = grow ? mx : m[u];
                }
#pragma unroll
                for (int i = 0; i < 8; ++i) l[u] += __builtin_amdgcn_exp2f(__builtin_fmaf(sv[i], a.scale_log2, -m[u]));
            }
        }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
        if constexpr (BOUNDED) {
#pragma unroll
            for (int x = 16; x <= 32; x *= 2) l[u] += __shfl_xor(l[u], x, 64);
            if (g == 0 && q0 + 16 * u + n < sq) lse[16 * u + n] = l[u];
            continue;
        }
#pragma unroll
        for (int x = 16; x <= 32; x *= 2) {
            const float m2 = __shfl_xor(m[u], x, 64), l2 = __shfl_xor(l[u], x, 64), top = fmaxf(m[u], m2);
            l[u] = l[u] * exp2f(m[u] - top) + l2 * exp2f(m2 - top);
            m[u] = top;
        }
        const float top = fmaxf(m[u], 0.f);
        if (g == 0 && q0 + 16 * u + n < sq)
            lse[16 * u + n] = top + log2f(l[u] * exp2f(m[u] - top) + exp2f(-top));
    }
}

// Address in LDS of byte `at` of the record of (query q, key token), REC bytes long.  Lanes that write (16 queries, one key) and lanes
// that read (16 keys of tile_row_token, one query) meet all banks.  For the second eight of 16 queries the halves of every 16 bytes
// are swapped (`swapped`).  What a query, a key and `at` contribute is independent.
template <int REC>
__device__ __forceinline__ int record_place(int q, int token, int at) {
    const int low = REC == 128 ? (token & 3) | (token >> 1 & 4) : REC == 64 ? (token >> 1 & 1) | (token >> 2 & 2) : token >> 3 & 1;
    return (q * kStep + token) * REC + at ^ (low << 4) ^ ((q & 15) << 4) ^ (q & 8);
}
__device__ __forceinline__ bool swapped(int q) { return q & 8; }
template <int HP>
__device__ __forceinline__ int mixed_place(int q, int slot, int g) { return (q * HP + (slot ^ (q & (HP - 1)))) * 64 + 16 * (g ^ ((q >> 2) & 3)); }

// SHARE: the heads of a wavefront have one key/value head.
template <int KS, int VT, int UH, int QT, bool SHARE>
__global__ void __launch_bounds__(64 * kMixWaves) __attribute__((amdgpu_waves_per_eu(2, 2))) talk_mix_kernel(TalkPrefillArgs a) {
    constexpr int HP = kMixWaves * UH, Q = 16 * QT;              // head slots, queries
    constexpr int kRec = 4 * HP;                                 // bytes of a record: every head's weight in two pieces
    constexpr int KP = UH == 4 ? 2 : 1, RT = UH == 4 ? 2 : 1;    // k-steps and head tiles of the mixture
    constexpr int UK = SHARE ? 1 : UH, UW = UH / UK;             // key heads of a wavefront, query heads of each
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    unsigned char* wbuf = lds;                                   // [Q][32 keys][kRec]
    unsigned char* pbuf = wbuf + Q * kStep * kRec;               // [Q][HP][32 keys] bf16
    bf16x8_t* talk = reinterpret_cast<bf16x8_t*>(pbuf + Q * HP * 2 * kStep);       // [2][KP][RT][64]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, n = lane & 15;
    Turn turn;
    const int die = blockIdx.x & 7u, dealt = blockIdx.x >> 3;
    if (a.turns.sorted) turn = turn_of(a.turns, dealt / a.turns.run * 8 + die, dealt % a.turns.run, a.nseq, a.cu_q, a.cu_k);
    else {                                            // a share of the sequences for every die, if that comes out even
        const int share = a.nseq % 8 == 0 ? a.nseq / 8 : a.nseq, i = a.nseq % 8 == 0 ? dealt : (int)blockIdx.x, rest = i / share, s = i - rest * share;
        turn = plain_turn(a.turns, a.nseq % 8 == 0 ? die * share + s : s, rest, a.nseq, a.cu_q, a.cu_k);
    }
    const auto [b, q_beg, sq, shift, qblk, split, parts] = turn;
    if (qblk < 0) return;
    const int sk = sq + shift;
    const int q0 = qblk * Q;
    const int last_q = q0 + Q < sq ? q0 + Q - 1 : sq - 1, all_steps = steps_of(last_q, shift), each = (all_steps + parts - 1) / parts;
    const int s0 = split * each, steps = s0 + each < all_steps ? s0 + each : all_steps;
    if (s0 >= steps) return;
    const int sum_parts = a.bounded ? parts_of_block(a.sums, sq, shift, q0 >> __builtin_ctz(a.sums.queries)) : 0;
    const int group = a.heads / a.kv_heads;

    PageWalk walk(a, b, s0);
    int64_t tile = walk.next(a), tile1 = s0 + 1 < steps ? walk.next(a) : tile, tile2 = s0 + 2 < steps ? walk.next(a) : tile1;
    bf16x8_t q[UH][QT][KS];
    float lse[UH][QT];
    int limit[QT];
    int64_t k_head[UK], v_head[UK];
#pragma unroll
    for (int u = 0; u < UH; ++u) {
        const int h = wave * UH + u < a.heads ? wave * UH + u : a.heads - 1;         // a surplus slot repeats the last head and meets zeros in T
        if (u % UW == 0) {
            k_head[u / UW] = (int64_t)(h / group) * a.block_size * a.key_pad;
            v_head[u / UW] = (int64_t)(h / group) * a.block_size * a.vdim_pad;
        }
#pragma unroll
        for (int t = 0; t < QT; ++t) {
            const int qi = q0 + 16 * t + n < sq ? q0 + 16 * t + n : sq - 1;
            limit[t] = qi + shift;
            lse[u][t] = a.lse[(int64_t)h * a.tokens + q_beg + qi];
            const __bf16* qp = a.q + (int64_t)(q_beg + qi) * a.q_stride + (int64_t)h * a.dim;
#pragma unroll
            for (int j = 0; j < KS; ++j) q[u][t][j] = query_operand(qp, 32 * j + 8 * g, a.dim);
        }
    }
    if (a.bounded) {
        for (int i = 1; i < sum_parts; ++i)
#pragma unroll
            for (int u = 0; u < UH; ++u)
#pragma unroll
                for (int t = 0; t < QT; ++t) {
                    const int h = wave * UH + u < a.heads ? wave * UH + u : a.heads - 1;
                    lse[u][t] += a.lse[((int64_t)i * a.heads + h) * a.tokens + q_beg + limit[t] - shift];
                }
#pragma unroll
        for (int u = 0; u < UH; ++u)
#pragma unroll
            for (int t = 0; t < QT; ++t) lse[u][t] = log2f(1.f + lse[u][t]);
    }
    const unsigned k_lane = 2u * (unsigned)tile_key_entry(tile_row_token(n, 0), 8 * g), v_lane = 2u * (unsigned)tile_value_entry(8 * g, n);
    bf16x8_t kf[KS];
    // half x of the keys of head uk; k-steps behind the size repeat the first one, which meets zeros in q
    auto fetch_k = [&](int64_t tile, int uk, int x) __attribute__((always_inline)) {
        const __bf16* src = a.keys + tile * kStep * a.key_pad + k_head[uk] + tile_key_entry(tile_row_token(0, x), 0);
#pragma unroll
        for (int j = 0; j < KS; ++j) kf[j] = load_operand(src + tile_key_entry(0, 32 * j < a.key_pad ? 32 * j : 0), k_lane);
    };
    // T^T: entry i of lane (g, n) is column (head) 16 s + 4 g + i / 2 of row (head) 16 r + n, once for either piece; behind it the same
    // for records whose halves are swapped
    for (int i = tid; i < 2 * KP * RT * 64; i += 64 * kMixWaves) {
        const int s = i / (64 * RT) % KP, r = i / 64 % RT, to = 16 * r + i % 16;
        bf16x8_t x;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int from = 16 * s + 4 * (i % 64 / 16) + (i < KP * RT * 64 ? e : e ^ 4) / 2;
            const bool in = from < HP && from < a.heads && to < a.heads;
            const __bf16 w = a.talk[in ? to * a.heads + from : 0];           // no branch around a load: behind each there would be a wait
            x[e] = in ? w : (__bf16)0.f;
        }
        talk[i] = x;
    }

    f32x4_t acc[UH][QT][VT];
#pragma unroll
    for (int u = 0; u < UH; ++u)
#pragma unroll
        for (int t = 0; t < QT; ++t)
#pragma unroll
            for (int v = 0; v < VT; ++v) acc[u][t][v] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    constexpr int kRing = UH == 2 ? 3 : 4;                                     // value operands under way
    bf16x8_t vf[kRing];
    // operand i of the step: tile i % VT of head i / VT; tiles behind the size repeat the first one and are not stored
    auto fetch_v = [&](int64_t tile, int i) __attribute__((always_inline)) {
        const int v = i % VT;
        vf[i % kRing] = load_operand(a.values + tile * kStep * a.vdim_pad + v_head[i / VT] + tile_value_entry(0, 16 * v < a.vdim_pad ? 16 * v : 0), v_lane);
    };
    const int w_fixed = record_place<kRec>(n, 8 * g, wave * UH * 4);
    const int whole = (q0 + shift + 1) / kStep;                  // steps of which the first query sees every key

    // scores and weights of step s, half of the keys of a key head at a time; its first keys are in kf
    auto scores = [&](auto masked, int s, int64_t tile) __attribute__((always_inline)) {
        constexpr bool MASKED = decltype(masked)::value;
        const int tok0 = s * kStep, w_base = renewed(w_fixed);
#pragma unroll
        for (int i = 0; i < 2 * UK; ++i) {
            const int uk = i / 2, x = i % 2;
            // two score tiles at a time: of two heads, or of two query tiles
            constexpr int GW = UW >= 2 ? 2 : 1, GT = UW >= 2 || QT == 1 ? 1 : 2;
#pragma unroll
            for (int w0 = 0; w0 < UW; w0 += GW)
#pragma unroll
                for (int t0 = 0; t0 < QT; t0 += GT) {
                    f32x4_t sc[GW][GT];
#pragma unroll
                    for (int w = 0; w < GW; ++w)
#pragma unroll
                        for (int t = 0; t < GT; ++t) sc[w][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int j = 0; j < KS; ++j)
#pragma unroll
                        for (int w = 0; w < GW; ++w)
#pragma unroll
                            for (int t = 0; t < GT; ++t)
                                sc[w][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[j], q[uk * UW + w0 + w][t0 + t][j], sc[w][t], 0, 0, 0);
                    if (w0 + GW == UW && t0 + GT == QT && i + 1 < 2 * UK) fetch_k(tile, (i + 1) / 2, (i + 1) % 2);   // these are used up
#pragma unroll
                    for (int t = 0; t < GT; ++t) {
                        uint32_t pieces[GW][4];
#pragma unroll
                        for (int w = 0; w < GW; ++w)
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                float p = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[w][t][e], a.scale_log2, -lse[uk * UW + w0 + w][t0 + t]));
                                if (MASKED && e > limit[t0 + t] - tok0 - 8 * g - 4 * x) p = 0.f;
                                pieces[w][e] = round_pack(head(p), p - head(p));
                            }
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            unsigned char* to = wbuf + (w_base ^ record_place<kRec>(0, 4 * x + e, (uk * UW + w0) * 4)) + (t0 + t) * (16 * kStep * kRec);
                            if constexpr (GW == 2) *reinterpret_cast<u32x2_t*>(to) = u32x2_t{pieces[0][e], pieces[1][e]};
                            else *reinterpret_cast<uint32_t*>(to) = pieces[0][e];
                        }
                    }
                }
        }
    };
    // the mixture, for queries 2 QT wave and on
    auto mix = [&]() __attribute__((always_inline)) {
        const int g = renewed(lane >> 4), n = renewed(lane & 15);
        bf16x8_t tf[KP][RT];
#pragma unroll
        for (int y = 0; y < KP; ++y)
#pragma unroll
            for (int r = 0; r < RT; ++r) tf[y][r] = talk[((swapped(2 * QT * wave) ? KP : 0) + y) * RT * 64 + r * 64 + lane];
#pragma unroll
        for (int k = 0; k < 2 * QT; ++k) {
            if (UH == 4) __builtin_amdgcn_sched_barrier(0);      // one query at a time: registers
            const int qi = 2 * QT * wave + k;
            f32x4_t mixed[RT][2];
#pragma unroll
            for (int x = 0; x < 2; ++x) {
#pragma unroll
                for (int r = 0; r < RT; ++r) mixed[r][x] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int y = 0; y < KP; ++y) {
                    const bf16x8_t wf = *reinterpret_cast<const bf16x8_t*>(wbuf + record_place<kRec>(qi, tile_row_token(n, x), 64 * y + 16 * (UH == 1 ? g & 1 : g) ^ (qi & 8)));
#pragma unroll
                    for (int r = 0; r < RT; ++r) mixed[r][x] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, tf[y][r], mixed[r][x], 0, 0, 0);
                }
            }
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                bf16x8_t p;
#pragma unroll
                for (int i = 0; i < 8; ++i) p[i] = (__bf16)mixed[r][i >> 2][i & 3];
                const int to = 16 * r + n;
                if (HP >= 16 || to < HP) *reinterpret_cast<bf16x8_t*>(pbuf + mixed_place<HP>(qi, to, g)) = p;
            }
        }
    };
    // weighted sum of the values of step s, the first of which are in vf; behind it kf has the first keys of next_tile
    auto sums = [&](auto masked, int s, int64_t tile, int64_t next_tile) __attribute__((always_inline)) {
        constexpr bool MASKED = decltype(masked)::value;         // some values lie behind the last one
        const int left = sk - s * kStep;
        const int g = renewed(lane >> 4), n = renewed(lane & 15);
#pragma unroll
        for (int uk = 0; uk < UK; ++uk) {
            bf16x8_t pb[UW][QT];
#pragma unroll
            for (int w = 0; w < UW; ++w)
#pragma unroll
                for (int t = 0; t < QT; ++t) pb[w][t] = *reinterpret_cast<const bf16x8_t*>(pbuf + mixed_place<HP>(16 * t + n, wave * UH + uk * UW + w, g));
#pragma unroll
            for (int v = 0; v < VT; ++v) {
                const int i = uk * VT + v;
                bf16x8_t x = vf[i % kRing];
                if constexpr (MASKED)                        // values behind the last one may be anything
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (8 * g + e >= left) x[e] = (__bf16)0.f;
#pragma unroll
                for (int w = 0; w < UW; ++w)
#pragma unroll
                    for (int t = 0; t < QT; ++t) acc[uk * UW + w][t][v] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, pb[w][t], acc[uk * UW + w][t][v], 0, 0, 0);
                if (i + kRing < UK * VT) fetch_v(tile, i + kRing);
                if (i + kRing == UK * VT) {                  // the next step's first keys take the place of the last values
                    __builtin_amdgcn_sched_barrier(0);
                    fetch_k(next_tile, 0, 0);
                }
            }
        }
    };
    auto first_values = [&](int64_t tile) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kRing; ++i) fetch_v(tile, i);
    };
    __syncthreads();                                             // T
    // A wavefront's part of the walk; both forms meet the same barriers.  Loops of their own, since accumulators that several branches
    // change would be copied where these meet.
    auto run = [&](auto first) __attribute__((always_inline)) {
        constexpr bool SUMS_FIRST = decltype(first)::value;
        fetch_k(tile, 0, 0);
        if (s0 < whole) scores(std::false_type{}, s0, tile);
        else scores(std::true_type{}, s0, tile);
        if constexpr (SUMS_FIRST) first_values(tile);
        else fetch_k(tile1, 0, 0);
        __syncthreads();
        auto step = [&](auto masked, int s) __attribute__((always_inline)) {
            mix();
            __syncthreads();
            if constexpr (SUMS_FIRST) {
                sums(masked, s, tile, tile1);
                if (!decltype(masked)::value || s + 1 < steps) scores(masked, s + 1, tile1);
                first_values(tile1);
            } else {
                if (!decltype(masked)::value || s + 1 < steps) scores(masked, s + 1, tile1);
                first_values(tile);
                sums(masked, s, tile, tile2);
            }
            __syncthreads();
            tile = tile1;
            tile1 = tile2;
            if (s + 3 < steps) tile2 = walk.next(a);
        };
        const int plain = whole < steps ? whole : steps;
        int s = s0;
        for (; s + 1 < plain; ++s) step(std::false_type{}, s);
        for (; s < steps; ++s) step(std::true_type{}, s);
    };
    if (wave < kMixWaves / 2) run(std::true_type{});
    else run(std::false_type{});
    // Results as they lie are 8 bytes of every 32 of a token's row; they go through LDS, which nobody needs any more, so that a head's
    // row is written in one piece.  With the pages looked up before the queries are asked for, so that their latency runs under these
    // loads, the call takes, us, before / now: 64 sequences of 61 .. 179 tokens 66.1 / 59.7, 23 of 67 .. 80 25.9 / 23.7, 8 of 700 .. 2300 311 / 302,
    // 6 of 1214 .. 2313 281 / 275, one of 600 36.4 / 36.3.
    constexpr int kOutRow = 32 * VT + 16, kRowLanes = 4 * VT;    // bytes; lanes that write a row
    static_assert(kMixWaves * 16 * kOutRow <= Q * kStep * kRec + Q * HP * 2 * kStep, "room in LDS");
    unsigned char* obuf = lds + wave * 16 * kOutRow;
    // The lane number is made anew: what is worked out of it is otherwise kept from before the walk, in registers that the walk is short of
    // (the form for 17 to 32 heads of 128: 81 spilled registers, 12 to 14 of them met in a step, against 18 and 3 or 4; 32 heads, 8 x 2048 1003 / 701 us, 64 sequences
    // of 61 .. 179 tokens 131 / 95).
    auto finish = [&](int lane, int g, int n) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < UH; ++u) {
            const int h = wave * UH + u;
            if (h >= a.heads) continue;
#pragma unroll
            for (int t = 0; t < QT; ++t) {
                const int qi = q0 + 16 * t + n;
                if (parts > 1) {
                    if (qi >= sq) continue;
                    float* part = a.part + (((int64_t)split * a.tokens + q_beg + qi) * a.heads + h) * a.vdim + 4 * g;
#pragma unroll
                    for (int v = 0; v < VT; ++v)
                        if (16 * v + 4 * g < a.vdim) *reinterpret_cast<f32x4_t*>(part + 16 * v) = acc[u][t][v];
                    continue;
                }
#pragma unroll
                for (int v = 0; v < VT; ++v) {
                    bf16x4_t x;
#pragma unroll
                    for (int e = 0; e < 4; ++e) x[e] = (__bf16)(acc[u][t][v][e] * a.out_scale);
                    *reinterpret_cast<bf16x4_t*>(obuf + n * kOutRow + 32 * v + 8 * g) = x;
                }
                const int row = lane / kRowLanes, col = 4 * (lane % kRowLanes);
#pragma unroll
                for (int i = 0; i < 16 * kRowLanes / 64; ++i) {
                    const int r = row + 64 / kRowLanes * i;
                    const bf16x4_t x = *reinterpret_cast<const bf16x4_t*>(obuf + r * kOutRow + 2 * col);
                    if (q0 + 16 * t + r < sq && col < a.vdim)
                        *reinterpret_cast<bf16x4_t*>(a.out + (int64_t)(q_beg + q0 + 16 * t + r) * a.out_stride + (int64_t)h * a.vdim + col) = x;
                }
            }
        }
    };
    const int late = renewed(lane);
    finish(late, late >> 4, late & 15);
}

// Sums of the parts of walks that were cut.  Workgroup: a token.
__global__ void __launch_bounds__(256) talk_sum_kernel(TalkPrefillArgs a) {
    const int cols = a.heads * a.vdim, b = blockIdx.y, q_beg = a.cu_q[b], sq = a.cu_q[b + 1] - q_beg, shift = a.cu_k[b + 1] - a.cu_k[b] - sq, qi = blockIdx.x;
    if (qi >= sq) return;
    const int block = qi / a.turns.queries, parts = parts_of_block(a.turns, sq, shift, block);
    if (parts < 2) return;
    const int end = (block + 1) * a.turns.queries, steps = steps_of((end < sq ? end : sq) - 1, shift), each = (steps + parts - 1) / parts, there = (steps + each - 1) / each;
    const float* from = a.part + (int64_t)(q_beg + qi) * cols;
    __bf16* out = a.out + (int64_t)(q_beg + qi) * a.out_stride;
    for (int i = 4 * threadIdx.x; i < cols; i += 1024) {
        f32x4_t sum = {0.f, 0.f, 0.f, 0.f};
        for (int s = 0; s < there; ++s) sum += *reinterpret_cast<const f32x4_t*>(from + s * a.tokens * cols + i);
        bf16x4_t x;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = (__bf16)(sum[e] * a.out_scale);
        *reinterpret_cast<bf16x4_t*>(out + i) = x;
    }
}

constexpr int64_t kUnits = 256;
// How long the mixture takes, in us as a model has it.  The walks of `blocks` workgroups, the longest of `longest` steps, are taken for eight lengths, `walks`, each of
// an eighth of them; those of more than `most` steps are cut.  A workgroup takes cost.fixed beside its steps (loads of the queries, the first step's way through LDS,
// stores), and kLeft more if it leaves a part.  The launch takes as long as its longest workgroup, as all work shared out over the units, and, since of the 256 k + 1
// longest workgroups some k + 1 are on one unit, k + 1 times the shortest of these; parts are written and read once more, mb of them a workgroup.
// The constants were fitted to what is chosen by them: 8, 16 and 32 heads of 128 and of 64 with 8 key heads, 16 and 32 ungrouped ones of 128, 40 batches each (1 to
// 24 sequences of 190 to 6000 tokens, equal and unequal ones, 64 to 100 of up to 600, 4 to 200 with 64 to 1500 new tokens behind 100 to 8000 cached), every cut that
// mix_turns() looks at timed.  What it takes is 2.1 % longer than the best of them on average (16 heads of 128: 1.9 %), in nine of ten cases 6.6 % at most, 25 % at worst (100 sequences
// with 64 new tokens behind 100 to 3000).  The call, us, with constants of 16 heads for all forms and nothing for what parts are in memory / now: 8 x 2048 with 8 heads
// 251 / 225, 16 heads 343 / 327, 32 heads 706 / 643, 16 x 1000 with 8 heads 158 / 127, of 64 115 / 94, 4 x 2048 with 16 of 64 174 / 151, 64 with 64 new tokens behind 4000 and
// 8, 16, 32 heads 363 / 343, 556 / 452, 863 / 687, and 65 of them whole / now 533 / 368, 681 / 595, 1340 / 1154; 8 of 700 .. 2300 with 16 heads 279 / 280, 6 of 1214 .. 2313 254 / 262.
constexpr int kShares = 8;
constexpr double kLeft = 7.1, kBusy = 1.08, kBusyCut = 1.23, kTraffic = 0.56;
struct Cost { double fixed, step; };
// values of up to 64 and of more; 64 and 32 queries of up to 8 heads, 32 and 16 of up to 16, 16 of up to 32
constexpr Cost kCosts[2][5] = {{{26.9, 3.63}, {18.7, 2.37}, {19.7, 4.26}, {5.6, 2.77}, {4.6, 2.31}}, {{25.8, 4.15}, {19.7, 2.89}, {19., 4.73}, {18.4, 3.35}, {12.3, 4.65}}};
double mix_time(const double (&walks)[kShares], double blocks, int longest, int most, const Cost& cost, double mb) {
    struct Piece { double time, count; } pieces[kShares];
    double number = 0., work = 0., left = 0.;
    for (int i = 0; i < kShares; ++i) {
        const int parts = std::max(1, (int)std::ceil(walks[i] / most - 1e-9));
        pieces[i] = {cost.fixed + (parts > 1 ? kLeft : 0.) + walks[i] / parts * cost.step, blocks / kShares * parts};
        number += pieces[i].count;
        work += pieces[i].count * pieces[i].time;
        if (parts > 1) left += pieces[i].count;
    }
    double t = std::max(cost.fixed + (most < longest ? kLeft : 0.) + most * cost.step, (most < longest ? kBusyCut : kBusy) / kUnits * work);
    if (number > kUnits) {
        std::sort(pieces, pieces + kShares, [](const Piece& a, const Piece& b) { return a.time > b.time; });
        double longer = 0.;
        int rounds = 1;
        for (const Piece& p : pieces)
            for (longer += p.count; rounds < 4 && longer > rounds * kUnits; ++rounds) t = std::max(t, (rounds + 1) * p.time);
    }
    return t + kTraffic * mb * left;
}
// Finding a turn takes 1 to 2 us, which is not worth it where walks are short or all run at once: 24 sequences of 151 .. 441 78 us against 74, 23 of 67 .. 80
// 28 against 25, but 32 of 100 .. 600 111 against 148.
Turns arranged(Turns t, int64_t num_seqs, int64_t max_seqlen_q, int64_t max_keys, int64_t at_once) {
    const int64_t blocks = (max_seqlen_q + t.queries - 1) / t.queries, steps = (max_keys + kStep - 1) / kStep;
    t.sorted = num_seqs <= kLanes && max_keys <= kMostKeys && steps > 16 && t.splits * blocks * num_seqs > at_once;
    if (!t.sorted) t.run = 1;
    t.units = (int)((blocks + t.run - 1) / t.run);
    return t;
}
// Steps of a token's walk: its sequence is about as long as the mean of the mean and the longest one, and it is in its middle
double steps_seen(int64_t num_seqs, int64_t tokens, int64_t max_seqlen_q, int64_t max_keys) {
    return ((double)(max_keys - max_seqlen_q) + 0.25 * ((double)tokens / num_seqs + (double)max_seqlen_q)) / kStep + 0.5;
}
// Walks of more sequences than can be sorted are cut as well, and go out as they lie.
Turns mix_turns(int64_t heads, int64_t vdim, int64_t num_seqs, int64_t tokens, int64_t max_seqlen_q, int64_t max_keys) {
    const int64_t steps = (max_keys + kStep - 1) / kStep;
    const double exponent = std::max((double)steps / steps_seen(num_seqs, tokens, max_seqlen_q, max_keys) - 1., 0.004);
    double walks[kShares];
    for (int i = 0; i < kShares; ++i) walks[i] = std::max(1., (double)steps * std::pow((kShares - i - 0.5) / kShares, exponent));
    const int wide = heads <= 8 ? 4 : heads <= 16 ? 2 : 1, narrow = heads <= 8 ? 2 : 1;
    Turns turns{};
    double best = 0.;
    for (int tiles = wide; tiles >= narrow; tiles /= 2) {
        const int queries = 16 * tiles;
        const double blocks = std::min((double)tokens / queries + 0.5 * num_seqs, (double)((max_seqlen_q + queries - 1) / queries) * num_seqs);
        const Cost& cost = kCosts[vdim > 64][(heads <= 8 ? 0 : heads <= 16 ? 2 : 4) + (tiles < wide)];
        int64_t last = 0;
        for (const double share : {1., 0.8, 0.65, 1. / 2, 0.4, 1. / 3, 1. / 4, 1. / 6, 1. / 8}) {
            const int64_t most = std::min(std::max<int64_t>(4, (int64_t)std::ceil(share * (double)steps - 1e-9)), steps);
            if (most == last) continue;                          // a short walk has few cuts, and its call waits for the host: 32 sequences of 27 to 85 tokens 18.9 -> 17.5 us
            last = most;
            const double t = mix_time(walks, blocks, (int)steps, (int)most, cost, 4e-6 * (double)(queries * heads * vdim));
            if (best > 0. && t >= best) continue;
            best = t;
            turns = Turns{queries, 2, (int)most, (int)((steps + most - 1) / most), true, 0};
        }
    }
    return arranged(turns, num_seqs, max_seqlen_q, max_keys, kUnits);
}
Turns sum_turns(int64_t heads, int64_t num_seqs, int64_t tokens, int64_t max_seqlen_q, int64_t max_keys, bool bounded) {
    const int64_t steps = (max_keys + kStep - 1) / kStep;
    // few queries: more wavefronts with fewer of them each
    Turns sums{(max_seqlen_q + 63) / 64 * num_seqs * heads < 2048 ? 128 : 256, 1, (int)steps, 1, true, 0};
    // Few workgroups: no walk longer than what a place for a wavefront has to do, eight of a unit.  More even out by themselves, and parts cost each what it takes
    // to begin; the call, us, cut / whole: 400 workgroups (one sequence of 6000) 431 / 468, 240 (2 of 900 .. 1000) 62.5 / 68.7, 660 (6 of 1214 .. 2313) 274 / 265, 820 (8 of
    // 700 .. 2300) 303 / 294, 930 (16 of 100 .. 1500) 213 / 209, 960 (32 of 100 .. 600) 126 / 123.
    if (bounded && ((double)tokens / sums.queries + 0.5 * num_seqs) * heads <= 2 * kUnits) {
        const double seen = steps_seen(num_seqs, tokens, max_seqlen_q, max_keys);
        const int64_t n = std::max<int64_t>({8, (int64_t)((double)tokens / 64 * heads * seen / (8 * kUnits)) + 1, (steps + 7) / 8});
        if (5 * n <= 4 * steps) {
            sums.most = (int)n;
            sums.splits = (int)((steps + n - 1) / n);
        }
    }
    return arranged(sums, num_seqs, max_seqlen_q, max_keys, 2 * kUnits);
}
// Floats of the denominators, or of the sums that they are made of, and of all parts
int64_t sum_floats(const Turns& sums, int64_t heads, int64_t tokens) { return (sums.splits * heads * tokens + 3) / 4 * 4; }
int64_t all_floats(const Turns& sums, const Turns& turns, int64_t heads, int64_t vdim, int64_t tokens) {
    return sum_floats(sums, heads, tokens) + (turns.splits > 1 ? turns.splits * tokens * heads * vdim : 0);
}
// Turns that there are at most
int64_t most_turns(const Turns& t, int64_t num_seqs, int64_t tokens) {
    if (!t.sorted) return (int64_t)t.splits * t.units * num_seqs;
    return t.splits * (tokens / (t.queries * t.run) + num_seqs);
}

template <int KS, int U>
int launch_lse_of(const TalkPrefillArgs& a, int64_t turns, hipStream_t st) {
    const int64_t total = a.sums.sorted ? turns * a.heads : (a.nseq * (int64_t)a.heads + 7) / 8 * 8 * a.sums.units * a.sums.splits;
    if (total > 0x7fffffff) return INFER_KV_EINVAL;
    if (a.bounded) hipLaunchKernelGGL((talk_lse_kernel<KS, U, true>), dim3((unsigned)total), dim3(64 * kLseWaves), 0, st, a);
    else hipLaunchKernelGGL((talk_lse_kernel<KS, U, false>), dim3((unsigned)total), dim3(64 * kLseWaves), 0, st, a);
    return (int)hipGetLastError();
}
template <int KS>
int launch_lse(const TalkPrefillArgs& a, int64_t turns, hipStream_t st) {
    return a.sums.queries == 32 * kLseWaves ? launch_lse_of<KS, 2>(a, turns, st) : launch_lse_of<KS, 4>(a, turns, st);
}

template <int KS, int VT, int UH, int QT, bool SHARE>
int launch_mix(const TalkPrefillArgs& a, int64_t turns, int64_t max_seqlen_q, hipStream_t st) {
    const int64_t total = (turns + 7) / 8 * 8 * a.turns.run;
    if (total > 0x7fffffff) return INFER_KV_EINVAL;
    auto kernel = &talk_mix_kernel<KS, VT, UH, QT, SHARE>;
    constexpr size_t lds = (size_t)16 * QT * kStep * kMixWaves * UH * (4 + 2) + (UH == 4 ? 4 : 1) * 2048;
    static_assert(lds <= 160 * 1024, "LDS of a compute unit");
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return (int)e;
    hipLaunchKernelGGL(kernel, dim3((unsigned)total), dim3(64 * kMixWaves), lds, st, a);
    if (a.turns.splits > 1) hipLaunchKernelGGL(talk_sum_kernel, dim3((unsigned)max_seqlen_q, (unsigned)a.nseq), dim3(256), 0, st, a);
    return (int)hipGetLastError();
}

template <int KS, int VT>
int launch(const TalkPrefillArgs& a, int64_t sum_turns, int64_t turns, int64_t max_seqlen_q, hipStream_t st) {
    const int rc = launch_lse<KS>(a, sum_turns, st);
    if (rc) return rc;
    const int group = a.heads / a.kv_heads, tiles = a.turns.queries / 16;
    if (a.heads <= 8) return tiles == 4 ? launch_mix<KS, VT, 1, 4, true>(a, turns, max_seqlen_q, st) : launch_mix<KS, VT, 1, 2, true>(a, turns, max_seqlen_q, st);
    if (a.heads <= 16 && group % 2 == 0)
        return tiles == 2 ? launch_mix<KS, VT, 2, 2, true>(a, turns, max_seqlen_q, st) : launch_mix<KS, VT, 2, 1, true>(a, turns, max_seqlen_q, st);
    if (a.heads <= 16) return tiles == 2 ? launch_mix<KS, VT, 2, 2, false>(a, turns, max_seqlen_q, st) : launch_mix<KS, VT, 2, 1, false>(a, turns, max_seqlen_q, st);
    return group % 4 == 0 ? launch_mix<KS, VT, 4, 1, true>(a, turns, max_seqlen_q, st) : launch_mix<KS, VT, 4, 1, false>(a, turns, max_seqlen_q, st);
}

}  // namespace

// 1 if the sizes are served
extern "C" int infer_talking_prefill_supported(int64_t heads, int64_t dim, int64_t vdim) {
    return heads >= 1 && heads <= 32 && dim >= 8 && dim <= 128 && dim % 8 == 0 && vdim >= 8 && vdim <= 128 && vdim % 8 == 0;
}

extern "C" int64_t infer_talking_prefill_workspace_floats(int64_t heads, int64_t vdim, int64_t num_seqs, int64_t tokens, int64_t max_seqlen_q,
                                                          int64_t max_keys) {
    if (heads < 1 || vdim < 1 || num_seqs < 1 || tokens < 1 || max_seqlen_q < 1 || max_keys < 1) return 0;
    return all_floats(sum_turns(heads, num_seqs, tokens, max_seqlen_q, max_keys, true), mix_turns(heads, vdim, num_seqs, tokens, max_seqlen_q, max_keys), heads, vdim, tokens);
}

extern "C" int infer_talking_prefill(const void* q, int64_t q_stride, const void* keys, const void* values, int64_t key_pad,
                                     int64_t vdim_pad, const int32_t* block_table, int64_t bt_stride, int64_t table_cols,
                                     int64_t block_size, int64_t num_blocks, const int32_t* seqs, const int32_t* cu_q,
                                     const int32_t* cu_k, int64_t num_seqs, int64_t tokens, int64_t max_seqlen_q,
                                     int64_t max_keys, int64_t heads,
                                     int64_t kv_heads, int64_t dim, int64_t vdim, float scale, const void* talk, float out_scale,
                                     float max_score, void* out, int64_t out_stride, float* workspace, int64_t workspace_floats, void* stream) {
    if (!infer_talking_prefill_supported(heads, dim, vdim)) return INFER_KV_EUNSUPPORTED;
    if (num_seqs < 0 || max_seqlen_q < 0 || tokens < 0 || max_seqlen_q > 0x7fffffff || max_seqlen_q > tokens || max_keys < max_seqlen_q ||
        max_keys > 0x7fffffe0 || num_seqs > 65535)
        return INFER_KV_EINVAL;
    if (num_seqs == 0 || max_seqlen_q == 0) return INFER_KV_OK;
    if (!q || !keys || !values || !block_table || !seqs || !cu_q || !cu_k || !talk || !out || kv_heads < 1 || heads % kv_heads ||
        q_stride < heads * dim || out_stride < heads * vdim || key_pad != (dim + 31) / 32 * 32 || vdim_pad != (vdim + 31) / 32 * 32 ||
        block_size < kStep || block_size % kStep || block_size > (1 << 20) || table_cols < 1 || table_cols * block_size > 0x7fffffff || bt_stride < table_cols || num_blocks < 1 ||
        num_blocks > 0x7fffffff || !(scale > 0.f))
        return INFER_KV_EINVAL;
    if (q_stride % 8 || out_stride % 4 || !ptr_aligned(q, 16) || !ptr_aligned(keys, 16) || !ptr_aligned(values, 16) || !ptr_aligned(out, 8))
        return INFER_KV_EALIGN;
    const bool bounded = max_score * kLog2e <= kBound;
    const Turns mix = mix_turns(heads, vdim, num_seqs, tokens, max_seqlen_q, max_keys), cut = sum_turns(heads, num_seqs, tokens, max_seqlen_q, max_keys, true);
    if (!workspace || !ptr_aligned(workspace, 16) || workspace_floats < all_floats(cut, mix, heads, vdim, tokens)) return INFER_KV_EWORKSPACE;
    const Turns sums = bounded ? cut : sum_turns(heads, num_seqs, tokens, max_seqlen_q, max_keys, false);
    const TalkPrefillArgs a{(const __bf16*)q, q_stride, (const __bf16*)keys, (const __bf16*)values, (int)key_pad, (int)vdim_pad, block_table,
                            bt_stride, (int)table_cols, (int)block_size, (int)num_blocks, seqs, cu_q, cu_k, (int)heads, (int)kv_heads, (int)dim,
                            (int)vdim, (int)num_seqs, scale * kLog2e, (const __bf16*)talk, out_scale, (__bf16*)out, out_stride, workspace, tokens, mix,
                            sums, bounded, workspace + sum_floats(sums, heads, tokens)};
    hipStream_t st = (hipStream_t)stream;
    const int64_t most_sums = most_turns(sums, num_seqs, tokens), most_mix = most_turns(mix, num_seqs, tokens);
    if (dim <= 64) return vdim <= 64 ? launch<2, 4>(a, most_sums, most_mix, max_seqlen_q, st) : launch<2, 8>(a, most_sums, most_mix, max_seqlen_q, st);
    return vdim <= 64 ? launch<4, 4>(a, most_sums, most_mix, max_seqlen_q, st) : launch<4, 8>(a, most_sums, most_mix, max_seqlen_q, st);
}
