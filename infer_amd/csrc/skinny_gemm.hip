// Split-K weight-streaming GEMM for decode-sized batches on gfx950 (MI355X):
//
//     y[M, N] = x[M, K] . w[N, K]^T          bf16 in, float32 accumulate, bf16 out,  M <= 128
//
// This is `Linear.forward` (infer/ops/MLP.py:103-149, `F.linear`; the op `matmul(input, weight,
// output)` of src/bindings.cpp:7) at the shapes of a decode step whose weight matrix has few rows
// (o_proj, down_proj: N = hidden size).  There a tiled library GEMM has too few output tiles to keep
// 256 compute units streaming; this kernel cuts K as well, so that every unit reads its share of
// the weights exactly once, and pays for it with float32 partial sums that a second kernel adds.
//
// * The weights stream through LDS (weight_stream.h): skinny_stream_kernel, whose wavefronts split K among themselves, past up to 8 rows of the batch, up to 32
//   with at most 5120 weight rows and K < 8192, and 17 to 64 with 8193 to 12288 weight rows (16 also past many with a short K); otherwise
//   skinny_shared_kernel, whose wavefronts share every step of K and with it the batch.  Up to 64 rows K is cut over workgroups only where there are few of
//   them.
// * SK == 1: the accumulators are rounded to bf16 and stored.  SK > 1: float32 partial sums
//   [SK][M][N] go to the workspace and `skinny_gemm_reduce_kernel` adds them and rounds once.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/infer_kv.h"
#include "decode_few.h"
#include "weight_stream.h"

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kBN = 128;         // weight rows per workgroup past more than 64 of the batch
constexpr int kKC = 128;         // K elements per chunk

struct GemmArgs {
    const uint16_t* x; int64_t x_stride0;
    const uint16_t* w;           // [N, K] row-major
    uint16_t* y; int64_t y_stride0;
    float* partial;              // [SK][M][N] when SK > 1
    int m, n, k;
    int chunks;                  // K chunks per split
};
static_assert(sizeof(GemmArgs) == 64, "a line: arguments in another one cost 0.2 us of 5");

// The weight rows n0 .. end - 1 of which a workgroup takes its ROWS (GATED: ROWS / 2 gate rows, and the up rows of the same places), and where it begins its
// walk over k (stream_start): 2^TURN workgroups at one place, 0 everybody at the front.  Gate rows and up rows are halves of one matrix, and a product of both
// has to add up as the two by themselves do.  So without a gate a workgroup that is not cut over k lies in one half (APART), and there 2^HALF_TURN of them begin
// at the place of the twice as many that have the same rows with a gate.  Us, two workgroups of other halves side by side / the halves one behind the other:
// 6144 x 4096, 48 of the batch 17.0 / 16.8, 151936 x 4096, 4 183.8 / 179.9.  APART is no argument: working it out in kernels of 5 us costs 0.1.
template <bool GATED, int ROWS, int TURN, bool APART, int HALF_TURN = TURN>
struct Share {
    static_assert(!(GATED && APART) && (TURN > 0 || !APART), "halves of which somebody else has the other, and walks that begin somewhere");
    int n0, end, turn;
    __device__ __forceinline__ explicit Share(const GemmArgs& a) {
        const int b = blockIdx.x, half = a.n / 2;
        if constexpr (APART) {
            const int each = (half + ROWS - 1) / ROWS, at = b >= each ? b - each : b;
            n0 = at * ROWS + (b >= each ? half : 0);
            end = b >= each ? a.n : half;
            turn = at >> HALF_TURN;
        } else {
            n0 = b * (GATED ? ROWS / 2 : ROWS);
            end = GATED ? half : a.n;
            turn = TURN == 0 ? 0 : b >> (GATED ? HALF_TURN + 1 : TURN);
        }
    }
};

__device__ __forceinline__ u32x4 load16(const uint16_t* p) { return *reinterpret_cast<const u32x4*>(p); }

__device__ __forceinline__ float round_bf16(float x) { return (float)(__bf16)x; }

// Four sums of row `row` at the places 16 r + 4 g of a workgroup whose weights begin at row n0 and end in front of row `end` (GATED: as described below)
template <bool GATED>
__device__ __forceinline__ void finish_tile(const GemmArgs& a, int end, int split, int n0, int r, int row, int g, f32x4_t sum) {
    if constexpr (GATED) {                         // lanes g = 0, 1 hold gates 4 g + e, lanes g + 2 the up columns of the same place
        bf16x4_t v;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float gate = round_bf16(sum[e]), up = __shfl_xor(gate, 32, 64);
            v[e] = (__bf16)(round_bf16(gate / (1.0f + expf(-gate))) * up);
        }
        const int col = n0 + 8 * r + 4 * g;
        if (g < 2 && col < end && row < a.m) *reinterpret_cast<bf16x4_t*>(a.y + (int64_t)row * a.y_stride0 + col) = v;
    } else {
        const int col = n0 + 16 * r + 4 * g;
        if (col >= end || row >= a.m) return;          // a multiple of 8: a quad is in or out as a whole
        if (a.partial) {
            *reinterpret_cast<f32x4_t*>(a.partial + ((int64_t)split * a.m + row) * a.n + col) = sum;
        } else {
            bf16x4_t v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = (__bf16)sum[e];
            *reinterpret_cast<bf16x4_t*>(a.y + (int64_t)row * a.y_stride0 + col) = v;
        }
    }
}

// 16 RT rows of weights past up to 16 MT rows of the batch, NW wavefronts with D steps each in LDS.  GATED: the weights are gate rows and as
// many up rows, a.n / 2 each; a tile is eight gate rows and the eight up rows of the same places, and y = silu(gate) * up with the
// roundings of storing both and reading them again.
template <int RT, int MT, int NW, int D, bool GATED, int TURN, bool APART>
__global__ void __launch_bounds__(64 * NW) skinny_stream_kernel(GemmArgs a) {
    constexpr int kRing = D * stream_stage_bytes(RT, MT), kLds = NW * (kRing > 1024 * RT * MT ? kRing : 1024 * RT * MT);
    __shared__ __attribute__((aligned(1024))) unsigned char lds[kLds];
    const int lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int half = a.n / 2, split = blockIdx.y;
    const Share<GATED, 16 * RT, TURN, APART> share(a);
    const int64_t k_lo = (int64_t)split * a.chunks * kKC;
    const __bf16* w[2 * RT];
    const __bf16* x[2 * MT];
#pragma unroll
    for (int i = 0; i < 2 * RT; ++i) {
        int row = share.n0 + stream_row() + 8 * (GATED ? i / 2 : i);
        row = (row < share.end ? row : share.end - 1) + (GATED && (i & 1) ? half : 0);
        w[i] = (const __bf16*)a.w + (int64_t)row * a.k + k_lo;
    }
#pragma unroll
    for (int i = 0; i < 2 * MT; ++i) {
        const int row = stream_row() + 8 * i;
        x[i] = (const __bf16*)a.x + (int64_t)(row < a.m ? row : a.m - 1) * a.x_stride0 + k_lo;
    }
    f32x4_t acc[RT][MT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[r][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    stream_product<RT, MT, NW, D, (TURN > 0)>(w, x, a.chunks * kKC, share.turn, wave, lds + wave * kRing, acc);
    stream_reduce<RT, MT, NW>(acc, wave, lds, [&](int r, int t, f32x4_t sum) { finish_tile<GATED>(a, share.end, split, share.n0, r, 16 * t + n, g, sum); });
}

// The same, the steps of k shared by the wavefronts (SharedStream)
template <int RT, int MT, bool GATED, bool APART>
__global__ void __launch_bounds__(256) skinny_shared_kernel(GemmArgs a) {
    __shared__ __attribute__((aligned(1024))) unsigned char lds[SharedStream<RT, MT>::kRing];
    const int lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15, half = a.n / 2, split = blockIdx.y;
    const Share<GATED, 16 * RT, 3, APART, 2> share(a);
    const int64_t k_lo = (int64_t)split * a.chunks * kKC;
    shared_product<RT, MT>(a.chunks * kKC, share.turn, lds,
        [&](int i) {
            int row = share.n0 + stream_row() + 8 * (GATED ? i / 2 : i);
            row = (row < share.end ? row : share.end - 1) + (GATED && (i & 1) ? half : 0);
            return (const __bf16*)a.w + (int64_t)row * a.k + k_lo;
        },
        [&](int i) {
            const int row = stream_row() + 8 * i;
            return (const __bf16*)a.x + (int64_t)(row < a.m ? row : a.m - 1) * a.x_stride0 + k_lo;
        },
        [&](int r, int t, f32x4_t sum) { finish_tile<GATED>(a, share.end, split, share.n0, r, 16 * t + n, g, sum); });
}

// What stands in front of a product of few rows: y = norm(x + residual) w^T, where x may still be the pieces of a split product.
struct NormSource {
    const float* partial; int splits; int64_t split_stride, partial_stride0;      // if partial: x[r] = bf16(sum over splits of partial[s][r])
    const uint16_t* x; int64_t x_stride0;
    const uint16_t* residual; int64_t residual_stride0;                            // or null
    uint16_t* sum; int64_t sum_stride0;                                            // x + residual
    const uint16_t* gain;
    float inv_k, eps;
};
constexpr int kFewRows = 2, kFewPieces = 8, kNormGroup = 512;       // rows of the batch; pieces of a row of kNormGroup elements in all
constexpr int kFewMany = 16384;                                     // from so many weight rows on a workgroup takes 32
constexpr int kFewPad = 64;                                         // bytes behind a row in LDS: rows meet other banks

// A product of few rows with the norm of its input in front of it.  Every workgroup norms the rows for itself, out of the second-level cache
// and while its weights are on their way, since a launch in between costs more: a step of a 0.6B model, one sequence, 1063 -> 949 us with
// 56 of its 252 launches less.  The first workgroup leaves x + residual, in another place than the residual, which others still read.
// NP: pieces of 64 x 8 elements per wavefront.  Sums, order and roundings are those of rms_norm_kernel and of skinny_stream_kernel: the
// same bits.
// What bounds it is what all workgroups read in front, rows times their bytes.  Norm and product, us, two launches / one, for 1, 2, 4 rows:
// 4096 x 1024 behind four pieces 6.2 / 4.2, 6.4 / 4.3, 6.4 / 6.8; 6144 x 1024 gated 7.6 / 5.7, 7.6 / 6.0, 7.7 / 8.0; 6144 x 4096 14.1 / 12.6,
// 13.5 / 13.3, 13.7 / 22.4; 24576 x 4096 gated 35.5 / 33.7, 33.8 / 42.4.  So one row up to 4096 elements, two of half as many.
template <int RT, int NP, bool GATED, int TURN, bool APART>
__global__ void __launch_bounds__(256) norm_product_kernel(GemmArgs a, NormSource f) {
    constexpr int NW = 4, D = 4, kRing = D * stream_stage_bytes(RT, 0);
    static_assert(NW * kRing >= NW * RT * 1024, "sums of the wavefronts");
    extern __shared__ __attribute__((aligned(1024))) unsigned char few_lds[];      // rings, then rows of x, then sums of squares
    const int lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int half = a.n / 2;
    const Share<GATED, 16 * RT, TURN, APART> share(a);
    const int row_bytes = 2 * a.k + kFewPad;
    unsigned char* xs = few_lds + NW * kRing;
    float* squares = reinterpret_cast<float*>(xs + a.m * row_bytes);               // [kFewRows][8]
    const __bf16* w[2 * RT];
#pragma unroll
    for (int i = 0; i < 2 * RT; ++i) {
        int row = share.n0 + stream_row() + 8 * (GATED ? i / 2 : i);
        row = (row < share.end ? row : share.end - 1) + (GATED && (i & 1) ? half : 0);
        w[i] = (const __bf16*)a.w + (int64_t)row * a.k;
    }
    const int groups = (a.k + kNormGroup - 1) / kNormGroup, pieces = a.m * groups;
    int row[NP], c[NP];
    bool in[NP];
    u32x4 gain[NP], res[NP], raw[NP];
    f32x4 lo[NP], hi[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const int p = wave + NW * i;
        row[i] = p / groups;
        c[i] = 64 * (p - row[i] * groups) + lane;
        in[i] = p < pieces && 8 * c[i] < a.k;
        if (!in[i]) row[i] = c[i] = 0;
        gain[i] = load16(f.gain + 8 * c[i]);
        if (f.residual) res[i] = load16(f.residual + row[i] * f.residual_stride0 + 8 * c[i]);
        if (!f.partial) raw[i] = load16(f.x + row[i] * f.x_stride0 + 8 * c[i]);
        lo[i] = hi[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    if (f.partial) {
        constexpr int kBatch = 4;                        // splits requested at once
        for (int s0 = 0; s0 < f.splits; s0 += kBatch) {
            f32x4 l[kBatch][NP], h[kBatch][NP];
#pragma unroll
            for (int b = 0; b < kBatch; ++b)
#pragma unroll
                for (int i = 0; i < NP; ++i) {
                    const float* p = f.partial + (s0 + b < f.splits ? s0 + b : s0) * f.split_stride + row[i] * f.partial_stride0 + 8 * c[i];
                    l[b][i] = *reinterpret_cast<const f32x4*>(p);
                    h[b][i] = *reinterpret_cast<const f32x4*>(p + 4);
                }
#pragma unroll
            for (int b = 0; b < kBatch; ++b)
                if (s0 + b < f.splits)
#pragma unroll
                    for (int i = 0; i < NP; ++i) { lo[i] += l[b][i]; hi[i] += h[b][i]; }
        }
    }
    auto norm = [&] {
        float v[NP][8];
#pragma unroll
        for (int i = 0; i < NP; ++i) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[i][e] = f.partial ? round_bf16(lo[i][e]) : __builtin_bit_cast(float, e & 1 ? raw[i][e / 2] & 0xffff0000u : raw[i][e / 2] << 16);
                v[i][4 + e] = f.partial ? round_bf16(hi[i][e]) : __builtin_bit_cast(float, e & 1 ? raw[i][2 + e / 2] & 0xffff0000u : raw[i][2 + e / 2] << 16);
            }
            if (f.residual) {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[i][e] += __builtin_bit_cast(float, e & 1 ? res[i][e / 2] & 0xffff0000u : res[i][e / 2] << 16);
                if (blockIdx.x == 0 && in[i]) {
                    bf16x8 o;
#pragma unroll
                    for (int e = 0; e < 8; ++e) o[e] = (__bf16)v[i][e];
                    *reinterpret_cast<bf16x8*>(f.sum + row[i] * f.sum_stride0 + 8 * c[i]) = o;
                }
            }
            float ss = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) ss += v[i][e] * v[i][e];
            if (!in[i]) ss = 0.f;
#pragma unroll
            for (int m = 32; m >= 1; m >>= 1) ss += __shfl_xor(ss, m, 64);
            const int p = wave + NW * i;
            if (lane == 0 && p < pieces) squares[8 * (p / groups) + p % groups] = ss;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            if (!in[i]) continue;
            float ss = 0.f;
            for (int j = 0; j < groups; ++j) ss += squares[8 * row[i] + j];
            const float rs = rsqrtf(ss * f.inv_k + f.eps);
            bf16x8 o;
#pragma unroll
            for (int e = 0; e < 8; ++e)
                o[e] = (__bf16)(round_bf16(v[i][e] * rs) * __builtin_bit_cast(float, e & 1 ? gain[i][e / 2] & 0xffff0000u : gain[i][e / 2] << 16));
            *reinterpret_cast<bf16x8*>(xs + row[i] * row_bytes + 16 * c[i]) = o;
        }
        __syncthreads();
    };
    f32x4_t acc[RT][1];
#pragma unroll
    for (int r = 0; r < RT; ++r) acc[r][0] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    stream_product_held<RT, NW, D, (TURN > 0)>(w, xs + (n < a.m ? n : a.m - 1) * row_bytes + 16 * g, a.k, share.turn, wave, few_lds + wave * kRing, norm, acc);
    stream_reduce<RT, 1, NW>(acc, wave, few_lds, [&](int r, int, f32x4_t sum) { finish_tile<GATED>(a, share.end, 0, share.n0, r, n, g, sum); });
}

// A product, split over k, of one sequence's attention that still lies in pieces (decode_few.h): a workgroup has up to kPieceHeads heads of k, whose pieces
// it adds up while its weights are on their way: a launch less in every layer, and what the pieces cost is a read of the second-level cache.  A step
// of 28 layers of a 0.6B model, 700 tokens, 779 -> 731 us (751 with the pieces added up eight by eight, a chain of eleven sums instead of seven).  Sums, order and roundings are those of few_decode_sum_kernel and of skinny_stream_kernel:
// the same bits.
constexpr int kPieceHeads = 4, kPieceSets = 4;                      // heads of a workgroup; sets of four pairs of pieces of a head
__global__ void __launch_bounds__(256) piece_product_kernel(GemmArgs a, FewDecode f) {
    constexpr int NW = 4, D = 4, kRing = D * stream_stage_bytes(1, 0);
    __shared__ __attribute__((aligned(1024))) unsigned char lds[NW * kRing];
    __shared__ f32x4 sums[2][kPieceHeads][32];
    __shared__ float2 mls[2][kPieceHeads];
    __shared__ __attribute__((aligned(16))) __bf16 xs[kPieceHeads * kKC];
    const int lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n0 = blockIdx.x * 16, split = blockIdx.y;
    const __bf16* w[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int row = n0 + stream_row() + 8 * i;
        w[i] = (const __bf16*)a.w + (int64_t)(row < a.n ? row : a.n - 1) * a.k + (int64_t)split * a.chunks * kKC;
    }
    // 32 lanes hold the columns of a head, the workgroup's halves two of the four parts of the pieces each
    const int c = threadIdx.x & 31, in = (threadIdx.x >> 5) & 3, half = threadIdx.x >> 7;
    const int head = split * a.chunks + (in < a.chunks ? in : 0), kv = head / f.group, q = head - kv * f.group, floats = few_record_floats(f.group);
    const float* rec = f.rec + (int64_t)kv * f.pieces * floats;
    f32x4 v[2][kPieceSets][2];
    float2 ml[2][kPieceSets][2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < kPieceSets; ++i)
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int p = few_piece(2 * half + j, i, e);
                const float* from = rec + (int64_t)(p < f.pieces ? p : 0) * floats;
                v[j][i][e] = *reinterpret_cast<const f32x4*>(from + q * kKC + 4 * c);
                ml[j][i][e] = *reinterpret_cast<const float2*>(from + f.group * kKC + 2 * q);
            }
    const int pieces = few_pieces_of(f, f.ctx[0]);
    auto add = [&] {
        f32x4 num[2];
        float2 s[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            few_part<kPieceSets>(num[j], s[j], 2 * half + j, pieces, v[j], ml[j]);
            if (half) {
                sums[j][in][c] = num[j];
                if (c == 0) mls[j][in] = s[j];
            }
        }
        __syncthreads();
        if (!half) {
            if (2 < pieces) few_add(num[0], s[0], num[1], s[1]);
#pragma unroll
            for (int j = 2; j < 4; ++j)
                if (2 * j < pieces) few_add(num[0], s[0], sums[j - 2][in][c], mls[j - 2][in]);
            const float inv = s[0].y > 0.f ? 1.f / s[0].y : 0.f;
            bf16x4_t o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = (__bf16)(num[0][e] * inv);
            if (in < a.chunks) *reinterpret_cast<bf16x4_t*>(xs + in * kKC + 4 * c) = o;
        }
        __syncthreads();
    };
    f32x4_t acc[1][1] = {{f32x4_t{0.f, 0.f, 0.f, 0.f}}};
    stream_product_held<1, NW, D, false>(w, reinterpret_cast<const unsigned char*>(xs) + 16 * g, a.chunks * kKC, 0, wave, lds + wave * kRing, add, acc);
    stream_reduce<1, 1, NW>(acc, wave, lds, [&](int r, int, f32x4_t sum) { finish_tile<false>(a, a.n, split, n0, r, n, g, sum); });
}

struct ReduceArgs {
    const float* partial;
    uint16_t* y; int64_t y_stride0;
    int m, n, splits;
};

// y[row][8 c .. 8 c + 7] = bf16(sum over splits), one thread per 8 outputs
__global__ void __launch_bounds__(256) skinny_gemm_reduce_kernel(ReduceArgs a) {
    const int per_row = a.n / 8;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (int64_t)a.m * per_row) return;
    const int row = (int)(i / per_row), c = (int)(i - (int64_t)row * per_row);
    f32x4 lo = {0.f, 0.f, 0.f, 0.f}, hi = {0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < a.splits; ++s) {
        const float* p = a.partial + ((int64_t)s * a.m + row) * a.n + 8 * c;
        lo += *reinterpret_cast<const f32x4*>(p);     // plain loads: lo and hi are two instructions on the same lines
        hi += *reinterpret_cast<const f32x4*>(p + 4);
    }
    union { __bf16 h[8]; u32x4 u; } r;
#pragma unroll
    for (int e = 0; e < 4; ++e) { r.h[e] = (__bf16)lo[e]; r.h[4 + e] = (__bf16)hi[e]; }
    *reinterpret_cast<u32x4*>(a.y + (int64_t)row * a.y_stride0 + 8 * c) = r.u;
}

// Weight rows of a workgroup.  At most 8 of the batch, and up to 32 past few rows: 16, wavefronts that split k (skinny_stream_kernel), which are as good
// as any (32 past many with a short k: n = 151936 48 us with k = 1024, 54 with 16 rows).  More of the batch: the activations, which every workgroup reads
// whole, want many rows, and the chip wants a workgroup for every compute unit: wavefronts that share the steps of k (skinny_shared_kernel), 16 times
// shared_tiles rows.  Us, wavefronts that split k (before they began in different places) / this:
//   64 of the batch   24576 x 4096 gate and up 42.8 / 33.7   151936 x 4096 240 / 202   151936 x 1024 66 / 59   32000 x 4096 56 / 41   49152 x 2048 50 / 33
//   32                24576 x 4096 34 / 31   151936 x 4096 213 / 192   16384 x 2048 17 / 12   8192 x 4096 16.1 / 12.8
//   16                24576 x 4096 34 / 31   151936 x 4096 209 / 184   16384 x 2048 17 / 11.5   4: 30.8 / 30.7, 187 / 181 (these now 175), 14.9 / 11.9 (12.6)
// Three tiles of rows are none of its shapes, and 48 rows fill the chip from 8193 to 12288 of them: there 17 to 64 split k (12288 x 4096 with 64 of the batch
// 21.2 / 22.6).  Few weight rows and a long k: 16 rows give every compute unit
// a workgroup that reads the batch once per 16 rows; 64 rows, cut over k, read it a quarter as often.  Unreduced sums, 16 / 64 rows (split k): n = 4096,
// k = 12288 9 of the batch 18.5 / 17.1, 16 20.2 / 17.3, 32 25.9 / 19.0 (now 17.3); with a shorter k the launch that adds the sums up for those who want
// them costs more than that (n = 4096, k = 4096, 16: 8.4 / 10.4 reduced).  More than 4096 weight rows and a very long k: tiles of 64 rows leave
// 160 workgroups that read the batch for half of k each; 128 rows, cut twice as often, read it half as often: 5120 x 25600, 64 of the batch 68 / 49 us (with 4096
// weight rows the further sums take what that gives: 4096 x 12288 20.7 / 20.2, a step that adds them up 776 / 783).
constexpr int64_t kMany = 40960, kLongK = 8192, kUnits = 256;
// 16-row tiles of a workgroup of skinny_shared_kernel: those with which the compute units are through first, counting what a tile takes as three and what every
// 16 of the batch take beside them as one (151936 x 4096, us per round of 2 / 4 / 8 / 12 / 16 / 20 tiles: 64 of the batch 15 / 24 / 43 / 58 / 74 / 101, 16
// 11 / 19 / 38 / 53 / 67 / 92).
int shared_tiles(int64_t m, int64_t n) {
    int best = 0;
    int64_t least = 0;
    for (int t : {2, 4, 6, 8, 10, 12, 14, 16, 20}) {
        const int64_t groups = (n + 16 * t - 1) / (16 * t), takes = (groups + kUnits - 1) / kUnits * (3 * t + (m <= 16 ? 1 : m <= 32 ? 2 : 4));
        if (best == 0 || takes <= least) {
            best = t;
            least = takes;
        }
    }
    return best;
}
int rows_per_workgroup(int64_t m, int64_t n, int64_t k) {
    if (m > 64) return kBN;
    if (n <= 5120) return m > 32 && n > 4096 && k >= 2 * kLongK ? 128 : m > 32 || (m > 8 && k >= kLongK) ? 64 : 16;
    if (m <= 16 && n >= kMany && k <= 2048) return 32;
    if (m <= 8) return 16;
    return m > 16 && n > 8192 && n <= 12288 ? 48 : 16 * shared_tiles(m, n);
}

// Split-K factor: a divisor of the chunk count that brings the grid to at least one workgroup per
// compute unit (256 on MI355X) while leaving every split at least four chunks to stream.
int choose_splits(int64_t m, int64_t n, int64_t k) {
    const int64_t rows = rows_per_workgroup(m, n, k), tiles = (n + rows - 1) / rows;
    const int64_t chunks = k / kKC;
    if (m <= 64 && n > 5120) return 1;          // what 180 workgroups lack of the chip is less than the sums of a split cost
    int best = 1;
    for (int s = 1; s <= 32; ++s) {
        if (chunks % s != 0 || chunks / s < 4) continue;
        best = s;
        if (tiles * s >= 256) break;
    }
    if (m <= 32 || m > 64) return best;
    // A workgroup's start and end cost as much as four chunks, and two of 64 rows fit a compute unit's LDS, but what the unit takes from memory they share:
    // of the smaller factors, the first with the shortest chain of chunks.  Unreduced sums, 64 of the batch, us, the first factor with 256 workgroups / this
    // (wavefronts that split k): 3072 x 4096 12.8 / 9.7, 2560 x 4096 12.3 / 9.3, 5120 x 3072 15.0 / 10.6, 2560 x 9728 20.0 / 17.2, 5120 x 12288 38.0 / 27.4.
    auto chain = [&](int s) { return (tiles * s + 255) / 256 * (chunks / s + 4); };
    for (int s = best - 1; s >= 1; --s)
        if (chunks % s == 0 && chain(s) <= chain(best)) best = s;
    return best;
}

// Whether wavefronts that split k begin at different places of it (stream_start).  With few workgroups or a short k, finding out where costs what it gives (a
// step of 28 layers of a 0.6B model 729 / 733 us).  Products that norm their input have the bits of those that do not: the rule is one for both.  What the order of
// a gate's sums in products without one costs (Share), steps of three layers of an 8B model, 1, 4, 24, 48, 64 sequences, without / with it: 417 / 422, 437 / 439,
// 500 / 500, 548 / 546, 579 / 577; by themselves 121 products of other sizes took 1.004 times as long, the most 40832 x 4736 with 25 of the batch 58.2 / 61.4.
bool begins_anywhere(int64_t n, int64_t k) { return k > 2048 && n > 8 * kUnits; }
// Whether the halves of the weight rows are dealt out apart (Share): where walks begin at different places and the halves can be gate and up
bool dealt_apart(const GemmArgs& a, bool turned, int splits) { return turned && splits == 1 && a.n % 16 == 0; }
// Workgroups for so many weight rows each; twice those of a half are no round of the compute units more
unsigned workgroups(const GemmArgs& a, bool apart, int rows) { return (unsigned)(apart ? 2 * ((a.n / 2 + rows - 1) / rows) : (a.n + rows - 1) / rows); }

template <bool GATED, int MT>
void launch_shared(const GemmArgs& a, int tiles, int splits, hipStream_t st) {
    const bool apart = !GATED && dealt_apart(a, SharedStream<2, MT>::turned(a.chunks * kKC), splits);
    const dim3 grid(workgroups(a, apart, 16 * tiles), (unsigned)splits);
#define GO(RT) case RT: \
        if (apart) hipLaunchKernelGGL((skinny_shared_kernel<RT, MT, GATED, !GATED>), grid, dim3(256), 0, st, a); \
        else hipLaunchKernelGGL((skinny_shared_kernel<RT, MT, GATED, false>), grid, dim3(256), 0, st, a); \
        return
    switch (tiles) { GO(2); GO(4); GO(6); GO(8); GO(10); GO(12); GO(14); GO(16); GO(20); }
#undef GO
}

template <bool GATED>
void launch_stream(const GemmArgs& a, int splits, hipStream_t st) {
    const int rows = rows_per_workgroup(a.m, a.n, a.k);
    const bool turned = begins_anywhere(a.n, a.chunks * kKC), apart = !GATED && a.m <= 64 && dealt_apart(a, turned, splits);
    const dim3 grid(workgroups(a, apart, rows), (unsigned)splits);
#define TURNED(RT, MT, NW, D, TURN) do { \
        if (apart) hipLaunchKernelGGL((skinny_stream_kernel<RT, MT, NW, D, GATED, TURN, !GATED && (TURN > 0)>), grid, dim3(64 * NW), 0, st, a); \
        else hipLaunchKernelGGL((skinny_stream_kernel<RT, MT, NW, D, GATED, TURN, false>), grid, dim3(64 * NW), 0, st, a); \
    } while (0)
#define GO(RT, MT, NW, D) do { if (turned) TURNED(RT, MT, NW, D, 3); else TURNED(RT, MT, NW, D, 0); } while (0)
    if (turned && a.m <= kFewRows && rows == 16 && a.n >= kFewMany && a.n < kMany) TURNED(1, 1, 4, 4, 4);      // in twos, as 32 rows with a norm in front
    else if (a.m <= 16 && rows == 16) GO(1, 1, 4, 4);
    else if (a.m <= 16 && a.n >= kMany && a.k <= 2048) TURNED(2, 1, 4, 3, 0);
    else if (a.m <= 32 && rows == 16) GO(1, 2, 4, 3);
    else if (a.m <= 32 && rows == 48) GO(3, 2, 4, 2);
    else if (a.m <= 64 && rows == 48) GO(3, 4, 4, 2);
    else if (a.m <= 64) {
        // half as many rows where 64 leave every second compute unit idle: 64 of the batch 4096 x 1024 5.5 / 4.6 us, 1024 x 3072 5.6 / 4.6
        const int tiles = a.n <= 5120 && (a.n + rows - 1) / rows * splits <= kUnits / 2 ? 2 : rows / 16;
        if (a.m <= 16) launch_shared<GATED, 1>(a, tiles, splits, st);
        else if (a.m <= 32) launch_shared<GATED, 2>(a, tiles, splits, st);
        else launch_shared<GATED, 4>(a, tiles, splits, st);
    }
    else if constexpr (!GATED) {
        // Rows of the batch in operand registers while weights came straight from memory into theirs / these, 128 of the batch, unreduced, us: 4096 x 12288
        // 29.7 / 25.3, 5120 x 25600 89 / 78, 4096 x 4096 15.1 / 13.2, 1024 x 3072 10.5 / 7.8 (with eight tiles 10.0); 72: 4096 x 4096 13.0 / 11.1
        if (grid.x * grid.y <= kUnits / 2)
            hipLaunchKernelGGL((skinny_shared_kernel<4, 8, false, false>), dim3((unsigned)((a.n + 63) / 64), (unsigned)splits), dim3(256), 0, st, a);
        else hipLaunchKernelGGL((skinny_shared_kernel<8, 8, false, false>), grid, dim3(256), 0, st, a);
    }
#undef TURNED
#undef GO
}

// Whether the kernels are ahead of the vendor's product, from a sweep of 3000 sizes (n of 64 to 262144, k of 128 to 28672) with weights that no
// cache holds, vendor / these, us.  Inside, 1.3 times as fast on average; outside, sizes of both signs:
//   65 to 128 of the batch: few weight rows give the vendor too few tiles to fill the chip (o_proj, down_proj: 4096 rows 27 and 68 us against
//     22 and 38); it is ahead on wider ones and on a short k.
//   few weight rows: all, except that a split over k whose pieces nobody takes has a launch more (33 to 64 of the batch: 5120 x 1536 8.7 / 11.5,
//     1024 x 2048 8.0 / 8.6, 1024 x 4096 14.2 / 9.8; 24: 256 x 1024 4.6 / 5.5), and that very few do not fill the chip without one (512 x 768,
//     40 5.0 / 6.7).
//   many: a short k (36864 x 128, 16 of the batch 5.7 / 8.4), a long one (5128 x 16384 35.7 / 46.8; 24584 x 28672, 64 275 / 348) and more rows than a
//     vocabulary has (262144 x 5120, 16 0.86 times as fast) are the vendor's.  From 17 of the batch the line is where workgroups of 32 to 160 rows that
//     stream by themselves fill their last round (33 to 64 of the batch 36864 rows 1.25 times as fast as the vendor, 65528 0.76 to 1.0 times).  Those that
//     share their steps are ahead behind it, too (64 of the batch 27648 x 4096 50 / 37, 64512 x 4096 121 / 80): widening it is open.
bool pays(int64_t m, int64_t n, int64_t k, bool reduced) {
    if (m > 64) return n <= 5120 && k >= 2048;
    if (n <= 5120) {
        if (!reduced || k > 2048) return true;
        if (m <= 32) return n >= 512 || k == 2048 || choose_splits(m, n, k) == 1;
        return n >= 2048 && (k == 2048 || choose_splits(m, n, k) == 1);
    }
    if ((k < 512 && n > 20480) || k > 12288 || n > 163840) return false;
    if (m <= 16) return true;
    const int64_t rows = m <= 32 ? (n >= 8192 ? 48 : 32) : n <= 8192 ? 32 : n >= 65536 ? 160 : n > 24576 ? 80 : 16 * ((n + 4095) / 4096);
    const int64_t groups = (n + rows - 1) / rows, rounds = (groups + kUnits - 1) / kUnits;
    if (m <= 32) return k <= 2048 || 10 * groups >= 7 * kUnits * rounds;
    return n <= 24576 || 20 * groups >= 17 * kUnits * rounds;
}

}  // namespace

extern "C" int infer_skinny_gemm_pays(int64_t m, int64_t n, int64_t k, int reduced) {
    return m > 0 && m <= 128 && n > 0 && k > 0 && k % kKC == 0 && n % 8 == 0 && pays(m, n, k, reduced != 0);
}

extern "C" size_t infer_skinny_gemm_workspace_bytes(int64_t m, int64_t n, int64_t k) {
    if (m <= 0 || m > 128 || n <= 0 || k <= 0 || k % kKC != 0) return 0;
    auto need = [&](int64_t rows) {
        const int s = choose_splits(rows, n, k);
        return s > 1 ? (size_t)s * (size_t)rows * (size_t)n * sizeof(float) : 0;
    };
    // enough for smaller batches as well: 33 rows may be cut less often than 32
    size_t most = need(m);
    for (int64_t rows : {8, 16, 32, 64})
        if (rows < m && need(rows) > most) most = need(rows);
    return most;
}

namespace {
// Launches the streaming kernel and, if asked and the shape was split, the reduction.  Returns the
// split count through `splits_out`.
int run_gemm(const void* x, int64_t x_stride0, const void* w, void* y, int64_t y_stride0, int64_t m, int64_t n,
             int64_t k, void* workspace, size_t workspace_bytes, bool reduce, int* splits_out, void* stream) {
    if (m < 0 || n <= 0 || k <= 0) return INFER_KV_EINVAL;
    if (splits_out) *splits_out = 0;
    if (m == 0) return INFER_KV_OK;
    if (!x || !w || !y) return INFER_KV_EINVAL;
    if (m > 128 || k % kKC != 0 || n % 8 != 0) return INFER_KV_EUNSUPPORTED;
    if (x_stride0 < k || y_stride0 < n) return INFER_KV_EINVAL;
    if ((((uintptr_t)x | (uintptr_t)w | (uintptr_t)y) & 15) || (x_stride0 & 7) || (y_stride0 & 7)) return INFER_KV_EALIGN;
    if (n > (1 << 24) || k > (1 << 24)) return INFER_KV_EINVAL;
    const int splits = choose_splits(m, n, k);
    const size_t need = splits > 1 ? (size_t)splits * (size_t)m * (size_t)n * sizeof(float) : 0;
    if (need && (!workspace || workspace_bytes < need)) return INFER_KV_EWORKSPACE;
    if (need && ((uintptr_t)workspace & 15)) return INFER_KV_EALIGN;
    GemmArgs a{(const uint16_t*)x, x_stride0, (const uint16_t*)w, (uint16_t*)y, y_stride0,
               splits > 1 ? (float*)workspace : nullptr, (int)m, (int)n, (int)k, (int)(k / kKC / splits)};
    launch_stream<false>(a, splits, (hipStream_t)stream);
    int rc = (int)hipGetLastError();
    if (splits_out) *splits_out = splits;
    if (rc != 0 || splits == 1 || !reduce) return rc;
    ReduceArgs r{(const float*)workspace, (uint16_t*)y, y_stride0, (int)m, (int)n, splits};
    const int64_t items = m * (n / 8);
    hipLaunchKernelGGL(skinny_gemm_reduce_kernel, dim3((unsigned)((items + 255) / 256)), dim3(256), 0, (hipStream_t)stream, r);
    return (int)hipGetLastError();
}
}  // namespace

extern "C" int infer_skinny_gemm_bf16(const void* x, int64_t x_stride0, const void* w, void* y, int64_t y_stride0,
                                      int64_t m, int64_t n, int64_t k, void* workspace, size_t workspace_bytes,
                                      void* stream) {
    return run_gemm(x, x_stride0, w, y, y_stride0, m, n, k, workspace, workspace_bytes, true, nullptr, stream);
}

extern "C" int infer_skinny_gemm_partial_bf16(const void* x, int64_t x_stride0, const void* w, void* y,
                                              int64_t y_stride0, int64_t m, int64_t n, int64_t k, void* workspace,
                                              size_t workspace_bytes, int* splits_out, void* stream) {
    if (!splits_out) return INFER_KV_EINVAL;
    return run_gemm(x, x_stride0, w, y, y_stride0, m, n, k, workspace, workspace_bytes, false, splits_out, stream);
}

extern "C" int infer_skinny_gate_silu_bf16(const void* x, int64_t x_stride0, const void* w, void* y, int64_t y_stride0, int64_t m, int64_t ff,
                                           int64_t k, void* stream) {
    if (m < 0 || ff <= 0 || k <= 0) return INFER_KV_EINVAL;
    if (m == 0) return INFER_KV_OK;
    if (!x || !w || !y) return INFER_KV_EINVAL;
    if (m > 64 || k % kKC != 0 || ff % 8 != 0) return INFER_KV_EUNSUPPORTED;
    if (x_stride0 < k || y_stride0 < ff || ff > (1 << 23) || k > (1 << 24)) return INFER_KV_EINVAL;
    if ((((uintptr_t)x | (uintptr_t)w | (uintptr_t)y) & 15) || (x_stride0 & 7) || (y_stride0 & 7)) return INFER_KV_EALIGN;
    const GemmArgs a{(const uint16_t*)x, x_stride0, (const uint16_t*)w, (uint16_t*)y, y_stride0, nullptr, (int)m, (int)(2 * ff), (int)k, (int)(k / kKC)};
    launch_stream<true>(a, 1, (hipStream_t)stream);
    return (int)hipGetLastError();
}

namespace {
template <bool GATED>
int launch_norm_product(const GemmArgs& a, const NormSource& f, hipStream_t st) {
    const int pieces = a.m * ((a.k + kNormGroup - 1) / kNormGroup), rows = a.n >= kFewMany ? 32 : 16;
    const size_t lds = 4 * 4 * stream_stage_bytes(rows / 16, 0) + (size_t)a.m * (2 * a.k + kFewPad) + kFewRows * 8 * sizeof(float);
    const bool turned = begins_anywhere(a.n, a.k), apart = !GATED && dealt_apart(a, turned, 1);
    const dim3 grid(workgroups(a, apart, rows));
    auto launch = [&](auto kernel) -> int {
        if (lds > 60 * 1024) {
            const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            if (e != hipSuccess) return (int)e;
        }
        hipLaunchKernelGGL(kernel, grid, dim3(256), lds, st, a, f);
        return (int)hipGetLastError();
    };
#define GO(RT, NP, TURN) return apart ? launch(&norm_product_kernel<RT, NP, GATED, TURN, !GATED && (TURN > 0)>) : launch(&norm_product_kernel<RT, NP, GATED, TURN, false>)
    // four pieces: one row of at most 2048, or two of 1024
    if (rows == 16) {
        if (pieces <= 4) GO(1, 1, 0);
        else if (turned) GO(1, 2, 3);
        else GO(1, 2, 0);
    } else {
        if (pieces <= 4) GO(2, 1, 0);
        else if (turned && a.n < kMany) GO(2, 2, 3);
        else if (turned) GO(2, 2, 2);          // as 16 rows without a norm, which a vocabulary meets: 151936 x 4096 174 us, in twos 180
        else GO(2, 2, 0);
    }
#undef GO
}
}  // namespace

extern "C" int infer_norm_product_supported(int64_t m, int64_t n, int64_t k, int gated) {
    if (m < 1 || m > kFewRows || n < 1 || k < 1 || k % kKC || n % (gated ? 16 : 8) || n > (1 << 24) || k > kFewPieces * kNormGroup) return 0;
    if (m * ((k + kNormGroup - 1) / kNormGroup) > kFewPieces || !pays(m, n, k, true)) return 0;
    return choose_splits(m, n, k) == 1;
}

extern "C" int infer_norm_product_bf16(const void* x, int64_t x_stride0, const float* partial, int64_t splits, int64_t split_stride,
                                       int64_t partial_stride0, const void* residual, int64_t residual_stride0, void* sum, int64_t sum_stride0,
                                       const void* gain, float eps, const void* w, void* y, int64_t y_stride0, int64_t m, int64_t n, int64_t k,
                                       int gated, void* stream) {
    if (!infer_norm_product_supported(m, n, k, gated)) return INFER_KV_EUNSUPPORTED;
    if (!(x || partial) || !gain || !w || !y || (residual && !sum)) return INFER_KV_EINVAL;
    if (partial ? splits < 1 || splits > 64 || partial_stride0 < k || (splits > 1 && split_stride < m * partial_stride0) : x_stride0 < k) return INFER_KV_EINVAL;
    if (residual && (residual_stride0 < k || sum_stride0 < k || sum == residual)) return INFER_KV_EINVAL;
    if (y_stride0 < (gated ? n / 2 : n)) return INFER_KV_EINVAL;
    uintptr_t all = (uintptr_t)gain | (uintptr_t)w | (uintptr_t)y | (uintptr_t)(partial ? (const void*)partial : x);
    if (residual) all |= (uintptr_t)residual | (uintptr_t)sum;
    if ((all & 15) || (y_stride0 & 7) || (partial ? (partial_stride0 | split_stride) & 3 : x_stride0 & 7) ||
        (residual && ((residual_stride0 | sum_stride0) & 7)))
        return INFER_KV_EALIGN;
    const GemmArgs a{nullptr, 0, (const uint16_t*)w, (uint16_t*)y, y_stride0, nullptr, (int)m, (int)n, (int)k, (int)(k / kKC)};
    const NormSource f{partial, (int)splits, split_stride, partial_stride0, (const uint16_t*)x, x_stride0, (const uint16_t*)residual, residual_stride0,
                       (uint16_t*)sum, sum_stride0, (const uint16_t*)gain, 1.0f / (float)k, eps};
    return gated ? launch_norm_product<true>(a, f, (hipStream_t)stream) : launch_norm_product<false>(a, f, (hipStream_t)stream);
}

// The split over k of a product of `hidden` rows past one sequence's attention in pieces, or 0 where the pieces are added up first.  A workgroup
// reads the pieces of its heads, 65 KB of four, which has to cost less than a launch, and none may wait for another's compute unit.  Attention with its
// front and the product, us, three launches / two, for 20, 700, 4000 and 20000 tokens: 16 heads on 8, 1024 rows 9.4 / 8.8, 11.1 / 9.5, 14.4 / 13.0, 26.2 / 24.7;
// 32 on 16, 512 rows 10.2 / 9.2, 11.9 / 10.4, 17.7 / 16.3, 39.4 / 38.2; but 24 on 8, 768 rows, 288 workgroups, with a sum some 0.8 longer, 9.7 / 9.9, 10.9 / 11.4,
// 13.5 / 14.0.
int few_product_splits(int64_t batch, int64_t num_q_heads, int64_t pieces, int64_t hidden) {
    const int64_t k = num_q_heads * kKC;
    if (batch != 1 || pieces < 1 || pieces > 8 * kPieceSets || hidden < 8 || hidden % 8 || hidden > 5120 || rows_per_workgroup(1, hidden, k) != 16) return 0;
    const int splits = choose_splits(1, hidden, k);
    return splits > 1 && (hidden + 15) / 16 * splits <= 256 && num_q_heads / splits <= kPieceHeads ? splits : 0;
}

int launch_few_product(const FewDecode& f, const void* w, int64_t hidden, float* sums, int splits, hipStream_t stream) {
    const int heads = f.group * f.num_kv_heads;
    const GemmArgs a{nullptr, 0, (const uint16_t*)w, nullptr, 0, sums, 1, (int)hidden, heads * kKC, heads / splits};
    hipLaunchKernelGGL(piece_product_kernel, dim3((unsigned)((hidden + 15) / 16), (unsigned)splits), dim3(256), 0, stream, a, f);
    return (int)hipGetLastError();
}
