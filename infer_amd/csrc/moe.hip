// Mixture of experts, for gfx950 (MI355X).
//
//   moe_logits_kernel / moe_route_*   router logits in float32, softmax, the choice of experts inside the best groups, weights, and
//                                     every choice's rank among the choices of its expert
//   moe_scatter_kernel    rows sorted by expert: place of every choice, token and expert of every place, row tiles
//   moe_block_kernel      products of many rows per expert: 256 rows x 256 columns per workgroup, straight from memory to LDS
//   moe_tile_kernel       products of large row tiles: 128 rows x 128 columns per workgroup, through registers to LDS
//   moe_span_kernel       products of up to 128 rows at a time: the weights pass the rows once
//   moe_uneven_kernel     the same, and blocks for the experts that have more
//   moe_row_kernel        products of up to 32 rows (decode): the weights stream past the rows; wavefronts split k or share its steps
//   moe_any_kernel        any size and element type
//
// The first product takes gate and up columns side by side and stores act = silu(gate) * up, the second stores one row per
// place; the weighted sum of a token's rows is part of the next residual step (pre_norm.hip).  A choice beyond the experts is
// the identity: place -1, no row.
#include "weight_stream.h"

#include <type_traits>

namespace {

constexpr int kThreads = 256;
constexpr int kMaxExperts = 1024;

template <class T>
struct RouteArgs {
    const T* h; int64_t h_stride;
    const T* router;                       // [all][width]
    const float* correction;               // [all] or nullptr
    int width, all, experts, top, groups, keep;
    float scale;
    int32_t* ids; float* weights; int32_t* ranks;      // [n][top]
    int32_t* counts;                       // [experts], zero before
    int n;
};

// the maximum over the wavefront's lanes, without a trip through LDS
__device__ __forceinline__ float wave_max(float x) {
    auto ror = [](float v, auto C) { return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), decltype(C)::value, 0xf, 0xf, false)); };
    x = fmaxf(x, ror(x, std::integral_constant<int, 0x128>{}));           // rotations by 8, 4, 2 and 1 within rows of 16 lanes
    x = fmaxf(x, ror(x, std::integral_constant<int, 0x124>{}));
    x = fmaxf(x, ror(x, std::integral_constant<int, 0x122>{}));
    x = fmaxf(x, ror(x, std::integral_constant<int, 0x121>{}));
    return max_xor16_32(x);
}

// The choices of one token by one wavefront; `z` are its logits in LDS.  Ties go to the lower index.
template <int NE, class T>
__device__ __forceinline__ void choose(const RouteArgs<T>& a, const float* z, int64_t token, int* hist, int* rank_out) {
    const int lane = threadIdx.x & 63, size = a.all / a.groups;
    float s[NE], c[NE];
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < NE; ++i) {
        const int e = lane + 64 * i;
        s[i] = e < a.all ? z[e] : -INFINITY;
        mx = fmaxf(mx, s[i]);
    }
    mx = wave_max(mx);
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < NE; ++i) {
        s[i] = expf(s[i] - mx);
        sum += s[i];
    }
    sum = wave_sum(sum);
    unsigned open = 0;
#pragma unroll
    for (int i = 0; i < NE; ++i) {
        const int e = lane + 64 * i;
        s[i] /= sum;
        c[i] = e < a.all ? s[i] + (a.correction ? a.correction[e] : 0.f) : -INFINITY;
        if (e < a.all && a.keep >= a.groups) open |= 1u << i;
    }
    // the largest of the entries whose bit in `of` is set, the first of equal ones (of numbers that do not compare: the first); -1: none
    auto best = [&](unsigned of) {
        float v = -INFINITY;
#pragma unroll
        for (int i = 0; i < NE; ++i)
            if (of >> i & 1u) v = fmaxf(v, c[i]);
        v = wave_max(v);
        int at = -1, any = -1;
#pragma unroll
        for (int i = 0; i < NE; ++i) {
            const uint64_t set = __ballot(of >> i & 1u), top = __ballot((of >> i & 1u) && c[i] == v);
            if (at < 0 && top) at = __builtin_ctzll(top) + 64 * i;
            if (any < 0 && set) any = __builtin_ctzll(set) + 64 * i;
        }
        return at < 0 ? any : at;
    };
    if (a.keep < a.groups) {               // groups in the order of their largest entry
        unsigned valid = 0;
#pragma unroll
        for (int i = 0; i < NE; ++i)
            if (lane + 64 * i < a.all) valid |= 1u << i;
        for (int k = 0; k < a.keep; ++k) {
            const int at = best(valid & ~open), grp = at < 0 ? -1 : at / size;
#pragma unroll
            for (int i = 0; i < NE; ++i)
                if (lane + 64 * i < a.all && (lane + 64 * i) / size == grp) open |= 1u << i;
        }
    }
    int id = 0;
    float w = 0.f;
    for (int k = 0; k < a.top; ++k) {
        const int at = best(open);
        float v = 0.f;
#pragma unroll
        for (int i = 0; i < NE; ++i)
            if (at == lane + 64 * i) { v = s[i]; open &= ~(1u << i); }
        v = at < 0 ? 0.f : __shfl(v, at & 63, 64);
        if (lane == k) { id = at < 0 ? a.all - 1 : at; w = v * a.scale; }
    }
    if (lane < a.top) {
        a.ids[token * a.top + lane] = id;
        a.weights[token * a.top + lane] = w;
        rank_out[lane] = id < a.experts ? atomicAdd(&hist[id], 1) : 0;
    }
}

// behind the choices of a workgroup's tokens: their ranks among all choices of their experts
template <class T>
__device__ __forceinline__ void finish_ranks(const RouteArgs<T>& a, int64_t token0, int tokens, int* hist, const int* ranks) {
    const int threads = blockDim.x;
    __syncthreads();
    for (int e = threadIdx.x; e < a.experts; e += threads) {
        const int c = hist[e];
        hist[e] = c ? atomicAdd(&a.counts[e], c) : 0;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < tokens * a.top; i += threads) {
        const int64_t at = token0 * a.top + i;
        const int id = a.ids[at];
        a.ranks[at] = id < a.experts ? hist[id] + ranks[i] : 0;
    }
}

// ET tiles of 16 experts, U tiles of 16 tokens per workgroup; wavefront w of W takes the k-steps w, w + W, ...  Few tokens: one tile
// and many wavefronts, so that the chain of requests is short; many tokens: two tiles, so that the router is read half as often.
template <int ET, int U, int W>
__global__ void __launch_bounds__(64 * W) moe_route_tile_kernel(RouteArgs<__bf16> a) {
    constexpr int kRow = 16 * ET + 1, kAhead = U + ET <= 3 ? 8 : U + ET <= 6 ? 4 : 2;
    __shared__ float z[16 * U * kRow];
    __shared__ int hist[kMaxExperts], ranks[16 * U * 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4, n = lane & 15;
    const int64_t token0 = (int64_t)blockIdx.x * (16 * U);
    for (int e = tid; e < a.experts; e += 64 * W) hist[e] = 0;
    f32x4_t acc[U][ET];
    const __bf16* hr[U];
    const __bf16* rr[ET];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int64_t t = token0 + 16 * u + n;
        hr[u] = a.h + (t < a.n ? t : a.n - 1) * a.h_stride + 8 * g;
#pragma unroll
        for (int i = 0; i < ET; ++i) acc[u][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int i = 0; i < ET; ++i) rr[i] = a.router + (int64_t)(16 * i + n < a.all ? 16 * i + n : a.all - 1) * a.width + 8 * g;
#pragma unroll kAhead
    for (int k = 32 * wave; k < a.width; k += 32 * W) {
        bf16x8_t x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) x[u] = *reinterpret_cast<const bf16x8_t*>(hr[u] + k);
#pragma unroll
        for (int i = 0; i < ET; ++i) {
            const bf16x8_t w = *reinterpret_cast<const bf16x8_t*>(rr[i] + k);
#pragma unroll
            for (int u = 0; u < U; ++u) acc[u][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, x[u], acc[u][i], 0, 0, 0);
        }
    }
    if constexpr (ET == 1 && U <= 2) {                 // every wavefront's part side by side, added by a thread per logit
        __shared__ float part[W][256 * U];
#pragma unroll
        for (int u = 0; u < U; ++u)
            *reinterpret_cast<f32x4_t*>(&part[wave][256 * u + 16 * n + 4 * g]) = acc[u][0];
        __syncthreads();
        for (int i = tid; i < 256 * U; i += 64 * W) {
            float sum = 0.f;
#pragma unroll
            for (int w = 0; w < W; ++w) sum += part[w][i];
            z[(i >> 4) * kRow + (i & 15)] = sum;
        }
        __syncthreads();
    } else {
        for (int w = 0; w < W; ++w) {
            if (wave == w)
#pragma unroll
                for (int u = 0; u < U; ++u)
#pragma unroll
                    for (int i = 0; i < ET; ++i)
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            float* p = z + (16 * u + n) * kRow + 16 * i + 4 * g + e;
                            *p = w == 0 ? acc[u][i][e] : *p + acc[u][i][e];
                        }
            __syncthreads();
        }
    }
    const int tokens = token0 + 16 * U < a.n ? 16 * U : (int)(a.n - token0);
    for (int t = wave; t < tokens; t += W) choose<(ET + 3) / 4>(a, z + t * kRow, token0 + t, hist, ranks + t * a.top);
    finish_ranks(a, token0, tokens, hist, ranks);
}

template <int ET>
void launch_route(const RouteArgs<__bf16>& a, hipStream_t st) {
    if (a.n <= 2048) hipLaunchKernelGGL((moe_route_tile_kernel<ET, 1, 16>), dim3((unsigned)((a.n + 15) / 16)), dim3(1024), 0, st, a);
    else if constexpr (ET == 1) hipLaunchKernelGGL((moe_route_tile_kernel<ET, 2, 16>), dim3((unsigned)((a.n + 31) / 32)), dim3(1024), 0, st, a);
    else hipLaunchKernelGGL((moe_route_tile_kernel<ET, 2, 4>), dim3((unsigned)((a.n + 31) / 32)), dim3(256), 0, st, a);
}

// any size: one token per wavefront, four per workgroup
template <class T>
__global__ void __launch_bounds__(kThreads) moe_route_any_kernel(RouteArgs<T> a) {
    __shared__ float z[4][kMaxExperts];
    __shared__ int hist[kMaxExperts], ranks[4 * 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t token0 = (int64_t)blockIdx.x * 4;
    const int tokens = token0 + 4 < a.n ? 4 : (int)(a.n - token0);
    for (int e = tid; e < a.experts; e += kThreads) hist[e] = 0;
    if (wave < tokens) {
        const T* h = a.h + (token0 + wave) * a.h_stride;
        for (int e = 0; e < a.all; ++e) {
            const T* r = a.router + (int64_t)e * a.width;
            float s = 0.f;
            for (int c = lane; c < a.width; c += 64) s += (float)h[c] * (float)r[c];
            s = wave_sum(s);
            if (lane == 0) z[wave][e] = s;
        }
    }
    __syncthreads();
    if (wave < tokens) choose<kMaxExperts / 64>(a, z[wave], token0 + wave, hist, ranks + wave * a.top);
    finish_ranks(a, token0, tokens, hist, ranks);
}

struct ScatterArgs {
    const int32_t* ids; const int32_t* ranks; const int32_t* counts;
    int experts, top, tile_rows, max_tiles;
    int64_t choices;
    int32_t* places;                       // [choices]
    int32_t* row_token; int32_t* row_expert;           // [place]
    int32_t* offsets;                      // [experts + 1]
    int32_t* tiles;                        // [max_tiles][2]: expert, first row inside the expert; behind the last: -1, number of tiles
};

// exclusive prefix sum over the workgroup
__device__ __forceinline__ int block_scan(int x, int* part) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int s = x;
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) {
        const int up = __shfl_up(s, m, 64);
        if (lane >= m) s += up;
    }
    if (lane == 63) part[wave] = s;
    __syncthreads();
    int before = 0;
    for (int i = 0; i < wave; ++i) before += part[i];
    return before + s - x;
}

__global__ void __launch_bounds__(kThreads) moe_scatter_kernel(ScatterArgs a) {
    __shared__ int off[kMaxExperts + 4], part[2][4];
    const int tid = threadIdx.x;
    constexpr int kPer = kMaxExperts / kThreads;
    int cnt[kPer], rows = 0, tiles = 0;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        const int e = kPer * tid + i;
        cnt[i] = e < a.experts ? a.counts[e] : 0;
        rows += cnt[i];
        tiles += (cnt[i] + a.tile_rows - 1) / a.tile_rows;
    }
    int row0 = block_scan(rows, part[0]), tile0 = block_scan(tiles, part[1]);
    const bool writer = blockIdx.x == 0;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        const int e = kPer * tid + i;
        off[e] = row0;
        if (writer && e < a.experts) {
            a.offsets[e] = row0;
            if (e + 1 == a.experts) a.offsets[e + 1] = row0 + cnt[i];
            for (int r = 0; r < cnt[i]; r += a.tile_rows, ++tile0)
                if (tile0 < a.max_tiles) { a.tiles[2 * tile0] = e; a.tiles[2 * tile0 + 1] = r; }
        }
        row0 += cnt[i];
    }
    if (writer) {
        int total = 0;
        for (int i = 0; i < 4; ++i) total += part[1][i];
        // part[1] holds every wavefront's number of tiles
        for (int t = total + tid; t < a.max_tiles; t += kThreads) a.tiles[2 * t] = -1, a.tiles[2 * t + 1] = total;
    }
    __syncthreads();
    const int64_t i = (int64_t)blockIdx.x * kThreads + tid;
    if (i >= a.choices) return;
    const int id = a.ids[i];
    if (id >= a.experts) {
        a.places[i] = -1;
        return;
    }
    const int place = off[id] + a.ranks[i];
    a.places[i] = place;
    a.row_token[place] = (int32_t)(i / a.top);
    a.row_expert[place] = id;
}

template <class T>
struct GemmArgs {
    const T* x; int64_t x_stride;
    const int32_t* row_token;              // row of x of every place, or nullptr: the place itself
    const int32_t* row_expert;
    const int32_t* offsets; const int32_t* tiles;
    const T* w; int64_t w_expert; int64_t w_stride;    // [expert][rows][k]
    int k, cols, up_row;                   // up_row > 0: columns of the result come from rows c (gate) and up_row + c (up)
    T* out; int64_t out_stride; int out_cols;          // columns from `cols` to out_cols are zero
    int32_t* zero; int num_zero;           // cleared by the launch
    int experts, max_tiles, col_blocks;
};

template <class T>
__device__ __forceinline__ void clear_counts(const GemmArgs<T>& a) {
    if (a.zero && blockIdx.x == 0)
        for (int i = threadIdx.x; i < a.num_zero; i += kThreads) a.zero[i] = 0;
}

// A workgroup: 128 rows of one expert x 128 rows of W (GATED: 64 gate rows and the same 64 up rows), k in steps of 64 through two LDS
// buffers.  Wavefront (wm, wn) has 64 rows x 64 rows of W as 4 x 4 tiles; with GATED, its first two tiles are gate and the other
// two up columns of the same place, so that the activation stays in registers.
constexpr int kBigRows = 128;
template <bool GATED>
__global__ void __launch_bounds__(kThreads, 2) moe_tile_kernel(GemmArgs<__bf16> a) {
    constexpr int kRow = 128 + 16, kMat = 128 * kRow;
    __shared__ __attribute__((aligned(16))) unsigned char lds[2][2 * kMat];
    clear_counts(a);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4, n = lane & 15;
    // Workgroups go to the eight dies round-robin: each die gets a contiguous run of (tile, columns), columns fastest within
    // groups of tiles, so that the rows and weights it reads stay in its cache.
    const unsigned total = gridDim.x, id = blockIdx.x, die = id & 7u, per_die = total >> 3, extra = total & 7u;
    const unsigned unit = die * per_die + (die < extra ? die : extra) + (id >> 3);
    const int tile = (int)(unit / a.col_blocks), cb = (int)(unit % a.col_blocks);
    const int expert = a.tiles[2 * tile];
    if (expert < 0 || expert >= a.experts) return;
    const int first = a.offsets[expert] + a.tiles[2 * tile + 1], end = a.offsets[expert + 1];
    const int rows = end - first < kBigRows ? end - first : kBigRows;
    const __bf16* w = a.w + (int64_t)expert * a.w_expert;
    const int c0 = cb * (GATED ? 64 : 128);
    // unit i of this thread: row tid / 8 + 32 i of each tile, 16 bytes at column 8 (tid % 8)
    const int kc = 8 * (tid & 7);
    const __bf16* xs[4];
    const __bf16* ws[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = (tid >> 3) + 32 * i, xr = first + (r < rows ? r : rows - 1);
        xs[i] = a.x + (int64_t)(a.row_token ? a.row_token[xr] : xr) * a.x_stride;
        int col = GATED ? c0 + 32 * (r >> 6) + (r & 31) : c0 + r;
        col = col < a.cols ? col : a.cols - 1;
        ws[i] = w + (int64_t)(GATED && (r & 32) ? a.up_row + col : col) * a.w_stride;
    }
    u32x4_t xreg[4], wreg[4];
    auto fetch = [&](int k) {
        const bool in = k + kc < a.k;
        const int at = in ? k + kc : 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            xreg[i] = *reinterpret_cast<const u32x4_t*>(xs[i] + at);
            wreg[i] = *reinterpret_cast<const u32x4_t*>(ws[i] + at);
        }
    };
    auto put = [&](unsigned char* buf, int k) {
        const bool in = k + kc < a.k;                            // k is a multiple of eight
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = (tid >> 3) + 32 * i;
            *reinterpret_cast<u32x4_t*>(buf + r * kRow + 2 * kc) = in ? xreg[i] : u32x4_t{0u, 0u, 0u, 0u};
            *reinterpret_cast<u32x4_t*>(buf + kMat + r * kRow + 2 * kc) = in ? wreg[i] : u32x4_t{0u, 0u, 0u, 0u};
        }
    };
    const int wm = wave & 1, wn = wave >> 1;
    f32x4_t acc[4][4];                                           // [tile of W][tile of rows]
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    fetch(0);
    put(lds[0], 0);
    const int steps = (a.k + 63) / 64;
    if (steps > 1) fetch(64);
    for (int s = 0; s < steps; ++s) {
        __syncthreads();
        const unsigned char* buf = lds[s & 1];
        if (s + 1 < steps) put(lds[(s + 1) & 1], 64 * (s + 1));
        if (s + 2 < steps) fetch(64 * (s + 2));
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            bf16x8_t xf[4], wf[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                xf[i] = *reinterpret_cast<const bf16x8_t*>(buf + (64 * wm + 16 * i + n) * kRow + 64 * k + 16 * g);
                wf[i] = *reinterpret_cast<const bf16x8_t*>(buf + kMat + (64 * wn + 16 * i + n) * kRow + 64 * k + 16 * g);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[i], xf[j], acc[i][j], 0, 0, 0);
        }
    }
    // lane (g, n): row n of a row tile, columns 4 g + e
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int r = 64 * wm + 16 * j + n;
        if (r >= rows) continue;
        __bf16* o = a.out + (int64_t)(first + r) * a.out_stride;
#pragma unroll
        for (int i = 0; i < (GATED ? 2 : 4); ++i) {
            const int c = c0 + (GATED ? 32 : 64) * wn + 16 * i + 4 * g;
            bf16x4_t v;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float x = acc[i][j][e];
                if constexpr (GATED) x = silu_f(x) * acc[i + 2][j][e];
                v[e] = (__bf16)(c + e < a.cols ? x : 0.f);
            }
            if (c + 4 <= a.out_cols) {
                *reinterpret_cast<bf16x4_t*>(o + c) = v;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (c + e < a.out_cols) o[c + e] = v[e];
            }
        }
    }
}

// A workgroup of four wavefronts: 256 rows of one expert x 256 rows of W (GATED: 128 gate rows and the same 128 up rows), k in steps
// of 64 (a multiple of which k is) through LDS buffers that are filled from memory without passing through registers.  Wavefront
// (wm, wn) has 128 rows x 128 rows of W as 8 x 8 tiles: one wavefront on a vector unit, with all of its registers.
//
// A step is two phases of 64 products each.  While the operands of one phase are multiplied, those of the next are read from LDS, and the
// reads and the requests are spread over the products, so that the matrix units wait for neither.  One barrier a step, between the
// phases: in front of it a wavefront has read the last of the step's buffers and its requests of the next step have landed; behind it
// the step's buffers are free for requests: rows two steps ahead go to them in the second phase, W two steps ahead went to the third of its
// buffers in the first (W comes from farther away, and requests in one phase alone are as many as a compute unit can issue in it).
//
// 8000 rows, three of 14 experts of 3072 x 4096 and two that return their row: 1015 + 560 us with eight wavefronts of 128 x 64 that read 1.5
// times as much of LDS and issued a step's requests and reads in front of its products, 870 + 490 us now (1.2 PFLOP/s; products alone, without
// reads and requests, 0.92 of it).  16000 rows 3010 -> 2690 us in all.
//
// A row of a buffer is eight units of 16 bytes, unit c at place c ^ (row % 8), so that reads of a column meet all banks.
constexpr int kBlockRows = 256, kBlockThreads = 256;
// What an earlier launch wrote and this one only reads, by the scalar path.  i: the same in all lanes
__device__ __forceinline__ int fixed_at(const int32_t* p, int64_t i) {
    return reinterpret_cast<const __attribute__((address_space(4))) int32_t*>((uintptr_t)p)[i];
}
// Tiles of an expert that are worked on side by side: a die's compute units then share that many blocks of rows and 32 / kSideTiles of W.
constexpr int kSideTiles = 8;
// Which tiles a launch has: all of them, or (MANY) those of experts with more than kSpan rows.
constexpr int kSpan = 128;
template <bool MANY>
struct BlockTiles {
    const GemmArgs<__bf16>& a;
    // Of the tiles t .. t + 64 kSets - 1, one a lane and set, those that count; all requests of a kind at once.  Behind the last tile there are no experts.
    static constexpr int kSets = 3;
    __device__ __forceinline__ void counted(int t, uint64_t (&set)[kSets]) const {
        int expert[kSets], rows[kSets];
#pragma unroll
        for (int i = 0; i < kSets; ++i) {
            const int at = t + 64 * i + (int)(threadIdx.x & 63);
            expert[i] = at < a.max_tiles ? a.tiles[2 * at] : -1;
        }
#pragma unroll
        for (int i = 0; i < kSets; ++i) rows[i] = expert[i] >= 0 && expert[i] < a.experts ? a.offsets[expert[i] + 1] - a.offsets[expert[i]] : 0;
#pragma unroll
        for (int i = 0; i < kSets; ++i) set[i] = __ballot(rows[i] > kSpan);
    }
    __device__ __forceinline__ int total() const {
        if constexpr (!MANY) {                                   // behind the last their number stands
            const int mark = fixed_at(a.tiles, 2 * (int64_t)a.max_tiles - 2), number = fixed_at(a.tiles, 2 * (int64_t)a.max_tiles - 1);
            return mark < 0 ? number : a.max_tiles;
        }
        int n = 0;
        for (int t = 0; t < a.max_tiles; t += 64 * kSets) {
            uint64_t set[kSets];
            counted(t, set);
#pragma unroll
            for (int i = 0; i < kSets; ++i) n += __popcll(set[i]);
        }
        return n;
    }
    // tile number `n` of them
    __device__ __forceinline__ int at(int n) const {
        if constexpr (!MANY) return n;
        const int lane = threadIdx.x & 63;
        for (int t = 0; t < a.max_tiles; t += 64 * kSets) {
            uint64_t set[kSets];
            counted(t, set);
#pragma unroll
            for (int i = 0; i < kSets; ++i) {
                const int here = __popcll(set[i]);
                if (n >= 0 && n < here) return t + 64 * i + __builtin_ctzll(__ballot((set[i] >> lane & 1) && __popcll(set[i] & ((1ull << lane) - 1)) == n));
                n -= here;
            }
        }
        return 0;
    }
};
// The unit of workgroup number `block`: false if there is none, otherwise its expert, rows first .. first + rows - 1 and columns c0 and on.  Workgroups go to the eight
// dies round-robin, and each die gets a contiguous run of (expert, group of tiles, columns, tile): those that run at the same time share rows and weights of one
// expert.  Units behind a die's last whole round, if they are half a round at most, are two workgroups each, of half the rows: a round of them takes
// some 0.6 of one of whole units.  Routing, both products and the sum, us, units of 256 rows / of 128 where an expert has no more left / and these:
// 14 experts of 4096 x 3072, three each, 8000 rows 1380 / 1370 / 1357, 6000 1095 / 1082 / 1054, 4000 759 / 748 / 731, 3000 648 / 626 / 623, 1500 457 / 449 / 424; of
// 2880 x 2880, 3000 rows 458 / 448 / 433; of 2048 x 1024, 6000 285 / 281 / 263.  In quarters, of half the columns, too, up to a quarter of a round: 1356, 1066, 734, 629, 418, 433, 260.
struct BlockUnit { int expert, first, rows, c0; };
constexpr unsigned kDieUnits = 32;                               // compute units of a die, of which each works on one unit
template <bool GATED, bool MANY>
__device__ __forceinline__ bool block_unit(const GemmArgs<__bf16>& a, const BlockTiles<MANY>& list, int total, unsigned columns, unsigned block, BlockUnit& u) {
    const unsigned units = (unsigned)total * columns, die = block & 7u, extra = units & 7u, of_die = units / 8 + (die < extra ? 1 : 0), last = of_die % kDieUnits;
    unsigned turn = block >> 3, part = 0;
    const bool halves = !MANY && last <= kDieUnits / 2 && turn >= of_die - last;
    if (halves) {
        part = (turn - (of_die - last)) & 1;
        turn = of_die - last + (turn - (of_die - last)) / 2;
    }
    if (turn >= of_die) return false;
    const unsigned unit = die * (units / 8) + (die < extra ? die : extra) + turn;
    const int some = (int)(unit / columns), listed = list.at(some);         // a tile of the unit's expert
    const int in_expert = fixed_at(a.tiles, 2 * (int64_t)listed + 1);
    u.expert = fixed_at(a.tiles, 2 * (int64_t)listed);
    if (u.expert < 0 || u.expert >= a.experts) return false;
    const int row0 = fixed_at(a.offsets, u.expert), end = fixed_at(a.offsets, u.expert + 1), tile0 = some - in_expert / kBlockRows;
    const unsigned tiles = (unsigned)(end - row0 + kBlockRows - 1) / kBlockRows, groups = (tiles + kSideTiles - 1) / kSideTiles;
    const unsigned side = (tiles + groups - 1) / groups, of_expert = unit - (unsigned)tile0 * columns, group = of_expert / (side * columns);
    const unsigned here = tiles - group * side < side ? tiles - group * side : side, rest = of_expert - group * side * columns;
    u.first = row0 + kBlockRows * (int)(group * side + rest % here);
    u.rows = end - u.first < kBlockRows ? end - u.first : kBlockRows;
    if (halves) {
        u.first += (int)part * (kBlockRows / 2);
        u.rows = part ? u.rows - kBlockRows / 2 : u.rows < kBlockRows / 2 ? u.rows : kBlockRows / 2;
        if (u.rows <= 0) return false;
    }
    u.c0 = (int)(rest / here) * (GATED ? 128 : 256);
    return true;
}
constexpr int kBlockLds = 5 * kBlockRows * 128;                  // bytes: three buffers of W, two of rows
template <bool GATED, int RT>
__device__ __forceinline__ void moe_block_tiles(const GemmArgs<__bf16>& a, const BlockUnit& u, unsigned char* lds) {
    constexpr int kMat = kBlockRows * 128;
    const int lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int first = u.first, rows = u.rows, c0 = u.c0;
    // load i of a wavefront fills rows 8 (8 wave + i) .. + 7 of W and 8 (RT wave + i) .. + 7 of the rows: lane l place l % 8 of row l / 8
    uint32_t x_off[RT], w_off[8];                                // bytes (checked on the host to fit)
    const uint32_t to = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds);
    const uint32_t to_w = to + 8192u * wave, to_x = to + 3 * kMat + 1024u * RT * wave;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int r = 8 * (8 * wave + i) + (lane >> 3), unit = (lane & 7) ^ (lane >> 3);
        int col = GATED ? c0 + 32 * (r >> 6) + (r & 31) : c0 + r;
        col = col < a.cols ? col : a.cols - 1;
        w_off[i] = 2u * ((uint32_t)(GATED && (r & 32) ? a.up_row + col : col) * (uint32_t)a.w_stride + 8u * unit);
    }
#pragma unroll
    for (int i = 0; i < RT; ++i) {
        const int r = 8 * (RT * wave + i) + (lane >> 3), unit = (lane & 7) ^ (lane >> 3), xr = first + (r < rows ? r : rows - 1);
        x_off[i] = 2u * ((uint32_t)(GATED ? a.row_token[xr] : xr) * (uint32_t)a.x_stride + 8u * unit);        // the second product's rows lie by expert
    }
    const __bf16* xs = a.x;
    const __bf16* ws = a.w + (int64_t)u.expert * a.w_expert;
    // Inline assembly, since the compiler would put a wait for all requests in front of every read of LDS.  Nothing else here uses M0.
    auto request = [&](uint32_t off, const __bf16* from, uint32_t at) {
        __asm__ volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" :: "v"(off), "s"(from), "s"(at) : "memory", "m0");
    };
    auto fetch_x = [&](int i, int s) { request(x_off[i], xs + 64 * s, to_x + (uint32_t)(s & 1) * kMat + 1024u * i); };
    auto fetch_w = [&](int i, int s, uint32_t buf) { request(w_off[i], ws + 64 * s, to_w + buf + 1024u * i); };
    const int wm = wave & 1, wn = wave >> 1;
    f32x4_t acc[8][RT];                                          // [tile of W][tile of rows]
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < RT; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const int steps = a.k / 64;
#pragma unroll
    for (int i = 0; i < 8; ++i) fetch_w(i, 0, 0);
#pragma unroll
    for (int i = 0; i < RT; ++i) fetch_x(i, 0);
    if (steps > 1) {
#pragma unroll
        for (int i = 0; i < 8; ++i) fetch_w(i, 1, kMat);
#pragma unroll
        for (int i = 0; i < RT; ++i) fetch_x(i, 1);
    }
    if (steps > 1) __builtin_amdgcn_s_waitcnt(RT == 8 ? 0x4F70 : 0x0F7C);        // step 0 has landed: 8 + RT requests at most are under way
    else __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();
    bf16x8_t xf[2][RT], wf[2][8];
    const unsigned char* xl = lds + 3 * kMat + 128 * 16 * RT * wm + n * 128 + 16 * (g ^ (n & 7));
    const unsigned char* wl = lds + 128 * 128 * wn + n * 128 + 16 * (g ^ (n & 7));
    const int flip = 64 - 2 * (16 * (g ^ (n & 7)) & 64);         // from the unit of the first phase to that of the second
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        wf[0][i] = *reinterpret_cast<const bf16x8_t*>(wl + 2048 * i);
        if (i < RT) xf[0][i] = *reinterpret_cast<const bf16x8_t*>(xl + 2048 * i);
    }
    // In place by assembly: all accumulation registers are taken, and the compiler, which moves results around, has none to move them through.
    // It does not know these for matrix instructions and so keeps no distance between them and others: operands come from LDS reads alone, which
    // it waits for, and nothing but products touches the accumulators between two calls of settle().  Every build is looked over for that
    // (check_products.py).
    auto product = [](f32x4_t& c, const bf16x8_t& w, const bf16x8_t& x) {
        __asm__ volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(w), "v"(x));
    };
    // 8 RT products, with `aux(i)`, i < 4 RT, behind two each
    auto phase = [&](const bf16x8_t (&w)[8], const bf16x8_t (&x)[RT], auto aux) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int j = 0; j < RT; j += 2) {
                product(acc[i][j], w[i], x[j]);
                product(acc[i][j + 1], w[i], x[j + 1]);
                aux(RT / 2 * i + j / 2);
                __builtin_amdgcn_sched_barrier(0);
            }
    };
    auto read = [&](bf16x8_t (&w)[8], bf16x8_t (&x)[RT], const unsigned char* wb, const unsigned char* xb, int i) {
        if (i < RT) x[i] = *reinterpret_cast<const bf16x8_t*>(xb + 2048 * i);
        else if (i < RT + 8) w[i - RT] = *reinterpret_cast<const bf16x8_t*>(wb + 2048 * (i - RT));
    };
    uint32_t at_w = 0, far_w = 2 * kMat;                         // buffers of W of this step and of the one after the next
    auto step = [&](int s, auto inner_tag) {
        constexpr bool kInner = decltype(inner_tag)::value;      // a step with two more behind it
        const unsigned char* xb = xl + (s & 1) * kMat;
        const unsigned char* wb = wl + at_w;
        phase(wf[0], xf[0], [&](int i) {
            if (kInner || s + 2 < steps)
                if (i % (RT / 2) == RT / 2 - 1) fetch_w(i / (RT / 2), s + 2, far_w);
            read(wf[1], xf[1], wb + flip, xb + flip, i);
        });
        far_w = at_w;
        at_w = at_w == 2 * kMat ? 0 : at_w + kMat;
        const bool more = kInner || s + 1 < steps;
        if (more) {
            if (kInner || s + 2 < steps) __builtin_amdgcn_s_waitcnt(0x0070 | 8);
            else __builtin_amdgcn_s_waitcnt(0x0070);
            __syncthreads();
        }
        xb = xl + ((s + 1) & 1) * kMat;
        wb = wl + at_w;
        phase(wf[1], xf[1], [&](int i) {
            if (kInner || s + 2 < steps)
                if (i % 4 == 3) fetch_x(i / 4, s + 2);
            if (more) read(wf[0], xf[0], wb, xb, i);
        });
    };
    auto settle = [&] {                                          // of accumulators: what is in front of this and behind it stays there
#pragma unroll
        for (int i = 0; i < 8 * RT; ++i) __asm__ volatile("" : "+a"(acc[i / RT][i % RT]));
        __asm__ volatile("s_nop 15\n\ts_nop 15");
#pragma unroll
        for (int i = 0; i < 8 * RT; ++i) __asm__ volatile("" : "+a"(acc[i / RT][i % RT]));
    };
    settle();
    int s = 0;
    for (; s + 2 < steps; ++s) step(s, std::true_type{});
    for (; s < steps; ++s) step(s, std::false_type{});
    settle();
    // Lane (g, n) has row n of a row tile, columns 4 g + e: 8 bytes of every 32 of a row.  They go through LDS, a wavefront's rows to a part of its own, so that
    // rows are written in one piece.  With the unit's place read by the scalar path (block_unit), us, before / now: 14 experts of 4096 x 3072, 8000 rows 1370 / 1346, 5000
    // 913 / 899, 1500 448 / 446; of 2880 x 2880, 3000 rows 442 / 435 (without the scalar path 1351, 901, 448, 435).
    constexpr int kCols = GATED ? 64 : 128, kPitch = 2 * kCols + 16, kRowLanes = kCols / 8;
    static_assert(4 * 128 * kPitch <= kBlockLds, "room in LDS");
    __syncthreads();                                             // everybody has read the last step's operands
    unsigned char* own = lds + wave * 16 * RT * kPitch;
#pragma unroll
    for (int j = 0; j < RT; ++j)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if (GATED && (i & 2)) continue;
            const int at = (GATED ? 32 * (i >> 2) + 16 * (i & 1) : 16 * i) + 4 * g, c = c0 + kCols * wn + at;
            bf16x4_t v;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float x = acc[i][j][e];
                if constexpr (GATED) x = silu_f(x) * acc[(i + 2) & 7][j][e];
                v[e] = (__bf16)(c + e < a.cols ? x : 0.f);
            }
            *reinterpret_cast<bf16x4_t*>(own + (16 * j + n) * kPitch + 2 * at) = v;
        }
    const int c = c0 + kCols * wn + 8 * (lane % kRowLanes);
#pragma unroll
    for (int i = 0; i < 16 * RT * kRowLanes / 64; ++i) {
        const int in = 64 / kRowLanes * i + lane / kRowLanes, r = 16 * RT * wm + in;
        const bf16x8_t v = *reinterpret_cast<const bf16x8_t*>(own + in * kPitch + 16 * (lane % kRowLanes));
        if (r < rows && c < a.out_cols) *reinterpret_cast<bf16x8_t*>(a.out + (int64_t)(first + r) * a.out_stride + c) = v;       // out_cols is a multiple of eight
    }
}

// Whole units, and those of at most half the rows: a step's requests of W are the same, its products half as many
template <bool GATED>
__device__ __forceinline__ void moe_block_product(const GemmArgs<__bf16>& a, const BlockUnit& u, unsigned char* lds) {
    if (u.rows > kBlockRows / 2) moe_block_tiles<GATED, 8>(a, u, lds);
    else moe_block_tiles<GATED, 4>(a, u, lds);
}

template <bool GATED>
__global__ void __launch_bounds__(kBlockThreads) __attribute__((amdgpu_waves_per_eu(1, 1))) moe_block_kernel(GemmArgs<__bf16> a) {
    __shared__ __attribute__((aligned(1024))) unsigned char lds[kBlockLds];
    clear_counts(a);
    const BlockTiles<false> list{a};
    BlockUnit u;
    if (block_unit<GATED>(a, list, list.total(), (unsigned)a.col_blocks, blockIdx.x, u)) moe_block_product<GATED>(a, u, lds);
}

// A workgroup: up to 32 rows of one expert x some rows of W (a tile: 16, GATED: 8 gate and 8 up), which stream past them; the second half of the rows
// costs only where there are that many.  64 rows, three of 16 experts of 3072 x 4096: 258 us with 32 rows of W past 16 rows through
// operand registers, 181 us with one tile and wavefronts that split k (5.9 TB/s of weights).  Two tiles and wavefronts that share the steps of k read the
// rows half as often, and every step is on its way for all of the workgroup: experts of a step of 64 rows (14 of 4096 x 3072, three each) 205 / 188 us, 100
// rows 242 / 205, 130 rows 277 / 234; 14 of 1024 x 768, 16 rows the second product 6.9 / 5.8, 120 rows 9.1 / 6.6.  Four to eight tiles leave compute units
// waiting at the end (64 rows 195 to 198), and so do two where few experts have rows: one token 62.8 / 67.1, 2 91.6 / 93.3, 9 160.3 / 160.5.
constexpr int kSmallRows = 32, kRowWaves = 4, kSharedTiles = 2;
constexpr int kRowRing = 3 * stream_stage_bytes(1, 1);           // of a wavefront: three steps with 16 rows, two with 32
static_assert(2 * stream_stage_bytes(1, 2) <= kRowRing, "both rings fit");

// Start of row 8 i + stream_row() of the rows of W that lie at column c0 and on
template <bool GATED>
__device__ __forceinline__ const __bf16* moe_weight_row(const GemmArgs<__bf16>& a, int expert, int c0, int i) {
    int col = c0 + stream_row() + 8 * (GATED ? i / 2 : i);
    col = col < a.cols ? col : a.cols - 1;
    return a.w + (int64_t)expert * a.w_expert + (int64_t)(GATED && (i & 1) ? a.up_row + col : col) * a.w_stride;
}
// Of the rows that are multiplied
__device__ __forceinline__ const __bf16* moe_input_row(const GemmArgs<__bf16>& a, int first, int rows, int i) {
    const int r = stream_row() + 8 * i, xr = first + (r < rows ? r : rows - 1);
    return a.x + (int64_t)(a.row_token ? a.row_token[xr] : xr) * a.x_stride;
}
// Four sums of row r at column c + 4 g
template <bool GATED>
__device__ __forceinline__ void moe_finish(const GemmArgs<__bf16>& a, int first, int rows, int r, int c, f32x4_t sum) {
    const int g = (threadIdx.x & 63) >> 4;
    if constexpr (GATED) {                             // lanes g = 0, 1 hold gates 4 g + e, lanes g + 2 the up columns of the same place
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float up = __shfl_xor(sum[e], 32, 64);
            sum[e] = silu_f(sum[e]) * up;
        }
        if (g >= 2) return;
    }
    if (r >= rows) return;
    c += 4 * g;
    bf16x4_t v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = (__bf16)(c + e < a.cols ? sum[e] : 0.f);
    if (c + 4 <= a.out_cols) *reinterpret_cast<bf16x4_t*>(a.out + (int64_t)(first + r) * a.out_stride + c) = v;       // out_cols is a multiple of eight
}
template <bool GATED, int MT>
__device__ __forceinline__ void moe_row_product(const GemmArgs<__bf16>& a, int expert, int first, int rows, int c0, unsigned char* lds) {
    const int n = threadIdx.x & 15, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const __bf16* w[2];
    const __bf16* x[2 * MT];
#pragma unroll
    for (int i = 0; i < 2; ++i) w[i] = moe_weight_row<GATED>(a, expert, c0, i);
#pragma unroll
    for (int i = 0; i < 2 * MT; ++i) x[i] = moe_input_row(a, first, rows, i);
    f32x4_t acc[1][MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[0][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    stream_product<1, MT, kRowWaves, MT == 1 ? 3 : 2, false>(w, x, a.k, 0, wave, lds + wave * kRowRing, acc);
    stream_reduce<1, MT, kRowWaves>(acc, wave, lds, [&](int, int t, f32x4_t sum) { moe_finish<GATED>(a, first, rows, 16 * t + n, c0, sum); });
}
// The same, RT tiles of W and up to 16 MT rows, steps shared; k: a multiple of 64
template <bool GATED, int RT, int MT>
__device__ __forceinline__ void moe_shared_product(const GemmArgs<__bf16>& a, int expert, int first, int rows, int c0, unsigned char* lds) {
    const int n = threadIdx.x & 15;
    shared_product<RT, MT>(a.k, (int)blockIdx.x >> 3, lds, [&](int i) { return moe_weight_row<GATED>(a, expert, c0, i); },
                           [&](int i) { return moe_input_row(a, first, rows, i); },
                           [&](int r, int t, f32x4_t sum) { moe_finish<GATED>(a, first, rows, 16 * t + n, c0 + (GATED ? 8 : 16) * r, sum); });
}
template <bool GATED, bool SHARED>
__global__ void __launch_bounds__(64 * kRowWaves) moe_row_kernel(GemmArgs<__bf16> a) {
    constexpr int kShared1 = SharedStream<kSharedTiles, 1>::kRing, kShared2 = SharedStream<kSharedTiles, 2>::kRing;
    __shared__ __attribute__((aligned(1024))) unsigned char lds[!SHARED ? kRowWaves * kRowRing : kShared1 > kShared2 ? kShared1 : kShared2];
    clear_counts(a);
    const int tile = blockIdx.x / a.col_blocks, cb = blockIdx.x % a.col_blocks;
    const int expert = a.tiles[2 * tile];
    if (expert < 0 || expert >= a.experts) return;
    const int first = a.offsets[expert] + a.tiles[2 * tile + 1], end = a.offsets[expert + 1];
    const int rows = end - first < kSmallRows ? end - first : kSmallRows, c0 = cb * (GATED ? 8 : 16) * (SHARED ? kSharedTiles : 1);
    if constexpr (SHARED) {
        if (rows <= 16) moe_shared_product<GATED, kSharedTiles, 1>(a, expert, first, rows, c0, lds);
        else moe_shared_product<GATED, kSharedTiles, 2>(a, expert, first, rows, c0, lds);
    } else {
        if (rows <= 16) moe_row_product<GATED, 1>(a, expert, first, rows, c0, lds);
        else moe_row_product<GATED, 2>(a, expert, first, rows, c0, lds);
    }
}

// A workgroup: four or eight tiles of W past up to kSpan rows of one expert at a time, which the four wavefronts share (SharedStream), for as many rows as a
// decode batch or a few short prompts bring.  The weights bound such a product, each of which should pass once: tiles of 32 rows read them again for every 32
// rows, and blocks and tiles of 128 and 256 rows compute what there is not.  A workgroup has what begins with its tile and ends before the next multiple of kSpan
// rows, or of a tile if that has more; the tiles in between have nothing to do.
//
// A step's experts, us, before / this: 14 of 4096 x 3072, three choices, 100 rows 199 / 192, 130 242 / 197, 160 278 / 201, 300 284 / 227, 500 305 / 247; 14 of
// 1024 x 3072, 200 rows 106 / 72; 128 of 2048 x 768, eight choices, 400 rows 305 / 246; 8 of 4096 x 14336, two, 104 rows 667 / 445, 400 703 / 566; 8 of
// 2048 x 8192, 200 rows 276 / 173.  Fewer or more choices per expert: 14 of 4096 x 3072, 64 rows (14 each) 184 / 189, 700 (150) 306 / 438, since most of them
// then have more than 128.
template <bool GATED, int RT>
__device__ __forceinline__ void moe_span_rows(const GemmArgs<__bf16>& a, int expert, int first, int rows, int cb, unsigned char* lds) {
    const int c0 = cb * (GATED ? 8 : 16) * RT;
    if (rows <= 32) moe_shared_product<GATED, RT, 2>(a, expert, first, rows, c0, lds);
    else if (rows <= 64) moe_shared_product<GATED, RT, 4>(a, expert, first, rows, c0, lds);
    else moe_shared_product<GATED, RT, 8>(a, expert, first, rows, c0, lds);
}
template <int RT>
constexpr int span_lds() {
    constexpr int k2 = SharedStream<RT, 2>::kRing, k4 = SharedStream<RT, 4>::kRing, k8 = SharedStream<RT, 8>::kRing, k24 = k2 > k4 ? k2 : k4;
    return k24 > k8 ? k24 : k8;
}
template <bool GATED, int RT>
__global__ void __launch_bounds__(64 * kRowWaves) moe_span_kernel(GemmArgs<__bf16> a, int tile_rows) {
    __shared__ __attribute__((aligned(1024))) unsigned char lds[span_lds<RT>()];
    clear_counts(a);
    const int tile = blockIdx.x / a.col_blocks, cb = blockIdx.x % a.col_blocks;
    const int expert = a.tiles[2 * tile], row0 = a.tiles[2 * tile + 1], span = tile_rows > kSpan ? tile_rows : kSpan;
    if (expert < 0 || expert >= a.experts || row0 % span) return;
    const int first = a.offsets[expert] + row0, end = a.offsets[expert + 1], rows = end - first < span ? end - first : span;
    for (int at = 0; at < rows; at += kSpan) {
        if (at > 0) __syncthreads();                   // everybody has read what lies in LDS
        moe_span_rows<GATED, RT>(a, expert, first + at, rows - at < kSpan ? rows - at : kSpan, cb, lds);
    }
}
// The same with tiles of 256 rows, but experts with more than kSpan rows go in blocks, which come first.  How many there are is known here alone: the host deals
// out workgroups for all that there can be, and those behind the last have nothing to do.  All experts in blocks / all in spans / this, us: 14 of 4096 x 3072, 500
// rows, at most 128 of an expert 303 / 251 / 252, 236 302 / 322 / 249, 402 301 / 333 / 263, all at three 161 / 274 / 162; 8 of 4096 x 14336, 400 rows, 120 705 / 588 /
// 585, 155 704 / 757 / 684, all at two 437 / 690 / 442; 128 of 2048 x 768, 1200 rows, 101 339 / 312 / 317, 356 377 / 363 / 328, all at half of them 231 / 294 / 240.
// (As two launches, each of which ends by itself: 255, 352, 337, 168 for the first four.)
template <bool GATED>
__global__ void __launch_bounds__(kBlockThreads) __attribute__((amdgpu_waves_per_eu(1, 1))) moe_uneven_kernel(GemmArgs<__bf16> a, unsigned block_columns) {
    constexpr int RT = 8, kSpanLds = span_lds<RT>();
    static_assert(kBlockThreads == 64 * kRowWaves, "both have four wavefronts");
    __shared__ __attribute__((aligned(1024))) unsigned char lds[kBlockLds > kSpanLds ? kBlockLds : kSpanLds];
    clear_counts(a);
    const BlockTiles<true> list{a};
    const int total = list.total();
    const unsigned blocks = ((unsigned)total * block_columns + 7) / 8 * 8;
    if (blockIdx.x < blocks) {
        BlockUnit u;
        if (block_unit<GATED>(a, list, total, block_columns, blockIdx.x, u)) moe_block_product<GATED>(a, u, lds);
        return;
    }
    const unsigned at = blockIdx.x - blocks, tile = at / (unsigned)a.col_blocks;
    const int expert = tile < (unsigned)a.max_tiles ? a.tiles[2 * tile] : -1;
    if (expert < 0 || expert >= a.experts) return;
    const int first = a.offsets[expert], rows = a.offsets[expert + 1] - first;
    if (rows <= kSpan) moe_span_rows<GATED, RT>(a, expert, first, rows, (int)(at % (unsigned)a.col_blocks), lds);       // its only tile
}

// one wavefront per (place, four columns)
template <class T, bool GATED>
__global__ void __launch_bounds__(kThreads) moe_any_kernel(GemmArgs<T> a) {
    clear_counts(a);
    const int lane = threadIdx.x & 63;
    const int64_t place = blockIdx.x / a.col_blocks;
    if (place >= a.offsets[a.experts]) return;
    const int expert = a.row_expert[place];
    const T* x = a.x + (int64_t)(a.row_token ? a.row_token[place] : place) * a.x_stride;
    const T* w = a.w + (int64_t)expert * a.w_expert;
    for (int i = 0; i < 4; ++i) {
        const int c = (blockIdx.x % a.col_blocks) * 16 + (threadIdx.x >> 6) * 4 + i;
        if (c >= a.out_cols) break;
        float s = 0.f, u = 0.f;
        if (c < a.cols)
            for (int k = lane; k < a.k; k += 64) {
                s += (float)x[k] * (float)w[(int64_t)c * a.w_stride + k];
                if (GATED) u += (float)x[k] * (float)w[(int64_t)(a.up_row + c) * a.w_stride + k];
            }
        s = wave_sum(s);
        if (GATED) s = silu_f(s) * wave_sum(u);
        if (lane == 0) a.out[place * a.out_stride + c] = (T)s;
    }
}

bool size_in(int64_t v, int64_t lo, int64_t hi) { return v >= lo && v <= hi; }

template <class T>
int gemm(GemmArgs<T>& a, bool gated, int tile_rows, int64_t tokens, int64_t choices, int64_t max_places, hipStream_t st) {
    const dim3 block(kThreads);
    int64_t grid;
    if constexpr (sizeof(T) == 2) {
        const int64_t block_columns = (a.out_cols + (gated ? 127 : 255)) / (gated ? 128 : 256);
        if (tile_rows >= kSmallRows && a.k % kStreamK == 0 && choices >= 18 * a.experts && choices <= 112 * a.experts) {
            // eight tiles of W, unless four have the compute units through earlier: a tile takes about three times what the rows beside it do (8 experts of
            // 1536 x 4096, 100 rows 79 / 68 us; 14 of 4096 x 3072, 130 rows 197 / 205)
            auto takes = [&](int64_t t) {
                const int64_t groups = a.experts * ((a.out_cols * (gated ? 2 : 1) + 16 * t - 1) / (16 * t));
                return (groups + 255) / 256 * (3 * t + 4);
            };
            const int tiles = takes(4) < takes(8) ? 4 : 8, per = (gated ? 8 : 16) * tiles;
            a.col_blocks = (a.out_cols + per - 1) / per;
            grid = (int64_t)a.max_tiles * a.col_blocks;
            // An expert with more rows than kSpan reads its weights again for every kSpan of them, and what it computes is bound by LDS.  Where blocks would serve if
            // all had that many, they serve those that have, next to the others.  With four tiles of W two workgroups share a compute unit, which one with a
            // block's LDS would not: 8 of 1536 x 4096, 300 rows, at most 151 of an expert 131 us with blocks for both products, 109 with blocks for the first alone.
            const bool uneven = tile_rows == kBlockRows && tokens > kSpan && tiles == 8;
            if (uneven) {
                const int64_t large = choices / (kSpan + 1) < a.experts ? choices / (kSpan + 1) : a.experts;     // so many have more than kSpan at most
                grid += ((choices / kBlockRows + large) * block_columns + 7) / 8 * 8;
            }
            if (grid > 0x7fffffff) return INFER_KV_EINVAL;
            if (uneven && gated) hipLaunchKernelGGL((moe_uneven_kernel<true>), dim3((unsigned)grid), block, 0, st, a, (unsigned)block_columns);
            else if (uneven) hipLaunchKernelGGL((moe_uneven_kernel<false>), dim3((unsigned)grid), block, 0, st, a, (unsigned)block_columns);
            else if (gated && tiles == 8) hipLaunchKernelGGL((moe_span_kernel<true, 8>), dim3((unsigned)grid), block, 0, st, a, tile_rows);
            else if (gated) hipLaunchKernelGGL((moe_span_kernel<true, 4>), dim3((unsigned)grid), block, 0, st, a, tile_rows);
            else if (tiles == 8) hipLaunchKernelGGL((moe_span_kernel<false, 8>), dim3((unsigned)grid), block, 0, st, a, tile_rows);
            else hipLaunchKernelGGL((moe_span_kernel<false, 4>), dim3((unsigned)grid), block, 0, st, a, tile_rows);
            return (int)hipGetLastError();
        }
        if (tile_rows == kBlockRows) {
            a.col_blocks = (int)block_columns;
            grid = (a.max_tiles * block_columns + 7) / 8 * 8 + 8 * (kDieUnits / 2);
            if (grid > 0x7fffffff) return INFER_KV_EINVAL;
            if (gated) hipLaunchKernelGGL((moe_block_kernel<true>), dim3((unsigned)grid), dim3(kBlockThreads), 0, st, a);
            else hipLaunchKernelGGL((moe_block_kernel<false>), dim3((unsigned)grid), dim3(kBlockThreads), 0, st, a);
            return (int)hipGetLastError();
        }
        if (tile_rows == kBigRows || tile_rows == kSmallRows) {
            const bool shared = tile_rows == kSmallRows && a.k % kStreamK == 0 && choices >= 2 * a.experts;
            const int per = tile_rows == kBigRows ? (gated ? 64 : 128) : (gated ? 8 : 16) * (shared ? kSharedTiles : 1);
            a.col_blocks = (a.out_cols + per - 1) / per;
            grid = (int64_t)a.max_tiles * a.col_blocks;
            if (grid > 0x7fffffff) return INFER_KV_EINVAL;
            if (tile_rows == kBigRows) {
                if (gated) hipLaunchKernelGGL((moe_tile_kernel<true>), dim3((unsigned)grid), block, 0, st, a);
                else hipLaunchKernelGGL((moe_tile_kernel<false>), dim3((unsigned)grid), block, 0, st, a);
            } else if (shared) {
                if (gated) hipLaunchKernelGGL((moe_row_kernel<true, true>), dim3((unsigned)grid), block, 0, st, a);
                else hipLaunchKernelGGL((moe_row_kernel<false, true>), dim3((unsigned)grid), block, 0, st, a);
            } else {
                if (gated) hipLaunchKernelGGL((moe_row_kernel<true, false>), dim3((unsigned)grid), block, 0, st, a);
                else hipLaunchKernelGGL((moe_row_kernel<false, false>), dim3((unsigned)grid), block, 0, st, a);
            }
            return (int)hipGetLastError();
        }
    }
    a.col_blocks = (a.out_cols + 15) / 16;
    grid = max_places * a.col_blocks;
    if (grid > 0x7fffffff) return INFER_KV_EINVAL;
    if (gated) hipLaunchKernelGGL((moe_any_kernel<T, true>), dim3((unsigned)grid), block, 0, st, a);
    else hipLaunchKernelGGL((moe_any_kernel<T, false>), dim3((unsigned)grid), block, 0, st, a);
    return (int)hipGetLastError();
}

// rows per tile: 0 where only the any-size kernels serve
int rows_per_tile(int elem, int64_t n, int64_t width, int64_t ff_pad, int64_t experts, int64_t top) {
    if (elem != INFER_ELEM_BF16 || width % 8 || ff_pad % 8) return 0;
    // The tiles that moe_row_kernel, moe_tile_kernel and moe_block_kernel work on; the figures are of these.  With 18 to 112 choices per expert and k in whole steps
    // moe_span_kernel takes what begins with every 128 rows, whatever the tiles, but for experts with more where tiles are blocks.
    // An expert with more than one tile of 32 rows reads its weights again, and around 32 choices per expert half of them have more.  That costs
    // little where the weights are few, more where there are many of them or many experts; us, tiles of 32 rows / the others: 8 experts of
    // 1536 x 4096, 32 choices each 105 / 136; 8 of 2048 x 8192, 28 234 / 275; 14 of 4096 x 3072, 25 261 / 282, 32 330 / 280; 8 of 4096 x 14336, 26
    // 685 / 642; 32 of 2880 x 2880, 25 405 / 380, 32 507 / 375; 128 of 2048 x 768, 26 351 / 305, 32 419 / 312.
    const double weights = 6.0 * experts * width * ff_pad;       // bytes
    if (n * top <= (weights <= 3.2e8 ? 32 : experts <= 16 && weights <= 2e9 ? 28 : 24) * experts) return kSmallRows;
    // Large blocks pay where they are enough to fill most of the chip (of 14 experts, tiles of 128 rows / blocks, us: 3072 x 4096, 200 rows
    // 319 / 295, 800 471 / 322, 2100 879 / 510; 768 x 1024, 600 rows 57 / 66, 1200 67 / 71, 2300 104 / 81).  More than a round of them, of few rows
    // and a short k, does not: with 33 choices each 14 experts of 1024 x 3072 109 / 133, 24 of 2048 x 3072 233 / 257, 8 of 2048 x 8192 274 / 293.
    // Their offsets are 32 bits.
    const int64_t far = 1ll << 31;
    const bool fits = width % 64 == 0 && ff_pad % 64 == 0 && n * width < far && n * top * ff_pad < far && 2 * ff_pad * width < far;
    const int64_t columns = (ff_pad + 127) / 128, blocks = (n * top / kBlockRows + experts / 2) * columns, work = n * top * width;   // first product, about
    const bool worth = width >= 2880 || experts * columns <= 256 || work >= 150000 * experts || work >= 2200000;
    return fits && (n * top >= 512 * experts || (blocks >= 160 && worth)) ? kBlockRows : kBigRows;
}

}  // namespace

// places (rows of the two products) and tiles of a step of n tokens, and the rows per tile: out[3]
extern "C" int infer_moe_layout(int elem, int64_t n, int64_t width, int64_t ff_pad, int64_t experts, int64_t top, int64_t* out) {
    if (n < 0 || width < 1 || experts < 1 || top < 1 || !out) return INFER_KV_EINVAL;
    const int per = rows_per_tile(elem, n, width, ff_pad, experts, top);
    out[0] = n * top;
    out[1] = per ? n * top / per + (experts < n * top ? experts : n * top) : 1;
    out[2] = per;
    return INFER_KV_OK;
}

extern "C" int infer_moe(int elem, const void* h, int64_t h_stride, const void* router, const float* correction, int64_t n, int64_t width,
                         int64_t experts, int64_t identity, int64_t top, int64_t groups, int64_t keep, float scale, const void* gate_up,
                         const void* down, int64_t ff, int64_t ff_pad, int32_t* counts, int32_t* ids, float* weights, int32_t* ranks,
                         int32_t* places, int32_t* row_token, int32_t* row_expert, int32_t* offsets, int32_t* tiles, int64_t max_tiles,
                         void* act, void* out, int64_t max_places, void* stream) {
    const int64_t all = experts + identity;
    if (!size_in(n, 0, 1 << 26) || !size_in(width, 1, 1 << 20) || !size_in(experts, 1, kMaxExperts) || identity < 0 || all > kMaxExperts ||
        !size_in(top, 1, 64) || top > all || !size_in(groups, 1, all) || all % groups || !size_in(keep, 1, groups) ||
        keep * (all / groups) < top || !size_in(ff, 1, 1 << 20) || ff_pad < ff || h_stride < width)
        return INFER_KV_EINVAL;
    if (n == 0) return INFER_KV_OK;
    int64_t layout[3];
    infer_moe_layout(elem, n, width, ff_pad, experts, top, layout);
    if (!h || !router || !gate_up || !down || !counts || !ids || !weights || !ranks || !places || !row_token || !row_expert || !offsets ||
        !tiles || !act || !out || max_places < layout[0] || max_tiles < layout[1] || n * top > 0x7fffffff)
        return INFER_KV_EINVAL;
    hipStream_t st = (hipStream_t)stream;
    auto go = [&](auto zero) -> int {
        using T = decltype(zero);
        const RouteArgs<T> r{(const T*)h, h_stride, (const T*)router, correction, (int)width, (int)all, (int)experts, (int)top, (int)groups,
                             (int)keep, scale, ids, weights, ranks, counts, (int)n};
        const bool aligned = width % 8 == 0 && h_stride % 8 == 0 && ptr_aligned(h, 16) && ptr_aligned(gate_up, 16) && ptr_aligned(down, 16) &&
                             ptr_aligned(act, 16) && ptr_aligned(out, 16);
        bool routed = false;
        if constexpr (sizeof(T) == 2) {
            if (aligned && width % 32 == 0 && all <= 256 && ptr_aligned(router, 16)) {
                if (all <= 16) launch_route<1>(r, st);
                else if (all <= 64) launch_route<4>(r, st);
                else if (all <= 128) launch_route<8>(r, st);
                else launch_route<16>(r, st);
                routed = true;
            }
        }
        if (!routed) hipLaunchKernelGGL((moe_route_any_kernel<T>), dim3((unsigned)((n + 3) / 4)), dim3(kThreads), 0, st, r);
        const int tile_rows = aligned ? (int)layout[2] : 0;
        if (tile_rows == kBlockRows && n * h_stride >= (1ll << 31)) return INFER_KV_EUNSUPPORTED;
        const int64_t choices = n * top;
        const ScatterArgs s{ids, ranks, counts, (int)experts, (int)top, tile_rows ? tile_rows : kBigRows, (int)max_tiles, choices, places, row_token,
                            row_expert, offsets, tiles};
        hipLaunchKernelGGL(moe_scatter_kernel, dim3((unsigned)((choices + kThreads - 1) / kThreads)), dim3(kThreads), 0, st, s);
        GemmArgs<T> up{(const T*)h, h_stride, row_token, row_expert, offsets, tiles, (const T*)gate_up, 2 * ff * width, width, (int)width, (int)ff,
                       (int)ff, (T*)act, ff_pad, (int)ff_pad, counts, (int)experts, (int)experts, (int)max_tiles, 0};
        int rc = gemm(up, true, tile_rows, n, choices, max_places, st);
        if (rc) return rc;
        GemmArgs<T> dn{(const T*)act, ff_pad, nullptr, row_expert, offsets, tiles, (const T*)down, width * ff_pad, ff_pad, (int)ff_pad, (int)width,
                       0, (T*)out, width, (int)width, nullptr, 0, (int)experts, (int)max_tiles, 0};
        return gemm(dn, false, tile_rows, n, choices, max_places, st);
    };
    if (elem == INFER_ELEM_BF16) return go(__bf16(0.f));
    if (elem == INFER_ELEM_F32) return go(0.f);
    return INFER_KV_EUNSUPPORTED;
}
