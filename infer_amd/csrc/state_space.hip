// Selective state space (Mamba-2: Dao and Gu, "Transformers are SSMs: Generalized Models and Efficient Algorithms Through
// Structured State Space Duality"), for gfx950 (MI355X).  Per head, over a float32 state S[state][vdim]:
//     S <- e^{a dt} S + dt B x^T ;   y = S^T C + D x ,   dt = softplus(. + bias), a = -e^{A_log}
// with x, B and C behind a causal convolution per channel and silu; groups of heads share B and C.  Behind it
// rms(y silu(z)) over equal parts of a token's channels.
//
//   ssm_step_kernel      one token per sequence (decode): convolution, step sizes and recurrence, one workgroup per
//                        (sequence, head), the state passes through registers once
//   ssm_conv_kernel      convolution and silu of prompt portions
//   ssm_chunk_kernel     prompt portions in chunks of 32 tokens on bf16 matrix instructions
//   ssm_join_kernel      carries the state over the segments that a long portion is cut into
//   ssm_scan_any_kernel  prompt portions of any size and element type, token by token
//   ssm_norm_kernel      gate and norm of all rows; keeps the last inputs of the convolution
//
// The convolution's inputs live in a ring of `taps` entries per slot (position mod taps), one more than it looks back, so a
// decode launch may write its entry while others read.  A sequence at position 0 starts from zeros whatever its slot holds.
//
// Chunk form.  With S the state before a chunk of n tokens and G the running sum of a dt,
//     y_i = e^{G_i} S^T C_i + sum_{j<=i} e^{G_i-G_j} dt_j (C_i B_j) x_j + D x_i ,   S' = e^{G_n} S + sum_j B_j (e^{G_n-G_j} dt_j x_j)^T .
// No exponent is positive.  x, B and C are bf16 already; the weighted x enters the state as three bf16 pieces (exact to
// float precision), the products of the output, which is rounded to bf16 next, take two (2^-17).
#include "elem.h"
#include "pieces.h"
#include "segments.h"

#include <type_traits>

namespace {

typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef short i16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) i16x4 lds_i16x4;
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

constexpr int kThreads = 256;
constexpr int kC = 32;          // tokens per chunk
constexpr int kSlab = 64;       // state columns per workgroup of the chunk kernel
constexpr int kTaps = 4;        // of the convolution inside the chunk kernel

struct Span { int32_t row0, count, slot, pos0; };       // consecutive tokens of one sequence

template <class T>
struct SsmArgs {
    const T* proj; int64_t proj_stride; int z_off, x_off, dt_off;   // [z: heads x vdim | x | B: groups x state | C | dt: heads]
    int heads, vdim, state_n, groups, channels, taps;
    const float* conv; const float* conv_bias;                      // [channels][taps] (last: the current token), [channels]
    const float* dt_bias; const float* a_log; const float* d;       // [heads]
    T* ring; float* state; int num_slots;                           // [slots][taps][channels], [slots][heads][state][vdim]
    T* y; int64_t y_stride;                                         // [row][heads * vdim]
    const T* xbc; int64_t xbc_stride; int64_t xbc_row0;             // rows from xbc_row0 on, behind convolution and silu
};

template <class T>
__device__ __forceinline__ float step_size(const SsmArgs<T>& a, int64_t row, int h) {
    return softplus_f((float)a.proj[row * a.proj_stride + a.dt_off + h] + a.dt_bias[h]);
}

// ------------------------------------------------------------------ decode
template <class T, int VEC>
__global__ void __launch_bounds__(kThreads) ssm_step_kernel(SsmArgs<T> a, const int32_t* slots, const int64_t* positions) {
    extern __shared__ float lds[];
    const int h = blockIdx.x, tid = threadIdx.x;
    const int64_t row = blockIdx.y;
    const int slot = slots[row];
    const int64_t pos = positions[row];
    const int n = a.state_n, inner = a.heads * a.vdim, per = a.heads / a.groups, grp = h / per;
    if (slot < 0 || slot >= a.num_slots) {               // padding
        for (int i = tid; i < a.vdim; i += kThreads) a.y[row * a.y_stride + h * a.vdim + i] = (T)0.f;
        return;
    }
    float* xs = lds;                                     // [vdim], then B and C [state] each, then the sums [rows][vdim]
    float* bs = xs + (a.vdim + 3) / 4 * 4;
    float* sums = bs + 2 * ((n + 3) / 4 * 4);
    float* cs = bs + (n + 3) / 4 * 4;
    const T* in = a.proj + row * a.proj_stride + a.x_off;
    T* ring = a.ring + (int64_t)slot * a.taps * a.channels;
    const int now = (int)(pos % a.taps);
    for (int i = tid; i < a.vdim + 2 * n; i += kThreads) {
        const int c = i < a.vdim ? h * a.vdim + i : i < a.vdim + n ? inner + grp * n + (i - a.vdim)
                                                                   : inner + (a.groups + grp) * n + (i - a.vdim - n);
        const T cur = in[c];
        float v = a.conv_bias[c] + (float)cur * a.conv[(int64_t)c * a.taps + a.taps - 1];
        int at = now;
        for (int k = 1; k < a.taps; ++k) {
            at = at == 0 ? a.taps - 1 : at - 1;
            if (pos >= k) v += (float)ring[(int64_t)at * a.channels + c] * a.conv[(int64_t)c * a.taps + a.taps - 1 - k];
        }
        if (i < a.vdim || h % per == 0) ring[(int64_t)now * a.channels + c] = cur;
        v = silu_f(v);
        if (i < a.vdim) xs[i] = v;
        else if (i < a.vdim + n) bs[i - a.vdim] = v;
        else cs[i - a.vdim - n] = v;
    }
    const float dt = step_size(a, row, h), decay = expf(-expf(a.a_log[h]) * dt);
    __syncthreads();
    const int quads = a.vdim / VEC, rows = kThreads / quads;
    const int q = tid % quads, r = tid / quads;
    float y[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) y[e] = 0.f;
    if (r < rows) {
        float* st = a.state + ((int64_t)slot * a.heads + h) * n * a.vdim + VEC * q;
        float dx[VEC];
#pragma unroll
        for (int e = 0; e < VEC; ++e) dx[e] = dt * xs[VEC * q + e];
        constexpr int kBatch = 8;
        for (int i0 = r; i0 < n; i0 += kBatch * rows) {
            float s[kBatch][VEC];
#pragma unroll
            for (int b = 0; b < kBatch; ++b) {
                const int i = i0 + b * rows;
#pragma unroll
                for (int e = 0; e < VEC; ++e) s[b][e] = 0.f;
                if (i < n && pos > 0) load_elems<VEC>(st + (int64_t)i * a.vdim, s[b]);
            }
#pragma unroll
            for (int b = 0; b < kBatch; ++b) {
                const int i = i0 + b * rows;
                if (i >= n) continue;
                const float bi = bs[i], ci = cs[i];
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    s[b][e] = decay * s[b][e] + bi * dx[e];
                    y[e] += s[b][e] * ci;
                }
                store_elems<VEC>(st + (int64_t)i * a.vdim, s[b]);
            }
        }
#pragma unroll
        for (int e = 0; e < VEC; ++e) sums[r * a.vdim + VEC * q + e] = y[e];
    }
    __syncthreads();
    const float dh = a.d[h];
    for (int i = tid; i < a.vdim; i += kThreads) {
        float v = dh * xs[i];
        for (int k = 0; k < rows; ++k) v += sums[k * a.vdim + i];
        a.y[row * a.y_stride + h * a.vdim + i] = (T)v;
    }
}

// ------------------------------------------------------------------ convolution of portions
constexpr int kConvTokens = 16, kFewTokens = 4;         // per thread; where only B and C are convolved, which 16 leave to too few threads (14.5 us, 13,800 tokens)

// VEC channels per thread over TOKENS consecutive tokens, from channel `first` on, in kFewTokens form `units` threads side by side; TAPS > 0: the inputs it looks
// back on stay in registers
template <class T, int VEC, int TAPS, int TOKENS = kConvTokens>
__global__ void __launch_bounds__(kThreads) ssm_conv_kernel(SsmArgs<T> a, const Span* spans, T* out, int first, int units) {
    const Span span = spans[blockIdx.z];
    const unsigned item = blockIdx.x * kThreads + threadIdx.x, block = TOKENS == kConvTokens ? blockIdx.y : item / (unsigned)units;
    const int c = first + (int)(TOKENS == kConvTokens ? item : item - block * units) * VEC, i0 = (int)block * TOKENS;
    if (c >= a.channels || i0 >= span.count || span.slot < 0 || span.slot >= a.num_slots) return;
    const T* in = a.proj + (int64_t)span.row0 * a.proj_stride + a.x_off + c;
    const T* ring = a.ring + (int64_t)span.slot * a.taps * a.channels + c;
    auto input = [&](int i, float (&x)[VEC]) {           // token i of the portion, in front of it if negative
        const int pos = span.pos0 + i;
        if (i >= 0) {
            load_elems<VEC>(in + (int64_t)i * a.proj_stride, x);
        } else if (pos >= 0) {
            load_elems<VEC>(ring + (int64_t)(pos % a.taps) * a.channels, x);
        } else {
#pragma unroll
            for (int e = 0; e < VEC; ++e) x[e] = 0.f;
        }
    };
    T* o = out + (span.row0 - a.xbc_row0 + i0) * a.xbc_stride + c;
    const int end = i0 + TOKENS < span.count ? TOKENS : span.count - i0;
    float bias[VEC];
    load_elems<VEC>(a.conv_bias + c, bias);
    if constexpr (TAPS > 0) {
        float w[TAPS][VEC], x[TAPS][VEC];
#pragma unroll
        for (int k = 0; k < TAPS; ++k)
#pragma unroll
            for (int e = 0; e < VEC; ++e) w[k][e] = a.conv[(int64_t)(c + e) * TAPS + k];
#pragma unroll
        for (int k = 0; k + 1 < TAPS; ++k) input(i0 + k - (TAPS - 1), x[k]);
        // inputs are requested in batches: the compiler moves no load in front of a store
        struct alignas(sizeof(T) * VEC < 16 ? sizeof(T) * VEC : 16) Raw { T e[VEC]; };
        constexpr int kBatch = TOKENS < 8 ? TOKENS : 8;
#pragma unroll
        for (int b = 0; b < TOKENS; b += kBatch) {
            if (b >= end) break;
            Raw raw[kBatch];
#pragma unroll
            for (int i = 0; i < kBatch; ++i)
                raw[i] = *reinterpret_cast<const Raw*>(in + (int64_t)(i0 + (b + i < end ? b + i : end - 1)) * a.proj_stride);
#pragma unroll
            for (int i = 0; i < kBatch; ++i) {
                float v[VEC];
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    x[TAPS - 1][e] = (float)raw[i].e[e];
                    v[e] = bias[e];
#pragma unroll
                    for (int k = 0; k < TAPS; ++k) v[e] += w[k][e] * x[k][e];
                    v[e] = silu_f(v[e]);
                }
                if (b + i < end) store_elems<VEC>(o + (int64_t)(b + i) * a.xbc_stride, v);
#pragma unroll
                for (int k = 0; k + 1 < TAPS; ++k)
#pragma unroll
                    for (int e = 0; e < VEC; ++e) x[k][e] = x[k + 1][e];
            }
        }
    } else {
        for (int i = 0; i < end; ++i) {
            float v[VEC];
#pragma unroll
            for (int e = 0; e < VEC; ++e) v[e] = bias[e];
            for (int k = 0; k < a.taps; ++k) {
                float x[VEC];
                input(i0 + i + k - (a.taps - 1), x);
#pragma unroll
                for (int e = 0; e < VEC; ++e) v[e] += x[e] * a.conv[(int64_t)(c + e) * a.taps + k];
            }
#pragma unroll
            for (int e = 0; e < VEC; ++e) v[e] = silu_f(v[e]);
            store_elems<VEC>(o + (int64_t)i * a.xbc_stride, v);
        }
    }
}

// ------------------------------------------------------------------ any size
// One workgroup per (16 columns of the state, head, span); thread (r, c): column c, state rows r, r + 16, ...
template <class T, int NI>
__global__ void __launch_bounds__(kThreads) ssm_scan_any_kernel(SsmArgs<T> a, const Span* spans) {
    __shared__ float part[2][4][16];
    const Span span = spans[blockIdx.z];
    const int h = blockIdx.y, tid = threadIdx.x, r = tid >> 4, p = blockIdx.x * 16 + (tid & 15);
    if (span.slot < 0 || span.slot >= a.num_slots) return;
    const int n = a.state_n, inner = a.heads * a.vdim, grp = h / (a.heads / a.groups);
    const bool live = p < a.vdim;
    float* st = a.state + ((int64_t)span.slot * a.heads + h) * n * a.vdim + p;
    float s[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int k = r + 16 * i;
        s[i] = live && k < n && span.pos0 > 0 ? st[(int64_t)k * a.vdim] : 0.f;
    }
    const float ah = -expf(a.a_log[h]), dh = a.d[h];
    for (int t = 0; t < span.count; ++t) {
        const int64_t row = span.row0 + t;
        const T* in = a.xbc + (row - a.xbc_row0) * a.xbc_stride;
        const float dt = step_size(a, row, h), decay = expf(ah * dt);
        const float x = live ? (float)in[h * a.vdim + p] : 0.f;
        const T* b = in + inner + grp * n;
        const T* c = b + a.groups * n;
        float y = 0.f;
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int k = r + 16 * i;
            if (k < n) {
                s[i] = decay * s[i] + dt * (float)b[k] * x;
                y += s[i] * (float)c[k];
            }
        }
        y += __shfl_xor(y, 16, 64);
        y += __shfl_xor(y, 32, 64);
        if ((tid & 63) < 16) part[t & 1][tid >> 6][tid & 15] = y;
        __syncthreads();
        if (tid < 16 && live) {
            const float(*q)[16] = part[t & 1];
            a.y[row * a.y_stride + h * a.vdim + p] = (T)(q[0][tid] + q[1][tid] + q[2][tid] + q[3][tid] + dh * x);
        }
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int k = r + 16 * i;
        if (live && k < n) st[(int64_t)k * a.vdim] = s[i];
    }
}

// ------------------------------------------------------------------ chunks
struct ChunkArgs {
    SsmArgs<__bf16> a;
    const Span* spans;
    int seg_len, max_seg, slabs;                 // most tokens of a segment (a multiple of kC), segments of the longest span
    float* ws;                                   // [span][max_seg][heads][state][vdim], then [span][max_seg][heads]: log2 of the decay
    float* ws_decay;
    Turns turns;
};

// A workgroup serves one head and 64 columns of its state over the chunks of one segment.  Wavefront w owns 16 columns as accumulators, of
// eight wavefronts half the state rows each: lane (g, n) holds state rows 16 t + 4 g + e of column n.  That is an operand of the product with C
// as it lies, when the state rows of a k-step of 32 are taken in the order 16 tau + 4 g + e.  The 32 x 32 products C_i B_j are shared
// out over the wavefronts of the first half, weighted, and exchanged through LDS; those of the second add up and write the results.
// OUT = false: only the final state, from zero.  RAW: x comes as it entered the convolution, four taps, which is done here, of the next chunk while this one's products run (the
// pass 175 -> 202 to 212 us under a profiler, the launch that it replaces took 54, the one of B and C that is left 11); the portion is one segment.
// A portion takes as long as its chunks one after the other, and a chunk as long as one wavefront's instructions and reads of LDS (four
// wavefronts: 445 and 30 reads, 3900 clocks with three barriers).  Eight halve what follows one another, and where two chunks lie in LDS one
// barrier is left, behind which a chunk's results are finished under the next one's products.  6 portions of 900 to 3700 tokens of 64 heads,
// the call: 324 us, 310 with the barriers alone, 286 with eight wavefronts.
template <int NS, int WAVES, bool OUT, bool RAW>
__global__ void __launch_bounds__(64 * WAVES, WAVES == 8 && NS <= 4 ? 4 : 2) ssm_chunk_kernel(ChunkArgs args) {
    constexpr int kRow = NS * 64 + 16, kXRow = 2 * kSlab + 16, kMRow = 2 * kC + 16;      // bytes
    constexpr int kThr = 64 * WAVES, kParts = WAVES / 4, NT = 2 * NS / kParts;      // tiles of 16 state rows per wavefront
    constexpr int kAhead = WAVES;                                // chunks whose step sizes are computed together, one per wavefront
    constexpr int NU = (NS * 2 * kC * 2 + kThr - 1) / kThr;      // 16-byte units of B (and of C) per thread
    constexpr int kBufs = NS > 4 || WAVES == 4 ? 1 : 2;                        // chunks of B, C and x in LDS
    extern __shared__ __attribute__((aligned(16))) unsigned char chunk_lds[];
    auto &bbufs = *reinterpret_cast<unsigned char(*)[kBufs][kC * kRow]>(chunk_lds), &cbufs = *reinterpret_cast<unsigned char(*)[kBufs][kC * kRow]>(chunk_lds + sizeof(bbufs));
    auto& xbufs = *reinterpret_cast<unsigned char(*)[kBufs][kC * kXRow]>(chunk_lds + (OUT ? 2 : 1) * sizeof(bbufs));
    unsigned char* behind = chunk_lds + (OUT ? 2 : 1) * sizeof(bbufs) + sizeof(xbufs);
    auto& sums = *reinterpret_cast<float(*)[2][kAhead][kC]>(behind);
    auto& steps = *reinterpret_cast<float(*)[2][kAhead][kC]>(behind + sizeof(sums));
    auto& weights = *reinterpret_cast<float(*)[2][kAhead][kC]>(behind + 2 * sizeof(sums));
    auto& mbufs = *reinterpret_cast<unsigned char(*)[2][2 * kC * kMRow]>(behind + 3 * sizeof(sums));               // OUT
    auto& ybufs = *reinterpret_cast<f32x4_t(*)[2][4][2][64]>(behind + 3 * sizeof(sums) + sizeof(mbufs));           // OUT
    auto& taps = *reinterpret_cast<float(*)[kTaps + 1][kSlab]>(behind + 3 * sizeof(sums) + (OUT ? sizeof(mbufs) + (kParts > 1 ? sizeof(ybufs) : 0) : 0));   // RAW; last: the bias
    const SsmArgs<__bf16>& a = args.a;
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, n = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), half = wave >> 2, cw = wave & 3;
    const int h = blockIdx.y, slab = blockIdx.x % args.slabs, seg = blockIdx.x / args.slabs;
    const int portion = portion_of_turn(&args.spans->row0, args.turns, blockIdx.z);
    const Span span = args.spans[portion];
    const int seg_len = own_segment(span.count, args.seg_len, kC), first = seg * seg_len;
    if (span.slot < 0 || span.slot >= a.num_slots || first >= span.count) return;
    const bool last_seg = first + seg_len >= span.count;
    if (!OUT && last_seg) return;                                // nobody needs its final state yet
    const int count = last_seg ? span.count - first : seg_len;
    const int row0 = span.row0 + first, chunks = (count + kC - 1) / kC;
    const int N = a.state_n, inner = a.heads * a.vdim, grp = h / (a.heads / a.groups);
    const int v0 = slab * kSlab + cw * 16, r0 = half * 16 * NT;  // this wavefront's first column and state row
    const int64_t state_len = (int64_t)N * a.vdim;
    float* from = a.state + ((int64_t)span.slot * a.heads + h) * state_len;
    float* to = from;
    const int64_t rec = ((int64_t)portion * args.max_seg + seg) * a.heads + h;
    if (args.max_seg > 1) {
        if (OUT) from = args.ws + rec * state_len;
        else to = args.ws + rec * state_len;
    }
    const bool load = OUT && (args.max_seg > 1 || span.pos0 > 0), col_live = v0 + n < a.vdim;

    f32x4_t s[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        s[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        if (load && col_live)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (r0 + 16 * t + 4 * g + e < N) s[t][e] = from[(int64_t)(r0 + 16 * t + 4 * g + e) * a.vdim + v0 + n];
    }
    // entries behind the real sizes stay zero
    for (int i = tid; i < (int)((OUT ? 2 : 1) * sizeof(bbufs) + sizeof(xbufs)) / 16; i += kThr) reinterpret_cast<u32x4_t*>(chunk_lds)[i] = u32x4_t{0u, 0u, 0u, 0u};

    const int units = N / 8;
    int u_tok[NU], u_col[NU];                                    // token -1: no such unit; its load repeats another one
#pragma unroll
    for (int i = 0; i < NU; ++i) {
        const int u = tid + kThr * i;
        u_tok[i] = u < kC * units ? u / units : -1;
        u_col[i] = 8 * (u % units);
    }
    constexpr int XV = RAW && kThr == 512 ? 4 : 8, XR = RAW ? kTaps : 1;       // columns of x and rows of the window that a thread brings
    typedef typename std::conditional<XV == 4, u32x2_t, u32x4_t>::type xvec_t;
    const int x_tok = tid / (kSlab / XV) % kC, x_col = XV * (tid % (kSlab / XV));
    const bool x_in = tid < kSlab / XV * kC && slab * kSlab + x_col < a.vdim;
    const int x_chan = h * a.vdim + (x_in ? slab * kSlab + x_col : 0);
    const __bf16* rows = a.xbc + (row0 - a.xbc_row0) * a.xbc_stride;
    const __bf16* b_src = rows + inner + grp * N;
    const __bf16* c_src = b_src + a.groups * N;
    const int64_t x_stride = RAW ? a.proj_stride : a.xbc_stride;
    const __bf16* x_src = RAW ? a.proj + (int64_t)row0 * a.proj_stride + a.x_off + x_chan : rows + x_chan;
    const __bf16* dt_src = a.proj + (int64_t)row0 * a.proj_stride + a.dt_off + h;
    u32x4_t breg[NU], creg[NU];
    xvec_t xreg[XR];
    __bf16 dtreg;
    auto fetch = [&](int c) {                                    // chunk c; tokens behind the last one re-read it
        const int last = count - 1, t0 = c * kC;
        auto tok = [&](int i) -> int64_t { return t0 + i < last ? t0 + i : last; };
#pragma unroll
        for (int i = 0; i < NU; ++i) {
            const int64_t r = tok(u_tok[i] > 0 ? u_tok[i] : 0) * a.xbc_stride;
            breg[i] = *reinterpret_cast<const u32x4_t*>(b_src + r + u_col[i]);
            if constexpr (OUT) creg[i] = *reinterpret_cast<const u32x4_t*>(c_src + r + u_col[i]);
        }
    };
    auto fetch_x = [&](int c) {                                  // behind fetch(c)
        const int last = count - 1, t = c * kC + x_tok;
        const __bf16* r = x_src + (int64_t)((t < last ? t : last) - (XR - 1)) * x_stride;
#pragma unroll
        for (int k = 0; k < XR; ++k) xreg[k] = *reinterpret_cast<const xvec_t*>(r + k * x_stride);
    };
    // the window of a portion's first tokens looks back on the ring, and on zeros in front of the sequence
    auto fetch_first = [&] {
        const int last = count - 1, t = x_tok < last ? x_tok : last;
#pragma unroll
        for (int k = 0; k < XR; ++k) {
            const int i = t + k - (XR - 1), pos = span.pos0 + i;
            xreg[k] = xvec_t{};
            if (i >= 0) xreg[k] = *reinterpret_cast<const xvec_t*>(x_src + (int64_t)i * x_stride);
            else if (pos >= 0) xreg[k] = *reinterpret_cast<const xvec_t*>(a.ring + ((int64_t)span.slot * kTaps + pos % kTaps) * a.channels + x_chan);
        }
    };
    auto fetch_dt = [&](int c) {
        const int t = c * kC + (lane & 31);
        dtreg = dt_src[(int64_t)(t < count ? t : count - 1) * a.proj_stride];
    };
    const float a2 = -expf(a.a_log[h]) * kLog2e, bias = a.dt_bias[h], dh = a.d[h];
    float total = 0.f;                                           // log2 of the segment's decay
    // step sizes of chunks c .. c + kAhead - 1, this wavefront's being c + wave
    auto put_steps = [&](int c) {
        const int group = (c / kAhead) & 1;
        const float dt = (c + wave) * kC + (lane & 31) < count ? softplus_f((float)dtreg + bias) : 0.f;
        float G = fmaxf(a2 * dt, -160.f);                        // nothing is left beyond, and sums stay precise
#pragma unroll
        for (int m = 1; m < kC; m <<= 1) {
            const float up = __shfl_up(G, m, 32);
            G += (lane & 31) >= m ? up : 0.f;
        }
        const float end = __shfl(G, kC - 1, 64);
        if (lane < kC) {
            sums[group][wave][lane] = G;
            steps[group][wave][lane] = dt;
            weights[group][wave][lane] = __builtin_amdgcn_exp2f(end - G) * dt;
        }
        fetch_dt(c + kAhead + wave);
    };
    // x of the chunk requested last, as it enters LDS: of eight wavefronts among the products, of four behind the stores of B and C
    constexpr bool kWithin = WAVES == 8;
    xvec_t xput;
    auto convolve = [&]() __attribute__((always_inline)) {
        if constexpr (!RAW) {
            xput = xreg[0];
        } else {
            float y[XV];
#pragma unroll
            for (int q = 0; q < XV; q += 4) {
                f32x4_t v = *reinterpret_cast<const f32x4_t*>(&taps[kTaps][x_col + q]);
#pragma unroll
                for (int k = 0; k < kTaps; ++k) {
                    const f32x4_t w = *reinterpret_cast<const f32x4_t*>(&taps[k][x_col + q]);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const uint32_t bits = xreg[k][(q + e) / 2];
                        v[e] += w[e] * __builtin_bit_cast(float, e & 1 ? bits & 0xffff0000u : bits << 16);
                    }
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) y[q + e] = silu_f(v[e]);
            }
            typedef __bf16 xbf_t __attribute__((ext_vector_type(XV)));
            xbf_t o;
#pragma unroll
            for (int e = 0; e < XV; ++e) o[e] = (__bf16)y[e];
            xput = __builtin_bit_cast(xvec_t, o);
        }
    };
    auto put = [&](int c) {
#pragma unroll
        for (int i = 0; i < NU; ++i)
            if (u_tok[i] >= 0) {
                *reinterpret_cast<u32x4_t*>(bbufs[c % kBufs] + u_tok[i] * kRow + 2 * u_col[i]) = breg[i];
                if constexpr (OUT) *reinterpret_cast<u32x4_t*>(cbufs[c % kBufs] + u_tok[i] * kRow + 2 * u_col[i]) = creg[i];
            }
        if constexpr (!kWithin) convolve();
        if (x_in) *reinterpret_cast<xvec_t*>(xbufs[c % kBufs] + x_tok * kXRow + 2 * x_col) = xput;
    };
    f32x4_t y[2];
    bf16x8_t xf;
    // what the chunk's own tokens add to the results, and their way out
    auto finish = [&](int c) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            if constexpr (kParts > 1) y[t] += ybufs[c & 1][cw][t][lane];
#pragma unroll
            for (int k = 1; k >= 0; --k) {
                const bf16x8_t mf = *reinterpret_cast<const bf16x8_t*>(mbufs[c & 1] + k * kC * kMRow + (16 * t + n) * kMRow + 16 * g);
                y[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf, mf, y[t], 0, 0, 0);
            }
            const int tok = c * kC + 16 * t + n;
            if (tok < count && v0 + 4 * g < a.vdim) {
                bf16x4_t o;
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = (__bf16)y[t][e];
                *reinterpret_cast<bf16x4_t*>(a.y + (row0 + tok) * a.y_stride + h * a.vdim + v0 + 4 * g) = o;
            }
        }
    };
    fetch(0);
    if constexpr (RAW) fetch_first();
    else fetch_x(0);
    fetch_dt(wave);
    if constexpr (RAW)
        for (int i = tid; i < (kTaps + 1) * kSlab; i += kThr) {
            const int k = i / kSlab, col = i % kSlab, c = h * a.vdim + slab * kSlab + col;
            const bool in = slab * kSlab + col < a.vdim;
            taps[k][col] = !in ? 0.f : k == kTaps ? a.conv_bias[c] : a.conv[(int64_t)c * kTaps + k];
        }
    __syncthreads();                                             // the zero fill
    put_steps(0);
    if constexpr (kWithin) convolve();
    put(0);
    if (chunks > 1) {
        fetch(1);
        fetch_x(1);
    }
    // Behind the barrier the chunk lies in LDS, and the products of the last chunk's tokens, whose results are finished while
    // this chunk's products run.  Everything that is written between two barriers was read last in front of the first.
#pragma unroll 1                                                 // unrolled it spills
    for (int c = 0; c < chunks; ++c) {
        __syncthreads();
        if constexpr (OUT)
            if (half == kParts - 1 && c > 0) finish(c - 1);
        unsigned char *bbuf = bbufs[c % kBufs], *cbuf = cbufs[c % kBufs], *xbuf = xbufs[c % kBufs], *mbuf = mbufs[c & 1];
        const float* sum = sums[(c / kAhead) & 1][c % kAhead];
        const float* step = steps[(c / kAhead) & 1][c % kAhead];
        const float* weight = weights[(c / kAhead) & 1][c % kAhead];
        const float G_end = sum[kC - 1];
        // x of this wavefront's columns: lane (g, n) has tokens 8 g .. 8 g + 7 of column n
        const unsigned char* xr = xbuf + (8 * g + (n >> 2)) * kXRow + (n & 3) * 8 + 32 * cw;
        const i16x4 xlo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)xr);
        const i16x4 xhi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(xr + 4 * kXRow));
        xf = __builtin_bit_cast(bf16x8_t, (i16x8)__builtin_shufflevector(xlo, xhi, 0, 1, 2, 3, 4, 5, 6, 7));
        if constexpr (OUT) {
            if (half == 0) {
                // products C_i B_j of one 16 x 16 tile: lane (g, n) gets tokens j = 4 g + e and i = n of it
                const int sj = cw >> 1, ti = cw & 1;
                f32x4_t m = {0.f, 0.f, 0.f, 0.f};
                if (sj <= ti) {
#pragma unroll
                    for (int k = 0; k < NS; ++k) {
                        const bf16x8_t bf = *reinterpret_cast<const bf16x8_t*>(bbuf + (16 * sj + n) * kRow + 64 * k + 16 * g);
                        const bf16x8_t cf = *reinterpret_cast<const bf16x8_t*>(cbuf + (16 * ti + n) * kRow + 64 * k + 16 * g);
                        m = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf, cf, m, 0, 0, 0);
                    }
                }
                const int i = 16 * ti + n, j0 = 16 * sj + 4 * g;
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int j = j0 + e;
                    v[e] = j <= i ? m[e] * __builtin_amdgcn_exp2f(sum[i] - sum[j]) * step[j] : 0.f;
                    if (j == i) v[e] += dh;
                }
                uint32_t p[2][2];
                split<2, 4>(v, p);
#pragma unroll
                for (int k = 0; k < 2; ++k)
                    *reinterpret_cast<uint2*>(mbuf + k * kC * kMRow + i * kMRow + 2 * j0) = uint2{p[k][0], p[k][1]};
            }
            // products of the state: lane (g, n) gets columns 4 g + e for token n
            y[0] = y[1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < NT / 2; ++k) {
                float sv[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) sv[e] = s[2 * k + e / 4][e % 4];
                bf16x8_t sp[2];
                split_frags<2>(sv, sp);
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const unsigned char* cr = cbuf + (16 * t + n) * kRow + 64 * (half * (NT / 2) + k) + 8 * g;
                    const uint2 lo = *reinterpret_cast<const uint2*>(cr), hi = *reinterpret_cast<const uint2*>(cr + 32);
                    const bf16x8_t cf = __builtin_bit_cast(bf16x8_t, u32x4_t{lo.x, lo.y, hi.x, hi.y});
                    y[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(sp[1], cf, y[t], 0, 0, 0);
                    y[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(sp[0], cf, y[t], 0, 0, 0);
                }
            }
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                y[t] *= __builtin_amdgcn_exp2f(sum[16 * t + n]);
                if (kParts > 1 && half == 0) ybufs[c & 1][cw][t][lane] = y[t];
            }
        }
        if constexpr (kWithin) convolve();
        // the state
        float wx[8], xv[8];
        widen(__builtin_bit_cast(u32x4_t, xf), xv);
#pragma unroll
        for (int e = 0; e < 8; ++e) wx[e] = xv[e] * weight[8 * g + e];
        bf16x8_t xp[3];
        split_frags<3>(wx, xp);
        const float carry = __builtin_amdgcn_exp2f(G_end);
        total += G_end;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const unsigned char* br = bbuf + (8 * g + (n >> 2)) * kRow + (n & 3) * 8 + 2 * r0 + 32 * t;
            const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)br);
            const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(br + 4 * kRow));
            const bf16x8_t bf = __builtin_bit_cast(bf16x8_t, (i16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
            s[t] *= carry;
#pragma unroll
            for (int k = 2; k >= 0; --k) s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf, xp[k], s[t], 0, 0, 0);
        }
        if (c + 1 < chunks) {
            if constexpr (kBufs == 1) __syncthreads();
            if ((c + 1) % kAhead == 0) put_steps(c + 1);
            put(c + 1);
            if (c + 2 < chunks) {
                fetch(c + 2);
                fetch_x(c + 2);
            }
        }
    }
    if constexpr (OUT) {
        __syncthreads();
        if (half == kParts - 1) finish(chunks - 1);
    }
    if (!OUT && slab == 0 && tid == 0) args.ws_decay[rec] = total;
    if (OUT && !last_seg) return;
    if (col_live)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (r0 + 16 * t + 4 * g + e < N) to[(int64_t)(r0 + 16 * t + 4 * g + e) * a.vdim + v0 + n] = s[t][e];
}

// final states of segments from zero -> the states in front of the segments
__global__ void __launch_bounds__(kThreads) ssm_join_kernel(ChunkArgs args) {
    const SsmArgs<__bf16>& a = args.a;
    const Span span = args.spans[blockIdx.z];
    const int h = blockIdx.y;
    const int64_t state_len = (int64_t)a.state_n * a.vdim, i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (i >= state_len || span.slot < 0 || span.slot >= a.num_slots) return;
    float cur = span.pos0 > 0 ? a.state[((int64_t)span.slot * a.heads + h) * state_len + i] : 0.f;
    const int seg_len = own_segment(span.count, args.seg_len, kC), segs = (span.count + seg_len - 1) / seg_len;
    for (int k = 0; k < segs; ++k) {
        const int64_t rec = ((int64_t)blockIdx.z * args.max_seg + k) * a.heads + h;
        float* w = args.ws + rec * state_len + i;
        const float own = k + 1 < segs ? *w : 0.f, decay = k + 1 < segs ? __builtin_amdgcn_exp2f(args.ws_decay[rec]) : 0.f;
        *w = cur;
        cur = cur * decay + own;
    }
}

// ------------------------------------------------------------------ gate and norm
template <class T>
struct NormArgs {
    SsmArgs<T> a;
    const float* norm;                     // [heads * vdim]
    int parts; float eps;
    const int32_t* ring_slot;              // [row][2]: slot, rows of the portion that follow
    const int64_t* positions;
    int64_t portion_row;                   // rows from here on belong to portions
    T* out; int64_t out_stride;
};

// Bound by memory: 13,800 rows of 4096 (two read, one written) 340 MB.  ONCE: rows that are kept, with the streaming hint.
constexpr int kKeep = 4;                   // chunks kept between the sum and the result; more are computed twice
template <class T, int VEC, bool ONCE>
__global__ void __launch_bounds__(kThreads) ssm_norm_kernel(NormArgs<T> b) {
    __shared__ float part[kThreads / 64];
    const SsmArgs<T>& a = b.a;
    const int64_t row = blockIdx.x;
    const int size = a.heads * a.vdim / b.parts, c0 = blockIdx.y * size, tid = threadIdx.x;
    const T* y = a.y + row * a.y_stride + c0;
    const T* z = a.proj + row * a.proj_stride + a.z_off + c0;
    float x[kKeep][VEC], ss = 0.f;
    auto gated = [&](int c, float (&v)[VEC]) {
        float w[VEC];
        load_once<VEC, ONCE>(y + c, v);
        load_once<VEC, ONCE>(z + c, w);
#pragma unroll
        for (int e = 0; e < VEC; ++e) v[e] *= silu_f(w[e]);
    };
#pragma unroll
    for (int j = 0; j < kKeep; ++j) {
        const int c = (tid + j * kThreads) * VEC;
        if (c < size) {
            gated(c, x[j]);
#pragma unroll
            for (int e = 0; e < VEC; ++e) ss += x[j][e] * x[j][e];
        }
    }
    for (int c = (tid + kKeep * kThreads) * VEC; c < size; c += kThreads * VEC) {
        float v[VEC];
        gated(c, v);
#pragma unroll
        for (int e = 0; e < VEC; ++e) ss += v[e] * v[e];
    }
    const float rs = rsqrtf(block_sum<kThreads / 64>(ss, part) / (float)size + b.eps);
    auto put = [&](int c, float (&v)[VEC]) {
        float w[VEC];
        load_elems<VEC>(b.norm + c0 + c, w);
#pragma unroll
        for (int e = 0; e < VEC; ++e) v[e] *= rs * w[e];
        store_elems<VEC>(b.out + row * b.out_stride + c0 + c, v);
    };
#pragma unroll
    for (int j = 0; j < kKeep; ++j) {
        const int c = (tid + j * kThreads) * VEC;
        if (c < size) put(c, x[j]);
    }
    for (int c = (tid + kKeep * kThreads) * VEC; c < size; c += kThreads * VEC) {
        float v[VEC];
        gated(c, v);
        put(c, v);
    }
    if (row >= b.portion_row && blockIdx.y == 0 && b.ring_slot[2 * row + 1] < a.taps - 1) {
        const int slot = b.ring_slot[2 * row];
        if (slot < 0 || slot >= a.num_slots) return;
        T* ring = a.ring + ((int64_t)slot * a.taps + b.positions[row] % a.taps) * a.channels;
        const T* in = a.proj + row * a.proj_stride + a.x_off;
        for (int c = tid; c < a.channels; c += kThreads) ring[c] = in[c];
    }
}

// ------------------------------------------------------------------ launches
bool chunked(int elem, int64_t vdim, int64_t state_n) { return elem == INFER_ELEM_BF16 && vdim % 8 == 0 && state_n % 8 == 0 && state_n <= 256; }

// How portions are walked: wavefronts of a workgroup, and the segments that they are cut into so that enough workgroups run (most tokens of a
// segment and their largest number).  Cut portions are walked twice, which pays below one workgroup of eight wavefronts or one and a half
// of four per compute unit.  Heads of 128 x 64, the call in us, four wavefronts cut for three workgroups per compute unit / eight cut for
// two: 6 portions of 900 to 3700 tokens of 64 heads 325 / 286, 5 of 1000 to 3000 248 / 211, 8 of 1000 174 / 158, 4 of 500 to 4000 252 / 245, 11 of
// 500 to 1500 of 32 heads 185 / 158, 1 of 300 40 / 36.  Two workgroups of eight fit a compute unit; where there are more, four are ahead
// (10 of 800 to 1800 of 64 heads 250 / 256), and with a long portion by itself, cut into equal segments: what the chip has to do in all
// counts there, not the longest chain.  1 of 3500 / 4319 / 6000 / 9000 / 13900, four / eight: 64 heads 105 / 101, 122.2 / 119.6, 154.4 / 157.1,
// 216 / 221, 311 / 322; 32 heads 75.2 / 71.0, 87.8 / 82.8, 100.1 / 97.1, 131.4 / 131.4, 203 / 202.
// Segments of one length per portion instead of one for the batch: 6 portions of 32 heads 228 -> 220.
struct Walk { int waves, seg_len, max_seg; };
Walk walk_of(int64_t heads, int64_t vdim, int64_t state_n, int64_t num_spans, int64_t max_span) {
    const int64_t units = heads * ((vdim + kSlab - 1) / kSlab) * num_spans, chunks = (max_span + kC - 1) / kC;
    const bool wide = units <= 512 && state_n <= 128 && !(num_spans == 1 && units * max_span > 64 * 5000);
    const int64_t full = wide ? 256 : 384;
    int64_t want = units > 0 && units < full ? (2 * full + units - 1) / units : 1;
    if (want > chunks / 4) want = chunks / 4;              // no segment shorter than four chunks
    if (want < 1) want = 1;
    const int64_t per = (chunks + want - 1) / want, seg_len = (per > 0 ? per : 1) * kC;
    return Walk{wide ? 8 : 4, (int)seg_len, (int)(max_span > 0 ? (max_span + seg_len - 1) / seg_len : 1)};
}

template <int NS, int WAVES, bool OUT, bool RAW>
int launch_chunk(const ChunkArgs& c, int64_t num_spans, hipStream_t st) {
    constexpr size_t bufs = NS > 4 || WAVES == 4 ? 1 : 2;
    constexpr size_t lds = kC * (bufs * ((OUT ? 2 : 1) * (NS * 64 + 16) + 2 * kSlab + 16) + (OUT ? 2 * 2 * (2 * kC + 16) : 0)) +
                           3 * 2 * WAVES * kC * sizeof(float) + (OUT && WAVES == 8 ? 2 * 4 * 2 * 64 * sizeof(f32x4_t) : 0) +
                           (RAW ? (kTaps + 1) * kSlab * sizeof(float) : 0);
    auto kernel = &ssm_chunk_kernel<NS, WAVES, OUT, RAW>;
    if (lds > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return (int)e;
    }
    hipLaunchKernelGGL(kernel, dim3((unsigned)(c.slabs * c.max_seg), (unsigned)c.a.heads, (unsigned)num_spans), dim3(64 * WAVES), lds, st, c);
    return (int)hipGetLastError();
}

template <int NS, int WAVES, bool RAW>
int launch_chunks(const ChunkArgs& c, int64_t num_spans, hipStream_t st) {
    if constexpr (RAW) return launch_chunk<NS, WAVES, true, true>(c, num_spans, st);        // one segment
    if (c.max_seg > 1) {
        const int rc = launch_chunk<NS, WAVES, false, false>(c, num_spans, st);
        if (rc) return rc;
        const int64_t state_len = (int64_t)c.a.state_n * c.a.vdim;
        hipLaunchKernelGGL(ssm_join_kernel, dim3((unsigned)((state_len + kThreads - 1) / kThreads), (unsigned)c.a.heads, (unsigned)num_spans),
                           dim3(kThreads), 0, st, c);
    }
    return launch_chunk<NS, WAVES, true, false>(c, num_spans, st);
}

template <class T>
int portions(SsmArgs<T>& a, const Span* spans, int64_t num_spans, int64_t max_span, int64_t row0, int64_t n, T* xbc, float* ws,
             int64_t ws_floats, hipStream_t st) {
    const int64_t rows = n - row0;
    if (!spans || !xbc || num_spans < 1 || num_spans > 65535 || max_span < 1 || max_span > rows) return INFER_KV_EINVAL;
    a.xbc = xbc;
    a.xbc_stride = a.channels;
    a.xbc_row0 = row0;
    const bool vec = a.channels % 8 == 0 && a.proj_stride % 8 == 0 && a.x_off % 8 == 0 && ptr_aligned(a.proj, 16) && ptr_aligned(xbc, 16) &&
                     ptr_aligned(a.ring, 16) && ptr_aligned(a.conv_bias, 16);
    const int64_t token_blocks = (max_span + kConvTokens - 1) / kConvTokens;
    if (token_blocks > 65535) return INFER_KV_EINVAL;
    const dim3 block(kThreads);
    auto convolve = [&] {
        const dim3 grid((unsigned)(((vec ? a.channels / 8 : a.channels) + kThreads - 1) / kThreads), (unsigned)token_blocks, (unsigned)num_spans);
        if (vec && a.taps == 4) hipLaunchKernelGGL((ssm_conv_kernel<T, 8, 4>), grid, block, 0, st, a, spans, xbc, 0, 0);
        else if (vec) hipLaunchKernelGGL((ssm_conv_kernel<T, 8, 0>), grid, block, 0, st, a, spans, xbc, 0, 0);
        else hipLaunchKernelGGL((ssm_conv_kernel<T, 1, 0>), grid, block, 0, st, a, spans, xbc, 0, 0);
        return (int)hipGetLastError();
    };
    if constexpr (sizeof(T) == 2) {
        if (chunked(INFER_ELEM_BF16, a.vdim, a.state_n) && vec && a.y_stride % 4 == 0 && ptr_aligned(a.y, 8)) {
            const Walk walk = walk_of(a.heads, a.vdim, a.state_n, num_spans, max_span);
            const int slabs = (a.vdim + kSlab - 1) / kSlab;
            ChunkArgs c{a, spans, walk.seg_len, walk.max_seg, slabs, nullptr, nullptr, walk.max_seg > 1 ? Turns{} : turns_of(num_spans, (int64_t)a.heads * slabs, rows)};
            if (c.max_seg > 1) {
                const int64_t records = num_spans * c.max_seg * a.heads, len = (int64_t)a.state_n * a.vdim;
                if (!ws || ws_floats < records * (len + 1)) return INFER_KV_EWORKSPACE;
                c.ws = ws;
                c.ws_decay = ws + records * len;
            }
            // x is convolved where it is used, and only B and C, which all heads of a group share, by a launch of their own, unless portions are cut,
            // since their x would be convolved twice (1 of 4000 tokens 123 -> 125 us).  The call, us, x by a launch / inside: 64 heads, 6 portions
            // of 900 to 3700 tokens 266 / 255, 8 of 1000 152 / 140, 10 of 800 to 1800 229 / 219, 32 of 60 to 200 109 / 107; 32 heads, 20 of 200 to 900 135 / 121,
            // 9 of 500 to 1500 134 / 127.
            const int64_t items = (int64_t)(a.channels - a.heads * a.vdim) / 8 * ((max_span + kFewTokens - 1) / kFewTokens);
            const bool raw = a.taps == kTaps && c.max_seg == 1 && items <= 0x7fffffff;
            if (raw) {
                hipLaunchKernelGGL((ssm_conv_kernel<T, 8, kTaps, kFewTokens>), dim3((unsigned)((items + kThreads - 1) / kThreads), 1, (unsigned)num_spans), block, 0, st,
                                   a, spans, xbc, a.heads * a.vdim, (a.channels - a.heads * a.vdim) / 8);
                const hipError_t e = hipGetLastError();
                if (e != hipSuccess) return (int)e;
            } else if (const int rc = convolve()) {
                return rc;
            }
            auto walked = [&](auto within) {
                constexpr bool RAW = decltype(within)::value;
                if (a.state_n > 128) return launch_chunks<8, 4, RAW>(c, num_spans, st);
                if (walk.waves == 8) return a.state_n <= 64 ? launch_chunks<2, 8, RAW>(c, num_spans, st) : launch_chunks<4, 8, RAW>(c, num_spans, st);
                return a.state_n <= 64 ? launch_chunks<2, 4, RAW>(c, num_spans, st) : launch_chunks<4, 4, RAW>(c, num_spans, st);
            };
            return raw ? walked(std::true_type{}) : walked(std::false_type{});
        }
    }
    if (const int rc = convolve()) return rc;
    const dim3 sgrid((unsigned)((a.vdim + 15) / 16), (unsigned)a.heads, (unsigned)num_spans);
    if (a.state_n <= 64) hipLaunchKernelGGL((ssm_scan_any_kernel<T, 4>), sgrid, block, 0, st, a, spans);
    else if (a.state_n <= 256) hipLaunchKernelGGL((ssm_scan_any_kernel<T, 16>), sgrid, block, 0, st, a, spans);
    else if (a.state_n <= 1024) hipLaunchKernelGGL((ssm_scan_any_kernel<T, 64>), sgrid, block, 0, st, a, spans);
    else return INFER_KV_EUNSUPPORTED;
    return (int)hipGetLastError();
}

bool size_in(int64_t v, int64_t lo, int64_t hi) { return v >= lo && v <= hi; }

}  // namespace

extern "C" int64_t infer_state_space_workspace_floats(int elem, int64_t heads, int64_t vdim, int64_t state_n, int64_t num_spans,
                                                      int64_t max_span) {
    if (!chunked(elem, vdim, state_n) || heads < 1 || num_spans < 1 || max_span < 1) return 0;
    const int64_t max_seg = walk_of(heads, vdim, state_n, num_spans, max_span).max_seg;
    return max_seg > 1 ? num_spans * max_seg * heads * (state_n * vdim + 1) : 0;
}

extern "C" int infer_state_space(int elem, const void* proj, int64_t proj_stride, int64_t z_off, int64_t x_off, int64_t dt_off,
                                 int64_t heads, int64_t vdim, int64_t state_n, int64_t groups, int64_t taps, const float* conv,
                                 const float* conv_bias, const float* dt_bias, const float* a_log, const float* d, const float* norm,
                                 int64_t norm_parts, float eps, void* ring, float* state, int64_t num_slots, const int32_t* slots,
                                 const int64_t* positions, int64_t decode_rows, const int32_t* spans, int64_t num_spans,
                                 int64_t max_span, const int32_t* ring_slot, int64_t n, void* xbc, void* y, float* workspace,
                                 int64_t workspace_floats, void* out, int64_t out_stride, void* stream) {
    if (n < 0 || n > 0x7fffffff || decode_rows < 0 || decode_rows > n) return INFER_KV_EINVAL;
    if (n == 0) return INFER_KV_OK;
    if (!size_in(heads, 1, 4096) || !size_in(vdim, 1, 1024) || !size_in(state_n, 1, 1024) || !size_in(groups, 1, heads) || heads % groups ||
        !size_in(taps, 1, 64) || norm_parts < 1 || heads * vdim % norm_parts || norm_parts > 65535 || num_slots < 1)
        return INFER_KV_EINVAL;
    const int64_t inner = heads * vdim, channels = inner + 2 * groups * state_n;
    if (!proj || !conv || !conv_bias || !dt_bias || !a_log || !d || !norm || !ring || !state || !y || !out || !positions || z_off < 0 ||
        x_off < 0 || dt_off < 0 || z_off + inner > proj_stride || x_off + channels > proj_stride || dt_off + heads > proj_stride ||
        out_stride < inner || proj_stride > (1 << 24) || (decode_rows > 0 && !slots) || (decode_rows < n && !ring_slot))
        return INFER_KV_EINVAL;
    hipStream_t st = (hipStream_t)stream;
    auto go = [&](auto zero) -> int {
        using T = decltype(zero);
        SsmArgs<T> a{(const T*)proj, proj_stride, (int)z_off, (int)x_off, (int)dt_off, (int)heads, (int)vdim, (int)state_n, (int)groups,
                     (int)channels, (int)taps, conv, conv_bias, dt_bias, a_log, d, (T*)ring, state, (int)num_slots, (T*)y, inner, nullptr, 0, 0};
        if (decode_rows > 0) {
            if (decode_rows > 65535) return INFER_KV_EINVAL;
            const bool vec = vdim % 4 == 0 && ptr_aligned(state, 16);
            const int64_t quads = vdim / (vec ? 4 : 1);
            if (quads > kThreads) return INFER_KV_EUNSUPPORTED;
            const size_t lds = sizeof(float) * ((vdim + 3) / 4 * 4 + 2 * ((state_n + 3) / 4 * 4) + kThreads / quads * vdim);
            const dim3 grid((unsigned)heads, (unsigned)decode_rows), block(kThreads);
            if (vec) hipLaunchKernelGGL((ssm_step_kernel<T, 4>), grid, block, lds, st, a, slots, positions);
            else hipLaunchKernelGGL((ssm_step_kernel<T, 1>), grid, block, lds, st, a, slots, positions);
        }
        if (decode_rows < n) {
            const int rc = portions<T>(a, (const Span*)spans, num_spans, max_span, decode_rows, n, (T*)xbc, workspace, workspace_floats, st);
            if (rc) return rc;
        }
        const NormArgs<T> b{a, norm, (int)norm_parts, eps, ring_slot, positions, decode_rows, (T*)out, out_stride};
        const int64_t size = inner / norm_parts;
        const bool vec = size % 8 == 0 && inner % 8 == 0 && proj_stride % 8 == 0 && z_off % 8 == 0 && out_stride % 8 == 0 &&
                         ptr_aligned(proj, 16) && ptr_aligned(y, 16) && ptr_aligned(out, 16) && ptr_aligned(norm, 16);
        const dim3 grid((unsigned)n, (unsigned)norm_parts), block(kThreads);
        if (vec && size <= 8 * kKeep * kThreads && beyond_caches(2 * n * inner * (int64_t)sizeof(T), inner > 2048 ? 35 : 38)) hipLaunchKernelGGL((ssm_norm_kernel<T, 8, true>), grid, block, 0, st, b);
        else if (vec) hipLaunchKernelGGL((ssm_norm_kernel<T, 8, false>), grid, block, 0, st, b);
        else hipLaunchKernelGGL((ssm_norm_kernel<T, 1, false>), grid, block, 0, st, b);
        return (int)hipGetLastError();
    };
    if (elem == INFER_ELEM_BF16) return go(__bf16(0.f));
    if (elem == INFER_ELEM_F32) return go(0.f);
    return INFER_KV_EUNSUPPORTED;
}
