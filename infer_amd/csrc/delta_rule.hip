// Gated delta rule with a decay per key channel, for gfx950 (MI355X).  Per head, over a float32 state S[dim][vdim]:
//     S <- e^g * S (rows);  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q
// with k, q unit vectors behind a short causal convolution and silu, g = -exp(A) softplus(a + dt) <= 0.
//
//   delta_step_kernel    one token per sequence (decode): convolution, norms, gates, recurrence, output norm and
//                        output gate in one launch; one workgroup per (sequence, head), the state passes
//                        through registers once
//   delta_prep_kernel    prompt portions in chunks of 16 tokens, all chunks in parallel: convolution, norms,
//                        gates and everything of a chunk that does not need the state
//   delta_scan_kernel    walks the chunks of a portion; a wavefront holds 16 columns of the state as float32 MFMA
//                        accumulators
//   delta_scan_slab_kernel   the same for few portions and heads: a workgroup per head and 16 to 64 columns, the rows shared out over its wavefronts
//   delta_out_kernel     output norm and gate of the scanned tokens; the convolution's tail goes to its ring
//   delta_scan_wide_kernel   scan, output norm and gate in one launch, for batches that fill the chip with one workgroup per
//                        (portion, head); delta_ring_kernel then writes the rings
//
// Chunk form.  Let G_i be the sum of g over the chunk's tokens up to i, S the state before the chunk.
//     u_i = beta_i (v_i - S^T (e^{G_i} k_i) - sum_{j<i} A_ij u_j),    A_ij = sum_d k_i[d] k_j[d] e^{G_i - G_j}[d]
// so U = T (beta V) - T (beta e^G K) S with T = (I + tril(beta A, -1))^-1, and
//     o_i = (e^{G_i} q_i)^T S + sum_{j<=i} B_ij u_j,                  B_ij = sum_d q_i[d] k_j[d] e^{G_i - G_j}[d]
//     S'  = e^{G_last} S + sum_j (e^{G_last - G_j} k_j) u_j^T.
// Every exponent is a difference that is <= 0, so nothing overflows however strong the decay is.  All of it is
// float32, the products included (v_mfma_f32_16x16x4_f32; in the wide and the slab scan six bf16 products of the pieces of a float).
//
// The last `taps` inputs of the convolution live in a ring per sequence (entry position % taps).  A position below
// zero counts as zero and a portion that starts at position 0 starts from a zero state, so a slot needs no clearing
// when another sequence takes it over.
#include "conv_window.h"
#include "pieces.h"
#include "segments.h"

#include <type_traits>

namespace {

constexpr int kC = 16;               // tokens per chunk
constexpr int kStepThreads = 256;

template <class T>
struct DeltaArgs {
    // inputs of a token row: [q: kv_heads x dim | k: kv_heads x dim | v: heads x vdim | ...], columns 0 .. channels - 1
    const T* proj; int64_t proj_stride;
    int beta_off;                                   // column of the write-strength logits in `proj`
    const T* decay; int64_t decay_stride;           // [row][heads * dim]
    const T* gate; int64_t gate_stride;             // [row][heads * vdim]
    const float* conv;                              // [channels][taps]
    const float* a_log; const float* dt_bias; const float* norm;   // [heads], [heads * dim], [vdim]
    T* ring;                                        // [slots][taps][channels]
    float* state;                                   // [slots][heads][dim_pad][vdim_pad]
    int num_slots;
    int heads, kv_heads, dim, vdim, dim_pad, vdim_pad, taps, channels;
    float eps, q_scale;
    T* out; int64_t out_stride;                     // [row][heads * vdim]
};

// silu of the convolution of channel c at position `pos`; row(p) is the batch row of position p >= first, earlier
// positions are in the ring
template <class T, class Row>
__device__ __forceinline__ float conv_silu(const DeltaArgs<T>& a, int c, int64_t pos, int64_t first, int slot, Row row) {
    const float* w = a.conv + (int64_t)c * a.taps;
    float s = 0.f;
    for (int j = 0; j < a.taps; ++j) {
        const int64_t p = pos - j;
        if (p < 0) break;
        const float x = p >= first ? (float)a.proj[row(p) * a.proj_stride + c]
                                   : (float)a.ring[((int64_t)slot * a.taps + p % a.taps) * a.channels + c];
        s += w[a.taps - 1 - j] * x;
    }
    return silu_f(s);
}

template <class T>
__device__ __forceinline__ float log2_decay(const DeltaArgs<T>& a, int64_t row, int h, int d, float rate) {
    const int i = h * a.dim + d;
    return -rate * softplus_f((float)a.decay[row * a.decay_stride + i] + a.dt_bias[i]) * kLog2e;
}

// ------------------------------------------------------------------ one token per sequence
// Thread (r, c): column group c (4 columns of the state), rows r, r + R, ...  NP = rows per thread kept in
// registers; NP = 0: the state is too large for that and is read twice.
template <class T, int NP>
__global__ void __launch_bounds__(kStepThreads) delta_step_kernel(DeltaArgs<T> a, const int32_t* slots, const int64_t* positions) {
    extern __shared__ __attribute__((aligned(16))) float sh[];
    const int row = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
    const int slot = slots[row];
    T* out = a.out + (int64_t)row * a.out_stride + (int64_t)h * a.vdim;
    if (slot < 0 || slot >= a.num_slots) {           // a padding row of a captured batch
        for (int v = tid; v < a.vdim; v += kStepThreads) out[v] = (T)0.f;
        return;
    }
    const int64_t pos = positions[row];
    const int group = a.heads / a.kv_heads, kvh = h / group;
    const int cgs = a.vdim_pad / 4, rgs = kStepThreads / cgs;
    float* ks = sh;                                  // [dim_pad]
    float* qs = ks + a.dim_pad;
    float* es = qs + a.dim_pad;                      // e^g
    float* vs = es + a.dim_pad;                      // [vdim_pad]
    float* red = vs + a.vdim_pad;                    // [rgs][vdim_pad]
    float* part = red + rgs * a.vdim_pad;            // [3][4]

    const int cg = tid % cgs, rg = tid / cgs;
    const bool works = rg < rgs;
    float* sp = a.state + (((int64_t)slot * a.heads + h) * a.dim_pad) * a.vdim_pad + 4 * cg;
    f32x4_t s[NP > 0 ? NP : 1];
    if constexpr (NP > 0) {
        if (works)
#pragma unroll
            for (int i = 0; i < NP; ++i) {
                const int d = rg + i * rgs;
                s[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
                if (pos > 0 && d < a.dim_pad) s[i] = *reinterpret_cast<const f32x4_t*>(sp + (int64_t)d * a.vdim_pad);
            }
    }
    auto this_row = [&](int64_t) { return (int64_t)row; };
    const float rate = expf(a.a_log[h]);
    float sk = 0.f, sq = 0.f;
    for (int d = tid; d < a.dim_pad; d += kStepThreads) {
        float k = 0.f, q = 0.f, e = 1.f;
        if (d < a.dim) {
            q = conv_silu(a, kvh * a.dim + d, pos, pos, slot, this_row);
            k = conv_silu(a, (a.kv_heads + kvh) * a.dim + d, pos, pos, slot, this_row);
            e = exp2f(log2_decay(a, row, h, d, rate));
        }
        sk += k * k;
        sq += q * q;
        ks[d] = k; qs[d] = q; es[d] = e;
    }
    for (int v = tid; v < a.vdim_pad; v += kStepThreads)
        vs[v] = v < a.vdim ? conv_silu(a, 2 * a.kv_heads * a.dim + h * a.vdim + v, pos, pos, slot, this_row) : 0.f;
    // The ring holds `taps` entries, one more than the convolution looks back: the entry this token overwrites is
    // not read by anyone, so every workgroup may write its own channels at any time.
    T* ring = a.ring + ((int64_t)slot * a.taps + pos % a.taps) * a.channels;
    const T* in = a.proj + (int64_t)row * a.proj_stride;
    if (h % group == 0)
        for (int d = tid; d < a.dim; d += kStepThreads) {
            ring[kvh * a.dim + d] = in[kvh * a.dim + d];
            ring[(a.kv_heads + kvh) * a.dim + d] = in[(a.kv_heads + kvh) * a.dim + d];
        }
    for (int v = tid; v < a.vdim; v += kStepThreads) {
        const int c = 2 * a.kv_heads * a.dim + h * a.vdim + v;
        ring[c] = in[c];
    }
    const float inv_k = rsqrtf(block_sum<4>(sk, part) + 1e-6f);
    const float inv_q = rsqrtf(block_sum<4>(sq, part + 4) + 1e-6f) * a.q_scale;
    const float beta = sigmoid_f((float)in[a.beta_off + h]);

    // S^T k after the decay
    f32x4_t dot = {0.f, 0.f, 0.f, 0.f};
    if (works) {
        if constexpr (NP > 0) {
#pragma unroll
            for (int i = 0; i < NP; ++i) {
                const int d = rg + i * rgs;
                if (d < a.dim_pad) {
                    s[i] *= es[d];
                    dot += s[i] * ks[d];
                }
            }
        } else if (pos > 0) {
            for (int d = rg; d < a.dim_pad; d += rgs) dot += *reinterpret_cast<const f32x4_t*>(sp + (int64_t)d * a.vdim_pad) * (es[d] * ks[d]);
        }
        *reinterpret_cast<f32x4_t*>(red + rg * a.vdim_pad + 4 * cg) = dot;
    }
    __syncthreads();
    f32x4_t u = {0.f, 0.f, 0.f, 0.f};
    if (works) {
        for (int r = 0; r < rgs; ++r) u += *reinterpret_cast<const f32x4_t*>(red + r * a.vdim_pad + 4 * cg);
        u = (*reinterpret_cast<const f32x4_t*>(vs + 4 * cg) - u * inv_k) * (beta * inv_k);     // k enters as ks * inv_k
    }
    __syncthreads();
    f32x4_t o = {0.f, 0.f, 0.f, 0.f};
    if (works) {
        if constexpr (NP > 0) {
#pragma unroll
            for (int i = 0; i < NP; ++i) {
                const int d = rg + i * rgs;
                if (d < a.dim_pad) {
                    s[i] += u * ks[d];
                    o += s[i] * qs[d];
                    *reinterpret_cast<f32x4_t*>(sp + (int64_t)d * a.vdim_pad) = s[i];
                }
            }
        } else {
            for (int d = rg; d < a.dim_pad; d += rgs) {
                f32x4_t x = {0.f, 0.f, 0.f, 0.f};
                if (pos > 0) x = *reinterpret_cast<const f32x4_t*>(sp + (int64_t)d * a.vdim_pad) * es[d];
                x += u * ks[d];
                o += x * qs[d];
                *reinterpret_cast<f32x4_t*>(sp + (int64_t)d * a.vdim_pad) = x;
            }
        }
        *reinterpret_cast<f32x4_t*>(red + rg * a.vdim_pad + 4 * cg) = o * inv_q;
    }
    __syncthreads();
    // vdim_pad <= 1024 = 4 column groups of threads; one thread per column group finishes the row
    float so = 0.f;
    f32x4_t y = {0.f, 0.f, 0.f, 0.f};
    if (tid < cgs) {
        for (int r = 0; r < rgs; ++r) y += *reinterpret_cast<const f32x4_t*>(red + r * a.vdim_pad + 4 * tid);
#pragma unroll
        for (int e = 0; e < 4; ++e) so += y[e] * y[e];       // padded columns are zero
    }
    const float rs = rsqrtf(block_sum<4>(so, part + 8) / (float)a.vdim + a.eps);
    if (tid < cgs) {
        const T* gr = a.gate + (int64_t)row * a.gate_stride + (int64_t)h * a.vdim;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int v = 4 * tid + e;
            if (v < a.vdim) out[v] = (T)(y[e] * rs * a.norm[v] * sigmoid_f((float)gr[v]));
        }
    }
}

// ------------------------------------------------------------------ prompt portions
struct ChunkDesc { int32_t row0, count, pos0, first_pos, slot, pad; };   // first_pos: where the portion starts
struct PortionDesc { int32_t chunk0, chunks, slot, pos0; };

// A chunk's record, floats, each part in the order in which the lanes of the scan read it (lane = 16 q + m takes the
// four consecutive floats at 4 * lane of a 256-float fragment):
//   W   [dim_pad / 16][256]   element (i, d):  T (beta e^G K)
//   Q   [dim_pad / 16][256]   element (i, d):  e^G q
//   K   [dim_pad / 16][256]   element (j, d):  e^{G_last - G_j} k_j, rows d
//   B   [256]                 element (i, j)
//   E   [dim_pad]             e^{G_last}
//   V   [vdim_pad / 16][256]  element (i, v):  T (beta V)
__host__ __device__ inline int64_t record_floats(int dim_pad, int vdim_pad) { return 48 * (int64_t)dim_pad + 256 + dim_pad + 16 * (int64_t)vdim_pad; }

// The convolution of four channels over tokens t0 .. t0 + 7 of a chunk, for four taps, the window in registers.
// c: first channel, dst: LDS row of token t0, column of the channel.  INNER: all 16 tokens exist and the window of
// the first one lies inside the portion.
template <class T, bool INNER>
__device__ __forceinline__ void conv4_silu(const DeltaArgs<T>& a, const ChunkDesc& cd, int c, int t0, float* dst, int pitch) {
    float x[11][4], w[4][4];
#pragma unroll
    for (int e = 0; e < 4; ++e) load_elems<4>(a.conv + 4 * (c + e), w[e]);
    if constexpr (INNER) {
        const T* src = a.proj + (int64_t)(cd.row0 + t0 - 3) * a.proj_stride + c;
#pragma unroll
        for (int j = 0; j < 11; ++j, src += a.proj_stride) load_elems<4>(src, x[j]);
    }
#pragma unroll
    for (int j = 0; j < (INNER ? 0 : 11); ++j) {
        const int t = t0 + j - 3;
        const WindowRow from = window_row(cd.count, cd.pos0, cd.first_pos, t);
#pragma unroll
        for (int e = 0; e < 4; ++e) x[j][e] = 0.f;
        if (from != WindowRow::kNone)
            load_elems<4>(from == WindowRow::kBatch ? a.proj + (int64_t)(cd.row0 + t) * a.proj_stride + c
                                                    : a.ring + ((int64_t)cd.slot * 4 + ((cd.pos0 + t) & 3)) * a.channels + c, x[j]);
    }
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        float y[4];
        const bool in = INNER || t0 + t < cd.count;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            y[e] = 0.f;
#pragma unroll
            for (int j = 0; j < 4; ++j) y[e] += w[e][j] * x[t + j][e];
            y[e] = in ? silu_f(y[e]) : 0.f;
        }
        store_elems<4>(dst + t * pitch, y);
    }
}

// softplus in units of log2: log2(1 + e^z)
__device__ __forceinline__ float softplus_log2(float z) {
    const float e = __builtin_amdgcn_exp2f(-fabsf(z) * kLog2e);
    const float l = e < 0.02f ? e * (1.f - e * (0.5f - e * (0.33333333f - 0.25f * e))) * kLog2e : __builtin_amdgcn_logf(1.f + e);
    return fmaxf(z, 0.f) * kLog2e + l;
}

// Decay of a whole chunk, in log2 units, up to which e^{G_i - G_j} may be split into two factors.
constexpr float kSplitRange = 48.f;

// x summed over the rows of 16 lanes of a wavefront, and over the 32 lanes of its halves, in all of them
__device__ __forceinline__ float row_sum(float x) {
    auto ror = [](float v, auto C) { return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), decltype(C)::value, 0xf, 0xf, false)); };
    x += ror(x, std::integral_constant<int, 0x128>{});          // rotations by 8, 4, 2 and 1
    x += ror(x, std::integral_constant<int, 0x124>{});
    x += ror(x, std::integral_constant<int, 0x122>{});
    x += ror(x, std::integral_constant<int, 0x121>{});
    return x;
}
__device__ __forceinline__ float half_sum(float x) {
    const unsigned u = __builtin_bit_cast(unsigned, row_sum(x));
    const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    const unsigned lo = r[0], hi = r[1];
    return __builtin_bit_cast(float, lo) + __builtin_bit_cast(float, hi);
}
template <int LANES>
__device__ __forceinline__ float lanes_sum(float x) {
    static_assert(LANES == 16 || LANES == 32, "lanes");
    return LANES == 16 ? row_sum(x) : half_sum(x);
}

// VEC: four channels at a time, four taps; otherwise any size, one element at a time.
template <class T, bool VEC>
__global__ void __launch_bounds__(256) delta_prep_kernel(DeltaArgs<T> a, const ChunkDesc* chunks, float* records) {
    extern __shared__ __attribute__((aligned(16))) float sh[];
    const int tid = threadIdx.x, h = blockIdx.y, lane = tid & 63, wave = tid >> 6;
    const ChunkDesc c = chunks[blockIdx.x];
    const int dp = a.dim_pad, pk = dp + 4, pv = a.vdim_pad + 4;
    float* qs = sh;                    // [16][pk] q, then e^G q
    float* ks = qs + kC * pk;          // [16][pk] k, then e^G k
    float* gs = ks + kC * pk;          // [16][pk] running log2 decay G, then e^{G_last - G} k
    float* vs = gs + kC * pk;          // [16][pv]
    float* pp = vs + kC * pv;          // [2][2][256] products of the token pairs (k k, q k), in two parts each
    float* lt = pp + 1024;             // [16][20] column s: beta * A of the tokens behind s
    float* tb = lt;                    // [16][20] T * beta, when those have been used
    float* gl = lt + kC * 20;          // [dp] G_last
    float* inv = gl + dp;              // [2][16] 1 / length of k and q
    float* bs = inv + 32;              // [16] beta
    const int group = a.heads / a.kv_heads, kvh = h / group;
    const int cq = kvh * a.dim, ck = (a.kv_heads + kvh) * a.dim, cv = 2 * a.kv_heads * a.dim + h * a.vdim;
    float* rec = records + ((int64_t)blockIdx.x * a.heads + h) * record_floats(dp, a.vdim_pad);
    const float rate = expf(a.a_log[h]);

    if constexpr (VEC) {
        const int nd = a.dim / 4, nv = a.vdim / 4, n = 2 * nd + nv;
        const bool inner = c.count == kC && c.pos0 - 3 >= c.first_pos;
        for (int i = tid; i < 2 * n; i += 256) {
            const int half = i >= n, j = i - half * n, t0 = 8 * half;
            const int col = j < nd ? 4 * j : j < 2 * nd ? 4 * (j - nd) : 4 * (j - 2 * nd);
            const int ch = col + (j < nd ? cq : j < 2 * nd ? ck : cv), pitch = j < 2 * nd ? pk : pv;
            float* dst = (j < nd ? qs : j < 2 * nd ? ks : vs) + t0 * pitch + col;
            if (inner) conv4_silu<T, true>(a, c, ch, t0, dst, pitch);
            else conv4_silu<T, false>(a, c, ch, t0, dst, pitch);
        }
        for (int i = tid; i < kC * nd; i += 256) {
            const int t = i / nd, d = 4 * (i - t * nd);
            float x[4] = {0.f, 0.f, 0.f, 0.f};
            if (t < c.count) {
                float dt[4];
                load_elems<4>(a.decay + (int64_t)(c.row0 + t) * a.decay_stride + h * a.dim + d, x);
                load_elems<4>(a.dt_bias + h * a.dim + d, dt);
#pragma unroll
                for (int e = 0; e < 4; ++e) x[e] = -rate * softplus_log2(x[e] + dt[e]);
            }
            store_elems<4>(gs + t * pk + d, x);
        }
        for (int i = tid; i < kC * (dp - a.dim); i += 256) {
            const int t = i / (dp - a.dim), d = a.dim + i % (dp - a.dim);
            qs[t * pk + d] = ks[t * pk + d] = gs[t * pk + d] = 0.f;
        }
        for (int i = tid; i < kC * (a.vdim_pad - a.vdim); i += 256) {
            const int t = i / (a.vdim_pad - a.vdim), v = a.vdim + i % (a.vdim_pad - a.vdim);
            vs[t * pv + v] = 0.f;
        }
    } else {
        auto row_of = [&](int64_t p) { return (int64_t)c.row0 + (p - c.pos0); };
        for (int i = tid; i < kC * dp; i += 256) {
            const int t = i / dp, d = i - t * dp;
            float q = 0.f, k = 0.f, g = 0.f;
            if (t < c.count && d < a.dim) {
                q = conv_silu(a, cq + d, c.pos0 + t, c.first_pos, c.slot, row_of);
                k = conv_silu(a, ck + d, c.pos0 + t, c.first_pos, c.slot, row_of);
                g = log2_decay(a, c.row0 + t, h, d, rate);
            }
            qs[t * pk + d] = q;
            ks[t * pk + d] = k;
            gs[t * pk + d] = g;
        }
        for (int i = tid; i < kC * a.vdim_pad; i += 256) {
            const int t = i / a.vdim_pad, v = i - t * a.vdim_pad;
            vs[t * pv + v] = t < c.count && v < a.vdim ? conv_silu(a, cv + v, c.pos0 + t, c.first_pos, c.slot, row_of) : 0.f;
        }
    }
    if (tid < kC) bs[tid] = tid < c.count ? sigmoid_f((float)a.proj[(int64_t)(c.row0 + tid) * a.proj_stride + a.beta_off + h]) : 0.f;
    __syncthreads();

    const int i = tid >> 4, j = tid & 15;
    int strong = 0;
    for (int d = tid; d < dp; d += 256) {
        float sum = 0.f;
#pragma unroll
        for (int t = 0; t < kC; ++t) {
            sum += gs[t * pk + d];
            gs[t * pk + d] = sum;
        }
        gl[d] = sum;
        strong |= sum < -kSplitRange;
    }
    {
        float sk = 0.f, sq = 0.f;
        for (int d = 4 * j; d < dp; d += 64) {
            const f32x4_t k = *reinterpret_cast<const f32x4_t*>(ks + i * pk + d), q = *reinterpret_cast<const f32x4_t*>(qs + i * pk + d);
#pragma unroll
            for (int e = 0; e < 4; ++e) { sk += k[e] * k[e]; sq += q[e] * q[e]; }
        }
#pragma unroll
        for (int m = 8; m >= 1; m >>= 1) { sk += __shfl_xor(sk, m, 64); sq += __shfl_xor(sq, m, 64); }
        if (j == 0) { inv[i] = rsqrtf(sk + 1e-6f); inv[16 + i] = rsqrtf(sq + 1e-6f) * a.q_scale; }
    }
    strong = __syncthreads_or(strong);
    float akk = 0.f, aqk = 0.f;                    // products of token pair (i, j), before the lengths
    if (strong && j <= i) {
        // some channel decays so much over the chunk that only differences of G can be exponentiated
        const float *ki = ks + i * pk, *qi = qs + i * pk, *gi = gs + i * pk, *kj = ks + j * pk, *gj = gs + j * pk;
        for (int d = 0; d < dp; d += 4) {
            const f32x4_t k1 = *reinterpret_cast<const f32x4_t*>(ki + d), q1 = *reinterpret_cast<const f32x4_t*>(qi + d);
            const f32x4_t g1 = *reinterpret_cast<const f32x4_t*>(gi + d), k2 = *reinterpret_cast<const f32x4_t*>(kj + d);
            const f32x4_t g2 = *reinterpret_cast<const f32x4_t*>(gj + d);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float w = k2[e] * __builtin_amdgcn_exp2f(g1[e] - g2[e]);
                akk += k1[e] * w;
                aqk += q1[e] * w;
            }
        }
    }
    if (strong) __syncthreads();
    for (int x = tid; x < kC * (dp / 4); x += 256) {
        const int t = x / (dp / 4), d = 4 * (x - t * (dp / 4));
        f32x4_t* g = reinterpret_cast<f32x4_t*>(gs + t * pk + d);
        f32x4_t* k = reinterpret_cast<f32x4_t*>(ks + t * pk + d);
        f32x4_t* q = reinterpret_cast<f32x4_t*>(qs + t * pk + d);
        const f32x4_t last = *reinterpret_cast<const f32x4_t*>(gl + d);
        f32x4_t gv = *g, kv = *k, qv = *q;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float up = __builtin_amdgcn_exp2f(gv[e]);
            gv[e] = kv[e] * __builtin_amdgcn_exp2f(last[e] - gv[e]);
            kv[e] *= up;
            qv[e] *= up;
        }
        *g = gv; *k = kv; *q = qv;
    }
    __syncthreads();
    const int lq = lane >> 4, lm = lane & 15;
    if (!strong) {
        // A_ij = sum_d (k_i e^{G_i - G_last}) (k_j e^{G_last - G_j}) on the matrix pipe: wavefronts 0 and 1 take half of the
        // channels each, 2 and 3 do the same for q
        f32x4_t acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = acc0;
        const float* left = (wave < 2 ? ks : qs) + lm * pk;
        for (int t = wave & 1; t < dp / 16; t += 2) {
            const int d = 16 * t + 4 * lq;
            const f32x4_t x1 = *reinterpret_cast<const f32x4_t*>(left + d), last = *reinterpret_cast<const f32x4_t*>(gl + d);
            const f32x4_t k2 = *reinterpret_cast<const f32x4_t*>(gs + lm * pk + d);
#pragma unroll
            for (int e = 0; e < 4; e += 2) {
                acc0 = __builtin_amdgcn_mfma_f32_16x16x4f32(x1[e] * __builtin_amdgcn_exp2f(-last[e]), k2[e], acc0, 0, 0, 0);
                acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(x1[e + 1] * __builtin_amdgcn_exp2f(-last[e + 1]), k2[e + 1], acc1, 0, 0, 0);
            }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) pp[wave * 256 + (4 * lq + e) * 16 + lm] = acc0[e] + acc1[e];    // row: token i, column: token j
        __syncthreads();
        akk = pp[tid] + pp[256 + tid];
        aqk = pp[512 + tid] + pp[768 + tid];
    }
    lt[j * 20 + i] = j < i ? bs[i] * akk * inv[i] * inv[j] : 0.f;
    rec[48 * dp + ((j >> 2) * 16 + i) * 4 + (j & 3)] = j <= i ? aqk * inv[16 + i] * inv[j] : 0.f;
    __syncthreads();
    if (wave == 0) {
        // T = (I + L)^-1 column by column: lane m holds column m, row s is final when it is used
        float t[kC];
#pragma unroll
        for (int r = 0; r < kC; ++r) t[r] = r == lm ? 1.f : 0.f;
#pragma unroll
        for (int s = 0; s < kC - 1; ++s)
#pragma unroll
            for (int r4 = 0; r4 < kC; r4 += 4)
                if (r4 + 3 > s) {
                    const f32x4_t l = *reinterpret_cast<const f32x4_t*>(lt + s * 20 + r4);      // zero for rows up to s
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (r4 + e > s) t[r4 + e] -= l[e] * t[s];
                }
        if (lane < kC) {
            const float b = bs[lm];
#pragma unroll
            for (int r = 0; r < kC; ++r) tb[r * 20 + lm] = t[r] * b;
        }
    } else {
        const float iq = inv[16 + lm];
        f32x4_t ik;
#pragma unroll
        for (int e = 0; e < 4; ++e) ik[e] = inv[4 * lq + e];
        for (int t = wave - 1; t < dp / 16; t += 3) {
            f32x4_t q = *reinterpret_cast<const f32x4_t*>(qs + lm * pk + 16 * t + 4 * lq), k;
            q *= iq;
#pragma unroll
            for (int e = 0; e < 4; ++e) k[e] = gs[(4 * lq + e) * pk + 16 * t + lm] * ik[e];
            *reinterpret_cast<f32x4_t*>(rec + 16 * dp + 256 * t + 4 * lane) = q;
            *reinterpret_cast<f32x4_t*>(rec + 32 * dp + 256 * t + 4 * lane) = k;
        }
        for (int d = tid - 64; d < dp; d += 192) rec[48 * dp + 256 + d] = __builtin_amdgcn_exp2f(gl[d]);
    }
    __syncthreads();
    const f32x4_t tv = *reinterpret_cast<const f32x4_t*>(tb + lm * 20 + 4 * lq);       // T beta, row lm
    for (int t = wave; t < dp / 16; t += 4) {      // W^T = (e^G K)^T (T beta)^T: row d, column i
        f32x4_t w = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < 4; ++e)
            w = __builtin_amdgcn_mfma_f32_16x16x4f32(ks[(4 * lq + e) * pk + 16 * t + lm] * inv[4 * lq + e], tv[e], w, 0, 0, 0);
        *reinterpret_cast<f32x4_t*>(rec + 256 * t + 4 * lane) = w;
    }
    float* uv = rec + 49 * dp + 256;
    for (int t = wave; t < a.vdim_pad / 16; t += 4) {
        f32x4_t w = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < 4; ++e) w = __builtin_amdgcn_mfma_f32_16x16x4f32(tv[e], vs[(4 * lq + e) * pv + 16 * t + lm], w, 0, 0, 0);
        *reinterpret_cast<f32x4_t*>(uv + 256 * t + 4 * lane) = w;
    }
}

// The same for bf16 heads of dim = vdim = 16 DT and four taps.  A record of 34 KB and 8 KB of inputs for a chunk and head of 128 pass through memory, which
// bounds it (4.6 TB/s; without the records' way to memory the call takes 66 us less).  The general form is bound by how long a chunk takes, of which four
// fit a compute unit: here three wavefronts convolve while the fourth does the gates and adds them up token by token in registers, the lengths of k and q
// come out of the pass that scales them, and sizes are constants.  8 portions of 500 to 2600 tokens, 32 heads of 128: the call 807 -> 735 us.  (Two, four
// or eight chunks one after the other in a workgroup, the next one's inputs requested ahead: 744, 752, 769.)
template <int DT>
__global__ void __launch_bounds__(256, 4) delta_prep_square_kernel(DeltaArgs<__bf16> a, const ChunkDesc* chunks, float* records) {
    constexpr int D = 16 * DT, P = D + 4, ND = D / 4, kConv = 6 * ND, CD = D / 64;      // CD: channels of a lane of the fourth wavefront
    static_assert(DT == 4 || DT == 8, "lanes of the gates, items of the convolution, halves of a wavefront per token");
    extern __shared__ __attribute__((aligned(16))) float sh[];
    float* qs = sh;                    // [16][P] q, then e^G q / |q|
    float* ks = qs + kC * P;           // [16][P] k, then e^G k / |k|
    float* gs = ks + kC * P;           // [16][P] running log2 decay G, then e^{G_last - G} k / |k|
    float* vs = gs + kC * P;           // [16][P]
    float* pp = vs + kC * P;           // [2][2][256] products of the token pairs (k k, q k), in two parts each
    float* lt = pp + 1024;             // [16][20] column s: beta * A of the tokens behind s
    float* tb = lt;                    // [16][20] T * beta, when those have been used
    float* gl = lt + kC * 20;          // [D] G_last
    float* gi = gl + D;                // [D] e^{-G_last}
    float* inv = gi + D;               // [2][16] 1 / length of k and q
    float* bs = inv + 32;              // [16] beta
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), h = blockIdx.y;
    const int lq = lane >> 4, lm = lane & 15, i = tid >> 4, j = tid & 15;
    const ChunkDesc c = chunks[blockIdx.x];
    const int row0 = c.count > 0 ? c.row0 : 0;                   // the gates of an empty chunk read row 0, which exists, and use nothing of it
    float* rec = records + ((int64_t)blockIdx.x * a.heads + h) * record_floats(D, D);
    const int group = a.heads / a.kv_heads, kvh = h / group;
    const float rate = expf(a.a_log[h]);
    const bool gates = wave == 3;
    // item of the convolution: matrix, four channels, half of the tokens
    const int item = tid < kConv ? tid : 0, t0 = 8 * (item / (3 * ND)), matrix = item / ND % 3, col = 4 * (item % ND);
    const int channel = col + (matrix == 0 ? kvh * D : matrix == 1 ? (a.kv_heads + kvh) * D : 2 * a.kv_heads * D + h * D);
    float* const conv_to = (matrix == 0 ? qs : matrix == 1 ? ks : vs) + t0 * P + col;
    const int d0 = CD * lane;
    float w[4][4], dt[CD];
#pragma unroll
    for (int e = 0; e < 4; ++e) load_elems<4>(a.conv + 4 * (channel + e), w[e]);
#pragma unroll
    for (int e = 0; e < CD; ++e) dt[e] = a.dt_bias[h * D + d0 + e];

    // Inputs: of the convolution tokens t0 - 3 .. t0 + 7, of the gates 16 tokens and a logit of the write strength
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    u32x2 raw[11];
    if (gates) {
        const __bf16* src = a.decay + (int64_t)row0 * a.decay_stride + h * D + d0;
        const int last = c.count > 0 ? c.count - 1 : 0;      // tokens behind the last one re-read it
#pragma unroll
        for (int t = 0; t < kC; ++t) {
            const __bf16* p = src + (t < last ? t : last) * a.decay_stride;
            raw[t / 2][t & 1] = CD == 2 ? *reinterpret_cast<const uint32_t*>(p) : *reinterpret_cast<const uint16_t*>(p);
        }
        raw[8][0] = *reinterpret_cast<const uint16_t*>(a.proj + (int64_t)(row0 + ((lane & 15) < last ? lane & 15 : last)) * a.proj_stride + a.beta_off + h);
    } else if (c.count == kC && c.pos0 - 3 >= c.first_pos) {
        const __bf16* src = a.proj + (int64_t)(row0 + t0 - 3) * a.proj_stride + channel;
#pragma unroll
        for (int x = 0; x < 11; ++x, src += a.proj_stride) raw[x] = *reinterpret_cast<const u32x2*>(src);
    } else {
#pragma unroll
        for (int x = 0; x < 11; ++x) {
            const int t = t0 + x - 3;
            const WindowRow from = window_row(c.count, c.pos0, c.first_pos, t);
            raw[x] = u32x2{0u, 0u};
            if (from != WindowRow::kNone)
                raw[x] = *reinterpret_cast<const u32x2*>(from == WindowRow::kBatch ? a.proj + (int64_t)(row0 + t) * a.proj_stride + channel
                                                                                   : a.ring + ((int64_t)c.slot * 4 + ((c.pos0 + t) & 3)) * a.channels + channel);
        }
    }
    int strong = 0;
    if (gates) {
        float sum[CD];
#pragma unroll
        for (int e = 0; e < CD; ++e) sum[e] = 0.f;
#pragma unroll
        for (int t = 0; t < kC; ++t)
#pragma unroll
            for (int e = 0; e < CD; ++e) {
                const uint32_t bits = raw[t / 2][t & 1];
                const float z = __builtin_bit_cast(float, e == 1 ? bits & 0xffff0000u : bits << 16) + dt[e], g = -rate * softplus_log2(z);
                sum[e] += t < c.count ? g : 0.f;
                gs[t * P + d0 + e] = sum[e];
            }
#pragma unroll
        for (int e = 0; e < CD; ++e) {
            gl[d0 + e] = sum[e];
            gi[d0 + e] = __builtin_amdgcn_exp2f(-sum[e]);
            strong |= sum[e] < -kSplitRange;
        }
        if (lane < kC) bs[lane] = lane < c.count ? sigmoid_f(__builtin_bit_cast(float, raw[8][0] << 16)) : 0.f;
    } else if (tid < kConv) {
        float x[4][4];                             // rows of the window, each in its place for four tokens
        auto widen_row = [&](int r) {
#pragma unroll
            for (int e = 0; e < 4; ++e) x[r & 3][e] = __builtin_bit_cast(float, e & 1 ? raw[r][e / 2] & 0xffff0000u : raw[r][e / 2] << 16);
        };
#pragma unroll
        for (int r = 0; r < 3; ++r) widen_row(r);
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            widen_row(t + 3);
            f32x4_t y;
            const bool in = t0 + t < c.count;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float s = 0.f;
#pragma unroll
                for (int k = 0; k < 4; ++k) s += w[e][k] * x[(t + k) & 3][e];
                y[e] = in ? silu_f(s) : 0.f;
            }
            *reinterpret_cast<f32x4_t*>(conv_to + t * P) = y;
            if (t & 1) __builtin_amdgcn_sched_barrier(0);
        }
    }
    strong = __syncthreads_or(strong);
    float akk = 0.f, aqk = 0.f;                    // products of token pair (i, j)
    if (strong) {
        if (j <= i) {
            // some channel decays so much over the chunk that only differences of G can be exponentiated
            const float *ki = ks + i * P, *qi = qs + i * P, *gi_ = gs + i * P, *kj = ks + j * P, *gj = gs + j * P;
            for (int d = 0; d < D; d += 4) {
                const f32x4_t k1 = *reinterpret_cast<const f32x4_t*>(ki + d), q1 = *reinterpret_cast<const f32x4_t*>(qi + d);
                const f32x4_t g1 = *reinterpret_cast<const f32x4_t*>(gi_ + d), k2 = *reinterpret_cast<const f32x4_t*>(kj + d);
                const f32x4_t g2 = *reinterpret_cast<const f32x4_t*>(gj + d);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float v = k2[e] * __builtin_amdgcn_exp2f(g1[e] - g2[e]);
                    akk += k1[e] * v;
                    aqk += q1[e] * v;
                }
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int x = 0; x < kC * ND / 256; ++x) {      // ND lanes side by side hold a token
        const int t = (tid + 256 * x) / ND, d = 4 * (tid % ND);
        f32x4_t* gp = reinterpret_cast<f32x4_t*>(gs + t * P + d);
        f32x4_t* kp = reinterpret_cast<f32x4_t*>(ks + t * P + d);
        f32x4_t* qp = reinterpret_cast<f32x4_t*>(qs + t * P + d);
        const f32x4_t last = *reinterpret_cast<const f32x4_t*>(gl + d);
        f32x4_t g = *gp, k = *kp, q = *qp;
        float sk = (k[0] * k[0] + k[1] * k[1]) + (k[2] * k[2] + k[3] * k[3]), sq = (q[0] * q[0] + q[1] * q[1]) + (q[2] * q[2] + q[3] * q[3]);
        sk = lanes_sum<ND>(sk);
        sq = lanes_sum<ND>(sq);
        const float ik = rsqrtf(sk + 1e-6f), iq = rsqrtf(sq + 1e-6f) * a.q_scale;
        if (tid % ND == 0) { inv[t] = ik; inv[16 + t] = iq; }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float up = __builtin_amdgcn_exp2f(g[e]), kn = k[e] * ik;
            g[e] = kn * __builtin_amdgcn_exp2f(last[e] - g[e]);
            k[e] = kn * up;
            q[e] *= up * iq;
        }
        *gp = g; *kp = k; *qp = q;
    }
    __syncthreads();
    if (!strong) {
        // A_ij = sum_d (k_i e^{G_i - G_last}) (k_j e^{G_last - G_j}) on the matrix pipe: wavefronts 0 and 1 take half of the
        // channels each, 2 and 3 do the same for q
        f32x4_t acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = acc0;
        const float* left = (wave < 2 ? ks : qs) + lm * P;
#pragma unroll
        for (int x = 0; x < DT / 2; ++x) {
            const int d = 16 * (2 * x + (wave & 1)) + 4 * lq;
            const f32x4_t x1 = *reinterpret_cast<const f32x4_t*>(left + d) * *reinterpret_cast<const f32x4_t*>(gi + d);
            const f32x4_t k2 = *reinterpret_cast<const f32x4_t*>(gs + lm * P + d);
#pragma unroll
            for (int e = 0; e < 4; e += 2) {
                acc0 = __builtin_amdgcn_mfma_f32_16x16x4f32(x1[e], k2[e], acc0, 0, 0, 0);
                acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(x1[e + 1], k2[e + 1], acc1, 0, 0, 0);
            }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) pp[wave * 256 + (4 * lq + e) * 16 + lm] = acc0[e] + acc1[e];    // row: token i, column: token j
        __syncthreads();
        akk = pp[tid] + pp[256 + tid];
        aqk = pp[512 + tid] + pp[768 + tid];
    } else {
        akk *= inv[i] * inv[j];
        aqk *= inv[16 + i] * inv[j];
    }
    lt[j * 20 + i] = j < i ? bs[i] * akk : 0.f;
    rec[48 * D + ((j >> 2) * 16 + i) * 4 + (j & 3)] = j <= i ? aqk : 0.f;
    __syncthreads();
    if (wave == 0) {
        // T = (I + L)^-1 column by column: lane m holds column m, row s is final when it is used
        float t[kC];
#pragma unroll
        for (int r = 0; r < kC; ++r) t[r] = r == lm ? 1.f : 0.f;
#pragma unroll
        for (int s = 0; s < kC - 1; ++s)
#pragma unroll
            for (int r4 = 0; r4 < kC; r4 += 4)
                if (r4 + 3 > s) {
                    const f32x4_t l = *reinterpret_cast<const f32x4_t*>(lt + s * 20 + r4);      // zero for rows up to s
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (r4 + e > s) t[r4 + e] -= l[e] * t[s];
                }
        if (lane < kC) {
            const float b = bs[lm];
#pragma unroll
            for (int r = 0; r < kC; ++r) tb[r * 20 + lm] = t[r] * b;
        }
    } else {
        for (int t = wave - 1; t < DT; t += 3) {
            f32x4_t k;
#pragma unroll
            for (int e = 0; e < 4; ++e) k[e] = gs[(4 * lq + e) * P + 16 * t + lm];
            *reinterpret_cast<f32x4_t*>(rec + 16 * D + 256 * t + 4 * lane) = *reinterpret_cast<const f32x4_t*>(qs + lm * P + 16 * t + 4 * lq);
            *reinterpret_cast<f32x4_t*>(rec + 32 * D + 256 * t + 4 * lane) = k;
        }
        if (tid - 64 < D) rec[48 * D + 256 + tid - 64] = __builtin_amdgcn_exp2f(gl[tid - 64]);
    }
    __syncthreads();
    const f32x4_t tv = *reinterpret_cast<const f32x4_t*>(tb + lm * 20 + 4 * lq);       // T beta, row lm
#pragma unroll
    for (int x = 0; x < DT / 4; ++x) {             // W^T = (e^G K)^T (T beta)^T: row d, column i; T beta V
        const int t = 4 * x + wave;
        f32x4_t wt = {0.f, 0.f, 0.f, 0.f}, vt = wt;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            wt = __builtin_amdgcn_mfma_f32_16x16x4f32(ks[(4 * lq + e) * P + 16 * t + lm], tv[e], wt, 0, 0, 0);
            vt = __builtin_amdgcn_mfma_f32_16x16x4f32(tv[e], vs[(4 * lq + e) * P + 16 * t + lm], vt, 0, 0, 0);
        }
        *reinterpret_cast<f32x4_t*>(rec + 256 * t + 4 * lane) = wt;
        *reinterpret_cast<f32x4_t*>(rec + 49 * D + 256 + 256 * t + 4 * lane) = vt;
    }
}

// Wavefront w of workgroup x owns state columns 16 (x * waves + w) .. + 15: DT accumulator tiles of 16 rows, lane (q, m)
// holding rows 16 t + 4 q + r of column m.  That is also the layout of the second operand of the next product, whose
// first operand the records hold in fragment order.
template <int DT>
__global__ void __launch_bounds__(256) delta_scan_kernel(const PortionDesc* portions, const ChunkDesc* chunks, const float* records,
                                                         float* state, float* o, int heads, int vdim_pad, Turns turns) {
    constexpr int dp = 16 * DT;
    constexpr int kShared = 48 * dp + 256 + dp;                  // floats of a record all wavefronts read
    extern __shared__ __attribute__((aligned(16))) float sh[];   // [2][kShared]
    const int tid = threadIdx.x, threads = blockDim.x, lane = tid & 63, wave = tid >> 6;
    const int q = lane >> 4, m = lane & 15;
    const int h = blockIdx.y;
    const PortionDesc p = portions[portion_of_turn(&portions->chunk0, turns, blockIdx.z)];
    const int vt = blockIdx.x * (threads >> 6) + wave;
    const bool live = vt < vdim_pad / 16;
    const int64_t rec_len = record_floats(dp, vdim_pad);
    float* sp = state + (((int64_t)p.slot * heads + h) * dp) * vdim_pad + 16 * vt + m;
    f32x4_t s[DT];
#pragma unroll
    for (int t = 0; t < DT; ++t) {
        s[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        if (live && p.pos0 > 0)
#pragma unroll
            for (int r = 0; r < 4; ++r) s[t][r] = sp[(int64_t)(16 * t + 4 * q + r) * vdim_pad];
    }
    constexpr int kVecs = kShared / 4;
    constexpr int kMaxStage = (kVecs + 63) / 64;                 // chunks of 16 bytes per thread of a one-wavefront workgroup
    constexpr int kStage = kMaxStage < 8 ? kMaxStage : 8;        // kept in registers; the rest goes straight to LDS
    f32x4_t stage[kStage];
    auto fetch = [&](int c) {
        const f32x4_t* src = reinterpret_cast<const f32x4_t*>(records + ((int64_t)(p.chunk0 + c) * heads + h) * rec_len);
#pragma unroll
        for (int i = 0; i < kStage; ++i)
            if (tid + i * threads < kVecs) stage[i] = src[tid + i * threads];
    };
    auto put = [&](int c, float* buf) {
        f32x4_t* dst = reinterpret_cast<f32x4_t*>(buf);
#pragma unroll
        for (int i = 0; i < kStage; ++i)
            if (tid + i * threads < kVecs) dst[tid + i * threads] = stage[i];
        const f32x4_t* src = reinterpret_cast<const f32x4_t*>(records + ((int64_t)(p.chunk0 + c) * heads + h) * rec_len);
        for (int i = tid + kStage * threads; i < kVecs; i += threads) dst[i] = src[i];
    };
    fetch(0);
    put(0, sh);
    __syncthreads();
    for (int c = 0; c < p.chunks; ++c) {
        const float* buf = sh + (c & 1) * kShared;
        const float* rec = records + ((int64_t)(p.chunk0 + c) * heads + h) * rec_len;
        f32x4_t u = {0.f, 0.f, 0.f, 0.f};
        if (live) u = *reinterpret_cast<const f32x4_t*>(rec + kShared + vt * 256 + 4 * lane);
        if (c + 1 < p.chunks) fetch(c + 1);
        const float* fr = buf + 4 * lane;
        f32x4_t ws0 = {0.f, 0.f, 0.f, 0.f}, ws1 = ws0, o0 = ws0, o1 = ws0;
#pragma unroll
        for (int t = 0; t < DT; ++t) {
            const f32x4_t w = *reinterpret_cast<const f32x4_t*>(fr + 256 * t);
            const f32x4_t qv = *reinterpret_cast<const f32x4_t*>(fr + 16 * dp + 256 * t);
#pragma unroll
            for (int r = 0; r < 4; r += 2) {
                ws0 = __builtin_amdgcn_mfma_f32_16x16x4f32(w[r], s[t][r], ws0, 0, 0, 0);
                o0 = __builtin_amdgcn_mfma_f32_16x16x4f32(qv[r], s[t][r], o0, 0, 0, 0);
                ws1 = __builtin_amdgcn_mfma_f32_16x16x4f32(w[r + 1], s[t][r + 1], ws1, 0, 0, 0);
                o1 = __builtin_amdgcn_mfma_f32_16x16x4f32(qv[r + 1], s[t][r + 1], o1, 0, 0, 0);
            }
        }
        u = u - (ws0 + ws1);
        const f32x4_t b = *reinterpret_cast<const f32x4_t*>(fr + 48 * dp);
#pragma unroll
        for (int r = 0; r < 4; ++r) o0 = __builtin_amdgcn_mfma_f32_16x16x4f32(b[r], u[r], o0, 0, 0, 0);
        const float* e = buf + 48 * dp + 256 + 4 * q;
#pragma unroll
        for (int t = 0; t < DT; ++t) {
            const f32x4_t k = *reinterpret_cast<const f32x4_t*>(fr + 32 * dp + 256 * t);
            s[t] *= *reinterpret_cast<const f32x4_t*>(e + 16 * t);
#pragma unroll
            for (int r = 0; r < 4; ++r) s[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[r], u[r], s[t], 0, 0, 0);
        }
        if (live) {
            const ChunkDesc d = chunks[p.chunk0 + c];
            const f32x4_t ov = o0 + o1;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (4 * q + r < d.count) o[((int64_t)(d.row0 + 4 * q + r) * heads + h) * vdim_pad + 16 * vt + m] = ov[r];
        }
        if (c + 1 < p.chunks) put(c + 1, sh + ((c + 1) & 1) * kShared);
        __syncthreads();
    }
    if (live)
#pragma unroll
        for (int t = 0; t < DT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) sp[(int64_t)(16 * t + 4 * q + r) * vdim_pad] = s[t][r];
}

// hi + mid + lo = x exactly, two floats at a time, hi and mid rounded to nearest, so that residuals have both signs: |mid| <= 2^-8 and
// |lo| <= 2^-17 of x's power of two (a float past the largest bf16, 3.39e38, is infinite).  A residual is one dot product with (-1, 0) or (0, -1) instead of a mask and a subtraction
// (829 -> 797 us with 8 x 500 .. 2600 tokens of 32 heads).  A pair lies along the sum that both enter, so an infinity spoils no other sum.
template <int N>
__device__ __forceinline__ void split3(const float (&x)[N], uint32_t (&p)[3][N / 2]) {
    typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
    uint32_t c0 = 0x0000bf80u, c1 = 0xbf800000u;       // (-1, 0) and (0, -1)
    asm("" : "+s"(c0), "+s"(c1));                      // in registers: as an inline constant the compiler writes -1.0, which is another pair
    const bf16x2_t first = __builtin_bit_cast(bf16x2_t, c0), second = __builtin_bit_cast(bf16x2_t, c1);
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
        p[0][i] = round_pack(x[2 * i], x[2 * i + 1]);
        const bf16x2_t hi = __builtin_bit_cast(bf16x2_t, p[0][i]);
        const float a = __builtin_amdgcn_fdot2_f32_bf16(hi, first, x[2 * i], false), b = __builtin_amdgcn_fdot2_f32_bf16(hi, second, x[2 * i + 1], false);
        p[1][i] = round_pack(a, b);
        const bf16x2_t mid = __builtin_bit_cast(bf16x2_t, p[1][i]);
        p[2][i] = pack(__builtin_amdgcn_fdot2_f32_bf16(mid, first, a, false), __builtin_amdgcn_fdot2_f32_bf16(mid, second, b, false));
    }
}

// Operands of products over 16 (tokens, or rows of the state) as pieces, two along the sum: six products of pieces are three instructions.
struct LeftPieces {
    bf16x8_t hm, hl;
    LeftPieces() = default;
    __device__ __forceinline__ explicit LeftPieces(f32x4_t x) {
        const float f[4] = {x[0], x[1], x[2], x[3]};
        uint32_t p[3][2];
        split3<4>(f, p);
        hm = __builtin_bit_cast(bf16x8_t, u32x4_t{p[0][0], p[0][1], p[1][0], p[1][1]});
        hl = __builtin_bit_cast(bf16x8_t, u32x4_t{p[0][0], p[0][1], p[2][0], p[2][1]});
    }
};
struct RightPieces {
    bf16x8_t hh, mm, lh;
    RightPieces() = default;
    __device__ __forceinline__ explicit RightPieces(f32x4_t x) {
        const float f[4] = {x[0], x[1], x[2], x[3]};
        uint32_t p[3][2];
        split3<4>(f, p);
        hh = __builtin_bit_cast(bf16x8_t, u32x4_t{p[0][0], p[0][1], p[0][0], p[0][1]});
        mm = __builtin_bit_cast(bf16x8_t, u32x4_t{p[1][0], p[1][1], p[1][0], p[1][1]});
        lh = __builtin_bit_cast(bf16x8_t, u32x4_t{p[2][0], p[2][1], p[0][0], p[0][1]});
    }
};
struct PieceSums {
    f32x4_t large = {0.f, 0.f, 0.f, 0.f}, middle = large, small = large;
    __device__ __forceinline__ void add(const LeftPieces& a, const RightPieces& b) {
        small = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.hl, b.lh, small, 0, 0, 0);
        middle = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.hm, b.mm, middle, 0, 0, 0);
        large = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.hm, b.hh, large, 0, 0, 0);
    }
    __device__ __forceinline__ f32x4_t sum() const { return large + (middle + small); }
};

// Few (portion, head) pairs: what counts is how long a chunk takes, and there are compute units enough for every 16 CT columns of a head to have one.
// Wavefront w of NW owns RT tiles of 16 rows of the state (w RT + r) and brings their parts of the records straight into registers, PD chunks ahead; what
// the products with all rows need, S^T K and S^T Q of a chunk, is added up through LDS, one barrier a chunk.  Two more wavefronts, each for every other
// chunk, bring V and B and finish the outputs, so that nobody else stores anything.  Workgroups of a pair lie on one die and walk its records side by side, so
// that these come from memory once.  Products as in delta_scan_wide_kernel, the state's sums by the vector unit.
// A chunk takes 1.0 us with one tile, 1.3 with two and 2.1 with four (delta_scan_kernel: 2.5 and more), of which the loads are nothing (the same record again and
// again: 3 % less), the products of S^T Q 13 % although they run while U is under way.  One portion of 2000 tokens, 32 heads of 128 x 128: the scan 262 -> 131 us under
// a profiler, the call 382 -> 184.  With float products 186 (one tile), 408 instead of 323 (four); one wavefront for the outputs 200; eight wavefronts of one
// row tile each 187.
template <int DT, int CT>
struct SlabSizes {
    static constexpr int RT = DT >= 8 ? 2 : 1, NW = DT / RT, PD = CT == 4 ? 2 : 3, threads = 64 * (NW + 2);
    static constexpr int lds = 2 * (2 * NW + 1) * CT * 1024;
};
template <int DT, int CT>
__global__ void __launch_bounds__((SlabSizes<DT, CT>::threads)) delta_scan_slab_kernel(const PortionDesc* portions, const ChunkDesc* chunks, const float* records,
                                                                                          float* state, float* o, int heads, int vdim_pad, int pairs, int slabs) {
    using Z = SlabSizes<DT, CT>;
    constexpr int dp = 16 * DT, RT = Z::RT, NW = Z::NW, PD = Z::PD;
    extern __shared__ __attribute__((aligned(16))) f32x4_t slab_lds[];
    f32x4_t* parts = slab_lds;                                  // [2][NW + 1][CT][64]: of S^T K, the last one -V
    f32x4_t* outs = slab_lds + 2 * (NW + 1) * CT * 64;          // [2][NW][CT][64]: of S^T Q
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), q = lane >> 4, m = lane & 15;
    const int die = blockIdx.x & 7, turn = blockIdx.x >> 3, pair = turn / slabs * 8 + die, slab = turn % slabs;
    if (pair >= pairs) return;
    const PortionDesc p = portions[pair / heads];
    const int h = pair % heads, vt0 = slab * CT, tiles = vdim_pad / 16;
    const int64_t rec_len = record_floats(dp, vdim_pad), rec_step = (int64_t)heads * rec_len;
    const float* rec = records + ((int64_t)p.chunk0 * heads + h) * rec_len;
    auto record = [&](int c) { return rec + (c < p.chunks ? c : p.chunks - 1) * rec_step; };
    auto part = [&](int c, int w, int t) -> f32x4_t& { return parts[(((c & 1) * (NW + 1) + w) * CT + t) * 64 + lane]; };
    auto out = [&](int c, int w, int t) -> f32x4_t& { return outs[(((c & 1) * NW + w) * CT + t) * 64 + lane]; };
    auto update = [&](int c, int t) {                           // U: V - S^T K
        f32x4_t u = part(c, NW, t);
#pragma unroll
        for (int w = 0; w < NW; ++w) u += part(c, w, t);
        return -u;
    };
    if (wave < NW) {
        f32x4_t s[RT][CT];
        auto state_at = [&](int r, int t, int e) {
            return state + (((int64_t)p.slot * heads + h) * dp + 16 * (wave * RT + r) + 4 * q + e) * vdim_pad + 16 * (vt0 + t) + m;
        };
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int t = 0; t < CT; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e) s[r][t][e] = p.pos0 > 0 && vt0 + t < tiles ? *state_at(r, t, e) : 0.f;
        if (p.chunks > 0) {
            struct Rows { f32x4_t w[RT], q[RT], k[RT], e[RT]; } ring[PD];
            auto request = [&](Rows& f, int c) {
                const float* src = record(c) + 256 * RT * wave + 4 * lane;
#pragma unroll
                for (int r = 0; r < RT; ++r) {
                    f.w[r] = *reinterpret_cast<const f32x4_t*>(src + 256 * r);
                    f.q[r] = *reinterpret_cast<const f32x4_t*>(src + 16 * dp + 256 * r);
                    f.k[r] = *reinterpret_cast<const f32x4_t*>(src + 32 * dp + 256 * r);
                    f.e[r] = *reinterpret_cast<const f32x4_t*>(record(c) + 48 * dp + 256 + 16 * (RT * wave + r) + 4 * q);
                }
            };
#pragma unroll
            for (int i = 0; i < PD; ++i) request(ring[i], i);
            LeftPieces w[RT], qv[RT], k[RT];
#pragma unroll
            for (int r = 0; r < RT; ++r) w[r] = LeftPieces(ring[0].w[r]);
            for (int c0 = 0; c0 < p.chunks; c0 += PD) {
#pragma unroll
                for (int i = 0; i < PD; ++i) {
                    const int c = c0 + i;
                    if (c >= p.chunks) break;
                    const Rows& f = ring[i];
                    RightPieces sp[RT][CT];
#pragma unroll
                    for (int t = 0; t < CT; ++t) {
#pragma unroll
                        for (int r = 0; r < RT; ++r) sp[r][t] = RightPieces(s[r][t]);
                        PieceSums x;
#pragma unroll
                        for (int r = 0; r < RT; ++r) x.add(w[r], sp[r][t]);
                        part(c, wave, t) = x.sum();
                    }
#pragma unroll
                    for (int r = 0; r < RT; ++r) {
                        qv[r] = LeftPieces(f.q[r]);
                        k[r] = LeftPieces(f.k[r]);
                    }
                    __syncthreads();
                    f32x4_t us[CT];
#pragma unroll
                    for (int t = 0; t < CT; ++t) us[t] = update(c, t);
#pragma unroll
                    for (int t = 0; t < CT; ++t) {
                        PieceSums y;
#pragma unroll
                        for (int r = 0; r < RT; ++r) y.add(qv[r], sp[r][t]);
                        out(c, wave, t) = y.sum();
                    }
#pragma unroll
                    for (int t = 0; t < CT; ++t) {
                        const RightPieces u(us[t]);
#pragma unroll
                        for (int r = 0; r < RT; ++r) {
                            PieceSums d;
                            d.add(k[r], u);
                            const f32x4_t ds = d.sum();
#pragma unroll
                            for (int e = 0; e < 4; ++e) s[r][t][e] = __builtin_fmaf(s[r][t][e], f.e[r][e], ds[e]);
                        }
                    }
#pragma unroll
                    for (int r = 0; r < RT; ++r) w[r] = LeftPieces(ring[(i + 1) % PD].w[r]);
                    request(ring[i], c + PD);
                }
            }
            __syncthreads();                                   // the last chunk's outputs
        }
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int t = 0; t < CT; ++t)
                if (vt0 + t < tiles)
#pragma unroll
                    for (int e = 0; e < 4; ++e) *state_at(r, t, e) = s[r][t][e];
    } else if (p.chunks > 0) {
        int zero = 0;
        asm volatile("" : "+v"(zero));                         // by the vector path: a scalar load in flight would be waited for with every read of LDS
        const int32_t* descs = &chunks[p.chunk0].row0 + zero;
        constexpr int kDesc = sizeof(ChunkDesc) / sizeof(int32_t), kRing = 2;
        struct Chunk { f32x4_t v[CT], b; int row0, count; } ring[kRing];
        auto request = [&](Chunk& f, int c) {
            const float* src = record(c);
#pragma unroll
            for (int t = 0; t < CT; ++t) f.v[t] = *reinterpret_cast<const f32x4_t*>(src + 49 * dp + 256 + 256 * (vt0 + t < tiles ? vt0 + t : 0) + 4 * lane);
            f.b = *reinterpret_cast<const f32x4_t*>(src + 48 * dp + 4 * lane);
            const int at = (c < p.chunks ? c : p.chunks - 1) * kDesc;
            f.row0 = descs[at];
            f.count = descs[at + 1];
        };
        const int64_t row_step = (int64_t)heads * vdim_pad;
        float* const column = o + (int64_t)h * vdim_pad + 16 * vt0 + m + 4 * q * row_step;
        f32x4_t y[CT];
        auto store = [&](const Chunk& f, int c) {
#pragma unroll
            for (int t = 0; t < CT; ++t)
#pragma unroll
                for (int w = 0; w < NW; ++w) y[t] += out(c, w, t);
            const int count = f.count - 4 * q;
            float* to = column + __builtin_amdgcn_readfirstlane(f.row0) * row_step;
#pragma unroll
            for (int e = 0; e < 4; ++e, to += row_step)
                if (e < count)
#pragma unroll
                    for (int t = 0; t < CT; ++t)
                        if (vt0 + t < tiles) to[16 * t] = y[t][e];
        };
        // Chunks of one parity: in front of its barrier -V, behind it the outputs, behind the next one their way out
        auto walk = [&](auto parity) {
            constexpr int kOdd = decltype(parity)::value;
#pragma unroll
            for (int i = 0; i < kRing; ++i) request(ring[i], 2 * i + kOdd);
            for (int c0 = 0; c0 < p.chunks; c0 += 2 * kRing)
#pragma unroll
                for (int i = 0; i < 2 * kRing; ++i) {
                    const int c = c0 + i;
                    if (c >= p.chunks) break;
                    if ((i & 1) == kOdd) {
#pragma unroll
                        for (int t = 0; t < CT; ++t) part(c, NW, t) = -ring[i / 2].v[t];
                    }
                    __syncthreads();
                    if ((i & 1) == kOdd) {
                        const LeftPieces b(ring[i / 2].b);
#pragma unroll
                        for (int t = 0; t < CT; ++t) {
                            PieceSums x;
                            x.add(b, RightPieces(update(c, t)));
                            y[t] = x.sum();
                        }
                    } else if (c > 0) {
                        Chunk& last = ring[(i + 2 * kRing - 1) / 2 % kRing];
                        store(last, c - 1);
                        request(last, c - 1 + 2 * kRing);
                    }
                }
            const int c = p.chunks - 1;
            __syncthreads();
            if ((c & 1) == kOdd) {
#pragma unroll
                for (int i = 0; i < kRing; ++i)
                    if (c / 2 % kRing == i) store(ring[i], c);
            }
        };
        if (wave == NW) walk(std::integral_constant<int, 0>{});
        else walk(std::integral_constant<int, 1>{});
    }
}

// A record in LDS: sums of three bf16 numbers, hi + mid + lo = the float exactly, so that the products run on the bf16 matrix pipe.  Of
// the nine products of two such sums six are added; the others, mid lo, lo mid and lo lo, are 2^-24 of the product at most, as much as a
// float product is rounded by, and of either sign.
struct WideBuffer {
    u32x4_t* p;
    int ks;
    __device__ __forceinline__ u32x4_t* wq(int which, int kk, int piece) const { return p + (((which * ks + kk) * 3 + piece) * 64); }
    __device__ __forceinline__ u32x4_t* k(int t, int form) const { return p + (6 * ks + 2 * t + form) * 64; }          // 0: [hi | mid], 1: [hi | lo]
    __device__ __forceinline__ u32x4_t* b(int form) const { return p + (10 * ks + form) * 64; }
    __device__ __forceinline__ u32x4_t* e() const { return p + (10 * ks + 2) * 64; }
};
__host__ __device__ constexpr int wide_buffer_units(int dt) { return 64 * (5 * dt + 2) + 4 * dt; }

// All columns of a head in one workgroup: eight wavefronts, of which `slabs` own 16 columns of the state each and all bring the next
// record to LDS, cut into pieces.  A chunk's outputs go through LDS to rows of a wavefront's half, which the next step norms and gates,
// so they do not pass through memory in between.
// A batch takes as long as its longest portion's chunks one after the other; a step of eight wavefronts on a compute unit is 3200 clocks
// of matrix pipe per wavefront with float products and 1200 with pieces, which cost about 180 vector instructions.  32 heads, 8 portions
// of 590 to 2560 tokens: scan, output and ring 662 us with delta_scan_kernel, 515 us here (kernels alone, under a profiler; the call 963 and
// 807 us).  What a step waits for is requested a step before, by every thread and without branches: with requests in branches, or
// stores between a request and its use, the compiler waits for everything in flight.  Tried as well, against 435 us of a first form: 830
// with such requests; float products for W S 690; the two wavefronts of a vector unit in opposite phases 550; four wavefronts that only
// serve eight that compute 460.
template <class T, int DT>
__global__ void __launch_bounds__(512, 2) delta_scan_wide_kernel(DeltaArgs<T> a, const PortionDesc* portions, const ChunkDesc* chunks,
                                                                 const float* records, int slabs, Turns turns) {
    constexpr int dp = 16 * DT, KS = DT / 2, kShared = 49 * dp + 256, kPitch = 132;
    extern __shared__ __attribute__((aligned(16))) u32x4_t lds[];     // [2] buffers, then outputs [2][16][kPitch]
    float* outputs = reinterpret_cast<float*>(lds + 2 * wide_buffer_units(DT));
    const int tid = threadIdx.x, lane = tid & 63, vt = __builtin_amdgcn_readfirstlane(tid >> 6), q = lane >> 4, m = lane & 15;
    const int h = blockIdx.x;
    const PortionDesc p = portions[portion_of_turn(&portions->chunk0, turns, blockIdx.y)];
    const bool live = vt < slabs;
    const int vdim_pad = a.vdim_pad;
    const int64_t rec_len = record_floats(dp, vdim_pad);
    const f32x4_t* rec = reinterpret_cast<const f32x4_t*>(records + ((int64_t)p.chunk0 * a.heads + h) * rec_len);
    const int64_t rec_step = (int64_t)a.heads * rec_len / 4;
    float* sp = a.state + (((int64_t)p.slot * a.heads + h) * dp) * vdim_pad + 16 * vt + m;
    f32x4_t s[DT];
#pragma unroll
    for (int t = 0; t < DT; ++t) {
        s[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        if (live && p.pos0 > 0)
#pragma unroll
            for (int r = 0; r < 4; ++r) s[t][r] = sp[(int64_t)(16 * t + 4 * q + r) * vdim_pad];
    }

    auto keep_state = [&] {
        if (!live) return;
#pragma unroll
        for (int t = 0; t < DT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) sp[(int64_t)(16 * t + 4 * q + r) * vdim_pad] = s[t][r];
    };
    if (p.chunks <= 0) return keep_state();            // an empty portion has no record to request

    // Every request is made by every thread, so that the compiler knows how many are in flight; what a thread has no use for is the
    // record's start.
    const int w_at = tid < 64 * DT ? (tid / (64 * KS)) * 4 * dp + ((tid >> 6) % KS) * 128 + lane : 0, k_at = tid < 64 * DT ? 8 * dp + tid : 0;
    const int b_at = tid < 64 + dp / 4 ? 12 * dp + tid : 0, v_at = live ? kShared / 4 + vt * 64 + lane : 0;
    f32x4_t w0, w1, kf, be, vn;
    auto fetch = [&](int c) {
        const f32x4_t* src = rec + (c < p.chunks ? c : p.chunks - 1) * rec_step;
        w0 = src[w_at];
        w1 = src[w_at + 64];
        kf = src[k_at];
        be = src[b_at];
        vn = src[v_at];
    };
    auto put = [&](int half) {
        const WideBuffer buf{lds + half * wide_buffer_units(DT), KS};
        auto two_forms = [&](f32x4_t x, u32x4_t* d0, u32x4_t* d1) {
            const float f[4] = {x[0], x[1], x[2], x[3]};
            uint32_t pc[3][2];
            split3<4>(f, pc);
            d0[lane] = u32x4_t{pc[0][0], pc[0][1], pc[1][0], pc[1][1]};
            d1[lane] = u32x4_t{pc[0][0], pc[0][1], pc[2][0], pc[2][1]};
        };
        if (DT == 8 || tid < 64 * DT) {
            const float f[8] = {w0[0], w0[1], w0[2], w0[3], w1[0], w1[1], w1[2], w1[3]};
            uint32_t pc[3][4];
            split3<8>(f, pc);
#pragma unroll
            for (int i = 0; i < 3; ++i) buf.wq(vt / KS, vt % KS, i)[lane] = u32x4_t{pc[i][0], pc[i][1], pc[i][2], pc[i][3]};
            two_forms(kf, buf.k(vt, 0), buf.k(vt, 1));
        }
        if (vt == 0) two_forms(be, buf.b(0), buf.b(1));
        else if (tid < 64 + dp / 4) buf.e()[tid - 64] = __builtin_bit_cast(u32x4_t, be);
    };
    auto mma = [](u32x4_t x, bf16x8_t y, f32x4_t acc) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, x), y, acc, 0, 0, 0); };

    // Rows 2 vt and 2 vt + 1 of a chunk's outputs, four columns per lane.  The gate is requested with the chunk, a step before it is used.
    const int out_row = 2 * vt + (lane >> 5), out_col = 4 * (lane & 31);
    const bool out_in = out_col < a.vdim;
    typedef T t4_t __attribute__((ext_vector_type(4)));
    t4_t gate;
    float norm[4];
    load_elems<4>(a.norm + (out_in ? out_col : 0), norm);
    const T* gates = a.gate + (int64_t)h * a.vdim + (out_in ? out_col : 0);
    T* outs = a.out + (int64_t)h * a.vdim + out_col;
    int done_row = 0, done_count = 0;
    const float inv_vdim = 1.f / (float)a.vdim;
    auto finish = [&](int half) {
        const f32x4_t x = *reinterpret_cast<const f32x4_t*>(outputs + (half * 16 + out_row) * kPitch + out_col);
        float ss = (x[0] * x[0] + x[1] * x[1]) + (x[2] * x[2] + x[3] * x[3]);
        ss = half_sum(ss);
        const float rs = rsqrtf(ss * inv_vdim + a.eps);
        float y[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) y[r] = x[r] * (rs * norm[r] * sigmoid_f((float)gate[r]));
        if (out_in && out_row < done_count) store_elems<4>(outs + (int64_t)(done_row + out_row) * a.out_stride, y);
    };

    // A step first brings the next record, requested a step ago, to LDS and requests the one behind it: what a step waits for has
    // had a whole step to arrive.
    int zero = 0;
    asm volatile("" : "+v"(zero));                     // by the vector path: a scalar load in flight would be waited for with every LDS read
    const int32_t* descs = &chunks[p.chunk0].row0 + zero;
    constexpr int kDesc = sizeof(ChunkDesc) / sizeof(int32_t);
    int next_row = descs[0], next_count = descs[1];
    int row = __builtin_amdgcn_readfirstlane(next_row), count = __builtin_amdgcn_readfirstlane(next_count);
    const int second = p.chunks > 1 ? kDesc : 0;
    next_row = descs[second];
    next_count = descs[second + 1];
    for (int i = tid; i < 2 * 16 * kPitch; i += 512) outputs[i] = 0.f;           // columns behind the last slab stay so
    fetch(0);
    f32x4_t v = vn;
    put(0);
    fetch(1);
    __syncthreads();
    // Loops of their own for wavefronts with columns and for others: where they met, the state would be copied.  Of the two wavefronts of a
    // vector unit the older one is served first, and the other one is alone for the rest of a step, when nothing covers its latencies (4500 and 6900
    // clocks): so the younger ones go first until U, the older ones behind it, if they have columns (heads of 64 x 64, where none of them has: 401 -> 383, of 128 x 64
    // 661 -> 647).  8 portions of 500 .. 2600 tokens, 32 heads, the call 737 -> 718 us, 16 of
    // 800 645 -> 637, 16 heads with 11 of 300 .. 1500 378 -> 365.  Half of the wavefronts with the next record behind the products instead: 734; the products
    // alone or the next record alone ahead: 733, 739.
    auto walk = [&](auto owner) __attribute__((always_inline)) {
        constexpr bool LIVE = decltype(owner)::value;
        for (int c = 0; c < p.chunks; ++c) {
            const WideBuffer buf{lds + (c & 1) * wide_buffer_units(DT), KS};
            if (LIVE && vt >= 4) __builtin_amdgcn_s_setprio(1);
            f32x4_t u = v;
            if (c + 1 < p.chunks) {
                v = vn;
                put((c + 1) & 1);
            }
            if (c > 0) finish((c - 1) & 1);
            fetch(c + 2);
            // rows behind a chunk's last repeat it; an empty chunk has none, and row 0 exists
            gate = *reinterpret_cast<const t4_t*>(gates + (int64_t)(count > 0 ? row + (out_row < count ? out_row : count - 1) : 0) * a.gate_stride);
            __builtin_amdgcn_sched_barrier(0);             // requests stay here, a step ahead of their use
            if constexpr (LIVE) {
                // The vector unit cuts the next part of the state while the matrix pipe works on one.  The pipe rounds its sums towards one
                // side, so nothing stays in its accumulators from chunk to chunk: the state takes a chunk's sum by the vector unit.  3200
                // tokens without decay, all of one sign: error of the state 5.7e-7 of its norm, 6.6e-6 with the state in the pipe's
                // accumulators and pieces cut off instead of rounded, 1.4e-6 in delta_scan_kernel; 794 -> 807 us for the call with the batch above.
                f32x4_t x1 = {0.f, 0.f, 0.f, 0.f}, x2 = x1, x3 = x1, o1 = x1, o2 = x1, o3 = x1;
                uint32_t pc[KS][3][4];
                u32x4_t w[KS][3], qv[KS][3];
                auto part = [&](int kk) {
                    const float f[8] = {s[2 * kk][0], s[2 * kk][1], s[2 * kk][2], s[2 * kk][3], s[2 * kk + 1][0], s[2 * kk + 1][1], s[2 * kk + 1][2], s[2 * kk + 1][3]};
#pragma unroll
                    for (int i = 0; i < 3; ++i) { w[kk][i] = buf.wq(0, kk, i)[lane]; qv[kk][i] = buf.wq(1, kk, i)[lane]; }
                    split3<8>(f, pc[kk]);
                };
                part(0);
#pragma unroll
                for (int kk = 0; kk < KS; ++kk) {
                    const bf16x8_t sh = frag(pc[kk][0]), sm = frag(pc[kk][1]), sl = frag(pc[kk][2]);
                    if (kk + 1 < KS) part(kk + 1);
                    x1 = mma(w[kk][0], sh, x1);
                    o1 = mma(qv[kk][0], sh, o1);
                    x2 = mma(w[kk][1], sh, x2);
                    o2 = mma(qv[kk][1], sh, o2);
                    x3 = mma(w[kk][2], sh, x3);
                    o3 = mma(qv[kk][2], sh, o3);
                    x2 = mma(w[kk][0], sm, x2);
                    o2 = mma(qv[kk][0], sm, o2);
                    x3 = mma(w[kk][1], sm, x3);
                    o3 = mma(qv[kk][1], sm, o3);
                    x3 = mma(w[kk][0], sl, x3);
                    o3 = mma(qv[kk][0], sl, o3);
                }
                if (vt >= 4) __builtin_amdgcn_s_setprio(0);
                else __builtin_amdgcn_s_setprio(1);
                u = u - (x1 + (x2 + x3));
                uint32_t uc[3][2];
                {
                    const float f[4] = {u[0], u[1], u[2], u[3]};
                    split3<4>(f, uc);
                }
                const bf16x8_t uhh = __builtin_bit_cast(bf16x8_t, u32x4_t{uc[0][0], uc[0][1], uc[0][0], uc[0][1]});
                const bf16x8_t umm = __builtin_bit_cast(bf16x8_t, u32x4_t{uc[1][0], uc[1][1], uc[1][0], uc[1][1]});
                const bf16x8_t ulh = __builtin_bit_cast(bf16x8_t, u32x4_t{uc[2][0], uc[2][1], uc[0][0], uc[0][1]});
                const u32x4_t b0 = buf.b(0)[lane], b1 = buf.b(1)[lane];
                o3 = mma(b1, ulh, o3);
                o2 = mma(b0, umm, o2);
                o1 = mma(b0, uhh, o1);
                const f32x4_t* e = reinterpret_cast<const f32x4_t*>(buf.e());
                u32x4_t k0[DT], k1[DT];
                f32x4_t ds[DT], et[DT];
#pragma unroll
                for (int t = 0; t < DT; ++t) {
                    k0[t] = buf.k(t, 0)[lane];
                    k1[t] = buf.k(t, 1)[lane];
                    et[t] = e[4 * t + q];
                }
#pragma unroll
                for (int t = 0; t < DT; ++t) ds[t] = mma(k1[t], ulh, f32x4_t{0.f, 0.f, 0.f, 0.f});
#pragma unroll
                for (int t = 0; t < DT; ++t) ds[t] = mma(k0[t], umm, ds[t]);
#pragma unroll
                for (int t = 0; t < DT; ++t) ds[t] = mma(k0[t], uhh, ds[t]);
#pragma unroll
                for (int t = 0; t < DT; ++t) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) s[t][r] = __builtin_fmaf(s[t][r], et[t][r], ds[t][r]);
                }
                const f32x4_t o = o1 + (o2 + o3);
                float* to = outputs + ((c & 1) * 16 + 4 * q) * kPitch + 16 * vt + m;
#pragma unroll
                for (int r = 0; r < 4; ++r) to[r * kPitch] = o[r];
            }
            __builtin_amdgcn_s_setprio(0);
            done_row = row;
            done_count = count;
            row = __builtin_amdgcn_readfirstlane(next_row);
            count = __builtin_amdgcn_readfirstlane(next_count);
            const int after = c + 2 < p.chunks ? c + 2 : p.chunks - 1;
            next_row = descs[after * kDesc];
            next_count = descs[after * kDesc + 1];
            __syncthreads();
        }
    };
    if (live) walk(std::true_type{});
    else walk(std::false_type{});
    finish((p.chunks - 1) & 1);
    keep_state();
}

// The inputs of the convolution that a portion's last tokens leave in its ring; a workgroup looks at 64 rows and copies VEC * 256 channels
// of those it finds.
template <class T, int VEC>
__global__ void __launch_bounds__(256) delta_ring_kernel(DeltaArgs<T> a, int64_t row0, int64_t rows, const int32_t* ring_slot, const int64_t* positions) {
    typedef T vec_t __attribute__((ext_vector_type(VEC)));
    const int64_t first = row0 + 64 * (int64_t)blockIdx.x, mine = first + (threadIdx.x & 63);
    const int c = (blockIdx.y * 256 + threadIdx.x) * VEC;
    const int slot = mine < row0 + rows ? ring_slot[2 * mine] : -1;
    const int follow = mine < row0 + rows ? ring_slot[2 * mine + 1] : a.taps;
    uint64_t found = __ballot(slot >= 0 && slot < a.num_slots && follow < a.taps);
    while (found) {
        const int i = __builtin_ctzll(found);
        found &= found - 1;
        const int64_t row = first + i, to = (int64_t)__builtin_amdgcn_readlane(slot, i) * a.taps + positions[row] % a.taps;
        if (c < a.channels) *reinterpret_cast<vec_t*>(a.ring + to * a.channels + c) = *reinterpret_cast<const vec_t*>(a.proj + row * a.proj_stride + c);
    }
}

// One workgroup per token row behind `row0`.  LANES lanes share a head, four values each (vdim = 4 LANES);
// LANES = 0: any vdim, one wavefront per head.
template <class T, int LANES>
__global__ void __launch_bounds__(256) delta_out_kernel(DeltaArgs<T> a, const float* o, int64_t row0, const int32_t* ring_slot,
                                                        const int64_t* positions) {
    const int64_t row = row0 + blockIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if constexpr (LANES > 0) {
        const int v = 4 * (threadIdx.x % LANES);
        float w[4];
        load_elems<4>(a.norm + v, w);
        for (int h = threadIdx.x / LANES; h < a.heads; h += 256 / LANES) {
            float x[4], g[4];
            load_elems<4>(o + (row * a.heads + h) * a.vdim_pad + v, x);
            load_elems<4>(a.gate + row * a.gate_stride + (int64_t)h * a.vdim + v, g);
            float ss = x[0] * x[0] + x[1] * x[1] + x[2] * x[2] + x[3] * x[3];
#pragma unroll
            for (int m = LANES / 2; m >= 1; m >>= 1) ss += __shfl_xor(ss, m, 64);
            const float rs = rsqrtf(ss / (float)a.vdim + a.eps);
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] *= rs * w[e] * sigmoid_f(g[e]);
            store_elems<4>(a.out + row * a.out_stride + (int64_t)h * a.vdim + v, x);
        }
    } else {
        for (int h = wave; h < a.heads; h += 4) {
            const float* x = o + (row * a.heads + h) * a.vdim_pad;
            float ss = 0.f;
            for (int v = lane; v < a.vdim; v += 64) ss += x[v] * x[v];
            const float rs = rsqrtf(wave_sum(ss) / (float)a.vdim + a.eps);
            const T* gr = a.gate + row * a.gate_stride + (int64_t)h * a.vdim;
            T* out = a.out + row * a.out_stride + (int64_t)h * a.vdim;
            for (int v = lane; v < a.vdim; v += 64) out[v] = (T)(x[v] * rs * a.norm[v] * sigmoid_f((float)gr[v]));
        }
    }
    const int slot = ring_slot[2 * row];
    if (slot < 0 || slot >= a.num_slots || ring_slot[2 * row + 1] >= a.taps) return;     // not among the portion's last inputs
    T* ring = a.ring + ((int64_t)slot * a.taps + positions[row] % a.taps) * a.channels;
    const T* in = a.proj + row * a.proj_stride;
    for (int c = threadIdx.x; c < a.channels; c += 256) ring[c] = in[c];
}

int tiles_of(int dim) {        // row tiles of the state, rounded up to what the scan is built for
    const int t = (dim + 15) / 16;
    for (int n : {1, 2, 3, 4, 6, 8, 12, 16})
        if (t <= n) return n;
    return 0;
}

template <int DT>
int launch_scan(const PortionDesc* p, int64_t portions, int64_t tokens, const ChunkDesc* c, const float* records, float* state, float* o,
                int heads, int vdim_pad, hipStream_t st) {
    const int slabs = vdim_pad / 16, waves = slabs < 4 ? slabs : 4;
    constexpr size_t lds = (size_t)2 * (49 * 16 * DT + 256) * sizeof(float);
    if (lds > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&delta_scan_kernel<DT>),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return (int)e;
    }
    hipLaunchKernelGGL((delta_scan_kernel<DT>), dim3((unsigned)((slabs + waves - 1) / waves), (unsigned)heads, (unsigned)portions),
                       dim3(64 * waves), lds, st, p, c, records, state, o, heads, vdim_pad, turns_of(portions, (int64_t)heads * ((slabs + waves - 1) / waves), tokens));
    return (int)hipGetLastError();
}

template <int DT, int CT>
int launch_scan_slab(const PortionDesc* p, int64_t portions, const ChunkDesc* c, const float* records, float* state, float* o,
                     int heads, int vdim_pad, hipStream_t st) {
    using Z = SlabSizes<DT, CT>;
    const int64_t pairs = portions * heads;
    const int slabs = (vdim_pad / 16 + CT - 1) / CT;
    auto kernel = &delta_scan_slab_kernel<DT, CT>;
    if (Z::lds > 60 * 1024) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, Z::lds);
        if (e != hipSuccess) return (int)e;
    }
    hipLaunchKernelGGL(kernel, dim3((unsigned)((pairs + 7) / 8 * 8 * slabs)), dim3(Z::threads), Z::lds, st, p, c, records, state, o, heads, vdim_pad, (int)pairs, slabs);
    return (int)hipGetLastError();
}
// Tiles of 16 columns per workgroup of delta_scan_slab_kernel, or 0 where the others are ahead.  Heads of 128 rows need a compute unit for a workgroup: one
// tile as long as there are enough of them, otherwise two or four.  Others share it, and one tile is ahead up to two and a half workgroups per unit.  The call,
// us, delta_scan_kernel (* delta_scan_wide_kernel) / 1 / 2 / 4 tiles, heads x portions of tokens: 128 x 128 16 x 1 of 2000 352 / 150 / 194 / 290, 32 x 1 of 12000 2197 / 1087 /
// 1277 / 1823, 16 x 4 of 500 to 3000 528 / 358 / 333 / 446, 32 x 2 of 1000 233 / 187 / 156 / 204, 32 x 3 267 / 295 / 270 / 240, 32 x 4 297 / 392 / 310 / 277, but 32 x 5 302* / 486 /
// 412 / 419; 64 x 64 32 x 4 of 1000 177 / 136 / 132 / 165, 32 x 5 176* / 196 / 212 / 195; 96 x 96 30 x 4 of 800 230 / 226 / 243 / 252; 256 x 128 16 x 5 of 600 355 / 303 /
// 429; 192 x 192 16 x 3 of 300 to 1200 364 / 274; 48 x 48 30 x 7 of 600 189 / 144; 32 x 32 32 x 5 of 300 to 900 117* / 93; 16 x 16 30 x 20 of 700 290 / 276.
int few_tiles(int dim_pad, int vdim_pad, int64_t pairs) {
    const int tiles = vdim_pad / 16;
    if (dim_pad != 128) return pairs * tiles <= 640 ? 1 : 0;
    for (int n : {1, 2, 4})
        if (pairs * ((tiles + n - 1) / n) <= 256) return n;
    return 0;
}
template <int DT>
int launch_few(const PortionDesc* p, int64_t portions, int64_t tokens, const ChunkDesc* c, const float* records, float* state, float* o,
               int heads, int vdim_pad, hipStream_t st) {
    const int tiles = few_tiles(16 * DT, vdim_pad, portions * heads);
    if (tiles == 1) return launch_scan_slab<DT, 1>(p, portions, c, records, state, o, heads, vdim_pad, st);
    if constexpr (DT == 8) {
        if (tiles == 2) return launch_scan_slab<DT, 2>(p, portions, c, records, state, o, heads, vdim_pad, st);
        if (tiles == 4) return launch_scan_slab<DT, 4>(p, portions, c, records, state, o, heads, vdim_pad, st);
    }
    return launch_scan<DT>(p, portions, tokens, c, records, state, o, heads, vdim_pad, st);
}

template <class T, int DT>
int launch_scan_wide(const DeltaArgs<T>& a, const PortionDesc* p, int64_t portions, int64_t tokens, const ChunkDesc* c, const float* records, hipStream_t st) {
    constexpr size_t lds = (size_t)2 * wide_buffer_units(DT) * 16 + 2 * 16 * 132 * sizeof(float);
    if (lds > 60 * 1024) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&delta_scan_wide_kernel<T, DT>),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return (int)e;
    }
    hipLaunchKernelGGL((delta_scan_wide_kernel<T, DT>), dim3((unsigned)a.heads, (unsigned)portions), dim3(512), lds, st, a, p, c, records,
                       a.vdim_pad / 16, turns_of(portions, a.heads, tokens));
    return (int)hipGetLastError();
}

template <class T>
int make_args(DeltaArgs<T>& a, const void* proj, int64_t proj_stride, int64_t beta_off, const void* decay, int64_t decay_stride,
              const void* gate, int64_t gate_stride, const float* conv, const float* a_log, const float* dt_bias, const float* norm,
              void* ring, float* state, int64_t num_slots, int64_t heads, int64_t kv_heads, int64_t dim, int64_t vdim, int64_t taps,
              float eps, void* out, int64_t out_stride) {
    if (!proj || !decay || !gate || !conv || !a_log || !dt_bias || !norm || !ring || !state || !out) return INFER_KV_EINVAL;
    if (heads < 1 || heads > 65535 || kv_heads < 1 || heads % kv_heads || dim < 1 || vdim < 1 || taps < 1 || taps > 64 || num_slots < 1 ||
        num_slots > (1 << 24))
        return INFER_KV_EINVAL;
    if (dim > 256 || vdim > 512) return INFER_KV_EUNSUPPORTED;
    const int64_t channels = 2 * kv_heads * dim + heads * vdim;
    if (beta_off < channels || proj_stride < beta_off + heads || decay_stride < heads * dim || gate_stride < heads * vdim ||
        out_stride < heads * vdim)
        return INFER_KV_EINVAL;
    if (!ptr_aligned(state, 16)) return INFER_KV_EALIGN;
    a = DeltaArgs<T>{(const T*)proj, proj_stride, (int)beta_off, (const T*)decay, decay_stride, (const T*)gate, gate_stride, conv, a_log,
                     dt_bias, norm, (T*)ring, state, (int)num_slots, (int)heads, (int)kv_heads, (int)dim, (int)vdim,
                     16 * tiles_of((int)dim), (int)((vdim + 15) / 16 * 16), (int)taps, (int)channels, eps, 1.0f / sqrtf((float)dim),
                     (T*)out, out_stride};
    return INFER_KV_OK;
}

template <class T>
int launch_step(const DeltaArgs<T>& a, const int32_t* slots, const int64_t* positions, int64_t rows, hipStream_t st) {
    const int cgs = a.vdim_pad / 4, rgs = kStepThreads / cgs, np = (a.dim_pad + rgs - 1) / rgs;
    const size_t lds = (size_t)(3 * a.dim_pad + a.vdim_pad + rgs * a.vdim_pad + 12) * sizeof(float);
    const dim3 grid((unsigned)rows, (unsigned)a.heads), block(kStepThreads);
#define GO(N) hipLaunchKernelGGL((delta_step_kernel<T, N>), grid, block, lds, st, a, slots, positions)
    if (np <= 1) GO(1);
    else if (np <= 2) GO(2);
    else if (np <= 4) GO(4);
    else if (np <= 8) GO(8);
    else if (np <= 16) GO(16);
    else if (np <= 32) GO(32);
    else GO(0);
#undef GO
    return (int)hipGetLastError();
}

template <int DT>
int launch_prep_square(const DeltaArgs<__bf16>& a, const ChunkDesc* chunks, int64_t num_chunks, float* records, hipStream_t st) {
    constexpr int D = 16 * DT;
    constexpr size_t lds = (size_t)(4 * kC * (D + 4) + 1024 + kC * 20 + 2 * D + 48) * sizeof(float);
    static_assert(lds <= 40 * 1024, "four workgroups a compute unit");
    hipLaunchKernelGGL((delta_prep_square_kernel<DT>), dim3((unsigned)num_chunks, (unsigned)a.heads), dim3(256), lds, st, a, chunks, records);
    return (int)hipGetLastError();
}

template <class T>
int launch_chunks(const DeltaArgs<T>& a, const PortionDesc* portions, int64_t num_portions, const ChunkDesc* chunks, int64_t num_chunks,
                  float* records, float* o, int64_t row0, int64_t rows, const int32_t* ring_slot, const int64_t* positions,
                  hipStream_t st) {
    const size_t lds = (size_t)(3 * kC * (a.dim_pad + 4) + kC * (a.vdim_pad + 4) + 1024 + kC * 20 + a.dim_pad + 48) * sizeof(float);
    // rows and channels that can be read four elements at a time
    auto fours = [](const void* p, int64_t stride) { return ptr_aligned(p, 4 * sizeof(T)) && stride % 4 == 0; };
    const bool rows4 = a.dim % 4 == 0 && a.vdim % 4 == 0;
    const bool vec = rows4 && a.taps == 4 && fours(a.proj, a.proj_stride) && fours(a.ring, a.channels) && fours(a.decay, a.decay_stride) &&
                     ptr_aligned(a.conv, 16) && ptr_aligned(a.dt_bias, 16);
    auto prep = vec ? &delta_prep_kernel<T, true> : &delta_prep_kernel<T, false>;
    if (lds > 60 * 1024) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(prep), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return (int)e;
    }
    int rc = INFER_KV_OK;
    bool prepared = false;
    if constexpr (sizeof(T) == 2)
        if (vec && a.dim == a.vdim && (a.dim == 64 || a.dim == 128) && a.decay_stride % 2 == 0) {
            rc = a.dim == 64 ? launch_prep_square<4>(a, chunks, num_chunks, records, st) : launch_prep_square<8>(a, chunks, num_chunks, records, st);
            prepared = true;
        }
    if (!prepared) {
        hipLaunchKernelGGL(prep, dim3((unsigned)num_chunks, (unsigned)a.heads), dim3(256), lds, st, a, chunks, records);
        rc = (int)hipGetLastError();
    }
    if (rc) return rc;
    const bool out4 = rows4 && fours(a.gate, a.gate_stride) && fours(a.out, a.out_stride) && ptr_aligned(o, 16) && ptr_aligned(a.norm, 16);
    // Up to 128 pairs of a portion and a head, and some more of small heads (few_tiles), the columns of a head go to several workgroups.  Beyond, one
    // workgroup for a head and its outputs wins, here against delta_scan_kernel: 32 heads, 16 portions of 800 tokens 853 us against 712, 60 of 110 512 against 428; heads
    // of 64 x 64, 5 of 800 183 against 156; of 128 x 16, 5 of 800 465 against 181.  Small heads give most of its eight wavefronts no
    // columns, which costs where there are more workgroups than compute units, unless delta_out_kernel has no form for the columns
    // either: 60 portions of 110, heads of 32 x 32 153 us against 195, 32 x 64 201 against 213, 64 x 32 220 against 253, but 32 x 48 210
    // against 197.
    const int64_t pairs = (int64_t)a.heads * num_portions;
    const bool small = a.dim_pad * a.vdim_pad <= 2048 && (a.vdim == 32 || a.vdim == 64);
    const bool slabs = pairs <= 128 || (few_tiles(a.dim_pad, a.vdim_pad, pairs) == 1 && pairs * (a.vdim_pad / 16) <= 320);
    if (out4 && !slabs && !(small && pairs > 256) && a.vdim_pad <= 128 && (a.dim_pad == 32 || a.dim_pad == 64 || a.dim_pad == 96 || a.dim_pad == 128)) {
#define GO(N) case N: rc = launch_scan_wide<T, N>(a, portions, num_portions, rows, chunks, records, st); break
        switch (a.dim_pad / 16) { GO(2); GO(4); GO(6); GO(8); }
#undef GO
        if (rc) return rc;
        const unsigned groups = (unsigned)((rows + 63) / 64);
        if (rows4 && fours(a.proj, a.proj_stride) && fours(a.ring, a.channels))
            hipLaunchKernelGGL((delta_ring_kernel<T, 4>), dim3(groups, (unsigned)((a.channels + 1023) / 1024)), dim3(256), 0, st, a, row0, rows, ring_slot, positions);
        else
            hipLaunchKernelGGL((delta_ring_kernel<T, 1>), dim3(groups, (unsigned)((a.channels + 255) / 256)), dim3(256), 0, st, a, row0, rows, ring_slot, positions);
        return (int)hipGetLastError();
    }
#define GO(N) case N: rc = launch_few<N>(portions, num_portions, rows, chunks, records, a.state, o, a.heads, a.vdim_pad, st); break
    switch (a.dim_pad / 16) { GO(1); GO(2); GO(3); GO(4); GO(6); GO(8); GO(12); GO(16); default: return INFER_KV_EUNSUPPORTED; }
#undef GO
    if (rc) return rc;
#define GO(N) hipLaunchKernelGGL((delta_out_kernel<T, N>), dim3((unsigned)rows), dim3(256), 0, st, a, (const float*)o, row0, ring_slot, positions)
    if (out4 && a.vdim == 32) GO(8);
    else if (out4 && a.vdim == 64) GO(16);
    else if (out4 && a.vdim == 128) GO(32);
    else if (out4 && a.vdim == 256) GO(64);
    else GO(0);
#undef GO
    return (int)hipGetLastError();
}

}  // namespace

// [0]: state rows per head, [1]: state columns per head, [2]: floats of a chunk record, [3]: tokens per chunk;
// 0 if the sizes are served, otherwise a negative code
extern "C" int infer_delta_layout(int64_t dim, int64_t vdim, int64_t* out4) {
    if (!out4 || dim < 1 || vdim < 1) return INFER_KV_EINVAL;
    if (dim > 256 || vdim > 512) return INFER_KV_EUNSUPPORTED;
    const int dp = 16 * tiles_of((int)dim), vp = (int)((vdim + 15) / 16 * 16);
    out4[0] = dp; out4[1] = vp; out4[2] = record_floats(dp, vp); out4[3] = kC;
    return INFER_KV_OK;
}

extern "C" int infer_delta_step(int elem, const void* proj, int64_t proj_stride, int64_t beta_off, const void* decay,
                                int64_t decay_stride, const void* gate, int64_t gate_stride, const float* conv, const float* a_log,
                                const float* dt_bias, const float* norm, void* ring, float* state, int64_t num_slots, int64_t heads,
                                int64_t kv_heads, int64_t dim, int64_t vdim, int64_t taps, float eps, const int32_t* slots,
                                const int64_t* positions, void* out, int64_t out_stride, int64_t rows, void* stream) {
    if (rows < 0 || rows > 0x7fffffff) return INFER_KV_EINVAL;
    if (rows == 0) return INFER_KV_OK;
    if (!slots || !positions) return INFER_KV_EINVAL;
    int rc;
    if (elem == INFER_ELEM_BF16) {
        DeltaArgs<__bf16> a;
        rc = make_args(a, proj, proj_stride, beta_off, decay, decay_stride, gate, gate_stride, conv, a_log, dt_bias, norm, ring, state,
                       num_slots, heads, kv_heads, dim, vdim, taps, eps, out, out_stride);
        return rc ? rc : launch_step(a, slots, positions, rows, (hipStream_t)stream);
    }
    if (elem == INFER_ELEM_F32) {
        DeltaArgs<float> a;
        rc = make_args(a, proj, proj_stride, beta_off, decay, decay_stride, gate, gate_stride, conv, a_log, dt_bias, norm, ring, state,
                       num_slots, heads, kv_heads, dim, vdim, taps, eps, out, out_stride);
        return rc ? rc : launch_step(a, slots, positions, rows, (hipStream_t)stream);
    }
    return INFER_KV_EUNSUPPORTED;
}

extern "C" int infer_delta_chunks(int elem, const void* proj, int64_t proj_stride, int64_t beta_off, const void* decay,
                                  int64_t decay_stride, const void* gate, int64_t gate_stride, const float* conv, const float* a_log,
                                  const float* dt_bias, const float* norm, void* ring, float* state, int64_t num_slots, int64_t heads,
                                  int64_t kv_heads, int64_t dim, int64_t vdim, int64_t taps, float eps, const int32_t* portions,
                                  int64_t num_portions, const int32_t* chunks, int64_t num_chunks, float* records, float* o,
                                  const int32_t* ring_slot, const int64_t* positions, void* out, int64_t out_stride, int64_t row0,
                                  int64_t rows, void* stream) {
    if (rows < 0 || rows > 0x7fffffff || row0 < 0 || num_portions < 0 || num_portions > 65535 || num_chunks < num_portions ||
        num_chunks > 0x7fffffff)
        return INFER_KV_EINVAL;
    if (rows == 0 || num_portions == 0) return INFER_KV_OK;
    if (!portions || !chunks || !records || !o || !ring_slot || !positions) return INFER_KV_EINVAL;
    if (!ptr_aligned(records, 16)) return INFER_KV_EALIGN;
    int rc;
    if (elem == INFER_ELEM_BF16) {
        DeltaArgs<__bf16> a;
        rc = make_args(a, proj, proj_stride, beta_off, decay, decay_stride, gate, gate_stride, conv, a_log, dt_bias, norm, ring, state,
                       num_slots, heads, kv_heads, dim, vdim, taps, eps, out, out_stride);
        return rc ? rc : launch_chunks(a, (const PortionDesc*)portions, num_portions, (const ChunkDesc*)chunks, num_chunks, records, o,
                                       row0, rows, ring_slot, positions, (hipStream_t)stream);
    }
    if (elem == INFER_ELEM_F32) {
        DeltaArgs<float> a;
        rc = make_args(a, proj, proj_stride, beta_off, decay, decay_stride, gate, gate_stride, conv, a_log, dt_bias, norm, ring, state,
                       num_slots, heads, kv_heads, dim, vdim, taps, eps, out, out_stride);
        return rc ? rc : launch_chunks(a, (const PortionDesc*)portions, num_portions, (const ChunkDesc*)chunks, num_chunks, records, o,
                                       row0, rows, ring_slot, positions, (hipStream_t)stream);
    }
    return INFER_KV_EUNSUPPORTED;
}
