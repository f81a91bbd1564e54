// Rows of weights streamed past a few rows of activations: y[16 MT][16 RT] = x w^T for one workgroup, the steps of k dealt out to its
// wavefronts, each of which brings its own steps to a ring in LDS and multiplies them without ever waiting for another one.
//
// A step is 64 elements of every row, a whole 128-byte line.  One request of a wavefront fills 1 KiB of LDS with eight rows of a step,
// straight from memory; 16-byte unit c of row r lies at place c ^ (r % 8), so that the reads of a matrix operand meet all banks.
// Weights carry the streaming hint, activations stay in the second-level cache.  What this is worth, 16 rows past 24576 x 4096 weights:
// requests of 64 bytes of 16 rows straight into operand registers 52.8 us (3.8 TB/s), this 35.3 us (5.7 TB/s); a read of the weights
// alone in lines takes 31.5 us with the hint and 33.7 without, in halves of lines 37.7.
#pragma once
#include <type_traits>

#include "elem.h"

constexpr int kStreamK = 64;                       // elements of a step
constexpr int stream_stage_bytes(int rt, int mt) { return 2048 * (rt + mt); }

// Where a lane of a request starts in the row it reads: row lane / 8 of eight, its unit of the step
__device__ __forceinline__ int stream_row() { return (threadIdx.x & 63) >> 3; }
__device__ __forceinline__ int stream_col() { return 8 * ((threadIdx.x & 7) ^ ((threadIdx.x & 63) >> 3)); }

// Where a workgroup begins its walk over k, of `steps`; behind the end it goes on at the front.  Rows of weights lie a power of two or a small multiple of
// one apart, so workgroups that all begin at the front read the same few channels of memory at any one time, and the same lines of the activations.
// Every eighth workgroup goes to the same die, whose 32 compute units begin evenly spread: `turn` counts eights of workgroups or so.  Everybody at the front / this,
// 64 of the batch, us: gate and up of 24576 x 4096 42.8 / 37.2, 65536 x 4096 108 / 90, 8192 x 4096 20.8 / 16.6; four: 16384 x 2048 14.9 / 12.6.  One turn behind the
// other: with the 32 places in the order of their bits in reverse 24576 x 4096, steps shared (below), 33.6 / 37.0, four of the batch 32.2 / 38.1.
__device__ __forceinline__ int stream_start(int turn, int steps) { return (int)((turn & 31) * (unsigned)steps >> 5); }

// w[i], x[i]: this lane's row stream_row() + 8 i of the weights and of the activations, at the first element of k (16-byte aligned);
// TURNED: the walk begins at stream_start(turn), otherwise at the front; k: elements, a multiple of eight; ring: D * stream_stage_bytes(RT, MT) bytes of the wavefront's own.  Adds to acc[r][t] (lane (g, n):
// row n of tile t of x, rows 4 g + e of tile r of w) what the steps `wave`, `wave` + NW, ... contribute.
template <int RT, int MT, int NW, int D, bool TURNED>
__device__ __forceinline__ void stream_product(const __bf16* const (&w)[2 * RT], const __bf16* const (&x)[2 * MT], int k, int turn, int wave,
                                               unsigned char* ring, f32x4_t (&acc)[RT][MT]) {
    constexpr int kRequests = 2 * (RT + MT), kStage = stream_stage_bytes(RT, MT);
    static_assert(D >= 2 && D <= 4 && (D - 1) * kRequests <= 63, "requests in flight are counted in six bits");
    const int lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15, col = stream_col();
    const int all = (k + kStreamK - 1) / kStreamK, steps = all > wave ? (all - wave + NW - 1) / NW : 0;
    const uint32_t base = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)ring);
    // Inline assembly, since the compiler would put a wait for all requests in front of every read of LDS.  Nothing else here uses M0.
    int ahead = TURNED ? stream_start(turn, steps) : 0, now = ahead;      // the steps to be requested and to be multiplied next
    auto request = [&](int stage) {
        const int at = (ahead * NW + wave) * kStreamK + col, from = at < k ? at : 0;   // behind the end: something, which meets zeros
        ahead = TURNED && ahead + 1 == steps ? 0 : ahead + 1;
#pragma unroll
        for (int i = 0; i < kRequests; ++i) {
            const uint32_t to = base + stage * kStage + 1024 * i;
            if (i < 2 * RT)
                __asm__ volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt" :: "v"(w[i < 2 * RT ? i : 0] + from), "s"(to) : "memory", "m0");
            else
                __asm__ volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" :: "v"(x[i < 2 * RT ? 0 : i - 2 * RT] + from), "s"(to) : "memory", "m0");
        }
    };
#pragma unroll
    for (int d = 0; d < D; ++d)
        if (d < steps) request(d);
    const int place = 128 * n + 16 * (g ^ (n & 7));
    int stage = 0;
    for (int s = 0; s < steps; ++s) {
        const int behind = steps - 1 - s;              // steps that have been requested and are not waited for: as many, at most D - 1
        if (behind >= D - 1) __asm__ volatile("s_waitcnt vmcnt(%0)" :: "n"((D - 1) * kRequests) : "memory");
        else if (D > 3 && behind == 2) __asm__ volatile("s_waitcnt vmcnt(%0)" :: "n"(D > 3 ? 2 * kRequests : 0) : "memory");
        else if (D > 2 && behind == 1) __asm__ volatile("s_waitcnt vmcnt(%0)" :: "n"(D > 2 ? kRequests : 0) : "memory");
        else __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
        bf16x8_t a[RT][2], b[MT][2];
        const unsigned char* p = ring + stage * kStage;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int r = 0; r < RT; ++r) a[r][h] = *reinterpret_cast<const bf16x8_t*>(p + 2048 * r + (place ^ (64 * h)));
#pragma unroll
            for (int t = 0; t < MT; ++t) b[t][h] = *reinterpret_cast<const bf16x8_t*>(p + 2048 * (RT + t) + (place ^ (64 * h)));
        }
        __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");         // read before the stage is filled again
        __builtin_amdgcn_sched_barrier(0);
        if (s + D < steps) request(stage);
        const int first = (now * NW + wave) * kStreamK;
        now = TURNED && now + 1 == steps ? 0 : now + 1;
        if (first + kStreamK > k)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                if (first + 32 * h + 8 * g >= k)
#pragma unroll
                    for (int t = 0; t < MT; ++t) b[t][h] = bf16x8_t{};
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int r = 0; r < RT; ++r) acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[r][h], b[t][h], acc[r][t], 0, 0, 0);
        stage = stage + 1 == D ? 0 : stage + 1;
    }
}

// The same past activations that lie in LDS as a whole: only the weights are requested, and `before` runs behind the first requests, while
// they are on their way; it puts the activations where x points (this lane's row, at element 8 g of the first step) and ends with a barrier.
// k: a multiple of kStreamK; ring: D * stream_stage_bytes(RT, 0) bytes.
template <int RT, int NW, int D, bool TURNED, class Before>
__device__ __forceinline__ void stream_product_held(const __bf16* const (&w)[2 * RT], const unsigned char* x, int k, int turn, int wave, unsigned char* ring,
                                                    Before before, f32x4_t (&acc)[RT][1]) {
    constexpr int kRequests = 2 * RT, kStage = stream_stage_bytes(RT, 0);
    static_assert(D >= 2 && D <= 4, "the waits below");
    const int lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15, col = stream_col();
    const int all = k / kStreamK, steps = all > wave ? (all - wave + NW - 1) / NW : 0;
    const uint32_t base = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)ring);
    int ahead = TURNED ? stream_start(turn, steps) : 0, now = ahead;
    auto request = [&](int stage) {
        const int from = (ahead * NW + wave) * kStreamK + col;
        ahead = TURNED && ahead + 1 == steps ? 0 : ahead + 1;
#pragma unroll
        for (int i = 0; i < kRequests; ++i)
            __asm__ volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt" :: "v"(w[i] + from), "s"(base + stage * kStage + 1024 * i) : "memory", "m0");
    };
#pragma unroll
    for (int d = 0; d < D; ++d)
        if (d < steps) request(d);
    before();
    const int place = 128 * n + 16 * (g ^ (n & 7));
    int stage = 0;
    for (int s = 0; s < steps; ++s) {
        // requests of later steps are the only ones behind this step's, or there are stores in between, with which this waits longer
        const int behind = steps - 1 - s;
        if (behind >= D - 1) __asm__ volatile("s_waitcnt vmcnt(%0)" :: "n"((D - 1) * kRequests) : "memory");
        else if (D > 3 && behind == 2) __asm__ volatile("s_waitcnt vmcnt(%0)" :: "n"(D > 3 ? 2 * kRequests : 0) : "memory");
        else if (D > 2 && behind == 1) __asm__ volatile("s_waitcnt vmcnt(%0)" :: "n"(D > 2 ? kRequests : 0) : "memory");
        else __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
        bf16x8_t a[RT][2], b[2];
        const unsigned char* p = ring + stage * kStage;
        const unsigned char* from = x + 2 * kStreamK * (now * NW + wave);
        now = TURNED && now + 1 == steps ? 0 : now + 1;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int r = 0; r < RT; ++r) a[r][h] = *reinterpret_cast<const bf16x8_t*>(p + 2048 * r + (place ^ (64 * h)));
            b[h] = *reinterpret_cast<const bf16x8_t*>(from + 64 * h);
        }
        __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");         // read before the stage is filled again
        __builtin_amdgcn_sched_barrier(0);
        if (s + D < steps) request(stage);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int r = 0; r < RT; ++r) acc[r][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[r][h], b[h], acc[r][0], 0, 0, 0);
        stage = stage + 1 == D ? 0 : stage + 1;
    }
}

// The sum of the wavefronts' parts of every tile, tile q = r * MT + t by wavefront q % NW, which gets it as f(r, t, sum) in the layout of
// acc.  `lds` holds NW * RT * MT KiB; everybody is past its own ring.
template <int RT, int MT, int NW, class F>
__device__ __forceinline__ void stream_reduce(const f32x4_t (&acc)[RT][MT], int wave, unsigned char* lds, F f) {
    f32x4_t* part = reinterpret_cast<f32x4_t*>(lds);
    const int lane = threadIdx.x & 63;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int t = 0; t < MT; ++t) part[(wave * RT * MT + r * MT + t) * 64 + lane] = acc[r][t];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < RT * MT; ++q) {
        if (q % NW != wave) continue;
        f32x4_t sum = part[q * 64 + lane];
#pragma unroll
        for (int v = 1; v < NW; ++v) sum += part[(v * RT * MT + q) * 64 + lane];
        f(q / MT, q % MT, sum);
    }
}

// Rows of weights past activations that the four wavefronts of a workgroup share: they go through one ring of D steps, of which every wavefront brings
// a quarter, and a wavefront multiplies RT / WR tiles of weight rows by all MT tiles of the batch: with all of a step's elements (WR = 4), or with one half
// of them (WR = 2; the sums of the two halves remain to be added).  One barrier a step: behind it the step has arrived for everybody, and the place
// of the one before is free.
//
// A wavefront that streams by itself (above) brings the batch for its own rows alone, and two steps of that are all that LDS holds; here the batch
// takes 8 KB of a step of up to 48.  And in eight times as many smaller steps what is under way hardly falls while one is multiplied.
template <int RT, int MT>
struct SharedStream {
    // Up to 96 rows leave room for a second workgroup on the compute unit, which begins while the other one ends
    static constexpr int kWaves = 4, WR = RT <= 6 || RT % 4 ? 2 : 4, kTiles = RT / WR, KH = WR == 4 ? 2 : 1;
    static constexpr int kStage = stream_stage_bytes(RT, MT), kFit = (RT <= 6 ? 80 : 160) * 1024 / kStage, D = kFit < 12 ? kFit : 12, kRing = D * kStage;
    static constexpr int kOfWeights = 2 * RT / kWaves, kRequests = kOfWeights + (2 * MT + kWaves - 1) / kWaves;
    static_assert(RT % WR == 0 && 2 * RT % kWaves == 0 && D >= 3 && (D - 2) * kRequests <= 63, "requests in flight are counted in six bits");
    const __bf16* from[kRequests];
    uint32_t to[kRequests];
    int ahead, steps;

    // Whether a walk over k begins at stream_start(turn): a short one would find out where for nothing
    static __host__ __device__ __forceinline__ bool turned(int k) { return k >= 2048; }
    // weights(i), batch(i): this lane's row stream_row() + 8 i of either, at the first element of k (a multiple of kStreamK)
    template <class Weights, class Batch>
    __device__ __forceinline__ SharedStream(int k, int turn, int wave, const unsigned char* ring, Weights weights, Batch batch) {
        const uint32_t base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)ring;
#pragma unroll
        for (int j = 0; j < kRequests; ++j) {
            const int i = wave + kWaves * j, of_batch = (i - 2 * RT) & (2 * MT - 1);       // one too many repeats another
            from[j] = (j < kOfWeights ? weights(i) : batch(of_batch)) + stream_col();
            to[j] = __builtin_amdgcn_readfirstlane(base + 1024 * (j < kOfWeights ? i : 2 * RT + of_batch));
        }
        steps = k / kStreamK;
        ahead = turned(k) ? stream_start(turn, steps) : 0;
    }
    __device__ __forceinline__ void request(int stage) {
#pragma unroll
        for (int j = 0; j < kRequests; ++j) {
            const uint32_t at = to[j] + stage * kStage;
            if (j < kOfWeights)
                __asm__ volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt" :: "v"(from[j] + ahead * kStreamK), "s"(at) : "memory", "m0");
            else
                __asm__ volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" :: "v"(from[j] + ahead * kStreamK), "s"(at) : "memory", "m0");
        }
        ahead = ahead + 1 == steps ? 0 : ahead + 1;
    }
    // Adds to acc[r][t]: tile kTiles (wave % WR) + r of the weights, tile t of the batch; layout as of stream_product
    __device__ __forceinline__ void product(int wave, const unsigned char* ring, f32x4_t (&acc)[kTiles][MT]) {
        const int lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15, first = wave % WR * kTiles;
        const int place = 128 * n + 16 * (g ^ (n & 7)) ^ (KH == 1 ? 64 * (wave / WR) : 0);
#pragma unroll
        for (int d = 0; d < D - 1; ++d)
            if (d < steps) request(d);
        int stage = 0, free = D - 1;                   // where step s lies, and where the one D - 1 behind it will
        auto step = [&](int s, auto behind) __attribute__((always_inline)) {       // behind: steps that have been requested and are not waited for
            __asm__ volatile("s_waitcnt vmcnt(%0)" :: "n"(decltype(behind)::value * kRequests) : "memory");
            __builtin_amdgcn_s_barrier();
            __asm__ volatile("" ::: "memory");
            bf16x8_t a[kTiles][KH], b[MT][KH];
            const unsigned char* p = ring + stage * kStage;
#pragma unroll
            for (int h = 0; h < KH; ++h) {
#pragma unroll
                for (int t = 0; t < MT; ++t) b[t][h] = *reinterpret_cast<const bf16x8_t*>(p + 2048 * (RT + t) + (place ^ (64 * h)));
#pragma unroll
                for (int r = 0; r < kTiles; ++r) a[r][h] = *reinterpret_cast<const bf16x8_t*>(p + 2048 * (first + r) + (place ^ (64 * h)));
            }
            if (s + D - 1 < steps) request(free);
            __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");     // read before the next barrier
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int h = 0; h < KH; ++h)
#pragma unroll
                for (int r = 0; r < kTiles; ++r)
#pragma unroll
                    for (int t = 0; t < MT; ++t) acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[r][h], b[t][h], acc[r][t], 0, 0, 0);
            stage = stage + 1 == D ? 0 : stage + 1;
            free = free + 1 == D ? 0 : free + 1;
        };
        int s = 0;
        for (; s + D - 2 < steps; ++s) step(s, std::integral_constant<int, D - 2>{});
        last_steps<D - 3>(s, step);
    }
    template <int B, class Step>
    __device__ __forceinline__ void last_steps(int s, Step& step) {
        if constexpr (B >= 0) {
            if (s + B == steps - 1) step(s++, std::integral_constant<int, B>{});
            last_steps<B - 1>(s, step);
        }
    }
};

// The product of RT tiles of weight rows and up to 16 MT rows of the batch by a workgroup: f(r, t, sum) gets tile r of the weights, t of the batch in the layout of
// stream_product, by some wavefront.  lds: SharedStream<RT, MT>::kRing bytes
template <int RT, int MT, class Weights, class Batch, class F>
__device__ __forceinline__ void shared_product(int k, int turn, unsigned char* lds, Weights weights, Batch batch, F f) {
    using Stream = SharedStream<RT, MT>;
    constexpr int TW = Stream::kTiles, WR = Stream::WR, WK = 4 / WR;
    static_assert(WK == 1 || 4096 * TW * MT <= Stream::kRing, "the sums fit the ring");
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wr = wave % WR;
    Stream stream(k, turn, wave, lds, weights, batch);
    f32x4_t acc[TW][MT];
#pragma unroll
    for (int r = 0; r < TW; ++r)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[r][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    stream.product(wave, lds, acc);
    auto finish = [&](int r, int t, f32x4_t sum) { f(wr * TW + r, t, sum); };
    if constexpr (WK == 1) {
#pragma unroll
        for (int r = 0; r < TW; ++r)
#pragma unroll
            for (int t = 0; t < MT; ++t) finish(r, t, acc[r][t]);
    } else {
        stream_reduce<TW, MT, WK>(acc, wave / WR, lds + wr * (1024 * WK * TW * MT), finish);
    }
}
