// How the recurrences over prompts cut a portion into segments, and in which order workgroups take the portions of a batch.  The kernels of the segments, the
// kernel that joins their states and the host, which counts their records, have to agree.
#pragma once
#include <hip/hip_runtime.h>

// Tokens of a segment of a portion of `count`: as many segments as `most` tokens each would make, all of one length (a multiple of `chunk`, as `most` is) but
// for the last one's rest, so that a portion a little longer than `most` does not leave a workgroup with almost nothing.  Never more than `most`, and never
// more segments than a portion of the longest count has.
__device__ __forceinline__ int own_segment(int count, int most, int chunk) {
    const int segs = (count + most - 1) / most;
    return segs > 1 ? ((count + segs - 1) / segs + chunk - 1) / chunk * chunk : most;
}

// Portions are walked token by token, so a batch is done when its longest one is, and workgroups start in the order of their numbers: a long portion that
// starts late, or beside another long one on the same compute unit, is waited for by itself.  So the longest go first, one workgroup to every compute unit, and
// the others in falling order behind them; the first ones rise, so that where a unit holds two workgroups, the longest of the others meets the shortest of
// the first.  6 portions of 900 to 3700 tokens, us, as they lie / in this order / falling throughout: state space of 64 heads 287 / 272 / 285.  As they
// lie where every workgroup has a compute unit to itself, where long ones are cut into segments, and where many short ones even out and are walked in little
// more time than it takes to find out whose turn it is (64 of 61 to 94 tokens, delta rule of 16 heads 188 / 199; 52 of 129 to 311, state space of 64 heads
// 231 / 236; but 22 of 397 to 737, retention of 16 heads 150 / 123).
struct Turns { int portions, first; };             // first: portions of the first round; 0: as they lie
static inline Turns turns_of(int64_t portions, int64_t groups_each, int64_t tokens) {
    constexpr int64_t kUnits = 256;
    if (portions < 2 || portions > 64 || portions * groups_each <= kUnits || tokens < 8 * portions * portions) return Turns{(int)portions, 0};
    const int64_t n = kUnits / groups_each;
    return Turns{(int)portions, (int)(n < 1 ? 1 : n)};
}
// The portion that workgroups number `turn` serve.  `spans`: four numbers per portion, the second its length.
__device__ __forceinline__ int portion_of_turn(const int32_t* spans, Turns t, int turn) {
    if (t.first == 0) return turn;
    const int lane = threadIdx.x & 63, mine = lane < t.portions ? spans[4 * lane + 1] : 0;
    int longer = 0;
    for (int i = 0; i < t.portions; ++i) {
        const int other = __builtin_amdgcn_readlane(mine, i);
        longer += other > mine || (other == mine && i < lane);
    }
    const uint64_t found = __ballot(lane < t.portions && longer == (turn < t.first ? t.first - 1 - turn : turn));
    return __builtin_ctzll(found);                 // ranks are a permutation: exactly one
}
