// How the recurrences over prompts cut a portion into segments.  The kernels of the segments, the kernel that joins their states and the host, which counts
// their records, have to agree.
#pragma once
#include <hip/hip_runtime.h>

// Tokens of a segment of a portion of `count`: as many segments as `most` tokens each would make, all of one length (a multiple of `chunk`, as `most` is) but
// for the last one's rest, so that a portion a little longer than `most` does not leave a workgroup with almost nothing.  Never more than `most`, and never
// more segments than a portion of the longest count has.
__device__ __forceinline__ int own_segment(int count, int most, int chunk) {
    const int segs = (count + most - 1) / most;
    return segs > 1 ? ((count + segs - 1) / segs + chunk - 1) / chunk * chunk : most;
}
