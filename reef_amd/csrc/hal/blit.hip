// Copies a few ranges in one launch: a recorded pass ends with one that puts a model's results into host
// memory.  The runtime's copy of 4 KB out of device memory takes 11.5 us for each of them; behind the
// last kernel of a pass the launch costs 2 us for all.
#include <hip/hip_runtime.h>

#include "hal/blit.h"

extern "C" __global__ void __launch_bounds__(256) reef_blit_ranges(BlitArgs a) {
    const uint32_t b = blockIdx.x;
    uint32_t r = 0, first = 0;
    while (r + 1 < a.ranges && b >= a.range[r].end) first = a.range[r++].end;
    const uint32_t at = (b - first) * kBlitBlock + threadIdx.x * 16u, bytes = a.range[r].bytes;
    if (at + 16u <= bytes) *(float4*)(a.range[r].dst + at) = *(const float4*)(a.range[r].src + at);
    else
        for (uint32_t i = at; i < bytes; ++i) a.range[r].dst[i] = a.range[r].src[i];
}
