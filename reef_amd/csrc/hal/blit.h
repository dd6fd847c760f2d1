// Arguments of the library's own copy kernel (hal/blit.hip).
#pragma once
#include <stdint.h>

constexpr unsigned kBlitRanges = 8, kBlitBlock = 4096;   // bytes a workgroup copies
struct BlitArgs {
    struct {
        const char* src;
        char* dst;          // both on 16 bytes
        uint32_t bytes, end;   // end: first workgroup of the next range
    } range[kBlitRanges];
    uint32_t ranges;
};
