// Device helpers shared by the multigrid kernels (mg_kernels.hip, mg_pass.hip).
#pragma once

#include <hip/hip_runtime.h>

namespace sr {

// r / d with a float reciprocal and one correction step, exact for r < 2^24
__device__ inline unsigned fdivu(unsigned r, unsigned d, float inv) {
    unsigned q = (unsigned)((float)r * inv);
    int rem = (int)r - (int)(q * d);
    q += (unsigned)(rem >= (int)d) - (unsigned)(rem < 0);
    return q;
}

}  // namespace sr
