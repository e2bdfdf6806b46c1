// Device helpers shared by the multigrid kernels (mg_kernels.hip, mg_pass.hip, mg_coarse.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "mg_layout.h"

namespace sr {

// r / d with a float reciprocal and one correction step, exact for r < 2^24
__device__ inline unsigned fdivu(unsigned r, unsigned d, float inv) {
    unsigned q = (unsigned)((float)r * inv);
    int rem = (int)r - (int)(q * d);
    q += (unsigned)(rem >= (int)d) - (unsigned)(rem < 0);
    return q;
}

// t = (a * n1 + b) * n2 + c for t < 2^24, split with float-reciprocal divisions (fdivu) instead of
// integer divisions: the single-workgroup kernels are bound by their VALU issue rate
struct Div3 {
    unsigned n1, n2;
    float i1, i2;
};
__device__ inline Div3 div3(int n1, int n2) {
    return Div3{(unsigned)n1, (unsigned)n2, 1.0f / (float)n1, 1.0f / (float)n2};
}
__device__ inline void split3(const Div3 &D, int t, int &a, int &b, int &c) {
    unsigned r = fdivu((unsigned)t, D.n2, D.i2);
    c = t - (int)(r * D.n2);
    unsigned q = fdivu(r, D.n1, D.i1);
    b = (int)(r - q * D.n1);
    a = (int)q;
}

// Diagonal of the 7-point operator at a node from the three directions' coefficient quadruples
// (c+, c-, c0, pad).  The FP64 quadruples store c0 = c+ + c- (rounded once, at set-up), so the sum
// is formed from c+ and c-, which the stencil loads anyway, with the same value as from c0; the FP32
// quadruples hold each value rounded separately and use c0.
template <typename T>
__device__ __forceinline__ T diag3(const T *X, const T *Y, const T *Z) {
    if constexpr (sizeof(T) == 8) return (X[0] + X[1]) + (Y[0] + Y[1]) + (Z[0] + Z[1]);
    else return X[2] + Y[2] + Z[2];
}

// Face-ghost images of an updated node: a node whose padded index is the source of a ghost of a
// periodic / mirror / anti direction writes that ghost (same colour, so no other thread of this
// half sweep reads it).  Edge and corner ghosts are not read by the 7-point stencil.
template <typename T>
__device__ inline void write_images(const Lay &L, T *u, int ip, int jp, int kp, T v, const Bc &bc) {
    int n[3] = {L.nx, L.ny, L.nz};
    int p[3] = {ip, jp, kp};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        int r = bc.rule[d];
        if (r > G_ANTI) continue;
        T w = (r == G_ANTI) ? -v : v;
        int g0 = ghost_src(r, 0, n[d]), g1 = ghost_src(r, n[d] + 1, n[d]);
        if (p[d] == g0) {
            int q[3] = {p[0], p[1], p[2]};
            q[d] = 0;
            u[lay_idx(L, q[0], q[1], q[2])] = w;
        }
        if (p[d] == g1) {
            int q[3] = {p[0], p[1], p[2]};
            q[d] = n[d] + 1;
            u[lay_idx(L, q[0], q[1], q[2])] = w;
        }
    }
}

}  // namespace sr
