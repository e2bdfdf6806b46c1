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

// The six neighbour products of L u.  The roundings are written out (x- rounded, the others fused onto it in
// order): left to the compiler they came out differently from kernel to kernel, and a refinement's
// iterates then differ by FP32 roundings, which a poorly conditioned grid amplifies to 1e-8.
template <typename T>
__device__ __forceinline__ T six(T x0, T xp, T x1, T xm, T y0, T yp, T y1, T ym, T z0, T zp, T z1, T zm) {
    T s = x1 * xm;
    s = fma(x0, xp, s);
    s = fma(y0, yp, s);
    s = fma(y1, ym, s);
    s = fma(z0, zp, s);
    return fma(z1, zm, s);
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

__device__ inline double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
__device__ inline double wave_max(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    return v;
}

// Whether this workgroup is the last of the grid to get here (a device-scope counter, zero before the
// launch, which the caller resets): what the others wrote before is then visible to it.
__device__ inline bool last_block_done(unsigned *counter) {
    __shared__ bool last;
    __syncthreads();
    if (threadIdx.x == 0) {
        __threadfence();
        last = atomicAdd(counter, 1u) == gridDim.x - 1;
    }
    __syncthreads();
    if (last) __threadfence();
    return last;
}

// alpha, beta of the step from the block sums; coef = {alpha, beta, (r q), (q q), (q p), (r p), (p p)}.
// When the orthogonalised direction has lost most of its norm to cancellation (or there is no
// previous direction) the step falls back to the minimal-residual step along e.
__device__ inline void gcr_coef_from(const double (&t)[5], double *coef) {
    double rq = t[0], qq = t[1], qp = t[2], rp = t[3], pp = t[4];
    double beta = pp > 0.0 ? qp / pp : 0.0;
    double qn = qq - 2.0 * beta * qp + beta * beta * pp;
    if (!(qn >= 1e-3 * qq)) {
        beta = 0.0;
        qn = qq;
    }
    double alpha = qn > 0.0 ? (rq - beta * rp) / qn : 0.0;
    coef[0] = alpha;
    coef[1] = beta;
    for (int i = 0; i < 5; i++) coef[2 + i] = t[i];
}

}  // namespace sr
