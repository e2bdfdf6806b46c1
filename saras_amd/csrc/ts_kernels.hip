// gfx950 kernels of the hydro time step on the reference's padded layout (k fastest).
//
//   k_deriv        derivative::calcDerivative1_* / calcDerivative2* (lib/field/derivative.cc:121-243)
//   k_build_rhs    hydro_d3.cc:259-300 fused, the three velocity components together: computeDiff / Re, computeNLin
//                  (vfield.cc:104-253), - grad P (sfield.cc:155-171), * dt, + V
//   k_jacobi_march one Jacobi sweep of solveVx/Vy/Vz (hydro_d3.cc:375-391) into the second buffer, with
//                  or without the residual of the current iterate from the same loads
//   k_jacobi_res   the convergence residual of the same routines (hydro_d3.cc:396-410), max-reduced
//   k_ghost_ops    a wave of ghost / wall operations (mpidata::syncData, lib/boundary/*.cc); k_ghost_pair
//                  syncData and the z walls in one launch
//   k_divergence   vfield::divergence (vfield.cc:299-320), optionally scaled (mgRHS = div / dt)
//   k_project      P += Pp and V -= dt grad Pp (hydro_d3.cc:354-362)
//   k_energy       tseries energy (tseries.cc:158-169), deterministic two-pass sum
//
// Field shapes (core sizes) follow field.h: P on nodes (N in every direction), V_c on faces in
// direction c (N-1) and nodes in the other two.  Derivative alignment: centred,
// out(r) = metric(r) (F(r+1) - F(r-1)) / (2h) over the core range along the direction.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <utility>

#include "columns.h"

namespace sr {

constexpr int kJacobiThreads = 1024;

__device__ inline long fidx(const FShape &f, int i, int j, int k) {
    return ((long)(i + 1) * (f.n[1] + 2) + (j + 1)) * (f.n[2] + 2) + (k + 1);
}

// metric arrays: [dim][node?0:1][q] with q 0 coordinate, 1 xi_x, 2 xi_xx, 3 xi_x^2, index -1 at 0
__device__ inline double metv(const Metrics &M, int d, int node, int q, int i) {
    return M.m[d][node ? 0 : 1][q][i + 1];
}

// ------------------------------------------------------------------------------------------------
// derivatives (for parity tests; the fused step kernel carries its own copies)
// ------------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_deriv(FShape f, Metrics M, const double *__restrict__ F,
                                               double *__restrict__ out, int order, int d, double ih) {
    int lo[3] = {-1, -1, -1}, sz[3] = {f.n[0] + 2, f.n[1] + 2, f.n[2] + 2};
    lo[d] = 0;
    sz[d] = f.n[d];
    long total = (long)sz[0] * sz[1] * sz[2];
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= total) return;
    int k = (int)(t % sz[2]) + lo[2];
    long r = t / sz[2];
    int j = (int)(r % sz[1]) + lo[1];
    int i = (int)(r / sz[1]) + lo[0];
    long st[3] = {(long)(f.n[1] + 2) * (f.n[2] + 2), (long)(f.n[2] + 2), 1};
    long c = fidx(f, i, j, k);
    int q = d == 0 ? i : d == 1 ? j : k;
    if (order == 1) {
        double v = (F[c + st[d]] - F[c - st[d]]) / 2.0;
        v *= ih;
        out[c] = metv(M, d, f.s[d], 1, q) * v;
    } else {
        double ih2 = ih * ih;
        double tmp = (F[c + st[d]] - F[c - st[d]]) / 2.0 * ih;
        double sec = (F[c + st[d]] - 2.0 * F[c] + F[c - st[d]]) * ih2;
        out[c] = metv(M, d, f.s[d], 2, q) * tmp + 0.5 * metv(M, d, f.s[d], 3, q) * sec;
    }
}

// ------------------------------------------------------------------------------------------------
// nseRHS of the three velocity components
// ------------------------------------------------------------------------------------------------
// All three components in one march (columns.h): the velocities and P are read once for the three, which
// move 7 arrays (8 with a temperature).  129^3: 104 -> 39 us.
template <bool BUOY>
__global__ void __launch_bounds__(kColThreads) k_build_rhs(ColGeo G, VelGeo S, Metrics M, const double *__restrict__ Vx,
                                                   const double *__restrict__ Vy, const double *__restrict__ Vz,
                                                   const double *__restrict__ P, double *__restrict__ Hx,
                                                   double *__restrict__ Hy, double *__restrict__ Hz, ColMet W,
                                                   double inverseRe, double dt, const double *__restrict__ T, double Fb) {
    // core entries get the right-hand side, pads a copy of V (the reference forms nseRHS over the
    // whole padded array, with zero terms outside the core)
    const Col C = column(G);   // core planes
    // x metrics of a face and of a node: first differences (a quarter of it on nodes, whose advecting
    // velocity is a mean of four), and the two parts of the second
    __shared__ double lx[6][kColPlanes];
    for (int q = (int)threadIdx.x; q < C.i1 - C.i0; q += kColThreads) {
        const int fi = min(C.i0 + q, S.N[0] - 2), ni = C.i0 + q;
        lx[0][q] = met1(M, 0, 0, fi, W.ih[0]);
        lx[1][q] = met2(M, 0, 0, fi, W.ih[0]);
        lx[2][q] = met3(M, 0, 0, fi, W.ih[0], W.half);
        lx[3][q] = 0.25 * met1(M, 0, 1, ni, W.ih[0]);
        lx[4][q] = met2(M, 0, 1, ni, W.ih[0]);
        lx[5][q] = met3(M, 0, 1, ni, W.ih[0], W.half);
    }
    __syncthreads();
    const long sx = S.sx(), sy = S.sy(), sz = S.sz();
    if ((long)C.t >= sx) return;
    const int row = S.N[2] + 2, rz = S.N[2] + 1;
    const int jp = (int)(C.t / (unsigned)row), kp = (int)C.t - jp * row;   // padded
    const bool in = jp >= 1 && kp >= 1 && jp <= S.N[1] && kp <= S.N[2];
    const bool hasy = jp <= S.N[1], hasz = kp <= S.N[2];             // rows and entries that Vy and Vz have
    const bool cy = in && jp < S.N[1], cz = in && kp < S.N[2];       // core of Vy and Vz
    // a pad entry takes part in the loads of the core entry next to it
    const int j = min(max(jp, 1), S.N[1]) - 1, k = min(max(kp, 1), S.N[2]) - 1;
    const unsigned o = (unsigned)((j + 1) * row + k + 1) * 8u, oz = (unsigned)((j + 1) * rz + k + 1) * 8u;
    const unsigned po = C.t * 8u, poz = (unsigned)(jp * rz + kp) * 8u;
    const int jf = min(j, S.N[1] - 2), kf = min(k, S.N[2] - 2);
    const double yf1 = met1(M, 1, 0, jf, W.ih[1]), yf2 = met2(M, 1, 0, jf, W.ih[1]), yf3 = met3(M, 1, 0, jf, W.ih[1], W.half);
    const double yn1 = 0.25 * met1(M, 1, 1, j, W.ih[1]), yn2 = met2(M, 1, 1, j, W.ih[1]), yn3 = met3(M, 1, 1, j, W.ih[1], W.half);
    const double zf1 = met1(M, 2, 0, kf, W.ih[2]), zf2 = met2(M, 2, 0, kf, W.ih[2]), zf3 = met3(M, 2, 0, kf, W.ih[2], W.half);
    const double zn1 = 0.25 * met1(M, 2, 1, k, W.ih[2]), zn2 = met2(M, 2, 1, k, W.ih[2]), zn3 = met3(M, 2, 1, k, W.ih[2], W.half);
    // the pad planes on either side
    if (C.i0 == 0) {
        std_(Hx, po, ldd(Vx, po));
        if (hasy) std_(Hy, po, ldd(Vy, po));
        if (hasz) std_(Hz, poz, ldd(Vz, poz));
    }
    if (C.i1 == S.N[0]) {
        if (hasy) std_(Hy + (S.N[0] + 1) * sy, po, ldd(Vy + (S.N[0] + 1) * sy, po));
        if (hasz) std_(Hz + (S.N[0] + 1) * sz, poz, ldd(Vz + (S.N[0] + 1) * sz, poz));
    }
    const long i0 = C.i0 + 1;
    Vx += i0 * sx;
    Vy += i0 * sy;
    Vz += i0 * sz;
    P += i0 * sx;
    if (BUOY) T += i0 * sx;
    Hx += i0 * sx;
    Hy += i0 * sy;
    Hz += i0 * sz;
    Vels v;
    vels_begin(v, Vx, Vy, Vz, S, o, oz, true);
    double p = ldd(P, o);
    for (int i = C.i0; i < C.i1; ++i) {
        const bool cx = i < S.N[0] - 1;
        vels_load(v, Vx, Vy, Vz, S, o, oz, true, !cx);
        const double pn = ldd(P + sx, o), pj = ldd(P + row, o), pk = ldd(P + 1, o);
        const double *const m = &lx[0][i - C.i0];
        const double xf1 = m[0], xf2 = m[kColPlanes], xf3 = m[2 * kColPlanes];
        const double xn1 = m[3 * kColPlanes], xn2 = m[4 * kColPlanes], xn3 = m[5 * kColPlanes];
        // computeDiff / Re, - computeNLin, - grad P on the component's faces (its metric over h is twice
        // that of a centred difference), * dt, + V
        const Cross ux = cross_x(v), uy = cross_y(v), uz = cross_z(v);
        double ax = inverseRe * diffuse(0.0, ux, xf2, xf3, yn2, yn3, zn2, zn3);
        double ay = inverseRe * diffuse(0.0, uy, xn2, xn3, yf2, yf3, zn2, zn3);
        double az = inverseRe * diffuse(0.0, uz, xn2, xn3, yn2, yn3, zf2, zf3);
        ax = advect<0>(ax, v, ux, xf1, yn1, zn1);
        ay = advect<1>(ay, v, uy, xn1, yf1, zn1);
        az = advect<2>(az, v, uz, xn1, yn1, zf1);
        // buoyantForce::addForcing: the z face between nodes k and k + 1 gets Fb times their mean
        if (BUOY) az += Fb * ((ldd(T, o) + ldd(T + 1, o)) / 2.0);
        ax = dt * (ax - 2.0 * xf1 * (pn - p)) + v.x;
        ay = dt * (ay - 2.0 * yf1 * (pj - p)) + v.y;
        az = dt * (az - 2.0 * zf1 * (pk - p)) + v.z;
        double vx = v.x, vy = v.y, vz = v.z;
        if (!in) {
            vx = ldd(Vx, po);
            if (hasy) vy = ldd(Vy, po);
            if (hasz) vz = ldd(Vz, poz);
        }
        std_(Hx, po, in && cx ? ax : vx);
        if (hasy) std_(Hy, po, cy ? ay : vy);
        if (hasz) std_(Hz, poz, cz ? az : vz);
        vels_next(v);
        p = pn;
        Vx += sx;
        Vy += sy;
        Vz += sz;
        P += sx;
        if (BUOY) T += sx;
        Hx += sx;
        Hy += sy;
        Hz += sz;
    }
}

// ------------------------------------------------------------------------------------------------
// Jacobi viscous solve of component c over its bulk
// ------------------------------------------------------------------------------------------------
// G = J(V) over the bulk and 0 elsewhere (the reference's guess field is written on the bulk only and
// copied whole into V); with RES also the convergence residual of V itself, as k_jacobi_res: the sweep
// that follows an iterate and that iterate's residual read the same neighbours.
//
// A march along x (columns.h).  The residual's maximum is combined by device-scope atomics, and the last
// workgroup leaves it in out and in the host's mirror and clears sync for the next launch, so that no
// second launch and no copy follow.  Workgroups of 1024 keep the atomics few.  129^3, us: 15.1 the sweep
// alone as before, 17.5 + 4.5 + 3 (maximum, copy) -> 17.7 with the residual (21.6 with one counter for
// all workgroups); V, R and G are 52 MB that the last-level cache holds.
template <bool RES>
__global__ void __launch_bounds__(kJacobiThreads) k_jacobi_march(ColGeo C0, FShape f, Metrics M, Bulk B,
                                                                 const double *__restrict__ V, const double *__restrict__ R,
                                                                 double *__restrict__ G, JacobiCoef J,
                                                                 JacobiSync *sync, unsigned long long *out,
                                                                 unsigned long long *host) {
    const Col C = column(C0);   // padded planes
    __shared__ double lx[kColPlanes];
    for (int q = (int)threadIdx.x; q < C.i1 - C.i0; q += kJacobiThreads)
        lx[q] = met(M, 0, J.ms[0], 3, max(0, min(C.i0 - 1 + q, f.n[0] - 1)));
    __syncthreads();
    const int row = f.n[2] + 2;
    const long ps = (long)(f.n[1] + 2) * row;
    double e = 0.0;
    if ((long)C.t < ps) {
        const int jp = (int)(C.t / (unsigned)row), kp = (int)C.t - jp * row;
        // an entry outside the bulk takes part in the loads of the bulk entry next to it
        const int j = min(max(jp - 1, B.lo[1]), B.hi[1]), k = min(max(kp - 1, B.lo[2]), B.hi[2]);
        const bool in = j == jp - 1 && k == kp - 1;
        const unsigned po = C.t * 8u, o = (unsigned)((j + 1) * row + k + 1) * 8u;
        const double my = met(M, 1, J.ms[1], 3, j), mz = met(M, 2, J.ms[2], 3, k);
        const int last = f.n[0] + 1;
        double xm = ldd(V + max(C.i0 - 1, 0) * ps, o), c = ldd(V + C.i0 * ps, o);
        for (int p0 = C.i0; p0 < C.i1; p0 += kColAhead) {
            double xp[kColAhead], rq[kColAhead], yp[kColAhead], ym[kColAhead], zp[kColAhead], zm[kColAhead];
#pragma unroll
            for (int u = 0; u < kColAhead; u++) {
                const double *const v = V + min(p0 + u, C.i1 - 1) * ps;
                xp[u] = ldd(V + min(p0 + u + 1, last) * ps, o);
                rq[u] = ldd(R + min(p0 + u, C.i1 - 1) * ps, o);
                yp[u] = ldd(v + row, o);
                ym[u] = ldd(v - row, o);
                zp[u] = ldd(v + 1, o);
                zm[u] = ldd(v - 1, o);
            }
            loaded(xp);
            loaded(rq);
#pragma unroll
            for (int u = 0; u < kColAhead; u++) {
                const int p = p0 + u;
                if (p >= C.i1) break;
                const double mx = lx[p - C.i0];
                const bool bulk = in && p - 1 >= B.lo[0] && p - 1 <= B.hi[0];
                const double a = J.hy2hz2 * mx * (xp[u] + xm) + J.hz2hx2 * my * (yp[u] + ym[u]) + J.hx2hy2 * mz * (zp[u] + zm[u]);
                const double d = J.hy2hz2 * mx + J.hz2hx2 * my + J.hx2hy2 * mz;
                const double g = (a * J.rA + rq[u]) / (1.0 + d * J.rD);
                std_(G + p * ps, po, bulk ? g : 0.0);
                if (RES) {
                    const double lap = c - (mx * (xp[u] - 2.0 * c + xm) * J.ih2[0] + my * (yp[u] - 2.0 * c + ym[u]) * J.ih2[1] +
                                            mz * (zp[u] - 2.0 * c + zm[u]) * J.ih2[2]) * J.lapS;
                    e = fmax(e, bulk ? fabs(lap - rq[u]) : 0.0);
                }
                xm = c;
                c = xp[u];
            }
        }
    }
    if (RES) {
        __shared__ double s[kJacobiThreads / 64];
#pragma unroll
        for (int w = 32; w > 0; w >>= 1) e = fmax(e, __shfl_xor(e, w, 64));
        if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = e;
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int w = 1; w < kJacobiThreads / 64; w++) e = fmax(e, s[w]);
            // the bits of non-negative doubles are in their order; one maximum per group of workgroups
            arrived(__hip_atomic_fetch_max(sync->max + 16 * grid_group(), (unsigned long long)__double_as_longlong(e),
                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
            if (grid_last(sync->words)) {
                unsigned long long m[kGridGroups], r = 0;
#pragma unroll
                for (int w = 0; w < kGridGroups; w++)
                    m[w] = __hip_atomic_exchange(sync->max + 16 * w, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
                for (int w = 0; w < kGridGroups; w++) r = max(r, m[w]);
                *out = r;
                if (host) {
                    *host = r;
                    __threadfence_system();
                }
            }
        }
    }
}

// max over the bulk of |V - 0.5 dt/Re lap V - R|: each logical block takes one contiguous range of
// the bulk (32-bit index arithmetic), so that an XCD's blocks cover neighbouring planes; one maximum
// per block into part; k_jacobi_res_final reduces them (a maximum: the same whatever the order)
__global__ void __launch_bounds__(256) k_jacobi_res(FShape f, Metrics M, Bulk B, const double *__restrict__ V,
                                                    const double *__restrict__ R, JacobiCoef J,
                                                    double *__restrict__ part) {
    unsigned sz1 = (unsigned)(B.hi[1] - B.lo[1] + 1), sz2 = (unsigned)(B.hi[2] - B.lo[2] + 1);
    unsigned total = (unsigned)(B.hi[0] - B.lo[0] + 1) * sz1 * sz2;
    long st[3] = {(long)(f.n[1] + 2) * (f.n[2] + 2), (long)(f.n[2] + 2), 1};
    const unsigned lb = xcd_block();
    // range of a block: a whole number of 256-entry strips
    const unsigned strips = (total + 255u) / 256u;
    const unsigned per = (strips + gridDim.x - 1u) / gridDim.x;
    const unsigned t0 = lb * per * 256u;
    const unsigned t1 = min(total, t0 + per * 256u);
    double e = 0.0;
    for (unsigned t = t0 + threadIdx.x; t < t1; t += 256u) {
        unsigned r = t / sz2;
        int k = (int)(t - r * sz2) + B.lo[2];
        unsigned i0 = r / sz1;
        int j = (int)(r - i0 * sz1) + B.lo[1];
        int i = (int)i0 + B.lo[0];
        long q = fidx(f, i, j, k);
        double mx = metv(M, 0, J.ms[0], 3, i), my = metv(M, 1, J.ms[1], 3, j), mz = metv(M, 2, J.ms[2], 3, k);
        double lap = V[q] - (mx * (V[q + st[0]] - 2.0 * V[q] + V[q - st[0]]) * J.ih2[0] +
                             my * (V[q + st[1]] - 2.0 * V[q] + V[q - st[1]]) * J.ih2[1] +
                             mz * (V[q + 1] - 2.0 * V[q] + V[q - 1]) * J.ih2[2]) * J.lapS;
        e = fmax(e, fabs(lap - R[q]));
    }
    __shared__ double s[4];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) e = fmax(e, __shfl_xor(e, o, 64));
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = e;
    __syncthreads();
    if (threadIdx.x == 0) part[lb] = fmax(fmax(s[0], s[1]), fmax(s[2], s[3]));
}

// maximum of the block maxima, stored as the bit pattern of the double; one block of up to 1024
// threads (a maximum: the same whatever the order)
__global__ void __launch_bounds__(1024) k_jacobi_res_final(const double *__restrict__ part, int n,
                                                           unsigned long long *__restrict__ out) {
    double m = 0.0;
#pragma unroll 8
    for (int q = threadIdx.x; q < n; q += blockDim.x) m = fmax(m, part[q]);
    __shared__ double s[16];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        double r = s[0];
        for (int w = 1; w < (int)(blockDim.x >> 6); w++) r = fmax(r, s[w]);
        out[0] = (unsigned long long)__double_as_longlong(r);
    }
}

// ------------------------------------------------------------------------------------------------
// ghost / wall operations: dst = a * F(src) + b over a plane (dim fixed) or a z-line (x, y fixed)
// ------------------------------------------------------------------------------------------------
// operation and place of thread t of a wave: destination p, source s; false past the last one
__device__ inline bool ghost_place(const GhostWave &W, long t, int &o, int (&p)[3], int (&s)[3]) {
    o = 0;
    while (o < W.nops && t >= W.ops[o].count) {
        t -= W.ops[o].count;
        o++;
    }
    if (o >= W.nops) return false;
    const GhostOp &op = W.ops[o];
    if (op.kind == 0) {      // plane: fixed index along op.dim, ranges on the other two
        const int na = op.hi[0] - op.lo[0] + 1;
        const int q = (int)((unsigned)t / (unsigned)na);
        const int ia = op.lo[0] + (int)t - q * na, ib = op.lo[1] + q;
        p[0] = s[0] = ia;
        p[1] = s[1] = op.dim == 0 ? ia : ib;
        p[2] = s[2] = ib;
        if (op.dim == 0) { p[0] = op.dst[0]; s[0] = op.src[0]; }
        if (op.dim == 1) { p[1] = op.dst[0]; s[1] = op.src[0]; }
        if (op.dim == 2) { p[2] = op.dst[0]; s[2] = op.src[0]; }
    } else {                 // z-line at fixed (x, y)
        p[2] = s[2] = op.lo[0] + (int)t;
        p[0] = op.dst[0]; p[1] = op.dst[1];
        s[0] = op.src[0]; s[1] = op.src[1];
    }
    return true;
}

__global__ void __launch_bounds__(256) k_ghost_ops(FShape f, double *__restrict__ F, GhostWave W) {
    int o, p[3], s[3];
    if (!ghost_place(W, (long)blockIdx.x * blockDim.x + threadIdx.x, o, p, s)) return;
    const GhostOp &op = W.ops[o];
    const double v = op.a == 0.0 ? 0.0 : op.a * F[fidx(f, s[0], s[1], s[2])];
    F[fidx(f, p[0], p[1], p[2])] = v + op.b;
}

// Two waves in one launch: copies onto x and y pads (S) and then z walls (W).  A wall entry over a pad
// takes its value from where S would have copied the pad from, and S leaves out the planes that W
// writes, so that neither reads what the other writes.
__global__ void __launch_bounds__(256) k_ghost_pair(FShape f, double *__restrict__ F, GhostWave S, GhostWave W, long ns) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    int o, p[3], s[3];
    if (t < ns) {
        ghost_place(S, t, o, p, s);
        for (int q = 0; q < W.nops; q++)
            if (p[2] == W.ops[q].dst[0]) return;
        F[fidx(f, p[0], p[1], p[2])] = F[fidx(f, s[0], s[1], s[2])];
        return;
    }
    if (!ghost_place(W, t - ns, o, p, s)) return;
    const double a = W.ops[o].a, b = W.ops[o].b;
    double v = 0.0;
    if (a != 0.0) {
        for (int q = 0; q < S.nops; q++) {
            const GhostOp &c = S.ops[q];
            if (c.kind == 1) {
                if (s[0] == c.dst[0] && s[1] == c.dst[1] && s[2] >= c.lo[0] && s[2] <= c.hi[0]) {
                    s[0] = c.src[0];
                    s[1] = c.src[1];
                    break;
                }
            } else {
                const int e = c.dim == 0 ? s[1] : s[0];
                if ((c.dim == 0 ? s[0] : s[1]) == c.dst[0] && e >= c.lo[0] && e <= c.hi[0] && s[2] >= c.lo[1] && s[2] <= c.hi[1]) {
                    if (c.dim == 0) s[0] = c.src[0];
                    else s[1] = c.src[0];
                    break;
                }
            }
        }
        v = a * F[fidx(f, s[0], s[1], s[2])];
    }
    F[fidx(f, p[0], p[1], p[2])] = v + b;
}

// ------------------------------------------------------------------------------------------------
// temperature right-hand side: core nodes T + dt (kappa sum d2 T - sum_d Vbar_d dT/dx_d), pads T
// ------------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(kColThreads) k_build_trhs(ColGeo G, VelGeo S, Metrics M, const double *__restrict__ Vx,
                                                    const double *__restrict__ Vy, const double *__restrict__ Vz,
                                                    const double *__restrict__ T, double *__restrict__ R, ColMet W,
                                                    double kappa, double dt) {
    const Col C = column(G);   // padded planes
    __shared__ double lx[3][kColPlanes];
    for (int q = (int)threadIdx.x; q < C.i1 - C.i0; q += kColThreads) {
        const int i = max(0, min(C.i0 - 1 + q, S.N[0] - 1));
        lx[0][q] = 0.5 * met1(M, 0, 1, i, W.ih[0]);
        lx[1][q] = met2(M, 0, 1, i, W.ih[0]);
        lx[2][q] = met3(M, 0, 1, i, W.ih[0], W.half);
    }
    __syncthreads();
    const long sx = S.sx(), sy = S.sy(), sz = S.sz();
    if ((long)C.t >= sx) return;
    const int row = S.N[2] + 2, rz = S.N[2] + 1;
    const int jp = (int)(C.t / (unsigned)row), kp = (int)C.t - jp * row;
    const bool in = jp >= 1 && kp >= 1 && jp <= S.N[1] && kp <= S.N[2];
    const int j = min(max(jp, 1), S.N[1]) - 1, k = min(max(kp, 1), S.N[2]) - 1;
    const unsigned o = C.t * 8u, oz = (unsigned)(jp * rz + kp) * 8u;
    const double y1 = 0.5 * met1(M, 1, 1, j, W.ih[1]), y2 = met2(M, 1, 1, j, W.ih[1]), y3 = met3(M, 1, 1, j, W.ih[1], W.half);
    const double z1 = 0.5 * met1(M, 2, 1, k, W.ih[2]), z2 = met2(M, 2, 1, k, W.ih[2]), z3 = met3(M, 2, 1, k, W.ih[2], W.half);
    const double *t = T + C.i0 * sx;
    Cross u;
    u.xm = C.i0 > 0 ? ldd(t - sx, o) : 0.0;
    u.c = ldd(t, o);
    double xm = C.i0 > 0 ? ldd(Vx + (C.i0 - 1) * sx, o) : 0.0;
#pragma unroll 2
    for (int p = C.i0; p < C.i1; ++p, t += sx) {
        double v = u.c;
        u.xp = p <= S.N[0] ? ldd(t + sx, o) : 0.0;
        const double x = p <= S.N[0] ? ldd(Vx + p * sx, o) : 0.0;
        if (in && p >= 1 && p <= S.N[0]) {
            u.yp = ldd(t + row, o);
            u.ym = ldd(t - row, o);
            u.zp = ldd(t + 1, o);
            u.zm = ldd(t - 1, o);
            const double *const Y = Vy + p * sy, *const Z = Vz + p * sz;
            const int q = p - C.i0;
            double acc = kappa * diffuse(0.0, u, lx[1][q], lx[2][q], y2, y3, z2, z3);
            acc -= (x + xm) * (lx[0][q] * (u.xp - u.xm));
            acc -= (ldd(Y, o) + ldd(Y - row, o)) * (y1 * (u.yp - u.ym));
            acc -= (ldd(Z, oz) + ldd(Z - 1, oz)) * (z1 * (u.zp - u.zm));
            v = dt * acc + u.c;
        }
        std_(R + p * sx, o, v);
        xm = x;
        u.xm = u.c;
        u.c = u.xp;
    }
}

// Nusselt partials: per block sums of (volume) and (w T volume), w the mean of the two z faces
__global__ void __launch_bounds__(256) k_nusselt(FShape fp, FShape fz, Metrics M, const double *__restrict__ Vz,
                                                 const double *__restrict__ T, double h0, double h1, double h2,
                                                 double *__restrict__ part) {
    long total = (long)fp.n[0] * fp.n[1] * fp.n[2];
    const unsigned lb = xcd_block();
    long t = (long)lb * blockDim.x + threadIdx.x;
    double vol = 0.0, uzt = 0.0;
    if (t < total) {
        int k = (int)(t % fp.n[2]);
        long r = t / fp.n[2];
        int j = (int)(r % fp.n[1]);
        int i = (int)(r / fp.n[1]);
        double dv = (h0 / metv(M, 0, 0, 1, i)) * (h1 / metv(M, 1, 0, 1, j)) * (h2 / metv(M, 2, 0, 1, k));
        double w = (Vz[fidx(fz, i, j, k)] + Vz[fidx(fz, i, j, k - 1)]) / 2.0;
        vol = dv;
        uzt = w * T[fidx(fp, i, j, k)] * dv;
    }
    __shared__ double sv[4], su[4];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        vol += __shfl_xor(vol, o, 64);
        uzt += __shfl_xor(uzt, o, 64);
    }
    if ((threadIdx.x & 63) == 0) { sv[threadIdx.x >> 6] = vol; su[threadIdx.x >> 6] = uzt; }
    __syncthreads();
    if (threadIdx.x == 0) {
        double a = 0, b = 0;
        for (int w = 0; w < 4; w++) { a += sv[w]; b += su[w]; }
        part[2 * (long)lb] = a;
        part[2 * (long)lb + 1] = b;
    }
}

// ------------------------------------------------------------------------------------------------
// divergence over the node core (pads untouched), times `scale`
// ------------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_divergence(FShape fp, FShape fx, FShape fy, FShape fz, Metrics M,
                                                    const double *__restrict__ Vx, const double *__restrict__ Vy,
                                                    const double *__restrict__ Vz, double *__restrict__ out,
                                                    double h0, double h1, double h2, double scale, int scaled) {
    long total = (long)fp.n[0] * fp.n[1] * fp.n[2];
    const unsigned lb = xcd_block();
    long t = (long)lb * blockDim.x + threadIdx.x;
    if (t >= total) return;
    int k = (int)(t % fp.n[2]);
    long r = t / fp.n[2];
    int j = (int)(r % fp.n[1]);
    int i = (int)(r / fp.n[1]);
    double a = metv(M, 0, 1, 1, i) * (Vx[fidx(fx, i, j, k)] - Vx[fidx(fx, i - 1, j, k)]) / h0;
    double b = metv(M, 1, 1, 1, j) * (Vy[fidx(fy, i, j, k)] - Vy[fidx(fy, i, j - 1, k)]) / h1;
    double c = metv(M, 2, 1, 1, k) * (Vz[fidx(fz, i, j, k)] - Vz[fidx(fz, i, j, k - 1)]) / h2;
    double d = a + b + c;
    out[fidx(fp, i, j, k)] = scaled ? d * scale : d;
}

// ------------------------------------------------------------------------------------------------
// projection: V_c(core) -= dt * grad_c Pp  (pads of the gradient are zero, so pads of V are kept)
// ------------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_project(int c, FShape fc, FShape fp, Metrics M, const double *__restrict__ Pp,
                                                 double *__restrict__ V, double hc, double dt) {
    long total = (long)fc.n[0] * fc.n[1] * fc.n[2];
    const unsigned lb = xcd_block();
    long t = (long)lb * blockDim.x + threadIdx.x;
    if (t >= total) return;
    int k = (int)(t % fc.n[2]);
    long r = t / fc.n[2];
    int j = (int)(r % fc.n[1]);
    int i = (int)(r / fc.n[1]);
    int idx[3] = {i, j, k};
    long sp[3] = {(long)(fp.n[1] + 2) * (fp.n[2] + 2), (long)(fp.n[2] + 2), 1};
    long pq = fidx(fp, i, j, k);
    double g = metv(M, c, 0, 1, idx[c]) * (Pp[pq + sp[c]] - Pp[pq]) / hc;
    g *= dt;
    long q = fidx(fc, i, j, k);
    V[q] = V[q] - g;
}

__global__ void __launch_bounds__(256) k_fill_d(double *__restrict__ p, long n, double v) {
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) p[t] = v;
}

__global__ void __launch_bounds__(256) k_axpy_full(double *__restrict__ y, const double *__restrict__ x, long n) {
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) y[t] += x[t];
}

// ------------------------------------------------------------------------------------------------
// energy partials: per block sums of (volume) and (energy density * volume), fixed order
// ------------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_energy(FShape fp, FShape fx, FShape fy, FShape fz, Metrics M,
                                                const double *__restrict__ Vx, const double *__restrict__ Vy,
                                                const double *__restrict__ Vz, double h0, double h1, double h2,
                                                double *__restrict__ part) {
    long total = (long)fp.n[0] * fp.n[1] * fp.n[2];
    const unsigned lb = xcd_block();
    long t = (long)lb * blockDim.x + threadIdx.x;
    double vol = 0.0, en = 0.0;
    if (t < total) {
        int k = (int)(t % fp.n[2]);
        long r = t / fp.n[2];
        int j = (int)(r % fp.n[1]);
        int i = (int)(r / fp.n[1]);
        double dv = (h0 / metv(M, 0, 0, 1, i)) * (h1 / metv(M, 1, 0, 1, j)) * (h2 / metv(M, 2, 0, 1, k));
        double u = (Vx[fidx(fx, i - 1, j, k)] + Vx[fidx(fx, i, j, k)]) / 2.0;
        double v = (Vy[fidx(fy, i, j - 1, k)] + Vy[fidx(fy, i, j, k)]) / 2.0;
        double w = (Vz[fidx(fz, i, j, k - 1)] + Vz[fidx(fz, i, j, k)]) / 2.0;
        vol = dv;
        en = (u * u + v * v + w * w) * dv;
    }
    __shared__ double sv[4], se[4];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        vol += __shfl_xor(vol, o, 64);
        en += __shfl_xor(en, o, 64);
    }
    if ((threadIdx.x & 63) == 0) { sv[threadIdx.x >> 6] = vol; se[threadIdx.x >> 6] = en; }
    __syncthreads();
    if (threadIdx.x == 0) {
        double a = 0, b = 0;
        for (int w = 0; w < 4; w++) { a += sv[w]; b += se[w]; }
        part[2 * (long)lb] = a;
        part[2 * (long)lb + 1] = b;
    }
}

__global__ void __launch_bounds__(256) k_energy_final(const double *__restrict__ part, int n, double *__restrict__ out) {
    double a = 0, b = 0;
#pragma unroll 8
    for (int q = threadIdx.x; q < n; q += blockDim.x) {
        a += part[2 * (long)q];
        b += part[2 * (long)q + 1];
    }
    __shared__ double sa[4], sb[4];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        a += __shfl_xor(a, o, 64);
        b += __shfl_xor(b, o, 64);
    }
    if ((threadIdx.x & 63) == 0) { sa[threadIdx.x >> 6] = a; sb[threadIdx.x >> 6] = b; }
    __syncthreads();
    if (threadIdx.x == 0) {
        double x = 0, y = 0;
        for (int w = 0; w < 4; w++) { x += sa[w]; y += sb[w]; }
        out[0] = x;
        out[1] = y;
    }
}

// max over the node core of a field (fxMax); the values are arbitrary signed doubles, reduced in
// a fixed order per block then by one block
__global__ void __launch_bounds__(256) k_max_partial(FShape fp, const double *__restrict__ F, double *__restrict__ part) {
    long total = (long)fp.n[0] * fp.n[1] * fp.n[2];
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    double m = -1.0e300;
    if (t < total) {
        int k = (int)(t % fp.n[2]);
        long r = t / fp.n[2];
        int j = (int)(r % fp.n[1]);
        int i = (int)(r / fp.n[1]);
        m = F[fidx(fp, i, j, k)];
    }
    __shared__ double s[4];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = fmax(fmax(s[0], s[1]), fmax(s[2], s[3]));
}

__global__ void __launch_bounds__(256) k_max_final(const double *__restrict__ part, int n, double *__restrict__ out) {
    double m = -1.0e300;
#pragma unroll 8
    for (int q = threadIdx.x; q < n; q += blockDim.x) m = fmax(m, part[q]);
    __shared__ double s[4];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) out[0] = fmax(fmax(s[0], s[1]), fmax(s[2], s[3]));
}

__global__ void k_tgv(FShape f, Metrics M, int c, double Lx, double Ly, double Lz, double *__restrict__ V) {
    long total = (long)(f.n[0] + 2) * (f.n[1] + 2) * (f.n[2] + 2);
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= total) return;
    int k = (int)(t % (f.n[2] + 2)) - 1;
    long r = t / (f.n[2] + 2);
    int j = (int)(r % (f.n[1] + 2)) - 1;
    int i = (int)(r / (f.n[1] + 2)) - 1;
    double x = metv(M, 0, f.s[0], 0, i), y = metv(M, 1, f.s[1], 0, j), z = metv(M, 2, f.s[2], 0, k);
    const double pi = 3.14159265358979323846;
    double v = 0.0;
    if (c == 0) v = sin(2.0 * pi * x / Lx) * cos(2.0 * pi * y / Ly) * cos(2.0 * pi * z / Lz);
    if (c == 1) v = -cos(2.0 * pi * x / Lx) * sin(2.0 * pi * y / Ly) * cos(2.0 * pi * z / Lz);
    V[t] = v;
}

// ------------------------------------------------------------------------------------------------
// launchers
// ------------------------------------------------------------------------------------------------
static inline unsigned nb(long n) { return (unsigned)((n + 255) / 256); }

void ts_deriv(const FShape &f, const Metrics &M, const double *F, double *out, int order, int d, double h,
              hipStream_t s) {
    long sz[3] = {f.n[0] + 2L, f.n[1] + 2L, f.n[2] + 2L};
    sz[d] = f.n[d];
    hipLaunchKernelGGL(k_deriv, dim3(nb(sz[0] * sz[1] * sz[2])), dim3(256), 0, s, f, M, F, out, order, d, 1.0 / h);
}

// the inverse grid spacings are formed on the host, like derivative's ihx, ihy, ihz (derivative.cc:66-68)
static ColMet col_met(const double *h) { return ColMet{{1.0 / h[0], 1.0 / h[1], 1.0 / h[2]}, 0.5}; }

void ts_build_rhs(const FShape &fp, const Metrics &M, const double *const *V, const double *P, double *const *H,
                  const double *h, double visc, double dt, const double *T, double Fb, hipStream_t s) {
    const VelGeo S{{fp.n[0], fp.n[1], fp.n[2]}};
    const ColGeo G = col_geo(fp.n[1] + 2, fp.n[2] + 2, fp.n[0]);
    hipLaunchKernelGGL((T ? k_build_rhs<true> : k_build_rhs<false>), dim3(col_blocks(G)), dim3(kColThreads), 0, s, G, S, M, V[0],
                       V[1], V[2], P, H[0], H[1], H[2], col_met(h), visc, dt, T, Fb);
}

void ts_build_trhs(const FShape &fp, const Metrics &M, const double *const *V, const double *T, double *R,
                   const double *h, double kappa, double dt, hipStream_t s) {
    const VelGeo S{{fp.n[0], fp.n[1], fp.n[2]}};
    const ColGeo G = col_geo(fp.n[1] + 2, fp.n[2] + 2, fp.n[0] + 2);
    hipLaunchKernelGGL(k_build_trhs, dim3(col_blocks(G)), dim3(kColThreads), 0, s, G, S, M, V[0], V[1], V[2], T, R, col_met(h),
                       kappa, dt);
}

void ts_nusselt(const FShape &fp, const FShape &fz, const Metrics &M, const double *Vz, const double *T,
                const double *h, double *part, double *out, hipStream_t s) {
    int n = ts_energy_parts(fp);
    hipLaunchKernelGGL(k_nusselt, dim3(n), dim3(256), 0, s, fp, fz, M, Vz, T, h[0], h[1], h[2], part);
    hipLaunchKernelGGL(k_energy_final, dim3(1), dim3(256), 0, s, part, n, out);
}

// the grid-uniform quotients of hydro_d3.cc:375-410 (form 0: 1/Re; form 1: the diffusivity vis,
// scalar_d3.cc:373-531), formed once on the host
static JacobiCoef with_quotients(JacobiCoef J) {
    if (J.form == 0) {
        J.rA = J.dt / (J.hx2hy2hz2 * 2.0 * J.Re);
        J.rD = J.dt / (J.Re * J.hx2hy2hz2);
    } else {
        J.rA = J.dt * J.vis / (J.hx2hy2hz2 * 2.0);
        J.rD = J.dt * J.vis / J.hx2hy2hz2;
    }
    J.ih2[0] = 1.0 / (J.hx * J.hx);
    J.ih2[1] = 1.0 / (J.hy * J.hy);
    J.ih2[2] = 1.0 / (J.hz * J.hz);
    J.lapS = 0.5 * J.dt * (J.form == 0 ? J.inverseRe : J.vis);
    return J;
}

void ts_jacobi(const FShape &f, const Metrics &M, const Bulk &B, const double *V, const double *R, double *G,
               const JacobiCoef &J, hipStream_t s) {
    const ColGeo C = col_geo(f.n[1] + 2, f.n[2] + 2, f.n[0] + 2, kJacobiThreads);
    hipLaunchKernelGGL(k_jacobi_march<false>, dim3(col_blocks(C)), dim3(kJacobiThreads), 0, s, C, f, M, B, V, R, G,
                       with_quotients(J), nullptr, nullptr, nullptr);
}

int ts_jacobi_res_parts() { return 1024; }

void ts_jacobi_res(const FShape &f, const Metrics &M, const Bulk &B, const double *V, const double *R,
                   const JacobiCoef &J, double *part, unsigned long long *out, hipStream_t s) {
    long n = (long)(B.hi[0] - B.lo[0] + 1) * (B.hi[1] - B.lo[1] + 1) * (B.hi[2] - B.lo[2] + 1);
    unsigned g = nb(n);
    if (g > (unsigned)ts_jacobi_res_parts()) g = (unsigned)ts_jacobi_res_parts();
    if (g == 0) g = 1;
    hipLaunchKernelGGL(k_jacobi_res, dim3(g), dim3(256), 0, s, f, M, B, V, R, with_quotients(J), part);
    hipLaunchKernelGGL(k_jacobi_res_final, dim3(1), dim3(1024), 0, s, part, (int)g, out);
}

void ts_jacobi_vres(const FShape &f, const Metrics &M, const Bulk &B, const double *V, const double *R, double *G,
                    const JacobiCoef &J, JacobiSync *sync, unsigned long long *out, unsigned long long *host,
                    hipStream_t s) {
    const ColGeo C = col_geo(f.n[1] + 2, f.n[2] + 2, f.n[0] + 2, kJacobiThreads);
    hipLaunchKernelGGL(k_jacobi_march<true>, dim3(col_blocks(C)), dim3(kJacobiThreads), 0, s, C, f, M, B, V, R, G,
                       with_quotients(J), sync, out, host);
}

static long wave_count(const GhostWave &W) {
    long n = 0;
    for (int o = 0; o < W.nops; o++) n += W.ops[o].count;
    return n;
}

void ts_ghost_wave(const FShape &f, double *F, const GhostWave &W, hipStream_t s) {
    const long n = wave_count(W);
    if (n > 0) hipLaunchKernelGGL(k_ghost_ops, dim3(nb(n)), dim3(256), 0, s, f, F, W);
}

// S copies within planes of z and W writes whole planes of z from planes that neither writes
static bool ghost_pair_ok(const FShape &f, const GhostWave &S, const GhostWave &W) {
    for (int o = 0; o < S.nops; o++)
        if (S.ops[o].a != 1.0 || S.ops[o].b != 0.0 || (S.ops[o].kind == 0 && S.ops[o].dim == 2)) return false;
    for (int o = 0; o < W.nops; o++) {
        if (W.ops[o].kind != 0 || W.ops[o].dim != 2 || W.ops[o].lo[0] != -1 || W.ops[o].lo[1] != -1 ||
            W.ops[o].hi[0] != f.n[0] || W.ops[o].hi[1] != f.n[1])
            return false;
        for (int q = 0; q < W.nops; q++)
            if (W.ops[o].a != 0.0 && W.ops[o].src[0] == W.ops[q].dst[0]) return false;
    }
    return S.nops > 0 && W.nops > 0;
}

void ts_ghost_waves(const FShape &f, double *F, const GhostWave *W, int n, hipStream_t s) {
    for (int w = 0; w < n; w++) {
        if (w + 1 < n && ghost_pair_ok(f, W[w], W[w + 1])) {
            const long ns = wave_count(W[w]), nw = wave_count(W[w + 1]);
            if (ns + nw > 0) hipLaunchKernelGGL(k_ghost_pair, dim3(nb(ns + nw)), dim3(256), 0, s, f, F, W[w], W[w + 1], ns);
            w++;
        } else {
            ts_ghost_wave(f, F, W[w], s);
        }
    }
}

JacobiCoef jacobi_coef(const double h[3], double dt, double Re) {
    JacobiCoef J{};
    J.hx = h[0];
    J.hy = h[1];
    J.hz = h[2];
    J.hx2hy2 = std::pow(J.hx, 2.0) * std::pow(J.hy, 2.0);
    J.hy2hz2 = std::pow(J.hy, 2.0) * std::pow(J.hz, 2.0);
    J.hz2hx2 = std::pow(J.hz, 2.0) * std::pow(J.hx, 2.0);
    J.hx2hy2hz2 = std::pow(J.hx, 2.0) * std::pow(J.hy, 2.0) * std::pow(J.hz, 2.0);
    J.dt = dt;
    J.Re = Re;
    J.inverseRe = Re > 0.0 ? 1.0 / Re : 0.0;
    return J;
}

Bulk jacobi_bulk(const FShape &f, const int per[3]) {
    Bulk B{};
    for (int k = 0; k < 3; k++) {
        B.lo[k] = 0;
        B.hi[k] = f.n[k] - 1;
        if (f.s[k] && !per[k]) {
            B.lo[k] = 1;
            B.hi[k] = f.n[k] - 2;
        }
    }
    return B;
}

int ts_jacobi_loop(const FShape &f, const Metrics &M, const Bulk &B, double *&F, double *&G, const double *R,
                   const JacobiCoef &J, const GhostWave *bc, int nbc, const JacobiIO &io, double tol, long max_iter,
                   int *sweeps, hipError_t *err) {
#define JCHK(x)                      \
    do {                             \
        hipError_t e_ = (x);         \
        if (e_ != hipSuccess) {      \
            *err = e_;               \
            return -1;               \
        }                            \
    } while (0)
    long iterCount = 0;
    int n = 0;
    ts_jacobi(f, M, B, F, R, G, J, io.s);
    std::swap(F, G);
    ts_ghost_waves(f, F, bc, nbc, io.s);
    int status = 0;
    while (true) {
        // not a maximum of absolute values: what is left here if the kernel's write does not land
        *io.hmax = ~0ull;
        ts_jacobi_vres(f, M, B, F, R, G, J, io.sync, io.dmax, io.hmax, io.s);
        JCHK(hipEventRecord(io.ev, io.s));
        ts_ghost_waves(f, G, bc, nbc, io.s);
        JCHK(hipGetLastError());
        JCHK(hipEventSynchronize(io.ev));
        double maxError;
        const unsigned long long bits = *(volatile unsigned long long *)io.hmax;
        if (bits == ~0ull) JCHK(hipErrorUnknown);
        std::memcpy(&maxError, &bits, sizeof(double));
        n += 1;
        if (maxError < tol) break;
        iterCount += 1;
        if (iterCount > max_iter) {
            status = 1;
            break;
        }
        std::swap(F, G);
    }
#undef JCHK
    *sweeps = n;
    return status;
}

void ts_divergence(const FShape &fp, const FShape *fv, const Metrics &M, const double *const *V, double *out,
                   const double *h, double scale, int scaled, hipStream_t s) {
    long n = (long)fp.n[0] * fp.n[1] * fp.n[2];
    hipLaunchKernelGGL(k_divergence, dim3(nb(n)), dim3(256), 0, s, fp, fv[0], fv[1], fv[2], M, V[0], V[1], V[2],
                       out, h[0], h[1], h[2], scale, scaled);
}

void ts_project(int c, const FShape &fc, const FShape &fp, const Metrics &M, const double *Pp, double *V,
                double hc, double dt, hipStream_t s) {
    long n = (long)fc.n[0] * fc.n[1] * fc.n[2];
    hipLaunchKernelGGL(k_project, dim3(nb(n)), dim3(256), 0, s, c, fc, fp, M, Pp, V, hc, dt);
}

void ts_axpy_full(double *y, const double *x, long n, hipStream_t s) {
    hipLaunchKernelGGL(k_axpy_full, dim3(nb(n)), dim3(256), 0, s, y, x, n);
}


void ts_fill(double *p, long n, double v, hipStream_t s) {
    if (n > 0) hipLaunchKernelGGL(k_fill_d, dim3(nb(n)), dim3(256), 0, s, p, n, v);
}

int ts_energy_parts(const FShape &fp) { return (int)nb((long)fp.n[0] * fp.n[1] * fp.n[2]); }

void ts_energy(const FShape &fp, const FShape *fv, const Metrics &M, const double *const *V, const double *h,
               double *part, double *out, hipStream_t s) {
    int n = ts_energy_parts(fp);
    hipLaunchKernelGGL(k_energy, dim3(n), dim3(256), 0, s, fp, fv[0], fv[1], fv[2], M, V[0], V[1], V[2], h[0],
                       h[1], h[2], part);
    hipLaunchKernelGGL(k_energy_final, dim3(1), dim3(256), 0, s, part, n, out);
}

void ts_max(const FShape &fp, const double *F, double *part, double *out, hipStream_t s) {
    int n = ts_energy_parts(fp);
    hipLaunchKernelGGL(k_max_partial, dim3(n), dim3(256), 0, s, fp, F, part);
    hipLaunchKernelGGL(k_max_final, dim3(1), dim3(256), 0, s, part, n, out);
}

void ts_tgv(const FShape &f, const Metrics &M, int c, double Lx, double Ly, double Lz, double *V, hipStream_t s) {
    long n = (long)(f.n[0] + 2) * (f.n[1] + 2) * (f.n[2] + 2);
    hipLaunchKernelGGL(k_tgv, dim3(nb(n)), dim3(256), 0, s, f, M, c, Lx, Ly, Lz, V);
}

}  // namespace sr
