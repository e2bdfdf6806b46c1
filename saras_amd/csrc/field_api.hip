// C ABI of the field operators on caller device arrays (include/saras_field.h): derivative
// (lib/field/derivative.cc:121-243), vfield / sfield computeDiff, computeNLin, divergence and
// gradient (vfield.cc:104-320, sfield.cc:86-171), the boundary classes with syncData, and the
// implicit Jacobi solves of hydro_d3 / scalar_d3.
//
// Kernels here march along x over the reference's padded natural layout (k fastest, columns.h), all
// components of a field operator in one launch, so that computeNLin reads each V_d once for the three
// components that it advects.  All are HBM-bound (well under one FP64 flop per byte).
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <string>
#include <utility>
#include <vector>

#include "../../include/saras_field.h"
#include "../../include/saras_mg.h"
#include "ghost_waves.h"
#include "columns.h"
#include "mg_state.h"
#include "ts_kernels.h"

using namespace sr;

#define HIPCHK(expr)                                                                                  \
    do {                                                                                              \
        hipError_t _e = (expr);                                                                       \
        if (_e != hipSuccess)                                                                         \
            return set_err(SR_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(_e));            \
    } while (0)

#define RETCHK(expr)                                                                                  \
    do {                                                                                              \
        int _r = (expr);                                                                              \
        if (_r != SR_OK) return _r;                                                                   \
    } while (0)

struct sr_fgrid {
    sr_fgrid_desc d{};
    int N[3] = {0, 0, 0};
    double h[3] = {0, 0, 0};
    double half = 0.5;                   // calcDerivative2*: factor of the xi^2 part (iScheme)
    FShape shape[4]{};                   // SR_LOC_NODE, SR_LOC_VX, SR_LOC_VY, SR_LOC_VZ
    double *dmet = nullptr;
    Metrics M{};
    hipStream_t s = nullptr;
    JacobiSync *jsync = nullptr;
    unsigned long long *dmax = nullptr, *hmax = nullptr;   // JacobiIO
    hipEvent_t jev = nullptr;            // marks a Jacobi residual's read-back
};

namespace {

__host__ __device__ inline long fsz(const FShape &f) { return (long)(f.n[0] + 2) * (f.n[1] + 2) * (f.n[2] + 2); }

// entry t of a padded plane with rows of n entries -> (j, k), counted from -1
__device__ inline void in_plane(unsigned t, int n, int &j, int &k) {
    const unsigned r = t / (unsigned)n;
    j = (int)r - 1;
    k = (int)(t - r * (unsigned)n) - 1;
}
__device__ inline long plane_of(const FShape &f) { return (long)(f.n[1] + 2) * (f.n[2] + 2); }

// calcDerivative1 / 2 along d over the whole padded array: the core range along d gets the
// derivative, the two pad layers along d get 0
template <int ORDER, bool ALONGX>
__global__ void __launch_bounds__(kColThreads) k_fd_deriv(ColGeo G, FShape f, Metrics M, const double *__restrict__ F,
                                                          double *__restrict__ out, int d, double ih, double half) {
    const Col C = column(G);
    const long ps = plane_of(f);
    // metrics of the planes (along x) or of this column
    __shared__ double lx[2][kColPlanes];
    if (ALONGX) {
        for (int q = (int)threadIdx.x; q < C.i1 - C.i0; q += kColThreads) {
            const int r = max(0, min(C.i0 - 1 + q, f.n[0] - 1));
            lx[0][q] = ORDER == 1 ? met1(M, 0, f.s[0], r, ih) : met2(M, 0, f.s[0], r, ih);
            lx[1][q] = ORDER == 1 ? 0.0 : met3(M, 0, f.s[0], r, ih, half);
        }
        __syncthreads();
    }
    if ((long)C.t >= ps) return;
    int j, k;
    in_plane(C.t, f.n[2] + 2, j, k);
    const int r = d == 1 ? j : k, n = d == 1 ? f.n[1] : f.n[2], sd = d == 1 ? f.s[1] : f.s[2];
    const bool column_in = ALONGX || (r >= 0 && r < n);
    // a pad entry along d takes part in the loads of the core entry next to it
    const int rc = max(0, min(r, n - 1)), st2 = d == 1 ? f.n[2] + 2 : 1;
    const unsigned o = C.t * 8u, os = ALONGX ? o : (unsigned)((int)C.t + (rc - r) * st2) * 8u;
    const long st = ALONGX ? ps : st2;
    double a2 = 0.0, a3 = 0.0;
    if (!ALONGX) {
        a2 = d == 1 ? met(M, 1, sd, ORDER, rc) : met(M, 2, sd, ORDER, rc);
        a2 *= 0.5 * ih;
        if (ORDER == 2) a3 = half * (d == 1 ? met(M, 1, sd, 3, rc) : met(M, 2, sd, 3, rc)) * (ih * ih);
    }
    for (int p0 = C.i0; p0 < C.i1; p0 += kColAhead) {
        double fp[kColAhead], fm[kColAhead], fc[kColAhead];
#pragma unroll
        for (int u = 0; u < kColAhead; u++) {
            const int p = ALONGX ? max(1, min(p0 + u, f.n[0])) : min(p0 + u, C.i1 - 1);
            const double *const c = F + p * ps;
            fp[u] = ldd(c + st, os);
            fm[u] = ldd(c - st, os);
            if (ORDER == 2) fc[u] = ldd(c, os);
        }
        loaded(fp);
        loaded(fm);
        if (ORDER == 2) loaded(fc);
#pragma unroll
        for (int u = 0; u < kColAhead; u++) {
            const int p = p0 + u;
            if (p >= C.i1) break;
            const bool in = ALONGX ? p >= 1 && p <= f.n[0] : column_in;
            const double b2 = ALONGX ? lx[0][p - C.i0] : a2, b3 = ALONGX ? lx[1][p - C.i0] : a3;
            const double v = ORDER == 1 ? b2 * (fp[u] - fm[u]) : b2 * (fp[u] - fm[u]) + b3 * (fp[u] - 2.0 * fc[u] + fm[u]);
            std_(out + p * ps, o, in ? v : 0.0);
        }
    }
}

// up to three fields with their own shapes, one per grid row
struct Fields {
    const double *F[3];
    double *H[3];
    FShape f[3];
};

// computeDiff: H(core) += d2xx, += d2yy, += d2zz in that order.  At 257^3 the field and H are read and
// H is written, 0.41 GB: 163 -> 116 us.
__global__ void __launch_bounds__(kColThreads) k_fd_diff(ColGeo G, Fields A, Metrics M, ColMet W) {
    const FShape f = A.f[blockIdx.y];
    const Col C = column(G);
    __shared__ double lx[2][kColPlanes];
    for (int q = (int)threadIdx.x; q < C.i1 - C.i0; q += kColThreads) {
        const int i = min(C.i0 + q, f.n[0] - 1);
        lx[0][q] = met2(M, 0, f.s[0], i, W.ih[0]);
        lx[1][q] = met3(M, 0, f.s[0], i, W.ih[0], W.half);
    }
    __syncthreads();
    int j, k;
    const int row = f.n[2] + 2, i1 = min(C.i1, f.n[0]);
    in_plane(C.t, row, j, k);
    if (j < 0 || k < 0 || j >= f.n[1] || k >= f.n[2] || C.i0 >= i1) return;
    const long ps = plane_of(f);
    const unsigned o = C.t * 8u;
    const double y2 = met2(M, 1, f.s[1], j, W.ih[1]), y3 = met3(M, 1, f.s[1], j, W.ih[1], W.half);
    const double z2 = met2(M, 2, f.s[2], k, W.ih[2]), z3 = met3(M, 2, f.s[2], k, W.ih[2], W.half);
    const double *F = A.F[blockIdx.y] + (C.i0 + 1) * ps;
    double *H = A.H[blockIdx.y] + (C.i0 + 1) * ps;
    Cross u;
    u.xm = ldd(F - ps, o);
    u.c = ldd(F, o);
    for (int i = C.i0; i < i1; i += kColAhead, F += kColAhead * ps, H += kColAhead * ps) {
        double xp[kColAhead], h[kColAhead];
#pragma unroll
        for (int w = 0; w < kColAhead; w++) {
            const long q = min(w, i1 - 1 - i) * ps;
            xp[w] = ldd(F + q + ps, o);
            h[w] = ldd(H + q, o);
        }
        loaded(xp);
        loaded(h);
#pragma unroll
        for (int w = 0; w < kColAhead; w++) {
            if (i + w >= i1) break;
            const double *const f = F + w * ps;
            u.xp = xp[w];
            u.yp = ldd(f + row, o);
            u.ym = ldd(f - row, o);
            u.zp = ldd(f + 1, o);
            u.zm = ldd(f - 1, o);
            const int q = i + w - C.i0;
            std_(H + w * ps, o, diffuse(h[w], u, lx[0][q], lx[1][q], y2, y3, z2, z3));
            u.xm = u.c;
            u.c = u.xp;
        }
    }
}

// computeNLin of a vector field U advected by V: for d = x, y, z, H(core) -= (sum of the slices of V_d)
// d_d U / nslices.  Slices of V_d onto component c's location: the core index alone when d == c, else
// {core, d-1, c+1, (c+1, d-1)} (field.cc:309-575).  SELF: U is V, whose loads then serve both.  which: the
// components to do, as bits.  At 257^3 three fields and three H are read and H is written, 1.22 GB: 560 ->
// 350 us for the three components.
template <bool SELF>
__global__ void __launch_bounds__(kColThreads) k_fd_nlin(ColGeo G, VelGeo S, Metrics M, const double *__restrict__ Ux,
                                                 const double *__restrict__ Uy, const double *__restrict__ Uz,
                                                 const double *__restrict__ Vx, const double *__restrict__ Vy,
                                                 const double *__restrict__ Vz, double *__restrict__ Hx,
                                                 double *__restrict__ Hy, double *__restrict__ Hz, ColMet W, int which) {
    const Col C = column(G);
    __shared__ double lx[2][kColPlanes];   // x metrics of faces (one slice) and a quarter of those of nodes
    for (int q = (int)threadIdx.x; q < C.i1 - C.i0; q += kColThreads) {
        lx[0][q] = met1(M, 0, 0, min(C.i0 + q, S.N[0] - 2), W.ih[0]);
        lx[1][q] = 0.25 * met1(M, 0, 1, C.i0 + q, W.ih[0]);
    }
    __syncthreads();
    int j, k;
    const int row = S.N[2] + 2, rz = S.N[2] + 1;
    in_plane(C.t, row, j, k);
    if (j < 0 || k < 0 || j >= S.N[1] || k >= S.N[2]) return;
    const long sx = S.sx(), sy = S.sy(), sz = S.sz();
    const unsigned o = C.t * 8u, oz = (unsigned)((j + 1) * rz + k + 1) * 8u;
    const bool cy = (which & 2) && j < S.N[1] - 1, cz = (which & 4) && k < S.N[2] - 1;
    const double yf = met1(M, 1, 0, min(j, S.N[1] - 2), W.ih[1]), yn = 0.25 * met1(M, 1, 1, j, W.ih[1]);
    const double zf = met1(M, 2, 0, min(k, S.N[2] - 2), W.ih[2]), zn = 0.25 * met1(M, 2, 1, k, W.ih[2]);
    const long i0 = C.i0 + 1;
    Vx += i0 * sx;
    Vy += i0 * sy;
    Vz += i0 * sz;
    Ux += i0 * sx;
    Uy += i0 * sy;
    Uz += i0 * sz;
    Hx += i0 * sx;
    Hy += i0 * sy;
    Hz += i0 * sz;
    Vels v;
    vels_begin(v, Vx, Vy, Vz, S, o, oz, SELF);
    Cross ux, uy, uz;
    if (!SELF) {
        ux.xm = ldd(Ux - sx, o);
        ux.c = ldd(Ux, o);
        uy.xm = ldd(Uy - sy, o);
        uy.c = ldd(Uy, o);
        uz.xm = ldd(Uz - sz, oz);
        uz.c = ldd(Uz, oz);
    }
    for (int i = C.i0; i < C.i1; ++i) {
        const bool cx = i < S.N[0] - 1;
        vels_load(v, Vx, Vy, Vz, S, o, oz, SELF, !cx);
        if (SELF) {
            ux = cross_x(v);
            uy = cross_y(v);
            uz = cross_z(v);
        } else {
            ux.xp = ldd(cx ? Ux + sx : Ux, o);
            ux.yp = ldd(Ux + row, o);
            ux.ym = ldd(Ux - row, o);
            ux.zp = ldd(Ux + 1, o);
            ux.zm = ldd(Ux - 1, o);
            uy.xp = ldd(Uy + sy, o);
            uy.yp = ldd(Uy + row, o);
            uy.ym = ldd(Uy - row, o);
            uy.zp = ldd(Uy + 1, o);
            uy.zm = ldd(Uy - 1, o);
            uz.xp = ldd(Uz + sz, oz);
            uz.yp = ldd(Uz + rz, oz);
            uz.ym = ldd(Uz - rz, oz);
            uz.zp = ldd(Uz + 1, oz);
            uz.zm = ldd(Uz - 1, oz);
        }
        const double hx = ldd(Hx, o), hy = ldd(Hy, o), hz = ldd(Hz, oz);
        const double xf = lx[0][i - C.i0], xn = lx[1][i - C.i0];
        if (cx && (which & 1)) std_(Hx, o, advect<0>(hx, v, ux, xf, yn, zn));
        if (cy) std_(Hy, o, advect<1>(hy, v, uy, xn, yf, zn));
        if (cz) std_(Hz, oz, advect<2>(hz, v, uz, xn, yn, zf));
        vels_next(v);
        if (!SELF) {
            ux.xm = ux.c;
            ux.c = ux.xp;
            uy.xm = uy.c;
            uy.c = uy.xp;
            uz.xm = uz.c;
            uz.c = uz.xp;
        }
        Vx += sx;
        Vy += sy;
        Vz += sz;
        Ux += sx;
        Uy += sy;
        Uz += sz;
        Hx += sx;
        Hy += sy;
        Hz += sz;
    }
}

// computeNLin of a node field: the slices of V_d are {core, d-1}
__global__ void __launch_bounds__(kColThreads) k_fd_nlin_node(ColGeo G, VelGeo S, Metrics M, const double *__restrict__ F,
                                                      const double *__restrict__ Vx, const double *__restrict__ Vy,
                                                      const double *__restrict__ Vz, double *__restrict__ H, ColMet W) {
    const Col C = column(G);
    __shared__ double lx[kColPlanes];
    for (int q = (int)threadIdx.x; q < C.i1 - C.i0; q += kColThreads) lx[q] = 0.5 * met1(M, 0, 1, C.i0 + q, W.ih[0]);
    __syncthreads();
    int j, k;
    const int row = S.N[2] + 2, rz = S.N[2] + 1;
    in_plane(C.t, row, j, k);
    if (j < 0 || k < 0 || j >= S.N[1] || k >= S.N[2]) return;
    const long sx = S.sx(), sy = S.sy(), sz = S.sz(), i0 = C.i0 + 1;
    const unsigned o = C.t * 8u, oz = (unsigned)((j + 1) * rz + k + 1) * 8u;
    const double ay = 0.5 * met1(M, 1, 1, j, W.ih[1]), az = 0.5 * met1(M, 2, 1, k, W.ih[2]);
    F += i0 * sx;
    H += i0 * sx;
    Vx += i0 * sx;
    Vy += i0 * sy;
    Vz += i0 * sz;
    double fm = ldd(F - sx, o), f0 = ldd(F, o), xm = ldd(Vx - sx, o);
    for (int i = C.i0; i < C.i1; i += kColAhead) {
        double fp[kColAhead], x[kColAhead], acc[kColAhead], y[kColAhead], ym[kColAhead], z[kColAhead], zm[kColAhead];
        double fy[kColAhead], fym[kColAhead], fz[kColAhead], fzm[kColAhead];
#pragma unroll
        for (int u = 0; u < kColAhead; u++) {
            const long q = min(u, C.i1 - 1 - i);
            const double *const f = F + q * sx, *const Y = Vy + q * sy, *const Z = Vz + q * sz;
            fp[u] = ldd(f + sx, o);
            x[u] = ldd(Vx + q * sx, o);
            acc[u] = ldd(H + q * sx, o);
            y[u] = ldd(Y, o);
            ym[u] = ldd(Y - row, o);
            z[u] = ldd(Z, oz);
            zm[u] = ldd(Z - 1, oz);
            fy[u] = ldd(f + row, o);
            fym[u] = ldd(f - row, o);
            fz[u] = ldd(f + 1, o);
            fzm[u] = ldd(f - 1, o);
        }
        loaded(fp);
        loaded(x);
        loaded(acc);
        loaded(y);
        loaded(z);
#pragma unroll
        for (int u = 0; u < kColAhead; u++) {
            if (i + u >= C.i1) break;
            acc[u] -= (x[u] + xm) * (lx[i + u - C.i0] * (fp[u] - fm));
            acc[u] -= (y[u] + ym[u]) * (ay * (fy[u] - fym[u]));
            acc[u] -= (z[u] + zm[u]) * (az * (fz[u] - fzm[u]));
            std_(H + u * sx, o, acc[u]);
            fm = f0;
            f0 = fp[u];
            xm = x[u];
        }
        F += kColAhead * sx;
        H += kColAhead * sx;
        Vx += kColAhead * sx;
        Vy += kColAhead * sy;
        Vz += kColAhead * sz;
    }
}

// gradient on the cores of its components: G_c = xi_c(face) (F(+1) - F) / h_c; which: the components to
// do, as bits.  One launch reads F once: 213 -> 134 us at 257^3.
__global__ void __launch_bounds__(kColThreads) k_fd_gradient(ColGeo G, VelGeo S, Metrics M, const double *__restrict__ F,
                                                     double *__restrict__ Gx, double *__restrict__ Gy,
                                                     double *__restrict__ Gz, ColMet W, int which) {
    const Col C = column(G);
    __shared__ double lx[kColPlanes];
    for (int q = (int)threadIdx.x; q < C.i1 - C.i0; q += kColThreads)
        lx[q] = met(M, 0, 0, 1, min(C.i0 + q, S.N[0] - 2)) * W.ih[0];
    __syncthreads();
    int j, k;
    const int row = S.N[2] + 2, rz = S.N[2] + 1;
    in_plane(C.t, row, j, k);
    if (j < 0 || k < 0 || j >= S.N[1] || k >= S.N[2]) return;
    const long sx = S.sx(), sy = S.sy(), sz = S.sz(), i0 = C.i0 + 1;
    const unsigned o = C.t * 8u, oz = (unsigned)((j + 1) * rz + k + 1) * 8u;
    const bool cy = (which & 2) && j < S.N[1] - 1, cz = (which & 4) && k < S.N[2] - 1;
    const double ay = met(M, 1, 0, 1, min(j, S.N[1] - 2)) * W.ih[1], az = met(M, 2, 0, 1, min(k, S.N[2] - 2)) * W.ih[2];
    F += i0 * sx;
    Gx += i0 * sx;
    Gy += i0 * sy;
    Gz += i0 * sz;
    double f0 = ldd(F, o);
    for (int i = C.i0; i < C.i1; i += kColAhead) {
        double fp[kColAhead], fy[kColAhead], fz[kColAhead];
#pragma unroll
        for (int u = 0; u < kColAhead; u++) {
            const double *const f = F + min(u, C.i1 - 1 - i) * sx;
            fp[u] = ldd(f + sx, o);
            fy[u] = ldd(f + row, o);
            fz[u] = ldd(f + 1, o);
        }
        loaded(fp);
#pragma unroll
        for (int u = 0; u < kColAhead; u++) {
            if (i + u >= C.i1) break;
            if (i + u < S.N[0] - 1 && (which & 1)) std_(Gx + u * sx, o, lx[i + u - C.i0] * (fp[u] - f0));
            if (cy) std_(Gy + u * sy, o, ay * (fy[u] - f0));
            if (cz) std_(Gz + u * sz, oz, az * (fz[u] - f0));
            f0 = fp[u];
        }
        F += kColAhead * sx;
        Gx += kColAhead * sx;
        Gy += kColAhead * sy;
        Gz += kColAhead * sz;
    }
}

// divergence over the whole padded node array: core from the face differences, pads 0.  Planes one by one:
// 257^3 117 us, 65 x 257 x 257 nodes 23.8, 129^3 13.1; by pairs 124, 24.3 and 13.4, one thread per entry
// 128, 23.7 and 13.7.
__global__ void __launch_bounds__(kColThreads) k_fd_divergence(ColGeo G, VelGeo S, Metrics M, const double *__restrict__ Vx,
                                                       const double *__restrict__ Vy, const double *__restrict__ Vz,
                                                       double *__restrict__ out, ColMet W) {
    const Col C = column(G);   // padded planes
    __shared__ double lx[kColPlanes];
    for (int q = (int)threadIdx.x; q < C.i1 - C.i0; q += kColThreads)
        lx[q] = met(M, 0, 1, 1, max(0, min(C.i0 - 1 + q, S.N[0] - 1))) * W.ih[0];
    __syncthreads();
    const long sx = S.sx(), sy = S.sy(), sz = S.sz();
    if ((long)C.t >= sx) return;
    int j, k;
    const int row = S.N[2] + 2, rz = S.N[2] + 1;
    in_plane(C.t, row, j, k);
    const bool in = j >= 0 && k >= 0 && j < S.N[1] && k < S.N[2];
    const unsigned po = C.t * 8u;
    // a pad entry takes part in the loads of the core entry next to it
    j = max(0, min(j, S.N[1] - 1));
    k = max(0, min(k, S.N[2] - 1));
    const unsigned o = (unsigned)((j + 1) * row + k + 1) * 8u, oz = (unsigned)((j + 1) * rz + k + 1) * 8u;
    const double ay = met(M, 1, 1, 1, j) * W.ih[1], az = met(M, 2, 1, 1, k) * W.ih[2];
    double xm = ldd(Vx + max(C.i0 - 1, 0) * sx, o);
    for (int p = C.i0; p < C.i1; p++) {
        const long q = min(p, S.N[0]);   // the last plane of Vx
        const double x = ldd(Vx + q * sx, o);
        const double y = ldd(Vy + q * sy, o), ym = ldd(Vy + q * sy - row, o);
        const double z = ldd(Vz + q * sz, oz), zm = ldd(Vz + q * sz - 1, oz);
        const double a = lx[p - C.i0] * (x - xm), b = ay * (y - ym);
        const double v = a + b + az * (z - zm);
        std_(out + p * sx, po, in && p >= 1 && p <= S.N[0] ? v : 0.0);
        xm = x;
    }
}

ColMet col_met(const sr_fgrid *g) {
    // the inverse grid spacings are formed on the host, like derivative's ihx, ihy, ihz (derivative.cc:66-68)
    return ColMet{{1.0 / g->h[0], 1.0 / g->h[1], 1.0 / g->h[2]}, g->half};
}
VelGeo vel_geo(const sr_fgrid *g) { return VelGeo{{g->N[0], g->N[1], g->N[2]}}; }
// Whether the components' outputs H can be written by one launch that reads the inputs U (one for each
// component) and V (all of them for every component): no output shares memory with another one, with
// another component's U or with a V.  A caller may let them (the components are then done in order, as
// if one by one, each reading what the ones before it left).
bool one_launch(const sr_fgrid *g, double *const H[3], const double *const *U, const double *const *V = nullptr) {
    auto apart = [&](const double *a, int c, const double *b, int e) {
        return a + fsz(g->shape[SR_LOC_VX + c]) <= b || b + fsz(g->shape[SR_LOC_VX + e]) <= a;
    };
    for (int c = 0; c < 3; c++)
        for (int e = 0; e < 3; e++) {
            if (V && !apart(H[c], c, V[e], e)) return false;
            if (e != c && (!apart(H[c], c, H[e], e) || (U && !apart(H[c], c, U[e], e)))) return false;
        }
    return true;
}
ColGeo node_geo(const sr_fgrid *g, int planes, int ahead = kColAhead) {
    return col_geo(g->N[1] + 2, g->N[2] + 2, planes, kColThreads, ahead);
}

int check_loc(const sr_fgrid *g, int loc) {
    if (!g) return set_err(SR_ERR_ARG, "null handle");
    if (loc < SR_LOC_NODE || loc > SR_LOC_VZ) return set_err(SR_ERR_ARG, "location must be SR_LOC_NODE..SR_LOC_VZ");
    return SR_OK;
}

// the boundary conditions as ordered waves: syncData, x walls, y walls, then top and bottom
int bc_waves(const sr_fgrid *g, const FShape &f, const sr_bc *bc, std::vector<GhostWave> &ws) {
    int per[3] = {g->d.xPer, g->d.yPer, g->d.zPer};
    for (int w = 0; w < 6; w++) {
        int kd = bc->kind[w];
        if (kd != SR_BC_PERIODIC && kd != SR_BC_DIRICHLET && kd != SR_BC_NEUMANN && kd != SR_BC_NONE)
            return set_err(SR_ERR_ARG, "boundary kind must be SR_BC_PERIODIC, _DIRICHLET, _NEUMANN or _NONE");
        bool p = per[w / 2] != 0;
        if ((kd == SR_BC_PERIODIC && !p) || (p && kd != SR_BC_PERIODIC && kd != SR_BC_NONE))
            return set_err(SR_ERR_ARG, "periodic walls must match the grid's periodic directions");
    }
    ws.clear();
    ws.push_back(sync_wave(f, per[0], per[1]));
    // wall_op kinds: 0 periodicCC, 1 periodicFC, 2 dirichletCC, 3 dirichletFC, 4 neumannCC, 5 neumannFC
    auto cls = [&](int w) {
        int node = f.s[w / 2];
        if (bc->kind[w] == SR_BC_PERIODIC) return node ? 0 : 1;
        if (bc->kind[w] == SR_BC_DIRICHLET) return node ? 2 : 3;
        return node ? 4 : 5;
    };
    for (int d = 0; d < 2; d++) {
        if (per[d]) continue;
        GhostWave w{};
        for (int q = 2 * d; q <= 2 * d + 1; q++)
            if (bc->kind[q] != SR_BC_NONE) add_op(w, wall_op(f, 0, q, cls(q), bc->value[q]));
        if (w.nops) ws.push_back(w);
    }
    GhostWave w{};
    for (int q : {5, 4})
        if (bc->kind[q] != SR_BC_NONE) add_op(w, wall_op(f, per[2], q, cls(q), bc->value[q]));
    if (w.nops) ws.push_back(w);
    return SR_OK;
}

}  // namespace

// ------------------------------------------------------------------------------------------------
// handle
// ------------------------------------------------------------------------------------------------
static int fgrid_create_impl(const sr_fgrid_desc *desc, sr_fgrid *g) {
    g->d = *desc;
    const sr_fgrid_desc &d = g->d;
    int ind[3] = {d.xInd, d.yInd, d.zInd};
    double L[3] = {d.Lx, d.Ly, d.Lz};
    int gt[3] = {d.xGrid, d.yGrid, d.zGrid};
    double beta[3] = {d.betaX, d.betaY, d.betaZ};
    for (int k = 0; k < 3; k++) {
        if (ind[k] < 2 || ind[k] > 12) return set_err(SR_ERR_ARG, "grid size index out of range 2..12");
        if (L[k] <= 0.0) return set_err(SR_ERR_ARG, "domain length must be positive");
    }
    g->half = d.iScheme == 1 ? 0.5 : 1.0;
    std::vector<double> hmet[3][2][4];
    for (int k = 0; k < 3; k++) {
        int n = (1 << ind[k]) + 1;
        g->N[k] = n;
        g->h[k] = 1.0 / (double)(n - 1);
        for (int face = 0; face < 2; face++) {
            for (int q = 0; q < 4; q++) hmet[k][face][q].assign((size_t)(face ? n + 1 : n + 2), 0.0);
            int r = sr_grid_axis(n, L[k], gt[k], beta[k], face, hmet[k][face][0].data(), hmet[k][face][1].data(),
                                 hmet[k][face][2].data(), hmet[k][face][3].data());
            if (r != SR_OK) return set_err(r, "invalid grid description");
        }
    }
    for (int k = 0; k < 3; k++) {
        g->shape[SR_LOC_NODE].n[k] = g->N[k];
        g->shape[SR_LOC_NODE].s[k] = 1;
    }
    for (int c = 0; c < 3; c++)
        for (int k = 0; k < 3; k++) {
            g->shape[SR_LOC_VX + c].n[k] = c == k ? g->N[k] - 1 : g->N[k];
            g->shape[SR_LOC_VX + c].s[k] = c == k ? 0 : 1;
        }
    HIPCHK(hipStreamCreateWithFlags(&g->s, hipStreamNonBlocking));
    size_t tot = 0;
    for (int k = 0; k < 3; k++)
        for (int face = 0; face < 2; face++)
            for (int q = 0; q < 4; q++) tot += hmet[k][face][q].size();
    HIPCHK(hipMalloc((void **)&g->dmet, sizeof(double) * tot));
    size_t off = 0;
    for (int k = 0; k < 3; k++)
        for (int face = 0; face < 2; face++)
            for (int q = 0; q < 4; q++) {
                const std::vector<double> &v = hmet[k][face][q];
                HIPCHK(hipMemcpy(g->dmet + off, v.data(), sizeof(double) * v.size(), hipMemcpyHostToDevice));
                g->M.m[k][face][q] = g->dmet + off;
                off += v.size();
            }
    HIPCHK(hipEventCreateWithFlags(&g->jev, hipEventDisableTiming));
    HIPCHK(hipMalloc((void **)&g->dmax, sizeof(unsigned long long)));
    HIPCHK(hipMalloc((void **)&g->jsync, sizeof(JacobiSync)));
    HIPCHK(hipMemsetAsync(g->jsync, 0, sizeof(JacobiSync), g->s));
    HIPCHK(hipHostMalloc((void **)&g->hmax, sizeof(unsigned long long), hipHostMallocDefault));
    return SR_OK;
}

extern "C" int sr_fgrid_create(const sr_fgrid_desc *desc, sr_fgrid **out) {
    if (!desc || !out) return set_err(SR_ERR_ARG, "null argument");
    *out = nullptr;
    sr_fgrid *g = new sr_fgrid();
    int r = fgrid_create_impl(desc, g);
    if (r != SR_OK) {
        std::string msg = sr_last_error();
        sr_fgrid_destroy(g);
        return set_err(r, msg);
    }
    *out = g;
    return SR_OK;
}

extern "C" int sr_fgrid_destroy(sr_fgrid *g) {
    if (!g) return SR_OK;
    if (g->s) (void)hipStreamSynchronize(g->s);
    if (g->dmet) (void)hipFree(g->dmet);
    if (g->jev) (void)hipEventDestroy(g->jev);
    if (g->dmax) (void)hipFree(g->dmax);
    if (g->jsync) (void)hipFree(g->jsync);
    if (g->hmax) (void)hipHostFree(g->hmax);
    if (g->s) (void)hipStreamDestroy(g->s);
    delete g;
    return SR_OK;
}

extern "C" int sr_fgrid_dims(const sr_fgrid *g, int loc, int *nx, int *ny, int *nz) {
    RETCHK(check_loc(g, loc));
    if (!nx || !ny || !nz) return set_err(SR_ERR_ARG, "null argument");
    *nx = g->shape[loc].n[0];
    *ny = g->shape[loc].n[1];
    *nz = g->shape[loc].n[2];
    return SR_OK;
}

extern "C" int sr_fgrid_stream(const sr_fgrid *g, void **hip_stream) {
    if (!g || !hip_stream) return set_err(SR_ERR_ARG, "null argument");
    *hip_stream = (void *)g->s;
    return SR_OK;
}

extern "C" int sr_fgrid_sync(sr_fgrid *g) {
    if (!g) return set_err(SR_ERR_ARG, "null handle");
    HIPCHK(hipStreamSynchronize(g->s));
    HIPCHK(hipGetLastError());
    return SR_OK;
}

// ------------------------------------------------------------------------------------------------
// operators
// ------------------------------------------------------------------------------------------------
static int deriv(sr_fgrid *g, int loc, int order, int dim, const double *F, double *out) {
    RETCHK(check_loc(g, loc));
    if (dim < 0 || dim > 2) return set_err(SR_ERR_ARG, "dim must be 0..2");
    if (!F || !out) return set_err(SR_ERR_ARG, "null array");
    if ((const double *)out == F) return set_err(SR_ERR_ARG, "out must not alias F");
    const FShape &f = g->shape[loc];
    const ColGeo G = col_geo(f.n[1] + 2, f.n[2] + 2, f.n[0] + 2);
    auto *const k = order == 1 ? (dim == 0 ? k_fd_deriv<1, true> : k_fd_deriv<1, false>)
                               : (dim == 0 ? k_fd_deriv<2, true> : k_fd_deriv<2, false>);
    hipLaunchKernelGGL(k, dim3(col_blocks(G)), dim3(kColThreads), 0, g->s, G, f, g->M, F, out, dim, 1.0 / g->h[dim],
                       g->half);
    HIPCHK(hipGetLastError());
    return SR_OK;
}

extern "C" int sr_deriv1(sr_fgrid *g, int loc, int dim, const double *F, double *out) {
    return deriv(g, loc, 1, dim, F, out);
}
extern "C" int sr_deriv2(sr_fgrid *g, int loc, int dim, const double *F, double *out) {
    return deriv(g, loc, 2, dim, F, out);
}

// computeDiff of n fields at locations loc, loc + 1, ...
static int diff(sr_fgrid *g, int loc, int n, const double *const *F, double *const *H) {
    Fields A{};
    for (int c = 0; c < n; c++) {
        if (!F[c] || !H[c]) return set_err(SR_ERR_ARG, "null array");
        if ((const double *)H[c] == F[c]) return set_err(SR_ERR_ARG, "H must not alias the field");
        A.F[c] = F[c];
        A.H[c] = H[c];
        A.f[c] = g->shape[loc + c];
    }
    const ColGeo G = node_geo(g, g->N[0]);
    hipLaunchKernelGGL(k_fd_diff, dim3(col_blocks(G), n), dim3(kColThreads), 0, g->s, G, A, g->M, col_met(g));
    HIPCHK(hipGetLastError());
    return SR_OK;
}

extern "C" int sr_vf_diff(sr_fgrid *g, const double *Vx, const double *Vy, const double *Vz, double *Hx, double *Hy,
                          double *Hz) {
    if (!g) return set_err(SR_ERR_ARG, "null handle");
    const double *F[3] = {Vx, Vy, Vz};
    double *H[3] = {Hx, Hy, Hz};
    if (one_launch(g, H, F)) return diff(g, SR_LOC_VX, 3, F, H);
    for (int c = 0; c < 3; c++) RETCHK(diff(g, SR_LOC_VX + c, 1, F + c, H + c));
    return SR_OK;
}

extern "C" int sr_sf_diff(sr_fgrid *g, const double *F, double *H) {
    if (!g) return set_err(SR_ERR_ARG, "null handle");
    return diff(g, SR_LOC_NODE, 1, &F, &H);
}

extern "C" int sr_vf_nlin(sr_fgrid *g, const double *Ux, const double *Uy, const double *Uz, const double *Vx,
                          const double *Vy, const double *Vz, double *Hx, double *Hy, double *Hz) {
    if (!g) return set_err(SR_ERR_ARG, "null handle");
    // each component's H is written from U_c and the three V_d; H_c must alias none of them,
    // including the other components' inputs
    const double *V[3] = {Vx, Vy, Vz};
    const double *U[3] = {Ux, Uy, Uz};
    double *H[3] = {Hx, Hy, Hz};
    for (int c = 0; c < 3; c++)
        for (int e = 0; e < 3; e++)
            if ((const double *)H[c] == U[e] || (const double *)H[c] == V[e])
                return set_err(SR_ERR_ARG, "H must not alias an input");
    for (int c = 0; c < 3; c++)
        if (!U[c] || !V[c] || !H[c]) return set_err(SR_ERR_ARG, "null array");
    const ColGeo G = node_geo(g, g->N[0]);
    const bool self = Ux == Vx && Uy == Vy && Uz == Vz;
    for (int part = 0, one = one_launch(g, H, U, V); part < (one ? 1 : 3); part++)
        hipLaunchKernelGGL((self ? k_fd_nlin<true> : k_fd_nlin<false>), dim3(col_blocks(G)), dim3(kColThreads), 0, g->s, G,
                           vel_geo(g), g->M, Ux, Uy, Uz, Vx, Vy, Vz, Hx, Hy, Hz, col_met(g), one ? 7 : 1 << part);
    HIPCHK(hipGetLastError());
    return SR_OK;
}

extern "C" int sr_sf_nlin(sr_fgrid *g, const double *Vx, const double *Vy, const double *Vz, const double *F,
                          double *H) {
    if (!g) return set_err(SR_ERR_ARG, "null handle");
    if (!F || !H || !Vx || !Vy || !Vz) return set_err(SR_ERR_ARG, "null array");
    if ((const double *)H == F || (const double *)H == Vx || (const double *)H == Vy || (const double *)H == Vz)
        return set_err(SR_ERR_ARG, "H must not alias an input");
    const ColGeo G = node_geo(g, g->N[0]);
    hipLaunchKernelGGL(k_fd_nlin_node, dim3(col_blocks(G)), dim3(kColThreads), 0, g->s, G, vel_geo(g), g->M, F, Vx, Vy, Vz, H,
                       col_met(g));
    HIPCHK(hipGetLastError());
    return SR_OK;
}

extern "C" int sr_divergence(sr_fgrid *g, const double *Vx, const double *Vy, const double *Vz, double *div) {
    if (!g) return set_err(SR_ERR_ARG, "null handle");
    if (!Vx || !Vy || !Vz || !div) return set_err(SR_ERR_ARG, "null array");
    if ((const double *)div == Vx || (const double *)div == Vy || (const double *)div == Vz)
        return set_err(SR_ERR_ARG, "div must not alias an input");
    const ColGeo G = node_geo(g, g->N[0] + 2, 1);
    hipLaunchKernelGGL(k_fd_divergence, dim3(col_blocks(G)), dim3(kColThreads), 0, g->s, G, vel_geo(g), g->M, Vx, Vy, Vz, div,
                       col_met(g));
    HIPCHK(hipGetLastError());
    return SR_OK;
}

extern "C" int sr_gradient(sr_fgrid *g, const double *F, double *Gx, double *Gy, double *Gz) {
    if (!g) return set_err(SR_ERR_ARG, "null handle");
    double *G[3] = {Gx, Gy, Gz};
    if (!F || !Gx || !Gy || !Gz) return set_err(SR_ERR_ARG, "null array");
    for (int c = 0; c < 3; c++)
        if ((const double *)G[c] == F) return set_err(SR_ERR_ARG, "the gradient must not alias F");
    const ColGeo C = node_geo(g, g->N[0]);
    for (int part = 0, one = one_launch(g, G, nullptr); part < (one ? 1 : 3); part++)
        hipLaunchKernelGGL(k_fd_gradient, dim3(col_blocks(C)), dim3(kColThreads), 0, g->s, C, vel_geo(g), g->M, F, Gx, Gy, Gz,
                           col_met(g), one ? 7 : 1 << part);
    HIPCHK(hipGetLastError());
    return SR_OK;
}

extern "C" int sr_bc_fill(sr_fgrid *g, int loc, const sr_bc *bc, double *F) {
    RETCHK(check_loc(g, loc));
    if (!bc || !F) return set_err(SR_ERR_ARG, "null argument");
    std::vector<GhostWave> ws;
    RETCHK(bc_waves(g, g->shape[loc], bc, ws));
    ts_ghost_waves(g->shape[loc], F, ws.data(), (int)ws.size(), g->s);
    HIPCHK(hipGetLastError());
    return SR_OK;
}

extern "C" int sr_jacobi_visc(sr_fgrid *g, int loc, const sr_jacobi_desc *jd, const sr_bc *bc, const double *R,
                              double *F, double *G, int *iters) {
    RETCHK(check_loc(g, loc));
    if (!jd || !bc || !R || !F || !G) return set_err(SR_ERR_ARG, "null argument");
    if (F == G || (const double *)F == R || (const double *)G == R) return set_err(SR_ERR_ARG, "F, G and R must be distinct arrays");
    if (jd->dt <= 0.0 || jd->cnTolerance <= 0.0) return set_err(SR_ERR_ARG, "dt and cnTolerance must be positive");
    if (jd->form == 0 && jd->Re <= 0.0) return set_err(SR_ERR_ARG, "Re must be positive");
    if (jd->form != 0 && jd->form != 1) return set_err(SR_ERR_ARG, "form must be 0 or 1");
    const FShape &f = g->shape[loc];
    std::vector<GhostWave> ws;
    RETCHK(bc_waves(g, f, bc, ws));
    JacobiCoef J = jacobi_coef(g->h, jd->dt, jd->form == 0 ? jd->Re : 0.0);
    J.vis = jd->coef;
    J.form = jd->form;
    for (int k = 0; k < 3; k++) J.ms[k] = f.s[k];
    if (jd->zCollocMetric) J.ms[2] = 0;
    int per[3] = {g->d.xPer, g->d.yPer, g->d.zPer};
    Bulk B = jacobi_bulk(f, per);
    long maxIterations = (long)(g->N[0] - 1) * (g->N[1] - 1) * (g->N[2] - 1);
    double *a = F, *b = G;
    JacobiIO io{g->jsync, g->dmax, g->hmax, g->jev, g->s};
    int sweeps = 0;
    hipError_t err = hipSuccess;
    int st = ts_jacobi_loop(f, g->M, B, a, b, R, J, ws.data(), (int)ws.size(), io, jd->cnTolerance, maxIterations,
                            &sweeps, &err);
    HIPCHK(err);
    int status = SR_OK;
    if (st == 1) status = set_err(SR_ERR_NOT_CONVERGED, "Jacobi iterations did not converge within the iteration limit");
    // the result lives in whichever buffer holds the converged iterate; the dropped iterate's BCs
    // are still on the stream, so the call waits for them too before G goes back to the caller
    if (a != F) HIPCHK(hipMemcpyAsync(F, a, sizeof(double) * fsz(f), hipMemcpyDeviceToDevice, g->s));
    HIPCHK(hipStreamSynchronize(g->s));
    if (iters) *iters = sweeps;
    return status;
}
