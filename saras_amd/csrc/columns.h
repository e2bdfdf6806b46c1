// Stencil kernels over padded fields (k fastest) that march along x: work split, loads and the
// advection stencils shared by the time step (ts_kernels.hip) and the field operators (field_api.hip).
//
// A thread takes one (j, k) column of a chunk of planes, consecutive lanes consecutive entries of the
// padded plane.  What does not change along x is formed once per column (the place in the plane, byte
// offsets, y and z metrics), the x neighbours of a value stay in registers, and every load is a plane's
// address plus a 32-bit offset.  One thread per entry instead spent some 300 instructions per wavefront
// on indices and metrics and was bound by them: 163 us for the second derivatives of a 257^3 field, which
// move 0.41 GB.  Here it is 116 us.  At 257^3 the L1 caches read 0.8 GB from the L2 caches for it and 2.6
// GB for the advection of a velocity (351 us), 7 TB/s, neighbouring rows among them, about 20 us per
// array; HBM carries 1.02 to 1.4 times what a kernel has to move, at 3.9-5.2 TB/s, where a large copy gets
// 4.75.  Workgroup size (256 or 1024), chunk length and order change these by a few per cent.
#pragma once

#include "ts_kernels.h"
#include "xcd.h"

namespace sr {

constexpr int kColThreads = 256;
// Workgroups per plane, chunks of planes, planes per chunk (quotient, remainder), and whether the
// workgroups of a chunk follow each other (by_chunk) or the chunks of a plane's part.
struct ColGeo {
    int nb, nch, cq, cr, by_chunk;
};
constexpr int kColPlanes = 64;   // most planes of a chunk
// Planes whose loads are issued together; 257^3 operators with 2 and 4: 1562 and 1580 us.
constexpr int kColAhead = 2;

// Padded planes of `rows` rows of `row` entries.  Eight workgroups per CU where the planes suffice, and at
// most kColPlanes planes each: the 257^3 operators with 1024 / 2048 / 4096 / 8192 / 16384 workgroups take
// 1611 / 1586 / 1571 / 1590 / 1683 us.  Short chunks hold an even number of planes where two are loaded
// together (ahead), as the last of an odd one leaves half of the loads unused (129^3: second derivatives
// 9.1 -> 8.7 us, one thread per entry 9.8; not with 1024 threads, of which two workgroups fill a CU: a
// Jacobi sweep 14.2 -> 16.6), and one plane only while that makes at most four workgroups per CU
// (257 x 5 x 257: advection of a node field 8.1 us with one plane, 6.5 with two; one thread per entry 6.0).
//
// Each XCD takes a contiguous eighth of the workgroups.  With the chunks of a plane's part after each
// other that is an eighth of the rows, whose neighbour rows belong to others: on 513 x 9 x 513 nodes one
// row and its two neighbours, and a node field's advection took 31.9 us, 23.8 with one thread per entry.
// There the workgroups of a chunk follow each other, an eighth of the planes per XCD: 21.6 us; 513 x 65 x
// 257 88.4 against 93.5.  From 16 rows per XCD on the first order is as good or better (129^3 20.0 / 20.4,
// 257^3 operators 1537 / 1562).
inline ColGeo col_geo(int rows, int row, int planes, int threads = kColThreads, int ahead = kColAhead) {
    const int scale = threads / kColThreads;
    ColGeo G;
    G.nb = (int)(((long)rows * row + threads - 1) / threads);
    G.nch = max(1, min(2048 / scale / G.nb, planes));
    const int len = (planes + G.nch - 1) / G.nch;
    if (planes < 2 * G.nch) {
        if ((long)G.nb * planes > 1024 / scale) G.nch = (planes + 1) / 2;
    } else if (scale == 1 && len < 8 && len % ahead) {
        const int even = (planes + len - 2) / (len - 1);
        if ((long)G.nb * even <= 2304) G.nch = even;
    }
    G.nch = max(G.nch, (planes + kColPlanes - 1) / kColPlanes);
    G.cq = planes / G.nch;
    G.cr = planes % G.nch;
    G.by_chunk = rows < 130 && planes > rows;
    return G;
}
inline unsigned col_blocks(const ColGeo &G) { return (unsigned)(G.nb * G.nch); }

// the thread's entry of the padded plane and the planes of its chunk, counted from 0
struct Col {
    unsigned t;
    int i0, i1;
};
__device__ inline Col column(const ColGeo &G) {
    const unsigned b = xcd_block(), inner = (unsigned)(G.by_chunk ? G.nb : G.nch), q = b / inner, r = b - q * inner;
    const unsigned tile = G.by_chunk ? r : q, chunk = G.by_chunk ? q : r;
    Col C;
    C.t = tile * blockDim.x + threadIdx.x;
    C.i0 = (int)chunk * G.cq + min((int)chunk, G.cr);
    C.i1 = C.i0 + G.cq + ((int)chunk < G.cr);
    return C;
}

// the values are loaded here, not where they are used: the compiler sinks loads into the guarded block of
// each plane otherwise, one plane's at a time
template <int N>
__device__ __forceinline__ void loaded(double (&a)[N]) {
#pragma unroll
    for (int u = 0; u < N; u++) asm volatile("" : "+v"(a[u]));
}

__device__ __forceinline__ double ldd(const double *base, unsigned off) {
    return *reinterpret_cast<const double *>(reinterpret_cast<const char *>(base) + off);
}
__device__ __forceinline__ void std_(double *base, unsigned off, double v) {
    *reinterpret_cast<double *>(reinterpret_cast<char *>(base) + off) = v;
}

// Metrics with the grid factors of the centred differences taken in: d1 F = a1 (F+ - F-) and
// d2 F = a2 (F+ - F-) + a3 (F+ - 2 F + F-).  The spacings are powers of two, so these are the
// reference's xi_x ((F+ - F-) / 2 ih) and so on to the last bit.
__device__ inline double met(const Metrics &M, int d, int node, int q, int i) { return M.m[d][node ? 0 : 1][q][i + 1]; }
__device__ inline double met1(const Metrics &M, int d, int node, int i, double ih) { return met(M, d, node, 1, i) * (0.5 * ih); }
__device__ inline double met2(const Metrics &M, int d, int node, int i, double ih) { return met(M, d, node, 2, i) * (0.5 * ih); }
__device__ inline double met3(const Metrics &M, int d, int node, int i, double ih, double half) {
    return half * met(M, d, node, 3, i) * (ih * ih);
}

// inverse spacings, and the weight of the second difference (1/2 where the solve is implicit)
struct ColMet {
    double ih[3], half;
};

// a staggered velocity's plane strides and row lengths (Vx and P share rows and in-plane offsets, Vy its
// rows, Vz has shorter rows)
struct VelGeo {
    int N[3];
    __host__ __device__ long sx() const { return (long)(N[1] + 2) * (N[2] + 2); }
    __host__ __device__ long sy() const { return (long)(N[1] + 1) * (N[2] + 2); }
    __host__ __device__ long sz() const { return (long)(N[1] + 2) * (N[2] + 1); }
};

// Velocities around node (i, j, k): a plain name is V(i, j, k), m/n the planes before/after, j/k the
// neighbours after it along y/z, d those before (along y for x, y, z with d; z with b: before along z).
struct Vels {
    double x, xm, xn, xj, xk, xmj, xmk, xd, xb;
    double y, ym, yn, yj, yk, yd, yb, ynd, ydk;
    double z, zm, zn, zj, zk, zd, zb, znb, zjb;
};

// the planes before the first one: everything that an iteration hands on to the next
__device__ __forceinline__ void vels_begin(Vels &v, const double *X, const double *Y, const double *Z, const VelGeo &G,
                                           unsigned o, unsigned oz, bool self) {
    const long sx = G.sx(), sy = G.sy(), sz = G.sz();
    const int r = G.N[2] + 2;
    v.xm = ldd(X - sx, o);
    v.xmj = ldd(X - sx + r, o);
    v.xmk = ldd(X - sx + 1, o);
    v.x = ldd(X, o);
    v.y = ldd(Y, o);
    v.yd = ldd(Y - r, o);
    v.z = ldd(Z, oz);
    v.zb = ldd(Z - 1, oz);
    if (self) {
        v.ym = ldd(Y - sy, o);
        v.zm = ldd(Z - sz, oz);
    }
}
// the loads of one plane and of the plane after it; lastx: Vx has none
__device__ __forceinline__ void vels_load(Vels &v, const double *X, const double *Y, const double *Z, const VelGeo &G,
                                          unsigned o, unsigned oz, bool self, bool lastx) {
    const long sx = G.sx(), sy = G.sy(), sz = G.sz();
    const int r = G.N[2] + 2, rz = G.N[2] + 1;
    v.xn = ldd(lastx ? X : X + sx, o);
    v.yn = ldd(Y + sy, o);
    v.ynd = ldd(Y + sy - r, o);
    v.zn = ldd(Z + sz, oz);
    v.znb = ldd(Z + sz - 1, oz);
    v.xj = ldd(X + r, o);
    v.xk = ldd(X + 1, o);
    v.yk = ldd(Y + 1, o);
    v.ydk = ldd(Y - r + 1, o);
    v.zj = ldd(Z + rz, oz);
    v.zjb = ldd(Z + rz - 1, oz);
    if (self) {
        v.xd = ldd(X - r, o);
        v.xb = ldd(X - 1, o);
        v.yj = ldd(Y + r, o);
        v.yb = ldd(Y - 1, o);
        v.zk = ldd(Z + 1, oz);
        v.zd = ldd(Z - rz, oz);
    }
}
// on to the next plane
__device__ __forceinline__ void vels_next(Vels &v) {
    v.xm = v.x;
    v.xmj = v.xj;
    v.xmk = v.xk;
    v.x = v.xn;
    v.ym = v.y;
    v.y = v.yn;
    v.yd = v.ynd;
    v.zm = v.z;
    v.z = v.zn;
    v.zb = v.znb;
}

// a field's values around a node: along x, y, z after (p) and before (m)
struct Cross {
    double c, xp, xm, yp, ym, zp, zm;
};
__device__ __forceinline__ Cross cross_x(const Vels &v) { return Cross{v.x, v.xn, v.xm, v.xj, v.xd, v.xk, v.xb}; }
__device__ __forceinline__ Cross cross_y(const Vels &v) { return Cross{v.y, v.yn, v.ym, v.yj, v.yd, v.yk, v.yb}; }
__device__ __forceinline__ Cross cross_z(const Vels &v) { return Cross{v.z, v.zn, v.zm, v.zj, v.zd, v.zk, v.zb}; }

// computeNLin of component C at its face, u its stencil: acc -= (mean of the slices of V_d) d_d u, d = x,
// y, z.  a: first-derivative metrics of the three directions, a quarter of them where four slices are
// averaged (field.cc:309-575)
template <int C>
__device__ __forceinline__ double advect(double acc, const Vels &v, const Cross &u, double ax, double ay, double az) {
    const double ix = C == 0 ? v.x : C == 1 ? v.x + v.xm + v.xj + v.xmj : v.x + v.xm + v.xk + v.xmk;
    const double iy = C == 0 ? v.y + v.yd + v.yn + v.ynd : C == 1 ? v.y : v.y + v.yd + v.yk + v.ydk;
    const double iz = C == 0 ? v.z + v.zb + v.zn + v.znb : C == 1 ? v.z + v.zb + v.zj + v.zjb : v.z;
    acc -= ix * (ax * (u.xp - u.xm));
    acc -= iy * (ay * (u.yp - u.ym));
    acc -= iz * (az * (u.zp - u.zm));
    return acc;
}

// the three second derivatives of u added to acc, x first; X, Y, Z: a2 and a3 of each direction
__device__ __forceinline__ double diffuse(double acc, const Cross &u, double x2, double x3, double y2, double y3, double z2,
                                          double z3) {
    acc += x2 * (u.xp - u.xm) + x3 * (u.xp - 2.0 * u.c + u.xm);
    acc += y2 * (u.yp - u.ym) + y3 * (u.yp - 2.0 * u.c + u.ym);
    acc += z2 * (u.zp - u.zm) + z3 * (u.zp - 2.0 * u.c + u.zm);
    return acc;
}

}  // namespace sr
