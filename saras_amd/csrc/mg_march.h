// Kernels that march over the planes of a level with a tile of rows per workgroup (mg_pass.hip,
// mg_outer.hip): work split, paired loads and stores, coefficient triples.
//
// A workgroup takes a tile of y rows with one halo row on either side, the whole of z and a chunk of x
// planes.  Thread row r stands for row j0 - 1 + r; thread t of it for the half-row entries 2t, 2t + 1.
#pragma once

#include "mg_device.h"

namespace sr {

template <typename T> struct Pair { T a, b; };

// the value, opaque to the compiler.  Used on a lane's offset from a base that is the same for the whole
// wave: the address then stays scalar base + 32-bit offset; without it every array's 64-bit lane
// addresses are formed before the loop and live in registers.
__device__ __forceinline__ unsigned here(unsigned v) {
    asm volatile("" : "+v"(v));
    return v;
}
// two consecutive entries at a 32-bit byte offset
template <typename T>
__device__ __forceinline__ Pair<T> ld2(const T *base, unsigned off) {
    typedef T V2 __attribute__((ext_vector_type(2)));
    const V2 v = *reinterpret_cast<const V2 *>(reinterpret_cast<const char *>(base) + off);
    return Pair<T>{v.x, v.y};
}
template <typename T>
__device__ __forceinline__ void st2(T *base, unsigned off, const Pair<T> &v) {
    typedef T V2 __attribute__((ext_vector_type(2)));
    V2 w;
    w.x = v.a;
    w.y = v.b;
    *reinterpret_cast<V2 *>(reinterpret_cast<char *>(base) + off) = w;
}
template <typename T>
__device__ __forceinline__ void st1(T *base, unsigned off, T v) {
    *reinterpret_cast<T *>(reinterpret_cast<char *>(base) + off) = v;
}

// coefficients of one direction at one index: c+, c- and, in FP32, the separately rounded centre
// (see diag3)
template <typename T> struct Co;
template <> struct alignas(16) Co<double> { double p, m; };
template <> struct alignas(16) Co<float> { float p, m, c, pad; };
__device__ __forceinline__ double cen(const Co<double> &q) { return q.p + q.m; }
__device__ __forceinline__ float cen(const Co<float> &q) { return q.c; }
__device__ __forceinline__ Co<double> ldco(const double *q) { return Co<double>{q[0], q[1]}; }
__device__ __forceinline__ Co<float> ldco(const float *q) { return Co<float>{q[0], q[1], q[2], 0.0f}; }

struct MarchGeo {
    int ntile, nch, tpr, R;   // row tiles, chunks of x, threads per row, thread rows
    int tq, tr, cq, cr;       // rows per tile and planes per chunk: quotient and remainder
    float inv_tpr;
};

struct MarchPlan {
    MarchGeo g;
    int blocks() const { return g.ntile * g.nch; }
    int threads() const { return g.R * g.tpr; }
};

// Tiles of up to 13 rows (15 thread rows with the halo rows: 15 % of colour 0 updated twice) and as
// many chunks of x as give every CU its share of workgroups: one of 1024 threads (257 nodes along z:
// 240 workgroups of 21 planes), two of half that.  More chunks cost two planes each, fewer leave CUs
// idle.  Measured (us per solve or step, R = 15 / 11 / 19 rows with 512 workgroups): 129^3 step
// 3077 / 3135 / 3343, 65^3 GCR solve 1424 / 1446 / 1499; 15 rows with 256 workgroups 3140 and 1464.
// At 257^3 in FP64 1024 threads and 256 workgroups take 12.56 ms per solve, 512 threads and 512
// workgroups 12.85 ms, 715 threads and 512 workgroups 13.26 ms.  planes: the least planes of a chunk.
inline MarchPlan march_plan(const Lay &L, int planes = 1) {
    MarchPlan P{};
    P.g.tpr = L.kh / 2;
    P.g.inv_tpr = 1.0f / (float)P.g.tpr;
    int R = 1024 / P.g.tpr;
    if (R > 15) R = 15;
    if (R > L.ny + 2) R = L.ny + 2;
    P.g.ntile = (L.ny + R - 3) / (R - 2);
    P.g.tq = L.ny / P.g.ntile;
    P.g.tr = L.ny % P.g.ntile;
    P.g.R = P.g.tq + (P.g.tr > 0) + 2;
    P.g.nch = (P.threads() > 512 ? 256 : 512) / P.g.ntile;
    if (P.g.nch > L.nx / planes) P.g.nch = L.nx / planes;
    if (P.g.nch < 1) P.g.nch = 1;
    P.g.cq = L.nx / P.g.nch;
    P.g.cr = L.nx % P.g.nch;
    return P;
}

// Rows of an even number of entries of which at least six fit a workgroup (a z direction of at most 513
// nodes; beyond that the halo rows outweigh the tile).
inline bool march_ok(const Lay &L) {
    return L.kh % 2 == 0 && L.nx >= 5 && L.ny >= 5 && L.nz >= 5 && L.kh / 2 <= 170;
}

}  // namespace sr
