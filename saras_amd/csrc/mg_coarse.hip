// The coarse end of the V-cycle in one workgroup: levels first..last of the down leg, the coarsest
// solve and the up leg back to `first`, with every level's u and f in LDS (poisson.cc:239-279 limited
// to those levels; poisson_d3.cc smooth / coarsen / solve / prolong).
//
// One workgroup of 1024 threads works through some thirty phases between barriers, so what counts is
// the length of each phase, not any rate.  Levels are kept without their ghost layers: the neighbour
// beyond a boundary is resolved to the core node it copies when a thread sets up its share of a
// smoothing, up to three entries of both half rows of one column, whose coefficients, right-hand sides
// and reciprocal diagonals then stay in registers; a half sweep is five or six LDS reads a node.  The
// residual that a restriction reads is formed once per fine node, the dense coarsest operator is
// applied by all threads, and all levels' coefficients come in one block.
//
// Per cycle at 257^3 (levels 17^3 to 3^3): 47 us in FP32 and 50 us in FP64, against 66 and 76 us with
// ghost layers whose images every update wrote, index arithmetic in every half sweep and a residual
// evaluated once per tap; V(4,4) with the iterated coarsest level (Taylor-Green) 79 against 186 us, of
// which the 65 coarsest iterations take 19 (about 100 before).  The four half sweeps at 17^3 take 7 us,
// 10 us as three nodes of each colour per thread with all indices kept, 8 us in FP32 but 16 in FP64 with
// everything in registers (spills).  A level of more than 1024 columns of three (33 x 17 x 9, the first of
// the 129 x 65 x 33 grid in FP32: 1122) takes a second round in every half sweep, which sets its columns
// up again: 58 us a cycle there.
#include "mg_kernels.h"

#include <type_traits>

#include "mg_device.h"

namespace sr {
namespace {

constexpr int kThreads = 1024;

// entries of one level without ghost layers: the red-black half rows of mg_layout.h for core (i, j)
__host__ __device__ inline int core_size(const Lay &L) { return L.nx * L.ny * 2 * L.kh; }
__device__ inline int core_idx(const Lay &L, int i, int j, int k) {
    return ((i * L.ny + j) * 2 + ((i + j + k) & 1)) * L.kh + ((k + 1) >> 1);
}

// 0-based core index of ghost -1 (side 0) or n (side 1)
__device__ inline int ghost_core(int rule, int side, int n) { return ghost_src(rule, side ? n + 1 : 0, n) - 1; }

// One node: its entry, the entries of its six neighbours (x+, x-, y+, y-, z+, z-), the coefficient
// entries of its three indices, and which neighbours are ghosts (bits 0..5) and antisymmetric ones
// (bits 8..13).
struct Node {
    int own, nb[6], cx, cy, cz;
    unsigned ghosts;
};

__device__ inline Node make_node(const Lay &L, const Bc &bc, int i, int j, int k) {
    Node N;
    const int p[3] = {i, j, k}, n[3] = {L.nx, L.ny, L.nz};
    N.own = core_idx(L, i, j, k);
    N.cx = 4 * (i + 1);
    N.cy = 4 * (j + 1);
    N.cz = 4 * (k + 1);
    N.ghosts = 0;
#pragma unroll
    for (int d = 0; d < 3; d++)
#pragma unroll
        for (int s = 0; s < 2; s++) {   // s = 0: plus
            int g = p[d] + (s ? -1 : 1);
            const bool out = g < 0 || g >= n[d];
            if (out) {
                N.ghosts |= 1u << (2 * d + s);
                if (bc.rule[d] == G_ANTI) N.ghosts |= 256u << (2 * d + s);
                g = ghost_core(bc.rule[d], s ? 0 : 1, n[d]);
            }
            N.nb[2 * d + s] = core_idx(L, d == 0 ? g : i, d == 1 ? g : j, d == 2 ? g : k);
        }
    return N;
}

template <typename T> struct Lvl {
    T *u, *f;
    const T *cx, *cy, *cz;
};

// the neighbour sum of the seven-point operator
template <typename T, bool ANTI>
__device__ __forceinline__ T nb_sum(const Lvl<T> &V, const Node &N, const T *X, const T *Y, const T *Z) {
    T w[6];
#pragma unroll
    for (int q = 0; q < 6; q++) {
        w[q] = V.u[N.nb[q]];
        if (ANTI && (N.ghosts >> (8 + q) & 1u)) w[q] = -w[q];
    }
    return six(X[0], w[0], X[1], w[1], Y[0], w[2], Y[1], w[3], Z[0], w[4], Z[1], w[5]);
}

// Gauss-Seidel update of one node
template <typename T, bool ANTI>
__device__ __forceinline__ T gs_value(const Lvl<T> &V, const Node &N) {
    const T *X = V.cx + N.cx, *Y = V.cy + N.cy, *Z = V.cz + N.cz;
    return (nb_sum<T, ANTI>(V, N, X, Y, Z) - V.f[N.own]) / diag3<T>(X, Y, Z);
}

// n / d from the reciprocal r of d: the quotient n r and one correction by its exact remainder
// (Markstein's division step), correctly rounded but for rare last-digit cases
__device__ __forceinline__ double quot(double n, double d, double r) {
    const double q = n * r;
    return __builtin_fma(__builtin_fma(-d, q, n), r, q);
}
__device__ __forceinline__ float quot(float n, float d, float r) {
    const float q = n * r;
    return __builtin_fmaf(__builtin_fmaf(-d, q, n), r, q);
}

// A thread's share of a smoothing: K entries from h0 of both half rows of one column (i, j).  The
// column's x and y coefficients, the nodes' z coefficients, right-hand sides and reciprocal diagonals
// stay in registers over the sweeps; a half sweep reads the four neighbouring columns' and the own
// column's other half row from LDS.
template <typename T, int K> struct Column {
    int h0, kb1;                    // parity of colour 1 (of colour 0: 1 - kb1)
    int own, xp, xm, yp, ym;        // first entries of the colour-0 half rows
    T sxp, sxm, syp, sym;           // signs of antisymmetric neighbours
    T X0, X1, Y0, Y1, cxy;
    T Z0[2][K], Z1[2][K], d[2][K], r[2][K], f[2][K];
    bool ok[2][K];
};

template <typename T, bool ANTI, int K>
__device__ __forceinline__ Column<T, K> make_column(const Lay &L, const Lvl<T> &V, const Bc &bc, int item, int nch) {
    Column<T, K> C;
    int i, j, ch;
    split3(div3(L.ny, nch), item, i, j, ch);
    const bool some = i < L.nx;
    i = min(i, L.nx - 1);
    C.h0 = ch * K;
    C.kb1 = (i + j) & 1;
    const int kh = L.kh;
    auto row = [&](int a, int b) { return (a * L.ny + b) * 2 * kh; };
    C.own = row(i, j);
    C.xp = row(i + 1 < L.nx ? i + 1 : ghost_core(bc.rule[0], 1, L.nx), j);
    C.xm = row(i > 0 ? i - 1 : ghost_core(bc.rule[0], 0, L.nx), j);
    C.yp = row(i, j + 1 < L.ny ? j + 1 : ghost_core(bc.rule[1], 1, L.ny));
    C.ym = row(i, j > 0 ? j - 1 : ghost_core(bc.rule[1], 0, L.ny));
    if (ANTI) {
        C.sxp = bc.rule[0] == G_ANTI && i + 1 == L.nx ? T(-1) : T(1);
        C.sxm = bc.rule[0] == G_ANTI && i == 0 ? T(-1) : T(1);
        C.syp = bc.rule[1] == G_ANTI && j + 1 == L.ny ? T(-1) : T(1);
        C.sym = bc.rule[1] == G_ANTI && j == 0 ? T(-1) : T(1);
    }
    const T *X = V.cx + 4 * (i + 1), *Y = V.cy + 4 * (j + 1);
    C.X0 = X[0]; C.X1 = X[1]; C.Y0 = Y[0]; C.Y1 = Y[1];
    if constexpr (sizeof(T) == 8) C.cxy = (X[0] + X[1]) + (Y[0] + Y[1]);
    else C.cxy = X[2] + Y[2];
#pragma unroll
    for (int c = 0; c < 2; c++)
#pragma unroll
        for (int q = 0; q < K; q++) {
            const int h = C.h0 + q, kp = 2 * h + (c ? C.kb1 : 1 - C.kb1);
            C.ok[c][q] = some && kp >= 1 && kp <= L.nz;
            const T *Z = V.cz + 4 * min(kp, L.nz + 1);
            C.Z0[c][q] = Z[0];
            C.Z1[c][q] = Z[1];
            const T cz = sizeof(T) == 8 ? Z[0] + Z[1] : Z[2];
            C.d[c][q] = C.cxy + cz;
            C.r[c][q] = T(1) / C.d[c][q];
            C.f[c][q] = V.f[C.own + c * kh + min(h, kh - 1)];
        }
    return C;
}

// neighbour sums of the column's nodes of colour c
template <typename T, bool ANTI, int K>
__device__ __forceinline__ void column_sums(const Lay &L, const Lvl<T> &V, const Bc &bc, const Column<T, K> &C, int c,
                                            T (&s)[K]) {
    const int kh = L.kh, o = (c ^ 1) * kh, kb = c ? C.kb1 : 1 - C.kb1;
    const T *u = V.u + o;
    // the other half row's entries h0 - 1 + kb .. h0 + K - 1 + kb.  Where kb is 1 that row holds the z
    // ghosts, its first and last entries: they are read from the nodes they copy.
    T z[K + 1];
#pragma unroll
    for (int q = 0; q <= K; q++) {
        const int e = C.h0 - 1 + kb + q;
        const bool lo = q == 0 && kb && e == 0, hi = q > 0 && e == kh - 1;
        const int g = lo || hi ? (ghost_core(bc.rule[2], hi, L.nz) + 1) >> 1 : min(max(e, 0), kh - 1);
        z[q] = u[C.own + g];
        if (ANTI && bc.rule[2] == G_ANTI && (lo || hi)) z[q] = -z[q];
    }
#pragma unroll
    for (int q = 0; q < K; q++) {
        const int h = min(C.h0 + q, kh - 1);
        T xp = u[C.xp + h], xm = u[C.xm + h], yp = u[C.yp + h], ym = u[C.ym + h];
        if (ANTI) {
            xp *= C.sxp;
            xm *= C.sxm;
            yp *= C.syp;
            ym *= C.sym;
        }
        s[q] = six(C.X0, xp, C.X1, xm, C.Y0, yp, C.Y1, ym, C.Z0[c][q], z[q + 1], C.Z1[c][q], z[q]);
    }
}

// `count` red-black sweeps; zero: u is not set and counts as zero.  With res, the residual f - L u of
// the colour-0 nodes is left there (slots (i, j, h)): a sweep ends on colour 1, whose residual is then
// zero.
template <typename T, bool ANTI, int K>
__device__ inline void smooth_columns(const Lay &L, const Lvl<T> &V, const Bc &bc, int count, bool zero, T *res) {
    const int kh = L.kh, nch = (kh - 2 + K) / K, n = L.nx * L.ny * nch;
    const bool one = n <= kThreads;   // every item has its own thread: set up once
    Column<T, K> C = make_column<T, ANTI, K>(L, V, bc, (int)threadIdx.x, nch);
#pragma unroll 1
    for (int sc = 0; sc < 2 * count + (res ? 1 : 0); sc++) {
#pragma unroll 1
        for (int t = threadIdx.x; t < n; t += kThreads) {
            if (!one) C = make_column<T, ANTI, K>(L, V, bc, t, nch);
            auto part = [&](auto cc) {
                constexpr int c = decltype(cc)::value;
                T s[K];
                if (zero && sc == 0) {
#pragma unroll
                    for (int q = 0; q < K; q++) s[q] = T(0);
                } else {
                    column_sums<T, ANTI, K>(L, V, bc, C, c, s);
                }
#pragma unroll
                for (int q = 0; q < K; q++) {
                    const int e = C.h0 + q;
                    if (!C.ok[c][q]) continue;
                    if (sc < 2 * count) V.u[C.own + c * kh + e] = quot(s[q] - C.f[c][q], C.d[c][q], C.r[c][q]);
                    else res[(C.own >> 1) + e] = C.f[c][q] - (s[q] - C.d[c][q] * V.u[C.own + c * kh + e]);
                }
            };
            if (sc & 1) part(std::integral_constant<int, 1>{});
            else part(std::integral_constant<int, 0>{});
        }
        __syncthreads();
    }
}

// one entry per thread where that fits the workgroup (short chains), three otherwise (fewer reads)
template <typename T, bool ANTI>
__device__ inline void smooth(const Lay &L, const Lvl<T> &V, const Bc &bc, int count, bool zero, T *res) {
    if (L.nx * L.ny * (L.kh - 1) <= kThreads) smooth_columns<T, ANTI, 1>(L, V, bc, count, zero, res);
    else smooth_columns<T, ANTI, 3>(L, V, bc, count, zero, res);
}

// a fine position along one direction as the residual pads give it: core index and factor
__device__ inline int pad_src(int rule, int q, int n, int &fac) {
    if (q >= 0 && q < n) return q;
    if (rule > G_ANTI) {
        fac = 0;
        return 0;
    }
    if (rule == G_ANTI) fac = -fac;
    return ghost_core(rule, q < 0 ? 0 : 1, n);
}

// Full weighting (poisson_d3.cc:250-298) to the coarse right-hand side fc.  rb: from the colour-0
// residuals alone, the coincident node and the 12 edge points; else from all 27 points of r, which has
// the level's own layout.
template <typename T>
__device__ inline void restrict_to(const Lay &F, const T *r, const Bc &tb, const Lay &C, T *fc, bool rb) {
    const Div3 dv = div3(C.ny, C.nz);
#pragma unroll 1
    for (int t = threadIdx.x; t < C.nx * C.ny * C.nz; t += kThreads) {
        int i, j, k;
        split3(dv, t, i, j, k);
        int ix[3], jx[3], kx[3], fi[3], fj[3], fk[3];
#pragma unroll
        for (int a = 0; a < 3; a++) {
            fi[a] = fj[a] = fk[a] = 1;
            ix[a] = pad_src(tb.rule[0], 2 * i + a - 1, F.nx, fi[a]);
            jx[a] = pad_src(tb.rule[1], 2 * j + a - 1, F.ny, fj[a]);
            kx[a] = pad_src(tb.rule[2], 2 * k + a - 1, F.nz, fk[a]);
        }
        auto R = [&](int a, int b, int e) -> T {
            const int fac = fi[a + 1] * fj[b + 1] * fk[e + 1];
            const int ii = ix[a + 1], jj = jx[b + 1], kk = kx[e + 1];
            const T v = rb ? r[(ii * F.ny + jj) * F.kh + ((kk + 1) >> 1)] : r[core_idx(F, ii, jj, kk)];
            return fac == 0 ? T(0) : fac < 0 ? -v : v;
        };
        T v;
        const T edgePoints = (R(1, 1, 0) + R(1, -1, 0) + R(-1, -1, 0) + R(-1, 1, 0) + R(0, 1, 1) + R(0, -1, 1) +
                              R(0, -1, -1) + R(0, 1, -1) + R(1, 0, 1) + R(1, 0, -1) + R(-1, 0, -1) + R(-1, 0, 1)) *
                             T(0.03125);
        if (rb) {
            v = edgePoints + R(0, 0, 0) * T(0.125);
        } else {
            const T facePoints = (R(1, 0, 0) + R(-1, 0, 0) + R(0, 1, 0) + R(0, -1, 0) + R(0, 0, 1) + R(0, 0, -1)) *
                                 T(0.0625);
            const T vertPoints = (R(1, 1, 1) + R(1, 1, -1) + R(1, -1, 1) + R(-1, 1, 1) + R(1, -1, -1) +
                                  R(-1, 1, -1) + R(-1, -1, 1) + R(-1, -1, -1)) *
                                 T(0.015625);
            v = facePoints + edgePoints + vertPoints + R(0, 0, 0) * T(0.125);
        }
        fc[core_idx(C, i, j, k)] = v;
    }
    __syncthreads();
}

// u += P e (trilinear, poisson_d3.cc:301-388) on the core nodes, or with color1 on the colour-1 nodes
// only: the post-smoothing that follows overwrites the others without reading them
template <typename T>
__device__ inline void prolong_add(const Lay &F, T *u, const Lay &C, const T *e, bool color1) {
    const int kc = color1 ? F.kh : F.nz;
    const Div3 dv = div3(F.ny, kc);
#pragma unroll 1
    for (int t = threadIdx.x; t < F.nx * F.ny * kc; t += kThreads) {
        int i, j, k;
        split3(dv, t, i, j, k);
        if (color1) {
            k = 2 * k + ((i + j) & 1) - 1;
            if (k < 0 || k >= F.nz) continue;
        }
        const int io = i & 1, jo = j & 1, ko = k & 1;
        const int ci = i >> 1, cj = j >> 1, ck = k >> 1;
        auto E = [&](int a, int b, int q) { return e[core_idx(C, ci + a, cj + b, ck + q)]; };
        T v;
        const int odd = io + jo + ko;
        if (odd == 3)
            v = (E(0, 0, 0) + E(1, 0, 0) + E(0, 1, 0) + E(0, 0, 1) + E(1, 1, 0) + E(1, 0, 1) + E(0, 1, 1) +
                 E(1, 1, 1)) / T(8.0);
        else if (odd == 1)
            v = (E(0, 0, 0) + E(io, jo, ko)) / T(2.0);
        else if (odd == 0)
            v = E(0, 0, 0);
        else   // the two in-between corners: four corners of the face, z pairs first
            v = ko ? (E(0, 0, 0) + E(0, 0, 1) + E(io, jo, 0) + E(io, jo, 1)) / T(4.0)
                   : (E(0, 0, 0) + E(0, 1, 0) + E(1, 0, 0) + E(1, 1, 0)) / T(4.0);
        u[core_idx(F, i, j, k)] += v;
    }
    __syncthreads();
}

// f -= (w f) / (w 1) on the coarsest level (coarseProject); one item per thread and round
template <typename T>
__device__ inline void project(const Lay &L, T *f, const double *wx, const double *wy, const double *wz, double wsum,
                               double *red) {
    const Div3 dv = div3(L.ny, L.nz);
    double s = 0;
    for (int t = threadIdx.x; t < L.nx * L.ny * L.nz; t += kThreads) {
        int i, j, k;
        split3(dv, t, i, j, k);
        s += wx[i] * wy[j] * wz[k] * (double)f[core_idx(L, i, j, k)];
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    double tot = 0;
    for (int w = 0; w < kThreads / 64; ++w) tot += red[w];
    const double c = tot / wsum;
    for (int t = threadIdx.x; t < L.nx * L.ny * L.nz; t += kThreads) {
        int i, j, k;
        split3(dv, t, i, j, k);
        const int o = core_idx(L, i, j, k);
        f[o] = (T)((double)f[o] - c);
    }
    __syncthreads();
}

// u = P f with the dense coarsest inverse (transposed: pt[j * nc + i] = P[i][j]; node order (i, j, k), k
// fastest).  The columns are shared out over the threads, `parts` groups per row; the partial sums
// (FP64) meet in scr in column order.  pv: entry threadIdx.x of pt, loaded at kernel start, when nc * nc
// <= kThreads.
template <typename T>
__device__ inline void direct(const Lay &L, T *u, const T *f, const T *__restrict__ pt, int nc, T pv, double *scr) {
    const int parts = nc * nc <= kThreads ? nc : max(1, kThreads / nc), per = (nc + parts - 1) / parts;
    const Div3 dv = div3(L.ny, L.nz);
    auto at = [&](int q) {
        int i, j, k;
        split3(dv, q, i, j, k);
        return core_idx(L, i, j, k);
    };
    const int part = (int)fdivu(threadIdx.x, (unsigned)nc, 1.0f / (float)nc), row = (int)threadIdx.x - part * nc;
    if (part < parts) {
        double acc = 0.0;
        if (per == 1) {
            acc = (double)pv * (double)f[at(part)];
        } else {
            const int j1 = min(nc, (part + 1) * per);
            for (int j0 = part * per; j0 < j1; j0 += 8) {
                T p[8];
#pragma unroll
                for (int q = 0; q < 8; q++) p[q] = pt[(long)min(j0 + q, j1 - 1) * nc + row];
#pragma unroll
                for (int q = 0; q < 8; q++)
                    if (j0 + q < j1) acc += (double)p[q] * (double)f[at(j0 + q)];
            }
        }
        scr[part * nc + row] = acc;
    }
    __syncthreads();
    if ((int)threadIdx.x < nc) {
        double acc = scr[threadIdx.x];
        for (int q = 1; q < parts; q++) acc += scr[q * nc + threadIdx.x];
        u[at((int)threadIdx.x)] = (T)acc;
    }
    __syncthreads();
}

// The coarsest-level iteration of poisson_d3.cc:190-247 with the red-black sweep: {ghosts; colour 0;
// ghosts; colour 1; max |r|} until max |r| < tol or more than max_count iterations.  The residual is
// evaluated before the next ghost update, so a colour-0 node sees its ghost neighbours, which copy
// colour-1 nodes, as they were before the colour-1 half sweep.  Whether the maximum is below tol is
// voted on by all nodes.  Returns the iteration count.

// at most 64 nodes: one wave, a node's value in its lane, neighbours by lane exchange
template <typename T, bool ANTI>
__device__ inline int gs_wave(const Lay &L, const Lvl<T> &V, const Bc &bc, double tol, int max_count) {
    const int lane = threadIdx.x, nc = L.nx * L.ny * L.nz;
    const Div3 dv = div3(L.ny, L.nz);
    int i = 0, j = 0, k = 0;
    if (lane < nc) split3(dv, lane, i, j, k);
    const bool own = lane < nc;
    const Node N = make_node(L, bc, i, j, k);
    int src[6];   // neighbour lanes
#pragma unroll
    for (int d = 0; d < 3; d++)
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const int n = d == 0 ? L.nx : d == 1 ? L.ny : L.nz, p = d == 0 ? i : d == 1 ? j : k;
            int g = p + (s ? -1 : 1);
            if (g < 0 || g >= n) g = ghost_core(bc.rule[d], s ? 0 : 1, n);
            src[2 * d + s] = d == 0 ? (g * L.ny + j) * L.nz + k : d == 1 ? (i * L.ny + g) * L.nz + k
                                                                         : (i * L.ny + j) * L.nz + g;
        }
    const T *X = V.cx + N.cx, *Y = V.cy + N.cy, *Z = V.cz + N.cz;
    const T c0 = X[0], c1 = X[1], c2 = Y[0], c3 = Y[1], c4 = Z[0], c5 = Z[1], dg = diag3<T>(X, Y, Z);
    const T fm = own ? V.f[N.own] : T(0);
    const int col = own ? (i + j + k) & 1 : 2;
    T v = T(0), w[6], x[6];
    auto gather = [&](T (&o)[6]) {
#pragma unroll
        for (int q = 0; q < 6; q++) {
            o[q] = __shfl(v, src[q], 64);
            if (ANTI && (N.ghosts >> (8 + q) & 1u)) o[q] = -o[q];
        }
    };
    auto sum = [&](const T (&o)[6]) { return six(c0, o[0], c1, o[1], c2, o[2], c3, o[3], c4, o[4], c5, o[5]); };
    int it = 0;
    gather(x);
    while (true) {
        if (col == 0) v = (sum(x) - fm) / dg;
        gather(w);
        if (col == 1) v = (sum(w) - fm) / dg;
        gather(x);
        T y[6];
#pragma unroll
        for (int q = 0; q < 6; q++) y[q] = col == 0 && (N.ghosts >> q & 1u) ? w[q] : x[q];
        const T lu = sum(y) - dg * v;
        const double m = fmax(-1.0e-10, fabs((double)fm - (double)lu));
        if (!__any(own && !(m < tol))) break;
        it += 1;
        if (it > max_count) break;
    }
    if (own) V.u[N.own] = v;
    return it;
}

// up to kThreads nodes: one node per thread, values in LDS
template <typename T, bool ANTI>
__device__ inline int gs_block(const Lay &L, const Lvl<T> &V, const Bc &bc, double tol, int max_count) {
    const int nc = L.nx * L.ny * L.nz;
    const bool own = (int)threadIdx.x < nc;
    int i, j, k;
    split3(div3(L.ny, L.nz), own ? (int)threadIdx.x : 0, i, j, k);
    const Node N = make_node(L, bc, i, j, k);
    const int col = own ? (i + j + k) & 1 : 2;
    if (own) V.u[N.own] = T(0);
    __syncthreads();
    int it = 0;
    while (true) {
        if (col == 0) V.u[N.own] = gs_value<T, ANTI>(V, N);
        __syncthreads();
        T w[6], v = T(0);
#pragma unroll
        for (int e = 0; e < 6; e++) w[e] = V.u[N.nb[e]];   // colour 0: the ghosts as its residual sees them
        if (col == 1) v = gs_value<T, ANTI>(V, N);
        __syncthreads();
        if (col == 1) V.u[N.own] = v;
        __syncthreads();
        const T *X = V.cx + N.cx, *Y = V.cy + N.cy, *Z = V.cz + N.cz;
#pragma unroll
        for (int e = 0; e < 6; e++) {
            if (!(col == 0 && (N.ghosts >> e & 1u))) w[e] = V.u[N.nb[e]];
            if (ANTI && (N.ghosts >> (8 + e) & 1u)) w[e] = -w[e];
        }
        const T lu = fma(-diag3<T>(X, Y, Z), V.u[N.own],
                         six(X[0], w[0], X[1], w[1], Y[0], w[2], Y[1], w[3], Z[0], w[4], Z[1], w[5]));
        const double m = fmax(-1.0e-10, fabs((double)V.f[N.own] - (double)lu));
        if (!__syncthreads_or(own && !(m < tol))) break;
        it += 1;
        if (it > max_count) break;
    }
    return it;
}

template <typename T, bool ANTI>
__global__ void __launch_bounds__(kThreads) k_coarse_cycle(CoarseDesc D, T *__restrict__ u_first,
                                                           const T *__restrict__ f_first, int *__restrict__ iters) {
    extern __shared__ unsigned char smem[];
    __shared__ double red[kThreads / 64];
    T *const base = (T *)smem;
    const int nl = D.last - D.first + 1, tid = (int)threadIdx.x;
    T *const scr = base + D.off_s;
    // the dense coarsest operator where one entry per thread holds it: loaded now, used at the bottom
    const T pv = D.pinv && tid < D.ncd * D.ncd && D.ncd * D.ncd <= kThreads ? ((const T *)D.pinv)[tid] : T(0);
    // coefficients of all levels (one block in LDS order) and the first level's right-hand side into
    // LDS; the loads are issued in batches before their LDS stores (each is a round trip to memory)
    {
        const Lay &L = D.L[0];
        const int n = core_size(L);
        const Div3 dv = div3(L.ny, 2 * L.kh);
        const T *cb = (const T *)D.coef;
        T *f = base + D.off_f[0];
#pragma unroll 1
        for (int t0 = tid; t0 < max(n, D.ncoef); t0 += 8 * kThreads) {
            T v[8];
#pragma unroll
            for (int q = 0; q < 8; q++) {
                int i, j, e;
                split3(dv, min(t0 + q * kThreads, n - 1), i, j, e);
                v[q] = f_first[((long)(i + 1) * (L.ny + 2) + (j + 1)) * 2 * L.khs + e];
            }
            const T c = t0 < D.ncoef ? cb[t0] : T(0);
#pragma unroll
            for (int q = 0; q < 8; q++)
                if (t0 + q * kThreads < n) f[t0 + q * kThreads] = v[q];
            if (t0 < D.ncoef) base[D.off_c[0][0] + t0] = c;
        }
        for (int t = tid + kThreads; t < D.ncoef; t += kThreads) base[D.off_c[0][0] + t] = cb[t];
    }
    __syncthreads();
    auto lvl = [&](int q) {
        return Lvl<T>{base + D.off_u[q], base + D.off_f[q], base + D.off_c[q][0], base + D.off_c[q][1],
                      base + D.off_c[q][2]};
    };
    // down leg, bottom and up leg in one loop: the kernel is straight-line work done once, and the
    // less code it runs through the fewer instruction fetches it waits for
#pragma unroll 1
    for (int step = 0; step < 2 * nl - 1; step++) {
        const bool down = step < nl - 1;
        const int q = down ? step : 2 * nl - 2 - step;
        const Lay L = D.L[q];
        const Lvl<T> V = lvl(q);
        if (step == nl - 1) {
            int it = 0;
            if (D.pinv) {
                direct<T>(L, V.u, V.f, (const T *)D.pinv, D.ncd, pv, (double *)scr);
            } else {
                if (D.project) project<T>(L, V.f, D.wc[0], D.wc[1], D.wc[2], D.wcsum, red);
                if (L.nx * L.ny * L.nz <= 64) {
                    if (tid < 64) it = gs_wave<T, ANTI>(L, V, D.bc, D.tol, D.max_count);
                } else {
                    it = gs_block<T, ANTI>(L, V, D.bc, D.tol, D.max_count);
                }
                __syncthreads();
            }
            if (tid == 0) iters[0] = it;
            continue;
        }
        if (!down) prolong_add<T>(L, V.u, D.L[q + 1], base + D.off_u[q + 1], D.post > 0);
        smooth<T, ANTI>(L, V, D.bc, down ? D.pre : D.post, down, down && D.pre > 0 ? scr : nullptr);
        if (!down) continue;
        if (D.pre == 0) {
            // without pre-smoothing u is zero and the residual is the right-hand side
            for (int t = tid; t < core_size(L); t += kThreads) V.u[t] = T(0);
        }
        restrict_to<T>(L, D.pre > 0 ? scr : V.f, D.tbc, D.L[q + 1], base + D.off_f[q + 1], D.pre > 0);
    }
    // the first level back, with its face-ghost images
    {
        const Lay &L = D.L[0];
        const T *u = base + D.off_u[0];
        const int row2 = 2 * L.kh;
        const Div3 dv = div3(L.ny, row2);
#pragma unroll 1
        for (int t = tid; t < core_size(L); t += kThreads) {
            int i, j, e;
            split3(dv, t, i, j, e);
            const int c = e >= L.kh ? 1 : 0, h = e - c * L.kh;
            const int ip = i + 1, jp = j + 1, kp = 2 * h + ((c + 1 + ip + jp) & 1);
            if (kp < 1 || kp > L.nz) continue;
            const T v = u[t];
            u_first[lay_row(L, ip, jp, c) + h] = v;
            if (ip == 2 || ip == L.nx - 1 || jp == 2 || jp == L.ny - 1 || kp == 2 || kp == L.nz - 1)
                write_images(L, u_first, ip, jp, kp, v, D.bc);
        }
    }
}

}  // namespace

// LDS offsets (elements of T) of the levels' arrays and the scratch, which holds one colour of the
// first level or the dense solve's partial sums; returns the bytes, or more than any limit when the
// coarsest level has more nodes than the workgroup has threads
template <typename T>
size_t coarse_cycle_plan(CoarseDesc &D) {
    size_t off = 0;
    auto take = [&](size_t n) { size_t o = off; off += (n + 7) & ~(size_t)7; return (int)o; };
    const int nl = D.last - D.first + 1;
    for (int q = 0; q < nl; q++) {
        D.off_u[q] = take((size_t)core_size(D.L[q]));
        D.off_f[q] = take((size_t)core_size(D.L[q]));
    }
    for (int q = 0; q < nl; q++) {
        D.off_c[q][0] = take(4 * (size_t)(D.L[q].nx + 2));
        D.off_c[q][1] = take(4 * (size_t)(D.L[q].ny + 2));
        D.off_c[q][2] = take(4 * (size_t)(D.L[q].nz + 2));
    }
    D.ncoef = (int)off - D.off_c[0][0];
    const size_t half = (size_t)core_size(D.L[0]) / 2, sums = kThreads * sizeof(double) / sizeof(T);
    D.off_s = take(half > sums ? half : sums);
    const Lay &C = D.L[nl - 1];
    if ((long)C.nx * C.ny * C.nz > kThreads) return ~(size_t)0;
    return off * sizeof(T);
}

template <typename T>
void launch_coarse_cycle(const CoarseDesc &D, size_t lds, T *u_first, const T *f_first, int *iters, hipStream_t s) {
    const bool anti = D.bc.rule[0] == G_ANTI || D.bc.rule[1] == G_ANTI || D.bc.rule[2] == G_ANTI;
    auto go = [&](auto k) { hipLaunchKernelGGL(k, dim3(1), dim3(kThreads), lds, s, D, u_first, f_first, iters); };
    anti ? go(k_coarse_cycle<T, true>) : go(k_coarse_cycle<T, false>);
}

template <typename T>
int coarse_cycle_attr(size_t lds) {
    const hipFuncAttribute a = hipFuncAttributeMaxDynamicSharedMemorySize;
    return hipFuncSetAttribute((const void *)k_coarse_cycle<T, false>, a, (int)lds) == hipSuccess &&
                   hipFuncSetAttribute((const void *)k_coarse_cycle<T, true>, a, (int)lds) == hipSuccess ? 0 : 1;
}

template size_t coarse_cycle_plan<double>(CoarseDesc &);
template size_t coarse_cycle_plan<float>(CoarseDesc &);
template void launch_coarse_cycle<double>(const CoarseDesc &, size_t, double *, const double *, int *, hipStream_t);
template void launch_coarse_cycle<float>(const CoarseDesc &, size_t, float *, const float *, int *, hipStream_t);
template int coarse_cycle_attr<double>(size_t);
template int coarse_cycle_attr<float>(size_t);

}  // namespace sr
