// One full red-black Gauss-Seidel sweep (colour 0, then colour 1) of a level in a single launch.
//
// Two half sweeps (k_rb_sweep) read the neighbour values of every node through seven vector loads and
// are held by the address unit, not by HBM: 121 us (FP64) and 63 us (FP32) a sweep at 257^3, where a
// sweep has to move 272 and 136 MB.  This kernel takes 55 and 40 us, 71 and 47 us as the last sweep of a
// smoothing, which stores colour 0 too.  FP64: 312 and 389 MB pass HBM, 5.4-5.7 TB/s, above the rate of a
// large copy.  FP32: 162 and 197 MB, 4.1 TB/s; its vector instructions (190 per four nodes) take 52-57 %
// of the time to issue, the rest goes with one workgroup per CU that waits at every plane's barrier.
//
// A workgroup marches over the planes of a chunk of x with a tile of y rows and the whole of z.  Each
// thread owns the two half-row entries 2t, 2t+1 of one row: its x neighbours stay in registers from
// plane to plane, its y and z neighbours come from LDS, and every u and f entry is loaded once (16 B
// in FP64).  Colour 1 of plane p - 1 is updated as soon as colour 0 of plane p is known.  Tiles and
// chunks overlap by one row and one plane in which colour 0 is updated twice, identically, by both
// neighbours.
//
// A neighbouring workgroup may still read colour 1 as it was before the sweep, so the new colour-1
// values go to another buffer than the old ones came from (bo != ub).  Colour 0 is never read before
// it is written, and only the last sweep of a smoothing stores it (LAST).
//
// Ghosts are not read: the neighbour beyond a boundary is resolved to the core node it copies
// (periodic, mirror, antisymmetric rules).  With LAST the face-ghost images of both colours are
// written, as k_rb_sweep writes them.
#include "mg_kernels.h"

#include "mg_march.h"
#include "xcd.h"

namespace sr {
template <typename T, bool ZERO, bool LAST, bool ZPER>
__global__ void __launch_bounds__(1024) k_rb_pass(Lay L, MarchGeo G, const T *__restrict__ ub, T *__restrict__ u,
                                                  T *__restrict__ bo, const T *__restrict__ f,
                                                  const T *__restrict__ cx, const T *__restrict__ cy,
                                                  const T *__restrict__ cz, Bc bc) {
    extern __shared__ unsigned char smem[];
    const int khs = L.khs, kh = L.kh, nx = L.nx, ny = L.ny;
    const unsigned b = xcd_block();
    const int chunk = (int)(b / (unsigned)G.ntile), tile = (int)b - chunk * G.ntile;
    const int j0 = 1 + tile * G.tq + min(tile, G.tr), j1 = j0 + G.tq + (tile < G.tr);
    const int i0 = 1 + chunk * G.cq + min(chunk, G.cr), i1 = i0 + G.cq + (chunk < G.cr);
    // thread rows: the tile's rows with one halo row on either side (rows past them repeat the last one)
    const int R = (int)blockDim.x / G.tpr;
    const int r = (int)fdivu(threadIdx.x, (unsigned)G.tpr, G.inv_tpr), t = (int)threadIdx.x - r * G.tpr;
    const int jp = min(j0 - 1 + r, j1);
    const bool halo = jp < j0 || jp >= j1, first = t == 0, last = t == G.tpr - 1;
    const int h0 = 2 * t;

    // core index of a position along x or y (0 and n+1 are ghosts), and whether its copy changes sign
    const bool antix = bc.rule[0] == G_ANTI, antiy = bc.rule[1] == G_ANTI;
    auto src = [&](int d, int q, int n) { return q >= 1 && q <= n ? q : ghost_src(bc.rule[d], q, n); };
    const int sj = src(1, jp, ny);
    const int sjm = src(1, sj - 1, ny), sjp = src(1, sj + 1, ny);
    const T ys = antiy && sj != jp ? T(-1) : T(1);
    const T ysm = antiy && sjm != sj - 1 ? T(-1) : T(1), ysp = antiy && sjp != sj + 1 ? T(-1) : T(1);
    const T zs = bc.rule[2] == G_ANTI ? T(-1) : T(1);
    const long ps = 2L * (ny + 2) * khs;
    // in-plane byte offsets of this thread's entries of colours 0 and 1, and of the rows beside it
    const unsigned w = sizeof(T), ob = khs * w;
    const unsigned vo0 = (unsigned)(sj * 2 * khs + h0) * w, vo1 = vo0 + ob;
    const unsigned vom = (unsigned)((sjm * 2 + 1) * khs + h0) * w, vop = (unsigned)((sjp * 2 + 1) * khs + h0) * w;

    // LDS: colour 1 (old) and colour 0 (new) of one plane each, two buffers; the z coefficients of
    // padded index 4t + q in entry q * tpr + t
    T *const lb = (T *)smem, *const la = lb + 2 * R * khs;
    const int lrow = r * khs;
    const unsigned lo2 = (unsigned)(lrow + h0) * w;
    const unsigned lom = r > 0 ? lo2 - ob : lo2, lop = r < R - 1 ? lo2 + ob : lo2;
    const int e0 = lrow + (first ? 0 : h0 - 1), e1 = lrow + (last ? h0 : h0 + 2);   // the third z neighbour
    Co<T> *const lz = (Co<T> *)(la + 2 * R * khs);
    for (int q = (int)threadIdx.x; q < 4 * G.tpr; q += (int)blockDim.x) {
        const int qq = (int)fdivu((unsigned)q, (unsigned)G.tpr, G.inv_tpr);
        lz[q] = ldco(cz + 4 * min(4 * (q - qq * G.tpr) + qq, L.nz + 1));
    }
    const Co<T> Y = ldco(cy + 4 * sj);

    // new value of one colour's entries of a row; own, xm, xp: the other colour in this row at the
    // plane and at the planes before and after; ym, yp: in the rows before and after; row: its LDS
    // rows, stored with sign ls
    auto update = [&](const Co<T> &X, const Pair<T> &own, const Pair<T> &xm, const Pair<T> &xp, const Pair<T> &ym,
                      const Pair<T> &yp, const T *row, T ls, const Pair<T> &fv, bool kb, const Co<T> &Z0,
                      const Co<T> &Z1) {
        const T ext = ls * row[kb ? e1 : e0];
        T lo = own.a, hi = own.b;
        if (ZPER) {
            if (first) lo = ls * row[lrow + kh - 2];
            if (last) hi = ls * row[lrow + 1];
        } else {
            lo = first ? zs * own.b : lo;
            hi = last ? zs * own.a : hi;
        }
        const T zm0 = kb ? lo : ext, zp0 = kb ? hi : own.a;
        const T zm1 = kb ? own.b : own.a, zp1 = kb ? ext : own.b;
        const T n0 = six(X.p, xp.a, X.m, xm.a, Y.p, yp.a, Y.m, ym.a, Z0.p, zp0, Z0.m, zm0) - fv.a;
        const T n1 = six(X.p, xp.b, X.m, xm.b, Y.p, yp.b, Y.m, ym.b, Z1.p, zp1, Z1.m, zm1) - fv.b;
        return Pair<T>{n0 / (cen(X) + cen(Y) + cen(Z0)), n1 / (cen(X) + cen(Y) + cen(Z1))};
    };
    // the entries of one colour's row at byte offset o.  Beside the core nodes a row holds its ghost
    // entries (kb = 0: first and last; kb = 1: the last is unused): they get their images, or, in
    // rows whose ghosts nobody reads, whatever was computed for them.
    auto store_row = [&](T *plane, unsigned o, const Pair<T> &v, bool kb) {
        if (!LAST) {
            st2(plane, o, v);
        } else if (!ZPER) {
            st2(plane, o, Pair<T>{first && !kb ? zs * v.b : v.a, last && !kb ? zs * v.a : v.b});
        } else {
            if (last) st1(plane, o, v.a);
            else if (first && !kb) st1(plane, o + w, v.b);
            else st2(plane, o, v);
            if (!kb && last) st1(plane, o - h0 * w, v.a);
            if (!kb && first) st1(plane, o + (kh - 1) * w, v.b);
        }
    };
    // the ghost row and the ghost plane that copy this row and a plane (at most one each: ny, nx >= 5)
    const int xs0 = ghost_src(bc.rule[0], 0, nx), xs1 = ghost_src(bc.rule[0], nx + 1, nx);
    const bool yi0 = sj == ghost_src(bc.rule[1], 0, ny), yimg = yi0 || sj == ghost_src(bc.rule[1], ny + 1, ny);
    // colour c at core plane i, with the face-ghost images of all directions where they are wanted
    auto store = [&](T *dst, int i, int c, const Pair<T> &v, bool kb) {
        const unsigned o = here(c ? vo1 : vo0);
        store_row(dst + i * ps, o, v, kb);
        if (!LAST) return;
        if (yimg)
            store_row(dst + i * ps, o + (unsigned)((yi0 ? 0 : ny + 1) - sj) * 2u * ob,
                      Pair<T>{antiy ? -v.a : v.a, antiy ? -v.b : v.b}, kb);
        if (i == xs0 || i == xs1)
            store_row(dst + (i == xs0 ? 0 : nx + 1) * ps, o, Pair<T>{antix ? -v.a : v.a, antix ? -v.b : v.b}, kb);
    };

    const Pair<T> none{T(0), T(0)};
    // rings over the planes: old colour 1 at p-1, p, p+1, p+2; new colour 0 at p-2, p-1, p; f of colour 0
    // at p, p+1 and of colour 1 at p-1, p; old colour 1 beside a halo row at p, p+1; x coefficients
    Pair<T> B[4] = {none, none, none, none}, A[4] = {none, none, none, none};
    Pair<T> F0[2] = {none, none}, F1[2] = {none, none}, Ym[2] = {none, none}, Yp[2] = {none, none};
    Co<T> Xs[4] = {};
    Pair<T> Bs = none;   // new colour 1, stored in the next turn
    int flip = 0;
    for (int p = i0 - 1; p <= i1; ++p, flip ^= 1) {
        Pair<T> &Bm = B[0], &Bc_ = B[1], &Bp = B[2], &Bn = B[3];
        Pair<T> &A2 = A[0], &A1 = A[1], &An = A[2];
        Co<T> &X1 = Xs[0], &X = Xs[1], &Xn = Xs[2];
        Pair<T> &f0 = F0[0], &f0n = F0[1], &f1 = F1[0], &f1n = F1[1];
        const int bsz = R * khs;
        T *const lbc = lb + flip * bsz, *const lbn = lb + bsz - flip * bsz;
        T *const lac = la + flip * bsz, *const lap = la + bsz - flip * bsz;
        const int s = src(0, p, nx);
        if (p == i0 - 1 || s != p || (p == i0 && i0 == 1)) {
            // the first plane, and the planes at a ghost plane, load all that their update needs
            X = ldco(cx + 4 * s);
            f0 = ld2(f + s * ps, here(vo0));
            if (!ZERO) {
                const int sm = src(0, s - 1, nx), sp = src(0, s + 1, nx);
                Bm = ld2(ub + sm * ps, here(vo1));
                Bc_ = ld2(ub + s * ps, here(vo1));
                Bp = ld2(ub + sp * ps, here(vo1));
                if (halo) {
                    Ym[0] = ld2(ub + s * ps, here(vom));
                    Yp[0] = ld2(ub + s * ps, here(vop));
                }
                if (antix && sm != s - 1) Bm = Pair<T>{-Bm.a, -Bm.b};
                if (antix && sp != s + 1) Bp = Pair<T>{-Bp.a, -Bp.b};
                // nobody reads this buffer: it was last read two planes ago
                st2(lbc, lo2, Pair<T>{ys * Bc_.a, ys * Bc_.b});
            }
            __syncthreads();
        } else if (!ZERO && antix && p == nx) {
            Bp = Pair<T>{-Bp.a, -Bp.b};
        }
        // The previous turn's results are stored here, behind the wait for this turn's loads and before
        // the next ones are issued: loads and stores retire in order, so a store issued at the end of a
        // turn would be waited for with the loads.
        if (!halo) {
            if (LAST && p > i0) store(u, p - 1, 0, A1, !((1 + p + jp) & 1));
            if (p > i0 + 1) store(bo, p - 2, 1, Bs, !((1 + p + jp) & 1));
        }
        // loads for the next plane: nothing uses them before the next turn
        if (p < i1) {
            const int s1 = src(0, p + 1, nx);
            Xn = ldco(cx + 4 * s1);
            f0n = ld2(f + s1 * ps, here(vo0));
            if (!ZERO) {
                Bn = ld2(ub + src(0, min(p + 2, nx + 1), nx) * ps, here(vo1));
                if (halo) {
                    Ym[1] = ld2(ub + s1 * ps, here(vom));
                    Yp[1] = ld2(ub + s1 * ps, here(vop));
                }
            }
            f1n = ld2(f + s * ps, here(vo1));
        }
        const bool kb = (1 + p + jp) & 1;
        const Co<T> Z0 = lz[(kb ? G.tpr : 0) + t], Z1 = lz[(kb ? 3 * G.tpr : 2 * G.tpr) + t];
        if (ZERO) {
            An.a = -f0.a / (cen(X) + cen(Y) + cen(Z0));
            An.b = -f0.b / (cen(X) + cen(Y) + cen(Z1));
        } else {
            Pair<T> m_ = ld2(lbc, lom), p_ = ld2(lbc, lop);
            if (halo) {
                m_ = Pair<T>{ysm * Ym[0].a, ysm * Ym[0].b};
                p_ = Pair<T>{ysp * Yp[0].a, ysp * Yp[0].b};
            }
            An = update(X, Bc_, Bm, Bp, m_, p_, lbc, ys, f0, kb, Z0, Z1);
        }
        if (antix && s != p) An = Pair<T>{-An.a, -An.b};
        // colour 1 of plane p - 1, whose parity is that of colour 0 here
        if (p > i0) Bs = update(X1, A1, A2, An, ld2(lap, lom), ld2(lap, lop), lap, T(1), f1, kb, Z0, Z1);
        if (p < i1) {
            st2(lac, lo2, Pair<T>{ys * An.a, ys * An.b});
            if (!ZERO) st2(lbn, lo2, Pair<T>{ys * Bp.a, ys * Bp.b});
            __syncthreads();
        }
        Bm = Bc_;
        Bc_ = Bp;
        Bp = Bn;
        A2 = A1;
        A1 = An;
        X1 = X;
        X = Xn;
        f0 = f0n;
        f1 = f1n;
        Ym[0] = Ym[1];
        Yp[0] = Yp[1];
    }
    if (!halo) store(bo, i1 - 1, 1, Bs, (1 + i1 + jp) & 1);
}

// Image rules only (and march_ok's sizes).
bool rb_pass_ok(const Lay &L, const Bc &bc) {
    for (int d = 0; d < 3; d++)
        if (bc.rule[d] > G_ANTI) return false;
    return march_ok(L);
}

template <typename T, bool ZERO, bool LAST, bool ZPER>
static int attr1() {
    return hipFuncSetAttribute((const void *)k_rb_pass<T, ZERO, LAST, ZPER>, hipFuncAttributeMaxDynamicSharedMemorySize,
                               80 * 1024) == hipSuccess ? 0 : 1;
}
template <typename T>
static int attr8() {
    return attr1<T, false, false, false>() | attr1<T, false, true, false>() | attr1<T, true, false, false>() |
           attr1<T, true, true, false>() | attr1<T, false, false, true>() | attr1<T, false, true, true>() |
           attr1<T, true, false, true>() | attr1<T, true, true, true>();
}
int rb_pass_attr() { return attr8<double>() | attr8<float>(); }

template <typename T>
void launch_rb_pass(const Lay &L, const T *ub, T *u, T *bo, const T *f, const T *cx, const T *cy, const T *cz,
                    const Bc &bc, bool zero, bool last, hipStream_t s) {
    const MarchPlan P = march_plan(L);
    const dim3 grid(P.blocks()), blk(P.threads());
    const size_t lds = 4 * (size_t)P.g.R * L.khs * sizeof(T) + 4 * (size_t)P.g.tpr * sizeof(Co<T>);
    auto go = [&](auto k) { hipLaunchKernelGGL(k, grid, blk, lds, s, L, P.g, ub, u, bo, f, cx, cy, cz, bc); };
    const bool zper = bc.rule[2] == G_PERIODIC;
    if (zero && last) zper ? go(k_rb_pass<T, true, true, true>) : go(k_rb_pass<T, true, true, false>);
    else if (zero) zper ? go(k_rb_pass<T, true, false, true>) : go(k_rb_pass<T, true, false, false>);
    else if (last) zper ? go(k_rb_pass<T, false, true, true>) : go(k_rb_pass<T, false, true, false>);
    else zper ? go(k_rb_pass<T, false, false, true>) : go(k_rb_pass<T, false, false, false>);
}

template void launch_rb_pass<double>(const Lay &, const double *, double *, double *, const double *, const double *,
                                     const double *, const double *, const Bc &, bool, bool, hipStream_t);
template void launch_rb_pass<float>(const Lay &, const float *, float *, float *, const float *, const float *,
                                    const float *, const float *, const Bc &, bool, bool, hipStream_t);

}  // namespace sr
