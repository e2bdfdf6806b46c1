// The outer step of the mixed-precision solves and the norms of the level-0 residual as marches over x
// (mg_march.h): every array is read once, the x neighbours stay in registers, the y and z neighbours
// come from LDS, and the last workgroup to finish combines the sums, so that a step is one launch.
//
//   k_march_residual   r = f - L u with its norms, u being read as it is (OUT_READ), u_in + e of a
//                      refinement step (OUT_ADD), or x_in + alpha (e - beta z) of a GCR step
//                      (OUT_GCR); or the norms alone, of both colours (OUT_NORM) or of colour 0 (OUT_NORM0)
//   k_march_dots       q = L e and p = L z in FP32 and the five products of the GCR step coefficients
//
// Per-node kernels of these steps (seven vector loads of neighbour values per quantity, ghosts filled, a
// second launch for the sums and a copy for the host) took at 257^3: GCR step and residual 82 + 147 + 5,
// products 87 + 8, norm of colour 0 58 + 5 us; these take 137, 71 and 65.  A GCR step has to move 0.75 GB
// (x, f, e, z read, x, z, r written) and is bound by HBM: 0.72 GB of it pass there, 5.3 TB/s.  The
// products (0.20 GB, 0.22 with the halos, 3.1 TB/s) and the norm (0.20, 0.23, 3.5) reach neither that nor
// the rate of their instructions, which take 32 and 18 % of the time to issue: one workgroup per CU waits
// for its loads and at a barrier in every plane.
//
// Ghosts are neither read nor written: the neighbour beyond a periodic or mirror boundary is resolved
// to the node it copies.  (Dirichlet walls keep the kernels of mg_kernels.hip.)
#include "mg_kernels.h"

#include "grid_last.h"
#include "mg_march.h"
#include "xcd.h"

namespace sr {
namespace {

// a workgroup's tile and chunk and a thread's place in them
struct Place {
    int j0, j1, i0, i1, r, t, jp, sj, h0;
    bool inner, first, last;
};

__device__ inline Place place(const Lay &L, const MarchGeo &G, int rule_y) {
    Place P;
    const unsigned b = xcd_block();
    const int chunk = (int)(b / (unsigned)G.ntile), tile = (int)b - chunk * G.ntile;
    P.j0 = 1 + tile * G.tq + min(tile, G.tr);
    P.j1 = P.j0 + G.tq + (tile < G.tr);
    P.i0 = 1 + chunk * G.cq + min(chunk, G.cr);
    P.i1 = P.i0 + G.cq + (chunk < G.cr);
    const int r = (int)fdivu(threadIdx.x, (unsigned)G.tpr, G.inv_tpr);
    P.t = (int)threadIdx.x - r * G.tpr;
    // threads past the last row repeat it
    P.jp = min(P.j0 - 1 + r, P.j1);
    P.r = min(r, G.R - 1);
    P.inner = P.jp >= P.j0 && P.jp < P.j1;
    P.first = P.t == 0;
    P.last = P.t == G.tpr - 1;
    P.h0 = 2 * P.t;
    P.sj = P.jp >= 1 && P.jp <= L.ny ? P.jp : ghost_src(rule_y, P.jp, L.ny);
    return P;
}

// z coefficients of padded index 4t + q in entry q * tpr + t
template <typename T>
__device__ inline void load_z(const Lay &L, const MarchGeo &G, const T *cz, Co<T> *lz) {
    for (int q = (int)threadIdx.x; q < 4 * G.tpr; q += (int)blockDim.x) {
        const int qq = (int)fdivu((unsigned)q, (unsigned)G.tpr, G.inv_tpr);
        lz[q] = ldco(cz + 4 * min(4 * (q - qq * G.tpr) + qq, L.nz + 1));
    }
}

// L a at a thread's entries of one colour: c its own values; own, xm, xp the other colour in this row
// at the plane and at the planes before and after, ym and yp in the rows before and after; row the
// other colour's LDS row
template <typename T>
__device__ __forceinline__ Pair<T> lap2(const Place &P, int kh, bool zper, bool kb, const Pair<T> &c, const Pair<T> &own,
                                        const Pair<T> &xm, const Pair<T> &xp, const Pair<T> &ym, const Pair<T> &yp,
                                        const T *row, const Co<T> &X, const Co<T> &Y, const Co<T> &Z0, const Co<T> &Z1) {
    const T ext = row[kb ? (P.last ? P.h0 : P.h0 + 2) : (P.first ? 0 : P.h0 - 1)];
    T lo = own.a, hi = own.b;
    if (zper) {
        if (P.first) lo = row[kh - 2];
        if (P.last) hi = row[1];
    } else {
        lo = P.first ? own.b : lo;
        hi = P.last ? own.a : hi;
    }
    const T zm0 = kb ? lo : ext, zp0 = kb ? hi : own.a;
    const T zm1 = kb ? own.b : own.a, zp1 = kb ? ext : own.b;
    const T d0 = cen(X) + cen(Y) + cen(Z0), d1 = cen(X) + cen(Y) + cen(Z1);
    return Pair<T>{fma(-d0, c.a, six(X.p, xp.a, X.m, xm.a, Y.p, yp.a, Y.m, ym.a, Z0.p, zp0, Z0.m, zm0)),
                   fma(-d1, c.b, six(X.p, xp.b, X.m, xm.b, Y.p, yp.b, Y.m, ym.b, Z1.p, zp1, Z1.m, zm1))};
}

// sums of W quantities and one maximum over the workgroup (a multiple of 64 threads), in thread 0
template <int W>
__device__ inline void block_sums(double (&s)[W], double &m) {
    __shared__ double sh[16][W + 1];
    const int wv = threadIdx.x >> 6, nw = (int)blockDim.x >> 6;
#pragma unroll
    for (int i = 0; i < W; i++) s[i] = wave_sum(s[i]);
    m = wave_max(m);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
        for (int i = 0; i < W; i++) sh[wv][i] = s[i];
        sh[wv][W] = m;
    }
    __syncthreads();
    if (threadIdx.x == 0)
        for (int w = 1; w < nw; w++) {
#pragma unroll
            for (int i = 0; i < W; i++) s[i] += sh[w][i];
            m = fmax(m, sh[w][W]);
        }
}

// Partials of all workgroups, combined by the last of them (grid_last.h) in a fixed order: true there,
// in thread 0, with the totals.
template <int W>
__device__ inline bool grid_sums(double (&s)[W], double &m, double *part, unsigned *counter) {
    __shared__ bool last;
    block_sums<W>(s, m);
    unsigned long long *const pq = reinterpret_cast<unsigned long long *>(part);
    if (threadIdx.x == 0) {
        unsigned long long old[W + 1];
#pragma unroll
        for (int i = 0; i <= W; i++)
            old[i] = __hip_atomic_exchange(pq + (W + 1) * blockIdx.x + i,
                                           (unsigned long long)__double_as_longlong(i < W ? s[i < W ? i : 0] : m),
                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int i = 0; i <= W; i++) arrived(old[i]);
        last = grid_last(counter);
    }
    __syncthreads();
    if (!last) return false;
#pragma unroll
    for (int i = 0; i < W; i++) s[i] = 0.0;
    m = 0.0;
    for (int b = (int)threadIdx.x; b < (int)gridDim.x; b += (int)blockDim.x) {
        double v[W + 1];
#pragma unroll
        for (int i = 0; i <= W; i++)
            v[i] = __longlong_as_double((long long)__hip_atomic_load(pq + (W + 1) * b + i, __ATOMIC_RELAXED,
                                                                     __HIP_MEMORY_SCOPE_AGENT));
#pragma unroll
        for (int i = 0; i < W; i++) s[i] += v[i];
        m = fmax(m, v[W]);
    }
    block_sums<W>(s, m);
    return threadIdx.x == 0;
}

enum { OUT_READ = 0, OUT_ADD = 1, OUT_GCR = 2, OUT_NORM = 3, OUT_NORM0 = 4 };

template <int MODE>
__global__ void __launch_bounds__(1024) k_march_residual(Lay L, MarchGeo G, const double *__restrict__ x_in,
                                                         const float *__restrict__ e, const float *__restrict__ z,
                                                         const double *__restrict__ coef, const double *__restrict__ f,
                                                         double *__restrict__ x_out, float *__restrict__ z_next,
                                                         float *__restrict__ r32, const double *__restrict__ cx,
                                                         const double *__restrict__ cy, const double *__restrict__ cz,
                                                         Bc bc, double *__restrict__ part, unsigned *counter,
                                                         const double *__restrict__ ft, double *__restrict__ out,
                                                         double *host) {
    extern __shared__ unsigned char smem[];
    constexpr int NC = MODE == OUT_NORM0 ? 1 : 2;   // colours whose residual is formed
    constexpr bool KEEP = MODE == OUT_READ || MODE == OUT_ADD || MODE == OUT_GCR;   // and stored
    const Place P = place(L, G, bc.rule[1]);
    const int khs = L.khs, kh = L.kh, nx = L.nx;
    const bool zper = bc.rule[2] == G_PERIODIC;
    auto src = [&](int p) { return p >= 1 && p <= nx ? p : ghost_src(bc.rule[0], p, nx); };
    const long ps = 2L * (L.ny + 2) * khs;
    const unsigned vo0 = (unsigned)(P.sj * 2 * khs + P.h0) * 8u;
    const double alpha = MODE == OUT_GCR ? coef[0] : 0.0, beta = MODE == OUT_GCR ? coef[1] : 0.0;

    // LDS: u of a plane, two buffers; a row holds the half rows of colour 1 and (two colours) colour 0
    double *const lu_ = (double *)smem;
    const int bsz = G.R * NC * khs, lrow = P.r * NC * khs;
    Co<double> *const lz = (Co<double> *)(lu_ + 2 * bsz);
    load_z(L, G, cz, lz);
    const Co<double> Y = ldco(cy + 4 * P.sj);

    struct Raw {
        Pair<double> x[2];
        Pair<float> e[2], z[2];
    };
    auto load = [&](int p) {
        const int s = src(p);
        Raw w;
#pragma unroll
        for (int c = 0; c < 2; c++) {
            w.x[c] = ld2(x_in + s * ps + c * khs, here(vo0));
            if (MODE == OUT_ADD || MODE == OUT_GCR) w.e[c] = ld2(e + s * ps + c * khs, here(vo0) / 2);
            if (MODE == OUT_GCR) w.z[c] = ld2(z + s * ps + c * khs, here(vo0) / 2);
        }
        return w;
    };
    // the plane's u, stored (own: a plane and row of this workgroup) where the step makes a new one
    auto value = [&](const Raw &w, int p, bool own, Pair<double> (&u)[2]) {
#pragma unroll
        for (int c = 0; c < 2; c++) {
            if (MODE != OUT_ADD && MODE != OUT_GCR) {
                u[c] = w.x[c];
            } else if (MODE == OUT_ADD) {
                u[c] = Pair<double>{w.x[c].a + (double)w.e[c].a, w.x[c].b + (double)w.e[c].b};
            } else {
                const double da = (double)w.e[c].a - beta * (double)w.z[c].a;
                const double db = (double)w.e[c].b - beta * (double)w.z[c].b;
                u[c] = Pair<double>{w.x[c].a + alpha * da, w.x[c].b + alpha * db};
                if (own) st2(z_next + p * ps + c * khs, here(vo0) / 2, Pair<float>{(float)da, (float)db});
            }
            if ((MODE == OUT_ADD || MODE == OUT_GCR) && own) st2(x_out + p * ps + c * khs, here(vo0), u[c]);
        }
    };
    auto keep = [&](int buf, const Pair<double> (&u)[2]) {
#pragma unroll
        for (int c = 0; c < NC; c++) st2(lu_ + buf * bsz, (unsigned)(lrow + c * khs + P.h0) * 8u, u[c ^ 1]);
    };

    Pair<double> Um[2], Uc[2], Up[2], fc[2], fn[2];
    Raw w{};
    value(load(P.i0 - 1), 0, false, Um);
    value(load(P.i0), P.i0, P.inner, Uc);
    value(load(P.i0 + 1), P.i0 + 1, P.inner && P.i0 + 1 < P.i1, Up);
    keep(0, Uc);
#pragma unroll
    for (int c = 0; c < NC; c++) fc[c] = ld2(f + P.i0 * ps + c * khs, here(vo0));
    Co<double> X = ldco(cx + 4 * P.i0), Xn = X;
    double s[1] = {0.0}, mm = 0.0;
    __syncthreads();
    int buf = 0;
    for (int p = P.i0; p < P.i1; ++p, buf ^= 1) {
        const bool more = p + 1 < P.i1;
        // the next plane into LDS, and the loads of the one after it: they are waited for at the end of
        // the turn, behind them come the turn's stores (loads and stores retire in order)
        if (more) {
            keep(buf ^ 1, Up);
            w = load(p + 2);
#pragma unroll
            for (int c = 0; c < NC; c++) fn[c] = ld2(f + (p + 1) * ps + c * khs, here(vo0));
            Xn = ldco(cx + 4 * (p + 1));
        }
        const double *const lp = lu_ + buf * bsz;
        const int rm = P.r > 0 ? lrow - NC * khs : lrow, rp = P.r < G.R - 1 ? lrow + NC * khs : lrow;
        Pair<float> rs[2];
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const bool kb = (c + 1 + p + P.jp) & 1;
            const Co<double> Z0 = lz[(kb ? G.tpr : 0) + P.t], Z1 = lz[(kb ? 3 * G.tpr : 2 * G.tpr) + P.t];
            const Pair<double> ym = ld2(lp, (unsigned)(rm + c * khs + P.h0) * 8u);
            const Pair<double> yp = ld2(lp, (unsigned)(rp + c * khs + P.h0) * 8u);
            const Pair<double> lu = lap2<double>(P, kh, zper, kb, Uc[c], Uc[c ^ 1], Um[c ^ 1], Up[c ^ 1], ym, yp,
                                                 lp + lrow + c * khs, X, Y, Z0, Z1);
            double ra = fc[c].a - lu.a, rb = fc[c].b - lu.b;
            if (!P.inner || (P.first && !kb)) ra = 0.0;   // halo rows, and entries that hold no node
            if (!P.inner || P.last) rb = 0.0;
            rs[c] = Pair<float>{(float)ra, (float)rb};
            s[0] += ra * ra;
            s[0] += rb * rb;
            mm = fmax(mm, fmax(fabs(ra), fabs(rb)));
        }
        if (more) __syncthreads();
#pragma unroll
        for (int c = 0; c < 2; c++) {
            Um[c] = Uc[c];
            Uc[c] = Up[c];
            fc[c] = fn[c];
        }
        X = Xn;
        if (more) value(w, p + 2, P.inner && p + 2 < P.i1, Up);
        if (KEEP && P.inner) {
#pragma unroll
            for (int c = 0; c < NC; c++) st2(r32 + p * ps + c * khs, here(vo0) / 2, rs[c]);
        }
    }
    if (grid_sums<1>(s, mm, part, counter)) {
        // the four quantities of computeError, on the device and in the host's mirror
        const double q[4] = {s[0], ft[1], mm, ft[3]};
        for (int i = 0; i < 4; i++) out[i] = q[i];
        if (host) {
            for (int i = 0; i < 4; i++) host[i] = q[i];
            __threadfence_system();
        }
    }
}

// Q1R: e ends on a colour-1 half sweep for r32, so L e = r32 on colour 1 and is read there
template <bool Q1R>
__global__ void __launch_bounds__(1024) k_march_dots(Lay L, MarchGeo G, const float *__restrict__ e,
                                                     const float *__restrict__ z, const float *__restrict__ r32,
                                                     const float *__restrict__ cx, const float *__restrict__ cy,
                                                     const float *__restrict__ cz, Bc bc, double *__restrict__ part,
                                                     unsigned *counter, double *__restrict__ coef) {
    extern __shared__ unsigned char smem[];
    constexpr int NF = Q1R ? 3 : 4;   // half rows in LDS: z of colours 0 and 1, e of colour 1, e of colour 0
    const Place P = place(L, G, bc.rule[1]);
    const int khs = L.khs, kh = L.kh, nx = L.nx;
    const bool zper = bc.rule[2] == G_PERIODIC;
    auto src = [&](int p) { return p >= 1 && p <= nx ? p : ghost_src(bc.rule[0], p, nx); };
    const long ps = 2L * (L.ny + 2) * khs;
    const unsigned vo0 = (unsigned)(P.sj * 2 * khs + P.h0) * 4u, ob = (unsigned)khs * 4u;
    float *const lf = (float *)smem;
    const int bsz = G.R * NF * khs, lrow = P.r * NF * khs;
    Co<float> *const lz = (Co<float> *)(lf + 2 * bsz);
    load_z(L, G, cz, lz);
    const Co<float> Y = ldco(cy + 4 * P.sj);

    struct Val {
        Pair<float> z[2], e[2];
    };
    auto load = [&](int p) {
        const int s = src(p);
        Val v;
#pragma unroll
        for (int c = 0; c < 2; c++) {
            v.z[c] = ld2(z + s * ps + c * khs, here(vo0));
            v.e[c] = ld2(e + s * ps + c * khs, here(vo0));
        }
        return v;
    };
    auto keep = [&](int buf, const Val &v) {
        float *const b = lf + buf * bsz;
        const unsigned o = (unsigned)(lrow + P.h0) * 4u;
        st2(b, o, v.z[0]);
        st2(b, o + ob, v.z[1]);
        st2(b, o + 2 * ob, v.e[1]);
        if (!Q1R) st2(b, o + 3 * ob, v.e[0]);
    };
    Val m = load(P.i0 - 1), c_ = load(P.i0), n = load(P.i0 + 1);
    keep(0, c_);
    Pair<float> rn[2], rc[2];
#pragma unroll
    for (int c = 0; c < 2; c++) rn[c] = ld2(r32 + P.i0 * ps + c * khs, here(vo0));
    Co<float> Xn = ldco(cx + 4 * P.i0);
    double s[5] = {0.0, 0.0, 0.0, 0.0, 0.0}, unused = 0.0;
    __syncthreads();
    int buf = 0;
    for (int p = P.i0; p < P.i1; ++p, buf ^= 1) {
        const Val pl = n;
        const Co<float> X = Xn;
        rc[0] = rn[0];
        rc[1] = rn[1];
        if (p + 1 < P.i1) {
            keep(buf ^ 1, pl);
            n = load(p + 2);
#pragma unroll
            for (int c = 0; c < 2; c++) rn[c] = ld2(r32 + (p + 1) * ps + c * khs, here(vo0));
            Xn = ldco(cx + 4 * (p + 1));
        }
        const float *const lp = lf + buf * bsz;
        const int rm = P.r > 0 ? lrow - NF * khs : lrow, rp = P.r < G.R - 1 ? lrow + NF * khs : lrow;
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const bool kb = (c + 1 + p + P.jp) & 1;
            const Co<float> Z0 = lz[(kb ? G.tpr : 0) + P.t], Z1 = lz[(kb ? 3 * G.tpr : 2 * G.tpr) + P.t];
            const int oz = (c ^ 1) * khs, oe = (c == 0 ? 2 : 3) * khs;
            const Pair<float> lzv =
                lap2<float>(P, kh, zper, kb, c_.z[c], c_.z[c ^ 1], m.z[c ^ 1], pl.z[c ^ 1],
                            ld2(lp, (unsigned)(rm + oz + P.h0) * 4u), ld2(lp, (unsigned)(rp + oz + P.h0) * 4u),
                            lp + lrow + oz, X, Y, Z0, Z1);
            Pair<float> q = rc[c];
            if (!(Q1R && c == 1))
                q = lap2<float>(P, kh, zper, kb, c_.e[c], c_.e[c ^ 1], m.e[c ^ 1], pl.e[c ^ 1],
                                ld2(lp, (unsigned)(rm + oe + P.h0) * 4u), ld2(lp, (unsigned)(rp + oe + P.h0) * 4u),
                                lp + lrow + oe, X, Y, Z0, Z1);
            if (!P.inner) continue;
            auto add = [&](double r, double qv, double pv) {
                s[0] += r * qv;
                s[1] += qv * qv;
                s[2] += qv * pv;
                s[3] += r * pv;
                s[4] += pv * pv;
            };
            if (!(P.first && !kb)) add((double)rc[c].a, (double)q.a, (double)lzv.a);
            if (!P.last) add((double)rc[c].b, (double)q.b, (double)lzv.b);
        }
        if (p + 1 < P.i1) __syncthreads();
        m = c_;
        c_ = pl;
    }
    if (grid_sums<5>(s, unused, part, counter)) gcr_coef_from(s, coef);
}

template <typename K>
int allow_lds(K k) {
    return hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024) == hipSuccess ? 0 : 1;
}
unsigned threads64(const MarchPlan &P) { return (unsigned)(P.threads() + 63) & ~63u; }

}  // namespace

// Two planes per chunk at least: one costs the reads of three.  Measured (us per solve, at most 512 / 256 /
// 128 / 64 workgroups): 129 x 65 x 33 refinement, one or two planes at 512 or 256, 3534 / 3486 / 3541 /
// 3698; 65^3 GCR 1238 / 1236 / 1245 / 1305; 257 x 257 x 129 time step 2051 / 2075 / 2388 / 3086.
static MarchPlan outer_plan(const Lay &L) { return march_plan(L, 2); }

// the sizes and ghost rules these kernels take
bool march_outer_ok(const Lay &L, const Bc &bc) {
    for (int d = 0; d < 3; d++)
        if (bc.rule[d] != G_PERIODIC && bc.rule[d] != G_MIRROR) return false;
    return march_ok(L);
}
int march_parts(const Lay &L) { return march_ok(L) ? outer_plan(L).blocks() : 0; }
int march_outer_attr() {
    return allow_lds(k_march_residual<OUT_READ>) | allow_lds(k_march_residual<OUT_ADD>) |
           allow_lds(k_march_residual<OUT_GCR>) | allow_lds(k_march_residual<OUT_NORM0>) |
           allow_lds(k_march_residual<OUT_NORM>) |
           allow_lds(k_march_dots<true>) | allow_lds(k_march_dots<false>);
}

void launch_march_residual(const Lay &L, const double *x_in, const float *e, const float *z, const double *coef,
                           const double *f, double *x_out, float *z_next, float *r32, const double *cx,
                           const double *cy, const double *cz, const Bc &bc, bool color0, const MarchSums &S, hipStream_t s) {
    const MarchPlan P = outer_plan(L);
    const int nc = color0 ? 1 : 2;
    const size_t lds = 2 * (size_t)P.g.R * nc * L.khs * sizeof(double) + 4 * (size_t)P.g.tpr * sizeof(Co<double>);
    auto go = [&](auto k) {
        hipLaunchKernelGGL(k, dim3(P.blocks()), dim3(threads64(P)), lds, s, L, P.g, x_in, e, z, coef, f, x_out, z_next,
                           r32, cx, cy, cz, bc, S.part, S.counter, S.fterms, S.out, S.host);
    };
    if (color0) go(k_march_residual<OUT_NORM0>);
    else if (!r32) go(k_march_residual<OUT_NORM>);
    else if (z) go(k_march_residual<OUT_GCR>);
    else if (e) go(k_march_residual<OUT_ADD>);
    else go(k_march_residual<OUT_READ>);
}

void launch_march_dots(const Lay &L, const float *e, const float *z, const float *r32, const float *cx, const float *cy,
                       const float *cz, const Bc &bc, bool q1r, double *part, unsigned *counter, double *coef,
                       hipStream_t s) {
    const MarchPlan P = outer_plan(L);
    const size_t lds = 2 * (size_t)P.g.R * (q1r ? 3 : 4) * L.khs * sizeof(float) + 4 * (size_t)P.g.tpr * sizeof(Co<float>);
    auto go = [&](auto k) {
        hipLaunchKernelGGL(k, dim3(P.blocks()), dim3(threads64(P)), lds, s, L, P.g, e, z, r32, cx, cy, cz, bc, part,
                           counter, coef);
    };
    q1r ? go(k_march_dots<true>) : go(k_march_dots<false>);
}

}  // namespace sr
