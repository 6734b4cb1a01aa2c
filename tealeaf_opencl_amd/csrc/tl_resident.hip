// Iteration phases of the device-resident driver on the resident solver
// (tl_resident.h): the CG, Chebyshev, PPCG and Jacobi loops of
// tea_solve.f90:147-332, one cooperative launch per phase.
#include <hip/hip_runtime.h>

#include "../../include/tealeaf_mi355x.h"
#include "tl_chunk.h"
#include "tl_common.h"
#include "tl_device.h"
#include "tl_kernels.h"
#include "tl_resident.h"
#include "tl_state.h"

namespace tl {
namespace res {

// The scalar algebra of a mode on the block's copy of the solver state in LDS,
// run by one thread (block 0's also records the histories); the other threads
// see the result after the next barrier.
__device__ __forceinline__ void tail(const RedArgs &ra, int mode, double tot, SolveState *st)
{
    RedArgs a = ra;
    a.mode = mode;
    if (blockIdx.x != 0) a.hist_a = a.hist_b = a.hist_e = nullptr;
    double t[MAX_RED] = {tot};
    finish_state(a, t, st);
}

// One CG iteration measured (the slope between two caps), none / diagonal / block,
// against two kernels and two finishers per iteration from a graph:
//   512^2    5.7 /  5.4 /  5.7 us   (17.8 to 18.2 us)
//   960^2    7.5 /  7.5 /  7.8 us   (27 to 29 us)
//   1024^2   7.9 /  7.8 /  8.1 us   (29 to 31 us)
// What bounds it is the two exchanges, at least 1.3 us each from a store to
// the load that sees it on another XCD; at 512^2 the vector units are busy 14 % of
// the time.
// CG iterations until the state halts or `iters` are done
// (tea_leaf_cg_cl.cl:45-160). An iteration's scalar algebra, beyond alpha and
// beta, is run by one thread while the others wait for the next iteration's
// p.w; a halt is acted on behind that sum, when the next iteration has formed
// its p but changed nothing.
template <int PREC, int NW, int S>
__global__ void __launch_bounds__(NW * 64) k_res_cg(Geom g, Ext e, Comm cm, double *u, double *r, double *z,
                                                    double *pA, double *pB, const double *W, Faces fc, RedArgs ra,
                                                    int iters)
{
    constexpr int R = S * STRIP;
    __shared__ Shared<NW, S, 1> sh;
    __shared__ SolveState st;
    constexpr bool LDS = S > 1 && PREC == PREC_BLOCK;
    __shared__ HeldMem<LDS, R, NW> um;
    Ctx<NW, S, 1> x(cm, sh);
    if (threadIdx.x == 0) {
        st = *ra.st;
        sh.fault = 0;
    }
    __syncthreads();
    const unsigned int closed = x.begin();
    if (st.halt) return;
    const Cells c = thread_cells(x, g, e);
    const int P = g.pitch;
    CellFaces<NW, S, 1> f;
    f.template from_cond<false>(x, g, fc, W, c);
    CellPrec<PREC, false, NW, S, 1> M;
    M.init(g, c, f);
    // p_{n-1} as the streaming kernels leave it
    const double *src = PREC == PREC_NONE ? r : z, *p_old = (st.n & 1) ? pA : pB;
    Held<LDS, R, NW> uv(um);
    double rv[R], zv[R], pv[R], za, zb, pa, pb, w[R], pn[R], acc[1][S], tot[1], *ph = x.side(0);
    load_cells(c, P, u, w);
    uv.put(w);
    load_cells(c, P, p_old, pv);
    load_cells(c, P, r, rv);
    load_cells(c, P, src, zv);
    double beta = uniform(st.beta), rro = uniform(st.rro), pw = 0.0;
    load_border(x.lane, c, e, P, p_old, pa, pb, w);
    load_border(x.lane, c, e, P, src, za, zb, pn);
    pa = fma(beta, pa, za);
    pb = fma(beta, pb, zb);
    if (x.ends())
#pragma unroll
        for (int q = 0; q < R; ++q) ph[q] = fma(beta, w[q], pn[q]);
    if (!x.begun(closed)) return;
    for (int it = 0;; ++it) {
#pragma unroll
        for (int q = 0; q < R; ++q) pn[q] = fma(beta, pv[q], zv[q]);
        cells_op(f, pn, pa, pb, ph, w);
        strip_dots<S>(pn, w, acc[0]);
        x.sum_begin(acc);
        if (it > 0 && threadIdx.x == TAIL_THREAD) {
            tail(ra, RED_CG_PW, pw, &st);
            tail(ra, RED_CG_RRN, rro, &st);
        }
        x.sum_end(tot);
        if (st.halt || sh.fault || it == iters) break;
        pw = uniform(tot[0]);
        const double alpha = uniform(rro / pw);
#pragma unroll
        for (int q = 0; q < R; ++q) {
            pv[q] = pn[q];
            uv(q) = fma(alpha, pn[q], uv(q));
            rv[q] = fma(-alpha, w[q], rv[q]);
        }
        M.apply(f, rv, zv);
        x.send(zv);
        strip_dots<S>(rv, zv, acc[0]);
        x.sum_begin(acc);
        x.template sum_end<true>(tot, za, zb);
        beta = uniform(tot[0] / rro);
        rro = uniform(tot[0]);
        // the border of the next p: this one's and z's
        pa = fma(beta, pa, za);
        pb = fma(beta, pb, zb);
        if (x.ends())
#pragma unroll
            for (int q = 0; q < R; ++q) ph[q] = fma(beta, ph[q], x.in()[q]);
    }
    if (sh.fault) return;
    uv.get(w);
    store_cells(c, P, u, w);
    store_cells(c, P, r, rv);
    if (PREC != PREC_NONE) store_cells(c, P, z, zv);
    // the last iteration's p where the streaming kernels write it
    store_cells(c, P, (st.cg_calc_steps & 1) ? pB : pA, pv);
    if (blockIdx.x == 0 && threadIdx.x == 0) *ra.st = st;
}

// The same on tall blocks. Per iteration, none / diagonal / block: 1100x1000 16.6 /
// 17.1 / 18.2 us, 2001x1503 24.0 / 24.9 / 27.5 us, 2048^2 29.9 / 36.4 / 38.0 us
// (launched: 32 / 34 / 35, 57 / 61 / 62 and 79 / 84 / 84 us, bound by the memory
// traffic that this form does not have). At 2001x1503 and 2048^2, block, the vector
// units are busy half of the time, 58 % of their instructions in FP64 (two faces of
// 11 instructions per cell in each of the two passes); the rest are the two exchanges
// (about 5 us), latencies that two wavefronts per SIMD leave open and, at 2048^2,
// r's traffic, which no longer fits the registers.
template <int PREC, int NW, int S>
__global__ void __launch_bounds__(NW * 64) k_tall_cg(Geom g, Ext e, Comm cm, double *u, double *r, double *z,
                                                     double *pA, double *pB, const double *W, Faces fc, RedArgs ra,
                                                     int iters)
{
    tall_cg<double, PREC, false, 1, NW, S, CondStream<double, false, NW, S>>(
        g, e, cm, u, r, z, pA, pB, W, (const double *)nullptr, fc, ra.st, iters,
        [&](double pw, const double *tot, SolveState *st) {
            tail(ra, RED_CG_PW, pw, st);
            tail(ra, RED_CG_RRN, tot[0], st);
        },
        [](const SolveState &st) { return (st.n & 1) != 0; },
        [](const SolveState &st) { return (st.cg_calc_steps & 1) != 0; });
}

// Jacobi sweeps (tea_leaf_jacobi_cl.cl:15-42) until the state halts or
// `iters` are done. One exchange per sweep: 200x148 2.1 us, 512^2 2.8 us,
// 1024^2 4.5 us (a sweep and its finisher launched: 9.6, 8.0 and 12.4 us). A
// sweep's scalar algebra runs, and its halt is acted on, during the next
// sweep's exchange.
template <int NW, int S>
__global__ void __launch_bounds__(NW * 64) k_res_jacobi(Geom g, Ext e, Comm cm, const double *u0, double *u,
                                                        const double *W, Faces fc, RedArgs ra, int iters)
{
    constexpr int R = S * STRIP;
    __shared__ Shared<NW, S, 1> sh;
    __shared__ SolveState st;
    Ctx<NW, S, 1> x(cm, sh);
    if (threadIdx.x == 0) {
        st = *ra.st;
        sh.fault = 0;
    }
    __syncthreads();
    const unsigned int closed = x.begin();
    if (st.halt) return;
    const Cells c = thread_cells(x, g, e);
    const int P = g.pitch;
    CellFaces<NW, S, 1> f;
    f.template from_cond<false>(x, g, fc, W, c);
    double b[R], uv[R], un[R], ua, ub, acc[1][S], tot[1];
    load_cells(c, P, u0, b);
    load_cells(c, P, u, uv);
    load_border(x.lane, c, e, P, u, ua, ub, un);
    if (x.ends())
#pragma unroll
        for (int q = 0; q < R; ++q) x.in()[q] = un[q];
    if (!x.begun(closed)) return;
    for (int it = 0;; ++it) {
#pragma unroll
        for (int q = 0; q < R; ++q) {
            const double w = dpp_shr1(uv[q], x.in()[q]), ee = dpp_shl1(uv[q], x.in()[q]);
            const double kx1 = f.east(q), a = q ? uv[q - 1] : ua, d = q < R - 1 ? uv[q + 1] : ub;
            un[q] = fma(f.ky[q], a, fma(f.ky[q + 1], d, fma(f.kx[q], w, fma(kx1, ee, b[q])))) /
                    (1.0 + (f.kx[q] + kx1) + (f.ky[q] + f.ky[q + 1]));
        }
        x.send(un);
#pragma unroll
        for (int s = 0; s < S; ++s) {
            acc[0][s] = 0.0;
#pragma unroll
            for (int q = s * STRIP; q < (s + 1) * STRIP; ++q)
                if (q < c.rows) acc[0][s] += fabs(un[q] - uv[q]);
        }
        x.sum_begin(acc);
        if (it > 0 && threadIdx.x == TAIL_THREAD) tail(ra, RED_JACOBI, tot[0], &st);
        x.template sum_end<true>(tot, ua, ub);
        if (st.halt || sh.fault || it == iters) break;
#pragma unroll
        for (int q = 0; q < R; ++q) uv[q] = un[q];
    }
    if (sh.fault) return;
    store_cells(c, P, u, uv);
    if (blockIdx.x == 0 && threadIdx.x == 0) *ra.st = st;
}

// Chebyshev iterations (tea_leaf_cheby_cl.cl:66-145) until the state halts or
// `iters` are done. Nothing is summed but every tenth residual norm
// (tea_solve.f90:223), and the launch's first; the state's algebra runs during the exchange of u. Per
// iteration without a norm, block Jacobi: 512^2 1.6 us, 1024^2 2.3 us (launched in
// pairs: 11.4 and 14.3 us).
template <int PREC, int NW, int S>
__global__ void __launch_bounds__(NW * 64) k_res_cheby(Geom g, Ext e, Comm cm, const double *u0, double *u, double *p,
                                                       const double *W, Faces fc, const double *ch_a,
                                                       const double *ch_b, RedArgs ra, int iters)
{
    constexpr int R = S * STRIP;
    __shared__ Shared<NW, S, 1> sh;
    __shared__ SolveState st;
    Ctx<NW, S, 1> x(cm, sh);
    if (threadIdx.x == 0) {
        st = *ra.st;
        sh.fault = 0;
    }
    __syncthreads();
    const unsigned int closed = x.begin();
    if (st.halt) return;
    const Cells c = thread_cells(x, g, e);
    const int P = g.pitch;
    CellFaces<NW, S, 1> f;
    f.template from_cond<false>(x, g, fc, W, c);
    CellPrec<PREC, false, NW, S, 1> M;
    M.init(g, c, f);
    double b[R], uv[R], pv[R], rv[R], zv[R], ua, ub, acc[1][S], tot[1] = {0.0};
    load_cells(c, P, u0, b);
    load_cells(c, P, u, uv);
    load_cells(c, P, p, pv);
    load_border(x.lane, c, e, P, u, ua, ub, rv);
    if (x.ends())
#pragma unroll
        for (int q = 0; q < R; ++q) x.in()[q] = rv[q];
    int n = st.n, step = st.cheby_calc_steps - 1;
    const int est_itc = st.est_itc;
    if (!x.begun(closed)) return;
    for (int it = 0; it < iters; ++it, ++n, ++step) {
        const double ca = ch_a[step], cb = ch_b[step];
        // (the first iteration's sum: see tl_resident.h, Beginning)
        const bool want = it == 0 || (n >= est_itc && n % 10 == 0);
        cells_op(f, uv, ua, ub, x.in(), rv);
#pragma unroll
        for (int q = 0; q < R; ++q) rv[q] = b[q] - rv[q];
        if (PREC == PREC_BLOCK) M.apply(f, rv, zv);
#pragma unroll
        for (int q = 0; q < R; ++q) {
            const double z = PREC == PREC_BLOCK ? cb * zv[q] : PREC == PREC_DIAG ? cb * M.mi[q] * rv[q] : cb * rv[q];
            pv[q] = fma(ca, pv[q], z);
            uv[q] = uv[q] + pv[q];
        }
        if (want) {
            strip_dots<S>(rv, rv, acc[0]);
            x.sum_begin(acc);
            x.sum_end(tot);
        }
        x.send(uv);
        x.recv(ua, ub, [&]() {
            if (threadIdx.x == TAIL_THREAD) tail(ra, RED_CHEBY, tot[0], &st);
        });
        if (st.halt || sh.fault) break;
    }
    if (sh.fault) return;
    store_cells(c, P, u, uv);
    store_cells(c, P, p, pv);
    if (blockIdx.x == 0 && threadIdx.x == 0) *ra.st = st;
}

// PPCG outer steps (tea_solve.f90:231-267 with tea_leaf_ppcg_cl.cl:4-155) of
// `inner` smoothing steps each, until the state halts or `iters` are done. An
// outer step exchanges z (whose border also gives that of sd = z / theta), sd
// before every smoothing step but the first, and sums p.w and r.z. fresh: r.z
// and p with the z of the last smoothing step (the fresh-z option). Per outer
// step of ten smoothing steps, none / diagonal / block: 512^2 22 / 23 / 23 us,
// 1024^2 31 / 34 / 35 us (launched: 57 / 60 / 60 and 120 / 123 / 135 us).
template <int PREC, int NW, int S>
__global__ void __launch_bounds__(NW * 64) k_res_ppcg(Geom g, Ext e, Comm cm, double *u, double *r, double *z,
                                                      double *pA, double *pB, const double *W, Faces fc,
                                                      const double *ch_a, const double *ch_b, int inner, int fresh,
                                                      RedArgs ra, int iters)
{
    constexpr int R = S * STRIP;
    __shared__ Shared<NW, S, 3> sh;
    __shared__ SolveState st;
    constexpr bool LDS = S > 1 && PREC != PREC_NONE;
    __shared__ HeldMem<LDS, R, NW> um, zm, pm;
    Ctx<NW, S, 3> x(cm, sh);
    if (threadIdx.x == 0) {
        st = *ra.st;
        sh.fault = 0;
    }
    __syncthreads();
    const unsigned int closed = x.begin();
    if (st.halt) return;
    const Cells c = thread_cells(x, g, e);
    const int P = g.pitch, n0 = st.n;
    CellFaces<NW, S, 3> f;
    f.template from_cond<false>(x, g, fc, W, c);
    CellPrec<PREC, false, NW, S, 3> M;
    M.init(g, c, f);
    const double *src = PREC == PREC_NONE ? r : z, *p_old = (n0 & 1) ? pA : pB;
    Held<LDS, R, NW> uv(um), zv(zm), pv(pm);
    double rv[R], sd[R], w[R], za, zb, pa, pb, sa, sb, acc[1][S], tot[1];
    double *ph = x.side(0), *zh = x.side(1), *sh0 = x.side(2);
    load_cells(c, P, u, w);
    uv.put(w);
    load_cells(c, P, src, w);
    zv.put(w);
    load_cells(c, P, p_old, w);
    pv.put(w);
    load_cells(c, P, r, rv);
    double beta = uniform(st.beta), rro = uniform(st.rro), pw = 0.0;
    const double theta = uniform(st.theta);
    load_border(x.lane, c, e, P, p_old, pa, pb, w);
    load_border(x.lane, c, e, P, src, za, zb, sd);
    pa = fma(beta, pa, za);
    pb = fma(beta, pb, zb);
    if (x.ends())
#pragma unroll
        for (int q = 0; q < R; ++q) ph[q] = fma(beta, w[q], sd[q]);
    if (!x.begun(closed)) return;
    int it = 0;
    for (;; ++it) {
        // p: sd is free until the smoothing
#pragma unroll
        for (int q = 0; q < R; ++q) sd[q] = fma(beta, pv(q), zv(q));
        cells_op(f, sd, pa, pb, ph, w);
        strip_dots<S>(sd, w, acc[0]);
        x.sum_begin(acc);
        if (it > 0 && threadIdx.x == TAIL_THREAD) {
            tail(ra, RED_PPCG_PW, pw, &st);
            tail(ra, RED_PPCG_RRN, rro, &st);
        }
        x.sum_end(tot);
        if (st.halt || sh.fault || it == iters) break;
        pw = uniform(tot[0]);
        const double alpha = uniform(rro / pw);
        pv.put(sd);
#pragma unroll
        for (int q = 0; q < R; ++q) {
            uv(q) = fma(alpha, sd[q], uv(q));
            rv[q] = fma(-alpha, w[q], rv[q]);
        }
        M.apply(f, rv, w);
        zv.put(w);
        x.swap(w, za, zb);
#pragma unroll
        for (int q = 0; q < R; ++q) sd[q] = w[q] / theta;
        sa = za / theta;
        sb = zb / theta;
        if (x.ends())
#pragma unroll
            for (int q = 0; q < R; ++q) {
                zh[q] = x.in()[q];
                sh0[q] = x.in()[q] / theta;
            }
        for (int k = 0; k < inner; ++k) {
            const double ca = ch_a[k], cb = ch_b[k];
            if (k) x.swap(sd, sa, sb);
            cells_op(f, sd, sa, sb, k ? x.in() : sh0, w);
#pragma unroll
            for (int q = 0; q < R; ++q) {
                uv(q) = uv(q) + sd[q];
                rv[q] -= w[q];
            }
            M.apply(f, rv, w);
#pragma unroll
            for (int q = 0; q < R; ++q)
                sd[q] = fma(ca, sd[q], PREC == PREC_DIAG ? cb * rv[q] * M.mi[q] : cb * w[q]);
        }
        // w holds M^-1 r of the last smoothing step
        if (PREC == PREC_NONE || fresh) {
            zv.put(w);
            x.send(w);
        } else {
            zv.get(w);
        }
        strip_dots<S>(rv, w, acc[0]);
        x.sum_begin(acc);
        if (PREC == PREC_NONE || fresh) {
            x.template sum_end<true>(tot, za, zb);
            zh = x.in();
        } else {
            x.sum_end(tot);
        }
        beta = uniform(tot[0] / rro);
        rro = uniform(tot[0]);
        pa = fma(beta, pa, za);
        pb = fma(beta, pb, zb);
        if (x.ends())
#pragma unroll
            for (int q = 0; q < R; ++q) ph[q] = fma(beta, ph[q], zh[q]);
        zh = x.side(1);
    }
    if (sh.fault) return;
    uv.get(w);
    store_cells(c, P, u, w);
    store_cells(c, P, r, rv);
    zv.get(w);
    if (PREC != PREC_NONE) store_cells(c, P, z, w);
    pv.get(w);
    // the last iteration's p where the streaming kernels write it
    store_cells(c, P, ((n0 + it - 1) & 1) ? pB : pA, w);
    if (blockIdx.x == 0 && threadIdx.x == 0) *ra.st = st;
}

// Chebyshev iterations on tall blocks: u and p in registers, u0 in LDS, faces
// and preconditioner factors formed anew in the iteration's one pass. A strip's
// new u takes the place of the old one at once: the strip below only needs its
// last row, kept in `up`. Per iteration without a norm, none / diagonal / block:
// 1100x1000 6.1 / 6.5 / 7.4 us, 2001x1503 8.4 / 9.4 / 10.5 us, 2048^2 11.0 / 11.9 / 13.7
// us (launched in pairs: 15, 22 and 30 us). At 2001x1503, block, the vector units are
// busy two thirds of the time.
template <int PREC, int NW, int S>
__global__ void __launch_bounds__(NW * 64) k_tall_cheby(Geom g, Ext e, Comm cm, const double *u0, double *u, double *p,
                                                        const double *W, Faces fc, const double *ch_a,
                                                        const double *ch_b, RedArgs ra, int iters)
{
    constexpr int R = S * STRIP;
    __shared__ Shared<NW, S, 1> sh;
    __shared__ SolveState st;
    __shared__ double bl[R][NW * 64];
    __shared__ double cwl[NW * R];
    Ctx<NW, S, 1> x(cm, sh);
    const int t = threadIdx.x;
    if (t == 0) {
        st = *ra.st;
        sh.fault = 0;
    }
    __syncthreads();
    const unsigned int closed = x.begin();
    if (st.halt) return;
    const Tall<NW, S> c(x, g, e);
    const CondStream<double, false, NW, S> F(x, c, g, e, fc, W, nullptr, cwl + x.wv * R);
    double uv[R], pv[R], ua, ub, tot[1] = {0.0};
    if (x.lane < S) sh.part[0][x.wv * S + x.lane] = 0.0;
    if (x.lane < R) sh.col[0][x.wv * R + x.lane] = sh.col[1][x.wv * R + x.lane] = 0.0;
    auto take = [](double *to) {
        return [to](int o, const double *v) {
#pragma unroll
            for (int q = 0; q < STRIP; ++q) to[o + q] = v[q];
        };
    };
    auto give = [](const double *from) {
        return [from](int o, double *v) {
#pragma unroll
            for (int q = 0; q < STRIP; ++q) v[q] = from[o + q];
        };
    };
    tall_load(c, u0, [&](int o, const double *v) {
#pragma unroll
        for (int q = 0; q < STRIP; ++q) bl[o + q][t] = v[q];
    });
    tall_load(c, (const double *)u, take(uv));
    tall_load(c, (const double *)p, take(pv));
    tall_border(x, c, g, e, ua, ub, sh.in, [&](int i) { return u[i]; });
    int n = st.n, step = st.cheby_calc_steps - 1;
    const int est_itc = st.est_itc;
    if (!x.begun(closed)) return;
    for (int it = 0; it < iters; ++it, ++n, ++step) {
        const double ca = ch_a[step], cb = ch_b[step];
        // (the first iteration's sum: see tl_resident.h, Beginning)
        const bool want = it == 0 || (n >= est_itc && n % 10 == 0);
        double up = ua;
        F.pass(c, [&](const Tall<NW, S> &d, int s, const double *kx0, const double *kx1, const double *ky) {
            const int o = s * STRIP;
            double rs[STRIP], zs[STRIP];
            tall_op<R>(s, uv, up, ub, x.in(), kx0, kx1, ky, rs);
            up = uv[o + STRIP - 1];
#pragma unroll
            for (int q = 0; q < STRIP; ++q) rs[q] = bl[o + q][t] - rs[q];
            if (want) {
                double acc = 0.0;
#pragma unroll
                for (int q = 0; q < STRIP; ++q) acc = fma(rs[q], rs[q], acc);
                x.strip_sum(0, s, acc);
            }
            if (PREC == PREC_BLOCK) strip_precondition<PREC>(g, d.ks + o, 0, kx0, kx1, ky, rs, zs);
#pragma unroll
            for (int q = 0; q < STRIP; ++q) {
                const double z = PREC == PREC_BLOCK  ? cb * zs[q]
                                 : PREC == PREC_DIAG ? cb * div_nr(1.0, diag_of(kx0[q], kx1[q], ky[q], ky[q + 1])) * rs[q]
                                                     : cb * rs[q];
                pv[o + q] = fma(ca, pv[o + q], z);
                uv[o + q] = uv[o + q] + pv[o + q];
            }
            if (x.ends())
#pragma unroll
                for (int q = 0; q < STRIP; ++q) sh.col[x.lane & 1][x.wv * R + o + q] = uv[o + q];
        });
        if (want) {
            x.sum_begin();
            x.sum_end(tot);
        }
        x.send(uv[0], uv[R - 1]);
        x.recv(ua, ub, [&]() {
            if (t == TAIL_THREAD) tail(ra, RED_CHEBY, tot[0], &st);
        });
        if (st.halt || sh.fault) break;
    }
    if (sh.fault) return;
    tall_store(c, u, give(uv));
    tall_store(c, p, give(pv));
    if (blockIdx.x == 0 && t == 0) *ra.st = st;
}

// The outer steps of k_res_ppcg on tall blocks. Per outer step of ten smoothing
// steps, none / diagonal / block: 1100x1000 80 / 90 / 99 us, 2001x1503 118 / 131 /
// 171 us, 2048^2 212 / 226 / 249 us (launched: 136 / 139 / 142, 286 / 295 / 298 and
// 393 / 401 / 403 us).
template <int PREC, int NW, int S>
__global__ void __launch_bounds__(NW * 64) k_tall_ppcg(Geom g, Ext e, Comm cm, double *u, double *r, double *z,
                                                       double *pA, double *pB, const double *W, Faces fc,
                                                       const double *ch_a, const double *ch_b, int inner, int fresh,
                                                       RedArgs ra, int iters)
{
    tall_ppcg<double, PREC, false, 1, NW, S, CondStream<double, false, NW, S>>(
        g, e, cm, u, r, z, pA, pB, W, (const double *)nullptr, fc, ch_a, ch_b, inner, fresh != 0, ra.st, iters,
        [&](double pw, const double *tot, SolveState *st) {
            tail(ra, RED_PPCG_PW, pw, st);
            tail(ra, RED_PPCG_RRN, tot[0], st);
        });
}

Comm next_comm(tl_chunk *c, unsigned int reds, unsigned int halos)
{
    const Ext e = ext_interior(c);
    Comm cm;
    cm.mem = c->res_mem;
    cm.fault = c->res_fault;
    cm.left = c->res_fault + 1;
    cm.closed = c->res_closed;
    // for tests (TL_TUNE_RESIDENT): a short wait, a launch closed before it begins
    if (c->resident < 0) *c->h_res_fault = FAULT_IMPATIENT;
    if (c->resident > 1 && ++c->res_launches >= c->resident - 1)
        (void)hipMemsetD32Async((hipDeviceptr_t)c->res_closed, (int)c->res_rseq, 1, c->s);
    cm.rseq = c->res_rseq;
    cm.hseq = c->res_hseq;
    c->res_rseq += reds + 2;
    c->res_hseq += halos + 2;
    cm.nbx = e.ntx;
    cm.nby = (e.nty + c->res_rows - 1) / c->res_rows;
    cm.nty = e.nty;
    return cm;
}

std::mutex &launch_mutex(const tl_chunk *c)
{
    static std::mutex mu[64];
    return mu[c->device & 63];
}

}  // namespace res

using namespace res;

// The fewest tile rows per block with which a block per compute unit covers
// the grid: more, smaller blocks have less to do between exchanges (one CG
// iteration, no preconditioner: 256^2 with 1, 2 and 4 tile rows per block 3.75, 3.9
// and 4.8 us; at 512^2, 5.6, 5.3 and 5.3 us, larger blocks' fewer words to poll are
// worth as much). The order of the sums by
// quads, or on tall blocks by piles of as many quads as a block owns, is a
// condition of the kernels.
int resident_rows(const Ext &e, int cus)
{
    if (!e.quad) return 0;
    for (int tr : {1, 2, 4})
        if (e.quad == 1 && e.ntx * ((e.nty + tr - 1) / tr) <= cus) return tr;
    const int tr = 4 * e.quad;
    return e.quad > 1 && e.ntx * ((e.nty + tr - 1) / tr) <= cus ? tr : 0;
}

size_t resident_bytes(const Ext &e, int rows)
{
    return sizeof(u64) * (RED_WORDS + (size_t)halo_words(rows * TILE_Y) * e.ntx * ((e.nty + rows - 1) / rows));
}

bool resident_eligible(const tl_chunk *c)
{
    return c->res_rows && c->faces.zl && c->faces.zr && c->faces.zb && c->faces.zt;
}

int resident_status(tl_chunk *c, hipError_t e, bool *left)
{
    volatile unsigned int *flag = c->h_res_fault;
    if (e != hipSuccess) (void)hipGetLastError();
    *left = e != hipSuccess || flag[1];
    const bool stuck = !*left && flag[0] == FAULT_STUCK;
    flag[0] = flag[1] = 0u;
    if (stuck) {
        set_error("resident solver: a block waited too long for another");
        return TL_ERR_SOLVER;
    }
    if (*left) c->res_left = true;
    return TL_OK;
}

#define TL_NO_TALL(P, NW, S) hipErrorNotSupported
hipError_t launch_res_cg(tl_chunk *c, int iters)
{
    const Ext e = ext_interior(c);
    const Comm cm = next_comm(c, 2u * iters + 2, iters);
    const RedArgs ra = red_args(c, RED_CG_RRN, true);
    double **f = c->f2;
#define TL_K(P, NW, S)                                                                                          \
    coop(c, k_res_cg<P, NW, S>, cm, NW, c->g, e, cm, f[F_U], f[F_R], f[F_Z], f[F_P], f[F_P2],                   \
         (const double *)f[F_COND], c->faces, ra, iters)
#define TL_L(P, NW, S)                                                                                          \
    coop(c, k_tall_cg<P, NW, S>, cm, NW, c->g, e, cm, f[F_U], f[F_R], f[F_Z], f[F_P], f[F_P2],                  \
         (const double *)f[F_COND], c->faces, ra, iters)
    return TL_RES_ANY(TL_K, TL_L);
#undef TL_K
#undef TL_L
}

hipError_t launch_res_cheby(tl_chunk *c, int iters)
{
    const Ext e = ext_interior(c);
    const Comm cm = next_comm(c, iters, iters);
    const RedArgs ra = red_args(c, RED_CHEBY, true);
    double **f = c->f2;
#define TL_K(P, NW, S)                                                                                            \
    coop(c, k_res_cheby<P, NW, S>, cm, NW, c->g, e, cm, (const double *)f[F_U0], f[F_U], f[F_P],                  \
         (const double *)f[F_COND], c->faces, (const double *)c->ch_a, (const double *)c->ch_b, ra, iters)
#define TL_L(P, NW, S)                                                                                            \
    coop(c, k_tall_cheby<P, NW, S>, cm, NW, c->g, e, cm, (const double *)f[F_U0], f[F_U], f[F_P],                 \
         (const double *)f[F_COND], c->faces, (const double *)c->ch_a, (const double *)c->ch_b, ra, iters)
    return TL_RES_ANY(TL_K, TL_L);
#undef TL_K
#undef TL_L
}

hipError_t launch_res_ppcg(tl_chunk *c, int inner, int iters)
{
    const Ext e = ext_interior(c);
    const Comm cm = next_comm(c, 2u * iters + 2, (unsigned)(inner + 1) * iters);
    const RedArgs ra = red_args(c, RED_PPCG_RRN, true);
    double **f = c->f2;
    const int fresh = c->ppcg_fresh_z;
#define TL_K(P, NW, S)                                                                                            \
    coop(c, k_res_ppcg<P, NW, S>, cm, NW, c->g, e, cm, f[F_U], f[F_R], f[F_Z], f[F_P], f[F_P2],                   \
         (const double *)f[F_COND], c->faces, (const double *)c->ch_a, (const double *)c->ch_b, inner, fresh, ra, \
         iters)
#define TL_L(P, NW, S)                                                                                            \
    coop(c, k_tall_ppcg<P, NW, S>, cm, NW, c->g, e, cm, f[F_U], f[F_R], f[F_Z], f[F_P], f[F_P2],                  \
         (const double *)f[F_COND], c->faces, (const double *)c->ch_a, (const double *)c->ch_b, inner, fresh, ra, \
         iters)
    return TL_RES_ANY(TL_K, TL_L);
#undef TL_K
#undef TL_L
}

hipError_t launch_res_jacobi(tl_chunk *c, int iters)
{
    const Ext e = ext_interior(c);
    const Comm cm = next_comm(c, iters + 1, iters + 1);
    const RedArgs ra = red_args(c, RED_JACOBI, true);
    double **f = c->f2;
#define TL_K(P, NW, S)                                                                                            \
    coop(c, k_res_jacobi<NW, S>, cm, NW, c->g, e, cm, (const double *)f[F_U0], f[F_U], (const double *)f[F_COND], \
         c->faces, ra, iters)
    return TL_RES_ROWS(TL_K, TL_NO_TALL, PREC_NONE);
#undef TL_K
}

}  // namespace tl
