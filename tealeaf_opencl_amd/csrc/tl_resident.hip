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

// the thread that runs the scalar algebra: not of the wavefront that publishes
// the block's sums
constexpr int TAIL_THREAD = 64;

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

// One CG iteration measured, none / diagonal / block, against two kernels and
// two finishers per iteration from a graph (before the resident solver, and
// with this library's small-grid kernels):
//   512^2    5.5 /  5.6 /  5.8 us   (25 and 19 us)
//   960^2    8.5 /  8.3 /  8.8 us   (31 and 28 us)
//   1024^2   8.4 /  8.3 /  8.7 us   (33 and 30 us)
// What bounds it is the two exchanges, at least 1.3 us each from a store to
// the load that sees it on another XCD; its arithmetic takes 1 to 3 us.
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
    __shared__ Shared<NW, S> sh;
    __shared__ SolveState st;
    Ctx<NW, S> x(cm, sh);
    if (threadIdx.x == 0) {
        st = *ra.st;
        sh.fault = 0;
    }
    __syncthreads();
    if (st.halt) return;
    const Cells c = thread_cells(x, g, e);
    const int P = g.pitch;
    CellFaces<NW, S> f;
    f.template from_cond<false>(x, g, fc, W, c);
    CellPrec<PREC, false, NW, S> M;
    M.init(g, c, f);
    // p_{n-1} as the streaming kernels leave it
    const double *src = PREC == PREC_NONE ? r : z, *p_old = (st.n & 1) ? pA : pB;
    double uv[R], rv[R], zv[R], pv[R], za, zb, pa, pb, w[R], pn[R], acc[1][S], tot[1], *ph = x.side();
    load_cells(c, P, u, uv);
    load_cells(c, P, r, rv);
    load_cells(c, P, src, zv);
    load_cells(c, P, p_old, pv);
    double beta = st.beta, rro = st.rro, pw = 0.0;
    const bool ends = x.lane == 0 || x.lane == 63;
    load_border(x.lane, c, e, P, p_old, pa, pb, w);
    load_border(x.lane, c, e, P, src, za, zb, pn);
    pa = fma(beta, pa, za);
    pb = fma(beta, pb, zb);
    if (ends)
#pragma unroll
        for (int q = 0; q < R; ++q) ph[q] = fma(beta, w[q], pn[q]);
    __syncthreads();
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
#pragma unroll
        for (int q = 0; q < R; ++q) pv[q] = pn[q];
        pw = tot[0];
        const double alpha = rro / pw;
#pragma unroll
        for (int q = 0; q < R; ++q) {
            uv[q] = fma(alpha, pv[q], uv[q]);
            rv[q] = fma(-alpha, w[q], rv[q]);
        }
        M.apply(f, rv, zv);
        x.send(zv);
        strip_dots<S>(rv, zv, acc[0]);
        x.sum_begin(acc);
        x.template sum_end<true>(tot, za, zb);
        beta = tot[0] / rro;
        rro = tot[0];
        // the border of the next p: this one's and z's
        pa = fma(beta, pa, za);
        pb = fma(beta, pb, zb);
        if (ends)
#pragma unroll
            for (int q = 0; q < R; ++q) ph[q] = fma(beta, ph[q], x.in()[q]);
    }
    if (sh.fault) return;
    store_cells(c, P, u, uv);
    store_cells(c, P, r, rv);
    if (PREC != PREC_NONE) store_cells(c, P, z, zv);
    // the last iteration's p where the streaming kernels write it
    store_cells(c, P, (st.cg_calc_steps & 1) ? pB : pA, pv);
    if (blockIdx.x == 0 && threadIdx.x == 0) *ra.st = st;
}

// A launch's parameters: the exchange memory with fresh tags for at most
// `reds` sums and `halos` exchanges
Comm next_comm(tl_chunk *c, unsigned int reds, unsigned int halos)
{
    const Ext e = ext_interior(c);
    Comm cm;
    cm.red = c->res_mem;
    cm.halo = c->res_mem + RED_WORDS;
    cm.fault = c->res_fault;
    cm.rseq = c->res_rseq;
    cm.hseq = c->res_hseq;
    c->res_rseq += reds + 2;
    c->res_hseq += halos + 2;
    cm.nbx = e.ntx;
    cm.nby = (e.nty + c->res_rows - 1) / c->res_rows;
    cm.nty = e.nty;
    return cm;
}

}  // namespace res

using namespace res;

// The fewest tile rows per block with which a block per compute unit covers
// the grid: more, smaller blocks have less to do between exchanges (one CG
// iteration, no preconditioner: 256^2 with 1, 2 and 4 tile rows per block
// 4.4, 4.6 and 5.5 us; 512^2 5.5, 5.6 and 6.1 us). The quad order of the sums
// is a condition of the kernels.
int resident_rows(const Ext &e, int cus)
{
    if (!e.quad) return 0;
    for (int tr : {1, 2, 4})
        if (e.ntx * ((e.nty + tr - 1) / tr) <= cus) return tr;
    return 0;
}

size_t resident_bytes(const Ext &e) { return sizeof(u64) * (RED_WORDS + (size_t)HALO_WORDS * e.ntx * e.nty); }

bool resident_eligible(const tl_chunk *c)
{
    return c->res_rows && c->faces.zl && c->faces.zr && c->faces.zb && c->faces.zt;
}

template <typename F, typename... A>
static hipError_t coop(tl_chunk *c, F *kernel, const Comm &cm, int nw, A... args)
{
    void *p[] = {(void *)&args...};
    return hipLaunchCooperativeKernel((const void *)kernel, dim3(cm.nbx * cm.nby), dim3(nw * 64), p, 0, c->s);
}

// the kernel's form for the chunk's tile rows per block and preconditioner:
// K(preconditioner, wavefronts, strips per wavefront)
#define TL_RES_ROWS(K, P) (c->res_rows == 1 ? K(P, 4, 1) : c->res_rows == 2 ? K(P, 8, 1) : K(P, 8, 2))
#define TL_RES_ANY(K)                                           \
    (c->prec == PREC_BLOCK  ? TL_RES_ROWS(K, PREC_BLOCK)        \
     : c->prec == PREC_DIAG ? TL_RES_ROWS(K, PREC_DIAG)         \
                            : TL_RES_ROWS(K, PREC_NONE))

hipError_t launch_res_cg(tl_chunk *c, int iters)
{
    const Ext e = ext_interior(c);
    const Comm cm = next_comm(c, 2u * iters + 2, iters);
    const RedArgs ra = red_args(c, RED_CG_RRN, true);
    double **f = c->f2;
#define TL_K(P, NW, S)                                                                                          \
    coop(c, k_res_cg<P, NW, S>, cm, NW, c->g, e, cm, f[F_U], f[F_R], f[F_Z], f[F_P], f[F_P2],                   \
         (const double *)f[F_COND], c->faces, ra, iters)
    return TL_RES_ANY(TL_K);
#undef TL_K
}

}  // namespace tl
