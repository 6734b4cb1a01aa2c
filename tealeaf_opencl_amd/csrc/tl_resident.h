// Resident solver: the iteration loops of the device-resident driver for
// grids whose whole solver state fits the chip's registers (about a million
// cells), one cooperative launch per solve phase instead of two to a dozen
// dependent launches per iteration.
//
// Decomposition: a block of NW wavefronts owns a column of NW strips, 64
// columns x 4 NW rows; a thread owns one column of one 4-row strip, as in the
// tile kernels, and keeps its cells' vectors, faces and preconditioner factors
// in registers for the whole phase. Neighbouring values come from the next
// lane (DPP), from the next wavefront (LDS), or from the neighbouring block.
//
// Exchange between blocks: a value crosses as two 64-bit words, each half of
// its bits with a 32-bit tag, stored and polled with relaxed device-scope
// atomics: a word whose tag is the expected one carries its half of the value,
// so no fence, flag or barrier stands between the store and its reader. The
// tag is the running number of the exchange (of one kind: sums or halos), and
// successive exchanges of a kind alternate between two slots: a block writes
// exchange n+2 only after it has read its readers' exchange n+1, which they
// send after reading n.
//
// Sums have the association of the tile kernels and their finisher (strips of
// a 64x16 tile, tiles in groups of 64, groups in order), so a phase gives
// bitwise what the same iterations give launched one by one. Every block forms
// every total from the tiles' partial sums and runs the scalar algebra on its
// own copy of the state; block 0 stores it back.
//
// Every poll is bounded (RES_TIMEOUT): a block that waits longer sets the
// launch's fault flag and leaves, and so does every other one.
#pragma once

#include <hip/hip_runtime.h>

#include <mutex>

#include "tl_chunk.h"
#include "tl_common.h"
#include "tl_device.h"

namespace tl {
namespace res {

typedef unsigned long long u64;

constexpr int MAX_Q = 2;                     // sums per reduction
constexpr int MAX_SLOTS = 4 * MAX_QUADS;     // one per tile at most
// Copies of the partial sums, one for the readers of every eighth block. With
// one copy, 256 blocks polling the same 4 KB took 3.6 us per sum (40 blocks
// 1.6 us); with eight a CG iteration of 512^2 went from 9 to 5.5 us.
constexpr int COPIES = 8;
constexpr int RED_WORDS = 2 * MAX_Q * COPIES * 2 * MAX_SLOTS;
constexpr int EDGE = 64;                     // values per edge of a block
constexpr int HALO_WORDS = 2 * 4 * 2 * EDGE; // per block: slots x edges x words
// ticks of the 100 MHz clock after which a poll gives up
constexpr long long RES_TIMEOUT = 500000000LL;

enum { EDGE_TOP = 0, EDGE_BOTTOM, EDGE_LEFT, EDGE_RIGHT };  // top: the block's first row

// what the host passes: the exchange memory and the first tags of the launch
struct Comm {
    u64 *red;
    u64 *halo;
    unsigned int *fault;
    unsigned int rseq, hseq;
    int nbx, nby;      // blocks
    int nty;           // tile rows
};

// NW wavefronts of S strips each: 64 columns x 4 S NW rows
template <int NW, int S>
struct Shared {
    double top[NW][64], bot[NW][64];   // first and last row of every wavefront, of the vector sent
    double part[MAX_Q][NW * S];        // strips' sums
    double grp[MAX_Q][MAX_SLOTS / 64]; // groups' sums
    double col[2][EDGE];               // lanes 0 and 63 of the vector sent (by row)
    double in[2][EDGE];                // the vector received beyond them
    double side[3][2][EDGE];           // vectors kept beyond them
    double kxe[EDGE];                  // Kx east of lane 63 (by row)
    int fault;
};

__device__ __forceinline__ void ll_put(u64 *w0, u64 *w1, double v, unsigned int tag)
{
    const u64 b = __builtin_bit_cast(u64, v), t = (u64)tag << 32;
    __hip_atomic_store(w0, (b & 0xffffffffull) | t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(w1, (b >> 32) | t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A poll of up to two values (each two words, `off` apart; null: none) until
// both carry their tags.
struct Want {
    const u64 *w;
    int off;
    unsigned int tag;
    double v;
};

__device__ __forceinline__ bool ll_take(Want &a, u64 x, u64 y)
{
    if ((unsigned int)(x >> 32) != a.tag || (unsigned int)(y >> 32) != a.tag) return false;
    a.v = __builtin_bit_cast(double, (x & 0xffffffffull) | (y << 32));
    return true;
}

__device__ __forceinline__ void ll_poll(Want &a, Want &b, unsigned int *fault, int *sh_fault)
{
    bool na = a.w != nullptr, nb = b.w != nullptr;
    long long t0 = 0;
    for (int spin = 1; na || nb; ++spin) {
        u64 x = 0, y = 0, p = 0, q = 0;
        if (na) {
            x = __hip_atomic_load(a.w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            y = __hip_atomic_load(a.w + a.off, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (nb) {
            p = __hip_atomic_load(b.w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            q = __hip_atomic_load(b.w + b.off, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (na) na = !ll_take(a, x, y);
        if (nb) nb = !ll_take(b, p, q);
        if ((spin & 1023) == 0) {
            const long long t = wall_clock64();
            if (t0 == 0) t0 = t;
            if (t - t0 > RES_TIMEOUT || __hip_atomic_load(fault, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM)) {
                __hip_atomic_store(fault, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                *sh_fault = 1;
                return;
            }
        }
    }
}

// a block's place and its running exchange numbers
template <int NW, int S>
struct Ctx {
    static constexpr int R = S * STRIP;                    // rows of a thread
    static constexpr int TR = NW * S / STRIPS_PER_TILE;    // tile rows of a block: 1, 2 or 4 of a quad
    static_assert(TR == 1 || TR == 2 || TR == 4, "a block's tile rows lie in one quad");
    static_assert(NW * R <= EDGE, "edge");
    const Comm &cm;
    Shared<NW, S> &sh;
    int lane, wv, bx, by;
    unsigned int rseq, hseq;

    __device__ __forceinline__ Ctx(const Comm &c, Shared<NW, S> &s) : cm(c), sh(s)
    {
        lane = threadIdx.x & 63;
        // wave-uniform
        wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        bx = (int)blockIdx.x % cm.nbx;
        by = (int)blockIdx.x / cm.nbx;
        rseq = cm.rseq;
        hseq = cm.hseq;
    }

    __device__ __forceinline__ u64 *edge(int bx_, int by_, int which, unsigned int seq) const
    {
        return cm.halo + ((((long)(by_ * cm.nbx + bx_) * 2 + (seq & 1)) * 4 + which) * 2) * EDGE;
    }
    __device__ __forceinline__ u64 *slot(int q, int copy, unsigned int seq) const
    {
        return cm.red + ((((seq & 1) * MAX_Q + q) * COPIES + copy) * 2) * MAX_SLOTS;
    }

    // Wavefronts' parts in an exchange: one each of the block's edges, and the
    // units of 64 partial sums starting at the fourth.
    static constexpr int W_LEFT = 1, W_RIGHT = 2, W_SLOTS = 3;

    // Sends this thread's cells of a vector to whoever reads their border:
    // rows to the neighbouring wavefronts through LDS, edges to the
    // neighbouring blocks (the columns by way of LDS, in recv). A
    // __syncthreads and recv follow.
    __device__ __forceinline__ void send(const double *v)
    {
        ++hseq;
        sh.top[wv][lane] = v[0];
        sh.bot[wv][lane] = v[R - 1];
        if (lane == 0 || lane == 63)
#pragma unroll
            for (int q = 0; q < R; ++q) sh.col[lane & 1][wv * R + q] = v[q];
        if (wv == 0 && by > 0) {
            u64 *w = edge(bx, by, EDGE_TOP, hseq);
            ll_put(w + lane, w + EDGE + lane, v[0], hseq);
        }
        if (wv == NW - 1 && by < cm.nby - 1) {
            u64 *w = edge(bx, by, EDGE_BOTTOM, hseq);
            ll_put(w + lane, w + EDGE + lane, v[R - 1], hseq);
        }
    }

    // publishes the columns and says what this lane reads of the border
    __device__ __forceinline__ Want want_border()
    {
        Want a{nullptr, EDGE, hseq, 0.0};
        const u64 *w = nullptr;
        if (wv == W_LEFT && bx > 0 && lane < NW * R) {
            u64 *o = edge(bx, by, EDGE_LEFT, hseq) + lane;
            ll_put(o, o + EDGE, sh.col[0][lane], hseq);
            w = edge(bx - 1, by, EDGE_RIGHT, hseq);
        }
        if (wv == W_RIGHT && bx < cm.nbx - 1 && lane < NW * R) {
            u64 *o = edge(bx, by, EDGE_RIGHT, hseq) + lane;
            ll_put(o, o + EDGE, sh.col[1][lane], hseq);
            w = edge(bx + 1, by, EDGE_LEFT, hseq);
        }
        if (wv == 0 && by > 0) w = edge(bx, by - 1, EDGE_BOTTOM, hseq);
        if (wv == NW - 1 && by < cm.nby - 1) w = edge(bx, by + 1, EDGE_TOP, hseq);
        if (w) a.w = w + lane;
        return a;
    }

    // The border of the cells sent last: the row above (va, index k - 1) and
    // below (vb), zero beyond the grid's walls; after the next __syncthreads
    // the columns west of lane 0 and east of lane 63 are in sh.in.
    __device__ __forceinline__ void take_border(const Want &a, double &va, double &vb)
    {
        va = wv > 0 ? sh.bot[wv - 1][lane] : a.v;
        vb = wv < NW - 1 ? sh.top[wv + 1][lane] : a.v;
        if (wv == W_LEFT && lane < NW * R) sh.in[0][lane] = a.v;
        if (wv == W_RIGHT && lane < NW * R) sh.in[1][lane] = a.v;
    }

    // this thread's place in sh.side[k] and sh.in (lane 0: west, lane 63: east;
    // the other lanes read along)
    __device__ __forceinline__ double *side(int k) const { return sh.side[k][lane >> 5] + wv * R; }
    __device__ __forceinline__ double *in() const { return sh.in[lane >> 5] + wv * R; }
    __device__ __forceinline__ bool ends() const { return lane == 0 || lane == 63; }

    // A vector's border with nothing to sum: its columns go to sh.in. `meanwhile`
    // runs between the barriers.
    template <typename F>
    __device__ __forceinline__ void swap(const double *v, double &va, double &vb, F &&meanwhile)
    {
        send(v);
        __syncthreads();
        meanwhile();
        Want a = want_border(), b{nullptr, 0, 0, 0.0};
        ll_poll(a, b, cm.fault, &sh.fault);
        take_border(a, va, vb);
        __syncthreads();
    }

    __device__ __forceinline__ void swap(const double *v, double &va, double &vb)
    {
        swap(v, va, vb, []() {});
    }

    // Totals of NQ sums over the grid, the same in every thread of every
    // block, in two calls with the block's barrier in the first: v[q][s] is
    // this thread's sum over its strip s.
    template <int NQ>
    __device__ __forceinline__ void sum_begin(const double (&v)[NQ][S])
    {
        ++rseq;
#pragma unroll
        for (int q = 0; q < NQ; ++q)
#pragma unroll
            for (int s = 0; s < S; ++s) {
                const double t = wave_sum(v[q][s]);
                if (lane == 0) sh.part[q][wv * S + s] = t;
            }
        __syncthreads();
    }

    // the partials' butterfly of the finisher from the point where a group's
    // 64 tiles have become 64 / TR slots
    static __device__ __forceinline__ double slot_sum(double v)
    {
        if (TR == 1) v = swap_add<32>(v);
        if (TR <= 2) v = swap_add<16>(v);
        v += dpp_ror<8>(v);
        v += dpp_ror<4>(v);
        v += dpp_ror<2>(v);
        v += dpp_ror<1>(v);
        return v;
    }

    // BORDER: together with the border of a vector sent before sum_begin
    template <bool BORDER, int NQ>
    __device__ __forceinline__ void sum_end(double (&tot)[NQ], double &va, double &vb)
    {
        // the block's tiles, those outside the grid counting zero
        const int t = threadIdx.x;
        const int quads = cm.nbx * ((cm.nty + 3) / 4), ngrp = (quads + 15) / 16;
        const int b = by * TR / 4 * cm.nbx + bx;      // the block's quad
        const bool alone = cm.nbx * cm.nby == 1;
        if (t < NQ * COPIES) {
            const int tq = t / COPIES;
            double x[TR];
#pragma unroll
            for (int i = 0; i < TR; ++i) {
                const double *p = sh.part[tq] + STRIPS_PER_TILE * i;
                x[i] = by * TR + i < cm.nty ? ((p[0] + p[1]) + p[2]) + p[3] : 0.0;
            }
            const double y = TR == 4 ? (x[0] + x[1 % TR]) + (x[2 % TR] + x[3 % TR]) : TR == 2 ? x[0] + x[1 % TR] : x[0];
            // slot within the group of 16 quads
            const int row = TR == 4 ? 0 : TR == 2 ? (by & 1) * 16 : (by & 1) * 32 + (by >> 1 & 1) * 16;
            const int i = b / 16 * (64 / TR) + row + b % 16;
            u64 *w = slot(tq, t % COPIES, rseq) + i;
            if (!alone) ll_put(w, w + MAX_SLOTS, y, rseq);
            else if (t % COPIES == 0) sh.grp[tq][0] = y;
        }
        Want edge{nullptr, 0, 0, 0.0}, sum{nullptr, MAX_SLOTS, rseq, 0.0};
        if (BORDER) edge = want_border();
        const int nunit = alone ? 0 : (ngrp * (64 / TR) + 63) / 64 * NQ;
        int u = (wv + NW - W_SLOTS) % NW;
        do {
            // unit u: slots sl of sum q
            const int q = u % NQ, sl = u / NQ * 64 + lane;
            // the slot's block: row y0
            const int in = sl % (64 / TR), bq = sl / (64 / TR) * 16 + (in & 15);
            const int y0 = bq / cm.nbx * (4 / TR) + (TR == 4 ? 0 : TR == 2 ? in >> 4 : (in >> 5) + 2 * (in >> 4 & 1));
            sum.w = u < nunit && y0 < cm.nby ? slot(q, blockIdx.x % COPIES, rseq) + sl : nullptr;
            sum.v = 0.0;
            ll_poll(edge, sum, cm.fault, &sh.fault);
            edge.w = nullptr;
            if (u < nunit) {
                const double y = slot_sum(sum.v);
                if (in == 0) sh.grp[q][sl / (64 / TR)] = y;
            }
            u += NW;
        } while (u < nunit);
        if (BORDER) take_border(edge, va, vb);
        __syncthreads();
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            double s = 0.0;
            for (int i = 0; i < ngrp; ++i) s += sh.grp[q][i];
            tot[q] = s;
        }
    }
    template <int NQ>
    __device__ __forceinline__ void sum_end(double (&tot)[NQ])
    {
        double va, vb;
        sum_end<false>(tot, va, vb);
    }
};

// ---------------------------------------------------------------------------
// a thread's cells: S strips of one column, their operator and preconditioner
// in registers
// ---------------------------------------------------------------------------

// which of the cells lie in the grid
struct Cells {
    int j, ks, i0;
    int rows;          // rows that do (from the first)
};

template <int NW, int S>
__device__ __forceinline__ Cells thread_cells(const Ctx<NW, S> &x, const Geom &g, const Ext &e)
{
    constexpr int R = S * STRIP;
    Cells c;
    c.j = e.j0 + x.bx * TILE_X + x.lane;
    c.ks = e.k0 + (x.by * NW + x.wv) * R;
    c.i0 = IX(g, c.j, c.ks);
    const int left = e.k1 - c.ks + 1;
    c.rows = c.j > e.j1 || left <= 0 ? 0 : left < R ? left : R;
    return c;
}

// Faces of the cells: Kx west of each, Ky above each and below the last. Those
// of cells outside the grid are zero. Kx east of a cell is the next lane's, of
// lane 63's cells sh.kxe.
template <int NW, int S>
struct CellFaces {
    static constexpr int R = S * STRIP;
    double kx[R], ky[R + 1];
    const double *kxe;

    // from the conductivity (or its 1/(2w))
    template <bool HALF_INV, typename T>
    __device__ __forceinline__ void from_cond(Ctx<NW, S> &x, const Geom &g, const Faces &fc, const T *W, const Cells &c)
    {
        set(x, c, [&](int o, double *k0, double *k1, double *y) {
            strip_k_cond<HALF_INV>(g, fc, W, c.i0 + o * g.pitch, g.pitch, c.j, c.ks + o, k0, k1, y);
        });
    }
    // read
    template <typename T>
    __device__ __forceinline__ void from_fields(Ctx<NW, S> &x, const Geom &g, const T *Kx, const T *Ky, const Cells &c)
    {
        set(x, c, [&](int o, double *k0, double *k1, double *y) {
            strip_k(Kx, Ky, c.i0 + o * g.pitch, g.pitch, k0, k1, y);
        });
    }
    __device__ __forceinline__ double east(int q) const { return dpp_shl1(kx[q], kxe[q]); }

  private:
    template <typename F>
    __device__ __forceinline__ void set(Ctx<NW, S> &x, const Cells &c, F &&strip)
    {
        double k1[R];
#pragma unroll
        for (int q = 0; q < R; ++q) kx[q] = k1[q] = ky[q] = 0.0;
        ky[R] = 0.0;
#pragma unroll
        for (int o = 0; o < R; o += STRIP) {
            if (o >= c.rows) continue;
            double y[STRIP + 1];
            strip(o, kx + o, k1 + o, y);
            if (o == 0) ky[0] = y[0];
#pragma unroll
            for (int q = 0; q < STRIP; ++q) ky[o + q + 1] = y[q + 1];
        }
#pragma unroll
        for (int q = 0; q < R; ++q)
            if (q >= c.rows) kx[q] = k1[q] = ky[q + 1] = 0.0;
        if (x.lane == 63)
#pragma unroll
            for (int q = 0; q < R; ++q) x.sh.kxe[x.wv * R + q] = k1[q];
        kxe = x.sh.kxe + x.wv * R;
    }
};

// M^-1 with the factors kept (bitwise strip_precondition)
template <int PREC, bool FAST, int NW, int S>
struct CellPrec {
    static constexpr int R = S * STRIP;
    double cp[R], bf[R];  // block: Thomas factors (first of a strip: 1 / b0 with FAST, else its refined reciprocal)
    double b0[S];
    double mi[R];         // diagonal: 1 / diag

    __device__ __forceinline__ void init(const Geom &g, const Cells &c, const CellFaces<NW, S> &f)
    {
        double kx1[R];
#pragma unroll
        for (int q = 0; q < R; ++q) kx1[q] = f.east(q);
        if (PREC == PREC_BLOCK) {
#pragma unroll
            for (int s = 0; s < S; ++s) {
                const int o = s * STRIP;
                double a[STRIP], b[STRIP], cc[STRIP];
                strip_abc(f.kx + o, kx1 + o, f.ky + o, a, b, cc);
                const int upper = o < c.rows ? block_top(g, c.ks + o) : 0;
                strip_factors<FAST ? DIV_RCP32 : DIV_NR>(upper, b, a, cc, cp + o, bf + o);
                b0[s] = b[0];
                if (!FAST) {
                    double y = __builtin_amdgcn_rcp(b[0]);
                    double e = fma(-b[0], y, 1.0);
                    y = fma(y, e, y);
                    e = fma(-b[0], y, 1.0);
                    bf[o] = fma(y, e, y);
                }
                if (upper <= 0) bf[o] = b0[s] = 0.0;
            }
        } else if (PREC == PREC_DIAG) {
#pragma unroll
            for (int q = 0; q < R; ++q) {
                const double dg = diag_of(f.kx[q], kx1[q], f.ky[q], f.ky[q + 1]);
                mi[q] = FAST ? rcp_fp32(dg) : div_nr(1.0, dg);
            }
        }
    }

    __device__ __forceinline__ void apply(const CellFaces<NW, S> &f, const double *r, double *z) const
    {
        if (PREC == PREC_BLOCK) {
#pragma unroll
            for (int s = 0; s < S; ++s) {
                const int o = s * STRIP;
                double dp[STRIP];
                if (FAST) {
                    dp[0] = r[o] * bf[o];
                } else {
                    // div_nr(r, b0)
                    const double q = r[o] * bf[o];
                    dp[0] = fma(fma(-b0[s], q, r[o]), bf[o], q);
                }
#pragma unroll
                for (int k = 1; k < STRIP; ++k) dp[k] = fma(f.ky[o + k], dp[k - 1], r[o + k]) * bf[o + k];
                z[o + STRIP - 1] = dp[STRIP - 1];
#pragma unroll
                for (int k = STRIP - 2; k >= 0; --k) z[o + k] = fma(-cp[o + k], z[o + k + 1], dp[k]);
            }
        } else if (PREC == PREC_DIAG) {
#pragma unroll
            for (int q = 0; q < R; ++q) z[q] = r[q] * mi[q];
        } else {
#pragma unroll
            for (int q = 0; q < R; ++q) z[q] = r[q];
        }
    }
};

// out = A v: va, vb the rows above and below, vh (a place in LDS or registers)
// the columns beyond lanes 0 and 63
template <int NW, int S>
__device__ __forceinline__ void cells_op(const CellFaces<NW, S> &f, const double *v, double va, double vb,
                                         const double *vh, double *out)
{
    constexpr int R = S * STRIP;
#pragma unroll
    for (int q = 0; q < R; ++q) {
        const double w = dpp_shr1(v[q], vh[q]), e = dpp_shl1(v[q], vh[q]);
        out[q] = opA(f.kx[q], f.east(q), f.ky[q], f.ky[q + 1], v[q], w, e, q ? v[q - 1] : va,
                     q < R - 1 ? v[q + 1] : vb);
    }
}

// a strip's sum of a b, as the tile kernels accumulate it
template <int S>
__device__ __forceinline__ void strip_dots(const double *a, const double *b, double (&acc)[S])
{
#pragma unroll
    for (int s = 0; s < S; ++s) {
        acc[s] = 0.0;
#pragma unroll
        for (int q = 0; q < STRIP; ++q) acc[s] = fma(a[s * STRIP + q], b[s * STRIP + q], acc[s]);
    }
}

template <int R, typename T>
__device__ __forceinline__ void load_cells(const Cells &c, int P, const T *f, double (&v)[R])
{
#pragma unroll
    for (int q = 0; q < R; ++q) v[q] = q < c.rows ? (double)f[c.i0 + q * P] : 0.0;
}

template <int R, typename T>
__device__ __forceinline__ void store_cells(const Cells &c, int P, T *f, const double (&v)[R])
{
#pragma unroll
    for (int q = 0; q < R; ++q)
        if (q < c.rows) f[c.i0 + q * P] = (T)v[q];
}

// the border of the cells read from the field (what an exchange gives for a
// vector that every block has stored); vh: the columns, in lanes 0 and 63
template <int R, typename T>
__device__ __forceinline__ void load_border(int lane, const Cells &c, const Ext &e, int P, const T *f, double &va,
                                            double &vb, double (&vh)[R])
{
    va = c.rows && c.ks > e.k0 ? (double)f[c.i0 - P] : 0.0;
    vb = c.rows == R && c.ks + R <= e.k1 ? (double)f[c.i0 + R * P] : 0.0;
    const bool lft = lane == 0 && c.j > e.j0, rgt = lane == 63 && c.j < e.j1;
#pragma unroll
    for (int q = 0; q < R; ++q) vh[q] = (lft || rgt) && q < c.rows ? (double)f[c.i0 + q * P + (lft ? -1 : 1)] : 0.0;
}

// the thread that runs the scalar algebra: not of the wavefront that publishes
// the block's sums
constexpr int TAIL_THREAD = 64;

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

// iterations, or exchanges, per launch
constexpr int RES_ITERS = 1024;

// a launch's parameters: the exchange memory with fresh tags for at most
// `reds` sums and `halos` exchanges
Comm next_comm(tl_chunk *c, unsigned int reds, unsigned int halos);

// held from a launch to its end: each needs every block on the device at once
std::mutex &launch_mutex();

template <typename F, typename... A>
hipError_t coop(tl_chunk *c, F *kernel, const Comm &cm, int nw, A... args)
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

}  // namespace res
}  // namespace tl
