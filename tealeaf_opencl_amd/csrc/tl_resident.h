// Resident solver: the iteration loops of the device-resident driver for
// grids whose vectors fit the chip's registers and LDS (up to about four
// million cells), one cooperative launch per solve phase instead of two to a
// dozen dependent launches per iteration.
//
// Decomposition: a block of NW wavefronts owns 64 columns x 4 S NW rows; a
// thread owns S strips of four rows of one column. Up to S = 2 (a million cells)
// it keeps its cells' vectors, faces and preconditioner factors in registers
// for the whole phase; with S = 4, 6 or 8 ("tall") the vectors, one of them in
// LDS, and it forms faces and factors anew from the coefficient field in each
// pass over its strips. Neighbouring values come from the next lane (DPP), from
// the next wavefront (LDS), or from the neighbouring block.
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
// a 64x16 tile, tiles in groups of 64, groups in order), so a CG, PPCG or Jacobi
// phase of the native driver gives bitwise what the same iterations give launched
// one by one. Chebyshev's residual norms and the refined solve's p.w are summed
// along bands where launched, and differ by rounding. Every block forms every
// total from the tiles' partial sums and runs the scalar algebra on its own copy
// of the state; block 0 stores it back.
//
// Beginning. A cooperative launch puts the blocks on the device together, but
// does not start them together. The first exchange of every launch is a sum over
// all blocks, to which a block sends after it has read the state: no block changes
// memory before every one has begun, nor stores the state before every one has
// read it.
//
// Every wait is bounded. A block that has looked RES_LOOKS times for a value closes
// the launch (Comm::closed): a block that begins after that sends nothing, says so
// (Comm::left) and leaves, so none passes the first sum, and the launch has changed
// nothing. One that began before has GRACE looks to send its part, and the launch
// goes on if it does. A block that has waited longer than that sets the fault flag
// and leaves, and so does every other one; if none has said that it left at the
// start, the launch was given up in the middle. (Looks are counted, not time: a
// process that is taken off the device does not wait.)
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
constexpr int MAX_SLOTS = 4 * MAX_PILES;     // one per tile of 256 quads at most
// Copies of the partial sums, one for the readers of every eighth block. With
// one copy, 256 blocks polling the same 4 KB, a CG iteration takes 6.4 us at 512^2
// and 9.3 us at 1024^2, with eight 5.6 and 7.7 us.
constexpr int COPIES = 8;
constexpr int RED_WORDS = 2 * MAX_Q * COPIES * 2 * MAX_SLOTS;
// values per edge of a block of `rows` rows, and words of its four edges (slots
// x edges x words)
constexpr int edge_len(int rows) { return rows > 64 ? rows : 64; }
constexpr int halo_words(int rows) { return 2 * 4 * 2 * edge_len(rows); }
// looks (of about a microsecond each) after which a poll closes the launch, and
// after how many more it gives up
constexpr unsigned int RES_LOOKS = 1u << 22, GRACE = 1u << 16;
// the fault flag: a block has left; the host has polls close at their first check
enum { FAULT_STUCK = 1, FAULT_IMPATIENT = 2 };

enum { EDGE_TOP = 0, EDGE_BOTTOM, EDGE_LEFT, EDGE_RIGHT };  // top: the block's first row

// what the host passes: the exchange memory and the first tags of the launch
struct Comm {
    u64 *mem;          // RED_WORDS of partial sums, then the blocks' edges
    unsigned int *fault, *left;
    unsigned int *closed;  // rseq of the launch given up last
    unsigned int rseq, hseq;
    int nbx, nby;      // blocks
    int nty;           // tile rows
};

// NW wavefronts of S strips each: 64 columns x 4 S NW rows. KEEP: vectors kept
// beyond the block's columns.
template <int NW, int S, int KEEP>
struct Shared {
    static constexpr int ROWS = NW * S * STRIP;
    double top[NW][64], bot[NW][64];   // first and last row of every wavefront, of the vector sent
    double part[MAX_Q][NW * S];        // strips' sums
    double grp[MAX_Q][MAX_SLOTS / 64]; // groups' sums
    double col[2][ROWS];               // lanes 0 and 63 of the vector sent (by row)
    double in[2][ROWS];                // the vector received beyond them
    double side[KEEP][2][ROWS];        // vectors kept beyond them
    double kxe[ROWS];                  // Kx east of lane 63 (by row)
    int fault;
};

__device__ __forceinline__ void ll_put(u64 *w0, u64 *w1, double v, unsigned int tag)
{
    const u64 b = __builtin_bit_cast(u64, v), t = (u64)tag << 32;
    __hip_atomic_store(w0, (b & 0xffffffffull) | t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(w1, (b >> 32) | t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A value to poll for (two words of the exchange memory at `at` and at + off;
// at < 0: none)
struct Want {
    int at;
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

// polls until every value has come
template <int N>
__device__ __forceinline__ void ll_poll(const Comm &cm, Want (&a)[N], int *sh_fault)
{
    const u64 *mem = cm.mem;
    bool need[N], any = false;
#pragma unroll
    for (int i = 0; i < N; ++i) any |= need[i] = a[i].at >= 0;
    for (unsigned int spin = 1; any; ++spin) {
        u64 x[N], y[N];
#pragma unroll
        for (int i = 0; i < N; ++i) {
            x[i] = y[i] = 0;
            if (need[i]) {
                x[i] = __hip_atomic_load(mem + a[i].at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                y[i] = __hip_atomic_load(mem + a[i].at + a[i].off, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        any = false;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            if (need[i]) need[i] = !ll_take(a[i], x[i], y[i]);
            any |= need[i];
        }
        if ((spin & 1023) == 0) {
            const unsigned int f = __hip_atomic_load(cm.fault, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            const unsigned int close = f == FAULT_IMPATIENT ? 1024u : RES_LOOKS;
            if (spin == close) __hip_atomic_store(cm.closed, cm.rseq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (f == FAULT_STUCK || spin >= close + GRACE) {
                __hip_atomic_store(cm.fault, (unsigned int)FAULT_STUCK, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                *sh_fault = 1;
                return;
            }
        }
    }
}

// LDS written by some lanes of a wavefront and then read by others of it
__device__ __forceinline__ void wave_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// a block's place and its running exchange numbers
template <int NW, int S, int KEEP>
struct Ctx {
    static constexpr int R = S * STRIP;                  // rows of a thread
    static constexpr int TR = NW * S / STRIPS_PER_TILE;  // tile rows of a block: 1 or 2 of a quad, or quads
    static constexpr int SL = TR == 1 ? 64 : TR == 2 ? 32 : 16;  // slots per group of 16 piles
    static constexpr int EDGE = edge_len(NW * R);
    static_assert(TR == 1 || TR == 2 || TR % 4 == 0, "a block's tile rows lie in one quad or are quads");
    static_assert(2 * R <= 64, "a wavefront exchanges its rows' columns with one lane each");
    const Comm &cm;
    Shared<NW, S, KEEP> &sh;
    int lane, wv, bx, by;
    unsigned int rseq, hseq;

    __device__ __forceinline__ Ctx(const Comm &c, Shared<NW, S, KEEP> &s) : cm(c), sh(s)
    {
        lane = threadIdx.x & 63;
        // wave-uniform
        wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        bx = (int)blockIdx.x % cm.nbx;
        by = (int)blockIdx.x / cm.nbx;
        rseq = cm.rseq;
        hseq = cm.hseq;
    }

    // Thread 0 looks whether the launch was closed, behind a barrier that follows its
    // read of the state; begun, with a barrier of the block, is false if it was. (The
    // loads of the block's cells are between the two.)
    __device__ __forceinline__ unsigned int begin() const
    {
        if (threadIdx.x != 0) return cm.rseq + 1;
        return __hip_atomic_load(cm.closed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __device__ __forceinline__ bool begun(unsigned int closed) const
    {
        if (closed == cm.rseq) {
            sh.fault = 1;
            __hip_atomic_store(cm.left, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            __hip_atomic_store(cm.fault, (unsigned int)FAULT_STUCK, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
        __syncthreads();
        return !sh.fault;
    }

    // places in the exchange memory: an edge's values, a sum's slots
    __device__ __forceinline__ int edge(int bx_, int by_, int which, unsigned int seq) const
    {
        return RED_WORDS + (((by_ * cm.nbx + bx_) * 2 + (int)(seq & 1)) * 4 + which) * 2 * EDGE;
    }
    __device__ __forceinline__ int slot(int q, int copy, unsigned int seq) const
    {
        return (((int)(seq & 1) * MAX_Q + q) * COPIES + copy) * 2 * MAX_SLOTS;
    }
    __device__ __forceinline__ void put(int at, int off, double v, unsigned int tag) const
    {
        ll_put(cm.mem + at, cm.mem + at + off, v, tag);
    }

    // Sends this thread's cells of a vector to whoever reads their border:
    // rows to the neighbouring wavefronts through LDS (first and last, the
    // thread's first and last row), edges to the neighbouring blocks. col(q):
    // row q, read in lanes 0 and 63. A __syncthreads and the reception follow.
    template <typename F>
    __device__ __forceinline__ void send(double first, double last, F &&col)
    {
        if (ends())
#pragma unroll
            for (int q = 0; q < R; ++q) sh.col[lane & 1][wv * R + q] = col(q);
        send(first, last);
    }
    // (the columns are in sh.col)
    __device__ __forceinline__ void send(double first, double last)
    {
        ++hseq;
        sh.top[wv][lane] = first;
        sh.bot[wv][lane] = last;
        if (wv == 0 && by > 0) put(edge(bx, by, EDGE_TOP, hseq) + lane, EDGE, first, hseq);
        if (wv == NW - 1 && by < cm.nby - 1) put(edge(bx, by, EDGE_BOTTOM, hseq) + lane, EDGE, last, hseq);
    }
    __device__ __forceinline__ void send(const double *v)
    {
        send(v[0], v[R - 1], [&](int q) { return v[q]; });
    }

    // lanes 0 .. R-1 exchange the rows' west column, R .. 2R-1 the east one
    __device__ __forceinline__ bool column() const
    {
        return lane < R ? bx > 0 : lane < 2 * R && bx < cm.nbx - 1;
    }
    // publishes them: before the block's barrier where the exchange stands alone,
    // behind it, off the way to the block's sums, where it goes with one
    __device__ __forceinline__ void put_column() const
    {
        const int i = wv * R + lane % R;
        if (column()) put(edge(bx, by, lane < R ? EDGE_LEFT : EDGE_RIGHT, hseq) + i, EDGE, sh.col[lane >= R][i], hseq);
    }
    __device__ __forceinline__ Want want_column() const
    {
        Want a{-1, EDGE, hseq, 0.0};
        if (column())
            a.at = (lane < R ? edge(bx - 1, by, EDGE_RIGHT, hseq) : edge(bx + 1, by, EDGE_LEFT, hseq)) + wv * R + lane % R;
        return a;
    }
    __device__ __forceinline__ Want want_row() const
    {
        Want a{-1, EDGE, hseq, 0.0};
        if (wv == 0 && by > 0) a.at = edge(bx, by - 1, EDGE_BOTTOM, hseq) + lane;
        if (wv == NW - 1 && by < cm.nby - 1) a.at = edge(bx, by + 1, EDGE_TOP, hseq) + lane;
        return a;
    }

    // The border of the cells sent last: the row above (va, index k - 1) and
    // below (vb), zero beyond the grid's walls; the columns west of lane 0 and
    // east of lane 63 go to sh.in, for this wavefront.
    __device__ __forceinline__ void take_border(const Want &column_, const Want &row, double &va, double &vb)
    {
        va = wv > 0 ? sh.bot[wv - 1][lane] : row.v;
        vb = wv < NW - 1 ? sh.top[wv + 1][lane] : row.v;
        if (lane < 2 * R) sh.in[lane >= R][wv * R + lane % R] = column_.v;
        wave_fence();
    }

    // this thread's place in sh.side[k] and sh.in (lane 0: west, lane 63: east;
    // the other lanes read along)
    __device__ __forceinline__ double *side(int k) const { return sh.side[k][lane >> 5] + wv * R; }
    __device__ __forceinline__ double *in() const { return sh.in[lane >> 5] + wv * R; }
    __device__ __forceinline__ bool ends() const { return lane == 0 || lane == 63; }

    // the border of a vector sent before, with nothing to sum. `meanwhile` runs
    // between the barriers.
    template <typename F>
    __device__ __forceinline__ void recv(double &va, double &vb, F &&meanwhile)
    {
        wave_fence();
        put_column();
        __syncthreads();
        meanwhile();
        Want a[2] = {want_column(), want_row()};
        ll_poll(cm, a, &sh.fault);
        take_border(a[0], a[1], va, vb);
        __syncthreads();
    }
    __device__ __forceinline__ void swap(const double *v, double &va, double &vb)
    {
        send(v);
        recv(va, vb, []() {});
    }

    // Totals of NQ sums over the grid, the same in every thread of every block:
    // strip_sum for each sum q and strip s of this thread, sum_begin (the
    // block's barrier), sum_end.
    __device__ __forceinline__ void strip_sum(int q, int s, double v)
    {
        const double t = wave_sum(v);
        if (lane == 0) sh.part[q][wv * S + s] = t;
    }
    __device__ __forceinline__ void sum_begin()
    {
        ++rseq;
        __syncthreads();
    }
    template <int NQ>
    __device__ __forceinline__ void sum_begin(const double (&v)[NQ][S])
    {
#pragma unroll
        for (int q = 0; q < NQ; ++q)
#pragma unroll
            for (int s = 0; s < S; ++s) strip_sum(q, s, v[q][s]);
        sum_begin();
    }

    // the finisher's butterfly from the point where a group's 64 threads have
    // become SL slots
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
        constexpr int PER = TR < 4 ? 4 / TR : 1;      // block rows per pile
        const int t = threadIdx.x;
        const int npile = cm.nbx * ((cm.nby + PER - 1) / PER), ngrp = (npile + 15) / 16;
        const bool alone = cm.nbx * cm.nby == 1;
        if (t < NQ * COPIES) {
            const int tq = t / COPIES;
            // the block's tiles, those outside the grid counting zero; the quads
            // of a pile are added first
            double x[4];
#pragma unroll
            for (int i = 0; i < (TR < 4 ? TR : 4); ++i) {
                x[i] = 0.0;
#pragma unroll
                for (int k = i; k < TR; k += 4) {
                    const double *p = sh.part[tq] + STRIPS_PER_TILE * k;
                    const double y = by * TR + k < cm.nty ? ((p[0] + p[1]) + p[2]) + p[3] : 0.0;
                    x[i] = k < 4 ? y : x[i] + y;
                }
            }
            const double y = TR >= 4 ? (x[0] + x[1]) + (x[2] + x[3]) : TR == 2 ? x[0] + x[1] : x[0];
            // slot within the group of 16 piles
            const int b = by / PER * cm.nbx + bx;
            const int row = TR >= 4 ? 0 : TR == 2 ? (by & 1) * 16 : (by & 1) * 32 + (by >> 1 & 1) * 16;
            const int i = b / 16 * SL + row + b % 16;
            if (!alone) put(slot(tq, t % COPIES, rseq) + i, MAX_SLOTS, y, rseq);
            else if (t % COPIES == 0) sh.grp[tq][0] = y;
        }
        constexpr int NP = BORDER ? 3 : 1;
        Want a[NP];
        if (BORDER) {
            put_column();
            a[NP - 1] = want_column();
            a[NP / 2] = want_row();
        }
        a[0] = {-1, MAX_SLOTS, rseq, 0.0};
        // units of 64 slots, the first one the second wavefront's
        const int nunit = alone ? 0 : (ngrp * SL + 63) / 64 * NQ;
        int u = (wv + NW - 1) % NW;
        do {
            const int q = u % NQ, sl = u / NQ * 64 + lane;
            // the slot's block: row y0
            const int in_ = sl % SL, bq = sl / SL * 16 + (in_ & 15);
            const int y0 = bq / cm.nbx * PER + (TR >= 4 ? 0 : TR == 2 ? in_ >> 4 : (in_ >> 5) + 2 * (in_ >> 4 & 1));
            a[0].at = u < nunit && y0 < cm.nby ? slot(q, blockIdx.x % COPIES, rseq) + sl : -1;
            a[0].v = 0.0;
            ll_poll(cm, a, &sh.fault);
            if (BORDER) a[NP - 1].at = a[NP / 2].at = -1;
            if (u < nunit) {
                const double y = slot_sum(a[0].v);
                if (in_ == 0) sh.grp[q][sl / SL] = y;
            }
            u += NW;
        } while (u < nunit);
        if (BORDER) take_border(a[NP - 1], a[NP / 2], va, vb);
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

template <int NW, int S, int KEEP>
__device__ __forceinline__ Cells thread_cells(const Ctx<NW, S, KEEP> &x, const Geom &g, const Ext &e)
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
template <int NW, int S, int KEEP>
struct CellFaces {
    static constexpr int R = S * STRIP;
    double kx[R], ky[R + 1];
    const double *kxe;

    // from the conductivity (or its 1/(2w))
    template <bool HALF_INV, typename T>
    __device__ __forceinline__ void from_cond(Ctx<NW, S, KEEP> &x, const Geom &g, const Faces &fc, const T *W, const Cells &c)
    {
        set(x, c, [&](int o, double *k0, double *k1, double *y) {
            strip_k_cond<HALF_INV>(g, fc, W, c.i0 + o * g.pitch, g.pitch, c.j, c.ks + o, k0, k1, y);
        });
    }
    // read
    template <typename T>
    __device__ __forceinline__ void from_fields(Ctx<NW, S, KEEP> &x, const Geom &g, const T *Kx, const T *Ky, const Cells &c)
    {
        set(x, c, [&](int o, double *k0, double *k1, double *y) {
            strip_k(Kx, Ky, c.i0 + o * g.pitch, g.pitch, k0, k1, y);
        });
    }
    __device__ __forceinline__ double east(int q) const { return dpp_shl1(kx[q], kxe[q]); }

  private:
    template <typename F>
    __device__ __forceinline__ void set(Ctx<NW, S, KEEP> &x, const Cells &c, F &&strip)
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
template <int PREC, bool FAST, int NW, int S, int KEEP>
struct CellPrec {
    static constexpr int R = S * STRIP;
    double cp[R], bf[R];  // block: Thomas factors (first of a strip: 1 / b0 with FAST, else its refined reciprocal)
    double b0[S];
    double mi[R];         // diagonal: 1 / diag

    __device__ __forceinline__ void init(const Geom &g, const Cells &c, const CellFaces<NW, S, KEEP> &f)
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

    __device__ __forceinline__ void apply(const CellFaces<NW, S, KEEP> &f, const double *r, double *z) const
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
template <int NW, int S, int KEEP>
__device__ __forceinline__ void cells_op(const CellFaces<NW, S, KEEP> &f, const double *v, double va, double vb,
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

// a wave-uniform value, in scalar registers
__device__ __forceinline__ double uniform(double v)
{
    const u64 b = __builtin_bit_cast(u64, v);
    const u64 lo = (unsigned int)__builtin_amdgcn_readfirstlane((int)b);
    const u64 hi = (unsigned int)__builtin_amdgcn_readfirstlane((int)(b >> 32));
    return __builtin_bit_cast(double, lo | hi << 32);
}

// A thread's R values of a vector that a step touches once: in LDS where two
// strips' vectors are more than the registers (a form that spills registers is
// not built: the compiler can place a spill where only some lanes of a
// wavefront are active), else in registers.
template <bool LDS, int R, int NW>
struct HeldMem {
    double v[LDS ? R : 1][LDS ? NW * 64 : 1];
};
template <bool LDS, int R, int NW>
struct Held {
    HeldMem<LDS, R, NW> &mem;
    double own[LDS ? 1 : R];
    __device__ __forceinline__ explicit Held(HeldMem<LDS, R, NW> &m) : mem(m) {}
    __device__ __forceinline__ double &operator()(int q) { return LDS ? mem.v[LDS ? q : 0][LDS ? threadIdx.x : 0] : own[LDS ? 0 : q]; }
    __device__ __forceinline__ void put(const double *v)
    {
#pragma unroll
        for (int q = 0; q < R; ++q) (*this)(q) = v[q];
    }
    __device__ __forceinline__ void get(double *v)
    {
#pragma unroll
        for (int q = 0; q < R; ++q) v[q] = (*this)(q);
    }
};

// the thread that runs the scalar algebra: not of the wavefront that publishes
// the block's sums
constexpr int TAIL_THREAD = 64;

// ---------------------------------------------------------------------------
// tall blocks: faces formed strip by strip in every pass
// ---------------------------------------------------------------------------

// A wavefront's rows and the place of its cells. Everything but the lane's
// column is wave-uniform, so that a cell's address is a scalar base and one
// 32-bit offset per thread.
template <int NW, int S>
struct Tall {
    static constexpr int R = S * STRIP;
    int ks, rows;         // first row; rows in the grid
    int i0, P;            // place of (lane 0's column, first row); pitch
    unsigned int lo;      // columns from lane 0's (the last one's beyond the grid)
    bool col, west;       // the column lies in the grid; so does the one west of it

    template <int KEEP>
    __device__ __forceinline__ Tall(const Ctx<NW, S, KEEP> &x, const Geom &g, const Ext &e)
    {
        const int jw = e.j0 + x.bx * TILE_X, last = min(TILE_X - 1, e.j1 - jw);
        ks = e.k0 + (x.by * NW + x.wv) * R;
        const int left = e.k1 - ks + 1;
        rows = left <= 0 ? 0 : left < R ? left : R;
        i0 = IX(g, jw, rows ? ks : e.k0);
        P = g.pitch;
        col = x.lane <= last;
        west = col && (x.lane > 0 || x.bx > 0);
        lo = (unsigned int)min(x.lane, last);
    }

    // The same for one pass, of which the compiler cannot tell that it is the
    // same in every pass: what a pass derives from it (row addresses, which rows
    // are in the grid) is formed when needed instead of kept in registers that
    // the vectors need.
    __device__ __forceinline__ Tall again() const
    {
        Tall c = *this;
        asm volatile("" : "+s"(c.ks), "+s"(c.rows), "+s"(c.i0), "+v"(c.lo));
        return c;
    }

    template <typename T>
    __device__ __forceinline__ T &at(T *f, int row) const
    {
        return *(T *)((uintptr_t)(f + (i0 + row * P)) + lo * (unsigned int)sizeof(T));
    }
    // cells o .. o+3, of which those outside the grid are not read
    template <typename T>
    __device__ __forceinline__ void read4(const T *f, int o, T *v) const
    {
#pragma unroll
        for (int q = 0; q < STRIP; ++q) {
            v[q] = (T)0;
            if (o + q < rows) v[q] = at(f, o + q);
        }
#pragma unroll
        for (int q = 0; q < STRIP; ++q) v[q] = col ? v[q] : (T)0;
    }
    template <typename T>
    __device__ __forceinline__ void write4(T *f, int o, const T *v) const
    {
        if (col)
#pragma unroll
            for (int q = 0; q < STRIP; ++q)
                if (o + q < rows) at(f, o + q) = v[q];
    }
};

// Faces from a per-cell field: the conductivity (bitwise those that
// tea_leaf_init_common stores) or, with HALF_INV, its 1/(2w). Every wall is
// closed (resident_eligible), so a face is formed or zero.
template <typename T, bool HALF_INV, int NW, int S>
struct CondStream {
    static constexpr int R = S * STRIP, FIELDS = 1;
    static constexpr bool NARROW = sizeof(T) < sizeof(double);
    const T *w;
    double rx, ry, above, below;
    const double *cw, *kxe;     // LDS: the field west of lane 0, Kx east of lane 63
    int k0, k1;                 // the grid's first and last row

    // face_coef_nr / face_coef_h, the product by the scale kept from being fused
    // into a sum of faces: which of two would be is the compiler's choice
    static __device__ __forceinline__ double face(double a, double b, double scale)
    {
#pragma clang fp contract(off)
        const double v = HALF_INV ? a + b : div_nr(a + b, 2.0 * a * b);
        return v * scale;
    }
    // cwl: R values of LDS
    template <int KEEP>
    __device__ __forceinline__ CondStream(Ctx<NW, S, KEEP> &x, const Tall<NW, S> &c, const Geom &g, const Ext &e,
                                          const Faces &fc, const T *W, const T *, double *cwl)
        : w(W), rx(fc.rx), ry(fc.ry), cw(cwl), kxe(x.sh.kxe + x.wv * R), k0(e.k0), k1(e.k1)
    {
        above = c.rows && c.ks > e.k0 ? (double)c.at(W, -1) : 1.0;
        below = c.rows == R && c.ks + R <= e.k1 ? (double)c.at(W, R) : 1.0;
        // one row per lane: the columns beyond the block are read once
        if (x.lane < R) {
            const int jw = e.j0 + x.bx * TILE_X, je = jw + TILE_X - 1, k = c.ks + x.lane;
            double a = 1.0, b = 0.0;
            if (x.lane < c.rows) {
                if (jw > e.j0) a = (double)W[IX(g, jw - 1, k)];
                if (je < e.j1) b = face((double)W[IX(g, je, k)], (double)W[IX(g, je + 1, k)], rx);
            }
            cwl[x.lane] = a;
            x.sh.kxe[x.wv * R + x.lane] = b;
        }
        wave_fence();
    }

    // Rows o .. o+3 of the field. A row beyond the grid repeats the last one, a
    // column beyond it the last one (Tall::lo): the cells there hold zeros and
    // are cut off by the zero face before them, so their own faces only have to
    // be numbers.
    __device__ __forceinline__ void rows4(const Tall<NW, S> &c, int o, double *v) const
    {
#pragma unroll
        for (int q = 0; q < STRIP; ++q) v[q] = (double)c.at(w, min(o + q, max(c.rows - 1, 0)));
    }

    // f(d, s, kx0, kx1, ky) for every strip s with rows in the grid, top to
    // bottom; d: c.again()
    template <typename F>
    __device__ __forceinline__ void pass(const Tall<NW, S> &c, F &&f) const
    {
        const Tall<NW, S> d = c.again();
        double cur[STRIP], nxt[STRIP] = {}, up = above;
        rows4(d, 0, cur);
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const int o = s * STRIP;
            if (o >= d.rows) continue;
            if (s + 1 < S) rows4(d, o + STRIP, nxt);
            const double down = s + 1 < S ? nxt[0] : below;
            double kx0[STRIP], kx1[STRIP], ky[STRIP + 1];
#pragma unroll
            for (int q = 0; q < STRIP; ++q) {
                const double kx = face(dpp_shr1(cur[q], cw[o + q]), cur[q], rx);
                kx0[q] = d.west ? kx : 0.0;
                kx1[q] = dpp_shl1(kx0[q], kxe[o + q]);
                ky[q] = face(q ? cur[q - 1] : up, cur[q], ry);
            }
            ky[STRIP] = face(cur[STRIP - 1], down, ry);
            // the walls above the first and below the last row
            if (s == 0 && d.ks == k0) ky[0] = 0.0;
            if (d.ks + o + STRIP > k1) {
#pragma unroll
                for (int q = 1; q <= STRIP; ++q)
                    if (o + q == d.rows) ky[q] = 0.0;
            }
            f(d, s, kx0, kx1, ky);
            up = cur[STRIP - 1];
#pragma unroll
            for (int q = 0; q < STRIP; ++q) cur[q] = nxt[q];
        }
    }
};

// Faces read from two fields, which hold zeros on the walls
template <typename T, int NW, int S>
struct FieldStream {
    static constexpr int R = S * STRIP, FIELDS = 2;
    static constexpr bool NARROW = sizeof(T) < sizeof(double);
    const T *kx, *ky;
    const double *kxe;

    template <int KEEP>
    __device__ __forceinline__ FieldStream(Ctx<NW, S, KEEP> &x, const Tall<NW, S> &c, const Geom &g, const Ext &e,
                                           const Faces &, const T *Kx, const T *Ky, double *)
        : kx(Kx), ky(Ky), kxe(x.sh.kxe + x.wv * R)
    {
        if (x.lane < R) {
            const int je = e.j0 + x.bx * TILE_X + TILE_X - 1, k = c.ks + x.lane;
            x.sh.kxe[x.wv * R + x.lane] = x.lane < c.rows && je < e.j1 ? (double)Kx[IX(g, je + 1, k)] : 0.0;
        }
        wave_fence();
    }

    // (rows beyond the grid lie in the fields' halos and margins)
    template <typename F>
    __device__ __forceinline__ void pass(const Tall<NW, S> &c, F &&f) const
    {
        const Tall<NW, S> d = c.again();
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const int o = s * STRIP;
            if (o >= d.rows) continue;
            double kx0[STRIP], kx1[STRIP], y[STRIP + 1];
#pragma unroll
            for (int q = 0; q < STRIP; ++q) kx0[q] = (double)d.at(kx, o + q);
#pragma unroll
            for (int q = 0; q < STRIP + 1; ++q) y[q] = (double)d.at(ky, o + q);
#pragma unroll
            for (int q = 0; q < STRIP; ++q) {
                kx0[q] = d.west ? kx0[q] : 0.0;
                kx1[q] = dpp_shl1(kx0[q], kxe[o + q]);
            }
            f(d, s, kx0, kx1, y);
        }
    }
};

// A v on strip s of an R-row column v (above, vb: the rows above the strip and
// below the column; vh: the columns beyond lanes 0 and 63)
template <int R, typename T>
__device__ __forceinline__ void tall_op(int s, const T *v, double above, double vb, const double *vh,
                                        const double *kx0, const double *kx1, const double *ky, double *out)
{
    const int o = s * STRIP;
#pragma unroll
    for (int q = 0; q < STRIP; ++q) {
        const double c = (double)v[o + q];
        const double w = dpp_shr1(c, vh[o + q]), e = dpp_shl1(c, vh[o + q]);
        out[q] = opA(kx0[q], kx1[q], ky[q], ky[q + 1], c, w, e, q ? (double)v[o + q - 1] : above,
                     o + q < R - 1 ? (double)v[o + q + 1] : vb);
    }
}

// strip by strip: f's cells, zero outside the grid, to put(o, four values), or
// from get(o, four values), of the first M strips (-1: all). The barriers keep the loads of all strips from
// being in flight, and in registers, at once.
template <int M = -1, int NW, int S, typename T, typename F>
__device__ __forceinline__ void tall_load(const Tall<NW, S> &c, const T *f, F &&put)
{
    const Tall<NW, S> d = c.again();
#pragma unroll
    for (int o = 0; o < (M < 0 ? S : M) * STRIP; o += STRIP) {
        T v[STRIP];
        d.read4(f, o, v);
        put(o, v);
        if (o % (2 * STRIP)) __builtin_amdgcn_sched_barrier(0);
    }
}

template <int M = -1, int NW, int S, typename T, typename F>
__device__ __forceinline__ void tall_store(const Tall<NW, S> &c, T *f, F &&get)
{
    const Tall<NW, S> d = c.again();
#pragma unroll
    for (int o = 0; o < (M < 0 ? S : M) * STRIP; o += STRIP) {
        T v[STRIP];
        get(o, v);
        d.write4(f, o, v);
    }
}

// the border of a vector that every block has stored, fn(place): the row above
// (va) and below (vb); the columns go to vh (of LDS: [2][ROWS]), one row per
// lane
template <int NW, int S, int KEEP, typename F>
__device__ __forceinline__ void tall_border(const Ctx<NW, S, KEEP> &x, const Tall<NW, S> &c, const Geom &g,
                                            const Ext &e, double &va, double &vb, double (*vh)[NW * S * STRIP], F &&fn)
{
    constexpr int R = S * STRIP;
    const int j = c.i0 + (int)c.lo;
    va = vb = 0.0;
    if (c.col && c.rows && c.ks > e.k0) va = fn(j - c.P);
    if (c.col && c.rows == R && c.ks + R <= e.k1) vb = fn(j + R * c.P);
    const int jw = e.j0 + x.bx * TILE_X, row = x.lane % R;
    const bool open = x.lane < R ? jw > e.j0 : x.lane < 2 * R && jw + TILE_X - 1 < e.j1;
    double v = 0.0;
    if (open && row < c.rows) v = fn(IX(g, x.lane < R ? jw - 1 : jw + TILE_X, c.ks + row));
    if (x.lane < 2 * R) vh[x.lane >= R][x.wv * R + row] = v;
    wave_fence();
}

// Strips of r that a thread keeps in registers, as many as fit without a spill;
// the others' r is read and written in memory.
template <typename Stream>
constexpr int tall_cg_r(int prec, int S)
{
    if (prec == PREC_NONE || S < 6) return S;
    if (Stream::NARROW) return S < 8 || Stream::FIELDS == 1 ? S : prec == PREC_BLOCK ? 2 : 4;
    return S == 8 ? 0 : prec == PREC_BLOCK ? 4 : S;
}
template <typename Stream>
constexpr int tall_ppcg_r(int prec, int S, int sums)
{
    if (Stream::NARROW) return S < 8 || prec != PREC_BLOCK ? S : 6;
    return S < 6 ? S : S == 8 ? (prec != PREC_BLOCK) : prec == PREC_BLOCK ? 2 : sums == 1 ? S : 3;
}

// Preconditioned CG on tall blocks (the iterations of k_res_cg and of the
// refined solve's k_rf_res_cg): r (tall_cg_r), p and z in the storage type T in
// registers, the solution (or its increment) in LDS. A p is formed again in the second
// pass instead of kept: its faces are formed there anyway, for the
// preconditioner. The state's algebra is run, and a halt acted on, at the end
// of the iteration. St: the solver state; tail(pw, totals, st) its algebra;
// old_in_a(st): p_{n-1} is in pA when the launch starts; last_in_b(st): the last
// p belongs in pB when it ends.
template <typename T, int PREC, bool FAST, int NQ, int NW, int S, typename Stream, typename St, typename Tail,
          typename Old, typename Last>
__device__ __forceinline__ void tall_cg(const Geom &g, const Ext &e, const Comm &cm, T *u, T *r, T *z, T *pA, T *pB,
                                        const T *W, const T *Wy, const Faces &fc, St *gst, int iters, Tail &&tail,
                                        Old &&old_in_a, Last &&last_in_b)
{
    constexpr int R = S * STRIP;
    // strips of r in registers, the others in memory
    constexpr int RM = tall_cg_r<Stream>(PREC, S);
    __shared__ Shared<NW, S, 1> sh;
    __shared__ St st;
    __shared__ T ul[R][NW * 64];
    __shared__ double cwl[NW * R];
    Ctx<NW, S, 1> x(cm, sh);
    const int t = threadIdx.x;
    if (t == 0) {
        st = *gst;
        sh.fault = 0;
    }
    __syncthreads();
    const unsigned int closed = x.begin();
    if (st.halt) return;
    const Tall<NW, S> c(x, g, e);
    const Stream F(x, c, g, e, fc, W, Wy, cwl + x.wv * R);
    const T *src = PREC == PREC_NONE ? r : z, *p_old = old_in_a(st) ? pA : pB;
    T rv[(RM ? RM : 1) * STRIP], zv[PREC == PREC_NONE ? 1 : R], pv[R];
    double za, zb, pa, pb, pw[1], tot[NQ], *ph = x.side(0);
    double beta = uniform(st.beta), rro = uniform(st.rro);
    // beta == 0 (first iteration) ignores p_old entirely
    auto next = [&](double zz, double pp) { return (double)(T)(beta != 0.0 ? fma(beta, pp, zz) : zz); };
    // strips outside the grid never form their sums, nor their columns
    if (x.lane < S)
        for (int q = 0; q < NQ; ++q) sh.part[q][x.wv * S + x.lane] = 0.0;
    if (x.lane < R) sh.col[0][x.wv * R + x.lane] = sh.col[1][x.wv * R + x.lane] = 0.0;
    auto take = [](T *to) {
        return [to](int o, const T *v) {
#pragma unroll
            for (int q = 0; q < STRIP; ++q) to[o + q] = v[q];
        };
    };
    tall_load(c, u, [&](int o, const T *v) {
#pragma unroll
        for (int q = 0; q < STRIP; ++q) ul[o + q][t] = v[q];
    });
    tall_load<RM>(c, r, take(rv));
    tall_load(c, p_old, take(pv));
    if (PREC != PREC_NONE) tall_load(c, z, take(zv));
    tall_border(x, c, g, e, pa, pb, sh.side[0], [&](int i) { return next((double)src[i], (double)p_old[i]); });
    if (!x.begun(closed)) return;
    for (int it = 0;;) {
#pragma unroll
        for (int q = 0; q < R; ++q) pv[q] = (T)next((double)(PREC == PREC_NONE ? rv[q] : zv[q]), (double)pv[q]);
        F.pass(c, [&](const Tall<NW, S> &, int s, const double *kx0, const double *kx1, const double *ky) {
            double w[STRIP], acc = 0.0;
            tall_op<R>(s, pv, s ? (double)pv[s * STRIP - 1] : pa, pb, ph, kx0, kx1, ky, w);
#pragma unroll
            for (int q = 0; q < STRIP; ++q) acc = fma((double)pv[s * STRIP + q], w[q], acc);
            x.strip_sum(0, s, acc);
        });
        x.sum_begin();
        x.sum_end(pw);
        if (sh.fault) break;
        const double alpha = uniform(rro / pw[0]);
        double zfirst = 0.0, zlast = 0.0;
        F.pass(c, [&](const Tall<NW, S> &d, int s, const double *kx0, const double *kx1, const double *ky) {
            const int o = s * STRIP;
            double w[STRIP], rs[STRIP], zs[STRIP], a0 = 0.0, a1 = 0.0;
            T zq[STRIP], rq[STRIP], *rr = s < RM ? rv + o : rq;
            if (s >= RM) d.read4((const T *)r, o, rq);
            tall_op<R>(s, pv, s ? (double)pv[o - 1] : pa, pb, ph, kx0, kx1, ky, w);
#pragma unroll
            for (int q = 0; q < STRIP; ++q) {
                ul[o + q][t] = (T)fma(alpha, (double)pv[o + q], (double)ul[o + q][t]);
                rr[q] = (T)fma(-alpha, w[q], (double)rr[q]);
                rs[q] = (double)rr[q];
            }
            if (s >= RM) d.write4(r, o, rq);
            strip_precondition<PREC, FAST>(g, d.ks + o, 0, kx0, kx1, ky, rs, zs);
#pragma unroll
            for (int q = 0; q < STRIP; ++q) {
                zq[q] = (T)zs[q];
                a0 = fma(rs[q], (double)zq[q], a0);
                if (NQ > 1) a1 = fma(rs[q], rs[q], a1);
                if (PREC != PREC_NONE) zv[o + q] = zq[q];
            }
            if (x.ends())
#pragma unroll
                for (int q = 0; q < STRIP; ++q) sh.col[x.lane & 1][x.wv * R + o + q] = (double)zq[q];
            if (s == 0) zfirst = (double)zq[0];
            if (s == S - 1) zlast = (double)zq[STRIP - 1];
            x.strip_sum(0, s, a0);
            if (NQ > 1) x.strip_sum(NQ - 1, s, a1);
        });
        x.send(zfirst, zlast);
        x.sum_begin();
        x.template sum_end<true>(tot, za, zb);
        beta = uniform(tot[0] / rro);
        rro = uniform(tot[0]);
        if (t == TAIL_THREAD) tail(pw[0], tot, &st);
        __syncthreads();
        if (st.halt || sh.fault || ++it == iters) break;
        pa = next(za, pa);
        pb = next(zb, pb);
        // the columns beyond the block, one row per lane
        if (x.lane < 2 * R) {
            double *s = &sh.side[0][x.lane >= R][x.wv * R + x.lane % R];
            *s = next(sh.in[x.lane >= R][x.wv * R + x.lane % R], *s);
        }
        wave_fence();
    }
    if (sh.fault) return;
    auto give = [](const T *from) {
        return [from](int o, T *v) {
#pragma unroll
            for (int q = 0; q < STRIP; ++q) v[q] = from[o + q];
        };
    };
    tall_store(c, u, [&](int o, T *v) {
#pragma unroll
        for (int q = 0; q < STRIP; ++q) v[q] = ul[o + q][t];
    });
    tall_store<RM>(c, r, give(rv));
    if (PREC != PREC_NONE) tall_store(c, z, give(zv));
    tall_store(c, last_in_b(st) ? pB : pA, give(pv));
    if (blockIdx.x == 0 && t == 0) *gst = st;
}

// PPCG on tall blocks (the outer steps of k_res_ppcg and of the refined solve's
// k_rf_res_ppcg): r and, by turns in the same registers, p, the smoothing
// direction sd and z; the solution in LDS; p, and z where the smoothing does not
// renew it, in memory, each read once per outer step by the thread that wrote
// it. A strip's new direction takes the place of the old one at once: the strip
// below only needs its last row, kept in `up`. The state's algebra runs with the
// next outer step's p.w, as in k_res_ppcg.
template <typename T, int PREC, bool FAST, int NQ, int NW, int S, typename Stream, typename St, typename Tail>
__device__ __forceinline__ void tall_ppcg(const Geom &g, const Ext &e, const Comm &cm, T *u, T *r, T *z, T *pA, T *pB,
                                          const T *W, const T *Wy, const Faces &fc, const double *ch_a,
                                          const double *ch_b, int inner, bool fresh, St *gst, int iters, Tail &&tail)
{
    constexpr int R = S * STRIP;
    constexpr int RM = tall_ppcg_r<Stream>(PREC, S, NQ);
    __shared__ Shared<NW, S, 2> sh;
    __shared__ St st;
    __shared__ T ul[R][NW * 64];
    __shared__ double cwl[NW * R];
    Ctx<NW, S, 2> x(cm, sh);
    const int t = threadIdx.x;
    if (t == 0) {
        st = *gst;
        sh.fault = 0;
    }
    __syncthreads();
    const unsigned int closed = x.begin();
    if (st.halt) return;
    const Tall<NW, S> c(x, g, e);
    const Stream F(x, c, g, e, fc, W, Wy, cwl + x.wv * R);
    // z is that of the last smoothing step
    const bool renew = PREC == PREC_NONE || fresh;
    const T *src = PREC == PREC_NONE ? r : z;
    T rv[(RM ? RM : 1) * STRIP], v[R];
    double za, zb, pa, pb, sa, sb, pw[1], tot[NQ], *ph = x.side(0);
    double beta = uniform(st.beta), rro = uniform(st.rro);
    const double theta = uniform(st.theta);
    auto next = [&](double zz, double pp) { return (double)(T)(beta != 0.0 ? fma(beta, pp, zz) : zz); };
    int n = st.n;
    const T *p_old = (n & 1) ? pA : pB;
    if (x.lane < S)
        for (int q = 0; q < NQ; ++q) sh.part[q][x.wv * S + x.lane] = 0.0;
    if (x.lane < R) sh.col[0][x.wv * R + x.lane] = sh.col[1][x.wv * R + x.lane] = 0.0;
    auto take = [](T *to) {
        return [to](int o, const T *w) {
#pragma unroll
            for (int q = 0; q < STRIP; ++q) to[o + q] = w[q];
        };
    };
    // the columns of v to sh.col
    auto ends4 = [&](int o) {
        if (x.ends())
#pragma unroll
            for (int q = 0; q < STRIP; ++q) sh.col[x.lane & 1][x.wv * R + o + q] = (double)v[o + q];
    };
    tall_load(c, u, [&](int o, const T *w) {
#pragma unroll
        for (int q = 0; q < STRIP; ++q) ul[o + q][t] = w[q];
    });
    tall_load<RM>(c, r, take(rv));
    tall_load(c, src, take(v));
    tall_border(x, c, g, e, pa, pb, sh.side[0], [&](int i) { return next((double)src[i], (double)p_old[i]); });
    if (!x.begun(closed)) return;
    for (int it = 0;; ++it, ++n) {
        T *p_new = (n & 1) ? pB : pA;
        p_old = (n & 1) ? pA : pB;
        tall_load(c, p_old, [&](int o, const T *w) {
#pragma unroll
            for (int q = 0; q < STRIP; ++q) v[o + q] = (T)next((double)v[o + q], (double)w[q]);
        });
        F.pass(c, [&](const Tall<NW, S> &, int s, const double *kx0, const double *kx1, const double *ky) {
            double w[STRIP], acc = 0.0;
            tall_op<R>(s, v, s ? (double)v[s * STRIP - 1] : pa, pb, ph, kx0, kx1, ky, w);
#pragma unroll
            for (int q = 0; q < STRIP; ++q) acc = fma((double)v[s * STRIP + q], w[q], acc);
            x.strip_sum(0, s, acc);
        });
        x.sum_begin();
        if (it > 0 && t == TAIL_THREAD) tail(pw[0], tot, &st);
        x.sum_end(pw);
        if (st.halt || sh.fault || it == iters) break;
        const double alpha = uniform(rro / pw[0]);
        double up = pa, zfirst = 0.0, zlast = 0.0;
        F.pass(c, [&](const Tall<NW, S> &d, int s, const double *kx0, const double *kx1, const double *ky) {
            const int o = s * STRIP;
            double w[STRIP], rs[STRIP], zs[STRIP];
            T rq[STRIP], *rr = s < RM ? rv + o : rq;
            if (s >= RM) d.read4((const T *)r, o, rq);
            tall_op<R>(s, v, up, pb, ph, kx0, kx1, ky, w);
            up = (double)v[o + STRIP - 1];
#pragma unroll
            for (int q = 0; q < STRIP; ++q) {
                ul[o + q][t] = (T)fma(alpha, (double)v[o + q], (double)ul[o + q][t]);
                rr[q] = (T)fma(-alpha, w[q], (double)rr[q]);
                rs[q] = (double)rr[q];
            }
            if (s >= RM) d.write4(r, o, rq);
            d.write4(p_new, o, v + o);
            strip_precondition<PREC, FAST>(g, d.ks + o, 0, kx0, kx1, ky, rs, zs);
#pragma unroll
            for (int q = 0; q < STRIP; ++q) v[o + q] = (T)zs[q];
            if (!renew) d.write4(z, o, v + o);
            ends4(o);
            if (s == 0) zfirst = (double)v[0];
            if (s == S - 1) zlast = (double)v[R - 1];
#pragma unroll
            for (int q = 0; q < STRIP; ++q) v[o + q] = (T)((double)v[o + q] / theta);
        });
        x.send(zfirst, zlast);
        x.recv(za, zb, []() {});
        sa = (double)(T)(za / theta);
        sb = (double)(T)(zb / theta);
        if (x.lane < 2 * R) {
            double *in = &sh.in[x.lane >= R][x.wv * R + x.lane % R];
            sh.side[1][x.lane >= R][x.wv * R + x.lane % R] = *in;
            *in = (double)(T)(*in / theta);
        }
        wave_fence();
        for (int k = 0; k < inner; ++k) {
            const double ca = ch_a[k], cb = ch_b[k];
            const bool last = k == inner - 1;
            if (k) {
                x.send((double)v[0], (double)v[R - 1]);
                x.recv(sa, sb, []() {});
            }
            up = sa;
            F.pass(c, [&](const Tall<NW, S> &d, int s, const double *kx0, const double *kx1, const double *ky) {
                const int o = s * STRIP;
                double w[STRIP], rs[STRIP], zs[STRIP];
                T rq[STRIP], *rr = s < RM ? rv + o : rq;
                if (s >= RM) d.read4((const T *)r, o, rq);
                tall_op<R>(s, v, up, sb, x.in(), kx0, kx1, ky, w);
                up = (double)v[o + STRIP - 1];
#pragma unroll
                for (int q = 0; q < STRIP; ++q) {
                    ul[o + q][t] = (T)((double)ul[o + q][t] + (double)v[o + q]);
                    rr[q] = (T)((double)rr[q] - w[q]);
                    rs[q] = (double)rr[q];
                }
                if (s >= RM) d.write4(r, o, rq);
                strip_precondition<PREC, FAST>(g, d.ks + o, 0, kx0, kx1, ky, rs, zs);
                if (!last) {
                    // (the products' order as in the kernels of each solve)
#pragma unroll
                    for (int q = 0; q < STRIP; ++q) {
                        const double m = PREC == PREC_DIAG && NQ == 1
                                             ? cb * rs[q] * div_nr(1.0, diag_of(kx0[q], kx1[q], ky[q], ky[q + 1]))
                                             : cb * zs[q];
                        v[o + q] = (T)fma(ca, (double)v[o + q], m);
                    }
                } else {
                    if (!renew) {
                        d.read4((const T *)z, o, v + o);
                    } else {
#pragma unroll
                        for (int q = 0; q < STRIP; ++q) v[o + q] = (T)zs[q];
                        if (PREC != PREC_NONE) d.write4(z, o, v + o);
                    }
                    double a0 = 0.0, a1 = 0.0;
#pragma unroll
                    for (int q = 0; q < STRIP; ++q) {
                        a0 = fma(rs[q], (double)v[o + q], a0);
                        if (NQ > 1) a1 = fma(rs[q], rs[q], a1);
                    }
                    x.strip_sum(0, s, a0);
                    if (NQ > 1) x.strip_sum(NQ - 1, s, a1);
                }
                ends4(o);
            });
        }
        if (renew) x.send((double)v[0], (double)v[R - 1]);
        x.sum_begin();
        if (renew) x.template sum_end<true>(tot, za, zb);
        else x.sum_end(tot);
        beta = uniform(tot[0] / rro);
        rro = uniform(tot[0]);
        pa = next(za, pa);
        pb = next(zb, pb);
        if (x.lane < 2 * R) {
            const int i = x.wv * R + x.lane % R, side = x.lane >= R;
            sh.side[0][side][i] = next(renew ? sh.in[side][i] : sh.side[1][side][i], sh.side[0][side][i]);
        }
        wave_fence();
    }
    if (sh.fault) return;
    tall_store(c, u, [&](int o, T *w) {
#pragma unroll
        for (int q = 0; q < STRIP; ++q) w[q] = ul[o + q][t];
    });
    tall_store<RM>(c, r, [&](int o, T *w) {
#pragma unroll
        for (int q = 0; q < STRIP; ++q) w[q] = rv[o + q];
    });
    if (blockIdx.x == 0 && t == 0) *gst = st;
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

// iterations, or exchanges, per launch
constexpr int RES_ITERS = 1024;

// a launch's parameters: the exchange memory with fresh tags for at most
// `reds` sums and `halos` exchanges
Comm next_comm(tl_chunk *c, unsigned int reds, unsigned int halos);

// held from a launch to its end: each needs every block on the chunk's device at
// once
std::mutex &launch_mutex(const tl_chunk *c);

template <typename F, typename... A>
hipError_t coop(tl_chunk *c, F *kernel, const Comm &cm, int nw, A... args)
{
    void *p[] = {(void *)&args...};
    // (for tests: a block too few)
    const int grid = cm.nbx * cm.nby - (c->resident == -1);
    return hipLaunchCooperativeKernel((const void *)kernel, dim3(grid), dim3(nw * 64), p, 0, c->s);
}

// the kernel's form for the chunk's tile rows per block and preconditioner:
// K, or for tall blocks L, (preconditioner, wavefronts, strips per wavefront)
#define TL_RES_ROWS(K, L, P)                                                                            \
    (c->res_rows == 1   ? K(P, 4, 1)                                                                    \
     : c->res_rows == 2 ? K(P, 8, 1)                                                                    \
     : c->res_rows == 4 ? K(P, 8, 2)                                                                    \
     : c->res_rows == 8 ? L(P, 8, 4)                                                                    \
     : c->res_rows == 12 ? L(P, 8, 6) : L(P, 8, 8))
#define TL_RES_ANY(K, L)                                           \
    (c->prec == PREC_BLOCK  ? TL_RES_ROWS(K, L, PREC_BLOCK)        \
     : c->prec == PREC_DIAG ? TL_RES_ROWS(K, L, PREC_DIAG)         \
                            : TL_RES_ROWS(K, L, PREC_NONE))

}  // namespace res
}  // namespace tl
