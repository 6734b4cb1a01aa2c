// Scalar algebra of the device-resident solver state: what the finisher of an
// iteration's reduction, or the resident solver (tl_resident.hip), does with
// the totals (tea_solve.f90:103-350).
#pragma once

#include <hip/hip_runtime.h>

#include "tl_common.h"

namespace tl {

// tea_solve.f90:322-331: error = SQRT(error), exit test, old_error, then the
// solver-switch test at the top of the next iteration (:151-165)
__device__ __forceinline__ void iteration_tail(SolveState *s, double *hist_e)
{
    s->error = sqrt(s->error);
    if (hist_e) hist_e[s->n] = s->error;
    if (fabs(s->error) < s->eps * s->initial_residual) {
        s->done = 1;
        s->halt = 1;
        s->exit_n = s->n;
        return;
    }
    s->old_error = s->error;
    if (s->n >= s->max_iters) {
        s->done = 1;
        s->halt = 1;
        s->exit_n = s->max_iters + 1;
        return;
    }
    s->n += 1;
    if (s->cheby_calc_steps == 0 && (s->solver == SOLVER_CHEBY || s->solver == SOLVER_PPCG)) {
        const bool sw = (!s->first && s->solver == SOLVER_PPCG && s->n > 1) ||
                        (fabs(s->old_error) <= s->epslim && s->n >= s->presteps);
        if (sw) {
            s->halt = 1;
            s->switch_n = s->n;
        }
    }
}

__device__ __forceinline__ bool cheby_norm_due(const SolveState *s)
{
    return s->n >= s->est_itc && (s->n % 10) == 0;
}

__device__ __forceinline__ void finish_results(const RedArgs &ra, const double *tot)
{
#pragma unroll
    for (int q = 0; q < MAX_RED; ++q) ra.result[q] = tot[q];
    // the release orders the totals before the flag for the host's reader
    if (ra.flag) __hip_atomic_store(ra.flag, ra.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The scalar algebra of the mode on s, a copy of the solver state in
// registers that the caller writes back
__device__ __forceinline__ void finish_state(const RedArgs &ra, const double *tot, SolveState *s)
{
    switch (ra.mode) {
    case RED_INIT_RESID:
        s->old_error = tot[0];
        s->initial_residual = sqrt(tot[0]);
        s->n = 1;
        break;
    case RED_INIT_RRO: {
        s->rro = tot[0];
        s->beta = 0.0;
        s->n = 1;
        if (s->solver == SOLVER_CHEBY || s->solver == SOLVER_PPCG) {
            const bool sw = fabs(s->old_error) <= s->epslim && s->n >= s->presteps;
            if (sw) {
                s->halt = 1;
                s->switch_n = 1;
            }
        }
        break;
    }
    case RED_CG_PW:
        s->pw = tot[0];
        s->alpha_prev = s->alpha;
        s->alpha = s->rro / s->pw;
        if (ra.hist_a) ra.hist_a[s->n] = s->alpha;
        break;
    case RED_CG_RRN:
        s->rrn = tot[0];
        s->beta = s->rrn / s->rro;
        if (ra.hist_b) ra.hist_b[s->n] = s->beta;
        s->error = s->rrn;
        s->rro = s->rrn;
        s->cg_calc_steps += 1;
        iteration_tail(s, ra.hist_e);
        break;
    case RED_PPCG_PW:
        s->pw = tot[0];
        s->alpha = s->rro / s->pw;
        break;
    case RED_PPCG_RRN:
        s->rrn = tot[0];
        s->beta = s->rrn / s->rro;
        s->error = s->rrn;
        s->rro = s->rrn;
        s->cheby_calc_steps += 1;
        iteration_tail(s, ra.hist_e);
        break;
    case RED_JACOBI:
        s->error = tot[0];
        iteration_tail(s, ra.hist_e);
        break;
    case RED_CHEBY:
        if (cheby_norm_due(s)) s->error = tot[0];
        s->cheby_calc_steps += 1;
        iteration_tail(s, ra.hist_e);
        break;
    case RED_CHEBY2:
        // two iterations; the first (odd n) never forms the norm
        s->cheby_calc_steps += 1;
        iteration_tail(s, ra.hist_e);
        if (s->halt) break;
        if (cheby_norm_due(s)) s->error = tot[0];
        s->cheby_calc_steps += 1;
        iteration_tail(s, ra.hist_e);
        break;
    case RED_EXACT:
        s->exact_error = sqrt(tot[0]);
        break;
    default:
        break;
    }
}

__device__ __forceinline__ bool iteration_mode(int mode)
{
    return mode == RED_CG_PW || mode == RED_CG_RRN || mode == RED_PPCG_PW || mode == RED_PPCG_RRN ||
           mode == RED_JACOBI || mode == RED_CHEBY || mode == RED_CHEBY2;
}

}  // namespace tl
