// Device functions of the BiCGSTAB recurrence shared by the Krylov kernels
// (kernels_linalg.hip, kernels_multicolour.hip): the scalar steps on the state block and
// the entry-wise vector updates.
#pragma once

#include <hip/hip_runtime.h>

#include "kernels_linalg.hpp"

namespace cfdg {

// Start of an iteration (bicgstab.cpp:97-109): iteration limit, it += 1,
// beta = (rho / rho_old)(alpha / omega) from the second iteration on.  Run
// at the end of the step before it (the start of the solve, or the end of the
// previous iteration), since nothing in between reads or writes the state.
__device__ inline void bicg_begin(double* ks) {
    if (ks[kKsIt] >= ks[kKsMaxIt]) {
        ks[kKsStatus] = kKsMaxIter;
        return;
    }
    ks[kKsIt] += 1.0;
    ks[kKsFirst] = (ks[kKsIt] == 1.0) ? 1.0 : 0.0;
    if (ks[kKsFirst] == 0.0) {
        const double beta = (ks[kKsRho] / ks[kKsRhoOld]) * (ks[kKsAlpha] / ks[kKsOmega]);
        if (!isfinite(beta)) {
            ks[kKsStatus] = kKsDiverged;
            return;
        }
        ks[kKsBeta] = beta;
        ks[kKsNbo] = -beta * ks[kKsOmega];
    }
}

// After x and r are updated (bicgstab.cpp:160-195): breakdown checks, the
// true residual norm when rr is given (every 32nd iteration), convergence;
// then the start of the next iteration.
__device__ inline void bicg_post(double* ks, const double* rr) {
    double rnorm = ks[kKsRnNew];
    const double omega_new = ks[kKsOmegaNew];
    ks[kKsRnorm] = rnorm;
    if (!isfinite(rnorm) || !isfinite(omega_new) || omega_new == 0.0) {
        ks[kKsStatus] = kKsDiverged;
        return;
    }
    if (rr) rnorm = sqrt(rr[0]);
    ks[kKsRnorm] = rnorm;
    if (rnorm <= ks[kKsTol]) {
        ks[kKsStatus] = kKsConverged;
        return;
    }
    const double rho_new = ks[kKsRhoNew];
    if (!isfinite(rho_new) || rho_new == 0.0) {
        ks[kKsStatus] = kKsDiverged;
        return;
    }
    ks[kKsRhoOld] = ks[kKsRho];
    ks[kKsRho] = rho_new;
    ks[kKsOmega] = omega_new;
    bicg_begin(ks);
}

// The end-of-iteration checks and the start of the next iteration inside a
// vector kernel: formed by thread 0 of every workgroup from the state ks_in
// alone, so every workgroup takes the same decision, workgroup 0 writing the
// result to ks_out; next (LDS) = status, first, beta, nbo of the next
// iteration.  False when the solve had ended before.
constexpr int kNextCount = 4;
__device__ __forceinline__ bool next_iteration(const double* ks_in, double* ks_out, double next[kNextCount]) {
    const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
    if (ks_in[kKsStatus] != 0.0) {  // ended before: carry the state over
        if (lead)
            for (int k = 0; k < kKsCount; ++k) ks_out[k] = ks_in[k];
        return false;
    }
    if (threadIdx.x == 0) {
        double st[kKsCount];
        for (int k = 0; k < kKsCount; ++k) st[k] = ks_in[k];
        bicg_post(st, nullptr);
        next[0] = st[kKsStatus];
        next[1] = st[kKsFirst];
        next[2] = st[kKsBeta];
        next[3] = st[kKsNbo];
        if (lead)
            for (int k = 0; k < kKsCount; ++k) ks_out[k] = st[k];
    }
    __syncthreads();
    return true;
}

// p = r on the first iteration, else p = ((p beta) + (-beta omega) v) + r
template <class T>
__device__ __forceinline__ T p_entry_of(double first, double beta, double nbo, T ri, const T* v, const T* p,
                                        long long i) {
    if (first != 0.0) return ri;
    T t = p[i] * static_cast<T>(beta);
    t += static_cast<T>(nbo) * v[i];
    t += static_cast<T>(1.0) * ri;
    return t;
}
template <class T>
__device__ __forceinline__ T p_entry(const double* ks, const T* r, const T* v, const T* p, long long i) {
    return p_entry_of(ks[kKsFirst], ks[kKsBeta], ks[kKsNbo], r[i], v, p, i);
}

// x = (x + alpha ph) + omega sh, written; returns r = s + (-omega) t
// (bicgstab.cpp:145-149)
template <class T>
__device__ __forceinline__ T xr_entry(const double* ks, const T* ph, const T* sh, const T* sv, const T* t, T* x,
                                      long long i) {
    const double alpha = ks[kKsAlpha], omega = ks[kKsOmegaNew];
    T xv = x[i];
    xv += static_cast<T>(alpha) * ph[i];
    xv += static_cast<T>(omega) * sh[i];
    x[i] = xv;
    T rv = sv[i];
    rv += static_cast<T>(-omega) * t[i];
    return rv;
}

// s = r + (-alpha) v
template <class T>
__device__ __forceinline__ T s_entry(const double* ks, const T* r, const T* v, long long i) {
    return r[i] + static_cast<T>(-ks[kKsAlpha]) * v[i];
}

}  // namespace cfdg
