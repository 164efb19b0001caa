// Launch wrappers of the BiCGSTAB iteration with the multicolour symmetric
// Gauss-Seidel preconditioner (kernels_multicolour.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "kernels.hpp"
#include "kernels_linalg.hpp"
#include "kernels_sell.hpp"

namespace cfdg {

// The vectors of one solve.
template <class T>
struct KrylovVecs {
    T *r, *r0, *p, *v, *s, *t, *ph, *sh;
};

// Start of a solve after launch_bicg_start: r = r0 = p = src (src may be w.r), and the
// first colour's forward solve of ph = M^-1 p.
template <class T>
void launch_mc_start(const SellArgs& b, const SellMatrix& m, const int* colour_slice, const T* src,
                     const KrylovVecs<T>& w, const double* ks, hipStream_t s);
// y = p (op 0) or s (op 1), and the first colour's forward solve of z = M^-1 y
template <class T>
void launch_mc_vec(int op, const SellArgs& b, const SellMatrix& m, const int* colour_slice, const KrylovVecs<T>& w,
                   const double* ks, hipStream_t s);
// the end of an iteration and launch_mc_vec(0) of the next (launch_xr_next of
// kernels_linalg.hpp)
template <class T>
void launch_mc_xr_next(const SellArgs& b, const SellMatrix& m, const int* colour_slice, const KrylovVecs<T>& w, T* x,
                       const double* ks_in, double* ks_out, hipStream_t s);
// v = A M^-1 p (op 0) or t = A M^-1 s (op 1) after launch_mc_vec, then the dot
// products of the step and its scalars (kStepAlpha, kStepOmega); first_slots: the most
// slots of a slice of the first colour
template <class T>
void launch_mc_product(int op, const SellArgs& b, const SellMatrix& m, const int* colour_slice, int colours,
                       int first_slots, const KrylovVecs<T>& w, double* partial, double* dots, double* ks, hipStream_t s);

}  // namespace cfdg
