// Launch wrappers of the multicolour BiCGSTAB iteration in its reduced form
// (kernels_reduced.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "kernels.hpp"
#include "kernels_linalg.hpp"
#include "kernels_sell.hpp"

namespace cfdg {

// The vectors of one reduced solve (sliced layout).  Of r, r0, p, v, s, t, ph
// and sh only the rows after the first colour are read or written (of r0 all rows
// are written, for the end of the solve); d holds a sweep's corrections of all
// colours but the last, g the first colour's part of the forward sweep.
template <class T>
struct RedVecs {
    T *r, *r0, *p, *v, *s, *t, *ph, *sh, *d, *g;
};

// After launch_bicg_init: g = A_{.0} D_0^-1 r_0 and r0 = r = src (the initial
// residual; src may be w.r).
template <class T>
void launch_red_start(const SellArgs& b, const SellMatrix& m, const int* colour_slice, const T* src,
                      const RedVecs<T>& w, const double* ks, hipStream_t s);
// y = p (op 0) or s (op 1), and the second colour's forward solve of z = M^-1 y
template <class T>
void launch_red_vec(int op, const SellArgs& b, const SellMatrix& m, const int* colour_slice, const RedVecs<T>& w,
                    const double* ks, hipStream_t s);
// the end of an iteration and launch_red_vec(0) of the next (launch_xr_next of
// kernels_linalg.hpp); x past the first colour
template <class T>
void launch_red_xr_next(const SellArgs& b, const SellMatrix& m, const int* colour_slice, const RedVecs<T>& w, T* x,
                        const double* ks_in, double* ks_out, hipStream_t s);
// v = A M^-1 p (op 0) or t = A M^-1 s (op 1) after launch_red_vec, then the dot
// products of the step and its scalars (kStepAlpha, kStepOmega)
template <class T>
void launch_red_product(int op, const SellArgs& b, const SellMatrix& m, const int* colour_slice, int colours,
                        const RedVecs<T>& w, double* partial, double* dots, double* ks, hipStream_t s);
// x of the first colour from the others at the end of a solve: D_0 x_0 = b_0 -
// r_0 - A_{0.} x
template <class T>
void launch_red_finish(const SellArgs& b, const SellMatrix& m, const int* colour_slice, const T* rhs,
                       const RedVecs<T>& w, T* x, const double* ks, hipStream_t s);

}  // namespace cfdg
