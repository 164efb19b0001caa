// BiCGSTAB iteration with the multicolour symmetric Gauss-Seidel preconditioner on
// the sliced block layout (gfx950).
//
// Colours 0 .. k-1; D_c the diagonal blocks of a colour, A_cj its blocks with
// columns of colour j.  A preconditioned product is the sweep z = M^-1 y
//
//   forward    z_c = D_c^-1 (y_c - sum_{j<c} A_cj z_j)
//   backward   z_c = D_c^-1 (y_c - sum_{j!=c} A_cj z_j)        c = k-2 .. 0
//
// and A z.  Every block product, and the order of every sum, is that of the plain
// sweeps and product (kernels_sell.hip).  The first colour's backward step and its
// rows of A z need the same products A_0j z_j, of vectors that are final by then:
// k_first_colour forms them once for both.  Its forward step reads no off-diagonal block
// and is done where y is formed.  With two colours a preconditioned product reads the
// upper blocks once and the lower blocks twice, where sweeps and product apart read both
// twice.
//
// Not used: the identities of this preconditioner (Eisenstat's trick) by which A z =
// y + sum_{j<c} A_cj d_j with the backward sweep's corrections d, and A z = y in the first
// colour.  They halve the bytes again, but put y where the product has D z, so that the
// error of the 5x5 solve, large where a block's rows differ by orders of magnitude as at
// low Mach number, no longer enters the residual and is never corrected: the update was
// 3 times (plate, one iteration) to 22 times (SA bump, two) further from 80-bit floats.
//
// Bound: HBM.  2.1M-cell plate (256 x 64 x 128) in FP64, per preconditioned product:
// k_sell_sweep 320 us, k_first_colour 354 us, k_sell_spmv over the other colour 302 us
// (5.0-5.3 TB/s).  A BiCGSTAB iteration, against five lanes per row on row-major blocks:
// 2.1M cells FP64 3.63 -> 2.39 ms, BF16 1.73 -> 0.93 ms; 262,144 cells 474 -> 302 and 193 ->
// 118 us; 663,552 tetrahedra FP64 1.24 -> 0.89 ms; 93,765 cells FP64 162 -> 123 us; 3,072
// cells, twelve launches of latency, 65 -> 60 us.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <stdexcept>

#include "kernels.hpp"
#include "kernels_krylov.hpp"
#include "kernels_multicolour.hpp"
#include "kernels_sell_device.hpp"
#include "reduce_device.hpp"

namespace cfdg {

namespace {

constexpr int kBlock = kSellBlock;

// z = D^-1 y
template <class TV>
__device__ __forceinline__ void diagonal_solve(const Rows& q, TV y[5], const TV* lu, const std::uint16_t* piv, TV* z) {
    TV L[25];
    load_lu<TV, TV>(lu, q.slice, q.lane, L);
    lu_solve(y, L, piv[q.slice * kSellRows + q.lane]);
#pragma unroll
    for (int k = 0; k < 5; ++k) z[q.at + k * kSellRows] = y[k];
}

// r = r0 = p = src and the first colour's (slices [0, first)) forward solve
template <class TV>
__global__ void __launch_bounds__(kBlock) k_mc_start(SellArgs b, int first, const double* ks, const TV* src, TV* r,
                                                     TV* r0, TV* p, const TV* lu, const std::uint16_t* piv, TV* z) {
    if (ks[kKsStatus] != 0.0) return;
    const int slice = wave_slice<1>();
    if (slice >= b.nslices) return;
    const Rows q = rows_of(b, slice);
    if (!q.on) return;
    TV y[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        const long long e = q.at + k * kSellRows;
        y[k] = src[e];
        r[e] = y[k];
        r0[e] = y[k];
        p[e] = y[k];
    }
    if (slice < first) diagonal_solve(q, y, lu, piv, z);
}

// y = p (kOp 0) or s (kOp 1), and the first colour's forward solve
template <int kOp, class TV>
__global__ void __launch_bounds__(kBlock) k_mc_vec(SellArgs b, int first, const double* ks, const TV* r, const TV* v,
                                                   TV* y, const TV* lu, const std::uint16_t* piv, TV* z) {
    if (ks[kKsStatus] != 0.0) return;
    const int slice = wave_slice<1>();
    if (slice >= b.nslices) return;
    const Rows q = rows_of(b, slice);
    if (!q.on) return;
    TV s[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        const long long e = q.at + k * kSellRows;
        s[k] = (kOp == 0) ? p_entry(ks, r, v, y, e) : s_entry(ks, r, v, e);
        y[e] = s[k];
    }
    if (slice < first) diagonal_solve(q, s, lu, piv, z);
}

// The end of one iteration and the start of the next (k_xr_next, kernels_linalg.hip)
template <class TV>
__global__ void __launch_bounds__(kBlock) k_mc_xr_next(SellArgs b, int first, const double* ks_in, double* ks_out,
                                                       TV* ph, const TV* sh, const TV* sv, const TV* t, TV* x, TV* r,
                                                       const TV* v, TV* p, const TV* lu, const std::uint16_t* piv) {
    __shared__ double next[kNextCount];
    if (!next_iteration(ks_in, ks_out, next)) return;
    const int slice = wave_slice<1>();
    if (slice >= b.nslices) return;
    const Rows q = rows_of(b, slice);
    if (!q.on) return;
    const bool go = next[0] == 0.0;  // uniform over the grid
    TV s[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        const long long e = q.at + k * kSellRows;
        const TV rv = xr_entry(ks_in, ph, sh, sv, t, x, e);
        r[e] = rv;
        if (go) {
            s[k] = p_entry_of(next[1], next[2], next[3], rv, v, p, e);
            p[e] = s[k];
        }
    }
    if (go && slice < first) diagonal_solve(q, s, lu, piv, ph);
}

// The backward step of the first colour, z_0 = D_0^-1 (y_0 - sum A_0j z_j), and its rows
// of the product, out_0 = D_0 z_0 + sum A_0j z_j.  The products of a row's first kHeld
// blocks are held between the two sums, in registers (kSplit 1) or by the waves that share
// the slice in LDS; those of a cell with more faces are formed again.
constexpr int kSharedHeld = 8;
template <class TS, class TV, int kSplit, int kHeld>
__global__ void __launch_bounds__(slice_threads<kSplit>()) k_first_colour(SellArgs b, int count,
                                                                          const word_t<TS>* off,
                                                                          const word_t<TS>* diag, const TV* lu,
                                                                          const std::uint16_t* piv, const TV* y, TV* z,
                                                                          TV* out, const double* ks) {
    __shared__ TV lds[kSplit == 1 ? 1 : kHeld * 5 * kSellRows];
    if (ks[kKsStatus] != 0.0) return;
    const int ls = wave_slice<kSplit>();
    if (ls >= count) return;
    const Rows q = rows_of(b, ls);
    const bool lead = lead_wave<kSplit>() && q.on;
    const int blocks = q.blocks();  // all upper, so the slots are in column order
    const auto product = [&](int k, TV t[5]) { slot_times<TS, TV>(off, b.cols, q.sl.x + k, q.lane, z, t); };
    TV held[kSplit == 1 ? kHeld : 1][5], acc[5], L[25];
    if constexpr (kSplit == 1) {
        if (!lead) return;
#pragma unroll
        for (int k = 0; k < kHeld; ++k)
            if (k < blocks) product(k, held[k]);
    } else {
        for (int k = static_cast<int>(threadIdx.x >> 6); k < kHeld && k < q.sl.z; k += kSplit) {
            TV t[5];
            if (k < blocks) product(k, t);
#pragma unroll
            for (int v = 0; v < 5; ++v)
                if (k < blocks) lds[(k * 5 + v) * kSellRows + q.lane] = t[v];
        }
        if (lead) load_lu<TV, TV>(lu, q.slice, q.lane, L);  // in flight with the products
        __syncthreads();
        if (!lead) return;
    }
    // f(k, product k) in column order
    const auto each = [&](auto&& f) {
#pragma unroll
        for (int k = 0; k < kHeld; ++k) {
            if (k >= blocks) break;
            TV t[5];
#pragma unroll
            for (int v = 0; v < 5; ++v)
                t[v] = kSplit == 1 ? held[kSplit == 1 ? k : 0][v] : lds[kSplit == 1 ? 0 : (k * 5 + v) * kSellRows + q.lane];
            f(k, t);
        }
        for (int k = kHeld; k < blocks; ++k) {
            TV t[5];
            product(k, t);
            f(k, t);
        }
    };
#pragma unroll
    for (int v = 0; v < 5; ++v) acc[v] = y[q.at + v * kSellRows];
    each([&](int, const TV t[5]) {
#pragma unroll
        for (int v = 0; v < 5; ++v) acc[v] -= t[v];
    });
    if (kSplit == 1) load_lu<TV, TV>(lu, q.slice, q.lane, L);
    lu_solve(acc, L, piv[q.slice * kSellRows + q.lane]);
    const int before = b.before[q.slice * kSellRows + q.lane];
    TV d[5];
    diagonal_times<TS, TV>(diag, q, acc, d);
    RowSum<TV> sum;
    each([&](int k, const TV t[5]) { sum.add(k, t, before, d); });
    sum.finish(blocks, before, d);
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        z[q.at + v * kSellRows] = acc[v];
        out[q.at + v * kSellRows] = sum.s[v];
    }
}

template <class TS, class TV, int kS, int kHeld>
void launch_first_as(const SellArgs& b, const SellMatrix& m, int count, const TV* y, TV* z, TV* out, const double* ks,
                     hipStream_t s) {
    hipLaunchKernelGGL((k_first_colour<TS, TV, kS, kHeld>), slice_grid<kS>(count), dim3(slice_threads<kS>()), 0, s, b,
                       count, static_cast<const word_t<TS>*>(m.off), static_cast<const word_t<TS>*>(m.diag),
                       static_cast<const TV*>(m.lu), m.piv, y, z, out, ks);
}

}  // namespace

template <class T>
void launch_mc_start(const SellArgs& b, const SellMatrix& m, const int* cs, const T* src, const KrylovVecs<T>& w,
                     const double* ks, hipStream_t s) {
    hipLaunchKernelGGL(k_mc_start<T>, grid_for_slices(b.nslices), dim3(kBlock), 0, s, b, cs[1], ks, src, w.r, w.r0, w.p,
                       static_cast<const T*>(m.lu), m.piv, w.ph);
}

template <class T>
void launch_mc_vec(int op, const SellArgs& b, const SellMatrix& m, const int* cs, const KrylovVecs<T>& w,
                   const double* ks, hipStream_t s) {
    const dim3 g = grid_for_slices(b.nslices), blk(kBlock);
    const T* L = static_cast<const T*>(m.lu);
    if (op == 0)
        hipLaunchKernelGGL((k_mc_vec<0, T>), g, blk, 0, s, b, cs[1], ks, w.r, w.v, w.p, L, m.piv, w.ph);
    else
        hipLaunchKernelGGL((k_mc_vec<1, T>), g, blk, 0, s, b, cs[1], ks, w.r, w.v, w.s, L, m.piv, w.sh);
}

template <class T>
void launch_mc_xr_next(const SellArgs& b, const SellMatrix& m, const int* cs, const KrylovVecs<T>& w, T* x,
                       const double* ks_in, double* ks_out, hipStream_t s) {
    hipLaunchKernelGGL(k_mc_xr_next<T>, grid_for_slices(b.nslices), dim3(kBlock), 0, s, b, cs[1], ks_in, ks_out, w.ph,
                       w.sh, w.s, w.t, x, w.r, w.v, w.p, static_cast<const T*>(m.lu), m.piv);
}

template <class T>
void launch_mc_product(int op, const SellArgs& b, const SellMatrix& m, const int* cs, int colours,
                       int first_slots, const KrylovVecs<T>& w, double* partial, double* dots, double* ks, hipStream_t s) {
    const T* y = op == 0 ? w.p : w.s;
    T* z = op == 0 ? w.ph : w.sh;
    T* out = op == 0 ? w.v : w.t;
    for (int c = 1; c < colours; ++c) launch_sell_sweep<T>(b, m, cs[c], cs[c + 1] - cs[c], false, y, z, s, ks);
    for (int c = colours - 2; c >= 1; --c) launch_sell_sweep<T>(b, m, cs[c], cs[c + 1] - cs[c], true, y, z, s, ks);
    with_form<T>(m, [&](auto ts) {
        typedef decltype(ts) TS;
        with_split(cs[1], [&](auto split) {
            constexpr int kS = decltype(split)::value;
            if constexpr (kS > 1)
                launch_first_as<TS, T, kS, kSharedHeld>(b, m, cs[1], y, z, out, ks, s);
            else if (first_slots <= 4)  // tetrahedra
                launch_first_as<TS, T, 1, 4>(b, m, cs[1], y, z, out, ks, s);
            else
                launch_first_as<TS, T, 1, 6>(b, m, cs[1], y, z, out, ks, s);
        });
    });
    launch_sell_spmv<T>(b, m, cs[1], b.nslices - cs[1], z, out, s, ks);
    const int parts = op == 0 ? launch_sell_dots<T>(b, 1, w.r0, w.v, w.v, partial, s, ks)
                              : launch_sell_dots<T>(b, 5, w.t, w.s, w.r0, partial, s, ks);
    launch_reduce_step(parts, op == 0 ? 1 : 5, partial, dots, ks, op == 0 ? kStepAlpha : kStepOmega, s);
}

#define CFDG_MC(T)                                                                                                   \
    template void launch_mc_start<T>(const SellArgs&, const SellMatrix&, const int*, const T*, const KrylovVecs<T>&, \
                                     const double*, hipStream_t);                                                    \
    template void launch_mc_vec<T>(int, const SellArgs&, const SellMatrix&, const int*, const KrylovVecs<T>&,        \
                                   const double*, hipStream_t);                                                      \
    template void launch_mc_xr_next<T>(const SellArgs&, const SellMatrix&, const int*, const KrylovVecs<T>&, T*,     \
                                       const double*, double*, hipStream_t);                                         \
    template void launch_mc_product<T>(int, const SellArgs&, const SellMatrix&, const int*, int, int,            \
                                       const KrylovVecs<T>&, double*, double*, double*, hipStream_t);
CFDG_MC(double)
CFDG_MC(float)
#undef CFDG_MC

}  // namespace cfdg
