// BiCGSTAB with the multicolour symmetric Gauss-Seidel preconditioner, on the
// sliced block layout, without the work that the preconditioner makes redundant.
//
// Colours 0 .. k-1; D_c the diagonal blocks of a colour, A_cj its blocks with
// columns of colour j.  z = M^-1 y is the sweep
//
//   forward    z'_c = D_c^-1 (y_c - sum_{j<c} A_cj z'_j)
//   backward   z_c  = D_c^-1 (y_c - sum_{j<c} A_cj z'_j - sum_{j>c} A_cj z_j)
//
// so that with d = z - z' (zero in the last colour)
//
//   (1)  d_c = - D_c^-1 sum_{j>c} A_cj z_j            no lower block is read again
//   (2)  (A z)_c = y_c + sum_{j<c} A_cj d_j           the product reads lower blocks only
//
// (2) gives (A z)_0 = y_0: in the first colour v = p and t = s, and every vector
// of the recurrence is a multiple of the initial residual r0 there, r_0 = a_r r0_0,
// p_0 = a_p r0_0, s_0 = a_s r0_0.  Three scalars of the state block and b0 =
// |r0_0|^2 stand for the first colour in all vector updates and dot products, and
// its part of the forward sweep is a_y g with g_c = A_c0 D_0^-1 r0_0 formed once per
// solve.  x_0 follows from the first block row of A x = b - r at the end.
//
// The sums are the preconditioned product's own, so the iterates are those of
// k_sell_sweep / k_sell_spmv up to rounding.  Rounding: the product of the
// rounded z and (2) differ by the residual of the 5x5 solves, a few eps |D| |z|,
// which is the size of the rounding of the product itself; relative error of
// the caller's system of 156,849 cells solved to 1e-8 against 64 bits 2.3e-8 both
// ways (the tolerance, not the rounding).
//
// Bound: HBM.  With two colours a preconditioned product reads the off-diagonal
// blocks once (upper of the first colour, lower of the second) and no diagonal
// block, where sweeps and product read them twice and the diagonal blocks once;
// with four (tetrahedra) the lower blocks once without, once with the first
// colour's columns, the upper blocks once.  2.1M-cell plate (256 x 64 x 128) in FP64:
// a backward step 315 us and a product with its dot products 287 us, 5.2-5.4 TB/s
// (a reduction that only reads reaches 6.0); a BiCGSTAB iteration 2.36 -> 1.20 ms, at
// 262,144 cells FP64 0.33 -> 0.18 ms, BF16 0.126 -> 0.070 ms.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <stdexcept>

#include "kernels.hpp"
#include "kernels_krylov.hpp"
#include "kernels_reduced.hpp"
#include "kernels_sell_device.hpp"
#include "reduce_device.hpp"

namespace cfdg {

namespace {

constexpr int kBlock = kSellBlock;

// A wave's slice: rows at component 0, whether the lane holds a row, its blocks.
struct Rows {
    int slice, lane;
    int4 sl;
    bool on;
    unsigned n;
    long long at;
};
__device__ __forceinline__ Rows rows_of(const SellArgs& b, int slice) {
    Rows q;
    q.slice = slice;
    q.lane = threadIdx.x & (kSellRows - 1);
    q.sl = b.slice[slice];
    q.on = q.lane < q.sl.w;
    q.n = q.on ? b.count[slice * kSellRows + q.lane] : 0;
    q.at = static_cast<long long>(slice) * (5 * kSellRows) + q.lane;
    return q;
}
__device__ __forceinline__ int first_lower(const SellArgs& b, const Rows& q) {
    return q.on ? static_cast<int>(b.lower0[q.slice * kSellRows + q.lane]) : 0;
}
template <int kSplit>
__device__ __forceinline__ bool lead_wave() {
    return kSplit == 1 || threadIdx.x < kSellRows;
}

// r0_0 = src_0 and d_0 = D_0^-1 src_0
template <class TV>
__global__ void __launch_bounds__(kBlock) k_red_start(SellArgs b, int count, const TV* src, TV* r0, TV* d,
                                                      const TV* lu, const std::uint16_t* piv, const double* ks) {
    if (ks[kKsStatus] != 0.0) return;
    const int slice = wave_slice<1>();
    if (slice >= count) return;
    const Rows q = rows_of(b, slice);
    if (!q.on) return;
    TV s[5], L[25];
    load_lu<TV, TV>(lu, slice, q.lane, L);
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        s[k] = src[q.at + k * kSellRows];
        r0[q.at + k * kSellRows] = s[k];
    }
    lu_solve(s, L, piv[slice * kSellRows + q.lane]);
#pragma unroll
    for (int k = 0; k < 5; ++k) d[q.at + k * kSellRows] = s[k];
}

// g_c = A_c0 d_0 and r0 = r = src in the rows after the first colour
template <class TS, class TV, int kSplit>
__global__ void __launch_bounds__(slice_threads<kSplit>()) k_red_g(SellArgs b, int first, int count,
                                                                   const word_t<TS>* off, const TV* d, const TV* src,
                                                                   TV* r, TV* r0, TV* g, const double* ks) {
    __shared__ TV lds[split_lds<kSplit, TV>()];
    if (ks[kKsStatus] != 0.0) return;
    const int ls = wave_slice<kSplit>();
    if (ls >= count) return;
    Rows q = rows_of(b, first + ls);
    // the row's lower blocks of the first colour come first
    q.n = static_cast<unsigned>(first_lower(b, q));
    TV acc[5] = {0, 0, 0, 0, 0};
    for_slots<kSplit, TS, TV>(off, b.cols, q.sl, q.n, 0, q.sl.y, 0, q.lane, d, lds, [&](const TV t[5]) {
#pragma unroll
        for (int k = 0; k < 5; ++k) acc[k] += t[k];
    });
    if (!lead_wave<kSplit>() || !q.on) return;
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        const long long e = q.at + k * kSellRows;
        const TV rv = src[e];
        g[e] = acc[k];
        r[e] = rv;
        r0[e] = rv;
    }
}

// z = D^-1 (y - a g) for a row whose lower blocks are all of the first colour
template <class TV>
__device__ __forceinline__ void second_colour_solve(const Rows& q, const TV y[5], double a, const TV* g, const TV* lu,
                                                    const std::uint16_t* piv, TV* z) {
    TV s[5], L[25];
    load_lu<TV, TV>(lu, q.slice, q.lane, L);
#pragma unroll
    for (int k = 0; k < 5; ++k) s[k] = y[k] - static_cast<TV>(a) * g[q.at + k * kSellRows];
    lu_solve(s, L, piv[q.slice * kSellRows + q.lane]);
#pragma unroll
    for (int k = 0; k < 5; ++k) z[q.at + k * kSellRows] = s[k];
}

// y = p (kOp 0) or s (kOp 1) in the rows after the first colour, and the second
// colour's (slices [first, second)) forward solve.
template <int kOp, class TV>
__global__ void __launch_bounds__(kBlock) k_red_vec(SellArgs b, int first, int second, const double* ks, const TV* r,
                                                    const TV* v, const TV* g, TV* y, const TV* lu,
                                                    const std::uint16_t* piv, TV* z) {
    if (ks[kKsStatus] != 0.0) return;
    const int slice = first + wave_slice<1>();
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
    if (slice < second) second_colour_solve(q, s, ks[kOp == 0 ? kKsAp : kKsAs], g, lu, piv, z);
}

// The end of one iteration and the start of the next (k_xr_next, kernels_linalg.hip)
template <class TV>
__global__ void __launch_bounds__(kBlock) k_red_xr_next(SellArgs b, int first, int second, const double* ks_in,
                                                        double* ks_out, TV* ph, const TV* sh, const TV* sv,
                                                        const TV* t, TV* x, TV* r, const TV* v, const TV* g, TV* p,
                                                        const TV* lu, const std::uint16_t* piv) {
    __shared__ double next[kNextCount];
    if (!next_iteration(ks_in, ks_out, next)) return;
    const int slice = first + wave_slice<1>();
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
    if (go && slice < second) second_colour_solve(q, s, next[4], g, lu, piv, ph);
}

// Forward sweep of a colour after the second: z = D^-1 (y - a g - sum A z over the
// lower blocks that g does not hold).
template <class TS, class TV, int kSplit>
__global__ void __launch_bounds__(slice_threads<kSplit>()) k_red_forward(SellArgs b, int first, int count, int scalar,
                                                                         const word_t<TS>* off, const TV* lu,
                                                                         const std::uint16_t* piv, const TV* y,
                                                                         const TV* g, TV* z, const double* ks) {
    __shared__ TV lds[split_lds<kSplit, TV>()];
    if (ks[kKsStatus] != 0.0) return;
    const int ls = wave_slice<kSplit>();
    if (ls >= count) return;
    const Rows q = rows_of(b, first + ls);
    const int skip = first_lower(b, q);
    const bool lead = lead_wave<kSplit>() && q.on;
    TV acc[5], L[25];
    if (lead) {
        const TV a = static_cast<TV>(ks[scalar]);
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            const long long e = q.at + k * kSellRows;
            acc[k] = y[e] - a * g[e];
        }
        if (kSplit > 1) load_lu<TV, TV>(lu, q.slice, q.lane, L);  // in flight with the slots
    }
    for_slots<kSplit, TS, TV>(off, b.cols, q.sl, q.n, 0, q.sl.y, skip, q.lane, z, lds, [&](const TV t[5]) {
#pragma unroll
        for (int k = 0; k < 5; ++k) acc[k] -= t[k];
    });
    if (!lead) return;
    if (kSplit == 1) load_lu<TV, TV>(lu, q.slice, q.lane, L);
    lu_solve(acc, L, piv[q.slice * kSellRows + q.lane]);
#pragma unroll
    for (int k = 0; k < 5; ++k) z[q.at + k * kSellRows] = acc[k];
}

// Backward sweep of a colour, (1): d = -D^-1 sum A z over the upper blocks, and
// past the first colour z += d.
template <class TS, class TV, int kSplit>
__global__ void __launch_bounds__(slice_threads<kSplit>()) k_red_backward(SellArgs b, int first, int count,
                                                                          const word_t<TS>* off, const TV* lu,
                                                                          const std::uint16_t* piv, TV* z, TV* d,
                                                                          int update, const double* ks) {
    __shared__ TV lds[split_lds<kSplit, TV>()];
    if (ks[kKsStatus] != 0.0) return;
    const int ls = wave_slice<kSplit>();
    if (ls >= count) return;
    const Rows q = rows_of(b, first + ls);
    const bool lead = lead_wave<kSplit>() && q.on;
    TV acc[5] = {0, 0, 0, 0, 0}, L[25];
    if (kSplit > 1 && lead) load_lu<TV, TV>(lu, q.slice, q.lane, L);
    for_slots<kSplit, TS, TV>(off, b.cols, q.sl, q.n, q.sl.y, q.sl.y + q.sl.z, 0, q.lane, z, lds, [&](const TV t[5]) {
#pragma unroll
        for (int k = 0; k < 5; ++k) acc[k] -= t[k];
    });
    if (!lead) return;
    if (kSplit == 1) load_lu<TV, TV>(lu, q.slice, q.lane, L);
    lu_solve(acc, L, piv[q.slice * kSellRows + q.lane]);
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        const long long e = q.at + k * kSellRows;
        d[e] = acc[k];
        if (update) z[e] += acc[k];
    }
}

// The product, (2), with the dot products of its step: v and (r0, v) (kOp 0), or
// t and (t,t), (t,s), (r0,t), (r0,s), (s,s) (kOp 1), whose operands are in
// registers but for r0.  A workgroup takes a run of slices (kSplit 1) or one
// (kSplit 8) and leaves its partial sums, in a fixed order.
template <int kOp, class TS, class TV, int kSplit>
__global__ void __launch_bounds__(slice_threads<kSplit>()) k_red_product(SellArgs b, int first, int count,
                                                                         const word_t<TS>* off, const TV* d,
                                                                         const TV* y, const TV* r0, TV* out,
                                                                         double* partial, const double* ks) {
    constexpr int kDots = kOp == 0 ? 1 : 5;
    __shared__ TV lds[split_lds<kSplit, TV>()];
    if (ks[kKsStatus] != 0.0) return;
    const int blk = xcd_block(blockIdx.x, gridDim.x);
    double dot[kDots];
#pragma unroll
    for (int j = 0; j < kDots; ++j) dot[j] = 0.0;
    const auto slice_product = [&](int slice) {
        const Rows q = rows_of(b, slice);
        const bool lead = lead_wave<kSplit>() && q.on;
        TV acc[5], yv[5], rv[5];
        if (lead) {
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                yv[k] = y[q.at + k * kSellRows];
                rv[k] = r0[q.at + k * kSellRows];
                acc[k] = yv[k];
            }
        }
        for_slots<kSplit, TS, TV>(off, b.cols, q.sl, q.n, 0, q.sl.y, 0, q.lane, d, lds, [&](const TV t[5]) {
#pragma unroll
            for (int k = 0; k < 5; ++k) acc[k] += t[k];
        });
        if (!lead) return;
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            out[q.at + k * kSellRows] = acc[k];
            const double a = static_cast<double>(acc[k]), r = static_cast<double>(rv[k]);
            if constexpr (kOp == 0) {
                dot[0] += r * a;
            } else {
                const double s = static_cast<double>(yv[k]);
                dot[0] += a * a;
                dot[1] += a * s;
                dot[2] += r * a;
                dot[3] += r * s;
                dot[4] += s * s;
            }
        }
    };
    if constexpr (kSplit == 1) {
        const int lo = static_cast<int>(static_cast<long long>(count) * blk / gridDim.x);
        const int hi = static_cast<int>(static_cast<long long>(count) * (blk + 1) / gridDim.x);
        for (int s = lo + static_cast<int>(threadIdx.x >> 6); s < hi; s += kBlockSlices) slice_product(first + s);
        __shared__ double sums[kBlockSlices * kDots];
#pragma unroll
        for (int j = 0; j < kDots; ++j) {
            const double s = wave_sum(dot[j]);
            if ((threadIdx.x & 63) == 0) sums[(threadIdx.x >> 6) * kDots + j] = s;
        }
        __syncthreads();
        if (threadIdx.x < kDots) {
            double s = 0.0;
            for (int w = 0; w < kBlockSlices; ++w) s += sums[w * kDots + static_cast<int>(threadIdx.x)];
            partial[blk * 5 + static_cast<int>(threadIdx.x)] = s;
        }
    } else {
        slice_product(first + blk);
        if (threadIdx.x >= kSellRows) return;
#pragma unroll
        for (int j = 0; j < kDots; ++j) {
            const double s = wave_sum(dot[j]);
            if (threadIdx.x == 0) partial[blk * 5 + j] = s;
        }
    }
}

// D_0 x_0 = rhs_0 - a_r r0_0 - A_{0.} x; x as it is when no iteration was done.
template <class TS, class TV, int kSplit>
__global__ void __launch_bounds__(slice_threads<kSplit>()) k_red_finish(SellArgs b, int count, const word_t<TS>* off,
                                                                        const TV* lu, const std::uint16_t* piv,
                                                                        const TV* rhs, const TV* r0, TV* x,
                                                                        const double* ks) {
    __shared__ TV lds[split_lds<kSplit, TV>()];
    if (ks[kKsIt] == 0.0) return;
    const int ls = wave_slice<kSplit>();
    if (ls >= count) return;
    const Rows q = rows_of(b, ls);
    const bool lead = lead_wave<kSplit>() && q.on;
    TV acc[5], L[25];
    if (lead) {
        const TV a = static_cast<TV>(ks[kKsAr]);
#pragma unroll
        for (int k = 0; k < 5; ++k) acc[k] = rhs[q.at + k * kSellRows] - a * r0[q.at + k * kSellRows];
        if (kSplit > 1) load_lu<TV, TV>(lu, q.slice, q.lane, L);
    }
    for_slots<kSplit, TS, TV>(off, b.cols, q.sl, q.n, q.sl.y, q.sl.y + q.sl.z, 0, q.lane, x, lds, [&](const TV t[5]) {
#pragma unroll
        for (int k = 0; k < 5; ++k) acc[k] -= t[k];
    });
    if (!lead) return;
    if (kSplit == 1) load_lu<TV, TV>(lu, q.slice, q.lane, L);
    lu_solve(acc, L, piv[q.slice * kSellRows + q.lane]);
#pragma unroll
    for (int k = 0; k < 5; ++k) x[q.at + k * kSellRows] = acc[k];
}

// f(storage type, waves per slice) for a launch over that many slices; the LU
// type follows the vector type, FP64 vectors only with FP64 blocks.
template <class TV, class F>
void with_form(const SellMatrix& m, int slices, F&& f) {
    with_split(slices, [&](auto split) {
        if constexpr (sizeof(TV) == sizeof(double)) {
            if (m.storage != kStoreF64) throw std::invalid_argument("FP64 SGS needs FP64 blocks");
            f(double{}, split);
        } else {
            with_storage(m.storage, [&](auto ts) { f(ts, split); });
        }
    });
}

template <class TS>
const word_t<TS>* words(const void* p) {
    return static_cast<const word_t<TS>*>(p);
}

}  // namespace

template <class T>
void launch_red_start(const SellArgs& b, const SellMatrix& m, const int* cs, const T* src, const RedVecs<T>& w,
                      const double* ks, hipStream_t s) {
    hipLaunchKernelGGL(k_red_start<T>, grid_for_slices(cs[1]), dim3(kBlock), 0, s, b, cs[1], src, w.r0, w.d,
                       static_cast<const T*>(m.lu), m.piv, ks);
    const int rest = b.nslices - cs[1];
    with_form<T>(m, rest, [&](auto ts, auto split) {
        typedef decltype(ts) TS;
        constexpr int kS = decltype(split)::value;
        hipLaunchKernelGGL((k_red_g<TS, T, kS>), slice_grid<kS>(rest), dim3(slice_threads<kS>()), 0, s, b, cs[1], rest,
                           words<TS>(m.off), w.d, src, w.r, w.r0, w.g, ks);
    });
}

template <class T>
void launch_red_vec(int op, const SellArgs& b, const SellMatrix& m, const int* cs, const RedVecs<T>& w,
                    const double* ks, hipStream_t s) {
    const dim3 g = grid_for_slices(b.nslices - cs[1]), blk(kBlock);
    const T* L = static_cast<const T*>(m.lu);
    if (op == 0)
        hipLaunchKernelGGL((k_red_vec<0, T>), g, blk, 0, s, b, cs[1], cs[2], ks, w.r, w.v, w.g, w.p, L, m.piv, w.ph);
    else
        hipLaunchKernelGGL((k_red_vec<1, T>), g, blk, 0, s, b, cs[1], cs[2], ks, w.r, w.v, w.g, w.s, L, m.piv, w.sh);
}

template <class T>
void launch_red_xr_next(const SellArgs& b, const SellMatrix& m, const int* cs, const RedVecs<T>& w, T* x,
                        const double* ks_in, double* ks_out, hipStream_t s) {
    hipLaunchKernelGGL(k_red_xr_next<T>, grid_for_slices(b.nslices - cs[1]), dim3(kBlock), 0, s, b, cs[1], cs[2], ks_in,
                       ks_out, w.ph, w.sh, w.s, w.t, x, w.r, w.v, w.g, w.p, static_cast<const T*>(m.lu), m.piv);
}

template <class T>
void launch_red_product(int op, const SellArgs& b, const SellMatrix& m, const int* cs, int colours,
                        const RedVecs<T>& w, double* partial, double* dots, double* ks, hipStream_t s) {
    const T* y = op == 0 ? w.p : w.s;
    T* z = op == 0 ? w.ph : w.sh;
    T* out = op == 0 ? w.v : w.t;
    const T* L = static_cast<const T*>(m.lu);
    for (int c = 2; c < colours; ++c) {
        const int n = cs[c + 1] - cs[c];
        with_form<T>(m, n, [&](auto ts, auto split) {
            typedef decltype(ts) TS;
            constexpr int kS = decltype(split)::value;
            hipLaunchKernelGGL((k_red_forward<TS, T, kS>), slice_grid<kS>(n), dim3(slice_threads<kS>()), 0, s, b,
                               cs[c], n, op == 0 ? kKsAp : kKsAs, words<TS>(m.off), L, m.piv, y, w.g, z, ks);
        });
    }
    for (int c = colours - 2; c >= 0; --c) {
        const int n = cs[c + 1] - cs[c];
        with_form<T>(m, n, [&](auto ts, auto split) {
            typedef decltype(ts) TS;
            constexpr int kS = decltype(split)::value;
            hipLaunchKernelGGL((k_red_backward<TS, T, kS>), slice_grid<kS>(n), dim3(slice_threads<kS>()), 0, s, b,
                               cs[c], n, words<TS>(m.off), L, m.piv, z, w.d, c > 0 ? 1 : 0, ks);
        });
    }
    const int rest = b.nslices - cs[1];
    int parts = 0;
    with_form<T>(m, rest, [&](auto ts, auto split) {
        typedef decltype(ts) TS;
        constexpr int kS = decltype(split)::value;
        const int runs = (rest + kBlockSlices - 1) / kBlockSlices;
        parts = kS > 1 ? rest : (runs < kReduceBlocks ? runs : kReduceBlocks);
        const dim3 g(static_cast<unsigned>(parts)), blk(slice_threads<kS>());
        if (op == 0)
            hipLaunchKernelGGL((k_red_product<0, TS, T, kS>), g, blk, 0, s, b, cs[1], rest, words<TS>(m.off), w.d, y,
                               w.r0, out, partial, ks);
        else
            hipLaunchKernelGGL((k_red_product<1, TS, T, kS>), g, blk, 0, s, b, cs[1], rest, words<TS>(m.off), w.d, y,
                               w.r0, out, partial, ks);
    });
    launch_reduce_step(parts, op == 0 ? 1 : 5, partial, dots, ks, op == 0 ? kStepAlpha : kStepOmega, s);
}

template <class T>
void launch_red_finish(const SellArgs& b, const SellMatrix& m, const int* cs, const T* rhs, const RedVecs<T>& w, T* x,
                       const double* ks, hipStream_t s) {
    with_form<T>(m, cs[1], [&](auto ts, auto split) {
        typedef decltype(ts) TS;
        constexpr int kS = decltype(split)::value;
        hipLaunchKernelGGL((k_red_finish<TS, T, kS>), slice_grid<kS>(cs[1]), dim3(slice_threads<kS>()), 0, s, b, cs[1],
                           words<TS>(m.off), static_cast<const T*>(m.lu), m.piv, rhs, w.r0, x, ks);
    });
}

#define CFDG_RED(T)                                                                                                    \
    template void launch_red_start<T>(const SellArgs&, const SellMatrix&, const int*, const T*, const RedVecs<T>&,     \
                                      const double*, hipStream_t);                                                     \
    template void launch_red_vec<T>(int, const SellArgs&, const SellMatrix&, const int*, const RedVecs<T>&,            \
                                    const double*, hipStream_t);                                                       \
    template void launch_red_xr_next<T>(const SellArgs&, const SellMatrix&, const int*, const RedVecs<T>&, T*,         \
                                        const double*, double*, hipStream_t);                                          \
    template void launch_red_product<T>(int, const SellArgs&, const SellMatrix&, const int*, int, const RedVecs<T>&,   \
                                        double*, double*, double*, hipStream_t);                                       \
    template void launch_red_finish<T>(const SellArgs&, const SellMatrix&, const int*, const T*, const RedVecs<T>&,    \
                                       T*, const double*, hipStream_t);
CFDG_RED(double)
CFDG_RED(float)
#undef CFDG_RED

}  // namespace cfdg
