// Multicolour Krylov kernels on the sliced block layout (gfx950).
//
// A wave takes one slice: 64 rows of one colour, a row per lane.  Entry e of
// the lanes' blocks in a slot is one run of 64 values, so every load of a
// block entry is one contiguous 512-byte (FP64), 256-byte (FP32, and two BF16
// entries per word) request of the wave, the rows of a colour are contiguous,
// and a sweep reads no block, factor or vector line it does not use.
//
//   k_sell_lu      diagonal-block LU with partial pivoting (bsr_helpers.hpp:278-321)
//   k_sell_spmv    y = A x
//   k_sell_sweep   one Gauss-Seidel step of a colour (bsr_helpers.hpp:390-435)
//
// with the vector kernels and sums of a solve's start and end.  The iterations of the
// solve have some more (kernels_multicolour.hip).
//
// Arithmetic per row component: products summed over the block's columns, the
// block sums added or subtracted in ascending mesh column, as on a row-major matrix;
// sums over the vectors in the order of the device rows, 5 values each
// (flat_dots).  Both are those of kernels_linalg.hip, so a solve's result does not
// depend on the layout: a loosely converged solve magnifies rounding, and in a
// sequence of time steps a different order of the sums shows within a few steps.
//
// Bound: HBM.  On the 2.1M-cell plate in FP64 (256 x 64 x 128) a sweep step moves
// its 1.6 GB in 320 us (5.0 TB/s, against 6.0 TB/s of a reduction that only reads);
// five lanes per row on row-major blocks in cell order took 1.4 times as long, because
// a colour's rows alternated with the other colours' and with the diagonal blocks a
// sweep does not read, at 200-byte blocks that start and end inside cache lines.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <stdexcept>
#include <type_traits>

#include "kernels.hpp"
#include "kernels_sell.hpp"
#include "kernels_sell_device.hpp"
#include "reduce_device.hpp"

namespace cfdg {

namespace {

constexpr int kBlock = kSellBlock;

inline dim3 grid_for(long long n) { return dim3(static_cast<unsigned>((n + kBlock - 1) / kBlock)); }

[[noreturn]] void throw_bad_combination(const char* what) { throw std::invalid_argument(what); }

template <class TS, class TL>
__global__ void __launch_bounds__(kBlock) k_sell_lu(SellArgs b, const word_t<TS>* diag, TL* lu, std::uint16_t* piv,
                                                    int* singular) {
    const int p = blockIdx.x * kBlock + threadIdx.x;
    if (p >= b.nslices * kSellRows) return;
    const int row = b.row[p];
    if (row < 0) return;
    const int slice = p >> 6, lane = p & (kSellRows - 1);
    double a[25];
    {
        word_t<TS> w[SellLayout<TS>::words];
        load_words<TS>(diag, slice, lane, w);
#pragma unroll
        for (int k = 0; k < 25; ++k) a[k] = entry<TS, double>(w, k);
    }
    unsigned pv = 0;
    bool ok = true;
    // fully unrolled so that the 25 entries stay in registers: the row swap is
    // a select over the (compile-time) candidate rows
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        int mrow = k;
        double mx = fabs(a[k * 5 + k]);
#pragma unroll
        for (int r = k + 1; r < 5; ++r) {
            const double v = fabs(a[r * 5 + k]);
            if (v > mx) {
                mx = v;
                mrow = r;
            }
        }
        pv |= static_cast<unsigned>(mrow) << (3 * k);
        ok = ok && (mx != 0.0);
#pragma unroll
        for (int r = k + 1; r < 5; ++r) {
            const bool sw = (mrow == r);
#pragma unroll
            for (int j = 0; j < 5; ++j) {
                const double tk = a[k * 5 + j], tr = a[r * 5 + j];
                a[k * 5 + j] = sw ? tr : tk;
                a[r * 5 + j] = sw ? tk : tr;
            }
        }
        const double inv_d = 1.0 / a[k * 5 + k];
#pragma unroll
        for (int r = k + 1; r < 5; ++r) {
            const double l = a[r * 5 + k] * inv_d;
            a[r * 5 + k] = l;
#pragma unroll
            for (int j = k + 1; j < 5; ++j) a[r * 5 + j] -= l * a[k * 5 + j];
        }
    }
    if (!ok) {
        atomicMax(singular, row + 1);  // integer flag: largest singular row + 1
        return;
    }
    TL* dst = lu + static_cast<long long>(slice) * (25 * kSellRows) + lane;
#pragma unroll
    for (int k = 0; k < 25; ++k) dst[k * kSellRows] = cvt<TL>(a[k]);
    piv[p] = static_cast<std::uint16_t>(pv);
}

// y = A x in the rows of slices [first, first + count).
template <class TS, class TV, int kSplit>
__global__ void __launch_bounds__(slice_threads<kSplit>()) k_sell_spmv(SellArgs b, int first, int count,
                                                                       const word_t<TS>* off, const word_t<TS>* diag,
                                                                       const TV* x, TV* y, const double* gate) {
    __shared__ TV lds[split_lds<kSplit, TV>()];
    if (gate && gate[kKsStatus] != 0.0) return;
    const int ls = wave_slice<kSplit>();
    if (ls >= count) return;
    const Rows q = rows_of(b, first + ls);
    const bool lead = lead_wave<kSplit>() && q.on;
    const int before = lead ? b.before[q.slice * kSellRows + q.lane] : 0;
    TV d[5];
    RowSum<TV> sum;
    if (lead) {
        TV xv[5];
#pragma unroll
        for (int v = 0; v < 5; ++v) xv[v] = x[q.at + v * kSellRows];
        diagonal_times<TS, TV>(diag, q, xv, d);
    }
    for_blocks<kSplit, true, TS, TV>(b, off, q, x, lds, [&](int k, const TV t[5]) { sum.add(k, t, before, d); });
    if (!lead) return;
    sum.finish(q.blocks(), before, d);
#pragma unroll
    for (int v = 0; v < 5; ++v) y[q.at + v * kSellRows] = sum.s[v];
}

// z_i = D_i^-1 (r_i - sum A_ij z_j) for the rows of one colour.
template <class TS, class TL, class TV, int kSplit, bool kAll>
__global__ void __launch_bounds__(slice_threads<kSplit>()) k_sell_sweep(SellArgs b, int first, int count,
                                                                        const word_t<TS>* off, const TL* lu,
                                                                        const std::uint16_t* piv, const TV* r, TV* z,
                                                                        const double* gate) {
    __shared__ TV lds[split_lds<kSplit, TV>()];
    if (gate && gate[kKsStatus] != 0.0) return;
    const int ls = wave_slice<kSplit>();
    if (ls >= count) return;
    const Rows q = rows_of(b, first + ls);
    const bool lead = lead_wave<kSplit>() && q.on;
    TV acc[5], L[25];
    if (lead) {
#pragma unroll
        for (int v = 0; v < 5; ++v) acc[v] = r[q.at + v * kSellRows];
        if (kSplit > 1) load_lu<TL, TV>(lu, q.slice, q.lane, L);  // in flight with the slots
    }
    for_blocks<kSplit, kAll, TS, TV>(b, off, q, z, lds, [&](int, const TV t[5]) {
#pragma unroll
        for (int v = 0; v < 5; ++v) acc[v] -= t[v];
    });
    if (!lead) return;
    if (kSplit == 1) load_lu<TL, TV>(lu, q.slice, q.lane, L);
    lu_solve(acc, L, piv[q.slice * kSellRows + q.lane]);
#pragma unroll
    for (int v = 0; v < 5; ++v) z[q.at + v * kSellRows] = acc[v];
}

__global__ void __launch_bounds__(kBlock) k_sell_gather(SellArgs b, const int* src_of, const double* src, double* dst) {
    const int p = blockIdx.x * kBlock + threadIdx.x;
    if (p >= b.nslices * kSellRows) return;
    const int row = b.row[p];
    if (row < 0) return;
    const double* u = src + 5LL * (src_of ? src_of[row] : row);
    double* d = dst + vec_at(p);
    for (int v = 0; v < 5; ++v) d[v * kSellRows] = u[v];
}

__global__ void __launch_bounds__(kBlock) k_sell_scatter(SellArgs b, const int* dst_of, const double* src, double* dst) {
    const int row = blockIdx.x * kBlock + threadIdx.x;
    if (row >= b.n) return;
    const double* u = src + vec_at(b.pos[row]);
    double* d = dst + 5LL * (dst_of ? dst_of[row] : row);
    for (int v = 0; v < 5; ++v) d[v] = u[v * kSellRows];
}

// Partial dot products of vectors of the layout, in the order of k_dots
// (kernels_linalg.hip) on flat vectors: element i is component i % 5 of device row
// i / 5, thread t of workgroup blk takes i = blk 256 + t and every nb 256th from there.
// load(row, component, v) gives an element's kVals factors; the products are v0 v0
// (one factor), v0 v1, or (kDots 2) v0 v0 and v1 v1, or (kDots 5) v0 v0, v0 v1, v2 v0,
// v2 v1, v1 v1.  Four elements are in flight at a time (eight are no faster).  5 rows < 2^32 in
// 288 GB.
template <int kDots, int kVals, class Load>
__device__ __forceinline__ void flat_dots(int blk, int nb, int rows, double* partial, Load&& load) {
    constexpr int kAhead = 4;
    __shared__ double lds[kBlock / 64 * 5];
    const unsigned n = 5u * static_cast<unsigned>(rows), stride = static_cast<unsigned>(nb) * kBlock;
    double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    for (unsigned long long i0 = static_cast<unsigned>(blk) * kBlock + threadIdx.x; i0 < n; i0 += kAhead * stride) {
        double v[kAhead][kVals];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const unsigned long long i = i0 + static_cast<unsigned>(u) * static_cast<unsigned long long>(stride);
            if (i < n) {
                const unsigned row = static_cast<unsigned>(i) / 5u;
                load(static_cast<int>(row), static_cast<int>(static_cast<unsigned>(i) - 5u * row), v[u]);
            }
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            if (i0 + static_cast<unsigned>(u) * static_cast<unsigned long long>(stride) >= n) break;
            const double* e = v[u];
            if constexpr (kDots == 1) {
                acc[0] += e[0] * e[kVals - 1];
            } else if constexpr (kDots == 2) {
                acc[0] += e[0] * e[0];
                acc[1] += e[1] * e[1];
            } else {
                acc[0] += e[0] * e[0];
                acc[1] += e[0] * e[1];
                acc[2] += e[2] * e[0];
                acc[3] += e[2] * e[1];
                acc[4] += e[1] * e[1];
            }
        }
    }
    const double s = block_sums(acc, kDots, lds);
    if (threadIdx.x < kDots) partial[blk * 5 + static_cast<int>(threadIdx.x)] = s;
}

// The dot products of a step or of a start: kDots 1 (v0, v1), 2 (v0, v0) and (v1, v1),
// 5 with v0 = t, v1 = s, v2 = r0.  Bound: HBM at 2.1M cells (two vectors 43 us, three
// 65 us, 3.9 TB/s: the rows' components are read in device order from colour order, in
// runs of about 13 rows), latency below a million.  Workgroups in XCD order: neighbours
// share lines.
template <int kDots, class TV>
__global__ void __launch_bounds__(kBlock) k_sell_dots(SellArgs b, const TV* v0, const TV* v1, const TV* v2,
                                                      double* partial, const double* gate) {
    if (gate && gate[kKsStatus] != 0.0) return;
    constexpr int kVals = kDots == 5 ? 3 : 2;
    const int nb = static_cast<int>(gridDim.x);
    flat_dots<kDots, kVals>(xcd_block(blockIdx.x, nb), nb, b.n, partial, [&](int row, int k, double v[kVals]) {
        const long long at = vec_at(b.pos[row]) + k * kSellRows;
        v[0] = static_cast<double>(v0[at]);
        v[1] = static_cast<double>(v1[at]);
        if constexpr (kVals == 3) v[2] = static_cast<double>(v2[at]);
    });
}

// b = -R, the implicit right-hand side (implicit_euler.hpp:81-92), x = 0 and the
// squares of R by component (as k_res_sq adds them) in the first nb_norms workgroups,
// (b, b) in the others: one launch where the norms, (b, b) and the fill took one each.
__global__ void __launch_bounds__(kBlock) k_sell_rhs(SellArgs b, int ld, const double* res, double* rhs, double* x,
                                                     double* partial, int nb_norms, int* singular,
                                                     unsigned long long* stamp, int jacobian_end) {
    stamp_stage(stamp, kStampLinear);
    if (jacobian_end) stamp_stage(stamp, kStampJacobianEnd);
    const int blk = static_cast<int>(blockIdx.x);
    if (blk >= nb_norms) {
        const int nb = static_cast<int>(gridDim.x) - nb_norms;
        flat_dots<1, 1>(xcd_block(blk - nb_norms, nb), nb, b.n, partial, [&](int row, int k, double v[1]) {
            v[0] = -res[static_cast<long long>(k) * ld + row];
        });
        return;
    }
    if (blk == 0 && threadIdx.x == 0) *singular = 0;
    __shared__ double lds[kBlock / 64 * 5];
    double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    for (int c = blk * kBlock + static_cast<int>(threadIdx.x); c < b.n; c += nb_norms * kBlock) {
        const long long at = vec_at(b.pos[c]);
        for (int v = 0; v < 5; ++v) {
            const double r = res[static_cast<long long>(v) * ld + c];
            acc[v] += r * r;
            rhs[at + v * kSellRows] = -r;
            x[at + v * kSellRows] = 0.0;
        }
    }
    const double s = block_sums(acc, 5, lds);
    if (threadIdx.x < 5) partial[kNormPartials + blk * 5 + static_cast<int>(threadIdx.x)] = s;
}

// The right-hand side of a defect correction's inner solve, b = r in FP32 and x = 0,
// and (b, b), likewise.
__global__ void __launch_bounds__(kBlock) k_sell_inner_rhs(SellArgs b, const double* r, float* rhs, float* x,
                                                           double* partial, int nb_copy) {
    const int blk = static_cast<int>(blockIdx.x);
    if (blk >= nb_copy) {
        const int nb = static_cast<int>(gridDim.x) - nb_copy;
        flat_dots<1, 1>(xcd_block(blk - nb_copy, nb), nb, b.n, partial, [&](int row, int k, double v[1]) {
            v[0] = static_cast<double>(static_cast<float>(r[vec_at(b.pos[row]) + k * kSellRows]));
        });
        return;
    }
    const long long end = 5LL * kSellRows * b.nslices;
    for (long long e = static_cast<long long>(blk) * kBlock + threadIdx.x; e < end;
         e += static_cast<long long>(nb_copy) * kBlock) {
        rhs[e] = static_cast<float>(r[e]);
        x[e] = 0.0f;
    }
}

// U = U + du (implicit_euler.hpp:53-61)
__global__ void __launch_bounds__(kBlock) k_sell_state_update(SellArgs b, int ld, const double* du, double* U,
                                                              double* du_cells, unsigned long long* stamp) {
    stamp_stage(stamp, kStampLinearEnd);
    const int row = blockIdx.x * kBlock + threadIdx.x;
    if (row >= b.n) return;
    const double* d = du + vec_at(b.pos[row]);
    for (int v = 0; v < 5; ++v) {
        double* u = U + static_cast<long long>(v) * ld + row;
        const double dv = d[v * kSellRows];
        *u = *u + dv;
        du_cells[5LL * row + v] = dv;
    }
}

// The 25 entries of the block with a code (>= 0: slot * 64 + lane, < 0: the
// diagonal block of position -1 - code), one thread per entry.
template <class TS>
__device__ __forceinline__ const word_t<TS>* block_words_of(int code, const word_t<TS>* off, const word_t<TS>* diag) {
    const int c = code >= 0 ? code : -1 - code;
    const long long slot = c >> 6;
    return (code >= 0 ? off : diag) + slot * (SellLayout<TS>::words * kSellRows) + (c & (kSellRows - 1));
}
template <class TS>
__device__ __forceinline__ TS block_entry(const word_t<TS>* w, int e) {
    if constexpr (sizeof(TS) == sizeof(bf16)) {
        const std::uint32_t u = w[(e >> 1) * kSellRows];
        return bf16{static_cast<std::uint16_t>((e & 1) ? (u >> 16) : (u & 0xffffu))};
    } else {
        return w[e * kSellRows];
    }
}

template <class TS>
__global__ void __launch_bounds__(kBlock) k_sell_get_blocks(const int* code, long long n, const word_t<TS>* off,
                                                            const word_t<TS>* diag, double* out) {
    const long long t = static_cast<long long>(blockIdx.x) * kBlock + threadIdx.x;
    if (t >= n * 25) return;
    out[t] = to_f64(block_entry<TS>(block_words_of<TS>(code[t / 25], off, diag), static_cast<int>(t % 25)));
}

// One thread per stored word, so that a bfloat16 pair has one writer.
template <class TS>
__global__ void __launch_bounds__(kBlock) k_sell_set_blocks(const int* code, long long n, const double* in,
                                                            word_t<TS>* off, word_t<TS>* diag) {
    constexpr int kW = SellLayout<TS>::words;
    const long long t = static_cast<long long>(blockIdx.x) * kBlock + threadIdx.x;
    if (t >= n * kW) return;
    const long long k = t / kW;
    const int q = static_cast<int>(t - k * kW);
    word_t<TS>* w = const_cast<word_t<TS>*>(block_words_of<TS>(code[k], off, diag)) + q * kSellRows;
    const double* v = in + k * 25;
    if constexpr (sizeof(TS) == sizeof(bf16)) {
        const std::uint32_t lo = cvt<bf16>(v[2 * q]).u;
        const std::uint32_t hi = 2 * q + 1 < 25 ? cvt<bf16>(v[2 * q + 1]).u : 0;
        *w = lo | (hi << 16);
    } else {
        *w = cvt<TS>(v[q]);
    }
}

template <class TS>
__global__ void __launch_bounds__(kBlock) k_sell_to_csr(const int* code, long long n, const word_t<TS>* off,
                                                        const word_t<TS>* diag, TS* values) {
    const long long t = static_cast<long long>(blockIdx.x) * kBlock + threadIdx.x;
    if (t >= n * 25) return;
    const long long k = t / 25;
    const int e = static_cast<int>(t - k * 25);
    values[k * BlockLayout<TS>::block + (e / 5) * BlockLayout<TS>::row + e % 5] =
        block_entry<TS>(block_words_of<TS>(code[k], off, diag), e);
}

}  // namespace

void launch_sell_lu(const SellArgs& b, const SellMatrix& m, void* lu, int lu_f32, std::uint16_t* piv, int* singular,
                    hipStream_t s) {
    if (b.nslices <= 0) return;
    const dim3 g = grid_for_slices(b.nslices), blk(kBlock);
    if (!lu_f32) {
        if (m.storage != kStoreF64) throw_bad_combination("FP64 LU needs FP64 blocks");
        hipLaunchKernelGGL((k_sell_lu<double, double>), g, blk, 0, s, b, static_cast<const double*>(m.diag),
                           static_cast<double*>(lu), piv, singular);
        return;
    }
    with_storage(m.storage, [&](auto ts) {
        typedef decltype(ts) TS;
        hipLaunchKernelGGL((k_sell_lu<TS, float>), g, blk, 0, s, b, static_cast<const word_t<TS>*>(m.diag),
                           static_cast<float*>(lu), piv, singular);
    });
}

template <class TV>
void launch_sell_spmv(const SellArgs& b, const SellMatrix& m, int first, int count, const TV* x, TV* y, hipStream_t s,
                      const double* gate) {
    if (count <= 0) return;
    with_split(count, [&](auto split) {
        with_storage(m.storage, [&](auto ts) {
            typedef decltype(ts) TS;
            constexpr int kS = decltype(split)::value;
            hipLaunchKernelGGL((k_sell_spmv<TS, TV, kS>), slice_grid<kS>(count), dim3(slice_threads<kS>()), 0, s, b,
                               first, count, static_cast<const word_t<TS>*>(m.off),
                               static_cast<const word_t<TS>*>(m.diag), x, y, gate);
        });
    });
}
template void launch_sell_spmv<double>(const SellArgs&, const SellMatrix&, int, int, const double*, double*,
                                       hipStream_t, const double*);
template void launch_sell_spmv<float>(const SellArgs&, const SellMatrix&, int, int, const float*, float*, hipStream_t,
                                      const double*);

template <class TV>
void launch_sell_sweep(const SellArgs& b, const SellMatrix& m, int first, int count, bool all, const TV* r, TV* z,
                       hipStream_t s, const double* gate) {
    if (count <= 0) return;
    const auto launch = [&](auto split, auto ts, auto whole) {
        typedef decltype(ts) TS;
        typedef std::conditional_t<sizeof(TV) == sizeof(double), double, float> TL;
        constexpr int kS = decltype(split)::value;
        hipLaunchKernelGGL((k_sell_sweep<TS, TL, TV, kS, decltype(whole)::value>), slice_grid<kS>(count),
                           dim3(slice_threads<kS>()), 0, s, b, first, count, static_cast<const word_t<TS>*>(m.off),
                           static_cast<const TL*>(m.lu), m.piv, r, z, gate);
    };
    with_split(count, [&](auto split) {
        with_form<TV>(m, [&](auto ts) {
            if (all)
                launch(split, ts, std::true_type{});
            else
                launch(split, ts, std::false_type{});
        });
    });
}
template void launch_sell_sweep<double>(const SellArgs&, const SellMatrix&, int, int, bool, const double*, double*,
                                        hipStream_t, const double*);
template void launch_sell_sweep<float>(const SellArgs&, const SellMatrix&, int, int, bool, const float*, float*,
                                       hipStream_t, const double*);

void launch_sell_gather(const SellArgs& b, const int* src_of, const double* src, double* dst, hipStream_t s) {
    if (b.nslices > 0)
        hipLaunchKernelGGL(k_sell_gather, grid_for_slices(b.nslices), dim3(kBlock), 0, s, b, src_of, src, dst);
}

void launch_sell_scatter(const SellArgs& b, const int* dst_of, const double* src, double* dst, hipStream_t s) {
    if (b.n > 0) hipLaunchKernelGGL(k_sell_scatter, grid_for(b.n), dim3(kBlock), 0, s, b, dst_of, src, dst);
}

template <class TV>
int launch_sell_dots(const SellArgs& b, int ndot, const TV* v0, const TV* v1, const TV* v2, double* partial,
                     hipStream_t s, const double* gate) {
    const int nb = reduction_blocks(5LL * b.n);
    const dim3 g(static_cast<unsigned>(nb)), blk(kBlock);
    if (ndot == 1)
        hipLaunchKernelGGL((k_sell_dots<1, TV>), g, blk, 0, s, b, v0, v1, v2, partial, gate);
    else if (ndot == 2)
        hipLaunchKernelGGL((k_sell_dots<2, TV>), g, blk, 0, s, b, v0, v1, v2, partial, gate);
    else
        hipLaunchKernelGGL((k_sell_dots<5, TV>), g, blk, 0, s, b, v0, v1, v2, partial, gate);
    return nb;
}
template int launch_sell_dots<double>(const SellArgs&, int, const double*, const double*, const double*, double*,
                                      hipStream_t, const double*);
template int launch_sell_dots<float>(const SellArgs&, int, const float*, const float*, const float*, double*,
                                     hipStream_t, const double*);

SellSums launch_sell_rhs(const SellArgs& b, int ld, const double* res, double* rhs, double* x, bool square,
                         double* partial, int* singular, unsigned long long* stamp, bool jacobian_end, hipStream_t s) {
    const SellSums n{square ? reduction_blocks(5LL * b.n) : 0, reduction_blocks(b.n)};
    hipLaunchKernelGGL(k_sell_rhs, dim3(static_cast<unsigned>(n.dots + n.norms)), dim3(kBlock), 0, s, b, ld, res, rhs, x,
                       partial, n.norms, singular, stamp, jacobian_end ? 1 : 0);
    return n;
}

SellSums launch_sell_inner_rhs(const SellArgs& b, const double* r, float* rhs, float* x, double* partial,
                               hipStream_t s) {
    const SellSums n{reduction_blocks(5LL * b.n), 0};
    const int copy = reduction_blocks(5LL * kSellRows * b.nslices);
    hipLaunchKernelGGL(k_sell_inner_rhs, dim3(static_cast<unsigned>(copy + n.dots)), dim3(kBlock), 0, s, b, r, rhs, x,
                       partial, copy);
    return n;
}

void launch_sell_state_update(const SellArgs& b, int ld, const double* du, double* U, double* du_cells,
                              unsigned long long* stamp, hipStream_t s) {
    if (b.n > 0)
        hipLaunchKernelGGL(k_sell_state_update, grid_for(b.n), dim3(kBlock), 0, s, b, ld, du, U, du_cells, stamp);
}

void launch_sell_get_blocks(const int* code, long long n, const SellMatrix& m, double* out, hipStream_t s) {
    if (n <= 0) return;
    with_storage(m.storage, [&](auto ts) {
        typedef decltype(ts) TS;
        hipLaunchKernelGGL(k_sell_get_blocks<TS>, grid_for(n * 25), dim3(kBlock), 0, s, code, n,
                           static_cast<const word_t<TS>*>(m.off), static_cast<const word_t<TS>*>(m.diag), out);
    });
}

void launch_sell_set_blocks(const int* code, long long n, const double* in, void* off, void* diag, int storage,
                            hipStream_t s) {
    if (n <= 0) return;
    with_storage(storage, [&](auto ts) {
        typedef decltype(ts) TS;
        hipLaunchKernelGGL(k_sell_set_blocks<TS>, grid_for(n * SellLayout<TS>::words), dim3(kBlock), 0, s, code, n, in,
                           static_cast<word_t<TS>*>(off), static_cast<word_t<TS>*>(diag));
    });
}

void launch_sell_to_csr(const int* code, long long n, const SellMatrix& m, void* values, hipStream_t s) {
    if (n <= 0) return;
    with_storage(m.storage, [&](auto ts) {
        typedef decltype(ts) TS;
        hipLaunchKernelGGL(k_sell_to_csr<TS>, grid_for(n * 25), dim3(kBlock), 0, s, code, n,
                           static_cast<const word_t<TS>*>(m.off), static_cast<const word_t<TS>*>(m.diag),
                           static_cast<TS*>(values));
    });
}

}  // namespace cfdg
