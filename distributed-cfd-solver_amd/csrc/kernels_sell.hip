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
// The iterations of the solve run on kernels_reduced.hip, which needs neither a
// whole product nor a whole sweep; these serve the residuals of the defect
// correction, the ABI's product and preconditioner calls, and the solves that the
// reduced form leaves (bicgstab, capi.cpp).
//
// Arithmetic per row component: products summed over the block's columns, the
// block sums added or subtracted in the order of the row's slots.
//
// Bound: HBM.  On the 2.1M-cell plate in FP64 (256 x 64 x 128) a sweep step moves
// its 1.6 GB in 273 us and the product its 2.96 GB of blocks in 525 us (5.6-5.8
// TB/s, against 6.0 TB/s of a reduction that only reads); five lanes per row on
// row-major blocks in cell order took 384 and 612 us, because a colour's rows
// alternated with the other colours' and with the diagonal blocks a sweep does not
// read, at 200-byte blocks that start and end inside cache lines.
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

template <class TS, class TV, int kSplit>
__global__ void __launch_bounds__(slice_threads<kSplit>()) k_sell_spmv(SellArgs b, const word_t<TS>* off,
                                                                       const word_t<TS>* diag, const TV* x, TV* y,
                                                                       const double* gate) {
    __shared__ TV lds[split_lds<kSplit, TV>()];
    if (gate && gate[kKsStatus] != 0.0) return;
    const int slice = wave_slice<kSplit>();
    if (slice >= b.nslices) return;
    const int lane = threadIdx.x & 63;
    const int4 sl = b.slice[slice];
    const bool lead = kSplit == 1 || threadIdx.x < kSellRows;
    const bool on = lane < sl.w;
    const unsigned n = on ? b.count[slice * kSellRows + lane] : 0;
    const long long at = static_cast<long long>(slice) * (5 * kSellRows) + lane;
    TV acc[5];
    if (lead && on) {
        word_t<TS> w[SellLayout<TS>::words];
        load_words<TS>(diag, slice, lane, w);
        TV xv[5];
#pragma unroll
        for (int v = 0; v < 5; ++v) xv[v] = x[at + v * kSellRows];
        block_times<TS, TV>(w, xv, acc);
    }
    for_slots<kSplit, TS, TV>(off, b.cols, sl, n, 0, sl.y + sl.z, 0, lane, x, lds, [&](const TV t[5]) {
#pragma unroll
        for (int v = 0; v < 5; ++v) acc[v] += t[v];
    });
    if (!lead || !on) return;
#pragma unroll
    for (int v = 0; v < 5; ++v) y[at + v * kSellRows] = acc[v];
}

// z_i = D_i^-1 (r_i - sum A_ij z_j) for the rows of one colour.
template <class TS, class TL, class TV, int kSplit>
__global__ void __launch_bounds__(slice_threads<kSplit>()) k_sell_sweep(SellArgs b, int first, int count, int all,
                                                                        const word_t<TS>* off, const TL* lu,
                                                                        const std::uint16_t* piv, const TV* r, TV* z,
                                                                        const double* gate) {
    __shared__ TV lds[split_lds<kSplit, TV>()];
    if (gate && gate[kKsStatus] != 0.0) return;
    const int ls = wave_slice<kSplit>();
    if (ls >= count) return;
    const int slice = first + ls;
    const int lane = threadIdx.x & 63;
    const int4 sl = b.slice[slice];
    const bool lead = kSplit == 1 || threadIdx.x < kSellRows;
    const bool on = lane < sl.w;
    const unsigned n = on ? b.count[slice * kSellRows + lane] : 0;
    const long long at = static_cast<long long>(slice) * (5 * kSellRows) + lane;
    TV acc[5], L[25];
    if (lead && on) {
#pragma unroll
        for (int v = 0; v < 5; ++v) acc[v] = r[at + v * kSellRows];
        if (kSplit > 1) load_lu<TL, TV>(lu, slice, lane, L);  // in flight with the slots
    }
    for_slots<kSplit, TS, TV>(off, b.cols, sl, n, 0, all ? sl.y + sl.z : sl.y, 0, lane, z, lds, [&](const TV t[5]) {
#pragma unroll
        for (int v = 0; v < 5; ++v) acc[v] -= t[v];
    });
    if (!lead || !on) return;
    if (kSplit == 1) load_lu<TL, TV>(lu, slice, lane, L);
    lu_solve(acc, L, piv[slice * kSellRows + lane]);
#pragma unroll
    for (int v = 0; v < 5; ++v) z[at + v * kSellRows] = acc[v];
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

// The positions of the sliced layout in grid-stride order, f(position, device row)
// for those that hold a row and as many workgroups as a reduction has partial sums.
template <class F>
__device__ __forceinline__ void for_rows(const SellArgs& b, F&& f) {
    const int end = b.nslices * kSellRows, stride = static_cast<int>(gridDim.x * blockDim.x);
    for (int p = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x); p < end; p += stride) {
        const int row = b.row[p];
        if (row >= 0) f(p, row);
    }
}

// Partial sums of squares for launch_bicg_start: by component, and the total of the
// positions before first_end.
struct Squares {
    double all[5] = {0.0, 0.0, 0.0, 0.0, 0.0}, first = 0.0;
    __device__ __forceinline__ void store(double* partial) const {
        __shared__ double lds[2][kBlock / 64 * 5];
        const double f[5] = {first, 0.0, 0.0, 0.0, 0.0};
        const double s = block_sums(all, 5, lds[0]);
        const double s0 = block_sums(f, 1, lds[1]);
        if (threadIdx.x < 5) partial[blockIdx.x * 5 + threadIdx.x] = s;
        if (threadIdx.x == 0) partial[5 * kMaxPartials + blockIdx.x] = s0;
    }
};

// b = -R, the implicit right-hand side (implicit_euler.hpp:81-92), x = 0, and the
// squares of R: one pass where the norms and (b, b) took one each and x a fill.
__global__ void __launch_bounds__(kBlock) k_sell_rhs(SellArgs b, int ld, const double* res, double* rhs, double* x,
                                                     int first_end, double* partial, int* singular,
                                                     unsigned long long* stamp, int jacobian_end) {
    stamp_stage(stamp, kStampLinear);
    if (jacobian_end) stamp_stage(stamp, kStampJacobianEnd);
    if (blockIdx.x == 0 && threadIdx.x == 0) *singular = 0;
    Squares q;
    for_rows(b, [&](int p, int row) {
        const long long at = vec_at(p);
        for (int v = 0; v < 5; ++v) {
            const double r = res[static_cast<long long>(v) * ld + row];
            rhs[at + v * kSellRows] = -r;
            x[at + v * kSellRows] = 0.0;
            q.all[v] += r * r;
            if (p < first_end) q.first += r * r;
        }
    });
    q.store(partial);
}

// The squares of a vector, added as the kernels above and below add theirs.
template <class TV>
__global__ void __launch_bounds__(kBlock) k_sell_squares(SellArgs b, const TV* u, int first_end, double* partial) {
    Squares q;
    for_rows(b, [&](int p, int) {
        const long long at = vec_at(p);
        for (int v = 0; v < 5; ++v) {
            const double d = static_cast<double>(u[at + v * kSellRows]);
            q.all[v] += d * d;
            if (p < first_end) q.first += d * d;
        }
    });
    q.store(partial);
}

// The right-hand side of a defect correction's inner solve, b = r in FP32, x = 0, and
// the squares of b.
__global__ void __launch_bounds__(kBlock) k_sell_inner_rhs(SellArgs b, const double* r, float* rhs, float* x,
                                                           int first_end, double* partial) {
    Squares q;
    for_rows(b, [&](int p, int) {
        const long long at = vec_at(p);
        for (int v = 0; v < 5; ++v) {
            const float f = static_cast<float>(r[at + v * kSellRows]);
            rhs[at + v * kSellRows] = f;
            x[at + v * kSellRows] = 0.0f;
            const double d = static_cast<double>(f);
            q.all[v] += d * d;
            if (p < first_end) q.first += d * d;
        }
    });
    q.store(partial);
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
void launch_sell_spmv(const SellArgs& b, const SellMatrix& m, const TV* x, TV* y, hipStream_t s, const double* gate) {
    if (b.nslices <= 0) return;
    with_split(b.nslices, [&](auto split) {
        with_storage(m.storage, [&](auto ts) {
            typedef decltype(ts) TS;
            constexpr int kS = decltype(split)::value;
            hipLaunchKernelGGL((k_sell_spmv<TS, TV, kS>), slice_grid<kS>(b.nslices), dim3(slice_threads<kS>()), 0, s,
                               b, static_cast<const word_t<TS>*>(m.off), static_cast<const word_t<TS>*>(m.diag), x, y,
                               gate);
        });
    });
}
template void launch_sell_spmv<double>(const SellArgs&, const SellMatrix&, const double*, double*, hipStream_t,
                                       const double*);
template void launch_sell_spmv<float>(const SellArgs&, const SellMatrix&, const float*, float*, hipStream_t,
                                      const double*);

template <class TV>
void launch_sell_sweep(const SellArgs& b, const SellMatrix& m, int first, int count, bool all, const TV* r, TV* z,
                       hipStream_t s, const double* gate) {
    if (count <= 0) return;
    with_split(count, [&](auto split) {
        constexpr int kS = decltype(split)::value;
        const dim3 g = slice_grid<kS>(count), blk(slice_threads<kS>());
        if constexpr (sizeof(TV) == sizeof(double)) {
            if (m.storage != kStoreF64) throw_bad_combination("FP64 SGS needs FP64 blocks");
            hipLaunchKernelGGL((k_sell_sweep<double, double, double, kS>), g, blk, 0, s, b, first, count, all ? 1 : 0,
                               static_cast<const double*>(m.off), static_cast<const double*>(m.lu), m.piv, r, z, gate);
        } else {
            with_storage(m.storage, [&](auto ts) {
                typedef decltype(ts) TS;
                hipLaunchKernelGGL((k_sell_sweep<TS, float, float, kS>), g, blk, 0, s, b, first, count, all ? 1 : 0,
                                   static_cast<const word_t<TS>*>(m.off), static_cast<const float*>(m.lu), m.piv, r, z,
                                   gate);
            });
        }
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

int launch_sell_rhs(const SellArgs& b, int ld, const double* res, double* rhs, double* x, int first_slices,
                    double* partial, int* singular, unsigned long long* stamp, bool jacobian_end, hipStream_t s) {
    const int nb = reduction_blocks(static_cast<long long>(b.nslices) * kSellRows);
    hipLaunchKernelGGL(k_sell_rhs, dim3(nb), dim3(kBlock), 0, s, b, ld, res, rhs, x, first_slices * kSellRows, partial,
                       singular, stamp, jacobian_end ? 1 : 0);
    return nb;
}

template <class TV>
int launch_sell_squares(const SellArgs& b, const TV* u, int first_slices, double* partial, hipStream_t s) {
    const int nb = reduction_blocks(static_cast<long long>(b.nslices) * kSellRows);
    hipLaunchKernelGGL(k_sell_squares<TV>, dim3(nb), dim3(kBlock), 0, s, b, u, first_slices * kSellRows, partial);
    return nb;
}
template int launch_sell_squares<double>(const SellArgs&, const double*, int, double*, hipStream_t);
template int launch_sell_squares<float>(const SellArgs&, const float*, int, double*, hipStream_t);

int launch_sell_inner_rhs(const SellArgs& b, const double* r, float* rhs, float* x, int first_slices, double* partial,
                          hipStream_t s) {
    const int nb = reduction_blocks(static_cast<long long>(b.nslices) * kSellRows);
    hipLaunchKernelGGL(k_sell_inner_rhs, dim3(nb), dim3(kBlock), 0, s, b, r, rhs, x, first_slices * kSellRows, partial);
    return nb;
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
