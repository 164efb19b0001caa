// Device functions and launch rules of the kernels on the sliced block layout
// (kernels_sell.hip, kernels_multicolour.hip): block and factor loads, the 5x5
// solve, and the walk over a slice's slots by one wave, four or eight.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <stdexcept>
#include <type_traits>

#include "kernels.hpp"
#include "kernels_sell.hpp"

namespace cfdg {

constexpr int kSellBlock = 256;
constexpr int kBlockSlices = kSellBlock / kSellRows;  // slices per workgroup, one per wave

inline dim3 grid_for_slices(int n) { return dim3(static_cast<unsigned>((n + kBlockSlices - 1) / kBlockSlices)); }

template <class TS>
using word_t = typename SellLayout<TS>::word;

// The 25 entries of the block in (slot, lane) as storage words.
template <class TS>
__device__ __forceinline__ void load_words(const word_t<TS>* v, long long slot, int lane, word_t<TS> w[]) {
    const word_t<TS>* p = v + slot * (SellLayout<TS>::words * kSellRows) + lane;
#pragma unroll
    for (int q = 0; q < SellLayout<TS>::words; ++q) w[q] = p[q * kSellRows];
}
// Entry e of a loaded block in the arithmetic type.
template <class TS, class TV>
__device__ __forceinline__ TV entry(const word_t<TS> w[], int e) {
    if constexpr (sizeof(TS) == sizeof(bf16)) {
        const std::uint32_t u = w[e >> 1];
        return static_cast<TV>(f32_from_bits((e & 1) ? (u & 0xffff0000u) : (u << 16)));
    } else {
        return load_as<TV>(w[e]);
    }
}

// Component 0 of the row at a position; component v follows at v * 64.
__device__ __forceinline__ long long vec_at(int position) {
    return static_cast<long long>(position >> 6) * (5 * kSellRows) + (position & (kSellRows - 1));
}

// t = A x of one block: t_a = a0 x0 + a1 x1 + ... in column order
template <class TS, class TV>
__device__ __forceinline__ void block_times(const word_t<TS> w[], const TV x[5], TV t[5]) {
#pragma unroll
    for (int a = 0; a < 5; ++a) {
        TV s = entry<TS, TV>(w, a * 5) * x[0];
#pragma unroll
        for (int b = 1; b < 5; ++b) s += entry<TS, TV>(w, a * 5 + b) * x[b];
        t[a] = s;
    }
}

// Solution of (LU) x = s with partial pivoting (lu_solve_block<5>,
// bsr_helpers.hpp:325-353); pivots as five 3-bit row numbers.
template <class TV>
__device__ __forceinline__ void lu_solve(TV s[5], const TV L[25], unsigned piv) {
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        const int pk = static_cast<int>((piv >> (3 * k)) & 7u);
        const TV sk = s[k];
        TV sp = sk;
#pragma unroll
        for (int q = k + 1; q < 5; ++q) {
            const bool sw = q == pk;
            sp = sw ? s[q] : sp;
            s[q] = sw ? sk : s[q];
        }
        s[k] = sp;
    }
#pragma unroll
    for (int a = 1; a < 5; ++a)
#pragma unroll
        for (int b = 0; b < a; ++b) s[a] -= L[a * 5 + b] * s[b];
#pragma unroll
    for (int a = 4; a >= 0; --a) {
#pragma unroll
        for (int b = a + 1; b < 5; ++b) s[a] -= L[a * 5 + b] * s[b];
        s[a] = s[a] / L[a * 5 + a];
    }
}

template <class TL, class TV>
__device__ __forceinline__ void load_lu(const TL* lu, int slice, int lane, TV L[25]) {
    const TL* p = lu + static_cast<long long>(slice) * (25 * kSellRows) + lane;
#pragma unroll
    for (int k = 0; k < 25; ++k) L[k] = load_as<TV>(p[k * kSellRows]);
}

// t = A x for the row's block in a slot.
template <class TS, class TV>
__device__ __forceinline__ void slot_times(const word_t<TS>* off, const int* cols, long long slot, int lane,
                                           const TV* x, TV t[5]) {
    word_t<TS> w[SellLayout<TS>::words];
    const TV* xb = x + vec_at(cols[slot * kSellRows + lane]);
    load_words<TS>(off, slot, lane, w);
    TV xv[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) xv[v] = xb[v * kSellRows];
    block_times<TS, TV>(w, xv, t);
}

// A wave's slice: its slots and rows, whether the lane holds a row, the row's blocks
// (lower | upper << 16) and where component 0 of its vector entries is.
struct Rows {
    int slice, lane;
    int4 sl;
    bool on;
    unsigned n;
    long long at;
    __device__ __forceinline__ int lower() const { return static_cast<int>(n & 0xffffu); }
    __device__ __forceinline__ int blocks() const { return lower() + static_cast<int>(n >> 16); }
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
// The products with x of a row's lower blocks, or with kAll of all its off-diagonal
// blocks, handed to add(k, t) in ascending mesh column (k counts them): the order of a
// row-major matrix, so that a row's sums do not depend on the colours or on the layout.
// In a slice with lower and upper slots that order is read from b.order; elsewhere the
// slots are in it.  kSplit = 1: by the wave alone, one after the other.  kSplit > 1: the kSplit
// waves of the workgroup, all on the same slice, form kSplit products at a time into LDS
// and the first wave adds them.
template <int kSplit, bool kAll, class TS, class TV, class F>
__device__ __forceinline__ void for_blocks(const SellArgs& b, const word_t<TS>* off, const Rows& q, const TV* x,
                                           TV* lds, F&& add) {
    const int most = kAll ? q.sl.y + q.sl.z : q.sl.y, mine = kAll ? q.blocks() : q.lower();
    const auto walk = [&](auto&& slot) {
        if constexpr (kSplit == 1) {
            for (int k = 0; k < most; ++k) {
                if (k >= mine) continue;
                TV t[5];
                slot_times<TS, TV>(off, b.cols, slot(k), q.lane, x, t);
                add(k, t);
            }
        } else {
            const int w = threadIdx.x >> 6;
            for (int k0 = 0; k0 < most; k0 += kSplit) {
                if (k0 + w < mine) {
                    TV t[5];
                    slot_times<TS, TV>(off, b.cols, slot(k0 + w), q.lane, x, t);
#pragma unroll
                    for (int v = 0; v < 5; ++v) lds[(w * 5 + v) * kSellRows + q.lane] = t[v];
                }
                __syncthreads();
                if (w == 0)
                    for (int k = 0; k < kSplit && k0 + k < mine; ++k) {
                        TV t[5];
#pragma unroll
                        for (int v = 0; v < 5; ++v) t[v] = lds[(k * 5 + v) * kSellRows + q.lane];
                        add(k0 + k, t);
                    }
                if (k0 + kSplit < most) __syncthreads();
            }
        }
    };
    const long long base = q.sl.x;
    if (kAll && q.sl.y > 0 && q.sl.z > 0)
        walk([&](int k) { return base + b.order[(base + k) * kSellRows + q.lane]; });
    else
        walk([&](int k) { return base + k; });
}

// The sum of a row's product y = A x: the off-diagonal products as for_blocks hands
// them over, and the diagonal one, d, in its place among them (before: the number of
// off-diagonal blocks that precede it).
template <class TV>
struct RowSum {
    TV s[5] = {0, 0, 0, 0, 0};
    __device__ __forceinline__ void add(const TV t[5]) {
#pragma unroll
        for (int v = 0; v < 5; ++v) s[v] += t[v];
    }
    __device__ __forceinline__ void add(int k, const TV t[5], int before, const TV d[5]) {
        if (k == before) add(d);
        add(t);
    }
    __device__ __forceinline__ void finish(int blocks, int before, const TV d[5]) {
        if (blocks == before) add(d);
    }
};
// d = D x for the row's diagonal block
template <class TS, class TV>
__device__ __forceinline__ void diagonal_times(const word_t<TS>* diag, const Rows& q, const TV x[5], TV d[5]) {
    word_t<TS> w[SellLayout<TS>::words];
    load_words<TS>(diag, q.slice, q.lane, w);
    block_times<TS, TV>(w, x, d);
}

template <int kSplit>
__device__ __forceinline__ bool lead_wave() {
    return kSplit == 1 || threadIdx.x < kSellRows;
}
template <int kSplit>
constexpr int slice_threads() {
    return kSplit == 1 ? kSellBlock : kSplit * kSellRows;
}
template <int kSplit, class TV>
constexpr int split_lds() {
    return kSplit == 1 ? 1 : kSplit * 5 * kSellRows;
}
// The slice of this wave among count, or count and above for none.
template <int kSplit>
__device__ __forceinline__ int wave_slice() {
    const int b = xcd_block(blockIdx.x, gridDim.x);
    return kSplit == 1 ? b * kBlockSlices + static_cast<int>(threadIdx.x >> 6) : b;
}

// Waves per slice.  A launch over few slices is bound by the latency of a row's
// chain of slots, so eight or four waves share a slice (a hexahedron's or tetrahedron's
// slots all at once, or in two goes); over many slices one wave each fills the chip and
// the split only adds barriers.  Per BiCGSTAB iteration with one / four / eight waves
// (slices of a colour): 24,576-cell plate (192) FP64 92 / 73 / 70 us, BF16 67 / 58 / 56;
// 93,765 cells (735) 122 / 123 / 132, 87 / 80 / 79; 156,849 cells (1,226) 217 / 189 / 201,
// 100 / 98 / 100; 196,608 cells (1,536) 241 / 230 / 244, 106 / 105 / 111; 162,000 tetrahedra
// (four colours) 239 / 231 / 254, 153 / 131 / 137; 262,144 cells (2,048) 302 / 318 / 336,
// 119 / 126 / 130.
constexpr int kEightSlices = 384, kSplitSlices = 1536;
template <int kSplit>
dim3 slice_grid(int slices) {
    return kSplit == 1 ? grid_for_slices(slices) : dim3(static_cast<unsigned>(slices));
}
// f(std::integral_constant<int, waves per slice>) for a launch over that many slices
template <class F>
void with_split(int slices, F&& f) {
    if (slices <= kEightSlices)
        f(std::integral_constant<int, 8>{});
    else if (slices <= kSplitSlices)
        f(std::integral_constant<int, 4>{});
    else
        f(std::integral_constant<int, 1>{});
}

// f(TS{}) for the storage kind
template <class F>
void with_storage(int storage, F&& f) {
    if (storage == kStoreF32)
        f(float{});
    else if (storage == kStoreBF16)
        f(bf16{});
    else
        f(double{});
}

// f(storage type) with the LU type that follows the vector type, FP64 vectors only
// with FP64 blocks.
template <class TV, class F>
void with_form(const SellMatrix& m, F&& f) {
    if constexpr (sizeof(TV) == sizeof(double)) {
        if (m.storage != kStoreF64) throw std::invalid_argument("FP64 SGS needs FP64 blocks");
        f(double{});
    } else {
        with_storage(m.storage, f);
    }
}

}  // namespace cfdg
