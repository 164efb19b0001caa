// Device functions and launch rules of the kernels on the sliced block layout
// (kernels_sell.hip, kernels_reduced.hip): block and factor loads, the 5x5
// solve, and the walk over a slice's slots by one wave, four or eight.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
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

// Whether the row with block counts n (lower | upper << 16) has a block in the
// j-th slot of its slice.
__device__ __forceinline__ bool has_block(const int4& sl, unsigned n, int j) {
    return j < sl.y ? j < static_cast<int>(n & 0xffffu) : j - sl.y < static_cast<int>(n >> 16);
}

// The products of slots [from, to) of a slice with x, of the row's blocks only
// (has_block), handed to add(t) in slot order.  skip: the row's first lower blocks
// that are left out.  kSplit = 1: by the wave alone, one slot after the other.  kSplit > 1:
// the kSplit waves of the workgroup, all on the same slice, form kSplit slots at a
// time into LDS and the first wave adds them, in the same order.
template <int kSplit, class TS, class TV, class F>
__device__ __forceinline__ void for_slots(const word_t<TS>* off, const int* cols, const int4& sl, unsigned n, int from,
                                          int to, int skip, int lane, const TV* x, TV* lds, F&& add) {
    if constexpr (kSplit == 1) {
        for (int j = from; j < to; ++j) {
            if (j < skip || !has_block(sl, n, j)) continue;
            TV t[5];
            slot_times<TS, TV>(off, cols, sl.x + j, lane, x, t);
            add(t);
        }
    } else {
        const int w = threadIdx.x >> 6;
        for (int j0 = from; j0 < to; j0 += kSplit) {
            const int j = j0 + w;
            if (j < to && j >= skip && has_block(sl, n, j)) {
                TV t[5];
                slot_times<TS, TV>(off, cols, sl.x + j, lane, x, t);
#pragma unroll
                for (int v = 0; v < 5; ++v) lds[(w * 5 + v) * kSellRows + lane] = t[v];
            }
            __syncthreads();
            if (w == 0)
                for (int k = 0; k < kSplit && j0 + k < to; ++k) {
                    if (j0 + k < skip || !has_block(sl, n, j0 + k)) continue;
                    TV t[5];
#pragma unroll
                    for (int v = 0; v < 5; ++v) t[v] = lds[(k * 5 + v) * kSellRows + lane];
                    add(t);
                }
            if (j0 + kSplit < to) __syncthreads();
        }
    }
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
// (slices of a colour): 24,576-cell plate (192) FP64 70 / 47 / 45 us, BF16 41 / 33 / 31;
// 93,765 cells (735) 80 / 77 / 81, 53 / 51 / 49; 156,849 cells (1,226) 132 / 116 / 116,
// 62 / 62 / 64; 196,608 cells (1,536) 157 / 153 / 160, 65 / 68 / 71; 162,000 tetrahedra
// (four colours) 157 / 151 / 166, 102 / 100 / 102; 262,144 cells (2,048) 193 / - / -, 73.
constexpr int kEightSlices = 384, kSplitSlices = 1536;
static_assert(kSplitSlices <= kMaxPartials, "a product over that many slices leaves one partial sum each");
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

}  // namespace cfdg
