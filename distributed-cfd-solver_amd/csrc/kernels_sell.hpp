// Launch wrappers of the multicolour Krylov kernels on the sliced block layout
// (kernels_sell.hip).  Blocks are passed untyped with their storage kind;
// vectors (5 values per row at (slice * 5 + v) * 64 + lane, SellArgs) are typed
// and fix the arithmetic type.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernels.hpp"
#include "kernels_linalg.hpp"

namespace cfdg {

// One matrix in the sliced layout: off-diagonal blocks, diagonal blocks, and
// the diagonal LU factors (25 entries of the LU type per row) with their pivots
// (five 3-bit row numbers per row).
struct SellMatrix {
    const void* off = nullptr;
    const void* diag = nullptr;
    int storage = kStoreF64;
    const void* lu = nullptr;
    const std::uint16_t* piv = nullptr;
};

// Elements of a vector of the layout.
inline long long sell_vector_size(int nslices) { return 5LL * kSellRows * nslices; }
// Bytes of one slot of blocks (64 blocks) in a storage type.
inline std::size_t sell_slot_bytes(int storage) {
    return storage == kStoreF64 ? 64 * 25 * 8 : (storage == kStoreF32 ? 64 * 25 * 4 : 64 * 13 * 4);
}

// LU factors with partial pivoting of the stored diagonal blocks, factorised in
// FP64 and kept in FP64 (lu_f32 = 0, FP64 blocks only) or FP32; singular takes
// the largest device row + 1 with a zero pivot.
void launch_sell_lu(const SellArgs& b, const SellMatrix& m, void* lu, int lu_f32, std::uint16_t* piv, int* singular,
                    hipStream_t s);
// y = A x in the rows of slices [first, first + count).  TV = float needs FP32
// vectors, any storage; TV = double any storage.
template <class TV>
void launch_sell_spmv(const SellArgs& b, const SellMatrix& m, int first, int count, const TV* x, TV* y, hipStream_t s,
                      const double* gate = nullptr);
// One sweep step over the slices [first, first + count) of a colour:
// z_i = D_i^-1 (r_i - sum A_ij z_j) over the row's lower blocks, or with all
// set over all its off-diagonal blocks.
template <class TV>
void launch_sell_sweep(const SellArgs& b, const SellMatrix& m, int first, int count, bool all, const TV* r, TV* z,
                       hipStream_t s, const double* gate = nullptr);
// dst (sliced) = src (5 values per cell, cell src_of[device row], or the device
// row itself when src_of is null), and back.
void launch_sell_gather(const SellArgs& b, const int* src_of, const double* src, double* dst, hipStream_t s);
void launch_sell_scatter(const SellArgs& b, const int* dst_of, const double* src, double* dst, hipStream_t s);
// Partial sums left for launch_bicg_start: 5-vectors of dot products, and of squared
// residuals.
struct SellSums {
    int dots = 0, norms = 0;
};
// Partial dot products (5 per workgroup, their number is returned): ndot 1 (v0, v1), 2
// (v0, v0) and (v1, v1), 5 (v0, v0), (v0, v1), (v2, v0), (v2, v1), (v1, v1); vectors
// that are not used repeat another.
template <class TV>
int launch_sell_dots(const SellArgs& b, int ndot, const TV* v0, const TV* v1, const TV* v2, double* partial,
                     hipStream_t s, const double* gate = nullptr);
// b = -R and x = 0 in the sliced layout, *singular = 0, with the partial sums of the
// norms and (square) of (b, b); jacobian_end: the launch directly after the Jacobian's.
SellSums launch_sell_rhs(const SellArgs& b, int ld, const double* res, double* rhs, double* x, bool square,
                         double* partial, int* singular, unsigned long long* stamp, bool jacobian_end, hipStream_t s);
// b = r in FP32, x = 0 and the partial sums of (b, b)
SellSums launch_sell_inner_rhs(const SellArgs& b, const double* r, float* rhs, float* x, double* partial,
                               hipStream_t s);
// U += du with du in the sliced layout, du also written per cell (5 values, device
// order); stamps the solve's end.
void launch_sell_state_update(const SellArgs& b, int ld, const double* du, double* U, double* du_cells,
                              unsigned long long* stamp, hipStream_t s);
// Row-major 25-entry blocks k0 .. k0 + n of a list of block codes (setup.hpp,
// sell_block_codes) from and to the sliced layout; to_csr keeps the storage
// type (block layout of precision.hpp).
void launch_sell_get_blocks(const int* code, long long n, const SellMatrix& m, double* out, hipStream_t s);
void launch_sell_set_blocks(const int* code, long long n, const double* in, void* off, void* diag, int storage,
                            hipStream_t s);
void launch_sell_to_csr(const int* code, long long n, const SellMatrix& m, void* values, hipStream_t s);

}  // namespace cfdg
