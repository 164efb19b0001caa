// Residual, time-step and Jacobian kernels (gfx950).
//
// Data: cell and face planes (structure of arrays, kernels.hpp).  Cells are
// in the device (tile) order; faces keep their mesh index.
//
//   k_primitives        U -> (p,u,v,w,T) into the cell records; boundary ghost
//                       states, one thread per boundary face
//   k_gradient_limiter  cell gradient (node-stencil least squares with the
//                       3x3 normal equations rebuilt per cell from neighbour
//                       centroids, or Green-Gauss) + MUSCL limiter, one thread
//                       per cell; k_gradient_limiter_lds is the same per cell
//                       with the tile's neighbour stencil staged in LDS
//   k_ghost_gradients   boundary ghost gradients
//   k_flux              tiled flux residual: a workgroup owns a tile of cells,
//                       evaluates each face touching the tile once into LDS,
//                       then every cell sums its faces in ascending face index
//   k_dt, k_jacobian    local time step; Picard Jacobian on the flux tiles, one
//                       thread per block row
//
// No floating-point atomics: every output element has a single writer and
// every sum has a fixed order.
#include <hip/hip_runtime.h>

#include "kernels.hpp"
#include "kernels_linalg.hpp"
#include "reduce_device.hpp"

namespace cfdg {

namespace {

constexpr int kBlock = 256;

__device__ __forceinline__ int face_owner(const MeshArgs& m, int f) { return m.fcells[f].x; }
// neighbour cell, or the ghost n_cells + (f - n_inner) of a boundary face
__device__ __forceinline__ int face_other(const MeshArgs& m, int f) { return m.fcells[f].y; }
__device__ __forceinline__ FaceRef frec(const MeshArgs& m, int f) { return FaceRef{m.fp, m.fld, f}; }
__device__ __forceinline__ CellRef crec(const FieldArgs& f, int c) { return CellRef{f.cs, f.ld, c}; }
__device__ __forceinline__ CellRefW crecw(const FieldArgs& f, int c) { return CellRefW{f.cs, f.ld, c}; }

// 1 / max((x_f - x_c) . n, 1e-14)   (boundary_traversal.hpp:98-108)
template <class FR, class CR>
__device__ __forceinline__ double rcfn_inverse(const FR& fr, const CR& cr) {
    const double rx = fr[kFC] - cr[kRC], ry = fr[kFC + 1] - cr[kRC + 1], rz = fr[kFC + 2] - cr[kRC + 2];
    const double r = rx * fr[kFN] + ry * fr[kFN + 1] + rz * fr[kFN + 2];
    return 1.0 / dmax(r, 1.0e-14);
}

__device__ __forceinline__ void cell_primitives(const MeshArgs& m, const FieldArgs& f, const NumArgs& nm, int c,
                                                double q[5]) {
    double U[5];
    for (int v = 0; v < 5; ++v) U[v] = f.U[static_cast<long long>(v) * m.nc + c];
    cons_to_prim(nm.gas, U, q);
}

// Ghost primitive states (bc/physical/*.hpp value kernels)
__device__ __forceinline__ void ghost_primitives(const MeshArgs& m, const FieldArgs& f, const NumArgs& nm,
                                                 const BcTable& bt, int bf) {
    const int fc = m.ninner + bf;
    const FaceRef fr = frec(m, fc);
    const int owner = face_owner(m, fc);
    const CellRef ri = crec(f, owner);
    const CellRefW rg = crecw(f, m.nc + bf);
    const BcDev bp = bt.bc[m.bface_bc[bf]];
    double qi[5], qg[5];
    cell_primitives(m, f, nm, owner, qi);
    const double nx = fr[kFN], ny = fr[kFN + 1], nz = fr[kFN + 2];
    switch (bp.type) {
        case kSupIn: {
            const double qf[5] = {bp.p, bp.u, bp.v, bp.w, bp.T};
            for (int v = 0; v < 5; ++v) qg[v] = 2.0 * qf[v] - qi[v];
            qg[0] = dmax(qg[0], 1.0);
            qg[4] = dmax(qg[4], 1.0);
            break;
        }
        case kSlip:
        case kSym: {
            const double vn2 = 2.0 * (qi[1] * nx + qi[2] * ny + qi[3] * nz);
            qg[1] = qi[1] - vn2 * nx;
            qg[2] = qi[2] - vn2 * ny;
            qg[3] = qi[3] - vn2 * nz;
            qg[0] = qi[0];
            qg[4] = qi[4];
            break;
        }
        case kFar: {
            double qb[5];
            bool so = false;
            farfield_state(bp, nm.gas.gamma, nm.gas.R, qi[0], qi[4], qi[1], qi[2], qi[3], nx, ny, nz, qb, so);
            if (so) {
                for (int v = 0; v < 5; ++v) qg[v] = qi[v];
            } else {
                for (int v = 0; v < 5; ++v) qg[v] = 2.0 * qb[v] - qi[v];
                qg[0] = dmax(qg[0], 1.0);
                qg[4] = dmax(qg[4], 1.0);
            }
            break;
        }
        case kNoSlip:
        case kSubIn:
            qg[0] = qi[0];
            qg[1] = 2.0 * bp.u - qi[1];
            qg[2] = 2.0 * bp.v - qi[2];
            qg[3] = 2.0 * bp.w - qi[3];
            qg[4] = 2.0 * bp.T - qi[4];
            qg[4] = dmax(qg[4], 1.0);
            break;
        case kNoSlipHF: {
            const double rinv = rcfn_inverse(fr, ri);
            qg[0] = qi[0];
            qg[1] = 2.0 * bp.u - qi[1];
            qg[2] = 2.0 * bp.v - qi[2];
            qg[3] = 2.0 * bp.w - qi[3];
            const double r = 1.0 / rinv;
            qg[4] = qi[4] + 2.0 * bp.tmp_grad * r;
            qg[4] = dmax(qg[4], 1.0);
            break;
        }
        case kSubOut:
            qg[0] = 2.0 * bp.p - qi[0];
            qg[0] = dmax(qg[0], 1.0);
            for (int v = 1; v < 5; ++v) qg[v] = qi[v];
            break;
        default:  // supersonic outlet: extrapolation
            for (int v = 0; v < 5; ++v) qg[v] = qi[v];
            break;
    }
    for (int v = 0; v < 5; ++v) rg[kRQ + v] = qg[v];
}

// U -> q for the cells (solver.hpp:185-188), the first cell_blocks workgroups, and
// the ghosts, the others: a ghost forms its owner's primitives itself, so the two
// need no order and one launch does both.
__global__ void __launch_bounds__(kBlock) k_primitives(MeshArgs m, FieldArgs f, NumArgs nm, BcTable bt,
                                                       int cell_blocks) {
    stamp_stage(f.stamp, kStampPrimitives);
    const int blk = static_cast<int>(blockIdx.x);
    if (blk >= cell_blocks) {
        const int bf = (blk - cell_blocks) * kBlock + static_cast<int>(threadIdx.x);
        if (bf < m.nf - m.ninner) ghost_primitives(m, f, nm, bt, bf);
        return;
    }
    const int c = xcd_block(blk, cell_blocks) * kBlock + static_cast<int>(threadIdx.x);
    if (c >= m.nc) return;
    double q[5];
    cell_primitives(m, f, nm, c, q);
    const CellRefW r = crecw(f, c);
    for (int v = 0; v < 5; ++v) r[kRQ + v] = q[v];
}

// Inverse of the weighted least-squares normal matrix of cell c over its
// vertex-sharing stencil (LeastSquaresCellNodeGradient::setup,
// gradient_operator.cpp:622-707): A = sum w dr dr^T + 1e-14 I with
// w = 1/max(|dr|^2, 1e-30), inverted by the adjugate (zero when |det| <= 1e-14).
// A is symmetric and so is its adjugate inverse entry for entry, so six values
// (00, 01, 02, 11, 12, 22) hold it.
__device__ __forceinline__ void lsq_inverse(const MeshArgs& m, const FieldArgs& f, int c, double out[6]) {
    const CellRef rc = crec(f, c);
    const double x0 = rc[kRC], y0 = rc[kRC + 1], z0 = rc[kRC + 2];
    double A0 = 0.0, A1 = 0.0, A2 = 0.0, A4 = 0.0, A5 = 0.0, A8 = 0.0;
    for (int j = m.ccn_off[c]; j < m.ccn_off[c + 1]; ++j) {
        const CellRef rn = crec(f, m.ccn[j]);
        const double dx = rn[kRC] - x0, dy = rn[kRC + 1] - y0, dz = rn[kRC + 2] - z0;
        const double r2 = dx * dx + dy * dy + dz * dz;
        const double w = 1.0 / dmax(r2, 1.0e-30);
        A0 += w * dx * dx;
        A1 += w * dx * dy;
        A2 += w * dx * dz;
        A4 += w * dy * dy;
        A5 += w * dy * dz;
        A8 += w * dz * dz;
    }
    const double A3 = A1, A6 = A2, A7 = A5;
    A0 += 1.0e-14;
    A4 += 1.0e-14;
    A8 += 1.0e-14;
    for (int k = 0; k < 6; ++k) out[k] = 0.0;
    const double det = A0 * (A4 * A8 - A5 * A7) - A1 * (A3 * A8 - A5 * A6) + A2 * (A3 * A7 - A4 * A6);
    if (!(fabs(det) <= 1.0e-14)) {
        const double id = 1.0 / det;
        out[0] = (A4 * A8 - A5 * A7) * id;
        out[1] = (A2 * A7 - A1 * A8) * id;
        out[2] = (A1 * A5 - A2 * A4) * id;
        out[3] = (A0 * A8 - A2 * A6) * id;
        out[4] = (A2 * A3 - A0 * A5) * id;
        out[5] = (A0 * A4 - A1 * A3) * id;
    }
}

// Set-up: the inverse normal matrix of every cell into planes kRInv..kRInv+5
// (centroids only, so once per mesh).
__global__ void __launch_bounds__(kBlock) k_lsq_setup(MeshArgs m, FieldArgs f) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= m.nc) return;
    double inv[6];
    lsq_inverse(m, f, c, inv);
    const CellRefW w = crecw(f, c);
    for (int k = 0; k < 6; ++k) w[kRInv + k] = inv[k];
}

// Cell gradient + MUSCL limiter of device cell c (gradient_operator.cpp:549-707,
// :197-278; muscl.hpp:26-104).  `self`, nbn(j) and nbf(j) point at 8 doubles
// laid out as the first half of a cell record (q, centroid) for the cell, its
// j-th vertex neighbour and its j-th face neighbour -- either the records in
// planes in HBM or their copies staged in LDS.
// Optional nu_tilde gradient formed in the same least-squares pass (the
// turbulence module's scalar, same coefficients, same order per term).
struct NoScalar {
    static constexpr bool kOn = false;
    __device__ double self() const { return 0.0; }
    template <class Nb>
    __device__ double nb(const Nb&) const { return 0.0; }
    __device__ void store(int, const double*) const {}
};
struct LdsScalar {
    static constexpr bool kOn = true;
    const double* s;       // LDS slots (the neighbour's slot comes with its view)
    int own;               // slot of the cell
    double* g;             // output: 3 planes of nc
    long long nc;
    __device__ double self() const { return s[own]; }
    template <class Nb>
    __device__ double nb(const Nb& rn) const { return s[rn.s]; }
    __device__ void store(int c, const double* v) const {
        g[c] = v[0];
        g[nc + c] = v[1];
        g[2 * nc + c] = v[2];
    }
};

template <class Self, class NbF, class FVec>
__device__ __forceinline__ void store_and_limit(const MeshArgs& m, const FieldArgs& f, const NumArgs& nm, int c,
                                                const Self& self, const double (&g)[5][3], NbF nbf, FVec fvec);

// fvec(e, k, x0, y0, z0, ex, ey, ez) gives x_f - x_c of the cell's k-th face
// (entry e of cf).
template <class Self, class NbN, class NbF, class FVec, class Sc = NoScalar>
__device__ __forceinline__ void gradient_limiter_cell(const MeshArgs& m, const FieldArgs& f, const NumArgs& nm, int c,
                                                      const Self& self, NbN nbn, NbF nbf, FVec fvec,
                                                      const Sc& sc = Sc{}) {
    const CellRefW rc = crecw(f, c);
    double qc[5];
    for (int v = 0; v < 5; ++v) qc[v] = self[kRQ + v];
    const double x0 = self[kRC], y0 = self[kRC + 1], z0 = self[kRC + 2];
    double g[5][3];
    for (int v = 0; v < 5; ++v) g[v][0] = g[v][1] = g[v][2] = 0.0;

    if (nm.gradient == 2) {
        // weighted least squares over the vertex-sharing stencil with the
        // inverse normal matrix of the cell (set-up time, lsq_inverse): the
        // coefficients C_j = A^-1 w_j dr_j are applied on the fly
        const int jb = m.ccn_off[c], je = m.ccn_off[c + 1];
        double gs[3] = {0.0, 0.0, 0.0};
        const double sc0 = sc.self();
        if (je > jb) {
            const CellRef ri{f.cs, f.ld, c};
            const double i0 = ri[kRInv], i1 = ri[kRInv + 1], i2 = ri[kRInv + 2], i4 = ri[kRInv + 3],
                         i5 = ri[kRInv + 4], i8 = ri[kRInv + 5];
            for (int j = jb, k = 0; j < je; ++j, ++k) {
                const auto rn = nbn(j, k);
                const double dx = rn[kRC] - x0, dy = rn[kRC + 1] - y0, dz = rn[kRC + 2] - z0;
                const double r2 = dx * dx + dy * dy + dz * dz;
                const double w = 1.0 / dmax(r2, 1.0e-30);
                const double rx = w * dx, ry = w * dy, rz = w * dz;
                const double cx = i0 * rx + i1 * ry + i2 * rz;
                const double cy = i1 * rx + i4 * ry + i5 * rz;
                const double cz = i2 * rx + i5 * ry + i8 * rz;
                for (int v = 0; v < 5; ++v) {
                    const double d = rn[kRQ + v] - qc[v];
                    g[v][0] += cx * d;
                    g[v][1] += cy * d;
                    g[v][2] += cz * d;
                }
                if constexpr (Sc::kOn) {
                    const double d = sc.nb(rn) - sc0;
                    gs[0] += cx * d;
                    gs[1] += cy * d;
                    gs[2] += cz * d;
                }
            }
        }
        if constexpr (Sc::kOn) sc.store(c, gs);
    } else {
        // Green-Gauss: the face scatter gathered per cell (both the face- and
        // cell-based variants form these sums)
        for (int e = m.cf_off[c]; e < m.cf_off[c + 1]; ++e) {
            const int fc = m.cf[e];
            const FaceRef fr = frec(m, fc);
            const int o = face_owner(m, fc);
            const int nb = face_other(m, fc);
            const double a05 = 0.5 * fr[kFA];
            const double hx = a05 * fr[kFN], hy = a05 * fr[kFN + 1], hz = a05 * fr[kFN + 2];
            const bool own = (o == c);
            const CellRef ro = crec(f, o);
            const CellRef rn = crec(f, nb);
            for (int v = 0; v < 5; ++v) {
                const double s = ro[kRQ + v] + rn[kRQ + v];
                const double fx = hx * s, fy = hy * s, fz = hz * s;
                if (own) {
                    g[v][0] += fx;
                    g[v][1] += fy;
                    g[v][2] += fz;
                } else {
                    g[v][0] -= fx;
                    g[v][1] -= fy;
                    g[v][2] -= fz;
                }
            }
        }
        const double iv = 1.0 / rc[kRVol];
        for (int v = 0; v < 5; ++v) {
            g[v][0] *= iv;
            g[v][1] *= iv;
            g[v][2] *= iv;
        }
    }
    store_and_limit(m, f, nm, c, self, g, nbf, fvec);
}

// The gradients g of device cell c stored, then the MUSCL limiter of the cell
// from them (muscl.hpp:26-104): the second half of gradient_limiter_cell.
template <class Self, class NbF, class FVec>
__device__ __forceinline__ void store_and_limit(const MeshArgs& m, const FieldArgs& f, const NumArgs& nm, int c,
                                                const Self& self, const double (&g)[5][3], NbF nbf, FVec fvec) {
    const CellRefW rc = crecw(f, c);
    double qc[5];
    for (int v = 0; v < 5; ++v) qc[v] = self[kRQ + v];
    const double x0 = self[kRC], y0 = self[kRC + 1], z0 = self[kRC + 2];
    for (int v = 0; v < 5; ++v)
        for (int d = 0; d < 3; ++d) rc[kRG + 3 * v + d] = g[v][d];

    if (!nm.muscl) return;
    double qmax[5], qmin[5];
    for (int v = 0; v < 5; ++v) qmax[v] = qmin[v] = qc[v];
    for (int j = m.ccf_off[c], k = 0; j < m.ccf_off[c + 1]; ++j, ++k) {
        const auto rn = nbf(j, k);
        for (int v = 0; v < 5; ++v) {
            const double qn = rn[kRQ + v];
            qmax[v] = dmax(qmax[v], qn);
            qmin[v] = dmin(qmin[v], qn);
        }
    }
    double ph[5] = {1.0, 1.0, 1.0, 1.0, 1.0};
    const double eps2 = nm.k3 * rc[kRVol];
    for (int e = m.cf_off[c], k = 0; e < m.cf_off[c + 1]; ++e, ++k) {
        double ex, ey, ez;
        fvec(e, k, x0, y0, z0, ex, ey, ez);
        for (int v = 0; v < 5; ++v) {
            const double df = g[v][0] * ex + g[v][1] * ey + g[v][2] * ez;
            const double dnb = (df > 0.0) ? (qmax[v] - qc[v]) : (qmin[v] - qc[v]);
            ph[v] = dmin(ph[v], limiter_phi(nm.limiter, dnb, df, eps2));
        }
    }
    for (int v = 0; v < 5; ++v) rc[kRPhi + v] = ph[v];
}

// One thread per cell, neighbours gathered from the records in HBM.
__global__ void __launch_bounds__(kBlock) k_gradient_limiter(MeshArgs m, FieldArgs f, NumArgs nm) {
    stamp_stage(f.stamp, kStampGradients);
    const int c = xcd_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
    if (c >= m.nc) return;
    gradient_limiter_cell(
        m, f, nm, c, crec(f, c), [&](int j, int) { return crec(f, m.ccn[j]); },
        [&](int j, int) { return crec(f, m.ccf[j]); },
        [&](int e, int, double x0, double y0, double z0, double& ex, double& ey, double& ez) {
            const FaceRef fr = frec(m, m.cf[e]);
            ex = fr[kFC] - x0;
            ey = fr[kFC + 1] - y0;
            ez = fr[kFC + 2] - z0;
        });
}

// Four consecutive 16-bit LDS slot indices of a stencil list, loaded as one
// 8-byte word; entry k of the chunk sits in bits 16 (k mod 4) and up.  Taking
// an entry by shifting the word (not by picking one of two 32-bit halves)
// keeps the chunk in registers: a pick between the halves by a run-time index
// was compiled into an indexed load from a stack copy.
typedef unsigned long long SlotChunk;
__device__ __forceinline__ int chunk_slot(SlotChunk ch, int k) {
    return static_cast<int>((ch >> ((k & 3) * 16)) & 0xffffULL);
}

// View of one LDS slot of the staged gradient kernel: planes 0-7 (q,
// centroid) stored as interleaved pairs like the cell planes, quantity k of
// slot s at sq[((k / 2) kSlots + s) 2 + k % 2], so one 16-byte LDS read
// brings two quantities of a neighbour.
template <int kSlots>
struct LdsSlot {
    const double* sq;
    int s;
    __device__ __forceinline__ double operator[](int k) const { return sq[((k >> 1) * kSlots + s) * 2 + (k & 1)]; }
};

// One workgroup per gradient tile (a flux tile, or a consecutive sub-range of
// one where the tile's stencil halo would not fit; blockDim.x >= its cells):
// the (q, centroid) planes of the tile's cells and of its stencil halo are
// staged once into LDS (structure of arrays, so that lanes reading different
// slots of one plane spread over the banks), then every cell reads its vertex
// and face neighbours from there.
template <bool kSA, int kSlots>
__global__ void __launch_bounds__(kTileCells) k_gradient_limiter_lds(MeshArgs m, FieldArgs f, NumArgs nm, SaArgs sa) {
    stamp_stage(f.stamp, kStampGradients);
    __shared__ __attribute__((aligned(16))) double sq[(kSA ? 9 : 8) * kSlots];  // 4 plane pairs (+ nu_tilde)
    const int t = xcd_block(blockIdx.x, gridDim.x);
    const int c0 = m.gtile_off[t], nt = m.gtile_off[t + 1] - c0;
    const int hb = m.tile_halo_off[t], ns = nt + (m.tile_halo_off[t + 1] - hb);
    // slot lists in chunks of four entries (8 bytes) per cell, consecutive
    // lanes on consecutive chunks; the first two chunks of each list are
    // loaded before the staging so that their latency overlaps it
    const bool live = static_cast<int>(threadIdx.x) < nt;
    const int nchn = (m.ccn_base[t + 1] - m.ccn_base[t]) / (4 * nt);
    const int nchf = (m.ccf_base[t + 1] - m.ccf_base[t]) / (4 * nt);
    const SlotChunk* chn = reinterpret_cast<const SlotChunk*>(m.ccn_slot + m.ccn_base[t]) + threadIdx.x;
    const SlotChunk* chf = reinterpret_cast<const SlotChunk*>(m.ccf_slot + m.ccf_base[t]) + threadIdx.x;
    SlotChunk curn = 0, nxtn = 0, curf = 0, nxtf = 0;
    if (live) {
        if (nchn > 0) curn = chn[0];
        if (nchn > 1) nxtn = chn[nt];
        if (nchf > 0) curf = chf[0];
        if (nchf > 1) nxtf = chf[nt];
    }
    for (int sl = threadIdx.x; sl < ns; sl += blockDim.x) {
        const int src = (sl < nt) ? c0 + sl : m.tile_halo[hb + sl - nt];
        for (int k = 0; k < 8; k += 2) {  // planes 0-7 = q, centroid: four 16-byte pair loads
            const double2 v = *reinterpret_cast<const double2*>(f.cs + plane_at(k, f.ld, src));
            *reinterpret_cast<double2*>(sq + ((k >> 1) * kSlots + sl) * 2) = v;
        }
        if constexpr (kSA) sq[8 * kSlots + sl] = sa.nu[src];
    }
    __syncthreads();
    if (!live) return;
    // entries are taken in order k = 0, 1, 2, ...: at each chunk boundary the
    // held next chunk becomes current and the one after it is requested
    const auto take = [&](int k, SlotChunk& cur, SlotChunk& nxt, const SlotChunk* ch, int nch) {
        if ((k & 3) == 0 && k > 0) {
            cur = nxt;
            if ((k >> 2) + 1 < nch) nxt = ch[((k >> 2) + 1) * nt];
        }
        return chunk_slot(cur, k);
    };
    const auto nbn = [&](int, int k) { return LdsSlot<kSlots>{sq, take(k, curn, nxtn, chn, nchn)}; };
    const auto nbf = [&](int, int k) { return LdsSlot<kSlots>{sq, take(k, curf, nxtf, chf, nchf)}; };
    // set-up-time face vectors, transposed per tile like the slot lists
    const long long vb = m.face_vec_base[t];
    const long long vw = (m.face_vec_base[t + 1] - vb) / (3LL * nt);
    const double* fvp = m.face_vec + vb + threadIdx.x;
    const auto fvec = [&](int, int k, double, double, double, double& ex, double& ey, double& ez) {
        ex = fvp[k * static_cast<long long>(nt)];
        ey = fvp[(vw + k) * nt];
        ez = fvp[(2 * vw + k) * nt];
    };
    if constexpr (kSA) {
        // the module's nu_tilde gradient in the same pass (k_sa_gradient's arithmetic)
        const LdsScalar sc{sq + 8 * kSlots, static_cast<int>(threadIdx.x), sa.g, m.nc};
        gradient_limiter_cell(m, f, nm, c0 + threadIdx.x, LdsSlot<kSlots>{sq, static_cast<int>(threadIdx.x)}, nbn, nbf,
                              fvec, sc);
    } else {
        gradient_limiter_cell(m, f, nm, c0 + threadIdx.x, LdsSlot<kSlots>{sq, static_cast<int>(threadIdx.x)}, nbn, nbf,
                              fvec);
    }
}

// The second half of gradient_limiter_cell for the variables var (those with on set) and
// their gradients gv of one of the two lanes of a cell: the same operations per variable.
constexpr int kRounds = 3;  // of five variables, per lane
template <class Self, class NbF, class FVec>
__device__ __forceinline__ void store_and_limit_split(const MeshArgs& m, const FieldArgs& f, const NumArgs& nm, int c,
                                                      const Self& self, const int (&var)[kRounds],
                                                      const bool (&on)[kRounds], const double (&gv)[kRounds][3],
                                                      NbF nbf, FVec fvec) {
    const CellRefW rc = crecw(f, c);
    double qc[kRounds], qmax[kRounds], qmin[kRounds], ph[kRounds];
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
        for (int d = 0; d < 3; ++d)
            if (on[r]) rc[kRG + 3 * var[r] + d] = gv[r][d];
        qc[r] = self[kRQ + var[r]];
        qmax[r] = qmin[r] = qc[r];
        ph[r] = 1.0;
    }
    if (!nm.muscl) return;
    for (int j = m.ccf_off[c], k = 0; j < m.ccf_off[c + 1]; ++j, ++k) {
        const auto rn = nbf(j, k);
#pragma unroll
        for (int r = 0; r < kRounds; ++r) {
            const double qn = rn[kRQ + var[r]];
            qmax[r] = dmax(qmax[r], qn);
            qmin[r] = dmin(qmin[r], qn);
        }
    }
    const double x0 = self[kRC], y0 = self[kRC + 1], z0 = self[kRC + 2];
    const double eps2 = nm.k3 * rc[kRVol];
    for (int e = m.cf_off[c], k = 0; e < m.cf_off[c + 1]; ++e, ++k) {
        double ex, ey, ez;
        fvec(e, k, x0, y0, z0, ex, ey, ez);
#pragma unroll
        for (int r = 0; r < kRounds; ++r) {
            const double df = gv[r][0] * ex + gv[r][1] * ey + gv[r][2] * ez;
            const double dnb = (df > 0.0) ? (qmax[r] - qc[r]) : (qmin[r] - qc[r]);
            ph[r] = dmin(ph[r], limiter_phi(nm.limiter, dnb, df, eps2));
        }
    }
#pragma unroll
    for (int r = 0; r < kRounds; ++r)
        if (on[r]) rc[kRPhi + var[r]] = ph[r];
}

// The neighbouring lane's value (lanes 2 k and 2 k + 1 exchange).
__device__ __forceinline__ double other_lane(double v) {
    constexpr int kSwapPairs = 0xb1;  // quad permutation 1, 0, 3, 2
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(b), kSwapPairs, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(b >> 32), kSwapPairs, 0xf, 0xf, false);
    return __longlong_as_double((static_cast<long long>(hi) << 32) | static_cast<unsigned>(lo));
}

// The staged forms with two lanes per cell (adjacent lanes, workgroups of up to 512), where
// one lane per cell leaves too few waves to hide the stencil loop's latencies
// (launch_gradient_limiter).  Node LSQ only (the only gradient the staged forms serve).
//
// Wide: the lanes split the cell's vertex stencil by chunks of four entries (lane h takes
// chunks h, h + 2, ...), each adding its entries in stencil order with the arithmetic of
// gradient_limiter_cell; the two lanes' sums are then added.  The limiter's variables
// are split over the lanes.
//
// Narrow: the lanes split the variables, lane 0 the first three, lane 1 the others (and
// nu_tilde), and each adds every entry in stencil order; the entries' coefficients, with
// the division the larger part of the work, are formed by the lanes in turn and
// exchanged.  The sums are those of the one-lane form that takes over beyond few tiles, so
// a cell's gradient does not depend on how many tiles the mesh has.
template <bool kSA, int kSlots>
__global__ void __launch_bounds__(2 * kTileCells) k_gradient_limiter_lanes(MeshArgs m, FieldArgs f, NumArgs nm,
                                                                           SaArgs sa) {
    constexpr bool kByVariable = kSlots == kGradSlots;
    constexpr int kStep = kByVariable ? 1 : 2;  // chunks of the stencil from one of a lane's to the next
    stamp_stage(f.stamp, kStampGradients);
    __shared__ __attribute__((aligned(16))) double sq[(kSA ? 9 : 8) * kSlots];
    const int t = xcd_block(blockIdx.x, gridDim.x);
    const int c0 = m.gtile_off[t], nt = m.gtile_off[t + 1] - c0;
    const int hb = m.tile_halo_off[t], ns = nt + (m.tile_halo_off[t + 1] - hb);
    const int cell = static_cast<int>(threadIdx.x) / 2, h = static_cast<int>(threadIdx.x) % 2;
    const bool live = cell < nt;
    const int nchn = (m.ccn_base[t + 1] - m.ccn_base[t]) / (4 * nt);
    const SlotChunk* chn = reinterpret_cast<const SlotChunk*>(m.ccn_slot + m.ccn_base[t]) + cell;
    // this lane's first two vertex-slot chunks, requested before the staging
    const int first = kByVariable ? 0 : h;
    SlotChunk cur = 0, nxt = 0;
    if (live) {
        if (first < nchn) cur = chn[first * nt];
        if (first + kStep < nchn) nxt = chn[(first + kStep) * nt];
    }
    for (int sl = threadIdx.x; sl < ns; sl += blockDim.x) {
        const int src = (sl < nt) ? c0 + sl : m.tile_halo[hb + sl - nt];
        for (int k = 0; k < 8; k += 2) {
            const double2 v = *reinterpret_cast<const double2*>(f.cs + plane_at(k, f.ld, src));
            *reinterpret_cast<double2*>(sq + ((k >> 1) * kSlots + sl) * 2) = v;
        }
        if constexpr (kSA) sq[8 * kSlots + sl] = sa.nu[src];
    }
    __syncthreads();
    const int c = c0 + cell;
    const LdsSlot<kSlots> self{sq, cell};
    int var[kRounds];
    bool on[kRounds];
    double gv[kRounds][3], gs[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
        const int v = kByVariable ? 3 * h + r : h + 2 * r;
        on[r] = v < 5;
        var[r] = on[r] ? v : 4;
        gv[r][0] = gv[r][1] = gv[r][2] = 0.0;
    }
    const double x0 = self[kRC], y0 = self[kRC + 1], z0 = self[kRC + 2];
    const double sc0 = kSA ? sq[8 * kSlots + cell] : 0.0;
    const CellRef ri{f.cs, f.ld, c};
    const int cnt = live ? m.ccn_off[c + 1] - m.ccn_off[c] : 0;
    double inv[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    if (live)
        for (int k = 0; k < 6; ++k) inv[k] = ri[kRInv + k];
    // the coefficients of the stencil entry in a slot
    const auto coefficients = [&](int slot, double k[3]) {
        const LdsSlot<kSlots> rn{sq, slot};
        const double dx = rn[kRC] - x0, dy = rn[kRC + 1] - y0, dz = rn[kRC + 2] - z0;
        const double r2 = dx * dx + dy * dy + dz * dz;
        const double wgt = 1.0 / dmax(r2, 1.0e-30);
        const double rx = wgt * dx, ry = wgt * dy, rz = wgt * dz;
        k[0] = inv[0] * rx + inv[1] * ry + inv[2] * rz;
        k[1] = inv[1] * rx + inv[3] * ry + inv[4] * rz;
        k[2] = inv[2] * rx + inv[4] * ry + inv[5] * rz;
    };
    if constexpr (kByVariable) {
        // where the lane's values lie in a slot; lane 1's third is nu_tilde, in a plane of its own
        int at[kRounds], stride[kRounds];
        double q0[kRounds];
#pragma unroll
        for (int r = 0; r < kRounds; ++r) {
            const int k = kRQ + var[r];
            const bool scalar = kSA && !on[r];
            at[r] = scalar ? 8 * kSlots : (k >> 1) * 2 * kSlots + (k & 1);
            stride[r] = scalar ? 1 : 2;
            q0[r] = sq[at[r] + stride[r] * cell];
        }
        for (int q = 0; 4 * q < cnt; ++q) {
            const SlotChunk ch = cur;
            cur = nxt;
            if (q + 2 < nchn) nxt = chn[(q + 2) * nt];
            for (int e = 0; e < 4 && 4 * q + e < cnt; e += 2) {  // the lanes of a cell together
                const bool both = 4 * q + e + 1 < cnt;
                double mine[3], theirs[3];
                coefficients(chunk_slot(ch, both ? e + h : e), mine);
#pragma unroll
                for (int d = 0; d < 3; ++d) theirs[d] = other_lane(mine[d]);
                for (int u = 0; u < (both ? 2 : 1); ++u) {
                    const int slot = chunk_slot(ch, e + u);
#pragma unroll
                    for (int r = 0; r < kRounds; ++r) {
                        const double dq = sq[at[r] + stride[r] * slot] - q0[r];
#pragma unroll
                        for (int d = 0; d < 3; ++d) gv[r][d] += (u == h ? mine[d] : theirs[d]) * dq;
                    }
                }
            }
        }
        if constexpr (kSA)
            for (int d = 0; d < 3; ++d) gs[d] = gv[kRounds - 1][d];
    } else {
        double g[5][3], qc[5];
        for (int v = 0; v < 5; ++v) {
            g[v][0] = g[v][1] = g[v][2] = 0.0;
            qc[v] = self[kRQ + v];
        }
        for (int q = h; 4 * q < cnt; q += kStep) {
            const SlotChunk ch = cur;
            cur = nxt;
            if (q + 2 * kStep < nchn) nxt = chn[(q + 2 * kStep) * nt];
            for (int e = 0; e < 4 && 4 * q + e < cnt; ++e) {
                const int slot = chunk_slot(ch, e);
                const LdsSlot<kSlots> rn{sq, slot};
                double k[3];
                coefficients(slot, k);
                for (int v = 0; v < 5; ++v) {
                    const double d = rn[kRQ + v] - qc[v];
                    for (int x = 0; x < 3; ++x) g[v][x] += k[x] * d;
                }
                if constexpr (kSA) {
                    const double d = sq[8 * kSlots + slot] - sc0;
                    for (int x = 0; x < 3; ++x) gs[x] += k[x] * d;
                }
            }
        }
        // the lanes' sums added (every lane takes part)
        for (int v = 0; v < 5; ++v)
            for (int d = 0; d < 3; ++d) g[v][d] += other_lane(g[v][d]);
        if constexpr (kSA)
            for (int d = 0; d < 3; ++d) gs[d] += other_lane(gs[d]);
#pragma unroll
        for (int r = 0; r < kRounds; ++r)
            for (int d = 0; d < 3; ++d) {
                gv[r][d] = g[0][d];
                for (int w = 1; w < 5; ++w) gv[r][d] = (var[r] == w) ? g[w][d] : gv[r][d];
            }
    }
    if (!live) return;
    if constexpr (kSA) {
        const long long nc = m.nc;
        if (h == 1) {
            sa.g[c] = gs[0];
            sa.g[nc + c] = gs[1];
            sa.g[2 * nc + c] = gs[2];
        }
    }
    // the limiter's face neighbours and face vectors, in order, as the one-lane form reads them
    const int nchf = (m.ccf_base[t + 1] - m.ccf_base[t]) / (4 * nt);
    const SlotChunk* chf = reinterpret_cast<const SlotChunk*>(m.ccf_slot + m.ccf_base[t]) + cell;
    SlotChunk curf = 0, nxtf = 0;
    if (nchf > 0) curf = chf[0];
    if (nchf > 1) nxtf = chf[nt];
    const auto nbf = [&](int, int k) {
        if ((k & 3) == 0 && k > 0) {
            curf = nxtf;
            if ((k >> 2) + 1 < nchf) nxtf = chf[((k >> 2) + 1) * nt];
        }
        return LdsSlot<kSlots>{sq, chunk_slot(curf, k)};
    };
    const long long vb = m.face_vec_base[t];
    const long long vw = (m.face_vec_base[t + 1] - vb) / (3LL * nt);
    const double* fvp = m.face_vec + vb + cell;
    const auto fvec = [&](int, int k, double, double, double, double& ex, double& ey, double& ez) {
        ex = fvp[k * static_cast<long long>(nt)];
        ey = fvp[(vw + k) * nt];
        ez = fvp[(2 * vw + k) * nt];
    };
    store_and_limit_split(m, f, nm, c, self, var, on, gv, nbf, fvec);
}

__device__ __forceinline__ void grad_dirichlet(double* g, const double* gi, double qin, double qfix, double nx,
                                               double ny, double nz, double rinv) {
    const double ddn = (qfix - qin) * rinv;
    const double gn = gi[0] * nx + gi[1] * ny + gi[2] * nz;
    const double fac = 2.0 * (ddn - gn);
    g[0] = gi[0] + fac * nx;
    g[1] = gi[1] + fac * ny;
    g[2] = gi[2] + fac * nz;
}

__device__ __forceinline__ void grad_neumann(double* g, const double* gi, double fixed, double nx, double ny,
                                             double nz) {
    const double gn = gi[0] * nx + gi[1] * ny + gi[2] * nz;
    const double fac = 2.0 * (fixed - gn);
    g[0] = gi[0] + fac * nx;
    g[1] = gi[1] + fac * ny;
    g[2] = gi[2] + fac * nz;
}

__device__ __forceinline__ void grad_slip(double* g, const double* gi, double qin, double qgh, double nx, double ny,
                                          double nz, double rinv) {
    const double gn = gi[0] * nx + gi[1] * ny + gi[2] * nz;
    const double ddn = 0.5 * (qgh - qin) * rinv;
    const double fac = 2.0 * (ddn - gn);
    g[0] = gi[0] + fac * nx;
    g[1] = gi[1] + fac * ny;
    g[2] = gi[2] + fac * nz;
}

// Ghost gradients (bc/physical/*.hpp gradient kernels, boundary_gradients.hpp)
__global__ void __launch_bounds__(kBlock) k_ghost_gradients(MeshArgs m, FieldArgs f, NumArgs nm, BcTable bt) {
    stamp_stage(f.stamp, kStampGhostGradients);
    const int bf = blockIdx.x * blockDim.x + threadIdx.x;
    const int nbf = m.nf - m.ninner;
    if (bf >= nbf) return;
    const int fc = m.ninner + bf;
    const FaceRef fr = frec(m, fc);
    const CellRef ri = crec(f, face_owner(m, fc));
    const CellRefW rg = crecw(f, m.nc + bf);
    const BcDev bp = bt.bc[m.bface_bc[bf]];
    const double nx = fr[kFN], ny = fr[kFN + 1], nz = fr[kFN + 2];
    const double rinv = rcfn_inverse(fr, ri);
    double gi[5][3], go[5][3], qi[5];
    for (int v = 0; v < 5; ++v) {
        qi[v] = ri[kRQ + v];
        for (int d = 0; d < 3; ++d) go[v][d] = gi[v][d] = ri[kRG + 3 * v + d];
    }
    switch (bp.type) {
        case kSupIn: {
            const double qf[5] = {bp.p, bp.u, bp.v, bp.w, bp.T};
            for (int v = 0; v < 5; ++v) grad_dirichlet(go[v], gi[v], qi[v], qf[v], nx, ny, nz, rinv);
            break;
        }
        case kSlip:
        case kSym:
            grad_neumann(go[0], gi[0], 0.0, nx, ny, nz);
            for (int v = 1; v < 4; ++v) grad_slip(go[v], gi[v], qi[v], rg[kRQ + v], nx, ny, nz, rinv);
            grad_neumann(go[4], gi[4], 0.0, nx, ny, nz);
            break;
        case kFar: {
            double qb[5];
            bool so = false;
            farfield_state(bp, nm.gas.gamma, nm.gas.R, qi[0], qi[4], qi[1], qi[2], qi[3], nx, ny, nz, qb, so);
            if (!so)
                for (int v = 0; v < 5; ++v) grad_dirichlet(go[v], gi[v], qi[v], qb[v], nx, ny, nz, rinv);
            break;
        }
        case kNoSlip:
        case kSubIn: {
            const double qw[4] = {bp.u, bp.v, bp.w, bp.T};
            for (int v = 1; v < 5; ++v) grad_dirichlet(go[v], gi[v], qi[v], qw[v - 1], nx, ny, nz, rinv);
            break;
        }
        case kNoSlipHF: {
            const double qw[3] = {bp.u, bp.v, bp.w};
            for (int v = 1; v < 4; ++v) grad_dirichlet(go[v], gi[v], qi[v], qw[v - 1], nx, ny, nz, rinv);
            grad_neumann(go[4], gi[4], bp.tmp_grad, nx, ny, nz);
            break;
        }
        case kSubOut:
            grad_dirichlet(go[0], gi[0], qi[0], bp.p, nx, ny, nz, rinv);
            break;
        default:  // supersonic outlet: extrapolation
            break;
    }
    for (int v = 0; v < 5; ++v)
        for (int d = 0; d < 3; ++d) rg[kRG + 3 * v + d] = go[v][d];
}

// Inviscid + viscous flux of one face times its area, and its spectral-radius
// contribution (residual_kernel.hpp:183-240 / 245-300 for one face, with the
// MUSCL states of muscl.hpp:108-157).
// fr views the face's planes, (c0, c1) = (owner, neighbour or ghost).
// r0 / r1 view the owner's and the other cell's planes (in HBM or staged in
// LDS), mutL / mutR are their eddy viscosities (kEddy = false: none, both 0).
// The owner -> neighbour centroid vector and its inverse length are formed
// here with the operations of face_distances (aux_geometry.cpp:11-51,120-156),
// so they equal the mesh-order face planes bit for bit.
template <bool kEddy, class FR, class R0, class R1, class ML, class MR>
__device__ __forceinline__ void face_flux(const NumArgs& nm, const FR& fr, bool inner, const R0& r0, const R1& r1,
                                          const ML& mut0, const MR& mut1, double F[5], double& lam_f) {
    const double nx = fr[kFN], ny = fr[kFN + 1], nz = fr[kFN + 2], A = fr[kFA];
    double qL[5], qR[5];
    if (inner && nm.muscl) {
        const double fx = fr[kFC], fy = fr[kFC + 1], fz = fr[kFC + 2];
        const double d0x = fx - r0[kRC], d0y = fy - r0[kRC + 1], d0z = fz - r0[kRC + 2];
        const double d1x = fx - r1[kRC], d1y = fy - r1[kRC + 1], d1z = fz - r1[kRC + 2];
        for (int v = 0; v < 5; ++v) {
            const double dot0 = r0[kRG + 3 * v] * d0x + r0[kRG + 3 * v + 1] * d0y + r0[kRG + 3 * v + 2] * d0z;
            qL[v] = r0[kRQ + v] + r0[kRPhi + v] * dot0;
            const double dot1 = r1[kRG + 3 * v] * d1x + r1[kRG + 3 * v + 1] * d1y + r1[kRG + 3 * v + 2] * d1z;
            qR[v] = r1[kRQ + v] + r1[kRPhi + v] * dot1;
        }
    } else {
        for (int v = 0; v < 5; ++v) {
            qL[v] = r0[kRQ + v];
            qR[v] = r1[kRQ + v];
        }
    }
    double UL[5], UR[5];
    prim_to_cons(nm.gas, qL, UL);
    prim_to_cons(nm.gas, qR, UR);
    double smax = 0.0;
    hllc_flux(nm.gas, UL, UR, nx, ny, nz, A, F, smax);
    lam_f = A * smax;
    if (nm.viscous) {
        double qa[5], qb[5], ga[12], gb[12];
        for (int v = 0; v < 5; ++v) {
            qa[v] = r0[kRQ + v];
            qb[v] = r1[kRQ + v];
        }
        for (int k = 0; k < 12; ++k) {
            ga[k] = r0[kRG + 3 + k];
            gb[k] = r1[kRG + 3 + k];
        }
        double dvx, dvy, dvz, inv_d;
        if (inner) {
            const double ex = r1[kRC] - r0[kRC], ey = r1[kRC + 1] - r0[kRC + 1], ez = r1[kRC + 2] - r0[kRC + 2];
            dvx = ex;
            dvy = ey;
            dvz = ez;
            inv_d = 1.0 / sqrt(ex * ex + ey * ey + ez * ez);
        } else {
            const double ex = fr[kFC] - r0[kRC], ey = fr[kFC + 1] - r0[kRC + 1], ez = fr[kFC + 2] - r0[kRC + 2];
            dvx = 2.0 * ex;
            dvy = 2.0 * ey;
            dvz = 2.0 * ez;
            inv_d = 1.0 / sqrt(4.0 * ex * ex + 4.0 * ey * ey + 4.0 * ez * ez);
        }
        double Fv[5];
        double lv = 0.0;
        const double mutL = kEddy ? mut0() : 0.0, mutR = kEddy ? mut1() : 0.0;  // read where they are used
        viscous_flux<kEddy>(nm.gas, inv_d, dvx, dvy, dvz, qa, qb, ga, gb, mutL, mutR, nx, ny, nz, A, Fv, lv);
        for (int v = 1; v < 5; ++v) F[v] += Fv[v];
        lam_f += lv;
    }
}

// View of a tile cell's planes staged in LDS: planes 0 .. kFluxPlanes-1 in
// the pair layout of the cell planes with a stride of kTileCells slots.
constexpr int kFluxPlanes = 30;  // q, centroid, limiter, volume, gradients (plane 29 unused)
struct LdsRec {
    const double* s;
    int i;  // slot = device id - tile start
    __device__ __forceinline__ double operator[](int k) const { return s[((k >> 1) * kTileCells + i) * 2 + (k & 1)]; }
};

// One entry of the tile face-list stream (non-temporal loads); the centroid's
// z, which shares its 16-byte pair with the packed cell ids, is held by value.
struct TileFaceRef {
    const double* b;
    long long ld;
    int e;
    double fz;
    __device__ __forceinline__ double operator[](int k) const {
        if (k == kFC + 2) return fz;
        const double* base = b + static_cast<long long>(k >> 1) * 2 * ld;
        return __builtin_nontemporal_load(base + (2u * static_cast<unsigned>(e) + static_cast<unsigned>(k & 1)));
    }
};

// Tiled flux residual: each face touching the tile is evaluated once (face-
// parallel, one face per lane) and each cell then adds its faces' fluxes in
// ascending face index, with + for the owner and - for the neighbour
// (residual_kernel.hpp:175-306 formed as a gather; only faces on a tile
// boundary are evaluated by both adjacent tiles).  The tile's own cells are
// staged into LDS first (coalesced), so only the halo and ghost side of a
// face on the tile boundary is read from HBM; the face list is grouped by
// which cells lie in the tile, so a wave mostly takes one of the three load
// paths.  After the face phase the staging area is reused for the fluxes.
// With turbulence the kernel also records each face's mass flux F[0] (from
// the tile that owns the face's owner cell); eddy viscosity follows the
// cells (residual_kernel.hpp:229-230, 282-283).
template <bool kTurb, int kThreads>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4, 4))) k_flux(MeshArgs m, FieldArgs f, NumArgs nm) {
    stamp_stage(f.stamp, kStampFlux);
    __shared__ double sc[kFluxPlanes * kTileCells];  // staged planes, then the fluxes sF[6][kTileFaces]
    __shared__ double smut[kTurb ? kTileCells : 1];
    __shared__ int scf[kTileCells + 1 + 2 * kTileFaces];  // the tile's cf_off (rebased), then its cf_slot entries
    static_assert(6 * kTileFaces <= kFluxPlanes * kTileCells, "flux area must fit the staging area");
    constexpr int kPerLane = kTileFaces / kThreads;  // faces per lane
    const int t = xcd_block(blockIdx.x, gridDim.x);
    const int c0 = m.tile_off[t], nt = m.tile_off[t + 1] - c0;
    const int fb = m.tile_face_off[t], nfl = m.tile_face_off[t + 1] - fb;
    const int i = threadIdx.x;
    int cx[kPerLane], cy[kPerLane];
    double fz[kPerLane];
#pragma unroll
    for (int r = 0; r < kPerLane; ++r) {  // this lane's faces: cells (and index), issued before the staging loads
        const int j = i + r * kThreads;
        cx[r] = cy[r] = 0;
        fz[r] = 0.0;
        if (j < nfl) {
            typedef double pair_t __attribute__((ext_vector_type(2)));
            const pair_t w = __builtin_nontemporal_load(
                reinterpret_cast<const pair_t*>(m.tf + plane_at(kTCells - 1, m.tld, fb + j)));
            const unsigned long long ids = static_cast<unsigned long long>(__double_as_longlong(w.y));
            fz[r] = w.x;
            cx[r] = static_cast<int>(static_cast<unsigned>(ids));
            cy[r] = static_cast<int>(static_cast<unsigned>(ids >> 32));
        }
    }
    // staging of the plane pairs the face fluxes read: q (pairs 0-2), centroid
    // and limiter (2-6) for MUSCL, gradients (7-14) for MUSCL or viscous terms
    {
        const int sl = i % kTileCells, g = i / kTileCells;
        constexpr int kGroups = kThreads / kTileCells, kPairs = kFluxPlanes / 2;
        const int p_hi = (nm.muscl || nm.viscous) ? kPairs : 3;
        if (sl < nt) {
            for (int p = g; p < p_hi; p += kGroups) {
                if (p > 3 && p < 7 && !nm.muscl) continue;  // centroid (pairs 2-3) stays: viscous terms need it
                const double2 v = *reinterpret_cast<const double2*>(f.cs + plane_at(2 * p, f.ld, c0 + sl));
                *reinterpret_cast<double2*>(sc + (p * kTileCells + sl) * 2) = v;
            }
            if (kTurb && g == 0) smut[sl] = f.mut[c0 + sl];
        }
        // the cells' face slots for the gather: a contiguous range of cf_slot
        // (at most two entries per tile face); ne > 2 kTileFaces cannot occur
        const int e0 = m.cf_off[c0], ne = m.cf_off[c0 + nt] - e0;
        if (i <= nt) scf[i] = m.cf_off[c0 + i] - e0;
        for (int e = i; e < ne; e += kThreads) scf[kTileCells + 1 + e] = m.cf_slot[e0 + e];
    }
    __syncthreads();
    double F[kPerLane][6];
#pragma unroll
    for (int r = 0; r < kPerLane; ++r) {
        const int j = i + r * kThreads;
        for (int v = 0; v < 6; ++v) F[r][v] = 0.0;
        if (j >= nfl) break;  // later faces of the lane are out of range too
        const TileFaceRef fr{m.tf, m.tld, fb + j, fz[r]};
        const bool inner = cy[r] < m.nc;  // boundary faces: the other cell is a ghost
        const unsigned s0 = static_cast<unsigned>(cx[r] - c0), s1 = static_cast<unsigned>(cy[r] - c0);
        const bool in0 = s0 < static_cast<unsigned>(nt), in1 = s1 < static_cast<unsigned>(nt);
        double* Fr = F[r];
        // eddy viscosities from LDS (tile cells) or HBM (halo and ghosts)
        const int g0 = cx[r], g1 = cy[r];
        const auto lds0 = [&] { return smut[s0]; };
        const auto lds1 = [&] { return smut[s1]; };
        const auto hbm0 = [&] { return f.mut[g0]; };
        const auto hbm1 = [&] { return f.mut[g1]; };
        if (in0 && in1) {
            face_flux<kTurb>(nm, fr, inner, LdsRec{sc, static_cast<int>(s0)}, LdsRec{sc, static_cast<int>(s1)}, lds0,
                             lds1, Fr, Fr[5]);
        } else if (in0) {
            face_flux<kTurb>(nm, fr, inner, LdsRec{sc, static_cast<int>(s0)}, crec(f, g1), lds0, hbm1, Fr, Fr[5]);
        } else {
            face_flux<kTurb>(nm, fr, inner, crec(f, g0), LdsRec{sc, static_cast<int>(s1)}, hbm0, lds1, Fr, Fr[5]);
        }
        if (kTurb) f.mdot_tile[fb + j] = Fr[0];
        if (!inner)  // a boundary face lies in exactly one tile: single writer; ghost id = cells + boundary index
            for (int v = 0; v < 5; ++v) f.bflux[static_cast<long long>(cy[r] - m.nc) * 5 + v] = Fr[v];
    }
    __syncthreads();  // every read of the staged planes is done
    double* sF = sc;
#pragma unroll
    for (int r = 0; r < kPerLane; ++r) {
        const int j = i + r * kThreads;
        if (j < nfl)
            for (int v = 0; v < 6; ++v) sF[v * kTileFaces + j] = F[r][v];
    }
    __syncthreads();
    if (i >= nt) return;
    const int c = c0 + i;
    double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    double lam = 0.0;
    for (int e = scf[i]; e < scf[i + 1]; ++e) {
        const int s = scf[kTileCells + 1 + e];
        if (s >= 0) {
            for (int v = 0; v < 5; ++v) acc[v] += sF[v * kTileFaces + s];
            lam += sF[5 * kTileFaces + s];
        } else {
            const int k = -s - 1;
            for (int v = 0; v < 5; ++v) acc[v] -= sF[v * kTileFaces + k];
            lam += sF[5 * kTileFaces + k];
        }
    }
    for (int v = 0; v < 5; ++v) __builtin_nontemporal_store(acc[v], f.res + static_cast<long long>(v) * m.nc + c);
    __builtin_nontemporal_store(lam, f.lam + c);
}

// Implicit local time step and diagonal shift (solver.hpp:256-287); unsteady
// = c0 / dt of dual time stepping (0 in steady mode)
__global__ void __launch_bounds__(kBlock) k_dt(int nc, const double* cs, long long ld, const double* lam, double cfl,
                                               double unsteady, double* dt, double* alpha,
                                               unsigned long long* flux_end) {
    if (flux_end) stamp_stage(flux_end, kStampFluxEnd);
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nc) return;
    const double vol = cs[plane_at(kRVol, ld, c)];
    const double inv_cfl = 1.0 / cfl;
    const double l = dmax(lam[c], 1.0e-14);
    dt[c] = cfl * vol / l;
    alpha[c] = (l * inv_cfl) + (vol * unsteady);
}

// Mesh-order face mass flux from the tile-order copy: entry of each face in
// the face list of the tile that holds its owner
__global__ void __launch_bounds__(kBlock) k_gather_mdot(int nf, const int* face_entry, const double* mdot_tile,
                                                        double* mdot) {
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= nf) return;
    mdot[f] = mdot_tile[face_entry[f]];
}

// Output fields of the solution files (Solver::write_fields, solver.hpp:856-878):
// rho, u, v, w, p = (gamma - 1) rho e (state_conversions.hpp:12-25), Mach =
// |rho v| / (rho a) with a = sqrt(gamma p / rho); out = 6 planes of nc
__global__ void __launch_bounds__(kBlock) k_output_fields(int nc, Gas g, const double* U, double* out) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nc) return;
    double u[5];
    for (int v = 0; v < 5; ++v) u[v] = U[static_cast<long long>(v) * nc + c];
    const double r = u[0];
    const double inv_rho = 1.0 / r;
    const double q2 = (u[1] * u[1] + u[2] * u[2] + u[3] * u[3]) * (inv_rho * inv_rho);
    const double e = (u[4] * inv_rho) - 0.5 * q2;
    const double p = (g.gamma - 1.0) * r * e;
    const double a = sqrt(g.gamma * p / r);
    double* o = out + c;
    o[0] = r;
    o[static_cast<long long>(nc)] = u[1] / r;
    o[2LL * nc] = u[2] / r;
    o[3LL * nc] = u[3] / r;
    o[4LL * nc] = p;
    o[5LL * nc] = sqrt(u[1] * u[1] + u[2] * u[2] + u[3] * u[3]) / (r * a);
}

// Five planes of nc between mesh order and device order: dst[r] = src[map[r]]
// (mesh cell of a device row), or back, dst[map[r]] = src[r].  A tile's rows are
// runs of neighbouring mesh cells, so either side falls in few cache lines.
template <bool kToDevice>
__global__ void __launch_bounds__(kBlock) k_permute_planes(int nc, const int* map, const double* src, double* dst) {
    const int r = xcd_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
    if (r >= nc) return;
    const int o = map[r];
    for (int v = 0; v < 5; ++v) {
        const long long p = static_cast<long long>(v) * nc;
        if (kToDevice)
            dst[p + r] = src[p + o];
        else
            dst[p + o] = src[p + r];
    }
}

// Forward Euler step in one pass over the residual: local time step alpha = dt / V
// = CFL / lambda (solver.hpp:278-285), U <- U - alpha R (update_ops.hpp:28-44) and
// the residual's squares (solver.hpp:740-756), summed as k_res_sq does.  Bound: HBM
// (three kernels read the residual twice and alpha back: 80 us at 2.1M cells).
__global__ void __launch_bounds__(kBlock) k_explicit_step(int nc, const double* cs, long long ld, const double* lam,
                                                          double cfl, const double* res, double* dt, double* alpha,
                                                          double* U, double* partial, unsigned long long* stamp) {
    __shared__ double lds[kBlock / 64 * 5];
    stamp_stage(stamp, kStampFluxEnd);
    double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    const int stride = static_cast<int>(gridDim.x * blockDim.x);
    for (int c = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x); c < nc; c += stride) {
        const double l = dmax(lam[c], 1.0e-14);
        const double a = cfl / l;
        dt[c] = a * cs[plane_at(kRVol, ld, c)];
        alpha[c] = a;
        for (int v = 0; v < 5; ++v) {
            const long long k = static_cast<long long>(v) * nc + c;
            const double r = res[k];
            acc[v] += r * r;
            U[k] = U[k] - a * r;
        }
    }
    const double s = block_sums(acc, 5, lds);
    if (threadIdx.x < 5) partial[blockIdx.x * 5 + threadIdx.x] = s;
}

__global__ void k_stamp(unsigned long long* stamp, int k, int k2) {
    stamp_stage(stamp, k);
    if (k2 >= 0) stamp_stage(stamp, k2);
}

// BDF pseudo-source of dual time stepping, R += V (c0 U + c1 U^n [+ c2 U^{n-1}])
// (solver.hpp:546-575); U^n, U^{n-1} as 5 planes of nc
__global__ void __launch_bounds__(kBlock) k_unsteady_source(int nc, const double* cs, long long ld, int bdf,
                                                            double inv_dt, const double* U, const double* Un,
                                                            const double* Unm1, double* res) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nc) return;
    const double vol = cs[plane_at(kRVol, ld, c)];
    for (int v = 0; v < 5; ++v) {
        const long long k = static_cast<long long>(v) * nc + c;
        if (bdf == 2) {
            const double c0 = 1.5 * inv_dt, c1 = -2.0 * inv_dt, c2 = 0.5 * inv_dt;
            res[k] += vol * (c0 * U[k] + c1 * Un[k] + c2 * Unm1[k]);
        } else {
            const double c0 = 1.0 * inv_dt, c1 = -1.0 * inv_dt;
            res[k] += vol * (c0 * U[k] + c1 * Un[k]);
        }
    }
}

// Stores one 5x5 block (values v, sign +1 or -1 applied as 0.0 + v / 0.0 - v,
// or as is) in the sliced layout: its words at dst, dst + 64, ...; the lanes of a wave
// write consecutive words.
template <class TS>
__device__ __forceinline__ void store_sell_block(typename SellLayout<TS>::word* dst, const double v[25], int sign) {
    const auto signed_value = [&](int k) { return sign > 0 ? 0.0 + v[k] : (sign < 0 ? 0.0 - v[k] : v[k]); };
    if constexpr (sizeof(TS) == sizeof(bf16)) {
#pragma unroll
        for (int q = 0; q < SellLayout<TS>::words; ++q) {
            const std::uint32_t lo = cvt<bf16>(signed_value(2 * q)).u;
            const std::uint32_t hi = 2 * q + 1 < 25 ? cvt<bf16>(signed_value(2 * q + 1)).u : 0;
            dst[q * kSellRows] = lo | (hi << 16);
        }
    } else {
#pragma unroll
        for (int k = 0; k < 25; ++k) dst[k * kSellRows] = cvt<TS>(signed_value(k));
    }
}

// J += Jv (plus) or J -= Jv for the dense viscous block Jv of
// viscous_jacobian_dense, touching only its 11 nonzero entries.  Adding the
// pattern's zeros would change no stored value: it can only turn a -0 entry
// into +0, and the diagonal sums start at +0 while every off-diagonal store
// forms 0 + v or 0 - v.
__device__ __forceinline__ void add_viscous_jacobian(const double m[9], bool plus, double J[25]) {
    const double d[11] = {m[0], m[3], m[1], m[3], m[2], m[3], m[4], m[5], m[6], m[7], m[8]};
    const int at[11] = {5, 6, 10, 12, 15, 18, 20, 21, 22, 23, 24};
    for (int k = 0; k < 11; ++k) J[at[k]] = plus ? J[at[k]] + d[k] : J[at[k]] - d[k];
}

// One face of a Jacobian row (jacobian_kernel.hpp:104-270 for one face): the
// row cell's state from LDS, the face from the tile face stream, the other
// cell from LDS (tile cell) or the cell planes (halo cell, ghost).  Adds the
// face's dF of the row's own side to dg (+ dFL as owner, - dFR as
// neighbour); at an interior face returns true with the other side's dF in J
// (dFR as owner, dFL as neighbour: the caller stores + J or - J).
template <bool kTurb>
__device__ __forceinline__ bool jacobian_face(const MeshArgs& m, const FieldArgs& f, const NumArgs& nm,
                                              const double* sq, const double* smut, int i, int c0, int nt, int j,
                                              bool own, double dg[25], double J[25]) {
    typedef double pair_t __attribute__((ext_vector_type(2)));
    // the row cell's state, re-read from LDS per face (fewer live registers)
    double qc[5], Uc[5];
    for (int v = 0; v < 5; ++v) qc[v] = sq[v * kTileCells + i];
    prim_to_cons(nm.gas, qc, Uc);
    const pair_t n01 = *reinterpret_cast<const pair_t*>(m.tf + plane_at(kFN, m.tld, j));
    const pair_t n2a = *reinterpret_cast<const pair_t*>(m.tf + plane_at(kFN + 2, m.tld, j));
    const pair_t zid = *reinterpret_cast<const pair_t*>(m.tf + plane_at(kTCells - 1, m.tld, j));
    const double nx = n01.x, ny = n01.y, nz = n2a.x, A = n2a.y;
    const unsigned long long ids = static_cast<unsigned long long>(__double_as_longlong(zid.y));
    const int cx = static_cast<int>(static_cast<unsigned>(ids));
    const int cy = static_cast<int>(static_cast<unsigned>(ids >> 32));
    const bool inner = cy < m.nc;  // boundary faces: the other cell is a ghost
    const int oc = own ? cy : cx;
    const unsigned so = static_cast<unsigned>(oc - c0);
    const bool oin = so < static_cast<unsigned>(nt);
    double qo[5], xo[3];
    double mo = 0.0;
    if (oin) {
        for (int v = 0; v < 5; ++v) qo[v] = sq[v * kTileCells + so];
        for (int d = 0; d < 3; ++d) xo[d] = sq[(5 + d) * kTileCells + so];
        if (kTurb) mo = smut[so];
    } else {
        const CellRef r = crec(f, oc);
        for (int v = 0; v < 5; ++v) qo[v] = r[kRQ + v];
        for (int d = 0; d < 3; ++d) xo[d] = r[kRC + d];
        if (kTurb) mo = f.mut[oc];
    }
    double Uo[5];
    prim_to_cons(nm.gas, qo, Uo);
    double qL[5], qR[5], UL[5], UR[5];
    for (int v = 0; v < 5; ++v) {
        qL[v] = own ? qc[v] : qo[v];
        qR[v] = own ? qo[v] : qc[v];
        UL[v] = own ? Uc[v] : Uo[v];
        UR[v] = own ? Uo[v] : Uc[v];
    }
    const double smax = hllc_smax(nm.gas, UL, UR, nx, ny, nz);
    const double half_area = 0.5 * A;
    const double diss = 0.5 * smax * A;
    double vm[9];
    if (nm.viscous) {
        // owner -> neighbour centroid vector and its inverse length with the
        // operations of face_distances (aux_geometry.cpp:11-51, 120-156)
        const double xc0 = sq[5 * kTileCells + i], xc1 = sq[6 * kTileCells + i], xc2 = sq[7 * kTileCells + i];
        double inv_d;
        if (inner) {
            const double ax = own ? xc0 : xo[0], ay = own ? xc1 : xo[1], az = own ? xc2 : xo[2];
            const double bx = own ? xo[0] : xc0, by = own ? xo[1] : xc1, bz = own ? xo[2] : xc2;
            const double ex = bx - ax, ey = by - ay, ez = bz - az;
            inv_d = 1.0 / sqrt(ex * ex + ey * ey + ez * ez);
        } else {  // the row cell owns a boundary face
            const pair_t fxy = *reinterpret_cast<const pair_t*>(m.tf + plane_at(kFC, m.tld, j));
            const double ex = fxy.x - xc0, ey = fxy.y - xc1, ez = zid.x - xc2;
            inv_d = 1.0 / sqrt(4.0 * ex * ex + 4.0 * ey * ey + 4.0 * ez * ez);
        }
        // jacobian_kernel.hpp:156-157, 209-210, 252-254: the ghost side carries no eddy viscosity
        const double mc = kTurb ? smut[i] : 0.0;
        const double mutL = kTurb ? (own ? mc : mo) : 0.0;
        const double mutR = (kTurb && inner) ? (own ? mo : mc) : 0.0;
        viscous_jacobian_entries<kTurb>(nm.gas, inv_d, qL, qR, mutL, mutR, A, vm);
    }
    // own side, dFL = 0.5 A J(UL) + diss I (+ viscous) as owner, dFR = 0.5 A
    // J(UR) - diss I (- viscous) as neighbour
    euler_jacobian_scaled(nm.gas, Uc, nx, ny, nz, half_area, J);
    for (int k = 0; k < 5; ++k) J[k * 6] = own ? (J[k * 6] + diss) : (J[k * 6] - diss);
    if (nm.viscous) add_viscous_jacobian(vm, own, J);
    if (own)
        for (int k = 0; k < 25; ++k) dg[k] += J[k];
    else
        for (int k = 0; k < 25; ++k) dg[k] -= J[k];
    if (!inner) return false;
    // other side: dFR as owner, dFL as neighbour
    euler_jacobian_scaled(nm.gas, Uo, nx, ny, nz, half_area, J);
    for (int k = 0; k < 5; ++k) J[k * 6] = own ? (J[k * 6] - diss) : (J[k * 6] + diss);
    if (nm.viscous) add_viscous_jacobian(vm, !own, J);
    return true;
}

// Picard Jacobian on the flux tiles (jacobian_kernel.hpp:74-270): one
// workgroup per tile, one thread per block row.  The tile's cells' primitive
// states, centroids (and eddy viscosities) are staged in LDS with coalesced
// loads; each of a row's faces is read from the tile face-list stream (normal,
// area, centroid, packed cell ids: contiguous per tile), so only the halo or
// ghost side of a face on the tile boundary is gathered from the cell planes.
// Row c forms, per face, the face's dF of its own side (added to the diagonal:
// + dFL as owner, - dFR as neighbour) and, at an interior face, the other
// side's dF, the off-diagonal block: + dFR as owner, - dFL as neighbour.
// The threads take the tile's rows in the order of the sliced matrix layout,
// so in a round (each row's r-th face in ascending face index) a wave's 64
// blocks lie on consecutive lanes of a slot -- on a hexahedral mesh, where a
// row's blocks keep the face order -- and every store instruction writes whole
// cache lines.  (Row-major blocks staged through LDS and stored word by word
// covered cache lines only partly at first touch and made the L2 fetch them:
// 2.64 GB read for 0.9 GB of inputs, and the stage's 51 KB of LDS; on the
// 2.1M-cell plate FP64 1,429 -> 985 us.)  Two waves per SIMD at 178 registers: a third
// wave at 168 spills ten of them and gains nothing (262,144 cells FP64 138 / 147 us,
// 524,288 cells 271 / 268, 663,552 tetrahedra with eddy viscosity 301 / 317).  The
// arithmetic and its order are those of the reference's face loop, so the
// blocks are the reference's bit for bit; each block has a single writer.
template <class TS, bool kTurb>
__global__ void __launch_bounds__(kTileCells)
__attribute__((amdgpu_waves_per_eu(2)))
k_jacobian(MeshArgs m, FieldArgs f, NumArgs nm, SellArgs b, const double* alpha,
           typename SellLayout<TS>::word* off, typename SellLayout<TS>::word* diag) {
    stamp_stage(f.stamp, kStampJacobian);
    constexpr long long kW = SellLayout<TS>::words;
    __shared__ double sq[8 * kTileCells];  // q (0-4) and centroid (5-7) of the tile's cells, one plane each
    __shared__ double smut[kTurb ? kTileCells : 1];
    const int t = xcd_block(blockIdx.x, gridDim.x);
    const int c0 = m.tile_off[t], nt = m.tile_off[t + 1] - c0;
    const int fb = m.tile_face_off[t];
    const int th = threadIdx.x;
    if (th < nt) {
        typedef double pair_t __attribute__((ext_vector_type(2)));
        for (int p = 0; p < 4; ++p) {
            const pair_t v = *reinterpret_cast<const pair_t*>(f.cs + plane_at(2 * p, f.ld, c0 + th));
            sq[(2 * p) * kTileCells + th] = v.x;
            sq[(2 * p + 1) * kTileCells + th] = v.y;
        }
        if (kTurb) smut[th] = f.mut[c0 + th];
    }
    __syncthreads();
    if (th >= nt) return;
    const int p = b.tile_pos[c0 + th];
    const int c = b.row[p], i = c - c0;
    const int4 sl = b.slice[p / kSellRows];
    const int lane = p % kSellRows;
    const int nl = static_cast<int>(b.count[p] & 0xffffu);
    const int vb = b.visit_base[t], rounds = (b.visit_base[t + 1] - vb) / nt;
    double dg[25];
    for (int k = 0; k < 25; ++k) dg[k] = 0.0;
    for (int rr = 0; rr < rounds; ++rr) {
        const unsigned v = b.visit[vb + rr * nt + th];
        if (v == kSellVisitNone) break;  // no face follows
        const bool own = (v & kSellVisitNeighbour) == 0;
        double J[25];
        if (jacobian_face<kTurb>(m, f, nm, sq, smut, i, c0, nt, fb + static_cast<int>(v & 0x7fffu), own, dg, J)) {
            const int blk = static_cast<int>(v >> 16);
            const long long slot = blk < nl ? sl.x + blk : sl.x + sl.y + (blk - nl);
            store_sell_block<TS>(off + slot * kW * kSellRows + lane, J, own ? 1 : -1);
        }
    }
    const double a = alpha[c];
    for (int k = 0; k < 5; ++k) dg[k * 6] += a;
    store_sell_block<TS>(diag + (p / kSellRows) * kW * kSellRows + lane, dg, 0);
}

// Per-patch boundary integrals (residual_kernel.hpp:96-169 forms F[0] and
// F[4]; the momentum components give the force on the patch).  One workgroup
// per patch; thread t sums the patch's faces t, t + 256, ... in order, then a
// fixed tree adds the thread sums.
__global__ void __launch_bounds__(kBlock) k_boundary_integrals(int nbf, const int* bface_bc, const double* bflux,
                                                               double* out) {
    __shared__ double red[kBlock];
    const int p = blockIdx.x;
    double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    for (int b = threadIdx.x; b < nbf; b += kBlock) {
        if (bface_bc[b] != p) continue;
        for (int v = 0; v < 5; ++v) acc[v] += bflux[static_cast<long long>(b) * 5 + v];
    }
    for (int v = 0; v < 5; ++v) {
        red[threadIdx.x] = acc[v];
        __syncthreads();
        for (int w = kBlock / 2; w > 0; w >>= 1) {
            if (static_cast<int>(threadIdx.x) < w) red[threadIdx.x] += red[threadIdx.x + w];
            __syncthreads();
        }
        if (threadIdx.x == 0) out[p * 5 + v] = red[0];
        __syncthreads();
    }
}

inline dim3 grid_for(long long n) { return dim3(static_cast<unsigned>((n + kBlock - 1) / kBlock)); }

}  // namespace

void launch_primitives(const MeshArgs& m, const FieldArgs& f, const NumArgs& nm, const BcTable& bcs, hipStream_t s) {
    const int cells = (m.nc + kBlock - 1) / kBlock, ghosts = (m.nf - m.ninner + kBlock - 1) / kBlock;
    if (cells + ghosts > 0)
        hipLaunchKernelGGL(k_primitives, dim3(static_cast<unsigned>(cells + ghosts)), dim3(kBlock), 0, s, m, f, nm, bcs,
                           cells);
}

// Tiles up to which each has a CU of its own.
constexpr int kFewTiles = 256;

template <bool kSA>
static void launch_staged_gradient(const MeshArgs& m, const FieldArgs& f, const NumArgs& nm, const SaArgs& sa,
                                   hipStream_t s) {
    const unsigned cells = static_cast<unsigned>(m.gblock);
    const dim3 g(static_cast<unsigned>(m.ngtiles));
    // Two lanes per cell in the wide form, whose LDS leaves room for two workgroups per
    // CU, and where there is no second workgroup for a CU anyway.  The narrow form with
    // one / two lanes: 12 tiles 14.6 / 13.6 us, 106 tiles 19.4 / 18.1, 256 tiles 20.0 / 18.8,
    // 320 tiles 23.5 / 25.9, 1,024 tiles 40 / 48.
    if (m.gslots > kGradSlots)
        hipLaunchKernelGGL((k_gradient_limiter_lanes<kSA, kGradSlotsBig>), g, dim3(2 * cells), 0, s, m, f, nm, sa);
    else if (m.ngtiles <= kFewTiles)
        hipLaunchKernelGGL((k_gradient_limiter_lanes<kSA, kGradSlots>), g, dim3(2 * cells), 0, s, m, f, nm, sa);
    else
        hipLaunchKernelGGL((k_gradient_limiter_lds<kSA, kGradSlots>), g, dim3(cells), 0, s, m, f, nm, sa);
}

bool launch_gradient_limiter(const MeshArgs& m, const FieldArgs& f, const NumArgs& nm, hipStream_t s,
                             const SaArgs* sa) {
    if (m.nc <= 0) return false;
    if (m.tile_halo_off != nullptr) {
        if (sa)
            launch_staged_gradient<true>(m, f, nm, *sa, s);
        else
            launch_staged_gradient<false>(m, f, nm, SaArgs{}, s);
        return sa != nullptr;
    }
    hipLaunchKernelGGL(k_gradient_limiter, grid_for(m.nc), dim3(kBlock), 0, s, m, f, nm);
    return false;
}

void launch_lsq_setup(const MeshArgs& m, const FieldArgs& f, hipStream_t s) {
    if (m.nc > 0) hipLaunchKernelGGL(k_lsq_setup, grid_for(m.nc), dim3(kBlock), 0, s, m, f);
}

void launch_ghost_gradients(const MeshArgs& m, const FieldArgs& f, const NumArgs& nm, const BcTable& bcs,
                            hipStream_t s) {
    const int nbf = m.nf - m.ninner;
    if (nbf > 0)
        hipLaunchKernelGGL(k_ghost_gradients, grid_for(nbf), dim3(kBlock), 0, s, m, f, nm, bcs);
    else
        launch_stamp(f.stamp, kStampGhostGradients, -1, s);  // the stage has no kernel on a closed mesh
}

template <int kThreads>
static void launch_flux_as(const MeshArgs& m, const FieldArgs& f, const NumArgs& nm, hipStream_t s) {
    const dim3 g(static_cast<unsigned>(m.ntiles)), b(kThreads);
    if (f.mut)
        hipLaunchKernelGGL((k_flux<true, kThreads>), g, b, 0, s, m, f, nm);
    else
        hipLaunchKernelGGL((k_flux<false, kThreads>), g, b, 0, s, m, f, nm);
}

void launch_flux(const MeshArgs& m, const FieldArgs& f, const NumArgs& nm, hipStream_t s) {
    if (m.ntiles <= 0) return;
    // One face per lane where every tile has a CU of its own, else two, so that two
    // tiles share a CU.  Two / one per lane: 12 tiles 16.2 / 14.9 us, 106 tiles 19.1 / 17.1,
    // 188 tiles of tetrahedra with eddy viscosity 35 / 29, 384 tiles 26.6 / 30.7, 1,024
    // tiles 54 / 63.
    if (m.ntiles <= kFewTiles)
        launch_flux_as<2 * kFluxThreads>(m, f, nm, s);
    else
        launch_flux_as<kFluxThreads>(m, f, nm, s);
}

void launch_boundary_integrals(const MeshArgs& m, const FieldArgs& f, int n_patches, double* out, hipStream_t s) {
    if (n_patches > 0)
        hipLaunchKernelGGL(k_boundary_integrals, dim3(static_cast<unsigned>(n_patches)), dim3(kBlock), 0, s,
                           m.nf - m.ninner, m.bface_bc, f.bflux, out);
}

void launch_output_fields(int nc, const Gas& g, const double* U, double* out, hipStream_t s) {
    if (nc > 0) hipLaunchKernelGGL(k_output_fields, grid_for(nc), dim3(kBlock), 0, s, nc, g, U, out);
}

void launch_gather_mdot(int nf, const int* face_entry, const double* mdot_tile, double* mdot, hipStream_t s) {
    if (nf > 0) hipLaunchKernelGGL(k_gather_mdot, grid_for(nf), dim3(kBlock), 0, s, nf, face_entry, mdot_tile, mdot);
}

void launch_dt(const MeshArgs& m, const FieldArgs& f, const double* lam, double cfl, double unsteady, double* dt,
               double* alpha, bool flux_end, hipStream_t s) {
    if (m.nc > 0)
        hipLaunchKernelGGL(k_dt, grid_for(m.nc), dim3(kBlock), 0, s, m.nc, f.cs, f.ld, lam, cfl, unsteady, dt, alpha,
                           flux_end ? f.stamp : nullptr);
}

void launch_planes_to_device(int nc, const int* mesh_of_row, const double* src, double* dst, hipStream_t s) {
    if (nc > 0) hipLaunchKernelGGL(k_permute_planes<true>, grid_for(nc), dim3(kBlock), 0, s, nc, mesh_of_row, src, dst);
}

void launch_planes_to_mesh(int nc, const int* mesh_of_row, const double* src, double* dst, hipStream_t s) {
    if (nc > 0) hipLaunchKernelGGL(k_permute_planes<false>, grid_for(nc), dim3(kBlock), 0, s, nc, mesh_of_row, src, dst);
}

int launch_explicit_step(const MeshArgs& m, const FieldArgs& f, const double* lam, double cfl, double* dt,
                         double* alpha, double* U, double* partial, hipStream_t s) {
    const int nb = reduction_blocks(m.nc);
    hipLaunchKernelGGL(k_explicit_step, dim3(nb), dim3(kBlock), 0, s, m.nc, f.cs, f.ld, lam, cfl, f.res, dt, alpha, U,
                       partial, f.stamp);
    return nb;
}

void launch_stamp(unsigned long long* stamp, int k, int k2, hipStream_t s) {
    hipLaunchKernelGGL(k_stamp, dim3(1), dim3(1), 0, s, stamp, k, k2);
}

void launch_unsteady_source(const MeshArgs& m, const FieldArgs& f, int bdf, double inv_dt, const double* Un,
                            const double* Unm1, hipStream_t s) {
    if (m.nc > 0)
        hipLaunchKernelGGL(k_unsteady_source, grid_for(m.nc), dim3(kBlock), 0, s, m.nc, f.cs, f.ld, bdf, inv_dt, f.U,
                           Un, Unm1, f.res);
}

template <class TS>
static void launch_jacobian_as(const MeshArgs& m, const FieldArgs& f, const NumArgs& nm, const SellArgs& b,
                               const double* alpha, void* off, void* diag, hipStream_t s) {
    typedef typename SellLayout<TS>::word word;
    const dim3 grid(static_cast<unsigned>(m.ntiles)), block(kTileCells);
    if (f.mut)
        hipLaunchKernelGGL((k_jacobian<TS, true>), grid, block, 0, s, m, f, nm, b, alpha, static_cast<word*>(off),
                           static_cast<word*>(diag));
    else
        hipLaunchKernelGGL((k_jacobian<TS, false>), grid, block, 0, s, m, f, nm, b, alpha, static_cast<word*>(off),
                           static_cast<word*>(diag));
}

void launch_jacobian(const MeshArgs& m, const FieldArgs& f, const NumArgs& nm, const SellArgs& b,
                     const double* alpha, void* off, void* diag, int storage, hipStream_t s) {
    if (m.nc <= 0) return;
    if (storage == kStoreF32)
        launch_jacobian_as<float>(m, f, nm, b, alpha, off, diag, s);
    else if (storage == kStoreBF16)
        launch_jacobian_as<bf16>(m, f, nm, b, alpha, off, diag, s);
    else
        launch_jacobian_as<double>(m, f, nm, b, alpha, off, diag, s);
}

}  // namespace cfdg
