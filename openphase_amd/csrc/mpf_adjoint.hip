// Adjoint (vector-Jacobian product) of one multiphase-field step on MI355X.
//
// Forward step t -> t+1 per interface cell c: the merged list of c (own entries, entries appended
// from neighbours) with Laplacians L_e(c) = sum_k w_k phi_e(c+k) and gradients
// G_e(c) = sum_k g_k phi_e(c+k) (src/PhaseField.cpp:566-615) feeds the cell update: pair energies
// (InterfaceProperties::SetSR, src/InterfaceProperties.cpp:603-762), double-obstacle pair
// increments psi (src/DoubleObstacle.cpp:502-571) with the constant driving force
// (src/DrivingForce.cpp:497-602), the sum-to-one limiter (PhaseField::NormalizeIncrementsSR,
// src/PhaseField.cpp:1351-1567), the merge (:1268-1299) and NodePF::finalize
// (include/Containers/NodePF.h:214-255). Bulk cells keep their single entry.
//
// Given the cotangent of the values of S_{t+1}, three stages return the cotangent of the values
// of S_t and add the cotangents of the pair tables:
//  1. adjoint_local_kernel, one thread per cell: the cell update of a two-entry list (in
//     registers) is recomputed in FP64 and swept backwards by hand - finalize and merge, then the
//     increments psi (pair energies with the cubic anisotropy, triple-junction and driving-force
//     terms). Longer lists go to a work list that adjoint_list_kernel takes (the list length C a
//     compile-time constant), sweeping the sum-to-one limiter backwards through its iterations,
//     recomputed from the increments entering it; lists of five or more entries (a few cells per
//     step) go on to a second list and adjoint_long_kernel (five entries in registers, six to
//     eight in private memory), so that their long code holds up only its own wavefronts.
//     Out: the direct part per own entry, the cotangents of each merged entry's Laplacian and
//     gradient, and the table cotangents - per block of cells, in thread order, and per listed
//     cell, folded into its block's sum in cell order by adjoint_fold_kernel.
//  2. adjoint_gather_kernel: the transpose of the stencils as a gather (Laplacian weights
//     symmetric, gradient weights antisymmetric in the offset):
//     lam_t(c, g) = direct(c, g) + sum_k w_k lamL(c+k, g) - sum_k g_k . lamG(c+k, g).
//  3. adjoint_grad_kernel: the per-block table cotangents summed over the blocks in a fixed order
//     and added to the caller's array. Results are the same from run to run.
// Derivatives follow the branches the forward step takes (clamps, erasures and limiter factors as
// evaluated); grain VolumeRatios are held fixed. FP32 states are differentiated at their values
// with FP64 arithmetic; S_{t+1}'s grain lists map the next-state cotangents to the entries.

#include <hip/hip_runtime.h>

#include "mpf_adjoint_cell.h"
#include "mpf_device.h"
#include "mpf_group.h"
#include "mpf_lists.h"

namespace mpf {

namespace {

constexpr int kAdjBlock = 64;      // one wavefront per block
enum AdjError { kAdjCapacity = 3 };  // status word: a cell needed more than kAdjSlots entries

constexpr int kAdjMid = 4;         // list capacity of the work-list kernel's register path
constexpr int kAdjListBlocks = 1024;  // blocks (wavefronts) of the work-list kernels

// Writes the adjoint outputs of a wide cell: merged entries with the cotangents of their
// Laplacians and gradients, and the direct part of the own entries.
template <int K, bool GRAD>
__device__ __forceinline__ void store_adjoint(const AdjointArgs& J, int64_t c, const CellList<K, double, GRAD>& L,
                                              const double (&lam_phi)[K], const double (&lam_lap)[K],
                                              const double (&lam_gr)[GRAD ? K : 1][3])
{
    const int64_t N = J.s.ncells;
    const int ne = L.ne;
    J.adj_cnt[c] = static_cast<uint8_t>(ne);
#pragma unroll
    for (int e = 0; e < K; ++e) {
        if (e >= ne) continue;
        J.adj_id[static_cast<int64_t>(e) * N + c] = static_cast<uint16_t>(L.eid[e]);
        J.adj_lap[static_cast<int64_t>(e) * N + c] = lam_lap[e];
        if (GRAD)
            for (int d = 0; d < 3; ++d) J.adj_grad[static_cast<int64_t>(3 * e + d) * N + c] = lam_gr[GRAD ? e : 0][d];
        if (e < L.n0) J.lam_own[static_cast<int64_t>(e) * N + c] = lam_phi[e];
    }
}

// Main local kernel: bulk cells and wide cells of two merged entries (lists in registers). Longer
// lists go to the work list (J.defer marks them by cell for the fold in cell order).
template <typename TV, bool GRAD>
__global__ __launch_bounds__(kAdjBlock) void adjoint_local_kernel(const AdjointArgs J)
{
    extern __shared__ double gsh[];  // [kAdjBlock][3 nphases^2] table cotangents per thread
    constexpr int K = 2;
    const StepArgs& A = J.s;
    const bool fp32 = sizeof(TV) == 4;
    const int G = 3 * A.nphases * A.nphases;
    double* gsl = gsh + static_cast<int>(threadIdx.x) * G;
    for (int e = 0; e < G; ++e) gsl[e] = 0.0;
    const int64_t c = static_cast<int64_t>(blockIdx.x) * kAdjBlock + threadIdx.x;
    if (c < A.ncells) {
        CellList<K, double, GRAD> L;
        const int r = gather_cell<K, TV, double, GRAD>(A, c, L);
        bool defer = r == kCellDeferred;
        if (r == kCellBulk) {
            // a bulk cell keeps its single entry
            J.adj_cnt[c] = 0;
            if (L.n0 == 1) {
                const NextList next(J, fp32, c);
                J.lam_own[c] = next.lam(J, c, next.find(J, c, L.eid[0], 0));
            }
        } else if (r == kCellWide) {
            double lam_phi[K], lam_lap[K], lam_gr[GRAD ? K : 1][3];
            cell_adjoint<2, GRAD, K>(J, fp32, c, L, lam_phi, lam_lap, lam_gr, gsl);
            store_adjoint<K, GRAD>(J, c, L, lam_phi, lam_lap, lam_gr);
        }
        J.defer[c] = defer ? 1 : 0;
        if (defer) J.list[atomicAdd(J.list_count, 1u)] = static_cast<uint32_t>(c);
    }
    __syncthreads();
    if (static_cast<int>(threadIdx.x) < G) {
        double s = 0.0;
        for (int t = 0; t < kAdjBlock; ++t) s += gsh[t * G + threadIdx.x];
        J.partial[static_cast<int64_t>(blockIdx.x) * G + threadIdx.x] = s;
    }
}

// One listed cell of at most kAdjMid merged entries (lists in registers): cotangents stored, its
// table cotangents to J.cellg[cell]. A longer list goes to the second work list.
template <typename TV, bool GRAD>
__device__ __forceinline__ void list_cell(const AdjointArgs& J, int64_t c, double* gsl)
{
    const StepArgs& A = J.s;
    const bool fp32 = sizeof(TV) == 4;
    const int G = 3 * A.nphases * A.nphases;
    constexpr int K = kAdjMid;
    CellList<K, double, GRAD> L;
    const int r = gather_cell<K, TV, double, GRAD>(A, c, L);
    if (r != kCellWide) {
        J.list_long[atomicAdd(J.long_count, 1u)] = static_cast<uint32_t>(c);
        return;
    }
    for (int e = 0; e < G; ++e) gsl[e] = 0.0;
    double lam_phi[K], lam_lap[K], lam_gr[GRAD ? K : 1][3];
    switch (L.ne) {
        case 2: cell_adjoint<2, GRAD, K>(J, fp32, c, L, lam_phi, lam_lap, lam_gr, gsl); break;
        case 3: cell_adjoint<3, GRAD, K>(J, fp32, c, L, lam_phi, lam_lap, lam_gr, gsl); break;
        default: cell_adjoint<4, GRAD, K>(J, fp32, c, L, lam_phi, lam_lap, lam_gr, gsl); break;
    }
    store_adjoint<K, GRAD>(J, c, L, lam_phi, lam_lap, lam_gr);
    for (int e = 0; e < G; ++e) J.cellg[c * G + e] = gsl[e];
}

// The list a group of lanes formed, as one lane's register list.
template <int K, bool GRAD>
__device__ __forceinline__ void take_list(const GroupMem<double, GRAD, kAdjSlots>& M, int n0, int ne, CellList<K, double, GRAD>& L)
{
    L.n0 = n0;
    L.ne = ne;
#pragma unroll
    for (int t = 0; t < K; ++t) {
        const bool in = t < ne;
        L.eid[t] = in ? M.eid[t] : 0u;
        L.phi[t] = in ? M.phi[t] : 0.0;
        L.lap[t] = in ? M.lap[t] : 0.0;
        L.keep[t] = t < n0;
        if (GRAD)
            for (int d = 0; d < 3; ++d) L.gr[GRAD ? t : 0][d] = in ? M.gr[GRAD ? t : 0][d] : 0.0;
    }
}

// Cells of the second work list, four by the groups of a wavefront (`run`): the list is formed by the
// group (a lane alone waits through it twice, with five and with eight entries), the reverse sweep
// runs in the group's first lane - five merged entries in registers (almost all of them), up to
// kAdjSlots in private memory; more is reported in the status word.
template <typename TV, bool GRAD>
__device__ __forceinline__ void long_cell(const AdjointArgs& J, bool run, int64_t c, GroupMem<double, GRAD, kAdjSlots>& M, double* gsl)
{
    static_assert(kAdjSlots == kGroupCap, "the group holds the adjoint's lists");
    const StepArgs& A = J.s;
    const bool fp32 = sizeof(TV) == 4;
    const int G = 3 * A.nphases * A.nphases, l = static_cast<int>(threadIdx.x) & (kGroupLanes - 1);
    const GroupList<double> P = group_gather<TV, double, GRAD, kGroupLanes, kAdjSlots>(A, run, c, M);
    if (l < kAdjSlots) {
        M.lap[l] = P.lap;
        M.phi[l] = P.phi;
        if (GRAD) { M.gr[GRAD ? l : 0][0] = P.gx; M.gr[GRAD ? l : 0][1] = P.gy; M.gr[GRAD ? l : 0][2] = P.gz; }
    }
    __syncthreads();
    if (run && l == 0) {
        for (int e = 0; e < G; ++e) gsl[e] = 0.0;
        if (P.over) {
            atomicOr(&A.status[kAdjCapacity], 1);
            J.adj_cnt[c] = 0;
        } else if (P.ne == 5) {
            constexpr int K = 5;
            CellList<K, double, GRAD> L;
            take_list<K, GRAD>(M, P.n0, P.ne, L);
            double lam_phi[K], lam_lap[K], lam_gr[GRAD ? K : 1][3];
            cell_adjoint<5, GRAD, K>(J, fp32, c, L, lam_phi, lam_lap, lam_gr, gsl);
            store_adjoint<K, GRAD>(J, c, L, lam_phi, lam_lap, lam_gr);
        } else {
            constexpr int K = kAdjSlots;
            CellList<K, double, GRAD> L;
            take_list<K, GRAD>(M, P.n0, P.ne, L);
            double lam_phi[K], lam_lap[K], lam_gr[GRAD ? K : 1][3];
            switch (P.ne) {
                case 6: cell_adjoint<6, GRAD, K>(J, fp32, c, L, lam_phi, lam_lap, lam_gr, gsl); break;
                case 7: cell_adjoint<7, GRAD, K>(J, fp32, c, L, lam_phi, lam_lap, lam_gr, gsl); break;
                default: cell_adjoint<8, GRAD, K>(J, fp32, c, L, lam_phi, lam_lap, lam_gr, gsl); break;
            }
            store_adjoint<K, GRAD>(J, c, L, lam_phi, lam_lap, lam_gr);
        }
        for (int e = 0; e < G; ++e) J.cellg[c * G + e] = gsl[e];
    }
    __syncthreads();
}

// Work-list kernel: the cells of three or four merged entries, spread over all wavefronts (a cell's
// latency, not the chip, bounds it: the fewer lengths a wavefront holds, the better).
template <typename TV, bool GRAD>
__global__ __launch_bounds__(kAdjBlock) void adjoint_list_kernel(const AdjointArgs J)
{
    extern __shared__ double gsh[];
    const int G = 3 * J.s.nphases * J.s.nphases;
    double* gsl = gsh + static_cast<int>(threadIdx.x) * G;
    const unsigned n = *J.list_count, per = (n + gridDim.x - 1) / gridDim.x, end = min(n, (blockIdx.x + 1) * per);
    for (unsigned i = blockIdx.x * per + threadIdx.x; i < end; i += kAdjBlock) list_cell<TV, GRAD>(J, J.list[i], gsl);
}

// Second work-list kernel: the few cells of five or more merged entries, at most one to a group of
// lanes while there are that few. 64 of them to a wavefront, each lane forming its own list, took
// 220 us at 2D 512^2 (1,150 cells falling to 90 in eight steps); now 145 us, the reverse sweep of one
// cell.
template <typename TV, bool GRAD>
__global__ __launch_bounds__(kAdjBlock) void adjoint_long_kernel(const AdjointArgs J)
{
    constexpr int C = kAdjBlock / kGroupLanes;
    extern __shared__ double gsh[];
    __shared__ GroupMem<double, GRAD, kAdjSlots> mem[C];
    const int G = 3 * J.s.nphases * J.s.nphases, group = static_cast<int>(threadIdx.x) / kGroupLanes;
    double* gsl = gsh + group * G;
    const unsigned n = *J.long_count;
    const unsigned used = min(static_cast<unsigned>(C), (n + gridDim.x - 1) / gridDim.x);
    for (unsigned base = blockIdx.x * used; base < n; base += gridDim.x * used) {
        const unsigned i = base + static_cast<unsigned>(group);
        const bool run = static_cast<unsigned>(group) < used && i < n;
        long_cell<TV, GRAD>(J, run, run ? J.list_long[i] : 0, mem[group], gsl);
    }
}

// One wavefront per main-kernel block: adds the table cotangents of the block's listed cells to
// the block's partial sums, summed over the 64 cells by a fixed shuffle tree.
__global__ __launch_bounds__(64) void adjoint_fold_kernel(const AdjointArgs J)
{
    const int64_t b = blockIdx.x;
    const int G = 3 * J.s.nphases * J.s.nphases;
    const int64_t c = b * kAdjBlock + threadIdx.x;
    const bool listed = c < J.s.ncells && J.defer[c];
    if (!__any(listed)) return;
    for (int e = 0; e < G; ++e) {
        double v = listed ? J.cellg[c * G + e] : 0.0;
        for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
        if (threadIdx.x == 0) J.partial[b * G + e] += v;
    }
}

// Cotangent of own entry s (grain g) of cell c by a search of every neighbour's entries, one after
// the other.
template <bool GRAD>
__device__ __forceinline__ double gather_entry(const AdjointArgs& J, int64_t c, int s, uint32_t g)
{
    const StepArgs& A = J.s;
    const int64_t N = A.ncells;
    const Box B = make_box(A, c);
    double acc = J.lam_own[static_cast<int64_t>(s) * N + c];
    for (int k = 0; k < 27; ++k) {
        if (!box_active(A, k)) continue;
        const int ii = k / 9 - 1, jj = (k / 3) % 3 - 1, kk = k % 3 - 1;
        const int nnz = (ii != 0) + (jj != 0) + (kk != 0);
        const int64_t nb = B.cell(k);
        const int m = min(static_cast<int>(J.adj_cnt[nb]), kAdjSlots);
        for (int e = 0; e < m; ++e) {
            if (J.adj_id[static_cast<int64_t>(e) * N + nb] != g) continue;
            acc += A.wl[nnz] * J.adj_lap[static_cast<int64_t>(e) * N + nb];
            if (GRAD && nnz) {
                const double gw = A.wg[nnz];
                const double gx = ii == 0 ? 0.0 : (ii < 0 ? -gw : gw);
                const double gy = jj == 0 ? 0.0 : (jj < 0 ? -gw : gw);
                const double gz = kk == 0 ? 0.0 : (kk < 0 ? -gw : gw);
                acc -= gx * J.adj_grad[static_cast<int64_t>(3 * e + 0) * N + nb] +
                       gy * J.adj_grad[static_cast<int64_t>(3 * e + 1) * N + nb] +
                       gz * J.adj_grad[static_cast<int64_t>(3 * e + 2) * N + nb];
            }
        }
    }
    return acc;
}

// One thread per cell. Latency bound, so the neighbours of a plane of the box (2D: of the whole box,
// whose two active axes form that plane) are looked up together: their nine counts, the first two
// grains of each, then the cotangents of those the cell holds, three neighbours at a time; the
// first four own entries are summed in one walk. Every entry's sum keeps the order of neighbours and
// of their entries. An own entry and a neighbour entry at a time it took 108 us at 2D 512^2; now
// 57 us.
template <typename TV, bool GRAD>
__global__ __launch_bounds__(kAdjBlock) void adjoint_gather_kernel(const AdjointArgs J)
{
    constexpr int S = 4;  // own entries of one walk
    const StepArgs& A = J.s;
    const int64_t N = A.ncells;
    const int64_t c = static_cast<int64_t>(blockIdx.x) * kAdjBlock + threadIdx.x;
    if (c >= N) return;
    const int n0 = min(ListCode<TV>::count(A.cnt_in[c]), kAdjSlots);
    uint32_t g[S];
    double acc[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        g[s] = s < n0 ? A.id_in[static_cast<int64_t>(s) * N + c] : ~0u;
        acc[s] = s < n0 ? J.lam_own[static_cast<int64_t>(s) * N + c] : 0.0;
    }
    // axes of the planes: (y, z) of a 3D grid, else the active ones in their order
    const bool cube = A.dnx && A.dny && A.dnz;
    const int NY = A.ny, NZ = A.nz;
    const int x = static_cast<int>(c / (static_cast<int64_t>(NY) * NZ)), y = static_cast<int>((c / NZ) % NY),
              z = static_cast<int>(c % NZ);
    const int ax1 = cube || !A.dnx ? 1 : 0, ax2 = !cube && A.dnx && A.dny ? 1 : 2;
    auto place = [&](int ax, int d) -> int64_t {  // offset of coordinate + d along an axis
        return ax == 0 ? static_cast<int64_t>(wrap1(x + d, A.nx)) * NY * NZ
                       : (ax == 1 ? static_cast<int64_t>(wrap1(y + d, NY)) * NZ : static_cast<int64_t>(wrap1(z + d, NZ)));
    };
    const bool on1 = ax1 == 0 ? A.dnx : A.dny, on2 = ax2 == 1 ? A.dny : A.dnz;
    // the coordinates that neither plane axis moves
    const int64_t rest = cube ? 0 : (ax1 != 0 ? place(0, 0) : 0) + (ax1 != 1 && ax2 != 1 ? place(1, 0) : 0) + (ax2 != 2 ? place(2, 0) : 0);
    int64_t p1[3], p2[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        p1[d] = place(ax1, on1 ? d - 1 : 0);
        p2[d] = place(ax2, on2 ? d - 1 : 0);
    }
#pragma unroll 1
    for (int ii = cube ? -1 : 0; ii <= (cube ? 1 : 0); ++ii) {
        const int64_t base = cube ? place(0, ii) : rest;
        int m[9];
        uint32_t id[9][2];
        bool any = false;
#pragma unroll
        for (int j = 0; j < 9; ++j) {
            const bool in = (j / 3 == 1 || on1) && (j % 3 == 1 || on2);
            const uint8_t cnt = J.adj_cnt[base + p1[j / 3] + p2[j % 3]];
            m[j] = in ? min(static_cast<int>(cnt), kAdjSlots) : 0;
            any = any || m[j] > 0;
        }
        if (!any || n0 == 0) continue;
#pragma unroll
        for (int j = 0; j < 9; ++j)
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int64_t nb = base + p1[j / 3] + p2[j % 3];
                const uint32_t v = J.adj_id[(e < m[j] ? static_cast<int64_t>(e) * N : 0) + nb];
                id[j][e] = e < m[j] ? v : ~1u;
            }
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            int hit[3][2];
            double lap[3][2], gr[GRAD ? 3 : 1][2][3];
#pragma unroll
            for (int q = 0; q < 3; ++q)
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const int j = 3 * r + q;
                    const int64_t nb = base + p1[r] + p2[q];
                    int h = -1;
#pragma unroll
                    for (int s = S - 1; s >= 0; --s) h = g[s] == id[j][e] ? s : h;
                    hit[q][e] = h;
                    lap[q][e] = 0.0;
                    if (h >= 0) {
                        lap[q][e] = J.adj_lap[static_cast<int64_t>(e) * N + nb];
                        if (GRAD)
                            for (int d = 0; d < 3; ++d) gr[GRAD ? q : 0][e][d] = J.adj_grad[static_cast<int64_t>(3 * e + d) * N + nb];
                    }
                }
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                const int j = 3 * r + q;
                const int jj = j / 3 - 1, kk = j % 3 - 1;
                const int nnz = (ii != 0) + (jj != 0) + (kk != 0);
                const double wl = A.wl[nnz], gw = A.wg[nnz];
                const double g0 = ii == 0 ? 0.0 : (ii < 0 ? -gw : gw), g1 = jj == 0 ? 0.0 : (jj < 0 ? -gw : gw),
                             g2 = kk == 0 ? 0.0 : (kk < 0 ? -gw : gw);
                // gradient weights along x, y, z
                const double gx = cube ? g0 : (ax1 == 0 ? g1 : 0.0);
                const double gy = cube || ax1 == 1 ? g1 : (ax2 == 1 ? g2 : 0.0);
                const double gz = ax2 == 2 ? g2 : 0.0;
#pragma unroll
                for (int e = 0; e < 2; ++e)
#pragma unroll
                    for (int s = 0; s < S; ++s)
                        if (hit[q][e] == s) {
                            acc[s] += wl * lap[q][e];
                            if (GRAD && nnz) acc[s] -= gx * gr[GRAD ? q : 0][e][0] + gy * gr[GRAD ? q : 0][e][1] + gz * gr[GRAD ? q : 0][e][2];
                        }
                for (int e = 2; e < m[j]; ++e) {
                    const int64_t nb = base + p1[r] + p2[q];
                    const uint32_t v = J.adj_id[static_cast<int64_t>(e) * N + nb];
#pragma unroll
                    for (int s = 0; s < S; ++s)
                        if (g[s] == v) {
                            acc[s] += wl * J.adj_lap[static_cast<int64_t>(e) * N + nb];
                            if (GRAD && nnz)
                                acc[s] -= gx * J.adj_grad[static_cast<int64_t>(3 * e + 0) * N + nb] +
                                          gy * J.adj_grad[static_cast<int64_t>(3 * e + 1) * N + nb] +
                                          gz * J.adj_grad[static_cast<int64_t>(3 * e + 2) * N + nb];
                        }
                }
            }
        }
    }
#pragma unroll
    for (int s = 0; s < S; ++s)
        if (s < A.slots) J.lam_prev[static_cast<int64_t>(s) * N + c] = s < n0 ? acc[s] : 0.0;
    for (int s = S; s < A.slots; ++s)
        J.lam_prev[static_cast<int64_t>(s) * N + c] =
            s < n0 ? gather_entry<GRAD>(J, c, s, A.id_in[static_cast<int64_t>(s) * N + c]) : 0.0;
}

__global__ void adjoint_reset_kernel(unsigned* count)
{
    if (threadIdx.x < 2) count[threadIdx.x] = 0u;
}

// One block per table entry e: grad[e] += sum over blocks of partial[block][e], in block order per
// thread, then a fixed tree.
__global__ __launch_bounds__(256) void adjoint_grad_kernel(const double* __restrict__ partial, int64_t nb, int G,
                                                           double* __restrict__ grad)
{
    __shared__ double lds[256];
    const int e = blockIdx.x;
    double v = 0.0;
    for (int64_t b = threadIdx.x; b < nb; b += 256) v += partial[b * G + e];
    lds[threadIdx.x] = v;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (static_cast<int>(threadIdx.x) < s) lds[threadIdx.x] = lds[threadIdx.x] + lds[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) grad[e] += lds[0];
}

template <typename TV, bool GRAD>
void launch_all(const AdjointArgs& a, hipStream_t s)
{
    const int64_t nb = adjoint_blocks(a.s.ncells);
    const int G = 3 * a.s.nphases * a.s.nphases;
    const dim3 grid(static_cast<unsigned>(nb));
    hipLaunchKernelGGL(adjoint_reset_kernel, dim3(1), dim3(64), 0, s, a.list_count);
    hipLaunchKernelGGL((adjoint_local_kernel<TV, GRAD>), grid, dim3(kAdjBlock), kAdjBlock * G * sizeof(double), s, a);
    hipLaunchKernelGGL((adjoint_list_kernel<TV, GRAD>), dim3(kAdjListBlocks), dim3(kAdjBlock),
                       kAdjBlock * G * sizeof(double), s, a);
    hipLaunchKernelGGL((adjoint_long_kernel<TV, GRAD>), dim3(kAdjListBlocks), dim3(kAdjBlock),
                       kAdjBlock / kGroupLanes * G * sizeof(double), s, a);
    hipLaunchKernelGGL(adjoint_fold_kernel, grid, dim3(kAdjBlock), 0, s, a);
    hipLaunchKernelGGL((adjoint_gather_kernel<TV, GRAD>), grid, dim3(kAdjBlock), 0, s, a);
    hipLaunchKernelGGL(adjoint_grad_kernel, dim3(G), dim3(256), 0, s, a.partial, nb, G, a.grad);
}

}  // namespace

int64_t adjoint_blocks(int64_t ncells) { return (ncells + kAdjBlock - 1) / kAdjBlock; }

int launch_adjoint(const AdjointArgs& a, bool fp32, void* stream)
{
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (fp32) {
        if (a.grad_energy) launch_all<float, true>(a, s);
        else launch_all<float, false>(a, s);
    } else {
        if (a.grad_energy) launch_all<double, true>(a, s);
        else launch_all<double, false>(a, s);
    }
    return static_cast<int>(hipGetLastError());
}

}  // namespace mpf
