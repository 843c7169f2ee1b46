// Quantities derived from the state on demand: per-cell phase fractions
// (PhaseField::CalculateFractions, src/PhaseField.cpp:411-423), and the interface energy of the
// double-obstacle functional summed over the grid:
// DoubleObstacle::PointEnergy (src/DoubleObstacle.cpp:903-923) per cell, added up by
// DoubleObstacle::Energy / AverageEnergyDensity (:953-967, :989-1005).
//
// Per wide-interface cell of the current state, over the pairs alpha < beta of its
// neighbour-merged list (zero-valued appended entries included), 4 E (phi_a phi_b - Eta^2/Pi^2
// grad_a . grad_b) / Eta. The gradients are those of the current lists
// (PhaseField::CalculateDerivativesSR, src/PhaseField.cpp:588-603); E is the energy
// InterfaceProperties::Properties holds for the pair, i.e. what the last IP.Set evaluated on the
// state it saw (`ip_*`, the step-start state when IP.Set ran before the last step): 0 for a pair
// absent from that cell's list then, or for a cell that was not a wide interface
// (NodeIP::get_energy, include/Containers/NodeIP.h:379-388).
//
// Each block sums its cells in a fixed order, and one block adds the partial sums in a fixed order, so the result is the same from run to run (it differs from the
// reference's sequential sum only in rounding).
#include <hip/hip_runtime.h>

#include "mpf_device.h"
#include "mpf_group.h"
#include "mpf_lists.h"
#include "mpf_step_ops.h"

namespace mpf {

namespace {

constexpr int kEnergyBlock = 256;  // cells of a block of energy_kernel; threads of the other kernels

__device__ __forceinline__ double block_sum(double v, double* lds)
{
    lds[threadIdx.x] = v;
    __syncthreads();
    for (int s = kEnergyBlock / 2; s > 0; s >>= 1) {
        if (static_cast<int>(threadIdx.x) < s) lds[threadIdx.x] = lds[threadIdx.x] + lds[threadIdx.x + s];
        __syncthreads();
    }
    return lds[0];
}

// Which of the grains eid[0 .. ne) the merged list of cell c of state B holds (bit t), and whether
// that cell is a wide interface at all (bit 31). Group-wide.
template <typename TV, int G>
__device__ __forceinline__ uint32_t group_members(const StepArgs& B, bool run, int64_t c, const uint32_t* eid, int ne)
{
    constexpr int NK = (27 + G - 1) / G;
    const int l = static_cast<int>(threadIdx.x) & (G - 1);
    const int64_t N = B.ncells;
    const uint32_t cc = static_cast<uint32_t>(run ? c : 0);
    const int NY = B.ny, NZ = B.nz;
    const int z0 = static_cast<int>(cc % static_cast<uint32_t>(NZ));
    const int y0 = static_cast<int>((cc / static_cast<uint32_t>(NZ)) % static_cast<uint32_t>(NY));
    const int x0 = static_cast<int>(cc / (static_cast<uint32_t>(NY) * static_cast<uint32_t>(NZ)));
    uint32_t nb[NK], mask = 0u;
    int m[NK], imp[NK];
#pragma unroll
    for (int j = 0; j < NK; ++j) {
        const int k = l + j * G;
        const int ii = k / 9 - 1, jj = (k / 3) % 3 - 1, kk = k % 3 - 1;
        const bool act = run && k < 27 && (ii == 0 || B.dnx) && (jj == 0 || B.dny) && (kk == 0 || B.dnz);
        nb[j] = static_cast<uint32_t>((wrap1(x0 + (act ? ii : 0), B.nx) * NY + wrap1(y0 + (act ? jj : 0), NY)) * NZ +
                                      wrap1(z0 + (act ? kk : 0), NZ));
        const uint8_t code = B.cnt_in[nb[j]];
        m[j] = act ? ListCode<TV>::count(code) : 0;
        imp[j] = ListCode<TV>::implicit(code);
        if (m[j] > 1) mask |= 1u << 31;
    }
#pragma unroll
    for (int j = 0; j < NK; ++j) {
        const bool own = l + j * G == 13;
        for (int q = 0; q < m[j]; ++q) {
            const int64_t at = static_cast<int64_t>(q) * N + nb[j];
            const uint32_t g = B.id_in[at];
            // a zero value is not merged (a lone implicit entry of FP32 has none stored: it is 1)
            const bool lone = ListCode<TV>::kImplicit && m[j] == 1 && imp[j] == 0;
            if (!own && !lone && load_val<TV>(B.val_in, at) == TV(0)) continue;
            for (int t = 0; t < ne; ++t)
                if (eid[t] == g) mask |= 1u << t;
        }
    }
#pragma unroll
    for (int k = 1; k < G; k <<= 1) mask |= static_cast<uint32_t>(__shfl_xor(static_cast<int>(mask), k));
    return mask;
}

// This lane's part of the energy of cell c (when `run`). `over`: the lists need more than CAP entries.
// FULL: the pair's energy needs the list IP.Set saw with its values and gradients (orientation
// dependent) or its order (tables that are not symmetric); otherwise only whether it held the pair.
template <typename TV, bool FULL, int G, int CAP>
__device__ __forceinline__ double group_energy(const EnergyArgs& E, const StepArgs& B, bool run, int64_t c,
                                               GroupMem<double, true, CAP>& M, GroupMem<double, true, CAP>* O,
                                               const uint16_t* pairs, bool& over)
{
    const StepArgs& A = E.cur;
    const int l = static_cast<int>(threadIdx.x) & (G - 1), NP = A.nphases;
    const GroupList<double> L = group_gather<TV, double, true, G, CAP>(A, run, c, M);
    over = run && L.over;
    const bool work = run && !L.over && L.wide;
    if (l < CAP) {
        M.gr[l][0] = L.gx; M.gr[l][1] = L.gy; M.gr[l][2] = L.gz;
        M.phi[l] = L.phi;
        M.ph[l] = work && l < L.ne ? A.gphase[L.eid] : 0;
    }
    uint32_t held = 0u;
    int ip_ne = 0;
    bool ip_wide = false;
    if (FULL) {
        const GroupList<double> P = group_gather<TV, double, true, G, CAP>(B, run, c, *O);
        over = over || (run && P.over);
        ip_ne = P.ne;
        ip_wide = P.wide;
        if (l < CAP) {
            O->gr[l][0] = P.gx; O->gr[l][1] = P.gy; O->gr[l][2] = P.gz;
            O->phi[l] = P.phi;
        }
    } else {
        __syncthreads();
        held = group_members<TV, G>(B, work, c, M.eid, work ? L.ne : 0);
        ip_wide = (held >> 31) != 0u;
    }
    __syncthreads();
    double e = 0.0;
    const int np = work && !over && ip_wide ? L.ne * (L.ne - 1) / 2 : 0;
    for (int p = l; p < np; p += G) {
        const int a = pairs[p] & 255, b = pairs[p] >> 8;
        double en = 0.0;  // a pair absent from the list IP.Set saw has no energy
        if (FULL) {
            int pa = -1, pb = -1;
            for (int t = 0; t < ip_ne; ++t) {
                if (O->eid[t] == M.eid[a]) pa = t;
                if (O->eid[t] == M.eid[b]) pb = t;
            }
            if (pa >= 0 && pb >= 0) {
                if (pa > pb) { const int q = pa; pa = pb; pb = q; }
                const int k = A.gphase[O->eid[pa]] * NP + A.gphase[O->eid[pb]];
                en = ip_pair_energy<double>(A, k, O->eid[pa], O->eid[pb], O->phi[pa], O->phi[pb], O->gr[pa], O->gr[pb]);
            }
        } else if ((held >> a) & (held >> b) & 1u) {
            en = A.sigma[M.ph[a] * NP + M.ph[b]];
        }
        const double dot = M.gr[a][0] * M.gr[b][0] + M.gr[a][1] * M.gr[b][1] + M.gr[a][2] * M.gr[b][2];
        e += 4.0 * en * (M.phi[a] * M.phi[b] - E.pref * dot) / E.eta;
    }
    __syncthreads();
    return e;
}

// A wavefront collects the wide-interface cells of its 256 cells, in order, and takes them four at a
// time, 16 lanes each (group_gather), the pairs dealt to the lanes. Every lane's sum and the sum over
// the lanes have a fixed order. What bounds it is the instructions of the two list walks. One thread
// per cell with both lists in private memory took 108 ms at 160^3; now 2.6 ms.
template <typename TV, bool FULL>
__global__ __launch_bounds__(64) void energy_kernel(const EnergyArgs E)
{
    constexpr int G = kGroupLanes, C = 64 / G;
    __shared__ GroupArena<double, true> mem;
    __shared__ __align__(16) unsigned char old_mem[FULL ? sizeof(GroupArena<double, true>) : 16];
    auto* old = reinterpret_cast<GroupArena<double, true>*>(old_mem);
    __shared__ uint16_t pairs[kPairTable];
    __shared__ uint16_t s_list[kEnergyBlock];
    const StepArgs& A = E.cur;
    const int lane = static_cast<int>(threadIdx.x);
    const int64_t base = static_cast<int64_t>(blockIdx.x) * kEnergyBlock;
    fill_pairs(pairs);
    int n = 0;
    for (int k = 0; k < kEnergyBlock; k += 64) {
        const int64_t c = base + k + lane;
        bool wide = false;
        if (c < A.ncells && E.ip_cnt != nullptr) {
            uint32_t codes[7];
            wide = load_codes<TV>(A, make_box(A, c), A.cnt_in[c], codes);
        }
        const unsigned long long m = __ballot(wide);
        if (wide) s_list[n + __popcll(m & ((1ull << lane) - 1ull))] = static_cast<uint16_t>(k + lane);
        n += __popcll(m);
    }
    __syncthreads();
    StepArgs B = A;
    B.cnt_in = E.ip_cnt;
    B.id_in = E.ip_id;
    B.val_in = E.ip_val;
    double e = 0.0;
    for (int i0 = 0; i0 < n; i0 += C) {
        const int i = i0 + lane / G;
        const bool run = i < n;
        const int64_t c = base + (run ? s_list[i] : 0);
        bool over = false;
        e += group_energy<TV, FULL, G, kGroupCap>(E, B, run, c, mem.cell[lane / G], FULL ? &old->cell[lane / G] : nullptr,
                                                  pairs, over);
        unsigned long long todo = __ballot(over && (lane & (G - 1)) == 0);
        while (todo) {
            const int from = next_long(todo);
            const int64_t cb = base + s_list[i0 + from / G];
            bool none = false;
            e += group_energy<TV, FULL, kLongLanes, kWideSlots>(E, B, true, cb, mem.longer[lane / kLongLanes],
                                                                FULL ? &old->longer[lane / kLongLanes] : nullptr, pairs, none);
            if (none && (lane & (kLongLanes - 1)) == 0) atomicOr(E.status, 1);
        }
    }
#pragma unroll
    for (int k = 32; k >= 1; k >>= 1) e += __shfl_xor(e, k);
    if (lane == 0) E.partial[blockIdx.x] = e;
}

// Adds the per-block sums in a fixed order: thread t sums blocks t, t + 256, ... in order, then the
// tree of block_sum.
__global__ __launch_bounds__(kEnergyBlock) void energy_total_kernel(const double* __restrict__ partial, int64_t n,
                                                                    double* __restrict__ out)
{
    __shared__ double lds[kEnergyBlock];
    double v = 0.0;
    for (int64_t i = threadIdx.x; i < n; i += kEnergyBlock) v += partial[i];
    const double s = block_sum(v, lds);
    if (threadIdx.x == 0) *out = s;
}

// One thread per cell: for every thermodynamic phase the sum of its grains' values in list order
// (the FP32 implicit entry as 1 - the others), out[phase * ncells + cell].
template <typename TV>
__global__ __launch_bounds__(kEnergyBlock) void fractions_kernel(const StepArgs A, double* __restrict__ out)
{
    const int64_t c = static_cast<int64_t>(blockIdx.x) * kEnergyBlock + threadIdx.x;
    if (c >= A.ncells) return;
    CellList<kMaxSlots, double, false> L;
    load_own<kMaxSlots, TV, double, false>(A, c, A.cnt_in[c], L);
    for (int n = 0; n < A.nphases; ++n) {
        double f = 0.0;
        for (int t = 0; t < L.n0; ++t)
            if (A.gphase[L.eid[t]] == n) f += L.phi[t];
        out[static_cast<int64_t>(n) * A.ncells + c] = f;
    }
}

}  // namespace

int launch_fractions(const StepArgs& a, bool fp32, double* out, void* stream)
{
    const hipStream_t s = static_cast<hipStream_t>(stream);
    const unsigned nb = static_cast<unsigned>((a.ncells + kEnergyBlock - 1) / kEnergyBlock);
    if (fp32)
        hipLaunchKernelGGL(fractions_kernel<float>, dim3(nb), dim3(kEnergyBlock), 0, s, a, out);
    else
        hipLaunchKernelGGL(fractions_kernel<double>, dim3(nb), dim3(kEnergyBlock), 0, s, a, out);
    return static_cast<int>(hipGetLastError());
}

int64_t energy_blocks(int64_t ncells) { return (ncells + kEnergyBlock - 1) / kEnergyBlock; }

int launch_energy(const EnergyArgs& a, bool fp32, double* out, void* stream)
{
    const hipStream_t s = static_cast<hipStream_t>(stream);
    const int64_t nb = energy_blocks(a.cur.ncells);
    const dim3 grid(static_cast<unsigned>(nb));
    if (fp32) {
        if (a.full) hipLaunchKernelGGL((energy_kernel<float, true>), grid, dim3(64), 0, s, a);
        else hipLaunchKernelGGL((energy_kernel<float, false>), grid, dim3(64), 0, s, a);
    } else {
        if (a.full) hipLaunchKernelGGL((energy_kernel<double, true>), grid, dim3(64), 0, s, a);
        else hipLaunchKernelGGL((energy_kernel<double, false>), grid, dim3(64), 0, s, a);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return static_cast<int>(e);
    hipLaunchKernelGGL(energy_total_kernel, dim3(1), dim3(kEnergyBlock), 0, s, a.partial, nb, out);
    return static_cast<int>(hipGetLastError());
}

}  // namespace mpf
