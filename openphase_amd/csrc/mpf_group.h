// A cell's neighbour-merged list formed by a group of lanes (PhaseField::CalculateDerivativesSR,
// src/PhaseField.cpp:566-615): every lane fetches the lists of its neighbours of the 3^d box (two
// round trips for the whole cell), the merged list is formed with one ballot per appended grain,
// and lane t ends up with entry t and its Laplacian and gradient, summed in stencil order. Used
// where single cells or irregular lists of cells are worked on: the deferred cells of the step
// (mpf_deferred.h), the interface energy (mpf_energy.hip), the curvature (mpf_dgavg.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <float.h>
#include <stdint.h>

#include "mpf_device.h"
#include "mpf_lists.h"

namespace mpf {

namespace {

constexpr int kGroupLanes = 16;  // lanes per cell
constexpr int kGroupCap = 8;     // merged entries a group has room for
constexpr int kLongLanes = 64;   // lanes of a cell of more (up to kWideSlots)

// One cell's list and tables in LDS.
template <typename TC, bool GRAD, int CAP> struct GroupMem {
    union {
        TC a[CAP][27];                 // value of merged entry t at box position k
        struct {
            double psi[CAP][CAP + 1];  // increment of (t, u), antisymmetric
            TC sig[CAP][CAP + 1];      // interface energy of (t, u)
        } p;
    };
    TC gr[GRAD ? CAP : 1][3];
    double phi[CAP];
    TC lap[CAP];
    TC ev[CAP];                        // value in the stencil arithmetic
    double lim1[CAP], lim2[CAP];
    double vr[CAP];
    int ph[CAP];
    uint32_t eid[CAP];
};

// Lane l's part of a merged list: entry l (below ne).
template <typename TC> struct GroupList {
    int n0, ne;          // own and merged entries
    bool wide;           // the box holds an interface cell (else the list is the own one, underived)
    bool over;           // more than CAP entries, or next to a longer list: nothing else is valid
    uint32_t eid;
    double phi;          // own value (0 for an appended entry), FP32's implicit one recovered
    TC lap, gx, gy, gz;
};

// Largest n over the wavefront's groups of G lanes (n uniform within a group), in a scalar.
template <int G> __device__ __forceinline__ int wave_max(int n)
{
#pragma unroll
    for (int k = G; k < 64; k <<= 1) n = max(n, __shfl_xor(n, k));
    return __builtin_amdgcn_readfirstlane(n);
}

// The ballot's bits of this lane's group, shifted to bit 0.
template <int G> __device__ __forceinline__ unsigned long long group_bits(unsigned long long m)
{
    if (G == 64) return m;
    const int lane = static_cast<int>(threadIdx.x) & 63;
    return (m >> (lane & ~(G - 1))) & ((1ull << (G & 63)) - 1ull);
}

// The merged list of cell c of state A (when `run`) by the G lanes of this lane's group; M.eid holds
// the grains afterwards. All lanes of the wavefront call it together; loops run to the longest list
// of its groups.
template <typename TV, typename TC, bool GRAD, int G, int CAP>
__device__ __forceinline__ GroupList<TC> group_gather(const StepArgs& A, bool run, int64_t c, GroupMem<TC, GRAD, CAP>& M)
{
    constexpr int NK = (27 + G - 1) / G;   // neighbours per lane
    constexpr int RQ = CAP;                // entries of a neighbour
    constexpr bool IMPL = ListCode<TV>::kImplicit;
    const int lane = static_cast<int>(threadIdx.x) & 63, l = lane & (G - 1);
    const int64_t N = A.ncells;
    const uint32_t N32 = static_cast<uint32_t>(N);
    const uint32_t cc = static_cast<uint32_t>(run ? c : 0);

    // ---- the box: positions l, l + G of stencil order
    const int NY = A.ny, NZ = A.nz;
    const int z0 = static_cast<int>(cc % static_cast<uint32_t>(NZ));
    const int y0 = static_cast<int>((cc / static_cast<uint32_t>(NZ)) % static_cast<uint32_t>(NY));
    const int x0 = static_cast<int>(cc / (static_cast<uint32_t>(NY) * static_cast<uint32_t>(NZ)));
    const __amdgpu_buffer_rsrc_t rc = plane_rsrc(A.cnt_in, N32);
    uint32_t nb[NK];
    bool act[NK];
    uint8_t code[NK];
#pragma unroll
    for (int j = 0; j < NK; ++j) {
        const int k = l + j * G;
        const int ii = k / 9 - 1, jj = (k / 3) % 3 - 1, kk = k % 3 - 1;
        act[j] = run && k < 27 && (ii == 0 || A.dnx) && (jj == 0 || A.dny) && (kk == 0 || A.dnz);
        nb[j] = static_cast<uint32_t>((wrap1(x0 + (act[j] ? ii : 0), A.nx) * NY + wrap1(y0 + (act[j] ? jj : 0), NY)) * NZ +
                                      wrap1(z0 + (act[j] ? kk : 0), NZ));
        code[j] = buffer_load<uint8_t>(rc, act[j] ? nb[j] : kNoLoad);
    }
    const uint8_t code0 = buffer_load<uint8_t>(rc, run ? cc : kNoLoad);
    const int n0 = ListCode<TV>::count(code0), imp0 = ListCode<TV>::implicit(code0);
    int m[NK], mtop = n0;
    bool multi = false;
#pragma unroll
    for (int j = 0; j < NK; ++j) {
        m[j] = ListCode<TV>::count(code[j]);
        multi = multi || m[j] > 1;
        mtop = max(mtop, m[j]);
    }
    // a neighbour's list longer than this form holds, or the own one
    const bool wide = group_bits<G>(__ballot(multi)) != 0ull;
    bool over = group_bits<G>(__ballot(mtop > CAP)) != 0ull;
#pragma unroll
    for (int k = 1; k < 64; k <<= 1) mtop = max(mtop, __shfl_xor(mtop, k));
    const int qtop = min(__builtin_amdgcn_readfirstlane(mtop), RQ);

    // ---- lists of the lane's neighbours, and entry l of the own list. An entry that is not there, or
    // holds no value, or is in the merged list already, is grain -1
    int32_t g[NK][RQ];
    TV v[NK][RQ];
#pragma unroll
    for (int q = 0; q < RQ; ++q) {
        if (q >= 2 && q >= qtop) {
#pragma unroll
            for (int j = 0; j < NK; ++j) { g[j][q] = -1; v[j][q] = TV(0); }
            continue;
        }
        // slot 0 of the cell in place of a slot it does not use: no branch between the loads
#pragma unroll
        for (int j = 0; j < NK; ++j) {
            const int64_t at = (q < m[j] ? static_cast<int64_t>(q) * N : 0) + nb[j];
            g[j][q] = A.id_in[at];
            v[j][q] = load_val<TV>(A.val_in, at);
        }
    }
    double phi = 0.0;
    uint32_t eid = 0u;
    if (l < n0 && l < CAP) {
        eid = A.id_in[static_cast<int64_t>(l) * N + cc];
        if (!(IMPL && l == imp0)) phi = static_cast<double>(load_val<TV>(A.val_in, static_cast<int64_t>(l) * N + cc));
    }
    const bool look = wide && !over;
#pragma unroll
    for (int q = 0; q < RQ; ++q) {
        if (q >= 2 && q >= qtop) continue;
#pragma unroll
        for (int j = 0; j < NK; ++j) {
            // a lone implicit entry (FP32) has no stored value: it is 1
            if (IMPL && q == 0 && m[j] == 1 && ListCode<TV>::implicit(code[j]) == 0) v[j][q] = TV(1);
            if (!look || q >= m[j] || v[j][q] == TV(0)) g[j][q] = -1;
        }
    }
    if (l < CAP) { M.phi[l] = phi; M.eid[l] = eid; }
    __syncthreads();
    if (IMPL) {
        double others = 0.0;
        for (int t = 0; t < CAP; ++t)
            if (t < n0 && t != imp0) others += M.phi[t];
        __syncthreads();
        if (l < CAP && l < n0 && l == imp0) {
            phi = 1.0 - others;
            M.phi[l] = phi;
        }
    }

    // ---- merged list: the own entries, then grains new to the box in stencil order. Row t of
    // M.a: the value of entry t at every box position
    int ne = over ? 0 : n0;
    auto row = [&](int t, int32_t gid, bool on) {
        TC a[NK];
#pragma unroll
        for (int j = 0; j < NK; ++j) a[j] = TC(0);
#pragma unroll
        for (int q = 0; q < RQ; ++q) {
            if (q >= 2 && q >= qtop) continue;
#pragma unroll
            for (int j = 0; j < NK; ++j) {
                const bool hit = g[j][q] == gid;
                a[j] = hit ? static_cast<TC>(v[j][q]) : a[j];
                g[j][q] = hit ? -1 : g[j][q];
            }
        }
#pragma unroll
        for (int j = 0; j < NK; ++j) {
            const int k = l + j * G;
            if (on && k < 27) M.a[t][k] = a[j];
        }
    };
    const int own_top = wave_max<G>(look ? ne : 0);
    for (int t = 0; t < own_top; ++t) {
        const bool on = look && t < ne;
        row(t, on ? static_cast<int32_t>(M.eid[t]) : -2, on);
    }
    while (true) {
        // the first grain left, in stencil order then list order
        int32_t cand = -1;
        unsigned long long who = 0ull;
#pragma unroll
        for (int j = NK - 1; j >= 0; --j) {
            int32_t next = -1;
#pragma unroll
            for (int q = RQ - 1; q >= 0; --q) {
                if (q >= 2 && q >= qtop) continue;
                next = g[j][q] >= 0 ? g[j][q] : next;
            }
            const unsigned long long b = group_bits<G>(__ballot(next >= 0));
            if (b) {
                who = b;
                cand = next;
            }
        }
        if (!__any(who != 0ull)) break;
        const int leader = who ? __ffsll(static_cast<long long>(who)) - 1 : 0;
        const int32_t gid = __shfl(cand, (lane & ~(G - 1)) + leader);
        bool on = who != 0ull;
        if (on && ne >= CAP) {
            over = true;
            on = false;
#pragma unroll
            for (int q = 0; q < RQ; ++q)
#pragma unroll
                for (int j = 0; j < NK; ++j) g[j][q] = -1;
        }
        row(ne, on ? gid : -2, on);
        if (on) {
            if (l == ne) eid = static_cast<uint32_t>(gid);
            ++ne;
        }
    }
    if (l < CAP) M.eid[l] = eid;
    const bool work = run && !over && wide;
    __syncthreads();

    // ---- Laplacian (gradient) of entry l, in stencil order
    TC lap = TC(0), gx = TC(0), gy = TC(0), gz = TC(0);
    if (work && l < ne) {
#pragma unroll
        for (int k = 0; k < 27; ++k) {
            const int ii = k / 9 - 1, jj = (k / 3) % 3 - 1, kk = k % 3 - 1;
            const int nz = (ii != 0) + (jj != 0) + (kk != 0);
            const TC a = M.a[l][k];
            lap += static_cast<TC>(A.wl[nz]) * a;
            if (GRAD && k != 13) {
                const TC w = static_cast<TC>(A.wg[nz]);
                if (ii) gx = gx + (ii < 0 ? -w : w) * a;
                if (jj) gy = gy + (jj < 0 ? -w : w) * a;
                if (kk) gz = gz + (kk < 0 ? -w : w) * a;
            }
        }
    }
    __syncthreads();  // M.p may take M.a's place
    return GroupList<TC>{n0, ne, wide, over, eid, phi, lap, gx, gy, gz};
}

// The groups' memory of one wavefront: four cells, or one of a longer list
template <typename TC, bool GRAD> union GroupArena {
    GroupMem<TC, GRAD, kGroupCap> cell[64 / kGroupLanes];
    GroupMem<TC, GRAD, kWideSlots> longer[64 / kLongLanes];
};

constexpr int kPairTable = kWideSlots * (kWideSlots - 1) / 2;

// The next cell of a wavefront's groups whose bit (at the group's first lane) is set in `todo`: that
// lane.
__device__ __forceinline__ int next_long(unsigned long long& todo)
{
    const int from = __ffsll(static_cast<long long>(todo)) - 1;
    todo &= todo - 1ull;
    return from;
}

// Pair p = b (b - 1) / 2 + a as a | b << 8. One wavefront.
__device__ __forceinline__ void fill_pairs(uint16_t* pairs)
{
    for (int p = static_cast<int>(threadIdx.x); p < kPairTable; p += 64) {
        int b = 1;
        while (b * (b + 1) / 2 <= p) ++b;
        pairs[p] = static_cast<uint16_t>((p - b * (b - 1) / 2) | (b << 8));
    }
}

}  // namespace

}  // namespace mpf
