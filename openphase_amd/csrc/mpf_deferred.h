// Deferred cells of the step: the cells whose neighbourhood the main step kernels cannot hold
// (merged lists of more than four entries, neighbours with long lists, too many grains in a tile).
// Included by mpf_kernels_variant.hip.
//
// A group of lanes takes one cell: 16 lanes, four cells per wavefront. What bounds such a cell is
// latency - one chain of dependent loads, list searches and divisions - so its work is spread over
// the group instead of run by one lane: the merged list is formed by the group (group_gather), lane t
// holds entry t (Laplacian, limiter bounds, merge, finalize) and the pair increments are dealt to
// the lanes. Sums that the reference forms in an order are formed by one lane in that order (stencil
// order, list order, pair order), so every value equals the one-lane form bit for bit.
//
// Lists are held in LDS with run-time lengths, so one kernel takes every length: a cell of more
// than kGroupCap merged entries, or next to a list of more than kGroupCap, is done again by the
// whole wavefront with room for kWideSlots. Measured against one thread per cell with register
// lists in three launches (2-6, 7-10 and up to 16 entries), mid-run states, FP64: 16 us instead of
// 114 at 2D 512^2 and 18 instead of 120 at 96^2 (a few hundred cells that waited on their own
// latency), 1.07 ms instead of 2.62 at 256^3; 64 FP32 domains in one launch 60 us instead of 354.
// Three wavefronts per SIMD: four spill (256^3, mid-run: 0.43 ms FP64, 0.48 FP32 where three take 0.34
// and 0.37; eight steps of a fresh start 28.7 and 27.2 ms instead of 26.9 and 24.4).
#pragma once

#include <hip/hip_runtime.h>
#include <float.h>
#include <stdint.h>

#include "mpf_device.h"
#include "mpf_group.h"
#include "mpf_lists.h"
#include "mpf_step_ops.h"

namespace mpf {

namespace {

constexpr int kVolSlots = 32;    // grains of the wavefront's volume table

struct VolTable {
    int32_t key[kVolSlots];
    unsigned long long acc[kVolSlots][kLimbs];
};

// Adds one entry's value to the wavefront's table of exact volume sums, or to the global sums
// when the table is full.
__device__ __forceinline__ void table_volume_add(VolTable& V, uint32_t g, double v, unsigned long long* acc, bool& bad)
{
    unsigned long long l[kLimbs];
    value_limbs(v, l, bad);
    unsigned long long* dst = acc + static_cast<int64_t>(g) * kLimbs;
    uint32_t h = (g * 0x9E3779B1u) >> 27;
    for (int i = 0; i < kVolSlots; ++i, h = (h + 1u) & (kVolSlots - 1)) {
        int k = *static_cast<volatile int32_t*>(&V.key[h]);
        if (k == -1) {
            k = atomicCAS(&V.key[h], -1, static_cast<int>(g));
            if (k == -1) k = static_cast<int>(g);
        }
        if (k == static_cast<int>(g)) {
            dst = V.acc[h];
            break;
        }
    }
#pragma unroll
    for (int i = 0; i < kLimbs; ++i)
        if (l[i]) atomicAdd(&dst[i], l[i]);
}

// The step of cell c (when `run`) by the G lanes of this lane's group. Returns true (uniform in
// the group) when the cell needs more than CAP entries: nothing was written then. All lanes of the
// wavefront call it together; loops run to the longest list of its groups.
template <typename TV, typename TC, bool GRAD, bool DG, int G, int CAP>
__device__ __forceinline__ bool group_cell(const StepArgs& A, bool run, int64_t c, GroupMem<TC, GRAD, CAP>& M,
                                           bool count_long, const uint16_t* pairs, VolTable& V, double& emax,
                                           double& mmax, bool& bad)
{
    constexpr bool IMPL = ListCode<TV>::kImplicit;
    const int lane = static_cast<int>(threadIdx.x) & 63, l = lane & (G - 1);
    const int64_t N = A.ncells;
    const GroupList<TC> L = group_gather<TV, TC, GRAD, G, CAP>(A, run, c, M);
    const int n0 = L.n0, ne = L.ne;
    const uint32_t eid = L.eid;
    double phi = L.phi;
    const bool go = run && !L.over;          // the cell's result is written by this call
    const bool work = go && L.wide;
    if (work && ne > 6 && count_long && l == 0) atomicAdd(&A.work_count[2], 1u);
    const int top = wave_max<G>(work ? ne : 0);
    double vr = 0.0;
    int ph = 0;
    if (work && l < ne) {
        ph = A.gphase[eid];
        vr = A.gvr[eid];
    }
    const TC ev = static_cast<TC>(phi);
    if (l < CAP) {
        M.lap[l] = L.lap;
        M.ev[l] = ev;
        M.ph[l] = ph;
        M.vr[l] = vr;
        if (GRAD) { M.gr[GRAD ? l : 0][0] = L.gx; M.gr[GRAD ? l : 0][1] = L.gy; M.gr[GRAD ? l : 0][2] = L.gz; }
    }
    __syncthreads();

    // ---- pair increments (compute_cell's formulas), pair p = b (b - 1) / 2 + a to lane p mod G
    const int NP = A.nphases;
    double localn = 0.0;
    if (A.consider_nucleus) {
        for (int t = 0; t < top; ++t) localn += t < ne ? M.vr[t] : 0.0;
    } else {
        localn = static_cast<double>(ne);
    }
    const double norm_1 = 1.0 / localn;
    const bool uni = A.uniform != 0 && group_bits<G>(__ballot(work && l < ne && vr != 1.0)) == 0ull;
    const TC P = static_cast<TC>(A.prefactor);
    const int np = work ? ne * (ne - 1) / 2 : 0;
    const int ptop = top * (top - 1) / 2;
    if (__any(work && !uni)) {
        for (int p0 = 0; p0 < ptop; p0 += G) {
            const int p = p0 + l;
            if (p < np && !uni) {
                const int a = pairs[p] & 255, b = pairs[p] >> 8;
                if (GRAD) {
                    TC da[3], db[3];
                    for (int d = 0; d < 3; ++d) { da[d] = M.gr[GRAD ? a : 0][d]; db[d] = M.gr[GRAD ? b : 0][d]; }
                    const TC en = ip_pair_energy<TC>(A, M.ph[a] * NP + M.ph[b], M.eid[a], M.eid[b], M.ev[a], M.ev[b], da, db);
                    M.p.sig[a][b] = en;
                    M.p.sig[b][a] = en;
                } else {
                    M.p.sig[a][b] = static_cast<TC>(A.sigma[M.ph[a] * NP + M.ph[b]]);
                    M.p.sig[b][a] = static_cast<TC>(A.sigma[M.ph[b] * NP + M.ph[a]]);
                }
            }
        }
        __syncthreads();
    }
    for (int p0 = 0; p0 < ptop; p0 += G) {
        const int p = p0 + l;
        if (p < np) {
            const int a = pairs[p] & 255, b = pairs[p] >> 8;
            const int k = M.ph[a] * NP + M.ph[b];
            TC d, mob;
            if (uni) {
                const TC s0 = static_cast<TC>(A.sigma0);
                const TC mf = static_cast<TC>(A.mu0) * static_cast<TC>(norm_1);
                d = s0 * ((M.lap[a] + P * M.ev[a]) - (M.lap[b] + P * M.ev[b]));
                d *= mf;
                mob = static_cast<TC>(A.mu0);
                emax = smax(emax, static_cast<double>(s0));
                mmax = smax(mmax, A.mu0);
            } else {
                const double scaled = sqrt(M.vr[a] * M.vr[b]);
                const TC scale = static_cast<TC>(scaled);
                const TC cf = TC(0.5) * (TC(1.0) + scale) * P;
                d = M.p.sig[a][b] * ((M.lap[a] + cf * M.ev[a]) - (M.lap[b] + cf * M.ev[b]));
                for (int g2 = 0; g2 < ne; ++g2) {
                    if (g2 == a || g2 == b) continue;
                    d += (M.p.sig[b][g2] - M.p.sig[a][g2]) * (M.lap[g2] + cf * M.ev[g2]);
                    if (A.tj_model == 0) {
                        if (A.tj_factor != 0.0 || scaled < 1.0) {
                            const int pg = M.ph[g2];
                            const TC e3 = static_cast<TC>(A.sigma[k]) + static_cast<TC>(A.sigma[M.ph[b] * NP + pg]) +
                                          static_cast<TC>(A.sigma[M.ph[a] * NP + pg]);
                            d += static_cast<TC>(smax(A.tj_factor, (1.0 - scaled))) * P * e3 *
                                 (M.ev[a] * M.ev[g2] - M.ev[b] * M.ev[g2]);
                        }
                    } else if (A.tj_model == 1) {
                        d += static_cast<TC>(A.tj_energy) * P * (M.ev[a] * M.ev[g2] - M.ev[b] * M.ev[g2]);
                    }
                }
                mob = static_cast<TC>(A.mu[k]);
                emax = smax(emax, static_cast<double>(M.p.sig[a][b]));
                mmax = smax(mmax, static_cast<double>(mob));
                if (DG && A.reg) {
                    d = d * mob * static_cast<TC>(norm_1) * scale;
                    if (A.reg_active) {
                        d *= static_cast<TC>(A.reg_factor);
                        if (A.curv != nullptr && n0 > 1 && b < n0) {
                            const TC kappa = static_cast<TC>(A.curv[static_cast<int64_t>(p) * N + c]);
                            d += kappa * mob * sqrt(M.ev[a] * M.ev[b]) * static_cast<TC>(A.dg_prefactor);
                        }
                    }
                } else {
                    d *= mob * static_cast<TC>(norm_1) * scale;
                }
            }
            if (DG && n0 > 1 && A.dg_mode[k] == 1) {
                const TC raw = dg_local<TC>(A, a, b, n0, c, k);
                const TC weight = sqrt(M.ev[a] * M.ev[b]);
                const TC allowed = static_cast<TC>(A.dg_allowed[k]);
                const TC dgl = allowed * tanh(raw / allowed);
                d += dgl * mob * weight * static_cast<TC>(A.dg_prefactor);
            }
            M.p.psi[a][b] = static_cast<double>(d);
            M.p.psi[b][a] = -static_cast<double>(d);
        }
    }
    __syncthreads();

    // ---- limiter (FP64): lane t holds the increments psi of (t, u) in registers, 0 where there is
    // none (the reference drops such a pair from the increment list; adding 0 changes no sum). Both
    // lanes of a pair scale it by the same factors, so the two stay exact negatives
    const double dt = A.dt;
    if (work && ne == 2 && l == 0) {
        double d = M.p.psi[0][1];
        const double va = d * dt;
        const double old = phi;
        if ((old == 0.0 && va < 0.0) || (old == 1.0 && va > 0.0)) {
            d = 0.0;
        } else {
            const double nv = old + va;
            double norm = 1.0;
            if (nv < 0.0) norm *= -old / va;
            else if (nv > 1.0) norm *= (1.0 - old) / va;
            if (norm > DBL_EPSILON) d *= norm;
            else d = 0.0;
        }
        M.p.psi[0][1] = d;
        M.p.psi[1][0] = -d;
    }
    __syncthreads();
    double psi[CAP];
#pragma unroll
    for (int u = 0; u < CAP; ++u) psi[u] = work && l < ne && u < ne && u != l ? M.p.psi[l][u] : 0.0;
    const bool many = work && ne > 2;
    if (__any(many)) {
        // zero the pairs that would push a field at 0 below or at 1 above, entry after entry
        int done = -1;
        while (true) {
            double dpsi = 0.0;
#pragma unroll
            for (int u = 0; u < CAP; ++u) dpsi += psi[u];
            const bool stop = many && l < ne && l > done && ((phi == 0.0 && dpsi < 0.0) || (phi == 1.0 && dpsi > 0.0));
            const unsigned long long b = group_bits<G>(__ballot(stop));
            if (!__any(stop)) break;
            if (b) {
                done = __ffsll(static_cast<long long>(b)) - 1;
#pragma unroll
                for (int u = 0; u < CAP; ++u) psi[u] = u == done || l == done ? 0.0 : psi[u];
            }
        }
        bool needed = many;
        for (int iter = 1; iter <= 25 && __any(needed); ++iter) {
            double pos = 0.0, neg = 0.0;
#pragma unroll
            for (int u = 0; u < CAP; ++u) {
                pos += fmax(psi[u], 0.0);
                neg += fmin(psi[u], 0.0);
            }
            double lim1 = 1.0, lim2 = 1.0;
            if (needed && l < ne) {
                const double npf = phi + (pos + neg) * dt;
                if (npf < 0.0) lim2 = smin(lim2, -(phi + pos * dt) / (neg * dt));
                if (npf > 1.0) lim1 = smin(lim1, (1.0 - (phi + neg * dt)) / (pos * dt));
            }
            // factors of 1 all over leave every increment as it is
            needed = needed && group_bits<G>(__ballot(lim1 < 1.0 || lim2 < 1.0)) != 0ull;
            if (!__any(needed)) break;
            if (l < CAP) {
                M.lim1[l] = lim1;
                M.lim2[l] = lim2;
            }
            __syncthreads();
            bool again = false;
            if (needed && l < ne) {
#pragma unroll
                for (int u = 0; u < CAP; ++u) {
                    // (a negative increment: entry l loses, u gains)
                    const double t = psi[u] < 0.0 ? smin(lim2, M.lim1[u]) : smin(lim1, M.lim2[u]);
                    again = again || (psi[u] != 0.0 && t < 1.0);
                    psi[u] = psi[u] != 0.0 ? psi[u] * t : 0.0;
                }
            }
            needed = needed && group_bits<G>(__ballot(again)) != 0ull;
            __syncthreads();
        }
        // plausibility check of the limited increments (warning count)
        if (many && l < ne) {
            double tv = phi;
#pragma unroll
            for (int u = 0; u < CAP; ++u) tv += fabs(psi[u] * dt) < DBL_EPSILON ? 0.0 : psi[u] * dt;
            if (tv < -FLT_EPSILON || tv > 1.0 + FLT_EPSILON) atomicAdd(A.warnings, 1ull);
        }
    }

    // ---- merge, then finalize (NodePF::finalize); a bulk cell keeps its list
    bool keep = go && l < ne;
    if (work && l < ne) {
#pragma unroll
        for (int u = 0; u < CAP; ++u) {
            const double value = psi[u] * dt;
            phi += fabs(value) >= DBL_EPSILON ? value : 0.0;
        }
        if (phi >= 1.0 - DBL_EPSILON) phi = 1.0;
        if (phi <= 0.0 + DBL_EPSILON) { phi = 0.0; keep = false; }
        M.phi[l] = phi;
    }
    unsigned long long kept = group_bits<G>(__ballot(keep));
    const int ns = __popcll(kept);
    __syncthreads();
    if (work) {
        double total = 0.0;
        for (int t = 0; t < ne; ++t) total += M.phi[t];
        if (ns > 1) {
            const double norm = 1.0 / total;
            if (keep) phi *= norm;
        } else if (ns == 1) {
            if (keep) phi = 1.0;
        }
        if (ns == 0 && l == 0) atomicOr(&A.status[kStatusEmpty], 1);
    }
    __syncthreads();

    // ---- store (store_cell): FP32 lists hold their first largest entry implicitly
    if (go && ns > A.slots) {
        if (l == 0) {
            atomicOr(&A.status[kStatusOverflow], 1);
            atomicMin(A.first_overflow, static_cast<unsigned long long>(c));
        }
        keep = false;
    } else if (go) {
        const int w = __popcll(kept & ((1ull << l) - 1ull));
        const TV sv = static_cast<TV>(phi);
        int imp = -1;
        if (IMPL) {
            if (l < CAP) M.phi[l] = phi;
            __builtin_amdgcn_wave_barrier();
            double vmax = -1.0, others = 0.0;
            for (int t = 0; t < ne; ++t)
                if (((kept >> t) & 1ull) && M.phi[t] > vmax) { vmax = M.phi[t]; imp = t; }
            for (int t = 0; t < ne; ++t)
                if (((kept >> t) & 1ull) && t != imp) others += static_cast<double>(static_cast<TV>(M.phi[t]));
            phi = l == imp ? 1.0 - others : static_cast<double>(sv);
        }
        if (keep) {
            A.id_out[static_cast<int64_t>(w) * N + c] = static_cast<uint16_t>(eid);
            if (!(IMPL && l == imp && ns == 1)) static_cast<TV*>(A.val_out)[static_cast<int64_t>(w) * N + c] = sv;
        }
        if (l == 0) {
            const int wi = IMPL && imp >= 0 ? __popcll(kept & ((1ull << imp) - 1ull)) : 0;
            A.cnt_out[c] = static_cast<uint8_t>(IMPL ? (ns | (wi << 4)) : ns);
        }
    }
    if (keep) table_volume_add(V, eid, phi, A.vol_acc, bad);
    return run && L.over;
}

// One wavefront per block; neighbours in a domain's list of deferred cells are neighbours in the grid.
template <typename TV, typename TC, bool GRAD, bool DG>
__global__ __launch_bounds__(64, 3) void deferred_kernel(const StepArgs* __restrict__ batch, int32_t ndom)
{
    constexpr int G = kGroupLanes, C = 64 / G;
    __shared__ GroupArena<TC, GRAD> mem;
    __shared__ uint16_t pairs[kPairTable];
    __shared__ VolTable V;
    const unsigned per = gridDim.x / static_cast<unsigned>(ndom);
    const unsigned dom = blockIdx.x / per, part = blockIdx.x - dom * per;
    const StepArgs& A = batch[dom];
    const unsigned n = A.work_count[0];
    if (n == 0u) return;
    // Runs of up to four rounds of C cells. Blocks go to the eight XCDs in turn; each XCD takes one
    // eighth of the list and its wavefronts take that part's runs in turn, so that what is worked on
    // at a time is one stretch of the list, whose neighbourhoods overlap in the XCD's L2 (256^3 FP64,
    // 750,000 cells: 0.81 instead of 2.7 GB from memory, 1.07 instead of 1.41 ms)
    const unsigned rounds = (n + C - 1) / C, length = min(4u, max(1u, rounds / per)), runs = (rounds + length - 1) / length;
    const unsigned xcds = per % 8u == 0u ? 8u : 1u, xcd = part % xcds;
    const unsigned last = static_cast<unsigned>(static_cast<uint64_t>(runs) * (xcd + 1u) / xcds);
    unsigned turn = static_cast<unsigned>(static_cast<uint64_t>(runs) * xcd / xcds) + part / xcds;
    if (turn >= last) return;
    const int lane = static_cast<int>(threadIdx.x);
    fill_pairs(pairs);
    if (lane < kVolSlots) V.key[lane] = -1;
    for (int i = lane; i < kVolSlots * kLimbs; i += 64) (&V.acc[0][0])[i] = 0ull;
    __syncthreads();
    double emax = 0.0, mmax = 0.0;
    bool bad = false;
    for (; turn < last; turn += per / xcds) {
        const unsigned begin = turn * length * C, end = min(n, begin + length * C);
        for (unsigned base = begin; base < end; base += C) {
            const unsigned i = base + static_cast<unsigned>(lane / G);
            const bool run = i < end;
            const uint32_t entry = run ? A.work_list[i] : 0u;
            const int64_t c = entry & ~(1u << 31);
            const bool uncounted = (entry >> 31) == 0u;   // as more than six merged entries
            const bool big = group_cell<TV, TC, GRAD, DG, G, kGroupCap>(A, run, c, mem.cell[lane / G], uncounted, pairs, V, emax,
                                                                        mmax, bad);
            unsigned long long todo = __ballot(big && (lane & (G - 1)) == 0);
            __syncthreads();
            while (todo) {
                const int from = next_long(todo);
                const int64_t cb = static_cast<int64_t>(__shfl(static_cast<int>(c), from));
                const bool first = __shfl(uncounted ? 1 : 0, from) != 0;
                if (group_cell<TV, TC, GRAD, DG, kLongLanes, kWideSlots>(A, true, cb, mem.longer[lane / kLongLanes], first, pairs,
                                                                         V, emax, mmax, bad) &&
                    (lane & (kLongLanes - 1)) == 0) {
                    atomicOr(&A.status[kStatusOverflow], 1);
                    atomicMin(A.first_overflow, static_cast<unsigned long long>(cb));
                }
                __syncthreads();
            }
        }
        // the run's volumes; another run's grains are others
        for (int i = lane; i < kVolSlots * kLimbs; i += 64) {
            const int s = i / kLimbs;
            const unsigned long long x = V.acc[s][i - s * kLimbs];
            if (x) atomicAdd(&A.vol_acc[static_cast<int64_t>(V.key[s]) * kLimbs + (i - s * kLimbs)], x);
            V.acc[s][i - s * kLimbs] = 0ull;
        }
        __syncthreads();
        if (lane < kVolSlots) V.key[lane] = -1;
        __syncthreads();
    }
    note_maxima(A.obs, emax, mmax);
    if (__any(bad) && lane == 0) atomicOr(&A.status[kStatusVolumeRange], 1);
}

}  // namespace

}  // namespace mpf
