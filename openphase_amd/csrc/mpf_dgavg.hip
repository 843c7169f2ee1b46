// MI355X (gfx950) kernels of the driving-force averaging over the interface
// (DrivingForce::Average with Averaging on, src/DrivingForce.cpp:242-255).
//
// The reference keeps a Force entry per VALUE-mode phase-field pair of every interface node
// (UserDrivingForce::SetDrivingForce, src/UserDrivingForce.cpp:152-175) with raw = Value(phaseA,
// phaseB) and weight = sqrt(phiA phiB) (SetWeights, :276-291). CollectAverage (:293-379) replaces
// raw by its weighted mean over the sphere of radius Range (tmp); DistributeAverage (:381-478)
// averages tmp again (average), which MergePhaseFieldIncrementsSR then limits and merges. Here no
// Force storage exists: an entry's raw value and weight follow from the node's own list (grains,
// values) and the phase-pair table, so both passes read the step-start state directly, the sphere's
// offsets x outer, z inner (the reference's loop order; every sum is formed in that order); a
// neighbour contributes when it is an interface cell holding both grains. tmp and the averaged value are stored per pair of own
// entries (a < b at plane b(b-1)/2 + a) for the step kernel, which reads them in place of the
// phase-pair value.
//
// Built with -ffp-contract=off like the step kernels: the FP64 sums are the reference's.

#include <hip/hip_runtime.h>
#include <float.h>
#include <stdint.h>

#include "mpf_device.h"
#include "mpf_group.h"
#include "mpf_lists.h"
#include "mpf_step_ops.h"

namespace mpf {

namespace {

__device__ __forceinline__ int pair_plane(int a, int b)  // a < b
{
    return b * (b - 1) / 2 + a;
}

// Value of own entry t of cell c (count code `code`). FP32 lists recover their implicit entry as
// 1 - (sum of the others in slot order), as the step does.
template <typename TV>
__device__ double entry_value(const StepArgs& A, int64_t c, uint8_t code, int t)
{
    const int64_t N = A.ncells;
    const int imp = ListCode<TV>::implicit(code);
    if (t != imp) return static_cast<double>(load_val<TV>(A.val_in, static_cast<int64_t>(t) * N + c));
    const int n = ListCode<TV>::count(code);
    double others = 0.0;
    for (int s = 0; s < n; ++s)
        if (s != imp) others += static_cast<double>(load_val<TV>(A.val_in, static_cast<int64_t>(s) * N + c));
    return 1.0 - others;
}

// Lane l's value of x (l uniform across the wavefront).
__device__ __forceinline__ double lane_value(double x, int l)
{
    const unsigned long long b = static_cast<unsigned long long>(__double_as_longlong(x));
    const unsigned lo = static_cast<unsigned>(__builtin_amdgcn_readlane(static_cast<int>(static_cast<unsigned>(b)), l));
    const unsigned hi = static_cast<unsigned>(__builtin_amdgcn_readlane(static_cast<int>(static_cast<unsigned>(b >> 32)), l));
    return __longlong_as_double(static_cast<long long>((static_cast<unsigned long long>(hi) << 32) | lo));
}

constexpr int kAvgCells = 64;                 // cells per block
constexpr int kAvgWaves = kAvgBlock / 64;     // wavefronts per block
constexpr int kAvgChunks = 2;                 // offsets of a lane looked up together

// The lists of the cells at the sphere's offsets t0 + 64 u + lane: all chunks' counts are loaded
// together, then their first four grains (branch-free buffer loads).
struct NearLists {
    uint32_t nb[kAvgChunks];
    uint8_t code[kAvgChunks];
    int n[kAvgChunks];            // entries of an interface cell, else 0
    uint32_t g[kAvgChunks][4];
};

template <typename TV>
__device__ __forceinline__ void near_lists(const SphereArgs& P, int x, int y, int z, int t0, NearLists& L)
{
    const StepArgs& A = P.s;
    const int64_t N = A.ncells;
    const uint32_t N32 = static_cast<uint32_t>(N);
    const int lane = static_cast<int>(threadIdx.x) & 63;
#pragma unroll
    for (int u = 0; u < kAvgChunks; ++u) {
        const int t = min(t0 + 64 * u + lane, P.noff - 1);
        const int ii = P.off[3 * t], jj = P.off[3 * t + 1], kk = P.off[3 * t + 2];
        L.nb[u] = (static_cast<uint32_t>(wrap1(x + ii, A.nx)) * static_cast<uint32_t>(A.ny) + static_cast<uint32_t>(wrap1(y + jj, A.ny))) *
                      static_cast<uint32_t>(A.nz) + static_cast<uint32_t>(wrap1(z + kk, A.nz));
    }
#pragma unroll
    for (int u = 0; u < kAvgChunks; ++u) L.code[u] = A.cnt_in[L.nb[u]];
#pragma unroll
    for (int u = 0; u < kAvgChunks; ++u) {
        const int n = t0 + 64 * u + lane < P.noff ? ListCode<TV>::count(L.code[u]) : 0;
        L.n[u] = n < 2 ? 0 : n;
#pragma unroll
        for (int s = 0; s < 4; ++s)
            L.g[u][s] = buffer_load<uint16_t>(plane_rsrc(A.id_in + s * N, N32 * 2u), s < L.n[u] ? L.nb[u] * 2u : kNoLoad);
    }
}

// A pair of grains at one neighbour: NodeDF::get_weight / get_raw / get_tmp
// (include/Containers/NodeDF.h:401-410). An entry exists on an interface cell (more than one own
// entry) whose list holds both grains (the pair's phases give the same mode everywhere); entries of
// zero-valued appended grains weigh 0 and never count.
struct PairTerm {
    bool has, fwd;   // fwd: ga precedes gb in the list (the entry's stored order; else the sign flips)
    double w, v;     // sqrt(phi_a phi_b) and, given `src`, the pair's stored value there
};

// The pair (ga, gb) at the cells of L, its values and stored values loaded together; false when none
// of the wavefront's cells holds it. Lanes without the pair read cell c.
template <typename TV>
__device__ __forceinline__ bool pair_terms(const StepArgs& A, const NearLists& L, int64_t c, uint32_t ga, uint32_t gb,
                                           const double* src, PairTerm (&T)[kAvgChunks])
{
    const int64_t N = A.ncells;
    int ia[kAvgChunks], ib[kAvgChunks];
    bool any = false;
#pragma unroll
    for (int u = 0; u < kAvgChunks; ++u) {
        ia[u] = ib[u] = -1;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            ia[u] = s < L.n[u] && L.g[u][s] == ga ? s : ia[u];
            ib[u] = s < L.n[u] && L.g[u][s] == gb ? s : ib[u];
        }
        for (int s = 4; s < L.n[u]; ++s) {
            const uint32_t gs = A.id_in[static_cast<int64_t>(s) * N + L.nb[u]];
            ia[u] = gs == ga ? s : ia[u];
            ib[u] = gs == gb ? s : ib[u];
        }
        T[u].has = ia[u] >= 0 && ib[u] >= 0;
        T[u].fwd = ia[u] < ib[u];
        any = any || T[u].has;
    }
    if (!__any(any)) return false;
    double va[kAvgChunks], vb[kAvgChunks];
#pragma unroll
    for (int u = 0; u < kAvgChunks; ++u) {
        T[u].v = 0.0;
        if constexpr (ListCode<TV>::kImplicit) {
            va[u] = vb[u] = 0.0;
            if (T[u].has) {
                va[u] = entry_value<TV>(A, L.nb[u], L.code[u], ia[u]);
                vb[u] = entry_value<TV>(A, L.nb[u], L.code[u], ib[u]);
            }
        } else {
            va[u] = load_val<TV>(A.val_in, T[u].has ? static_cast<int64_t>(ia[u]) * N + L.nb[u] : c);
            vb[u] = load_val<TV>(A.val_in, T[u].has ? static_cast<int64_t>(ib[u]) * N + L.nb[u] : c);
        }
        if (src != nullptr) {
            const int plane = T[u].fwd ? pair_plane(ia[u], ib[u]) : pair_plane(ib[u], ia[u]);
            T[u].v = src[T[u].has ? static_cast<int64_t>(plane) * N + L.nb[u] : c];
        }
    }
#pragma unroll
    for (int u = 0; u < kAvgChunks; ++u) T[u].w = sqrt(va[u] * vb[u]);
    return true;
}

// Adds the weights and terms that count of kAvgChunks chunks to `acc` in offset order (even lanes: the
// sum of the weights, odd lanes: that of the terms) and returns how many there were. They are
// compacted into LDS and added eight at a time by every lane, padded with +0, which changes no sum
// here (none is ever -0): two instructions per term, where reading each from its lane's registers took
// about twelve and made up half of the first pass.
__device__ __forceinline__ int ordered_add(double (&buf)[64 * kAvgChunks + 8][2], const bool (&ok)[kAvgChunks],
                                           const double (&wt)[kAvgChunks], const double (&term)[kAvgChunks], double& acc)
{
    const int lane = static_cast<int>(threadIdx.x) & 63;
    int m = 0;
#pragma unroll
    for (int u = 0; u < kAvgChunks; ++u) {
        const unsigned long long okm = __ballot(ok[u]);
        if (ok[u]) {
            const int at = m + __popcll(okm & ((1ull << lane) - 1ull));
            buf[at][0] = wt[u];
            buf[at][1] = term[u];
        }
        m += __popcll(okm);
    }
    if (m == 0) return 0;
    if (lane < 16) buf[m + (lane >> 1)][lane & 1] = 0.0;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    for (int i = 0; i < m; i += 8) {
        double e[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) e[q] = buf[i + q][lane & 1];
#pragma unroll
        for (int q = 0; q < 8; ++q) acc += e[q];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    return m;
}

// SECOND = false: CollectAverage into tmp; true: DistributeAverage into avg, of the driving force or
// (CURV) of the curvature, for spheres too large for staged tiles (sphere_tile_kernel). A block takes
// 64 consecutive cells and compacts their interface cells in LDS; its wavefronts take them in turn.
// Lane p holds pair p of the cell (64 at a time): its bounds, own value and sums. The 64 lanes look up
// the lists at 64 kAvgChunks sphere offsets at once, every pair of the cell is matched against them, and its
// terms are added in offset order, chunk after chunk, as the reference's sums are formed.
//
// The curvature: collect is InterfaceRegularization::CollectAverageSR
// (src/InterfaceRegularization.cpp:196-223), distribute DistributeAverageSR (:225-274); the pair's
// weight is sqrt(phi_a phi_b) (SetWeightsSR, :178-194) on interface cells. Collect: for a weight above
// the threshold, the mean of the neighbours' raw weighted by weight * (Range - |offset|), over terms
// above DBL_EPSILON, if their sum exceeds DBL_EPSILON (else the fresh entry's 0). Distribute: for a
// weight above DBL_EPSILON, the plain mean of the tmp of the neighbours whose weight exceeds the
// threshold, or the own tmp. No grain is a Seed here (grains enter as Stable; only nucleation makes
// seeds), so the entries below those bounds keep 0.
//
// What bounds it is the lookups' round trips. 96^3, 485 offsets (collect / distribute): lists looked up
// for each pair anew and terms read from lane registers 0.64 / 1.88 ms, terms added from LDS and two
// chunks in flight 0.33 / 1.74 ms, lists looked up once for all pairs of a cell 0.31 / 1.32 ms.
// Tiles against this kernel (ms, 20 steps in 2D, 4 in 3D): curvature, 25 offsets in 2D and 93 in 3D,
// 256^2 4.07 / 3.63, 512^2 5.36 / 6.51, 48^3 5.89 / 3.77, 64^3 5.40 / 5.91, 96^3 8.17 / 10.6: tiles from
// kSphereGrid cells on. Driving force, 69 offsets in 2D, 128^2 3.03 / 1.95, 512^2 4.86 / 3.75: in 2D two
// chunks hold the sphere, and tiles stay to kSphereOffsets2d.
template <typename TV, bool SECOND, bool CURV>
__global__ __launch_bounds__(kAvgBlock) void sphere_wave_kernel(const SphereArgs P)
{
    __shared__ uint16_t s_list[kAvgCells];
    __shared__ int s_count;
    __shared__ double s_terms[kAvgWaves][64 * kAvgChunks + 8][2];
    const StepArgs& A = P.s;
    const int64_t N = A.ncells;
    const int tid = static_cast<int>(threadIdx.x), lane = tid & 63, wave = tid >> 6;
    const int64_t base = static_cast<int64_t>(blockIdx.x) * kAvgCells;
    if (wave == 0) {
        // pairs of own entries live on interface cells (more than one own entry) only
        const int64_t c0 = base + lane;
        const bool inter = lane < kAvgCells && c0 < N && ListCode<TV>::count(A.cnt_in[c0]) >= 2;
        const unsigned long long m = __ballot(inter);
        if (inter) s_list[__popcll(m & ((1ull << lane) - 1ull))] = static_cast<uint16_t>(lane);
        if (lane == 0) s_count = __popcll(m);
    }
    __syncthreads();
    const int ninter = s_count;
    const int64_t nyz = static_cast<int64_t>(A.ny) * A.nz;
    const int NP = A.nphases;
    const double* src = SECOND ? P.tmp : (CURV ? P.raw : nullptr);
    for (int i = wave; i < ninter; i += kAvgWaves) {
        const int64_t c = base + s_list[i];
        const uint8_t code = A.cnt_in[c];
        const int n = ListCode<TV>::count(code);
        const int x = static_cast<int>(c / nyz), y = static_cast<int>((c / A.nz) % A.ny), z = static_cast<int>(c % A.nz);
        const int npairs = n * (n - 1) / 2;
        for (int p0 = 0; p0 < npairs; p0 += 64) {
            // ---- lane's pair (a, b), a < b, at plane b (b - 1) / 2 + a
            const int p = p0 + lane;
            uint32_t ga = 0u, gb = 0u;
            double cut = 0.0, vab = 0.0, vba = 0.0, own = 0.0;
            bool entry = false, run = false;
            if (p < npairs) {
                int b = 1;
                while (b * (b + 1) / 2 <= p) ++b;
                const int a = p - b * (b - 1) / 2;
                ga = A.id_in[static_cast<int64_t>(a) * N + c];
                gb = A.id_in[static_cast<int64_t>(b) * N + c];
                const double w = sqrt(entry_value<TV>(A, c, code, a) * entry_value<TV>(A, c, code, b));
                if (CURV) {
                    entry = true;
                    run = SECOND ? (w > DBL_EPSILON) : (w > P.threshold);
                } else {
                    const int pa = A.gphase[ga], pb = A.gphase[gb];
                    entry = A.dg_mode[pa * NP + pb] == 1;  // else no Force entry for this pair
                    const double scale = A.gvr[ga] * A.gvr[gb];
                    cut = P.threshold * scale;
                    vab = A.dg_value[pa * NP + pb];
                    vba = A.dg_value[pb * NP + pa];
                    run = entry && (SECOND ? (w > 0.0) : (w > cut));
                }
                // own value the pass falls back to: raw or 0 (collect), tmp (distribute)
                if (entry) own = SECOND ? P.tmp[static_cast<int64_t>(p) * N + c] : (CURV ? 0.0 : vab);
            }
            double sum = 0.0, value = 0.0;
            int counted = 0;
            const unsigned long long pairs = __ballot(run);
            for (int t0 = 0; pairs != 0ull && t0 < P.noff; t0 += 64 * kAvgChunks) {
                NearLists L;
                near_lists<TV>(P, x, y, z, t0, L);
                double ow[kAvgChunks];
#pragma unroll
                for (int u = 0; u < kAvgChunks; ++u)
                    ow[u] = (CURV ? !SECOND : P.weights == 1) ? P.off_w[min(t0 + 64 * u + lane, P.noff - 1)] : 1.0;
                for (unsigned long long left = pairs; left != 0ull; left &= left - 1ull) {
                    const int q = __ffsll(static_cast<long long>(left)) - 1;
                    PairTerm T[kAvgChunks];
                    if (!pair_terms<TV>(A, L, c, static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(ga), q)),
                                        static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(gb), q)), src, T))
                        continue;
                    bool ok[kAvgChunks];
                    double wt[kAvgChunks], term[kAvgChunks];
#pragma unroll
                    for (int u = 0; u < kAvgChunks; ++u) {
                        if (CURV) {
                            const double v = T[u].fwd ? T[u].v : -T[u].v;
                            wt[u] = SECOND ? 0.0 : T[u].w * ow[u];
                            ok[u] = T[u].has && (SECOND ? T[u].w > P.threshold : wt[u] > DBL_EPSILON);
                            term[u] = SECOND ? v : wt[u] * v;
                        } else {
                            wt[u] = P.weights == 0 ? T[u].w : ow[u];
                            ok[u] = T[u].has && (SECOND ? (T[u].w > lane_value(cut, q)) : (T[u].w > 0.0));
                            if (SECOND) term[u] = wt[u] * (T[u].fwd ? T[u].v : -T[u].v);
                            else term[u] = wt[u] * (T[u].fwd ? lane_value(vab, q) : -lane_value(vba, q));
                        }
                    }
                    // value += weight * v and sum += weight in offset order
                    double acc = lane & 1 ? lane_value(value, q) : lane_value(sum, q);
                    const int m = ordered_add(s_terms[wave], ok, wt, term, acc);
                    const double s0 = lane_value(acc, 0), s1 = lane_value(acc, 1);
                    if (lane == q) {
                        sum = s0;
                        value = s1;
                        counted += m;
                    }
                }
            }
            // DistributeAverage's weight-0 branch (Seed grains) cannot occur: own entries are above the
            // finalize cutoff and no grain is a Seed
            if (entry) {
                double result = 0.0;  // a fresh entry's tmp / average
                if (run) {
                    if (CURV ? SECOND : P.weights == 2) result = counted != 0 ? value / static_cast<double>(counted) : own;
                    else result = sum > (CURV ? DBL_EPSILON : 0.0) ? value / sum : own;
                }
                (SECOND ? P.avg : P.tmp)[static_cast<int64_t>(p) * N + c] = result;
            }
        }
    }
}

// ---- interface regularization (FP64 state) -------------------------------------------------

constexpr int kRawCells = 256;     // most cells per block (one wavefront) of the raw pass
constexpr int kRawWaves = 8192;    // wavefronts that fill the chip: 1024 SIMDs x 8

// The curvature DoubleObstacle's regularization overload adds per pair of non-zero entries of a
// wide-interface cell (src/DoubleObstacle.cpp:702-763): loc_increment (the pair's increment before
// the mobility, over the neighbour-merged list) * Eta/Pi * scale * norm_1 / sqrt(phi_a phi_b) *
// (CurvatureFactor - RegularizationFactor). Only own entries are non-zero, so only interface cells
// (more than one own entry) hold such pairs. A group of lanes takes the cell (group_gather), its
// own pairs dealt to the lanes; energies per pair from the phase-pair table (GRAD false) or the
// orientation. Returns true when the cell needs more than CAP entries: nothing was written then.
template <bool GRAD, int G, int CAP>
__device__ __forceinline__ bool raw_cell(const CurvArgs& P, bool run, int64_t c, GroupMem<double, GRAD, CAP>& M,
                                         const uint16_t* pairs)
{
    const StepArgs& A = P.s;
    const int64_t N = A.ncells;
    const int l = static_cast<int>(threadIdx.x) & (G - 1), NP = A.nphases;
    const GroupList<double> L = group_gather<double, double, GRAD, G, CAP>(A, run, c, M);
    const bool work = run && !L.over && L.wide;
    const int ne = work ? L.ne : 0, n0 = work ? L.n0 : 0;
    if (l < CAP) {
        M.lap[l] = L.lap;
        M.phi[l] = L.phi;
        M.ph[l] = l < ne ? A.gphase[L.eid] : 0;
        M.vr[l] = l < ne ? A.gvr[L.eid] : 0.0;
        if (GRAD) { M.gr[GRAD ? l : 0][0] = L.gx; M.gr[GRAD ? l : 0][1] = L.gy; M.gr[GRAD ? l : 0][2] = L.gz; }
    }
    __syncthreads();
    double localn = 0.0;
    if (A.consider_nucleus) {
        for (int t = 0; t < ne; ++t) localn += M.vr[t];
    } else {
        localn = static_cast<double>(ne);
    }
    const double norm_1 = 1.0 / localn;
    const double Pf = A.prefactor;
    // InterfaceProperties energy of a pair (the lower list position first)
    for (int p = l; p < ne * (ne - 1) / 2; p += G) {
        const int a = pairs[p] & 255, b = pairs[p] >> 8;
        double en;
        if (GRAD) {
            double da[3], db[3];
            for (int d = 0; d < 3; ++d) { da[d] = M.gr[GRAD ? a : 0][d]; db[d] = M.gr[GRAD ? b : 0][d]; }
            en = ip_pair_energy<double>(A, M.ph[a] * NP + M.ph[b], M.eid[a], M.eid[b], M.phi[a], M.phi[b], da, db);
        } else {
            en = A.sigma[M.ph[a] * NP + M.ph[b]];
        }
        M.p.sig[a][b] = en;
        M.p.sig[b][a] = en;
    }
    __syncthreads();
    for (int p = l; p < n0 * (n0 - 1) / 2; p += G) {
        const int a = pairs[p] & 255, b = pairs[p] >> 8;
        const double scale = sqrt(M.vr[a] * M.vr[b]);
        const double cf = 0.5 * (1.0 + scale) * Pf;
        double d = M.p.sig[a][b] * ((M.lap[a] + cf * M.phi[a]) - (M.lap[b] + cf * M.phi[b]));
        for (int g = 0; g < ne; ++g) {
            if (g == a || g == b) continue;
            d += (M.p.sig[b][g] - M.p.sig[a][g]) * (M.lap[g] + cf * M.phi[g]);
            if (A.tj_model == 0) {
                if (A.tj_factor != 0.0 || scale < 1.0) {
                    const int pa = M.ph[a], pb = M.ph[b], pg = M.ph[g];
                    const double e3 = A.sigma[pa * NP + pb] + A.sigma[pb * NP + pg] + A.sigma[pa * NP + pg];
                    d += smax(A.tj_factor, (1.0 - scale)) * Pf * e3 * (M.phi[a] * M.phi[g] - M.phi[b] * M.phi[g]);
                }
            } else if (A.tj_model == 1) {
                d += A.tj_energy * Pf * (M.phi[a] * M.phi[g] - M.phi[b] * M.phi[g]);
            }
        }
        double kappa = d * P.prefactor2 * scale * norm_1 / sqrt(M.phi[a] * M.phi[b]);
        kappa *= P.factor;
        P.sphere.raw[static_cast<int64_t>(p) * N + c] = kappa;
    }
    __syncthreads();
    return run && L.over;
}

// A wavefront collects the interface cells of its 256 cells in LDS and takes them four at a time
// (longer lists, up to 16 merged entries, one at a time; more than that the step itself reports as
// an overflow). What bounds it is the instructions of the list walk; one thread per cell with
// register lists took 4.0 ms at 160^3 (256 VGPRs and spills, one wavefront per SIMD), now 1.23 ms.
template <bool GRAD>
__global__ __launch_bounds__(64) void curvature_raw_kernel(const CurvArgs P, int cells)
{
    constexpr int G = kGroupLanes, C = 64 / G;
    __shared__ GroupArena<double, GRAD> mem;
    __shared__ uint16_t pairs[kPairTable];
    __shared__ uint16_t s_list[kRawCells];
    const int lane = static_cast<int>(threadIdx.x);
    const int64_t base = static_cast<int64_t>(blockIdx.x) * cells;
    fill_pairs(pairs);
    int n = 0;
    for (int k = 0; k < cells; k += 64) {
        const int64_t c = base + k + lane;
        const bool in = k + lane < cells && c < P.s.ncells && ListCode<double>::count(P.s.cnt_in[c]) >= 2;
        const unsigned long long m = __ballot(in);
        if (in) s_list[n + __popcll(m & ((1ull << lane) - 1ull))] = static_cast<uint16_t>(k + lane);
        n += __popcll(m);
    }
    __syncthreads();
    for (int i0 = 0; i0 < n; i0 += C) {
        const int i = i0 + lane / G;
        const bool run = i < n;
        const bool big = raw_cell<GRAD, G, kGroupCap>(P, run, base + (run ? s_list[i] : 0), mem.cell[lane / G], pairs);
        unsigned long long todo = __ballot(big && (lane & (G - 1)) == 0);
        while (todo) {
            const int from = next_long(todo);
            (void)raw_cell<GRAD, kLongLanes, kWideSlots>(P, true, base + s_list[i0 + from / G], mem.longer[lane / kLongLanes], pairs);
        }
    }
}

// ---- both averagings on staged tiles

constexpr int kSphereBlock = kSphereCells;     // threads of a block

struct __align__(16) PairCell {
    double w, v;   // weight and value of the staged pair at a cell (absent: 0, 0)
};
static_assert(sizeof(PairCell) + sizeof(unsigned long long) + 1 == kSphereCellBytes, "LDS of a staged cell");

// Grain of entry t of cell c, `rec` holding its first four.
__device__ __forceinline__ uint32_t listed_grain(const StepArgs& A, unsigned long long rec, int64_t c, int t)
{
    return t < 4 ? static_cast<uint32_t>(rec >> (16 * t)) & 0xFFFFu : A.id_in[static_cast<int64_t>(t) * A.ncells + c];
}

// SECOND = false: CollectAverage into tmp; true: DistributeAverage into avg, of the driving force or
// (CURV) of the curvature: the sums of sphere_wave_kernel, on tiles.
//
// A block stages the lists' grains of its tile plus the sphere's reach in LDS, and then takes the
// pairs of grains its cells hold one after another (ascending): the pair's weight and value at every
// staged cell go to LDS (0 where it is absent: such a term never counts), and every lane sums the
// sphere around one of the tile's cells that hold the pair, x outer, z inner as the reference does,
// from LDS at fixed distances. Values are staged in the orientation (lower grain, higher grain); a
// sum in the other orientation is its exact negative. So a pair is looked up once per staged cell
// and not once per cell and offset, and a wavefront holds 64 cells' sums instead of one. What
// bounds it is the chain of the sums (an LDS read and about 11 instructions per offset) of the
// pairs that only a few of the tile's cells hold. Collect / Distribute of the curvature, 93
// offsets, 160^3: 7.66 / 5.70 ms when a wavefront took a cell, 1.68 / 1.54 ms on tiles. The driving
// force with 485 offsets, 96^3: 0.31 / 1.32 ms a wavefront per cell, 0.61 / 2.70 ms on tiles: so
// tiles are staged up to kSphereOffsets offsets.
template <typename TV, bool CURV, bool SECOND>
__global__ __launch_bounds__(kSphereBlock) void sphere_tile_kernel(const SphereArgs P)
{
    extern __shared__ __align__(16) unsigned char s_dyn[];
    __shared__ uint32_t s_item[kSphereBlock];
    __shared__ uint32_t s_key, s_items;
    const StepArgs& A = P.s;
    const int64_t N = A.ncells;
    const int NP = A.nphases;
    const int tid = static_cast<int>(threadIdx.x);
    const int HY = P.ty + 2 * P.ry, HZ = P.tz + 2 * P.rz, H = (P.tx + 2 * P.rx) * HY * HZ;
    PairCell* s_pair = reinterpret_cast<PairCell*>(s_dyn);
    unsigned long long* s_rec = reinterpret_cast<unsigned long long*>(s_pair + H);
    uint32_t* s_row = reinterpret_cast<uint32_t*>(s_rec + H);   // first cell of a staged row of z
    uint8_t* s_code = reinterpret_cast<uint8_t*>(s_row + H / HZ);
    const unsigned b = A.xcd_order ? xcd_block(blockIdx.x, gridDim.x) : blockIdx.x;
    const unsigned ntz = static_cast<unsigned>((A.nz + P.tz - 1) / P.tz), nty = static_cast<unsigned>((A.ny + P.ty - 1) / P.ty);
    const int z0 = static_cast<int>(b % ntz) * P.tz, y0 = static_cast<int>((b / ntz) % nty) * P.ty,
              x0 = static_cast<int>(b / (ntz * nty)) * P.tx;
    for (int r = tid; r < H / HZ; r += kSphereBlock) {
        const int x = (x0 - P.rx + r / HY + A.nx) % A.nx, y = (y0 - P.ry + r % HY + A.ny) % A.ny;
        s_row[r] = static_cast<uint32_t>((x * A.ny + y) * A.nz);
    }
    __syncthreads();
    // a thread stages the cells of one z in every step-th row
    const int step = kSphereBlock / HZ, row0 = tid / HZ < step ? tid / HZ : H / HZ, hz = tid % HZ;
    const uint32_t zg = static_cast<uint32_t>((z0 - P.rz + hz + A.nz) % A.nz);
    for (int r = row0; r < H / HZ; r += step) {
        const int64_t c = s_row[r] + zg;
        const uint8_t code = A.cnt_in[c];
        const int n = ListCode<TV>::count(code);
        unsigned long long rec = 0ull;
#pragma unroll
        for (int s = 0; s < 4; ++s)
            if (s < n) rec |= static_cast<unsigned long long>(A.id_in[static_cast<int64_t>(s) * N + c]) << (16 * s);
        s_rec[r * HZ + hz] = rec;
        s_code[r * HZ + hz] = code;
    }
    // the thread's own cell
    const int lx = tid / (P.ty * P.tz), ly = (tid / P.tz) % P.ty, lz = tid % P.tz;
    const bool own = lx < P.tx && x0 + lx < A.nx && y0 + ly < A.ny && z0 + lz < A.nz;
    const int hown = own ? ((lx + P.rx) * HY + ly + P.ry) * HZ + lz + P.rz : 0;
    const int64_t cown = own ? (static_cast<int64_t>(x0 + lx) * A.ny + y0 + ly) * A.nz + z0 + lz : 0;
    __syncthreads();
    const int nown = own ? ListCode<TV>::count(s_code[hown]) : 0;
    const unsigned long long rown = s_rec[hown];
    // key of the own pair (d, e): its grains, lower first, ~0 for a driving force's pair of phases
    // without one (no Force entry); those of the first four entries are kept
    auto own_key = [&](int d, int e) -> uint32_t {
        const uint32_t gd = listed_grain(A, rown, cown, d), ge = listed_grain(A, rown, cown, e);
        if (!CURV && A.dg_mode[A.gphase[gd] * NP + A.gphase[ge]] != 1) return ~0u;
        return min(gd, ge) << 16 | max(gd, ge);
    };
    uint32_t key4[6];
#pragma unroll
    for (int e = 1; e < 4; ++e)
#pragma unroll
        for (int d = 0; d < e; ++d) key4[pair_plane(d, e)] = e < nown ? own_key(d, e) : ~0u;
    uint32_t last = 0u;  // keys (lower grain << 16 | higher grain) are not 0
    while (true) {
        if (tid == 0) {
            s_key = ~0u;
            s_items = 0u;
        }
        __syncthreads();
        uint32_t next = ~0u;
#pragma unroll
        for (int p = 0; p < 6; ++p) next = key4[p] > last ? min(next, key4[p]) : next;
        for (int e = 4; e < nown; ++e)
            for (int d = 0; d < e; ++d) {
                const uint32_t k = own_key(d, e);
                next = k > last ? min(next, k) : next;
            }
#pragma unroll
        for (int k = 32; k >= 1; k >>= 1) next = min(next, static_cast<uint32_t>(__shfl_xor(static_cast<int>(next), k)));
        if ((tid & 63) == 0 && next != ~0u) atomicMin(&s_key, next);
        __syncthreads();
        const uint32_t key = s_key;
        if (key == ~0u) break;
        last = key;
        const uint32_t glo = key >> 16, ghi = key & 0xFFFFu;
        const int plo = A.gphase[glo], phi = A.gphase[ghi];
        double cut = P.threshold;
        if (!CURV) cut *= A.gvr[glo] * A.gvr[ghi];
        // the tile's cells that hold the pair; those whose weight is too small keep a fresh entry's 0
        int plane = -1, ia = 0, ib = 0;
#pragma unroll
        for (int e = 1; e < 4; ++e)
#pragma unroll
            for (int d = 0; d < e; ++d)
                if (key4[pair_plane(d, e)] == key) { plane = pair_plane(d, e); ia = d; ib = e; }
        for (int e = 4; e < nown && plane < 0; ++e)
            for (int d = 0; d < e; ++d)
                if (own_key(d, e) == key) { plane = pair_plane(d, e); ia = d; ib = e; }
        if (plane >= 0) {
            const uint8_t code = s_code[hown];
            const double w = sqrt(entry_value<TV>(A, cown, code, ia) * entry_value<TV>(A, cown, code, ib));
            const bool back = listed_grain(A, rown, cown, ia) != glo;
            if (CURV ? (SECOND ? w > DBL_EPSILON : w > P.threshold) : (SECOND ? w > 0.0 : w > cut))
                s_item[atomicAdd(&s_items, 1u)] = static_cast<uint32_t>(tid) | static_cast<uint32_t>(plane) << 16 | (back ? 1u << 31 : 0u);
            else
                (SECOND ? P.avg : P.tmp)[static_cast<int64_t>(plane) * N + cown] = 0.0;
        }
        __syncthreads();
        const uint32_t items = s_items;
        if (items) {
            const double* __restrict__ src = SECOND ? P.tmp : P.raw;
            const double fwd = CURV ? 0.0 : A.dg_value[plo * NP + phi], rev = CURV ? 0.0 : -A.dg_value[phi * NP + plo];
            for (int r = row0; r < H / HZ; r += step) {
                const int h = r * HZ + hz;
                const uint8_t code = s_code[h];
                const int n = ListCode<TV>::count(code);
                const unsigned long long rec = s_rec[h];
                PairCell p{0.0, 0.0};
                if (n > 1) {
                    int ja = -1, jb = -1;
#pragma unroll
                    for (int s = 0; s < 4; ++s) {
                        const uint32_t g = static_cast<uint32_t>(rec >> (16 * s)) & 0xFFFFu;
                        ja = s < n && g == glo ? s : ja;
                        jb = s < n && g == ghi ? s : jb;
                    }
                    const int64_t c = s_row[r] + zg;
                    if (n > 4 && (ja < 0 || jb < 0)) {
                        for (int s = 4; s < n; ++s) {
                            const uint32_t g = A.id_in[static_cast<int64_t>(s) * N + c];
                            ja = g == glo ? s : ja;
                            jb = g == ghi ? s : jb;
                        }
                    }
                    if (ja >= 0 && jb >= 0) {
                        if (SECOND || CURV) p.v = src[static_cast<int64_t>(pair_plane(min(ja, jb), max(ja, jb))) * N + c];
                        p.w = sqrt(entry_value<TV>(A, c, code, ja) * entry_value<TV>(A, c, code, jb));
                        if (SECOND || CURV) p.v = ja < jb ? p.v : -p.v;
                        else p.v = ja < jb ? fwd : rev;
                    }
                }
                s_pair[h] = p;
            }
        }
        __syncthreads();
        for (uint32_t i = static_cast<uint32_t>(tid); i < items; i += kSphereBlock) {
            const int t0 = static_cast<int>(s_item[i] & 0xFFFFu);
            const int plane = static_cast<int>((s_item[i] >> 16) & 0x7FFFu);
            const bool back = (s_item[i] >> 31) != 0u;
            const int cx = t0 / (P.ty * P.tz), cy = (t0 / P.tz) % P.ty, cz = t0 % P.tz;
            const int64_t here = static_cast<int64_t>(plane) * N + (static_cast<int64_t>(x0 + cx) * A.ny + y0 + cy) * A.nz + z0 + cz;
            const PairCell* at = s_pair + ((cx + P.rx) * HY + cy + P.ry) * HZ + cz + P.rz;
            double value = 0.0, sum = 0.0;
            int counter = 0;
#pragma unroll 8
            for (int t = 0; t < P.noff; ++t) {
                const PairCell p = at[P.tile_off[t]];
                // terms that do not count add +0, which leaves the sums as they are (never -0)
                if (CURV && SECOND) {
                    const bool ok = p.w > P.threshold;
                    value += ok ? p.v : 0.0;
                    counter += ok ? 1 : 0;
                } else {
                    const double wt = CURV ? p.w * P.off_w[t] : (P.weights == 0 ? p.w : (P.weights == 1 ? P.off_w[t] : 1.0));
                    const bool ok = CURV ? wt > DBL_EPSILON : (SECOND ? p.w > cut : p.w > 0.0);
                    value += ok ? wt * p.v : 0.0;
                    sum += ok ? wt : 0.0;
                }
            }
            if (back) value = -value;
            double result;
            if (CURV) {
                if (SECOND) result = counter != 0 ? value / static_cast<double>(counter) : P.tmp[here];
                else result = sum > DBL_EPSILON ? value / sum : 0.0;
            } else {
                // COUNTER weights are 1: their sum is the count
                if (sum > 0.0) result = value / sum;
                else result = SECOND ? P.tmp[here] : A.dg_value[back ? phi * NP + plo : plo * NP + phi];
            }
            (SECOND ? P.avg : P.tmp)[here] = result;
        }
    }
}

}  // namespace

// LDS of a staged tile: pair field, grains and count byte per cell, first cell per row.
static size_t sphere_lds(const SphereArgs& a)
{
    const size_t rows = static_cast<size_t>(a.tx + 2 * a.rx) * (a.ty + 2 * a.ry);
    return rows * ((a.tz + 2 * a.rz) * kSphereCellBytes + sizeof(uint32_t));
}

template <typename TV, bool CURV>
static void launch_sphere(const SphereArgs& a, hipStream_t s)
{
    if (a.tx) {
        const size_t lds = sphere_lds(a);
        const int64_t blocks = static_cast<int64_t>((a.s.nx + a.tx - 1) / a.tx) * ((a.s.ny + a.ty - 1) / a.ty) * ((a.s.nz + a.tz - 1) / a.tz);
        const dim3 grid(static_cast<unsigned>(blocks));
        hipLaunchKernelGGL((sphere_tile_kernel<TV, CURV, false>), grid, dim3(kSphereBlock), lds, s, a);
        hipLaunchKernelGGL((sphere_tile_kernel<TV, CURV, true>), grid, dim3(kSphereBlock), lds, s, a);
    } else {
        const dim3 grid(static_cast<unsigned>((a.s.ncells + kAvgCells - 1) / kAvgCells));
        hipLaunchKernelGGL((sphere_wave_kernel<TV, false, CURV>), grid, dim3(kAvgBlock), 0, s, a);
        hipLaunchKernelGGL((sphere_wave_kernel<TV, true, CURV>), grid, dim3(kAvgBlock), 0, s, a);
    }
}

int sphere_lds_limit()
{
    // more than 64 KiB of dynamic LDS has to be asked for, once per kernel
    const void* kernels[] = {reinterpret_cast<const void*>(&sphere_tile_kernel<double, true, false>),
                             reinterpret_cast<const void*>(&sphere_tile_kernel<double, true, true>),
                             reinterpret_cast<const void*>(&sphere_tile_kernel<double, false, false>),
                             reinterpret_cast<const void*>(&sphere_tile_kernel<double, false, true>),
                             reinterpret_cast<const void*>(&sphere_tile_kernel<float, false, false>),
                             reinterpret_cast<const void*>(&sphere_tile_kernel<float, false, true>)};
    for (const void* k : kernels) {
        const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, kSphereLds);
        if (e != hipSuccess) return static_cast<int>(e);
    }
    return 0;
}

int launch_curvature(const CurvArgs& a, void* stream)
{
    hipStream_t s = static_cast<hipStream_t>(stream);
    // a wavefront takes 256 cells, whose interface cells fill its groups of lanes; fewer on a grid that
    // would not give every SIMD eight wavefronts: 20 regularized steps 64^2 6.0 -> 2.7 ms, 512^2 6.5 -> 5.4 ms,
    // four at 96^3 8.6 -> 8.2 ms
    int cells = kRawCells;
    while (cells > 64 / kGroupLanes && a.s.ncells / cells < kRawWaves) cells /= 2;
    const dim3 raw_grid(static_cast<unsigned>((a.s.ncells + cells - 1) / cells));
    if (a.grad) hipLaunchKernelGGL((curvature_raw_kernel<true>), raw_grid, dim3(64), 0, s, a, cells);
    else hipLaunchKernelGGL((curvature_raw_kernel<false>), raw_grid, dim3(64), 0, s, a, cells);
    launch_sphere<double, true>(a.sphere, s);
    return static_cast<int>(hipGetLastError());
}

int launch_dg_average(const SphereArgs& a, bool fp32, void* stream)
{
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (fp32) launch_sphere<float, false>(a, s);
    else launch_sphere<double, false>(a, s);
    return static_cast<int>(hipGetLastError());
}

}  // namespace mpf
