// Drives group_gather (openphase_amd/csrc/mpf_group.h) on the host's lanes (lane_runtime.h): random
// states with lists of every length, each cell's merged list and Laplacians by groups of 16 lanes and by
// a wavefront against a plain walk over the box. Prints "gather ok" and the forms it saw.
#include "mpf_group.h"

#include <random>
#include <algorithm>

using namespace mpf;

namespace {

int fails = 0;

void check(bool ok, const char* what, long c)
{
    if (ok) return;
    ++fails;
    std::fprintf(stderr, "cell %ld: %s\n", c, what);
}

// A state of lists of up to `longest` of `pool` grains; FP32: the implicit (largest) entry comes last.
template <typename TV> struct State {
    StepArgs A{};
    std::vector<uint8_t> cnt;
    std::vector<uint16_t> id;
    std::vector<TV> val;
    State(int nx, int ny, int nz, int pool, int longest, unsigned seed)
    {
        A.nx = nx ? nx : 1; A.ny = ny ? ny : 1; A.nz = nz ? nz : 1;
        A.dnx = nx > 0; A.dny = ny > 0; A.dnz = nz > 0;
        A.ncells = static_cast<int64_t>(A.nx) * A.ny * A.nz;
        A.slots = kMaxSlots;
        for (int i = 0; i < 4; ++i) { A.wl[i] = 0.7 - 0.31 * i; A.wg[i] = 0.2 + 0.11 * i; }
        const size_t N = static_cast<size_t>(A.ncells);
        cnt.resize(N);
        id.resize(N * kMaxSlots);
        val.resize(N * kMaxSlots);
        std::mt19937 rng(seed);
        std::vector<int> order(pool);
        for (size_t c = 0; c < N; ++c) {
            const int n = rng() % 3 == 0 ? 1 : 1 + static_cast<int>(rng() % longest);
            for (int i = 0; i < pool; ++i) order[i] = i;
            for (int i = 0; i < n; ++i) std::swap(order[i], order[i + rng() % (pool - i)]);
            cnt[c] = static_cast<uint8_t>(ListCode<TV>::kImplicit ? n | ((n - 1) << 4) : n);
            for (int q = 0; q < n; ++q) {
                id[q * N + c] = static_cast<uint16_t>(order[q]);
                // some entries hold 0: those are not merged
                val[q * N + c] = n == 1 ? TV(1) : (rng() % 8 == 0 ? TV(0) : TV((1 + q + rng() % 4) / 256.0));
            }
            // (a lone implicit entry stores nothing)
            if (ListCode<TV>::kImplicit && n == 1) val[c] = TV(-7);
        }
        A.cnt_in = cnt.data();
        A.id_in = id.data();
        A.val_in = val.data();
    }
};

template <typename TV, bool GRAD, int G, int CAP> void compare(const State<TV>& S, int& held, int& longer)
{
    const StepArgs& A = S.A;
    const int64_t N = A.ncells;
    constexpr int C = 64 / G;
    static GroupMem<TV, GRAD, CAP> mem[C];
    GroupList<TV> got[64];
    for (int64_t base = 0; base < N; base += C) {
        lanes::run([&] {
            const int64_t c = base + lanes::here / G;
            got[lanes::here] = group_gather<TV, TV, GRAD, G, CAP>(A, c < N, c < N ? c : 0, mem[lanes::here / G]);
        });
        for (int g = 0; g < C && base + g < N; ++g) {
            // ---- the plain walk: own entries, then grains new to the box, in stencil order
            const int64_t c = base + g;
            std::vector<uint32_t> list;
            std::vector<TV> lap, gx;
            int own = ListCode<TV>::count(S.cnt[c]), most = 0;
            bool wide = false;
            for (int q = 0; q < own; ++q) list.push_back(S.id[q * N + c]);
            for (int pass = 0; pass < 2; ++pass) {
                lap.assign(list.size(), TV(0));
                gx.assign(list.size(), TV(0));
                for (int k = 0; k < 27; ++k) {
                    const int ii = k / 9 - 1, jj = (k / 3) % 3 - 1, kk = k % 3 - 1, nz = (ii != 0) + (jj != 0) + (kk != 0);
                    if ((ii && !A.dnx) || (jj && !A.dny) || (kk && !A.dnz)) continue;
                    const int64_t x = (c / (A.ny * A.nz) + ii + A.nx) % A.nx, y = (c / A.nz + jj + A.ny) % A.ny, z = (c % A.nz + kk + A.nz) % A.nz;
                    const int64_t nb = (x * A.ny + y) * A.nz + z;
                    const int n = ListCode<TV>::count(S.cnt[nb]);
                    most = std::max(most, n);
                    wide = wide || n > 1;
                    for (int q = 0; q < n; ++q) {
                        const TV v = ListCode<TV>::kImplicit && n == 1 ? TV(1) : S.val[q * N + nb];
                        if (v == TV(0)) continue;
                        size_t t = 0;
                        while (t < list.size() && list[t] != S.id[q * N + nb]) ++t;
                        if (t == list.size()) { list.push_back(S.id[q * N + nb]); lap.push_back(TV(0)); gx.push_back(TV(0)); }
                        lap[t] += static_cast<TV>(A.wl[nz]) * v;
                        if (ii) gx[t] += (ii < 0 ? -1 : 1) * static_cast<TV>(A.wg[nz]) * v;
                    }
                }
            }
            const GroupList<TV>* L = got + g * G;
            const bool over = wide ? static_cast<int>(list.size()) > CAP || most > CAP : own > CAP;
            check(L->over == over, "over", c);
            check(L->wide == wide && L->n0 == own, "own list", c);
            if (over || !wide) { longer += over; continue; }
            ++held;
            check(L->ne == static_cast<int>(list.size()), "merged length", c);
            double others = 0.0;
            const int imp = ListCode<TV>::implicit(S.cnt[c]);
            for (int q = 0; q < own; ++q)
                if (q != imp) others += static_cast<double>(S.val[q * N + c]);
            for (size_t t = 0; t < list.size(); ++t) {
                const double phi = static_cast<int>(t) >= own ? 0.0 : (static_cast<int>(t) == imp ? 1.0 - others : static_cast<double>(S.val[t * N + c]));
                check(L[t].eid == list[t], "grain", c);
                check(L[t].phi == phi, "value", c);
                check(L[t].lap == lap[t] && (!GRAD || L[t].gx == gx[t]), "Laplacian or gradient", c);
            }
        }
    }
}

template <typename TV, bool GRAD> void states()
{
    int held = 0, longer = 0, held16 = 0, longer16 = 0;
    const int sizes[][3] = {{9, 7, 0}, {6, 0, 5}, {0, 0, 11}, {4, 5, 3}};
    for (const auto& n : sizes)
        for (int longest : {2, 5, 9, 14}) {
            const State<TV> S(n[0], n[1], n[2], longest < 9 ? longest + 2 : 18, longest, 7u * n[0] + longest);
            compare<TV, GRAD, kGroupLanes, kGroupCap>(S, held, longer);
            compare<TV, GRAD, kLongLanes, kWideSlots>(S, held16, longer16);
        }
    std::printf("%d bytes: 16 lanes %d held, %d longer; 64 lanes %d held, %d longer\n", static_cast<int>(sizeof(TV)), held, longer,
                held16, longer16);
    if (!held || !longer || !held16 || !longer16) ++fails;
}

}  // namespace

int main()
{
    states<double, true>();
    states<float, false>();
    if (fails) return 1;
    std::puts("gather ok");
    return 0;
}
