// Teams of different sizes (plan_resident in csrc/resident_plan.hip): every
// system is in one list and fits its team, every work-group has one place,
// a team sits on one XCD, the teams' slots do not overlap, and the plan is
// never longer than the best one with teams of one size.
#include <cstdio>
#include <cstdlib>
#include <random>
#include <set>

#include "../hornofusion-full3d_amd/csrc/resident_plan.hip"

#define CHECK(c, ...)                                \
    do {                                             \
        if (!(c)) {                                  \
            std::printf("line %d: ", __LINE__);      \
            std::printf(__VA_ARGS__);                \
            std::printf("\n");                       \
            std::exit(1);                            \
        }                                            \
    } while (0)

namespace eafp {
int device_cus() { return RES_CUS; }
}

using namespace eafp;

static int slots(int nz, int rows) { return (int)(((long)nz * rows + 511) / 512); }
static size_t lds(int nz, int, int lrows, int hrows) { return 4096 + ((size_t)lrows * 8 + (size_t)hrows * 16) * nz; }
static int pitch(int nz) { return nz; }
static const ResLimits kLim = {8, slots, lds, {1.2f, 3.4f, 3.4f, 3.4f, 3.4f, 4.1f, 4.8f, 5.1f, 7.3f}, 0.5f};

static long g_mixed = 0, g_plans = 0;

static float uniform_est(const std::vector<SysGeom>& g) {
    std::vector<long> xoff(g.size(), 0);
    const Priced c = price(g, kLim, xoff);
    float best = 0.f;
    for (int lt = 0; lt < LT; ++lt) {
        int n[LT] = {};
        n[lt] = std::min((int)g.size(), RES_CUS >> lt);
        const float t = assign(c, kLim, n, nullptr, nullptr);
        if (t > 0.f && (best == 0.f || t < best)) best = t;
    }
    return best;
}

static void check(const std::vector<SysGeom>& g) {
    const ResPlan p = plan_resident(g, kLim, pitch);
    const float est = uniform_est(g);
    CHECK(p.ok == (est > 0.f), "plan %d, uniform %f", (int)p.ok, est);
    if (!p.ok) return;
    ++g_plans;
    CHECK(p.est_us <= est * 1.0001f && (p.T || p.est_us <= 0.9501f * est), "%f against %f", p.est_us, est);
    CHECK((int)p.team_begin.size() == p.nteam + 1 && p.team_begin[0] == 0 && p.team_begin[p.nteam] == (int)g.size(), "lists");
    std::set<int> seen;
    for (int t = 0; t < p.nteam; ++t)
        for (int i = p.team_begin[t]; i < p.team_begin[t + 1]; ++i) {
            const ResItem& I = p.items[i];
            const int T = p.T ? p.T : p.teams[t].T;
            int pr, pth, rows, lrows;
            CHECK(seen.insert(I.sys).second && I.nr == g[I.sys].nr && I.nz == g[I.sys].nz, "system %d", I.sys);
            res_grid(I.nr, I.nth, T, pr, pth);
            res_extent(I.nr, I.nth, pr, pth, rows, lrows);
            CHECK(pr == I.pr && pth == I.pth && pr * pth <= T, "grid of system %d", I.sys);
            CHECK(slots(I.nz, rows) <= p.slots && p.slots <= 8 && lds(I.nz, rows, lrows, lrows - rows) <= p.lds &&
                      p.lds <= (size_t)RES_LDS, "system %d does not fit", I.sys);
        }
    CHECK(seen.size() == g.size() && p.max_items >= 1, "systems");
    if (p.T) return;
    ++g_mixed;
    CHECK((int)p.teams.size() == p.nteam && (int)p.member.size() >= p.blocks && p.blocks <= RES_CUS, "tables");
    std::set<std::pair<int, int>> places;
    std::vector<int> xcd(p.nteam, -1);
    for (int b = 0; b < (int)p.member.size(); ++b) {
        const int t = p.member[b].x, m = p.member[b].y;
        if (t < 0) continue;
        CHECK(b < p.blocks && t < p.nteam && m >= 0 && m < p.teams[t].T, "work-group %d", b);
        CHECK(places.insert({t, m}).second, "a place twice");
        CHECK(xcd[t] < 0 || xcd[t] == b % NXCD, "team %d over several XCDs", t);
        xcd[t] = b % NXCD;
    }
    int total = 0, slot = 0;
    for (int t = 0; t < p.nteam; ++t) {
        const int T = p.teams[t].T;
        CHECK(p.teams[t].slot0 == slot && T >= 1 && T <= 32, "slots of team %d", t);
        slot += 2 * T;
        const bool used = p.team_begin[t + 1] > p.team_begin[t];
        CHECK((xcd[t] >= 0) == used, "team %d has items but no place", t);
        total += used ? T : 0;
    }
    CHECK(total == p.members && (int)places.size() == total && slot == p.nslot, "members");
}

int main() {
    std::mt19937 rng(5);
    for (int S : {1, 2, 3, 5, 8, 16, 31, 32, 33, 64, 96, 200, 400})
        for (int rep = 0; rep < 12; ++rep) {
            std::vector<SysGeom> g(S);
            long off = 0;
            const int hi = rep % 3 == 0 ? 12 : rep % 3 == 1 ? 40 : 64;
            for (auto& s : g) {
                s = SysGeom{};
                s.nr = 1 + (int)(rng() % hi);
                s.nth = 1 + (int)(rng() % (hi + 20));
                s.nz = 1 + (int)(rng() % hi);
                s.n = s.nr * s.nth * s.nz;
                s.off = off;
                off += s.n;
            }
            check(g);
        }
    CHECK(g_mixed > 20, "%ld of %ld plans mix", g_mixed, g_plans);
    std::printf("ok %ld %ld\n", g_plans, g_mixed);
    return 0;
}
