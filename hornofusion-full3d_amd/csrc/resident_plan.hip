// resident_plan.hip -- host side of the resident solvers (resident_plan.hpp).
#include <algorithm>
#include <condition_variable>
#include <mutex>

#include "resident_plan.hpp"

namespace eafp {

namespace {
constexpr int MAX_DEV = 64;
std::mutex g_res_mu;
std::condition_variable g_res_cv;
int g_res_used[MAX_DEV];
unsigned long g_res_next[MAX_DEV], g_res_serving[MAX_DEV];
}  // namespace

ResidentGate::ResidentGate(int blocks) : dev_(0), n_(blocks) {
    (void)hipGetDevice(&dev_);
    if (dev_ < 0 || dev_ >= MAX_DEV) dev_ = 0;
    std::unique_lock<std::mutex> lk(g_res_mu);
    const unsigned long mine = g_res_next[dev_]++;   // first come, first served
    g_res_cv.wait(lk, [&] { return g_res_serving[dev_] == mine && g_res_used[dev_] + n_ <= RES_CUS; });
    g_res_used[dev_] += n_;
    ++g_res_serving[dev_];
    lk.unlock();
    g_res_cv.notify_all();
}

ResidentGate::~ResidentGate() {
    {
        std::lock_guard<std::mutex> lk(g_res_mu);
        g_res_used[dev_] -= n_;
    }
    g_res_cv.notify_all();
}

namespace {

constexpr int LT = 9;                  // team sizes 1, 2, 4 .. 256
constexpr int LT_MIXED = 6;            // and those that mixed teams take: a team on one XCD
constexpr int MIXED_SYS = 512;         // systems, at most, for mixed teams

// The systems, largest first, and what each takes with teams of each size.
struct Priced {
    std::vector<int> order;
    std::vector<int> u[LT];            // slots per thread (0: does not fit)
    std::vector<size_t> lds[LT];
    std::vector<ResItem> item[LT];
};

Priced price(const std::vector<SysGeom>& g, const ResLimits& lim, const std::vector<long>& xoff) {
    const int S = (int)g.size();
    Priced c;
    c.order.resize(S);
    for (int s = 0; s < S; ++s) c.order[s] = s;
    std::stable_sort(c.order.begin(), c.order.end(), [&](int a, int b) { return g[a].n > g[b].n; });
    for (int lt = 0; lt < LT; ++lt) {
        c.u[lt].assign(S, 0);
        c.lds[lt].assign(S, 0);
        c.item[lt].assign(S, ResItem{});
        for (int s = 0; s < S; ++s) {
            const SysGeom& G = g[s];
            ResItem& I = c.item[lt][s];
            I.sys = s;
            I.nr = G.nr;
            I.nth = G.nth;
            I.nz = G.nz;
            I.off = G.off;
            I.xoff = xoff[s];
            res_grid(G.nr, G.nth, 1 << lt, I.pr, I.pth);
            int rows, lrows;
            res_extent(G.nr, G.nth, I.pr, I.pth, rows, lrows);
            const int u = lim.slots(G.nz, rows);
            c.lds[lt][s] = lim.lds(G.nz, rows, lrows, lrows - rows);
            if (u >= 1 && u <= lim.max_slots && c.lds[lt][s] <= (size_t)RES_LDS) c.u[lt][s] = u;
        }
    }
    return c;
}

// count[lt] teams of size 1 << lt, largest first: systems go to the teams
// largest first, each to the team that is done with it soonest.  Returns the
// longest list's time (0: a system fits none); the lists, where asked for.
float assign(const Priced& c, const ResLimits& lim, const int (&count)[LT], std::vector<std::vector<ResItem>>* lists,
             std::vector<int>* size) {
    std::vector<std::pair<float, int>> heap[LT];      // the teams of a size by (time so far, team)
    int nteam = 0;
    for (int lt = LT - 1; lt >= 0; --lt)
        for (int q = 0; q < count[lt]; ++q) {
            heap[lt].push_back({0.f, nteam++});
            if (size) size->push_back(1 << lt);
        }
    const auto later = [](const std::pair<float, int>& x, const std::pair<float, int>& y) { return x > y; };
    for (auto& h : heap) std::make_heap(h.begin(), h.end(), later);
    if (lists) lists->resize(nteam);
    float longest = 0.f;
    for (int s : c.order) {
        int best = -1;
        float t_best = 0.f;
        for (int lt = 0; lt < LT; ++lt) {
            if (heap[lt].empty() || !c.u[lt][s]) continue;
            const float t = heap[lt].front().first + lim.sync_us[lt] + lim.slot_us * (float)c.u[lt][s];
            if (best < 0 || t < t_best) {
                best = lt;
                t_best = t;
            }
        }
        if (best < 0) return 0.f;
        std::pop_heap(heap[best].begin(), heap[best].end(), later);
        heap[best].back().first = t_best;
        if (lists) (*lists)[heap[best].back().second].push_back(c.item[best][s]);
        std::push_heap(heap[best].begin(), heap[best].end(), later);
        longest = std::max(longest, t_best);
    }
    return longest;
}

}  // namespace

// Every power of two T is priced: a team's iteration is its sums (sync_us)
// and its slots, a launch runs as many teams as fit the CUs, and the longest
// team list sets the time.  Then teams of different sizes, each on one XCD:
// from the sizes up to the best one's, two teams are made one, or one two,
// as long as that shortens the longest list.  One large system else sets the
// size for all, and in a large team the sums outlast the cells: 32 uneven
// systems of 22 to 112 thousand cells in FP64 took 19.2 ms in eight teams of 32
// and take 15.1, 96 of them mixed 39.8 and 32.4.
ResPlan plan_resident(const std::vector<SysGeom>& g, const ResLimits& lim, int (*xpitch)(int nz)) {
    ResPlan p;
    if (device_cus() < RES_CUS) return p;
    const int S = (int)g.size();
    std::vector<long> xoff(S);
    for (int s = 0; s < S; ++s) {
        xoff[s] = p.xlen;
        p.xlen += ((long)g[s].nr * g[s].nth * xpitch(g[s].nz) + 31) / 32 * 32;
    }
    const Priced c = price(g, lim, xoff);
    int count[LT] = {}, uniform = -1;
    for (int lt = 0; lt < LT; ++lt) {
        int n[LT] = {};
        n[lt] = std::min(S, RES_CUS >> lt);
        const float t = assign(c, lim, n, nullptr, nullptr);
        if (t > 0.f && (uniform < 0 || t < p.est_us)) {
            uniform = lt;
            p.est_us = t;
        }
    }
    if (uniform < 0) return ResPlan{};
    count[uniform] = std::min(S, RES_CUS >> uniform);
    if (S > 1 && S <= MIXED_SYS) {
        const float gain = 0.95f;      // what the tables' look-up and the model's error are worth
        float best = gain * p.est_us;
        for (int lt = 0; lt <= std::min(uniform, LT_MIXED - 1); ++lt) {
            // teams of this size, and one of the smallest that holds the systems that do not fit it
            int n[LT] = {}, need = lt;
            for (int s = 0; s < S; ++s)
                while (need < LT_MIXED && !c.u[need][s]) ++need;
            if (need >= LT_MIXED) continue;
            n[need] = 1;
            n[lt] += (RES_CUS - (1 << need)) >> lt;
            float t = assign(c, lim, n, nullptr, nullptr);
            for (bool moved = true; moved;) {
                moved = false;
                int keep[LT];
                std::copy(n, n + LT, keep);
                for (int q = 0; q + 1 < LT_MIXED; ++q)
                    for (int up = 0; up < 2; ++up) {
                        int m[LT];
                        std::copy(n, n + LT, m);
                        m[q] += up ? -2 : 2;
                        m[q + 1] += up ? 1 : -1;
                        if (m[q] < 0 || m[q + 1] < 0) continue;
                        const float v = assign(c, lim, m, nullptr, nullptr);
                        if (v > 0.f && v < 0.999f * t) {
                            t = v;
                            std::copy(m, m + LT, keep);
                            moved = true;
                        }
                    }
                std::copy(keep, keep + LT, n);
            }
            if (t > 0.f && t < best) {
                best = p.est_us = t;
                std::copy(n, n + LT, count);
                uniform = -1;
            }
        }
    }
    std::vector<std::vector<ResItem>> lists;
    std::vector<int> size;
    p.est_us = assign(c, lim, count, &lists, &size);
    p.ok = true;
    p.nsys = S;
    p.T = uniform < 0 ? 0 : 1 << uniform;
    p.nteam = (int)lists.size();
    for (int t = 0; t < p.nteam; ++t) {
        p.team_begin.push_back((int)p.items.size());
        p.items.insert(p.items.end(), lists[t].begin(), lists[t].end());
        p.max_items = std::max(p.max_items, (int)lists[t].size());
        int lt = 0;
        while (1 << lt < size[t]) ++lt;
        for (const ResItem& I : lists[t]) {
            p.slots = std::max(p.slots, c.u[lt][I.sys]);
            p.lds = std::max(p.lds, c.lds[lt][I.sys]);
        }
    }
    p.team_begin.push_back((int)p.items.size());
    if (p.T) {
        p.blocks = res_grid_blocks(p.nteam, p.T);
        p.members = p.T > 1 ? p.nteam * p.T : 0;
        p.nslot = p.nteam * 2 * p.T;
        return p;
    }
    // teams onto the XCDs' work-groups, largest first: powers of two leave no gap
    int used[NXCD] = {};
    p.member.assign(RES_CUS, int2{-1, 0});
    for (int t = 0; t < p.nteam; ++t) {
        p.teams.push_back(ResTeam{size[t], p.nslot});
        p.nslot += 2 * size[t];
        if (lists[t].empty()) continue;
        const int x = (int)(std::min_element(used, used + NXCD) - used);
        for (int m = 0; m < size[t]; ++m) p.member[(used[x] + m) * NXCD + x] = int2{t, m};
        used[x] += size[t];
        p.members += size[t];
    }
    p.blocks = *std::max_element(used, used + NXCD) * NXCD;
    return p;
}

int ResDevice::init(ResPlan&& p, hipStream_t stream) {
    EAFP_TRY_RC(items.alloc(p.items.size()));
    EAFP_TRY_RC(team_begin.alloc(p.team_begin.size()));
    EAFP_TRY_RC(slots.alloc((size_t)p.nslot * SLOT_WORDS));
    EAFP_TRY_RC(gate.alloc(2));
    EAFP_TRY(hipMemcpy(items.p, p.items.data(), sizeof(ResItem) * p.items.size(), hipMemcpyHostToDevice));
    EAFP_TRY(hipMemcpy(team_begin.p, p.team_begin.data(), sizeof(int) * p.team_begin.size(), hipMemcpyHostToDevice));
    if (!p.T) {
        EAFP_TRY_RC(teams.alloc(p.teams.size()));
        EAFP_TRY_RC(member.alloc(p.member.size()));
        EAFP_TRY(hipMemcpy(teams.p, p.teams.data(), sizeof(ResTeam) * p.teams.size(), hipMemcpyHostToDevice));
        EAFP_TRY(hipMemcpy(member.p, p.member.data(), sizeof(int2) * p.member.size(), hipMemcpyHostToDevice));
    }
    EAFP_TRY(hipMemsetAsync(slots.p, 0, sizeof(u64) * slots.n, stream));
    EAFP_TRY(hipMemsetAsync(gate.p, 0, sizeof(unsigned) * 2, stream));
    tag = 1;
    plan = std::move(p);
    return EAFP_OK;
}

int ResDevice::create(ResPlan&& p, std::unique_ptr<ResDevice>& out, hipStream_t stream) {
    if (!p.ok) return EAFP_OK;
    auto d = std::make_unique<ResDevice>();
    const int rc = d->init(std::move(p), stream);
    if (rc == EAFP_OK) out = std::move(d);
    if (rc != (int)hipErrorOutOfMemory) return rc;
    (void)hipGetLastError();
    return EAFP_OK;
}

constexpr int RES_RETRY = 100;
void ResDevice::gave_up(std::chrono::steady_clock::time_point since) {
    const auto now = std::chrono::steady_clock::now();
    retry = now + RES_RETRY * (now - since);
    ++given_up;
}

ResLaunch ResDevice::launch() const {
    ResLaunch L{};
    L.items = items.p;
    L.team_begin = team_begin.p;
    L.teams = teams.p;
    L.member = member.p;
    L.nteam = plan.nteam;
    L.T = plan.T;
    L.slots = slots.p;
    L.gate = gate.p;
    L.expected = plan.members + absent;
    return L;
}

__global__ void k_res_arm(unsigned* gate, unsigned tag) {
    gate[0] = 0;
    gate[1] = tag;
}

int ResDevice::take_tags(long tags, hipStream_t stream, unsigned* first) {
    if ((unsigned long)tag + (unsigned long)tags > 0xF0000000ul) {   // before the tags wrap, forget the old ones
        EAFP_TRY(hipMemsetAsync(slots.p, 0, sizeof(u64) * slots.n, stream));
        tag = 1;
    }
    *first = tag;
    tag += (unsigned)tags;
    return EAFP_OK;
}

int ResDevice::arm(long tags, hipStream_t stream) {
    unsigned first = 0;
    EAFP_TRY_RC(take_tags(tags, stream, &first));
    k_res_arm<<<1, 1, 0, stream>>>(gate.p, first);
    EAFP_TRY(hipGetLastError());
    return EAFP_OK;
}

}  // namespace eafp
