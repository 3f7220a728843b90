// resident_plan.hip -- host side of the resident solvers (resident_plan.hpp).
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

// Every power of two T is priced: a team's iteration is its sums (sync_us)
// and its slots, a launch runs as many teams as fit the CUs, and the longest
// team list sets the time.  Systems go to the teams largest first, each to
// the team with the fewest cells so far.
ResPlan plan_resident(const std::vector<SysGeom>& g, const ResLimits& lim, int (*xpitch)(int nz)) {
    ResPlan best;
    if (device_cus() < RES_CUS) return best;
    const int S = (int)g.size();
    std::vector<int> order(S);
    for (int s = 0; s < S; ++s) order[s] = s;
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return g[a].n > g[b].n; });
    std::vector<long> xoff(S);
    long xlen = 0;
    for (int s = 0; s < S; ++s) {
        xoff[s] = xlen;
        xlen += ((long)g[s].nr * g[s].nth * xpitch(g[s].nz) + 31) / 32 * 32;
    }
    for (int lt = 0, T = 1; T <= RES_CUS; ++lt, T *= 2) {
        ResPlan p;
        p.nsys = S;
        p.T = T;
        p.nteam = std::min(S, RES_CUS / T);
        std::vector<std::vector<ResItem>> lists(p.nteam);
        std::vector<float> cost(p.nteam, 0.f);
        bool fits = true;
        for (int s : order) {
            const SysGeom& G = g[s];
            ResItem I{};
            I.sys = s;
            I.nr = G.nr;
            I.nth = G.nth;
            I.nz = G.nz;
            I.off = G.off;
            I.xoff = xoff[s];
            res_grid(G.nr, G.nth, T, I.pr, I.pth);
            int rows, lrows;
            res_extent(G.nr, G.nth, I.pr, I.pth, rows, lrows);
            const int hrows = lrows - rows;
            const int u = lim.slots(G.nz, rows);
            const size_t lds = lim.lds(G.nz, rows, lrows, hrows);
            if (u < 1 || u > lim.max_slots || lds > (size_t)RES_LDS) {
                fits = false;
                break;
            }
            p.slots = std::max(p.slots, u);
            p.lds = std::max(p.lds, lds);
            int t = 0;
            for (int q = 1; q < p.nteam; ++q)
                if (cost[q] < cost[t]) t = q;
            lists[t].push_back(I);
            cost[t] += lim.sync_us[lt] + lim.slot_us * (float)u;
        }
        if (!fits) continue;
        for (float c : cost) p.est_us = std::max(p.est_us, c);
        if (best.ok && p.est_us >= best.est_us) continue;
        p.ok = true;
        p.xlen = xlen;
        p.blocks = res_grid_blocks(p.nteam, T);
        for (const auto& l : lists) {
            p.team_begin.push_back((int)p.items.size());
            p.items.insert(p.items.end(), l.begin(), l.end());
            p.max_items = std::max(p.max_items, (int)l.size());
        }
        p.team_begin.push_back((int)p.items.size());
        best = p;
    }
    return best;
}

int ResDevice::init(ResPlan&& p, hipStream_t stream) {
    EAFP_TRY_RC(items.alloc(p.items.size()));
    EAFP_TRY_RC(team_begin.alloc(p.team_begin.size()));
    EAFP_TRY_RC(slots.alloc((size_t)p.nteam * 2 * p.T * SLOT_WORDS));
    EAFP_TRY_RC(gate.alloc(2));
    EAFP_TRY(hipMemcpy(items.p, p.items.data(), sizeof(ResItem) * p.items.size(), hipMemcpyHostToDevice));
    EAFP_TRY(hipMemcpy(team_begin.p, p.team_begin.data(), sizeof(int) * p.team_begin.size(), hipMemcpyHostToDevice));
    EAFP_TRY(hipMemsetAsync(slots.p, 0, sizeof(u64) * slots.n, stream));
    EAFP_TRY(hipMemsetAsync(gate.p, 0, sizeof(unsigned) * 2, stream));
    tag = 1;
    plan = std::move(p);
    return EAFP_OK;
}

ResLaunch ResDevice::launch() const {
    ResLaunch L{};
    L.items = items.p;
    L.team_begin = team_begin.p;
    L.nteam = plan.nteam;
    L.T = plan.T;
    L.slots = slots.p;
    L.gate = gate.p;
    L.expected = plan.T > 1 ? plan.nteam * plan.T : 0;
    return L;
}

__global__ void k_res_arm(unsigned* gate, unsigned tag) {
    gate[0] = 0;
    gate[1] = tag;
}

int ResDevice::arm(long tags, hipStream_t stream) {
    if ((unsigned long)tag + (unsigned long)tags > 0xF0000000ul) {   // before the tags wrap, forget the old ones
        EAFP_TRY(hipMemsetAsync(slots.p, 0, sizeof(u64) * slots.n, stream));
        tag = 1;
    }
    k_res_arm<<<1, 1, 0, stream>>>(gate.p, tag);
    EAFP_TRY(hipGetLastError());
    tag += (unsigned)tags;
    return EAFP_OK;
}

}  // namespace eafp
