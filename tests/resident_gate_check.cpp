// Who may launch (ResidentGate in csrc/resident_plan.hip): threads with plans of
// their own never hold more than the chip between them, come in the order in
// which they asked, and a plan of teams of one takes places too.  And where the
// rows cross: one double per cell for FP64, two floats for the mixed solver with
// rows of four cells or more, no two systems in the same place.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <thread>

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

static ResPlan plan(int S, int nr, int nth, int nz) {
    std::vector<SysGeom> g(S);
    for (auto& s : g) {
        s = SysGeom{};
        s.nr = nr;
        s.nth = nth;
        s.nz = nz;
        s.n = nr * nth * nz;
    }
    return plan_resident(g, kLim, pitch);
}

static std::atomic<int> g_held{0};
static std::atomic<long> g_launches{0};

static void hold(int n) {
    const ResidentGate gate(n);
    const int now = g_held.fetch_add(n) + n;
    CHECK(now <= RES_CUS, "%d work-groups at once", now);
    ++g_launches;
    std::this_thread::sleep_for(std::chrono::microseconds(50));
    g_held.fetch_sub(n);
}

static int pitch1(int nz) { return (nz + 3) / 4 * 4; }
static int pitch2(int nz) { return (nz + 7) / 8 * 8; }

static void exchange() {
    std::mt19937 rng(11);
    for (int rep = 0; rep < 200; ++rep) {
        std::vector<SysGeom> g(1 + rng() % 40);
        for (auto& s : g) {
            s = SysGeom{};
            s.nr = 1 + (int)(rng() % 30);
            s.nth = 1 + (int)(rng() % 40);
            s.nz = (rep % 2 ? 4 : 1) + (int)(rng() % 60);
        }
        const long ncells = layout_systems(g);
        for (int (*pt)(int) : {pitch, pitch1, pitch2}) {
            const ResPlan p = plan_resident(g, kLim, pt);
            if (!p.ok) continue;
            if (pt == pitch) CHECK(p.xlen <= ncells, "%ld of %ld", p.xlen, ncells);
            if (rep % 2) CHECK(p.xlen <= 2 * ncells, "%ld of %ld", p.xlen, 2 * ncells);
            std::vector<std::pair<long, long>> part;
            for (const ResItem& I : p.items) part.push_back({I.xoff, I.xoff + (long)I.nr * I.nth * pt(I.nz)});
            std::sort(part.begin(), part.end());
            CHECK(part.front().first == 0 && part.back().second <= p.xlen, "ends");
            for (size_t q = 1; q < part.size(); ++q)
                CHECK(part[q].first >= part[q - 1].second && part[q].first % 32 == 0, "part %zu", q);
        }
    }
}

int main() {
    exchange();
    // plans and what they take
    const ResPlan many = plan(5000, 8, 8, 8), one = plan(1, 60, 120, 84), few = plan(3, 20, 30, 33);
    CHECK(many.ok && many.T == 1 && many.members == 0, "teams of %d", many.T);
    CHECK(many.places() == many.nteam && many.places() == RES_CUS, "%d places", many.places());
    CHECK(one.places() == one.members && one.places() > 64, "%d places", one.places());
    CHECK(few.places() == few.members && few.places() < RES_CUS, "%d places", few.places());

    // never more than the chip
    std::vector<std::thread> t;
    for (int q = 0; q < 6; ++q)
        t.emplace_back([&, q] {
            std::mt19937 rng(q);
            for (int r = 0; r < 200; ++r) {
                const int pick = (int)(rng() % 4);
                hold(pick == 0 ? many.places() : pick == 1 ? one.places() : pick == 2 ? few.places() : 1 + (int)(rng() % RES_CUS));
            }
        });
    for (auto& x : t) x.join();
    CHECK(g_launches == 1200 && g_held == 0, "%ld launches", g_launches.load());

    // first come, first served: a small plan does not pass a large one that waits
    std::vector<int> order;
    std::atomic<int> asked{0};
    std::thread a, b;
    {
        const ResidentGate held(200);
        a = std::thread([&] {
            ++asked;
            const ResidentGate g(100);
            order.push_back(100);
            std::this_thread::sleep_for(std::chrono::milliseconds(20));
        });
        while (asked < 1) std::this_thread::yield();
        std::this_thread::sleep_for(std::chrono::milliseconds(50));
        b = std::thread([&] {
            ++asked;
            const ResidentGate g(200);
            order.push_back(200);
        });
        while (asked < 2) std::this_thread::yield();
        std::this_thread::sleep_for(std::chrono::milliseconds(50));
        CHECK(order.empty(), "a waiting plan ran");
    }
    a.join();
    b.join();
    CHECK(order.size() == 2 && order[0] == 100 && order[1] == 200, "order");
    std::printf("ok %ld\n", g_launches.load());
    return 0;
}
