// resident_check.cpp -- host-side check of the resident solvers' division of
// a system among a team's members, and of what each member reads.
//
// For every mesh and team size it checks that
//   - the members' rectangles cover every z-row exactly once and stay inside
//     the extents that the plan sizes LDS and registers by,
//   - in a member's LDS box every own row finds its four neighbours: own rows,
//     halo rows that exactly one halo index fills, zeros beyond the r walls,
//     the other end of an uncut ring,
//   - every halo row belongs to a member that res_neighbours names (the one
//     whose words the fetch waits for) and is an edge row there,
//   - a launch's work-groups take every (team, member) exactly once.
// Prints "ok <cases>" and exits 0, or the first violation and exits 1.
#include <cstdio>
#include <cstdlib>
#include <set>
#include <utility>
#include <vector>

#include "../hornofusion-full3d_amd/csrc/resident.hpp"

using namespace eafp;

static long g_cases = 0;

#define CHECK(cond, ...)                                                   \
    do {                                                                   \
        if (!(cond)) {                                                     \
            std::printf("FAIL %s:%d: %s: ", __FILE__, __LINE__, #cond);    \
            std::printf(__VA_ARGS__);                                      \
            std::printf("\n");                                             \
            std::exit(1);                                                  \
        }                                                                  \
    } while (0)

static void check_grid(int nr, int nth, int T) {
    ResItem I{};
    I.nr = nr;
    I.nth = nth;
    I.nz = 3;
    res_grid(nr, nth, T, I.pr, I.pth);
    CHECK(I.pr >= 1 && I.pth >= 1 && I.pr * I.pth <= T, "%d %d T %d: %d x %d", nr, nth, T, I.pr, I.pth);
    int rows, lrows;
    res_extent(nr, nth, I.pr, I.pth, rows, lrows);
    std::vector<int> owner(nr * nth, -1);
    for (int m = 0; m < I.pr * I.pth; ++m) {
        const ResRect R = res_rect(I, m);
        CHECK(R.i0 < R.i1 && R.j0 < R.j1 && R.i1 <= nr && R.j1 <= nth, "member %d", m);
        const ResBox X(R, I.pth);
        CHECK(X.rows() <= rows && X.lds_rows() <= lrows, "%d %d T %d member %d", nr, nth, T, m);
        CHECK(X.halo_rows(R, nr) <= lrows - rows || X.rows() < rows, "halo rows of member %d", m);
        for (int i = R.i0; i < R.i1; ++i)
            for (int j = R.j0; j < R.j1; ++j) {
                CHECK(owner[i * nth + j] < 0, "row %d %d twice", i, j);
                owner[i * nth + j] = m;
            }
    }
    for (int o : owner) CHECK(o >= 0, "%d %d T %d: a row without a member", nr, nth, T);
    for (int m = 0; m < I.pr * I.pth; ++m) {
        const ResRect R = res_rect(I, m);
        const ResBox X(R, I.pth);
        std::vector<int> box(X.lds_rows(), -1);   // -1: zeros
        for (int li = 0; li < X.bi; ++li)
            for (int lj = 0; lj < X.bj; ++lj) {
                const int l = X.lds_row(li, lj);
                CHECK(l >= X.pitch && l < (int)box.size(), "row in LDS");
                box[l] = (R.i0 + li) * nth + R.j0 + lj;
            }
        int mem[4];
        res_neighbours(I, m, mem);
        std::set<int> filled;
        const int nh = X.halo_rows(R, nr);
        for (int h = 0; h < nh; ++h) {
            int grow, lrow;
            X.halo(h, R, nr, nth, grow, lrow);
            CHECK(grow >= 0 && grow < nr * nth && lrow >= 0 && lrow < (int)box.size(), "halo %d", h);
            CHECK(box[lrow] < 0 && filled.insert(lrow).second, "halo %d fills a row again", h);
            box[lrow] = grow;
            const int o = owner[grow];
            CHECK(o == mem[0] || o == mem[1] || o == mem[2] || o == mem[3], "halo %d of member %d from %d", h, m, o);
            ResItem J = I;
            const ResRect Q = res_rect(J, o);
            const ResBox Y(Q, I.pth);
            const int li = grow / nth - Q.i0, lj = grow % nth - Q.j0;
            const bool edge = (li == 0 && Q.i0 > 0) || (li == Y.bi - 1 && Q.i1 < nr) ||
                              (Y.hs && (lj == 0 || lj == Y.bj - 1));
            CHECK(edge, "halo row %d is not published by member %d", grow, o);
        }
        for (int li = 0; li < X.bi; ++li)
            for (int lj = 0; lj < X.bj; ++lj) {
                const int l = X.lds_row(li, lj), i = R.i0 + li, j = R.j0 + lj;
                const int S = X.hs || lj > 0 ? l - 1 : l + X.bj - 1;
                const int N = X.hs || lj < X.bj - 1 ? l + 1 : l - (X.bj - 1);
                CHECK(box[l - X.pitch] == (i > 0 ? (i - 1) * nth + j : -1), "W of %d %d", i, j);
                CHECK(box[l + X.pitch] == (i < nr - 1 ? (i + 1) * nth + j : -1), "E of %d %d", i, j);
                CHECK(box[S] == i * nth + (j + nth - 1) % nth, "S of %d %d", i, j);
                CHECK(box[N] == i * nth + (j + 1) % nth, "N of %d %d", i, j);
            }
    }
    ++g_cases;
}

static void check_members(int nteam, int T) {
    std::set<std::pair<int, int>> seen;
    const int G = res_grid_blocks(nteam, T);
    CHECK(G >= nteam * T, "grid");
    for (int b = 0; b < G; ++b) {
        int team, m;
        res_member(b, nteam, T, team, m);
        CHECK(m >= 0 && m < T && team >= 0, "block %d", b);
        if (team < nteam) CHECK(seen.insert({team, m}).second, "block %d takes a member again", b);
        if (T <= 32 && team < nteam) CHECK(b % NXCD == team % NXCD, "team %d over several XCDs", team);
    }
    CHECK((int)seen.size() == nteam * T, "%d teams of %d: %d members", nteam, T, (int)seen.size());
    ++g_cases;
}

int main() {
    const int rs[] = {1, 2, 3, 5, 7, 12, 18, 35, 60, 75, 120}, ts[] = {1, 2, 3, 6, 17, 36, 66, 120, 240};
    for (int T = 1; T <= RES_CUS; T *= 2) {
        for (int nr : rs)
            for (int nth : ts) check_grid(nr, nth, T);
        for (int n = 1; n <= RES_CUS / T; ++n) check_members(n, T);
    }
    std::printf("ok %ld\n", g_cases);
    return 0;
}
