// The parts of an overlapped line-TDMA sweep (chain_part and the rest in
// csrc/tdma_line.hpp), line by line: with the parts of a launch taken in
// either order, each line finds what it reads done, moved and prepared;
// nothing is written that a later kernel still needs as it was; and the parts
// of a pass are all of it, once.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../hornofusion-full3d_amd/csrc/tdma_line.hpp"

using namespace eafp::tdma;

#define CHECK(c, ...)                                                        \
    do {                                                                     \
        if (!(c)) {                                                          \
            std::printf("line %d: ", __LINE__);                              \
            std::printf(__VA_ARGS__);                                        \
            std::printf("\n");                                               \
            std::exit(1);                                                    \
        }                                                                    \
    } while (0)

struct Grid {
    int nu, nv;
    std::vector<char> x;
    Grid(int u, int v) : nu(u), nv(v), x((size_t)(u + 2) * (v + 2), 0) {}
    char& at(int u, int v) { return x[(size_t)v * (nu + 2) + u]; }
};

// The lines of diagonals span of a pass: the updated neighbours done.
static void run(Grid& done, const TdSpan& span) {
    for (int w = span.lo; w < span.hi; ++w) {
        int lo, hi;
        diagonal_range(w, done.nu, done.nv, lo, hi);
        for (int v = lo; v <= hi; ++v) {
            const int u = w + 2 - v;
            CHECK(!done.at(u, v) && (u == 1 || done.at(u - 1, v)) && (v == 1 || done.at(u, v - 1)), "line (%d,%d)", u, v);
            done.at(u, v) = 1;
        }
    }
}

static void check(int nr, int nth, int nz, int parts, bool forward) {
    TdSys s{};
    s.nr = nr;
    s.nth = nth;
    s.nz = nz;
    Grid r(nth, nz), th(nr, nz), z(nr, nth), prep1(nr, nz), prep2(nr, nth);
    std::vector<char> plane((size_t)nz + 2, 0), column((size_t)nr + 2, 0);
    auto r_part = [&](int c) {
        run(r, chain_part(s, 0, c, parts));
    };
    auto hand_planes = [&](int c) {
        for (int k = 1; k <= nz; ++k) {
            PackTile t{};
            t.k0 = (k - 1) / TD_PT * TD_PT;
            if (!in_move_part(s, 0, t, c, parts)) continue;
            CHECK(!plane[(size_t)k], "plane %d twice", k);
            for (int j = 1; j <= nth; ++j) CHECK(r.at(j, k), "r line (%d,%d) moved before it is done", j, k);
            for (int i = 1; i <= nr; ++i) CHECK(!th.at(i, k), "theta line (%d,%d) overwritten", i, k);
            plane[(size_t)k] = 1;
        }
        for (int i = 1; i <= nr; ++i)
            for (int k = 1; k <= nz; ++k)
                if (in_prep_part(s, 1, i | k << 16, c, parts)) {
                    CHECK(!prep1.at(i, k) && plane[(size_t)k] && (k == nz || plane[(size_t)k + 1]), "prep of (%d,%d)", i, k);
                    CHECK(!th.at(i, k) && (i == nr || !th.at(i + 1, k)) && (k == nz || !th.at(i, k + 1)), "late prep");
                    prep1.at(i, k) = 1;
                }
    };
    auto th_part = [&](int c) {
        const TdSpan sp = chain_part(s, 1, c, parts);
        run(th, sp);
        for (int w = sp.lo; w < sp.hi; ++w)
            for (int k = 1; k <= nz; ++k)
                if (const int i = w + 2 - k; i >= 1 && i <= nr) CHECK(prep1.at(i, k), "theta line (%d,%d) not prepared", i, k);
    };
    auto hand_columns = [&](int c) {
        for (int i = 1; i <= nr; ++i) {
            PackTile t{};
            t.i0 = (i - 1) / TD_PT * TD_PT;
            if (!in_move_part(s, 1, t, c, parts)) continue;
            CHECK(!column[(size_t)i], "column %d twice", i);
            for (int k = 1; k <= nz; ++k) CHECK(th.at(i, k), "theta line (%d,%d) moved before it is done", i, k);
            for (int j = 1; j <= nth; ++j) CHECK(!z.at(i, j), "z line (%d,%d) overwritten", i, j);
            column[(size_t)i] = 1;
        }
        for (int i = 1; i <= nr; ++i)
            for (int j = 1; j <= nth; ++j)
                if (in_prep_part(s, 2, i | j << 16, c, parts)) {
                    CHECK(!prep2.at(i, j) && column[(size_t)i] && (i == nr || column[(size_t)i + 1]), "prep of (%d,%d)", i, j);
                    CHECK(!z.at(i, j) && !z.at(i, j == nth ? 1 : j + 1) && !z.at(i, j == 1 ? nth : 1) &&
                              (i == nr || !z.at(i + 1, j)), "late prep");
                    prep2.at(i, j) = 1;
                }
    };
    auto z_part = [&](int c) {
        const TdSpan sp = chain_part(s, 2, c, parts);
        run(z, sp);
        for (int w = sp.lo; w < sp.hi; ++w)
            for (int j = 1; j <= nth; ++j)
                if (const int i = w + 2 - j; i >= 1 && i <= nr) CHECK(prep2.at(i, j), "z line (%d,%d) not prepared", i, j);
    };
    // the launches of a sweep: r part a, theta part a - 1 and z part
    // a - parts - 1 side by side, then portion a is handed on
    for (int a = 0; a <= 2 * parts; ++a) {
        for (int q = 0; q < 3; ++q) {
            const int P = forward ? q : 2 - q;
            if (P == 0 && a < parts) r_part(a);
            if (P == 1 && a >= 1 && a < 2 * parts) th_part(a - 1);
            if (P == 2 && a > parts) z_part(a - parts - 1);
        }
        if (a < parts) hand_planes(a);
        else if (a < 2 * parts) hand_columns(a - parts);
    }
    for (int k = 1; k <= nz; ++k) {
        for (int j = 1; j <= nth; ++j) CHECK(r.at(j, k), "r line (%d,%d) left out", j, k);
        for (int i = 1; i <= nr; ++i) CHECK(th.at(i, k) && prep1.at(i, k), "theta line (%d,%d) left out", i, k);
    }
    for (int i = 1; i <= nr; ++i)
        for (int j = 1; j <= nth; ++j) CHECK(z.at(i, j) && prep2.at(i, j), "z line (%d,%d) left out", i, j);
}

int main() {
    long n = 0;
    for (int nr : {1, 2, 15, 16, 17, 32, 33, 60, 63, 70})
        for (int nth : {1, 2, 16, 31, 66, 120})
            for (int nz : {1, 2, 16, 17, 31, 32, 33, 34, 48, 49, 64, 65, 84})
                for (int parts : {1, 2, 3, 4, 5, 8})
                    for (int order = 0; order < 2; ++order, ++n) check(nr, nth, nz, parts, order != 0);
    std::printf("ok %ld\n", n);
    return 0;
}
