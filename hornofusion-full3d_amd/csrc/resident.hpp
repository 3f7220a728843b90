// resident.hpp -- systems kept on chip for a whole solve.
//
// A p' system of 604,800 cells needs 53 MB in FP64; the 256 CUs hold 128 MB
// of registers and 40 MB of LDS.  The resident solvers therefore give every
// system to a team of T work-groups (one per CU), each of which keeps a
// rectangle of the system's z-rows in registers and LDS through all
// iterations.  Only the rows on a rectangle's edge and the dot products'
// partial sums cross between work-groups, through memory that every XCD
// sees (agent-scope relaxed stores and loads, which go past the XCDs' own
// L2s).
//
// Sum over a team: every member stores its partial sums as 8-byte words, 32
// bits of the value and a 32-bit tag in each, and reads every member's
// words until all carry the tag of this sum.  Data and flag travel in one
// word, so a sum costs one store and one load through memory, and all
// members add the same words in the same order: the same bits everywhere.
// Measured on MI355X (store to the last member's sum): 1.1 us for 2..16
// members, 1.9 us for 32, 2.5 us for 256.  The slots are double-buffered by
// the tag's parity: a member stores sum n+2 only after sum n+1, which every
// member joins after it has read sum n.
//
// Edge rows are stored before a sum and read after it.  A wave waits for its
// own stores before the work-group's words go out, so a complete sum means
// that every member's rows are in memory.  Tagged words for the rows (no
// wait, the neighbours poll them) were slower: the exchange of 1848 doubles
// with the sum took 6.1 us over 256 members against 4.5, the words being
// twice the bytes.
//
// All work-groups of a launch must be on the GPU at once.  The host gives
// out at most one work-group per CU (ResidentGate), and a launch begins
// with a gate: a work-group that finds the others missing for GATE_TICKS
// marks the launch as given up, all its work-groups leave without having
// written anything, and the host solves with the streaming kernels instead.
// Past the gate every wait ends because all the members run; should one
// last WAIT_TICKS all the same, the work-group raises the same mark and
// leaves.
//
// How long a sum takes also hangs on where the slots lie in memory: the same
// code on the same mesh took 2.4 or 2.6 us per FP64 iteration of 18x36x24, and
// 18.5 or 20.3 for 32 uneven systems, with the slots at other addresses.
#pragma once
#include <algorithm>

#include "eafp_common.hpp"

namespace eafp {

typedef unsigned long long u64;

constexpr int RB = 512;                    // threads of a resident work-group
constexpr int RW = RB / 64;
constexpr int RES_CUS = 256;               // one work-group per CU
constexpr int RES_LDS = 160 * 1024;        // LDS of a CU
constexpr int RES_LDS_ALONE = 84 * 1024;   // a work-group that takes this much is alone on its CU
constexpr int SLOT_WORDS = 8;              // words per member and parity: up to 4 doubles
constexpr long long GATE_TICKS = 20000000;    // 0.2 s of the 100 MHz clock
constexpr long long WAIT_TICKS = 400000000;   // 4 s

// One system of a resident launch.
struct ResItem {
    int sys;
    int nr, nth, nz;
    int pr, pth;        // the team's grid of rectangles, pr * pth <= T
    int pad_;
    long off;           // first cell of the system in the arenas
    long xoff;          // first element of the system in the exchange buffer
};

// A team of a launch whose teams differ in size: its work-groups and the
// first slot of its own.
struct ResTeam {
    int T, slot0;
};

// A launch: teams of T work-groups, or (T = 0) of the sizes of `teams`, with
// the team and member of each work-group in `member`; team t takes the items
// [team_begin[t], team_begin[t+1]) one after another.
struct ResLaunch {
    const ResItem* items;
    const int* team_begin;
    const ResTeam* teams;
    const int2* member;
    int nteam, T;
    u64* slots;         // 2 * T * SLOT_WORDS of every team
    unsigned* gate;     // [0] arrivals and the give-up mark, [1] the next launch's first tag
    int expected;       // work-groups that pass the gate
    int pad_;
};

constexpr unsigned GATE_GIVEN_UP = 0x80000000u;

// The rectangle of member m: rows i0..i1-1 x j0..j1-1.
struct ResRect {
    int i0, i1, j0, j1;
};
__host__ __device__ __forceinline__ ResRect res_rect(const ResItem& I, int m) {
    const int a = m / I.pth, b = m % I.pth;
    return {(int)((long)I.nr * a / I.pr), (int)((long)I.nr * (a + 1) / I.pr), (int)((long)I.nth * b / I.pth),
            (int)((long)I.nth * (b + 1) / I.pth)};
}

// The members next to m that own its halo rows (-1: none): r below, r above,
// theta below, theta above.
__host__ __device__ __forceinline__ void res_neighbours(const ResItem& I, int m, int (&mem)[4]) {
    const int a = m / I.pth, b = m % I.pth;
    const bool in = m < I.pr * I.pth;
    mem[0] = in && a > 0 ? m - I.pth : -1;
    mem[1] = in && a + 1 < I.pr ? m + I.pth : -1;
    mem[2] = in && I.pth > 1 ? a * I.pth + (b > 0 ? b - 1 : I.pth - 1) : -1;
    mem[3] = in && I.pth > 1 ? a * I.pth + (b + 1 < I.pth ? b + 1 : 0) : -1;
}

// A rectangle's rows in LDS: one row more on either side in r (beyond a
// wall it holds zeros), and in theta where the ring is cut (pth > 1); an
// uncut ring wraps inside the rectangle.
struct ResBox {
    int bi, bj, hs, pitch;
    __host__ __device__ ResBox(const ResRect& r, int pth) {
        bi = r.i1 - r.i0;
        bj = r.j1 - r.j0;
        hs = pth > 1 ? 1 : 0;
        pitch = bj + 2 * hs;
    }
    __host__ __device__ int rows() const { return bi * bj; }
    __host__ __device__ int lds_rows() const { return (bi + 2) * pitch; }
    __host__ __device__ int lds_row(int li, int lj) const { return (li + 1) * pitch + lj + hs; }
    // rows read from other members (or, where the ring is cut in two, twice from the same one)
    __host__ __device__ int halo_rows(const ResRect& r, int nr) const {
        return ((r.i0 > 0) + (r.i1 < nr)) * bj + 2 * hs * bi;
    }
    // halo row h: its global row (i*nth + j) and its row in LDS
    __host__ __device__ void halo(int h, const ResRect& r, int nr, int nth, int& grow, int& lrow) const {
        int li, lj;
        const int up = r.i0 > 0 ? bj : 0, dn = r.i1 < nr ? bj : 0;
        if (h < up) {
            li = -1;
            lj = h;
        } else if (h < up + dn) {
            li = bi;
            lj = h - up;
        } else {
            const int q = h - up - dn;
            li = q < bi ? q : q - bi;
            lj = q < bi ? -1 : bj;
        }
        int j = r.j0 + lj;
        j = j < 0 ? j + nth : (j >= nth ? j - nth : j);
        grow = (r.i0 + li) * nth + j;
        lrow = lds_row(li, lj);
    }
};

// Largest number of rows and of LDS rows of any member for a pr x pth grid.
inline void res_extent(int nr, int nth, int pr, int pth, int& rows, int& lds_rows) {
    const int bi = (nr + pr - 1) / pr, bj = (nth + pth - 1) / pth;
    rows = bi * bj;
    lds_rows = (bi + 2) * (bj + (pth > 1 ? 2 : 0));
}

// The grid of at most T rectangles with the fewest rows per member, then the
// fewest halo rows.
inline void res_grid(int nr, int nth, int T, int& pr, int& pth) {
    long best = -1;
    pr = pth = 1;
    for (int a = 1; a <= T && a <= nr; ++a) {
        const int b = std::min(T / a, nth);
        // not more columns than the same column width needs
        const int bj = (nth + b - 1) / b, bb = (nth + bj - 1) / bj;
        const int bi = (nr + a - 1) / a, aa = (nr + bi - 1) / bi;
        const long cost = (long)bi * bj * 1024 + (a > 1 ? 2 * bj : 0) + (bb > 1 ? 2 * bi : 0);
        if (best < 0 || cost < best) {
            best = cost;
            pr = aa;
            pth = bb;
        }
    }
}

// Work-groups of a launch and the team and member of each.  Hardware deals
// work-groups to the XCDs round robin; a team of at most 32 sits on one XCD.
inline int res_grid_blocks(int nteam, int T) { return T <= 32 ? NXCD * ((nteam + NXCD - 1) / NXCD) * T : nteam * T; }
__host__ __device__ __forceinline__ void res_member(int b, int nteam, int T, int& team, int& m) {
    const int x = b % NXCD, q = b / NXCD;
    if (T <= 32) {
        team = (q / T) * NXCD + x;
        m = q % T;
    } else {
        const int L = x * (nteam * T / NXCD) + q;
        team = L / T;
        m = L % T;
    }
}

// ---------------------------------------------------------------------------
// Device side
// ---------------------------------------------------------------------------
// The team and member of this work-group; false when it has none.
__device__ __forceinline__ bool res_place(const ResLaunch& L, int& team, int& m, int& T, u64*& slots) {
    int slot0;
    if (L.T) {
        res_member((int)blockIdx.x, L.nteam, L.T, team, m);
        if (team >= L.nteam) return false;
        T = L.T;
        slot0 = team * 2 * T;
    } else {
        const int2 b = L.member[blockIdx.x];
        team = __builtin_amdgcn_readfirstlane(b.x);
        m = __builtin_amdgcn_readfirstlane(b.y);
        if (team < 0) return false;
        T = __builtin_amdgcn_readfirstlane(L.teams[team].T);
        slot0 = __builtin_amdgcn_readfirstlane(L.teams[team].slot0);
    }
    slots = L.slots + (size_t)slot0 * SLOT_WORDS;
    return true;
}

__device__ __forceinline__ u64 ld_agent(const u64* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_agent(u64* p, u64 v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double ld_agent_d(const double* p) {
    return __longlong_as_double((long long)ld_agent(reinterpret_cast<const u64*>(p)));
}
__device__ __forceinline__ void st_agent_d(double* p, double v) {
    st_agent(reinterpret_cast<u64*>(p), (u64)__double_as_longlong(v));
}
// LDS scratch of team_sum: two copies (by the tag's parity), per value one
// entry per wave for the member's own sum and one per reading wave.
struct TeamLds {
    double own[2][4][RW];
    double all[2][4][RW];
    int dead;
};

struct Team {
    u64* slots;
    unsigned* gate;
    int T, m;
    unsigned tag;
};

// Every store this wave has issued has reached memory.
__device__ __forceinline__ void drain_stores() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// The launch's gate (see the head of this file).  Called by every thread;
// returns false when the launch was given up.
__device__ __forceinline__ bool res_gate(const ResLaunch& L, TeamLds& S) {
    if (threadIdx.x == 0) {
        int dead = 0;
        if (L.expected > 1) {
            unsigned w = __hip_atomic_fetch_add(L.gate, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u;
            const long long t0 = wall_clock64();
            while (!(w & GATE_GIVEN_UP) && w < (unsigned)L.expected) {
                if (wall_clock64() - t0 > GATE_TICKS) {
                    // marks the launch unless the last member has arrived meanwhile
                    if (__hip_atomic_compare_exchange_strong(L.gate, &w, w | GATE_GIVEN_UP, __ATOMIC_RELAXED,
                                                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                        w |= GATE_GIVEN_UP;
                    continue;
                }
                __builtin_amdgcn_s_sleep(1);
                w = __hip_atomic_load(L.gate, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            dead = (w & GATE_GIVEN_UP) ? 1 : 0;
        }
        S.dead = dead;
    }
    __syncthreads();
    return S.dead == 0;
}

__device__ __forceinline__ bool res_waited_too_long(const Team& t, long long t0) {
    const bool given_up = (__hip_atomic_load(t.gate, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & GATE_GIVEN_UP) != 0;
    if (!given_up && wall_clock64() - t0 <= WAIT_TICKS) return false;
    __hip_atomic_fetch_or(t.gate, GATE_GIVEN_UP, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
}

// Lane q < 4 of the wave waits for member mem[q]'s words of the coming sum
// (-1: none): what that member published before it is then in memory.
__device__ __forceinline__ void wait_members(const Team& t, TeamLds& S, const int (&mem)[4]) {
    const int lane = threadIdx.x & 63;
    const int m = lane == 0 ? mem[0] : lane == 1 ? mem[1] : lane == 2 ? mem[2] : lane == 3 ? mem[3] : -1;
    if (m >= 0) {
        const u64* s = t.slots + ((size_t)(t.tag & 1u) * t.T + m) * SLOT_WORDS;
        const long long t0 = wall_clock64();
        int n = 0;
        while ((unsigned)(ld_agent(s) >> 32) != t.tag)
            if ((++n & 255) == 0 && res_waited_too_long(t, t0)) {
                S.dead = 1;
                break;
            }
    }
    asm volatile("" ::: "memory");   // the fetches stay behind the wait
}

// v[c] summed over the work-group's threads and the team's members, the
// same bits in every thread of the team.  Called by every thread of the
// work-group; false: the launch was given up.  `publish`: what the team's
// threads stored before (st_agent) is in memory once the sum is complete.
// Waves without members' words to read call aside(w, n), w of n, to fetch
// the neighbours' rows (wait_members) while the rest of the team is waited
// for; a team of one has none.
//
// A member's words have 64 bytes of their own and are read 16 bytes at a
// time.  The sum alone over 256 members takes 2.5 us so; 8-byte reads took
// 2.8, several members' words in one line 3.6 (16 bytes apart) or 4.1 us
// (word by word).
typedef unsigned res_u4 __attribute__((ext_vector_type(4)));

template <int NV, typename Aside>
__device__ __forceinline__ bool team_sum(Team& t, double (&v)[NV], TeamLds& S, bool publish, Aside aside) {
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const unsigned par = t.tag & 1u;
#pragma unroll
    for (int c = 0; c < NV; ++c) {
        const double w = wave_sum(v[c]);
        if (lane == 0) S.own[par][c][wid] = w;
    }
    if (publish) drain_stores();
    __syncthreads();
    if (t.T == 1) {
#pragma unroll
        for (int c = 0; c < NV; ++c) {
            double s = 0.0;
#pragma unroll
            for (int w = 0; w < RW; ++w) s += S.own[par][c][w];
            v[c] = s;
        }
        ++t.tag;
        return true;
    }
    u64* base = t.slots + (size_t)par * t.T * SLOT_WORDS;
    if (tid < 2 * NV) {
        const int c = tid >> 1;
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < RW; ++w) s += S.own[par][c][w];
        const u64 bits = (u64)__double_as_longlong(s);
        st_agent(base + t.m * SLOT_WORDS + tid, (u64)t.tag << 32 | ((tid & 1) ? bits >> 32 : bits & 0xFFFFFFFFull));
    }
    const int nw = (t.T + 63) >> 6;   // the waves that read members: T <= 256, so 4 of 8 at most
    if (wid < nw) {
        double x[NV];
#pragma unroll
        for (int c = 0; c < NV; ++c) x[c] = 0.0;
        if (tid < t.T) {
            const auto rs = __builtin_amdgcn_make_buffer_rsrc(base, 0, t.T * SLOT_WORDS * 8, 0x00020000);
            constexpr int SC1 = 16;    // the load's scope: the agent
            res_u4 w[NV];
            const long long t0 = wall_clock64();
            int n = 0;
            for (;;) {
                unsigned bad = 0;
#pragma unroll
                for (int c = 0; c < NV; ++c)
                    w[c] = __builtin_amdgcn_raw_buffer_load_b128(rs, tid * SLOT_WORDS * 8 + c * 16, 0, SC1);
#pragma unroll
                for (int c = 0; c < NV; ++c) bad |= (w[c].y ^ t.tag) | (w[c].w ^ t.tag);
                if (!bad) break;
                if ((++n & 255) == 0 && res_waited_too_long(t, t0)) {
                    S.dead = 1;
                    break;
                }
                asm volatile("" ::: "memory");   // the words are read again
            }
#pragma unroll
            for (int c = 0; c < NV; ++c) x[c] = __hiloint2double((int)w[c].z, (int)w[c].x);
        }
#pragma unroll
        for (int c = 0; c < NV; ++c) {
            const double y = wave_sum(x[c]);
            if (lane == 0) S.all[par][c][wid] = y;
        }
    } else if (publish) {
        aside(wid - nw, RW - nw);
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < NV; ++c) {
        double s = 0.0;
        for (int w = 0; w < nw; ++w) s += S.all[par][c][w];
        v[c] = s;
    }
    ++t.tag;
    return S.dead == 0;
}

struct NoAside {
    __device__ void operator()(int, int) const {}
};

// Hides a value from the optimiser, so that what is derived from it inside a
// loop is formed there again instead of being kept in registers.
__device__ __forceinline__ int fresh(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

// The value is formed by here: what leads to it is not put off past this
// point (to after a whole loop over the thread's cells, say, with everything
// it needs kept in registers meanwhile).
__device__ __forceinline__ void formed(float& v) { asm volatile("" : "+v"(v)); }
__device__ __forceinline__ void formed(double& v) { asm volatile("" : "+v"(v)); }

// A value that is the same in every lane, in scalar registers.
template <typename R>
__device__ __forceinline__ R uniform(const R& v) {
    static_assert(sizeof(R) % 4 == 0, "whole words");
    int w[sizeof(R) / 4];
    __builtin_memcpy(w, &v, sizeof(R));
#pragma unroll
    for (int i = 0; i < (int)(sizeof(R) / 4); ++i) w[i] = __builtin_amdgcn_readfirstlane(w[i]);
    R r;
    __builtin_memcpy(&r, w, sizeof(R));
    return r;
}

// Row and place in the row of element c (c < 2^24) of consecutive rows of n.
__device__ __forceinline__ void row_of(int c, int n, float inv_n, int& row, int& k) {
    row = fdiv(c, n, inv_n);
    k = c - row * n;
}

}  // namespace eafp
