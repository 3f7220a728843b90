// cg64_resident.hip -- the FP64 Jacobi-PCG of cg_3d_mpi
// (src/mod_solver_3d.f90:485-620) with the system kept on chip.
//
// The streaming kernels (cg64.hip) read and write 152 bytes per cell and
// iteration in two launches; at 604,800 cells an iteration took 25.2 us, two
// thirds of it launch and drain latency.  Here one launch runs the solve.  A
// team of work-groups (resident.hpp) holds the system: a thread keeps its
// cells' seven coefficients, x, r and z (or q) in registers, the search
// direction p of the rectangle and its halo rows is in LDS, and an
// iteration reads and writes memory only for the halo rows of z and the two
// team sums.  What bounds it now is those two sums and the exchange of z
// between them: 604,800 cells on 256 work-groups take 9.4 us per iteration,
// 7.3 of it the sums and the exchange and 2.1 the cells (5 per thread);
// 4,608 cells on 16 take 3.8 (14 streaming); 32 uneven systems of 15,000 to
// 115,000 cells on 8 teams of 32 take 27 us per iteration of all (52
// streaming).  The matrix is taken as given: seven coefficients, no symmetry.
//
// The recurrences, their tests and their order are the streaming kernels':
//   p = z + beta p (own rows, and the halo rows from the neighbours' z)
//   q = A p, p.q                                          -> team sum
//   breakdown test, alpha; x += alpha p, r -= alpha q, z = r/max(|aP|,SMALL)
//   r.r, r.z, edge rows of z to the exchange buffer       -> team sum
//   residual, stop tests, beta
// The halo rows of p are formed from the same z, beta and old p as in the
// member that owns them, so every member has the same p.
#include "cg64.hpp"
#include "resident_plan.hpp"

namespace eafp {

struct R64Args {
    Cg64Args a;
    ResLaunch L;
    double* zx;          // edge rows of z for the neighbours, ResItem::xoff + row * nz + k: the
                         // streaming kernels' q, which has the same places and is free here
    int iters;           // iterations per item and launch at most
};

// Cells per thread, U; RB * U cells per work-group.
constexpr int R64_MAX_U = 8;

// LDS: the team's scratch, then p of the box rows (with one element in
// front, so that the cell below a box's first exists), then per halo element
// its place in the system and in p, then the halo elements of z, then x
// where the registers do not hold it.
static int r64_slots(int nz, int rows) {
    const long cells = (long)nz * rows;
    return cells <= (long)RB * R64_MAX_U ? (int)((cells + RB - 1) / RB) : 0;
}
__host__ __device__ constexpr size_t r64_scratch() { return (sizeof(TeamLds) + 15) / 16 * 16; }
static size_t r64_lds(int nz, int rows, int lds_rows, int halo_rows) {
    return r64_scratch() + ((size_t)lds_rows * nz + 2) * sizeof(double) +
           (size_t)halo_rows * nz * (sizeof(int2) + sizeof(double)) +
           (size_t)r64_slots(nz, rows) * RB * sizeof(double);
}

// From six cells per thread on, x is in LDS and each cell's work is a block
// of its own, skipped where the rectangle has no such cells: run together,
// the cells' loads and divisions would not fit the 256 registers (eight
// cells per thread spilled 158).
constexpr int R64_TIGHT = 6;
#define R64_CELL(u) if (U < R64_TIGHT || (u) < nu)

template <int U>
__global__ __launch_bounds__(RB, 2) void k64_resident(R64Args g) {
    extern __shared__ double r64_dyn[];
    TeamLds& S = *reinterpret_cast<TeamLds*>(r64_dyn);
    double* P = r64_dyn + r64_scratch() / sizeof(double) + 1;
    const int tid = threadIdx.x;
    Team t;
    int team;
    if (!res_place(g.L, team, t.m, t.T, t.slots)) return;
    if (!res_gate(g.L, S)) return;
    t.gate = g.L.gate;
    t.tag = uniform(g.L.gate[1]);
    const Cg64Args& a = g.a;

    const int it_end = uniform(g.L.team_begin[team + 1]);
    for (int item = uniform(g.L.team_begin[team]); item < it_end; ++item) {
        const ResItem I = uniform(g.L.items[item]);
        const int s = I.sys, nz = I.nz;
        CgSlot st = uniform(a.slot[1][s]);
        if (st.done) continue;
        const CgConst K = uniform(a.cst[s]);
        const bool member = t.m < I.pr * I.pth;   // the others only join the sums
        const ResRect R = res_rect(I, member ? t.m : 0);
        const ResBox X(R, I.pth);
        const int rows = member ? X.rows() : 0, cells = rows * nz;
        const int nhalo = member ? X.halo_rows(R, I.nr) * nz : 0;
        const int plen = X.lds_rows() * nz;
        int2* H = reinterpret_cast<int2*>(P + plen + 1);
        const int nu = (cells + RB - 1) / RB;
        const float inv_nz = 1.0f / (float)nz, inv_bj = 1.0f / (float)X.bj;
        const int dr = X.pitch * nz;               // LDS distance of the r neighbours
        const int wrap = (X.bj - 1) * nz;          // theta neighbours across an uncut ring
        double* Zh = reinterpret_cast<double*>(H + nhalo);
        double* zx = g.zx + I.xoff;
        int mem[4];
        res_neighbours(I, t.m, mem);

        __syncthreads();                           // the previous item's p is no longer read
        for (int q = tid - 1; q < plen + 1; q += RB) P[q] = 0.0;
        for (int h = tid; h < nhalo; h += RB) {
            int hr, k, grow, lrow;
            row_of(h, nz, inv_nz, hr, k);
            X.halo(hr, R, I.nr, I.nth, grow, lrow);
            H[h] = make_int2(grow * nz + k, lrow * nz + k);
        }

        // the thread's cells: c = tid + u*RB of the rectangle's rows in order
        double cf[U][7], xr[U < R64_TIGHT ? U : 1], r[U], z[U];
        double* XL = Zh + nhalo;                    // x, with R64_TIGHT cells or more
        auto x = [&](int u) -> double& { return U < R64_TIGHT ? xr[U < R64_TIGHT ? u : 0] : XL[tid + u * RB]; };
        int lo[U], go[U];                           // its place in p, in the system
        unsigned flag[U];
        enum { F_CELL = 1, F_EDGE = 2, F_B = 4, F_T = 8, F_S = 16, F_N = 32 };
        auto cell = [&](int u, int& li, int& lj, int& k) {
            const int c = tid + u * RB;
            int row;
            row_of(c < cells ? c : 0, nz, inv_nz, row, k);
            row_of(row, X.bj, inv_bj, li, lj);
            return c < cells;
        };
#pragma unroll
        for (int u = 0; u < U; ++u) {
            int li, lj, k;
            const bool ok = cell(u, li, lj, k);
            lo[u] = X.lds_row(li, lj) * nz + k;
            flag[u] = 0;
            if (ok) {
                const bool edge = (li == 0 && R.i0 > 0) || (li == X.bi - 1 && R.i1 < I.nr) ||
                                  (X.hs && (lj == 0 || lj == X.bj - 1));
                flag[u] = F_CELL | (edge ? F_EDGE : 0) | (k > 0 ? F_B : 0) | (k < nz - 1 ? F_T : 0) |
                          (!X.hs && lj == 0 ? F_S : 0) | (!X.hs && lj == X.bj - 1 ? F_N : 0);
            }
            go[u] = ((R.i0 + li) * I.nth + R.j0 + lj) * nz + k;
            const long o = I.off + go[u];
            cf[u][0] = ok ? a.aP[o] : 1.0;
            cf[u][1] = ok ? a.aW[o] : 0.0;
            cf[u][2] = ok ? a.aE[o] : 0.0;
            cf[u][3] = ok ? a.aS[o] : 0.0;
            cf[u][4] = ok ? a.aN[o] : 0.0;
            cf[u][5] = ok ? a.aB[o] : 0.0;
            cf[u][6] = ok ? a.aT[o] : 0.0;
        }
        // q = A p of the thread's cell u, p from LDS
        auto apply = [&](int u, double pc) {
            const double* p = P + fresh(lo[u]);
            const unsigned f = (unsigned)fresh((int)flag[u]);
            const double pW = p[-dr], pE = p[dr];
            const double pS = p[(f & F_S) ? wrap : -nz], pN = p[(f & F_N) ? -wrap : nz];
            const double b = p[-1], tt = p[1];
            const double pB = (f & F_B) ? b : 0.0, pT = (f & F_T) ? tt : 0.0;
            return cf[u][0] * pc - cf[u][1] * pW - cf[u][2] * pE - cf[u][3] * pS - cf[u][4] * pN - cf[u][5] * pB -
                   cf[u][6] * pT;
        };
        // edge rows of z for the neighbours
        auto publish = [&]() {
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (fresh((int)flag[u]) & F_EDGE) st_agent_d(zx + fresh(go[u]), z[u]);
        };
        // the neighbours' edge rows, into Zh
        auto fetch = [&](int w, int n) {
            constexpr int Q = U >= R64_TIGHT ? 4 : 8;
            for (int h0 = w * 64 + (tid & 63), first = 1; first || h0 < nhalo; h0 += Q * 64 * n, first = 0) {
                int src[Q];
#pragma unroll
                for (int q = 0; q < Q; ++q) {
                    const int h = h0 + q * 64 * n;
                    src[q] = h < nhalo ? H[h].x : 0;
                }
                if (first) wait_members(t, S, mem);
                double v[Q];
#pragma unroll
                for (int q = 0; q < Q; ++q) v[q] = ld_agent_d(zx + src[q]);
#pragma unroll
                for (int q = 0; q < Q; ++q)
                    if (h0 + q * 64 * n < nhalo) Zh[h0 + q * 64 * n] = v[q];
            }
        };
        __syncthreads();

        bool alive = true;
        int iters = 0;
        if (st.bnorm < 0.0) {
            // r = Su - A x0 (src/mod_solver_3d.f90:509-530), x0 in P meanwhile
            for (int h = tid; h < nhalo; h += RB) P[H[h].y] = a.x0[I.off + H[h].x];
            double su[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const bool ok = flag[u] & F_CELL;
                const long o = I.off + go[u];
                const double x0 = ok ? a.x0[o] : 0.0;
                R64_CELL(u) x(u) = x0;
                su[u] = ok ? a.b[o] : 0.0;
                r[u] = ok ? a.fold[o] : 0.0;
                if (ok) P[lo[u]] = x0;
            }
            __syncthreads();
            double acc[3] = {0.0, 0.0, 0.0};
#pragma unroll
            for (int u = 0; u < U; ++u) R64_CELL(u) {
                const bool ok = flag[u] & F_CELL;
                const double ax = apply(u, P[lo[u]]);
                const double rr = su[u] - (ax - r[u]);
                const double zz = rr / fmax(fabs(cf[u][0]), SMALL);
                r[u] = ok ? rr : 0.0;
                z[u] = ok ? zz : 0.0;
                acc[0] += r[u] * r[u];
                acc[1] += r[u] * z[u];
                acc[2] += su[u] * su[u];
            }
            publish();
            alive = team_sum<3>(t, acc, S, true, fetch);   // its barriers: P is read
            for (int h = tid; h < nhalo; h += RB) P[H[h].y] = 0.0;
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (flag[u] & F_CELL) P[lo[u]] = 0.0;
            st.bnorm = sqrt(acc[2]);
            st.n_iter = 0;
            st.it = 1;
            st.beta = 0.0;
            if (st.bnorm < SMALL) {
                st.residual = 0.0;
                st.done = 1;
                st.status = EAFP_STOP_ZERO_RHS;
            } else {
                st.residual = sqrt(acc[0]) / st.bnorm;
                st.rz = acc[1];
                if (K.max_iter <= 0) {
                    st.done = 1;
                    st.status = EAFP_STOP_MAX_ITER;
                }
            }
        } else {
            // the launch before left the state in memory
            for (int h = tid; h < nhalo; h += RB) {
                P[H[h].y] = a.p[0][I.off + H[h].x];
                Zh[h] = a.z[I.off + H[h].x];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const bool ok = flag[u] & F_CELL;
                const long o = I.off + go[u];
                R64_CELL(u) x(u) = ok ? a.x[o] : 0.0;
                r[u] = ok ? a.r[o] : 0.0;
                z[u] = ok ? a.z[o] : 0.0;
                if (ok) P[lo[u]] = a.p[0][o];
            }
        }

        while (alive && !st.done && iters < g.iters) {
            ++iters;
            // p = z + beta p, own rows and halo rows (each element by one thread)
            const double beta = st.beta;
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (flag[u] & F_CELL) P[lo[u]] = z[u] + beta * P[lo[u]];
            for (int h = tid; h < nhalo; h += RB) {
                const int dst = H[h].y;
                P[dst] = Zh[h] + beta * P[dst];
            }
            __syncthreads();
            double acc1[1] = {0.0};
#pragma unroll
            for (int u = 0; u < U; ++u) R64_CELL(u) {
                const double pc = P[lo[u]];
                z[u] = (flag[u] & F_CELL) ? apply(u, pc) : 0.0;   // q, until z is formed again
                acc1[0] += pc * z[u];
                formed(z[u]);
                formed(acc1[0]);
            }
            alive = team_sum<1>(t, acc1, S, false, NoAside());
            if (!alive) break;
            const double pq = acc1[0];
            if (fabs(pq) < SMALL) {
                st.done = 1;
                st.status = EAFP_STOP_BREAKDOWN;
                break;
            }
            const double alpha = st.rz / pq;
            st.alpha = alpha;
            double acc[2] = {0.0, 0.0};
#pragma unroll
            for (int u = 0; u < U; ++u) R64_CELL(u) {
                const bool ok = flag[u] & F_CELL;
                const double rr = r[u] - alpha * z[u];
                const double zz = rr / fmax(fabs(cf[u][0]), SMALL);
                x(u) += alpha * P[lo[u]];
                r[u] = ok ? rr : 0.0;
                z[u] = ok ? zz : 0.0;
                acc[0] += r[u] * r[u];
                acc[1] += r[u] * z[u];
                formed(x(u));
                formed(r[u]);
                formed(z[u]);
                formed(acc[0]);
                formed(acc[1]);
            }
            publish();
            alive = team_sum<2>(t, acc, S, true, fetch);
            if (!alive) break;
            st.residual = sqrt(acc[0]) / st.bnorm;
            st.n_iter = st.it;
            if (st.residual < K.tol) {
                st.done = 1;
                st.status = EAFP_STOP_CONVERGED;
            } else if (st.it >= K.max_iter) {
                st.done = 1;
                st.status = EAFP_STOP_MAX_ITER;
            } else {
                st.beta = acc[1] / fmax(st.rz, SMALL);
                st.rz = acc[1];
            }
            ++st.it;
        }
        if (!alive) return;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (!(flag[u] & F_CELL)) continue;
            const long o = I.off + go[u];
            a.x[o] = x(u);
            if (!st.done) {
                a.r[o] = r[u];
                a.z[o] = z[u];
                a.p[0][o] = P[lo[u]];
            }
        }
        if (t.m == 0 && tid == 0) store_state(&a.slot[1][s], st);
    }
}

static const ResLimits kLimits = {
    R64_MAX_U, r64_slots, r64_lds,
    // T = 1, 2, 4, 8, 16, 32, 64, 128, 256, fitted to iterations measured at 1 to
    // 5 cells per thread: 3.75 us (T 16, 1 cell), 4.2 (8, 2), 5.0 (2, 5), 6.75
    // (32, 5), 6.45 (64, 3), 6.3 (128, 3), 9.9 (256, 5)
    {1.2f, 3.4f, 3.4f, 3.4f, 3.4f, 4.1f, 4.8f, 5.1f, 7.3f},
    0.5f,
};
static int r64_xpitch(int nz) { return nz; }

// The FP64 batch's resident plan (not ok: the batch streams).
ResPlan plan_resident64(const Batch& B) { return plan_resident(B.geom, kLimits, r64_xpitch); }

template <int U>
static int launch_u(const R64Args& g, int blocks, size_t lds, hipStream_t st) {
    EAFP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(&k64_resident<U>),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    k64_resident<U><<<blocks, RB, lds, st>>>(g);
    EAFP_TRY(hipGetLastError());
    return EAFP_OK;
}

// Fresh slots and the solve's constants for every system; opens the first
// launch's gate.
__global__ void k64_res_start(CgSlot* slot, CgConst* cst, int nsys, double tol, int max_iter, unsigned* gate,
                              unsigned tag) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s == 0) {
        gate[0] = 0;
        gate[1] = tag;
    }
    if (s >= nsys) return;
    CgSlot n{};
    n.bnorm = -1.0;
    slot[s] = n;
    cst[s] = CgConst{tol, max_iter, 0};
}

static long launch_tags(const ResDevice& D, int iters) { return (long)D.plan.max_items * (2L * iters + 2); }

int start_resident64(Batch& B, ResDevice& D, CgSlot* slot, CgConst* cst, double tol, int max_iter, int iters) {
    unsigned tag = 0;
    EAFP_TRY_RC(D.take_tags(launch_tags(D, iters), B.stream, &tag));
    k64_res_start<<<(B.nsys + 255) / 256, 256, 0, B.stream>>>(slot, cst, B.nsys, tol, max_iter, D.gate.p, tag);
    EAFP_TRY(hipGetLastError());
    return EAFP_OK;
}

// The slots and the gate word, straight into the host's memory: one launch
// instead of two copies.
__global__ void k64_res_report(const CgSlot* slot, const unsigned* gate, int nsys, CgSlot* out, unsigned* gate_out) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s == 0) *gate_out = gate[0];
    if (s < nsys) out[s] = slot[s];
}

int report_resident64(Batch& B, ResDevice& D, const CgSlot* slot, CgSlot* slots_host, unsigned* gate_host) {
    CgSlot* out = nullptr;
    unsigned* gate_out = nullptr;
    EAFP_TRY(hipHostGetDevicePointer((void**)&out, slots_host, 0));
    EAFP_TRY(hipHostGetDevicePointer((void**)&gate_out, gate_host, 0));
    k64_res_report<<<(B.nsys + 255) / 256, 256, 0, B.stream>>>(slot, D.gate.p, B.nsys, out, gate_out);
    EAFP_TRY(hipGetLastError());
    return EAFP_OK;
}

// One launch: at most `iters` iterations of every unfinished system.  The
// slots, x0, b, fold and the coefficients are the streaming kernels' own.
// `first`: start_resident64 has opened the gate.
int launch_resident64(Batch& B, ResDevice& D, const Cg64Args& a, int iters, bool first) {
    const ResPlan& p = D.plan;
    ++D.launches;
    if (!first) EAFP_TRY_RC(D.arm(launch_tags(D, iters), B.stream));
    R64Args g{};
    g.a = a;
    g.L = D.launch();
    g.zx = a.q;
    g.iters = iters;
    const size_t lds = std::max(p.lds, p.members > 0 ? (size_t)RES_LDS_ALONE : (size_t)0);
    switch (p.slots) {
        case 1: return launch_u<1>(g, p.blocks, lds, B.stream);
        case 2: return launch_u<2>(g, p.blocks, lds, B.stream);
        case 3: return launch_u<3>(g, p.blocks, lds, B.stream);
        case 4: return launch_u<4>(g, p.blocks, lds, B.stream);
        case 5: return launch_u<5>(g, p.blocks, lds, B.stream);
        case 6: return launch_u<6>(g, p.blocks, lds, B.stream);
        default: return launch_u<8>(g, p.blocks, lds, B.stream);
    }
}

}  // namespace eafp
