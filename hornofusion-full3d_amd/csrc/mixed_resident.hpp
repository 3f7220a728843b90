// mixed_resident.hpp -- the inner iterations of the mixed solver with the
// systems' vectors kept on chip.
//
// One launch runs the `interval` inner iterations between two refinement
// steps for every system, instead of 2*interval launches of the streaming
// kernels (mixed.hip) that move 56 bytes per cell and iteration with BF16
// weights.  A team of work-groups (resident.hpp) holds a system: a thread
// keeps r, d and q (or z) of its cells in registers, p of the rectangle and
// its halo rows is in LDS, and z crosses to the neighbours by its edge rows.
// The weights and the preconditioner (12 bytes per cell with BF16) are read
// again in every iteration, from the L2s and the memory-side cache, which
// hold them: 18,900 cells per work-group would not fit the registers with
// them.
//
// A lane holds CQ quads, 4*CQ consecutive cells, of a z-row; nl lanes make a
// row and a wave takes as many whole rows as fit.  The z neighbours and the
// line preconditioner's recurrences then stay inside a wave.  M^-1 is two
// scans of affine maps over the wave's lanes (row shifts, then the three row
// ends): a row's first l is 0, so its first map forgets what comes before,
// and several rows per wave need no masks.
//
// The arithmetic per cell is k_mspmv's and k_mupdate_line's; the order of the
// sums differs.
//
// What bounds it: 604,800 cells on 256 work-groups take 8.4 us per BF16 z-line
// iteration (17.5 streaming), the waves waiting 74 % of it for the two sums and
// the exchange of z and the vector ALU busy 22 %; eight such systems at once,
// 32 work-groups each, take 15.9 us (50 streaming), the vector ALU busy 55 % of
// it (261 instructions per quad).  4.8 million cells on 256 work-groups take
// 21.4 us (60 streaming), the vector ALU busy 36 %; 69 MB per iteration come
// from beyond the L2s, 3.2 TB/s over the whole of it.
#pragma once
#include "mixed.hpp"
#include "resident_plan.hpp"

namespace eafp {

struct RMxArgs {
    MxArgs a;
    ResLaunch L;
    float* xz;           // exchange buffer, rows of nl*CQ quads
    int interval;
};

__host__ __device__ __forceinline__ int rmx_lanes(int nz, int cq) { return (nz + 4 * cq - 1) / (4 * cq); }
__host__ __device__ constexpr size_t rmx_scratch() { return (sizeof(TeamLds) + 15) / 16 * 16; }

// Four weights at any cell: a quad begins anywhere in the arena when nz is not
// a multiple of 4.
template <int F>
struct WQuad;
template <>
struct WQuad<EAFP_COEF_FP32> {
    F4 v;
    __device__ __forceinline__ void load(const void* w, const float*, unsigned o) {
        __builtin_memcpy(&v, (const float*)w + o, 16);
    }
    __device__ __forceinline__ float get(int k) const { return v.v[k]; }
};
template <>
struct WQuad<EAFP_COEF_BF16> {
    unsigned w2[2];
    __device__ __forceinline__ void load(const void* w, const float*, unsigned o) {
        __builtin_memcpy(w2, (const unsigned short*)w + o, 8);
    }
    __device__ __forceinline__ float get(int k) const {
        return __uint_as_float((k & 1) ? w2[k >> 1] & 0xFFFF0000u : w2[k >> 1] << 16);
    }
};
template <>
struct WQuad<EAFP_COEF_FP16> {
    _Float16 h[4];
    F4 s;
    __device__ __forceinline__ void load(const void* w, const float* sc, unsigned o) {
        __builtin_memcpy(h, (const _Float16*)w + o, 8);
        __builtin_memcpy(&s, sc + o, 16);
    }
    __device__ __forceinline__ float get(int k) const { return (float)h[k] * s.v[k]; }
};

// a where bit `n` of f is set, else b: a sign-extended bit and a bitwise
// select (a compare and a conditional move wait for each other, 17 cycles
// against 9).
template <int BIT>
__device__ __forceinline__ int pick(unsigned f, int a, int b) {
    constexpr int n = __builtin_ctz(BIT);
    const int m = (int)(f << (31 - n)) >> 31;
    return (a & m) | (b & ~m);
}

// The six weight pieces of a lane's quads, loaded one slot ahead of their use.
template <int F, int CQ>
struct WSet {
    WQuad<F> wr[CQ], wrm[CQ], wt[CQ], wtm[CQ], wz[CQ], e[CQ];
};

// Lane shifts over the whole wave; the end lane gets 0.
__device__ __forceinline__ float from_prev_lane(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xF, 0xF, true));   // wave_shr:1
}
__device__ __forceinline__ float from_next_lane(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xF, 0xF, true));   // wave_shl:1
}
__device__ __forceinline__ float readlane_f(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// The value that flows into each lane: lane n's map y -> A y + B applied to
// what flows into it flows into lane n+1 (UP) or n-1; 0 flows into the end.
// Steps of 1, 2, 4, 8 lanes inside the rows of 16, two instructions each (a
// lane without a source adds 0 to B and keeps A); then the row ends.  The
// shifted operand is part of the multiply: as moves of their own, each step
// took 40 cycles of the wave instead of 12.  A shifted operand needs two
// wait states after its write, which the other chain and the s_nop make.
template <bool UP>
__device__ __forceinline__ float scan_lanes(float A, float B) {
    if (UP) {
        asm("s_nop 1\n\t"
            "v_fmac_f32_dpp %1, %1, %0 row_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
            "v_mul_f32_dpp %0, %0, %0 row_shr:1 row_mask:0xf bank_mask:0xf\n\t"
            "s_nop 0\n\t"
            "v_fmac_f32_dpp %1, %1, %0 row_shr:2 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
            "v_mul_f32_dpp %0, %0, %0 row_shr:2 row_mask:0xf bank_mask:0xf\n\t"
            "s_nop 0\n\t"
            "v_fmac_f32_dpp %1, %1, %0 row_shr:4 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
            "v_mul_f32_dpp %0, %0, %0 row_shr:4 row_mask:0xf bank_mask:0xf\n\t"
            "s_nop 0\n\t"
            "v_fmac_f32_dpp %1, %1, %0 row_shr:8 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
            "v_mul_f32_dpp %0, %0, %0 row_shr:8 row_mask:0xf bank_mask:0xf\n\t"
            // the end of rows 0 and 2 into rows 1 and 3, then of row 1 into rows 2 and 3
            "s_nop 0\n\t"
            "v_fmac_f32_dpp %1, %1, %0 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
            "v_mul_f32_dpp %0, %0, %0 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
            "s_nop 0\n\t"
            "v_fmac_f32_dpp %1, %1, %0 row_bcast:31 row_mask:0xc bank_mask:0xf"
            : "+v"(A), "+v"(B));
        return from_prev_lane(B);
    }
    asm("s_nop 1\n\t"
        "v_fmac_f32_dpp %1, %1, %0 row_shl:1 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
        "v_mul_f32_dpp %0, %0, %0 row_shl:1 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 0\n\t"
        "v_fmac_f32_dpp %1, %1, %0 row_shl:2 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
        "v_mul_f32_dpp %0, %0, %0 row_shl:2 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 0\n\t"
        "v_fmac_f32_dpp %1, %1, %0 row_shl:4 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
        "v_mul_f32_dpp %0, %0, %0 row_shl:4 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 0\n\t"
        "v_fmac_f32_dpp %1, %1, %0 row_shl:8 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
        "v_mul_f32_dpp %0, %0, %0 row_shl:8 row_mask:0xf bank_mask:0xf"
        : "+v"(A), "+v"(B));
    // what flows out of the first lanes of rows 3, 2 and 1 flows into rows 2, 1 and 0
    const float x2 = readlane_f(B, 48);
    const float x1 = readlane_f(A, 32) * x2 + readlane_f(B, 32);
    const float x0 = readlane_f(A, 16) * x1 + readlane_f(B, 16);
    asm("s_nop 1\n\t"
        "v_fmac_f32_dpp %0, %1, %2 quad_perm:[0,1,2,3] row_mask:0x4 bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %3 quad_perm:[0,1,2,3] row_mask:0x2 bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %4 quad_perm:[0,1,2,3] row_mask:0x1 bank_mask:0xf"
        : "+v"(B)
        : "v"(A), "v"(x2), "v"(x1), "v"(x0));
    return from_next_lane(B);
}

// z = M^-1 r for the wave's rows: L y = r upwards, L^T z = y/d downwards.
template <int NC>
__device__ __forceinline__ void line_solve_lanes(const float (&r)[NC], const float (&l)[NC], const float (&iv)[NC],
                                                 float (&z)[NC]) {
    float A = -l[0], B = r[0];
#pragma unroll
    for (int k = 1; k < NC; ++k) {
        A = -l[k] * A;
        B = r[k] - l[k] * B;
    }
    float y = scan_lanes<true>(A, B);
    float u[NC];
#pragma unroll
    for (int k = 0; k < NC; ++k) {
        y = r[k] - l[k] * y;
        u[k] = y * iv[k];
    }
    const float ln = from_next_lane(l[0]);   // 0 in a row's last lane: the next row's first l
    A = -ln;
    B = u[NC - 1];
#pragma unroll
    for (int k = NC - 2; k >= 0; --k) {
        A = -l[k + 1] * A;
        B = u[k] - l[k + 1] * B;
    }
    const float zin = scan_lanes<false>(A, B);
    z[NC - 1] = u[NC - 1] - ln * zin;
#pragma unroll
    for (int k = NC - 2; k >= 0; --k) z[k] = u[k] - l[k + 1] * z[k + 1];
}

template <int F, bool LINE, int CQ, int U>
__global__ __launch_bounds__(RB, 2) void k_mresident(RMxArgs g) {
    extern __shared__ float4 rmx_dyn[];
    TeamLds& S = *reinterpret_cast<TeamLds*>(rmx_dyn);
    float4* P = rmx_dyn + rmx_scratch() / sizeof(float4);
    constexpr int NC = 4 * CQ;
    // the weights of the next slot are loaded ahead, unless 32-bit weights (or
    // 16-bit ones with their scales) leave no registers for them
    constexpr bool AHEAD = F == EAFP_COEF_BF16 || U * CQ <= 6;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    Team t;
    int team;
    if (!res_place(g.L, team, t.m, t.T, t.slots)) return;
    if (!res_gate(g.L, S)) return;
    t.gate = g.L.gate;
    t.tag = uniform(g.L.gate[1]);
    const MxArgs& a = g.a;

    const int it_end = uniform(g.L.team_begin[team + 1]);
    for (int item = uniform(g.L.team_begin[team]); item < it_end; ++item) {
        const ResItem I = uniform(g.L.items[item]);
        const int s = I.sys, nz = I.nz;
        MxDyn D = uniform(a.dyn[1][s]);
        if (D.done || D.broken) continue;
        const bool member = t.m < I.pr * I.pth;   // the others only join the sums
        const ResRect R = res_rect(I, member ? t.m : 0);
        const ResBox X(R, I.pth);
        const int rows = member ? X.rows() : 0;
        const int nl = rmx_lanes(nz, CQ), nq = nl * CQ, lpw = 64 / nl;   // quads of a row in LDS; rows per wave
        const int nhalo = member ? X.halo_rows(R, I.nr) * nq : 0;
        const int plen = X.lds_rows() * nq;
        float4* Zh = P + plen;
        int2* H = reinterpret_cast<int2*>(Zh + nhalo);   // halo quads: place in the exchange buffer, in P
        // this wave's slots: the others hold no row and are left out of the
        // stencil and the update (worked through with zeros, 96 uneven systems
        // took 33.1 ms instead of 31.6, one of 60x120x84 13.5 instead of 13.2)
        const int per = RW * lpw, first_row = __builtin_amdgcn_readfirstlane(wid) * lpw;
        const int nu = rows > first_row ? (rows - first_row + per - 1) / per : 0;
        const float inv_nq = 1.0f / (float)nq, inv_bj = 1.0f / (float)X.bj;
        const int dr = X.pitch * nq, wrap = (X.bj - 1) * nq;
        int mem[4];
        res_neighbours(I, t.m, mem);
        const auto rs = __builtin_amdgcn_make_buffer_rsrc(g.xz + I.xoff, 0, I.nr * I.nth * nq * 16, 0x00020000);
        constexpr int SC1 = 16;                    // the accesses' scope: the agent
        // the operand from the system's first cell on; `pad`: the zeros past the arena
        const unsigned pad = (unsigned)(a.sink - I.off), span = (unsigned)(I.nth * nz);
        const bool whole = nz % NC == 0;           // no lane's cells end before its quads do
        const char* w0 = (const char*)a.w[0] + I.off * (F == EAFP_COEF_FP32 ? 4 : 2);
        const char* w1 = (const char*)a.w[1] + I.off * (F == EAFP_COEF_FP32 ? 4 : 2);
        const char* w2 = (const char*)a.w[2] + I.off * (F == EAFP_COEF_FP32 ? 4 : 2);
        const char* we = (const char*)a.e + I.off * (F == EAFP_COEF_FP32 ? 4 : 2);
        const float* sc = F == EAFP_COEF_FP16 ? a.scale + I.off : nullptr;
        const float* pre = (LINE ? (const float*)a.fac : a.dinv) + I.off;

        // the lane's place in its rows (a lane past the wave's rows stands at
        // the beginning of a row it does not own)
        const int row_in_wave = lane / nl;
        const bool in_row = row_in_wave < lpw;
        const int j = in_row ? lane - row_in_wave * nl : 0;
        const int k0 = j * NC;
        // rows in order: wave by wave, slot by slot
        float r[U][NC], d[U][NC], q[U][NC];
        int lo[U], go[U];                          // first quad in LDS; first cell in the system, or the pad's
        unsigned flag[U];
        enum { F_CELL = 1, F_EDGE = 2, F_W = 4, F_S = 8, F_N = 16, F_J0 = 32 };

        __syncthreads();                           // the previous item's p is no longer read
        for (int h = tid; h < plen; h += RB) P[h] = make_float4(0.f, 0.f, 0.f, 0.f);
        __syncthreads();
        float* Pf = reinterpret_cast<float*>(P);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int n = (u * RW + wid) * lpw + row_in_wave;
            const bool ok = in_row && n < rows;
            int li, lj;
            row_of(ok ? n : 0, X.bj, inv_bj, li, lj);
            const int gi = R.i0 + li, gj = R.j0 + lj;
            const bool edge = (li == 0 && R.i0 > 0) || (li == X.bi - 1 && R.i1 < I.nr) ||
                              (X.hs && (lj == 0 || lj == X.bj - 1));
            flag[u] = (ok ? F_CELL : 0) | (ok && edge ? F_EDGE : 0) | (gi > 0 || !ok ? F_W : 0) |
                      (!X.hs && lj == 0 ? F_S : 0) | (!X.hs && lj == X.bj - 1 ? F_N : 0) | (ok && gj == 0 ? F_J0 : 0);
            lo[u] = X.lds_row(li, lj) * nq + j * CQ;
            go[u] = ok ? (gi * I.nth + gj) * nz + k0 : (int)pad;
            const long o = I.off + go[u];
#pragma unroll
            for (int k = 0; k < NC; ++k) {
                const bool c = ok && k0 + k < nz;
                r[u][k] = c ? a.r[o + k] : 0.f;
                q[u][k] = c ? a.z[o + k] : 0.f;     // z, until the stencil leaves q here
                d[u][k] = 0.f;
                if (c) Pf[4 * lo[u] + k] = a.p[0][o + k];
            }
        }
        for (int h = tid; h < nhalo; h += RB) {
            int hr, hq, grow, lrow;
            row_of(h, nq, inv_nq, hr, hq);
            X.halo(hr, R, I.nr, I.nth, grow, lrow);
            const long o = I.off + (long)grow * nz + 4 * hq;
            float zv[4], pv[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const bool c = 4 * hq + k < nz;
                zv[k] = c ? a.z[o + k] : 0.f;
                pv[k] = c ? a.p[0][o + k] : 0.f;
            }
            H[h] = make_int2((grow * nq + hq) * 16, lrow * nq + hq);
            Zh[h] = make_float4(zv[0], zv[1], zv[2], zv[3]);
            P[lrow * nq + hq] = make_float4(pv[0], pv[1], pv[2], pv[3]);
        }
        // edge rows of z for the neighbours, and theirs into Zh
        auto publish = [&]() {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int f = fresh((int)flag[u]);
                if (f & F_EDGE) {
                    const int o = fresh(go[u]);
                    const int gq = whole ? o >> 2 : (o - k0) / nz * nq + j * CQ;
#pragma unroll
                    for (int c = 0; c < CQ; ++c) {
                        res_u4 v;
                        v.x = __float_as_uint(q[u][4 * c]);
                        v.y = __float_as_uint(q[u][4 * c + 1]);
                        v.z = __float_as_uint(q[u][4 * c + 2]);
                        v.w = __float_as_uint(q[u][4 * c + 3]);
                        __builtin_amdgcn_raw_buffer_store_b128(v, rs, (gq + c) * 16, 0, SC1);
                    }
                }
            }
        };
        auto fetch = [&](int w, int n) {
            constexpr int Q = 4;
            for (int h0 = w * 64 + lane, first = 1; first || h0 < nhalo; h0 += Q * 64 * n, first = 0) {
                int src[Q];
#pragma unroll
                for (int c = 0; c < Q; ++c) {
                    const int h = h0 + c * 64 * n;
                    src[c] = h < nhalo ? H[h].x : 0;
                }
                if (first) wait_members(t, S, mem);
                res_u4 v[Q];
#pragma unroll
                for (int c = 0; c < Q; ++c) v[c] = __builtin_amdgcn_raw_buffer_load_b128(rs, src[c], 0, SC1);
#pragma unroll
                for (int c = 0; c < Q; ++c) {
                    const int h = h0 + c * 64 * n;
                    if (h < nhalo)
                        Zh[h] = make_float4(__uint_as_float(v[c].x), __uint_as_float(v[c].y), __uint_as_float(v[c].z),
                                            __uint_as_float(v[c].w));
                }
            }
        };
        const int eW = (int)span * (I.nr - 1), eS = (int)span - nz;
        // A slot without a row stands at the pad, inside the arena for its W and
        // S weights too; its q is cleared and its z comes out 0.  Beyond the inner
        // wall stands the outer wall's row of w_r, whose weights are 0.
        auto load_w = [&](int u, WSet<F, CQ>& w) {
            const unsigned f = (unsigned)fresh((int)flag[u]), o = (unsigned)fresh(go[u]);
            const unsigned oW = o + (unsigned)pick<F_W>(f, -(int)span, eW), oS = o + (unsigned)pick<F_J0>(f, eS, -nz);
#pragma unroll
            for (int c = 0; c < CQ; ++c) {
                w.wr[c].load(w0, sc, o + 4 * c);
                w.wrm[c].load(w0, sc, oW + 4 * c);
                w.wt[c].load(w1, sc, o + 4 * c);
                w.wtm[c].load(w1, sc, oS + 4 * c);
                w.wz[c].load(w2, sc, o + 4 * c);
                w.e[c].load(we, sc, o + 4 * c);
            }
        };
        auto load_pre = [&](int u, F4 (&v)[CQ]) {
            const unsigned o = (unsigned)fresh(go[u]);
#pragma unroll
            for (int c = 0; c < CQ; ++c) __builtin_memcpy(&v[c], pre + o + 4 * c, 16);
        };

        double acc[1] = {0.0};
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int k = 0; k < NC; ++k) acc[0] += (double)r[u][k] * (double)q[u][k];
        bool alive = team_sum<1>(t, acc, S, false, NoAside());
        double rz = acc[0];

        for (int it = 0; alive && it < g.interval; ++it) {
            if (!(rz > 0.0)) {
                D.broken = 1;   // r.z lost positivity: wait for the next refinement step
                break;
            }
            D.beta = D.fresh ? 0.0 : rz / D.rz;
            D.rz = rz;
            D.fresh = 0;
            const float fb = (float)D.beta;
            WSet<F, CQ> w;
            if (AHEAD) load_w(0, w);
            // p = z + beta p, own rows and halo rows (each quad by one thread);
            // read several slots ahead of the writes
            constexpr int PG = U * CQ <= 6 ? U : 5;
#pragma unroll
            for (int u0 = 0; u0 < U; u0 += PG) {
                float4 v[PG][CQ];
#pragma unroll
                for (int u = u0; u < u0 + PG && u < U; ++u)
#pragma unroll
                    for (int c = 0; c < CQ; ++c) v[u - u0][c] = P[fresh(lo[u]) + c];
#pragma unroll
                for (int u = u0; u < u0 + PG && u < U; ++u) {
#pragma unroll
                    for (int c = 0; c < CQ; ++c) {
                        float4& x = v[u - u0][c];
                        x.x = q[u][4 * c] + fb * x.x;
                        x.y = q[u][4 * c + 1] + fb * x.y;
                        x.z = q[u][4 * c + 2] + fb * x.z;
                        x.w = q[u][4 * c + 3] + fb * x.w;
                    }
                    if (flag[u] & F_CELL)
#pragma unroll
                        for (int c = 0; c < CQ; ++c) P[lo[u] + c] = v[u - u0][c];
                }
            }
            for (int h = tid; h < nhalo; h += RB) {
                float4* p = P + H[h].y;
                const float4 z = Zh[h];
                float4 v = *p;
                v.x = z.x + fb * v.x;
                v.y = z.y + fb * v.y;
                v.z = z.z + fb * v.z;
                v.w = z.w + fb * v.w;
                *p = v;
            }
            __syncthreads();
            // q = A p (flux form)
            acc[0] = 0.0;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (u >= nu) continue;
                WSet<F, CQ> wn;
                if (AHEAD && u + 1 < U) load_w(u + 1 < U ? u + 1 : 0, wn);
                if (!AHEAD) load_w(u, w);
                const unsigned f = (unsigned)fresh((int)flag[u]);
                const float4* p = P + fresh(lo[u]);
                const int lS = pick<F_S>(f, wrap, -nq), lN = pick<F_N>(f, -wrap, nq);
                float pc[NC], y[NC], wz[NC];
#pragma unroll
                for (int c = 0; c < CQ; ++c) {
                    const float4 v = p[c], vE = p[dr + c], vW = p[c - dr], vN = p[lN + c], vS = p[lS + c];
                    const float vc[4] = {v.x, v.y, v.z, v.w}, ve[4] = {vE.x, vE.y, vE.z, vE.w},
                                vw[4] = {vW.x, vW.y, vW.z, vW.w}, vn[4] = {vN.x, vN.y, vN.z, vN.w},
                                vs[4] = {vS.x, vS.y, vS.z, vS.w};
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        pc[4 * c + k] = vc[k];
                        wz[4 * c + k] = w.wz[c].get(k);
                        float x = w.e[c].get(k) * vc[k];
                        x += w.wr[c].get(k) * (vc[k] - ve[k]);
                        x += w.wrm[c].get(k) * (vc[k] - vw[k]);
                        x += w.wt[c].get(k) * (vc[k] - vn[k]);
                        x += w.wtm[c].get(k) * (vc[k] - vs[k]);
                        y[4 * c + k] = x;
                    }
                }
                const float pT = from_next_lane(pc[0]), pB = from_prev_lane(pc[NC - 1]);
                const float wl = from_prev_lane(wz[NC - 1]);
                const float wB = j > 0 ? wl : 0.f;
#pragma unroll
                for (int k = 0; k < NC; ++k) {
                    y[k] += wz[k] * (pc[k] - (k + 1 < NC ? pc[k + 1 < NC ? k + 1 : 0] : pT));
                    y[k] += (k > 0 ? wz[k > 0 ? k - 1 : 0] : wB) * (pc[k] - (k > 0 ? pc[k > 0 ? k - 1 : 0] : pB));
                }
                const int live = pick<F_CELL>(f, -1, 0);
                if (!whole)
#pragma unroll
                    for (int k = 0; k < NC; ++k) y[k] = k0 + k < nz ? y[k] : 0.f;
#pragma unroll
                for (int k = 0; k < NC; ++k) {
                    q[u][k] = __int_as_float(__float_as_int(y[k]) & live);
                    acc[0] += (double)pc[k] * (double)q[u][k];
                    formed(q[u][k]);
                }
                formed(acc[0]);
                if (AHEAD && u + 1 < U) w = wn;
                __builtin_amdgcn_sched_barrier(0);   // the loads of one slot ahead, not of all
            }
            F4 fv[CQ];
            load_pre(0, fv);
            alive = team_sum<1>(t, acc, S, false, NoAside());
            if (!alive) break;
            const double pq = acc[0];
            if (!(fabs(pq) > SMALL)) {
                D.broken = 1;
                break;
            }
            D.alpha = D.rz / pq;
            D.total_inner += 1;
            const float fa = (float)D.alpha;
            // d += alpha p, r -= alpha q, z = M^-1 r
            acc[0] = 0.0;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (u >= nu) continue;
                F4 fn[CQ];
                if (u + 1 < U) load_pre(u + 1 < U ? u + 1 : 0, fn);
                const float4* p = P + fresh(lo[u]);
                float l[NC], iv[NC], zn[NC];
#pragma unroll
                for (int c = 0; c < CQ; ++c) {
                    const float4 v = p[c];
                    const float vc[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        d[u][4 * c + k] += fa * vc[k];
                        r[u][4 * c + k] -= fa * q[u][4 * c + k];
                        if (LINE) unpack_fac(fv[c].v[k], l[4 * c + k], iv[4 * c + k]);
                        else zn[4 * c + k] = fv[c].v[k] * r[u][4 * c + k];
                    }
                }
                if (LINE) line_solve_lanes<NC>(r[u], l, iv, zn);
#pragma unroll
                for (int k = 0; k < NC; ++k) {
                    // past the row's last cell r is 0 and dinv is another row's: z is 0 there
                    q[u][k] = zn[k];
                    acc[0] += (double)r[u][k] * (double)zn[k];
                    formed(q[u][k]);
                    formed(d[u][k]);
                }
                formed(acc[0]);
                if (u + 1 < U)
#pragma unroll
                    for (int c = 0; c < CQ; ++c) fv[c] = fn[c];
                __builtin_amdgcn_sched_barrier(0);
            }
            if (it + 1 == g.interval) break;   // the refinement step replaces r and z
            publish();
            alive = team_sum<1>(t, acc, S, true, fetch);
            rz = acc[0];
        }
        if (!alive) return;
        // d and p for the refinement step, and the state
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (!(flag[u] & F_CELL)) continue;
            const long o = I.off + go[u];
#pragma unroll
            for (int k = 0; k < NC; ++k)
                if (k0 + k < nz) {
                    a.d[o + k] = d[u][k];
                    a.p[0][o + k] = Pf[4 * lo[u] + k];
                }
        }
        if (t.m == 0 && tid == 0) store_state(&a.dyn[1][s], D);
    }
}

template <int F, bool LINE, int CQ, int U>
int launch_rmx(const RMxArgs& g, int blocks, size_t lds, hipStream_t st) {
    k_mresident<F, LINE, CQ, U><<<blocks, RB, lds, st>>>(g);
    return (int)hipGetLastError();
}
template <int F, bool LINE, int CQ, int U>
int prepare_rmx() {
    return (int)hipFuncSetAttribute(reinterpret_cast<const void*>(&k_mresident<F, LINE, CQ, U>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, RES_LDS);
}

// The kernel for `slots` rows per wave and lane: the next size there is.
#define EAFP_RMX_DISPATCH(fn, ...)                                                          \
    if (cq == 1) {                                                                          \
        if (slots <= 1) return line ? fn<F, true, 1, 1>(__VA_ARGS__) : fn<F, false, 1, 1>(__VA_ARGS__);   \
        if (slots <= 2) return line ? fn<F, true, 1, 2>(__VA_ARGS__) : fn<F, false, 1, 2>(__VA_ARGS__);   \
        if (slots <= 3) return line ? fn<F, true, 1, 3>(__VA_ARGS__) : fn<F, false, 1, 3>(__VA_ARGS__);   \
        if (slots <= 4) return line ? fn<F, true, 1, 4>(__VA_ARGS__) : fn<F, false, 1, 4>(__VA_ARGS__);   \
        if (slots <= 6) return line ? fn<F, true, 1, 6>(__VA_ARGS__) : fn<F, false, 1, 6>(__VA_ARGS__);   \
        if (slots <= 8) return line ? fn<F, true, 1, 8>(__VA_ARGS__) : fn<F, false, 1, 8>(__VA_ARGS__);   \
        return line ? fn<F, true, 1, 10>(__VA_ARGS__) : fn<F, false, 1, 10>(__VA_ARGS__);   \
    }                                                                                       \
    if (slots <= 1) return line ? fn<F, true, 2, 1>(__VA_ARGS__) : fn<F, false, 2, 1>(__VA_ARGS__);   \
    if (slots <= 2) return line ? fn<F, true, 2, 2>(__VA_ARGS__) : fn<F, false, 2, 2>(__VA_ARGS__);   \
    if (slots <= 3) return line ? fn<F, true, 2, 3>(__VA_ARGS__) : fn<F, false, 2, 3>(__VA_ARGS__);   \
    if (slots <= 4) return line ? fn<F, true, 2, 4>(__VA_ARGS__) : fn<F, false, 2, 4>(__VA_ARGS__);   \
    return line ? fn<F, true, 2, 5>(__VA_ARGS__) : fn<F, false, 2, 5>(__VA_ARGS__);

template <int F>
int rmx_launch(bool line, int cq, int slots, const RMxArgs& g, int blocks, size_t lds, hipStream_t st) {
    EAFP_RMX_DISPATCH(launch_rmx, g, blocks, lds, st)
}
template <int F>
int rmx_prepare(bool line, int cq, int slots) {
    EAFP_RMX_DISPATCH(prepare_rmx)
}

// One translation unit per weight format (mixed_resident_*.hip).
int rmx_launch_fp32(bool line, int cq, int slots, const RMxArgs& g, int blocks, size_t lds, hipStream_t st);
int rmx_launch_bf16(bool line, int cq, int slots, const RMxArgs& g, int blocks, size_t lds, hipStream_t st);
int rmx_launch_fp16(bool line, int cq, int slots, const RMxArgs& g, int blocks, size_t lds, hipStream_t st);
int rmx_prepare_fp32(bool line, int cq, int slots);
int rmx_prepare_bf16(bool line, int cq, int slots);
int rmx_prepare_fp16(bool line, int cq, int slots);

}  // namespace eafp
