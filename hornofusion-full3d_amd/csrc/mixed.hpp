// mixed.hpp -- state, arguments and weight formats of the mixed-precision
// solver, shared by its streaming kernels (mixed.hip) and its resident kernel
// (mixed_resident.hpp).
#pragma once
#include "batch.hpp"

namespace eafp {

// Per-system state of the mixed solver, double-buffered by kernel role:
// MxDyn changes every inner iteration (k_mspmv reads slot 1 and writes
// slot 0, k_mupdate the reverse); MxStat changes once per refinement step
// (k_res copies slot 1 to slot 0, k_mreplace writes slot 1 from slot 0).
// Every thread loads the few MxDyn fields it needs and the writer stores
// its new values straight from registers.
struct MxDyn {
    double rz, alpha, beta;
    int fresh;          // next k_mspmv starts a new Krylov sequence (beta = 0)
    int broken;         // inner breakdown: idle until the next refinement step
    int total_inner;
    int done;           // mirror of MxStat::done for the inner kernels
};

struct MxStat {
    double bnorm, b1, res_l2, res_l1;
    double res_first, res_least;   // res_l2 of the first step, the smallest so far
    double mean_x[MAX_COMP];
    int n_refine, done, status, xbuf;
};

struct MxConst {
    double tol;
    double inv_cnt[MAX_COMP];
    int ncomp, max_steps, restart, pad;
};

constexpr int NRES = 4 + 2 * MAX_COMP;   // r.r, |r|, Su.Su, |Su|, sum r per comp, sum x per comp

struct MxArgs {
    const TileDesc* tiles;
    int ntiles;
    int nsys;
    const ColDesc* cols;   // column segments (column-marching stencil)
    // FP64 operand
    const double *aW, *aE, *aS, *aN, *aB, *aT, *aP, *b, *fold, *x0;
    const unsigned char* comp;
    double* X[2];        // FP64 iterate, ping-pong per refinement step
    double* r64;         // FP64 residual of the current refinement step
    double* xout;        // projected result
    // compressed operand
    void* w[3];          // +r, +theta, +z face weights (format dependent)
    float* scale;        // FP16 only: per-cell scale (the owner's aP)
    void* e;             // diagonal excess, in the weight format (FP16: scaled like the weights)
    float* dinv;         // Jacobi inverse of the rounded operator
    const LineTile* lt;  // line tiles (z-line preconditioner)
    unsigned* fac;       // z-line factors per cell: FP16 l (low half), BF16 1/d (high half)
    int line;            // 1: z-line preconditioner; the r.z partials are per line tile
    int state_first;     // 1 (batches): read the system's state before the cell loads, so the
                         // blocks of converged systems load nothing; 0 (one system): overlap them
    // inner FP32 vectors
    float *d, *r, *z, *q;
    float* p[2];
    long sink;           // a 16-byte slot past the cells of p[0], p[1] and q: stores that must be issued but not kept
    double* partR;       // ntiles * NRES (k_res)
    double* sumR;        // nsys * NRES: partR reduced per system (k_rsum)
    const SysGeom* geom; // per-system geometry and tile ranges
    double* partA;       // ntiles        (k_mspmv: p.q)
    double* partB;       // ntiles * 2, or nltiles * 2 with `line` (k_mreplace, k_mupdate: r.r, r.z)
    MxDyn* dyn[2];
    MxStat* stat[2];
    const MxConst* cst;
    int* ndone;          // finished systems; of them, set aside (k_mcount)
};

// ---------------------------------------------------------------------------
// Weight storage formats
// ---------------------------------------------------------------------------
__device__ __forceinline__ unsigned short f32_to_bf16_rne(float v) {
    unsigned u = __float_as_uint(v);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
}

template <int F>
struct WFmt;

template <>
struct WFmt<EAFP_COEF_FP32> {
    using T = float;
    __device__ static float load(const void* w, const float*, long o) { return ((const float*)w)[o]; }
    __device__ static F4 load4(const void* w, const float*, long o) { return ld4((const float*)w + o); }
    __device__ static T enc(float v, float) { return v; }
    __device__ static float dec(T h, float) { return h; }
};

template <>
struct WFmt<EAFP_COEF_BF16> {
    using T = unsigned short;
    __device__ static float load(const void* w, const float*, long o) {
        return __uint_as_float((unsigned)((const unsigned short*)w)[o] << 16);
    }
    __device__ static F4 load4(const void* w, const float*, long o) {
        unsigned short h[4];
        __builtin_memcpy(h, __builtin_assume_aligned((const unsigned short*)w + o, 8), 8);
        F4 r;
#pragma unroll
        for (int q = 0; q < 4; ++q) r.v[q] = __uint_as_float((unsigned)h[q] << 16);
        return r;
    }
    __device__ static T enc(float v, float) { return f32_to_bf16_rne(v); }
    __device__ static float dec(T h, float) { return __uint_as_float((unsigned)h << 16); }
};

template <>
struct WFmt<EAFP_COEF_FP16> {
    using T = _Float16;
    __device__ static float load(const void* w, const float* sc, long o) {
        return (float)((const _Float16*)w)[o] * sc[o];
    }
    __device__ static F4 load4(const void* w, const float* sc, long o) {
        _Float16 h[4];
        __builtin_memcpy(h, __builtin_assume_aligned((const _Float16*)w + o, 8), 8);
        F4 r = ld4(sc + o);
#pragma unroll
        for (int q = 0; q < 4; ++q) r.v[q] *= (float)h[q];
        return r;
    }
    __device__ static T enc(float v, float s) { return (_Float16)(v / s); }
    __device__ static float dec(T h, float s) { return (float)h * s; }
};

// z-line factors of a cell: FP16 l (low half), BF16 1/d (high half).
__device__ __forceinline__ void unpack_fac(float bits, float& l, float& inv) {
    const unsigned u = __float_as_uint(bits);
    const unsigned short lb = (unsigned short)(u & 0xFFFFu);
    _Float16 lh;
    __builtin_memcpy(&lh, &lb, 2);
    l = (float)lh;
    inv = __uint_as_float(u & 0xFFFF0000u);
}

constexpr long SINK_CELLS = 64;   // past the arenas: the column stencil's discarded stores, and the
                                  // rest of a quad that begins at the last cell of a row

}  // namespace eafp
