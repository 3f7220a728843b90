// cg64.hpp -- state and arguments of the FP64 CG, shared by its streaming
// kernels (cg64.hip) and its resident kernel (cg64_resident.hip).
#pragma once
#include "batch.hpp"

namespace eafp {

struct CgSlot {
    double bnorm;      // ||Su||; < 0 until the first k64_spmv after k64_init
    double residual;   // relative recurrence residual of the last completed iteration
    double rz, alpha, beta;
    int it;            // iteration in progress (set by k64_spmv)
    int n_iter;        // completed iterations
    int done, status;
};

struct CgConst {
    double tol;
    int max_iter;
    int pad;
};

struct Cg64Args {
    const TileDesc* tiles;
    int ntiles;
    int nsys;
    const double *aW, *aE, *aS, *aN, *aB, *aT, *aP;
    const double *b, *fold, *x0;
    double *x, *r, *z, *q;
    double* p[2];
    double* partA;       // ntiles:     p.q
    double* partB;       // ntiles * 3: r.r, r.z, Su.Su
    CgSlot* slot[2];
    const CgConst* cst;
    int* ndone;          // finished systems, counted after each chunk
    int state_first;     // 1 (batches): read a system's state before its cell loads; 0: overlap them
};

}  // namespace eafp
