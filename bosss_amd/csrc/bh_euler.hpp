// Explicit DG Euler / HLLC operator (see bh_euler.hip).
#pragma once
#include "bh_internal.hpp"

namespace bh {

struct EulerOp;
// out = R(U), or with c != 0 a stage of the time step, out = base + c (U - base + h R(U))
// (base null: U; out may be base, not U) (bh_eulerrhs.hip); false if (D, k, nodes) is not supported
bool euler_stage(EulerOp* e, const void* U, void* out, int prec, const void* base = nullptr, double c = 0, double h = 0);

struct EulerOp {
    bh_ctx* ctx;
    bh_grid* g;
    int D, k, nq1, Np, nv;
    int64_t N;
    double gamma, MS;
    int scale_exp = 0;        // 2^scale_exp is near sqrt(det J) of the grid's cells (geometric mean of the widest and narrowest)
    DevBuf work;
    DevBuf tab64, tab32;      // 1D tables of the right-hand side (built on first use)
    std::vector<double> h_tab;
    EulerOp(bh_grid* g, int k, int nq1, double gamma, double mach);
    void rhs(const void* U, void* out, int prec);
    void tvd3(void* U, double dt, int steps, int prec);
    void stage(const void* U, void* out, int prec, const void* base, double c, double h);
};

// Newton-Krylov solve of the backward-Euler step U - Un - dt R(U) = 0 (bh_newton.cpp)
void newton_euler(EulerOp* E, const double* Un, double* U, double dt, double conv, int maxit, int restart, int* info,
                  double* res);

}  // namespace bh

struct bh_euler {
    bh::EulerOp* e = nullptr;
};
