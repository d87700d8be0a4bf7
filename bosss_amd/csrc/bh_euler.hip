// Explicit DG for the compressible Euler equations with the HLLC flux, on a
// periodic Cartesian grid (gfx950).
//
// What: dU/dt = R(U) = int F(U).grad(phi) - oint Fhat(U-, U+, n) phi, with the
// fluxes of OptimizedHLLC{Density,Momentum,Energy}Flux (Flux() and
// InnerEdgeFlux(), L3-solution/BoSSS.Solution.CompressibleFlowCommon/
// Convection/OptimizedHLLCDensityFlux.cs:45-190 and the Momentum/Energy
// variants) and the non-dimensionalisation MachScaling = gamma*Mach^2 used
// there; time stepping with RungeKuttaScheme.TVD3 (L3-solution/
// BoSSS.Solution/TimeStepping/RungeKuttaScheme.cs:145-167).
//
// How (MI355X): the right-hand side is one launch of euler_rhs_kernel
// (bh_eulerrhs.hip: sum-factorised, one lane per cell and node plane, the stage's
// combination in its epilogue); this
// file holds the operator set-up and the TVD3 stages.
#include <algorithm>
#include <cmath>

#include "bh_internal.hpp"
#include "bh_euler.hpp"

namespace bh {

// ------------------------------------------------------------------ host
EulerOp::EulerOp(bh_grid* g_, int k_, int nq1_, double gamma_, double mach) : g(g_), k(k_), nq1(nq1_), gamma(gamma_) {
    ctx = g->ctx;
    D = g->D;
    MS = gamma * mach * mach;
    Np = basis_count(D, k);
    nv = D + 2;
    N = (int64_t)g->J * nv * Np;
    // exponent of the scale that the right-hand side works in (see euler_rhs_kernel)
    double v = 1;
    for (int d = 0; d < D; ++d) {
        const auto w = std::minmax_element(g->width[d].begin(), g->width[d].end());
        v *= std::sqrt(0.5 * std::sqrt(*w.first) * std::sqrt(*w.second));
    }
    if (std::frexp(v, &scale_exp) < std::sqrt(0.5)) --scale_exp;   // the nearest power
}

void EulerOp::stage(const void* U, void* out, int prec, const void* base, double c, double h) {
    if (!euler_stage(this, U, out, prec, base, c, h)) throw Error(-3, "Euler: unsupported (D, k, quadrature points) combination");
}

void EulerOp::rhs(const void* U, void* out, int prec) { stage(U, out, prec, nullptr, 0, 0); }

// The scheme of the reference, k1 = R(U), k2 = R(U + h k1), k3 = R(U + h/4 (k1 + k2)),
// U += h/6 (k1 + k2) + 2h/3 k3, in terms of the stage values (Shu-Osher): each stage is one
// launch and no k is stored.  The increments are taken as differences to U, so that the
// weights 1/3 and 2/3 of a convex combination, whose roundings do not add up to one, never
// scale the state; a step rounds the state at most 11/6 times (three before).
// Bounded by the three right-hand sides: 4.30 ms for a step at 96^3, k = 2, FP64; the
// combinations as launches of their own, which move 12 N of vectors a step, cost 0.4 ms.
void EulerOp::tvd3(void* U, double dt, int steps, int prec) {
    const size_t bytes = N * (prec == BH_FP32 ? sizeof(float) : sizeof(double));
    if (work.bytes < 2 * bytes) work.alloc(2 * bytes);
    void* t1 = work.p;
    void* t2 = (char*)work.p + bytes;
    for (int s = 0; s < steps; ++s) {
        stage(U, t1, prec, nullptr, 1.0, dt);
        stage(t1, t2, prec, U, 0.25, dt);
        stage(t2, U, prec, U, 2.0 / 3.0, dt);
    }
}

}  // namespace bh
