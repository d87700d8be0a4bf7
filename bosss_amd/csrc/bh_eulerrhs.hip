// Explicit DG Euler right-hand side with the HLLC flux (gfx950), sum-factorised on the
// vector units: OptimizedHLLC{Density,Momentum,Energy}Flux, L3-solution/
// BoSSS.Solution.CompressibleFlowCommon/Convection/OptimizedHLLCDensityFlux.cs:45-190,
// periodic Cartesian grid.
//
// NQ lanes share a cell (NQ = Gauss points per direction): lane q takes the nodes whose
// index in the last direction is q.  The tensor basis then splits every contraction:
//   volume: a line of nodes along x needs, per variable, its K + 1 line coefficients
//   (the modes contracted with the line's transverse values), K + 1 multiply-adds per
//   node, and the fluxes are contracted along x in registers before they meet the
//   transverse directions (y in registers, the last one across the lanes);
//   faces: a lane takes the face nodes of one index of the last tangential direction,
//   with line coefficients of both sides' traces, the HLLC flux per node in registers,
//   and the flux contracted along its row before the last direction.
// Each lane keeps partial sums; the NQ partials of a cell are added through LDS.
//
// Bounded by vector instructions (counted): 9,208 per wave of 16 cells at 3D, k = 2, FP64
// (four reciprocals and four square roots per face node; each face is evaluated from both
// of its cells), at four cycles each and 2.4 GHz 0.83 ms of issue at 96^3 against 1.50 ms
// measured (mean of 73 launches, 1.36 at best), at the two waves per SIMD that 240
// registers allow.  FP32, 8,026 per wave and three waves per SIMD: 0.72 ms of issue, 0.78
// measured (0.70 at best), the limit.  Dense node-by-mode products on the matrix
// cores, whose FP64 and FP32 rates are the vector units' here, need four times the
// multiply-adds with their padding to 16 x 16 x 4 tiles: 2.05 ms at 96^3 FP64, and 173 us
// against 96 us here for FP32 at 47 x 61 x 35.
#include <algorithm>
#include <cmath>
#include <vector>

#include "bh_internal.hpp"
#include "bh_euler.hpp"

namespace bh {

namespace {

// tables, per node q: P[q][j], w_q P[q][j], w_q P'[q][j] of the orthonormal Legendre
// polynomials at the Gauss nodes
template <int K, int NQ>
struct EulerTab {
    static constexpr int P = 0, WP = P + NQ * (K + 1), WD = WP + NQ * (K + 1), TOTAL = WD + NQ * (K + 1);
};

// Reciprocal and square root by Newton's and Goldschmidt's iterations from the hardware's
// approximations, to about one unit in the last place.  In FP64 they hold for zero and
// infinity too.  In FP32 the approximations take denormal numbers for zero, and the
// iterations turn that, zero and infinity into NaN: is_normal tells, and the caller
// then uses the exact operations (EXACT).
__device__ __forceinline__ bool is_normal(float x) { return __builtin_amdgcn_classf(x, 0x108); }
__device__ __forceinline__ bool is_normal(double x) { return __builtin_amdgcn_class(x, 0x108); }
template <bool EXACT>
__device__ __forceinline__ double rcp_n(double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = fma(fma(-x, r, 1.0), r, r);
    r = fma(fma(-x, r, 1.0), r, r);
    return __builtin_amdgcn_div_fixup(r, x, 1.0);
}
template <bool EXACT>
__device__ __forceinline__ float rcp_n(float x) {
    if constexpr (EXACT) return 1.0f / x;
    const float r = __builtin_amdgcn_rcpf(x);
    return fmaf(fmaf(-x, r, 1.0f), r, r);
}
template <bool EXACT>
__device__ __forceinline__ double sqrt_n(double x) {
    const double r = __builtin_amdgcn_rsq(x);
    double g = x * r, h = 0.5 * r;
    double e = fma(-h, g, 0.5);
    g = fma(g, e, g);
    h = fma(h, e, h);
    g = fma(fma(-g, g, x), h, g);
    return __builtin_amdgcn_class(x, 0x260) ? x : g;   // zeros and +infinity
}
template <bool EXACT>
__device__ __forceinline__ float sqrt_n(float x) {
    if constexpr (EXACT) return sqrtf(x);
    const float r = __builtin_amdgcn_rsqf(x);
    const float g = x * r;
    return fmaf(fmaf(-g, g, x), 0.5f * r, g);
}

// n values in 16-byte loads (the array need only be aligned to its elements)
template <int n, typename R>
__device__ __forceinline__ void load_row(const R* __restrict__ p, R* r) {
    constexpr int W = 16 / sizeof(R);
    typedef R V __attribute__((ext_vector_type(W), aligned(sizeof(R))));
#pragma unroll
    for (int i = 0; i + W <= n; i += W) {
        const V v = *(const V*)(p + i);
#pragma unroll
        for (int t = 0; t < W; ++t) r[i + t] = v[t];
    }
#pragma unroll
    for (int i = n / W * W; i < n; ++i) r[i] = p[i];
}

// index of the pair (a, b), a + b <= k
__host__ __device__ constexpr int pair_of(int k, int a, int b) { return a * (k + 1) - a * (a - 1) / 2 + b; }

template <typename R>
struct Gas {
    R gm1, MS, iMS, iMach, hg;   // hg = (gamma + 1) / (2 gamma), iMach = sqrt(gamma / MS)
};

// HLLC as OptimizedHLLC*Flux.InnerEdgeFlux (normal = sgn * e_dn).  The wave speeds
// a q = sqrt(gamma / MS (p + hg max(p* - p, 0)) / rho) and the star state's energy term
// f (rho s* MS + p / (s - v)) (s* - v) with f = (s - v) / (s - s*) need four reciprocals and
// four square roots per node.  False (FP32) where one of them left the range of the fast
// forms; F is then to be taken from EXACT.
template <int D, int dn, bool EXACT, typename R>
__device__ __forceinline__ bool hllc(const Gas<R>& g, const R* Ui, const R* Uo, R sgn, R* F) {
    const R rIn = Ui[0], rOut = Uo[0], EIn = Ui[D + 1], EOut = Uo[D + 1];
    const R irIn = rcp_n<EXACT>(rIn), irOut = rcp_n<EXACT>(rOut);
    R m2In = 0, m2Out = 0;
#pragma unroll
    for (int d = 0; d < D; ++d) { m2In = fma(Ui[d + 1], Ui[d + 1], m2In); m2Out = fma(Uo[d + 1], Uo[d + 1], m2Out); }
    const R vnIn = sgn * Ui[dn + 1] * irIn, vnOut = sgn * Uo[dn + 1] * irOut;
    const R pIn = g.gm1 * (EIn - g.MS * R(0.5) * m2In * irIn), pOut = g.gm1 * (EOut - g.MS * R(0.5) * m2Out * irOut);
    const R aIn = sqrt_n<EXACT>(pIn * irIn), aOut = sqrt_n<EXACT>(pOut * irOut);
    const R pStar = fmax(R(0), R(0.5) * (pIn + pOut) - R(0.125) * g.MS * g.iMach * (vnOut - vnIn) * (aIn + aOut) * (rIn + rOut));
    const R sIn = vnIn - g.iMach * sqrt_n<EXACT>(irIn * fma(g.hg, fmax(pStar - pIn, R(0)), pIn));
    const R sOut = vnOut + g.iMach * sqrt_n<EXACT>(irOut * fma(g.hg, fmax(pStar - pOut, R(0)), pOut));
    const R cIn = rIn * (sIn - vnIn), cOut = rOut * (sOut - vnOut);
    const R rc = rcp_n<EXACT>(cOut - cIn);
    const R sStar = (cOut * vnOut - cIn * vnIn + (pIn - pOut) * g.iMS) * rc;
    const bool left = sStar > R(0);
    const R rS = left ? rIn : rOut, irS = left ? irIn : irOut, vnS = left ? vnIn : vnOut, pS = left ? pIn : pOut;
    const R ES = left ? EIn : EOut, sK = left ? sIn : sOut;
    R Us[D];
#pragma unroll
    for (int c = 0; c < D; ++c) Us[c] = left ? Ui[c + 1] : Uo[c + 1];
    // the outer flux, and the star region's correction where the wave has passed the face
    const bool star = left ? sIn <= R(0) : sOut >= R(0);
    const R d1 = rcp_n<EXACT>(sK - sStar), f = (sK - vnS) * d1, dv = sStar - vnS, rf = rS * f;
    auto put = [&](int v, R outer, R corr) { F[v] = star ? fma(sK, corr, outer) : outer; };   // corr may be infinite or NaN where unused
    put(0, vnS * rS, rf - rS);
#pragma unroll
    for (int c = 0; c < D; ++c) {
        const R pn = c == dn ? sgn * pS * g.iMS : R(0), un = Us[c] * irS + (c == dn ? sgn * dv : R(0));
        put(c + 1, vnS * Us[c] + pn, rf * un - Us[c]);
    }
    const R fe = fma(rf * sStar * g.MS + pS * d1, dv, f * ES);
    put(D + 1, vnS * (ES + pS), fe - ES);
    // NaN or infinity of any reciprocal or root shows in these three (a speed of sound that is
    // zero included); single tests would cost as much as the exact operations
    if constexpr (sizeof(R) == 4 && !EXACT) return is_normal(aIn + aOut) && is_normal(rc) && is_normal(d1);
    return true;
}

}  // namespace

template <int K, int NQ, typename R>
struct EulerArgs {
    int J, n0, n1, n2, nmax;
    const double* __restrict__ width;   // [4][3][nmax]: h, 1/h, sqrt(h), 1/sqrt(h)
    const R* __restrict__ tab;          // the tables for lane-dependent nodes
    // the same by value: kernel arguments are scalar loads wherever they are used
    R P[NQ * (K + 1)], WP[NQ * (K + 1)], WD[NQ * (K + 1)];
    Gas<R> gas;
    R sc, isc;                          // 2^-e and 2^e, 2^e near the grid's sqrt(det J)
    const R* __restrict__ U;
    // a stage of the time step in the same launch: out = base + c (U - base + h R(U)), base the
    // step's first state (null: U itself); c = 0 writes R(U).  out may be base
    const R* base;
    R c, h;
    R* out;
};

template <int D, int K, int NQ, typename R>
__global__ __launch_bounds__(256, 2) void euler_rhs_kernel(EulerArgs<K, NQ, R> a) {
    using T = EulerTab<K, NQ>;
    constexpr int Np = binom(K + D, D), NV = D + 2, ROW = NV * Np, K1 = K + 1;
    constexpr int CW = 64 / NQ;                  // cells per wave
    constexpr int LS = ROW | 1, LY = Np | 1;     // odd strides: no bank conflicts between cells / lanes
    __shared__ R sU[4][CW * LS], sY[4][64 * LY], sZ[4][CW * ROW];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int cl = lane / NQ < CW ? lane / NQ : CW - 1, ql = lane - (lane / NQ) * NQ;   // the last lanes repeat a cell
    const int c0 = ((int)blockIdx.x * 4 + wave) * CW;
    if (c0 >= a.J) return;                       // whole wave; no barrier in this kernel
    const int nc = min(CW, a.J - c0);
    R* __restrict__ su = sU[wave];
    R* __restrict__ sy = sY[wave];
    R* __restrict__ sz = sZ[wave];
    for (int t = lane; t < nc * ROW; t += 64) {
        const int i = t / ROW;
        su[i * LS + t - i * ROW] = a.sc * a.U[(size_t)c0 * ROW + t];
    }
    const int c = c0 + min(cl, nc - 1);
    const R* __restrict__ u = su + min(cl, nc - 1) * LS;
    int idx[3];
    if (D == 2) { idx[0] = c / a.n1; idx[1] = c - idx[0] * a.n1; idx[2] = 0; }
    else { const int sl = a.n0 * a.n1; idx[2] = c / sl; const int rr = c - idx[2] * sl; idx[1] = rr / a.n0; idx[0] = rr - idx[1] * a.n0; }
    const int nn[3] = {a.n0, a.n1, a.n2};
    // g_d = 2 / h_d.  The physical states are the modal sums over sqrt(det J); the fluxes are
    // homogeneous of degree one in the state, so the kernel works with the sums, the
    // neighbour's rescaled to the cell's volume, over a power of two near the grid's
    // sqrt(det J) (EulerArgs::sc): no rounding, and squares and quotients of the states stay in
    // the type's range whatever the size of the cells.
    R gd[3] = {1, 1, 1};
#pragma unroll
    for (int d = 0; d < D; ++d) gd[d] = R(2) * (R)a.width[(3 + d) * a.nmax + idx[d]];
    // the lane's values in its own direction
    R pq[K1], wq[K1], dq[K1];
#pragma unroll
    for (int j = 0; j < K1; ++j) {
        pq[j] = a.tab[T::P + ql * K1 + j];
        wq[j] = a.tab[T::WP + ql * K1 + j];
        dq[j] = a.tab[T::WD + ql * K1 + j];
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    constexpr int N2 = D == 3 ? (K + 1) * (K + 2) / 2 : K1;   // mode pairs (2D: exponents)
    // Face terms of direction d; the lanes run along t2, a lane's row along t1 (2D: one node
    // per lane).  H[v][(e_t1, e_d)] += the flux against the face's test functions without
    // their t2 factor.
    auto faces = [&](auto DD, R (&H)[NV][N2]) {
        constexpr int d = DD;
        constexpr int t2 = d == D - 1 ? D - 2 : D - 1, t1 = D == 3 ? 3 - d - t2 : 0;
        constexpr int KR = D == 3 ? K1 : 1;      // row coefficients
#pragma unroll 1
        for (int sd = 0; sd < 2; ++sd) {
            const R sgn = sd ? R(1) : R(-1);
            int nidx[3] = {idx[0], idx[1], idx[2]};
            nidx[d] += sd ? 1 : -1;
            nidx[d] = nidx[d] < 0 ? nn[d] - 1 : (nidx[d] == nn[d] ? 0 : nidx[d]);
            const int cn = D == 2 ? nidx[0] * a.n1 + nidx[1] : nidx[0] + nidx[1] * a.n0 + nidx[2] * a.n0 * a.n1;
            const R* __restrict__ un = a.U + (size_t)cn * ROW;
            // sqrt(det J of the cell / det J of the neighbour): they differ in the width along d
            const R rs = a.sc * (R)(a.width[(6 + d) * a.nmax + idx[d]] * a.width[(9 + d) * a.nmax + nidx[d]]);
            R Li[NV][KR], Lo[NV][KR], G[NV][KR];
            static_for<NV>([&](auto VV) {
                constexpr int v = VV;
                R uo[Np];
                load_row<Np>(un + v * Np, uo);
#pragma unroll
                for (int i = 0; i < KR; ++i) { Li[v][i] = 0; Lo[v][i] = 0; G[v][i] = 0; }
                static_for<Np>([&](auto NN) {
                    constexpr int n = NN, j = mode_exponent(D, K, n, d), e2 = mode_exponent(D, K, n, t2);
                    constexpr int e1 = D == 3 ? mode_exponent(D, K, n, t1) : 0;
                    // p_j(sgn) = sgn^j s_j on the own side, (-sgn)^j s_j on the neighbour's
                    const R pv = R(sqrt_half(j)) * pq[e2], po = (j & 1) ? pv * sgn : pv;
                    Li[v][e1] = fma(po, u[v * Np + n], Li[v][e1]);
                    Lo[v][e1] = fma((j & 1) ? -po : po, uo[n], Lo[v][e1]);
                });
#pragma unroll
                for (int i = 0; i < KR; ++i) Lo[v][i] *= rs;
                // keep the loads of the later variables out of the registers of the earlier ones
                if constexpr (v == 2) asm volatile("" ::: "memory");
            });
            const R wf = -gd[d];                 // dA / det J
#pragma unroll 1
            for (int q = 0; q < (D == 3 ? NQ : 1); ++q) {
                R F[NV];
                auto flux = [&](auto EX) {
                    R Ui[NV], Uo[NV];
#pragma unroll
                    for (int v = 0; v < NV; ++v) {
                        if constexpr (D == 3) {
                            Ui[v] = a.P[q * K1] * Li[v][0];
                            Uo[v] = a.P[q * K1] * Lo[v][0];
#pragma unroll
                            for (int i = 1; i < K1; ++i) {
                                Ui[v] = fma(a.P[q * K1 + i], Li[v][i], Ui[v]);
                                Uo[v] = fma(a.P[q * K1 + i], Lo[v][i], Uo[v]);
                            }
                        } else {
                            Ui[v] = Li[v][0];
                            Uo[v] = Lo[v][0];
                        }
                    }
                    return hllc<D, d, EX, R>(a.gas, Ui, Uo, sgn, F);
                };
                if (!flux(std::false_type{})) flux(std::true_type{});   // FP64: never
                // FP32 has registers for the row's sum (93.9 against 99.5 us at 47 x 61 x 35,
                // k = 2); in FP64 it spills (4659 against 4611 us for a step at 96^3)
                if constexpr (D == 3 && sizeof(R) == 4) {
#pragma unroll
                    for (int v = 0; v < NV; ++v)
#pragma unroll
                        for (int i = 0; i < K1; ++i) G[v][i] = fma(a.WP[q * K1 + i], F[v], G[v][i]);
                } else {
                    static_for<K1>([&](auto JJ) {
                        constexpr int j = JJ;
                        const R pj = R(sqrt_half(j)) * wf * ((j & 1) ? sgn : R(1));
                        static_for<D == 3 ? K1 - j : 1>([&](auto II) {
                            constexpr int i = II, ij = D == 2 ? j : (t1 < d ? pair_of(K, i, j) : pair_of(K, j, i));   // lower direction first
                            const R t = D == 2 ? pj : pj * a.WP[q * K1 + i];
#pragma unroll
                            for (int v = 0; v < NV; ++v) H[v][ij] = fma(t, F[v], H[v][ij]);
                        });
                    });
                }
            }
            if constexpr (D == 3 && sizeof(R) == 4) {
                static_for<K1>([&](auto JJ) {
                    constexpr int j = JJ;
                    const R pj = R(sqrt_half(j)) * wf * ((j & 1) ? sgn : R(1));
                    static_for<K1 - j>([&](auto II) {
                        constexpr int i = II, ij = t1 < d ? pair_of(K, i, j) : pair_of(K, j, i);
#pragma unroll
                        for (int v = 0; v < NV; ++v) H[v][ij] = fma(pj, G[v][i], H[v][ij]);
                    });
                });
            }
        }
    };
    // Sum over the lanes of a cell of one variable's partials r(n), cell by cell: put(slot, sum)
    auto lane_sum = [&](const R* r, auto&& put) {
#pragma unroll
        for (int n = 0; n < Np; ++n) sy[lane * LY + n] = r[n];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int t0 = 0; t0 < CW * Np; t0 += 64) {
            const int t = t0 + lane, i = t / Np, n = t - i * Np;
            if (i < nc) {
                R s = sy[i * NQ * LY + n];
#pragma unroll
                for (int q = 1; q < NQ; ++q) s += sy[(i * NQ + q) * LY + n];
                put(i, n, s);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    // ---------------- faces of the last direction (lanes along the one before): summed over
    // the lanes now, so that only the other terms' partials stay in registers
    {
        R H[NV][N2];
#pragma unroll
        for (int v = 0; v < NV; ++v)
#pragma unroll
            for (int i = 0; i < N2; ++i) H[v][i] = 0;
        faces(std::integral_constant<int, D - 1>{}, H);
        static_for<NV>([&](auto VV) {
            constexpr int v = VV;
            R r[Np];
            static_for<Np>([&](auto NN) {
                constexpr int n = NN, e0 = mode_exponent(D, K, n, 0), e1 = mode_exponent(D, K, n, 1);
                if constexpr (D == 3) r[n] = wq[e1] * H[v][pair_of(K, e0, mode_exponent(D, K, n, 2))];
                else r[n] = wq[e0] * H[v][e1];
            });
            lane_sum(r, [&](int i, int n, R s) { sz[i * ROW + v * Np + n] = s; });
        });
    }
    // ---------------- the other faces (lanes along the last direction, as in the volume)
    R XY[NV][N2], Z[NV][D == 3 ? N2 : K1];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
#pragma unroll
        for (int i = 0; i < N2; ++i) XY[v][i] = 0;
#pragma unroll
        for (int i = 0; i < (D == 3 ? N2 : K1); ++i) Z[v][i] = 0;
    }
    static_for<D - 1>([&](auto DD) { faces(DD, XY); });
    // ---------------- volume
#pragma unroll 1
    for (int qy = 0; qy < (D == 3 ? NQ : 1); ++qy) {
        // line coefficients of the states; X, Y, L: the fluxes of the first, second and (3D)
        // third direction contracted along the line
        R w[NV][K1], X_[NV][K1], Y_[NV][K1], L_[NV][K1];
        static_for<NV>([&](auto VV) {
            constexpr int v = VV;
#pragma unroll
            for (int i = 0; i < K1; ++i) { w[v][i] = 0; X_[v][i] = 0; Y_[v][i] = 0; L_[v][i] = 0; }
            static_for<Np>([&](auto NN) {
                constexpr int n = NN, i = mode_exponent(D, K, n, 0), j = mode_exponent(D, K, n, 1);
                if constexpr (D == 3) {
                    constexpr int l = mode_exponent(D, K, n, 2);
                    w[v][i] = fma(a.P[qy * K1 + j] * pq[l], u[v * Np + n], w[v][i]);
                } else {
                    w[v][i] = fma(pq[j], u[v * Np + n], w[v][i]);
                }
            });
            asm volatile("" ::: "memory");
        });
#pragma unroll
        for (int qx = 0; qx < NQ; ++qx) {
            R s[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                s[v] = a.P[qx * K1] * w[v][0];
#pragma unroll
                for (int i = 1; i < K1; ++i) s[v] = fma(a.P[qx * K1 + i], w[v][i], s[v]);
            }
            R irho = rcp_n<false>(s[0]);
            if (sizeof(R) == 4 && !is_normal(irho)) irho = rcp_n<true>(s[0]);
            R m2 = 0;
#pragma unroll
            for (int d = 0; d < D; ++d) m2 = fma(s[d + 1], s[d + 1], m2);
            const R p = a.gas.gm1 * (s[D + 1] - a.gas.MS * R(0.5) * m2 * irho), pM = p * a.gas.iMS, Ep = s[D + 1] + p;
            static_for<D>([&](auto DD) {
                constexpr int d = DD;
                const R ud = s[d + 1] * irho;
                static_for<NV>([&](auto VV) {
                    constexpr int v = VV;
                    R f;
                    if constexpr (v == 0) f = s[d + 1];
                    else if constexpr (v == D + 1) f = ud * Ep;
                    else f = v == d + 1 ? fma(s[v], ud, pM) : s[v] * ud;
                    if constexpr (d == 0) {
#pragma unroll
                        for (int i = 1; i < K1; ++i) X_[v][i] = fma(a.WD[qx * K1 + i], f, X_[v][i]);
                    } else {
                        R* A = d == 1 ? Y_[v] : L_[v];
#pragma unroll
                        for (int i = 0; i < K; ++i) A[i] = fma(a.WP[qx * K1 + i], f, A[i]);
                    }
                });
            });
        }
        if constexpr (D == 3) {
            // contract along y: values for the x and z fluxes, derivatives for the y flux
            static_for<K1>([&](auto JJ) {
                constexpr int j = JJ;
                const R wp = a.WP[qy * K1 + j], wd = a.WD[qy * K1 + j];
                const R wx = wp * gd[0], wy = wd * gd[1], wz = wp * gd[2];
                static_for<NV>([&](auto VV) {
                    constexpr int v = VV;
                    static_for<K1 - j>([&](auto II) {
                        constexpr int i = II, ij = pair_of(K, i, j);
                        if constexpr (i > 0) XY[v][ij] = fma(wx, X_[v][i], XY[v][ij]);
                        if constexpr (j > 0) XY[v][ij] = fma(wy, Y_[v][i], XY[v][ij]);
                        if constexpr (i + j < K) Z[v][ij] = fma(wz, L_[v][i], Z[v][ij]);
                    });
                });
            });
        } else {
            static_for<NV>([&](auto VV) {
                constexpr int v = VV;
#pragma unroll
                for (int i = 0; i < K1; ++i) {
                    if (i > 0) XY[v][i] = fma(gd[0], X_[v][i], XY[v][i]);
                    if (i < K) Z[v][i] = gd[1] * Y_[v][i];
                }
            });
        }
    }
    // ---------------- contract along the lane's direction and add the lanes' partials
    static_for<NV>([&](auto VV) {
        constexpr int v = VV;
        R r[Np];
        static_for<Np>([&](auto NN) {
            constexpr int n = NN, i = mode_exponent(D, K, n, 0), j = mode_exponent(D, K, n, 1);
            constexpr int l = D == 3 ? mode_exponent(D, K, n, 2) : j, ij = D == 3 ? pair_of(K, i, j) : i;
            r[n] = wq[l] * XY[v][ij];
            if constexpr (l > 0) r[n] = fma(dq[l], Z[v][ij], r[n]);
        });
        lane_sum(r, [&](int i, int n, R s) {
            const size_t o = ((size_t)(c0 + i) * NV + v) * Np + n;
            R y = a.isc * (s + sz[i * ROW + v * Np + n]);
            if (a.c != R(0)) {
                const R x = a.isc * su[i * LS + v * Np + n], b = a.base ? a.base[o] : x;
                y = fma(a.c, fma(a.h, y, x - b), b);
            }
            a.out[o] = y;
        });
    });
}

template <int D, int K, int NQ>
static void ensure_tables(EulerOp* e) {
    if (e->tab64.p) return;
    using T = EulerTab<K, NQ>;
    std::vector<double> x(NQ), w(NQ), h(T::TOTAL), val(K + 1), der(K + 1);
    gauss_rule(NQ, x.data(), w.data());
    for (int q = 0; q < NQ; ++q) {
        // orthonormal Legendre polynomials and derivatives by the three-term recursion
        std::vector<double> p(K + 2), dp(K + 2);
        p[0] = 1;
        p[1] = x[q];
        dp[0] = 0;
        dp[1] = 1;
        for (int n = 2; n <= K; ++n) {
            p[n] = ((2 * n - 1) * x[q] * p[n - 1] - (n - 1) * p[n - 2]) / n;
            dp[n] = dp[n - 2] + (2 * n - 1) * p[n - 1];
        }
        for (int j = 0; j <= K; ++j) {
            const double s = std::sqrt(j + 0.5);
            h[T::P + q * (K + 1) + j] = s * p[j];
            h[T::WP + q * (K + 1) + j] = w[q] * s * p[j];
            h[T::WD + q * (K + 1) + j] = w[q] * s * dp[j];
        }
    }
    e->h_tab = h;
    e->tab64.alloc(h.size() * sizeof(double));
    e->ctx->upload(e->tab64.p, h.data(), h.size() * sizeof(double));
    std::vector<float> h32(h.begin(), h.end());
    e->tab32.alloc(h32.size() * sizeof(float));
    e->ctx->upload(e->tab32.p, h32.data(), h32.size() * sizeof(float));
}

template <int D, int K, int NQ, typename R>
static void launch_rhs(EulerOp* e, const R* U, R* out, const R* base, double c, double h) {
    ensure_tables<D, K, NQ>(e);
    EulerArgs<K, NQ, R> a;
    a.J = e->g->J;
    a.n0 = e->g->n[0]; a.n1 = e->g->n[1]; a.n2 = e->g->n[2];
    a.nmax = e->g->nmax;
    a.width = e->g->d_width.as<double>();
    a.tab = (const R*)(sizeof(R) == 4 ? e->tab32.p : e->tab64.p);
    using T = EulerTab<K, NQ>;
    for (int i = 0; i < NQ * (K + 1); ++i) {
        a.P[i] = (R)e->h_tab[T::P + i];
        a.WP[i] = (R)e->h_tab[T::WP + i];
        a.WD[i] = (R)e->h_tab[T::WD + i];
    }
    a.gas.gm1 = (R)(e->gamma - 1.0);
    a.gas.MS = (R)e->MS;
    a.gas.iMS = (R)(1.0 / e->MS);
    a.gas.iMach = (R)std::sqrt(e->gamma / e->MS);
    a.gas.hg = (R)(0.5 * (e->gamma + 1.0) / e->gamma);
    constexpr int emax = sizeof(R) == 4 ? 120 : 1000;   // both powers are normal numbers
    const int ex = std::min(std::max(e->scale_exp, -emax), emax);
    a.sc = (R)std::ldexp(1.0, -ex);
    a.isc = (R)std::ldexp(1.0, ex);
    a.U = U;
    a.base = base;
    a.c = (R)c;
    a.h = (R)h;
    a.out = out;
    constexpr int CB = 4 * (64 / NQ);   // cells per workgroup
    hipLaunchKernelGGL((euler_rhs_kernel<D, K, NQ, R>), dim3((a.J + CB - 1) / CB), dim3(256), 0, e->ctx->stream, a);
    BH_HIP(hipGetLastError());
}

bool euler_stage(EulerOp* e, const void* U, void* out, int prec, const void* base, double c, double h) {
#define BH_CASE(DD, KK, QQ)                                                                                  \
    if (e->D == DD && e->k == KK && e->nq1 == QQ) {                                                          \
        if (prec == BH_FP32) launch_rhs<DD, KK, QQ, float>(e, (const float*)U, (float*)out, (const float*)base, c, h);                 \
        else launch_rhs<DD, KK, QQ, double>(e, (const double*)U, (double*)out, (const double*)base, c, h);                              \
        return true;                                                                                         \
    }
    BH_CASE(3, 1, 3) BH_CASE(3, 2, 4) BH_CASE(3, 1, 2) BH_CASE(2, 2, 4) BH_CASE(2, 3, 5) BH_CASE(2, 1, 3)
#undef BH_CASE
    return false;
}

}  // namespace bh
