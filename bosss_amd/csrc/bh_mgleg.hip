// Legs of a multigrid cycle on assembled levels of small blocks (gfx950): the way down from
// a level (residual, restriction and the coarse level's first block-Jacobi sweep) and the
// way up (residual, sweep and the prolongation to the finer level) as one launch each.  The
// reference runs them one after the other (AS/OrthonormalizationMultigrid.cs:797-1100,
// AS/BlockJacobi.cs:150-240).
//
// Below the finest level a cycle is bounded by launches and by the chains of dependent loads
// in them, not by bytes: at 32^3 cells of 4 modes the sweep, residual and restriction took
// 4.4 + 5.2 + 6.1 us and three launch gaps.  What a launch needs of its neighbours is only
// the vector that the residual multiplies; sweep, transfer and prolongation touch a row and
// its aggregate, so they ride along with the launch that makes their input: 5.1 us down and
// 6.5 us up as the mean of the 32^3 and 16^3 levels, the dense solve of 2048 with its
// prolongation 7.4 us (FP32); at 48^3 cells, 50 MB of blocks, 16 and 12 us.
#include "bh_internal.hpp"
#include "bh_mg.hpp"

namespace bh {

namespace {

// value of the lane j ^ X of the quad (X = 1, 2), and of its lane M
template <int CTRL, typename T>
__device__ __forceinline__ T quad_move(T v) {
    if constexpr (sizeof(T) == 8) {
        const long long b = __double_as_longlong(v);
        const int lo = __builtin_amdgcn_mov_dpp((int)b, CTRL, 0xf, 0xf, true);
        const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xf, 0xf, true);
        return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
    } else {
        return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
    }
}
template <typename T> __device__ __forceinline__ T quad_xor1(T v) { return quad_move<0xB1>(v); }
template <typename T> __device__ __forceinline__ T quad_xor2(T v) { return quad_move<0x4E>(v); }

// lane j of a quad: sum over the quad's lanes of their s[j]
template <typename T>
__device__ __forceinline__ T quad_transpose_sum(const T* s, int j) {
    const bool hi = j & 2, odd = j & 1;
    const T a0 = (hi ? s[2] : s[0]) + quad_xor2(hi ? s[0] : s[2]);
    const T a1 = (hi ? s[3] : s[1]) + quad_xor2(hi ? s[1] : s[3]);
    return (odd ? a1 : a0) + quad_xor1(odd ? a0 : a1);
}
// sum_m A[m] v_m, v_m the value of the quad's lane m
template <int BS, typename T>
__device__ __forceinline__ T quad_dot(const T* A, T v) {
    T s = A[0] * quad_move<0x00>(v);
    if constexpr (BS > 1) s += A[1] * quad_move<0x55>(v);
    if constexpr (BS > 2) s += A[2] * quad_move<0xAA>(v);
    if constexpr (BS > 3) s += A[3] * quad_move<0xFF>(v);
    return s;
}

}  // namespace

namespace {

// One column of a block, BS consecutive values, and nothing behind them: the matrix's last
// block ends its allocation.  A vector of four is one load; a vector type of three has the
// size (and in FP64 the load) of four, so other widths are loaded value by value and the
// compiler joins what it may.
template <int BS, typename T>
struct BlockColumn {
    T v[BS];
    __device__ __forceinline__ void load(const T* __restrict__ p) {
        if constexpr (BS == 4) {
            typedef T V __attribute__((ext_vector_type(BS), aligned(sizeof(T))));
            static_assert(sizeof(V) == BS * sizeof(T), "a column's load holds its values only");
            const V a = *(const V*)p;
#pragma unroll
            for (int m = 0; m < BS; ++m) v[m] = a[m];
        } else {
#pragma unroll
            for (int m = 0; m < BS; ++m) v[m] = p[m];
        }
    }
};

// Sum over the blocks of a row of their column j times x_j(c), c the block's column: eight
// blocks' loads in flight at once (a row has seven on a 3D grid).  x_of(c): x_j(c).
template <int BS, typename T, typename X>
__device__ __forceinline__ void row_times(int64_t p0, int64_t p1, int j, const int* __restrict__ col, const T* __restrict__ vals,
                                          const X& x_of, T* acc) {
    for (int64_t p = p0; p < p1; p += 8) {
        int c[8];
        BlockColumn<BS, T> a[8];
        T s[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) c[t] = col[p + t < p1 ? p + t : p1 - 1];
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const int64_t q = p + t < p1 ? p + t : p1 - 1;
            a[t].load(vals + ((size_t)q * BS + j) * BS);
            s[t] = x_of(c[t]);
        }
#pragma unroll
        for (int t = 0; t < 8; ++t)
            if (p + t < p1) {
#pragma unroll
                for (int m = 0; m < BS; ++m) acc[m] += a[t].v[m] * s[t];
            }
    }
}

}  // namespace

// bc = R (b - A x) and, where xc is given, the coarse level's sweep xc = omega Dc^-1 bc.  A
// quad of lanes takes a row, lane j its column j of every block; eight quads take the
// children of an aggregate (at most two per direction), so the restriction adds over the
// half-wave in registers.
template <typename T, int BS>
__global__ __launch_bounds__(256) void bsr_down_k(int Jc, const int* __restrict__ cptr, const int* __restrict__ cidx,
                                                  const int* __restrict__ pidx, const T* __restrict__ P,
                                                  const int64_t* __restrict__ rowptr, const int* __restrict__ col,
                                                  const T* __restrict__ vals, const T* __restrict__ b, const T* __restrict__ x,
                                                  T* __restrict__ bc, const T* __restrict__ Dc, T omega, T* __restrict__ xc) {
    const int lane = threadIdx.x & 63, j = lane & 3, q = (lane & 31) >> 2;
    const int I = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 2 + (lane >> 5);
    const bool in = I < Jc && j < BS;
    T acc[4] = {0, 0, 0, 0}, Pj[BS], Dj[BS], bj = 0;
    int row = -1;
#pragma unroll
    for (int m = 0; m < BS; ++m) { Pj[m] = 0; Dj[m] = 0; }
    if (in) {
        const int p = cptr[I] + q;
        if (p < cptr[I + 1]) row = cidx[p];
        if (xc) {
#pragma unroll
            for (int m = 0; m < BS; ++m) Dj[m] = Dc[((size_t)I * BS + m) * BS + j];
        }
    }
    if (row >= 0) {
        bj = b[(size_t)row * BS + j];
        const T* __restrict__ Pi = P + (size_t)pidx[row] * BS * BS + j;
#pragma unroll
        for (int m = 0; m < BS; ++m) Pj[m] = Pi[m * BS];
        row_times<BS>(rowptr[row], rowptr[row + 1], j, col, vals, [&](int c) { return x[(size_t)c * BS + j]; }, acc);
    }
    T t = quad_dot<BS>(Pj, bj - quad_transpose_sum(acc, j));
    if (row < 0) t = 0;
#pragma unroll
    for (int off = 4; off < 32; off <<= 1) t += __shfl_xor(t, off, 64);
    const T s = quad_dot<BS>(Dj, t);
    if (in && q == 0) {
        bc[(size_t)I * BS + j] = t;
        if (xc) xc[(size_t)I * BS + j] = omega * s;
    }
}

// xf += P y over the children of coarse row I: lane j of a quad, whose lanes hold y, takes
// component j; all children's loads before the first store
template <int BS, typename T>
__device__ __forceinline__ void prolong_children(const UpFine<T>& f, int I, int j, const T* y) {
    const int q1 = f.cptr[I + 1];
    for (int q = f.cptr[I]; q < q1; q += 8) {
        int i[8];
        T v[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) i[t] = f.cidx[q + t < q1 ? q + t : q1 - 1];
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const T* __restrict__ Pi = f.P + ((size_t)f.pidx[i[t]] * BS + j) * BS;
            v[t] = f.xf[(size_t)i[t] * BS + j];
#pragma unroll
            for (int n = 0; n < BS; ++n) v[t] += Pi[n] * y[n];
        }
#pragma unroll
        for (int t = 0; t < 8; ++t)
            if (q + t < q1) f.xf[(size_t)i[t] * BS + j] = v[t];
    }
}

// x = x0 + omega D^-1 (b - A x0), written to x or prolongated to the finer level's vector
template <typename T, int BS>
__global__ __launch_bounds__(256) void bsr_up_k(int nrows, const int64_t* __restrict__ rowptr, const int* __restrict__ col,
                                                const T* __restrict__ vals, const T* __restrict__ Dinv,
                                                const T* __restrict__ b, const T* __restrict__ x0, T omega,
                                                T* __restrict__ x, UpFine<T> f) {
    const int lane = threadIdx.x & 63, j = lane & 3;
    const int row = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 16 + (lane >> 2);
    const bool on = row < nrows && j < BS;
    T acc[4] = {0, 0, 0, 0}, Dj[BS], bj = 0, own = 0;
#pragma unroll
    for (int m = 0; m < BS; ++m) Dj[m] = 0;
    if (on) {
        bj = b[(size_t)row * BS + j];
        own = x0[(size_t)row * BS + j];
#pragma unroll
        for (int m = 0; m < BS; ++m) Dj[m] = Dinv[((size_t)row * BS + m) * BS + j];
        row_times<BS>(rowptr[row], rowptr[row + 1], j, col, vals, [&](int c) { return x0[(size_t)c * BS + j]; }, acc);
    }
    const T s = quad_dot<BS>(Dj, bj - quad_transpose_sum(acc, j));
    const T y = own + omega * s;
    const T yq[4] = {quad_move<0x00>(y), quad_move<0x55>(y), quad_move<0xAA>(y), quad_move<0xFF>(y)};
    if (!on) return;
    if (f.xf) prolong_children<BS>(f, row, j, yq);
    else x[(size_t)row * BS + j] = y;
}

// The coarsest level's dense solve, prolongated: xf += P (Ainv b).  A workgroup takes the BS
// rows of a cell, a wave a row (accumulated in double), and its first quad the children.
template <typename T, typename M, int BS>
__global__ __launch_bounds__(64 * BS) void dense_up_k(int n, const M* __restrict__ Ainv, const T* __restrict__ b, UpFine<T> f) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const M* __restrict__ Ar = Ainv + (size_t)(blockIdx.x * BS + wave) * n;
    double s0 = 0, s1 = 0;
    int c = 4 * lane;
    for (; c + 259 < n; c += 512) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            s0 += (double)Ar[c + e] * (double)b[c + e];
            s1 += (double)Ar[c + 256 + e] * (double)b[c + 256 + e];
        }
    }
    for (; c < n; c += 256)
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (c + e < n) s0 += (double)Ar[c + e] * (double)b[c + e];
    double s = s0 + s1;
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    __shared__ T y[BS];
    if (lane == 0) y[wave] = (T)s;
    __syncthreads();
    if (threadIdx.x < BS) {
        T yq[BS];
#pragma unroll
        for (int m = 0; m < BS; ++m) yq[m] = y[m];
        prolong_children<BS>(f, blockIdx.x, threadIdx.x, yq);
    }
}

template <typename T>
void bsr_down(bh_bsr* A, int Jc, const int* cptr, const int* cidx, const int* pidx, const T* P, const T* b, const T* x, T* bc,
              const T* Dc, double omega, T* xc) {
    const T* vals = (const T*)(sizeof(T) == 4 ? A->vals32.p : A->vals.p);
    const dim3 g((unsigned)((Jc + 7) / 8));
#define BH_CASE(B)                                                                                                          \
    case B:                                                                                                                 \
        hipLaunchKernelGGL((bsr_down_k<T, B>), g, dim3(256), 0, A->ctx->stream, Jc, cptr, cidx, pidx, P,                    \
                           A->rowptr.as<int64_t>(), A->col.as<int>(), vals, b, x, bc, Dc, (T)omega, xc);                    \
        break;
    switch (A->bs) {
        BH_CASE(3) BH_CASE(4)
        default: throw Error(-3, "multigrid leg: unsupported block size");
    }
#undef BH_CASE
    BH_HIP(hipGetLastError());
}

template <typename T>
void bsr_up(bh_bsr* A, const T* Dinv, const T* b, const T* x0, double omega, T* x, const UpFine<T>& f) {
    const T* vals = (const T*)(sizeof(T) == 4 ? A->vals32.p : A->vals.p);
    const dim3 g((unsigned)((A->nrows + 63) / 64));
#define BH_CASE(B)                                                                                                          \
    case B:                                                                                                                 \
        hipLaunchKernelGGL((bsr_up_k<T, B>), g, dim3(256), 0, A->ctx->stream, A->nrows, A->rowptr.as<int64_t>(),            \
                           A->col.as<int>(), vals, Dinv, b, x0, (T)omega, x, f);                                            \
        break;
    switch (A->bs) {
        BH_CASE(3) BH_CASE(4)
        default: throw Error(-3, "multigrid leg: unsupported block size");
    }
#undef BH_CASE
    BH_HIP(hipGetLastError());
}

template <typename T, typename M>
void dense_up(bh_ctx* ctx, int n, int bs, const M* Ainv, const T* b, const UpFine<T>& f) {
    BH_CHECK((bs == 3 || bs == 4) && n % bs == 0, "multigrid leg: unsupported block size");
    const dim3 g((unsigned)(n / bs));
    if (bs == 3) hipLaunchKernelGGL((dense_up_k<T, M, 3>), g, dim3(192), 0, ctx->stream, n, Ainv, b, f);
    else hipLaunchKernelGGL((dense_up_k<T, M, 4>), g, dim3(256), 0, ctx->stream, n, Ainv, b, f);
    BH_HIP(hipGetLastError());
}
template void dense_up<float, float>(bh_ctx*, int, int, const float*, const float*, const UpFine<float>&);
template void dense_up<float, double>(bh_ctx*, int, int, const double*, const float*, const UpFine<float>&);
template void dense_up<double, double>(bh_ctx*, int, int, const double*, const double*, const UpFine<double>&);

#define BH_INST(T)                                                                                                          \
    template void bsr_down<T>(bh_bsr*, int, const int*, const int*, const int*, const T*, const T*, const T*, T*, const T*, \
                              double, T*);                                                                                  \
    template void bsr_up<T>(bh_bsr*, const T*, const T*, const T*, double, T*, const UpFine<T>&);
BH_INST(float)
BH_INST(double)
#undef BH_INST

}  // namespace bh
