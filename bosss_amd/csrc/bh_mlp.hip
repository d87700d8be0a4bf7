// Learned per-cell coarse correction: a 3-layer MLP (IN -> H -> H -> OUT,
// ReLU) evaluated per cell, BF16 weights with FP32 accumulation on MFMA
// (v_mfma_f32_16x16x32_bf16) for inference; FP32 forward/backward
// (v_mfma_f32_16x16x4_f32) and Adam for training, all on the device.  No reference counterpart (the reference
// has no learned components); it is an extra correction inside the
// preconditioner, guarded by residual minimisation with fallback to the plain
// multigrid (the acceptance rule of OrthonormalizationMultigrid.AddSol /
// MinimizeResidual, AS/OrthonormalizationMultigrid.cs:149-215).
//
// Feature map per cell j over its face adjacency (k-th mode residual r_jk,
// mean residual mode r_n0 of the 2D face neighbours n, diffusion nu):
//   s_j = sqrt(||r_j||^2 + sum_n r_n0^2) + tiny,
//   x_j = [ r_j / s_j , r_n0 / s_j for the 2D face neighbours (boundary: 0) ,
//           log10(nu_n / nu_j) for the same neighbours (boundary: +2) , 0-padding ]
// (Np + 4D inputs).  Output y_j maps to the correction e_j = s_j * (h_j^2 / nu_j) * y_j.
#include <algorithm>
#include <cmath>
#include <mutex>
#include <string>

#include "bh_internal.hpp"

#include "bh_mlp.hpp"

namespace bh {

// ------------------------------------------------------------------ bf16
__host__ __device__ inline uint16_t f32_to_bf16(float f) {
    uint32_t u;
    memcpy(&u, &f, 4);
    if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)(u >> 16);  // inf / nan
    u += 0x7fffu + ((u >> 16) & 1u);                                    // round to nearest even
    return (uint16_t)(u >> 16);
}
__host__ __device__ inline float bf16_to_f32(uint16_t b) {
    uint32_t u = (uint32_t)b << 16;
    float f;
    memcpy(&f, &u, 4);
    return f;
}

// ------------------------------------------------------------------ features
// X[j][:] as described above (fp32, row stride IN_P), scale s[j].
template <typename T, int D>
__global__ __launch_bounds__(256) void mlp_features_k(int J, int Np, int n0, int n1, int n2, const T* __restrict__ r,
                                                      const double* __restrict__ nu, int in_p, float* __restrict__ X,
                                                      float* __restrict__ s) {
    // one segment of in_p lanes (16 or 32) per cell: lane t of the segment owns
    // feature slot t (coalesced reads of the residual row and writes of the
    // feature row); the patch norm is a butterfly inside the segment
    const int segs = 256 / in_p;
    const int t = threadIdx.x & (in_p - 1);
    const int nn[3] = {n0, n1, n2};
    for (int j = blockIdx.x * segs + threadIdx.x / in_p; j < J; j += gridDim.x * segs) {
        int q[3];
        if (D == 2) { q[0] = j / n1; q[1] = j - q[0] * n1; q[2] = 0; }
        else { const int sl = n0 * n1; q[2] = j / sl; const int rr = j - q[2] * sl; q[1] = rr / n0; q[0] = rr - q[1] * n0; }
        // the neighbour across face f = 2d + side of slots Np + f and Np + 2D + f (-1: boundary)
        int nbc = -1;
        if (t >= Np && t < Np + 4 * D) {
            const int f = (t - Np) % (2 * D), d = f >> 1, side = f & 1;
            int qq[3] = {q[0], q[1], q[2]};
            qq[d] += side ? 1 : -1;
            if (qq[d] >= 0 && qq[d] < nn[d]) nbc = D == 2 ? qq[0] * n1 + qq[1] : qq[0] + qq[1] * n0 + qq[2] * n0 * n1;
        }
        double v = 0.0;
        if (t < Np) v = (double)r[(size_t)j * Np + t];
        else if (t < Np + 2 * D && nbc >= 0) v = (double)r[(size_t)nbc * Np];
        double sq = v * v;
        for (int off = in_p >> 1; off > 0; off >>= 1) sq += __shfl_xor(sq, off, 64);
        const double sc = sqrt(sq) + 1e-30;
        float out = 0.f;
        if (t < Np + 2 * D) {
            out = (float)(v / sc);
        } else if (t < Np + 4 * D) {
            out = nbc < 0 ? 2.0f : log10f((float)nu[nbc]) - log10f((float)nu[j]);
        }
        X[(size_t)j * in_p + t] = out;
        if (t == 0) s[j] = (float)sc;
    }
}

// correction e_j += w * s_j * (h_j^2/nu_j) * y_j  (h^2 = product of widths^(2/D))
template <typename T, int D>
__global__ void mlp_apply_scale_k(int J, int Np, int n0, int n1, const double* __restrict__ width, int nmax,
                                  const double* __restrict__ nu, const float* __restrict__ s, const float* __restrict__ Y,
                                  int out_p, T* __restrict__ e) {
    const int64_t tot = (int64_t)J * Np;
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < tot; t += (int64_t)gridDim.x * blockDim.x) {
        const int j = (int)(t / Np), m = (int)(t - (int64_t)j * Np);
        int idx[3];
        if (D == 2) { idx[0] = j / n1; idx[1] = j - idx[0] * n1; idx[2] = 0; }
        else { int sl = n0 * n1; idx[2] = j / sl; int rr = j - idx[2] * sl; idx[1] = rr / n0; idx[0] = rr - idx[1] * n0; }
        double vol = 1;
        for (int d = 0; d < D; ++d) vol *= width[d * nmax + idx[d]];
        const double h2 = pow(vol, 2.0 / D);
        e[t] = (T)((double)s[j] * h2 / nu[j] * (double)Y[(size_t)j * out_p + m]);
    }
}

// targets T[j][m] = e_jm / (s_j h_j^2 / nu_j)
template <int D>
__global__ void mlp_targets_k(int J, int Np, int n0, int n1, const double* __restrict__ width, int nmax,
                              const double* __restrict__ nu, const float* __restrict__ s, const double* __restrict__ e,
                              int out_p, float* __restrict__ Tg) {
    const int64_t tot = (int64_t)J * out_p;
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < tot; t += (int64_t)gridDim.x * blockDim.x) {
        const int j = (int)(t / out_p), m = (int)(t - (int64_t)j * out_p);
        if (m >= Np) { Tg[t] = 0.f; continue; }
        int idx[3];
        if (D == 2) { idx[0] = j / n1; idx[1] = j - idx[0] * n1; idx[2] = 0; }
        else { int sl = n0 * n1; idx[2] = j / sl; int rr = j - idx[2] * sl; idx[1] = rr / n0; idx[0] = rr - idx[1] * n0; }
        double vol = 1;
        for (int d = 0; d < D; ++d) vol *= width[d * nmax + idx[d]];
        const double h2 = pow(vol, 2.0 / D);
        Tg[t] = (float)(e[(size_t)j * Np + m] / ((double)s[j] * h2 / nu[j]));
    }
}

// upstream gradient of a loss L(e) through the correction map e_j = sigma_j y_j
// (sigma_j = s_j h_j^2 / nu_j): dY[j][m] = c * sigma_j * g[j][m], with g = dL/de / c
template <int D>
__global__ void mlp_upstream_k(int J, int Np, int n0, int n1, const double* __restrict__ width, int nmax,
                               const double* __restrict__ nu, const float* __restrict__ s, const double* __restrict__ g,
                               double c, int out_p, float* __restrict__ dY) {
    const int64_t tot = (int64_t)J * out_p;
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < tot; t += (int64_t)gridDim.x * blockDim.x) {
        const int j = (int)(t / out_p), m = (int)(t - (int64_t)j * out_p);
        if (m >= Np) { dY[t] = 0.f; continue; }
        int idx[3];
        if (D == 2) { idx[0] = j / n1; idx[1] = j - idx[0] * n1; idx[2] = 0; }
        else { int sl = n0 * n1; idx[2] = j / sl; int rr = j - idx[2] * sl; idx[1] = rr / n0; idx[0] = rr - idx[1] * n0; }
        double vol = 1;
        for (int d = 0; d < D; ++d) vol *= width[d * nmax + idx[d]];
        const double h2 = pow(vol, 2.0 / D);
        dY[t] = (float)(c * (double)s[j] * h2 / nu[j] * g[(size_t)j * Np + m]);
    }
}

// ------------------------------------------------------------------ inference (MFMA)
typedef float float4_t __attribute__((ext_vector_type(4)));
// four floats at any float's address: callers' arrays are only known to be float-aligned
typedef float float4_u __attribute__((ext_vector_type(4), aligned(4)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

// The layers are computed transposed, H^T = W X^T, on v_mfma_f32_16x16x32_bf16:
//   A (16 x 32, weights):      lane l holds A[l%16][8*(l/16) + j], j = 0..7
//   B (32 x 16, activations):  lane l holds B[8*(l/16) + j][l%16]
//   C (16 x 16):               lane l holds C[4*(l/16) + i][l%16], i = 0..3
// so a lane's outputs (units 16 t + 4 g + i of cell l%16, g = l/16) are, for two
// consecutive unit tiles t, eight of the inputs the next layer's B operand wants of
// the same cell: with the K slot (g, j) of step S standing for unit
// 32 S + 16 (j / 4) + 4 g + j % 4 (the weights are staged in that order) the
// activations go from one layer to the next in registers, without LDS or barriers.
// The weights sit in LDS as whole A fragments (consecutive lanes read consecutive
// 16-byte chunks, no bank conflicts); each fragment read serves the RT cell tiles
// (16 cells each) of a wave.
// Bound: a 16-cell tile needs 44 MFMA of 16 cycles and 44 KB of fragment reads per wave,
// so one tile per wave is LDS-bound and RT = 4 is bound by the matrix cores and
// the ReLU / rounding work (two conversions per unit and cell).  262144 cells, widths
// 22 -> 128 -> 128 -> 10: 21 us (570 TFLOP/s of BF16, 2.4 TB/s of rows); 200 us with
// 16x16x16 MFMA and the activations passed through an unpadded LDS tile (16-way bank
// conflicts on every read).
template <int INP, int H, int OUTP, int RT>
__global__ __launch_bounds__(256, 2) void mlp_infer_k(int J, const float* __restrict__ X, const uint16_t* __restrict__ W1t,
                                                      const float* __restrict__ b1, const uint16_t* __restrict__ W2t,
                                                      const float* __restrict__ b2, const uint16_t* __restrict__ W3t,
                                                      const float* __restrict__ b3, float* __restrict__ Y) {
    constexpr int WAVES = 4, NT = H / 16, KS = H / 32, OT = OUTP / 16;
    __shared__ __attribute__((aligned(16))) uint16_t sW1[NT * 512], sW2[NT * KS * 512], sW3[OT * KS * 512];
    __shared__ __attribute__((aligned(16))) float sb[2 * H + OUTP];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m = lane & 15, g = lane >> 4;
    // fragments: 16 bytes per lane, two 8-byte pieces of a weight row
    for (int i = tid; i < NT * 64; i += blockDim.x) {
        const int t = i >> 6, r = i & 15, q = (i >> 4) & 3;
        uint2 lo{0, 0}, hi{0, 0};
        if (8 * q < INP) {
            const uint2* src = (const uint2*)(W1t + (size_t)(16 * t + r) * INP + 8 * q);
            lo = src[0];
            hi = src[1];
        }
        ((uint4*)sW1)[i] = uint4{lo.x, lo.y, hi.x, hi.y};
    }
    auto stage = [&](uint16_t* dst, const uint16_t* src, int tiles) {
        for (int i = tid; i < tiles * KS * 64; i += blockDim.x) {
            const int t = i / (KS * 64), S = (i >> 6) % KS, r = i & 15, q = (i >> 4) & 3;
            const uint16_t* row = src + (size_t)(16 * t + r) * H + 32 * S + 4 * q;
            const uint2 lo = *(const uint2*)row, hi = *(const uint2*)(row + 16);
            ((uint4*)dst)[i] = uint4{lo.x, lo.y, hi.x, hi.y};
        }
    };
    stage(sW2, W2t, NT);
    stage(sW3, W3t, OT);
    for (int i = tid; i < H; i += blockDim.x) { sb[i] = b1[i]; sb[H + i] = b2[i]; }
    for (int i = tid; i < OUTP; i += blockDim.x) sb[2 * H + i] = b3[i];
    __syncthreads();
    const int ngroups = (J + 16 * RT - 1) / (16 * RT);
    for (int grp = blockIdx.x * WAVES + wave; grp < ngroups; grp += gridDim.x * WAVES) {
        const int c0 = grp * 16 * RT;
        // the lane offset is opaque per iteration, or the compiler keeps all fragments of the
        // loop in registers (256 VGPRs and 140 spilled) instead of reading them from LDS
        int fl = lane;
        asm volatile("" : "+v"(fl));
        const bf16x8_t* F1 = (const bf16x8_t*)sW1 + fl;
        const bf16x8_t* F2 = (const bf16x8_t*)sW2 + fl;
        const bf16x8_t* F3 = (const bf16x8_t*)sW3 + fl;
        const float* fb = sb + 4 * (fl >> 4);
        bf16x8_t xb[RT], h1[KS][RT], h2[KS][RT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            const int c = c0 + 16 * rt + m;
            float4_t lo{0, 0, 0, 0}, hi{0, 0, 0, 0};
            if (8 * g < INP && c < J) {
                const float4_u* src = (const float4_u*)(X + (size_t)c * INP + 8 * g);
                lo = src[0];
                hi = src[1];
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) { xb[rt][j] = (__bf16)lo[j]; xb[rt][4 + j] = (__bf16)hi[j]; }
        }
        auto relu_out = [&](const float4_t& a, bf16x8_t& f, int half) {
#pragma unroll
            for (int i = 0; i < 4; ++i) f[4 * half + i] = (__bf16)fmaxf(a[i], 0.f);
        };
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const bf16x8_t w = F1[t * 64];
            const float4_t bias = *(const float4_t*)(fb + 16 * t);
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
                relu_out(__builtin_amdgcn_mfma_f32_16x16x32_bf16(w, xb[rt], bias, 0, 0, 0), h1[t / 2][rt], t & 1);
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const float4_t bias = *(const float4_t*)(fb + H + 16 * t);
            float4_t acc[RT];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) acc[rt] = bias;
#pragma unroll
            for (int S = 0; S < KS; ++S) {
                const bf16x8_t w = F2[(t * KS + S) * 64];
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, h1[S][rt], acc[rt], 0, 0, 0);
            }
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) relu_out(acc[rt], h2[t / 2][rt], t & 1);
        }
#pragma unroll
        for (int t = 0; t < OT; ++t) {
            const float4_t bias = *(const float4_t*)(fb + 2 * H + 16 * t);
            float4_t acc[RT];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) acc[rt] = bias;
#pragma unroll
            for (int S = 0; S < KS; ++S) {
                const bf16x8_t w = F3[(t * KS + S) * 64];
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, h2[S][rt], acc[rt], 0, 0, 0);
            }
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const int c = c0 + 16 * rt + m;
                if (c < J) *(float4_u*)(Y + (size_t)c * OUTP + 16 * t + 4 * g) = acc[rt];
            }
        }
    }
}

// ------------------------------------------------------------------ training (FP32)
// Forward + backward on the FP32 matrix cores (v_mfma_f32_16x16x4_f32), one workgroup
// of 8 waves per tile of 32 cells, looping over tiles.  Weights used are the
// BF16-rounded values (as in inference), the activations stay FP32.  UPSTREAM: Tg
// holds dLoss/dy per cell (the loss is defined outside the network, e.g. the residual
// after the correction) and no loss is reported; otherwise Tg holds targets of the
// mean-squared error.
//
// Wave w owns hidden units 16 w .. 16 w + 15 of both hidden layers.  Operands of the MFMA:
//   A (16 x 4): lane l holds A[l%16][l/16],  B (4 x 16): lane l holds B[l/16][l%16],
//   C (16 x 16): lane l holds C[4*(l/16) + i][l%16], i = 0..3.
// The hidden layers' forward products take K in ascending order, so a preactivation is the
// chain of fused multiply-adds bias, k = 0, 1, ... (the MFMA rounds as that chain): a
// unit within rounding of its ReLU kink is on or off as in plain FP32 code, and one
// unit that differs moves the whole gradient by 1e-6.  Elsewhere the four K slots
// g = l/16 of four consecutive MFMA stand for the indices 16 S + 4 g + j (j the MFMA),
// so an operand that is contiguous along K is one 16-byte LDS read per four MFMA, and
// a wave's own output tile (C layout: cells 4 g + i, unit l%16) is, without any
// exchange, the A or B operand of the weight-gradient products, whose K index is
// the cell.  A wave's slices of the weights (forward and transposed) and
// its slices of the weight gradients stay in registers for all tiles; LDS
// holds only the activations of the tile (54 KB).  Per-workgroup gradient partials are
// written once (no atomics) and summed by mlp_reduce_k.
// Bound: 248 MFMA of 32 cycles per wave and tile at 2 waves per SIMD: 32768 cells are 4
// tiles per workgroup of 256, 26 us of MFMA issue.  Measured with the reduction: 61 us
// (73 TFLOP/s); 3270 us with one thread per hidden unit walking the cells one by one.
constexpr int TRT = 32;   // cells per tile
template <int INP, int H, int OUTP, bool UPSTREAM>
__global__ __launch_bounds__(512, 2) void mlp_train_k(int B, const int* __restrict__ idx, const float* __restrict__ X,
                                                      const float* __restrict__ Tg, int nout, const uint16_t* __restrict__ W1,
                                                      const float* __restrict__ b1, const uint16_t* __restrict__ W2,
                                                      const float* __restrict__ b2, const uint16_t* __restrict__ W3,
                                                      const float* __restrict__ b3, float* __restrict__ part,
                                                      float* __restrict__ lossp) {
    static_assert(H == 128, "8 waves of 16 hidden units");
    constexpr int RT = TRT / 16, IT = INP / 16, OT = OUTP / 16, HT = H / 16;
    constexpr int KSP = 8 / (RT * OT);         // output layer: K split over the waves left
    constexpr int SK = HT / KSP;               // ... into SK groups of 16 hidden units
    constexpr int LH = H + 4, LI = INP + 4, LO = OUTP + 4;
    __shared__ __attribute__((aligned(16))) float xs[TRT][LI], h1s[TRT][LH], h2s[TRT][LH], g2s[TRT][LH];
    __shared__ __attribute__((aligned(16))) float yp[KSP][TRT][OUTP], dys[TRT][LO];
    __shared__ float lred[8];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int m = lane & 15, g = lane >> 4;
    const int u = 16 * w + m;
    constexpr int NW = H * INP + H + H * H + H + OUTP * H + OUTP;
    // the wave's weights
    float w1[INP / 4], w2[H / 4], w2t[HT][4], w3t[OT][4], w3[SK][4];
    const int rt3 = w % RT, ot3 = (w / RT) % OT, ks3 = w / (RT * OT);
#pragma unroll
    for (int s = 0; s < INP / 4; ++s) w1[s] = bf16_to_f32(W1[u * INP + 4 * s + g]);
#pragma unroll
    for (int s = 0; s < H / 4; ++s) w2[s] = bf16_to_f32(W2[u * H + 4 * s + g]);
#pragma unroll
    for (int S = 0; S < HT; ++S)
#pragma unroll
        for (int j = 0; j < 4; ++j) w2t[S][j] = bf16_to_f32(W2[(16 * S + 4 * g + j) * H + u]);
#pragma unroll
    for (int S = 0; S < OT; ++S)
#pragma unroll
        for (int j = 0; j < 4; ++j) w3t[S][j] = bf16_to_f32(W3[(16 * S + 4 * g + j) * H + u]);
#pragma unroll
    for (int S = 0; S < SK; ++S)
#pragma unroll
        for (int j = 0; j < 4; ++j) w3[S][j] = bf16_to_f32(W3[(16 * ot3 + m) * H + 16 * (ks3 * SK + S) + 4 * g + j]);
    const float bias1 = b1[u], bias2 = b2[u];
    const float4_t z{0, 0, 0, 0};
    float4_t gW1[IT], gW2[HT], gW3[OT];
#pragma unroll
    for (int t = 0; t < IT; ++t) gW1[t] = z;
#pragma unroll
    for (int t = 0; t < HT; ++t) gW2[t] = z;
#pragma unroll
    for (int t = 0; t < OT; ++t) gW3[t] = z;
    float gb1 = 0, gb2 = 0, gb3 = 0, lacc = 0;
    const float dsc = 2.f / ((float)B * (float)nout);
    const int ntiles = (B + TRT - 1) / TRT;
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int s0 = tile * TRT;
        if (tid < TRT * INP / 4) {
            const int r = tid / (INP / 4), q = tid - r * (INP / 4);
            float4_t v = z;
            if (s0 + r < B) {
                const int c = idx ? idx[s0 + r] : s0 + r;
                v = *(const float4_u*)(X + (size_t)c * INP + 4 * q);
            }
            *(float4_t*)&xs[r][4 * q] = v;
        }
        __syncthreads();
        float4_t a1[RT], a2[RT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            a1[rt] = float4_t{bias1, bias1, bias1, bias1};
#pragma unroll
            for (int s = 0; s < INP / 4; ++s)
                a1[rt] = __builtin_amdgcn_mfma_f32_16x16x4f32(xs[16 * rt + m][4 * s + g], w1[s], a1[rt], 0, 0, 0);
        }
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                a1[rt][i] = fmaxf(a1[rt][i], 0.f);
                h1s[16 * rt + 4 * g + i][u] = a1[rt][i];
            }
        __syncthreads();
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) a2[rt] = float4_t{bias2, bias2, bias2, bias2};
#pragma unroll
        for (int s = 0; s < H / 4; ++s)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
                a2[rt] = __builtin_amdgcn_mfma_f32_16x16x4f32(h1s[16 * rt + m][4 * s + g], w2[s], a2[rt], 0, 0, 0);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                a2[rt][i] = fmaxf(a2[rt][i], 0.f);
                h2s[16 * rt + 4 * g + i][u] = a2[rt][i];
            }
        __syncthreads();
        {
            float4_t o = z;
#pragma unroll
            for (int S = 0; S < SK; ++S) {
                const float4_t a = *(const float4_t*)&h2s[16 * rt3 + m][16 * (ks3 * SK + S) + 4 * g];
#pragma unroll
                for (int j = 0; j < 4; ++j) o = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], w3[S][j], o, 0, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) yp[ks3][16 * rt3 + 4 * g + i][16 * ot3 + m] = o[i];
        }
        __syncthreads();
#pragma unroll
        for (int e = tid; e < TRT * OUTP; e += 512) {
            const int r = e / OUTP, o = e - r * OUTP;
            float d = 0.f;
            if (s0 + r < B && o < nout) {
                const int c = idx ? idx[s0 + r] : s0 + r;
                const float t = Tg[(size_t)c * OUTP + o];
                if (UPSTREAM) {
                    d = t;
                } else {
                    float y = b3[o];
#pragma unroll
                    for (int k = 0; k < KSP; ++k) y += yp[k][r][o];
                    const float diff = y - t;
                    d = dsc * diff;
                    lacc += diff * diff;
                }
            }
            dys[r][o] = d;
        }
        __syncthreads();
        // hidden layer 2: g2 = (dy W3) where h2 > 0; W3 and its bias
        float4_t g2[RT], g1[RT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            g2[rt] = z;
#pragma unroll
            for (int S = 0; S < OT; ++S) {
                const float4_t a = *(const float4_t*)&dys[16 * rt + m][16 * S + 4 * g];
#pragma unroll
                for (int j = 0; j < 4; ++j) g2[rt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], w3t[S][j], g2[rt], 0, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                g2[rt][i] = a2[rt][i] > 0.f ? g2[rt][i] : 0.f;
                gb2 += g2[rt][i];
                g2s[16 * rt + 4 * g + i][u] = g2[rt][i];
            }
#pragma unroll
            for (int t = 0; t < OT; ++t)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    gW3[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(dys[16 * rt + 4 * g + j][16 * t + m], a2[rt][j], gW3[t], 0, 0, 0);
        }
        if (tid < OUTP)
            for (int r = 0; r < TRT; ++r) gb3 += dys[r][tid];
        __syncthreads();
        // hidden layer 1: g1 = (g2 W2) where h1 > 0; then W2 and W1
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) g1[rt] = z;
#pragma unroll
        for (int S = 0; S < HT; ++S)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const float4_t a = *(const float4_t*)&g2s[16 * rt + m][16 * S + 4 * g];
#pragma unroll
                for (int j = 0; j < 4; ++j) g1[rt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], w2t[S][j], g1[rt], 0, 0, 0);
            }
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int t = 0; t < HT; ++t)
                    gW2[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(g2[rt][j], h1s[16 * rt + 4 * g + j][16 * t + m], gW2[t], 0, 0, 0);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float v = a1[rt][j] > 0.f ? g1[rt][j] : 0.f;
                gb1 += v;
#pragma unroll
                for (int t = 0; t < IT; ++t)
                    gW1[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(v, xs[16 * rt + 4 * g + j][16 * t + m], gW1[t], 0, 0, 0);
            }
        __syncthreads();
    }
    // partials: rows of a weight gradient are the wave's units (W3: the outputs)
    float* P = part + (size_t)blockIdx.x * NW;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = 16 * w + 4 * g + i;
#pragma unroll
        for (int t = 0; t < IT; ++t) P[r * INP + 16 * t + m] = gW1[t][i];
#pragma unroll
        for (int t = 0; t < HT; ++t) P[H * INP + H + r * H + 16 * t + m] = gW2[t][i];
#pragma unroll
        for (int t = 0; t < OT; ++t) P[H * INP + H + H * H + H + (16 * t + 4 * g + i) * H + u] = gW3[t][i];
    }
    gb1 += __shfl_xor(gb1, 16, 64);
    gb2 += __shfl_xor(gb2, 16, 64);
    gb1 += __shfl_xor(gb1, 32, 64);
    gb2 += __shfl_xor(gb2, 32, 64);
    if (g == 0) {
        P[H * INP + u] = gb1;
        P[H * INP + H + H * H + u] = gb2;
    }
    if (tid < OUTP) P[H * INP + H + H * H + H + OUTP * H + tid] = gb3;
    for (int off = 32; off > 0; off >>= 1) lacc += __shfl_xor(lacc, off, 64);
    if (lane == 0) lred[w] = lacc;
    __syncthreads();
    if (tid == 0) {
        float t = 0;
        for (int i = 0; i < 8; ++i) t += lred[i];
        lossp[blockIdx.x] = t;
    }
}

// grad[i] = sum over the nb partials, in a fixed order: a workgroup takes 64 consecutive
// entries, wave v the partials [v nb / 8, (v + 1) nb / 8), and the eight sums are added
// in wave order.  (One thread per entry walked all partials alone: 61 us for 256 x 22,672
// entries, a chain of dependent loads.)  grad_out (may be null) receives the same
// values.  The last workgroup, launched when loss is not null, adds the loss partials in
// block order in double, as the host does.
__global__ __launch_bounds__(512) void mlp_reduce_k(int nb, int nw, const float* __restrict__ part, float* __restrict__ grad,
                                                    float* __restrict__ grad_out, const float* __restrict__ lossp, double denom,
                                                    double* __restrict__ loss) {
    __shared__ float sm[512];
    const int lane = threadIdx.x & 63, v = threadIdx.x >> 6;
    if ((int)blockIdx.x == (nw + 63) / 64) {
        if ((int)threadIdx.x < nb) sm[threadIdx.x] = lossp[threadIdx.x];
        __syncthreads();
        if (threadIdx.x == 0) {
            double l = 0;
            for (int b = 0; b < nb; ++b) l += sm[b];
            *loss = l / denom;
        }
        return;
    }
    const int i = blockIdx.x * 64 + lane;
    float s = 0;
    if (i < nw) {
        const int p0 = v * nb / 8, p1 = (v + 1) * nb / 8;
#pragma unroll 8
        for (int b = p0; b < p1; ++b) s += part[(size_t)b * nw + i];
    }
    sm[threadIdx.x] = s;
    __syncthreads();
    if (v == 0 && i < nw) {
#pragma unroll
        for (int q = 1; q < 8; ++q) s += sm[64 * q + lane];
        grad[i] = s;
        if (grad_out) grad_out[i] = s;
    }
}

// Adam (Kingma & Ba 2015) on the flat FP32 master parameters
__global__ void adam_k(int n, float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m, float* __restrict__ v,
                       float lr, float b1, float b2, float eps, float c1, float c2) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const float gi = g[i];
        const float mi = b1 * m[i] + (1.f - b1) * gi;
        const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        w[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    }
}

// master FP32 (row = output unit) -> transposed BF16 inference copies
__global__ void mlp_to_bf16_k(int rows, int cols, const float* __restrict__ W, uint16_t* __restrict__ Wt) {
    // W[r][c] with r = output unit, c = input: the inference layout is also
    // [output unit][input] (B fragment = 4 consecutive inputs), i.e. the same order
    const int n = rows * cols;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) Wt[i] = f32_to_bf16(W[i]);
}

// ------------------------------------------------------------------ host
Mlp::Mlp(bh_ctx* c, int in_, int hid_, int out_, uint64_t seed) : ctx(c), in(in_), hid(hid_), out(out_) {
    BH_CHECK(hid == 128, "MLP: hidden width must be 128");
    in_p = (in + 15) / 16 * 16;
    out_p = (out + 15) / 16 * 16;
    BH_CHECK(in_p == 16 || in_p == 32, "MLP: input width must be <= 32");
    BH_CHECK(out_p == 16 || out_p == 32, "MLP: output width must be <= 32");
    nw = hid * in_p + hid + hid * hid + hid + out_p * hid + out_p;
    // He-uniform initialisation with a fixed LCG (padded rows/cols zero)
    std::vector<float> w(nw, 0.f);
    uint64_t st = seed * 6364136223846793005ULL + 1442695040888963407ULL;
    auto rnd = [&]() {
        st = st * 6364136223846793005ULL + 1442695040888963407ULL;
        return (double)(st >> 11) / 9007199254740992.0 * 2.0 - 1.0;
    };
    size_t o = 0;
    const double a1 = std::sqrt(6.0 / in), a2 = std::sqrt(6.0 / hid), a3 = std::sqrt(3.0 / hid) * 0.1;
    for (int r = 0; r < hid; ++r) for (int c = 0; c < in_p; ++c) w[o + r * in_p + c] = c < in ? (float)(a1 * rnd()) : 0.f;
    o += hid * in_p + hid;
    for (int r = 0; r < hid; ++r) for (int c = 0; c < hid; ++c) w[o + r * hid + c] = (float)(a2 * rnd());
    o += hid * hid + hid;
    for (int r = 0; r < out_p; ++r) for (int c = 0; c < hid; ++c) w[o + r * hid + c] = r < out ? (float)(a3 * rnd()) : 0.f;
    params.alloc(nw * sizeof(float));
    grad.alloc(nw * sizeof(float));
    m1.alloc(nw * sizeof(float));
    m2.alloc(nw * sizeof(float));
    wbf.alloc((hid * in_p + hid * hid + out_p * hid) * sizeof(uint16_t));
    set_params(w.data());
}

void Mlp::set_params(const float* w) {
    ctx->upload(params.p, w, nw * sizeof(float));
    BH_HIP(hipMemsetAsync(m1.p, 0, nw * sizeof(float), ctx->stream));
    BH_HIP(hipMemsetAsync(m2.p, 0, nw * sizeof(float), ctx->stream));
    step = 0;
    refresh_bf16();
}

void Mlp::refresh_bf16() {
    const float* P = params.as<float>();
    uint16_t* Wb = wbf.as<uint16_t>();
    hipLaunchKernelGGL(mlp_to_bf16_k, dim3(64), dim3(256), 0, ctx->stream, hid, in_p, P + off_W1(), Wb);
    hipLaunchKernelGGL(mlp_to_bf16_k, dim3(64), dim3(256), 0, ctx->stream, hid, hid, P + off_W2(), Wb + hid * in_p);
    hipLaunchKernelGGL(mlp_to_bf16_k, dim3(64), dim3(256), 0, ctx->stream, out_p, hid, P + off_W3(), Wb + hid * in_p + hid * hid);
    BH_HIP(hipGetLastError());
}

void Mlp::infer(int J, const float* X, float* Y) {
    const float* P = params.as<float>();
    const uint16_t* Wb = wbf.as<uint16_t>();
    // Cell tiles per wave: 4 (each weight fragment read from LDS serves four MFMA) once that
    // still gives every SIMD a wave (1024 waves of 64 cells), else 1 (more waves, shorter chains).
    // Persistent workgroups of 4 waves (two per CU, by registers) loop over their groups, so the
    // weight staging is paid once per workgroup.
    const bool wide = J >= 64 * 1024;
    const int groups = (J + (wide ? 63 : 15)) / (wide ? 64 : 16);
    const int blocks = std::max(1, std::min((groups + 3) / 4, 512));
#define BH_RUN(I, O, R)                                                                                             \
    hipLaunchKernelGGL((mlp_infer_k<I, 128, O, R>), dim3(blocks), dim3(256), 0, ctx->stream, J, X, Wb, P + off_b1(), \
                       Wb + hid * in_p, P + off_b2(), Wb + hid * in_p + hid * hid, P + off_b3(), Y)
#define BH_CASE(I, O)                          \
    if (in_p == I && out_p == O) {             \
        if (wide) BH_RUN(I, O, 4);             \
        else BH_RUN(I, O, 1);                  \
        BH_HIP(hipGetLastError());             \
        return;                                \
    }
    BH_CASE(16, 16) BH_CASE(16, 32) BH_CASE(32, 16) BH_CASE(32, 32)
#undef BH_CASE
#undef BH_RUN
    throw Error(-3, "MLP: unsupported widths");
}

// One training pass: mlp_train_k writes every entry of the nb per-block gradient
// partials and the nb loss partials, and mlp_reduce_k sums the partials in block
// order into grad (no atomics, so results do not depend on scheduling).
void Mlp::launch_gradient(int B, int nb, const int* idx, const float* X, const float* Tg, float* part, float* lossp,
                          bool upstream, float* grad_out, double* loss_dev) {
    const float* P = params.as<float>();
    const uint16_t* Wb = wbf.as<uint16_t>();
#define BH_RUN(I, O, U)                                                                                                  \
    hipLaunchKernelGGL((mlp_train_k<I, 128, O, U>), dim3(nb), dim3(512), 0, ctx->stream, B, idx, X, Tg, out, Wb, P + off_b1(), \
                       Wb + hid * in_p, P + off_b2(), Wb + hid * in_p + hid * hid, P + off_b3(), part, lossp)
#define BH_CASE(I, O)                        \
    if (in_p == I && out_p == O) {           \
        if (upstream) BH_RUN(I, O, true);    \
        else BH_RUN(I, O, false);            \
    } else
    BH_CASE(16, 16) BH_CASE(16, 32) BH_CASE(32, 16) BH_CASE(32, 32) { throw Error(-3, "MLP: unsupported widths"); }
#undef BH_CASE
#undef BH_RUN
    BH_HIP(hipGetLastError());
    hipLaunchKernelGGL(mlp_reduce_k, dim3((nw + 63) / 64 + (loss_dev ? 1 : 0)), dim3(512), 0, ctx->stream, nb, nw, part,
                       grad.as<float>(), grad_out, lossp, (double)B * out, loss_dev);
    BH_HIP(hipGetLastError());
}

double Mlp::gradient(int B, const int* idx, const float* X, const float* Tg) {
    const int nb = gradient_blocks(B);
    if (part.bytes < (size_t)nb * nw * sizeof(float)) part.alloc((size_t)256 * nw * sizeof(float));
    if (lossp.bytes < 256 * sizeof(float)) lossp.alloc(256 * sizeof(float));
    launch_gradient(B, nb, idx, X, Tg, part.as<float>(), lossp.as<float>(), false);
    std::vector<float> lp(nb);
    ctx->download(lp.data(), lossp.p, nb * sizeof(float));
    double l = 0;
    for (float v : lp) l += v;
    return l / ((double)B * out);
}

// Gradient of a loss defined outside the network from its upstream gradient dY
// [B][out_p] (first `out` columns used), into grad; same kernels and partials as
// gradient().
void Mlp::backward(int B, const float* X, const float* dY) {
    const int nb = gradient_blocks(B);
    if (part.bytes < (size_t)nb * nw * sizeof(float)) part.alloc((size_t)256 * nw * sizeof(float));
    if (lossp.bytes < 256 * sizeof(float)) lossp.alloc(256 * sizeof(float));
    launch_gradient(B, nb, nullptr, X, dY, part.as<float>(), lossp.as<float>(), true);
}

// ------------------------------------------------------------------ allocation-free gradient
// Fixed workspace of gradient_noalloc: the per-block gradient partials (at most
// 256 blocks of the largest parameter count the widths allow, in_p = out_p = 32)
// followed by the per-block loss partials.  One copy per GPU, 25.5 MB, held until
// the process ends.  In host code `scratch` is only a stand-in for the symbol:
// the kernels receive the device address that hipGetSymbolAddress returns for the
// current GPU (noalloc_ptr), never the array's name.
constexpr size_t kNoallocBlocks = 256;
constexpr size_t kNoallocMaxParams = 128 * 32 + 128 + 128 * 128 + 128 + 32 * 128 + 32;
constexpr size_t kNoallocFloats = kNoallocBlocks * kNoallocMaxParams + kNoallocBlocks;
static __device__ __align__(256) float scratch[kNoallocFloats];

constexpr int kMaxDevices = 64;
static float* noalloc_ptr[kMaxDevices] = {};
static std::mutex noalloc_mu;

size_t mlp_noalloc_capacity() { return kNoallocFloats; }

// Called once per context from bh_init, with the context's device current.
void mlp_noalloc_setup(int device) {
    BH_CHECK(device >= 0 && device < kMaxDevices, "bh_init: device index beyond the allocation-free workspace table");
    std::lock_guard<std::mutex> lock(noalloc_mu);
    if (noalloc_ptr[device]) return;
    void* p = nullptr;
    BH_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    BH_CHECK(p != nullptr, "bh_init: no device address for the allocation-free workspace");
    noalloc_ptr[device] = (float*)p;
}

void Mlp::gradient_noalloc(int B, const float* X, const float* Tg, float* grad_out, double* loss_dev) {
    const int nb = gradient_blocks(B);
    const size_t need = (size_t)nb * nw + (size_t)nb;
    BH_CHECK(need <= kNoallocFloats, "bh_mlp_gradient_noalloc: " + std::to_string(nb) + " blocks x " + std::to_string(nw) +
                                         " parameters exceed the fixed workspace of " + std::to_string(kNoallocFloats) +
                                         " floats");
    float* base = nullptr;
    {
        std::lock_guard<std::mutex> lock(noalloc_mu);
        base = (ctx->device >= 0 && ctx->device < kMaxDevices) ? noalloc_ptr[ctx->device] : nullptr;
    }
    BH_CHECK(base != nullptr, "bh_mlp_gradient_noalloc: the workspace of this GPU is not set up (bh_init)");
    float* part = base;
    float* lossp = base + (size_t)nb * nw;
    launch_gradient(B, nb, nullptr, X, Tg, part, lossp, false, grad_out, loss_dev);
}

void Mlp::adam(float lr) {
    ++step;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.f - std::pow(b1, (float)step), c2 = 1.f - std::pow(b2, (float)step);
    hipLaunchKernelGGL(adam_k, dim3((nw + 255) / 256), dim3(256), 0, ctx->stream, nw, params.as<float>(), grad.as<float>(),
                       m1.as<float>(), m2.as<float>(), lr, b1, b2, 1e-8f, c1, c2);
    BH_HIP(hipGetLastError());
    refresh_bf16();
}

void mlp_features(bh_op* op, const void* r, int prec, float* X, float* s, int in_p) {
    bh_grid* g = op->grid;
    const int J = g->J;
    BH_CHECK((in_p == 16 || in_p == 32) && op->Np + 4 * op->D <= in_p,
             "mlp_features: input width must be 16 or 32 and hold Np + 4 D features");
    const int segs = 256 / in_p;
    dim3 grd((J + segs - 1) / segs > 8192 ? 8192 : (J + segs - 1) / segs), blk(256);
    if (op->D == 2) {
        if (prec == BH_FP32) hipLaunchKernelGGL((mlp_features_k<float, 2>), grd, blk, 0, op->ctx->stream, J, op->Np, g->n[0], g->n[1], g->n[2], (const float*)r, op->nu.as<double>(), in_p, X, s);
        else hipLaunchKernelGGL((mlp_features_k<double, 2>), grd, blk, 0, op->ctx->stream, J, op->Np, g->n[0], g->n[1], g->n[2], (const double*)r, op->nu.as<double>(), in_p, X, s);
    } else {
        if (prec == BH_FP32) hipLaunchKernelGGL((mlp_features_k<float, 3>), grd, blk, 0, op->ctx->stream, J, op->Np, g->n[0], g->n[1], g->n[2], (const float*)r, op->nu.as<double>(), in_p, X, s);
        else hipLaunchKernelGGL((mlp_features_k<double, 3>), grd, blk, 0, op->ctx->stream, J, op->Np, g->n[0], g->n[1], g->n[2], (const double*)r, op->nu.as<double>(), in_p, X, s);
    }
    BH_HIP(hipGetLastError());
}

void mlp_correction(bh_op* op, const float* s, const float* Y, int out_p, void* e, int prec) {
    bh_grid* g = op->grid;
    const int64_t tot = (int64_t)g->J * op->Np;
    dim3 grd((unsigned)std::min<int64_t>((tot + 255) / 256, 8192)), blk(256);
    const double* w = g->d_width.as<double>();
    if (op->D == 2) {
        if (prec == BH_FP32) hipLaunchKernelGGL((mlp_apply_scale_k<float, 2>), grd, blk, 0, op->ctx->stream, g->J, op->Np, g->n[0], g->n[1], w, g->nmax, op->nu.as<double>(), s, Y, out_p, (float*)e);
        else hipLaunchKernelGGL((mlp_apply_scale_k<double, 2>), grd, blk, 0, op->ctx->stream, g->J, op->Np, g->n[0], g->n[1], w, g->nmax, op->nu.as<double>(), s, Y, out_p, (double*)e);
    } else {
        if (prec == BH_FP32) hipLaunchKernelGGL((mlp_apply_scale_k<float, 3>), grd, blk, 0, op->ctx->stream, g->J, op->Np, g->n[0], g->n[1], w, g->nmax, op->nu.as<double>(), s, Y, out_p, (float*)e);
        else hipLaunchKernelGGL((mlp_apply_scale_k<double, 3>), grd, blk, 0, op->ctx->stream, g->J, op->Np, g->n[0], g->n[1], w, g->nmax, op->nu.as<double>(), s, Y, out_p, (double*)e);
    }
    BH_HIP(hipGetLastError());
}

void mlp_upstream(bh_op* op, const float* s, const double* g, double c, int out_p, float* dY) {
    bh_grid* gr = op->grid;
    const int64_t tot = (int64_t)gr->J * out_p;
    dim3 grd((unsigned)std::min<int64_t>((tot + 255) / 256, 8192)), blk(256);
    const double* w = gr->d_width.as<double>();
    if (op->D == 2) hipLaunchKernelGGL((mlp_upstream_k<2>), grd, blk, 0, op->ctx->stream, gr->J, op->Np, gr->n[0], gr->n[1], w, gr->nmax, op->nu.as<double>(), s, g, c, out_p, dY);
    else hipLaunchKernelGGL((mlp_upstream_k<3>), grd, blk, 0, op->ctx->stream, gr->J, op->Np, gr->n[0], gr->n[1], w, gr->nmax, op->nu.as<double>(), s, g, c, out_p, dY);
    BH_HIP(hipGetLastError());
}

void mlp_targets(bh_op* op, const float* s, const double* e, int out_p, float* Tg) {
    bh_grid* g = op->grid;
    const int64_t tot = (int64_t)g->J * out_p;
    dim3 grd((unsigned)std::min<int64_t>((tot + 255) / 256, 8192)), blk(256);
    const double* w = g->d_width.as<double>();
    if (op->D == 2) hipLaunchKernelGGL((mlp_targets_k<2>), grd, blk, 0, op->ctx->stream, g->J, op->Np, g->n[0], g->n[1], w, g->nmax, op->nu.as<double>(), s, e, out_p, Tg);
    else hipLaunchKernelGGL((mlp_targets_k<3>), grd, blk, 0, op->ctx->stream, g->J, op->Np, g->n[0], g->n[1], w, g->nmax, op->nu.as<double>(), s, e, out_p, Tg);
    BH_HIP(hipGetLastError());
}

}  // namespace bh
