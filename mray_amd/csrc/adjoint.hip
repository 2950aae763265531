// Adjoint of the bounded-MESE preparation (MIXED, FP64): given dL/dlambda,
// dL/dmoments of lambda = prepare(moments) (prepare_mixed_kernel's
// mathematics: bias lerp, Herglotz transform, Toeplitz solve, autocorrelation,
// imaginary correlation; src/mese/MESE_dynamic.h:35-211). The reference has no
// gradients; this is new.
//
// With the solution P = P_0 a of T P = e_0 (T Hermitian Toeplitz, t_0 = 2 Re
// E_0, t_l = E_l), R_n = sum_j a_j conj(a_j+n) and
//     lambda_k = 2 P_0 Im sum_j R_k+j E_j,
// the reverse needs no recursion:
//  * R and E get the correlation and the convolution of dL/dlambda with each
//    other's values, and the solution g = dL/dP from R's and P_0's;
//  * dL = -Re(y^H dT P) with y = T^-1 g, by Gohberg and Semencul's formula,
//    T^-1 = (L(P) L(P)^H - L(Z) L(Z)^H) / P_0 with L(v) the lower triangular
//    Toeplitz matrix of first column v and Z = (0, conj(P_n-1) .. conj(P_1));
//    then dL/dt_l = -sum_k (y_k+l conj(P_k) + conj(y_k) P_k+l);
//  * E(z) = E_0 exp(2 pi i sum_l T_l z^l), so dL/dT_k = -2 pi Im sum_j
//    conj(dL/dE_j+k) E_j (half of it for T_0, through E_0).
// n is the order of the solution: where the |u|^2 >= 1 guard fired, the later
// reflection coefficients are the constant 0 and P solves the system of the
// order reached.
//
// Every pass but the forward's is a sum of shifted arrays, sum_k c_k S^k X, by
// Horner's rule: the accumulators move by one element per step (a renaming of
// registers and one DPP move, mese_lattice.hpp), X stays, and c_k is read from
// LDS, the same address in the pixel's lanes. 52 operations per element and
// step in all. G lanes per pixel: 4 up to 40 moments, then 8 and 16, so that
// the five arrays live at once fit two wavefronts per SIMD.
// Measured (512 x 512 pixels, 40 moments): 2.46 ms by the reverse sweep of
// the Levinson recursion this replaces, 1.00 ms now; bound by VALU issue.
#include <hip/hip_runtime.h>

#include "device_common.hpp"
#include "launch.hpp"
#include "mese_lattice.hpp"

namespace mray
{

namespace
{

// acc <- (acc moved down by one element) + c X
template <int G, int C>
__device__ __forceinline__ void horner_left(dc (&acc)[C], dc c, const dc (&X)[C], bool last)
{
    const dc nx = shl1<G>(acc[0], last);
#pragma unroll
    for (int i = 0; i < C; ++i)
    {
        const dc n = (i + 1 < C) ? acc[i + 1 < C ? i + 1 : 0] : nx;
        acc[i].x = fma(-c.y, X[i].y, fma_moved(c.x, X[i].x, n.x));
        acc[i].y = fma(c.y, X[i].x, fma_moved(c.x, X[i].y, n.y));
    }
}

// acc <- (acc moved up by one element) + c X
template <int G, int C>
__device__ __forceinline__ void horner_right(dc (&acc)[C], dc c, const dc (&X)[C], bool first)
{
    const dc px = shr1<G>(acc[C - 1], first);
#pragma unroll
    for (int i = C - 1; i >= 0; --i)
    {
        const dc n = (i > 0) ? acc[i > 0 ? i - 1 : 0] : px;
        acc[i].x = fma(-c.y, X[i].y, fma_moved(c.x, X[i].x, n.x));
        acc[i].y = fma(c.y, X[i].x, fma_moved(c.x, X[i].y, n.y));
    }
}

// acc += c X, in place
template <int C> __device__ __forceinline__ void add_scaled(dc (&acc)[C], dc c, const dc (&X)[C])
{
#pragma unroll
    for (int i = 0; i < C; ++i)
    {
        acc[i].x = fma(c.x, X[i].x, fma(-c.y, X[i].y, acc[i].x));
        acc[i].y = fma(c.x, X[i].y, fma(c.y, X[i].x, acc[i].y));
    }
}

template <int C> __device__ __forceinline__ void clear(dc (&a)[C])
{
#pragma unroll
    for (int i = 0; i < C; ++i)
        a[i] = dc{0.0, 0.0};
}

template <int C> __device__ __forceinline__ void store_block(dc *to, int g, const dc (&a)[C])
{
#pragma unroll
    for (int i = 0; i < C; ++i)
        to[g * C + i] = a[i];
    wave_sync();
}

__device__ __forceinline__ dc conj(dc a) { return dc{a.x, -a.y}; }

template <int G, int C>
__global__ __launch_bounds__(64, (C <= 10) ? 2 : 1) void prepare_adjoint_kernel(const float *__restrict__ mom,
                                                                                const uint32_t *__restrict__ index,
                                                                                int npix, int m, float bias,
                                                                                const float *__restrict__ grad_lag,
                                                                                float *__restrict__ grad_mom)
{
    constexpr int N = G * C, PX = 64 / G, S = lattice_stride(N);
    __shared__ dc lds_a[PX * S], lds_b[PX * S];
    const int lane = threadIdx.x;
    const int g = lane % G, q = lane / G;
    const bool first = g == 0, last = g == G - 1;
    const int pix = blockIdx.x * PX + q;
    const bool in = pix < npix;
    const int nm = in ? (index ? min((int)(index[pix + 1] - index[pix]), m) : m) : 0;
    const size_t off = in ? (index ? (size_t)index[pix] : (size_t)pix * m) : 0;
    int nw = nm;
#pragma unroll
    for (int o = G; o < 64; o <<= 1)
        nw = max(nw, __shfl_xor(nw, o, 64));
    nw = __builtin_amdgcn_readfirstlane(nw);
    if (nw == 0)
        return;
    dc *A = lds_a + q * S, *B = lds_b + q * S;
    double *Ad = reinterpret_cast<double *>(A);

    // ---- forward: E, a, 1 / sigma = P_0, R ----
    dc ED[C], aD[C], RD[C];
    double P0;
    int order;
    {
        double V[C];
        const double t0 = load_weights<G, C>(mom, off, nm, (double)bias, g, Ad, V);
        double sn, cs;
        sincos(kPi * t0 - 0.5 * kPi, &sn, &cs);
        const dc e0 = dc{cs * (0.25 / kPi), sn * (0.25 / kPi)};
        herglotz<G, C>(V, e0, nw, nm, g, last, A);
        order = lattice<G, C>(A, e0, nw, nm, g, last, aD, P0);
    }
#pragma unroll
    for (int c = 0; c < C; ++c)
    {
        const int i = g * C + c;
        const dc e = A[min(i, nw - 1)];
        ED[c] = (i < nm) ? e : dc{0.0, 0.0};
        if (i >= order)
            aD[c] = dc{0.0, 0.0};
    }
    if (first)
        B[N] = dc{0.0, 0.0};
    store_block<C>(B, g, aD);
    // conj(R)_n = sum_j conj(a_j) a_j+n
    clear<C>(RD);
    for (int j = nw - 1; j >= 0; --j)
        horner_left<G, C>(RD, conj(B[j]), aD, last);

    // ---- dL/dlambda into A, with it dL/dE (up to 2 P_0) through the imaginary
    // correlation and dL/dR (up to 2 P_0) ----
#pragma unroll
    for (int r = 0; r < C; ++r)
    {
        const int e = G * r + g;
        Ad[e] = (e < nm) ? (double)grad_lag[off + e] : 0.0;
    }
    wave_sync();
    dc EB[C], Rb[C];
    clear<C>(EB);
    clear<C>(Rb);
    for (int k = nw - 1; k >= 0; --k)
    {
        const double lb = Ad[k];
        const dc nx = shl1<G>(EB[0], last), px = shr1<G>(Rb[C - 1], first);
#pragma unroll
        for (int i = 0; i < C; ++i)
        {
            const dc n = (i + 1 < C) ? EB[i + 1 < C ? i + 1 : 0] : nx;
            EB[i].x = fma_moved(-lb, RD[i].y, n.x); // RD holds conj(R)
            EB[i].y = fma_moved(lb, RD[i].x, n.y);
        }
#pragma unroll
        for (int i = C - 1; i >= 0; --i)
        {
            const dc n = (i > 0) ? Rb[i > 0 ? i - 1 : 0] : px;
            Rb[i].x = fma_moved(lb, ED[i].y, n.x);
            Rb[i].y = fma_moved(lb, ED[i].x, n.y);
        }
    }
    // sum_k lb_k Im sum_j R_k+j E_j, for P_0's part
    double dot = 0.0;
#pragma unroll
    for (int c = 0; c < C; ++c)
        dot = fma(EB[c].x, ED[c].x, fma(EB[c].y, ED[c].y, dot));
#pragma unroll
    for (int o = 1; o < G; o <<= 1)
        dot += __shfl_xor(dot, o, 64);
    // R_n for n >= nm is no output's operand
#pragma unroll
    for (int c = 0; c < C; ++c)
        if (g * C + c >= nm)
            Rb[c] = dc{0.0, 0.0};
    wave_sync();

    // ---- g = dL/dP: sum_n (Rb_n a_j+n + conj(Rb_n) a_j-n), times 2, and P_0's ----
    store_block<C>(A, g, Rb);
    dc G1[C], G2[C];
    clear<C>(G1);
    clear<C>(G2);
    for (int k = nw - 1; k >= 0; --k)
    {
        const dc r = A[k];
        horner_left<G, C>(G1, r, aD, last);
        horner_right<G, C>(G2, conj(r), aD, first);
    }
#pragma unroll
    for (int c = 0; c < C; ++c)
    {
        const bool on = g * C + c < order;
        G1[c] = on ? dc{2.0 * (G1[c].x + G2[c].x), 2.0 * (G1[c].y + G2[c].y)} : dc{0.0, 0.0};
    }
    if (first)
        G1[0].x -= 2.0 * dot;

    // ---- y = T^-1 g (up to P_0): L(a)^H g and L(z)^H g, then L(a) and L(z) ----
    dc W1[C], W2[C];
    clear<C>(W1);
    clear<C>(W2);
    for (int k = nw - 1; k >= 0; --k)
    {
        // conj(z_k) = a_n-k, 0 for k = 0 (a_n) and k > n
        const dc a = B[k], z = B[k <= order ? order - k : N];
        horner_left<G, C>(W1, conj(a), G1, last);
        horner_left<G, C>(W2, z, G1, last);
    }
    dc Y[C];
    clear<C>(Y);
    for (int k = nw - 1; k >= 0; --k)
    {
        const dc a = B[k], z = conj(B[k <= order ? order - k : N]);
        horner_right<G, C>(Y, a, W1, first);
        add_scaled<C>(Y, dc{-z.x, -z.y}, W2);
    }
#pragma unroll
    for (int c = 0; c < C; ++c)
        if (g * C + c >= order)
            Y[c] = dc{0.0, 0.0};

    // ---- dL/dE += dL/dt: -P_0^2 sum_k (y_k+l conj(a_k) + conj(y_k) a_k+l) ----
    store_block<C>(A, g, Y);
#pragma unroll
    for (int c = 0; c < C; ++c)
        aD[c] = B[g * C + c];
    dc D[C];
    clear<C>(D);
    for (int k = nw - 1; k >= 0; --k)
    {
        const dc a = B[k], y = A[k];
        horner_left<G, C>(D, conj(a), Y, last);
        add_scaled<C>(D, conj(y), aD);
    }
    const double s1 = 2.0 * P0, s2 = -(P0 * P0);
#pragma unroll
    for (int c = 0; c < C; ++c)
    {
        const bool on = g * C + c < nm;
        EB[c] = on ? dc{fma(s2, D[c].x, s1 * EB[c].x), fma(s2, D[c].y, s1 * EB[c].y)} : dc{0.0, 0.0};
    }
    wave_sync();

    // ---- dL/dT_k = -2 pi Im sum_j conj(EB_j+k) E_j ----
    store_block<C>(A, g, ED);
    double TB[C];
#pragma unroll
    for (int c = 0; c < C; ++c)
        TB[c] = 0.0;
    for (int j = nw - 1; j >= 0; --j)
    {
        const dc e = A[j];
        const double nx = shl1<G>(TB[0], last);
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            const double n = (c + 1 < C) ? TB[c + 1 < C ? c + 1 : 0] : nx;
            TB[c] = fma(-EB[c].y, e.x, fma_moved(EB[c].x, e.y, n));
        }
    }
    wave_sync();
#pragma unroll
    for (int c = 0; c < C; ++c)
        Ad[g * C + c] = TB[c];
    wave_sync();
    const double scale = -2.0 * kPi * (1.0 - (double)bias);
#pragma unroll
    for (int r = 0; r < C; ++r)
    {
        const int e = G * r + g;
        if (e < nm)
            grad_mom[off + e] = (float)((e == 0 ? 0.5 * scale : scale) * Ad[e]);
    }
}

} // namespace

int launch_prepare_adjoint(const float *moments, const uint32_t *index, int W, int H, int m, float bias,
                           const float *grad_lagrange, float *grad_moments, hipStream_t stream)
{
    const int npix = W * H;
#define MRAY_PADJ_CASE(GG, CC)                                                                                        \
    if (m <= GG * CC)                                                                                                 \
    {                                                                                                                 \
        hipLaunchKernelGGL((prepare_adjoint_kernel<GG, CC>), dim3((npix + 64 / GG - 1) / (64 / GG)), dim3(64), 0,     \
                           stream, moments, index, npix, m, bias, grad_lagrange, grad_moments);                       \
        return 0;                                                                                                     \
    }
    MRAY_PADJ_CASE(4, 2)
    MRAY_PADJ_CASE(4, 4)
    MRAY_PADJ_CASE(4, 5)
    MRAY_PADJ_CASE(4, 6)
    MRAY_PADJ_CASE(4, 7)
    MRAY_PADJ_CASE(4, 8)
    MRAY_PADJ_CASE(4, 9)
    MRAY_PADJ_CASE(4, 10)
    MRAY_PADJ_CASE(8, 6)
    MRAY_PADJ_CASE(8, 7)
    MRAY_PADJ_CASE(8, 8)
    MRAY_PADJ_CASE(8, 10)
    MRAY_PADJ_CASE(16, 6)
    MRAY_PADJ_CASE(16, 7)
    MRAY_PADJ_CASE(16, 8)
    MRAY_PADJ_CASE(16, 10)
    MRAY_PADJ_CASE(16, 13)
    MRAY_PADJ_CASE(16, 16)
#undef MRAY_PADJ_CASE
    return MRAY_ERR_UNSUPPORTED;
}

} // namespace mray
