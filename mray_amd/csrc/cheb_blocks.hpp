// Chebyshev sums over moments by products: j = q P + r,
//     2 T_qP T_r = T_qP+r + T_qP-r.
// A series or a set of sums over T_0 .. T_M-1 of one x costs one operation per
// order in the products' basis and about P + 2 M / P more for T_r (r <= P) and
// T_qP, where the recurrences over the orders cost two per order. The change of
// basis (forwards for coefficients, transposed for sums) is a short alternating
// sum per order, done once per ray in FP64. P near sqrt(M).
#pragma once

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define MRAY_DEV __device__ __forceinline__
#else
#include <cmath>
#define MRAY_DEV inline
using std::fma;
#endif

namespace mray
{

template <int M> constexpr int block_width() { return M <= 12 ? 4 : M <= 30 ? 5 : M <= 56 ? 7 : M <= 72 ? 8 : 10; }

// T_1 .. T_P of x (T[0] is not written)
template <int P> MRAY_DEV void cheb_low(double (&T)[P + 1], double x)
{
    const double x2 = x + x;
    T[0] = 1.0;
    T[1] = x;
#pragma unroll
    for (int r = 2; r <= P; ++r)
        T[r] = fma(x2, T[r - 1], -T[r - 2]);
}

// a_qr += (w T_qP) T_r, j = FIRST .. M - 1
template <int M, int FIRST>
MRAY_DEV void block_sums(double (&a)[M], double w, const double (&T)[block_width<M>() + 1])
{
    constexpr int P = block_width<M>();
    const double y2 = T[P] + T[P];
    double z1 = w, z = w;
#pragma unroll
    for (int q = 0; q * P < M; ++q)
    {
        if (q == 1)
            z = w * T[P];
        else if (q > 1)
        {
            const double zn = fma(y2, z, -z1);
            z1 = z;
            z = zn;
        }
#pragma unroll
        for (int r = 0; r < P; ++r)
        {
            const int j = q * P + r;
            if (j >= M || j < FIRST)
                continue;
            if (r == 0)
                a[j] += z;
            else
                a[j] = fma(z, T[r], a[j]);
        }
    }
}

// sums over T_j from block_sums' products: s_qP+r = 2 a_qr - s_qP-r for q,
// r >= 1 (the other slots are products with T_0)
template <int M> MRAY_DEV void untangle_sums(double (&a)[M])
{
    constexpr int P = block_width<M>();
#pragma unroll
    for (int j = P + 1; j < M; ++j)
        if (j % P != 0)
            a[j] = fma(2.0, a[j], -a[j / P * P - j % P]);
}

// coefficients of the products from those of T_j (in place):
// c_qr = 2 mu_qP+r - c_(q+1)(P-r) for q, r >= 1, c_0r = mu_r - c_1(P-r) / 2
template <int M> MRAY_DEV void block_coefficients(double (&c)[M])
{
    constexpr int P = block_width<M>();
#pragma unroll
    for (int j = M - 1; j >= 1; --j)
    {
        const int q = j / P, r = j % P, partner = (q + 1) * P + P - r;
        if (r == 0)
            continue;
        const double other = (partner < M) ? c[partner < M ? partner : 0] : 0.0;
        c[j] = (q > 0) ? fma(2.0, c[j], -other) : fma(-0.5, other, c[j]);
    }
}

// sum_q T_qP sum_r c_qr T_r: Clenshaw's recurrence over q on T_P
template <int M>
MRAY_DEV double block_series(const double (&c)[M], const double (&T)[block_width<M>() + 1])
{
    constexpr int P = block_width<M>(), Q = (M + P - 1) / P;
    const double y2 = T[P] + T[P];
    double b1 = 0.0, b2 = 0.0;
#pragma unroll
    for (int q = Q - 1; q >= 0; --q)
    {
        double t = c[q * P];
        if (q < Q - 2)
            t -= b2;
        if (q < Q - 1)
            t = fma(q > 0 ? y2 : T[P], b1, t);
#pragma unroll
        for (int r = 1; r < P; ++r)
            if (q * P + r < M)
                t = fma(c[q * P + r < M ? q * P + r : 0], T[r], t);
        b2 = b1;
        b1 = t;
    }
    return b1;
}

} // namespace mray
