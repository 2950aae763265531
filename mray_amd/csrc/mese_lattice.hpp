// FP64 building blocks of the MIXED preparation and its reverse: G lanes (4, 8 or 16) hold a
// pixel, lane g elements gC .. gC + C - 1 of its arrays in registers. Every
// recursion is arranged so that one of its operands moves down by one element
// per step (shl: register renaming inside a lane, one DPP move across lanes)
// and the element a step needs in all lanes is always element 0 or 1
// (bcast0: one DPP move), so that no step reads LDS, sums over lanes or
// indexes registers at run time.
#pragma once

#include "device_common.hpp"

namespace mray
{

struct dc
{
    double x, y;
};

// Orders LDS accesses of the lanes of one wavefront (they execute in lockstep).
__device__ __forceinline__ void wave_sync() { __builtin_amdgcn_wave_barrier(); __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront"); }

// 1 / d by the hardware reciprocal and two Newton steps (within an ulp of
// the IEEE quotient; d is in (0, 1] here)
__device__ __forceinline__ double recip_nr(double d)
{
    double r = __builtin_amdgcn_rcp(d);
    r = fma(r, fma(-d, r, 1.0), r);
    return fma(r, fma(-d, r, 1.0), r);
}

template <int CTRL, int BANKS = 0xF> __device__ __forceinline__ double dpp_f64(double old, double v)
{
    int2 w, o;
    __builtin_memcpy(&w, &v, 8);
    __builtin_memcpy(&o, &old, 8);
    o.x = __builtin_amdgcn_update_dpp(o.x, w.x, CTRL, 0xF, BANKS, false);
    o.y = __builtin_amdgcn_update_dpp(o.y, w.y, CTRL, 0xF, BANKS, false);
    __builtin_memcpy(&v, &o, 8);
    return v;
}

// the value of the group's lane 0 in all its lanes
template <int G> __device__ __forceinline__ double bcast0(double v)
{
    if constexpr (G == 4)
        return dpp_f64<0x00>(v, v); // quad_perm 0 0 0 0
    else if constexpr (G == 16)
        return dpp_f64<0x150>(v, v); // row_newbcast:0
    else
        return dpp_f64<0x158, 0xC>(dpp_f64<0x150>(v, v), v); // lane 8 for the row's upper half
}

// the next lane's value; last: the group's last lane, which gets 0
template <int G> __device__ __forceinline__ double shl1(double v, bool last)
{
    const double n = (G == 4) ? dpp_f64<0xF9>(v, v) : dpp_f64<0x101>(v, v); // quad_perm 1 2 3 3, row_shl:1
    return last ? 0.0 : n;
}

template <int G> __device__ __forceinline__ dc bcast0(dc v) { return dc{bcast0<G>(v.x), bcast0<G>(v.y)}; }
template <int G> __device__ __forceinline__ dc shl1(dc v, bool last)
{
    return dc{shl1<G>(v.x, last), shl1<G>(v.y, last)};
}

// a b + c in registers of its own: where an array moves down by one element
// per step, the compiler's two-operand form would sum in place and copy
__device__ __forceinline__ double fma_moved(double a, double b, double c)
{
    double r;
    asm("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// the lane before's value; first: the group's lane 0, which gets 0
template <int G> __device__ __forceinline__ double shr1(double v, bool first)
{
    const double n = (G == 4) ? dpp_f64<0x90>(v, v) : dpp_f64<0x111>(v, v); // quad_perm 0 0 1 2, row_shr:1
    return first ? 0.0 : n;
}
template <int G> __device__ __forceinline__ dc shr1(dc v, bool first)
{
    return dc{shr1<G>(v.x, first), shr1<G>(v.y, first)};
}

// LDS stride of a pixel's N complex doubles: odd, so that the pixels of a
// wavefront use different banks
constexpr int lattice_stride(int N) { return N | 1; }

// 2 pi / j
struct TwoPiOver
{
    double v[256];
    constexpr TwoPiOver() : v()
    {
        v[0] = 0.0;
        for (int j = 1; j < 256; ++j)
            v[j] = 2.0 * kPi / j;
    }
};
static __constant__ TwoPiOver kTwoPiOver;

// The biased moments of a pixel (lerp in FP64: near the boundary of the moment
// space the recursions amplify a one-ulp change of the input) from memory in
// coalesced order through its LDS block (T, 2 S doubles) to the lanes' blocks,
// as the weights V_i = (i + 1) T_i+1 of the Herglotz recursion. Returns T_0
// (1/2 for a pixel without moments).
template <int G, int C>
__device__ __forceinline__ double load_weights(const float *__restrict__ mom, size_t off, int nm, double bias, int g,
                                               double *T, double (&V)[C])
{
#pragma unroll
    for (int r = 0; r < C; ++r)
    {
        const int e = G * r + g;
        const double v = (e < nm) ? (double)mom[off + e] : 0.0;
        T[e] = (e < nm) ? (1.0 - bias) * v + (e == 0 ? bias * 0.5 : 0.0) : 0.0;
    }
    T[G * C] = 0.0;
    wave_sync();
#pragma unroll
    for (int c = 0; c < C; ++c)
        V[c] = (double)(g * C + c + 1) * T[g * C + c + 1];
    const double t0 = (nm > 0) ? T[0] : 0.5;
    wave_sync();
    return t0;
}

// Herglotz transform: trigonometric -> exponential moments
// (trigonometricToExponentialMoments, src/mese/MESE_dynamic.h:35-54), into the
// pixel's LDS block E (zero from nm on, up to the next multiple of four of
// nw); e0 = E_0, not doubled.
template <int G, int C>
__device__ __forceinline__ void herglotz(const double (&V)[C], dc e0, int nw, int nm, int g, bool last, dc *E)
{
    static_assert((G * C) % 4 == 0, "E is read up to the next multiple of four");
    if (g == 0)
        E[0] = (nm > 0) ? e0 : dc{0.0, 0.0};
    dc X[C];
#pragma unroll
    for (int c = 0; c < C; ++c)
        X[c] = dc{V[c] * e0.x, V[c] * e0.y};
    for (int j = 1; j < nw; ++j)
    {
        const double f = kTwoPiOver.v[j];
        const dc x0 = bcast0<G>(X[0]);
        const dc ej = dc{-f * x0.y, f * x0.x};
        if (g == 0)
            E[j] = (j < nm) ? ej : dc{0.0, 0.0};
        const dc nx = shl1<G>(X[0], last);
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            const dc xn = (c + 1 < C) ? X[c + 1 < C ? c + 1 : 0] : nx;
            X[c] = dc{fma_moved(V[c], ej.x, xn.x), fma_moved(V[c], ej.y, xn.y)};
        }
    }
    if (g < 4 && nw + g < G * C)
        E[nw + g] = dc{0.0, 0.0};
    wave_sync();
}

// The lattice (levinsonsAlgorithm, src/mese/MESE_dynamic.h:100-135; see
// prepare.hip): F becomes the monic solution a_0 = 1, a_1, ..., rs = 1 / sigma
// (the solution's element 0). Returns the order: the entries of a that are
// not zero by the count or by the |u|^2 >= 1 guard.
template <int G, int C>
__device__ __forceinline__ int lattice(const dc *E, dc e0, int nw, int nm, int g, bool last, dc (&F)[C], double &rs)
{
    dc B[C];
#pragma unroll
    for (int c = 0; c < C; ++c)
    {
        const int i = g * C + c;
        const dc e = E[min(i, nw - 1)];
        F[c] = (i < nw) ? e : dc{0.0, 0.0};
        B[c] = (i < nw - 1) ? e : (i == nw - 1) ? dc{1.0, 0.0} : dc{0.0, 0.0};
        if (c == 0 && g == 0 && nw > 1)
            B[c] = dc{2.0 * e0.x, 0.0};
    }
    rs = 1.0 / (2.0 * e0.x);
    int order = nm;
    for (int L = (nw - 2) / C; L >= 0; --L)
    {
#pragma unroll
        for (int cs = C - 1; cs >= 0; --cs)
        {
            const int seam = L * C + cs; // nw - 2 - seam steps are done
            if (seam > nw - 2)
                continue;
            const int j = nw - 1 - seam;
            const dc f1 = bcast0<G>(F[1]);
            dc k = dc{-f1.x * rs, -f1.y * rs};
            double k2 = fma(k.x, k.x, k.y * k.y);
            if (j >= order || k2 >= 1.0)
            {
                k = dc{0.0, 0.0};
                k2 = 0.0;
                order = min(order, j);
            }
            rs *= recip_nr(1.0 - k2);
            const dc nx = shl1<G>(F[0], last);
#pragma unroll
            for (int c = 0; c < C; ++c)
            {
                const dc f = (c + 1 < C) ? F[c + 1 < C ? c + 1 : 0] : nx, b = B[c];
                F[c] = dc{fma(k.x, b.x, fma(-k.y, b.y, f.x)), fma(k.x, b.y, fma(k.y, b.x, f.y))};
                B[c] = dc{fma(k.x, f.x, fma(k.y, f.y, b.x)), fma(k.x, f.y, fma(-k.y, f.x, b.y))};
            }
            if (g == L)
                B[cs] = dc{k.x, -k.y};
        }
    }
    if (g == 0)
        F[0] = dc{1.0, 0.0};
    return order;
}

} // namespace mray
