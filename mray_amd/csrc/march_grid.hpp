// The gridded march of generate.hip: its rule of which rays it takes and the
// weights it gives the grid's nodes, for the kernels and for a check on the host.
#pragma once

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define MRAY_GRID_FN __host__ __device__ __forceinline__
#else
#include <cmath>
#define MRAY_GRID_FN inline
using std::fma;
#endif

namespace mray
{

// how far from t = 0, in steps, a gridded ray may reach
constexpr float kGridReach = 8192.0f;

// Whether the march from t_near to t_far in steps of s resolves m moments on a
// uniform grid of phases: the largest order turns by at most 1 per step, and
// |t| <= 8192 s at both ends and so in between. There a float of t has 2^-10 s
// or less between neighbours, so t + s advances by s (1 +- 2^-11): the
// increments are uniform to that, and the march ends. t_near may be negative
// (a camera inside or behind the box with a negative znear), where a box
// reaching far behind the camera leaves t + s == t.
MRAY_GRID_FN bool grid_resolves(int m, float dphi, float t_near, float t_far, float s)
{
    return (float)(m - 1) * dphi <= 1.0f && t_far <= kGridReach * s && t_near >= -kGridReach * s && t_near + s < t_far;
}

// The grid's step at the node reached: t's float increment there and the
// reciprocal of the phase it spans.
struct GridStep
{
    float ds;
    double rstep;

    // the first increment; phase_per_t = pi / range
    MRAY_GRID_FN void start(float inc, double phase_per_t)
    {
        ds = inc;
        rstep = 1.0 / ((double)inc * phase_per_t);
    }

    // Where the increment changes to inc (rare; t passes a power of two): the
    // change of the step's phase. The stencils of the nodes that follow are
    // weighted for the new step: next to 8192 steps from t = 0 the segments
    // overlap by up to 2^-12 of a step and the step changes by 2^-11 of
    // itself, and with the first step kept a ray's moments were off by up to
    // 2e-7 (1.6e-8 now, from the nodes whose stencils span the change; the
    // sums node by node reach 4e-8 on their FP32 terms).
    MRAY_GRID_FN double change(float inc, double phase_per_t)
    {
        const double shift = ((double)inc - (double)ds) * phase_per_t;
        start(inc, phase_per_t);
        return shift;
    }

    // cpp c'' + cp c' as weights of the differences (WeightRing::push). Where
    // the step changes by `shift` behind the node, the second difference picks
    // up a first one.
    MRAY_GRID_FN double second(double cpp) const { return cpp * rstep * rstep; }
    MRAY_GRID_FN double first(double cp, double A, double shift) const
    {
        return fma(-1.2690476190476190 * A, shift, cp) * rstep;
    }
};

// Pending weights of the eight grid nodes around the newest one (the 9-point
// stencils of the first two derivatives, error (j Delta)^8 / 630 and / 3150 of
// the term). push adds node k's functional d c + cp c' + cpp c'' and returns
// the finished weight of node k - 4; A = cpp / Delta^2, B = cp / Delta. The
// ring moves on by writing each sum into the next slot (no copies).
struct WeightRing
{
    double w[8];

    // r = a b + c with r a register of its own (left to the compiler, each
    // sum is formed in its old slot's registers and copied over)
    static MRAY_GRID_FN void fma_to(double &r, double a, double b, double c)
    {
#if defined(__HIP_DEVICE_COMPILE__)
        asm("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "s"(a), "v"(b), "v"(c));
#else
        r = fma(a, b, c);
#endif
    }

    MRAY_GRID_FN WeightRing()
    {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            w[i] = 0.0;
    }

    MRAY_GRID_FN double push(double d, double A, double B)
    {
        constexpr double a0 = -205.0 / 72.0, a1 = 8.0 / 5.0, a2 = -1.0 / 5.0, a3 = 8.0 / 315.0, a4 = -1.0 / 560.0;
        constexpr double b1 = 4.0 / 5.0, b2 = -1.0 / 5.0, b3 = 4.0 / 105.0, b4 = -1.0 / 280.0;
        const double out = fma(a4, A, fma(-b4, B, w[0]));
        fma_to(w[0], a3, A, fma(-b3, B, w[1]));
        fma_to(w[1], a2, A, fma(-b2, B, w[2]));
        fma_to(w[2], a1, A, fma(-b1, B, w[3]));
        fma_to(w[3], a0, A, w[4] + d);
        fma_to(w[4], a1, A, fma(b1, B, w[5]));
        fma_to(w[5], a2, A, fma(b2, B, w[6]));
        fma_to(w[6], a3, A, fma(b3, B, w[7]));
        w[7] = fma(a4, A, b4 * B);
        return out;
    }

    MRAY_GRID_FN double pop()
    {
        const double out = w[0];
#pragma unroll
        for (int i = 0; i < 7; ++i)
            w[i] = w[i + 1];
        w[7] = 0.0;
        return out;
    }
};

} // namespace mray
