// The gridded march's rule of which rays it takes (generate.hip), for the
// kernels and for a check on the host.
#pragma once

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define MRAY_GRID_FN __host__ __device__ __forceinline__
#else
#define MRAY_GRID_FN inline
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

} // namespace mray
