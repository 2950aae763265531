// The arithmetic decoder's choice of a symbol by the lanes of a wavefront
// (entropy.hip), for the kernel and for a check on the host.
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define MRAY_LANE_FN __host__ __device__ __forceinline__
#else
#define MRAY_LANE_FN inline
#endif

namespace mray
{

// What a lane holds for symbol k of an alphabet of A: the distribution d(k);
// as the end of the lane's last symbol (end) 1 for k = A, so that base + length
// * 1 is the reference's base + length; a NaN past the alphabet, where nothing
// qualifies.
MRAY_LANE_FN double lane_dist(uint32_t k, uint32_t A, double dk, bool end)
{
    return (k < A) ? dk : (end && k == A) ? 1.0 : __builtin_nan("");
}

// Whether a candidate whose interval starts at z may be the symbol of a code
// value v: the reference takes the last one that is not above v. Ordered, so
// that a NaN (no symbol) fails, also for the infinite v that a malformed code
// reaches (the value leaves the interval and grows by 2^16 per
// renormalisation).
MRAY_LANE_FN bool candidate(double z, double v) { return z <= v; }

// A lane's offer among its R symbols d[0 .. R - 1]: whether the first
// qualifies, the last that does and that one's interval
struct LaneOffer
{
    bool any;
    uint32_t sub;
    double x, y;
};
template <int R> MRAY_LANE_FN LaneOffer lane_offer(const double (&d)[R + 1], double base, double length, double v)
{
    double z[R + 1];
#pragma unroll
    for (int r = 0; r <= R; ++r)
        z[r] = base + length * d[r];
    LaneOffer o{candidate(z[0], v), 0u, z[0], z[1]};
#pragma unroll
    for (int r = 1; r < R; ++r)
    {
        const bool q = candidate(z[r], v);
        o.x = q ? z[r] : o.x;
        o.y = q ? z[r + 1 <= R ? r + 1 : R] : o.y;
        o.sub = q ? (uint32_t)r : o.sub;
    }
    return o;
}

} // namespace mray
