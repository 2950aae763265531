// FP64 building blocks of the MIXED preparation: G lanes (4, 8 or 16) hold a
// pixel, lane g elements gC .. gC + C - 1 of its arrays in registers. Every
// recursion is arranged so that one of its operands moves down by one element
// per step (shl: register renaming inside a lane, one DPP move across lanes)
// and the element a step needs in all lanes is always element 0 or 1
// (bcast0: one DPP move), so that no step reads LDS, sums over lanes or
// indexes registers at run time.
#pragma once

#include "mese_f64.hpp"

namespace mray
{

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

// LDS stride of a pixel's N complex doubles: odd, so that the pixels of a
// wavefront use different banks
constexpr int lattice_stride(int N) { return N | 1; }

} // namespace mray
