// The arithmetic encoder's code as a ring of 16-bit digits (entropy.hip), for
// the kernel and for a check on the host. W supplies what the lanes of a
// wavefront do together: u32 (one value per lane) and its operations.
#pragma once

#include <stddef.h>
#include <stdint.h>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define MRAY_RING_FN __device__ __forceinline__
#else
#define MRAY_RING_FN inline
#endif

namespace mray
{

// A renormalisation shifts out two bytes, one digit. The newest digits are in
// the ring (128 of them); a carry adds 1 to the newest one without looking at
// it, and the digits are brought into [0, 2^16) when 64 of them leave the ring
// together (flush). At least 32 stay, so that a carry finds its digit in the
// ring.
template <typename W> struct DigitRing
{
    uint8_t *out;
    size_t cap;
    uint32_t *ring;
    uint32_t nd, flushed; // digits so far, and of them in out

    MRAY_RING_FN void put(uint32_t a)
    {
        if (W::first())
            ring[nd & 127u] = a;
        ++nd;
        if (__builtin_expect(nd - flushed >= 96u, 0))
            flush(64u);
    }

    MRAY_RING_FN void carry()
    {
        if (W::first() && nd > 0)
            W::add(&ring[(nd - 1u) & 127u], 1u);
    }

    // the next n <= 64 digits of the ring to out
    MRAY_RING_FN void flush(uint32_t n)
    {
        W::sync();
        typename W::u32 v = W::load(ring, flushed, n);
        uint32_t carried = 0;
        while (W::any_above(v, 0xFFFFu))
        {
            const typename W::u32 c = W::shift_right(v, 16);
            carried += W::lane0(c);
            v = W::plus(W::low_bits(v, 0xFFFFu), W::from_next(c));
        }
        if (carried)
        {
            // into the bytes already out
            W::fence();
            if (W::first())
            {
                size_t p = 2 * (size_t)flushed - 1;
                while (p < cap && out[p] == 0xFFu)
                    out[p--] = 0;
                if (p < cap)
                    out[p] = (uint8_t)(out[p] + 1);
            }
            W::fence();
        }
        W::store(out, cap, 2 * (size_t)flushed, v, n);
        flushed += n;
        W::sync();
    }

    MRAY_RING_FN void flush_all()
    {
        while (flushed < nd)
            flush(nd - flushed < 64u ? nd - flushed : 64u);
    }
};

} // namespace mray
