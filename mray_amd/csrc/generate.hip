// Moment generation: ray march accumulating bounded trigonometric moments of
// the density along each ray (src/raymarch_generate.h:35-148).
//
// Two forms share the sample loop (pixel ray, slab test, t loop, trilinear
// fetch, map_density, min/max bound) so both see exactly the reference's
// samples and produce its 16-bit bounds bit for bit:
//
//  PLAIN  the reference's per-segment update_moments: 2(m-1) sin/cos per
//         sample, one thread per ray, accumulators in LDS (what a direct port
//         of generate_moments_kernel does).
//
//  MIXED  the same integral written per node instead of per segment. For
//         contiguous segments with slopes g_s the i/j terms telescope and
//             trig_j = (1/j^2) sum_k (g_k - g_{k+1}) cos(j phi_k)
//                      - (f_0 / j) sin(j phi_0).
//         The reference's segments are [p_k - dphi, p_k] with p_k recomputed
//         from t, so neighbours overlap by a few ulp (delta), and its lines
//         use the slope (f_k - f_{k-1}) / dphi, so they miss f_k by a few ulp
//         (eps); both enter to first order, their squares are ~1e-13 (more
//         where t is thousands of steps, see GridStep):
//             + sum_k [ -delta_k f_k cos(j p_k) + h_k sin(j p_k) / j ].
//         Two marches sum these terms. Where the samples resolve the largest
//         order (almost every ray), the ulp-sized terms become weights of
//         plain cosines on the ray's uniform phase grid (WeightRing), and a
//         moment costs one FP64 operation per node (block_sums); the
//         other rays are summed node by node from each node's own phasor,
//         five operations per moment (accumulate_node). gfx950 issues FP64
//         FMAs at the rate of unpacked FP32 ones, so the cosine sums and
//         trig_0 (the exact integral of the reference's lines) are FP64; the
//         moments are rounded to float once. Moments live in registers
//         (template M >= m); more than 60 are split into chunks over
//         workgroups (CHUNK).
#include "cheb_blocks.hpp"
#include "device_common.hpp"
#include "launch.hpp"
#include "march_grid.hpp"
#include "sph_common.hpp"
#include <type_traits>

namespace mray
{

struct GenArgs
{
    int W, H, m;
    float step;
    float data_min, data_max;
    float data_rinv; // host_reciprocal(data_max - data_min)
    int transform_to_bounds;
    int compact_image;
    float bound_eps;
};

// Sample at t along r (origin + t * dir in float, as the reference).
template <typename T>
__device__ __forceinline__ float sample_at(const VolumeView<T> &vol, const Ray &r, float t, const GenArgs &a)
{
    float px = r.o.x + t * r.d.x, py = r.o.y + t * r.d.y, pz = r.o.z + t * r.d.z;
    return map_density(sample_volume(vol, px, py, pz), a.data_min, a.data_max);
}

// ---------------------------------------------------------------------------
// PLAIN
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void generate_plain_kernel(VolumeView<T> vol, DevCamera cam, GenArgs a,
                                                             float *__restrict__ out, uint32_t *__restrict__ bounds,
                                                             int32_t *__restrict__ samples,
                                                             float2 *__restrict__ ray_range)
{
    extern __shared__ float lds_trig[]; // [m][blockDim.x], strided per thread
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int stride = blockDim.x;
    const uint32_t ntiles = ((a.W + 7) / 8) * ((a.H + 7) / 8);
    const uint32_t tile = xcd_tile_block(a.W, blockDim.x / 64) * (blockDim.x / 64) + (tid >> 6);
    if (tile >= ntiles)
        return;
    int x, y;
    tile_pixel(tile, a.W, lane, x, y);
    if (x >= a.W || y >= a.H)
        return;
    const int m = a.m;
    float *trig = lds_trig + tid;
#define TRIG(j) trig[(j)*stride]
    for (int j = 0; j < m; ++j)
        TRIG(j) = 0.0f;

    Ray r = pixel_ray(cam, a.W, a.H, x, y);
    float t_near, t_far;
    bool hit = intersect_aabb(r, vol.dmin, vol.dmax, t_near, t_far);
    t_near = rmax(t_near, cam.znear);
    size_t pix = (size_t)y * a.W + x;
    float *mo = out + pix * (size_t)m;
    if (!(hit && (t_far > 0)))
    {
        if (!(a.transform_to_bounds && a.compact_image))
            for (int j = 0; j < m; ++j)
                mo[j] = 0.f;
        if (bounds)
            bounds[pix] = 0;
        if (ray_range)
            ray_range[pix] = make_float2(0.0f, 1.0f);
        if (samples)
            samples[pix] = 0;
        return;
    }
    const float s = a.step;
    float lo = 1.f, hi = 0.f;
    float t = t_near;
    float pi_trange_inv = (float)(kPi / (double)(t_far - t_near));
    float p = (float)(-kPi);
    float dphi = (float)(kPi * (double)(s / (t_far - t_near)));
    float fs = sample_at(vol, r, t, a);
    int ns = 1;
    lo = rmin(lo, fs);
    hi = rmax(hi, fs);

    auto update = [&](float p_next, float step_size, float f0, float f1) {
        // update_moments (src/raymarch_generate.h:35-58)
        float p_prev = p_next - step_size;
        float gradient = (f1 - f0) / step_size;
        float yint = f0 - gradient * p_prev;
        for (int j = 1; j < m; ++j)
        {
            float jf = (float)j;
            float jSq = jf * jf;
            float csx = gradient / jSq, csy = yint / jf;
            float sn, cn, sp, cp;
            sincosf(-jf * p_next, &sn, &cn);
            sincosf(-jf * p_prev, &sp, &cp);
            float ay = csy + gradient * jf * p_next / jSq;
            float by = csy + gradient * jf * p_prev / jSq;
            float acc = TRIG(j);
            acc += (csx + 0.0f) * cn - ay * sn;
            acc -= (csx + 0.0f) * cp - by * sp;
            TRIG(j) = acc;
        }
        float t0 = TRIG(0);
        t0 = (float)((double)t0 + (0.5 * gradient * (double)(p_next * p_next) + (double)(yint * p_next)));
        t0 = (float)((double)t0 - (0.5 * gradient * (double)(p_prev * p_prev) + (double)(yint * p_prev)));
        TRIG(0) = t0;
    };

    float bs;
    const int cap = march_cap(t_near, t_far, s);
    for (int it = 0; t + s < t_far && it < cap; ++it)
    {
        t += s;
        p = (float)((double)((t - t_near) * pi_trange_inv) - kPi);
        bs = sample_at(vol, r, t, a);
        ++ns;
        lo = rmin(lo, bs);
        hi = rmax(hi, bs);
        update(p, dphi, fs, bs);
        fs = bs;
    }
    float last_step = 0.0f - p;
    bs = sample_at(vol, r, t_far, a);
    ++ns;
    lo = rmin(lo, bs);
    hi = rmax(hi, bs);
    update(0.0f, last_step, fs, bs);

    // normalisation (src/raymarch_generate.h:116-135)
    if (a.transform_to_bounds)
    {
        lo = rmax(lo - a.bound_eps, 0.0f);
        hi = rmin(hi + a.bound_eps, 1.0f);
        double inv = 1.0 / (double)(hi - lo);
        mo[0] = (float)((double)(TRIG(0) * kInvPiF - lo) * inv);
        for (int j = 1; j < m; ++j)
            mo[j] = (float)((double)(TRIG(j) * kInvPiF) * inv);
    }
    else
        for (int j = 0; j < m; ++j)
            mo[j] = TRIG(j) * kInvPiF;
#undef TRIG
    if (bounds)
        bounds[pix] = pack_bound(lo, hi);
    if (ray_range)
        ray_range[pix] = make_float2(lo, hi);
    if (samples)
        samples[pix] = ns;
}

// ---------------------------------------------------------------------------
// MIXED
// ---------------------------------------------------------------------------

// The chunk j0 .. j0 + M - 1 of a march whose moments are split into chunks:
// sc_i += w cos((j0 + i) q_n) by the recurrence from w cos(j0 q_n) and
// w cos((j0 + 1) q_n) (c0, c1), two operations per moment.
template <int M> __device__ __forceinline__ void accumulate_chunk(double (&sc)[M], double w, double x, double c0, double c1)
{
    const double x2 = x + x;
    double v1 = w * c0, v = w * c1;
    sc[0] += v1;
    sc[1] += v;
#pragma unroll
    for (int i = 2; i < M; ++i)
    {
        const double n = fma(x2, v, -v1);
        v1 = v;
        v = n;
        sc[i] += v;
    }
}

// One node of an exactly summed ray (see the kernel), its terms at its own phase,
// moments j = 1..M-1:
//     sc[j] += (d + j^2 e) cos(j phi)   (FP64)
//     ss[j] += h sin(j phi)             (FP32)
// the moment being (sc[j] + j ss[j]) / j^2. cos(j phi) by the Chebyshev
// recurrence v_j = 2x v_{j-1} - v_{j-2} in FP64 from x = cos(phi) (gfx950
// issues FP64 FMAs at the rate of unpacked FP32 ones); the sine terms carry
// only the first-order corrections of the reference's ulp offsets (h is a few
// ulps of the slopes), so their recurrence from y = sin(phi) and their sums
// are FP32. The weight d + j^2 e is built up by the odd numbers,
// w_j = w_{j-1} + (2j - 1) e, one FMA whose small odd factor is an
// instruction literal (an FMA by j^2 into a fresh register would need a copy
// of d first: gfx950's three-operand forms take no literal): five operations
// and three registers per moment.
template <int M>
__device__ __forceinline__ void accumulate_node(double (&sc)[M], float (&ss)[M], double d, double e, float h,
                                                double x, float y)
{
    const double x2 = x + x;
    const float x2f = (float)x2;
    double cm2 = 1.0, cm1 = x;
    float sm2 = 0.0f, sm1 = y;
    double w = d + e;
    sc[1] = fma(w, cm1, sc[1]);
    ss[1] = __builtin_fmaf(h, sm1, ss[1]);
#pragma unroll
    for (int j = 2; j < M; ++j)
    {
        const double c = fma(x2, cm1, -cm2);
        const float sn = __builtin_fmaf(x2f, sm1, -sm2);
        w = fma((double)(2 * j - 1), e, w);
        sc[j] = fma(w, c, sc[j]);
        ss[j] = __builtin_fmaf(h, sn, ss[j]);
        cm2 = cm1;
        cm1 = c;
        sm2 = sm1;
        sm1 = sn;
    }
}

// accumulate_node for the moment chunk j = j0 + i, i = 0..M-1, of a march
// whose moments are split into chunks (more than fit in one thread's
// registers): (c0, s0) and (c1, s1) are cos and sin of j0 phi and (j0 + 1) phi,
// the recurrences run from there. The weight d + j^2 e = D + i E2 + i^2 e
// (D = d + j0^2 e, E2 = 2 j0 e) is built up as w_i = w_{i-1} + (2i - 1) e
// + E2: one operation per moment more than accumulate_node's. Slot i = 0 of
// the chunk j0 = 0 (moment 0) gets d, which nothing reads.
template <int M>
__device__ __forceinline__ void accumulate_node_chunk(double (&sc)[M], float (&ss)[M], double d, double e, float h,
                                                      double x, double c0, float s0, double c1, float s1, double j0)
{
    const double x2 = x + x;
    const float x2f = (float)x2;
    const double D = fma(j0 * j0, e, d);
    const double E2 = (j0 + j0) * e;
    double cm2 = c0, cm1 = c1;
    float sm2 = s0, sm1 = s1;
    double w = D;
    sc[0] = fma(w, c0, sc[0]);
    ss[0] = __builtin_fmaf(h, s0, ss[0]);
#pragma unroll
    for (int i = 1; i < M; ++i)
    {
        double c;
        float sn;
        if (i == 1)
        {
            c = c1;
            sn = s1;
        }
        else
        {
            c = fma(x2, cm1, -cm2);
            sn = __builtin_fmaf(x2f, sm1, -sm2);
            cm2 = cm1;
            cm1 = c;
            sm2 = sm1;
            sm1 = sn;
        }
        w = fma((double)(2 * i - 1), e, w) + E2;
        sc[i] = fma(w, c, sc[i]);
        ss[i] = __builtin_fmaf(h, sn, ss[i]);
    }
}

// accumulate_node_chunk for a chunk start J0 known at compile time: the
// weight d + j^2 e continues the odd-number recurrence of accumulate_node
// from D = d + J0^2 e, w_j = w_{j-1} + (2j - 1) e with the odd factor an
// instruction literal, five operations per moment as in the first chunk.
template <int M, int J0>
__device__ __forceinline__ void accumulate_node_chunk_c(double (&sc)[M], float (&ss)[M], double d, double e, float h,
                                                        double x, double c0, float s0, double c1, float s1)
{
    const double x2 = x + x;
    const float x2f = (float)x2;
    double cm2 = c0, cm1 = c1;
    float sm2 = s0, sm1 = s1;
    double w = fma((double)(J0 * J0), e, d);
    sc[0] = fma(w, c0, sc[0]);
    ss[0] = __builtin_fmaf(h, s0, ss[0]);
#pragma unroll
    for (int i = 1; i < M; ++i)
    {
        double c;
        float sn;
        if (i == 1)
        {
            c = c1;
            sn = s1;
        }
        else
        {
            c = fma(x2, cm1, -cm2);
            sn = __builtin_fmaf(x2f, sm1, -sm2);
            cm2 = cm1;
            cm1 = c;
            sm2 = sm1;
            sm1 = sn;
        }
        w = fma((double)(2 * (J0 + i) - 1), e, w);
        sc[i] = fma(w, c, sc[i]);
        ss[i] = __builtin_fmaf(h, sn, ss[i]);
    }
}

// a value of another lane of the quad (CTRL: quad_perm)
template <int CTRL> __device__ __forceinline__ float dpp_quad(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
template <int CTRL> __device__ __forceinline__ double dpp_quad(double v)
{
    int2 w = __builtin_bit_cast(int2, v);
    w.x = __builtin_amdgcn_update_dpp(0, w.x, CTRL, 0xF, 0xF, true);
    w.y = __builtin_amdgcn_update_dpp(0, w.y, CTRL, 0xF, 0xF, true);
    return __builtin_bit_cast(double, w);
}

// wavefronts per SIMD a kernel's registers are held to. Up to 30 moments (28 in
// general domains) a GRID kernel comes to 168 to 184 without a bound, and 3 to 14
// of them spilled cost less than the third wavefront is worth (128^3 f32, 509 x
// 387 rays, 30 moments: 350 us by two, 320 by three; in a domain of 0.9^3 396
// and 422). Node by node 30 moments come to 170 to 174 (512 x 512 rays, 487 and
// 460 us). Particle sets and volumes beyond 32-bit offsets, whose samples wait
// on memory, are better off without (node by node 1229 and 1363 us, 1100^3
// voxels 836 and 948; 28 moments on the grid 867 and 1008).
template <typename T, int M, bool OFF32, bool POW2, bool GRID, int S> constexpr int mixed_wavefronts()
{
    if (!GRID)
        return (M == 30 && OFF32 && !std::is_same<T, SphParticle>::value) ? 3 : 1;
    return (S == 1 && M <= (!OFF32 ? 24 : POW2 ? 30 : 28)) ? 3 : 2;
}

// The integral per node. A segment [u, p] of the reference with slope g
// contributes, with c(phi) = cos(j phi) and rho the line's values at its ends,
//     (1/j^2) [ g c(p) - rho_p c'(p) - g c(u) + rho_u c'(u) ].
// Node k gathers the end of segment k (at p_k) and the start of segment k + 1
// (at u_k+1 = p_k + delta, the reference's p_k+1 - dphi in float). Expanded
// around the uniform grid q_k = (t_k - t_near) pi / range - pi (p_k = q_k +
// eps; eps, delta are a few float ulps of the phase, their squares ~1e-13, and
// next to 8192 steps from t = 0 delta is up to 2^-12 of dphi: GridStep):
//     d c + cp c' + cpp c''   at q_k,
//     d   = g_k - g_k+1
//     cp  = d eps - g_k+1 delta - g_k (width_k - dphi)
//     cpp = f_k delta
// On the uniform grid the derivatives are 9-point differences of c at the
// neighbouring nodes, so a node's terms become weights of plain cosines
// (WeightRing) and a moment costs one FP64 operation per node (five before:
// cosine, sine and weight recurrences and two sums). The stencils reach past
// the ray's ends: c is defined there too. This needs the largest order
// resolved by the grid, (m - 1) dphi <= 1 (at 1: 1.6e-3 of cp's terms, i.e.
// ~1e-10 of the moments), and t's float increments uniform (|t| <= 8192 s:
// where t passes a power of two they change by at most 2^-11): grid_resolves;
// GridStep has what a change next to 8192 s costs.
// The wavefronts with a ray that fails it (a few samples for many moments)
// are summed node by node: the terms at p_k itself, cosine sums in FP64 and
// the ulp-sized sine terms in FP32, five operations per moment. GRID: each
// wavefront takes the form its rays allow, in one launch, so that neither form
// waits for the other's last wavefronts (128^3 f32 from a perspective camera,
// 50 moments, 256 steps: 512 x 512 rays 522 us as two launches over the same
// tiles, 499 all node by node, 364 in one; 90 x 70 rays 322, 266 and 240).
// !GRID: node by node throughout.
//
// A pass that records the rays' normalisation is the forward of a gradient
// (generate_backward) and is summed node by node for every ray: the bounded
// MESE amplifies the last bit of a moment to up to 1e-2 of the gradient's
// norm (mixing layers of 60 to 120 voxels: 1 to 9e-3 between two sums that
// are both within a moment's rounding), so that pass keeps one rounding.
//
// CHUNK: more moments than one thread's registers hold are split into chunks
// of M; each chunk's workgroups march the same rays and accumulate moments
// j0 .. j0 + M - 1. The first chunk is the unchunked kernel (M moments of an
// image of m > M: it writes moments 0 .. M - 1, the bounds, the ray range and
// the sample counts); the CHUNK kernel runs the later ones,
// j0 = (blockIdx.y + 1) M.
// J0C: a chunk start known at compile time.
// S = 4: four lanes per ray, each the terms of a quarter of its nodes (from the
// segment that ends at the first of them to the one that starts at the last),
// their sums added at the end. For images of few rays, which leave most SIMDs
// without a wavefront: a lone wavefront takes 0.5 us per node. A tile that is
// summed node by node leaves three of its wavefronts without work.
// Measured (128^3, 30 moments): 100 steps, up to 16384 rays 62 us by one lane,
// 28 by four; 1000 steps 541 and 179 (each lane first adds up its t).
//
// Measured (1024^3 f32, 1024 x 1024 rays, 50 moments): 11.6 ms node by node,
// 7.1 ms gridded (8.1 before the corners came in pairs); 2048 x 2048 x 1920
// u8, 2048 x 2048 rays, 100 moments: 132 and 76 ms (the bytes' divisions and
// the corner addresses are a third of that gain). Bound by VALU issue, then by
// load latency at two wavefronts per SIMD.
template <typename T, int M, bool OFF32, bool POW2, bool CHUNK, bool GRID, int J0C, int S = 1>
__global__ __launch_bounds__(256, (mixed_wavefronts<T, M, OFF32, POW2, GRID, S>())) void generate_mixed_kernel(VolumeView<T> vol, DevCamera cam, GenArgs a,
                                                             float *__restrict__ out, uint32_t *__restrict__ bounds,
                                                             int32_t *__restrict__ samples,
                                                             float2 *__restrict__ ray_range)
{
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const uint32_t ntiles = ((a.W + 7) / 8) * ((a.H + 7) / 8);
    static_assert(S == 1 || (S == 4 && GRID && !CHUNK), "four lanes per ray: the gridded march, unchunked");
    const int quad = tid & 3; // S = 4: a workgroup's tile, 16 rays per wavefront
    const uint32_t tile = S == 4 ? xcd_tile_block(a.W, 1) : xcd_tile_block(a.W, 4) * 4 + (tid >> 6);
    if (tile >= ntiles)
        return;
    int x, y;
    tile_pixel(tile, a.W, S == 4 ? tid >> 2 : lane, x, y);
    if (S == 1 && (x >= a.W || y >= a.H))
        return;
    const int m = a.m;
    const int j0 = CHUNK ? (J0C ? J0C : (int)(blockIdx.y + 1) * M) : 0;
    const bool first_chunk = !CHUNK;
    const int jend = CHUNK ? min(m, j0 + M) : min(m, M);
    Ray r = pixel_ray(cam, a.W, a.H, x, y);
    float t_near, t_far;
    bool hit = intersect_aabb(r, vol.dmin, vol.dmax, t_near, t_far);
    t_near = rmax(t_near, cam.znear);
    bool tile_gridded = false;
    if constexpr (S == 4)
    {
        // whether the tile's rays are gridded: as its wavefront decides with
        // one lane per ray
        const bool inside = x < a.W && y < a.H;
        const float step_phase = (float)(kPi * (double)(a.step / (t_far - t_near)));
        tile_gridded = !__syncthreads_or(inside && hit && t_far > 0 && !grid_resolves(m, step_phase, t_near, t_far, a.step));
        if (!tile_gridded)
        {
            // one wavefront of the tile's 64 rays, as with one lane per ray
            if (tid >= 64)
                return;
            tile_pixel(tile, a.W, lane, x, y);
            r = pixel_ray(cam, a.W, a.H, x, y);
            hit = intersect_aabb(r, vol.dmin, vol.dmax, t_near, t_far);
            t_near = rmax(t_near, cam.znear);
        }
        if (x >= a.W || y >= a.H)
            return;
    }
    size_t pix = (size_t)y * a.W + x;
    float *mo = out + pix * (size_t)m;
    if (!(hit && (t_far > 0)))
    {
        if (!(a.transform_to_bounds && a.compact_image))
            for (int j = j0; j < jend; ++j)
                mo[j] = 0.f;
        if (first_chunk)
        {
            if (bounds)
                bounds[pix] = 0;
            if (ray_range)
                ray_range[pix] = make_float2(0.0f, 1.0f);
            if (samples)
                samples[pix] = 0;
        }
        return;
    }

    const float s = a.step;
    const float pi_trange_inv = (float)(kPi / (double)(t_far - t_near));
    const float dphi = (float)(kPi * (double)(s / (t_far - t_near)));
    // by wavefront: whether its rays are gridded
    bool gridded = false;
    if constexpr (GRID)
        gridded = S == 4 ? tile_gridded : __ballot(!grid_resolves(m, dphi, t_near, t_far, s)) == 0ull;
    const bool one_lane = S == 1 || !gridded;

    float t = t_near;
    const float f_first = sample_at(vol, r, t, a);
    float lo = rmin(1.f, f_first), hi = rmax(0.f, f_first);
    int ns = 1;

    // phase of node 0: start of the first segment, p_1 - dphi (or -pi when the
    // ray has no interior sample), as update_moments forms p_prev.
    float phase0;
    if (t + s < t_far)
    {
        float t1 = t + s;
        float p1 = (float)((double)((t1 - t_near) * pi_trange_inv) - kPi);
        phase0 = p1 - dphi;
    }
    else
        phase0 = (float)(-kPi);

    double sc[M];
#pragma unroll
    for (int j = 0; j < M; ++j)
        sc[j] = 0.0;
    const double j0d = (double)j0;
    double trap = 0.0; // trig_0, the exact integral of the reference's lines

    const int cap = march_cap(t_near, t_far, s);
    // the next sample's loads are issued one step ahead (at t + s while the
    // march continues, else at t_far for the last segment)
    auto issue_at = [&](PendingSample<T, OFF32, POW2> &ps, float tt) {
        ps.issue(vol, r.o.x + tt * r.d.x, r.o.y + tt * r.d.y, r.o.z + tt * r.d.z);
    };
    PendingSample<T, OFF32, POW2> pending;
    auto density = [&](float sv) { return map_density_r<POW2>(sv, a.data_min, a.data_max, a.data_rinv); };

    // state of the node reached: its density, phase (float, as FP64) and the
    // slope and surplus width (width - dphi) of the segment that ends there
    double f_prev = (double)f_first, p_prev = (double)phase0;
    double g_left = 0.0, w_left = 0.0;
    const double dphid = (double)dphi, rdphi = 1.0 / dphid;
    // the grid's phase per unit of t, and its first step
    const double ptid = (double)pi_trange_inv;
    GridStep step_at;
    step_at.start((t + s) - t, ptid);
    const float ds0 = step_at.ds;

    // S = 4: the lane's nodes first .. until - 1 of 0 .. nodes (its sums are
    // those nodes' terms), begun at the node before; t_back is t four nodes
    // before the first, where the first finished weight belongs
    int first = 0, until = 0, last_node = 0;
    float t_back = t_near;
    if (!one_lane)
    {
        for (float tt = t_near; tt + s < t_far; tt += s)
            ++last_node;
        const int per = (last_node + 4) / 4;
        first = quad * per;
        until = min(first + per, last_node + 1);
        if (first <= last_node && first > 0)
        {
            for (int i = 0; i < first - 1; ++i)
            {
                if (i == first - 4)
                    t_back = t;
                t += s;
            }
            if (first > 1)
            {
                p_prev = (double)(float)((double)((t - t_near) * pi_trange_inv) - kPi);
                f_prev = (double)sample_at(vol, r, t, a);
            }
            ns = first;
        }
    }

    // advances to the next sample and to the terms of the node behind it; the
    // last segment [p_K, 0] (src/raymarch_generate.h:107-114) starts exactly
    // at p_K and its line ends exactly at its sample
    auto segment = [&](double eps, double &d, double &cp, double &cpp, double &shift) __attribute__((always_inline)) {
        const float tn = t + s, dn = tn - t;
        shift = 0.0;
        if (__builtin_expect(dn != step_at.ds, 0))
        {
            asm volatile(""); // rare: a branch, not a select of its result
            shift = step_at.change(dn, ptid);
        }
        t = tn;
        const float p = (float)((double)((t - t_near) * pi_trange_inv) - kPi);
        const float f = density(pending.value());
        // the loaded values die here: keeping the next loads below this point
        // lets them land in the same registers (no copies that would wait
        // for them at the end of the iteration)
        __builtin_amdgcn_sched_barrier(0);
        issue_at(pending, fminf(t + s, t_far));
        lo = fminf(lo, f); // f is in [0, 1]
        hi = fmaxf(hi, f);
        const double fd = (double)f, pd = (double)p;
        const double u = (double)(p - dphi);
        const double g = (fd - f_prev) * rdphi;
        const double width = pd - u;
        trap = fma(width, fma(0.5 * g, width, f_prev), trap);
        const double delta = (ns > 1) ? u - p_prev : 0.0; // node 0 is the start of the first segment
        d = g_left - g;
        cp = fma(d, eps, -fma(g, delta, g_left * w_left));
        cpp = f_prev * delta;
        g_left = g;
        w_left = width - dphid;
        f_prev = fd;
        p_prev = pd;
        ++ns;
    };
    auto last_segment = [&](double eps, double &d, double &cp) __attribute__((always_inline)) {
        const float f = density(pending.value());
        lo = rmin(lo, f);
        hi = rmax(hi, f);
        const double dl = 0.0 - p_prev;
        const double g = ((double)f - f_prev) / dl;
        trap = fma(dl, fma(0.5 * g, dl, f_prev), trap);
        d = g_left - g;
        cp = fma(d, eps, -g_left * w_left);
        g_left = g;
        ++ns;
    };

    if (GRID && gridded)
    {
        issue_at(pending, fminf(t + s, t_far));
        // the phasor of the node whose weight is finished, four nodes behind,
        // turned by the grid's step; td is that node's t
        WeightRing ring;
        float dsd = ds0, td = t_near;
        double step = (double)ds0 * ptid;
        double rs, rc, zs, zc, js, jc, kr = 0.0, ki = 0.0;
        sincos_small(step, rs, rc);
        if constexpr (S == 4)
        {
            td = t_back;
            sincos_small(first >= 4 ? fma((double)t_back - (double)t_near, ptid, -kPi)
                                    : (double)(first - 4) * step - kPi,
                         zs, zc);
        }
        else
            sincos_small(-kPi - 4.0 * step, zs, zc);
        if constexpr (CHUNK)
        {
            sincos_small(j0d * step, js, jc);
            sincos_small(j0d * (-kPi - 4.0 * step), ki, kr);
        }
        auto add = [&](double w) __attribute__((always_inline)) {
            // a weight of exactly zero (inside a stretch of zero density) adds
            // nothing; where every lane of the wavefront has one, skipped
            if (w != 0.0)
            {
                if constexpr (CHUNK)
                    accumulate_chunk<M>(sc, w, zc, kr, fma(kr, zc, -ki * zs));
                else
                {
                    // moment 0 is integrated apart (trap)
                    double cheb[block_width<M>() + 1];
                    cheb_low<block_width<M>()>(cheb, zc);
                    block_sums<M, 1>(sc, w, cheb);
                }
            }
        };
        auto turn = [&]() __attribute__((always_inline)) {
            const double nc = fma(zc, rc, -zs * rs);
            zs = fma(zs, rc, zc * rs);
            zc = nc;
            if constexpr (CHUNK)
            {
                const double nk = fma(kr, jc, -ki * js);
                ki = fma(ki, jc, kr * js);
                kr = nk;
            }
        };
        // the turn to the next real node: t's increment changes where t
        // passes a power of two
        auto turn_real = [&]() __attribute__((always_inline)) {
            const float tn = td + s;
            if (__builtin_expect(tn - td != dsd, 0))
            {
                dsd = tn - td;
                sincos_small((double)dsd * ptid, rs, rc);
                if constexpr (CHUNK)
                    sincos_small(j0d * ((double)dsd * ptid), js, jc);
            }
            td = tn;
            turn();
        };
        double eps = p_prev + kPi; // of node 0, at q_0 = -pi
        int it = 0;
        if constexpr (S == 4)
        {
            it = first;
            if (first > 0 && first <= last_node)
            {
                // the segment that ends at the first node: its left slope
                double d, cp, cpp, shift;
                segment(eps, d, cp, cpp, shift);
                eps = p_prev - fma((double)t - (double)t_near, ptid, -kPi);
                trap = 0.0;
            }
        }
        while (S == 4 ? it < min(until, last_node) : t + s < t_far) // t advances by s (1 - 2^-11) or more
        {
            double d, cp, cpp, shift;
            segment(eps, d, cp, cpp, shift);
            eps = p_prev - fma((double)t - (double)t_near, ptid, -kPi);
            const double A = step_at.second(cpp);
            add(ring.push(d, A, step_at.first(cp, A, shift)));
            if (it++ >= 4)
                turn_real();
            else
                turn();
        }
        if constexpr (S == 4)
        {
            const bool last = first <= last_node && until > last_node;
            if (last)
            {
                double d, cp;
                last_segment(eps, d, cp);
                add(ring.push(d, 0.0, cp * step_at.rstep));
            }
            if (first <= last_node)
            {
                // node of the phasor and of the ring's first pending weight
                // (turned already behind a push of the loop)
                int node = it - 4;
                for (int i = 0; i < 8; ++i)
                {
                    if (i > 0 || last)
                    {
                        if (node >= 0 && node < last_node)
                            turn_real();
                        else
                            turn();
                        ++node;
                    }
                    add(ring.pop());
                }
            }
            else
                ns = 0;
            auto quad_sum = [](double v) __attribute__((always_inline)) {
                v += dpp_quad<0xB1>(v);
                return v + dpp_quad<0x4E>(v);
            };
            g_left = quad_sum(last ? g_left : 0.0);
            trap = quad_sum(trap);
#pragma unroll
            for (int j = 0; j < M; ++j)
                sc[j] = quad_sum(sc[j]);
            lo = fminf(lo, dpp_quad<0xB1>(lo));
            lo = fminf(lo, dpp_quad<0x4E>(lo));
            hi = fmaxf(hi, dpp_quad<0xB1>(hi));
            hi = fmaxf(hi, dpp_quad<0x4E>(hi));
            ns = last_node + 2;
            untangle_sums<M>(sc);
        }
        else
        {
            double d, cp;
            last_segment(eps, d, cp);
            add(ring.push(d, 0.0, cp * step_at.rstep));
            // the nodes whose weights are still pending: real ones up to the
            // last, then the grid continued
            const int nodes = ns - 2; // index of the last node
            for (int i = 0; i < 8; ++i)
            {
                if (nodes - 4 + i >= 0 && i < 4)
                    turn_real();
                else
                    turn();
                add(ring.pop());
            }
            if constexpr (!CHUNK)
                untangle_sums<M>(sc);
        }
    }
    else
    {
        issue_at(pending, fminf(t + s, t_far));
        float ss[M];
#pragma unroll
        for (int j = 0; j < M; ++j)
            ss[j] = 0.0f;
        // cos and sin of the node phase (FP64, of the float phase); CHUNK: of
        // j0 phi and (j0 + 1) phi too (the product j0 phi is exact in FP64)
        float node_phase = phase0, fp = f_first, gl = 0.0f;
        double zs, zc, kc = 1.0, ks = 0.0, kc1, ks1;
        sincos_small((double)node_phase, zs, zc);
        bool turned = false; // kc, ks already are those of the node
        auto chunk_start = [&](float ph) __attribute__((always_inline)) {
            if constexpr (CHUNK)
            {
                if (!turned)
                    sincos_small(j0d * (double)ph, ks, kc);
                kc1 = fma(kc, zc, -ks * zs);
                ks1 = fma(ks, zc, kc * zs);
            }
        };
        chunk_start(node_phase);
        auto add = [&](double d, double e, double h) __attribute__((always_inline)) {
            if constexpr (CHUNK && J0C > 0)
                accumulate_node_chunk_c<M, J0C>(sc, ss, d, e, (float)h, zc, kc, (float)ks, kc1, (float)ks1);
            else if constexpr (CHUNK)
                accumulate_node_chunk<M>(sc, ss, d, e, (float)h, zc, kc, (float)ks, kc1, (float)ks1, j0d);
            else
                accumulate_node<M>(sc, ss, d, e, (float)h, zc, (float)zs);
        };
        const float rdphif = host_reciprocal(dphi); // for the segment slopes
        for (int it = 0; t + s < t_far && it < cap; ++it)
        {
            t += s;
            const float p = (float)((double)((t - t_near) * pi_trange_inv) - kPi);
            const float f = density(pending.value());
            __builtin_amdgcn_sched_barrier(0);
            issue_at(pending, (t + s < t_far && it + 1 < cap) ? t + s : t_far);
            ++ns;
            lo = rmin(lo, f);
            hi = rmax(hi, f);
            const float u = p - dphi;
            const float g = div_rn(f - fp, dphi, rdphif);
            const double width = (double)p - (double)u;
            trap += width * ((double)fp + 0.5 * (double)g * width);
            const double delta = (it > 0) ? (double)u - (double)node_phase : 0.0;
            const double h = fma((double)g, delta, (double)gl * w_left);
            const double dn = (double)gl - (double)g, en = -delta * (double)fp;
            if (dn != 0.0 || en != 0.0 || h != 0.0)
                add(dn, en, h);
            gl = g;
            w_left = width - dphid;
            fp = f;
            // the phasor turned by the exact difference of the two float
            // phases while that is small (Taylor terms to dp^5 and dp^6); that
            // of j0 phi, j0 known at compile time, by j0 dp likewise
            // (|j0 dp| <= 50 / 64 < pi / 4)
            const double dp = (double)p - (double)node_phase;
            turned = false;
            if (M <= 56 && fabs(dp) <= 0.015625)
            {
                const double d2 = dp * dp;
                const double sd = fma(dp * d2, fma(d2, 1.0 / 120.0, -1.0 / 6.0), dp);
                const double cd = fma(fma(fma(d2, -1.0 / 720.0, 1.0 / 24.0), d2, -0.5), d2, 1.0);
                const double nc = fma(zc, cd, -zs * sd);
                zs = fma(zs, cd, zc * sd);
                zc = nc;
                if constexpr (CHUNK && J0C > 0)
                {
                    static_assert(J0C <= 50, "the turn by J0C dp must stay within pi / 4");
                    double sj, cj;
                    sincos_quarter((double)J0C * dp, sj, cj);
                    const double nkc = fma(kc, cj, -ks * sj);
                    ks = fma(ks, cj, kc * sj);
                    kc = nkc;
                    turned = true;
                }
            }
            else
                sincos_small((double)p, zs, zc);
            node_phase = p;
            chunk_start(p);
        }
        // last segment [p_K, 0] (src/raymarch_generate.h:107-114): it starts
        // exactly at p_K and its line ends exactly at its sample
        const float f = density(pending.value());
        ++ns;
        lo = rmin(lo, f);
        hi = rmax(hi, f);
        const float dl = 0.0f - node_phase;
        const float g = (f - fp) / dl;
        trap += (double)dl * ((double)fp + 0.5 * (double)g * (double)dl);
        add((double)gl - (double)g, 0.0, (double)gl * w_left);
        g_left = (double)g;
#pragma unroll
        for (int j = 0; j < M; ++j)
            sc[j] = fma(j0d + (double)j, (double)ss[j], sc[j]);
    }
    // node at phase 0: cos(j*0) = 1, sin(j*0) = 0
#pragma unroll
    for (int j = CHUNK ? 0 : 1; j < M; ++j)
        sc[j] += g_left;

    // trig_j = sc_j / j^2 - f_0 sin(j phi_0) / j in FP64 (phi_0 the start of
    // the first segment), sin by the recurrence over j, then moment_j =
    // trig_j / pi, normalised and rounded to float once
    double norm = 0.31830988618379067154; // 1 / pi
    if (a.transform_to_bounds)
    {
        lo = rmax(lo - a.bound_eps, 0.0f);
        hi = rmin(hi + a.bound_eps, 1.0f);
        const double inv = 1.0 / (double)(hi - lo);
        if (first_chunk)
            mo[0] = (float)((trap * norm - (double)lo) * inv);
        norm *= inv;
    }
    else if (first_chunk)
        mo[0] = (float)(trap * norm);
    {
        double z0s, z0c, k0s = 0.0, k0c = 1.0;
        sincos_small((double)phase0, z0s, z0c);
        if constexpr (CHUNK)
            sincos_small(j0d * (double)phase0, k0s, k0c);
        const double x2 = z0c + z0c;
        double sm2 = k0s, sm1 = fma(k0s, z0c, k0c * z0s); // sin(j0 phi_0), sin((j0 + 1) phi_0)
#pragma unroll
        for (int i = 0; i < M; ++i)
        {
            const double jd = j0d + (double)i;
            const int j = j0 + i;
            double sj = (i == 0) ? sm2 : sm1;
            if (i >= 1)
            {
                const double n = fma(x2, sm1, -sm2);
                sm2 = sm1;
                sm1 = n;
            }
            if (j >= 1 && j < jend && (one_lane || (j & 3) == quad))
                mo[j] = (float)((sc[i] / (jd * jd) - (double)f_first * sj / jd) * norm);
        }
    }
    if (first_chunk)
    {
        const uint32_t b = pack_bound(lo, hi);
        if (bounds)
            bounds[pix] = b;
        if (ray_range)
            ray_range[pix] = make_float2(lo, hi);
        if (samples)
            samples[pix] = ns;
    }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
// images of few rays take four lanes per ray: up to two wavefronts of 16 rays,
// which is what the registers hold, on each of the 1024 SIMDs (192 x 160 rays:
// 66 us by one lane, 44 by four; 256 x 192: 68 and 68; 256 x 256: 70 and 83)
constexpr uint64_t kFewRays = 32768;

// one launch of generate_mixed_kernel over `chunks` rows of blockIdx.y
template <typename T, int M, bool CHUNK, bool GRID, int J0C>
static void launch_mixed_kernel(const VolumeView<T> &v, const DevCamera &c, const GenArgs &a, float *o, uint32_t *b,
                                int32_t *s, float2 *rr, hipStream_t st, uint32_t blocks, int chunks)
{
    const bool off32 = offsets_fit(v.nx, v.ny, v.nz, sizeof(T));
    // power-of-two domain extents and data range: divisions become products
    const bool pow2 = exact_pow2(v.dmax.x - v.dmin.x) && exact_pow2(v.dmax.y - v.dmin.y) &&
                      exact_pow2(v.dmax.z - v.dmin.z) && exact_pow2(a.data_max - a.data_min);
    const dim3 grid(blocks, chunks);
    if constexpr (std::is_same<T, SphParticle>::value)
    {
        // particle sets: the gather ignores OFF32 and POW2 (the data range
        // division takes the exact path)
        hipLaunchKernelGGL((generate_mixed_kernel<T, M, true, false, CHUNK, GRID, J0C>), grid, dim3(256), 0, st, v, c, a,
                           o, b, s, rr);
    }
    else
    {
        if (off32 && pow2)
            hipLaunchKernelGGL((generate_mixed_kernel<T, M, true, true, CHUNK, GRID, J0C>), grid, dim3(256), 0, st, v, c,
                               a, o, b, s, rr);
        else if (off32)
            hipLaunchKernelGGL((generate_mixed_kernel<T, M, true, false, CHUNK, GRID, J0C>), grid, dim3(256), 0, st, v, c,
                               a, o, b, s, rr);
        else
            hipLaunchKernelGGL((generate_mixed_kernel<T, M, false, false, CHUNK, GRID, J0C>), grid, dim3(256), 0, st, v,
                               c, a, o, b, s, rr);
    }
}

// `chunks` > 1 marches the moments in chunks of M: the unchunked kernel for
// the first, then the later ones over blockIdx.y (or, of two, the second from
// j0 = M as a compile-time start)
template <typename T, int M, bool GRID, bool CHUNK = false>
static void launch_mixed(const VolumeView<T> &v, const DevCamera &c, const GenArgs &a, float *o, uint32_t *b,
                         int32_t *s, float2 *rr, hipStream_t st, uint32_t blocks, int chunks = 1)
{
    launch_mixed_kernel<T, M, false, GRID, 0>(v, c, a, o, b, s, rr, st, blocks, 1);
    if constexpr (CHUNK)
    {
        if (chunks == 2)
            launch_mixed_kernel<T, M, true, GRID, M>(v, c, a, o, b, s, rr, st, blocks, 1);
        else if (chunks > 1)
            launch_mixed_kernel<T, M, true, GRID, 0>(v, c, a, o, b, s, rr, st, blocks, chunks - 1);
    }
}

// the march by four lanes per ray (grids only); false if this call doesn't take it
template <typename T>
static bool launch_few_rays(const VolumeView<T> &v, const DevCamera &c, const GenArgs &a, float *o, uint32_t *b,
                            int32_t *s, hipStream_t st)
{
    if (a.m > 56 || (uint64_t)a.W * (uint64_t)a.H > kFewRays || !offsets_fit(v.nx, v.ny, v.nz, sizeof(T)))
        return false;
    const bool pow2 = exact_pow2(v.dmax.x - v.dmin.x) && exact_pow2(v.dmax.y - v.dmin.y) &&
                      exact_pow2(v.dmax.z - v.dmin.z) && exact_pow2(a.data_max - a.data_min);
    const dim3 grid((uint32_t)(((a.W + 7) / 8) * ((a.H + 7) / 8)));
    float2 *none = nullptr;
#define MRAY_FEW_CASE(MM)                                                                                             \
    if (a.m <= MM)                                                                                                    \
    {                                                                                                                 \
        if (pow2)                                                                                                     \
            hipLaunchKernelGGL((generate_mixed_kernel<T, MM, true, true, false, true, 0, 4>), grid, dim3(256), 0, st, \
                               v, c, a, o, b, s, none);                                                               \
        else                                                                                                          \
            hipLaunchKernelGGL((generate_mixed_kernel<T, MM, true, false, false, true, 0, 4>), grid, dim3(256), 0,    \
                               st, v, c, a, o, b, s, none);                                                           \
        return true;                                                                                                  \
    }
    MRAY_FEW_CASE(8)
    MRAY_FEW_CASE(16)
    MRAY_FEW_CASE(24)
    MRAY_FEW_CASE(30)
    MRAY_FEW_CASE(36)
    MRAY_FEW_CASE(40)
    MRAY_FEW_CASE(44)
    MRAY_FEW_CASE(50)
    MRAY_FEW_CASE(56)
#undef MRAY_FEW_CASE
    return false;
}

template <typename T, bool GRID>
static int dispatch_widths(const VolumeView<T> &v, const DevCamera &c, const GenArgs &a, float *o, uint32_t *b,
                           int32_t *s, float2 *rr, hipStream_t st, uint32_t blocks)
{
    const int m = a.m;
#define MRAY_GEN_CASE(MM)                                                                                             \
    if (m <= MM)                                                                                                      \
    {                                                                                                                 \
        launch_mixed<T, MM, GRID>(v, c, a, o, b, s, rr, st, blocks);                                                  \
        return 0;                                                                                                     \
    }
    MRAY_GEN_CASE(4)
    MRAY_GEN_CASE(8)
    MRAY_GEN_CASE(12)
    MRAY_GEN_CASE(16)
    MRAY_GEN_CASE(20)
    MRAY_GEN_CASE(24)
    MRAY_GEN_CASE(28)
    MRAY_GEN_CASE(30)
    MRAY_GEN_CASE(32)
    MRAY_GEN_CASE(36)
    MRAY_GEN_CASE(40)
    MRAY_GEN_CASE(44)
    MRAY_GEN_CASE(48)
    MRAY_GEN_CASE(50)
    MRAY_GEN_CASE(52)
    MRAY_GEN_CASE(56)
    MRAY_GEN_CASE(60)
#undef MRAY_GEN_CASE
    // 61..255 moments: K chunks of at most 50 (an unchunked M = 64 loses half
    // its occupancy, and so does a chunk of 56), each M >= ceil(m / K) wide
    if (m <= 255)
    {
        const int chunks = (m + 49) / 50;
        const int per = (m + chunks - 1) / chunks;
        if (per <= 40)
            launch_mixed<T, 40, GRID, true>(v, c, a, o, b, s, rr, st, blocks, chunks);
        else
            launch_mixed<T, 50, GRID, true>(v, c, a, o, b, s, rr, st, blocks, chunks);
        return 0;
    }
    return MRAY_ERR_UNSUPPORTED;
}

// The kernel that lets each wavefront take the gridded march, unless none can:
// a pass that records the rays' normalisation (ray_range) is summed node by
// node throughout (see the kernel), and so is an image whose longest possible
// ray has too few samples for its moments. Particle sets, too: a sample of
// theirs is a walk over cells that costs many times the sums, and the gridded
// march's registers take wavefronts that hide its loads (10^6 particles, 256 x
// 256 rays, 128 steps, 30 moments: 8.0 ms node by node, 13.2 gridded).
template <typename T>
static int dispatch_mixed(const VolumeView<T> &v, const DevCamera &c, const GenArgs &a, float *o, uint32_t *b,
                          int32_t *s, float2 *rr, hipStream_t st, uint32_t blocks)
{
    if constexpr (std::is_same<T, SphParticle>::value)
        return dispatch_widths<T, false>(v, c, a, o, b, s, rr, st, blocks);
    else
    {
        const float ex = v.dmax.x - v.dmin.x, ey = v.dmax.y - v.dmin.y, ez = v.dmax.z - v.dmin.z;
        const Vec3 d = c.dir;
        // directions of perspective rays are unit vectors, an orthographic
        // camera's is as given
        const float len = c.orthographic ? sqrtf(d.x * d.x + d.y * d.y + d.z * d.z) : 1.0f;
        const float longest = sqrtf(ex * ex + ey * ey + ez * ez) / len;
        if (rr || !((float)(a.m - 1) * (float)kPi * (a.step / longest) <= 1.01f))
            return dispatch_widths<T, false>(v, c, a, o, b, s, rr, st, blocks);
        if (launch_few_rays(v, c, a, o, b, s, st))
            return 0;
        return dispatch_widths<T, true>(v, c, a, o, b, s, rr, st, blocks);
    }
}

// PLAIN keeps m floats per thread in LDS: 256-thread blocks while that fits
// in 64 KiB, else one wave per block.
static int plain_block(int m) { return (256 * m * (int)sizeof(float) <= 65536) ? 256 : 64; }

// ---------------------------------------------------------------------------
// ADJOINT (F32 volumes): dL/dvolume from dL/dmoments
// ---------------------------------------------------------------------------

// A trilinear sample of the march that keeps what its reverse needs: the
// cell, the weights and the voxel values (same arithmetic as sample_volume;
// loads issued in issue(), used in value()).
template <bool POW2> struct GradSample
{
    float ax, ay, az;
    int cx, cy, cz; // clamped (x0, y0, z0)
    uint32_t fl;    // bit 0/1/2: x1 > x0, y1 > y0, z1 > z0 (0 at a clamped edge)
    float v[8];

    __device__ __forceinline__ void issue(const VolumeView<float> &vol, float px, float py, float pz)
    {
        const float ipx = div_c<POW2>(px - vol.dmin.x, vol.dmax.x - vol.dmin.x, vol.rext.x) * (float)vol.nx;
        const float ipy = div_c<POW2>(py - vol.dmin.y, vol.dmax.y - vol.dmin.y, vol.rext.y) * (float)vol.ny;
        const float ipz = div_c<POW2>(pz - vol.dmin.z, vol.dmax.z - vol.dmin.z, vol.rext.z) * (float)vol.nz;
        const float flx = floorf(ipx), fly = floorf(ipy), flz = floorf(ipz);
        ax = ipx - flx;
        ay = ipy - fly;
        az = ipz - flz;
        const int xl = (int)flx, yl = (int)fly, zl = (int)flz;
        cx = iclamp(xl, 0, vol.nx - 1);
        cy = iclamp(yl, 0, vol.ny - 1);
        cz = iclamp(zl, 0, vol.nz - 1);
        const int x1 = iclamp(xl + 1, 0, vol.nx - 1), y1 = iclamp(yl + 1, 0, vol.ny - 1),
                  z1 = iclamp(zl + 1, 0, vol.nz - 1);
        fl = (uint32_t)(x1 > cx) | ((uint32_t)(y1 > cy) << 1) | ((uint32_t)(z1 > cz) << 2);
        const uint32_t sxy = (uint32_t)(vol.ny * vol.nx);
        const uint32_t dx = fl & 1u, dy = (fl & 2u) ? (uint32_t)vol.nx : 0u;
        const float *p0 = vol.data + ((size_t)cz * sxy + (uint32_t)(cy * vol.nx + cx));
        const float *p1 = p0 + ((fl & 4u) ? sxy : 0u);
        v[0] = p0[0];
        v[1] = p0[dx];
        v[2] = p0[dy];
        v[3] = p0[dy + dx];
        v[4] = p1[0];
        v[5] = p1[dx];
        v[6] = p1[dy];
        v[7] = p1[dy + dx];
    }

    __device__ __forceinline__ float value() const
    {
        return (1.f - ax) * (1.f - ay) * (1.f - az) * v[0] + ax * (1.f - ay) * (1.f - az) * v[1] +
               (1.f - ax) * ay * (1.f - az) * v[2] + ax * ay * (1.f - az) * v[3] + (1.f - ax) * (1.f - ay) * az * v[4] +
               ax * (1.f - ay) * az * v[5] + (1.f - ax) * ay * az * v[6] + ax * ay * az * v[7];
    }
};

// Where the gradient of a cell's eight voxels goes: a workgroup's LDS window
// over a box of voxels (summed there, added to the volume once per voxel and
// chunk of the march) or, for corners
// outside the window, straight to the volume with float atomics. The window's
// 64 KiB hold 8192 voxels in 64-bit fixed point (integer LDS atomics, the
// fast kind) or 16384 in float (LDS float atomics cost several times more,
// but less than the global atomics a box too large for 8192 would take).
enum WinMode : int
{
    kWinGlobal = 0, // no window: float atomics to the volume
    kWinFixed = 1,  // 64-bit fixed point at scale 2^kfix
    kWinFloat = 2,  // float
};
struct GradTarget
{
    float *grad;
    unsigned long long *win; // LDS window, x fastest (as 8192 x u64 or 16384 x f32)
    int kfix;
    int ox, oy, oz, ex, ey, ez;
    int mode; // WinMode, the same in the whole workgroup
    int nx;
    uint32_t sxy;

    // adds w[i] to corner i of the cell (corner i: bit 0 / 1 / 2 of i select
    // x1 / y1 / z1)
    __device__ __forceinline__ void add(int cx, int cy, int cz, uint32_t fl, const float (&w)[8]) const
    {
        const int fx = fl & 1, fy = (fl >> 1) & 1, fz = (fl >> 2) & 1;
        const int lx = cx - ox, ly = cy - oy, lz = cz - oz;
        if (mode != kWinGlobal && lx >= 0 && ly >= 0 && lz >= 0 && lx + fx < ex && ly + fy < ey && lz + fz < ez)
        {
            const int i0 = lx + ex * (ly + ey * lz);
            const int dy = fy * ex, dz = fz * ex * ey;
            if (mode == kWinFixed)
            {
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    atomicAdd(win + i0 + ((i & 1) ? fx : 0) + ((i & 2) ? dy : 0) + ((i & 4) ? dz : 0),
                              to_fixed(w[i], kfix));
            }
            else
            {
                float *wf = reinterpret_cast<float *>(win);
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    atomicAdd(wf + i0 + ((i & 1) ? fx : 0) + ((i & 2) ? dy : 0) + ((i & 4) ? dz : 0), w[i]);
            }
            return;
        }
        float *p0 = grad + ((size_t)cz * sxy + (uint32_t)(cy * nx + cx));
        const uint32_t dy = fy ? (uint32_t)nx : 0u, dz = fz ? sxy : 0u;
#pragma unroll
        for (int i = 0; i < 8; ++i)
            unsafeAtomicAdd(p0 + ((i & 1) ? (uint32_t)fx : 0u) + ((i & 2) ? dy : 0u) + ((i & 4) ? (size_t)dz : 0u), w[i]);
    }
};

// Accumulates gs times the trilinear weights of a sample. Consecutive
// samples of a ray in the same cell are merged in registers; the eight
// corners go to the target when the ray leaves the cell (one code path for
// every lane: keeping a shared face in registers saved atomics but split the
// wavefront over six cases). Clamp-to-edge duplicates receive both weights.
struct CellScatter
{
    int cx = -1, cy = 0, cz = 0;
    uint32_t fl = 0;
    float w[8] = {0, 0, 0, 0, 0, 0, 0, 0};

    __device__ __forceinline__ void flush(const GradTarget &tg)
    {
        if (cx < 0)
            return;
        tg.add(cx, cy, cz, fl, w);
        cx = -1;
    }

    template <bool POW2> __device__ __forceinline__ void add(const GradTarget &tg, const GradSample<POW2> &sm, float gs)
    {
        // the same corner with other neighbour flags is another cell (a
        // sample just outside the domain clamps onto the edge voxel)
        if (!(sm.cx == cx && sm.cy == cy && sm.cz == cz && sm.fl == fl))
        {
            flush(tg);
#pragma unroll
            for (int i = 0; i < 8; ++i)
                w[i] = 0.0f;
            cx = sm.cx;
            cy = sm.cy;
            cz = sm.cz;
            fl = sm.fl;
        }
        const float ax = sm.ax, ay = sm.ay, az = sm.az;
        w[0] += gs * ((1.f - ax) * (1.f - ay) * (1.f - az));
        w[1] += gs * (ax * (1.f - ay) * (1.f - az));
        w[2] += gs * ((1.f - ax) * ay * (1.f - az));
        w[3] += gs * (ax * ay * (1.f - az));
        w[4] += gs * ((1.f - ax) * (1.f - ay) * az);
        w[5] += gs * (ax * (1.f - ay) * az);
        w[6] += gs * ((1.f - ax) * ay * az);
        w[7] += gs * (ax * ay * az);
    }
};

// Reverse mode of the generate march for dL/dmoments (dense W*H*m). The
// derivative of the exact integral of the reference's piecewise-linear
// segment [pp, pn] (length sg, slope denominator seg, r = sg / seg) is
//   d trig_j / d f1 =  (cos j pn - cos j pp) / (j^2 seg) + r sin(j pn) / j
//   d trig_j / d f0 = -(cos j pn - cos j pp) / (j^2 seg) + (1 - r) sin(j pn) / j - sin(j pp) / j
//   d trig_0 / d f1 = sg^2 / (2 seg),  d trig_0 / d f0 = sg - sg^2 / (2 seg).
// Summed over j with the incoming gradients g_j these need, at each end
// point, C(phi) = sum g_j / j^2 cos(j phi) and S(phi) = sum g_j / j sin(j phi):
// two Clenshaw sums in FP64 per node (their differences between neighbouring
// nodes are small next to their values). A segment starts where the previous
// one ended up to the reference's float rounding, pp = phi_k + delta; that
// offset enters to first order, C(pp) = C_k - delta S_k and S(pp) = S_k +
// delta S'_k, with S' = sum g_j cos(j phi) from a central difference of S
// over the neighbouring nodes (delta is a few ulps, so its accuracy hardly
// matters). Then through map_density (slope 1 / (data_max - data_min) where
// it does not clamp) and the trilinear weights to the voxels. The bounds are
// constants (a first pass recomputes them for the normalisation); cos and
// sin of the node phases come from sincos_small. One thread per ray, nothing
// stored per sample.
// CHUNK: moments j0 .. j0 + M - 1 with j0 = blockIdx.y * M (more moments
// than one thread's registers hold); the reverse is linear in the incoming
// gradient, so the chunks' passes add their shares to the volume gradient.
template <int M, bool POW2, bool CHUNK = false>
__global__ __launch_bounds__(256) void generate_adjoint_kernel(VolumeView<float> vol, DevCamera cam, GenArgs a,
                                                               const float *__restrict__ grad_mom,
                                                               const float2 *__restrict__ ray_range,
                                                               float *__restrict__ grad_vol)
{
    // The workgroup's 256 rays advance in chunks of kChunk nodes. Per chunk
    // they agree on the box of voxels they can touch; gradients go to an LDS
    // window over that box (when it fits), which is then added to the volume
    // with one atomic per voxel instead of one per ray, sample and corner.
    constexpr int kWin = 8192; // voxels of LDS window in 64-bit fixed point (twice as many in float)
    constexpr int kChunk = 32; // nodes per chunk and ray
    __shared__ unsigned long long win[kWin];
    __shared__ int bbox[6];
    __shared__ uint32_t bound_bits;
    const int tid = threadIdx.x;
    for (int i = tid; i < kWin; i += blockDim.x)
        win[i] = 0ull;
    if (tid == 0)
        bound_bits = 0u;
    __syncthreads();

    const int lane = tid & 63;
    const uint32_t ntiles = ((a.W + 7) / 8) * ((a.H + 7) / 8);
    const uint32_t tile = xcd_tile_block(a.W, 4) * 4 + (tid >> 6);
    int x = 0, y = 0;
    bool active = tile < ntiles;
    if (active)
    {
        tile_pixel(tile, a.W, lane, x, y);
        active = x < a.W && y < a.H;
    }
    Ray r = pixel_ray(cam, a.W, a.H, active ? x : 0, active ? y : 0);
    float t_near, t_far;
    const bool hit = intersect_aabb(r, vol.dmin, vol.dmax, t_near, t_far);
    t_near = rmax(t_near, cam.znear);
    active = active && hit && (t_far > 0);
    const int m = a.m;
    const size_t pix = active ? (size_t)y * a.W + x : 0;
    const float s = a.step;
    const float pi_trange_inv = (float)(kPi / (double)(t_far - t_near));
    const float dphi = (float)(kPi * (double)(s / (t_far - t_near)));
    const int cap = active ? march_cap(t_near, t_far, s) : 0;
    auto issue_at = [&](GradSample<POW2> &sm, float tt) {
        sm.issue(vol, r.o.x + tt * r.d.x, r.o.y + tt * r.d.y, r.o.z + tt * r.d.z);
    };
    auto density = [&](const GradSample<POW2> &sm) {
        return map_density_r<POW2>(sm.value(), a.data_min, a.data_max, a.data_rinv);
    };

    // normalisation of the forward: inv = 1 / (hi - lo) with the bounds of the
    // ray, as the forward recorded them or from a pass over the samples
    double inv = 1.0;
    if (active && a.transform_to_bounds && ray_range)
    {
        const float2 b = ray_range[pix];
        inv = 1.0 / (double)(b.y - b.x);
    }
    else if (active && a.transform_to_bounds)
    {
        float lo = 1.f, hi = 0.f;
        GradSample<POW2> sm;
        float t = t_near;
        issue_at(sm, t);
        for (int it = 0;; ++it)
        {
            const bool more = t + s < t_far && it < cap;
            const float f = density(sm);
            lo = rmin(lo, f);
            hi = rmax(hi, f);
            if (!more && t == t_far)
                break;
            t = more ? t + s : t_far;
            __builtin_amdgcn_sched_barrier(0);
            issue_at(sm, t);
            if (!more)
            {
                const float fl = density(sm);
                lo = rmin(lo, fl);
                hi = rmax(hi, fl);
                break;
            }
        }
        lo = rmax(lo - a.bound_eps, 0.0f);
        hi = rmin(hi + a.bound_eps, 1.0f);
        inv = 1.0 / (double)(hi - lo);
    }
    // dL/dtrig_j = dL/dmoment_j * inv / pi
    // Chebyshev coefficients g_j / j^2 of C in FP64 registers (slot i holds
    // moment j0 + i; moment 0 enters through g0, in the first chunk)
    const int j0 = CHUNK ? (int)blockIdx.y * M : 0;
    double cc[M];
    const double scale = inv / kPi;
    const double g0 = (active && j0 == 0) ? (double)grad_mom[pix * m] * scale : 0.0;
#pragma unroll
    for (int i = 0; i < M; ++i)
    {
        const int j = j0 + i;
        cc[i] = (active && j >= 1 && j < m) ? (double)grad_mom[pix * m + j] * scale / (double)(j * j) : 0.0;
    }
    // C and S at a node with cos / sin (co, si) of its phase: Clenshaw's
    // recurrence b_l = c_l + 2x b_{l+1} - b_{l+2} gives C = x b_1 - b_2, and
    // its derivative in x, b'_l = 2 b_{l+1} + 2x b'_{l+1} - b'_{l+2}, gives
    // S = -dC/dphi = sin(phi) dC/dx = sin(phi) (b_1 + x b'_1 - b'_2), since
    // S = sum j c_j sin(j phi) for the same coefficients c_j = g_j / j^2.
    //
    // CHUNK: the chunk's sum is C = b_0 T_j0 - b_1 T_j0-1 (Clenshaw down to
    // slot 0), and with T'_n(cos phi) sin(phi) = n sin(n phi),
    // S = sin(phi) (d_0 T_j0 - d_1 T_j0-1) + b_0 j0 sin(j0 phi)
    //     - b_1 (j0 - 1) sin((j0 - 1) phi);
    // cos and sin of j0 phi by binary powering of the node's phasor (j0 is
    // the same in the whole workgroup), so that they are the Chebyshev values
    // of the x the recurrence uses.
    auto sums = [&](double co, double si, double &C, double &S) {
        const double x2 = co + co;
        double b1 = 0.0, b2 = 0.0, d1 = 0.0, d2 = 0.0;
        if constexpr (!CHUNK)
        {
#pragma unroll
            for (int l = M - 1; l >= 1; --l)
            {
                const double tb = fma(x2, b1, cc[l] - b2);
                const double td = fma(x2, d1, fma(2.0, b1, -d2));
                b2 = b1;
                b1 = tb;
                d2 = d1;
                d1 = td;
            }
            C = fma(co, b1, -b2);
            S = si * (b1 + fma(co, d1, -d2));
        }
        else
        {
#pragma unroll
            for (int l = M - 1; l >= 0; --l)
            {
                const double tb = fma(x2, b1, cc[l] - b2);
                const double td = fma(x2, d1, fma(2.0, b1, -d2));
                b2 = b1;
                b1 = tb;
                d2 = d1;
                d1 = td;
            }
            // b1, b2, d1, d2 now hold b_0, b_1, d_0, d_1
            double pc = 1.0, ps = 0.0, bc = co, bs = si;
            for (int e = j0; e > 0; e >>= 1)
            {
                if (e & 1)
                {
                    const double nc = fma(pc, bc, -ps * bs);
                    ps = fma(pc, bs, ps * bc);
                    pc = nc;
                }
                const double sc = fma(bc, bc, -bs * bs);
                bs = 2.0 * bc * bs;
                bc = sc;
            }
            const double qc = fma(pc, co, ps * si), qs = fma(ps, co, -pc * si); // (j0 - 1) phi
            C = fma(b1, pc, -b2 * qc);
            S = fma(si, fma(d1, pc, -d2 * qc), fma(b1 * (double)j0, ps, -b2 * (double)(j0 - 1) * qs));
        }
    };
    const float dscale = 1.0f / (a.data_max - a.data_min);
    // fixed-point scale of the window: a node adds at most |fbar| |dscale| to
    // a voxel (trilinear weights sum to 1), |fbar| <= |A| + |B| <= 6.2 sum_j j |c_j|
    // + 2 pi |g0| (|C'| and |S| <= sum_j j |c_j|); 8 (...) with margin, times the
    // kChunk + 1 nodes a ray adds per chunk, over the workgroup
    {
        double sj = 0.0;
#pragma unroll
        for (int i = 0; i < M; ++i)
            sj = fma((double)(j0 + i), fabs(cc[i]), sj);
        const float lb = active ? (float)(8.0 * (sj + fabs(g0)) * (double)fabsf(dscale) * (kChunk + 1)) : 0.0f;
        atomicMax(&bound_bits, __float_as_uint(lb));
    }
    __syncthreads();
    // the same value in every lane: read as a scalar, so the branches on it
    // are uniform
    const float bsum = __uint_as_float(__builtin_amdgcn_readfirstlane(bound_bits)) * (float)blockDim.x;
    const int kfix = fixed_scale(bsum);
    // not finite: no window, float atomics straight to the volume
    const bool fixed = fixed_usable(bsum);
    // d f / d s of map_density
    auto dmap = [&](float sv) {
        const float u = div_c<POW2>(sv - a.data_min, a.data_max - a.data_min, a.data_rinv);
        return (u > 0.0f && u < 1.0f) ? dscale : 0.0f;
    };
    // clamped cell of the sample at t
    auto cell_at = [&](float tt, int &qx, int &qy, int &qz) {
        const float px = r.o.x + tt * r.d.x, py = r.o.y + tt * r.d.y, pz = r.o.z + tt * r.d.z;
        qx = iclamp((int)floorf(div_c<POW2>(px - vol.dmin.x, vol.dmax.x - vol.dmin.x, vol.rext.x) * (float)vol.nx), 0,
                    vol.nx - 1);
        qy = iclamp((int)floorf(div_c<POW2>(py - vol.dmin.y, vol.dmax.y - vol.dmin.y, vol.rext.y) * (float)vol.ny), 0,
                    vol.ny - 1);
        qz = iclamp((int)floorf(div_c<POW2>(pz - vol.dmin.z, vol.dmax.z - vol.dmin.z, vol.rext.z) * (float)vol.nz), 0,
                    vol.nz - 1);
    };

    const double rdphi = 1.0 / (double)dphi;
    // node 0: the ray's first sample, at the start of the first segment
    // (p_1 - dphi in float, or -pi when the ray has no interior sample)
    float t = t_near;
    float phi_prev;
    if (t + s < t_far && cap > 0)
        phi_prev = (float)((double)((t + s - t_near) * pi_trange_inv) - kPi) - dphi;
    else
        phi_prev = (float)(-kPi);
    // cur: the sample of the node behind the current segment; its loads are
    // issued one node ahead and used after the next node's sums
    GradSample<POW2> cur;
    double co = 1.0, si = 0.0, C_prev = 0.0, S_prev = 0.0;
    if (active)
    {
        issue_at(cur, t);
        sincos_small((double)phi_prev, si, co);
        sums(co, si, C_prev, S_prev);
    }
    double S_prev2 = S_prev, phi_prev2 = (double)phi_prev; // node k-2 for S'
    double fbar = 0.0; // pending gradient of the node behind the current segment
    CellScatter cells;
    GradTarget tg;
    tg.grad = grad_vol;
    tg.win = win;
    tg.kfix = kfix;
    tg.nx = vol.nx;
    tg.sxy = (uint32_t)(vol.nx * vol.ny);
    int it = 0;
    bool done = !active;
    while (__syncthreads_or(!done))
    {
        if (tid == 0)
        {
            bbox[0] = bbox[1] = bbox[2] = 0x7fffffff;
            bbox[3] = bbox[4] = bbox[5] = -1;
        }
        __syncthreads();
        if (!done)
        {
            // this chunk reads samples in [t, t + (kChunk + 1) s], or up to t_far
            // when it ends the ray; one cell of margin on each side
            float tb = t + (float)(kChunk + 1) * s;
            if (tb > t_far || it + kChunk >= cap)
                tb = t_far;
            int ax0, ay0, az0, ax1, ay1, az1;
            cell_at(t, ax0, ay0, az0);
            cell_at(tb, ax1, ay1, az1);
            atomicMin(&bbox[0], max(min(ax0, ax1) - 1, 0));
            atomicMin(&bbox[1], max(min(ay0, ay1) - 1, 0));
            atomicMin(&bbox[2], max(min(az0, az1) - 1, 0));
            atomicMax(&bbox[3], min(max(ax0, ax1) + 2, vol.nx - 1));
            atomicMax(&bbox[4], min(max(ay0, ay1) + 2, vol.ny - 1));
            atomicMax(&bbox[5], min(max(az0, az1) + 2, vol.nz - 1));
        }
        __syncthreads();
        tg.ox = __builtin_amdgcn_readfirstlane(bbox[0]);
        tg.oy = __builtin_amdgcn_readfirstlane(bbox[1]);
        tg.oz = __builtin_amdgcn_readfirstlane(bbox[2]);
        tg.ex = __builtin_amdgcn_readfirstlane(bbox[3]) - tg.ox + 1;
        tg.ey = __builtin_amdgcn_readfirstlane(bbox[4]) - tg.oy + 1;
        tg.ez = __builtin_amdgcn_readfirstlane(bbox[5]) - tg.oz + 1;
        {
            const long long nbox = (tg.ex > 0 && tg.ey > 0 && tg.ez > 0) ? (long long)tg.ex * tg.ey * tg.ez : -1;
            tg.mode = (nbox < 0) ? kWinGlobal
                      : (fixed && nbox <= kWin) ? kWinFixed
                      : (nbox <= 2 * kWin) ? kWinFloat
                                           : kWinGlobal;
        }
        for (int k = 0; k < kChunk && !done; ++k, ++it)
        {
            const bool last = !(t + s < t_far) || it >= cap;
            float p_next, seg;
            if (!last)
            {
                t += s;
                p_next = (float)((double)((t - t_near) * pi_trange_inv) - kPi);
                seg = dphi;
            }
            else
            {
                p_next = 0.0f;
                seg = 0.0f - phi_prev;
            }
            // the segment [pp, pn]: pp = p_next - seg in float (= phi_prev + delta)
            const double pn = (double)p_next;
            const double pp = (double)(p_next - seg);
            const double sg = pn - pp;
            const double delta = pp - (double)phi_prev;
            // cos / sin at the new node: rotated from the previous node by the
            // exact phase difference (Taylor terms to d^8 while it is below
            // 0.05; the rounding drift over a ray stays far below what the
            // sums resolve), else evaluated afresh
            {
                const double d = pn - (double)phi_prev;
                if (fabs(d) < 0.05)
                {
                    const double d2 = d * d;
                    const double cd = fma(d2, fma(d2, fma(d2, fma(d2, 1.0 / 40320, -1.0 / 720), 1.0 / 24), -0.5), 1.0);
                    const double sd = d * fma(d2, fma(d2, fma(d2, -1.0 / 5040, 1.0 / 120), -1.0 / 6), 1.0);
                    const double nc = fma(co, cd, -si * sd);
                    si = fma(si, cd, co * sd);
                    co = nc;
                }
                else
                    sincos_small(pn, si, co);
            }
            double Cn, Sn;
            sums(co, si, Cn, Sn);
            // S' at the previous node by a central difference (one-sided at the
            // first); it only multiplies delta, a few ulps, so float suffices
            const float dS = __fdividef((float)((it == 0) ? Sn - S_prev : Sn - S_prev2),
                                        (float)((it == 0) ? pn - (double)phi_prev : pn - phi_prev2));
            const double Cpp = C_prev - delta * S_prev;
            const double Spp = S_prev + delta * (double)dS;
            const double X = Cn - Cpp, V = Sn - Spp;
            const double rseg = last ? 1.0 / (double)seg : rdphi;
            const double xs = X * rseg;
            const double rr = sg * rseg;
            const double half = 0.5 * sg * rr;
            const double A = -xs + V - rr * Sn + g0 * (sg - half);
            const double B = xs + rr * Sn + g0 * half;
            fbar += A;
            const float gs0 = (float)fbar * dmap(cur.value());
            if (gs0 != 0.0f)
                cells.add(tg, cur, gs0);
            fbar = B;
            S_prev2 = S_prev;
            phi_prev2 = (double)phi_prev;
            C_prev = Cn;
            S_prev = Sn;
            phi_prev = p_next;
            __builtin_amdgcn_sched_barrier(0);
            issue_at(cur, last ? t_far : t);
            if (last)
            {
                const float gl = (float)fbar * dmap(cur.value());
                if (gl != 0.0f)
                    cells.add(tg, cur, gl);
                done = true;
            }
        }
        cells.flush(tg);
        __syncthreads();
        if (tg.mode != kWinGlobal)
        {
            // the window back to all-zero bits (a float sum may end as -0)
            // as its sums go to the volume
            // the window's voxel i at (lx, ly, lz), i = lx + ex (ly + ey lz):
            // each thread steps through i by blockDim.x, carrying lx and ly
            // over (no integer divisions in the loop)
            const int n = tg.ex * tg.ey * tg.ez;
            const int step = (int)blockDim.x;
            const int sx = step % tg.ex, sy = (step / tg.ex) % tg.ey, sz = step / (tg.ex * tg.ey);
            int lx = tid % tg.ex, ly = (tid / tg.ex) % tg.ey, lz = tid / (tg.ex * tg.ey);
            uint32_t *win32 = reinterpret_cast<uint32_t *>(win);
            for (int i = tid; i < n; i += step)
            {
                float v = 0.0f;
                bool any = false;
                if (tg.mode == kWinFixed)
                {
                    const unsigned long long q = win[i];
                    any = q != 0ull;
                    if (any)
                    {
                        win[i] = 0ull;
                        v = from_fixed(q, kfix);
                    }
                }
                else
                {
                    const uint32_t b = win32[i];
                    any = b != 0u;
                    if (any)
                    {
                        win32[i] = 0u;
                        v = __uint_as_float(b);
                    }
                }
                if (any)
                    unsafeAtomicAdd(grad_vol + ((size_t)(tg.oz + lz) * tg.sxy +
                                                (uint32_t)((tg.oy + ly) * vol.nx + tg.ox + lx)),
                                    v);
                lx += sx;
                ly += sy;
                lz += sz;
                if (lx >= tg.ex)
                {
                    lx -= tg.ex;
                    ++ly;
                }
                if (ly >= tg.ey)
                {
                    ly -= tg.ey;
                    ++lz;
                }
            }
        }
    }
}

int launch_generate_adjoint(const float *vox, int nx, int ny, int nz, const float *dmin, const float *dmax,
                            const mray_camera &cam, const mray_gen_params &p, int W, int H, int m,
                            const float *grad_moments, const float *ray_range, float *grad_volume,
                            hipStream_t stream)
{
    const float2 *rr = reinterpret_cast<const float2 *>(ray_range);
    GenArgs a;
    a.W = W;
    a.H = H;
    a.m = m;
    a.step = p.step_size;
    a.data_min = p.data_min;
    a.data_max = p.data_max;
    a.data_rinv = host_reciprocal(p.data_max - p.data_min);
    a.transform_to_bounds = p.transform_to_bounds;
    a.compact_image = p.compact_image;
    a.bound_eps = p.transform_bound_eps;
    DevCamera c = make_dev_camera(cam);
    const uint32_t ntiles = (uint32_t)(((W + 7) / 8) * ((H + 7) / 8));
    const uint32_t blocks = (ntiles + 3) / 4;
    VolumeView<float> v = make_volume_view(vox, nx, ny, nz, dmin, dmax);
    const bool pow2 = exact_pow2(v.dmax.x - v.dmin.x) && exact_pow2(v.dmax.y - v.dmin.y) &&
                      exact_pow2(v.dmax.z - v.dmin.z) && exact_pow2(a.data_max - a.data_min);
#define MRAY_GADJ_CASE(MM)                                                                                            \
    if (m <= MM)                                                                                                      \
    {                                                                                                                 \
        if (pow2)                                                                                                     \
            hipLaunchKernelGGL((generate_adjoint_kernel<MM, true>), dim3(blocks), dim3(256), 0, stream, v, c, a,      \
                               grad_moments, rr, grad_volume);                                                        \
        else                                                                                                          \
            hipLaunchKernelGGL((generate_adjoint_kernel<MM, false>), dim3(blocks), dim3(256), 0, stream, v, c, a,     \
                               grad_moments, rr, grad_volume);                                                        \
        return 0;                                                                                                     \
    }
    // 65..255 moments: chunks of at most 56 over blockIdx.y
#define MRAY_GADJ_CHUNK_CASE(MM)                                                                                      \
    if (m > 64 && m <= 255 && per <= MM)                                                                              \
    {                                                                                                                 \
        const dim3 grid(blocks, chunks);                                                                              \
        if (pow2)                                                                                                     \
            hipLaunchKernelGGL((generate_adjoint_kernel<MM, true, true>), grid, dim3(256), 0, stream, v, c, a,        \
                               grad_moments, rr, grad_volume);                                                        \
        else                                                                                                          \
            hipLaunchKernelGGL((generate_adjoint_kernel<MM, false, true>), grid, dim3(256), 0, stream, v, c, a,       \
                               grad_moments, rr, grad_volume);                                                        \
        return 0;                                                                                                     \
    }
    const int chunks = (m + 55) / 56;
    const int per = (m + chunks - 1) / chunks;
    MRAY_GADJ_CHUNK_CASE(40)
    MRAY_GADJ_CHUNK_CASE(48)
    MRAY_GADJ_CHUNK_CASE(56)
#undef MRAY_GADJ_CHUNK_CASE
    // the Clenshaw sums run over all M slots: widths close to the common
    // moment counts
    MRAY_GADJ_CASE(8)
    MRAY_GADJ_CASE(16)
    MRAY_GADJ_CASE(20)
    MRAY_GADJ_CASE(24)
    MRAY_GADJ_CASE(28)
    MRAY_GADJ_CASE(32)
    MRAY_GADJ_CASE(36)
    MRAY_GADJ_CASE(40)
    MRAY_GADJ_CASE(44)
    MRAY_GADJ_CASE(48)
    MRAY_GADJ_CASE(50)
    MRAY_GADJ_CASE(52)
    MRAY_GADJ_CASE(56)
    MRAY_GADJ_CASE(60)
    MRAY_GADJ_CASE(64)
#undef MRAY_GADJ_CASE
    return MRAY_ERR_UNSUPPORTED;
}

int launch_generate(const void *vox, int dtype, int nx, int ny, int nz, const float *dmin, const float *dmax,
                    const mray_camera &cam, const mray_gen_params &p, int form, int W, int H, int m, float *moments,
                    uint32_t *bounds, int32_t *samples, float *ray_range, hipStream_t stream)
{
    float2 *rr = reinterpret_cast<float2 *>(ray_range);
    GenArgs a;
    a.W = W;
    a.H = H;
    a.m = m;
    a.step = p.step_size;
    a.data_min = p.data_min;
    a.data_max = p.data_max;
    a.data_rinv = host_reciprocal(p.data_max - p.data_min);
    a.transform_to_bounds = p.transform_to_bounds;
    a.compact_image = p.compact_image;
    a.bound_eps = p.transform_bound_eps;
    DevCamera c = make_dev_camera(cam);
    uint32_t ntiles = (uint32_t)(((W + 7) / 8) * ((H + 7) / 8));
    uint32_t blocks = (ntiles + 3) / 4;
    if (dtype == MRAY_DTYPE_PARTICLES)
    {
        // a particle set: vox is its SphBuffers (host struct of device buffers)
        const SphBuffers *sb = static_cast<const SphBuffers *>(vox);
        VolumeView<SphParticle> v;
        v.s = sb->view();
        v.nx = v.ny = v.nz = 1;
        v.dmin = {dmin[0], dmin[1], dmin[2]};
        v.dmax = {dmax[0], dmax[1], dmax[2]};
        v.rext = {host_reciprocal(dmax[0] - dmin[0]), host_reciprocal(dmax[1] - dmin[1]),
                  host_reciprocal(dmax[2] - dmin[2])};
        if (form == MRAY_FORM_PLAIN)
        {
            int bs = plain_block(m);
            hipLaunchKernelGGL(generate_plain_kernel<SphParticle>, dim3((ntiles + bs / 64 - 1) / (bs / 64)), dim3(bs),
                               bs * m * sizeof(float), stream, v, c, a, moments, bounds, samples, rr);
            return 0;
        }
        return dispatch_mixed<SphParticle>(v, c, a, moments, bounds, samples, rr, stream, blocks);
    }
    if (dtype == MRAY_DTYPE_F32)
    {
        VolumeView<float> v = make_volume_view((const float *)vox, nx, ny, nz, dmin, dmax);
        if (form == MRAY_FORM_PLAIN)
        {
            int bs = plain_block(m);
            hipLaunchKernelGGL(generate_plain_kernel<float>, dim3((ntiles + bs / 64 - 1) / (bs / 64)), dim3(bs),
                               bs * m * sizeof(float), stream, v, c, a, moments, bounds, samples, rr);
            return 0;
        }
        return dispatch_mixed<float>(v, c, a, moments, bounds, samples, rr, stream, blocks);
    }
    VolumeView<uint8_t> v = make_volume_view((const uint8_t *)vox, nx, ny, nz, dmin, dmax);
    if (form == MRAY_FORM_PLAIN)
    {
        int bs = plain_block(m);
        hipLaunchKernelGGL(generate_plain_kernel<uint8_t>, dim3((ntiles + bs / 64 - 1) / (bs / 64)), dim3(bs),
                           bs * m * sizeof(float), stream, v, c, a, moments, bounds, samples, rr);
        return 0;
    }
    return dispatch_mixed<uint8_t>(v, c, a, moments, bounds, samples, rr, stream, blocks);
}

} // namespace mray
