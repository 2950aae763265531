// Bounded-MESE preparation: moments -> Lagrange multipliers per pixel
// (MomentImageHost::prepare_moments, src/moment_image.cpp:154-183 ->
// prepare_moments_from_std_coding, src/moment_preparation.h:55-64 ->
// prepareMESELagrange, src/mese/MESE_dynamic.h:194-211).
//
//  PLAIN  the reference FP32 arithmetic operation for operation, one thread
//         per pixel, the three complex temporaries strided through LDS (as
//         prepareMomentsKernel). sinf / cosf of the zeroth exponential
//         moment reproduce the host C library's results (host_sincosf.hpp),
//         so the multipliers are bit-identical to the reference CPU path's.
//
//  MIXED  the Herglotz transform (trigonometric -> exponential moments) and
//         the Toeplitz solve in FP64, where conditioning at 50+ moments needs
//         it; the autocorrelation and correlation stay FP64 too since FP64
//         FMA is full rate on gfx950. Four lanes work on a pixel (8 or 16
//         above 100 moments or in small images), its arrays in registers (mese_lattice.hpp).
//         The reflection coefficients come from Schur's recursion on the
//         moments instead of Levinson's inner products, together with the
//         solution polynomial in one lattice (see the kernel).
#include "launch.hpp"
#include "mese_f32.hpp"
#include "mese_lattice.hpp"

namespace mray
{


// ---------------------------------------------------------------------------
// PLAIN (FP32, one thread per pixel)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(64) void prepare_plain_kernel(const float *__restrict__ mom,
                                                           const uint32_t *__restrict__ index, int npix, int m,
                                                           float bias, float *__restrict__ out)
{
    extern __shared__ cf lds_cf[]; // 3 arrays of [m][64]
    const int tid = threadIdx.x;
    const int pix = blockIdx.x * 64 + tid;
    if (pix >= npix)
        return;
    const int nm = index ? min((int)(index[pix + 1] - index[pix]), m) : m;
    const size_t off = index ? (size_t)index[pix] : (size_t)pix * m;
    if (nm <= 0)
        return;
    const Col E{lds_cf + tid, 64}, P{lds_cf + 64 * m + tid, 64}, R{lds_cf + 2 * 64 * m + tid, 64};
    const float *t = mom + off;
    // prepare_moments_from_std_coding (src/moment_preparation.h:55-64):
    // bias lerp toward the uniform density, then prepareMESELagrange
    // (src/mese/MESE_dynamic.h:194-211)
    trig_to_exp(nm, E, [&](int i) { return i == 0 ? lerp_bias(t[0], 0.5f, bias) : lerp_bias(t[i], 0.0f, bias); });
    levinson(nm, P, E);
    lagrange_from_levinson(nm, out + off, E, P, R);
}

// ---------------------------------------------------------------------------
// MIXED (FP64, G lanes per pixel)
// ---------------------------------------------------------------------------

// For the Hermitian Toeplitz matrix of t (t_0 real) the lattice of order n
//     a^n = a^n-1 + k z b^n-1,        b^n = z b^n-1 + conj(k) a^n-1
// gives the (monic) solution polynomial a and its reverse b; the sequences
// f_i = sum_k a_k t_i-k and e_i = sum_k b_k t_i-k obey the same recursion from
// f = e = t, f_n^n-1 and the error e_n-1^n-1 = sigma are the step's only
// inner products, k = -f_n / sigma, and sigma shrinks by 1 - |k|^2 (the
// reference's |u|^2 >= 1 guard is on u = -k). Of f and e, step n needs the
// entries above n; a and b have n entries: one pair of arrays of N elements
// holds both,
//     F = f_n .. f_N-1, a_1 .. a_n          B = e_n .. e_N-2, b_0 .. b_n-1, 1
// and a step is F_i <- F_i+1 + k B_i, B_i <- B_i + conj(k) F_i+1 for all i,
// with k from F_1 and b_0 = conj(k) set at the seam i = N - n - 2, which moves
// down by one element per step (its register is known at compile time: the
// steps are unrolled by C). The other passes shift one operand down likewise:
// the Herglotz recursion X_i <- X_i+1 + (i + 1) T_i+1 E_j, whose X_0 is next
// E_j+1 up to 2 pi i / (j + 1), and the two correlations.
//
// A step costs 8 C FMAs and about 35 operations for k, the seam, two
// broadcasts and the shift, none of them LDS: at 50 moments (1024 x 1024
// pixels, FP64 multipliers) the LDS-bound Levinson kernel before took 4.37 ms,
// this one 1.92 (VALU issue in 85 to 89 % of the cycles); a compact 1000 x 777 image
// of 8 to 96 moments 6.8 and 2.85 ms. G = 4 makes the
// share of the per-step overhead small (16 pixels per wavefront) while the two
// arrays fit the registers of two wavefronts per SIMD (C <= 25).
// OutT: float multipliers, or FP64 ones for mray_hip_prepare_f64
template <int G, int C, typename OutT>
__global__ __launch_bounds__(64, 2) void prepare_mixed_kernel(const float *__restrict__ mom,
                                                           const uint32_t *__restrict__ index, int npix, int m,
                                                           float bias, OutT *__restrict__ out)
{
    constexpr int N = G * C, PX = 64 / G, S = lattice_stride(N);
    static_assert(C >= 2, "element 1 is lane 0's slot 1");
    __shared__ dc lds_c[PX * S];
    const int lane = threadIdx.x;
    const int g = lane % G, q = lane / G;
    const bool last = g == G - 1;
    const int pix = blockIdx.x * PX + q;
    const bool in = pix < npix;
    const int nm = in ? (index ? min((int)(index[pix + 1] - index[pix]), m) : m) : 0;
    const size_t off = in ? (index ? (size_t)index[pix] : (size_t)pix * m) : 0;
    // the wavefront's largest count bounds its loops
    int nw = nm;
#pragma unroll
    for (int o = G; o < 64; o <<= 1)
        nw = max(nw, __shfl_xor(nw, o, 64));
    nw = __builtin_amdgcn_readfirstlane(nw);
    if (nw == 0)
        return;

    dc *E = lds_c + q * S;
    double *T = reinterpret_cast<double *>(E);
    double V[C];
    const double t0 = load_weights<G, C>(mom, off, nm, (double)bias, g, T, V);
    double sn, cs;
    sincos(kPi * t0 - 0.5 * kPi, &sn, &cs);
    const dc e0 = dc{cs * (0.25 / kPi), sn * (0.25 / kPi)};
    herglotz<G, C>(V, e0, nw, nm, g, last, E);
    dc F[C];
    double rs;
    lattice<G, C>(E, e0, nw, nm, g, last, F, rs);

    // autocorrelation of a (computeAutocorrelation): R_i = sum_j a_j conj(a_j+i)
    dc R[C];
#pragma unroll
    for (int c = 0; c < C; ++c)
        R[c] = dc{0.0, 0.0};
    // four steps per pass: the moves of F end in a renaming of its registers
    // (one at a time they are copied, half the loop); the steps past nw add zeros
    for (int j = 0; j < nw; j += 4)
    {
#pragma unroll
        for (int u = 0; u < 4; ++u)
        {
            const dc a = bcast0<G>(F[0]);
            const dc nx = shl1<G>(F[0], last);
#pragma unroll
            for (int c = 0; c < C; ++c)
            {
                const dc b = F[c];
                R[c].x = fma(a.x, b.x, fma(a.y, b.y, R[c].x));
                R[c].y = fma(a.y, b.x, fma(-a.x, b.y, R[c].y));
                F[c] = (c + 1 < C) ? F[c + 1 < C ? c + 1 : 0] : nx;
            }
        }
    }

    // imaginary correlation with E (E_0 not doubled) and normalisation
    // (computeImaginaryCorrelation): with the solution P = a / sigma,
    // lambda = Im(sum_j 4 pi^2 (P * P)_j+i E_j) / (2 pi^2 P_0)
    double acc[C];
#pragma unroll
    for (int c = 0; c < C; ++c)
        acc[c] = 0.0;
    for (int j = 0; j < nw; j += 4)
    {
        dc e[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            e[u] = E[j + u];
#pragma unroll
        for (int u = 0; u < 4; ++u)
        {
            const dc nx = shl1<G>(R[0], last);
#pragma unroll
            for (int c = 0; c < C; ++c)
            {
                acc[c] = fma(R[c].x, e[u].y, fma(R[c].y, e[u].x, acc[c]));
                R[c] = (c + 1 < C) ? R[c + 1 < C ? c + 1 : 0] : nx;
            }
        }
    }
    wave_sync();
    const double nf = 2.0 * rs;
#pragma unroll
    for (int c = 0; c < C; ++c)
        T[g * C + c] = nf * acc[c];
    wave_sync();
#pragma unroll
    for (int r = 0; r < C; ++r)
    {
        const int e = G * r + g;
        if (e < nm)
            out[off + e] = (OutT)T[e];
    }
}

size_t g_lds_limit = 65536;

void set_lds_limit(size_t bytes) { g_lds_limit = bytes; }

namespace
{
// the MIXED preparation into float or FP64 multipliers
template <typename OutT>
int launch_prepare_mixed(const float *moments, const uint32_t *index, int npix, int m, float bias, OutT *lagrange,
                         hipStream_t stream)
{
#define MRAY_PREP_CASE(GG, CC)                                                                                        \
    if (m <= GG * CC)                                                                                                 \
    {                                                                                                                 \
        hipLaunchKernelGGL((prepare_mixed_kernel<GG, CC, OutT>), dim3((npix + 64 / GG - 1) / (64 / GG)), dim3(64), 0, \
                           stream, moments, index, npix, m, bias, lagrange);                                          \
        return 0;                                                                                                     \
    }
    // Four lanes per pixel cost the least work; where they leave SIMDs without
    // a wavefront (fewer than 1024 wavefronts of 16 pixels), more lanes make
    // each wavefront's chain of steps shorter (64 x 48 pixels, 30 moments:
    // 33 us, 15 now)
    if (npix <= 4 * 1024)
    {
        MRAY_PREP_CASE(16, 2)
        MRAY_PREP_CASE(16, 3)
        MRAY_PREP_CASE(16, 4)
        MRAY_PREP_CASE(16, 5)
        MRAY_PREP_CASE(16, 6)
        MRAY_PREP_CASE(16, 7)
        MRAY_PREP_CASE(16, 8)
        MRAY_PREP_CASE(16, 10)
        MRAY_PREP_CASE(16, 13)
        MRAY_PREP_CASE(16, 16)
    }
    if (npix <= 8 * 1024)
    {
        MRAY_PREP_CASE(8, 2)
        MRAY_PREP_CASE(8, 3)
        MRAY_PREP_CASE(8, 4)
        MRAY_PREP_CASE(8, 5)
        MRAY_PREP_CASE(8, 6)
        MRAY_PREP_CASE(8, 7)
        MRAY_PREP_CASE(8, 8)
        MRAY_PREP_CASE(8, 10)
        MRAY_PREP_CASE(8, 13)
    }
    MRAY_PREP_CASE(4, 2)
    MRAY_PREP_CASE(4, 3)
    MRAY_PREP_CASE(4, 4)
    MRAY_PREP_CASE(4, 5)
    MRAY_PREP_CASE(4, 6)
    MRAY_PREP_CASE(4, 7)
    MRAY_PREP_CASE(4, 8)
    MRAY_PREP_CASE(4, 9)
    MRAY_PREP_CASE(4, 10)
    MRAY_PREP_CASE(4, 11)
    MRAY_PREP_CASE(4, 12)
    MRAY_PREP_CASE(4, 13)
    MRAY_PREP_CASE(4, 14)
    MRAY_PREP_CASE(4, 15)
    MRAY_PREP_CASE(4, 16)
    MRAY_PREP_CASE(4, 18)
    MRAY_PREP_CASE(4, 20)
    MRAY_PREP_CASE(4, 22)
    MRAY_PREP_CASE(4, 24)
    MRAY_PREP_CASE(4, 25)
    // more moments than four lanes' registers hold
    MRAY_PREP_CASE(8, 16)
    MRAY_PREP_CASE(8, 20)
    MRAY_PREP_CASE(8, 24)
    MRAY_PREP_CASE(16, 13)
    MRAY_PREP_CASE(16, 16)
#undef MRAY_PREP_CASE
    return MRAY_ERR_UNSUPPORTED;
}
} // namespace

int launch_prepare(const float *moments, const uint32_t *index, int W, int H, int m, float bias, int form,
                   float *lagrange, hipStream_t stream)
{
    const int npix = W * H;
    if (form == MRAY_FORM_PLAIN)
    {
        size_t lds = (size_t)3 * 64 * m * sizeof(cf);
        if (lds > g_lds_limit)
            return MRAY_ERR_UNSUPPORTED;
        hipLaunchKernelGGL(prepare_plain_kernel, dim3((npix + 63) / 64), dim3(64), lds, stream, moments, index, npix,
                           m, bias, lagrange);
        return 0;
    }
    return launch_prepare_mixed<float>(moments, index, npix, m, bias, lagrange, stream);
}

int launch_prepare_f64(const float *moments, const uint32_t *index, int W, int H, int m, float bias,
                       double *lagrange, hipStream_t stream)
{
    return launch_prepare_mixed<double>(moments, index, W * H, m, bias, lagrange, stream);
}

} // namespace mray
