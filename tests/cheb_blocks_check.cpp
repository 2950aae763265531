// Check of mray_amd/csrc/cheb_blocks.hpp against direct sums of cos(j theta) in
// long double, for every width 1..128. Built and run by
// tests/test_cheb_blocks.py. Prints the largest error of the series and of the
// sums, each relative to the sum of its terms' magnitudes.
#include <cstdio>
#include <cstdlib>
#include <cmath>

#include "../mray_amd/csrc/cheb_blocks.hpp"

static double worst_series = 0.0, worst_sums = 0.0;

static double uniform(double lo, double hi) { return lo + (hi - lo) * (rand() / (double)RAND_MAX); }

template <int M> void check()
{
    constexpr int P = mray::block_width<M>();
    double mu[M], c[M], sums[M];
    long double ref[M], mag = 0.0L;
    for (int j = 0; j < M; ++j)
    {
        mu[j] = c[j] = uniform(-1e3, 1e3);
        sums[j] = 0.0;
        ref[j] = 0.0L;
        mag += std::fabs(mu[j]);
    }
    mray::block_coefficients<M>(c);
    long double wmag = 0.0L;
    for (int i = 0; i < 200; ++i)
    {
        // the ends of [0, pi] among the angles
        const double theta = (i == 0) ? 0.0 : (i == 1) ? M_PI : uniform(0.0, M_PI);
        const double x = std::cos(theta), w = uniform(-50.0, 50.0);
        const long double th = acosl((long double)x);
        double T[P + 1];
        mray::cheb_low<P>(T, x);
        long double s = 0.0L;
        for (int j = 0; j < M; ++j)
        {
            s += mu[j] * cosl(j * th);
            ref[j] += w * cosl(j * th);
        }
        wmag += std::fabs(w);
        worst_series = std::fmax(worst_series, (double)(fabsl(s - mray::block_series<M>(c, T)) / mag));
        mray::block_sums<M, 0>(sums, w, T);
    }
    mray::untangle_sums<M>(sums);
    for (int j = 0; j < M; ++j)
        worst_sums = std::fmax(worst_sums, (double)(fabsl(ref[j] - sums[j]) / wmag));
}

template <int M> void all()
{
    check<M>();
    if constexpr (M > 1)
        all<M - 1>();
}

int main()
{
    srand(1);
    all<128>();
    printf("%.3e %.3e\n", worst_series, worst_sums);
    return 0;
}
