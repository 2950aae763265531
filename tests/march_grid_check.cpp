// Check of mray_amd/csrc/march_grid.hpp: marches, as the gridded march does, the
// rays that grid_resolves takes. Built and run by tests/test_march_grid.py.
// Prints "<rays taken> <marches that don't end> <largest |increment / s - 1|>".
#include <cmath>
#include <cstdio>
#include <cstdlib>

#include "../mray_amd/csrc/march_grid.hpp"

static double uniform(double lo, double hi) { return lo + (hi - lo) * (rand() / (double)RAND_MAX); }

// steps before t = 0 around the rule's limit and where t + s == t
static const float kReachEdge[] = {8191.0f, 8192.0f, 8193.0f, 16384.0f, 16777216.0f, 33554432.0f};
static const int kEdges = 6;

int main()
{
    srand(1);
    long taken = 0, endless = 0;
    double worst = 0.0;
    for (int i = 0; i < 300000; ++i)
    {
        const float s = (float)std::exp(uniform(std::log(1e-4), std::log(10.0)));
        // up to 2^27 steps before t = 0 and 2^14 behind it, or all behind it
        const float t_far = (float)(s * std::exp(uniform(0.0, 14 * std::log(2.0))));
        const float t_near = (i % 3 == 0) ? (float)(t_far * uniform(0.0, 1.0))
                             : (i % 3 == 1) ? -(float)(s * std::exp(uniform(0.0, 27 * std::log(2.0))))
                                            : -kReachEdge[i / 3 % kEdges] * s;
        const int m = 1 + rand() % 60;
        const float dphi = (float)(3.14159265358979323846 * (double)(s / (t_far - t_near)));
        if (!mray::grid_resolves(m, dphi, t_near, t_far, s))
            continue;
        ++taken;
        int it = 0;
        for (float t = t_near; t + s < t_far && it <= 20000; t += s, ++it)
        {
            const float inc = (t + s) - t;
            worst = std::fmax(worst, std::fabs((double)inc / s - 1.0));
        }
        endless += it > 20000; // 16384 steps from end to end, 2^-11 longer at most
    }
    printf("%ld %ld %.9f\n", taken, endless, worst);
    return 0;
}
