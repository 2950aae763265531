// Check of mray_amd/csrc/march_grid.hpp. Built and run by tests/test_march_grid.py.
// Without arguments: marches, as the gridded march does, the rays that
// grid_resolves takes, and prints
//   <rays taken> <marches that don't end> <largest |increment / s - 1|>
// With a count: sums the moments of that many rays, most of them next to the
// rule's reach, with GridStep and WeightRing, and prints their largest
// distance from the reference's integral in long double, and how many of the
// rays had an increment change.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../mray_amd/csrc/march_grid.hpp"

static double uniform(double lo, double hi) { return lo + (hi - lo) * (rand() / (double)RAND_MAX); }

// steps before t = 0 around the rule's limit and where t + s == t
static const float kReachEdge[] = {8191.0f, 8192.0f, 8193.0f, 16384.0f, 16777216.0f, 33554432.0f};
static const int kEdges = 6;

static float density(int kind, float x)
{
    const float v = kind == 0 ? 0.5f + 0.45f * sinf(40.0f * x) : kind == 1 ? (x > 0.37f ? 0.9f : 0.1f)
                    : kind == 2 ? 1.0f : 0.5f + 0.5f * tanhf((x - 0.5f) / 0.03f);
    return std::min(1.0f, std::max(0.0f, v));
}

// the ray's moments as generate.hip's gridded march sums them, against the sum
// over the reference's segments; the largest difference over the orders
static double moments_error(float t_near, float t_far, float s, int m, int kind, bool &changed)
{
    const double pi = 3.14159265358979323846;
    const float pti = (float)(pi / (double)(t_far - t_near)), dphi = (float)(pi * (double)(s / (t_far - t_near)));
    const double ptid = pti, dphid = dphi, rdphi = 1.0 / dphid;
    std::vector<long double> ref(m, 0.0L);
    std::vector<double> sc(m, 0.0);
    auto at = [&](float t) { return density(kind, (t - t_near) / (t_far - t_near)); };
    auto phase = [&](float t) { return (float)((double)((t - t_near) * pti) - pi); };
    auto grid = [&](float t) { return fma((double)t - (double)t_near, ptid, -pi); };
    // a line of slope g from (u, f) to p
    auto segment = [&](long double u, long double p, long double g, long double f) {
        const long double fp = f + g * (p - u);
        for (int j = 1; j < m; ++j)
            ref[j] += (g * cosl(j * p) + fp * j * sinl(j * p) - g * cosl(j * u) - f * j * sinl(j * u)) / ((long double)j * j);
    };
    float t = t_near;
    const float f0 = at(t), phase0 = phase(t + s) - dphi;
    mray::GridStep step;
    step.start((t + s) - t, ptid);
    const double step0 = (double)step.ds * ptid;
    mray::WeightRing ring;
    std::vector<double> weight, q(1, -pi);
    double f_prev = f0, p_prev = phase0, g_left = 0.0, w_left = 0.0, eps = p_prev + pi;
    changed = false;
    for (int ns = 1; t + s < t_far; ++ns)
    {
        const float tn = t + s, inc = tn - t;
        double shift = 0.0;
        if (inc != step.ds)
        {
            shift = step.change(inc, ptid);
            changed = true;
        }
        t = tn;
        const float p = phase(t), f = at(t);
        const double u = (double)(p - dphi), g = ((double)f - f_prev) * rdphi, width = (double)p - u;
        segment(u, p, ((long double)f - f_prev) / dphi, f_prev);
        const double delta = ns > 1 ? u - p_prev : 0.0, d = g_left - g;
        const double cp = fma(d, eps, -fma(g, delta, g_left * w_left)), A = step.second(f_prev * delta);
        weight.push_back(ring.push(d, A, step.first(cp, A, shift)));
        g_left = g;
        w_left = width - dphid;
        f_prev = f;
        p_prev = p;
        q.push_back(grid(t));
        eps = p_prev - q.back();
    }
    const float f = at(t_far);
    const double dl = 0.0 - p_prev, g = ((double)f - f_prev) / dl, d = g_left - g;
    segment(p_prev, 0.0L, ((long double)f - f_prev) / dl, f_prev);
    weight.push_back(ring.push(d, 0.0, fma(d, eps, -g_left * w_left) * step.rstep));
    for (int i = 0; i < 8; ++i)
        weight.push_back(ring.pop());
    const int last = (int)q.size() - 1;
    const double step1 = (double)step.ds * ptid;
    for (size_t i = 0; i < weight.size(); ++i)
    {
        // the grid continued past the ray's ends
        const int k = (int)i - 4;
        const double x = k < 0 ? -pi + k * step0 : k <= last ? q[k] : q[last] + (k - last) * step1;
        for (int j = 1; j < m; ++j)
            sc[j] += weight[i] * std::cos(j * x);
    }
    double worst = 0.0;
    for (int j = 1; j < m; ++j)
    {
        const double v = (sc[j] + g) / ((double)j * j) - (double)f0 * std::sin(j * (double)phase0) / j;
        worst = std::max(worst, (double)fabsl(v - ref[j]) / pi);
    }
    return worst;
}

static int check_moments(int rays)
{
    double worst = 0.0;
    int changes = 0;
    for (int i = 0; i < rays; ++i)
    {
        // ends at 0.3 to 1 of the reach; long rays, short ones and ones that begin behind the camera
        const float s = (float)std::exp(uniform(std::log(1e-4), std::log(1e-1)));
        const float t_far = (float)(mray::kGridReach * s * uniform(0.3, 0.9999));
        const int m = 4 + rand() % 50;
        const double length = (m - 1) * 3.2 * s * std::exp(uniform(0.0, 2.0));
        float t_near = (float)(t_far - length);
        if (i % 8 == 0)
            t_near = -(float)(s * uniform(1.0, 2000.0));
        const float dphi = (float)(3.14159265358979323846 * (double)(s / (t_far - t_near)));
        if (!mray::grid_resolves(m, dphi, t_near, t_far, s))
            continue;
        bool changed;
        worst = std::max(worst, moments_error(t_near, t_far, s, m, i % 4, changed));
        changes += changed;
    }
    bool changed;
    for (int kind = 0; kind < 4; ++kind)
    {
        // rays whose increment changes next to the reach
        worst = std::max(worst, moments_error(15.3f, 16.5f, 0.002017f, 16, kind, changed));
        worst = std::max(worst, moments_error(7.8248f, 8.8147f, 0.0012374f, 40, kind, changed));
    }
    printf("%.3e %d\n", worst, changes);
    return 0;
}

int main(int argc, char **argv)
{
    srand(1);
    if (argc > 1)
        return check_moments(atoi(argv[1]));
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
