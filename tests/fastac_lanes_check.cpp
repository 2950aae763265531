// Check of mray_amd/csrc/fastac_lanes.hpp: codes decoded by 64 lanes as the
// entropy kernel does, against the reference's bisection on the same model
// (double arithmetic in the reference's order). Built and run by
// tests/test_fastac_lanes.py with the width, the code's byte (-1: random
// bytes) and the symbol count; prints "<first symbol that differs, or -1>
// <1 if the code's value went to infinity>".
#include <cstdio>
#include <cstdlib>
#include <cmath>
#include <vector>

#include "../mray_amd/csrc/fastac_lanes.hpp"

using mray::LaneOffer;
constexpr double kOut = 65536.0, kMin = 1.0 / 65536.0, kLsb = 1.0 / 281474976710656.0, kLeak = 2.0 * kLsb;

struct Model
{
    uint32_t A, total = 0, cycle, until = 0;
    std::vector<uint32_t> count;
    std::vector<double> d;
    explicit Model(uint32_t n) : A(n), cycle(n), count(n, 1u), d(n)
    {
        update();
        cycle = until = (A + 6) >> 1;
    }
    void update()
    {
        if ((total += cycle) > (1u << 17))
        {
            total = 0;
            for (uint32_t &c : count)
                total += c = (c + 1) >> 1;
        }
        uint32_t run = 0;
        const double scale = 1.0 / (double)total;
        for (uint32_t k = 0; k < A; ++k)
        {
            d[k] = scale * (double)run;
            run += count[k];
        }
        cycle = (5 * cycle) >> 2;
        const uint32_t cap = (A + 6) << 3;
        cycle = until = cycle > cap ? cap : cycle;
    }
};

struct State
{
    double base = 0.0, length = 1.0, value = 0.0;
    size_t pos = 0;
};

static int code_byte;
static std::vector<uint8_t> code;
static double byte(size_t i) { return code_byte >= 0 ? code_byte : code[i]; }

static void narrow(State &S, double x, double y)
{
    S.base = x;
    S.length = y - x;
    if (S.base >= 1.0)
    {
        S.base -= 1.0;
        S.value -= 1.0;
    }
    if ((S.length -= kLeak) <= kMin)
        do
        {
            S.base *= kOut;
            const double a = (double)(uint32_t)S.base;
            S.base -= a;
            S.value = (kOut * S.value - a) + kLsb * (256.0 * byte(S.pos) + byte(S.pos + 1));
            S.pos += 2;
        } while ((S.length *= kOut) <= kMin);
}

static uint32_t bisect(State &S, const Model &M)
{
    uint32_t s = 0, n = M.A, mid = n >> 1;
    double x = S.base, y = S.base + S.length;
    const double sv = S.value + kLsb;
    do
    {
        const double z = S.base + S.length * M.d[mid];
        if (z > sv)
        {
            y = z;
            n = mid;
        }
        else
        {
            x = z;
            s = mid;
        }
    } while ((mid = (s + n) >> 1) != s);
    narrow(S, x, y);
    return s;
}

template <int R> static uint32_t lanes(State &S, const Model &M)
{
    LaneOffer o[64];
    int j = 0;
    for (int i = 0; i < 64; ++i)
    {
        double d[R + 1];
        for (int r = 0; r <= R; ++r)
        {
            const uint32_t k = (uint32_t)(i * R + r);
            d[r] = mray::lane_dist(k, M.A, k < M.A ? M.d[k] : 0.0, r == R);
        }
        o[i] = mray::lane_offer<R>(d, S.base, S.length, S.value + kLsb);
        // the ballot's population count: the qualifying lanes are a prefix
        j += o[i].any;
    }
    j = j > 0 ? j - 1 : 0;
    narrow(S, o[j].x, o[j].y);
    return (uint32_t)(j * R) + o[j].sub;
}

int main(int argc, char **argv)
{
    const int bits = atoi(argv[1]);
    code_byte = atoi(argv[2]);
    const long n = atol(argv[3]);
    if (code_byte < 0)
    {
        srand(bits);
        code.resize((size_t)(2 * n) + 64);
        for (uint8_t &b : code)
            b = (uint8_t)(rand() >> 7);
    }
    Model M(1u << bits);
    State A, B;
    for (size_t k = 0; k < 6; ++k)
        A.value = 256.0 * A.value + kLsb * byte(k);
    A.pos = 6;
    B = A;
    long first = -1;
    for (long i = 0; i < n && first < 0; ++i)
    {
        const uint32_t want = bisect(A, M);
        const uint32_t got = bits <= 6 ? lanes<1>(B, M) : bits == 7 ? lanes<2>(B, M) : lanes<4>(B, M);
        if (got != want || A.base != B.base || A.length != B.length)
            first = i;
        ++M.count[want];
        if (--M.until == 0)
            M.update();
    }
    printf("%ld %d\n", first, (int)std::isinf(A.value));
    return 0;
}
