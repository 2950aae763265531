// Check of mray_amd/csrc/digit_ring.hpp: sequences of digits and carries through
// the ring, 64 lanes emulated, against bytes written and carried one by one.
// Built and run by tests/test_digit_ring.py; prints "<sequences> <that differ>
// <carries into bytes already out> <flushes that ran more than one round>".
#include <array>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../mray_amd/csrc/digit_ring.hpp"

static long rounds, late_carries, long_flushes;

struct HostWave
{
    using u32 = std::array<uint32_t, 64>;
    template <typename F> static u32 each(F f)
    {
        u32 r;
        for (uint32_t i = 0; i < 64; ++i)
            r[i] = f(i);
        return r;
    }
    static bool first() { return true; }
    static void add(uint32_t *p, uint32_t v) { *p += v; }
    static void sync()
    {
        long_flushes += rounds > 1;
        rounds = 0;
    }
    static void fence() { ++late_carries; }
    static u32 load(const uint32_t *ring, uint32_t at, uint32_t n)
    {
        return each([&](uint32_t i) { return i < n ? ring[(at + i) & 127u] : 0u; });
    }
    static bool any_above(const u32 &v, uint32_t top)
    {
        for (uint32_t x : v)
            if (x > top)
            {
                ++rounds;
                return true;
            }
        return false;
    }
    static u32 shift_right(const u32 &v, int k) { return each([&](uint32_t i) { return v[i] >> k; }); }
    static u32 low_bits(const u32 &v, uint32_t m) { return each([&](uint32_t i) { return v[i] & m; }); }
    static u32 plus(const u32 &a, const u32 &b) { return each([&](uint32_t i) { return a[i] + b[i]; }); }
    static uint32_t lane0(const u32 &v) { return v[0]; }
    static u32 from_next(const u32 &v) { return each([&](uint32_t i) { return i < 63 ? v[i + 1] : 0u; }); }
    static void store(uint8_t *out, size_t cap, size_t at, const u32 &v, uint32_t n)
    {
        for (uint32_t i = 0; i < n; ++i)
        {
            const size_t p = at + 2 * (size_t)i;
            if (p < cap)
                out[p] = (uint8_t)(v[i] >> 8);
            if (p + 1 < cap)
                out[p + 1] = (uint8_t)v[i];
        }
    }
};

// digits with a carry behind some of them, to capacity cap
static bool differs(const std::vector<uint32_t> &digits, const std::vector<char> &carry, size_t cap)
{
    std::vector<uint8_t> a(2 * digits.size() + 8, 0xA5), b(a);
    uint32_t ring[128];
    for (uint32_t &r : ring)
        r = 0xDEADBEEFu;
    mray::DigitRing<HostWave> R{a.data(), cap, ring, 0u, 0u};
    size_t pos = 0;
    for (size_t i = 0; i < digits.size(); ++i)
    {
        R.put(digits[i]);
        for (uint32_t byte : {digits[i] >> 8, digits[i] & 0xFFu})
        {
            if (pos < cap)
                b[pos] = (uint8_t)byte;
            ++pos;
        }
        if (carry[i])
        {
            R.carry();
            // the reference's propagate_carry
            size_t p = pos - 1;
            while (p < cap && b[p] == 0xFFu)
                b[p--] = 0;
            if (p < cap)
                b[p] = (uint8_t)(b[p] + 1);
        }
    }
    R.flush_all();
    return a != b;
}

int main()
{
    long n = 0, bad = 0;
    srand(1);
    // a run of 0xFFFF of every length up to 200 behind `lead` digits, the carry
    // right behind its last digit, `tail` digits after it (none, up to past the next flush)
    for (int lead : {1, 31, 32, 33, 63, 64, 65, 95, 96, 97, 130})
        for (int run = 0; run <= 200; ++run)
            for (int tail : {0, 1, 40, 70, 100})
            {
                std::vector<uint32_t> d;
                for (int i = 0; i < lead; ++i)
                    d.push_back((uint32_t)rand() & 0x7FFFu);
                d.insert(d.end(), (size_t)run, 0xFFFFu);
                std::vector<char> c(d.size(), 0);
                c.back() = 1;
                for (int i = 0; i < tail; ++i)
                {
                    d.push_back((uint32_t)rand() & 0xFFFFu);
                    c.push_back(0);
                }
                ++n;
                bad += differs(d, c, 2 * d.size() + 8);
            }
    // random digits, many of them 0xFFFF or 0, carries where they leave a code
    // below 1, and capacities that truncate the code without a carry
    for (int k = 0; k < 20000; ++k)
    {
        std::vector<uint32_t> d(1, 0x1234u);
        std::vector<char> c(1, 0);
        const int len = rand() % 400;
        const int kind = rand() % 3;
        bool full = false; // the newest digits already carried into
        for (int i = 0; i < len; ++i)
        {
            const uint32_t v = kind == 0 ? (uint32_t)rand() & 0xFFFFu : (rand() % 16 ? 0xFFFFu : (uint32_t)rand() & 0xFFFFu);
            d.push_back(v);
            // one carry at most into each run of 0xFFFF: it leaves zeros behind
            const bool room = !full;
            c.push_back(room && rand() % (kind == 2 ? 64 : 8) == 0);
            full = c.back() || (full && v == 0xFFFFu);
        }
        const bool cut = k % 4 == 0;
        if (cut)
            std::fill(c.begin(), c.end(), 0);
        ++n;
        bad += differs(d, c, cut ? (size_t)(rand() % (2 * len + 3)) : 2 * d.size() + 8);
    }
    printf("%ld %ld %ld %ld\n", n, bad, late_carries / 2, long_flushes);
    return 0;
}
