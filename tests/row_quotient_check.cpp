// ternainfer_amd/csrc/row_quotient.h against the division it stands for, bit for bit: built with g++ (no contraction) and run by test_row_quotient.py.
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <thread>
#include <vector>

#pragma GCC diagnostic ignored "-Wunknown-pragmas"
#include "../ternainfer_amd/csrc/row_quotient.h"

static float from_bits(uint32_t u)
{
    float f;
    std::memcpy(&f, &u, 4);
    return f;
}
static uint32_t bits(float f)
{
    uint32_t u;
    std::memcpy(&u, &f, 4);
    return u;
}

// The first of the sums +-first, +-(first + 2 step), ... up to about `last` whose quotients by `scale` are not the division's, or 0.  NaNs agree whatever their bits.
static int64_t unequal(float scale, int64_t first, int64_t last, int64_t step)
{
    const terna::RowQuotient by(scale);
    constexpr int F = 16;
    for (int64_t n = first; n <= last; n += F * step) {
        float x[F], want[F];
        for (int v = 0; v < F; ++v) {
            x[v] = static_cast<float>((v & 1 ? -1 : 1) * (n + v / 2 * 2 * step));
            want[v] = x[v] / scale;
        }
        by.of(x);
        for (int v = 0; v < F; ++v)
            if (bits(x[v]) != bits(want[v]) && !(std::isnan(x[v]) && std::isnan(want[v]))) return n + v / 2 * 2 * step;
    }
    return 0;
}

int main()
{
    std::vector<std::thread> threads;
    std::vector<int> failed(8, 0);
    for (int t = 0; t < 8; ++t)
        threads.emplace_back([t, &failed] {
            auto check = [&](float scale, int64_t first, int64_t last, int64_t step) {
                const int64_t at = unequal(scale, first, last, step);
                if (at != 0) std::printf("%a at %lld\n", scale, static_cast<long long>(at)), failed[t] = 1;
            };
            for (uint32_t mantissa = t; mantissa < 128; mantissa += 8) {
                // a power of two more or less moves every intermediate by as much; 127 / s of a row is within 2^-20 .. 2^24 for all but absurd rows
                const float scale = from_bits((127u << 23) | (mantissa << 16));
                check(scale, 1, 1 << 22, 1);                           // odd sums of both signs,
                check(scale, 2, 1 << 22, 1);                           // even ones
                check(scale, (1 << 22) + 1, 0x7fffffffll - 4096, 4099);
                for (int exponent : {1, 20, 66, 67, 68, 100, 150, 186, 187, 188, 230, 254}) {
                    const float there = from_bits((static_cast<uint32_t>(exponent) << 23) | (mantissa << 16));
                    check(there, 1, 1 << 12, 1);
                    check(there, 1 << 22, 0x7fffffffll - 65536, 104729);
                    check(-there, 1, 1 << 8, 1);
                }
            }
        });
    for (auto& t : threads) t.join();
    for (uint32_t special : {0x00000000u, 0x80000000u, 0x00010000u, 0x007f0000u, 0x7f800000u, 0xff800000u, 0x7fc00000u, 0x7f7f0000u}) {
        float zero[1] = {0.0f}, one[1] = {1.0f};
        const terna::RowQuotient by(from_bits(special));
        by.of(zero);
        by.of(one);
        const float want0 = 0.0f / from_bits(special), want1 = 1.0f / from_bits(special);
        if ((bits(zero[0]) != bits(want0) && !std::isnan(want0)) || std::isnan(zero[0]) != std::isnan(want0) || (bits(one[0]) != bits(want1) && !std::isnan(want1)) ||
            std::isnan(one[0]) != std::isnan(want1))
            std::printf("special %08x\n", special), failed[0] = 1;
    }
    for (int f : failed)
        if (f) return 1;
    std::printf("row quotient ok\n");
    return 0;
}
