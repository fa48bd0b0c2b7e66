// Runs the scalar functions of the projection over whole ranges of floats against the host's exp, log and division.
// Prints a line per sweep: its name, the values compared, those that differ, and the first few of these.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <mutex>
#include <thread>
#include <vector>

#include "trips_math.h"

namespace
{
double2 g_table[trips::kLogTable];

bool same(float a, float b) { return __float_as_uint(a) == __float_as_uint(b) || (a != a && b != b); }

// f(u, report) for u in [first, last], by pieces, on all threads; report(u) notes a difference
template <typename F>
void sweep(const char* name, uint64_t first, uint64_t last, F&& f)
{
    constexpr uint64_t kPiece = 1u << 18;
    std::atomic<uint64_t> next{first}, bad{0};
    std::mutex mutex;
    std::vector<uint64_t> which;
    auto report = [&](uint64_t u)
    {
        bad += 1;
        std::lock_guard<std::mutex> lock(mutex);
        if (which.size() < 4) which.push_back(u);
    };
    std::vector<std::thread> threads;
    for (unsigned i = 0; i < std::max(1u, std::thread::hardware_concurrency()); ++i)
        threads.emplace_back(
            [&]()
            {
                for (uint64_t at = next.fetch_add(kPiece); at <= last; at = next.fetch_add(kPiece))
                    for (uint64_t u = at; u < at + kPiece && u <= last; ++u) f(u, report);
            });
    for (auto& t : threads) t.join();
    std::printf("%s %llu %llu", name, (unsigned long long)(last - first + 1), (unsigned long long)bad.load());
    std::sort(which.begin(), which.end());
    for (uint64_t u : which) std::printf(" 0x%llx", (unsigned long long)u);
    std::printf("\n");
    std::fflush(stdout);
}

uint64_t mix(uint64_t z)  // splitmix64
{
    z += 0x9e3779b97f4a7c15ull;
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}
}  // namespace

int main()
{
    using namespace trips;
    for (int i = 0; i < kLogTable; ++i) g_table[i] = log_table_entry(i);
    // the exponential, and softplus with its derivative, of every float of a sign with magnitude 2^-27 to 200
    auto softplus_of = [](uint64_t u, auto& report)
    {
        const float x = __uint_as_float((uint32_t)u), e = (float)std::exp((double)x);
        if (!same(exp_rn(x), e)) report(u);
        float d = 0.f;
        const float y = softplus(x, g_table, &d);
        if (!same(y, x > 20.f ? x : (float)std::log((double)(1.f + e))) || !same(d, x > 20.f ? 1.f : e / (e + 1.f))) report(u);
    };
    const uint32_t small = __float_as_uint(0x1p-27f), most = __float_as_uint(200.f), sign = 0x80000000u;
    sweep("softplus+", small, most, softplus_of);
    sweep("softplus-", (uint64_t)sign | small, (uint64_t)sign | most, softplus_of);
    // below, where the exponential is 1: every 97th, zero and the denormals among them
    sweep("softplus0", 0, 2 * (small / 97), [&](uint64_t i, auto& report) { softplus_of((i / 2) * 97 | (i % 2 ? sign : 0u), report); });
    // the logarithm of every float from 1 to 1 + exp(20)
    sweep("log", __float_as_uint(1.f), __float_as_uint(1.f + (float)std::exp(20.0)),
          [](uint64_t u, auto& report)
          {
              const float z = __uint_as_float((uint32_t)u);
              if (!same(log_rn(z, g_table), (float)std::log((double)z))) report(u);
          });
    // quotients by positive numbers: any two floats; two whose quotient lies below the normal numbers; and of these the ones that
    // are the middle between two floats, a = m b with an odd number m of half units
    auto divide = [](float a, float b, uint64_t i, auto& report)
    {
        t_rcp_units = (int)(i % 3) - 1;
        const double reciprocal = reciprocal_of(b);
        if (!same(quotient_of_any_size(a, b, reciprocal), a / b)) report(i);
        if (!(std::fabs(a / b) < 0x1p-126f) && !same(quotient(a, reciprocal), a / b)) report(i);
    };
    constexpr uint64_t kMany = 20000000;
    sweep("quotient", 0, kMany,
          [&](uint64_t i, auto& report)
          {
              const uint64_t r = mix(i);
              const uint32_t b = std::min((uint32_t)(r >> 33) + 1u, 0x7f7fffffu);
              divide(__uint_as_float((uint32_t)r), __uint_as_float(b), i, report);
          });
    sweep("quotient_small", 0, kMany,
          [&](uint64_t i, auto& report)
          {
              const uint64_t r = mix(i);
              const int eb = 24 + (int)(r % 230), ea = std::min(std::max(eb - 127 - (int)((r >> 8) % 26), 0), 254);  // biased exponents
              divide(__uint_as_float((uint32_t)(ea << 23) | ((uint32_t)(r >> 16) & 0x807fffffu)),
                     __uint_as_float((uint32_t)(eb << 23) | ((uint32_t)(r >> 41) & 0x7fffffu)), i, report);
          });
    sweep("quotient_middle", 0, kMany,
          [&](uint64_t i, auto& report)
          {
              const uint64_t r = mix(i);
              const int bits = 2 + (int)(r % 22);  // of b's odd part; m has the rest of 24
              const uint64_t odd_b = (r >> 8) % (1ull << bits) | 1ull, m = (r >> 32) % (1ull << (24 - bits)) | 1ull;
              const int k = 1 + (int)((r >> 56) % 100);
              const float b = std::ldexp((float)odd_b, k), a = std::ldexp((float)(odd_b * m), k - 150);
              if (b < INFINITY && (double)a / (double)b == std::ldexp((double)m, -150)) divide(a, b, i, report);
          });
    return 0;
}
