// GPU check of the shared-divisor quotients of physics.hpp against the host's IEEE results, bit
// for bit: quot with recip, with recip_kb (the reciprocal of rho kb from that of rho) and with a
// correctly rounded reciprocal as tables and kernel arguments hold it, and speed_sqrt.  Operands
// are random over wide exponent ranges with significands that are also near all ones or near a
// power of two; square roots add zeros, infinity, NaN, negative arguments and perfect squares.
// Prints "<name>: N values, M mismatches" per check; exits 0 only when every M is 0.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <vector>

#include "physics.hpp"

namespace {

uint64_t next(uint64_t& s)
{
    s ^= s << 13;
    s ^= s >> 7;
    s ^= s << 17;
    return s;
}

double draw(uint64_t& s, int emin, int emax)
{
    uint64_t sig = next(s) & ((1ull << 52) - 1);
    switch (next(s) % 4) {
    case 0: sig = ((1ull << 52) - 1) - (sig & 0xFF); break;
    case 1: sig &= 0xFF; break;
    default: break;
    }
    int const e = emin + (int)(next(s) % (uint64_t)(emax - emin + 1));
    uint64_t const bits = ((uint64_t)(e + 1023) << 52) | sig;
    double d;
    std::memcpy(&d, &bits, 8);
    return d;
}

__global__ void k_check(const double* a, const double* b, const double* y, double* out, int n)
{
    int const t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    double const rho = b[t];
    out[t] = hclpp::quot(a[t], rho, hclpp::recip(rho));
    out[t + n] = hclpp::quot(a[t], rho * hclpp::kKb, hclpp::PerfectGas::recip_kb(rho, hclpp::recip(rho)));
    out[t + 2 * n] = hclpp::quot(a[t], rho, y[t]);
    out[t + 3 * n] = hclpp::speed_sqrt(a[t]);
}

bool same(double x, double y)
{
    if (std::isnan(x) || std::isnan(y)) return std::isnan(x) && std::isnan(y);
    return std::memcmp(&x, &y, 8) == 0;
}

}  // namespace

int main()
{
    int const n = 1 << 22;
    std::vector<double> a(n), b(n), y(n), out(4 * (size_t)n);
    uint64_t s = 0x9E3779B97F4A7C15ull;
    double const special[] = {0.0, -0.0, INFINITY, NAN, -1.0, 1.0, 4.0, 1e-200};
    for (int i = 0; i < n; ++i) {
        a[i] = draw(s, -300, 300);
        b[i] = draw(s, -300, 300);
        if (i % 1024 < 8) a[i] = special[i % 1024];
        else if (i % 16 == 9) a[i] = std::floor(std::ldexp(draw(s, 0, 20), 3)) * std::floor(std::ldexp(draw(s, 0, 20), 3));
        y[i] = 1 / b[i];
    }
    double *da, *db, *dy, *d;
    auto ok = [](hipError_t e) {
        if (e != hipSuccess) std::printf("%s\n", hipGetErrorString(e));
        return e == hipSuccess;
    };
    size_t const bytes = sizeof(double) * n;
    if (!ok(hipMalloc(&da, bytes)) || !ok(hipMalloc(&db, bytes)) || !ok(hipMalloc(&dy, bytes)) || !ok(hipMalloc(&d, 4 * bytes))) return 2;
    if (!ok(hipMemcpy(da, a.data(), bytes, hipMemcpyHostToDevice)) || !ok(hipMemcpy(db, b.data(), bytes, hipMemcpyHostToDevice)) ||
        !ok(hipMemcpy(dy, y.data(), bytes, hipMemcpyHostToDevice)))
        return 2;
    hipLaunchKernelGGL(k_check, dim3(n / 256), dim3(256), 0, nullptr, da, db, dy, d, n);
    if (!ok(hipGetLastError()) || !ok(hipMemcpy(out.data(), d, 4 * bytes, hipMemcpyDeviceToHost))) return 2;
    char const* names[] = {"recip", "recip_kb", "table", "speed_sqrt"};
    int total = 0;
    for (int c = 0; c < 4; ++c) {
        int bad = 0;
        for (int i = 0; i < n; ++i) {
            double const want = c == 1 ? a[i] / (b[i] * hclpp::kKb) : (c == 3 ? std::sqrt(a[i]) : a[i] / b[i]);
            if (!same(out[(size_t)c * n + i], want)) ++bad;
        }
        std::printf("%s: %d values, %d mismatches\n", names[c], n, bad);
        total += bad;
    }
    return total ? 1 : 0;
}
