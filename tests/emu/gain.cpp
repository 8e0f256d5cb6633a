// CPU check that the FP32 operators have no systematic gain: the mean change
// of |a|^2 by rounding over many random values, which adds up linearly over
// the z-slices.  Prints <label> <relative bias of the power>.
#include <hip/hip_runtime.h>
#include <cstdio>
#include <random>
#include <vector>
#include "../../cuopo3d_amd/csrc/opo_tables.hpp"
using namespace opo;

// Table entries exp(-la + i theta), 4e6 values.
void multiply(const char *label, double theta, double la) {
    std::mt19937_64 rng(1);
    std::normal_distribution<double> g;
    const double c = std::exp(-la) * std::cos(theta), s = std::exp(-la) * std::sin(theta);
    const cplx<float> hi = {(float)c, (float)s}, lo = {(float)(c - hi.x), (float)(s - hi.y)};
    double bias = 0, den = 0;
    for (int i = 0; i < 4000000; ++i) {
        const cplx<float> a = {(float)g(rng), (float)g(rng)}, b = cmul_hl(a, hi, lo);
        const double x = a.x * c - a.y * s, y = a.x * s + a.y * c;
        bias += 2 * (x * (b.x - x) + y * (b.y - y));
        den += x * x + y * y;
    }
    std::printf("%s %.6e\n", label, bias / den);
}

// One time-line operator with quadratic phases up to theta on fresh noise.
template <int N> void line(const char *label, double theta) {
    const int L = 4000000 / N;
    std::mt19937_64 rng(N);
    std::normal_distribution<double> g;
    const LineShape s = line_shape<float>(N, USE_T);
    std::vector<cplx<float>> tw(2 * N + 1), tab(2 * N), f(N);
    tw_fill(s, [&](size_t i, double t, double r) { tw[i] = {(float)t, (float)r}; });
    for (int i = 0; i < N; ++i) {
        const int k = tw_slot_bin(s, i);
        const double u = (k < N / 2 ? k : k - N) / (0.5 * N), c = std::cos(theta * u * u) / N, q = std::sin(theta * u * u) / N;
        tab[2 * i] = {(float)c, (float)q};
        tab[2 * i + 1] = {(float)(c - tab[2 * i].x), (float)(q - tab[2 * i].y)};
    }
    double n0 = 0, n1 = 0;
    for (int l = 0; l < L; ++l) {
        for (auto &v : f) {
            v = {(float)g(rng), (float)g(rng)};
            n0 += (double)v.x * v.x + (double)v.y * v.y;
        }
        line_op<float, N, 1, N, 1, false, TwShear>(f.data(), 1, tw.data(), tab.data(), 0, 1);
        for (auto &v : f) n1 += (double)v.x * v.x + (double)v.y * v.y;
    }
    std::printf("%s %.6e\n", label, (n1 - n0) / n0);
}

int main() {
    multiply("mul_1e-4", 1e-4, 0.0);
    multiply("mul_5e-4", 5e-4, 0.0);
    multiply("mul_1e-3", 1e-3, 0.0);
    multiply("mul_0.3", 0.3, 0.0);
    multiply("mul_2.8", 2.8, 0.0);
    multiply("mul_absorbing", 3e-4, 5.05e-6);
    line<64>("line_64", 5.2e-4);
    line<256>("line_256", 5.2e-4);
    line<2048>("line_2048", 5.2e-4);
    return 0;
}
