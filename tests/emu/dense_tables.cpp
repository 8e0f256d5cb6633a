// CPU check of the FP64 dense tables (dense_fill<double>): the operator that a
// table stands for, applied in long double, against the exact operator with
// the same phases.  Prints <label> <relative rms error>.
#include <hip/hip_runtime.h>
#include <complex>
#include <cstdio>
#include <random>
#include <vector>
#include "../../cuopo3d_amd/csrc/opo_tables.hpp"
using namespace opo;
typedef long double LD;
typedef std::complex<LD> cl;

// Quadratic phases up to `phase`, absorption la.
template <int N> void table(const char *label, double phase, double la) {
    constexpr int N1 = N / 8;
    const LD pi = acosl(-1.0L);
    std::vector<double> ph(N);
    for (int k = 0; k < N; ++k) {
        const double f = (k < N / 2 ? k : k - N) / (0.5 * N);
        ph[k] = -phase * f * f;
    }
    DenseRootsOf<dense_acc<double>> w;
    w.fill(N);
    std::vector<cl> M(2 * N), r(N), x(N), v(N), o(N), want(N);
    dense_fill<double>(N, -1, w, [&](int k, dense_acc<double> &re, dense_acc<double> &im) {
        dense_increment<dense_acc<double>>(ph[k], std::expm1((dense_acc<double>)-la), re, im);
    }, [&](int i, double re, double im, unsigned) { M[i] = cl(re, im); }, dense_c<double>(N1), true);
    for (int k1 = 0; k1 < N1; ++k1) M[16 * k1 + 7] += (LD)dense_c<double>(N1);
    for (int j = 0; j < N; ++j) r[j] = std::polar((LD)1, 2 * pi * j / N);
    std::mt19937_64 rng(N);
    std::normal_distribution<double> g;
    for (auto &a : x) a = cl(g(rng), g(rng));
    for (int k = 0; k < N; ++k) {
        cl a = 0;
        for (int n = 0; n < N; ++n) a += x[n] * std::conj(r[n * k % N]);
        a *= std::polar(expl(-(LD)la) / N, (LD)ph[k]);
        for (int n = 0; n < N; ++n) want[n] += a * r[n * k % N];
    }
    for (int b = 0; b < 8; ++b)
        for (int k1 = 0; k1 < N1; ++k1) {
            cl a = 0;
            for (int n1 = 0; n1 < N1; ++n1) a += x[8 * n1 + b] * std::conj(r[8 * n1 * k1 % N]);
            v[b * N1 + k1] = a;
        }
    for (int a = 0; a < 8; ++a)
        for (int k1 = 0; k1 < N1; ++k1) {
            cl s = 0;
            for (int b = 0; b < 8; ++b) s += M[16 * k1 + b - a + 7] * v[b * N1 + k1];
            o[a * N1 + k1] = s;
        }
    LD e = 0, d = 0;
    for (int a = 0; a < 8; ++a)
        for (int n1 = 0; n1 < N1; ++n1) {
            cl s = 0;
            for (int k1 = 0; k1 < N1; ++k1) s += o[a * N1 + k1] * r[8 * n1 * k1 % N];
            e += std::norm(s - want[8 * n1 + a]);
            d += std::norm(want[8 * n1 + a]);
        }
    std::printf("%s %.6e\n", label, (double)std::sqrt(e / d));
}

int main() {
    table<16>("slice_16", 0.03, 5e-6);
    table<32>("slice_32", 0.12, 5e-6);
    table<64>("slice_64", 0.49, 5e-6);
    table<96>("slice_96", 1.1, 5e-6);
    table<128>("slice_128", 2.0, 5e-6);
    table<96>("absorbing_96", 1.1, 0.3);
    table<64>("space_64", 48.0, 0.0);
    table<128>("space_128", 196.0, 0.0);
    return 0;
}
