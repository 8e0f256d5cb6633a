// CPU check of the FP32 matrix-core line operator in its own order of
// operations: the bf16 residual product rounded once, the FP32 products of
// v_mfma_f32_16x16x4_f32 as a chain of fused operations over the lane groups
// (even points' real parts, their imaginary parts, then the odd points), then
// dense_c() x.  Prints <label> <value>: the relative L2 error of 100 slices
// against FP64 (drift_*), or the relative change of the power by rounding in
// one slice (gain_*).
#include <hip/hip_runtime.h>
#include <complex>
#include <cstdio>
#include <random>
#include <vector>
#include "../../cuopo3d_amd/csrc/opo_tables.hpp"
using namespace opo;
typedef std::complex<double> cd;

static float bits(unsigned u) {
    float x;
    std::memcpy(&x, &u, 4);
    return x;
}
static float top_half(float x) {
    unsigned u;
    std::memcpy(&u, &x, 4);
    return bits(u & 0xffff0000u);
}

template <int N> struct Line {
    static constexpr int N1 = N / 8;
    static constexpr float c = dense_c<float>(N1);
    std::vector<cplx<float>> hi, lo;
    // entries (1 + e(k)) / N
    template <typename E> explicit Line(E e) : hi(2 * N), lo(2 * N) {
        DenseRoots w;
        w.fill(N);
        dense_fill<float>(N, -1, w, e, [&](int i, float re, float im, unsigned l) {
            hi[i] = {re, im};
            lo[i] = {bits(l << 16), bits(l & 0xffff0000u)};
        }, c);
    }
    void apply(cplx<float> *x) const {
        cplx<float> v[8][N1];
        for (int n = 0; n < N; ++n) v[n % 8][n / 8] = x[n];
        for (int b = 0; b < 8; ++b) dft<N1, -1>(v[b]);
        for (int k1 = 0; k1 < N1; ++k1) {
            cplx<float> out[8];
            for (int a = 0; a < 8; ++a) {
                const cplx<float> *l = &lo[16 * k1 - a + 7], *h = &hi[16 * k1 - a + 7];
                double dr = 0, di = 0;
                for (int b = 0; b < 8; ++b) {
                    const double zx = top_half(v[b][k1].x), zy = top_half(v[b][k1].y);
                    dr += l[b].x * zx - l[b].y * zy;
                    di += l[b].x * zy + l[b].y * zx;
                }
                float re = (float)dr, im = (float)di;
                for (int p = 0; p < 2; ++p) {
                    for (int b = p; b < 8; b += 2) re = fmaf(h[b].x, v[b][k1].x, re), im = fmaf(h[b].y, v[b][k1].x, im);
                    for (int b = p; b < 8; b += 2) re = fmaf(-h[b].y, v[b][k1].y, re), im = fmaf(h[b].x, v[b][k1].y, im);
                }
                out[a] = {fmaf(v[a][k1].x, c, re), fmaf(v[a][k1].y, c, im)};
            }
            for (int b = 0; b < 8; ++b) v[b][k1] = out[b];
        }
        for (int b = 0; b < 8; ++b) idft<N1, -1>(v[b]);
        for (int n = 0; n < N; ++n) x[n] = v[n % 8][n / 8];
    }
};

// The factor of a slice: quadratic phase up to `phase`, absorption `la`.
template <int N> struct Slice {
    double phase, la;
    void operator()(int k, double &re, double &im) const {
        const double f = (k < N / 2 ? k : k - N) / (0.5 * N), r = -phase * f * f, h = std::sin(0.5 * r), a = std::expm1(-la);
        re = a - (1 + a) * 2 * h * h;
        im = (1 + a) * std::sin(r);
    }
};

template <int N> void drift(const char *label, double phase, bool beam) {
    constexpr int L = 16, K = 100;
    std::mt19937_64 rng(N);
    std::normal_distribution<double> g;
    const Slice<N> e{phase, 0.0};
    const Line<N> line(e);
    std::vector<cd> root(N);
    for (int k = 0; k < N; ++k) root[k] = std::polar(1.0, 2 * M_PI * k / N);
    double num = 0, den = 0;
    for (int l = 0; l < L; ++l) {
        std::vector<cplx<float>> y(N);
        std::vector<cd> X(N);
        for (int n = 0; n < N; ++n) {
            const double u = (n - 0.5 * N) / (N / 6.0);
            const cd v = beam ? std::polar(std::exp(-u * u) * (1 + 0.1 * l), 0.3 * u * u) : cd(g(rng), g(rng));
            y[n] = {(float)v.real(), (float)v.imag()};
        }
        for (int k = 0; k < N; ++k) {
            cd a = 0;
            for (int n = 0; n < N; ++n) a += cd(y[n].x, y[n].y) * std::conj(root[(long)n * k % N]);
            double re, im;
            e(k, re, im);
            X[k] = a * std::pow(cd(1 + re, im), K) / (double)N;
        }
        for (int s = 0; s < K; ++s) line.apply(y.data());
        for (int n = 0; n < N; ++n) {
            cd a = 0;
            for (int k = 0; k < N; ++k) a += X[k] * root[(long)n * k % N];
            num += std::norm(a - cd(y[n].x, y[n].y));
            den += std::norm(a);
        }
    }
    std::printf("%s %.6e\n", label, std::sqrt(num / den));
}

// Slices in sequence on noise, 6e7 values in all.
template <int N> void gain(const char *label, double phase, double la) {
    constexpr int K = 50, L = 60000000 / (K * N);
    std::mt19937_64 rng(N + 1);
    std::normal_distribution<double> g;
    const Line<N> line(Slice<N>{phase, la});
    double n0 = 0, n1 = 0;
    std::vector<cplx<float>> y(N);
    for (int l = 0; l < L; ++l) {
        for (auto &v : y) {
            v = {(float)g(rng), (float)g(rng)};
            n0 += (double)v.x * v.x + (double)v.y * v.y;
        }
        for (int s = 0; s < K; ++s) line.apply(y.data());
        for (auto &v : y) n1 += (double)v.x * v.x + (double)v.y * v.y;
    }
    std::printf("%s %.6e\n", label, (std::log(n1 / n0) + 2 * la * K) / K);
}

int main() {
    drift<32>("drift_beam_32", 0.12, true);
    drift<64>("drift_beam_64", 0.49, true);
    drift<96>("drift_beam_96", 1.1, true);
    drift<128>("drift_beam_128", 2.0, true);
    drift<96>("drift_noise_96", 1.1, false);
    drift<128>("drift_noise_128", 2.0, false);
    drift<256>("drift_noise_256", 7.8, false);
    gain<64>("gain_64", 0.49, 5.05e-6);
    gain<96>("gain_96", 1.1, 5.05e-6);
    gain<128>("gain_128", 2.0, 5.05e-6);
    return 0;
}
