// Host program: RMS error (relative to the RMS of the result) of the row transforms of
// hy_fft.hpp in binary64 against a long-double DFT of the same rows.  Prints
// "LEN forward inverse x-inverse" per length: level A then B with table twiddles,
// the inverse of the y and z passes (split twiddles), and that of the x
// passes (B then A).
#include <cmath>
#include <cstdio>
#include <random>
#include <vector>

#include "hy_fft.hpp"

using C = double2;

template <int LEN, int A, int B, int S, bool SPLIT>
std::vector<C> row(const std::vector<C>& x, const C* tw) {
    std::vector<C> y(LEN), out(LEN);
    for (int t = 0; t < B; ++t) {
        C v[32], w[32], lo[32], hi[32];
        for (int n = 0; n < A; ++n) v[n] = x[t + B * n];
        hy::dft_reg<A, S>(v);
        if (SPLIT) {
            hy::tl_twiddle_load_split<A, LEN>(lo, hi, t, tw, 1);
            hy::tl_twiddle_apply_split<A, S>(v, lo, hi);
        } else {
            hy::tl_twiddle_load<A, LEN>(w, t, tw, 1);
            hy::tl_twiddle_apply<A, S>(v, w);
        }
        for (int k = 0; k < A; ++k) y[k * B + t] = v[k];
    }
    for (int t = 0; t < A; ++t) {
        C v[32];
        for (int n = 0; n < B; ++n) v[n] = y[t * B + n];
        hy::dft_reg<B, S>(v);
        for (int k = 0; k < B; ++k) out[t + A * k] = v[k];
    }
    return out;
}

template <int LEN>
void measure() {
    const long double two_pi = 2.0L * 3.141592653589793238462643383279502884L;
    std::vector<long double> c(LEN), s(LEN);
    std::vector<C> tw(LEN);
    for (int m = 0; m < LEN; ++m) {
        c[m] = std::cos(two_pi * m / LEN);
        s[m] = std::sin(two_pi * m / LEN);
        tw[m] = {(double)c[m], -(double)s[m]};
    }
    constexpr int A = hy::TwoLevel<LEN>::A, B = hy::TwoLevel<LEN>::B;
    std::mt19937_64 rng(LEN);
    std::normal_distribution<double> normal;
    long double err[3] = {0, 0, 0}, norm = 0;
    for (int rep = 0; rep < 20000 / LEN + 8; ++rep) {
        std::vector<C> x(LEN);
        for (C& v : x) v = {normal(rng), normal(rng)};
        const std::vector<C> got[3] = {row<LEN, A, B, -1, false>(x, tw.data()), row<LEN, A, B, 1, true>(x, tw.data()),
                                       row<LEN, B, A, 1, true>(x, tw.data())};
        for (int k = 0; k < LEN; ++k) {
            long double re[2] = {0, 0}, im[2] = {0, 0};  // forward, inverse
            for (int n = 0; n < LEN; ++n) {
                const int m = (int)((long)k * n % LEN);
                const long double xc = x[n].x * c[m], xs = x[n].x * s[m], yc = x[n].y * c[m], ys = x[n].y * s[m];
                re[0] += xc + ys;
                im[0] += yc - xs;
                re[1] += xc - ys;
                im[1] += yc + xs;
            }
            norm += re[0] * re[0] + im[0] * im[0];
            for (int i = 0; i < 3; ++i) {
                const long double dx = got[i][k].x - re[i > 0], dy = got[i][k].y - im[i > 0];
                err[i] += dx * dx + dy * dy;
            }
        }
    }
    std::printf("%d %.4Le %.4Le %.4Le\n", LEN, std::sqrt(err[0] / norm), std::sqrt(err[1] / norm),
                std::sqrt(err[2] / norm));
}

int main() {
    measure<6>(); measure<12>(); measure<24>(); measure<48>(); measure<96>(); measure<192>(); measure<384>();
    measure<8>(); measure<16>(); measure<32>(); measure<64>(); measure<128>(); measure<256>(); measure<512>();
    measure<1024>();
}
