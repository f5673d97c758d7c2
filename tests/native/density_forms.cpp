// Host evaluation of what the FP64 density pairs are made of (common.hpp), for the CPU tests: the
// sums of their brackets (kernVG) and of the reference's pieces (kernWdW), each against the sums in 128
// bits, and the root from an estimate (rootStep) against the correctly rounded one.  Prints
//   sums <pairs> <rms error of sum W: pieces, kernVG> <rms error of sum -q dW/dq - 3W: pieces, kernVG>
//   root <samples> <samples that are not the nearest double>
#include "../../cosmosphere_amd/csrc/common.hpp"

#include <cmath>
#include <cstdio>
#include <random>

using csph::kGe;
using csph::kGp;
using csph::kGw;
using csph::kWw;
typedef __float128 quad;

static quad up(quad c, quad q) { return q < c ? c - q : quad(0); }

// W and -q dW/dq - 3W at q^2 = x (the root by one Newton step from the double's)
static void exact(double x, quad& w, quad& g)
{
    quad q = std::sqrt(x);
    if (x > 0.0) q = (q + quad(x) / q) / 2;
#ifdef COSMO_KERNEL_QUINTIC
    const quad a = up(3, q), b = up(2, q), c = up(1, q);
    w = a * a * a * a * a - 6 * b * b * b * b * b + 15 * c * c * c * c * c;
    g = 5 * q * (a * a * a * a - 6 * b * b * b * b + 15 * c * c * c * c) - 3 * w;
#else
    const quad a = up(2, q), b = up(1, q);
    w = (a * a * a - 4 * b * b * b) / 4;
    g = 3 * q * (a * a - 4 * b * b) / 4 - 3 * w;
#endif
}

int main()
{
    std::mt19937_64 gen(7);
    std::uniform_real_distribution<double> uni(0.0, 1.0);
    const int sets = 20000, lanes = 3;   // a particle's pairs on three lanes, then their sum
    for (int n : {58, 113, 500})
    {
        double ew[2] = {0, 0}, eg[2] = {0, 0};
        for (int k = 0; k < sets; ++k)
        {
            double sw[2][lanes] = {}, sg[2][lanes] = {};
            quad W = 0, G = 0;
            for (int j = 0; j < n; ++j)
            {
                const double x = j ? csph::kRad2 * std::pow(uni(gen), 2.0 / 3.0) : 0.0;   // a ball; the self pair
                quad w, g;
                exact(x, w, g);
                W += w;
                G += g;
                const double q = std::sqrt(x);
                double a, d, V, H;
                csph::kernWdW<double>(x, q, a, d);
                sw[0][j % lanes] += a;
                sg[0][j % lanes] += -q * d - 3.0 * a;
                const double x1 = x + 0x1p-900;
                double e;
                const double r = csph::rootStep(x1, (1.0 / std::sqrt(x1)) * (1.0 + (uni(gen) - 0.5) * 0x1p-23), e);
                csph::kernVG<double>(r, x1, V, H);
                sw[1][j % lanes] += V;
                sg[1][j % lanes] += H;
            }
            for (int f = 0; f < 2; ++f)
            {
                const double w = (sw[f][0] + sw[f][1]) + sw[f][2], g = (sg[f][0] + sg[f][1]) + sg[f][2];
                const quad dw = quad(f ? kWw * csph::kVs * w : w) - W, dg = quad(f ? (kGp + kGw) * csph::kVs * g : g) - G;
                ew[f] += (double)(dw * dw / (W * W));
                eg[f] += (double)(dg * dg / (W * W));
            }
        }
        std::printf("sums %d %.6e %.6e %.6e %.6e\n", n, std::sqrt(ew[0] / sets), std::sqrt(ew[1] / sets),
                    std::sqrt(eg[0] / sets), std::sqrt(eg[1] / sets));
    }
    long wrong = 0;
    const long samples = 2000000;
    for (long k = 0; k < samples; ++k)
    {
        const double x = std::ldexp(1.0 + uni(gen), (int)(-200 * uni(gen)) + 3);
        double e;
        if (csph::rootStep(x, (1.0 / std::sqrt(x)) * (1.0 + (uni(gen) - 0.5) * 0x1p-22), e) != std::sqrt(x)) ++wrong;
    }
    std::printf("root %ld %ld\n", samples, wrong);
    return 0;
}
