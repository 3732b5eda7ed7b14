// Host check of the inner-loop functions of device_common.hpp (square root,
// exponential, quotient) against long double, and of the split e-e-n
// polynomial of een_poly.hpp against the direct term sum, orders 2 to 5.
// Exit status 1 if a deviation exceeds its bound.
#include "../../champ_amd/csrc/een_poly.hpp"

#include <cmath>
#include <cstdio>
#include <random>

using namespace champ;

static double ulps(double a, long double b) { return (double)(std::fabs((long double)a - b) / (std::fabs(b) * 0x1p-53L)); }

template <int N>
static double split(std::mt19937_64 &g)
{
    constexpr EenTable<N> ET{};
    constexpr EenSplit<N> ES{};
    constexpr int NP = een_nsep<N>();
    std::uniform_real_distribution<double> U(-1, 1), P(0.0, 1.0);
    double worst = 0;
    for (int trial = 0; trial < 2000; trial++) {
        double c[40], ref = 0, big = 1;
        for (double &v : c) v = U(g);
        const double u = P(g), x = P(g), y = P(g);
        for (int t = 0; t < ET.n; t++) {
            const double v = c[t] * std::pow(u, ET.k[t]) * (std::pow(x, ET.l[t]) + std::pow(y, ET.l[t])) * std::pow(x * y, ET.m[t]);
            ref += v;
            big += std::fabs(v);
        }
        double xp[N + 1], yp[N + 1], s[NP] = {0};
        een_powers<N>(x, xp);
        een_powers<N>(y, yp);
        een_uncoupled<N>(c, xp, s);
        een_uncoupled<N>(c, yp, s);
        double got = 0;
        for (int n = 1; n <= NP; n++) got += xp[n] * een_coupled<N>(c, yp, 0, n);
        for (int k = NP; k >= 1; k--) {
            double mk = s[k - 1];
            for (int n = 1; n <= N; n++)
                if (ES.idx[k][n] >= 0) mk += xp[n] * een_coupled<N>(c, yp, k, n);
            got += std::pow(u, k) * mk;
        }
        worst = std::max(worst, std::fabs(got - ref) / big);
    }
    return worst;
}

int main()
{
    std::mt19937_64 g(99);
    std::uniform_real_distribution<double> E(-40, 40), Z(-60, 0), V(-3, 3);
    double ws = 0, we = 0, wd = 0;
    for (int t = 0; t < 200000; t++) {
        const double x = std::exp2(E(g)), z = t % 2 ? Z(g) : -std::exp2(E(g) / 4), a = V(g), b = std::exp2(E(g) / 8);
        ws = std::max(ws, ulps(sqrt_inner(x), sqrtl((long double)x)));
        if (z > -700) we = std::max(we, ulps(exp_neg(z), expl((long double)z)));
        wd = std::max(wd, ulps(div_inner(a, b), (long double)a / b));
    }
    // one rounding each plus the last step's (square root, quotient); the
    // exponential adds the roundings of its reduced argument and polynomial
    int bad = !(ws <= 2.0) + !(wd <= 2.0) + !(we <= 4.0);
    const double inf = INFINITY;
    bad += sqrt_inner(0.0) != 0.0 || sqrt_inner(inf) != inf || exp_neg(0.0) != 1.0 || exp_neg(-inf) != 0.0 ||
           exp_neg(-1e300) != 0.0 || !std::isnan(exp_neg(NAN)) || !std::isnan(sqrt_inner(NAN));
    const double w[] = {split<2>(g), split<3>(g), split<4>(g), split<5>(g)};
    for (double v : w) bad += !(v < 1e-14);
    std::printf("ulp/2: sqrt %.2f exp %.2f div %.2f; split %.1e %.1e %.1e %.1e\n", ws, we, wd, w[0], w[1], w[2], w[3]);
    // the matrix part at orders 2..5: 0, 1, 3 and 6 entries
    bad += EenSplit<2>{}.nc != 0 || EenSplit<3>{}.nc != 1 || EenSplit<4>{}.nc != 3 || EenSplit<5>{}.nc != 6;
    return bad != 0;
}
