// Real spherical harmonics and Legendre coefficients of the moment form
// (ann_amd/csrc/harm_dev.h) on the host, in FP64 except for the FP32 adjoint:
//   sum_m Y_lm(u) Y_lm(v) = P_l(u . v),   c^m = sum_l k(m, l) P_l(c),
//   the derivative along a tangential direction and the adjoint's gradient
//   against central differences, and the moment form of a triplet sum against
//   the sum itself: sum_{j<k} (1/2 + lambda c_jk / 2)^zeta e_j e_k
//   = sum_l a_l (sum_m T_lm^2 - sum_j e_j^2) / 2.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>

#include "harm_dev.h"

using namespace ann;

static std::mt19937 rng(7);

static void require(bool ok, const char* what, int z, double err) {
    if (ok) return;
    std::printf("%s, degree bound %d: error %.3e\n", what, z, err);
    std::exit(1);
}

static void unit(double (&x)[3]) {
    std::normal_distribution<double> g;
    for (double& c : x) c = g(rng);
    const double r = std::sqrt(x[0] * x[0] + x[1] * x[1] + x[2] * x[2]);
    for (double& c : x) c /= r;
}

static double legendre(int l, double c) {
    double p0 = 1.0, p1 = c;
    if (l == 0) return 1.0;
    for (int k = 2; k <= l; ++k) {
        const double p2 = ((2.0 * k - 1.0) * c * p1 - (k - 1.0) * p0) / k;
        p0 = p1;
        p1 = p2;
    }
    return p1;
}

template <int Z>
static void values(const double (&x)[3], double (&Y)[nharm(Z)]) {
    double C[Z + 1], S[Z + 1], q[qidx(Z, Z) + 1];
    harm_factors<Z, double>(x[0], x[1], x[2], C, S, q);
    harm_values<Z, double>(C, S, q, Y);
}

template <int Z>
static void check() {
    std::uniform_real_distribution<double> uni(-1.0, 1.0);
    for (int trial = 0; trial < 200; ++trial) {
        double u[3], v[3], a[nharm(Z)], b[nharm(Z)];
        unit(u);
        unit(v);
        if (trial < 6) {                                // the poles and the axes
            for (double& c : u) c = 0.0;
            u[trial / 2] = trial % 2 ? -1.0 : 1.0;
        }
        values<Z>(u, a);
        values<Z>(v, b);
        const double c = u[0] * v[0] + u[1] * v[1] + u[2] * v[2];
        for (int l = 0; l <= Z; ++l) {
            double s = 0.0, n = 0.0;
            for (int f = l * l; f < (l + 1) * (l + 1); ++f) {
                s += a[f] * b[f];
                n += a[f] * a[f];
            }
            require(std::fabs(s - legendre(l, c)) < 1e-13, "addition theorem", Z, s - legendre(l, c));
            require(std::fabs(n - 1.0) < 1e-13, "normalisation", Z, n - 1.0);
        }
        // tangential derivative against central differences of the normalised vector
        double t[3], up[3], um[3], C[Z + 1], S[Z + 1], q[qidx(Z, Z) + 1], D[nharm(Z)], yp[nharm(Z)], ym[nharm(Z)];
        unit(t);
        const double tu = t[0] * u[0] + t[1] * u[1] + t[2] * u[2], h = 1e-5;
        double rp = 0.0, rm = 0.0;
        for (int k = 0; k < 3; ++k) {
            t[k] -= tu * u[k];
            up[k] = u[k] + h * t[k];
            um[k] = u[k] - h * t[k];
            rp += up[k] * up[k];
            rm += um[k] * um[k];
        }
        for (int k = 0; k < 3; ++k) {
            up[k] /= std::sqrt(rp);
            um[k] /= std::sqrt(rm);
        }
        harm_factors<Z, double>(u[0], u[1], u[2], C, S, q);
        harm_along<Z, double>(C, S, q, t[0], t[1], t[2], D);
        values<Z>(up, yp);
        values<Z>(um, ym);
        for (int f = 0; f < nharm(Z); ++f) {
            const double d = (yp[f] - ym[f]) / (2.0 * h);
            require(std::fabs(D[f] - d) < 1e-8, "tangential derivative", Z, D[f] - d);
        }
        // the adjoint: radial sum, and its gradient along t
        float4 W[nharm(Z)];
        for (float4& w : W) w = make_float4((float)uni(rng), (float)uni(rng), (float)uni(rng), (float)uni(rng));
        const float4 e = make_float4(0.9f, 0.5f, 0.3f, 0.1f), d = make_float4(-0.2f, 0.4f, 0.7f, -0.6f);
        float rad, g0, g1, g2;
        harm_adjoint<Z>((float)u[0], (float)u[1], (float)u[2], e, d, W, rad, g0, g1, g2);
        double wr = 0.0, wt = 0.0;
        for (int f = 0; f < nharm(Z); ++f) {
            wr += a[f] * (d.x * W[f].x + d.y * W[f].y + d.z * W[f].z + d.w * W[f].w);
            wt += D[f] * (e.x * W[f].x + e.y * W[f].y + e.z * W[f].z + e.w * W[f].w);
        }
        // at most 36 terms of size below 2 (values) and 2 l (derivatives), FP32
        require(std::fabs(rad - wr) < 1e-5, "radial sum of the adjoint", Z, rad - wr);
        require(std::fabs(g0 * t[0] + g1 * t[1] + g2 * t[2] - wt) < 5e-5, "gradient of the adjoint", Z,
                g0 * t[0] + g1 * t[1] + g2 * t[2] - wt);
        for (int m = 0; m <= Z; ++m) {
            double s = 0.0;
            for (int l = 0; l <= m; ++l) s += legendre_of_power(m, l) * legendre(l, c);
            require(std::fabs(s - std::pow(c, m)) < 1e-13, "powers in Legendre polynomials", Z, s - std::pow(c, m));
        }
    }
    // a triplet sum and its moment form
    constexpr int n = 40;
    static double x[n][3], ev[n], Y[n][nharm(Z)];
    double T[nharm(Z)] = {}, D2 = 0.0;
    for (int j = 0; j < n; ++j) {
        unit(x[j]);
        values<Z>(x[j], Y[j]);
        ev[j] = 0.5 + 0.5 * uni(rng);
        D2 += ev[j] * ev[j];
        for (int f = 0; f < nharm(Z); ++f) T[f] += ev[j] * Y[j][f];
    }
    for (int zeta = 1; zeta <= Z; ++zeta)
        for (int lam = -1; lam <= 1; ++lam) {
            double ref = 0.0, sum = 0.0;
            for (int j = 0; j < n; ++j)
                for (int k = j + 1; k < n; ++k) {
                    const double c = x[j][0] * x[k][0] + x[j][1] * x[k][1] + x[j][2] * x[k][2];
                    ref += std::pow(0.5 + 0.5 * lam * c, zeta) * ev[j] * ev[k];
                }
            for (int l = 0; l <= zeta; ++l) {
                double A = 0.0, al = 0.0;
                for (int f = l * l; f < (l + 1) * (l + 1); ++f) A += T[f] * T[f];
                for (int m = l; m <= zeta; m += 2) {
                    double k = std::pow(2.0, m - zeta) * std::pow(0.5 * lam, m);
                    for (int q = 0; q < m; ++q) k = k * (zeta - q) / (q + 1);
                    al += k * legendre_of_power(m, l);
                }
                sum += al * 0.5 * (A - D2);
            }
            require(std::fabs(sum - ref) < 1e-12 * n * n, "moment form", Z, sum - ref);
        }
}

int main() {
    check<1>();
    check<2>();
    check<3>();
    check<4>();
    check<5>();
    std::puts("ok");
    return 0;
}
