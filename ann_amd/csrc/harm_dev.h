// harm_dev.h -- real spherical harmonics up to degree Z on unit vectors, in the
// normalisation of the addition theorem  P_l(u . v) = sum_m Y_lm(u) Y_lm(v).
//
// With x, y, z the unit vector's components, C_m + i S_m = (x + i y)^m and
// q_lm(z) = n_lm d^m P_l / dz^m, n_l0 = 1, n_lm^2 = 2 (l - m)! / (l + m)!,
// the functions are q_l0, q_lm C_m and q_lm S_m (m = 1 .. l): 2l + 1 of degree
// l, (Z + 1)^2 in all, numbered l^2 (m = 0), l^2 + 2m - 1 (C_m), l^2 + 2m (S_m),
// so a smaller degree bound is a prefix.  q follows the upward recurrence
// (l - m) Q_l = (2l - 1) z Q_(l-1) - (l + m - 1) Q_(l-2) of the associated
// Legendre functions, every coefficient a compile-time constant.
#pragma once
#include "common.h"

namespace ann {

__host__ __device__ constexpr int nharm(int Z) { return (Z + 1) * (Z + 1); }
__host__ __device__ constexpr int qidx(int l, int m) { return l * (l + 1) / 2 + m; }

constexpr double csqrt(double v) {
    double r = v > 1.0 ? v : 1.0;
    for (int k = 0; k < 60; ++k) r = 0.5 * (r + v / r);
    return r;
}

template <int Z>
struct HarmCoef {
    double a[qidx(Z, Z) + 1], b[qidx(Z, Z) + 1];   // q_lm = a z q_(l-1)m - b q_(l-2)m (l > m)
    double s[Z + 1];                               // q_mm
    double d[qidx(Z, Z) + 1];                      // dq_lm / dz = d q_l(m+1) (m < l)
    constexpr HarmCoef() : a(), b(), s(), d() {
        double n[qidx(Z, Z) + 1] = {};
        for (int l = 0; l <= Z; ++l)
            for (int m = 0; m <= l; ++m) {
                double w = m == 0 ? 1.0 : 2.0;
                for (int k = l - m + 1; k <= l + m; ++k) w /= k;
                n[qidx(l, m)] = csqrt(w);
            }
        for (int m = 0; m <= Z; ++m) {
            double f = 1.0;
            for (int k = 2 * m - 1; k > 1; k -= 2) f *= k;
            s[m] = f * n[qidx(m, m)];
        }
        for (int l = 1; l <= Z; ++l)
            for (int m = 0; m < l; ++m) {
                a[qidx(l, m)] = (2.0 * l - 1.0) / (l - m) * n[qidx(l, m)] / n[qidx(l - 1, m)];
                b[qidx(l, m)] = l - 2 >= m ? (l + m - 1.0) / (l - m) * n[qidx(l, m)] / n[qidx(l - 2, m)] : 0.0;
                d[qidx(l, m)] = n[qidx(l, m)] / n[qidx(l, m + 1)];
            }
    }
};

// C_m, S_m and q_lm of one unit vector
template <int Z, typename T>
__device__ __forceinline__ void harm_factors(T x, T y, T z, T (&C)[Z + 1], T (&S)[Z + 1], T (&q)[qidx(Z, Z) + 1]) {
    constexpr HarmCoef<Z> hc{};
    C[0] = T(1);
    S[0] = T(0);
#pragma unroll
    for (int m = 1; m <= Z; ++m) {
        C[m] = m == 1 ? x : x * C[m - 1] - y * S[m - 1];
        S[m] = m == 1 ? y : x * S[m - 1] + y * C[m - 1];
    }
#pragma unroll
    for (int m = 0; m <= Z; ++m) {
        q[qidx(m, m)] = T(hc.s[m]);
#pragma unroll
        for (int l = m + 1; l <= Z; ++l) {
            const T up = T(hc.a[qidx(l, m)]) * z;
            q[qidx(l, m)] = l - 2 >= m ? up * q[qidx(l - 1, m)] - T(hc.b[qidx(l, m)]) * q[qidx(l - 2, m)]
                                       : up * q[qidx(l - 1, m)];
        }
    }
}

// every function's value
template <int Z, typename T>
__device__ __forceinline__ void harm_values(const T (&C)[Z + 1], const T (&S)[Z + 1], const T (&q)[qidx(Z, Z) + 1],
                                            T (&Y)[nharm(Z)]) {
#pragma unroll
    for (int l = 0; l <= Z; ++l) {
        Y[l * l] = q[qidx(l, 0)];
#pragma unroll
        for (int m = 1; m <= l; ++m) {
            Y[l * l + 2 * m - 1] = q[qidx(l, m)] * C[m];
            Y[l * l + 2 * m] = q[qidx(l, m)] * S[m];
        }
    }
}

// every function's derivative along a direction d tangential to the sphere
template <int Z, typename T>
__device__ __forceinline__ void harm_along(const T (&C)[Z + 1], const T (&S)[Z + 1], const T (&q)[qidx(Z, Z) + 1],
                                           T dx, T dy, T dz, T (&D)[nharm(Z)]) {
    constexpr HarmCoef<Z> hc{};
#pragma unroll
    for (int m = 0; m <= Z; ++m) {
        T dC = T(0), dS = T(0);
        if (m > 0) {
            dC = T(m) * (dx * C[m - 1] - dy * S[m - 1]);
            dS = T(m) * (dx * S[m - 1] + dy * C[m - 1]);
        }
#pragma unroll
        for (int l = m; l <= Z; ++l) {
            const T dq = l > m ? T(hc.d[qidx(l, m)]) * q[qidx(l, m + 1 <= l ? m + 1 : m)] * dz : T(0);
            if (m == 0) {
                D[l * l] = dq;
            } else {
                D[l * l + 2 * m - 1] = q[qidx(l, m)] * dC + dq * C[m];
                D[l * l + 2 * m] = q[qidx(l, m)] * dS + dq * S[m];
            }
        }
    }
}

// Adjoint of one neighbour: the angular energy sum_u e_u(r) sum_f W_f[u] Y_f with
// e4 = e_u and f4 = de_u/dr.  Returns rad = sum_u f_u sum_f W_f[u] Y_f and the
// gradient g of sum_u e_u sum_f W_f[u] Y_f in the Cartesian components of the
// unit vector (its tangential part is what counts).  Per function: four products
// for V_f = sum_u e_u W_f[u], four for the sums per width, one each for the
// m-resolved sums of the gradient.
template <int Z>
__device__ __forceinline__ void harm_adjoint(float x, float y, float z, const float4 e4, const float4 f4,
                                             const float4* __restrict__ W, float& rad, float& g0, float& g1, float& g2) {
    constexpr HarmCoef<Z> hc{};
    float C[Z + 1], S[Z + 1], q[qidx(Z, Z) + 1];
    harm_factors<Z, float>(x, y, z, C, S, q);
    float p0 = 0.0f, p1 = 0.0f, p2 = 0.0f, p3 = 0.0f;
    g0 = g1 = g2 = 0.0f;
#pragma unroll
    for (int m = 0; m <= Z; ++m) {
        float A = 0.0f, B = 0.0f, zA = 0.0f, zB = 0.0f;      // sums over l with q and with dq/dz
#pragma unroll
        for (int l = m; l <= Z; ++l) {
            const float ql = q[qidx(l, m)], dq = l > m ? (float)hc.d[qidx(l, m)] * q[qidx(l, m + 1 <= l ? m + 1 : m)] : 0.0f;
            {
                const float4 w = W[m == 0 ? l * l : l * l + 2 * m - 1];
                const float V = e4.x * w.x + e4.y * w.y + e4.z * w.z + e4.w * w.w;
                const float Y = m == 0 ? ql : ql * C[m];
                p0 += Y * w.x; p1 += Y * w.y; p2 += Y * w.z; p3 += Y * w.w;
                A += ql * V;
                if (l > m) zA += dq * V;
            }
            if (m > 0) {
                const float4 w = W[l * l + 2 * m];
                const float V = e4.x * w.x + e4.y * w.y + e4.z * w.z + e4.w * w.w;
                const float Y = ql * S[m];
                p0 += Y * w.x; p1 += Y * w.y; p2 += Y * w.z; p3 += Y * w.w;
                B += ql * V;
                if (l > m) zB += dq * V;
            }
        }
        if (m == 0) {
            g2 += zA;
        } else {
            const float mA = (float)m * A, mB = (float)m * B;
            g0 += mA * C[m - 1] + mB * S[m - 1];
            g1 += mB * C[m - 1] - mA * S[m - 1];
            g2 += zA * C[m] + zB * S[m];
        }
    }
    rad = f4.x * p0 + f4.y * p1 + f4.z * p2 + f4.w * p3;
}

// Coefficients of c^m in Legendre polynomials: c^m = sum_l k(m, l) P_l(c),
// l = m, m - 2, ...; k(m, l) = (2l + 1) m! / (2^((m - l) / 2) ((m - l) / 2)! (l + m + 1)!!)
__host__ __device__ constexpr double legendre_of_power(int m, int l) {
    if (l > m || (m - l) % 2) return 0.0;
    double k = 2.0 * l + 1.0;
    for (int t = 2; t <= m; ++t) k *= t;
    for (int t = 1; t <= (m - l) / 2; ++t) k /= 2.0 * t;
    for (int t = l + m + 1; t > 1; t -= 2) k /= t;
    return k;
}

}  // namespace ann
