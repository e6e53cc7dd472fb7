// Beta policy head math for the rollout buffer of the shared-policy loop: the
// log-density of a draw, the entropy, and their derivatives with respect to the
// head's raw outputs (u, v), for shapes a = softplus(u) + f, b = softplus(v) + f
// with the policy's shape floor f (1 by default; below 1 the shapes may be
// below 1) (complete_port/patches/pufferlib_core.diff:944-1000,
// beta_continuous_head; :1008-1014 beta_kl).
//
//   log p(x)  = (a - 1) log x + (b - 1) log(1 - x) - ln B(a, b)
//   H         = ln B(a, b) - (a - 1) psi(a) - (b - 1) psi(b) + (a + b - 2) psi(a + b)
//   d log p / da = log x - psi(a) + psi(a + b)
//   d H / da     = -(a - 1) psi'(a) + (a + b - 2) psi'(a + b)
//   d a / du     = softplus'(u) = sigmoid(u)
//
// ln Gamma, psi and psi' together, from one shift to z >= 8 and the asymptotic
// series there (Abramowitz & Stegun 6.1.40, 6.3.18, 6.4.12, eight Bernoulli
// terms: truncation below 4e-16); shapes are positive.
//
//   KL(Beta(a1, b1) || Beta(a2, b2)) = ln B(a2, b2) - ln B(a1, b1) + (a1 - a2) psi(a1)
//                                      + (b1 - b2) psi(b1) + (a2 - a1 + b2 - b1) psi(a1 + b1)
// (the difference of the cross-entropy E_1[-log p_2] and the entropy of p_1,
// with E_1[log x] = psi(a1) - psi(a1 + b1) and E_1[log(1 - x)] = psi(b1) - psi(a1 + b1)).
#pragma once
#include <hip/hip_runtime.h>

namespace sbk {

// What ln Gamma, psi and psi' of x > 0 share. For x < 8, with z = x + 8 and
// P = x (x + 1) .. (x + 7): ln Gamma(x) = ln Gamma(z) - ln P, psi(x) = psi(z) -
// P'/P, psi'(x) = psi'(z) + (P'/P)^2 - P''/P; for x >= 8, z = x and P = 1. P is a
// polynomial of q = x (x + 7): q (q + 6) (q + 10) (q + 12). No loop and one
// division (for P and z), where a recurrence takes up to ten of each for psi and for
// psi' and ln Gamma a shift of its own: the PPO kernel (4,096 envs x 186 heads)
// 413 -> 64 us.
struct GammaAt {
    double z, iz, i2, P, ip, s1, s2, lz;
};

__device__ __forceinline__ GammaAt gamma_at(double x) {
    GammaAt g;
    const bool low = x < 8.0;
    const double t = 2.0 * x + 7.0, q = x * (x + 7.0);
    const double p1 = q * (q + 6.0), p2 = (q + 10.0) * (q + 12.0);
    const double d1 = 2.0 * q + 6.0, d2 = 2.0 * q + 22.0;
    const double dP = d1 * p2 + p1 * d2, ddP = 2.0 * (p2 + d1 * d2 + p1);
    g.P = low ? p1 * p2 : 1.0;
    g.z = low ? x + 8.0 : x;
    const double inv = 1.0 / (g.P * g.z);   // (P z is below 5e9, or z)
    g.ip = g.z * inv;
    g.iz = g.P * inv;
    g.s1 = low ? dP * t * g.ip : 0.0;
    g.s2 = low ? g.s1 * g.s1 - (ddP * t * t + 2.0 * dP) * g.ip : 0.0;
    g.i2 = g.iz * g.iz;
    g.lz = log(g.z);
    return g;
}

// ln Gamma(x) + ln P
__device__ __forceinline__ double gamma_ln(const GammaAt& g) {
    const double i2 = g.i2;
    const double s = g.iz * (1.0 / 12 - i2 * (1.0 / 360 - i2 * (1.0 / 1260 - i2 * (1.0 / 1680 - i2 * (1.0 / 1188
                     - i2 * (691.0 / 360360 - i2 * (1.0 / 156 - i2 * (3617.0 / 122400))))))));
    return (g.z - 0.5) * g.lz - g.z + 0.91893853320467274178 + s;   // ln(2 pi) / 2
}

__device__ __forceinline__ double gamma_psi(const GammaAt& g) {
    const double i2 = g.i2;
    const double s = i2 * (1.0 / 12 - i2 * (1.0 / 120 - i2 * (1.0 / 252 - i2 * (1.0 / 240 - i2 * (1.0 / 132
                     - i2 * (691.0 / 32760 - i2 * (1.0 / 12 - i2 * (3617.0 / 8160))))))));
    return g.lz - 0.5 * g.iz - s - g.s1;
}

__device__ __forceinline__ double gamma_psi1(const GammaAt& g) {
    const double i2 = g.i2;
    const double s = i2 * g.iz * (1.0 / 6 - i2 * (1.0 / 30 - i2 * (1.0 / 42 - i2 * (1.0 / 30 - i2 * (5.0 / 66
                     - i2 * (691.0 / 2730 - i2 * (7.0 / 6 - i2 * (3617.0 / 510))))))));
    return g.iz + 0.5 * i2 + s + g.s2;
}

// The sampler's shape map (float, as the draws use it) and its derivative.
__device__ __forceinline__ float beta_shape(float raw, float floor) {
    return (raw > 20.0f ? raw : log1pf(expf(raw))) + floor;
}
__device__ __forceinline__ double beta_shape_grad(float raw) {
    return raw > 20.0f ? 1.0 : 1.0 / (1.0 + exp(-(double)raw));
}

// Draws are floats in (0, 1); a ratio of gamma draws can round to 0 or 1, so
// the density is evaluated at x clamped to [2^-24, 1 - 2^-24].
__device__ __forceinline__ double beta_clamp_x(float x) {
    const double lo = 5.9604644775390625e-8;
    return x < lo ? lo : (x > 1.0 - lo ? 1.0 - lo : (double)x);
}

struct BetaHead {
    double logp, entropy;
    double g[4];   // d logp / du, d logp / dv, d H / du, d H / dv
};

// A head's shapes and what both its density and a divergence from or to it use.
struct BetaAt {
    double a, b, s;
    GammaAt ga, gb, gs;
    double lnb;
};

__device__ __forceinline__ BetaAt beta_at(float u, float v, float floor) {
    BetaAt t;
    t.a = beta_shape(u, floor);
    t.b = beta_shape(v, floor);
    t.s = t.a + t.b;
    t.ga = gamma_at(t.a);
    t.gb = gamma_at(t.b);
    t.gs = gamma_at(t.s);
    // (each P is 1 or below 2.6e8)
    t.lnb = gamma_ln(t.ga) + gamma_ln(t.gb) - gamma_ln(t.gs) - log(t.ga.P * t.gb.P * t.gs.ip);
    return t;
}

__device__ __forceinline__ BetaHead beta_head(const BetaAt& t, float u, float v, float x) {
    const double xc = beta_clamp_x(x);
    const double lx = log(xc), l1 = log(1.0 - xc);   // (1 - x is exact in double for a float x >= 2^-24)
    const double pa = gamma_psi(t.ga), pb = gamma_psi(t.gb), ps = gamma_psi(t.gs);
    BetaHead h;
    h.logp = (t.a - 1.0) * lx + (t.b - 1.0) * l1 - t.lnb;
    h.entropy = t.lnb - (t.a - 1.0) * pa - (t.b - 1.0) * pb + (t.s - 2.0) * ps;
    const double ta = gamma_psi1(t.ga), tb = gamma_psi1(t.gb), ts = gamma_psi1(t.gs);
    const double su = beta_shape_grad(u), sv = beta_shape_grad(v);
    h.g[0] = (lx - pa + ps) * su;
    h.g[1] = (l1 - pb + ps) * sv;
    h.g[2] = (-(t.a - 1.0) * ta + (t.s - 2.0) * ts) * su;
    h.g[3] = (-(t.b - 1.0) * tb + (t.s - 2.0) * ts) * sv;
    return h;
}

__device__ __forceinline__ BetaHead beta_head(float u, float v, float x, float floor) {
    return beta_head(beta_at(u, v, floor), u, v, x);
}

// The density and entropy by the two lanes of a pair: this lane's shape is a
// on the even lane (which 0), b on the odd one, `mate` the other's. Each takes
// the gamma functions of its own shape and of the sum; both lanes return the
// same values.
struct PairTerms {
    double logp, entropy;
};

__device__ __forceinline__ PairTerms beta_pair(float own, float mate, int which, float x) {
    const double c = (double)own, s = c + (double)mate, xc = beta_clamp_x(x);
    const GammaAt g = gamma_at(c), gs = gamma_at(s);
    const double l = (c - 1.0) * log(which ? 1.0 - xc : xc);
    const double ln = gamma_ln(g), e = (c - 1.0) * gamma_psi(g);
    const double P = g.P * __shfl_xor(g.P, 1);
    const double lnb = ln + __shfl_xor(ln, 1) - gamma_ln(gs) - log(P * gs.ip);
    PairTerms t;
    t.logp = l + __shfl_xor(l, 1) - lnb;
    t.entropy = lnb - (e + __shfl_xor(e, 1)) + (s - 2.0) * gamma_psi(gs);
    return t;
}

// KL(p || q)
__device__ __forceinline__ double beta_kl(const BetaAt& p, const BetaAt& q) {
    return q.lnb - p.lnb + (p.a - q.a) * gamma_psi(p.ga) + (p.b - q.b) * gamma_psi(p.gb)
           + (q.a - p.a + q.b - p.b) * gamma_psi(p.gs);
}

}  // namespace sbk
