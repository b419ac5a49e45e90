// wall_pairs.hpp -- the no-slip wall image system of StkWallFMM (Lib/src/StkWallFMM.cpp:154-292) as one
// pair formula: a source and its image against one target, the whole system in one evaluation.
//
// The reference sums a Stokeslet or RPY kernel, Laplace charges, dipoles and (RPY) quadrupoles at the
// source and at its image (x, y, -z) and combines their potentials, gradients and Hessians with the
// target's height at the end: 7 sums for Stokes, 10 for RPY, each with its own displacement, reciprocal
// square root and outputs that the assembly does not use.  Collected by powers of 1/r per pair (units of
// 1/(8 pi)), with r = (dx, dy, d1 = x3 - z), s = 1/|r| to the source, R = (dx, dy, d2 = x3 + z),
// S = 1/|R| to the image, x3 the target's and z the source's height, g = f1 dx + f2 dy:
//   * the parts at the source are exactly the free-space kernel of the whole force (the charges' terms
//     meet in the factor x3 - z = d1);
//   * the parts at the image depend on h = f3 d2 - g, the image force (-f1, -f2, f3) along R.
// The terms that cancel near the wall cancel inside a pair here and not between sums of all pairs.
// Both distances keep the coincidence mask of the constituent kernels (s or S = 0 at distance 0).
//
// Each struct has the micro-kernels' members (ukernels.hpp) except that eval_wall takes the heights.
#pragma once

#include "ukernels.hpp"

namespace stkp2p {

// f(3) -> u(3).  With m = 2 x3 z:
//   u_x = f1 (s - S - m S^3) + dx c,   u_y likewise,   c = c1 - c2
//   u_z = f3 (s - S + m S^3) + d1 c1 - d2 c2 - 2 z h S^3
//   c1 = (g + f3 d1) s^3,   c2 = (g + f3 d1) S^3 + 3 m h S^5
// evaluated as 2 u from w = 2 s, W = 2 S (twice_rsqrt, one operation fewer each): 1/4 of f in g and h and
// 1/4 of m make every power's factor 1; staged f, f/4, z/2, 2 z.  42 FP64 operations and two reciprocal
// square roots and masks per pair, for about 180 of the seven sums.
struct UkWallStokes {
    static constexpr int KS = 3, KS1 = 3, KL = 7, KT = 3;
    static constexpr bool WALL = true;
    __host__ __device__ static constexpr double post(int) { return 0.5; }
    __host__ __device__ static void stage(const double *in, double *o) {
        for (int i = 0; i < 3; ++i) {
            o[i] = in[i];
            o[3 + i] = 0.25 * in[i];
        }
    }
    // the source's height joins its staged values
    __host__ __device__ static void stage_height(double z, double *o) { o[6] = 0.5 * z; }
    template <class R>
    __device__ static void eval_wall(R *u, R dx, R dy, R d1, R d2, R x3, const R *f) {
        const R rho2 = dx * dx + dy * dy;
        const R w = twice_rsqrt<true>(d1 * d1 + rho2);
        const R W = twice_rsqrt<true>(d2 * d2 + rho2);
        const R g = f[3] * dx + f[4] * dy;
        const R a = f[5] * d1 + g;
        const R h = f[5] * d2 - g;
        const R w3 = (w * w) * w;
        const R W2 = W * W;
        const R W3 = W2 * W;
        const R e = (f[6] * x3) * W3;
        const R t = w - W;
        const R c1 = a * w3;
        const R c2 = a * W3 + (R(3.0) * e) * (h * W2);
        const R c = c1 - c2;
        const R A = t - e;
        u[0] += f[0] * A;
        u[0] += dx * c;
        u[1] += f[1] * A;
        u[1] += dy * c;
        u[2] += f[2] * (t + e);
        u[2] += d1 * c1;
        u[2] -= d2 * c2;
        u[2] -= (R(4.0) * f[6] * h) * W3;
    }
};

// [f(3), b] -> [u(3), lap u(3)].  With B = b^2/3, m = 2 x3 z, P = S^3, q = d2 S^2, H = h S^2:
//   at the source UkRpyULapU of (f1, f2, f3, b); at the image
//   u_x = f1 F + dx C,  F = y d2 - S - (B + m) P,  y = 6 x3 B S^5,
//     C = P (t - 3 (B + m) H) - y (f3 - 5 d2 H),  t = h - 2 x3 f3
//   u_z = -f3 (S + (B - m) P) + d2 C - y k + P (6 B d2 H - 2 z h),  k = f3 d2 + h
//   lap u_x = 6 (f1 F' + dx S^5 G),  F' = -P/3 + 2 S^5 (z d2 + B - 5 B d2 q),
//     G = -t + 10 (H (z d2 + B - 7 B d2 q) + 2 B q f3)
//   lap u_z = 6 (-f3 P/3 + d2 S^5 G + S^5 (10 (2 B d2 H + f3 B d2 q) - 2 z k - 6 B f3))
// post() applies the 6 of the Laplacian.
struct UkWallRpy {
    static constexpr int KS = 4, KS1 = 4, KL = 5, KT = 6;
    static constexpr bool WALL = true;
    __host__ __device__ static constexpr double post(int k) { return k < 3 ? 1.0 : 6.0; }
    __host__ __device__ static void stage(const double *in, double *o) {
        o[0] = in[0]; o[1] = in[1]; o[2] = in[2];
        // b^2/3 (the reference has 1/6 b^2 in the dipoles and quadrupoles, which remain of a source on the
        // wall, and 0.3333333333333 b^2 in the RPY kernels, which cancel there)
        o[3] = (in[3] * in[3]) / 3.0;
    }
    __host__ __device__ static void stage_height(double z, double *o) { o[4] = z; }
    template <class R>
    __device__ static void eval_wall(R *u, R dx, R dy, R d1, R d2, R x3, const R *f) {
        const R B = f[3], z = f[4];
        const R rho2 = dx * dx + dy * dy;
        const R s = rsqrt_masked(d1 * d1 + rho2);
        const R S = rsqrt_masked(d2 * d2 + rho2);
        const R g = f[0] * dx + f[1] * dy;
        const R h = f[2] * d2 - g;
        const R s2 = s * s;
        const R s3 = s2 * s;
        const R g3 = (f[2] * d1 + g) * s3;
        const R g5 = g3 * s2;
        const R b1 = g3 - (R(3.0) * B) * g5;
        const R S2 = S * S;
        const R P = S2 * S;
        const R S5 = P * S2;
        const R H = h * S2;
        const R q = d2 * S2;
        const R m = (R(2.0) * x3) * z;
        const R t = h - (R(2.0) * x3) * f[2];
        const R y = (R(6.0) * x3) * (B * S5);
        const R Bm = B + m;
        const R dH = d2 * H;
        const R C = P * (t - R(3.0) * (Bm * H)) - y * (f[2] - R(5.0) * dH);
        // s + B s^3 and S + B S^3 as two differences: they cancel to a multiple of z near the wall
        const R v = s3 - P;
        const R D = B * v + (s - S);
        const R mP = m * P;
        const R F = D + (y * d2 - mP);
        const R cu = b1 + C;
        const R k = f[2] * d2 + h;
        const R bq = (B * d2) * q;
        const R zB = z * d2 + B;
        const R z2 = R(2.0) * z;
        u[0] += f[0] * F;
        u[0] += dx * cu;
        u[1] += f[1] * F;
        u[1] += dy * cu;
        u[2] += f[2] * (D + mP);
        u[2] += d1 * b1;
        u[2] += d2 * C;
        u[2] -= y * k;
        u[2] += P * ((R(6.0) * B) * dH - z2 * h);
        const R v3 = R(1.0 / 3.0) * v;
        const R F3 = v3 + (R(2.0) * S5) * (zB - R(5.0) * bq);
        const R E = S5 * (R(10.0) * (H * (zB - R(7.0) * bq) + (R(2.0) * B) * (q * f[2])) - t);
        const R cl = E - g5;
        u[3] += f[0] * F3;
        u[3] += dx * cl;
        u[4] += f[1] * F3;
        u[4] += dy * cl;
        u[5] += f[2] * v3;
        u[5] += d2 * E;
        u[5] -= d1 * g5;
        u[5] += S5 * ((R(20.0) * B) * dH + f[2] * (R(10.0) * bq - R(6.0) * B) - z2 * k);
    }
};

template <> struct UkerOf<25> { using type = UkWallStokes; };
template <> struct UkerOf<26> { using type = UkWallRpy; };

} // namespace stkp2p
