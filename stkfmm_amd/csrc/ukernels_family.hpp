// ukernels_family.hpp -- the rest of the STKFMM kernel family, for gfx950: Stokes PVelGrad,
// PVelLaplacian and Traction (single and double layer), the regularised force/torque kernels of
// StokesRegVelOmega, and the Laplace quadrupole kernels of LapQPGradGrad.
//
// Same contract as ukernels.hpp (KS, KS1, KL, KT, SRC_SCALE_MASK, deg, post, stage, eval).
//
// These kernels carry powers of 1/r up to r^-9 (r^-7 for the double layers) in the reference's
// algebra.  Formed literally, rinv^9 overflows FP32 for a close pair (r < ~1e-4 in the work item's
// level-scaled frame), so the FP32 form of every kernel here is the unit-direction form: with
// s = 1/|r| (masked) and n = r s, a term  poly_k(r) * rinv^(k+m)  with poly_k homogeneous of degree
// k equals  poly_k(n) * s^m, and each output becomes a polynomial in n (entries bounded by the
// source strengths) times one power of s -- the power the output's own magnitude needs.
// Coincident pairs: s = 0 gives n = 0 and every output carries at least one factor of s, so they
// contribute exactly 0, as the reference's masked approx_rsqrt does.
//
// FP64 takes powers of w = 2/r (twice_rsqrt) up to w^7, which every output stands for separations of 9e-44 to 4e43
// (LapQPGradGrad; the others, up to w^5, from 1e-61 to 1e61): farther than the reference's own powers reach in each
// kernel (1e-34 to 1e34 with r^-9, 1e-43 to 1e44 with r^-7, 1e-61 to 1e62 with r^-5), though not as far as the
// unit-direction form (1e-61, 1e-76 or 1e-102).  It saves the three products of n,
// and accumulates in a basis of its own (ACC64, ukernels.hpp): a symmetric tensor as six sums, an
// antisymmetric part as three, the multiple of the unit matrix once, constant factors at the end.  The
// kernels are bound by FP64 issue, so a pair's time follows its operations; 262,144-point U-list, 1.06e9
// pairs, item kernel + reduce (ms), unit-direction form with every output apart -> this form (which also
// drops the coincidence mask on clear tiles): PVelGrad 2.96 -> 2.20, DoublePVelGrad 2.48 -> 2.23,
// PVelLaplacian 1.57 -> 1.34, DoubleLaplacian 1.74 -> 1.56, Traction 1.51 -> 1.15, DoubleTraction 2.36 ->
// 1.76, RegFTVelOmega 2.70 -> 2.16, VelOmega 1.40 -> 1.26, LapQPGradGrad 2.98 -> 2.29, LapQuadP 1.27 ->
// 0.90, RegFTVel 1.68 -> 1.41 (and LapPGradGrad 1.32 -> 1.15, its double layer 2.20 -> 1.66).
//
// Each struct cites the reference lines it restates and shows the rewrite from the reference's
// expression to the unit-direction form.
#pragma once

#include "ukernels.hpp"

namespace stkp2p {

// single-layer Stokes source [fx, fy, fz, TrD].  The reference keeps one running coefficient,
// c = f.r, and updates it in place: c - TrD for u, (c - TrD) + TrD for grad p / lap u, and
// ((c - TrD) + TrD) - TrD for grad u (StokesSingleLayerKernel.hpp:76-98, 139-145).  When
// |f.r| << |TrD| (close pairs) each round trip through TrD costs f.r relative accuracy, and the
// reference's results carry that; FP64 reproduces the sequence (SlFrame64) so that it agrees with the
// reference to rounding.  FP32 uses the exact expressions (there the round trip would cost ~1e-7 |TrD| /
// |f.r|) in unit-direction form: with s = 1/r, n = r s,  c s^k r-powers become  (c s) s^(k-1).
template <class R>
struct SlFrame {
    R s, nx, ny, nz;
    R c0, c1, c2, c3; // (f.r) s, (f.r - TrD) s, and the two later states of the coefficient, times s
    __device__ SlFrame(R dx, R dy, R dz, const R *f) {
        const R r2 = dx * dx + dy * dy + dz * dz;
        s = rsqrt_masked(r2);
        nx = dx * s;
        ny = dy * s;
        nz = dz * s;
        c0 = f[0] * nx + f[1] * ny + f[2] * nz;
        c1 = c0 - f[3] * s;
        c2 = c0;
        c3 = c1;
    }
};
// FP64 with w = 2/r: the coefficient's states over 4 (f/4 and TrD/4 staged as f[3..6]; f itself f[0..2])
struct SlFrame64 {
    double w, w2, w3, c0, c1, c2, c3;
    template <bool M>
    __device__ static SlFrame64 of(double dx, double dy, double dz, const double *f) {
        SlFrame64 a;
        a.w = twice_rsqrt_f64<M>(dx * dx + dy * dy + dz * dz);
        a.w2 = a.w * a.w;
        a.w3 = a.w2 * a.w;
        a.c0 = f[3] * dx + f[4] * dy + f[5] * dz;
        a.c1 = a.c0 - f[6];
        a.c2 = a.c1 + f[6];
        a.c3 = a.c2 - f[6];
        return a;
    }
};
__host__ __device__ inline void stage_sl64(const double *in, double *o) {
    for (int i = 0; i < 3; ++i) {
        o[i] = in[i];
        o[3 + i] = 0.25 * in[i];
    }
    o[6] = 0.25 * in[3];
}
// p (1), 2 u, 4 grad p: u_i = (f_i w + r_i (c1/4) w^3)/2, grad p_i = (f_i w^3 - 3 r_i (c2/4) w^5)/4
__device__ __forceinline__ void sl_pvel_gradp64(double *a, const SlFrame64 &q, double dx, double dy, double dz,
                                                const double *f) {
    const double b = q.c1 * q.w3;
    const double k = -3.0 * ((q.c2 * q.w3) * q.w2);
    a[0] += q.c0 * q.w3;
    a[1] += f[0] * q.w;
    a[1] += dx * b;
    a[2] += f[1] * q.w;
    a[2] += dy * b;
    a[3] += f[2] * q.w;
    a[3] += dz * b;
    a[4] += f[0] * q.w3;
    a[4] += dx * k;
    a[5] += f[1] * q.w3;
    a[5] += dy * k;
    a[6] += f[2] * q.w3;
    a[6] += dz * k;
}

// stokes_pvelgrad, StokesSingleLayerKernel.hpp:61-110; source [fx, fy, fz, TrD] ->
// [p, u(3), grad p(3), grad u(9) row-major du_i/dx_j].  With r^2 s^2 = 1 (c0..c3 of SlFrame):
//   p = 2 (f.r) s^3 = 2 c0 s^2
//   u_i = s^3 (r^2 f_i + (f.r - TrD) r_i) = s f_i + (c1 s) n_i
//   dp/dx_i = 2 s^5 (r^2 f_i - 3 r_i (f.r)) = 2 s^3 (f_i - 3 n_i c2)
//   du_i/dx_j = s^5 ((r^2 d_ij - 3 r_i r_j)(f.r - TrD) + r^2 (r_i f_j - r_j f_i))
//             = s^2 (d_ij c3 - 3 n_i n_j c3 + n_i f_j - n_j f_i)
// post() applies the 2 of p and grad p.
// FP64 (ACC64): besides p, u and grad p as sl_pvel_gradp64, grad u as the symmetric part -3 r_i r_j K (K =
// (c3/4) w^5), the antisymmetric part (r_i f_j - r_j f_i) w^3 and the multiple of the unit matrix (c3/4) w^3
// (8, 8 and 2 times their value): 55 operations a pair, and the reciprocal square root, for about 100 with
// the nine entries apart.
struct UkStokesPVelGrad {
    static constexpr int KS = 4, KS1 = 4, KL = 4, KL_FP64 = 7, KT = 16, ACC64 = 17;
    static constexpr bool STAGE_BY_PRECISION = true;
    static constexpr unsigned SRC_SCALE_MASK = 0x8u;
    __host__ __device__ static constexpr int deg(int k) { return k == 0 ? 2 : (k < 4 ? 1 : (k < 7 ? 3 : 2)); }
    __host__ __device__ static constexpr double post(int k) { return (k == 0 || (k >= 4 && k < 7)) ? 2.0 : 1.0; }
    template <int PREC>
    __host__ __device__ static void stage_p(const double *in, double *o) {
        if constexpr (PREC == 0) {
            stage_sl64(in, o);
        } else {
            o[0] = in[0]; o[1] = in[1]; o[2] = in[2]; o[3] = in[3];
        }
    }
    // a: p, u, grad p; 7 the unit matrix; 8-10 diagonal, 11-13 xy, xz, yz of r r K; 14-16 yz, zx, xy of r x f w^3
    template <bool M>
    __device__ static void eval64(double *a, double dx, double dy, double dz, const double *f) {
        const SlFrame64 q = SlFrame64::of<M>(dx, dy, dz, f);
        sl_pvel_gradp64(a, q, dx, dy, dz, f);
        const double m = q.c3 * q.w3;
        const double K = m * q.w2;
        const double kx = dx * K, ky = dy * K, kz = dz * K;
        const double vx = dx * q.w3, vy = dy * q.w3, vz = dz * q.w3;
        a[7] += m;
        a[8] += dx * kx;
        a[9] += dy * ky;
        a[10] += dz * kz;
        a[11] += dx * ky;
        a[12] += dx * kz;
        a[13] += dy * kz;
        a[14] += vy * f[2];
        a[14] -= vz * f[1];
        a[15] += vz * f[0];
        a[15] -= vx * f[2];
        a[16] += vx * f[1];
        a[16] -= vy * f[0];
    }
    __device__ static void finish64(const double *a, double *o) {
        o[0] = 0.5 * a[0];
        for (int i = 0; i < 3; ++i) {
            o[1 + i] = 0.5 * a[1 + i];
            o[4 + i] = 0.125 * a[4 + i];
            o[7 + 4 * i] = 0.5 * a[7] - 0.375 * a[8 + i];
        }
        o[8] = 0.125 * a[16] - 0.375 * a[11];
        o[10] = -0.125 * a[16] - 0.375 * a[11];
        o[9] = -0.125 * a[15] - 0.375 * a[12];
        o[13] = 0.125 * a[15] - 0.375 * a[12];
        o[12] = 0.125 * a[14] - 0.375 * a[13];
        o[14] = -0.125 * a[14] - 0.375 * a[13];
    }
    template <class R>
    __device__ static void eval(R *u, R dx, R dy, R dz, const R *f) {
        if constexpr (sizeof(R) == 8) {
            eval_by_acc64<UkStokesPVelGrad>(u, dx, dy, dz, f);
            return;
        }
        const SlFrame<R> a(dx, dy, dz, f);
        const R n[3] = {a.nx, a.ny, a.nz};
        const R s2 = a.s * a.s;
        const R s3 = s2 * a.s;
        const R ms = a.c1 * a.s;
        const R g = R(3.0) * a.c2;
        u[0] += a.c0 * s2;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            u[1 + i] += f[i] * a.s;
            u[1 + i] += n[i] * ms;
            u[4 + i] += s3 * (f[i] - n[i] * g);
        }
        const R M = a.c3 * s2;
        R p3[3], ns[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            p3[i] = R(3.0) * n[i] * M;
            ns[i] = n[i] * s2;
        }
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                if (i == j) {
                    u[7 + 3 * i + j] += M - p3[i] * n[j];
                } else {
                    u[7 + 3 * i + j] += ns[i] * f[j] - p3[i] * n[j];
                    u[7 + 3 * i + j] -= ns[j] * f[i];
                }
            }
    }
};

// stokes_pvellaplacian, StokesSingleLayerKernel.hpp:125-154: [p, u(3), lap u(3)];
//   lap u_i = 2 s^5 (f_i r^2 - 3 r_i (f.r)) = 2 s^3 (f_i - 3 n_i c2)   (= grad p of PVelGrad)
// FP64: sl_pvel_gradp64.
struct UkStokesPVelLaplacian {
    static constexpr int KS = 4, KS1 = 4, KL = 4, KL_FP64 = 7, KT = 7, ACC64 = 7;
    static constexpr bool STAGE_BY_PRECISION = true;
    static constexpr unsigned SRC_SCALE_MASK = 0x8u;
    __host__ __device__ static constexpr int deg(int k) { return k == 0 ? 2 : (k < 4 ? 1 : 3); }
    __host__ __device__ static constexpr double post(int k) { return (k == 0 || k >= 4) ? 2.0 : 1.0; }
    template <int PREC>
    __host__ __device__ static void stage_p(const double *in, double *o) {
        if constexpr (PREC == 0) {
            stage_sl64(in, o);
        } else {
            o[0] = in[0]; o[1] = in[1]; o[2] = in[2]; o[3] = in[3];
        }
    }
    template <bool M>
    __device__ static void eval64(double *a, double dx, double dy, double dz, const double *f) {
        sl_pvel_gradp64(a, SlFrame64::of<M>(dx, dy, dz, f), dx, dy, dz, f);
    }
    __device__ static void finish64(const double *a, double *o) {
        o[0] = 0.5 * a[0];
        for (int i = 0; i < 3; ++i) {
            o[1 + i] = 0.5 * a[1 + i];
            o[4 + i] = 0.125 * a[4 + i];
        }
    }
    template <class R>
    __device__ static void eval(R *u, R dx, R dy, R dz, const R *f) {
        if constexpr (sizeof(R) == 8) {
            eval_by_acc64<UkStokesPVelLaplacian>(u, dx, dy, dz, f);
            return;
        }
        const SlFrame<R> a(dx, dy, dz, f);
        const R n[3] = {a.nx, a.ny, a.nz};
        const R s2 = a.s * a.s;
        const R s3 = s2 * a.s;
        const R ms = a.c1 * a.s;
        const R g = R(3.0) * a.c2;
        u[0] += a.c0 * s2;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            u[1 + i] += f[i] * a.s;
            u[1 + i] += n[i] * ms;
            u[4 + i] += s3 * (f[i] - n[i] * g);
        }
    }
};

// stokes_traction, StokesSingleLayerKernel.hpp:169-194 (ScaleFactor -3/(4 pi), :166): stress row-major
//   sigma_ij = r_i r_j (f.r - TrD) s^5 + d_ij TrD r^2 s^5 / 3 = n_i n_j c1 s^2 + d_ij (TrD/3) s^3
// Staged: fx, fy, fz, TrD, TrD * invthree (the reference's invthree = 0.3333333333333333333).
// FP64: the stress is symmetric: r_i r_j (f.r - TrD) w^5 (32 times) as six sums, (TrD/3) w^3 (8 times) once.
struct UkStokesTraction {
    static constexpr int KS = 4, KS1 = 4, KL = 5, KT = 9, ACC64 = 7;
    static constexpr unsigned SRC_SCALE_MASK = 0x8u;
    __host__ __device__ static constexpr int deg(int) { return 2; }
    __host__ __device__ static constexpr double post(int k) { return ((void)k, 1.0); }
    __device__ static void stage(const double *in, double *o) {
        o[0] = in[0]; o[1] = in[1]; o[2] = in[2]; o[3] = in[3];
        o[4] = in[3] * 0.3333333333333333333;
    }
    template <bool M>
    __device__ static void eval64(double *a, double dx, double dy, double dz, const double *f) {
        const double w = twice_rsqrt_f64<M>(dx * dx + dy * dy + dz * dz);
        const double w2 = w * w;
        const double w3 = w2 * w;
        const double c = (f[0] * dx + f[1] * dy + f[2] * dz) - f[3];
        const double K = (c * w3) * w2;
        const double kx = dx * K, ky = dy * K, kz = dz * K;
        a[0] += f[4] * w3;
        a[1] += dx * kx;
        a[2] += dy * ky;
        a[3] += dz * kz;
        a[4] += dx * ky;
        a[5] += dx * kz;
        a[6] += dy * kz;
    }
    __device__ static void finish64(const double *a, double *o) {
        for (int i = 0; i < 3; ++i)
            o[4 * i] = 0.03125 * a[1 + i] + 0.125 * a[0];
        o[1] = o[3] = 0.03125 * a[4];
        o[2] = o[6] = 0.03125 * a[5];
        o[5] = o[7] = 0.03125 * a[6];
    }
    template <class R>
    __device__ static void eval(R *u, R dx, R dy, R dz, const R *f) {
        if constexpr (sizeof(R) == 8) {
            eval_by_acc64<UkStokesTraction>(u, dx, dy, dz, f);
            return;
        }
        const SlFrame<R> a(dx, dy, dz, f);
        const R n[3] = {a.nx, a.ny, a.nz};
        const R s2 = a.s * a.s;
        const R mm = a.c1 * s2;
        const R diag = f[4] * (s2 * a.s);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const R ai = n[i] * mm;
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                u[3 * i + j] += ai * n[j];
                if (i == j)
                    u[3 * i + j] += diag;
            }
        }
    }
};

// ---- double layer (StokesDoubleLayerKernel.hpp) --------------------------------------------------
// Every double-layer kernel depends on D through S = D + D^T and trD only.  Staged (FP64, the
// reference's source-only sums, :88-103): S = [2 Dxx, 2 Dyy, 2 Dzz, Dxy + Dyx, Dxz + Dzx,
// Dyz + Dzy], trD = Dxx + Dyy + Dzz.  Per pair: c = S n (the reference's (D r + D^T r) / r),
// Qh = n.D.n = (n.c)/2 (the reference's r.D.r / r^2).
__device__ inline void stage_sym(const double *in, double *o) {
    o[0] = in[0] + in[0];
    o[1] = in[4] + in[4];
    o[2] = in[8] + in[8];
    o[3] = in[1] + in[3];
    o[4] = in[2] + in[6];
    o[5] = in[5] + in[7];
    o[6] = in[0] + in[4] + in[8];
}

// FP64: staged H = S/2 (its off-diagonal entries halves of sums) and tr D / 2.  Per pair, w = 2/r:
// q = H r, t = 4 (r.D.r)/r^2 = (r.q) w^2, and with g = (5/8) t r - (trD/2) r - q, e = (5/8) t r - q
//   p = w^3 (trD/2 - (3/8) t)/2,  u = -(3/32) t w^3 r,  grad p = (3/8) w^5 g,
//   grad u_ij = (3/16) w^5 r_i e_j - d_ij (3/32) t w^3
__host__ __device__ inline void stage_sym64(const double *in, double *o) {
    o[0] = in[0];
    o[1] = in[4];
    o[2] = in[8];
    o[3] = 0.5 * (in[1] + in[3]);
    o[4] = 0.5 * (in[2] + in[6]);
    o[5] = 0.5 * (in[5] + in[7]);
    o[6] = 0.5 * (in[0] + in[4] + in[8]);
}
struct DlFrame64 {
    double w2, w3, w5, q[3], t;
    template <bool M>
    __device__ static DlFrame64 of(double dx, double dy, double dz, const double *h) {
        DlFrame64 a;
        const double w = twice_rsqrt_f64<M>(dx * dx + dy * dy + dz * dz);
        a.w2 = w * w;
        a.w3 = a.w2 * w;
        a.w5 = a.w3 * a.w2;
        a.q[0] = h[0] * dx + h[3] * dy + h[4] * dz;
        a.q[1] = h[3] * dx + h[1] * dy + h[5] * dz;
        a.q[2] = h[4] * dx + h[5] * dy + h[2] * dz;
        a.t = (a.q[0] * dx + a.q[1] * dy + a.q[2] * dz) * a.w2;
        return a;
    }
};
// p (2), u (-32/3), grad p (8/3): a[0..6]; returns t w^3
__device__ __forceinline__ double dl_pvel_gradp64(double *a, const DlFrame64 &b, double dx, double dy, double dz,
                                                  double trh) {
    const double v = b.t * b.w3;
    const double k = 0.625 * b.t - trh;
    a[0] += b.w3 * (trh - 0.375 * b.t);
    a[1] += dx * v;
    a[2] += dy * v;
    a[3] += dz * v;
    a[4] += b.w5 * (k * dx - b.q[0]);
    a[5] += b.w5 * (k * dy - b.q[1]);
    a[6] += b.w5 * (k * dz - b.q[2]);
    return v;
}
// before post() 2 (p), 1 (u), 6 (grad p)
__device__ inline void dl_pvel_gradp_finish64(const double *a, double *o) {
    o[0] = 0.25 * a[0];
    for (int i = 0; i < 3; ++i) {
        o[1 + i] = -0.09375 * a[1 + i];
        o[4 + i] = 0.0625 * a[4 + i];
    }
}

template <class R>
struct DlFrame {
    R s, n[3], c[3], qh;
    __device__ DlFrame(R dx, R dy, R dz, const R *g) {
        const R r2 = dx * dx + dy * dy + dz * dz;
        s = rsqrt_masked(r2);
        n[0] = dx * s;
        n[1] = dy * s;
        n[2] = dz * s;
        c[0] = g[0] * n[0] + g[3] * n[1] + g[4] * n[2];
        c[1] = g[3] * n[0] + g[1] * n[1] + g[5] * n[2];
        c[2] = g[4] * n[0] + g[5] * n[1] + g[2] * n[2];
        qh = R(0.5) * (n[0] * c[0] + n[1] * c[1] + n[2] * c[2]);
    }
};

// stokes_doublepvel part of the double-layer gradient kernels (:106-111, :192-197):
//   p = 2 s^5 (r^2 trD - 3 r.D.r) = 2 s^3 (trD - 3 Qh),   u_i = -3 r_i (r.D.r) s^5 = -3 Qh s^2 n_i
//   dp/dx_i (:115-118, :201-204, with its rinv7 *= -3):
//     = 6 s^7 (5 r_i (r.D.r) - r^2 ((D r + D^T r)_i + r_i trD)) = 6 s^4 ((5 Qh - trD) n_i - c_i)
// post(): 2 for p, 6 for grad p.
template <class R>
__device__ inline void dl_pvel_gradp(R *u, const DlFrame<R> &a, R trd) {
    const R s2 = a.s * a.s;
    const R s3 = s2 * a.s;
    const R s4 = s2 * s2;
    const R h = R(-3.0) * a.qh;
    u[0] += s3 * (trd + h);
    const R v = h * s2;
    const R w = R(5.0) * a.qh - trd;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        u[1 + i] += a.n[i] * v;
        u[4 + i] += s4 * (w * a.n[i] - a.c[i]);
    }
}

// stokes_doublepvelgrad, StokesDoubleLayerKernel.hpp:71-142; D row-major (9) -> 16.
//   du_i/dx_j (:131-141, rinv7 already times -3; the bracket is of degree 4 in r):
//     = -3 s^7 (-5 (r.D.r) r_i r_j + r^2 r_i (D r + D^T r)_j + r^2 (r.D.r) d_ij)
//     = 3 s^3 (5 Qh n_i n_j - n_i c_j - Qh d_ij);   post() 3
struct UkStokesDoublePVelGrad {
    static constexpr int KS = 9, KS1 = 9, KL = 7, KT = 16, ACC64 = 17;
    static constexpr bool STAGE_BY_PRECISION = true;
    static constexpr unsigned SRC_SCALE_MASK = 0x1FFu;
    __host__ __device__ static constexpr int deg(int k) { return k == 0 ? 2 : (k < 4 ? 1 : (k < 7 ? 3 : 2)); }
    __host__ __device__ static constexpr double post(int k) { return k == 0 ? 2.0 : (k < 4 ? 1.0 : (k < 7 ? 6.0 : 3.0)); }
    template <int PREC>
    __host__ __device__ static void stage_p(const double *in, double *o) {
        if constexpr (PREC == 0)
            stage_sym64(in, o);
        else
            stage_sym(in, o);
    }
    // a: p, u, grad p; 7-15 r_i e_j w^5; 16 t w^3
    template <bool M>
    __device__ static void eval64(double *a, double dx, double dy, double dz, const double *h) {
        const DlFrame64 b = DlFrame64::of<M>(dx, dy, dz, h);
        a[16] += dl_pvel_gradp64(a, b, dx, dy, dz, h[6]);
        const double r[3] = {dx, dy, dz};
        const double t5 = 0.625 * b.t;
        double e[3];
#pragma unroll
        for (int j = 0; j < 3; ++j)
            e[j] = b.w5 * (t5 * r[j] - b.q[j]);
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j)
                a[7 + 3 * i + j] += r[i] * e[j];
    }
    __device__ static void finish64(const double *a, double *o) {
        dl_pvel_gradp_finish64(a, o);
        for (int k = 0; k < 9; ++k)
            o[7 + k] = 0.0625 * a[7 + k] - (k % 4 == 0 ? 0.03125 * a[16] : 0.0);
    }
    template <class R>
    __device__ static void eval(R *u, R dx, R dy, R dz, const R *g) {
        if constexpr (sizeof(R) == 8) {
            eval_by_acc64<UkStokesDoublePVelGrad>(u, dx, dy, dz, g);
            return;
        }
        const DlFrame<R> a(dx, dy, dz, g);
        dl_pvel_gradp(u, a, g[6]);
        const R s3 = a.s * a.s * a.s;
        const R q5 = R(5.0) * a.qh;
        const R dq = s3 * a.qh;
        R e[3];
#pragma unroll
        for (int j = 0; j < 3; ++j)
            e[j] = s3 * (q5 * a.n[j] - a.c[j]);
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                u[7 + 3 * i + j] += a.n[i] * e[j];
                if (i == j)
                    u[7 + 3 * i + j] -= dq;
            }
    }
};

// stokes_doublelaplacian, StokesDoubleLayerKernel.hpp:157-205; D (9) -> [p, u(3), lap u(3)]
// (lap u has the expression of the double-layer grad p, :202-204)
struct UkStokesDoubleLaplacian {
    static constexpr int KS = 9, KS1 = 9, KL = 7, KT = 7, ACC64 = 7;
    static constexpr bool STAGE_BY_PRECISION = true;
    static constexpr unsigned SRC_SCALE_MASK = 0x1FFu;
    __host__ __device__ static constexpr int deg(int k) { return k == 0 ? 2 : (k < 4 ? 1 : 3); }
    __host__ __device__ static constexpr double post(int k) { return k == 0 ? 2.0 : (k < 4 ? 1.0 : 6.0); }
    template <int PREC>
    __host__ __device__ static void stage_p(const double *in, double *o) {
        if constexpr (PREC == 0)
            stage_sym64(in, o);
        else
            stage_sym(in, o);
    }
    template <bool M>
    __device__ static void eval64(double *a, double dx, double dy, double dz, const double *h) {
        (void)dl_pvel_gradp64(a, DlFrame64::of<M>(dx, dy, dz, h), dx, dy, dz, h[6]);
    }
    __device__ static void finish64(const double *a, double *o) { dl_pvel_gradp_finish64(a, o); }
    template <class R>
    __device__ static void eval(R *u, R dx, R dy, R dz, const R *g) {
        if constexpr (sizeof(R) == 8) {
            eval_by_acc64<UkStokesDoubleLaplacian>(u, dx, dy, dz, g);
            return;
        }
        const DlFrame<R> a(dx, dy, dz, g);
        dl_pvel_gradp(u, a, g[6]);
    }
};

// stokes_doubletraction, StokesDoubleLayerKernel.hpp:220-272 (ScaleFactor -3/(8 pi), :217):
//   np = facp r^2 s^7 (r^2 trD - 3 r.D.r) = facp s^3 (trD - 3 Qh)    (facp = 0.66666666666666)
//   tv_ij = s^7 (-5 (r.D.r) r_i r_j + r^2 r_i (D r + D^T r)_j + r^2 (r.D.r) d_ij)   (degree 4)
//         = s^3 (-5 Qh n_i n_j + n_i c_j + Qh d_ij)
//   sigma_ij = d_ij np + tv_ij + tv_ji = d_ij (np + 2 s^3 Qh) + n_i h_j + n_j h_i,
//   h_j = s^3 (c_j - 5 Qh n_j)
struct UkStokesDoubleTraction {
    static constexpr int KS = 9, KS1 = 9, KL = 7, KT = 9, ACC64 = 7;
    static constexpr bool STAGE_BY_PRECISION = true;
    static constexpr unsigned SRC_SCALE_MASK = 0x1FFu;
    __host__ __device__ static constexpr int deg(int) { return 2; }
    __host__ __device__ static constexpr double post(int k) { return ((void)k, 1.0); }
    template <int PREC>
    __host__ __device__ static void stage_p(const double *in, double *o) {
        if constexpr (PREC == 0)
            stage_sym64(in, o);
        else
            stage_sym(in, o);
    }
    // FP64: sigma_ij = -(w^5/16) (r_i e_j + r_j e_i) + d_ij (w^3/8) (facp trD - (3 facp - 2) t/4): the unit
    // matrix's multiple, r_i e_i w^5 and (r_i e_j + r_j e_i) w^5 as seven sums
    template <bool M>
    __device__ static void eval64(double *a, double dx, double dy, double dz, const double *h) {
        const DlFrame64 b = DlFrame64::of<M>(dx, dy, dz, h);
        constexpr double facp = 0.66666666666666;
        const double t5 = 0.625 * b.t;
        const double ex = b.w5 * (t5 * dx - b.q[0]), ey = b.w5 * (t5 * dy - b.q[1]), ez = b.w5 * (t5 * dz - b.q[2]);
        a[0] += b.w3 * (2.0 * facp * h[6] - (0.25 * (3.0 * facp - 2.0)) * b.t);
        a[1] += dx * ex;
        a[2] += dy * ey;
        a[3] += dz * ez;
        a[4] += dx * ey;
        a[4] += dy * ex;
        a[5] += dx * ez;
        a[5] += dz * ex;
        a[6] += dy * ez;
        a[6] += dz * ey;
    }
    __device__ static void finish64(const double *a, double *o) {
        for (int i = 0; i < 3; ++i)
            o[4 * i] = 0.125 * a[0] - 0.125 * a[1 + i];
        o[1] = o[3] = -0.0625 * a[4];
        o[2] = o[6] = -0.0625 * a[5];
        o[5] = o[7] = -0.0625 * a[6];
    }
    template <class R>
    __device__ static void eval(R *u, R dx, R dy, R dz, const R *g) {
        if constexpr (sizeof(R) == 8) {
            eval_by_acc64<UkStokesDoubleTraction>(u, dx, dy, dz, g);
            return;
        }
        const DlFrame<R> a(dx, dy, dz, g);
        const R s3 = a.s * a.s * a.s;
        const R np = R(0.66666666666666) * (s3 * (g[6] - R(3.0) * a.qh));
        const R diag = np + R(2.0) * (s3 * a.qh);
        const R q5 = R(5.0) * a.qh;
        R h[3];
#pragma unroll
        for (int j = 0; j < 3; ++j)
            h[j] = s3 * (a.c[j] - q5 * a.n[j]);
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                u[3 * i + j] += a.n[i] * h[j];
                u[3 * i + j] += a.n[j] * h[i];
                if (i == j)
                    u[3 * i + j] += diag;
            }
    }
};

// ---- regularised force + torque (StokesRegSingleLayerKernel.hpp) ----------------------------------
// Source [fx, fy, fz, tx, ty, tz, eps]; rho^2 = r^2 + eps^2, s = 1/rho (masked at rho = 0, where the
// reference divides by zero), n = r s, q = r^2 s^2, e = eps^2 s^2 (q + e = 1).  Staged: f, t, eps^2.
template <class R>
struct RegFrame {
    R s, n[3], q, e;
    __device__ RegFrame(R dx, R dy, R dz, R eps2) {
        const R r2 = dx * dx + dy * dy + dz * dz;
        s = rsqrt_masked(r2 + eps2);
        n[0] = dx * s;
        n[1] = dy * s;
        n[2] = dz * s;
        const R ss = s * s;
        q = r2 * ss;
        e = eps2 * ss;
    }
};

// velocity of stokes_regftvel (:85-87) and stokes_regftvelomega (:143-145):
//   H1 f + H2 (f.r) r + rc (t x r),  H1 = (r^2 + 2 eps^2) s^3 = (q + 2e) s,  H2 r_i r_j = s n_i n_j,
//   rc (t x r) = (2 r^2 + 5 eps^2) s^5 / 2 (t x r) = (2q + 5e)/2 s^2 (t x n)
template <class R>
__device__ inline void reg_velocity(R *u, const RegFrame<R> &a, const R *f, R rc2) {
    const R h1 = (a.q + R(2.0) * a.e) * a.s;
    const R fn = f[0] * a.n[0] + f[1] * a.n[1] + f[2] * a.n[2];
    const R b = fn * a.s;
    const R tx = f[4] * a.n[2] - f[5] * a.n[1];
    const R ty = f[5] * a.n[0] - f[3] * a.n[2];
    const R tz = f[3] * a.n[1] - f[4] * a.n[0];
    u[0] += f[0] * h1;
    u[0] += a.n[0] * b;
    u[0] += rc2 * tx;
    u[1] += f[1] * h1;
    u[1] += a.n[1] * b;
    u[1] += rc2 * ty;
    u[2] += f[2] * h1;
    u[2] += a.n[2] * b;
    u[2] += rc2 * tz;
}

// FP64: with eps^2 = rho^2 - r^2 eliminated, eta = eps^2 s^2:  H1 = s (1 + eta), rc = s^3 (1 + 3/2 eta),
// D1 = s^3 (15 eta^2 - 3 eta - 2)/4, D2 = s^5 (15 eta + 6)/4; the cross products take rc r once.
struct RegFrame64 {
    double s, s2, s3, eta, rc[3], b;
    template <bool M>
    __device__ static RegFrame64 of(double dx, double dy, double dz, const double *f) {
        RegFrame64 a;
        a.s = rsqrt_f64<M>(dx * dx + (dy * dy + (dz * dz + f[6])));
        a.s2 = a.s * a.s;
        a.s3 = a.s2 * a.s;
        a.eta = f[6] * a.s2;
        const double rc = a.s3 * (1.5 * a.eta + 1.0);
        a.rc[0] = rc * dx;
        a.rc[1] = rc * dy;
        a.rc[2] = rc * dz;
        a.b = (f[0] * dx + f[1] * dy + f[2] * dz) * a.s3;
        return a;
    }
    // a[0..2] += t x v
    __device__ static void cross(double *a, const double *t, const double *v) {
        a[0] += t[1] * v[2];
        a[0] -= t[2] * v[1];
        a[1] += t[2] * v[0];
        a[1] -= t[0] * v[2];
        a[2] += t[0] * v[1];
        a[2] -= t[1] * v[0];
    }
    __device__ void velocity(double *a, double dx, double dy, double dz, const double *f) const {
        const double h1 = eta * s + s;
        a[0] += f[0] * h1;
        a[0] += dx * b;
        a[1] += f[1] * h1;
        a[1] += dy * b;
        a[2] += f[2] * h1;
        a[2] += dz * b;
        cross(a, f + 3, rc);
    }
};

// stokes_regftvel, StokesRegSingleLayerKernel.hpp:55-88: [f, t, eps] -> u(3)
struct UkStokesRegFTVel {
    static constexpr int KS = 7, KS1 = 7, KL = 7, KT = 3, ACC64 = 3;
    static constexpr unsigned SRC_SCALE_MASK = 0x78u;
    __host__ __device__ static constexpr int deg(int) { return 1; }
    __host__ __device__ static constexpr double post(int k) { return ((void)k, 1.0); }
    __device__ static void stage(const double *in, double *o) {
        for (int k = 0; k < 6; ++k)
            o[k] = in[k];
        o[6] = in[6] * in[6];
    }
    template <bool M>
    __device__ static void eval64(double *a, double dx, double dy, double dz, const double *f) {
        RegFrame64::of<M>(dx, dy, dz, f).velocity(a, dx, dy, dz, f);
    }
    __device__ static void finish64(const double *a, double *o) {
        for (int k = 0; k < KT; ++k)
            o[k] = a[k];
    }
    template <class R>
    __device__ static void eval(R *u, R dx, R dy, R dz, const R *f) {
        if constexpr (sizeof(R) == 8) {
            eval_by_acc64<UkStokesRegFTVel>(u, dx, dy, dz, f);
            return;
        }
        const RegFrame<R> a(dx, dy, dz, f[6]);
        const R rc2 = (R(2.0) * a.q + R(5.0) * a.e) * (R(0.5) * (a.s * a.s));
        reg_velocity(u, a, f, rc2);
    }
};

// stokes_regftvelomega, StokesRegSingleLayerKernel.hpp:103-150: [f, t, eps] -> [u(3), omega(3)]
//   omega = D1 t + D2 (t.r) r + rc (f x r),
//   D1 = (10 eps^4 - 7 eps^2 r^2 - 2 r^4) s^7 / 4 = (10 e^2 - 7 e q - 2 q^2)/4 s^3,
//   D2 r_i r_j = (21 eps^2 + 6 r^2) s^7 / 4 r_i r_j = (21 e + 6 q)/4 s^3 n_i n_j
struct UkStokesRegFTVelOmega {
    static constexpr int KS = 7, KS1 = 7, KL = 7, KT = 6, ACC64 = 6;
    static constexpr unsigned SRC_SCALE_MASK = 0x78u;
    __host__ __device__ static constexpr int deg(int k) { return k < 3 ? 1 : 2; }
    __host__ __device__ static constexpr double post(int k) { return ((void)k, 1.0); }
    __device__ static void stage(const double *in, double *o) { UkStokesRegFTVel::stage(in, o); }
    template <bool M>
    __device__ static void eval64(double *a, double dx, double dy, double dz, const double *f) {
        const RegFrame64 q = RegFrame64::of<M>(dx, dy, dz, f);
        q.velocity(a, dx, dy, dz, f);
        const double d1 = (q.eta * (15.0 * q.eta - 3.0) - 2.0) * (0.25 * q.s3);
        const double d2 = (q.s3 * q.s2) * (3.75 * q.eta + 1.5);
        const double b = d2 * (f[3] * dx + f[4] * dy + f[5] * dz);
        a[3] += f[3] * d1;
        a[3] += dx * b;
        a[4] += f[4] * d1;
        a[4] += dy * b;
        a[5] += f[5] * d1;
        a[5] += dz * b;
        RegFrame64::cross(a + 3, f, q.rc);
    }
    __device__ static void finish64(const double *a, double *o) {
        for (int k = 0; k < KT; ++k)
            o[k] = a[k];
    }
    template <class R>
    __device__ static void eval(R *u, R dx, R dy, R dz, const R *f) {
        if constexpr (sizeof(R) == 8) {
            eval_by_acc64<UkStokesRegFTVelOmega>(u, dx, dy, dz, f);
            return;
        }
        const RegFrame<R> a(dx, dy, dz, f[6]);
        const R ss = a.s * a.s;
        const R rc2 = (R(2.0) * a.q + R(5.0) * a.e) * (R(0.5) * ss);
        reg_velocity(u, a, f, rc2);
        const R s34 = R(0.25) * (ss * a.s);
        const R d1 = (a.e * (R(10.0) * a.e - R(7.0) * a.q) - R(2.0) * (a.q * a.q)) * s34;
        const R d2 = (R(21.0) * a.e + R(6.0) * a.q) * s34;
        const R tn = f[3] * a.n[0] + f[4] * a.n[1] + f[5] * a.n[2];
        const R b = d2 * tn;
        const R fx = f[1] * a.n[2] - f[2] * a.n[1];
        const R fy = f[2] * a.n[0] - f[0] * a.n[2];
        const R fz = f[0] * a.n[1] - f[1] * a.n[0];
        u[3] += f[3] * d1;
        u[3] += a.n[0] * b;
        u[3] += rc2 * fx;
        u[4] += f[4] * d1;
        u[4] += a.n[1] * b;
        u[4] += rc2 * fy;
        u[5] += f[5] * d1;
        u[5] += a.n[2] * b;
        u[5] += rc2 * fz;
    }
};

// stokes_velomega, StokesRegSingleLayerKernel.hpp:165-201 (L2T kernel of StokesRegVelOmega, :223-229):
// f(3) -> [u(3), omega(3)];  u = f s + (f.n) s n  (the Stokeslet),  omega = r^2 s^5 (f x r) = s^2 (f x n)
// FP64: w = 2/r, f and f/4 staged: u = (f w + r ((f/4).r) w^3)/2, omega = f x (r w^3)/8.
struct UkStokesVelOmega {
    static constexpr int KS = 3, KS1 = 3, KL = 3, KL_FP64 = 6, KT = 6, ACC64 = 6;
    static constexpr bool STAGE_BY_PRECISION = true;
    static constexpr unsigned SRC_SCALE_MASK = 0u;
    __host__ __device__ static constexpr int deg(int k) { return k < 3 ? 1 : 2; }
    __host__ __device__ static constexpr double post(int k) { return ((void)k, 1.0); }
    template <int PREC>
    __host__ __device__ static void stage_p(const double *in, double *o) {
        for (int i = 0; i < 3; ++i) {
            o[i] = in[i];
            if constexpr (PREC == 0)
                o[3 + i] = 0.25 * in[i];
        }
    }
    template <bool M>
    __device__ static void eval64(double *a, double dx, double dy, double dz, const double *f) {
        const double w = twice_rsqrt_f64<M>(dx * dx + dy * dy + dz * dz);
        const double w3 = (w * w) * w;
        const double b = (f[3] * dx + f[4] * dy + f[5] * dz) * w3;
        a[0] += f[0] * w;
        a[0] += dx * b;
        a[1] += f[1] * w;
        a[1] += dy * b;
        a[2] += f[2] * w;
        a[2] += dz * b;
        const double v[3] = {dx * w3, dy * w3, dz * w3};
        RegFrame64::cross(a + 3, f, v);
    }
    __device__ static void finish64(const double *a, double *o) {
        for (int k = 0; k < 3; ++k) {
            o[k] = 0.5 * a[k];
            o[3 + k] = 0.125 * a[3 + k];
        }
    }
    template <class R>
    __device__ static void eval(R *u, R dx, R dy, R dz, const R *f) {
        if constexpr (sizeof(R) == 8) {
            eval_by_acc64<UkStokesVelOmega>(u, dx, dy, dz, f);
            return;
        }
        const R r2 = dx * dx + dy * dy + dz * dz;
        const R s = rsqrt_masked(r2);
        const R nx = dx * s, ny = dy * s, nz = dz * s;
        const R b = (f[0] * nx + f[1] * ny + f[2] * nz) * s;
        const R ss = s * s;
        u[0] += f[0] * s;
        u[0] += nx * b;
        u[1] += f[1] * s;
        u[1] += ny * b;
        u[2] += f[2] * s;
        u[2] += nz * b;
        u[3] += ss * (f[1] * nz - f[2] * ny);
        u[4] += ss * (f[2] * nx - f[0] * nz);
        u[5] += ss * (f[0] * ny - f[1] * nx);
    }
};

// ---- Laplace quadrupole (LaplaceLayerKernel.hpp) ----------------------------------------------------
// Q row-major (9), staged like the Stokes double layer (S = Q + Q^T, trQ).

// laplace_quadp, LaplaceLayerKernel.hpp:209-231:  p = (3 r.Q.r - r^2 trQ) s^5 = s^3 (3 Qh - trQ)
// FP64: 3 (r.Q.r)/r^2 - trQ with z^2 = r^2 - x^2 - y^2 (as UkStokesDoublePVel) and w = 2/r: staged 3/4 (Qxx -
// Qzz), 3/4 (Qyy - Qzz), 3 Qzz - trQ, 3/4 (Qxy + Qyx), 3/4 (Qxz + Qzx), 3/4 (Qyz + Qzy).
struct UkLaplaceQuadP {
    static constexpr int KS = 9, KS1 = 9, KL = 7, KL_FP64 = 6, KT = 1, ACC64 = 1;
    static constexpr bool STAGE_BY_PRECISION = true;
    static constexpr unsigned SRC_SCALE_MASK = 0u;
    __host__ __device__ static constexpr int deg(int) { return 3; }
    __host__ __device__ static constexpr double post(int k) { return ((void)k, 1.0); }
    template <int PREC>
    __host__ __device__ static void stage_p(const double *in, double *o) {
        if constexpr (PREC == 0) {
            o[0] = 0.75 * (in[0] - in[8]);
            o[1] = 0.75 * (in[4] - in[8]);
            o[2] = 3.0 * in[8] - (in[0] + in[4] + in[8]);
            o[3] = 0.75 * (in[1] + in[3]);
            o[4] = 0.75 * (in[2] + in[6]);
            o[5] = 0.75 * (in[5] + in[7]);
        } else {
            stage_sym(in, o);
        }
    }
    template <bool M>
    __device__ static void eval64(double *a, double dx, double dy, double dz, const double *g) {
        const double w = twice_rsqrt_f64<M>(dx * dx + dy * dy + dz * dz);
        const double w2 = w * w;
        const double x = g[0] * dx + g[3] * dy + g[4] * dz;
        const double y = g[1] * dy + g[5] * dz;
        a[0] += (w2 * w) * ((dx * x + dy * y) * w2 + g[2]);
    }
    __device__ static void finish64(const double *a, double *o) { o[0] = 0.125 * a[0]; }
    template <class R>
    __device__ static void eval(R *u, R dx, R dy, R dz, const R *g) {
        if constexpr (sizeof(R) == 8) {
            eval_by_acc64<UkLaplaceQuadP>(u, dx, dy, dz, g);
            return;
        }
        const DlFrame<R> a(dx, dy, dz, g);
        u[0] += (a.s * a.s * a.s) * (R(3.0) * a.qh - g[6]);
    }
};

// laplace_quadpgradgrad, LaplaceLayerKernel.hpp:241-311: [p, grad(3), Hessian xx,xy,xz,yy,yz,zz]
//   grad_i = -3 s^7 (5 r_i r.Q.r - r^2 (S r + r trQ)_i) = -3 s^4 ((5 Qh - trQ) n_i - c_i)    post -3
//   H_ij = s^9 (105 r_i r_j r.Q.r - 15 r^2 (d_ij r.Q.r + r_j (S r)_i + r_i (S r)_j + r_i r_j trQ)
//               + 3 r^4 (d_ij trQ + S_ij))
//        = 3 s^5 (n_i n_j (35 Qh - 5 trQ) - 5 (n_j c_i + n_i c_j) + S_ij + d_ij (trQ - 5 Qh))  post 3
struct UkLaplaceQuadPGradGrad {
    static constexpr int KS = 9, KS1 = 9, KL = 7, KT = 10, ACC64 = 11;
    static constexpr bool STAGE_BY_PRECISION = true;
    static constexpr unsigned SRC_SCALE_MASK = 0u;
    __host__ __device__ static constexpr int deg(int k) { return k == 0 ? 3 : (k < 4 ? 4 : 5); }
    __host__ __device__ static constexpr double post(int k) { return k == 0 ? 1.0 : (k < 4 ? -3.0 : 3.0); }
    template <int PREC>
    __host__ __device__ static void stage_p(const double *in, double *o) {
        if constexpr (PREC == 0)
            stage_sym64(in, o);
        else
            stage_sym(in, o);
    }
    // FP64 (b, t, q, g as the Stokes double layer): p = w^3/4 ((3/8) t - trQ/2), grad = -3 w^5/16 g (a before
    // post()), H_ij/3 = (10/128) w^7 (r_i y_j + r_j y_i) + (w^5/32) S_ij - d_ij (w^5/16) ((5/8) t - trQ/2),
    // y = ((7/16) t - trQ/4) r - q.  Sums: 0 p, 1-3 grad, 4 the unit matrix, 5-7 and 8-10 the diagonal and
    // off-diagonal of r y w^7 with S w^5 joined to them (S_ij = 2 H_ij: 0.8 H_ij off, 0.4 H_ii on the diagonal)
    template <bool M>
    __device__ static void eval64(double *a, double dx, double dy, double dz, const double *h) {
        const DlFrame64 b = DlFrame64::of<M>(dx, dy, dz, h);
        const double k = 0.625 * b.t - h[6];
        a[0] += b.w3 * (0.375 * b.t - h[6]);
        a[1] += b.w5 * (k * dx - b.q[0]);
        a[2] += b.w5 * (k * dy - b.q[1]);
        a[3] += b.w5 * (k * dz - b.q[2]);
        a[4] += b.w5 * k;
        const double y = 0.4375 * b.t - 0.5 * h[6];
        const double w7 = b.w5 * b.w2, wo = 0.8 * b.w5, wd = 0.4 * b.w5;
        const double yx = w7 * (y * dx - b.q[0]), yy = w7 * (y * dy - b.q[1]), yz = w7 * (y * dz - b.q[2]);
        a[5] += dx * yx;
        a[5] += wd * h[0];
        a[6] += dy * yy;
        a[6] += wd * h[1];
        a[7] += dz * yz;
        a[7] += wd * h[2];
        a[8] += dx * yy;
        a[8] += dy * yx;
        a[8] += wo * h[3];
        a[9] += dx * yz;
        a[9] += dz * yx;
        a[9] += wo * h[4];
        a[10] += dy * yz;
        a[10] += dz * yy;
        a[10] += wo * h[5];
    }
    __device__ static void finish64(const double *a, double *o) {
        o[0] = 0.25 * a[0];
        for (int i = 0; i < 3; ++i)
            o[1 + i] = 0.0625 * a[1 + i];
        const double d = 0.0625 * a[4];
        o[4] = 0.15625 * a[5] - d;
        o[7] = 0.15625 * a[6] - d;
        o[9] = 0.15625 * a[7] - d;
        o[5] = 0.078125 * a[8];
        o[6] = 0.078125 * a[9];
        o[8] = 0.078125 * a[10];
    }
    template <class R>
    __device__ static void eval(R *u, R dx, R dy, R dz, const R *g) {
        if constexpr (sizeof(R) == 8) {
            eval_by_acc64<UkLaplaceQuadPGradGrad>(u, dx, dy, dz, g);
            return;
        }
        const DlFrame<R> a(dx, dy, dz, g);
        const R trq = g[6];
        const R s2 = a.s * a.s;
        const R s3 = s2 * a.s;
        const R s4 = s2 * s2;
        const R s5 = s4 * a.s;
        u[0] += s3 * (R(3.0) * a.qh - trq);
        const R w = R(5.0) * a.qh - trq;
#pragma unroll
        for (int i = 0; i < 3; ++i)
            u[1 + i] += s4 * (w * a.n[i] - a.c[i]);
        // S_ij of the staged layout: diagonal g[0..2], off-diagonal xy g[3], xz g[4], yz g[5]
        const R A = R(35.0) * a.qh - R(5.0) * trq;
        const R dg = trq - R(5.0) * a.qh;
        R nA[3], c5[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            nA[i] = a.n[i] * A;
            c5[i] = R(5.0) * a.c[i];
        }
        constexpr int I[6] = {0, 0, 0, 1, 1, 2}, J[6] = {0, 1, 2, 1, 2, 2}, SIDX[6] = {0, 3, 4, 1, 5, 2};
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            const int i = I[k], j = J[k];
            R h = nA[i] * a.n[j] - (a.n[j] * c5[i] + a.n[i] * c5[j]) + g[SIDX[k]];
            if (i == j)
                h += dg;
            u[4 + k] += s5 * h;
        }
    }
};

} // namespace stkp2p
