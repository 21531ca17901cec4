// kernels.hpp -- gfx950 device code of liboctofmm: FP64 pair arithmetic, the
// FP32 pairs of mixed precision, kernel arguments and the tree passes' shifts.
//
// Pair arithmetic gives what Octo-Tiger's templates give
// (octotiger/multipole_interactions/kernel/compute_kernel_templates.hpp:67-391,
//  octotiger/monopole_interactions/kernel/monopole_kernel_templates.hpp:16-239):
// the order-3 contraction of a partner's moments with the derivatives of -1/r,
// and the angular-momentum correction from the order-4 ones.  The FP64 pairs
// form no derivative tensor for it (see below); the FP32 pairs do.
#pragma once

#include <hip/hip_runtime.h>

#include "octofmm.h"
#include "octofmm_internal.hpp"

namespace octofmm {

// ---------------------------------------------------------------------------
// Pair arithmetic
//
// The derivatives of -1/r are harmonic, so every trace over two of their
// indices vanishes: at separation x, with d1 = 1/r^3, d2 = -3/r^5, d3 = 15/r^7,
// 3 d1 + d2 r^2 = 0 and 5 d2 + d3 r^2 = 0.  The pair functions therefore never
// form the tensors D_ab and D_abc.  They contract the partner's moments with
// the separation (vectors Q x, scalars x Q x, p x, B x x x) and accumulate
// sums of a few radial powers times those, from which a target's expansion is
// formed once, after its last pair (acc_finish):
//   - only the trace-free parts of the quadrupole Q and of the octupole B act
//     on L, so the staged record holds those;
//   - L_ab and L_abc are the trace-free parts of the sums R_ab (Acc::hd, ho)
//     and T_abc (Acc::t), which leave out every term that only adds a trace;
//   - the angular-momentum correction uses the order-4 derivatives without
//     their d4 term, -[d2 tau_d + d3 (B_dbc x_b x_c + x_d tau x)] with tau the
//     trace of B.  Split into trace-free part and trace, the d2 term cancels:
//     -d3 [B0_dbc x_b x_c + 7/5 x_d tau x];
//   - the target's own octupole enters the correction linearly, as the mass
//     ratio m0 / mc0 times the same form, so its part needs only the sums
//     W_bc = sum m0 d3 x_b x_c.
// FP64 VALU issue bounds the level kernels, so the instructions per pair are
// what counts: 115 (RHO) and 102 (DRHODT) per far pair, where forming the
// tensors took 177 and 132.  A pass over 4096 sub-grids went 2.97 -> 2.19 ms
// (RHO) and 2.42 -> 2.00 ms (DRHODT), over 512 0.386 -> 0.293 ms, with the
// errors against 64-bit sums no larger.  The identities hold for separations
// above the floor r^2 >= 1e-20, which exists so that a pair of coincident
// empty cells gives zero, not NaN.
//
// Powers: one Newton step of the hardware estimate gives P = 2/r (rsqrt2), and
// d1' = P^3, e2 = P^5, e3 = P^7 carry the factors 8, 32, 128, which the
// record's scales and acc_finish take back.
//
// Record of one partner cell, 24 doubles:
//   0      m0
//   1..3   5/4 p
//   4..8   15/32 of the trace-free M_ab: xx xy xz yy yz
//   9..20  RHO: 5/64 of the trace-free part of M_abc, xxx xyy xzz xxy yyy yzz
//          xxz yyz xyz, then 7/10 of the trace of 5/64 M_abc
//          DRHODT: the same trace-free part as the coefficients of the 8 cubic
//          monomials of cubic_monomials (9..16), zeros
//   21..23 centre of mass
// ---------------------------------------------------------------------------

// Sum over the 8 lanes of an aligned group, by three DPP lane moves (VALU ops,
// no LDS round trip): the pair of xor 1, the pair of xor 2 within each quad,
// then the mirrored lane of the other quad (7 - i within each half row, once
// every lane holds its quad's sum).  Every lane ends with the same value:
// ((v0 + v1) + (v2 + v3)) + ((v4 + v5) + (v6 + v7)), in the same order on
// every run.  The 8 lanes of a group must be active together.
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)b, CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xF, 0xF, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

__device__ __forceinline__ double sum8(double v) {
    v += dpp_move<0xB1>(v);    // quad_perm [1, 0, 3, 2]
    v += dpp_move<0x4E>(v);    // quad_perm [2, 3, 0, 1]
    v += dpp_move<0x141>(v);   // row_half_mirror
    return v;
}

// 2/sqrt(x): the hardware estimate (relative error <= 5.2e-8, measured on
// MI355X over x in [1e-12, 1e6]) refined by one Newton step, which squares the
// error: <= 4.1e-15 (a second step would give 1.4e-16).  The expansion's
// highest power scales it by at most 7, far inside the 1e-12 gate.  Without
// the step's factor 1/2 it is one instruction shorter.
__device__ __forceinline__ double rsqrt2(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    return y * fma(-(x * y), y, 3.0);
}

// Running sums of one target cell over its partners (see the top of the
// file); scales as acc_finish takes them.
template <bool RHO>
struct Acc {
    double a0, aq;      // potential
    double l[3];        // gradient
    double hd[3], ho[3];   // second order: diagonal xx yy zz, off-diagonal xy xz yz
    double t[8];        // third order
    double u[RHO ? 9 : 3];   // RHO: W xx yy zz xy xz yz, correction; DRHODT: dipole rows
};

template <bool RHO>
__device__ __forceinline__ void acc_clear(Acc<RHO>& s) {
    s.a0 = s.aq = 0.0;
#pragma unroll
    for (int i = 0; i < 3; ++i) s.l[i] = s.hd[i] = s.ho[i] = 0.0;
#pragma unroll
    for (int i = 0; i < 8; ++i) s.t[i] = 0.0;
#pragma unroll
    for (int i = 0; i < (RHO ? 9 : 3); ++i) s.u[i] = 0.0;
}

// Squares of the separation and the radial powers of a pair, with the
// reference's floor r^2 >= 1e-20.
struct Radial {
    double xx, yy, zz;
    double P, d1, e2, e3;   // 2/r and its powers 3, 5, 7
};

__device__ __forceinline__ void radial_powers(double P, Radial& g) {
    const double rho = P * P;
    g.P = P;
    g.d1 = P * rho;
    g.e2 = rho * g.d1;
    g.e3 = rho * g.e2;
}

__device__ __forceinline__ void radial(double x, double y, double z, Radial& g) {
    g.xx = x * x;
    g.yy = y * y;
    g.zz = z * z;
    const double r2 = fmax(g.xx + g.yy + g.zz, 1.0e-20);   // one v_max_f64; r2 of finite separations is never NaN
    radial_powers(rsqrt2(r2), g);
}

// Record fields by index from the 12 double2 of a record.
__device__ __forceinline__ double rec_at(const double2* v, int i) { return (i & 1) ? v[i >> 1].y : v[i >> 1].x; }

// Potential and gradient rows of mass and quadrupole.
template <bool RHO>
__device__ __forceinline__ void add_gradient(const double2* v, double x, double y, double z, const Radial& g, double e2x,
    Acc<RHO>& s) {
    const double m0 = rec_at(v, 0);
    const double qxx = rec_at(v, 4), qxy = rec_at(v, 5), qxz = rec_at(v, 6), qyy = rec_at(v, 7), qyz = rec_at(v, 8);
    const double qzz = -(qxx + qyy);
    const double qx = fma(qxz, z, fma(qxy, y, qxx * x));
    const double qy = fma(qyz, z, fma(qyy, y, qxy * x));
    const double qz = fma(qzz, z, fma(qyz, y, qxz * x));
    const double sq = fma(qz, z, fma(qy, y, qx * x));
    s.a0 = fma(m0, g.P, s.a0);
    s.aq = fma(g.e2, sq, s.aq);
    const double e = fma(g.e3, sq, m0 * g.d1);
    s.l[0] = fma(-e2x, qx, fma(e, x, s.l[0]));
    s.l[1] = fma(-e2x, qy, fma(e, y, s.l[1]));
    s.l[2] = fma(-e2x, qz, fma(e, z, s.l[2]));
}

// z_a x_b + z_b x_a of the second-order sums (z_a x_a on the diagonal).
template <bool RHO>
__device__ __forceinline__ void add_second(double zx, double zy, double zz, double x, double y, double z, Acc<RHO>& s) {
    s.hd[0] = fma(zx, x, s.hd[0]);
    s.hd[1] = fma(zy, y, s.hd[1]);
    s.hd[2] = fma(zz, z, s.hd[2]);
    s.ho[0] = fma(zy, x, fma(zx, y, s.ho[0]));
    s.ho[1] = fma(zz, x, fma(zx, z, s.ho[1]));
    s.ho[2] = fma(zz, y, fma(zy, z, s.ho[2]));
}

// Quadratic monomials of the trace-free octupole forms, B_dbc x_b x_c / 2 =
// B_dxx h1 + B_dyy h2 + B_dxy xy + B_dxz xz + B_dyz yz.
struct Quadratic {
    double h1, h2, xy, xz, yz;
};

__device__ __forceinline__ Quadratic quadratic(double x, double y, double z, const Radial& g) {
    Quadratic q;
    const double h = 0.5 * g.zz;
    q.h1 = fma(0.5, g.xx, -h);
    q.h2 = fma(0.5, g.yy, -h);
    q.xy = x * y;
    q.xz = x * z;
    q.yz = y * z;
    return q;
}

// b: xxx xyy xzz xxy yyy yzz xxz yyz xyz
__device__ __forceinline__ void octupole_vector(const double* b, const Quadratic& q, double* v) {
    v[0] = fma(b[8], q.yz, fma(b[6], q.xz, fma(b[3], q.xy, fma(b[1], q.h2, b[0] * q.h1))));
    v[1] = fma(b[7], q.yz, fma(b[8], q.xz, fma(b[1], q.xy, fma(b[4], q.h2, b[3] * q.h1))));
    v[2] = fma(b[5], q.yz, fma(b[2], q.xz, fma(b[8], q.xy, fma(b[7], q.h2, b[6] * q.h1))));
}

// Partner part of the correction (and, with the potential a0, the partner's
// octupole on it): c += e3 (v + x tau x).
__device__ __forceinline__ void add_correction(const double* b, const double* tau, double x, double y, double z,
    const Quadratic& q, double e3, double* a0, double* c) {
    double v[3];
    octupole_vector(b, q, v);
    if (a0) *a0 = fma(e3, fma(v[2], z, fma(v[1], y, v[0] * x)), *a0);
    const double tx = fma(tau[2], z, fma(tau[1], y, tau[0] * x));
    c[0] = fma(e3, fma(x, tx, v[0]), c[0]);
    c[1] = fma(e3, fma(y, tx, v[1]), c[1]);
    c[2] = fma(e3, fma(z, tx, v[2]), c[2]);
}

// W += m0 e3 x x, the sums the target's own octupole meets.
__device__ __forceinline__ void add_w(double g3, const Radial& g, const Quadratic& q, double* w) {
    w[0] = fma(g3, g.xx, w[0]);
    w[1] = fma(g3, g.yy, w[1]);
    w[2] = fma(g3, g.zz, w[2]);
    w[3] = fma(g3, q.xy, w[3]);
    w[4] = fma(g3, q.xz, w[4]);
    w[5] = fma(g3, q.yz, w[5]);
}

// Third-order sums of the RHO kernels.
__device__ __forceinline__ void add_third(double g3, double x, double y, double z, const Radial& g, const Quadratic& q,
    double* t) {
    const double gx = g3 * x, gy = g3 * y, gz = g3 * z;
    t[0] = fma(gx, q.h1 - g.zz, t[0]);
    t[1] = fma(gx, q.h2, t[1]);
    t[2] = fma(gy, q.h1, t[2]);
    t[3] = fma(gy, q.h2 - g.zz, t[3]);
    t[4] = fma(gz, q.h1, t[4]);
    t[5] = fma(gz, q.h2, t[5]);
    t[6] = fma(gz, g.zz, t[6]);
    t[7] = fma(gx, q.yz, t[7]);
}

// The 8 cubic monomials that both the third-order sums and the octupole's
// potential of the DRHODT kernels use (twice those of add_third, but for the
// last two).
__device__ __forceinline__ void cubic_monomials(double x, double y, double z, const Radial& g, double* c) {
    const double h1 = g.xx - g.zz, h2 = g.yy - g.zz;
    c[0] = x * fma(-2.0, g.zz, h1);
    c[1] = x * h2;
    c[2] = y * h1;
    c[3] = y * fma(-2.0, g.zz, h2);
    c[4] = z * h1;
    c[5] = z * h2;
    c[6] = z * g.zz;
    c[7] = x * (y * z);
}

// Dipole rows of the DRHODT kernels (compute_kernel_non_rho, :374-389).  The
// reference subtracts the whole first row of the second-order tensor from
// each gradient component; kept as is.
__device__ __forceinline__ void add_dipole_rows(const double2* v, double x, double y, double z, const Radial& g,
    double px, Acc<false>& s) {
    s.aq = fma(g.d1, px, s.aq);
    const double es = -0.75 * (g.e2 * (x + y + z));
    s.u[0] = fma(rec_at(v, 1), fma(es, x, g.d1), s.u[0]);
    s.u[1] = fma(rec_at(v, 2), fma(es, y, g.d1), s.u[1]);
    s.u[2] = fma(rec_at(v, 3), fma(es, z, g.d1), s.u[2]);
}

// A partner record held in registers (24 doubles as 12 double2).
struct Rec {
    double2 v[12];
};

__device__ __forceinline__ void load_rec(const double* __restrict__ p, Rec& r) {
    const double2* p2 = reinterpret_cast<const double2*>(p);
#pragma unroll
    for (int i = 0; i < 12; ++i) r.v[i] = p2[i];
}

// One far M2L pair: partner record r onto the target at X.
template <bool RHO>
__device__ __forceinline__ void m2l_far_rec(const Rec& r, double X0, double X1, double X2, Acc<RHO>& s) {
    const double2* v = r.v;
    const double x = X0 - rec_at(v, kRecY), y = X1 - rec_at(v, kRecY + 1), z = X2 - rec_at(v, kRecY + 2);
    Radial g;
    radial(x, y, z, g);
    const double e2x = 1.6 * g.e2, m0 = rec_at(v, 0);
    add_gradient<RHO>(v, x, y, z, g, e2x, s);
    const double px = fma(rec_at(v, 3), z, fma(rec_at(v, 2), y, rec_at(v, 1) * x));
    const double k = fma(g.e3, px, m0 * g.e2);
    add_second<RHO>(fma(k, x, -(e2x * rec_at(v, 1))), fma(k, y, -(e2x * rec_at(v, 2))), fma(k, z, -(e2x * rec_at(v, 3))),
        x, y, z, s);
    const double g3 = m0 * g.e3;
    if constexpr (RHO) {
        const Quadratic q = quadratic(x, y, z, g);
        add_third(g3, x, y, z, g, q, s.t);
        add_w(g3, g, q, s.u);
        double b[9], tau[3];
#pragma unroll
        for (int i = 0; i < 9; ++i) b[i] = rec_at(v, 9 + i);
#pragma unroll
        for (int i = 0; i < 3; ++i) tau[i] = rec_at(v, 18 + i);
        add_correction(b, tau, x, y, z, q, g.e3, &s.a0, s.u + 6);
    } else {
        double c[8], o = 0.0;
        cubic_monomials(x, y, z, g, c);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            s.t[i] = fma(g3, c[i], s.t[i]);
            o = i == 0 ? rec_at(v, 9) * c[0] : fma(rec_at(v, 9 + i), c[i], o);
        }
        s.a0 = fma(g.e3, o, s.a0);
        add_dipole_rows(v, x, y, z, g, px, s);
    }
}

// The same pair from a record in global memory.
template <bool RHO>
__device__ __forceinline__ void m2l_far(const double* __restrict__ p, double X0, double X1, double X2, Acc<RHO>& s) {
    Rec r;
    load_rec(p, r);
    m2l_far_rec<RHO>(r, X0, X1, X2, s);
}

// One near pair with a monopole-only partner of mass mn at Y.
template <bool RHO>
__device__ __forceinline__ void m2l_near(double mn, double Y0, double Y1, double Y2, double X0, double X1,
    double X2, Acc<RHO>& s) {
    const double x = X0 - Y0, y = X1 - Y1, z = X2 - Y2;
    Radial g;
    radial(x, y, z, g);
    s.a0 = fma(mn, g.P, s.a0);
    const double e = mn * g.d1, k = mn * g.e2, g3 = mn * g.e3;
    s.l[0] = fma(e, x, s.l[0]);
    s.l[1] = fma(e, y, s.l[1]);
    s.l[2] = fma(e, z, s.l[2]);
    add_second<RHO>(k * x, k * y, k * z, x, y, z, s);
    if constexpr (RHO) {
        const Quadratic q = quadratic(x, y, z, g);
        add_third(g3, x, y, z, g, q, s.t);
        add_w(g3, g, q, s.u);
    } else {
        double c[8];
        cubic_monomials(x, y, z, g, c);
#pragma unroll
        for (int i = 0; i < 8; ++i) s.t[i] = fma(g3, c[i], s.t[i]);
    }
}

// The target's own octupole (its record trec, mass reciprocal inv_mc0) meets
// the sums W; c = partner part in, whole correction out (scale of acc_finish).
__device__ __forceinline__ void fold_w(const double* __restrict__ trec, double inv_mc0, const double* w, double* c) {
    const Quadratic q = {0.5 * (w[0] - w[2]), 0.5 * (w[1] - w[2]), w[3], w[4], w[5]};
    double b[9], v[3];
#pragma unroll
    for (int i = 0; i < 9; ++i) b[i] = trec[9 + i];
    octupole_vector(b, q, v);
    const double t0 = trec[18], t1 = trec[19], t2 = trec[20];
    v[0] = fma(t2, w[4], fma(t1, w[3], fma(t0, w[0], v[0])));
    v[1] = fma(t2, w[5], fma(t1, w[1], fma(t0, w[3], v[1])));
    v[2] = fma(t2, w[2], fma(t1, w[5], fma(t0, w[4], v[2])));
#pragma unroll
    for (int d = 0; d < 3; ++d) c[d] = fma(-inv_mc0, v[d], c[d]);
}

// Number of sums of a target after acc_fold.
constexpr int kFolded = 21;

// Folds a target's sums to the kFolded linear ones that partial sums of one
// target add up in: potential, gradient 3, second order 6, third order 8,
// correction 3 (zeros for DRHODT).
template <bool RHO>
__device__ __forceinline__ void acc_fold_expansion(const Acc<RHO>& s, double* f) {
    f[0] = fma(0.2, s.aq, s.a0);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        f[1 + i] = RHO ? s.l[i] : fma(-0.8, s.u[i], s.l[i]);
        f[4 + i] = s.hd[i];
        f[7 + i] = s.ho[i];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) f[10 + i] = s.t[i];
}

template <bool RHO>
__device__ __forceinline__ void acc_fold(const Acc<RHO>& s, const double* __restrict__ trec, double* f) {
    acc_fold_expansion<RHO>(s, f);
    if constexpr (RHO) {
        double c[3] = {s.u[6], s.u[7], s.u[8]};
        fold_w(trec, 1.0 / trec[0], s.u, c);
        f[18] = c[0];
        f[19] = c[1];
        f[20] = c[2];
    } else {
        f[18] = f[19] = f[20] = 0.0;
    }
}

constexpr double kCorrectionScale = -1.5;

// Expansion and correction of a target from its folded sums.
template <bool RHO>
__device__ __forceinline__ void acc_finish(const double* f, double* L, double* C) {
    L[0] = -0.5 * f[0];
#pragma unroll
    for (int i = 0; i < 3; ++i) L[1 + i] = 0.125 * f[1 + i];
    const double tr = (f[4] + f[5] + f[6]) * (1.0 / 3.0);
    L[4] = -(3.0 / 32.0) * (f[4] - tr);
    L[7] = -(3.0 / 32.0) * (f[5] - tr);
    L[9] = -(3.0 / 32.0) * (f[6] - tr);
    L[5] = -(3.0 / 64.0) * f[7];
    L[6] = -(3.0 / 64.0) * f[8];
    L[8] = -(3.0 / 64.0) * f[9];
    const double k = 15.0 / 128.0, h = RHO ? 2.0 : 1.0;
    const double* t = f + 10;
    // T with its xzz, yzz components zero, less the trace part
    const double xxx = h * t[0], xyy = h * t[1], xxy = h * t[2], yyy = h * t[3], xxz = h * t[4], yyz = h * t[5],
                 zzz = -2.0 * t[6];
    const double sx = 0.2 * (xxx + xyy), sy = 0.2 * (xxy + yyy), sz = 0.2 * (xxz + yyz + zzz);
    L[10] = k * (xxx - 3.0 * sx);
    L[11] = k * (xxy - sy);
    L[12] = k * (xxz - sz);
    L[13] = k * (xyy - sx);
    L[14] = k * t[7];
    L[15] = -k * sx;
    L[16] = k * (yyy - 3.0 * sy);
    L[17] = k * (yyz - sz);
    L[18] = -k * sy;
    L[19] = k * (zzz - 3.0 * sz);
#pragma unroll
    for (int d = 0; d < 3; ++d) C[d] = RHO ? kCorrectionScale * f[18 + d] : 0.0;
}

// One p2m pair: refined-neighbour multipole record r onto a leaf cell at X
// (compute_interaction_p2m_rho, monopole_kernel_templates.hpp:69-187): the
// potential and gradient rows, and the partner part of the correction.
template <bool RHO>
__device__ __forceinline__ void p2m_pair_rec(const Rec& r, double X0, double X1, double X2, Acc<RHO>& s) {
    const double2* v = r.v;
    const double x = X0 - rec_at(v, kRecY), y = X1 - rec_at(v, kRecY + 1), z = X2 - rec_at(v, kRecY + 2);
    Radial g;
    radial(x, y, z, g);
    add_gradient<RHO>(v, x, y, z, g, 1.6 * g.e2, s);
    if constexpr (RHO) {
        double b[9], tau[3];
#pragma unroll
        for (int i = 0; i < 9; ++i) b[i] = rec_at(v, 9 + i);
#pragma unroll
        for (int i = 0; i < 3; ++i) tau[i] = rec_at(v, 18 + i);
        add_correction(b, tau, x, y, z, quadratic(x, y, z, g), g.e3, &s.a0, s.u + 6);
    } else {
        double c[8];
        cubic_monomials(x, y, z, g, c);
        double o = rec_at(v, 9) * c[0];
#pragma unroll
        for (int i = 1; i < 8; ++i) o = fma(rec_at(v, 9 + i), c[i], o);
        s.a0 = fma(g.e3, o, s.a0);
        add_dipole_rows(v, x, y, z, g, fma(rec_at(v, 3), z, fma(rec_at(v, 2), y, rec_at(v, 1) * x)), s);
    }
}

// L0..3 and the correction of a leaf target from its p2m sums.
template <bool RHO>
__device__ __forceinline__ void p2m_finish(const Acc<RHO>& s, double* L, double* C) {
    L[0] = fma(-0.5, s.a0, -0.1 * s.aq);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        L[1 + i] = RHO ? 0.125 * s.l[i] : fma(-0.1, s.u[i], 0.125 * s.l[i]);
        C[i] = RHO ? kCorrectionScale * s.u[6 + i] : 0.0;
    }
}

// Multiplicity factors of the FP32 half of the mixed-precision pairs, folded
// into the FP32 moments of the mixed record: m4, m7, m9 halved and the octupole
// m10..m19 times {1,3,3,3,6,3,1,3,3,1}/6, so every term of its contraction is
// one fused multiply-add.
__host__ __device__ constexpr double record_scale(int c) {
    return (c == 4 || c == 7 || c == 9) ? 0.5
        : (c == 10 || c == 16 || c == 19) ? 1.0 / 6.0
        : (c == 14) ? 1.0
        : (c >= 11 && c <= 18) ? 0.5
        : 1.0;
}

// FP32 half of a mixed-precision far pair: the derivative tensor of -1/r at
// the separation (x, y, z), already rounded to FP32, and the 20-component
// contraction with the factor-scaled partner multipole m, accumulated into
// the FP32 partial sums Lf.  Returns the FP32 estimate of 1/r, from which the
// FP64 correction starts.
template <bool RHO>
__device__ __forceinline__ float m2l_fp32_core(float x, float y, float z, const float* m, float* Lf) {
    const float x00 = x * x, x11 = y * y, x22 = z * z;
    float r2 = fmaf(z, z, fmaf(y, y, x00));
    r2 = fmaxf(r2, 1.0e-20f);   // one v_max_f32; r2 of finite separations is never NaN
    const float ri = __builtin_amdgcn_rsqf(r2);
    const float r2inv = ri * ri;
    const float d1 = ri * r2inv;
    const float d2 = (-3.0f * r2inv) * d1;
    const float d3 = (-5.0f * r2inv) * d2;
    float D[20];
    D[0] = -ri;
    D[1] = x * d1;
    D[2] = y * d1;
    D[3] = z * d1;
    D[4] = fmaf(d2, x00, d1);
    D[5] = d2 * (x * y);
    D[6] = d2 * (x * z);
    D[7] = fmaf(d2, x11, d1);
    D[8] = d2 * (y * z);
    D[9] = fmaf(d2, x22, d1);
    const float d2x = d2 * x, d2y = d2 * y, d2z = d2 * z;
    const float d3x00 = d3 * x00, d3x11 = d3 * x11, d3x22 = d3 * x22;
    D[10] = fmaf(d3x00, x, 3.0f * d2x);
    D[11] = fmaf(d3x00, y, d2y);
    D[12] = fmaf(d3x00, z, d2z);
    D[13] = fmaf(d3x11, x, d2x);
    D[14] = (d3 * x) * (y * z);
    D[15] = fmaf(d3x22, x, d2x);
    D[16] = fmaf(d3x11, y, 3.0f * d2y);
    D[17] = fmaf(d3x11, z, d2z);
    D[18] = fmaf(d3x22, y, d2y);
    D[19] = fmaf(d3x22, z, 3.0f * d2z);
#pragma unroll
    for (int i = 0; i < 4; ++i) Lf[i] = fmaf(m[0], D[i], Lf[i]);
    if constexpr (!RHO) {
        Lf[0] = fmaf(-m[1], D[1], Lf[0]);
        Lf[0] = fmaf(-m[2], D[2], Lf[0]);
        Lf[0] = fmaf(-m[3], D[3], Lf[0]);
        Lf[1] = fmaf(-m[1], D[4] + D[5] + D[6], Lf[1]);
        Lf[2] = fmaf(-m[2], D[5] + D[7] + D[8], Lf[2]);
        Lf[3] = fmaf(-m[3], D[6] + D[8] + D[9], Lf[3]);
    }
    float l0 = Lf[0], l1 = Lf[1], l2 = Lf[2], l3 = Lf[3];
    l0 = fmaf(m[4], D[4], l0);   l1 = fmaf(m[4], D[10], l1);  l2 = fmaf(m[4], D[11], l2);  l3 = fmaf(m[4], D[12], l3);
    l0 = fmaf(m[5], D[5], l0);   l1 = fmaf(m[5], D[11], l1);  l2 = fmaf(m[5], D[13], l2);  l3 = fmaf(m[5], D[14], l3);
    l0 = fmaf(m[6], D[6], l0);   l1 = fmaf(m[6], D[12], l1);  l2 = fmaf(m[6], D[14], l2);  l3 = fmaf(m[6], D[15], l3);
    l0 = fmaf(m[7], D[7], l0);   l1 = fmaf(m[7], D[13], l1);  l2 = fmaf(m[7], D[16], l2);  l3 = fmaf(m[7], D[17], l3);
    l0 = fmaf(m[8], D[8], l0);   l1 = fmaf(m[8], D[14], l1);  l2 = fmaf(m[8], D[17], l2);  l3 = fmaf(m[8], D[18], l3);
    l0 = fmaf(m[9], D[9], l0);   l1 = fmaf(m[9], D[15], l1);  l2 = fmaf(m[9], D[18], l2);  l3 = fmaf(m[9], D[19], l3);
#pragma unroll
    for (int k = 10; k < 20; ++k) l0 = fmaf(-m[k], D[k], l0);
    Lf[0] = l0; Lf[1] = l1; Lf[2] = l2; Lf[3] = l3;
    static constexpr int kRowB[6][3] = {{10, 11, 12}, {11, 13, 14}, {12, 14, 15}, {13, 16, 17}, {14, 17, 18},
        {15, 18, 19}};
#pragma unroll
    for (int i = 0; i < 6; ++i) {
        float t = fmaf(m[0], D[4 + i], Lf[4 + i]);
        t = fmaf(-m[1], D[kRowB[i][0]], t);
        t = fmaf(-m[2], D[kRowB[i][1]], t);
        Lf[4 + i] = fmaf(-m[3], D[kRowB[i][2]], t);
    }
#pragma unroll
    for (int i = 10; i < 20; ++i) Lf[i] = fmaf(m[0], D[i], Lf[i]);
    return ri;
}

// FP64 half of a mixed-precision far pair (RHO): the angular-momentum
// correction at the FP64 separation, with 1/r refined from the FP32 estimate
// ri by one FP64 Newton step.  b7 and tau: the partner's scaled FP64 octupole
// without xzz and yzz, which its vanishing traces give.  Adds to the sums
// W (s.u[0..5]) and the partner part of the correction (s.u[6..8]).
__device__ __forceinline__ void mixed_correction(double x, double y, double z, float ri, double m0, const double* b7,
    const double* tau, double* u) {
    Radial g;
    g.xx = x * x;
    g.yy = y * y;
    g.zz = z * z;
    const double r2 = fmax(g.xx + g.yy + g.zz, 1.0e-20);
    const double y0 = (double)ri;
    radial_powers(y0 * fma(-(r2 * y0), y0, 3.0), g);
    const Quadratic q = quadratic(x, y, z, g);
    add_w(m0 * g.e3, g, q, u);
    const double b[9] = {b7[0], b7[1], -(b7[0] + b7[1]), b7[2], b7[3], -(b7[2] + b7[3]), b7[4], b7[5], b7[6]};
    add_correction(b, tau, x, y, z, q, g.e3, nullptr, u + 6);
}

// Mixed-precision partner record (192 bytes, 12 chunks of 16), written by the
// staging kernel beside the FP64 record for mixed-precision plans: chunks 0-4
// the factor-scaled multipole m0..m19 rounded to FP32, chunk 5 (Y0, Y1),
// chunk 6 (Y2, m0), chunks 7-11 the FP64 octupole fields of the FP64 record
// (xxx xyy xxy yyy xxz yyz xyz, trace 3).
constexpr int kRecmY01 = 5;
constexpr int kRecmY2M0 = 6;
constexpr int kRecmOct = 7;

// Mixed precision far pair from a mixed-precision record r (12 double2, in
// LDS or registers): the separation is formed in FP64 and rounded to FP32 for
// the derivative tensor and the 20-component contraction, which accumulate
// into the FP32 partial sums Lf of the current image (at most 8 pairs, added
// to the FP64 expansion by the caller).  The correction stays FP64, in u.
template <bool RHO>
__device__ __forceinline__ void m2l_far_m32(const double2* __restrict__ r, double X0, double X1, double X2, float* Lf,
    double* u) {
    const double2 y01 = r[kRecmY01], y2m = r[kRecmY2M0];
    const double xd = X0 - y01.x, yd = X1 - y01.y, zd = X2 - y2m.x;
    float m[20];
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        const float4 v = __builtin_bit_cast(float4, r[i]);
        m[4 * i] = v.x;
        m[4 * i + 1] = v.y;
        m[4 * i + 2] = v.z;
        m[4 * i + 3] = v.w;
    }
    const float ri = m2l_fp32_core<RHO>((float)xd, (float)yd, (float)zd, m, Lf);
    if constexpr (RHO) {
        double o[10];
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            const double2 v = r[kRecmOct + k];
            o[2 * k] = v.x;
            o[2 * k + 1] = v.y;
        }
        mixed_correction(xd, yd, zd, ri, y2m.y, o, o + 7, u);
    }
}

// ---------------------------------------------------------------------------
// Kernel arguments
// ---------------------------------------------------------------------------
struct StageArgs {
    const double* M;        // [nslots][512][20]
    const double* com;      // [nslots][512][3]
    const double* mon;      // [nslots][512]
    const int32_t* kind;    // [nslots]
    const double* fxbase;   // [nslots][3] frame origin for leaf-cell centres
    const int32_t* foff;    // [nslots][3] frame offset of the slot's cell (0,0,0)
    double* rec;            // [nslots][512][24]
    double* recm;           // mixed-precision records [nslots][512][24], or null
    const int32_t* list;    // slots to stage (null: all nslots)
    double dx;
    int32_t nslots;         // slots to stage (length of list when given)
    int32_t rho;            // record form: RHO or DRHODT octupole fields
};

// Levels of one stage_records launch, and the most slots (of 4 workgroups each)
// of levels that share one: four workgroups a CU, one round of the chip.
constexpr int kStageLevels = 6;
constexpr int kStageTogether = 256;
struct StageGroup {
    StageArgs a[kStageLevels];
};

struct LevelArgs {
    const double* rec;      // partner records
    const double* com;      // input centres of mass (leaf targets)
    const double* xbase;    // [nslots][3] and cell size, whole-tree solves
    double dx;
    double* L;
    double* Lc;
    const int32_t* nbr;     // [nslots][27]
    const int32_t* kind;    // [nslots]
    const int2* items;      // (slot, flags)
    const Tables* tab;
    const uint64_t* mixbits;   // per coarse offset: byte k, bit j = far pair evaluated in FP32
    // mixed-precision plans, lane mapping 7: the mixed-precision records, and
    // the entries of the far schedule (Tables::sched) in the order they run,
    // the first mix_n64 in FP64 and then those whose offset has every far pair
    // evaluated in FP32
    const double* recm;
    const int32_t* mixorder;
    int32_t mix_n64;
    const double* mon;      // [nslots][512] monopoles (p2p window of leaf targets)
    // leaf targets with refined neighbours: the p2m sums (L0..3, L_c, 0) of
    // each cell, [p2m item][512][8], written by p2m_kernel for leaf_kernel
    double* p2m_out;
    // its work lists (P2mPacks)
    const int32_t* p2m_hdr;
    const int32_t* p2m_units;
    const int32_t* p2m_idx;
    const int32_t* p2m_di;
    // Whole-tree solves (l2l != 0): the level's expansions are written, not
    // accumulated, as interactions + the parent cell's final expansion
    // re-expanded about the cell's centre of mass (and L_c + the parent's
    // L_c); leaf cells also get phi and g.  parent / octant per slot, pL /
    // pLc / pcom of the level above (null on level 0).
    const int32_t* parent;
    const int32_t* octant;
    const double* pL;
    const double* pLc;
    const double* pcom;
    double* g;
    double G;
    int32_t l2l;
    int32_t correct_am;
    int32_t overwrite;      // outside whole-tree solves: L is written, not accumulated
    int32_t leaf_rows;      // whole-tree solves: 0 = leaf cells get g (and L_c) only, no L rows
    // persistent form of lane mapping 7: 8 work counters, one per XCD
    // (cleared by queue_reset before each launch)
    uint32_t* queue;
    // variant 704 on small levels: workgroups per coarse block (0 or 1: the
    // plain form), and their folded sums
    // [item * 8 + block][part][kFolded][64]
    double* wide_sums;
    int32_t parts;
    int32_t nitems;
    int32_t item0;          // first item of this launch
    int32_t leaf0;          // first leaf item
    double inv_dx;
    double neg_inv_dx;
};

struct RootArgs {
    const double* rec;      // records of the root slot (512 x 24)
    const Tables* tab;
    double* partial;        // [kRootChunks][512][24]
};

// tree_sums_kernel: the root's pairs, and per level the workgroups of its sums
// (items x 8 x parts) and of its p2m (packs).
struct TreeSums {
    RootArgs root;
    int32_t sums[kStageLevels];
    int32_t packs[kStageLevels];
    LevelArgs a[kStageLevels];
};

// Leaf targets of up to kLeafLevels levels, one after another.
constexpr int kLeafLevels = 4;
struct LeafGroup {
    int32_t n[kLeafLevels];
    LevelArgs a[kLeafLevels];
};

struct RootReduceArgs {
    const double* partial;
    double* L;              // [512][20]
    double* Lc;             // [512][3]
    int32_t nchunks;
    int32_t rho;
    int32_t overwrite;      // whole-tree solve: L is written, not accumulated
};

// ---------------------------------------------------------------------------
// Tree passes: expansion shifts of taylor<4> (octotiger/taylor.hpp:222-311)
// ---------------------------------------------------------------------------
__host__ __device__ constexpr int tmap2(int a, int b) {
    const int i = a < b ? a : b, j = a < b ? b : a;
    return 4 + i * 3 - (i * (i - 1)) / 2 + (j - i);
}

__host__ __device__ constexpr int tmap3(int a, int b, int c) {
    const int t[27] = {10, 11, 12, 11, 13, 14, 12, 14, 15, 11, 13, 14, 13, 16, 17, 14, 17, 18,
        12, 14, 15, 14, 17, 18, 15, 18, 19};
    return t[a * 9 + b * 3 + c];
}

// taylor::operator>>= : B = A moved from its centre by X (X = old - new centre).
// Each order takes the finished lower one as a factor: with T_ac = A_ac + A_a X_c,
//   B_a = A_a + A X_a,  B_ab = A_ab + A_a X_b + X_a B_b,
//   B_abc = A_abc + A_ab X_c + X_b T_ac + X_a B_bc,
// 51 fused multiply-adds, where the expanded sums take about 190 operations.
__device__ __forceinline__ void multipole_shift(const double* A, const double* X, double* B) {
    B[0] = A[0];
#pragma unroll
    for (int a = 0; a < 3; ++a) B[1 + a] = fma(A[0], X[a], A[1 + a]);
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int b = a; b < 3; ++b) B[tmap2(a, b)] = fma(X[a], B[1 + b], fma(A[1 + a], X[b], A[tmap2(a, b)]));
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int c = a; c < 3; ++c) {
            const double t = fma(A[1 + a], X[c], A[tmap2(a, c)]);
#pragma unroll
            for (int b = a; b <= c; ++b)
                B[tmap3(a, b, c)] =
                    fma(X[a], B[tmap2(b, c)], fma(X[b], t, fma(A[tmap2(a, b)], X[c], A[tmap3(a, b, c)])));
        }
}

// multipole_shift for A = (m, 0, ..., 0), a cell that holds only its mass:
// the terms of the general form that remain, each formed in the same order.
__device__ __forceinline__ void monopole_shift(double m, const double* X, double* B) {
    B[0] = m;
#pragma unroll
    for (int a = 0; a < 3; ++a) B[1 + a] = m * X[a];
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int b = a; b < 3; ++b) B[tmap2(a, b)] = m * X[a] * X[b];
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int b = a; b < 3; ++b)
#pragma unroll
            for (int c = b; c < 3; ++c) B[tmap3(a, b, c)] = m * X[a] * X[b] * X[c];
}

// taylor::operator<<= : B = local expansion A re-expanded at +X.  With w_ab =
// A_abc X_c, v_a = w_ab X_b and q_a = A_ab X_b,
//   B_ab = A_ab + w_ab,  B_a = A_a + q_a + v_a / 2,
//   B = A + X_a (A_a + q_a / 2 + v_a / 6),
// 57 operations, where the expanded sums take about 280.
__device__ __forceinline__ void local_shift(const double* A, const double* X, double* B) {
    double w[10];   // by tmap2
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int b = a; b < 3; ++b)
            w[tmap2(a, b)] =
                fma(A[tmap3(a, b, 2)], X[2], fma(A[tmap3(a, b, 1)], X[1], A[tmap3(a, b, 0)] * X[0]));
    B[0] = A[0];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const double v = fma(w[tmap2(a, 2)], X[2], fma(w[tmap2(a, 1)], X[1], w[tmap2(a, 0)] * X[0]));
        const double q = fma(A[tmap2(a, 2)], X[2], fma(A[tmap2(a, 1)], X[1], A[tmap2(a, 0)] * X[0]));
        B[1 + a] = fma(0.5, v, A[1 + a] + q);
        B[0] = fma(fma(1.0 / 6.0, v, fma(0.5, q, A[1 + a])), X[a], B[0]);
    }
#pragma unroll
    for (int i = 4; i < 10; ++i) B[i] = A[i] + w[i];
#pragma unroll
    for (int i = 10; i < 20; ++i) B[i] = A[i];
}

// parent cell holding coarse cell (ip, jp, kp) of a node in octant o
// (node_server::compute_fmm, src/node_server.cpp:613-636, 756-768)
__host__ __device__ __forceinline__ int parent_cell(int o, int ip, int jp, int kp) {
    return (ip + 4 * (o & 1)) * 64 + (jp + 4 * ((o >> 1) & 1)) * 8 + (kp + 4 * ((o >> 2) & 1));
}

struct M2MArgs {
    const double* M;        // [n][512][20] this level
    double* com;            // [n][512][3]  this level (leaf centres written for RHO)
    const double* mon;      // [n][512]
    const int32_t* parent;
    const int32_t* octant;
    const int32_t* order;   // [n] nodes of the level: nleaf leaves, then the refined ones
    const double* xbase;    // [n][3]
    double* pM;             // parent level [np][512][20]
    double* pcom;           // parent level [np][512][3]
    double dx;
    int32_t nleaf;
};

}   // namespace octofmm
