// Device kernels of small_strain_J2_plasticity_damage (viscoplastic J2 with nonlinear kinematic
// hardening and Lemaitre-Chaboche scalar damage): the predictor, one thread per quadrature point,
// and the return map of the points that yield, four lanes per point.
//
// Reference behaviour (paths relative to the neon repository root):
//   update_internal_variables  src/constitutive/mechanics/solid/small_strain_J2_plasticity_damage.cpp:34-120
//   perform_radial_return      :122-250 (16 unknowns: plastic and damage multipliers, kinetic
//                              stress (6), kinetic back stress (6), damage, energy release rate)
//   yield functions            :252-265; energy release rate :267-285
//   material constants         src/material/isotropic_elastic_plastic_damage.cpp:9-45
//   Voigt / Mandel conventions src/numeric/tensor_operations.hpp:207-214, 373-376, 425-439, 509-515
//
// The return map's 16 x 16 Newton systems are solved by Gaussian elimination with complete
// pivoting (the algorithm of Eigen's FullPivLU the reference calls), and the tangent takes the
// 6 x 6 stress block of the last iteration's inverse from one factorisation and six solves.  A
// point's system (2 KB, indexed by its pivots) is in LDS, 64 points per workgroup side by side, its
// rows dealt to four lanes that hold the point's other values alike.  In private memory, one thread
// per point, the systems of a workgroup went through the caches and 22 K points filled a third of
// the compute units with one wavefront per SIMD: 3.65 ms per update (14 x 13 x 15 cells, all
// yielding) against 0.71 ms here,
// bound by the chain of 16 dependent pivots (an LDS scan each) per iteration.
// History (plastic strain, effective plastic strain, back stress, damage) is updated in place
// at every call, as neon does; the tangent is general (36 coefficients, row-major 6 x 6).
#pragma once

#include "element_kernels.hpp"

namespace neon_amd
{
constexpr int kGeneralCoefs = 36;

// isotropic_elastic_plastic_damage constants: kinematic hardening modulus C, softening multiplier
// gamma, plasticity viscous denominator s_p and exponent n_p, damage viscous denominator s_d and
// exponent n_d
struct damage_constants
{
    double C, gamma, sp, np, sd, nd;
};

// J2 damage state beyond the J2 arrays of qp_state (stride Q): back stress 6 (tensor components
// 11, 22, 33, 23, 13, 12), damage 1, energy release rate 1
struct damage_state
{
    double* beta;
    double* dmg;
    double* energy;
};

namespace damage_detail
{
// kinetic Voigt (11, 22, 33, 23, 13, 12) <-> 3 x 3 row-major
__device__ inline void kin(const double* a, double* v)
{
    v[0] = a[0], v[1] = a[4], v[2] = a[8], v[3] = a[5], v[4] = a[2], v[5] = a[1];
}
__device__ inline void kin_from(const double* v, double* a)
{
    a[0] = v[0], a[4] = v[1], a[8] = v[2];
    a[5] = a[7] = v[3];
    a[2] = a[6] = v[4];
    a[1] = a[3] = v[5];
}
// C * kinematic(e) for the isotropic C_e (lambda, G) scaled by s: the stress-like vector of
// compute_stress_like_vector_voigt (:280-285)
__device__ inline void ce_times(double lam, double G, double s, const double* e, double* v)
{
    double const tr = e[0] + e[4] + e[8];
    v[0] = s * (lam * tr + 2.0 * G * e[0]);
    v[1] = s * (lam * tr + 2.0 * G * e[4]);
    v[2] = s * (lam * tr + 2.0 * G * e[8]);
    v[3] = s * G * 2.0 * e[5];
    v[4] = s * G * 2.0 * e[2];
    v[5] = s * G * 2.0 * e[1];
}
__device__ inline double ddot9(const double* a, const double* b)
{
    double s = 0.0;
    for (int i = 0; i < 9; ++i) s += a[i] * b[i];
    return s;
}
__device__ inline double mandel_factor(int i, int j)
{
    if (i >= 3 && j >= 3) return 2.0;
    if ((i < 3) != (j < 3)) return 1.4142135623730951; // sqrt(2)
    return 1.0;
}
// the isotropic elastic moduli (isotropic_linear_elasticity.cpp:55-67) entry (i, j)
__device__ inline double ce_entry(double lam, double G, int i, int j)
{
    if (i < 3 && j < 3) return lam + (i == j ? 2.0 * G : 0.0);
    return i == j ? G : 0.0;
}

// residual and the nonzero entries put(i, j, value) of the 16 x 16 Jacobian of the return map at y
template <typename PUT>
__device__ __forceinline__ void system(double kp, double kd, double G, double lam, double sy, double E,
                                       const damage_constants& dc, double dt,
                                       const double* eps_e_t, const double* beta_t, double dmg_t, const double* y, double* res,
                                       PUT put)
{
    double const s32 = sqrt(1.5);
    double const dlp = y[0], dld = y[1];
    double sig[9], bet[9];
    kin_from(y + 2, sig);
    kin_from(y + 8, bet);
    double const D = y[14], omD = 1.0 - D, Y = y[15];
    double dev[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) dev[i] = sig[i] - bet[i];
    double const m = (dev[0] + dev[4] + dev[8]) / 3.0;
    dev[0] -= m, dev[4] -= m, dev[8] -= m;
    double const nd = sqrt(ddot9(dev, dev));
    double const vm = s32 * nd;
    double N[9], ee[9], dNdD[9], dfdb[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) N[i] = s32 * dev[i] / (nd * omD);
#pragma unroll
    for (int i = 0; i < 9; ++i) ee[i] = eps_e_t[i] - dlp * N[i];
    double const fp = fmax(0.0, vm / omD + 0.5 * dc.gamma / dc.C * ddot9(bet, bet) - sy);
    double const fd = fmax(0.0, Y - sy * sy / (2.0 * E));
#pragma unroll
    for (int i = 0; i < 9; ++i) dfdb[i] = dc.gamma / dc.C * bet[i] - N[i];
#pragma unroll
    for (int i = 0; i < 9; ++i) dNdD[i] = N[i] / omD;
    double const dfdD = vm / (omD * omD);
    // dN/dsigma in kinetic Voigt: sqrt(3/2) / (1 - D) (P / |dev| - dev (x) dev / |dev|^3)
    double dv[6];
    kin(dev, dv);
    double const a1 = s32 / omD / nd, a2 = s32 / omD / (nd * nd * nd);
    auto dNds = [&](int i, int j) {
        double p = 0.0;
        if (i < 3 && j < 3)
            p = i == j ? 2.0 / 3.0 : -1.0 / 3.0;
        else if (i == j)
            p = 1.0;
        return a1 * p - a2 * dv[i] * dv[j];
    };
    put(0, 0, 1.0);
    put(1, 1, 1.0);
    put(14, 14, 1.0);
    put(15, 15, 1.0);
    double Cee[6], Ceem[9];
    ce_times(lam, G, 1.0, ee, Cee);
    kin_from(Cee, Ceem);
    res[0] = dlp - kp * pow(fp, dc.np) * dt;
    res[1] = dld - kd * pow(fd, dc.nd) * dt;
    {
        double const tr = ee[0] + ee[4] + ee[8];
        double t[9], v[6];
#pragma unroll
        for (int i = 0; i < 9; ++i) t[i] = sig[i] - omD * ((i % 4 == 0 ? lam * tr : 0.0) + 2.0 * G * ee[i]);
        kin(t, v);
#pragma unroll
        for (int i = 0; i < 6; ++i) res[2 + i] = v[i];
#pragma unroll
        for (int i = 0; i < 9; ++i) t[i] = bet[i] - beta_t[i] - dlp * (dc.C * N[i] - dc.gamma * bet[i]);
        kin(t, v);
#pragma unroll
        for (int i = 0; i < 6; ++i) res[8 + i] = v[i];
    }
    res[14] = D - dmg_t - dld;
    res[15] = Y - 0.5 * ddot9(ee, Ceem);
    double const cfp = -dc.np * kp * pow(fp, dc.np - 1.0) * dt;
    {
        double v[6], w[6];
        kin(N, v);
        kin(dfdb, w);
#pragma unroll
        for (int j = 0; j < 6; ++j)
        {
            put(0, 2 + j, cfp * v[j]);
            put(0, 8 + j, cfp * w[j]);
        }
    }
    put(0, 14, cfp * dfdD);
    put(1, 15, -dc.nd * kd * pow(fd, dc.nd - 1.0) * dt);
    {
        double v[6];
        ce_times(lam, G, omD, N, v);
#pragma unroll
        for (int i = 0; i < 6; ++i) put(2 + i, 0, v[i]);
    }
    // mandel((1 - D) C_e) mandel(dlp dN/dsigma); the back-stress block is its negative
#pragma unroll
    for (int i = 0; i < 6; ++i)
#pragma unroll
        for (int j = 0; j < 6; ++j)
        {
            double p = 0.0;
#pragma unroll
            for (int k = 0; k < 6; ++k)
                p += omD * ce_entry(lam, G, i, k) * mandel_factor(i, k) * dlp * dNds(k, j) * mandel_factor(k, j);
            put(2 + i, 2 + j, (i == j ? 1.0 : 0.0) + p);
            put(2 + i, 8 + j, -p);
        }
    {
        double t[9], v[6];
#pragma unroll
        for (int i = 0; i < 9; ++i) t[i] = omD * dlp * dNdD[i] + ee[i];
        ce_times(lam, G, 1.0, t, v);
#pragma unroll
        for (int i = 0; i < 6; ++i) put(2 + i, 14, v[i]);
#pragma unroll
        for (int i = 0; i < 9; ++i) t[i] = dc.gamma * bet[i] - dc.C * N[i];
        kin(t, v);
#pragma unroll
        for (int i = 0; i < 6; ++i) put(8 + i, 0, v[i]);
#pragma unroll
        for (int i = 0; i < 9; ++i) t[i] = -dc.C * dlp * dNdD[i];
        kin(t, v);
#pragma unroll
        for (int i = 0; i < 6; ++i) put(8 + i, 14, v[i]);
    }
#pragma unroll
    for (int i = 0; i < 6; ++i)
#pragma unroll
        for (int j = 0; j < 6; ++j)
        {
            double const d = dNds(i, j);
            put(8 + i, 2 + j, -dc.C * dlp * d);
            put(8 + i, 8 + j, (i == j ? 1.0 + dc.gamma * dlp : 0.0) + dc.C * dlp * d);
        }
    put(14, 1, -1.0);
    put(15, 0, ddot9(N, Ceem));
#pragma unroll
    for (int j = 0; j < 6; ++j)
    {
        double t = 0.0;
#pragma unroll
        for (int k = 0; k < 6; ++k) t += dNds(j, k) * Cee[k];
        put(15, 2 + j, dlp * t);
        put(15, 8 + j, -dlp * t);
    }
    put(15, 14, dlp * ddot9(dNdD, Ceem));
}

// The systems of a workgroup in LDS: entry (i, j) of point q at a[(16 i + j) 64 + q], its right-hand
// side or solution at r / x[64 i + q].  Lane sub (0..3) of a point owns the rows i with i % 4 = sub.
constexpr int kDamagePoints = 64; // per workgroup
struct damage_lds
{
    double a[256 * kDamagePoints];
    double r[16 * kDamagePoints];
    double x[16 * kDamagePoints];
};

// The four lanes' LDS accesses so far come before those that follow (one wavefront holds all four and
// its LDS accesses execute in order; this keeps the compiler to that order)
__device__ inline void lanes_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// In-place LU with complete pivoting of a point's system: rowp / colp receive the exchanges, four bits
// each; multipliers below the diagonal.  false when a pivot is exactly zero.
__device__ bool lu_full(double* A, int sub, uint64_t& rowp, uint64_t& colp)
{
    auto at = [&](int i, int j) -> double& { return A[(i * 16 + j) * kDamagePoints]; };
    rowp = 0;
    colp = 0xfedcba9876543210ull;
    for (int k = 0; k < 16; ++k)
    {
        // the first largest entry in row-major order
        double big = -1.0;
        int where = 256;
        for (int i = k + ((sub - k) & 3); i < 16; i += 4)
            for (int j = k; j < 16; ++j)
            {
                double const v = fabs(at(i, j));
                if (v > big)
                {
                    big = v;
                    where = i * 16 + j;
                }
            }
#pragma unroll
        for (int m = 1; m <= 2; m <<= 1)
        {
            double const ob = __shfl_xor(big, m, 64);
            int const ow = __shfl_xor(where, m, 64);
            if (ob > big || (ob == big && ow < where))
            {
                big = ob;
                where = ow;
            }
        }
        // no entry compared greater (all are NaN): the diagonal
        int const pr = where < 256 ? where >> 4 : k, pc = where < 256 ? where & 15 : k;
        if (big == 0.0) return false;
        rowp |= uint64_t(pr) << (4 * k);
        lanes_sync();
        // the trailing columns only: each stored multiplier stays with the position it was
        // computed at, so lu_solve can apply exchanges and eliminations step by step
        if (pr != k)
            for (int j = k + ((sub - k) & 3); j < 16; j += 4)
            {
                double const t = at(k, j);
                at(k, j) = at(pr, j);
                at(pr, j) = t;
            }
        lanes_sync();
        if (pc != k)
        {
            for (int i = sub; i < 16; i += 4)
            {
                double const t = at(i, k);
                at(i, k) = at(i, pc);
                at(i, pc) = t;
            }
            uint64_t const d = ((colp >> (4 * k)) ^ (colp >> (4 * pc))) & 15u;
            colp ^= d << (4 * k) | d << (4 * pc);
        }
        lanes_sync();
        double const pivot = at(k, k);
        for (int i = k + 1 + ((sub - k - 1) & 3); i < 16; i += 4)
        {
            double const f = at(i, k) / pivot;
            at(i, k) = f;
            if (f == 0.0) continue;
            for (int j = k + 1; j < 16; ++j) at(i, j) -= f * at(k, j);
        }
        lanes_sync();
    }
    return true;
}

// x = A^-1 r from lu_full's factors (r is overwritten)
__device__ void lu_solve(const double* A, int sub, uint64_t rowp, uint64_t colp, double* r, double* x)
{
    auto at = [&](int i, int j) { return A[(i * 16 + j) * kDamagePoints]; };
    lanes_sync();
    for (int k = 0; k < 16; ++k)
    {
        int const pr = int(rowp >> (4 * k)) & 15;
        double const rk = r[pr * kDamagePoints], old = r[k * kDamagePoints];
        lanes_sync();
        if (sub == 0 && pr != k)
        {
            r[k * kDamagePoints] = rk;
            r[pr * kDamagePoints] = old;
        }
        lanes_sync();
        for (int i = k + 1 + ((sub - k - 1) & 3); i < 16; i += 4)
        {
            double const f = at(i, k);
            if (f != 0.0) r[i * kDamagePoints] -= f * rk;
        }
        lanes_sync();
    }
    for (int k = 15; k >= 0; --k)
    {
        double const yk = r[k * kDamagePoints] / at(k, k);
        if (sub == 0) x[(int(colp >> (4 * k)) & 15) * kDamagePoints] = yk;
        for (int i = sub; i < k; i += 4) r[i * kDamagePoints] -= at(i, k) * yk;
        lanes_sync();
    }
}
} // namespace damage_detail

namespace damage_detail
{
// A point's elastic predictor (with damage) from its committed history: strain, stress, relative von
// Mises stress, energy and the two yield functions (stress_routines.hpp:38-44)
struct predictor
{
    double lam, G, sy, Emod;
    double ep[9], beta[9], ee[9], sig[9];
    double dmg, eb, vm, energy;
    bool elastic;
};
__device__ inline double von_mises_rel(const double* s, const double* b)
{
    double d[9];
    for (int i = 0; i < 9; ++i) d[i] = s[i] - b[i];
    double const m = (d[0] + d[4] + d[8]) / 3.0;
    d[0] -= m, d[4] -= m, d[8] -= m;
    return sqrt(1.5) * sqrt(ddot9(d, d));
}
__device__ __forceinline__ void predict(predictor& t, const double* H, element_params prm, qp_state const& st,
                                        damage_state const& ds, damage_constants const& dc, int64_t e, int64_t qp)
{
    int64_t const Q = st.Q;
    double const bulk = prm.p[4 * e], G = prm.p[4 * e + 1], sy = prm.p[4 * e + 2];
    double const lam = bulk - 2.0 * G / 3.0;
    t.lam = lam, t.G = G, t.sy = sy;
    t.Emod = 9.0 * bulk * G / (3.0 * bulk + G); // isotropic_elastic_property.hpp:16
    double ev[6];
    for (int k = 0; k < 6; ++k) ev[k] = st.eps_p[k * Q + qp];
    kin_from(ev, t.ep);
    for (int k = 0; k < 6; ++k) ev[k] = ds.beta[k * Q + qp];
    kin_from(ev, t.beta);
    t.dmg = ds.dmg[qp];
    t.eb = st.ebar[qp];
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j) t.ee[i * 3 + j] = 0.5 * (H[i * 3 + j] + H[j * 3 + i]) - t.ep[i * 3 + j];
    double const tr = t.ee[0] + t.ee[4] + t.ee[8];
    for (int i = 0; i < 9; ++i) t.sig[i] = (1.0 - t.dmg) * ((i % 4 == 0 ? lam * tr : 0.0) + 2.0 * G * t.ee[i]);
    t.vm = von_mises_rel(t.sig, t.beta);
    double v[6], m[9];
    ce_times(lam, G, 1.0, t.ee, v);
    kin_from(v, m);
    t.energy = 0.5 * ddot9(t.ee, m);
    double const fp0 = t.vm / (1.0 - t.dmg) + 0.5 * dc.gamma / dc.C * ddot9(t.beta, t.beta) - sy;
    double const fd0 = t.energy - sy * sy / (2.0 * t.Emod);
    t.elastic = fp0 <= 0.0 && fd0 <= 0.0;
}
__device__ inline void store_stress(qp_state const& st, damage_state const& ds, int64_t qp, const double* sig, double vm,
                                    double energy, uint32_t* status)
{
    ds.energy[qp] = energy;
    st.vm[qp] = vm;
    double sv[6];
    kin(sig, sv);
    bool finite = true;
    for (int k = 0; k < 6; ++k)
    {
        st.sigma[k * st.Q + qp] = sv[k];
        finite = finite && isfinite(sv[k]);
    }
    if (!finite) atomicOr(status, STATUS_NAN);
}
} // namespace damage_detail

// One thread per quadrature point (qp = 8 e + l); the per-element parameters are (K, G, yield
// stress, unused).  Elastic points are done; the others' numbers go to yield[1 ...], their count to
// yield[0] (zero before), in any order.
__global__ __launch_bounds__(kBlock) void damage_predict_kernel(int32_t E, const int32_t* __restrict__ conn,
                                                                const double* __restrict__ X,
                                                                const double* __restrict__ u, element_params prm,
                                                                qp_state st, damage_state ds, damage_constants dc,
                                                                uint32_t* __restrict__ status, int32_t* yield)
{
    using namespace damage_detail;
    int64_t const qp = int64_t(blockIdx.x) * kBlock + threadIdx.x;
    if (qp >= 8ll * E) return;
    int64_t const e = qp >> 3;
    double H[9], F[9];
    qp_kinematics(conn, X, u, e, int(qp & 7), H, F);
    double const Jdet = det3(F);
    st.detF[qp] = Jdet;
    if (signbit(Jdet)) atomicOr(status, STATUS_NEGATIVE_JACOBIAN);
    predictor t;
    predict(t, H, prm, st, ds, dc, e, qp);
    // the wavefront's yielding points take consecutive places (one atomic)
    uint64_t const mask = __ballot(!t.elastic);
    if (mask)
    {
        int const lane = threadIdx.x & 63, leader = __ffsll((unsigned long long)mask) - 1;
        int base = 0;
        if (lane == leader) base = atomicAdd(yield, int(__popcll(mask)));
        base = __shfl(base, leader, 64);
        if (!t.elastic) yield[1 + base + __popcll(mask & ((1ull << lane) - 1))] = int32_t(qp);
    }
    if (!t.elastic) return;
    for (int i = 0; i < 6; ++i)
        for (int j = 0; j < 6; ++j) st.coef[int64_t(i * 6 + j) * st.Q + qp] = ce_entry(t.lam, t.G, i, j);
    store_stress(st, ds, qp, t.sig, t.vm, t.energy, status);
}

// perform_radial_return of the points listed in yield: four lanes per point, 64 points per workgroup
// at a time.  kp, kd: the constants' s^-n powers.
__global__ __launch_bounds__(256, 1) void damage_return_kernel(const int32_t* __restrict__ conn,
                                                               const double* __restrict__ X,
                                                               const double* __restrict__ u, element_params prm,
                                                               qp_state st, damage_state ds, damage_constants dc,
                                                               double kp, double kd, double dt,
                                                               uint32_t* __restrict__ status,
                                                               const int32_t* __restrict__ yield)
{
    using namespace damage_detail;
    extern __shared__ __align__(16) unsigned char damage_smem[];
    damage_lds& lds = *reinterpret_cast<damage_lds*>(damage_smem);
    int const q = threadIdx.x >> 2, sub = threadIdx.x & 3;
    double* const A = lds.a + q;
    double* const r = lds.r + q;
    double* const x = lds.x + q;
    int32_t const count = yield[0];
    int64_t const Q = st.Q;
    for (int32_t n = int32_t(blockIdx.x) * kDamagePoints + q; n < count; n += int32_t(gridDim.x) * kDamagePoints)
    {
        int64_t const qp = yield[1 + n];
        int64_t const e = qp >> 3;
        double H[9], F[9];
        qp_kinematics(conn, X, u, e, int(qp & 7), H, F);
        predictor t;
        predict(t, H, prm, st, ds, dc, e, qp);
        auto form = [&](const double* y, double* res) {
            lanes_sync();
            for (int i = sub; i < 16; i += 4)
                for (int j = 0; j < 16; ++j) A[(i * 16 + j) * kDamagePoints] = 0.0;
            system(kp, kd, t.G, t.lam, t.sy, t.Emod, dc, dt, t.ee, t.beta, t.dmg, y, res,
                   [&](int i, int j, double v) {
                       if ((i & 3) == sub) A[(i * 16 + j) * kDamagePoints] = v;
                   });
            lanes_sync();
        };
        double y[16], yprev[16], res[16];
        uint64_t rowp = 0, colp = 0;
        y[0] = y[1] = 0.0;
        kin(t.sig, y + 2);
        kin(t.beta, y + 8);
        y[14] = t.dmg;
        y[15] = t.energy;
        double rn = 2.0; // the reference starts from a residual of ones (norm 4)
        int it = 0;
        bool ok = true;
        while (rn > 1.0e-6 && it < 50)
        {
            form(y, res);
            double s = 0.0;
#pragma unroll
            for (int i = 0; i < 16; ++i) s += res[i] * res[i];
            rn = sqrt(s);
            if (!lu_full(A, sub, rowp, colp))
            {
                ok = false;
                break;
            }
#pragma unroll
            for (int i = 0; i < 16; ++i)
                if ((i & 3) == sub) r[i * kDamagePoints] = res[i];
            lu_solve(A, sub, rowp, colp, r, x);
#pragma unroll
            for (int i = 0; i < 16; ++i)
            {
                yprev[i] = y[i];
                y[i] -= x[i * kDamagePoints];
            }
            ++it;
            // the reference tests the residual of the iterate it just solved from (its loop
            // condition reads the residual the last system computed)
        }
        if ((!ok || it == 50 || y[14] > 1.0) && sub == 0) atomicOr(status, STATUS_RETURN_MAP);
        double const pinc = y[0] > 0.0 ? y[0] : 0.0;
        double sig[9], beta[9];
        kin_from(y + 2, sig);
        kin_from(y + 8, beta);
        double const dmg = y[14] > t.dmg ? y[14] : t.dmg;
        // tangent (1 - D) mandel(C_e) mandel(inverse(J)[2:8, 2:8]) with the Jacobian of the
        // last iteration: rebuild it at the iterate it was formed at and factor once
        double inv22[36];
#pragma unroll
        for (int i = 0; i < 36; ++i) inv22[i] = 0.0;
        if (it > 0 && ok)
        {
            form(yprev, res);
            if (!lu_full(A, sub, rowp, colp))
            {
                if (sub == 0) atomicOr(status, STATUS_RETURN_MAP);
            }
            else
#pragma unroll
                for (int c = 0; c < 6; ++c)
                {
                    for (int i = sub; i < 16; i += 4) r[i * kDamagePoints] = i == 2 + c ? 1.0 : 0.0;
                    lu_solve(A, sub, rowp, colp, r, x);
#pragma unroll
                    for (int k = 0; k < 6; ++k) inv22[k * 6 + c] = x[(2 + k) * kDamagePoints];
                    lanes_sync();
                }
        }
#pragma unroll
        for (int i = 0; i < 6; ++i)
            if ((i & 3) == sub)
#pragma unroll
                for (int j = 0; j < 6; ++j)
                {
                    double p = 0.0;
#pragma unroll
                    for (int k = 0; k < 6; ++k)
                        p += ce_entry(t.lam, t.G, i, k) * mandel_factor(i, k) * inv22[k * 6 + j] * mandel_factor(k, j);
                    st.coef[int64_t(i * 6 + j) * Q + qp] = (1.0 - dmg) * p;
                }
        if (sub != 0) continue;
        // update_internal_variables after the return map (:104-119)
        double d[9];
        for (int i = 0; i < 9; ++i) d[i] = sig[i] - beta[i];
        double const m = (d[0] + d[4] + d[8]) / 3.0;
        d[0] -= m, d[4] -= m, d[8] -= m;
        double const nd = sqrt(ddot9(d, d));
        double const inc = pinc * dt;
        double ep[9], ev[6];
        for (int i = 0; i < 9; ++i) ep[i] = t.ep[i] + inc * sqrt(1.5) * d[i] / (nd * (1.0 - dmg));
        kin(ep, ev);
        for (int k = 0; k < 6; ++k) st.eps_p[k * Q + qp] = ev[k];
        st.ebar[qp] = t.eb + inc / (1.0 - dmg);
        kin(beta, ev);
        for (int k = 0; k < 6; ++k) ds.beta[k * Q + qp] = ev[k];
        ds.dmg[qp] = dmg;
        store_stress(st, ds, qp, sig, von_mises_rel(sig, beta), y[15], status);
    }
}
} // namespace neon_amd
