// Two-scale fatigue damage per Gauss point, FP64, device-resident state.
//
// Restates the functor Kokkos_Kernel::operator() (kokkos_kernel.h:44-344, constants
// damage.h:8-17) launched by kokkos_host_ (kokkos_host.cpp:37-190): one lane per
// Gauss point walks the nip temporal interpolation points of the slab in order,
// with the elastic predictor / plastic corrector / Lemaitre damage update of the
// reference.
//
// The return map branches on the trial stress at every time point; at load
// reversals the trial stress lies on the yield surface, so a last-bit difference
// flips branches and the history variables diverge.  The kernel therefore keeps
// the reference's exact operation sequence (same products, same summation order; the
// 0.0 that the reference starts its sums from changes at most the sign of a zero and is
// left out) with floating-point contraction disabled in this file, and evaluates the
// damage power (Y/S)^0.5 as the correctly rounded sqrt, the same choice as the oracle.
// Division and sqrt are IEEE correctly rounded on gfx950, so every lane reproduces the
// CPU restatement bit for bit.
//
// What bounds it: FP64 instructions, about 280 an elastic step (the law's multiplications
// and additions, which may not be fused) at 2 waves a SIMD (256 registers).  Off the elastic
// step are taken, without a change of any result: what depends on the damage alone (3
// divisions, kept until it changes), the divisions by 3 (div3) and the root of the yield
// test (its square against the largest double whose root is at most sig_f; the root itself
// only where the corrector or the end asks for it); in the corrector 20 of 34 divisions have a
// reciprocal at hand (quotients), 8 are by 3 and 2 are of constants (a block of 630 elements
// that damages, 688 points: 0.69 -> 0.48 ms).  345600 points, 2560 time points: 11.9 -> 9.7 ms,
// with the displacements written a time point ahead 8.8; 5400 waves on 1024 SIMDs leave
// 12 % of it to the last round.
//
// Work sharing: the 8 Gauss points of a C3D8 element interpolate the same 24
// nodal displacements disp = sum_k Nt_k u_k (kokkos_kernel.h:58-71).  The 8
// lanes of an element each interpolate one node (identical operations to the
// reference) and exchange the 24 values through LDS, so the interpolation costs
// 36 instead of 288 FP64 operations per lane and time point.  The per-GP state
// stays in registers across the nip steps and is written back once.
// Element status (chkelesta, delelement.f90:109-136) is a second small kernel.
#include <cmath>
#include <limits>

#include "xt_common.h"

#pragma clang fp contract(off)

namespace xt {

// Material constants of the damage law.  Defaults: damage.h:9-17 (Cy = 1740, h = 0.2,
// S = 0.5, s = 0.5, sig_f = 180, sig_u = 577, eps_D = 0.08); the damage threshold is
// wd = (sig_u - sig_f) eps_D (kokkos_kernel.h:47).
struct DamageParams {
    double sigf = 180.0, sigu = 577.0, epsd = 0.08, cy = 1740.0, h = 0.2, S = 0.5, sexp = 0.5;
};
#define XT_CY dp.cy
#define XT_H dp.h
#define XT_S dp.S
#define XT_SIGF dp.sigf
#define XT_WD ((dp.sigu - dp.sigf) * dp.epsd)

// x / 3 and x / den, correctly rounded, from a correctly rounded reciprocal: a quotient
// within one unit in the last place, its exact remainder by one fma and the correction by
// another (Markstein, IBM J. Res. Dev. 34, 1990).  For 3 the product with the reciprocal is
// that close; for any other divisor a first correction makes it so.  The remainder is exact
// unless the quotient is subnormal (or, den other than 3, x is outside 2^-900 .. 2^900): such
// values, infinities and NaNs go through the division itself.  3 and 5 operations in place
// of the 11 and a quarter-rate reciprocal of a division.
static __device__ inline double div3(double x) {
    const double r = 1.0 / 3.0;
    const double q = x * r;
    double y = fma(fma(-3.0, q, x), r, q);
    const bool odd = __builtin_amdgcn_class(q, 0x297);   // NaN, infinite, subnormal
    if (__builtin_amdgcn_ballot_w64(odd)) y = odd ? x / 3.0 : y;   // (a branch, not a select)
    return y;
}

static __device__ inline bool ordinary(double v) {   // 2^-100 .. 2^100
    const int e = __builtin_amdgcn_frexp_exp(v);
    return e > -100 && e < 100 && !__builtin_amdgcn_class(v, 0x267);
}
// x[i] / den, r = 1 / den correctly rounded
template <int N>
static __device__ inline void quotients(double (&x)[N], double den, double r, bool ord_den) {
    double y[N];
    int lo = 0, hi = 0;
    bool inf = false;
    for (int i = 0; i < N; ++i) {
        const int e = __builtin_amdgcn_frexp_exp(x[i]);   // (0 for 0, infinities and NaNs)
        lo = min(lo, e);
        hi = max(hi, e);
        inf |= __builtin_amdgcn_class(x[i], 0x207);
        const double q = x[i] * r;
        const double q1 = fma(fma(-den, q, x[i]), r, q);
        y[i] = fma(fma(-den, q1, x[i]), r, q1);
    }
    const bool odd = !ord_den || inf || lo < -900 || hi > 900;
    if (__builtin_amdgcn_ballot_w64(odd))
        for (int i = 0; i < N; ++i) y[i] = odd ? x[i] / den : y[i];
    for (int i = 0; i < N; ++i) x[i] = y[i];
}
// 1.5 and 3 times the squares of a deviator, summed in the reference's order
static __device__ inline double equivalent2(const double (&t)[6]) {
    double e = 1.5 * t[0] * t[0];
    for (int i = 1; i < 3; ++i) e += 1.5 * t[i] * t[i];
    for (int i = 3; i < 6; ++i) e += 3.0 * t[i] * t[i];
    return e;
}

// Block = one wave of 64 lanes = 8 elements x 8 Gauss points (GP ii = 8 e + g).
__global__ void __launch_bounds__(64, 2)
damage_kernel(int ngp, int nn, int nip, const int *__restrict__ nodes,
              const double *__restrict__ Nx, const double *__restrict__ Ny,
              const double *__restrict__ Nz, const double *__restrict__ Nt,
              const double *__restrict__ sol, const double *__restrict__ ym,
              const double *__restrict__ nu, double *__restrict__ eps_old,
              double *__restrict__ eps_pl, double *__restrict__ sig_eff,
              double *__restrict__ sig_back, double *__restrict__ pp, double *__restrict__ dd,
              double *__restrict__ wsv, double *__restrict__ del_po_v,
              double *__restrict__ sig_d_v, const DamageParams dp, const double sigf2,
              const double r2s, const double rs) {
    __shared__ double xch[2][64][4];  // [parity][lane][disp of the lane's node, padded]
    // what only the corrector reads, out of the registers: c4, gamma, p, ws, del_po, G, Kb,
    // (1 + nu) / 2 E and nu / 2 E
    __shared__ double rare[9][64];
    const int lane = threadIdx.x;
    const int ii = blockIdx.x * 64 + lane;
    const bool act = ii < ngp;
    const int g = lane & 7;       // node of the element this lane interpolates
    const int e0 = lane & ~7;     // first lane of this lane's element
    // nodal temporal coefficients of node g: sl[k][j] = sol(k, node, j)
    double sl[6][3];
    double nx[8], ny[8], nz[8];
    double nui = 0.3, ymi = 1.0;
    double eo[6], ep[6], se[6], sb[6];
    double d = 0.0, sig_d = 0.0;
    if (act) {
        const size_t plane = (size_t)nn * 3;
        const size_t nd = (size_t)(nodes[(size_t)ii * 8 + g] - 1) * 3;
        for (int k = 0; k < 6; ++k)
            for (int j = 0; j < 3; ++j) sl[k][j] = sol[k * plane + nd + j];
        for (int a = 0; a < 8; ++a) {
            nx[a] = Nx[(size_t)ii * 8 + a];
            ny[a] = Ny[(size_t)ii * 8 + a];
            nz[a] = Nz[(size_t)ii * 8 + a];
        }
        nui = nu[ii];
        ymi = ym[ii];
        for (int c = 0; c < 6; ++c) {
            eo[c] = eps_old[(size_t)ii * 6 + c];
            ep[c] = eps_pl[(size_t)ii * 6 + c];
            se[c] = sig_eff[(size_t)ii * 6 + c];
            sb[c] = sig_back[(size_t)ii * 6 + c];
        }
        d = dd[ii]; sig_d = sig_d_v[ii];
        rare[2][lane] = pp[ii]; rare[3][lane] = wsv[ii]; rare[4][lane] = del_po_v[ii];
    } else {
        for (int k = 0; k < 6; ++k) for (int j = 0; j < 3; ++j) sl[k][j] = 0.0;
        for (int a = 0; a < 8; ++a) { nx[a] = 0.0; ny[a] = 0.0; nz[a] = 0.0; }
        for (int c = 0; c < 6; ++c) { eo[c] = 0.0; ep[c] = 0.0; se[c] = 0.0; sb[c] = 0.0; }
    }
    // constants of kokkos_kernel.h:49-53 and the elastic matrix of :88-100
    const double a = (1.0 + nui) / (3.0 * (1.0 - nui));
    const double b = 2.0 * (4.0 - 5.0 * nui) / (15.0 * (1.0 - nui));
    rare[5][lane] = ymi / (2.0 * (1.0 + nui));
    rare[6][lane] = ymi / (3.0 * (1.0 - 2.0 * nui));
    rare[7][lane] = (1.0 + nui) / (2.0 * ymi);
    rare[8][lane] = nui / (2.0 * ymi);
    const double coef = ymi / ((1. + nui) * (1. - 2. * nui));
    const double dl = coef * nui;
    const double dg = coef * (1.0 - nui);
    const double dsh = coef * (1.0 - 2.0 * nui) / 2.0;
    // functions of the damage alone (kokkos_kernel.h:104-115, :196, :213), kept until it changes
    double c1, c2, c3;
    auto with_damage = [&]() {
        const double om = 1.0 - b * d;
        c1 = 1.0 / om;
        c2 = (a - b) * d / (om * (1.0 - a * d));
        c3 = b * (1.0 - d) / om;
        const double G = rare[5][lane], Kb = rare[6][lane];
        rare[0][lane] = Kb * (a - b) * d / (om * (1.0 - a * d));             // c4
        rare[1][lane] = XT_CY * (1.0 - d) + 3.0 * G * (1.0 - b) / om;        // gamma
    };
    with_damage();
    bool squared = false;   // sig_d holds the square of the equivalent stress

    // disp of node g at a time point (kokkos_kernel.h:60-71: disp += Nt_k * sol, k ascending)
    auto interpolate = [&](const double (&nt)[6], double *out) {
        for (int j = 0; j < 3; ++j) {
            double s = nt[0] * sl[0][j];
            for (int k = 1; k < 6; ++k) s += nt[k] * sl[k][j];
            out[j] = s;
        }
    };
    auto table = [&](int jj, double (&nt)[6]) {
        for (int k = 0; k < 6; ++k) nt[k] = Nt[(size_t)(jj < nip ? jj : nip - 1) * 6 + k];
    };
    // The displacements of a time point are written during the one before (and the table's
    // row read one earlier still), so that their way through LDS is not waited for.  (One
    // wave: its LDS accesses complete in order.)
    double nt[6];
    table(0, nt);
    interpolate(nt, xch[0][lane]);
    table(1, nt);
    for (int jj = 0; jj < nip; ++jj) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        double (*buf)[4] = xch[jj & 1];
        // strain (kokkos_kernel.h:74-84)
        double strain[6];
        for (int i = 0; i < 8; ++i) {
            const double d0 = buf[e0 + i][0], d1 = buf[e0 + i][1], d2 = buf[e0 + i][2];
            const double t[6] = {nx[i] * d0, ny[i] * d1, nz[i] * d2, ny[i] * d0 + nx[i] * d1,
                                 nz[i] * d1 + ny[i] * d2, nz[i] * d0 + nx[i] * d2};
            for (int c = 0; c < 6; ++c) strain[c] = i ? strain[c] + t[c] : t[c];
        }
        interpolate(nt, xch[(jj + 1) & 1][lane]);
        table(jj + 2, nt);
        if (!act) continue;
        // elastic predictor (kokkos_kernel.h:104-171)
        double tel[6], tee[6];
        for (int i = 0; i < 6; ++i) tel[i] = c1 * strain[i] + c3 * ep[i];
        double tr = strain[0] + strain[1] + strain[2];
        tr = div3(c2 * tr);
        for (int i = 0; i < 3; ++i) tel[i] += tr;
        for (int i = 0; i < 6; ++i) tee[i] = tel[i] - ep[i];
        // D_el * tee with the reference's row sums (zero entries contribute exact zeros)
        double tse[6];
        tse[0] = (dg * tee[0] + dl * tee[1]) + dl * tee[2];
        tse[1] = (dl * tee[0] + dg * tee[1]) + dl * tee[2];
        tse[2] = (dl * tee[0] + dl * tee[1]) + dg * tee[2];
        tse[3] = dsh * tee[3];
        tse[4] = dsh * tee[4];
        tse[5] = dsh * tee[5];
        const double trs = div3(tse[0] + tse[1] + tse[2]);
        double tsig[6];
        tsig[0] = (tse[0] - trs) - sb[0];
        tsig[1] = (tse[1] - trs) - sb[1];
        tsig[2] = (tse[2] - trs) - sb[2];
        tsig[3] = tse[3] - sb[3];
        tsig[4] = tse[4] - sb[4];
        tsig[5] = tse[5] - sb[5];
        const double teq2 = equivalent2(tsig);
        if (teq2 <= sigf2) {   // the equivalent stress, its root, is at most sig_f
            for (int i = 0; i < 6; ++i) { se[i] = tse[i]; eo[i] = strain[i]; }
            sig_d = teq2;
            squared = true;
            continue;
        }
        // plastic corrector (kokkos_kernel.h:175-263)
        if (squared) sig_d = sqrt(sig_d);
        squared = false;
        double ds_[6], dsig[6];
        for (int i = 0; i < 6; ++i) ds_[i] = strain[i] - eo[i];
        dsig[0] = (dg * ds_[0] + dl * ds_[1]) + dl * ds_[2];
        dsig[1] = (dl * ds_[0] + dg * ds_[1]) + dl * ds_[2];
        dsig[2] = (dl * ds_[0] + dl * ds_[1]) + dg * ds_[2];
        dsig[3] = dsh * ds_[3];
        dsig[4] = dsh * ds_[4];
        dsig[5] = dsh * ds_[5];
        const double om = 1.0 - b * d, c4 = rare[0][lane], gamma = rare[1][lane];
        quotients(dsig, om, c1, ordinary(om));
        const double trd = ds_[0] + ds_[1] + ds_[2];
        for (int i = 0; i < 3; ++i) dsig[i] += c4 * trd;
        double Qs[6];
        for (int i = 0; i < 6; ++i) Qs[i] = sb[i] - se[i] - dsig[i];
        const double trq = div3(Qs[0] + Qs[1] + Qs[2]);
        double dq[6] = {Qs[0] - trq, Qs[1] - trq, Qs[2] - trq, Qs[3], Qs[4], Qs[5]};
        const double qeq = sqrt(equivalent2(dq));
        const double tr_sigs = -trq;
        const double del_p = (qeq - XT_SIGF) / gamma;
        rare[2][lane] += del_p;
        double c5q[1] = {gamma * del_p};
        quotients(c5q, XT_SIGF, 2.0 * r2s, ordinary(XT_SIGF));
        const double c5 = 1.0 + c5q[0];
        double dvs[6];
        for (int i = 0; i < 6; ++i) dvs[i] = -dq[i];
        quotients(dvs, c5, 1.0 / c5, ordinary(c5));
        double sigs[6] = {dvs[0] + tr_sigs, dvs[1] + tr_sigs, dvs[2] + tr_sigs, dvs[3], dvs[4], dvs[5]};
        double dpl[6];
        for (int i = 0; i < 6; ++i) dpl[i] = 3.0 * dvs[i] * del_p;
        quotients(dpl, 2.0 * XT_SIGF, r2s, ordinary(XT_SIGF));
        for (int i = 0; i < 6; ++i) ep[i] += dpl[i];
        for (int i = 0; i < 6; ++i) sb[i] += div3(2.0 * XT_CY * (1.0 - d) * dpl[i]);
        for (int i = 0; i < 6; ++i) se[i] = sigs[i] + sb[i];
        const double tse2 = div3(se[0] + se[1] + se[2]);
        double dse[6] = {se[0] - tse2, se[1] - tse2, se[2] - tse2, se[3], se[4], se[5]};
        const double seq = sqrt(equivalent2(dse));
        const double sig_new = fabs(seq - XT_SIGF);
        const double sig_old = fabs(sig_d - XT_SIGF);
        const double ws = rare[3][lane] + (sig_new * del_p + sig_old * rare[4][lane]) / 2.0;
        rare[3][lane] = ws;
        const double d_was = d;
        if (ws >= XT_WD) {
            // Lemaitre damage increment (kokkos_kernel.h:293-330)
            double sp[3] = {0.0, 0.0, 0.0}, sn[3] = {0.0, 0.0, 0.0};
            for (int i = 0; i < 3; ++i) {
                if (se[i] < 0.0) sn[i] = se[i];
                else sp[i] = se[i];
            }
            const double y1 = rare[7][lane], y2 = rare[8][lane];
            const double hr = (1.0 - d) / (1.0 - XT_H * d);
            const double Yp = y1 *
                              (sp[0] * sp[0] + sp[1] * sp[1] + sp[2] * sp[2] +
                               XT_H * hr * hr * (sn[0] * sn[0] + sn[1] * sn[1] + sn[2] * sn[2]));
            double trt = 0.0;
            for (int i = 0; i < 3; ++i) trt += se[i];
            double Yn;
            if (trt >= 0.0) Yn = y2 * trt * trt;
            else Yn = y2 * XT_H * hr * hr * trt * trt;
            // (Y/S)^s: s = 0.5 as the correctly rounded sqrt (the reference's value)
            double ys[1] = {Yp - Yn};
            quotients(ys, XT_S, rs, ordinary(XT_S));
            d += (dp.sexp == 0.5 ? sqrt(ys[0]) : pow(ys[0], dp.sexp)) * del_p;
        } else {
            d = 0.0;
        }
        if (d != d_was) with_damage();
        for (int i = 0; i < 6; ++i) eo[i] = strain[i];
        sig_d = seq;
        rare[4][lane] = del_p;
    }
    if (!act) return;
    if (squared) sig_d = sqrt(sig_d);
    for (int c = 0; c < 6; ++c) {
        eps_old[(size_t)ii * 6 + c] = eo[c];
        eps_pl[(size_t)ii * 6 + c] = ep[c];
        sig_eff[(size_t)ii * 6 + c] = se[c];
        sig_back[(size_t)ii * 6 + c] = sb[c];
    }
    pp[ii] = rare[2][lane];
    dd[ii] = d;
    wsv[ii] = rare[3][lane];
    del_po_v[ii] = rare[4][lane];
    sig_d_v[ii] = sig_d;
}

// element e failed iff any of its ngpe Gauss points has D >= Dc
__global__ void __launch_bounds__(256)
elestatus_kernel(int ne, int ngpe, double Dc, const double *__restrict__ D, int *elesta,
                 int *gpsta, int *failed) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= ne) return;
    int any = 0;
    for (int g = 0; g < ngpe; ++g) any |= (D[(size_t)e * ngpe + g] >= Dc);
    failed[e] = any;
    if (any) {
        elesta[e] = 0;
        for (int g = 0; g < ngpe; ++g) gpsta[(size_t)e * ngpe + g] = 0;
    }
}

// kokkos_damage.f90:102-107: a failed Gauss point carries D = ws = 0
__global__ void __launch_bounds__(256)
zero_failed_kernel(int ngp, const int *__restrict__ gpsta, double *D, double *ws) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g < ngp && gpsta[g] == 0) {
        D[g] = 0.0;
        ws[g] = 0.0;
    }
}

// The largest double whose square root rounds to at most v (v > 0)
static double largest_square(double v) {
    double t = v * v;
    while (std::sqrt(t) > v) t = std::nextafter(t, 0.0);
    while (t < std::numeric_limits<double>::infinity() &&
           std::sqrt(std::nextafter(t, std::numeric_limits<double>::infinity())) <= v)
        t = std::nextafter(t, std::numeric_limits<double>::infinity());
    return t;
}

}  // namespace xt

using namespace xt;

extern "C" int xt_damage_device_params(int ne, int nn, int nip, const int *nodes,
                                       const double *Nx, const double *Ny, const double *Nz,
                                       const double *Nt, const double *sol, const double *ym,
                                       const double *nu, double *eps_old, double *eps_pl,
                                       double *sig_eff, double *sig_back, double *p, double *D,
                                       double *ws, double *del_po, double *sig_d,
                                       const double *params, void *stream) {
    XT_ARG(ne >= 0 && nn > 0 && nip >= 0, "damage sizes");
    DamageParams dp;
    if (params) {
        dp.sigf = params[0]; dp.sigu = params[1]; dp.epsd = params[2]; dp.cy = params[3];
        dp.h = params[4]; dp.S = params[5]; dp.sexp = params[6];
        XT_ARG(dp.sigf > 0.0 && dp.sigu > dp.sigf && dp.S > 0.0, "damage parameters");
    }
    XT_ARG(nodes && Nx && Ny && Nz && (nip == 0 || Nt) && sol && ym && nu && eps_old && eps_pl &&
               sig_eff && sig_back && p && D && ws && del_po && sig_d,
           "damage arrays");
    const int ngp = 8 * ne;
    if (ngp == 0 || nip == 0) return XT_OK;
    const bool prof = prof_on(XT_PROF_DAMAGE);
    if (prof) prof_begin(XT_PROF_DAMAGE, (hipStream_t)stream);
    hipLaunchKernelGGL(damage_kernel, dim3(ceil_div(ngp, 64)), dim3(64), 0,
                       (hipStream_t)stream, ngp, nn, nip, nodes, Nx, Ny, Nz, Nt, sol, ym, nu,
                       eps_old, eps_pl, sig_eff, sig_back, p, D, ws, del_po, sig_d, dp,
                       largest_square(dp.sigf), 1.0 / (2.0 * dp.sigf), 1.0 / dp.S);
    if (prof)   // state 31 FP64 read + written, 24 derivatives + 8 node ids, Nt, 24 disp gathers per step
        prof_end(XT_PROF_DAMAGE, (hipStream_t)stream,
                 (double)ngp * (31 * 16 + 24 * 8 + 8 * 4) + 8.0 * 6 * nip + 8.0 * 18 * nn, 0.0);
    XT_HIP(hipGetLastError());
    return XT_OK;
}

extern "C" int xt_damage_device(int ne, int nn, int nip, const int *nodes, const double *Nx,
                                const double *Ny, const double *Nz, const double *Nt,
                                const double *sol, const double *ym, const double *nu,
                                double *eps_old, double *eps_pl, double *sig_eff,
                                double *sig_back, double *p, double *D, double *ws,
                                double *del_po, double *sig_d, void *stream) {
    return xt_damage_device_params(ne, nn, nip, nodes, Nx, Ny, Nz, Nt, sol, ym, nu, eps_old,
                                   eps_pl, sig_eff, sig_back, p, D, ws, del_po, sig_d, nullptr,
                                   stream);
}

namespace xt {
int elestatus_device(int ne, int ngpe, double Dc, const double *D, int *elesta, int *gpsta,
                     int *failed, hipStream_t s) {
    if (ne == 0) return XT_OK;
    hipLaunchKernelGGL(elestatus_kernel, dim3(ceil_div(ne, 256)), dim3(256), 0, s, ne, ngpe, Dc,
                       D, elesta, gpsta, failed);
    XT_HIP(hipGetLastError());
    return XT_OK;
}
}  // namespace xt

extern "C" int xt_elestatus_device(int ne, int ngpe, double Dc, const double *D, int *elesta,
                                   int *gpsta, int *failed, void *stream) {
    XT_ARG(ne >= 0 && ngpe > 0, "elestatus sizes");
    if (ne == 0) return XT_OK;
    XT_ARG(D && elesta && gpsta && failed, "elestatus arrays");
    return elestatus_device(ne, ngpe, Dc, D, elesta, gpsta, failed, (hipStream_t)stream);
}

extern "C" int xt_damage_zero_failed(int ngp, const int *gpsta, double *D, double *ws,
                                     void *stream) {
    XT_ARG(ngp >= 0, "zero_failed size");
    if (ngp == 0) return XT_OK;
    XT_ARG(gpsta && D && ws, "zero_failed arrays");
    hipLaunchKernelGGL(zero_failed_kernel, dim3(ceil_div(ngp, 256)), dim3(256), 0,
                       (hipStream_t)stream, ngp, gpsta, D, ws);
    XT_HIP(hipGetLastError());
    return XT_OK;
}
