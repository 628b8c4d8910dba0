// Vertical solve with the density/pressure update of the acoustic substep
// (Vertical_Eq, thor_vertical_int.h:52-563, and the column part of
// Density_Pressure_Eqs, thor_fastmodes.h:255-847), production form of both
// precisions: 16 columns per 256-thread block, 16 rows, row r owning the
// interfaces [lo, hi) of its column and the cells lo .. hi - 1 above them (row 0
// cell 0 too).
#pragma once
#include "dyn_kernels.h"

namespace thor {

// Per-level constants of k_solve, [6][nv + 1] (one block): 1 / (Alt[l] -
// Alt[l - 1]); gravity times the weights of the cells below and above
// interface l; r^2 of interface l; and per cell 1 / dr2dz and 1 / (dz r2m).
__global__ void k_solve_levels(Geo g, double *out) {
    const int l = threadIdx.x, nv = g.nv, N = nv + 1;
    if (l > nv) return;
    const double A = g.A, rh = g.Alth[l] + A;
    out[3 * N + l] = g.deep ? rh * rh : 1.0;
    out[l] = out[N + l] = out[2 * N + l] = out[4 * N + l] = out[5 * N + l] = 0.0;
    if (l >= 1 && l < nv) {
        const double alt = g.Alt[l], altl = g.Alt[l - 1], alth = g.Alth[l], q = A / (A + alt);
        const double gr = g.ghv ? g.Gravit * q * q : g.Gravit;
        out[l] = 1.0 / (alt - altl);
        out[N + l] = gr * (alth - alt) / (altl - alt);
        out[2 * N + l] = gr * (alth - altl) / (alt - altl);
    }
    if (l < nv) {
        const double dz = g.Alth[l + 1] - g.Alth[l], rt = g.Alth[l + 1] + A, rm = g.Alt[l] + A;
        out[4 * N + l] = g.deep ? 3.0 / (rt * rt * rt - rh * rh * rh) : 1.0 / dz;
        out[5 * N + l] = g.deep ? 1.0 / (dz * rm * rm) : 1.0 / dz;
    }
}

// v^y for v > 0 as exp(y log v), the series of pm::log and pm::exp with fused
// multiply-adds (half the instructions; one rounding less per term).
__device__ __forceinline__ double pow_fma(double v, double y) {
    if (!(v > 1e-300 && v < 1e300)) return pm::pow(v, y);  // subnormal, zero, negative, infinite or NaN
    const uint64_t u = pm::bits(v);
    int e = (int)(u >> 52) - 1023;
    double m = pm::from_bits((u & 0x000fffffffffffffull) | 0x3ff0000000000000ull);
    if (m > 1.4142135623730951) {
        m = m * 0.5;
        e += 1;
    }
    const double s = (m - 1.0) / (m + 1.0), s2 = s * s;
    double q = 1.0 / 27.0;
#pragma unroll
    for (int k = 25; k >= 3; k -= 2) q = __builtin_fma(q, s2, 1.0 / k);
    const double lm = __builtin_fma(2.0 * s, s2 * q, 2.0 * s), de = (double)e;
    const double t = y * (__builtin_fma(de, pm::LN2_HI, lm) + de * pm::LN2_LO);
    const double n = rint(t * pm::INV_LN2);
    if (!(fabs(n) < 1000.0)) return pm::exp(t);
    const double r = __builtin_fma(n, -pm::LN2_LO, __builtin_fma(n, -pm::LN2_HI, t));
    double f = 1.0 / 355687428096000.0, k = 355687428096000.0;  // 1 / 17!
#pragma unroll
    for (int i = 17; i >= 3; i--) {
        k /= i;  // (i - 1)!, a compile-time constant
        f = __builtin_fma(f, r, 1.0 / k);
    }
    return __builtin_fma(r, __builtin_fma(r, f, 1.0), 1.0) * pm::from_bits((uint64_t)((int64_t)n + 1023) << 52);
}

// The density/pressure update of one cell from the horizontal flux
// divergences and the divergences dw, dwpt of the vertical mass and pressure
// fluxes. With pf = ps + pk, 1/q = (pf / P_Ref)^(-Cv/Cp) and x = -Rd (nflxpt +
// dwptdz) dt / (P_Ref q) the reference's new pressure is pf (1 + x)^(Cp/Cv), so
// pnew - pk = ps + pf ((1 + x)^(Cp/Cv) - 1), formed without the cancellation of
// pnew - pk: for |x| < 2^-7 by the binomial series to x^9, else by a power.
struct DpConst {
    double dt, kap, gam, iP, RoP, RoCdt;  // Cv / Cp, Cp / Cv, 1 / P_Ref, Rd dt / P_Ref, Rd dt / Cv
    __device__ __forceinline__ DpConst(const Geo &g, double dt_)
        : dt(dt_), kap((g.Cp - g.Rd) / g.Cp), gam(g.Cp / (g.Cp - g.Rd)), iP(1.0 / g.P_Ref), RoP(g.Rd * dt_ / g.P_Ref),
          RoCdt(g.Rd / (g.Cp - g.Rd) * dt_) {}
};
__device__ __forceinline__ double dp_pressure(const DpConst &k, double ps, double pk, double flux, double dpr, double q) {
    const double pf = ps + pk;
    const double x = -flux * k.RoP * pow_fma(pf * k.iP, -k.kap);
    double dp;
    if (fabs(x) < 0.0078125) {
        double c[10];
        c[1] = k.gam;
#pragma unroll
        for (int i = 2; i <= 9; i++) c[i] = c[i - 1] * (k.gam - (i - 1)) * (1.0 / i);
        double h = c[9];
#pragma unroll
        for (int i = 8; i >= 1; i--) h = __builtin_fma(h, x, c[i]);
        dp = pf * (h * x);
    } else {
        // a cell of no pressure (x is infinite or NaN): pnew = P_Ref (-Rd flux dt / P_Ref)^(Cp/Cv)
        const bool none = pf == 0.0;
        const double q1 = pow_fma(none ? -flux * k.RoP : 1.0 + x, k.gam);
        dp = none ? q1 / k.iP : pf * (q1 - 1.0);
    }
    return ps + dp + (dpr * k.dt + k.RoCdt * q);
}

// The forward elimination x_l = (-C_l - x_{l-1} AA_l) TT_l and the back
// substitution w_l = x_l - CC_l w_{l+1} are first-order linear recurrences: each
// row composes its interfaces into one affine map, the maps are scanned in row
// order (four rows of a wave by lane shuffles, the four waves through LDS) and
// each row then runs its interfaces from its true start, all in registers.
// Every value is read from HBM once, with buffer loads on one 32-bit offset
// per interface, before the first scan; the level constants come from a table
// in LDS, so a cell costs one logarithm and one exponential and no division
// of its own. The form before it (k_thomas_dp_seg: about nine FP64 divisions,
// 64-bit addresses per value, the update's loads behind the sweeps, a chain
// over up to 15 rows in LDS) took 24 cycles of a CU per cell, VALU as much as
// memory: 77 us at 40 962 x 48, 22.9 at 10 242 x 40 and 10.7 at 2 562 x 20 in the
// mixed form; here 59, 16.1 and 7.9. Its floor there: 140 bytes per cell (14 FP64
// planes and diffpr in, 3 out; Qheat, where it is not known to be zero, 8 more;
// FP64 form 4 more), so 58 us at the 4.73 TB/s of a large copy, and 6.7 and 0.8 at
// the 8.5 TB/s of one within the 256 MB cache.
// SEG: interfaces per row, ceil((nv - 1) / 16). DP = false: the solve alone
// (k_dp_solve then applies the update after a physics hook).
template <int SEG, bool DP, bool MX>
__global__ __launch_bounds__(256) void k_solve(Geo g, Fields f, double deltat) {
    constexpr int CB = 16, NROW = 16;
    __shared__ double sc[6 * (NROW * SEG + 2)], sa[2][4][CB], sb[2][4][CB];
    const int nv = g.nv, N = nv + 1, t = threadIdx.x, c = t % CB, row = t / CB, wave = t >> 6, sub = row & 3;
    const int p = blockIdx.x * CB + c;
    const unsigned S8 = (unsigned)g.S * 8u;
    for (int i = t; i < 6 * N; i += 256) sc[i] = g.tlv[i];
    const int seg = (nv - 1 + NROW - 1) / NROW, lo = 1 + row * seg, hi = min(nv, lo + seg);
    const int n = p < g.P ? max(0, hi - lo) : 0;  // interfaces lo .. lo + n - 1
    const unsigned none = 0x80000000u;            // an offset outside every buffer: loads 0, stores nothing
    const unsigned base = (unsigned)(lo - 1) * S8 + 8u * (unsigned)p;
    unsigned off[SEG + 2];  // of level lo - 1 + i
#pragma unroll
    for (int i = 0; i < SEG + 2; i++) off[i] = n > 0 && i <= n + 1 ? base + i * S8 : none;
    const size_t b1 = (size_t)nv * S8, bi = (size_t)N * S8;
    const auto rR = rsrc(f.Rhos, b1), rP = rsrc(f.ps, b1), rS = rsrc(f.SlowRho, b1), rF = rsrc(f.hflx_r, b1),
               rSp = rsrc(f.Sp, b1), rSw = rsrc(f.SlowWh, bi), rW = rsrc(f.Whs, bi), rA = rsrc(f.tAA, b1),
               rT = rsrc(f.tTT, b1), rC = rsrc(f.tCC, b1);
    // cells lo - 1 .. lo + n - 1
    double cR[SEG + 1], cP[SEG + 1], cD[SEG + 1], cSp[SEG + 1];
    double a[SEG], tt[SEG], cc[SEG], x[SEG];
#pragma unroll
    for (int i = 0; i <= SEG; i++) {
        const unsigned o = i <= n ? off[i] : none;
        cR[i] = ldb_d(rR, o, 0);
        cP[i] = ldb_d(rP, o, 0);
        cD[i] = ldb_d(rS, o, 0);
        const double fr = ldb_d(rF, o, 0);
        cD[i] = cD[i] - fr;  // Sd: SlowRho less the horizontal mass flux divergence
        cSp[i] = ldb_d(rSp, o, 0);
    }
#pragma unroll
    for (int i = 0; i < SEG; i++) {
        const unsigned o = i < n ? off[i + 1] : none;
        x[i] = deltat * ldb_d(rSw, o, 0);
        if (g.nonhydro) x[i] = x[i] + ldb_d(rW, o, 0);
        a[i] = ldb_d(rA, o, 0);
        tt[i] = ldb_d(rT, o, 0);
        cc[i] = ldb_d(rC, o, 0);
    }
    // the update's own inputs: cells 0 .. n (0 on row 0 only), interfaces lo .. lo + n
    double ePk[SEG + 1], eF[SEG + 1], eD[SEG + 1], eQ[SEG + 1], hW[SEG + 1], hP[SEG + 1];
    if constexpr (DP) {
        const auto rPk = rsrc(f.pk, b1), rFp = rsrc(f.hflx_pt, b1), rQ = rsrc(f.Qheat, f.Qheat ? b1 : 0), rWk = rsrc(f.Whk, bi),
                   rPt = rsrc(f.pth, bi), rD = rsrc(FS<MX>::diffpr(f), MX ? b1 / 2 : b1);
#pragma unroll
        for (int i = 0; i <= SEG; i++) {
            const unsigned o = i <= n && (i > 0 || row == 0) ? off[i] : none, oh = i <= n ? off[i + 1] : none;
            ePk[i] = ldb_d(rPk, o, 0);
            eF[i] = ldb_d(rFp, o, 0);
            if constexpr (MX) eD[i] = ldb_f(rD, o == none ? none : o >> 1, 0);
            else eD[i] = ldb_d(rD, o, 0);
            eQ[i] = ldb_d(rQ, o, 0);
            hW[i] = ldb_d(rWk, oh, 0);
            hP[i] = ldb_d(rPt, oh, 0);
        }
    }
    __syncthreads();  // sc
    const double *kz = sc, *kl = sc + N, *ku = sc + 2 * N;
    const double CvR = (g.Cp - g.Rd) / (g.Rd * deltat * deltat), dt2 = deltat * deltat;
    double ma = 1.0, mb = 0.0;  // the row's map x_{hi-1} = ma x_{lo-1} + mb
    {
        double al = dt2 * cSp[0] + deltat * cP[0], bl = dt2 * cD[0] + deltat * cR[0];
#pragma unroll
        for (int i = 0; i < SEG; i++) {
            const double au = dt2 * cSp[i + 1] + deltat * cP[i + 1], bu = dt2 * cD[i + 1] + deltat * cR[i + 1];
            const int l = min(lo + i, nv);
            // -C0
            const double r = CvR * (x[i] - (au - al) * kz[l] - (kl[l] * bl + ku[l] * bu));
            al = au;
            bl = bu;
            if (i < n) {
                const bool first = lo + i == 1;  // TT[1] holds the pivot itself
                const double piv = first ? 1.0 / tt[i] : tt[i];
                a[i] = first ? 0.0 : -a[i] * piv;
                x[i] = r * piv;
                ma = a[i] * ma;
                mb = a[i] * mb + x[i];
            }
        }
    }
    // exclusive scan of the maps over the rows: x at the interface below the row
    auto compose = [&](double pa, double pb, bool on) {  // this map after (pa, pb)
        if (on) {
            mb = ma * pb + mb;
            ma = ma * pa;
        }
    };
    double xs;
    {
        const double a1 = __shfl_up(ma, 16), b1s = __shfl_up(mb, 16);
        compose(a1, b1s, sub >= 1);
        const double a2 = __shfl_up(ma, 32), b2s = __shfl_up(mb, 32);
        compose(a2, b2s, sub >= 2);
        const double ea = __shfl_up(ma, 16), eb = __shfl_up(mb, 16);
        if (sub == 3) {
            sa[0][wave][c] = ma;
            sb[0][wave][c] = mb;
        }
        __syncthreads();
        xs = 0.0;
        for (int w = 0; w < wave; w++) xs = sa[0][w][c] * xs + sb[0][w][c];
        if (sub >= 1) xs = ea * xs + eb;
    }
    ma = 1.0;
    mb = 0.0;
#pragma unroll
    for (int i = 0; i < SEG; i++)
        if (i < n) {
            xs = a[i] * xs + x[i];
            x[i] = xs;
        }
    // the row's map w_lo = ma w_hi + mb of the back substitution, from the top down
#pragma unroll
    for (int i = SEG - 1; i >= 0; i--)
        if (i < n) {
            ma = -cc[i] * ma;
            mb = x[i] - cc[i] * mb;
        }
    // w: Whs at interface hi (0 at the top); wlo: at lo, the same number that the
    // row below starts from, so both cells of an interface use one flux
    double w, wlo;
    {
        const double a1 = __shfl_down(ma, 16), b1s = __shfl_down(mb, 16);
        compose(a1, b1s, sub <= 2);
        const double a2 = __shfl_down(ma, 32), b2s = __shfl_down(mb, 32);
        compose(a2, b2s, sub <= 1);
        const double ea = __shfl_down(ma, 16), eb = __shfl_down(mb, 16);
        if (sub == 0) {
            sa[1][wave][c] = ma;
            sb[1][wave][c] = mb;
        }
        __syncthreads();
        w = 0.0;
        for (int v = 3; v > wave; v--) w = sa[1][v][c] * w + sb[1][v][c];
        wlo = ma * w + mb;
        if (sub <= 2) w = ea * w + eb;
    }
    // down through the row's cells
    const double *kr = sc + 3 * N, *kd = p >= g.P - 2 ? sc + 5 * N : sc + 4 * N, *kp = sc + 5 * N;
    const DpConst K(g, deltat);
    bool nan = false;
    double fw = 0.0, fp = 0.0;  // vertical mass and pressure flux times r^2 at the interface above the cell
    if constexpr (DP) {
        const double r2 = kr[min(hi, nv)];
        fw = w * r2;
#pragma unroll
        for (int i = 0; i <= SEG; i++)  // interface lo + n
            if (i == n) fp = (w + hW[i]) * hP[i] * r2;
    }
#pragma unroll
    for (int i = SEG - 1; i >= -1; i--) {
        // interface lo + i and the cell above it (i = -1: cell 0, no flux through the ground)
        if (i >= n || (i < 0 && (row != 0 || n == 0))) continue;
        if (i >= 0) {
            w = i == 0 ? wlo : x[i] - cc[i] * w;
            stb_d(rW, off[i + 1], 0, w);
        }
        if constexpr (DP) {
            const int l = lo + i;
            double gw = 0.0, gp = 0.0;
            if (i >= 0) {
                const double r2 = kr[l];
                gw = w * r2;
                gp = (w + hW[i < 0 ? 0 : i]) * hP[i < 0 ? 0 : i] * r2;
            }
            const double flux = eF[i + 1] + (fp - gp) * kp[l];
            stb_d(rR, off[i + 1], 0, cR[i + 1] + (cD[i + 1] - (fw - gw) * kd[l]) * deltat);
            const double ps = dp_pressure(K, cP[i + 1], ePk[i + 1], flux, eD[i + 1], eQ[i + 1]);
            stb_d(rP, off[i + 1], 0, ps);
            nan |= isnan(ps);
            fw = gw;
            fp = gp;
        }
    }
    if (DP && nan) atomicOr(f.flags, FLAG_NAN_P);
}

// The update alone, after a solve and a physics hook: one thread per (point,
// level), the same numbers as in k_solve.
template <bool MX> __global__ __launch_bounds__(256) void k_dp_solve(Geo g, Fields f, double deltat) {
    const int p = blockIdx.x * 256 + threadIdx.x, l = blockIdx.y, nv = g.nv, N = nv + 1;
    if (p >= g.P) return;
    const size_t S = g.S;
    const double *kr = g.tlv + 3 * N, *kd = g.tlv + (p >= g.P - 2 ? 5 : 4) * N, *kp = g.tlv + 5 * N;
    const DpConst K(g, deltat);
    double fw = 0.0, fp = 0.0, gw = 0.0, gp = 0.0;
    {
        const double w = l + 1 < nv ? LV(f.Whs, l + 1) : 0.0, r2 = kr[l + 1];
        fw = w * r2;
        fp = (w + LV(f.Whk, l + 1)) * LV(f.pth, l + 1) * r2;
    }
    if (l > 0) {
        const double w = LV(f.Whs, l), r2 = kr[l];
        gw = w * r2;
        gp = (w + LV(f.Whk, l)) * LV(f.pth, l) * r2;
    }
    const double cD = LV(f.SlowRho, l) - LV(f.hflx_r, l);
    const double flux = LV(f.hflx_pt, l) + (fp - gp) * kp[l];
    LV(f.Rhos, l) = LV(f.Rhos, l) + (cD - (fw - gw) * kd[l]) * deltat;
    const double ps = dp_pressure(K, LV(f.ps, l), LV(f.pk, l), flux, (double)LV(FS<MX>::diffpr(f), l),
                                  f.Qheat ? LV(f.Qheat, l) : 0.0);
    LV(f.ps, l) = ps;
    if (isnan(ps)) atomicOr(f.flags, FLAG_NAN_P);
}

} // namespace thor
