// Column part of a Runge-Kutta stage's start, production form of both
// precisions: the update of the stage before (UpdateRK2, thor_auxiliary.h:420-529),
// the thermodynamic diagnostics (Compute_Temperature_H_Pt_Geff,
// thor_auxiliary.h:55-309), the vertical advection and Coriolis terms
// (Compute_Advec_Cori2, thor_adv_cor.h:366-536) and the factorisation of the
// stage's vertical solve (the coefficients of Vertical_Eq,
// thor_vertical_int.h:52-563).
#pragma once
#include "dyn_kernels_solve.h"

namespace thor {

// Per-level constants of k_column_w, [kColConst][nv + 1] (one block). Per
// interface l: the weights of the cells below and above, 1 / (Alt[l] - Alt[l - 1]),
// r^2 and the coefficients of the tridiagonal rows (k_thomas_factor's dzph or2,
// inttm, intl, dzmh or2, tor3 and GCoR). Per cell: the weights of its lower and
// upper interface, 1 / (dz r2m).
constexpr int kColConst = 13;
enum { CC_WL, CC_WU, CC_IDA, CC_R2, CC_K1, CC_K2, CC_K3, CC_K4, CC_T3, CC_GC, CC_CL, CC_CU, CC_IDZ };
__global__ void k_column_consts(Geo g, double *out) {
    const int l = threadIdx.x, nv = g.nv, N = nv + 1;
    if (l > nv) return;
    const double A = g.A, rh = g.Alth[l] + A;
    for (int i = 0; i < kColConst; i++) out[i * N + l] = 0.0;
    out[CC_R2 * N + l] = g.deep ? rh * rh : 1.0;
    if (l < nv) {
        const double lo = g.Alth[l], hi = g.Alth[l + 1], c = g.Alt[l], rm = c + A;
        out[CC_CL * N + l] = (c - hi) / (lo - hi);
        out[CC_CU * N + l] = (c - lo) / (hi - lo);
        out[CC_IDZ * N + l] = g.deep ? 1.0 / ((hi - lo) * rm * rm) : 1.0 / (hi - lo);
    }
    if (l >= 1 && l < nv) {
        const double alt = g.Alt[l], altl = g.Alt[l - 1], alth = g.Alth[l], altht = g.Alth[l + 1], althl = g.Alth[l - 1];
        out[CC_WL * N + l] = (alth - alt) / (altl - alt);
        out[CC_WU * N + l] = (alth - altl) / (alt - altl);
        out[CC_IDA * N + l] = 1.0 / (alt - altl);
        const double dzp = 1.0 / (altht - alth), dzh = 1.0 / (alt - altl), dzm = 1.0 / (alth - althl);
        const double or2 = g.deep ? 1.0 / (rh * rh) : 1.0, CvR = (g.Cp - g.Rd) / g.Rd;
        const double ql = A / (A + altl), qu = A / (A + alt);
        const double gl = (g.ghv ? g.Gravit * ql * ql : g.Gravit) * CvR, gu = (g.ghv ? g.Gravit * qu * qu : g.Gravit) * CvR;
        out[CC_K1 * N + l] = dzp * dzh * or2;
        out[CC_K2 * N + l] = -(altl - alth) * dzm * dzh;
        out[CC_K3 * N + l] = (alt - alth) * dzp * dzh;
        out[CC_K4 * N + l] = dzm * dzh * or2;
        out[CC_T3 * N + l] = g.deep ? 2.0 / (rh * rh * rh) : 0.0;
        out[CC_GC * N + l] = (gl * (alt - alth) + gu * (alth - altl)) * dzh;
    }
}

// 16 columns per 256-thread block, 16 rows; row r owns the cells c0 = r SEG ..
// c0 + SEG - 1 (SEG = ceil(nv / 16)) and the interfaces below them (the last row
// the top one too). Neighbouring rows exchange their edge cells and interfaces
// through LDS, so every value is read and formed once; the level constants come
// from a table, leaving two divisions and one power per cell. The pivot
// recurrence c'_l = cc_l / (bb_l - aa_l c'_{l-1}) is composed per row as a Moebius
// map and scanned over the rows (by lane shuffles within a wave).
// UPD: the cells are the stage before plus its deviations, written out as the
// new stage values; else they are read as they are. f: the fields of that
// stage (UPD) or of this one; dt: this stage's substep.
// Three kernels did this (k_update_rk2, k_column_prep_lv, k_thomas_factor_seg):
// about 20 FP64 divisions and two powers per cell, the stage values, hh and
// gtilh written and read again: 50 + 77 + 29 us at 40 962 x 48, 11.4 + 21 + 10 at
// 10 242 x 40, 3.7 + 12.2 + 5.0 at 2 562 x 20 (mixed). Here 111, 22 and 10.7 with
// the update (240 bytes per cell: 100 us of HBM at 40 962 x 48), 73, 17 and 9.3
// without. Three waves per SIMD at three cells per row.
template <int SEG, bool UPD, bool MX>
__global__ __launch_bounds__(256) void k_column_w(Geo g, Fields f, double dt) {
    constexpr int CB = 16, NROW = 16;
    __shared__ double sc[kColConst * (NROW * SEG + 1)];
    __shared__ double sx[2][7][NROW][CB];  // first and last cell of each row; then interfaces and maps
    const int nv = g.nv, N = nv + 1, t = threadIdx.x, c = t % CB, row = t / CB, wave = t >> 6, sub = row & 3;
    const int p = blockIdx.x * CB + c;
    const unsigned S8 = (unsigned)g.S * 8u, none = 0x80000000u;
    for (int i = t; i < kColConst * N; i += 256) sc[i] = g.ccl[i];
    const int c0 = row * SEG, n = p < g.P ? max(0, min(nv, c0 + SEG) - c0) : 0;
    const bool top = n > 0 && c0 + n == nv;
    const size_t b1 = (size_t)nv * S8, bi = (size_t)N * S8;
    const unsigned base = (unsigned)c0 * S8 + 8u * (unsigned)p;
    unsigned off[SEG + 1];  // of level c0 + i (interfaces: i <= n)
#pragma unroll
    for (int i = 0; i <= SEG; i++) off[i] = n > 0 && i <= n ? base + i * S8 : none;
    auto oc = [&](int i) { return i < n ? off[i] : none; };  // of a cell
    const unsigned cb = (unsigned)b1;  // bytes of a component
    const double fr[3] = {p < g.P ? g.fr[p] : 0.0, p < g.P ? g.fr[g.S + p] : 0.0, p < g.P ? g.fr[2 * (size_t)g.S + p] : 0.0};
    // cells j = 0 (row below), 1 .. SEG, SEG + 1 (row above)
    double wp[SEG + 2], wr[SEG + 2], wh[SEG + 2], wt[SEG + 2], wv[SEG + 2][3], W[SEG + 1];
    {
        const auto rM = rsrc(f.Mhk, 3 * b1), rR = rsrc(f.Rhok, b1), rP = rsrc(f.pk, b1), rW = rsrc(f.Whk, bi);
        const auto sM = rsrc(FS<MX>::Mhs(f), UPD ? (MX ? 3 * b1 / 2 : 3 * b1) : 0), sR = rsrc(f.Rhos, UPD ? b1 : 0),
                   sP = rsrc(f.ps, UPD ? b1 : 0), sW = rsrc(f.Whs, UPD ? bi : 0), rWk = rsrc(f.Wk, b1);
        double m[SEG][3], wk[SEG];
#pragma unroll
        for (int i = 0; i <= SEG; i++) {
            W[i] = ldb_d(rW, off[i], 0);
            if constexpr (UPD) W[i] = W[i] + ldb_d(sW, off[i], 0);
        }
#pragma unroll
        for (int i = 0; i < SEG; i++) {
            const unsigned o = oc(i);
#pragma unroll
            for (int k = 0; k < 3; k++) {
                m[i][k] = ldb_d(rM, o, k * cb);
                if constexpr (UPD) {
                    if constexpr (MX) m[i][k] = m[i][k] + (double)ldb_f(sM, o == none ? none : o >> 1, k * (cb >> 1));
                    else m[i][k] = m[i][k] + ldb_d(sM, o, k * cb);
                }
            }
            wr[i + 1] = ldb_d(rR, o, 0);
            wp[i + 1] = ldb_d(rP, o, 0);
            if constexpr (UPD) {
                wr[i + 1] = wr[i + 1] + ldb_d(sR, o, 0);
                wp[i + 1] = wp[i + 1] + ldb_d(sP, o, 0);
            } else {
                wk[i] = ldb_d(rWk, o, 0);
            }
        }
        __syncthreads();  // sc
        if constexpr (UPD) {
            if (c0 == 0) W[0] = 0.0;
            const auto oM = rsrc(f.Mhk_out, 3 * b1), oR = rsrc(f.Rhok_out, b1), oP = rsrc(f.pk_out, b1),
                       oW = rsrc(f.Whk_out, bi), oWk = rsrc(f.Wk_out, b1);
#pragma unroll
            for (int i = 0; i <= SEG; i++) {
                if (top && i == n) W[i] = 0.0;
                if (i < n || (top && i == n)) stb_d(oW, off[i], 0, W[i]);
            }
#pragma unroll
            for (int i = 0; i < SEG; i++) {
                const unsigned o = oc(i);
                const double aux = m[i][0] * fr[0] + m[i][1] * fr[1] + m[i][2] * fr[2];
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    m[i][k] = m[i][k] - aux * fr[k];
                    stb_d(oM, o, k * cb, m[i][k]);
                }
                stb_d(oR, o, 0, wr[i + 1]);
                stb_d(oP, o, 0, wp[i + 1]);
                const int l = min(c0 + i, nv);
                wk[i] = W[i] * sc[CC_CL * N + l] + W[i + 1] * sc[CC_CU * N + l];
                stb_d(oWk, o, 0, wk[i]);
            }
        }
        const double Rd = g.Rd, Cv = g.Cp - g.Rd, iRd = 1.0 / Rd, CpoR = g.Cp / Rd, PoR = g.P_Ref / Rd, iP = 1.0 / g.P_Ref, kap = Cv / g.Cp;
        const auto oT = rsrc(f.T, b1), oh = rsrc(f.h, b1), opt = rsrc(f.pt, b1), ohp = rsrc(f.mhpt, MX ? b1 : 0);
#pragma unroll
        for (int i = 0; i < SEG; i++) {
            const unsigned o = oc(i);
            const double inv = 1.0 / wr[i + 1], pr = wp[i + 1] * inv;
            const double T = pr * iRd;
            wh[i + 1] = CpoR * pr;  // Cv T + p / rho
            wt[i + 1] = PoR * inv * (i < n ? pow_fma(wp[i + 1] * iP, kap) : 1.0);
            const double w = wk[i] * inv;
#pragma unroll
            for (int k = 0; k < 3; k++) wv[i + 1][k] = m[i][k] * inv + w * fr[k];
            stb_d(oT, o, 0, T);
            stb_d(oh, o, 0, wh[i + 1]);
            stb_d(opt, o, 0, wt[i + 1]);
            if constexpr (MX) {
                stb_f(ohp, o == none ? none : o >> 1, 0, (float)wh[i + 1]);
                stb_f(ohp, o == none ? none : o >> 1, cb >> 1, (float)wt[i + 1]);
            }
        }
    }
    auto edge = [&](int which, int j) {
        sx[which][0][row][c] = wp[j];
        sx[which][1][row][c] = wr[j];
        sx[which][2][row][c] = wh[j];
        sx[which][3][row][c] = wt[j];
#pragma unroll
        for (int k = 0; k < 3; k++) sx[which][4 + k][row][c] = wv[j][k];
    };
    edge(0, 1);
    edge(1, SEG);
    __syncthreads();
    auto take = [&](int which, int rr, int j) {
        wp[j] = sx[which][0][rr][c];
        wr[j] = sx[which][1][rr][c];
        wh[j] = sx[which][2][rr][c];
        wt[j] = sx[which][3][rr][c];
#pragma unroll
        for (int k = 0; k < 3; k++) wv[j][k] = sx[which][4 + k][rr][c];
    };
    take(1, max(row - 1, 0), 0);
    take(0, min(row + 1, NROW - 1), SEG + 1);
    __syncthreads();  // sx is reused
    // interfaces i = 0 .. n (level c0 + i): hh, gtilh, and the fluxes of v and p
    double hh[SEG + 1], gt[SEG + 1], F[SEG + 1][3], wg[SEG + 1];
    const double *Alt = g.Alt, *Alth = g.Alth;
    const auto ohh = rsrc(f.hh, bi), opth = rsrc(f.pth, bi), ogt = rsrc(f.gtilh, bi);
#pragma unroll
    for (int i = 0; i <= SEG; i++) {
        const int l = min(c0 + i, nv);
        double pth;
        if (c0 + i == 0) {  // ground: cells 1 and 2 of the window
            const double a0 = Alt[0], a1 = Alt[1], q = g.A / (g.A + a0), gr = g.ghv ? g.Gravit * q * q : g.Gravit;
            const double pl = wp[2] - wr[1] * gr * (-a0 - a1);
            const double rl = wr[2] + (wr[2] - wr[1]) * ((-a0 - a1) / (a1 - a0));
            hh[i] = wh[1];
            gt[i] = -(wp[1] - pl) / (2.0 * a0 * (0.5 * (wr[1] + rl)));
            pth = wt[2] + (wt[2] - wt[1]) * ((Alth[0] - a1) / (a1 - a0));
            wg[i] = F[i][0] = F[i][1] = F[i][2] = 0.0;
        } else if (i > 0 && top && i == n) {  // lid: the two cells below
            const double a1 = Alt[nv - 1], a2 = Alt[nv - 2], at = Alth[nv], q = g.A / (g.A + a1),
                         gr = g.ghv ? g.Gravit * q * q : g.Gravit, ex = (2 * at - a1 - a2) / (a1 - a2);
            const double p2 = wp[i > 0 ? i - 1 : 0], r1 = wr[i], r2 = wr[i > 0 ? i - 1 : 0], t2 = wt[i > 0 ? i - 1 : 0];
            const double rp = r2 + (r1 - r2) * ex;
            const double pp = p2 - r1 * gr * (2 * at - a1 - a2);
            hh[i] = wh[i];
            gt[i] = -(pp - wp[i]) / (2.0 * (at - a1) * (0.5 * (r1 + rp)));
            pth = t2 + (wt[i] - t2) * ex;
            wg[i] = F[i][0] = F[i][1] = F[i][2] = 0.0;
        } else {
            const double wl = sc[CC_WL * N + l], wu = sc[CC_WU * N + l];
            hh[i] = wh[i] * wl + wh[i + 1] * wu;
            pth = wt[i] * wl + wt[i + 1] * wu;
            gt[i] = -(wp[i + 1] - wp[i]) * sc[CC_IDA * N + l] / (wr[i] * wl + wr[i + 1] * wu);
            wg[i] = W[i] * gt[i];
            const double wr2 = W[i] * sc[CC_R2 * N + l];
#pragma unroll
            for (int k = 0; k < 3; k++) F[i][k] = (wv[i][k] * wl + wv[i + 1][k] * wu) * wr2;
        }
        const unsigned o = i < n || (top && i == n) ? off[i] : none;
        stb_d(ohh, o, 0, hh[i]);
        stb_d(opth, o, 0, pth);
        stb_d(ogt, o, 0, gt[i]);
    }
    // cells: gtil, vertical advection and Coriolis
    {
        const auto ogl = rsrc(f.gtil, b1), oA = rsrc(FS<MX>::Adv(f), MX ? 3 * b1 / 2 : 3 * b1);
        const double Om = 2.0 * g.Omega;
#pragma unroll
        for (int i = 0; i < SEG; i++) {
            const int l = min(c0 + i, nv);
            const unsigned o = oc(i);
            stb_d(ogl, o, 0, wg[i] * sc[CC_CL * N + l] + wg[i + 1] * sc[CC_CU * N + l]);
            const double *v = wv[i + 1], r = Om * wr[i + 1], iz = sc[CC_IDZ * N + l];
            double a[3];
            if (g.deep) {
                a[0] = -r * v[1];
                a[1] = r * v[0];
                a[2] = 0.0;
            } else {
                a[0] = r * (v[2] * fr[2] * fr[1] - v[1] * fr[2] * fr[2]);
                a[1] = -r * (v[2] * fr[2] * fr[0] - v[0] * fr[2] * fr[2]);
                a[2] = r * (v[1] * fr[2] * fr[0] - v[0] * fr[2] * fr[1]);
            }
#pragma unroll
            for (int k = 0; k < 3; k++) {
                const double ad = (F[i + 1][k] - F[i][k]) * iz + a[k];
                if constexpr (MX) stb_f(oA, o == none ? none : o >> 1, k * (cb >> 1), (float)ad);
                else stb_d(oA, o, k * cb, ad);
            }
        }
    }
    // factorisation: rows l = c0 + i, 1 <= l < nv, from hh and gtilh at l - 1, l, l + 1
    double hm, gm;
    sx[0][0][row][c] = hh[SEG - 1];
    sx[0][1][row][c] = gt[SEG - 1];
    __syncthreads();
    hm = sx[0][0][max(row - 1, 0)][c];
    gm = sx[0][1][max(row - 1, 0)][c];
    const double CRdd = (g.Cp - g.Rd) / (g.Rd * dt * dt);
    double ra[SEG], rb[SEG], rc[SEG];
    double m00 = 1.0, m01 = 0.0, m10 = 0.0, m11 = 1.0;  // c'_{last} = (m00 x + m01) / (m10 x + m11)
    // the product of two maps, scaled by a power of two to stay in range
    auto scale = [&]() {
        const double big = fmax(fmax(fabs(m00), fabs(m01)), fmax(fabs(m10), fabs(m11)));
        const int e = -__builtin_amdgcn_frexp_exp(big);
        m00 = ldexp(m00, e);
        m01 = ldexp(m01, e);
        m10 = ldexp(m10, e);
        m11 = ldexp(m11, e);
    };
#pragma unroll
    for (int i = 0; i < SEG; i++) {
        const int l = min(c0 + i, nv);
        const double k1 = sc[CC_K1 * N + l], k2 = sc[CC_K2 * N + l], k3 = sc[CC_K3 * N + l], k4 = sc[CC_K4 * N + l],
                     t3 = sc[CC_T3 * N + l], gc = sc[CC_GC * N + l];
        const double Hm = (i ? hh[i > 0 ? i - 1 : 0] : hm) * sc[CC_R2 * N + max(l - 1, 0)], H = hh[i] * sc[CC_R2 * N + l],
                     Hp = hh[i + 1] * sc[CC_R2 * N + min(l + 1, nv)];
        const double gml = i ? gt[i > 0 ? i - 1 : 0] : gm;
        rc[i] = -k1 * Hp - k2 * (gt[i + 1] + gc - t3 * Hp);
        rb[i] = (k1 + k4) * H + (k3 - k2) * (gt[i] + gc - t3 * H);
        if (g.nonhydro) rb[i] = rb[i] + CRdd;
        ra[i] = -k4 * Hm + k3 * (gml + gc - t3 * Hm);
        if (i < n && c0 + i > 0) {
            const double a = c0 + i == 1 ? 0.0 : -ra[i];  // c'_0 does not enter the first interface
            const double n00 = rc[i] * m10, n01 = rc[i] * m11;
            const double n10 = a * m00 + rb[i] * m10, n11 = a * m01 + rb[i] * m11;
            m00 = n00;
            m01 = n01;
            m10 = n10;
            m11 = n11;
            scale();
        }
    }
    double x;
    {
        auto after = [&](int d, bool on) {  // this map after the one d rows below
            const double p00 = __shfl_up(m00, 16 * d), p01 = __shfl_up(m01, 16 * d), p10 = __shfl_up(m10, 16 * d),
                         p11 = __shfl_up(m11, 16 * d);
            if (on) {
                const double n00 = m00 * p00 + m01 * p10, n01 = m00 * p01 + m01 * p11;
                const double n10 = m10 * p00 + m11 * p10, n11 = m10 * p01 + m11 * p11;
                m00 = n00;
                m01 = n01;
                m10 = n10;
                m11 = n11;
                scale();
            }
        };
        after(1, sub >= 1);
        after(2, sub >= 2);
        const double e00 = __shfl_up(m00, 16), e01 = __shfl_up(m01, 16), e10 = __shfl_up(m10, 16), e11 = __shfl_up(m11, 16);
        if (sub == 3) {
            sx[1][0][wave][c] = m00;
            sx[1][1][wave][c] = m01;
            sx[1][2][wave][c] = m10;
            sx[1][3][wave][c] = m11;
        }
        __syncthreads();
        x = 0.0;  // c' below the wave, then below the row
        for (int w = 0; w < wave; w++)
            x = (sx[1][0][w][c] * x + sx[1][1][w][c]) / (sx[1][2][w][c] * x + sx[1][3][w][c]);
        if (sub >= 1) x = (e00 * x + e01) / (e10 * x + e11);
    }
    const auto oAA = rsrc(f.tAA, b1), oCC = rsrc(f.tCC, b1), oTT = rsrc(f.tTT, b1);
#pragma unroll
    for (int i = 0; i < SEG; i++) {
        if (i < n && c0 + i > 0) {
            const bool first = c0 + i == 1;
            const double tt = 1.0 / (first ? rb[i] : rb[i] - x * ra[i]);
            x = rc[i] * tt;
            stb_d(oAA, off[i], 0, ra[i]);
            stb_d(oCC, off[i], 0, x);
            stb_d(oTT, off[i], 0, first ? rb[i] : tt);
        }
    }
}

} // namespace thor
