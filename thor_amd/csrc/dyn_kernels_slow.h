// Slow tendencies of a Runge-Kutta stage (Compute_Slow_Modes,
// thor_slowmodes.h:48-683, with UpdateRK, thor_auxiliary.h:311-418), production
// form of both precisions over level chunks.
#pragma once
#include "dyn_kernels.h"

namespace thor {

// Per-level constants of k_slow_w, [kSlowConst][nv + 1] (one block): per cell
// rscale, 1 / dr2dz, 1 / (dz r2m), gravity, 1 / (Alt + A); per interface r^2, the
// weights of the cells below and above, 1 / (Alt[l] - Alt[l - 1]).
constexpr int kSlowConst = 9;
enum { SC_RS, SC_IDR, SC_IDZ, SC_G, SC_IR, SC_R2, SC_WL, SC_WU, SC_IDA };
__global__ void k_slow_consts(Geo g, double *out) {
    const int l = threadIdx.x, nv = g.nv, N = nv + 1;
    if (l > nv) return;
    const double A = g.A, rh = g.Alth[l] + A;
    for (int i = 0; i < kSlowConst; i++) out[i * N + l] = 0.0;
    out[SC_R2 * N + l] = g.deep ? rh * rh : 1.0;
    if (l < nv) {
        const double dz = g.Alth[l + 1] - g.Alth[l], rt = g.Alth[l + 1] + A, rm = g.Alt[l] + A, q = A / rm;
        out[SC_RS * N + l] = g.deep ? q : 1.0;
        out[SC_IDR * N + l] = g.deep ? 3.0 / (rt * rt * rt - rh * rh * rh) : 1.0 / dz;
        out[SC_IDZ * N + l] = g.deep ? 1.0 / (dz * rm * rm) : 1.0 / dz;
        out[SC_G * N + l] = g.ghv ? g.Gravit * q * q : g.Gravit;
        out[SC_IR * N + l] = 1.0 / rm;
    }
    if (l >= 1 && l < nv) {
        const double alt = g.Alt[l], altl = g.Alt[l - 1], alth = g.Alth[l];
        out[SC_WL * N + l] = (alth - alt) / (altl - alt);
        out[SC_WU * N + l] = (alth - altl) / (alt - altl);
        out[SC_IDA * N + l] = 1.0 / (alt - altl);
    }
}

// The neighbour weights serve gradient and divergence (THOR's operators share
// them, checked at create), in registers for the chunk; a slot's mass flux
// div . M is formed once and multiplies h and theta. Values of the point alone
// go through 64-bit scalar bases and one 32-bit offset (only the four staged
// fields take buffer descriptors), level constants come from a table in LDS,
// and the forcing tendencies are read only where there are any (null: zero).
// k_slow_lc2 (the reference's order, 24 weight planes in LDS, about 30 buffer
// descriptors, a dozen divisions per cell) spilled 24 vector and 245 scalar
// registers at two blocks per CU: 168 us (mixed) and 228 (FP64) at 40 962 x 48,
// 38.6 and 52.7 at 10 242 x 40, 16.5 and 18.9 at 2 562 x 20; here 135, 142, 27.1,
// 33.1, 11.4 and 13.1 (110 and 140 for the traffic at 40 962 x 48).
// dm: the damping pass 1 (k_divm1_lc, k_divm1_lw). At the first stage the
// deviations start from zero, so the first substep's damping and pressure
// gradient vanish and its momentum equation is Mhs = dt SlowMh (tangential):
// written here, without launches of its own.
template <bool MX>
__global__ __launch_bounds__(256, 2) void k_slow_w(Geo g, Fields f, const typename FS<MX>::R *dm, int divdamp, int rk,
                                                   double dt, int lc) {
#pragma clang fp contract(fast)
    using R = typename FS<MX>::R;
    int r, l0, l1;
    if (!block_tile_lc(g, lc, r, l0, l1)) return;
    const size_t S = g.S;
    const int nv = g.nv;
    if (r == g.nr) {
        PoleCtx c;
        int lev;
        if (!pole_ctx_lc(g, l0, l1, c, lev)) return;
        const int p = c.p;
        double DivM[3] = {0.0, 0.0, 0.0};
        if (divdamp)
            for (int k = 0; k < 3; k++) DivM[k] = VEC(dm, k, lev, p);
        slow_sums<MX, 3>(
            g, f, p, lev, true, rk, DivM, [&](int s) { return LVP(f.pk, lev, c.gi(s)); },
            [&](int s) { return LVP(f.h, lev, c.gi(s)); }, [&](int s, int k) { return VEC(f.Mhk, k, lev, c.gi(s)); });
        if (rk == 0) {
            const auto *Sm = FS<MX>::SlowMh(f);
            const double m[3] = {VEC(Sm, 0, lev, p) * dt, VEC(Sm, 1, lev, p) * dt, VEC(Sm, 2, lev, p) * dt};
            const double mr = m[0] * g.fr[p] + m[1] * g.fr[S + p] + m[2] * g.fr[2 * S + p];
            for (int k = 0; k < 3; k++) VEC(FS<MX>::Mhs(f), k, lev, p) = (R)(m[k] - mr * g.fr[(size_t)k * S + p]);
        }
        return;
    }
    // staged point: (M_x, M_y), (M_z, p), (h, pt)
    __shared__ double2 sA[2][NHL2], sB[2][NHL2], sC[2][NHL2];
    __shared__ double sK[kSlowConst][kLcMax + 1];
    const int N = nv + 1;
    for (int i = threadIdx.x; i < kSlowConst * (l1 - l0 + 1); i += 256)
        sK[i / (l1 - l0 + 1)][i % (l1 - l0 + 1)] = g.scl[(i / (l1 - l0 + 1)) * N + l0 + i % (l1 - l0 + 1)];
    const LcThread T = lc_thread(g, r);
    const int p = T.p;
    double w[24];  // gradient, then the divergence weights of slot 0
    load_packed(g.pgrad, S, p, w);
    const double *wd0 = w + 21;
    const double fr[3] = {g.fr[p], g.fr[S + p], g.fr[2 * S + p]};
    const unsigned p8 = (unsigned)S * 8u, pR = (unsigned)(S * sizeof(R));  // bytes of a level plane
    const size_t c8 = (size_t)nv * p8, cR = (size_t)nv * pR;               // of a component
    // values of the point alone: component k of a vector (or a scalar) at a 32-bit offset
    auto ld = [&](const auto *b, int k, size_t cs, unsigned off) {
        return *(decltype(b))((const char *)b + (size_t)k * cs + (size_t)off);
    };
    auto st = [&](auto *b, int k, size_t cs, unsigned off, double v) {
        using V = std::remove_pointer_t<decltype(b)>;
        *(V *)((char *)b + (size_t)k * cs + (size_t)off) = (V)v;
    };
    const auto rM = rsrc(f.Mhk, 3 * c8), rP = rsrc(f.pk, c8), rH = rsrc(f.h, c8), rT = rsrc(f.pt, c8);
    struct Stg {
        double om[3], op, oh, ot, hm[3], hp, hh, ht;
    };
    auto load = [&](Stg &v, int lev) {
        const unsigned l8 = (unsigned)lev * p8;
#pragma unroll
        for (int k = 0; k < 3; k++) {
            v.om[k] = ldb_d(rM, T.o8, (unsigned)(k * c8) + l8);
            v.hm[k] = ldb_d(rM, T.h8, (unsigned)(k * c8) + l8);
        }
        v.op = ldb_d(rP, T.o8, l8);
        v.hp = ldb_d(rP, T.h8, l8);
        v.oh = ldb_d(rH, T.o8, l8);
        v.hh = ldb_d(rH, T.h8, l8);
        v.ot = ldb_d(rT, T.o8, l8);
        v.ht = ldb_d(rT, T.h8, l8);
    };
    auto put = [&](const Stg &v, int b) {
        sA[b][T.ir] = make_double2(v.om[0], v.om[1]);
        sB[b][T.ir] = make_double2(v.om[2], v.op);
        sC[b][T.ir] = make_double2(v.oh, v.ot);
        if (T.hp >= 0) {
            sA[b][T.hp] = make_double2(v.hm[0], v.hm[1]);
            sB[b][T.hp] = make_double2(v.hm[2], v.hp);
            sC[b][T.hp] = make_double2(v.hh, v.ht);
        }
    };
    const R *Adv = FS<MX>::Adv(f), *dmh = FS<MX>::diffmh(f), *dfw = FS<MX>::diffw(f), *drh = FS<MX>::diffrh(f),
            *dpr = FS<MX>::diffpr(f);
    R *SlowMh = FS<MX>::SlowMh(f), *Mhs = FS<MX>::Mhs(f);
    // the radial advection, hydrostatic: its metric form (the same operations
    // wherever a chunk begins)
    auto dot = [](const double a[3], const double c[3]) {
        return __builtin_fma(a[2], c[2], __builtin_fma(a[1], c[1], a[0] * c[0]));
    };
    // the cell below: radial advection (or its hydrostatic form), rho, p, vertical diffusion, gravity
    double c_advr = 0.0, c_rho = 0.0, c_p = 0.0, c_dw = 0.0, c_g = 0.0;
    if (l0 > 0) {
        c_g = g.scl[SC_G * N + l0 - 1];
        const unsigned o8 = T.o8 + (unsigned)(l0 - 1) * p8, oR = (unsigned)(T.p * sizeof(R)) + (unsigned)(l0 - 1) * pR;
        c_rho = ld(f.Rhok, 0, 0, o8);
        c_p = ld(f.pk, 0, 0, o8);
        c_dw = ld(dfw, 0, 0, oR);
        const double m[3] = {ld(f.Mhk, 0, c8, o8), ld(f.Mhk, 1, c8, o8), ld(f.Mhk, 2, c8, o8)};
        const double a[3] = {(double)ld(Adv, 0, cR, oR), (double)ld(Adv, 1, cR, oR), (double)ld(Adv, 2, cR, oR)};
        c_advr = g.nonhydro ? dot(a, fr) : dot(m, m) / c_rho * g.scl[SC_IR * N + l0 - 1];
    }
    double whl = ld(f.Whk, 0, 0, T.o8 + (unsigned)l0 * p8), hhl = ld(f.hh, 0, 0, T.o8 + (unsigned)l0 * p8);
    const double RoC = g.Rd / (g.Cp - g.Rd);
    Stg A;
    load(A, l0);
    put(A, 0);
    __syncthreads();
    for (int lev = l0; lev < l1; lev++) {
        const int b = (lev - l0) & 1, i = lev - l0;
        const unsigned o8 = T.o8 + (unsigned)lev * p8, oR = (unsigned)(T.p * sizeof(R)) + (unsigned)lev * pR;
        // the point's own values, then the next level's tile
        double adv[3], src[3], y[3];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            adv[k] = ld(Adv, k, cR, oR);
            src[k] = ld(dmh, k, cR, oR);
            if (divdamp) src[k] += ld(dm, k, cR, oR);
            y[k] = rk ? ld(f.Mh, k, c8, o8) : 0.0;
        }
        const double rho = ld(f.Rhok, 0, 0, o8), wht = ld(f.Whk, 0, 0, o8 + p8), hht = ld(f.hh, 0, 0, o8 + p8),
                     dw = ld(dfw, 0, 0, oR), v_drh = ld(drh, 0, 0, oR), v_dpr = ld(dpr, 0, 0, oR),
                     v_gt = ld(f.gtil, 0, 0, o8);
        double yr = 0.0, yp = 0.0, yw = 0.0;
        if (rk) {
            yr = ld(f.Rho, 0, 0, o8);
            yp = ld(f.p, 0, 0, o8);
            yw = ld(f.Wh, 0, 0, o8);
        }
        double v_q = f.Qheat ? ld(f.Qheat, 0, 0, o8) : 0.0, v_dwh = 0.0;
        if (f.dMh) {
            v_dwh = ld(f.dWh, 0, 0, o8);
#pragma unroll
            for (int k = 0; k < 3; k++) src[k] += ld(f.dMh, k, c8, o8);
        }
        if constexpr (!MX)
            if (f.diffmv) {
#pragma unroll
                for (int k = 0; k < 3; k++) src[k] += ld(f.diffmv, k, c8, o8);
            }
        load(A, min(lev + 1, l1 - 1));
        double gp[3], nr, nh, nt, m0[3], p0;
        {
            const double2 a = sA[b][T.pos[0]], q = sB[b][T.pos[0]], h = sC[b][T.pos[0]];
            m0[0] = a.x;
            m0[1] = a.y;
            m0[2] = q.x;
            p0 = q.y;
            const double d = wd0[0] * a.x + wd0[1] * a.y + wd0[2] * q.x;
#pragma unroll
            for (int k = 0; k < 3; k++) gp[k] = w[k] * p0;
            nr = d;
            nh = d * h.x;
            nt = d * h.y;
        }
#pragma unroll
        for (int s = 1; s < 7; s++) {
            const double2 a = sA[b][T.pos[s]], q = sB[b][T.pos[s]], h = sC[b][T.pos[s]];
            const double d = w[s * 3] * a.x + w[s * 3 + 1] * a.y + w[s * 3 + 2] * q.x;
#pragma unroll
            for (int k = 0; k < 3; k++) gp[k] += w[s * 3 + k] * q.y;
            nr += d;
            nh += d * h.x;
            nt += d * h.y;
        }
        const double rs = sK[SC_RS][i];
        st(f.hflx_ptk, 0, 0, o8, rs * nt);
        // horizontal momentum: tangential part of gradient and advection, and the tendencies
        double advr = dot(adv, fr);
        const double gr = rs * (gp[0] * fr[0] + gp[1] * fr[1] + gp[2] * fr[2]);
        double vgp = 0.0, sm[3];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const double gt = rs * gp[k] - gr * fr[k];
            vgp += gt * m0[k];
            sm[k] = src[k] - gt - (adv[k] - advr * fr[k]);
            st(SlowMh, k, cR, oR, sm[k]);
        }
        if (!g.nonhydro) advr = dot(m0, m0) / rho * sK[SC_IR][i];
        // vertical momentum at the interface below
        if (lev > 0) {
            const double wl = sK[SC_WL][i], wu = sK[SC_WU][i];
            double lo = c_rho * c_g, up = rho * sK[SC_G][i];
            if (g.deep) {
                lo += c_advr;
                up += advr;
            }
            if (g.nonhydro) {
                lo -= c_dw;
                up -= dw;
            }
            st(f.SlowWh, 0, 0, o8, -(lo * wl + up * wu + (p0 - c_p) * sK[SC_IDA][i] - v_dwh));
        } else {
            whl = 0.0;
            st(f.SlowWh, 0, 0, o8, 0.0);
            LV(f.SlowWh, nv) = 0.0;
        }
        c_g = sK[SC_G][i];
        const double ul = whl * sK[SC_R2][i], ut = wht * sK[SC_R2][i + 1];
        st(f.SlowRho, 0, 0, o8, v_drh - (rs * nr + (ut - ul) * sK[SC_IDR][i]));
        double sp = RoC * (v_q + vgp / rho - rs * nh - v_gt - (ut * hht - ul * hhl) * sK[SC_IDZ][i]);
        sp += !MX && g.energy ? RoC * v_dpr : v_dpr;  // thor_slowmodes.h:375-377
        st(f.Slowp, 0, 0, o8, sp);
        // deviations at the start of the stage
        if (rk == 0) {
            const double mr = sm[0] * fr[0] + sm[1] * fr[1] + sm[2] * fr[2];
#pragma unroll
            for (int k = 0; k < 3; k++) st(Mhs, k, cR, oR, dt * (sm[k] - mr * fr[k]));
            st(f.Rhos, 0, 0, o8, 0.0);
            st(f.ps, 0, 0, o8, 0.0);
            st(f.Whs, 0, 0, o8, 0.0);
        } else {
            const double Mx = y[0] - m0[0], My = y[1] - m0[1], Mz = y[2] - m0[2];
            const double mr = Mx * fr[0] + My * fr[1] + Mz * fr[2];
            st(Mhs, 0, cR, oR, Mx - mr * fr[0]);
            st(Mhs, 1, cR, oR, My - mr * fr[1]);
            st(Mhs, 2, cR, oR, Mz - mr * fr[2]);
            st(f.Rhos, 0, 0, o8, yr - rho);
            st(f.ps, 0, 0, o8, yp - p0);
            st(f.Whs, 0, 0, o8, lev == 0 ? 0.0 : yw - whl);
        }
        if (lev == nv - 1) LV(f.Whs, nv) = 0.0;
        c_advr = advr;
        c_rho = rho;
        c_p = p0;
        c_dw = dw;
        whl = wht;
        hhl = hht;
        if (lev + 1 < l1) put(A, b ^ 1);
        __syncthreads();
    }
}

} // namespace thor
