// FP64 horizontal operators of the production build over level chunks.
//
// The Laplacian and the divergence-damping operator are linear in their
// inputs, with coefficients fixed by the geometry and the level's rscale
// (dyn_kernels.h, k_probe_weights). Walking a point's triangles level by level
// (dyn_kernels_ml.h) costs 60-100 doubles of geometry and a chain of divisions
// per point and level group: those kernels ran at 8-36 % VALU and 1.5 TB/s,
// waiting on the next triangle's geometry. Here each thread holds its point's
// FP64 operator weights in registers for a chunk of levels and the next
// levels' tiles are loaded while the current one is summed (the pipeline of
// the mixed form's _lc kernels), so a level costs its field traffic. The sums
// are those of the triangle walk in another order: the parity build, which is
// compared bit for bit, keeps the triangle walk.
//
// Measured at 40 962 x 48 (us per launch, triangle walk -> here; the field
// traffic at the 4.7 TB/s of a large copy in brackets): advection and first
// Laplacian 243 -> 78 [60], last Laplacian 224 -> 60 [43], damping pass 0 100 ->
// 38 [24], pass 1 64 -> 30 [20], momentum 107 -> 49 [43]; the FP64 step
// 7.70 -> 5.00 ms. At 2 562 x 23, one level per block: 27.6 -> 9.3, 22.4 -> 7.1,
// 17.0 -> 9.5, 13.9 -> 7.2, 20.2 -> 10.2.
#pragma once
#include "dyn_kernels.h"

namespace thor {

// The operator weights of every point, for rscale = 1, from the triangle walk
// on unit inputs: wlap [6] (slots 1..6 of the Laplacian's difference form), wdd
// [63] and udd [21] (divergence damping, as Geo::wdd64/udd64), and for the
// outputs that are projected on the tangent plane anyway (divergence-damping
// pass 1, the pressure gradient in the momentum equation) the weights of their
// two tangential components: et [6] a tangent basis e1, e2 of the point, wdt
// [42] and wgt [14] the components of wdd and of the gradient along it.
__global__ __launch_bounds__(256) void k_probe_weights64(Geo gu, double *wlap, double *wdd, double *udd, double *et,
                                                         double *wdt, double *wgt) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= gu.P) return;
    const size_t S = gu.S;
    const bool pole = p >= gu.P - 2;
    const int nf = pole ? 5 : gu.nfc[p];
    {
        double out[7];
        laplacians<7>(gu, p, nf, 1.0, [&](int v, int s) { return v == s ? 1.0 : 0.0; }, out);
        for (int s = 1; s < 7; s++) wlap[(size_t)(s - 1) * S + p] = out[s];
    }
    // e1 along the axis least aligned with the radial direction, e2 = f x e1
    const double f[3] = {gu.fr[p], gu.fr[S + p], gu.fr[2 * S + p]};
    int ax = 0;
    for (int k = 1; k < 3; k++)
        if (fabs(f[k]) < fabs(f[ax])) ax = k;
    double e1[3], e2[3], n = 0.0;
    for (int k = 0; k < 3; k++) {
        e1[k] = (k == ax ? 1.0 : 0.0) - f[ax] * f[k];
        n += e1[k] * e1[k];
    }
    n = sqrt(n);
    for (int k = 0; k < 3; k++) e1[k] /= n;
    for (int k = 0; k < 3; k++) e2[k] = f[(k + 1) % 3] * e1[(k + 2) % 3] - f[(k + 2) % 3] * e1[(k + 1) % 3];
    for (int k = 0; k < 3; k++) {
        et[(size_t)k * S + p] = e1[k];
        et[(size_t)(3 + k) * S + p] = e2[k];
    }
    auto zero = [&](int) { return 0.0; };
    for (int s0 = 0; s0 < 7; s0++) {
        for (int k0 = 0; k0 < 3; k0++) {
            double o3[3];
            divm_nf<false>(
                gu, p, 0, nf, pole, [&](int s, int k) { return (s == s0 && k == k0) ? 1.0 : 0.0; }, zero, zero, o3);
            for (int c = 0; c < 3; c++) wdd[(size_t)(c * 21 + s0 * 3 + k0) * S + p] = o3[c];
            wdt[(size_t)(s0 * 3 + k0) * S + p] = e1[0] * o3[0] + e1[1] * o3[1] + e1[2] * o3[2];
            wdt[(size_t)(21 + s0 * 3 + k0) * S + p] = e2[0] * o3[0] + e2[1] * o3[1] + e2[2] * o3[2];
        }
        double o3[3];
        divm_nf<false>(
            gu, p, 0, nf, pole, [&](int, int) { return 0.0; }, [&](int s) { return s == s0 ? 1.0 : 0.0; }, zero, o3);
        const double dz0 = 1.0 / (gu.Alth[0] - gu.Alth[1]);
        for (int c = 0; c < 3; c++) udd[(size_t)(c * 7 + s0) * S + p] = o3[c] / dz0;
        const double gx = gu.grad[(size_t)(s0 * 3) * S + p], gy = gu.grad[(size_t)(s0 * 3 + 1) * S + p],
                     gz = gu.grad[(size_t)(s0 * 3 + 2) * S + p];
        wgt[(size_t)s0 * S + p] = e1[0] * gx + e1[1] * gy + e1[2] * gz;
        wgt[(size_t)(7 + s0) * S + p] = e2[0] * gx + e2[1] * gy + e2[2] * gz;
    }
}

// The level loop of a chunked kernel: level lev is computed from one LDS buffer
// while lev + 1 is put into the other and lev + 2 is being loaded.
#define LW_LOOP()                                   \
    In A, B;                                        \
    load(A, l0);                                    \
    load(B, min(l0 + 1, l1 - 1));                   \
    put(A, 0);                                      \
    __syncthreads();                                \
    for (int lev = l0; lev < l1; lev += 2) {        \
        body(lev, B, A);                            \
        if (lev + 1 < l1) body(lev + 1, A, B);      \
    }

// Divergence-damping pass 0 (DivM_Op, thor_div.h:49-315) on the deviations Mhs /
// Whs, or with STAGE on the stage values Mhk / Whk. Bound by its field traffic
// (7 doubles per cell: M 3 and W in, 3 out) and the 84 weights per point and chunk,
// read from L2.
template <bool STAGE>
__global__ __launch_bounds__(256, 2) void k_divm0_lw(Geo g, Fields f, int lc) {
#pragma clang fp contract(fast)
    int r, l0, l1;
    if (!block_tile_lc(g, lc, r, l0, l1)) return;
    const size_t S = g.S;
    const int nv = g.nv;
    const double *Mv = STAGE ? f.Mhk : f.Mhs, *Wv = STAGE ? f.Whk : f.Whs;
    if (r == g.nr) {
        PoleCtx c;
        int lev;
        if (!pole_ctx_lc(g, l0, l1, c, lev)) return;
        const int p = c.p;
        const double rs = rscale_at(g, lev), rs2 = rs * rs, rdz = rs / (g.Alth[lev] - g.Alth[lev + 1]);
        double o[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int s = 0; s < 7; s++) {
            const int q = c.gi(s);
            const double dw = (LVP(Wv, lev, q) - LVP(Wv, lev + 1, q)) * rdz;
            for (int cc = 0; cc < 3; cc++) {
                double sum = 0.0;
                for (int k = 0; k < 3; k++) sum += g.wdd64[(size_t)(cc * 21 + s * 3 + k) * S + p] * VEC(Mv, k, lev, q);
                o[cc] += rs2 * sum + g.udd64[(size_t)(cc * 7 + s) * S + p] * dw;
            }
        }
        for (int k = 0; k < 3; k++) VEC(f.divg, k, lev, p) = o[k];
        return;
    }
    // staged point: (M_x, M_y) and (M_z, (Wl - Wt) rs^-1 dz), two 16-byte LDS words
    __shared__ double2 sA[2][NHL2], sB[2][NHL2];
    __shared__ double sRs2[kLcMax], sDz[kLcMax];
    if ((int)threadIdx.x < l1 - l0) {
        const int lev = l0 + threadIdx.x;
        const double rs = rscale_at(g, lev);
        sRs2[threadIdx.x] = rs * rs;
        sDz[threadIdx.x] = rs / (g.Alth[lev] - g.Alth[lev + 1]);
    }
    const LcThread T = lc_thread(g, r);
    const int p = T.p;
    double wd[63], wu[21];
    load_packed(g.pwd64, S, p, wd);
    load_packed(g.pwu64, S, p, wu);
    const size_t pl8 = S * 8;
    const auto rM = rsrc(Mv, 3 * nv * pl8), rW = rsrc(Wv, (nv + 1) * pl8), rD = rsrc(f.divg, 3 * nv * pl8);
    struct In {
        double om[3], hm[3], ow, hw;  // momentum and the top interface's W
    };
    auto load = [&](In &v, int lev) {
#pragma unroll
        for (int k = 0; k < 3; k++) {
            v.om[k] = ldb_d(rM, T.o8, (unsigned)((k * nv + lev) * pl8));
            v.hm[k] = ldb_d(rM, T.h8, (unsigned)((k * nv + lev) * pl8));
        }
        v.ow = ldb_d(rW, T.o8, (unsigned)((lev + 1) * pl8));
        v.hw = ldb_d(rW, T.h8, (unsigned)((lev + 1) * pl8));
    };
    double owl = ldb_d(rW, T.o8, (unsigned)(l0 * pl8)), hwl = ldb_d(rW, T.h8, (unsigned)(l0 * pl8));
    auto put = [&](const In &v, int b) {
        sA[b][T.ir] = make_double2(v.om[0], v.om[1]);
        sB[b][T.ir] = make_double2(v.om[2], owl - v.ow);
        owl = v.ow;
        if (T.hp >= 0) {
            sA[b][T.hp] = make_double2(v.hm[0], v.hm[1]);
            sB[b][T.hp] = make_double2(v.hm[2], hwl - v.hw);
        }
        hwl = v.hw;
    };
    auto body = [&](int lev, In &R, In &L) {
        load(L, min(lev + 2, l1 - 1));
        const int b = (lev - l0) & 1;
        const double rs2 = sRs2[lev - l0], rdz = sDz[lev - l0];
        double o[3] = {0.0, 0.0, 0.0}, u[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int s = 0; s < 7; s++) {
            const double2 a = sA[b][T.pos[s]], q = sB[b][T.pos[s]];
#pragma unroll
            for (int c = 0; c < 3; c++) {
                o[c] += wd[c * 21 + s * 3] * a.x;
                o[c] += wd[c * 21 + s * 3 + 1] * a.y;
                o[c] += wd[c * 21 + s * 3 + 2] * q.x;
                u[c] += wu[c * 7 + s] * q.y;
            }
        }
#pragma unroll
        for (int c = 0; c < 3; c++) stb_d(rD, T.o8, (unsigned)((c * nv + lev) * pl8), rs2 * o[c] + rdz * u[c]);
        if (lev + 1 < l1) put(R, b ^ 1);
        __syncthreads();
    };
    LW_LOOP()
}

// Divergence-damping pass 1 on the deviations + Momentum_Eq
// (thor_fastmodes.h:54-253). Both the damping and the pressure gradient are
// projected on the tangent plane, so only their two components along the
// point's tangent basis are formed (56 weights instead of 84).
__global__ __launch_bounds__(256, 2) void k_momentum_lw(Geo g, Fields f, int divdamp, double dt, int lc) {
#pragma clang fp contract(fast)
    int r, l0, l1;
    if (!block_tile_lc(g, lc, r, l0, l1)) return;
    const size_t S = g.S;
    const int nv = g.nv;
    if (r == g.nr) {
        PoleCtx c;
        int lev;
        if (!pole_ctx_lc(g, l0, l1, c, lev)) return;
        const int p = c.p;
        const double rs = rscale_at(g, lev), kz = rs * rs * g.Kdhz[lev];
        double t[2];
        for (int e = 0; e < 2; e++) {
            double sg = 0.0, sd = 0.0, sm = 0.0;
#pragma unroll
            for (int s = 0; s < 7; s++) {
                const int q = c.gi(s);
                sg += g.wgt64[(size_t)(e * 7 + s) * S + p] * LVP(f.ps, lev, q);
                if (divdamp)
                    for (int k = 0; k < 3; k++)
                        sd += g.wdt64[(size_t)(e * 21 + s * 3 + k) * S + p] * VEC(f.divg, k, lev, q);
            }
            for (int k = 0; k < 3; k++) sm += g.et64[(size_t)(e * 3 + k) * S + p] * VEC(f.SlowMh, k, lev, p);
            t[e] = (sm - rs * sg - kz * sd) * dt;
        }
        for (int k = 0; k < 3; k++)
            VEC(f.Mhs, k, lev, p) += t[0] * g.et64[(size_t)k * S + p] + t[1] * g.et64[(size_t)(3 + k) * S + p];
        return;
    }
    // staged point: (divg_x, divg_y) and (divg_z, ps)
    __shared__ double2 sA[2][NHL2], sB[2][NHL2];
    __shared__ double sRs[kLcMax], sKz[kLcMax];
    if ((int)threadIdx.x < l1 - l0) {
        const int lev = l0 + threadIdx.x;
        const double rs = rscale_at(g, lev);
        sRs[threadIdx.x] = rs;
        sKz[threadIdx.x] = rs * rs * g.Kdhz[lev];
    }
    const LcThread T = lc_thread(g, r);
    const int p = T.p;
    double wd[42] = {}, wg[20];  // wg: gradient, then the tangent basis
    if (divdamp) load_packed(g.pwt64, S, p, wd);
    load_packed(g.pwg64, S, p, wg);
    const double *e = wg + 14;
    const size_t pl8 = S * 8;
    // without damping the divg loads fall outside an empty buffer and return 0
    const auto rG = rsrc(f.divg, divdamp ? 3 * nv * pl8 : 0), rP = rsrc(f.ps, nv * pl8), rS = rsrc(f.SlowMh, 3 * nv * pl8),
               rM = rsrc(f.Mhs, 3 * nv * pl8);
    struct In {
        double sm[3], mh[3], og[3], op, hg[3], hpv;
    };
    auto load = [&](In &v, int lev) {
#pragma unroll
        for (int k = 0; k < 3; k++) {
            v.sm[k] = ldb_d(rS, T.o8, (unsigned)((k * nv + lev) * pl8));
            v.mh[k] = ldb_d(rM, T.o8, (unsigned)((k * nv + lev) * pl8));
        }
#pragma unroll
        for (int k = 0; k < 3; k++) {
            v.og[k] = ldb_d(rG, T.o8, (unsigned)((k * nv + lev) * pl8));
            v.hg[k] = ldb_d(rG, T.h8, (unsigned)((k * nv + lev) * pl8));
        }
        v.op = ldb_d(rP, T.o8, (unsigned)(lev * pl8));
        v.hpv = ldb_d(rP, T.h8, (unsigned)(lev * pl8));
    };
    auto put = [&](const In &v, int b) {
        sA[b][T.ir] = make_double2(v.og[0], v.og[1]);
        sB[b][T.ir] = make_double2(v.og[2], v.op);
        if (T.hp >= 0) {
            sA[b][T.hp] = make_double2(v.hg[0], v.hg[1]);
            sB[b][T.hp] = make_double2(v.hg[2], v.hpv);
        }
    };
    auto body = [&](int lev, In &R, In &L) {
        const double s1 = e[0] * L.sm[0] + e[1] * L.sm[1] + e[2] * L.sm[2];
        const double s2 = e[3] * L.sm[0] + e[4] * L.sm[1] + e[5] * L.sm[2];
        const double mh[3] = {L.mh[0], L.mh[1], L.mh[2]};
        load(L, min(lev + 2, l1 - 1));
        const int b = (lev - l0) & 1;
        double d1 = 0.0, d2 = 0.0, g1 = 0.0, g2 = 0.0;
#pragma unroll
        for (int s = 0; s < 7; s++) {
            const double2 a = sA[b][T.pos[s]], q = sB[b][T.pos[s]];
            d1 += wd[s * 3] * a.x;
            d2 += wd[21 + s * 3] * a.x;
            d1 += wd[s * 3 + 1] * a.y;
            d2 += wd[21 + s * 3 + 1] * a.y;
            d1 += wd[s * 3 + 2] * q.x;
            d2 += wd[21 + s * 3 + 2] * q.x;
            g1 += wg[s] * q.y;
            g2 += wg[7 + s] * q.y;
        }
        const double rs = sRs[lev - l0], kz = sKz[lev - l0];
        const double t1 = (s1 - rs * g1 - kz * d1) * dt, t2 = (s2 - rs * g2 - kz * d2) * dt;
#pragma unroll
        for (int k = 0; k < 3; k++)
            stb_d(rM, T.o8, (unsigned)((k * nv + lev) * pl8), mh[k] + (t1 * e[k] + t2 * e[3 + k]));
        if (lev + 1 < l1) put(R, b ^ 1);
        __syncthreads();
    };
    LW_LOOP()
}

// Divergence-damping pass 1 of the slow part (thor_slowmodes.h:82-105) into dm
// [3][nv], for k_slow_w<false>.
__global__ __launch_bounds__(256, 3) void k_divm1_lw(Geo g, Fields f, double *dm, int lc) {
#pragma clang fp contract(fast)
    int r, l0, l1;
    if (!block_tile_lc(g, lc, r, l0, l1)) return;
    const size_t S = g.S;
    const int nv = g.nv;
    if (r == g.nr) {
        PoleCtx c;
        int lev;
        if (!pole_ctx_lc(g, l0, l1, c, lev)) return;
        const double rs = rscale_at(g, lev), kz = -(rs * rs) * g.Kdhz[lev];
        double t[2] = {0.0, 0.0};
#pragma unroll
        for (int s = 0; s < 7; s++)
#pragma unroll
            for (int k = 0; k < 3; k++) {
                const double a = VEC(f.divg, k, lev, c.gi(s));
                t[0] += g.wdt64[(size_t)(s * 3 + k) * S + c.p] * a;
                t[1] += g.wdt64[(size_t)(21 + s * 3 + k) * S + c.p] * a;
            }
        for (int k = 0; k < 3; k++)
            VEC(dm, k, lev, c.p) = kz * (t[0] * g.et64[(size_t)k * S + c.p] + t[1] * g.et64[(size_t)(3 + k) * S + c.p]);
        return;
    }
    __shared__ double2 sA[2][NHL2];
    __shared__ double sB[2][NHL2], sKz[kLcMax];
    if ((int)threadIdx.x < l1 - l0) {
        const int lev = l0 + threadIdx.x;
        const double rs = rscale_at(g, lev);
        sKz[threadIdx.x] = -(rs * rs) * g.Kdhz[lev];
    }
    const LcThread T = lc_thread(g, r);
    const int p = T.p;
    double wd[42], e[6];
    load_packed(g.pwt64, S, p, wd);
#pragma unroll
    for (int i = 0; i < 6; i++) e[i] = g.et64[(size_t)i * S + p];
    const size_t pl8 = S * 8;
    const auto rG = rsrc(f.divg, 3 * nv * pl8), rD = rsrc(dm, 3 * nv * pl8);
    struct In {
        double og[3], hg[3];
    };
    auto load = [&](In &v, int lev) {
#pragma unroll
        for (int k = 0; k < 3; k++) {
            v.og[k] = ldb_d(rG, T.o8, (unsigned)((k * nv + lev) * pl8));
            v.hg[k] = ldb_d(rG, T.h8, (unsigned)((k * nv + lev) * pl8));
        }
    };
    auto put = [&](const In &v, int b) {
        sA[b][T.ir] = make_double2(v.og[0], v.og[1]);
        sB[b][T.ir] = v.og[2];
        if (T.hp >= 0) {
            sA[b][T.hp] = make_double2(v.hg[0], v.hg[1]);
            sB[b][T.hp] = v.hg[2];
        }
    };
    auto body = [&](int lev, In &R, In &L) {
        load(L, min(lev + 2, l1 - 1));
        const int b = (lev - l0) & 1;
        double d1 = 0.0, d2 = 0.0;
#pragma unroll
        for (int s = 0; s < 7; s++) {
            const double2 a = sA[b][T.pos[s]];
            const double z = sB[b][T.pos[s]];
            d1 += wd[s * 3] * a.x;
            d2 += wd[21 + s * 3] * a.x;
            d1 += wd[s * 3 + 1] * a.y;
            d2 += wd[21 + s * 3 + 1] * a.y;
            d1 += wd[s * 3 + 2] * z;
            d2 += wd[21 + s * 3 + 2] * z;
        }
        const double kz = sKz[lev - l0];
#pragma unroll
        for (int k = 0; k < 3; k++)
            stb_d(rD, T.o8, (unsigned)((k * nv + lev) * pl8), kz * (d1 * e[k] + d2 * e[3 + k]));
        if (lev + 1 < l1) put(R, b ^ 1);
        __syncthreads();
    };
    LW_LOOP()
}

// Horizontal advection (Compute_Advec_Cori1, thor_adv_cor.h:51-235) added to
// the vertical part, and the first Laplacian pass of the hyperdiffusion
// (thor_diff.h:54-522). Each staged point carries u = M / rho, v = u + (W / rho) r,
// rho, W / rho and T; a slot's mass flux div . M is formed once and multiplies
// the three components of v, and every Laplacian is a difference form.
__global__ __launch_bounds__(256, 2) void k_adv_diff1_lw(Geo g, Fields f, int hydiff, int lc) {
#pragma clang fp contract(fast)
    int r, l0, l1;
    if (!block_tile_lc(g, lc, r, l0, l1)) return;
    const size_t S = g.S;
    const int nv = g.nv;
    const double cT = g.energy ? g.Cp - g.Rd : g.Rd;  // variable 5: internal energy (thor_diff.h:196-202) or Rd T
    if (r == g.nr) {
        PoleCtx c;
        int lev;
        if (!pole_ctx_lc(g, l0, l1, c, lev)) return;
        const int p = c.p;
        const double rs = rscale_at(g, lev);
        double adv[3] = {0.0, 0.0, 0.0}, lap[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, a0[6];
#pragma unroll
        for (int s = 0; s < 7; s++) {
            const int q = c.gi(s);
            const double rho = LVP(f.Rhok, lev, q), wr = LVP(f.Wk, lev, q) / rho;
            double u[3], mf = 0.0;
            for (int k = 0; k < 3; k++) {
                const double m = VEC(f.Mhk, k, lev, q);
                u[k] = m / rho;
                mf += g.div[(size_t)(s * 3 + k) * S + p] * m;
            }
            for (int k = 0; k < 3; k++) adv[k] += (u[k] + wr * g.fr[(size_t)k * S + q]) * mf;
            const double a[6] = {rho, u[0], u[1], u[2], wr, LVP(f.T, lev, q)};
            for (int v = 0; v < 6; v++) {
                if (s == 0) a0[v] = a[v];
                else lap[v] += g.wlap64[(size_t)(s - 1) * S + p] * (a[v] - a0[v]);
            }
        }
        for (int k = 0; k < 3; k++) VEC(f.Adv, k, lev, p) += rs * adv[k];
        if (hydiff)
            for (int v = 0; v < 6; v++) VEC(f.diff, v, lev, p) = (v == 5 ? cT : 1.0) * (rs * rs) * lap[v];
        return;
    }
    // staged point: (u_x, u_y), (u_z, rho), (v_x, v_y), (v_z, W / rho), T
    __shared__ double2 sU[2][NHL2], sR[2][NHL2], sV[2][NHL2], sW[2][NHL2];
    __shared__ double sT[2][NHL2], sRs[kLcMax];
    if ((int)threadIdx.x < l1 - l0) sRs[threadIdx.x] = rscale_at(g, l0 + threadIdx.x);
    const LcThread T = lc_thread(g, r);
    const int p = T.p;
    double wd[21], wl[6];
    load_packed(g.pdiv, S, p, wd);
#pragma unroll
    for (int s = 0; s < 6; s++) wl[s] = g.wlap64[(size_t)s * S + p];
    const int qh = T.hp >= 0 ? g.halo[r * NHALO + threadIdx.x] : -1;
    double ofr[3], hfr[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        ofr[k] = g.fr[(size_t)k * S + p];
        hfr[k] = qh >= 0 ? g.fr[(size_t)k * S + qh] : 0.0;
    }
    const size_t pl8 = S * 8;
    const auto rAd = rsrc(f.Adv, 3 * nv * pl8), rD0 = rsrc(f.diff, 3 * nv * pl8),
               rD1 = rsrc(f.diff + 3 * nv * S, 3 * nv * pl8), rM = rsrc(f.Mhk, 3 * nv * pl8), rRk = rsrc(f.Rhok, nv * pl8),
               rWk = rsrc(f.Wk, nv * pl8), rTk = rsrc(f.T, nv * pl8);
    struct In {
        double adv[3], om[3], orho, ow, ot, hm[3], hrho, hw, ht;
    };
    auto load = [&](In &v, int lev) {
#pragma unroll
        for (int k = 0; k < 3; k++) {
            v.adv[k] = ldb_d(rAd, T.o8, (unsigned)((k * nv + lev) * pl8));
            v.om[k] = ldb_d(rM, T.o8, (unsigned)((k * nv + lev) * pl8));
            v.hm[k] = ldb_d(rM, T.h8, (unsigned)((k * nv + lev) * pl8));
        }
        const unsigned l8 = (unsigned)(lev * pl8);
        v.orho = ldb_d(rRk, T.o8, l8);
        v.hrho = ldb_d(rRk, T.h8, l8);
        v.ow = ldb_d(rWk, T.o8, l8);
        v.hw = ldb_d(rWk, T.h8, l8);
        v.ot = ldb_d(rTk, T.o8, l8);
        v.ht = ldb_d(rTk, T.h8, l8);
    };
    auto put1 = [&](int b, int pos, const double m[3], double rho, double w, double t, const double fr[3]) {
        const double wr = w / rho, ux = m[0] / rho, uy = m[1] / rho, uz = m[2] / rho;
        sU[b][pos] = make_double2(ux, uy);
        sR[b][pos] = make_double2(uz, rho);
        sV[b][pos] = make_double2(ux + wr * fr[0], uy + wr * fr[1]);
        sW[b][pos] = make_double2(uz + wr * fr[2], wr);
        sT[b][pos] = t;
    };
    auto put = [&](const In &v, int b) {
        put1(b, T.ir, v.om, v.orho, v.ow, v.ot, ofr);
        // a missing pentagon corner is never read; its loads returned 0
        if (qh >= 0) put1(b, T.hp, v.hm, v.hrho, v.hw, v.ht, hfr);
    };
    auto body = [&](int lev, In &R, In &L) {
        const double adv[3] = {L.adv[0], L.adv[1], L.adv[2]};
        load(L, min(lev + 2, l1 - 1));
        const int b = (lev - l0) & 1;
        double ad[3] = {0.0, 0.0, 0.0}, a0[6], lap[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int s = 0; s < 7; s++) {
            const int q = T.pos[s];
            const double2 u = sU[b][q], ur = sR[b][q], v = sV[b][q], vw = sW[b][q];
            const double mf = ur.y * (wd[s * 3] * u.x + wd[s * 3 + 1] * u.y + wd[s * 3 + 2] * ur.x);
            ad[0] += v.x * mf;
            ad[1] += v.y * mf;
            ad[2] += vw.x * mf;
            const double a[6] = {ur.y, u.x, u.y, ur.x, vw.y, sT[b][q]};
#pragma unroll
            for (int i = 0; i < 6; i++) {
                if (s == 0) a0[i] = a[i];
                else lap[i] += wl[s - 1] * (a[i] - a0[i]);
            }
        }
        const double rs = sRs[lev - l0], rs2 = rs * rs;
#pragma unroll
        for (int k = 0; k < 3; k++) stb_d(rAd, T.o8, (unsigned)((k * nv + lev) * pl8), adv[k] + rs * ad[k]);
        if (hydiff) {
#pragma unroll
            for (int i = 0; i < 3; i++) {
                stb_d(rD0, T.o8, (unsigned)((i * nv + lev) * pl8), rs2 * lap[i]);
                stb_d(rD1, T.o8, (unsigned)((i * nv + lev) * pl8), (i == 2 ? cT * rs2 : rs2) * lap[3 + i]);
            }
        }
        if (lev + 1 < l1) put(R, b ^ 1);
        __syncthreads();
    };
    LW_LOOP()
}

// A further hyperdiffusion pass of the six fields src. LAST: the last one with
// Correct_Horizontal (thor_diff.h:524-915, variables 1..5 weighted by the stage
// density, scaled by -Kdh4 sign, the diffusive sponge added, the radial part
// of the momentum removed) into diffmh, diffw, diffrh, diffpr; else an
// intermediate pass of HyDiffOrder >= 6 into dst.
template <bool LAST>
__global__ __launch_bounds__(256, 3) void k_diff_lw(Geo g, Fields f, const double *src, double *dst, double sign,
                                                    int lc) {
#pragma clang fp contract(fast)
    int r, l0, l1;
    if (!block_tile_lc(g, lc, r, l0, l1)) return;
    const size_t S = g.S;
    const int nv = g.nv;
    if (r == g.nr) {
        PoleCtx c;
        int lev;
        if (!pole_ctx_lc(g, l0, l1, c, lev)) return;
        const int p = c.p;
        const double rs = rscale_at(g, lev);
        double out[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, a0[6];
#pragma unroll
        for (int s = 0; s < 7; s++) {
            const int q = c.gi(s);
            const double rho = LAST ? LVP(f.Rhok, lev, q) : 1.0;
            for (int v = 0; v < 6; v++) {
                const double a = VEC(src, v, lev, q) * (v == 0 ? 1.0 : rho);
                if (s == 0) a0[v] = a;
                else out[v] += g.wlap64[(size_t)(s - 1) * S + p] * (a - a0[v]);
            }
        }
        for (int v = 0; v < 6; v++) out[v] *= rs * rs;
        if constexpr (LAST) diff2_tail<false>(g, f, p, lev, true, sign, out, LV(f.Rhok, lev));
        else
            for (int v = 0; v < 6; v++) VEC(dst, v, lev, p) = out[v];
        return;
    }
    __shared__ double2 sA[2][3][NHL2];  // variables (0, 1), (2, 3), (4, 5) of a point
    __shared__ double sK[kLcMax];
    if ((int)threadIdx.x < l1 - l0) {
        const int lev = l0 + threadIdx.x;
        const double rs = rscale_at(g, lev);
        sK[threadIdx.x] = LAST ? rs * rs * (-g.Kdh4[lev] * sign) : rs * rs;
    }
    const LcThread T = lc_thread(g, r);
    const int p = T.p;
    double wl[6];
#pragma unroll
    for (int s = 0; s < 6; s++) wl[s] = g.wlap64[(size_t)s * S + p];
    const double fx = g.fr[p], fy = g.fr[S + p], fz = g.fr[2 * S + p];
    const size_t pl8 = S * 8;
    const auto r0 = rsrc(src, 3 * nv * pl8), r1 = rsrc(src + 3 * nv * S, 3 * nv * pl8), rR = rsrc(f.Rhok, nv * pl8);
    const auto q0 = rsrc(LAST ? f.diffmh : dst, 3 * nv * pl8),
               q1 = rsrc(LAST ? f.diffrh : dst + 3 * nv * S, (LAST ? 1 : 3) * nv * pl8), q2 = rsrc(f.diffw, nv * pl8),
               q3 = rsrc(f.diffpr, nv * pl8);
    struct In {
        double od[6], hd[6], orho, hrho;
    };
    auto load = [&](In &v, int lev) {
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const unsigned o = (unsigned)((k * nv + lev) * pl8);
            v.od[k] = ldb_d(r0, T.o8, o);
            v.od[3 + k] = ldb_d(r1, T.o8, o);
            v.hd[k] = ldb_d(r0, T.h8, o);
            v.hd[3 + k] = ldb_d(r1, T.h8, o);
        }
        if constexpr (LAST) {
            v.orho = ldb_d(rR, T.o8, (unsigned)(lev * pl8));
            v.hrho = ldb_d(rR, T.h8, (unsigned)(lev * pl8));
        }
    };
    auto put1 = [&](int b, int pos, const double d[6], double rho) {
        const double q = LAST ? rho : 1.0;
        sA[b][0][pos] = make_double2(d[0], d[1] * q);
        sA[b][1][pos] = make_double2(d[2] * q, d[3] * q);
        sA[b][2][pos] = make_double2(d[4] * q, d[5] * q);
    };
    auto put = [&](const In &v, int b) {
        put1(b, T.ir, v.od, v.orho);
        if (T.hp >= 0) put1(b, T.hp, v.hd, v.hrho);
    };
    auto body = [&](int lev, In &R, In &L) {
        const double rho = L.orho;
        load(L, min(lev + 2, l1 - 1));
        const int b = (lev - l0) & 1;
        double out[6];
#pragma unroll
        for (int h = 0; h < 3; h++) {
            const double2 a0 = sA[b][h][T.pos[0]];
            double x = 0.0, y = 0.0;
#pragma unroll
            for (int s = 1; s < 7; s++) {
                const double2 a = sA[b][h][T.pos[s]];
                x += wl[s - 1] * (a.x - a0.x);
                y += wl[s - 1] * (a.y - a0.y);
            }
            out[2 * h] = sK[lev - l0] * x;
            out[2 * h + 1] = sK[lev - l0] * y;
        }
        if constexpr (LAST) {
            if (f.dsp) {  // diffusive sponge, as diff2_tail
                const double k2 = g.ssp * rho * g.Kdh2[lev] * g.dsp_scale;
                for (int var = 1; var <= 4; var++) out[var] += k2 * VEC(f.dsp, var, lev, p);
            }
            const unsigned l8 = (unsigned)(lev * pl8);
            stb_d(q1, T.o8, l8, out[0]);
            stb_d(q2, T.o8, l8, out[4]);
            stb_d(q3, T.o8, l8, out[5]);
            const double dr = fx * out[1] + fy * out[2] + fz * out[3];
            stb_d(q0, T.o8, l8, out[1] - fx * dr);
            stb_d(q0, T.o8, (unsigned)((nv + lev) * pl8), out[2] - fy * dr);
            stb_d(q0, T.o8, (unsigned)((2 * nv + lev) * pl8), out[3] - fz * dr);
        } else {
#pragma unroll
            for (int k = 0; k < 3; k++) {
                const unsigned o = (unsigned)((k * nv + lev) * pl8);
                stb_d(q0, T.o8, o, out[k]);
                stb_d(q1, T.o8, o, out[3 + k]);
            }
        }
        if (lev + 1 < l1) put(R, b ^ 1);
        __syncthreads();
    };
    LW_LOOP()
}

// Prepare_Implicit_Vertical (thor_vertical_int.h:566-771) and the horizontal
// flux divergences of Density_Pressure_Eqs with the stage part of the pressure
// flux divergence taken from f.hflx_ptk (k_slow_w) and Sd left to
// the vertical solve, as k_prepare_lc<true>: the stage momentum is not read
// and one plane less is written in every substep (10 doubles per cell instead
// of 14: 63 -> 45 us at 40 962 x 48, 19.4 -> 14.2 at 10 242 x 40).
__global__ __launch_bounds__(256, 2) void k_prepare_lw(Geo g, Fields f, int lc) {
#pragma clang fp contract(fast)
    int r, l0, l1;
    if (!block_tile_lc(g, lc, r, l0, l1)) return;
    const size_t S = g.S;
    const int nv = g.nv;
    const double RoC = g.Rd / (g.Cp - g.Rd);
    if (r == g.nr) {
        PoleCtx c;
        int lev;
        if (pole_ctx_lc(g, l0, l1, c, lev))
            prepare_point<kPoleUnroll>(
                g, f, c.p, lev, [&](int s, int k) { return VEC(f.Mhs, k, lev, c.gi(s)); },
                [&](int s) { return LVP(f.h, lev, c.gi(s)); },
                [&](int s, int k) { return VEC(f.Mhs, k, lev, c.gi(s)) + VEC(f.Mhk, k, lev, c.gi(s)); },
                [&](int s) { return LVP(f.pt, lev, c.gi(s)); });
        return;
    }
    // staged point: (M_x, M_y), (M_z, h), pt
    __shared__ double2 sA[2][NHL2], sB[2][NHL2];
    __shared__ double sT[2][NHL2], sRs[kLcMax];
    if ((int)threadIdx.x < l1 - l0) sRs[threadIdx.x] = rscale_at(g, l0 + threadIdx.x);
    const LcThread T = lc_thread(g, r);
    const int p = T.p;
    double wv[21];
    load_packed(g.pdiv, S, p, wv);
    const size_t pl8 = S * 8;
    const auto rM = rsrc(f.Mhs, 3 * nv * pl8), rH = rsrc(f.h, nv * pl8), rPt = rsrc(f.pt, nv * pl8),
               rSp = rsrc(f.Slowp, nv * pl8), rPk = rsrc(f.hflx_ptk, nv * pl8), wSp = rsrc(f.Sp, nv * pl8),
               wFr = rsrc(f.hflx_r, nv * pl8), wFp = rsrc(f.hflx_pt, nv * pl8);
    struct In {
        double slowp, ptk, om[3], hm[3], oh, hh, opt, hpt;
    };
    auto load = [&](In &v, int lev) {
        const unsigned l8 = (unsigned)(lev * pl8);
        v.slowp = ldb_d(rSp, T.o8, l8);
        v.ptk = ldb_d(rPk, T.o8, l8);
#pragma unroll
        for (int k = 0; k < 3; k++) {
            v.om[k] = ldb_d(rM, T.o8, (unsigned)((k * nv + lev) * pl8));
            v.hm[k] = ldb_d(rM, T.h8, (unsigned)((k * nv + lev) * pl8));
        }
        v.oh = ldb_d(rH, T.o8, l8);
        v.opt = ldb_d(rPt, T.o8, l8);
        v.hh = ldb_d(rH, T.h8, l8);
        v.hpt = ldb_d(rPt, T.h8, l8);
    };
    auto put = [&](const In &v, int b) {
        sA[b][T.ir] = make_double2(v.om[0], v.om[1]);
        sB[b][T.ir] = make_double2(v.om[2], v.oh);
        sT[b][T.ir] = v.opt;
        if (T.hp >= 0) {
            sA[b][T.hp] = make_double2(v.hm[0], v.hm[1]);
            sB[b][T.hp] = make_double2(v.hm[2], v.hh);
            sT[b][T.hp] = v.hpt;
        }
    };
    auto body = [&](int lev, In &R, In &L) {
        const double slowp = L.slowp, ptk = L.ptk;
        load(L, min(lev + 2, l1 - 1));
        const int b = (lev - l0) & 1;
        double sr = 0.0, sp = 0.0, st = 0.0;
#pragma unroll
        for (int s = 0; s < 7; s++) {
            const double2 a = sA[b][T.pos[s]], q = sB[b][T.pos[s]];
            const double d = wv[s * 3] * a.x + wv[s * 3 + 1] * a.y + wv[s * 3 + 2] * q.x;
            sr += d;
            sp += d * q.y;
            st += d * sT[b][T.pos[s]];
        }
        const double rs = sRs[lev - l0];
        const unsigned l8 = (unsigned)(lev * pl8);
        stb_d(wSp, T.o8, l8, slowp - RoC * rs * sp);
        stb_d(wFr, T.o8, l8, rs * sr);
        stb_d(wFp, T.o8, l8, ptk + rs * st);
        if (lev + 1 < l1) put(R, b ^ 1);
        __syncthreads();
    };
    LW_LOOP()
}
#undef LW_LOOP

} // namespace thor
