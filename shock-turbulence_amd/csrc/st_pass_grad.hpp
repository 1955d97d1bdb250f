// First-derivative passes of the right-hand side (one translation unit per
// direction: st_pass_gradx.hip, st_pass_gradz.hip, st_pass_grady.hip).
#pragma once

#include "st_pass.hpp"

namespace st {

// ---------------------------------------------------------------------
// P1: first derivatives, own-direction second derivatives and convective
// terms of one direction, from the state Q.
//   RHS_x  src/rhsv_periodic_sf.f:36-461
//   RHS_yz src/rhsv_periodic_sf.f:546-880 (y and z parts of the same terms)
// The load phase stages the primitives (u, v, w, T, rho) of
// src/rhsv_periodic_sf.f:92-104.  Per direction d (velocity u_d):
//   dQ_i += D1(-rho u_i u_d/2 - delta_id P) - D1(rho u_d) u_i/2
//           - (rho u_d/2) du_i/dx_d + w_id mu d2u_i/dx_d^2,  w_id = 4/3+bulk (i=d) else 1
//   dQ_4 += -D1(rho u_d)
//   dQ_5 += D1(-(rho T + rho |u|^2/2) u_d) + sum_i u_i w_id mu d2u_i/dx_d^2
//           + Pr^-1 (mu d2T/dx_d^2 + mu' (dT/dx_d)^2)
//   G(., d) = D1(u, v, w, T);  L2e += D2(T)/gamma   (e = T/gamma)
// D1 of a sum replaces the reference's sum of D1s of the same operator,
// rho*E + P = rho T + rho |u|^2 / 2, and D2(T)/gamma replaces D2(T/gamma);
// all three differ from the reference's evaluation only by rounding.
// ---------------------------------------------------------------------
// DIR: the sweep's direction, fixed at compile time, so that the operators
// are unrolled with every component known (a loop over them costs each
// accumulation a fused multiply-add per candidate row and each flux both of
// its forms: 606 -> 421 vector instructions per point of the x pass).
// MW: occupancy target (waves per SIMD) handed to the register allocator.
// CROSS (y lines, after the x and z passes have left their partial sums):
// the store phase also assembles the right-hand side of the first-derivative
// part -- the y terms, the z and x partials and the viscous terms built from
// products of first derivatives -- and |S| and C_beta, from the derivatives
// of all three directions at the point (the y ones carried from the early
// store in registers).  The viscosity is formed once per point, in the load
// phase, and staged in a slot of its own, which the compute phase and the
// store read.
// NMX: stored first derivatives staged as well, whose D1 along the sweep
// gives the mixed second derivatives of the viscous terms
// (src/rhsv_periodic_sf.f:1062-1070,1281-1363):
//   y (4): D1y of du/dx, dv/dx, dv/dz, dw/dz;  z (2): D1z of du/dx, dw/dx
// each times (1/3 + bulk) mu into the momentum component it belongs to and,
// times that velocity, into the energy.  The x sweep runs first, so the z
// and y sweeps find the derivatives they need.
// TWO (the z sweep, two rounds of staging): the two mixed inputs are staged in
// the slots of v and rho, whose values wait in registers (NHOLD) until the
// mixed terms are done (compute_a); five slots instead of seven.  At 8 points
// per lane 8-line tiles of 256 threads then fit two workgroups per CU (0.70 ->
// 0.645 ms at 256^3); at 4 to 7, 16-line tiles of 512 threads, which stream (128^3
// stage 710 -> 699 us), while on 256 threads the extra phase costs more than it
// gives (256^3 at 4 points per lane 0.70 -> 0.79 ms).
template <int DIR, int MW, bool TWO_ = false>
struct PassGrad {
    static constexpr bool TWO = TWO_, CROSS = DIR == 1;
    static constexpr int NMX = DIR == 0 ? 0 : DIR == 2 ? 2 : 4;
    static_assert(!TWO || NMX == 2, "two-round staging is the z sweep's");
    // slots: u, v, w, T, rho, the mixed inputs; CROSS: the viscosity
    static constexpr int NSLOT = TWO ? 5 : 5 + NMX + (CROSS ? 1 : 0), NOUT = 5, NEARLY = 5;
    static constexpr int MUSLOT = 9;
    static constexpr int NHOLD = TWO ? 2 : 0;
    // CROSS: u, v, w and T of each point go from the load phase to the late
    // store in registers (the store assembles the right-hand side from them)
    static constexpr int NLCARRY = CROSS ? 4 : 0;
    HD static constexpr int hold_slot(int j) { return j == 0 ? 1 : 4; }
    static constexpr bool REUSE = true;
    // (CROSS: the y derivatives and the Laplacian of e)
    static constexpr int NCARRY = CROSS ? 5 : 0;
    // CROSS: |S| and the Laplacian of e, complete here, are differentiated
    // twice along y while their lines are at hand (the first terms of Lap|S|
    // and Lap(Lap e)): a pass less, two fields fewer
    static constexpr int NPOST = CROSS ? 2 : 0;
    // CROSS: the staged inputs of the mixed terms (du/dx, dv/dx, dv/dz,
    // dw/dz) and the viscosity reach the store after the late results
    static constexpr int NKEEP = CROSS ? NMX + 1 : 0;
    static constexpr int MIN_WAVES = MW;
    static constexpr int STREAM = DIR == 2 && !TWO ? 0 : STREAM_LOADS | STREAM_STORES | (DIR == 1 ? STREAM_Y : 0);
    static constexpr int LOAD_UNROLL = 8;
    static constexpr int NPF = 0;
    // the additive LDS layout for the x and y sweeps (fewer address
    // registers: the x pass at 8 points per lane no longer spills, and the y
    // pass runs 2% faster) and for z at 8 points per lane; the swizzled one
    // for z at 4 points per lane, whose 4-line tiles would take 4-way bank
    // conflicts in the staging
    HD static constexpr bool lds_add(int m) { return NMX != 2 || m >= 8 || TWO; }
    // CROSS: the store phases' global reads (sfetch_early: the z and x
    // partials of the Laplacian of e; sfetch: four x and z derivatives, and
    // the z and x partial sums) go out for all the thread's points (two at a
    // time) before the first store
    static constexpr int NSFE = CROSS ? 2 : 0, NSF = CROSS ? 14 : 0, SF_BATCH = 2;
    template <class A>
    DEV static void prefetch(const Geo &, const A &, long, double *) {}
    // G index of mixed input m: y: gxx=0, gyx=1, gyz=7, gzz=8; z: gxx=0, gzx=2
    HD static constexpr int msrc(int m) { return NMX == 4 ? (m == 0 ? 0 : m == 1 ? 1 : m == 2 ? 7 : 8) : (m == 0 ? 0 : 2); }
    // momentum component that D1 of mixed input m feeds
    HD static constexpr int mdst(int m) { return NMX == 4 ? (m == 1 ? 0 : m == 2 ? 2 : 1) : (m == 0 ? 2 : 0); }
    // slot of mixed input m
    HD static constexpr int mslot(int m) { return TWO ? (m == 0 ? 1 : 4) : 5 + m; }
    template <class A>
    DEV static void load(const Geo &, const A &a, long gi, double (&v)[NSLOT + NHOLD + NLCARRY])
    {
        const Prim pr = prim(a.ph, a.Q[gi], a.Q[a.N + gi], a.Q[2 * a.N + gi], a.Q[3 * a.N + gi], a.Q[4 * a.N + gi]);
        v[0] = pr.u;
        v[2] = pr.w;
        v[3] = pr.T;
        if constexpr (CROSS) {
            v[MUSLOT] = visc(a.ph, pr.T);
            v[NSLOT] = pr.u;
            v[NSLOT + 1] = pr.v;
            v[NSLOT + 2] = pr.w;
            v[NSLOT + 3] = pr.T;
        }
        if constexpr (TWO) {
            v[5] = pr.v;
            v[6] = a.Q[3 * a.N + gi];
        } else {
            v[1] = pr.v;
            v[4] = a.Q[3 * a.N + gi];
        }
#pragma unroll
        for (int m = 0; m < NMX; m++) v[mslot(m)] = a.G[msrc(m) * a.N + gi];
    }

    // ---- the operators of one lane's M points ----
    // Each step below ends with a compiler fence, and its sums are pinned:
    // the slots are read again by the next step instead of being kept in
    // registers, and no step's tail is put off into a later one (without
    // either, the unrolled steps spill 250-390 registers).
    template <int M>
    DEV static void pin(double (&r)[M])
    {
#pragma unroll
        for (int k = 0; k < M; k++) asm volatile("" : "+v"(r[k]));
    }
    DEV static void fence()
    {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    }

    template <int M, int P, bool NP, bool AL, class F, class A>
    DEV static void d1(const A &a, const Lane<M, P, NP, AL> &L, const F &f, double (&r)[M])
    {
        double v[M], w[M + 2 * d_halo<NP, M>()];
#pragma unroll
        for (int k = 0; k < M; k++) v[k] = f(k);
        window<M>(v, L, w);
        op_d1<M>(w, a.K1, a.tab()->op[0], L, r);
    }
    // the viscosity: from its slot, or formed here (TWO: in compute_a, which
    // leaves it in the row of the continuity equation)
    template <int M, int P, bool NP, bool AL, class A>
    DEV static void viscosity(const A &a, const Lane<M, P, NP, AL> &L, double (&mu)[M])
    {
#pragma unroll
        for (int k = 0; k < M; k++) mu[k] = CROSS ? L.ld(MUSLOT, k) : visc(a.ph, L.ld(3, k));
    }
    // mixed-derivative term m into its momentum component and the energy
    // (SET: the first term of that row)
    template <int m, bool SET, bool SETE, int M, int P, bool NP, bool AL, class A>
    DEV static void mixed(const A &a, const Lane<M, P, NP, AL> &L, const double (&mu)[M], double (&out)[5][M])
    {
        if constexpr (m < NMX) {
            constexpr int comp = mdst(m);
            const double cb = a.ph.bulk + 1.0 / 3.0;
            double r[M];
            d1<M, P, NP>(a, L, [&](int k) { return L.ld(mslot(m), k); }, r);
#pragma unroll
            for (int k = 0; k < M; k++) {
                const double t = (cb * mu[k]) * r[k];
                out[comp][k] = SET ? t : out[comp][k] + t;
                out[4][k] = SETE ? L.ld(comp, k) * t : fma(L.ld(comp, k), t, out[4][k]);
            }
            pin<M>(out[comp]);
            pin<M>(out[4]);
            fence();
        }
    }
    template <int M, int P, bool NP, bool AL, class A>
    DEV static void mixed_all(const A &a, const Lane<M, P, NP, AL> &L, const double (&mu)[M], double (&out)[5][M])
    {
        if constexpr (NMX > 0) {
            mixed<0, true, true, M, P, NP>(a, L, mu, out);
            mixed<1, true, false, M, P, NP>(a, L, mu, out);
            mixed<2, true, false, M, P, NP>(a, L, mu, out);
            mixed<3, false, false, M, P, NP>(a, L, mu, out);
        }
    }
    // rows that the mixed terms have started: z: 2, 0, energy; y: 1, 0, 2, energy
    HD static constexpr bool started(int row) { return NMX == 4 ? row != 3 : NMX == 2 && (row == 0 || row == 2 || row == 4); }
    // TWO: the mixed terms, while their inputs hold the slots of v and rho.
    template <int M, int P, bool NP, bool AL, class A>
    DEV static void compute_a(const Geo &, const A &a, const Lane<M, P, NP, AL> &L, double (&out)[5][M])
    {
        viscosity<M, P, NP>(a, L, out[3]);
        mixed_all<M, P, NP>(a, L, out[3], out);
    }
    template <int ROW, int M>
    DEV static void add(double (&out)[5][M], const double (&r)[M])
    {
#pragma unroll
        for (int k = 0; k < M; k++) out[ROW][k] = started(ROW) ? out[ROW][k] + r[k] : r[k];
    }
    // momentum flux of component i (with the pressure in the sweep's own)
    template <int i, int M, int P, bool NP, bool AL, class A>
    DEV static void momentum(const A &a, const Lane<M, P, NP, AL> &L, double (&out)[5][M])
    {
        const double pfac = a.ph.gm1 * a.ph.ginv;
        double r[M];
        d1<M, P, NP>(a, L, [&](int k) {
            const double f = -0.5 * L.ld(4, k) * L.ld(i, k) * L.ld(DIR, k);
            return i == DIR ? f - L.ld(4, k) * L.ld(3, k) * pfac : f;
        }, r);
        add<i, M>(out, r);
        pin<M>(out[i]);
        fence();
    }
    // velocity i: second, then first derivatives; the latter takes its slot
    template <int i, int M, int P, bool NP, bool AL, class A>
    DEV static void velocity(const A &a, const Lane<M, P, NP, AL> &L, const double (&mu)[M], double (&out)[5][M])
    {
        const double wd = i == DIR ? 4.0 / 3.0 + a.ph.bulk : 1.0;
        constexpr int H = d_halo<NP, M>();
        double v[M], w[M + 2 * H], r[M];
#pragma unroll
        for (int k = 0; k < M; k++) v[k] = L.ld(i, k);
        window<M>(v, L, w);
        op_d2<M>(w, a.K2, a.tab()->op[1], L, r);
#pragma unroll
        for (int k = 0; k < M; k++) {
            const double vt = i == DIR ? wd * mu[k] * r[k] : mu[k] * r[k];
            out[i][k] += vt;
            out[4][k] = fma(w[H + k], vt, out[4][k]);
        }
        op_d1<M>(w, a.K1, a.tab()->op[0], L, r);
#pragma unroll
        for (int k = 0; k < M; k++) {
            const double rud = -0.5 * L.ld(4, k) * L.ld(DIR, k);
            out[i][k] = fma(rud, r[k], out[i][k]);
            L.st(i, k, r[k]);
        }
        pin<M>(out[i]);
        pin<M>(out[4]);
        fence();
    }

    // Operator order: the mixed terms; the fluxes and the mass flux, while u,
    // v, w, T and rho are all needed; then the velocities (u_d last), whose
    // slots take their derivatives; then T, whose slot takes dT/dx_d and
    // rho's slot the Laplacian of e.
    template <int M, int P, bool NP, bool AL, class A>
    DEV static void compute(const Geo &, const A &a, const Lane<M, P, NP, AL> &L, double (&out)[5][M])
    {
        const Phys &ph = a.ph;
        // the viscosity is held through the flux solves where the mixed terms
        // need it before them and it has no slot
        constexpr bool EARLY = NMX > 0 && !CROSS;
        double mu[M];
        if constexpr (TWO) {
#pragma unroll
            for (int k = 0; k < M; k++) mu[k] = out[3][k];
        } else if constexpr (NMX > 0) {
            viscosity<M, P, NP>(a, L, mu);
            mixed_all<M, P, NP>(a, L, mu, out);
        }
        momentum<0, M, P, NP>(a, L, out);
        momentum<1, M, P, NP>(a, L, out);
        momentum<2, M, P, NP>(a, L, out);
        // energy flux
        {
            double r[M];
            d1<M, P, NP>(a, L, [&](int k) {
                const double u = L.ld(0, k), v = L.ld(1, k), w = L.ld(2, k), rho = L.ld(4, k);
                const double ud = DIR == 0 ? u : DIR == 1 ? v : w;
                return -((rho * L.ld(3, k) + 0.5 * rho * (u * u + v * v + w * w)) * ud);
            }, r);
            add<4, M>(out, r);
            pin<M>(out[4]);
            fence();
        }
        // skew-symmetric part and continuity with the mass flux rho u_d
        {
            double r[M];
            d1<M, P, NP>(a, L, [&](int k) { return L.ld(4, k) * L.ld(DIR, k); }, r);
#pragma unroll
            for (int k = 0; k < M; k++) {
                const double t = -0.5 * r[k];
                out[0][k] = fma(t, L.ld(0, k), out[0][k]);
                out[1][k] = fma(t, L.ld(1, k), out[1][k]);
                out[2][k] = fma(t, L.ld(2, k), out[2][k]);
                out[3][k] = -r[k];
            }
#pragma unroll
            for (int i = 0; i < 4; i++) pin<M>(out[i]);
            fence();
        }
        if constexpr (!EARLY) viscosity<M, P, NP>(a, L, mu);
        velocity<(DIR + 1) % 3, M, P, NP>(a, L, mu, out);
        velocity<(DIR + 2) % 3, M, P, NP>(a, L, mu, out);
        velocity<DIR, M, P, NP>(a, L, mu, out);
        // T: first and second derivatives; the Laplacian of e = T/gamma is
        // D2(T)/gamma (the operator is linear).  CROSS: the store has mu' and
        // adds its term.
        {
            constexpr int H = d_halo<NP, M>();
            double v[M], w[M + 2 * H], r[M];
#pragma unroll
            for (int k = 0; k < M; k++) v[k] = L.ld(3, k);
            window<M>(v, L, w);
            op_d2<M>(w, a.K2, a.tab()->op[1], L, r);
#pragma unroll
            for (int k = 0; k < M; k++) {
                L.st(4, k, r[k] * ph.ginv);
                out[4][k] = fma(ph.pr_inv * mu[k], r[k], out[4][k]);
            }
            op_d1<M>(w, a.K1, a.tab()->op[0], L, r);
#pragma unroll
            for (int k = 0; k < M; k++) {
                L.st(3, k, r[k]);
                if constexpr (!CROSS) {
                    const double mup = dvisc(ph, w[H + k], mu[k]);
                    out[4][k] += ph.pr_inv * (mup * r[k] * r[k]);
                }
            }
        }
    }

    template <class A>
    DEV static void store_early(const Geo &g, const A &a, long gi, const double *v)
    {
#pragma unroll
        for (int c = 0; c < 3; c++) a.G[(g.dir * 3 + c) * a.N + gi] = v[c];
        a.G[(9 + g.dir) * a.N + gi] = v[3];
        if (a.L2e) upd(a.L2e[gi], v[4], a.first);
    }
    template <class A>
    DEV static void store(const Geo &, const A &a, long gi, const double *v)
    {
#pragma unroll
        for (int c = 0; c < 5; c++) upd(a.dQ[c * a.N + gi], v[c], a.first);
    }

    // CROSS: G(., y) and dT/dy go out and stay in the carry; the Laplacian
    // of e adds the z, then the x partial.
    template <class A>
    DEV static void sfetch_early(const Geo &, const A &a, long gi, double *sf)
    {
        sf[0] = a.L2e ? a.L2ep[gi] : 0.0;
        sf[1] = a.L2e ? a.L2ep[a.N + gi] : 0.0;
    }
    template <class A>
    DEV static void store_early(const Geo &, const A &a, long gi, const double *v, double *cr,
                                const double *sf)
    {
        const long N = a.N;
#pragma unroll
        for (int c = 0; c < 3; c++) a.G[(3 + c) * N + gi] = v[c];
        a.G[10 * N + gi] = v[3];
#pragma unroll
        for (int c = 0; c < 4; c++) cr[c] = v[c];
        cr[4] = (v[4] + sf[0]) + sf[1];
        if (a.L2e) a.L2e[gi] = cr[4];
    }
    // the store phase's reads: du/dz, dw/dx, dT/dx, dT/dz, the z partials
    // (5), the x partials (5)
    template <class A>
    DEV static void sfetch(const Geo &, const A &a, long gi, double *sf)
    {
        const long N = a.N;
        sf[0] = a.G[2 * N + gi];
        sf[1] = a.G[6 * N + gi];
        sf[2] = a.G[9 * N + gi];
        sf[3] = a.G[11 * N + gi];
#pragma unroll
        for (int c = 0; c < 10; c++) sf[4 + c] = a.dQp[c * N + gi];
    }
    // CROSS: viscous terms built from products of first derivatives
    // (src/rhsv_periodic_sf.f:1128-1154 without the mixed and own-direction
    // second derivatives, and :1252-1275), plus |S| (src/hyper_dynamic.f:
    // 12-33, 227-245) and the dilatation sensor C_beta
    // (src/hyper_dynamic.f:142-160; skipped when Cb is null: the
    // constant-coefficient src/hyper_routines.f); |S| and C_beta only with
    // the artificial transport on (L2e set).
    template <class A>
    DEV static void store(const Geo &, const A &a, long gi, const double *v, const double *cr,
                          const double *sf, const double *lc, double *po)
    {
        const long N = a.N;
        const Phys &ph = a.ph;
        struct { double u, v, w, T; } pr = {lc[0], lc[1], lc[2], lc[3]};
        static_assert(!CROSS || (NMX == 4 && msrc(0) == 0 && msrc(1) == 1 && msrc(2) == 7 && msrc(3) == 8),
                      "the kept slots are du/dx, dv/dx, dv/dz, dw/dz and mu");
        const double gxx = v[5], gyx = v[6], gzx = sf[0];
        const double gxy = cr[0], gyy = cr[1], gzy = cr[2];
        const double gxz = sf[1], gyz = v[7], gzz = v[8];
        const double mu = v[9], mup = dvisc(ph, pr.T, mu);
        const double tx = mup * sf[2], ty = mup * cr[3], tz = mup * sf[3];
        const double f1 = ph.bulk - 2.0 / 3.0;
        const double dil = gxx + gyy + gzz;
        const double t1 = gyx + gxy, t2 = gzx + gxz, t3 = gzy + gyz;
        const double fX = tx * (2.0 * gxx + f1 * dil) + ty * t1 + tz * t2;
        const double fY = ty * (2.0 * gyy + f1 * dil) + tx * t1 + tz * t3;
        const double fZ = tz * (2.0 * gzz + f1 * dil) + tx * t2 + ty * t3;
        const double *Pz = sf + 4, *Px = sf + 9;
        a.dQ[gi] = ((v[0] + Pz[0]) + Px[0]) + fX;
        a.dQ[N + gi] = ((v[1] + Pz[1]) + Px[1]) + fY;
        a.dQ[2 * N + gi] = ((v[2] + Pz[2]) + Px[2]) + fZ;
        a.dQ[3 * N + gi] = (v[3] + Pz[3]) + Px[3];
        a.dQ[4 * N + gi] = ((v[4] + Pz[4]) + Px[4])
                           + (pr.u * fX + pr.v * fY + pr.w * fZ
                              + mu * (2.0 * (gxx * gxx + gyy * gyy + gzz * gzz) + f1 * dil * dil)
                              + mu * (t1 * t1 + t2 * t2 + t3 * t3)
                              + ph.pr_inv * (ty * cr[3]));
        po[0] = 0.0;
        po[1] = cr[4];
        if (a.L2e) {
            const double s12 = 0.5 * (gxy + gyx), s13 = 0.5 * (gxz + gzx), s23 = 0.5 * (gyz + gzy);
            po[0] = sqrt(0.5 * (gxx * gxx + gyy * gyy + gzz * gzz + 2.0 * (s12 * s12 + s13 * s13 + s23 * s23)));
            a.S[gi] = po[0];
            if (a.Cb) {
                const double wx = gzy - gyz, wy = gxz - gzx, wz = gyx - gxy;
                const double om2 = wx * wx + wy * wy + wz * wz;
                const double fac = 0.5 * (1.0 - tanh(2.5 + 10.0 * dil));
                a.Cb[gi] = fac * dil * dil / (dil * dil + om2 + 1.0e-7) + 1.0e-20;
            }
        }
    }
    // CROSS: D2y of |S| and Lap e
    template <class A>
    DEV static bool post_on(const A &a) { return (bool)a.L2e; }
    template <int M, int P, bool NP, bool AL, class A>
    DEV static void compute_post(const A &a, const Lane<M, P, NP, AL> &L)
    {
#pragma unroll 1
        for (int m = 0; m < 2; m++) {
            double f[M], w[M + 2 * d_halo<NP, M>()], r[M];
#pragma unroll
            for (int k = 0; k < M; k++) f[k] = L.ld(m, k);
            window<M>(f, L, w);
            op_d2<M>(w, a.K2, a.tab()->op[1], L, r);
#pragma unroll
            for (int k = 0; k < M; k++) L.st(m, k, r[k]);
        }
    }
    template <class A>
    DEV static void store_post(const A &a, long gi, const double *v)
    {
        a.L2S[gi] = v[0];
        a.L4e[gi] = v[1];
    }
};

}  // namespace st
