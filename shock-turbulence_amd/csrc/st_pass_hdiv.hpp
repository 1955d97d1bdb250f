// Divergence of the artificial stress and heat flux, shared by the
// hyper_div pass and its fused form with the stage update and x filter.
#pragma once

#include "st_pass.hpp"

namespace st {

// ---------------------------------------------------------------------
// P5: divergence of the artificial stress and heat flux
// (src/hyper_rhs.f:159-491), x and y.  For direction d the staged fields are
// the momentum fluxes tau_xd, tau_yd, tau_zd and the energy flux
// u tau_xd + v tau_yd + w tau_zd + kappa* dT/dx_d (the reference takes the
// D1 of each energy term separately; the sum of the D1s is the D1 of the
// sum), which the z pass has formed at the points where it made the
// coefficients.  So this pass moves 12 fields instead of the 23 of forming
// them again from Hc, eight gradients and the state, and divides nowhere.
// ---------------------------------------------------------------------
struct PassHyperDiv {
    static constexpr int STREAM = STREAM_LOADS;
    static constexpr int NSLOT = 4, NOUT = 0, NEARLY = 4;
    static constexpr bool REUSE = true;
    static constexpr int MIN_WAVES = 1;
    static constexpr int LOAD_UNROLL = 8;
    static constexpr int NPF = 4;            // dQ 1, 2, 3, 5 before this pass
    template <class A>
    DEV static void prefetch(const Geo &, const A &a, long gi, double *p)
    {
        p[0] = a.dQ[gi];
        p[1] = a.dQ[a.N + gi];
        p[2] = a.dQ[2 * a.N + gi];
        p[3] = a.dQ[4 * a.N + gi];
    }
    template <class A>
    DEV static void load(const Geo &g, const A &a, long gi, double (&v)[4])
    {
        const long N = a.N;
        const bool x = g.dir == 0;           // the same on every lane
        v[0] = a.dQp[(x ? FLUX_XX : FLUX_XY) * N + gi];
        v[1] = a.dQp[(x ? FLUX_XY : FLUX_YY) * N + gi];
        v[2] = a.dQp[(x ? FLUX_XZ : FLUX_YZ) * N + gi];
        v[3] = a.dQp[(x ? FLUX_EX : FLUX_EY) * N + gi];
    }
    template <int M, int P, bool NP, bool AL, class A>
    DEV static void compute(const Geo &, const A &a, const Lane<M, P, NP, AL> &L, double (&)[1][M])
    {
#pragma unroll 1
        for (int m = 0; m < 4; m++) {
            double f[M], w[M + 2 * d_halo<NP, M>()], r[M];
#pragma unroll
            for (int k = 0; k < M; k++) f[k] = L.ld(m, k);
            window<M>(f, L, w);
            op_d1<M>(w, a.K1, a.tab()->op[0], L, r);
#pragma unroll
            for (int k = 0; k < M; k++) L.st(m, k, r[k]);
        }
    }
    template <class A>
    DEV static void store(const Geo &, const A &, long, const double *) {}
    template <class A>
    DEV static void store_early(const Geo &, const A &a, long gi, const double *v)
    {
        a.dQ[gi] = v[4] + v[0];
        a.dQ[a.N + gi] = v[5] + v[1];
        a.dQ[2 * a.N + gi] = v[6] + v[2];
        a.dQ[4 * a.N + gi] = v[7] + v[3];
    }
};

}  // namespace st
