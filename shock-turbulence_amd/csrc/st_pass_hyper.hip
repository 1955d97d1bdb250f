// Artificial-transport passes: second Laplacians, Gaussian smoothing, flux divergence.
#include "st_pass_hdiv.hpp"

namespace st {

// ---------------------------------------------------------------------
// P3: Laplacian of Lap|S| (src/hyper_dynamic.f:272-279), x pass: adds D2x
// to the z pass's partial in L4S.
// ---------------------------------------------------------------------
struct PassLap2 : NoReuse {
    static constexpr int STREAM = STREAM_LOADS;
    static constexpr int NSLOT = 1, NOUT = 1, NEARLY = 0;
    template <class A>
    DEV static void load(const Geo &, const A &a, long gi, double (&v)[1]) { v[0] = a.L2S[gi]; }
    template <int M, int P, bool NP, bool AL, class A>
    DEV static void compute(const Geo &, const A &a, const Lane<M, P, NP, AL> &L, double (&out)[1][M])
    {
        double f[M], w[M + 2 * d_halo<NP, M>()];
#pragma unroll
        for (int k = 0; k < M; k++) f[k] = L.ld(0, k);
        window<M>(f, L, w);
        op_d2<M>(w, a.K2, a.tab()->op[1], L, out[0]);
    }
    template <class A>
    DEV static void store(const Geo &, const A &a, long gi, const double *v) { upd(a.L4S[gi], v[0], a.first); }
};

// D2 along the sweep of the first staged slot, in place.
template <int M, int P, bool NP, bool AL, class A>
DEV void d2_slot(const A &a, const Lane<M, P, NP, AL> &L, int m)
{
    double f[M], w[M + 2 * d_halo<NP, M>()], r[M];
#pragma unroll
    for (int k = 0; k < M; k++) f[k] = L.ld(m, k);
    window<M>(f, L, w);
    op_d2<M>(w, a.K2, a.tab()->op[1], L, r);
#pragma unroll
    for (int k = 0; k < M; k++) L.st(m, k, r[k]);
}

// ---------------------------------------------------------------------
// The z pass that completes Lap|S| and Lap(Lap e) (the last direction of
// the D2 of |S| and Lap e, after x and y) and starts Lap(Lap|S|) on the
// same z lines:
//   compute   D2z of |S| and Lap e
//   mid       per point: L2S and L4e += those (written)
//   compute2  D2z of L2S
//   store     L4S = D2z L2S (the first direction of the second Laplacian)
// ---------------------------------------------------------------------
struct PassLapSELap2 {
    static constexpr int STREAM = STREAM_LOADS;
    static constexpr int NSLOT = 2, NOUT = 0, NEARLY = 1;
    static constexpr bool REUSE = true;
    static constexpr bool MID = true;
    static constexpr int MIN_WAVES = 1;
    static constexpr int LOAD_UNROLL = 8;
    static constexpr int NPF = 0;
    template <class A>
    DEV static void prefetch(const Geo &, const A &, long, double *) {}
    template <class A>
    DEV static void load(const Geo &, const A &a, long gi, double (&v)[2])
    {
        v[0] = a.S[gi];
        v[1] = a.L2e[gi];
    }
    template <int M, int P, bool NP, bool AL, class A>
    DEV static void compute(const Geo &, const A &a, const Lane<M, P, NP, AL> &L, double (&)[1][M])
    {
#pragma unroll 1
        for (int m = 0; m < 2; m++) d2_slot<M, P, NP>(a, L, m);
    }
    // the sums so far, of all the thread's points before the first is stored
    static constexpr int NMF = 2, MF_BATCH = 8;
    template <class A>
    DEV static void mfetch(const Geo &, const A &a, long gi, double *m)
    {
        m[0] = a.L2S[gi];
        m[1] = a.L4e[gi];
    }
    template <class A>
    DEV static void mid(const Geo &, const A &a, long gi, int, double (&v)[2], const double *m)
    {
        const double l2s = m[0] + v[0];            // as the accumulating D2 pass of |S| and Lap e
        a.L2S[gi] = l2s;
        a.L4e[gi] = m[1] + v[1];
        v[0] = l2s;
        v[1] = 0.0;
    }
    template <int M, int P, bool NP, bool AL, class A>
    DEV static void compute2(const Geo &, const A &a, const Lane<M, P, NP, AL> &L)
    {
        d2_slot<M, P, NP>(a, L, 0);
    }
    template <class A>
    DEV static void store(const Geo &, const A &, long, const double *) {}
    template <class A>
    DEV static void store_early(const Geo &, const A &a, long gi, const double *v) { a.L4S[gi] = v[0]; }
};

// ---------------------------------------------------------------------
// The y pass that completes Lap(Lap|S|) (after z and x), forms the transport
// drivers eta = (rho |Lap^2 S|, (rho/T) c |Lap^2 e|) (src/hyper_dynamic.f:
// 278-297) and smooths them along y (the first Gaussian direction):
//   compute   D2y of L2S
//   mid       per point: |L4S + D2y|, |L4e| and the state give eta
//   compute2  Gaussian along y of both eta fields
//   store     eta
// ---------------------------------------------------------------------
struct PassLap2Gauss {
    static constexpr int STREAM = STREAM_LOADS | STREAM_STORES | STREAM_Y;
    static constexpr int NSLOT = 2, NOUT = 0, NEARLY = 2;
    static constexpr bool REUSE = true;
    static constexpr bool MID = true;
    static constexpr int MIN_WAVES = 1;
    static constexpr int LOAD_UNROLL = 8;
    static constexpr int NPF = 0;
    template <class A>
    DEV static void prefetch(const Geo &, const A &, long, double *) {}
    template <class A>
    DEV static void load(const Geo &, const A &a, long gi, double (&v)[2])
    {
        v[0] = a.L2S[gi];
        v[1] = 0.0;
    }
    template <int M, int P, bool NP, bool AL, class A>
    DEV static void compute(const Geo &, const A &a, const Lane<M, P, NP, AL> &L, double (&)[1][M])
    {
        d2_slot<M, P, NP>(a, L, 0);
    }
    template <class A>
    DEV static void mid(const Geo &, const A &a, long gi, int, double (&v)[2])
    {
        const Phys &ph = a.ph;
        const double d4S = fabs(a.L4S[gi] + v[0]);
        const double d4e = fabs(a.L4e[gi]);
        const double q4 = qf(a, 3, gi);
        const Prim pr = prim(ph, qf(a, 0, gi), qf(a, 1, gi), qf(a, 2, gi), q4, qf(a, 4, gi));
        const double fac3 = (q4 / pr.T) * sqrt(ph.gamma * pr.p * pr.vs);
        v[0] = q4 * d4S;
        v[1] = fac3 * d4e;
    }
    template <int M, int P, bool NP, bool AL, class A>
    DEV static void compute2(const Geo &, const A &a, const Lane<M, P, NP, AL> &L)
    {
#pragma unroll 1
        for (int m = 0; m < 2; m++) {
            double f[M], w[M + 2 * HALO], r[M];
#pragma unroll
            for (int k = 0; k < M; k++) f[k] = L.ld(m, k);
            window<M>(f, L, w);
            op_gauss<M>(w, a.C, r);
#pragma unroll
            for (int k = 0; k < M; k++) L.st(m, k, r[k]);
        }
    }
    template <class A>
    DEV static void store(const Geo &, const A &, long, const double *) {}
    template <class A>
    DEV static void store_early(const Geo &, const A &a, long gi, const double *v)
    {
        a.eta[gi] = v[0];
        a.eta[a.N + gi] = v[1];
    }
};

// ---------------------------------------------------------------------
// Gaussian smoothing of eta (in place), the x pass (y is done in
// PassLap2Gauss, z in PassGaussHdiv).
// ---------------------------------------------------------------------
struct PassGaussEta : NoReuse {
    static constexpr int STREAM = STREAM_LOADS;
    static constexpr int NSLOT = 2, NOUT = 2, NEARLY = 0;
    template <class A>
    DEV static void load(const Geo &, const A &a, long gi, double (&v)[2])
    {
        v[0] = a.eta[gi];
        v[1] = a.eta[a.N + gi];
    }
    template <int M, int P, bool NP, bool AL, class A>
    DEV static void compute(const Geo &, const A &a, const Lane<M, P, NP, AL> &L, double (&out)[2][M])
    {
#pragma unroll
        for (int m = 0; m < 2; m++) {
            double f[M], w[M + 2 * HALO];
#pragma unroll
            for (int k = 0; k < M; k++) f[k] = L.ld(m, k);
            window<M>(f, L, w);
            op_gauss<M>(w, a.C, out[m]);
        }
    }
    template <class A>
    DEV static void store(const Geo &, const A &a, long gi, const double *v)
    {
        a.eta[gi] = v[0];
        a.eta[a.N + gi] = v[1];
    }
};

// ---------------------------------------------------------------------
// The z pass of the Gaussian smoothing fused with the z pass of the
// divergence: the smoothed eta gives the transport coefficients beta*,
// mu*, kappa* (src/hyper_dynamic.f:303-314) and, at the same point, all the
// artificial stresses and energy fluxes (src/hyper_rhs.f:159-491).  Those of
// the z direction are staged and their D1z added into dQ; those of x and y
// are written for their passes, which then read four fields each instead of
// the coefficients, eight gradients and the state.  The pass is bound by
// memory: 34 fields a point (37 with the coefficients written, which only
// the last stage of a step needs).  256^3: this pass 745 -> 895 us at 26 ->
// 34 fields, the x pass 698 -> 336 us (23 -> 12), the y pass 959 -> 703 us
// (36 -> 29, streamed).
//   compute   Gaussian along z of the two eta fields
//   mid       per point: beta*, mu*, kappa*, the x and y fluxes (written),
//             the staged z fluxes
//   compute2  D1z of the fluxes
// ---------------------------------------------------------------------
struct PassGaussHdiv {
    static constexpr int STREAM = STREAM_LOADS | STREAM_STORES;
    static constexpr int NSLOT = 4, NOUT = 0, NEARLY = 4;
    static constexpr bool REUSE = true;
    static constexpr bool MID = true;
    static constexpr int MIN_WAVES = 1;
    static constexpr int LOAD_UNROLL = 8;
    static constexpr int NPF = PassHyperDiv::NPF;
    template <class A>
    DEV static void prefetch(const Geo &g, const A &a, long gi, double *p) { PassHyperDiv::prefetch(g, a, gi, p); }
    template <class A>
    DEV static void load(const Geo &, const A &a, long gi, double (&v)[4])
    {
        v[0] = a.eta[gi];
        v[1] = a.eta[a.N + gi];
        v[2] = 0.0;
        v[3] = 0.0;
    }
    template <int M, int P, bool NP, bool AL, class A>
    DEV static void compute(const Geo &, const A &a, const Lane<M, P, NP, AL> &L, double (&)[1][M])
    {
#pragma unroll
        for (int m = 0; m < 2; m++) {
            double f[M], w[M + 2 * HALO], r[M];
#pragma unroll
            for (int k = 0; k < M; k++) f[k] = L.ld(m, k);
            window<M>(f, L, w);
            op_gauss<M>(w, a.C, r);
#pragma unroll
            for (int k = 0; k < M; k++) L.st(m, k, r[k]);
        }
    }
    // the 12 gradients, the momenta and density, C_beta
    static constexpr int NMF = 17, MF_BATCH = 2;
    template <class A>
    DEV static void mfetch(const Geo &, const A &a, long gi, double *m)
    {
#pragma unroll
        for (int c = 0; c < 12; c++) m[c] = a.G[c * a.N + gi];
#pragma unroll
        for (int c = 0; c < 4; c++) m[12 + c] = a.Q[c * a.N + gi];
        // constant C_beta = 1 without the sensor (src/hyper_routines.f:99-101,204)
        m[16] = a.Cb ? (double)a.Cb[gi] : 1.0;
    }
    template <class A>
    DEV static void mid(const Geo &, const A &a, long gi, int, double (&v)[4], const double *m)
    {
        const Phys &ph = a.ph;
        const long N = a.N;
        const double beta = m[16] * v[0] * ph.dx6;
        const double mu = ph.cmu * v[0] * ph.dx6;
        const double kap = ph.ck * v[1] * ph.dx5;
        if (a.keep_hc) {
            a.Hc[gi] = beta;
            a.Hc[N + gi] = mu;
            a.Hc[2 * N + gi] = kap;
        }
        const double gxx = m[0], gyy = m[4], gzz = m[8];
        const double dil = gxx + gyy + gzz;
        const double uh = m[12] / m[15], vh = m[13] / m[15], wh = m[14] / m[15];
        const double tt = 2.0 / 3.0;
        const double bulkterm = (beta - tt * mu) * dil;
        const double xx = 2.0 * mu * gxx + bulkterm, yy = 2.0 * mu * gyy + bulkterm, zz = 2.0 * mu * gzz + bulkterm;
        const double xy = mu * (m[3] + m[1]), xz = mu * (m[6] + m[2]), yz = mu * (m[7] + m[5]);
        a.dQp[FLUX_XX * N + gi] = xx;
        a.dQp[FLUX_XY * N + gi] = xy;
        a.dQp[FLUX_XZ * N + gi] = xz;
        a.dQp[FLUX_EX * N + gi] = uh * xx + vh * xy + wh * xz + kap * m[9];
        a.dQp[FLUX_YY * N + gi] = yy;
        a.dQp[FLUX_YZ * N + gi] = yz;
        a.dQp[FLUX_EY * N + gi] = uh * xy + vh * yy + wh * yz + kap * m[10];
        v[0] = xz;
        v[1] = yz;
        v[2] = zz;
        v[3] = uh * xz + vh * yz + wh * zz + kap * m[11];
    }
    template <int M, int P, bool NP, bool AL, class A>
    DEV static void compute2(const Geo &g, const A &a, const Lane<M, P, NP, AL> &L)
    {
        double o[1][M];
        PassHyperDiv::compute<M, P, NP>(g, a, L, o);
    }
    template <class A>
    DEV static void store(const Geo &, const A &, long, const double *) {}
    template <class A>
    DEV static void store_early(const Geo &g, const A &a, long gi, const double *v)
    {
        PassHyperDiv::store_early(g, a, gi, v);
    }
};


// The fluxes are stored for x and y alone, and the pass that forms them takes
// the z derivative.
static bool flux_dir(int kind, int dir)
{
    return kind == K_HDIV ? dir != 2 : kind == K_GAUSS_ETA_LAST ? dir == 2 : true;
}

hipError_t launch_hyper(int kind, const DirTab &t, int nt, int dir, int My, int Mz, int Mx, const PassArgs &a, hipStream_t s)
{
    if (!flux_dir(kind, dir)) return hipErrorInvalidValue;
    switch (kind) {
    case K_LAP2: return launch<PassLap2>(t, nt, dir, My, Mz, Mx, a, s);
    case K_LAP2_LAST: return launch<PassLap2Gauss, false>(t, nt, dir, My, Mz, Mx, a, s);
    case K_LAPSE_LAP2: return launch<PassLapSELap2, false>(t, nt, dir, My, Mz, Mx, a, s);
    case K_GAUSS_ETA: return launch<PassGaussEta>(t, nt, dir, My, Mz, Mx, a, s);
    case K_GAUSS_ETA_LAST: return launch<PassGaussHdiv, false>(t, nt, dir, My, Mz, Mx, a, s);
    case K_HDIV: return launch<PassHyperDiv>(t, nt, dir, My, Mz, Mx, a, s);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_hyper_ragged(int kind, const RaggedSpec &sp, hipStream_t s)
{
    if (!flux_dir(kind, sp.dir)) return hipErrorInvalidValue;
    switch (kind) {
    case K_LAP2: return launch_ragged<PassLap2>(sp, s);
    case K_LAP2_LAST: return launch_ragged<PassLap2Gauss>(sp, s);
    case K_LAPSE_LAP2: return launch_ragged<PassLapSELap2>(sp, s);
    case K_GAUSS_ETA: return launch_ragged<PassGaussEta>(sp, s);
    case K_GAUSS_ETA_LAST: return launch_ragged<PassGaussHdiv>(sp, s);
    case K_HDIV: return launch_ragged<PassHyperDiv>(sp, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace st
