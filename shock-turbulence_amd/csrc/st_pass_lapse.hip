// Second derivatives of |S| and of the Laplacian of e (the artificial
// transport's fourth-order drivers), x.
#include "st_pass.hpp"

namespace st {

// ---------------------------------------------------------------------
// D2 along x of |S| and of Lap e, added to the y terms that the y gradient
// pass left in L2S = Lap|S| and L4e = Lap(Lap e) (src/hyper_dynamic.f:
// 272-276); z joins the first pass of the artificial transport.
// ---------------------------------------------------------------------
struct PassLapSE {
    static constexpr int STREAM = STREAM_LOADS;
    static constexpr int NSLOT = 2, NOUT = 0, NEARLY = 2;
    static constexpr bool REUSE = true;
    static constexpr int MIN_WAVES = 1;
    static constexpr int LOAD_UNROLL = 8;
    static constexpr int NPF = 2;
    template <class A>
    DEV static void prefetch(const Geo &, const A &a, long gi, double *p)
    {
        p[0] = a.L2S[gi];
        p[1] = a.L4e[gi];
    }
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
    DEV static void store(const Geo &, const A &, long, const double *) {}
    template <class A>
    DEV static void store_early(const Geo &, const A &a, long gi, const double *v)
    {
        a.L2S[gi] = v[2] + v[0];
        a.L4e[gi] = v[3] + v[1];
    }
};


hipError_t launch_lapse(int kind, const DirTab &t, int nt, int dir, int My, int Mz, int Mx, const PassArgs &a, hipStream_t s)
{
    if (kind != K_LAPSE) return hipErrorInvalidValue;
    return launch<PassLapSE>(t, nt, dir, My, Mz, Mx, a, s);
}

hipError_t launch_lapse_ragged(int kind, const RaggedSpec &sp, hipStream_t s)
{
    if (kind != K_LAPSE) return hipErrorInvalidValue;
    return launch_ragged<PassLapSE>(sp, s);
}

}  // namespace st
