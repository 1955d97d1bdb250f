// The last filter pass of a stage fused with the x gradient pass of the next.
#include "st_pass_grad.hpp"

namespace st {

// ---------------------------------------------------------------------
// Between the stages of a step: the x filter and Fix_Pressure
// (src/lddrk4_periodic_sf.f:354-356,436-473) end one stage, the x gradient
// pass starts the next on the same lines and the same state:
//   compute   filter of the five fields along x
//   mid       per point: Fix_Pressure, the state written, its primitives staged
//   compute2  the x gradient pass
//   store     as that pass
// The state is read once instead of twice and a launch goes.  Same bits as
// the two passes in the same lane layout.
// ---------------------------------------------------------------------
struct PassFqGrad {
    typedef PassGrad<0, 1> Grad;
    static constexpr int NSLOT = 5, NOUT = 5, NEARLY = 5;
    static constexpr bool REUSE = true;
    static constexpr bool MID = true;
    static constexpr int STREAM = STREAM_LOADS | STREAM_STORES;
    static constexpr int MIN_WAVES = 1;
    static constexpr int LOAD_UNROLL = 8;
    static constexpr int NPF = 0;
    HD static constexpr bool lds_add(int) { return true; }
    template <class A>
    DEV static void prefetch(const Geo &, const A &, long, double *) {}
    template <class A>
    DEV static void load(const Geo &, const A &a, long gi, double (&v)[5])
    {
#pragma unroll
        for (int c = 0; c < 5; c++) v[c] = a.Q[c * a.N + gi];
    }
    template <int M, int P, bool NP, bool AL, class A>
    DEV static void compute(const Geo &, const A &a, const Lane<M, P, NP, AL> &L, double (&)[5][M])
    {
        CTab &T = a.tab()->op[2];
#pragma unroll 1
        for (int m = 0; m < 5; m++) {
            double f[M], w[M + 2 * HALO], r[M];
#pragma unroll
            for (int k = 0; k < M; k++) f[k] = L.ld(m, k);
            window<M>(f, L, w);
            op_filt<M>(w, a.C, T.scale, T, L, r);
#pragma unroll
            for (int k = 0; k < M; k++) L.st(m, k, r[k]);
        }
    }
    template <class A>
    DEV static void mid(const Geo &, const A &a, long gi, int, double (&v)[5])
    {
        v[4] = fixed_energy(a.ph, v[0], v[1], v[2], v[3], v[4]);
#pragma unroll
        for (int c = 0; c < 5; c++) a.Q[c * a.N + gi] = v[c];
        const Prim pr = prim(a.ph, v[0], v[1], v[2], v[3], v[4]);
        v[4] = v[3];
        v[0] = pr.u;
        v[1] = pr.v;
        v[2] = pr.w;
        v[3] = pr.T;
    }
    template <int M, int P, bool NP, bool AL, class A>
    DEV static void compute2(const Geo &g, const A &a, const Lane<M, P, NP, AL> &L, double (&out)[5][M])
    {
        Grad::compute<M, P, NP>(g, a, L, out);
    }
    template <class A>
    DEV static void store_early(const Geo &g, const A &a, long gi, const double *v)
    {
        Grad::store_early(g, a, gi, v);
    }
    template <class A>
    DEV static void store(const Geo &g, const A &a, long gi, const double *v)
    {
        Grad::store(g, a, gi, v);
    }
};

hipError_t launch_fqgrad(const DirTab &t, int nt, int My, int Mz, int Mx, const PassArgs &a, hipStream_t s)
{
    return launch<PassFqGrad>(t, nt, 0, My, Mz, Mx, a, s);
}

hipError_t launch_fqgrad_ragged(const RaggedSpec &sp, hipStream_t s) { return launch_ragged<PassFqGrad>(sp, s); }

}  // namespace st
