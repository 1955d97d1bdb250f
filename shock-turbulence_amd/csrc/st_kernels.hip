// HIP kernels for the per-RK-stage pipeline (gfx950, FP64).
//
// The reference evaluates one stage as ~110 separate compact operators,
// each copying bands, transposing and re-eliminating
// (src/derivCDopt6_periodic.f, src/pentadiagonal.f90).  Here a stage is a
// short chain of directional passes; each pass loads its inputs once,
// applies every operator of that direction the dataflow allows, folds the
// pointwise algebra of src/rhsv_periodic_sf.f and src/hyper_rhs.f into
// its load and store phases, and writes its results once.
#include <hip/hip_runtime.h>

#include "st_engine.hpp"
#include "st_kernels.h"

namespace st {

// Launch shape of a pass: the lane layout (wide: M points per lane on P lanes;
// narrow: M/2 on 2P) and the threads per workgroup.  Measured with each pass
// varied in turn and the whole stage timed (us per stage).
// Grids below STREAM_POINTS live in the caches and launch few workgroups: the
// narrow layout halves each lane's serial work and 256-thread tiles give the
// most workgroups (against the shapes of 256^3: 64^3 190 -> 153, 48^3 149 ->
// 117, 32^3 113 -> 88, 96^3 410 -> 353).
// Larger grids are bound by memory.  y passes keep the narrow layout and 256
// threads (the plain update and filter 512: 128^3 without artificial transport
// 393 -> 387).  Strided passes take tiles of 16 lines, whose rows are whole
// 128-byte lines that can stream (256^3: x gradient 5579 -> 5465, z Gaussian and
// divergence 5476 -> 5405), on 32 lanes per line (128^3: z Gaussian and
// divergence narrow 737, wide 751); but the x filter and x gradient passes and
// their fused form keep the wide layout (128^3: fused 713 wide, 730 narrow),
// and the filters alone, with much arithmetic for ten fields, 256 threads, more
// than one workgroup per CU (256^3 filter z 5382 against 5447).  The layout
// decides the rounding, so it depends on the instance alone and not on how
// many share the launch.
void pass_default_cfg(int kind, int dir, const DirTab &wide, long ni, long N, int *narrow, int *nt)
{
    *narrow = 1;
    *nt = 256;
    const bool big = ni >= STREAM_POINTS, many = N >= STREAM_POINTS;
    if (dir == 1) {
        if (kind == K_RKF && many) *nt = 512;
        return;
    }
    const bool filt = kind == K_FQ || kind == K_FQ_FIX, xgrad = kind == K_FQ_GRAD || (kind == K_GRAD && dir == 0);
    if (big) *narrow = !(filt || xgrad) && wide.P < 32;
    if (many && !filt) {
        const bool split = wide.M % 2 == 0 && 2 * wide.P <= 64;       // a narrow layout exists
        const int P = *narrow && split ? 2 * wide.P : wide.P;
        const int M = *narrow && split ? wide.M / 2 : wide.M;
        *nt = P <= 16 ? 256 : P == 32 ? 512 : 1024;
        // the z gradient pass has its 512-thread form for 4 to 7 points per lane
        if (kind == K_GRAD && dir == 2 && !(P == 32 && M >= 4 && M <= 7)) *nt = 256;
    }
}

hipError_t run_pass(int kind, const DirTab &t, int nt, int dir, int My, int Mz, int Mx, const PassArgs &a, hipStream_t s)
{
    switch (kind) {
    case K_D1: case K_D2: case K_FILT: case K_GAUSS: case K_VGRAD:
        return launch_ops(kind, t, nt, dir, My, Mz, Mx, a, s);
    // x first (no mixed terms), z with two, y last with four and the
    // pointwise assembly
    case K_GRAD:
        if (dir == 0) return launch_grad_x(t, nt, My, Mz, Mx, a, s);
        if (dir == 2) return launch_grad_z(t, nt, My, Mz, Mx, a, s);
        return hipErrorInvalidValue;
    case K_GRAD_CROSS:
        return dir == 1 ? launch_grad_y(t, nt, My, Mz, Mx, a, s) : hipErrorInvalidValue;
    case K_LAPSE:
        return launch_lapse(kind, t, nt, dir, My, Mz, Mx, a, s);
    case K_LAP2: case K_LAP2_LAST: case K_GAUSS_ETA: case K_GAUSS_ETA_LAST: case K_HDIV: case K_LAPSE_LAP2:
        return launch_hyper(kind, t, nt, dir, My, Mz, Mx, a, s);
    case K_RKF: case K_FQ: case K_FQ_FIX:
        return launch_filter(kind, t, nt, dir, My, Mz, Mx, a, s);
    case K_FQ_GRAD:
        return dir == 0 ? launch_fqgrad(t, nt, My, Mz, Mx, a, s) : hipErrorInvalidValue;
    case K_HDIV_RKF:
        return launch_hdivrk(kind, t, nt, dir, My, Mz, Mx, a, s);
    default: return hipErrorInvalidValue;
    }
}

int ragged_member(int n)
{
    for (int c = 0; c < 4; c++)
        if (RAGGED_N[c] == n) return c;
    return -1;
}

hipError_t run_pass_ragged(int kind, const RaggedSpec &sp, hipStream_t s)
{
    switch (kind) {
    case K_GRAD:
        if (sp.dir == 0) return launch_grad_x_ragged(sp, s);
        if (sp.dir == 2) return launch_grad_z_ragged(sp, s);
        return hipErrorInvalidValue;
    case K_GRAD_CROSS:
        return sp.dir == 1 ? launch_grad_y_ragged(sp, s) : hipErrorInvalidValue;
    case K_LAPSE:
        return launch_lapse_ragged(kind, sp, s);
    case K_LAP2: case K_LAP2_LAST: case K_GAUSS_ETA: case K_GAUSS_ETA_LAST: case K_HDIV: case K_LAPSE_LAP2:
        return launch_hyper_ragged(kind, sp, s);
    case K_RKF: case K_FQ: case K_FQ_FIX:
        return launch_filter_ragged(kind, sp, s);
    case K_FQ_GRAD:
        return sp.dir == 0 ? launch_fqgrad_ragged(sp, s) : hipErrorInvalidValue;
    case K_HDIV_RKF:
        return launch_hdivrk_ragged(kind, sp, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace st

// ---------------------------------------------------------------------
// reductions: one partial per block and slot, partial[(slot*nb + block)*NV + v]
// (slot: the slot number, not its index in the launch)
// ---------------------------------------------------------------------
namespace st {

template <int NV, class OP>
DEV void block_reduce(double (&v)[NV], OP op, double *partial, int slot)
{
    __shared__ double sh[NV][256 / 64];          // one array per NV: a kernel may reduce 2, then 3 values
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < NV; i++) {
        double x = v[i];
        for (int o = 32; o > 0; o >>= 1) x = op(x, __shfl_xor(x, o));
        if (lane == 0) sh[i][wave] = x;
    }
    __syncthreads();
    if (threadIdx.x < NV) {
        double x = sh[threadIdx.x][0];
        for (int w = 1; w < (int)(blockDim.x >> 6); w++) x = op(x, sh[threadIdx.x][w]);
        partial[((long)slot * gridDim.x + blockIdx.x) * NV + threadIdx.x] = x;
    }
}

struct OpMax { DEV double operator()(double a, double b) const { return a > b ? a : b; } };
struct OpMin { DEV double operator()(double a, double b) const { return a < b ? a : b; } };
struct OpSum { DEV double operator()(double a, double b) const { return a + b; } };

// Compute_CFL src/lddrk4_periodic_sf.f:29-56
__global__ void __launch_bounds__(256) k_cfl(PassArgs a, double *partial)
{
    const int slot = a.slots ? a.slots[blockIdx.y] : blockIdx.y;
    if (a.act && !a.act[slot]) return;
    const long N = a.N, off = (long)slot * a.ni;
    double v[2] = {-INFINITY, -INFINITY};
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < a.ni; i += (long)gridDim.x * blockDim.x) {
        const long gi = off + i;
        double w1, w2;
        cfl_point(a.ph, a.Q[gi], a.Q[N + gi], a.Q[2 * N + gi], a.Q[3 * N + gi], a.Q[4 * N + gi], w1, w2);
        v[0] = w1 > v[0] ? w1 : v[0];
        v[1] = w2 > v[1] ? w2 : v[1];
    }
    block_reduce<2>(v, OpMax(), partial, slot);
}

// The three dt limits of Compute_Tstep at a point
// (src/lddrk4_periodic_sf.f:105-132)
DEV void limit_point(const Phys &ph, double q1, double q2, double q3, double q4, double q5, double beta, double mu,
                     double kap, double (&l)[3])
{
    const double fac = ph.gamma * ph.gm1;
    const double del = ph.D[0];
    const double t1 = 1.0 / q4;
    const double br = q5 - 0.5 * t1 * (q1 * q1 + q2 * q2 + q3 * q3);
    const double t2 = sqrt(fac * t1 * br);
    const double T = ph.gamma * t1 * br;
    l[0] = q4 * (del * del) / mu;
    l[1] = q4 * (del * del) / beta;
    l[2] = q4 * ((del * t2) * (del * t2)) / (kap * T);
}

// Compute_Tstep src/lddrk4_periodic_sf.f:105-132 (beta*, mu*, kappa* in Hc)
__global__ void __launch_bounds__(256) k_tstep(PassArgs a, double *partial)
{
    const int slot = a.slots ? a.slots[blockIdx.y] : blockIdx.y;
    if (a.act && !a.act[slot]) return;
    const long N = a.N, off = (long)slot * a.ni;
    double v[3] = {INFINITY, INFINITY, INFINITY};
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < a.ni; i += (long)gridDim.x * blockDim.x) {
        const long gi = off + i;
        double l[3];
        limit_point(a.ph, a.Q[gi], a.Q[N + gi], a.Q[2 * N + gi], a.Q[3 * N + gi], a.Q[4 * N + gi], a.Hc[gi],
                    a.Hc[N + gi], a.Hc[2 * N + gi], l);
        for (int k = 0; k < 3; k++) v[k] = l[k] < v[k] ? l[k] : v[k];
    }
    block_reduce<3>(v, OpMin(), partial, slot);
}

// Both in one sweep, for the steps whose dt is formed on the device: Q is
// read once instead of twice.  The same expressions and the same order within
// a block as the two above, so the same bits; pt null: no limits (artificial
// transport off).
__global__ void __launch_bounds__(256) k_cfl_tstep(PassArgs a, double *pc, double *pt)
{
    const int slot = a.slots ? a.slots[blockIdx.y] : blockIdx.y;
    if (a.act && !a.act[slot]) return;
    const long N = a.N, off = (long)slot * a.ni;
    const Phys &ph = a.ph;
    double v[2] = {-INFINITY, -INFINITY}, u[3] = {INFINITY, INFINITY, INFINITY};
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < a.ni; i += (long)gridDim.x * blockDim.x) {
        const long gi = off + i;
        const double q1 = a.Q[gi], q2 = a.Q[N + gi], q3 = a.Q[2 * N + gi], q4 = a.Q[3 * N + gi], q5 = a.Q[4 * N + gi];
        double w[2];
        cfl_point(ph, q1, q2, q3, q4, q5, w[0], w[1]);
        for (int k = 0; k < 2; k++) v[k] = w[k] > v[k] ? w[k] : v[k];
        if (pt) {
            double l[3];
            limit_point(ph, q1, q2, q3, q4, q5, a.Hc[gi], a.Hc[N + gi], a.Hc[2 * N + gi], l);
            for (int k = 0; k < 3; k++) u[k] = l[k] < u[k] ? l[k] : u[k];
        }
    }
    block_reduce<2>(v, OpMax(), pc, slot);
    if (pt) block_reduce<3>(u, OpMin(), pt, slot);
}

// Compute_Mom/KE/Mass/Energy/Entropy src/lddrk4_periodic_sf.f:153-302 (sums)
__global__ void __launch_bounds__(256) k_diag(PassArgs a, double *partial)
{
    const int slot = a.slots ? a.slots[blockIdx.y] : blockIdx.y;
    if (a.act && !a.act[slot]) return;
    const long N = a.N, off = (long)slot * a.ni;
    const Phys &ph = a.ph;
    double v[7] = {0, 0, 0, 0, 0, 0, 0};
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < a.ni; i += (long)gridDim.x * blockDim.x) {
        const long gi = off + i;
        const double q1 = a.Q[gi], q2 = a.Q[N + gi], q3 = a.Q[2 * N + gi], q4 = a.Q[3 * N + gi], q5 = a.Q[4 * N + gi];
        const double t = 1.0 / q4;
        const double u1 = q1 * t, u2 = q2 * t, u3 = q3 * t;
        v[0] += q1;
        v[1] += q2;
        v[2] += q3;
        v[3] += q4 * u1 * u1 + q4 * u2 * u2 + q4 * u3 * u3;
        v[4] += q4;
        v[5] += q5;
        const double p = ph.gm1 * (q5 - 0.5 * t * (q1 * q1 + q2 * q2 + q3 * q3));
        v[6] += q4 * log(p * pow(t, ph.gamma));
    }
    block_reduce<7>(v, OpSum(), partial, slot);
}

__global__ void __launch_bounds__(256) k_fill(double *p, long n, double v)
{
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) p[i] = v;
}

// p[f*N + s*ni + i] = v for the launch's slots s (blockIdx.y = f*nslot + index)
__global__ void __launch_bounds__(256) k_fill_slots(double *p, long N, long ni, int nslot, const int *slots,
                                                     const int *act, double v)
{
    const int f = blockIdx.y / nslot, si = blockIdx.y - f * nslot;
    const int slot = slots ? slots[si] : si;
    if (act && !act[slot]) return;
    double *q = p + f * N + (long)slot * ni;
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < ni; i += (long)gridDim.x * blockDim.x) q[i] = v;
}

// Fix_Pressure on a resident array (src/lddrk4_periodic_sf.f:436-473), slot 0
__global__ void __launch_bounds__(256) k_fixp(PassArgs a, double *Qx)
{
    const long N = a.N;
    const Phys &ph = a.ph;
    for (long gi = blockIdx.x * (long)blockDim.x + threadIdx.x; gi < a.ni; gi += (long)gridDim.x * blockDim.x) {
        Qx[4 * N + gi] = fixed_energy(ph, Qx[gi], Qx[N + gi], Qx[2 * N + gi], Qx[3 * N + gi], Qx[4 * N + gi]);
    }
}

// Device-side Compute_Tstep for every slot (one workgroup per slot): fold the
// CFL and dt-limit partials, dt = cfl_cal/cfl_resv, then the hyper limits
// when the slot's step passes the driver's rule (src/lddrk4_periodic_sf.f:96-142;
// first_step = 1 applies them from the first step,
// src/lddrk4_nonperiodic_sf.f:105).  stepc is the driver's step counter
// (1 before the first step).  A slot runs this step (run = 1) while it is
// active and its counter is below its target.  hist and seen (a single run's
// march): hist[step - hist0] records the dt, and a slot whose dt is not positive
// and finite does not run, now or later (active is cleared); seen, in host
// memory, tells the host how many steps have their dt, -1 for such a slot.
// The fold of up to 1024 partials a slot is a chain of dependent loads in one
// thread (219 us at 64^3); 256 threads take four partials each (5 us).  A
// maximum or minimum does not depend on the order, NaNs are passed over.
__global__ void __launch_bounds__(256)
k_dt(const double *pc, const double *pt, int nb, int *active, const int *target, const int *stepc, double cfl_cal,
     int hyper, int first_step, int *run, double *dt, double *dt_last, double *hist, int hist0, int *seen)
{
    __shared__ double sh[4][4];
    const int slot = blockIdx.x;
    const int step = stepc[slot], go = active[slot] && step < target[slot];
    if (!go) {                                      // the same on every thread
        if (threadIdx.x == 0) run[slot] = 0;
        return;
    }
    const bool lim = hyper == 1 && (step > 1 || first_step);
    double v[4] = {-INFINITY, INFINITY, INFINITY, INFINITY};
    for (int b = threadIdx.x; b < nb; b += blockDim.x) {
        const double x = pc[((long)slot * nb + b) * 2 + 1];
        v[0] = x > v[0] ? x : v[0];
        if (lim)
            for (int i = 0; i < 3; i++) {
                const double y = pt[((long)slot * nb + b) * 3 + i];
                v[1 + i] = y < v[1 + i] ? y : v[1 + i];
            }
    }
    for (int i = 0; i < 4; i++) {
        for (int o = 32; o > 0; o >>= 1) {
            const double x = __shfl_xor(v[i], o);
            v[i] = (i == 0 ? x > v[i] : x < v[i]) ? x : v[i];
        }
        if ((threadIdx.x & 63) == 0) sh[i][threadIdx.x >> 6] = v[i];
    }
    __syncthreads();
    if (threadIdx.x) return;
    for (int i = 0; i < 4; i++)
        for (int w = 1; w < 4; w++) {
            const double x = sh[i][w];
            v[i] = (i == 0 ? x > v[i] : x < v[i]) ? x : v[i];
        }
    double t = cfl_cal / v[0];
    if (lim) {
        const double p2 = (double)0.2f;                 // default-real literal 0.2
        for (int i = 1; i < 4; i++)
            if (p2 * v[i] < t) t = p2 * v[i];
    }
    dt[slot] = t;
    dt_last[slot] = t;
    run[slot] = 1;
    if (!hist) return;
    hist[step - hist0] = t;
    const bool ok = t > 0.0 && t < INFINITY;
    if (!ok) active[slot] = run[slot] = 0;
    __hip_atomic_store(seen, ok ? step - hist0 + 1 : -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// time += dt after each RK loop; step += 1 after the second
// (src/lddrk4_periodic_sf.f:372,419-420)
__global__ void k_clock(int nslot, const int *run, const double *dt, double *time, int *stepc, int bump)
{
    const int slot = blockIdx.x * blockDim.x + threadIdx.x;
    if (slot >= nslot || !run[slot]) return;
    time[slot] = time[slot] + dt[slot];
    if (bump) stepc[slot] = stepc[slot] + 1;
}

// Sponge_Forcing (src/sponge1d.f:85-95): dQ -= sigma(x) (Q - Qref) with
// sigma per x index in spg[0..Mx) and the reference states of the left
// and right layers in spg[Mx..Mx+5) and spg[Mx+5..Mx+10).
__global__ void __launch_bounds__(256) k_sponge(PassArgs a, const double *spg, int Mx, int nleft)
{
    const int slot = a.slots ? a.slots[blockIdx.y] : blockIdx.y;
    if (a.act && !a.act[slot]) return;
    const long N = a.N, off = (long)slot * a.ni, plane = a.ni / Mx;
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < a.ni; i += (long)gridDim.x * blockDim.x) {
        const int ix = (int)(i / plane);
        const double sg = spg[ix];
        if (sg == 0.0) continue;
        const double *ref = spg + Mx + (ix < nleft ? 0 : 5);
        const long gi = off + i;
#pragma unroll
        for (int l = 0; l < 5; l++) a.dQ[l * N + gi] = fma(-sg, a.Q[l * N + gi] - ref[l], a.dQ[l * N + gi]);
    }
}

hipError_t run_sponge(const PassArgs &a, const double *spg, int Mx, int nleft, hipStream_t s)
{
    long blocks = (a.ni + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(k_sponge, dim3((unsigned)blocks, (unsigned)a.nslot), dim3(256), 0, s, a, spg, Mx, nleft);
    return hipGetLastError();
}

// ---------------------------------------------------------------------
// Compute_hyper outside a stage (src/hyper_dynamic.f:173-318; the static
// variant src/hyper_routines.f:66-214) and Compute_Grad (src/grad.f:13-115):
// the pointwise steps between single-operator passes.  Each acts on one
// slot: the pointers already carry the slot's offset, fields are N apart.
// ---------------------------------------------------------------------

// |S| of the symmetrised /GRAD/ (0 when G is null: the coefficients of a
// start without gradients, src/main.f:100) (src/hyper_dynamic.f:227-245,
// :12-33) and e (:251-266).
__global__ void __launch_bounds__(256) k_hyp_prep(const double *Q, const double *G, long N, long ni, double *S, double *e)
{
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < ni; i += (long)gridDim.x * blockDim.x) {
        const double q1 = Q[i], q2 = Q[N + i], q3 = Q[2 * N + i], q4 = Q[3 * N + i];
        const double t = 1.0 / q4;
        double s = 0.0;
        if (G) {
            const double s11 = G[i], s22 = G[4 * N + i], s33 = G[8 * N + i];
            const double s12 = 0.5 * (G[3 * N + i] + G[N + i]);
            const double s13 = 0.5 * (G[6 * N + i] + G[2 * N + i]);
            const double s23 = 0.5 * (G[7 * N + i] + G[5 * N + i]);
            s = sqrt(0.5 * (s11 * s11 + s22 * s22 + s33 * s33 + 2.0 * (s12 * s12 + s13 * s13 + s23 * s23)));
        }
        S[i] = s;
        e[i] = t * (Q[4 * N + i] - 0.5 * t * (q1 * q1 + q2 * q2 + q3 * q3));
    }
}

// C_beta from the nine velocity gradients g[3d + i] = du_i/dx_d: vorticity and
// dilatation (src/hyper_dynamic.f:105-160)
__global__ void __launch_bounds__(256) k_hyp_cb(const double *g, long N, long ni, double *Cb)
{
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < ni; i += (long)gridDim.x * blockDim.x) {
        const double g1 = g[5 * N + i] - g[7 * N + i], g2 = g[6 * N + i] - g[2 * N + i], g3 = g[N + i] - g[3 * N + i];
        const double g4 = (g[i] + g[4 * N + i]) + g[8 * N + i];
        const double fac = 0.5 * (1.0 - tanh(2.5 + 10.0 * g4));
        const double om2 = g1 * g1 + g2 * g2 + g3 * g3;
        Cb[i] = fac * g4 * g4 / (g4 * g4 + om2 + 1.0e-7) + 1.0e-20;
    }
}

// beta*, mu*, kappa* from the smoothed eta (src/hyper_dynamic.f:303-314;
// C_beta = 1 without the sensor, src/hyper_routines.f:204)
__global__ void __launch_bounds__(256) k_hyp_coef(const double *g1, const double *g2, const double *Cb, long N,
                                                  long ni, Phys ph, double *Hc)
{
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < ni; i += (long)gridDim.x * blockDim.x) {
        Hc[i] = (Cb ? Cb[i] : 1.0) * g1[i] * ph.dx6;
        Hc[N + i] = ph.cmu * g1[i] * ph.dx6;
        Hc[2 * N + i] = ph.ck * g2[i] * ph.dx5;
    }
}

// Compute_Grad's reductions (src/grad.f:100-115): max |dil| and the sum of
// |omega|^2 over one slot, from /GRAD/ (G fields 0..8), partials per block.
__global__ void __launch_bounds__(256) k_gradred(const double *G, long N, long ni, double *partial)
{
    __shared__ double sh[2][4];
    double mx = 0.0, s = 0.0;
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < ni; i += (long)gridDim.x * blockDim.x) {
        const double dux_dx = G[i], duy_dx = G[N + i], duz_dx = G[2 * N + i];
        const double dux_dy = G[3 * N + i], duy_dy = G[4 * N + i], duz_dy = G[5 * N + i];
        const double dux_dz = G[6 * N + i], duy_dz = G[7 * N + i], duz_dz = G[8 * N + i];
        const double w1 = duz_dy - duy_dz, w2 = dux_dz - duz_dx, w3 = duy_dx - dux_dy;
        const double dil = fabs(dux_dx + duy_dy + duz_dz);
        mx = dil > mx ? dil : mx;
        s += w1 * w1 + w2 * w2 + w3 * w3;
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int o = 32; o > 0; o >>= 1) {
        const double a = __shfl_xor(mx, o);
        mx = a > mx ? a : mx;
        s += __shfl_xor(s, o);
    }
    if (lane == 0) {
        sh[0][wave] = mx;
        sh[1][wave] = s;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double m = sh[0][0], t = sh[1][0];
        for (int w = 1; w < (int)(blockDim.x >> 6); w++) {
            m = sh[0][w] > m ? sh[0][w] : m;
            t += sh[1][w];
        }
        partial[2 * blockIdx.x] = m;
        partial[2 * blockIdx.x + 1] = t;
    }
}

static long pw_blocks(long ni)
{
    long b = (ni + 255) / 256;
    return b > 4096 ? 4096 : b;
}

hipError_t run_hyp_prep(const double *Q, const double *G, long N, long ni, double *S, double *e, hipStream_t s)
{
    hipLaunchKernelGGL(k_hyp_prep, dim3((unsigned)pw_blocks(ni)), dim3(256), 0, s, Q, G, N, ni, S, e);
    return hipGetLastError();
}

hipError_t run_hyp_cb(const double *g, long N, long ni, double *Cb, hipStream_t s)
{
    hipLaunchKernelGGL(k_hyp_cb, dim3((unsigned)pw_blocks(ni)), dim3(256), 0, s, g, N, ni, Cb);
    return hipGetLastError();
}

hipError_t run_hyp_coef(const double *g1, const double *g2, const double *Cb, long N, long ni, const Phys &ph,
                        double *Hc, hipStream_t s)
{
    hipLaunchKernelGGL(k_hyp_coef, dim3((unsigned)pw_blocks(ni)), dim3(256), 0, s, g1, g2, Cb, N, ni, ph, Hc);
    return hipGetLastError();
}

int gradred_blocks(long ni)
{
    long b = (ni + 255) / 256;
    return (int)(b > 1024 ? 1024 : b);
}

hipError_t run_gradred(const double *G, long N, long ni, double *partial, hipStream_t s)
{
    hipLaunchKernelGGL(k_gradred, dim3((unsigned)gradred_blocks(ni)), dim3(256), 0, s, G, N, ni, partial);
    return hipGetLastError();
}

static long red_blocks(long N)
{
    long b = (N + 255) / 256;
    return b > 1024 ? 1024 : b;
}

hipError_t run_reduce(int which, const PassArgs &a, double *partial, int *nblocks, hipStream_t s)
{
    const long nb = red_blocks(a.ni);
    *nblocks = (int)nb;
    const dim3 grid((unsigned)nb, (unsigned)a.nslot);
    if (which == 0) hipLaunchKernelGGL(k_cfl, grid, dim3(256), 0, s, a, partial);
    else if (which == 1) hipLaunchKernelGGL(k_tstep, grid, dim3(256), 0, s, a, partial);
    else hipLaunchKernelGGL(k_diag, grid, dim3(256), 0, s, a, partial);
    return hipGetLastError();
}

int reduce_blocks(long ni) { return (int)red_blocks(ni); }

hipError_t run_fill(double *p, long n, double v, hipStream_t s)
{
    long nb = (n + 255) / 256;
    if (nb > 4096) nb = 4096;
    hipLaunchKernelGGL(k_fill, dim3((unsigned)nb), dim3(256), 0, s, p, n, v);
    return hipGetLastError();
}

hipError_t run_fill_slots(double *p, int nfields, long N, long ni, int nslot, const int *slots, const int *act,
                          double v, hipStream_t s)
{
    long nb = (ni + 255) / 256;
    if (nb > 1024) nb = 1024;
    hipLaunchKernelGGL(k_fill_slots, dim3((unsigned)nb, (unsigned)(nfields * nslot)), dim3(256), 0, s, p, N, ni, nslot,
                       slots, act, v);
    return hipGetLastError();
}

hipError_t run_fixp(const PassArgs &a, double *Qx, hipStream_t s)
{
    const long nb = red_blocks(a.ni) * 4;
    hipLaunchKernelGGL(k_fixp, dim3((unsigned)nb), dim3(256), 0, s, a, Qx);
    return hipGetLastError();
}

hipError_t run_cfl_tstep(const PassArgs &a, double *pc, double *pt, int *nblocks, hipStream_t s)
{
    const long nb = red_blocks(a.ni);
    *nblocks = (int)nb;
    hipLaunchKernelGGL(k_cfl_tstep, dim3((unsigned)nb, (unsigned)a.nslot), dim3(256), 0, s, a, pc, pt);
    return hipGetLastError();
}

hipError_t run_dt(const double *pc, const double *pt, int nb, int nslot, int *active, const int *target,
                  const int *stepc, double cfl_cal, int hyper, int first_step, int *run, double *dt, double *dt_last,
                  double *hist, int hist0, int *seen, hipStream_t s)
{
    hipLaunchKernelGGL(k_dt, dim3((unsigned)nslot), dim3(256), 0, s, pc, pt, nb, active, target, stepc, cfl_cal, hyper,
                       first_step, run, dt, dt_last, hist, hist0, seen);
    return hipGetLastError();
}

// The clock of one run: active, its target, step and time
__global__ void k_clock_set(int *active, int *target, int *stepc, double *time, int steps, int step, double t)
{
    *active = 1;
    *target = step + steps;
    *stepc = step;
    *time = t;
}

hipError_t run_clock_set(int *active, int *target, int *stepc, double *time, int steps, int step, double t,
                         hipStream_t s)
{
    hipLaunchKernelGGL(k_clock_set, dim3(1), dim3(1), 0, s, active, target, stepc, time, steps, step, t);
    return hipGetLastError();
}

hipError_t run_clock(int nslot, const int *run, const double *dt, double *time, int *stepc, int bump, hipStream_t s)
{
    hipLaunchKernelGGL(k_clock, dim3((unsigned)((nslot + 63) / 64)), dim3(64), 0, s, nslot, run, dt, time, stepc, bump);
    return hipGetLastError();
}

}  // namespace st

