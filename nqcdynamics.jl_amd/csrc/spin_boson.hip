// spin_boson.hip -- FSSH / Ehrenfest for the spin-boson model (two states coupled to a
// harmonic bath), BABwithTsit5 (bab_electronics.jl:48-91) with the hop callback
// (surface_hopping.jl:2-16).
//
// V(R) = [[eps + c.R, Delta], [Delta, -eps - c.R]] + R^T W^2 R / 2
// (docs/src/NQCModels/systembathmodels.md:21-27).  The state-dependent part of dV/dR_j
// is c_j sigma_z, so every per-mode quantity the reference forms per degree of freedom
// (U^T dV_j U, the coupling d_j, v.d, the rescaling vectors) is c_j times a 2x2 quantity
// of the collective coordinate X = sum_j c_j R_j.  One trajectory per lane; the bath
// positions and velocities live in registers; all trajectories run the same number of
// steps, so the launch is a plain grid (no refill queue).
#include "spin_boson.h"

#include <cmath>

#include "ensemble.h"
#include <vector>

namespace nqcd {

constexpr int kBathModes = 100;  // instantiated bath size
constexpr int kSbBlock = 64;     // one wavefront per workgroup
constexpr int kSbAhead = 2;      // chunks of four modes whose coefficients are loaded together, one group ahead

struct SbArgs {
    int64_t ntraj;
    int32_t method, rescaling, nsub, save_every;
    int32_t nsave, initial_state, diabatic, pad;
    double dt, t0, eps, Delta, S2, cnorm;  // S2 = sum c^2/m, cnorm = |c|
    int64_t nsteps;
    uint64_t key;
    const double* w2;    // [NB] omega^2
    const double* c;     // [NB] coupling
    const double* invm;  // [NB] 1/m
    const double* kd;    // [NB/4][3][4] half-kick coefficients dt/2 w^2/m, dt/2 c/m, and c (FP64)
    const float* kf;     // [NB/4][3][4] the same in FP32
    const double* r0;    // [NB][ntraj] sampled initial positions
    const double* v0;    // [NB][ntraj] sampled initial velocities
    double* r;           // [NB][ntraj]
    double* v;           // [NB][ntraj]
    double* sig;         // [4][ntraj]
    int32_t* state;
    int32_t* steps;
    int32_t* nhops;
    double* save_pop_ad; // [nsave][2][ntraj]
    double* save_pop_di; // [nsave][2][ntraj]
    int32_t* save_state; // [nsave][ntraj]
};

template <class T>
__device__ __forceinline__ const T* sb_opaque(const T* p) {
    asm volatile("" : "+s"(p));
    return p;
}

// U^T sigma_z U for the 2x2 eigenvectors U (row-major).
__device__ __forceinline__ void rotate_sz(const double U[4], double& g00, double& g11, double& g01) {
    g00 = U[0] * U[0] - U[2] * U[2];
    g11 = U[1] * U[1] - U[3] * U[3];
    g01 = U[0] * U[1] - U[2] * U[3];
}

__device__ __forceinline__ void sb_save(const SbArgs* Ap, int64_t tid, int slot, int method, int st, double tr,
                                        const Sig2& s, const double U[4]) {
    const SbArgs& A = *sb_opaque(Ap);
    if (slot >= A.nsave) return;
    const int64_t n = A.ntraj;
    double pa0, pa1;
    if (method == 0) { pa0 = (st == 0) ? 1.0 : 0.0; pa1 = 1.0 - pa0; }
    else { pa0 = 0.5 * (tr + s.q); pa1 = 0.5 * (tr - s.q); }
    const double pd0 = U[0] * U[0] * pa0 + U[1] * U[1] * pa1 + 2.0 * U[0] * U[1] * s.x;
    const double pd1 = U[2] * U[2] * pa0 + U[3] * U[3] * pa1 + 2.0 * U[2] * U[3] * s.x;
    A.save_pop_ad[((int64_t)slot * 2) * n + tid] = pa0;
    A.save_pop_ad[((int64_t)slot * 2 + 1) * n + tid] = pa1;
    A.save_pop_di[((int64_t)slot * 2) * n + tid] = pd0;
    A.save_pop_di[((int64_t)slot * 2 + 1) * n + tid] = pd1;
    A.save_state[(int64_t)slot * n + tid] = st;
}

// The coefficient table through a constant-address-space pointer in scalar registers, made opaque where it is
// used: its entries are scalar loads there, and go into the vector instructions as scalar operands.
// Four modes make a chunk, so that a coefficient of a chunk is one four-wide load.
template <typename R>
using SbVec = R __attribute__((ext_vector_type(4)));
template <typename R>
using SbTab = __attribute__((address_space(4))) const SbVec<R>*;

__device__ __forceinline__ const double* kick_table(const SbArgs& A, double) { return A.kd; }
__device__ __forceinline__ const float* kick_table(const SbArgs& A, float) { return A.kf; }

template <typename R>
__device__ __forceinline__ SbTab<R> sb_table(const SbArgs& A) {
    return (SbTab<R>)uniform_sgpr((uint64_t)kick_table(A, (R)0));
}

template <typename R>
__device__ __forceinline__ SbTab<R> sb_here(SbTab<R> p) {
    asm volatile("" : "+s"(p));
    return p;
}

// A step is two passes over the modes with the electronics between them.  Both half kicks that meet at a step
// end see the same positions and the same force factor F (the acceleration of the step end stands, also after a
// hop), so one pass applies them together: v = u - a is the velocity at the step end, whose projection on c the
// coupling needs, and u' = u - 2 a the one after the next step's first half kick.  The kick a is formed first, so
// that a velocity is rounded at its own size once a step (velocity Verlet step by step rounds it twice).
//
// The positions of the last NL modes stay in LDS ([chunk][lane], 16 bytes a lane and access), the rest and all
// velocities in registers: with all 2 NB values in registers a wavefront took 352 registers, so the 1,563
// wavefronts of 1e5 trajectories ran one to a SIMD in two rounds; with 48 of the FP32 positions in LDS two fit.
// Bound by FP32 and FP64 issue: 2,240 vector instructions a wavefront-step by the counters (700 for the bath, about 450
// for the electronics, the hop's pass in nearly every step, as a lane hops in every sixteenth), 7.5 ms where two
// wavefronts share a SIMD.  1e5 FSSH trajectories x 1000 steps: 23.7 -> 9.3 ms; before, the coefficients were vector
// loads through the argument pointer, each waited for, 25 round trips to the cache per pass.
template <int NB, int NL, typename R>
__device__ __forceinline__ void sb_body(const SbArgs* __restrict__ Ap, SbVec<R>* lds) {
    static_assert(NB % 4 == 0 && NL % 4 == 0 && NL < NB, "chunks of four modes");
    constexpr int NC = NB / 4, NCR = (NB - NL) / 4;   // chunks, and those whose positions are in registers
    const SbArgs& A = *Ap;
    const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (tid >= A.ntraj) return;   // no barriers below: a lane reads only what it wrote
    const int method = A.method;
    SbVec<R>* xl = lds + threadIdx.x;
    R x[NB - NL], v[NB];
    // the four positions of chunk q, from registers or LDS
    auto load_x = [&](int q) -> SbVec<R> {
        if (q < NCR) return SbVec<R>{x[4 * q], x[4 * q + 1], x[4 * q + 2], x[4 * q + 3]};
        return xl[(q - NCR) * kSbBlock];
    };
    auto store_x = [&](int q, const SbVec<R>& xq) {
        if (q < NCR) {
#pragma unroll
            for (int k = 0; k < 4; ++k) x[4 * q + k] = xq[k];
        } else {
            xl[(q - NCR) * kSbBlock] = xq;
        }
    };
    const SbTab<R> K0 = sb_table<R>(A);
    // collective coordinate X = sum c_j x_j of the initial positions
    R X = (R)0;
    {
        const SbArgs& B = *sb_opaque(Ap);
        const SbTab<R> K = sb_here<R>(K0);
#pragma unroll
        for (int q = 0; q < NC; ++q) {
            SbVec<R> xq;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                xq[k] = (R)B.r0[(int64_t)(4 * q + k) * B.ntraj + tid];
                v[4 * q + k] = (R)B.v0[(int64_t)(4 * q + k) * B.ntraj + tid];
            }
            const SbVec<R> c = K[3 * q + 2];
#pragma unroll
            for (int k = 0; k < 4; ++k) X += c[k] * xq[k];
            store_x(q, xq);
        }
    }
    double E0, E1, U[4];
    eigen2(A.eps + (double)X, A.Delta, -A.eps - (double)X, E0, E1, U, false);
    // initial density: pure adiabatic state, or U^T rho U for a diabatic one (density_matrix_dynamics.jl:37-75)
    double a, b, sx;
    if (A.diabatic) {
        const double u0 = U[A.initial_state * 2], u1 = U[A.initial_state * 2 + 1];
        a = u0 * u0; b = u1 * u1; sx = u0 * u1;
    } else {
        a = (A.initial_state == 0) ? 1.0 : 0.0; b = 1.0 - a; sx = 0.0;
    }
    const double tr = a + b;
    Sig2 s; s.q = a - b; s.x = sx; s.y = 0.0;
    int st = A.initial_state;
    if (method == 0 && A.diabatic) {  // fssh.jl:54
        const double u = philox_uniform((uint64_t)tid, 0u, STREAM_STATE, A.key) * tr;
        st = (u < a) ? 0 : 1;
    }
    double g00, g11, g01;
    rotate_sz(U, g00, g11, g01);
    // system force factor F: k_j = -(w2_j x_j + c_j F) / m_j
    double F = (method == 0) ? ((st == 0) ? g00 : g11) : (g00 * a + g11 * b + 2.0 * g01 * sx);
    double dEc = 0.0, wc = 0.0, tc = 0.0, t = A.t0;
    int nh = 0;
    sb_save(Ap, tid, 0, method, st, tr, s, U);
    // the step loop's launch arguments in scalar registers
    const int nsteps = (int)uniform_sgpr(A.nsteps), save_every = uniform_sgpr(A.save_every), nsub = uniform_sgpr(A.nsub);
    const int rescaling = uniform_sgpr(A.rescaling);
    const double dt = uniform_sgpr(A.dt), eps = uniform_sgpr(A.eps), Delta = uniform_sgpr(A.Delta);
    const double S2 = uniform_sgpr(A.S2), cnorm = uniform_sgpr(A.cnorm);
    const uint64_t key = uniform_sgpr(A.key);
    const R dtR = (R)dt;
    // v -= f (K x + C F), f = 1 (step_B!: v += dt/2 * k) or -1
    auto half_kick = [&](R f, double Fd) {
        const SbTab<R> K = sb_here<R>(K0);
        const R Fr = (R)Fd;
#pragma unroll
        for (int q = 0; q < NC; ++q) {
            const SbVec<R> kx = K[3 * q], kf = K[3 * q + 1];
            const SbVec<R> xq = load_x(q);
#pragma unroll
            for (int k = 0; k < 4; ++k) v[4 * q + k] -= f * (kx[k] * xq[k] + kf[k] * Fr);
        }
    };
    if (nsteps > 0) half_kick((R)1, F);
#pragma unroll 1
    for (int step = 0; step < nsteps; ++step) {
        R Xn = (R)0;
        {
            const SbTab<R> K = sb_here<R>(K0);
            // the next group's coefficients and LDS positions are on their way while one is used
            SbVec<R> c[2][kSbAhead], xa[2][kSbAhead];
#pragma unroll
            for (int i = 0; i < kSbAhead; ++i) c[0][i] = K[3 * i + 2];
#pragma unroll
            for (int q0 = 0; q0 < NC; q0 += kSbAhead) {
                const int cur = (q0 / kSbAhead) & 1;
#pragma unroll
                for (int i = 0; i < kSbAhead; ++i) {
                    const int q = q0 + kSbAhead + i;
                    if (q < NC) c[cur ^ 1][i] = K[3 * q + 2];
                    if (q < NC && q >= NCR) xa[cur ^ 1][i] = load_x(q);
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < kSbAhead; ++i) {
                    const int q = q0 + i;
                    if (q >= NC) break;
                    SbVec<R> xq = q < NCR ? load_x(q) : xa[cur][i];
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        xq[k] = xq[k] + dtR * v[4 * q + k];          // step_A!
                        Xn += c[cur][i][k] * xq[k];
                    }
                    store_x(q, xq);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        double inv_gap;
        eigen2_gap(eps + (double)Xn, Delta, -eps - (double)Xn, E0, E1, inv_gap, U, true);  // update_cache!
        rotate_sz(U, g00, g11, g01);
        {
            const double aa = 0.5 * (tr + s.q), bb = 0.5 * (tr - s.q);
            F = (method == 0) ? ((st == 0) ? g00 : g11) : (g00 * aa + g11 * bb + 2.0 * g01 * s.x);
        }
        R Vc = (R)0;
        {
            const SbTab<R> K = sb_here<R>(K0);
            const R Fn = (R)F;
            SbVec<R> c[2][kSbAhead][3], xa[2][kSbAhead];
#pragma unroll
            for (int i = 0; i < 3 * kSbAhead; ++i) c[0][i / 3][i % 3] = K[i];
#pragma unroll
            for (int q0 = 0; q0 < NC; q0 += kSbAhead) {
                const int cur = (q0 / kSbAhead) & 1;
#pragma unroll
                for (int i = 0; i < 3 * kSbAhead; ++i)
                    if (q0 + kSbAhead + i / 3 < NC) c[cur ^ 1][i / 3][i % 3] = K[3 * (q0 + kSbAhead) + i];
#pragma unroll
                for (int i = 0; i < kSbAhead; ++i)
                    if (q0 + kSbAhead + i < NC && q0 + kSbAhead + i >= NCR) xa[cur ^ 1][i] = load_x(q0 + kSbAhead + i);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < kSbAhead; ++i) {
                    const int q = q0 + i;
                    if (q >= NC) break;
                    const SbVec<R> xq = q < NCR ? load_x(q) : xa[cur][i];
#pragma unroll
                    for (int k = 0; k < 4; ++k) {                    // step_B! twice
                        const R a = c[cur][i][0][k] * xq[k] + c[cur][i][1][k] * Fn;
                        Vc += c[cur][i][2][k] * (v[4 * q + k] - a);
                        v[4 * q + k] = v[4 * q + k] - (R)2 * a;
                        asm volatile("" : "+v"(v[4 * q + k]));   // formed here: left to be sunk, a and the old v both live on
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        const double gap = E1 - E0;
        const double d01c = g01 * inv_gap;             // d_j[0][1] = c_j * d01c
        const double w = d01c * (double)Vc;
        const double tn = t + dt;
        const double dEn = E0 - E1;
        const double inv = nr_rcp(tn - tc);
        Interp2 P;
        P.dE0 = dEc; P.dE1 = (dEn - dEc) * inv; P.w0 = wc; P.w1 = (w - wc) * inv;
        // 100 modes carry a step's difference on: held two orders tighter beside FP64 nuclei
        propagate2<R>(P, s, t, tc, dt, nsub, nsub == 5, 1e-14);
        dEc = dEn; wc = w; tc = tn; t = tn;
        // the save precedes the hop callback (a save time holds the state before the step's callbacks)
        if (save_every > 0 && ((step + 1) % save_every) == 0) sb_save(Ap, tid, (step + 1) / save_every, method, st, tr, s, U);
        if (method == 0) {
            const double sss = 0.5 * (tr + ((st == 0) ? s.q : -s.q));
            const double ratio = s.x / sss;
            const double dsm = (st == 0) ? d01c : -d01c;
            double p = 2.0 * (double)Vc * ratio * dsm * dt;
            // the velocities' change of an accepted or reflected hop, v_j -= (s1 / m_j + s2) c_j
            double s1 = 0.0, s2 = 0.0;
            if (p > 0.0) {
                p = fmin(p, 1.0);
                const double rnd = philox_uniform((uint64_t)tid, (uint32_t)step, STREAM_HOP, key);
                if (p > rnd) {
                    // rescale along d_j = c_j * dms (coupling[new, old]); surface_hopping.jl:64-99
                    const double dms = -dsm;
                    const double dE = (st == 0) ? gap : -gap;
                    bool accept = true;
                    if (rescaling != 2) {
                        const double aq = 0.5 * dms * dms * S2;
                        const double bq = dms * (double)Vc;
                        const double disc = bq * bq - 4.0 * aq * dE;
                        if (disc < 0.0) {
                            accept = false;
                            if (rescaling == 1) {
                                const double nrm = fabs(dms) * cnorm;
                                s2 = 2.0 * (bq / nrm) * (dms / nrm);
                            }
                        } else {
                            const double root = sqrt(disc);
                            const double gam = (bq < 0.0) ? (bq + root) / (2.0 * aq) : (bq - root) / (2.0 * aq);
                            s1 = gam * dms;
                        }
                    }
                    if (accept) { st = 1 - st; ++nh; }
                }
            }
            // one pass for the wavefront (a zero change leaves the other lanes' velocities as they are), so the
            // velocities are not copied around a divergent region every step
            if (__ballot(s1 != 0.0 || s2 != 0.0) != 0) {
                const SbTab<double> cm = (SbTab<double>)uniform_sgpr((uint64_t)sb_opaque(Ap)->c);
                const SbTab<double> im = (SbTab<double>)uniform_sgpr((uint64_t)sb_opaque(Ap)->invm);
#pragma unroll
                for (int q = 0; q < NC; ++q) {
                    const SbVec<double> cq = cm[q], iq = im[q];
#pragma unroll
                    for (int k = 0; k < 4; ++k) v[4 * q + k] = (R)((double)v[4 * q + k] - (s1 * iq[k] + s2) * cq[k]);
                    __builtin_amdgcn_sched_barrier(0);   // chunk by chunk: converted all at once they spill
                }
            }
        }
    }
    if (nsteps > 0) half_kick((R)-1, F);   // the next step's first half kick taken back
    const SbArgs& B = *sb_opaque(Ap);
    const int64_t n = B.ntraj;
#pragma unroll
    for (int q = 0; q < NC; ++q) {
        const SbVec<R> xq = load_x(q);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            B.r[(int64_t)(4 * q + k) * n + tid] = (double)xq[k];
            B.v[(int64_t)(4 * q + k) * n + tid] = (double)v[4 * q + k];
        }
    }
    B.sig[tid] = 0.5 * (tr + s.q);
    B.sig[n + tid] = 0.5 * (tr - s.q);
    B.sig[2 * n + tid] = s.x;
    B.sig[3 * n + tid] = s.y;
    B.state[tid] = st;
    B.steps[tid] = (int32_t)nsteps;
    B.nhops[tid] = nh;
}

constexpr int kSbLds32 = 48, kSbLds64 = 40;   // modes whose positions are in LDS (12 KB, 20 KB a wavefront)
__global__ __launch_bounds__(kSbBlock) __attribute__((amdgpu_waves_per_eu(2)))
void sb_kernel_f32(const SbArgs* __restrict__ Ap) {
    __shared__ SbVec<float> lds[kSbLds32 / 4 * kSbBlock];
    sb_body<kBathModes, kSbLds32, float>(Ap, lds);
}
__global__ __launch_bounds__(kSbBlock) void sb_kernel_f64(const SbArgs* __restrict__ Ap) {
    __shared__ SbVec<double> lds[kSbLds64 / 4 * kSbBlock];
    sb_body<kBathModes, kSbLds64, double>(Ap, lds);
}

// ---------------------------------------------------------------------------
// Host side.
// ---------------------------------------------------------------------------
int32_t sb_sample_initial(nqcd_handle_t* h, const nqcd_sampler_desc* S, uint64_t seed) {
    const int nb = (int)h->sb_omega.size();
    if (nb != kBathModes)
        return fail(h, NQCD_ERR_UNSUPPORTED, "spin-boson kernels are built for 100 bath modes");
    if (h->D != nb) return fail(h, NQCD_ERR_ARG, "problem dofs must equal the number of bath modes");
    if (S->nparams != 4 * nb || !S->params)
        return fail(h, NQCD_ERR_ARG, "bath sampler params: mu_r[nb], sd_r[nb], mu_v[nb], sd_v[nb]");
    h->ntraj = S->ntraj;
    HIPCHK(h, h->bath.ensure(sizeof(double) * 10 * nb + sizeof(float) * 3 * nb));
    std::vector<double> tab(10 * nb);
    for (int j = 0; j < nb; ++j) {
        tab[j] = h->sb_omega[j] * h->sb_omega[j];
        tab[nb + j] = h->sb_c[j];
        tab[2 * nb + j] = h->inv_mass[j];
        for (int k = 0; k < 4; ++k) tab[3 * nb + 4 * j + k] = S->params[k * nb + j];  // per-mode interleave
    }
    const double hdt = 0.5 * h->prob.dt;
    std::vector<float> tabf(3 * nb);
    for (int j = 0; j < nb; ++j) {
        double* t4 = tab.data() + 7 * nb + 12 * (j / 4) + j % 4;   // chunks of four modes: kick, force and c
        t4[0] = hdt * tab[j] * tab[2 * nb + j];
        t4[4] = hdt * tab[nb + j] * tab[2 * nb + j];
        t4[8] = tab[nb + j];
        for (int k = 0; k < 3; ++k) tabf[12 * (j / 4) + 4 * k + j % 4] = (float)t4[4 * k];
    }
    HIPCHK(h, hipMemcpy(h->bath.p, tab.data(), sizeof(double) * 10 * nb, hipMemcpyHostToDevice));
    HIPCHK(h, hipMemcpy(h->bath.as<char>() + sizeof(double) * 10 * nb, tabf.data(), sizeof(float) * 3 * nb,
                        hipMemcpyHostToDevice));
    // harmonic Wigner sampling: counter (traj, mode, stream 0) -> z0 for R, z1 for V
    HIPCHK(h, h->r0.ensure(sizeof(double) * nb * h->ntraj));
    HIPCHK(h, h->v0.ensure(sizeof(double) * nb * h->ntraj));
    HIPCHK(h, launch_sample_gaussian(h->ntraj, nb, h->bath.as<double>() + 3 * nb, seed, h->r0.as<double>(),
                                     h->v0.as<double>(), h->stream));
    HIPCHK(h, hipStreamSynchronize(h->stream));
    h->sb_state = S->initial_state;
    h->sb_diabatic = S->state_basis == 1;
    h->sb_seed = seed;
    return NQCD_OK;
}

int32_t sb_run(nqcd_handle_t* h, double t0, int64_t nsteps, const nqcd_term_desc* term, uint64_t key) {
    if (term && term->kind != NQCD_TERM_NONE)
        return fail(h, NQCD_ERR_UNSUPPORTED, "termination predicates are not supported for system-bath models");
    const int nb = kBathModes;
    const int64_t n = h->ntraj;
    HIPCHK(h, h->r.ensure(sizeof(double) * nb * n));
    HIPCHK(h, h->v.ensure(sizeof(double) * nb * n));
    HIPCHK(h, h->sig.ensure(sizeof(double) * 4 * n));
    HIPCHK(h, h->state.ensure(sizeof(int32_t) * n));
    HIPCHK(h, h->steps.ensure(sizeof(int32_t) * n));
    HIPCHK(h, h->nhops.ensure(sizeof(int32_t) * n));
    HIPCHK(h, h->save_ad.ensure(sizeof(double) * 2 * h->nsave * n));
    HIPCHK(h, h->save_di.ensure(sizeof(double) * 2 * h->nsave * n));
    HIPCHK(h, h->save_state.ensure(sizeof(int32_t) * h->nsave * n));
    HIPCHK(h, launch_zero(h->save_ad.p, sizeof(double) * 2 * h->nsave * n, h->stream));
    HIPCHK(h, launch_zero(h->save_di.p, sizeof(double) * 2 * h->nsave * n, h->stream));
    HIPCHK(h, launch_zero(h->save_state.p, sizeof(int32_t) * h->nsave * n, h->stream));
    SbArgs A{};
    A.ntraj = n;
    A.method = (h->prob.method == NQCD_METHOD_FSSH) ? 0 : 1;
    A.rescaling = h->prob.rescaling;
    A.nsub = h->prob.electronic_substeps > 0 ? h->prob.electronic_substeps : 5;
    A.save_every = h->save_every;
    A.nsave = h->nsave;
    A.initial_state = h->sb_state;
    A.diabatic = h->sb_diabatic ? 1 : 0;
    A.dt = h->prob.dt;
    A.t0 = t0;
    A.eps = h->sb_eps;
    A.Delta = h->sb_delta;
    double S2 = 0.0, c2 = 0.0;
    for (int j = 0; j < nb; ++j) { S2 += h->sb_c[j] * h->sb_c[j] * h->inv_mass[j]; c2 += h->sb_c[j] * h->sb_c[j]; }
    A.S2 = S2;
    A.cnorm = std::sqrt(c2);
    A.nsteps = nsteps;
    A.key = key;
    const double* tab = h->bath.as<double>();
    A.w2 = tab; A.c = tab + nb; A.invm = tab + 2 * nb;
    A.kd = tab + 7 * nb;
    A.kf = reinterpret_cast<const float*>(h->bath.as<char>() + sizeof(double) * 10 * nb);
    A.r0 = h->r0.as<double>(); A.v0 = h->v0.as<double>();
    A.r = h->r.as<double>(); A.v = h->v.as<double>(); A.sig = h->sig.as<double>();
    A.state = h->state.as<int32_t>(); A.steps = h->steps.as<int32_t>(); A.nhops = h->nhops.as<int32_t>();
    A.save_pop_ad = h->save_ad.as<double>(); A.save_pop_di = h->save_di.as<double>();
    A.save_state = h->save_state.as<int32_t>();
    HIPCHK(h, h->args_dev.ensure(sizeof(SbArgs)));
    HIPCHK(h, hipMemcpyAsync(h->args_dev.p, &A, sizeof(SbArgs), hipMemcpyHostToDevice, h->stream));
    const int block = kSbBlock;
    const int grid = (int)((n + block - 1) / block);
    HIPCHK(h, hipEventRecord(h->ev0, h->stream));
    if (h->prob.precision == NQCD_PREC_FP64)
        hipLaunchKernelGGL(sb_kernel_f64, dim3(grid), dim3(block), 0, h->stream, h->args_dev.as<const SbArgs>());
    else
        hipLaunchKernelGGL(sb_kernel_f32, dim3(grid), dim3(block), 0, h->stream, h->args_dev.as<const SbArgs>());
    HIPCHK(h, hipGetLastError());
    HIPCHK(h, hipEventRecord(h->ev1, h->stream));
    h->stats.block = block;
    h->stats.grid = grid;
    h->stats.launches = 1;
    return NQCD_OK;
}

}  // namespace nqcd
