// iesh.hip -- independent-electron surface hopping (IESH) and EhrenfestNA on the Newns-Anderson
// impurity model, one trajectory per workgroup.
//
// Reference path: VerletwithElectronics (src/DynamicsMethods/IntegrationAlgorithms/
// verlet_with_electronics.jl:42-69), the wavefunction propagator (src/DynamicsUtils/
// wavefunction_dynamics.jl:15-58), the IESH force and hop (src/DynamicsMethods/SurfaceHoppingMethods/
// iesh.jl:190-207,231-335,390-441) and the EhrenfestNA force (src/DynamicsMethods/EhrenfestMethods/
// ehrenfest_na.jl:72-86).
//
// Model: N = M + 1 states, impurity h(x) = U1 - U0 coupled with a constant V to M bath levels
// eps_k = a + k (b - a)/(M - 1), V = sqrt(Gamma (b - a)/(M - 1) / 2 pi).  The Hamiltonian is an
// arrowhead matrix, so per step:
//   * eigen: root i of the secular function f(l) = l - h - V^2 sum_k 1/(l - eps_k) lies in
//     (eps_{i-1}, eps_i); rational-model iteration from the previous step's root, one thread per
//     root (3 to 5 evaluations of f per root and step).
//     The impurity component of eigenvector i is u_i = f'(E_i)^(-1/2) > 0 (a continuous gauge).
//   * dV/dx only touches the impurity entry, so U^T dV U = dh u u^T and the nonadiabatic coupling
//     is d_ij = dh u_i u_j / (E_j - E_i).
//   * propagator: psi <- exp(-i dt (diag(E) - i v d)) psi, applied as a Taylor series whose length
//     follows from the bound ||dt H|| <= dt max|E| + ||dt v d||_F (remainder below 1e-17); each term is one real GEMM
//     (-dt v dh W) [Re psi | Im psi] on FP64 MFMA 16x16x4 plus the diagonal part.  The reference
//     diagonalises H with zheevr and forms U exp(-i Lambda dt) U^H; both give exp(-i H dt) to
//     rounding.
//   * IESH hop: S = psi[occ, :], det S and S^-1 by one Gauss-Jordan elimination (partial pivoting) in
//     registers, the reference's early-exit estimate, and on the steps that pass it the replaced-row determinants by the
//     determinant lemma det(S with row n <- psi_m) = det(S) (psi_m S^-1)_n, so
//     P(n -> m) = 2 dt Re((psi_m S^-1)_n) v_dot_d[m, n]; cumulative selection electrons outer,
//     unoccupied states inner (iesh.jl:318-335).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "ensemble.h"
#include "handle.h"
#include "iesh.h"
#include "nqcd_device.h"

namespace nqcd {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int kIeMaxNe = 64;
constexpr int kIeMaxStates = 128;
constexpr double kFarPole = 1e300;  // pads the bath levels to a multiple of 16: nothing in the secular sums
constexpr size_t kIeLdsBytes = 160 * 1024;  // LDS of one gfx950 compute unit

struct IeshArgs {
    int64_t ntraj;
    int64_t nsteps;
    int32_t N, M, Ne, cw;         // states, bath levels, electrons, psi columns in use (16 * column tiles)
    int32_t sb_len, pad0;         // doubles of the S / probability workspace in LDS
    int32_t method;               // 0 = IESH, 1 = EhrenfestNA
    int32_t rescaling, estimate, edc;
    int32_t save_every, nsave;
    int32_t P, pad1;              // ring-polymer beads (1: no ring polymer)
    double dt, mass, edc_C;
    double wn;                    // ring-polymer frequency P kT
    uint64_t key;
    double mw2, g, dG, V, a, de;  // model
    const double* r0; const double* v0; const int32_t* occ0; const double* psi0;  // psi0 may be null
    double* r; double* v; double* psi; int32_t* occ; int32_t* nhops; int32_t* steps;
    double* save_di;              // (nsave, N, ntraj)
    double* save_ad;              // (nsave, N, ntraj)
};

template <int NT>
__device__ __forceinline__ double block_max(double v, double* red) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = red[0];
#pragma unroll
    for (int j = 1; j < NT; ++j) s = fmax(s, red[j]);
    return s;
}

struct Scalars { double h, dh, dU0; };

__device__ __forceinline__ Scalars na_scalars(const IeshArgs& A, double x) {
    Scalars s;
    const double U0 = 0.5 * A.mw2 * x * x;
    const double U1 = 0.5 * A.mw2 * (x - A.g) * (x - A.g) + A.dG;
    s.h = U1 - U0;
    s.dh = A.mw2 * (x - A.g) - A.mw2 * x;
    s.dU0 = A.mw2 * x;
    return s;
}

// 1/x from the hardware estimate and two Newton-Raphson corrections (within an ulp).
__device__ __forceinline__ double rcp_nr(double x) {
    double r = __builtin_amdgcn_rcp(x);
    double e = fma(-x, r, 1.0);
    r = fma(r, e, r);
    e = fma(-x, r, 1.0);
    return fma(r, e, r);
}

// Root i of the secular function f(l) = l - h - V^2 sum_k 1/(l - eps_k), which increases from
// -inf to +inf on its interval (lo, hi) = (eps_{i-1}, eps_i) (the outer roots have one finite end).
// Each iteration evaluates f, f' once and steps to the root of a two-pole rational model that
// matches f and f' at the current point ("middle way", R.-C. Li, LAPACK Working Note 89):
//   F(y) = c + bl / (y - eps_{i-1}) + bh / (y - eps_i),
// where the poles below and above the interval carry their own parts of f' and the slope of the
// linear term is shared between them; the model's root is a quadratic's, and a step that leaves
// the bracket (kept from the signs of f) bisects instead.  Stops when |f| is at its rounding level,
// when the step is a few ulps or when the bracket is narrower than tol.  Returns E_i and
// f'(E_i) = 1 + V^2 sum_k 1/(E_i - eps_k)^2.
// G lanes (1, 2 or 4 consecutive lanes, sub = lane mod G) share a root: lane sub sums the poles
// k = sub, sub + G, ..., and the partial sums are combined by DPP exchanges whose results have
// the same bits in every lane of the group, so the group iterates in lockstep.
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double x) {
    const long long bits = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(bits & 0xffffffffll), CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(bits >> 32), CTRL, 0xF, 0xF, false);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

template <int G>
__device__ __forceinline__ double group_sum(double v) {
    if (G >= 2) v += dpp_f64<0xB1>(v);  // quad_perm [1,0,3,2]
    if (G >= 4) v += dpp_f64<0x4E>(v);  // quad_perm [2,3,0,1]
    return v;
}

template <int G = 1>
__device__ double secular_root(const double* eps, int M, int i, double V2, double h, double lo, double hi,
                               double guess, double tol, double& fp, int sub = 0) {
    const bool has_lo = i > 0, has_hi = i < M;
    const double dl = has_lo ? eps[i - 1] : lo, dh = has_hi ? eps[i] : hi;
    const double wl = has_lo ? (has_hi ? 0.5 : 1.0) : 0.0;  // share of the linear term's slope at the lower pole
    double lam = (guess > lo && guess < hi) ? guess : 0.5 * (lo + hi);
    fp = 1.0;
    for (int it = 0; it < 100; ++it) {
        // q_k > 0 below the interval, < 0 above it; four poles at a time (eps is padded with far poles)
        double sl = 0.0, sl2 = 0.0, sh = 0.0, sh2 = 0.0;
        for (int k = sub; k < M; k += 4 * G) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const double q = rcp_nr(lam - eps[k + u * G]);
                const double ql = fmax(q, 0.0), qh = fmin(q, 0.0);
                sl += ql;
                sh += qh;
                sl2 = fma(ql, ql, sl2);
                sh2 = fma(qh, qh, sh2);
            }
        }
        if (G > 1) {
            sl = group_sum<G>(sl);
            sh = group_sum<G>(sh);
            sl2 = group_sum<G>(sl2);
            sh2 = group_sum<G>(sh2);
        }
        const double f = lam - h - V2 * (sl + sh);
        fp = 1.0 + V2 * (sl2 + sh2);
        if (fabs(f) <= 8.0 * __DBL_EPSILON__ * (fabs(lam) + fabs(h) + V2 * (sl - sh))) break;
        if (f > 0.0) hi = lam;
        else lo = lam;
        const double ql = has_lo ? -(V2 * sl2 + wl) * (lam - dl) : 0.0, qh = has_hi ? -(V2 * sh2 + (1.0 - wl)) * (lam - dh) : 0.0;
        const double bl = ql * (lam - dl), bh = qh * (lam - dh);
        const double c = f - ql - qh;
        double nl;
        if (has_lo && has_hi) {
            // c t (t - D) + bl (t - D) + bh t = 0 with t = y - dl, D = dh - dl; root in (0, D)
            const double D = dh - dl;
            const double a1 = bl + bh - c * D, a0 = -bl * D;
            const double sq = sqrt(fmax(a1 * a1 - 4.0 * c * a0, 0.0));
            const double den = a1 > 0.0 ? -a1 - sq : -a1 + sq;
            nl = dl + den * rcp_nr(2.0 * c);
            if (!(nl >= lo && nl <= hi)) nl = dl + 2.0 * a0 * rcp_nr(den);
        } else if (has_hi) {
            nl = dh - bh * rcp_nr(c);
        } else {
            nl = dl - bl * rcp_nr(c);
        }
        if (fabs(nl - lam) <= 4.0 * __DBL_EPSILON__ * fabs(lam) || (hi - lo) <= tol) break;
        if (!(nl > lo && nl < hi)) nl = 0.5 * (lo + hi);
        lam = nl;
    }
    return lam;
}

__device__ __forceinline__ double readlane_f64(double x, int lane) {
    const long long bits = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_readlane((int)(bits & 0xffffffffll), lane);
    const int hi = __builtin_amdgcn_readlane((int)(bits >> 32), lane);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

// Sums over rows of 16 lanes and over the wavefront, the same value in every lane: butterflies inside the rows, then
// the four rows.
__device__ __forceinline__ double row_sum(double v) {
    v += dpp_f64<0xB1>(v);
    v += dpp_f64<0x4E>(v);
    v += dpp_f64<0x141>(v);  // row_half_mirror
    v += dpp_f64<0x140>(v);  // row_mirror
    return v;
}
__device__ __forceinline__ double wave_sum(double v) {
    v = row_sum(v);
    return (readlane_f64(v, 0) + readlane_f64(v, 16)) + (readlane_f64(v, 32) + readlane_f64(v, 48));
}

// Eigenvalue ir of the Newns-Anderson matrix at impurity energy h: the secular root on its
// bracket (the outer brackets reach past the band and h by the coupling norm zn = sqrt(M) V);
// warm starts from `guess` (from `prev` where that leaves the bracket), a cold start from below the bracket.
// Also returns f'(E_ir).
template <int G = 1>
__device__ __forceinline__ double na_root(const double* eps, int M, double a, double V2, double zn, double h, int ir,
                                          bool warm, double guess, double prev, double& fp, int sub = 0) {
    const double lo = (ir == 0) ? fmin(h, eps[0]) - zn - 1e-3 * (zn + 1e-300) : eps[ir - 1];
    const double hi = (ir == M) ? fmax(h, eps[M - 1]) + zn + 1e-3 * (zn + 1e-300) : eps[ir];
    const double scale = fmax(fmax(fabs(a), fabs(eps[M - 1])), fabs(h)) + zn;
    return secular_root<G>(eps, M, ir, V2, h, lo, hi, warm ? ((guess > lo && guess < hi) ? guess : prev) : lo - 1.0,
                           4.0e-16 * scale, fp, sub);
}

// One step of a wavefront arg-max over (mag, idx) with the DPP lane pattern CTRL (larger mag
// wins, the lower idx on ties).
template <int CTRL>
__device__ __forceinline__ void argmax_dpp(double& mag, int& idx) {
    const long long bits = __double_as_longlong(mag);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(bits & 0xffffffffll), CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(bits >> 32), CTRL, 0xF, 0xF, false);
    const int oi = __builtin_amdgcn_update_dpp(0, idx, CTRL, 0xF, 0xF, false);
    const double om = __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
    if (om > mag || (om == mag && oi < idx)) { mag = om; idx = oi; }
}

// Wavefront-uniform arg-max of (mag, idx), the lowest idx among equal maxima: butterflies inside
// each row of 16 lanes (quad_perm [1,0,3,2], [2,3,0,1], row_half_mirror, row_mirror), then the
// four row results compared in lane order.
__device__ __forceinline__ void wave_argmax(double& mag, int& idx) {
    argmax_dpp<0xB1>(mag, idx);
    argmax_dpp<0x4E>(mag, idx);
    argmax_dpp<0x141>(mag, idx);
    argmax_dpp<0x140>(mag, idx);
    double bm = readlane_f64(mag, 0);
    int bi = __builtin_amdgcn_readlane(idx, 0);
#pragma unroll
    for (int row = 1; row < 4; ++row) {
        const double m = readlane_f64(mag, 16 * row);
        const int i = __builtin_amdgcn_readlane(idx, 16 * row);
        if (m > bm || (m == bm && i < bi)) { bm = m; bi = i; }
    }
    mag = bm;
    idx = bi;
}

// Inverse and determinant of an Ne x Ne complex matrix (Ne <= 64) by Gauss-Jordan elimination in place with partial
// pivoting (largest |.| in the column among the rows not yet used, lowest row on ties), by NT wavefronts: lane r holds
// row r, wavefront w the columns w, w + NT, ..., rotated so that its next pivot column is always x[0].  Rows are never
// moved: with row q_p the pivot row of column p, entry (p, q_c) of the inverse ends in row q_p, column c, and the sign
// of the pivot permutation comes from counting, at each step, the unused rows above the pivot row.  The column's owner
// picks the pivot and leaves the multipliers in LDS; one barrier a pivot (two buffers), everything else in registers.
// In place of one wavefront's LU through LDS followed by a workgroup's Gauss-Jordan through LDS, with the populations
// saved by a matrix product and the secular sums four poles at a time: 8192 trajectories of 41 states, 100 steps,
// 65.9 -> 56 ms; 2048 of 101 states, 50 steps, 95.5 -> 66 ms.  buf: 2 x 136 doubles; piv[p] = q_p; myp: the column whose
// pivot row this lane's row was; on return x[j] is column w + NT ((j + rot) % KC).  False for a singular matrix (a zero
// pivot column).  Called by whole workgroups of 64 NT lanes; the caller's previous use of buf and piv ends with a barrier.
template <int NT, int KC>
__device__ __forceinline__ bool block_inverse(double (&xr)[KC], double (&xi)[KC], int Ne, int w, int l, double* buf, int* piv,
                                              double& dre, double& dim, int& myp, int& rot) {
    bool used = l >= Ne;
    double ar = 1.0, ai = 0.0;
    int inv = 0, owner = 0;
    myp = 0;
    rot = 0;
    for (int p = 0; p < Ne; ++p) {
        double* B = buf + (p & 1) * 136;
        if (w == owner) {
            double mag = used ? -1.0 : xr[0] * xr[0] + xi[0] * xi[0];
            int q = l;
            wave_argmax(mag, q);
            const bool ok = mag > 0.0;
            const double pr = readlane_f64(xr[0], q), pi = readlane_f64(xi[0], q), ip = 1.0 / mag;
            B[2 * l] = (xr[0] * pr + xi[0] * pi) * ip;      // S[r][p] / pivot
            B[2 * l + 1] = (xi[0] * pr - xr[0] * pi) * ip;
            if (l == 0) {
                B[128] = pr;
                B[129] = pi;
                B[130] = pr * ip;                           // 1 / pivot
                B[131] = -pi * ip;
                piv[p] = ok ? q : -1;
            }
        }
        __syncthreads();
        const int q = __builtin_amdgcn_readfirstlane(piv[p]);
        if (q < 0) { dre = 0.0; dim = 0.0; return false; }
        const double pr = B[128], pi = B[129];
        const double fr = l == q ? -B[130] : B[2 * l], fi = l == q ? -B[131] : B[2 * l + 1];
        {
            const double nr = ar * pr - ai * pi, ni = ar * pi + ai * pr;
            ar = nr;
            ai = ni;
        }
        inv += __popcll(__ballot(!used && l < q));
        if (l == q) { used = true; myp = p; }
#pragma unroll
        for (int j = 0; j < KC; ++j) {  // rows r != q: x - f y; row q: y / pivot
            const double yr = readlane_f64(xr[j], q), yi = readlane_f64(xi[j], q);
            const double zr = l == q ? 0.0 : xr[j], zi = l == q ? 0.0 : xi[j];
            xr[j] = fma(fi, yi, fma(-fr, yr, zr));
            xi[j] = fma(-fi, yr, fma(-fr, yi, zi));
        }
        if (w == owner) {  // the pivot column's own place takes the identity's column; then the next one to the front
            const double tr = -fr, ti = -fi;
#pragma unroll
            for (int j = 0; j + 1 < KC; ++j) { xr[j] = xr[j + 1]; xi[j] = xi[j + 1]; }
            xr[KC - 1] = tr;
            xi[KC - 1] = ti;
            ++rot;
        }
        if (++owner == NT) owner = 0;
    }
    dre = (inv & 1) ? -ar : ar;
    dim = (inv & 1) ? -ai : ai;
    return true;
}

// Norms of dt H above which the Taylor series takes another term: the remainder x^(K+1) / (K+1)! e^x of K terms passes
// 1e-17 at kTaylorFrom[K] (rounded down).  The last entry lies above the 0.5 of a sub-step.
__constant__ float kTaylorFrom[16] = {
    9.999990e-18f, 4.472131e-09f, 3.914859e-06f, 1.244626e-04f, 1.036921e-03f, 4.391071e-03f, 1.257669e-02f, 2.812954e-02f,
    5.324670e-02f, 8.955433e-02f, 1.380727e-01f, 1.992883e-01f, 2.732652e-01f, 3.597589e-01f, 4.583142e-01f, 5.683443e-01f};

// The thread index made opaque where a phase of the step begins: what a phase derives from it (LDS addresses, row
// and column numbers) is then computed there, instead of being hoisted out of the step loop and held in registers
// through every other phase.
__device__ __forceinline__ int ie_tid() {
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}
#define IE_IDS const int tid = ie_tid(), w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63; (void)w; (void)l;

// Bound by the propagator (8 or 9 terms of N x N x 2 Ne on FP64 MFMA, two barriers and an LDS round trip a term: the
// matrix cores are busy for 17.7 of 55 ms at 41 states and 29.4 of 66 ms at 101, where seven wavefronts share four
// SIMDs) and, up to 64 states, by the latency of the phases around it, which one workgroup cannot hide: there the
// registers are held to three wavefronts a SIMD, so that three or four trajectories share a compute unit.  Larger
// problems fill the LDS with one trajectory and keep two wavefronts' registers.  The phases exchange sums once
// (coupling norm, hop bound, orbital weight ride on the propagator's registers and barriers), divide by Newton-Raphson
// reciprocals, save populations by a product on the matrix cores and invert S in registers.
// 8192 trajectories of 41 states, 100 steps: 91 -> 56 ms; 2048 of 101 states, 50 steps: 103 -> 66 ms.
// RPB: ring polymer (BCBWavefunction), a separate instantiation so the one-bead kernels carry none of it
template <int NT, int CTM, bool RPB>
__global__ __launch_bounds__(64 * NT) __attribute__((amdgpu_waves_per_eu(NT <= 4 && CTM <= 4 && !RPB ? 3 : 2))) void iesh_kernel(const IeshArgs A) {
    constexpr int NP = 16 * NT;  // padded state count (rows of psi / W tiles)
    constexpr int B = 64 * NT;
    constexpr int KF = 4 * NT;   // A-fragments per lane (K = NP in steps of 4)
    extern __shared__ double smem[];
    constexpr int CW = 16 * CTM; // row stride of psi in LDS (compile time, so LDS offsets are immediates)
    const int N = A.N, M = A.M, Ne = A.Ne, CT = A.cw / 16;
    double* Tb = smem;                       // NP x CW: psi (Re, Im interleaved per electron) / Taylor term
    double* Sb = Tb + NP * CW;               // Ne x Ne complex S^-1
    double* E = Sb + A.sb_len;               // NP adiabatic energies
    double* U = E + NP;                      // NP impurity components of the eigenvectors
    double* eps = U + NP;                    // NP bath levels
    double* red = eps + NP;                  // NT reduction slots
    double* pcol = red + 8;                  // max(NP, 2 kIeMaxNe) per-state / per-electron temporaries
    double* part = pcol + (NP > 2 * kIeMaxNe ? NP : 2 * kIeMaxNe);  // 8 kIeMaxNe partial sums / probabilities
    double* scal = part + 8 * kIeMaxNe;      // 8 broadcast scalars
    int* occ = reinterpret_cast<int*>(scal + 8);  // kIeMaxNe occupied states
    int* isocc = occ + kIeMaxNe;                  // NP electron index occupying the state, -1 if empty
    int* piv = isocc + NP;                        // kIeMaxNe pivot rows
    int* unocc = piv + kIeMaxNe;                  // NP unoccupied states, ascending
    // ring polymers (P > 1): bead positions, velocities, accelerations, normal-mode pair, and the
    // eigenpairs of one bead (these arrays are allocated only when P > 1)
    const int P = RPB ? A.P : 1;
    constexpr bool rp = RPB;
    double* brl = reinterpret_cast<double*>(unocc + NP);
    double* bvl = brl + 64;
    double* bal = bvl + 64;
    double* bq = bal + 64;
    double* bp = bq + 64;
    double* Eb = bp + 64;
    double* Ub = Eb + NP;

    const int tid = threadIdx.x, w = tid >> 6, l = tid & 63;
    const double dt = A.dt;
    const double V2 = A.V * A.V;
    for (int k = tid; k < NP; k += B) eps[k] = (k < M) ? A.a + k * A.de : kFarPole;
    __syncthreads();
    const double zn = sqrt((double)M) * A.V;
    const float order_from = (threadIdx.x & 63) < 16 ? kTaylorFrom[threadIdx.x & 15] : __builtin_inff();

    for (int64_t traj = blockIdx.x; traj < A.ntraj; traj += gridDim.x) {
        __syncthreads();
        // ---- load the trajectory --------------------------------------------------------------
        for (int idx = tid; idx < NP * CW; idx += B) {
            const int row = idx / CW, col = idx - row * CW;
            double val = 0.0;
            if (A.psi0 && row < N && col < 2 * Ne) val = A.psi0[(((size_t)traj * N + row) * Ne + (col >> 1)) * 2 + (col & 1)];
            Tb[idx] = val;
        }
        for (int s = tid; s < NP; s += B) isocc[s] = -1;
        if (tid < Ne) occ[tid] = A.occ0[(size_t)traj * Ne + tid];
        __syncthreads();
        if (tid < Ne) {
            isocc[occ[tid]] = tid;
            if (!A.psi0) Tb[occ[tid] * CW + 2 * tid] = 1.0;  // psi[state_e, e] = 1 (iesh.jl:174-180)
        }
        // The determinant bound of the hop estimate (below) needs orthonormal electron orbitals:
        // true for psi[state_e, e] = 1, checked for a given psi; propagation keeps it, EDC does not.
        bool det_bound = A.method == 0 && A.estimate && !A.edc;
        if (det_bound && A.psi0) {
            __syncthreads();
            double dev = 0.0;
            for (int k = tid; k < Ne * Ne; k += B) {
                const int e1 = k / Ne, e2 = k - e1 * Ne;
                double gr = (e1 == e2) ? -1.0 : 0.0, gi = 0.0;
                for (int a = 0; a < N; ++a) {
                    const double xr = Tb[a * CW + 2 * e1], xi = Tb[a * CW + 2 * e1 + 1];
                    const double yr = Tb[a * CW + 2 * e2], yi = Tb[a * CW + 2 * e2 + 1];
                    gr += xr * yr + xi * yi;
                    gi += xr * yi - xi * yr;
                }
                dev = fmax(dev, fmax(fabs(gr), fabs(gi)));
            }
            det_bound = block_max<NT>(dev, red) <= 1e-10;
            __syncthreads();
        }
        auto bead_mean = [&](const double* a) {
            double m = 0.0;
            for (int b = 0; b < P; ++b) m += a[b];
            return m / P;
        };
        double x, v;
        if (rp) {
            if (tid < P) {
                brl[tid] = A.r0[(size_t)traj * P + tid];
                bvl[tid] = A.v0[(size_t)traj * P + tid];
            }
            __syncthreads();
            x = bead_mean(brl);
            v = bead_mean(bvl);
        } else {
            x = A.r0[traj];
            v = A.v0[traj];
        }
        double Eprev = -1.0, u2prev = 0.0, hprev = 0.0;
        bool warm = false;
        int nh = 0;

        // eigen at x (all threads); leaves E, U in LDS and returns the model scalars
        auto eigen = [&](double xx) -> Scalars {
            IE_IDS
            const Scalars s = na_scalars(A, xx);
            // four lanes per root, roots dealt round-robin over the wavefronts (16 NT >= N slots)
            const int ir = (l >> 2) * NT + w, sub = l & 3;
            if (ir < N) {
                double fp;
                // first-order start: dE/dh = u^2 (the impurity entry alone depends on x)
                const double lam = na_root<4>(eps, M, A.a, V2, zn, s.h, ir, warm, Eprev + (s.h - hprev) * u2prev, Eprev, fp, sub);
                const double u = 1.0 / sqrt(fp);
                if (sub == 0) {
                    E[ir] = lam;
                    U[ir] = u;
                }
                Eprev = lam;
                u2prev = u * u;
            } else if (ir < NP && sub == 0) {
                E[ir] = 0.0;
                U[ir] = 0.0;
            }
            warm = true;
            hprev = s.h;
            __syncthreads();
            return s;
        };
        // eigenpairs at a bead position into Eb, Ub (cold start: no roots are kept per bead)
        auto bead_eigen = [&](double xx) -> Scalars {
            IE_IDS
            const Scalars s = na_scalars(A, xx);
            const int ir = (l >> 2) * NT + w, sub = l & 3;
            if (ir < N) {
                double fp;
                const double lam = na_root<4>(eps, M, A.a, V2, zn, s.h, ir, false, 0.0, 0.0, fp, sub);
                if (sub == 0) {
                    Eb[ir] = lam;
                    Ub[ir] = 1.0 / sqrt(fp);
                }
            }
            __syncthreads();
            return s;
        };
        // acceleration at the eigenpairs whose impurity components are Uv, with the wavefunction in Tb
        // (iesh.jl:190-207, ehrenfest_na.jl:72-86; per bead rpiesh.jl:20-38, rpehrenfest_na.jl:14-40).  Ends without a
        // barrier: pcol (EhrenfestNA), occ, Uv and Tb are still being read, and the caller puts a workgroup barrier
        // before the next write to any of them.
        auto accel = [&](const Scalars& s, const double* Uv) -> double {
            IE_IDS
            // summed by every wavefront for itself (Ne <= 64)
            double t = 0.0;
            if (A.method == 0) {
                if (l < Ne) { const double u = Uv[occ[l]]; t = u * s.dh * u; }
            } else {
                if (tid < Ne) {
                    double re = 0.0, im = 0.0;
                    for (int a = 0; a < N; ++a) {
                        re += Uv[a] * Tb[a * CW + 2 * tid];
                        im += Uv[a] * Tb[a * CW + 2 * tid + 1];
                    }
                    pcol[tid] = s.dh * (re * re + im * im);
                }
                __syncthreads();
                if (l < Ne) t = pcol[l];
            }
            return -(s.dU0 + wave_sum(t)) / A.mass;
        };
        // Diabatic populations: component a of eigenvector b is U_ab = u_b (a = 0, impurity) or
        // V u_b / (E_b - eps_{a-1}) (bath level a - 1).  IESH (iesh.jl:351-369): per electron
        // diag(U rho U^T), rho = offdiag(c c^T) + e_s e_s^T with c = Re psi_e, i.e.
        // (sum_b U_ab c_b)^2 - sum_b U_ab^2 c_b^2 + U_as^2; EhrenfestNA: sum_e |(U psi)_{a e}|^2.
        auto save = [&](int slot) {
            IE_IDS
            if (slot >= A.nsave) return;
            // U psi on the matrix cores, as a term of the propagator; IESH takes the real columns and puts the rest,
            // sum_b U_ab^2 ([b occupied] - sum_e c_b^2), in weights
            const int g = l >> 4, own = (16 * w + g) * CW + (l & 15);
            const bool drop = A.method == 0 && (l & 1);
            double rs[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                double q = 0.0;
                for (int ct = 0; ct < CT; ++ct) { const double c = Tb[own + 4 * r * CW + 16 * ct]; q += c * c; }
                rs[r] = row_sum(drop ? 0.0 : q);
                if ((l & 15) == 0) {
                    const int b = 16 * w + 4 * r + g;
                    pcol[b] = (isocc[b] >= 0 ? 1.0 : 0.0) - rs[r];
                }
            }
            __syncthreads();
            {
                const int a = 16 * w + (l & 15);
                const double ea = (a > 0 && a < N) ? eps[a - 1] : 0.0;
                double Af[KF], corr = 0.0;
#pragma unroll
                for (int kk = 0; kk < KF; ++kk) {
                    const int k = 4 * kk + g;
                    double u = (a == 0) ? U[k] : A.V * U[k] * rcp_nr(E[k] - ea);
                    if (a >= N || k >= N) u = 0.0;
                    Af[kk] = u;
                    corr += u * u * pcol[k];
                }
                corr += __shfl_xor(corr, 16);
                corr += __shfl_xor(corr, 32);
                double pa[4] = {0.0, 0.0, 0.0, 0.0};
                const double* bcol = Tb + g * CW + (l & 15);
                for (int ct = 0; ct < CT; ++ct) {
                    d4 Y = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
                    for (int kk = 0; kk < KF; ++kk) {
                        if (kk > KF - 4 && 4 * kk >= N) continue;  // padding
                        Y = __builtin_amdgcn_mfma_f64_16x16x4f64(Af[kk], bcol[4 * kk * CW + 16 * ct], Y, 0, 0, 0);
                    }
#pragma unroll
                    for (int r = 0; r < 4; ++r) pa[r] += Y[r] * Y[r];
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int b = 16 * w + 4 * r + g;
                    double pd = row_sum(drop ? 0.0 : pa[r]);
                    const double cb = __shfl(corr, 4 * r + g);
                    if (A.method == 0) pd += cb;
                    if ((l & 15) == 0 && b < N) {
                        A.save_di[((size_t)slot * N + b) * A.ntraj + traj] = pd;
                        // one-hot (iesh.jl:371-375); ehrenfest_na.jl:119-126
                        A.save_ad[((size_t)slot * N + b) * A.ntraj + traj] = A.method == 0 ? (isocc[b] >= 0 ? 1.0 : 0.0) : rs[r];
                    }
                }
            }
            __syncthreads();
        };

        // bead accelerations into bal (one bead at a time over the whole workgroup)
        auto bead_accels = [&]() {
            IE_IDS
            for (int b = 0; b < P; ++b) {
                const Scalars s = bead_eigen(brl[b]);
                const double a = accel(s, Ub);
                if (tid == 0) bal[b] = a;
                __syncthreads();  // Ub and pcol are the next bead's
            }
        };
        // y = H x for the two bead vectors (H: the discrete Hartley transform, orthogonal and its own
        // inverse; modes l and P - l share the frequency, so the Cayley step per Hartley mode is the
        // free ring polymer's), one bead per lane of wavefront 0
        auto hartley2 = [&](const double* x1, const double* x2, double* y1, double* y2) {
            IE_IDS
            if (tid < P) {
                double a1 = 0.0, a2 = 0.0;
                for (int k = 0; k < P; ++k) {
                    double sn, cs;
                    sincospi(2.0 * (double)((tid * k) % P) / (double)P, &sn, &cs);
                    a1 += (cs + sn) * x1[k];
                    a2 += (cs + sn) * x2[k];
                }
                const double sP = 1.0 / sqrt((double)P);
                y1[tid] = a1 * sP;
                y2[tid] = a2 * sP;
            }
            __syncthreads();
        };

        Scalars sc = eigen(x);
        double kacc = 0.0;
        if (rp) bead_accels();
        else kacc = accel(sc, U);
        __syncthreads();  // accel's reads of pcol end here, before save writes it
        save(0);

        for (int64_t step = 0; step < A.nsteps; ++step) {
            if (!rp) {
                // ---- nuclei: B A (update) B (verlet_with_electronics.jl:58-66) ----------------------
                const double vt = v + (dt / 2) * kacc;
                x = x + dt * vt;
                sc = eigen(x);
                kacc = accel(sc, U);  // EhrenfestNA uses psi of the step start
                v = vt + (dt / 2) * kacc;
            } else {
                // ---- ring polymer: B, C in normal modes, B (bcb_wavefunction.jl:46-66); the bead
                // forces see psi of the step start, and the wavefunction step below the centroid
                // eigenpairs and velocity of the step start (E, U, sc, v are not updated here) ---
                if (tid < P) bvl[tid] += (dt / 2) * bal[tid];
                __syncthreads();
                hartley2(brl, bvl, bq, bp);
                if (tid < P) {  // Cayley map of mode tid, half = false (ring_polymer.jl:71-82)
                    const double wk = 2.0 * A.wn * sinpi((double)tid / (double)P);
                    const double uu = dt * dt * wk * wk / 4.0, sc1 = 1.0 / (1.0 + uu);
                    const double c11 = (1.0 - uu) * sc1, c12 = dt * sc1, c21 = -dt * wk * wk * sc1;
                    const double qn = c11 * bq[tid] + c12 * bp[tid], pn = c21 * bq[tid] + c11 * bp[tid];
                    bq[tid] = qn;
                    bp[tid] = pn;
                }
                __syncthreads();
                hartley2(bq, bp, brl, bvl);
                bead_accels();
                if (tid < P) bvl[tid] += (dt / 2) * bal[tid];
                __syncthreads();
            }

            double dtvd;  // dt sum |v_dot_d[m, n]| over unoccupied m and electrons n (iesh.jl:285-298)
            // ---- wavefunction: psi <- exp(-i dt H) psi, H = diag(E) - i v d ---------------------------
            {
            IE_IDS
                const double sW = dt * v * sc.dh;
                const int ia = 16 * w + (l & 15);
                const bool free_row = isocc[ia] < 0;
                const double Ei = E[ia], sU = -sW * U[ia];
                double Af[KF];
                double loc = 0.0, lvd = 0.0;
#pragma unroll
                for (int kk = 0; kk < KF; ++kk) {
                    const int k = 4 * kk + (l >> 4);
                    double val = sU * (U[k] * rcp_nr(E[k] - Ei));
                    if (ia >= N || k >= N || ia == k) val = 0.0;
                    Af[kk] = val;
                    loc += val * val;
                    if (!RPB && free_row && isocc[k] >= 0) lvd += fabs(val);
                }
                loc = wave_sum(loc);
                if (!RPB) lvd = wave_sum(lvd);
                if (l == 0) {
                    part[w] = loc;
                    part[8 + w] = lvd;
                }
                __syncthreads();
                loc = part[0];
                dtvd = part[8];
#pragma unroll
                for (int j = 1; j < NT; ++j) {
                    loc += part[j];
                    dtvd += part[8 + j];
                }
                // ||dt H||_2 <= dt max|E_i| + ||dt v d||_F; the energies ascend
                const double theta = dt * fmax(fabs(E[0]), fabs(E[N - 1])) + sqrt(loc);
                // Sub-steps of norm <= 0.5, at most 1024 of them; a non-finite bound leaves psi as is.
                const bool finite = theta <= 512.0;
                const int ns = (finite && theta > 0.5) ? __builtin_amdgcn_readfirstlane((int)ceil(theta / 0.5)) : 1;
                const double inv_ns = 1.0 / ns;
                const double ths = finite ? theta * inv_ns : 0.0;
                const int K = (int)__popcll(__ballot((float)ths > order_from));
                if (ns > 1) {
#pragma unroll
                    for (int kk = 0; kk < KF; ++kk) Af[kk] *= inv_ns;
                }
                double dg[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int ir = 16 * w + 4 * r + (l >> 4);
                    // the sign of the Re / Im column this lane holds goes with it
                    dg[r] = (ir < N) ? ((l & 1) ? -dt : dt) * E[ir] * inv_ns : 0.0;
                }
                d4 P[CTM];
                const int own = (16 * w + (l >> 4)) * CW + (l & 15);
#pragma unroll
                for (int ct = 0; ct < CTM; ++ct) {
                    P[ct] = d4{0.0, 0.0, 0.0, 0.0};
                    if (ct < CT) {
#pragma unroll
                        for (int r = 0; r < 4; ++r) P[ct][r] = Tb[own + 4 * r * CW + 16 * ct];
                    }
                }
                // All column tiles of a term are computed, then written back over it: two barriers a term.
                const double* bcol = Tb + (l >> 4) * CW + (l & 15);
                for (int sub = 0; sub < ns && K > 0; ++sub) {
                    for (int k = 1; k <= K; ++k) {
                        const double ik = rcp_nr((double)k);
                        const bool last = (k == K);
                        d4 Y[CTM];
#pragma unroll
                        for (int ct = 0; ct < CTM; ++ct) {
                            if (ct < CT) {
                                Y[ct] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
                                for (int kk = 0; kk < KF; ++kk) {
                                    if (kk > KF - 4 && 4 * kk >= N) continue;  // padding
                                    Y[ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(Af[kk], bcol[4 * kk * CW + 16 * ct], Y[ct], 0, 0, 0);
                                }
#pragma unroll
                                for (int r = 0; r < 4; ++r) {
                                    Y[ct][r] = (Y[ct][r] + dg[r] * Tb[(own ^ 1) + 4 * r * CW + 16 * ct]) * ik;
                                    P[ct][r] += Y[ct][r];
                                }
                            }
                        }
                        __syncthreads();
#pragma unroll
                        for (int ct = 0; ct < CTM; ++ct) {
                            if (ct < CT) {
#pragma unroll
                                for (int r = 0; r < 4; ++r) Tb[own + 4 * r * CW + 16 * ct] = last ? P[ct][r] : Y[ct][r];
                            }
                        }
                        if (sub + 1 < ns || !last) __syncthreads();
                    }
                }
                // the weight of the orbitals outside the occupied states
                double lt2 = 0.0;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    double q = 0.0;
#pragma unroll
                    for (int ct = 0; ct < CTM; ++ct) q += P[ct][r] * P[ct][r];
                    if (isocc[16 * w + 4 * r + (l >> 4)] < 0) lt2 += q;
                }
                lt2 = wave_sum(lt2);
                if (l == 0) part[16 + w] = lt2;
                __syncthreads();
            }

            if (rp) {  // centroid at the step end: eigenpairs and velocity for the hop and the next step
                x = bead_mean(brl);
                v = bead_mean(bvl);
                sc = eigen(x);
            }

            // the save precedes the hop and decoherence callbacks (a save time holds the state before the
            // step's callbacks: DiffEqBase saves the due saveat points before affect!)
            if (A.save_every > 0 && (step + 1) % A.save_every == 0) save((int)((step + 1) / A.save_every));

            // ---- IESH hop (iesh.jl:390-407) -------------------------------------------------------------
            if (A.method == 0) {
            IE_IDS
                const double rnd = philox_uniform((uint64_t)traj, (uint32_t)step, STREAM_HOP, A.key);
                const int Nu = N - Ne;
                // t2 = ||psi[unoccupied, :]||_F^2, the weight of the orbitals outside the occupied rows; a ring
                // polymer's eigenpairs and velocity are those of the step end
                double t2 = part[16];
#pragma unroll
                for (int j = 1; j < NT; ++j) t2 += part[16 + j];
                if (RPB) {
                    double lvd = 0.0;
                    for (int k = tid; k < N * Ne; k += B) {
                        const int m = k / Ne, n = k - m * Ne;
                        if (isocc[m] < 0) {
                            const int o = occ[n];
                            lvd += fabs(v * (sc.dh * (U[m] * U[o] / (E[o] - E[m]))));
                        }
                    }
                    lvd = wave_sum(lvd);
                    if (l == 0) part[24 + w] = lvd;
                    __syncthreads();
                    dtvd = part[24];
#pragma unroll
                    for (int j = 1; j < NT; ++j) dtvd += part[24 + j];
                    dtvd *= dt;
                }
                // The estimate 2 dtvd (|Re det S| + |Im det S|) / |det S|^2 (iesh.jl:250-253) is at
                // most 2 dtvd sqrt(2) / |det S|, and for orthonormal orbitals (S^H S + T^H T = I,
                // T = psi[unoccupied, :]) |det S|^2 = prod(1 - s_i^2(T)) >= 1 - t2.  Where that bound
                // is already below the uniform, the reference's estimate is too: no hop, and the LU is
                // skipped (1e-6 absorbs the orbitals' rounding-level loss of orthonormality; 1e-8 and
                // the 1e-4 floor, which bounds cond(S) by 100, absorb the rounding of the estimate).
                bool skip = false;
                if (det_bound) {
                    const double L2 = 1.0 - t2 - 1e-6;
                    skip = L2 > 1e-4 && 2.0 * dtvd * 1.4142135623730951 * (1.0 + 1e-8) < rnd * sqrt(L2);
                }
                bool evaluate = false;
                if (!skip) {
                    IE_IDS
                    if (w == 0) {  // unoccupied states in ascending order (DynamicsUtils.jl:162-171)
                        int c = 0;
                        for (int m = l; m - l < N; m += 64) {
                            const uint64_t f = __ballot(m < N && isocc[min(m, N - 1)] < 0);
                            if ((f >> l) & 1) unocc[c + __popcll(f & ((1ull << l) - 1))] = m;
                            c += __popcll(f);
                        }
                    }
                    // S_je = psi[occ_j, e] (iesh.jl:309-316): row j on lane j; det S (FastDeterminant.jl:20-22) and S^-1
                    constexpr int KC = CTM > NT ? 16 : 8;  // columns of a wavefront: 2 Ne <= 16 CTM, Ne <= N <= 16 NT
                    double xr[KC], xi[KC];
                    const double* srow = Tb + occ[min(l, Ne - 1)] * CW;
#pragma unroll
                    for (int j = 0; j < KC; ++j) {
                        const int c = w + NT * j;
                        const bool in = l < Ne && c < Ne;
                        xr[j] = in ? srow[2 * c] : 0.0;
                        xi[j] = in ? srow[2 * c + 1] : 0.0;
                    }
                    double dre, dim;
                    int myp, rot;
                    const bool singular = !block_inverse<NT, KC>(xr, xi, Ne, w, l, part + 32, piv, dre, dim, myp, rot);
                    const double Akk = dre * dre + dim * dim;
                    const double est = 2.0 / Akk * dtvd * (fabs(dre) + fabs(dim));
                    evaluate = !singular && Akk > 0.0 && (!A.estimate || !(est < rnd));
                    if (evaluate && l < Ne) {  // S^-1, interleaved complex, row-major
#pragma unroll
                        for (int j = 0; j < KC; ++j) {
                            const int c = w + NT * ((j + rot) % KC);
                            if (c < Ne) {
                                const int at = 2 * (myp * Ne + piv[c]);
                                Sb[at] = xr[j];
                                Sb[at + 1] = xi[j];
                            }
                        }
                    }
                }
                if (evaluate) {
                    IE_IDS
                    __syncthreads();  // S^-1 and the unoccupied states are in place
                    // P(n -> m) = 2 dt Re((psi_m S^-1)_n) v_dot_d[m, n]: det(S with row n replaced by
                    // psi_m) = det(S) (psi_m S^-1)_n, so Re(det S conj(det S_{n<-m})) / |det S|^2 is that real part.
                    // pass 1: per-electron totals, partial sums over interleaved chunks of unoccupied states
                    const int nch = max(1, min(8, B / Ne));
                    if (tid < Ne * nch) {
                        const int n = tid % Ne, ch = tid / Ne;
                        const int o = occ[n];
                        double part_sum = 0.0;
                        for (int mi = ch; mi < Nu; mi += nch) {
                            const int m = unocc[mi];
                            double zr = 0.0;
                            for (int e = 0; e < Ne; ++e)
                                zr += Tb[m * CW + 2 * e] * Sb[2 * (e * Ne + n)] - Tb[m * CW + 2 * e + 1] * Sb[2 * (e * Ne + n) + 1];
                            const double vd = -v * (sc.dh * (U[m] * U[o] / (E[o] - E[m])));
                            part_sum += fmin(fmax(2.0 * dt * zr * vd, 0.0), 1.0);
                        }
                        part[n * 8 + ch] = part_sum;
                    }
                    __syncthreads();
                    for (int n = tid; n < Ne; n += B) {
                        double sn = 0.0;
                        for (int ch = 0; ch < nch; ++ch) sn += part[n * 8 + ch];
                        pcol[n] = sn;
                    }
                    __syncthreads();
                    if (w == 0) {  // the electron whose cumulative total passes the uniform, if any
                        const double mine = l < Ne ? pcol[l] : 0.0;
                        double cum = 0.0;
                        int hn = -1;
                        for (int n = 0; n < Ne; ++n) {
                            const double pn = readlane_f64(mine, n);
                            if (rnd < cum + pn) { hn = n; break; }
                            cum += pn;
                        }
                        if (l == 0) {
                            scal[3] = (double)hn;
                            scal[4] = cum;
                        }
                    }
                    __syncthreads();
                    const int hsel = (int)scal[3];
                    if (hsel >= 0) {  // pass 2: that electron's probabilities, in unoccupied order
                        const int o = occ[hsel];
                        for (int mi = tid; mi < Nu; mi += B) {
                            const int m = unocc[mi];
                            double zr = 0.0;
                            for (int e = 0; e < Ne; ++e)
                                zr += Tb[m * CW + 2 * e] * Sb[2 * (e * Ne + hsel)] - Tb[m * CW + 2 * e + 1] * Sb[2 * (e * Ne + hsel) + 1];
                            const double vd = -v * (sc.dh * (U[m] * U[o] / (E[o] - E[m])));
                            part[mi] = fmin(fmax(2.0 * dt * zr * vd, 0.0), 1.0);
                        }
                    }
                    __syncthreads();
                    if (tid == 0) {  // cumulative selection, electrons outer, unoccupied inner (iesh.jl:318-335)
                        int hn = -1, hm = -1;
                        if (hsel >= 0) {
                            double cum = scal[4];
                            for (int mi = 0; mi < Nu; ++mi) {
                                cum += part[mi];
                                if (rnd < cum) { hn = hsel; hm = unocc[mi]; break; }
                            }
                        }
                        scal[5] = v;
                        scal[6] = 0.0;
                        if (hn >= 0) {  // rescale along d[new, old] (surface_hopping.jl:65-92)
                            const int old = occ[hn];
                            bool ok = true;
                            double vn = v;
                            if (A.rescaling != NQCD_RESCALE_OFF) {
                                const double dd = sc.dh * (U[hm] * U[old] / (E[old] - E[hm]));
                                const double aq = dd * dd / A.mass / 2.0, bq = dd * v, cq = E[hm] - E[old];
                                const double disc = bq * bq - 4.0 * aq * cq;
                                if (disc < 0.0) {
                                    ok = false;
                                    if (A.rescaling == NQCD_RESCALE_VINVERSION) {
                                        const double inc = 2.0 * (v * (dd / fabs(dd))) * (dd / fabs(dd));
                                        vn = v - inc;
                                        scal[6] = -inc;
                                    }
                                } else {
                                    const double root = sqrt(disc);
                                    const double gam = (bq < 0.0) ? (bq + root) / (2.0 * aq) : (bq - root) / (2.0 * aq);
                                    vn = v - gam * dd / A.mass;
                                    scal[6] = -(gam * dd / A.mass);
                                }
                            }
                            if (ok) {
                                isocc[old] = -1;
                                isocc[hm] = hn;
                                occ[hn] = hm;
                                ++nh;
                            }
                            scal[5] = vn;
                        }
                    }
                    __syncthreads();
                    v = scal[5];
                    if (rp) {  // every bead takes the centroid's change (rpsh.jl:24-44)
                        const double inc = scal[6];
                        __syncthreads();
                        if (tid < P) bvl[tid] = bvl[tid] - (-inc);
                        __syncthreads();
                        v = bead_mean(bvl);
                    }
                    __syncthreads();
                }
                // ---- Granucci-Persico EDC per electron (decoherence_corrections.jl:21-39, iesh.jl:424-433)
                if (A.edc) {
                    IE_IDS
                    const double Ekin = 0.5 * A.mass * v * v;
                    if (tid < Ne) {
                        const int s = occ[tid];
                        double nrm = 0.0;
                        for (int a = 0; a < N; ++a) {
                            if (a == s) continue;
                            const double tau = (1.0 + A.edc_C / Ekin) / fabs(E[a] - E[s]);
                            const double f = exp(-dt / tau);
                            const double re = Tb[a * CW + 2 * tid] * f, im = Tb[a * CW + 2 * tid + 1] * f;
                            Tb[a * CW + 2 * tid] = re;
                            Tb[a * CW + 2 * tid + 1] = im;
                            nrm += re * re + im * im;
                        }
                        const double cr = Tb[s * CW + 2 * tid], ci = Tb[s * CW + 2 * tid + 1];
                        const double fac = sqrt((1.0 - nrm) / (cr * cr + ci * ci));
                        Tb[s * CW + 2 * tid] = cr * fac;
                        Tb[s * CW + 2 * tid + 1] = ci * fac;
                    }
                    __syncthreads();
                }
            }
        }

        // ---- store --------------------------------------------------------------------------------
        if (rp) {
            if (tid < P) {
                A.r[(size_t)traj * P + tid] = brl[tid];
                A.v[(size_t)traj * P + tid] = bvl[tid];
            }
        } else if (tid == 0) {
            A.r[traj] = x;
            A.v[traj] = v;
        }
        if (tid == 0) {
            A.nhops[traj] = nh;
            A.steps[traj] = (int32_t)A.nsteps;
        }
        if (tid < Ne) A.occ[(size_t)traj * Ne + tid] = occ[tid];
        for (int idx = tid; idx < N * 2 * Ne; idx += B) {
            const int row = idx / (2 * Ne), col = idx - row * 2 * Ne;
            A.psi[(size_t)traj * N * 2 * Ne + idx] = Tb[row * CW + col];
        }
    }
}

// Determinants of nmat complex Ne x Ne matrices (re, im planes, row-major) by block_inverse, one
// workgroup per matrix: the test hook of the IESH estimate's determinant.
__global__ __launch_bounds__(256) void det_kernel(const double* __restrict__ re, const double* __restrict__ im, int Ne,
                                                  double* __restrict__ out) {
    __shared__ double buf[2 * 136];
    __shared__ int piv[kIeMaxNe];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63;
    const size_t base = (size_t)blockIdx.x * Ne * Ne;
    double xr[16], xi[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const int c = w + 4 * j;
        const bool in = l < Ne && c < Ne;
        xr[j] = in ? re[base + (size_t)l * Ne + c] : 0.0;
        xi[j] = in ? im[base + (size_t)l * Ne + c] : 0.0;
    }
    double dr, di;
    int myp, rot;
    const bool ok = block_inverse<4, 16>(xr, xi, Ne, w, l, buf, piv, dr, di, myp, rot);
    if (threadIdx.x == 0) {
        out[3 * blockIdx.x] = dr;
        out[3 * blockIdx.x + 1] = di;
        out[3 * blockIdx.x + 2] = ok ? 1.0 : 0.0;
    }
}

// The energies the Fermi-Dirac occupation chain weighs, at each trajectory's initial position: the
// adiabatic energies (iesh.jl:113-114), or for the diabatic basis the diagonal of the model matrix,
// [h(x0), eps_0, ..., eps_{M-1}] (iesh.jl:150-153), followed then by the adiabatic energies E_b and
// the impurity components u_b of the eigenvectors (row stride 3N; N for the adiabatic basis).  One
// wavefront per trajectory, root ir on lane ir % 64.
__global__ __launch_bounds__(256) void ie_initial_energies(const IeshArgs A, int diabatic, double* __restrict__ W) {
    __shared__ double eps[kIeMaxStates];
    for (int k = threadIdx.x; k < kIeMaxStates; k += blockDim.x) eps[k] = k < A.M ? A.a + k * A.de : kFarPole;
    __syncthreads();
    const int64_t traj = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (traj >= A.ntraj) return;
    double x0 = A.r0[traj];
    if (A.P > 1) {  // the centroid (the hopping eigenvalues of a ring polymer, SurfaceHoppingMethods.jl:85-87)
        x0 = 0.0;
        for (int b = 0; b < A.P; ++b) x0 += A.r0[(size_t)traj * A.P + b];
        x0 /= A.P;
    }
    const Scalars s = na_scalars(A, x0);
    const double zn = sqrt((double)A.M) * A.V;
    double* row = W + traj * (diabatic ? 3 * A.N : A.N);
    for (int ir = threadIdx.x & 63; ir < A.N; ir += 64) {
        double fp;
        const double lam = na_root(eps, A.M, A.a, A.V * A.V, zn, s.h, ir, false, 0.0, 0.0, fp);
        if (diabatic) {
            row[ir] = (ir == 0) ? s.h : eps[ir - 1];
            row[A.N + ir] = lam;
            row[2 * A.N + ir] = 1.0 / sqrt(fp);
        } else {
            row[ir] = lam;
        }
    }
}

// Position of the k-th set bit (k < popcount) of a 64-bit word.
__device__ __forceinline__ int select_bit64(uint64_t w, int k) {
    int pos = 0;
#pragma unroll
    for (int sh = 32; sh > 0; sh >>= 1) {
        const int c = __popcll(w & ((1ull << sh) - 1));
        if (k >= c) { k -= c; w >>= sh; pos += sh; }
    }
    return pos;
}

// Fermi-Dirac occupations by the Boltzmann-factor Metropolis chain of
// sample_fermi_dirac_distribution (DynamicsUtils.jl:191-205), one lane per trajectory: start from
// the n_e lowest available states, then n_avail * n_e moves; move `it` draws Philox counter (traj,
// it, STREAM_OCCUPATION) = (o0, o1, o2, o3), takes the occupied slot (o0 n_e) >> 32 of the state
// array and the unoccupied available state number (o1 n_free) >> 32 in ascending order, and
// accepts when exp(-beta (E_j - E_i)) > u53(o2, o3) (beta = inf: when E_j < E_i).  The slot array
// lives in LDS ([slot][lane]); the occupied set is a 128-bit mask, so the sorted result is its set
// bits in order.
__global__ __launch_bounds__(256) void ie_fermi_dirac_chain(int64_t ntraj, int N, int Ne, uint64_t avail_lo,
                                                            uint64_t avail_hi, double beta, uint64_t key,
                                                            const double* __restrict__ E0, int stride,
                                                            int32_t* __restrict__ occ0) {
    extern __shared__ int slots[];  // Ne x blockDim.x
    const int tid = threadIdx.x, B = blockDim.x;
    const int64_t traj = (int64_t)blockIdx.x * B + tid;
    if (traj >= ntraj) return;
    const int navail = __popcll(avail_lo) + __popcll(avail_hi), nfree = navail - Ne;
    const double* E = E0 + traj * stride;
    uint64_t occ_lo = 0, occ_hi = 0;
    for (int e = 0; e < Ne; ++e) {  // the first Ne available states
        const uint64_t flo = avail_lo & ~occ_lo, fhi = avail_hi & ~occ_hi;
        const int st = flo ? __ffsll((unsigned long long)flo) - 1 : 64 + __ffsll((unsigned long long)fhi) - 1;
        slots[e * B + tid] = st;
        if (st < 64) occ_lo |= 1ull << st; else occ_hi |= 1ull << (st - 64);
    }
    const bool cold = isinf(beta);
    const int64_t nmoves = (int64_t)navail * Ne;
    for (int64_t it = 0; it < nmoves; ++it) {
        uint32_t c0 = (uint32_t)traj, c1 = (uint32_t)(traj >> 32), c2 = (uint32_t)it, c3 = STREAM_OCCUPATION;
        philox4x32_10(c0, c1, c2, c3, (uint32_t)key, (uint32_t)(key >> 32));
        const int ci = (int)(((uint64_t)c0 * (uint64_t)Ne) >> 32);
        const int kk = (int)(((uint64_t)c1 * (uint64_t)nfree) >> 32);
        const uint64_t flo = avail_lo & ~occ_lo, fhi = avail_hi & ~occ_hi;
        const int nlo = __popcll(flo);
        const int j = kk < nlo ? select_bit64(flo, kk) : 64 + select_bit64(fhi, kk - nlo);
        const int i = slots[ci * B + tid];
        const double dE = E[j] - E[i];
        const bool accept = cold ? (dE < 0.0) : (exp(-beta * dE) > u53(c2, c3));
        if (accept) {
            slots[ci * B + tid] = j;
            if (i < 64) occ_lo &= ~(1ull << i); else occ_hi &= ~(1ull << (i - 64));
            if (j < 64) occ_lo |= 1ull << j; else occ_hi |= 1ull << (j - 64);
        }
    }
    int e = 0;
    for (uint64_t w = occ_lo; w; w &= w - 1) occ0[traj * Ne + e++] = __ffsll((unsigned long long)w) - 1;
    for (uint64_t w = occ_hi; w; w &= w - 1) occ0[traj * Ne + e++] = 64 + __ffsll((unsigned long long)w) - 1;
}

// Diabatic Fermi-Dirac occupations to IESH orbitals (iesh.jl:159-182), one lane per trajectory:
// for each sampled diabatic state d (ascending), an adiabatic state is drawn with weights U_db^2
// (U_db = component d of eigenvector b: u_b for the impurity, V u_b / (E_b - eps_{d-1}) for a bath
// level) until one not yet taken comes up -- StatsBase's sample(Weights(w)): t = rand() * sum(w), the
// first b whose running sum reaches t -- and the electron's orbital is row d of U times the sign of
// U_d0, psi_b = U_db U_d0 / sqrt(U_d0^2) (real).  Draw k of a trajectory is Philox counter
// (traj, 2^31 + k, STREAM_OCCUPATION), u = u53(o0, o1).  The orbitals stay in sampling order and
// the occupations are sorted, as the reference leaves them.  A trajectory that needs more than
// 4096 draws for one electron (free states of vanishing weight) gets occupation -1.
__global__ __launch_bounds__(256) void ie_diabatic_orbitals(int64_t ntraj, int N, int Ne, double V, double a, double de,
                                                            uint64_t key, const double* __restrict__ W,
                                                            const int32_t* __restrict__ dstate,
                                                            int32_t* __restrict__ occ0, double* __restrict__ psi0) {
    const int64_t traj = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (traj >= ntraj) return;
    const double* E = W + traj * 3 * N + N;
    const double* u = E + N;
    uint64_t tk_lo = 0, tk_hi = 0;
    uint32_t draw = 0;
    bool failed = false;
    for (int i = 0; i < Ne && !failed; ++i) {
        const int d = dstate[traj * Ne + i];
        const double ed = (d == 0) ? 0.0 : a + (d - 1) * de;
        auto Ud = [&](int b) { return (d == 0) ? u[b] : V * u[b] / (E[b] - ed); };
        double sw = 0.0;
        for (int b = 0; b < N; ++b) { const double x = Ud(b); sw += x * x; }
        int pick = -1;
        for (int tries = 0; tries < 4096 && pick < 0; ++tries) {
            uint32_t c0 = (uint32_t)traj, c1 = (uint32_t)(traj >> 32), c2 = 0x80000000u + draw++, c3 = STREAM_OCCUPATION;
            philox4x32_10(c0, c1, c2, c3, (uint32_t)key, (uint32_t)(key >> 32));
            const double t = u53(c0, c1) * sw;
            int k = 0;
            double x = Ud(0), cw = x * x;
            while (cw < t && k < N - 1) {
                ++k;
                x = Ud(k);
                cw += x * x;
            }
            const bool taken = (k < 64) ? (tk_lo >> k) & 1 : (tk_hi >> (k - 64)) & 1;
            if (!taken) pick = k;
        }
        if (pick < 0) { failed = true; break; }
        if (pick < 64) tk_lo |= 1ull << pick; else tk_hi |= 1ull << (pick - 64);
        const double u0 = Ud(0), nrm = sqrt(u0 * u0);
        for (int b = 0; b < N; ++b) {
            double* p = psi0 + (((size_t)traj * N + b) * Ne + i) * 2;
            p[0] = (Ud(b) * u0) / nrm;
            p[1] = 0.0;
        }
    }
    if (failed) {
        for (int e = 0; e < Ne; ++e) occ0[traj * Ne + e] = -1;
        return;
    }
    int e = 0;
    for (uint64_t w = tk_lo; w; w &= w - 1) occ0[traj * Ne + e++] = __ffsll((unsigned long long)w) - 1;
    for (uint64_t w = tk_hi; w; w &= w - 1) occ0[traj * Ne + e++] = 64 + __ffsll((unsigned long long)w) - 1;
}

// S^-1, interleaved complex; an odd number of rows is reserved, the size that the limit on problems is stated for
int ie_sb_len(int Ne) { return 2 * Ne * (Ne | 1); }

size_t ie_lds_bytes(int NT, int cw, int N, int Ne, int P) {
    const int NP = 16 * NT;
    return sizeof(double) * ((size_t)NP * cw + ie_sb_len(Ne) + 3 * NP + 8 + std::max(NP, 2 * kIeMaxNe) + 8 * kIeMaxNe + 8) +
           sizeof(int) * (2 * kIeMaxNe + 2 * NP) + (P > 1 ? sizeof(double) * (5 * 64 + 2 * (size_t)NP) : 0);
}

typedef void (*IeKernel)(const IeshArgs);

IeKernel ie_pick(int NT, bool wide, bool rp) {
#define NQCD_IE(nt)                                                                                    \
    case nt:                                                                                           \
        if (rp) return wide ? (IeKernel)iesh_kernel<nt, 8, true> : (IeKernel)iesh_kernel<nt, nt, true>; \
        return wide ? (IeKernel)iesh_kernel<nt, 8, false> : (IeKernel)iesh_kernel<nt, nt, false>;
    switch (NT) {
        NQCD_IE(1) NQCD_IE(2) NQCD_IE(3) NQCD_IE(4) NQCD_IE(5) NQCD_IE(6) NQCD_IE(7) NQCD_IE(8)
    default: return nullptr;
    }
#undef NQCD_IE
}

// Model parameters in the handle's slot 0: m, omega, g, dG, Gamma, a, b, M.
struct IeModel { double mw2, g, dG, V, a, de; int M; };

IeModel ie_model(const nqcd_handle_t* h) {
    const double* p = h->models[0].p;
    IeModel m;
    m.M = (int)p[7];
    m.mw2 = p[0] * p[1] * p[1];
    m.g = p[2];
    m.dG = p[3];
    m.a = p[5];
    m.de = (p[6] - p[5]) / (m.M - 1);
    m.V = std::sqrt(p[4] / (2.0 * M_PI)) * std::sqrt(m.de);
    return m;
}

}  // namespace

int32_t ie_check_problem(nqcd_handle_t* h) {
    const nqcd_problem_desc& d = h->prob;
    if (d.nbeads <= 1 && d.algorithm != NQCD_ALG_VERLET_ELECTRONICS)
        return fail(h, NQCD_ERR_UNSUPPORTED, "IESH / EhrenfestNA integrate with VerletwithElectronics");
    if (d.nbeads > 1 && d.algorithm != NQCD_ALG_BCB_WAVEFUNCTION)
        return fail(h, NQCD_ERR_UNSUPPORTED, "ring-polymer IESH / EhrenfestNA integrate with BCBWavefunction");
    if (d.ndofs * d.natoms != 1)
        return fail(h, NQCD_ERR_UNSUPPORTED, "IESH / EhrenfestNA: one degree of freedom");
    if (d.nbeads > 64) return fail(h, NQCD_ERR_UNSUPPORTED, "ring-polymer IESH / EhrenfestNA: at most 64 beads");
    if (d.nbeads > 1 && !(d.temperature > 0.0))
        return fail(h, NQCD_ERR_ARG, "ring polymers need a positive temperature");
    if (d.nbeads > 1 && d.decoherence != NQCD_DECOHERENCE_NONE)
        return fail(h, NQCD_ERR_UNSUPPORTED, "the EDC decoherence correction is not defined for ring polymers");
    if (d.n_states < 3 || d.n_states > kIeMaxStates)
        return fail(h, NQCD_ERR_UNSUPPORTED, "IESH / EhrenfestNA: n_states must be in 3..128");
    if (d.n_electrons < 1 || d.n_electrons >= d.n_states || d.n_electrons > kIeMaxNe)
        return fail(h, NQCD_ERR_ARG, "n_electrons must be in 1..min(64, n_states - 1)");
    if (d.precision != NQCD_PREC_FP64) return fail(h, NQCD_ERR_UNSUPPORTED, "IESH / EhrenfestNA run in FP64");
    if (d.decoherence < 0 || d.decoherence > 1) return fail(h, NQCD_ERR_ARG, "unknown decoherence correction");
    if (d.decoherence == NQCD_DECOHERENCE_EDC && d.method != NQCD_METHOD_IESH)
        return fail(h, NQCD_ERR_UNSUPPORTED, "the EDC decoherence correction applies to IESH");
    return NQCD_OK;
}

int32_t ie_set_model(nqcd_handle_t* h, int32_t slot, const double* p, int64_t n) {
    if (slot != 0) return fail(h, NQCD_ERR_UNSUPPORTED, "the Newns-Anderson model must use slot 0");
    if (n != 8) return fail(h, NQCD_ERR_ARG, "Newns-Anderson params: m, omega, g, dG, Gamma, a, b, M");
    const double M = p[7];
    if (!(M >= 2 && M == std::floor(M) && M + 1 <= kIeMaxStates))
        return fail(h, NQCD_ERR_ARG, "Newns-Anderson: M must be an integer in 2..127");
    if (!(p[4] > 0.0)) return fail(h, NQCD_ERR_ARG, "Newns-Anderson: Gamma must be positive");
    if (!(p[6] > p[5])) return fail(h, NQCD_ERR_ARG, "Newns-Anderson: the band needs b > a");
    if (!(p[0] > 0.0)) return fail(h, NQCD_ERR_ARG, "Newns-Anderson: m must be positive");
    ModelSlot m{};
    m.kind = NQCD_MODEL_NEWNS_ANDERSON;
    for (int i = 0; i < 8; ++i) m.p[i] = p[i];
    h->models[0] = m;
    h->model_set[0] = true;
    return NQCD_OK;
}

static int32_t ie_check_occ(nqcd_handle_t* h, int64_t ntraj, const int32_t* occ) {
    const int N = h->prob.n_states, Ne = h->prob.n_electrons;
    std::vector<char> seen(N);
    for (int64_t i = 0; i < ntraj; ++i) {
        std::fill(seen.begin(), seen.end(), 0);
        for (int e = 0; e < Ne; ++e) {
            const int32_t s = occ[(size_t)i * Ne + e];
            if (s < 0 || s >= N) return fail(h, NQCD_ERR_ARG, "occupied state out of range");
            if (seen[s]) return fail(h, NQCD_ERR_ARG, "an adiabatic state is occupied twice");
            seen[s] = 1;
        }
    }
    return NQCD_OK;
}

int32_t ie_load_initial(nqcd_handle_t* h, int64_t ntraj, const double* r, const double* v, const double* psi_re,
                        const double* psi_im, const int32_t* occ) {
    const int N = h->prob.n_states, Ne = h->prob.n_electrons;
    if (!occ) return fail(h, NQCD_ERR_ARG, "IESH / EhrenfestNA need the occupied states (n_electrons per trajectory)");
    if ((psi_re == nullptr) != (psi_im == nullptr)) return fail(h, NQCD_ERR_ARG, "give both psi parts or neither");
    if (int32_t rc = ie_check_occ(h, ntraj, occ)) return rc;
    h->ntraj = ntraj;
    const int P = h->prob.nbeads > 1 ? h->prob.nbeads : 1;  // (nbeads, ntraj) column-major for ring polymers
    HIPCHK(h, h->r0.ensure(sizeof(double) * P * ntraj));
    HIPCHK(h, h->v0.ensure(sizeof(double) * P * ntraj));
    HIPCHK(h, h->state0.ensure(sizeof(int32_t) * Ne * ntraj));
    HIPCHK(h, hipMemcpy(h->r0.p, r, sizeof(double) * P * ntraj, hipMemcpyHostToDevice));
    HIPCHK(h, hipMemcpy(h->v0.p, v, sizeof(double) * P * ntraj, hipMemcpyHostToDevice));
    HIPCHK(h, hipMemcpy(h->state0.p, occ, sizeof(int32_t) * Ne * ntraj, hipMemcpyHostToDevice));
    h->ie_psi_given = psi_re != nullptr;
    if (psi_re) {  // (N, Ne, ntraj) column-major -> per trajectory rows of (Re, Im) pairs
        std::vector<double> t((size_t)2 * N * Ne * ntraj);
        for (int64_t i = 0; i < ntraj; ++i)
            for (int a = 0; a < N; ++a)
                for (int e = 0; e < Ne; ++e) {
                    const size_t src = ((size_t)i * Ne + e) * N + a;
                    const size_t dst = (((size_t)i * N + a) * Ne + e) * 2;
                    t[dst] = psi_re[src];
                    t[dst + 1] = psi_im[src];
                }
        HIPCHK(h, h->sig0.ensure(sizeof(double) * t.size()));
        HIPCHK(h, hipMemcpy(h->sig0.p, t.data(), sizeof(double) * t.size(), hipMemcpyHostToDevice));
    }
    return NQCD_OK;
}

int32_t ie_sample_initial(nqcd_handle_t* h, const nqcd_sampler_desc* S, uint64_t seed) {
    if (h->prob.nbeads > 1)
        return fail(h, NQCD_ERR_UNSUPPORTED, "ring-polymer IESH / EhrenfestNA take their beads from nqcd_mi355x_load_initial");
    if (S->kind != NQCD_SAMPLER_GAUSSIAN || S->nparams != 4 || !S->params)
        return fail(h, NQCD_ERR_ARG, "IESH / EhrenfestNA sampler: GAUSSIAN with mu_r, sd_r, mu_v, sd_v");
    const int Ne = h->prob.n_electrons;
    const int64_t n = S->ntraj;
    h->ntraj = n;
    HIPCHK(h, h->r0.ensure(sizeof(double) * n));
    HIPCHK(h, h->v0.ensure(sizeof(double) * n));
    HIPCHK(h, h->small.ensure(sizeof(double) * 4));
    HIPCHK(h, hipMemcpy(h->small.p, S->params, sizeof(double) * 4, hipMemcpyHostToDevice));
    HIPCHK(h, launch_sample_gaussian(n, 1, h->small.as<double>(), seed, h->r0.as<double>(), h->v0.as<double>(), h->stream));
    // lowest n_electrons adiabatic states occupied: the zero-temperature limit of the
    // Fermi-Dirac occupation sampling (DynamicsUtils.jl:176-208)
    std::vector<int32_t> occ((size_t)Ne * n);
    for (int64_t i = 0; i < n; ++i)
        for (int e = 0; e < Ne; ++e) occ[(size_t)i * Ne + e] = e;
    HIPCHK(h, h->state0.ensure(sizeof(int32_t) * occ.size()));
    HIPCHK(h, hipMemcpyAsync(h->state0.p, occ.data(), sizeof(int32_t) * occ.size(), hipMemcpyHostToDevice, h->stream));
    HIPCHK(h, hipStreamSynchronize(h->stream));
    h->ie_psi_given = false;
    return NQCD_OK;
}

int32_t ie_sample_fermi_dirac(nqcd_handle_t* h, double beta, const int32_t* avail, int32_t navail, int32_t basis,
                              uint64_t seed) {
    if (!h->have_initial || h->ntraj < 1)
        return fail(h, NQCD_ERR_STATE, "load or sample the nuclear initial conditions first");
    if (!h->model_set[0] || h->models[0].kind != NQCD_MODEL_NEWNS_ANDERSON)
        return fail(h, NQCD_ERR_STATE, "Fermi-Dirac occupations need the Newns-Anderson model in slot 0");
    if (!(beta >= 0.0)) return fail(h, NQCD_ERR_ARG, "beta must be >= 0 (inf for zero temperature)");
    if (basis != 0 && basis != 1) return fail(h, NQCD_ERR_ARG, "basis must be 0 (adiabatic) or 1 (diabatic)");
    if (basis == 1 && h->prob.method != NQCD_METHOD_IESH)
        return fail(h, NQCD_ERR_UNSUPPORTED, "diabatic Fermi-Dirac occupations are defined for IESH (iesh.jl:138)");
    const IeModel md = ie_model(h);
    const int N = h->prob.n_states, Ne = h->prob.n_electrons;
    if (md.M + 1 != N) return fail(h, NQCD_ERR_ARG, "n_states must equal M + 1 for the Newns-Anderson model");
    if (N > kIeMaxStates) return fail(h, NQCD_ERR_UNSUPPORTED, "Fermi-Dirac occupations support up to 128 states");
    uint64_t am[2] = {0, 0};
    if (!avail) {
        for (int s = 0; s < N; ++s) am[s >> 6] |= 1ull << (s & 63);
    } else {
        for (int32_t k = 0; k < navail; ++k) {
            const int s = avail[k];
            if (s < 0 || s >= N) return fail(h, NQCD_ERR_ARG, "available state out of range");
            if (am[s >> 6] >> (s & 63) & 1) return fail(h, NQCD_ERR_ARG, "available states repeat");
            am[s >> 6] |= 1ull << (s & 63);
        }
    }
    const int na = __builtin_popcountll(am[0]) + __builtin_popcountll(am[1]);
    if (na <= Ne) return fail(h, NQCD_ERR_ARG, "need more available states than electrons");
    const int64_t n = h->ntraj;
    IeshArgs A{};
    A.ntraj = n;
    A.N = N; A.M = md.M; A.Ne = Ne;
    A.mw2 = md.mw2; A.g = md.g; A.dG = md.dG; A.V = md.V; A.a = md.a; A.de = md.de;
    A.r0 = h->r0.as<double>();
    A.P = h->prob.nbeads > 1 ? h->prob.nbeads : 1;
    const int stride = basis ? 3 * N : N;
    HIPCHK(h, h->tmp.ensure(sizeof(double) * (size_t)stride * n));
    hipLaunchKernelGGL(ie_initial_energies, dim3((unsigned)((n + 3) / 4)), dim3(256), 0, h->stream, A, basis,
                       h->tmp.as<double>());
    HIPCHK(h, hipGetLastError());
    HIPCHK(h, h->state0.ensure(sizeof(int32_t) * (size_t)Ne * n));
    HIPCHK(h, h->state.ensure(sizeof(int32_t) * (size_t)Ne * n));
    int32_t* chain_out = basis ? h->state.as<int32_t>() : h->state0.as<int32_t>();  // diabatic states: scratch
    const int block = 256;
    hipLaunchKernelGGL(ie_fermi_dirac_chain, dim3((unsigned)((n + block - 1) / block)), dim3(block),
                       sizeof(int) * (size_t)Ne * block, h->stream, n, N, Ne, am[0], am[1], beta, seed,
                       h->tmp.as<double>(), stride, chain_out);
    HIPCHK(h, hipGetLastError());
    if (basis) {
        HIPCHK(h, h->sig0.ensure(sizeof(double) * 2 * (size_t)N * Ne * n));
        hipLaunchKernelGGL(ie_diabatic_orbitals, dim3((unsigned)((n + block - 1) / block)), dim3(block), 0, h->stream,
                           n, N, Ne, md.V, md.a, md.de, seed, h->tmp.as<double>(), h->state.as<int32_t>(),
                           h->state0.as<int32_t>(), h->sig0.as<double>());
        HIPCHK(h, hipGetLastError());
        HIPCHK(h, hipStreamSynchronize(h->stream));
        std::vector<int32_t> occ((size_t)Ne * n);
        HIPCHK(h, hipMemcpy(occ.data(), h->state0.p, sizeof(int32_t) * occ.size(), hipMemcpyDeviceToHost));
        for (int32_t o : occ)
            if (o < 0) return fail(h, NQCD_ERR_ARG, "diabatic Fermi-Dirac occupations: no free adiabatic state of nonzero weight");
        h->ie_psi_given = true;
        return NQCD_OK;
    }
    HIPCHK(h, hipStreamSynchronize(h->stream));
    h->ie_psi_given = false;
    return NQCD_OK;
}

int32_t ie_run(nqcd_handle_t* h, double t0, int64_t nsteps, const nqcd_term_desc* term, uint64_t key) {
    (void)t0;
    if (term && term->kind != NQCD_TERM_NONE)
        return fail(h, NQCD_ERR_UNSUPPORTED, "termination predicates are not supported for IESH / EhrenfestNA");
    if (!h->model_set[0] || h->models[0].kind != NQCD_MODEL_NEWNS_ANDERSON)
        return fail(h, NQCD_ERR_STATE, "IESH / EhrenfestNA need the Newns-Anderson model in slot 0");
    const IeModel md = ie_model(h);
    const int N = h->prob.n_states, Ne = h->prob.n_electrons;
    if (md.M + 1 != N) return fail(h, NQCD_ERR_ARG, "n_states must equal M + 1 for the Newns-Anderson model");
    const int64_t n = h->ntraj;
    const int NT = (N + 15) / 16;
    const int CT = (2 * Ne + 15) / 16;
    const bool wide = CT > NT;
    IeKernel kern = ie_pick(NT, wide, h->prob.nbeads > 1);
    if (!kern) return fail(h, NQCD_ERR_UNSUPPORTED, "n_states");
    const int P = h->prob.nbeads > 1 ? h->prob.nbeads : 1;
    const size_t lds = ie_lds_bytes(NT, 16 * (wide ? 8 : NT), N, Ne, P);
    if (lds > kIeLdsBytes)
        return fail(h, NQCD_ERR_UNSUPPORTED,
                    "IESH / EhrenfestNA with " + std::to_string(N) + " states and " + std::to_string(Ne) +
                        " electrons needs " + std::to_string(lds) + " bytes of LDS per workgroup (" +
                        std::to_string(kIeLdsBytes) + " available)");
    HIPCHK(h, hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    const int block = 64 * NT;
    int bpc = 0;
    HIPCHK(h, hipOccupancyMaxActiveBlocksPerMultiprocessor(&bpc, (const void*)kern, block, lds));
    if (bpc < 1) return fail(h, NQCD_ERR_UNSUPPORTED, "IESH kernel does not fit on a compute unit");
    int64_t grid = (int64_t)bpc * h->cu_count;
    if (grid > n) grid = n;

    HIPCHK(h, h->r.ensure(sizeof(double) * P * n));
    HIPCHK(h, h->v.ensure(sizeof(double) * P * n));
    HIPCHK(h, h->sig.ensure(sizeof(double) * 2 * N * Ne * n));
    HIPCHK(h, h->state.ensure(sizeof(int32_t) * Ne * n));
    HIPCHK(h, h->steps.ensure(sizeof(int32_t) * n));
    HIPCHK(h, h->nhops.ensure(sizeof(int32_t) * n));
    HIPCHK(h, h->save_ad.ensure(sizeof(double) * N * h->nsave * n));
    HIPCHK(h, h->save_di.ensure(sizeof(double) * N * h->nsave * n));
    HIPCHK(h, launch_zero(h->save_ad.p, sizeof(double) * N * h->nsave * n, h->stream));
    HIPCHK(h, launch_zero(h->save_di.p, sizeof(double) * N * h->nsave * n, h->stream));

    IeshArgs A{};
    A.ntraj = n;
    A.nsteps = nsteps;
    A.N = N; A.M = md.M; A.Ne = Ne; A.cw = 16 * CT;
    A.sb_len = ie_sb_len(Ne);
    A.method = (h->prob.method == NQCD_METHOD_IESH) ? 0 : 1;
    A.rescaling = h->prob.rescaling;
    A.estimate = h->prob.disable_estimate ? 0 : 1;
    A.edc = h->prob.decoherence == NQCD_DECOHERENCE_EDC;
    A.save_every = h->save_every;
    A.nsave = h->nsave;
    A.dt = h->prob.dt;
    A.P = P;
    A.wn = P * h->prob.temperature;  // omega_n = P kT (ring_polymer.jl:6-39)
    A.mass = h->masses[0];
    A.edc_C = h->prob.edc_C > 0.0 ? h->prob.edc_C : 0.1;
    A.key = key;
    A.mw2 = md.mw2; A.g = md.g; A.dG = md.dG; A.V = md.V; A.a = md.a; A.de = md.de;
    A.r0 = h->r0.as<double>(); A.v0 = h->v0.as<double>(); A.occ0 = h->state0.as<int32_t>();
    A.psi0 = h->ie_psi_given ? h->sig0.as<double>() : nullptr;
    A.r = h->r.as<double>(); A.v = h->v.as<double>(); A.psi = h->sig.as<double>(); A.occ = h->state.as<int32_t>();
    A.nhops = h->nhops.as<int32_t>(); A.steps = h->steps.as<int32_t>();
    A.save_di = h->save_di.as<double>(); A.save_ad = h->save_ad.as<double>();
    HIPCHK(h, hipEventRecord(h->ev0, h->stream));
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(block), lds, h->stream, A);
    HIPCHK(h, hipGetLastError());
    HIPCHK(h, hipEventRecord(h->ev1, h->stream));
    h->stats.block = block;
    h->stats.grid = (int)grid;
    h->stats.launches = 1;
    return NQCD_OK;
}

int32_t ie_download(nqcd_handle_t* h, int32_t field, void* out, int64_t bytes) {
    const int64_t nt = h->ntraj;
    const int N = h->prob.n_states, Ne = h->prob.n_electrons, ns = h->nsave;
    switch (field) {
    case NQCD_FIELD_R:
    case NQCD_FIELD_V:  // (nbeads, ntraj) for ring polymers
        if (bytes != (int64_t)sizeof(double) * nt * (h->prob.nbeads > 1 ? h->prob.nbeads : 1))
            return fail(h, NQCD_ERR_ARG, "bytes mismatch");
        HIPCHK(h, hipMemcpy(out, field == NQCD_FIELD_R ? h->r.p : h->v.p, bytes, hipMemcpyDeviceToHost));
        return NQCD_OK;
    case NQCD_FIELD_SIGMA_RE:
    case NQCD_FIELD_SIGMA_IM: {  // (N, Ne, ntraj) column-major
        if (bytes != (int64_t)sizeof(double) * N * Ne * nt) return fail(h, NQCD_ERR_ARG, "bytes mismatch");
        std::vector<double> t((size_t)2 * N * Ne * nt);
        HIPCHK(h, hipMemcpy(t.data(), h->sig.p, sizeof(double) * t.size(), hipMemcpyDeviceToHost));
        double* o = static_cast<double*>(out);
        const int c = field == NQCD_FIELD_SIGMA_RE ? 0 : 1;
        for (int64_t i = 0; i < nt; ++i)
            for (int a = 0; a < N; ++a)
                for (int e = 0; e < Ne; ++e) o[((size_t)i * Ne + e) * N + a] = t[(((size_t)i * N + a) * Ne + e) * 2 + c];
        return NQCD_OK;
    }
    case NQCD_FIELD_STATE:
        if (bytes != (int64_t)sizeof(int32_t) * Ne * nt) return fail(h, NQCD_ERR_ARG, "bytes mismatch");
        HIPCHK(h, hipMemcpy(out, h->state.p, bytes, hipMemcpyDeviceToHost));
        return NQCD_OK;
    case NQCD_FIELD_STEPS:
    case NQCD_FIELD_NHOPS:
        if (bytes != (int64_t)sizeof(int32_t) * nt) return fail(h, NQCD_ERR_ARG, "bytes mismatch");
        HIPCHK(h, hipMemcpy(out, field == NQCD_FIELD_STEPS ? h->steps.p : h->nhops.p, bytes, hipMemcpyDeviceToHost));
        return NQCD_OK;
    case NQCD_FIELD_SAVE_POP_AD:
    case NQCD_FIELD_SAVE_POP_DI: {  // (N, nsave, ntraj)
        if (bytes != (int64_t)sizeof(double) * N * ns * nt) return fail(h, NQCD_ERR_ARG, "bytes mismatch");
        return download_rows(h, field == NQCD_FIELD_SAVE_POP_AD ? h->save_ad : h->save_di, 0, N * ns,
                             static_cast<double*>(out));
    }
    default: return fail(h, NQCD_ERR_UNSUPPORTED, "field not available for IESH / EhrenfestNA");
    }
}

int32_t ie_test_det(nqcd_handle_t* h, const double* re, const double* im, int32_t Ne, int32_t nmat, double* out) {
    if (Ne < 1 || Ne > kIeMaxNe) return fail(h, NQCD_ERR_ARG, "1 <= n <= 64 required");
    if (nmat < 1 || nmat > 65536) return fail(h, NQCD_ERR_ARG, "1 <= nmat <= 65536 required");
    HIPCHK(h, hipSetDevice(h->device));
    const size_t n = (size_t)nmat * Ne * Ne;
    DevBuf a, b, o;
    HIPCHK(h, a.ensure(sizeof(double) * n));
    HIPCHK(h, b.ensure(sizeof(double) * n));
    HIPCHK(h, o.ensure(sizeof(double) * 3 * nmat));
    hipError_t e = hipMemcpy(a.p, re, sizeof(double) * n, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(b.p, im, sizeof(double) * n, hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(det_kernel, dim3(nmat), dim3(256), 0, h->stream, a.as<double>(), b.as<double>(), Ne, o.as<double>());
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(out, o.p, sizeof(double) * 3 * nmat, hipMemcpyDeviceToHost);
    a.release(); b.release(); o.release();
    if (e != hipSuccess) return fail(h, NQCD_ERR_DEVICE, std::string("determinant test: ") + hipGetErrorString(e));
    return NQCD_OK;
}

}  // namespace nqcd
