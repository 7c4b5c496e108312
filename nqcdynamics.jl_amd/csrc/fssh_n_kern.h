// fssh_n_kern.h -- device templates of the n-state FSSH / Ehrenfest kernel (fssh_n.hip describes the
// method and the layout); included by the two translation units that instantiate the state counts.
#pragma once
#include "fssh_n.h"

namespace nqcd {

template <class T>
__device__ __forceinline__ const T* ns_opaque(const T* p) {
    asm volatile("" : "+s"(p));
    return p;
}

// index of the upper pair (i, j), i < j, of an NM x NM matrix
template <int NM>
__host__ __device__ constexpr int pidx(int i, int j) {
    return i * NM - i * (i + 1) / 2 + (j - i - 1);
}

template <int NM, typename R>
struct LaneN {
    static constexpr int NP = NM * (NM - 1) / 2;
    R r, v, k;
    double a[NM], x[NP > 0 ? NP : 1], y[NP > 0 ? NP : 1];  // sigma: diagonal, upper real / imaginary parts
    double U[NM * NM];                                     // eigenvectors, row-major, column j = state j
    double Ec[NM], Wc[NP > 0 ? NP : 1];                    // electronic buffer at the step start
    double tc, t;
    const double* tab;                                     // MORSE_N table of the trajectory's model (LDS or global), or null
    ModelRegs m;
    int64_t tid;
    int32_t n, st, nh, step;
};

// Model matrix V (diagonal vd, upper vo) and derivative (dd, dof) of the trajectory's model at x.
template <int NM, typename R>
__device__ __forceinline__ void ns_model(const LaneN<NM, R>& L, R x, double vd[NM], double vo[], double dd[NM],
                                         double dof[]) {
    constexpr int NP = LaneN<NM, R>::NP;
#pragma unroll
    for (int i = 0; i < NM; ++i) { vd[i] = 0.0; dd[i] = 0.0; }
#pragma unroll
    for (int p = 0; p < NP; ++p) { vo[p] = 0.0; dof[p] = 0.0; }
    if (!L.tab) {  // two-state closed-form models (Tully 1/2/3, double well)
        R v11, v22, v12, d11, d22, d12;
        model1d_eval<R>(L.m, x, v11, v22, v12, d11, d22, d12);
        vd[0] = (double)v11; dd[0] = (double)d11;
        if (NM > 1) { vd[1] = (double)v22; dd[1] = (double)d22; vo[0] = (double)v12; dof[0] = (double)d12; }
        return;
    }
    // n-state Morse (Coker and Xiao, J. Chem. Phys. 102, 496 (1995)):
    //   V_ii = D_i (1 - e^{-beta_i (x - r_i)})^2 + c_i,   V_ij = A_ij e^{-a_ij (x - r_ij)^2}
    const double xd = (double)x;
    const double* q = L.tab;
    const int n = L.n;
#pragma unroll
    for (int i = 0; i < NM; ++i) {
        if (i < n) {
            const double Dm = q[4 * i], be = q[4 * i + 1], r0 = q[4 * i + 2], c = q[4 * i + 3];
            const double e = exp(-be * (xd - r0));
            vd[i] = Dm * (1.0 - e) * (1.0 - e) + c;
            dd[i] = 2.0 * Dm * be * e * (1.0 - e);
        }
    }
    // pairs of the n-state table are numbered for n, those of the registers for NM
    int tp = 0;
#pragma unroll
    for (int i = 0; i < NM; ++i)
#pragma unroll
        for (int j = i + 1; j < NM; ++j) {
            if (j < n) {
                const double* c = q + 4 * n + 3 * tp;
                const double u = xd - c[2];
                const double w = c[0] * exp(-c[1] * u * u);
                vo[pidx<NM>(i, j)] = w;
                dof[pidx<NM>(i, j)] = -2.0 * c[1] * u * w;
                ++tp;
            }
        }
}

// Cyclic Jacobi on the leading n x n block of the symmetric matrix (vd, vo): eigenvalues ascending in
// E, eigenvectors in U (columns), signs by the fresh rule or tracked against Uprev (= U on entry).
// warm: the sweeps start from the basis U holds on entry (an orthogonal matrix that is the identity outside
// the leading block, such as the previous step's eigenvectors): A = U^T V U and Q = U, so a basis close to
// the new one needs one or two sweeps to meet the convergence test instead of four or five.  From the
// identity the warm start is the cold one bit for bit (products with exact ones and zeros).
template <int NM>
__device__ __forceinline__ void ns_eigen(int n, const double vd[NM], const double vo[], double E[NM], double U[NM * NM],
                                         bool track, bool warm = false) {
    constexpr int NP = NM * (NM - 1) / 2;
    double A[NM * NM], Q[NM * NM];
#pragma unroll
    for (int i = 0; i < NM; ++i)
#pragma unroll
        for (int j = 0; j < NM; ++j) {
            A[i * NM + j] = (i == j) ? vd[i] : (i < j ? vo[pidx<NM>(i, j)] : vo[pidx<NM>(j, i)]);
            Q[i * NM + j] = warm ? U[i * NM + j] : ((i == j) ? 1.0 : 0.0);
        }
    if (warm) {
        double T[NM * NM];
#pragma unroll
        for (int i = 0; i < NM; ++i)  // T = V U
#pragma unroll
            for (int j = 0; j < NM; ++j) {
                double t = 0.0;
#pragma unroll
                for (int k = 0; k < NM; ++k) t += A[i * NM + k] * U[k * NM + j];
                T[i * NM + j] = t;
            }
#pragma unroll
        for (int i = 0; i < NM; ++i)  // A = U^T T, the upper triangle mirrored
#pragma unroll
            for (int j = i; j < NM; ++j) {
                double t = 0.0;
#pragma unroll
                for (int k = 0; k < NM; ++k) t += U[k * NM + i] * T[k * NM + j];
                A[i * NM + j] = t;
                A[j * NM + i] = t;
            }
    }
    (void)NP;
    for (int sweep = 0; sweep < 100; ++sweep) {
        double off = 0.0, tot = 0.0;
#pragma unroll
        for (int i = 0; i < NM; ++i)
#pragma unroll
            for (int j = 0; j < NM; ++j) {
                const double a2 = (i < n && j < n) ? A[i * NM + j] * A[i * NM + j] : 0.0;
                tot += a2;
                if (i != j) off += a2;
            }
        if (off <= 1e-30 * tot || off == 0.0) break;
#pragma unroll
        for (int p = 0; p < NM - 1; ++p)
#pragma unroll
            for (int q = p + 1; q < NM; ++q) {
                const double apq = A[p * NM + q];
                // t = tan of the rotation angle, the smaller root: 2 a_pq sgn(h) / (|h| + sqrt(h^2 + 4 a_pq^2)),
                // h = a_qq - a_pp.  Square roots and reciprocals by the hardware estimate and Newton steps: a
                // rotation's last bit only moves what the next sweep removes.
                const double h = A[q * NM + q] - A[p * NM + p], t2 = 2.0 * apq, r2 = fma(h, h, t2 * t2);
                if (q < n && apq != 0.0 && r2 > 0.0) {
                    const double t = (h >= 0.0 ? t2 : -t2) * nr_rcp(fabs(h) + r2 * nr_rsq(r2));
                    const double c = nr_rsq(fma(t, t, 1.0)), s = t * c;
                    A[p * NM + p] -= t * apq;   // A <- J^T A J, the pair annihilated
                    A[q * NM + q] += t * apq;
                    A[p * NM + q] = 0.0;
                    A[q * NM + p] = 0.0;
#pragma unroll
                    for (int k = 0; k < NM; ++k) {
                        if (k == p || k == q) continue;
                        const double akp = A[k * NM + p], akq = A[k * NM + q];
                        A[k * NM + p] = A[p * NM + k] = c * akp - s * akq;
                        A[k * NM + q] = A[q * NM + k] = s * akp + c * akq;
                    }
#pragma unroll
                    for (int k = 0; k < NM; ++k) {
                        const double ukp = Q[k * NM + p], ukq = Q[k * NM + q];
                        Q[k * NM + p] = c * ukp - s * ukq;
                        Q[k * NM + q] = s * ukp + c * ukq;
                    }
                }
            }
    }
    if (warm) {
        // one Newton-Schulz step Q <- Q (3 I - Q^T Q) / 2: a basis carried from step to step would otherwise
        // lose orthogonality by rounding, step after step
        double G[NM * NM], Qn[NM * NM];
#pragma unroll
        for (int i = 0; i < NM; ++i)
#pragma unroll
            for (int j = i; j < NM; ++j) {
                double g = 0.0;
#pragma unroll
                for (int k = 0; k < NM; ++k) g += Q[k * NM + i] * Q[k * NM + j];
                G[i * NM + j] = ((i == j) ? 1.5 : 0.0) - 0.5 * g;
                G[j * NM + i] = G[i * NM + j];
            }
#pragma unroll
        for (int i = 0; i < NM; ++i)
#pragma unroll
            for (int j = 0; j < NM; ++j) {
                double t = 0.0;
#pragma unroll
                for (int k = 0; k < NM; ++k) t += Q[i * NM + k] * G[k * NM + j];
                Qn[i * NM + j] = t;
            }
#pragma unroll
        for (int i = 0; i < NM * NM; ++i) Q[i] = Qn[i];
    }
#pragma unroll
    for (int i = 0; i < NM; ++i) E[i] = A[i * NM + i];
    // ascending order over the first n (a stable exchange sort on fixed indices)
#pragma unroll
    for (int pass = 0; pass < NM - 1; ++pass)
#pragma unroll
        for (int j = 0; j < NM - 1 - pass; ++j) {
            if (j + 1 < n && E[j + 1] < E[j]) {
                const double te = E[j]; E[j] = E[j + 1]; E[j + 1] = te;
#pragma unroll
                for (int k = 0; k < NM; ++k) {
                    const double tq = Q[k * NM + j]; Q[k * NM + j] = Q[k * NM + j + 1]; Q[k * NM + j + 1] = tq;
                }
            }
        }
#pragma unroll
    for (int j = 0; j < NM; ++j) {
        double flip;
        if (track) {
            double s = 0.0;
#pragma unroll
            for (int i = 0; i < NM; ++i) s += Q[i * NM + j] * U[i * NM + j];
            flip = (s < 0.0) ? -1.0 : 1.0;
        } else {
            double amax = -1.0, vmax = 0.0;
#pragma unroll
            for (int i = 0; i < NM; ++i) {
                const double av = fabs(Q[i * NM + j]);
                if (i < n && av > amax) { amax = av; vmax = Q[i * NM + j]; }
            }
            flip = (vmax < 0.0) ? -1.0 : 1.0;
        }
#pragma unroll
        for (int i = 0; i < NM; ++i) U[i * NM + j] = flip * Q[i * NM + j];
    }
#pragma unroll
    for (int i = 0; i < NM; ++i) if (i >= n) E[i] = 0.0;
}

// G = U^T dV U (upper triangle with diagonal): Gd[i] = G_ii, Go[p(i,j)] = G_ij.
template <int NM>
__device__ __forceinline__ void ns_rotate(const double U[NM * NM], const double dd[NM], const double dof[], double Gd[NM],
                                          double Go[]) {
    double T[NM * NM];  // T = dV U
#pragma unroll
    for (int a = 0; a < NM; ++a)
#pragma unroll
        for (int j = 0; j < NM; ++j) {
            double s = 0.0;
#pragma unroll
            for (int b = 0; b < NM; ++b) {
                const double dab = (a == b) ? dd[a] : (a < b ? dof[pidx<NM>(a, b)] : dof[pidx<NM>(b, a)]);
                s += dab * U[b * NM + j];
            }
            T[a * NM + j] = s;
        }
#pragma unroll
    for (int i = 0; i < NM; ++i)
#pragma unroll
        for (int j = i; j < NM; ++j) {
            double s = 0.0;
#pragma unroll
            for (int a = 0; a < NM; ++a) s += U[a * NM + i] * T[a * NM + j];
            if (i == j) Gd[i] = s; else Go[pidx<NM>(i, j)] = s;
        }
}

// Right-hand side of the density equation at energies e and couplings W = w (upper, antisymmetric), written out
// for the real diagonal a and the upper elements x + i y of sigma:
//   a_i'  = -2 sum_k W_ik x_ki
//   x_ij' = (e_i - e_j) y_ij - W_ij (a_j - a_i) - sum_{k != i, j} (W_ik x_kj + W_jk x_ki)
//   y_ij' = -(e_i - e_j) x_ij - sum_{k != i, j} (W_ik y_kj - W_jk y_ki)
// ADD: added to ka, kx, ky (every product is then a fused multiply-add), else stored there.
template <int NM, bool ADD>
__device__ __forceinline__ void ns_rhs(const double e[NM], const double w[], const double a[NM], const double x[],
                                       const double y[], double ka[NM], double kx[], double ky[]) {
    auto W = [&](int i, int k) -> double { return i < k ? w[pidx<NM>(i, k)] : -w[pidx<NM>(k, i)]; };
    auto X = [&](int k, int j) -> double { return k < j ? x[pidx<NM>(k, j)] : x[pidx<NM>(j, k)]; };
    auto Y = [&](int k, int j) -> double { return k < j ? y[pidx<NM>(k, j)] : -y[pidx<NM>(j, k)]; };
#pragma unroll
    for (int i = 0; i < NM; ++i) {
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < NM; ++k)
            if (k != i) s = fma(W(i, k), X(i, k), s);
        ka[i] = ADD ? fma(-2.0, s, ka[i]) : -2.0 * s;
    }
#pragma unroll
    for (int i = 0; i < NM; ++i)
#pragma unroll
        for (int j = i + 1; j < NM; ++j) {
            const int p = pidx<NM>(i, j);
            const double de = e[i] - e[j];
            double fx = ADD ? kx[p] : 0.0, fy = ADD ? ky[p] : 0.0;
#pragma unroll
            for (int k = 0; k < NM; ++k) {
                if (k == i || k == j) continue;
                fx = fma(-W(i, k), X(k, j), fma(-W(j, k), X(k, i), fx));
                fy = fma(-W(i, k), Y(k, j), fma(W(j, k), Y(k, i), fy));
            }
            kx[p] = fma(de, y[p], fma(-w[p], a[j] - a[i], fx));
            ky[p] = fma(-de, x[p], fy);
        }
}

// 1 / k!, read with scalar loads by the rolled series
constexpr int kNsMaxOrders = 63;
struct InvFactorials {
    double v[kNsMaxOrders + 1];
};
constexpr InvFactorials ns_inv_factorials() {
    InvFactorials t{};
    long double f = 1.0L;
    for (int k = 0; k <= kNsMaxOrders; ++k) {
        if (k > 1) f *= k;
        t.v[k] = (double)(1.0L / f);
    }
    return t;
}
__constant__ InvFactorials kInvFactorial = ns_inv_factorials();

// The density over a nuclear step as one power series (series_step2 in nqcd_device.h, for the n-state equation):
// over the step the energies and couplings are e + e1 s, w + w1 s for s in [0, 1] (times dt), so the derivatives
// obey u^(k+1) = f(e, w; u^(k)) + k f(e1, w1; u^(k-1)), two right-hand sides an order in place of the 31 and the
// stage sums of five Tsit5 sub-steps.  Orders by z2 = |A0|^2 + 4 |A1| as there, with
// |A| <= spread of the energies + 2 sum |w|.  Bound by FP64 issue; without the stages of five sub-steps the
// three-state FP32 kernel needs 214 registers instead of 256 and runs two wavefronts a SIMD (1e5 three-state Morse
// trajectories x 1000 steps, with the cheaper Jacobi rotations and the tables in LDS: 20.8 -> 8.9 ms).
__device__ __forceinline__ int ns_series_orders(double z2) {
    return z2 > 0.0041 ? (z2 > 0.022 ? (z2 > 0.075 ? (z2 > 0.19 ? (z2 > 0.35 ? (z2 > 0.65 ? 20 : 18) : 16) : 14) : 12) : 10) : 8;
}

// Orders of each of `parts` equal parts of a step whose generator starts at a norm of m - m1 and changes by m1 (z2 >= 4,
// FP32 nuclei; rp = 1 / parts).  A later part starts from what the generator has grown to, so each is taken to start
// from m / parts, and z bounds the norm at its end.  The count leaves less than 1e-10 of the majorant series (computed
// for z from 2 to 12 and every share of m1 in it); at z = 12 its cancellation costs 2e-11.  Few long parts: a unit
// of z takes about three orders where parts of z = 2 take ten (100 steps of 1e5 three-state trajectories, at a norm of 6:
// 3.9 -> 2.0 ms, at 25: 10.2 -> 5.1; five sub-steps: 2.3 ms, off by 7e-4 a step at 6 and unstable at 25).  Beyond a
// norm of 500 to 760, where the 64 parts end, no accuracy is promised.
__device__ __forceinline__ int ns_long_orders(int parts, double rp, double m, double m1) {
    const double z = parts > 1 ? rp * fma(rp, m1, m) : m;
    const double share = (parts > 1 ? rp * rp * m1 : m1) / z;
    return (int)fmin(fma(3.2, z, 14.0) + 11.0 * sqrt(share), (double)kNsMaxOrders);
}

template <int NM>
__device__ __forceinline__ double ns_norm(int n, const double e[NM], const double w[]) {
    constexpr int NP = NM * (NM - 1) / 2;
    double lo = e[0], hi = e[0], sw = 0.0;
#pragma unroll
    for (int i = 1; i < NM; ++i)
        if (i < n) { lo = fmin(lo, e[i]); hi = fmax(hi, e[i]); }
#pragma unroll
    for (int p = 0; p < NP; ++p) sw += fabs(w[p]);
    return fma(2.0, sw, hi - lo);
}

template <int NM>
__device__ __forceinline__ void ns_series(const double e[NM], const double w[], const double e1[NM], const double w1[],
                                          int orders, double a[NM], double x[], double y[]) {
    constexpr int NP = NM * (NM - 1) / 2;
    constexpr int NQ = NP > 0 ? NP : 1;
    double ka[NM], kx[NQ], ky[NQ], pa[NM], px[NQ], py[NQ];   // u^(k) and u^(k-1)
    double ek[NM], wk[NQ];                                     // k times the slopes
#pragma unroll
    for (int i = 0; i < NM; ++i) { ka[i] = a[i]; pa[i] = 0.0; ek[i] = 0.0; }
#pragma unroll
    for (int p = 0; p < NP; ++p) { kx[p] = x[p]; ky[p] = y[p]; px[p] = 0.0; py[p] = 0.0; wk[p] = 0.0; }
#pragma unroll 1
    for (int k = 1; k <= orders; ++k) {
        const double rf = kInvFactorial.v[k];
        double fa[NM], fx[NQ], fy[NQ];
        ns_rhs<NM, false>(ek, wk, pa, px, py, fa, fx, fy);
        ns_rhs<NM, true>(e, w, ka, kx, ky, fa, fx, fy);
#pragma unroll
        for (int i = 0; i < NM; ++i) { pa[i] = ka[i]; ka[i] = fa[i]; a[i] = fma(fa[i], rf, a[i]); ek[i] += e1[i]; }
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            px[p] = kx[p]; kx[p] = fx[p]; x[p] = fma(fx[p], rf, x[p]);
            py[p] = ky[p]; ky[p] = fy[p]; y[p] = fma(fy[p], rf, y[p]);
            wk[p] += w1[p];
        }
    }
}

// One Tsit5 step of size h from tau (electronic_dynamics.jl:104-130 integrated by Tsit5, the stage
// arithmetic of the oracle: u + h (sum a_ij k_j)); the parameters at stage time tau + c h are the
// linear interpolation e = Ec + (En - Ec) loc, loc = (tau - tc) / (tn - tc).
template <int NM>
struct NsInterp {
    static constexpr int NP = NM * (NM - 1) / 2 > 0 ? NM * (NM - 1) / 2 : 1;
    double Ec[NM], En[NM], Wc[NP], Wn[NP];
    double tc, tn;
};

template <int NM>
__device__ __forceinline__ void ns_params(const NsInterp<NM>& I, double tau, double e[NM], double w[]) {
    constexpr int NP = NM * (NM - 1) / 2;
    double loc = (tau - I.tc) / (I.tn - I.tc);
    if (loc != loc) loc = 0.0;
#pragma unroll
    for (int i = 0; i < NM; ++i) e[i] = I.Ec[i] + (I.En[i] - I.Ec[i]) * loc;
#pragma unroll
    for (int p = 0; p < NP; ++p) w[p] = I.Wc[p] + (I.Wn[p] - I.Wc[p]) * loc;
}

template <int NM>
__device__ __forceinline__ void ns_tsit5(const NsInterp<NM>& I, double tau, double h, double a[NM], double x[], double y[]) {
    using namespace ts5;
    constexpr int NP = NM * (NM - 1) / 2;
    constexpr int NQ = NP > 0 ? NP : 1;
    double e[NM], w[NQ];
    double ka[6][NM], kx[6][NQ], ky[6][NQ];
    double ta[NM], tx[NQ], ty[NQ];
    const double cs[6] = {0.0, c1, c2, c3, c4, 1.0};
    const double A[6][5] = {{0, 0, 0, 0, 0},
                            {a21, 0, 0, 0, 0},
                            {a31, a32, 0, 0, 0},
                            {a41, a42, a43, 0, 0},
                            {a51, a52, a53, a54, 0},
                            {a61, a62, a63, a64, a65}};
#pragma unroll
    for (int st = 0; st < 6; ++st) {
#pragma unroll
        for (int i = 0; i < NM; ++i) {
            double s = 0.0;
#pragma unroll
            for (int j = 0; j < st; ++j) s = (j == 0) ? A[st][0] * ka[0][i] : s + A[st][j] * ka[j][i];
            ta[i] = (st == 0) ? a[i] : a[i] + h * s;
        }
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            double sx = 0.0, sy = 0.0;
#pragma unroll
            for (int j = 0; j < st; ++j) {
                sx = (j == 0) ? A[st][0] * kx[0][p] : sx + A[st][j] * kx[j][p];
                sy = (j == 0) ? A[st][0] * ky[0][p] : sy + A[st][j] * ky[j][p];
            }
            tx[p] = (st == 0) ? x[p] : x[p] + h * sx;
            ty[p] = (st == 0) ? y[p] : y[p] + h * sy;
        }
        ns_params<NM>(I, tau + cs[st] * h, e, w);
        ns_rhs<NM, false>(e, w, ta, tx, ty, ka[st], kx[st], ky[st]);
    }
    const double b[6] = {a71, a72, a73, a74, a75, a76};
#pragma unroll
    for (int i = 0; i < NM; ++i) {
        double s = b[0] * ka[0][i];
#pragma unroll
        for (int j = 1; j < 6; ++j) s += b[j] * ka[j][i];
        a[i] = a[i] + h * s;
    }
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        double sx = b[0] * kx[0][p], sy = b[0] * ky[0][p];
#pragma unroll
        for (int j = 1; j < 6; ++j) { sx += b[j] * kx[j][p]; sy += b[j] * ky[j][p]; }
        x[p] = x[p] + h * sx;
        y[p] = y[p] + h * sy;
    }
}

// A: FsshNArgs, or NsHot (its fields in scalar registers)
template <int NM, typename R, class AT>
__device__ __forceinline__ void ns_accel(const AT& A, LaneN<NM, R>& L, const double Gd[NM], const double Go[],
                                         const double* aa, const double* xx) {
    constexpr int NP = LaneN<NM, R>::NP;
    double f;
    if (A.method == 0) {
        f = 0.0;
#pragma unroll
        for (int i = 0; i < NM; ++i) f = (i == L.st) ? Gd[i] : f;
    } else {  // sum_ij Re sigma_ij G_ij
        f = 0.0;
#pragma unroll
        for (int i = 0; i < NM; ++i) f += Gd[i] * aa[i];
#pragma unroll
        for (int p = 0; p < NP; ++p) f += 2.0 * Go[p] * xx[p];
    }
    L.k = (R)(-f * A.inv_mass);
}

template <int NM, typename R>
__device__ __forceinline__ void ns_save(const FsshNArgs* Ap, const LaneN<NM, R>& L, int slot) {
    const FsshNArgs& A = *ns_opaque(Ap);
    if (slot >= A.nsave) return;
    const int64_t nt = A.ntraj;
    double pa[NM];
#pragma unroll
    for (int i = 0; i < NM; ++i) pa[i] = (A.method == 0) ? ((i == L.st) ? 1.0 : 0.0) : L.a[i];
    if (A.save_pop_ad)
#pragma unroll
        for (int i = 0; i < NM; ++i) A.save_pop_ad[((int64_t)slot * NM + i) * nt + L.tid] = pa[i];
    if (A.save_pop_di) {
        // diag(U S U^T), S = Re sigma, with the diagonal replaced by the active state for FSSH
        // (fssh.jl:132-142, ehrenfest.jl:75-83)
#pragma unroll
        for (int i = 0; i < NM; ++i) {
            double p = 0.0;
#pragma unroll
            for (int q = 0; q < NM; ++q) p += L.U[i * NM + q] * L.U[i * NM + q] * pa[q];
#pragma unroll
            for (int q = 0; q < NM; ++q)
#pragma unroll
                for (int r = q + 1; r < NM; ++r) p += 2.0 * L.U[i * NM + q] * L.U[i * NM + r] * L.x[pidx<NM>(q, r)];
            A.save_pop_di[((int64_t)slot * NM + i) * nt + L.tid] = p;
        }
    }
    if (A.save_state) A.save_state[(int64_t)slot * nt + L.tid] = L.st;
}

template <int NM, typename R>
__device__ __forceinline__ void ns_load(const FsshNArgs* Ap, LaneN<NM, R>& L, int64_t tid, const double* tabs) {
    const FsshNArgs& A = *ns_opaque(Ap);
    constexpr int NP = LaneN<NM, R>::NP;
    const int64_t nt = A.ntraj;
    L.tid = tid;
    const int mid = A.model_id ? A.model_id[tid] : 0;
    L.n = A.slot_n[mid];
    L.tab = A.slot_tab[mid] >= 0 ? tabs + A.slot_tab[mid] : nullptr;
    L.m = model_regs(A.models, mid);
    L.r = (R)A.r0[tid];
    L.v = (R)A.v0[tid];
    double vd[NM], vo[NP > 0 ? NP : 1], dd[NM], dof[NP > 0 ? NP : 1], E[NM], Gd[NM], Go[NP > 0 ? NP : 1];
    ns_model<NM, R>(L, L.r, vd, vo, dd, dof);
    ns_eigen<NM>(L.n, vd, vo, E, L.U, false);                     // initialize! (bab_electronics.jl:48-59)
    ns_rotate<NM>(L.U, dd, dof, Gd, Go);
    if (A.init_diabatic >= 0) {  // sigma = U^T e_d e_d^T U (density_matrix_dynamics.jl:37-46,64-75)
        const int d = A.init_diabatic;
#pragma unroll
        for (int i = 0; i < NM; ++i) {
            double ud = 0.0;
#pragma unroll
            for (int q = 0; q < NM; ++q) ud = (q == d) ? L.U[q * NM + i] : ud;
            L.a[i] = ud * ud;
        }
#pragma unroll
        for (int i = 0; i < NM; ++i)
#pragma unroll
            for (int j = i + 1; j < NM; ++j) {
                double ui = 0.0, uj = 0.0;
#pragma unroll
                for (int q = 0; q < NM; ++q) { ui = (q == d) ? L.U[q * NM + i] : ui; uj = (q == d) ? L.U[q * NM + j] : uj; }
                L.x[pidx<NM>(i, j)] = ui * uj;
                L.y[pidx<NM>(i, j)] = 0.0;
            }
    } else {
#pragma unroll
        for (int i = 0; i < NM; ++i) L.a[i] = A.sig0_re[(int64_t)(i + NM * i) * nt + tid];
#pragma unroll
        for (int i = 0; i < NM; ++i)
#pragma unroll
            for (int j = i + 1; j < NM; ++j) {  // sigma_ij = element (i, j) of the column-major (NM, NM) matrix
                L.x[pidx<NM>(i, j)] = A.sig0_re[(int64_t)(i + NM * j) * nt + tid];
                L.y[pidx<NM>(i, j)] = A.sig0_im[(int64_t)(i + NM * j) * nt + tid];
            }
    }
    int st = A.state0 ? A.state0[tid] : -1;
    if (A.method == 0 && st < 0) {  // fssh.jl:54: sample(Weights(diag(real.(sigma))))
        double tot = 0.0;
#pragma unroll
        for (int i = 0; i < NM; ++i) tot += L.a[i];
        const double u = philox_uniform((uint64_t)tid, 0u, STREAM_STATE, A.key) * tot;
        double cum = 0.0;
        st = L.n - 1;
        bool found = false;
#pragma unroll
        for (int i = 0; i < NM; ++i) {
            cum += L.a[i];
            if (!found && i < L.n && u < cum) { st = i; found = true; }
        }
    }
    L.st = st;
    ns_accel<NM, R>(A, L, Gd, Go, L.a, L.x);
#pragma unroll
    for (int i = 0; i < NM; ++i) L.Ec[i] = 0.0;
#pragma unroll
    for (int p = 0; p < NP; ++p) L.Wc[p] = 0.0;
    L.tc = 0.0;  // zero buffers stamped t = 0 (electronic_dynamics.jl:118-127)
    L.t = A.t0;
    L.nh = 0;
    L.step = 0;
    ns_save<NM, R>(Ap, L, 0);
}

template <int NM, typename R>
__device__ __forceinline__ void ns_finish(const FsshNArgs* Ap, const LaneN<NM, R>& L) {
    const FsshNArgs& A = *ns_opaque(Ap);
    const int64_t nt = A.ntraj;
    A.r[L.tid] = (double)L.r;
    A.v[L.tid] = (double)L.v;
#pragma unroll
    for (int i = 0; i < NM; ++i)
#pragma unroll
        for (int j = 0; j < NM; ++j) {
            double re, im;
            if (i == j) { re = L.a[i]; im = 0.0; }
            else if (i < j) { re = L.x[pidx<NM>(i, j)]; im = L.y[pidx<NM>(i, j)]; }
            else { re = L.x[pidx<NM>(j, i)]; im = -L.y[pidx<NM>(j, i)]; }
            A.sig_re[(int64_t)(i + NM * j) * nt + L.tid] = re;
            A.sig_im[(int64_t)(i + NM * j) * nt + L.tid] = im;
        }
    A.state[L.tid] = L.st;
    A.steps[L.tid] = L.step;
    A.nhops[L.tid] = L.nh;
}

// The launch arguments the step reads, in scalar registers for the whole persistent loop (read per step through the
// argument pointer, each is a vector-memory round trip with a full wait).
struct NsHot {
    int32_t method, rescaling, nsub, save_every, cell_mode, term_kind;
    int64_t nsteps;
    double dt, inv_mass, term_value;
    uint64_t key;
};

__device__ __forceinline__ NsHot ns_hot(const FsshNArgs& A) {
    NsHot H;
    H.method = uniform_sgpr(A.method); H.rescaling = uniform_sgpr(A.rescaling); H.nsub = uniform_sgpr(A.nsub);
    H.save_every = uniform_sgpr(A.save_every); H.cell_mode = uniform_sgpr(A.cell.mode);
    H.term_kind = uniform_sgpr(A.term_kind); H.nsteps = uniform_sgpr(A.nsteps);
    H.dt = uniform_sgpr(A.dt); H.inv_mass = uniform_sgpr(A.inv_mass); H.term_value = uniform_sgpr(A.term_value);
    H.key = uniform_sgpr(A.key);
    return H;
}

// SER: the default five sub-steps, by the power series where it serves; otherwise any number of sub-steps.
template <int NM, typename R, bool SER>
__device__ __forceinline__ void ns_step(const FsshNArgs* Ap, const FsshNArgs& A, const NsHot& H, LaneN<NM, R>& L) {
    constexpr int NP = LaneN<NM, R>::NP;
    constexpr int NQ = NP > 0 ? NP : 1;
    const R hdt = (R)(0.5 * H.dt), dtR = (R)H.dt;
    const R vt = L.v + hdt * L.k;                                     // step_B!
    L.r = L.r + dtR * vt;                                             // step_A!
    double vd[NM], vo[NQ], dd[NM], dof[NQ], E[NM], Gd[NM], Go[NQ];
    ns_model<NM, R>(L, L.r, vd, vo, dd, dof);                         // update_cache!
    // from the identity, not from the previous step's basis: where two states cross with a coupling of 1e-20 the sign
    // of their overlaps hangs on components that small, which rotations of V itself give to full relative accuracy
    ns_eigen<NM>(L.n, vd, vo, E, L.U, true);
    ns_rotate<NM>(L.U, dd, dof, Gd, Go);
    ns_accel<NM, R>(H, L, Gd, Go, L.a, L.x);                          // sigma of the step start
    L.v = vt + hdt * L.k;                                             // step_B!
    // nonadiabatic couplings d_ij = G_ij / (E_j - E_i) and W = v d on the trajectory's n states
    double d[NQ];
    NsInterp<NM> I;
#pragma unroll
    for (int i = 0; i < NM; ++i)
#pragma unroll
        for (int j = i + 1; j < NM; ++j) {
            const int p = pidx<NM>(i, j);
            d[p] = (j < L.n) ? Go[p] * nr_rcp(E[j] - E[i]) : 0.0;
            I.Wn[p] = d[p] * (double)L.v;
            I.Wc[p] = L.Wc[p];
        }
#pragma unroll
    for (int i = 0; i < NM; ++i) { I.Ec[i] = L.Ec[i]; I.En[i] = E[i]; }
    const double tn = L.t + H.dt;
    I.tc = L.tc; I.tn = tn;
    // step!(electronic_integrator, dt, true) (bab_electronics.jl:87-90)
    bool series = SER;
    if constexpr (SER) {
        // energies and couplings at the step start and their change over the step, times dt
        const double inv = nr_rcp(tn - L.tc), off = (L.t - L.tc) * inv, len = H.dt * inv;
        double e0[NM], w0[NQ], e1[NM], w1[NQ];
#pragma unroll
        for (int i = 0; i < NM; ++i) {
            const double d1 = E[i] - L.Ec[i];
            e0[i] = H.dt * fma(d1, off, L.Ec[i]);
            e1[i] = (H.dt * len) * d1;
        }
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const double d1 = I.Wn[p] - L.Wc[p];
            w0[p] = H.dt * fma(d1, off, L.Wc[p]);
            w1[p] = (H.dt * len) * d1;
        }
        const double m0 = ns_norm<NM>(L.n, e0, w0), m1 = ns_norm<NM>(L.n, e1, w1);
        const double z2 = fma(4.0, m1, m0 * m0);
        int parts = 1;
        if constexpr (sizeof(R) == 8) {
            // FP64 nuclei: where the sub-steps' own error and theirs on the change of A stay below 1e-12 a step
            // (series_step2's comment), so that leaving both out changes nothing; else the sub-steps
            const double m = m0 + m1, mm = m * m;
            series = 1.4e-8 * (mm * mm) * (mm + m1) < 1e-12;
        } else {
            // FP32 nuclei: the series throughout, on parts of a step whose generator passes a norm of 12
            if (z2 >= 4.0) parts = (int)fmin(ceil(fma(0.5, m1, m0 + m1) * (1.0 / 12.0)), 64.0);
        }
        if (series) {
            if constexpr (sizeof(R) == 8) {
                ns_series<NM>(e0, w0, e1, w1, ns_series_orders(z2), L.a, L.x, L.y);
            } else {
                const double rp = nr_rcp((double)parts);
                const int orders = z2 >= 4.0 ? ns_long_orders(parts, rp, m0 + m1, m1) : ns_series_orders(z2);
#pragma unroll
                for (int i = 0; i < NM; ++i) { e0[i] *= rp; e1[i] *= rp * rp; }
#pragma unroll
                for (int p = 0; p < NP; ++p) { w0[p] *= rp; w1[p] *= rp * rp; }
#pragma unroll 1
                for (int q = 0; q < parts; ++q) {
                    ns_series<NM>(e0, w0, e1, w1, orders, L.a, L.x, L.y);
#pragma unroll
                    for (int i = 0; i < NM; ++i) e0[i] += e1[i];
#pragma unroll
                    for (int p = 0; p < NP; ++p) w0[p] += w1[p];
                }
            }
        }
    }
    if constexpr (!SER || sizeof(R) == 8) {
        if (!series) {   // nsub sub-steps clipped to t + dt
            const double h = H.dt / (double)H.nsub;
            double tau = L.t;
            for (int s = 0; s < H.nsub; ++s) {
                const double hs = fmin(h, tn - tau);
                ns_tsit5<NM>(I, tau, hs, L.a, L.x, L.y);
                tau = (s == H.nsub - 1) ? tn : tau + hs;
            }
        }
    }
#pragma unroll
    for (int i = 0; i < NM; ++i) L.Ec[i] = E[i];
#pragma unroll
    for (int p = 0; p < NP; ++p) L.Wc[p] = I.Wn[p];
    L.tc = tn;
    L.t = tn;
    // the save precedes the hop callback (a save time holds the state before the step's callbacks)
    if (H.save_every > 0 && ((L.step + 1) % H.save_every) == 0) ns_save<NM, R>(Ap, L, (L.step + 1) / H.save_every);
    if (H.method == 0) {  // HoppingCallback (surface_hopping.jl:2-16), fssh.jl:96-121
        const int s = L.st;
        double ass = 0.0;
#pragma unroll
        for (int i = 0; i < NM; ++i) ass = (i == s) ? L.a[i] : ass;
        double cum[NM];
        double run = 0.0;
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            double pm = 0.0;
            if (m != s && m < L.n) {
                double xms = 0.0, dsm = 0.0;  // Re sigma_ms and d_sm
#pragma unroll
                for (int q = 0; q < NM; ++q) {
                    if (q == s) {
                        if (m < q) { xms = L.x[pidx<NM>(m, q)]; dsm = -d[pidx<NM>(m, q)]; }
                        else if (m > q) { xms = L.x[pidx<NM>(q, m)]; dsm = d[pidx<NM>(q, m)]; }
                    }
                }
                pm = 2.0 * (double)L.v * (xms / ass) * dsm * H.dt;
                pm = fmin(fmax(pm, 0.0), 1.0);
            }
            run += pm;
            cum[m] = run;
        }
        if (run > 0.0) {
            const double rnd = philox_uniform((uint64_t)L.tid, (uint32_t)L.step, STREAM_HOP, H.key);
            int ns = s;
            bool found = false;
#pragma unroll
            for (int m = 0; m < NM; ++m)
                if (!found && m != s && m < L.n && cum[m] > rnd) { ns = m; found = true; }
            if (found) {
                double dno = 0.0, dE = 0.0;  // coupling[new, old], E_new - E_old
#pragma unroll
                for (int i = 0; i < NM; ++i)
#pragma unroll
                    for (int j = i + 1; j < NM; ++j) {
                        if (i == ns && j == s) dno = d[pidx<NM>(i, j)];
                        if (i == s && j == ns) dno = -d[pidx<NM>(i, j)];
                    }
#pragma unroll
                for (int i = 0; i < NM; ++i) { if (i == ns) dE += E[i]; if (i == s) dE -= E[i]; }
                R vv[1] = {L.v};
                const double dc[1] = {dno};
                const double im[1] = {H.inv_mass};
                if (rescale_velocity<1, R>(H.rescaling, vv, im, dc, dE)) { L.st = ns; ++L.nh; }
                L.v = vv[0];
            }
        }
    }
    if (H.cell_mode == 1) {  // CellBoundaryCallback after the hop callback; the step-end acceleration is kept
        R rr[1] = {L.r};
        if (cell_outside<1, 1, R>(A.cell, rr)) { cell_wrap<1, 1, R>(A.cell, rr); L.r = rr[0]; }
    }
    ++L.step;
}

template <int NM, typename R, bool SER>
__device__ __forceinline__ void ns_body(const FsshNArgs* __restrict__ Ap, double* tabs) {
    const FsshNArgs& A = *Ap;
    const NsHot H = ns_hot(A);
    for (int i = threadIdx.x; i < A.ntab; i += blockDim.x) tabs[i] = A.mtab[i];   // the models' tables, read every step
    __syncthreads();
    const int lane = __lane_id();
    const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    LaneN<NM, R> L;
    bool active = false, exhausted = false;
    for (;;) {
        const uint64_t want = __ballot(!active && !exhausted);
        if (want) {
            const int cnt = __popcll(want);
            const int leader = __ffsll((unsigned long long)want) - 1;
            unsigned long long base = 0;
            if (lane == leader) base = atomicAdd(ns_opaque(Ap)->queue, (unsigned long long)cnt);
            base = __shfl(base, leader);
            if (!active && !exhausted) {
                const unsigned long long q = base + (unsigned long long)__popcll(want & below);
                if (q < (unsigned long long)A.ntraj) {
                    const int32_t* order = ns_opaque(Ap)->order;
                    ns_load<NM, R>(Ap, L, order ? (int64_t)order[q] : (int64_t)q, tabs);
                    if (H.nsteps <= 0) ns_finish<NM, R>(Ap, L); else active = true;
                } else {
                    exhausted = true;
                }
            }
        }
        if (__ballot(active) == 0) break;
        if (active) {
            ns_step<NM, R, SER>(Ap, A, H, L);
            // TerminatingCallback after each step, not at t0 (callbacks.jl:15-29)
            const R rr[1] = {L.r};
            if (L.step >= H.nsteps || (H.cell_mode == 2 && cell_outside<1, 1, R>(A.cell, rr)) ||
                term_hit(H.term_kind, (double)L.r, H.term_value)) {
                ns_finish<NM, R>(Ap, L);
                active = false;
            }
        }
    }
}

// f32s, f64s: the default five sub-steps (the power series); f32, f64: other counts.
#define NQCD_NS_KERNEL(NAME, NM, R, SER)                                                                 \
    __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu((NM) <= 3 ? 2 : 1)))            \
    void NAME(const FsshNArgs* __restrict__ Ap) {                                                        \
        extern __shared__ double ns_tabs[];                                                              \
        ns_body<NM, R, SER>(Ap, ns_tabs);                                                                \
    }
#define NQCD_NS_KERNELS(NM)                                                                              \
    NQCD_NS_KERNEL(fssh_n_f64_##NM, NM, double, false)                                                   \
    NQCD_NS_KERNEL(fssh_n_f64s_##NM, NM, double, true)                                                   \
    NQCD_NS_KERNEL(fssh_n_f32_##NM, NM, float, false)                                                    \
    NQCD_NS_KERNEL(fssh_n_f32s_##NM, NM, float, true)

// The kernel of a precision and of the default (five) or another count of sub-steps.
#define NQCD_NS_PICK(NM, precision, five)                                                                \
    ((precision) == 0 ? ((five) ? (NsKernelPtr)fssh_n_f64s_##NM : (NsKernelPtr)fssh_n_f64_##NM)                \
                      : ((five) ? (NsKernelPtr)fssh_n_f32s_##NM : (NsKernelPtr)fssh_n_f32_##NM))

}  // namespace nqcd
