// Density-based implicit updates of SEMO's dual-time solvers
// (src/solvers/linearSolver.cpp) on the device:
//   - calcLinearSolver (:666-725): per cell, res <- (P + 1.5 dtau/dt T)^-1 res;
//   - calcSingleLinearSolver (:729-787): per cell, res <- T^-1 res;
//   - calcLinearSolverLUSGS (:144-389): a forward then a backward Gauss-Seidel
//     sweep over the cells in lib_RCM's order, the off-diagonal blocks being
//     the faces' upwind flux Jacobians (getNumericalFluxJacobianUpwind,
//     :394-640) times dtau / V * area.
// P and T are constructMatrix's (:791-890); the block inverse is
// GaussSeidelSOR's (src/math/math.cpp:141-200): Doolittle LU without
// pivoting, then a forward and a back substitution per unit column.  The
// arithmetic is the reference's, in its order; pow(x, 2.0) is written x * x.
//
// The sweeps are sequential by definition: cell i reads the already-updated
// residuals of its neighbours that come before it (forward) or after it
// (backward).  Their dependency graph is levelled on the host once per mesh:
// a cell's forward level is one more than the largest level of its earlier
// neighbours, so the cells of one level depend only on lower levels.  A sweep
// is one launch whose wavefronts take up to 16 cells of one level at a time,
// in level order, and wait for the neighbours' values themselves
// (k_lusgs_sweep), with the sequential sweep's result.
// The diagonal block (the same in both sweeps) is formed and inverted once,
// fully parallel, and stored (dinv_at).
//
// Cell state records, [n][12 + 3 nsp] in device order: P, U, V, W, T, rho,
// C, Ht, dRhoDP, dHtDP, dRhoDT, dHtDT, Ur, dtPseudo, Y_0..Y_{nsp-1},
// dRhoDY_0..dRhoDY_{nsp-2}, dHtDY_0..dHtDY_{nsp-2}; residuals [n][4 + nsp].
#include "common.hpp"
#include "kern.hpp"

namespace semo {
namespace {

enum { sP = 0, sU, sV, sW, sT, sRHO, sC, sHT, sDRDP, sDHDP, sDRDT, sDHDT, sUR, sDTP, sY0 };

template <int NSP>
struct LS {
    static constexpr int N = 4 + NSP, K = 12 + 3 * NSP;
};

template <int NSP>
__device__ inline void load_rec(const double* __restrict__ st, int i, double (&s)[LS<NSP>::K]) {
    const double* p = st + (size_t)i * LS<NSP>::K;
#pragma unroll
    for (int k = 0; k < LS<NSP>::K; ++k) s[k] = p[k];
}

// constructMatrix (linearSolver.cpp:791-890)
template <int NSP>
__device__ inline void construct(const double (&s)[LS<NSP>::K], double (&Pm)[4 + NSP][4 + NSP],
                                 double (&Tm)[4 + NSP][4 + NSP]) {
    constexpr int N = 4 + NSP;
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
        for (int j = 0; j < N; ++j) Tm[i][j] = 0.0;
    const double DRDP = s[sDRDP], DHDP = s[sDHDP], DRDT = s[sDRDT], DHDT = s[sDHDT];
    const double Rho = s[sRHO], U = s[sU], V = s[sV], W = s[sW], Ht = s[sHT];
    Tm[0][0] = DRDP; Tm[1][0] = DRDP * U; Tm[2][0] = DRDP * V; Tm[3][0] = DRDP * W;
    Tm[4][0] = DRDP * Ht + Rho * DHDP - 1.0;
    Tm[1][1] = Rho; Tm[4][1] = Rho * U;
    Tm[2][2] = Rho; Tm[4][2] = Rho * V;
    Tm[3][3] = Rho; Tm[4][3] = Rho * W;
    Tm[0][4] = DRDT; Tm[1][4] = DRDT * U; Tm[2][4] = DRDT * V; Tm[3][4] = DRDT * W;
    Tm[4][4] = DRDT * Ht + Rho * DHDT;
#pragma unroll
    for (int a = 0; a < NSP - 1; ++a) {
        const int q = 5 + a;
        const double Y = s[sY0 + a], dRdY = s[sY0 + NSP + a], dHdY = s[sY0 + 2 * NSP - 1 + a];
        Tm[q][0] = DRDP * Y;
        Tm[q][4] = DRDT * Y;
#pragma unroll
        for (int b = 0; b < NSP - 1; ++b) Tm[q][5 + b] = Y * s[sY0 + NSP + b];
        Tm[q][q] += Rho;
        Tm[0][q] = dRdY; Tm[1][q] = dRdY * U; Tm[2][q] = dRdY * V; Tm[3][q] = dRdY * W;
        Tm[4][q] = dRdY * Ht + Rho * dHdY;
    }
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
        for (int j = 0; j < N; ++j) Pm[i][j] = Tm[i][j];
    const double beta = 1.0 / (s[sUR] * s[sUR]) + DRDP - 1.0 / (s[sC] * s[sC]);
    Pm[0][0] = beta; Pm[1][0] = beta * U; Pm[2][0] = beta * V; Pm[3][0] = beta * W;
    Pm[4][0] = beta * Ht + Rho * DHDP - 1.0;
#pragma unroll
    for (int a = 0; a < NSP - 1; ++a) Pm[5 + a][0] = beta * s[sY0 + a];
}

// getNumericalFluxJacobianUpwind (linearSolver.cpp:394-640), side "R" when
// RIGHT, else "L": 0.5 dF/dQ of that side's state +/- 0.5 of the Roe-type
// dissipation of the face averages (none in the species rows).  The rows are
// handed to `use(i, row)` one after the other, so that a caller that consumes
// them as they come holds one row and not the matrix.
template <int NSP, bool RIGHT, class RowF>
__device__ inline void jacobian(const double (&L)[LS<NSP>::K], const double (&R)[LS<NSP>::K], const double n[3],
                                RowF use) {
    constexpr int N = 4 + NSP;
    const double UnL = L[sU] * n[0] + L[sV] * n[1] + L[sW] * n[2];
    const double UnR = R[sU] * n[0] + R[sV] * n[1] + R[sW] * n[2];
    const double RT = sqrt(L[sRHO] / R[sRHO]);
    const double Rhohat = 0.5 * (L[sRHO] + R[sRHO]);
    const double Chat = 0.5 * (L[sC] + R[sC]);
    const double Unhat = 0.5 * (UnL + UnR);
    const double hat[3] = {(RT * L[sU] + R[sU]) / (RT + 1.0), (RT * L[sV] + R[sV]) / (RT + 1.0),
                           (RT * L[sW] + R[sW]) / (RT + 1.0)};
    const double Hthat = (RT * L[sHT] + R[sHT]) / (RT + 1.0);
    const double fgL = RIGHT ? 0.0 : 1.0, fgR = RIGHT ? 1.0 : 0.0;
    const double vel[3] = {L[sU] * fgL + R[sU] * fgR, L[sV] * fgL + R[sV] * fgR, L[sW] * fgL + R[sW] * fgR};
    const double HtLR = L[sHT] * fgL + R[sHT] * fgR, RhoLR = L[sRHO] * fgL + R[sRHO] * fgR;
    const double DRDPLR = L[sDRDP] * fgL + R[sDRDP] * fgR, DHDPLR = L[sDHDP] * fgL + R[sDHDP] * fgR;
    const double DRDTLR = L[sDRDT] * fgL + R[sDRDT] * fgR, DHDTLR = L[sDHDT] * fgL + R[sDHDT] * fgR;
    const double UnLR = UnL * fgL + UnR * fgR;
    double YLR[NSP], DRDYLR[NSP], DHDYLR[NSP];
#pragma unroll
    for (int a = 0; a < NSP - 1; ++a) {
        YLR[a] = L[sY0 + a] * fgL + R[sY0 + a] * fgR;
        DRDYLR[a] = L[sY0 + NSP + a] * fgL + R[sY0 + NSP + a] * fgR;
        DHDYLR[a] = L[sY0 + 2 * NSP - 1 + a] * fgL + R[sY0 + 2 * NSP - 1 + a] * fgR;
    }
    const double dissUp = (Chat - fabs(Unhat)) / Rhohat / Chat / Chat;
    const double dissUu = Unhat / Chat;
    const double dissPp = Unhat / Chat;
    const double dissPu = (Chat - fabs(Unhat)) * Rhohat;
    const double AD = fabs(Unhat);
#pragma unroll
    for (int i = 0; i < N; ++i) {
        // row i of the convective part (fluxLRdot) and of the dissipation
        // (dissimat, 5 x 5)
        double F[N], D[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
        if (i == 0) {
            F[0] = DRDPLR * UnLR;
#pragma unroll
            for (int d = 0; d < 3; ++d) F[1 + d] = RhoLR * n[d];
            F[4] = DRDTLR * UnLR;
#pragma unroll
            for (int a = 0; a < NSP - 1; ++a) F[5 + a] = DRDYLR[a] * UnLR;
            D[0] = AD * DRDPLR + dissUp * Rhohat;
#pragma unroll
            for (int c = 0; c < 3; ++c) D[1 + c] = dissUu * n[c] * Rhohat;
            D[4] = AD * DRDTLR;
        } else if (i < 4) {
            const int r = i - 1;
            F[0] = DRDPLR * UnLR * vel[r] + n[r];
#pragma unroll
            for (int d = 0; d < 3; ++d)
                F[1 + d] = r == d ? RhoLR * n[d] * vel[r] + RhoLR * UnLR : RhoLR * n[d] * vel[r];
            F[4] = DRDTLR * UnLR * vel[r];
#pragma unroll
            for (int a = 0; a < NSP - 1; ++a) F[5 + a] = DRDYLR[a] * UnLR * vel[r];
            D[0] = AD * DRDPLR * vel[r] + dissUp * Rhohat * hat[r] + dissPp * n[r];
#pragma unroll
            for (int c = 0; c < 3; ++c)
                D[1 + c] = r == c ? AD * RhoLR + dissUu * n[c] * Rhohat * hat[r] + dissPu * n[c] * n[r]
                                  : dissUu * n[c] * Rhohat * hat[r] + dissPu * n[c] * n[r];
            D[4] = AD * DRDTLR * vel[r];
        } else if (i == 4) {
            F[0] = DRDPLR * UnLR * HtLR + RhoLR * UnLR * DHDPLR;
#pragma unroll
            for (int d = 0; d < 3; ++d) F[1 + d] = RhoLR * n[d] * HtLR + RhoLR * UnLR * vel[d];
            F[4] = DRDTLR * UnLR * HtLR + RhoLR * UnLR * DHDTLR;
#pragma unroll
            for (int a = 0; a < NSP - 1; ++a) F[5 + a] = DRDYLR[a] * UnLR * HtLR + RhoLR * UnLR * DHDYLR[a];
            D[0] = AD * (DRDPLR * HtLR + RhoLR * DHDPLR - 1.0) + dissUp * Rhohat * Hthat + dissPp * Unhat;
#pragma unroll
            for (int c = 0; c < 3; ++c)
                D[1 + c] = AD * RhoLR * vel[c] + dissUu * n[c] * Rhohat * Hthat + dissPu * n[c] * Unhat;
            D[4] = AD * (DRDTLR * HtLR + RhoLR * DHDTLR);
        } else {
            const int a = i - 5;
            F[0] = DRDPLR * YLR[a] * UnLR;
#pragma unroll
            for (int d = 0; d < 3; ++d) F[1 + d] = RhoLR * YLR[a] * n[d];
            F[4] = DRDTLR * YLR[a] * UnLR;
#pragma unroll
            for (int b = 0; b < NSP - 1; ++b) F[5 + b] = DRDYLR[b] * YLR[a] * UnLR;
            F[i] += RhoLR * UnLR;
        }
        double J[N];
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const double d = (i < 5 && j < 5) ? D[j < 5 ? j : 0] : 0.0;
            J[j] = RIGHT ? 0.5 * F[j] - 0.5 * d : 0.5 * F[j] + 0.5 * d;
        }
        use(i, J);
    }
}

// Division of several numbers by the same b: y = 1 / b once, then per
// quotient q = a y corrected by its exact remainder (Markstein, IBM J. Res.
// Dev. 34 (1990) 111), three operations instead of a division of some twelve.
// The quotient is a / b as rounded by the division while no step leaves the
// normal range: the divisor is checked (div_ok), a quotient that overflows or
// starts from a non-finite a is found by the caller among its results, which
// are then formed again with plain divisions.  Below 1e-292 the last bit may
// differ.
template <bool PLAIN>
__device__ inline double quot(double a, double b, double y) {
    if constexpr (PLAIN) return a / b;
    const double q = a * y;
    return __builtin_fma(__builtin_fma(-b, q, a), y, q);
}
__device__ inline bool div_ok(double b) { return fabs(b) > 0x1p-900 && fabs(b) < 0x1p900; }

// GaussSeidelSOR (math.cpp:141-200), in place: A's upper triangle becomes U,
// its strict lower triangle the multipliers L (which the reference keeps in
// a separate matrix; the elimination never reads them back).  Y: the
// reciprocals of U's diagonal.  False if quot needs PLAIN for one of them.
template <int N, bool PLAIN>
__device__ inline bool lu_nopivot(double (&A)[N][N], double (&Y)[N]) {
    bool ok = true;
#pragma unroll
    for (int k = 0; k < N; ++k) {
        if constexpr (!PLAIN) { Y[k] = 1.0 / A[k][k]; ok = ok && div_ok(A[k][k]); }
#pragma unroll
        for (int i = k + 1; i < N; ++i) {
            const double coeff = quot<PLAIN>(A[i][k], A[k][k], Y[k]);
#pragma unroll
            for (int j = k + 1; j < N; ++j) A[i][j] = A[i][j] - coeff * A[k][j];
            A[i][k] = coeff;
        }
    }
    return ok;
}

// Column k of the inverse: forward substitution of the unit vector e_k
// through L, back substitution through U.  The zeros above row k stay zero:
// without PLAIN their products are left out (a non-finite L shows in its own
// column).  k_lusgs_diag keeps PLAIN: at 256 registers the second pass over a
// cell that the check needs costs it a wavefront per SIMD.
template <int N, bool PLAIN>
__device__ inline void inverse_column(const double (&A)[N][N], const double (&Y)[N], int k, double (&X)[N]) {
    double Dv[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
        Dv[i] = i == k ? 1.0 : 0.0;
#pragma unroll
        for (int j = 0; j < i; ++j)
            if (PLAIN || j >= k) Dv[i] = Dv[i] - A[i][j] * Dv[j];
    }
    X[N - 1] = quot<PLAIN>(Dv[N - 1], A[N - 1][N - 1], Y[N - 1]);
#pragma unroll
    for (int i = N - 2; i >= 0; --i) {
        X[i] = Dv[i];
#pragma unroll
        for (int j = N - 1; j >= i + 1; --j) X[i] = X[i] - A[i][j] * X[j];
        X[i] = quot<PLAIN>(X[i], A[i][i], Y[i]);
    }
}

// use(k, X) for the columns of A's inverse; false: to be done again with PLAIN
template <int N, bool PLAIN, class Use>
__device__ inline bool inverse(double (&A)[N][N], Use use) {
    double Y[N];
    bool ok = lu_nopivot<N, PLAIN>(A, Y);
#pragma unroll
    for (int k = 0; k < N; ++k) {
        double X[N];
        inverse_column<N, PLAIN>(A, Y, k, X);
        if constexpr (!PLAIN)
#pragma unroll
            for (int j = 0; j < N; ++j) ok = ok && __builtin_isfinite(X[j]);
        use(k, X);
    }
    return ok;
}

// calcLinearSolver (SINGLE false) / calcSingleLinearSolver (SINGLE true):
// one thread per cell; the inverse's columns are applied as they come, which
// is the reference's k-ordered sum sum_k Ainv[j][k] b[k].  Bound by FP64
// arithmetic (some 2400 operations a cell with three species, 70 divisions
// among them, against 280 bytes): with seven reciprocals in place of the
// divisions and the substitutions' zeros left out 309,690 cells take 20.8 us
// against 27, their bytes 14.
template <int NSP, bool SINGLE>
__global__ __launch_bounds__(TPB) void k_linsol_point(int n, const double* __restrict__ st, double time_step,
                                                      double* __restrict__ res) {
    constexpr int N = 4 + NSP;
    const int i = xcd_block() * TPB + (int)threadIdx.x;
    if (i >= n) return;
    double out[N];
    auto cell = [&](auto plain) {
        double s[LS<NSP>::K];
        load_rec<NSP>(st, i, s);
        double A[N][N];
        {
            double Pm[N][N], Tm[N][N];
            construct<NSP>(s, Pm, Tm);
            const double f = 1.5 * s[sDTP] / time_step;
#pragma unroll
            for (int a = 0; a < N; ++a)
#pragma unroll
                for (int c = 0; c < N; ++c) A[a][c] = SINGLE ? Tm[a][c] : Pm[a][c] + f * Tm[a][c];
        }
        double b[N];
#pragma unroll
        for (int a = 0; a < N; ++a) { b[a] = res[(size_t)i * N + a]; out[a] = 0.0; }
        return inverse<N, decltype(plain)::value>(A, [&](int k, const double (&X)[N]) {
#pragma unroll
            for (int j = 0; j < N; ++j) out[j] += X[j] * b[k];
        });
    };
    if (!cell(std::false_type{})) cell(std::true_type{});
#pragma unroll
    for (int a = 0; a < N; ++a) res[(size_t)i * N + a] = out[a];
}

__device__ inline void face_normal(const double* __restrict__ nrm, int f, bool own_is_owner, double n[3]) {
#pragma unroll
    for (int a = 0; a < 3; ++a) n[a] = own_is_owner ? nrm[3 * (size_t)f + a] : -nrm[3 * (size_t)f + a];
}

// place of entry 0 of cell i's inverted diagonal block; entry e lies 64 e
// further: 64 cells together, entry by entry, so that a wavefront's stores of
// one entry are one run and so are a sweep unit's loads of it (cells of one
// level are mostly consecutive)
template <int N>
__device__ inline size_t dinv_at(int i) { return (size_t)(i >> 6) * (64 * N * N) + (i & 63); }

// LU-SGS diagonal blocks: P + 1.5 (dtau / dt) T + sum over the cell's faces
// (ascending) of dtau / V * J_L * area, inverted.  FP64 arithmetic and the
// 144-byte records of seven cells a thread bound it: 128^3, two species,
// 770 -> 550 us once each Jacobian row was added as it was formed (212
// registers, two wavefronts per SIMD, against 310 and one) and the blocks
// were stored in runs.
template <int NSP>
__global__ __launch_bounds__(TPB) void k_lusgs_diag(int n, int nif, const int* __restrict__ cf_ptr,
                                                    const int* __restrict__ cf_idx, const int* __restrict__ owner,
                                                    const int* __restrict__ nbr, const double* __restrict__ nrm,
                                                    const double* __restrict__ area, const double* __restrict__ vol,
                                                    const double* __restrict__ st, double time_step,
                                                    double* __restrict__ dinv) {
    constexpr int N = 4 + NSP;
    const int i = xcd_block() * TPB + (int)threadIdx.x;
    if (i >= n) return;
    double s[LS<NSP>::K];
    load_rec<NSP>(st, i, s);
    const double rDtauPerVol = s[sDTP] / vol[i];
    double DS[N][N];
#pragma unroll
    for (int a = 0; a < N; ++a)
#pragma unroll
        for (int c = 0; c < N; ++c) DS[a][c] = 0.0;
    for (int k = cf_ptr[i]; k < cf_ptr[i + 1]; ++k) {
        const int f = cf_idx[k];
        const int o = owner[f];
        double nv[3];
        face_normal(nrm, f, o == i, nv);
        const double A = area[f];
        // row by row, each added before the next is formed
        auto add = [&](int a, const double (&J)[N]) {
#pragma unroll
            for (int c = 0; c < N; ++c) {
                DS[a][c] += rDtauPerVol * J[c] * A;
                asm volatile("" : "+v"(DS[a][c]));
            }
        };
        double sn[LS<NSP>::K];
        load_rec<NSP>(st, f < nif ? (o == i ? nbr[f] : o) : i, sn);
        jacobian<NSP, false>(s, sn, nv, add);
    }
    double M[N][N];
    {
        double Pm[N][N], Tm[N][N];
        construct<NSP>(s, Pm, Tm);
        const double timeFrac = s[sDTP] / time_step;
#pragma unroll
        for (int a = 0; a < N; ++a)
#pragma unroll
            for (int c = 0; c < N; ++c) {
                M[a][c] = Pm[a][c] + 1.5 * timeFrac * Tm[a][c];
                M[a][c] += DS[a][c];
            }
    }
    inverse<N, true>(M, [&](int k, const double (&X)[N]) {
#pragma unroll
        for (int j = 0; j < N; ++j) dinv[dinv_at<N>(i) + (size_t)(j * N + k) * 64] = X[j];
    });
}

// Broadcast within each quad of lanes (DPP quad_perm): every lane gets lane
// SRC's value of its quad.
template <int SRC>
__device__ inline double quad_bcast(double v) {
    constexpr int CTRL = SRC * 0x55;
    int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xF, 0xF, false);
    int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}

// A value no sweep result can be: a signaling NaN, which arithmetic quiets.
constexpr unsigned long long LS_EMPTY = 0x7FF4A5A5C3C35A5Aull;
// polls of one neighbour before a sweep gives up (about ten seconds): never
// reached by the argument at k_lusgs_sweep, so that a mistake in the schedule
// ends in an error instead of a hang
constexpr int LS_POLL_LIMIT = 1 << 23;

// words of the control array: per sweep one ticket counter for each wavefront
// of a block, 256 bytes apart, then the error word
constexpr int LS_STEP = 64, LS_WAVES = TPB / 64, LS_ERR = 2 * LS_WAVES * LS_STEP, LS_CTL = LS_ERR + LS_STEP;

// the results emptied, tickets and error word cleared: max(n, LS_CTL) threads
__global__ __launch_bounds__(TPB) void k_lusgs_empty(size_t n, unsigned long long* __restrict__ v,
                                                     int* __restrict__ ctl) {
    size_t k = (size_t)blockIdx.x * TPB + threadIdx.x;
    if (k < LS_CTL) ctl[k] = 0;
    if (k < n) v[k] = LS_EMPTY;
}

__device__ inline double ls_load(const double* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void ls_store(double* p, double v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One sweep, four lanes (a quad) per cell, 16 cells of one level per unit of
// work (slots 16 u .. 16 u + 15; the last unit of a level is filled up with
// copies of its first slot, whose results are not stored).  Slot t holds its
// cell, and the cell's faces toward earlier (FWD) /
// later cells in ascending face order as (neighbour, face) pairs, the face
// stored as ~f when the cell is the face's neighbour (normal reversed): the
// first four in the slot's 48-byte record (one load round gives a lane its
// cell and its pair), the rest in an overflow list.  Lane l of the quad takes
// pairs l, l + 4, ...: its term dtau / V * (J_R r_ngb) * area; the quad adds
// the terms in pair order (the reference's sum), then forward: r <- Dinv (r -
// sum), backward: r <- r - Dinv sum, rows l and l + 4 on lane l.  Control
// flow is uniform within a quad, so every DPP source lane is active.
//
// A lane forms its face's Jacobian first and then polls the neighbour's
// result in `out`, which starts as LS_EMPTY: the value is its own flag, so a
// dependency costs one store and one load through the memory side (the XCDs'
// L2s do not share lines), not a flag and then the data, and not a launch.
// Units are taken in level order by tickets, unit u by the wavefronts of
// place u mod 4 in their block (one counter would be taken at 14 ns a ticket,
// 1.9 ms a sweep at 128^3): every block has wavefronts of all four places and
// each holds, besides its current unit, at most two later ones of the same
// counter.  So the lowest unfinished unit is some wavefront's current one or
// is come to without a wait: what lies before it on its counter is finished,
// as is all it waits for.  Every wait ends, whatever else runs on the device.
// A unit's cells are of one level: no lane waits for another lane of its
// wavefront.
// Bound by that chain: 128^3 hexes (382 levels a sweep) 2.8 us a level,
// against 6.1 us with a launch per level (4.65 -> 2.16 ms for both sweeps).
template <int NSP, bool FWD>
__global__ __launch_bounds__(TPB) void k_lusgs_sweep(int nunits, const int4* __restrict__ slots,
                                                     const int2* __restrict__ ovf,
                                                     const double* __restrict__ nrm, const double* __restrict__ area,
                                                     const double* __restrict__ vol, const double* __restrict__ st,
                                                     const double* __restrict__ dinv, const double* __restrict__ rin,
                                                     double* out, double* __restrict__ res, int* __restrict__ ctl) {
    constexpr int N = 4 + NSP;
    static_assert(N <= 8, "two rows per lane");
    const int lane = (int)threadIdx.x & 63, l = lane & 3;
    const int place = (int)threadIdx.x >> 6;
    int* ticket = ctl + ((FWD ? 0 : LS_WAVES) + place) * LS_STEP;
    // a unit's slot records are requested while the unit before it is worked
    // on, its ticket one unit earlier still
    const int4* mine = slots + 3 * (lane >> 2);
    auto take = [&] { return lane == 0 ? atomicAdd(ticket, 1) : 0; };
    auto unit = [&](int tk) { return __builtin_amdgcn_readfirstlane(tk) * LS_WAVES + place; };
    int u = unit(take());
    if (u >= nunits) return;
    // slot record: {cell, pair count, overflow offset, to be stored}, pairs 0..3
    int4 h = mine[48 * (size_t)u], qq = mine[48 * (size_t)u + 1 + (l >> 1)];
    int tk = take();
    for (;;) {
        const int i = h.x, p1 = h.y, ovf0 = h.z, act = h.w;
        const int2 q0 = (l & 1) ? make_int2(qq.z, qq.w) : make_int2(qq.x, qq.y);
        u = unit(tk);
        if (u < nunits) {
            h = mine[48 * (size_t)u];
            qq = mine[48 * (size_t)u + 1 + (l >> 1)];
            tk = take();
        }
        double s[LS<NSP>::K];
        load_rec<NSP>(st, i, s);
        const double rDtauPerVol = s[sDTP] / vol[i];
        // the cell's own residual and this lane's Dinv rows do not depend on
        // the neighbours: in flight during the neighbour terms
        double ri[N], D0[N], D1[N];
        const double* Di = dinv + dinv_at<N>(i);
#pragma unroll
        for (int a = 0; a < N; ++a) {
            ri[a] = rin[(size_t)i * N + a];
            D0[a] = Di[64 * (l * N + a)];
            D1[a] = l + 4 < N ? Di[64 * ((l + 4) * N + a)] : 0.0;
        }
        double LU[N];
#pragma unroll
        for (int a = 0; a < N; ++a) LU[a] = 0.0;
        for (int base = 0; base < p1; base += 4) {
            const int p = base + l;
            double c[N];
#pragma unroll
            for (int a = 0; a < N; ++a) c[a] = 0.0;
            if (p < p1) {
                const int2 q = p < 4 ? q0 : ovf[ovf0 + p - 4];
                const int g = q.x;
                const bool own_is_owner = q.y >= 0;
                const int f = own_is_owner ? q.y : ~q.y;
                double nv[3];
                face_normal(nrm, f, own_is_owner, nv);
                double sn[LS<NSP>::K], J[N][N], rg[N];
                load_rec<NSP>(st, g, sn);
                double A = area[f];
                // formed before the wait, not sunk behind it
                jacobian<NSP, true>(s, sn, nv, [&](int a, const double (&Ja)[N]) {
#pragma unroll
                    for (int k = 0; k < N; ++k) {
                        J[a][k] = Ja[k];
                        asm volatile("" : "+v"(J[a][k]));
                    }
                });
                for (int poll = 0;; ++poll) {
                    bool ready = true;
#pragma unroll
                    for (int k = 0; k < N; ++k) rg[k] = ls_load(out + (size_t)g * N + k);
#pragma unroll
                    for (int k = 0; k < N; ++k)
                        ready = ready && (unsigned long long)__double_as_longlong(rg[k]) != LS_EMPTY;
                    if (ready) break;
                    if (poll >= LS_POLL_LIMIT) { ctl[LS_ERR] = 1; break; }
                    __builtin_amdgcn_s_sleep(1);
                }
#pragma unroll
                for (int a = 0; a < N; ++a) {
                    double sig = 0.0;
#pragma unroll
                    for (int k = 0; k < N; ++k) sig += rg[k] * J[a][k];
                    c[a] = rDtauPerVol * sig * A;
                }
            }
#pragma unroll
            for (int a = 0; a < N; ++a) {
                const double v0 = quad_bcast<0>(c[a]), v1 = quad_bcast<1>(c[a]);
                const double v2 = quad_bcast<2>(c[a]), v3 = quad_bcast<3>(c[a]);
                LU[a] += v0;
                if (base + 1 < p1) LU[a] += v1;
                if (base + 2 < p1) LU[a] += v2;
                if (base + 3 < p1) LU[a] += v3;
            }
        }
        double b[N];
#pragma unroll
        for (int a = 0; a < N; ++a) b[a] = FWD ? ri[a] - LU[a] : LU[a];
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const int j = l + 4 * r;
            if (j < N && act) {
                double v = 0.0;
#pragma unroll
                for (int k = 0; k < N; ++k) v += (r == 0 ? D0[k] : D1[k]) * b[k];
                if (!FWD) v = ri[j] - v;
                ls_store(out + (size_t)i * N + j, v);
                if (!FWD) res[(size_t)i * N + j] = v;
            }
        }
        if (u >= nunits) break;
    }
}

// Blocks of a sweep: one wavefront per SIMD.  Fewer leave units of the next
// levels unprepared; more only poll, and the polls slow the values down: with
// 128 / 192 / 256 / 384 / 512 blocks an update took 3.48 / 3.01 / 2.91 / 3.71 /
// 3.85 ms on 128^3 hexes, 1.06 / 1.09 / 1.14 / 1.15 / 1.14 ms on 144000 tets.
constexpr int LS_BLOCKS = 256;

// lib_RCM's order in device numbering (rank[i] = position of cell i) and
// the forward / backward level lists of the sweeps.
void lusgs_schedule(semo_ctx* c) {
    if (c->ls_ready) return;
    const int nc = c->nc, nif = c->nif;
    std::vector<int> rank(nc), order(nc);
    if (c->reordered) {
        std::iota(rank.begin(), rank.end(), 0);
    } else {   // lib_RCM's adjacency (RCM.cpp:79-126): internal faces in ascending order
        std::vector<int> cnt(nc + 1, 0);
        for (int f = 0; f < nif; ++f) { cnt[c->h_owner[f] + 1]++; cnt[c->h_nbr[f] + 1]++; }
        for (int i = 0; i < nc; ++i) cnt[i + 1] += cnt[i];
        std::vector<int> adj(cnt[nc]), pos(cnt.begin(), cnt.end() - 1);
        for (int f = 0; f < nif; ++f) {
            adj[pos[c->h_owner[f]]++] = c->h_nbr[f];
            adj[pos[c->h_nbr[f]]++] = c->h_owner[f];
        }
        std::vector<int> perm(nc);
        genrcm(nc, cnt.data(), adj.data(), perm.data(), rank.data());
    }
    for (int i = 0; i < nc; ++i) order[rank[i]] = i;
    for (int dir = 0; dir < 2; ++dir) {
        std::vector<int> lev(nc, 0);
        int nlev = 0;
        for (int p = 0; p < nc; ++p) {
            const int i = order[dir == 0 ? p : nc - 1 - p];
            int l = 0;
            for (int k = c->h_cf_ptr[i]; k < c->h_cf_ptr[i + 1]; ++k) {
                const int f = c->h_cf_idx[k];
                if (f >= nif) continue;
                const int g = c->h_owner[f] == i ? c->h_nbr[f] : c->h_owner[f];
                if (dir == 0 ? rank[g] < rank[i] : rank[g] > rank[i]) l = std::max(l, lev[g] + 1);
            }
            lev[i] = l;
            nlev = std::max(nlev, l + 1);
        }
        std::vector<int> ptr(nlev + 1, 0);
        for (int i = 0; i < nc; ++i) ptr[lev[i] + 1]++;
        for (int l = 0; l < nlev; ++l) ptr[l + 1] += ptr[l];
        std::vector<int> cells(nc), fill(ptr.begin(), ptr.end() - 1);
        for (int p = 0; p < nc; ++p) {   // within a level, in sweep order
            const int i = order[dir == 0 ? p : nc - 1 - p];
            cells[fill[lev[i]]++] = i;
        }
        // per slot: {cell, pair count, overflow offset, 1} and its first four
        // (neighbour, face) pairs toward earlier (later) cells, ascending;
        // a level's last unit of 16 is filled with copies of its first slot,
        // {.., 0}
        std::vector<int4> rec;
        rec.reserve(3 * ((size_t)nc + 16 * (size_t)nlev));
        std::vector<int2> ovf;
        for (int l = 0; l < nlev; ++l) {
            for (int t = ptr[l]; t < ptr[l + 1]; ++t) {
                const int i = cells[t];
                int np = 0;
                int2 q[4] = {};
                const int off = (int)ovf.size();
                for (int k = c->h_cf_ptr[i]; k < c->h_cf_ptr[i + 1]; ++k) {
                    const int f = c->h_cf_idx[k];
                    if (f >= nif) continue;
                    const bool own = c->h_owner[f] == i;
                    const int g = own ? c->h_nbr[f] : c->h_owner[f];
                    if (!(dir == 0 ? rank[g] < rank[i] : rank[g] > rank[i])) continue;
                    const int2 pq = make_int2(g, own ? f : ~f);
                    if (np < 4) q[np] = pq;
                    else ovf.push_back(pq);
                    ++np;
                }
                rec.push_back(make_int4(i, np, off, 1));
                rec.push_back(make_int4(q[0].x, q[0].y, q[1].x, q[1].y));
                rec.push_back(make_int4(q[2].x, q[2].y, q[3].x, q[3].y));
            }
            while (rec.size() % 48) {
                const size_t first = rec.size() / 48 * 48;
                for (int k = 0; k < 3; ++k) {
                    int4 r = rec[first + k];
                    if (k == 0) r.w = 0;
                    rec.push_back(r);
                }
            }
        }
        if (ovf.empty()) ovf.push_back(make_int2(0, 0));
        c->ls_slots[dir].upload(rec, c->stream);
        c->ls_ovf[dir].upload(ovf, c->stream);
        SEMO_HIP(hipStreamSynchronize(c->stream));   // rec and ovf are temporaries
    }
    c->ls_ready = true;
}

template <int NSP>
void linsol_run(semo_ctx* c, int method, double time_step, const double* st, double* res) {
    constexpr int N = 4 + NSP, K = 12 + 3 * NSP;
    const int n = c->nc;
    dim3 g(nblk(n)), b(TPB);
    if (method == SEMO_LINSOL_POINT) {
        SEMO_LAUNCH(c, "linsol_point", (double)n * (K + 2 * N) * 8.0, (k_linsol_point<NSP, false>), g, b, n, st,
                    time_step, res);
        return;
    }
    if (method == SEMO_LINSOL_SINGLE) {
        SEMO_LAUNCH(c, "linsol_single", (double)n * (K + 2 * N) * 8.0, (k_linsol_point<NSP, true>), g, b, n, st,
                    time_step, res);
        return;
    }
    lusgs_schedule(c);
    c->ls_dinv.ensure((size_t)N * N * 64 * ((n + 63) / 64));
    const double sides = (double)c->h_cf_idx.size();
    SEMO_LAUNCH(c, "lusgs_diag", (double)n * (K + N * N + 3) * 8.0 + sides * (4.0 + 8.0 + 32.0 + K * 8.0),
                k_lusgs_diag<NSP>, g, b, n, c->nif, c->d_cf_ptr.p, c->d_cf_idx.p, c->d_owner.p, c->d_nbr.p,
                c->f_nrm.p, c->f_area.p, c->c_vol.p, st, time_step, c->ls_dinv.p);
    // forward results, backward results; tickets and error word
    const size_t nv = (size_t)N * n;
    c->ls_out.ensure(2 * nv);
    c->ls_ctl.ensure(LS_CTL);
    SEMO_LAUNCH(c, "lusgs_empty", 16.0 * nv, k_lusgs_empty, dim3(nblk(std::max(2 * (long)nv, (long)LS_CTL))), b, 2 * nv,
                reinterpret_cast<unsigned long long*>(c->ls_out.p), c->ls_ctl.p);
    // per cell: record, Dinv, own residual read + write, slot record; per
    // earlier (later) neighbour: its record and residual, the face's normal
    // and area (half the sides)
    const double bytes = (double)n * ((K + N * N + 2 * N + 1) * 8.0 + 48.0) + 0.5 * sides * ((K + N) * 8.0 + 40.0);
    for (int dir = 0; dir < 2; ++dir) {
        const int nu = (int)(c->ls_slots[dir].n / 48);
        // more wavefronts than can be resident only wait for a slot
        const dim3 gu(std::min(nblk(64L * nu), LS_BLOCKS));
        if (dir == 0)
            SEMO_LAUNCH(c, "lusgs_sweep", bytes, (k_lusgs_sweep<NSP, true>), gu, b, nu, c->ls_slots[0].p,
                        c->ls_ovf[0].p, c->f_nrm.p, c->f_area.p, c->c_vol.p, st, c->ls_dinv.p,
                        (const double*)res, c->ls_out.p, (double*)nullptr, c->ls_ctl.p);
        else
            SEMO_LAUNCH(c, "lusgs_sweep", bytes, (k_lusgs_sweep<NSP, false>), gu, b, nu, c->ls_slots[1].p,
                        c->ls_ovf[1].p, c->f_nrm.p, c->f_area.p, c->c_vol.p, st, c->ls_dinv.p,
                        (const double*)c->ls_out.p, c->ls_out.p + nv, res, c->ls_ctl.p);
    }
    int err = 0;
    SEMO_HIP(hipMemcpyAsync(&err, c->ls_ctl.p + LS_ERR, sizeof(int), hipMemcpyDeviceToHost, c->stream));
    SEMO_HIP(hipStreamSynchronize(c->stream));
    SEMO_CHECK(err == 0, SEMO_EHIP, "LU-SGS sweep: a neighbour's update did not arrive");
}

// updateValues (src/solvers/densityBased.cpp:366-512), per cell: the
// under-relaxed increments of P, U, V, W, T and the first nsp - 1 mass
// fractions, the limits (P, U, V, W, T: a value at or beyond a bound takes
// it), the mass fractions clipped to [0, 1] and the last one closing the sum.
// cells[n][5 + nsp] = (P, U, V, W, T, MF_0..MF_{nsp-1}); lim = (minP, maxP,
// minU, maxU, minV, maxV, minW, maxW, minT, maxT).
__global__ __launch_bounds__(TPB) void k_update_cells(int n, int nsp, double uP, double uU, double uT, double uMF,
                                                      const double* __restrict__ lim, const double* __restrict__ res,
                                                      double* __restrict__ cells) {
    const int i = xcd_block() * TPB + (int)threadIdx.x;
    if (i >= n) return;
    const int N = 4 + nsp, K = 5 + nsp;
    double* c = cells + (size_t)i * K;
    const double* r = res + (size_t)i * N;
    double v[5] = {c[0] + uP * r[0], c[1] + uU * r[1], c[2] + uU * r[2], c[3] + uU * r[3], c[4] + uT * r[4]};
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        if (v[k] <= lim[2 * k]) v[k] = lim[2 * k];
        if (v[k] >= lim[2 * k + 1]) v[k] = lim[2 * k + 1];
        c[k] = v[k];
    }
    double tmp = 0.0;
    for (int a = 0; a < nsp - 1; ++a) {
        double y = c[5 + a] + uMF * r[5 + a];
        y = y < 1.0 ? y : 1.0;      // std::min(1.0, y): (y < 1) ? y : 1
        y = 0.0 < y ? y : 0.0;      // std::max(0.0, y): (0 < y) ? y : 0
        c[5 + a] = y;
        tmp += y;
    }
    c[5 + nsp - 1] = 1.0 - tmp;
}

// per internal face: Un += URF_U * (wC r_own + (1 - wC) r_ngb) . n over the
// momentum increments, in the caller's orientation (a face the renumbering
// flipped takes the other side's weight and the negated normal)
__global__ __launch_bounds__(TPB) void k_update_un(int nif, int nsp, double uU, const int* __restrict__ owner,
                                                   const int* __restrict__ nbr, const int8_t* __restrict__ flip,
                                                   const double* __restrict__ wC, const double* __restrict__ nrm,
                                                   const double* __restrict__ res, double* __restrict__ un) {
    const int f = xcd_block() * TPB + (int)threadIdx.x;
    if (f >= nif) return;
    const int N = 4 + nsp;
    const bool fl = flip[f] != 0;
    const int o = fl ? nbr[f] : owner[f], g = fl ? owner[f] : nbr[f];
    const double wCL = fl ? 1.0 - wC[f] : wC[f], wCR = 1.0 - wCL;
    double n[3];
    for (int a = 0; a < 3; ++a) n[a] = fl ? -nrm[3 * (size_t)f + a] : nrm[3 * (size_t)f + a];
    const double* ro = res + (size_t)o * N;
    const double* rg = res + (size_t)g * N;
    un[f] += uU * ((wCL * ro[1] + wCR * rg[1]) * n[0] + (wCL * ro[2] + wCR * rg[2]) * n[1] +
                   (wCL * ro[3] + wCR * rg[3]) * n[2]);
}

}  // namespace

void update_values_device(semo_ctx* c, int nsp, const double* urf, const double* d_lim, const double* res,
                          double* cells, double* un) {
    const int N = 4 + nsp;
    SEMO_LAUNCH(c, "update_cells", (double)c->nc * (2.0 * (5 + nsp) + N) * 8.0, k_update_cells,
                dim3(nblk(c->nc)), dim3(TPB), c->nc, nsp, urf[0], urf[1], urf[2], urf[3], d_lim, res, cells);
    if (c->nif)
        SEMO_LAUNCH(c, "update_un", (double)c->nif * (8.0 + 1.0 + 8.0 + 24.0 + 16.0) + 6.0 * 8.0 * c->nif,
                    k_update_un, dim3(nblk(c->nif)), dim3(TPB), c->nif, nsp, urf[1], c->d_owner.p, c->d_nbr.p,
                    c->d_fflip.p, c->f_wC.p, c->f_nrm.p, res, un);
}

void linsol_device(semo_ctx* c, int method, int nsp, double time_step, const double* st, double* res) {
    switch (nsp) {
    case 1: linsol_run<1>(c, method, time_step, st, res); break;
    case 2: linsol_run<2>(c, method, time_step, st, res); break;
    case 3: linsol_run<3>(c, method, time_step, st, res); break;
    case 4: linsol_run<4>(c, method, time_step, st, res); break;
    default: SEMO_CHECK(false, SEMO_EINVAL, "linear solver: 1 <= nsp <= 4");
    }
}

}  // namespace semo
