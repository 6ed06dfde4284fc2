// Block-coupled pressure-velocity solve: one 4x4 block per cell pair (BSR4).
//
// SEMO's calcCoupledEq (src/solvers/eqCoupled.cpp:12-1250) is commented out in
// the reference: only its design survives -- four unknowns per cell
// (p', u', v', w'), B_n = 4 (eqCoupled.cpp:26), global index
// startCellGlobal*B_n + n*var + i, i.e. variable-major (eqCoupled.cpp:249-305),
// a continuity row with the p' Laplacian and momentum rows with upwind
// convection plus the face-interpolated p' gradient (eqCoupled.cpp:470-640),
// one solveAMGCL call (:1246).  This file builds that system from the live
// assembly of this library, so its blocks are exactly:
//   momentum rows (k = 1..3): the momentum matrix of calcMomentumEqs on the
//     (k, k) entries, plus the linearised pressure force: for a face f with
//     owner P and neighbour N, row P gets +n_k A (wC p'_P + (1-wC) p'_N), row
//     N the opposite; a zeroGradient-p boundary face adds n_k A p'_P;
//   continuity row (0): the pressure-correction matrix of calcPressureEq on
//     (0, 0), plus the face flux of the velocity correction,
//     +A (wC n.u'_P + (1-wC) n.u'_N) in row P and the opposite in row N
//     (zeroGradient / outflowing inletOutlet boundary faces add A n.u'_P);
//   right-hand sides: the momentum and pressure right-hand sides.
// The solution updates p += urf_p p', U += urf_u u'.  At a converged outer
// iteration both right-hand sides vanish, so the coupled and the segregated
// (SIMPLE) iterations share their fixed point.
//
// Storage (device numbering): of an off-diagonal block's 16 entries eight are
// zero and the others are five numbers -- the pressure-matrix entry (0, 0), the
// momentum-matrix entry (1..3, 1..3) and one coupling per component, the same
// in (0, k) and (k, 0) -- kept as five arrays over the slots of the scalar
// pattern (sliced ELL, entry pairs); a diagonal block is its two scalar
// diagonals and six couplings.  Vectors interleaved [n][4] = (p, u, v, w).
// Solver: FP64 BiCGStab, right-preconditioned by a SIMPLE-type block
// factorisation whose Schur-complement step is one FP32 V-cycle of the scalar
// pressure hierarchy (see precond below).
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdlib>

#include "kern.hpp"

namespace semo {

struct Coupled {
    bool built = false;
    int n = 0;
    int64_t nnzb = 0;                           // off-diagonal blocks
    DBuf<double> rhs;                           // [n][4]
    // the blocks, FP64: momentum / pressure entries and couplings per slot
    // (mval, pval [nv], gval [3][nv]; padding slots of gval hold 0), the
    // diagonal blocks' scalar entries and their couplings (0, 1..3), (1..3, 0)
    // (dval [6][n])
    DBuf<double> mval, mdiag, mrhs, pval, pdiag, prhs, gval, dval;
    DBuf<double> x;                             // [n][4] last solution
    // the couplings the preconditioner reads, FP32 (gval and dval rounded:
    // gc [3][nv], dd [6][n]) and im [n] = 1 / diag(M)
    DBuf<float> gc, dd;
    DBuf<double> im;
    DBuf<double> kv;                            // Krylov vectors
    DBuf<double> tp, zp;                        // Schur-complement right side / solution [n]
    DBuf<double> red, sc;                       // reduction partials, scalars
    GraphCache graphs;                          // a captured BiCGStab iteration
    int last_iters = 0;
    double last_relres = 0.0;
};

void coupled_free(Coupled* p) { delete p; }

namespace {

// ---------------------------------------------------------------- assembly --
// Forms the couplings and the right-hand side; the scalar entries are the two
// assembled systems' own arrays.  (Writing 16-value blocks instead took 665 us
// on 1.05M cells, 1.0 GB of stores; the couplings alone 233 us.)
__global__ void __launch_bounds__(TPB) k_cpl_row(
    int nc, int nif, const int* __restrict__ cf_sl, const int* __restrict__ cf_ell, const int* __restrict__ bpatch,
    const semo_patch_bc* __restrict__ bcs, const double* __restrict__ nrm, const double* __restrict__ area,
    const double* __restrict__ wCv, const int* __restrict__ slot_own, const int* __restrict__ slot_nbr,
    const double* __restrict__ mdiag, const double* __restrict__ mrhs, const double* __restrict__ prhs,
    const double* __restrict__ U, const double* __restrict__ V, const double* __restrict__ W,
    double* __restrict__ gval, double* __restrict__ dval, double* __restrict__ rhs, int64_t nv,
    float* __restrict__ gc, float* __restrict__ dd, double* __restrict__ im) {
    int i = xcd_block() * blockDim.x + threadIdx.x;
    if (i >= nc) return;
    double D[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};    // continuity row's u'_k, momentum rows' p'
    double uc[3] = {U[i], V[i], W[i]};
    CELL_FACES_BEGIN(i, cf_sl, cf_ell, f, own)
        const double* n = nrm + 3 * (size_t)f;
        double A = area[f];
        if (f < nif) {
            double wC = wCv[f];
            // no other face adds to this slot (one face per pair of cells)
            int slot = own ? slot_own[f] : slot_nbr[f];
            double wi = own ? wC : 1.0 - wC, wj = 1.0 - wi, sg = own ? 1.0 : -1.0;
            for (int k = 0; k < 3; ++k) {
                double g = sg * n[k] * A;
                D[k] += g * wi;
                D[3 + k] += g * wi;
                double gj = g * wj;
                gval[k * nv + slot] = gj;
                gc[k * nv + slot] = (float)gj;
            }
            continue;
        }
        semo_patch_bc bc = bcs[bpatch[f - nif]];
        if (bc.p_type != SEMO_BC_FIXED_VALUE)
            for (int k = 0; k < 3; ++k) D[3 + k] += n[k] * A;
        bool flux = bc.u_type == SEMO_BC_ZERO_GRADIENT ||
                    (bc.u_type == SEMO_BC_INLET_OUTLET && uc[0] * n[0] + uc[1] * n[1] + uc[2] * n[2] > 0.0);
        if (flux)
            for (int k = 0; k < 3; ++k) D[k] += n[k] * A;
    }
    size_t N = (size_t)nc;
    for (int k = 0; k < 6; ++k) {
        dval[k * N + i] = D[k];
        dd[k * N + i] = (float)D[k];
    }
    im[i] = 1.0 / mdiag[i];
    double2* Ro = reinterpret_cast<double2*>(rhs + 4 * (size_t)i);
    Ro[0] = make_double2(prhs[i], mrhs[i]);
    Ro[1] = make_double2(mrhs[N + i], mrhs[2 * N + i]);
}

// the columns of entries e, e + 1 (e even) of the scalar pattern, from
// int16 offsets column - row or from int32 columns
template <bool NARROW>
__device__ inline int2 pat_cols(const int* __restrict__ col, const int16_t* __restrict__ dcol, int e, int row) {
    if constexpr (NARROW) {
        int w = *reinterpret_cast<const int*>(dcol + e);
        return make_int2(row + (int)(int16_t)(w & 0xffff), row + (w >> 16));
    } else {
        return *reinterpret_cast<const int2*>(col + e);
    }
}

// ------------------------------------------------------------- block product --
// the block matrix as the product reads it
struct BlkMat {
    const int* __restrict__ sl_ptr;
    const int* __restrict__ col;
    const int16_t* __restrict__ dcol;
    const double* __restrict__ m;       // momentum entries per slot
    const double* __restrict__ p;       // pressure entries per slot
    const double* __restrict__ g;       // couplings [3][nv]
    const double* __restrict__ md;      // scalar diagonals
    const double* __restrict__ pd;
    const double* __restrict__ d;       // the diagonal blocks' couplings [6][n]
    int64_t nv;
};

// OP 0: y = A x;  OP 1: y = b - A x;  OP 2: y = A x with block partials of
// y.w, OP 3 also of y.y (the rows are in registers: 1.05M cells 79 us and 86 /
// 81 us with the dots, which cost 14 us each as passes of their own).  One lane per block row: a wavefront's
// load of each of the five value arrays is one contiguous 1 KB run, a
// neighbour costs one 32-byte gather.  Bound by HBM: 40 B per off-diagonal
// block and 128 B per row with the vectors, against 132 B and 192 B when full
// 16-value blocks were read (four lanes per row, block CSR): 1.05M cells
// 200 -> 79 us a product, 5.0 TB/s.  The omitted products are by exact zeros, and the
// rest are added in the same order.
template <int OP, bool NARROW>
__global__ void __launch_bounds__(TPB) k_blk(int n, BlkMat a, const double* __restrict__ x,
                                             const double* __restrict__ b, double* __restrict__ y,
                                             const double* __restrict__ w, double* __restrict__ part) {
    int row = xcd_block() * TPB + threadIdx.x;
    int s = row >> 6, lane = row & (SL - 1);
    bool in = s < (n + SL - 1) / SL;
    if constexpr (OP < 2) { if (!in) return; }
    double2 wa = make_double2(0.0, 0.0), wb = wa;
    if (OP >= 2 && row < n) {
        wa = *reinterpret_cast<const double2*>(w + 4 * (size_t)row);
        wb = *reinterpret_cast<const double2*>(w + 4 * (size_t)row + 2);
    }
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
    if (row < n) {
        size_t N = (size_t)n;
        double2 xa = *reinterpret_cast<const double2*>(x + 4 * (size_t)row);
        double2 xb = *reinterpret_cast<const double2*>(x + 4 * (size_t)row + 2);
        double dm = a.md[row];
        s0 = a.pd[row] * xa.x + a.d[row] * xa.y + a.d[N + row] * xb.x + a.d[2 * N + row] * xb.y;
        s1 = a.d[3 * N + row] * xa.x + dm * xa.y;
        s2 = a.d[4 * N + row] * xa.x + dm * xb.x;
        s3 = a.d[5 * N + row] * xa.x + dm * xb.y;
    }
    int end = in ? a.sl_ptr[s + 1] : 0;
    const double* g1 = a.g + a.nv;
    const double* g2 = g1 + a.nv;
    for (int e = in ? a.sl_ptr[s] + 2 * lane : 0; e < end; e += 2 * SL) {
        int2 j = pat_cols<NARROW>(a.col, a.dcol, e, row);
        double2 q = *reinterpret_cast<const double2*>(a.p + e);
        double2 m = *reinterpret_cast<const double2*>(a.m + e);
        double2 c0 = *reinterpret_cast<const double2*>(a.g + e);
        double2 c1 = *reinterpret_cast<const double2*>(g1 + e);
        double2 c2 = *reinterpret_cast<const double2*>(g2 + e);
        double2 u0 = *reinterpret_cast<const double2*>(x + 4 * (size_t)j.x);
        double2 u1 = *reinterpret_cast<const double2*>(x + 4 * (size_t)j.x + 2);
        double2 v0 = *reinterpret_cast<const double2*>(x + 4 * (size_t)j.y);
        double2 v1 = *reinterpret_cast<const double2*>(x + 4 * (size_t)j.y + 2);
        s0 += q.x * u0.x + c0.x * u0.y + c1.x * u1.x + c2.x * u1.y;
        s1 += c0.x * u0.x + m.x * u0.y;
        s2 += c1.x * u0.x + m.x * u1.x;
        s3 += c2.x * u0.x + m.x * u1.y;
        s0 += q.y * v0.x + c0.y * v0.y + c1.y * v1.x + c2.y * v1.y;
        s1 += c0.y * v0.x + m.y * v0.y;
        s2 += c1.y * v0.x + m.y * v1.x;
        s3 += c2.y * v0.x + m.y * v1.y;
    }
    if constexpr (OP < 2) { if (row >= n) return; }
    if constexpr (OP == 1) {
        double2 ba = *reinterpret_cast<const double2*>(b + 4 * (size_t)row);
        double2 bb = *reinterpret_cast<const double2*>(b + 4 * (size_t)row + 2);
        s0 = ba.x - s0; s1 = ba.y - s1; s2 = bb.x - s2; s3 = bb.y - s3;
    }
    if (OP < 2 || row < n) {
        *reinterpret_cast<double2*>(y + 4 * (size_t)row) = make_double2(s0, s1);
        *reinterpret_cast<double2*>(y + 4 * (size_t)row + 2) = make_double2(s2, s3);
    }
    if constexpr (OP >= 2) {
        double yw = 0.0, yy = 0.0;
        if (row < n) {
            yw = s0 * wa.x + s1 * wa.y + s2 * wb.x + s3 * wb.y;
            if (OP == 3) yy = s0 * s0 + s1 * s1 + s2 * s2 + s3 * s3;
        }
        block_sum2(yw, yy, part);
    }
}

// ------------------------------------------ SIMPLE-type block preconditioner --
// Block factorisation of K = [[Lp, D], [G, M]] (continuity row: the
// pressure-correction matrix Lp on p', the velocity-correction flux D on u';
// momentum rows: the pressure force G on p', the momentum matrix M on u'):
//   u* = diag(M)^-1 r_u;  p' = S^-1 (r_p - D u*);  u' = u* - diag(M)^-1 G p'
// with the Schur complement S = Lp - D diag(M)^-1 G replaced by Lp, applied
// as one FP32 V-cycle of the scalar pressure hierarchy.  (Scaling that
// approximation by 1.3, 1.6 or 2 -- the part D diag(M)^-1 G adds to smooth
// modes -- raised the BiCGStab iterations of the 1.05M-cell channel from
// 11.6 to 12.3, 14.1 and 15.2 per outer iteration.)
// The two kernels around the V-cycle walk the scalar pattern one lane per
// row (sliced ELL, entry pairs: the three coupling arrays and the columns
// are one 8-byte load per lane per pair, a wavefront's load one contiguous
// run); u* is formed where it is read (r_u 1/diag(M), the same product the
// correction forms), so no pass writes it.

constexpr int PC_PAIRS = 2;   // entry pairs per trip: their loads, then their gathers

// tp = r_p - D u*
template <bool NARROW>
__global__ void __launch_bounds__(TPB) k_sp_schur_rhs(int n, const int* __restrict__ sl_ptr,
                                                      const int* __restrict__ col, const int16_t* __restrict__ dcol,
                                                      const float* __restrict__ gc, int64_t nv,
                                                      const float* __restrict__ dd, const double* __restrict__ r,
                                                      const double* __restrict__ im, double* __restrict__ tp) {
    int row = xcd_block() * TPB + threadIdx.x;
    int s = row >> 6, lane = row & (SL - 1);
    if (s >= (n + SL - 1) / SL) return;
    double t = 0.0;
    if (row < n) {
        double2 r01 = *reinterpret_cast<const double2*>(r + 4 * (size_t)row);
        double2 r23 = *reinterpret_cast<const double2*>(r + 4 * (size_t)row + 2);
        double m = im[row];
        t = r01.x;
        t -= (double)dd[row] * (r01.y * m) + (double)dd[(size_t)n + row] * (r23.x * m) +
             (double)dd[2 * (size_t)n + row] * (r23.y * m);
    }
    int end = sl_ptr[s + 1];
    for (int e = sl_ptr[s] + 2 * lane; e < end; e += 2 * SL * PC_PAIRS) {
        int2 j[PC_PAIRS];
        float2 a0[PC_PAIRS], a1[PC_PAIRS], a2[PC_PAIRS];
#pragma unroll
        for (int u = 0; u < PC_PAIRS; ++u) {
            int ee = e + 2 * SL * u;
            if (ee < end) {
                j[u] = pat_cols<NARROW>(col, dcol, ee, row);
                a0[u] = *reinterpret_cast<const float2*>(gc + ee);
                a1[u] = *reinterpret_cast<const float2*>(gc + nv + ee);
                a2[u] = *reinterpret_cast<const float2*>(gc + 2 * nv + ee);
            } else {
                j[u] = make_int2(-1, -1);
            }
        }
        double2 x0[PC_PAIRS], x1[PC_PAIRS], y0[PC_PAIRS], y1[PC_PAIRS];
        double m0[PC_PAIRS], m1[PC_PAIRS];
#pragma unroll
        for (int u = 0; u < PC_PAIRS; ++u)
            if (j[u].x >= 0) {
                x0[u] = *reinterpret_cast<const double2*>(r + 4 * (size_t)j[u].x);
                x1[u] = *reinterpret_cast<const double2*>(r + 4 * (size_t)j[u].x + 2);
                y0[u] = *reinterpret_cast<const double2*>(r + 4 * (size_t)j[u].y);
                y1[u] = *reinterpret_cast<const double2*>(r + 4 * (size_t)j[u].y + 2);
                m0[u] = im[j[u].x];
                m1[u] = im[j[u].y];
            }
#pragma unroll
        for (int u = 0; u < PC_PAIRS; ++u)
            if (j[u].x >= 0) {
                t -= (double)a0[u].x * (x0[u].y * m0[u]) + (double)a1[u].x * (x1[u].x * m0[u]) +
                     (double)a2[u].x * (x1[u].y * m0[u]);
                t -= (double)a0[u].y * (y0[u].y * m1[u]) + (double)a1[u].y * (y1[u].x * m1[u]) +
                     (double)a2[u].y * (y1[u].y * m1[u]);
            }
    }
    if (row < n) tp[row] = t;
}
// z_p = p', z_u = u* - diag(M)^-1 G p'
template <bool NARROW>
__global__ void __launch_bounds__(TPB) k_sp_correct(int n, const int* __restrict__ sl_ptr,
                                                    const int* __restrict__ col, const int16_t* __restrict__ dcol,
                                                    const float* __restrict__ gc, int64_t nv,
                                                    const float* __restrict__ dd, const double* __restrict__ r,
                                                    const double* __restrict__ im, const double* __restrict__ zp,
                                                    double* __restrict__ z) {
    int row = xcd_block() * TPB + threadIdx.x;
    int s = row >> 6, lane = row & (SL - 1);
    if (s >= (n + SL - 1) / SL) return;
    double p = 0.0, g0 = 0.0, g1 = 0.0, g2 = 0.0;
    if (row < n) {
        p = zp[row];
        g0 = (double)dd[3 * (size_t)n + row] * p;
        g1 = (double)dd[4 * (size_t)n + row] * p;
        g2 = (double)dd[5 * (size_t)n + row] * p;
    }
    int end = sl_ptr[s + 1];
    for (int e = sl_ptr[s] + 2 * lane; e < end; e += 2 * SL * PC_PAIRS) {
        int2 j[PC_PAIRS];
        float2 a0[PC_PAIRS], a1[PC_PAIRS], a2[PC_PAIRS];
#pragma unroll
        for (int u = 0; u < PC_PAIRS; ++u) {
            int ee = e + 2 * SL * u;
            if (ee < end) {
                j[u] = pat_cols<NARROW>(col, dcol, ee, row);
                a0[u] = *reinterpret_cast<const float2*>(gc + ee);
                a1[u] = *reinterpret_cast<const float2*>(gc + nv + ee);
                a2[u] = *reinterpret_cast<const float2*>(gc + 2 * nv + ee);
            } else {
                j[u] = make_int2(-1, -1);
            }
        }
        double q0[PC_PAIRS], q1[PC_PAIRS];
#pragma unroll
        for (int u = 0; u < PC_PAIRS; ++u)
            if (j[u].x >= 0) { q0[u] = zp[j[u].x]; q1[u] = zp[j[u].y]; }
#pragma unroll
        for (int u = 0; u < PC_PAIRS; ++u)
            if (j[u].x >= 0) {
                g0 += (double)a0[u].x * q0[u]; g1 += (double)a1[u].x * q0[u]; g2 += (double)a2[u].x * q0[u];
                g0 += (double)a0[u].y * q1[u]; g1 += (double)a1[u].y * q1[u]; g2 += (double)a2[u].y * q1[u];
            }
    }
    if (row >= n) return;
    double m = im[row];
    double2 r01 = *reinterpret_cast<const double2*>(r + 4 * (size_t)row);
    double2 r23 = *reinterpret_cast<const double2*>(r + 4 * (size_t)row + 2);
    double* zi = z + 4 * (size_t)row;
    *reinterpret_cast<double2*>(zi) = make_double2(p, r01.y * m - g0 * m);
    *reinterpret_cast<double2*>(zi + 2) = make_double2(r23.x * m - g1 * m, r23.y * m - g2 * m);
}

// ----------------------------------------------------------- Krylov kernels --
// |a|^2, block partials (fixed order) in part[2b]
__global__ void __launch_bounds__(TPB) k_norm2(size_t n, const double* __restrict__ a, double* __restrict__ part) {
    size_t i = (size_t)xcd_block() * blockDim.x + threadIdx.x;
    double s = 0.0;
    for (size_t k = i; k < n; k += (size_t)gridDim.x * blockDim.x) s += a[k] * a[k];
    block_sum2(s, 0.0, part);
}

// P += urf_p x0, U += urf_u x(1..3), clipped; partial sums of |dx|^2 and |x_new|^2
__global__ void __launch_bounds__(TPB) k_cpl_update(int nc, double urf_p, double urf_u, double lim,
                                                    const double* __restrict__ x, double* __restrict__ P,
                                                    double* __restrict__ U, double* __restrict__ V,
                                                    double* __restrict__ W, double* __restrict__ part) {
    int i = xcd_block() * blockDim.x + threadIdx.x;
    double nd = 0.0, np = 0.0;
    if (i < nc) {
        const double* xi = x + 4 * (size_t)i;
        double* f[4] = {P, U, V, W};
        for (int q = 0; q < 4; ++q) {
            double d = (q == 0 ? urf_p : urf_u) * xi[q];
            double v = f[q][i] + d;
            if (v <= -lim) v = -lim;
            if (v >= lim) v = lim;
            f[q][i] = v;
            nd += d * d; np += v * v;
        }
    }
    block_sum2(nd, np, part);
}

// device scalars of the block BiCGStab (zero denominators give zero steps,
// so that an iteration issued past convergence leaves x unchanged)
enum { C_RHO = 0, C_ALPHA, C_OMEGA, C_BETA };
enum { F_START = 0, F_ALPHA, F_OMEGA, F_RR, F_RESTART };

constexpr int CTPB = 1024;
// the squared norms (|b|^2, |r|^2) also go to the host
__global__ void __launch_bounds__(CTPB) k_cfinish(int nb, const double* __restrict__ part, double* __restrict__ sc,
                                                  int what, Ring ring) {
    double a0 = 0.0, a1 = 0.0;
    for (int i = threadIdx.x; i < nb; i += CTPB) { a0 += part[2 * i]; a1 += part[2 * i + 1]; }
    __shared__ double sh[2][CTPB];
    sh[0][threadIdx.x] = a0; sh[1][threadIdx.x] = a1;
    __syncthreads();
    for (int w = CTPB / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) { sh[0][threadIdx.x] += sh[0][threadIdx.x + w]; sh[1][threadIdx.x] += sh[1][threadIdx.x + w]; }
        __syncthreads();
    }
    if (threadIdx.x != 0) return;
    double d0 = sh[0][0], d1 = sh[1][0];
    switch (what) {
    // a (re)start: rh = r, so rho = |r|^2, and p = r by beta = 0 (p = v = 0)
    case F_START:
    case F_RESTART: sc[C_RHO] = d0; sc[C_BETA] = 0.0; sc[C_OMEGA] = 1.0; break;
    case F_ALPHA: sc[C_ALPHA] = d0 != 0.0 ? sc[C_RHO] / d0 : 0.0; break;     // d0 = rh.v
    case F_OMEGA: sc[C_OMEGA] = d1 != 0.0 ? d0 / d1 : 0.0; break;            // d0 = t.s, d1 = t.t
    case F_RR:       // d0 = r.r, d1 = rh.r
        sc[C_BETA] = (sc[C_RHO] != 0.0 && sc[C_OMEGA] != 0.0) ? (d1 / sc[C_RHO]) * (sc[C_ALPHA] / sc[C_OMEGA]) : 0.0;
        sc[C_RHO] = d1;
        break;
    default: break;
    }
    if (what == F_START || what == F_RR) ring_put(ring, &d0, 1);
}

// p = r + beta (p - omega v)
__global__ void __launch_bounds__(TPB) k_cb_p(size_t n, const double* __restrict__ sc, const double* __restrict__ r,
                                              const double* __restrict__ v, double* __restrict__ p) {
    size_t i = (size_t)xcd_block() * blockDim.x + threadIdx.x;
    if (i >= n) return;
    p[i] = r[i] + sc[C_BETA] * (p[i] - sc[C_OMEGA] * v[i]);
}
// s = r - alpha v
__global__ void __launch_bounds__(TPB) k_cb_s(size_t n, const double* __restrict__ sc, const double* __restrict__ r,
                                              const double* __restrict__ v, double* __restrict__ s) {
    size_t i = (size_t)xcd_block() * blockDim.x + threadIdx.x;
    if (i >= n) return;
    s[i] = r[i] - sc[C_ALPHA] * v[i];
}
// x += alpha ph + omega sh; r = s - omega t; partials of r.r and of rh.r for
// the next direction (1.05M cells: 34 us without it, 41 with; a pass of its
// own 14 and one more finish)
__global__ void __launch_bounds__(TPB) k_cb_x(size_t n, const double* __restrict__ sc, const double* __restrict__ ph,
                                              const double* __restrict__ sh, const double* __restrict__ s,
                                              const double* __restrict__ t, const double* __restrict__ rh,
                                              double* __restrict__ x, double* __restrict__ r,
                                              double* __restrict__ part) {
    size_t i = (size_t)xcd_block() * blockDim.x + threadIdx.x;
    double rr = 0.0, hr = 0.0;
    if (i < n) {
        double a = sc[C_ALPHA], w = sc[C_OMEGA];
        x[i] += a * ph[i] + w * sh[i];
        double ri = s[i] - w * t[i];
        r[i] = ri;
        rr = ri * ri; hr = rh[i] * ri;
    }
    block_sum2(rr, hr, part);
}
// restart from the current x (r = b - A x already formed): rh = r,
// p = v = 0; partials of r.r
__global__ void __launch_bounds__(TPB) k_cb_restart(size_t n, const double* __restrict__ r, double* __restrict__ rh,
                                                    double* __restrict__ p, double* __restrict__ v,
                                                    double* __restrict__ part) {
    size_t i = (size_t)xcd_block() * blockDim.x + threadIdx.x;
    double rr = 0.0;
    if (i < n) {
        double ri = r[i];
        rh[i] = ri; p[i] = 0.0; v[i] = 0.0;
        rr = ri * ri;
    }
    block_sum2(rr, 0.0, part);
}
// r = rh = b, x = p = v = 0; partials of b.b
__global__ void __launch_bounds__(TPB) k_cb_init(size_t n, const double* __restrict__ b, double* __restrict__ x,
                                                 double* __restrict__ r, double* __restrict__ rh,
                                                 double* __restrict__ p, double* __restrict__ v,
                                                 double* __restrict__ part) {
    size_t i = (size_t)xcd_block() * blockDim.x + threadIdx.x;
    double bb = 0.0;
    if (i < n) {
        double bi = b[i];
        r[i] = bi; rh[i] = bi; x[i] = 0.0; p[i] = 0.0; v[i] = 0.0;
        bb = bi * bi;
    }
    block_sum2(bb, 0.0, part);
}

// --------------------------------------------------------------- host side --
int nb_of(size_t n) { return (int)std::min<size_t>((n + TPB - 1) / TPB, 2048); }


// z = P^-1 r with the SIMPLE-type factorisation (FP64 vectors, FP32
// couplings and pressure V-cycle); captured: the V-cycle's kernels one by one
void precond(semo_ctx* c, Coupled& C, const double* r, double* z, bool captured) {
    int n = C.n;
    const DevSell<double>& A = c->Amat;
    int64_t nv = (int64_t)c->pat.col.size();
    int nb = nblk((long)c->pat.nslices * SL);
    bool narrow = A.dcol.p != nullptr;
    double idx = narrow ? 2.0 : 4.0;
    if (narrow)
        SEMO_LAUNCH(c, "cpl_precond_schur_rhs", (idx + 12.0) * nv + 60.0 * n, k_sp_schur_rhs<true>, dim3(nb),
                    dim3(TPB), n, A.sl_ptr.p, A.col.p, A.dcol.p, C.gc.p, nv, C.dd.p, r, C.im.p, C.tp.p);
    else
        SEMO_LAUNCH(c, "cpl_precond_schur_rhs", (idx + 12.0) * nv + 60.0 * n, k_sp_schur_rhs<false>, dim3(nb),
                    dim3(TPB), n, A.sl_ptr.p, A.col.p, A.dcol.p, C.gc.p, nv, C.dd.p, r, C.im.p, C.tp.p);
    if (captured) pressure_vcycle_kernels(c, C.tp.p, C.zp.p, true);
    else pressure_vcycle(c, C.tp.p, C.zp.p, true);
    if (narrow)
        SEMO_LAUNCH(c, "cpl_precond_correct", (idx + 12.0) * nv + 84.0 * n, k_sp_correct<true>, dim3(nb),
                    dim3(TPB), n, A.sl_ptr.p, A.col.p, A.dcol.p, C.gc.p, nv, C.dd.p, r, C.im.p, C.zp.p, z);
    else
        SEMO_LAUNCH(c, "cpl_precond_correct", (idx + 12.0) * nv + 84.0 * n, k_sp_correct<false>, dim3(nb),
                    dim3(TPB), n, A.sl_ptr.p, A.col.p, A.dcol.p, C.gc.p, nv, C.dd.p, r, C.im.p, C.zp.p, z);
}

BlkMat blk_mat(semo_ctx* c, const Coupled& C) {
    const DevSell<double>& A = c->Amat;
    return BlkMat{A.sl_ptr.p, A.col.p, A.dcol.p, C.mval.p, C.pval.p, C.gval.p, C.mdiag.p, C.pdiag.p, C.dval.p,
                  (int64_t)c->pat.col.size()};
}
// y = A x (OP 0), y = b - A x (OP 1), y = A x with partials of y.w (OP 2) and
// also of y.y (OP 3)
template <int OP>
void blk_product(semo_ctx* c, Coupled& C, const double* x, const double* b, double* y, const char* tag,
                 const double* w = nullptr) {
    bool narrow = c->Amat.dcol.p != nullptr;
    double bytes = (40.0 + (narrow ? 2.0 : 4.0)) * C.nnzb + (64.0 + 64.0 + (OP ? 32.0 : 0.0)) * C.n;
    dim3 g(nblk((long)c->pat.nslices * SL)), t(TPB);
    BlkMat a = blk_mat(c, C);
    if (narrow) SEMO_LAUNCH(c, tag, bytes, (k_blk<OP, true>), g, t, C.n, a, x, b, y, w, C.red.p);
    else SEMO_LAUNCH(c, tag, bytes, (k_blk<OP, false>), g, t, C.n, a, x, b, y, w, C.red.p);
}
void spmv64(semo_ctx* c, Coupled& C, const double* x, double* y) {
    blk_product<0>(c, C, x, nullptr, y, "cpl_blk_spmv");
}

// work arrays (once per mesh)
void coupled_setup(semo_ctx* c, Coupled& C) {
    int n = c->nc;
    C.n = n;
    C.nnzb = 2 * (int64_t)c->nif;
    hipStream_t s = c->stream;
    size_t nv = std::max<size_t>(c->pat.col.size(), 1);
    C.rhs.alloc(4 * (size_t)n);
    C.x.alloc(4 * (size_t)n); C.x.zero(s);
    for (DBuf<double>* b : {&C.mval, &C.pval}) b->alloc(nv);
    for (DBuf<double>* b : {&C.mdiag, &C.pdiag, &C.prhs}) b->alloc(n);
    C.mrhs.alloc(3 * (size_t)n);
    C.kv.alloc(8 * 4 * (size_t)n);
    C.tp.alloc((size_t)n + 64); C.zp.alloc((size_t)n + 64);
    C.red.alloc(2 * (size_t)nblk(4 * (long)n) + 64);
    C.sc.alloc(16);
    C.gval.alloc(3 * nv); C.gval.zero(s);       // padding slots stay 0
    C.gc.alloc(3 * nv); C.gc.zero(s);
    C.dval.alloc(6 * (size_t)n); C.dd.alloc(6 * (size_t)n);
    C.im.alloc(n);
    SEMO_HIP(hipStreamSynchronize(s));
    C.built = true;
}

}  // namespace

// momentum + pressure assembly of the current state, then the block system
void assemble_coupled(semo_ctx* c) {
    for (const semo_patch_bc& b : c->bcs)
        SEMO_CHECK(b.p_type != SEMO_BC_SWITCH, SEMO_EINVAL_BC,
                   "coupled system: the Mach-switched pressure boundary has no block form here");
    if (!c->cpl) c->cpl = new Coupled();
    Coupled& C = *c->cpl;
    int n = c->nc;
    size_t nv = c->pat.col.size();
    assemble_pressure(c);
    if (!C.built) coupled_setup(c, C);
    // the Schur-complement preconditioner's hierarchy: built for the
    // pressure-correction operator, its finest level refreshed on the device
    // when the values change (the outer Krylov iteration sees the exact system)
    pressure_amg_update(c, [](const Amg&) { return true; });
    copy_d(c, C.pval.p, c->Amat.val.p, nv);
    copy_d(c, C.pdiag.p, c->Amat.diag.p, n);
    copy_d(c, C.prhs.p, c->Bvec.p, n);
    assemble_momentum(c);
    copy_d(c, C.mval.p, c->Amat.val.p, nv);
    copy_d(c, C.mdiag.p, c->Amat.diag.p, n);
    copy_d(c, C.mrhs.p, c->Bvec.p, 3 * (size_t)n);
    SEMO_LAUNCH(c, "cpl_assemble",
                cell_faces_bytes(c, 48.0) + (8.0 + 72.0) * c->nif + (24.0 + 8.0 + 32.0 + 72.0 + 8.0 + 32.0) * n,
                k_cpl_row, dim3(nblk(n)), dim3(TPB), n, c->nif, c->d_cf_sl.p, c->d_cf_ell.p, c->d_bpatch.p,
                c->d_bcs.p, c->f_nrm.p, c->f_area.p, c->f_wC.p, c->d_slot_own.p, c->d_slot_nbr.p, C.mdiag.p,
                C.mrhs.p, C.prhs.p, c->U.p, c->V.p, c->W.p, C.gval.p, C.dval.p, C.rhs.p, (int64_t)nv, C.gc.p, C.dd.p,
                C.im.p);
    c->last_eq = 3;
}

void coupled_spmv(semo_ctx* c, const double* x, double* y) {
    SEMO_CHECK(c->cpl && c->cpl->built, SEMO_ESTATE, "no coupled system assembled");
    spmv64(c, *c->cpl, x, y);
}

// right-preconditioned BiCGStab, x0 = 0, stop at ||b - A x|| <= tol ||b||.
// The Krylov scalars stay on the device; the host reads one residual per
// iteration, one iteration behind, so the stream never drains while it waits.
// An iteration's 12 kernels and two V-cycles are one graph.  Restarted from
// the current iterate (true residual, new shadow vector) when RESTART_AFTER
// iterations have not halved the smallest residual seen since the last
// (re)start: in transients the unrestarted iteration was seen to stall for
// hundreds of iterations.
constexpr int RESTART_AFTER = 30, MAX_RESUMES = 3;
void coupled_solve(semo_ctx* c, const double* b, double* x, semo_solve_stats* st) {
    SEMO_CHECK(c->cpl && c->cpl->built, SEMO_ESTATE, "no coupled system assembled");
    Coupled& C = *c->cpl;
    size_t N = 4 * (size_t)C.n;
    double* r = C.kv.p; double* rh = r + N; double* p = rh + N; double* v = p + N; double* ph = v + N;
    double* sv = ph + N; double* sh = sv + N; double* t = sh + N;
    double* sc = C.sc.p;
    int nbv = nblk((long)N);
    auto fin = [&](int nb, int what) {
        SEMO_LAUNCH(c, "cpl_finish", 16.0 * nb + 8.0, k_cfinish, dim3(1), dim3(CTPB), nb, C.red.p, sc, what,
                    ring_of(c));
    };
    int nbp = nblk((long)c->pat.nslices * SL);              // blocks of a product
    bool graph = c->graphs && !c->prof.on;
    auto record = [&] {                                     // one iteration, one ring word (|r|^2)
        SEMO_LAUNCH(c, "cpl_bicg_p", 32.0 * N, k_cb_p, dim3(nbv), dim3(TPB), N, sc, r, v, p);
        precond(c, C, p, ph, graph);
        blk_product<2>(c, C, ph, nullptr, v, "cpl_blk_spmv", rh);
        fin(nbp, F_ALPHA);
        SEMO_LAUNCH(c, "cpl_bicg_s", 24.0 * N, k_cb_s, dim3(nbv), dim3(TPB), N, sc, r, v, sv);
        precond(c, C, sv, sh, graph);
        blk_product<3>(c, C, sh, nullptr, t, "cpl_blk_spmv", sv);
        fin(nbp, F_OMEGA);
        SEMO_LAUNCH(c, "cpl_bicg_x", 64.0 * N, k_cb_x, dim3(nbv), dim3(TPB), N, sc, ph, sh, sv, t, rh, x, r, C.red.p);
        fin(nbv, F_RR);
    };
    int wb = ring_expect(c, 1);
    SEMO_LAUNCH(c, "cpl_bicg_init", 48.0 * N, k_cb_init, dim3(nbv), dim3(TPB), N, b, x, r, rh, p, v, C.red.p);
    fin(nbv, F_START);
    hipGraphExec_t exec = nullptr;
    if (graph) {
        std::vector<const void*> key = pressure_vcycle_signature(c, C.tp.p, C.zp.p, true);
        BlkMat a = blk_mat(c, C);
        for (const void* q : {(const void*)a.sl_ptr, (const void*)a.col, (const void*)a.dcol, (const void*)a.m,
                              (const void*)a.p, (const void*)a.g, (const void*)a.md, (const void*)a.pd,
                              (const void*)a.d, (const void*)C.gc.p, (const void*)C.dd.p, (const void*)C.im.p,
                              (const void*)C.kv.p, (const void*)x, (const void*)C.red.p, (const void*)sc,
                              (const void*)c->pin, (const void*)c->d_seq.p, reinterpret_cast<const void*>(N)})
            key.push_back(q);
        exec = C.graphs.get(c->stream, key, record);
    }
    // r = b - A x formed before: rh = r, p = v = 0, rho = |r|^2
    auto restart = [&] {
        SEMO_LAUNCH(c, "cpl_bicg_restart", 32.0 * N, k_cb_restart, dim3(nbv), dim3(TPB), N, r, rh, p, v, C.red.p);
        fin(nbv, F_RESTART);
    };
    int it = 0;
    double tol = c->sp.tol_u;
    ConvCheck cc(c, tol * tol, wb);
    double bb = 0.0, best = 0.0;
    C.last_relres = 0.0;
    for (int attempt = 0;; ++attempt) {
        int since = 0;
        for (++it; it <= c->sp.maxit_u; ++it) {
            int w = ring_expect(c, 1);
            if (graph) SEMO_HIP(hipGraphLaunch(exec, c->stream));
            else record();
            if (it == 1) {
                best = bb = cc.bb();
                if (!(bb > 0.0)) break;                      // b = 0, or not finite
            }
            if (cc.done(it, w)) break;
            if (cc.r1 < 0.25 * best) { best = cc.r1; since = 0; }       // squared residuals
            else if (++since >= RESTART_AFTER) {
                blk_product<1>(c, C, x, b, r, "cpl_blk_resid");
                restart();
                since = 0;
                best = cc.r1;
            }
        }
        if (!(bb > 0.0)) {
            zero_d(c, x, N * sizeof(double));                // 0 * z is NaN where the preconditioner overflows
            it = 0;
            break;
        }
        it = std::min(it, c->sp.maxit_u);
        // true residual
        blk_product<1>(c, C, x, b, r, "cpl_blk_resid");
        int nb = nb_of(N);
        SEMO_LAUNCH(c, "cpl_norm2", 8.0 * N, k_norm2, dim3(nb), dim3(TPB), N, r, C.red.p);
        double rr = sum_to_host(c, nb, C.red.p).x;
        C.last_relres = std::sqrt(rr) / std::sqrt(bb);
        // the recurrence can run ahead of the residual (seen where a flow has
        // become steady and the right-hand side is round-off): such a solve
        // goes on from its iterate
        if (!std::isfinite(rr) || C.last_relres <= solve_limit(tol) || it >= c->sp.maxit_u || attempt == MAX_RESUMES)
            break;
        restart();
        cc = ConvCheck(c, tol * tol * bb, rr);
        cc.read = it;
        best = rr;
    }
    C.last_iters = it;
    if (st) {
        *st = semo_solve_stats{};
        st->iters[0] = it;
        st->rel_res[0] = C.last_relres;
        st->n_levels = (int)c->amg_p.lv.size();
    }
    check_converged(bb > 0.0 ? C.last_relres : bb, c->sp.tol_u, "coupled");
}

void coupled_solve_assembled(semo_ctx* c, semo_solve_stats* st) {
    SEMO_CHECK(c->cpl && c->cpl->built, SEMO_ESTATE, "no coupled system assembled");
    coupled_solve(c, c->cpl->rhs.p, c->cpl->x.p, st);
}

double coupled_update(semo_ctx* c) {
    Coupled& C = *c->cpl;
    int nb = nblk(c->nc);
    SEMO_LAUNCH(c, "cpl_update", 96.0 * c->nc + 16.0 * nb, k_cpl_update, dim3(nb), dim3(TPB), c->nc, c->cs.urf_p,
                c->cs.urf_mom, c->cs.limit, C.x.p, c->P.p, c->U.p, c->V.p, c->W.p, c->red.p);
    double2 s = sum_to_host(c, nb, c->red.p);
    return s.y > 0.0 ? std::sqrt(s.x) / std::sqrt(s.y) : std::sqrt(s.x);
}

// block COO (diagonal blocks first, then row by row) and rhs, device numbering
void coupled_export(semo_ctx* c, std::vector<int>& rows, std::vector<int>& cols, std::vector<double>& blocks,
                    std::vector<double>& rhs) {
    SEMO_CHECK(c->cpl && c->cpl->built, SEMO_ESTATE, "no coupled system assembled");
    Coupled& C = *c->cpl;
    int n = C.n;
    size_t nv = c->pat.col.size(), N = (size_t)n;
    std::vector<double> mv(nv), pv(nv), gv(3 * nv), dv(6 * N), md(N), pd(N);
    rhs.resize(4 * N);
    C.mval.download(mv.data(), nv, c->stream); C.pval.download(pv.data(), nv, c->stream);
    C.gval.download(gv.data(), 3 * nv, c->stream); C.dval.download(dv.data(), 6 * N, c->stream);
    C.mdiag.download(md.data(), N, c->stream); C.pdiag.download(pd.data(), N, c->stream);
    C.rhs.download(rhs.data(), rhs.size(), c->stream);
    SEMO_HIP(hipStreamSynchronize(c->stream));
    rows.clear(); cols.clear();
    size_t nb = N + (size_t)C.nnzb;
    rows.reserve(nb); cols.reserve(nb);
    blocks.assign(16 * nb, 0.0);
    auto block = [&](int i, int j, double p, double m) {
        double* B = blocks.data() + 16 * rows.size();
        rows.push_back(i); cols.push_back(j);
        B[0] = p; B[5] = B[10] = B[15] = m;
        return B;
    };
    for (int i = 0; i < n; ++i) {
        double* B = block(i, i, pd[i], md[i]);
        for (int k = 0; k < 3; ++k) { B[1 + k] = dv[k * N + i]; B[4 * (1 + k)] = dv[(3 + k) * N + i]; }
    }
    for (int i = 0; i < n; ++i) {
        int base = c->pat.sl_ptr[i / SL], w = (c->pat.sl_ptr[i / SL + 1] - base) / SL;
        for (int q = 0; q < w; ++q) {
            int e = sell_pos(base, q, i % SL);
            if (c->pat.col[e] == i) break;                  // padding follows a row's last entry
            double* B = block(i, c->pat.col[e], pv[e], mv[e]);
            for (int k = 0; k < 3; ++k) B[1 + k] = B[4 * (1 + k)] = gv[k * nv + e];
        }
    }
}

}  // namespace semo
