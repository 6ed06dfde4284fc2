// Linear algebra and Krylov solvers on the device.
//
// * row kernels over two operator formats: sliced ELL (one lane per row,
//   coalesced val/col loads; short regular rows such as the fine-mesh
//   operator and the prolongation) and CSR with 4..64 lanes per row (long or
//   ragged rows: AMG restriction and Galerkin coarse operators);
// * fused Chebyshev steps (SpMV + residual/direction/iterate updates in one
//   pass) and a fused post-smoother start (A x, residual, first direction);
// * deterministic reductions fused into the kernels that produce their
//   operands: per-block partials in a fixed order, then one single-block
//   kernel sums them in a fixed order and computes the Krylov scalars, so
//   they never leave the GPU except for the convergence test.  (A
//   last-block-done scheme would need a device-scope release fence in every
//   block, i.e. an L2 write-back per block on this chip: measured ~0.3 ms per
//   launch at 2M rows, against ~5 us for the extra launch.)
// * AMG V-cycle with Chebyshev smoothing, smoothed-aggregation transfer
//   operators and a dense FP64 coarsest solve (explicit inverse, one GEMV);
// * flexible PCG for the pressure (FP64 AMG, or FP32 AMG inside the FP64
//   Krylov loop) and Jacobi-BiCGStab for momentum.
//
// Replaces the solve half of solveAMGCL (src/solvers/solveAMGCL.cpp:179-1271)
// and AMGCL's amg/idrs/fgmres (lib/amgcl/mpi/amg.hpp:342-380,
// lib/amgcl/solver/idrs.hpp, fgmres.hpp).
#include <chrono>
#include <cmath>
#include <limits>

#include "common.hpp"

namespace semo {

struct HCsr;
void amg_build_csr(semo_ctx* c, Amg& amg, int n, const std::vector<int>& ptr,
                   const std::vector<int>& col, const std::vector<double>& val);

namespace {

constexpr int TPB = 256;
constexpr int RB = 1024;   // grid of the grid-stride reductions
inline int nblk(long n) { return (int)((n + TPB - 1) / TPB); }
inline int rblk(long n) { return (int)std::min<long>(RB, std::max<long>(1, (n + TPB - 1) / TPB)); }

// ------------------------------------------------------------- reductions --
template <class T>
__device__ inline T wave_sum(T v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    return v;
}

// Sums the two per-thread values over the block in a fixed order and stores
// them as this block's partials part[2b], part[2b+1].  Every thread of the
// block must call it.
__device__ inline void block_partials(double (&v)[2], double* __restrict__ part) {
    __shared__ double sh[2][TPB / 64];
    v[0] = wave_sum(v[0]); v[1] = wave_sum(v[1]);
    if ((threadIdx.x & 63) == 0) { sh[0][threadIdx.x >> 6] = v[0]; sh[1][threadIdx.x >> 6] = v[1]; }
    __syncthreads();
    if (threadIdx.x == 0) {
        double t0 = 0.0, t1 = 0.0;
        for (int w = 0; w < TPB / 64; ++w) { t0 += sh[0][w]; t1 += sh[1][w]; }
        part[2 * blockIdx.x] = t0; part[2 * blockIdx.x + 1] = t1;
    }
}

// Krylov scalars in device memory (slots of c->scal)
enum { S_RZ = 0, S_ALPHA = 10, S_BETA = 11, S_OMEGA = 12,
       S_TT = 14, S_TS = 15, S_RHO = 16, S_AV = 20,
       S_RZ2 = 24, S_ALPHA2 = 26 };   // r.z and alpha of even / odd iterations (in-kernel totals)

// what the last block does with the totals d[0], d[1]
enum { W_NONE = 0,       // nothing is kept
       W_FCG_ALPHA,      // d0 = p.Ap:  alpha = rz / p.Ap
       W_FCG_BETA,       // d0 = r.z, d1 = z.Ap: Polak-Ribiere beta, rz = d0
       W_FCG_START,      // d0 = r.z of the first direction: rz = d0, beta = 0
       W_BICG_INIT,      // d0 = b.b: rho = b.b, beta = 0, alpha = omega = 1
       W_BICG_ALPHA,     // d0 = rh.v: alpha = rho / rh.v
       W_BICG_OMEGA,     // d0 = t.t, d1 = t.s: omega = t.s / t.t
       W_BICG_RHO };     // d0 = r.r, d1 = rh.r: beta = (rho'/rho)(alpha/omega), rho = rho'

__device__ inline double fcg_alpha(double rz, double pq) { return pq != 0.0 ? rz / pq : 0.0; }
__device__ inline double fcg_beta(double rz_old, double alpha, double zq) {
    return rz_old != 0.0 ? -alpha * zq / rz_old : 0.0;
}

__device__ void finish_scalars(int what, const double (&d)[2], double* s) {
    switch (what) {
    // zero denominators (an exactly solved system) give zero steps, so that
    // an iteration issued past convergence leaves x unchanged
    case W_FCG_ALPHA: s[S_ALPHA] = fcg_alpha(s[S_RZ], d[0]); break;
    // z.(r - r_old) = -alpha z.Ap, so r_old is not kept
    case W_FCG_BETA: s[S_BETA] = fcg_beta(s[S_RZ], s[S_ALPHA], d[1]); s[S_RZ] = d[0]; break;
    case W_FCG_START: s[S_BETA] = 0.0; s[S_RZ] = d[0]; break;
    case W_BICG_INIT:
        s[S_RHO] = d[0];
        s[S_BETA] = 0.0; s[S_ALPHA] = 1.0; s[S_OMEGA] = 1.0;
        break;
    case W_BICG_ALPHA: s[S_AV] = d[0]; s[S_ALPHA] = d[0] != 0.0 ? s[S_RHO] / d[0] : 0.0; break;
    case W_BICG_OMEGA: s[S_TT] = d[0]; s[S_TS] = d[1]; s[S_OMEGA] = d[0] != 0.0 ? d[1] / d[0] : 0.0; break;
    case W_BICG_RHO:
        s[S_BETA] = (s[S_RHO] != 0.0 && s[S_OMEGA] != 0.0) ? (d[1] / s[S_RHO]) * (s[S_ALPHA] / s[S_OMEGA]) : 0.0;
        s[S_RHO] = d[1];
        break;
    default: break;
    }
}

struct Red {                 // where a launch leaves its block partials
    double* part;
};

__device__ inline void reduce2(double (&v)[2], const Red& rd) { block_partials(v, rd.part); }

// ordered sum of nb partial pairs, then the scalar update `what`; one
// 1024-thread block, so each thread streams only a few partials
constexpr int FTPB = 1024;
// ring (optional): the host gets d0, and d1 where nput = 2
__global__ void __launch_bounds__(FTPB) k_finish(int nb, const double* __restrict__ part, double* __restrict__ s,
                                                 int what, Ring ring, int nput) {
    double a0 = 0.0, a1 = 0.0;
    const double2* p2 = reinterpret_cast<const double2*>(part);
    for (int i = threadIdx.x; i < nb; i += FTPB) { double2 v = p2[i]; a0 += v.x; a1 += v.y; }
    __shared__ double sh[2][FTPB];
    sh[0][threadIdx.x] = a0; sh[1][threadIdx.x] = a1;
    __syncthreads();
    for (int w = FTPB / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) {
            sh[0][threadIdx.x] += sh[0][threadIdx.x + w];
            sh[1][threadIdx.x] += sh[1][threadIdx.x + w];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        double d[2] = {sh[0][0], sh[1][0]};
        finish_scalars(what, d, s);
        ring_put(ring, d, nput);
    }
}

// the smallest of the partials' first values
__global__ void __launch_bounds__(FTPB) k_finish_min(int nb, const double* __restrict__ part, double start, Ring ring) {
    double m = start;
    for (int i = threadIdx.x; i < nb; i += FTPB) { double v = part[2 * (size_t)i]; m = v < m ? v : m; }
    __shared__ double sh[FTPB];
    sh[threadIdx.x] = m;
    __syncthreads();
    for (int w = FTPB / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w && sh[threadIdx.x + w] < sh[threadIdx.x]) sh[threadIdx.x] = sh[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) ring_put(ring, sh, 1);
}

// The totals of nb partial pairs, formed by every block of a kernel that needs
// them, in one order for all (256 threads each).  Up to TOTAL_MAX pairs this
// costs no more device time than k_finish before it and saves its launch: at
// 222650 cells (870 pairs) k_fcg_update takes 7.3 us with its own totals
// against 5.1 + 2.8 us, k_spmv_xpby 9.7 against 7.0 + 2.8 us.
constexpr int TOTAL_MAX = 1024;
__device__ inline double2 block_total(int nb, const double* __restrict__ part) {
    __shared__ double sh[2][TPB / 64];
    double a0 = 0.0, a1 = 0.0;
    const double2* p2 = reinterpret_cast<const double2*>(part);
    for (int i = threadIdx.x; i < nb; i += TPB) { double2 v = p2[i]; a0 += v.x; a1 += v.y; }
    a0 = wave_sum(a0); a1 = wave_sum(a1);
    if ((threadIdx.x & 63) == 0) { sh[0][threadIdx.x >> 6] = a0; sh[1][threadIdx.x >> 6] = a1; }
    __syncthreads();
    double2 t = make_double2(0.0, 0.0);
    for (int w = 0; w < TPB / 64; ++w) { t.x += sh[0][w]; t.y += sh[1][w]; }
    return t;
}

// a.b (+ c.d) over a grid-stride range
__global__ void __launch_bounds__(TPB) k_dot(int n, const double* __restrict__ a, const double* __restrict__ b,
                                             const double* __restrict__ cc, const double* __restrict__ d, Red rd) {
    double v[2] = {0.0, 0.0};
    for (int i = xcd_block() * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        v[0] += a[i] * b[i];
        if (cc) v[1] += cc[i] * d[i];
    }
    reduce2(v, rd);
}

// ------------------------------------------------------------ row kernels --
enum { OP_Y = 0,       // y = A x
       OP_RES = 1,     // y = b - A x
       OP_ADD = 2,     // y += A x
       OP_CHEB = 3,    // Chebyshev step: x = d_k, y = d_k+1, r -= D^-1 A d_k, xo += d_k+1
       OP_CHEBX = 4,   // Chebyshev start from x != 0: r = D^-1 (b - A x), y = r c1, xo = x + y
       OP_YPREP = 6 }; // y = A x and xo = c1 D^-1 y (restriction writing the next level's b and
                       // its degree-1 smoothed start, rounded as k_cheb_init forms it)

template <class T>
struct RowArgs {
    int n;
    const int* __restrict__ ptr;    // slice offsets (sliced ELL) or row offsets (CSR)
    const int* __restrict__ col;
    const int16_t* __restrict__ dcol;   // sliced ELL: column - row (null: use col)
    const T* __restrict__ val;
    const T* __restrict__ diag;     // null: no diagonal part
    const T* __restrict__ x;        // gathered operand
    const T* __restrict__ b;
    T* __restrict__ y;
    const T* __restrict__ dinv;
    T* __restrict__ r;
    T* __restrict__ xo;
    double* __restrict__ zo;        // optional FP64 copy of the new iterate
    T c1, c2;
};

// entries per trip of the row sums: 2 pairs on sliced-ELL slices (rows of
// ~6-7 entries), 8 per lane of the CSR kernels (coarse rows of 30-60 entries
// over avg/4 lanes; measured best of 1/2/4/8 on MI355X)
constexpr int SELL_PAIRS = 2, CSR_UNR = 8;
// One lane's sum over its row of a sliced-ELL slice, entries e0, e0 + 64, ...
// below e1, in entry order: acc += val[e] * opnd(col(e)).  U entries per
// trip: their indices and values are loaded first, then their gathers are
// issued together, so the gathers' latency is paid once per trip instead of
// once per entry.  The sum is the same as the one-entry loop's, bit for bit.
// (STRIDE 64; the CSR kernels use it with STRIDE = lanes per row.)
template <int U, int STRIDE, class T, class ColF, class OpF>
__device__ inline T sell_row_sum(int e0, int e1, const T* __restrict__ val, ColF colf, OpF opnd) {
    T acc = 0;
    for (int e = e0; e < e1; e += STRIDE * U) {
        int j[U];
        T v[U], x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            int ee = e + STRIDE * u;
            j[u] = ee < e1 ? colf(ee) : -1;
            v[u] = ee < e1 ? val[ee] : T(0);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) x[u] = j[u] >= 0 ? opnd(j[u]) : T(0);
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (j[u] >= 0) acc += v[u] * x[u];
    }
    return acc;
}

// One lane's sum over its row of a sliced-ELL slice (entry pairs, sell_pos):
// pair m of the row at base + 128 m + 2 lane, P pairs per trip, their values
// and columns loaded (one load each per pair) before their gathers are
// issued together.  acc += val * opnd(col) in entry order, bit for bit the
// sum of the one-entry loop.  colf2(e) gives the columns of entries e, e + 1.
template <int P, class T, class ColF2, class OpF>
__device__ inline T sell2_row_sum(int base, int end, int lane, const T* __restrict__ val, ColF2 colf2, OpF opnd) {
    using T2 = typename std::conditional<sizeof(T) == 8, double2, float2>::type;
    T acc = 0;
    for (int e = base + 2 * lane; e < end; e += 2 * SL * P) {
        int2 j[P];
        T2 v[P];
        T x0[P], x1[P];
#pragma unroll
        for (int u = 0; u < P; ++u) {
            int ee = e + 2 * SL * u;
            bool in = ee < end;
            j[u] = in ? colf2(ee) : make_int2(-1, -1);
            if (in) v[u] = *reinterpret_cast<const T2*>(val + ee);
        }
#pragma unroll
        for (int u = 0; u < P; ++u)
            if (j[u].x >= 0) { x0[u] = opnd(j[u].x); x1[u] = opnd(j[u].y); }
#pragma unroll
        for (int u = 0; u < P; ++u)
            if (j[u].x >= 0) { acc += v[u].x * x0[u]; acc += v[u].y * x1[u]; }
    }
    return acc;
}
// the two columns of entries e, e + 1 (e even) from int32 columns or from
// int16 offsets column - row
__device__ inline int2 sell2_col(const int* __restrict__ col, int e) {
    return *reinterpret_cast<const int2*>(col + e);
}
__device__ inline int2 sell2_dcol(const int16_t* __restrict__ dcol, int e, int row) {
    int w = *reinterpret_cast<const int*>(dcol + e);
    return make_int2(row + (int)(int16_t)(w & 0xffff), row + (w >> 16));
}

// G == 0: sliced ELL, one lane per row.  G > 0: CSR, G consecutive lanes per
// row, strided partial sums combined by a fixed shuffle tree (the result is
// deterministic for a given G).
// the row's own operands of the epilogue: diagonal and x (for the
// diagonal term, and x for the Chebyshev start), b (OP_ADD: y), D^-1
template <class T>
struct Own {
    T d, x, b, dv;
};
template <class T, int OP>
__device__ inline Own<T> load_own(const RowArgs<T>& a, int row) {
    Own<T> o{};
    if (a.diag) o.d = a.diag[row];
    if (a.diag || OP == OP_CHEBX || OP == OP_CHEB) o.x = a.x[row];
    if constexpr (OP == OP_RES || OP == OP_CHEBX) o.b = a.b[row];
    if constexpr (OP == OP_ADD) o.b = a.y[row];
    if constexpr (OP == OP_YPREP || OP == OP_CHEB || OP == OP_CHEBX) o.dv = a.dinv[row];
    return o;
}

template <class T, int G, int OP>
__global__ void __launch_bounds__(TPB) k_row(RowArgs<T> a) {
    int gid = xcd_block() * TPB + threadIdx.x;
    int row;
    T acc = 0;
    Own<T> own{};
    if constexpr (G == 0) {
        row = gid;
        int s = row >> 6, lane = row & 63;
        if (s >= ((a.n + 63) >> 6)) return;
        // the row's own operands are requested before the gathers
        if (row < a.n) own = load_own<T, OP>(a, row);
        auto opnd = [&](int j) { return a.x[j]; };
        if (a.dcol)
            acc = sell2_row_sum<SELL_PAIRS>(a.ptr[s], a.ptr[s + 1], lane, a.val,
                                            [&](int e) { return sell2_dcol(a.dcol, e, row); }, opnd);
        else
            acc = sell2_row_sum<SELL_PAIRS>(a.ptr[s], a.ptr[s + 1], lane, a.val,
                                            [&](int e) { return sell2_col(a.col, e); }, opnd);
        if (row >= a.n) return;
    } else {
        row = gid / G;
        int sub = gid & (G - 1);
        if (row >= a.n) return;
        // in flight during the gathers (128^3, 263552-row level, FP32: residual
        // 21.9 -> 20.6 us, smoothing step 17.1 -> 16.2; 8 lanes a row with four
        // entries a lane stays best: 4 lanes 26 us, 16 lanes 26 us)
        if (sub == 0) own = load_own<T, OP>(a, row);
        acc = sell_row_sum<CSR_UNR, G, T>(a.ptr[row] + sub, a.ptr[row + 1], a.val, [&](int e) { return a.col[e]; },
                                            [&](int j) { return a.x[j]; });
#pragma unroll
        for (int o = G / 2; o > 0; o >>= 1) acc += __shfl_down(acc, o, G);
        if (sub) return;
    }
    if (a.diag) acc += own.d * own.x;
    if constexpr (OP == OP_YPREP) {
        a.y[row] = acc;
        T rj = own.dv * acc;
        a.xo[row] = rj * a.c1;
    } else if constexpr (OP == OP_Y) {
        a.y[row] = acc;
    } else if constexpr (OP == OP_RES) {
        a.y[row] = own.b - acc;
    } else if constexpr (OP == OP_ADD) {
        a.y[row] = own.b + acc;
    } else if constexpr (OP == OP_CHEB) {
        T ri = a.r[row] - own.dv * acc;
        T di = a.c1 * own.x + a.c2 * ri;
        a.r[row] = ri; a.y[row] = di;
        T xn = a.xo[row] + di;
        a.xo[row] = xn;
        if (a.zo) a.zo[row] = (double)xn;
    } else {
        // r, y and xo may be null: a degree-1 smoother reads none of r and
        // y afterwards, and at the finest level only the FP64 copy zo
        T ri = own.dv * (own.b - acc);
        T di = ri * a.c1;
        if (a.r) a.r[row] = ri;
        if (a.y) a.y[row] = di;
        T xn = own.x + di;
        if (a.xo) a.xo[row] = xn;
        if (a.zo) a.zo[row] = (double)xn;
    }
}

template <class T, int OP>
void row_launch(semo_ctx* c, const DevSell<T>& A, RowArgs<T> a, const char* tag, double bytes) {
    if (A.n == 0) return;
    a.n = A.n; a.ptr = A.sl_ptr.p; a.col = A.col.p; a.val = A.val.p; a.diag = A.diag.p;
    a.dcol = (A.lanes == 0 && A.dcol.n) ? A.dcol.p : nullptr;
    ProfScope ps(c, tag, bytes);
    long rows = A.n;
    switch (A.lanes) {
    case 0: hipLaunchKernelGGL((k_row<T, 0, OP>), dim3(nblk((long)A.nslices * 64)), dim3(TPB), 0, c->stream, a); break;
    case 4: hipLaunchKernelGGL((k_row<T, 4, OP>), dim3(nblk(rows * 4)), dim3(TPB), 0, c->stream, a); break;
    case 8: hipLaunchKernelGGL((k_row<T, 8, OP>), dim3(nblk(rows * 8)), dim3(TPB), 0, c->stream, a); break;
    case 16: hipLaunchKernelGGL((k_row<T, 16, OP>), dim3(nblk(rows * 16)), dim3(TPB), 0, c->stream, a); break;
    case 32: hipLaunchKernelGGL((k_row<T, 32, OP>), dim3(nblk(rows * 32)), dim3(TPB), 0, c->stream, a); break;
    case 64: hipLaunchKernelGGL((k_row<T, 64, OP>), dim3(nblk(rows * 64)), dim3(TPB), 0, c->stream, a); break;
    default: throw Error(SEMO_EINVAL, "operator with an unsupported lane count");
    }
}

// algorithmic bytes of one pass over A: values + columns of the real
// entries, row/slice offsets, plus `vec` vector accesses of n entries
template <class T>
double op_bytes(const DevSell<T>& A, int vec) {
    double ptrs = A.lanes ? 4.0 * (A.n + 1) : 4.0 * (A.nslices + 1);
    double idx = (A.lanes == 0 && A.dcol.n) ? 2.0 : 4.0;
    double nd = A.diag.n ? (double)A.n : 0.0;          // diagonal entries: a value, no index
    return ((double)A.nnz - nd) * (sizeof(T) + idx) + nd * sizeof(T) + ptrs + (double)A.n * sizeof(T) * vec;
}

template <class T, int OP>
void spmv(semo_ctx* c, const DevSell<T>& A, const T* x, const T* b, T* y, const char* tag) {
    RowArgs<T> a{};
    a.x = x; a.b = b; a.y = y;
    row_launch<T, OP>(c, A, a, tag, op_bytes(A, OP == OP_Y ? 2 : 3));
}

// y = A x (sliced ELL, FP64) with d0 = (a0 ? a0 : y).y and d1 = a1.y
__global__ void __launch_bounds__(TPB) k_spmv_dot(int n, const int* __restrict__ sl_ptr, const int* __restrict__ col,
                                                  const int16_t* __restrict__ dcol,
                                                  const double* __restrict__ val, const double* __restrict__ diag,
                                                  const double* __restrict__ x, double* __restrict__ y,
                                                  const double* __restrict__ a0, const double* __restrict__ a1, Red rd) {
    int row = xcd_block() * blockDim.x + threadIdx.x;
    int s = row >> 6, lane = row & 63;
    double v[2] = {0.0, 0.0};
    if (s < ((n + 63) >> 6)) {
        bool own = row < n;     // the row's own operands before the gathers
        double dr = own ? diag[row] : 0.0, xr = own ? x[row] : 0.0;
        auto opnd = [&](int j) { return x[j]; };
        double acc = dcol ? sell2_row_sum<SELL_PAIRS>(sl_ptr[s], sl_ptr[s + 1], lane, val,
                                                      [&](int e) { return sell2_dcol(dcol, e, row); }, opnd)
                          : sell2_row_sum<SELL_PAIRS>(sl_ptr[s], sl_ptr[s + 1], lane, val,
                                                      [&](int e) { return sell2_col(col, e); }, opnd);
        if (own) {
            acc += dr * xr;
            y[row] = acc;
            v[0] = (a0 ? a0[row] : acc) * acc;
            if (a1) v[1] = a1[row] * acc;
        }
    }
    reduce2(v, rd);
}

// Where an FCG kernel finds a scalar it needs: nb > 0 -- it forms the totals
// of the partials itself (block_total) and one thread keeps what the next
// kernels need in the slots of this iteration's parity; nb == 0 -- k_finish
// left it in its slot.
struct FcgIn {
    const double* __restrict__ part;
    int nb, par, first;
};

// FCG direction update fused into its product: pn = z + beta po, q = A pn,
// partials pn.q; the first direction is z.  po and pn are distinct buffers:
// neighbours read po while the row writes pn.  z comes as the V-cycle left
// it: FP32 (TZ = float) from an FP32 one.
template <class TZ>
__global__ void __launch_bounds__(TPB) k_spmv_xpby(int n, const int* __restrict__ sl_ptr,
                                                   const int* __restrict__ col, const int16_t* __restrict__ dcol,
                                                   const double* __restrict__ val, const double* __restrict__ diag,
                                                   double* __restrict__ s, FcgIn in, const TZ* __restrict__ z,
                                                   const double* __restrict__ po, double* __restrict__ pn,
                                                   double* __restrict__ q, Red rd) {
    int row = xcd_block() * blockDim.x + threadIdx.x;
    int sl = row >> 6, lane = row & 63;
    double v[2] = {0.0, 0.0};
    double beta = 0.0;
    if (in.nb) {
        double2 t = block_total(in.nb, in.part);                  // r.z, z.Ap_old
        if (!in.first) beta = fcg_beta(s[S_RZ2 + (in.par ^ 1)], s[S_ALPHA2 + (in.par ^ 1)], t.y);
        if (blockIdx.x == 0 && threadIdx.x == 0) s[S_RZ2 + in.par] = t.x;
    } else if (!in.first) {
        beta = s[S_BETA];
    }
    if (sl < ((n + 63) >> 6)) {
        // the row's own operands are requested before the gathers
        bool own = row < n;
        double zr = own ? (double)z[row] : 0.0, dr = own ? diag[row] : 0.0;
        double por = own && !in.first ? po[row] : 0.0;
        auto sum = [&](auto opnd) {
            return dcol ? sell2_row_sum<SELL_PAIRS>(sl_ptr[sl], sl_ptr[sl + 1], lane, val,
                                                    [&](int e) { return sell2_dcol(dcol, e, row); }, opnd)
                        : sell2_row_sum<SELL_PAIRS>(sl_ptr[sl], sl_ptr[sl + 1], lane, val,
                                                    [&](int e) { return sell2_col(col, e); }, opnd);
        };
        double acc = in.first ? sum([&](int j) { return (double)z[j]; })
                              : sum([&](int j) { return (double)z[j] + beta * po[j]; });
        if (own) {
            double pr = in.first ? zr : zr + beta * por;
            pn[row] = pr;
            acc += dr * pr;
            q[row] = acc;
            v[0] = pr * acc;
        }
    }
    reduce2(v, rd);
}

// the V-cycle's last step at the finest level, x + c1 D^-1 (b - A x) into z
// (its own precision), with the dots the next direction needs: r.z and z.q
template <class T>
__global__ void __launch_bounds__(TPB) k_chebx_dot(RowArgs<T> a, const double* __restrict__ r,
                                                   const double* __restrict__ q, Red rd) {
    int row = xcd_block() * TPB + threadIdx.x;
    int s = row >> 6, lane = row & 63;
    double v[2] = {0.0, 0.0};
    if (s < ((a.n + 63) >> 6)) {
        Own<T> own{};
        double ri = 0.0, qi = 0.0;
        if (row < a.n) {
            own = load_own<T, OP_CHEBX>(a, row);
            ri = r[row]; qi = q[row];
        }
        auto opnd = [&](int j) { return a.x[j]; };
        T acc = a.dcol ? sell2_row_sum<SELL_PAIRS>(a.ptr[s], a.ptr[s + 1], lane, a.val,
                                                   [&](int e) { return sell2_dcol(a.dcol, e, row); }, opnd)
                       : sell2_row_sum<SELL_PAIRS>(a.ptr[s], a.ptr[s + 1], lane, a.val,
                                                   [&](int e) { return sell2_col(a.col, e); }, opnd);
        if (row < a.n) {
            acc += own.d * own.x;
            T res = own.dv * (own.b - acc);
            T di = res * a.c1;
            T xn = own.x + di;
            a.xo[row] = xn;
            v[0] = ri * (double)xn; v[1] = qi * (double)xn;
        }
    }
    reduce2(v, rd);
}

// |b - A x|^2 (sliced ELL, FP64), the residual itself not stored
__global__ void __launch_bounds__(TPB) k_resid_norm(int n, const int* __restrict__ sl_ptr, const int* __restrict__ col,
                                                    const int16_t* __restrict__ dcol, const double* __restrict__ val,
                                                    const double* __restrict__ diag, const double* __restrict__ x,
                                                    const double* __restrict__ b, Red rd) {
    int row = xcd_block() * blockDim.x + threadIdx.x;
    int s = row >> 6, lane = row & 63;
    double v[2] = {0.0, 0.0};
    if (s < ((n + 63) >> 6)) {
        bool own = row < n;
        double dr = own ? diag[row] : 0.0, xr = own ? x[row] : 0.0, br = own ? b[row] : 0.0;
        auto opnd = [&](int j) { return x[j]; };
        double acc = dcol ? sell2_row_sum<SELL_PAIRS>(sl_ptr[s], sl_ptr[s + 1], lane, val,
                                                      [&](int e) { return sell2_dcol(dcol, e, row); }, opnd)
                          : sell2_row_sum<SELL_PAIRS>(sl_ptr[s], sl_ptr[s + 1], lane, val,
                                                      [&](int e) { return sell2_col(col, e); }, opnd);
        if (own) {
            acc += dr * xr;
            double t = br - acc;
            v[0] = t * t;
        }
    }
    reduce2(v, rd);
}

// ------------------------------------------------------- Krylov vectors --
// Level-0 input of the next FP32 V-cycle, written by the kernel that
// produces the residual r (null b32: not used): b32 = (float) r and the
// degree-1 smoothed start x32 = c1 D^-1 b32, rounded as the V-cycle's own
// fused smoothing step forms them.
// (b64 / x64: the same for an FP64 V-cycle.)
struct Prep {
    float* __restrict__ b32;
    float* __restrict__ x32;
    const float* __restrict__ dinv32;
    float c1;
    double* __restrict__ b64;
    double* __restrict__ x64;
    const double* __restrict__ dinv64;
    double c1d;
};
__device__ inline void prep_store(const Prep& pp, int i, double ri) {
    if (pp.b32) {
        float bf = (float)ri;
        pp.b32[i] = bf;
        float rj = pp.dinv32[i] * bf;
        pp.x32[i] = rj * pp.c1;
    } else if (pp.b64) {
        pp.b64[i] = ri;
        double rj = pp.dinv64[i] * ri;
        pp.x64[i] = rj * pp.c1d;
    }
}

// r = b, d0 = b.b
__global__ void __launch_bounds__(TPB) k_fcg_init(int n, const double* __restrict__ b, double* __restrict__ r, Red rd,
                                                  Prep pp) {
    int i = xcd_block() * blockDim.x + threadIdx.x;
    double v[2] = {0.0, 0.0};
    if (i < n) { double bi = b[i]; r[i] = bi; v[0] = bi * bi; prep_store(pp, i, bi); }
    reduce2(v, rd);
}

// x += alpha p (the first step from x = 0); r -= alpha q ; d0 = r.r
__global__ void __launch_bounds__(TPB) k_fcg_update(int n, double* __restrict__ s, FcgIn in, double* __restrict__ x,
                                                    double* __restrict__ r, const double* __restrict__ p,
                                                    const double* __restrict__ q, Red rd, Prep pp) {
    int i = xcd_block() * blockDim.x + threadIdx.x;
    double v[2] = {0.0, 0.0};
    double a;
    if (in.nb) {
        a = fcg_alpha(s[S_RZ2 + in.par], block_total(in.nb, in.part).x);
        if (blockIdx.x == 0 && threadIdx.x == 0) s[S_ALPHA2 + in.par] = a;
    } else {
        a = s[S_ALPHA];
    }
    if (i < n) {
        x[i] = in.first ? a * p[i] : x[i] + a * p[i];
        double ri = r[i];
        ri -= a * q[i];
        r[i] = ri;
        v[0] = ri * ri;
        prep_store(pp, i, ri);
    }
    reduce2(v, rd);
}

template <class TA, class TB>
__global__ void __launch_bounds__(TPB) k_cast(int n, const TA* __restrict__ a, TB* __restrict__ b) {
    int i = xcd_block() * blockDim.x + threadIdx.x;
    if (i < n) b[i] = (TB)a[i];
}

// x = 0, r = rh = b, p = v = 0, d0 = b.b
__global__ void __launch_bounds__(TPB) k_bicg_init(int n, const double* __restrict__ b, double* __restrict__ x,
                                                   double* __restrict__ r, double* __restrict__ rh,
                                                   double* __restrict__ p, double* __restrict__ v, Red rd) {
    int i = xcd_block() * blockDim.x + threadIdx.x;
    double w[2] = {0.0, 0.0};
    if (i < n) {
        double bi = b[i];
        x[i] = 0.0; r[i] = bi; rh[i] = bi; p[i] = 0.0; v[i] = 0.0;
        w[0] = bi * bi;
    }
    reduce2(w, rd);
}
// p = r + beta (p - omega v) ; ph = D^-1 p
__global__ void __launch_bounds__(TPB) k_bicg_p(int n, const double* __restrict__ s, const double* __restrict__ r,
                                                const double* __restrict__ v, const double* __restrict__ dinv,
                                                double* __restrict__ p, double* __restrict__ ph) {
    int i = xcd_block() * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double pi = r[i] + s[S_BETA] * (p[i] - s[S_OMEGA] * v[i]);
    p[i] = pi; ph[i] = dinv[i] * pi;
}
// sv = r - alpha v ; sh = D^-1 sv
__global__ void __launch_bounds__(TPB) k_bicg_s(int n, const double* __restrict__ s, const double* __restrict__ r,
                                                const double* __restrict__ v, const double* __restrict__ dinv,
                                                double* __restrict__ sv, double* __restrict__ sh) {
    int i = xcd_block() * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double si = r[i] - s[S_ALPHA] * v[i];
    sv[i] = si; sh[i] = dinv[i] * si;
}
// x += alpha ph + omega sh ; r = sv - omega t ; d0 = r.r, d1 = rh.r
__global__ void __launch_bounds__(TPB) k_bicg_x(int n, const double* __restrict__ s, const double* __restrict__ ph,
                                                const double* __restrict__ sh, const double* __restrict__ sv,
                                                const double* __restrict__ t, const double* __restrict__ rh,
                                                double* __restrict__ x, double* __restrict__ r, Red rd) {
    int i = xcd_block() * blockDim.x + threadIdx.x;
    double w[2] = {0.0, 0.0};
    if (i < n) {
        x[i] += s[S_ALPHA] * ph[i] + s[S_OMEGA] * sh[i];
        double ri = sv[i] - s[S_OMEGA] * t[i];
        r[i] = ri;
        w[0] = ri * ri; w[1] = rh[i] * ri;
    }
    reduce2(w, rd);
}

// ------------------------------------------ three right-hand sides at once --
// The momentum components U, V, W share one matrix: BiCGStab on the three
// systems runs in lockstep, so every matrix pass serves all three.  Vectors
// are [3][n] (component k at +k*n); the Krylov scalars of component k live
// in slots Q_* + k of the device scalar array.
enum { Q_RHO = 32, Q_ALPHA = 35, Q_OMEGA = 38, Q_BETA = 41, Q_BB = 44 };
enum { F3_INIT = 0, F3_ALPHA, F3_OMEGA, F3_RHO, F3_STORE };

__device__ inline void block_partials6(double (&v)[6], double* __restrict__ part) {
    __shared__ double sh[6][TPB / 64];
#pragma unroll
    for (int q = 0; q < 6; ++q) v[q] = wave_sum(v[q]);
    if ((threadIdx.x & 63) == 0)
        for (int q = 0; q < 6; ++q) sh[q][threadIdx.x >> 6] = v[q];
    __syncthreads();
    if (threadIdx.x == 0)
        for (int q = 0; q < 6; ++q) {
            double t = 0.0;
            for (int w = 0; w < TPB / 64; ++w) t += sh[q][w];
            part[6 * blockIdx.x + q] = t;
        }
}

// INIT and STORE send the three squared norms to the host, RHO the largest
// relative one
__global__ void __launch_bounds__(1024) k_finish6(int nb, const double* __restrict__ part, double* __restrict__ s,
                                                  int what, Ring ring) {
    double a[6] = {0, 0, 0, 0, 0, 0};
    for (int i = threadIdx.x; i < nb; i += 1024)
        for (int q = 0; q < 6; ++q) a[q] += part[6 * i + q];
    __shared__ double sh[6][1024];
    for (int q = 0; q < 6; ++q) sh[q][threadIdx.x] = a[q];
    __syncthreads();
    for (int w = 512; w > 0; w >>= 1) {
        if (threadIdx.x < w)
            for (int q = 0; q < 6; ++q) sh[q][threadIdx.x] += sh[q][threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x != 0) return;
    double d[6];
    for (int q = 0; q < 6; ++q) d[q] = sh[q][0];
    double mx = 0.0;
    for (int k = 0; k < 3; ++k) {
        switch (what) {
        case F3_INIT:
            s[Q_BB + k] = d[k]; s[Q_RHO + k] = d[k];
            s[Q_ALPHA + k] = 1.0; s[Q_OMEGA + k] = 1.0; s[Q_BETA + k] = 0.0;
            break;
        case F3_ALPHA: s[Q_ALPHA + k] = d[k] != 0.0 ? s[Q_RHO + k] / d[k] : 0.0; break;
        case F3_OMEGA: s[Q_OMEGA + k] = d[3 + k] != 0.0 ? d[k] / d[3 + k] : 0.0; break;
        case F3_RHO: {
            double rho = s[Q_RHO + k], om = s[Q_OMEGA + k];
            s[Q_BETA + k] = (rho != 0.0 && om != 0.0) ? (d[3 + k] / rho) * (s[Q_ALPHA + k] / om) : 0.0;
            s[Q_RHO + k] = d[3 + k];
            double bb = s[Q_BB + k];
            double rel = bb > 0.0 ? d[k] / bb : 0.0;
            mx = (rel > mx || rel != rel) ? rel : mx;
            break;
        }
        default: break;
        }
    }
    if (what == F3_RHO) ring_put(ring, &mx, 1);
    else if (what == F3_INIT || what == F3_STORE) ring_put(ring, d, 3);
}

__global__ void __launch_bounds__(TPB) k_bicg3_init(int n, const double* __restrict__ b, double* __restrict__ x,
                                                    double* __restrict__ r, double* __restrict__ rh,
                                                    double* __restrict__ p, double* __restrict__ v,
                                                    double* __restrict__ part) {
    int i = xcd_block() * blockDim.x + threadIdx.x;
    double w[6] = {0, 0, 0, 0, 0, 0};
    if (i < n)
        for (int k = 0; k < 3; ++k) {
            size_t j = (size_t)k * n + i;
            double bi = b[j];
            x[j] = 0.0; r[j] = bi; rh[j] = bi; p[j] = 0.0; v[j] = 0.0;
            w[k] = bi * bi;
        }
    block_partials6(w, part);
}
// p = r + beta (p - omega v) ; ph = D^-1 p
__global__ void __launch_bounds__(TPB) k_bicg3_p(int n, const double* __restrict__ s, const double* __restrict__ r,
                                                 const double* __restrict__ v, const double* __restrict__ dinv,
                                                 double* __restrict__ p, double* __restrict__ ph) {
    int i = xcd_block() * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double di = dinv[i];
    for (int k = 0; k < 3; ++k) {
        size_t j = (size_t)k * n + i;
        double pi = r[j] + s[Q_BETA + k] * (p[j] - s[Q_OMEGA + k] * v[j]);
        p[j] = pi; ph[j] = di * pi;
    }
}
// sv = r - alpha v ; sh = D^-1 sv
__global__ void __launch_bounds__(TPB) k_bicg3_s(int n, const double* __restrict__ s, const double* __restrict__ r,
                                                 const double* __restrict__ v, const double* __restrict__ dinv,
                                                 double* __restrict__ sv, double* __restrict__ sh) {
    int i = xcd_block() * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double di = dinv[i];
    for (int k = 0; k < 3; ++k) {
        size_t j = (size_t)k * n + i;
        double si = r[j] - s[Q_ALPHA + k] * v[j];
        sv[j] = si; sh[j] = di * si;
    }
}
// x += alpha ph + omega sh ; r = sv - omega t ; partials r.r (0..2), rh.r (3..5)
__global__ void __launch_bounds__(TPB) k_bicg3_x(int n, const double* __restrict__ s, const double* __restrict__ ph,
                                                 const double* __restrict__ sh, const double* __restrict__ sv,
                                                 const double* __restrict__ t, const double* __restrict__ rh,
                                                 double* __restrict__ x, double* __restrict__ r,
                                                 double* __restrict__ part) {
    int i = xcd_block() * blockDim.x + threadIdx.x;
    double w[6] = {0, 0, 0, 0, 0, 0};
    if (i < n)
        for (int k = 0; k < 3; ++k) {
            size_t j = (size_t)k * n + i;
            x[j] += s[Q_ALPHA + k] * ph[j] + s[Q_OMEGA + k] * sh[j];
            double ri = sv[j] - s[Q_OMEGA + k] * t[j];
            r[j] = ri;
            w[k] = ri * ri; w[3 + k] = rh[j] * ri;
        }
    block_partials6(w, part);
}
// y_k = A x_k on the fine sliced-ELL operator for k = 0..2, with the dots
// MODE 0: a_k.y_k (0..2);  MODE 1: y_k.a_k (0..2), y_k.y_k (3..5);
// MODE 2: y_k = a_k - A x_k and y_k.y_k (0..2)
template <int MODE>
__global__ void __launch_bounds__(TPB) k_spmv3(int n, const int* __restrict__ sl_ptr, const int* __restrict__ col,
                                               const int16_t* __restrict__ dcol, const double* __restrict__ val,
                                               const double* __restrict__ diag, const double* __restrict__ x,
                                               double* __restrict__ y, const double* __restrict__ a,
                                               double* __restrict__ part) {
    int row = xcd_block() * blockDim.x + threadIdx.x;
    int s = row >> 6, lane = row & 63;
    double w[6] = {0, 0, 0, 0, 0, 0};
    size_t N = (size_t)n;
    if (s < ((n + 63) >> 6)) {
        bool own = row < n;     // the row's own operands before the gathers
        double d = own ? diag[row] : 0.0;
        double xr0 = own ? x[row] : 0.0, xr1 = own ? x[N + row] : 0.0, xr2 = own ? x[2 * N + row] : 0.0;
        double acc0 = 0.0, acc1 = 0.0, acc2 = 0.0;
        for (int e = sl_ptr[s] + 2 * lane; e < sl_ptr[s + 1]; e += 2 * SL) {     // entry pairs
            int2 j = dcol ? sell2_dcol(dcol, e, row) : sell2_col(col, e);
            double2 v = *reinterpret_cast<const double2*>(val + e);
            acc0 += v.x * x[j.x]; acc1 += v.x * x[N + j.x]; acc2 += v.x * x[2 * N + j.x];
            acc0 += v.y * x[j.y]; acc1 += v.y * x[N + j.y]; acc2 += v.y * x[2 * N + j.y];
        }
        if (own) {
            double acc[3] = {acc0 + d * xr0, acc1 + d * xr1, acc2 + d * xr2};
            for (int k = 0; k < 3; ++k) {
                size_t jj = (size_t)k * N + row;
                double yk = MODE == 2 ? a[jj] - acc[k] : acc[k];
                y[jj] = yk;
                if (MODE == 0) w[k] = a[jj] * yk;
                else if (MODE == 1) { w[k] = yk * a[jj]; w[3 + k] = yk * yk; }
                else w[k] = yk * yk;
            }
        }
    }
    block_partials6(w, part);
}

// ---------------------------------------------------------- Chebyshev ----
// start from x = 0: r = D^-1 b, d = r/theta, x = d.  bsrc (optional): FP64
// right-hand side, converted into b on the way.  zo (optional): FP64 copy of x.
template <class T>
__global__ void __launch_bounds__(TPB) k_cheb_init(int n, const T* __restrict__ dinv, T* __restrict__ b,
                                                   const double* __restrict__ bsrc, T theta_inv, T* __restrict__ r,
                                                   T* __restrict__ d, T* __restrict__ x, double* __restrict__ zo) {
    int i = xcd_block() * blockDim.x + threadIdx.x;
    if (i >= n) return;
    T bi;
    if (bsrc) { bi = (T)bsrc[i]; b[i] = bi; } else bi = b[i];
    T ri = dinv[i] * bi;
    T di = ri * theta_inv;
    r[i] = ri; d[i] = di; x[i] = di;
    if (zo) zo[i] = (double)di;
}

// coarse dense solve: y = Ainv x (FP64), x/y of type T
template <class T>
__global__ void __launch_bounds__(TPB) k_dense_gemv(int n, const double* __restrict__ M, const T* __restrict__ x,
                                                    T* __restrict__ y) {
    int row = blockIdx.x * (TPB / 64) + (threadIdx.x >> 6);
    int lane = threadIdx.x & 63;
    if (row >= n) return;
    double acc = 0.0;
    for (int j = lane; j < n; j += 64) acc += M[(size_t)row * n + j] * (double)x[j];
    acc = wave_sum(acc);
    if (lane == 0) y[row] = (T)acc;
}

// flag = 1 where some value of the na + nb differs from its key
__global__ void __launch_bounds__(TPB) k_neq(size_t na, const double* __restrict__ a, const double* __restrict__ ka,
                                             size_t nb, const double* __restrict__ b, const double* __restrict__ kb,
                                             int* __restrict__ flag) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < na ? a[i] != ka[i] : (i - na < nb && b[i - na] != kb[i - na])) *flag = 1;
}
// the flag to the host, and cleared for the next comparison
__global__ void k_flag_put(int* __restrict__ flag, Ring ring) {
    double v = *flag;
    *flag = 0;
    ring_put(ring, &v, 1);
}

// --------------------------------------------------------------- V-cycle --
template <class T> const DevSell<T>& opA(const AmgLevel& L);
template <> const DevSell<double>& opA<double>(const AmgLevel& L) { return L.A64; }
template <> const DevSell<float>& opA<float>(const AmgLevel& L) { return L.A32; }
template <class T> const DevSell<T>& opP(const AmgLevel& L);
template <> const DevSell<double>& opP<double>(const AmgLevel& L) { return L.P64; }
template <> const DevSell<float>& opP<float>(const AmgLevel& L) { return L.P32; }
template <class T> const DevSell<T>& opR(const AmgLevel& L);
template <> const DevSell<double>& opR<double>(const AmgLevel& L) { return L.R64; }
template <> const DevSell<float>& opR<float>(const AmgLevel& L) { return L.R32; }
template <class T> DBuf<T>& bx(AmgLevel& L);
template <> DBuf<double>& bx<double>(AmgLevel& L) { return L.x64; }
template <> DBuf<float>& bx<float>(AmgLevel& L) { return L.x32; }
template <class T> DBuf<T>& bw(AmgLevel& L);
template <> DBuf<double>& bw<double>(AmgLevel& L) { return L.w64; }
template <> DBuf<float>& bw<float>(AmgLevel& L) { return L.w32; }
template <class T> T* vb(AmgLevel& L);
template <> double* vb<double>(AmgLevel& L) { return L.b64.p; }
template <> float* vb<float>(AmgLevel& L) { return L.b32.p; }
template <class T> T* vr(AmgLevel& L);
template <> double* vr<double>(AmgLevel& L) { return L.r64.p; }
template <> float* vr<float>(AmgLevel& L) { return L.r32.p; }
template <class T> T* vt(AmgLevel& L);
template <> double* vt<double>(AmgLevel& L) { return L.t64.p; }
template <> float* vt<float>(AmgLevel& L) { return L.t32.p; }
template <class T> T* vu(AmgLevel& L);
template <> double* vu<double>(AmgLevel& L) { return L.u64.p; }
template <> float* vu<float>(AmgLevel& L) { return L.u32.p; }
template <class T> const T* vdinv(const AmgLevel& L);
template <> const double* vdinv<double>(const AmgLevel& L) { return L.dinv64.p; }
template <> const float* vdinv<float>(const AmgLevel& L) { return L.dinv32.p; }

struct Tags { const char *cheb, *chebx, *resid, *restrict_, *prolong; };
Tags level_tags(int l, bool fp64) {
    if (l == 0)
        return fp64 ? Tags{"amg_cheb_fp64_L0", "amg_chebx_fp64_L0", "amg_resid_fp64_L0", "amg_restrict_fp64_L0",
                           "amg_prolong_fp64_L0"}
                    : Tags{"amg_cheb_fp32_L0", "amg_chebx_fp32_L0", "amg_resid_fp32_L0", "amg_restrict_fp32_L0",
                           "amg_prolong_fp32_L0"};
    const char* t = fp64 ? "amg_coarse_fp64" : "amg_coarse_fp32";
    return Tags{t, t, t, t, t};
}

// Chebyshev polynomial smoother in D^-1 A on [lmax/10, 1.1 lmax] for the
// iterate held in the level's x buffer.  x_zero: start from x = 0 (no SpMV
// for the start).  bsrc: FP64 right-hand side to convert into b first.  zo:
// FP64 copy of the final iterate.
// Chebyshev interval [lo, hi] of a level's smoother
inline void cheb_interval(const AmgLevel& L, double& lo, double& hi) { hi = 1.1 * L.lmax; lo = hi / 10.0; }

// what the last step of a V-cycle does for the FCG loop around it (degree 1):
// its result goes to z in the V-cycle's precision, with the block partials of
// r.z and z.q
// (the finest operator sliced ELL)
struct VcDot {
    void* z;
    const double *r, *q;
    double* part;
};

template <class T>
void cheb_smooth(semo_ctx* c, AmgLevel& L, T* b, int degree, bool x_zero, const double* bsrc, double* zo,
                 const Tags& tg, const VcDot* vd = nullptr) {
    const DevSell<T>& A = opA<T>(L);
    int n = L.n;
    T* dA = vt<T>(L); T* dB = vu<T>(L); T* r = vr<T>(L);
    double hi, lo;
    cheb_interval(L, lo, hi);
    double theta = 0.5 * (hi + lo), delta = 0.5 * (hi - lo);
    double sigma = theta / delta, rho = 1.0 / sigma;
    if (x_zero) {
        SEMO_LAUNCH(c, tg.chebx,
                    (double)sizeof(T) * 5 * n + (bsrc ? 8.0 * n : 0.0) + (degree == 1 && zo ? 8.0 * n : 0.0),
                    k_cheb_init<T>, dim3(nblk(n)), dim3(TPB), n, vdinv<T>(L), b, bsrc, (T)(1.0 / theta), r, dA,
                    bx<T>(L).p, degree == 1 ? zo : nullptr);
    } else if (degree == 1 && vd) {
        RowArgs<T> a{};
        a.n = A.n; a.ptr = A.sl_ptr.p; a.col = A.col.p; a.val = A.val.p; a.diag = A.diag.p;
        a.dcol = A.dcol.n ? A.dcol.p : nullptr;
        a.x = bx<T>(L).p; a.b = b; a.dinv = vdinv<T>(L); a.xo = static_cast<T*>(vd->z); a.c1 = (T)(1.0 / theta);
        SEMO_LAUNCH(c, tg.chebx, op_bytes(A, 4) + 16.0 * n, k_chebx_dot<T>, dim3(nblk((long)A.nslices * 64)),
                    dim3(TPB), a, vd->r, vd->q, Red{vd->part});
    } else if (degree == 1) {
        // the only step: r and y are dead, and with zo (the finest level)
        // so is the T iterate, which keeps the level's x buffer in place
        RowArgs<T> a{};
        a.x = bx<T>(L).p; a.b = b; a.dinv = vdinv<T>(L); a.zo = zo; a.c1 = (T)(1.0 / theta);
        if (!zo) a.xo = bw<T>(L).p;
        row_launch<T, OP_CHEBX>(c, A, a, tg.chebx, op_bytes(A, 3) + (zo ? 8.0 * n : (double)sizeof(T) * n));
        if (!zo) std::swap(bx<T>(L), bw<T>(L));
    } else {
        RowArgs<T> a{};
        a.x = bx<T>(L).p; a.b = b; a.y = dA; a.dinv = vdinv<T>(L); a.r = r; a.xo = bw<T>(L).p;
        a.c1 = (T)(1.0 / theta);
        row_launch<T, OP_CHEBX>(c, A, a, tg.chebx, op_bytes(A, 6));
        std::swap(bx<T>(L), bw<T>(L));       // the new iterate is the level's x from here on
    }
    T* x = bx<T>(L).p;
    for (int k = 1; k < degree; ++k) {
        double rho_new = 1.0 / (2.0 * sigma - rho);
        double c1 = rho_new * rho, c2 = 2.0 * rho_new / delta;
        rho = rho_new;
        RowArgs<T> a{};
        a.x = dA; a.y = dB; a.dinv = vdinv<T>(L); a.r = r; a.xo = x; a.c1 = (T)c1; a.c2 = (T)c2;
        a.zo = k == degree - 1 ? zo : nullptr;
        row_launch<T, OP_CHEB>(c, A, a, tg.cheb, op_bytes(A, 8));
        std::swap(dA, dB);
    }
}

// one V-cycle for level l on b; the result is left in the level's x buffer
// (and, at the finest level, converted into zo)
// prepared (degree 1): b and the smoothed start x of level l were written by
// the kernel that produced b (the Krylov residual update at level 0, the
// restriction below it)
template <class T>
void vcycle(semo_ctx* c, Amg& amg, int l, int degree, const double* bsrc, double* zo, bool prepared = false,
            const VcDot* vd = nullptr) {
    AmgLevel& L = amg.lv[l];
    int n = L.n;
    T* b = vb<T>(L);
    if (l + 1 == (int)amg.lv.size()) {     // coarsest: dense direct solve in FP64
        if (bsrc) SEMO_LAUNCH(c, (sizeof(T) == 8 ? "amg_coarse_fp64" : "amg_coarse_fp32"), (8.0 + sizeof(T)) * n,
                              (k_cast<double, T>), dim3(nblk(n)), dim3(TPB), n, bsrc, b);
        SEMO_LAUNCH(c, (sizeof(T) == 8 ? "amg_coarse_fp64" : "amg_coarse_fp32"), 8.0 * n * n + 2.0 * sizeof(T) * n,
                    k_dense_gemv<T>, dim3((n + 3) / 4), dim3(TPB), n, amg.coarse_inv.p, b, bx<T>(L).p);
        if (zo) SEMO_LAUNCH(c, (sizeof(T) == 8 ? "amg_coarse_fp64" : "amg_coarse_fp32"), (8.0 + sizeof(T)) * n,
                            (k_cast<T, double>), dim3(nblk(n)), dim3(TPB), n, bx<T>(L).p, zo);
        return;
    }
    AmgLevel& C = amg.lv[l + 1];
    Tags tg = level_tags(l, sizeof(T) == 8);
    T* t = vt<T>(L);
    const DevSell<T>& A = opA<T>(L);
    if (degree == 1 && prepared) {
        spmv<T, OP_RES>(c, A, bx<T>(L).p, b, t, tg.resid);
    } else {
        cheb_smooth<T>(c, L, b, degree, true, bsrc, nullptr, tg);
        spmv<T, OP_RES>(c, A, bx<T>(L).p, b, t, tg.resid);
    }
    // a coarse level that smooths (not the coarsest) gets its b and its
    // degree-1 smoothed start from the restriction
    bool prep_next = degree == 1 && l + 2 < (int)amg.lv.size();
    if (prep_next) {
        double chi, clo;
        cheb_interval(C, clo, chi);
        RowArgs<T> a{};
        a.x = t; a.y = vb<T>(C); a.dinv = vdinv<T>(C); a.xo = bx<T>(C).p; a.c1 = (T)(1.0 / (0.5 * (chi + clo)));
        row_launch<T, OP_YPREP>(c, opR<T>(L), a, tg.restrict_,
                                op_bytes(opR<T>(L), 0) + (double)sizeof(T) * (n + 3.0 * C.n));
    } else {
        spmv<T, OP_Y>(c, opR<T>(L), t, (const T*)nullptr, vb<T>(C), tg.restrict_);
    }
    vcycle<T>(c, amg, l + 1, degree, nullptr, nullptr, prep_next);
    spmv<T, OP_ADD>(c, opP<T>(L), bx<T>(C).p, (const T*)nullptr, bx<T>(L).p, tg.prolong);
    cheb_smooth<T>(c, L, b, degree, false, nullptr, zo, tg, vd);
}

// z = M^-1 r with one V-cycle in precision T.  The V-cycle is a fixed
// sequence of ~22 kernels over fixed buffers, so it is captured once as a HIP
// graph and replayed: one submission instead of ~22.  It holds no memset and
// no library call.  Profiling (per-kernel events) runs it eagerly.
int cheb_degree(const semo_ctx* c) { return c->sp.cheb_degree > 0 ? c->sp.cheb_degree : 2; }

template <class T>
void sig_op(std::vector<const void*>& s, const DevSell<T>& M) {
    s.push_back(M.sl_ptr.p); s.push_back(M.col.p); s.push_back(M.dcol.p); s.push_back(M.val.p);
    s.push_back(M.diag.p);
}
// every device address a V-cycle in precision T passes to its kernels
template <class T>
std::vector<const void*> vcycle_signature(const Amg& amg, const double* r64, const double* z64, const VcDot* vd) {
    std::vector<const void*> s{r64, z64, amg.coarse_inv.p};
    if (vd)
        for (const void* p : {(const void*)vd->z, (const void*)vd->r, (const void*)vd->q, (const void*)vd->part})
            s.push_back(p);
    for (const AmgLevel& L : amg.lv) {
        if (sizeof(T) == 8) {
            for (const void* p : {(const void*)L.x64.p, (const void*)L.b64.p, (const void*)L.r64.p,
                                  (const void*)L.t64.p, (const void*)L.u64.p, (const void*)L.w64.p,
                                  (const void*)L.dinv64.p})
                s.push_back(p);
        } else {
            for (const void* p : {(const void*)L.x32.p, (const void*)L.b32.p, (const void*)L.r32.p,
                                  (const void*)L.t32.p, (const void*)L.u32.p, (const void*)L.w32.p,
                                  (const void*)L.dinv32.p})
                s.push_back(p);
        }
        sig_op(s, opA<T>(L)); sig_op(s, opP<T>(L)); sig_op(s, opR<T>(L));
    }
    std::sort(s.begin(), s.end());
    return s;
}

// what a graph of the V-cycle depends on: its addresses (sorted) and options
template <class T>
std::vector<const void*> vcycle_key(const semo_ctx* c, const Amg& amg, const double* r64, const double* z64,
                                    bool prepared, const VcDot* vd) {
    std::vector<const void*> s = vcycle_signature<T>(amg, r64, z64, vd);
    for (size_t v : {(size_t)cheb_degree(c), sizeof(T), (size_t)prepared, (size_t)(vd != nullptr), amg.builds})
        s.push_back(reinterpret_cast<const void*>(v));
    return s;
}

template <class T>
void precondition(semo_ctx* c, Amg& amg, const double* r64, double* z64) {
    int deg = cheb_degree(c);
    if (!c->graphs || c->prof.on) {
        vcycle<T>(c, amg, 0, deg, r64, z64);
        return;
    }
    std::vector<const void*> key = vcycle_key<T>(c, amg, r64, z64, false, nullptr);
    hipGraphExec_t x = amg.graphs.get(c->stream, key, [&] { vcycle<T>(c, amg, 0, deg, r64, z64); });
    SEMO_HIP(hipGraphLaunch(x, c->stream));
}

Red red_of(semo_ctx* c) { return Red{c->red.p}; }


// sums the partials of the previous launch (nb blocks) and applies `what`
void finish(semo_ctx* c, int nb, int what, const double* part = nullptr) {
    SEMO_LAUNCH(c, "krylov_finish", 16.0 * nb + 8.0, k_finish, dim3(1), dim3(FTPB), nb, part ? part : c->red.p,
                c->scal.p, what, Ring{nullptr, nullptr}, 0);
}
// ... and sends d0 (and d1: nput = 2) to the host: the caller has asked for
// the words (ring_expect)
void finish_put(semo_ctx* c, int nb, int what, const double* part = nullptr, int nput = 1) {
    SEMO_LAUNCH(c, "krylov_finish", 16.0 * nb + 8.0, k_finish, dim3(1), dim3(FTPB), nb, part ? part : c->red.p,
                c->scal.p, what, ring_of(c), nput);
}

// y = A x with dots of y (see k_spmv_dot), for the fine-level sliced-ELL operator
void spmv_dot(semo_ctx* c, const DevSell<double>& A, const double* x, double* y, const double* a0,
              const double* a1, int what) {
    int nb = nblk((long)A.nslices * 64);
    SEMO_LAUNCH(c, "spmv_fp64", op_bytes(A, 2 + (a0 ? 1 : 0) + (a1 ? 1 : 0)), k_spmv_dot, dim3(nb), dim3(TPB),
                A.n, A.sl_ptr.p, A.col.p, A.dcol.n ? A.dcol.p : nullptr, A.val.p, A.diag.p, x, y, a0, a1,
                red_of(c));
    finish(c, nb, what);
}

// x = 0 for b = 0: the iteration issued before |b|^2 arrived leaves 0 * z, NaN
// where the preconditioner overflows
void zero_x(semo_ctx* c, double* x, size_t n) { zero_d(c, x, n * sizeof(double)); }

// flexible (Polak-Ribiere) PCG with the AMG preconditioner.  x0 = 0,
// stop at ||r|| <= tol ||b||.
//
// An iteration is the V-cycle (its last step leaves z and the dots r.z, z.q),
// the direction and its product, the update of x and r (which also writes
// the next V-cycle's level-0 input) and the residual's way to the host: three
// kernels after the V-cycle's, with the scalars of small systems formed where
// they are used (block_total), five with k_finish for large ones.  (With
// the dots, the scalars and the residual's copy as launches of their own and
// r_old kept, a time step took 1.18 ms at 16^3, now 0.99; at 128^3 the V-cycle's
// last step and the dots take 32.0 us instead of 25.4 + 9.1.)
int fpcg(semo_ctx* c, Amg& amg, const DevSell<double>& A, const double* b, double* x, double tol, int maxit,
         bool mixed, double* relres) {
    SEMO_CHECK(A.lanes == 0, SEMO_EINVAL, "Krylov operator must be sliced ELL");
    int n = A.n;
    size_t ln = (size_t)n + 64;
    c->kv64.ensure(8 * ln);
    double* r = c->kv64.p; double* z = r + ln; double* p = z + ln; double* q = p + ln; double* p2 = q + ln;
    // degree-1 smoothing, at least two levels: the kernels that produce r also
    // write the V-cycle's level-0 input, and its last step the dots, where the
    // finest operator is sliced ELL (rows of more than ten or very unequal
    // numbers of neighbours are CSR: k_row smooths, k_dot follows)
    Prep pp{};
    bool prep = cheb_degree(c) == 1 && amg.lv.size() >= 2 && amg.lv[0].n == n;
    if (prep) {
        AmgLevel& L0 = amg.lv[0];
        double hi, lo;
        cheb_interval(L0, lo, hi);
        if (mixed) {
            pp.b32 = vb<float>(L0); pp.x32 = bx<float>(L0).p; pp.dinv32 = vdinv<float>(L0);
            pp.c1 = (float)(1.0 / (0.5 * (hi + lo)));
        } else {
            pp.b64 = vb<double>(L0); pp.x64 = bx<double>(L0).p; pp.dinv64 = vdinv<double>(L0);
            pp.c1d = 1.0 / (0.5 * (hi + lo));
        }
    }
    int nbr = nblk(n), nbs = nblk((long)A.nslices * 64);
    // partials of the three reductions of an iteration
    double* part_z = c->red.p;
    double* part_p = part_z + 2 * (size_t)std::max(nbs, RB);
    double* part_r = part_p + 2 * (size_t)nbs;
    bool own_totals = std::max(nbs, nbr) <= TOTAL_MAX;
    const VcDot vd{z, r, q, part_z};
    bool fused = prep && (mixed ? amg.lv[0].A32.lanes : amg.lv[0].A64.lanes) == 0;
    int nbz = fused ? nbs : rblk(n);                      // blocks of the r.z, z.q partials
    bool z32 = fused && mixed;                            // z as the FP32 V-cycle leaves it
    const VcDot* d = fused ? &vd : nullptr;
    const int16_t* dc = A.dcol.n ? A.dcol.p : nullptr;
    double prep_bytes = prep ? (mixed ? 8.0 : 16.0) * n : 0.0;     // the V-cycle's b and x written
    // iteration `it`: one ring word, its squared residual; the first is
    // preceded by the start (one more word, |b|^2)
    auto record = [&](int it) {
        bool first = it == 1;
        const double* po = (it & 1) ? p : p2;               // directions alternate between two buffers
        double* pn = (it & 1) ? p2 : p;
        if (first) {
            SEMO_LAUNCH(c, "fcg_init", 16.0 * n + prep_bytes, k_fcg_init, dim3(nbr), dim3(TPB), n, b, r, Red{part_r},
                        pp);
            finish_put(c, nbr, W_NONE, part_r);
        }
        if (mixed) vcycle<float>(c, amg, 0, cheb_degree(c), r, z, prep, d);
        else vcycle<double>(c, amg, 0, cheb_degree(c), r, z, prep, d);
        if (!fused)
            SEMO_LAUNCH(c, "krylov_dot", 32.0 * n, k_dot, dim3(nbz), dim3(TPB), n, r, z, z, q, Red{part_z});
        FcgIn in{part_z, own_totals ? nbz : 0, it & 1, first ? 1 : 0};
        if (!own_totals) finish(c, nbz, first ? W_FCG_START : W_FCG_BETA, part_z);
        // p = z + beta p, q = A p
        if (z32)
            SEMO_LAUNCH(c, "spmv_xpby_fp64", op_bytes(A, 3) + 4.0 * n, k_spmv_xpby<float>, dim3(nbs), dim3(TPB), n,
                        A.sl_ptr.p, A.col.p, dc, A.val.p, A.diag.p, c->scal.p, in,
                        reinterpret_cast<const float*>(z), po, pn, q, Red{part_p});
        else
            SEMO_LAUNCH(c, "spmv_xpby_fp64", op_bytes(A, 4), k_spmv_xpby<double>, dim3(nbs), dim3(TPB), n, A.sl_ptr.p,
                        A.col.p, dc, A.val.p, A.diag.p, c->scal.p, in, z, po, pn, q, Red{part_p});
        in.part = part_p;
        if (own_totals) in.nb = nbs;
        else finish(c, nbs, W_FCG_ALPHA, part_p);
        SEMO_LAUNCH(c, "fcg_update", 48.0 * n + prep_bytes, k_fcg_update, dim3(nbr), dim3(TPB), n, c->scal.p, in, x, r,
                    pn, q, Red{part_r}, pp);
        finish_put(c, nbr, W_NONE, part_r);
    };
    // The kernels of an iteration go out as one graph, the first iteration's
    // with the start, the even and the odd ones' each their own.  (As a graph
    // of the V-cycle between launches, an iteration of small systems waited
    // for the switch between the two: five captured and three plain empty
    // kernels take 34 us, eight captured ones 21 us.)
    bool graph = c->graphs && !c->prof.on;
    std::vector<const void*> key;
    if (graph) {
        ring_init(c);
        key = mixed ? vcycle_key<float>(c, amg, r, z, prep, d) : vcycle_key<double>(c, amg, r, z, prep, d);
        for (const void* a : {(const void*)A.sl_ptr.p, (const void*)A.col.p, (const void*)dc, (const void*)A.val.p,
                              (const void*)A.diag.p, (const void*)c->scal.p, (const void*)r, (const void*)z,
                              (const void*)p, (const void*)p2, (const void*)q, (const void*)x, (const void*)part_z,
                              (const void*)part_p, (const void*)part_r, (const void*)c->pin,
                              (const void*)c->d_seq.p, reinterpret_cast<const void*>((size_t)n)})
            key.push_back(a);
        // where an iteration leaves the next one's V-cycle its b and start: the
        // V-cycle's own list is sorted, and smoothing of another degree swaps
        // the level's x with a work array
        for (const void* a : {(const void*)pp.b32, (const void*)pp.x32, (const void*)pp.b64, (const void*)pp.x64})
            key.push_back(a);
        key.push_back(nullptr);                              // b (first iteration), which iteration
        key.push_back(nullptr);
    }
    hipGraphExec_t exec[3] = {};
    auto issue = [&](int it) {
        if (!graph) { record(it); return; }
        int kind = it == 1 ? 0 : 1 + (it & 1);
        if (!exec[kind]) {
            key[key.size() - 2] = it == 1 ? b : nullptr;
            key[key.size() - 1] = reinterpret_cast<const void*>((size_t)kind);
            exec[kind] = amg.graphs.get(c->stream, key, [&] { record(it); });
        }
        SEMO_HIP(hipGraphLaunch(exec[kind], c->stream));
    };
    int it = 0, w = ring_expect(c, 2);
    ConvCheck cc(c, tol * tol, w++);
    double bb = 0.0;
    for (it = 1; it <= maxit; ++it) {
        issue(it);
        if (it == 1 && (bb = cc.bb()) == 0.0) { zero_x(c, x, n); *relres = 0.0; return 0; }
        if (cc.done(it, w)) break;
        if (it < maxit) w = ring_expect(c, 1);
    }
    // true residual in FP64
    w = ring_expect(c, 1);
    SEMO_LAUNCH(c, "true_resid_fp64", op_bytes(A, 2), k_resid_norm, dim3(nbs), dim3(TPB), n, A.sl_ptr.p, A.col.p,
                dc, A.val.p, A.diag.p, x, b, Red{part_r});
    finish_put(c, nbs, W_NONE, part_r);
    *relres = std::sqrt(ring_read(c, w)) / std::sqrt(bb);
    return std::min(it, maxit);
}

// right-preconditioned (Jacobi) BiCGStab, x0 = 0
// z = M^-1 r for one component of a momentum / volume-fraction solve: one
// V-cycle of `amg` in the solve's precision, through fixed staging buffers,
// so that one captured V-cycle graph serves every component and call
void stage_vcycle(semo_ctx* c, Amg& amg, const double* r, double* z) {
    size_t n = c->nc;
    double* sr = c->mom_stage.p;
    double* sz = sr + n + 64;
    copy_d(c, sr, r, n);
    if (c->sp.precision == SEMO_PREC_MIXED) precondition<float>(c, amg, sr, sz);
    else precondition<double>(c, amg, sr, sz);
    copy_d(c, z, sz, n);
}

int bicgstab(semo_ctx* c, const DevSell<double>& A, const double* dinv, const double* b, double* x, double tol,
             int maxit, double* relres, Amg* pre = nullptr) {
    SEMO_CHECK(A.lanes == 0, SEMO_EINVAL, "Krylov operator must be sliced ELL");
    int n = A.n;
    size_t ln = (size_t)n + 64;
    c->kv64.ensure(8 * ln);
    double* r = c->kv64.p; double* rh = r + ln; double* p = rh + ln; double* v = p + ln; double* sv = v + ln;
    double* t = sv + ln; double* ph = t + ln; double* sh = ph + ln;
    double* s = c->scal.p;
    int w = ring_expect(c, 1);
    SEMO_LAUNCH(c, "bicg_init", 48.0 * n, k_bicg_init, dim3(nblk(n)), dim3(TPB), n, b, x, r, rh, p, v, red_of(c));
    finish_put(c, nblk(n), W_BICG_INIT);
    int it;
    ConvCheck cc(c, tol * tol, w);
    double bb = 0.0;
    for (it = 1; it <= maxit; ++it) {
        w = ring_expect(c, 1);
        SEMO_LAUNCH(c, "bicg_p", 48.0 * n, k_bicg_p, dim3(nblk(n)), dim3(TPB), n, s, r, v, dinv, p, ph);
        if (pre) stage_vcycle(c, *pre, p, ph);                            // ph = M^-1 p (AMG)
        spmv_dot(c, A, ph, v, rh, nullptr, W_BICG_ALPHA);                 // v = A ph, alpha
        SEMO_LAUNCH(c, "bicg_s", 40.0 * n, k_bicg_s, dim3(nblk(n)), dim3(TPB), n, s, r, v, dinv, sv, sh);
        if (pre) stage_vcycle(c, *pre, sv, sh);
        spmv_dot(c, A, sh, t, nullptr, sv, W_BICG_OMEGA);                 // t = A sh, omega
        SEMO_LAUNCH(c, "bicg_x", 64.0 * n, k_bicg_x, dim3(nblk(n)), dim3(TPB), n, s, ph, sh, sv, t, rh, x, r,
                    red_of(c));
        finish_put(c, nblk(n), W_BICG_RHO);
        if (it == 1 && (bb = cc.bb()) == 0.0) { zero_x(c, x, n); *relres = 0.0; return 0; }
        if (cc.done(it, w)) break;
    }
    int nbs = nblk((long)A.nslices * 64);
    w = ring_expect(c, 1);
    SEMO_LAUNCH(c, "true_resid_fp64", op_bytes(A, 2), k_resid_norm, dim3(nbs), dim3(TPB), n, A.sl_ptr.p, A.col.p,
                A.dcol.n ? A.dcol.p : nullptr, A.val.p, A.diag.p, x, b, red_of(c));
    finish_put(c, nbs, W_NONE);
    *relres = std::sqrt(ring_read(c, w)) / std::sqrt(bb);
    return std::min(it, maxit);
}

// BiCGStab on the three momentum components in lockstep (Jacobi, x0 = 0);
// stops when every component has ||r_k|| <= tol ||b_k||
int bicgstab3(semo_ctx* c, const DevSell<double>& A, const double* dinv, const double* b, double* x, double tol,
              int maxit, semo_solve_stats* st, Amg* pre = nullptr) {
    SEMO_CHECK(A.lanes == 0, SEMO_EINVAL, "Krylov operator must be sliced ELL");
    int n = A.n;
    size_t ln = 3 * (size_t)n + 64;
    c->kv64.ensure(8 * ln);
    double* r = c->kv64.p; double* rh = r + ln; double* p = rh + ln; double* v = p + ln; double* sv = v + ln;
    double* t = sv + ln; double* ph = t + ln; double* sh = ph + ln;
    double* s = c->scal.p;
    int nb = nblk(n), nbs = nblk((long)A.nslices * 64);
    size_t need = 6 * (size_t)std::max(nb, nbs) + 64;
    if (c->red.n < need) c->red.alloc(need);
    double* part = c->red.p;
    const int16_t* dc = A.dcol.n ? A.dcol.p : nullptr;
    auto fin = [&](int blocks, int what) {
        SEMO_LAUNCH(c, "bicg3_finish", 48.0 * blocks + 8.0, k_finish6, dim3(1), dim3(1024), blocks, part, s, what,
                    ring_of(c));
    };
    auto spmv3 = [&](int mode, const double* xin, double* y, const double* a) {
        // matrix once, three gathered operands, three results, three dot operands
        ProfScope ps(c, mode == 2 ? "spmv3_res_fp64" : "spmv3_fp64", op_bytes(A, 9));
        if (mode == 0)
            hipLaunchKernelGGL(k_spmv3<0>, dim3(nbs), dim3(TPB), 0, c->stream, n, A.sl_ptr.p, A.col.p, dc, A.val.p,
                               A.diag.p, xin, y, a, part);
        else if (mode == 1)
            hipLaunchKernelGGL(k_spmv3<1>, dim3(nbs), dim3(TPB), 0, c->stream, n, A.sl_ptr.p, A.col.p, dc, A.val.p,
                               A.diag.p, xin, y, a, part);
        else
            hipLaunchKernelGGL(k_spmv3<2>, dim3(nbs), dim3(TPB), 0, c->stream, n, A.sl_ptr.p, A.col.p, dc, A.val.p,
                               A.diag.p, xin, y, a, part);
    };
    SEMO_LAUNCH(c, "bicg3_init", 144.0 * n, k_bicg3_init, dim3(nb), dim3(TPB), n, b, x, r, rh, p, v, part);
    int wb = ring_expect(c, 3);
    fin(nb, F3_INIT);
    int it = 0;
    double bb[3] = {0.0, 0.0, 0.0};
    ConvCheck cc(c, tol * tol, 1.0);
    for (it = 1; it <= maxit; ++it) {
        SEMO_LAUNCH(c, "bicg3_p", 128.0 * n, k_bicg3_p, dim3(nb), dim3(TPB), n, s, r, v, dinv, p, ph);
        if (pre)                                               // ph_k = M^-1 p_k (AMG)
            for (int k = 0; k < 3; ++k) stage_vcycle(c, *pre, p + (size_t)k * n, ph + (size_t)k * n);
        spmv3(0, ph, v, rh);                                   // v = A ph, rh.v
        fin(nbs, F3_ALPHA);
        SEMO_LAUNCH(c, "bicg3_s", 104.0 * n, k_bicg3_s, dim3(nb), dim3(TPB), n, s, r, v, dinv, sv, sh);
        if (pre)
            for (int k = 0; k < 3; ++k) stage_vcycle(c, *pre, sv + (size_t)k * n, sh + (size_t)k * n);
        spmv3(1, sh, t, sv);                                   // t = A sh, t.s, t.t
        fin(nbs, F3_OMEGA);
        SEMO_LAUNCH(c, "bicg3_x", 192.0 * n, k_bicg3_x, dim3(nb), dim3(TPB), n, s, ph, sh, sv, t, rh, x, r, part);
        int w = ring_expect(c, 1);
        fin(nb, F3_RHO);
        if (it == 1) {                       // later iterations' words come around to these
            for (int k = 0; k < 3; ++k) bb[k] = ring_read(c, wb + k);
            if (!(bb[0] > 0.0 || bb[1] > 0.0 || bb[2] > 0.0)) break;
        }
        if (cc.done(it, w)) break;
    }
    it = std::min(it, maxit);
    // true residuals in FP64
    int wr = ring_expect(c, 3);
    spmv3(2, x, r, b);
    fin(nbs, F3_STORE);
    double rr[3];
    for (int k = 0; k < 3; ++k) rr[k] = ring_read(c, wr + k);
    if (!(bb[0] > 0.0 || bb[1] > 0.0 || bb[2] > 0.0)) { zero_x(c, x, 3 * (size_t)n); it = 0; }
    for (int k = 0; k < 3; ++k) {
        double rel = bb[k] > 0.0 ? std::sqrt(rr[k] / bb[k]) : 0.0;
        if (st) { st->iters[k] = bb[k] > 0.0 ? it : 0; st->rel_res[k] = rel; }
        check_converged(std::isfinite(bb[k]) ? rel : bb[k], tol, "momentum");
    }
    return it;
}

// level-0 operator of the hierarchy refreshed from the assembled system
// (same pattern, new values): off-diagonals through the slot map, diagonal,
// D^-1, FP32 copies
__global__ void __launch_bounds__(TPB) k_refresh_offdiag(size_t nv, const int* __restrict__ map,
                                                         const double* __restrict__ src, double* __restrict__ v64,
                                                         float* __restrict__ v32) {
    size_t e = (size_t)xcd_block() * blockDim.x + threadIdx.x;
    if (e >= nv) return;
    int m = map[e];
    double v = m >= 0 ? src[m] : 0.0;
    v64[e] = v; v32[e] = (float)v;
}
__global__ void __launch_bounds__(TPB) k_refresh_diag(int n, const double* __restrict__ d, double* __restrict__ d64,
                                                      float* __restrict__ d32, double* __restrict__ di64,
                                                      float* __restrict__ di32) {
    int i = xcd_block() * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double v = d[i], iv = 1.0 / v;
    d64[i] = v; d32[i] = (float)v; di64[i] = iv; di32[i] = (float)iv;
}

__global__ void __launch_bounds__(TPB) k_dinv(int n, const double* __restrict__ d, double* __restrict__ o) {
    int i = xcd_block() * blockDim.x + threadIdx.x;
    if (i < n) o[i] = 1.0 / d[i];
}

}  // namespace

// ---------------------------------------------------------------- uploads --
template <class T>
void sell_upload(DevSell<T>& M, const SellPattern& p, const std::vector<double>& vals,
                 const std::vector<double>& diag, hipStream_t s) {
    M.n = p.n; M.ncols = p.ncols; M.nslices = p.nslices; M.lanes = 0;
    M.nnz = p.nnz_offdiag + (int64_t)diag.size();
    M.sl_ptr.upload(p.sl_ptr, s);
    M.col.upload(p.col, s);
    sell_narrow(p, M.dcol, s);
    std::vector<T> v(vals.begin(), vals.end());
    M.val.upload(v, s);
    if (!diag.empty()) {
        std::vector<T> d(diag.begin(), diag.end());
        M.diag.upload(d, s);
    } else M.diag.release();
    SEMO_HIP(hipStreamSynchronize(s));
}
template void sell_upload<double>(DevSell<double>&, const SellPattern&, const std::vector<double>&,
                                  const std::vector<double>&, hipStream_t);
template void sell_upload<float>(DevSell<float>&, const SellPattern&, const std::vector<double>&,
                                 const std::vector<double>&, hipStream_t);

// column - row as int16 when every entry of a square pattern allows it;
// entries of the rows past n in the last slice (value 0) point at row n - 1.
// Leaves d empty otherwise.
void sell_narrow(const SellPattern& p, DBuf<int16_t>& d, hipStream_t s) {
    d.release();
    if (p.n != p.ncols || p.n == 0) return;
    std::vector<int16_t> h(p.col.size());
    for (int sl = 0; sl < p.nslices; ++sl)
        for (int e = p.sl_ptr[sl]; e < p.sl_ptr[sl + 1]; ++e) {
            int row = sl * SL + sell_lane(p.sl_ptr[sl], e);
            long dv = row < p.n ? (long)p.col[e] - row : (long)(p.n - 1) - row;
            if (dv < -32767 || dv > 32767) return;
            h[e] = (int16_t)dv;
        }
    d.upload(h, s);
    SEMO_HIP(hipStreamSynchronize(s));
}

template <class T>
void csr_upload(DevSell<T>& M, int n, int ncols, const std::vector<int>& ptr, const std::vector<int>& col,
                const std::vector<double>& vals, const std::vector<double>& diag, int lanes, hipStream_t s) {
    SEMO_CHECK(n >= 0 && ncols >= 1 && (int)ptr.size() == n + 1 && ptr[0] == 0 && ptr[n] == (int)col.size() &&
                   vals.size() == col.size() && (diag.empty() || (int)diag.size() == n),
               SEMO_EINVAL, "CSR operator: inconsistent arrays");
    SEMO_CHECK(lanes == 4 || lanes == 8 || lanes == 16 || lanes == 32 || lanes == 64, SEMO_EINVAL,
               "CSR operator: lanes per row");
    for (int r = 0; r < n; ++r) SEMO_CHECK(ptr[r + 1] >= ptr[r], SEMO_EINVAL, "CSR operator: row pointers");
    for (int cidx : col) SEMO_CHECK(cidx >= 0 && cidx < ncols, SEMO_EINVAL, "CSR operator: column out of range");
    M.n = n; M.ncols = ncols; M.nslices = (n + SL - 1) / SL; M.lanes = lanes;
    M.nnz = (int64_t)col.size() + (int64_t)diag.size();
    M.sl_ptr.upload(ptr, s);
    M.col.upload(col, s);
    std::vector<T> v(vals.begin(), vals.end());
    M.val.upload(v, s);
    if (!diag.empty()) {
        std::vector<T> d(diag.begin(), diag.end());
        M.diag.upload(d, s);
    } else M.diag.release();
    SEMO_HIP(hipStreamSynchronize(s));
}
template void csr_upload<double>(DevSell<double>&, int, int, const std::vector<int>&, const std::vector<int>&,
                                 const std::vector<double>&, const std::vector<double>&, int, hipStream_t);
template void csr_upload<float>(DevSell<float>&, int, int, const std::vector<int>&, const std::vector<int>&,
                                const std::vector<double>&, const std::vector<double>&, int, hipStream_t);

// partials for reductions over up to n rows (two values per block, three
// reductions at a time)
void reduction_alloc(semo_ctx* c, long n) {
    size_t need = 6 * (size_t)std::max(nblk(std::max<long>(n, 1) + 64), RB) + 64;
    if (c->red.n < need) c->red.alloc(need);
    if (c->scal.n < 64) c->scal.alloc(64);
}

// ----------------------------------------------------- equation solves ----
// The pressure hierarchy for the operator in c->Amat: built when missing;
// when the values changed, the finest level is refreshed on the device while
// keep_coarse says the coarse levels still serve, else rebuilt.
// the hierarchy `amg` for the operator in c->Amat, whose values it was built
// from are kept in key_val / key_diag (device copies)
void amg_update(semo_ctx* c, Amg& amg, DBuf<double>& key_val, DBuf<double>& key_diag,
                bool (*keep_coarse)(const Amg&)) {
    bool rebuild = !amg.built;
    if (amg.built) {
        // device-side comparison with the values the hierarchy was built from
        DBuf<int>& flag = c->d_flag1;
        if (!flag.n) { flag.alloc(1); zero_d(c, flag.p, sizeof(int)); }
        size_t nv = c->Amat.val.n, nd = (size_t)c->nc;
        int w = ring_expect(c, 1);
        SEMO_LAUNCH(c, "amg_values_changed", 16.0 * (nv + nd), k_neq, dim3((unsigned)((nv + nd + TPB - 1) / TPB)),
                    dim3(TPB), nv, c->Amat.val.p, key_val.p, nd, c->Amat.diag.p, key_diag.p, flag.p);
        SEMO_LAUNCH(c, "amg_values_changed", 16.0, k_flag_put, dim3(1), dim3(1), flag.p, ring_of(c));
        double f = ring_read(c, w);
        rebuild = f != 0.0;
    }
    // New values on the same pattern (a variable-density flow): refresh the
    // finest level on the device and keep the coarse levels, as long as the
    // flexible CG converges within 1.5x (+3) the iterations it needed right
    // after the last full set-up; otherwise, or without a slot map, rebuild.
    // The outer Krylov method always uses the current operator, so this only
    // affects the preconditioner's quality, never the solution.
    bool refresh = false;
    if (rebuild && amg.built && amg.l0_map.n == amg.lv[0].A64.val.n && amg.l0_map.n > 0 && keep_coarse(amg)) {
        refresh = true;
        rebuild = false;
    }
    if (refresh) {
        AmgLevel& L0 = amg.lv[0];
        size_t nv = L0.A64.val.n;
        SEMO_LAUNCH(c, "amg_refresh_L0", 24.0 * nv, k_refresh_offdiag, dim3((unsigned)((nv + TPB - 1) / TPB)),
                    dim3(TPB), nv, amg.l0_map.p, c->Amat.val.p, L0.A64.val.p, L0.A32.val.p);
        SEMO_LAUNCH(c, "amg_refresh_L0", 32.0 * c->nc, k_refresh_diag, dim3(nblk(c->nc)), dim3(TPB), c->nc,
                    c->Amat.diag.p, L0.A64.diag.p, L0.A32.diag.p, L0.dinv64.p, L0.dinv32.p);
        copy_d(c, key_val.p, c->Amat.val.p, c->Amat.val.n);
        copy_d(c, key_diag.p, c->Amat.diag.p, c->Amat.diag.n);
        amg.fresh = false;
    }
    if (rebuild) {
        amg.built = false;
        amg_build(c, amg, c->Amat);
        key_val.alloc(c->Amat.val.n);
        key_diag.alloc(c->nc);
        SEMO_HIP(hipMemcpyAsync(key_val.p, c->Amat.val.p, c->Amat.val.bytes(), hipMemcpyDeviceToDevice, c->stream));
        SEMO_HIP(hipMemcpyAsync(key_diag.p, c->Amat.diag.p, c->Amat.diag.bytes(), hipMemcpyDeviceToDevice, c->stream));
        amg.fresh = true;
    }
}

void pressure_amg_update(semo_ctx* c, bool (*keep_coarse)(const Amg&)) {
    amg_update(c, c->amg_p, c->amg_key_val, c->amg_key_diag, keep_coarse);
}

// z = M^-1 r: one V-cycle of the pressure hierarchy, FP32 (fp32) or FP64,
// FP64 in and out (the Schur-complement step of the coupled solver)
void pressure_vcycle(semo_ctx* c, const double* r64, double* z64, bool fp32) {
    SEMO_CHECK(c->amg_p.built, SEMO_ESTATE, "pressure hierarchy not built");
    if (fp32) precondition<float>(c, c->amg_p, r64, z64);
    else precondition<double>(c, c->amg_p, r64, z64);
}
void pressure_vcycle_kernels(semo_ctx* c, const double* r64, double* z64, bool fp32) {
    SEMO_CHECK(c->amg_p.built, SEMO_ESTATE, "pressure hierarchy not built");
    if (fp32) vcycle<float>(c, c->amg_p, 0, cheb_degree(c), r64, z64);
    else vcycle<double>(c, c->amg_p, 0, cheb_degree(c), r64, z64);
}
std::vector<const void*> pressure_vcycle_signature(semo_ctx* c, const double* r64, const double* z64, bool fp32) {
    return fp32 ? vcycle_key<float>(c, c->amg_p, r64, z64, false, nullptr)
                : vcycle_key<double>(c, c->amg_p, r64, z64, false, nullptr);
}

double2 sum_to_host(semo_ctx* c, int nb, const double* part) {
    int w = ring_expect(c, 2);
    finish_put(c, nb, W_NONE, part, 2);
    double a = ring_read(c, w);
    return make_double2(a, ring_read(c, w + 1));
}
double min_to_host(semo_ctx* c, int nb, const double* part) {
    int w = ring_expect(c, 1);
    SEMO_LAUNCH(c, "krylov_finish", 16.0 * nb + 8.0, k_finish_min, dim3(1), dim3(FTPB), nb, part,
                std::numeric_limits<double>::infinity(), ring_of(c));
    return ring_read(c, w);
}

// flexible CG: the coarse levels serve while the iteration count stays
// within 1.5x (+3) of the count right after the last full set-up
bool fcg_keeps_coarse(const Amg& amg) {
    return amg.iters_ref >= 0 && amg.last_iters <= std::max((3 * amg.iters_ref) / 2, amg.iters_ref + 3);
}

// pressure: hierarchy (re)built when the operator's values changed
void solve_pressure(semo_ctx* c, const double* b, double* x, semo_solve_stats* st) {
    Amg& amg = c->amg_p;
    pressure_amg_update(c, fcg_keeps_coarse);
    reduction_alloc(c, c->nc);
    double rr = 0;
    int it = fpcg(c, amg, c->Amat, b, x, c->sp.tol_p, c->sp.maxit_p, c->sp.precision == SEMO_PREC_MIXED, &rr);
    if (amg.fresh) { amg.iters_ref = it; amg.fresh = false; }
    amg.last_iters = it;
    if (st) {
        st->iters[0] = it; st->rel_res[0] = rr; st->n_levels = (int)amg.lv.size(); st->setup_ms = amg.setup_ms;
    }
    check_converged(rr, c->sp.tol_p, "pressure");
}

// BiCGStab keeps the coarse levels of its AMG preconditioner while it
// converges within 1.5x (+3) the iterations right after the last build
bool bicg_keeps_coarse(const Amg& amg) {
    return amg.iters_ref >= 0 && amg.last_iters <= std::max((3 * amg.iters_ref) / 2, amg.iters_ref + 3);
}

// momentum (nrhs = 3, one operator, three right-hand sides in lockstep) and
// volume fraction (nrhs = 1): BiCGStab right-preconditioned by Jacobi, or by
// an AMG V-cycle of the system's own hierarchy (SEMO_MSOLVER_AMG, or
// SEMO_MSOLVER_AUTO once a Jacobi solve of that system has needed more than
// MSOLVER_AUTO_ITERS iterations), as SEMO's AMGCL solves precondition them
// with aggregation AMG (solveAMGCL.cpp:881-927, 1195-1258)
constexpr int MSOLVER_AUTO_ITERS = 30;
void solve_momentum(semo_ctx* c, int nrhs, semo_solve_stats* st) {
    int n = c->nc;
    reduction_alloc(c, n);
    DBuf<double>& dinv = c->dinv_mom;
    dinv.alloc(n + 64);
    SEMO_LAUNCH(c, "jacobi_dinv", 16.0 * n, k_dinv, dim3(nblk(n)), dim3(TPB), n, c->Amat.diag.p, dinv.p);
    bool mom = nrhs == 3;
    bool& auto_on = mom ? c->amg_mom_on : c->amg_vf_on;
    Amg* pre = nullptr;
    if (c->msolver == SEMO_MSOLVER_AMG || (c->msolver == SEMO_MSOLVER_AUTO && auto_on)) {
        Amg& amg = mom ? c->amg_m : c->amg_vf;
        amg_update(c, amg, mom ? c->amg_m_kv : c->amg_vf_kv, mom ? c->amg_m_kd : c->amg_vf_kd, bicg_keeps_coarse);
        c->mom_stage.ensure(2 * ((size_t)n + 64));
        pre = &amg;
    }
    int it = 0;
    if (nrhs == 3) {
        it = bicgstab3(c, c->Amat, dinv.p, c->Bvec.p, c->Xvec.p, c->sp.tol_u, c->sp.maxit_u, st, pre);
    } else {
        for (int k = 0; k < nrhs; ++k) {
            double rr = 0;
            int ik = bicgstab(c, c->Amat, dinv.p, c->Bvec.p + (size_t)k * n, c->Xvec.p + (size_t)k * n,
                              c->sp.tol_u, c->sp.maxit_u, &rr, pre);
            if (st) { st->iters[k] = ik; st->rel_res[k] = rr; }
            check_converged(rr, c->sp.tol_u, "momentum/volume-fraction");
            it = std::max(it, ik);
        }
    }
    if (pre) {
        if (pre->fresh) { pre->iters_ref = it; pre->fresh = false; }
        pre->last_iters = it;
        if (st) { st->n_levels = (int)pre->lv.size(); st->setup_ms = pre->setup_ms; }
    } else if (c->msolver == SEMO_MSOLVER_AUTO && it > MSOLVER_AUTO_ITERS) {
        auto_on = true;
    }
}

// standalone COO system (seam 2)
void solve_coo(semo_ctx* c, const char* eq, int n, int64_t nnz, const int* rows, const int* cols,
               const double* vals, int nrhs, const double* b, double* x, semo_solve_stats* st) {
    SEMO_CHECK(n > 0 && nnz >= n && nrhs >= 1 && nrhs <= 4, SEMO_EINVAL, "solve_coo sizes");
    for (int64_t k = 0; k < nnz; ++k) {
        SEMO_CHECK(rows[k] >= 0 && rows[k] < n && cols[k] >= 0 && cols[k] < n, SEMO_EINVAL, "COO index out of range");
        SEMO_CHECK(std::isfinite(vals[k]), SEMO_EINVAL, "COO value is not finite");
    }
    for (int64_t k = 0; k < (int64_t)n * nrhs; ++k)
        SEMO_CHECK(std::isfinite(b[k]), SEMO_EINVAL, "right-hand side is not finite");
    // CSR with summed duplicates, sorted columns
    std::vector<int> ptr(n + 1, 0);
    for (int64_t k = 0; k < nnz; ++k) ptr[rows[k] + 1]++;
    for (int i = 0; i < n; ++i) ptr[i + 1] += ptr[i];
    std::vector<std::pair<int, double>> ent(nnz);
    {
        std::vector<int> pos(ptr.begin(), ptr.end() - 1);
        for (int64_t k = 0; k < nnz; ++k) ent[pos[rows[k]]++] = {cols[k], vals[k]};
    }
    std::vector<int> cptr(n + 1, 0), ccol; std::vector<double> cval;
    for (int i = 0; i < n; ++i) {
        std::sort(ent.begin() + ptr[i], ent.begin() + ptr[i + 1],
                  [](const auto& a, const auto& b2) { return a.first < b2.first; });
        for (int k = ptr[i]; k < ptr[i + 1]; ++k) {
            if (!ccol.empty() && (int)ccol.size() > cptr[i] && ccol.back() == ent[k].first) { cval.back() += ent[k].second; continue; }
            ccol.push_back(ent[k].first); cval.push_back(ent[k].second);
        }
        cptr[i + 1] = (int)ccol.size();
    }
    // device operator
    std::vector<int> optr(n + 1, 0), ocol; std::vector<double> oval, diag(n, 0.0);
    for (int i = 0; i < n; ++i) {
        for (int k = cptr[i]; k < cptr[i + 1]; ++k) {
            if (ccol[k] == i) diag[i] = cval[k];
            else { ocol.push_back(ccol[k]); oval.push_back(cval[k]); }
        }
        optr[i + 1] = (int)ocol.size();
    }
    for (int i = 0; i < n; ++i) SEMO_CHECK(diag[i] != 0.0, SEMO_EZERO_PIVOT, "zero diagonal");
    std::vector<int> pos;
    SellPattern p = sell_from_csr(n, n, optr, ocol, &pos);
    std::vector<double> pv(p.col.size(), 0.0);
    for (size_t k = 0; k < ocol.size(); ++k) pv[pos[k]] = oval[k];
    DevSell<double> A;
    sell_upload<double>(A, p, pv, diag, c->stream);
    DBuf<double> db, dx;
    db.upload(b, (size_t)n * nrhs, c->stream);
    dx.alloc((size_t)n * nrhs);
    reduction_alloc(c, n);
    std::string e(eq ? eq : "");
    if (e == "pressure") {
        Amg amg;
        amg_build_csr(c, amg, n, cptr, ccol, cval);
        for (int k = 0; k < nrhs; ++k) {
            double rr = 0;
            int it = fpcg(c, amg, A, db.p + (size_t)k * n, dx.p + (size_t)k * n, c->sp.tol_p, c->sp.maxit_p,
                          c->sp.precision == SEMO_PREC_MIXED, &rr);
            if (st) { st->iters[k] = it; st->rel_res[k] = rr; st->n_levels = (int)amg.lv.size(); st->setup_ms = amg.setup_ms; }
            check_converged(rr, c->sp.tol_p, "pressure");
        }
        // the local hierarchy and its graph go out of scope here
        SEMO_HIP(hipStreamSynchronize(c->stream));
    } else {
        DBuf<double> dinv; dinv.alloc(n + 64);
        SEMO_LAUNCH(c, "jacobi_dinv", 16.0 * n, k_dinv, dim3(nblk(n)), dim3(TPB), n, A.diag.p, dinv.p);
        for (int k = 0; k < nrhs; ++k) {
            double rr = 0;
            int it = bicgstab(c, A, dinv.p, db.p + (size_t)k * n, dx.p + (size_t)k * n, c->sp.tol_u, c->sp.maxit_u, &rr);
            if (st) { st->iters[k] = it; st->rel_res[k] = rr; }
            check_converged(rr, c->sp.tol_u, "solve");
        }
    }
    dx.download(x, (size_t)n * nrhs, c->stream);
    SEMO_HIP(hipStreamSynchronize(c->stream));
}

}  // namespace semo
