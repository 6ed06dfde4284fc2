// Compact clusters of cells for the vertex-stencil passes (LSQ gradients,
// curvature divergence), built once per mesh on the device.
//
// The storage order is lib_RCM's: 256 consecutive cells are a thin piece of a
// level, and the cells their stencils touch are 12 times as many.  Cut from a
// space-filling order instead, 256 cells touch 2 (hexes) to 4 (tets) times
// as many, few enough for a workgroup to bring them into LDS once and gather
// from there; the stencils become 16-bit places in that list.  Entry order,
// and so every sum, stays the stencil's own.
#include <algorithm>
#include <climits>

#include "kern.hpp"

namespace semo {
namespace {

constexpr int HASH = 4096;            // LDS table of a cluster's distinct cells
constexpr int CL_SHORT = 512;

// place of a cell centre on the Hilbert curve (Butz's algorithm in the form of
// Hamilton, "Compact Hilbert Indices", 2006) through a grid of 1024^3 points
// of spacing 1 / inv_h from lo.  Built from the top bit down: at each level the
// octant's place is the Gray rank of its three bits in the current frame (a
// permutation of the axes and a reflection), and the next frame is the one in
// which the sub-curve enters where the curve so far left off.
__global__ void __launch_bounds__(TPB) k_cluster_key(int nc, const double* __restrict__ cxyz, double lo0, double lo1,
                                                     double lo2, double inv_h, uint32_t* __restrict__ key) {
    int i = blockIdx.x * TPB + threadIdx.x;
    if (i >= nc) return;
    const double lo[3] = {lo0, lo1, lo2};
    uint32_t v[3];
    for (int a = 0; a < 3; ++a) {
        double q = (cxyz[3 * (size_t)i + a] - lo[a]) * inv_h;
        v[a] = (uint32_t)fmin(fmax(q, 0.0), 1023.0);
    }
    // frame: corner e the curve enters the octant at, axis d along which it
    // leaves it; bits are read rotated by d + 1 after the reflection by e
    uint32_t k = 0, e = 0;
    int d = 0;
    auto rotr = [](uint32_t x, int n) { return n ? ((x >> n) | (x << (3 - n))) & 7u : x; };
    auto rotl = [](uint32_t x, int n) { return n ? ((x << n) | (x >> (3 - n))) & 7u : x; };
    for (int b = 9; b >= 0; --b) {
        uint32_t l = ((v[0] >> b) & 1u) | ((v[1] >> b) & 1u) << 1 | ((v[2] >> b) & 1u) << 2;
        int r = (d + 1) % 3;
        uint32_t t = rotr(l ^ e, r);
        uint32_t w = t ^ (t >> 1);                    // inverse Gray code of three bits
        w ^= t >> 2;
        k = (k << 3) | w;
        // entry corner and direction of sub-octant w in the unrotated frame
        uint32_t g = w == 0 ? 0u : ((w - 1) & ~1u);
        uint32_t ent = g ^ (g >> 1);
        int dir = w == 0 ? 0 : (w & 1 ? __ffs((int)~w) - 1 : __ffs((int)~(w - 1)) - 1) % 3;
        e ^= rotl(ent, r);
        d = (d + dir + 1) % 3;
    }
    key[i] = k;
}

// ascending bitonic sort of N ints in LDS by the whole block
template <int N>
__device__ inline void lds_sort(int* v) {
    for (int k = 2; k <= N; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1) {
            __syncthreads();
            for (int t = threadIdx.x; t < N; t += TPB) {
                int o = t ^ j;
                if (o > t) {
                    int a = v[t], b = v[o];
                    if ((a > b) == ((t & k) == 0)) { v[t] = b; v[o] = a; }
                }
            }
        }
    __syncthreads();
}

// the cells of each cluster in ascending order, their entry counts, and the
// widths of its four 64-cell slices (even)
__global__ void __launch_bounds__(TPB) k_cluster_order(int nc, const int* __restrict__ order,
                                                       const int* __restrict__ st_ptr, int* __restrict__ cell,
                                                       int* __restrict__ num, int* __restrict__ width) {
    __shared__ int v[TPB];
    size_t p = (size_t)blockIdx.x * TPB + threadIdx.x;
    v[threadIdx.x] = p < (size_t)nc ? order[p] : INT_MAX;
    lds_sort<TPB>(v);
    int i = v[threadIdx.x];
    int n = i == INT_MAX ? 0 : st_ptr[i + 1] - st_ptr[i];
    cell[p] = i == INT_MAX ? -1 : i;
    num[p] = n;
    for (int o = 32; o > 0; o >>= 1) n = max(n, __shfl_xor(n, o, 64));
    if ((threadIdx.x & 63) == 0) width[p >> 6] = (n + 1) & ~1;
}

// the distinct cells of a cluster and its stencils, ascending, and the
// stencil entries as places in that list (pairs: sell_pos); *over is raised
// when a cluster has more than CL_LIST
__global__ void __launch_bounds__(TPB) k_cluster_lists(const int* __restrict__ cell, const int* __restrict__ num,
                                                       const int* __restrict__ st_ptr, const int* __restrict__ st_idx,
                                                       const int* __restrict__ sl, int* __restrict__ cnt,
                                                       int* __restrict__ list, uint16_t* __restrict__ ell,
                                                       int* __restrict__ over) {
    __shared__ int table[HASH];
    __shared__ int arr[CL_LIST];
    __shared__ int distinct, fill;
    for (int t = threadIdx.x; t < HASH; t += TPB) table[t] = -1;
    for (int t = threadIdx.x; t < CL_LIST; t += TPB) arr[t] = INT_MAX;
    if (threadIdx.x == 0) { distinct = 0; fill = 0; }
    __syncthreads();
    size_t p = (size_t)blockIdx.x * TPB + threadIdx.x;
    int i = cell[p], n = num[p];
    size_t e0 = i >= 0 ? (size_t)st_ptr[i] : 0;
    auto insert = [&](int key) {
        unsigned h = ((unsigned)key * 2654435761u) >> 20;             // 12 bits
        for (int probe = 0; probe < HASH; ++probe) {
            int old = atomicCAS(&table[(h + probe) & (HASH - 1)], -1, key);
            if (old == -1) { atomicAdd(&distinct, 1); return; }
            if (old == key) return;
        }
        atomicAdd(&distinct, HASH);                                   // the table is full
    };
    if (i >= 0) insert(i);
    for (int k = 0; k < n; ++k) {
        if (*(volatile int*)&distinct > CL_LIST) break;
        insert(st_idx[e0 + k]);
    }
    __syncthreads();
    if (distinct > CL_LIST) {
        if (threadIdx.x == 0) { cnt[blockIdx.x] = 0; atomicOr(over, 1); }
        return;
    }
    for (int t = threadIdx.x; t < HASH; t += TPB)
        if (table[t] >= 0) arr[atomicAdd(&fill, 1)] = table[t];
    lds_sort<CL_LIST>(arr);
    int m = distinct;
    if (threadIdx.x == 0) cnt[blockIdx.x] = m;
    for (int t = threadIdx.x; t < m; t += TPB) list[(size_t)blockIdx.x * CL_LIST + t] = arr[t];
    int base = sl[p >> 6], lane = threadIdx.x & 63, w = (sl[(p >> 6) + 1] - base) / SL;
    for (int k = 0; k < w; ++k) {
        int at = 0;
        if (k < n) {
            int key = st_idx[e0 + k], lo = 0, hi = m - 1;
            while (lo < hi) {
                int mid = (lo + hi) >> 1;
                if (arr[mid] < key) lo = mid + 1; else hi = mid;
            }
            at = lo;
        }
        ell[base + (k >> 1) * (2 * SL) + 2 * lane + (k & 1)] = (uint16_t)at;
    }
}

}  // namespace

// Space order by a counting sort of the keys (the cells' own mean spacing),
// then lists on the device.  For long stencils (tets) at any size, for short
// ones (hexes: 26 cells) up to CL_SHORT clusters: there a gathering pass leaves
// the chip waiting (91125 hexes, U, V, W and five fields: staged 26 and 31 us,
// gathered 33 and 35), beyond it the scattered stores of cells far apart in
// storage cost more than the gathers (222650: 47 and 59 against 45 and 54;
// 2.1M: 314 and 413 against 314 and 376).  On 96 x 48 x 48 cubes of six tets the lists average
// 1123 cells and reach 1470 (in Morton order 1244 and 1611), on 128^3 hexes 578
// and 600.
void stencil_clusters(semo_ctx* c) {
    Clusters& K = c->clu;
    K.ok = false;
    const int nc = c->nc;
    K.n = (nc + TPB - 1) / TPB;
    if (K.n > CL_SHORT && (double)c->d_st_idx.n < LSQ_LANES_LONG_STENCIL * nc) return;
    double ext[3], vol = 1.0, big = 0.0;
    for (int a = 0; a < 3; ++a) {
        ext[a] = c->bb_hi[a] - c->bb_lo[a];
        vol *= ext[a];
        big = std::max(big, ext[a]);
    }
    if (!(vol > 0.0) || !std::isfinite(vol)) return;
    double h = std::max(std::cbrt(vol / nc), big / 1023.0);
    hipStream_t s = c->stream;
    DBuf<uint32_t> dkey;
    dkey.alloc(nc);
    SEMO_LAUNCH(c, "setup_clusters", 28.0 * nc, k_cluster_key, dim3(nblk(nc)), dim3(TPB), nc, c->c_xyz.p, c->bb_lo[0],
                c->bb_lo[1], c->bb_lo[2], 1.0 / h, dkey.p);
    std::vector<uint32_t> key(nc);
    dkey.download(key.data(), nc, s);
    SEMO_HIP(hipStreamSynchronize(s));
    std::vector<int> a(nc), b(nc);
    std::iota(a.begin(), a.end(), 0);
    for (int shift = 0; shift < 30; shift += 10) {
        std::vector<int> pos(1025, 0);
        for (int i = 0; i < nc; ++i) ++pos[((key[i] >> shift) & 1023) + 1];
        for (int d = 0; d < 1024; ++d) pos[d + 1] += pos[d];
        for (int i : a) b[pos[(key[i] >> shift) & 1023]++] = i;
        a.swap(b);
    }
    DBuf<int> order, width, over;
    order.upload(a, s);
    const size_t np = (size_t)K.n * TPB, ns = np / SL;
    K.cell.alloc(np); K.num.alloc(np); K.cnt.alloc(K.n);
    width.alloc(ns);
    SEMO_LAUNCH(c, "setup_clusters", 20.0 * nc, k_cluster_order, dim3(K.n), dim3(TPB), nc, order.p, c->d_st_ptr.p,
                K.cell.p, K.num.p, width.p);
    std::vector<int> w(ns), sl(ns + 1, 0);
    width.download(w.data(), ns, s);
    SEMO_HIP(hipStreamSynchronize(s));
    for (size_t k = 0; k < ns; ++k) {
        if ((int64_t)sl[k] + (int64_t)w[k] * SL > INT_MAX) return;
        sl[k + 1] = sl[k] + w[k] * SL;
    }
    K.sl.upload(sl, s);
    K.ell.alloc((size_t)sl[ns] + 2 * SL);
    K.list.alloc((size_t)K.n * CL_LIST);
    over.alloc(1);
    zero_d(c, over.p, sizeof(int));
    SEMO_LAUNCH(c, "setup_clusters", 6.0 * (double)c->d_st_idx.n, k_cluster_lists, dim3(K.n), dim3(TPB), K.cell.p,
                K.num.p, c->d_st_ptr.p, c->d_st_idx.p, K.sl.p, K.cnt.p, K.list.p, K.ell.p, over.p);
    int ov = 0;
    std::vector<int> cnt(K.n);
    over.download(&ov, 1, s);
    K.cnt.download(cnt.data(), cnt.size(), s);
    SEMO_HIP(hipStreamSynchronize(s));
    K.most = *std::max_element(cnt.begin(), cnt.end());
    K.total = 0;
    for (int v : cnt) K.total += v;
    K.ok = ov == 0;
    if (!K.ok) { K.list.release(); K.ell.release(); }
}

}  // namespace semo
