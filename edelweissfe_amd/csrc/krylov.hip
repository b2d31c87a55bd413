// Krylov solvers for the assembled tangent on gfx950.
//
// Operator layout: sliced ELL of 3x3 blocks, slice height 64 (one wavefront).
// Lane l of a slice s's workgroup has row slot p = 64 s + l, the row of node slotNode[p] (rows
// sorted by length inside windows of nodes), whose blocks its wavefronts share; block slot k of that row
// stores its 9 values at Kval[slice_off[s]*9 + (9k+v)*64 + l], so every value
// load of a wavefront is one contiguous 512 B (FP64) / 256 B (FP32) segment and
// the block column index (1 int per 9 values) is shared by the three rows of a
// node.  Padding slots hold zeros and point at the row itself.
//
// PCG with 3x3 block-Jacobi, in place of the reference's direct solve
// (nonlinearimplicitstatic.py:727-751) on symmetric tangents.  One iteration is
// three kernels:
//   A: q = K p, per-workgroup partials of p.q
//   B: alpha = rz/pq; r -= alpha q; z = Minv r; partials of r.z, r.r
//   C: x += alpha p; beta = rz_new/rz; convergence test; p = z + beta p
// (small assembled systems two: C's test and p in the next A, x in B).
// Global scalars are never stored by one workgroup for the others of its launch: every
// workgroup re-reduces the (few thousand) partials of the previous kernel in the
// same fixed order, so all workgroups hold bitwise identical scalars and the
// whole solve is deterministic.  What the first workgroup stores for the next launches (alpha, the stop
// flags, which alternate with the iteration) no kernel reads that stores it.  A runs on the product's grid, B and C on a smaller
// grid of their own (their partials re-reduced by every workgroup cost less).  The two
// r.z partial buffers alternate with the iteration parity, so a batch of an even number
// of iterations is a fixed sequence of launches that is captured once into a hipGraph
// and replayed.
// With the hexa8 brick operator (matrix-free FP32, and FP64), A is the brick product alone, its
// partials the bricks' shares of p.Kp (Dirichlet DOFs masked), and B gathers each node's
// brick partials itself (q is never stored): p.q = the bricks' sum + the sum of p^2 over the
// Dirichlet DOFs, whose partials C (and the init) form with p.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "efe_internal.h"

struct KrylovWork {
    int D = 0, N = 0;
    // grids: the vector kernels (init, update, direction) nwgv workgroups of block threads, krv rows each;
    // the hexa20 matrix-free product's gather nwgg of gblock, krg; the assembled product nwgs of krs slices
    int block = 0, krv = 1, nwgv = 0;
    int gblock = 0, krg = 1, nwgg = 0;
    int krs = 1, nwgs = 0;
    double* pb = nullptr;  // second direction vector of the folded iteration
    int ps = 0;  // row stride of the partials array (the largest workgroup count)
    // FP64 and FP32 vector sets
    double *x64 = nullptr, *r64 = nullptr, *z64 = nullptr, *p64 = nullptr, *q64 = nullptr;
    float *x32 = nullptr, *r32 = nullptr, *z32 = nullptr, *p32 = nullptr, *q32 = nullptr;
    double* part = nullptr;  // [6][ps]: pq, rz0, rz1, rr, bb, p.p over the Dirichlet DOFs
    int* flags = nullptr;    // device: [done, nan, iters_local, done of odd iterations]
    double* dscal = nullptr; // device: [tol2, scratch sum, alpha, scratch sum]
    int* hflags = nullptr;   // pinned host copy
    double* hpart = nullptr; // pinned host scalars
    hipStream_t ks = nullptr;
    hipEvent_t evA = nullptr, evB = nullptr, t0 = nullptr, t1 = nullptr;
    hipGraphExec_t graph[4] = {};  // FP64 assembled, FP32 assembled, FP32 matrix-free, FP64 bricks
    int graph_batch[4] = {};
    int graph_block[4] = {};
    // the operator buffers a batch graph was captured with (a graph keeps their addresses)
    const void* graph_ops[4][4] = {};
};

namespace {

// Workgroups of a launch are dealt round-robin to the 8 XCDs of the MI355X, each with
// its own L2.  Renumbering them so that every XCD owns one contiguous range of node
// rows keeps the x gathers of an XCD inside a slab of the mesh (plus halo), which
// fits its L2.  The grid size of these launches is a multiple of 8.
__device__ __forceinline__ int xcd_block() {
    const int per = gridDim.x >> 3;
    return (blockIdx.x & 7) * per + (blockIdx.x >> 3);
}

__host__ __forceinline__ int round8(int n) { return (n + 7) & ~7; }

// Deterministic workgroup sums.  Within a wavefront an xor butterfly: the two lanes of a
// pair add the same two values (a + b == b + a exactly), so after every step all lanes
// hold bitwise identical sums.  Across the BS/64 wavefronts the per-wave sums are added in
// wave order.  One barrier pair per call, however many values are summed together.
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

template <int BS, int K>
__device__ __forceinline__ void block_sums(double (&v)[K], double* sh) {
    constexpr int NW = BS / 64;
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = wave_sum(v[k]);
    if (NW == 1) return;
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
        for (int k = 0; k < K; ++k) sh[k * NW + w] = v[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
        double r = sh[k * NW];
        for (int i = 1; i < NW; ++i) r += sh[k * NW + i];
        v[k] = r;
    }
    __syncthreads();
}

template <int BS>
__device__ __forceinline__ double block_sum(double v, double* sh) {
    double a[1] = {v};
    block_sums<BS, 1>(a, sh);
    return a[0];
}

// Sums of K partial arrays (each n long, at part + offs[k]) in a fixed order, computed
// identically by every workgroup.
template <int BS, int K>
__device__ __forceinline__ void reduce_partials_n(const double* __restrict__ part, const int (&offs)[K], int n,
                                                  double (&out)[K], double* sh) {
#pragma unroll
    for (int k = 0; k < K; ++k) out[k] = 0.0;
    for (int i = threadIdx.x; i < n; i += BS) {
#pragma unroll
        for (int k = 0; k < K; ++k) out[k] += part[offs[k] + i];
    }
    block_sums<BS, K>(out, sh);
}

// reduce_partials_n with a count per array and its first loads (start) apart from the rest; each array's
// sum is formed in the same order as reduce_partials_n would form it.
template <int BS, int K>
struct PartialSums {
    double out[K];
    __device__ __forceinline__ void start(const double* __restrict__ part, const int* offs, const int* ns) {
#pragma unroll
        for (int k = 0; k < K; ++k) out[k] = (int)threadIdx.x < ns[k] ? part[offs[k] + threadIdx.x] : 0.0;
    }
    __device__ __forceinline__ void finish(const double* __restrict__ part, const int* offs, const int* ns, double* sh) {
        int nmax = 0;
#pragma unroll
        for (int k = 0; k < K; ++k) nmax = ns[k] > nmax ? ns[k] : nmax;
        for (int i = threadIdx.x + BS; i < nmax; i += BS) {
#pragma unroll
            for (int k = 0; k < K; ++k)
                if (i < ns[k]) out[k] += part[offs[k] + i];
        }
        block_sums<BS, K>(out, sh);
    }
};

template <int BS>
__device__ __forceinline__ double reduce_partials(const double* __restrict__ part, int n, double* sh) {
    const int offs[1] = {0};
    double out[1];
    reduce_partials_n<BS, 1>(part, offs, n, out, sh);
    return out[0];
}

// y = K x, a workgroup per ks slices, its wavefronts each a range of a slice's blocks (as in the GMRES
// product, gmres.hip); with part, the workgroup's partial of x . y.  One product, a lane per row ->
// 8 wavefronts per slice: hexa8 FP64 20^3 13.6 -> 5.4 us, 48^3 40.2 -> 38.9, 64^3 102 -> 94 (5.9 TB/s),
// hexa20 FP64 6^3 35.7 -> 10.3, 16^3 50.6 -> 26.2; 4 wavefronts the same within 5 %, 2 up to 30 % slower.
// At most 2048 workgroups, whose partials every update adds up: FP32 CG 64^3 63.9 us at 2048, 67.7 at
// 1024, 80^3 121 at 2048, 119 at 4096.
constexpr int kSpmvWaves = 8;

template <typename T>
__global__ __launch_bounds__(64 * kSpmvWaves) void spmv_kernel(int N, const int32_t* __restrict__ slice_off,
                                                               const int32_t* __restrict__ scol,
                                                               const int32_t* __restrict__ slotNode,
                                                               const T* __restrict__ K, const T* __restrict__ x,
                                                               T* __restrict__ y, double* __restrict__ part,
                                                               const int* __restrict__ flags, int ks) {
    constexpr int W = kSpmvWaves;
    __shared__ T sh[W - 1][3][64];
    if (flags && flags[0]) return;
    const int blk = xcd_block(), l = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    double dot = 0.0;
    for (int it = 0; it < ks; ++it) {
        const int s = blk * ks + it;
        if (s * kSlice >= N) break;
        const int ps = s * kSlice + l;  // row slot
        const int o0 = slice_off[s], deg = (slice_off[s + 1] - o0) / kSlice;
        const int n = ps < N ? slotNode[ps] : -1;
        const int32_t* cp = scol + o0 + l;
        const T* kp = K + (int64_t)o0 * 9 + l;
        T y0 = 0, y1 = 0, y2 = 0;
        const int k1 = (wave + 1) * deg / W;
        // matrix values and indices are streamed once per product: non-temporal loads
        // keep them from displacing the gathered x in L2
        if (n >= 0)
#pragma unroll 3
            for (int k = wave * deg / W; k < k1; ++k) {
                const int m = __builtin_nontemporal_load(cp + k * kSlice);
                const T x0 = x[3 * m], x1 = x[3 * m + 1], x2 = x[3 * m + 2];
                const T* v = kp + (int64_t)k * 9 * kSlice;
                T a[9];
#pragma unroll
                for (int i = 0; i < 9; ++i) a[i] = __builtin_nontemporal_load(v + i * kSlice);
                y0 += a[0] * x0 + a[1] * x1 + a[2] * x2;
                y1 += a[3] * x0 + a[4] * x1 + a[5] * x2;
                y2 += a[6] * x0 + a[7] * x1 + a[8] * x2;
            }
        if (it > 0) __syncthreads();  // the first wavefront has read the last slice's sums
        if (wave > 0) {
            sh[wave - 1][0][l] = y0;
            sh[wave - 1][1][l] = y1;
            sh[wave - 1][2][l] = y2;
        }
        __syncthreads();
        if (wave > 0 || n < 0) continue;
#pragma unroll
        for (int w = 0; w < W - 1; ++w) {
            y0 += sh[w][0][l];
            y1 += sh[w][1][l];
            y2 += sh[w][2][l];
        }
        y[3 * n] = y0;
        y[3 * n + 1] = y1;
        y[3 * n + 2] = y2;
        if (part) dot += (double)x[3 * n] * y0 + (double)x[3 * n + 1] * y1 + (double)x[3 * n + 2] * y2;
    }
    if (part && wave == 0) {
        dot = wave_sum(dot);
        if (threadIdx.x == 0) part[blk] = dot;
    }
}

// The iteration of a small assembled system in two launches: the direction (stop test, p = z + beta p)
// in the product that follows it.  Every gather forms its entry of p, the row's owner stores it, and the
// two p alternate, as neighbours still gather the old one.  The first blocks of a row are loaded beside
// the scalars' reduction, once the flag has come with the slice's offsets: behind the loads, the idle
// iterations after the stop read the whole operator (a solve of 2 of 32 iterations at 28^3 FP64 494 us,
// now 247; the iteration is no slower).  What an update ends with is tested by the next launch of this kernel, which
// stores the flag of the update and of the launch after it (doneNext) and reads its own (done): the two
// alternate, so that the wavefronts of a workgroup agree on it.  PCG
// iteration in three launches -> two: hexa8 FP64 525 nodes 11.1 -> 9.4 us, 3375 11.7 -> 9.7, 9261 13.3 ->
// 10.3, 24389 19.0 -> 18.1, 35937 22.4 -> 22.4; FP32 9261 11.1 -> 8.7; hexa20R FP64 2673 19.8 -> 16.0, 26353
// 36.2 -> 29.1.  (On 64^3 the same fold cost more than the launch: a second gathered vector.)
template <typename T>
__global__ __launch_bounds__(64 * kSpmvWaves) void pcg_fold_kernel(
    int N, const int32_t* __restrict__ slice_off, const int32_t* __restrict__ scol,
    const int32_t* __restrict__ slotNode, const T* __restrict__ K, const T* __restrict__ z, const T* __restrict__ p,
    T* __restrict__ pNew, T* __restrict__ q, double* __restrict__ part, int ps, int nvec, int par, int jlocal,
    const double* __restrict__ dtol2, const int* __restrict__ done, int* __restrict__ doneNext,
    int* __restrict__ flags) {
    constexpr int W = kSpmvWaves, U = 4;
    __shared__ T sh[W - 1][3][64];
    __shared__ double sd[3 * W];
    const int s = xcd_block(), l = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const bool slice = s * kSlice < N;
    const int ps_ = s * kSlice + l;  // row slot
    const int n = slice && ps_ < N ? slotNode[ps_] : -1;
    int o0 = 0, k0 = 0, k1 = 0;
    if (slice) {
        o0 = slice_off[s];
        const int deg = (slice_off[s + 1] - o0) / kSlice;
        k0 = wave * deg / W;
        k1 = (wave + 1) * deg / W;
    }
    const int32_t* cp = scol + o0 + l;
    const T* kp = K + (int64_t)o0 * 9 + l;
    T a[U][9], zv[U][3], pv[U][3];
    auto load = [&](int k) {
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (k + u < k1) {  // uniform over the wavefront
                const int m = cp[(k + u) * kSlice];
#pragma unroll
                for (int i = 0; i < 9; ++i) a[u][i] = kp[(int64_t)((k + u) * 9 + i) * kSlice];
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    zv[u][i] = z[3 * m + i];
                    pv[u][i] = p[3 * m + i];
                }
            }
    };
    const bool first = blockIdx.x == 0 && threadIdx.x == 0;
    if (*done) {
        if (first) *doneNext = 1;
        return;
    }
    if (n >= 0) load(k0);
    const int offs[3] = {(1 + par) * ps, (2 - par) * ps, 3 * ps};
    double sc[3];
    reduce_partials_n<64 * W, 3>(part, offs, nvec, sc, sd);
    const double rz = sc[0], rzo = sc[1], rr = sc[2];
    const bool bad = !(rr == rr) || !(rz == rz);
    // the last iteration's result; there is none before the first, whose r.z before is infinite
    const bool stop = bad || (rr <= dtol2[0] && rzo < INFINITY);
    if (first) {
        if (stop) {
            flags[2] = jlocal;
            flags[1] = bad ? 1 : 0;
        }
        *doneNext = stop ? 1 : 0;
    }
    if (stop) return;
    const T beta = (T)(rz / rzo);
    T y0 = 0, y1 = 0, y2 = 0;
    if (n >= 0)
        for (int k = k0; k < k1; k += U) {
            if (k > k0) load(k);
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (k + u < k1) {
                    const T x0 = zv[u][0] + beta * pv[u][0], x1 = zv[u][1] + beta * pv[u][1],
                            x2 = zv[u][2] + beta * pv[u][2];
                    y0 += a[u][0] * x0 + a[u][1] * x1 + a[u][2] * x2;
                    y1 += a[u][3] * x0 + a[u][4] * x1 + a[u][5] * x2;
                    y2 += a[u][6] * x0 + a[u][7] * x1 + a[u][8] * x2;
                }
        }
    if (wave > 0) {
        sh[wave - 1][0][l] = y0;
        sh[wave - 1][1][l] = y1;
        sh[wave - 1][2][l] = y2;
    }
    __syncthreads();
    if (wave > 0) return;
    double dot = 0.0;
    if (n >= 0) {
#pragma unroll
        for (int w = 0; w < W - 1; ++w) {
            y0 += sh[w][0][l];
            y1 += sh[w][1][l];
            y2 += sh[w][2][l];
        }
        const T y[3] = {y0, y1, y2};
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const T v = z[3 * n + i] + beta * p[3 * n + i];
            pNew[3 * n + i] = v;
            q[3 * n + i] = y[i];
            dot += (double)v * y[i];
        }
    }
    dot = wave_sum(dot);
    if (threadIdx.x == 0) part[s] = dot;
}

// x = 0, r = b (b_dir = b on Dirichlet DOFs is part of the system), z = Minv r, p = z,
// partials r.z -> part[1], b.b -> part[4].
template <typename T, int BS, bool DP2 = false>
__global__ __launch_bounds__(BS) void pcg_init_kernel(int N, const double* __restrict__ b, const T* __restrict__ Minv,
                                                      T* __restrict__ x, T* __restrict__ r, T* __restrict__ z,
                                                      T* __restrict__ p, double* __restrict__ part, int ps,
                                                      int* __restrict__ flags, int kr,
                                                      const uint8_t* __restrict__ dirflag = nullptr) {
    __shared__ double sh[BS];
    const int blk = xcd_block();
    double rz = 0, bb = 0, pd = 0;
    for (int it = 0; it < kr; ++it) {
        const int n = (blk * kr + it) * BS + threadIdx.x;
        if (n >= N) break;
        T rv[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            rv[i] = (T)b[3 * n + i];
            x[3 * n + i] = 0;
            r[3 * n + i] = rv[i];
            bb += (double)b[3 * n + i] * b[3 * n + i];
        }
        const T* M = Minv + (int64_t)n * 9;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            T zi = M[3 * i] * rv[0] + M[3 * i + 1] * rv[1] + M[3 * i + 2] * rv[2];
            z[3 * n + i] = zi;
            p[3 * n + i] = zi;
            rz += (double)rv[i] * zi;
            if (DP2 && dirflag[3 * n + i]) pd += (double)zi * zi;
        }
    }
    constexpr int NS = DP2 ? 3 : 2;
    double sums[NS];
    sums[0] = rz;
    sums[1] = bb;
    if constexpr (DP2) sums[2] = pd;
    block_sums<BS, NS>(sums, sh);
    const double s1 = sums[0], s2 = sums[1];
    if (threadIdx.x == 0) {
        part[1 * ps + blk] = s1;
        part[4 * ps + blk] = s2;
        if constexpr (DP2) part[5 * ps + blk] = sums[NS - 1];
        // the folded iteration's beta = r.z / (r.z before) and stop test: 0 and no before the first
        part[2 * ps + blk] = INFINITY;
        part[3 * ps + blk] = INFINITY;
        if (blk == 0) {
            flags[0] = 0;
            flags[1] = 0;
            flags[2] = 0;
            flags[3] = 0;
        }
    }
}

// What the update reads of row n, loaded before the scalars are reduced.  BRICK: q is the sum of the
// node's brick partials (gptr, gF), p on its Dirichlet DOFs; else it is stored (gF).
template <typename T, bool BRICK>
struct UpdateRow {
    T r[3], M[9], q[3];
    __device__ __forceinline__ void load(int n, const T* __restrict__ rv, const T* __restrict__ Minv,
                                         const T* __restrict__ p, const int32_t* __restrict__ gptr,
                                         const T* __restrict__ gF, const uint8_t* __restrict__ dirflag) {
        int g0 = 0, g1 = 0;
        if constexpr (BRICK) {
            g0 = gptr[n];
            g1 = gptr[n + 1];
        }
#pragma unroll
        for (int i = 0; i < 3; ++i) r[i] = rv[3 * (int64_t)n + i];
#pragma unroll
        for (int i = 0; i < 9; ++i) M[i] = Minv[(int64_t)n * 9 + i];
        if constexpr (BRICK) {
            bool d[3];
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                d[i] = dirflag[3 * (int64_t)n + i];
                q[i] = (T)0;
            }
            for (int c = g0; c < g1; ++c)
#pragma unroll
                for (int i = 0; i < 3; ++i) q[i] += gF[3 * (int64_t)c + i];
#pragma unroll
            for (int i = 0; i < 3; ++i)
                if (d[i]) q[i] = p[3 * (int64_t)n + i];
        } else {
#pragma unroll
            for (int i = 0; i < 3; ++i) q[i] = gF[3 * (int64_t)n + i];
        }
    }
};

// B: alpha = r.z / p.q, r -= alpha q, z = Minv r and their partials; p.q = the operator's partials (nop
// of them), on the bricks + the Dirichlet p.p partials.  x waits for C, which reads p anyway; alpha
// goes to *alphaOut.  The first row's loads run beside the scalars' reduction, behind its first loads and
// the flag, which the idle iterations after the stop end at (both kernels: a solve of 2 of 32 iterations
// on the 90^3 FP64 bricks 862 us with the flag behind the row, now 696; the iteration 177.3 and 176.3 us,
// FP32 64^3 39.6 and 39.5).  PCG iteration on the
// bricks with x updated here and the loads behind the reduction -> now (both kernels, and the
// fixed-pitch brick tables): FP64 20^3 20.4 -> 19.3, 40^3 33.0 -> 30.0, 64^3 62.7 -> 59.0 us, FP32 96^3
// 118.4 -> 113.3 us.
// FOLD: x is updated here, after pcg_fold_kernel.
template <typename T, int BS, bool BRICK, bool FOLD = false>
__global__ __launch_bounds__(BS) void pcg_update_kernel(
    int N, const T* __restrict__ Minv, T* __restrict__ r, T* __restrict__ z, const T* __restrict__ p,
    const int32_t* __restrict__ gptr, const T* __restrict__ gF, const uint8_t* __restrict__ dirflag,
    double* __restrict__ part, int ps, int nop, int nvec, int par, const int* __restrict__ done,
    double* __restrict__ alphaOut, int kr,
    T* __restrict__ x = nullptr) {
    __shared__ double sh[BS];
    const int blk = xcd_block();
    int n = blk * kr * BS + threadIdx.x;
    UpdateRow<T, BRICK> row;
    constexpr int NS = BRICK ? 3 : 2;
    const int offs[3] = {0, (1 + par) * ps, 5 * ps};
    const int ns[3] = {nop, nvec, nvec};
    PartialSums<BS, NS> sc;
    sc.start(part, offs, ns);
    if (*done) return;
    if (n < N) row.load(n, r, Minv, p, gptr, gF, dirflag);
    sc.finish(part, offs, ns, sh);
    double pq = sc.out[0];
    if constexpr (BRICK) pq += sc.out[NS - 1];
    const double al = sc.out[1] / pq;
    const T alpha = (T)al;
    if (blk == 0 && threadIdx.x == 0) *alphaOut = al;
    double rzn = 0, rr = 0;
    for (int it = 0; it < kr && n < N; ++it) {
        T rv[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            rv[i] = row.r[i] - alpha * row.q[i];
            r[3 * (int64_t)n + i] = rv[i];
            rr += (double)rv[i] * rv[i];
        }
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const T zi = row.M[3 * i] * rv[0] + row.M[3 * i + 1] * rv[1] + row.M[3 * i + 2] * rv[2];
            z[3 * (int64_t)n + i] = zi;
            rzn += (double)rv[i] * zi;
        }
        if constexpr (FOLD)
#pragma unroll
            for (int i = 0; i < 3; ++i) x[3 * (int64_t)n + i] += alpha * p[3 * (int64_t)n + i];
        n += BS;
        if (it + 1 < kr && n < N) row.load(n, r, Minv, p, gptr, gF, dirflag);
    }
    double sums[2] = {rzn, rr};
    block_sums<BS, 2>(sums, sh);
    if (threadIdx.x == 0) {
        part[(2 - par) * ps + blk] = sums[0];
        part[3 * ps + blk] = sums[1];
    }
}

// C: x += alpha p, the convergence test, p = z + beta p and, on the bricks, the Dirichlet p.p partials.
// As every workgroup has to add its alpha p in the last iteration too, the flag of the next iteration
// (doneNext) is not the one this kernel reads (done): the two alternate.
template <typename T, int BS, bool BRICK>
__global__ __launch_bounds__(BS) void pcg_direction_kernel(
    int N, T* __restrict__ x, const T* __restrict__ z, T* __restrict__ p, double* __restrict__ part, int ps, int nvec,
    int par, int jlocal, const double* __restrict__ dtol2, const double* __restrict__ alphaIn,
    const int* __restrict__ done, int* __restrict__ doneNext, int* __restrict__ flags, int kr,
    const uint8_t* __restrict__ dirflag) {
    __shared__ double sh[BS];
    const int blk = xcd_block();
    int n = blk * kr * BS + threadIdx.x;
    T xv[3], zv[3], pv[3];
    auto load = [&] {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            xv[i] = x[3 * (int64_t)n + i];
            zv[i] = z[3 * (int64_t)n + i];
            pv[i] = p[3 * (int64_t)n + i];
        }
    };
    const int offs[3] = {(1 + par) * ps, (2 - par) * ps, 3 * ps}, ns[3] = {nvec, nvec, nvec};
    PartialSums<BS, 3> sc;
    sc.start(part, offs, ns);
    if (*done) {
        if (blk == 0 && threadIdx.x == 0) *doneNext = 1;
        return;
    }
    if (n < N) load();
    const T alpha = (T)*alphaIn;
    sc.finish(part, offs, ns, sh);
    const double rzo = sc.out[0], rzn = sc.out[1], rr = sc.out[2];
    const bool bad = !(rr == rr) || !(rzn == rzn);
    const bool stop = bad || rr <= dtol2[0];
    if (blk == 0 && threadIdx.x == 0) {
        if (stop) {
            flags[2] = jlocal + 1;
            flags[1] = bad ? 1 : 0;
        }
        *doneNext = stop ? 1 : 0;
    }
    const T beta = (T)(rzn / rzo);
    double pd = 0;
    for (int it = 0; it < kr && n < N; ++it) {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            x[3 * (int64_t)n + i] = xv[i] + alpha * pv[i];
            if (!stop) {
                const T v = zv[i] + beta * pv[i];
                p[3 * (int64_t)n + i] = v;
                if (BRICK && dirflag[3 * (int64_t)n + i]) pd += (double)v * v;
            }
        }
        n += BS;
        if (it + 1 < kr && n < N) load();
    }
    if constexpr (BRICK) {
        const double s = block_sum<BS>(pd, sh);
        if (threadIdx.x == 0) part[5 * ps + blk] = s;
    }
}

// x_out = x (converted), with Dirichlet DOFs taken from b exactly.
template <typename T>
__global__ void pcg_finish_kernel(int D, const T* __restrict__ x, const double* __restrict__ b,
                                  const uint8_t* __restrict__ dirflag, int ndir, double* __restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= D) return;
    out[i] = (ndir && dirflag[i]) ? b[i] : (double)x[i];
}

// Convergence quantities: max|R| (first index on ties), max|ddU|, sum|F|, NaN flag.
template <int BS>
__global__ __launch_bounds__(BS) void norms_stage1(int D, const double* __restrict__ R, const double* __restrict__ ddU,
                                                   const double* __restrict__ F, double* __restrict__ part,
                                                   int nwg) {
    __shared__ double sh[BS / 64 * 5];
    NormSums v;
#pragma unroll 4
    for (int i = blockIdx.x * BS + threadIdx.x; i < D; i += BS * gridDim.x)
        v.add((double)i, R[i], ddU ? ddU[i] : 0.0, F[i]);
    v.reduce<BS / 64>(sh);
    if (threadIdx.x == 0) {
        part[0 * nwg + blockIdx.x] = v.mr;
        part[1 * nwg + blockIdx.x] = v.ir;
        part[2 * nwg + blockIdx.x] = v.md;
        part[3 * nwg + blockIdx.x] = v.sf;
        part[4 * nwg + blockIdx.x] = v.nan;
    }
}

// Fixed-order sum of n partials by one 256-thread workgroup.
__global__ __launch_bounds__(256) void sum_partials_kernel(const double* __restrict__ part, int n,
                                                           double* __restrict__ out) {
    __shared__ double sh[256];
    const double s = reduce_partials<256>(part, n, sh);
    if (threadIdx.x == 0) *out = s;
}

// Final reduction of the per-workgroup norms by one 256-thread workgroup (fixed order).
__global__ __launch_bounds__(256) void norms_stage2(const double* __restrict__ part, int nwg,
                                                    double* __restrict__ out) {
    __shared__ double sh[4 * 5];
    NormSums v;
#pragma unroll 4
    for (int w = threadIdx.x; w < nwg; w += 256) {
        NormSums o;
        o.mr = part[w];
        o.ir = part[nwg + w];
        o.md = part[2 * nwg + w];
        o.sf = part[3 * nwg + w];
        o.nan = part[4 * nwg + w];
        v.merge(o);
    }
    v.reduce<4>(sh);
    if (threadIdx.x == 0) {
        out[0] = v.mr < 0 ? 0.0 : v.mr;
        out[1] = v.mr < 0 ? 0.0 : v.ir;
        out[2] = v.md;
        out[3] = v.sf;
        out[4] = v.nan;
    }
}

// Assembled systems of up to this many nodes take the folded iteration (at 35937 it is no faster).
constexpr int kFoldNodes = 28000;
inline bool fold_iteration(const efe_ctx* c) { return c->N <= kFoldNodes; }

template <typename T, int BS>
void launch_iter(efe_ctx* c, KrylovWork* w, hipStream_t st, T* x, T* r, T* z, T* p, T* q, const T* K,
                 const T* Minv, bool bricks, int par, int j) {
    const int gv = w->nwgv, krv = w->krv;
    const int *done = w->flags + (par ? 3 : 0);
    int* doneNext = w->flags + (par ? 0 : 3);
    if (bricks) {  // hexa8 bricks: the product's partials gathered by the update
        const T* gF;
        if constexpr (sizeof(T) == 8) gF = c->mfbF64;
        else gF = c->mfbF;
        efe_mf_launch_apply_partials(c, st, p, w->part, done);
        pcg_update_kernel<T, BS, true><<<gv, BS, 0, st>>>(c->N, Minv, r, z, p, c->mfbPptr, gF, c->dirflag, w->part,
                                                          w->ps, round8(c->mfbG), gv, par, done, w->dscal + 2, krv);
        pcg_direction_kernel<T, BS, true><<<gv, BS, 0, st>>>(c->N, x, z, p, w->part, w->ps, gv, par, j, w->dscal,
                                                             w->dscal + 2, done, doneNext, w->flags, krv, c->dirflag);
        return;
    }
    int nop = w->nwgg;
    if (K && fold_iteration(c)) {
        nop = w->nwgs;
        T *pa = p, *pb = (T*)w->pb;
        T *pOld = par ? pb : pa, *pNew = par ? pa : pb;
        pcg_fold_kernel<T><<<nop, 64 * kSpmvWaves, 0, st>>>(c->N, c->slice_off, c->scol, c->slotNode, K, z, pOld, pNew, q,
                                                            w->part, w->ps, gv, par, j, w->dscal, done, doneNext,
                                                            w->flags);
        pcg_update_kernel<T, BS, false, true><<<gv, BS, 0, st>>>(c->N, Minv, r, z, pNew, nullptr, q, nullptr, w->part,
                                                                 w->ps, nop, gv, par, doneNext, w->dscal + 2, krv, x);
        return;
    }
    if (K) {
        nop = w->nwgs;
        spmv_kernel<T><<<nop, 64 * kSpmvWaves, 0, st>>>(c->N, c->slice_off, c->scol, c->slotNode, K, p, q, w->part, done,
                                                        w->krs);
    } else {  // matrix-free FP32 operator of hexa20
        efe_mf_launch_operator(c, st, (const float*)p, (float*)q, w->part, done, nop, w->gblock, w->krg);
    }
    pcg_update_kernel<T, BS, false><<<gv, BS, 0, st>>>(c->N, Minv, r, z, p, nullptr, q, nullptr, w->part, w->ps, nop, gv,
                                                       par, done, w->dscal + 2, krv);
    pcg_direction_kernel<T, BS, false><<<gv, BS, 0, st>>>(c->N, x, z, p, w->part, w->ps, gv, par, j, w->dscal,
                                                          w->dscal + 2, done, doneNext, w->flags, krv, nullptr);
}

template <typename T>
void launch_iter_bs(efe_ctx* c, KrylovWork* w, hipStream_t st, T* x, T* r, T* z, T* p, T* q, const T* K,
                    const T* Minv, bool bricks, int par, int j) {
    switch (w->block) {
        case 64: launch_iter<T, 64>(c, w, st, x, r, z, p, q, K, Minv, bricks, par, j); break;
        case 128: launch_iter<T, 128>(c, w, st, x, r, z, p, q, K, Minv, bricks, par, j); break;
        case 512: launch_iter<T, 512>(c, w, st, x, r, z, p, q, K, Minv, bricks, par, j); break;
        default: launch_iter<T, 256>(c, w, st, x, r, z, p, q, K, Minv, bricks, par, j); break;
    }
}

template <typename T>
void launch_init_bs(efe_ctx* c, KrylovWork* w, hipStream_t st, const double* b, const T* Minv, T* x, T* r, T* z,
                    T* p, bool dp2) {
    if (dp2) {  // the brick operator's Dirichlet p.p partials
        switch (w->block) {
            case 64: pcg_init_kernel<T, 64, true><<<w->nwgv, 64, 0, st>>>(c->N, b, Minv, x, r, z, p, w->part, w->ps, w->flags, w->krv, c->dirflag); break;
            case 128: pcg_init_kernel<T, 128, true><<<w->nwgv, 128, 0, st>>>(c->N, b, Minv, x, r, z, p, w->part, w->ps, w->flags, w->krv, c->dirflag); break;
            case 512: pcg_init_kernel<T, 512, true><<<w->nwgv, 512, 0, st>>>(c->N, b, Minv, x, r, z, p, w->part, w->ps, w->flags, w->krv, c->dirflag); break;
            default: pcg_init_kernel<T, 256, true><<<w->nwgv, 256, 0, st>>>(c->N, b, Minv, x, r, z, p, w->part, w->ps, w->flags, w->krv, c->dirflag); break;
        }
        return;
    }
    switch (w->block) {
        case 64: pcg_init_kernel<T, 64><<<w->nwgv, 64, 0, st>>>(c->N, b, Minv, x, r, z, p, w->part, w->ps, w->flags, w->krv); break;
        case 128: pcg_init_kernel<T, 128><<<w->nwgv, 128, 0, st>>>(c->N, b, Minv, x, r, z, p, w->part, w->ps, w->flags, w->krv); break;
        case 512: pcg_init_kernel<T, 512><<<w->nwgv, 512, 0, st>>>(c->N, b, Minv, x, r, z, p, w->part, w->ps, w->flags, w->krv); break;
        default: pcg_init_kernel<T, 256><<<w->nwgv, 256, 0, st>>>(c->N, b, Minv, x, r, z, p, w->part, w->ps, w->flags, w->krv); break;
    }
}

int ensure_work(efe_ctx* c) {
    int block = c->kblock;
    // Unless set: small meshes' rows over as many CUs as they give wavefronts.  PCG iteration at 64 / 128
    // / 256 / 512: 525 nodes 10.9 / 11.4 / 11.6 / 12.7 us, 3375 11.8 / 12.0 / 12.4 / 13.5, 9261 14.2 / 13.2 / 13.4 /
    // 14.2, 274625 76.7 / 63.4 / 59.3 / 63.4.
    if (block <= 0) block = c->N <= 4096 ? 64 : 256;
    if (block != 64 && block != 128 && block != 256 && block != 512) block = 256;
    // Unless set, the gather of the hexa20 matrix-free product keeps 256 at every size: at 64 a lane stages
    // four times as many force slots, and the LDS that holds them serves one wavefront.  PCG iteration at 64
    // / 256: C3D20 81 nodes 66.2 / 60.5 us, 2673 68.6 / 63.7; C3D20R 81 35.2 / 29.8, 2673 41.0 / 36.2.
    const int gblock = c->kblock > 0 ? block : 256;
    KrylovWork* w = c->kw;
    // the brick operator writes one p.Kp partial per brick into the partials array
    const int need = c->mfb ? round8(c->mfbG) : 0;
    if (w && w->block == block && w->gblock == gblock && w->ps >= need) return EFE_OK;
    if (!w) {
        w = new KrylovWork();
        c->kw = w;
        w->D = c->D;
        w->N = c->N;
        size_t D = (size_t)c->D;
        EFE_HIP(hipMalloc(&w->x64, D * sizeof(double)));
        EFE_HIP(hipMalloc(&w->r64, D * sizeof(double)));
        EFE_HIP(hipMalloc(&w->z64, D * sizeof(double)));
        EFE_HIP(hipMalloc(&w->p64, D * sizeof(double)));
        EFE_HIP(hipMalloc(&w->q64, D * sizeof(double)));
        EFE_HIP(hipMalloc(&w->x32, D * sizeof(float)));
        EFE_HIP(hipMalloc(&w->r32, D * sizeof(float)));
        EFE_HIP(hipMalloc(&w->z32, D * sizeof(float)));
        EFE_HIP(hipMalloc(&w->p32, D * sizeof(float)));
        EFE_HIP(hipMalloc(&w->q32, D * sizeof(float)));
        EFE_HIP(hipMalloc(&w->flags, 4 * sizeof(int)));
        EFE_HIP(hipMalloc(&w->dscal, 4 * sizeof(double)));
        if (fold_iteration(c)) EFE_HIP(hipMalloc(&w->pb, D * sizeof(double)));
        EFE_HIP(hipHostMalloc(&w->hflags, 4 * sizeof(int), hipHostMallocDefault));
        EFE_HIP(hipHostMalloc(&w->hpart, 8 * sizeof(double), hipHostMallocDefault));
        EFE_HIP(hipStreamCreateWithFlags(&w->ks, hipStreamNonBlocking));
        EFE_HIP(hipEventCreateWithFlags(&w->evA, hipEventDisableTiming));
        EFE_HIP(hipEventCreateWithFlags(&w->evB, hipEventDisableTiming));
        EFE_HIP(hipEventCreate(&w->t0));
        EFE_HIP(hipEventCreate(&w->t1));
    }
    for (int i = 0; i < 4; ++i) {
        if (w->graph[i]) hipGraphExecDestroy(w->graph[i]);
        w->graph[i] = nullptr;
    }
    if (w->part) hipFree(w->part);
    w->block = block;
    w->gblock = gblock;
    // bounded workgroup counts: every workgroup re-reduces all partials in a fixed order, so their number
    // must stay bounded at any mesh size (uncapped, the reductions dominate at 96^3).  The vector kernels
    // stream less per row than the product and re-reduce every partial of the previous kernel in every
    // workgroup, so they take at most 512 workgroups of several rows per thread.  Measured at 64^3 (history
    // Krylov iteration, FP64 / mixed): the product's grid 125.6 / 48.6 us, at most 512 123.7 / 47.4, 256
    // 123.1 / 47.4, 128 125.9 / 49.7.  The FP32 operators are fastest with at most ~1024.
    auto grid = [&](int threads, int cap, int* rows, int* wgs) {
        *rows = ((c->N + threads - 1) / threads + cap - 1) / cap;
        *wgs = round8((c->N + threads * *rows - 1) / (threads * *rows));
    };
    grid(block, 512, &w->krv, &w->nwgv);
    grid(gblock, 1024, &w->krg, &w->nwgg);
    const int slices = (c->N + kSlice - 1) / kSlice, scap = 2048;
    w->krs = (slices + scap - 1) / scap;
    w->nwgs = round8((slices + w->krs - 1) / w->krs);
    w->ps = std::max(std::max(w->nwgv, w->nwgg), std::max(w->nwgs, need));
    EFE_HIP(hipMalloc(&w->part, (size_t)6 * w->ps * sizeof(double)));
    return EFE_OK;
}

template <typename T>
int pcg_solve(efe_ctx* c, const double* b, double* xout, const efe_solve_opts* o, efe_solve_info* info, T* x, T* r,
              T* z, T* p, T* q, const T* K, const T* Minv, bool bricks, int gi) {
    KrylovWork* w = c->kw;
    hipStream_t st = w->ks;
    // order after the caller's stream
    EFE_HIP(hipEventRecord(w->evA, c->stream));
    EFE_HIP(hipStreamWaitEvent(st, w->evA, 0));
    launch_init_bs<T>(c, w, st, b, Minv, x, r, z, p, bricks);
    EFE_HIP(hipGetLastError());
    // b.b (host) to fix the absolute tolerance
    sum_partials_kernel<<<1, 256, 0, st>>>(w->part + 4 * w->ps, w->nwgv, w->dscal + 1);
    EFE_HIP(hipMemcpyAsync(w->hpart, w->dscal + 1, sizeof(double), hipMemcpyDeviceToHost, st));
    EFE_HIP(hipStreamSynchronize(st));
    const double bnorm = sqrt(w->hpart[0]);
    info->rhs_norm = bnorm;
    info->iterations = 0;
    info->status = EFE_OK;
    info->residual = bnorm;
    const int D = c->D;
    if (bnorm == 0.0 || !(bnorm == bnorm)) {
        pcg_finish_kernel<T><<<(D + 255) / 256, 256, 0, st>>>(D, x, b, c->dirflag, c->ndir, xout);
        EFE_HIP(hipEventRecord(w->evB, st));
        EFE_HIP(hipStreamWaitEvent(c->stream, w->evB, 0));
        if (!(bnorm == bnorm)) info->status = EFE_NAN;
        return EFE_OK;
    }
    const double tol = fmax(o->rtol * bnorm, o->atol);
    const double tol2 = tol * tol;
    int batch = o->check_every > 0 ? o->check_every : 16;
    if (batch & 1) batch += 1;
    const int maxit = o->max_iter > 0 ? o->max_iter : 10000;
    w->hpart[1] = tol2;
    EFE_HIP(hipMemcpyAsync(w->dscal, w->hpart + 1, sizeof(double), hipMemcpyHostToDevice, st));
    // (re)build the captured batch when its shape or an operator buffer changed
    const void* ops[4] = {K, Minv, sizeof(T) == 8 ? (void*)c->mfC64 : (void*)c->mfC,
                          sizeof(T) == 8 ? (void*)c->mfbF64 : (void*)c->mfbF};
    bool same = true;
    for (int i = 0; i < 4; ++i) same = same && w->graph_ops[gi][i] == ops[i];
    if (!w->graph[gi] || w->graph_batch[gi] != batch || w->graph_block[gi] != w->block || !same) {
        if (w->graph[gi]) hipGraphExecDestroy(w->graph[gi]);
        w->graph[gi] = nullptr;
        hipGraph_t g;
        EFE_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeRelaxed));
        for (int j = 0; j < batch; ++j) launch_iter_bs<T>(c, w, st, x, r, z, p, q, K, Minv, bricks, j & 1, j);
        EFE_HIP(hipStreamEndCapture(st, &g));
        EFE_HIP(hipGraphInstantiate(&w->graph[gi], g, nullptr, nullptr, 0));
        EFE_HIP(hipGraphDestroy(g));
        w->graph_batch[gi] = batch;
        w->graph_block[gi] = w->block;
        for (int i = 0; i < 4; ++i) w->graph_ops[gi][i] = ops[i];
    }
    int it = 0;
    EFE_HIP(hipEventRecord(w->t0, st));
    while (true) {
        EFE_HIP(hipGraphLaunch(w->graph[gi], st));
        EFE_HIP(hipMemcpyAsync(w->hflags, w->flags, 3 * sizeof(int), hipMemcpyDeviceToHost, st));
        EFE_HIP(hipStreamSynchronize(st));
        if (w->hflags[0]) {
            it += w->hflags[2];
            if (w->hflags[1]) info->status = EFE_NAN;
            break;
        }
        it += batch;
        if (it >= maxit) {
            info->status = EFE_NOT_CONVERGED;
            break;
        }
    }
    EFE_HIP(hipEventRecord(w->t1, st));
    pcg_finish_kernel<T><<<(D + 255) / 256, 256, 0, st>>>(D, x, b, c->dirflag, c->ndir, xout);
    EFE_HIP(hipGetLastError());
    EFE_HIP(hipEventRecord(w->evB, st));
    EFE_HIP(hipStreamWaitEvent(c->stream, w->evB, 0));
    // final residual of the recursion
    sum_partials_kernel<<<1, 256, 0, st>>>(w->part + 3 * w->ps, w->nwgv, w->dscal + 1);
    EFE_HIP(hipMemcpyAsync(w->hpart, w->dscal + 1, sizeof(double), hipMemcpyDeviceToHost, st));
    // a folded iteration's result is tested by the next one: that of the last iteration allowed here, by its
    // r.r and r.z (the r.z of odd iterations, as a batch ends with one)
    const bool untested = info->status == EFE_NOT_CONVERGED && K && fold_iteration(c);
    if (untested) {
        sum_partials_kernel<<<1, 256, 0, st>>>(w->part + w->ps, w->nwgv, w->dscal + 3);
        EFE_HIP(hipMemcpyAsync(w->hpart + 1, w->dscal + 3, sizeof(double), hipMemcpyDeviceToHost, st));
    }
    EFE_HIP(hipStreamSynchronize(st));
    info->residual = sqrt(w->hpart[0]);
    if (untested) {
        if (!(w->hpart[0] == w->hpart[0]) || !(w->hpart[1] == w->hpart[1])) info->status = EFE_NAN;
        else if (w->hpart[0] <= tol2) info->status = EFE_OK;
    }
    info->iterations = it;
    float ms = 0;
    hipEventElapsedTime(&ms, w->t0, w->t1);
    c->t_kry = it > 0 ? ms / it : 0.0;
    c->tot[EFE_T_KRYLOV] += ms;
    c->tot[EFE_T_KRYLOV_ITERS] += it;
    c->tot[EFE_T_SOLVES] += 1;
    return EFE_OK;
}

}  // namespace

int efe_krylov_solve(efe_ctx* c, const double* b, double* x, const efe_solve_opts* o, efe_solve_info* info) {
    if (c->Kprec < 0) {
        efe_set_error("no assembled operator: call efe_compute_elements first");
        return EFE_ERR_STATE;
    }
    if (o->precision != c->Kprec) {
        efe_set_error("solve precision differs from the precision K was assembled in");
        return EFE_ERR_ARG;
    }
    if (o->precision == EFE_FP32_MATFREE && (o->solver != EFE_SOLVER_CG || o->precond != EFE_PRECOND_BLOCK_JACOBI)) {
        efe_set_error("the matrix-free operator runs with block-Jacobi CG");
        return EFE_ERR_ARG;
    }
    if (o->solver == EFE_SOLVER_GMRES) return efe_gmres_solve(c, b, x, o, info);
    if (o->solver != EFE_SOLVER_CG || o->precond != EFE_PRECOND_BLOCK_JACOBI) {
        efe_set_error("CG runs with the block-Jacobi preconditioner (ILU(0) is available with GMRES)");
        return EFE_ERR_ARG;
    }
    int rc = ensure_work(c);
    if (rc != EFE_OK) return rc;
    KrylovWork* w = c->kw;
    if (o->precision == EFE_FP32_MATFREE)
        return pcg_solve<float>(c, b, x, o, info, w->x32, w->r32, w->z32, w->p32, w->q32, nullptr, c->Minv32, c->mfb, 2);
    if (o->precision == EFE_FP32)
        return pcg_solve<float>(c, b, x, o, info, w->x32, w->r32, w->z32, w->p32, w->q32, c->K32, c->Minv32, false, 1);
    // hexa8 with a symmetric tangent: the FP64 brick product moves 614 bytes per element where the
    // assembled one moves 2135.  PCG iteration at 32^3 / 40^3 / 64^3: 22.4 / 39.5 / 118 us assembled,
    // 22.2 / 30.0 / 59.0 us on the bricks.  The assembled operator serves smaller meshes
    // (kSplitElements), the other elements and materials, and a Dirichlet set changed since the pass.
    if (efe_mf_bricks64(c))
        return pcg_solve<double>(c, b, x, o, info, w->x64, w->r64, w->z64, w->p64, w->q64, nullptr, c->Minv64, true, 3);
    return pcg_solve<double>(c, b, x, o, info, w->x64, w->r64, w->z64, w->p64, w->q64, c->K64, c->Minv64, false, 0);
}

int efe_launch_spmv64(efe_ctx* c, const double* x, double* y) {
    if (c->Kprec != EFE_FP64) {
        efe_set_error("efe_spmv needs an FP64 operator");
        return EFE_ERR_STATE;
    }
    spmv_kernel<double><<<round8((c->N + kSlice - 1) / kSlice), 64 * kSpmvWaves, 0, c->stream>>>(
        c->N, c->slice_off, c->scol, c->slotNode, c->K64, x, y, nullptr, nullptr, 1);
    EFE_HIP(hipGetLastError());
    return EFE_OK;
}

int efe_launch_norms(efe_ctx* c, const double* R, const double* ddU, const double* F, double* out) {
    const int BS = 256;
    int nwg = (c->D + BS - 1) / BS;
    if (nwg > 1024) nwg = 1024;
    norms_stage1<BS><<<nwg, BS, 0, c->stream>>>(c->D, R, ddU, F, c->red + 8, nwg);
    norms_stage2<<<1, 256, 0, c->stream>>>(c->red + 8, nwg, c->red);
    EFE_HIP(hipGetLastError());
    EFE_HIP(hipMemcpyAsync(out, c->red, 5 * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    EFE_HIP(hipStreamSynchronize(c->stream));
    return EFE_OK;
}


void efe_krylov_free(efe_ctx* c) {
    KrylovWork* w = c->kw;
    if (!w) return;
    for (int i = 0; i < 4; ++i)
        if (w->graph[i]) hipGraphExecDestroy(w->graph[i]);
    hipFree(w->x64); hipFree(w->r64); hipFree(w->z64); hipFree(w->p64); hipFree(w->q64);
    hipFree(w->x32); hipFree(w->r32); hipFree(w->z32); hipFree(w->p32); hipFree(w->q32);
    hipFree(w->part); hipFree(w->flags); hipFree(w->dscal); hipFree(w->pb);
    hipHostFree(w->hflags); hipHostFree(w->hpart);
    if (w->ks) hipStreamDestroy(w->ks);
    if (w->evA) hipEventDestroy(w->evA);
    if (w->evB) hipEventDestroy(w->evB);
    if (w->t0) hipEventDestroy(w->t0);
    if (w->t1) hipEventDestroy(w->t1);
    delete w;
    c->kw = nullptr;
}
