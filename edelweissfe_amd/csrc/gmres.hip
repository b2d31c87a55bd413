// GMRES(m) with multicolor block ILU(0) or block-Jacobi right preconditioning, for the
// non-symmetric tangents of non-associative plasticity, in place of the reference's
// unsymmetric direct solve (PARDISO mtype 11, linsolve/pardiso/pardiso.pyx:104-151).
//
// Block ILU(0): the zero-fill incomplete factorisation on the 3x3-block pattern of K, in
// the elimination order (color, node) of a greedy coloring of the node graph.  The
// factor is formed in block CSR with rows in that order, so every color is one contiguous
// range of mutually independent rows: the factorisation and both triangular sweeps take
// one launch per color (8 on a hexa8 grid) instead of one per dependency level.  The sweeps
// read a copy of it in slices.
//
// GMRES: right preconditioning (the Arnoldi residual is the true residual of K x = b),
// classical Gram-Schmidt with one re-orthogonalisation (all projections of a step in one
// pass over the basis), Givens rotations on the host, which the device writes each step's
// projections to and runs one step ahead of.
#include <algorithm>
#include <array>
#include <cstdlib>
#include <cmath>
#include <cstring>
#include <vector>

#include "efe_internal.h"

// One color of a sweep: slices of 64 / G rows by decreasing length, so step k belongs to the first
// count[k] slices, at base[k] + slice; kernel arguments, so that no load waits for an offset.
constexpr int kSweepLevels = 8;
struct SweepColor {
    int slices = 0, levels = 0, row0 = 0, more = 0, G = 0;  // more: first of levels kSweepLevels.. in Sweep::more
    int base[kSweepLevels] = {}, count[kSweepLevels] = {};
};

struct GmresWork {
    int D = 0, N = 0, m = 0, nwg = 0;
    // ILU structure
    bool ilu_ready = false;
    int ncolors = 0;
    std::vector<int> cstart;
    std::vector<int> cup;  // per color: most blocks after the diagonal in a row
    int32_t *fptr = nullptr, *fcol = nullptr, *fidx = nullptr, *dslot = nullptr, *perm = nullptr;
    int64_t nbF = 0;
    int maxUpper = 0;  // most blocks in a row's upper part
    int maxRow = 0;    // most blocks in a row
    double *F64 = nullptr, *Dinv64 = nullptr;
    float *F32 = nullptr, *Dinv32 = nullptr;
    int factored_version[2] = {-1, -1};
    // the sweeps' copy of the factor: [0] the blocks before the diagonal, [1] those after it
    struct Sweep {
        std::vector<SweepColor> color;
        int64_t steps = 0;
        int2* rows = nullptr;          // [slices][64/G] (node, factor row), node -1: none
        int2* more = nullptr;          // levels past SweepColor's own: (first step, slices)
        int32_t *col = nullptr, *src = nullptr;  // [steps][64] node of the entry (kNoBlock: none), its block
        double* v64 = nullptr;         // [steps][9][64]
        float* v32 = nullptr;
    } sweep[2];
    // Krylov basis and work vectors (one precision at a time)
    void* V = nullptr;   // [(m+1)][D]
    void* w = nullptr;
    void* z = nullptr;
    void* x = nullptr;
    int vprec = -1;
    double *part = nullptr, *pnorm = nullptr;  // [(m+1)][nwg]; behind it the partial norms
    double* hdev = nullptr;  // [m+2]: ||w||^2 of a start, coefficients of the solution
    double* hhost = nullptr; // pinned, [2][3][m+2]: h1, h2, ||w||^2 of the even and the odd steps
    hipEvent_t step[2] = {nullptr, nullptr};  // their ends
    hipStream_t ks = nullptr;
    hipEvent_t evA = nullptr, evB = nullptr;
    hipEvent_t t0 = nullptr, t1 = nullptr, t2 = nullptr;  // timing: solve start, factor done, end
    // one captured hipGraph per Arnoldi step j (the launches between two readbacks) and the
    // pointers and sizes it was captured with
    std::vector<hipGraphExec_t> stepGraph;
    std::vector<std::array<int64_t, 8>> stepKey;
};

namespace {
void drop_step_graphs(GmresWork* g) {
    for (hipGraphExec_t& e : g->stepGraph)
        if (e) hipGraphExecDestroy(e);
    g->stepGraph.clear();
    g->stepKey.clear();
}
}  // namespace

namespace {

constexpr int BS = 256;
constexpr int kFactorCap = 128;  // upper-part blocks of a row the LDS factor kernel stages

__device__ __forceinline__ int xcd_block_g() {
    const int per = gridDim.x >> 3;
    return (blockIdx.x & 7) * per + (blockIdx.x >> 3);
}

inline int round8g(int n) { return (n + 7) & ~7; }

__device__ __forceinline__ double bsum(double v, double* sh) {
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int s = BS / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
        __syncthreads();
    }
    double r = sh[0];
    __syncthreads();
    return r;
}

template <typename T>
__device__ __forceinline__ void mat3mul(const T* a, const T* b, T* o) {
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) o[i * 3 + j] = a[i * 3] * b[j] + a[i * 3 + 1] * b[3 + j] + a[i * 3 + 2] * b[6 + j];
}

__device__ __forceinline__ void inv3d(const double m[9], double o[9]) {
    const double det = m[0] * (m[4] * m[8] - m[5] * m[7]) - m[1] * (m[3] * m[8] - m[5] * m[6]) +
                       m[2] * (m[3] * m[7] - m[4] * m[6]);
    const double id = 1.0 / det;
    o[0] = (m[4] * m[8] - m[5] * m[7]) * id;
    o[1] = (m[2] * m[7] - m[1] * m[8]) * id;
    o[2] = (m[1] * m[5] - m[2] * m[4]) * id;
    o[3] = (m[5] * m[6] - m[3] * m[8]) * id;
    o[4] = (m[0] * m[8] - m[2] * m[6]) * id;
    o[5] = (m[2] * m[3] - m[0] * m[5]) * id;
    o[6] = (m[3] * m[7] - m[4] * m[6]) * id;
    o[7] = (m[1] * m[6] - m[0] * m[7]) * id;
    o[8] = (m[0] * m[4] - m[1] * m[3]) * id;
}

// F <- K in the factor's block-CSR order (thread per operator node row).
template <typename T>
__global__ __launch_bounds__(BS) void ilu_copy_kernel(int N, const int32_t* __restrict__ bptr,
                                                      const int32_t* __restrict__ slice_off,
                                                      const int32_t* __restrict__ nodeSlot,
                                                      const T* __restrict__ K, const int32_t* __restrict__ fidx,
                                                      T* __restrict__ F) {
    const int n = blockIdx.x * BS + threadIdx.x;
    if (n >= N) return;
    const int ps = nodeSlot[n];
    const int s = ps / kSlice, l = ps - (ps / kSlice) * kSlice;
    const int64_t vb = (int64_t)slice_off[s] * 9 + l;
    const int b0 = bptr[n], nb = bptr[n + 1] - b0;
    // several blocks in flight per lane; measured on the 48^3 hexa20 operator: FP64 2.25 / 1.98
    // / 2.66 ms at 1 / 4 / 8 blocks, FP32 1.44 / 1.20 / 1.04 ms
    constexpr int kUnroll = sizeof(T) == 8 ? 4 : 8;
#pragma unroll kUnroll
    for (int k = 0; k < nb; ++k) {
        T* dst = F + (int64_t)fidx[b0 + k] * 9;
#pragma unroll
        for (int v = 0; v < 9; ++v) dst[v] = K[vb + (int64_t)(k * 9 + v) * kSlice];
    }
}

// Rows [r0, r1) of one color: IKJ block ILU(0).  Rows k < i in elimination order are final.
// A group of G lanes works on one row; the row's block at position p belongs to lane
// (p - b0) % G, which alone reads and writes it.  For each k in the row's lower part
// (in order) the owner of (i, k) forms L_ik = A_ik Dinv_k and broadcasts it; every lane
// then updates its own blocks (i, j), j after k, for which (k, j) is in row k's upper part
// (binary search: a row's columns are sorted in elimination order).
template <typename T, int G>
__global__ __launch_bounds__(BS) void ilu_factor_kernel(int r0, int r1, const int32_t* __restrict__ fptr,
                                                        const int32_t* __restrict__ fcol,
                                                        const int32_t* __restrict__ dslot, T* __restrict__ F,
                                                        T* __restrict__ Dinv) {
    const int tid = blockIdx.x * BS + threadIdx.x;
    const int i = r0 + tid / G, lane = tid % G;
    if (i >= r1) return;  // a whole group leaves together
    const int b0 = fptr[i], b1 = fptr[i + 1], d = b0 + dslot[i];
    for (int kb = b0; kb < d; ++kb) {
        const int k = fcol[kb];
        const int owner = (kb - b0) % G;
        T lik[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
        if (lane == owner) {
            T a[9];
#pragma unroll
            for (int v = 0; v < 9; ++v) a[v] = F[(int64_t)kb * 9 + v];
            mat3mul(a, Dinv + (int64_t)k * 9, lik);
#pragma unroll
            for (int v = 0; v < 9; ++v) F[(int64_t)kb * 9 + v] = lik[v];
        }
#pragma unroll
        for (int v = 0; v < 9; ++v) lik[v] = __shfl(lik[v], owner, G);
        const int u0 = fptr[k] + dslot[k] + 1, u1 = fptr[k + 1];
        const int first = kb + 1 + ((lane - (kb + 1 - b0) % G) % G + G) % G;  // first owned position > kb
        for (int jb = first; jb < b1; jb += G) {
            const int cj = fcol[jb];
            int lo = u0, hi = u1;
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (fcol[mid] < cj) lo = mid + 1;
                else hi = mid;
            }
            if (lo < u1 && fcol[lo] == cj) {
                T u[9], p[9];
#pragma unroll
                for (int v = 0; v < 9; ++v) u[v] = F[(int64_t)lo * 9 + v];
                mat3mul(lik, u, p);
#pragma unroll
                for (int v = 0; v < 9; ++v) F[(int64_t)jb * 9 + v] -= p[v];
            }
        }
    }
    if (lane == (d - b0) % G) {
        double dd[9], di[9];
#pragma unroll
        for (int v = 0; v < 9; ++v) dd[v] = (double)F[(int64_t)d * 9 + v];
        inv3d(dd, di);
#pragma unroll
        for (int v = 0; v < 9; ++v) Dinv[(int64_t)i * 9 + v] = (T)di[v];
    }
}

// ilu_factor_kernel with row k's upper column list staged in LDS: the G lanes of a row load it
// together (coalesced), then each searches its columns there instead of through dependent
// global loads.  The same updates in the same order: the factor is bitwise identical.
// Needs every row's upper part to hold at most CAP blocks.
template <typename T, int G, int CAP>
__global__ __launch_bounds__(BS) void ilu_factor_lds_kernel(int r0, int r1, const int32_t* __restrict__ fptr,
                                                            const int32_t* __restrict__ fcol,
                                                            const int32_t* __restrict__ dslot, T* __restrict__ F,
                                                            T* __restrict__ Dinv) {
    __shared__ int32_t cols[(BS / G) * CAP];
    const int tid = blockIdx.x * BS + threadIdx.x;
    const int i = r0 + tid / G, lane = tid % G;
    int32_t* kc = cols + (threadIdx.x / G) * CAP;  // this row group's list (groups lie inside one wave)
    if (i >= r1) return;  // a whole group leaves together
    const int b0 = fptr[i], b1 = fptr[i + 1], d = b0 + dslot[i];
    for (int kb = b0; kb < d; ++kb) {
        const int k = fcol[kb];
        const int owner = (kb - b0) % G;
        const int u0 = fptr[k] + dslot[k] + 1, nu = fptr[k + 1] - u0;
        for (int t = lane; t < nu; t += G) kc[t] = fcol[u0 + t];
        T lik[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
        if (lane == owner) {
            T a[9];
#pragma unroll
            for (int v = 0; v < 9; ++v) a[v] = F[(int64_t)kb * 9 + v];
            mat3mul(a, Dinv + (int64_t)k * 9, lik);
#pragma unroll
            for (int v = 0; v < 9; ++v) F[(int64_t)kb * 9 + v] = lik[v];
        }
#pragma unroll
        for (int v = 0; v < 9; ++v) lik[v] = __shfl(lik[v], owner, G);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const int first = kb + 1 + ((lane - (kb + 1 - b0) % G) % G + G) % G;  // first owned position > kb
        for (int jb = first; jb < b1; jb += G) {
            const int cj = fcol[jb];
            int lo = 0, hi = nu;
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (kc[mid] < cj) lo = mid + 1;
                else hi = mid;
            }
            if (lo < nu && kc[lo] == cj) {
                T u[9], p[9];
                const int64_t ub = (int64_t)(u0 + lo) * 9;
#pragma unroll
                for (int v = 0; v < 9; ++v) u[v] = F[ub + v];
                mat3mul(lik, u, p);
#pragma unroll
                for (int v = 0; v < 9; ++v) F[(int64_t)jb * 9 + v] -= p[v];
            }
        }
        // every lane's searches are done before the list is overwritten
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    if (lane == (d - b0) % G) {
        double dd[9], di[9];
#pragma unroll
        for (int v = 0; v < 9; ++v) dd[v] = (double)F[(int64_t)d * 9 + v];
        inv3d(dd, di);
#pragma unroll
        for (int v = 0; v < 9; ++v) Dinv[(int64_t)i * 9 + v] = (T)di[v];
    }
}

// ilu_factor_lds_kernel with the row's own blocks held in registers: the G lanes of a row own
// its blocks b0 + lane + t G (t < NT) from the start, update them there and write them once at
// the end.  What remains per elimination step k is k's upper column list (LDS), Dinv_k and the
// U_kj blocks the row meets.  The same updates in the same order as ilu_factor_kernel: the
// factor is bitwise identical.  Needs rows of at most G NT blocks and upper parts of at most
// CAP blocks.
template <typename T, int G, int NT, int CAP>
__global__ __launch_bounds__(BS) void ilu_factor_reg_kernel(int r0, int r1, const int32_t* __restrict__ fptr,
                                                            const int32_t* __restrict__ fcol,
                                                            const int32_t* __restrict__ dslot, T* __restrict__ F,
                                                            T* __restrict__ Dinv) {
    __shared__ int32_t cols[(BS / G) * CAP];
    const int tid = blockIdx.x * BS + threadIdx.x;
    const int i = r0 + tid / G, lane = tid % G;
    int32_t* kc = cols + (threadIdx.x / G) * CAP;
    if (i >= r1) return;  // a whole group leaves together
    const int b0 = fptr[i], b1 = fptr[i + 1], d = b0 + dslot[i];
    T blk[NT][9];
    int col[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int jb = b0 + lane + t * G;
        col[t] = jb < b1 ? fcol[jb] : -1;
#pragma unroll
        for (int v = 0; v < 9; ++v) blk[t][v] = jb < b1 ? F[(int64_t)jb * 9 + v] : (T)0;
    }
    for (int kb = b0; kb < d; ++kb) {
        const int rel = kb - b0, owner = rel % G, tk = rel / G;
        int ck = 0;
#pragma unroll
        for (int t = 0; t < NT; ++t)
            if (t == tk) ck = col[t];
        const int k = __shfl(ck, owner, G);
        const int u0 = fptr[k] + dslot[k] + 1, nu = fptr[k + 1] - u0;
        for (int t = lane; t < nu; t += G) kc[t] = fcol[u0 + t];
        T lik[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
        if (lane == owner) {
            T a[9];
#pragma unroll
            for (int t = 0; t < NT; ++t)
                if (t == tk)
#pragma unroll
                    for (int v = 0; v < 9; ++v) a[v] = blk[t][v];
            mat3mul(a, Dinv + (int64_t)k * 9, lik);
#pragma unroll
            for (int t = 0; t < NT; ++t)
                if (t == tk)
#pragma unroll
                    for (int v = 0; v < 9; ++v) blk[t][v] = lik[v];
        }
#pragma unroll
        for (int v = 0; v < 9; ++v) lik[v] = __shfl(lik[v], owner, G);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int jb = b0 + lane + t * G;
            if (jb <= kb || jb >= b1) continue;
            const int cj = col[t];
            int lo = 0, hi = nu;
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (kc[mid] < cj) lo = mid + 1;
                else hi = mid;
            }
            if (lo < nu && kc[lo] == cj) {
                T u[9], p[9];
                const int64_t ub = (int64_t)(u0 + lo) * 9;
#pragma unroll
                for (int v = 0; v < 9; ++v) u[v] = F[ub + v];
                mat3mul(lik, u, p);
#pragma unroll
                for (int v = 0; v < 9; ++v) blk[t][v] -= p[v];
            }
        }
        // every lane's searches are done before the list is overwritten
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int jb = b0 + lane + t * G;
        if (jb >= b1) continue;
#pragma unroll
        for (int v = 0; v < 9; ++v) F[(int64_t)jb * 9 + v] = blk[t][v];
        if (jb == d) {
            double dd[9], di[9];
#pragma unroll
            for (int v = 0; v < 9; ++v) dd[v] = (double)blk[t][v];
            inv3d(dd, di);
#pragma unroll
            for (int v = 0; v < 9; ++v) Dinv[(int64_t)i * 9 + v] = (T)di[v];
        }
    }
}

// Sum of the 3-vectors of a group of G lanes (fixed butterfly order).
template <typename T, int G>
__device__ __forceinline__ void group_sum3(T& a, T& b, T& c) {
#pragma unroll
    for (int off = G / 2; off > 0; off >>= 1) {
        a += __shfl_xor(a, off, G);
        b += __shfl_xor(b, off, G);
        c += __shfl_xor(c, off, G);
    }
}

// ---- triangular sweeps ---------------------------------------------------------------------------
//
// A color is 1/20 of a hexa20 mesh's rows (1/8 of hexa8's) and must be complete before the next one
// starts, so at ordinary sizes a sweep is bound by the latency of its launches: each of the 38 per
// application waits for its dependent loads and little else.  The sweeps therefore read a copy of
// the factor in the order they take it: a wavefront has a slice of 64 / G rows, sorted by length
// within the color, G lanes per row; its blocks lie in steps of 64 (one per lane), a block's 9 values
// 64 apart, and where a step lies follows from the kernel's arguments.  Nodes, columns and values
// then take one round of loads, each contiguous over the wavefront, and the entries of z, the row's
// own values and its Dinv a second.  z is in node order and takes the forward values in place (color
// 0 has none: its rows read v), so that no vector is permuted.  A CU fills its L1 at 64 bytes a cycle,
// so few workgroups per color leave most of that idle: a wavefront is a workgroup of its own, and G
// is the smallest of 8, 16 and 32 with which a row's blocks take one batch of kSweepUnroll steps (a
// second batch is a third round of loads).  hexa20R FP64, GMRES iteration 24 x 22 x 20 / 8 x 8 x 8:
// row pointers, columns, z and strided 72-byte blocks in turn 309 / 257 us; this layout in
// workgroups of 4 wavefronts, G = 16 314 / 247; of one 297 / 219 (G = 32 throughout 310 / 217; next
// color's lines fetched into the L2 by further workgroups 297 / 216 but 697 for 613 at 40 x 36 x 32).

constexpr int32_t kNoBlock = INT32_MIN;
constexpr int kSweepUnroll = 4;  // steps loaded together

__device__ __forceinline__ int2 sweep_level(const SweepColor& sc, const int2* more, int k) {
    return k < kSweepLevels ? make_int2(sc.base[k], sc.count[k]) : more[sc.more + k - kSweepLevels];
}

// col and src of every entry of a color's slices: entry (step k, lane) is block G k + lane of the row
// (before the diagonal: from the row's first; after it: from the one after the diagonal).  Columns of
// color 0 (factor rows below c1) are marked -1 - node in the forward sweep.
template <int G>
__global__ __launch_bounds__(BS) void sweep_fill_kernel(SweepColor sc, int upper, int c1, const int2* __restrict__ more,
                                                        const int2* __restrict__ rows,
                                                        const int32_t* __restrict__ fptr,
                                                        const int32_t* __restrict__ fcol,
                                                        const int32_t* __restrict__ dslot,
                                                        const int32_t* __restrict__ perm, int32_t* __restrict__ col,
                                                        int32_t* __restrict__ src) {
    const int w = (blockIdx.x * BS + threadIdx.x) / 64, lane = threadIdx.x & 63;
    if (w >= sc.slices) return;
    const int2 rw = rows[sc.row0 + w * (64 / G) + lane / G];
    int b = 0, e = 0;
    if (rw.x >= 0) {
        const int d = fptr[rw.y] + dslot[rw.y];
        b = upper ? d + 1 : fptr[rw.y];
        e = upper ? fptr[rw.y + 1] : d;
    }
    for (int s = 0, k = b + lane % G; s < sc.levels; ++s, k += G) {
        const int2 lv = sweep_level(sc, more, s);
        if (w >= lv.y) break;
        const int64_t i = (int64_t)(lv.x + w) * 64 + lane;
        if (k < e) {
            const int f = fcol[k], m = perm[f];
            col[i] = !upper && f < c1 ? -1 - m : m;
            src[i] = k;
        } else {
            col[i] = kNoBlock;
            src[i] = -1;
        }
    }
}

// the values of a sweep's entries from the factor
template <typename T>
__global__ __launch_bounds__(BS) void sweep_pack_kernel(int64_t steps, const int32_t* __restrict__ src,
                                                        const T* __restrict__ F, T* __restrict__ val) {
    const int64_t s = ((int64_t)blockIdx.x * BS + threadIdx.x) / 64;
    const int lane = threadIdx.x & 63;
    if (s >= steps) return;
    const int k = src[s * 64 + lane];
#pragma unroll
    for (int v = 0; v < 9; ++v) val[(s * 9 + v) * 64 + lane] = k >= 0 ? F[(int64_t)k * 9 + v] : (T)0;
}

// One color of a sweep: z_n = own_n - sum of the row's blocks times their entries (columns marked
// -1 - m read v, the others z), times Dinv when given.
template <typename T, int G>
__global__ __launch_bounds__(64) void sweep_kernel(SweepColor sc, const int2* __restrict__ more,
                                                   const int2* __restrict__ rows, const int32_t* __restrict__ col,
                                                   const T* __restrict__ val, const T* __restrict__ Dinv,
                                                   const T* __restrict__ v, const T* own, T* z) {
    constexpr int U = kSweepUnroll;
    const int w = xcd_block_g();  // slice
    // All arguments in one round of loads: the compiler loads them where they are first used, and each
    // batch of them is then a wait of its own at the head of the kernel's chain.  24 x 22 x 20 hexa20R
    // FP64 259 -> 247 us per GMRES iteration.  (In the PCG's kernels, whose first loads need few of their
    // arguments, the same cost 0.2 to 0.6 us an iteration.)
    asm volatile("" ::"s"(sc.slices), "s"(sc.row0), "s"(sc.base[0]), "s"(sc.base[1]), "s"(sc.base[2]), "s"(sc.base[3]),
                 "s"(sc.count[0]), "s"(sc.count[1]), "s"(sc.count[2]), "s"(sc.count[3]), "s"(sc.count[4]),
                 "s"(sc.levels), "s"(rows), "s"(col), "s"(val), "s"(Dinv), "s"(v), "s"(own), "s"(z));
    const int lane = threadIdx.x, r = lane % G;
    if (w >= sc.slices) return;
    const int2 rw = rows[sc.row0 + w * (64 / G) + lane / G];
    T y0 = 0, y1 = 0, y2 = 0, o[3] = {0, 0, 0}, m[3] = {0, 0, 0};
    auto steps = [&](int b0, int c0, int b1, int c1, int b2, int c2, int b3, int c3, bool first) {
        const int bs[U] = {b0, b1, b2, b3}, ct[U] = {c0, c1, c2, c3};
        int c[U];
        T a[U][9], x[U][3];
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (w < ct[u]) {  // uniform over the wavefront
                const int64_t i = bs[u] + w;
                c[u] = col[i * 64 + lane];
#pragma unroll
                for (int k = 0; k < 9; ++k) a[u][k] = val[(i * 9 + k) * 64 + lane];
            }
        if (first && r < 3 && rw.x >= 0) {
#pragma unroll
            for (int k = 0; k < 3; ++k) o[k] = own[3 * (int64_t)rw.x + k];
            if (Dinv)
#pragma unroll
                for (int k = 0; k < 3; ++k) m[k] = Dinv[(int64_t)rw.y * 9 + 3 * r + k];
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (w < ct[u]) {
                x[u][0] = x[u][1] = x[u][2] = (T)0;
                if (c[u] != kNoBlock) {
                    const T* xs = c[u] < 0 ? v + 3 * (int64_t)(-1 - c[u]) : z + 3 * (int64_t)c[u];
#pragma unroll
                    for (int k = 0; k < 3; ++k) x[u][k] = xs[k];
                }
            }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (w < ct[u]) {
                y0 += a[u][0] * x[u][0] + a[u][1] * x[u][1] + a[u][2] * x[u][2];
                y1 += a[u][3] * x[u][0] + a[u][4] * x[u][1] + a[u][5] * x[u][2];
                y2 += a[u][6] * x[u][0] + a[u][7] * x[u][1] + a[u][8] * x[u][2];
            }
    };
    steps(sc.base[0], sc.count[0], sc.base[1], sc.count[1], sc.base[2], sc.count[2], sc.base[3], sc.count[3], true);
    if (w < sc.count[U])
        steps(sc.base[4], sc.count[4], sc.base[5], sc.count[5], sc.base[6], sc.count[6], sc.base[7], sc.count[7], false);
    for (int k = kSweepLevels; k < sc.levels; ++k) {
        const int2 lv = more[sc.more + k - kSweepLevels];
        if (w >= lv.y) break;
        steps(lv.x, lv.y, 0, 0, 0, 0, 0, 0, false);
    }
    group_sum3<T, G>(y0, y1, y2);
    if (r < 3 && rw.x >= 0) {
        y0 = o[0] - y0;
        y1 = o[1] - y1;
        y2 = o[2] - y2;
        T out = r == 0 ? y0 : r == 1 ? y1 : y2;
        if (Dinv) out = m[0] * y0 + m[1] * y1 + m[2] * y2;
        z[3 * (int64_t)rw.x + r] = out;
    }
}

template <typename T>
__global__ void bjacobi_kernel(int N, const T* __restrict__ Minv, const T* __restrict__ v, T* __restrict__ z) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= N) return;
    const T* M = Minv + (int64_t)n * 9;
    const T a = v[3 * n], b = v[3 * n + 1], c = v[3 * n + 2];
    z[3 * n] = M[0] * a + M[1] * b + M[2] * c;
    z[3 * n + 1] = M[3] * a + M[4] * b + M[5] * c;
    z[3 * n + 2] = M[6] * a + M[7] * b + M[8] * c;
}

// y = K x (sliced ELL), optionally y = b - K x.  A workgroup has one slice, its wavefronts each a range
// of the rows' blocks: with a lane for a whole row of up to 81 blocks the chain of their loads set the
// time wherever the slices are fewer than some thousands.  hexa20R GMRES iteration at 1 / 2 / 4 / 8
// wavefronts: 8 x 8 x 8 FP64 200 / 179 / 167 / 165 us, 24 x 22 x 20 FP64 (the product 58 us) 292 / 276 /
// 270 / 269, 40 x 36 x 32 FP64 615 / 617 / 595 / 587, FP32 394 / 394 / 388 / 384.
constexpr int kSpmvWaves = 8;
template <typename T>
__global__ __launch_bounds__(64 * kSpmvWaves) void gm_spmv_kernel(int N, const int32_t* __restrict__ slice_off,
                                                         const int32_t* __restrict__ scol,
                                                         const int32_t* __restrict__ slotNode, const T* __restrict__ K,
                                                         const T* __restrict__ x, T* __restrict__ y,
                                                         const double* __restrict__ b) {
    constexpr int W = kSpmvWaves;
    __shared__ T sh[W - 1][3][64];
    const int s = xcd_block_g(), l = threadIdx.x & 63;
    const int part = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int ps = s * kSlice + l;  // row slot
    if (s * kSlice >= N) return;
    const int o0 = slice_off[s], deg = (slice_off[s + 1] - o0) / kSlice;
    const int n = ps < N ? slotNode[ps] : -1;
    const int32_t* cp = scol + o0 + l;
    const T* kp = K + (int64_t)o0 * 9 + l;
    T y0 = 0, y1 = 0, y2 = 0;
    constexpr int kUnroll = sizeof(T) == 8 ? 2 : 3;
    const int k1 = (part + 1) * deg / W;
    if (n >= 0)
#pragma unroll kUnroll
        for (int k = part * deg / W; k < k1; ++k) {
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
    if (part > 0) {
        sh[part - 1][0][l] = y0;
        sh[part - 1][1][l] = y1;
        sh[part - 1][2][l] = y2;
    }
    __syncthreads();
    if (part > 0 || n < 0) return;
#pragma unroll
    for (int w = 0; w < W - 1; ++w) {
        y0 += sh[w][0][l];
        y1 += sh[w][1][l];
        y2 += sh[w][2][l];
    }
    if (b) {
        y[3 * n] = (T)b[3 * n] - y0;
        y[3 * n + 1] = (T)b[3 * n + 1] - y1;
        y[3 * n + 2] = (T)b[3 * n + 2] - y2;
    } else {
        y[3 * n] = y0;
        y[3 * n + 1] = y1;
        y[3 * n + 2] = y2;
    }
}

// partial sums of w . w, and their sum
template <typename T>
__global__ __launch_bounds__(BS) void norm_kernel(int D, const T* __restrict__ w, double* __restrict__ part, int nwg) {
    __shared__ double sh[BS];
    double s = 0.0;
#pragma unroll 4
    for (int i = blockIdx.x * BS + threadIdx.x; i < D; i += nwg * BS) s += (double)w[i] * (double)w[i];
    s = bsum(s, sh);
    if (threadIdx.x == 0) part[blockIdx.x] = s;
}

__global__ __launch_bounds__(BS) void norm_reduce_kernel(const double* __restrict__ part, int nwg,
                                                         double* __restrict__ out) {
    __shared__ double sh[BS];
    double s = 0.0;
    for (int i = threadIdx.x; i < nwg; i += BS) s += part[i];
    s = bsum(s, sh);
    if (threadIdx.x == 0) *out = s;
}

// sum over the wavefront of the NV values of each lane: lane l gets that of value l / (64 / NV)
template <int NV>
__device__ __forceinline__ double wave_sums(double (&s)[NV]) {
    const int lane = threadIdx.x & 63;
    int m = 32;
#pragma unroll
    for (int n = NV / 2; n >= 1; n >>= 1, m >>= 1) {
        const bool hi = lane & m;
#pragma unroll
        for (int q = 0; q < n; ++q) {
            const double send = hi ? s[q] : s[q + n], keep = hi ? s[q + n] : s[q];
            s[q] = keep + __shfl_xor(send, m);
        }
    }
    for (; m >= 1; m >>= 1) s[0] += __shfl_xor(s[0], m);
    return s[0];
}

// Classical Gram-Schmidt of w against V_0..V_{nv-1}.  A dot product has to be complete before the next
// step, and at ordinary sizes a launch costs more than its data: the dot kernel leaves the partial
// sums of its workgroups, and each workgroup of the kernel that needs them adds them up for itself.
// So that this stays short, the workgroups per group of kDotVecs vectors get fewer as the groups get
// more.  hexa20R 24 x 22 x 20 FP64, GMRES(50) iteration: with a reduction launch per dot and the norm
// apart (9 launches) 297 us, now (5) 279.  Several vectors held in registers across the correction and
// the second dot spill from 24 on (FP64), and the restart length is the caller's: not done.
constexpr int kDotVecs = 8, kCombineWG = 512, kMaxVecs = 257;

inline int dot_wgs(int nv) { return nv <= kDotVecs ? 256 : nv <= 3 * kDotVecs ? 128 : 64; }

// part[k][workgroup] = partial sums of V_k . w, kDotVecs vectors per workgroup
template <typename T>
__global__ __launch_bounds__(BS) void orth_dot_kernel(int D, int nv, const T* __restrict__ V, const T* __restrict__ w,
                                                      double* __restrict__ part) {
    constexpr int NV = kDotVecs, W = BS / 64;
    __shared__ double red[W][NV];
    const int nwg = gridDim.x, k0 = blockIdx.y * NV;
    const T* v[NV];
    double s[NV];
#pragma unroll
    for (int q = 0; q < NV; ++q) {
        v[q] = V + (int64_t)(k0 + q < nv ? k0 + q : nv - 1) * D;
        s[q] = 0.0;
    }
#pragma unroll 2
    for (int i = blockIdx.x * BS + threadIdx.x; i < D; i += nwg * BS) {
        const double x = (double)w[i];
#pragma unroll
        for (int q = 0; q < NV; ++q) s[q] += (double)v[q][i] * x;
    }
    const double t = wave_sums<NV>(s);
    const int lane = threadIdx.x & 63;
    if (lane % (64 / NV) == 0) red[threadIdx.x / 64][lane / (64 / NV)] = t;
    __syncthreads();
    if ((int)threadIdx.x < NV && k0 + (int)threadIdx.x < nv) {
        double y = 0.0;
#pragma unroll
        for (int q = 0; q < W; ++q) y += red[q][threadIdx.x];
        part[(int64_t)(k0 + threadIdx.x) * nwg + blockIdx.x] = y;
    }
}

// h_k = sum of part[k] (to hout from the first workgroup), w -= sum h_k V_k; with NORM, pnorm = the
// workgroups' partial sums of w . w
template <typename T, bool NORM>
__global__ __launch_bounds__(BS) void orth_combine_kernel(int D, int nv, int nwg, const T* __restrict__ V,
                                                          T* __restrict__ w, const double* __restrict__ part,
                                                          double* __restrict__ hout, double* __restrict__ pnorm) {
    constexpr int PRE = 8;
    __shared__ double hs[kMaxVecs], red[BS / 64];
    int i = blockIdx.x * BS + threadIdx.x;
    T a[PRE], x = 0;
    if (i < D) {  // in flight while the sums are formed
        x = w[i];
#pragma unroll
        for (int q = 0; q < PRE; ++q) a[q] = V[(int64_t)(q < nv ? q : nv - 1) * D + i];
    }
    for (int k = threadIdx.x / 8; k < nv; k += BS / 8) {
        double h = 0.0;
#pragma unroll 8
        for (int q = threadIdx.x & 7; q < nwg; q += 8) h += part[(int64_t)k * nwg + q];
        h += __shfl_xor(h, 1);
        h += __shfl_xor(h, 2);
        h += __shfl_xor(h, 4);
        if ((threadIdx.x & 7) == 0) {
            hs[k] = h;
            if (blockIdx.x == 0) hout[k] = h;
        }
    }
    __syncthreads();
    double nrm = 0.0;
    for (bool first = true; i < D; i += gridDim.x * BS, first = false) {
        double acc;
        int k = 0;
        if (first) {
            acc = (double)x;
            const int n = nv < PRE ? nv : PRE;
#pragma unroll
            for (int q = 0; q < PRE; ++q)
                if (q < n) acc -= hs[q] * (double)a[q];
            k = n;
        } else {
            acc = (double)w[i];
        }
#pragma unroll 8
        for (; k < nv; ++k) acc -= hs[k] * (double)V[(int64_t)k * D + i];
        const T y = (T)acc;
        w[i] = y;
        nrm += (double)y * (double)y;
    }
    if (NORM) {
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) nrm += __shfl_xor(nrm, m);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x / 64] = nrm;
        __syncthreads();
        if (threadIdx.x == 0) pnorm[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
    }
}

// v = w / ||w|| with ||w||^2 the sum of the np <= kCombineWG values pin
template <typename T>
__global__ __launch_bounds__(BS) void orth_scale_kernel(int D, int np, const T* __restrict__ w, const double* __restrict__ pin,
                                                        double* __restrict__ nrm2, T* __restrict__ v) {
    __shared__ double red[BS / 64];
    const int i = blockIdx.x * BS + threadIdx.x;
    const T x = i < D ? w[i] : (T)0;
    static_assert(kCombineWG == 2 * BS, "two values per thread");
    double s = ((int)threadIdx.x < np ? pin[threadIdx.x] : 0.0) + ((int)threadIdx.x + BS < np ? pin[threadIdx.x + BS] : 0.0);
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) s += __shfl_xor(s, m);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x / 64] = s;
    __syncthreads();
    s = (red[0] + red[1]) + (red[2] + red[3]);
    if (i == 0) *nrm2 = s;
    if (i < D) v[i] = (T)((double)x / sqrt(s));
}

// w = sum_i h_i V_i
template <typename T>
__global__ void combine_kernel(int D, int nv, const T* __restrict__ V, const double* __restrict__ h,
                               T* __restrict__ w) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= D) return;
    double acc = 0.0;
#pragma unroll 4
    for (int k = 0; k < nv; ++k) acc += h[k] * (double)V[(int64_t)k * D + i];
    w[i] = (T)acc;
}

template <typename T>
__global__ void scale_kernel(int D, const T* __restrict__ w, const double* __restrict__ nrm2, T* __restrict__ v) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= D) return;
    v[i] = (T)((double)w[i] / sqrt(nrm2[0]));
}

template <typename T>
__global__ void axpy_kernel(int D, const T* __restrict__ z, T* __restrict__ x) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < D) x[i] += z[i];
}

template <typename T>
__global__ void zero_kernel(int D, T* __restrict__ x) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < D) x[i] = 0;
}

template <typename T>
__global__ void finish_kernel(int D, const T* __restrict__ x, const double* __restrict__ b,
                              const uint8_t* __restrict__ dirflag, int ndir, double* __restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= D) return;
    out[i] = (ndir && dirflag[i]) ? b[i] : (double)x[i];
}

int grid_of(int n) { return (n + BS - 1) / BS; }

// The slices and levels of one sweep.
int build_sweep(GmresWork* g, int upper, const std::vector<int32_t>& fptr, const std::vector<int32_t>& dslot,
                const std::vector<int32_t>& perm) {
    GmresWork::Sweep& sw = g->sweep[upper];
    std::vector<int32_t> order, place;
    std::vector<int2> rows, more;
    sw.color.assign(g->ncolors, SweepColor());
    sw.steps = 0;
    auto len = [&](int i) { return upper ? fptr[i + 1] - fptr[i] - dslot[i] - 1 : dslot[i]; };
    for (int col = 0; col < g->ncolors; ++col) {
        const int r0 = g->cstart[col], r1 = g->cstart[col + 1];
        SweepColor& sc = sw.color[col];
        // by decreasing length, equal ones in order: counted, as a sort by comparison took 14 ms of the
        // first solve's 104 at 64^3 hexa8
        place.assign(g->maxRow + 1, 0);
        for (int i = r0; i < r1; ++i) ++place[len(i)];
        for (int l = g->maxRow, at = 0; l >= 0; --l) {
            const int n = place[l];
            place[l] = at;
            at += n;
        }
        order.resize(r1 - r0);
        for (int i = r0; i < r1; ++i) order[place[len(i)]++] = i;
        const int most = order.empty() ? 0 : len(order[0]);
        const int G = sc.G = most <= kSweepUnroll * 8 ? 8 : most <= kSweepUnroll * 16 ? 16 : 32, R = 64 / G;
        sc.row0 = (int)rows.size();
        sc.slices = (int)((order.size() + R - 1) / R);
        sc.more = (int)more.size();
        for (int k = 0; k < sc.slices * R; ++k)
            rows.push_back(k < (int)order.size() ? make_int2(perm[order[k]], order[k]) : make_int2(-1, -1));
        for (int k = 0, n = sc.slices;; ++k) {
            while (n > 0 && len(order[(n - 1) * R]) <= k * G) --n;  // slices with a step k
            if (n == 0) break;
            if (k < kSweepLevels) {
                sc.base[k] = (int)sw.steps;
                sc.count[k] = n;
            } else {
                more.push_back(make_int2((int)sw.steps, n));
            }
            sc.levels = k + 1;
            sw.steps += n;
        }
    }
    const size_t ne = std::max<size_t>(1, (size_t)sw.steps * 64);
    EFE_HIP(hipMalloc(&sw.rows, std::max<size_t>(1, rows.size()) * sizeof(int2)));
    EFE_HIP(hipMalloc(&sw.more, std::max<size_t>(1, more.size()) * sizeof(int2)));
    EFE_HIP(hipMalloc(&sw.col, ne * sizeof(int32_t)));
    EFE_HIP(hipMalloc(&sw.src, ne * sizeof(int32_t)));
    EFE_HIP(hipMemcpy(sw.rows, rows.data(), rows.size() * sizeof(int2), hipMemcpyHostToDevice));
    EFE_HIP(hipMemcpy(sw.more, more.data(), more.size() * sizeof(int2), hipMemcpyHostToDevice));
    for (const SweepColor& sc : sw.color) {
        if (sc.slices == 0) continue;
        const int grid = grid_of(sc.slices * 64), c1 = g->cstart[1];
        const auto fill = sc.G == 8 ? sweep_fill_kernel<8> : sc.G == 16 ? sweep_fill_kernel<16> : sweep_fill_kernel<32>;
        fill<<<grid, BS, 0, g->ks>>>(sc, upper, c1, sw.more, sw.rows, g->fptr, g->fcol, g->dslot, g->perm, sw.col, sw.src);
    }
    EFE_HIP(hipGetLastError());
    return EFE_OK;
}

int build_ilu(efe_ctx* c, GmresWork* g) {
    IluPattern ip;
    std::string err;
    if (!efe_build_ilu_pattern(c->hp, ip, err)) {
        efe_set_error(err);
        return EFE_ERR_ARG;
    }
    const int N = c->N;
    // block CSR of the factor in elimination order; fidx: operator block -> factor block
    std::vector<int32_t> fptr(N + 1, 0), fcol, fidx(c->hp.bptr[N]), dslot(N);
    for (int i = 0; i < N; ++i) fptr[i + 1] = fptr[i] + ip.rowlen[i];
    fcol.resize(fptr[N]);
    std::vector<std::pair<int32_t, int32_t>> row;
    for (int i = 0; i < N; ++i) {
        const int n = ip.perm[i];
        dslot[i] = ip.dslot[i];
        row.clear();
        for (int32_t b = c->hp.bptr[n]; b < c->hp.bptr[n + 1]; ++b) row.emplace_back(ip.iperm[c->hp.bcol[b]], b);
        std::sort(row.begin(), row.end());
        for (int k = 0; k < ip.rowlen[i]; ++k) {
            fcol[fptr[i] + k] = row[k].first;
            fidx[row[k].second] = fptr[i] + k;
        }
    }
    g->maxUpper = 0;
    g->maxRow = 0;
    for (int i = 0; i < N; ++i) {
        g->maxUpper = std::max(g->maxUpper, fptr[i + 1] - fptr[i] - dslot[i] - 1);
        g->maxRow = std::max(g->maxRow, fptr[i + 1] - fptr[i]);
    }
    g->ncolors = ip.ncolors;
    g->cstart.assign(ip.color_start.begin(), ip.color_start.end());
    g->cup.assign(g->ncolors, 0);
    for (int col = 0; col < g->ncolors; ++col)
        for (int i = g->cstart[col]; i < g->cstart[col + 1]; ++i) {
            g->cup[col] = std::max(g->cup[col], fptr[i + 1] - fptr[i] - dslot[i] - 1);
        }
    g->nbF = fptr[N];
    EFE_HIP(hipMalloc(&g->fptr, fptr.size() * sizeof(int32_t)));
    EFE_HIP(hipMalloc(&g->fcol, fcol.size() * sizeof(int32_t)));
    EFE_HIP(hipMalloc(&g->fidx, fidx.size() * sizeof(int32_t)));
    EFE_HIP(hipMalloc(&g->dslot, dslot.size() * sizeof(int32_t)));
    EFE_HIP(hipMalloc(&g->perm, (size_t)N * sizeof(int32_t)));
    EFE_HIP(hipMemcpy(g->fptr, fptr.data(), fptr.size() * sizeof(int32_t), hipMemcpyHostToDevice));
    EFE_HIP(hipMemcpy(g->fcol, fcol.data(), fcol.size() * sizeof(int32_t), hipMemcpyHostToDevice));
    EFE_HIP(hipMemcpy(g->fidx, fidx.data(), fidx.size() * sizeof(int32_t), hipMemcpyHostToDevice));
    EFE_HIP(hipMemcpy(g->dslot, dslot.data(), dslot.size() * sizeof(int32_t), hipMemcpyHostToDevice));
    EFE_HIP(hipMemcpy(g->perm, ip.perm.data(), (size_t)N * sizeof(int32_t), hipMemcpyHostToDevice));
    for (int up = 0; up < 2; ++up)
        if (int rc = build_sweep(g, up, fptr, dslot, ip.perm)) return rc;
    g->ilu_ready = true;
    return EFE_OK;
}

template <typename T>
T* sweep_values(const GmresWork::Sweep& sw) {
    if constexpr (sizeof(T) == 8) return sw.v64;
    else return sw.v32;
}

template <typename T>
int ilu_factor(efe_ctx* c, GmresWork* g, const T* K, T*& F, T*& Dinv, int pi, hipStream_t st) {
    if (!F) {
        EFE_HIP(hipMalloc(&F, (size_t)g->nbF * 9 * sizeof(T)));
        EFE_HIP(hipMalloc(&Dinv, (size_t)c->N * 9 * sizeof(T)));
    }
    if (g->factored_version[pi] == c->Kversion) return EFE_OK;
    ilu_copy_kernel<T><<<grid_of(c->N), BS, 0, st>>>(c->N, c->bptr, c->slice_off, c->nodeSlot, K, g->fidx, F);
    for (int col = 0; col < g->ncolors; ++col) {
        const int r0 = g->cstart[col], r1 = g->cstart[col + 1];
        if (r1 <= r0) continue;
        // the row in registers: hexa8 rows have up to 27 blocks, hexa20 rows up to 81.  (Issuing
        // the next steps' row-k loads ahead, with a second LDS list buffer, was measured: no
        // gain at 48^3 hexa20, the extra registers cost as much as the hidden latency.)
        if (g->maxUpper <= kFactorCap && g->maxRow <= 32) {
            ilu_factor_reg_kernel<T, 16, 2, kFactorCap><<<grid_of((r1 - r0) * 16), BS, 0, st>>>(
                r0, r1, g->fptr, g->fcol, g->dslot, F, Dinv);
        } else if (g->maxUpper <= kFactorCap && g->maxRow <= 96) {
            ilu_factor_reg_kernel<T, 32, 3, kFactorCap><<<grid_of((r1 - r0) * 32), BS, 0, st>>>(
                r0, r1, g->fptr, g->fcol, g->dslot, F, Dinv);
        } else if (g->maxUpper <= kFactorCap) {  // row k's upper columns staged in LDS
            if (c->NN == 8)
                ilu_factor_lds_kernel<T, 8, kFactorCap><<<grid_of((r1 - r0) * 8), BS, 0, st>>>(
                    r0, r1, g->fptr, g->fcol, g->dslot, F, Dinv);
            else
                ilu_factor_lds_kernel<T, 16, kFactorCap><<<grid_of((r1 - r0) * 16), BS, 0, st>>>(
                    r0, r1, g->fptr, g->fcol, g->dslot, F, Dinv);
        } else if (c->NN == 8) {
            ilu_factor_kernel<T, 8><<<grid_of((r1 - r0) * 8), BS, 0, st>>>(r0, r1, g->fptr, g->fcol, g->dslot, F, Dinv);
        } else {
            ilu_factor_kernel<T, 16><<<grid_of((r1 - r0) * 16), BS, 0, st>>>(r0, r1, g->fptr, g->fcol, g->dslot, F,
                                                                             Dinv);
        }
    }
    for (GmresWork::Sweep& sw : g->sweep) {
        if (!sweep_values<T>(sw))
            EFE_HIP(hipMalloc(sizeof(T) == 8 ? (void**)&sw.v64 : (void**)&sw.v32,
                              std::max<size_t>(1, (size_t)sw.steps * 64 * 9) * sizeof(T)));
        if (sw.steps)
            sweep_pack_kernel<T><<<(unsigned)((sw.steps * 64 + BS - 1) / BS), BS, 0, st>>>(sw.steps, sw.src, F, sweep_values<T>(sw));
    }
    EFE_HIP(hipGetLastError());
    g->factored_version[pi] = c->Kversion;
    return EFE_OK;
}

// z = M^{-1} v
template <typename T>
void apply_precond(efe_ctx* c, GmresWork* g, int precond, const T* F, const T* Dinv, const T* Minv, const T* v, T* z,
                   hipStream_t st) {
    const int N = c->N;
    if (precond == EFE_PRECOND_ILU0) {
        const int last = g->ncolors - 1;
        // color 0 has no forward sweep (nothing comes before it: its forward values are v's); the
        // last color's backward sweep rides on its forward sweep when its rows have no blocks after them
        const bool fuseLast = last > 0 && g->cup[last] == 0;
        auto launch = [&](int up, int col, const T* D) {
            const GmresWork::Sweep& sw = g->sweep[up];
            const SweepColor& sc = sw.color[col];
            if (sc.slices == 0) return;
            const auto kernel = sc.G == 8 ? sweep_kernel<T, 8> : sc.G == 16 ? sweep_kernel<T, 16> : sweep_kernel<T, 32>;
            kernel<<<round8g(sc.slices), 64, 0, st>>>(sc, sw.more, sw.rows, sw.col, sweep_values<T>(sw), D, v,
                                                      up && col > 0 ? z : v, z);
        };
        for (int col = 1; col < g->ncolors; ++col) launch(0, col, fuseLast && col == last ? Dinv : nullptr);
        for (int col = fuseLast ? last - 1 : last; col >= 0; --col) launch(1, col, Dinv);
    } else {
        bjacobi_kernel<T><<<grid_of(N), BS, 0, st>>>(N, Minv, v, z);
    }
}

inline double* step_results(const GmresWork* g, int j) { return g->hhost + (j & 1) * 3 * (g->m + 2); }

// Arnoldi step j: w = K M^{-1} V_j, two classical Gram-Schmidt passes against V_0..V_j
// (projections into h[0..], h[m+2..], h = step_results), ||w||^2 into h[2(m+2)], V_{j+1} = w / ||w||.
template <typename T>
void gmres_step_launch(efe_ctx* c, GmresWork* g, int precond, const T* F, const T* Dinv, const T* Minv, const T* K,
                       int j, hipStream_t st) {
    const int D = c->D, N = c->N, m = g->m;
    const int gd = grid_of(D), gs = round8g((N + kSlice - 1) / kSlice);
    T* V = (T*)g->V;
    T* w = (T*)g->w;
    T* z = (T*)g->z;
    apply_precond<T>(c, g, precond, F, Dinv, Minv, V + (int64_t)j * D, z, st);
    gm_spmv_kernel<T><<<gs, 64 * kSpmvWaves, 0, st>>>(N, c->slice_off, c->scol, c->slotNode, K, z, w, nullptr);
    const int nv = j + 1, nwg = dot_wgs(nv), gc = std::min(gd, kCombineWG);
    double* h = step_results(g, j);
    const dim3 gdot(nwg, (nv + kDotVecs - 1) / kDotVecs);
    orth_dot_kernel<T><<<gdot, BS, 0, st>>>(D, nv, V, w, g->part);
    orth_combine_kernel<T, false><<<gc, BS, 0, st>>>(D, nv, nwg, V, w, g->part, h, nullptr);
    orth_dot_kernel<T><<<gdot, BS, 0, st>>>(D, nv, V, w, g->part);
    orth_combine_kernel<T, true><<<gc, BS, 0, st>>>(D, nv, nwg, V, w, g->part, h + (m + 2), g->pnorm);
    orth_scale_kernel<T><<<gd, BS, 0, st>>>(D, gc, w, g->pnorm, h + 2 * (m + 2), V + (int64_t)nv * D);
}

// Step j as one replayed hipGraph (captured on first use for these buffers); with
// EFE_GMRES_NO_GRAPH set, the launches go to the stream one by one.
template <typename T>
int run_step(efe_ctx* c, GmresWork* g, int precond, const T* F, const T* Dinv, const T* Minv, const T* K, int j,
             hipStream_t st) {
    static const bool graphs = std::getenv("EFE_GMRES_NO_GRAPH") == nullptr;
    if (!graphs) {
        gmres_step_launch<T>(c, g, precond, F, Dinv, Minv, K, j, st);
        EFE_HIP(hipGetLastError());
        return EFE_OK;
    }
    if ((int)g->stepGraph.size() < g->m) {
        g->stepGraph.resize(g->m, nullptr);
        g->stepKey.resize(g->m);
    }
    const std::array<int64_t, 8> key = {precond,
                                        (int64_t)sizeof(T),
                                        (int64_t)(intptr_t)F,
                                        (int64_t)(intptr_t)Dinv,
                                        (int64_t)(intptr_t)Minv,
                                        (int64_t)(intptr_t)K,
                                        (int64_t)(intptr_t)g->V,
                                        g->ncolors};
    if (!g->stepGraph[j] || g->stepKey[j] != key) {
        if (g->stepGraph[j]) hipGraphExecDestroy(g->stepGraph[j]);
        g->stepGraph[j] = nullptr;
        hipGraph_t gr;
        EFE_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeRelaxed));
        gmres_step_launch<T>(c, g, precond, F, Dinv, Minv, K, j, st);
        EFE_HIP(hipStreamEndCapture(st, &gr));
        EFE_HIP(hipGraphInstantiate(&g->stepGraph[j], gr, nullptr, nullptr, 0));
        EFE_HIP(hipGraphDestroy(gr));
        g->stepKey[j] = key;
    }
    EFE_HIP(hipGraphLaunch(g->stepGraph[j], st));
    return EFE_OK;
}

template <typename T>
int gmres_solve(efe_ctx* c, GmresWork* g, const double* b, double* xout, const efe_solve_opts* o,
                efe_solve_info* info, const T* K, const T* Minv, int pi) {
    hipStream_t st = g->ks;
    const int D = c->D, N = c->N, m = g->m;
    EFE_HIP(hipEventRecord(g->evA, c->stream));
    EFE_HIP(hipStreamWaitEvent(st, g->evA, 0));
    EFE_HIP(hipEventRecord(g->t0, st));
    T *F = nullptr, *Dinv = nullptr;
    if (o->precond == EFE_PRECOND_ILU0) {
        if (!g->ilu_ready) {
            int rc = build_ilu(c, g);
            if (rc) return rc;
        }
        T*& Fr = pi ? (T*&)g->F32 : (T*&)g->F64;
        T*& Dr = pi ? (T*&)g->Dinv32 : (T*&)g->Dinv64;
        int rc = ilu_factor<T>(c, g, K, Fr, Dr, pi, st);
        if (rc) return rc;
        F = Fr;
        Dinv = Dr;
    }
    EFE_HIP(hipEventRecord(g->t1, st));
    T* V = (T*)g->V;
    T* w = (T*)g->w;
    T* z = (T*)g->z;
    T* x = (T*)g->x;
    const int gd = grid_of(D);
    const int gs = round8g((N + kSlice - 1) / kSlice);
    double* hh = g->hhost;
    // ||b||
    zero_kernel<T><<<gd, BS, 0, st>>>(D, x);
    gm_spmv_kernel<T><<<gs, 64 * kSpmvWaves, 0, st>>>(N, c->slice_off, c->scol, c->slotNode, K, x, w, b);
    norm_kernel<T><<<g->nwg, BS, 0, st>>>(D, w, g->part, g->nwg);
    norm_reduce_kernel<<<1, BS, 0, st>>>(g->part, g->nwg, g->hdev);
    EFE_HIP(hipMemcpyAsync(hh, g->hdev, sizeof(double), hipMemcpyDeviceToHost, st));
    EFE_HIP(hipStreamSynchronize(st));
    const double bnorm = sqrt(hh[0]);
    info->rhs_norm = bnorm;
    info->iterations = 0;
    info->status = EFE_OK;
    info->residual = bnorm;
    const double tol = fmax(o->rtol * bnorm, o->atol);
    const int maxit = o->max_iter > 0 ? o->max_iter : 10000;
    std::vector<double> H((size_t)(m + 1) * m), cs(m), sn(m), gv(m + 1), y(m);
    double beta = bnorm;
    int it = 0;
    bool done = !(bnorm > tol), bad = !(bnorm == bnorm);
    while (!done && !bad) {
        // r = b - K x is in w; V_0 = r / beta
        scale_kernel<T><<<gd, BS, 0, st>>>(D, w, g->hdev, V);
        std::fill(gv.begin(), gv.end(), 0.0);
        gv[0] = beta;
        int jend = -1, sent = 0;
        for (int j = 0; j < m; ++j) {
            // step j + 1 goes out before the host has seen step j, so that the device does not wait
            // for it: the last step of a solve is followed by one whose results nothing reads
            for (; sent <= j + 1 && sent < m && it + sent - j < maxit; ++sent) {
                if (int rc = run_step<T>(c, g, o->precond, F, Dinv, Minv, K, sent, st)) return rc;
                EFE_HIP(hipEventRecord(g->step[sent & 1], st));
            }
            EFE_HIP(hipEventSynchronize(g->step[j & 1]));
            ++it;
            const double* h = step_results(g, j);
            double* col = &H[(size_t)j * (m + 1)];
            for (int i = 0; i <= j; ++i) col[i] = h[i] + h[(m + 2) + i];
            col[j + 1] = sqrt(h[2 * (m + 2)]);
            for (int i = 0; i < j; ++i) {
                const double a = cs[i] * col[i] + sn[i] * col[i + 1];
                col[i + 1] = -sn[i] * col[i] + cs[i] * col[i + 1];
                col[i] = a;
            }
            const double r = std::hypot(col[j], col[j + 1]);
            cs[j] = r > 0 ? col[j] / r : 1.0;
            sn[j] = r > 0 ? col[j + 1] / r : 0.0;
            col[j] = r;
            col[j + 1] = 0.0;
            gv[j + 1] = -sn[j] * gv[j];
            gv[j] = cs[j] * gv[j];
            const double res = fabs(gv[j + 1]);
            info->residual = res;
            jend = j;
            if (!(res == res)) {
                bad = true;
                break;
            }
            if (res <= tol) {
                done = true;
                break;
            }
            if (it >= maxit) break;
        }
        if (bad || jend < 0) break;
        // y = H^{-1} g, u = V y, x += M^{-1} u
        for (int i = jend; i >= 0; --i) {
            double s = gv[i];
            for (int k = i + 1; k <= jend; ++k) s -= H[(size_t)k * (m + 1) + i] * y[k];
            y[i] = s / H[(size_t)i * (m + 1) + i];
        }
        EFE_HIP(hipMemcpyAsync(g->hdev, y.data(), (jend + 1) * sizeof(double), hipMemcpyHostToDevice, st));
        combine_kernel<T><<<gd, BS, 0, st>>>(D, jend + 1, V, g->hdev, w);
        apply_precond<T>(c, g, o->precond, F, Dinv, Minv, w, z, st);
        axpy_kernel<T><<<gd, BS, 0, st>>>(D, z, x);
        if (done || it >= maxit) break;
        // restart: w = b - K x
        gm_spmv_kernel<T><<<gs, 64 * kSpmvWaves, 0, st>>>(N, c->slice_off, c->scol, c->slotNode, K, x, w, b);
        norm_kernel<T><<<g->nwg, BS, 0, st>>>(D, w, g->part, g->nwg);
        norm_reduce_kernel<<<1, BS, 0, st>>>(g->part, g->nwg, g->hdev);
        EFE_HIP(hipMemcpyAsync(hh, g->hdev, sizeof(double), hipMemcpyDeviceToHost, st));
        EFE_HIP(hipStreamSynchronize(st));
        beta = sqrt(hh[0]);
        info->residual = beta;
        if (!(beta == beta)) bad = true;
        if (beta <= tol) done = true;
    }
    EFE_HIP(hipEventRecord(g->t2, st));
    finish_kernel<T><<<gd, BS, 0, st>>>(D, x, b, c->dirflag, c->ndir, xout);
    EFE_HIP(hipGetLastError());
    EFE_HIP(hipEventRecord(g->evB, st));
    EFE_HIP(hipStreamWaitEvent(c->stream, g->evB, 0));
    EFE_HIP(hipStreamSynchronize(st));
    info->iterations = it;
    float fms = 0, ims = 0;
    hipEventElapsedTime(&fms, g->t0, g->t1);
    hipEventElapsedTime(&ims, g->t1, g->t2);
    c->t_kry = it > 0 ? ims / it : 0.0;
    c->tot[EFE_T_KRYLOV] += ims;
    c->tot[EFE_T_KRYLOV_ITERS] += it;
    c->tot[EFE_T_SOLVES] += 1;
    c->tot[EFE_T_PRECOND] += fms;
    if (bad) info->status = EFE_NAN;
    else if (!done) info->status = EFE_NOT_CONVERGED;
    return EFE_OK;
}

int ensure_gmres(efe_ctx* c, int m, int prec) {
    GmresWork* g = c->gw;
    if (!g) {
        g = new GmresWork();
        c->gw = g;
        g->D = c->D;
        g->N = c->N;
        EFE_HIP(hipStreamCreateWithFlags(&g->ks, hipStreamNonBlocking));
        EFE_HIP(hipEventCreateWithFlags(&g->evA, hipEventDisableTiming));
        EFE_HIP(hipEventCreateWithFlags(&g->evB, hipEventDisableTiming));
        for (hipEvent_t& e : g->step) EFE_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        EFE_HIP(hipEventCreate(&g->t0));
        EFE_HIP(hipEventCreate(&g->t1));
        EFE_HIP(hipEventCreate(&g->t2));
        g->nwg = 512;
        EFE_HIP(hipHostMalloc(&g->hhost, 2 * 3 * 258 * sizeof(double), hipHostMallocDefault));
    }
    if (g->m != m || g->vprec != prec) {
        if (m > 256) {
            efe_set_error("GMRES restart length above 256");
            return EFE_ERR_ARG;
        }
        drop_step_graphs(g);
        hipFree(g->V); hipFree(g->w); hipFree(g->z); hipFree(g->x);
        hipFree(g->part); hipFree(g->hdev);
        const size_t es = prec == EFE_FP32 ? sizeof(float) : sizeof(double);
        const size_t D = (size_t)c->D;
        EFE_HIP(hipMalloc(&g->V, (size_t)(m + 1) * D * es));
        EFE_HIP(hipMalloc(&g->w, D * es));
        EFE_HIP(hipMalloc(&g->z, D * es));
        EFE_HIP(hipMalloc(&g->x, D * es));
        EFE_HIP(hipMalloc(&g->part, ((size_t)(m + 1) * g->nwg + kCombineWG) * sizeof(double)));
        g->pnorm = g->part + (size_t)(m + 1) * g->nwg;
        EFE_HIP(hipMalloc(&g->hdev, (size_t)(m + 2) * sizeof(double)));
        g->m = m;
        g->vprec = prec;
    }
    return EFE_OK;
}

}  // namespace

int efe_gmres_solve(efe_ctx* c, const double* b, double* x, const efe_solve_opts* o, efe_solve_info* info) {
    const int m = o->restart > 0 ? o->restart : 50;
    int rc = ensure_gmres(c, m, o->precision);
    if (rc) return rc;
    if (o->precision == EFE_FP32) return gmres_solve<float>(c, c->gw, b, x, o, info, c->K32, c->Minv32, 1);
    return gmres_solve<double>(c, c->gw, b, x, o, info, c->K64, c->Minv64, 0);
}

void efe_gmres_free(efe_ctx* c) {
    GmresWork* g = c->gw;
    if (!g) return;
    void* bufs[] = {g->fptr, g->fcol, g->fidx, g->dslot, g->perm, g->F64, g->Dinv64, g->F32, g->Dinv32,
                    g->V, g->w, g->z, g->x, g->part, g->hdev};
    for (void* p : bufs)
        if (p) hipFree(p);
    for (GmresWork::Sweep& sw : g->sweep) {
        void* sb[] = {sw.rows, sw.more, sw.col, sw.src, sw.v64, sw.v32};
        for (void* p : sb)
            if (p) hipFree(p);
    }
    drop_step_graphs(g);
    if (g->hhost) hipHostFree(g->hhost);
    if (g->ks) hipStreamDestroy(g->ks);
    if (g->evA) hipEventDestroy(g->evA);
    if (g->evB) hipEventDestroy(g->evB);
    for (hipEvent_t e : {g->t0, g->t1, g->t2, g->step[0], g->step[1]})
        if (e) hipEventDestroy(e);
    delete g;
    c->gw = nullptr;
}
