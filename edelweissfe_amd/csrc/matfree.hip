// Matrix-free products K p from the tangents at the QPs.
//
// The element pass stores, per element and QP, the compact tangent
// w detJ [A, B, cnn, (cn1, c1n,)] and the deviatoric direction n as n_11, n_22, n_12, n_13,
// n_23 (n_33 = -n_11 - n_22) of
// C = A 1(x)1 + B Idev + cnn n(x)n + cn1 n(x)1 + c1n 1(x)n.  y = K p is then, per element (one
// thread):
//   J   = sum_a dN_a/dxi (x) (x_a - x_0)              (rebuilt: cheaper than storing J^-1)
//   H   = sum_a p_a (x) dN_a/dxi                      (3x3)
//   eps = sym(H J^-1)                                 (engineering Voigt)
//   sig = C eps                                       (compact form, ~30 flops)
//   M_ik = sum_j sig_ij J^-1_jk
//   f_a = M dN_a/dxi
// followed by a sum of the element forces per node in a fixed order, so the product is
// deterministic.  Dirichlet DOFs are eliminated symmetrically, as in the assembled operator: p is
// read as 0 on them and their rows return p (unit diagonal).  The same kernels with the
// prescribed values as p and no elimination give the right-hand-side correction
// K[:, dir] dir_values.
//
// hexa20 (EFE_FP32_MATFREE): 8 or 10 floats per QP in [QP][field][element] order, the forces to
// node-sorted slots, one per (element, node), summed per node by a second kernel.
//
// hexa8: bricks of up to 256 elements (bricks.cpp), in FP32 (EFE_FP32_MATFREE) and in FP64: the
// FP64 tangent pass of elastic and J2 models stores its compact tangents too, and the FP64 CG
// runs on them instead of the assembled operator.  Bytes per element and product: 64 NC / 8 (FP32
// half of it) for the tangents (NC = 7), ~1.6 staged nodes of 48 + 2 x 24 (12) bytes, 16 of local
// indices: 614 in FP64, against 2135 of the assembled blocks at 64^3 (27 x 72 + 27 x 4 per node).
// Measured at 64^3 in FP64: 94 us per assembled product (5.9 TB/s), 43 us per brick product with
// the tangents from HBM, ~34 us with them in the Infinity Cache; PCG iteration 123.7 -> 59.0 us.
// Meshes of up to kSplitElements elements have, in FP32, bricks of 32 with 8 lanes per element and, in
// FP64, the assembled operator.
#include <algorithm>
#include <cstring>
#include <type_traits>
#include <vector>

#include "efe_internal.h"

namespace {

// slots staged per chunk by the gather: 2048 x 12 B (+1/8 skew) = 27 KiB of LDS, one chunk
// for the 256 nodes of a workgroup of an interior hexa8 region
constexpr int kGatherChunk = 2048;

__device__ __forceinline__ int xcd_block_mf() {
    const int per = gridDim.x >> 3;
    return (blockIdx.x & 7) * per + (blockIdx.x >> 3);
}

// Deterministic workgroup sum: xor butterfly inside each wavefront (all lanes end with
// bitwise identical sums), then the per-wave sums in wave order.
template <int BS>
__device__ __forceinline__ double block_sum_mf(double v, double* sh) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    constexpr int NW = BS / 64;
    if (NW == 1) return v;
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    double r = sh[0];
    for (int i = 1; i < NW; ++i) r += sh[i];
    __syncthreads();
    return r;
}

// Sum of the force slots of node n0 + threadIdx.x, for the BS consecutive nodes
// n0 .. n0 + BS - 1 of a workgroup (block-uniform call).  Their slots are one contiguous
// range of the node-sorted force list; it is staged through LDS in chunks with coalesced
// loads (consecutive lanes, consecutive words), then every lane sums its own node's slots
// in slot order, the same order as a direct per-node loop.  LDS layout: component-major
// with a skew of one word per 8 slots (lane l starts near slot 8 l, so the skewed word
// index 9 l + .. falls into distinct banks) and a row pitch of CHP words (CHP = 1 mod 64,
// so the three components of one slot, stored by neighbouring lanes, differ in bank too).
// A workgroup in which no lane wants its sum (frozen specimens) reads nothing.
template <int BS>
__device__ __forceinline__ void gather_slots(int n0, int N, const int32_t* __restrict__ nptr,
                                             const float* __restrict__ Fe, bool want, float* buf, float (&y)[3]) {
    constexpr int CH = kGatherChunk, CHP = kGatherChunk + kGatherChunk / 8 + 1;
    constexpr int R = (3 * CH + BS - 1) / BS;  // staged words per lane
    y[0] = y[1] = y[2] = 0.0f;
    if (!__syncthreads_or(want)) return;
    const int n = n0 + threadIdx.x;
    const int s0 = nptr[n0], s1 = nptr[min(n0 + BS, N)];
    const int mb = want ? nptr[n] : 0, me = want ? nptr[n + 1] : 0;
    for (int c0 = s0; c0 < s1; c0 += CH) {
        const int cnt = min(CH, s1 - c0);
        const float* src = Fe + (int64_t)c0 * 3;
        // all loads first (independent, so they are in flight together), then the stores
        float tmp[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int i = threadIdx.x + r * BS;
            tmp[r] = i < 3 * cnt ? src[i] : 0.0f;
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int i = threadIdx.x + r * BS;
            if (i < 3 * cnt) {
                const int c = i / 3, k = i - 3 * (i / 3);
                buf[k * CHP + c + (c >> 3)] = tmp[r];
            }
        }
        __syncthreads();
        const int lo = max(mb, c0), hi = min(me, c0 + cnt);
        for (int c = lo; c < hi; ++c) {
            const int w = (c - c0) + ((c - c0) >> 3);
            y[0] += buf[w];
            y[1] += buf[CHP + w];
            y[2] += buf[2 * CHP + w];
        }
        __syncthreads();
    }
}

constexpr int kGatherLds = 3 * (kGatherChunk + kGatherChunk / 8 + 1);

// gather_slots for short lists (brick partials, ~2.4 per node): each lane reads its node's
// entries directly, in the same order, so the sums are bitwise those of gather_slots.
__device__ __forceinline__ void gather_direct(int n, const int32_t* __restrict__ nptr, const float* __restrict__ Fe,
                                              bool want, float (&y)[3]) {
    y[0] = y[1] = y[2] = 0.0f;
    if (!want) return;
    const int b = nptr[n], e = nptr[n + 1];
    for (int c = b; c < e; ++c) {
        y[0] += Fe[3 * (int64_t)c];
        y[1] += Fe[3 * (int64_t)c + 1];
        y[2] += Fe[3 * (int64_t)c + 2];
    }
}

// One thread per element: element force f_e = K_e p_e.  J is rebuilt from the node
// coordinates relative to the element's first node (formed in FP64, so that FP32 keeps the
// element's own scale), the compact tangent is read per QP, and f_a is written to the
// node-sorted slot pos[a][e] of the force list, so the gather reads contiguous memory.
template <int NN, int Q, int NC, typename TP>
__global__ __launch_bounds__(256) void mf_apply_kernel(int E, int N, const int32_t* __restrict__ conn,
                                                       const double* __restrict__ coords,
                                                       const float* __restrict__ dnxi,
                                                       const float* __restrict__ mfC, const TP* __restrict__ p,
                                                       const uint8_t* __restrict__ dirflag, int mask,
                                                       const int* __restrict__ flags,
                                                       const int32_t* __restrict__ pos, float* __restrict__ Fs,
                                                       const int* __restrict__ active,
                                                       const int32_t* __restrict__ specOfElem) {
    if (flags && flags[0]) return;
    const int e = xcd_block_mf() * 256 + threadIdx.x;
    if (e >= E) return;
    if (active && !active[specOfElem[e]]) return;  // frozen specimen of a batched solve
    float pe[NN][3], fe[NN][3], xe[NN][3];
    double x0[3];
    // the tangents are streamed once per product: non-temporal loads keep them from
    // evicting the gathered p and coordinates from L2 (measured: 131 us instead of 151 us
    // at 96^3; for the connectivity and slot indices plain loads are faster)
#pragma unroll
    for (int a = 0; a < NN; ++a) {
        const int nd = conn[(int64_t)a * E + e];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            float v = (float)p[3 * nd + i];
            if (mask && dirflag[3 * nd + i]) v = 0.0f;
            pe[a][i] = v;
            fe[a][i] = 0.0f;
            const double xc = coords[(int64_t)i * N + nd];
            if (a == 0) x0[i] = xc;
            xe[a][i] = (float)(xc - x0[i]);
        }
    }
    for (int q = 0; q < Q; ++q) {
        const float* dn = dnxi + q * NN * 3;
        const float* dj = dnxi + (Q + q) * NN * 3;  // the table J is formed with
        float H[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};  // H[i*3+k] = sum_a p_a,i dN_a/dxi_k
        float J[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};  // J[k*3+c] = sum_a dJ_a/dxi_k x_a,c
#pragma unroll
        for (int a = 0; a < NN; ++a) {
            const float d[3] = {dn[a * 3], dn[a * 3 + 1], dn[a * 3 + 2]};
            const float dk[3] = {dj[a * 3], dj[a * 3 + 1], dj[a * 3 + 2]};
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    H[i * 3 + k] += pe[a][i] * d[k];
                    J[k * 3 + i] += dk[k] * xe[a][i];
                }
        }
        const float det = J[0] * (J[4] * J[8] - J[5] * J[7]) - J[1] * (J[3] * J[8] - J[5] * J[6]) +
                          J[2] * (J[3] * J[7] - J[4] * J[6]);
        const float id = 1.0f / det;
        const float iJ[9] = {(J[4] * J[8] - J[5] * J[7]) * id, (J[2] * J[7] - J[1] * J[8]) * id,
                             (J[1] * J[5] - J[2] * J[4]) * id, (J[5] * J[6] - J[3] * J[8]) * id,
                             (J[0] * J[8] - J[2] * J[6]) * id, (J[2] * J[3] - J[0] * J[5]) * id,
                             (J[3] * J[7] - J[4] * J[6]) * id, (J[1] * J[6] - J[0] * J[7]) * id,
                             (J[0] * J[4] - J[1] * J[3]) * id};
        // du_i/dx_j = sum_k H_ik iJ_jk
        float g[9];
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j)
                g[i * 3 + j] = H[i * 3] * iJ[j * 3] + H[i * 3 + 1] * iJ[j * 3 + 1] + H[i * 3 + 2] * iJ[j * 3 + 2];
        const float ep[6] = {g[0], g[4], g[8], g[1] + g[3], g[2] + g[6], g[5] + g[7]};
        float cf[NC];
#pragma unroll
        for (int k = 0; k < NC; ++k) cf[k] = __builtin_nontemporal_load(mfC + (int64_t)(q * NC + k) * E + e);
        const float A = cf[0], B = cf[1], cnn = cf[2];
        const float cn1 = NC == 10 ? cf[3] : 0.0f, c1n = NC == 10 ? cf[4] : 0.0f;
        const float* nc = cf + (NC == 10 ? 5 : 3);
        const float n[6] = {nc[0], nc[1], -(nc[0] + nc[1]), nc[2], nc[3], nc[4]};  // n deviatoric
        const float tr = ep[0] + ep[1] + ep[2];
        const float ne = n[0] * ep[0] + n[1] * ep[1] + n[2] * ep[2] + n[3] * ep[3] + n[4] * ep[4] + n[5] * ep[5];
        const float t3 = tr * (1.0f / 3.0f);
        const float sn = cnn * ne + cn1 * tr;     // coefficient of n
        const float s1 = A * tr + c1n * ne;       // coefficient of 1
        float sg[6];
#pragma unroll
        for (int i = 0; i < 3; ++i) sg[i] = s1 + B * (ep[i] - t3) + sn * n[i];
#pragma unroll
        for (int i = 3; i < 6; ++i) sg[i] = 0.5f * B * ep[i] + sn * n[i];
        // tensor sigma (Voigt 11,22,33,12,13,23); M_ik = sum_j sig_ij iJ_jk
        const float S[9] = {sg[0], sg[3], sg[4], sg[3], sg[1], sg[5], sg[4], sg[5], sg[2]};
        float M[9];
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int k = 0; k < 3; ++k)
                M[i * 3 + k] = S[i * 3] * iJ[k] + S[i * 3 + 1] * iJ[3 + k] + S[i * 3 + 2] * iJ[6 + k];
#pragma unroll
        for (int a = 0; a < NN; ++a) {
            const float d0 = dn[a * 3], d1 = dn[a * 3 + 1], d2 = dn[a * 3 + 2];
#pragma unroll
            for (int i = 0; i < 3; ++i) fe[a][i] += M[i * 3] * d0 + M[i * 3 + 1] * d1 + M[i * 3 + 2] * d2;
        }
    }
#pragma unroll
    for (int a = 0; a < NN; ++a) {
        float* dst = Fs + (int64_t)pos[(int64_t)a * E + e] * 3;
#pragma unroll
        for (int i = 0; i < 3; ++i) dst[i] = fe[a][i];
    }
}

// Hexa8 with 2x2x2 Gauss points: the product with the trilinear interpolation written in
// monomials.  A nodal field v gives v(x, y, z) = c0 + c_x x + c_y y + c_z z + c_xy xy +
// c_yz yz + c_xz xz + c_xyz xyz with c = (1/8) H v (H: the +-1 Walsh matrix of the node
// signs, applied as a 3-stage butterfly), so its natural gradient at a point costs 3 FMA per
// direction instead of a sum over the 8 nodes; the element forces f_a = sum_q M_q grad N_a(q)
// are accumulated in the same monomial basis and mapped back to the nodes by the transposed
// butterfly.  J (from the coordinates) and H = grad p use the first form, the forces the
// second: 90 instead of 216 multiply-adds per QP.  The evaluation point of QP q is the
// reference's exchanged point (eta_q, xi_q, zeta_q).
//
// Node order (xi, eta, zeta) signs: n0 (-,-,-) n1 (-,-,+) n2 (+,-,+) n3 (+,-,-) n4 (-,+,-)
// n5 (-,+,+) n6 (+,+,+) n7 (+,+,-); canonical butterfly index k = [xi>0] + 2 [eta>0] +
// 4 [zeta>0]:
__constant__ int8_t kHex8Canon[8] = {0, 3, 4, 7, 1, 2, 5, 6};  // node of canonical index k

// in place: w[k] (canonical order) -> r[k] = sum_j prod_{i in bits(k)} s_i(j) w[j]
template <typename T>
__device__ __forceinline__ void walsh3(T (&w)[8]) {
#pragma unroll
    for (int h = 1; h < 8; h <<= 1)
#pragma unroll
        for (int k = 0; k < 8; ++k)
            if (!(k & h)) {
                const T lo = w[k], hi = w[k | h];
                w[k] = lo + hi;
                w[k | h] = hi - lo;
            }
}

// in place: A[k] (monomial coefficients, A[0] = 0) -> f[k] = sum_S A_S prod_{i in S} s_i(k)
template <typename T>
__device__ __forceinline__ void walsh3_t(T (&w)[8]) {
#pragma unroll
    for (int h = 1; h < 8; h <<= 1)
#pragma unroll
        for (int k = 0; k < 8; ++k)
            if (!(k & h)) {
                const T lo = w[k], hi = w[k | h];
                w[k] = lo - hi;
                w[k | h] = lo + hi;
            }
}

// One QP at (x, y, z): adds its share of the element's forces in the monomial basis (fa, x 8), from
// the coefficients of p (cp) and of the coordinates (cx) and its NC values cf.
template <int NC, typename T>
__device__ __forceinline__ void brick_qp(const T (&cf)[NC ? NC : 1], T bulk, T shear2, T x, T y, T z,
                                         const T (&cp)[3][8], const T (&cx)[3][8], T (&fa)[3][8]) {
    const T xy = x * y, yz = y * z, xz = x * z;
    // natural gradients: d/dx = c1 + c3 y + c5 z + c7 yz, d/dy = c2 + c3 x + c6 z + c7 xz,
    // d/dz = c4 + c5 x + c6 y + c7 xy   (index = canonical monomial bits)
    T H[9], J[9];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        H[i * 3 + 0] = cp[i][1] + cp[i][3] * y + cp[i][5] * z + cp[i][7] * yz;
        H[i * 3 + 1] = cp[i][2] + cp[i][3] * x + cp[i][6] * z + cp[i][7] * xz;
        H[i * 3 + 2] = cp[i][4] + cp[i][5] * x + cp[i][6] * y + cp[i][7] * xy;
        J[0 * 3 + i] = cx[i][1] + cx[i][3] * y + cx[i][5] * z + cx[i][7] * yz;
        J[1 * 3 + i] = cx[i][2] + cx[i][3] * x + cx[i][6] * z + cx[i][7] * xz;
        J[2 * 3 + i] = cx[i][4] + cx[i][5] * x + cx[i][6] * y + cx[i][7] * xy;
    }
    const T det = J[0] * (J[4] * J[8] - J[5] * J[7]) - J[1] * (J[3] * J[8] - J[5] * J[6]) +
                  J[2] * (J[3] * J[7] - J[4] * J[6]);
    const T id = (T)1 / det;
    const T iJ[9] = {(J[4] * J[8] - J[5] * J[7]) * id, (J[2] * J[7] - J[1] * J[8]) * id,
                     (J[1] * J[5] - J[2] * J[4]) * id, (J[5] * J[6] - J[3] * J[8]) * id,
                     (J[0] * J[8] - J[2] * J[6]) * id, (J[2] * J[3] - J[0] * J[5]) * id,
                     (J[3] * J[7] - J[4] * J[6]) * id, (J[1] * J[6] - J[0] * J[7]) * id,
                     (J[0] * J[4] - J[1] * J[3]) * id};
    T gr[9];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j)
            gr[i * 3 + j] = H[i * 3] * iJ[j * 3] + H[i * 3 + 1] * iJ[j * 3 + 1] + H[i * 3 + 2] * iJ[j * 3 + 2];
    const T ep[6] = {gr[0], gr[4], gr[8], gr[1] + gr[3], gr[2] + gr[6], gr[5] + gr[7]};
    // the Gauss weights of hexa8 are 1: w detJ = det
    const T A = NC == 10 ? cf[0] : bulk * det;
    const T B = NC == 10 ? cf[1] : (NC == 7 ? cf[0] : shear2 * det);
    const T tr = ep[0] + ep[1] + ep[2], t3 = tr * (T)(1.0 / 3.0);
    T s1 = A * tr, sg[6];
    if constexpr (NC != 0) {
        const T* nc = cf + (NC == 10 ? 5 : 2);
        const T n[6] = {nc[0], nc[1], -(nc[0] + nc[1]), nc[2], nc[3], nc[4]};  // n deviatoric
        const T ne_ = n[0] * ep[0] + n[1] * ep[1] + n[2] * ep[2] + n[3] * ep[3] + n[4] * ep[4] + n[5] * ep[5];
        T sn = (NC == 10 ? cf[2] : cf[1]) * ne_;
        if constexpr (NC == 10) {
            sn += cf[3] * tr;
            s1 += cf[4] * ne_;
        }
#pragma unroll
        for (int i = 0; i < 3; ++i) sg[i] = s1 + B * (ep[i] - t3) + sn * n[i];
#pragma unroll
        for (int i = 3; i < 6; ++i) sg[i] = (T)0.5 * B * ep[i] + sn * n[i];
    } else {
#pragma unroll
        for (int i = 0; i < 3; ++i) sg[i] = s1 + B * (ep[i] - t3);
#pragma unroll
        for (int i = 3; i < 6; ++i) sg[i] = (T)0.5 * B * ep[i];
    }
    const T S[9] = {sg[0], sg[3], sg[4], sg[3], sg[1], sg[5], sg[4], sg[5], sg[2]};
    // f_a,i += sum_k M_ik dN_a/dxi_k with M_ik = sum_j sig_ij iJ_jk, in monomials:
    // fa[1] += M0, fa[2] += M1, fa[4] += M2, fa[3] += M0 y + M1 x, fa[5] += M0 z + M2 x,
    // fa[6] += M1 z + M2 y, fa[7] += M0 yz + M1 xz + M2 xy   (M_k = column k, x 1/8)
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const T m0 = S[i * 3] * iJ[0] + S[i * 3 + 1] * iJ[3] + S[i * 3 + 2] * iJ[6];
        const T m1 = S[i * 3] * iJ[1] + S[i * 3 + 1] * iJ[4] + S[i * 3 + 2] * iJ[7];
        const T m2 = S[i * 3] * iJ[2] + S[i * 3 + 1] * iJ[5] + S[i * 3 + 2] * iJ[8];
        fa[i][1] += m0;
        fa[i][2] += m1;
        fa[i][4] += m2;
        fa[i][3] += m0 * y + m1 * x;
        fa[i][5] += m0 * z + m2 * x;
        fa[i][6] += m1 * z + m2 * y;
        fa[i][7] += m0 * yz + m1 * xz + m2 * xy;
    }
}

// The sum over the element's QPs, whose tangents start at Cg.  HOT: plain loads, which leave the
// tangents in the Infinity Cache for the next product; else non-temporal ones.  The loop is not
// unrolled: unrolled, it hoists the tangent loads of all QPs and needs half as many registers again.
template <int NC, typename T, bool HOT>
__device__ __forceinline__ void brick_qps(const T* __restrict__ Cg, T bulk, T shear2, const T (&cp)[3][8],
                                          const T (&cx)[3][8], T (&fa)[3][8]) {
    const T gq = (T)0.57735026918962576451;
#pragma unroll 1
    for (int q = 0; q < 8; ++q) {
        // evaluation point (eta_q, xi_q, zeta_q) of the QP table xi = (-,-,-,-,+,+,+,+),
        // eta = (-,-,+,+,-,-,+,+), zeta = (-,+,+,-,-,+,+,-) (times 1/sqrt 3)
        const int r = q & 3;
        T cf[NC ? NC : 1];
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            const T* src = Cg + (q * NC + k) * kBrick;
            if constexpr (HOT) cf[k] = *src;
            else cf[k] = __builtin_nontemporal_load(src);
        }
        brick_qp<NC, T>(cf, bulk, shear2, (r < 2 ? -gq : gq), (q < 4 ? -gq : gq), ((r == 1 || r == 2) ? gq : -gq), cp,
                        cx, fa);
    }
}

// What a workgroup of the brick product reads besides the tangents (bricks.cpp).
struct BrickTables {
    const int32_t *lnode, *lpos, *spec;
    const uint16_t *linc, *lidx;
    const double* X;  // [3][G * NB] coordinates of the staged nodes
    int G, hot;
};

// Hexa8 product by bricks: workgroup g takes the up to kBrick / P elements of brick g, P = 1 or 8
// lanes each.
// The brick's distinct nodes (p with Dirichlet DOFs masked, and the coordinates, which lie in
// staging order) go to LDS once, after two dependent loads (the node, then its values: the tables
// have a fixed pitch, and the flags are waited for beside them); each lane forms its element's forces in the monomial basis and
// leaves them in LDS; each staged node's forces are summed in element order into one partial
// per (brick, node), stored at its slot of the node-ordered partial list.
//
// NC values per QP are read: 7 (w detJ [B, c_nn], n_11, n_22, n_12, n_13, n_23), with the
// volumetric coefficient A = K w detJ formed from the element's bulk modulus and the determinant
// at hand; 10 with Drucker-Prager (A, B, c_nn, c_n1, c_1n and n as stored); 0 when every
// element is linear elastic (B = 2 G w detJ likewise).  T is the precision of the arithmetic,
// the tangents and the partials.
//
// P = 8 (split bricks): a lane has one QP; its forces on the 8 nodes are summed over the element's
// lanes by halving exchanges, which leave each lane one node's.  This repeats the element's set-up in
// 8 lanes, but takes the tangents in one round of loads and needs 32 elements per CU, not 256: the
// product of a small mesh is a chain of latencies (320 elements: 9.3 us on two whole bricks).
template <int NC, typename T, typename TP, int P>
__global__ __launch_bounds__(kBrick) void brick_apply_kernel(
    BrickTables bt, const T* __restrict__ el, const T* __restrict__ C, const TP* __restrict__ p,
    const uint8_t* __restrict__ dirflag, int mask, const int* __restrict__ flags, T* __restrict__ Fpart,
    const int* __restrict__ active, double* __restrict__ part) {
    constexpr int EB = kBrick / P, NB = P == 1 ? kBrickNodes : 8 * EB;
    // LDS, reused: first the staged nodes (x 3 doubles, p 3 T), then the element forces (24 T each)
    constexpr int kStage = 3 * NB * (int)(sizeof(double) + sizeof(T));
    constexpr int kForce = 24 * EB * (int)sizeof(T);
    __shared__ __align__(16) char lds[kStage > kForce ? kStage : kForce];
    __shared__ double red[kBrick / 64];
    double* sx = (double*)lds;
    T* sp = (T*)(lds + 3 * NB * sizeof(double));
    T* sf = (T*)lds;
    const int g = xcd_block_mf();
    if (g >= bt.G) {  // the grid is rounded up to a multiple of 8
        if (part && threadIdx.x == 0) part[g] = 0.0;
        return;
    }
    constexpr int NS = NB / kBrick;  // staged nodes per lane
    const int t = threadIdx.x;
    const int64_t l0 = (int64_t)g * NB + t;
    int nd[NS];
#pragma unroll
    for (int k = 0; k < NS; ++k) nd[k] = bt.lnode[l0 + k * kBrick];
    // the element's 8 staged entries in one 16-byte load; 0xffff: no element for this lane
    const int el0 = g * EB + t / P;  // the lane's element
    const uint4 li4 = *reinterpret_cast<const uint4*>(bt.lidx + (int64_t)el0 * 8);
    const T bulk = NC != 10 ? el[el0] : (T)0;
    const T shear2 = NC == 0 ? el[(int64_t)bt.G * EB + el0] : (T)0;
    if (flags && flags[0]) return;
    // batched solves: a brick of a frozen specimen leaves its partials alone (nobody reads them)
    if (active && !active[bt.spec[g]]) return;
    const T* Cg = C + (int64_t)g * (8 / P * NC * kBrick) + t;
    T cf[NC ? NC : 1];  // P = 8: the lane's tangent
    if constexpr (P == 8)
#pragma unroll
        for (int k = 0; k < NC; ++k) cf[k] = Cg[k * kBrick];
#pragma unroll
    for (int k = 0; k < NS; ++k)
        if (nd[k] >= 0) {
            const int i = t + k * kBrick;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                T v = (T)p[3 * (int64_t)nd[k] + c];
                if (mask && dirflag[3 * (int64_t)nd[k] + c]) v = (T)0;
                sp[c * NB + i] = v;
                sx[c * NB + i] = bt.X[(int64_t)c * bt.G * NB + l0 + k * kBrick];
            }
        }
    const bool live = (li4.x & 0xffffu) != 0xffffu;
    __syncthreads();
    T cp[3][8], cx[3][8];
    if (live) {
        const uint32_t lw[4] = {li4.x, li4.y, li4.z, li4.w};
        int loc[8];
#pragma unroll
        for (int a = 0; a < 8; ++a) loc[a] = (int)((lw[a >> 1] >> (16 * (a & 1))) & 0xffffu);
        // coordinates relative to node 0, the difference formed in FP64, so that FP32 keeps the
        // element's own scale
        double x0[3];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int l = loc[kHex8Canon[k]];
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                cp[i][k] = sp[i * NB + l];
                const double xc = sx[i * NB + l];
                if (k == 0) x0[i] = xc;
                cx[i][k] = (T)(xc - x0[i]);
            }
        }
    }
    __syncthreads();  // the staging area becomes the force area
    // with part given: the brick's sum of p_e . f_e (its share of p . K p), formed in the
    // monomial basis: f = H^T fa / 8 and cp = H p / 8 with H H = 8 I give p . f = cp . fa
    double en = 0.0;
    uint4 inc[NS];
    int lp[NS];
    auto load_lists = [&] {  // of the staged nodes, for the sums at the end
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            inc[k] = *reinterpret_cast<const uint4*>(bt.linc + (l0 + k * kBrick) * 8);
            lp[k] = bt.lpos[l0 + k * kBrick];
        }
    };
    if (live) {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            walsh3(cp[i]);
            walsh3(cx[i]);
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                cp[i][k] *= (T)0.125;
                cx[i][k] *= (T)0.125;
            }
        }
        T fa[3][8];
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int k = 0; k < 8; ++k) fa[i][k] = (T)0;
        if constexpr (P == 8) {
            const T gq = (T)0.57735026918962576451;
            const int q = t & 7, r = q & 3;  // as in brick_qps
            brick_qp<NC, T>(cf, bulk, shear2, (r < 2 ? -gq : gq), (q < 4 ? -gq : gq), ((r == 1 || r == 2) ? gq : -gq),
                            cp, cx, fa);
        } else if (g < bt.hot) {
            brick_qps<NC, T, true>(Cg, bulk, shear2, cp, cx, fa);
        } else {
            brick_qps<NC, T, false>(Cg, bulk, shear2, cp, cx, fa);
        }
        if (part)
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int k = 0; k < 8; ++k) en += (double)cp[i][k] * (double)fa[i][k];
        load_lists();
#pragma unroll
        for (int i = 0; i < 3; ++i) walsh3_t(fa[i]);
        if constexpr (P == 8) {
            // lanes with the bit of the halved index set keep the upper half
            const bool b4 = t & 4, b2 = t & 2, b1 = t & 1;
            const int slot = t - (t & 7) + kHex8Canon[t & 7];
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                T u[4], v[2];
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    u[k] = (b4 ? fa[i][k + 4] : fa[i][k]) + lane_xor8<4>(b4 ? fa[i][k] : fa[i][k + 4]);
#pragma unroll
                for (int k = 0; k < 2; ++k) v[k] = (b2 ? u[k + 2] : u[k]) + lane_xor8<2>(b2 ? u[k] : u[k + 2]);
                sf[i * 8 * EB + slot] = (T)0.125 * ((b1 ? v[1] : v[0]) + lane_xor8<1>(b1 ? v[0] : v[1]));
            }
        } else {
            // forces [i][a][t]: consecutive lanes in consecutive banks
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int a = kHex8Canon[k];
#pragma unroll
                for (int i = 0; i < 3; ++i) sf[(i * 8 + a) * kBrick + t] = (T)0.125 * fa[i][k];
            }
        }
    } else {
        load_lists();
    }
    __syncthreads();
    // one partial per staged node: its up to 8 incidences in element order
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        if (nd[k] < 0) continue;
        const uint32_t w[4] = {inc[k].x, inc[k].y, inc[k].z, inc[k].w};
        T f0 = (T)0, f1 = (T)0, f2 = (T)0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t s = (w[j >> 1] >> (16 * (j & 1))) & 0xffffu;
            if (s != 0xffffu) {
                f0 += sf[s];
                f1 += sf[8 * EB + s];
                f2 += sf[16 * EB + s];
            }
        }
        T* dst = Fpart + (int64_t)lp[k] * 3;
        dst[0] = f0;
        dst[1] = f1;
        dst[2] = f2;
    }
    if (part) {
        const double sum = block_sum_mf<kBrick>(en, red);
        if (threadIdx.x == 0) part[g] = sum;
    }
}

// Batched solves (hexa20): q = K p on the nodes of active specimens and the per-node p.q values
// that the per-specimen reductions sum; nodes of frozen specimens are left alone (p.q 0).
__global__ __launch_bounds__(256) void mf_gather_batched_kernel(int N, const int32_t* __restrict__ nptr,
                                                                const float* __restrict__ Fe,
                                                                const float* __restrict__ p,
                                                                const uint8_t* __restrict__ dirflag,
                                                                const int32_t* __restrict__ spec,
                                                                const int* __restrict__ active, float* __restrict__ q,
                                                                double* __restrict__ npq) {
    __shared__ float buf[kGatherLds];
    const int n0 = blockIdx.x * 256, n = n0 + threadIdx.x;
    const bool valid = n < N;
    const bool act = valid && active[spec[n]];
    float yv[3];
    gather_slots<256>(n0, N, nptr, Fe, act, buf, yv);
    if (!valid) return;
    if (!act) {
        npq[n] = 0.0;
        return;
    }
    double dot = 0.0;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const float pv = p[3 * n + i];
        if (dirflag[3 * n + i]) yv[i] = pv;
        q[3 * n + i] = yv[i];
        dot += (double)pv * yv[i];
    }
    npq[n] = dot;
}

// MODE 0 (operator): y = sum of the node's element forces in element order on free DOFs,
// y = p on Dirichlet DOFs, per-workgroup partials of p.y.  MODE 1 (correction): y = the
// sum on free DOFs, 0 on Dirichlet DOFs.
template <int BS, int MODE, typename TP, typename TY, bool DIRECT = false>
__global__ __launch_bounds__(BS) void mf_gather_kernel(int N, const int32_t* __restrict__ nptr,
                                                       const int32_t* __restrict__ nlist,
                                                       const float* __restrict__ Fe, const TP* __restrict__ p,
                                                       const uint8_t* __restrict__ dirflag,
                                                       TY* __restrict__ y, double* __restrict__ part,
                                                       const int* __restrict__ flags, int kr) {
    __shared__ float buf[DIRECT ? 1 : kGatherLds];
    __shared__ double sh[BS / 64];
    if (flags && flags[0]) return;
    const int blk = xcd_block_mf();
    double dot = 0.0;
    for (int it = 0; it < kr; ++it) {
        const int n0 = (blk * kr + it) * BS;
        if (n0 >= N) break;
        const int n = n0 + threadIdx.x;
        const bool valid = n < N;
        float yv[3];
        if (DIRECT) gather_direct(n, nptr, Fe, valid, yv);
        else gather_slots<BS>(n0, N, nptr, Fe, valid, buf, yv);
        if (!valid) continue;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const bool d = dirflag[3 * n + i];  // always allocated; not ndir, which a captured graph would freeze
            if (MODE == 0) {
                const float pv = (float)p[3 * n + i];
                if (d) yv[i] = pv;
                dot += (double)pv * yv[i];
            } else if (d) {
                yv[i] = 0.0f;
            }
            y[3 * n + i] = (TY)yv[i];
        }
    }
    if (MODE == 0 && part) {
        const double s = block_sum_mf<BS>(dot, sh);
        if (threadIdx.x == 0) part[blk] = s;
    }
}

// Diagonal 3x3 blocks (element order), symmetric Dirichlet elimination inside the block,
// block-Jacobi inverse, and the P / F gather of the element residuals.
__global__ __launch_bounds__(256) void mf_diag_kernel(
    int N, const int32_t* __restrict__ nptr, const int32_t* __restrict__ nlist, const float* __restrict__ Kscr,
    const double* __restrict__ Pscr, const uint8_t* __restrict__ dirflag, int ndir, float* __restrict__ Minv,
    double* __restrict__ P, double* __restrict__ F, const int* __restrict__ specActive,
    const int32_t* __restrict__ specOfNode) {
    // XCD-aware numbering: each XCD sums a contiguous node range, so the element blocks that
    // neighbouring node rows share are fetched into one L2, not into several
    const int n = xcd_block_mf() * blockDim.x + threadIdx.x;
    if (n >= N) return;
    if (specActive && !specActive[specOfNode[n]]) return;  // a skipped specimen keeps its rows
    // K_nn = sum of the K_aa blocks [e][a][9] of the (element, local node) pairs of node n,
    // in element order (the order of the diagonal block's contributions in the assembly)
    float acc[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll 4
    for (int c = nptr[n]; c < nptr[n + 1]; ++c) add_block(Kscr + (int64_t)nlist[c] * kBlockPitch, acc);
    double dg[9];
#pragma unroll
    for (int v = 0; v < 9; ++v) dg[v] = acc[v];
    if (nptr[n] == nptr[n + 1]) dg[0] = dg[4] = dg[8] = 1.0;  // a node outside every element, as in the assembly
    if (ndir) {
        const bool fr[3] = {(bool)dirflag[3 * n], (bool)dirflag[3 * n + 1], (bool)dirflag[3 * n + 2]};
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j)
                if (fr[i] || fr[j]) dg[i * 3 + j] = (i == j) ? 1.0 : 0.0;
    }
    const double det = dg[0] * (dg[4] * dg[8] - dg[5] * dg[7]) - dg[1] * (dg[3] * dg[8] - dg[5] * dg[6]) +
                       dg[2] * (dg[3] * dg[7] - dg[4] * dg[6]);
    const double id = 1.0 / det;
    const double iv[9] = {(dg[4] * dg[8] - dg[5] * dg[7]) * id, (dg[2] * dg[7] - dg[1] * dg[8]) * id,
                          (dg[1] * dg[5] - dg[2] * dg[4]) * id, (dg[5] * dg[6] - dg[3] * dg[8]) * id,
                          (dg[0] * dg[8] - dg[2] * dg[6]) * id, (dg[2] * dg[3] - dg[0] * dg[5]) * id,
                          (dg[3] * dg[7] - dg[4] * dg[6]) * id, (dg[1] * dg[6] - dg[0] * dg[7]) * id,
                          (dg[0] * dg[4] - dg[1] * dg[3]) * id};
#pragma unroll
    for (int v = 0; v < 9; ++v) Minv[(int64_t)n * 9 + v] = (float)iv[v];
    double p0 = 0, p1 = 0, p2 = 0, f0 = 0, f1 = 0, f2 = 0;
#pragma unroll 4
    for (int c = nptr[n]; c < nptr[n + 1]; ++c) {
        const double* src = Pscr + (int64_t)nlist[c] * 3;
        p0 += src[0];
        p1 += src[1];
        p2 += src[2];
        f0 += fabs(src[0]);
        f1 += fabs(src[1]);
        f2 += fabs(src[2]);
    }
    P[3 * n] = p0;
    P[3 * n + 1] = p1;
    P[3 * n + 2] = p2;
    F[3 * n] = f0;
    F[3 * n + 1] = f1;
    F[3 * n + 2] = f2;
}

inline int round8_mf(int n) { return (n + 7) & ~7; }

#define MF_ARGS \
    c->E, c->N, c->conn, c->coords, c->dnxi32, c->mfC, p, c->dirflag, mask, flags, c->elemPos, c->mfF, active, \
        c->specOfElem

// T: precision of the product (float: the matrix-free operator; double: bricks of the FP64 pass)
template <typename T, typename TP>
void launch_bricks(efe_ctx* c, hipStream_t st, const TP* p, int mask, const int* flags, const int* active,
                   double* part) {
    // The Infinity Cache (256 MB) serves the tangents from one product to the next when they and
    // what a PCG iteration touches beside them fit: plain loads then, else non-temporal ones, which
    // keep the tangents from displacing the rest.  PCG iteration at 64^3 FP64 (117 + 90 MB) 69.6 ->
    // 62.7 us, 80^3 FP32 (115 + 90 MB) 82 -> 72 us; beyond it plain loads cost more: 80^3 FP64
    // (229 + 160 MB) 129 -> 152 us, 96^3 FP32 119 -> 139 us.  Below ~24 MB the L2s hold them either
    // way (36^3 FP64 25.3 us non-temporal, 26.4 plain).
    const int64_t tangents = (int64_t)c->E * 8 * c->mfNC * (int64_t)sizeof(T);
    const int64_t rest = c->mfbL * (int64_t)(48 + 3 * sizeof(T)) + (int64_t)c->E * (16 + sizeof(T)) +
                         (int64_t)c->N * 21 * (int64_t)sizeof(T);
    const bool hot = tangents > (int64_t)24e6 && tangents + rest <= (int64_t)216e6;
    const BrickTables bt{c->mfbLnode, c->mfbLpos, c->mfbSpec, c->mfbLinc, c->mfbLidx, c->mfbX,
                         c->mfbG,     hot ? c->mfbG : 0};
    const int grid = round8_mf(c->mfbG);
    const T *el, *C;
    T* F;
    if constexpr (sizeof(T) == 8) {
        el = c->mfbEl64;
        C = c->mfC64;
        F = c->mfbF64;
    } else {
        el = c->mfbEl;
        C = c->mfC;
        F = c->mfbF;
    }
#define BRICK_ARGS <<<grid, kBrick, 0, st>>>(bt, el, C, p, c->dirflag, mask, flags, F, active, part)
    if constexpr (sizeof(T) == 4) {
        if (c->mfbE != kBrick) {
            if (c->mfNC == 10) brick_apply_kernel<10, T, TP, 8> BRICK_ARGS;
            else if (c->mfNC == 7) brick_apply_kernel<7, T, TP, 8> BRICK_ARGS;
            else brick_apply_kernel<0, T, TP, 8> BRICK_ARGS;
            return;
        }
        if (c->mfNC == 10) {
            brick_apply_kernel<10, T, TP, 1> BRICK_ARGS;
            return;
        }
    }
    if (c->mfNC == 7) brick_apply_kernel<7, T, TP, 1> BRICK_ARGS;
    else brick_apply_kernel<0, T, TP, 1> BRICK_ARGS;
#undef BRICK_ARGS
}

// the element forces of the hexa20 product
template <typename TP>
void launch_apply(efe_ctx* c, hipStream_t st, const TP* p, int mask, const int* flags, const int* active = nullptr) {
    const int grid = round8_mf((c->E + 255) / 256);
    const bool dp = c->mfNC == 10;
    if (c->eltype == EFE_C3D20) {
        if (dp) mf_apply_kernel<20, 27, 10, TP><<<grid, 256, 0, st>>>(MF_ARGS);
        else mf_apply_kernel<20, 27, 8, TP><<<grid, 256, 0, st>>>(MF_ARGS);
    } else {
        if (dp) mf_apply_kernel<20, 8, 10, TP><<<grid, 256, 0, st>>>(MF_ARGS);
        else mf_apply_kernel<20, 8, 8, TP><<<grid, 256, 0, st>>>(MF_ARGS);
    }
}

template <int BS>
void launch_gather_op(efe_ctx* c, hipStream_t st, const float* p, float* q, double* part, const int* flags,
                      int nwg, int kr) {
    mf_gather_kernel<BS, 0, float, float><<<nwg, BS, 0, st>>>(c->N, c->nptr, c->nlist, c->mfF, p, c->dirflag, q, part,
                                                              flags, kr);
}

// y from FP64 vectors: the product (MODE 0, p masked) or the correction (MODE 1) of mf_gather_kernel
template <int MODE>
void launch_fp64_vectors(efe_ctx* c, const double* p, double* y) {
    const int grid = round8_mf((c->N + 255) / 256), mask = MODE == 0;
    if (c->mfb) {
        launch_bricks<float, double>(c, c->stream, p, mask, nullptr, nullptr, nullptr);
        mf_gather_kernel<256, MODE, double, double, true><<<grid, 256, 0, c->stream>>>(
            c->N, c->mfbPptr, c->nlist, c->mfbF, p, c->dirflag, y, nullptr, nullptr, 1);
    } else {
        launch_apply<double>(c, c->stream, p, mask, nullptr);
        mf_gather_kernel<256, MODE, double, double><<<grid, 256, 0, c->stream>>>(c->N, c->nptr, c->nlist, c->mfF, p,
                                                                                 c->dirflag, y, nullptr, nullptr, 1);
    }
}

}  // namespace

namespace {
// bulk modulus and 2 G of the elements, brick by brick (n places)
template <typename T>
__global__ void brick_moduli_kernel(int E, const double* __restrict__ props, int propStride,
                                    const int32_t* __restrict__ pos, int64_t n, T* __restrict__ el) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= E) return;
    const double y = propStride ? props[e] : props[0], nu = propStride ? props[propStride + e] : props[1];
    el[pos[e]] = (T)(y / (3.0 * (1.0 - 2.0 * nu)));
    el[n + pos[e]] = (T)(y / (1.0 + nu));
}

// the tangents, the moduli and the partials of one precision, in one allocation (at *C); with
// `optional`, *C stays null when there is no memory for them
template <typename T>
int alloc_bricks(efe_ctx* c, T** C, T** el, T** F, bool optional) {
    const size_t n = (size_t)c->mfbG * c->mfbE, nc = n * 8 * (c->mfNC ? c->mfNC : 1);
    const hipError_t e = hipMalloc((void**)C, (nc + 2 * n + (size_t)c->mfbL * 3) * sizeof(T));
    if (e != hipSuccess) *C = nullptr;
    if (optional && e == hipErrorOutOfMemory) {
        (void)hipGetLastError();  // the next launch's check is not to find it
        return EFE_OK;
    }
    EFE_HIP(e);
    *el = *C + nc;
    *F = *el + 2 * n;
    brick_moduli_kernel<T><<<(c->E + 255) / 256, 256, 0, c->stream>>>(c->E, c->props, c->props_per_element ? c->E : 0,
                                                                      c->mfbPos, (int64_t)n, *el);
    EFE_HIP(hipGetLastError());
    return EFE_OK;
}
}  // namespace

// The brick tables, once per context.  (The element passes keep the element order: walking the
// bricks, whose state lies in runs of ~8 elements, took the 64^3 tangent pass from 0.87 to 1.06 ms.)
// One allocation and one copy hold them all.
int efe_mf_upload_bricks(efe_ctx* c, const BrickPattern& bp, const double* coords) {
    const size_t L = bp.lnode.size();
    std::vector<double> X(3 * L, 0.0);
    for (size_t i = 0; i < L; ++i)
        if (bp.lnode[i] >= 0)
            for (int k = 0; k < 3; ++k) X[k * L + i] = coords[(size_t)3 * bp.lnode[i] + k];
    struct Part {
        const void* src;
        size_t bytes;
        void** dst;
    };
    auto part = [](const auto& v, auto** dst) { return Part{v.data(), v.size() * sizeof(v[0]), (void**)dst}; };
    const Part parts[] = {part(bp.pos, &c->mfbPos),   part(bp.lnode, &c->mfbLnode), part(bp.lpos, &c->mfbLpos),
                          part(bp.pptr, &c->mfbPptr), part(bp.linc, &c->mfbLinc),   part(bp.lidx, &c->mfbLidx),
                          part(bp.spec, &c->mfbSpec), part(X, &c->mfbX)};
    size_t total = 0;
    for (const Part& q : parts) total += (q.bytes + 255) & ~(size_t)255;
    std::vector<char> host(total);
    EFE_HIP(hipMalloc(&c->mfbTables, total));
    size_t off = 0;
    for (const Part& q : parts) {
        if (q.bytes) memcpy(host.data() + off, q.src, q.bytes);
        *q.dst = (char*)c->mfbTables + off;
        off += (q.bytes + 255) & ~(size_t)255;
    }
    EFE_HIP(hipMemcpy(c->mfbTables, host.data(), total, hipMemcpyHostToDevice));
    c->mfbL = bp.L;
    c->mfbG = bp.G;
    c->mfbE = bp.EB;
    c->mfb = true;
    return EFE_OK;
}

int efe_mf_alloc_bricks(efe_ctx* c, bool fp64) {
    if (!fp64) return c->mfC ? EFE_OK : alloc_bricks(c, &c->mfC, &c->mfbEl, &c->mfbF, false);
    if (c->mfC64 || c->noBricks64) return EFE_OK;
    const int rc = alloc_bricks(c, &c->mfC64, &c->mfbEl64, &c->mfbF64, true);
    c->noBricks64 = !c->mfC64;  // asked for once: the passes and captured rounds keep one operator
    return rc;
}

bool efe_mf_bricks64(const efe_ctx* c, const uint8_t* which) {
    if (!c->mfC64 || c->mf64Dir.empty()) return false;
    for (int s = 0; s < c->nspec; ++s)
        if ((!which || which[s]) && c->mf64Dir[s] != c->dirVersion) return false;
    return true;
}

void efe_mf_mark64(efe_ctx* c, const uint8_t* which) {
    c->mf64Dir.resize(c->nspec, -1);
    for (int s = 0; s < c->nspec; ++s)
        if (!which || which[s]) c->mf64Dir[s] = c->dirVersion;
}

int efe_mf_alloc(efe_ctx* c) {
    const int NC = c->mfNC;
    if (c->mfC) return EFE_OK;
    if (!c->Minv32) EFE_HIP(hipMalloc(&c->Minv32, (size_t)c->N * 9 * sizeof(float)));
    if (c->eltype == EFE_C3D8) {
        if (!c->mfb) {
            BrickPattern bp;
            bp.EB = c->mfbE;
            efe_build_bricks(bp, c->N, c->E, c->brickConn.data(), c->brickXyz.data(), nullptr);
            if (int rc = efe_mf_upload_bricks(c, bp, c->brickXyz.data())) return rc;
            std::vector<int32_t>().swap(c->brickConn);
            std::vector<double>().swap(c->brickXyz);
        }
        return efe_mf_alloc_bricks(c, false);
    }
    const size_t EQ = (size_t)c->E * c->Q;
    const int64_t L = (int64_t)c->E * c->NN;
    EFE_HIP(hipMalloc(&c->mfC, EQ * NC * sizeof(float)));
    EFE_HIP(hipMalloc(&c->mfF, (size_t)L * 3 * sizeof(float)));
    // FP32 copies of the natural shape-function derivatives at the evaluation points and of
    // the table J is formed with, one after the other
    const size_t nd = (size_t)c->Q * c->NN * 3;
    std::vector<double> h(2 * nd);
    std::vector<float> hf(2 * nd);
    EFE_HIP(hipMemcpy(h.data(), c->dNdxi, nd * sizeof(double), hipMemcpyDeviceToHost));
    EFE_HIP(hipMemcpy(h.data() + nd, c->dJdxi, nd * sizeof(double), hipMemcpyDeviceToHost));
    for (size_t i = 0; i < 2 * nd; ++i) hf[i] = (float)h[i];
    EFE_HIP(hipMalloc(&c->dnxi32, 2 * nd * sizeof(float)));
    EFE_HIP(hipMemcpy(c->dnxi32, hf.data(), 2 * nd * sizeof(float), hipMemcpyHostToDevice));
    return EFE_OK;
}

// Diagonal blocks, Minv, P, F and (optionally) the right-hand-side correction K[:, dir] dir_values.
int efe_launch_mf_assembly(efe_ctx* c, double* P, double* F, const double* dir_values, double* dir_correction) {
    const int grid = (c->N + 255) / 256;
    mf_diag_kernel<<<round8_mf(grid), 256, 0, c->stream>>>(c->N, c->nptr, c->nlist, (const float*)c->Kscr, c->Pscr,
                                                           c->dirflag, c->ndir, c->Minv32, P, F,
                                                           c->useActive ? c->specActive : nullptr, c->specOfNode);
    EFE_HIP(hipGetLastError());
    if (dir_values) {
        launch_fp64_vectors<1>(c, dir_values, dir_correction);
        EFE_HIP(hipGetLastError());
    }
    c->Kprec = EFE_FP32_MATFREE;
    c->Kversion++;
    return EFE_OK;
}

// q = K p (FP32, Dirichlet eliminated) with per-workgroup partials of p.q, for the hexa20 PCG:
// nwg workgroups of bs threads with kr rows per thread.
void efe_mf_launch_operator(efe_ctx* c, hipStream_t st, const float* p, float* q, double* part, const int* flags,
                            int nwg, int bs, int kr) {
    launch_apply<float>(c, st, p, 1, flags);
    switch (bs) {
        case 64: launch_gather_op<64>(c, st, p, q, part, flags, nwg, kr); break;
        case 128: launch_gather_op<128>(c, st, p, q, part, flags, nwg, kr); break;
        case 512: launch_gather_op<512>(c, st, p, q, part, flags, nwg, kr); break;
        default: launch_gather_op<256>(c, st, p, q, part, flags, nwg, kr); break;
    }
}

// The brick product alone (hexa8 bricks only): the node partials of K p for the caller's own
// gather, and per brick the partial of p . K p (Dirichlet DOFs masked) at part[g], g below
// round8(mfbG).
void efe_mf_launch_apply_partials(efe_ctx* c, hipStream_t st, const float* p, double* part, const int* flags,
                                  const int* active) {
    launch_bricks<float, float>(c, st, p, 1, flags, active, part);
}

void efe_mf_launch_apply_partials(efe_ctx* c, hipStream_t st, const double* p, double* part, const int* flags,
                                  const int* active) {
    launch_bricks<double, double>(c, st, p, 1, flags, active, part);
}

// y = K x for FP64 vectors with the matrix-free FP32 operator (Dirichlet eliminated).
int efe_launch_spmv_mf(efe_ctx* c, const double* x, double* y) {
    launch_fp64_vectors<0>(c, x, y);
    EFE_HIP(hipGetLastError());
    return EFE_OK;
}

// Batched hexa20 PCG: q = K p for the active specimens, per-node p.q into npq.
void efe_mf_launch_operator_batched(efe_ctx* c, hipStream_t st, const float* p, float* q, double* npq,
                                    const int* active) {
    launch_apply<float>(c, st, p, 1, nullptr, active);
    mf_gather_batched_kernel<<<(c->N + 255) / 256, 256, 0, st>>>(c->N, c->nptr, c->mfF, p, c->dirflag, c->specOfNode,
                                                                 active, q, npq);
}

void efe_mf_free(efe_ctx* c) {
    // mfC and mfC64 hold the bricks' moduli and partials too
    void* b[] = {c->mfC, c->mfF, c->dnxi32, c->mfC64, c->mfbTables};
    for (void* q : b)
        if (q) hipFree(q);
    c->mfC = c->mfF = c->dnxi32 = nullptr;
    c->mfC64 = nullptr;
    c->mfb = false;
}
