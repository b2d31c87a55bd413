// Element, material and assembly kernels for gfx950.
//
// hex8_kernel (hexa8) is described at its definition; element_kernel (hexa20) follows the same
// three phases, one, two or four 64-lane wavefronts owning EPW elements.
//   phase 1: the nodes' coordinates and increments to LDS, one lane per (element, node); one
//            lane per (element, QP): Jacobian from the coordinates and the shape-function
//            derivatives at the reference's evaluation point; dN/dx over all lanes; one lane
//            per (element, QP): strain increment, FP64 material update of the reference state
//            into the temporary state, and (w detJ) C and (w detJ) sigma staged in LDS;
//   phase 2, one lane per (element, node a, node b), b >= a for symmetric
//            tangents: the 3x3 block
//            K_ab = sum_q B_a^T (w detJ C_q) B_b in KT precision (and K_ba = K_ab^T), written to the
//            element scratch at position cpos[e][a][b] of the contribution order
//            (block slot, then element), so that a row's contributions are
//            contiguous for the assembly;
//   phase 3, one lane per (element, node a): Pe_a = -sum_q B_a^T (w detJ sigma_q).
//   Follows DisplacementElement.computeYourself
//   (edelweissfe/elements/displacementelement/element.py:290-346).
//
// assemble_kernel: one thread per node row-block.  For every block slot of its
//   row it sums the element blocks stored for that slot, in element order (the
//   order of updateCSR, csrgenerator.pyx:112-113), eliminates Dirichlet rows and
//   columns symmetrically, writes the sliced-ELL value layout, inverts its
//   diagonal block for block Jacobi, and gathers P = sum Pe and F = sum |Pe|
//   (nonlinearimplicitstatic.py:843-844) in element order.  No atomics: the
//   result is bitwise reproducible.
#include <cstdlib>
#include <type_traits>

#include "efe_internal.h"
#include "materials.h"

namespace {

template <int MAT>
struct MatState {
    static constexpr int n = (MAT == EFE_LINEAR_ELASTIC) ? 0 : 1;
};

// The compact tangent of QP q of element e for the matrix-free product, from cc = [A, B, cnn, cn1,
// c1n, n]: ncw = 8 [A, B, cnn, n], 7 (A left out), 10 [A, B, cnn, cn1, c1n, n] (cn1 = c1n = 0 but
// DP) or 0 values, the coefficients times f = w detJ; n is deviatoric (n_33 = -n_11 - n_22): its
// five other components are stored.  Element e lies at its place mfPos in the bricks of mfEB elements
// (hexa8), or in element order.  (Constant indices into cc only: a variable one would put it into scratch memory.)
template <typename CT>
__device__ __forceinline__ void store_compact(CT* __restrict__ mfC, const int32_t* __restrict__ mfPos, int mfEB, int E,
                                              int Q, int e, int q, int ncw, double f, const double (&cc)[11]) {
    if (!ncw) return;
    CT* dc;
    int64_t stride = E;
    if (mfPos) {
        const int64_t slot = brick_slot(mfPos[e], q, mfEB);
        stride = kBrick;
        dc = mfC + slot / kBrick * ncw * kBrick + slot % kBrick;
    } else {
        dc = mfC + (int64_t)q * ncw * E + e;
    }
    if (ncw != 7) {
        *dc = (CT)(f * cc[0]);
        dc += stride;
    }
    dc[0] = (CT)(f * cc[1]);
    dc[stride] = (CT)(f * cc[2]);
    dc += 2 * stride;
    if (ncw == 10) {
        dc[0] = (CT)(f * cc[3]);
        dc[stride] = (CT)(f * cc[4]);
        dc += 2 * stride;
    }
    dc[0] = (CT)cc[5];
    dc[stride] = (CT)cc[6];
    dc[2 * stride] = (CT)cc[8];
    dc[3 * stride] = (CT)cc[9];
    dc[4 * stride] = (CT)cc[10];
}

// MF (matrix-free form, KT = float): phase 1 also stores the compact tangent
// w detJ [A, B, cnn, (cn1, c1n,)] and the deviatoric n (five components) per QP for the
// matrix-free operator, and phase 2 forms
// only the diagonal blocks K_aa (for block Jacobi), stored element-major [e][a][9] at the
// start of the element scratch.
// Phase 1 is bound by the latency of its loads, phase 2 by FP64 VALU issue and the block stores.
// With a gather of every node by every QP lane, and the gradients on the 16 (hexa20R: 2 x 8) or 27
// QP lanes alone, a residual pass of 17x15x13 hexa20 J2 took 47 us against 37 us now, of 24x22x20
// hexa20R DP 56 against 43 us, the matrix-free pass of the latter mesh (J2) 51 against 40 us; the
// FP64 tangent passes 147 -> 139 us and 263 -> 255 us.  Coordinates, inverse Jacobians and
// increments lie where the gradients and the weighted stresses follow: in LDS of their own (3 KB
// more) the hexa20R tangent pass got slower (32^3 DP: 705 -> 770 us; as it is, 698 us).
// W wavefronts per workgroup: the tasks of every phase over all of them, each with its own stage
// for the block stores.
template <int NN, int Q, int MAT, typename KT, int EPW, bool MF, int W>
__global__ __launch_bounds__(64 * W) void element_kernel(int E, int N, const double* __restrict__ coords,
                                                     const int32_t* __restrict__ conn,
                                                     const double* __restrict__ props, int propStride,
                                                     const double* __restrict__ dNdxi,
                                                     const double* __restrict__ dJdxi,
                                                     const double* __restrict__ qpw,
                                                     const double* __restrict__ dU,
                                                     const double* __restrict__ sRef, double* __restrict__ sTmp,
                                                     KT* __restrict__ Kscr, double* __restrict__ Pscr,
                                                     int* __restrict__ status,
                                                     float* __restrict__ mfC,
                                                     int* __restrict__ specStatus,
                                                     const int32_t* __restrict__ specOfElem,
                                                     const int32_t* __restrict__ cpos,
                                                     const int* __restrict__ specActive, int formK,
                                                     const int32_t* __restrict__ elist, int ecount, int ncw) {
    constexpr int NS = 12 + MatState<MAT>::n;
    constexpr int NP = (MAT == EFE_LINEAR_ELASTIC) ? 2 : 6;
    // the tangent of every QP in compact form, w detJ [A - B/3, B/2, c_nn, (c_n1, c_1n)] then n:
    // C = A 1(x)1 + B Idev + c_nn n(x)n (+ c_n1 n(x)1 + c_1n 1(x)n for Drucker-Prager)
    constexpr int NCC = (MAT == EFE_DRUCKER_PRAGER) ? 11 : 9;
    // g_s holds the node coordinates until the gradients are formed; w_s in turn the inverse
    // Jacobians, the nodes' increments, and the weighted stresses with the tangents
    __shared__ double g_s[EPW][Q * NN * 3];
    constexpr int kW = EPW * Q * 6 + (EPW * Q * NCC * (int)sizeof(KT) + 7) / 8;
    static_assert(EPW * Q * 9 <= kW && EPW * NN * 3 <= kW, "inverse Jacobians and increments fit");
    static_assert(EPW * Q <= 64 && EPW * NN <= 64, "a lane per (element, QP) and per (element, node)");
    __shared__ double w_s[kW];
    double(*iJ_s)[Q][9] = reinterpret_cast<double(*)[Q][9]>(w_s);
    double(*u_s)[NN][3] = reinterpret_cast<double(*)[NN][3]>(w_s);
    double(*fs_s)[Q][6] = reinterpret_cast<double(*)[Q][6]>(w_s);
    KT(*fC_s)[Q * NCC] = reinterpret_cast<KT(*)[Q * NCC]>(w_s + EPW * Q * 6);
    // assembled passes: blocks staged for word-by-word stores, and their positions (and those
    // of their transposes, -1: none)
    constexpr int kStage = 32;
    __shared__ KT stg_w[MF ? 1 : W][MF ? 1 : kStage][9];
    __shared__ int spos_w[MF ? 1 : W][MF ? 1 : 2 * kStage];
    const int tid = threadIdx.x, lane = tid & 63, wave = W > 1 ? tid >> 6 : 0;
    KT(*stg_s)[9] = stg_w[MF ? 0 : wave];
    int* spos_s = spos_w[MF ? 0 : wave];
    const int64_t EQ = (int64_t)E * Q;
    // Grid-stride over the element list: a grid smaller than the list (a persistent launch)
    // takes EPW elements per workgroup and round.
    for (int e0 = blockIdx.x * EPW; e0 < ecount; e0 += gridDim.x * EPW) {
    // Element el of this round: entry e0 + el of the group's element list (elist, or all
    // elements in order when it is null); -1 past the end and, in batched contexts, for
    // specimens the pass skips.
    auto elem = [&](int el) {
        const int i = e0 + el;
        if (i >= ecount) return -1;
        const int e = elist ? elist[i] : i;
        return (specActive && !specActive[specOfElem[e]]) ? -1 : e;
    };

    // Every node of an element is read once, not once per QP.
    const int nel = tid / NN, na = tid - (tid / NN) * NN;
    const bool hasNode = tid < EPW * NN && elem(nel) >= 0;
    double un[3] = {0, 0, 0};
    if (hasNode) {
        const int nd = conn[(int64_t)na * E + elem(nel)];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            g_s[nel][na * 3 + c] = coords[(int64_t)c * N + nd];
            un[c] = dU[3 * (int64_t)nd + c];
        }
    }
    __syncthreads();
    const int qel = tid / Q, q = tid - (tid / Q) * Q;
    const int e = tid < EPW * Q ? elem(qel) : -1;
    double det = 0.0;
    if (e >= 0) {
        const double* dj = dJdxi + (size_t)q * NN * 3;
        double J[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll 4
        for (int a = 0; a < NN; ++a) {
#pragma unroll
            for (int r = 0; r < 3; ++r) {
                const double d = dj[a * 3 + r];
#pragma unroll
                for (int c = 0; c < 3; ++c) J[r * 3 + c] += d * g_s[qel][a * 3 + c];
            }
        }
        det = J[0] * (J[4] * J[8] - J[5] * J[7]) - J[1] * (J[3] * J[8] - J[5] * J[6]) +
              J[2] * (J[3] * J[7] - J[4] * J[6]);
        const double id = 1.0 / det;
        double* iJ = iJ_s[qel][q];
        iJ[0] = (J[4] * J[8] - J[5] * J[7]) * id;
        iJ[1] = (J[2] * J[7] - J[1] * J[8]) * id;
        iJ[2] = (J[1] * J[5] - J[2] * J[4]) * id;
        iJ[3] = (J[5] * J[6] - J[3] * J[8]) * id;
        iJ[4] = (J[0] * J[8] - J[2] * J[6]) * id;
        iJ[5] = (J[2] * J[3] - J[0] * J[5]) * id;
        iJ[6] = (J[3] * J[7] - J[4] * J[6]) * id;
        iJ[7] = (J[1] * J[6] - J[0] * J[7]) * id;
        iJ[8] = (J[0] * J[4] - J[1] * J[3]) * id;
    }
    __syncthreads();
    for (int t = tid; t < EPW * Q * NN; t += 64 * W) {  // the gradients over all lanes
        const int el = t / (Q * NN), r = t - el * Q * NN;
        if (elem(el) < 0) continue;
        const double d0 = dNdxi[r * 3 + 0], d1 = dNdxi[r * 3 + 1], d2 = dNdxi[r * 3 + 2];
        const double* iJ = iJ_s[el][r / NN];
#pragma unroll
        for (int c = 0; c < 3; ++c) g_s[el][r * 3 + c] = iJ[c * 3 + 0] * d0 + iJ[c * 3 + 1] * d1 + iJ[c * 3 + 2] * d2;
    }
    __syncthreads();
    if (hasNode) {
#pragma unroll
        for (int c = 0; c < 3; ++c) u_s[nel][na][c] = un[c];
    }
    __syncthreads();
    double gr[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};  // gr[i*3+j] = d u_i / d x_j
    if (e >= 0) {
#pragma unroll 4
        for (int a = 0; a < NN; ++a)
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int j = 0; j < 3; ++j) gr[i * 3 + j] += u_s[qel][a][i] * g_s[qel][(q * NN + a) * 3 + j];
    }
    __syncthreads();
    if (e >= 0) {
        double de[6] = {gr[0], gr[4], gr[8], gr[1] + gr[3], gr[2] + gr[6], gr[5] + gr[7]};
        const int64_t sidx = (int64_t)e * Q + q;
        double s[6], ms = 0.0;
#pragma unroll
        for (int c = 0; c < 6; ++c) s[c] = sRef[c * EQ + sidx];
        if (MatState<MAT>::n) ms = sRef[12 * EQ + sidx];
        double p[NP];
#pragma unroll
        for (int k = 0; k < NP; ++k) p[k] = propStride ? props[(int64_t)k * propStride + e] : props[k];
        double C[36], cc[11];
        int st = 0;
        if (MAT == EFE_LINEAR_ELASTIC) st = efe::le_update(p, s, de, C, cc);
        else if (MAT == EFE_VONMISES) st = efe::vm_update(p, s, ms, de, C, cc);
        else st = efe::dp_update(p, s, ms, de, C, cc);
        if (st) {
            *status = 1;
            if (specStatus) specStatus[specOfElem[e]] = 1;  // which specimen asked (batched contexts)
        }
        if (mfC && formK) store_compact(mfC, (const int32_t*)nullptr, 0, E, Q, e, q, ncw, det * qpw[q], cc);
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            sTmp[c * EQ + sidx] = s[c];
            sTmp[(6 + c) * EQ + sidx] = sRef[(6 + c) * EQ + sidx] + de[c];
        }
        if (MatState<MAT>::n) sTmp[12 * EQ + sidx] = ms;
        (void)NS;
        const double f = det * qpw[q];
        if (formK) {
            fC_s[qel][q * NCC + 0] = (KT)(f * (cc[0] - cc[1] * (1.0 / 3.0)));
            fC_s[qel][q * NCC + 1] = (KT)(f * (0.5 * cc[1]));
#pragma unroll
            for (int k = 2; k < NCC - 6; ++k) fC_s[qel][q * NCC + k] = (KT)(f * cc[k]);
#pragma unroll
            for (int k = 0; k < 6; ++k) fC_s[qel][q * NCC + NCC - 6 + k] = (KT)cc[5 + k];
        }
#pragma unroll
        for (int k = 0; k < 6; ++k) fs_s[qel][q][k] = f * s[k];
    }
    __syncthreads();

    // Symmetric tangents (linear elastic, J2): only the blocks a <= b are formed; K_ba is
    // stored as K_ab^T.  Drucker-Prager (non-associative in general) forms all NN^2 blocks.
    constexpr bool SYM = !MF && MAT != EFE_DRUCKER_PRAGER;
    constexpr int NB = MF ? NN : (SYM ? NN * (NN + 1) / 2 : NN * NN);  // blocks per element formed here
    // a residual-only pass (formK = 0) leaves the tangent blocks alone
    // Lanes take an element's blocks one after the other.  The assembled
    // passes write their blocks through LDS, kStage blocks (and their transposes) at a time:
    // the wavefront then stores consecutive words, about seven 72-byte blocks per store
    // instruction instead of one scattered block per lane (48^3 hexa20R DP: 2.34 -> 2.27 ms).
    const int ntask = formK ? EPW * NB : 0;
    for (int t0 = 64 * wave; t0 < ntask; t0 += 64 * W) {
        const int t = t0 + lane;
        const int el = t / NB, r0 = t - (t / NB) * NB;
        int a = 0, b = 0;
        if (MF) {
            a = b = r0;
        } else if (SYM) {  // r0 -> (a, b), upper triangle row by row
            int r = r0;
            while (r >= NN - a) {
                r -= NN - a;
                ++a;
            }
            b = a + r;
        } else {
            a = r0 / NN;
            b = r0 - a * NN;
        }
        const int e = t < ntask ? elem(el) : -1;
        KT acc[9], tr = (KT)0;
#pragma unroll
        for (int k = 0; k < 9; ++k) acc[k] = (KT)0;
        if (e >= 0) {
            for (int q = 0; q < Q; ++q) {
                const KT ax = (KT)g_s[el][(q * NN + a) * 3 + 0], ay = (KT)g_s[el][(q * NN + a) * 3 + 1], az = (KT)g_s[el][(q * NN + a) * 3 + 2];
                const KT bx = (KT)g_s[el][(q * NN + b) * 3 + 0], by = (KT)g_s[el][(q * NN + b) * 3 + 1], bz = (KT)g_s[el][(q * NN + b) * 3 + 2];
                // the block as in hex8_kernel: lambda = A - B/3, mu = B/2 and h = n g
                const KT* cq = fC_s[el] + q * NCC;
                const KT lam = cq[0], mu = cq[1], cnn = cq[2];
                const KT* n = cq + NCC - 6;
                const KT av[3] = {ax, ay, az}, bv[3] = {bx, by, bz};
                const KT ha[3] = {n[0] * ax + n[3] * ay + n[4] * az, n[3] * ax + n[1] * ay + n[5] * az,
                                  n[4] * ax + n[5] * ay + n[2] * az};
                const KT hb[3] = {n[0] * bx + n[3] * by + n[4] * bz, n[3] * bx + n[1] * by + n[5] * bz,
                                  n[4] * bx + n[5] * by + n[2] * bz};
                KT u[3], v[3], w[3];
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    u[i] = lam * av[i];
                    v[i] = cnn * ha[i];
                    w[i] = mu * av[i];
                    if (NCC == 11) {
                        u[i] += cq[3] * ha[i];
                        v[i] += cq[4] * av[i];
                    }
                }
                tr += w[0] * bx + w[1] * by + w[2] * bz;
#pragma unroll
                for (int i = 0; i < 3; ++i)
#pragma unroll
                    for (int j = 0; j < 3; ++j) acc[i * 3 + j] += u[i] * bv[j] + v[i] * hb[j] + w[j] * bv[i];
            }
#pragma unroll
            for (int i = 0; i < 3; ++i) acc[i * 4] += tr;
        }
        if (MF) {  // K_aa element-major at the start of the scratch: [e][a][9]
            if (e >= 0) store_block(Kscr + ((int64_t)e * NN + a) * kBlockPitch, acc);
            continue;
        }
        // the block at position cp[a][b] and, for a symmetric tangent with a != b, its
        // transpose at cp[b][a]; staged kStage lanes at a time, then stored word by word
        const int32_t* cp = cpos + (int64_t)(e >= 0 ? e : 0) * NN * NN;
        const int p0 = e >= 0 ? cp[a * NN + b] : -1;
        const int p1 = (e >= 0 && SYM && a != b) ? cp[b * NN + a] : -1;
        const int nlive = ntask - t0 < 64 ? ntask - t0 : 64;
        for (int s0 = 0; s0 < nlive; s0 += kStage) {
            const int sl = lane - s0;
            if (sl >= 0 && sl < kStage) {
#pragma unroll
                for (int k = 0; k < 9; ++k) stg_s[sl][k] = acc[k];
                spos_s[sl] = p0;
                spos_s[kStage + sl] = p1;
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            const int nb = (nlive - s0 < kStage ? nlive - s0 : kStage);
            for (int w = lane; w < (SYM ? 2 : 1) * kStage * 9; w += 64) {
                const int bi = w / 9, v = w - bi * 9;
                const int src = bi < kStage ? bi : bi - kStage;
                const int pos = src < nb ? spos_s[bi] : -1;
                if (pos >= 0) {
                    const int vv = bi < kStage ? v : (v % 3) * 3 + v / 3;  // K_ba = K_ab^T
                    Kscr[(int64_t)pos * kBlockPitch + v] = stg_s[src][vv];
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
    }

    for (int t = tid; t < EPW * NN; t += 64 * W) {
        const int el = t / NN, a = t - (t / NN) * NN;
        const int e = elem(el);
        if (e < 0) continue;
        double p0 = 0, p1 = 0, p2 = 0;
        for (int q = 0; q < Q; ++q) {
            const double ax = g_s[el][(q * NN + a) * 3 + 0], ay = g_s[el][(q * NN + a) * 3 + 1], az = g_s[el][(q * NN + a) * 3 + 2];
            const double* s = fs_s[el][q];
            p0 += ax * s[0] + ay * s[3] + az * s[4];
            p1 += ay * s[1] + ax * s[3] + az * s[5];
            p2 += az * s[2] + ax * s[4] + ay * s[5];
        }
        double* dst = Pscr + ((int64_t)e * NN + a) * 3;
        dst[0] = -p0;
        dst[1] = -p1;
        dst[2] = -p2;
    }
    __syncthreads();  // the LDS tiles are refilled by the next round
    }
}

// ---- hexa8 passes --------------------------------------------------------------------------------
//
// One wavefront takes 8 elements, lane 8 el + j standing for node j, QP j and block row j of element
// el in turn:
//   fields   each lane loads one node (its coordinates and increment: every node of an element once,
//            not once per QP); three butterfly steps over the lanes of an element turn the nodal
//            values into the coefficients of 1, x, y, xy, ... (the trilinear field in monomials), and
//            a natural gradient at a QP then takes 9 FMA instead of 24;
//   QP       J^-1, strain increment, material update; loads of the state start before the fields;
//   forces   M = w detJ sigma J^-T of every QP to LDS; lane a sums M_q grad N_a(q) over the QPs;
//   blocks   g_a = grad N_a and h_a = n g_a of every QP to LDS; lane a accumulates the blocks
//            (a, a + o), o = 0..4 for a symmetric tangent (36 blocks of the 64, o = 4 for a < 4),
//            four passes of two o otherwise.  With C = A 1(x)1 + B Idev + cnn n(x)n + cn1 n(x)1 +
//            c1n 1(x)n, lambda = A - B/3, mu = B/2:
//              K_ab = sum_q (lambda g_a + cn1 h_a) g_b^T + (c1n g_a + cnn h_a) h_b^T
//                     + mu (g_b g_a^T + (g_a . g_b) I),
//            30 FMA per block and QP (the 6x6 form took about 100), the factors of g_a and h_a
//            formed once per lane and QP for all its blocks.
// What bounds it: the blocks' scattered 72-byte stores (1.2 GB at 64^3 in FP64) and, with 210 VGPRs
// and 26 KB of LDS a wavefront, 6 wavefronts per CU to hide the gathers behind; the residual pass moves
// 0.49 GB at 4.2 TB/s.  64^3 J2, one lane per (element, QP) with table gradients before -> now:
// residual pass 221 -> 117 us (3 wavefronts per SIMD; held to 128 VGPRs it spills and takes 133), FP64
// tangent pass 865 -> 630, FP32 731 -> 411, matrix-free 225 -> 184; linear elastic FP64 828 -> 540;
// Drucker-Prager FP64 985 -> 878.
//
// The QP evaluated at (eta_q, xi_q, zeta_q) of the table lies in the octant of node q, so a
// lane's sign pattern serves it as node and as QP.

// value of lane 0 of the 8 lanes of an element
__device__ __forceinline__ double lane_first8(double v, bool upper) {
    int lo = __double2loint(v), hi = __double2hiint(v);
    lo = __builtin_amdgcn_update_dpp(0, lo, 0x00, 0xF, 0xF, true);  // lane 0 of each quad
    hi = __builtin_amdgcn_update_dpp(0, hi, 0x00, 0xF, 0xF, true);
    const int lm = __builtin_amdgcn_update_dpp(0, lo, 0x141, 0xF, 0xF, true);  // row_half_mirror
    const int hm = __builtin_amdgcn_update_dpp(0, hi, 0x141, 0xF, 0xF, true);
    return __hiloint2double(upper ? hm : hi, upper ? lm : lo);
}

// octant of node (and QP) j: node numbers run (-,-,-) (-,-,+) (+,-,+) (+,-,-), then the same with +y
__host__ __device__ constexpr bool oct_x(int j) { return (j & 2) != 0; }
__host__ __device__ constexpr bool oct_y(int j) { return j >= 4; }
__host__ __device__ constexpr bool oct_z(int j) { return (j & 3) == 1 || (j & 3) == 2; }

template <int MAT, typename KT, bool MF, bool TAN>
struct Hex8Lds {
    static constexpr bool SYM = MAT != EFE_DRUCKER_PRAGER;
    static constexpr int NSC = SYM ? 3 : 5;                 // factors per QP: lambda, mu, cnn (, cn1, c1n)
    static constexpr int QS = 6 * 64 + 1;                   // pitch of a QP's g and h: the lanes of a store, 8
                                                            // QPs of 8 elements, spread over the banks
    static constexpr int kBlocks = SYM ? 288 : 128;         // blocks staged for the stores at a time
    static constexpr size_t fields = 6 * 64 * sizeof(double), forces = 9 * 64 * sizeof(double);
    static constexpr size_t grads = TAN ? (8 * QS + 8 * 8 * NSC) * sizeof(KT) : 0;
    static constexpr size_t stage = TAN && !MF ? kBlocks * (9 * sizeof(KT) + (SYM ? 2 : 1) * sizeof(int)) : 0;
    static constexpr size_t ab = fields > forces ? fields : forces;
    // one pass: the blocks take the place of g and h; two: g and h stay for the second
    static constexpr size_t stageAt = SYM ? 0 : (grads + 7) / 8 * 8;
    static constexpr size_t cd = grads > stageAt + stage ? grads : stageAt + stage;
    static constexpr size_t bytes = ab > cd ? ab : cd;
};

template <int MAT, typename KT, bool MF, bool TAN>
__global__ __launch_bounds__(64) void hex8_kernel(
    int E, int N, const double* __restrict__ coords, const int32_t* __restrict__ conn,
    const double* __restrict__ props, int propStride, const double* __restrict__ dU,
    const double* __restrict__ sRef, double* __restrict__ sTmp, KT* __restrict__ Kscr, double* __restrict__ Pscr,
    int* __restrict__ status, KT* __restrict__ mfC, const int32_t* __restrict__ mfPos, int* __restrict__ specStatus,
    const int32_t* __restrict__ specOfElem, const int32_t* __restrict__ cpos, const int* __restrict__ specActive,
    const int32_t* __restrict__ elist, int ecount, int ncw, int mfEB) {
    using L = Hex8Lds<MAT, KT, MF, TAN>;
    constexpr int NP = (MAT == EFE_LINEAR_ELASTIC) ? 2 : 6;
    constexpr bool HAS_K = MatState<MAT>::n != 0;
    __shared__ __align__(16) char lds[L::bytes];
    const int lane = threadIdx.x, el = lane >> 3, j = lane & 7;
    const int64_t EQ = (int64_t)E * 8;
    int e = -1;  // -1 past the end and, in batched contexts, for specimens the pass skips
    {
        const int i = blockIdx.x * 8 + el;
        if (i < ecount) {
            e = elist ? elist[i] : i;
            if (specActive && !specActive[specOfElem[e]]) e = -1;
        }
    }
    const bool live = e >= 0;
    const int64_t sidx = (int64_t)(live ? e : 0) * 8 + j;
    double s[6], eps[6], ms = 0.0;
#pragma unroll
    for (int c = 0; c < 6; ++c) s[c] = eps[c] = 0.0;
    double w[6] = {0, 0, 0, 0, 0, 0};
    if (live) {
        const int nd = conn[(int64_t)((0x65217430u >> (4 * j)) & 7) * E + e];  // the node of octant bits j
#pragma unroll
        for (int c = 0; c < 6; ++c) s[c] = sRef[c * EQ + sidx];
#pragma unroll
        for (int c = 0; c < 6; ++c) eps[c] = sRef[(6 + c) * EQ + sidx];
        if (HAS_K) ms = sRef[12 * EQ + sidx];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            w[c] = coords[(int64_t)c * N + nd];
            w[3 + c] = dU[3 * (int64_t)nd + c];
        }
    }
    {
        const double s1 = (j & 1) ? -1.0 : 1.0, s2 = (j & 2) ? -1.0 : 1.0, s4 = (j & 4) ? -1.0 : 1.0;
        double* cf = (double*)lds;
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            // lanes with the bit set take own - other, the others own + other
            // (values relative to the first node, so that round-off goes with the element's own scale)
            double v = w[c] - lane_first8(w[c], (j & 4) != 0);
            v = fma(s1, lane_xor8<1>(v), v);
            v = fma(s2, lane_xor8<2>(v), v);
            v = fma(s4, lane_xor8<4>(v), v);
            cf[c * 64 + lane] = 0.125 * v;
        }
    }
    __syncthreads();
    const double g0 = 0.57735026918962576451;
    const double x = oct_x(j) ? g0 : -g0, y = oct_y(j) ? g0 : -g0, z = oct_z(j) ? g0 : -g0;
    double J[9], H[9];
    {
        const double* cf = (const double*)lds + el * 8;
        const double xy = x * y, yz = y * z, xz = x * z;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const double* cx = cf + i * 64;
            const double* cu = cf + (3 + i) * 64;
            // d/dx = c1 + c3 y + c5 z + c7 yz, d/dy = c2 + c3 x + c6 z + c7 xz, d/dz = c4 + c5 x + c6 y + c7 xy
            J[0 * 3 + i] = cx[1] + cx[3] * y + cx[5] * z + cx[7] * yz;
            J[1 * 3 + i] = cx[2] + cx[3] * x + cx[6] * z + cx[7] * xz;
            J[2 * 3 + i] = cx[4] + cx[5] * x + cx[6] * y + cx[7] * xy;
            H[i * 3 + 0] = cu[1] + cu[3] * y + cu[5] * z + cu[7] * yz;
            H[i * 3 + 1] = cu[2] + cu[3] * x + cu[6] * z + cu[7] * xz;
            H[i * 3 + 2] = cu[4] + cu[5] * x + cu[6] * y + cu[7] * xy;
        }
    }
    const double det = J[0] * (J[4] * J[8] - J[5] * J[7]) - J[1] * (J[3] * J[8] - J[5] * J[6]) +
                       J[2] * (J[3] * J[7] - J[4] * J[6]);  // the Gauss weights are 1
    const double id = live ? 1.0 / det : 0.0;
    const double iJ[9] = {(J[4] * J[8] - J[5] * J[7]) * id, (J[2] * J[7] - J[1] * J[8]) * id,
                          (J[1] * J[5] - J[2] * J[4]) * id, (J[5] * J[6] - J[3] * J[8]) * id,
                          (J[0] * J[8] - J[2] * J[6]) * id, (J[2] * J[3] - J[0] * J[5]) * id,
                          (J[3] * J[7] - J[4] * J[6]) * id, (J[1] * J[6] - J[0] * J[7]) * id,
                          (J[0] * J[4] - J[1] * J[3]) * id};
    double cc[11];
#pragma unroll
    for (int k = 0; k < 11; ++k) cc[k] = 0.0;
    if (live) {
        double gr[9];  // d u_i / d x_k
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int k = 0; k < 3; ++k)
                gr[i * 3 + k] = H[i * 3] * iJ[k * 3] + H[i * 3 + 1] * iJ[k * 3 + 1] + H[i * 3 + 2] * iJ[k * 3 + 2];
        const double de[6] = {gr[0], gr[4], gr[8], gr[1] + gr[3], gr[2] + gr[6], gr[5] + gr[7]};
        double p[NP];
#pragma unroll
        for (int k = 0; k < NP; ++k) p[k] = propStride ? props[(int64_t)k * propStride + e] : props[k];
        double C[36];
        int st = 0;
        if (MAT == EFE_LINEAR_ELASTIC) st = efe::le_update(p, s, de, C, cc);
        else if (MAT == EFE_VONMISES) st = efe::vm_update(p, s, ms, de, C, cc);
        else st = efe::dp_update(p, s, ms, de, C, cc);
        if (st) {
            *status = 1;
            if (specStatus) specStatus[specOfElem[e]] = 1;  // which specimen asked (batched contexts)
        }
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            sTmp[c * EQ + sidx] = s[c];
            sTmp[(6 + c) * EQ + sidx] = eps[c] + de[c];
        }
        if (HAS_K) sTmp[12 * EQ + sidx] = ms;
        if (TAN && mfC) store_compact(mfC, mfPos, mfEB, E, 8, e, j, ncw, det, cc);
    }
    // reference gradients of an octant pair: t*(b)[c] = (1 +- g s)(1 +- g s) / 8 of the two other axes
    double tx[2][2], ty[2][2], tz[2][2];
    {
        const double px[2] = {1.0 - x, 1.0 + x}, py[2] = {1.0 - y, 1.0 + y}, pz[2] = {1.0 - z, 1.0 + z};
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                tx[a][b] = 0.125 * py[a] * pz[b];
                ty[a][b] = 0.125 * px[a] * pz[b];
                tz[a][b] = 0.125 * px[a] * py[b];
            }
    }
    // forces
    double* Ms = (double*)lds;
    __syncthreads();  // the coefficients have been read
    {
        const double S[9] = {s[0], s[3], s[4], s[3], s[1], s[5], s[4], s[5], s[2]};
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int k = 0; k < 3; ++k)
                Ms[el * 72 + (i * 3 + k) * 8 + j] =
                    det * (S[i * 3] * iJ[k] + S[i * 3 + 1] * iJ[3 + k] + S[i * 3 + 2] * iJ[6 + k]);
    }
    __syncthreads();
    {
        const double sx = oct_x(j) ? 1.0 : -1.0, sy = oct_y(j) ? 1.0 : -1.0, sz = oct_z(j) ? 1.0 : -1.0;
        double f[3] = {0, 0, 0};
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const double* M = Ms + el * 72 + i * 24;
            double fx = 0, fy = 0, fz = 0;
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                fx += M[q] * tx[oct_y(q)][oct_z(q)];
                fy += M[8 + q] * ty[oct_x(q)][oct_z(q)];
                fz += M[16 + q] * tz[oct_x(q)][oct_y(q)];
            }
            f[i] = sx * fx + sy * fy + sz * fz;
        }
        if (live) {
            double* dst = Pscr + ((int64_t)e * 8 + j) * 3;
            dst[0] = -f[0];
            dst[1] = -f[1];
            dst[2] = -f[2];
        }
    }
    if constexpr (TAN) {
        __syncthreads();
        KT* gh = (KT*)lds;
        KT* sc = gh + 8 * L::QS;
        {
            const double nn[9] = {cc[5], cc[8], cc[9], cc[8], cc[6], cc[10], cc[9], cc[10], cc[7]};
#pragma unroll
            for (int a = 0; a < 8; ++a) {
                const double d0 = oct_x(a) ? tx[oct_y(a)][oct_z(a)] : -tx[oct_y(a)][oct_z(a)];
                const double d1 = oct_y(a) ? ty[oct_x(a)][oct_z(a)] : -ty[oct_x(a)][oct_z(a)];
                const double d2 = oct_z(a) ? tz[oct_x(a)][oct_y(a)] : -tz[oct_x(a)][oct_y(a)];
                double g[3];
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    g[c] = iJ[c * 3] * d0 + iJ[c * 3 + 1] * d1 + iJ[c * 3 + 2] * d2;
                    gh[j * L::QS + c * 64 + el * 8 + a] = (KT)g[c];
                }
                if (MAT != EFE_LINEAR_ELASTIC)
#pragma unroll
                    for (int c = 0; c < 3; ++c)
                        gh[j * L::QS + (3 + c) * 64 + el * 8 + a] =
                            (KT)(nn[c * 3] * g[0] + nn[c * 3 + 1] * g[1] + nn[c * 3 + 2] * g[2]);
            }
            KT* d = sc + (j * 8 + el) * L::NSC;
            d[0] = (KT)(det * (cc[0] - cc[1] * (1.0 / 3.0)));
            d[1] = (KT)(det * (0.5 * cc[1]));
            d[2] = (KT)(det * cc[2]);
            if (!L::SYM) {
                d[L::NSC - 2] = (KT)(det * cc[3]);
                d[L::NSC - 1] = (KT)(det * cc[4]);
            }
        }
        __syncthreads();
        constexpr int NO = MF ? 1 : (L::SYM ? 5 : 2);  // blocks per lane and pass
        constexpr int NPASS = MF || L::SYM ? 1 : 4;
#pragma unroll 1
        for (int pass = 0; pass < NPASS; ++pass) {
            KT acc[NO][9], tr[NO];
#pragma unroll
            for (int o = 0; o < NO; ++o) {
                tr[o] = (KT)0;
#pragma unroll
                for (int k = 0; k < 9; ++k) acc[o][k] = (KT)0;
            }
#pragma unroll 1
            for (int q = 0; q < 8; ++q) {
                const KT* gq = gh + q * L::QS + el * 8;
                const KT* d = sc + (q * 8 + el) * L::NSC;
                KT u[3], v[3], wv[3];
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const KT ga = gq[c * 64 + j];
                    u[c] = d[0] * ga;
                    wv[c] = d[1] * ga;
                    if (MAT != EFE_LINEAR_ELASTIC) {
                        const KT ha = gq[(3 + c) * 64 + j];
                        v[c] = d[2] * ha;
                        if (!L::SYM) {
                            u[c] += d[L::NSC - 2] * ha;
                            v[c] += d[L::NSC - 1] * ga;
                        }
                    }
                }
#pragma unroll
                for (int o = 0; o < NO; ++o) {
                    const int b = (j + o + pass * NO) & 7;
                    KT gb[3], hb[3];
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        gb[c] = gq[c * 64 + b];
                        if (MAT != EFE_LINEAR_ELASTIC) hb[c] = gq[(3 + c) * 64 + b];
                    }
                    tr[o] += wv[0] * gb[0] + wv[1] * gb[1] + wv[2] * gb[2];
#pragma unroll
                    for (int i = 0; i < 3; ++i)
#pragma unroll
                        for (int k = 0; k < 3; ++k) {
                            KT t = acc[o][i * 3 + k] + u[i] * gb[k] + wv[k] * gb[i];
                            if (MAT != EFE_LINEAR_ELASTIC) t += v[i] * hb[k];
                            acc[o][i * 3 + k] = t;
                        }
                }
            }
#pragma unroll
            for (int o = 0; o < NO; ++o)
#pragma unroll
                for (int i = 0; i < 3; ++i) acc[o][i * 4] += tr[o];
            if constexpr (MF) {  // K_aa element-major at the start of the scratch: [e][a][9]
                if (live) store_block(Kscr + ((int64_t)e * 8 + j) * kBlockPitch, acc[0]);
            } else {
                // the blocks, then their positions (and those of the transposes, -1: none), in LDS; the
                // wavefront stores them word by word, about seven 72-byte blocks per instruction
                KT* stg = (KT*)(lds + L::stageAt);
                int* pos = (int*)(stg + L::kBlocks * 9);
                const int32_t* cp = cpos + (int64_t)(live ? e : 0) * 64;
                int p0[NO], p1[NO];
#pragma unroll
                for (int o = 0; o < NO; ++o) {
                    const int b = (j + o + pass * NO) & 7;
                    const bool mine = live && (!L::SYM || o < 4 || j < 4);
                    p0[o] = mine ? cp[j * 8 + b] : -1;
                    p1[o] = L::SYM && mine && o ? cp[b * 8 + j] : -1;
                }
                __syncthreads();  // g and h have been read
#pragma unroll
                for (int o = 0; o < NO; ++o) {
                    if (L::SYM && o == 4 && j >= 4) continue;
                    // slots 0..255: the offsets 0..3; 256..287: offset 4 of the lanes j < 4
                    const int slot = o < 4 ? o * 64 + lane : 256 + el * 4 + j;
#pragma unroll
                    for (int k = 0; k < 9; ++k) stg[slot * 9 + k] = acc[o][k];
                    pos[slot] = p0[o];
                    if (L::SYM) pos[L::kBlocks + slot] = p1[o];
                }
                __syncthreads();
                for (int t = lane; t < L::kBlocks * 9; t += 64) {
                    const int bi = t / 9, v = t - bi * 9;
                    const int pb = pos[bi];
                    if (pb >= 0) Kscr[(int64_t)pb * kBlockPitch + v] = stg[t];
                    if constexpr (L::SYM) {  // K_ba = K_ab^T
                        const int pt = pos[L::kBlocks + bi];
                        const int vt = (v % 3) * 3 + v / 3;
                        if (pt >= 0) Kscr[(int64_t)pt * kBlockPitch + v] = stg[bi * 9 + vt];
                    }
                }
                if (pass + 1 < NPASS) __syncthreads();  // the staged blocks have been read
            }
        }
    }
}

__device__ __forceinline__ void inv3(const double m[9], double o[9]) {
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

template <typename KT>
__global__ __launch_bounds__(256) void assemble_kernel(
    int N, const int32_t* __restrict__ bptr, const int32_t* __restrict__ bcol, const int32_t* __restrict__ coff,
    const int32_t* __restrict__ nptr, const int32_t* __restrict__ nlist,
    const int32_t* __restrict__ slice_off, const KT* __restrict__ Kscr, const double* __restrict__ Pscr,
    const uint8_t* __restrict__ dirflag, int ndir, const double* __restrict__ dirv, double* __restrict__ dircorr,
    KT* __restrict__ Kval, KT* __restrict__ Minv, double* __restrict__ P, double* __restrict__ F,
    const int32_t* __restrict__ slotNode, const int32_t* __restrict__ cslice, const int* __restrict__ specActive,
    const int32_t* __restrict__ specOfNode) {
    // Threads walk the row slots of the sliced layout: the value stores of a wavefront are
    // contiguous, and so are its reads of the element scratch, where contribution j of the
    // 64 rows of a slice is one run of 64 blocks.
    const int per = gridDim.x >> 3;
    const int blk = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    const int ps = blk * blockDim.x + threadIdx.x;
    if (ps >= N) return;
    const int n = slotNode[ps];
    if (specActive && !specActive[specOfNode[n]]) {
        // a skipped specimen keeps its rows; its increment is not solved, so its right-hand
        // side correction is zero
        if (dirv) dircorr[3 * n] = dircorr[3 * n + 1] = dircorr[3 * n + 2] = 0.0;
        return;
    }
    const int s = ps / kSlice, l = ps - (ps / kSlice) * kSlice;
    const int64_t vbase = (int64_t)slice_off[s] * 9 + l;
    bool fr[3] = {false, false, false};
    if (ndir) {
        fr[0] = dirflag[3 * n];
        fr[1] = dirflag[3 * n + 1];
        fr[2] = dirflag[3 * n + 2];
    }
    double t0 = 0, t1 = 0, t2 = 0;
    double dg[9] = {1, 0, 0, 0, 1, 0, 0, 0, 1};
    const int b0 = bptr[n], b1 = bptr[n + 1];
    // block position of this row's contribution c: cbase + (c - coff[b0]) * kSlice
    const int64_t cbase = (int64_t)cslice[s] * kSlice + l - (int64_t)coff[b0] * kSlice;
    for (int b = b0; b < b1; ++b) {
        const int m = bcol[b];
        KT acc[9];
#pragma unroll
        for (int v = 0; v < 9; ++v) acc[v] = (KT)0;
        // the slot's contributions are contiguous and in element order; unrolled so that
        // the loads of several contributions are in flight together
#pragma unroll 4
        for (int c = coff[b]; c < coff[b + 1]; ++c) add_block(Kscr + (cbase + (int64_t)c * kSlice) * kBlockPitch, acc);
        if (dirv) {
            const double d0 = dirv[3 * m], d1 = dirv[3 * m + 1], d2 = dirv[3 * m + 2];
            t0 += (double)acc[0] * d0 + (double)acc[1] * d1 + (double)acc[2] * d2;
            t1 += (double)acc[3] * d0 + (double)acc[4] * d1 + (double)acc[5] * d2;
            t2 += (double)acc[6] * d0 + (double)acc[7] * d1 + (double)acc[8] * d2;
        }
        if (ndir) {
            const bool fc[3] = {(bool)dirflag[3 * m], (bool)dirflag[3 * m + 1], (bool)dirflag[3 * m + 2]};
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int j = 0; j < 3; ++j)
                    if (fr[i] || fc[j]) acc[i * 3 + j] = (m == n && i == j) ? (KT)1 : (KT)0;
        }
        const int k = b - b0;
#pragma unroll
        for (int v = 0; v < 9; ++v) Kval[vbase + (int64_t)(k * 9 + v) * kSlice] = acc[v];
        if (m == n) {
#pragma unroll
            for (int v = 0; v < 9; ++v) dg[v] = (double)acc[v];
        }
    }
    double iv[9];
    inv3(dg, iv);
#pragma unroll
    for (int v = 0; v < 9; ++v) Minv[(int64_t)n * 9 + v] = (KT)iv[v];
    if (P) {
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
    if (dirv) {
        dircorr[3 * n] = fr[0] ? 0.0 : t0;
        dircorr[3 * n + 1] = fr[1] ? 0.0 : t1;
        dircorr[3 * n + 2] = fr[2] ? 0.0 : t2;
    }
}

// assemble_kernel with the element scratch read run by run and the row's blocks shared out over W
// wavefronts: a workgroup takes one slice, wavefront w the w-th part of every row's blocks.  It loads
// each contribution run of its part (the j-th contributions of the 64 rows, 64 contiguous blocks)
// with nine coalesced 512-byte loads (FP64), stages it in LDS and each lane takes its own block
// from there, loading the next run meanwhile.  A block is summed by one lane in the order of
// assemble_kernel, so K and Minv are bitwise the same for every W; P and F are summed by the last
// wavefront, the correction from the W parts in order.  The one block of a node outside every element
// has no contributions (every other block of the pattern has): its K stays zero and its Minv is the
// identity.
template <typename KT, int W>
__global__ __launch_bounds__(64 * W) void assemble_runs_kernel(
    int N, const int32_t* __restrict__ bptr, const int32_t* __restrict__ bcol, const int32_t* __restrict__ coff,
    const int32_t* __restrict__ nptr, const int32_t* __restrict__ nlist,
    const int32_t* __restrict__ slice_off, const KT* __restrict__ Kscr, const double* __restrict__ Pscr,
    const uint8_t* __restrict__ dirflag, int ndir, const double* __restrict__ dirv, double* __restrict__ dircorr,
    KT* __restrict__ Kval, KT* __restrict__ Minv, double* __restrict__ P, double* __restrict__ F,
    const int32_t* __restrict__ slotNode, const int32_t* __restrict__ cslice, const int* __restrict__ specActive,
    const int32_t* __restrict__ specOfNode) {
    constexpr int RUN = 9 * kSlice;  // values of one contribution run
    __shared__ KT runbuf[W][RUN];
    const int per = gridDim.x >> 3;
    const int s = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (s * kSlice >= N) return;  // the whole workgroup
    const int l = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int ps = s * kSlice + l;
    KT* buf = runbuf[wv];
    const bool valid = ps < N;
    const int n = valid ? slotNode[ps] : 0;
    const bool work = valid && !(specActive && !specActive[specOfNode[n]]);
    bool fr[3] = {false, false, false};
    if (work && ndir) {
        fr[0] = dirflag[3 * n];
        fr[1] = dirflag[3 * n + 1];
        fr[2] = dirflag[3 * n + 2];
    }
    double t0 = 0, t1 = 0, t2 = 0;
    double dg[9] = {1, 0, 0, 0, 1, 0, 0, 0, 1};
    bool haveDiag = false;
    const int64_t vbase = (int64_t)slice_off[s] * 9 + l;
    int b0 = 0, b = 0, b1 = 0, c0 = 0, c1 = 0, cend = 0;  // this part's blocks [b, b1), contributions [c0, c1)
    if (work) {
        b0 = bptr[n];
        const int deg = bptr[n + 1] - b0;
        b = b0 + deg * wv / W;
        b1 = b0 + deg * (wv + 1) / W;
        const int first = coff[b0];
        c0 = coff[b] - first;
        c1 = coff[b1] - first;
        if (b < b1) cend = coff[b + 1] - first;
        haveDiag = b < b1 && c0 == c1;  // a block without contributions: dg as it is
    }
    KT acc[9];
#pragma unroll
    for (int v = 0; v < 9; ++v) acc[v] = (KT)0;
    // the runs of this part over the 64 rows (rows of one kind, the same for all)
    int jlo = c0 < c1 ? c0 : 0x7fffffff, jhi = c1;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        jlo = min(jlo, __shfl_xor(jlo, o, 64));
        jhi = max(jhi, __shfl_xor(jhi, o, 64));
    }
    jlo = __builtin_amdgcn_readfirstlane(jlo);
    jhi = __builtin_amdgcn_readfirstlane(jhi);
    if (jlo < jhi) {
        const KT* runs = Kscr + (int64_t)cslice[s] * RUN;
        KT nxt[9];
#pragma unroll
        for (int t = 0; t < 9; ++t) nxt[t] = __builtin_nontemporal_load(runs + (int64_t)jlo * RUN + t * kSlice + l);
        for (int j = jlo; j < jhi; ++j) {
#pragma unroll
            for (int t = 0; t < 9; ++t) buf[t * kSlice + l] = nxt[t];
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            if (j + 1 < jhi) {
                const KT* nr = runs + (int64_t)(j + 1) * RUN;
#pragma unroll
                for (int t = 0; t < 9; ++t) nxt[t] = __builtin_nontemporal_load(nr + t * kSlice + l);
            }
            if (j >= c0 && j < c1) {
#pragma unroll
                for (int v = 0; v < 9; ++v) acc[v] += buf[l * 9 + v];
                if (j + 1 == cend) {  // the last contribution of block b: finish it
                    const int m = bcol[b];
                    if (dirv) {
                        const double d0 = dirv[3 * m], d1 = dirv[3 * m + 1], d2 = dirv[3 * m + 2];
                        t0 += (double)acc[0] * d0 + (double)acc[1] * d1 + (double)acc[2] * d2;
                        t1 += (double)acc[3] * d0 + (double)acc[4] * d1 + (double)acc[5] * d2;
                        t2 += (double)acc[6] * d0 + (double)acc[7] * d1 + (double)acc[8] * d2;
                    }
                    if (ndir) {
                        const bool fc[3] = {(bool)dirflag[3 * m], (bool)dirflag[3 * m + 1], (bool)dirflag[3 * m + 2]};
#pragma unroll
                        for (int i = 0; i < 3; ++i)
#pragma unroll
                            for (int jj = 0; jj < 3; ++jj)
                                if (fr[i] || fc[jj]) acc[i * 3 + jj] = (m == n && i == jj) ? (KT)1 : (KT)0;
                    }
                    const int k = b - b0;
#pragma unroll
                    for (int v = 0; v < 9; ++v) Kval[vbase + (int64_t)(k * 9 + v) * kSlice] = acc[v];
                    if (m == n) {
                        haveDiag = true;
#pragma unroll
                        for (int v = 0; v < 9; ++v) dg[v] = (double)acc[v];
                    }
#pragma unroll
                    for (int v = 0; v < 9; ++v) acc[v] = (KT)0;
                    ++b;
                    if (b < b1) cend = coff[b + 1] - coff[b0];
                }
            }
            // every lane has read its block before the next run overwrites the buffer
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
    }
    if (work && haveDiag) {
        double iv[9];
        inv3(dg, iv);
#pragma unroll
        for (int v = 0; v < 9; ++v) Minv[(int64_t)n * 9 + v] = (KT)iv[v];
    }
    if (work && P && wv == W - 1) {
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
    if (dirv) {
        double(*sum)[3][64] = (double(*)[3][64])runbuf;  // [W][3][64], within the run buffers
        static_assert(sizeof(runbuf) >= (size_t)W * 3 * 64 * sizeof(double), "the parts' sums fit");
        __syncthreads();
        sum[wv][0][l] = t0;
        sum[wv][1][l] = t1;
        sum[wv][2][l] = t2;
        __syncthreads();
        if (wv == 0 && valid) {
            // a skipped specimen's increment is not solved: its correction is zero
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                double t = 0;
                for (int k = 0; k < W; ++k) t += sum[k][i][l];
                dircorr[3 * n + i] = !work || fr[i] ? 0.0 : t;
            }
        }
    }
}

// Body force (element.py:348-371): Pe = sum_q N_q (x) f detJ_q w_q with N at the table
// point and detJ of the element's J at the evaluation point (dJdxi); written to the
// element scratch, then gathered.
// One thread per listed element (elems[k], or element k when elems is NULL).
template <int NN, int Q>
__global__ __launch_bounds__(64) void body_force_kernel(int n, int E, int N, const int32_t* __restrict__ elems,
                                                        const double* __restrict__ coords,
                                                        const int32_t* __restrict__ conn,
                                                        const double* __restrict__ dNdxi,
                                                        const double* __restrict__ shapeN,
                                                        const double* __restrict__ qpw, double fx, double fy,
                                                        double fz, double* __restrict__ Pscr) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const int e = elems ? elems[k] : k;
    double acc[NN];
#pragma unroll
    for (int a = 0; a < NN; ++a) acc[a] = 0.0;
    for (int q = 0; q < Q; ++q) {
        const double* dn = dNdxi + (size_t)q * NN * 3;
        double J[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
        for (int a = 0; a < NN; ++a) {
            const int nd = conn[(int64_t)a * E + e];
            const double x = coords[nd], y = coords[N + nd], z = coords[2 * N + nd];
#pragma unroll
            for (int r = 0; r < 3; ++r) {
                J[r * 3 + 0] += dn[a * 3 + r] * x;
                J[r * 3 + 1] += dn[a * 3 + r] * y;
                J[r * 3 + 2] += dn[a * 3 + r] * z;
            }
        }
        const double det = J[0] * (J[4] * J[8] - J[5] * J[7]) - J[1] * (J[3] * J[8] - J[5] * J[6]) +
                           J[2] * (J[3] * J[7] - J[4] * J[6]);
#pragma unroll
        for (int a = 0; a < NN; ++a) acc[a] += shapeN[q * NN + a] * det * qpw[q];
    }
#pragma unroll
    for (int a = 0; a < NN; ++a) {
        double* dst = Pscr + ((int64_t)e * NN + a) * 3;
        dst[0] = acc[a] * fx;
        dst[1] = acc[a] * fy;
        dst[2] = acc[a] * fz;
    }
}

// Surface traction (the distributed load of nonlinearimplicitstatic.py:460-508 with type
// "surface traction"): the consistent nodal force f_a = t * integral N_a dA of a uniform
// traction t on element faces.  Faces are numbered by local node numbers as in Abaqus
// (1: 1-2-3-4, 2: 5-8-7-6, 3: 1-5-6-2, 4: 2-6-7-3, 5: 3-7-8-4, 6: 4-8-5-1; hexa20 adds the
// mid-side nodes between consecutive corners), the numbering of the box generator's
// surfaces (boxgen.py:438-446).  2x2 Gauss points on 4-node faces, 3x3 on 8-node
// (serendipity) faces.  One thread per loaded element: its faces (bit f-1 of fmask) are
// summed in face order into the element's force slots.
__constant__ int8_t kFace8[6][4] = {{0, 1, 2, 3}, {4, 7, 6, 5}, {0, 4, 5, 1},
                                    {1, 5, 6, 2}, {2, 6, 7, 3}, {3, 7, 4, 0}};
__constant__ int8_t kFace20[6][8] = {{0, 1, 2, 3, 8, 9, 10, 11},   {4, 7, 6, 5, 15, 14, 13, 12},
                                     {0, 4, 5, 1, 16, 12, 17, 8},  {1, 5, 6, 2, 17, 13, 18, 9},
                                     {2, 6, 7, 3, 18, 14, 19, 10}, {3, 7, 4, 0, 19, 15, 16, 11}};

// N, dN/ds, dN/dt of the NF-node face (4: bilinear; 8: serendipity) at (s, t); node order:
// corners (-1,-1), (1,-1), (1,1), (-1,1), then mid-sides (0,-1), (1,0), (0,1), (-1,0)
template <int NF>
__device__ __forceinline__ void face_shape(double s, double t, double* N, double* Ns, double* Nt) {
    const double cs[4] = {-1, 1, 1, -1}, ct[4] = {-1, -1, 1, 1};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const double a = 1 + s * cs[i], b = 1 + t * ct[i];
        if (NF == 4) {
            N[i] = a * b / 4;
            Ns[i] = cs[i] * b / 4;
            Nt[i] = ct[i] * a / 4;
        } else {
            N[i] = a * b * (s * cs[i] + t * ct[i] - 1) / 4;
            Ns[i] = cs[i] * b * (2 * s * cs[i] + t * ct[i]) / 4;
            Nt[i] = ct[i] * a * (s * cs[i] + 2 * t * ct[i]) / 4;
        }
    }
    if (NF == 8) {
        N[4] = (1 - s * s) * (1 - t) / 2;
        Ns[4] = -s * (1 - t);
        Nt[4] = -(1 - s * s) / 2;
        N[5] = (1 + s) * (1 - t * t) / 2;
        Ns[5] = (1 - t * t) / 2;
        Nt[5] = -t * (1 + s);
        N[6] = (1 - s * s) * (1 + t) / 2;
        Ns[6] = -s * (1 + t);
        Nt[6] = (1 - s * s) / 2;
        N[7] = (1 - s) * (1 - t * t) / 2;
        Ns[7] = -(1 - t * t) / 2;
        Nt[7] = -t * (1 - s);
    }
}

template <int NN>
__global__ __launch_bounds__(256) void surface_traction_kernel(int n, int E, int N, const int32_t* __restrict__ elems,
                                                               const uint8_t* __restrict__ fmask,
                                                               const double* __restrict__ coords,
                                                               const int32_t* __restrict__ conn, double tx, double ty,
                                                               double tz, double* __restrict__ Pscr) {
    constexpr int NF = NN == 8 ? 4 : 8, NG = NN == 8 ? 2 : 3;
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const int e = elems[k], mask = fmask[k];
    const double gp2[2] = {-0.57735026918962576451, 0.57735026918962576451}, gw2[2] = {1.0, 1.0};
    const double gp3[3] = {-0.77459666924148337704, 0.0, 0.77459666924148337704};
    const double gw3[3] = {5.0 / 9.0, 8.0 / 9.0, 5.0 / 9.0};
    double acc[NN];
#pragma unroll
    for (int a = 0; a < NN; ++a) acc[a] = 0.0;
    for (int f = 0; f < 6; ++f) {
        if (!((mask >> f) & 1)) continue;
        int loc[NF];
        double X[NF][3];
#pragma unroll
        for (int j = 0; j < NF; ++j) {
            loc[j] = NN == 8 ? kFace8[f][j] : kFace20[f][j];
            const int nd = conn[(int64_t)loc[j] * E + e];
            X[j][0] = coords[nd];
            X[j][1] = coords[N + nd];
            X[j][2] = coords[2 * N + nd];
        }
        for (int i = 0; i < NG; ++i)
            for (int j2 = 0; j2 < NG; ++j2) {
                const double s = NG == 2 ? gp2[i] : gp3[i], t = NG == 2 ? gp2[j2] : gp3[j2];
                const double w = NG == 2 ? gw2[i] * gw2[j2] : gw3[i] * gw3[j2];
                double Nf[NF], Ns[NF], Nt[NF];
                face_shape<NF>(s, t, Nf, Ns, Nt);
                double xs[3] = {0, 0, 0}, xt[3] = {0, 0, 0};
#pragma unroll
                for (int j = 0; j < NF; ++j)
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        xs[c] += Ns[j] * X[j][c];
                        xt[c] += Nt[j] * X[j][c];
                    }
                const double cx = xs[1] * xt[2] - xs[2] * xt[1], cy = xs[2] * xt[0] - xs[0] * xt[2],
                             cz = xs[0] * xt[1] - xs[1] * xt[0];
                const double dA = sqrt(cx * cx + cy * cy + cz * cz) * w;
#pragma unroll
                for (int j = 0; j < NF; ++j) acc[loc[j]] += Nf[j] * dA;
            }
    }
#pragma unroll
    for (int a = 0; a < NN; ++a) {
        double* dst = Pscr + ((int64_t)e * NN + a) * 3;
        dst[0] = acc[a] * tx;
        dst[1] = acc[a] * ty;
        dst[2] = acc[a] * tz;
    }
}

// P and F of a residual-only pass: the element residuals of every node summed in element
// order, as the assembly's gather sums them.  Nodes of specimens the pass skips (batched
// contexts) keep P and F, as in the assembly.
__global__ void pf_gather_kernel(int N, const int32_t* __restrict__ nptr, const int32_t* __restrict__ nlist,
                                 const double* __restrict__ Pscr, double* __restrict__ P, double* __restrict__ F,
                                 const int* __restrict__ specActive, const int32_t* __restrict__ specOfNode) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= N) return;
    if (specActive && !specActive[specOfNode[n]]) return;
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

__global__ void gather_add_kernel(int N, const int32_t* __restrict__ nptr, const int32_t* __restrict__ nlist,
                                  const double* __restrict__ Pscr, double* __restrict__ out) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= N) return;
    double p0 = 0, p1 = 0, p2 = 0;
    for (int c = nptr[n]; c < nptr[n + 1]; ++c) {
        const double* src = Pscr + (int64_t)nlist[c] * 3;
        p0 += src[0];
        p1 += src[1];
        p2 += src[2];
    }
    out[3 * n] += p0;
    out[3 * n + 1] += p1;
    out[3 * n + 2] += p2;
}

template <typename KT>
__global__ void export_csr_kernel(int N, const int32_t* __restrict__ bptr, const int32_t* __restrict__ slice_off,
                                  const int32_t* __restrict__ nodeSlot, const KT* __restrict__ Kval,
                                  double* __restrict__ out) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= N) return;
    const int ps = nodeSlot[n];
    const int s = ps / kSlice, l = ps - (ps / kSlice) * kSlice;
    const int64_t vbase = (int64_t)slice_off[s] * 9 + l;
    const int deg = bptr[n + 1] - bptr[n];
    const int64_t r0 = (int64_t)9 * bptr[n];
    for (int k = 0; k < deg; ++k)
        for (int i = 0; i < 3; ++i)
            for (int j = 0; j < 3; ++j)
                out[r0 + (int64_t)3 * i * deg + 3 * k + j] = (double)Kval[vbase + (int64_t)(k * 9 + i * 3 + j) * kSlice];
}

template <int NN, int Q, int MAT, typename KT, int EPW>
void launch_elem_t(efe_ctx* c, const double* dU) {
    static const int cap = std::getenv("EFE_ELEMENT_GRID_CAP") ? std::atoi(std::getenv("EFE_ELEMENT_GRID_CAP")) : 0;
    int grid = (c->curCount + EPW - 1) / EPW;
    if (grid == 0) return;
    if (cap > 0 && grid > cap) grid = cap;  // persistent: the workgroups loop over the list
    const int propStride = c->props_per_element ? c->E : 0;
    const int* act = c->useActive ? c->specActive : nullptr;
    auto launch = [&](auto kern, int threads, auto* K, float* mfC, int reserve = 0) {
        kern<<<grid, threads, reserve, c->stream>>>(c->E, c->N, c->coords, c->conn, c->props, propStride, c->dNdxi, c->dJdxi,
                                              c->qpw, dU, c->stateRef, c->stateTmp, K, c->Pscr, c->status, mfC,
                                              c->specStatus, c->specOfElem, c->cpos, act, c->formK, c->curList,
                                              c->curCount, c->mfNC);
    };
    // Two wavefronts per workgroup where 27 QPs' blocks are formed: the LDS of 27 QPs leaves eight
    // workgroups per CU, too few wavefronts to hide the LDS reads of the blocks (17x15x13 hexa20 J2:
    // 139 -> 122 us in FP64, 118 -> 107 us in FP32; 27 elements: 49 -> 31 us; 32^3: 1074 -> 1026 us).
    // With 8 QPs a second wavefront only took registers and stage space (32^3 hexa20R DP: 698 ->
    // 722 us), and passes without blocks leave it idle (residual of 17x15x13: 37 -> 42 us).
    // Up to three workgroups per CU the chip has wavefronts to spare, and four share an element's
    // blocks: 8^3 hexa20 J2 45 -> 33 us, 9^3 (729 workgroups) 46 -> 38 us, but 10^3 (1000) 47 -> 52;
    // hexa20R DP 9^3 67 -> 36 us, 11^3 (666) 68 -> 41, 12^3 (864) 70 -> 59, 16^3 (2048) 100 -> 105.
    constexpr int kSmallGrid = 3 * 256;
    constexpr int W = Q > 8 ? 2 : 1;
    // Large FP64 passes of hexa20R store 400 scattered 72-byte blocks per element from 12 workgroups per CU,
    // more than the memory merges: 48^3 Drucker-Prager 2110 us while the gradients were formed by the QP
    // lanes alone, 2530 with them over all lanes, which leaves the stores a larger part of each workgroup's
    // time.  LDS that nobody uses keeps it to 11: 40^3 1289 -> 1280 us, 44^3 1715 -> 1670, 48^3 2530 -> 2157,
    // 56^3 4322 -> 3438 (J2 48^3 2693 -> 2667, linear elastic 2713 -> 2673).  36^3 (23328 workgroups) takes
    // 953 us either way, 32^3 683 with 12 and 701 with 11; in FP32, whose blocks are half as large, 48^3
    // takes 1597 with 12 and 1694 with 11.
    constexpr int kReserve = Q == 8 && EPW == 2 && sizeof(KT) == 8 ? 2400 : 0, kLargeGrid = 25000;
    if (c->mfPass)
        launch(element_kernel<NN, Q, MAT, float, EPW, true, 1>, 64, (float*)c->Kscr, c->mfC);
    else if (c->formK && grid <= kSmallGrid)
        launch(element_kernel<NN, Q, MAT, KT, EPW, false, 4>, 256, (KT*)c->Kscr, (float*)nullptr);
    else if (c->formK)
        launch(element_kernel<NN, Q, MAT, KT, EPW, false, W>, 64 * W, (KT*)c->Kscr, (float*)nullptr,
               grid > kLargeGrid ? kReserve : 0);
    else
        launch(element_kernel<NN, Q, MAT, KT, EPW, false, 1>, 64, (KT*)c->Kscr, (float*)nullptr);
}

template <int NN, int Q, int MAT, typename KT>
int launch_elem_epw(efe_ctx* c, const double* dU) {
    // default: hexa20R 2, hexa20 1
    int epw = c->epw;
    if (epw <= 0) epw = Q == 8 ? 2 : 1;
    switch (epw) {
        case 1: launch_elem_t<NN, Q, MAT, KT, 1>(c, dU); break;
        case 2: launch_elem_t<NN, Q, MAT, KT, 2>(c, dU); break;
        default:
            efe_set_error("elements per workgroup must be 1, 2, 4 or 8 (hexa20: 1 or 2)");
            return EFE_ERR_ARG;
    }
    return EFE_OK;
}

// hexa8: 8 elements per wavefront whatever is set (of the choices there are)
template <int MAT, typename KT>
int launch_hex8(efe_ctx* c, const double* dU) {
    if (c->epw > 0 && c->epw != 1 && c->epw != 2 && c->epw != 4 && c->epw != 8) {
        efe_set_error("elements per workgroup must be 1, 2, 4 or 8 (hexa20: 1 or 2)");
        return EFE_ERR_ARG;
    }
    const int grid = (c->curCount + 7) / 8;
    if (grid == 0) return EFE_OK;
    const int propStride = c->props_per_element ? c->E : 0;
    const int* act = c->useActive ? c->specActive : nullptr;
#define HEX8_ARGS(T, C)                                                                                            \
    c->E, c->N, c->coords, c->conn, c->props, propStride, dU, c->stateRef, c->stateTmp, (T*)c->Kscr, c->Pscr,         \
        c->status, C, c->mfbPos, c->specStatus, c->specOfElem, c->cpos, act, c->curList, c->curCount, c->mfNC, c->mfbE
    if (!c->formK)
        hex8_kernel<MAT, double, false, false><<<grid, 64, 0, c->stream>>>(HEX8_ARGS(double, (double*)nullptr));
    else if (c->mfPass)
        hex8_kernel<MAT, float, true, true><<<grid, 64, 0, c->stream>>>(HEX8_ARGS(float, c->mfC));
    else if constexpr (sizeof(KT) == 8)
        hex8_kernel<MAT, double, false, true><<<grid, 64, 0, c->stream>>>(HEX8_ARGS(double, c->mfC64));
    else
        hex8_kernel<MAT, float, false, true><<<grid, 64, 0, c->stream>>>(HEX8_ARGS(float, (float*)nullptr));
#undef HEX8_ARGS
    return EFE_OK;
}

template <int NN, int Q, typename KT>
int launch_elem_mat(efe_ctx* c, const double* dU) {
    switch (c->curMat) {
        case EFE_LINEAR_ELASTIC: return launch_elem_epw<NN, Q, EFE_LINEAR_ELASTIC, KT>(c, dU);
        case EFE_VONMISES: return launch_elem_epw<NN, Q, EFE_VONMISES, KT>(c, dU);
        case EFE_DRUCKER_PRAGER: return launch_elem_epw<NN, Q, EFE_DRUCKER_PRAGER, KT>(c, dU);
    }
    efe_set_error("unknown material");
    return EFE_ERR_ARG;
}

template <typename KT>
int launch_elem_type(efe_ctx* c, const double* dU) {
    switch (c->eltype) {
        case EFE_C3D8:
            switch (c->curMat) {
                case EFE_LINEAR_ELASTIC: return launch_hex8<EFE_LINEAR_ELASTIC, KT>(c, dU);
                case EFE_VONMISES: return launch_hex8<EFE_VONMISES, KT>(c, dU);
                case EFE_DRUCKER_PRAGER: return launch_hex8<EFE_DRUCKER_PRAGER, KT>(c, dU);
            }
            efe_set_error("unknown material");
            return EFE_ERR_ARG;
        case EFE_C3D20: return launch_elem_mat<20, 27, KT>(c, dU);
        case EFE_C3D20R: return launch_elem_mat<20, 8, KT>(c, dU);
    }
    efe_set_error("unknown element type");
    return EFE_ERR_ARG;
}

}  // namespace

int efe_launch_elements(efe_ctx* c, const double* dU, int precision) {
    c->mfPass = precision == EFE_FP32_MATFREE;
    for (int g = 0; g < c->ngroups; ++g) {  // one launch per material group (section)
        c->curMat = c->groupMat[g];
        c->curList = c->groupElems[g];
        c->curCount = c->groupCount[g];
        int rc = (precision == EFE_FP64) ? launch_elem_type<double>(c, dU) : launch_elem_type<float>(c, dU);
        if (rc != EFE_OK) return rc;
        EFE_HIP(hipGetLastError());
    }
    return EFE_OK;
}

int efe_launch_residual(efe_ctx* c, const double* dU, double* P, double* F, int precision) {
    c->formK = 0;
    const int rc = efe_launch_elements(c, dU, precision);  // the precision's launch shape; same residual
    c->formK = 1;
    if (rc != EFE_OK) return rc;
    pf_gather_kernel<<<(c->N + 255) / 256, 256, 0, c->stream>>>(c->N, c->nptr, c->nlist, c->Pscr, P, F,
                                                                 c->useActive ? c->specActive : nullptr,
                                                                 c->specOfNode);
    EFE_HIP(hipGetLastError());
    return EFE_OK;
}

int efe_launch_assembly(efe_ctx* c, double* P, double* F, const double* dir_values, double* dir_correction,
                        int precision) {
    const int bs = 256, grid = (((c->N + bs - 1) / bs) + 7) & ~7;  // a multiple of 8 (XCD mapping)
    static const bool perLane = std::getenv("EFE_ASSEMBLY_PER_LANE") != nullptr;  // the per-lane form, for comparison
    if (!perLane) {
#define ASM_ARGS(KT, K, M)                                                                                           \
    c->N, c->bptr, c->bcol, c->coff, c->nptr, c->nlist, c->slice_off, (const KT*)c->Kscr, c->Pscr, c->dirflag,       \
        c->ndir, dir_values, dir_correction, K, M, P, F, c->slotNode, c->cslice, c->useActive ? c->specActive : nullptr, \
        c->specOfNode
#define ASM_LAUNCH(W)                                                                                                  \
    do {                                                                                                               \
        if (precision == EFE_FP32)                                                                                     \
            assemble_runs_kernel<float, W><<<gs, 64 * W, 0, c->stream>>>(ASM_ARGS(float, c->K32, c->Minv32));          \
        else                                                                                                           \
            assemble_runs_kernel<double, W><<<gs, 64 * W, 0, c->stream>>>(ASM_ARGS(double, c->K64, c->Minv64));        \
    } while (0)
        const int gs = (c->nslices + 7) & ~7;
        // a row's contributions are one dependent walk (80 to 160 runs in hexa20): 8 wavefronts per
        // slice take it in parts, 4 where the slices alone fill the chip and the values are FP64.
        // At 1 / 4 / 8 / 16 wavefronts: 525 nodes 55 / 36 / 31 / 37 us, hexa20 17 x 15 x 13 148 / 103 /
        // 100 / 121 us, 64^3 hexa8 477 / 468 / 473 / 494 us, FP32 373 / 287 / 275 / 301 us (one wavefront
        // per slice and four slices per workgroup before: 67, 186, 520 and 390 us).
        if (precision == EFE_FP64 && c->nslices >= 1536) ASM_LAUNCH(4);
        else ASM_LAUNCH(8);
#undef ASM_LAUNCH
#undef ASM_ARGS
        EFE_HIP(hipGetLastError());
        c->Kprec = precision;
        c->Kversion++;
        return EFE_OK;
    }
    if (precision == EFE_FP32) {
        assemble_kernel<float><<<grid, bs, 0, c->stream>>>(
            c->N, c->bptr, c->bcol, c->coff, c->nptr, c->nlist, c->slice_off, (const float*)c->Kscr,
            c->Pscr, c->dirflag, c->ndir, dir_values, dir_correction, c->K32, c->Minv32, P, F, c->slotNode, c->cslice,
            c->useActive ? c->specActive : nullptr, c->specOfNode);
    } else {
        assemble_kernel<double><<<grid, bs, 0, c->stream>>>(
            c->N, c->bptr, c->bcol, c->coff, c->nptr, c->nlist, c->slice_off, (const double*)c->Kscr,
            c->Pscr, c->dirflag, c->ndir, dir_values, dir_correction, c->K64, c->Minv64, P, F, c->slotNode, c->cslice,
            c->useActive ? c->specActive : nullptr, c->specOfNode);
    }
    EFE_HIP(hipGetLastError());
    c->Kprec = precision;
    c->Kversion++;
    return EFE_OK;
}

int efe_launch_body_force(efe_ctx* c, const int32_t* elems, int n, const double* f3, double* PExt) {
    // a subset leaves the other elements' slots at zero
    if (elems) EFE_HIP(hipMemsetAsync(c->Pscr, 0, (size_t)c->E * c->NN * 3 * sizeof(double), c->stream));
    c->pscrValid = false;
    const int grid = (n + 63) / 64;
    if (n > 0) switch (c->eltype) {
        case EFE_C3D8:
            body_force_kernel<8, 8><<<grid, 64, 0, c->stream>>>(n, c->E, c->N, elems, c->coords, c->conn, c->dJdxi,
                                                               c->shapeN, c->qpw, f3[0], f3[1], f3[2], c->Pscr);
            break;
        case EFE_C3D20:
            body_force_kernel<20, 27><<<grid, 64, 0, c->stream>>>(n, c->E, c->N, elems, c->coords, c->conn, c->dJdxi,
                                                                 c->shapeN, c->qpw, f3[0], f3[1], f3[2], c->Pscr);
            break;
        case EFE_C3D20R:
            body_force_kernel<20, 8><<<grid, 64, 0, c->stream>>>(n, c->E, c->N, elems, c->coords, c->conn, c->dJdxi,
                                                                c->shapeN, c->qpw, f3[0], f3[1], f3[2], c->Pscr);
            break;
        default:
            efe_set_error("unknown element type");
            return EFE_ERR_ARG;
    }
    gather_add_kernel<<<(c->N + 255) / 256, 256, 0, c->stream>>>(c->N, c->nptr, c->nlist, c->Pscr, PExt);
    EFE_HIP(hipGetLastError());
    return EFE_OK;
}

int efe_launch_surface_traction(efe_ctx* c, const int32_t* elems, const uint8_t* fmask, int n, const double* t3,
                                double* PExt) {
    EFE_HIP(hipMemsetAsync(c->Pscr, 0, (size_t)c->E * c->NN * 3 * sizeof(double), c->stream));
    c->pscrValid = false;
    const int grid = (n + 255) / 256;
    if (n > 0) {
        if (c->NN == 8)
            surface_traction_kernel<8><<<grid, 256, 0, c->stream>>>(n, c->E, c->N, elems, fmask, c->coords, c->conn,
                                                                    t3[0], t3[1], t3[2], c->Pscr);
        else
            surface_traction_kernel<20><<<grid, 256, 0, c->stream>>>(n, c->E, c->N, elems, fmask, c->coords, c->conn,
                                                                     t3[0], t3[1], t3[2], c->Pscr);
    }
    gather_add_kernel<<<(c->N + 255) / 256, 256, 0, c->stream>>>(c->N, c->nptr, c->nlist, c->Pscr, PExt);
    EFE_HIP(hipGetLastError());
    return EFE_OK;
}

// Geostatic initial stress at every QP of the listed elements (all when elems is NULL):
// sigma_yy = p1 + (p2 - p1) (y - h1) / (h2 - h1) at the QP's y coordinate, sigma_xx =
// xLateral sigma_yy, sigma_zz = zLateral sigma_yy; shear stresses and all other state stay.
template <int NN>
__global__ __launch_bounds__(256) void geostatic_kernel(int E, int Q, int n, int N, const int32_t* __restrict__ elems,
                                                        const double* __restrict__ coords,
                                                        const int32_t* __restrict__ conn,
                                                        const double* __restrict__ shapeNe, double p1, double h1,
                                                        double p2, double h2, double xl, double zl,
                                                        double* __restrict__ stateRef) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)n * Q) return;
    const int k = (int)(i / Q), q = (int)(i - (int64_t)k * Q);
    const int e = elems ? elems[k] : k;
    double y = 0.0;
#pragma unroll
    for (int a = 0; a < NN; ++a) y += shapeNe[q * NN + a] * coords[N + conn[(int64_t)a * E + e]];
    const double sy = p1 + (p2 - p1) * (y - h1) / (h2 - h1);
    const int64_t EQ = (int64_t)E * Q, idx = (int64_t)e * Q + q;
    stateRef[idx] = xl * sy;
    stateRef[EQ + idx] = sy;
    stateRef[2 * EQ + idx] = zl * sy;
}

int efe_launch_geostatic(efe_ctx* c, const double* def, const int32_t* elements, int32_t n) {
    const int32_t* de = nullptr;
    if (elements) {
        if (!c->geoElems) EFE_HIP(hipMalloc(&c->geoElems, (size_t)c->E * sizeof(int32_t)));
        EFE_HIP(hipMemcpyAsync(c->geoElems, elements, (size_t)n * sizeof(int32_t), hipMemcpyHostToDevice,
                               c->stream));
        de = c->geoElems;
    }
    if (n == 0) return EFE_OK;
    const int64_t work = (int64_t)n * c->Q;
    const unsigned grid = (unsigned)((work + 255) / 256);
    if (c->NN == 8)
        geostatic_kernel<8><<<grid, 256, 0, c->stream>>>(c->E, c->Q, n, c->N, de, c->coords, c->conn, c->shapeNe,
                                                          def[0], def[1], def[2], def[3], def[4], def[5],
                                                          c->stateRef);
    else
        geostatic_kernel<20><<<grid, 256, 0, c->stream>>>(c->E, c->Q, n, c->N, de, c->coords, c->conn, c->shapeNe,
                                                           def[0], def[1], def[2], def[3], def[4], def[5],
                                                           c->stateRef);
    EFE_HIP(hipGetLastError());
    return EFE_OK;
}

// Element matrices in the layout of the native element ABI (MarmotElement::computeYourself,
// marmotelement/element.pxd:97-103: Ke column-major nDof x nDof, Pe nDof, DOFs node-major):
// thread per (listed element, block a b); the block is read from its contribution position.
template <typename KT>
__global__ void export_element_kernel(int n, int NN, const int32_t* __restrict__ elems,
                                      const int32_t* __restrict__ cpos, const KT* __restrict__ Kscr,
                                      const double* __restrict__ Pscr, double* __restrict__ Ke,
                                      double* __restrict__ Pe) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t nb = (int64_t)NN * NN;
    if (t >= (int64_t)n * nb) return;
    const int k = (int)(t / nb), ab = (int)(t - (int64_t)k * nb);
    const int a = ab / NN, b = ab - (ab / NN) * NN;
    const int e = elems[k];
    const int nd = 3 * NN;
    const KT* src = Kscr + (int64_t)cpos[(int64_t)e * nb + ab] * kBlockPitch;
    double* dst = Ke + (int64_t)k * nd * nd;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) dst[(int64_t)(3 * b + j) * nd + 3 * a + i] = (double)src[i * 3 + j];
    if (Pe && b == 0) {
#pragma unroll
        for (int i = 0; i < 3; ++i) Pe[(int64_t)k * nd + 3 * a + i] = Pscr[((int64_t)e * NN + a) * 3 + i];
    }
}

int efe_launch_export_elements(efe_ctx* c, const int32_t* elems, int n, double* Ke, double* Pe) {
    const int64_t total = (int64_t)n * c->NN * c->NN;
    const unsigned grid = (unsigned)((total + 255) / 256);
    if (c->Kprec == EFE_FP32)
        export_element_kernel<float><<<grid, 256, 0, c->stream>>>(n, c->NN, elems, c->cpos, (const float*)c->Kscr,
                                                                   c->Pscr, Ke, Pe);
    else
        export_element_kernel<double><<<grid, 256, 0, c->stream>>>(n, c->NN, elems, c->cpos,
                                                                    (const double*)c->Kscr, c->Pscr, Ke, Pe);
    EFE_HIP(hipGetLastError());
    return EFE_OK;
}

int efe_launch_export_csr(efe_ctx* c, double* values) {
    const int grid = (c->N + 255) / 256;
    if (c->Kprec == EFE_FP32)
        export_csr_kernel<float><<<grid, 256, 0, c->stream>>>(c->N, c->bptr, c->slice_off, c->nodeSlot, c->K32,
                                                               values);
    else
        export_csr_kernel<double><<<grid, 256, 0, c->stream>>>(c->N, c->bptr, c->slice_off, c->nodeSlot, c->K64,
                                                                values);
    EFE_HIP(hipGetLastError());
    return EFE_OK;
}
