// The native element ABI on the GPU: MarmotElement::computeYourself
// (marmotelement/element.pxd:97-103, called per element by NISTParallelForMarmotElements,
// solvers/nonlinearimplicitstaticparallel.pyx:65-167) for a list of elements in one launch,
// with caller-owned arrays:
//   dQ        [n][nDof]            increment of the element's DOFs (node-major, 3 a + c)
//   stateRef  [n][Q][nState]       QP state at the start of the increment (stress 6, strain 6,
//                                  material state; element.py:222-236)
//   stateTemp [n][Q][nState]       the updated state (may be stateRef: in place)
//   Pe        [n][nDof]            -sum_q B^T sigma detJ w
//   Ke        [n][nDof][nDof]      column-major sum_q B^T C B detJ w, or none
// The element formulation is the context's (DisplacementElement.computeYourself,
// element.py:290-346, with the reference's Jacobian), and so are its material and properties.
// One workgroup per EPW elements, in four phases: the nodes' coordinates and increments to LDS; thread
// per (element, QP): J, strain increment, material update; thread per (element, QP, node): g =
// grad N_a and h = n g; thread per (element, node a, pair of nodes b): two 3x3 blocks of Ke.
#include <vector>

#include "efe_internal.h"
#include "materials.h"

namespace {

// The tangent in compact form, as in the element passes (elements.hip): with C = A 1(x)1 + B Idev +
// cnn n(x)n + cn1 n(x)1 + c1n 1(x)n, lambda = A - B/3, mu = B/2,
//   K_ab = sum_q (lambda g_a + cn1 h_a) g_b^T + (c1n g_a + cnn h_a) h_b^T + mu (g_b g_a^T + (g_a . g_b) I),
// 30 FMA per block and QP where C as a 6x6 matrix took 81.  A thread's two blocks share what goes
// with a, and consecutive threads have consecutive a, whose rows lie side by side in a column of Ke
// (with b running fastest a store went to 64 columns).  What bounds it now is the chain of a
// workgroup's phases; Ke alone is 29 KB per hexa20 element.  Kernel for 1716 hexa20R Drucker-Prager
// elements, one wavefront per two elements and C as a matrix 63.8 us, now 41.1 (49 MB of Ke); the whole
// call 89 -> 69 us, 13824 hexa8 J2 elements 129 -> 99, 64 hexa20R 79 -> 48.  Held to 128 VGPRs 82 / 111 /
// 53, 512 threads 89 / 117 / 45, one hexa20R element per 128 threads 77 / 99 / 47.
//
// KE: whether the call wants Ke.  Without it a wavefront is enough for the phases that are left, and the
// LDS of h goes.  Whole call with 256 -> 64 threads: hexa20 12^3 Drucker-Prager 56.0 -> 49.7 us, 24^3 J2
// 187 -> 142, hexa20R 24^3 134 -> 89.  hexa8 takes 4 elements then in lists of up to 65536 (27000 elements:
// Drucker-Prager 120.6 -> 113.1, 118.6 with 8; linear elastic 108.9 -> 110.7, 115.0 with 8) and 8 in
// longer ones (216000 J2 elements 658 -> 625, 661 with 4).
template <int NN, int Q, int MAT, int EPW, bool KE>
__global__ __launch_bounds__(KE ? 256 : 64) void element_abi_kernel(
    int cnt, const int32_t* __restrict__ kmap, const int32_t* __restrict__ emap, int E, int N,
    const double* __restrict__ coords, const int32_t* __restrict__ conn, const double* __restrict__ props,
    int propStride, const double* __restrict__ dNdxi, const double* __restrict__ dJdxi,
    const double* __restrict__ qpw, const double* __restrict__ dQ, const double* __restrict__ sRef,
    double* __restrict__ sTmp, int ns, double* __restrict__ Pe, double* __restrict__ Ke, int* __restrict__ status) {
    constexpr int NP = (MAT == EFE_LINEAR_ELASTIC) ? 2 : 6;
    constexpr int ND = 3 * NN, kBS = KE ? 256 : 64;
    constexpr bool LE = MAT == EFE_LINEAR_ELASTIC;
    static_assert(NN % 2 == 0, "blocks in pairs");
    __shared__ double x_s[EPW][NN][6];                         // coordinates, increment
    __shared__ double iJ_s[EPW][Q][9];
    __shared__ double g_s[EPW][Q][NN][3];
    constexpr bool H = KE && !LE;
    __shared__ double h_s[H ? EPW : 1][H ? Q : 1][H ? NN : 1][3];
    __shared__ double c_s[EPW][Q][5], n_s[LE ? 1 : EPW][LE ? 1 : Q][6];  // w detJ [lambda, mu, cnn, cn1, c1n]; n
    __shared__ double fs_s[EPW][Q][6];
    const int tid = threadIdx.x;
    const int i0 = blockIdx.x * EPW;
    const int ne = cnt - i0 < EPW ? cnt - i0 : EPW;

    for (int t = tid; t < ne * NN; t += kBS) {
        const int el = t / NN, a = t - (t / NN) * NN;
        const int nd = conn[(int64_t)a * E + emap[i0 + el]];
        const double* du = dQ + (int64_t)kmap[i0 + el] * ND + 3 * a;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            x_s[el][a][c] = coords[(int64_t)c * N + nd];
            x_s[el][a][3 + c] = du[c];
        }
    }
    __syncthreads();

    double det = 0.0;
    if (tid < ne * Q) {
        const int el = tid / Q, q = tid - (tid / Q) * Q;
        const double* dj = dJdxi + (size_t)q * NN * 3;
        double J[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll 4
        for (int a = 0; a < NN; ++a) {
#pragma unroll
            for (int r = 0; r < 3; ++r) {
                const double d = dj[a * 3 + r];
#pragma unroll
                for (int c = 0; c < 3; ++c) J[r * 3 + c] += d * x_s[el][a][c];
            }
        }
        det = J[0] * (J[4] * J[8] - J[5] * J[7]) - J[1] * (J[3] * J[8] - J[5] * J[6]) +
              J[2] * (J[3] * J[7] - J[4] * J[6]);
        const double id = 1.0 / det;
        double* iJ = iJ_s[el][q];
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

    for (int t = tid; t < ne * Q * NN; t += kBS) {
        const int el = t / (Q * NN), r = t - el * Q * NN, q = r / NN, a = r - (r / NN) * NN;
        const double* dn = dNdxi + ((size_t)q * NN + a) * 3;
        const double d0 = dn[0], d1 = dn[1], d2 = dn[2];
        const double* iJ = iJ_s[el][q];
#pragma unroll
        for (int c = 0; c < 3; ++c) g_s[el][q][a][c] = iJ[c * 3 + 0] * d0 + iJ[c * 3 + 1] * d1 + iJ[c * 3 + 2] * d2;
    }
    __syncthreads();

    if (tid < ne * Q) {
        const int el = tid / Q, q = tid - (tid / Q) * Q;
        const int k = kmap[i0 + el], e = emap[i0 + el];
        double gr[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll 4
        for (int a = 0; a < NN; ++a)
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int j = 0; j < 3; ++j) gr[i * 3 + j] += x_s[el][a][3 + i] * g_s[el][q][a][j];
        const double de[6] = {gr[0], gr[4], gr[8], gr[1] + gr[3], gr[2] + gr[6], gr[5] + gr[7]};
        const double* sr = sRef + ((int64_t)k * Q + q) * ns;
        double* st = sTmp + ((int64_t)k * Q + q) * ns;
        double s[6], eps[6], ms = 0.0;
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            s[c] = sr[c];
            eps[c] = sr[6 + c];
        }
        if (!LE && ns > 12) ms = sr[12];
        double p[NP];
#pragma unroll
        for (int m = 0; m < NP; ++m) p[m] = propStride ? props[(int64_t)m * propStride + e] : props[m];
        double C[36], cc[11];
        int fail = 0;
        if (LE) fail = efe::le_update(p, s, de, C, cc);
        else if (MAT == EFE_VONMISES) fail = efe::vm_update(p, s, ms, de, C, cc);
        else fail = efe::dp_update(p, s, ms, de, C, cc);
        if (fail) *status = 1;
        // the state out: other columns (a wider state of another section) are carried over
        for (int c = 0; c < ns; ++c) st[c] = sr[c];
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            st[c] = s[c];
            st[6 + c] = eps[c] + de[c];
        }
        if (!LE && ns > 12) st[12] = ms;
        const double f = det * qpw[q];
        c_s[el][q][0] = f * (cc[0] - cc[1] * (1.0 / 3.0));
        c_s[el][q][1] = f * (0.5 * cc[1]);
#pragma unroll
        for (int m = 2; m < 5; ++m) c_s[el][q][m] = f * cc[m];
        if (!LE)
#pragma unroll
            for (int m = 0; m < 6; ++m) n_s[el][q][m] = cc[5 + m];
#pragma unroll
        for (int m = 0; m < 6; ++m) fs_s[el][q][m] = f * s[m];
    }
    __syncthreads();

    if constexpr (KE) {
        if constexpr (!LE) {
            for (int t = tid; t < ne * Q * NN; t += kBS) {
                const int el = t / (Q * NN), r = t - el * Q * NN, q = r / NN, a = r - (r / NN) * NN;
                const double* n = n_s[el][q];
                const double x = g_s[el][q][a][0], y = g_s[el][q][a][1], z = g_s[el][q][a][2];
                h_s[el][q][a][0] = n[0] * x + n[3] * y + n[4] * z;
                h_s[el][q][a][1] = n[3] * x + n[1] * y + n[5] * z;
                h_s[el][q][a][2] = n[4] * x + n[5] * y + n[2] * z;
            }
            __syncthreads();
        }
        constexpr int NB2 = NN / 2;
        for (int t = tid; t < ne * NN * NB2; t += kBS) {
            const int el = t / (NN * NB2), r = t - el * NN * NB2, b0 = r / NN, a = r - (r / NN) * NN;
            double acc[2][9], tr[2] = {0, 0};
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int k = 0; k < 9; ++k) acc[h][k] = 0.0;
            for (int q = 0; q < Q; ++q) {
                const double* c = c_s[el][q];
                double u[3], v[3], w[3];
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    const double g = g_s[el][q][a][i];
                    u[i] = c[0] * g;
                    w[i] = c[1] * g;
                    if constexpr (!LE) {
                        const double hh = h_s[el][q][a][i];
                        v[i] = c[2] * hh;
                        if constexpr (MAT == EFE_DRUCKER_PRAGER) {
                            u[i] += c[3] * hh;
                            v[i] += c[4] * g;
                        }
                    }
                }
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const double* gb = g_s[el][q][b0 + h * NB2];
                    tr[h] += w[0] * gb[0] + w[1] * gb[1] + w[2] * gb[2];
#pragma unroll
                    for (int i = 0; i < 3; ++i)
#pragma unroll
                        for (int j = 0; j < 3; ++j) acc[h][i * 3 + j] += u[i] * gb[j] + w[j] * gb[i];
                    if constexpr (!LE) {
                        const double* hb = h_s[el][q][b0 + h * NB2];
#pragma unroll
                        for (int i = 0; i < 3; ++i)
#pragma unroll
                            for (int j = 0; j < 3; ++j) acc[h][i * 3 + j] += v[i] * hb[j];
                    }
                }
            }
            double* dst = Ke + (int64_t)kmap[i0 + el] * ND * ND;
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int j = 0; j < 3; ++j)
#pragma unroll
                    for (int i = 0; i < 3; ++i)
                        dst[(int64_t)(3 * (b0 + h * NB2) + j) * ND + 3 * a + i] =
                            i == j ? acc[h][i * 3 + j] + tr[h] : acc[h][i * 3 + j];
        }
    }

    for (int t = tid; t < ne * NN; t += kBS) {
        const int el = t / NN, a = t - (t / NN) * NN;
        double p0 = 0, p1 = 0, p2 = 0;
        for (int q = 0; q < Q; ++q) {
            const double ax = g_s[el][q][a][0], ay = g_s[el][q][a][1], az = g_s[el][q][a][2];
            const double* s = fs_s[el][q];
            p0 += ax * s[0] + ay * s[3] + az * s[4];
            p1 += ay * s[1] + ax * s[3] + az * s[5];
            p2 += az * s[2] + ax * s[4] + ay * s[5];
        }
        double* dst = Pe + (int64_t)kmap[i0 + el] * ND + 3 * a;
        dst[0] = -p0;
        dst[1] = -p1;
        dst[2] = -p2;
    }
}

template <int NN, int Q, int MAT>
void launch_abi(efe_ctx* c, int cnt, const int32_t* kmap, const int32_t* emap, const double* dQ, const double* sRef,
                double* sTmp, double* Pe, double* Ke) {
    constexpr int EPW = (NN == 8) ? 8 : (Q == 8 ? 2 : 1);
    static_assert(EPW * Q <= 64, "a thread per (element, QP)");
    if (cnt == 0) return;
    auto launch = [&](auto kernel, int epw, int threads) {
        kernel<<<(cnt + epw - 1) / epw, threads, 0, c->stream>>>(
            cnt, kmap, emap, c->E, c->N, c->coords, c->conn, c->props, c->props_per_element ? c->E : 0, c->dNdxi,
            c->dJdxi, c->qpw, dQ, sRef, sTmp, c->nstate, Pe, Ke, c->status);
    };
    if (Ke) launch(element_abi_kernel<NN, Q, MAT, EPW, true>, EPW, 256);
    else if (NN == 8 && cnt <= 65536) launch(element_abi_kernel<NN, Q, MAT, NN == 8 ? 4 : EPW, false>, 4, 64);
    else launch(element_abi_kernel<NN, Q, MAT, EPW, false>, EPW, 64);
}

template <int NN, int Q>
void launch_abi_mat(efe_ctx* c, int mat, int cnt, const int32_t* kmap, const int32_t* emap, const double* dQ,
                    const double* sRef, double* sTmp, double* Pe, double* Ke) {
    if (mat == EFE_LINEAR_ELASTIC) launch_abi<NN, Q, EFE_LINEAR_ELASTIC>(c, cnt, kmap, emap, dQ, sRef, sTmp, Pe, Ke);
    else if (mat == EFE_VONMISES) launch_abi<NN, Q, EFE_VONMISES>(c, cnt, kmap, emap, dQ, sRef, sTmp, Pe, Ke);
    else launch_abi<NN, Q, EFE_DRUCKER_PRAGER>(c, cnt, kmap, emap, dQ, sRef, sTmp, Pe, Ke);
}

}  // namespace

extern "C" int efe_element_compute(efe_ctx* c, const int32_t* elements, int32_t n, const double* QTotal,
                                   const double* dQ, const double* stateRef, double* stateTemp, double* Pe,
                                   double* Ke, const double* time, double dT, double* pNewDT) {
    (void)QTotal;
    (void)time;
    (void)dT;
    if (!c) {
        efe_set_error("null context");
        return EFE_ERR_ARG;
    }
    if (n < 0 || (n > 0 && (!elements || !dQ || !stateRef || !stateTemp || !Pe)) || !pNewDT) {
        efe_set_error("efe_element_compute: invalid arguments");
        return EFE_ERR_ARG;
    }
    // the listed elements by material group (the order of each group kept), positions k in
    // the caller's arrays and element indices e of the context
    std::vector<int32_t> km, em;
    km.reserve(n);
    em.reserve(n);
    std::vector<int> gcount(c->ngroups, 0);
    for (int32_t i = 0; i < n; ++i)
        if (elements[i] < 0 || elements[i] >= c->E) {
            efe_set_error("efe_element_compute: element out of range");
            return EFE_ERR_ARG;
        }
    for (int g = 0; g < c->ngroups; ++g)
        for (int32_t i = 0; i < n; ++i)
            if (c->ngroups == 1 || c->matOf[elements[i]] == c->groupMat[g]) {
                km.push_back(i);
                em.push_back(elements[i]);
                ++gcount[g];
            }
    if (n == 0) return EFE_OK;
    const size_t need = 2 * (size_t)n;
    if (need > c->resCap) {
        hipFree(c->resIdx);
        c->resIdx = nullptr;
        c->resCap = 0;
        EFE_HIP(hipMalloc(&c->resIdx, need * sizeof(int32_t)));
        c->resCap = need;
    }
    std::vector<int32_t> both(km);
    both.insert(both.end(), em.begin(), em.end());
    EFE_HIP(hipMemcpyAsync(c->resIdx, both.data(), need * sizeof(int32_t), hipMemcpyHostToDevice, c->stream));
    EFE_HIP(hipMemsetAsync(c->status, 0, sizeof(int), c->stream));
    int off = 0;
    for (int g = 0; g < c->ngroups; ++g) {
        const int32_t* kmap = c->resIdx + off;
        const int32_t* emap = c->resIdx + n + off;
        const int cnt = gcount[g], mat = c->groupMat[g];
        switch (c->eltype) {
            case EFE_C3D8: launch_abi_mat<8, 8>(c, mat, cnt, kmap, emap, dQ, stateRef, stateTemp, Pe, Ke); break;
            case EFE_C3D20: launch_abi_mat<20, 27>(c, mat, cnt, kmap, emap, dQ, stateRef, stateTemp, Pe, Ke); break;
            default: launch_abi_mat<20, 8>(c, mat, cnt, kmap, emap, dQ, stateRef, stateTemp, Pe, Ke); break;
        }
        EFE_HIP(hipGetLastError());
        off += cnt;
    }
    int hs = 0;
    EFE_HIP(hipMemcpyAsync(&hs, c->status, sizeof(int), hipMemcpyDeviceToHost, c->stream));
    EFE_HIP(hipStreamSynchronize(c->stream));  // both must outlive the copy
    if (hs) {
        *pNewDT = *pNewDT < 0.5 ? *pNewDT : 0.5;
        return EFE_CUTBACK;
    }
    return EFE_OK;
}
