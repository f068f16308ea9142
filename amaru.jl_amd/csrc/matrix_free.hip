// Element data of the matrix-free operator of the PCG (pcg_mf_kernel in
// kernels_solve.hip): K x of a model whose materials are all LinearElastic as
// the sum over the elements of Be' (coef De) Be xe, from per-IP geometry
// instead of the assembled matrix.
//
// What it reads per element is 72 B per IP (HEX20 with 27 IPs: 1.9 KB, HEX8
// 0.6 KB, TET10 0.3 KB) against 38 to 76 B per 3x3 block of the assembled matrix
// (HEX20: 9 to 18 KB of blocks per element).
//
// Layout.  Elements are taken in groups of 16, one wave per group.  Lane l =
// 16 g + c of a group holds, of element 16 grp + c, the nodes 4 s + g (slot
// s) and the IPs 4 k + g (slot k): the operand and result layout of
// v_mfma_f64_4x4x4 (four blocks of 4x4x4), so that the products with the
// shape-derivative tables need no exchange between lanes.
#include <cmath>
#include <type_traits>
#include <vector>

#include "amr_internal.h"

namespace {

constexpr int NSLOT = 5, KSLOT = 7;  // largest numbers of node and IP slots (HEX20, 27 IPs)

// One thread per (group, IP slot, lane): A = inv(J) sqrt(det J w) of the IP (0
// for the padding elements and IPs), so that P = A' sigma(A' ...) carries the
// IP's weight once; per element lambda and mu of De (Mandel De is lambda
// tr(eps) I + 2 mu eps, src/mech/mat/linear-elastic.jl:98-123).  flag: bit 0 an
// IP without a positive determinant, bit 1 an element too soft or small for
// mount_K's |Ke_ij| < eps filter to be without effect on the product.
__global__ void __launch_bounds__(256) mf_geometry_kernel(int64_t n, int NN, int NQ, int KS, int64_t ne,
                                                          const double *__restrict__ X,
                                                          const int32_t *__restrict__ conn,
                                                          const int32_t *__restrict__ emat,
                                                          const AmrMat *__restrict__ mats,
                                                          const double *__restrict__ dNdR,
                                                          const double *__restrict__ wip, double *__restrict__ geo,
                                                          double *__restrict__ lm, int32_t *__restrict__ flag)
{
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= n) return;
    const int lane = (int)(t & 63), g = lane >> 4, c = lane & 15;
    const int64_t gk = t >> 6, grp = gk / KS;
    const int q = 4 * (int)(gk - grp * KS) + g;
    const int64_t e = grp * 16 + c;
    double A[9] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    if (e < ne && q < NQ) {
        double J[9] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        const double *dq = dNdR + (int64_t)q * NN * 3;
        for (int a = 0; a < NN; a++) {
            const double *x = X + (int64_t)conn[e * NN + a] * 3;
            for (int i = 0; i < 3; i++)
                for (int j = 0; j < 3; j++) J[i * 3 + j] = fma(x[i], dq[a * 3 + j], J[i * 3 + j]);
        }
        double C[9];
        for (int i = 0; i < 3; i++)
            for (int j = 0; j < 3; j++) {
                const int i1 = (i + 1) % 3, i2 = (i + 2) % 3, j1 = (j + 1) % 3, j2 = (j + 2) % 3;
                C[i * 3 + j] = J[i1 * 3 + j1] * J[i2 * 3 + j2] - J[i1 * 3 + j2] * J[i2 * 3 + j1];
            }
        const double det = J[0] * C[0] + J[1] * C[1] + J[2] * C[2];
        const double coef = det * wip[q];
        const AmrMat m = mats[emat[e]];
        const double E = m.p[0], nu = m.p[1], s = E / ((1.0 + nu) * (1.0 - 2.0 * nu));
        const double mu = 0.5 * (s * (1.0 - 2.0 * nu));
        if (!(det > 0.0) || !(coef > 0.0) || !std::isfinite(coef)) atomicOr(flag, 1);
        if (!(mu * cbrt(coef * NQ) >= 1.0)) atomicOr(flag, 2);
        const double f = sqrt(coef) / det;
        for (int i = 0; i < 3; i++)
            for (int j = 0; j < 3; j++) A[i * 3 + j] = C[j * 3 + i] * f;
        if (q == 0) {
            lm[grp * 32 + c] = s * nu;
            lm[grp * 32 + 16 + c] = mu;
        }
    } else if (q == 0) {
        lm[grp * 32 + c] = lm[grp * 32 + 16 + c] = 0.0;
    }
    for (int r = 0; r < 9; r++) geo[(gk * 9 + r) * 64 + lane] = A[r];
}

// One thread per (group, node slot, lane): the lane's node (node 0 of the
// mesh for padding; its table entries are 0).
__global__ void __launch_bounds__(256) mf_conn_kernel(int64_t n, int NN, int NS, int64_t ne,
                                                      const int32_t *__restrict__ conn,
                                                      int32_t *__restrict__ mfconn)
{
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= n) return;
    const int lane = (int)(t & 63);
    const int64_t gs = t >> 6, grp = gs / NS;
    const int a = 4 * (int)(gs - grp * NS) + (lane >> 4);
    const int64_t e = grp * 16 + (lane & 15);
    mfconn[t] = e < ne ? conn[e * NN + (a < NN ? a : 0)] : 0;
}

// One thread per incidence p of the force-gather map (node -> (element, local
// node), ascending element): where the group's wave stores component 0 of
// that element node's product.
__global__ void __launch_bounds__(256) mf_src_kernel(int64_t n, int NN, int NS, const int32_t *__restrict__ fsrc,
                                                     int32_t *__restrict__ src)
{
    const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (p >= n) return;
    const int32_t v = fsrc[p], e = v / NN, a = v - e * NN;
    src[p] = ((e >> 4) * NS + (a >> 2)) * 192 + (a & 3) * 16 + (e & 15);
}

// One thread per entry of the nodes' records: the places of a node's first
// eight products (-1: fewer), 32 bytes per node read without the dependent
// load of the list's bounds.  Nodes of structured hexahedra have at most
// eight, most nodes of tetrahedra fewer.
__global__ void __launch_bounds__(256) mf_rec_kernel(int64_t n, const int32_t *__restrict__ fptr,
                                                     const int32_t *__restrict__ src, int32_t *__restrict__ rec)
{
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= n) return;
    const int64_t k = fptr[t >> 3] + (t & 7);
    rec[t] = k < fptr[(t >> 3) + 1] ? src[k] : -1;
}

}  // namespace

// Tables of the two products, 16 values per 4x4 block (the four blocks of an
// instruction share them; lane m + 4 b + 16 kk reads value m + 4 kk).  First
// part, slot (k, j), node slot s: dN_a/dR_j at IP q = 4 k + m with a = 4 s + kk
// (rows IPs, inner dimension nodes).  Second part: dN_a/dR_j at IP q = 4 k + kk
// with a = 4 s + m (rows nodes, inner dimension IPs).  Entries past NN or NQ
// are 0.
static std::vector<double> mf_tables(int NN, int NQ, const double *dNdR)
{
    const int NS = (NN + 3) / 4, KS = (NQ + 3) / 4, half = KS * 3 * NS * 16;
    std::vector<double> T((size_t)2 * half, 0.0);
    auto at = [&](int q, int a, int j) { return q < NQ && a < NN ? dNdR[(q * NN + a) * 3 + j] : 0.0; };
    for (int k = 0; k < KS; k++)
        for (int j = 0; j < 3; j++)
            for (int s = 0; s < NS; s++)
                for (int l = 0; l < 16; l++) {
                    const int m = l & 3, kk = l >> 2, o = ((k * 3 + j) * NS + s) * 16 + l;
                    T[o] = at(4 * k + m, 4 * s + kk, j);
                    T[half + o] = at(4 * k + kk, 4 * s + m, j);
                }
    return T;
}

// Queues the element data of an all-elastic model on its stream (nothing for
// other models).
int amr_mf_build(amr_model *m, const double *dNdR_host)
{
    m->mf_ok = false;
    if (!m->all_elastic || m->ne == 0) return AMR_OK;
    const int NN = m->nn, NQ = m->nips, NS = (NN + 3) / 4, KS = (NQ + 3) / 4;
    static_assert(NSLOT * 4 >= AMR_MAXNN && KSLOT * 4 >= AMR_MAXIP, "slots");
    const int64_t ngrp = (m->ne + 15) / 16;
    // the product's offsets are 32-bit
    if (ngrp * NS * 192 >= ((int64_t)1 << 31) || m->ne * NN >= ((int64_t)1 << 31)) return AMR_OK;
    m->mf_ngrp = ngrp;
    m->mf_tab_h = mf_tables(NN, NQ, dNdR_host);
    // the arrays as slices of one block (one allocation), 256-byte aligned
    size_t off = 0;
    auto slice = [&off](size_t bytes) {
        const size_t o = off;
        off = (off + bytes + 255) & ~(size_t)255;
        return o;
    };
    const size_t o_tab = slice(m->mf_tab_h.size() * 8), o_geo = slice((size_t)ngrp * KS * 9 * 64 * 8),
                 o_lm = slice((size_t)ngrp * 32 * 8), o_f = slice((size_t)ngrp * NS * 192 * 8),
                 o_conn = slice((size_t)ngrp * NS * 64 * 4), o_src = slice((size_t)m->ne * NN * 4), o_rec = slice((size_t)m->nnodes * 32),
                 o_flag = slice(4);
    const int rc = amr_dalloc(m, (void **)&m->mf_block, off);
    if (rc == AMR_ERR_NOMEM) {
        // the model does without: it iterates on the assembled matrix (so it
        // does when a later allocation needs the block, amr_hip_malloc)
        (void)hipGetLastError();
        m->mf_block = nullptr;
        return AMR_OK;
    }
    if (rc) return rc;
    auto at = [&](auto **p, size_t o) { *p = (std::remove_reference_t<decltype(**p)> *)(m->mf_block + o); };
    at(&m->mf_tab, o_tab);
    at(&m->mf_geo, o_geo);
    at(&m->mf_lm, o_lm);
    at(&m->mf_f, o_f);
    at(&m->mf_conn, o_conn);
    at(&m->mf_src, o_src);
    at(&m->mf_rec, o_rec);
    at(&m->mf_flag, o_flag);
    hipStream_t s = m->stream;
    AMR_HIP(hipMemcpyAsync(m->mf_tab, m->mf_tab_h.data(), m->mf_tab_h.size() * sizeof(double),
                           hipMemcpyHostToDevice, s));
    AMR_HIP(hipMemsetAsync(m->mf_flag, 0, sizeof(int32_t), s));
    const int64_t n0 = ngrp * KS * 64, n1 = ngrp * NS * 64, n2 = m->ne * NN;
    auto grid = [](int64_t n) { return dim3((unsigned)((n + 255) / 256)); };
    hipLaunchKernelGGL(mf_geometry_kernel, grid(n0), dim3(256), 0, s, n0, NN, NQ, KS, m->ne, m->X, m->conn, m->emat,
                       m->mats, m->dNdR, m->wip, m->mf_geo, m->mf_lm, m->mf_flag);
    hipLaunchKernelGGL(mf_conn_kernel, grid(n1), dim3(256), 0, s, n1, NN, NS, m->ne, m->conn, m->mf_conn);
    hipLaunchKernelGGL(mf_src_kernel, grid(n2), dim3(256), 0, s, n2, NN, NS, m->fsrc, m->mf_src);
    hipLaunchKernelGGL(mf_rec_kernel, grid(m->nnodes * 8), dim3(256), 0, s, m->nnodes * 8, m->fptr, m->mf_src,
                       m->mf_rec);
    AMR_HIP(hipGetLastError());
    return AMR_OK;
}

// After a wait for amr_mf_build's work: whether the operator may be used.
int amr_mf_check(amr_model *m)
{
    std::vector<double>().swap(m->mf_tab_h);
    if (!m->mf_block) return AMR_OK;
    int32_t flag = 0;
    AMR_HIP(hipMemcpyAsync(&flag, m->mf_flag, sizeof flag, hipMemcpyDeviceToHost, m->stream));
    AMR_HIP(hipStreamSynchronize(m->stream));
    if (flag == 0) m->mf_ok = true;
    else amr_mf_free(m);
    return AMR_OK;
}

void amr_mf_free(amr_model *m)
{
    amr_release(m, m->mf_block);
    m->mf_block = nullptr;
    m->mf_ok = false;
}
