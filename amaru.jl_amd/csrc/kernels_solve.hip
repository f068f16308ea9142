// Solver kernels for gfx950: node-block (3x3) SpMV and Jacobi-PCG, replacing
// the UMFPACK solve of solve_system! (src/solver.jl:42-43), plus the vector
// kernels of the device-resident stage driver.
//
// Vectors live in node order (3 dofs per node).  The operator is K with the
// prescribed dofs masked out: y = mask .* (K x).  With x zero at prescribed
// dofs this is K11 x on the unknowns, so one resident copy of K serves K11,
// K12 U2 (right-hand side) and K21 U1 + K22 U2 (reactions).
//
// Pools.  The PCG kernels work on a pool of independent systems (models) at
// once: a descriptor per model holds its matrix, vectors, partials and
// scalars, and every launch walks a work list of (model, row tile) or
// (model, vector block) entries, so one launch per PCG phase advances every
// model of the pool.  Each model's tile and block decomposition depends on
// that model alone, and each model's scalars are reduced from its own
// partials in a fixed order, so a model's iterates are bit-identical whether
// it is solved alone (a pool of one, which is what amr_pcg_solve does) or
// together with any others.  Models join and leave the pool between steps
// (continuous batching at the granularity of one step of check_every
// iterations).
//
// Reductions need no atomics and no fences: a reducing kernel writes one
// partial per workgroup, and every workgroup of the next kernel that needs
// the scalar sums those partials itself in index order (kernel boundaries
// make them visible).
//
// Precision.  Matrix-free members (all-elastic models) multiply in FP64 from
// the element geometry in every mode.  Plain path: FP64 PCG.  Mixed paths: the same CG recurrences
// with FP64 vectors, FP64 dot products and FP64 solution update, but the
// SpMV reads FP32 values (with an FP32 copy of the search direction and FP32
// accumulation for AMR_PREC_MIXED, FP64 gather and accumulation for
// AMR_PREC_MIXED_F64ACC) and the preconditioner is applied in FP32.  The
// FP64 residual r = b - K x is recomputed with the FP64 matrix whenever the
// recursive residual has dropped 10x since the last recomputation and at the
// end (residual replacement), which keeps the iteration converging to the
// FP64 solution without restarting the Krylov process; a model whose FP32
// operator drifts too far from K falls back to the FP64 operator.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "amr_internal.h"
#include "wave_ops.h"

namespace {

constexpr int WGV = 256;  // vector kernels
constexpr int WGS = 512;  // SpMV kernels
constexpr int MAX_GR = 8192, MAX_GV = 1024;

// scalar and control slots of one model: S_NSCAL doubles, then C_NCTL ints
// S_RZP0/1: r.z published per parity slot (the sum of that slot's partials)
// S_BETA: the running iteration's beta (members whose operator forms the direction)
enum { S_RZ = 0, S_RR, S_BB, S_THR, S_KX, S_RES, S_ERRN, S_ERRD, S_GAP, S_RZP0, S_RZP1, S_BETA, S_NSCAL = 16 };
__device__ inline int rz_pub(int slot) { return slot ? S_RZP1 : S_RZP0; }
// C_DONE is read by every workgroup at kernel entry and written only where
// all workgroups of the model in the running launch agree on it
// (breakdown); the convergence test writes C_STOP, which the next operator
// launch promotes to C_DONE.  Where pcg_dir_kernel tests, it reads no C_STOP,
// so none of its workgroups sees a flag of its own launch.  Where the operator
// forms the direction, its first tile tests: later tiles of that launch may
// see C_STOP and leave, earlier ones work on; either is right, since the
// update kernel reads C_STOP first, uses nothing of a stopped iteration and
// promotes the flag itself.  The direction is not stored then (REZ_FORM).
// C_ITERS is advanced by the operator's first tile and read by the kernels
// after it.  C_PREV is the number of completed iterations, advanced by the
// update kernel: the tiles of an operator that forms the direction read it
// (one of them writes C_ITERS in the same launch).
enum { C_DONE = 0, C_ITERS, C_BREAK, C_NAN, C_STOP, C_PREV, C_NCTL = 16 };
constexpr int SEG_DBL = 32;  // doubles per model in a pool's scalar array
static_assert(S_NSCAL + C_NCTL / 2 <= SEG_DBL, "scalar block");
// partial buffers inside m->part
enum { P_PQ = 0, P_RZ0 = 8192, P_RZ1 = 9216, P_RR0 = 10240, P_RR1 = 11264, P_CY0 = 12288, P_CY1 = 12800, P_A = 13312,
       P_B = 21504, P_C = 29696, P_D = 37888, P_END = 46080 };
static_assert(P_END == AMR_PART_DBL, "partials layout");
constexpr int MAX_CW = 512;  // coarse-product workgroups per model (4 coarse rows each)

// Pointers taken from a descriptor are generic; device buffers are all in
// the global address space, and saying so lets the compiler use global
// (not flat) memory instructions.
template <typename T>
__device__ inline const __attribute__((address_space(1))) T *gl(const T *p)
{
    return (const __attribute__((address_space(1))) T *)p;
}
template <typename T>
__device__ inline __attribute__((address_space(1))) T *glw(T *p)
{
    return (__attribute__((address_space(1))) T *)p;
}

template <int NT>
__device__ inline double block_sum(double v)
{
    __shared__ double sh[NT / 64];
    v = wave_sum(v);
    __syncthreads();
    if (threadIdx.x % 64 == 0) sh[threadIdx.x / 64] = v;
    __syncthreads();
    double t = 0.0;
    for (int i = 0; i < NT / 64; i++) t += sh[i];
    return t;  // same value in every thread
}

// N block sums at once; thread t < N gets sum t.
template <int NT, int N>
__device__ inline double block_sums(const double v[N])
{
    __shared__ double sh[NT / 64][N];
    __syncthreads();
    double w[N];
#pragma unroll
    for (int k = 0; k < N; k++) w[k] = wave_sum(v[k]);
    if (threadIdx.x % 64 == 0)
#pragma unroll
        for (int k = 0; k < N; k++) sh[threadIdx.x / 64][k] = w[k];
    __syncthreads();
    double t = 0.0;
    if (threadIdx.x < N)
        for (int i = 0; i < NT / 64; i++) t += sh[i][threadIdx.x];
    return t;
}

template <int NT>
__device__ inline double block_max(double v)
{
    __shared__ double sh[NT / 64];
    for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_down(v, off, 64));
    __syncthreads();
    if (threadIdx.x % 64 == 0) sh[threadIdx.x / 64] = v;
    __syncthreads();
    double t = 0.0;
    for (int i = 0; i < NT / 64; i++) t = fmax(t, sh[i]);
    return t;
}

// A thread's share of the sum of n partials (block_sum adds the shares: a
// fixed order).
template <int NT>
__device__ inline double thread_partials(const double *__restrict__ P, int n)
{
    double v = 0.0;
    const auto *Pg = gl(P);
    // a thread's loads are issued before its additions, which keep the order
    // i, i + NT, ...; addresses past the end are clamped, so that the loads
    // need no branches
    const int last = n - 1;
    if (n <= 4 * NT) {
        double a[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int i = (int)threadIdx.x + k * NT;
            a[k] = Pg[i < n ? i : last];
        }
#pragma unroll
        for (int k = 0; k < 4; k++) v = (int)threadIdx.x + k * NT < n ? v + a[k] : v;
        return v;
    }
    for (int i = threadIdx.x; i < n; i += 16 * NT) {
        double a[16];
#pragma unroll
        for (int k = 0; k < 16; k++) a[k] = Pg[i + k * NT < n ? i + k * NT : last];
#pragma unroll
        for (int k = 0; k < 16; k++) v = i + k * NT < n ? v + a[k] : v;
    }
    return v;
}

// Sum of n partials in a fixed order; every thread gets the result.
template <int NT>
__device__ inline double sum_partials(const double *__restrict__ P, int n)
{
    return block_sum<NT>(thread_partials<NT>(P, n));
}

typedef int32_t i32x4 __attribute__((ext_vector_type(4)));

// One model of a pool, as the kernels see it.
struct SegDesc {
    const int32_t *rowptr, *col;
    const int16_t *col16;         // column - row per block when every offset fits 16 bits, else null
    const double *Kv;
    const float *Kv32;
    const double *mask;
    const double *dinv, *binv;    // Jacobi / nodal block-Jacobi inverses
    const float *dinv32, *binv32;
    const double *b;              // right-hand side (node order, 0 at prescribed dofs)
    double *x, *r, *z, *p, *q, *rt;
    float *p32;                   // FP32 copy of p (AMR_PREC_MIXED)
    double *part, *scal;
    int32_t *ctl;
    int64_t nnodes, nblk;
    double thr_fac;               // recursive-residual stop: rr <= thr_fac * bb
    int R, ntiles, nvblk, maxiter;
    int f32;                      // preconditioner applied in FP32
    int block;                    // nodal block Jacobi
    int wp32;                     // keep p32 up to date
    int tl;                       // two-level: add the coarse correction Phi Kc^-1 Phi^T r
    // two-level coarse space
    int nagg, nc, ncw;
    const int32_t *agg, *aggptr, *aggnodes;
    const double *cent, *X, *Kinv;
    double *cvec, *yvec;
    // the nodes in aggregate order in chunks of one workgroup each (first
    // node, end, aggregate), the chunks of each aggregate, and the chunks'
    // parts of c
    const i32x4 *chunk;
    const int32_t *aggch;
    double *cpart;
    int nchunk;
    int cparts;                   // the update kernel goes by chunks and writes the parts of c
    int nred;                     // partials of r.z and r.r from the update kernel
    // matrix-free operator (null geo: the assembled matrix): element data of
    // matrix_free.hip, tiles of mfG groups of 16 elements per wave (or team of waves), and the map
    // node -> element products (CSR over nodes)
    const double *geo, *lm, *tab;
    const int32_t *mfconn, *mfrec, *fptr, *mfsrc;
    double *mff;
    int64_t ngrp;
    int mfG;
    int npq;                      // partials of p.q
    int fuse;                     // p = z + beta p formed by the operator and update kernels
};

// r.z with z = M r: the Jacobi part's partials plus, two-level, the coarse
// part c.y = (Phi^T r).(Kc^-1 Phi^T r)
__device__ inline double sum_rz(const SegDesc &d, int slot)
{
    double v = sum_partials<WGV>(d.part + (slot ? P_RZ1 : P_RZ0), d.nvblk);
    if (d.tl) v += sum_partials<WGV>(d.part + (slot ? P_CY1 : P_CY0), d.ncw);
    return v;
}

// coarse correction at dof c of node nd: (R_nd y_agg(nd))_c, masked
__device__ inline double coarse_term(const SegDesc &d, int64_t nd, int c)
{
    const int32_t a = gl(d.agg)[nd];
    const auto *y = gl(d.yvec) + (int64_t)a * 6;
    const auto *X = gl(d.X), *cent = gl(d.cent);
    const double dx = X[nd * 3] - cent[a * 3], dy = X[nd * 3 + 1] - cent[a * 3 + 1],
                 dz = X[nd * 3 + 2] - cent[a * 3 + 2];
    double v;
    if (c == 0) v = fma(-dy, y[5], fma(dz, y[4], y[0]));
    else if (c == 1) v = fma(dx, y[5], fma(-dz, y[3], y[1]));
    else v = fma(-dx, y[4], fma(dy, y[3], y[2]));
    return gl(d.mask)[nd * 3 + c] != 0.0 ? v : 0.0;
}

// Preconditioner: Jacobi (inverse diagonal) or 3x3 nodal block Jacobi
// (inverse of each node's diagonal block restricted to its free dofs), in
// FP64 or applied in FP32 (mixed paths).
__device__ inline void apply_prec(const SegDesc &P, int64_t node, const double r[3], double z[3])
{
    const int64_t i = node * 3;
    if (P.block) {
        if (P.f32) {
            const auto *B = gl(P.binv32) + node * 9;
            const float r0 = (float)r[0], r1 = (float)r[1], r2 = (float)r[2];
            for (int d = 0; d < 3; d++) z[d] = (double)fmaf(B[d * 3 + 2], r2, fmaf(B[d * 3 + 1], r1, B[d * 3] * r0));
        } else {
            const auto *B = gl(P.binv) + node * 9;
            for (int d = 0; d < 3; d++) z[d] = fma(B[d * 3 + 2], r[2], fma(B[d * 3 + 1], r[1], B[d * 3] * r[0]));
        }
    } else if (P.f32) {
        for (int d = 0; d < 3; d++) z[d] = (double)(gl(P.dinv32)[i + d] * (float)r[d]);
    } else {
        for (int d = 0; d < 3; d++) z[d] = gl(P.dinv)[i + d] * r[d];
    }
}

// ------------------------------------------------------------------ SpMV
//
// Row tiles: a workgroup owns block rows [t*R, (t+1)*R) of one model (R a
// power of two fixed per model), stages their row pointers in LDS and walks
// them with L lanes per row.  Each row's sum is formed over 64 virtual slots
// (slot j takes blocks rb+j, rb+j+64, ... in order) reduced by one fixed
// binary tree, whatever L is: a lane holds 64/L slots and performs the tree
// levels above L itself, the levels below L are cross-lane shuffles.
// Per-row dot contributions go to LDS and are reduced by a fixed tree too.
// So neither the row sums nor the partials depend on L, and L can be
// chosen per model for speed alone.


// The nine values of block k, converted to the accumulation type.
typedef double f64x2 __attribute__((ext_vector_type(2)));

template <typename VT, typename AT> struct BlockLoad;

// FP64 values (kv_at layout): four 2-wide loads and one scalar load
template <typename AT> struct BlockLoad<double, AT> {
    __device__ static inline void load(const double *__restrict__ vals, int64_t k, AT v[9])
    {
        const auto *base = gl(vals) + (k >> 6) * 576;
        const auto *pr = gl(reinterpret_cast<const f64x2 *>(vals + (k >> 6) * 576)) + (k & 63);
#pragma unroll
        for (int p = 0; p < 4; p++) {
            const f64x2 w = pr[p * 64];
            v[2 * p] = (AT)w.x;
            v[2 * p + 1] = (AT)w.y;
        }
        v[8] = (AT)base[512 + (k & 63)];
    }
};

// FP32 values (kv32_at layout): two 4-wide loads and one scalar load
typedef float f32x4 __attribute__((ext_vector_type(4)));
template <typename AT> struct BlockLoad<float, AT> {
    __device__ static inline void load(const float *__restrict__ vals, int64_t k, AT v[9])
    {
        const auto *base = gl(vals) + (k >> 6) * 576;
        const auto *pq = gl(reinterpret_cast<const f32x4 *>(vals + (k >> 6) * 576)) + (k & 63);
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const f32x4 w = pq[q * 64];
            v[4 * q] = (AT)w.x;
            v[4 * q + 1] = (AT)w.y;
            v[4 * q + 2] = (AT)w.z;
            v[4 * q + 3] = (AT)w.w;
        }
        v[8] = (AT)base[512 + (k & 63)];
    }
};

template <typename VT, typename AT>
__device__ inline void load_block(const VT *__restrict__ vals, int64_t k, AT v[9])
{
    BlockLoad<VT, AT>::load(vals, k, v);
}

// Column of block k: col[k], or with 16-bit column offsets row + col16[k].
template <typename CT>
__device__ inline int64_t block_col(const CT *__restrict__ col, int64_t k, int64_t row);
template <>
__device__ inline int64_t block_col<int32_t>(const int32_t *__restrict__ col, int64_t k, int64_t)
{
    return gl(col)[k];
}
template <>
__device__ inline int64_t block_col<int16_t>(const int16_t *__restrict__ col, int64_t k, int64_t row)
{
    return row + gl(col)[k];
}

// FUSE: the operand is z + beta x, formed as it is gathered.
template <int L, bool ABS, typename VT, typename XT, typename AT, typename CT = int32_t, bool FUSE = false>
__device__ inline void row_sum(int32_t rb, int32_t re, int sub, const CT *__restrict__ col,
                               const VT *__restrict__ vals, const XT *__restrict__ x, AT y[3], int64_t row = 0,
                               const double *__restrict__ z = nullptr, double beta = 0.0)
{
    constexpr int NS = 64 / L;
    AT acc[NS][3];
#pragma unroll
    for (int t = 0; t < NS; t++) acc[t][0] = acc[t][1] = acc[t][2] = (AT)0;
    for (int32_t base = rb; base < re; base += 64) {
#pragma unroll
        for (int t = 0; t < NS; t++) {
            const int32_t k = base + sub + L * t;
            if (k < re) {
                const int64_t c = block_col<CT>(col, k, row);
                const auto *xc = gl(x) + c * 3;
                AT x0 = (AT)xc[0], x1 = (AT)xc[1], x2 = (AT)xc[2];
                if (FUSE) {
                    const auto *zc = gl(z) + c * 3;
                    x0 = fma(beta, x0, zc[0]);
                    x1 = fma(beta, x1, zc[1]);
                    x2 = fma(beta, x2, zc[2]);
                }
                AT v[9];
                load_block<VT, AT>(vals, k, v);
                if (ABS) {
                    acc[t][0] += fabs(v[0] * x0) + fabs(v[1] * x1) + fabs(v[2] * x2);
                    acc[t][1] += fabs(v[3] * x0) + fabs(v[4] * x1) + fabs(v[5] * x2);
                    acc[t][2] += fabs(v[6] * x0) + fabs(v[7] * x1) + fabs(v[8] * x2);
                } else {
                    acc[t][0] = fma(v[2], x2, fma(v[1], x1, fma(v[0], x0, acc[t][0])));
                    acc[t][1] = fma(v[5], x2, fma(v[4], x1, fma(v[3], x0, acc[t][1])));
                    acc[t][2] = fma(v[8], x2, fma(v[7], x1, fma(v[6], x0, acc[t][2])));
                }
            }
        }
    }
    // tree levels with offset >= L combine slots held by the same lane
#pragma unroll
    for (int off = 32; off >= L; off >>= 1) {
#pragma unroll
        for (int t = 0; t < off / L; t++)
#pragma unroll
            for (int d = 0; d < 3; d++) acc[t][d] = acc[t][d] + acc[t + off / L][d];
    }
#pragma unroll
    for (int d = 0; d < 3; d++) {
        AT v = acc[0][d];
#pragma unroll
        for (int off = L / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, L);
        y[d] = v;
    }
}

// row_sum<L, false> (y = K x) and row_sum<L, true> (a = |K| |x|) of the
// same row in one pass over its blocks: each sum has the same slots and the
// same tree as alone, so the same bits.
template <int L, typename VT, typename XT, typename AT, typename CT = int32_t>
__device__ inline void row_sum_pair(int32_t rb, int32_t re, int sub, const CT *__restrict__ col,
                                    const VT *__restrict__ vals, const XT *__restrict__ x, AT y[3], AT a[3],
                                    int64_t row = 0)
{
    constexpr int NS = 64 / L;
    AT acc[NS][3], abs_[NS][3];
#pragma unroll
    for (int t = 0; t < NS; t++)
#pragma unroll
        for (int d = 0; d < 3; d++) acc[t][d] = abs_[t][d] = (AT)0;
    for (int32_t base = rb; base < re; base += 64) {
#pragma unroll
        for (int t = 0; t < NS; t++) {
            const int32_t k = base + sub + L * t;
            if (k < re) {
                const int64_t c = block_col<CT>(col, k, row);
                const auto *xc = gl(x) + c * 3;
                const AT x0 = (AT)xc[0], x1 = (AT)xc[1], x2 = (AT)xc[2];
                AT v[9];
                load_block<VT, AT>(vals, k, v);
                acc[t][0] = fma(v[2], x2, fma(v[1], x1, fma(v[0], x0, acc[t][0])));
                acc[t][1] = fma(v[5], x2, fma(v[4], x1, fma(v[3], x0, acc[t][1])));
                acc[t][2] = fma(v[8], x2, fma(v[7], x1, fma(v[6], x0, acc[t][2])));
                abs_[t][0] += fabs(v[0] * x0) + fabs(v[1] * x1) + fabs(v[2] * x2);
                abs_[t][1] += fabs(v[3] * x0) + fabs(v[4] * x1) + fabs(v[5] * x2);
                abs_[t][2] += fabs(v[6] * x0) + fabs(v[7] * x1) + fabs(v[8] * x2);
            }
        }
    }
#pragma unroll
    for (int off = 32; off >= L; off >>= 1) {
#pragma unroll
        for (int t = 0; t < off / L; t++)
#pragma unroll
            for (int d = 0; d < 3; d++) {
                acc[t][d] = acc[t][d] + acc[t + off / L][d];
                abs_[t][d] = abs_[t][d] + abs_[t + off / L][d];
            }
    }
#pragma unroll
    for (int d = 0; d < 3; d++) {
        AT u = acc[0][d], w = abs_[0][d];
#pragma unroll
        for (int off = L / 2; off > 0; off >>= 1) {
            u += __shfl_xor(u, off, L);
            w += __shfl_xor(w, off, L);
        }
        y[d] = u;
        a[d] = w;
    }
}

// Smallest power of two >= R: LDS reduction arrays are that long, zero
// padded, so the tree is the same fixed binary tree for any R.
__host__ __device__ inline int pow2ceil(int R)
{
    int p = 1;
    while (p < R) p <<= 1;
    return p;
}

// Fixed-order tree sum of R (power of two) LDS values; result in every thread.
__device__ inline double lds_tree_sum(double *s, int R)
{
    for (int h = R / 2; h > 0; h >>= 1) {
        for (int i = threadIdx.x; i < h; i += blockDim.x) s[i] = s[i] + s[i + h];
        __syncthreads();
    }
    const double t = s[0];
    __syncthreads();
    return t;
}

// lds_tree_sum's tree (R a power of two, 64 <= R <= 1024) done by the first
// wave alone, after the barrier that completes s: lane i reduces
// s[i + 64 m] over m in registers (the levels h >= 64, same pairs in the
// same order), then the levels h = 32..1 by shuffles.  The result is in lane
// 0; the other waves need not wait.
__device__ inline double wave_tree_sum(const double *s, int R)
{
    const int M = R / 64;
    double v[16];
#pragma unroll
    for (int m = 0; m < 16; m++) v[m] = m < M ? s[threadIdx.x + 64 * m] : 0.0;
#pragma unroll
    for (int H = 8; H > 0; H >>= 1)
        if (H < M)
#pragma unroll
            for (int m = 0; m < H; m++) v[m] = v[m] + v[m + H];
    double a = v[0];
#pragma unroll
    for (int h = 32; h > 0; h >>= 1) a = a + __shfl_down(a, h, 64);
    return a;
}

// Dynamic LDS layout of the row-tile kernels: R+1 row pointers, then up to
// four double arrays of pow2ceil(R) entries (sized for the largest R of the
// launch).
__device__ inline int32_t *tile_rowptr(char *sm) { return (int32_t *)sm; }
__device__ inline double *tile_dbl(char *sm, int R, int j)
{
    const int off = ((R + 1) * 4 + 15) & ~15;
    return (double *)(sm + off) + (int64_t)j * pow2ceil(R);
}

// Entry i of a launch's work list.  A step with one member needs none: the
// launch passes a null list and that member's descriptor, which takes one
// dependent load off the start of every workgroup (a pass through the kernels
// of a small model's iteration is a chain of such loads).
__device__ inline int2 list_entry(const int2 *__restrict__ l, int64_t i)
{
    return l ? l[i] : make_int2(0, (int)i);
}

// Loads written before this stay before it: the kernels of an iteration issue
// their first loads together with the control words and only then test them,
// and address past-the-end operands clamped instead of under a branch.  On
// small models a wave of these kernels waits for memory three quarters of its
// time, about 0.45 us per dependent load: this, DPP reductions and no work
// list together took an iteration of the HEX8 20x4x4 model from 14.6 to 12.0
// us, of the HEX20 64x7x8 one from 18.0 to 14.9.
#define AMR_ISSUED() asm volatile("" ::: "memory")

// Workgroups are dispatched round-robin over the 8 XCDs (workgroup b runs on
// XCD b % 8).  Entry t(b) gives each XCD one contiguous run of the work
// list, so the slice of x a run of row tiles gathers stays in that XCD's L2.
__device__ inline int64_t xcd_tile(int64_t b, int64_t G)
{
    const int64_t x = b & 7, i = b >> 3, q = G >> 3, rm = G & 7;
    return x * q + (x < rm ? x : rm) + i;
}

__device__ inline int load_rows(const int32_t *__restrict__ rowptr, int64_t nrows, int R, int64_t tile,
                                int32_t *srp, int64_t &r0)
{
    r0 = tile * R;
    const int nr = (int)std::min<int64_t>(R, nrows - r0);
    for (int i = threadIdx.x; i <= nr; i += blockDim.x) srp[i] = gl(rowptr)[r0 + i];
    __syncthreads();
    return nr;
}

// y = K x (mode 0) or mask .* (K x) (mode 1), FP64, one model
template <int L>
__global__ void __launch_bounds__(WGS) spmv_kernel(int64_t nrows, int R, const int32_t *__restrict__ rowptr,
                                                   const int32_t *__restrict__ col, const double *__restrict__ vals,
                                                   const double *__restrict__ x, double *__restrict__ y,
                                                   const double *__restrict__ mask, int mode)
{
    extern __shared__ __align__(16) char sm[];
    int32_t *srp = tile_rowptr(sm);
    int64_t r0;
    const int nr = load_rows(rowptr, nrows, R, xcd_tile(blockIdx.x, gridDim.x), srp, r0);
    constexpr int RPW = WGS / L;
    const int sub = threadIdx.x % L;
    for (int i = threadIdx.x / L; i < nr; i += RPW) {
        double yy[3];
        row_sum<L, false, double, double, double>(srp[i], srp[i + 1], sub, col, vals, x, yy);
        if (sub == 0) {
            const int64_t row = r0 + i;
            for (int d = 0; d < 3; d++)
                y[row * 3 + d] = (mode == 1 && mask[row * 3 + d] == 0.0) ? 0.0 : yy[d];
        }
    }
}

// rt = mask .* (b - K x) in FP64; per-tile partials ||rt||^2, ||b||^2,
// || |K||x| + |b| ||^2 and the drift ||rt - r||^2 (r: recursive residual)
template <int L>
__global__ void __launch_bounds__(WGS) residual_kernel(const SegDesc *__restrict__ D, const int2 *__restrict__ tl)
{
    const int2 te = tl[xcd_tile(blockIdx.x, gridDim.x)];
    const SegDesc &d = D[te.x];
    const int R = d.R;
    extern __shared__ __align__(16) char sm[];
    int32_t *srp = tile_rowptr(sm);
    double *s_rr = tile_dbl(sm, R, 0), *s_bb = tile_dbl(sm, R, 1), *s_kx = tile_dbl(sm, R, 2),
           *s_gap = tile_dbl(sm, R, 3);
    const int RP = pow2ceil(R);
    for (int i = threadIdx.x; i < RP; i += WGS) s_rr[i] = s_bb[i] = s_kx[i] = s_gap[i] = 0.0;
    int64_t r0;
    const int nr = load_rows(d.rowptr, d.nnodes, R, te.y, srp, r0);
    constexpr int RPW = WGS / L;
    const int sub = threadIdx.x % L;
    const auto *__restrict__ b = gl(d.b);
    const auto *__restrict__ mask = gl(d.mask);
    for (int i = threadIdx.x / L; i < nr; i += RPW) {
        double y[3], a[3];
        if (d.col16)
            row_sum_pair<L, double, double, double, int16_t>(srp[i], srp[i + 1], sub, d.col16, d.Kv, d.x, y, a,
                                                             r0 + i);
        else
            row_sum_pair<L, double, double, double>(srp[i], srp[i + 1], sub, d.col, d.Kv, d.x, y, a);
        if (sub == 0) {
            double rr = 0.0, bb = 0.0, kx = 0.0, gap = 0.0;
            for (int c = 0; c < 3; c++) {
                const int64_t k = (r0 + i) * 3 + c;
                const bool fr = mask[k] != 0.0;
                const double ri = fr ? b[k] - y[c] : 0.0;
                const double bi = fr ? b[k] : 0.0;
                const double ai = fr ? a[c] + fabs(b[k]) : 0.0;
                glw(d.rt)[k] = ri;
                rr = fma(ri, ri, rr);
                bb = fma(bi, bi, bb);
                kx = fma(ai, ai, kx);
                const double g = ri - gl(d.r)[k];
                gap = fma(g, g, gap);
            }
            s_rr[i] = rr;
            s_bb[i] = bb;
            s_kx[i] = kx;
            s_gap[i] = gap;
        }
    }
    __syncthreads();
    const double trr = lds_tree_sum(s_rr, RP), tbb = lds_tree_sum(s_bb, RP), tkx = lds_tree_sum(s_kx, RP),
                 tgap = lds_tree_sum(s_gap, RP);
    if (threadIdx.x == 0) {
        glw(d.part)[P_A + te.y] = trr;
        glw(d.part)[P_B + te.y] = tbb;
        glw(d.part)[P_C + te.y] = tkx;
        glw(d.part)[P_D + te.y] = tgap;
    }
}

// ------------------------------------------------------------------- PCG
//
// Iteration k of a model (parity pi = k % 2), three kernels; without a coarse
// correction the first forms the direction as it gathers (matrix-free members
// and small assembled ones) and pcg_dir is not launched:
//   pcg_spmv / pcg_mf: q = A p, partial p.q                   -> P_PQ
//   pcg_update: a = rz_k / pq; x += a p; r -= a q; z = M r;
//               partials rz_{k+1}, rr                         -> P_RZ[pi], P_RR[pi]
//   pcg_dir:    b = rz_{k+1} / rz_k; p = z + b p; convergence test;
//               publishes rz_{k+1} in scalar slot rz_pub(pi)
// rz_k is the sum of P_RZ[1-pi], published in rz_pub(1-pi) by iteration
// k-1's pcg_dir, by the initialisation or by a residual replacement.

template <typename VT>
__device__ inline const VT *seg_vals(const SegDesc &d);
template <>
__device__ inline const double *seg_vals<double>(const SegDesc &d) { return d.Kv; }
template <>
__device__ inline const float *seg_vals<float>(const SegDesc &d) { return d.Kv32; }
template <typename XT>
__device__ inline const XT *seg_px(const SegDesc &d);
template <>
__device__ inline const double *seg_px<double>(const SegDesc &d) { return d.p; }
template <>
__device__ inline const float *seg_px<float>(const SegDesc &d) { return d.p32; }

// FUSE (small models without a coarse correction): the kernel gathers
// p = z + beta p as pcg_mf_kernel does, with its bookkeeping; pcg_update stores
// it.  For the gather's second vector an iteration saves the direction's
// launch (about 5 us).
template <int L, typename VT, typename XT, typename AT, bool FUSE>
__global__ void __launch_bounds__(WGS) pcg_spmv_kernel(const SegDesc *__restrict__ D, const int2 *__restrict__ tl,
                                                       int first)
{
    const int2 te = list_entry(tl, xcd_tile(blockIdx.x, gridDim.x));
    if (te.x < 0) return;  // padding of a captured step's list
    const SegDesc &d = D[te.x];
    auto *ctl = glw(d.ctl);
    if (ctl[C_DONE]) return;
    if (ctl[C_STOP]) {
        // converged in the previous iteration: every workgroup leaves, and
        // the first tile raises C_DONE for the kernels that follow
        if (te.y == 0 && threadIdx.x == 0) ctl[C_DONE] = 1;
        return;
    }
    // the step's first iteration takes p as it is: p + 0 p
    const double *z = FUSE && !first ? d.z : d.p;
    double beta = 0.0;
    if (FUSE && !first) {
        const int it = ctl[C_PREV], pi = (it - 1) & 1;
        const double rzt = thread_partials<WGS>(d.part + (pi ? P_RZ1 : P_RZ0), d.nred);
        const double rrt = te.y == 0 ? thread_partials<WGS>(d.part + (pi ? P_RR1 : P_RR0), d.nred) : 0.0;
        const double rzn = block_sum<WGS>(rzt);
        beta = rzn / glw(d.scal)[rz_pub(1 - pi)];
        if (te.y == 0) {
            const double rr = block_sum<WGS>(rrt);
            if (threadIdx.x == 0) {
                glw(d.scal)[S_RR] = rr;
                glw(d.scal)[S_RZ] = rzn;
                glw(d.scal)[rz_pub(pi)] = rzn;
                glw(d.scal)[S_BETA] = beta;
                if (rr <= glw(d.scal)[S_THR] || it >= d.maxiter || !std::isfinite(rr)) ctl[C_STOP] = 1;
                else ctl[C_ITERS] = it + 1;
            }
        }
    } else if (te.y == 0 && threadIdx.x == 0) {
        ctl[C_ITERS] = (FUSE ? ctl[C_PREV] : ctl[C_ITERS]) + 1;
    }
    const int R = d.R;
    extern __shared__ __align__(16) char sm[];
    int32_t *srp = tile_rowptr(sm);
    double *sdot = tile_dbl(sm, R, 0);
    static_assert(sizeof(AT) >= sizeof(VT), "accumulate at least in the storage precision");
    const int RP = pow2ceil(R);
    for (int i = threadIdx.x; i < RP; i += WGS) sdot[i] = 0.0;
    int64_t r0;
    const int nr = load_rows(d.rowptr, d.nnodes, R, te.y, srp, r0);
    constexpr int RPW = WGS / L;
    const int sub = threadIdx.x % L;
    const VT *vals = seg_vals<VT>(d);
    const XT *px = seg_px<XT>(d);
    for (int i = threadIdx.x / L; i < nr; i += RPW) {
        // lanes 0..2 of the row group fetch the row's mask and p entries
        // before its blocks, so the row's tail waits on no load
        const int64_t k3 = (r0 + i) * 3 + (sub < 3 ? sub : 0);
        double mk = 0.0, pk = 0.0;
        if (sub < 3) {
            mk = gl(d.mask)[k3];
            pk = gl(d.p)[k3];
            if (FUSE) pk = fma(beta, pk, gl(z)[k3]);
        }
        AT y[3];
        if (d.col16)
            row_sum<L, false, VT, XT, AT, int16_t, FUSE>(srp[i], srp[i + 1], sub, d.col16, vals, px, y, r0 + i, z, beta);
        else
            row_sum<L, false, VT, XT, AT, int32_t, FUSE>(srp[i], srp[i + 1], sub, d.col, vals, px, y, 0, z, beta);
        // lane e < 3 stores q of component e; lane 0 forms the row's p.q,
        // fma(p2, q2, fma(p1, q1, fma(p0, q0, 0)))
        const double qk = mk != 0.0 ? (double)(sub == 0 ? y[0] : sub == 1 ? y[1] : y[2]) : 0.0;
        if (sub < 3) glw(d.q)[k3] = qk;
        const double q1 = __shfl_down(qk, 1, L), q2 = __shfl_down(qk, 2, L);
        const double p1 = __shfl_down(pk, 1, L), p2 = __shfl_down(pk, 2, L);
        if (sub == 0) sdot[i] = fma(p2, q2, fma(p1, q1, fma(pk, qk, 0.0)));
    }
    __syncthreads();
    if (RP <= 1024) {
        if (threadIdx.x < 64) {
            const double pq = wave_tree_sum(sdot, RP);
            if (threadIdx.x == 0) glw(d.part)[P_PQ + te.y] = pq;
        }
    } else {
        const double pq = lds_tree_sum(sdot, RP);
        if (threadIdx.x == 0) glw(d.part)[P_PQ + te.y] = pq;
    }
}

// ------------------------------------------------- matrix-free operator
//
// f_e = Be' (coef De) Be p_e for the elements of a tile and the tile's partial
// of p.q = sum_e p_e . f_e (p is 0 at prescribed dofs); pcg_update sums the f_e
// of each node into q.  One wave per group of 16 elements (lane l = 16 g + c:
// element c, node slots 4 s + g, IP slots 4 k + g; see matrix_free.hip).  Per
// IP slot: H = du/dR by FP64 matrix instructions (inner dimension the nodes),
// sigma and P = A' sigma in registers, f += B' P by matrix instructions (inner
// dimension the IPs).  Every intermediate stays in the lane that needs it.
//
// With d.fuse (no coarse correction) and first == 0 the kernel forms the
// direction itself, p = z + beta p with the rounding of pcg_dir_kernel: a
// node's p is gathered by the few elements around it, so forming it in the
// gather costs less than a kernel of its own; pcg_update stores it.  The
// first tile then does pcg_dir_kernel's bookkeeping.
//
// Bound on the 40^3 HEX20 block (27 IPs, 64,000 elements) by memory: 35 us a
// launch, in which 144 MB are read (72 B of geometry per IP, most of it) and
// 31 MB written past the L2, 5.0 TB/s, the rate of a 1 GiB copy; the matrix
// cores are busy 55% of its cycles (630 v_mfma_f64_4x4x4 per group, 16 cycles
// each), without LDS bank conflicts.  In small models by one wave's chain (see
// mf_geom).  The 4x4x4 form is used because its operand and result lanes agree
// (no exchange) and its rows need no padding to 16; measured alone it reaches
// 68 TFLOP/s here against 43 for 16x16x4.  Medians of a kernel trace, and of
// the SpMV on the assembled matrix with FP32 and with FP64 values: the block 35
// us against 142 and 235; HEX20 17x19x15 10.9 against 15.8 and 20.9; HEX20
// 64x7x8 with 8 IPs 6.2 against 16.1 and 21.2; HEX8 83x21x20 9.2 against 12.8
// and 18.2; TET10 49x12x13 10.3 against 22.6 and 33.3 us.
template <int NN, int NQ>
struct MfShape {
    static constexpr int NS = (NN + 3) / 4, KS = (NQ + 3) / 4, HALF = KS * 3 * NS * 16;
};

template <int NN, int NQ, int W>
__global__ void __launch_bounds__(256, 2) pcg_mf_kernel(const SegDesc *__restrict__ D, const int2 *__restrict__ tl,
                                                        int first)
{
    using S = MfShape<NN, NQ>;
    constexpr int NS = S::NS, KS = S::KS;
    const int2 te = list_entry(tl, xcd_tile(blockIdx.x, gridDim.x));
    if (te.x < 0) return;
    const SegDesc d = D[te.x];
    auto *ctl = glw(d.ctl);
    __shared__ __align__(16) double sT[2 * S::HALF];
    const bool fuse = d.fuse && !first;
    // W waves share a group, each with the IP slots sub, sub + W, ...
    constexpr int NG = 4 / W;
    __shared__ double sF[W > 1 ? 4 : 1][W > 1 ? NS * 192 : 1];
    __shared__ double sU[W > 1 ? NG : 1][W > 1 ? NS * 192 : 1];
    constexpr int NW = (NS + W - 1) / W;  // node slots gathered by a wave: sub, sub + W, ...
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, sub = wave % W;
    const auto *__restrict__ p = gl(d.p);
    // (p again, unused, where the direction is already formed)
    const auto *__restrict__ z = fuse ? gl(d.z) : gl(d.p);
    const int64_t g0 = (int64_t)te.y * NG * d.mfG + wave / W;
    const auto *mfconn = gl(d.mfconn);
    const int done = ctl[C_DONE], stop = ctl[C_STOP], it = ctl[C_PREV];
    int32_t nd[NW];
    double u[NS][3], pv[NW][3], zv[NW][3], f[NS][3];
    auto load_nodes = [&](int64_t grp) {
#pragma unroll
        for (int t = 0; t < NW; t++) {
            const int s = sub + W * t;
            nd[t] = mfconn[(grp * NS + (s < NS ? s : 0)) * 64 + lane];
        }
    };
    auto gather = [&]() {
#pragma unroll
        for (int t = 0; t < NW; t++)
#pragma unroll
            for (int c = 0; c < 3; c++) {
                pv[t][c] = p[(int64_t)nd[t] * 3 + c];
                zv[t][c] = z[(int64_t)nd[t] * 3 + c];
            }
    };
    // the geometry of an IP slot is loaded one slot ahead where waves share a
    // group; with a group per wave the registers cost more than it hides (HEX20
    // with 27 IPs, 40^3 block: 34.4 against 32.9 us)
    constexpr bool AHEAD = W > 1;
    double An[9];
    auto load_geo = [&](int64_t grp, int k) {
        const auto *geo = gl(d.geo) + (grp * KS + k) * 576 + lane;
#pragma unroll
        for (int r = 0; r < 9; r++) An[r] = geo[r * 64];
    };
    // first loads: the first group's nodes and geometry, the tables, the shares of the r.z
    // (and, first tile, r.r) partials of both parity slots
    load_nodes(g0 < d.ngrp ? g0 : 0);
    if (AHEAD) load_geo(g0 < d.ngrp ? g0 : 0, sub);
    constexpr int NT2 = (S::HALF + 255) / 256;  // 16-byte table loads per thread
    f64x2 tb[NT2];
#pragma unroll
    for (int k = 0; k < NT2; k++) {
        const int i = (int)threadIdx.x + k * 256;
        tb[k] = gl((const f64x2 *)d.tab)[i < S::HALF ? i : 0];
    }
    double rzs[2] = {0.0, 0.0}, rrs[2] = {0.0, 0.0}, rzp[2] = {0.0, 0.0}, thr = 0.0;
    if (fuse) {
        rzs[0] = thread_partials<256>(d.part + P_RZ0, d.nred);
        rzs[1] = thread_partials<256>(d.part + P_RZ1, d.nred);
        rzp[0] = glw(d.scal)[S_RZP0];
        rzp[1] = glw(d.scal)[S_RZP1];
        if (te.y == 0) {
            rrs[0] = thread_partials<256>(d.part + P_RR0, d.nred);
            rrs[1] = thread_partials<256>(d.part + P_RR1, d.nred);
            thr = glw(d.scal)[S_THR];
        }
    }
    AMR_ISSUED();
    if (done) return;
    if (stop) {
        if (te.y == 0 && threadIdx.x == 0) ctl[C_DONE] = 1;
        return;
    }
    gather();
#pragma unroll
    for (int k = 0; k < NT2; k++) {
        const int i = (int)threadIdx.x + k * 256;
        if (i < S::HALF) ((f64x2 *)sT)[i] = tb[k];
    }
    double beta = 0.0;
    if (fuse) {
        const int pi = (it - 1) & 1;
        const double rzn = block_sum<256>(pi ? rzs[1] : rzs[0]);
        beta = rzn / (pi ? rzp[0] : rzp[1]);
        if (te.y == 0) {
            const double rr = block_sum<256>(pi ? rrs[1] : rrs[0]);
            if (threadIdx.x == 0) {
                glw(d.scal)[S_RR] = rr;
                glw(d.scal)[S_RZ] = rzn;
                glw(d.scal)[rz_pub(pi)] = rzn;
                glw(d.scal)[S_BETA] = beta;
                // stopped: the update kernel of this iteration does nothing
                if (rr <= thr || it >= d.maxiter || !std::isfinite(rr)) ctl[C_STOP] = 1;
                else ctl[C_ITERS] = it + 1;
            }
        }
    } else if (te.y == 0 && threadIdx.x == 0) {
        ctl[C_ITERS] = it + 1;
    }
    __syncthreads();
    double pq = 0.0;
    for (int w = 0; w < d.mfG; w++) {
        const int64_t grp = g0 + NG * w;
        if (W == 1 && grp >= d.ngrp) break;  // (a shared group's waves meet at a barrier; mfG is 1 there)
        if (W == 1 && w > 0) {
            load_nodes(grp);
            gather();
        }
        // the waves of a shared group each gathered some of its nodes (the
        // scattered loads are the L1's work, one line per lane)
        double *su = sU[W > 1 ? wave / W : 0];
#pragma unroll
        for (int t = 0; t < NW; t++)
#pragma unroll
            for (int c = 0; c < 3; c++) {
                const double v = fuse ? fma(beta, pv[t][c], zv[t][c]) : pv[t][c];
                if (W == 1) u[t][c] = v;
                else if (sub + W * t < NS) su[((sub + W * t) * 3 + c) * 64 + lane] = v;
            }
        if (W > 1) __syncthreads();
#pragma unroll
        for (int s = 0; s < NS; s++)
#pragma unroll
            for (int c = 0; c < 3; c++) {
                if (W > 1) u[s][c] = su[(s * 3 + c) * 64 + lane];
                f[s][c] = 0.0;
            }
        const auto *lmp = gl(d.lm) + (grp < d.ngrp ? grp : 0) * 32 + (lane & 15);
        const double lam = lmp[0], mu = lmp[16];
#pragma unroll 1
        for (int k = sub; k < KS; k += W) {
            double A[3][3], H[3][3];
            if (!AHEAD) load_geo(grp, k);
#pragma unroll
            for (int r = 0; r < 9; r++) A[r / 3][r % 3] = An[r];
            if (AHEAD && k + W < KS) load_geo(grp < d.ngrp ? grp : 0, k + W);
            const double *t1 = sT + k * (3 * NS * 16) + (lane & 3) + 4 * (lane >> 4);
#pragma unroll
            for (int j = 0; j < 3; j++) {
#pragma unroll
                for (int c = 0; c < 3; c++) H[c][j] = 0.0;
#pragma unroll
                for (int s = 0; s < NS; s++) {
                    const double a = t1[(j * NS + s) * 16];
#pragma unroll
                    for (int c = 0; c < 3; c++)
                        H[c][j] = __builtin_amdgcn_mfma_f64_4x4x4f64(a, u[s][c], H[c][j], 0, 0, 0);
                }
            }
            // G = H A (du_c/dX_m), sigma = lambda tr I + mu (G + G'), P = sigma A'
            double G[3][3], P[3][3];
#pragma unroll
            for (int c = 0; c < 3; c++)
#pragma unroll
                for (int m = 0; m < 3; m++) G[c][m] = fma(H[c][2], A[2][m], fma(H[c][1], A[1][m], H[c][0] * A[0][m]));
            const double lt = lam * (G[0][0] + G[1][1] + G[2][2]);
            const double s00 = fma(2.0 * mu, G[0][0], lt), s11 = fma(2.0 * mu, G[1][1], lt),
                         s22 = fma(2.0 * mu, G[2][2], lt);
            const double s12 = mu * (G[1][2] + G[2][1]), s02 = mu * (G[0][2] + G[2][0]), s01 = mu * (G[0][1] + G[1][0]);
#pragma unroll
            for (int j = 0; j < 3; j++) {
                P[0][j] = fma(s02, A[j][2], fma(s01, A[j][1], s00 * A[j][0]));
                P[1][j] = fma(s12, A[j][2], fma(s11, A[j][1], s01 * A[j][0]));
                P[2][j] = fma(s22, A[j][2], fma(s12, A[j][1], s02 * A[j][0]));
            }
            const double *t2 = t1 + S::HALF;
#pragma unroll
            for (int j = 0; j < 3; j++)
#pragma unroll
                for (int s = 0; s < NS; s++) {
                    const double a = t2[(j * NS + s) * 16];
#pragma unroll
                    for (int c = 0; c < 3; c++)
                        f[s][c] = __builtin_amdgcn_mfma_f64_4x4x4f64(a, P[c][j], f[s][c], 0, 0, 0);
                }
        }
        auto *o = glw(d.mff) + grp * (NS * 192) + lane;
#pragma unroll
        for (int s = 0; s < NS; s++)
#pragma unroll
            for (int c = 0; c < 3; c++) {
                if (W == 1) o[(s * 3 + c) * 64] = f[s][c];
                else sF[wave][(s * 3 + c) * 64 + lane] = f[s][c];
                if (W == 1 || grp < d.ngrp) pq = fma(u[s][c], f[s][c], pq);
            }
        if (W > 1) {
            // the group's waves add their parts, a row of 64 each in turn
            __syncthreads();
            if (grp < d.ngrp)
                for (int r = sub; r < NS * 3; r += W) {
                    double v = sF[wave - sub][r * 64 + lane];
#pragma unroll
                    for (int x = 1; x < W; x++) v += sF[wave - sub + x][r * 64 + lane];
                    o[r * 64] = v;
                }
        }
    }
    pq = block_sum<256>(pq);
    if (threadIdx.x == 0) glw(d.part)[P_PQ + te.y] = pq;
}

// q of a node: its elements' products in element order, 0 at prescribed
// dofs.  b: the node's record (matrix_free.hip), its first eight products'
// places (-1: none); a ninth one and later ones come from the incidence list.
__device__ inline void mf_load_q(const SegDesc &d, const int32_t b[8], double v[8][3])
{
    const auto *f = gl(d.mff);
#pragma unroll
    for (int j = 0; j < 8; j++)
#pragma unroll
        for (int c = 0; c < 3; c++) v[j][c] = f[(b[j] >= 0 ? b[j] : 0) + 64 * c];
}

__device__ inline void mf_sum_q(const SegDesc &d, int64_t nd, const int32_t b[8], double v[8][3], const double m[3],
                                double q[3])
{
    double a[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int j = 0; j < 8; j++)
#pragma unroll
        for (int c = 0; c < 3; c++) a[c] = b[j] >= 0 ? a[c] + v[j][c] : a[c];
    if (b[7] >= 0) {
        const auto *f = gl(d.mff);
        const auto *fp = gl(d.fptr), *src = gl(d.mfsrc);
        const int32_t k1 = fp[nd + 1];
        // eight at a time: a corner node of tetrahedra has up to 24
        for (int32_t k = fp[nd] + 8; k < k1; k += 8) {
            int32_t e[8];
#pragma unroll
            for (int j = 0; j < 8; j++) e[j] = src[k + j < k1 ? k + j : k];
#pragma unroll
            for (int j = 0; j < 8; j++)
#pragma unroll
                for (int c = 0; c < 3; c++) v[j][c] = f[e[j] + 64 * c];
#pragma unroll
            for (int j = 0; j < 8; j++)
#pragma unroll
                for (int c = 0; c < 3; c++) a[c] = k + j < k1 ? a[c] + v[j][c] : a[c];
        }
    }
    for (int c = 0; c < 3; c++) q[c] = m[c] != 0.0 ? a[c] : 0.0;
}

// MF: members on the matrix-free operator (q summed from its element
// products); the others read the SpMV's q.  TL: two-level members on an
// assembled matrix; a workgroup takes a chunk of an aggregate's nodes and also
// writes the chunk's part of c = Phi^T r, while r is in registers (a kernel of
// its own for it read r and X again: 3.7 us of a 36 us iteration on the
// 40x40x20 footing).
// FZ: members on an assembled matrix whose SpMV forms the direction.
template <bool MF, bool TL, bool FZ>
__global__ void __launch_bounds__(WGV) pcg_update_kernel(const SegDesc *__restrict__ D, const int2 *__restrict__ vl,
                                                         int first)
{
    const int2 ve = list_entry(vl, blockIdx.x);
    if (ve.x < 0) return;
    const SegDesc d = D[ve.x];
    auto *ctl = glw(d.ctl);
    constexpr bool FUSE = MF || FZ;  // the operator may form the direction
    const bool fuse = FUSE && d.fuse && !first;
    const int done = ctl[C_DONE], stop = FUSE ? (int)ctl[C_STOP] : 0, iters = ctl[C_ITERS];
    const int pi = (iters - 1) & 1;
    auto *__restrict__ x = glw(d.x);
    auto *__restrict__ r = glw(d.r);
    // (no __restrict__: where the direction is formed, z and p are read through
    // zs and written here)
    auto *z = glw(d.z);
    auto *p = glw(d.p);
    const auto *__restrict__ q = gl(d.q);
    const double beta = FUSE ? (double)glw(d.scal)[S_BETA] : 0.0;
    const double rzp0 = glw(d.scal)[S_RZP0], rzp1 = glw(d.scal)[S_RZP1];
    // z is read where the direction is formed here (else p again, unused, so
    // that the loads need no branch)
    const auto *zs = fuse ? gl(d.z) : gl(d.p);
    // a node's operands; with MF also its record and mask, from which
    // mf_load_q and mf_sum_q gather q
    struct Node {
        double p[3], q[3], x[3], r[3], z[3], m[3], X[3];
        int32_t b[8];
    };
    auto load_node = [&](int64_t n, Node &v) {
        for (int c = 0; c < 3; c++) {
            v.p[c] = p[n * 3 + c];
            if (FUSE) v.z[c] = zs[n * 3 + c];
            v.x[c] = x[n * 3 + c];
            v.r[c] = r[n * 3 + c];
            if (MF) v.m[c] = gl(d.mask)[n * 3 + c];
            else v.q[c] = q[n * 3 + c];
            if (TL) v.X[c] = gl(d.X)[n * 3 + c];
        }
        if (MF) {
            const auto *b = gl((const i32x4 *)d.mfrec) + 2 * n;
            const i32x4 b0 = b[0], b1 = b[1];
            for (int j = 0; j < 4; j++) {
                v.b[j] = b0[j];
                v.b[4 + j] = b1[j];
            }
        }
    };
    // the first node's operands are loaded before the control words are tested
    // and the partials are summed, so that their latencies overlap
    // positions first + thread, + stride, ... below end: nodes, or places in
    // the aggregate-ordered node list
    i32x4 ch = {0, 0, 0, 0};
    if (TL) ch = gl(d.chunk)[ve.y];
    const int64_t stride = TL ? WGV : (int64_t)d.nvblk * WGV, end = TL ? ch.y : d.nnodes;
    int64_t pos = (TL ? (int64_t)ch.x : (int64_t)ve.y * WGV) + threadIdx.x;
    auto node_at = [&](int64_t k) { return TL ? (int64_t)gl(d.aggnodes)[k] : k; };
    Node v = {};
    int64_t nd = node_at(pos < end ? pos : end - 1);
    load_node(nd, v);
    AMR_ISSUED();
    if (done) return;
    if (FUSE && stop) {
        // converged before this iteration (seen by the operator's first tile)
        if (ve.y == 0 && threadIdx.x == 0) ctl[C_DONE] = 1;
        return;
    }
    if (FUSE && ve.y == 0 && threadIdx.x == 0) ctl[C_PREV] = iters;
    double fv[8][3];
    if (MF) mf_load_q(d, v.b, fv);
    const double pqt = thread_partials<WGV>(d.part + P_PQ, d.npq);
    AMR_ISSUED();
    if (MF) mf_sum_q(d, nd, v.b, fv, v.m, v.q);
    const double pq = block_sum<WGV>(pqt);
    const double rz = pi ? rzp0 : rzp1;
    if (!(pq > 0.0) || !std::isfinite(pq)) {
        if (ve.y == 0 && threadIdx.x == 0) {
            ctl[C_BREAK] = 1;
            ctl[C_DONE] = 1;
        }
        return;
    }
    const double a = rz / pq;
    double rzn = 0.0, rr = 0.0, cp[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, cen[3] = {0.0, 0.0, 0.0};
    if (TL)
        for (int c = 0; c < 3; c++) cen[c] = gl(d.cent)[ch.z * 3 + c];
    // one node per pass; the dot contributions in node order
    while (pos < end) {
        double rv[3], zv[3];
        for (int c = 0; c < 3; c++) {
            const int64_t i = nd * 3 + c;
            if (fuse) {
                v.p[c] = fma(beta, v.p[c], v.z[c]);
                p[i] = v.p[c];
            }
            x[i] = fma(a, v.p[c], v.x[c]);
            rv[c] = fma(-a, v.q[c], v.r[c]);
            r[i] = rv[c];
        }
        apply_prec(d, nd, rv, zv);
        for (int c = 0; c < 3; c++) {
            z[nd * 3 + c] = zv[c];
            rzn = fma(rv[c], zv[c], rzn);
            rr = fma(rv[c], rv[c], rr);
        }
        if (TL) {
            const double dx = v.X[0] - cen[0], dy = v.X[1] - cen[1], dz = v.X[2] - cen[2];
            cp[0] += rv[0];
            cp[1] += rv[1];
            cp[2] += rv[2];
            cp[3] += fma(dy, rv[2], -dz * rv[1]);
            cp[4] += fma(dz, rv[0], -dx * rv[2]);
            cp[5] += fma(dx, rv[1], -dy * rv[0]);
        }
        pos += stride;
        if (pos < end) {
            nd = node_at(pos);
            load_node(nd, v);
            if (MF) {
                mf_load_q(d, v.b, fv);
                mf_sum_q(d, nd, v.b, fv, v.m, v.q);
            }
        }
    }
    // thread 0 writes the r.z partial, 1 the r.r one, 2..7 the part of c
    constexpr int NSUM = TL ? 8 : 2;
    double sums[NSUM];
    sums[0] = rzn;
    sums[1] = rr;
    if (TL)
        for (int c = 0; c < 6; c++) sums[2 + c] = cp[c];
    const double t = block_sums<WGV, NSUM>(sums);
    if (threadIdx.x == 0) glw(d.part)[(pi ? P_RZ1 : P_RZ0) + ve.y] = t;
    else if (threadIdx.x == 1) glw(d.part)[(pi ? P_RR1 : P_RR0) + ve.y] = t;
    else if (TL && threadIdx.x < 8) glw(d.cpart)[(int64_t)ve.y * 6 + threadIdx.x - 2] = t;
}

// p = z + beta p, for two-level members p = z + Phi y + beta p: a workgroup
// takes a chunk of an aggregate's nodes, so that y and the centroid are the
// same for all of them (per dof with the aggregate looked up: 12.9 us on the
// 40^3 HEX20 block).
template <bool TL>
__global__ void __launch_bounds__(WGV) pcg_dir_kernel(const SegDesc *__restrict__ D, const int2 *__restrict__ vl)
{
    const int2 ve = list_entry(vl, blockIdx.x);
    if (ve.x < 0) return;
    const SegDesc d = D[ve.x];
    auto *ctl = glw(d.ctl);
    const int done = ctl[C_DONE], it = ctl[C_ITERS], pi = (it - 1) & 1;
    auto *__restrict__ p = glw(d.p);
    auto *__restrict__ p32 = d.wp32 ? glw(d.p32) : nullptr;
    const auto *__restrict__ z = gl(d.z);
    // non-TL: one dof per pass; TL: one node per pass
    constexpr int NC = TL ? 3 : 1;
    i32x4 ch = {0, 0, 0, 0};
    if (TL) ch = gl(d.chunk)[ve.y];
    const int64_t stride = TL ? WGV : (int64_t)d.nvblk * WGV, end = TL ? (int64_t)ch.y : d.nnodes * 3;
    int64_t pos = (TL ? (int64_t)ch.x : (int64_t)ve.y * WGV) + threadIdx.x;
    double pv[NC], zv[NC], X[NC], mk[NC];
    int64_t i0 = 0;
    auto load = [&](int64_t k) {
        i0 = TL ? (int64_t)gl(d.aggnodes)[k] * 3 : k;
#pragma unroll
        for (int c = 0; c < NC; c++) {
            pv[c] = p[i0 + c];
            zv[c] = z[i0 + c];
            X[c] = TL ? gl(d.X)[i0 + c] : 0.0;
            mk[c] = TL ? gl(d.mask)[i0 + c] : 0.0;
        }
    };
    // the first operands, the aggregate's correction, the shares of both
    // parity slots' partials and the published r.z
    load(pos < end ? pos : end - 1);
    double y[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, cen[3] = {0.0, 0.0, 0.0};
    if (TL) {
        for (int c = 0; c < 6; c++) y[c] = gl(d.yvec)[(int64_t)ch.z * 6 + c];
        for (int c = 0; c < 3; c++) cen[c] = gl(d.cent)[ch.z * 3 + c];
    }
    double rzs[2], rrs[2] = {0.0, 0.0};
    rzs[0] = thread_partials<WGV>(d.part + P_RZ0, d.nred);
    rzs[1] = thread_partials<WGV>(d.part + P_RZ1, d.nred);
    if (TL) {
        rzs[0] += thread_partials<WGV>(d.part + P_CY0, d.ncw);
        rzs[1] += thread_partials<WGV>(d.part + P_CY1, d.ncw);
    }
    if (ve.y == 0) {
        rrs[0] = thread_partials<WGV>(d.part + P_RR0, d.nred);
        rrs[1] = thread_partials<WGV>(d.part + P_RR1, d.nred);
    }
    const double rzp0 = glw(d.scal)[S_RZP0], rzp1 = glw(d.scal)[S_RZP1], thr = glw(d.scal)[S_THR];
    AMR_ISSUED();
    if (done) return;
    // rz of the previous iteration was published in the other parity slot;
    // the first workgroup publishes this one's and tests convergence
    const double rzn = block_sum<WGV>(pi ? rzs[1] : rzs[0]);
    const double beta = rzn / (pi ? rzp0 : rzp1);
    if (ve.y == 0) {
        const double rr = block_sum<WGV>(pi ? rrs[1] : rrs[0]);
        if (threadIdx.x == 0) {
            glw(d.scal)[S_RR] = rr;
            glw(d.scal)[S_RZ] = rzn;
            glw(d.scal)[rz_pub(pi)] = rzn;
            if (rr <= thr || it >= d.maxiter || !std::isfinite(rr)) ctl[C_STOP] = 1;
        }
    }
    while (pos < end) {
        if (TL) {
            // Phi y at the node (coarse_term)
            const double dx = X[0] - cen[0], dy = X[NC - 2] - cen[1], dz = X[NC - 1] - cen[2];
            const double t[3] = {fma(-dy, y[5], fma(dz, y[4], y[0])), fma(dx, y[5], fma(-dz, y[3], y[1])),
                                 fma(-dx, y[4], fma(dy, y[3], y[2]))};
#pragma unroll
            for (int c = 0; c < NC; c++) zv[c] += mk[c] != 0.0 ? t[c] : 0.0;
        }
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const double pn = fma(beta, pv[c], zv[c]);
            p[i0 + c] = pn;
            if (p32) p32[i0 + c] = (float)pn;
        }
        pos += stride;
        if (pos < end) load(pos);
    }
}

// Two-level pieces, for the members with d.tl (mode 0: inside the iteration,
// skipped once the member is done; mode 1: initialisation and resume)
//   restrict: c_a = sum_{i in a} R_i^T r_i, four waves per aggregate (inside
//             an iteration only for the members whose update kernel does not
//             write c's parts)
//   coarse:   y = Kc^-1 c, one wave per coarse row, and partials of c.y
//   prolong:  p = z + Phi y (start of a search direction)
constexpr int WGR = 256;  // restriction
__global__ void __launch_bounds__(WGR) tl_restrict_kernel(const SegDesc *__restrict__ D, const int2 *__restrict__ al,
                                                         int mode)
{
    const int2 e = list_entry(al, blockIdx.x);
    if (e.x < 0) return;
    const SegDesc d = D[e.x];
    const int done = mode == 0 ? (int)glw(d.ctl)[C_DONE] : 0;
    const int32_t a = e.y;
    const auto *cent = gl(d.cent), *X = gl(d.X), *rv = gl(d.r);
    const auto *aggptr = gl(d.aggptr), *aggnodes = gl(d.aggnodes);
    const double cx = cent[a * 3], cy = cent[a * 3 + 1], cz = cent[a * 3 + 2];
    double v[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    // a thread's nodes k = k0 + tid + 256 j in order of j, eight at a time:
    // the eight nodes' loads are issued before their sums.  Bound by that chain
    // of loads: on 256 aggregates of 1,057 nodes one wave each took 9.9 us, four
    // take 6.6; with 261 nodes in each a TET10 step went from 7.43 to 7.30 ms
    constexpr int NB = 8;
    const int32_t k0 = aggptr[a], k1 = aggptr[a + 1];
    AMR_ISSUED();
    if (done) return;
    for (int32_t kb = k0 + (int32_t)threadIdx.x; kb < k1; kb += WGR * NB) {
        int64_t nd[NB];
#pragma unroll
        for (int j = 0; j < NB; j++) nd[j] = kb + WGR * j < k1 ? aggnodes[kb + WGR * j] : -1;
        double r[NB][3], x[NB][3];
#pragma unroll
        for (int j = 0; j < NB; j++)
            if (nd[j] >= 0)
                for (int c = 0; c < 3; c++) {
                    r[j][c] = rv[nd[j] * 3 + c];
                    x[j][c] = X[nd[j] * 3 + c];
                }
#pragma unroll
        for (int j = 0; j < NB; j++)
            if (nd[j] >= 0) {
                const double r0 = r[j][0], r1 = r[j][1], r2 = r[j][2];
                const double dx = x[j][0] - cx, dy = x[j][1] - cy, dz = x[j][2] - cz;
                v[0] += r0;
                v[1] += r1;
                v[2] += r2;
                v[3] += fma(dy, r2, -dz * r1);
                v[4] += fma(dz, r0, -dx * r2);
                v[5] += fma(dx, r1, -dy * r0);
            }
    }
    __shared__ double s[6][WGR / 64];
    for (int q = 0; q < 6; q++) {
        const double t = wave_sum(v[q]);
        if (threadIdx.x % 64 == 0) s[q][threadIdx.x / 64] = t;
    }
    __syncthreads();
    const int q = threadIdx.x;
    if (q < 6) glw(d.cvec)[a * 6 + q] = (s[q][0] + s[q][1]) + (s[q][2] + s[q][3]);
}

__global__ void __launch_bounds__(256) tl_coarse_kernel(const SegDesc *__restrict__ D, const int2 *__restrict__ wl,
                                                        int mode)
{
    const int2 e = list_entry(wl, blockIdx.x);
    if (e.x < 0) return;
    const SegDesc d = D[e.x];
    const int done = mode == 0 ? (int)glw(d.ctl)[C_DONE] : 0;
    const int pi = (glw(d.ctl)[C_ITERS] - 1) & 1;
    const int row = e.y * 4 + (int)(threadIdx.x / 64), lane = threadIdx.x % 64;
    // columns lane + 64 j in order of j; the first sixteen entries of the row
    // and the workgroup's share of c are in flight together (c staged in LDS
    // ahead of the row's loads took the kernel from 6.0 to 7.7 us on 1,020
    // coarse dofs)
    constexpr int NB = 16, NCV = MAX_CW * 4 / 256;
    const auto *Kr = gl(d.Kinv) + (int64_t)(row < d.nc ? row : 0) * d.nc;
    double kv[NB], cs[NCV];
#pragma unroll
    for (int j = 0; j < NB; j++) kv[j] = Kr[lane + 64 * j < d.nc ? lane + 64 * j : 0];
    // c: inside an iteration from the chunks' parts where the update kernel
    // writes them, else as tl_restrict_kernel left it
    const bool parts = mode == 0 && d.cparts;
    const auto *src = parts ? gl(d.cpart) : gl(d.cvec);
    __shared__ double cvec[MAX_CW * 4];
    if (!parts || d.nchunk == d.nagg) {
#pragma unroll
        for (int t = 0; t < NCV; t++) {
            const int k = (int)threadIdx.x + 256 * t;
            cs[t] = src[k < d.nc ? k : 0];
        }
    } else {
#pragma unroll
        for (int t = 0; t < NCV; t++) {
            const int k = (int)threadIdx.x + 256 * t, a = k / 6, q = k - 6 * a;
            cs[t] = 0.0;
            if (k < d.nc)
                for (int32_t h = gl(d.aggch)[a], h1 = gl(d.aggch)[a + 1]; h < h1; h++)
                    cs[t] += src[(int64_t)h * 6 + q];
        }
    }
    AMR_ISSUED();
    if (done) return;
#pragma unroll
    for (int t = 0; t < NCV; t++) cvec[threadIdx.x + 256 * t] = cs[t];
    __syncthreads();
    double acc = 0.0;
    if (row < d.nc)
        for (int cb = lane; cb < d.nc; cb += 64 * NB) {
            if (cb >= 64 * NB)
#pragma unroll
                for (int j = 0; j < NB; j++) kv[j] = Kr[cb + 64 * j < d.nc ? cb + 64 * j : 0];
#pragma unroll
            for (int j = 0; j < NB; j++)
                acc = cb + 64 * j < d.nc ? fma(kv[j], cvec[cb + 64 * j], acc) : acc;
        }
    acc = wave_sum(acc);
    __shared__ double cyw[4];
    if (lane == 0) {
        if (row < d.nc) glw(d.yvec)[row] = acc;
        cyw[threadIdx.x / 64] = row < d.nc ? cvec[row] * acc : 0.0;
    }
    __syncthreads();
    if (threadIdx.x == 0) glw(d.part)[(pi ? P_CY1 : P_CY0) + e.y] = ((cyw[0] + cyw[1]) + cyw[2]) + cyw[3];
}

__global__ void __launch_bounds__(WGV) tl_prolong_kernel(const SegDesc *__restrict__ D, const int2 *__restrict__ vl)
{
    const int2 ve = vl[blockIdx.x];
    const SegDesc &d = D[ve.x];
    float *__restrict__ p32 = d.wp32 ? d.p32 : nullptr;
    const int64_t n = d.nnodes * 3, stride = (int64_t)d.nvblk * WGV;
    for (int64_t i = (int64_t)ve.y * WGV + threadIdx.x; i < n; i += stride) {
        const double pn = d.z[i] + coarse_term(d, i / 3, (int)(i % 3));
        d.p[i] = pn;
        if (p32) p32[i] = (float)pn;
    }
}

// x = 0, r = b, z = M r, p = z; partials rz -> P_RZ1, rr -> P_RR1
__global__ void __launch_bounds__(WGV) pcg_init_kernel(const SegDesc *__restrict__ D, const int2 *__restrict__ vl)
{
    const int2 ve = vl[blockIdx.x];
    const SegDesc &d = D[ve.x];
    // iteration 0: the two-level kernels after this one write the parity
    // slot of C_ITERS - 1, i.e. slot 1, like the Jacobi partials below
    if (ve.y == 0 && threadIdx.x == 0) glw(d.ctl)[C_ITERS] = glw(d.ctl)[C_PREV] = 0;
    double rz = 0.0, rr = 0.0;
    float *__restrict__ p32 = d.wp32 ? d.p32 : nullptr;
    const int64_t stride = (int64_t)d.nvblk * WGV;
    for (int64_t nd = (int64_t)ve.y * WGV + threadIdx.x; nd < d.nnodes; nd += stride) {
        double rv[3], zv[3];
        for (int c = 0; c < 3; c++) rv[c] = d.b[nd * 3 + c];
        apply_prec(d, nd, rv, zv);
        for (int c = 0; c < 3; c++) {
            const int64_t i = nd * 3 + c;
            d.x[i] = 0.0;
            d.r[i] = rv[c];
            d.z[i] = zv[c];
            d.p[i] = zv[c];
            if (p32) p32[i] = (float)zv[c];
            rz = fma(rv[c], zv[c], rz);
            rr = fma(rv[c], rv[c], rr);
        }
    }
    rz = block_sum<WGV>(rz);
    rr = block_sum<WGV>(rr);
    if (threadIdx.x == 0) {
        glw(d.part)[P_RZ1 + ve.y] = rz;
        glw(d.part)[P_RR1 + ve.y] = rr;
    }
}

// r = rt; z = M r; rz partials into the slot the next iteration reads as
// "previous".  The search direction the next iteration takes as it is:
//   REZ_KEEP     already in p (pcg_dir_kernel formed it)
//   REZ_RESTART  p = z: it starts afresh
//   REZ_FORM     p = z + beta p with the z and beta of the stop: a member whose
//                operator forms the direction (d.fuse) stopped inside a step,
//                before anything stored it; p still is the direction of the
//                iteration before, orthogonal to r, and no later iteration
//                would leave that state
enum { REZ_KEEP = 0, REZ_RESTART, REZ_FORM, REZ_NMODE };
__global__ void __launch_bounds__(WGV) pcg_rez_kernel(const SegDesc *__restrict__ D, const int2 *__restrict__ vl,
                                                      int mode)
{
    const int2 ve = vl[blockIdx.x];
    const SegDesc &d = D[ve.x];
    const int slot_pi = 1 - (glw(d.ctl)[C_ITERS] & 1);
    const double beta = d.scal[S_BETA];
    float *__restrict__ p32 = d.wp32 ? d.p32 : nullptr;
    double rz = 0.0;
    const int64_t stride = (int64_t)d.nvblk * WGV;
    for (int64_t nd = (int64_t)ve.y * WGV + threadIdx.x; nd < d.nnodes; nd += stride) {
        double rv[3], zv[3];
        for (int c = 0; c < 3; c++) rv[c] = d.rt[nd * 3 + c];
        apply_prec(d, nd, rv, zv);
        for (int c = 0; c < 3; c++) {
            const int64_t i = nd * 3 + c;
            if (mode == REZ_FORM) d.p[i] = fma(beta, d.p[i], d.z[i]);
            d.r[i] = rv[c];
            d.z[i] = zv[c];
            if (mode == REZ_RESTART) {
                d.p[i] = zv[c];
                if (p32) p32[i] = (float)zv[c];
            }
            rz = fma(rv[c], zv[c], rz);
        }
    }
    rz = block_sum<WGV>(rz);
    if (threadIdx.x == 0) glw(d.part)[(slot_pi ? P_RZ1 : P_RZ0) + ve.y] = rz;
}

// One workgroup per listed model publishes scalars from partials.
//   mode 0 (after init):        rz, rr = bb from slot 1; recursive threshold; reset control
//   mode 1 (after replacement): rr, bb, kx, drift from the residual partials
//   mode 2 (resume):            rz from the slot written by pcg_rez; clear the stop flags
__global__ void __launch_bounds__(WGV) pcg_finalize_kernel(const SegDesc *__restrict__ D,
                                                           const int32_t *__restrict__ sl, int mode)
{
    const SegDesc &d = D[sl[blockIdx.x]];
    auto *ctl = glw(d.ctl);
    double *scal = d.scal;
    if (mode == 0) {
        const double rz = sum_rz(d, 1);
        const double rr = sum_partials<WGV>(d.part + P_RR1, d.nvblk);
        if (threadIdx.x == 0) {
            scal[S_RZ] = rz;
            scal[rz_pub(1)] = rz;
            scal[S_RR] = rr;
            scal[S_BB] = rr;
            scal[S_KX] = 0.0;
            scal[S_GAP] = 0.0;
            scal[S_THR] = d.thr_fac * rr;
            ctl[C_ITERS] = 0;
            ctl[C_PREV] = 0;
            ctl[C_BREAK] = 0;
            ctl[C_STOP] = 0;
            ctl[C_DONE] = rr == 0.0 ? 1 : 0;
        }
    } else if (mode == 1) {
        const double rr = sum_partials<WGV>(d.part + P_A, d.ntiles);
        const double bb = sum_partials<WGV>(d.part + P_B, d.ntiles);
        const double kx = sum_partials<WGV>(d.part + P_C, d.ntiles);
        const double gap = sum_partials<WGV>(d.part + P_D, d.ntiles);
        if (threadIdx.x == 0) {
            scal[S_RR] = rr;
            scal[S_BB] = bb;
            scal[S_KX] = kx;
            scal[S_GAP] = gap;
        }
    } else {
        const int slot_pi = 1 - (ctl[C_ITERS] & 1);
        const double rz = sum_rz(d, slot_pi);
        if (threadIdx.x == 0) {
            scal[S_RZ] = rz;
            scal[rz_pub(slot_pi)] = rz;
            ctl[C_PREV] = ctl[C_ITERS];
            ctl[C_DONE] = 0;
            ctl[C_STOP] = 0;
            ctl[C_BREAK] = 0;
        }
    }
}

__global__ void fill_f32_kernel(int64_t n, float *__restrict__ x, float v)
{
    for (int64_t i = (int64_t)blockIdx.x * WGV + threadIdx.x; i < n; i += (int64_t)gridDim.x * WGV) x[i] = v;
}

__global__ void fill_kernel(int64_t n, double *__restrict__ x, double v)
{
    for (int64_t i = (int64_t)blockIdx.x * WGV + threadIdx.x; i < n; i += (int64_t)gridDim.x * WGV) x[i] = v;
}

// Row tiles of a model: R = 64 rows, a whole number of the row passes of a
// 512-thread workgroup at every lanes value (16 rows per pass at 32 lanes,
// 8 at 64, 32 at 16, 64 at 8); models of more than 64 * MAX_GR nodes take
// the next multiple of 64 that keeps MAX_GR tiles.  On the 40^3 HEX20 block
// (L = 32) the SpMV took 153.9 us with R = 64 and 154.5 us with 48 against
// 155.8-160.0 us with 40, 56, 72, 80 and 96 (rows that leave the last pass
// partly idle, or longer tiles) and 162.6 us with 128.  Vector kernels: at
// most MAX_GV workgroups.
struct Geom {
    int R, ntiles, nvblk;
};

Geom model_geom(const amr_model *m)
{
    Geom g;
    const int64_t n = std::max<int64_t>(1, m->nnodes);
    int64_t R = 64;
    if ((n + R - 1) / R > MAX_GR) R = ((n + MAX_GR - 1) / MAX_GR + 63) / 64 * 64;
    g.R = (int)R;
    g.ntiles = (int)((n + R - 1) / R);
    const int64_t nv = (m->nnodes * 3 + WGV - 1) / WGV;
    g.nvblk = (int)std::max<int64_t>(1, std::min<int64_t>(nv, MAX_GV));
    return g;
}

// Tiles of the matrix-free operator.  With few groups the waves of a
// workgroup share a group where its IP slots can be divided (four waves a group
// for 27 IPs, two for the hex rules with 8): such a launch is bound by one
// wave's chain of matrix instructions, not by throughput.  The line is at two
// groups per CU, 512.  Up to there all workgroups run at once, two per CU with
// four waves a group (65 KB of LDS each), one with two; a workgroup more
// waits for a place, or shares a CU with another.  Launches between events, one wave a group against shared,
// at 512 and 529 groups: HEX20 with 27 IPs 15.3 / 13.8 and 15.3 / 17.7 us, with
// 8 IPs 10.8 / 10.0 and 11.0 / 11.4, HEX8 8.31 / 8.12 and 8.26 / 8.50; at 46
// and 938 groups with 27 IPs 13.7 / 9.9 and 15.4 / 21.3.  Above, a wave takes
// a group of its own, G groups in turn only where the p.q partials would not
// fit otherwise (two groups a wave made the 40^3 HEX20 block no faster and the
// TET10 49x12x13 box 10% slower).
struct MfGeom {
    int W, G, ntiles;
};

MfGeom mf_geom(const amr_model *m)
{
    MfGeom g;
    g.W = m->mf_ngrp > 2 * (int64_t)m->ncu ? 1 : m->nips == 27 ? 4 : m->nips == 8 ? 2 : 1;
    if (m->test_tiles) g.W = 1;  // (a shared group's waves take one group only)
    const int64_t ng = 4 / g.W, most = m->test_tiles ? m->test_tiles : MAX_GR;
    g.G = (int)std::max<int64_t>(1, (m->mf_ngrp + ng * most - 1) / (ng * most));
    g.ntiles = (int)((m->mf_ngrp + ng * g.G - 1) / (ng * g.G));
    return g;
}

size_t tile_lds(int R, int ndbl) { return (size_t)(((R + 1) * 4 + 15) & ~15) + (size_t)ndbl * pow2ceil(R) * 8; }

// SpMV operand kinds: FP64 values; FP32 values with FP32 p and FP32
// accumulation; FP32 values with FP64 gather and accumulation.
enum { K_F64 = 0, K_F32, K_F32D, K_NKIND };
// Launch groups after those: the matrix-free operator of each element shape,
// with one wave per group and with shared groups
enum { K_MF = K_NKIND, K_FZ = K_MF + 8, K_NGROUP = K_FZ + 2 };
// K_FZ: the SpMV that forms the direction, FP64 values; + 1: FP32 values

int lanes_index(int lanes) { return lanes == 8 ? 0 : lanes == 16 ? 1 : lanes == 32 ? 2 : 3; }
constexpr int LANES[4] = {8, 16, 32, 64};

int kind_lanes(const amr_model *m, int kind)
{
    return kind == K_F64 ? m->lanes64 : kind == K_F32 ? m->lanes32 : m->lanes32d;
}

void launch_pcg_spmv(int kind, int lanes, unsigned grid, int Rmax, hipStream_t s, const SegDesc *D, const int2 *tl,
                     int first)
{
    const size_t lds = tile_lds(Rmax, 1);
#define AMR_PCG_SPMV(LN, VT, XT, AT, FZ) \
    hipLaunchKernelGGL((pcg_spmv_kernel<LN, VT, XT, AT, FZ>), dim3(grid), dim3(WGS), lds, s, D, tl, first)
#define AMR_PCG_KIND(LN)                                                     \
    do {                                                                     \
        if (kind == K_F64) AMR_PCG_SPMV(LN, double, double, double, false);  \
        else if (kind == K_F32) AMR_PCG_SPMV(LN, float, float, float, false); \
        else if (kind == K_F32D) AMR_PCG_SPMV(LN, float, double, double, false); \
        else if (kind == K_FZ) AMR_PCG_SPMV(LN, double, double, double, true); \
        else AMR_PCG_SPMV(LN, float, double, double, true);                  \
    } while (0)
    switch (lanes) {
    case 8: AMR_PCG_KIND(8); break;
    case 16: AMR_PCG_KIND(16); break;
    case 32: AMR_PCG_KIND(32); break;
    default: AMR_PCG_KIND(64); break;
    }
#undef AMR_PCG_KIND
#undef AMR_PCG_SPMV
}

int mf_kind(const amr_model *m)
{
    const int shape = m->etype == AMR_HEX8 ? 0 : m->etype == AMR_TET10 ? 3 : m->nips == 27 ? 1 : 2;
    return K_MF + 2 * shape + (mf_geom(m).W > 1 ? 1 : 0);
}

void launch_pcg_mf(int kind, unsigned grid, hipStream_t s, const SegDesc *D, const int2 *tl, int first)
{
#define AMR_MF(NN, NQ, W) hipLaunchKernelGGL((pcg_mf_kernel<NN, NQ, W>), dim3(grid), dim3(256), 0, s, D, tl, first)
    switch (kind - K_MF) {
    case 0: AMR_MF(8, 8, 1); break;
    case 1: AMR_MF(8, 8, 2); break;
    case 2: AMR_MF(20, 27, 1); break;
    case 3: AMR_MF(20, 27, 4); break;
    case 4: AMR_MF(20, 8, 1); break;
    case 5: AMR_MF(20, 8, 2); break;
    default: AMR_MF(10, 4, 1); break;
    }
#undef AMR_MF
}

void launch_residual(int lanes, unsigned grid, int Rmax, hipStream_t s, const SegDesc *D, const int2 *tl)
{
    const size_t lds = tile_lds(Rmax, 4);
#define AMR_RES(LN) hipLaunchKernelGGL((residual_kernel<LN>), dim3(grid), dim3(WGS), lds, s, D, tl)
    switch (lanes) {
    case 8: AMR_RES(8); break;
    case 16: AMR_RES(16); break;
    case 32: AMR_RES(32); break;
    default: AMR_RES(64); break;
    }
#undef AMR_RES
}

}  // namespace

// ------------------------------------------------------------- the pool

namespace {

struct Member {
    amr_model *m = nullptr;
    amr_solve_opts o{};
    const double *b = nullptr;
    double *x = nullptr;
    int state = 0;  // 0 free, 1 joining, 2 active
    bool mixed = false, f32x = false;
    bool mf = false;     // iterates on the matrix-free FP64 operator
    bool pc32 = false;   // a mixed precision was asked for: preconditioner in FP32
    double bb = 0.0, rr_ref = 0.0, rr_true_prev = INFINITY, relres = 0.0;
    int converged = 0, broke = 0, replacements = 0, iters = 0, fell_back = 0, breakdowns = 0;
    int last_rep = 0;  // iteration of the last residual replacement
    bool form = false;  // its coarse operator is to be formed before it starts
    // per-step scratch
    bool rep = false, done = false;
    bool unformed = false;  // stopped before its next direction was stored (REZ_FORM)
    double rr_rec = 0.0;
    int early = 0;  // early stops still to come (amr_test_early_stops)
};

// M_WAIT: joined, but work the model queued on its own stream before
// joining (assembly), or the formation of its coarse operator, may still be
// running; it starts at the first step that finds that work done, so that a
// slow joiner does not hold up the members already solving
enum { M_FREE = 0, M_JOIN, M_ACTIVE, M_WAIT };

}  // namespace

struct amr_pool {
    int device = 0;
    hipStream_t stream = nullptr;
    bool own_stream = false;
    int cap = 0, check = 32;
    std::vector<Member> mem;
    std::vector<amr_model *> attached;
    // device descriptors and scalars, with pinned host mirrors
    SegDesc *dD = nullptr, *hD = nullptr;
    double *dS = nullptr, *hS = nullptr;
    // work lists: staged in pinned memory, uploaded in one copy per use
    char *dL = nullptr, *hL = nullptr;
    size_t lcap = 0, lused = 0;
    bool pending = false;  // an upload from the pinned mirrors may still be in flight
    hipEvent_t ev_upload = nullptr;  // recorded after each upload
    bool desc_dirty = false;
    // a step launched by amr_pool_step_begin and not yet collected
    bool in_flight = false;
    hipEvent_t ev_step = nullptr;    // recorded after the step's scalar read-back
    std::vector<int> fl_act;         // members of the in-flight step
    // models that left the pool at the last step and still run on its
    // stream; they return to their own streams when the next step is queued
    // (or at amr_pool_hand_back), so that the work queued for them in
    // between (the NR finish) runs ahead of that step
    std::vector<amr_model *> leaving;
    // SpMV timing
    bool timing = false;
    std::vector<hipEvent_t> ev;
    double t_spmv_ms = 0.0;
    int64_t n_spmv = 0;
    // captured iteration blocks of a step (check_every iterations of every
    // PCG phase), keyed by their launch shapes; replayed while the shapes
    // stay (work lists padded to size classes, members joining and leaving
    // change only the lists' contents)
    struct StepGraph {
        std::vector<int64_t> key;
        hipGraphExec_t exec = nullptr;
        uint64_t used = 0;
    };
    std::vector<StepGraph> graphs;
    bool use_graphs = false;
    uint64_t graph_clock = 0;
    int64_t graph_captures = 0, graph_replays = 0;
    // coarse operators of two-level joiners are formed in batches: on the
    // side stream for joiners that start at a later step (the members
    // already solving are not held up), on the pool's stream for those that
    // start at once
    hipStream_t side = nullptr;
    AmrStaging stg_side, stg_pool;
    int64_t coarse_batches = 0, coarse_formed = 0;
    int64_t iter_kernels = 0, iter_submits = 0;  // of the steps' PCG iterations
    int64_t member_kernels = 0;  // the same iterations launched member by member
};

namespace {

int pool_sync(amr_pool *p)
{
    AMR_HIP(hipStreamSynchronize(p->stream));
    p->pending = false;
    return AMR_OK;
}

// Make the pinned mirrors writable: wait for any upload still reading them
// (only for the copy, not for the kernels queued after it).
int pool_begin_host_writes(amr_pool *p)
{
    if (!p->pending) return AMR_OK;
    AMR_HIP(hipEventSynchronize(p->ev_upload));
    p->pending = false;
    return AMR_OK;
}

void drop_graphs(amr_pool *p)
{
    for (auto &g : p->graphs)
        if (g.exec) (void)hipGraphExecDestroy(g.exec);
    p->graphs.clear();
}

int pool_reserve_lists(amr_pool *p, size_t bytes)
{
    if (bytes <= p->lcap) return AMR_OK;
    // kernels queued earlier may still read the device list buffer
    if (int rc = pool_sync(p)) return rc;
    drop_graphs(p);  // they point into the old buffer
    size_t ncap = std::max<size_t>(bytes, 2 * p->lcap);
    ncap = std::max<size_t>(ncap, 1 << 16);
    if (p->dL) AMR_HIP(hipFree(p->dL));
    if (p->hL) AMR_HIP(hipHostFree(p->hL));
    p->dL = p->hL = nullptr;
    p->lcap = 0;
    AMR_HIP(hipMalloc(&p->dL, ncap));
    AMR_HIP(hipHostMalloc(&p->hL, ncap, hipHostMallocDefault));
    p->lcap = ncap;
    return AMR_OK;
}

// List staging: reset, append, upload.  Offsets are 16-byte aligned.
struct Lists {
    amr_pool *p;
    size_t off = 0;
    template <typename T>
    T *dev_at(size_t o) const { return (T *)(p->dL + o); }
    template <typename T>
    size_t push(const std::vector<T> &v)
    {
        const size_t o = off;
        if (!v.empty()) std::memcpy(p->hL + o, v.data(), v.size() * sizeof(T));
        off = (o + v.size() * sizeof(T) + 15) & ~(size_t)15;
        return o;
    }
};

template <typename T>
size_t padded(const std::vector<T> &v) { return (v.size() * sizeof(T) + 15) & ~(size_t)15; }

int upload(amr_pool *p, size_t bytes, bool desc)
{
    if (bytes) AMR_HIP(hipMemcpyAsync(p->dL, p->hL, bytes, hipMemcpyHostToDevice, p->stream));
    if (desc) {
        AMR_HIP(hipMemcpyAsync(p->dD, p->hD, sizeof(SegDesc) * p->cap, hipMemcpyHostToDevice, p->stream));
        p->desc_dirty = false;
    }
    if (bytes || desc) {
        AMR_HIP(hipEventRecord(p->ev_upload, p->stream));
        p->pending = true;
    }
    return AMR_OK;
}

// A model's work runs on its own stream, and on the pool's stream while it
// is a member; the switches are ordered with events, without waiting.
int handoff(amr_model *m, hipStream_t from, hipStream_t to)
{
    if (from == to) return AMR_OK;
    if (!m->ev_handoff) AMR_HIP(hipEventCreateWithFlags(&m->ev_handoff, hipEventDisableTiming));
    AMR_HIP(hipEventRecord(m->ev_handoff, from));
    AMR_HIP(hipStreamWaitEvent(to, m->ev_handoff, 0));
    m->stream = to;
    return AMR_OK;
}

// Members on an assembled matrix without a coarse correction: up to this many
// nodes the direction is formed in the SpMV's gather (a launch less per
// iteration).  Passes with and without: HEX20 31x4x5 dynamic (3,400 nodes) 97.1
// and 100.3 ms, TET10 20x5x5 von Mises (5,000) 25.0 and 25.9, HEX8 64x16x16
// (18,800) 12.9 and 13.5, HEX20 40x10x10 with 27 IPs (20,000) 39.7 and 39.1.
constexpr int64_t FUSE_MAX = 16384;

// Two-level members on an assembled matrix: the update kernel by chunks, with
// the restriction.  On the matrix-free operator it stays in node order: summing
// the elements' products in aggregate order lost more (TET10 49x12x13: 13.3 ->
// 19.8 us, 40^3 HEX20: 17.6 -> 28.4 us) than the restriction's own launch (5.0
// and 10.1 us).
void set_cparts(SegDesc &d, bool on)
{
    d.cparts = on ? 1 : 0;
    d.nred = on ? d.nchunk : d.nvblk;
}

// The recursion stops where |r|^2 falls to this times |b|^2: half the
// tolerance, or, for the early stops a test asks for, the next power of
// early_rtol.
double stop_factor(const Member &M)
{
    const double rtol = M.early > 0 ? std::pow(M.m->test_early_rtol, M.m->test_early - M.early + 1) : M.o.rtol;
    const double tr = 0.5 * rtol;
    return tr * tr;
}

void fill_desc(amr_pool *p, int slot)
{
    Member &M = p->mem[slot];
    amr_model *m = M.m;
    const Geom g = model_geom(m);
    SegDesc &d = p->hD[slot];
    std::memset(&d, 0, sizeof d);
    d.rowptr = m->rowptr;
    d.col = m->col;
    d.col16 = m->col16;
    d.Kv = m->Kv;
    d.Kv32 = m->Kv32;
    d.mask = m->mask;
    d.dinv = m->dinv;
    d.binv = m->binv;
    d.dinv32 = m->dinv32;
    d.binv32 = m->binv32;
    d.b = M.b;
    d.x = M.x;
    d.r = m->v[1];
    d.z = m->v[2];
    d.p = m->v[3];
    d.q = m->v[4];
    d.rt = m->v[5];
    d.p32 = m->f[0];
    d.part = m->part;
    d.scal = p->dS + (size_t)slot * SEG_DBL;
    d.ctl = (int32_t *)(d.scal + S_NSCAL);
    d.nnodes = m->nnodes;
    d.nblk = m->pat.nblk;
    d.thr_fac = stop_factor(M);
    d.R = g.R;
    d.ntiles = g.ntiles;
    d.nvblk = g.nvblk;
    d.maxiter = M.o.maxiter;
    d.f32 = M.mixed || (M.mf && M.pc32) ? 1 : 0;
    d.npq = g.ntiles;
    d.nred = g.nvblk;
    d.block = M.o.precond == AMR_PRECOND_BLOCK_JACOBI ? 1 : 0;
    d.wp32 = (M.mixed && M.f32x) ? 1 : 0;
    d.tl = M.o.precond == AMR_PRECOND_TWO_LEVEL ? 1 : 0;
    if (d.tl) {
        d.nagg = m->nagg;
        d.nc = m->ncoarse;
        d.ncw = (m->ncoarse + 3) / 4;
        d.agg = m->c_agg;
        d.aggptr = m->c_aggptr;
        d.aggnodes = m->c_aggnodes;
        d.cent = m->c_cent;
        d.X = m->X;
        d.Kinv = m->Kinv;
        d.cvec = m->c_vec;
        d.yvec = m->y_vec;
        d.chunk = (const i32x4 *)m->c_chunk;
        d.aggch = m->c_aggch;
        d.cpart = m->c_part;
        d.nchunk = m->nchunk;
        set_cparts(d, !M.mf);
    }
    if (!d.tl && !(M.mixed && M.f32x) && m->nnodes <= FUSE_MAX) d.fuse = 1;
    if (M.mf) {
        const MfGeom mg = mf_geom(m);
        d.geo = m->mf_geo;
        d.lm = m->mf_lm;
        d.tab = m->mf_tab;
        d.mfconn = m->mf_conn;
        d.fptr = m->fptr;
        d.mfsrc = m->mf_src;
        d.mfrec = m->mf_rec;
        d.mff = m->mf_f;
        d.ngrp = m->mf_ngrp;
        d.mfG = mg.G;
        d.npq = mg.ntiles;
        d.fuse = d.tl ? 0 : 1;
    }
}

std::vector<int2> agg_list(amr_pool *p, const std::vector<int> &slots)
{
    std::vector<int2> v;
    for (int s : slots)
        if (p->hD[s].tl)
            for (int a = 0; a < p->hD[s].nagg; a++) v.push_back(make_int2(s, a));
    return v;
}

std::vector<int2> cw_list(amr_pool *p, const std::vector<int> &slots)
{
    std::vector<int2> v;
    for (int s : slots)
        if (p->hD[s].tl)
            for (int w = 0; w < p->hD[s].ncw; w++) v.push_back(make_int2(s, w));
    return v;
}

std::vector<int> tl_only(amr_pool *p, const std::vector<int> &slots)
{
    std::vector<int> v;
    for (int s : slots)
        if (p->hD[s].tl) v.push_back(s);
    return v;
}

// the two-level steps after an initialisation or a resume: c, y, and with
// `prolong` the search direction p = z + Phi y
void launch_tl_fresh(amr_pool *p, const Lists &Ls, size_t o_al, unsigned nal, size_t o_cw, unsigned ncw,
                     size_t o_pv, unsigned npv)
{
    hipStream_t st = p->stream;
    if (nal) hipLaunchKernelGGL(tl_restrict_kernel, dim3(nal), dim3(WGR), 0, st, p->dD, Ls.dev_at<int2>(o_al), 1);
    if (ncw) hipLaunchKernelGGL(tl_coarse_kernel, dim3(ncw), dim3(256), 0, st, p->dD, Ls.dev_at<int2>(o_cw), 1);
    if (npv) hipLaunchKernelGGL(tl_prolong_kernel, dim3(npv), dim3(WGV), 0, st, p->dD, Ls.dev_at<int2>(o_pv));
}

int member_kind(const Member &M) { return !M.mixed ? K_F64 : (M.f32x ? K_F32 : K_F32D); }

// Tile lists of the given members grouped by (kind, lanes); for residual
// launches kind is ignored and the FP64 lanes are used.
struct Group {
    int kind, lanes, Rmax;
    size_t off;     // device offset of the group's entries
    unsigned n;
};

void build_groups(amr_pool *p, const std::vector<int> &slots, bool residual, std::vector<std::vector<int2>> &ent,
                  std::vector<Group> &gr)
{
    ent.assign(K_NGROUP * 4, {});
    std::vector<int> rmax(K_NGROUP * 4, 0);
    for (int s : slots) {
        const Member &M = p->mem[s];
        if (M.mf && !residual) {
            const int key = mf_kind(M.m) * 4;
            for (int t = 0; t < p->hD[s].npq; t++) ent[key].push_back(make_int2(s, t));
            continue;
        }
        const int kind = residual ? K_F64 : member_kind(M);
        const SegDesc &d = p->hD[s];
        const int gk = !residual && d.fuse ? K_FZ + (kind == K_F32D ? 1 : 0) : kind;
        const int key = gk * 4 + lanes_index(kind_lanes(M.m, kind));
        for (int t = 0; t < d.ntiles; t++) ent[key].push_back(make_int2(s, t));
        rmax[key] = std::max(rmax[key], d.R);
    }
    gr.clear();
    for (int key = 0; key < K_NGROUP * 4; key++)
        if (!ent[key].empty()) gr.push_back({key / 4, LANES[key % 4], rmax[key], 0, (unsigned)ent[key].size()});
}

// Work lists of a captured step are padded with empty entries (member -1,
// which the kernels skip) to a size class: 64, then 2^k and 3*2^(k-1).
size_t size_class(size_t n)
{
    if (n <= 64) return 64;
    size_t c = 64;
    while (c < n) {
        if (c + c / 2 >= n) return c + c / 2;
        c *= 2;
    }
    return c;
}

void pad_list(std::vector<int2> &v)
{
    if (!v.empty()) v.resize(size_class(v.size()), make_int2(-1, -1));
}

// the chunks of the two-level members (aggregate-ordered vector work)
std::vector<int2> chunk_list(amr_pool *p, const std::vector<int> &slots)
{
    std::vector<int2> v;
    for (int s : slots)
        for (int j = 0; j < p->hD[s].nchunk; j++) v.push_back(make_int2(s, j));
    return v;
}

std::vector<int2> vec_list(amr_pool *p, const std::vector<int> &slots)
{
    std::vector<int2> v;
    for (int s : slots)
        for (int j = 0; j < p->hD[s].nvblk; j++) v.push_back(make_int2(s, j));
    return v;
}

int ensure_events(amr_pool *p)
{
    if ((int)p->ev.size() >= 2 * p->check) return AMR_OK;
    for (hipEvent_t e : p->ev) (void)hipEventDestroy(e);
    p->ev.assign(2 * p->check, nullptr);
    for (hipEvent_t &e : p->ev) AMR_HIP(hipEventCreate(&e));
    return AMR_OK;
}

void finish(amr_pool *p, int slot, std::vector<amr_pool_result> &out)
{
    Member &M = p->mem[slot];
    amr_pool_result r;
    r.m = M.m;
    r.info.iterations = M.iters;
    r.info.refinements = M.replacements;
    r.info.converged = M.converged;
    r.info.fallback = M.fell_back;
    r.info.relres = M.relres;
    out.push_back(r);
    M = Member();
}

}  // namespace

int amr_pool_new(amr_pool **out, int device, int cap, int check, hipStream_t stream)
{
    if (cap < 1 || cap > (1 << 16)) {
        amr_set_error("amr_pool_create: max_members must be in [1, 65536]");
        return AMR_ERR_ARG;
    }
    AMR_HIP(hipSetDevice(device));
    amr_pool *p = new amr_pool();
    p->device = device;
    p->cap = cap;
    p->check = std::max(1, std::min(check > 0 ? check : 32, 256));
    p->mem.assign(cap, Member());
    // steps launch kernel by kernel unless AMR_POOL_GRAPHS=1 (or
    // amr_pool_set_graphs) asks for captured ones: on MI355X the replayed
    // graphs ran the pooled workloads 4-12% slower than the same kernels
    // launched one by one
    if (const char *g = std::getenv("AMR_POOL_GRAPHS")) p->use_graphs = std::atoi(g) != 0;
    int rc = AMR_OK;
    auto fail = [&](hipError_t e) {
        amr_set_error(std::string("HIP error: ") + hipGetErrorString(e) + " creating a pool");
        amr_pool_free(p);
        return AMR_ERR_HIP;
    };
    hipError_t e;
    if (stream) p->stream = stream;
    else {
        if ((e = hipStreamCreateWithFlags(&p->stream, hipStreamNonBlocking)) != hipSuccess) return fail(e);
        p->own_stream = true;
    }
    if ((e = hipEventCreateWithFlags(&p->ev_upload, hipEventDisableTiming)) != hipSuccess) return fail(e);
    if ((e = hipEventCreateWithFlags(&p->ev_step, hipEventDisableTiming)) != hipSuccess) return fail(e);
    if ((e = hipMalloc(&p->dD, sizeof(SegDesc) * cap)) != hipSuccess) return fail(e);
    if ((e = hipHostMalloc(&p->hD, sizeof(SegDesc) * cap, hipHostMallocDefault)) != hipSuccess) return fail(e);
    if ((e = hipMalloc(&p->dS, sizeof(double) * SEG_DBL * cap)) != hipSuccess) return fail(e);
    if ((e = hipHostMalloc(&p->hS, sizeof(double) * SEG_DBL * cap, hipHostMallocDefault)) != hipSuccess)
        return fail(e);
    std::memset(p->hD, 0, sizeof(SegDesc) * cap);
    if ((e = hipMemsetAsync(p->dS, 0, sizeof(double) * SEG_DBL * cap, p->stream)) != hipSuccess) return fail(e);
    if ((e = hipStreamSynchronize(p->stream)) != hipSuccess) return fail(e);
    (void)rc;
    *out = p;
    return AMR_OK;
}

void amr_pool_free(amr_pool *p)
{
    if (!p) return;
    (void)hipSetDevice(p->device);
    if (p->stream) (void)hipStreamSynchronize(p->stream);
    for (amr_model *m : p->attached) {
        m->stream = m->own_stream;
        m->pool = nullptr;
    }
    if (p->dD) (void)hipFree(p->dD);
    if (p->hD) (void)hipHostFree(p->hD);
    if (p->dS) (void)hipFree(p->dS);
    if (p->hS) (void)hipHostFree(p->hS);
    if (p->dL) (void)hipFree(p->dL);
    if (p->hL) (void)hipHostFree(p->hL);
    for (hipEvent_t e : p->ev)
        if (e) (void)hipEventDestroy(e);
    if (p->ev_upload) (void)hipEventDestroy(p->ev_upload);
    if (p->ev_step) (void)hipEventDestroy(p->ev_step);
    if (p->side) (void)hipStreamSynchronize(p->side);
    amr_staging_free(p->stg_side);
    amr_staging_free(p->stg_pool);
    if (p->side) (void)hipStreamDestroy(p->side);
    drop_graphs(p);
    if (p->own_stream && p->stream) (void)hipStreamDestroy(p->stream);
    delete p;
}

int amr_pool_attach_model(amr_pool *p, amr_model *m)
{
    if (m->pool == p) return AMR_OK;
    if (m->pool) {
        amr_set_error("the model is attached to another pool");
        return AMR_ERR_ARG;
    }
    if (m->device != p->device) {
        amr_set_error("the model and the pool are on different devices");
        return AMR_ERR_ARG;
    }
    m->pool = p;
    p->attached.push_back(m);
    return AMR_OK;
}

int amr_pool_detach_model(amr_model *m)
{
    amr_pool *p = m->pool;
    if (!p) return AMR_OK;
    bool member = false;
    for (int s = 0; s < p->cap; s++)
        if (p->mem[s].m == m) {
            p->mem[s] = Member();
            member = true;
        }
    if (member || m->stream != m->own_stream) {
        // its kernels may still be queued on the pool's stream (or, for its
        // coarse operator, on the side stream)
        AMR_HIP(hipStreamSynchronize(p->stream));
        if (p->side) AMR_HIP(hipStreamSynchronize(p->side));
        p->fl_act.erase(std::remove_if(p->fl_act.begin(), p->fl_act.end(),
                                       [&](int s) { return p->mem[s].state == M_FREE; }),
                        p->fl_act.end());
        m->stream = m->own_stream;
    }
    p->attached.erase(std::remove(p->attached.begin(), p->attached.end(), m), p->attached.end());
    p->leaving.erase(std::remove(p->leaving.begin(), p->leaving.end(), m), p->leaving.end());
    m->pool = nullptr;
    return AMR_OK;
}

bool amr_pool_is_member(const amr_model *m)
{
    if (!m->pool) return false;
    for (const Member &M : m->pool->mem)
        if (M.m == m) return true;
    return false;
}

int amr_pool_count(const amr_pool *p)
{
    int n = 0;
    for (const Member &M : p->mem) n += M.state != M_FREE;
    return n;
}

// Join: the model's system K11 x = b starts at the next step.
int amr_pool_join(amr_pool *p, amr_model *m, const double *b, double *x, const amr_solve_opts *o)
{
    if (m->pool != p && m->self_pool != p) {
        amr_set_error("amr_pool_add: the model is not attached to this pool");
        return AMR_ERR_ARG;
    }
    for (const Member &M : p->mem)
        if (M.m == m) {
            amr_set_error("amr_pool_add: the model is already solving in this pool");
            return AMR_ERR_ARG;
        }
    int slot = -1;
    for (int s = 0; s < p->cap && slot < 0; s++)
        if (p->mem[s].state == M_FREE) slot = s;
    if (slot < 0) {
        amr_set_error("amr_pool_add: the pool is full");
        return AMR_ERR_ARG;
    }
    if (int rc = amr_choose_lanes(m)) return rc;
    bool form = false;
    if (o->precond == AMR_PRECOND_TWO_LEVEL) {
        if (int rc = amr_coarse_build(m)) return rc;
        if ((m->ncoarse + 3) / 4 > MAX_CW) {
            amr_set_error("two-level preconditioner: too many aggregates for the coarse product");
            return AMR_ERR_ARG;
        }
        form = amr_coarse_due(m);
    }
    Member M;
    M.form = form;
    M.m = m;
    M.o = *o;
    M.b = b;
    M.x = x;
    M.state = M_JOIN;
    // all-elastic models iterate on the matrix-free FP64 operator in every
    // precision: it moves fewer bytes than the FP32 matrix
    M.pc32 = o->precision == AMR_PREC_MIXED || o->precision == AMR_PREC_MIXED_F64ACC;
    M.mf = m->mf_ok && m->mf_plain;
    M.mixed = M.pc32 && !M.mf;
    M.f32x = o->precision == AMR_PREC_MIXED;
    M.early = m->test_early;
    if (int rc = pool_begin_host_writes(p)) return rc;
    // the model's queued work (assembly, right-hand side) precedes its solve
    if (m->stream != p->stream) {
        if (!m->ev_handoff) AMR_HIP(hipEventCreateWithFlags(&m->ev_handoff, hipEventDisableTiming));
        AMR_HIP(hipEventRecord(m->ev_handoff, m->stream));
        m->stream = p->stream;
        M.state = M_WAIT;
    }
    p->mem[slot] = M;
    fill_desc(p, slot);
    p->desc_dirty = true;
    return AMR_OK;
}

// A step: initialise joining members, run check_every PCG iterations for
// every member, then residual replacements and convergence decisions.
// amr_pool_step_launch queues the iterations and the read-back of the
// members' scalars without waiting; amr_pool_step_collect waits for them,
// decides, queues the replacements and resumes, and appends the members
// that finished (converged or failed) to `out`; they leave the pool, and
// their models' work returns to their own streams when the next step is
// queued.  Members that join while a step is in flight start at the next
// one.
int amr_pool_step_launch(amr_pool *p)
{
    if (p->in_flight) {
        amr_set_error("amr_pool_step_begin: the previous step has not been collected");
        return AMR_ERR_ARG;
    }
    AMR_HIP(hipSetDevice(p->device));
    // joiners whose own work is done start now; if nobody else is solving,
    // the waiting ones start too, the pool's stream waiting for them
    // (a joiner whose coarse operator is due is formed first: on the side
    // stream when others can start now, else on the pool's stream)
    std::vector<int> waiting, side;
    bool ready = false;
    for (int s = 0; s < p->cap; s++) {
        Member &M = p->mem[s];
        if (M.state == M_WAIT) {
            const hipError_t q = hipEventQuery(M.m->ev_handoff);
            if (q == hipSuccess) {
                if (M.form) side.push_back(s);
                else M.state = M_JOIN;
            } else if (q == hipErrorNotReady) {
                (void)hipGetLastError();  // not an error: clear it
                waiting.push_back(s);
            } else {
                AMR_HIP(q);
            }
        }
        ready = ready || M.state == M_JOIN || M.state == M_ACTIVE;
    }
    if (!ready) {
        for (int s : waiting) {
            AMR_HIP(hipStreamWaitEvent(p->stream, p->mem[s].m->ev_handoff, 0));
            p->mem[s].state = M_JOIN;
        }
        for (int s : side) p->mem[s].state = M_JOIN;
        side.clear();
    }
    if (!side.empty()) {
        if (!p->side) AMR_HIP(hipStreamCreateWithFlags(&p->side, hipStreamNonBlocking));
        std::vector<amr_model *> ms;
        for (int s : side) ms.push_back(p->mem[s].m);
        if (int rc = amr_coarse_form(p->side, ms.data(), (int)ms.size(), p->stg_side)) return rc;
        p->coarse_batches++;
        p->coarse_formed += (int64_t)ms.size();
        // they start at the first step that finds the formation done
        for (int s : side) {
            AMR_HIP(hipEventRecord(p->mem[s].m->ev_handoff, p->side));
            p->mem[s].form = false;
        }
    }
    {
        std::vector<amr_model *> ms;
        for (int s = 0; s < p->cap; s++)
            if (p->mem[s].state == M_JOIN && p->mem[s].form) {
                ms.push_back(p->mem[s].m);
                p->mem[s].form = false;
            }
        if (!ms.empty()) {
            if (int rc = amr_coarse_form(p->stream, ms.data(), (int)ms.size(), p->stg_pool)) return rc;
            p->coarse_batches++;
            p->coarse_formed += (int64_t)ms.size();
        }
    }
    std::vector<int> join, act;
    for (int s = 0; s < p->cap; s++) {
        if (p->mem[s].state == M_JOIN) join.push_back(s);
        if (p->mem[s].state == M_JOIN || p->mem[s].state == M_ACTIVE) act.push_back(s);
    }
    if (int rc = amr_pool_hand_back(p)) return rc;
    if (act.empty()) return AMR_OK;
    const int check = p->check;
    hipStream_t st = p->stream;

    // (a) lists for the iterations (first, so that their offsets depend on
    // their own sizes only) and for the initialisation of joiners
    const bool graph = p->use_graphs && !p->timing;
    // one member: its launches need no lists (list_entry), only their sizes
    const bool one = !graph && act.size() == 1;
    const SegDesc *const D = one ? p->dD + act[0] : p->dD;
    std::vector<std::vector<int2>> ent;
    std::vector<Group> gr;
    if (int rc = pool_begin_host_writes(p)) return rc;
    // vector work: update kernels of members on the matrix-free operator, on
    // an assembled matrix, and two-level on an assembled matrix (by chunks of
    // their aggregates); restrictions of the matrix-free two-level members;
    // direction kernels for the one-level members that have one in every
    // iteration (V_D), for all of them in the step's last one (V_L), and for
    // the two-level members (V_T)
    enum { V_M, V_A, V_AF, V_AT, V_RS, V_D, V_L, V_T, V_CW, NV };
    std::vector<int> sv[NV];
    for (int s : act) {
        const SegDesc &d = p->hD[s];
        sv[p->mem[s].mf ? V_M : d.tl ? V_AT : d.fuse ? V_AF : V_A].push_back(s);
        if (d.tl && p->mem[s].mf) sv[V_RS].push_back(s);
        if (!d.tl) {
            sv[V_L].push_back(s);
            if (!d.fuse) sv[V_D].push_back(s);
        } else {
            sv[V_T].push_back(s);
            sv[V_CW].push_back(s);
        }
    }
    std::vector<int2> vl[NV];
    unsigned nv[NV];
    if (one) {
        const SegDesc &d = p->hD[act[0]];
        const Member &M = p->mem[act[0]];
        const int kind = member_kind(M);
        if (M.mf) gr.push_back({mf_kind(M.m), 0, 0, 0, (unsigned)d.npq});
        else
            gr.push_back({d.fuse ? K_FZ + (kind == K_F32D ? 1 : 0) : kind, kind_lanes(M.m, kind), d.R, 0,
                          (unsigned)d.ntiles});
    } else {
        build_groups(p, act, false, ent, gr);
        for (int k = 0; k < NV; k++)
            vl[k] = k == V_CW               ? cw_list(p, sv[k])
                    : k == V_RS             ? agg_list(p, sv[k])
                    : k == V_AT || k == V_T ? chunk_list(p, sv[k])
                                            : vec_list(p, sv[k]);
    }
    if (graph) {
        for (auto &e : ent) pad_list(e);
        int gi = 0;
        for (const auto &e : ent)
            if (!e.empty()) {
                gr[gi].n = (unsigned)e.size();
                gr[gi].Rmax = (gr[gi].Rmax + 63) / 64 * 64;
                gi++;
            }
        for (auto &v : vl) pad_list(v);
    }
    std::vector<int2> vj = vec_list(p, join);
    std::vector<int32_t> sj(join.begin(), join.end());
    std::vector<int2> aj = agg_list(p, join), cj = cw_list(p, join), pj = vec_list(p, tl_only(p, join));
    size_t need = padded(vj) + padded(sj) + padded(aj) + padded(cj) + padded(pj);
    for (const auto &v : vl) need += padded(v);
    for (const auto &e : ent) need += padded(e);
    if (int rc = pool_reserve_lists(p, need)) return rc;
    Lists Ls{p};
    size_t o_v[NV];
    for (int k = 0; k < NV; k++) o_v[k] = Ls.push(vl[k]);
    {
        int gi = 0;
        for (const auto &e : ent)
            if (!e.empty()) gr[gi++].off = Ls.push(e);
    }
    // launch sizes, and the lists' addresses (none for one member)
    const SegDesc &d1 = p->hD[act[0]];
    for (int k = 0; k < NV; k++)
        nv[k] = !one            ? (unsigned)vl[k].size()
                : sv[k].empty() ? 0
                : k == V_CW     ? (unsigned)d1.ncw
                : k == V_RS     ? (unsigned)d1.nagg
                : k == V_AT || k == V_T ? (unsigned)d1.nchunk
                                        : (unsigned)d1.nvblk;
    auto list = [&](size_t o) { return one ? (const int2 *)nullptr : Ls.dev_at<int2>(o); };
    const size_t o_vj = Ls.push(vj), o_sj = Ls.push(sj);
    const size_t o_aj = Ls.push(aj), o_cj = Ls.push(cj), o_pj = Ls.push(pj);
    if (int rc = upload(p, Ls.off, p->desc_dirty)) return rc;
    if (!join.empty()) {
        hipLaunchKernelGGL(pcg_init_kernel, dim3((unsigned)vj.size()), dim3(WGV), 0, st, p->dD,
                           Ls.dev_at<int2>(o_vj));
        launch_tl_fresh(p, Ls, o_aj, (unsigned)aj.size(), o_cj, (unsigned)cj.size(), o_pj, (unsigned)pj.size());
        hipLaunchKernelGGL(pcg_finalize_kernel, dim3((unsigned)sj.size()), dim3(WGV), 0, st, p->dD,
                           Ls.dev_at<int32_t>(o_sj), 0);
    }
    if (p->timing)
        if (int rc = ensure_events(p)) return rc;
    // (b) check_every iterations of every phase
    auto iterations = [&]() {
        for (int j = 0; j < check; j++) {
            if (p->timing) (void)hipEventRecord(p->ev[2 * j], st);
            // the step's first iteration takes p as it is (the last one of
            // the previous step formed it)
            const int first = j == 0 ? 1 : 0;
            for (const Group &g : gr) {
                if (g.kind >= K_MF && g.kind < K_FZ) launch_pcg_mf(g.kind, g.n, st, D, list(g.off), first);
                else launch_pcg_spmv(g.kind, g.lanes, g.n, g.Rmax, st, D, list(g.off), first);
            }
            if (p->timing) (void)hipEventRecord(p->ev[2 * j + 1], st);
            auto launch = [&](int k, auto kernel, int threads, auto... args) {
                if (nv[k])
                    hipLaunchKernelGGL(kernel, dim3(nv[k]), dim3(threads), 0, st, D, list(o_v[k]), args...);
            };
            launch(V_M, pcg_update_kernel<true, false, false>, WGV, first);
            launch(V_A, pcg_update_kernel<false, false, false>, WGV, first);
            launch(V_AF, pcg_update_kernel<false, false, true>, WGV, first);
            launch(V_AT, pcg_update_kernel<false, true, false>, WGV, first);
            launch(V_RS, tl_restrict_kernel, WGR, 0);
            launch(V_CW, tl_coarse_kernel, 256, 0);
            launch(j == check - 1 ? V_L : V_D, pcg_dir_kernel<false>, WGV);
            launch(V_T, pcg_dir_kernel<true>, WGV);
        }
    };
    // kernels of the step's iterations, and the host submissions that queue
    // them: one each kernel by kernel, one graph launch when captured
    auto has = [&](int k) { return (int64_t)(nv[k] ? 1 : 0); };
    const int64_t iter_kernels =
        (int64_t)check * ((int64_t)gr.size() + has(V_M) + has(V_A) + has(V_AF) + has(V_AT) + has(V_RS) + has(V_CW) + has(V_T)) +
        (check - 1) * has(V_D) + has(V_L);
    p->iter_kernels += iter_kernels;
    p->iter_submits += graph ? 1 : iter_kernels;
    // launching each member alone would take its own operator, update and
    // direction kernels (and restrict and coarse product, two-level) per
    // iteration; the direction only once per step where it is fused
    for (int s : act)
        p->member_kernels += p->hD[s].fuse ? 2 * (int64_t)check + 1 : (int64_t)check * (p->hD[s].tl ? (p->hD[s].cparts ? 4 : 5) : 3);
    if (!graph) {
        iterations();
    } else {
        std::vector<int64_t> key = {check, (int64_t)(intptr_t)p->dL};
        for (const auto &v : vl) key.push_back((int64_t)v.size());
        for (const Group &g : gr) key.insert(key.end(), {g.kind, g.lanes, g.Rmax, (int64_t)g.n});
        amr_pool::StepGraph *hit = nullptr;
        for (auto &g : p->graphs)
            if (g.key == key) hit = &g;
        if (!hit) {
            // capture the iterations once for these shapes (no memset nodes:
            // the kernels write every value they later read)
            AMR_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeRelaxed));
            iterations();
            const hipError_t le = hipGetLastError();
            hipGraph_t g = nullptr;
            const hipError_t ce = hipStreamEndCapture(st, &g);
            AMR_HIP(le);
            AMR_HIP(ce);
            hipGraphExec_t ex = nullptr;
            const hipError_t ie = hipGraphInstantiateWithFlags(&ex, g, 0);
            (void)hipGraphDestroy(g);
            AMR_HIP(ie);
            if (p->graphs.size() >= 8) {
                auto lru = std::min_element(p->graphs.begin(), p->graphs.end(),
                                            [](const auto &a, const auto &b) { return a.used < b.used; });
                AMR_HIP(hipStreamSynchronize(st));   // it may still be running
                (void)hipGraphExecDestroy(lru->exec);
                p->graphs.erase(lru);
            }
            p->graphs.push_back({key, ex, 0});
            hit = &p->graphs.back();
            p->graph_captures++;
        } else {
            p->graph_replays++;
        }
        hit->used = ++p->graph_clock;
        AMR_HIP(hipGraphLaunch(hit->exec, st));
    }
    AMR_HIP(hipGetLastError());
    const size_t sbytes = sizeof(double) * SEG_DBL * p->cap;
    AMR_HIP(hipMemcpyAsync(p->hS, p->dS, sbytes, hipMemcpyDeviceToHost, st));
    AMR_HIP(hipEventRecord(p->ev_step, st));
    p->fl_act = act;
    p->in_flight = true;
    return AMR_OK;
}

namespace {

int step_decide(amr_pool *p, std::vector<amr_pool_result> &out)
{
    const std::vector<int> act = p->fl_act;
    const int check = p->check;
    const double kEps = 2.220446049250313e-16, kFloorC = 64.0, kGrow = 1e4;
    const int kForceEvery = 256;
    hipStream_t st = p->stream;
    const size_t sbytes = sizeof(double) * SEG_DBL * p->cap;
    std::vector<std::vector<int2>> ent;
    std::vector<Group> gr;
    Lists Ls{p};
    size_t need = 0;

    // (b) decisions; residual replacement for members that stopped or whose
    // recursive residual dropped enough (mixed paths)
    int real_max = 0;
    std::vector<int> rep;
    for (int s : act) {
        Member &M = p->mem[s];
        const double *hs = p->hS + (size_t)s * SEG_DBL;
        const int32_t *hc = (const int32_t *)(hs + S_NSCAL);
        const int prev = M.state == M_JOIN ? 0 : M.iters;
        if (M.state == M_JOIN) {
            M.state = M_ACTIVE;
            M.bb = hs[S_BB];
            M.rr_ref = M.bb;
            if (M.bb == 0.0) {
                M.converged = 1;
                finish(p, s, out);
                continue;
            }
        }
        real_max = std::max(real_max, std::min(hc[C_ITERS] - prev, check));
        M.iters = hc[C_ITERS];
        M.broke = hc[C_BREAK];
        M.done = hc[C_DONE] != 0 || hc[C_STOP] != 0;
        // (after a step's last iteration pcg_dir_kernel forms it)
        M.unformed = p->hD[s].fuse && M.done && !M.broke && M.iters - prev < check;
        const double rr = hs[S_RR];
        const double ratio = M.o.replace_ratio > 0.0 ? M.o.replace_ratio : 0.1;
        // mixed: replace when the recursive residual fell by `ratio`, and
        // also when it rose far above the last true residual or no
        // replacement happened for a while, so that a refinement that does
        // not contract is seen (and abandoned) early
        const bool mixed_due = M.mixed && (rr <= ratio * ratio * M.rr_ref || rr > kGrow * M.rr_ref ||
                                           M.iters - M.last_rep >= kForceEvery);
        if (!(M.done || mixed_due)) {
            if (M.broke || M.iters >= M.o.maxiter) finish(p, s, out);
            continue;
        }
        M.rr_rec = rr;
        rep.push_back(s);
    }
    if (p->timing) {
        // the SpMVs of iterations in which some member was active executed
        for (int j = 0; j < real_max; j++) {
            float ms = 0.f;
            AMR_HIP(hipEventElapsedTime(&ms, p->ev[2 * j], p->ev[2 * j + 1]));
            p->t_spmv_ms += ms;
            p->n_spmv++;
        }
    }
    if (rep.empty()) return AMR_OK;

    // rt = b - K x in FP64 for the replacing members
    if (int rc = pool_begin_host_writes(p)) return rc;
    build_groups(p, rep, true, ent, gr);
    std::vector<int32_t> sr(rep.begin(), rep.end());
    need = padded(sr);
    for (const auto &e : ent) need += padded(e);
    if (int rc = pool_reserve_lists(p, need)) return rc;
    Ls.off = 0;
    const size_t o_sr = Ls.push(sr);
    {
        int gi = 0;
        for (const auto &e : ent)
            if (!e.empty()) gr[gi++].off = Ls.push(e);
    }
    if (int rc = upload(p, Ls.off, false)) return rc;
    for (const Group &g : gr) launch_residual(g.lanes, g.n, g.Rmax, st, p->dD, Ls.dev_at<int2>(g.off));
    hipLaunchKernelGGL(pcg_finalize_kernel, dim3((unsigned)sr.size()), dim3(WGV), 0, st, p->dD,
                       Ls.dev_at<int32_t>(o_sr), 1);
    AMR_HIP(hipGetLastError());
    AMR_HIP(hipMemcpyAsync(p->hS, p->dS, sbytes, hipMemcpyDeviceToHost, st));
    if (int rc = pool_sync(p)) return rc;

    std::vector<int> cont[REZ_NMODE];  // members to resume, by their direction (pcg_rez_kernel)
    std::vector<std::pair<int, double>> early;  // members stopped early, their next thresholds
    bool desc_changed = false;
    for (int s : rep) {
        Member &M = p->mem[s];
        const double *hs = p->hS + (size_t)s * SEG_DBL;
        M.replacements++;
        M.last_rep = M.iters;
        const double rr = hs[S_RR];
        M.relres = M.bb > 0.0 ? std::sqrt(rr / M.bb) : 0.0;
        const double floor2 = kFloorC * kFloorC * kEps * kEps * hs[S_KX];
        if (rr <= M.o.rtol * M.o.rtol * M.bb || rr <= floor2) {
            M.converged = 1;
            finish(p, s, out);
            continue;
        }
        if (!std::isfinite(rr) || M.iters >= M.o.maxiter) {
            finish(p, s, out);
            continue;
        }
        bool restart = M.broke != 0;
        const double drift = M.o.drift_limit > 0.0 ? M.o.drift_limit : 0.3;
        if (M.mixed && (hs[S_GAP] > drift * drift * std::max(rr, M.rr_rec) || rr > M.rr_true_prev)) {
            // the FP32 operator is too coarse for this model: the recursive
            // residual drifted from the true one, or the refinement stopped
            // contracting; finish on the FP64 operator
            M.mixed = false;
            M.fell_back = 1;
            restart = true;
        } else if (M.mf && (M.broke || M.replacements >= 2)) {
            // the recursion on the matrix-free operator stopped above the
            // tolerance twice, or broke down: finish on the assembled matrix,
            // whose residual decides
            M.mf = false;
            M.fell_back = 1;
            restart = true;
        } else if ((M.done && !M.broke && rr > 0.25 * M.rr_true_prev) || (M.broke && ++M.breakdowns > 3)) {
            finish(p, s, out);  // stagnation above both bounds, or repeated breakdown
            continue;
        }
        SegDesc &d = p->hD[s];
        const int f32 = M.mixed || (M.mf && M.pc32) ? 1 : 0, wp32 = (M.mixed && M.f32x) ? 1 : 0;
        if (d.f32 != f32 || d.wp32 != wp32 || (d.geo && !M.mf)) {
            d.f32 = f32;
            d.wp32 = wp32;
            if (!M.mf) {
                d.geo = nullptr;
                d.fuse = !d.tl && M.m->nnodes <= FUSE_MAX ? 1 : 0;
                d.npq = d.ntiles;
                if (d.tl) set_cparts(d, true);
            }
            desc_changed = true;
        }
        if (M.early > 0 && M.done && !M.broke) {
            M.early--;
            d.thr_fac = stop_factor(M);
            early.push_back({s, d.thr_fac * M.bb});
            desc_changed = true;
        }
        M.broke = 0;
        M.rr_true_prev = rr;
        M.rr_ref = rr;
        cont[restart ? REZ_RESTART : M.unformed ? REZ_FORM : REZ_KEEP].push_back(s);
    }
    // resume: r = rt, z = M r, the direction, rz, clear the stop flags
    std::vector<int2> vc[REZ_NMODE];
    std::vector<int32_t> sc;
    size_t nvc = 0;
    for (int k = 0; k < REZ_NMODE; k++) {
        vc[k] = vec_list(p, cont[k]);
        nvc += padded(vc[k]);
        sc.insert(sc.end(), cont[k].begin(), cont[k].end());
    }
    if (sc.empty()) return AMR_OK;
    for (const auto &e : early)
        AMR_HIP(hipMemcpyAsync(p->hD[e.first].scal + S_THR, &e.second, sizeof(double), hipMemcpyHostToDevice, st));
    if (!early.empty())
        if (int rc = pool_sync(p)) return rc;
    std::vector<int> call(sc.begin(), sc.end());
    std::vector<int2> ac = agg_list(p, call), cc = cw_list(p, call), pc = vec_list(p, tl_only(p, cont[REZ_RESTART]));
    if (int rc = pool_reserve_lists(p, nvc + padded(sc) + padded(ac) + padded(cc) + padded(pc))) return rc;
    Ls.off = 0;
    size_t o_vc[REZ_NMODE];
    for (int k = 0; k < REZ_NMODE; k++) o_vc[k] = Ls.push(vc[k]);
    const size_t o_sc = Ls.push(sc);
    const size_t o_ac = Ls.push(ac), o_cc = Ls.push(cc), o_pc = Ls.push(pc);
    if (int rc = upload(p, Ls.off, desc_changed || p->desc_dirty)) return rc;
    for (int k = 0; k < REZ_NMODE; k++)
        if (!vc[k].empty())
            hipLaunchKernelGGL(pcg_rez_kernel, dim3((unsigned)vc[k].size()), dim3(WGV), 0, st, p->dD,
                               Ls.dev_at<int2>(o_vc[k]), k);
    launch_tl_fresh(p, Ls, o_ac, (unsigned)ac.size(), o_cc, (unsigned)cc.size(), o_pc, (unsigned)pc.size());
    hipLaunchKernelGGL(pcg_finalize_kernel, dim3((unsigned)sc.size()), dim3(WGV), 0, st, p->dD,
                       Ls.dev_at<int32_t>(o_sc), 2);
    AMR_HIP(hipGetLastError());
    return AMR_OK;
}

}  // namespace

int amr_pool_step_collect(amr_pool *p, std::vector<amr_pool_result> &out)
{
    if (!p->in_flight) return AMR_OK;
    AMR_HIP(hipSetDevice(p->device));
    AMR_HIP(hipEventSynchronize(p->ev_step));
    p->in_flight = false;
    const size_t first = out.size();
    const int rc = step_decide(p, out);
    for (size_t i = first; i < out.size(); i++)
        if (out[i].m->stream != out[i].m->own_stream) p->leaving.push_back(out[i].m);
    return rc;
}

// The models that left the pool at its last step return to their own
// streams, after the work queued for them on the pool's stream so far.
int amr_pool_hand_back(amr_pool *p)
{
    if (p->leaving.empty()) return AMR_OK;
    AMR_HIP(hipSetDevice(p->device));
    for (amr_model *m : p->leaving)
        if (m->stream == p->stream && m->pool == p && !amr_pool_is_member(m))
            if (int rc = handoff(m, p->stream, m->own_stream)) return rc;
    p->leaving.clear();
    return AMR_OK;
}

int amr_pool_step_members(const amr_pool *p) { return p->in_flight ? (int)p->fl_act.size() : 0; }

int amr_pool_step_query(amr_pool *p, int *done)
{
    *done = 1;
    if (!p->in_flight) return AMR_OK;
    AMR_HIP(hipSetDevice(p->device));
    const hipError_t q = hipEventQuery(p->ev_step);
    if (q == hipErrorNotReady) {
        (void)hipGetLastError();  // not an error: clear it
        *done = 0;
        return AMR_OK;
    }
    AMR_HIP(q);
    return AMR_OK;
}

int amr_pool_run(amr_pool *p, std::vector<amr_pool_result> &out)
{
    if (int rc = amr_pool_step_launch(p)) return rc;
    return amr_pool_step_collect(p, out);
}

extern "C" int amr_test_early_stops(amr_model *m, int n, double rtol)
{
    if (!m || n < 0 || (n > 0 && !(rtol > 0.0 && rtol < 1.0))) return AMR_ERR_ARG;
    m->test_early = n;
    m->test_early_rtol = rtol;
    return AMR_OK;
}

extern "C" int amr_test_limits(amr_model *m, int tiles, int chunks)
{
    if (!m || tiles < 0 || tiles > MAX_GR || chunks < 0 || chunks > MAX_GV) return AMR_ERR_ARG;
    m->test_tiles = tiles;
    m->test_chunks = chunks;
    return AMR_OK;
}

int amr_pool_set_timing(amr_pool *p, int enable, double *ms, int64_t *n)
{
    if (enable && !p->timing) {
        p->t_spmv_ms = 0.0;
        p->n_spmv = 0;
    }
    p->timing = enable != 0;
    if (ms) *ms = p->t_spmv_ms;
    if (n) *n = p->n_spmv;
    return AMR_OK;
}

int amr_pool_graphs(amr_pool *p, int enable, int64_t *captures, int64_t *replays)
{
    if (enable >= 0) {
        if (p->in_flight) {
            amr_set_error("amr_pool_graphs: a step is in flight");
            return AMR_ERR_ARG;
        }
        p->use_graphs = enable != 0;
    }
    if (captures) *captures = p->graph_captures;
    if (replays) *replays = p->graph_replays;
    return AMR_OK;
}

int amr_pool_counts(amr_pool *p, int64_t *out)
{
    out[0] = p->coarse_batches;
    out[1] = p->coarse_formed;
    out[2] = p->iter_kernels;
    out[3] = p->iter_submits;
    out[4] = p->member_kernels;
    return AMR_OK;
}

// ------------------------------------------------- single-model wrappers

namespace {

int self_pool(amr_model *m, amr_pool **out)
{
    if (!m->self_pool) {
        if (int rc = amr_pool_new(&m->self_pool, m->device, 1, 32, m->stream)) return rc;
    }
    m->self_pool->stream = m->stream;
    *out = m->self_pool;
    return AMR_OK;
}

// SpMV lanes per block row.  Measured on MI355X: alone, a model's SpMV is
// fastest with 8 lanes below about 0.75M blocks and with 32 above 4M blocks,
// the choices in between within 10% of each other (64 lanes never best); in
// a pool, members with the same lanes and operand kind share one launch per
// iteration, and one lanes value for all (16) beat the per-model best by
// 8-10% on both pooled workloads (256 Tet10 cantilevers, 48 Hex8/Tet10
// boxes).  So: 16 lanes, 32 for the FP64 operator from 0.75M blocks (16
// lanes cost 20% more there) and for every operator from 4M blocks (the
// 811,923-DOF Hex20 block: 10% less time than with 16).
int choose_lanes(const amr_model *m, int kind)
{
    const int64_t nb = m->pat.nblk;
    return (nb >= 4 * 1024 * 1024 || (kind == K_F64 && nb >= 768 * 1024)) ? 32 : 16;
}

}  // namespace

// y = K x (mask_mode 0) or mask .* (K x) (mask_mode 1), FP64, node order.
int amr_spmv_full(amr_model *m, const double *x, double *y, int mask_mode)
{
    return amr_spmv_vals(m, m->Kv, x, y, mask_mode);
}

int amr_spmv_vals(amr_model *m, const double *vals, const double *x, double *y, int mask_mode)
{
    if (int rc = amr_choose_lanes(m)) return rc;
    const Geom g = model_geom(m);
    const size_t lds = tile_lds(g.R, 0);
#define AMR_SPMV(LN)                                                                                               \
    hipLaunchKernelGGL((spmv_kernel<LN>), dim3((unsigned)g.ntiles), dim3(WGS), lds, m->stream, m->nnodes, g.R,     \
                       m->rowptr, m->col, vals, x, y, m->mask, mask_mode)
    switch (m->lanes64) {
    case 8: AMR_SPMV(8); break;
    case 16: AMR_SPMV(16); break;
    case 32: AMR_SPMV(32); break;
    default: AMR_SPMV(64); break;
    }
#undef AMR_SPMV
    AMR_HIP(hipGetLastError());
    return AMR_OK;
}

// Lanes per row for the three operand kinds, unless set explicitly.  Every
// choice gives bit-identical results (see row_sum); the choice depends only
// on the matrix, so it needs no device work.
int amr_choose_lanes(amr_model *m)
{
    if (!m->lanes64) m->lanes64 = choose_lanes(m, K_F64);
    if (!m->lanes32) m->lanes32 = choose_lanes(m, K_F32);
    if (!m->lanes32d) m->lanes32d = choose_lanes(m, K_F32D);
    return AMR_OK;
}

// Time every lanes choice for the three operand kinds on this model's matrix
// and keep the fastest (explicit tuning; amr_choose_lanes is the default).
int amr_tune_lanes(amr_model *m)
{
    if (amr_pool_is_member(m)) {
        amr_set_error("the model is solving in a pool; tune it before adding it");
        return AMR_ERR_ARG;
    }
    amr_pool *p;
    if (int rc = self_pool(m, &p)) return rc;
    if (int rc = pool_begin_host_writes(p)) return rc;
    // a descriptor whose vectors are scratch: p = 1, q, x, r written freely
    Member &M = p->mem[0];
    M = Member();
    M.m = m;
    M.o.maxiter = 1 << 30;
    M.o.rtol = 1.0;
    M.b = m->v[5];
    M.x = m->v[6];
    fill_desc(p, 0);
    M = Member();  // not a solving member
    const Geom g = model_geom(m);
    std::vector<int2> tl;
    for (int t = 0; t < g.ntiles; t++) tl.push_back(make_int2(0, t));
    if (int rc = pool_reserve_lists(p, padded(tl))) return rc;
    Lists Ls{p};
    const size_t o = Ls.push(tl);
    if (int rc = upload(p, Ls.off, true)) return rc;
    p->desc_dirty = true;  // the next real member rewrites it
    const int64_t n = m->nnodes * 3;
    const unsigned gv = (unsigned)g.nvblk;
    AMR_HIP(hipMemsetAsync(p->dS, 0, sizeof(double) * SEG_DBL, p->stream));
    hipLaunchKernelGGL(fill_kernel, dim3(gv), dim3(WGV), 0, p->stream, n, m->v[3], 1.0);
    hipLaunchKernelGGL(fill_f32_kernel, dim3(gv), dim3(WGV), 0, p->stream, n, m->f[0], 1.0f);
    AMR_HIP(hipGetLastError());
    hipEvent_t e0, e1;
    AMR_HIP(hipEventCreate(&e0));
    AMR_HIP(hipEventCreate(&e1));
    int *dst[K_NKIND] = {&m->lanes64, &m->lanes32, &m->lanes32d};
    for (int kind = 0; kind < K_NKIND; kind++) {
        float best = 1e30f;
        int bestL = 64;
        for (int L : LANES) {
            launch_pcg_spmv(kind, L, (unsigned)g.ntiles, g.R, p->stream, p->dD, Ls.dev_at<int2>(o), 1);  // warm
            AMR_HIP(hipEventRecord(e0, p->stream));
            for (int rep = 0; rep < 3; rep++)
                launch_pcg_spmv(kind, L, (unsigned)g.ntiles, g.R, p->stream, p->dD, Ls.dev_at<int2>(o), 1);
            AMR_HIP(hipEventRecord(e1, p->stream));
            AMR_HIP(hipEventSynchronize(e1));
            float ms = 0.f;
            AMR_HIP(hipEventElapsedTime(&ms, e0, e1));
            if (ms < best) {
                best = ms;
                bestL = L;
            }
        }
        *dst[kind] = bestL;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    p->pending = false;  // the event waits above drained the stream
    return AMR_OK;
}

// Solve K11 x = b (node order, b zero at prescribed dofs), x FP64: a pool of
// one, stepped until the model leaves it.
int amr_pcg_solve(amr_model *m, const double *b, double *x, const amr_solve_opts *o, amr_solve_info *info)
{
    if (amr_pool_is_member(m)) {
        amr_set_error("the model is solving in a pool; wait for it to leave before solving it alone");
        return AMR_ERR_ARG;
    }
    amr_pool *p;
    if (int rc = amr_choose_lanes(m)) return rc;
    if (int rc = self_pool(m, &p)) return rc;
    p->check = std::max(1, std::min(o->check_every > 0 ? o->check_every : 32, 256));
    p->timing = m->timing;
    p->t_spmv_ms = 0.0;
    p->n_spmv = 0;
    if (int rc = amr_pool_join(p, m, b, x, o)) return rc;
    std::vector<amr_pool_result> res;
    while (res.empty()) {
        if (int rc = amr_pool_run(p, res)) {
            p->mem[0] = Member();
            return rc;
        }
    }
    if (m->timing) {
        m->t_spmv_ms += p->t_spmv_ms;
        m->n_spmv += p->n_spmv;
    }
    const amr_solve_info &r = res[0].info;
    if (info) *info = r;
    if (!r.converged) {
        char buf[256];
        snprintf(buf, sizeof buf, "PCG did not reach rtol=%.3e (relres %.3e after %d iterations, %d replacements)",
                 o->rtol, r.relres, r.iterations, r.refinements);
        amr_set_error(buf);
        return AMR_ERR_SOLVE;
    }
    return AMR_OK;
}

// ----------------------------------------------------------- stage vectors
namespace {

__global__ void inc_begin_kernel(int64_t n, double dT, double acr, int add, const double *__restrict__ Uex,
                                 const double *__restrict__ Fex, const double *__restrict__ Rc,
                                 double *__restrict__ dFex, double *__restrict__ R, double *__restrict__ dUa,
                                 double *__restrict__ dUi)
{
    for (int64_t i = (int64_t)blockIdx.x * WGV + threadIdx.x; i < n; i += (int64_t)gridDim.x * WGV) {
        double f = dT * Fex[i];
        if (add) f = f + acr * Rc[i];
        dFex[i] = f;
        R[i] = f;
        dUa[i] = 0.0;
        dUi[i] = dT * Uex[i];
    }
}

__global__ void prescribed_part_kernel(int64_t n, const double *__restrict__ mask, const double *__restrict__ u,
                                       double *__restrict__ u2)
{
    for (int64_t i = (int64_t)blockIdx.x * WGV + threadIdx.x; i < n; i += (int64_t)gridDim.x * WGV)
        u2[i] = mask[i] != 0.0 ? 0.0 : u[i];
}

__global__ void masked_diff_kernel(int64_t n, const double *__restrict__ mask, const double *__restrict__ a,
                                   const double *__restrict__ b, double *__restrict__ out)
{
    for (int64_t i = (int64_t)blockIdx.x * WGV + threadIdx.x; i < n; i += (int64_t)gridDim.x * WGV)
        out[i] = mask[i] != 0.0 ? a[i] - b[i] : 0.0;
}

__global__ void combine_kernel(int64_t n, const double *__restrict__ mask, const double *__restrict__ x,
                               double *__restrict__ u)
{
    for (int64_t i = (int64_t)blockIdx.x * WGV + threadIdx.x; i < n; i += (int64_t)gridDim.x * WGV)
        if (mask[i] != 0.0) u[i] = x[i];
}

__global__ void vadd_kernel(int64_t n, const double *__restrict__ a, const double *__restrict__ b,
                            double *__restrict__ out)
{
    for (int64_t i = (int64_t)blockIdx.x * WGV + threadIdx.x; i < n; i += (int64_t)gridDim.x * WGV) out[i] = a[i] + b[i];
}

__global__ void scale_kernel(int64_t n, double a, const double *__restrict__ x, double *__restrict__ out)
{
    for (int64_t i = (int64_t)blockIdx.x * WGV + threadIdx.x; i < n; i += (int64_t)gridDim.x * WGV) out[i] = a * x[i];
}

// flag = 1 if any entry of v is NaN (flag cleared by the caller)
__global__ void nan_flag_kernel(int64_t n, const double *__restrict__ v, int32_t *__restrict__ flag)
{
    bool any = false;
    for (int64_t i = (int64_t)blockIdx.x * WGV + threadIdx.x; i < n; i += (int64_t)gridDim.x * WGV)
        any = any || v[i] != v[i];
    if (__any(any) && threadIdx.x % 64 == 0) atomicOr(flag, 1);
}

// ΔUa += ΔUi; R = mask .* (ΔFex - ΔFin); per-workgroup max|R|, max|ΔUi|,
// max|ΔUa| and a NaN-in-ΔFin flag
__global__ void __launch_bounds__(WGV) nr_post_kernel(int64_t n, const double *__restrict__ mask,
                                                      const double *__restrict__ dFex,
                                                      const double *__restrict__ dFin,
                                                      const double *__restrict__ dUi, double *__restrict__ dUa,
                                                      double *__restrict__ R, double *__restrict__ part)
{
    double mr = 0.0, mi = 0.0, ma = 0.0, bad = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * WGV + threadIdx.x; i < n; i += (int64_t)gridDim.x * WGV) {
        const double ua = dUa[i] + dUi[i];
        dUa[i] = ua;
        const double fi = dFin[i];
        const double r = mask[i] != 0.0 ? dFex[i] - fi : 0.0;
        R[i] = r;
        if (fi != fi) bad = 1.0;
        mr = fmax(mr, fabs(r));
        mi = fmax(mi, fabs(dUi[i]));
        ma = fmax(ma, fabs(ua));
    }
    mr = block_max<WGV>(mr);
    mi = block_max<WGV>(mi);
    ma = block_max<WGV>(ma);
    bad = block_max<WGV>(bad);
    if (threadIdx.x == 0) {
        part[P_A + blockIdx.x] = mr;
        part[P_B + blockIdx.x] = mi;
        part[P_C + blockIdx.x] = ma;
        part[P_D + blockIdx.x] = bad;
    }
}

__global__ void __launch_bounds__(WGV) nr_finalize_kernel(int nv, const double *__restrict__ part,
                                                          int32_t *__restrict__ ctl, double *__restrict__ scal)
{
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    const int off[4] = {P_A, P_B, P_C, P_D};
    for (int i = threadIdx.x; i < nv; i += WGV)
        for (int k = 0; k < 4; k++) v[k] = fmax(v[k], part[off[k] + i]);
    for (int k = 0; k < 4; k++) v[k] = block_max<WGV>(v[k]);
    if (threadIdx.x == 0) {
        scal[S_RES] = v[0];
        scal[S_ERRN] = v[1];
        scal[S_ERRD] = v[2];
        ctl[C_NAN] = v[3] != 0.0;
    }
}

__global__ void commit_kernel(int64_t n, double acr, const double *__restrict__ dUa, const double *__restrict__ dFin,
                              const double *__restrict__ R, double *__restrict__ U, double *__restrict__ F,
                              double *__restrict__ Rc)
{
    for (int64_t i = (int64_t)blockIdx.x * WGV + threadIdx.x; i < n; i += (int64_t)gridDim.x * WGV) {
        U[i] += dUa[i];
        F[i] += dFin[i];
        Rc[i] = (1.0 - acr) * Rc[i] + R[i];
    }
}

int read_scalars(amr_model *m, double *hs, int32_t *hc)
{
    AMR_HIP(hipMemcpyAsync(hs, m->scal, sizeof(double) * S_NSCAL, hipMemcpyDeviceToHost, m->stream));
    AMR_HIP(hipMemcpyAsync(hc, m->scal + S_NSCAL, sizeof(int32_t) * C_NCTL, hipMemcpyDeviceToHost, m->stream));
    AMR_HIP(hipStreamSynchronize(m->stream));
    return AMR_OK;
}

unsigned vec_grid(const amr_model *m)
{
    const int64_t nv = (m->nnodes * 3 + WGV - 1) / WGV;
    return (unsigned)std::max<int64_t>(1, std::min<int64_t>(nv, MAX_GV));
}

}  // namespace

int amr_vec_inc_begin(amr_model *m, double dT, double acr, int add)
{
    double **v = m->sv;
    hipLaunchKernelGGL(inc_begin_kernel, dim3(vec_grid(m)), dim3(WGV), 0, m->stream, m->nnodes * 3, dT, acr, add,
                       v[SV_UEX], v[SV_FEX], v[SV_RC], v[SV_DFEX], v[SV_R], v[SV_DUA], v[SV_DUI]);
    AMR_HIP(hipGetLastError());
    return AMR_OK;
}

int amr_vec_fill(amr_model *m, double *x, double val)
{
    hipLaunchKernelGGL(fill_kernel, dim3(vec_grid(m)), dim3(WGV), 0, m->stream, m->nnodes * 3, x, val);
    AMR_HIP(hipGetLastError());
    return AMR_OK;
}

int amr_vec_fill_n(amr_model *m, double *x, int64_t n, double val)
{
    const int64_t g = std::max<int64_t>(1, std::min<int64_t>((n + WGV - 1) / WGV, 4 * MAX_GV));
    hipLaunchKernelGGL(fill_kernel, dim3((unsigned)g), dim3(WGV), 0, m->stream, n, x, val);
    AMR_HIP(hipGetLastError());
    return AMR_OK;
}

// b = mask .* (R - K (prescribed part of dUi)); u2/ky are scratch
int amr_vec_solve_prep(amr_model *m, const double *dUi, const double *R, double *u2, double *ky, double *b)
{
    const int64_t n = m->nnodes * 3;
    hipLaunchKernelGGL(prescribed_part_kernel, dim3(vec_grid(m)), dim3(WGV), 0, m->stream, n, m->mask, dUi, u2);
    AMR_HIP(hipGetLastError());
    int rc = amr_spmv_full(m, u2, ky, 0);
    if (rc) return rc;
    hipLaunchKernelGGL(masked_diff_kernel, dim3(vec_grid(m)), dim3(WGV), 0, m->stream, n, m->mask, R, ky, b);
    AMR_HIP(hipGetLastError());
    return AMR_OK;
}

int amr_vec_combine(amr_model *m, const double *x, double *dUi)
{
    hipLaunchKernelGGL(combine_kernel, dim3(vec_grid(m)), dim3(WGV), 0, m->stream, m->nnodes * 3, m->mask, x, dUi);
    AMR_HIP(hipGetLastError());
    return AMR_OK;
}

int amr_vec_scale(amr_model *m, double a, const double *x, double *out)
{
    hipLaunchKernelGGL(scale_kernel, dim3(vec_grid(m)), dim3(WGV), 0, m->stream, m->nnodes * 3, a, x, out);
    AMR_HIP(hipGetLastError());
    return AMR_OK;
}

int amr_vec_nan_flag(amr_model *m, const double *v, int32_t *flag)
{
    AMR_HIP(hipMemsetAsync(flag, 0, sizeof(int32_t), m->stream));
    hipLaunchKernelGGL(nan_flag_kernel, dim3(vec_grid(m)), dim3(WGV), 0, m->stream, m->nnodes * 3, v, flag);
    AMR_HIP(hipGetLastError());
    return AMR_OK;
}

int amr_vec_add(amr_model *m, const double *a, const double *b, double *out)
{
    hipLaunchKernelGGL(vadd_kernel, dim3(vec_grid(m)), dim3(WGV), 0, m->stream, m->nnodes * 3, a, b, out);
    AMR_HIP(hipGetLastError());
    return AMR_OK;
}

int amr_vec_nr_post(amr_model *m, double *res, double *dui_max, double *dua_max, int *nan_flag)
{
    double **v = m->sv;
    int32_t *ctl = (int32_t *)(m->scal + S_NSCAL);
    const unsigned g = vec_grid(m);
    hipLaunchKernelGGL(nr_post_kernel, dim3(g), dim3(WGV), 0, m->stream, m->nnodes * 3, m->mask, v[SV_DFEX],
                       v[SV_DFIN], v[SV_DUI], v[SV_DUA], v[SV_R], m->part);
    hipLaunchKernelGGL(nr_finalize_kernel, dim3(1), dim3(WGV), 0, m->stream, (int)g, m->part, ctl, m->scal);
    AMR_HIP(hipGetLastError());
    double hs[S_NSCAL];
    int32_t hc[C_NCTL];
    if (int rc = read_scalars(m, hs, hc)) return rc;
    *res = hs[S_RES];
    *dui_max = hs[S_ERRN];
    *dua_max = hs[S_ERRD];
    *nan_flag = hc[C_NAN];
    return AMR_OK;
}

// The same as amr_vec_nr_post without waiting: the scalars are copied into
// hs/hc (pinned host memory) in stream order
int amr_vec_nr_post_async(amr_model *m, double *hs, int32_t *hc)
{
    double **v = m->sv;
    int32_t *ctl = (int32_t *)(m->scal + S_NSCAL);
    const unsigned g = vec_grid(m);
    hipLaunchKernelGGL(nr_post_kernel, dim3(g), dim3(WGV), 0, m->stream, m->nnodes * 3, m->mask, v[SV_DFEX],
                       v[SV_DFIN], v[SV_DUI], v[SV_DUA], v[SV_R], m->part);
    hipLaunchKernelGGL(nr_finalize_kernel, dim3(1), dim3(WGV), 0, m->stream, (int)g, m->part, ctl, m->scal);
    AMR_HIP(hipGetLastError());
    AMR_HIP(hipMemcpyAsync(hs, m->scal, sizeof(double) * S_NSCAL, hipMemcpyDeviceToHost, m->stream));
    AMR_HIP(hipMemcpyAsync(hc, m->scal + S_NSCAL, sizeof(int32_t) * C_NCTL, hipMemcpyDeviceToHost, m->stream));
    return AMR_OK;
}

int amr_nr_post_slots(int *res, int *errn, int *errd, int *nan)
{
    *res = S_RES;
    *errn = S_ERRN;
    *errd = S_ERRD;
    *nan = C_NAN;
    return AMR_OK;
}

int amr_vec_commit(amr_model *m)
{
    double **v = m->sv;
    hipLaunchKernelGGL(commit_kernel, dim3(vec_grid(m)), dim3(WGV), 0, m->stream, m->nnodes * 3, m->acr, v[SV_DUA],
                       v[SV_DFIN], v[SV_R], v[SV_U], v[SV_F], v[SV_RC]);
    AMR_HIP(hipGetLastError());
    return AMR_OK;
}
