// Device solve of an assembled system (kernels).
//
// x_A = A^-1 (b_A - D x_D) with x_D the Dirichlet values (mat::eliminate,
// src/formulation/mat.cpp:78-103; the reference then factorizes with MUMPS,
// src/expression/operation/sl.cpp:1565-1627).  Here: FP64 iterative
// refinement (FP64 CSR residuals) around a Jacobi-preconditioned FP32
// conjugate-gradient inner solve, for symmetric positive definite A.
//
// One inner iteration is three kernels:
//   K1  q = A p (FP32 values),             partials of p.q
//   K2  d += a p, r -= a q, z = r / diag,  partials of r.z and r.r  (a = rz / pq)
//   K3  p = z + beta p                     (beta = rz' / rz)
// The partials are summed, in one order, by every block that needs the scalar
// (at most SLX_SOLVE_BLOCKS values from the L2) instead of by one-block kernels
// between them: at 16^3 x 6 P2 elasticity those took 10 of 44 us an iteration.
// Every reduction is deterministic: a grid fixed by the system's sizes, partial
// sums in a fixed order, and fixed lanes per row for the products.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cmath>
#include <vector>
#include "solve.h"

namespace slx {

enum { SC_PQ = 1, SC_RR = 3, SC_DOT = 5 };

// block sum of one double per thread (256 threads); result valid in thread 0
__device__ inline double block_sum(double v, double* sh) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = 0.0;
    if (threadIdx.x == 0) s = (sh[0] + sh[1]) + (sh[2] + sh[3]);
    __syncthreads();
    return s;
}

// ordered sum of n partials, in every thread of a 256-thread block
__device__ inline double all_sum(const double* __restrict__ part, int n, double* sh) {
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) s += part[i];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
    __syncthreads();
    const double t = (sh[0] + sh[1]) + (sh[2] + sh[3]);
    __syncthreads();
    return t;
}

// y[r] = c0 f[r] - c1 (A x)[r] over one CSR matrix, LPR lanes per row (the
// lanes of a row group share r, so the width-LPR shuffles stay inside
// active lanes)
template <int LPR, typename VT, typename XT, typename YT>
__global__ void __launch_bounds__(256) spmv_kernel(int64_t nrows, const int64_t* __restrict__ rowp, const int32_t* __restrict__ col,
                                                   const VT* __restrict__ val, const XT* __restrict__ x, const YT* f, YT c0, YT c1, YT* y) {
    const int l = threadIdx.x % LPR;
    const int64_t rstride = (int64_t)gridDim.x * (256 / LPR);
    for (int64_t r = (int64_t)blockIdx.x * (256 / LPR) + threadIdx.x / LPR; r < nrows; r += rstride) {
        YT s = 0;
        const int64_t e = rowp[r + 1];
        for (int64_t k = rowp[r] + l; k < e; k += LPR) s += (YT)val[k] * (YT)x[col[k]];
#pragma unroll
        for (int o = LPR / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, LPR);
        if (l == 0) y[r] = (f ? c0 * f[r] : (YT)0) - c1 * s;
    }
}

// lanes per row from the mean row length (a few products per lane)
static int spmv_lpr(int64_t nrows, int64_t nnz) {
    const double avg = nrows ? (double)nnz / (double)nrows : 0.0;
    if (avg >= 96) return 32;
    if (avg >= 40) return 16;
    if (avg >= 16) return 8;
    if (avg >= 6) return 4;
    return 2;
}

template <typename VT, typename XT, typename YT>
static void spmv(int64_t nrows, int64_t nnz, const int64_t* rowp, const int32_t* col, const VT* val, const XT* x, const YT* f, YT c0,
                 YT c1, YT* y, hipStream_t st) {
    if (nrows <= 0) return;
    const int lpr = spmv_lpr(nrows, nnz);
    const unsigned grid = (unsigned)std::min<int64_t>((nrows * lpr + 255) / 256, 1 << 20);
#define SLX_SPMV_CASE(L)                                                                                                          \
    case L:                                                                                                                       \
        hipLaunchKernelGGL((spmv_kernel<L, VT, XT, YT>), dim3(grid), dim3(256), 0, st, nrows, rowp, col, val, x, f, c0, c1, y);       \
        break;
    switch (lpr) {
        SLX_SPMV_CASE(2)
        SLX_SPMV_CASE(4)
        SLX_SPMV_CASE(8)
        SLX_SPMV_CASE(16)
        SLX_SPMV_CASE(32)
    }
#undef SLX_SPMV_CASE
}

// q = A p over FP32 values, streamed by row blocks: a block loads the
// nonzeros of its rows with coalesced loads, keeps the products in LDS
// and reduces each row from there (lanes per row from the rows in the block);
// a row longer than SLX_STREAM_NNZ is summed by the whole block.  The fixed
// grid walks the row blocks; each block writes its partial sum of p.q.
// Workgroups are dispatched round-robin over the 8 XCDs (workgroup w on XCD
// w % 8): each XCD takes one contiguous eighth of the row blocks, so the
// entries of x its rows gather stay within a range its own L2 can hold.
__global__ void __launch_bounds__(256) spmv_stream_f32(int64_t nblk, const int64_t* __restrict__ rblk, const int64_t* __restrict__ rowp,
                                                       const int32_t* __restrict__ col, const float* __restrict__ val, int64_t nnz,
                                                       const float* __restrict__ x, float* __restrict__ y, double* __restrict__ part) {
    __shared__ float prod[SLX_STREAM_NNZ];
    __shared__ double sh[4];
    double acc = 0.0;
    const int xcd = blockIdx.x % SLX_XCDS;
    const int64_t b_end = nblk * (xcd + 1) / SLX_XCDS;
    for (int64_t b = nblk * xcd / SLX_XCDS + blockIdx.x / SLX_XCDS; b < b_end; b += gridDim.x / SLX_XCDS) {
        const int64_t r0 = rblk[b], r1 = rblk[b + 1];
        const int64_t k0 = rowp[r0], k1 = rowp[r1];
        if (k1 - k0 > SLX_STREAM_NNZ) {
            // one long row (block-uniform branch)
            double s = 0.0;
            for (int64_t k = k0 + threadIdx.x; k < k1; k += 256) s += (double)(val[k] * x[col[k]]);
            const double t = block_sum(s, sh);
            if (threadIdx.x == 0) {
                y[r0] = (float)t;
                acc += (double)x[r0] * (double)(float)t;
            }
            continue;
        }
        // consecutive lanes take consecutive nonzeros: the x entries one
        // wave gathers then share cache lines more often than with 16-byte
        // loads per lane (measured: 1.54 vs 1.75 ms per product, 64^3 P2 elasticity)
        const int64_t kb = k0;
        for (int64_t k = k0 + threadIdx.x; k < k1; k += 256) prod[k - k0] = val[k] * x[col[k]];
        __syncthreads();
        const int rows = (int)(r1 - r0);
        int lpr = 32;
        while (lpr > 1 && rows * lpr > 256) lpr >>= 1;
        const int g = threadIdx.x / lpr, l = threadIdx.x % lpr;
        for (int rr = g; rr < rows; rr += 256 / lpr) {
            const int a = (int)(rowp[r0 + rr] - kb), e = (int)(rowp[r0 + rr + 1] - kb);
            float s = 0.f;
            for (int k = a + l; k < e; k += lpr) s += prod[k];
            for (int o = lpr / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, lpr);
            if (l == 0) {
                y[r0 + rr] = s;
                acc += (double)x[r0 + rr] * (double)s;
            }
        }
        __syncthreads();
    }
    const double t = block_sum(acc, sh);
    if (threadIdx.x == 0) part[blockIdx.x] = t;
}

// q = A p over FP32 values, LPR lanes per row, U nonzeros of a lane in
// flight at once (values and columns, then the eight gathers): the product of
// the inner iterations for rows of ordinary length.  The streaming kernel
// above waits for its row block's loads, the LDS exchange and the row sums in
// turn: 26.9 us at 16^3 x 6 P2 elasticity (8.5e6 nonzeros, 81 a row), 23.9 us
// here, bound by the L1's line accesses (1.3e7, most of them gathers of x).
// Rows go to the XCDs in contiguous eighths, as above.
template <int LPR, int U>
__global__ void __launch_bounds__(512) spmv_rows_f32(int64_t nrows, const int64_t* __restrict__ rowp, const int32_t* __restrict__ col,
                                                     const float* __restrict__ val, const float* __restrict__ x, float* __restrict__ y,
                                                     double* __restrict__ part) {
    constexpr int RPB = 512 / LPR;
    __shared__ double sh[8];
    const int l = threadIdx.x % LPR, g = threadIdx.x / LPR;
    const int xcd = blockIdx.x % SLX_XCDS;
    const int64_t nb = (nrows + RPB - 1) / RPB, b_end = nb * (xcd + 1) / SLX_XCDS;
    double acc = 0.0;
    for (int64_t b = nb * xcd / SLX_XCDS + blockIdx.x / SLX_XCDS; b < b_end; b += gridDim.x / SLX_XCDS) {
        const int64_t r = b * RPB + g;
        if (r < nrows) {
            const int64_t k0 = rowp[r];
            const int n = (int)(rowp[r + 1] - k0);
            float s = 0.f;
            for (int k = l; k < n; k += U * LPR) {
                float v[U], xv[U];
                int c[U];
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const int kk = k + u * LPR;
                    const int64_t at = k0 + (kk < n ? kk : k);
                    v[u] = kk < n ? val[at] : 0.f;
                    c[u] = col[at];
                }
#pragma unroll
                for (int u = 0; u < U; u++) xv[u] = x[c[u]];
#pragma unroll
                for (int u = 0; u < U; u++) s += v[u] * (k + u * LPR < n ? xv[u] : 0.f);
            }
#pragma unroll
            for (int o = LPR / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, LPR);
            if (l == 0) {
                y[r] = s;
                acc += (double)x[r] * (double)s;
            }
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
#pragma unroll
        for (int i = 0; i < 8; i++) t += sh[i];
        part[blockIdx.x] = t;
    }
}

// The FP32 product of the inner iterations.  The row kernel takes
//  - rows of at most SLX_ROWS_MAX nonzeros, or of 64 and 256 where one lane and
//    two walk a row: a long row is a chain of loads there.  With 1 % of the rows
//    512 long, 4e5 rows of 5: 91 us, streaming 41; 2e4 rows of 20 (four lanes):
//    20 us, streaming 36.
//  - rows of nearly one length (the longest up to 1.5 times the mean) of any
//    number, others up to SLX_ROWS_SMALL of them and SLX_ROWS_AREA: with short and
//    long rows in a wave its loads spread over more lines than the caches of many
//    rows in flight hold, where the streaming kernel reads in one sweep.
// Whole CG iterations, us, row kernel and streaming: P1 2D Poisson 3.6e5 rows 24.6
// and 26.7, P2 elasticity 1.2e5 rows 42.8 and 50, 3.5e5 88 and 79, 2.7e6 833 and
// 668, orders 1 to 5 of hexahedra 2.3e4 rows 32 and 38, 8.5e4 84 and 59, P3 2D Poisson 9.8e5
// rows 106 and 71.
// *npart: partial sums of x.y written, at most SLX_STREAM_BLOCKS and at most
// nrows of them where they are more than SLX_SOLVE_BLOCKS.
static hipError_t inner_product(int64_t nrows, int64_t nnz, int max_row, int64_t nblk, const int64_t* blk, const int64_t* rowp,
                                const int32_t* col, const float* val, const float* x, float* y, double* part, int* npart, hipStream_t st) {
    // the fewest lanes whose batches of six or eight hold the mean row
    const int64_t avg = nrows ? (nnz + nrows - 1) / nrows : 1;
    int lpr = 1;
    while (lpr < 32 && lpr * 8 < avg) lpr *= 2;
    if (max_row > std::min(SLX_ROWS_MAX, 64 * lpr * lpr) || (2 * (int64_t)max_row > 3 * avg && (nrows > SLX_ROWS_SMALL || nrows * max_row > SLX_ROWS_AREA))) {
        // eight blocks on a CU: four took 124 us where eight take 84 (5e5 rows of 60)
        int64_t grid = std::min<int64_t>(SLX_STREAM_BLOCKS, (nblk + SLX_XCDS - 1) / SLX_XCDS * SLX_XCDS);
        if (grid > nrows) grid = std::min<int64_t>(grid, SLX_SOLVE_BLOCKS);
        *npart = (int)grid;
        hipLaunchKernelGGL(spmv_stream_f32, dim3((unsigned)grid), dim3(256), 0, st, nblk, blk, rowp, col, val, nnz, x, y, part);
        return hipGetLastError();
    }
    const bool six = lpr * 6 >= avg;
    const int64_t blocks = (nrows * lpr + 511) / 512;
    const unsigned grid = (unsigned)std::min<int64_t>(SLX_SOLVE_BLOCKS, (blocks + SLX_XCDS - 1) / SLX_XCDS * SLX_XCDS);
    *npart = (int)grid;
#define SLX_ROWS_CASE(L)                                                                                                          \
    case L:                                                                                                                       \
        if (six) hipLaunchKernelGGL((spmv_rows_f32<L, 6>), dim3(grid), dim3(512), 0, st, nrows, rowp, col, val, x, y, part);      \
        else hipLaunchKernelGGL((spmv_rows_f32<L, 8>), dim3(grid), dim3(512), 0, st, nrows, rowp, col, val, x, y, part);          \
        break;
    switch (lpr) {
        SLX_ROWS_CASE(1)
        SLX_ROWS_CASE(2)
        SLX_ROWS_CASE(4)
        SLX_ROWS_CASE(8)
        SLX_ROWS_CASE(16)
        SLX_ROWS_CASE(32)
    }
#undef SLX_ROWS_CASE
    return hipGetLastError();
}

void stream_row_blocks(const int64_t* rowp, int64_t nrows, std::vector<int64_t>& out) {
    out.clear();
    out.push_back(0);
    int64_t r = 0;
    while (r < nrows) {
        int64_t e = r;
        while (e < nrows && e - r < 256 && rowp[e + 1] - rowp[r] <= SLX_STREAM_NNZ) e++;
        if (e == r) e = r + 1;
        out.push_back(e);
        r = e;
    }
}

__global__ void gather_kernel(int64_t n, const int64_t* __restrict__ idx, const double* __restrict__ src, double* __restrict__ dst) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[idx[i]];
}

__global__ void scatter_kernel(int64_t n, const int64_t* __restrict__ idx, const double* __restrict__ src, double* __restrict__ dst) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[idx[i]] = src[i];
}

// Jacobi preconditioner (FP32) and the FP32 copy of the matrix values, 16
// lanes per row (one row per lane read the values a row apart: 0.29 ms
// instead of 0.03 at 16^3 x 6 P2 elasticity)
__global__ void __launch_bounds__(256) prep_kernel(int64_t nrows, const int64_t* __restrict__ rowp, const int32_t* __restrict__ col,
                                                   const double* __restrict__ val, float* __restrict__ val32, float* __restrict__ dinv) {
    const int64_t r = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / 16;
    if (r >= nrows) return;
    const int l = threadIdx.x % 16;
    double d = 0.0;
    for (int64_t k = rowp[r] + l; k < rowp[r + 1]; k += 16) {
        const double v = val[k];
        val32[k] = (float)v;
        if (col[k] == r) d = v;
    }
    // the diagonal sits in one lane; the others hold zero
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) d += __shfl_xor(d, o, 16);
    if (l == 0) dinv[r] = d != 0.0 ? (float)(1.0 / d) : 1.0f;
}

// partials of a.b (FP64 accumulation) over the fixed grid
template <typename T>
__global__ void __launch_bounds__(256) dot_partial(int64_t n, const T* __restrict__ a, const T* __restrict__ b, double* __restrict__ part) {
    __shared__ double sh[4];
    double s = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) s += (double)a[i] * (double)b[i];
    const double t = block_sum(s, sh);
    if (threadIdx.x == 0) part[blockIdx.x] = t;
}

// sc[out] = ordered sum of n partials
__global__ void __launch_bounds__(256) sum_partials(const double* __restrict__ part, int n, int out, double* __restrict__ sc) {
    __shared__ double sh[4];
    const double t = all_sum(part, n, sh);
    if (threadIdx.x == 0) sc[out] = t;
}

// inner start: r32 = r, z = r / diag, p = z, d = 0; partials of r.z and r.r
__global__ void __launch_bounds__(256) pcg_start(int64_t n, const double* __restrict__ r, const float* __restrict__ dinv,
                                                 float* __restrict__ r32, float* __restrict__ z, float* __restrict__ p,
                                                 float* __restrict__ d, double* __restrict__ prz, double* __restrict__ prr) {
    __shared__ double sh[4];
    double rz = 0.0, rr = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        const float rv = (float)r[i];
        const float zv = dinv[i] * rv;
        r32[i] = rv;
        z[i] = zv;
        p[i] = zv;
        d[i] = 0.f;
        rz += (double)rv * (double)zv;
        rr += (double)rv * (double)rv;
    }
    const double a = block_sum(rz, sh);
    const double b = block_sum(rr, sh);
    if (threadIdx.x == 0) {
        prz[blockIdx.x] = a;
        prr[blockIdx.x] = b;
    }
}

// d += a p ; r -= a q ; z = r / diag   (a = rz / pq, summed from their
// partials); partials of the new r.z and r.r
__global__ void __launch_bounds__(256) pcg_update(int64_t n, const double* __restrict__ ppq, int npq, const double* __restrict__ prz,
                                                  int nrz, float* __restrict__ d, float* __restrict__ r, const float* __restrict__ p,
                                                  const float* __restrict__ q, const float* __restrict__ dinv, float* __restrict__ z,
                                                  double* __restrict__ prz_new, double* __restrict__ prr) {
    __shared__ double sh[4];
    const double pq = all_sum(ppq, npq, sh), rz0 = all_sum(prz, nrz, sh);
    const float alpha = pq != 0.0 ? (float)(rz0 / pq) : 0.f;
    double rz = 0.0, rr = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        d[i] += alpha * p[i];
        const float rv = r[i] - alpha * q[i];
        const float zv = dinv[i] * rv;
        r[i] = rv;
        z[i] = zv;
        rz += (double)rv * (double)zv;
        rr += (double)rv * (double)rv;
    }
    const double a = block_sum(rz, sh);
    const double b = block_sum(rr, sh);
    if (threadIdx.x == 0) {
        prz_new[blockIdx.x] = a;
        prr[blockIdx.x] = b;
    }
}

// p = z + beta p   (beta = rz' / rz)
__global__ void __launch_bounds__(256) pcg_direction(int64_t n, const double* __restrict__ prz_new, const double* __restrict__ prz, int nrz,
                                                     const float* __restrict__ z, float* __restrict__ p) {
    __shared__ double sh[4];
    const double rzn = all_sum(prz_new, nrz, sh), rz = all_sum(prz, nrz, sh);
    const float beta = rz != 0.0 ? (float)(rzn / rz) : 0.f;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) p[i] = z[i] + beta * p[i];
}

__global__ void to_f32(int64_t n, const double* __restrict__ a, float* __restrict__ b) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) b[i] = (float)a[i];
}

__global__ void add_f32_to_f64(int64_t n, const float* __restrict__ d, double* __restrict__ x) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] += (double)d[i];
}

static unsigned blocks(int64_t n) { return (unsigned)((n + 255) / 256); }

// ---- GMRES (FP32 vectors, FP64 sums) ----

// One iteration is six kernels and no host work: q = A (dinv v_j), twice the
// dots with the basis and the subtraction, then the norm, v_{j+1} and the
// Givens rotations.  The host reads the residual history every
// SLX_GMRES_CHECK iterations and drops the ones past convergence (columns of
// H up to there do not depend on later ones).  Before, each iteration waited
// for the host three times and the dots ran a 2048-block grid over one basis
// vector after the other: 225 us an iteration at 4e3 rows, 30 us now.

// partials of V_i . w: block (c, g) takes chunk c of the rows for the four
// vectors 4 g .. 4 g + 3; part[i * gridDim.x + c]
__global__ void __launch_bounds__(256) basis_dots(int64_t n, int64_t chunk, const float* __restrict__ V, int nv, const float* __restrict__ w,
                                                  double* __restrict__ part) {
    __shared__ double sh[4];
    const int i0 = 4 * blockIdx.y;
    const int64_t k0 = blockIdx.x * chunk, k1 = min(n, k0 + chunk);
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    const float* v[4];
#pragma unroll
    for (int u = 0; u < 4; u++) v[u] = V + (size_t)min(i0 + u, nv - 1) * n;
    for (int64_t k = k0 + threadIdx.x; k < k1; k += 256) {
        const double wk = (double)w[k];
#pragma unroll
        for (int u = 0; u < 4; u++) s[u] += (double)v[u][k] * wk;
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const double t = block_sum(s[u], sh);
        if (threadIdx.x == 0 && i0 + u < nv) part[(size_t)(i0 + u) * gridDim.x + blockIdx.x] = t;
    }
}

// out[i] = ordered sum of partial row i (one block per row)
__global__ void __launch_bounds__(256) sum_rows(const double* __restrict__ part, int n, double* __restrict__ out) {
    __shared__ double sh[4];
    const double t = all_sum(part + (size_t)blockIdx.x * n, n, sh);
    if (threadIdx.x == 0) out[blockIdx.x] = t;
}

// w -= sum_i h_i V_i, h_i the ordered sum of its np partials; 64 rows per block
// step, four groups of the vectors side by side.  Block 0 keeps h in hcol
// (add: on top of the first pass's); partials of w.w
__global__ void __launch_bounds__(256) basis_update(int64_t n, const float* __restrict__ V, int nv, const double* __restrict__ part, int np,
                                                    int add, double* __restrict__ hcol, float* __restrict__ w, double* __restrict__ pnorm) {
    __shared__ float h[SLX_GMRES_MAX + 4];
    __shared__ float red[4][64];
    __shared__ double sh[4];
    const int t = threadIdx.x;
    for (int i = t; i < nv; i += 256) {
        double s = 0.0;
        for (int c = 0; c < np; c++) s += part[(size_t)i * np + c];
        h[i] = (float)s;
        if (blockIdx.x == 0) hcol[i] = add ? hcol[i] + s : s;
    }
    __syncthreads();
    const int l = t & 63, g = t >> 6, i0 = nv * g / 4, i1 = nv * (g + 1) / 4;
    double nn = 0.0;
    for (int64_t b = blockIdx.x; b * 64 < n; b += gridDim.x) {
        const int64_t k = b * 64 + l;
        float acc = 0.f;
        if (k < n) {
            int i = i0;
            for (; i + 8 <= i1; i += 8) {
                float v[8];
#pragma unroll
                for (int u = 0; u < 8; u++) v[u] = V[(size_t)(i + u) * n + k];
#pragma unroll
                for (int u = 0; u < 8; u++) acc += h[i + u] * v[u];
            }
            for (; i < i1; i++) acc += h[i] * V[(size_t)i * n + k];
        }
        red[g][l] = acc;
        __syncthreads();
        if (g == 0 && k < n) {
            const float wk = w[k] - ((red[0][l] + red[1][l]) + (red[2][l] + red[3][l]));
            w[k] = wk;
            nn += (double)wk * (double)wk;
        }
        __syncthreads();
    }
    const double s = block_sum(nn, sh);
    if (t == 0) pnorm[blockIdx.x] = s;
}

// v = w / |w| (zero when w is), z = dinv .* v; with j >= 0 block 0 also rotates
// column j of H (hcol: j + 1 entries, then |w|) and stores |g_{j+1}| and |w|
__global__ void __launch_bounds__(256) basis_next(int64_t n, const double* __restrict__ pnorm, int np, const float* __restrict__ w,
                                                  const float* __restrict__ dinv, float* __restrict__ v, float* __restrict__ z, int j,
                                                  double* __restrict__ hcol, double* __restrict__ cs, double* __restrict__ sn,
                                                  double* __restrict__ gv, double* __restrict__ hist) {
    __shared__ double sh[4];
    __shared__ double hl[SLX_GMRES_MAX + 1], cl[SLX_GMRES_MAX], sl[SLX_GMRES_MAX];
    const double nrm = sqrt(all_sum(pnorm, np, sh));
    const float inv = nrm > 0.0 ? (float)(1.0 / nrm) : 0.f;
    for (int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x; k < n; k += (int64_t)gridDim.x * 256) {
        const float x = inv * w[k];
        v[k] = x;
        z[k] = dinv[k] * x;
    }
    if (blockIdx.x != 0) return;
    if (j < 0) {
        if (threadIdx.x == 0) {
            gv[0] = nrm;
            hist[0] = nrm;
        }
        return;
    }
    for (int i = threadIdx.x; i <= j; i += 256) {
        hl[i] = hcol[i];
        if (i < j) {
            cl[i] = cs[i];
            sl[i] = sn[i];
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 0; i < j; i++) {
            const double a = hl[i], b = hl[i + 1];
            hl[i] = cl[i] * a + sl[i] * b;
            hl[i + 1] = -sl[i] * a + cl[i] * b;
        }
        const double a = hl[j], b = nrm, rr = hypot(a, b);
        const double c = rr > 0.0 ? a / rr : 1.0, s = rr > 0.0 ? b / rr : 0.0;
        hl[j] = rr;
        cs[j] = c;
        sn[j] = s;
        const double g = gv[j];
        gv[j + 1] = -s * g;
        gv[j] = c * g;
        hist[2 * j] = fabs(s * g);
        hist[2 * j + 1] = nrm;
    }
    __syncthreads();
    for (int i = threadIdx.x; i <= j; i += 256) hcol[i] = hl[i];
}

// d = dinv .* sum_i y_i V_i   (right preconditioning)
__global__ void basis_combine(int64_t n, const float* __restrict__ V, int nv, const double* __restrict__ y, const float* __restrict__ dinv,
                              float* __restrict__ d) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    float acc = 0.f;
    for (int i = 0; i < nv; i++) acc += (float)y[i] * V[(size_t)i * n + k];
    d[k] = dinv[k] * acc;
}

// position of column c in CSR row r (sorted columns), or -1
__device__ inline int64_t find_col(const int64_t* __restrict__ rowp, const int32_t* __restrict__ col, int64_t r, int64_t c) {
    int64_t lo = rowp[r], hi = rowp[r + 1];
    while (lo < hi) {
        const int64_t mid = (lo + hi) / 2;
        if (col[mid] < c) lo = mid + 1;
        else hi = mid;
    }
    return (lo < rowp[r + 1] && col[lo] == c) ? lo : -1;
}

// any entry a_rc whose transpose partner a_cr is missing or differs by more
// than 1e-5 (|a_rc| + |a_cr|) + 1e-6 (|a_rr| + |a_cc|) sets *flag (every
// writer stores 1); the diagonal term keeps rounding noise (FP64, or the
// 1e-7 of the mixed-precision element matrices) on entries that cancel to
// almost zero from counting as asymmetry.  SLX_SYM_LPR lanes share a row
// (one entry each per step), so the binary searches of a row run side by side.
#define SLX_SYM_LPR 16
__global__ void __launch_bounds__(256) sym_kernel(int64_t n, const int64_t* __restrict__ rowp, const int32_t* __restrict__ col,
                                                  const double* __restrict__ val, int* __restrict__ flag) {
    const int64_t r = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / SLX_SYM_LPR;
    const int l = threadIdx.x % SLX_SYM_LPR;
    if (r >= n) return;
    const int64_t kd = find_col(rowp, col, r, r);
    const double drr = kd >= 0 ? fabs(val[kd]) : 0.0;
    bool bad = false;
    for (int64_t k = rowp[r] + l; k < rowp[r + 1] && !bad; k += SLX_SYM_LPR) {
        const int32_t c = col[k];
        const int64_t kt = find_col(rowp, col, c, r);
        if (kt < 0) {
            bad = true;
        } else {
            // the partner's diagonal only where the rest of the bound does not settle it
            const double diff = fabs(val[k] - val[kt]), lim = 1e-5 * (fabs(val[k]) + fabs(val[kt])) + 1e-6 * drr;
            if (!(diff <= lim)) {
                const int64_t kc = find_col(rowp, col, c, c);
                const double dcc = kc >= 0 ? fabs(val[kc]) : 0.0;
                bad = diff > 1e-5 * (fabs(val[k]) + fabs(val[kt])) + 1e-6 * (drr + dcc);
            }
        }
    }
    if (bad) flag[0] = 1;
}

hipError_t check_symmetric(const SolveSystem& s, int* flag_dev, int* nonsym, hipStream_t st) {
    HIPERR(hipMemsetAsync(flag_dev, 0, sizeof(int), st));
    if (s.nfree > 0)
        hipLaunchKernelGGL(sym_kernel, dim3(blocks(s.nfree * SLX_SYM_LPR)), dim3(256), 0, st, s.nfree, s.Arow, s.Acol, s.Aval, flag_dev);
    HIPERR(hipMemcpyAsync(nonsym, flag_dev, sizeof(int), hipMemcpyDeviceToHost, st));
    return hipStreamSynchronize(st);
}

static hipError_t read_scalar(const double* dsc, int idx, double* h, hipStream_t st);

// One cycle of right-preconditioned GMRES on A d = r32 (FP32 vectors, FP64
// sums, classical Gram-Schmidt applied twice), at most min(restart,
// max_inner) iterations or until the FP32 residual estimate falls below
// inner_tol of its start.  d = 0 when r32 = 0.
static hipError_t gmres_cycle(const SolveSystem& s, const SolveParams& prm, SolveWork& w, int& iters, hipStream_t st) {
    const int64_t n = s.nfree;
    const int m = std::max(1, std::min(prm.restart, prm.max_inner));
    // mpart: the dots' partials, then the column store [m][m + 1], cs, sn, g and the history
    // (up to eight partials of a dot are summed by the kernel that needs it)
    const int nchunk = n <= 32768 ? (int)std::min<int64_t>(8, (n + 1023) / 1024) : (int)std::min<int64_t>(SLX_SOLVE_BLOCKS, (n + 4095) / 4096);
    const int64_t chunk = (n + nchunk - 1) / nchunk;
    double* part = w.mpart;
    double* H = part + (size_t)(m + 1) * SLX_SOLVE_BLOCKS;
    double* cs = w.mpart + (size_t)(m + 1) * 2 * SLX_SOLVE_BLOCKS - 5 * (m + 1);
    double *sn = cs + m, *gv = sn + m, *hist = gv + m + 1;
    const unsigned gu = (unsigned)std::min<int64_t>(SLX_SOLVE_BLOCKS, (n + 63) / 64);
    const unsigned gn = (unsigned)std::min<int64_t>(SLX_SOLVE_BLOCKS, (n + 255) / 256);
    const unsigned gd = (unsigned)std::min<int64_t>(SLX_SOLVE_BLOCKS, (n + 255) / 256);
    double beta = 0.0;
    hipLaunchKernelGGL((dot_partial<float>), dim3(gd), dim3(256), 0, st, n, w.r32, w.r32, w.part);
    hipLaunchKernelGGL(basis_next, dim3(gn), dim3(256), 0, st, n, w.part, (int)gd, w.r32, w.dinv, w.V, w.z, -1, H, cs, sn, gv, hist);
    HIPERR(read_scalar(hist, 0, &beta, st));
    if (!(beta > 0.0)) {
        HIPERR(hipMemsetAsync(w.d, 0, n * sizeof(float), st));
        return hipSuccess;
    }
    std::vector<double> hh(2 * (size_t)m);
    int k = 0;
    for (int j = 0; j < m && k == 0; j++) {
        int npart = 0;
        HIPERR(inner_product(n, s.nnzA, s.max_row, s.nblk, s.Ablk, s.Arow, s.Acol, w.val32, w.z, w.q, w.part, &npart, st));
        double* hcol = H + (size_t)j * (m + 1);
        // two passes of classical Gram-Schmidt against v_0 .. v_j
        for (int pass = 0; pass < 2; pass++) {
            hipLaunchKernelGGL(basis_dots, dim3(nchunk, (j + 4) / 4), dim3(256), 0, st, n, chunk, w.V, j + 1, w.q, part);
            const double* src = part;
            int np = nchunk;
            if (nchunk > 8) {
                hipLaunchKernelGGL(sum_rows, dim3(j + 1), dim3(256), 0, st, part, nchunk, w.hv);
                src = w.hv;
                np = 1;
            }
            hipLaunchKernelGGL(basis_update, dim3(gu), dim3(256), 0, st, n, w.V, j + 1, src, np, pass, hcol, w.q, w.part);
        }
        hipLaunchKernelGGL(basis_next, dim3(gn), dim3(256), 0, st, n, w.part, (int)gu, w.q, w.dinv, w.V + (size_t)(j + 1) * n, w.z, j, hcol,
                           cs, sn, gv, hist);
        if ((j + 1) % SLX_GMRES_CHECK == 0 || j + 1 == m) {
            HIPERR(hipMemcpyAsync(hh.data(), hist, 2 * (size_t)(j + 1) * sizeof(double), hipMemcpyDeviceToHost, st));
            HIPERR(hipStreamSynchronize(st));
            for (int i = j + 1 - std::min(j + 1, SLX_GMRES_CHECK); i <= j && k == 0; i++)
                if (hh[2 * i] <= prm.inner_tol * beta || !(hh[2 * i + 1] > 0.0)) k = i + 1;
            if (j + 1 == m && k == 0) k = m;
        }
    }
    iters += k;
    // y = H(0:k, 0:k)^-1 g(0:k)
    std::vector<double> R((size_t)k * (m + 1)), g(k), y(k, 0.0);
    HIPERR(hipMemcpyAsync(R.data(), H, R.size() * sizeof(double), hipMemcpyDeviceToHost, st));
    HIPERR(hipMemcpyAsync(g.data(), gv, (size_t)k * sizeof(double), hipMemcpyDeviceToHost, st));
    HIPERR(hipStreamSynchronize(st));
    for (int i = k - 1; i >= 0; i--) {
        double t = g[i];
        for (int c = i + 1; c < k; c++) t -= R[(size_t)c * (m + 1) + i] * y[c];
        const double d = R[(size_t)i * (m + 1) + i];
        y[i] = d != 0.0 ? t / d : 0.0;
    }
    HIPERR(hipMemcpyAsync(w.hv, y.data(), (size_t)k * sizeof(double), hipMemcpyHostToDevice, st));
    hipLaunchKernelGGL(basis_combine, dim3(blocks(n)), dim3(256), 0, st, n, w.V, k, w.hv, w.dinv, w.d);
    return hipStreamSynchronize(st);
}

static hipError_t read_scalar(const double* dsc, int idx, double* h, hipStream_t st) {
    HIPERR(hipMemcpyAsync(h, dsc + idx, sizeof(double), hipMemcpyDeviceToHost, st));
    return hipStreamSynchronize(st);
}

hipError_t eliminate_system(const SolveSystem& s, const double* b, double* out, double* xd, hipStream_t st) {
    const int64_t n = s.nfree;
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(gather_kernel, dim3(blocks(n)), dim3(256), 0, st, n, s.free_dofs, b, out);
    if (s.ncons > 0) {
        hipLaunchKernelGGL(gather_kernel, dim3(blocks(s.ncons)), dim3(256), 0, st, s.ncons, s.cons_dofs, b, xd);
        spmv<double, double, double>(n, s.nnzD, s.Drow, s.Dcol, s.Dval, xd, out, 1.0, 1.0, out, st);
    }
    return hipGetLastError();
}

hipError_t matvec_system(const SolveSystem& s, const double* x, double* y, double* xa, double* xd, double* ya, hipStream_t st) {
    const int64_t n = s.nfree;
    HIPERR(hipMemcpyAsync(y, x, s.n_dofs * sizeof(double), hipMemcpyDeviceToDevice, st));
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(gather_kernel, dim3(blocks(n)), dim3(256), 0, st, n, s.free_dofs, x, xa);
    spmv<double, double, double>(n, s.nnzA, s.Arow, s.Acol, s.Aval, xa, (const double*)nullptr, 0.0, -1.0, ya, st);
    if (s.ncons > 0) {
        hipLaunchKernelGGL(gather_kernel, dim3(blocks(s.ncons)), dim3(256), 0, st, s.ncons, s.cons_dofs, x, xd);
        spmv<double, double, double>(n, s.nnzD, s.Drow, s.Dcol, s.Dval, xd, ya, 1.0, -1.0, ya, st);
    }
    hipLaunchKernelGGL(scatter_kernel, dim3(blocks(n)), dim3(256), 0, st, n, s.free_dofs, ya, y);
    return hipGetLastError();
}

hipError_t spmv_stream_probe(int64_t nrows, const int64_t* rowp, const int32_t* col, const float* val, int64_t nnz, int max_row,
                             const int64_t* blk, int64_t nblk, const float* x, float* y, double* part, double* sc, hipStream_t st) {
    int npart = 0;
    HIPERR(inner_product(nrows, nnz, max_row, nblk, blk, rowp, col, val, x, y, part, &npart, st));
    hipLaunchKernelGGL(sum_partials, dim3(1), dim3(256), 0, st, part, npart, (int)SC_PQ, sc);
    return hipGetLastError();
}

hipError_t solve_system(const SolveSystem& s, const SolveParams& prm, SolveWork& w, SolveStats& out, hipStream_t st) {
    const int64_t n = s.nfree;
    out = SolveStats{};
    if (n == 0) return hipSuccess;
    // at most SLX_SOLVE_BLOCKS blocks (every block of the next kernel sums their partials)
    const unsigned G = (unsigned)std::min<int64_t>(SLX_SOLVE_BLOCKS, (n + 255) / 256);
    double *prz = w.part + SLX_SOLVE_BLOCKS, *prz_new = prz + SLX_SOLVE_BLOCKS, *prr = prz_new + SLX_SOLVE_BLOCKS;
    // the product's partials: the streaming kernel's may be more than a quarter of
    // w.part takes, and the full solution's place is free until the end
    double* ppq = s.n_dofs > SLX_SOLVE_BLOCKS ? w.xfull : w.part;
    // f = b_A - D x_D ; x_D = Dirichlet values from the rhs
    hipLaunchKernelGGL(gather_kernel, dim3(blocks(n)), dim3(256), 0, st, n, s.free_dofs, s.rhs, w.f);
    if (s.ncons > 0) {
        hipLaunchKernelGGL(gather_kernel, dim3(blocks(s.ncons)), dim3(256), 0, st, s.ncons, s.cons_dofs, s.rhs, w.xd);
        spmv<double, double, double>(n, s.nnzD, s.Drow, s.Dcol, s.Dval, w.xd, w.f, 1.0, 1.0, w.f, st);
    }
    hipLaunchKernelGGL(prep_kernel, dim3(blocks(16 * n)), dim3(256), 0, st, n, s.Arow, s.Acol, s.Aval, w.val32, w.dinv);
    HIPERR(hipMemsetAsync(w.x, 0, n * sizeof(double), st));
    double h = 0.0;
    hipLaunchKernelGGL((dot_partial<double>), dim3(G), dim3(256), 0, st, n, w.f, w.f, w.part);
    hipLaunchKernelGGL(sum_partials, dim3(1), dim3(256), 0, st, w.part, (int)G, (int)SC_DOT, w.sc);
    HIPERR(read_scalar(w.sc, SC_DOT, &h, st));
    const double fnorm = sqrt(h);
    // r = f (x = 0)
    HIPERR(hipMemcpyAsync(w.r, w.f, n * sizeof(double), hipMemcpyDeviceToDevice, st));
    double rnorm = fnorm;
    for (int it = 0; it < prm.max_outer; it++) {
        if (rnorm <= prm.rel_tol * fnorm) break;
        out.outer++;
        if (prm.gmres) {
            hipLaunchKernelGGL(to_f32, dim3(blocks(n)), dim3(256), 0, st, n, w.r, w.r32);
            HIPERR(gmres_cycle(s, prm, w, out.inner, st));
        } else {
        // inner FP32 PCG on A d = r
        hipLaunchKernelGGL(pcg_start, dim3(G), dim3(256), 0, st, n, w.r, w.dinv, w.r32, w.z, w.p, w.d, prz, prr);
        hipLaunchKernelGGL(sum_partials, dim3(1), dim3(256), 0, st, prr, (int)G, (int)SC_RR, w.sc);
        HIPERR(read_scalar(w.sc, SC_RR, &h, st));
        const double r0 = sqrt(h);
        for (int k = 0; k < prm.max_inner; k++) {
            int npq = 0;
            HIPERR(inner_product(n, s.nnzA, s.max_row, s.nblk, s.Ablk, s.Arow, s.Acol, w.val32, w.p, w.q, ppq, &npq, st));
            hipLaunchKernelGGL(pcg_update, dim3(G), dim3(256), 0, st, n, ppq, npq, prz, (int)G, w.d, w.r32, w.p, w.q, w.dinv, w.z, prz_new, prr);
            out.inner++;
            if ((k + 1) % 8 == 0 || k + 1 == prm.max_inner) {
                hipLaunchKernelGGL(sum_partials, dim3(1), dim3(256), 0, st, prr, (int)G, (int)SC_RR, w.sc);
                HIPERR(read_scalar(w.sc, SC_RR, &h, st));
                if (sqrt(h) <= prm.inner_tol * r0) break;
            }
            hipLaunchKernelGGL(pcg_direction, dim3(G), dim3(256), 0, st, n, prz_new, prz, (int)G, w.z, w.p);
            std::swap(prz, prz_new);
        }
        }
        hipLaunchKernelGGL(add_f32_to_f64, dim3(blocks(n)), dim3(256), 0, st, n, w.d, w.x);
        // FP64 residual r = f - A x
        spmv<double, double, double>(n, s.nnzA, s.Arow, s.Acol, s.Aval, w.x, w.f, 1.0, 1.0, w.r, st);
        hipLaunchKernelGGL((dot_partial<double>), dim3(G), dim3(256), 0, st, n, w.r, w.r, w.part);
        hipLaunchKernelGGL(sum_partials, dim3(1), dim3(256), 0, st, w.part, (int)G, (int)SC_DOT, w.sc);
        HIPERR(read_scalar(w.sc, SC_DOT, &h, st));
        rnorm = sqrt(h);
    }
    out.rel_residual = fnorm > 0 ? rnorm / fnorm : 0.0;
    // full solution: free entries from x, constrained entries the Dirichlet values
    HIPERR(hipMemcpyAsync(w.xfull, s.rhs, s.n_dofs * sizeof(double), hipMemcpyDeviceToDevice, st));
    hipLaunchKernelGGL(scatter_kernel, dim3(blocks(n)), dim3(256), 0, st, n, s.free_dofs, w.x, w.xfull);
    return hipGetLastError();
}

}  // namespace slx
