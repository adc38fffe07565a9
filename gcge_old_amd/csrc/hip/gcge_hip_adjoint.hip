// Gradients of eigenvalue and eigenvector losses with respect to the matrix
// entries and to per-element coefficients.
//
// For B-normalised eigenpairs (A - lambda_c B) x_c = 0 of symmetric A, B and a
// loss L(lambda), dL/dA = sum_c gbar_c x_c x_c^T and dL/dB = -sum_c gbar_c
// lambda_c x_c x_c^T; only the entries on the sparsity pattern are formed
// (pattern_gradient, weights gbar or -gbar lambda).  When A = sum_e kappa_e
// A_e (Q1 stiffness on the E^3 mesh, A_e = kappa-free element matrix),
// dL/dkappa_e = sum_c gbar_c x_c|e^T A_e x_c|e (q1_element_gradient).  Both
// take a second block Y for the bilinear form y^T A_e x of eigenvector-loss
// adjoints (Y = X for eigenvalue losses).
//
//   k_pattern_grad   one lane per sliced-ELLPACK entry position, k columns
//                    summed in registers, scattered to the CSR position;
//                    HBM-bound: nnz (4 + 4 + 8) + gathers of X and Y
//   k_q1_elem_grad   a thread marches up a column of elements: node values of
//                    x and y (zero on Dirichlet nodes) read once per plane,
//                    36 Khat diagonal in the sums and differences per axis
#include <hip/hip_runtime.h>

#include "gcge_hip_internal.h"

namespace gcge_hip {

namespace {

constexpr int kBlock = 256;
constexpr int kWave = 64;

__global__ __launch_bounds__(kBlock) void k_pattern_grad(int n, int nslices,
                                                        const int *__restrict__ sptr,
                                                        const int *__restrict__ sw,
                                                        const int *__restrict__ scol,
                                                        const int *__restrict__ spos,
                                                        const double *__restrict__ X, long ldx,
                                                        const double *__restrict__ Y, long ldy,
                                                        int k, const double *__restrict__ w,
                                                        double *__restrict__ grad)
{
    const int slice = blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
    if (slice >= nslices) return;
    const int lane = threadIdx.x % kWave;
    const int row = slice * kWave + lane;
    if (row >= n) return;
    const int off = sptr[slice], width = sw[slice];
    for (int j = 0; j < width; ++j) {
        const long pos = off + (long)j * kWave + lane;
        const int p = spos[pos];
        if (p < 0) continue;
        const int col = scol[pos];
        double s = 0.0;
        for (int c = 0; c < k; ++c) {
            const double *xc = X + (long)c * ldx, *yc = Y + (long)c * ldy;
            s += w[c] * 0.5 * (xc[row] * yc[col] + yc[row] * xc[col]);
        }
        grad[p] = s;
    }
}

// Element gradient, bound by the reads of X (8 n k bytes): a thread owns the
// Z elements ez0 .. ez0 + Z - 1 above one in-plane element (consecutive
// threads along x, then y) and, for every column, reads the Z + 1 node planes
// they touch once: 4 (Z + 1) values, all in flight together, instead of 8 per
// element and operand.  The 8 corner values of an element enter through sums
// s and differences d along each axis, in which the element matrix is
// diagonal: per axis x^T k y = d_x d_y and x^T (6 m) y = 3/2 s_x s_y + 1/2
// d_x d_y, so x^T (36 Khat) y = 9/4 (one difference) + 3/2 (two) + 3/4
// (three), about 30 operations per element and column instead of 144, and
// the in-plane half of the transform is shared by the elements below and
// above a plane.  SPLIT threads of a workgroup share an element column, each
// taking every SPLIT-th column of X (combined through LDS in a fixed order).
// SAME: Y is X (read once).  MAP: node numbers go through node_row, once per
// thread.  Measured (kernel alone, X = Y; before: one thread per element, 16
// loads and 8 x 8 products): 128^3 elements x 100 columns 1799 -> 617 us (2.7
// TB/s of X), 64^3 x 20 52 -> 21, 24^3 x 60 46 -> 15, permuted rows at 128^3
// x 100 17.9 -> 7.0 ms.  Two elements along y per thread (fewer loads each)
// measured the same, Z = 4 16 % slower at 128^3.
template <int Z, int SPLIT, bool SAME, bool MAP>
__global__ __launch_bounds__(kBlock) void k_q1_elem_grad(int E, double scale,
                                                        const double *__restrict__ X, long ldx,
                                                        const double *__restrict__ Y, long ldy,
                                                        int k, const double *__restrict__ w,
                                                        const int *__restrict__ node_row,
                                                        double *__restrict__ grad)
{
    constexpr int EL = kBlock / SPLIT;  // in-plane elements of a workgroup
    const int N = E - 1, EE = E * E, tiles = (EE + EL - 1) / EL;
    const int blk = xcd_remap(blockIdx.x, gridDim.x);
    const int ez0 = blk / tiles * Z;
    const int part = threadIdx.x / EL, ip = blk % tiles * EL + threadIdx.x % EL;
    const int ex = ip % E, ey = ip / E;
    bool ok[4];
    int off[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int ix = ex + (q & 1), iy = ey + (q >> 1);
        ok[q] = ip < EE && ix >= 1 && ix <= N && iy >= 1 && iy <= N;
        off[q] = ok[q] ? (ix - 1) + N * (iy - 1) : 0;
    }
    int row[MAP ? Z + 1 : 1][4];
    if constexpr (MAP) {
#pragma unroll
        for (int p = 0; p <= Z; ++p) {
            const int iz = ez0 + p;
            const bool in = iz >= 1 && iz <= N;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                row[p][q] = in && ok[q] ? node_row[(long)(iz - 1) * N * N + off[q]] : 0;
        }
    }
    // corner values of the Z + 1 planes (planes and nodes outside the mesh
    // read an inside one and count as zero), then the in-plane sums and
    // differences (x fastest: ss, ds, sd, dd)
    auto planes = [&](const double *__restrict__ col, double (&t)[Z + 1][4]) {
#pragma unroll
        for (int p = 0; p <= Z; ++p) {
            const double *base = MAP ? col : col + (long)(min(max(ez0 + p, 1), N) - 1) * N * N;
#pragma unroll
            for (int q = 0; q < 4; ++q) t[p][q] = base[MAP ? row[MAP ? p : 0][q] : off[q]];
        }
#pragma unroll
        for (int p = 0; p <= Z; ++p) {
            const bool in = ez0 + p >= 1 && ez0 + p <= N;
            double v[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] = in && ok[q] ? t[p][q] : 0.0;
            const double s0 = v[0] + v[1], d0 = v[1] - v[0], s1 = v[2] + v[3], d1 = v[3] - v[2];
            t[p][0] = s0 + s1;
            t[p][1] = d0 + d1;
            t[p][2] = s1 - s0;
            t[p][3] = d1 - d0;
        }
    };
    double total[Z];
#pragma unroll
    for (int z = 0; z < Z; ++z) total[z] = 0.0;
    for (int c = part; c < k; c += SPLIT) {
        double tx[Z + 1][4], ty[SAME ? 1 : Z + 1][4];
        planes(X + (long)c * ldx, tx);
        if constexpr (!SAME) planes(Y + (long)c * ldy, ty);
        const double wc = w[c];
#pragma unroll
        for (int z = 0; z < Z; ++z) {
            double m[8];  // products of the z sums (0..3) and differences (4..7)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const double xs = tx[z + 1][q] + tx[z][q], xd = tx[z + 1][q] - tx[z][q];
                double ys = xs, yd = xd;
                if constexpr (!SAME) {
                    ys = ty[z + 1][q] + ty[z][q];
                    yd = ty[z + 1][q] - ty[z][q];
                }
                m[q] = xs * ys;
                m[4 + q] = xd * yd;
            }
            total[z] += wc * (2.25 * (m[1] + m[2] + m[4]) + 1.5 * (m[3] + m[5] + m[6]) + 0.75 * m[7]);
        }
    }
    if constexpr (SPLIT > 1) {
        __shared__ double red[SPLIT - 1][Z][EL];
        if (part > 0) {
#pragma unroll
            for (int z = 0; z < Z; ++z) red[part - 1][z][threadIdx.x % EL] = total[z];
        }
        __syncthreads();
        if (part > 0) return;
#pragma unroll
        for (int z = 0; z < Z; ++z)
#pragma unroll
            for (int q = 0; q < SPLIT - 1; ++q) total[z] += red[q][z][threadIdx.x];
    }
    if (ip < EE) {
#pragma unroll
        for (int z = 0; z < Z; ++z)
            if (ez0 + z < E) grad[(long)(ez0 + z) * EE + ip] = scale * total[z];
    }
}

template <int Z, int SPLIT, bool SAME>
void launch_elem_grad(int E, double scale, const double *X, long ldx, const double *Y, long ldy,
                      int k, const double *d_w, const int *d_node_row, double *d_grad)
{
    constexpr int EL = kBlock / SPLIT;
    const long nb = ((long)E * E + EL - 1) / EL * ((E + Z - 1) / Z);
    if (d_node_row)
        hipLaunchKernelGGL((k_q1_elem_grad<Z, SPLIT, SAME, true>), dim3((unsigned)nb), dim3(kBlock), 0,
                           state().stream, E, scale, X, ldx, Y, ldy, k, d_w, d_node_row, d_grad);
    else
        hipLaunchKernelGGL((k_q1_elem_grad<Z, SPLIT, SAME, false>), dim3((unsigned)nb), dim3(kBlock), 0,
                           state().stream, E, scale, X, ldx, Y, ldy, k, d_w, d_node_row, d_grad);
}

}  // namespace

void pattern_gradient(const Mat *A, const double *X, long ldx, const double *Y, long ldy, int k,
                      const double *d_w, double *d_grad)
{
    if (k <= 0 || A->nrows <= 0) return;
    const int nb = (A->nslices + kBlock / kWave - 1) / (kBlock / kWave);
    ProfScope prof("pattern_grad", (double)A->nnz * 16.0 + 16.0 * k * (double)A->nrows);
    hipLaunchKernelGGL(k_pattern_grad, dim3(nb), dim3(kBlock), 0, state().stream, A->nrows,
                       A->nslices, A->d_slice_ptr, A->d_slice_w, A->d_col, A->d_csrpos, X, ldx, Y,
                       ldy, k, d_w, d_grad);
    HIP_CHECK(hipGetLastError());
}

void q1_element_gradient(int E, const double *X, long ldx, const double *Y, long ldy, int k,
                         const double *d_w, double *d_grad, const int *d_node_row)
{
    if (E < 2 || k <= 0) return;
    const long ne = (long)E * E * E;
    const double h = 1.0 / E;
    const bool same = X == Y && ldx == ldy;  // read once
    ProfScope prof("q1_elem_grad", (same ? 8.0 : 16.0) * k * (double)(E - 1) * (E - 1) * (E - 1) + 8.0 * ne);
    // eight planes per thread (two operands: four, for the registers) where
    // that gives six wavefronts per CU, from about E = 90: 617 against 712 us
    // at 128^3 x 100, 86 against 91 at 97^3 x 33; below, four planes and the
    // columns of X shared by four threads: 21 against 28 us at 64^3 x 20, 15
    // against 68 at 24^3 x 60
    const long waves = ((long)E * E + kWave - 1) / kWave * ((E + 7) / 8);
    const bool many = waves >= 6L * num_cus();
    if (many && same)
        launch_elem_grad<8, 1, true>(E, h / 36.0, X, ldx, Y, ldy, k, d_w, d_node_row, d_grad);
    else if (many)
        launch_elem_grad<4, 1, false>(E, h / 36.0, X, ldx, Y, ldy, k, d_w, d_node_row, d_grad);
    else if (same)
        launch_elem_grad<4, 4, true>(E, h / 36.0, X, ldx, Y, ldy, k, d_w, d_node_row, d_grad);
    else
        launch_elem_grad<4, 4, false>(E, h / 36.0, X, ldx, Y, ldy, k, d_w, d_node_row, d_grad);
    HIP_CHECK(hipGetLastError());
}

}  // namespace gcge_hip
