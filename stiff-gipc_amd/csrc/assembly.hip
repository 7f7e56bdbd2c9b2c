// Hessian assembly for gfx950: element kernels that write 3x3 triplets and
// the triplet -> unique upper BCOO conversion.
//
//  * stable Neo-Hookean tet (StiffGIPC/femEnergy.cu:1719-1857, PK1 :432-459,
//    projection :1641-1717): the PSD projection uses the analytic eigensystem
//    of dP/dF (three twist, three flip and three scaling modes built from a
//    rotation-variant 3x3 SVD), accumulated directly in the 12x12 vertex
//    space as sum_i max(l_i,0) g_i g_i^T with g_i = dF/dx^T vec(Q_i), so no
//    9x9 or 12x12 dense product is ever formed;
//  * point-triangle barrier, GIPC rank-2 variant (StiffGIPC/GIPC.cu:4733-4984):
//    rank-1 Hessian lambda0(I5) g g^T with g the gradient of dist/sqrt(dHat);
//    the lower blocks are moved to (col,row) and zeroed as the reference's
//    contact partition does (StiffGIPC/GIPC.cu:10329-10363);
//  * mass diagonal (StiffGIPC/GIPC.cu:10466-10485);
//  * conversion (Converter::srbk_convert, StiffGIPC/linear_system/utils/
//    converter.cu:32-238): a stable rocPRIM radix sort over only the bits the
//    (row, col) key needs, then every unique block is summed by one thread in
//    sorted (= arena) order, a block of more than 64 triplets as the ordered
//    sum of its 64-triplet chunk sums (each chunk by its own thread), which
//    makes the result deterministic.
#include <algorithm>
#include <cstring>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include "assembly.hpp"
#include "pcg.hpp"
#include "vertex_sums.hpp"
#include "wave_ops.hpp"

namespace sgipc {

namespace {

// ------------------------------------------------------------------ 3x3 helpers
__device__ __forceinline__ void jacobi3(double A[3][3], double V[3][3])
{
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) V[i][j] = (i == j) ? 1.0 : 0.0;
    for (int sweep = 0; sweep < 10; ++sweep) {
        const double off = A[0][1] * A[0][1] + A[0][2] * A[0][2] + A[1][2] * A[1][2];
        const double dia = A[0][0] * A[0][0] + A[1][1] * A[1][1] + A[2][2] * A[2][2];
        if (off <= 1e-34 * dia || off == 0.0) break;
#pragma unroll
        for (int pq = 0; pq < 3; ++pq) {
            const int p = pq == 2 ? 1 : 0;
            const int q = pq == 0 ? 1 : 2;
            const double apq = A[p][q];
            if (apq == 0.0) continue;
            const double theta = (A[q][q] - A[p][p]) / (2.0 * apq);
            const double t = (theta >= 0 ? 1.0 : -1.0) / (fabs(theta) + sqrt(theta * theta + 1.0));
            const double c = 1.0 / sqrt(t * t + 1.0), s = t * c;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const double akp = A[k][p], akq = A[k][q];
                A[k][p] = c * akp - s * akq;
                A[k][q] = s * akp + c * akq;
            }
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const double apk = A[p][k], aqk = A[q][k];
                A[p][k] = c * apk - s * aqk;
                A[q][k] = s * apk + c * aqk;
            }
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const double vkp = V[k][p], vkq = V[k][q];
                V[k][p] = c * vkp - s * vkq;
                V[k][q] = s * vkp + c * vkq;
            }
        }
    }
}

__device__ __forceinline__ double det3(const double F[3][3])
{
    return F[0][0] * (F[1][1] * F[2][2] - F[1][2] * F[2][1]) - F[0][1] * (F[1][0] * F[2][2] - F[1][2] * F[2][0]) +
           F[0][2] * (F[1][0] * F[2][1] - F[1][1] * F[2][0]);
}

__device__ __forceinline__ void cross3(const double a[3], const double b[3], double c[3])
{
    c[0] = a[1] * b[2] - a[2] * b[1];
    c[1] = a[2] * b[0] - a[0] * b[2];
    c[2] = a[0] * b[1] - a[1] * b[0];
}

// Rotation-variant SVD F = U diag(S) V^T with det U = det V = +1 (S[2] may be
// negative), from the eigen-decomposition of F^T F.  Columns of U/V are u_i/v_i.
__device__ void svd3_rv(const double F[3][3], double U[3][3], double S[3], double V[3][3])
{
    double B[3][3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) B[i][j] = F[0][i] * F[0][j] + F[1][i] * F[1][j] + F[2][i] * F[2][j];
    jacobi3(B, V);
    double ev[3] = {B[0][0], B[1][1], B[2][2]};
    // sort eigenvalues descending (swap V columns alongside)
#pragma unroll
    for (int pass = 0; pass < 2; ++pass)
#pragma unroll
        for (int i = 0; i < 2; ++i)
            if (ev[i] < ev[i + 1]) {
                double t = ev[i]; ev[i] = ev[i + 1]; ev[i + 1] = t;
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    double w = V[k][i]; V[k][i] = V[k][i + 1]; V[k][i + 1] = w;
                }
            }
    if (det3(V) < 0.0) {
#pragma unroll
        for (int k = 0; k < 3; ++k) V[k][2] = -V[k][2];
    }
    double fv[3][3];  // F v_i as columns
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int r = 0; r < 3; ++r) fv[r][i] = F[r][0] * V[0][i] + F[r][1] * V[1][i] + F[r][2] * V[2][i];
    double u0[3] = {fv[0][0], fv[1][0], fv[2][0]};
    double n0 = sqrt(u0[0] * u0[0] + u0[1] * u0[1] + u0[2] * u0[2]);
    if (n0 > 1e-300) {
#pragma unroll
        for (int k = 0; k < 3; ++k) u0[k] /= n0;
    } else {
        u0[0] = 1.0; u0[1] = 0.0; u0[2] = 0.0;
    }
    double u1[3] = {fv[0][1], fv[1][1], fv[2][1]};
    const double pr = u1[0] * u0[0] + u1[1] * u0[1] + u1[2] * u0[2];
#pragma unroll
    for (int k = 0; k < 3; ++k) u1[k] -= pr * u0[k];
    double n1 = sqrt(u1[0] * u1[0] + u1[1] * u1[1] + u1[2] * u1[2]);
    if (n1 > 1e-14 * (n0 > 0 ? n0 : 1.0)) {
#pragma unroll
        for (int k = 0; k < 3; ++k) u1[k] /= n1;
    } else {
        // any unit vector orthogonal to u0
        double e[3] = {fabs(u0[0]) < 0.9 ? 1.0 : 0.0, fabs(u0[0]) < 0.9 ? 0.0 : 1.0, 0.0};
        cross3(u0, e, u1);
        double nn = sqrt(u1[0] * u1[0] + u1[1] * u1[1] + u1[2] * u1[2]);
#pragma unroll
        for (int k = 0; k < 3; ++k) u1[k] /= nn;
    }
    double u2[3];
    cross3(u0, u1, u2);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        U[k][0] = u0[k];
        U[k][1] = u1[k];
        U[k][2] = u2[k];
    }
    S[0] = u0[0] * fv[0][0] + u0[1] * fv[1][0] + u0[2] * fv[2][0];
    S[1] = u1[0] * fv[0][1] + u1[1] * fv[1][1] + u1[2] * fv[2][1];
    S[2] = u2[0] * fv[0][2] + u2[1] * fv[1][2] + u2[2] * fv[2][2];
}

__device__ __forceinline__ int up12(int r, int c) { return r * 12 - r * (r - 1) / 2 + (c - r); }

// acc += lam * g g^T (upper triangle of 12x12)
__device__ __forceinline__ void rank1_upper(double acc[78], const double g[12], double lam)
{
#pragma unroll
    for (int r = 0; r < 12; ++r) {
        const double lr = lam * g[r];
#pragma unroll
        for (int c = r; c < 12; ++c) acc[up12(r, c)] += lr * g[c];
    }
}

// ------------------------------------------------------------------ tet kernel
// One thread per tet; the 12x12 Hessian is summed from the clamped rank-one
// modes in registers.  Bound by its scattered writes: the 10 blocks of a tet
// are 720 consecutive bytes, and a thread writing them for itself touches 64
// lines with every instruction, so a wave passes two blocks of its 64 tets at
// a time through LDS and stores 144-byte runs; and an atomic to memory per
// gradient component costs more than all stores, so a thread parks its twelve
// in LDS and the workgroup sums them by vertex (VertexSums) after the blocks.
// 1.5 M tets with gradient, 1.37 GB: 0.90 -> 0.64 ms; the staged stores
// alone change nothing (0.90).  The modes keep the order of their sums:
// forming the blocks in the singular bases (U M_ab U^T) took 0.41 ms but
// raised the error against 64 bits from 1.2e-15 to 1.4e-15.
// kFew: below kTetFew tets the chip is not full and a thread's own stores and
// atomics are over before the workgroup has met (with the launch: 750 and 13k
// tets 42 and 45 us against 46 and 48; 41k 63 against 52).
constexpr int kTetThreads = 128, kTetFew = 20000;
template <bool kFew>
__global__ __launch_bounds__(kTetThreads) void k_tet_snh(int n_tets, const double* __restrict__ x,
                                                 const uint4* __restrict__ tets, const double* __restrict__ dm_inv,
                                                 const double* __restrict__ vol, const double* __restrict__ mu_,
                                                 const double* __restrict__ lam_, double dt2, int hess_offset,
                                                 double* __restrict__ grad, double* __restrict__ tvals,
                                                 int* __restrict__ trows, int* __restrict__ tcols)
{
    __shared__ double stage[kFew ? 1 : kTetThreads / 64][kFew ? 1 : 64 * 18];
    __shared__ double forces[kFew ? 1 : kTetThreads][13];
    __shared__ VertexSums<kFew ? 2 : 256> sums;
    if constexpr (!kFew)
        if (grad) sums.init();
    const int t0 = blockIdx.x * blockDim.x + threadIdx.x;
    const bool act = t0 < n_tets;
    const int t = act ? t0 : n_tets - 1;  // spare lanes repeat the last tet and write nothing
    const uint4 tv = tets[t];
    const unsigned vid[4] = {tv.x, tv.y, tv.z, tv.w};
    double xs[4][3];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int d = 0; d < 3; ++d) xs[a][d] = x[3 * (long)vid[a] + d];
    double Dmi[3][3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) Dmi[i][j] = dm_inv[9 * (long)t + 3 * i + j];
    // F = Ds Dm^-1, Ds columns x1-x0, x2-x0, x3-x0
    double F[3][3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            double s = 0.0;
#pragma unroll
            for (int k = 0; k < 3; ++k) s += (xs[k + 1][i] - xs[0][i]) * Dmi[k][j];
            F[i][j] = s;
        }
    // d_a: dF(:,j)/dx_a coefficients
    double D[4][3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        D[0][j] = -(Dmi[0][j] + Dmi[1][j] + Dmi[2][j]);
#pragma unroll
        for (int a = 1; a < 4; ++a) D[a][j] = Dmi[a - 1][j];
    }
    const double mu = mu_[t], lam = lam_[t];
    const double J = det3(F);
    const double c = lam * (J - 1.0) - mu;
    const double scale = dt2 * vol[t];

    if (grad) {
        double cof[3][3];
        cof[0][0] = F[1][1] * F[2][2] - F[1][2] * F[2][1];
        cof[0][1] = F[1][2] * F[2][0] - F[1][0] * F[2][2];
        cof[0][2] = F[1][0] * F[2][1] - F[1][1] * F[2][0];
        cof[1][0] = F[2][1] * F[0][2] - F[2][2] * F[0][1];
        cof[1][1] = F[2][2] * F[0][0] - F[2][0] * F[0][2];
        cof[1][2] = F[2][0] * F[0][1] - F[2][1] * F[0][0];
        cof[2][0] = F[0][1] * F[1][2] - F[1][1] * F[0][2];
        cof[2][1] = F[0][2] * F[1][0] - F[0][0] * F[1][2];
        cof[2][2] = F[0][0] * F[1][1] - F[0][1] * F[1][0];
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                double s = 0.0;
#pragma unroll
                for (int j = 0; j < 3; ++j) s += (mu * F[d][j] + c * cof[d][j]) * D[a][j];
                if constexpr (kFew) {
                    if (act) atomic_add(grad + 3 * (long)vid[a] + d, scale * s);
                } else {
                    if (act) forces[threadIdx.x][3 * a + d] = scale * s;
                }
            }
    }

    double U[3][3], S[3], V[3][3];
    svd3_rv(F, U, S, V);
    // w[a][i] = v_i . d_a
    double w[4][3];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int i = 0; i < 3; ++i) w[a][i] = V[0][i] * D[a][0] + V[1][i] * D[a][1] + V[2][i] * D[a][2];

    double acc[78];
#pragma unroll
    for (int e = 0; e < 78; ++e) acc[e] = 0.0;
    const double rs2 = 0.70710678118654752440;
    // twist (Q = (u_j v_i^T - u_i v_j^T)/sqrt2) and flip (Q = (u_i v_j^T + u_j v_i^T)/sqrt2)
    // modes for axis k with (i, j) the other two axes; eigenvalues mu +/- c S[k]
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int i = k == 0 ? 1 : 0;
        const int j = k == 2 ? 1 : 2;
#pragma unroll
        for (int flip = 0; flip < 2; ++flip) {
            const double l = flip ? (mu - c * S[k]) : (mu + c * S[k]);
            if (l <= 0.0) continue;
            double g[12];
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int d = 0; d < 3; ++d)
                    g[3 * a + d] = flip ? rs2 * (U[d][i] * w[a][j] + U[d][j] * w[a][i])
                                        : rs2 * (U[d][j] * w[a][i] - U[d][i] * w[a][j]);
            rank1_upper(acc, g, l);
        }
    }
    // scaling modes: eigen-decomposition of the 3x3 block in singular space
    {
        const double ev = lam * (2.0 * J - 1.0) - mu;
        double A[3][3];
        A[0][0] = mu + lam * S[1] * S[1] * S[2] * S[2];
        A[1][1] = mu + lam * S[0] * S[0] * S[2] * S[2];
        A[2][2] = mu + lam * S[0] * S[0] * S[1] * S[1];
        A[0][1] = A[1][0] = ev * S[2];
        A[0][2] = A[2][0] = ev * S[1];
        A[1][2] = A[2][1] = ev * S[0];
        double E[3][3];
        jacobi3(A, E);
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            const double l = A[m][m];
            if (l <= 0.0) continue;
            double g[12];
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int d = 0; d < 3; ++d)
                    g[3 * a + d] = E[0][m] * U[d][0] * w[a][0] + E[1][m] * U[d][1] * w[a][1] + E[2][m] * U[d][2] * w[a][2];
            rank1_upper(acc, g, l);
        }
    }
    // 10 upper blocks, local (ii <= jj), stored at (min, max) of the global
    // ids: transposed when the ids are in the other order
    constexpr int kI[10] = {0, 0, 0, 0, 1, 1, 1, 2, 2, 3}, kJ[10] = {0, 1, 2, 3, 1, 2, 3, 2, 3, 3};
    if constexpr (kFew) {
        if (!act) return;
#pragma unroll
        for (int k = 0; k < 10; ++k) {
            const long at = 10 * (long)t + k;
            const int ii = kI[k], jj = kJ[k];
            const int a = (int)vid[ii] + hess_offset, b = (int)vid[jj] + hess_offset;
            const bool keep = a <= b;
            trows[at] = min(a, b);
            tcols[at] = max(a, b);
#pragma unroll
            for (int r = 0; r < 3; ++r)
#pragma unroll
                for (int cc = 0; cc < 3; ++cc) {
                    const int R = 3 * ii + r, C = 3 * jj + cc, R2 = 3 * jj + r, C2 = 3 * ii + cc;
                    const double hv = acc[R <= C ? up12(R, C) : up12(C, R)];
                    const double ht = acc[R2 <= C2 ? up12(R2, C2) : up12(C2, R2)];
                    tvals[9 * at + cc * 3 + r] = scale * (keep ? hv : ht);
                }
        }
        return;
    }
    const int lane = threadIdx.x & 63;
    double* const st = stage[threadIdx.x >> 6];
    const long w0 = (long)blockIdx.x * blockDim.x + (threadIdx.x & ~63);  // the wave's first tet
    const int nw = n_tets > w0 ? (int)(n_tets - w0 < 64 ? n_tets - w0 : 64) : 0;  // its tets
    // where value lane + 64 i of a staged pair of blocks goes (576 values are 32 tets)
    unsigned ofs[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) {
        const unsigned e = lane + 64 * i;
        ofs[i] = 90u * (e / 18u) + e % 18u;
    }
#pragma unroll
    for (int k0 = 0; k0 < 10; k0 += 2) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int ii = kI[k0 + k], jj = kJ[k0 + k];
            const bool keep = vid[ii] <= vid[jj];
            double* const q = st + 18 * lane + 9 * k;
#pragma unroll
            for (int r = 0; r < 3; ++r)
#pragma unroll
                for (int cc = 0; cc < 3; ++cc) {
                    const int R = 3 * ii + r, C = 3 * jj + cc;
                    q[keep ? cc * 3 + r : r * 3 + cc] = scale * acc[R <= C ? up12(R, C) : up12(C, R)];
                }
        }
        wave_lds_sync();
        double* const dst = tvals + 90 * w0 + 9 * k0;
#pragma unroll
        for (int i = 0; i < 18; ++i)
            if (lane + 64 * i < 18 * nw) dst[ofs[i % 9] + (i / 9) * 32u * 90u] = st[lane + 64 * i];
        wave_lds_sync();
    }
    int* const si = reinterpret_cast<int*>(st);
#pragma unroll
    for (int side = 0; side < 2; ++side) {
#pragma unroll
        for (int k = 0; k < 10; ++k) {
            const int a = (int)vid[kI[k]] + hess_offset, b = (int)vid[kJ[k]] + hess_offset;
            si[10 * lane + k] = side == 0 ? min(a, b) : max(a, b);
        }
        wave_lds_sync();
        int* const dst = (side == 0 ? trows : tcols) + 10 * w0;
        for (int e = lane; e < 10 * nw; e += 64) dst[e] = si[e];
        wave_lds_sync();
    }
    if (grad) {
        if (act)
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const double* const f = forces[threadIdx.x] + 3 * a;
                sums.add((int)vid[a], f[0], f[1], f[2], grad);
            }
        sums.flush(grad);
    }
}

// ------------------------------------------------------------------ barrier kernel
__device__ __forceinline__ double barrier_lambda0(double I5, double dh, double kappa)
{
    const double L = log(I5);
    return -(4.0 * kappa * dh * dh *
             (4.0 * I5 + L - 3.0 * I5 * I5 * L * L + 6.0 * I5 * L - 2.0 * I5 * I5 + I5 * L * L - 7.0 * I5 * I5 * L - 2.0)) /
           I5;
}

__global__ __launch_bounds__(128) void k_barrier_pt(int n_pairs, const double* __restrict__ x,
                                                    const int4* __restrict__ pairs, const double* __restrict__ pair_x,
                                                    double dh, double kappa, int hess_offset,
                                                    double* __restrict__ grad, double* __restrict__ tvals,
                                                    int* __restrict__ trows, int* __restrict__ tcols)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n_pairs) return;
    const int4 pr = pairs[p];
    const int vid[4] = {-pr.x - 1, pr.y, pr.z, pr.w};
    double P[4][3];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int d = 0; d < 3; ++d)
            P[a][d] = pair_x ? pair_x[12 * (long)p + 3 * a + d] : x[3 * (long)vid[a] + d];
    double e1[3], e2[3], w[3], b[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        e1[d] = P[2][d] - P[1][d];
        e2[d] = P[3][d] - P[1][d];
        w[d] = P[0][d] - P[1][d];
    }
    cross3(e1, e2, b);
    const double bb = b[0] * b[0] + b[1] * b[1] + b[2] * b[2];
    const double aTb = w[0] * b[0] + w[1] * b[1] + w[2] * b[2];
    const double d2 = aTb * aTb / bb;
    const double dis = sqrt(d2);
    const double sq = sqrt(dh);
    const double I5 = d2 / dh;
    const double nb = sqrt(bb), sgn = aTb >= 0 ? 1.0 : -1.0;
    double c1[3], c2[3];
    cross3(w, e2, c1);
    cross3(e1, w, c2);
    const double be1 = (c1[0] * b[0] + c1[1] * b[1] + c1[2] * b[2]) / bb;
    const double be2 = (c2[0] * b[0] + c2[1] * b[1] + c2[2] * b[2]) / bb;
    const double be0 = 1.0 - be1 - be2;
    const double coef[4] = {1.0, -be0, -be1, -be2};
    double g[12];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int d = 0; d < 3; ++d) g[3 * a + d] = sgn * coef[a] * b[d] / (nb * sq);
    const double gass = 1e-6;
    const double lam0 = barrier_lambda0(d2 < gass * dh ? gass : I5, dh, kappa);
    if (grad) {
        const double L = log(I5);
        const double pk = 2.0 * (2.0 * kappa * dh * dh * L * (I5 - 1.0) * (I5 + I5 * L - 1.0)) / I5;
        const double s = dis / sq;
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int d = 0; d < 3; ++d) atomic_add(grad + 3 * (long)vid[a] + d, g[3 * a + d] * s * pk);
    }
    const long base = 16 * (long)p;
#pragma unroll
    for (int ii = 0; ii < 4; ++ii)
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
            const int kk = ii * 4 + jj;
            const int row = vid[ii] + hess_offset, col = vid[jj] + hess_offset;
            double* dst = tvals + 9 * (base + kk);
            if (row <= col) {
                trows[base + kk] = row;
                tcols[base + kk] = col;
#pragma unroll
                for (int r = 0; r < 3; ++r)
#pragma unroll
                    for (int cc = 0; cc < 3; ++cc) dst[cc * 3 + r] = lam0 * g[3 * ii + r] * g[3 * jj + cc];
            } else {
                trows[base + kk] = col;
                tcols[base + kk] = row;
#pragma unroll
                for (int e = 0; e < 9; ++e) dst[e] = 0.0;
            }
        }
}

__global__ void k_mass_diag(int n, const double* __restrict__ mass, int hess_offset, double* __restrict__ tvals,
                            int* __restrict__ trows, int* __restrict__ tcols)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double m = mass[i];
    double* dst = tvals + 9 * (long)i;
#pragma unroll
    for (int e = 0; e < 9; ++e) dst[e] = (e == 0 || e == 4 || e == 8) ? m : 0.0;
    trows[i] = i + hess_offset;
    tcols[i] = i + hess_offset;
}

// ------------------------------------------------------------------ conversion
__global__ void k_make_keys(const int* __restrict__ rows, const int* __restrict__ cols, long n, int kbits,
                            uint64_t* __restrict__ keys, int* __restrict__ idx, int* __restrict__ bad)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int r = rows[i], c = cols[i];
    if (r < 0 || c < 0 || r > c || (kbits < 31 && (r >> kbits) != 0) || (kbits < 31 && (c >> kbits) != 0)) atomicOr(bad, 1);
    keys[i] = ((uint64_t)(uint32_t)r << kbits) | (uint64_t)(uint32_t)c;
    idx[i] = (int)i;
}

__global__ void k_head_flags(const uint64_t* __restrict__ sk, long n, int* __restrict__ flag)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    flag[i] = (i == 0 || sk[i] != sk[i - 1]) ? 1 : 0;
}

__global__ void k_heads(const uint64_t* __restrict__ sk, const int* __restrict__ flag, const int* __restrict__ pos,
                        long n, int kbits, int* __restrict__ head_pos, int* __restrict__ orows,
                        int* __restrict__ ocols, int capacity)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (i == n - 1 && pos[i] <= capacity) head_pos[pos[i]] = (int)n;  // sentinel
    if (!flag[i]) return;
    const int u = pos[i] - 1;
    if (u > capacity) return;
    // u == capacity: the first block past the capacity, whose start ends the
    // last block kept (head_pos holds capacity + 1 entries)
    head_pos[u] = (int)i;
    if (u == capacity) return;
    const uint64_t k = sk[i];
    orows[u] = (int)(k >> kbits);
    ocols[u] = (int)(k & ((1ull << kbits) - 1ull));
}

// Unique blocks of more than kSegChunk triplets (on coarse MAS levels and
// affine-body rows thousands of triplets merge into one block) are summed in
// chunks of kSegChunk consecutive sorted triplets, each by its own thread,
// and then the chunk sums in order; shorter blocks by one thread in sorted
// order.  Fixed order either way (deterministic).
constexpr int kSegChunk = 64;

// chunks of every unique block u < cap (0: summed directly)
__global__ void k_seg_chunks(const int* __restrict__ head_pos, const int* __restrict__ pos, long n, int cap,
                             int* __restrict__ cnt)
{
    const int u = blockIdx.x * blockDim.x + threadIdx.x;
    if (u >= cap) return;
    const int m = pos[n - 1] < cap ? pos[n - 1] : cap;
    int c = 0;
    if (u < m) {
        const int len = head_pos[u + 1] - head_pos[u];
        if (len > kSegChunk) c = (len + kSegChunk - 1) / kSegChunk;
    }
    cnt[u] = c;
}

// chunk t of the long blocks (cofs: exclusive prefix of cnt over cap blocks)
__global__ __launch_bounds__(256) void k_chunk_sum(const double* __restrict__ tvals, const int* __restrict__ sidx,
                                                   const int* __restrict__ head_pos, const int* __restrict__ cnt,
                                                   const int* __restrict__ cofs, int cap, long bound,
                                                   double* __restrict__ part)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= bound) return;
    const long total = (long)cofs[cap - 1] + cnt[cap - 1];
    if (t >= total) return;
    // the block holding chunk t: the last u with cofs[u] <= t
    int lo = 0, hi = cap;  // first index with cofs > t lies in (lo, hi]
    while (lo + 1 < hi) {
        const int mid = (lo + hi) >> 1;
        if ((long)cofs[mid] <= t) lo = mid;
        else hi = mid;
    }
    const int u = lo;
    const int b = head_pos[u] + (int)(t - cofs[u]) * kSegChunk;
    const int e = min(b + kSegChunk, head_pos[u + 1]);
    double s[9];
#pragma unroll
    for (int q = 0; q < 9; ++q) s[q] = 0.0;
    for (int p = b; p < e; ++p) {
        const double* v = tvals + 9 * (long)sidx[p];
#pragma unroll
        for (int q = 0; q < 9; ++q) s[q] += v[q];
    }
    double* o = part + 9 * t;
#pragma unroll
    for (int q = 0; q < 9; ++q) o[q] = s[q];
}

// One thread per unique block: its triplets in sorted (= arena) order, or
// its chunk sums in order.
__global__ __launch_bounds__(256) void k_segment_sum(const double* __restrict__ tvals, const int* __restrict__ sidx,
                                                     const int* __restrict__ head_pos, const int* __restrict__ pos,
                                                     long n, double* __restrict__ ovals, int capacity,
                                                     const int* __restrict__ cnt, const int* __restrict__ cofs,
                                                     const double* __restrict__ part)
{
    const int u = blockIdx.x * blockDim.x + threadIdx.x;
    const int nnz = pos[n - 1];
    if (u >= nnz || u >= capacity) return;
    double s[9];
#pragma unroll
    for (int q = 0; q < 9; ++q) s[q] = 0.0;
    if (cnt[u] > 0) {
        const long c0 = cofs[u], c1 = c0 + cnt[u];
        for (long c = c0; c < c1; ++c) {
            const double* v = part + 9 * c;
#pragma unroll
            for (int q = 0; q < 9; ++q) s[q] += v[q];
        }
    } else {
        const int b = head_pos[u], e = head_pos[u + 1];
        for (int p = b; p < e; ++p) {
            const double* v = tvals + 9 * (long)sidx[p];
#pragma unroll
            for (int q = 0; q < 9; ++q) s[q] += v[q];
        }
    }
    double* o = ovals + 9 * (long)u;
#pragma unroll
    for (int q = 0; q < 9; ++q) o[q] = s[q];
}

// ------------------------------------------------------------------ conversion by rows
// The general conversion above sorts 64-bit (row, column) keys over all their
// bits, five passes over 16 M triplets at C1.  Triplets of one row are few (61
// on average), so here they are put into row order by counting -- a
// workgroup counts its rows in an LDS table, so memory sees one atomic per
// distinct row and not one per triplet -- and each row is sorted by (column,
// triplet) on its own: by one wave in registers up to 256 triplets, by one
// workgroup in LDS up to 2048.  The triplets of longer rows (hubs, the zero
// blocks of boundary hinges) are sorted together by a radix sort of their own,
// whose keys hold a row's rank; where they are more than half of all, the
// general conversion runs instead.  The sums then read their triplets in
// exactly the general order, 9 lanes per block (72-byte runs).  16 M triplets
// (1.47 GB in and out): counting 81 + 103 us, row sorts 147, sums 440 (1.67 GB
// with the keys at 3.8 TB/s; a large copy reaches 4.75 on this part), 0.87 ms
// with the index check and the read-back against 1.73 ms for the general
// conversion.  With long rows: 48 M
// triplets of a 1024^2 cloth (one row of 65 k) 2.9 ms against 4.7; 1.9 M of
// two 72^2 sheets (one row of 9 k) 0.42 against 0.42.
constexpr int kRowTable = 1024;  // slots of the LDS row table
constexpr int kRowItems = 8;     // triplets per thread
constexpr int kRowShort = 256, kRowMid = 2048;
// words behind the row counts: bad index, rows past kRowShort, rows past
// kRowMid and their triplets, unique blocks
enum { kBad = 0, kNMid, kNLong, kLongSum, kUnique, kRowWords = 8 };

// Counts of the rows (scatter = false), or the triplets' keys (column, then
// index) to their row's segment (true; start: exclusive scan of the counts,
// which are used up).  The order inside a segment is left to the row sort.
template <bool scatter>
__global__ __launch_bounds__(256) void k_rows_bin(const int* __restrict__ rows, const int* __restrict__ cols, long n,
                                                  int n_rows, int* __restrict__ cnt, int* __restrict__ words,
                                                  const int* __restrict__ start, uint64_t* __restrict__ key)
{
    __shared__ int srow[kRowTable], scnt[kRowTable], sbase[kRowTable];
    for (int i = threadIdx.x; i < kRowTable; i += 256) {
        srow[i] = -1;
        scnt[i] = 0;
    }
    __syncthreads();
    const long b0 = (long)blockIdx.x * (256 * kRowItems) + threadIdx.x;
    int row[kRowItems], col[kRowItems], slot[kRowItems], at[kRowItems];
    bool bad = false;
#pragma unroll
    for (int i = 0; i < kRowItems; ++i) {
        const long k = b0 + 256 * i;
        row[i] = k < n ? rows[k] : -1;
        col[i] = k < n ? cols[k] : -1;
    }
#pragma unroll
    for (int i = 0; i < kRowItems; ++i) {
        slot[i] = -1;
        if (b0 + 256 * i >= n) continue;
        if (row[i] < 0 || row[i] > col[i] || col[i] >= n_rows) {
            bad = true;
            row[i] = -1;
            continue;
        }
        unsigned h = ((unsigned)row[i] * 2654435761u) >> 22;  // kRowTable slots
        for (int t = 0; t < 6; ++t, h = (h + 1) & (kRowTable - 1)) {
            const int r = atomicCAS(&srow[h], -1, row[i]);
            if (r == -1 || r == row[i]) {
                slot[i] = (int)h;
                at[i] = atomicAdd(&scnt[h], 1);
                break;
            }
        }
    }
    if (!scatter && bad) atomicOr(words + kBad, 1);
    __syncthreads();
    for (int i = threadIdx.x; i < kRowTable; i += 256)
        if (scnt[i] > 0) {
            if (scatter) sbase[i] = start[srow[i]] + atomicSub(cnt + srow[i], scnt[i]) - scnt[i];
            else atomicAdd(cnt + srow[i], scnt[i]);
        }
    if (scatter) __syncthreads();
#pragma unroll
    for (int i = 0; i < kRowItems; ++i) {
        if (row[i] < 0) continue;
        if (scatter) {
            const int p = slot[i] >= 0 ? sbase[slot[i]] + at[i] : start[row[i]] + atomicSub(cnt + row[i], 1) - 1;
            key[p] = ((uint64_t)(uint32_t)col[i] << 32) | (uint32_t)(b0 + 256 * i);
        } else if (slot[i] < 0) {
            atomicAdd(cnt + row[i], 1);
        }
    }
}

// One wave per row: its keys sorted in place and its unique columns counted;
// longer rows are listed.  Bitonic over 64 M elements, element i in lane
// i % 64, register i / 64; the kernel is bound by its instructions (about 100
// per row at M = 1; ranking every key against all others took 250, C1: 226
// us against 147).
template <int M>
__device__ __forceinline__ int sort_row(uint64_t* __restrict__ seg, int k)
{
    const int lane = threadIdx.x & 63;
    uint64_t v[M];
#pragma unroll
    for (int m = 0; m < M; ++m) v[m] = lane + 64 * m < k ? seg[lane + 64 * m] : ~0ull;
#pragma unroll
    for (int size = 2; size <= 64 * M; size <<= 1)
#pragma unroll
        for (int d = size >> 1; d > 0; d >>= 1) {
            if (d >= 64) {
#pragma unroll
                for (int m = 0; m < M; ++m) {
                    const int q = m ^ (d / 64);
                    if (q < m) continue;
                    const bool up = ((64 * m) & size) == 0;
                    const uint64_t x = v[m], y = v[q];
                    const bool swap = (x > y) == up;
                    v[m] = swap ? y : x;
                    v[q] = swap ? x : y;
                }
            } else {
#pragma unroll
                for (int m = 0; m < M; ++m) {
                    const uint64_t x = v[m], y = __shfl_xor(x, d, 64);
                    const bool up = ((64 * m + lane) & size) == 0, low = (lane & d) == 0;
                    v[m] = (x < y) == (low == up) ? x : y;  // equal keys are all padding
                }
            }
        }
    int u = 0;
    uint32_t before = 0;  // last column of the registers so far
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const uint32_t col = (uint32_t)(v[m] >> 32);
        uint32_t prev = __shfl_up(col, 1, 64);
        if (lane == 0) prev = before;
        before = __shfl(col, 63, 64);
        const bool in = lane + 64 * m < k;
        if (in) seg[lane + 64 * m] = v[m];
        u += __popcll(__ballot(in && ((m == 0 && lane == 0) || col != prev)));
    }
    return u;
}
__global__ __launch_bounds__(256) void k_rows_sort(int n_rows, const int* __restrict__ start, uint64_t* __restrict__ key,
                                                   int* __restrict__ ucnt, int* __restrict__ words,
                                                   int* __restrict__ list, int* __restrict__ base)
{
    const int r = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (r > n_rows) return;
    if (r == n_rows) {
        if (lane == 0) ucnt[r] = 0;  // the scan's last element is the total
        return;
    }
    const int b = start[r], k = start[r + 1] - b;
    int u = 0;
    if (k == 0) {
    } else if (k <= 64) {
        u = sort_row<1>(key + b, k);
    } else if (k <= 128) {
        u = sort_row<2>(key + b, k);
    } else if (k <= kRowShort) {
        u = sort_row<4>(key + b, k);
    } else {
        // listed from the front (up to kRowMid) or the back of the list, there
        // with its place among the long rows' triplets
        if (lane == 0) {
            ucnt[r] = 0;  // until its own kernel sets it
            if (k <= kRowMid) {
                list[atomicAdd(words + kNMid, 1)] = r;
            } else {
                const int q = atomicAdd(words + kNLong, 1);
                list[n_rows - 1 - q] = r;
                base[q] = atomicAdd(words + kLongSum, k);
            }
        }
        return;
    }
    if (lane == 0) ucnt[r] = u;
}

// Rows past kRowShort, one workgroup each (a fixed grid walks the list):
// bitonic sort in LDS, padded to a power of two.
__global__ __launch_bounds__(256) void k_rows_sort_mid(const int* __restrict__ start, uint64_t* __restrict__ key,
                                                       int* __restrict__ ucnt, const int* __restrict__ words,
                                                       const int* __restrict__ list)
{
    constexpr int NT = 256;
    __shared__ uint64_t sk[kRowMid];
    __shared__ int su[NT / 64];
    const int cnt = words[kNMid];
    for (int q = blockIdx.x; q < cnt; q += gridDim.x) {
        const int r = list[q];
        const int b = start[r], k = start[r + 1] - b;
        int p2 = 2 * kRowShort;
        while (p2 < k) p2 <<= 1;
        for (int i = threadIdx.x; i < p2; i += NT) sk[i] = i < k ? key[b + i] : ~0ull;
        __syncthreads();
        for (int size = 2; size <= p2; size <<= 1)
            for (int d = size >> 1; d > 0; d >>= 1) {
                for (int t = threadIdx.x; t < p2 / 2; t += NT) {
                    const int i = 2 * t - (t & (d - 1)), j = i + d;
                    const uint64_t x = sk[i], y = sk[j];
                    if ((x > y) == ((i & size) == 0)) {
                        sk[i] = y;
                        sk[j] = x;
                    }
                }
                __syncthreads();
            }
        int u = 0;
        for (int i = threadIdx.x; i < k; i += NT) {
            key[b + i] = sk[i];
            u += (i == 0 || (sk[i - 1] >> 32) != (sk[i] >> 32)) ? 1 : 0;
        }
        u = wave_sum(u);
        if ((threadIdx.x & 63) == 0) su[threadIdx.x >> 6] = u;
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int w = 1; w < NT / 64; ++w) u += su[w];
            ucnt[r] = u;
        }
        __syncthreads();
    }
}

// sum of value e of the triplets key[j0 .. j1) in order, four loads in flight
__device__ __forceinline__ double sum_run(const double* __restrict__ tvals, const uint64_t* __restrict__ key, int j0,
                                          int j1, int e)
{
    double s = 0.0;
    int j = j0;
    for (; j + 4 <= j1; j += 4) {
        double v[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) v[t] = tvals[9 * (long)(uint32_t)key[j + t] + e];
#pragma unroll
        for (int t = 0; t < 4; ++t) s += v[t];
    }
    for (; j < j1; ++j) s += tvals[9 * (long)(uint32_t)key[j] + e];
    return s;
}

// Unique blocks of the short rows, one wave per row, 9 lanes per block, 7
// blocks at a time; a block of more than kSegChunk triplets is the ordered
// sum of its chunk sums, as in the general conversion.
// Leaves at once while the long rows' blocks are not counted (n_long: how many
// are).
__global__ __launch_bounds__(256) void k_rows_sum(const double* __restrict__ tvals, int n_rows, int n_long,
                                                  const int* __restrict__ start, const uint64_t* __restrict__ key,
                                                  const int* __restrict__ uofs, int cap, double* __restrict__ ovals,
                                                  int* __restrict__ orows, int* __restrict__ ocols,
                                                  int* __restrict__ words)
{
    __shared__ uint64_t sm[4][kRowShort];
    __shared__ int hd[4][kRowShort + 1];
    if (words[kNLong] != n_long) return;
    const int r = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (r >= n_rows) {
        if (r == n_rows && lane == 0) words[kUnique] = uofs[n_rows];
        return;
    }
    const int b = start[r], k = start[r + 1] - b;
    if (k == 0 || k > kRowShort) return;
    uint64_t* const sk = sm[threadIdx.x >> 6];
    int* const h = hd[threadIdx.x >> 6];
    const int o = uofs[r];
    int u = 0, before = -1;  // last column of the previous 64
    for (int i0 = 0; i0 < k; i0 += 64) {
        const int i = i0 + lane;
        const uint64_t w = i < k ? key[b + i] : 0ull;
        const int col = (int)(w >> 32);
        int prev = __shfl_up(col, 1, 64);
        if (lane == 0) prev = before;
        before = __shfl(col, 63, 64);
        const bool head = i < k && col != prev;
        const uint64_t m = __ballot(head);
        if (i < k) sk[i] = w;
        if (head) {
            const int q = u + __popcll(m & ((1ull << lane) - 1ull));
            h[q] = i;
            if (o + q < cap) {
                orows[o + q] = r;
                ocols[o + q] = col;
            }
        }
        u += __popcll(m);
    }
    if (lane == 0) h[u] = k;
    wave_lds_sync();
    const int g = lane / 9, e = lane % 9;
    if (g == 7) return;
    for (int q = g; q < u; q += 7) {
        const int j0 = h[q], j1 = h[q + 1];
        double s = 0.0;
        if (j1 - j0 <= kSegChunk) {
            s = sum_run(tvals, sk, j0, j1, e);
        } else {
            for (int c = j0; c < j1; c += kSegChunk) s += sum_run(tvals, sk, c, min(c + kSegChunk, j1), e);
        }
        if (o + q < cap) ovals[9 * (long)(o + q) + e] = s;
    }
}

// Unique blocks of the rows past kRowShort, one workgroup per row: the 9-lane groups
// of all waves take the blocks' chunks in turn (blocks without chunks count
// as one), then the chunk sums of each block are added in order.
__global__ __launch_bounds__(256) void k_rows_sum_mid(const double* __restrict__ tvals, int n_long,
                                                      const int* __restrict__ start, const uint64_t* __restrict__ key,
                                                      const int* __restrict__ uofs, int cap,
                                                      double* __restrict__ ovals, int* __restrict__ orows,
                                                      int* __restrict__ ocols, const int* __restrict__ words,
                                                      const int* __restrict__ list)
{
    constexpr int NT = 256;
    // chunk sums of the blocks past kSegChunk: their count is below 2 kRowMid / kSegChunk
    __shared__ double part[9 * (2 * kRowMid / kSegChunk)];
    __shared__ int head[kRowMid + 1];  // block starts
    __shared__ int wsum[NT / 64];
    constexpr int kGroups = 7 * (NT / 64);
    if (words[kNLong] != n_long) return;
    const int cnt = words[kNMid];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (int t = blockIdx.x; t < cnt; t += gridDim.x) {
        const int r = list[t];
        const int b = start[r], k = start[r + 1] - b, o = uofs[r];
        // block starts in order
        int u = 0;
        for (int i0 = 0; i0 < k; i0 += NT) {
            const int i = i0 + (int)threadIdx.x;
            const uint64_t w = i < k ? key[b + i] : 0ull;
            const bool hdf = i < k && (i == 0 || (key[b + i - 1] >> 32) != (w >> 32));
            const uint64_t m = __ballot(hdf);
            if (lane == 0) wsum[wv] = __popcll(m);
            __syncthreads();
            int before = u, all = 0;
            for (int q = 0; q < NT / 64; ++q) {
                if (q < wv) before += wsum[q];
                all += wsum[q];
            }
            if (hdf) {
                const int q = before + __popcll(m & ((1ull << lane) - 1ull));
                head[q] = i;
                if (o + q < cap) {
                    orows[o + q] = r;
                    ocols[o + q] = (int)(w >> 32);
                }
            }
            u += all;
            __syncthreads();
        }
        if (threadIdx.x == 0) head[u] = k;
        __syncthreads();
        const int g = wv * 7 + lane / 9, e = lane % 9;
        const bool use = lane < 63;
        // blocks of at most kSegChunk triplets, and the chunks of the others
        int some = 0;
        for (int q = g; q < u && use; q += kGroups) {
            const int j0 = head[q], j1 = head[q + 1];
            if (j1 - j0 > kSegChunk) {
                some = 1;
                continue;
            }
            const double s = sum_run(tvals, key + b, j0, j1, e);
            if (o + q < cap) ovals[9 * (long)(o + q) + e] = s;
        }
        if (__syncthreads_or(some) == 0) continue;
        int c = 0;  // chunks so far; every lane walks the blocks
        for (int q = 0; q < u; ++q) {
            const int j0 = head[q], j1 = head[q + 1];
            if (j1 - j0 <= kSegChunk) continue;
            const int nc = (j1 - j0 + kSegChunk - 1) / kSegChunk;
            // the group that takes chunk x is x % kGroups
            for (int x = c + (g - c % kGroups + kGroups) % kGroups; x < c + nc && use; x += kGroups) {
                const int f = j0 + (x - c) * kSegChunk;
                part[9 * x + e] = sum_run(tvals, key + b, f, min(f + kSegChunk, j1), e);
            }
            c += nc;
        }
        __syncthreads();
        c = 0;
        for (int q = 0, nl = 0; q < u; ++q) {
            const int j0 = head[q], j1 = head[q + 1];
            if (j1 - j0 <= kSegChunk) continue;
            const int nc = (j1 - j0 + kSegChunk - 1) / kSegChunk;
            if (nl++ % kGroups == g && use) {
                double s = 0.0;
                for (int x = c; x < c + nc; ++x) s += part[9 * x + e];
                if (o + q < cap) ovals[9 * (long)(o + q) + e] = s;
            }
            c += nc;
        }
        __syncthreads();
    }
}

// ---- long rows: their triplets sorted together
// rank of the row, column and index of every triplet in one key
__global__ __launch_bounds__(256) void k_long_pack(int n_rows, const int* __restrict__ list,
                                                   const int* __restrict__ base, const int* __restrict__ start,
                                                   const uint64_t* __restrict__ key, int cbits, int ibits,
                                                   uint64_t* __restrict__ out)
{
    const int q = blockIdx.x, r = list[n_rows - 1 - q];
    const int b = start[r], k = start[r + 1] - b;
    for (int i = blockIdx.y * 256 + threadIdx.x; i < k; i += gridDim.y * 256) {
        const uint64_t w = key[b + i];
        out[base[q] + i] = ((uint64_t)q << (cbits + ibits)) | ((w >> 32) << ibits) | (uint32_t)w;
    }
}
__global__ void k_long_flags(const uint64_t* __restrict__ p, int m, int ibits, int* __restrict__ flag)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < m) flag[t] = (t == 0 || (p[t] >> ibits) != (p[t - 1] >> ibits)) ? 1 : 0;
}
// triplet indices in order; per block its first triplet, row rank and column;
// per row its first block (pos: inclusive scan of the flags)
// and, added to the 0 there, its block count
__global__ void k_long_heads(const uint64_t* __restrict__ p, const int* __restrict__ flag, const int* __restrict__ pos,
                             int m, int n_rows, const int* __restrict__ list, int cbits, int ibits,
                             int* __restrict__ idx, int* __restrict__ head, int2* __restrict__ id,
                             int* __restrict__ first, int* __restrict__ ucnt)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= m) return;
    const uint64_t w = p[t];
    const int q = (int)(w >> (cbits + ibits)), at = pos[t];
    idx[t] = (int)(w & ((1ull << ibits) - 1ull));
    if (flag[t]) {
        head[at - 1] = t;
        id[at - 1] = make_int2(q, (int)((w >> ibits) & ((1ull << cbits) - 1ull)));
    }
    if (t == 0 || (int)(p[t - 1] >> (cbits + ibits)) != q) {
        first[q] = at - 1;
        atomicSub(ucnt + list[n_rows - 1 - q], at - 1);
    }
    if (t == m - 1 || (int)(p[t + 1] >> (cbits + ibits)) != q) atomicAdd(ucnt + list[n_rows - 1 - q], at);
    if (t == m - 1) head[at] = m;
}
// Chunk sums of the blocks past kSegChunk, 9 lanes per chunk.  Of 64 sorted
// triplets, at most one starts a later chunk of a block and one the first
// chunk of the next such block: places 2 w and 2 w + 1 for triplets 64 w on.
__device__ __forceinline__ int long_chunk_place(int t, bool is_first) { return 2 * (t / kSegChunk) + (is_first ? 1 : 0); }
__global__ __launch_bounds__(256) void k_long_chunks(const double* __restrict__ tvals, const int* __restrict__ idx,
                                                     const int* __restrict__ head, const int* __restrict__ pos, int m,
                                                     double* __restrict__ part)
{
    const int lane = threadIdx.x & 63, e = lane % 9;
    const long g = (blockIdx.x * 4L + (threadIdx.x >> 6)) * 7 + lane / 9;
    const long t0 = g / 2 * kSegChunk;
    if (lane == 63 || t0 >= m) return;
    const bool is_first = (g & 1) != 0;
    const int t1 = (int)min(t0 + kSegChunk, (long)m);
    const int u = pos[is_first ? t1 - 1 : t0] - 1;  // the last block that starts here, or the one that t0 lies in
    const int b = head[u], end = head[u + 1];
    const int c = is_first ? b : b + ((int)t0 - b + kSegChunk - 1) / kSegChunk * kSegChunk;
    if (end - b <= kSegChunk || c < t0 || c >= min(t1, end) || is_first != (c == b)) return;
    double s = 0.0;
#pragma unroll 4
    for (int t = c; t < min(c + kSegChunk, end); ++t) s += tvals[9 * (long)idx[t] + e];
    part[9 * g + e] = s;
}
// 9 lanes per block, 7 blocks per wave: its triplets in order, or its chunk
// sums in order
__global__ __launch_bounds__(256) void k_long_sum(const double* __restrict__ tvals, const int* __restrict__ idx,
                                                  const int* __restrict__ head, const int2* __restrict__ id,
                                                  const int* __restrict__ first, const int* __restrict__ n_blocks,
                                                  int n_rows, const int* __restrict__ list,
                                                  const double* __restrict__ part, const int* __restrict__ uofs,
                                                  int cap, double* __restrict__ ovals, int* __restrict__ orows,
                                                  int* __restrict__ ocols)
{
    const int lane = threadIdx.x & 63, e = lane % 9;
    const long u = (blockIdx.x * 4L + (threadIdx.x >> 6)) * 7 + lane / 9;
    if (lane == 63 || u >= *n_blocks) return;
    const int2 w = id[u];
    const int r = list[n_rows - 1 - w.x];
    const long o = uofs[r] + (u - first[w.x]);
    if (o >= cap) return;
    double s = 0.0;
    const int b = head[u], end = head[u + 1];
    if (end - b > kSegChunk) {
#pragma unroll 4
        for (int t = b; t < end; t += kSegChunk) s += part[9L * long_chunk_place(t, t == b) + e];
    } else {
#pragma unroll 4
        for (int t = b; t < end; ++t) s += tvals[9 * (long)idx[t] + e];
    }
    ovals[9 * o + e] = s;
    if (e == 0) {
        orows[o] = r;
        ocols[o] = w.y;
    }
}

// One atomic per workgroup (at most 512): a wave's atomic each, 1024 of them
// on one address, took longer than the 128 MB of C1's indices.
__global__ __launch_bounds__(256) void k_max_index(const int* __restrict__ rows, const int* __restrict__ cols, long n,
                                                   int* __restrict__ out)
{
    __shared__ int sm[4];
    int m = 0;
    const long stride = (long)gridDim.x * blockDim.x;
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i + 3 * stride < n; i += 4 * stride) {
        int v[8];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            v[2 * k] = rows[i + k * stride];
            v[2 * k + 1] = cols[i + k * stride];
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) m = max(m, v[k]);
    }
    for (; i < n; i += stride) m = max(m, max(rows[i], cols[i]));
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) atomicMax(out, max(max(sm[0], sm[1]), max(sm[2], sm[3])));
}

inline int g256(long n) { return (int)((n + 255) / 256); }

}  // namespace

void launch_tet_snh(hipStream_t s, int n_tets, const double* x, const uint32_t* tets, const double* dm_inv,
                    const double* vol, const double* mu, const double* lam, double dt, int hess_offset,
                    double* grad, double* tvals, int* trows, int* tcols)
{
    if (n_tets <= 0) return;
    const auto kernel = n_tets < kTetFew ? &k_tet_snh<true> : &k_tet_snh<false>;
    kernel<<<(n_tets + kTetThreads - 1) / kTetThreads, kTetThreads, 0, s>>>(
        n_tets, x, reinterpret_cast<const uint4*>(tets), dm_inv, vol, mu, lam, dt * dt, hess_offset, grad, tvals, trows,
        tcols);
    SGIPC_LAUNCH_CHECK();
}

void launch_barrier_pt(hipStream_t s, int n_pairs, const double* x, const int* pairs, const double* pair_x,
                       double dhat_sq, double kappa, int hess_offset, double* grad, double* tvals, int* trows,
                       int* tcols)
{
    if (n_pairs <= 0) return;
    k_barrier_pt<<<(n_pairs + 127) / 128, 128, 0, s>>>(n_pairs, x, reinterpret_cast<const int4*>(pairs), pair_x,
                                                       dhat_sq, kappa, hess_offset, grad, tvals, trows, tcols);
    SGIPC_LAUNCH_CHECK();
}

void launch_mass_diag(hipStream_t s, int n, const double* mass, int hess_offset, double* tvals, int* trows,
                      int* tcols)
{
    if (n <= 0) return;
    k_mass_diag<<<g256(n), 256, 0, s>>>(n, mass, hess_offset, tvals, trows, tcols);
    SGIPC_LAUNCH_CHECK();
}

int convert_max_index(hipStream_t s, const int* rows, const int* cols, long n, int* ints)
{
    launch_fill<int>(s, ints, 0, 1);
    k_max_index<<<(int)std::min<long>(512, g256(n)), 256, 0, s>>>(rows, cols, n, ints);
    SGIPC_LAUNCH_CHECK();
    int m = 0;
    SGIPC_HIP(hipMemcpyAsync(&m, ints, sizeof(int), hipMemcpyDeviceToHost, s));
    SGIPC_HIP(hipStreamSynchronize(s));
    return m;
}

size_t convert_temp_bytes(hipStream_t s, long n)
{
    size_t need = 0, need2 = 0;
    const int kbits = 31;
    SGIPC_HIP(rocprim::radix_sort_pairs(nullptr, need, static_cast<uint64_t*>(nullptr), static_cast<uint64_t*>(nullptr),
                                        static_cast<int*>(nullptr), static_cast<int*>(nullptr), (size_t)n, 0, 2 * kbits,
                                        s));
    SGIPC_HIP(rocprim::inclusive_scan(nullptr, need2, static_cast<int*>(nullptr), static_cast<int*>(nullptr), (size_t)n,
                                      rocprim::plus<int>(), s));
    size_t need3 = 0;
    SGIPC_HIP(rocprim::exclusive_scan(nullptr, need3, static_cast<int*>(nullptr), static_cast<int*>(nullptr), 0,
                                      (size_t)n, rocprim::plus<int>(), s));
    return std::max(need, std::max(need2, need3));
}

int convert_into(hipStream_t s, const ConvertScratch& w, const double* tvals, const int* trows, const int* tcols,
                 long n, int index_bound, double* ovals, int* orows, int* ocols, int capacity, int* unique)
{
    *unique = 0;
    if (n <= 0) return 0;
    SGIPC_CHECK(n < (1L << 31), SGIPC_CAPACITY, "too many triplets");
    const int kbits = Converter::index_bits(index_bound);
    // at most n unique blocks: the kernels see the capacity clamped to n
    // (same results), so the block starts need n + 1 entries at most
    const int cap = capacity < n ? capacity : (int)n;
    launch_fill<int>(s, w.ints, 0, 1);
    k_make_keys<<<g256(n), 256, 0, s>>>(trows, tcols, n, kbits, w.keys, w.idx, w.ints);
    SGIPC_LAUNCH_CHECK();
    size_t need = 0, need2 = 0;
    SGIPC_HIP(rocprim::radix_sort_pairs(nullptr, need, w.keys, w.skeys, w.idx, w.sidx, (size_t)n, 0, 2 * kbits, s));
    SGIPC_HIP(rocprim::inclusive_scan(nullptr, need2, w.flag, w.pos, (size_t)n, rocprim::plus<int>(), s));
    SGIPC_CHECK(need <= w.temp_bytes && need2 <= w.temp_bytes, SGIPC_CAPACITY,
                "conversion scratch smaller than the sort needs");
    SGIPC_HIP(rocprim::radix_sort_pairs(w.temp, need, w.keys, w.skeys, w.idx, w.sidx, (size_t)n, 0, 2 * kbits, s));
    k_head_flags<<<g256(n), 256, 0, s>>>(w.skeys, n, w.flag);
    SGIPC_LAUNCH_CHECK();
    SGIPC_HIP(rocprim::inclusive_scan(w.temp, need2, w.flag, w.pos, (size_t)n, rocprim::plus<int>(), s));
    k_heads<<<g256(n), 256, 0, s>>>(w.skeys, w.flag, w.pos, n, kbits, w.head, orows, ocols, cap);
    SGIPC_LAUNCH_CHECK();
    if (cap > 0) {
        // long blocks in chunks: counts into flag, their exclusive prefix into
        // idx, the chunk sums into keys (both free after the sort and scan;
        // at most 2 n / kSegChunk chunks of 9 doubles fit in n words)
        int* cnt = w.flag;
        int* cofs = w.idx;
        double* part = reinterpret_cast<double*>(w.keys);
        k_seg_chunks<<<g256(cap), 256, 0, s>>>(w.head, w.pos, n, cap, cnt);
        SGIPC_LAUNCH_CHECK();
        size_t need3 = 0;
        SGIPC_HIP(rocprim::exclusive_scan(nullptr, need3, cnt, cofs, 0, (size_t)cap, rocprim::plus<int>(), s));
        SGIPC_CHECK(need3 <= w.temp_bytes, SGIPC_CAPACITY, "conversion scratch smaller than the scan needs");
        SGIPC_HIP(rocprim::exclusive_scan(w.temp, need3, cnt, cofs, 0, (size_t)cap, rocprim::plus<int>(), s));
        const long bound = 2 * n / kSegChunk + 1;
        k_chunk_sum<<<g256(bound), 256, 0, s>>>(tvals, w.sidx, w.head, cnt, cofs, cap, bound, part);
        SGIPC_LAUNCH_CHECK();
        k_segment_sum<<<g256(cap), 256, 0, s>>>(tvals, w.sidx, w.head, w.pos, n, ovals, cap, cnt, cofs, part);
        SGIPC_LAUNCH_CHECK();
    }
    int h[2] = {0, 0};
    SGIPC_HIP(hipMemcpyAsync(&h[0], w.pos + (n - 1), sizeof(int), hipMemcpyDeviceToHost, s));
    SGIPC_HIP(hipMemcpyAsync(&h[1], w.ints, sizeof(int), hipMemcpyDeviceToHost, s));
    SGIPC_HIP(hipStreamSynchronize(s));
    SGIPC_CHECK(h[1] == 0, SGIPC_BAD_INDEX, "triplet with row > col, a negative index or an index beyond the bound");
    *unique = h[0];
    SGIPC_CHECK(h[0] <= capacity, SGIPC_CAPACITY, "unique block count exceeds the output capacity");
    return h[0];
}

int Converter::index_bits(int bound)
{
    int k = 1;
    while (k < 31 && (1L << k) < (long)bound) ++k;
    return k;
}

int Converter::max_index(hipStream_t s, const int* rows, const int* cols, long n)
{
    scratch_int_.reserve(4);
    return convert_max_index(s, rows, cols, n, scratch_int_.get());
}

bool Converter::convert_rows(hipStream_t s, const double* tvals, const int* trows, const int* tcols, long n,
                             int n_rows, double* ovals, int* orows, int* ocols, int capacity, int* unique)
{
    const long R = n_rows;
    row_cnt_.reserve(R + 1 + kRowWords);
    row_start_.reserve(R + 1);
    row_ucnt_.reserve(R + 1);
    row_uofs_.reserve(R + 1);
    row_list_.reserve(R > 0 ? R : 1);
    row_base_.reserve(n / kRowMid + 1);
    keys_.reserve(n);
    int* const cnt = row_cnt_.get();
    int* const words = cnt + R + 1;
    size_t need = 0;
    SGIPC_HIP(rocprim::exclusive_scan(nullptr, need, cnt, row_start_.get(), 0, (size_t)(R + 1), rocprim::plus<int>(), s));
    temp_.reserve(need);
    launch_fill<int>(s, cnt, 0, R + 1 + kRowWords);
    const int gb = (int)((n + 256 * kRowItems - 1) / (256 * kRowItems));
    k_rows_bin<false><<<gb, 256, 0, s>>>(trows, tcols, n, n_rows, cnt, words, nullptr, nullptr);
    SGIPC_LAUNCH_CHECK();
    SGIPC_HIP(rocprim::exclusive_scan(temp_.get(), need, cnt, row_start_.get(), 0, (size_t)(R + 1),
                                      rocprim::plus<int>(), s));
    k_rows_bin<true><<<gb, 256, 0, s>>>(trows, tcols, n, n_rows, cnt, words, row_start_.get(), keys_.get());
    SGIPC_LAUNCH_CHECK();
    const int gr = (int)((R + 1 + 3) / 4);
    k_rows_sort<<<gr, 256, 0, s>>>(n_rows, row_start_.get(), keys_.get(), row_ucnt_.get(), words, row_list_.get(),
                                   row_base_.get());
    SGIPC_LAUNCH_CHECK();
    // rows past kRowShort: a grid that walks the list (its length stays on the device)
    const int g_mid = (int)std::min<long>(1024, n / kRowShort);
    if (g_mid > 0) {
        k_rows_sort_mid<<<g_mid, 256, 0, s>>>(row_start_.get(), keys_.get(), row_ucnt_.get(), words, row_list_.get());
        SGIPC_LAUNCH_CHECK();
    }
    // the blocks' places and sums, but those of n_long long rows
    auto sums = [&](int n_long) {
        SGIPC_HIP(rocprim::exclusive_scan(temp_.get(), need, row_ucnt_.get(), row_uofs_.get(), 0, (size_t)(R + 1),
                                          rocprim::plus<int>(), s));
        k_rows_sum<<<gr, 256, 0, s>>>(tvals, n_rows, n_long, row_start_.get(), keys_.get(), row_uofs_.get(), capacity,
                                      ovals, orows, ocols, words);
        SGIPC_LAUNCH_CHECK();
        if (g_mid > 0) {
            k_rows_sum_mid<<<g_mid, 256, 0, s>>>(tvals, n_long, row_start_.get(), keys_.get(), row_uofs_.get(),
                                                 capacity, ovals, orows, ocols, words, row_list_.get());
            SGIPC_LAUNCH_CHECK();
        }
    };
    int h[kRowWords];
    auto read_words = [&] {
        SGIPC_HIP(hipMemcpyAsync(h, words, sizeof(h), hipMemcpyDeviceToHost, s));
        SGIPC_HIP(hipStreamSynchronize(s));
    };
    sums(0);
    read_words();
    SGIPC_CHECK(h[kBad] == 0, SGIPC_BAD_INDEX,
                "triplet with row > col, a negative index or an index beyond the bound");
    const int n_long = h[kNLong], m = h[kLongSum];
    if (n_long > 0) {
        const int qbits = index_bits(n_long), cbits = index_bits(n_rows), ibits = index_bits((int)n);
        if (m > n / 2 || qbits + cbits + ibits > 64) return false;
        skeys_.reserve(2L * m);
        idx_.reserve(m);
        flag_.reserve(m);
        pos_.reserve(m);
        head_.reserve(m + 1L);
        long_id_.reserve(m);
        row_first_.reserve(n_long);
        uint64_t* const packed = skeys_.get();
        uint64_t* const sorted = packed + m;
        size_t n1 = 0, n2 = 0;
        SGIPC_HIP(rocprim::radix_sort_keys(nullptr, n1, packed, sorted, (size_t)m, 0, qbits + cbits + ibits, s));
        SGIPC_HIP(rocprim::inclusive_scan(nullptr, n2, flag_.get(), pos_.get(), (size_t)m, rocprim::plus<int>(), s));
        temp_.reserve(std::max(std::max(n1, n2), need));
        const unsigned gy = (unsigned)std::min<long>(64, m / n_long / 1024 + 1);
        k_long_pack<<<dim3(n_long, gy), 256, 0, s>>>(n_rows, row_list_.get(), row_base_.get(), row_start_.get(),
                                                     keys_.get(), cbits, ibits, packed);
        SGIPC_LAUNCH_CHECK();
        SGIPC_HIP(rocprim::radix_sort_keys(temp_.get(), n1, packed, sorted, (size_t)m, 0, qbits + cbits + ibits, s));
        k_long_flags<<<g256(m), 256, 0, s>>>(sorted, m, ibits, flag_.get());
        SGIPC_LAUNCH_CHECK();
        SGIPC_HIP(rocprim::inclusive_scan(temp_.get(), n2, flag_.get(), pos_.get(), (size_t)m, rocprim::plus<int>(), s));
        k_long_heads<<<g256(m), 256, 0, s>>>(sorted, flag_.get(), pos_.get(), m, n_rows, row_list_.get(), cbits, ibits,
                                             idx_.get(), head_.get(), long_id_.get(), row_first_.get(), row_ucnt_.get());
        SGIPC_LAUNCH_CHECK();
        sums(n_long);
        // chunk sums over the packed keys (2 of 9 doubles for every 64 triplets)
        double* const part = reinterpret_cast<double*>(packed);
        const long places = 2 * ((m + (long)kSegChunk - 1) / kSegChunk);
        k_long_chunks<<<(int)((places + 27) / 28), 256, 0, s>>>(tvals, idx_.get(), head_.get(), pos_.get(), m, part);
        SGIPC_LAUNCH_CHECK();
        k_long_sum<<<(m + 27) / 28, 256, 0, s>>>(tvals, idx_.get(), head_.get(), long_id_.get(), row_first_.get(),
                                                 pos_.get() + (m - 1), n_rows, row_list_.get(), part, row_uofs_.get(),
                                                 capacity, ovals, orows, ocols);
        SGIPC_LAUNCH_CHECK();
        read_words();
    }
    *unique = h[kUnique];
    SGIPC_CHECK(*unique <= capacity, SGIPC_CAPACITY, "unique block count exceeds the output capacity");
    return true;
}

int Converter::convert(hipStream_t s, const double* tvals, const int* trows, const int* tcols, long n,
                       int index_bound, double* ovals, int* orows, int* ocols, int capacity, bool long_rows)
{
    if (n <= 0) return 0;
    SGIPC_CHECK(n < (1L << 31), SGIPC_CAPACITY, "too many triplets");
    // By rows unless the rows are so few that they must be long, or so many
    // that their tables outweigh the triplets, or the caller or the count says
    // that much lies in long rows (0.35 M triplets, a third of them in 8 rows:
    // 0.70 ms by rows, each long one sorted by a workgroup, against 0.34).
    // Coarse levels with 400 to 1600 triplets a row: 44k to 1.4 M of them
    // 0.12 .. 0.28 ms against 0.21 .. 0.36, 5.6 M 0.68 against 0.70.
    if (!long_rows && index_bound < (1L << 31) - 8 && n <= 2048L * index_bound && index_bound <= 4 * n + 4096 &&
        convert_rows(s, tvals, trows, tcols, n, index_bound, ovals, orows, ocols, capacity, &last_unique))
        return last_unique;
    keys_.reserve(n);
    skeys_.reserve(n);
    idx_.reserve(n);
    sidx_.reserve(n);
    flag_.reserve(n);
    pos_.reserve(n);
    head_.reserve((size_t)(capacity < n ? capacity : n) + 1);
    scratch_int_.reserve(4);
    temp_.reserve(convert_temp_bytes(s, n));
    ConvertScratch w;
    w.keys = keys_.get();
    w.skeys = skeys_.get();
    w.idx = idx_.get();
    w.sidx = sidx_.get();
    w.flag = flag_.get();
    w.pos = pos_.get();
    w.head = head_.get();
    w.ints = scratch_int_.get();
    w.temp = temp_.get();
    w.temp_bytes = temp_.n;
    return convert_into(s, w, tvals, trows, tcols, n, index_bound, ovals, orows, ocols, capacity, &last_unique);
}

}  // namespace sgipc
