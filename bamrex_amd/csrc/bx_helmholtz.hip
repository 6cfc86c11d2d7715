// Variable-coefficient pressure Helmholtz solve of the IMEX (PEEK/PESK)
// schemes on one 2D periodic level: the operator, a geometric multigrid with
// the semantics of AMReX MLMG (the reference's "plain MLMG" solver) and an
// FP64 flexible GMRES whose preconditioner is a multigrid V-cycle or a
// V-cycle whose fine-level smoothing is a learned convolutional correction.
//
// Reference path (Source/IMEX/IMEX_O1.cpp:392-414, 570-640):
//   A p = alpha a p - beta div(b grad p) + gamma c . grad p
//   alpha = 1, a = eps/(gamma-1), beta = adt^2, b = face-averaged enthalpy,
//   gamma = -eps adt/2 (split KE) or 0 (PEEK)      setup_pressure_op
//   apply:   mlalapgrad_adotx   Source/LinearSolver/MLALapGrad_2D_K.H:9-33
//   smooth:  alapgrad_gsrb      Source/LinearSolver/MLALapGrad_2D_K.H:179-229
//            with dhx = beta/(h*h), cdhx = gamma/(2h) (MLALaplacianGrad.H:1243-1249)
//   coarse coefficients: average_down of a and c, average_down_faces of b
//            (MLALaplacianGrad.H:950-1027)
// MLMG defaults restated (AMReX is not available here): V-cycle, 2 pre- and
// 2 post-smoothing red-black sweeps, cell-average restriction, piecewise
// constant interpolation, coarsening by 2 while both extents stay even and
// >= 8; the bottom level gets nu_bottom (default 16) red-black sweep pairs
// (AMReX's GPU default bottom solver is BiCGStab; on these mass-term
// operators the coarsest level is diagonally dominant and the sweeps
// converge it).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/bamrex_hip.h"
#include "bx_helmholtz.h"
#include "bx_mail.h"
#include "bx_smooth.h"

namespace bx {

// ------------------------------------------------------------- kernels
// Cell operations shared by the grid kernels and the single-workgroup tail
// of the V-cycle, so both give the same bits.

// (A x) of one cell from its value, its four neighbours' and its
// coefficients (mlalapgrad_adotx); dhx = beta dxinv dxinv, dhy likewise
template <class T>
__device__ __forceinline__ T apply_vals(T xc, T xl, T xr, T xd, T xu, T a_c, T bxl, T bxr,
                                        T byl, T byr, T cx, T cy, bool with_c, T alpha,
                                        T dhx, T dhy, T gamma, T dxinv, T dyinv)
{
    T v = alpha * a_c * xc - dhx * (bxr * (xr - xc) - bxl * (xc - xl))
          - dhy * (byr * (xu - xc) - byl * (xc - xd));
    if (with_c)
    {
        const T chdx = gamma * cx * T(0.5) * dxinv;
        const T chdy = gamma * cy * T(0.5) * dyinv;
        v = v + chdx * (xr - xl) + chdy * (xu - xd);
    }
    return v;
}

// (A x)_ij on a periodic level (mlalapgrad_adotx)
template <class T>
__device__ __forceinline__ T apply_at(const T *__restrict__ x, const T *__restrict__ a,
                                      const T *__restrict__ bX, const T *__restrict__ bY,
                                      const T *__restrict__ cX, const T *__restrict__ cY,
                                      int nx, int ny, T alpha, T beta, T gamma, T dxinv,
                                      T dyinv, int i, int j)
{
    const int im = i == 0 ? nx - 1 : i - 1, ip = i == nx - 1 ? 0 : i + 1;
    const int jm = j == 0 ? ny - 1 : j - 1, jp = j == ny - 1 ? 0 : j + 1;
    const long long c   = (long long)j * nx + i;
    const T         xc  = x[c];
    const T         dhx = beta * dxinv * dxinv;
    const T         dhy = beta * dyinv * dyinv;
    // faces: bX(i,j) at j*(nx+1)+i, bY(i,j) at j*nx+i
    const T bxl = bX[(long long)j * (nx + 1) + i];
    const T bxr = bX[(long long)j * (nx + 1) + i + 1];
    const T byl = bY[(long long)j * nx + i];
    const T byr = bY[(long long)(j + 1) * nx + i];
    const T xl = x[(long long)j * nx + im], xr = x[(long long)j * nx + ip];
    const T xd = x[(long long)jm * nx + i], xu = x[(long long)jp * nx + i];
    return apply_vals(xc, xl, xr, xd, xu, a[c], bxl, bxr, byl, byr, cX ? cX[c] : T(0),
                      cY ? cY[c] : T(0), cX != nullptr, alpha, dhx, dhy, gamma, dxinv, dyinv);
}

// red/black Gauss-Seidel update of cell (i, j) (alapgrad_gsrb; periodic
// level: no boundary correction, delta = 0)
// the cell update of red/black Gauss-Seidel from its neighbours' values
template <class T>
__device__ __forceinline__ T gsrb_value(T rhs_c, T a_c, T bxl, T bxr, T byl, T byr, T cx,
                                        T cy, bool with_c, T pl, T pr, T pd, T pu, T phi_c,
                                        T alpha, T dhx, T dhy, T cdhx, T cdhy)
{
    const T gamma = alpha * a_c + dhx * (bxl + bxr) + dhy * (byl + byr);
    T rho = dhx * (bxl * pl + bxr * pr) + dhy * (byl * pd + byr * pu);
    if (with_c)
        rho = rho - cdhx * cx * (pr - pl) - cdhy * cy * (pu - pd);
    return (rhs_c + rho - phi_c * T(0)) / (gamma - T(0));
}

template <class T>
__device__ __forceinline__ void gsrb_at(T *__restrict__ phi, const T *__restrict__ rhs,
                                        const T *__restrict__ a, const T *__restrict__ bX,
                                        const T *__restrict__ bY, const T *__restrict__ cX,
                                        const T *__restrict__ cY, int nx, int ny, T alpha,
                                        T dhx, T dhy, T cdhx, T cdhy, int i, int j)
{
    const int im = i == 0 ? nx - 1 : i - 1, ip = i == nx - 1 ? 0 : i + 1;
    const int jm = j == 0 ? ny - 1 : j - 1, jp = j == ny - 1 ? 0 : j + 1;
    const long long c   = (long long)j * nx + i;
    const T bxl = bX[(long long)j * (nx + 1) + i];
    const T bxr = bX[(long long)j * (nx + 1) + i + 1];
    const T byl = bY[(long long)j * nx + i];
    const T byr = bY[(long long)(j + 1) * nx + i];
    const T pl = phi[(long long)j * nx + im], pr = phi[(long long)j * nx + ip];
    const T pd = phi[(long long)jm * nx + i], pu = phi[(long long)jp * nx + i];
    phi[c] = gsrb_value(rhs[c], a[c], bxl, bxr, byl, byr, cX ? cX[c] : T(0),
                        cY ? cY[c] : T(0), cX != nullptr, pl, pr, pd, pu, phi[c], alpha, dhx,
                        dhy, cdhx, cdhy);
}

template <class T>
__device__ __forceinline__ T restrict_at(const T *__restrict__ f, int ncx, int I, int J)
{
    const int       nfx = 2 * ncx;
    const long long f0  = (long long)(2 * J) * nfx + 2 * I;
    return T(0.25) * (f[f0] + f[f0 + 1] + f[f0 + nfx] + f[f0 + nfx + 1]);
}

template <class T>
__global__ __launch_bounds__(256) void k_apply(
    const T *__restrict__ x, T *__restrict__ y, const T *__restrict__ a,
    const T *__restrict__ bX, const T *__restrict__ bY,
    const T *__restrict__ cX, const T *__restrict__ cY, int nx, int ny,
    const T *__restrict__ sc, T dxinv, T dyinv, const T *__restrict__ rhs)
{
    // sc = (alpha, beta, gamma) in device memory, so that a captured graph
    // stays valid when the scalars change from one solve to the next
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int j = blockIdx.y;
    if (i >= nx)
        return;
    const long long c = (long long)j * nx + i;
    const T v = apply_at(x, a, bX, bY, cX, cY, nx, ny, sc[0], sc[1], sc[2], dxinv, dyinv, i, j);
    // residual form when rhs is given: y = rhs - A x
    y[c] = rhs ? rhs[c] - v : v;
}

template <class T>
__global__ __launch_bounds__(256) void k_gsrb(
    T *__restrict__ phi, const T *__restrict__ rhs, const T *__restrict__ a,
    const T *__restrict__ bX, const T *__restrict__ bY,
    const T *__restrict__ cX, const T *__restrict__ cY, int nx, int ny,
    const T *__restrict__ sc, T hx, T hy, int redblack)
{
    const T alpha = sc[0];
    const T dhx = sc[1] / (hx * hx), dhy = sc[1] / (hy * hy);
    const T cdhx = sc[2] / (2 * hx), cdhy = sc[2] / (2 * hy);
    // thread covers cells of one colour: i = 2*t + ((j + redblack) & 1)
    const int j = blockIdx.y;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int i = 2 * t + ((j + redblack) & 1);
    if (i >= nx)
        return;
    gsrb_at(phi, rhs, a, bX, bY, cX, cY, nx, ny, alpha, dhx, dhy, cdhx, cdhy, i, j);
}

template <class T>
__global__ __launch_bounds__(256) void k_restrict(const T *__restrict__ f,
                                                  T *__restrict__ c, int ncx,
                                                  int ncy)
{
    const int I = blockIdx.x * blockDim.x + threadIdx.x;
    const int J = blockIdx.y;
    if (I >= ncx)
        return;
    c[(long long)J * ncx + I] = restrict_at(f, ncx, I, J);
}

template <class T>
__global__ __launch_bounds__(256) void k_prolong_add(const T *__restrict__ c,
                                                     T *__restrict__ f, int nfx,
                                                     int nfy)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int j = blockIdx.y;
    if (i >= nfx)
        return;
    f[(long long)j * nfx + i] += c[(long long)(j >> 1) * (nfx >> 1) + (i >> 1)];
}

// coarse rhs = R (rhs - A x) on the fine level in one launch (the residual
// values and the averaging order of k_apply + k_restrict)
template <class T>
__global__ __launch_bounds__(256) void k_resid_restrict(
    const T *__restrict__ x, const T *__restrict__ rhs, const T *__restrict__ a,
    const T *__restrict__ bX, const T *__restrict__ bY, const T *__restrict__ cX,
    const T *__restrict__ cY, int nx, int ny, const T *__restrict__ sc, T dxinv, T dyinv,
    T *__restrict__ crhs)
{
    const int I = blockIdx.x * blockDim.x + threadIdx.x;
    const int J = blockIdx.y;
    const int ncx = nx >> 1;
    if (I >= ncx)
        return;
    const T alpha = sc[0], beta = sc[1], gamma = sc[2];
    T r[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
    {
        const int i = 2 * I + (q & 1), j = 2 * J + (q >> 1);
        r[q] = rhs[(long long)j * nx + i]
               - apply_at(x, a, bX, bY, cX, cY, nx, ny, alpha, beta, gamma, dxinv, dyinv, i, j);
    }
    crhs[(long long)J * ncx + I] = T(0.25) * (r[0] + r[1] + r[2] + r[3]);
}

// coarse face coefficients: average of the two fine faces on the coarse face
template <class T>
__global__ void k_avg_faces_x(const T *__restrict__ f, T *__restrict__ c,
                              int ncx, int ncy)
{
    const int I = blockIdx.x * blockDim.x + threadIdx.x; // 0..ncx
    const int J = blockIdx.y;
    if (I > ncx)
        return;
    const int nfx = 2 * ncx;
    c[(long long)J * (ncx + 1) + I]
        = T(0.5) * (f[(long long)(2 * J) * (nfx + 1) + 2 * I]
                    + f[(long long)(2 * J + 1) * (nfx + 1) + 2 * I]);
}

// One launch per coarse level for all its coefficients: a (and c) by cell
// average (k_restrict), bX / bY by face average (k_avg_faces_x / _y); the
// same expressions, so the same bits.  Grid (ncx + 1) x (ncy + 1).
template <class T>
__device__ __forceinline__ void coarsen_at(
    const T *__restrict__ fa, const T *__restrict__ fbX, const T *__restrict__ fbY,
    const T *__restrict__ fcX, const T *__restrict__ fcY, T *__restrict__ ca,
    T *__restrict__ cbX, T *__restrict__ cbY, T *__restrict__ ccX, T *__restrict__ ccY,
    int ncx, int ncy, int I, int J)
{
    const int nfx = 2 * ncx;
    if (J < ncy)
    {
        cbX[(long long)J * (ncx + 1) + I]
            = T(0.5) * (fbX[(long long)(2 * J) * (nfx + 1) + 2 * I]
                        + fbX[(long long)(2 * J + 1) * (nfx + 1) + 2 * I]);
        if (I < ncx)
        {
            ca[(long long)J * ncx + I] = restrict_at(fa, ncx, I, J);
            if (fcX)
            {
                ccX[(long long)J * ncx + I] = restrict_at(fcX, ncx, I, J);
                ccY[(long long)J * ncx + I] = restrict_at(fcY, ncx, I, J);
            }
        }
    }
    if (I < ncx)
        cbY[(long long)J * ncx + I] = T(0.5)
                                      * (fbY[(long long)(2 * J) * nfx + 2 * I]
                                         + fbY[(long long)(2 * J) * nfx + 2 * I + 1]);
}

template <class T>
__global__ __launch_bounds__(256) void k_coarsen_coeffs(
    const T *__restrict__ fa, const T *__restrict__ fbX, const T *__restrict__ fbY,
    const T *__restrict__ fcX, const T *__restrict__ fcY, T *__restrict__ ca,
    T *__restrict__ cbX, T *__restrict__ cbY, T *__restrict__ ccX, T *__restrict__ ccY,
    int ncx, int ncy)
{
    const int I = blockIdx.x * blockDim.x + threadIdx.x; // 0..ncx
    const int J = blockIdx.y;                            // 0..ncy
    if (I <= ncx)
        coarsen_at(fa, fbX, fbY, fcX, fcY, ca, cbX, cbY, ccX, ccY, ncx, ncy, I, J);
}

// The small coarse levels of a hierarchy, finest first, in one workgroup
// (a barrier between levels): the same expressions as k_coarsen_coeffs.
constexpr int COARSEN_MAX_LEVELS = 12;
constexpr int COARSEN_SMALL      = 64 * 64; // coarse levels up to this many cells
template <class T> struct CoarsenLevel
{
    const T *fa, *fbX, *fbY, *fcX, *fcY;
    T       *ca, *cbX, *cbY, *ccX, *ccY;
    int      ncx, ncy;
};
template <class T> struct CoarsenList
{
    int             n;
    CoarsenLevel<T> lev[COARSEN_MAX_LEVELS];
};

template <class T>
__global__ __launch_bounds__(1024) void k_coarsen_small(CoarsenList<T> cl)
{
    for (int l = 0; l < cl.n; ++l)
    {
        const CoarsenLevel<T> &c  = cl.lev[l];
        const int              w  = c.ncx + 1;
        const int              nq = w * (c.ncy + 1);
        for (int q = threadIdx.x; q < nq; q += 1024)
        {
            const int J = q / w, I = q - J * w;
            coarsen_at(c.fa, c.fbX, c.fbY, c.fcX, c.fcY, c.ca, c.cbX, c.cbY, c.ccX, c.ccY,
                       c.ncx, c.ncy, I, J);
        }
        __syncthreads();
    }
}

template <class T>
__global__ void k_avg_faces_y(const T *__restrict__ f, T *__restrict__ c,
                              int ncx, int ncy)
{
    const int I = blockIdx.x * blockDim.x + threadIdx.x;
    const int J = blockIdx.y; // 0..ncy
    if (I >= ncx)
        return;
    const int nfx = 2 * ncx;
    c[(long long)J * ncx + I] = T(0.5)
                                * (f[(long long)(2 * J) * nfx + 2 * I]
                                   + f[(long long)(2 * J) * nfx + 2 * I + 1]);
}

template <class TO, class TI>
__global__ __launch_bounds__(256) void k_convert(const TI *__restrict__ in,
                                                 TO *__restrict__ out,
                                                 long long n, TI scale)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
        out[i] = (TO)(in[i] * scale);
}

// Level-0 coefficients of a hierarchy from FP64 arrays, and its scalars
// (alpha, beta, gamma) into device memory, one launch:
// a, c over nx*ny cells, bX over (nx+1)*ny faces, bY over nx*(ny+1).
template <class T>
__global__ __launch_bounds__(256) void k_convert_coeffs(
    const double *__restrict__ a, const double *__restrict__ bX,
    const double *__restrict__ bY, const double *__restrict__ cX,
    const double *__restrict__ cY, T *__restrict__ oa, T *__restrict__ obX,
    T *__restrict__ obY, T *__restrict__ ocX, T *__restrict__ ocY, int nx, int ny,
    T *__restrict__ sc, T alpha, T beta, T gamma)
{
    if (blockIdx.x == 0 && threadIdx.x == 0)
    {
        sc[0] = alpha;
        sc[1] = beta;
        sc[2] = gamma;
    }
    const long long n   = (long long)nx * ny;
    const long long nbx = (long long)(nx + 1) * ny;
    const long long nby = (long long)nx * (ny + 1);
    const long long nm  = nbx > nby ? nbx : nby;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < nm;
         i += (long long)gridDim.x * blockDim.x)
    {
        if (i < n)
        {
            oa[i] = (T)a[i];
            if (cX)
            {
                ocX[i] = (T)cX[i];
                ocY[i] = (T)cY[i];
            }
        }
        if (i < nbx)
            obX[i] = (T)bX[i];
        if (i < nby)
            obY[i] = (T)bY[i];
    }
}

template <class T>
__global__ __launch_bounds__(256) void k_fill(T *__restrict__ p, long long n,
                                              T v)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
        p[i] = v;
}

// y += alpha * x  (alpha from a device scalar times a host factor)
__global__ __launch_bounds__(256) void k_axpy(double *__restrict__ y,
                                              const double *__restrict__ x,
                                              long long n, double alpha)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
        y[i] = y[i] + alpha * x[i];
}

__global__ __launch_bounds__(256) void k_scale(double *__restrict__ y,
                                               const double *__restrict__ x,
                                               long long n, double s)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
        y[i] = x[i] * s;
}

// partial dot products of w with k vectors V[0..k-1] (stride n)
__global__ __launch_bounds__(256) void k_multidot(
    const double *__restrict__ V, const double *__restrict__ w, long long n,
    int k, double *__restrict__ partial)
{
    __shared__ double sh[8][16];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (int v0 = 0; v0 < k; v0 += 16)
    {
        const int nv = min(16, k - v0);
        double    acc[16];
#pragma unroll
        for (int q = 0; q < 16; ++q)
            acc[q] = 0;
        for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
             i < n; i += (long long)gridDim.x * blockDim.x)
        {
            const double wi = w[i];
#pragma unroll
            for (int q = 0; q < 16; ++q)
                if (q < nv)
                    acc[q] += V[(long long)(v0 + q) * n + i] * wi;
        }
#pragma unroll
        for (int q = 0; q < 16; ++q)
        {
            double s = acc[q];
            for (int off = 32; off > 0; off >>= 1)
                s += __shfl_xor(s, off);
            if (lane == 0)
                sh[wv][q] = s;
        }
        __syncthreads();
        if (threadIdx.x < nv)
        {
            double s = 0;
            for (int q = 0; q < (int)(blockDim.x >> 6); ++q)
                s += sh[q][threadIdx.x];
            partial[(long long)(v0 + threadIdx.x) * gridDim.x + blockIdx.x] = s;
        }
        __syncthreads();
    }
}

// r = rhs - A x (k_apply's residual) and, in the same pass, the sums of r^2
// and with BN of rhs^2, in the next message: partial sums (rows 0 and 1 of
// `partial`) with the grid, the per-thread order and the reduction tree of
// k_multidot(., ., k = 1), added by the last block in the order of
// k_reduce_partials.  With stop.stop the message says instead of the second
// sum whether the solve goes on (the first sum's root, the residual norm,
// above tol), and its end is recorded if not.  Launched with nb_dot blocks of
// 256 threads; the level has at most 2^31 - 1 cells.  Bound by memory at large
// sizes, by latency at small ones; with a launch of its own for the sum of the
// partials it took 12.7 + 5.4 us at 1024^2, now 15.8, and 4.7 + 4.1 at 160 x
// 96, now 6.3.
template <bool BN>
__global__ __launch_bounds__(256) void k_residual_sumsq(
    const double *__restrict__ x, double *__restrict__ r, const double *__restrict__ rhs,
    const double *__restrict__ a, const double *__restrict__ bX,
    const double *__restrict__ bY, const double *__restrict__ cX,
    const double *__restrict__ cY, int nx, int ny, const double *__restrict__ sc,
    double dxinv, double dyinv, double *partial, StopCheck stop, NormMail nm)
{
    __shared__ double sh[2][4], red[BN ? 2 : 1][256];
    if (stop())
        return;
    const int    lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int    n    = nx * ny;
    const double al = sc[0], be = sc[1], ga = sc[2];
    double       acc[2] = { 0, 0 };
    for (long long q = (long long)blockIdx.x * 256 + threadIdx.x; q < n;
         q += (long long)gridDim.x * 256)
    {
        const int    c  = (int)q, j = c / nx, i = c - j * nx;
        const double bi = rhs[c];
        const double ri = bi - apply_at(x, a, bX, bY, cX, cY, nx, ny, al, be, ga, dxinv,
                                        dyinv, i, j);
        r[c] = ri;
        acc[0] += ri * ri;
        if (BN)
            acc[1] += bi * bi;
    }
#pragma unroll
    for (int v = 0; v < (BN ? 2 : 1); ++v)
    {
        double s = acc[v];
        for (int off = 32; off > 0; off >>= 1)
            s += __shfl_xor(s, off);
        if (lane == 0)
            sh[v][wv] = s;
    }
    __syncthreads();
    if (threadIdx.x < (BN ? 2 : 1))
    {
        double t = 0;
        for (int q = 0; q < 4; ++q)
            t += sh[threadIdx.x][q];
        put_partial(partial + (long long)threadIdx.x * gridDim.x + blockIdx.x, t);
    }
    if (!last_block(nm.count))
        return;
    double v[2] = { 0, 0 };
#pragma unroll
    for (int q = 0; q < (BN ? 2 : 1); ++q)
        v[q] = block_sum_partials(partial + (long long)q * gridDim.x, gridDim.x, red[q]);
    if (threadIdx.x == 0)
        nm.post(v[0], v[1], stop);
}

// y = x / sqrt(d[0]) when d[0] > 0 (the new Arnoldi vector)
__global__ __launch_bounds__(256) void k_scale_inv_norm(double *__restrict__ y,
                                                        const double *__restrict__ x,
                                                        long long n,
                                                        const double *__restrict__ d)
{
    const double hn = sqrt(d[0]);
    if (!(hn > 0))
        return;
    const double s = 1.0 / hn;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
        y[i] = x[i] * s;
}

__global__ void k_reduce_partials(const double *__restrict__ partial, int nb,
                                  int k, double *__restrict__ out)
{
    // one block per vector
    __shared__ double sh[256];
    const int v = blockIdx.x;
    double    s = 0;
    for (int b = threadIdx.x; b < nb; b += blockDim.x)
        s += partial[(long long)v * nb + b];
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int off = blockDim.x / 2; off > 0; off >>= 1)
    {
        if ((int)threadIdx.x < off)
            sh[threadIdx.x] += sh[threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0)
        out[v] = sh[0];
}

// w -= sum_q h[q] V[q]
__global__ __launch_bounds__(256) void k_subtract_combo(
    double *__restrict__ w, const double *__restrict__ V,
    const double *__restrict__ h, int k, long long n)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
    {
        double s = w[i];
        for (int q = 0; q < k; ++q)
            s -= h[q] * V[(long long)q * n + i];
        w[i] = s;
    }
}

// x += sum_q y[q] Z[q]
__global__ __launch_bounds__(256) void k_add_combo(double *__restrict__ x,
                                                   const double *__restrict__ Z,
                                                   const double *__restrict__ y,
                                                   int k, long long n)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
    {
        double s = x[i];
        for (int q = 0; q < k; ++q)
            s += y[q] * Z[(long long)q * n + i];
        x[i] = s;
    }
}

// ---- one FGMRES iteration's vector work in fewer passes ----------------
// The kernels hold K >= k sums per thread (K a compile-time 1, 2, 4, 8 or 16,
// so that the sums are registers); the sums and their order do not depend on
// K.  Bound by memory: k_apply_multidot at 1024^2 with one vector took 19.5 us
// with 16 sums (in scratch memory: their loops were not unrolled).
// Block partial sums of k dot products, one row of gridDim.x partials per
// vector (layout as k_multidot's), from per-thread sums.
template <int K>
__device__ __forceinline__ void block_partials(const double (&acc)[K], int k,
                                               double *__restrict__ partial)
{
    __shared__ double sh[4][K];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
    for (int q = 0; q < K; ++q)
    {
        double v = acc[q];
        for (int off = 32; off > 0; off >>= 1)
            v += __shfl_xor(v, off);
        if (lane == 0)
            sh[wv][q] = v;
    }
    __syncthreads();
    if ((int)threadIdx.x < k)
        partial[(long long)threadIdx.x * gridDim.x + blockIdx.x]
            = (sh[0][threadIdx.x] + sh[1][threadIdx.x]) + (sh[2][threadIdx.x] + sh[3][threadIdx.x]);
}

// w = A z (FP64 operator, the k_apply expression) and the partial dot
// products of w with V[0..k) (the first Gram-Schmidt projection); 256
// threads per block, grid-stride over cells
template <int K>
__global__ __launch_bounds__(256) void k_apply_multidot(
    const double *__restrict__ z, double *__restrict__ w, const double *__restrict__ a,
    const double *__restrict__ bX, const double *__restrict__ bY,
    const double *__restrict__ cX, const double *__restrict__ cY, int nx, int ny,
    const double *__restrict__ sc, double dxinv, double dyinv,
    const double *__restrict__ V, int k, double *__restrict__ partial)
{
    const int n = nx * ny;
    double    acc[K];
#pragma unroll
    for (int q = 0; q < K; ++q)
        acc[q] = 0;
    for (long long q0 = (long long)blockIdx.x * blockDim.x + threadIdx.x; q0 < n;
         q0 += (long long)gridDim.x * blockDim.x)
    {
        const int    c = (int)q0, j = c / nx, i = c - j * nx;
        const double v = apply_at(z, a, bX, bY, cX, cY, nx, ny, sc[0], sc[1], sc[2], dxinv,
                                  dyinv, i, j);
        w[c] = v;
#pragma unroll
        for (int q = 0; q < K; ++q)
            if (q < k)
                acc[q] += V[(long long)q * n + c] * v;
    }
    block_partials(acc, k, partial);
}

// w -= sum_q h[q] V[q] (q < k, the previous projection's coefficients), then
// the partial dot products of the new w with V[0..k) (second = true) or
// with itself (second = false: its squared norm, one row)
template <int K>
__global__ __launch_bounds__(256) void k_subtract_dots(double *__restrict__ w,
                                                       const double *__restrict__ V,
                                                       const double *__restrict__ h, int k,
                                                       long long n, int second,
                                                       double *__restrict__ partial)
{
    double acc[K];
#pragma unroll
    for (int q = 0; q < K; ++q)
        acc[q] = 0;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
    {
        double vq[K];
        double s = w[i];
#pragma unroll
        for (int q = 0; q < K; ++q)
            if (q < k)
            {
                vq[q] = V[(long long)q * n + i];
                s -= h[q] * vq[q];
            }
        w[i] = s;
        if (second)
        {
#pragma unroll
            for (int q = 0; q < K; ++q)
                if (q < k)
                    acc[q] += vq[q] * s;
        }
        else
            acc[0] += s * s;
    }
    block_partials(acc, second ? k : 1, partial);
}

// FGMRES least-squares state on the device: the Hessenberg matrix H
// ((m+1) x m, row stride m), the Givens rotations (cs, sn), the rotated
// right-hand side g, the solution y of the triangular system, and a status
// word the host reads (est = |g[j+1]|, the new column's norm, and whether y
// came out non-finite).
struct Arnoldi
{
    double *H, *cs, *sn, *g, *y, *status;
    int     m;
};

// g = beta e_0
__global__ void k_arnoldi_init(Arnoldi a, double beta)
{
    if (threadIdx.x == 0 && blockIdx.x == 0)
        for (int i = 0; i <= a.m; ++i)
            a.g[i] = i == 0 ? beta : 0.0;
}

// Column j of H from the two Gram-Schmidt passes (d1 + d2) and the new
// vector's squared norm d3, its previous rotations, a new rotation that
// zeroes H[j+1][j], and g rotated with it: one thread, in the order of a
// textbook Givens update (Saad, Iterative Methods, Alg. 6.9).
__device__ void arnoldi_step(Arnoldi a, const double *__restrict__ d1,
                             const double *__restrict__ d2, const double *__restrict__ d3,
                             int j)
{
    const int m  = a.m;
    double   *H  = a.H;
    for (int i = 0; i <= j; ++i)
        H[i * m + j] = d1[i] + d2[i];
    const double hn    = sqrt(d3[0]);
    H[(j + 1) * m + j] = hn;
    for (int i = 0; i < j; ++i)
    {
        const double t0    = a.cs[i] * H[i * m + j] + a.sn[i] * H[(i + 1) * m + j];
        const double t1    = -a.sn[i] * H[i * m + j] + a.cs[i] * H[(i + 1) * m + j];
        H[i * m + j]       = t0;
        H[(i + 1) * m + j] = t1;
    }
    const double den   = hypot(H[j * m + j], H[(j + 1) * m + j]);
    a.cs[j]            = den > 0 ? H[j * m + j] / den : 1.0;
    a.sn[j]            = den > 0 ? H[(j + 1) * m + j] / den : 0.0;
    H[j * m + j]       = den;
    H[(j + 1) * m + j] = 0;
    a.g[j + 1]         = -a.sn[j] * a.g[j];
    a.g[j]             = a.cs[j] * a.g[j];
    a.status[0]        = fabs(a.g[j + 1]);
    a.status[1]        = hn;
}

// the norm's partials summed by one block, then (thread 0) the Arnoldi step
// and the residual estimate and new column's norm mailed
__global__ __launch_bounds__(256) void k_norm_arnoldi(const double *__restrict__ partial, int nb,
                                                      double *__restrict__ d3, Arnoldi ar,
                                                      const double *__restrict__ d1,
                                                      const double *__restrict__ d2, int j,
                                                      Mail *m, unsigned long long seq)
{
    __shared__ double sh[256];
    const double      s = block_sum_partials(partial, nb, sh);
    if (threadIdx.x == 0)
    {
        d3[0] = s;
        arnoldi_step(ar, d1, d2, d3, j);
        mail_post(m, seq, ar.status[0], ar.status[1]);
    }
}

// y = R^-1 g over the first j columns (back substitution); a non-finite y
// is replaced by zeros (the iterate is kept) and flagged in *bad (pinned host
// memory, read after the next message)
__global__ void k_arnoldi_solve(Arnoldi a, int j, double *bad)
{
    if (threadIdx.x != 0 || blockIdx.x != 0)
        return;
    const int m      = a.m;
    bool      finite = true;
    for (int i = j - 1; i >= 0; --i)
    {
        double t = a.g[i];
        for (int q = i + 1; q < j; ++q)
            t -= a.H[i * m + q] * a.y[q];
        a.y[i] = t / a.H[i * m + i];
        finite = finite && isfinite(a.y[i]);
    }
    if (!finite)
        for (int i = 0; i < j; ++i)
            a.y[i] = 0.0;
    *bad = finite ? 0.0 : 1.0;
    __threadfence_system();
}

// doubles of the least-squares state for restart length up to m_max
static long long arnoldi_doubles(int m_max)
{
    return (long long)(m_max + 1) * m_max + 3LL * m_max + (m_max + 1) + 4;
}
static Arnoldi arnoldi_view(double *buf, int m, int m_max)
{
    Arnoldi a;
    a.m      = m;
    a.H      = buf;
    a.cs     = a.H + (long long)(m_max + 1) * m_max;
    a.sn     = a.cs + m_max;
    a.g      = a.sn + m_max;
    a.y      = a.g + (m_max + 1);
    a.status = a.y + m_max;
    return a;
}

// ------------------------------------------------------------ host class
static dim3 grid2(int nx, int ny, int bs = 256)
{
    return dim3((unsigned)((nx + bs - 1) / bs), (unsigned)ny, 1);
}

template <class T> struct MGLevel
{
    int nx = 0, ny = 0;
    T   hx = 0, hy = 0;       // cell sizes (smoother: beta / h^2)
    T   dxinv = 0, dyinv = 0; // 1 / h (operator apply)
    T  *a = nullptr, *bX = nullptr, *bY = nullptr, *cX = nullptr, *cY = nullptr;
    T  *x = nullptr, *rhs = nullptr, *res = nullptr;
};

template <class T> struct MGHierarchy
{
    std::vector<MGLevel<T>> lev;
    T                       alpha = 0, beta = 0, gamma = 0;
    T                       host_sc[3] = { 0, 0, 0 };
    T                      *d_sc       = nullptr; // (alpha, beta, gamma) on the device
    bool                    with_c     = false;
    int                     tail_l0    = -1;      // first level run by k_vcycle_tail
    int                     tail_lds   = 0;       // its LDS bytes
    TailArgs<T>             tail{};
    int                     nu1 = 2, nu2 = 2, nu_bottom = 16;
    StopCheck               stop; // of the iteration being launched
    // the finest level's coefficient arrays are the solver's own FP64
    // copies (FP64 hierarchy): not freed here
    bool                    alias0 = false;

    void free_all()
    {
        for (size_t l = 0; l < lev.size(); ++l)
        {
            const MGLevel<T> &L = lev[l];
            if (!(l == 0 && alias0))
                for (T *p : { L.a, L.bX, L.bY, L.cX, L.cY })
                    if (p)
                        (void)hipFree(p);
            for (T *p : { L.x, L.rhs, L.res })
                if (p)
                    (void)hipFree(p);
        }
        alias0 = false;
        lev.clear();
        if (d_sc)
            (void)hipFree(d_sc);
        d_sc = nullptr;
        tail_l0 = -1;
    }
};

} // namespace bx

using namespace bx;

struct bx_helm
{
    int    nx = 0, ny = 0;
    double dx = 0, dy = 0;
    long long n = 0;
    bool   has_c = false;
    double alpha = 0, beta = 0, gamma = 0;
    // fine-level FP64 operator (owned copies)
    double *a = nullptr, *bX = nullptr, *bY = nullptr, *cX = nullptr,
           *cY = nullptr;
    MGHierarchy<double> mg64;
    // the FP32 hierarchy of the FGMRES preconditioner, built from the
    // current coefficients when a preconditioner first needs it after
    // bx_helm_set_coeffs (multigrid solves never do)
    MGHierarchy<float>  mg32;
    bool                mg32_stale   = true;
    int                 precond_fp32 = 1;
    // FGMRES workspace (restart length m <= m_max, the allocated basis)
    int     m = 20, m_max = 20;
    double *V = nullptr, *Z = nullptr, *w = nullptr, *r = nullptr,
           *partial = nullptr, *dots = nullptr, *hdev = nullptr;
    int     nb_dot = 512; // blocks (and partials) of a sum over the level
    // the least-squares state (Arnoldi) lives in arn
    double            *arn  = nullptr;
    MailBox mail;
    unsigned long long *stop = nullptr, solve = 0; // StopCheck
    unsigned           *count = nullptr;           // last_block
    // learned smoother
    bx_cnn *cnn       = nullptr;
    double  cnn_omega = 1.0;
    int     cnn_mode  = BX_CNN_SMOOTHER;
    double *tmp1 = nullptr, *tmp2 = nullptr;
    float  *fr = nullptr, *fe = nullptr;
    bool    coeffs_set = false;
    // preconditioner replayed as captured graphs (FGMRES), one per
    // (network attached or not, input vector, output vector): FGMRES applies
    // it to its basis vectors V_j into Z_j, a bounded set, so the graphs
    // read and write those vectors directly; an entry is recaptured when
    // anything it bakes in changes (gen, the network's weights epoch)
    struct PGraph
    {
        int            slot;
        const double  *in;
        double        *out;
        hipGraphExec_t exec;
        long long      gen, epoch;
    };
    int                 use_graph  = 1;
    int                 fused      = 1; // blocked-smoother V-cycle in the FGMRES preconditioner
    hipStream_t         cap_stream = nullptr;
    std::vector<PGraph> pgraphs;
    long long           gen = 0;
};

static thread_local std::string g_helm_err;
static int herr(int code, const std::string &m)
{
    g_helm_err = m;
    return code;
}
#define H_CHECK(expr)                                                           \
    do                                                                          \
    {                                                                           \
        hipError_t e__ = (expr);                                                \
        if (e__ != hipSuccess)                                                  \
            return herr(BX_ERR_HIP, std::string(#expr) + ": "                   \
                                        + hipGetErrorString(e__));              \
    } while (0)

extern "C" const char *bx_helm_last_error(void) { return g_helm_err.c_str(); }

int bx_helm_fail(int code, const std::string &msg) { return herr(code, msg); }

template <class T> static int halloc(T **p, long long n)
{
    H_CHECK(hipMalloc((void **)p, sizeof(T) * std::max<long long>(n, 1)));
    return BX_OK;
}

// src*: the FP64 finest-level coefficients the hierarchy is built from
// (copied into, or converted to, its level 0)
template <class T>
static int build_hierarchy(bx_helm *h, MGHierarchy<T> &mg, hipStream_t s,
                           bool *reallocated, const double *src_a, const double *src_bX,
                           const double *src_bY, const double *src_cX,
                           const double *src_cY)
{
    mg.alpha      = (T)h->alpha;
    mg.beta       = (T)h->beta;
    mg.gamma      = (T)h->gamma;
    mg.host_sc[0] = mg.alpha;
    mg.host_sc[1] = mg.beta;
    mg.host_sc[2] = mg.gamma;
    int rc;
    // the level arrays depend only on the sizes and on whether the gradient
    // term is present: keep them (and every pointer a captured graph holds)
    // when those are unchanged, and refresh the values only
    const bool keep = !mg.lev.empty() && mg.with_c == h->has_c;
    if (!keep)
    {
        *reallocated = true;
        mg.free_all();
        if ((rc = halloc(&mg.d_sc, 3)))
            return rc;
        mg.with_c = h->has_c;
    }
    // the FP64 hierarchy's finest level is the solver's own FP64 copy of the
    // coefficients
    constexpr bool alias = std::is_same<T, double>::value;
    int nx = h->nx, ny = h->ny;
    double dx = h->dx, dy = h->dy;
    while (!keep)
    {
        MGLevel<T> L;
        L.nx    = nx;
        L.ny    = ny;
        L.hx    = (T)dx;
        L.hy    = (T)dy;
        L.dxinv = (T)(1.0 / dx);
        L.dyinv = (T)(1.0 / dy);
        const long long nc = (long long)nx * ny;
        if (alias && mg.lev.empty())
        {
            L.a  = (T *)h->a;
            L.bX = (T *)h->bX;
            L.bY = (T *)h->bY;
            L.cX = h->has_c ? (T *)h->cX : nullptr;
            L.cY = h->has_c ? (T *)h->cY : nullptr;
            mg.alias0 = true;
        }
        else
        {
            if ((rc = halloc(&L.a, nc)) || (rc = halloc(&L.bX, (long long)(nx + 1) * ny))
                || (rc = halloc(&L.bY, (long long)nx * (ny + 1))))
                return rc;
            if (h->has_c && ((rc = halloc(&L.cX, nc)) || (rc = halloc(&L.cY, nc))))
                return rc;
        }
        if ((rc = halloc(&L.x, nc)) || (rc = halloc(&L.rhs, nc)) || (rc = halloc(&L.res, nc)))
            return rc;
        mg.lev.push_back(L);
        // coarsen only to even extents: on a periodic level of odd extent
        // the cells on either side of the seam have the same red/black
        // colour, so one colour pass would update neighbours concurrently
        if (nx % 4 || ny % 4 || nx / 2 < 8 || ny / 2 < 8)
            break;
        nx /= 2;
        ny /= 2;
        dx *= 2;
        dy *= 2;
    }
    if (!keep)
    {
        // the coarsest levels whose arrays fit in LDS run in one launch, the
        // first of them with a quad per thread
        const int nl  = (int)mg.lev.size();
        int       dev = 0, lds_max = 0;
        H_CHECK(hipGetDevice(&dev));
        H_CHECK(hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
        // beside the kernel's static array of level scalars
        const long long tail_bytes = std::min<long long>(lds_max, TAIL_LDS_BYTES)
                                     - TAIL_MAX_LEVELS * 4 * (long long)sizeof(T);
        for (int l0 = nl - 1; l0 >= 0 && nl - l0 <= TAIL_MAX_LEVELS; --l0)
        {
            if ((long long)mg.lev[l0].nx * mg.lev[l0].ny > 4LL * TAIL_THREADS)
                break;
            TailArgs<T> ta{};
            long long   used = 0;
            for (int l = l0; l < nl; ++l)
            {
                const MGLevel<T> &L  = mg.lev[l];
                TailLevel<T>     &tl = ta.lev[l - l0];
                tl.a = L.a; tl.bX = L.bX; tl.bY = L.bY; tl.cX = L.cX; tl.cY = L.cY;
                tl.x = L.x; tl.rhs = L.rhs;
                tl.nx = L.nx; tl.ny = L.ny; tl.hx = L.hx; tl.hy = L.hy;
                tl.dxinv = L.dxinv; tl.dyinv = L.dyinv;
                used = tail_place(tl, l == l0, used);
            }
            if (used * (long long)sizeof(T) > tail_bytes)
                break;
            mg.tail     = ta;
            mg.tail_l0  = l0;
            mg.tail_lds = (int)(used * sizeof(T));
        }
    }
    // level 0 and the scalars in one launch, then one averaging launch per
    // large coarse level and one for all the small ones (the set-up is
    // bound by launches, not bytes)
    MGLevel<T> &L0 = mg.lev[0];
    const bool  c  = h->has_c;
    hipLaunchKernelGGL((k_convert_coeffs<T>), dim3(1024), dim3(256), 0, s, src_a, src_bX,
                       src_bY, c ? src_cX : nullptr, c ? src_cY : nullptr, L0.a, L0.bX, L0.bY,
                       L0.cX, L0.cY, h->nx, h->ny, mg.d_sc, mg.alpha, mg.beta, mg.gamma);
    CoarsenList<T> small{};
    for (size_t l = 1; l < mg.lev.size(); ++l)
    {
        MGLevel<T> &F = mg.lev[l - 1], &C = mg.lev[l];
        if ((long long)C.nx * C.ny <= COARSEN_SMALL && small.n < COARSEN_MAX_LEVELS)
        {
            small.lev[small.n++] = { F.a,  F.bX, F.bY, c ? F.cX : nullptr, c ? F.cY : nullptr,
                                     C.a,  C.bX, C.bY, C.cX, C.cY, C.nx, C.ny };
            continue;
        }
        if (small.n) // levels coarsen in order: flush before a large one
        {
            hipLaunchKernelGGL((k_coarsen_small<T>), dim3(1), dim3(1024), 0, s, small);
            small.n = 0;
        }
        hipLaunchKernelGGL((k_coarsen_coeffs<T>), grid2(C.nx + 1, C.ny + 1), dim3(256), 0, s,
                           F.a, F.bX, F.bY, c ? F.cX : nullptr, c ? F.cY : nullptr, C.a, C.bX,
                           C.bY, C.cX, C.cY, C.nx, C.ny);
    }
    if (small.n)
        hipLaunchKernelGGL((k_coarsen_small<T>), dim3(1), dim3(1024), 0, s, small);
    H_CHECK(hipGetLastError());
    return BX_OK;
}

template <class T>
static void launch_apply(const MGLevel<T> &L, const MGHierarchy<T> &mg,
                         const T *x, T *y, const T *rhs, hipStream_t s)
{
    hipLaunchKernelGGL((k_apply<T>), grid2(L.nx, L.ny), dim3(256), 0, s, x, y,
                       L.a, L.bX, L.bY, L.cX, L.cY, L.nx, L.ny, mg.d_sc, L.dxinv,
                       L.dyinv, rhs);
}

template <class T>
static void launch_smooth(const MGLevel<T> &L, const MGHierarchy<T> &mg,
                          T *phi, const T *rhs, int redblack, hipStream_t s)
{
    hipLaunchKernelGGL((k_gsrb<T>), grid2((L.nx + 1) / 2, L.ny), dim3(256), 0,
                       s, phi, rhs, L.a, L.bX, L.bY, L.cX, L.cY, L.nx, L.ny,
                       mg.d_sc, L.hx, L.hy, redblack);
}

template <class T, int TX, int TY, int PM, int RES>
static void launch_quad_tiles(const SmoothArgs<T> &A, hipStream_t s)
{
    const dim3 grid((unsigned)((A.nx + TX - 1) / TX), (unsigned)((A.ny + TY - 1) / TY));
    const dim3 block(quad_threads(TX, TY, PM, RES));
    if (A.cX)
        hipLaunchKernelGGL((k_gsrb_quads<T, TX, TY, PM, RES, true>), grid, block, 0, s, A);
    else
        hipLaunchKernelGGL((k_gsrb_quads<T, TX, TY, PM, RES, false>), grid, block, 0, s, A);
}

// A.pairs (1..4; 1..3 with A.crhs; on a bottom level 1..8) blocked red/black
// pairs on level L.  Tiles:
// 64 x 16, or 32 x 8 when the level has fewer 64 x 16 tiles than an MI355X
// has CUs (256): a small level is bound by latency, and more, shorter
// workgroups end sooner.  Two pairs with the restriction, FP64: 64 x 16 tiles on
// 1024^2 and 512^2 13.6 us a launch on average, without it 10.4 (a thread per
// cell: 16.8); 32 x 8 tiles on 256^2 and 128^2 4.6 (6.3).
template <class T, int TX, int TY> static void launch_quad_pairs(const SmoothArgs<T> &A, hipStream_t s)
{
    if (A.r_out)
    {
        if constexpr (std::is_same_v<T, double> && TX == 32)
            launch_quad_tiles<T, TX, TY, 2, SM_RESIDUAL>(A, s);
    }
    else if (A.crhs)
    {
        if (A.pairs <= 2)
            launch_quad_tiles<T, TX, TY, 2, SM_RESTRICT>(A, s);
        else
            launch_quad_tiles<T, TX, TY, 3, SM_RESTRICT>(A, s);
    }
    else if (A.pairs <= 2)
        launch_quad_tiles<T, TX, TY, 2, SM_PLAIN>(A, s);
    else if (A.pairs <= 4)
        launch_quad_tiles<T, TX, TY, 4, SM_PLAIN>(A, s);
    else if constexpr (TX == 32)
        launch_quad_tiles<T, 16, 8, 8, SM_PLAIN>(A, s);
}
constexpr int SM_MAXP = 4; // most pairs of one launch (3 with the restriction)
// and on a bottom level outside the tail: 8, in tiles of 16 x 8, where each has
// a CU to itself.  The halo makes that 7.5 times the tile's work, but latency
// bounds the launch: 16 pairs of 150 x 110, FP64, take 15.7 us in two launches
// (17.7 in tiles of 32 x 8) and took 20.6 in four of 4 pairs.
template <class T> static int bottom_pairs(const MGLevel<T> &L)
{
    const long long tiles = (long long)((L.nx + 15) / 16) * ((L.ny + 7) / 8);
    return tiles <= 256 ? 8 : SM_MAXP;
}

template <class T>
static SmoothArgs<T> smooth_args(const MGLevel<T> &L, const MGHierarchy<T> &mg, const T *in,
                                 T *out, int pairs)
{
    SmoothArgs<T> A{};
    A.phi = in; A.phi_out = out; A.rhs = L.rhs;
    A.a = L.a; A.bX = L.bX; A.bY = L.bY; A.cX = L.cX; A.cY = L.cY;
    A.nx = L.nx; A.ny = L.ny; A.sc = mg.d_sc;
    A.hx = L.hx; A.hy = L.hy; A.dxinv = L.dxinv; A.dyinv = L.dyinv;
    A.pairs = pairs;
    A.stop  = mg.stop;
    return A;
}

static bool large_tiles(int nx, int ny)
{
    return (long long)((nx + 63) / 64) * ((ny + 15) / 16) >= 256;
}
template <class T> static void launch_quads(const SmoothArgs<T> &A, hipStream_t s)
{
    if (large_tiles(A.nx, A.ny))
        launch_quad_pairs<T, 64, 16>(A, s);
    else
        launch_quad_pairs<T, 32, 8>(A, s);
}

// Level l takes the blocked path of vcycle().
template <class T>
static bool blocked_level(const MGHierarchy<T> &mg, int l, bool fused)
{
    const bool tail   = mg.tail_l0 >= 0 && l == mg.tail_l0;
    const bool bottom = l + 1 == (int)mg.lev.size();
    return !tail && !bottom && fused && mg.nu2 > 0 && mg.nu1 <= SM_MAXP && mg.nu2 <= SM_MAXP;
}

// Level l's blocked path also restricts the residual in its pre-smoothing
// launch, so no other launch reads the level's right-hand side array.
template <class T>
static bool direct_io_level(const MGHierarchy<T> &mg, int l, bool fused)
{
    return blocked_level(mg, l, fused) && mg.nu1 > 0 && mg.nu1 < SM_MAXP;
}

// One V-cycle from level l, from a zero guess on it (L.x need not be zeroed:
// a path that reads it zeroes it first).  acc (level 0 only): when the
// blocked path runs, its last smoothing adds the correction to acc (acc += e,
// as k_axpy) instead of storing it, and the call returns true; otherwise the
// correction is in mg.lev[l].x and the call returns false.  rhs_in / out64
// (only where direct_io_level holds): level l's right-hand side is read from
// rhs_in (FP64) and the correction written to out64 (FP64) by the smoothing
// launches themselves.
// end (level 0, with acc; see solve_mg): the last smoothing forms
// acc = end->x + e, the residual and its norm's message (SM_RESIDUAL).
template <class T> struct CycleEnd
{
    const T *x, *b;
    T       *r_out;
    double  *partial;
    NormMail nm;
};
template <class T>
static bool vcycle(MGHierarchy<T> &mg, int l, hipStream_t s, bool fused = false,
                   T *acc = nullptr, const double *rhs_in = nullptr, double *out64 = nullptr,
                   const CycleEnd<T> *end = nullptr)
{
    MGLevel<T> &L       = mg.lev[l];
    const bool  tail    = mg.tail_l0 >= 0 && l == mg.tail_l0;
    const bool  bottom  = l + 1 == (int)mg.lev.size();
    const bool  blocked = blocked_level(mg, l, fused);
    if (tail)
    {
        const int nl = (int)mg.lev.size() - l;
        if (mg.with_c)
            hipLaunchKernelGGL((k_vcycle_tail<T, true>), dim3(1), dim3(TAIL_THREADS),
                               mg.tail_lds, s, mg.tail, nl, mg.nu1, mg.nu2, mg.nu_bottom,
                               mg.d_sc, mg.stop);
        else
            hipLaunchKernelGGL((k_vcycle_tail<T, false>), dim3(1), dim3(TAIL_THREADS),
                               mg.tail_lds, s, mg.tail, nl, mg.nu1, mg.nu2, mg.nu_bottom,
                               mg.d_sc, mg.stop);
        return false;
    }
    if (bottom)
    {
        // a bottom level too large for the tail: its sweeps in blocked
        // launches, ending in L.x
        const int most = bottom_pairs(L);
        int       left = mg.nu_bottom;
        for (int k = (left + most - 1) / most; k > 0; --k)
        {
            T *const      out   = k % 2 ? L.x : L.res;
            const int     pairs = std::min(left, most);
            SmoothArgs<T> A     = smooth_args(L, mg, k % 2 ? L.res : L.x, out, pairs);
            A.zero_in           = left == mg.nu_bottom;
            launch_quads(A, s);
            left -= pairs;
        }
        return false;
    }
    if (!(blocked && mg.nu1 > 0))
        hipLaunchKernelGGL((k_fill<T>), dim3(2048), dim3(256), 0, s, L.x,
                           (long long)L.nx * L.ny, (T)0);
    MGLevel<T> &C = mg.lev[l + 1];
    if (blocked)
    {
        // two launches per level: blocked pre-smoothing with the residual's
        // restriction, prolongation + blocked post-smoothing.
        // pre-smoothing 0 -> res, post-smoothing res + P e_c -> x (the res
        // array is free in this path: the residual goes straight to C.rhs)
        const T *xs = L.x;
        if (mg.nu1 > 0)
        {
            SmoothArgs<T> A = smooth_args(L, mg, (const T *)L.x, L.res, mg.nu1);
            A.zero_in       = 1;
            A.rhs_in        = rhs_in;
            if (mg.nu1 < SM_MAXP)
                A.crhs = C.rhs;
            launch_quads(A, s);
            xs = L.res;
        }
        if (!(mg.nu1 > 0 && mg.nu1 < SM_MAXP))
            hipLaunchKernelGGL((k_resid_restrict<T>), grid2(C.nx, C.ny), dim3(256), 0, s, xs,
                               L.rhs, L.a, L.bX, L.bY, L.cX, L.cY, L.nx, L.ny, mg.d_sc,
                               L.dxinv, L.dyinv, C.rhs);
        vcycle(mg, l + 1, s, fused);
        SmoothArgs<T> A = smooth_args(L, mg, xs, acc ? acc : L.x, mg.nu2);
        A.coarse        = C.x;
        A.rhs_in        = rhs_in;
        A.accumulate    = acc != nullptr;
        A.out64         = acc ? nullptr : out64;
        if (xs == A.phi_out) // nu1 == 0: the iterate is still zero
        {
            // in and out must differ: smooth 0 + P e_c from the res array
            hipLaunchKernelGGL((k_fill<T>), dim3(2048), dim3(256), 0, s, L.res,
                               (long long)L.nx * L.ny, (T)0);
            A.phi = L.res;
        }
        if (end)
        {
            A.x_in    = end->x;
            A.b       = end->b;
            A.r_out   = end->r_out;
            A.partial = end->partial;
            A.nm      = end->nm;
        }
        launch_quads(A, s);
        return acc != nullptr;
    }
    for (int it = 0; it < mg.nu1; ++it)
    {
        launch_smooth(L, mg, L.x, L.rhs, 0, s);
        launch_smooth(L, mg, L.x, L.rhs, 1, s);
    }
    launch_apply(L, mg, L.x, L.res, L.rhs, s);
    hipLaunchKernelGGL((k_restrict<T>), grid2(C.nx, C.ny), dim3(256), 0, s,
                       L.res, C.rhs, C.nx, C.ny);
    vcycle(mg, l + 1, s, fused);
    hipLaunchKernelGGL((k_prolong_add<T>), grid2(L.nx, L.ny), dim3(256), 0, s,
                       C.x, L.x, L.nx, L.ny);
    for (int it = 0; it < mg.nu2; ++it)
    {
        launch_smooth(L, mg, L.x, L.rhs, 0, s);
        launch_smooth(L, mg, L.x, L.rhs, 1, s);
    }
    return false;
}

// coarse-grid part of the V-cycle only (levels >= 1), from L.res on level 0
template <class T>
static void coarse_correction(MGHierarchy<T> &mg, hipStream_t s, bool fused)
{
    MGLevel<T> &L = mg.lev[0];
    MGLevel<T> &C = mg.lev[1];
    hipLaunchKernelGGL((k_restrict<T>), grid2(C.nx, C.ny), dim3(256), 0, s,
                       L.res, C.rhs, C.nx, C.ny);
    vcycle(mg, 1, s, fused);
    hipLaunchKernelGGL((k_prolong_add<T>), grid2(L.nx, L.ny), dim3(256), 0, s,
                       C.x, L.x, L.nx, L.ny);
}

// r = b - A x at FP64
static void residual64(bx_helm *h, const double *b, const double *x, double *r,
                       hipStream_t s)
{
    launch_apply(h->mg64.lev[0], h->mg64, x, r, b, s);
}

// r = b - A x and its squared norm in the next message (v[0]), with bn also
// that of b (v[1]).  sc, tol: the solve's end (StopCheck).
static void launch_residual_norms(bx_helm *h, const double *b, const double *x, double *r,
                                  bool bn, const StopCheck &sc, double tol, hipStream_t s)
{
    const MGLevel<double> &L = h->mg64.lev[0];
    const dim3             g(h->nb_dot), t(256);
    const NormMail         nm{ h->count, h->mail.dev, ++h->mail.seq, tol };
    if (bn)
        hipLaunchKernelGGL(k_residual_sumsq<true>, g, t, 0, s, x, r, b, L.a, L.bX, L.bY, L.cX,
                           L.cY, L.nx, L.ny, h->mg64.d_sc, L.dxinv, L.dyinv, h->partial, sc, nm);
    else
        hipLaunchKernelGGL(k_residual_sumsq<false>, g, t, 0, s, x, r, b, L.a, L.bX, L.bY, L.cX,
                           L.cY, L.nx, L.ny, h->mg64.d_sc, L.dxinv, L.dyinv, h->partial, sc, nm);
}

// the same, waited for
static int residual_norms(bx_helm *h, const double *b, const double *x, double *r,
                          hipStream_t s, double *rnorm, double *bnorm)
{
    launch_residual_norms(h, b, x, r, bnorm != nullptr, StopCheck(), 0.0, s);
    H_CHECK(h->mail.wait(h->mail.seq, s));
    *rnorm = std::sqrt(h->mail[h->mail.seq].v[0]);
    if (bnorm)
        *bnorm = std::sqrt(h->mail[h->mail.seq].v[1]);
    return BX_OK;
}

// ------------------------------------------------------------- C ABI
extern "C" int bx_helm_create(int nx, int ny, double dx, double dy,
                              int periodic, bx_helm **out)
{
    if (!out || nx < 8 || ny < 8 || !(dx > 0) || !(dy > 0))
        return herr(BX_ERR_INVALID, "bx_helm_create: bad argument");
    if (!periodic)
        return herr(BX_ERR_UNSUPPORTED,
                    "bx_helm_create: only periodic levels are implemented");
    // red/black Gauss-Seidel on a periodic level needs even extents (an odd
    // extent makes the two cells across the seam the same colour)
    if (nx % 2 || ny % 2)
        return herr(BX_ERR_UNSUPPORTED, "bx_helm_create: nx and ny must be even");
    if ((long long)nx * ny > 2147483647LL)
        return herr(BX_ERR_UNSUPPORTED, "bx_helm_create: more than 2^31 - 1 cells");
    bx_helm *h = new bx_helm();
    h->nx = nx;
    h->ny = ny;
    h->dx = dx;
    h->dy = dy;
    h->n  = (long long)nx * ny;
    // one cell per thread until the chip is full (8 blocks per CU)
    h->nb_dot = (int)std::min<long long>((h->n + 255) / 256, 2048);
    // a partial per tile of the smoothing (SM_RESIDUAL), whichever its size
    const long long tiles = (long long)((nx + 31) / 32) * ((ny + 7) / 8);
    int rc;
    if ((rc = halloc(&h->a, h->n)) || (rc = halloc(&h->bX, (long long)(nx + 1) * ny))
        || (rc = halloc(&h->bY, (long long)nx * (ny + 1)))
        || (rc = halloc(&h->V, h->n * (h->m_max + 1))) || (rc = halloc(&h->Z, h->n * h->m_max))
        || (rc = halloc(&h->w, h->n)) || (rc = halloc(&h->r, h->n))
        || (rc = halloc(&h->tmp1, h->n)) || (rc = halloc(&h->tmp2, h->n))
        || (rc = halloc(&h->fr, h->n)) || (rc = halloc(&h->fe, h->n))
        || (rc = halloc(&h->partial, std::max((long long)h->nb_dot * (h->m_max + 1), tiles)))
        || (rc = halloc(&h->dots, 2 * (h->m_max + 1) + 3))
        || (rc = halloc(&h->count, (COUNT_GROUPS + 1) * COUNT_LINE)) || (rc = halloc(&h->hdev, h->m_max + 1))
        || (rc = halloc(&h->arn, arnoldi_doubles(h->m_max))))
    {
        bx_helm_destroy(h);
        return rc;
    }
    // the last word of the scalars
    h->stop = (unsigned long long *)(h->dots + 2 * (h->m_max + 1) + 2);
    const size_t counts = (COUNT_GROUPS + 1) * COUNT_LINE * sizeof(*h->count);
    if (hipMemset(h->stop, 0, sizeof(*h->stop)) != hipSuccess
        || hipMemset(h->count, 0, counts) != hipSuccess
        || hipStreamSynchronize(nullptr) != hipSuccess || h->mail.open() != hipSuccess)
    {
        bx_helm_destroy(h);
        return herr(BX_ERR_HIP, "bx_helm_create: allocation failed");
    }
    *out = h;
    return BX_OK;
}

extern "C" void bx_helm_destroy(bx_helm *h)
{
    if (!h)
        return;
    h->mg64.free_all();
    h->mg32.free_all();
    for (const auto &pg : h->pgraphs)
        if (pg.exec)
            (void)hipGraphExecDestroy(pg.exec);
    if (h->cap_stream)
        (void)hipStreamDestroy(h->cap_stream);
    for (void *p : { (void *)h->a, (void *)h->bX, (void *)h->bY, (void *)h->cX,
                     (void *)h->cY, (void *)h->V, (void *)h->Z, (void *)h->w,
                     (void *)h->r, (void *)h->partial, (void *)h->dots,
                     (void *)h->hdev, (void *)h->tmp1, (void *)h->tmp2,
                     (void *)h->fr, (void *)h->fe,
                     (void *)h->arn, (void *)h->count })
        if (p)
            (void)hipFree(p);
    h->mail.close(); // hipFree above has waited for the device
    delete h;
}

extern "C" int bx_helm_set_coeffs(bx_helm *h, double alpha, double beta,
                                  double gamma, const double *a,
                                  const double *bXf, const double *bYf,
                                  const double *cX, const double *cY,
                                  void *stream)
{
    if (!h || !a || !bXf || !bYf || ((cX == nullptr) != (cY == nullptr)))
        return herr(BX_ERR_INVALID, "bx_helm_set_coeffs: bad argument");
    hipStream_t s = (hipStream_t)stream;
    h->alpha = alpha;
    h->beta  = beta;
    h->gamma = gamma;
    h->has_c = cX != nullptr && gamma != 0.0;
    int rc;
    if (h->has_c && !h->cX && ((rc = halloc(&h->cX, h->n)) || (rc = halloc(&h->cY, h->n))))
        return rc;
    // the FP64 hierarchy's level 0 is the solver's copy (h->a, ...): its
    // level-0 launch copies the caller's arrays there
    bool realloc = false;
    if ((rc = build_hierarchy(h, h->mg64, s, &realloc, a, bXf, bYf, cX, cY)))
        return rc;
    if (realloc)
        ++h->gen;
    h->mg32_stale = true;
    H_CHECK(hipStreamSynchronize(s));
    h->coeffs_set = true;
    return BX_OK;
}

// Builds the FP32 hierarchy if a preconditioner will read it and it is
// older than the coefficients.  Never called inside a graph capture.
static int ensure_mg32(bx_helm *h, hipStream_t s)
{
    if (!h->mg32_stale || !h->precond_fp32)
        return BX_OK;
    bool realloc = false;
    int  rc;
    if ((rc = build_hierarchy(h, h->mg32, s, &realloc, h->a, h->bX, h->bY, h->cX, h->cY)))
        return rc;
    if (realloc)
        ++h->gen;
    h->mg32_stale = false;
    return BX_OK;
}

extern "C" int bx_helm_set_options(bx_helm *h, int nu1, int nu2, int nu_bottom,
                                   int precond_fp32, int restart)
{
    if (!h || nu1 < 0 || nu2 < 0 || nu_bottom < 1 || restart < 1 || restart > h->m_max)
        return herr(BX_ERR_INVALID, "bx_helm_set_options: bad argument");
    for (auto *mg : { &h->mg64 })
    {
        mg->nu1       = nu1;
        mg->nu2       = nu2;
        mg->nu_bottom = nu_bottom;
    }
    h->mg32.nu1       = nu1;
    h->mg32.nu2       = nu2;
    h->mg32.nu_bottom = nu_bottom;
    h->precond_fp32   = precond_fp32;
    h->m              = restart;
    ++h->gen;
    return BX_OK;
}

extern "C" int bx_helm_set_fused(bx_helm *h, int fused)
{
    if (!h)
        return herr(BX_ERR_INVALID, "bx_helm_set_fused: null solver");
    h->fused = fused ? 1 : 0;
    ++h->gen;
    return BX_OK;
}

extern "C" int bx_helm_set_graph(bx_helm *h, int use_graph)
{
    if (!h)
        return herr(BX_ERR_INVALID, "bx_helm_set_graph: null solver");
    h->use_graph = use_graph ? 1 : 0;
    return BX_OK;
}

extern "C" int bx_helm_apply(bx_helm *h, const double *x, double *y,
                             void *stream)
{
    if (!h || !h->coeffs_set || !x || !y)
        return herr(BX_ERR_STATE, "bx_helm_apply: coefficients not set");
    launch_apply(h->mg64.lev[0], h->mg64, x, y, (const double *)nullptr,
                 (hipStream_t)stream);
    H_CHECK(hipGetLastError());
    return BX_OK;
}

extern "C" int bx_helm_residual(bx_helm *h, const double *b, const double *x,
                                double *r, void *stream)
{
    if (!h || !h->coeffs_set || !b || !x || !r)
        return herr(BX_ERR_STATE, "bx_helm_residual: coefficients not set");
    residual64(h, b, x, r, (hipStream_t)stream);
    H_CHECK(hipGetLastError());
    return BX_OK;
}

extern "C" int bx_helm_smooth(bx_helm *h, double *phi, const double *rhs,
                              int redblack, void *stream)
{
    if (!h || !h->coeffs_set || !phi || !rhs)
        return herr(BX_ERR_STATE, "bx_helm_smooth: coefficients not set");
    launch_smooth(h->mg64.lev[0], h->mg64, phi, rhs, redblack & 1,
                  (hipStream_t)stream);
    H_CHECK(hipGetLastError());
    return BX_OK;
}

// e = M r : one V-cycle from a zero guess (FP32 or FP64), optionally with the
// learned correction as fine-level smoother:
//   e  = omega * CNN(r)                 (learned pre-smoothing)
//   e += P Vcycle_coarse(R (r - A e))
//   e += omega * CNN(r - A e)           (learned post-smoothing)
static int precond_vcycle(bx_helm *h, const double *rv, double *e, hipStream_t s);

static int precond(bx_helm *h, const double *rv, double *e, hipStream_t s)
{
    const long long n = h->n;
    if (h->cnn && h->cnn_mode == BX_CNN_CORRECTOR)
    {
        // e = V(r); e += omega * CNN(r - A e)
        int rc;
        if ((rc = precond_vcycle(h, rv, e, s)))
            return rc;
        residual64(h, rv, e, h->tmp1, s);
        if ((rc = bx_cnn_forward(h->cnn, h->tmp1, h->tmp2, h->nx, h->ny,
                                 h->cnn_omega, s)))
            return rc;
        hipLaunchKernelGGL(k_axpy, dim3(2048), dim3(256), 0, s, e, h->tmp2, n, 1.0);
        H_CHECK(hipGetLastError());
        return BX_OK;
    }
    if (h->cnn)
    {
        int rc;
        // pre: e = omega*CNN(r)
        if ((rc = bx_cnn_forward(h->cnn, rv, e, h->nx, h->ny, h->cnn_omega, s)))
            return rc;
        // residual r1 = r - A e (FP64), coarse correction in FP32 or FP64
        residual64(h, rv, e, h->tmp1, s);
        if (h->mg64.lev.size() < 2)
        {
            // single-level hierarchy: no coarse correction
        }
        else if (h->precond_fp32)
        {
            MGHierarchy<float> &mg = h->mg32;
            hipLaunchKernelGGL((k_convert<float, double>), dim3(2048), dim3(256), 0,
                               s, h->tmp1, mg.lev[0].res, n, 1.0);
            hipLaunchKernelGGL((k_fill<float>), dim3(2048), dim3(256), 0, s,
                               mg.lev[0].x, n, 0.f);
            coarse_correction(mg, s, h->fused);
            hipLaunchKernelGGL((k_convert<double, float>), dim3(2048), dim3(256), 0,
                               s, mg.lev[0].x, h->tmp2, n, 1.0f);
        }
        else
        {
            MGHierarchy<double> &mg = h->mg64;
            hipLaunchKernelGGL((k_scale), dim3(2048), dim3(256), 0, s,
                               mg.lev[0].res, h->tmp1, n, 1.0);
            hipLaunchKernelGGL((k_fill<double>), dim3(2048), dim3(256), 0, s,
                               mg.lev[0].x, n, 0.0);
            coarse_correction(mg, s, h->fused);
            hipLaunchKernelGGL((k_scale), dim3(2048), dim3(256), 0, s, h->tmp2,
                               mg.lev[0].x, n, 1.0);
        }
        if (h->mg64.lev.size() >= 2)
            hipLaunchKernelGGL(k_axpy, dim3(2048), dim3(256), 0, s, e, h->tmp2, n,
                               1.0);
        // post: e += omega*CNN(r - A e)
        residual64(h, rv, e, h->tmp1, s);
        if ((rc = bx_cnn_forward(h->cnn, h->tmp1, h->tmp2, h->nx, h->ny,
                                 h->cnn_omega, s)))
            return rc;
        hipLaunchKernelGGL(k_axpy, dim3(2048), dim3(256), 0, s, e, h->tmp2, n, 1.0);
        H_CHECK(hipGetLastError());
        return BX_OK;
    }
    return precond_vcycle(h, rv, e, s);
}

// e = one V-cycle on r from a zero guess, FP32 or FP64 hierarchy
static int precond_vcycle(bx_helm *h, const double *rv, double *e, hipStream_t s)
{
    const long long n = h->n;
    // where the finest level's smoothing launches can read r and write e
    // themselves, no conversion launches
    if (h->precond_fp32)
    {
        MGHierarchy<float> &mg = h->mg32;
        if (direct_io_level(mg, 0, h->fused != 0))
            vcycle(mg, 0, s, true, (float *)nullptr, rv, e);
        else
        {
            hipLaunchKernelGGL((k_convert<float, double>), dim3(2048), dim3(256), 0, s,
                               rv, mg.lev[0].rhs, n, 1.0);
            vcycle(mg, 0, s, h->fused != 0);
            hipLaunchKernelGGL((k_convert<double, float>), dim3(2048), dim3(256), 0, s,
                               mg.lev[0].x, e, n, 1.0f);
        }
    }
    else
    {
        MGHierarchy<double> &mg = h->mg64;
        if (direct_io_level(mg, 0, h->fused != 0))
            vcycle(mg, 0, s, true, (double *)nullptr, rv, e);
        else
        {
            hipLaunchKernelGGL((k_scale), dim3(2048), dim3(256), 0, s, mg.lev[0].rhs,
                               rv, n, 1.0);
            vcycle(mg, 0, s, h->fused != 0);
            hipLaunchKernelGGL((k_scale), dim3(2048), dim3(256), 0, s, e,
                               mg.lev[0].x, n, 1.0);
        }
    }
    H_CHECK(hipGetLastError());
    return BX_OK;
}

extern "C" int bx_helm_precond(bx_helm *h, const double *r, double *e,
                               void *stream)
{
    if (!h || !h->coeffs_set || !r || !e)
        return herr(BX_ERR_STATE, "bx_helm_precond: coefficients not set");
    int rc;
    if ((rc = ensure_mg32(h, (hipStream_t)stream)))
        return rc;
    return precond(h, r, e, (hipStream_t)stream);
}

extern "C" int bx_helm_attach_cnn(bx_helm *h, bx_cnn *cnn, double omega, int mode)
{
    if (!h || (mode != BX_CNN_SMOOTHER && mode != BX_CNN_CORRECTOR))
        return herr(BX_ERR_INVALID, "bx_helm_attach_cnn: bad argument");
    h->cnn       = cnn;
    h->cnn_omega = omega;
    h->cnn_mode  = mode;
    ++h->gen;
    return BX_OK;
}

// e = M r through the captured graph for (r, e)
static int precond_replay(bx_helm *h, const double *rv, double *e, hipStream_t s)
{
    if (!h->use_graph)
        return precond(h, rv, e, s);
    const int       slot  = h->cnn ? 1 : 0;
    const long long epoch = h->cnn ? bx_cnn_epoch(h->cnn) : 0;
    bx_helm::PGraph *pg   = nullptr;
    for (auto &q : h->pgraphs)
        if (q.slot == slot && q.in == rv && q.out == e)
            pg = &q;
    if (!pg)
    {
        h->pgraphs.push_back({ slot, rv, e, nullptr, -1, -1 });
        pg = &h->pgraphs.back();
    }
    if (!pg->exec || pg->gen != h->gen || pg->epoch != epoch)
    {
        if (pg->exec)
        {
            H_CHECK(hipGraphExecDestroy(pg->exec));
            pg->exec = nullptr;
        }
        if (!h->cap_stream)
            H_CHECK(hipStreamCreateWithFlags(&h->cap_stream, hipStreamNonBlocking));
        // everything the capture touches must be allocated beforehand
        if (h->cnn)
        {
            int rc = bx_cnn_reserve(h->cnn, h->n);
            if (rc)
                return rc;
        }
        H_CHECK(hipStreamSynchronize(s));
        hipGraph_t g = nullptr;
        H_CHECK(hipStreamBeginCapture(h->cap_stream, hipStreamCaptureModeThreadLocal));
        int rc = precond(h, rv, e, h->cap_stream);
        hipError_t ec = hipStreamEndCapture(h->cap_stream, &g);
        if (rc)
        {
            if (g)
                (void)hipGraphDestroy(g);
            return rc;
        }
        if (ec != hipSuccess)
            return herr(BX_ERR_HIP, std::string("precond capture: ") + hipGetErrorString(ec));
        ec = hipGraphInstantiate(&pg->exec, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        if (ec != hipSuccess)
        {
            pg->exec = nullptr;
            return herr(BX_ERR_HIP, std::string("precond instantiate: ") + hipGetErrorString(ec));
        }
        pg->gen   = h->gen;
        pg->epoch = epoch;
    }
    H_CHECK(hipGraphLaunch(pg->exec, s));
    return BX_OK;
}

// Multigrid iteration k (from 0) of a solve on the device: x += V(r) with r in
// the finest level's right-hand side, then the new residual there and its
// squared norm in the next message.  With `ends` one launch does
// what follows the V-cycle's last smoothing; the residual and x then alternate
// between two arrays each.
static void mg_iteration(bx_helm *h, const double *b, double *x, bool fused, const StopCheck &sc,
                         double tol, hipStream_t s, bool ends, int k)
{
    MGHierarchy<double> &mg = h->mg64;
    mg.stop                 = sc;
    if (ends)
    {
        double *const r = mg.lev[0].rhs, *const xs[2] = { x, h->w }, *const rs[2] = { r, h->r };
        const CycleEnd<double> e{ xs[k % 2], b, rs[(k + 1) % 2], h->partial,
                                  NormMail{ h->count, h->mail.dev, ++h->mail.seq, tol } };
        mg.lev[0].rhs = rs[k % 2];
        vcycle(mg, 0, s, fused, xs[(k + 1) % 2], nullptr, nullptr, &e);
        mg.lev[0].rhs = r;
        mg.stop       = StopCheck();
        return;
    }
    if (!vcycle(mg, 0, s, fused, x))
        hipLaunchKernelGGL(k_axpy, dim3(2048), dim3(256), 0, s, x, mg.lev[0].x, h->n, 1.0);
    mg.stop = StopCheck();
    launch_residual_norms(h, b, x, mg.lev[0].rhs, false, sc, tol, s);
}

// Every kernel of an iteration can be told to end at once: the blocked path
// from the finest level to the tail or the bottom (and the finest level is
// neither, so that its last smoothing adds to x).
static bool can_run_ahead(const bx_helm *h, bool fused)
{
    const MGHierarchy<double> &mg = h->mg64;
    const int nb = mg.tail_l0 >= 0 ? mg.tail_l0 : (int)mg.lev.size() - 1;
    for (int l = 0; l < nb; ++l)
        if (!direct_io_level(mg, l, fused))
            return false;
    return nb > 0;
}

// Plain multigrid solve (MLMG::solve semantics, FP64): x <- x + V(b - A x)
// until ||b - A x||_2 <= rtol ||b||_2.  The iterations are launched kernel by
// kernel: at 1024^2 the GPU is the bottleneck, and a captured iteration
// (which needs copies of b and x into fixed buffers) measured slower.  The
// residual lives in the finest level's right-hand side.  Where the path
// allows it (can_run_ahead) the next iteration is launched before the host
// has read the last one's norm, so the GPU does not wait for the host; only
// while the convergence so far says that it will be needed, since the
// kernels launched past the end cost about as much as two such waits.
// 160 x 96, 14 iterations: 902 -> 823 us a step.
// rn >= 0: the right-hand side already holds b - A x, of norm rn.
static int solve_mg(bx_helm *h, const double *b, double *x, double rtol,
                    int maxiter, double bnorm, bx_solve_stats *st,
                    hipStream_t s, bool fused = false, double rn = -1)
{
    const double tol = rtol * bnorm;
    int          rc;
    if (rn < 0 && (rc = residual_norms(h, b, x, h->mg64.lev[0].rhs, s, &rn, nullptr)))
        return rc;
    const bool ahead = can_run_ahead(h, fused);
    // SM_RESIDUAL smooths two pairs, in small tiles.  160 x 96: 8.2 us for 4.7 +
    // 6.3; in large ones its wider halo costs what the launch saves (600 x 440
    // 18.5 us for 8.7 + 10.3, 1024^2 33.7 for 16.2 + 15.8)
    const bool ends = ahead && h->mg64.nu2 <= 2 && !large_tiles(h->nx, h->ny);
    StopCheck  sc;
    if (ahead)
        sc = StopCheck{ h->stop, ++h->solve };
    double rate = 0.02; // of one iteration, until one has been seen
    const unsigned long long first = h->mail.seq; // message first + it: iteration it
    int                      it = 0, launched = 0;
    bool                     go = rn > tol;
    while (go && it < maxiter)
    {
        ++it;
        const int want = ahead && rn * rate > tol ? it + 1 : it;
        for (; launched < std::min(want, maxiter); ++launched)
            mg_iteration(h, b, x, fused, sc, tol, s, ends, launched);
        H_CHECK(h->mail.wait(first + it, s));
        const Mail  &m  = h->mail[first + it];
        const double r1 = std::sqrt(m.v[0]);
        rate            = r1 / rn;
        rn              = r1;
        go              = ahead ? m.v[1] != 0 : rn > tol;
        ++st->precond_applies;
    }
    if (ends && it % 2)
        H_CHECK(hipMemcpyAsync(x, h->w, sizeof(double) * h->n, hipMemcpyDeviceToDevice, s));
    st->iters += it;
    st->rel_resid = rn / bnorm;
    st->converged = !go && rn <= tol;
    return BX_OK;
}

template <int K>
static void gram_schmidt(bx_helm *h, double *zj, int j, double *d1, double *d2, hipStream_t s)
{
    // w = A z with the first projection's partial sums, then each subtraction
    // with the next pass's partial sums (the last: of the norm)
    const MGLevel<double> &L0 = h->mg64.lev[0];
    const dim3             g(h->nb_dot), t(256);
    hipLaunchKernelGGL(k_apply_multidot<K>, g, t, 0, s, zj, h->w, L0.a, L0.bX, L0.bY, L0.cX,
                       L0.cY, L0.nx, L0.ny, h->mg64.d_sc, L0.dxinv, L0.dyinv, h->V, j + 1,
                       h->partial);
    hipLaunchKernelGGL(k_reduce_partials, dim3(j + 1), t, 0, s, h->partial, h->nb_dot, j + 1,
                       d1);
    hipLaunchKernelGGL(k_subtract_dots<K>, g, t, 0, s, h->w, h->V, d1, j + 1, h->n, 1,
                       h->partial);
    hipLaunchKernelGGL(k_reduce_partials, dim3(j + 1), t, 0, s, h->partial, h->nb_dot, j + 1,
                       d2);
    hipLaunchKernelGGL(k_subtract_dots<K>, g, t, 0, s, h->w, h->V, d2, j + 1, h->n, 0,
                       h->partial);
}

// Flexible GMRES(m), right preconditioned, FP64 vectors and dot products,
// classical Gram-Schmidt applied twice.  The Hessenberg matrix, the Givens
// rotations and the triangular solve stay on the device; the host reads two
// status words per iteration (the residual estimate and the new column's
// norm), the one synchronisation an iteration needs to decide whether to
// go on.  Stall detection: if the residual has not dropped by 2x over 8
// iterations, or the iteration cap is reached, the caller falls back to
// plain multigrid.  rn0 >= 0: h->r already holds b - A x, of norm rn0.
static int solve_fgmres(bx_helm *h, const double *b, double *x, double rtol,
                        int maxiter, double bnorm, bx_solve_stats *st,
                        hipStream_t s, bool *stalled, double rn0 = -1)
{
    const long long n = h->n;
    const int       m = h->m;
    const Arnoldi   A = arnoldi_view(h->arn, m, h->m_max);
    *stalled          = false;
    int    total      = 0;
    double best       = 1e300;
    int    best_at    = 0;
    int    rc;
    bool   stop       = false; // a stall found inside the last cycle
    int    pending_j  = 0;     // directions added by the last cycle
    double beta       = rn0;
    while (true)
    {
        if (beta < 0)
        {
            if ((rc = residual_norms(h, b, x, h->r, s, &beta, nullptr)))
                return rc;
        }
        if (pending_j > 0)
        {
            if (h->mail.slots[0].v[3] != 0) // non-finite y: the iterate was kept
                stop = true;
            else
                st->iters += pending_j;
            pending_j = 0;
        }
        st->rel_resid = beta / bnorm;
        if (beta <= rtol * bnorm)
        {
            st->converged = 1;
            break;
        }
        if (stop || total >= maxiter)
        {
            *stalled = true;
            break;
        }
        hipLaunchKernelGGL(k_scale, dim3(2048), dim3(256), 0, s, h->V, h->r, n,
                           1.0 / beta);
        hipLaunchKernelGGL(k_arnoldi_init, dim3(1), dim3(64), 0, s, A, beta);
        beta  = -1;
        int j = 0;
        for (; j < m && total < maxiter; ++j)
        {
            double *vj = h->V + (long long)j * n;
            double *zj = h->Z + (long long)j * n;
            if (j > 0) // the last iteration's w, normalised
                hipLaunchKernelGGL(k_scale_inv_norm, dim3(2048), dim3(256), 0, s, vj, h->w, n,
                                   h->dots + 2 * (m + 1));
            if ((rc = precond_replay(h, vj, zj, s)))
                return rc;
            ++st->precond_applies;
            // CGS2 chained on the device (the projections are read from
            // device memory)
            double *d1 = h->dots, *d2 = h->dots + (m + 1), *d3 = h->dots + 2 * (m + 1);
            const int k = j + 1;
            if (k == 1)
                gram_schmidt<1>(h, zj, j, d1, d2, s);
            else if (k == 2)
                gram_schmidt<2>(h, zj, j, d1, d2, s);
            else if (k <= 4)
                gram_schmidt<4>(h, zj, j, d1, d2, s);
            else if (k <= 8)
                gram_schmidt<8>(h, zj, j, d1, d2, s);
            else if (k <= 16)
                gram_schmidt<16>(h, zj, j, d1, d2, s);
            else
            {
                launch_apply(h->mg64.lev[0], h->mg64, zj, h->w,
                             (const double *)nullptr, s);
                for (double *d : { d1, d2 })
                {
                    hipLaunchKernelGGL(k_multidot, dim3(h->nb_dot), dim3(256), 0, s, h->V, h->w,
                                       n, k, h->partial);
                    hipLaunchKernelGGL(k_reduce_partials, dim3(k), dim3(256), 0, s, h->partial,
                                       h->nb_dot, k, d);
                    hipLaunchKernelGGL(k_subtract_combo, dim3(2048), dim3(256), 0, s, h->w,
                                       h->V, d, k, n);
                }
                hipLaunchKernelGGL(k_multidot, dim3(h->nb_dot), dim3(256), 0, s, h->w, h->w, n,
                                   1, h->partial);
            }
            hipLaunchKernelGGL(k_norm_arnoldi, dim3(1), dim3(256), 0, s, h->partial, h->nb_dot,
                               d3, A, d1, d2, j, h->mail.dev, ++h->mail.seq);
            H_CHECK(h->mail.wait(h->mail.seq, s));
            const double est = h->mail[h->mail.seq].v[0], hn = h->mail[h->mail.seq].v[1];
            ++total;
            if (!std::isfinite(est) || !std::isfinite(hn))
            {
                // a non-finite preconditioner output: drop this direction
                stop = true;
                break;
            }
            if (est < best * 0.5)
            {
                best    = est;
                best_at = total;
            }
            if (est <= rtol * bnorm * 0.5 || hn == 0)
            {
                ++j;
                break;
            }
            if (total - best_at >= 8)
            {
                stop = true;
                ++j;
                break;
            }
        }
        // x += Z y, y from the triangular system of the first j columns
        if (j > 0)
        {
            hipLaunchKernelGGL(k_arnoldi_solve, dim3(1), dim3(64), 0, s, A, j,
                               &h->mail.dev[0].v[3]);
            hipLaunchKernelGGL(k_add_combo, dim3(2048), dim3(256), 0, s, x, h->Z, A.y, j, n);
            H_CHECK(hipGetLastError());
            pending_j = j;
        }
    }
    return BX_OK;
}

extern "C" int bx_helm_solve(bx_helm *h, const double *b, double *x, int method,
                             double rtol, int maxiter, bx_solve_stats *st,
                             void *stream)
{
    if (!h || !h->coeffs_set || !b || !x || !st || !(rtol > 0) || maxiter < 1
        || method < BX_SOLVE_MG || method > BX_SOLVE_MG_FUSED)
        return herr(BX_ERR_INVALID, "bx_helm_solve: bad argument");
    if (method == BX_SOLVE_FGMRES_CNN && !h->cnn)
        return herr(BX_ERR_STATE, "bx_helm_solve: no network attached");
    hipStream_t s = (hipStream_t)stream;
    std::memset(st, 0, sizeof(*st));
    const auto t0 = std::chrono::steady_clock::now();
    double     bnorm = 0, rn0 = 0;
    int        rc;
    const bool mg = method == BX_SOLVE_MG || method == BX_SOLVE_MG_FUSED;
    // the initial residual where the method starts from it, its norm and ||b||
    if ((rc = residual_norms(h, b, x, mg ? h->mg64.lev[0].rhs : h->r, s, &rn0, &bnorm)))
        return rc;
    if (bnorm == 0)
    {
        hipLaunchKernelGGL((k_fill<double>), dim3(2048), dim3(256), 0, s, x, h->n,
                           0.0);
        st->converged = 1;
        H_CHECK(hipStreamSynchronize(s));
        return BX_OK;
    }
    if (mg)
    {
        if ((rc = solve_mg(h, b, x, rtol, maxiter, bnorm, st, s,
                           method == BX_SOLVE_MG_FUSED, rn0)))
            return rc;
    }
    else
    {
        if ((rc = ensure_mg32(h, s)))
            return rc;
        bx_cnn *saved = h->cnn;
        if (method == BX_SOLVE_FGMRES_MG)
            h->cnn = nullptr;
        bool stalled = false;
        rc           = solve_fgmres(h, b, x, rtol, maxiter, bnorm, st, s, &stalled, rn0);
        h->cnn       = saved;
        if (rc)
            return rc;
        if (!st->converged)
        {
            // fall back to plain multigrid from the current iterate
            st->fell_back = 1;
            if ((rc = solve_mg(h, b, x, rtol, 1000, bnorm, st, s)))
                return rc;
        }
    }
    // The message that carried the final norm is posted by the launch that
    // still stores the iterate, and more may follow it: the copy of an iterate
    // that ended in the other array, kernels of an iteration launched ahead.
    H_CHECK(hipStreamSynchronize(s));
    st->seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0)
                      .count();
    return BX_OK;
}
