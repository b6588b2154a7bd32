// Batched Newton-Krylov for many independent 1D problems ("pores") packed
// into one device problem (see Problem::npores).
//
// Every pore is its own nonlinear system: the reference solves one such
// problem with newton_solver (src/dft_newton.c:131-196), a Schur-complement
// GMRES per step (src/dft_HardSphereLinProbMgr.cpp:345-428) and the damped
// update of update_solution (:266-380).  Here all pores advance in lockstep:
//
//  * the fill, the Schur products and the Newton update run once over the
//    whole packed batch (the stencil kernels see each pore between wall gaps);
//  * GMRES keeps one Krylov basis over the packed vector but a separate
//    Arnoldi process per pore: the Gram-Schmidt inner products are segmented
//    by pore, each pore has its own Hessenberg matrix and Givens rotations
//    and stops (freezes its iteration count) at its own tolerance;
//  * damping (frac_min), the convergence test and the iteration counts are
//    per pore; converged pores take no further updates.
//
// One Newton step is three device-only stages with no host synchronisation
// inside -- prefix (fill, norms, Schur right-hand side), a GMRES restart
// cycle of m Arnoldi steps, and the update -- each captured once into a HIP
// graph on a library-owned stream and replayed every iteration.  The host
// reads two counters per step (pores still active, pores whose GMRES has not
// converged).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <stdexcept>
#include <string>
#include <vector>

#include "tmi_device.hpp"
#include "tmi_internal.hpp"

namespace tmi {

namespace {

using namespace dev;

constexpr int kSegBlock = 512;
constexpr int kChunk = 8;   // Arnoldi steps per captured graph

__device__ inline double seg_block_sum(double v, double *sh)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) sh[wid] = v;
    __syncthreads();
    double t = 0.0;
    if (threadIdx.x < 64) {
        t = (threadIdx.x < kSegBlock / 64) ? sh[threadIdx.x] : 0.0;
        for (int o = 32; o > 0; o >>= 1) t += __shfl_down(t, o, 64);
    }
    return t;   // valid in thread 0
}

// out[p*ldo + j] = sum over pore p of V_j . w   (rows x nodes of the pore): one workgroup per pore,
// kSegGroup vectors per sweep over the pore's elements (w re-read per group, from cache) and one
// reduction round per group
constexpr int kSegGroup = 8;
__global__ __launch_bounds__(kSegBlock) void k_seg_dots(const double *__restrict__ V, long long ldv, int k,
                                                        const double *__restrict__ w, int rows, int N,
                                                        const int *__restrict__ off, double *__restrict__ out, int ldo,
                                                        const int *__restrict__ done)
{
    __shared__ double sh[kSegBlock / 64][kSegGroup];
    const int p = blockIdx.x;
    if (done[p]) return;
    const int i0 = off[p], n = off[p + 1] - i0;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    for (int j0 = 0; j0 < k; j0 += kSegGroup) {
        double acc[kSegGroup];
#pragma unroll
        for (int g = 0; g < kSegGroup; ++g) acc[g] = 0.0;
        for (int r = 0; r < rows; ++r) {
            const size_t base = (size_t)r * N + i0;
            for (int i = threadIdx.x; i < n; i += kSegBlock) {
                const double wv = w[base + i];
#pragma unroll
                for (int g = 0; g < kSegGroup; ++g)
                    if (j0 + g < k) acc[g] += V[(size_t)(j0 + g) * ldv + base + i] * wv;
            }
        }
#pragma unroll
        for (int g = 0; g < kSegGroup; ++g) {
            double a = acc[g];
            for (int o = 32; o > 0; o >>= 1) a += __shfl_down(a, o, 64);
            if (lane == 0) sh[wid][g] = a;
        }
        __syncthreads();
        if (threadIdx.x < kSegGroup && j0 + (int)threadIdx.x < k) {
            double t = 0.0;
            for (int q = 0; q < kSegBlock / 64; ++q) t += sh[q][threadIdx.x];
            out[(size_t)p * ldo + j0 + threadIdx.x] = t;
        }
        __syncthreads();   // sh is reused by the next group
    }
}

// w[e] += alpha * sum_j V_j[e] coef[pore(e)][j] (pores whose GMRES is done: w left alone)
__global__ void k_seg_gemv(const double *__restrict__ V, long long ldv, int k, const double *__restrict__ coef, int ldc,
                           double alpha, double *__restrict__ w, int rows, int N, const int *__restrict__ pore_of,
                           const int *__restrict__ done)
{
    const long long e = (long long)blockIdx.x * kBlock + threadIdx.x;
    if (e >= (long long)rows * N) return;
    const int i = (int)(e % N);
    if (done[pore_of[i]]) return;
    const double *c = coef + (size_t)pore_of[i] * ldc;
    double s = 0.0;
    for (int j = 0; j < k; ++j) s += V[(size_t)j * ldv + e] * c[j];
    w[e] += alpha * s;
}

__global__ void k_fill(double *__restrict__ y, double v, long long n)
{
    const long long i = (long long)blockIdx.x * kBlock + threadIdx.x;
    if (i < n) y[i] = v;
}

// y = a - b
__global__ void k_sub(const double *__restrict__ a, const double *__restrict__ b, double *__restrict__ y, long long n)
{
    const long long i = (long long)blockIdx.x * kBlock + threadIdx.x;
    if (i < n) y[i] = a[i] - b[i];
}

// out[p rows + r] = sum over row r of pore p of x^2: one workgroup per row, so that few pores still
// reach many CUs
__global__ __launch_bounds__(kBlock) void k_seg_sumsq(const double *__restrict__ x, int N, const int *__restrict__ off,
                                                      double *__restrict__ out)
{
    __shared__ double sh[kBlock / 64];
    const int p = blockIdx.x, r = blockIdx.y;
    const int i0 = off[p], n = off[p + 1] - i0;
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += kBlock) {
        const double v = x[(size_t)r * N + i0 + i];
        s += v * v;
    }
    for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int q = 0; q < kBlock / 64; ++q) t += sh[q];
        out[(size_t)p * gridDim.y + r] = t;
    }
}

// Normalise pore p's segment of w into v and store the norm in hn[p] (and hn2[p]).
__global__ __launch_bounds__(kSegBlock) void k_seg_normalize(const double *__restrict__ w, double *__restrict__ v,
                                                             int rows, int N, const int *__restrict__ off,
                                                             double *__restrict__ hn, double *__restrict__ hn2)
{
    __shared__ double sh[kSegBlock / 64];
    __shared__ double nrm;
    const int p = blockIdx.x;
    const int i0 = off[p], n = off[p + 1] - i0;
    double s = 0.0;
    for (int e = threadIdx.x; e < rows * n; e += kSegBlock) {
        const int r = e / n, i = e - r * n;
        const double t = w[(size_t)r * N + i0 + i];
        s += t * t;
    }
    s = seg_block_sum(s, sh);
    if (threadIdx.x == 0) {
        nrm = sqrt(s);
        hn[p] = nrm;
        if (hn2) hn2[p] = nrm;
    }
    __syncthreads();
    const double inv = nrm > 0.0 ? 1.0 / nrm : 0.0;
    for (int e = threadIdx.x; e < rows * n; e += kSegBlock) {
        const int r = e / n, i = e - r * n;
        const size_t q = (size_t)r * N + i0 + i;
        v[q] = w[q] * inv;
    }
}

// One thread: the new Hessenberg column h[0 .. k] and norm hn of segment p under the rotations cs, sn of the
// columns before it (h, cs, sn: LDS), its own rotation, the residual and the convergence flag; mirror
// (optional, pinned host memory): the flag and the step count.
__device__ inline void givens_column(double *h, double hn, int k, const double *cs, const double *sn, const GmresState &st, int p,
                                     double tol, double *mirror)
{
    const int m = st.m;
    double up = h[0];
    for (int j = 0; j < k; ++j) {
        const double b = h[j + 1];
        h[j] = cs[j] * up + sn[j] * b;
        up = -sn[j] * up + cs[j] * b;
    }
    const double den = sqrt(up * up + hn * hn);
    const double c = den > 0.0 ? up / den : 1.0, sv = den > 0.0 ? hn / den : 0.0;
    h[k] = den;
    st.cs[(size_t)p * m + k] = c;
    st.sn[(size_t)p * m + k] = sv;
    double *g = st.g + (size_t)p * (m + 1);
    const double gk = g[k], gn = -sv * gk;
    g[k + 1] = gn;
    g[k] = c * gk;
    st.kdone[p] = k + 1;
    const int done = fabs(gn) <= tol * st.bn[p] || hn == 0.0;
    if (done) st.done[p] = 1;
    if (mirror) {
        mirror[0] = done;
        mirror[1] = k + 1;
    }
}

// One Arnoldi step of every segment in one launch: classical Gram-Schmidt of w against V_0 .. V_k with
// one reorthogonalisation pass, the normalised result as V_k+1, the new Hessenberg column with its
// Givens rotations, and the convergence flag.  One workgroup per segment (the segments are
// independent), w in registers, so that the step reads w once and each V_j four times where separate
// launches read w six times more and wait for each other five times.  Bound by one CU's reads of V from
// the L2 (4 k sweeps of the segment) for long segments, by its dependent reductions for short ones.
// Finished segments only clear their next vector.  Measured per step against the six launches: 256 pores (up to 3002
// unknowns, k about 10) 89 -> 22 us, 16 slits (up to 6464) 97 -> 40 us.
constexpr int kOrthoGroup = 8;
constexpr int kOrthoMaxM = 512;   // longest restart cycle of the LDS bookkeeping
template <int BT, int NPT>
__global__ __launch_bounds__(BT) void k_seg_ortho(double *__restrict__ V, long long ldv, int k,
                                                  const double *__restrict__ w, int rows, int N,
                                                  const int *__restrict__ off, GmresState st, double tol,
                                                  double *__restrict__ mirror)
{
    constexpr int NW = BT / 64;
    __shared__ double h[kOrthoMaxM + 1], hs[kOrthoMaxM + 1], cs[kOrthoMaxM], sn[kOrthoMaxM];
    __shared__ double red[2][NW][kOrthoGroup];
    __shared__ double nrm;
    const int p = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int i0 = off[p], n = off[p + 1] - i0, len = rows * n, m = st.m;
    if (st.done[p]) {   // finite values: the stencil kernels read across the gap between segments with zero weights
        for (int e = tid; e < len; e += BT) {
            const int r = e / n;
            V[(size_t)(k + 1) * ldv + (size_t)r * N + i0 + (e - r * n)] = 0.0;
        }
        return;
    }
    double wv[NPT];
    int ix[NPT];
#pragma unroll
    for (int t = 0; t < NPT; ++t) {   // element e of the segment: row e / n, node e mod n
        const int e = tid + t * BT, r = e < len ? e / n : 0;
        ix[t] = e < len ? r * N + i0 + (e - r * n) : i0;
        wv[t] = e < len ? w[ix[t]] : 0.0;
    }
    for (int j = tid; j < k; j += BT) {
        cs[j] = st.cs[(size_t)p * m + j];
        sn[j] = st.sn[(size_t)p * m + j];
    }
    // out[j] = V_j . w, kOrthoGroup vectors per reduction round
    int buf = 0;
    auto dots = [&](double *out) {
        for (int j0 = 0; j0 <= k; j0 += kOrthoGroup) {
            double acc[kOrthoGroup];
#pragma unroll
            for (int g = 0; g < kOrthoGroup; ++g) acc[g] = 0.0;
            const double *Vj = V + (size_t)j0 * ldv;
#pragma unroll(NPT <= 4 ? NPT : 4)
            for (int t = 0; t < NPT; ++t) {
#pragma unroll
                for (int g = 0; g < kOrthoGroup; ++g)
                    if (j0 + g <= k) acc[g] += Vj[(size_t)g * ldv + ix[t]] * wv[t];
            }
            // sums over the wave: halve the values held per lane while pairing lanes, then fold the rest
#pragma unroll
            for (int s = kOrthoGroup / 2, msk = 1; s >= 1; s >>= 1, msk <<= 1) {
                const bool hi = lane & msk;
#pragma unroll
                for (int i = 0; i < kOrthoGroup / 2; ++i)
                    if (i < s) {
                        const double give = hi ? acc[i] : acc[i + s], keep = hi ? acc[i + s] : acc[i];
                        acc[i] = keep + __shfl_xor(give, msk, 64);
                    }
            }
            for (int msk = kOrthoGroup; msk < 64; msk <<= 1) acc[0] += __shfl_xor(acc[0], msk, 64);
            // lane l < 8 holds value g = (l bit 0) * 4 + (l bit 1) * 2 + (l bit 2)
            if (lane < kOrthoGroup) red[buf][wid][((lane & 1) << 2) | (lane & 2) | ((lane >> 2) & 1)] = acc[0];
            __syncthreads();
            if (tid < kOrthoGroup && j0 + tid <= k) {
                double t = 0.0;
#pragma unroll
                for (int q = 0; q < NW; ++q) t += red[buf][q][tid];
                out[j0 + tid] = t;
            }
            buf ^= 1;   // the other half is written next: its readers passed this barrier
        }
        __syncthreads();
    };
    auto update = [&](const double *c) {   // w -= V c
        double s[NPT];
#pragma unroll
        for (int t = 0; t < NPT; ++t) s[t] = 0.0;
#pragma unroll(NPT <= 4 ? 4 : 2)
        for (int j = 0; j <= k; ++j) {
            const double cj = c[j];
#pragma unroll
            for (int t = 0; t < NPT; ++t) s[t] += V[(size_t)j * ldv + ix[t]] * cj;
        }
#pragma unroll
        for (int t = 0; t < NPT; ++t) wv[t] = tid + t * BT < len ? wv[t] - s[t] : 0.0;
    };
    dots(h);
    update(h);
    dots(hs);
    update(hs);
    double q = 0.0;
#pragma unroll
    for (int t = 0; t < NPT; ++t) q += wv[t] * wv[t];
    for (int o = 32; o > 0; o >>= 1) q += __shfl_down(q, o, 64);
    if (lane == 0) red[buf][wid][0] = q;
    for (int j = tid; j <= k; j += BT) h[j] += hs[j];   // read again by thread 0 past the barrier
    __syncthreads();
    if (tid == 0) {
        double t = 0.0;
#pragma unroll
        for (int v = 0; v < NW; ++v) t += red[buf][v][0];
        nrm = sqrt(t);
    }
    __syncthreads();
    const double hn = nrm;
    if (tid == 0) givens_column(h, hn, k, cs, sn, st, p, tol, mirror);
    const double inv = hn > 0.0 ? 1.0 / hn : 0.0;
    double *out = V + (size_t)(k + 1) * ldv;
#pragma unroll
    for (int t = 0; t < NPT; ++t)
        if (tid + t * BT < len) out[ix[t]] = wv[t] * inv;
    __syncthreads();
    double *H = st.H + (size_t)p * (m + 1) * m;
    for (int j = tid; j <= k; j += BT) H[(size_t)j * m + k] = h[j];
}

// longest segment (unknowns) of one workgroup
constexpr int kOrthoMaxLen = 16384;

// start of a restart cycle: hn[p] = beta_p (already normalised V0);
// done_p is set for inactive pores and pores already at tolerance
__global__ void k_gmres_start(int P, GmresState st, const int *__restrict__ active, double tol)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= P) return;
    const int m = st.m;
    const double beta = st.hn[p];
    double *g = st.g + (size_t)p * (m + 1);
    for (int j = 0; j <= m; ++j) g[j] = 0.0;
    g[0] = beta;
    st.kdone[p] = 0;
    st.done[p] = (!active[p] || beta <= tol * st.bn[p] || beta == 0.0) ? 1 : 0;
}

// the same for one problem; mirror (pinned host memory): the flag and the step count
__global__ void k_line_start(GmresState st, const int *__restrict__ active, double tol, double *__restrict__ mirror)
{
    const double beta = st.hn[0];
    for (int j = threadIdx.x; j <= st.m; j += blockDim.x) st.g[j] = j ? 0.0 : beta;
    if (threadIdx.x == 0) {
        const int done = !active[0] || beta <= tol * st.bn[0] || beta == 0.0;
        st.kdone[0] = 0;
        st.done[0] = done;
        mirror[0] = done;
        mirror[1] = 0.0;
    }
}

// the column of one problem's step k whose Gram-Schmidt ran over the chip (dev_cgs2's coefficients, |w|^2 last)
__global__ __launch_bounds__(64) void k_line_givens(GmresState st, int k, const double *__restrict__ coef, double tol,
                                                    double *__restrict__ mirror)
{
    __shared__ double h[kOrthoMaxM + 1], cs[kOrthoMaxM], sn[kOrthoMaxM];
    const int m = st.m;
    for (int j = threadIdx.x; j <= k; j += 64) {
        h[j] = coef[j] + coef[k + 1 + j];
        if (j < k) {
            cs[j] = st.cs[j];
            sn[j] = st.sn[j];
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) givens_column(h, sqrt(coef[2 * (k + 1)]), k, cs, sn, st, 0, tol, mirror);
    __syncthreads();
    for (int j = threadIdx.x; j <= k; j += 64) st.H[(size_t)j * m + k] = h[j];
}

// Arnoldi step k: new column (h1 + h2, hn) of each active pore's Hessenberg
// matrix, previous rotations applied, new rotation formed, residual updated.
__global__ void k_gmres_givens(int P, int k, GmresState st, double tol)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= P || st.done[p]) return;
    const int m = st.m;
    double *H = st.H + (size_t)p * (m + 1) * m;
    double *cs = st.cs + (size_t)p * m, *sn = st.sn + (size_t)p * m, *g = st.g + (size_t)p * (m + 1);
    const double *h1 = st.h1 + (size_t)p * (m + 1), *h2 = st.h2 + (size_t)p * (m + 1);
    for (int j = 0; j <= k; ++j) H[(size_t)j * m + k] = h1[j] + h2[j];
    const double hn = st.hn[p];
    H[(size_t)(k + 1) * m + k] = hn;
    for (int j = 0; j < k; ++j) {
        const double a = H[(size_t)j * m + k], b = H[(size_t)(j + 1) * m + k];
        H[(size_t)j * m + k] = cs[j] * a + sn[j] * b;
        H[(size_t)(j + 1) * m + k] = -sn[j] * a + cs[j] * b;
    }
    const double a = H[(size_t)k * m + k], b = H[(size_t)(k + 1) * m + k];
    const double den = sqrt(a * a + b * b);
    cs[k] = den > 0.0 ? a / den : 1.0;
    sn[k] = den > 0.0 ? b / den : 0.0;
    H[(size_t)k * m + k] = den;
    H[(size_t)(k + 1) * m + k] = 0.0;
    g[k + 1] = -sn[k] * g[k];
    g[k] = cs[k] * g[k];
    st.kdone[p] = k + 1;
    if (fabs(g[k + 1]) <= tol * st.bn[p] || hn == 0.0) st.done[p] = 1;
}

// y = R^{-1} g over each pore's kdone steps (zero beyond), one wave per pore: each y_i is taken out of
// the remaining right-hand side by all lanes at once; iteration counts
__global__ __launch_bounds__(64) void k_gmres_solve(GmresState st)
{
    const int p = blockIdx.x, lane = threadIdx.x;
    const int m = st.m, k = st.kdone[p];
    const double *H = st.H + (size_t)p * (m + 1) * m, *g = st.g + (size_t)p * (m + 1);
    double *y = st.y + (size_t)p * m;
    __shared__ double r[kOrthoMaxM];
    for (int j = lane; j < m; j += 64) {
        y[j] = 0.0;
        r[j] = g[j];
    }
    __syncthreads();
    for (int i = k - 1; i >= 0; --i) {
        const double yi = r[i] / H[(size_t)i * m + i];
        if (lane == 0) y[i] = yi;
        for (int j = lane; j < i; j += 64) r[j] -= H[(size_t)j * m + i] * yi;
        __syncthreads();
    }
    if (lane == 0) st.its[p] += k;
}

// x2 += dinv (V y) over each pore's steps
__global__ void k_seg_update(const double *__restrict__ V, long long ldv, GmresState st, const double *__restrict__ dinv,
                             double *__restrict__ x2, int rows, int N, const int *__restrict__ pore_of)
{
    const long long e = (long long)blockIdx.x * kBlock + threadIdx.x;
    if (e >= (long long)rows * N) return;
    const int p = pore_of ? pore_of[(int)(e % N)] : 0;
    const int k = st.kdone[p];
    const double *y = st.y + (size_t)p * st.m;
    double s = 0.0;
    for (int j = 0; j < k; ++j) s += V[(size_t)j * ldv + e] * y[j];
    x2[e] += dinv[e] * s;
}

// pores still running: count[0] = #(active), or #(active and GMRES not done)
__global__ void k_count(int P, const int *__restrict__ active, const int *__restrict__ done, int *__restrict__ count)
{
    __shared__ int sh[kBlock];
    int c = 0;
    for (int p = threadIdx.x; p < P; p += kBlock) c += (active[p] && (!done || !done[p])) ? 1 : 0;
    sh[threadIdx.x] = c;
    __syncthreads();
    for (int s = kBlock / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) count[0] = sh[0];
}

// Newton bookkeeping after a fill (rn2: the rows' sums of squares): pores whose ||F_p|| < tol stop.
__global__ void k_newton_flags(int P, int rows, const double *__restrict__ rn2, double tol, int iter, int *__restrict__ active,
                               int *__restrict__ conv, int *__restrict__ iters, double *__restrict__ rnorm)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= P) return;
    double ss = 0.0;
    for (int r = 0; r < rows; ++r) ss += rn2[(size_t)p * rows + r];
    const double rn = sqrt(ss);
    rnorm[p] = rn;
    if (!active[p]) return;
    if (rn < tol) {
        active[p] = 0;
        conv[p] = 1;
        iters[p] = iter;
    } else if (!(rn == rn)) {
        active[p] = 0;   // NaN: stop this pore, reported as not converged
        iters[p] = iter;
    }
}

// update_solution per pore: frac_p = min over the pore's densities of
// max(min(1, x/(-dx)), scaling) where x + dx < 0
__global__ __launch_bounds__(kSegBlock) void k_seg_frac_min(const double *__restrict__ x, const double *__restrict__ dx,
                                                            int C, int N, const int *__restrict__ off, double scaling,
                                                            const int *__restrict__ active, double *__restrict__ frac)
{
    __shared__ double sh[kSegBlock];
    const int p = blockIdx.x;
    const int i0 = off[p], n = off[p + 1] - i0;
    double mn = 1.0;
    for (int e = threadIdx.x; e < C * n; e += kSegBlock) {
        const int r = e / n, i = e - r * n;
        const size_t q = (size_t)r * N + i0 + i;
        const double xv = x[q], d = dx[q];
        if (xv + d < 0.0) mn = fmin(mn, fmax(fmin(1.0, xv / (-d)), scaling));
    }
    sh[threadIdx.x] = mn;
    __syncthreads();
    for (int s = kSegBlock / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) sh[threadIdx.x] = fmin(sh[threadIdx.x], sh[threadIdx.x + s]);
        __syncthreads();
    }
    if (threadIdx.x == 0) frac[p] = active[p] ? sh[0] : 0.0;
}

// x += frac_p dx with the clamps of update_solution (src/dft_newton.c:266-380)
__global__ void k_seg_apply_update(double *__restrict__ x, const double *__restrict__ dx, long long n, int C, int N,
                                   int iu_n3, const int *__restrict__ pore_of, const double *__restrict__ frac)
{
    const long long e = (long long)blockIdx.x * kBlock + threadIdx.x;
    if (e >= n) return;
    const int u = (int)(e / N), i = (int)(e % N);
    const double f = frac[pore_of[i]];
    if (f == 0.0) return;
    const double xv = x[e], d = dx[e];
    // the limiting density goes to 0.1 x as in exact arithmetic, not to the rounding residue of
    // x + f dx (k_apply_update)
    const bool limited = u < C && xv + d < 0.0 && fmin(1.0, xv / (-d)) <= f;
    if (u < C && (xv + f * d < 1.e-99 || limited))
        x[e] = 0.1 * xv;
    else if (u == iu_n3 && xv + f * d > 1.0)
        x[e] = xv + 0.5 * (1.0 - xv);
    else
        x[e] = xv + f * d;
}

inline unsigned nblk(long long n, int b = kBlock) { return (unsigned)((n + b - 1) / b); }

}  // namespace

// ---------------------------------------------------------------- work buffers
struct BatchWork {
    int P = 0, m = 0, longest = 0;   // pores, restart length, nodes of the largest pore
    size_t ntot = 0, n2 = 0;
    hipStream_t stream = nullptr;
    double *buf = nullptr;     // all doubles below
    int *ibuf = nullptr;       // all ints below
    int *h_counts = nullptr;   // pinned [2]
    // vectors
    double *x;   // the solve's own copy of the unknowns: the graphs do not depend on the caller's buffer
    double *F, *b, *dx, *bS, *dinv, *V, *z, *w, *t1, *r;
    // per pore
    double *rn2, *rnorm, *frac;
    GmresState gs;
    int *active, *conv, *niters, *counts;
    // graphs
    hipGraphExec_t g_pre = nullptr, g_start0 = nullptr, g_start = nullptr, g_finish = nullptr, g_post = nullptr;
    std::vector<hipGraphExec_t> g_steps;   // Arnoldi steps [j*kChunk, (j+1)*kChunk)
    // what their launches depend on besides the buffers (graph_prec -1: none captured)
    int graph_prec = -1, graph_rev = 0;
    double graph_tol[2] = {0, 0};
};

void free_batch_work(Problem &P)
{
    BatchWork *W = P.batch_work;
    if (!W) return;
    for (hipGraphExec_t g : {W->g_pre, W->g_start0, W->g_start, W->g_finish, W->g_post})
        if (g) (void)hipGraphExecDestroy(g);
    for (hipGraphExec_t g : W->g_steps)
        if (g) (void)hipGraphExecDestroy(g);
    (void)hipFree(W->buf);
    (void)hipFree(W->ibuf);
    if (W->h_counts) (void)hipHostFree(W->h_counts);
    if (W->stream) (void)hipStreamDestroy(W->stream);
    delete W;
    P.batch_work = nullptr;
}

static BatchWork &batch_work(Problem &P, int m)
{
    if (P.batch_work && P.batch_work->m == m) return *P.batch_work;
    free_batch_work(P);
    auto *W = new BatchWork();
    P.batch_work = W;
    W->P = P.npores;
    W->m = m;
    const int Pn = P.npores;
    for (int p = 0; p < Pn; ++p) W->longest = std::max(W->longest, P.pore_off[p + 1] - P.pore_off[p]);
    W->ntot = (size_t)P.nunk * P.N;
    W->n2 = (size_t)P.p.ncomp * P.N;
    const size_t nt = W->ntot, n2 = W->n2;
    const size_t nd = 4 * nt + n2 /*bS*/ + n2 /*dinv*/ + (size_t)(m + 1) * n2 /*V*/ + 3 * n2 /*z w r*/ +
                      (size_t)(P.nrb + P.nmf) * P.N /*t1*/ + (2 + (size_t)P.nunk) * (size_t)Pn +
                      (size_t)Pn * ((size_t)(m + 1) * m + 2 * m + (m + 1) + m + 2 * (m + 1) + 2);
    const size_t ni = (size_t)Pn * 6 + 2;
    try {
        TMI_HIP_CHECK(hipStreamCreateWithFlags(&W->stream, hipStreamNonBlocking));
        TMI_HIP_CHECK(hipMalloc((void **)&W->buf, nd * sizeof(double)));
        TMI_HIP_CHECK(hipMalloc((void **)&W->ibuf, ni * sizeof(int)));
        TMI_HIP_CHECK(hipHostMalloc((void **)&W->h_counts, 2 * sizeof(int), hipHostMallocDefault));
    } catch (...) {   // no half-built work for the next solve of this length to take
        free_batch_work(P);
        throw;
    }
    double *q = W->buf;
    auto take = [&](size_t n) {
        double *r = q;
        q += n;
        return r;
    };
    W->x = take(nt);
    W->F = take(nt);
    W->b = take(nt);
    W->dx = take(nt);
    W->bS = take(n2);
    W->dinv = take(n2);
    W->V = take((size_t)(m + 1) * n2);
    W->z = take(n2);
    W->w = take(n2);
    W->r = take(n2);
    W->t1 = take((size_t)(P.nrb + P.nmf) * P.N);
    W->rn2 = take((size_t)P.nunk * Pn);
    W->rnorm = take(Pn);
    W->frac = take(Pn);
    W->gs.m = m;
    W->gs.H = take((size_t)Pn * (m + 1) * m);
    W->gs.cs = take((size_t)Pn * m);
    W->gs.sn = take((size_t)Pn * m);
    W->gs.g = take((size_t)Pn * (m + 1));
    W->gs.y = take((size_t)Pn * m);
    W->gs.h1 = take((size_t)Pn * (m + 1));
    W->gs.h2 = take((size_t)Pn * (m + 1));
    W->gs.hn = take(Pn);
    W->gs.bn = take(Pn);
    int *iq = W->ibuf;
    W->gs.kdone = iq;
    iq += Pn;
    W->gs.done = iq;
    iq += Pn;
    W->gs.its = iq;
    iq += Pn;
    W->active = iq;
    iq += Pn;
    W->conv = iq;
    iq += Pn;
    W->niters = iq;
    iq += Pn;
    W->counts = iq;
    return *W;
}

// ---------------------------------------------------------------- stages
// Schur product S v (v: density rows) in the chosen precision
static void schur_apply(Problem &P, const double *x, const double *v, double *t1, double *y, int prec, hipStream_t s)
{
    if (prec == TMI_PREC_MIXED)
        launch_schur_apply<float>(P, x, v, t1, y, s);
    else
        launch_schur_apply<double>(P, x, v, t1, y, s);
}

// prefix: F(x) and its per-pore sums of squares, b = -F, Schur right-hand
// side bS and its per-pore norms, A22^{-1}, x2 = 0
static void stage_pre(Problem &P, BatchWork &W, const double *x, hipStream_t s)
{
    const int Pn = W.P, C = P.p.ncomp, N = P.N;
    launch_residual(P, x, W.F, s);
    hipLaunchKernelGGL(k_seg_sumsq, dim3(Pn, P.nunk), dim3(kBlock), 0, s, W.F, N, P.d_pore_off, W.rn2);
    dev_scale_copy(-1.0, W.F, W.b, (long long)W.ntot, s);
    launch_schur_rhs(P, x, W.b, W.bS, s);
    dev_a22_inverse_diag(P, x, W.dinv, s);
    // bn_p = |bS|_p; x2 = 0, so bS is also the first cycle's residual and bS / bn its V0
    hipLaunchKernelGGL(k_seg_normalize, dim3(Pn), dim3(kSegBlock), 0, s, W.bS, W.V, C, N, P.d_pore_off, W.gs.bn, W.gs.hn);
    hipLaunchKernelGGL(k_fill, dim3(nblk((long long)W.n2)), dim3(kBlock), 0, s, W.dx, 0.0, (long long)W.n2);
    TMI_HIP_CHECK(hipGetLastError());
}

// One GMRES restart cycle on S x2 = bS per pore (x2 = dx[0 : C N]) in three
// parts: start (r = bS - S x2, V0, per-pore beta), Arnoldi steps [k0, k1),
// finish (per-pore least squares, x2 update).  Each part ends with the count
// of pores whose GMRES is still running, so the host can skip the remaining
// steps of a cycle once every pore has converged.
static void stage_cycle_begin(Problem &P, BatchWork &W, double tol, hipStream_t s)
{
    hipLaunchKernelGGL(k_gmres_start, dim3(nblk(W.P)), dim3(kBlock), 0, s, W.P, W.gs, W.active, tol);
    hipLaunchKernelGGL(k_count, dim3(1), dim3(kBlock), 0, s, W.P, W.active, W.gs.done, W.counts + 1);
    TMI_HIP_CHECK(hipGetLastError());
}
static void stage_cycle_start(Problem &P, BatchWork &W, const double *x, double tol, int prec, hipStream_t s)
{
    const int Pn = W.P, C = P.p.ncomp, N = P.N;
    const long long n2 = (long long)W.n2;
    schur_apply(P, x, W.dx, W.t1, W.w, prec, s);
    hipLaunchKernelGGL(k_sub, dim3(nblk(n2)), dim3(kBlock), 0, s, W.bS, W.w, W.r, n2);
    hipLaunchKernelGGL(k_seg_normalize, dim3(Pn), dim3(kSegBlock), 0, s, W.r, W.V, C, N, P.d_pore_off, W.gs.hn, nullptr);
    stage_cycle_begin(P, W, tol, s);
}

// Shape of the one-launch Arnoldi step for segments of up to len unknowns: threads by values per thread,
// enough of them that a segment's loads are in flight together, few enough values to stay in registers
static void launch_ortho(double *V, long long ldv, int k, const double *w, int rows, int N, const int *off, int Pn, int len,
                         const GmresState &st, double tol, double *mirror, hipStream_t s)
{
    auto go = [&](auto kernel, int bt) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)Pn), dim3(bt), 0, s, V, ldv, k, w, rows, N, off, st, tol, mirror);
    };
    if (len <= 2048)
        go(k_seg_ortho<512, 4>, 512);
    else if (len <= 4096)
        go(k_seg_ortho<1024, 4>, 1024);
    else if (len <= 8192)
        go(k_seg_ortho<1024, 8>, 1024);
    else
        go(k_seg_ortho<1024, 16>, 1024);
    TMI_HIP_CHECK(hipGetLastError());
}
static bool ortho_fits(long long len, int rows, int N, int m)
{
    return len <= kOrthoMaxLen && (long long)rows * N <= INT32_MAX && m <= kOrthoMaxM;
}

static void stage_cycle_steps(Problem &P, BatchWork &W, const double *x, double tol, int prec, int k0, int k1,
                              hipStream_t s)
{
    const int Pn = W.P, C = P.p.ncomp, N = P.N, m = W.m;
    const long long n2 = (long long)W.n2;
    const bool fused = schur_one_launch(P), one = ortho_fits((long long)C * W.longest, C, N, m);
    const int *done = one ? W.gs.done : nullptr;   // the separate kernels go on with every pore's vectors
    for (int k = k0; k < k1; ++k) {
        double *Vk = W.V + (size_t)k * n2;
        if (fused) {
            if (prec == TMI_PREC_MIXED)
                one_launch_schur<float>(P, x, Vk, W.dinv, W.w, done, s);
            else
                one_launch_schur<double>(P, x, Vk, W.dinv, W.w, done, s);
        } else {
            dev_mul(W.dinv, Vk, W.z, n2, s);
            schur_apply(P, x, W.z, W.t1, W.w, prec, s);
        }
        if (one) {
            launch_ortho(W.V, n2, k, W.w, C, N, P.d_pore_off, Pn, C * W.longest, W.gs, tol, nullptr, s);
            continue;
        }
        for (double *h : {W.gs.h1, W.gs.h2}) {
            hipLaunchKernelGGL(k_seg_dots, dim3(Pn), dim3(kSegBlock), 0, s, W.V, n2, k + 1, W.w, C, N, P.d_pore_off, h,
                               m + 1, W.gs.done);
            hipLaunchKernelGGL(k_seg_gemv, dim3(nblk(n2)), dim3(kBlock), 0, s, W.V, n2, k + 1, h, m + 1, -1.0, W.w, C, N,
                               P.d_pore_of, W.gs.done);
        }
        hipLaunchKernelGGL(k_seg_normalize, dim3(Pn), dim3(kSegBlock), 0, s, W.w, W.V + (size_t)(k + 1) * n2, C, N,
                           P.d_pore_off, W.gs.hn, nullptr);
        hipLaunchKernelGGL(k_gmres_givens, dim3(nblk(Pn)), dim3(kBlock), 0, s, Pn, k, W.gs, tol);
    }
    hipLaunchKernelGGL(k_count, dim3(1), dim3(kBlock), 0, s, Pn, W.active, W.gs.done, W.counts + 1);
    TMI_HIP_CHECK(hipGetLastError());
}

static void stage_cycle_finish(Problem &P, BatchWork &W, hipStream_t s)
{
    hipLaunchKernelGGL(k_gmres_solve, dim3(W.P), dim3(64), 0, s, W.gs);
    hipLaunchKernelGGL(k_seg_update, dim3(nblk((long long)W.n2)), dim3(kBlock), 0, s, W.V, (long long)W.n2, W.gs, W.dinv,
                       W.dx, P.p.ncomp, P.N, P.d_pore_of);
    TMI_HIP_CHECK(hipGetLastError());
}

// back-substitution of the nonlocal unknowns, per-pore damping and update
static void stage_post(Problem &P, BatchWork &W, double *x, double scaling, hipStream_t s)
{
    const int Pn = W.P, C = P.p.ncomp, N = P.N;
    launch_schur_backsub(P, x, W.b, W.dx, s);
    hipLaunchKernelGGL(k_seg_frac_min, dim3(Pn), dim3(kSegBlock), 0, s, x, W.dx, C, N, P.d_pore_off, scaling,
                       W.active, W.frac);
    hipLaunchKernelGGL(k_seg_apply_update, dim3(nblk((long long)W.ntot)), dim3(kBlock), 0, s, x, W.dx,
                       (long long)W.ntot, C, N, P.iu_rb, P.d_pore_of, W.frac);
    TMI_HIP_CHECK(hipGetLastError());
}

template <typename F>
static hipGraphExec_t capture(hipStream_t s, F &&enqueue)
{
    hipGraph_t g = nullptr;
    TMI_HIP_CHECK(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
    try {
        enqueue();
    } catch (...) {
        hipGraph_t tmp = nullptr;
        (void)hipStreamEndCapture(s, &tmp);
        if (tmp) (void)hipGraphDestroy(tmp);
        throw;
    }
    TMI_HIP_CHECK(hipStreamEndCapture(s, &g));
    hipGraphExec_t ex = nullptr;
    hipError_t e = hipGraphInstantiate(&ex, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    TMI_HIP_CHECK(e);
    return ex;
}

int batch_newton_solve(Problem &P, double *x_caller, const tmi_newton_opts &o, tmi_newton_stats &st, int *pore_iters,
                       int *pore_conv, int *pore_gmres, double *pore_resid, hipStream_t caller)
{
    if (P.npores < 1) throw std::logic_error("not a batched problem");
    const int m = std::max(1, std::min(o.gmres_restart, 200));
    BatchWork &W = batch_work(P, m);
    const int Pn = W.P;
    const char *ge = std::getenv("TMI_BATCH_GRAPH");
    const bool use_graph = !(ge && std::string(ge) == "0");
    hipStream_t s = W.stream;
    double *x = W.x;
    TMI_HIP_CHECK(hipStreamSynchronize(caller));
    TMI_HIP_CHECK(hipMemcpyAsync(x, x_caller, W.ntot * sizeof(double), hipMemcpyDeviceToDevice, s));
    auto t0 = std::chrono::steady_clock::now();
    st = tmi_newton_stats{};
    // per-pore state
    {
        std::vector<int> ones(Pn, 1), zeros(Pn, 0);
        TMI_HIP_CHECK(hipMemcpyAsync(W.active, ones.data(), Pn * sizeof(int), hipMemcpyHostToDevice, s));
        TMI_HIP_CHECK(hipMemcpyAsync(W.conv, zeros.data(), Pn * sizeof(int), hipMemcpyHostToDevice, s));
        TMI_HIP_CHECK(hipMemcpyAsync(W.niters, zeros.data(), Pn * sizeof(int), hipMemcpyHostToDevice, s));
        TMI_HIP_CHECK(hipMemcpyAsync(W.gs.its, zeros.data(), Pn * sizeof(int), hipMemcpyHostToDevice, s));
        TMI_HIP_CHECK(hipStreamSynchronize(s));
    }
    const int maxcycles = std::max(1, (o.gmres_max_iter + m - 1) / m);
    const int nchunks = (m + kChunk - 1) / kChunk;
    // the Newton iteration number only enters k_newton_flags, launched outside the graphs
    auto enqueue_pre = [&] { stage_pre(P, W, x, s); };
    auto enqueue_start0 = [&] { stage_cycle_begin(P, W, o.gmres_tol, s); };
    auto enqueue_start = [&] { stage_cycle_start(P, W, x, o.gmres_tol, o.precision, s); };
    auto enqueue_steps = [&](int j) {
        stage_cycle_steps(P, W, x, o.gmres_tol, o.precision, j * kChunk, std::min(m, (j + 1) * kChunk), s);
    };
    auto enqueue_finish = [&] { stage_cycle_finish(P, W, s); };
    auto enqueue_post = [&] { stage_post(P, W, x, o.update_scaling, s); };
    if (use_graph && (W.graph_prec != o.precision || W.graph_rev != P.launch_rev || W.graph_tol[0] != o.gmres_tol ||
                      W.graph_tol[1] != o.update_scaling)) {
        W.graph_prec = -1;   // until every part is captured
        for (hipGraphExec_t *g : {&W.g_pre, &W.g_start0, &W.g_start, &W.g_finish, &W.g_post})
            if (*g) {
                (void)hipGraphExecDestroy(*g);
                *g = nullptr;
            }
        for (hipGraphExec_t &g : W.g_steps)
            if (g) {
                (void)hipGraphExecDestroy(g);
                g = nullptr;
            }
        W.g_steps.assign(nchunks, nullptr);
        W.g_pre = capture(s, enqueue_pre);
        W.g_start0 = capture(s, enqueue_start0);
        W.g_start = capture(s, enqueue_start);
        for (int j = 0; j < nchunks; ++j) W.g_steps[j] = capture(s, [&] { enqueue_steps(j); });
        W.g_finish = capture(s, enqueue_finish);
        W.g_post = capture(s, enqueue_post);
        W.graph_prec = o.precision;
        W.graph_rev = P.launch_rev;
        W.graph_tol[0] = o.gmres_tol;
        W.graph_tol[1] = o.update_scaling;
    }
    auto run = [&](hipGraphExec_t g, auto &&enqueue) {
        if (use_graph)
            TMI_HIP_CHECK(hipGraphLaunch(g, s));
        else
            enqueue();
    };
    auto running = [&] {   // pores whose GMRES has not converged (one host read)
        TMI_HIP_CHECK(hipMemcpyAsync(W.h_counts + 1, W.counts + 1, sizeof(int), hipMemcpyDeviceToHost, s));
        TMI_HIP_CHECK(hipStreamSynchronize(s));
        return W.h_counts[1];
    };
    int iter = 0;
    while (true) {
        run(W.g_pre, enqueue_pre);
        hipLaunchKernelGGL(k_newton_flags, dim3(nblk(Pn)), dim3(kBlock), 0, s, Pn, P.nunk, W.rn2, o.resid_tol, iter, W.active,
                           W.conv, W.niters, W.rnorm);
        hipLaunchKernelGGL(k_count, dim3(1), dim3(kBlock), 0, s, Pn, W.active, (const int *)nullptr, W.counts);
        TMI_HIP_CHECK(hipMemcpyAsync(W.h_counts, W.counts, sizeof(int), hipMemcpyDeviceToHost, s));
        TMI_HIP_CHECK(hipStreamSynchronize(s));
        const int nactive = W.h_counts[0];
        if (o.verbose) std::fprintf(stderr, "[tmi batch] iter %d: %d of %d pores active\n", iter, nactive, Pn);
        if (nactive == 0 || iter >= o.max_iter) break;
        for (int c = 0; c < maxcycles; ++c) {
            if (c == 0)
                run(W.g_start0, enqueue_start0);
            else
                run(W.g_start, enqueue_start);
            int left = running();
            for (int j = 0; j < nchunks && left > 0; ++j) {
                if (use_graph)
                    TMI_HIP_CHECK(hipGraphLaunch(W.g_steps[j], s));
                else
                    enqueue_steps(j);
                left = running();
            }
            run(W.g_finish, enqueue_finish);
            if (left == 0) break;
        }
        run(W.g_post, enqueue_post);
        ++iter;
    }
    TMI_HIP_CHECK(hipMemcpyAsync(x_caller, x, W.ntot * sizeof(double), hipMemcpyDeviceToDevice, s));
    // pores still active at the iteration limit
    std::vector<int> act(Pn), conv(Pn), nit(Pn), gits(Pn);
    std::vector<double> rn(Pn);
    TMI_HIP_CHECK(hipMemcpyAsync(act.data(), W.active, Pn * sizeof(int), hipMemcpyDeviceToHost, s));
    TMI_HIP_CHECK(hipMemcpyAsync(conv.data(), W.conv, Pn * sizeof(int), hipMemcpyDeviceToHost, s));
    TMI_HIP_CHECK(hipMemcpyAsync(nit.data(), W.niters, Pn * sizeof(int), hipMemcpyDeviceToHost, s));
    TMI_HIP_CHECK(hipMemcpyAsync(gits.data(), W.gs.its, Pn * sizeof(int), hipMemcpyDeviceToHost, s));
    TMI_HIP_CHECK(hipMemcpyAsync(rn.data(), W.rnorm, Pn * sizeof(double), hipMemcpyDeviceToHost, s));
    TMI_HIP_CHECK(hipStreamSynchronize(s));
    double rsum = 0.0;
    int nconv = 0, gtot = 0;
    for (int p = 0; p < Pn; ++p) {
        if (act[p]) nit[p] = iter;
        rsum += rn[p] * rn[p];
        nconv += conv[p];
        gtot += gits[p];
        if (pore_iters) pore_iters[p] = nit[p];
        if (pore_conv) pore_conv[p] = conv[p];
        if (pore_gmres) pore_gmres[p] = gits[p];
        if (pore_resid) pore_resid[p] = rn[p];
    }
    st.iters = iter;
    st.converged = (nconv == Pn) ? 1 : 0;
    st.gmres_iters_total = gtot;
    st.resid_norm = std::sqrt(rsum);
    st.seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    return 0;
}

// One small 1D problem (the whole vector is one segment): two launches per Arnoldi step, and the host
// reads the convergence flag every kLineSteps steps; steps past convergence return at once.
// The rule: the Schur product in one launch, up to 8192 unknowns (601 nodes of two components: Newton 4.1 ->
// 2.2 ms), and while the basis is one that a workgroup sweeps faster than eight launches over the chip do:
// `sweep` values of it, fewer where a thread holds more than four values of w.  From there on the
// Gram-Schmidt passes run over the chip, with the rotations still on the device and one host read per step.
// A step on average, 84 of them at 3001 unknowns: 105 us in one workgroup throughout, 102 so, 136 with the rotations
// on the host (gmres_schur_t); 83 at 8001: 222, 108 and 136 us.
bool gmres_line(Problem &P, const double *x, const double *bS, double *x2, double rtol, int m, int maxit, int prec,
                double *work, int *iters, hipStream_t s)
{
    constexpr int kLineSteps = 4, kLineMax = 8192;
    const int C = P.p.ncomp, N = P.N;
    const long long n = (long long)C * N, sweep = n <= 4096 ? 200000 : 70000;
    if (P.npores > 0 || !line_available(P) || !schur_one_launch(P) || n > kLineMax || m > kOrthoMaxM) return false;
    if (P.line_gs_m != m) {
        (void)hipFree(P.d_line_gs);
        (void)hipFree(P.d_line_gi);
        P.d_line_gs = nullptr;
        P.d_line_gi = nullptr;
        P.line_gs_m = 0;
        TMI_HIP_CHECK(hipMalloc((void **)&P.d_line_gs, ((size_t)(m + 1) * m + 4 * (size_t)(m + 1) + 2) * sizeof(double)));
        TMI_HIP_CHECK(hipMalloc((void **)&P.d_line_gi, 6 * sizeof(int)));
        const int init[6] = {0, N, 1, 0, 0, 0};   // segment offsets, active; done, steps, iterations
        TMI_HIP_CHECK(hipMemcpy(P.d_line_gi, init, sizeof(init), hipMemcpyHostToDevice));
        P.line_gs_m = m;
    }
    GmresState st{};
    double *q = P.d_line_gs;
    st.m = m;
    st.H = q;
    q += (size_t)(m + 1) * m;
    st.cs = q;
    q += m + 1;
    st.sn = q;
    q += m + 1;
    st.g = q;
    q += m + 1;
    st.y = q;
    q += m + 1;
    st.hn = q;
    st.bn = q + 1;
    const int *off = P.d_line_gi, *active = P.d_line_gi + 2;
    st.done = P.d_line_gi + 3;
    st.kdone = P.d_line_gi + 4;
    st.its = P.d_line_gi + 5;
    double *V = work, *w = V + (size_t)(m + 1) * n, *r = w + n, *dinv = r + n;
    dev_a22_inverse_diag(P, x, dinv, s);
    hipLaunchKernelGGL(k_fill, dim3(nblk(n)), dim3(kBlock), 0, s, x2, 0.0, n);
    auto product = [&](const double *v, const double *mul, const int *done) {
        if (prec == TMI_PREC_MIXED)
            line_schur<float>(P, x, v, mul, w, done, s);
        else
            line_schur<double>(P, x, v, mul, w, done, s);
    };
    auto normalise = [&](const double *from, double *hn2) {
        hipLaunchKernelGGL(k_seg_normalize, dim3(1), dim3(kSegBlock), 0, s, from, V, C, N, off, st.hn, hn2);
        hipLaunchKernelGGL(k_line_start, dim3(1), dim3(64), 0, s, st, active, rtol, P.h_red_dev);
    };
    int its = 0;
    normalise(bS, st.bn);
    while (its < maxit) {
        const int steps = std::min(m, maxit - its);
        int k = 0, done = 0;
        while (k < steps && !done) {
            const int narrow = (int)std::min<long long>(steps, sweep / n);   // steps of one workgroup
            if (k < narrow) {
                for (const int end = std::min(narrow, k + kLineSteps); k < end; ++k) {
                    product(V + (size_t)k * n, dinv, st.done);
                    launch_ortho(V, n, k, w, C, N, off, 1, (int)n, st, rtol, P.h_red_dev, s);
                }
            } else {
                double *coef = P.d_red + kRedPartials;
                product(V + (size_t)k * n, dinv, nullptr);
                dev_cgs2<double>(P, V, n, k + 1, w, n, V + (size_t)(k + 1) * n, coef, s);
                hipLaunchKernelGGL(k_line_givens, dim3(1), dim3(64), 0, s, st, k, coef, rtol, P.h_red_dev);
                ++k;
            }
            TMI_HIP_CHECK(hipStreamSynchronize(s));
            done = P.h_red[0] != 0.0;
        }
        k = (int)P.h_red[1];
        its += k;
        if (k > 0) {
            hipLaunchKernelGGL(k_gmres_solve, dim3(1), dim3(64), 0, s, st);
            hipLaunchKernelGGL(k_seg_update, dim3(nblk(n)), dim3(kBlock), 0, s, V, n, st, dinv, x2, C, N, (const int *)nullptr);
        }
        if (done || its >= maxit) break;
        product(x2, nullptr, nullptr);   // r = bS - S x2
        hipLaunchKernelGGL(k_sub, dim3(nblk(n)), dim3(kBlock), 0, s, bS, w, r, n);
        normalise(r, nullptr);
    }
    TMI_HIP_CHECK(hipGetLastError());
    *iters = its;
    return true;
}

}  // namespace tmi
