// The stencil rows of one-component 2D problems and batches of 2D pieces on the matrix cores.
//
// A workgroup owns 16 x 16 nodes of one piece and stages the densities (attraction reach around the
// tile) and the four adjoint fields (FMT reach) in LDS, boundary values included, so no padded copy of
// either is built in memory.  Every sum is a chain of Toeplitz products: for each column offset dx,
//   D[i][j] += sum_k A_dx[i][k] B_dx[k][j],   A_dx[i][k] = w(dy = k - i - f, dx),
//   B_dx[k][j] = field(row k of the window, column j + dx),
// 4 window rows k per v_mfma 16x16x4, over the rows where the offset's column of the stencil is
// non-zero.  Operand lanes: A[i][k] at lane i + 16 k, B[k][j] at lane j + 16 k; D[i][j] at lane
// j + 16 (i % 4), register i / 4 in FP64 and at lane j + 16 (i / 4), register i % 4 in FP32.  B comes from
// LDS (16 consecutive values of 4 rows), A from a table transposed and zero-padded per dx, so that a
// wave reads 19 consecutive weights from one or two cache lines without bounds checks.
//
// Half of the waves share out the attraction offsets, a quarter takes the rho-bar sums (theta, delta,
// delta x, delta y), a quarter the Euler-Lagrange sums (one adjoint field each); waves are dealt to the
// four SIMDs in turn, so each SIMD gets an equal part of all three.  A Schur product needs the rho-bar
// sums before the adjoint fields: k_plane_schur forms the fields at the nodes, k_plane then runs the
// attraction and Euler-Lagrange sums.
// Bound by the FP64 matrix rate (64 cycles a product and SIMD) and the window loads before it: 256^2 nodes
// at dx = 0.05 sigma, attraction reach 2.5 sigma: 1.0e6 products, 26 us; a workgroup spends 40k cycles on
// its windows and 82k on 62k cycles' worth of products.  There a fill's rows take 59 us, the fill 81 us
// (132 us as FFT sums); 16 pieces of 64 columns at dx = 0.1 sigma (73,088 nodes): Schur product 42 us
// (98 us in separate launches), mixed Newton solve of the batch 9.5 ms (16.3 ms).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <string>
#include <type_traits>
#include <vector>

#include "tmi_device.hpp"
#include "tmi_fmt.hpp"
#include "tmi_internal.hpp"

namespace tmi {

// Tiles, weight tables and buffers of one problem.
struct PlanePlan {
    int ntiles = 0;
    int4 *tiles = nullptr;   // x0, first node row, first and one past the last node row of its piece
    // weights [sum][dx][2 f + kPlanePad] (sums: theta, delta, delta x, delta y) and [dx][2 h + kPlanePad], and the
    // window rows [klo, khi) a dx needs
    double *wf = nullptr, *wu = nullptr;
    float *wf32 = nullptr, *wu32 = nullptr;
    int2 *kf = nullptr, *ku = nullptr;
    int fx = 0, fy = 0, hx = 0, hy = 0;
    void *adj = nullptr;     // [4][N] adjoint fields at the nodes (Schur products)
    bool on = false, rows = true;   // serves the problem; calls for the rows alone as well
};

namespace {

using namespace dev;

constexpr int kPlanePad = 34;   // 15 zeros before a column's weights, 18 after (whole 4-row steps)

template <typename T>
struct Mfma16;
template <>
struct Mfma16<double> {
    typedef double v4 __attribute__((ext_vector_type(4)));
    __device__ static v4 step(double a, double b, v4 c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
    __device__ static int row(int kq, int r) { return kq + 4 * r; }   // tile row of register r
};
template <>
struct Mfma16<float> {
    typedef float v4 __attribute__((ext_vector_type(4)));
    __device__ static v4 step(float a, float b, v4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
    __device__ static int row(int kq, int r) { return 4 * kq + r; }
};

template <typename T>
struct PlaneArgs {
    const int4 *tiles;
    const T *wf, *wu;
    const int2 *kf, *ku;
    int nx, bcx[2], bcy[2], N;   // bcy: of a piece (walls in a batch)
    int fx, fy, hx, hy;          // reach of the FMT and attraction stencils
    int wr, wld, ar, ald;        // LDS rows and row lengths of the density window and of each adjoint window
    CompConsts cc;
    int func, nwall, rows, att;  // rows: write the rho-bar and mean-field rows; att: attraction
    const double *mu_row;        // [N] chemical-potential term of the node's piece (batches)
    const double *rho, *mul;     // densities or direction, optional factor
    const unsigned char *zero, *elzero;
    const double *in_rb, *sub_rb, *in_mf, *sub_mf;
    double *out_rb, *out_mf;
    const double *x_rb, *dn_rb, *x_rho, *in_rho, *el_mf, *vext, *add;
    const T *adj;                // adjoint fields at the nodes (Schur products)
    T *adj_out;
    double *out_el;
    double *ss;
    const int *done, *pore_of;
};

// code (0: node, -1: bulk, -2: wall) of column x and row y of a piece of ny rows starting at node row r0,
// in the order and with the codes of map_pad
__device__ inline int plane_map(const int *bcx, const int *bcy, int nx, int ny, int r0, int x, int y, int &src, int &refl)
{
    refl = 0;
    if (x < 0 || x >= nx) {
        const int b = bcx[x < 0 ? 0 : 1];
        if (b == TMI_IN_BULK) return -1;
        if (b == TMI_IN_WALL) return -2;
        if (b == TMI_PERIODIC) {
            x += x < 0 ? nx : -nx;
            if (x < 0 || x >= nx) return -2;   // columns past a ragged tile's last output
        } else {
            refl |= 1;
            const int side = x < 0 ? 0 : 1;
            x = side ? 2 * (nx - 1) - x : -x;
            if (x < 0 || x >= nx) return bcx[1 - side] == TMI_IN_BULK ? -1 : -2;
        }
    }
    if (y < 0 || y >= ny) {
        const int b = bcy[y < 0 ? 0 : 1];
        if (b == TMI_IN_BULK) return -1;
        if (b == TMI_IN_WALL) return -2;
        if (b == TMI_PERIODIC) {
            y += y < 0 ? ny : -ny;
            if (y < 0 || y >= ny) return -2;
        } else {
            refl |= 2;
            const int side = y < 0 ? 0 : 1;
            y = side ? 2 * (ny - 1) - y : -y;
            if (y < 0 || y >= ny) return bcy[1 - side] == TMI_IN_BULK ? -1 : -2;
        }
    }
    src = x + (r0 + y) * nx;
    return 0;
}

// rows of a window of `rows` x `cols` values around the tile (reach gx, gy), zeros past them up to whole
// LDS rows; value(code, src, refl, at) writes the position's values at LDS offset at
template <int NT, typename F>
__device__ inline void plane_window(const int *bcx, const int *bcy, int nx, const int4 &t, int gx, int gy, int lds_rows, int ld,
                                    F &&value)
{
    const int cols = 16 + 2 * gx, rows = 16 + 2 * gy;
    for (int e = threadIdx.x; e < lds_rows * ld; e += NT) {
        const int r = e / ld, c = e - r * ld;
        int src = 0, refl = 0, code = -2;
        if (r < rows && c < cols) code = plane_map(bcx, bcy, nx, t.w - t.z, t.z, t.x - gx + c, t.y - t.z - gy + r, src, refl);
        value(code, src, refl, e);
    }
}

// one Toeplitz chain: offsets dx0, dx0 + ddx, ... < ndx of one weight table over one LDS window
template <typename T>
__device__ inline void plane_chain(const T *win, int ld, const T *__restrict__ w, int wlen, const int2 *__restrict__ kr,
                                   int dx0, int ddx, int ndx, int lo, int kq, typename Mfma16<T>::v4 &acc)
{
    for (int dx = dx0; dx < ndx; dx += ddx) {
        const int2 k = kr[dx];
        const T *a = w + (size_t)dx * wlen + 15 + kq - lo;
        const T *b = win + kq * ld + dx + lo;
#pragma unroll 4
        for (int k0 = k.x; k0 < k.y; k0 += 4) acc = Mfma16<T>::step(a[k0], b[k0 * ld], acc);
    }
}

template <typename T>
__device__ inline void plane_put(T *tile, const typename Mfma16<T>::v4 &acc, int lo, int kq)
{
#pragma unroll
    for (int r = 0; r < 4; ++r) tile[16 * Mfma16<T>::row(kq, r) + lo] = acc[r];
}

__device__ inline void plane_rb(const double *__restrict__ rb, size_t N, int i, double (&v)[8])
{
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = rb[(size_t)q * N + i];
}

// adjoint fields A, B_x, B_y, S3 of one component from the rho-bar values r (solution order; LINEAR: and dr)
template <bool LINEAR>
__device__ inline void plane_adjoint(const CompConsts &cc, int func, const double (&r)[8], const double (&dr)[8],
                                     double (&out)[4])
{
    const double n[8] = {r[3], r[2], r[1], r[0], r[6], r[7], r[4], r[5]};
    double o[8];
    if constexpr (LINEAR) {
        const double dn[8] = {dr[3], dr[2], dr[1], dr[0], dr[6], dr[7], dr[4], dr[5]};
        fmt_hvp<2>(func, n, dn, o);
    } else {
        fmt_dphi<2>(func, n, o);
    }
    out[0] = o[0] * cc.i4pirsq[0] + o[1] * cc.i4pir[0] + o[2];
    out[1] = o[4] * cc.i4pir[0] + o[6];
    out[2] = o[5] * cc.i4pir[0] + o[7];
    out[3] = o[3];
}

// true when every node of the tile belongs to a finished piece
__device__ inline bool plane_done(const int *done, const int *pore_of, int nx, const int4 &t)
{
    return done && done[pore_of ? pore_of[t.z * nx] : 0];
}

// MODE 0: residual, 1: Jacobian-vector product, 2: second half of a Schur product (adjoint fields given)
template <typename T, int MODE, int NW>
__global__ __launch_bounds__(64 * NW) void k_plane(PlaneArgs<T> a)
{
    typedef typename Mfma16<T>::v4 v4;
    constexpr int NT = 64 * NW, NM = NW / 2, NR = NW / 4;   // waves: attraction, rho-bar, Euler-Lagrange (NR each)
    extern __shared__ __attribute__((aligned(32))) char smem_raw[];
    T *win = reinterpret_cast<T *>(smem_raw);               // [wr][wld]
    T *adj = win + (a.rho ? a.wr * a.wld : 0);              // [4][ar][ald]
    const int4 t = a.tiles[blockIdx.x];
    if (MODE == 2 && plane_done(a.done, a.pore_of, a.nx, t)) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lo = lane & 15, kq = lane >> 4;
    const size_t N = a.N;
    const bool el = a.out_el != nullptr;
    if (a.rho)
        plane_window<NT>(a.bcx, a.bcy, a.nx, t, a.hx, a.hy, a.wr, a.wld, [&](int code, int src, int, int at) {
            double v = code == -1 && MODE == 0 ? a.cc.rho_b[0] : 0.0;
            if (code == 0) {
                const double rv = a.rho[src], m = a.mul ? a.mul[src] : 1.0;
                v = a.zero[src] ? 0.0 : rv * m;
            }
            win[at] = (T)v;
        });
    if (el) {
        const int an = a.ar * a.ald;
        plane_window<NT>(a.bcx, a.bcy, a.nx, t, a.fx, a.fy, a.ar, a.ald, [&](int code, int src, int refl, int at) {
            T v[4] = {(T)0, (T)0, (T)0, (T)0};
            if (code == 0) {
                if constexpr (MODE == 2) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) v[q] = a.adj[(size_t)q * N + src];
                } else {
                    double r[8], dr[8], o[4];
                    plane_rb(a.x_rb, N, src, r);
                    if constexpr (MODE == 1) plane_rb(a.dn_rb, N, src, dr);
                    plane_adjoint<MODE == 1>(a.cc, a.func, r, dr, o);
#pragma unroll
                    for (int q = 0; q < 4; ++q) v[q] = (T)o[q];
                }
                if (refl & 1) v[1] = -v[1];
                if (refl & 2) v[2] = -v[2];
            } else if (code == -1 && MODE == 0) {
                v[0] = (T)a.cc.Ab[0];
                v[3] = (T)a.cc.S3b;
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) adj[q * an + at] = v[q];
        });
    }
    __syncthreads();
    v4 acc[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) acc[q] = (v4){(T)0, (T)0, (T)0, (T)0};
    const int nfx = 2 * a.fx + 1, wfl = 2 * a.fy + kPlanePad;
    if (wave < NM) {
        if (a.rho && a.att)
            plane_chain<T>(win, a.wld, a.wu, 2 * a.hy + kPlanePad, a.ku, wave, NM, 2 * a.hx + 1, lo, kq, acc[0]);
    } else if (wave < NM + NR) {
        if (a.rho && a.rows) {   // the FMT stencils' window inside the density window
            const T *w0 = win + (a.hy - a.fy) * a.wld + (a.hx - a.fx);
#pragma unroll
            for (int q = 0; q < 4 / NR; ++q) {
                const int s = (wave - NM) + q * NR;
                plane_chain<T>(w0, a.wld, a.wf + (size_t)s * nfx * wfl, wfl, a.kf, 0, 1, nfx, lo, kq, acc[q]);
            }
        }
    } else if (el) {
#pragma unroll
        for (int q = 0; q < 4 / NR; ++q) {   // field A: delta, B_x: delta x, B_y: delta y, S3: theta
            const int f = (wave - NM - NR) + q * NR, s = f == 3 ? 0 : f + 1;
            plane_chain<T>(adj + f * a.ar * a.ald, a.ald, a.wf + (size_t)s * nfx * wfl, wfl, a.kf, 0, 1, nfx, lo, kq, acc[q]);
        }
    }
    __syncthreads();
    // partial tiles over the windows: attraction [NM][256], rho-bar sums [4][256], Euler-Lagrange fields [4][256]
    T *pm = reinterpret_cast<T *>(smem_raw), *pr = pm + NM * 256, *pe = pr + 4 * 256;
    if (wave < NM) {
        plane_put<T>(pm + wave * 256, acc[0], lo, kq);
    } else if (wave < NM + NR) {
#pragma unroll
        for (int q = 0; q < 4 / NR; ++q) plane_put<T>(pr + ((wave - NM) + q * NR) * 256, acc[q], lo, kq);
    } else {
#pragma unroll
        for (int q = 0; q < 4 / NR; ++q) plane_put<T>(pe + ((wave - NM - NR) + q * NR) * 256, acc[q], lo, kq);
    }
    __syncthreads();
    // rows: Euler-Lagrange, then the 8 rho-bar rows, then the mean-field row; 4 waves per row
    double ssq = 0.0;
    const bool has_mf = a.rho && a.att;
    const int n_out = 1 + (a.rows ? 8 + (has_mf ? 1 : 0) : 0);
    for (int e = tid; e < n_out * 256; e += NT) {
        const int row = e >> 8, p = e & 255, x = t.x + (p & 15), y = t.y + (p >> 4);
        if (x >= a.nx || y >= t.w) continue;
        const int i = x + y * a.nx;
        T mf = 0;
        if (has_mf && (row == 9 || (MODE == 2 && row == 0)))
            for (int w = 0; w < NM; ++w) mf += pm[w * 256 + p];
        double v;
        if (row == 0) {
            if (!el) continue;
            const double in = a.in_rho ? a.in_rho[i] * (a.mul ? a.mul[i] : 1.0) : 0.0;
            if (a.elzero[i]) {
                v = in;
            } else {
                v = (double)(pe[3 * 256 + p] + pe[p] - pe[256 + p] - pe[2 * 256 + p]);
                const double xv = a.x_rho[i];
                if constexpr (MODE == 0) {
                    v += log(xv) + (a.mu_row ? a.mu_row[i] : a.cc.mu[0]);
                    if (a.nwall > 0) v += a.vext[i];
                } else {
                    if (a.in_rho) v += in / xv;
                }
                if constexpr (MODE == 2)
                    v += (double)mf;
                else if (a.el_mf)
                    v += a.el_mf[i];
            }
            if (a.add) v += a.add[i];
            a.out_el[i] = v;
        } else if (row < 9) {
            const int q = row - 1;   // n3 n2 n1 n0 nv2_x nv2_y nv1_x nv1_y from theta, delta, delta x, delta y
            const int s = q == 0 ? 0 : (q < 4 ? 1 : 2 + ((q - 4) & 1));
            const T sum = pr[s * 256 + p];
            v = (double)(q == 2 || q > 5 ? (T)a.cc.i4pir[0] * sum : (q == 3 ? (T)a.cc.i4pirsq[0] * sum : sum));
            const size_t at = (size_t)q * N + i;
            if (a.in_rb) v -= a.in_rb[at];
            if (a.sub_rb) v -= a.sub_rb[at];
            a.out_rb[at] = v;
        } else {
            v = (double)mf;
            if (a.in_mf) v -= a.in_mf[i];
            if (a.sub_mf) v -= a.sub_mf[i];
            a.out_mf[i] = v;
        }
        ssq += v * v;
    }
    if (a.ss) {
        __shared__ double sh[NW];
        for (int o = 32; o > 0; o >>= 1) ssq += __shfl_down(ssq, o, 64);
        if (lane == 0) sh[wave] = ssq;
        __syncthreads();
        if (tid == 0) {
            double s = 0.0;
            for (int w = 0; w < NW; ++w) s += sh[w];
            a.ss[blockIdx.x] = s;
        }
    }
}

// First half of a Schur product: rho-bar sums of the direction (FMT reach), the Hessian product at the
// nodes, the adjoint fields into adj_out [4][N].  8 waves: each sum split over two (even and odd dx).
template <typename T>
__global__ __launch_bounds__(512) void k_plane_schur(PlaneArgs<T> a)
{
    typedef typename Mfma16<T>::v4 v4;
    extern __shared__ __attribute__((aligned(32))) char smem_raw[];
    T *win = reinterpret_cast<T *>(smem_raw);   // [ar][ald]
    __shared__ T part[8][256];
    const int4 t = a.tiles[blockIdx.x];
    if (plane_done(a.done, a.pore_of, a.nx, t)) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lo = lane & 15, kq = lane >> 4;
    const size_t N = a.N;
    plane_window<512>(a.bcx, a.bcy, a.nx, t, a.fx, a.fy, a.ar, a.ald, [&](int code, int src, int, int at) {
        double v = 0.0;
        if (code == 0) {
            const double rv = a.rho[src], m = a.mul ? a.mul[src] : 1.0;
            v = a.zero[src] ? 0.0 : rv * m;
        }
        win[at] = (T)v;
    });
    const int x = t.x + (tid & 15), y = t.y + ((tid & 255) >> 4), i = x + y * a.nx;
    const bool live = tid < 256 && x < a.nx && y < t.w;
    double r[8];
    if (live) plane_rb(a.x_rb, N, i, r);
    __syncthreads();
    const int nfx = 2 * a.fx + 1, wfl = 2 * a.fy + kPlanePad;
    v4 acc = (v4){(T)0, (T)0, (T)0, (T)0};
    plane_chain<T>(win, a.ald, a.wf + (size_t)(wave >> 1) * nfx * wfl, wfl, a.kf, wave & 1, 2, nfx, lo, kq, acc);
    plane_put<T>(part[wave], acc, lo, kq);
    __syncthreads();
    if (!live) return;
    T s[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) s[q] = part[2 * q][tid] + part[2 * q + 1][tid];
    const T f1 = (T)a.cc.i4pir[0], f0 = (T)a.cc.i4pirsq[0];
    const double dr[8] = {(double)s[0], (double)s[1], (double)(f1 * s[1]), (double)(f0 * s[1]),
                          (double)s[2], (double)s[3], (double)(f1 * s[2]), (double)(f1 * s[3])};
    double o[4];
    plane_adjoint<true>(a.cc, a.func, r, dr, o);
#pragma unroll
    for (int q = 0; q < 4; ++q) a.adj_out[(size_t)q * N + i] = (T)o[q];
}

// LDS row length for `cols` values: the four rows of an operand read (32 banks each) should fall on
// different halves of the 64 banks
template <typename T>
int plane_ld(int cols)
{
    int best = cols, cost = 1 << 30;
    for (int ld = cols; ld < cols + 16; ++ld) {
        int hit[64] = {};
        for (int r = 0; r < 4; ++r)
            for (int j = 0; j < 16 * (int)sizeof(T) / 4; ++j) ++hit[(r * ld * (int)sizeof(T) / 4 + j) & 63];
        int worst = 0;
        for (int b : hit) worst = std::max(worst, b);
        if (worst < cost) cost = worst, best = ld;
        if (cost <= (int)sizeof(T) / 4) break;
    }
    return best;
}

struct PlaneShape {
    int wr, wld, ar, ald;
    size_t elems, schur;   // LDS values of k_plane and of k_plane_schur
};
template <typename T>
PlaneShape plane_shape(const PlanePlan &L)
{
    PlaneShape s;
    auto rows = [](int g) { return (16 + 2 * g + 3) & ~3; };
    s.wr = std::max(rows(L.hy), L.hy - L.fy + rows(L.fy));   // whole steps of the FMT sums inside it too
    s.wld = plane_ld<T>(16 + 2 * L.hx);
    s.ar = rows(L.fy);
    s.ald = plane_ld<T>(16 + 2 * L.fx);
    s.schur = (size_t)s.ar * s.ald;
    s.elems = std::max((size_t)s.wr * s.wld + 4 * s.schur, (size_t)16 * 256);
    return s;
}
constexpr size_t kPlaneTwo = 80 * 1024;   // LDS of a workgroup of which a CU holds two
inline int plane_waves_for(size_t lds) { return lds <= kPlaneTwo - 1024 ? 8 : 16; }

template <typename T>
PlaneArgs<T> plane_args(const Problem &P, const PlaneShape &s)
{
    const PlanePlan &L = *P.plane;
    PlaneArgs<T> a{};
    a.tiles = L.tiles;
    if constexpr (sizeof(T) == 8) {
        a.wf = L.wf;
        a.wu = L.wu;
    } else {
        a.wf = L.wf32;
        a.wu = L.wu32;
    }
    a.kf = L.kf;
    a.ku = L.ku;
    a.nx = P.p.nx[0];
    a.N = P.N;
    for (int e = 0; e < 2; ++e) {
        a.bcx[e] = P.p.bc[0][e];
        a.bcy[e] = P.npores > 0 ? TMI_IN_WALL : P.p.bc[1][e];
    }
    a.fx = L.fx;
    a.fy = L.fy;
    a.hx = L.hx;
    a.hy = L.hy;
    a.wr = s.wr;
    a.wld = s.wld;
    a.ar = s.ar;
    a.ald = s.ald;
    a.cc = make_consts(P);
    a.func = P.p.type_func;
    a.nwall = P.p.nwall;
    a.att = P.nmf > 0 ? 1 : 0;
    a.mu_row = P.d_mu;
    a.zero = P.d_zero;
    a.elzero = P.d_elzero;
    a.vext = P.d_vext;
    a.pore_of = P.d_pore_of;
    return a;
}

template <typename T, int MODE>
void plane_launch(const Problem &P, const PlaneShape &s, const PlaneArgs<T> &a, hipStream_t st)
{
    const size_t lds = s.elems * sizeof(T);
    auto go = [&](auto kernel, int nw) {
        if (lds > 64 * 1024)
            TMI_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                              (int)lds));
        hipLaunchKernelGGL(kernel, dim3((unsigned)P.plane->ntiles), dim3(64 * nw), lds, st, a);
    };
    if (plane_waves_for(lds) == 8)
        go(k_plane<T, MODE, 8>, 8);
    else
        go(k_plane<T, MODE, 16>, 16);
    TMI_HIP_CHECK(hipGetLastError());
}

}  // namespace

bool plane_on(const Problem &P) { return P.plane && P.plane->on; }
bool plane_built(const Problem &P) { return P.plane != nullptr; }
void plane_set(Problem &P, bool on)
{
    if (P.plane) P.plane->on = on;
}
void plane_set_rows(Problem &P, bool on)
{
    if (P.plane) P.plane->rows = on;
}
bool plane_rows(const Problem &P) { return P.plane && P.plane->rows; }
int plane_waves(const Problem &P) { return P.plane ? plane_waves_for(plane_shape<double>(*P.plane).elems * sizeof(double)) : 0; }
long long plane_partials(const Problem &P) { return plane_on(P) ? P.plane->ntiles : 0; }

void plane_free(Problem &P)
{
    PlanePlan *L = P.plane;
    if (!L) return;
    for (void *q : {(void *)L->tiles, (void *)L->wf, (void *)L->wu, (void *)L->wf32, (void *)L->wu32, (void *)L->kf, (void *)L->ku,
                    L->adj})
        (void)hipFree(q);
    delete L;
    P.plane = nullptr;
}

// Tables and tiles of a one-component 2D problem whose windows fit a CU's LDS (TMI_PLANE2D=0, or a
// switch that asks for one of the separate kernels: none; 2: without timing it against the FFT forms)
void plane_setup(Problem &P)
{
    if (P.p.ndim != 2 || P.p.ncomp != 1) return;
    for (const char *name : {"TMI_PLANE2D", "TMI_MF2D_MFMA", "TMI_RB2D_MFMA"}) {
        const char *env = std::getenv(name);
        if (env && std::string(env) == "0") return;
    }
    const char *kern = std::getenv("TMI_STENCIL_KERNEL");
    if (kern && std::string(kern) == "gather") return;
    auto *L = new PlanePlan();
    P.plane = L;
    try {
        auto reach = [&](const HostStencil &hs, int &gx, int &gy) {
            for (int k = 0; k < hs.L; ++k) {
                gx = std::max(gx, std::abs(hs.off[3 * (size_t)k]));
                gy = std::max(gy, std::abs(hs.off[3 * (size_t)k + 1]));
            }
        };
        const HostStencil &th = P.hs[TMI_THETA][0], &de = P.hs[TMI_DELTA][0], &ua = P.hs[TMI_UATT][0];
        reach(th, L->fx, L->fy);
        reach(de, L->fx, L->fy);
        L->hx = L->fx;
        L->hy = L->fy;
        if (P.nmf) reach(ua, L->hx, L->hy);
        int dev = 0, lds = 0;
        TMI_HIP_CHECK(hipGetDevice(&dev));
        TMI_HIP_CHECK(hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
        if (plane_shape<double>(*L).elems * sizeof(double) + 512 > (size_t)lds) {
            plane_free(P);
            return;
        }
        // a column's weights at [15 + dy + g], and the window rows its products need
        auto tables = [&](int gx, int gy, int nsum, auto &&fill, double **wd, float **wf, int2 **kr) {
            const int ndx = 2 * gx + 1, len = 2 * gy + kPlanePad;
            std::vector<double> w((size_t)nsum * ndx * len, 0.0);
            fill([&](int s, int dx, int dy) -> double & { return w[((size_t)s * ndx + (dx + gx)) * len + 15 + dy + gy]; });
            std::vector<int2> k(ndx, int2{0, 0});
            for (int dx = 0; dx < ndx; ++dx) {
                int lo = 1 << 30, hi = -1;
                for (int s = 0; s < nsum; ++s)
                    for (int j = 0; j <= 2 * gy; ++j)
                        if (w[((size_t)s * ndx + dx) * len + 15 + j] != 0.0) {
                            lo = std::min(lo, j);
                            hi = std::max(hi, j);
                        }
                if (hi >= 0) k[dx] = int2{lo & ~3, hi + 16};   // rows k with lo <= k - i <= hi for some i in [0, 16)
            }
            std::vector<float> f(w.begin(), w.end());
            TMI_HIP_CHECK(hipMalloc((void **)wd, w.size() * sizeof(double)));
            TMI_HIP_CHECK(hipMalloc((void **)wf, f.size() * sizeof(float)));
            TMI_HIP_CHECK(hipMalloc((void **)kr, k.size() * sizeof(int2)));
            TMI_HIP_CHECK(hipMemcpy(*wd, w.data(), w.size() * sizeof(double), hipMemcpyHostToDevice));
            TMI_HIP_CHECK(hipMemcpy(*wf, f.data(), f.size() * sizeof(float), hipMemcpyHostToDevice));
            TMI_HIP_CHECK(hipMemcpy(*kr, k.data(), k.size() * sizeof(int2), hipMemcpyHostToDevice));
        };
        tables(L->fx, L->fy, 4, [&](auto &&at) {
            for (int k = 0; k < th.L; ++k) at(0, th.off[3 * (size_t)k], th.off[3 * (size_t)k + 1]) += th.w[k];
            for (int k = 0; k < de.L; ++k) {
                const int *o = &de.off[3 * (size_t)k];
                at(1, o[0], o[1]) += de.w[k];
                for (int d = 0; d < 2; ++d) at(2 + d, o[0], o[1]) += de.w[k] * ((double)o[d] * P.p.dx[d] * P.bulk.inv_rad[0]);
            }
        }, &L->wf, &L->wf32, &L->kf);
        if (P.nmf)
            tables(L->hx, L->hy, 1, [&](auto &&at) {
                for (int k = 0; k < ua.L; ++k) at(0, ua.off[3 * (size_t)k], ua.off[3 * (size_t)k + 1]) += ua.w[k];
            }, &L->wu, &L->wu32, &L->ku);
        // tiles, piece by piece
        std::vector<int4> tiles;
        const int nx = P.p.nx[0];
        auto piece = [&](int r0, int r1) {
            for (int y = r0; y < r1; y += 16)
                for (int x = 0; x < nx; x += 16) tiles.push_back(int4{x, y, r0, r1});
        };
        if (P.npores > 0)
            for (int q = 0; q < P.npores; ++q) piece(P.pore_off[q] / nx, P.pore_off[q + 1] / nx);
        else
            piece(0, P.p.nx[1]);
        L->ntiles = (int)tiles.size();
        TMI_HIP_CHECK(hipMalloc((void **)&L->tiles, tiles.size() * sizeof(int4)));
        TMI_HIP_CHECK(hipMemcpy(L->tiles, tiles.data(), tiles.size() * sizeof(int4), hipMemcpyHostToDevice));
        TMI_HIP_CHECK(hipMalloc(&L->adj, (size_t)4 * P.N * sizeof(double)));
    } catch (...) {
        plane_free(P);
        throw;
    }
}

template <typename T>
void plane_rows_el(Problem &P, bool linear, const double *rho, const double *in_rb, const double *sub_rb, double *out_rb,
                   const double *in_mf, const double *sub_mf, double *out_mf, const double *x, const double *dn_rb,
                   const double *in_rho, const double *el_mf, const double *add, double *out_el, hipStream_t s, double *ss)
{
    const PlaneShape sh = plane_shape<T>(*P.plane);
    PlaneArgs<T> a = plane_args<T>(P, sh);
    const size_t N = P.N;
    a.rho = rho;
    a.rows = rho ? 1 : 0;
    a.in_rb = in_rb;
    a.sub_rb = sub_rb;
    a.out_rb = out_rb;
    a.in_mf = in_mf;
    a.sub_mf = sub_mf;
    a.out_mf = out_mf;
    if (out_el) {
        a.x_rb = x + (size_t)P.iu_rb * N;
        a.x_rho = x + (size_t)P.iu_rho * N;
    }
    a.dn_rb = dn_rb;
    a.in_rho = in_rho;
    a.el_mf = el_mf;
    a.add = add;
    a.out_el = out_el;
    a.ss = ss;
    if (linear)
        plane_launch<T, 1>(P, sh, a, s);
    else
        plane_launch<T, 0>(P, sh, a, s);
}
template void plane_rows_el<double>(Problem &, bool, const double *, const double *, const double *, double *,
                                    const double *, const double *, double *, const double *, const double *,
                                    const double *, const double *, const double *, double *, hipStream_t, double *);
template void plane_rows_el<float>(Problem &, bool, const double *, const double *, const double *, double *,
                                   const double *, const double *, double *, const double *, const double *,
                                   const double *, const double *, const double *, double *, hipStream_t, double *);

template <typename T>
void plane_schur(Problem &P, const double *x, const double *x2, const double *mul, double *y2, const int *done, hipStream_t s)
{
    const PlaneShape sh = plane_shape<T>(*P.plane);
    PlaneArgs<T> a = plane_args<T>(P, sh);
    const size_t N = P.N;
    a.rho = x2;
    a.mul = mul;
    a.x_rb = x + (size_t)P.iu_rb * N;
    a.x_rho = x + (size_t)P.iu_rho * N;
    a.in_rho = x2;
    a.adj = a.adj_out = (T *)P.plane->adj;
    a.out_el = y2;
    a.done = done;
    hipLaunchKernelGGL(k_plane_schur<T>, dim3((unsigned)P.plane->ntiles), dim3(512), sh.schur * sizeof(T), s, a);
    plane_launch<T, 2>(P, sh, a, s);
}
template void plane_schur<double>(Problem &, const double *, const double *, const double *, double *, const int *,
                                  hipStream_t);
template void plane_schur<float>(Problem &, const double *, const double *, const double *, double *, const int *,
                                 hipStream_t);

}  // namespace tmi
