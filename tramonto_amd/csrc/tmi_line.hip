// The stencil rows of 1D problems and batches of 1D pores in one launch.
//
// A 1D fill is six dependent-looking launches (density halo, rho-bar rows, mean-field rows,
// pointwise derivatives, adjoint halo, Euler-Lagrange rows) of a few microseconds each, and its
// kernels leave most SIMDs with one wave that waits for its own loads.  Here one workgroup owns TN
// consecutive padded positions, keeps the densities and the adjoint fields of its span (halos
// included) in LDS, and its waves share out the stencil sums: one (stencil, component, span) sum per
// wave at a time, so that the long attraction sums and the short FMT ones run side by side.
//  * Residual and Jacobian-vector product: the rows and the Euler-Lagrange sums depend on the
//    inputs alone, so both run in the same pass.
//  * Schur product (CHAIN): the rho-bar sums are formed on the span and its FMT halo (recomputed by
//    the neighbours), become adjoint fields in LDS, and feed the Euler-Lagrange sums: no row leaves
//    the chip.
// Each lane owns B consecutive outputs, so every LDS value read feeds B multiply-adds per stencil
// against weights in scalar registers.  Small problems are bound by latency and take B = 1 and 64
// positions a workgroup, which puts 401 nodes on 7 CUs instead of 1; large ones are bound by the FP64
// multiply-adds and LDS reads of the sums (256 pores, 221,378 nodes: 0.8 GFLOP, 14 us at the FP64
// peak with the halo's recomputed sums) and take B = 4.
// Measured, FP64: residual kernels of the 401-node hard wall 40 -> 9 us (with its sum of squares),
// Schur product of 256 pores 87 -> 34 us.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "tmi_device.hpp"
#include "tmi_fmt.hpp"
#include "tmi_internal.hpp"

namespace tmi {

// Positions per lane by the span: 64 B positions a workgroup, so that small problems still reach many
// CUs and large ones read LDS once per 4 outputs.
int line_lanes(const Problem &P)
{
    const long long span = (long long)P.pad_u.P[0] - 2LL * P.pad_u.h[0];
    return span <= 64LL * 256 ? 1 : (span <= 128LL * 256 ? 2 : 4);
}

namespace {

using namespace dev;

constexpr int kLineWaves = 8;
constexpr int kLineBlock = 64 * kLineWaves;
constexpr size_t kLineLds = 64 * 1024;   // dynamic LDS of a launch

template <typename T>
struct LineRow {
    const T *w, *wv;
    int lo0, L;
};

template <typename T>
struct LineArgs {
    Geo g;   // the density geometry; the adjoint fields use its positions too (its gaps are at least the FMT halo)
    LineRow<T> th[kNC], de[kNC], u[kNC * kNC];
    CompConsts cc;
    int TN, hr, hf;   // positions per workgroup, density halo in LDS, FMT halo
    int rho_ld, rb_ld, mf_ld, adj_ld, chain_ld;   // LDS row lengths; CHAIN: of the densities' and adjoint fields' shared space
    int nmf, func, nwall;
    const double *rho, *mul;   // densities or direction [C][N] (null: no rows), optional factor
    const unsigned char *zero, *elzero;
    const double *in_rb, *sub_rb, *in_mf, *sub_mf;
    double *out_rb, *out_mf;
    const double *x_rb, *dn_rb, *x_rho, *in_rho, *el_mf, *vext, *add;
    double *out_el;            // null: no Euler-Lagrange rows
    double *ss;                // optional: the workgroup's sum of squares of the rows written
    const int *done, *pore_of; // optional: skip a workgroup all of whose pores (null pore_of: the problem) are done
};

// code and source node of padded position q, which may lie outside the padded copy (map_pad in 1D)
__device__ inline int line_map(const Geo &g, int q, int &src, int &refl)
{
    refl = 0;
    if (g.pad_node) {
        src = (q >= 0 && q < (int)g.np) ? g.pad_node[q] : -1;
        return src >= 0 ? 0 : -2;
    }
    const int n = g.nx[0];
    int v = q - g.h[0];
    if (v >= 0 && v < n) {
        src = v;
        return 0;
    }
    const int side = v < 0 ? 0 : 1, b = g.bc[0][side];
    if (b == TMI_IN_BULK) return -1;
    if (b == TMI_IN_WALL) return -2;
    if (b == TMI_PERIODIC) {
        v += side ? -n : n;
        if (v < 0 || v >= n) return -2;   // further than one period: read by no output
    } else {
        refl = 1;
        v = side ? 2 * (n - 1) - v : -v;
        if (v < 0 || v >= n) return g.bc[0][1 - side] == TMI_IN_BULK ? -1 : -2;
    }
    src = v;
    return 0;
}

constexpr int kLineStep = 8;   // positions read per step of a stencil sum

// kLineStep LDS values from a multiple of B
template <typename T, int B>
__device__ __forceinline__ void lds_read(const T *p, T (&v)[kLineStep])
{
    if constexpr (B > 1) {
        typedef T VB __attribute__((ext_vector_type(B)));
#pragma unroll
        for (int q = 0; q < kLineStep / B; ++q) {
            const VB t = reinterpret_cast<const VB *>(p)[q];
#pragma unroll
            for (int i = 0; i < B; ++i) v[q * B + i] = t[i];
        }
    } else {
#pragma unroll
        for (int i = 0; i < kLineStep; ++i) v[i] = p[i];
    }
}

// acc[s][b] += sum_j w_s[j] row[a0 + b + j] for NS weight rows of one stencil (row: LDS, a0: the
// wave's first position plus the stencil's first offset, lane_a: the lane's, a multiple of B).  With
// B = 1 (few waves on the chip) the next step's values and weights are requested before this step's
// multiply-adds, so a wave does not wait for each of its LDS and scalar loads in turn; otherwise the
// CU's other waves cover the wait and the registers buy more of them.
template <typename T, int B, int NS>
__device__ __forceinline__ void line_sum(const T *row, int a0, int lane_a, const T *__restrict__ w0,
                                         const T *__restrict__ w1, int L, T (&acc)[NS][B])
{
    constexpr int K = kLineStep, NW = K + B - 1;
    const int sh = a0 & (B - 1);   // wave-uniform: reads start on a multiple of B
    const T *src = row + (a0 - sh) + lane_a;
    const int back = kRowPad - sh - (B - 1);
    // constant address space: wave-uniform weights go through the scalar cache into scalar registers
    typedef const T __attribute__((address_space(4))) *ConstW;
    const ConstW w[2] = {(ConstW)(w0 + back), (ConstW)((NS > 1 ? w1 : w0) + back)};
    const int nk = (L + sh + B - 1 + K - 1) / K;
    T v[2][K], wk[2][NS][NW];
    auto load = [&](int k, int p) {
        lds_read<T, B>(src + k * K, v[p]);
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int j = 0; j < NW; ++j) wk[p][s][j] = w[s][k * K + j];
    };
    auto fma_step = [&](int p) {
#pragma unroll
        for (int i = 0; i < K; ++i)
#pragma unroll
            for (int s = 0; s < NS; ++s)
#pragma unroll
                for (int b = 0; b < B; ++b) acc[s][b] += wk[p][s][i - b + B - 1] * v[p][i];
    };
    if constexpr (B == 1) {
        load(0, 0);
        for (int k = 0; k < nk; k += 2) {   // a step past the last reads zero weights and the row's slack
            load(k + 1, 1);
            fma_step(0);
            load(k + 2, 0);
            fma_step(1);
        }
    } else {
        for (int k = 0; k < nk; ++k) {
            load(k, 0);
            fma_step(0);
        }
    }
}

// the rho-bar rows of node src (solution order)
__device__ inline void line_rb(const double *__restrict__ rb, size_t N, int src, double (&v)[6])
{
#pragma unroll
    for (int q = 0; q < 6; ++q) v[q] = rb[(size_t)q * N + src];
}

// adjoint fields A_c, B_c (c < C), S3 from the rho-bar values r (LINEAR: and the direction's dr)
template <typename T, bool LINEAR>
__device__ inline void line_adjoint(int C, const CompConsts &cc, int func, const double (&r)[6], const double (&dr)[6],
                                    int refl, T *out, int ld)
{
    const double n[6] = {r[3], r[2], r[1], r[0], r[5], r[4]};
    double o[6];
    if constexpr (LINEAR) {
        const double dn[6] = {dr[3], dr[2], dr[1], dr[0], dr[5], dr[4]};
        fmt_hvp<1>(func, n, dn, o);
    } else {
        fmt_dphi<1>(func, n, o);
    }
    for (int c = 0; c < C; ++c) {
        out[(2 * c) * ld] = (T)(o[0] * cc.i4pirsq[c] + o[1] * cc.i4pir[c] + o[2]);
        const T b = (T)(o[4] * cc.i4pir[c] + o[5]);
        out[(2 * c + 1) * ld] = refl ? -b : b;
    }
    out[2 * C * ld] = (T)o[3];
}

template <typename T, int B, bool CHAIN, bool LINEAR>
__global__ __launch_bounds__(kLineBlock, B == 1 ? 2 : 6) void k_line(LineArgs<T> a)
{
    extern __shared__ __attribute__((aligned(32))) char smem_raw[];
    const Geo &g = a.g;
    const int C = g.C, TN = a.TN, hf = a.hf, hr = a.hr;
    const size_t N = g.N;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int p0 = g.h[0] + (int)blockIdx.x * TN;   // first position of the span
    if (a.done) {
        int live = 0;
        for (int t = tid; t < TN; t += kLineBlock) {
            int src, refl;
            if (line_map(g, p0 + t, src, refl) == 0 && !a.done[a.pore_of ? a.pore_of[src] : 0]) live = 1;
        }
        if (!__syncthreads_or(live)) return;
    }
    const int rb_n = CHAIN ? TN + 2 * hf : TN, adj_n = TN + 2 * hf, ext = CHAIN ? hf : 0;
    T *rho = reinterpret_cast<T *>(smem_raw);               // [C][rho_ld]
    // CHAIN: the adjoint fields replace the densities once the sums are formed
    T *adj = CHAIN ? rho : rho + (a.rho ? C * a.rho_ld : 0);   // [2 C + 1][adj_ld]
    T *srb = CHAIN ? rho + a.chain_ld : adj + (a.out_el ? (2 * C + 1) * a.adj_ld : 0);   // [C][3][rb_ld]: theta, delta, vector delta
    T *smf = srb + (a.rho ? 3 * C * a.rb_ld : 0);           // [C][C][mf_ld]
    T *sel = CHAIN ? srb : smf + (a.rho && a.nmf ? C * C * a.mf_ld : 0);   // [C][3][mf_ld]
    // densities with their halo, by the last threads first (the adjoint fields take the first ones)
    if (a.rho) {
        for (int r = kLineBlock - 1 - tid; r < a.rho_ld; r += kLineBlock) {
            int src = 0, refl = 0, code = -2;
            if (r < TN + 2 * hr) code = line_map(g, p0 - hr + r, src, refl);
            for (int c = 0; c < C; ++c) {
                double v = code == -1 && !LINEAR ? a.cc.rho_b[c] : 0.0;
                if (code == 0) {   // every load unconditional: none waits for another
                    const size_t q = (size_t)c * N + src;
                    const double rv = a.rho[q], m = a.mul ? a.mul[q] : 1.0;
                    v = a.zero[q] ? 0.0 : rv * m;
                }
                rho[c * a.rho_ld + r] = (T)v;
            }
        }
    }
    // adjoint fields with their halo
    auto adjoint_halo = [&](int r, int code) {   // no node: bulk or wall values
        const bool bulk = code == -1 && !LINEAR;
        for (int c = 0; c < C; ++c) {
            adj[(2 * c) * a.adj_ld + r] = bulk ? (T)a.cc.Ab[c] : (T)0;
            adj[(2 * c + 1) * a.adj_ld + r] = (T)0;
        }
        adj[2 * C * a.adj_ld + r] = bulk ? (T)a.cc.S3b : (T)0;
    };
    if (!CHAIN && a.out_el) {
        for (int r = tid; r < a.adj_ld; r += kLineBlock) {
            int src = 0, refl = 0, code = -2;
            if (r < adj_n) code = line_map(g, p0 - hf + r, src, refl);
            if (code == 0) {
                double xr[6], dr[6];
                line_rb(a.x_rb, N, src, xr);
                if constexpr (LINEAR) line_rb(a.dn_rb, N, src, dr);
                line_adjoint<T, LINEAR>(C, a.cc, a.func, xr, dr, refl, adj + r, a.adj_ld);
            } else {
                adjoint_halo(r, code);
            }
        }
    }
    // Node inputs of this thread's first adjoint position (CHAIN) and first output row, with B = 1 requested
    // before the sums.  Output rows: the Euler-Lagrange rows, then the rho-bar rows, then the mean-field rows;
    // thread e takes position e mod TN of row e / TN.
    const int n_out = (a.out_el ? C : 0) + (!CHAIN && a.rho ? 6 + a.nmf : 0);
    struct AdjIn {
        int src, refl, code;
        double x[6];
    };
    auto adj_in = [&](int r) {
        AdjIn v;
        v.src = v.refl = 0;
        v.code = -2;
        if (r < adj_n) v.code = line_map(g, p0 - hf + r, v.src, v.refl);
        if (v.code == 0) line_rb(a.x_rb, N, v.src, v.x);
        return v;
    };
    struct RowIn {
        int i;   // node (< 0: none)
        unsigned char fixed;
        double x, in, sub, vext, mf, add, mu;
    };
    auto row_in = [&](int e) {
        RowIn v;
        v.i = -1;
        v.fixed = 0;
        v.x = 1.0;
        v.in = v.sub = v.vext = v.mf = v.add = v.mu = 0.0;
        const int row = e / TN, q = p0 + e - row * TN;
        int refl;
        if (row >= n_out || q >= g.P[0] - g.h[0] || line_map(g, q, v.i, refl) != 0) {
            v.i = -1;
            return v;
        }
        if (a.out_el && row < C) {
            const size_t at = (size_t)row * N + v.i;
            v.fixed = a.elzero[at];
            v.x = a.x_rho[at];
            if (a.in_rho) v.in = a.in_rho[at];
            if (a.mul) v.in *= a.mul[at];
            if (!LINEAR && a.nwall > 0) v.vext = a.vext[at];
            if (!CHAIN && a.el_mf) v.mf = a.el_mf[at];
            if (a.add) v.add = a.add[at];
            if constexpr (!LINEAR) v.mu = g.mu ? g.mu[at] : a.cc.mu[row];
        } else {
            const int r = row - (a.out_el ? C : 0);
            const size_t at = (size_t)(r < 6 ? r : r - 6) * N + v.i;
            const double *in = r < 6 ? a.in_rb : a.in_mf, *sub = r < 6 ? a.sub_rb : a.sub_mf;
            if (in) v.in = in[at];
            if (sub) v.sub = sub[at];
        }
        return v;
    };
    AdjIn ain;
    RowIn rin;
    if constexpr (B == 1) {
        if constexpr (CHAIN) ain = adj_in(tid);
        rin = row_in(tid);
    }
    __syncthreads();
    // stencil sums, one item per wave at a time, the longest first
    constexpr int W = 64 * B;
    const int nt = (TN + W - 1) / W, ntr = (rb_n + W - 1) / W;
    const int n_mf = a.rho && a.nmf ? C * C * nt : 0, n_rb = a.rho ? C * ntr : 0, n_el = !CHAIN && a.out_el ? C * nt : 0;
    auto put = [&](T *row, int t0, int n, const T (&v)[B]) {
#pragma unroll
        for (int b = 0; b < B; ++b)
            if (t0 + lane * B + b < n) row[t0 + lane * B + b] = v[b];
    };
    auto el_item = [&](int it) {   // three items per component and span: delta A, vector delta B, theta S3
        const int kind = it % 3, t = (it / 3) % nt, c = it / (3 * nt);
        const LineRow<T> st = kind == 2 ? a.th[c] : a.de[c];
        const T *row = adj + (kind == 2 ? 2 * C : 2 * c + kind) * a.adj_ld;
        T acc[1][B] = {};
        line_sum<T, B, 1>(row, t * W + hf + st.lo0, lane * B, kind == 1 ? st.wv : st.w, nullptr, st.L, acc);
        put(sel + (3 * c + kind) * a.mf_ld, t * W, TN, acc[0]);
    };
    for (int it = wave; it < n_mf + 2 * n_rb + 3 * n_el; it += kLineWaves) {
        if (it < n_mf) {
            const int t = it % nt, q = it / nt, c = q / C, cj = q - c * C;
            const LineRow<T> u = a.u[c + C * cj];
            T acc[1][B] = {};
            line_sum<T, B, 1>(rho + cj * a.rho_ld, t * W + hr + u.lo0, lane * B, u.w, nullptr, u.L, acc);
            put(smf + q * a.mf_ld, t * W, TN, acc[0]);
        } else if (it < n_mf + 2 * n_rb) {
            const int j = it - n_mf, th = j >= n_rb, q = th ? j - n_rb : j, t = q % ntr, c = q / ntr;
            if (th) {
                const LineRow<T> st = a.th[c];
                T acc[1][B] = {};
                line_sum<T, B, 1>(rho + c * a.rho_ld, t * W - ext + hr + st.lo0, lane * B, st.w, nullptr, st.L, acc);
                put(srb + (3 * c) * a.rb_ld, t * W, rb_n, acc[0]);
            } else {
                const LineRow<T> st = a.de[c];
                T acc[2][B] = {};
                line_sum<T, B, 2>(rho + c * a.rho_ld, t * W - ext + hr + st.lo0, lane * B, st.w, st.wv, st.L, acc);
                put(srb + (3 * c + 1) * a.rb_ld, t * W, rb_n, acc[0]);
                put(srb + (3 * c + 2) * a.rb_ld, t * W, rb_n, acc[1]);
            }
        } else {
            el_item(it - n_mf - 2 * n_rb);
        }
    }
    __syncthreads();
    // rho-bar value q (solution order) at index r of the sums
    auto rb_val = [&](int q, int r) {
        const int k = q == 0 ? 0 : (q < 4 ? 1 : 2);
        T v = 0;
        for (int c = 0; c < C; ++c) {
            const T sum = srb[(3 * c + k) * a.rb_ld + r];
            const T f = q == 2 || q == 5 ? (T)a.cc.i4pir[c] : (q == 3 ? (T)a.cc.i4pirsq[c] : (T)1);
            v += f * sum;
        }
        return (double)v;
    };
    if constexpr (CHAIN) {
        auto adj_out = [&](int r, const AdjIn &v) {
            // across a mirror the node's own sums; a mirror node outside the span serves no output here
            const int rs = v.refl ? v.src + g.h[0] - (p0 - hf) : r;
            if (v.code == 0 && rs >= 0 && rs < rb_n) {
                double dr[6];
#pragma unroll
                for (int q = 0; q < 6; ++q) dr[q] = rb_val(q, rs);
                line_adjoint<T, true>(C, a.cc, a.func, v.x, dr, v.refl, adj + r, a.adj_ld);
            } else {
                adjoint_halo(r, v.code == 0 ? -2 : v.code);
            }
        };
        if (B == 1 && tid < a.adj_ld) adj_out(tid, ain);
        for (int r = B == 1 ? tid + kLineBlock : tid; r < a.adj_ld; r += kLineBlock) adj_out(r, adj_in(r));
        __syncthreads();
        for (int it = wave; it < 3 * C * nt; it += kLineWaves) el_item(it);
        __syncthreads();
    }
    // rows
    double ssq = 0.0;
    auto mf_sum = [&](int c, int t) {
        T mf = 0;
        for (int cj = 0; cj < C; ++cj) mf += smf[(c * C + cj) * a.mf_ld + t];
        return (double)mf;
    };
    auto row_out = [&](int e, const RowIn &v) {
        if (v.i < 0) return;
        const int row = e / TN, t = e - row * TN;
        double r;
        if (a.out_el && row < C) {
            if (v.fixed) {
                r = v.in;
            } else {
                const T *s = sel + 3 * row * a.mf_ld + t;
                r = (double)(s[2 * a.mf_ld] + s[0] - s[a.mf_ld]);
                if constexpr (!LINEAR) {
                    r += log(v.x) + v.mu;
                    if (a.nwall > 0) r += v.vext;
                } else {
                    if (a.in_rho) r += v.in / v.x;
                }
                if (CHAIN ? a.nmf > 0 : a.el_mf != nullptr) r += CHAIN ? mf_sum(row, t) : v.mf;
            }
            if (a.add) r += v.add;
            a.out_el[(size_t)row * N + v.i] = r;
        } else {
            const int q = row - (a.out_el ? C : 0);
            r = (q < 6 ? rb_val(q, t) : mf_sum(q - 6, t)) - v.in - v.sub;
            (q < 6 ? a.out_rb + (size_t)q * N : a.out_mf + (size_t)(q - 6) * N)[v.i] = r;
        }
        ssq += r * r;
    };
    if constexpr (B == 1) row_out(tid, rin);
    for (int e = B == 1 ? tid + kLineBlock : tid; e < n_out * TN; e += kLineBlock) row_out(e, row_in(e));
    if (a.ss) {
        __shared__ double sh[kLineWaves];
        for (int o = 32; o > 0; o >>= 1) ssq += __shfl_down(ssq, o, 64);
        if (lane == 0) sh[wave] = ssq;
        __syncthreads();
        if (tid == 0) {
            double s = 0.0;
            for (int w = 0; w < kLineWaves; ++w) s += sh[w];
            a.ss[blockIdx.x] = s;
        }
    }
}

// A call's LDS must fit (wide stencils on fine grids and many components keep the row kernels).
struct LineShape {
    int B, TN, hr, hf, rho_ld, rb_ld, mf_ld, adj_ld, chain_ld, blocks;
    size_t elems;
};
LineShape line_shape(const Problem &P, bool chain, bool rows, bool el)
{
    LineShape s;
    const int C = P.p.ncomp, hu = P.pad_u.h[0];
    s.B = line_lanes(P);
    s.TN = 64 * s.B;
    s.hf = P.pad_f.h[0];
    s.hr = chain ? std::max(hu, 2 * s.hf) : hu;
    auto ld = [&](int n) { return (n + (s.B == 1 ? 40 : 20) + 3) & ~3; };   // zero positions that a sum's last steps read
    s.rho_ld = ld(s.TN + 2 * s.hr);
    s.rb_ld = (s.TN + (chain ? 2 * s.hf : 0) + 3) & ~3;
    s.mf_ld = s.TN;
    s.adj_ld = ld(s.TN + 2 * s.hf);
    const size_t n_rho = (size_t)C * s.rho_ld, n_adj = (size_t)(2 * C + 1) * s.adj_ld;
    s.chain_ld = (int)std::max(n_rho, n_adj);
    s.elems = chain ? s.chain_ld : (rows ? n_rho : 0) + (el ? n_adj + 3 * (size_t)C * s.mf_ld : 0);
    if (rows) s.elems += 3 * (size_t)C * s.rb_ld + (P.nmf ? (size_t)C * C * s.mf_ld : 0);
    const long long span = (long long)P.pad_u.P[0] - 2LL * hu;
    s.blocks = (int)((span + s.TN - 1) / s.TN);
    return s;
}

template <typename T>
LineRow<T> line_row(const DevRow1DT<T> &d)
{
    return LineRow<T>{d.w, d.wv, d.lo0, d.L};
}

template <typename T>
LineArgs<T> line_args(const Problem &P, const LineShape &s)
{
    LineArgs<T> a{};
    const int C = P.p.ncomp;
    a.g = make_geo(P, P.pad_u);
    for (int c = 0; c < C; ++c) {
        a.th[c] = line_row(dev_row<T>(P, TMI_THETA, c));
        a.de[c] = line_row(dev_row<T>(P, TMI_DELTA, c));
    }
    if (P.nmf)
        for (int q = 0; q < C * C; ++q) a.u[q] = line_row(dev_row<T>(P, TMI_UATT, q));
    a.cc = make_consts(P);
    a.TN = s.TN;
    a.hr = s.hr;
    a.hf = s.hf;
    a.rho_ld = s.rho_ld;
    a.rb_ld = s.rb_ld;
    a.mf_ld = s.mf_ld;
    a.adj_ld = s.adj_ld;
    a.chain_ld = s.chain_ld;
    a.nmf = P.nmf;
    a.func = P.p.type_func;
    a.nwall = P.p.nwall;
    a.zero = P.d_zero;
    a.elzero = P.d_elzero;
    a.vext = P.d_vext;
    return a;
}

template <typename T, bool CHAIN, bool LINEAR>
void line_launch(const LineShape &s, const LineArgs<T> &a, hipStream_t st)
{
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)s.blocks), dim3(kLineBlock), s.elems * sizeof(T), st, a);
    };
    if (s.B == 1)
        go(k_line<T, 1, CHAIN, LINEAR>);
    else if (s.B == 2)
        go(k_line<T, 2, CHAIN, LINEAR>);
    else
        go(k_line<T, 4, CHAIN, LINEAR>);
    TMI_HIP_CHECK(hipGetLastError());
}

}  // namespace

// Every call of a 1D problem through k_line: dense row weights, the exact Jacobian's adjoint fields,
// and LDS for the largest form (FP64).  The FMT halo never exceeds the density halo.
bool line_available(const Problem &P)
{
    if (!P.line1d || !P.use_rows1d || P.pad_f.h[0] > P.pad_u.h[0]) return false;
    const size_t most = std::max(line_shape(P, true, true, true).elems, line_shape(P, false, true, true).elems);
    return most * sizeof(double) + 256 <= kLineLds;
}
long long line_partials(const Problem &P) { return line_available(P) ? line_shape(P, false, true, true).blocks : 0; }

template <typename T>
void line_rows_el(Problem &P, bool linear, const double *rho, const double *in_rb, const double *sub_rb, double *out_rb,
                  const double *in_mf, const double *sub_mf, double *out_mf, const double *x, const double *dn_rb,
                  const double *in_rho, const double *el_mf, const double *add, double *out_el, hipStream_t s, double *ss)
{
    const LineShape sh = line_shape(P, false, rho != nullptr, out_el != nullptr);
    LineArgs<T> a = line_args<T>(P, sh);
    const size_t N = P.N;
    a.rho = rho;
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
        line_launch<T, false, true>(sh, a, s);
    else
        line_launch<T, false, false>(sh, a, s);
}
template void line_rows_el<double>(Problem &, bool, const double *, const double *, const double *, double *,
                                   const double *, const double *, double *, const double *, const double *,
                                   const double *, const double *, const double *, double *, hipStream_t, double *);
template void line_rows_el<float>(Problem &, bool, const double *, const double *, const double *, double *,
                                  const double *, const double *, double *, const double *, const double *,
                                  const double *, const double *, const double *, double *, hipStream_t, double *);

template <typename T>
void line_schur(Problem &P, const double *x, const double *x2, const double *mul, double *y2, const int *done, hipStream_t s)
{
    const LineShape sh = line_shape(P, true, true, true);
    LineArgs<T> a = line_args<T>(P, sh);
    const size_t N = P.N;
    a.rho = x2;
    a.mul = mul;
    a.x_rb = x + (size_t)P.iu_rb * N;
    a.x_rho = x + (size_t)P.iu_rho * N;
    a.in_rho = x2;
    a.out_el = y2;
    a.done = done;
    a.pore_of = P.d_pore_of;
    line_launch<T, true, true>(sh, a, s);
}
template void line_schur<double>(Problem &, const double *, const double *, const double *, double *, const int *,
                                 hipStream_t);
template void line_schur<float>(Problem &, const double *, const double *, const double *, double *, const int *,
                                hipStream_t);

}  // namespace tmi
