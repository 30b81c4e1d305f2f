/*
 * wf_planes.hip -- pressure solve by real coefficient planes: three launches
 * per solve, for any transform lengths, on the matrix cores.
 *
 * f is real, so its x-transform has nx real coefficients per row: Re F_r for
 * r = 0 .. nx/2 and Im F_r for 1 <= r <= (nx-1)/2.  Along y and z each
 * coefficient is a real plane of its own (the tridiagonal systems are real and
 * depend on kx^2 + ky^2 alone), so a whole plane (ny x nz reals) can be
 * y-transformed, solved in z and transformed back by one workgroup in LDS:
 *
 *   P1 k_pl_rhs   : f of 16 rows of a slab, x-analysis      -> planes U[coef][k][j]
 *   P2 k_pl_solve : one plane: y-analysis, Thomas, y-synthesis, in LDS (or, where
 *                   that does not hold it or measured slower, k_pl_y, k_pl_tri, k_pl_y)
 *   P3 k_pl_inv   : x-synthesis of 16 rows of a slab, p, periodic duplicates,
 *                   max |dp| per workgroup
 *
 * against five dependent launches with the half spectrum read and written
 * three times in between (wf_pressure.hip).  Up to 128 nodes across, a launch
 * of that form takes 4-8 us however little it moves, so the launches were the
 * time; and its run-time stages evaluate a prime factor p of the length with p
 * terms to every output.
 *
 * The transforms are products with the cosine and sine matrices on MFMA
 * (v_mfma_f64_16x16x4f64), on the sums and differences
 * x_i +- x_{n-i}, which halve the terms of every output: n^2/2 multiply-adds
 * per real row.  That is the work of a prime length at any factorisation, and
 * costs nothing for the short lengths, where the rows would leave the lanes of
 * a mixed-radix plan idle; long lengths of small factors stay on the passes
 * (wf_pl_takes).  Memory: 8 bytes a node for U and 4 for the tables of the
 * tridiagonal solves (pl_l, pl_ru), where the passes hold 8 and 0.5.
 *
 * FP64 only.  The mixed form's p is a few 1e-5 from the FP64 one, all of it
 * the state's FP32 rounding carried through the divergence, and any other
 * order of operations in its transforms gives another draw of that rounding:
 * as accurate (2.6e-7 per solve against 3.7e-7) and 1.3 to 1.7 times as fast when
 * tried, but results that differ by more than its users' comparisons allow.
 */
#include <math.h>

#include "wf_common.h"
#include "wf_kernels.h"
#include "wf_pressure_dev.h"

namespace WF_NS {

typedef double wf_acc __attribute__((ext_vector_type(4)));
__device__ __forceinline__ wf_acc wf_mfma(double a, double b, wf_acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
/* row of accumulator element q in lane group lg = lane / 16 (column lane % 16) */
__device__ __forceinline__ int wf_acc_row(int lg, int q) { return lg + 4 * q; }

/* levels per workgroup of the transforms of planes that do not fit LDS */
#define WF_PL_LEVELS 32

/* Operand tables of length n, in the order the lanes read them:
 * [tile][step][cos, sin][lane], entry (r, i) = (16 tile + lane % 16,
 * 4 step + lane / 16), 4 steps per 16 terms.
 *   forward: cos(2 pi r i / n) and -sin(2 pi r i / n), applied to the sums and
 *            differences x_i +- x_{n-i} (output r, term i);
 *   inverse: w_i cos(2 pi r i / n) and -2 sin(2 pi r i / n), w = 1 for the
 *            bins without a conjugate and 2 for the others (output r, bin i).
 * Entries outside the lengths, and sines that vanish, are 0. */
void wf_pl_matrix(int n, std::vector<double> &fwd, std::vector<double> &inv) {
    const int h = wf_pl_half(n), T = wf_pl_tiles(n), S = 4 * T;
    std::vector<double> co(n), si(n);
    for (int e = 0; e < n; e++) {
        co[e] = cos(2.0 * M_PI * (double)e / (double)n);
        si[e] = sin(2.0 * M_PI * (double)e / (double)n);
    }
    fwd.assign((size_t)T * S * 128, 0.0);
    inv.assign((size_t)T * S * 128, 0.0);
    for (int t = 0; t < T; t++)
        for (int s = 0; s < S; s++)
            for (int l = 0; l < 64; l++) {
                const int r = 16 * t + (l & 15), i = 4 * s + (l >> 4);
                if (r >= h || i >= h) continue;
                const int e = r * i % n;
                const size_t o = ((size_t)t * S + s) * 128 + l;
                const bool single = (i == 0 || 2 * i == n);
                fwd[o] = co[e];
                inv[o] = (single ? 1.0 : 2.0) * co[e];
                if (!single && r != 0 && 2 * r != n) {
                    fwd[o + 64] = -si[e];
                    inv[o + 64] = -2.0 * si[e];
                }
            }
}

/* t / d by the reciprocal m = 2^32 / d rounded up (exact for t < 2^16, d <= 2^10) */
__device__ __forceinline__ unsigned wf_pl_magic(int d) { return 0xffffffffu / (unsigned)d + 1u; }
__device__ __forceinline__ int wf_pl_div(int t, unsigned m, int d) {
    return (d == 1) ? t : (int)__umulhi((unsigned)t, m);
}

/* Keeps the loads of x ahead of the branch that follows: the convergence flag
 * and a pass's first operands are then fetched together, one round trip
 * instead of two (a pass of these sizes is a few round trips long). */
__device__ __forceinline__ void wf_pin(wf_real &x) { asm volatile("" : "+v"(x)); }

/* Matrix operands of 4 steps (cosines in [2u], sines in [2u + 1]). */
struct WfPlMat {
    wf_real m[8];
    __device__ __forceinline__ void load(const wf_real *M, int s0) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            m[2 * u] = M[(s0 + u) * 128];
            m[2 * u + 1] = M[(s0 + u) * 128 + 64];
        }
    }
};

/* Products of TPW data tiles with one tile of the cosine and sine matrices
 * over S steps (a multiple of 4).  The matrix operands come from L2 (every
 * workgroup reads the same tables), two groups of 4 steps ahead of their use:
 * one group runs for 512 cycles of the matrix core, about what a load takes.
 * first holds the operands of steps 0 .. 3.  data(s, t, x, y) reads the data
 * operands of step s.  MA: the matrix is the first factor. */
template <bool MA, int TPW, typename F>
__device__ __forceinline__ void wf_pl_product(const wf_real *M, int S, const WfPlMat &first, F data,
                                              wf_acc (&c)[TPW], wf_acc (&d)[TPW]) {
    WfPlMat cur = first, next;
    next.load(M, (S > 4) ? 4 : 0);
    for (int s0 = 0; s0 < S; s0 += 4) {
        WfPlMat after;
        after.load(M, (s0 + 8 < S) ? s0 + 8 : s0);
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
            for (int t = 0; t < TPW; t++) {
                wf_real x, y;
                data(s0 + u, t, x, y);
                c[t] = MA ? wf_mfma(cur.m[2 * u], x, c[t]) : wf_mfma(x, cur.m[2 * u], c[t]);
                d[t] = MA ? wf_mfma(cur.m[2 * u + 1], y, d[t]) : wf_mfma(y, cur.m[2 * u + 1], d[t]);
            }
        cur = next;
        next = after;
    }
}

/* ----------------------------------------------------------------- P1 ---- */

/* f (form MODE) of rows j0 .. j0 + 15 of a slab and its x-analysis.  A thread
 * evaluates f at i and nx - i and leaves their sum and difference in LDS; the
 * waves then take 16 coefficients each.  What bounds it is the latency of the
 * 28 stencil loads of a node pair: `slots` node pairs per thread follow one
 * another, so the launch takes enough threads for about two (wf_pl_rhs_nt). */
template <int MODE>
__device__ __forceinline__ void wf_pl_rhs_body(const WfConst &c, const WfSpectral &sp, const WfState &Ys,
                                               const WfState &Yn, const wf_real *p, int block, int check) {
    extern __shared__ wf_real smem_r[];
    /* the first solve of a step is never done */
    const int done = (MODE == WF_F_ITER) ? wf_first_pass_returns(sp.ctl->done, check) : 0;
    const int nx = sp.nx, ny = sp.ny, hx = sp.hx, ld = wf_pl_stride(nx + 1);
    const int g = block % sp.pl_groups, ks = block / sp.pl_groups;
    const int k = 1 + ks;
    const int j0 = g * WF_PL_ROWS;
    const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), W = (int)(blockDim.x >> 6);
    const int T = wf_pl_tiles(nx), S = 4 * T;
    WfPlMat first;
    first.load(sp.pl_fx + (long)((w < T) ? w : 0) * S * 128 + lane, 0);
    const unsigned mh = wf_pl_magic(hx);
    const int n = WF_PL_ROWS * hx;
    for (int t0 = threadIdx.x; t0 - (int)threadIdx.x < n; t0 += blockDim.x) {
        const int t = (t0 < n) ? t0 : n - 1;
        const int row = wf_pl_div(t, mh, hx), i = t - row * hx;
        const int i2 = (i == 0 || 2 * i == nx) ? i : nx - i;
        const int j = (j0 + row < ny) ? j0 + row : ny - 1;
        wf_real f1 = wf_fx_input<MODE>(c, sp, Ys, Yn, p, i, j, k);
        wf_real f2 = wf_fx_input<MODE>(c, sp, Ys, Yn, p, i2, j, k);
        if (k == sp.nz - 1) { /* the known top plane, moved to the right-hand side */
            const long o = c.plane * (long)(c.Nz - 1) + (long)c.Nx * j;
            f1 = f1 - p[o + i] / (wf_real)sp.top_div;
            f2 = f2 - p[o + i2] / (wf_real)sp.top_div;
        }
        if (MODE == WF_F_ITER && t0 == (int)threadIdx.x) {
            wf_pin(f1);
            wf_pin(f2);
            if (done) return;
        }
        smem_r[row * ld + i] = (i2 == i) ? f1 : f1 + f2;
        smem_r[row * ld + ((i2 == i) ? nx : i2)] = (i2 == i) ? WR(0.0) : f1 - f2;
    }
    __syncthreads();
    const wf_real *rowp = smem_r + lr * ld;
    const long cs = (long)sp.nz * sp.pl_ld; /* coefficient stride */
    wf_real *out = sp.U + (long)k * sp.pl_ld + j0 + lr;
    for (int t = w; t < T; t += W) {
        const wf_real *A = sp.pl_fx + (long)t * S * 128 + lane;
        if (t != w) first.load(A, 0);
        wf_acc ac[1] = {}, as[1] = {};
        wf_pl_product<true, 1>(
            A, S, first,
            [&](int st, int, wf_real &x, wf_real &y) {
                const int ia = min(4 * st + lg, hx - 1);
                x = rowp[ia];
                y = rowp[nx - ia];
            },
            ac, as);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int r = 16 * t + wf_acc_row(lg, q);
            if (r < hx) out[r * cs] = ac[0][q];
            if (r >= 1 && 2 * r < nx) out[(hx + r - 1) * cs] = as[0][q];
        }
    }
}

template <int MODE>
__global__ __launch_bounds__(512) void k_pl_rhs(WfConst c, WfSpectral sp, WfState Ys, WfState Yn, const wf_real *p,
                                                 double tol, double rtol, int check, int max_iter) {
    const int b = wf_checked_block(sp, tol, rtol, check, max_iter);
    if (b >= 0) wf_pl_rhs_body<MODE>(c, sp, Ys, Yn, p, b, check);
}
template <int MODE>
__global__ __launch_bounds__(512) void k_pl_rhs_batch(const WfPressItem *__restrict__ tab, int check) {
    const WfPressItem it = wf_press_load(tab);
    const int b = wf_checked_block(it.sp, it.tol, it.rtol, check, it.max_iter);
    if (b >= 0) wf_pl_rhs_body<MODE>(it.c, it.sp, it.ys, it.yn, it.p, b, check);
}

/* ----------------------------------------------------------------- P2 ---- */

/* Operands of a wave's chunk of LC levels of 64 tridiagonal systems: the
 * multipliers l_k and reciprocal pivots 1/u_k, from tables formed once
 * (k_pl_pivots).  l_0 and the entries of the levels past the last
 * (rounded up to whole chunks) are 0, and so is c past the last level, which
 * makes the first and last rows of the system and the empty levels ordinary
 * ones. */
template <int LC>
struct WfPlTri {
    double l[LC], ru[LC];
    __device__ __forceinline__ void load(const WfSpectral &sp, int g, int ch, const double *L, const double *RU) {
        const int ny = sp.ny, hy = wf_pl_half(ny), nzp = wf_pl_levels(sp.nz);
        const int sys = g * 64 + (int)(threadIdx.x & 63), sc = (sys < ny) ? sys : 0;
        const int s = (sc < hy) ? sc : sc - hy + 1;
        const int k0 = min(ch * LC, nzp - LC);
#pragma unroll
        for (int t = 0; t < LC; t++) {
            l[t] = L[(k0 + t) * hy + s];
            ru[t] = RU[(k0 + t) * hy + s];
        }
    }
};

/* Tridiagonal solves of one plane in LDS (Z[k][s], systems s across lanes),
 * as wf_thomas_solve: a wave takes a chunk of LC levels of 64 systems, forward
 * elimination and back substitution run from a zero entry value with the
 * coefficient of the entry value carried along, and the chunks combine
 * through LDS in order.  With the tables a level costs two fused operations
 * instead of two divisions.  The waves take gp groups of 64 systems at a time, of
 * groups gfirst .. gend - 1, C chunks each; tri holds the operands of the first. */
template <int LC>
__device__ __forceinline__ void wf_pl_thomas(const WfSpectral &sp, wf_real *Z, int ld, int r, const double *L,
                                             const double *RU, WfPlTri<LC> &tri, int gfirst, int gend, int gp,
                                             int C, wf_cx<double> *comb) {
#pragma clang fp contract(fast)
    const int ny = sp.ny, nz = sp.nz, hy = wf_pl_half(ny);
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int gs = w % gp, ch = w / gp, k0 = ch * LC; /* ch >= C: idle */
    const double K2r = sp.kx2[r];
    const double *tc = sp.tc;
    for (int g0 = gfirst; g0 < gend; g0 += gp) {
        const int sys = (g0 + gs) * 64 + lane;
        const int sc = (sys < ny) ? sys : 0;
        const int s = (sc < hy) ? sc : sc - hy + 1;
        const bool ok = sys < ny && ch < C;
        if (g0 > gfirst && ch < C) tri.load(sp, g0 + gs, ch, L, RU);
        const double c0 = sp.c0a - 0.5 * sp.dz0 * (K2r + sp.ky2[s]) - sp.c0b;
        double y[LC], G[LC];
        double acc = 0.0, g = 1.0;
        if (ch < C) {
#pragma unroll
            for (int t = 0; t < LC; t++) y[t] = Z[min(k0 + t, nz - 1) * ld + sc];
#pragma unroll
            for (int t = 0; t < LC; t++) {
                acc = y[t] - tri.l[t] * acc;
                g = -tri.l[t] * g;
                y[t] = acc;
                G[t] = g;
            }
            comb[w * 64 + lane] = wf_cx<double>{acc, g};
        }
        __syncthreads();
        /* value entering the chunk from the chunks below, 4 of them read at a time */
        double in = 0.0;
        if (ch < C)
            for (int q0 = 0; q0 < ch; q0 += 4) {
                wf_cx<double> e[4];
#pragma unroll
                for (int u = 0; u < 4; u++) e[u] = comb[(min(q0 + u, ch - 1) * gp + gs) * 64 + lane];
#pragma unroll
                for (int u = 0; u < 4; u++) in = (q0 + u < ch) ? e[u].x + e[u].y * in : in;
            }
        __syncthreads();
        acc = 0.0;
        g = 1.0;
        if (ch < C) {
#pragma unroll
            for (int t = LC - 1; t >= 0; t--) {
                const double ck = (t == 0 && ch == 0) ? c0 : tc[k0 + t];
                acc = (y[t] + G[t] * in - ck * acc) * tri.ru[t];
                g = (-ck * tri.ru[t]) * g;
                y[t] = acc;
                G[t] = g;
            }
            comb[w * 64 + lane] = wf_cx<double>{acc, g};
        }
        __syncthreads();
        in = 0.0;
        for (int q0 = C - 1; q0 > ch; q0 -= 4) {
            wf_cx<double> e[4];
#pragma unroll
            for (int u = 0; u < 4; u++) e[u] = comb[(max(q0 - u, ch + 1) * gp + gs) * 64 + lane];
#pragma unroll
            for (int u = 0; u < 4; u++) in = (q0 - u > ch) ? e[u].x + e[u].y * in : in;
        }
#pragma unroll
        for (int t = 0; t < LC; t++)
            if (ok && k0 + t < nz) Z[(k0 + t) * ld + sc] = y[t] + G[t] * in;
        __syncthreads();
    }
}

/* One plane: y-analysis, tridiagonal solves, y-synthesis.  TPW: 16-level
 * tiles a wave takes with one set of matrix operands; LC: levels per lane of
 * the tridiagonal solves. */
template <int TPW, int LC>
__device__ __forceinline__ void wf_pl_solve_body(const WfSpectral &sp, int coef) {
    extern __shared__ wf_real smem_r[];
    const int done = wf_pass_returns(sp.ctl->done);
    const int ny = sp.ny, nz = sp.nz, hx = sp.hx, hy = wf_pl_half(ny), ld = wf_pl_stride(ny + 1);
    wf_real *Z = smem_r;
    wf_cx<double> *comb = (wf_cx<double> *)(smem_r + (((long)nz * ld + 3) & ~3l));
    const int tid = threadIdx.x, nt = (int)blockDim.x;
    const int lane = tid & 63, lr = lane & 15, lg = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), W = nt >> 6;
    const int T = wf_pl_tiles(ny), S = 4 * T;
    const int KG = W / T, jt = w % T, kg = w / T; /* kg >= KG: no tile */
    wf_real *plane = sp.U + (long)coef * nz * sp.pl_ld;
    const wf_real *Mf = sp.pl_fy + (long)jt * S * 128 + lane, *Mi = sp.pl_iy + (long)jt * S * 128 + lane;
    const int r = (coef < hx) ? coef : coef - hx + 1;
    const long to = (long)r * wf_pl_levels(nz) * hy;
    const int C = (nz + LC - 1) / LC, gp = max(1, W / C); /* chunks, system groups at a time */
    const int ng = (ny + 63) / 64;
    WfPlMat first;
    WfPlTri<LC> tri;
    /* sums and differences of rows 1 .. nz-1 (row 0 follows from row 1); the
     * first matrix and tridiagonal operands go out with the first loads */
    {
        constexpr int B = 4;
        const unsigned mh = wf_pl_magic(hy);
        const int n = (nz - 1) * hy;
        for (int t0 = tid; t0 - tid < n; t0 += B * nt) {
            wf_real a[B], b[B];
            int row[B], j[B], j2[B];
#pragma unroll
            for (int u = 0; u < B; u++) {
                const int t = (t0 + u * nt < n) ? t0 + u * nt : n - 1;
                const int rr = wf_pl_div(t, mh, hy);
                row[u] = 1 + rr;
                j[u] = t - rr * hy;
                j2[u] = (j[u] == 0 || 2 * j[u] == ny) ? j[u] : ny - j[u];
                a[u] = plane[(long)row[u] * sp.pl_ld + j[u]];
                b[u] = plane[(long)row[u] * sp.pl_ld + j2[u]];
            }
            if (t0 == tid) {
                first.load(Mf, 0);
                tri.load(sp, w % gp, w / gp, sp.pl_l + to, sp.pl_ru + to);
#pragma unroll
                for (int u = 0; u < B; u++) {
                    wf_pin(a[u]);
                    wf_pin(b[u]);
                }
                if (done) return;
            }
#pragma unroll
            for (int u = 0; u < B; u++) {
                if (t0 + u * nt < n) {
                    Z[row[u] * ld + j[u]] = (j2[u] == j[u]) ? a[u] : a[u] + b[u];
                    Z[row[u] * ld + ((j2[u] == j[u]) ? ny : j2[u])] = (j2[u] == j[u]) ? WR(0.0) : a[u] - b[u];
                }
            }
        }
    }
    __syncthreads();
    wf_acc ac[TPW] = {}, as[TPW] = {};
    int rp[TPW];
    if (kg < KG) {
#pragma unroll
        for (int t = 0; t < TPW; t++) {
            int kr = 16 * (kg + t * KG) + lr;
            kr = (kr < 1) ? 1 : (kr < nz) ? kr : nz - 1;
            rp[t] = kr * ld;
        }
        wf_pl_product<false, TPW>(
            Mf, S, first,
            [&](int st, int t, wf_real &x, wf_real &y) {
                const int ja = min(4 * st + lg, hy - 1);
                x = Z[rp[t] + ja];
                y = Z[rp[t] + ny - ja];
            },
            ac, as);
    }
    __syncthreads();
    if (kg < KG) {
        const int s = 16 * jt + lr;
#pragma unroll
        for (int t = 0; t < TPW; t++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int k = 16 * (kg + t * KG) + wf_acc_row(lg, q);
                /* level 0 holds half a spacing of level 1's f */
                const wf_real f = (k == 0) ? WR(0.5) * (wf_real)sp.dz0 : WR(1.0);
                if (k < nz && s < hy) Z[k * ld + s] = f * ac[t][q];
                if (k < nz && s >= 1 && 2 * s < ny) Z[k * ld + hy + s - 1] = f * as[t][q];
            }
    }
    __syncthreads();
    first.load(Mi, 0);
    wf_pl_thomas<LC>(sp, Z, ld, r, sp.pl_l + to, sp.pl_ru + to, tri, 0, ng, gp, C, comb);
    if (kg >= KG) return;
    wf_acc ec[TPW] = {}, es[TPW] = {};
#pragma unroll
    for (int t = 0; t < TPW; t++) {
        const int kr = 16 * (kg + t * KG) + lr;
        rp[t] = ((kr < nz) ? kr : nz - 1) * ld;
    }
    wf_pl_product<false, TPW>(
        Mi, S, first,
        [&](int st, int t, wf_real &x, wf_real &y) {
            const int jj = 4 * st + lg;
            x = Z[rp[t] + min(jj, hy - 1)];
            y = Z[rp[t] + min(hy - 1 + jj, ny - 1)];
        },
        ec, es);
    const int j = 16 * jt + lr;
#pragma unroll
    for (int t = 0; t < TPW; t++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int k = 16 * (kg + t * KG) + wf_acc_row(lg, q);
            if (k < nz && j < hy) {
                plane[(long)k * sp.pl_ld + j] = ec[t][q] + es[t][q];
                if (j >= 1 && 2 * j < ny) plane[(long)k * sp.pl_ld + ny - j] = ec[t][q] - es[t][q];
            }
        }
}

template <int NT, int TPW, int LC>
__global__ __launch_bounds__(NT) void k_pl_solve(WfSpectral sp) {
    wf_pl_solve_body<TPW, LC>(sp, (int)blockIdx.x);
}
template <int NT, int TPW, int LC>
__global__ __launch_bounds__(NT) void k_pl_solve_batch(const WfPressItem *__restrict__ tab) {
    const WfPressItem it = wf_press_load(tab);
    wf_pl_solve_body<TPW, LC>(it.sp, (int)blockIdx.x);
}

/* The same in three launches (where: wf_pl_solve_nt): the y-analysis
 * (INV = false) or synthesis of WF_PL_LEVELS levels of a plane, in place ... */
template <bool INV>
__device__ __forceinline__ void wf_pl_y_body(const WfSpectral &sp) {
    if (wf_pass_returns(sp.ctl->done)) return;
    extern __shared__ wf_real smem_r[];
    const int ny = sp.ny, nz = sp.nz, hy = wf_pl_half(ny), ld = wf_pl_stride(ny + 1);
    const int tid = threadIdx.x, nt = (int)blockDim.x;
    const int lane = tid & 63, lr = lane & 15, lg = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), W = nt >> 6;
    const int T = wf_pl_tiles(ny), S = 4 * T;
    const int kb = (int)blockIdx.y * WF_PL_LEVELS, nk = min(nz - kb, WF_PL_LEVELS);
    wf_real *plane = sp.U + (long)blockIdx.x * nz * sp.pl_ld;
    {
        constexpr int B = 4;
        const unsigned mh = wf_pl_magic(hy);
        const int n = nk * hy;
        for (int t0 = tid; t0 - tid < n; t0 += B * nt) {
            wf_real a[B], b[B];
            int row[B], j[B], j2[B];
#pragma unroll
            for (int u = 0; u < B; u++) {
                const int t = (t0 + u * nt < n) ? t0 + u * nt : n - 1;
                row[u] = wf_pl_div(t, mh, hy);
                j[u] = t - row[u] * hy;
                const bool single = (j[u] == 0 || 2 * j[u] == ny);
                j2[u] = single ? ny : INV ? hy + j[u] - 1 : ny - j[u];
                /* level 0 follows from level 1 */
                const wf_real *src = plane + (long)(INV ? kb + row[u] : max(kb + row[u], 1)) * sp.pl_ld;
                a[u] = src[j[u]];
                b[u] = src[single ? j[u] : j2[u]];
            }
#pragma unroll
            for (int u = 0; u < B; u++) {
                if (t0 + u * nt < n) {
                    const bool single = j2[u] == ny;
                    wf_real *z = smem_r + row[u] * ld;
                    z[j[u]] = (INV || single) ? a[u] : a[u] + b[u];
                    z[j2[u]] = single ? WR(0.0) : INV ? b[u] : a[u] - b[u];
                }
            }
        }
    }
    __syncthreads();
    const wf_real *tab = INV ? sp.pl_iy : sp.pl_fy;
    for (int e = w; e < T * (WF_PL_LEVELS / 16); e += W) {
        const int jt = e % T, kt = e / T;
        const wf_real *M = tab + (long)jt * S * 128 + lane;
        const wf_real *z = smem_r + min(16 * kt + lr, nk - 1) * ld;
        WfPlMat first;
        first.load(M, 0);
        wf_acc ac[1] = {}, as[1] = {};
        wf_pl_product<false, 1>(
            M, S, first,
            [&](int st, int, wf_real &x, wf_real &y) {
                const int jj = min(4 * st + lg, hy - 1);
                x = z[jj];
                y = z[INV ? min(hy - 1 + jj, ny - 1) : ny - jj];
            },
            ac, as);
        const int j = 16 * jt + lr;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int kl = 16 * kt + wf_acc_row(lg, q);
            if (kl < nk && j < hy) {
                wf_real *dst = plane + (long)(kb + kl) * sp.pl_ld;
                const bool two = j >= 1 && 2 * j < ny;
                if constexpr (INV) {
                    dst[j] = ac[0][q] + as[0][q];
                    if (two) dst[ny - j] = ac[0][q] - as[0][q];
                } else {
                    const wf_real f = (kb + kl == 0) ? WR(0.5) * (wf_real)sp.dz0 : WR(1.0);
                    dst[j] = f * ac[0][q];
                    if (two) dst[hy + j - 1] = f * as[0][q];
                }
            }
        }
    }
}
/* ... and the tridiagonal solves of 64 systems of a plane, in place. */
template <int LC>
__device__ __forceinline__ void wf_pl_tri_body(const WfSpectral &sp) {
    if (wf_pass_returns(sp.ctl->done)) return;
    __shared__ wf_cx<double> comb[1024];
    const int coef = blockIdx.x, g = blockIdx.y, nz = sp.nz, hy = wf_pl_half(sp.ny);
    const int r = (coef < sp.hx) ? coef : coef - sp.hx + 1;
    const int C = (nz + LC - 1) / LC;
    const int ch = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    wf_real *plane = sp.U + (long)coef * nz * sp.pl_ld;
    const long to = (long)r * wf_pl_levels(nz) * hy;
    WfPlTri<LC> tri;
    tri.load(sp, g, ch, sp.pl_l + to, sp.pl_ru + to);
    wf_pl_thomas<LC>(sp, plane, sp.pl_ld, r, sp.pl_l + to, sp.pl_ru + to, tri, g, g + 1, 1, C, comb);
}
template <bool INV>
__global__ __launch_bounds__(512) void k_pl_y(WfSpectral sp) {
    wf_pl_y_body<INV>(sp);
}
template <bool INV>
__global__ __launch_bounds__(512) void k_pl_y_batch(const WfPressItem *__restrict__ tab) {
    const WfPressItem it = wf_press_load(tab);
    wf_pl_y_body<INV>(it.sp);
}
template <int LC>
__global__ __launch_bounds__(1024) void k_pl_tri(WfSpectral sp) {
    wf_pl_tri_body<LC>(sp);
}
template <int LC>
__global__ __launch_bounds__(1024) void k_pl_tri_batch(const WfPressItem *__restrict__ tab) {
    const WfPressItem it = wf_press_load(tab);
    wf_pl_tri_body<LC>(it.sp);
}

/* Thomas multipliers and reciprocal pivots of every (kx, ky, level), formed
 * once with the operations of k_pivots. */
__global__ void k_pl_pivots(WfSpectral sp) {
    const int hy = wf_pl_half(sp.ny), nz = sp.nz;
    const int s = blockIdx.x * blockDim.x + threadIdx.x, r = blockIdx.y;
    if (s >= hy) return;
    const double K2 = sp.kx2d[r] + sp.ky2d[s];
    const double c0 = sp.c0a - 0.5 * sp.dz0 * K2 - sp.c0b;
    const int nzp = wf_pl_levels(nz);
    double u = sp.b0, l = 0.0;
    for (int k = 0; k < nzp; k++) {
        if (k > 0 && k < nz) u = wf_pivot_next<double>(sp, u, k, K2, c0, &l);
        const double lk = (k < nz) ? l : 0.0, ru = (k < nz) ? 1.0 / u : 0.0;
        const long o = ((long)r * nzp + k) * hy + s;
        sp.pl_l[o] = lk;
        sp.pl_ru[o] = ru;
    }
}

/* ----------------------------------------------------------------- P3 ---- */

__device__ __forceinline__ void wf_pl_norm(double pv, double pold, double &dmax) {
    const double d = fabs(pv - pold);
    dmax = (d > dmax) ? d : dmax;
}

/* x-synthesis of rows j0 .. j0 + 15 of slab k, p = (.)/(nx ny), its periodic
 * duplicates and max |p_new - p_old|; the last workgroup refreshes the
 * periodic copies of the top plane, as in wf_inv_fx_body.  Every global load
 * (coefficients, old p) goes out before the first wait. */
__device__ __forceinline__ void wf_pl_inv_body(const WfConst &c, const WfSpectral &sp, wf_real *p) {
    extern __shared__ wf_real smem_r[];
    const int done = wf_pass_returns(sp.ctl->done);
    double dmax = 0.0;
    if (blockIdx.x == gridDim.x - 1) {
        if (done) return;
        wf_top_duplicates(c, p, dmax);
    } else {
        const int nx = sp.nx, ny = sp.ny, hx = sp.hx, ld = sp.pl_ld;
        const int g = (int)blockIdx.x % sp.pl_groups, k = (int)blockIdx.x / sp.pl_groups;
        const int j0 = g * WF_PL_ROWS;
        const long cs = (long)sp.nz * ld;
        const wf_real *src = sp.U + (long)k * ld + j0;
        const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
        const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), W = (int)(blockDim.x >> 6);
        const int T = wf_pl_tiles(nx), S = 4 * T;
        const wf_real inv_scale = WR(1.0) / ((wf_real)nx * (wf_real)ny);
        const long slab = c.plane * (long)k, dup = slab + (long)c.Nx * (c.Ny - 1);
        /* old p at i and nx - i (i = 0: at its duplicate, column Nx-1) of the
         * tile's rows, and of the duplicate row Ny-1 of row 0 */
        wf_real po[4], po2[4], pd, pd2;
        WfPlMat first;
        int i, i2;
        const auto load_old = [&](int t) {
            i = (16 * t + lr < hx) ? 16 * t + lr : hx - 1;
            i2 = (i == 0) ? nx : nx - i;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int j = j0 + wf_acc_row(lg, q);
                const long o = slab + (long)c.Nx * ((j < ny) ? j : ny - 1);
                po[q] = p[o + i];
                po2[q] = p[o + i2];
            }
            pd = pd2 = WR(0.0);
            if (g == 0) {
                pd = p[dup + i];
                pd2 = p[dup + i2];
            }
            first.load(sp.pl_ix + (long)t * S * 128 + lane, 0);
        };
        {
            constexpr int B = 4;
            const int n = nx * WF_PL_ROWS, nt = (int)blockDim.x;
            for (int t0 = threadIdx.x; t0 - (int)threadIdx.x < n; t0 += B * nt) {
                wf_real a[B];
#pragma unroll
                for (int u = 0; u < B; u++) {
                    const int t = (t0 + u * nt < n) ? t0 + u * nt : n - 1;
                    a[u] = src[(long)(t >> 4) * cs + (t & 15)];
                }
                if (t0 == (int)threadIdx.x) {
                    if (w < T) load_old(w);
#pragma unroll
                    for (int u = 0; u < B; u++) wf_pin(a[u]);
                    if (done) return;
                }
#pragma unroll
                for (int u = 0; u < B; u++)
                    if (t0 + u * nt < n) smem_r[t0 + u * nt] = a[u];
            }
        }
        __syncthreads();
        for (int t = w; t < T; t += W) {
            if (t != w) load_old(t);
            wf_acc ec[1] = {}, es[1] = {};
            wf_pl_product<false, 1>(
                sp.pl_ix + (long)t * S * 128 + lane, S, first,
                [&](int st, int, wf_real &x, wf_real &y) {
                    const int rr = 4 * st + lg;
                    x = smem_r[min(rr, hx - 1) * 16 + lr];
                    y = smem_r[min(hx - 1 + rr, nx - 1) * 16 + lr];
                },
                ec, es);
            const bool in = 16 * t + lr < hx;
            const bool two = in && 2 * i != nx; /* i2 is another node */
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int j = j0 + wf_acc_row(lg, q);
                if (j < ny) {
                    const long o = slab + (long)c.Nx * j;
                    const wf_real v1 = (ec[0][q] + es[0][q]) * inv_scale;
                    const wf_real v2 = (i == 0) ? v1 : (ec[0][q] - es[0][q]) * inv_scale;
                    if (in) {
                        wf_pl_norm(v1, po[q], dmax);
                        p[o + i] = v1;
                    }
                    if (two) {
                        wf_pl_norm(v2, po2[q], dmax);
                        p[o + i2] = v2;
                    }
                    if (j == 0) { /* its duplicate, row j = Ny-1 */
                        if (in) {
                            wf_pl_norm(v1, pd, dmax);
                            p[dup + i] = v1;
                        }
                        if (two) {
                            wf_pl_norm(v2, pd2, dmax);
                            p[dup + i2] = v2;
                        }
                    }
                }
            }
        }
    }
    wf_block_max_store(dmax, &sp.pmax[blockIdx.x]);
}
__global__ __launch_bounds__(512) void k_pl_inv(WfConst c, WfSpectral sp, wf_real *p) { wf_pl_inv_body(c, sp, p); }
__global__ __launch_bounds__(512) void k_pl_inv_batch(const WfPressItem *__restrict__ tab) {
    const WfPressItem it = wf_press_load(tab);
    wf_pl_inv_body(it.c, it.sp, it.p);
}

/* ----------------------------------------------------------- launchers ---- */

/* threads of P1: enough for two node pairs each, at most 512 (two workgroups
 * a CU, so that one's products run beside the other's loads) */
static int wf_pl_rhs_nt(const WfSpectral &sp) { return (WF_PL_ROWS * sp.hx <= 512) ? 256 : 512; }
/* threads of P3: a tile per wave up to 8 where the workgroups leave CUs idle */
static int wf_pl_inv_nt(const WfSpectral &sp) {
    return (wf_pl_tiles(sp.nx) > 4 && sp.npmax <= 512) ? 512 : 256;
}
static size_t wf_pl_rhs_lds(const WfSpectral &sp) { return sizeof(wf_real) * WF_PL_ROWS * (size_t)wf_pl_stride(sp.nx + 1); }
static size_t wf_pl_y_lds(const WfSpectral &sp) { return sizeof(wf_real) * WF_PL_LEVELS * (size_t)wf_pl_stride(sp.ny + 1); }

/* The LDS above 64 KB that the kernels ask for (the x and y passes take at most
 * 133 KB beside their static reductions). */
static hipError_t wf_pl_allow(const void *kernel, int bytes = 144 * 1024) {
    return hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
}
static hipError_t wf_pl_allow_all() {
    hipError_t e = hipSuccess;
#define WF_PL_ALLOW(...) \
    if (e == hipSuccess) e = wf_pl_allow((const void *)__VA_ARGS__);
#define WF_PL_ATTR(NT, TPW, LC)                                                                                  \
    if (e == hipSuccess) e = wf_pl_allow((const void *)k_pl_solve<NT, TPW, LC>, WF_PL_LDS_MAX);                  \
    if (e == hipSuccess) e = wf_pl_allow((const void *)k_pl_solve_batch<NT, TPW, LC>, WF_PL_LDS_MAX);
    WF_PL_SOLVES(WF_PL_ATTR)
    WF_PL_ALLOW(k_pl_rhs<WF_F_ITER>)
    WF_PL_ALLOW(k_pl_rhs<WF_F_FIRST>)
    WF_PL_ALLOW(k_pl_rhs<WF_F_CONST>)
    WF_PL_ALLOW(k_pl_rhs_batch<WF_F_ITER>)
    WF_PL_ALLOW(k_pl_rhs_batch<WF_F_FIRST>)
    WF_PL_ALLOW(k_pl_rhs_batch<WF_F_CONST>)
    WF_PL_ALLOW(k_pl_inv)
    WF_PL_ALLOW(k_pl_inv_batch)
    WF_PL_ALLOW(k_pl_y<false>)
    WF_PL_ALLOW(k_pl_y<true>)
    WF_PL_ALLOW(k_pl_y_batch<false>)
    WF_PL_ALLOW(k_pl_y_batch<true>)
#undef WF_PL_ATTR
#undef WF_PL_ALLOW
    return e;
}
hipError_t wf_pl_prepare(const WfSpectral &sp, hipStream_t s) {
    /* once per process: the library runs on one device */
    static const hipError_t allowed = wf_pl_allow_all();
    if (allowed != hipSuccess) return allowed;
    hipLaunchKernelGGL(k_pl_pivots, dim3((wf_pl_half(sp.ny) + 63) / 64, sp.hx), dim3(64), 0, s, sp);
    return hipGetLastError();
}

hipError_t wf_launch_pl_rhs(const WfConst &c, const WfSpectral &sp, const WfState &Ys, const WfState &Yn,
                            const wf_real *p, int mode, double tol, double rtol, int check, int max_iter,
                            hipStream_t s) {
    const dim3 grd((unsigned)(sp.pl_groups * (sp.nz - 1) + (check >= 0))), blk(wf_pl_rhs_nt(sp));
    const size_t lds = wf_pl_rhs_lds(sp);
    if (mode == WF_F_ITER)
        hipLaunchKernelGGL(k_pl_rhs<WF_F_ITER>, grd, blk, lds, s, c, sp, Ys, Yn, p, tol, rtol, check, max_iter);
    else if (mode == WF_F_FIRST)
        hipLaunchKernelGGL(k_pl_rhs<WF_F_FIRST>, grd, blk, lds, s, c, sp, Ys, Yn, p, tol, rtol, check, max_iter);
    else if (mode == WF_F_CONST)
        hipLaunchKernelGGL(k_pl_rhs<WF_F_CONST>, grd, blk, lds, s, c, sp, Ys, Yn, p, tol, rtol, check, max_iter);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t wf_launch_pl_solve(const WfSpectral &sp, hipStream_t s) {
    if (sp.pl_nt == 0) { /* three launches (wf_pl_solve_nt) */
        const dim3 grd(sp.nx, (sp.nz + WF_PL_LEVELS - 1) / WF_PL_LEVELS), tri(sp.nx, (sp.ny + 63) / 64);
        hipLaunchKernelGGL(k_pl_y<false>, grd, dim3(512), wf_pl_y_lds(sp), s, sp);
        if (sp.nz <= 128)
            hipLaunchKernelGGL(k_pl_tri<8>, tri, dim3(64 * ((sp.nz + 7) / 8)), 0, s, sp);
        else
            hipLaunchKernelGGL(k_pl_tri<16>, tri, dim3(64 * ((sp.nz + 15) / 16)), 0, s, sp);
        hipLaunchKernelGGL(k_pl_y<true>, grd, dim3(512), wf_pl_y_lds(sp), s, sp);
        return hipGetLastError();
    }
    int tpw, lc;
    wf_pl_shape(sp.ny, sp.nz, sp.pl_nt, &tpw, &lc);
    const size_t lds = (size_t)wf_pl_lds(sp.ny, sp.nz, sp.pl_nt);
#define WF_PL_GO(NT, TPW, LC)                                                               \
    if (sp.pl_nt == NT && tpw == TPW && lc == LC) {                                         \
        hipLaunchKernelGGL((k_pl_solve<NT, TPW, LC>), dim3(sp.nx), dim3(NT), lds, s, sp);   \
        return hipGetLastError();                                                           \
    }
    WF_PL_SOLVES(WF_PL_GO)
#undef WF_PL_GO
    return hipErrorInvalidValue;
}

hipError_t wf_launch_pl_inv(const WfConst &c, const WfSpectral &sp, wf_real *p, hipStream_t s) {
    hipLaunchKernelGGL(k_pl_inv, dim3(sp.npmax), dim3(wf_pl_inv_nt(sp)), sizeof(wf_real) * WF_PL_ROWS * sp.nx, s, c, sp, p);
    return hipGetLastError();
}

/* Batched launchers: one size class, z = the member (wf_pressure.hip). */
hipError_t wf_launch_pl_rhs_batch(const WfSpectral &sp, const WfPressItem *tab, int nm, int mode, int check,
                                  hipStream_t s) {
    const dim3 grd((unsigned)(sp.pl_groups * (sp.nz - 1) + (check >= 0)), 1, nm), blk(wf_pl_rhs_nt(sp));
    const size_t lds = wf_pl_rhs_lds(sp);
    if (mode == WF_F_ITER)
        hipLaunchKernelGGL(k_pl_rhs_batch<WF_F_ITER>, grd, blk, lds, s, tab, check);
    else if (mode == WF_F_FIRST)
        hipLaunchKernelGGL(k_pl_rhs_batch<WF_F_FIRST>, grd, blk, lds, s, tab, check);
    else if (mode == WF_F_CONST)
        hipLaunchKernelGGL(k_pl_rhs_batch<WF_F_CONST>, grd, blk, lds, s, tab, check);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}
hipError_t wf_launch_pl_solve_batch(const WfSpectral &sp, const WfPressItem *tab, int nm, hipStream_t s) {
    if (sp.pl_nt == 0) { /* three launches (wf_pl_solve_nt) */
        const dim3 grd(sp.nx, (sp.nz + WF_PL_LEVELS - 1) / WF_PL_LEVELS, nm), tri(sp.nx, (sp.ny + 63) / 64, nm);
        hipLaunchKernelGGL(k_pl_y_batch<false>, grd, dim3(512), wf_pl_y_lds(sp), s, tab);
        if (sp.nz <= 128)
            hipLaunchKernelGGL(k_pl_tri_batch<8>, tri, dim3(64 * ((sp.nz + 7) / 8)), 0, s, tab);
        else
            hipLaunchKernelGGL(k_pl_tri_batch<16>, tri, dim3(64 * ((sp.nz + 15) / 16)), 0, s, tab);
        hipLaunchKernelGGL(k_pl_y_batch<true>, grd, dim3(512), wf_pl_y_lds(sp), s, tab);
        return hipGetLastError();
    }
    int tpw, lc;
    wf_pl_shape(sp.ny, sp.nz, sp.pl_nt, &tpw, &lc);
    const size_t lds = (size_t)wf_pl_lds(sp.ny, sp.nz, sp.pl_nt);
#define WF_PL_GO(NT, TPW, LC)                                                                            \
    if (sp.pl_nt == NT && tpw == TPW && lc == LC) {                                                      \
        hipLaunchKernelGGL((k_pl_solve_batch<NT, TPW, LC>), dim3(sp.nx, 1, nm), dim3(NT), lds, s, tab);  \
        return hipGetLastError();                                                                        \
    }
    WF_PL_SOLVES(WF_PL_GO)
#undef WF_PL_GO
    return hipErrorInvalidValue;
}
hipError_t wf_launch_pl_inv_batch(const WfSpectral &sp, const WfPressItem *tab, int nm, hipStream_t s) {
    hipLaunchKernelGGL(k_pl_inv_batch, dim3(sp.npmax, 1, nm), dim3(wf_pl_inv_nt(sp)), sizeof(wf_real) * WF_PL_ROWS * sp.nx, s,
                       tab);
    return hipGetLastError();
}

}  // namespace WF_NS
