/*
 * wf_pressure.hip -- pressure Poisson solve: FFT in x,y, tridiagonal in z.
 *
 * The reference (src/cu/pressure.cu:506-606) forms f on the (Nx-1)(Ny-1)(Nz-1)
 * unique nodes, runs a batched 2-D complex FFT per z-slab, solves one complex
 * tridiagonal system in z per (kx, ky), transforms back and keeps the real part
 * divided by (Nx-1)(Ny-1).  Here f is real, so the x-transform is a real
 * transform that keeps kx bins 0..nx/2 (two rows per complex FFT), the
 * y-transform runs on that half spectrum, and the Thomas solve runs on the
 * nx/2+1 retained kx bins only; the discarded half is the complex conjugate.
 *
 *   P1 k_rhs_fx   : f (or the top pressure plane) -> x half-spectrum   [row-pair group, slab]
 *   P2 k_fy       : y-transform of sp.fy_cols kx columns, one slab      [forward and inverse]
 *   P3 k_thomas   : tridiagonal solve, 64 (kx, ky) systems per workgroup, z split over its waves
 *   P5 k_inv_fx   : inverse x-transform, p, periodic duplicates, max |dp| per workgroup
 *   k_iter_check  : convergence test of the solve
 *
 * Spectral layout: F[k][kx][ky] with ky fastest (column stride ldj), so a
 * y-transform reads whole contiguous columns and the tridiagonal solve reads
 * 64 consecutive ky per wavefront.
 *
 * The variable-density fixed-point loop is controlled on the device
 * (WfIterCtl): every kernel of a solve returns at once after convergence, so
 * the host queues solves without waiting for each norm.
 */
#include "wf_common.h"
#include "wf_fft.h"
#include "wf_kernels.h"
#include "wf_pressure_dev.h"

namespace WF_NS {

/* FP32 chunks of 8 levels: 8 waves per SIMD, so that two 16-wave workgroups
 * share a CU (256x256x128: 512 workgroups, one round of them) */
#define WF_THOMAS_ATTR(LC) __attribute__((amdgpu_waves_per_eu((WF_MIXED && (LC) == 8) ? 8 : 4)))
/* row pairs whose loads are in flight before the one worked on (FP64 P1) */
#define WF_FX_AHEAD 1
#define WF_NX_SHORT 300
/* Row pairs of an x-transform workgroup compiled for length NX, and the most
 * elements a thread of it takes.  NX = 0 and -1 are the run-time lengths up
 * to 300 and above. */
template <int NX>
struct WfFx {
    static constexpr int LEN = (NX > 0) ? NX : (NX == 0) ? WF_NX_SHORT : 1024;
    static constexpr int PAIRS = wf_pairs_for(LEN);
    static constexpr bool RX = NX > 0 && wf_rx_a(NX) != 0; /* register form of the plan */
    /* compile-time lengths (2^m - 1): a row of LEN + 1 lanes per row pair, so
     * that the rows of a wavefront, and with them every address but the
     * column, are uniform; other lengths are packed */
    static constexpr bool UNI = NX > 0;
    static_assert(!UNI || (((NX + 1) & NX) == 0 && PAIRS * (NX + 1) % WF_NT == 0), "whole rows of lanes");
    static constexpr int PER = (PAIRS * (UNI ? NX + 1 : LEN) + WF_NT - 1) / WF_NT;
    /* LDS stride of a sequence: the register form's rows are 16 banks apart */
    __device__ __forceinline__ static int stride(int n) { return RX ? NX + 9 : n; }
};
/* Element pi of this thread among the PAIRS rows of length nx: row pair s and
 * column i, clamped to the last; true where it is one. */
template <int NX>
__device__ __forceinline__ bool wf_fx_elem(int pi, int nx, const WfDiv &by_nx, int *s, int *i) {
    const int t = (int)threadIdx.x + pi * WF_NT;
    if constexpr (WfFx<NX>::UNI) {
        const int x = t & NX;
        *s = __builtin_amdgcn_readfirstlane(t) / (NX + 1);
        *i = min(x, NX - 1);
        return x < NX;
    } else {
        const int n = WfFx<NX>::PAIRS * nx, tc = min(t, n - 1);
        *s = by_nx(tc);
        *i = tc - *s * nx;
        return t < n;
    }
}
/* F at an even ky and the next of a kx column: the spectra of a row pair */
struct alignas(2 * sizeof(wf_real2)) WfPairF {
    wf_real2 a, b;
};
/* Transform of the PAIRS sequences in buf: the register form of the plan from
 * phase A's values on, the in-place plan (NX > 0), or the run-time radices with
 * scratch buffer bufb; tw: twx for the first, else the table in LDS.  Returns
 * the result buffer; ends with a barrier. */
template <int NX, int SIGN>
__device__ __forceinline__ wfc *wf_rx_finish(wfc *buf, wfc *bufb, const wf_real2 *__restrict__ twx) {
    constexpr int PAIRS = WfFx<NX>::PAIRS, NA = wf_rx_a(NX);
    static_assert(PAIRS * wf_rx_b(NX) <= WF_NT && PAIRS * NA <= WF_NT, "a thread takes one DFT of a phase");
    __syncthreads();
    if (threadIdx.x < PAIRS * NA) {
        const int s = threadIdx.x / NA, j = threadIdx.x - s * NA;
        const int o = s * WfFx<NX>::stride(NX);
        wf_rx_phase_b<NX, SIGN>(buf + o, twx, j, [&](int k, wfc X) { bufb[o + k] = X; });
    }
    __syncthreads();
    return bufb;
}
template <int NX>
__device__ __forceinline__ wfc *wf_transform(wfc *buf, wfc *bufb, int n, const int *rad, const wfc *tw) {
    constexpr int PAIRS = WfFx<NX>::PAIRS;
    if constexpr (NX > 0) {
        wf_fft_ip<NX, PAIRS, WF_NT>(buf, tw);
        return buf;
    } else {
        return wf_lds_fft(buf, bufb, n, PAIRS, rad, tw);
    }
}

/* Each pass below is a device function (the body) run by two kernels: the
 * solo kernel k_*, with the operands as arguments, and the batched kernel
 * k_*_batch, which runs the body for member blockIdx.z of an ensemble's
 * size class with that member's operands read from a table.  The grid's x
 * and y are the solo launch's, so every member computes exactly what its
 * solo launch computes. */

/* rho^n = T_inf rho_inf / T^n on every node, once per step. */
__device__ __forceinline__ void wf_density_body(const WfConst &c, const wf_real *T, wf_real *rho) {
    long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q < c.N) rho[q] = c.T_inf * c.rho_inf / T[q];
}
__global__ void k_density(WfConst c, const wf_real *T, wf_real *rho) { wf_density_body(c, T, rho); }

__device__ __forceinline__ void wf_iter_reset_body(WfIterCtl *ctl) {
    ctl->done = 0;
    ctl->iters = 0;
    ctl->solves = 0;
    ctl->err = 0.0;
}
__global__ void k_iter_reset(WfIterCtl *ctl) { wf_iter_reset_body(ctl); }

__global__ __launch_bounds__(WF_NT) void k_iter_check(WfSpectral sp, double tol, double rtol, int m, int max_iter) {
    wf_iter_check_body(sp, tol, rtol, m, max_iter);
}

/* P1: f on slab k (1..nz-1; the top plane for WF_F_TOP) for one group of row
 * pairs (rows ja = 2m, jb = 2m+1 packed as ja + i jb), forward x
 * half-spectrum into F[k][kx][j].  NX > 0 selects the compile-time plan. */
template <int NX, int MODE>
__device__ __forceinline__ void wf_rhs_fx_body(const WfConst &c, const WfSpectral &sp, const WfState &Ys,
                                               const WfState &Yn, const wf_real *p, int block, int nblocks,
                                               int check, const wf_real2 *__restrict__ twx) {
    if (MODE != WF_F_TOP && wf_first_pass_returns(sp.ctl->done, check)) return;
    extern __shared__ wfc smem[];
    __shared__ int rad[WF_MAX_RADICES];
    constexpr int PAIRS = WfFx<NX>::PAIRS, PER = WfFx<NX>::PER;
    constexpr bool RX = WfFx<NX>::RX;
    const int nx = (NX > 0) ? NX : sp.nx, S = WfFx<NX>::stride(nx);
    const int ny = sp.ny, hx = sp.hx, ldj = sp.ldj;
    wfc *tw = smem, *bufa = RX ? smem : smem + nx, *bufb = bufa + PAIRS * S;
    int g, ks;
    wf_tile_decode_at(block, nblocks, sp.ngroups, (MODE == WF_F_TOP) ? 1 : sp.nz - 1, &g, &ks);
    const int k = (MODE == WF_F_TOP) ? c.Nz - 1 : 1 + ks;
    const int j0 = 2 * g * PAIRS;
    if constexpr (!RX)
        for (int t = threadIdx.x; t < nx; t += blockDim.x) tw[t] = *(const wfc *)&sp.twx[t];
    if (NX <= 0 && threadIdx.x < WF_MAX_RADICES) rad[threadIdx.x] = sp.radx[threadIdx.x];
    const WfDiv by_nx(nx);
#if !WF_MIXED
    if constexpr (MODE == WF_F_ITER && WfFx<NX>::UNI) {
        /* What bounds this pass in FP64 is the cache's data path: 18 values a
         * row pair by wf_pair_load against 30 node by node.  A row pair per
         * batch, WF_FX_AHEAD batches of loads in flight before the one that is
         * worked on, which the scheduling barriers keep so.  us at
         * 256x256x128: node by node 76, with none ahead 69, one 67.5, two
         * 68.4.  FP32, whose input is half of that, gains nothing (32.4-33.9
         * against 32.7). */
        const wf_real dzc = c.zc[WF_ZC * k + WF_Z_DZC];
        WfPairIn v[PER];
        const auto load = [&](int pi) {
            int s, i;
            (void)wf_fx_elem<NX>(pi, nx, by_nx, &s, &i);
            wf_pair_load(c, sp.A, sp.rho, p, i, min(j0 + 2 * s, ny - 1), k, v[pi]);
        };
#pragma unroll
        for (int pi = 0; pi < PER + WF_FX_AHEAD; pi++) {
            if (pi < PER) load(pi);
            __builtin_amdgcn_sched_barrier(0);
            if (pi < WF_FX_AHEAD) continue;
            const int po = pi - WF_FX_AHEAD;
            int s, i;
            const bool ok = wf_fx_elem<NX>(po, nx, by_nx, &s, &i);
            const int ja = j0 + 2 * s, jb = ja + 1;
            wf_real fa, fb;
            wf_pair_eval(c, v[po], i, dzc, &fa, &fb);
            if (ok) bufa[s * S + i] = wfc{(ja < ny) ? fa : WR(0.0), (jb < ny) ? fb : WR(0.0)};
            __builtin_amdgcn_sched_barrier(0);
        }
    } else
#endif
    {
        /* one row pair per batch: both cells' loads unconditional (indices clamped
         * to a valid node, padding results dropped), so a batch is one basic block
         * with all 28 loads in flight; the scheduling barrier keeps the batches
         * apart, which bounds the registers */
#pragma unroll
        for (int pi = 0; pi < PER; pi++) {
            if (NX <= 0 && pi * WF_NT >= PAIRS * nx) break;
            int s, i;
            const bool ok = wf_fx_elem<NX>(pi, nx, by_nx, &s, &i);
            const int ja = j0 + 2 * s, jb = ja + 1;
            if constexpr (MODE != WF_F_FIRST) {
                const wf_real fa = wf_fx_input<MODE>(c, sp, Ys, Yn, p, i, (ja < ny) ? ja : ny - 1, k);
                const wf_real fb = wf_fx_input<MODE>(c, sp, Ys, Yn, p, i, (jb < ny) ? jb : ny - 1, k);
                if (ok) bufa[s * S + i] = wfc{(ja < ny) ? fa : WR(0.0), (jb < ny) ? fb : WR(0.0)};
                __builtin_amdgcn_sched_barrier(0);
            } else if (ok) {
                wf_real fa = WR(0.0), fb = WR(0.0);
                if (ja < ny) fa = wf_fx_input<MODE>(c, sp, Ys, Yn, p, i, ja, k);
                if (jb < ny) fb = wf_fx_input<MODE>(c, sp, Ys, Yn, p, i, jb, k);
                bufa[s * S + i] = wfc{fa, fb};
            }
        }
    }
    __syncthreads();
    wfc *res;
    if constexpr (RX) {
        constexpr int NA = wf_rx_a(NX), NB = wf_rx_b(NX);
        if (threadIdx.x < PAIRS * NB) {
            const int s = threadIdx.x / NB, g = threadIdx.x - s * NB;
            wfc x[NA]; /* phase A writes where it read */
#pragma unroll
            for (int m = 0; m < NA; m++) x[m] = bufa[s * S + g + NB * m];
            wf_rx_phase_a<NX, -1>(x, bufa + s * S, twx, g);
        }
        res = wf_rx_finish<NX, -1>(bufa, bufb, twx);
    } else {
        res = wf_transform<NX>(bufa, bufb, nx, rad, tw);
    }
    /* a thread unpacks both rows of a pair */
    wf_real2 *dst = (MODE == WF_F_TOP) ? sp.Ptop : sp.F + (long)k * hx * ldj;
    for (int t = threadIdx.x; t < PAIRS * hx; t += WF_NT) {
        const int s = t % PAIRS, r = t / PAIRS, ja = j0 + 2 * s;
        const int rm = (r == 0) ? 0 : nx - r;
        wfc A, B;
        wf_unpack_pair(res[s * S + r], res[s * S + rm], &A, &B);
        wf_real2 *d = dst + (unsigned)(r * ldj + ja);
        if (ja + 1 < ny)
            *(WfPairF *)d = WfPairF{wf_make2(A.re, A.im), wf_make2(B.re, B.im)};
        else if (ja < ny)
            *d = wf_make2(A.re, A.im);
    }
}
template <int NX, int MODE>
__global__ __launch_bounds__(WF_NT) void k_rhs_fx(WfConst c, WfSpectral sp, WfState Ys, WfState Yn,
                                                  const wf_real *p, double tol, double rtol, int check,
                                                  int max_iter, const wf_real2 *__restrict__ twx) {
    const int b = wf_checked_block(sp, tol, rtol, check, max_iter);
    if (b >= 0) wf_rhs_fx_body<NX, MODE>(c, sp, Ys, Yn, p, b, (int)gridDim.x - (check >= 0), check, twx);
}

/* P2/P4: y-transform of sp.fy_cols kx columns (each contiguous over ky) of
 * slab slab0 + blockIdx.y; sign -1 forward, +1 inverse. */
template <int NY, int SIGN>
__device__ __forceinline__ void wf_fy_f2(const WfSpectral &sp, wf_real2 *base, wfc *buf, int r0,
                                         const wf_real2 *__restrict__ twy) {
    constexpr int N1 = wf_f2_n1(NY), N2 = wf_f2_n2(NY), NSEQ = wf_f2_nseq(NY);
    const int hx = sp.hx, ldj = sp.ldj;
    const int t = threadIdx.x;
    if (t < N1 * NSEQ) {
        const int s = t / N1, n1 = t - s * N1;
        wf_f2_phase_a<N1, N2, SIGN>(buf, twy, s, n1, [&](int ss, int n) {
            wfc v = {WR(0.0), WR(0.0)};
            if (r0 + ss < hx) {
                const wf_real2 x = base[(long)(r0 + ss) * ldj + n];
                v.re = x.x;
                v.im = x.y;
            }
            return v;
        });
    }
    __syncthreads();
    if (t < N2 * NSEQ) {
        const int s = t / N2, k2 = t - s * N2;
        if (r0 + s < hx) {
            wf_real2 *col = base + (long)(r0 + s) * ldj + k2;
            wf_f2_phase_b<N1, N2, SIGN>(buf, twy, s, k2, [&](int k1, wfc X) { col[N2 * k1] = wf_make2(X.re, X.im); });
        }
    }
}

/* twy: the y twiddle table again, as a read-only argument of its own, so
 * that the compiler may keep its loads apart from the column stores (scalar
 * loads for the DFT constants, vector loads issued early for the rest). */
template <int NY, bool BATCH>
__device__ __forceinline__ void wf_fy_body(const WfSpectral &sp, wf_real2 *buf, long slab_stride, int slab0, int sign,
                                           int guarded, const wf_real2 *__restrict__ twy) {
    if (guarded && wf_pass_returns(sp.ctl->done)) return;
    extern __shared__ wfc smem[];
    wf_real2 *base = buf + (long)(slab0 + blockIdx.y) * slab_stride;
    const int cols = sp.fy_cols;
    /* first column: the in-place plan's column count is a compile-time one */
    const int r0 = blockIdx.x * ((NY > 0 && wf_f2_n1(NY) == 0) ? wf_fy_ip_cols(NY, BATCH) : cols);
    if constexpr (NY > 0 && wf_f2_n1(NY) != 0) {
        if (sign < 0)
            wf_fy_f2<NY, -1>(sp, base, smem, r0, twy);
        else
            wf_fy_f2<NY, 1>(sp, base, smem, r0, twy);
    } else if constexpr (NY > 0) {
        /* compile-time in-place plan (lengths without a two-factor split,
         * such as the prime 127): wf_fy_ip_cols(NY, BATCH) columns in LDS */
        constexpr int COLS = wf_fy_ip_cols(NY, BATCH);
        const int hx = sp.hx, ldj = sp.ldj;
        wfc *tw = smem, *bufa = smem + NY;
        for (int t = threadIdx.x; t < NY; t += blockDim.x) {
            const wf_real2 w = twy[t];
            tw[t].re = w.x;
            tw[t].im = (sign > 0) ? -w.y : w.y;
        }
        for (int t = threadIdx.x; t < COLS * NY; t += blockDim.x) {
            const int cc = t / NY, jj = t - cc * NY;
            wfc v = {WR(0.0), WR(0.0)};
            if (r0 + cc < hx) {
                const wf_real2 x = base[(long)(r0 + cc) * ldj + jj];
                v.re = x.x;
                v.im = x.y;
            }
            bufa[t] = v;
        }
        __syncthreads();
        wf_fft_ip<NY, COLS, WF_NT>(bufa, tw);
        for (int t = threadIdx.x; t < COLS * NY; t += blockDim.x) {
            const int cc = t / NY, jj = t - cc * NY;
            if (r0 + cc < hx) base[(long)(r0 + cc) * ldj + jj] = wf_make2(bufa[t].re, bufa[t].im);
        }
    } else {
        __shared__ int rad[WF_MAX_RADICES];
        const int ny = sp.ny, hx = sp.hx, ldj = sp.ldj;
        wfc *tw = smem, *bufa = smem + ny, *bufb = bufa + cols * ny;
        for (int t = threadIdx.x; t < ny; t += blockDim.x) {
            wf_real2 w = sp.twy[t];
            tw[t].re = w.x;
            tw[t].im = (sign > 0) ? -w.y : w.y;
        }
        if (threadIdx.x < WF_MAX_RADICES) rad[threadIdx.x] = sp.rady[threadIdx.x];
        const WfDiv by_ny(ny);
        constexpr int B = 4;
        for (int t0 = threadIdx.x; t0 < cols * ny; t0 += B * WF_NT) {
            wf_real2 x[B];
#pragma unroll
            for (int u = 0; u < B; u++) {
                const int t = min(t0 + u * WF_NT, cols * ny - 1);
                const int cc = by_ny(t), jj = t - cc * ny;
                x[u] = base[(long)min(r0 + cc, hx - 1) * ldj + jj];
            }
#pragma unroll
            for (int u = 0; u < B; u++)
                if (t0 + u * WF_NT < cols * ny) bufa[t0 + u * WF_NT] = wfc{x[u].x, x[u].y};
        }
        __syncthreads();
        wfc *res = wf_lds_fft(bufa, bufb, ny, cols, rad, tw);
        for (int t = threadIdx.x; t < cols * ny; t += blockDim.x) {
            const int cc = by_ny(t), jj = t - cc * ny;
            if (r0 + cc < hx) base[(long)(r0 + cc) * ldj + jj] = wf_make2(res[t].re, res[t].im);
        }
    }
}
template <int NY>
__global__ __launch_bounds__(WF_NT) void k_fy(WfSpectral sp, wf_real2 *buf, long slab_stride, int slab0, int sign,
                                              int guarded, const wf_real2 *__restrict__ twy) {
    wf_fy_body<NY, false>(sp, buf, slab_stride, slab0, sign, guarded, twy);
}

__global__ void k_pivots(WfSpectral sp, double *UB) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    const int r = blockIdx.y;
    if (j >= sp.ny) return;
    const int nz = sp.nz, lc = sp.thomas_lc;
    const long slab = (long)sp.hx * sp.ldj;
    const long o = (long)r * sp.ldj + j;
    const double K2 = sp.kx2d[r] + sp.ky2d[j];
    const double c0 = sp.c0a - 0.5 * sp.dz0 * K2 - sp.c0b;
    double u = sp.b0;
    for (int k = 1; k < nz; k++) {
        if (k % lc == 0) UB[o + (k / lc) * slab] = u; /* u_{k-1} enters chunk k/lc */
        double l;
        u = wf_pivot_next<double>(sp, u, k, K2, c0, &l);
    }
}

/* P3: tridiagonal solve for 64 consecutive ky of one kx column per workgroup,
 * in place in F (src/cu/pressure.cu:418-443 with the right-hand side of
 * 473-504):  y_0 = d_0, y_k = d_k - L_k y_{k-1};  x_{nz-1} = y_{nz-1}/u_{nz-1},
 * x_k = (y_k - c_k x_{k+1})/u_k, in arithmetic type TA.
 * Wave w owns levels [w LC, w LC + LC) of its systems and keeps them in
 * registers.  Both recurrences are affine in the value entering the chunk, so
 * each wave runs them from a zero entry value while carrying the coefficient
 * of the entry value (products of -L_k, resp. of -c_k/u_k); the waves then
 * combine their chunk ends through LDS in order and add the correction.
 * A lane holds NC components of its system (ky j of kx r): both (64 systems
 * to a wave), or component comp alone (32 systems).  Loads go out before what
 * uses them (see SPREAD) and no level has a branch of its own: the levels above the top read the top's
 * entries, and the tables (padded to whole chunks: a = c = 0, beta = 1) keep
 * their values finite and apart from the others. */
template <typename TA, int NC>
struct WfThomasLds {
    struct alignas(NC * sizeof(TA)) V { /* one LDS access (two would meet in the banks) */
        TA c[NC];
    } v[WF_THOMAS_MAX_CHUNKS][64];
    TA g[WF_THOMAS_MAX_CHUNKS][64];
};
template <int LC, typename TA, int NC>
__device__ __forceinline__ void wf_thomas_solve(const WfSpectral &sp, WfThomasLds<TA, NC> &L, int j, int r,
                                                int comp) {
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int C = blockDim.x >> 6;
    const int nz = sp.nz;
    const bool ok = j < sp.ny;
    const long slab = (long)sp.hx * sp.ldj;
    const long row = (long)r * sp.ldj; /* uniform: a level's entries are at a scalar base + at */
    const unsigned jj = ok ? j : 0, at = 2 * jj + comp;
    const int k0 = w * LC;
    /* the operands of the pivots first: their chain of divisions runs while the
     * right-hand sides arrive */
    TA u = w ? (TA)(sp.UB + row + w * slab)[jj] : (TA)sp.b0; /* pivot entering the chunk */
    const TA K2 = wf_tab<TA>(sp.kx2, sp.kx2d, r) + wf_tab<TA>(sp.ky2, sp.ky2d, jj);
    __builtin_amdgcn_sched_barrier(0);
    TA y[LC][NC], g[LC], ru[LC], pt[NC];
    const auto load = [&](int t) {
        int k = min(k0 + t, nz - 1);
        if (t == 0) k = max(k, 1); /* level 0 takes level 1's right-hand side */
#pragma unroll
        for (int q = 0; q < NC; q++) y[t][q] = (TA)((const wf_real *)(sp.F + row + k * slab))[at + q];
    };
    /* FP64 (one workgroup per CU): a level's load before each level's
     * divisions, so that the memory has work while a round computes (all
     * first: 33.0 us against 31.8 at 256x256x128, 68 against 51 at 160 levels) */
    constexpr bool SPREAD = sizeof(TA) * NC == 16;
    if constexpr (!SPREAD) {
#pragma unroll
        for (int t = 0; t < LC; t++) load(t);
    }
#pragma unroll
    for (int q = 0; q < NC; q++)
        pt[q] = (k0 + LC >= nz) ? (TA)((const wf_real *)(sp.Ptop + row))[at + q] : (TA)0.0;
    const TA half_dz0 = (TA)0.5 * (TA)sp.dz0;
    const TA c0 = (TA)sp.c0a - half_dz0 * K2 - (TA)sp.c0b;
    const TA ck0 = w ? wf_tab<TA>(sp.tc, sp.tcd, k0) : c0; /* c_{k0} */
    /* the pivots u_k (wf_pivot_next's operations), L_k and 1/u_k */
#pragma unroll
    for (int t = 0; t < LC; t++) {
        if constexpr (SPREAD) load(t);
        const int km = (t > 0) ? k0 + t - 1 : max(k0 - 1, 0);
        const TA bk = -(K2 + wf_tab<TA>(sp.beta, sp.betad, k0 + t));
        const TA l = wf_tab<TA>(sp.ta, sp.tad, km) / u;
        u = bk - l * ((t == 1) ? ck0 : wf_tab<TA>(sp.tc, sp.tcd, km));
        g[t] = l;
        if (t == 0) {
            u = w ? u : (TA)sp.b0;
            g[0] = w ? l : (TA)0.0;
        }
        ru[t] = (TA)1.0 / u;
        if constexpr (SPREAD) __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_sched_barrier(0);
    /* forward elimination, entry value 0, coefficient G of the entry value */
    TA acc[NC], G = (TA)1.0;
#pragma unroll
    for (int q = 0; q < NC; q++) {
        if (k0 + LC >= nz) pt[q] = pt[q] / (TA)sp.top_div;
        acc[q] = (TA)0.0;
        y[0][q] = w ? y[0][q] : half_dz0 * y[0][q];
    }
#pragma unroll
    for (int t = 0; t < LC; t++) {
        const TA m = g[t];
#pragma unroll
        for (int q = 0; q < NC; q++) {
            const TA d = y[t][q] - ((k0 + t == nz - 1) ? pt[q] : (TA)0.0);
            y[t][q] = acc[q] = d - m * acc[q];
        }
        g[t] = G = -m * G;
    }
    typename WfThomasLds<TA, NC>::V e;
#pragma unroll
    for (int q = 0; q < NC; q++) e.c[q] = acc[q];
    L.v[w][lane] = e;
    L.g[w][lane] = G;
    __syncthreads();
    TA Y[NC];
#pragma unroll
    for (int q = 0; q < NC; q++) Y[q] = (TA)0.0;
#pragma unroll 4
    for (int s = 0; s < w; s++) {
        const TA gs = L.g[s][lane];
        const auto vs = L.v[s][lane];
#pragma unroll
        for (int q = 0; q < NC; q++) Y[q] = vs.c[q] + gs * Y[q];
    }
#pragma unroll
    for (int t = 0; t < LC; t++)
#pragma unroll
        for (int q = 0; q < NC; q++) y[t][q] = y[t][q] + g[t] * Y[q];
    __syncthreads();
    /* back substitution, entry value x_{k0+LC} = 0, coefficient H */
    TA xa[NC], H = (TA)1.0;
#pragma unroll
    for (int q = 0; q < NC; q++) xa[q] = (TA)0.0;
#pragma unroll
    for (int t = LC - 1; t >= 0; t--) {
        const TA ck = (t == 0) ? ck0 : wf_tab<TA>(sp.tc, sp.tcd, k0 + t); /* 0 at the top and above */
#pragma unroll
        for (int q = 0; q < NC; q++) y[t][q] = xa[q] = (y[t][q] - ck * xa[q]) * ru[t];
        g[t] = H = (-ck * ru[t]) * H;
    }
#pragma unroll
    for (int q = 0; q < NC; q++) e.c[q] = xa[q];
    L.v[w][lane] = e;
    L.g[w][lane] = H;
    __syncthreads();
    TA X[NC];
#pragma unroll
    for (int q = 0; q < NC; q++) X[q] = (TA)0.0;
#pragma unroll 4
    for (int s = C - 1; s > w; s--) {
        const TA hs = L.g[s][lane];
        const auto vs = L.v[s][lane];
#pragma unroll
        for (int q = 0; q < NC; q++) X[q] = vs.c[q] + hs * X[q];
    }
    if (!ok) return;
#pragma unroll
    for (int t = 0; t < LC; t++) {
        const int k = k0 + t;
        if (k >= nz) break;
#pragma unroll
        for (int q = 0; q < NC; q++)
            ((wf_real *)(sp.F + row + k * slab))[at + q] = (wf_real)(y[t][q] + g[t] * X[q]);
    }
}

template <int LC>
__device__ __forceinline__ void wf_thomas_body(const WfSpectral &sp) {
    if (wf_pass_returns(sp.ctl->done)) return;
    const int lane = threadIdx.x & 63, jlo = blockIdx.x * 64;
#if WF_MIXED
    /* a tile of 64 systems holding one of the lowest wavenumbers (kx index
     * below low_kx, ky index within low_ky of 0 or of ny) is solved in FP64:
     * those systems are singular or nearly so under the Neumann z conditions.
     * Two workgroups share such a tile, a component of a system to a lane: the
     * kernel can then be held to 64 registers (two workgroups of 16 waves to a
     * CU; 18 of the FP64 half's values spill, 68 bytes a lane, which the FP32
     * tiles do not touch), and its chain of FP64 divisions and
     * combines, the longest of the launch, has half the work.  The second
     * halves are low_kx rows of workgroups before the kx columns'.  us, with
     * a complex FP64 system to a lane, 105 registers and a branch per level
     * before: 64x64x32 8.6 -> 5.3, 128x128x64 10.8 -> 8.2, 201x151x81 16 ->
     * 13.8, 256x256x128 23.2 -> 18.8 (16.2 without the FP64 systems, whose
     * extra workgroups there start when the first others end); in FP64, all
     * systems complex, 256x256x64 16.4 -> 15.4, 256x256x128 as before (32.4).
     * Both halves by one workgroup in turn: 9.5, 16.1, 20.7, 29.4. */
    __shared__ union {
        WfThomasLds<float, 2> f;
        WfThomasLds<double, 1> d;
    } L;
    const int second = (int)blockIdx.y < sp.low_kx;
    const int r = second ? (int)blockIdx.y : (int)blockIdx.y - sp.low_kx;
    const int jhi = (jlo + 63 < sp.ny - 1) ? jlo + 63 : sp.ny - 1;
    const bool low = r < sp.low_kx && (jlo < sp.low_ky || sp.ny - jhi < sp.low_ky);
    if (low)
        wf_thomas_solve<LC, double, 1>(sp, L.d, jlo + 32 * second + (lane >> 1), r, lane & 1);
    else if (!second)
        wf_thomas_solve<LC, float, 2>(sp, L.f, jlo + lane, r, 0);
#else
    /* a component to a lane also where 16 levels of both (72 spilled
     * registers) do not fit: 256x256x160, 47.8 us
     * (51.6 before with 41 of them, 73 in this form of the solve) */
    constexpr int NC = (LC > 8) ? 1 : 2;
    __shared__ WfThomasLds<double, NC> L;
    if constexpr (NC == 1)
        wf_thomas_solve<LC, double, 1>(sp, L, (int)blockIdx.x * 32 + (lane >> 1), (int)blockIdx.y, lane & 1);
    else
        wf_thomas_solve<LC, double, 2>(sp, L, jlo + lane, (int)blockIdx.y, 0);
#endif
}
template <int LC>
__global__ __launch_bounds__(64 * WF_THOMAS_MAX_CHUNKS) WF_THOMAS_ATTR(LC) void k_thomas(WfSpectral sp) {
    wf_thomas_body<LC>(sp);
}

#if !WF_MIXED /* FP64 only: it has no FP64 path for the lowest wavenumbers */
/* P3 for nz <= 2 WF_THOMAS_MAX_CHUNKS LC (LC = 4: the 128-level grids): the
 * same chunked solve with each wave taking 32 systems and its two half-waves
 * two consecutive chunks, so a 16-wave workgroup covers 32 chunks with a
 * quarter of the registers per lane; two workgroups then fit a CU and one's
 * loads overlap the other's pivot chain and combine.  The tridiagonal
 * coefficient tables are staged in LDS (the chunk index, and so k, differs
 * between the half-waves); the pivots are re-formed with the operations of
 * k_pivots. */
template <int LC>
__device__ __forceinline__ void wf_thomas_h_body(const WfSpectral &sp) {
    if (wf_pass_returns(sp.ctl->done)) return;
    constexpr int CH = 2 * WF_THOMAS_MAX_CHUNKS;
    __shared__ wf_real2 sv[CH][32];
    __shared__ wf_real sg[CH][32];
    __shared__ wf_real s_ta[CH * LC], s_tc[CH * LC], s_beta[CH * LC];
    const int nz = sp.nz;
    for (int t = threadIdx.x; t < nz; t += blockDim.x) {
        s_ta[t] = (t < nz - 1) ? sp.ta[t] : WR(0.0);
        s_tc[t] = (t < nz - 1) ? sp.tc[t] : WR(0.0);
        s_beta[t] = sp.beta[t];
    }
    const int lane = threadIdx.x & 63, ls = lane & 31;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ch = 2 * w + (lane >> 5);
    const int C = 2 * (int)(blockDim.x >> 6);
    const int j = blockIdx.x * 32 + ls, r = blockIdx.y;
    const bool ok = j < sp.ny;
    const long slab = (long)sp.hx * sp.ldj;
    const long o = (long)r * sp.ldj + (ok ? j : 0);
    const int k0 = ch * LC;
    const wf_real K2 = ok ? sp.kx2[r] + sp.ky2[j] : WR(0.0);
    const wf_real c0 = sp.c0a - WR(0.5) * sp.dz0 * K2 - sp.c0b;
    __syncthreads();
    wf_real2 y[LC];
    wf_real g[LC], ru[LC];
    /* pivot entering the chunk (a chunk wholly above the top, possible when the
     * chunk count is odd, has no table entry and no levels) */
    wf_real u = (ch > 0 && ok && k0 < nz) ? sp.UB[o + ch * slab] : sp.b0;
#pragma unroll
    for (int t = 0; t < LC; t++) {
        const int k = k0 + t;
        y[t] = wf_make2(WR(0.0), WR(0.0));
        g[t] = WR(0.0);
        ru[t] = WR(0.0);
        if (ok && k < nz) {
            if (k == 0) {
                wf_real2 f1 = sp.F[o + slab];
                y[t] = wf_make2(WR(0.5) * sp.dz0 * f1.x, WR(0.5) * sp.dz0 * f1.y);
                u = sp.b0;
            } else {
                wf_real2 d = sp.F[o + k * slab];
                if (k == nz - 1) {
                    wf_real2 pt = sp.Ptop[o];
                    d.x = d.x - pt.x / sp.top_div;
                    d.y = d.y - pt.y / sp.top_div;
                }
                y[t] = d;
                /* wf_pivot_next with the staged tables */
                const wf_real ck1 = (k == 1) ? c0 : s_tc[k - 1];
                const wf_real bk = (k == nz - 1) ? -(K2 + sp.beta_top) : -(K2 + s_beta[k]);
                const wf_real l = s_ta[k - 1] / u;
                u = bk - l * ck1;
                g[t] = l;
            }
            ru[t] = WR(1.0) / u;
        }
    }
    /* forward elimination, entry value 0, coefficient G of the entry value */
    wf_real2 acc = wf_make2(WR(0.0), WR(0.0));
    wf_real G = WR(1.0);
#pragma unroll
    for (int t = 0; t < LC; t++) {
        const int k = k0 + t;
        if (k == 0) {
            acc = y[0];
            G = WR(0.0);
        } else {
            const wf_real m = g[t];
            acc.x = y[t].x - m * acc.x;
            acc.y = y[t].y - m * acc.y;
            G = -m * G;
            y[t] = acc;
        }
        g[t] = G;
    }
    sv[ch][ls] = acc;
    sg[ch][ls] = G;
    __syncthreads();
    wf_real2 Y = wf_make2(WR(0.0), WR(0.0));
    for (int q = 0; q < ch; q++) {
        const wf_real2 e = sv[q][ls];
        const wf_real gq = sg[q][ls];
        Y.x = e.x + gq * Y.x;
        Y.y = e.y + gq * Y.y;
    }
#pragma unroll
    for (int t = 0; t < LC; t++) {
        y[t].x = y[t].x + g[t] * Y.x;
        y[t].y = y[t].y + g[t] * Y.y;
    }
    __syncthreads();
    /* back substitution, entry value x_{k0+LC} = 0, coefficient H */
    wf_real2 xa = wf_make2(WR(0.0), WR(0.0));
    wf_real H = WR(1.0);
#pragma unroll
    for (int t = LC - 1; t >= 0; t--) {
        const int k = k0 + t;
        if (k >= nz) continue;
        if (k == nz - 1) {
            xa.x = y[t].x * ru[t];
            xa.y = y[t].y * ru[t];
            H = WR(0.0);
        } else {
            const wf_real ck = (k == 0) ? c0 : s_tc[k];
            xa.x = (y[t].x - ck * xa.x) * ru[t];
            xa.y = (y[t].y - ck * xa.y) * ru[t];
            H = (-ck * ru[t]) * H;
        }
        y[t] = xa;
        g[t] = H;
    }
    sv[ch][ls] = xa;
    sg[ch][ls] = H;
    __syncthreads();
    wf_real2 X = wf_make2(WR(0.0), WR(0.0));
    for (int q = C - 1; q > ch; q--) {
        const wf_real2 e = sv[q][ls];
        const wf_real hq = sg[q][ls];
        X.x = e.x + hq * X.x;
        X.y = e.y + hq * X.y;
    }
    if (!ok) return;
#pragma unroll
    for (int t = 0; t < LC; t++) {
        const int k = k0 + t;
        if (k < nz) sp.F[o + k * slab] = wf_make2(y[t].x + g[t] * X.x, y[t].y + g[t] * X.y);
    }
}
template <int LC>
__global__ __launch_bounds__(64 * WF_THOMAS_MAX_CHUNKS) __attribute__((amdgpu_waves_per_eu(8))) void k_thomas_h(
    WfSpectral sp) { /* 8 waves per SIMD: <= 64 VGPRs, which this fits without spills */
    wf_thomas_h_body<LC>(sp);
}
#endif

/* P5: inverse x-transform of one row-pair group of slab k (0..nz-1):
 * p = Re(.)/(nx ny) (multiplied by the reciprocal) on unique nodes, duplicate
 * planes i = Nx-1 and j = Ny-1 set from their images [Q6], and max
 * |p_new - p_old| of the workgroup into sp.pmax[blockIdx.x].  The last
 * workgroup refreshes the periodic copies on the top plane, which the solve
 * never writes on unique nodes. */

/* P5: every global load (half spectra, the old p of the
 * group's unique nodes and of their periodic duplicates) is issued before the
 * transform, unconditionally with clamped indices, so a workgroup waits for
 * one memory round trip; the stores of the duplicates use no branches inside
 * the main loop (column i = Nx-1 from threads 0 .. 2*PAIRS-1, row j = Ny-1 by
 * the group that holds j = 0). */
template <int NX>
__device__ __forceinline__ void wf_inv_fx_rows(const WfConst &c, const WfSpectral &sp, wf_real *p, wfc *smem,
                                                  const int *rad, int g, int k, wf_real &dmax, wf_real &pabs,
                                               const wf_real2 *__restrict__ twx) {
    constexpr int PAIRS = WfFx<NX>::PAIRS, PER = WfFx<NX>::PER;
    constexpr int PERY = (WfFx<NX>::LEN + 1 + WF_NT - 1) / WF_NT; /* row j = Ny-1: i = 0 .. Nx-1 */
    constexpr bool RX = WfFx<NX>::RX;
    const int nx = (NX > 0) ? NX : sp.nx, S = WfFx<NX>::stride(nx);
    const WfDiv by_nx(nx);
    const int ny = sp.ny, hx = sp.hx, ldj = sp.ldj;
    const int j0 = 2 * g * PAIRS;
    const wf_real2 *src = sp.F + (long)k * hx * ldj;
    const wf_real inv_scale = WR(1.0) / ((wf_real)nx * (wf_real)ny);
    const int tid = threadIdx.x;
    wfc *tw = smem, *buf = RX ? smem : smem + nx;
    /* loads: half spectra of a row pair (thread t -> pair t % PAIRS and bin, or
     * phase A's block, t / PAIRS, so consecutive threads read consecutive ky of
     * one kx column) */
    constexpr int NA = RX ? wf_rx_a(NX) : PER, NB = RX ? wf_rx_b(NX) : 1;
    WfPairF xp[NA];
    const int sA = tid % PAIRS, gA = tid / PAIRS, jA = j0 + 2 * sA;
    const int jl = min(jA, (ny - 1) & ~1);
#pragma unroll
    for (int m = 0; m < NA; m++) {
        if (NX <= 0 && m * WF_NT >= PAIRS * nx) break;
        const int r = RX ? min(gA, NB - 1) + NB * m : min(gA + m * (WF_NT / PAIRS), nx - 1);
        const int rr = (r >= hx) ? nx - r : r;
        xp[m] = *(const WfPairF *)&src[(unsigned)(rr * ldj + jl)];
    }
    /* old p of the unique nodes */
    wf_real pa[PER], pb[PER];
#pragma unroll
    for (int pi = 0; pi < PER; pi++) {
        if (NX <= 0 && pi * WF_NT >= PAIRS * nx) break;
        int s, i;
        (void)wf_fx_elem<NX>(pi, nx, by_nx, &s, &i);
        const int ja = j0 + 2 * s, jb = ja + 1;
        pa[pi] = wf_ldp(p + wf_q(c, 0, (ja < ny) ? ja : ny - 1, k), (unsigned)i);
        pb[pi] = wf_ldp(p + wf_q(c, 0, (jb < ny) ? jb : ny - 1, k), (unsigned)i);
    }
    /* old p of the duplicates: column i = Nx-1 of the group's rows, and
     * row j = Ny-1 (i = 0 .. Nx-1) when the group holds j = 0 */
    const int jr = j0 + ((tid < 2 * PAIRS) ? tid : 0);
    const wf_real pdx = p[wf_q(c, c.Nx - 1, (jr < ny) ? jr : ny - 1, k)];
    wf_real pdy[PERY];
    if (g == 0) {
#pragma unroll
        for (int pi = 0; pi < PERY; pi++) {
            const int i = tid + pi * WF_NT;
            pdy[pi] = p[wf_q(c, (i <= nx) ? i : nx, c.Ny - 1, k)];
        }
    }
    /* entry m of this thread as a bin of the packed pair */
    const auto packed = [&](int m, bool conj) {
        const wfc A = {xp[m].a.x, xp[m].a.y};
        wfc B = {WR(0.0), WR(0.0)};
        if (jA + 1 < ny) B = wfc{xp[m].b.x, xp[m].b.y};
        return wf_pack_pair(A, B, conj);
    };
    if constexpr (RX) {
        if (tid < PAIRS * NB) {
            wfc x[NA];
#pragma unroll
            for (int m = 0; m < NA; m++) x[m] = packed(m, gA + NB * m >= NX / 2 + 1);
            wf_rx_phase_a<NX, 1>(x, buf + sA * S, twx, gA);
        }
        buf = wf_rx_finish<NX, 1>(buf, buf + PAIRS * S, twx);
    } else {
        for (int t = tid; t < nx; t += WF_NT) {
            const wf_real2 w = sp.twx[t];
            tw[t].re = w.x;
            tw[t].im = -w.y;
        }
#pragma unroll
        for (int m = 0; m < NA; m++) {
            if (NX <= 0 && m * WF_NT >= PAIRS * nx) break;
            const int r = gA + m * (WF_NT / PAIRS);
            if (r < nx) buf[sA * nx + r] = packed(m, r >= hx);
        }
        __syncthreads();
        buf = wf_transform<NX>(buf, buf + PAIRS * nx, nx, rad, tw);
    }
    /* unique nodes */
#pragma unroll
    for (int pi = 0; pi < PER; pi++) {
        if (NX <= 0 && pi * WF_NT >= PAIRS * nx) break;
        int s, i;
        const bool ok = wf_fx_elem<NX>(pi, nx, by_nx, &s, &i);
        const int ja = j0 + 2 * s, jb = ja + 1;
        if (ok) {
            const wfc v = buf[s * S + i];
            if (ja < ny) {
                const wf_real pv = v.re * inv_scale;
                const wf_real d = fabs(pv - pa[pi]);
                dmax = (d > dmax) ? d : dmax;
                if constexpr (WF_MIXED) pabs = (fabs(pv) > pabs) ? fabs(pv) : pabs;
                (p + wf_q(c, 0, ja, k))[(unsigned)i] = pv;
            }
            if (jb < ny) {
                const wf_real pv = v.im * inv_scale;
                const wf_real d = fabs(pv - pb[pi]);
                dmax = (d > dmax) ? d : dmax;
                if constexpr (WF_MIXED) pabs = (fabs(pv) > pabs) ? fabs(pv) : pabs;
                (p + wf_q(c, 0, jb, k))[(unsigned)i] = pv;
            }
        }
    }
    /* duplicate column i = Nx-1 of rows j0 .. j0 + 2 PAIRS - 1 (value of i = 0) */
    if (tid < 2 * PAIRS && jr < ny) {
        const wfc v = buf[(tid >> 1) * S];
        const wf_real pv = ((tid & 1) ? v.im : v.re) * inv_scale;
        const wf_real d = fabs(pv - pdx);
        dmax = (d > dmax) ? d : dmax;
        p[wf_q(c, c.Nx - 1, jr, k)] = pv;
    }
    /* duplicate row j = Ny-1 (value of j = 0; its corner i = Nx-1 that of i = 0) */
    if (g == 0) {
#pragma unroll
        for (int pi = 0; pi < PERY; pi++) {
            const int i = tid + pi * WF_NT;
            if (i <= nx) {
                const wf_real pv = buf[(i < nx) ? i : 0].re * inv_scale;
                const wf_real d = fabs(pv - pdy[pi]);
                dmax = (d > dmax) ? d : dmax;
                p[wf_q(c, i, c.Ny - 1, k)] = pv;
            }
        }
    }
}

template <int NX>
__device__ __forceinline__ void wf_inv_fx_body(const WfConst &c, const WfSpectral &sp, wf_real *p,
                                               const wf_real2 *__restrict__ twx) {
    if (wf_pass_returns(sp.ctl->done)) return;
    extern __shared__ wfc smem[];
    __shared__ int rad[WF_MAX_RADICES];
    if (blockIdx.x == gridDim.x - 1) {
        double dtop = 0.0;
        wf_top_duplicates(c, p, dtop);
        wf_block_max_store(dtop, &sp.pmax[blockIdx.x]);
        if constexpr (WF_MIXED) {
            __syncthreads();
            wf_block_max_store(0.0, &sp.pmax[sp.npmax + blockIdx.x]);
        }
        return;
    }
    wf_real dmax = WR(0.0), pabs = WR(0.0);
    /* the tiles are blocks 0 .. gridDim.x - 2 (the last block is the one above) */
    int g, k;
    wf_tile_decode_at((int)blockIdx.x, (int)gridDim.x - 1, sp.ngroups, sp.nz, &g, &k);
    if (NX <= 0 && threadIdx.x < WF_MAX_RADICES) rad[threadIdx.x] = sp.radx[threadIdx.x];
    wf_inv_fx_rows<NX>(c, sp, p, smem, rad, g, k, dmax, pabs, twx);
    wf_block_max_store((double)dmax, &sp.pmax[blockIdx.x]);
    if constexpr (WF_MIXED) {
        __syncthreads();
        wf_block_max_store((double)pabs, &sp.pmax[sp.npmax + blockIdx.x]);
    }
}
template <int NX>
__global__ __launch_bounds__(WF_NT) void k_inv_fx(WfConst c, WfSpectral sp, wf_real *p,
                                                  const wf_real2 *__restrict__ twx) {
    wf_inv_fx_body<NX>(c, sp, p, twx);
}

/* ------------------------------------------------- batched size classes ---- */

__global__ void k_density_batch(const WfPressItem *__restrict__ tab) {
    const WfPressItem it = wf_press_load(tab);
    wf_density_body(it.c, it.yn.T, it.rho);
}

__global__ void k_iter_reset_batch(const WfPressItem *__restrict__ tab) {
    const WfPressItem it = wf_press_load(tab);
    wf_iter_reset_body(it.sp.ctl);
}

template <int NX, int MODE>
__global__ __launch_bounds__(WF_NT) void k_rhs_fx_batch(const WfPressItem *__restrict__ tab, int check,
                                                        const wf_real2 *__restrict__ twx) {
    const WfPressItem it = wf_press_load(tab);
    const int b = wf_checked_block(it.sp, it.tol, it.rtol, check, it.max_iter);
    if (b >= 0) wf_rhs_fx_body<NX, MODE>(it.c, it.sp, it.ys, it.yn, it.p, b, (int)gridDim.x - (check >= 0), check, twx);
}

/* twy: the class's y twiddle table (it depends on ny alone, so every member's
 * table holds the same values), as an argument of its own for the reason
 * given at k_fy */
template <int NY>
__global__ __launch_bounds__(WF_NT) void k_fy_batch(const WfPressItem *__restrict__ tab, long slab_stride, int slab0,
                                                    int sign, int guarded, const wf_real2 *__restrict__ twy) {
    const WfPressItem it = wf_press_load(tab);
    wf_fy_body<NY, true>(it.sp, it.sp.F, slab_stride, slab0, sign, guarded, twy);
}

template <int LC>
__global__ __launch_bounds__(64 * WF_THOMAS_MAX_CHUNKS) WF_THOMAS_ATTR(LC) void k_thomas_batch(const WfPressItem *__restrict__ tab) {
    const WfPressItem it = wf_press_load(tab);
    wf_thomas_body<LC>(it.sp);
}

#if !WF_MIXED
template <int LC>
__global__ __launch_bounds__(64 * WF_THOMAS_MAX_CHUNKS) __attribute__((amdgpu_waves_per_eu(8))) void k_thomas_h_batch(
    const WfPressItem *__restrict__ tab) {
    const WfPressItem it = wf_press_load(tab);
    wf_thomas_h_body<LC>(it.sp);
}
#endif

template <int NX>
__global__ __launch_bounds__(WF_NT) void k_inv_fx_batch(const WfPressItem *__restrict__ tab,
                                                        const wf_real2 *__restrict__ twx) {
    const WfPressItem it = wf_press_load(tab);
    wf_inv_fx_body<NX>(it.c, it.sp, it.p, twx);
}

__global__ __launch_bounds__(WF_NT) void k_iter_check_batch(const WfPressItem *__restrict__ tab, int m) {
    const WfPressItem it = wf_press_load(tab);
    wf_iter_check_body(it.sp, it.tol, it.rtol, m, it.max_iter);
}

/* ------------------------------------------------------------- launchers ---- */

/* dynamic LDS of an x-transform kernel: twiddles + one buffer (compile-time
 * plan, in place) or two buffers (run-time radices) */
static size_t wf_fx_lds(int n, int nseq) {
    if (wf_rx_a(n)) return sizeof(wfc) * (size_t)(n + 9) * 2 * (size_t)nseq;
    return sizeof(wfc) * (size_t)n * (1 + (wf_planned(n) ? 1 : 2) * (size_t)nseq);
}

/* dynamic LDS of the y-transform: the two-factor plans use one buffer of nseq
 * sequences; the other compile-time plans the twiddle table and one buffer;
 * run-time radices the twiddle table and two buffers */
static size_t wf_fy_lds(int n, int nseq) {
    if (wf_f2_n1(n)) return sizeof(wfc) * (size_t)n * (size_t)nseq;
    if (wf_planned(n)) return sizeof(wfc) * (size_t)n * (1 + (size_t)nseq);
    return sizeof(wfc) * (size_t)n * (1 + 2 * (size_t)nseq);
}

#define WF_DISPATCH_N(n, KERNEL, grd, blk, lds, s, ...)                                                  \
    do {                                                                                                \
        switch (n) {                                                                                    \
            case 63: hipLaunchKernelGGL(KERNEL<63>, grd, blk, lds, s, __VA_ARGS__); break;              \
            case 127: hipLaunchKernelGGL(KERNEL<127>, grd, blk, lds, s, __VA_ARGS__); break;            \
            case 255: hipLaunchKernelGGL(KERNEL<255>, grd, blk, lds, s, __VA_ARGS__); break;            \
            case 511: hipLaunchKernelGGL(KERNEL<511>, grd, blk, lds, s, __VA_ARGS__); break;            \
            default:                                                                                    \
                if (n <= WF_NX_SHORT)                                                                   \
                    hipLaunchKernelGGL(KERNEL<0>, grd, blk, lds, s, __VA_ARGS__);                       \
                else                                                                                    \
                    hipLaunchKernelGGL(KERNEL<-1>, grd, blk, lds, s, __VA_ARGS__);                      \
                break;                                                                                  \
        }                                                                                               \
    } while (0)

#define WF_DISPATCH_F2(n, KERNEL, grd, blk, lds, s, ...)                                                 \
    do {                                                                                                \
        switch (n) {                                                                                    \
            case 63: hipLaunchKernelGGL(KERNEL<63>, grd, blk, lds, s, __VA_ARGS__); break;              \
            case 127: hipLaunchKernelGGL(KERNEL<127>, grd, blk, lds, s, __VA_ARGS__); break;            \
            case 255: hipLaunchKernelGGL(KERNEL<255>, grd, blk, lds, s, __VA_ARGS__); break;            \
            case 511: hipLaunchKernelGGL(KERNEL<511>, grd, blk, lds, s, __VA_ARGS__); break;            \
            default: hipLaunchKernelGGL(KERNEL<0>, grd, blk, lds, s, __VA_ARGS__); break;               \
        }                                                                                               \
    } while (0)

#define WF_DISPATCH_NM(KERNEL, n, MODE, grd, blk, lds, s, ...)                                           \
    do {                                                                                                \
        switch (n) {                                                                                    \
            case 63: hipLaunchKernelGGL((KERNEL<63, MODE>), grd, blk, lds, s, __VA_ARGS__); break;      \
            case 127: hipLaunchKernelGGL((KERNEL<127, MODE>), grd, blk, lds, s, __VA_ARGS__); break;    \
            case 255: hipLaunchKernelGGL((KERNEL<255, MODE>), grd, blk, lds, s, __VA_ARGS__); break;    \
            case 511: hipLaunchKernelGGL((KERNEL<511, MODE>), grd, blk, lds, s, __VA_ARGS__); break;    \
            default:                                                                                    \
                if (n <= WF_NX_SHORT)                                                                   \
                    hipLaunchKernelGGL((KERNEL<0, MODE>), grd, blk, lds, s, __VA_ARGS__);               \
                else                                                                                    \
                    hipLaunchKernelGGL((KERNEL<-1, MODE>), grd, blk, lds, s, __VA_ARGS__);              \
                break;                                                                                  \
        }                                                                                               \
    } while (0)

hipError_t wf_launch_density(const WfConst &c, const wf_real *T, wf_real *rho, hipStream_t s) {
    hipLaunchKernelGGL(k_density, dim3((unsigned)((c.N + 255) / 256)), dim3(256), 0, s, c, T, rho);
    return hipGetLastError();
}

hipError_t wf_launch_iter_reset(WfIterCtl *ctl, hipStream_t s) {
    hipLaunchKernelGGL(k_iter_reset, dim3(1), dim3(1), 0, s, ctl);
    return hipGetLastError();
}

hipError_t wf_launch_pressure_rhs_fx(const WfConst &c, const WfSpectral &sp, const WfState &Ys, const WfState &Yn,
                                     const wf_real *p, int mode, double tol, double rtol, int check, int max_iter,
                                     hipStream_t s) {
    const int nslabs = (mode == WF_F_TOP) ? 1 : sp.nz - 1;
    dim3 grd((unsigned)(sp.ngroups * nslabs + (check >= 0)));
    size_t lds = wf_fx_lds(sp.nx, sp.fx_pairs);
    switch (mode) {
        case WF_F_ITER: WF_DISPATCH_NM(k_rhs_fx, sp.nx, WF_F_ITER, grd, dim3(WF_NT), lds, s, c, sp, Ys, Yn, p, tol, rtol,
                                        check, max_iter, (const wf_real2 *)sp.twx);
            break;
        case WF_F_FIRST: WF_DISPATCH_NM(k_rhs_fx, sp.nx, WF_F_FIRST, grd, dim3(WF_NT), lds, s, c, sp, Ys, Yn, p, tol, rtol,
                                        check, max_iter, (const wf_real2 *)sp.twx);
            break;
        case WF_F_CONST: WF_DISPATCH_NM(k_rhs_fx, sp.nx, WF_F_CONST, grd, dim3(WF_NT), lds, s, c, sp, Ys, Yn, p, tol, rtol,
                                        check, max_iter, (const wf_real2 *)sp.twx);
            break;
        default: WF_DISPATCH_NM(k_rhs_fx, sp.nx, WF_F_TOP, grd, dim3(WF_NT), lds, s, c, sp, Ys, Yn, p, tol, rtol,
                                        check, max_iter, (const wf_real2 *)sp.twx);
            break;
    }
    return hipGetLastError();
}

hipError_t wf_launch_fy(const WfSpectral &sp, wf_real2 *buf, long slab_stride, int slab0, int nslabs, int sign,
                        int guarded, hipStream_t s) {
    if (nslabs <= 0) return hipSuccess;
    dim3 grd((sp.hx + sp.fy_cols - 1) / sp.fy_cols, nslabs, 1);
    size_t lds = wf_fy_lds(sp.ny, sp.fy_cols);
    const int nt = wf_f2_n1(sp.ny) ? wf_f2_threads(sp.ny) : WF_NT;
    WF_DISPATCH_F2(sp.ny, k_fy, grd, dim3(nt), lds, s, sp, buf, slab_stride, slab0, sign, guarded,
                   (const wf_real2 *)sp.twy);
    return hipGetLastError();
}

hipError_t wf_launch_pivots(const WfSpectral &sp, double *UB, hipStream_t s) {
    dim3 grd((sp.ny + 63) / 64, sp.hx, 1);
    hipLaunchKernelGGL(k_pivots, grd, dim3(64), 0, s, sp, UB);
    return hipGetLastError();
}

/* workgroups per kx column: 64 systems each, 32 with a component to a lane (see wf_thomas_body) */
static int wf_thomas_tiles(const WfSpectral &sp) {
    const int per = (!WF_MIXED && sp.thomas_lc > 8) ? 32 : 64;
    return (sp.ny + per - 1) / per;
}

hipError_t wf_launch_thomas(const WfSpectral &sp, hipStream_t s) {
    const int chunks = (sp.nz + sp.thomas_lc - 1) / sp.thomas_lc;
    dim3 grd(wf_thomas_tiles(sp), sp.hx + sp.low_kx, 1);
    if (sp.thomas_lc == 4) {
#if WF_MIXED
        return hipErrorInvalidValue;
#else
        if (chunks > 2 * WF_THOMAS_MAX_CHUNKS) return hipErrorInvalidValue;
        hipLaunchKernelGGL(k_thomas_h<4>, dim3((sp.ny + 31) / 32, sp.hx, 1), dim3(64 * ((chunks + 1) / 2)), 0, s, sp);
        return hipGetLastError();
#endif
    }
    if (chunks > WF_THOMAS_MAX_CHUNKS) return hipErrorInvalidValue;
    if (sp.thomas_lc == 8)
        hipLaunchKernelGGL(k_thomas<8>, grd, dim3(64 * chunks), 0, s, sp);
    else if (sp.thomas_lc == 16)
        hipLaunchKernelGGL(k_thomas<16>, grd, dim3(64 * chunks), 0, s, sp);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t wf_launch_iter_check(const WfSpectral &sp, double tol, double rtol, int m, int max_iter, hipStream_t s) {
    hipLaunchKernelGGL(k_iter_check, dim3(1), dim3(WF_NT), 0, s, sp, tol, rtol, m, max_iter);
    return hipGetLastError();
}

hipError_t wf_launch_inverse_fx(const WfConst &c, const WfSpectral &sp, wf_real *p, hipStream_t s) {
    dim3 grd((unsigned)sp.npmax);
    size_t lds = wf_fx_lds(sp.nx, sp.fx_pairs);
    WF_DISPATCH_N(sp.nx, k_inv_fx, grd, dim3(WF_NT), lds, s, c, sp, p, (const wf_real2 *)sp.twx);
    return hipGetLastError();
}

/* Batched launchers: tab holds the nm members of one size class; sp and c are
 * any member's (the grids depend only on the class).  Each launch is the solo
 * launch's grid with z = nm. */
hipError_t wf_launch_density_batch(const WfConst &c, const WfPressItem *tab, int nm, hipStream_t s) {
    hipLaunchKernelGGL(k_density_batch, dim3((unsigned)((c.N + 255) / 256), 1, nm), dim3(256), 0, s, tab);
    return hipGetLastError();
}

hipError_t wf_launch_iter_reset_batch(const WfPressItem *tab, int nm, hipStream_t s) {
    hipLaunchKernelGGL(k_iter_reset_batch, dim3(1, 1, nm), dim3(1), 0, s, tab);
    return hipGetLastError();
}

hipError_t wf_launch_pressure_rhs_fx_batch(const WfSpectral &sp, const WfPressItem *tab, int nm, int mode, int check,
                                           hipStream_t s) {
    const int nslabs = (mode == WF_F_TOP) ? 1 : sp.nz - 1;
    dim3 grd((unsigned)(sp.ngroups * nslabs + (check >= 0)), 1, nm);
    size_t lds = wf_fx_lds(sp.nx, sp.fx_pairs);
    switch (mode) {
        case WF_F_ITER: WF_DISPATCH_NM(k_rhs_fx_batch, sp.nx, WF_F_ITER, grd, dim3(WF_NT), lds, s, tab, check,
                                        (const wf_real2 *)sp.twx);
            break;
        case WF_F_FIRST: WF_DISPATCH_NM(k_rhs_fx_batch, sp.nx, WF_F_FIRST, grd, dim3(WF_NT), lds, s, tab, check,
                                        (const wf_real2 *)sp.twx);
            break;
        case WF_F_CONST: WF_DISPATCH_NM(k_rhs_fx_batch, sp.nx, WF_F_CONST, grd, dim3(WF_NT), lds, s, tab, check,
                                        (const wf_real2 *)sp.twx);
            break;
        default: return hipErrorInvalidValue; /* the top plane is solo only */
    }
    return hipGetLastError();
}

hipError_t wf_launch_fy_batch(const WfSpectral &sp, const WfPressItem *tab, int nm, long slab_stride, int slab0,
                              int nslabs, int sign, int guarded, hipStream_t s) {
    if (nslabs <= 0) return hipSuccess;
    const int cols = (!wf_f2_n1(sp.ny) && wf_planned(sp.ny)) ? wf_fy_ip_cols(sp.ny, true) : sp.fy_cols;
    dim3 grd((sp.hx + cols - 1) / cols, nslabs, nm);
    size_t lds = wf_fy_lds(sp.ny, cols);
    const int nt = wf_f2_n1(sp.ny) ? wf_f2_threads(sp.ny) : WF_NT;
    WF_DISPATCH_F2(sp.ny, k_fy_batch, grd, dim3(nt), lds, s, tab, slab_stride, slab0, sign, guarded,
                   (const wf_real2 *)sp.twy);
    return hipGetLastError();
}

hipError_t wf_launch_thomas_batch(const WfSpectral &sp, const WfPressItem *tab, int nm, hipStream_t s) {
    const int chunks = (sp.nz + sp.thomas_lc - 1) / sp.thomas_lc;
    dim3 grd(wf_thomas_tiles(sp), sp.hx + sp.low_kx, nm);
    if (sp.thomas_lc == 4) {
#if WF_MIXED
        return hipErrorInvalidValue;
#else
        if (chunks > 2 * WF_THOMAS_MAX_CHUNKS) return hipErrorInvalidValue;
        hipLaunchKernelGGL(k_thomas_h_batch<4>, dim3((sp.ny + 31) / 32, sp.hx, nm), dim3(64 * ((chunks + 1) / 2)), 0,
                           s, tab);
        return hipGetLastError();
#endif
    }
    if (chunks > WF_THOMAS_MAX_CHUNKS) return hipErrorInvalidValue;
    if (sp.thomas_lc == 8)
        hipLaunchKernelGGL(k_thomas_batch<8>, grd, dim3(64 * chunks), 0, s, tab);
    else if (sp.thomas_lc == 16)
        hipLaunchKernelGGL(k_thomas_batch<16>, grd, dim3(64 * chunks), 0, s, tab);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t wf_launch_inverse_fx_batch(const WfSpectral &sp, const WfPressItem *tab, int nm, hipStream_t s) {
    dim3 grd((unsigned)sp.npmax, 1, nm);
    size_t lds = wf_fx_lds(sp.nx, sp.fx_pairs);
    WF_DISPATCH_N(sp.nx, k_inv_fx_batch, grd, dim3(WF_NT), lds, s, tab, (const wf_real2 *)sp.twx);
    return hipGetLastError();
}

hipError_t wf_launch_iter_check_batch(const WfPressItem *tab, int nm, int m, hipStream_t s) {
    hipLaunchKernelGGL(k_iter_check_batch, dim3(1, 1, nm), dim3(WF_NT), 0, s, tab, m);
    return hipGetLastError();
}

}  // namespace WF_NS
