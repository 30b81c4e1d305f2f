/*
 * wf_fft.h -- FFT building blocks of the pressure solve.
 *
 * Lengths 63, 127, 255 and 511 (64 to 512 nodes) have compile-time plans (below):
 * two factors in registers (y-transforms of 63 and 255), three odd radices with
 * two of them in registers (FP32 x-transforms of 255), or in place in LDS.  Any
 * other length runs a mixed-radix Stockham transform in LDS with run-time
 * radices (wf_lds_fft): stage with radix R after radices of product
 * Ns (natural order, decimation in time): butterfly j in [0, n/R) reads
 * in[j + r n/R], r < R, and writes out[(j/Ns) Ns R + j%Ns + q Ns], q < R, with
 *   out = sum_r W_{Ns R}^{r (j%Ns + q Ns)} in[j + r n/R],  W_m = exp(sign 2 pi i / m).
 * wf_stockham_output states one output element of a stage, for the CPU checks
 * alone; the kernels run wf_rt_stage, which is host/device-neutral, and a CPU
 * check compares the two at every length.
 */
#ifndef WF_FFT_H
#define WF_FFT_H

#if defined(__HIPCC__)
#define WF_HD __host__ __device__ __forceinline__
#define WF_HDM WF_HD
#else
#define WF_HD static inline
#define WF_HDM inline
#endif

#define WF_MAX_RADICES 16

/* wfc: a complex value in the precision of the compilation (wf_prec.h); the
 * C check of the plan (no HIP) uses FP64 */
#if defined(__HIPCC__)
#include "wf_prec.h"
namespace WF_NS {
typedef struct {
    wf_real re, im;
} wfc;
#else
typedef double wf_real;
#define WR(x) (x)
typedef struct {
    double re, im;
} wfc;
#endif

/* Output element o of one Stockham stage over a sequence of length n stored at
 * `in`; tw[e] = exp(sign 2 pi i e / n). */
WF_HD wfc wf_stockham_output(const wfc *in, int n, int R, int Ns, const wfc *tw, int o) {
    int kq = o % Ns;
    int rest = o / Ns;
    int q = rest % R;
    int jb = (rest / R) * Ns + kq;
    int m = n / R;
    int scale = n / (Ns * R);
    int step = ((kq + q * Ns) * scale) % n;
    wf_real ar = WR(0.0), ai = WR(0.0);
    int e = 0;
    for (int r = 0; r < R; r++) {
        wfc x = in[jb + r * m];
        wfc w = tw[e];
        ar += w.re * x.re - w.im * x.im;
        ai += w.re * x.im + w.im * x.re;
        e += step;
        if (e >= n) e -= n;
    }
    wfc y;
    y.re = ar;
    y.im = ai;
    return y;
}

/* Spectra of two real sequences a, b packed as z = a + i b, at bin r:
 * A[r] = (Z[r] + conj Z[n-r]) / 2, B[r] = (Z[r] - conj Z[n-r]) / (2i). */
WF_HD void wf_unpack_pair(wfc zr, wfc zm, wfc *A, wfc *B) {
    A->re = WR(0.5) * (zr.re + zm.re);
    A->im = WR(0.5) * (zr.im - zm.im);
    B->re = WR(0.5) * (zr.im + zm.im);
    B->im = WR(0.5) * (zm.re - zr.re);
}

/* Bin r of Z = A + i B for the inverse of two half spectra (r < n/2+1 read
 * directly, r above it from the conjugate-symmetric partner). */
WF_HD wfc wf_pack_pair(wfc A, wfc B, int conj) {
    wfc z;
    if (!conj) {
        z.re = A.re - B.im;
        z.im = A.im + B.re;
    } else {
        z.re = A.re + B.im;
        z.im = B.re - A.im;
    }
    return z;
}

#if defined(__cplusplus)
/* Quotients by a run-time divisor d through its reciprocal rounded up (exact
 * for t < 2^16, d <= 2^10: t (2^32/d + 1) < 2^32 (t/d + 1/d)). */
struct WfDiv {
    unsigned m;
    int d;
    WF_HDM explicit WfDiv(int div) : m(0xffffffffu / (unsigned)div + 1u), d(div) {}
    WF_HDM int operator()(int t) const {
        return (d == 1) ? t : (int)(((unsigned long long)(unsigned)t * m) >> 32);
    }
};

/* Run-time Stockham stages, wf_stockham_output's terms in its order.  What
 * bounds them is instructions: the index arithmetic of an output (five
 * run-time divisions), and for every term two LDS reads and 8 separate
 * roundings.  So a small radix takes a whole butterfly per thread (its R inputs
 * read once, one set of indices for R outputs), and the others WF_RT_SEQ
 * sequences per thread, which share indices and twiddles (two measured best:
 * four leave too few threads, 32 us against 24 for the x pass of length 200).
 * The term r = 0 has the factor (1, 0) and starts the sum.  FP32, us per pass,
 * one output per thread before: y of length 150 at 201x151x81 30 -> 20, x of
 * length 200 35 -> 24 and 32 -> 21; length 199 (prime) at 200x200x90 y 206 ->
 * 132, x 166 -> 136. */
template <int R>
WF_HD void wf_rt_butterfly(const wfc *a, wfc *b, int n, int nseq, int Ns, const wfc *tw, int tid, int nt) {
    const int m = n / R, scale = m / Ns;
    const WfDiv by_m(m), by_ns(Ns);
    for (int t = tid; t < m * nseq; t += nt) {
        const int s = by_m(t), j = t - s * m, jq = by_ns(j), kq = j - jq * Ns;
        const wfc *in = a + s * n + j;
        wfc *out = b + s * n + jq * Ns * R + kq;
        wfc x[R];
#pragma unroll
        for (int r = 0; r < R; r++) x[r] = in[r * m];
#pragma unroll
        for (int q = 0; q < R; q++) {
            const int step = kq * scale + q * m;
            wfc acc = x[0];
            int e = 0;
#pragma unroll
            for (int r = 1; r < R; r++) {
                e += step;
                e = (e >= n) ? e - n : e;
                const wfc w = tw[e];
                acc.re += w.re * x[r].re - w.im * x[r].im;
                acc.im += w.re * x[r].im + w.im * x[r].re;
            }
            out[q * Ns] = acc;
        }
    }
}
#define WF_RT_SEQ 2
WF_HD void wf_rt_outputs(const wfc *a, wfc *b, int n, int nseq, int R, int Ns, const wfc *tw, int tid, int nt) {
    constexpr int S = WF_RT_SEQ;
    const int m = n / R, scale = m / Ns;
    const WfDiv by_n(n), by_ns(Ns), by_r(R);
    for (int t = tid; t < n * (nseq / S); t += nt) {
        const int sg = by_n(t), o = t - sg * n;
        const int rest = by_ns(o), kq = o - rest * Ns, jq = by_r(rest), q = rest - jq * R;
        const wfc *in = a + sg * S * n + jq * Ns + kq;
        const int step = kq * scale + q * m;
        wfc acc[S];
#pragma unroll
        for (int s = 0; s < S; s++) acc[s] = in[s * n];
        int e = 0;
#pragma unroll 4
        for (int r = 1; r < R; r++) {
            e += step;
            e = (e >= n) ? e - n : e;
            in += m;
            const wfc w = tw[e];
#pragma unroll
            for (int s = 0; s < S; s++) {
                const wfc x = in[s * n];
                acc[s].re += w.re * x.re - w.im * x.im;
                acc[s].im += w.re * x.im + w.im * x.re;
            }
        }
#pragma unroll
        for (int s = 0; s < S; s++) b[(sg * S + s) * n + o] = acc[s];
    }
}
/* Thread tid's part (of nt) of a stage of radix R after radices of product Ns,
 * over nseq sequences (a multiple of WF_RT_SEQ) of length n, a -> b. */
WF_HD void wf_rt_stage(const wfc *a, wfc *b, int n, int nseq, int R, int Ns, const wfc *tw, int tid, int nt) {
    switch (R) {
        case 2: wf_rt_butterfly<2>(a, b, n, nseq, Ns, tw, tid, nt); break;
        case 3: wf_rt_butterfly<3>(a, b, n, nseq, Ns, tw, tid, nt); break;
        case 4: wf_rt_butterfly<4>(a, b, n, nseq, Ns, tw, tid, nt); break;
        case 5: wf_rt_butterfly<5>(a, b, n, nseq, Ns, tw, tid, nt); break;
        case 7: wf_rt_butterfly<7>(a, b, n, nseq, Ns, tw, tid, nt); break;
        default: wf_rt_outputs(a, b, n, nseq, R, Ns, tw, tid, nt); break;
    }
}
#endif

#if defined(__HIPCC__)
/* One full FFT of `nseq` sequences (a multiple of WF_RT_SEQ) of run-time
 * length n held in LDS (a -> b -> a ...), for lengths without a compile-time
 * plan.  Returns the buffer that holds the result. */
__device__ __forceinline__ wfc *wf_lds_fft(wfc *a, wfc *b, int n, int nseq, const int *rad, const wfc *tw) {
    int Ns = 1;
    for (int p = 0; p < WF_MAX_RADICES; p++) {
        const int R = rad[p];
        if (R == 0) break;
        wf_rt_stage(a, b, n, nseq, R, Ns, tw, (int)threadIdx.x, (int)blockDim.x);
        __syncthreads();
        wfc *tmp = a;
        a = b;
        b = tmp;
        Ns *= R;
    }
    return a;
}

__device__ __forceinline__ wfc wf_cmul(wfc a, wfc b) {
#pragma clang fp contract(fast)
    wfc r;
    r.re = a.re * b.re - a.im * b.im;
    r.im = a.re * b.im + a.im * b.re;
    return r;
}

/* ------------------------------------------------------------------------
 * Compile-time plans for the transform lengths of the supported grids.
 * The radix sequence of N is the one the host factoriser produces (4s, then
 * 2, then odd primes ascending), so every stage's sizes are constants and the
 * index arithmetic folds into multiplications and shifts.
 * ---------------------------------------------------------------------- */

constexpr int wf_radix_of(int n, int idx) {
    int cnt = 0;
    while (n % 4 == 0) {
        if (cnt == idx) return 4;
        cnt++;
        n /= 4;
    }
    while (n % 2 == 0) {
        if (cnt == idx) return 2;
        cnt++;
        n /= 2;
    }
    for (int p = 3; n > 1; p += 2) {
        while (n % p == 0) {
            if (cnt == idx) return p;
            cnt++;
            n /= p;
        }
    }
    return 0;
}


/* One Stockham stage of radix R after radices of product NS over `nseq`
 * sequences of length N (same mathematics as wf_stockham_output).  Radices up
 * to 8 run one butterfly per thread with its R values in registers; larger
 * prime radices run one output per thread to keep the workgroup busy. */
/* R-point DFT of x (twiddled inputs) into y, W_R^m = tw[m * WR]. */
template <int R, int WR>
__device__ __forceinline__ void wf_dft_generic(const wfc *x, wfc *y, const wfc *tw) {
#pragma clang fp contract(fast)
#pragma unroll
    for (int q = 0; q < R; q++) {
        wfc acc = x[0];
#pragma unroll
        for (int r = 1; r < R; r++) {
            wfc p = wf_cmul(x[r], tw[((r * q) % R) * WR]);
            acc.re += p.re;
            acc.im += p.im;
        }
        y[q] = acc;
    }
}

constexpr int wf_cmin(int a, int b) { return a < b ? a : b; }
constexpr int wf_cmax(int a, int b) { return a > b ? a : b; }

/* One in-place Stockham stage of radix R after radices of product NS over
 * NSEQ sequences of length N in LDS, NT threads (same mathematics as
 * wf_stockham_output).  Every thread first computes its outputs into
 * registers, then the workgroup synchronises and writes them back, so one
 * buffer suffices.  Ends with a barrier.
 *
 * Odd R: with a_r = x_r + x_{R-r}, b_r = x_r - x_{R-r} (twiddled inputs),
 *   X_q     = x_0 + sum_{r<=H} a_r Re W^{rq} + i sum_{r<=H} b_r Im W^{rq},
 *   X_{R-q} = x_0 + sum_{r<=H} a_r Re W^{rq} - i sum_{r<=H} b_r Im W^{rq},
 * H = (R-1)/2, W = exp(sign 2 pi i / R) (uses W^{R-m} = conj W^m): a quarter of
 * the multiplications of the direct sum.  QS threads share one butterfly, each
 * streaming over the inputs and accumulating only its own pairs (q, R-q), so
 * few registers are live and large radices still fill the workgroup.
 * Even R (2, 4): one butterfly per thread, direct sum. */
template <int N, int R, int NS, int NSEQ, int NT>
__device__ __forceinline__ void wf_stage_ip(wfc *buf, const wfc *tw) {
#pragma clang fp contract(fast)
    constexpr int M = N / R;
    constexpr int SC = N / (NS * R);
    constexpr int WR = N / R;
    constexpr int NB = NSEQ * M; /* butterflies */
    if constexpr (R % 2 == 1) {
        constexpr int H = (R - 1) / 2;
        /* threads per butterfly: as many as the workgroup has for it, up to
         * H; for a radix above 17, at most (H+3)/4, so that each thread
         * accumulates at least 4 output pairs from every input pair it reads
         * from LDS, even where that leaves threads idle in this stage (the
         * workgroups beside it on the CU take their issue slots) */
        constexpr int QS0 = wf_cmax(1, wf_cmin(H, NT / NB));
        constexpr int QS = (R > 17) ? wf_cmin(QS0, (H + 3) / 4) : QS0;
        constexpr int QN = (H + QS - 1) / QS;               /* output pairs per thread */
        constexpr int NW = NB * QS;
        constexpr int PER = (NW + NT - 1) / NT;
        wfc y0[PER], yp[PER][QN], ym[PER][QN];
#pragma unroll
        for (int pi = 0; pi < PER; pi++) {
            const int t = threadIdx.x + pi * NT;
            if (t < NW) {
                const int bf = t / QS, u = t - bf * QS;
                const int s = bf / M, j = bf - s * M;
                const int kq = j % NS;
                const wfc *src = buf + s * N + j;
                const wfc x0 = src[0];
                wf_real c0r = x0.re, c0i = x0.im;
                wf_real cr[QN], ci[QN], sr[QN], si[QN];
                int m[QN]; /* (r q) mod R for this thread's q = 1 + u + qi QS */
#pragma unroll
                for (int qi = 0; qi < QN; qi++) {
                    cr[qi] = x0.re;
                    ci[qi] = x0.im;
                    sr[qi] = WR(0.0);
                    si[qi] = WR(0.0);
                    m[qi] = 0;
                }
                constexpr int UNR = (H <= 8) ? H : 4;
#pragma unroll UNR
                for (int r = 1; r <= H; r++) {
                    wfc xa = src[r * M], xb = src[(R - r) * M];
                    if constexpr (NS > 1) {
                        xa = wf_cmul(xa, tw[kq * r * SC]);
                        xb = wf_cmul(xb, tw[kq * (R - r) * SC]);
                    }
                    const wf_real ar = xa.re + xb.re, ai = xa.im + xb.im;
                    const wf_real br = xa.re - xb.re, bi = xa.im - xb.im;
                    c0r += ar;
                    c0i += ai;
#pragma unroll
                    for (int qi = 0; qi < QN; qi++) {
                        const int q = 1 + u + qi * QS;
                        int mm = m[qi] + q;
                        mm = (mm >= R) ? mm - R : mm;
                        m[qi] = mm;
                        /* tw[m N/R] = W^m (its imaginary part carries the sign
                         * of W^{R-m} = conj W^m) */
                        const wfc W = tw[mm * WR];
                        cr[qi] += ar * W.re;
                        ci[qi] += ai * W.re;
                        sr[qi] += bi * W.im;
                        si[qi] += br * W.im;
                    }
                }
                y0[pi].re = c0r;
                y0[pi].im = c0i;
#pragma unroll
                for (int qi = 0; qi < QN; qi++) {
                    yp[pi][qi].re = cr[qi] - sr[qi];
                    yp[pi][qi].im = ci[qi] + si[qi];
                    ym[pi][qi].re = cr[qi] + sr[qi];
                    ym[pi][qi].im = ci[qi] - si[qi];
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int pi = 0; pi < PER; pi++) {
            const int t = threadIdx.x + pi * NT;
            if (t < NW) {
                const int bf = t / QS, u = t - bf * QS;
                const int s = bf / M, j = bf - s * M;
                const int kq = j % NS;
                wfc *dst = buf + s * N + (j / NS) * NS * R + kq;
                if (u == 0) dst[0] = y0[pi];
#pragma unroll
                for (int qi = 0; qi < QN; qi++) {
                    const int q = 1 + u + qi * QS;
                    if (q <= H) {
                        dst[q * NS] = yp[pi][qi];
                        dst[(R - q) * NS] = ym[pi][qi];
                    }
                }
            }
        }
        __syncthreads();
    } else {
        constexpr int PER = (NB + NT - 1) / NT;
        wfc v[PER][R];
#pragma unroll
        for (int pi = 0; pi < PER; pi++) {
            const int t = threadIdx.x + pi * NT;
            if (t < NB) {
                const int s = t / M, j = t - s * M;
                const int kq = j % NS;
                const wfc *src = buf + s * N + j;
                wfc x[R];
#pragma unroll
                for (int r = 0; r < R; r++) x[r] = src[r * M];
                if constexpr (NS > 1) {
#pragma unroll
                    for (int r = 1; r < R; r++) x[r] = wf_cmul(x[r], tw[kq * r * SC]);
                }
                wf_dft_generic<R, WR>(x, v[pi], tw);
            }
        }
        __syncthreads();
#pragma unroll
        for (int pi = 0; pi < PER; pi++) {
            const int t = threadIdx.x + pi * NT;
            if (t < NB) {
                const int s = t / M, j = t - s * M;
                const int kq = j % NS;
                wfc *dst = buf + s * N + (j / NS) * NS * R + kq;
#pragma unroll
                for (int q = 0; q < R; q++) dst[q * NS] = v[pi][q];
            }
        }
        __syncthreads();
    }
}

template <int N, int IDX, int NS, int NSEQ, int NT>
struct WfStagesIP {
    static __device__ __forceinline__ void run(wfc *buf, const wfc *tw) {
        constexpr int R = wf_radix_of(N, IDX);
        if constexpr (R != 0) {
            wf_stage_ip<N, R, NS, NSEQ, NT>(buf, tw);
            WfStagesIP<N, IDX + 1, NS * R, NSEQ, NT>::run(buf, tw);
        }
    }
};

/* In-place transform of NSEQ sequences of compile-time length N held in LDS
 * (natural order in and out), NT threads.  The caller synchronises after
 * filling buf; the transform ends with a barrier. */
template <int N, int NSEQ, int NT>
__device__ __forceinline__ void wf_fft_ip(wfc *buf, const wfc *tw) {
    WfStagesIP<N, 0, 1, NSEQ, NT>::run(buf, tw);
}
/* ------------------------------------------------------------------------
 * Two-factor register FFT for N = N1 N2 (N1, N2 odd, <= 17): the transform
 * lengths of the 64- and 256-node grids (63 = 7 x 9, 255 = 15 x 17).
 *   n = n1 + N1 n2, k = k2 + N2 k1:
 *   Y[n1][k2] = sum_{n2} x[n1 + N1 n2] W_{N2}^{n2 k2}          (phase A)
 *   X[k2 + N2 k1] = sum_{n1} W_N^{n1 k2} Y[n1][k2] W_{N1}^{n1 k1} (phase B)
 * Phase A: one thread per (sequence, n1) loads its N2 inputs, transforms them
 * in registers, twiddles and writes Y to LDS at n1 + N1 k2 (the positions it
 * read, when the input is that LDS buffer).  Phase B: one thread per
 * (sequence, k2) reads its N1 contiguous values of Y, transforms them and
 * hands X[k2 + N2 k1] to the caller.  The DFT constants W_R^m = tw[m N/R]
 * have compile-time offsets into the N-point table (scalar loads).
 * ---------------------------------------------------------------------- */

/* Factor pair of the lengths with a two-factor plan (0 if none). */
__host__ __device__ constexpr int wf_f2_n1(int n) { return n == 255 ? 15 : n == 63 ? 7 : 0; }
__host__ __device__ constexpr int wf_f2_n2(int n) { return n == 255 ? 17 : n == 63 ? 9 : 0; }
/* sequences per workgroup: the most that max(N1, N2) threads each fit in
 * 256 threads, or WF_FY_NSEQ255 for length 255 (fewer sequences, less LDS
 * and a smaller workgroup, so more workgroups per CU) */
#ifndef WF_FY_NSEQ255
#define WF_FY_NSEQ255 12
#endif
__host__ __device__ constexpr int wf_f2_nmax(int n) { return wf_f2_n1(n) > wf_f2_n2(n) ? wf_f2_n1(n) : wf_f2_n2(n); }
__host__ __device__ constexpr int wf_f2_nseq(int n) {
    return !wf_f2_n1(n) ? 0 : (n == 255 && WF_FY_NSEQ255 > 0) ? WF_FY_NSEQ255 : 256 / wf_f2_nmax(n);
}
/* threads of a two-factor workgroup: whole waves covering both phases */
__host__ __device__ constexpr int wf_f2_threads(int n) { return (wf_f2_nmax(n) * wf_f2_nseq(n) + 63) / 64 * 64; }
static_assert(wf_f2_threads(255) <= 256 && wf_f2_threads(63) <= 256, "two-factor workgroup above 256 threads");

/* Odd R-point DFT of x (registers) with W = exp(SIGN 2 pi i / R) taken from
 * the forward N-point table tw (W_R^m = tw[m TS] or its conjugate), outputs
 * handed to out(k, X_k) in the order 0, 1, R-1, 2, R-2, ... (pairs q, R-q
 * share their sums: X_q, X_{R-q} = x_0 + sum a_r Re W^{rq} +- i sum b_r Im W^{rq}). */
template <int R, int TS, int SIGN, class Out>
__device__ __forceinline__ void wf_dft_reg(const wfc *x, const wf_real2 *tw, Out &&out) {
#pragma clang fp contract(fast)
    constexpr int H = (R - 1) / 2;
    wfc a[H + 1], b[H + 1];
    wfc y0 = x[0];
#pragma unroll
    for (int r = 1; r <= H; r++) {
        a[r].re = x[r].re + x[R - r].re;
        a[r].im = x[r].im + x[R - r].im;
        b[r].re = x[r].re - x[R - r].re;
        b[r].im = x[r].im - x[R - r].im;
        y0.re += a[r].re;
        y0.im += a[r].im;
    }
    out(0, y0);
#pragma unroll
    for (int q = 1; q <= H; q++) {
        wf_real cr = x[0].re, ci = x[0].im, sr = WR(0.0), si = WR(0.0);
#pragma unroll
        for (int r = 1; r <= H; r++) {
            const wf_real2 W = tw[((r * q) % R) * TS];
            const wf_real c = W.x, sn = (SIGN < 0) ? W.y : -W.y;
            cr += a[r].re * c;
            ci += a[r].im * c;
            sr += b[r].im * sn;
            si += b[r].re * sn;
        }
        wfc yp, ym;
        yp.re = cr - sr;
        yp.im = ci + si;
        ym.re = cr + sr;
        ym.im = ci - si;
        out(q, yp);
        out(R - q, ym);
    }
}

/* Phase A for sequence s, n1 = this thread's row: load(s, n) gives input n;
 * Y is written to buf[s N + n1 + N1 k2]. */
template <int N1, int N2, int SIGN, class Load>
__device__ __forceinline__ void wf_f2_phase_a(wfc *buf, const wf_real2 *tw, int s, int n1, Load &&load) {
#pragma clang fp contract(fast)
    constexpr int N = N1 * N2;
    /* this row's twiddles W_N^{n1 k2} (n1 k2 < N) are loaded together with
     * its inputs, not one by one where they are used */
    wf_real2 wt[N2];
#pragma unroll
    for (int k2 = 1; k2 < N2; k2++) wt[k2] = tw[n1 * k2];
    wfc x[N2];
#pragma unroll
    for (int n2 = 0; n2 < N2; n2++) x[n2] = load(s, n1 + N1 * n2);
    wfc *row = buf + s * N + n1;
    wf_dft_reg<N2, N1, SIGN>(x, tw, [&](int k2, wfc y) {
        if (k2 != 0) {
            const wf_real2 W = wt[k2];
            const wf_real wi = (SIGN < 0) ? W.y : -W.y;
            wfc t;
            t.re = y.re * W.x - y.im * wi;
            t.im = y.re * wi + y.im * W.x;
            y = t;
        }
        row[N1 * k2] = y;
    });
}

/* Phase B for sequence s, k2 = this thread's column: X[k2 + N2 k1] -> out(k1, X). */
template <int N1, int N2, int SIGN, class Out>
__device__ __forceinline__ void wf_f2_phase_b(const wfc *buf, const wf_real2 *tw, int s, int k2, Out &&out) {
    constexpr int N = N1 * N2;
    wfc y[N1];
    const wfc *col = buf + s * N + N1 * k2;
#pragma unroll
    for (int n1 = 0; n1 < N1; n1++) y[n1] = col[n1];
    wf_dft_reg<N1, N2, SIGN>(y, tw, out);
}

/* ------------------------------------------------------------------------
 * Register form of the compile-time Stockham plan with three odd radices
 * R1 R2 R3 (255 = 3 5 17), for the FP32 x-transforms.  The stages compute what
 * wf_stage_ip computes, term for term and bit for bit (a twiddle's products
 * are spelled out in the form its compiled contraction takes, the sums of a
 * DFT are the same chains), but the values between the first two stay in
 * registers, each value crosses LDS once, not three times, with two barriers
 * instead of six, and the DFT constants come by scalar loads, not from LDS
 * one by one: 7.2 M vector instructions instead of 16 M in P5 at 256x256x128,
 * whose time, bound by them before and by its two phases' latency now, goes
 * from 30.4 to 25.5 us; P1 stays at 32.7 (its loads).  With 4 row pairs to a
 * workgroup instead of 8, 32.6 and 33.2.  In FP64 its registers (145-198)
 * leave too few waves: P5 47 us against 44 in place, P1 84 against 76.  The
 * form is for three odd radices of which the last is at most PAIRS threads'
 * share of a workgroup: 255 = 3 5 17 and, of the planned lengths, 63 = 3 3 7,
 * where it gains nothing (5.2 and 5.4 us in either form, the launch's latency,
 * at 64x64x32), so it is instantiated for 255 alone; 127 and 511 = 7 73 have
 * fewer radices.
 * Input of block g of the last radix: x[g + R3 m], m < R1 R2.
 * Phase A: one thread per (sequence, g) runs the radices R1 and R2 on its
 * R1 R2 inputs and twiddles the outputs for the last radix.
 * Phase B: one thread per (sequence, j), j < R1 R2, runs the radix R3.
 * ---------------------------------------------------------------------- */
__host__ __device__ constexpr int wf_rx_a(int n) { return (WF_MIXED && n == 255) ? 15 : 0; }
__host__ __device__ constexpr int wf_rx_b(int n) { return (WF_MIXED && n == 255) ? 17 : 0; }

/* a w, or a conj(w) for the inverse transform */
template <int SIGN>
__device__ __forceinline__ wfc wf_twiddle(wfc a, wf_real2 w) {
    const wf_real wi = (SIGN < 0) ? w.y : -w.y;
    wfc r;
    r.re = wf_fma(a.re, w.x, -(a.im * wi));
    r.im = wf_fma(a.im, w.x, a.re * wi);
    return r;
}

/* Phase A: x the inputs x[g + R3 m], outputs to row[g + R3 n], n < R1 R2. */
template <int N, int SIGN>
__device__ __forceinline__ void wf_rx_phase_a(const wfc *x, wfc *row, const wf_real2 *__restrict__ tw, int g) {
    constexpr int R1 = wf_radix_of(N, 0), R2 = wf_radix_of(N, 1), R3 = wf_rx_b(N), NA = R1 * R2;
    static_assert(NA == wf_rx_a(N) && R3 == wf_radix_of(N, 2) && NA * R3 == N, "three-radix plan");
    wf_real2 wt[NA]; /* the last radix's twiddles W_N^{g n} */
#pragma unroll
    for (int n = 1; n < NA; n++) wt[n] = tw[g * n];
    wfc v[R2][R1];
#pragma unroll
    for (int r = 0; r < R2; r++) {
        wfc in[R1];
#pragma unroll
        for (int s = 0; s < R1; s++) in[s] = x[r + R2 * s];
        wf_dft_reg<R1, N / R1, SIGN>(in, tw, [&](int q, wfc y) { v[r][q] = y; });
    }
#pragma unroll
    for (int kq = 0; kq < R1; kq++) {
        wfc in[R2];
#pragma unroll
        for (int r = 0; r < R2; r++) in[r] = (r && kq) ? wf_twiddle<SIGN>(v[r][kq], tw[kq * r * R3]) : v[r][kq];
        wf_dft_reg<R2, N / R2, SIGN>(in, tw, [&](int q, wfc y) {
            const int n = kq + R1 * q;
            row[g + R3 * n] = n ? wf_twiddle<SIGN>(y, wt[n]) : y;
        });
    }
}
/* Phase B: row[j R3 + r], r < R3 (phase A's outputs n = j) -> out(k, X_k), k = j + R1 R2 q. */
template <int N, int SIGN, class Out>
__device__ __forceinline__ void wf_rx_phase_b(const wfc *row, const wf_real2 *__restrict__ tw, int j, Out &&out) {
    constexpr int R3 = wf_rx_b(N), NA = wf_rx_a(N);
    wfc x[R3];
#pragma unroll
    for (int r = 0; r < R3; r++) x[r] = row[j * R3 + r];
    wf_dft_reg<R3, N / R3, SIGN>(x, tw, [&](int q, wfc y) { out(j + NA * q, y); });
}
#endif

#if defined(__HIPCC__)
}  // namespace WF_NS
#endif

#endif /* WF_FFT_H */
