/*
 * wf_planes_rule.h -- which solves the coefficient-plane form takes, and by
 * which instance of the plane solve (wf_planes.hip).  Host/device-neutral: the
 * CPU check runs the same rules over every size.
 */
#ifndef WF_PLANES_RULE_H
#define WF_PLANES_RULE_H

#if defined(__HIPCC__)
#define WF_PLR_HD __host__ __device__ static __forceinline__
#else
#define WF_PLR_HD static inline
#endif

#define WF_PL_LEN_MAX 512 /* longest transform */
#define WF_PL_LDS_MAX (160 * 1024)

/* LDS row stride of n reals: 4 times an odd number, so that the MFMA operand
 * reads (16 rows x 4 consecutive entries) hit distinct banks */
WF_PLR_HD int wf_pl_stride(int n) { return 4 * (((n + 3) / 4) | 1); }
/* levels of the tridiagonal tables: nz rounded up to whole chunks */
WF_PLR_HD int wf_pl_levels(int nz) { return (nz + 15) & ~15; }
/* half length (cosine terms) of n, and that rounded up to whole MFMA tiles */
WF_PLR_HD int wf_pl_half(int n) { return n / 2 + 1; }
WF_PLR_HD int wf_pl_tiles(int n) { return (wf_pl_half(n) + 15) / 16; }

/* LDS of a plane solve: the plane and the chunk ends of nt threads */
WF_PLR_HD long wf_pl_lds(int ny, int nz, int nt) {
    return 8 * (((long)nz * wf_pl_stride(ny + 1) + 3) & ~3l) + 16l * nt;
}

/* 16-level tiles per wave and levels per lane of a plane solve of nt threads
 * (0: more than the kernels are built for) */
WF_PLR_HD void wf_pl_shape(int ny, int nz, int nt, int *tpw, int *lc) {
    const int W = nt / 64, T = wf_pl_tiles(ny), nkt = (nz + 15) / 16;
    const int KG = W / T;
    const int need = (KG > 0) ? (nkt + KG - 1) / KG : 99;
    *tpw = (need <= 4) ? need : 0;
    *lc = ((nz + 3) / 4 * ((ny + 63) / 64) <= W) ? 4 : ((nz + 7) / 8 <= W) ? 8 : 0;
}

/* The instances (threads, tiles per wave, levels per lane) of the plane solve:
 * the ones that wf_pl_solve_nt and wf_pl_shape can choose. */
#define WF_PL_SOLVES(X) \
    X(256, 1, 4) X(256, 1, 8) X(512, 1, 4) X(512, 1, 8) X(512, 2, 8) X(1024, 1, 4) X(1024, 1, 8) X(1024, 2, 8) \
    X(1024, 3, 8) X(1024, 4, 8)

/* Threads of the one-launch plane solve; 0 where three launches take it: planes
 * that do not fit LDS or its kernels (more than 128 levels: 16 to a lane spill
 * 125-131 registers), and the planes of 16 waves, one to a CU, with two or more
 * tiles to a wave where half of the CUs have none.  us per solve, a step's wall
 * time over its solves, one launch against three:
 *     16 levels to a lane: 63x63x160 70 | 52, 100x100x160 142 | 101, 256x64x160 165 | 158, 300x10x250 130 | 103
 *     nx <= 128: 64x64x99 57 | 50, 128x128x99 123 | 111, 64x256x64 125 | 93, 128x300x49 164 | 135
 *     above: 144x128x99 128 | 127, 160x64x99 78 | 79, 200x200x63 160 | 168, 401x401x39 476 | 545
 *     one tile to a wave: 127x63x127 55 | 62, 32x280x11 43 | 55, 32x32x99 34 | 31
 * (Three and four tiles to a wave spill 3 and 25 registers.) */
WF_PLR_HD int wf_pl_solve_nt(int nx, int ny, int nz) {
    for (int n = 256; n <= 1024; n *= 2) {
        int tpw, lc;
        wf_pl_shape(ny, nz, n, &tpw, &lc);
        const int most = (n == 256) ? 1 : (n == 512) ? 2 : 4;
        if (tpw == 0 || tpw > most || lc == 0 || wf_pl_lds(ny, nz, n) > WF_PL_LDS_MAX) continue;
        return (n == 1024 && tpw > 1 && nx <= 128) ? 0 : n;
    }
    return 0;
}

/* lengths whose mixed-radix passes are fast: a two-factor or three-radix
 * compile-time plan, or run-time radices of a butterfly per thread (and 11) */
WF_PLR_HD int wf_pl_planned(int n) { return n == 63 || n == 255 || n == 511; }
WF_PLR_HD int wf_pl_quick(int n) {
    if (wf_pl_planned(n)) return 1;
    for (int p = 2; p <= 11; p++)
        while (n % p == 0) n /= p;
    return n == 1;
}

/* Whether the planes take the solve, and the threads of the one-launch plane
 * solve.  They do up to 512 x 512 unless both lengths are quick and the n^2/2
 * multiply-adds of a length, one chain of matrix instructions to a wave, cost
 * more than two passes over memory: a length near 512, more than 256 planes (a
 * second one for some CUs) of at least 128 columns, long x beside few columns,
 * planes that do not fit LDS from 200 x 200 on, and planned lengths with 255 or
 * 511 columns.  us per solve (a step's wall time over its solves),
 * planes | passes:
 *   by planes:  127x127x63 60 | 111    254x254x63 197 | 839    256x64x64 72 | 97      200x320x39 169 | 173
 *               240x300x39 173 | 182   300x80x39 83 | 92       128x128x160 153 | 176  257x257x39 236 | 1243
 *               310x310x39 278 | 366   401x401x39 476 | 3863
 *   by passes:  512x512x39 977 | 768   300x300x39 269 | 224    352x352x39 365 | 321   400x128x39 169 | 152
 *               128x400x39 185 | 165   240x384x39 235 | 233    512x8x11 95 | 55       16x500x39 119 | 83
 *               511x63x127 215 | 195   225x225x99 324 | 289    200x200x127 312 | 290  400x16x11 73 | 50
 * What the rule leaves: by planes 64x360x39 107 | 95, 255x300x39 174 | 164 and
 * 400x100x39 149 | 126 (but 420x120x29 105 | 117), by passes 462x220x29 209 | 215
 * and 240x400x39 243 | 248. */
WF_PLR_HD int wf_pl_takes(int nx, int ny, int nz, int *nt) {
    *nt = wf_pl_solve_nt(nx, ny, nz);
    if (nx > WF_PL_LEN_MAX || ny > WF_PL_LEN_MAX) return 0;
    if (!wf_pl_quick(nx) || !wf_pl_quick(ny)) return 1;
    if (wf_pl_planned(nx) && wf_pl_planned(ny) && ny >= 255) return 0;
    if (nx >= 480 || ny >= 384 || (nx > 256 && ny >= 128) || (nx >= 320 && ny <= 32)) return 0;
    return !(nx >= 200 && ny >= 200 && *nt == 0);
}

#endif
