/* The rules of the coefficient planes (wildfires_amd/csrc/hip/wf_planes_rule.h)
 * for the CPU check in tests/test_pressure_passes.py; test code only. */
#include "../../wildfires_amd/csrc/hip/wf_planes_rule.h"

/* threads, tiles per wave and levels per lane of an nx x ny x nz solve (threads
 * 0: three launches); 0: by the passes */
int plane_form(int nx, int ny, int nz, int *nt, int *tpw, int *lc) {
    const int takes = wf_pl_takes(nx, ny, nz, nt);
    *tpw = *lc = 0;
    if (takes && *nt) wf_pl_shape(ny, nz, *nt, tpw, lc);
    return takes;
}

/* Every solve up to 512 x 512 x 256 against the instances: 0, or 1 + the
 * number of one whose instance, LDS or work split is not there; used[q] counts
 * the solves of instance q, *ninst the instances. */
long plane_sweep(long *used, int *ninst) {
#define ONE(NT, TPW, LC) {NT, TPW, LC},
    static const int inst[][3] = {WF_PL_SOLVES(ONE)};
    const int n = sizeof(inst) / sizeof(inst[0]);
    *ninst = n;
    long at = 0;
    for (int nx = 4; nx <= WF_PL_LEN_MAX; nx++)
        for (int ny = 4; ny <= WF_PL_LEN_MAX; ny++)
            for (int nz = 5; nz <= 256; nz++) {
                int nt, tpw, lc, q = 0;
                at++;
                if (!plane_form(nx, ny, nz, &nt, &tpw, &lc) || nt == 0) continue;
                while (q < n && (inst[q][0] != nt || inst[q][1] != tpw || inst[q][2] != lc)) q++;
                if (q == n) return at;
                used[q]++;
                const int W = nt / 64, T = wf_pl_tiles(ny), KG = W / T, C = (nz + lc - 1) / lc;
                if (wf_pl_lds(ny, nz, nt) > WF_PL_LDS_MAX) return at;
                if (KG < 1 || 16 * KG * tpw < nz || C > W) return at; /* all levels have a tile and a chunk */
            }
    return 0;
}
