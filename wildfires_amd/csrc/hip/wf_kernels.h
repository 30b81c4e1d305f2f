/*
 * wf_kernels.h -- kernel launchers and device helpers shared between the
 * stage, pressure and projection translation units.
 */
#ifndef WF_KERNELS_H
#define WF_KERNELS_H

#include <vector>

#include "wf_common.h"
#include "wf_closure.h"
#include "wf_iter.h"
#include "wf_planes_rule.h"

namespace WF_NS {

/* k_stage modes (RK combination written by the stage pass) */
#define WF_MODE_PHI 0   /* out = k_s */
#define WF_MODE_FIRST 1 /* acc = k_1, out = y_n + a k_1 */
#define WF_MODE_MID 2   /* acc += 2 k_s, out = y_n + a k_s */
#define WF_MODE_LAST 3  /* out = y_n + a (acc + k_s) */
#define WF_MODE_EULER 4 /* out = y_n + a k_s */

/* Thermal conductivity by Sutherland's law and its T-derivative
 * (src/cu/pde.cu:692-695). */
__device__ __forceinline__ void wf_sutherland_k(wf_real T, wf_real *kT, wf_real *dk) {
    *kT = WR(0.0241) * pow(T / WR(273.15), WR(1.5)) * (WR(273.15) + 194) / (T + 194);
    *dk = WR(0.0241) * (WR(1.5) * pow(T / WR(273.15), WR(0.5)) * (WR(273.15) + 194) / (T + 194) -
                        pow(T / WR(273.15), WR(1.5)) * (WR(273.15) + 194) / ((T + 194) * (T + 194)));
}

/* Heat source q of the temperature RHS (src/cu/pde.cu:663-699): combustion
 * H_C Y K(T)/c_p minus the gas-solid exchange, with the gas/solid temperatures
 * of the fuel zone k <= Nz_Y.  The exchange term is h_c alpha_s sigma_s (...),
 * identically +-0 when alpha_s sigma_s = 0, in which case it is not formed
 * (q - (+-0) = q).  h_c is evaluated per node from the parameter value.
 * *Yout receives the node's fuel fraction (0 outside the stored fuel; read
 * from the FP64 Y and used in wf_real arithmetic). */
__device__ __forceinline__ wf_real wf_heat_source_y(const WfConst &c, int col, int i, int j, int k, wf_real T,
                                                    wf_real T_kp1, const double *Yf, wf_real *Yout) {
    wf_real K_T = wf_rate(c, T);
    wf_real T_gas = c.T_inf, T_solid = c.T_inf, Y = WR(0.0);
    int nzy = c.nzy[col];
    if (k <= nzy) {
        if (k < nzy)
            Y = (wf_real)Yf[(long)col + c.plane * (long)k];
        else
            T_gas = T_kp1;
        if (Y > WR(0.0))
            T_solid = T;
        else
            T_gas = T;
    }
    wf_real q = c.H_C * Y * K_T / c.c_p;
    if (c.exchange_on) {
        const wf_real *z = c.z;
        wf_real dz_k = (k < c.Nz - 1) ? z[k + 1] - z[k] : z[k] - z[k - 1];
        wf_real h_c = c.h_c * dz_k * pow(fabs(T_gas - T_solid) / dz_k, WR(1.0 / 4.0));
        q = q - h_c * c.alpha_s * c.sigma_s * (T_gas - T_solid) / (c.c_p * c.T_inf * c.rho_inf / T_gas);
    }
    *Yout = Y;
    return q;
}

__device__ __forceinline__ wf_real wf_heat_source(const WfConst &c, int col, int i, int j, int k, wf_real T,
                                                  wf_real T_kp1, const double *Yf) {
    wf_real Y;
    return wf_heat_source_y(c, col, i, j, k, T, T_kp1, Yf, &Y);
}

/* stage pass (wf_stage.hip) */
/* The derived pass (all derived fields), or with the learned closure and
 * mu_only mu_sgs and the u_tau plane alone, then the network pass over the
 * queued nodes. */
hipError_t wf_launch_derived(const WfConst &c, const WfState &X, const WfDerived &D, const WfClosure *cl,
                             const WfClosureQueue *cq, hipStream_t s, bool mu_only = false);
hipError_t wf_launch_closure_eval(const WfClosure &cl, const wf_real *feat, long n, wf_real *nu, int *learned,
                                  hipStream_t s);
hipError_t wf_launch_stage(const WfConst &c, const WfState &X, const WfDerived &D, const WfState &Yn,
                           const WfState &acc, const WfState &out, int mode, double a, bool closure, hipStream_t s);
/* The stage in one pass that evaluates the derived fields on the chip (u_tau
 * plane, stage tiles, column completion); D supplies the u_tau plane and the
 * kept raw RHS, and with the learned closure (closure) mu_sgs and u_tau as the
 * derived pass's mu-only form and the network pass left them.  shape: stage tile 32x8,
 * 16x16 or 16x8 (0, 1, 2); every shape gives the same results. */
hipError_t wf_launch_stage_fd(const WfConst &c, const WfState &X, const WfDerived &D, const WfState &Yn,
                              const WfState &acc, const WfState &out, int mode, double a, int shape, bool closure,
                              hipStream_t s);
/* the stage tiles alone (u_tau and the column completion not included) */
hipError_t wf_launch_stage_fd_only(const WfConst &c, const WfState &X, const WfDerived &D, const WfState &Yn,
                                   const WfState &acc, const WfState &out, int mode, double a, int shape, bool closure,
                                   hipStream_t s);
/* One member's operands of a batched RK stage (wf_launch_stage_batch). */
struct WfBatchStage {
    WfConst c;
    WfState X, Yn, acc, out;
    WfDerived D;
    int mode;
    double a;
};
/* Launch shape of the batched passes: the stage pass's tile shape (index
 * into 32x8, 16x16, 16x8), whether it is compiled for the exchange term and
 * Sutherland laws (general), and the workgroups of the u_tau, stage and
 * column launches (stage: > 0 a fixed grid looping over the items, < 0 one
 * workgroup per item, -grid[1] items). */
#define WF_BATCH_SHAPES 3
#define WF_STAGE_SHAPES WF_BATCH_SHAPES
#define WF_BATCH_PASSES (WF_BATCH_SHAPES + 2)
struct WfBatchShape {
    int shape;
    int general;
    int grid[3];
};
/* work items of a member: u_tau pass, stage pass per tile shape, column pass */
void wf_batch_items(const WfConst &c, int items[WF_BATCH_PASSES]);
/* One RK stage of nm members, one launch per pass (u_tau, stage with the
 * derived fields on the chip, column completion).  first holds
 * WF_BATCH_PASSES prefix arrays of nm + 1 entries (member m owns items
 * [first[m], first[m+1]) of that pass). */
hipError_t wf_launch_stage_batch(const WfBatchStage *B, const int *first, int nm, const WfBatchShape &sh,
                                 hipStream_t s);
hipError_t wf_launch_utau_batch(const WfBatchStage *B, const int *first, int nm, const WfBatchShape &sh,
                                hipStream_t s);
hipError_t wf_launch_stage_only_batch(const WfBatchStage *B, const int *first, int nm, const WfBatchShape &sh,
                                      hipStream_t s);
hipError_t wf_launch_columns_batch(const WfBatchStage *B, const int *first, int nm, const WfBatchShape &sh,
                                   hipStream_t s);
/* reference layout (FP64, z fastest) <-> internal layout in type D (wf_real
 * for u, v, w, T, p; double for Y) */
template <typename D>
hipError_t wf_launch_to_internal(const double *src, D *dst, int Nx, int Ny, int nz, hipStream_t s);
template <typename D>
hipError_t wf_launch_to_reference(const D *src, double *dst, int Nx, int Ny, int nz, hipStream_t s);

/* pressure pass (wf_pressure.hip) */

/* Device-side control of the variable-density pressure iteration. */
struct WfIterCtl {
    int done;   /* once converged or out of iterations, 1 + the last solve's index (wf_iter.h) */
    int iters;  /* the count the reference reports */
    int solves; /* solves performed */
    double err; /* last max |p_new - p_old| */
};
/* Its copy in mapped host memory, written by every check (done, 0 or 1, last): the
 * host follows the iteration by it and takes the results from it. */
struct WfHostFlag {
    int done, solves, iters;
    double err;
};

/* Row pairs per workgroup in the x-transforms and kx columns per workgroup in
 * the y-transform, for a transform length n. */
#ifndef WF_FX_PAIRS
#define WF_FX_PAIRS 4
#endif
__host__ __device__ constexpr int wf_pairs_for(int n) {
    return (WF_MIXED && n == 255) ? 8 : (n <= 300) ? WF_FX_PAIRS : 2;
}
/* lengths with a compile-time plan */
__host__ __device__ constexpr bool wf_planned(int n) { return n == 63 || n == 127 || n == 255 || n == 511; }
#define WF_FY_COLS 4
/* kx columns per workgroup of the in-place y-transform (lengths without a
 * two-factor plan).  Batched launches (many members, workgroups to spare) of
 * the prime 127 take 16: its single radix-127 stage then gives each of 16
 * threads per column 4 output pairs to accumulate from every input pair it
 * reads from LDS, against one pair each of 64 threads with 4 columns.  A
 * single grid keeps 4, for 4 times the workgroups.  Each output is summed in
 * the same order either way, so the results do not depend on the choice. */
__host__ __device__ constexpr int wf_fy_ip_cols(int n, bool batch) { return (batch && n == 127) ? 16 : WF_FY_COLS; }
/* z-levels per lane in the chunked tridiagonal solve and the largest nz */
#define WF_THOMAS_MAX_CHUNKS 16
/* half-wave chunks of 4 levels (k_thomas_h) for up to 128 levels: measured
 * slower (37.5 us against 33.0 us at 256x256x128, its 32-chunk combine is a
 * longer serial LDS chain), so off by default */
#ifndef WF_THOMAS_HALF
#define WF_THOMAS_HALF 0
#endif
#define WF_NZ_MAX (16 * WF_THOMAS_MAX_CHUNKS)

struct WfSpectral {
    int nx, ny, nz; /* unique nodes per direction: Nx-1, Ny-1, Nz-1 */
    int hx;         /* nx/2 + 1 retained x-wavenumbers */
    int ldj;        /* ny rounded up to a multiple of 8: stride of one kx column */
    int fx_pairs;   /* row pairs per workgroup in the x-transforms */
    int fy_cols;    /* kx columns per workgroup in the y-transform */
    int ngroups;    /* row-pair groups per slab in the x-transforms */
    int npmax;      /* workgroups of the inverse x-transform (partial maxima) */
    wf_real2 *F;    /* [nz][hx][ldj] spectral working buffer (ky fastest) */
    wf_real2 *Ptop; /* [hx][ldj] spectrum of the top pressure plane */
    wf_real *A;     /* Nx*Ny*Nz: p-independent part of the Poisson RHS */
    const double *UB;    /* [chunk][hx][ldj]: Thomas pivot u_{k0-1} entering each z-chunk (chunk >= 1), FP64 */
    int thomas_lc;       /* z-levels per chunk of the tridiagonal solve */
    double *pmax;        /* npmax partial maxima of |p_new - p_old| (mixed form: then npmax of |p_new|) */
    const wf_real *kx2;  /* hx: kx^2 of the retained x-wavenumbers */
    const wf_real *ky2;  /* ny */
    const wf_real *ta;   /* nz-1: sub-diagonal a_k (k-only), 0 up to a multiple of 16 */
    const wf_real *tc;   /* nz-1: super-diagonal c_k for k >= 1 (c_0 depends on K^2), 0 up to a multiple of 16 */
    /* the same tables in FP64, for the systems solved in FP64 (all of them in
     * the wf64 compilation, the lowest wavenumbers in the mixed one) */
    const double *kx2d, *ky2d, *tad, *tcd, *betad;
    int low_kx, low_ky;  /* mixed form: kx < low_kx and min(ky, ny-ky) < low_ky are solved in FP64 */
    const wf_real2 *twx; /* nx twiddles exp(-2 pi i e / nx) */
    const wf_real2 *twy; /* ny twiddles exp(-2 pi i e / ny) */
    const int *radx;     /* radices of nx, 0-terminated (<= 16 entries) */
    const int *rady;
    double dz0, top_div, c0a, c0b; /* c_0 = c0a - 0.5 dz0 K^2 - c0b */
    double b0;                     /* b_0 = -1/dz0 */
    double beta_top;               /* 2/(dz_{Nz-2} dz_{Nz-1}) */
    const wf_real *beta;           /* nz: 2/(dz_{k-1} dz_k) for 1 <= k <= nz-1, 1 up to a multiple of 16 */
    const wf_real *rho;            /* rho^n on every node (variable density) */
    WfIterCtl *ctl;
    WfHostFlag *hflag;             /* mapped host memory */
    /* coefficient-plane form (wf_planes.hip, FP64), used when pl is set (wf_pl_takes) */
    int pl;
    int pl_ld;          /* row stride of a plane: ny rounded up to 16 */
    int pl_groups;      /* 16-row groups per slab */
    int pl_nt;          /* threads of the plane solve; 0: three launches */
    wf_real *U;         /* [nx][nz][pl_ld] planes of real x-coefficients */
    const wf_real *pl_fx, *pl_ix, *pl_fy, *pl_iy; /* MFMA operands of the transforms (wf_pl_matrix) */
    wf_real *pl_l, *pl_ru;  /* [hx][nz up to 16][ny/2+1]: Thomas multipliers l_k and reciprocal pivots 1/u_k */
};

/* Forms of the x-transform input: the Poisson RHS of a later iteration (stored
 * p-independent part + pressure term), of the first iteration (also stores
 * that part), of the constant-density solve, and the top pressure plane. */
enum { WF_F_ITER = 0, WF_F_FIRST = 1, WF_F_CONST = 2, WF_F_TOP = 3 };

hipError_t wf_launch_pressure_rhs_fx(const WfConst &c, const WfSpectral &sp, const WfState &Ys, const WfState &Yn,
                                     const wf_real *p, int mode, double tol, double rtol, int check, int max_iter,
                                     hipStream_t s);
hipError_t wf_launch_fy(const WfSpectral &sp, wf_real2 *buf, long slab_stride, int slab0, int nslabs, int sign,
                        int guarded, hipStream_t s);
hipError_t wf_launch_density(const WfConst &c, const wf_real *T, wf_real *rho, hipStream_t s);
hipError_t wf_launch_iter_reset(WfIterCtl *ctl, hipStream_t s);
hipError_t wf_launch_thomas(const WfSpectral &sp, hipStream_t s);
hipError_t wf_launch_pivots(const WfSpectral &sp, double *UB, hipStream_t s);
hipError_t wf_launch_inverse_fx(const WfConst &c, const WfSpectral &sp, wf_real *p, hipStream_t s);
hipError_t wf_launch_iter_check(const WfSpectral &sp, double tol, double rtol, int m, int max_iter, hipStream_t s);

/* Coefficient-plane form of the solve (wf_planes.hip). */
#define WF_PL_ROWS 16     /* rows per workgroup in the x-transforms */
/* MFMA operand tables of a real transform of length n: forward and inverse */
void wf_pl_matrix(int n, std::vector<double> &fwd, std::vector<double> &inv);
hipError_t wf_pl_prepare(const WfSpectral &sp, hipStream_t s);
hipError_t wf_launch_pl_rhs(const WfConst &c, const WfSpectral &sp, const WfState &Ys, const WfState &Yn,
                            const wf_real *p, int mode, double tol, double rtol, int check, int max_iter,
                            hipStream_t s);
hipError_t wf_launch_pl_solve(const WfSpectral &sp, hipStream_t s);
hipError_t wf_launch_pl_inv(const WfConst &c, const WfSpectral &sp, wf_real *p, hipStream_t s);

/* One member's operands for the batched pressure passes of an ensemble.  The
 * members of a size class (same grid, precision and iteration limit) run each
 * pass as one launch: the solo launch's grid, with z the member in the class's
 * table. */
struct WfPressItem {
    WfConst c;
    WfSpectral sp;
    WfState ys, yn; /* y* and y_n of the solve */
    wf_real *p;
    wf_real *rho; /* rho^n, written by the density pass (sp.rho reads it) */
    double tol, rtol;
    int max_iter;
};
hipError_t wf_launch_density_batch(const WfConst &c, const WfPressItem *tab, int nm, hipStream_t s);
hipError_t wf_launch_iter_reset_batch(const WfPressItem *tab, int nm, hipStream_t s);
hipError_t wf_launch_pressure_rhs_fx_batch(const WfSpectral &sp, const WfPressItem *tab, int nm, int mode, int check,
                                           hipStream_t s);
hipError_t wf_launch_fy_batch(const WfSpectral &sp, const WfPressItem *tab, int nm, long slab_stride, int slab0,
                              int nslabs, int sign, int guarded, hipStream_t s);
hipError_t wf_launch_thomas_batch(const WfSpectral &sp, const WfPressItem *tab, int nm, hipStream_t s);
hipError_t wf_launch_inverse_fx_batch(const WfSpectral &sp, const WfPressItem *tab, int nm, hipStream_t s);
hipError_t wf_launch_iter_check_batch(const WfPressItem *tab, int nm, int m, hipStream_t s);
hipError_t wf_launch_pl_rhs_batch(const WfSpectral &sp, const WfPressItem *tab, int nm, int mode, int check,
                                  hipStream_t s);
hipError_t wf_launch_pl_solve_batch(const WfSpectral &sp, const WfPressItem *tab, int nm, hipStream_t s);
hipError_t wf_launch_pl_inv_batch(const WfSpectral &sp, const WfPressItem *tab, int nm, hipStream_t s);

/* Temperature source applied at the end of a step (src/cu/functions.cu:325-403). */
struct WfSource {
    int mode;  /* 0 none, 1 max(T, T at t_0), 2 delayed shape */
    int shape; /* mode 2: 1 gaussian, 2 parallelepiped, 0 none */
    wf_real scale, T_inf, T_source;
    wf_real xc, yc, zc, sx, sy, sz;
    wf_real x0, x1, y0, y1, z0, z1;
    const wf_real *x, *y; /* node coordinates */
    const wf_real *T_src; /* mode 1: T at the start of the run (internal layout) */
};

/* checkpoint reports (wf_reports.hip): WF_REP_N partial values per workgroup,
 * max |u|, |v|, |w|, min T, max T, min Y, max Y (fuel box), sum of the kinetic
 * energy, burned fuel columns, fuel columns, nodes with a learned viscosity */
#define WF_REP_N 11
#define WF_REP_BLOCKS 2048
hipError_t wf_launch_reports(const WfConst &c, const WfState &X, const wf_real *mu_sgs, const int *in_box,
                             double *part, int nblocks, unsigned long long *nan_first, hipStream_t s);

/* projection pass (wf_project.hip) */
hipError_t wf_launch_project(const WfConst &c, const WfState &Ys, const WfState &Yn, const wf_real *p,
                             const WfState &out, const WfSource &src, hipStream_t s);

}  // namespace WF_NS

/* library-wide helpers (wf_api.hip), outside the precision namespaces */
int wf_set_error(int code, const char *msg);
uint16_t wf_bf16_bits(float f);

/* Scratch of the entry points that allocate nothing (wf_noalloc.hip): a
 * static device array of WF_NOALLOC_DOUBLES doubles per GPU holding the
 * report partials of up to WF_REP_BLOCKS workgroups, the reduced values at
 * WF_NA_FINAL and the first-NaN slot at WF_NA_NAN. */
#define WF_NA_FINAL (WF_REP_N * WF_REP_BLOCKS)
#define WF_NA_NAN (WF_NA_FINAL + WF_REP_N)
#define WF_NOALLOC_DOUBLES (WF_NA_NAN + 1)
/* device address of the scratch array on `device` (looked up once per device) */
hipError_t wf_noalloc_scratch(int device, double **base);
hipError_t wf_launch_fill_u64(unsigned long long *p, unsigned long long v, hipStream_t s);
/* fin[0..WF_REP_N) <- reduction of nb partial rows, as the host reduction of
 * wf_solver_reports */
hipError_t wf_launch_reports_final(const double *part, int nb, double *fin, hipStream_t s);

#endif
