/*
 * Solver.hip -- host side of the time step, in one precision: device
 * workspace, the step sequence of src/cu/solver.cu:178-265 and the pieces the
 * C-ABI exposes (wf_api.hip dispatches to the wf64 or the wf32 compilation).
 *
 * Device buffers (internal layout, see wf_common.h):
 *   state[4]  four state vectors: u, v, w, T in wf_real and Y in FP64
 *             (max(Nz_Y_max, 1) planes); y_n, two stage inputs and the running
 *             RK combination; roles rotate between steps
 *   derived   8 N + 21 Nx Ny: per-node fields the SGS divergence reads at
 *             neighbours, u_tau and the kept raw RHS of the column passes
 *   p, A      pressure and the p-independent part of the Poisson RHS
 *   F, Ptop   x-half-spectrum working buffer [Nz-1][(Nx-1)/2+1][ldj] and the
 *             spectrum of the top pressure plane; UB the Thomas pivots (FP64)
 */
#include <math.h>
#include <stdint.h>
#include <cmath>
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <vector>

#include "../../../include/wildfires.h"
#include "wf_common.h"
#include "wf_core.h"
#include "wf_fft.h"
#include "wf_kernels.h"

#define WF_MAX_EVENTS 512
/* mixed form: relative stopping tolerance of the pressure iteration */
#ifndef WF_MIXED_PRESSURE_RTOL
#define WF_MIXED_PRESSURE_RTOL 3e-5
#endif

#define WF_HIP(call)                                                                              \
    do {                                                                                          \
        hipError_t e_ = (call);                                                                   \
        if (e_ != hipSuccess)                                                                     \
            return wf_fail(WF_E_DEVICE, "%s:%d %s: %s", __FILE__, __LINE__, #call, hipGetErrorString(e_)); \
    } while (0)

namespace WF_NS {

struct Solver {
    Parameters P;
    WfConst c;
    WfSpectral sp;
    long N, S, plane;
    long ny_planes;  /* Y planes on the device: max(Nz_Y_max, 1) */
    size_t sbytes;   /* bytes of one device state vector */
    int device;      /* the HIP device of the solver's buffers and stream */
    hipStream_t stream;
    char *state[4];
    int i_yn, i_x0, i_x1, i_acc;
    wf_real *derived;
    wf_real *p, *A;
    double *UB, *pmax;
    wf_real2 *F, *Ptop;
    wf_real *z, *cd2, *delta_k, *zc, *topo, *kx2, *ky2, *ta, *tc, *beta, *x, *y;
    double *kx2d, *ky2d, *tad, *tcd, *betad; /* FP64 copies (the mixed form's low wavenumbers) */
    /* learned closure (off unless wf_solver_set_closure gave parameters) */
    float *cl_prm;
    wf_bf16x8 *cl_frag;
    int closure_on;
    unsigned *clq_count, *clq_node; /* queue of the nodes the network evaluates */
    wf_bf16x8 *clq_x;
    wf_real *clq_rho;
    unsigned clq_cap;
    int clq_parity; /* which of the two counter sets the next derived pass appends to */
    int *cut, *nzy, *radx, *rady;
    wf_real *U, *pl_tab, *pl_piv; /* coefficient-plane form of the pressure solve */
    wf_real2 *twx, *twy;
    double *scratch; /* S doubles: host transfers in the reference layout */
    wf_real *Tsrc, *rho;
    int have_Tsrc;
    WfIterCtl *ctl;
    WfHostFlag *hflag;     /* mapped pinned host memory */
    WfHostFlag *hflag_dev; /* its device address */
    int method; /* 0 Euler, 1 RK2, 2 RK4 */
    int stage_split; /* 1: derived pass + stage pass also without the closure (WF_STAGE_FORM=split) */
    int stage_shape; /* stage tile shape (-1 until tuned at the first stage) */
    int cl_inplace_min; /* WfClosure::inplace_min (WF_CL_INPLACE_MIN) */
    float stage_ms[WF_STAGE_SHAPES]; /* the tuning's per-shape stage times (ms) */
    long press_solves, steps;
    double press_rtol; /* mixed form: relative stopping tolerance of the pressure iteration */
    /* checkpoint reports: fuel-box column mask, per-workgroup partials, first NaN */
    int *in_box;
    double *rep_part;
    unsigned long long *rep_nan;
    /* asynchronous checkpoints (allocated at the first one): the state and p in
     * the reference layout on the device and in pinned host memory, the copy
     * stream and its events */
    double *ck_dev, *ck_host;
    hipStream_t ck_stream;
    hipEvent_t ck_conv, ck_done;
    int ck_pending;
    double last_err;
    int last_iters;
    /* profiling */
    int profiling;
    hipEvent_t ev[2 * WF_MAX_EVENTS];
    int ev_kind[WF_MAX_EVENTS];
    int n_ev;
    double k_ms[WF_K_COUNT];
    long k_count[WF_K_COUNT];
};

/* u, v, w, T (wf_real) followed by Y (FP64; 4 N wf_real is a multiple of 8 bytes) */
static WfState wf_view(const Solver *s, char *base) {
    WfState v;
    wf_real *f = (wf_real *)base;
    v.u = f;
    v.v = f + s->N;
    v.w = f + 2 * s->N;
    v.T = f + 3 * s->N;
    v.Y = (double *)(base + sizeof(wf_real) * 4 * s->N);
    return v;
}

static WfDerived wf_derived_view(const Solver *s) {
    WfDerived d;
    wf_real *b = s->derived;
    long N = s->N;
    d.mu = b;
    d.s11 = b + N;
    d.s12 = b + 2 * N;
    d.s13 = b + 3 * N;
    d.s22 = b + 4 * N;
    d.s23 = b + 5 * N;
    d.s33 = b + 6 * N;
    d.divU = b + 7 * N;
    d.utau = b + 8 * N;
    d.col = b + 8 * N + s->plane;
    return d;
}

static int wf_factor(int n, int *rad) {
    int cnt = 0;
    while (n % 4 == 0 && cnt < WF_MAX_RADICES - 1) {
        rad[cnt++] = 4;
        n /= 4;
    }
    while (n % 2 == 0 && cnt < WF_MAX_RADICES - 1) {
        rad[cnt++] = 2;
        n /= 2;
    }
    for (int p = 3; n > 1 && cnt < WF_MAX_RADICES - 1; p += 2)
        while (n % p == 0 && cnt < WF_MAX_RADICES - 1) {
            rad[cnt++] = p;
            n /= p;
        }
    if (n != 1) return -1;
    for (int q = cnt; q < WF_MAX_RADICES; q++) rad[q] = 0;
    return cnt;
}

template <typename T>
static int wf_upload(T **dst, const T *src, size_t count) {
    WF_HIP(hipMalloc((void **)dst, sizeof(T) * (count > 0 ? count : 1)));
    if (count > 0) WF_HIP(hipMemcpy(*dst, src, sizeof(T) * count, hipMemcpyHostToDevice));
    return WF_OK;
}

/* an FP64 host table in wf_real on the device (rounded once, on the host) */
static int wf_upload_real(wf_real **dst, const double *src, size_t count) {
    std::vector<wf_real> v(src, src + count);
    return wf_upload(dst, v.data(), count);
}
static int wf_upload_real2(wf_real2 **dst, const std::vector<double2> &src) {
    std::vector<wf_real2> v(src.size());
    for (size_t q = 0; q < src.size(); q++) {
        v[q].x = (wf_real)src[q].x;
        v[q].y = (wf_real)src[q].y;
    }
    return wf_upload(dst, v.data(), v.size());
}

/* ------------------------------------------------------------ profiling ---- */

static int wf_prof_begin(Solver *s, int kind) {
    if (!s->profiling || s->n_ev >= WF_MAX_EVENTS) return -1;
    int slot = s->n_ev++;
    s->ev_kind[slot] = kind;
    (void)hipEventRecord(s->ev[2 * slot], s->stream);
    return slot;
}

static void wf_prof_end(Solver *s, int slot) {
    if (slot >= 0) (void)hipEventRecord(s->ev[2 * slot + 1], s->stream);
}

static int wf_prof_collect(Solver *s) {
    if (!s->profiling) return WF_OK;
    WF_HIP(hipStreamSynchronize(s->stream));
    for (int q = 0; q < s->n_ev; q++) {
        float ms = 0.0f;
        WF_HIP(hipEventElapsedTime(&ms, s->ev[2 * q], s->ev[2 * q + 1]));
        s->k_ms[s->ev_kind[q]] += (double)ms;
        s->k_count[s->ev_kind[q]] += 1;
    }
    s->n_ev = 0;
    return WF_OK;
}

#define WF_LAUNCH(solver, kind, expr)                                                        \
    do {                                                                                     \
        int slot_ = wf_prof_begin((solver), (kind));                                         \
        hipError_t e_ = (expr);                                                              \
        wf_prof_end((solver), slot_);                                                        \
        if (e_ != hipSuccess)                                                                \
            return wf_fail(WF_E_DEVICE, "launch %s: %s", #expr, hipGetErrorString(e_));     \
    } while (0)

/* ----------------------------------------------------------- lifecycle ---- */

static int wf_validate(const Parameters *P) {
    if (P->Nx < 5 || P->Ny < 5) return wf_fail(WF_E_ARG, "Nx and Ny must be at least 5 (got %d, %d)", P->Nx, P->Ny);
    if (P->Nx - 1 > 1024 || P->Ny - 1 > 1024)
        return wf_fail(WF_E_ARG, "Nx-1 and Ny-1 must not exceed 1024 (got %d, %d)", P->Nx - 1, P->Ny - 1);
    if (P->Nz < 6) return wf_fail(WF_E_ARG, "Nz must be at least 6 (got %d)", P->Nz);
    if (P->Nz - 1 > WF_NZ_MAX) return wf_fail(WF_E_ARG, "Nz-1 must not exceed %d (got %d)", WF_NZ_MAX, P->Nz - 1);
    if ((long)P->Nx * P->Ny * P->Nz > (1L << 28))
        return wf_fail(WF_E_ARG, "Nx*Ny*Nz must not exceed 2^28 (got %ld)", (long)P->Nx * P->Ny * P->Nz);
    if (P->z == NULL || P->cut_nodes == NULL || P->Nz_Y == NULL || P->topography == NULL)
        return wf_fail(WF_E_ARG, "parameters have no grids or terrain mask");
    long cols = (long)P->Nx * P->Ny;
    for (long q = 0; q < cols; q++)
        if (P->cut_nodes[q] > P->Nz - 4 || P->cut_nodes[q] < 0)
            return wf_fail(WF_E_ARG, "terrain reaches the top: cut node %d of column %ld exceeds Nz-4", P->cut_nodes[q], q);
    return WF_OK;
}

static int wf_method(const Parameters *P) {
    if (strncmp(P->method, "Euler", 5) == 0) return 0;
    if (strncmp(P->method, "RK2", 3) == 0) return 1;
    if (strncmp(P->method, "RK4", 3) == 0) return 2;
    return -1;
}

static int wf_create_impl(Solver *s, const Parameters *P) {
    int rc = wf_validate(P);
    if (rc != WF_OK) return rc;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1)
        return wf_fail(WF_E_DEVICE, "no HIP device available");
    WF_HIP(hipSetDevice(0));
    s->device = 0;
    s->P = *P;
    const int Nx = P->Nx, Ny = P->Ny, Nz = P->Nz, Nzm = P->Nz_Y_max;
    s->plane = (long)Nx * Ny;
    s->N = s->plane * Nz;
    s->S = 4 * s->N + s->plane * Nzm;
    s->ny_planes = (Nzm > 0) ? Nzm : 1;
    s->sbytes = sizeof(wf_real) * 4 * s->N + sizeof(double) * s->plane * s->ny_planes;
    s->method = wf_method(P);
    {
        const char *form = getenv("WF_STAGE_FORM");
        s->stage_split = (form != NULL && strcmp(form, "split") == 0) ? 1 : 0;
        const char *shp = getenv("WF_STAGE_SHAPE");
        s->stage_shape = (shp != NULL) ? atoi(shp) % WF_STAGE_SHAPES : -1;
        const char *inp = getenv("WF_CL_INPLACE_MIN");
        s->cl_inplace_min = (inp != NULL) ? atoi(inp) : WfClosure{}.inplace_min;
    }
    WF_HIP(hipStreamCreate(&s->stream));
    for (int q = 0; q < 4; q++) {
        WF_HIP(hipMalloc((void **)&s->state[q], s->sbytes));
        WF_HIP(hipMemset(s->state[q], 0, s->sbytes));
    }
    s->i_yn = 0;
    s->i_x0 = 1;
    s->i_x1 = 2;
    s->i_acc = 3;
    WF_HIP(hipMalloc((void **)&s->derived, sizeof(wf_real) * (8 * s->N + 21 * s->plane)));
    WF_HIP(hipMemset(s->derived, 0, sizeof(wf_real) * (8 * s->N + 21 * s->plane)));
    WF_HIP(hipMalloc((void **)&s->p, sizeof(wf_real) * s->N));
    WF_HIP(hipMemset(s->p, 0, sizeof(wf_real) * s->N));
    WF_HIP(hipMalloc((void **)&s->A, sizeof(wf_real) * s->N));
    WF_HIP(hipMalloc((void **)&s->scratch, sizeof(double) * s->S));
    WF_HIP(hipMalloc((void **)&s->Tsrc, sizeof(wf_real) * s->N));
    WF_HIP(hipMalloc((void **)&s->rho, sizeof(wf_real) * s->N));
    WF_HIP(hipMalloc((void **)&s->ctl, sizeof(WfIterCtl)));
    WF_HIP(hipMemset(s->ctl, 0, sizeof(WfIterCtl)));
    WF_HIP(hipHostMalloc((void **)&s->hflag, sizeof(WfHostFlag), hipHostMallocMapped));
    WF_HIP(hipHostGetDevicePointer((void **)&s->hflag_dev, s->hflag, 0));
    memset(s->hflag, 0, sizeof(WfHostFlag));

    /* grid tables evaluated on the host exactly as the reference evaluates them */
    const double *z = P->z;
    std::vector<double> cd2(Nz), delta_k(Nz);
    for (int k = 0; k < Nz; k++) {
        double dz_k = (k < Nz - 1) ? z[k + 1] - z[k] : z[k] - z[k - 1];
        delta_k[k] = pow(P->dx * P->dy * dz_k, 1.0 / 3.0);
        cd2[k] = pow(P->C_s * delta_k[k], 2.0);
    }
    /* z-stencil coefficients: the weights of the reference's difference
     * formulas (src/cu/pde.cu:363-385, 497-500, 539-542, 572) per plane */
    std::vector<double> zc((size_t)WF_ZC * Nz, 0.0);
    for (int k = 0; k < Nz; k++) {
        double *e = &zc[(size_t)WF_ZC * k];
        if (k <= Nz - 3) {
            double h0 = z[k + 1] - z[k], h1 = z[k + 2] - z[k + 1];
            e[WF_Z_D1F + 0] = -(2 * h0 + h1) / (h0 * (h0 + h1));
            e[WF_Z_D1F + 1] = (h0 + h1) / (h0 * h1);
            e[WF_Z_D1F + 2] = -h0 / (h1 * (h0 + h1));
        }
        if (k >= 2) {
            double hm2 = z[k - 1] - z[k - 2], hm1 = z[k] - z[k - 1];
            e[WF_Z_D1B + 0] = hm1 / (hm2 * (hm2 + hm1));
            e[WF_Z_D1B + 1] = -(hm2 + hm1) / (hm2 * hm1);
            e[WF_Z_D1B + 2] = (hm2 + 2 * hm1) / (hm1 * (hm2 + hm1));
        }
        if (k >= 1 && k <= Nz - 2) {
            double hm1 = z[k] - z[k - 1], h0 = z[k + 1] - z[k];
            e[WF_Z_D2M + 0] = 2 / (hm1 * (hm1 + h0));
            e[WF_Z_D2M + 1] = -2 / (hm1 * h0);
            e[WF_Z_D2M + 2] = 2 / (h0 * (hm1 + h0));
            e[WF_Z_DZC] = 1 / (hm1 + h0);
        }
        if (k == 0) {
            double h0 = z[1] - z[0], h1 = z[2] - z[1], h2 = z[3] - z[2];
            e[WF_Z_D2F + 0] = (6 * h0 + 4 * h1 + 2 * h2) / (h0 * (h0 + h1) * (h0 + h1 + h2));
            e[WF_Z_D2F + 1] = -(4 * h0 + 4 * h1 + 2 * h2) / (h0 * h1 * (h1 + h2));
            e[WF_Z_D2F + 2] = (4 * h0 + 2 * h1 + 2 * h2) / (h1 * h2 * (h0 + h1));
            e[WF_Z_D2F + 3] = -(4 * h0 + 2 * h1) / (h2 * (h1 + h2) * (h0 + h1 + h2));
        }
        if (k == Nz - 1) {
            double hm1 = z[k] - z[k - 1], hm2 = z[k - 1] - z[k - 2], hm3 = z[k - 2] - z[k - 3];
            e[WF_Z_D2B + 0] = -(2 * hm2 + 4 * hm1) / (hm3 * (hm3 + hm2) * (hm3 + hm2 + hm1));
            e[WF_Z_D2B + 1] = (2 * hm3 + 2 * hm2 + 4 * hm1) / (hm3 * hm2 * (hm2 + hm1));
            e[WF_Z_D2B + 2] = -(2 * hm3 + 4 * hm2 + 4 * hm1) / (hm2 * hm1 * (hm3 + hm2));
            e[WF_Z_D2B + 3] = (2 * hm3 + 4 * hm2 + 6 * hm1) / (hm1 * (hm2 + hm1) * (hm3 + hm2 + hm1));
        }
    }
    if ((rc = wf_upload_real(&s->z, z, Nz))) return rc;
    if ((rc = wf_upload_real(&s->cd2, cd2.data(), Nz))) return rc;
    if ((rc = wf_upload_real(&s->delta_k, delta_k.data(), Nz))) return rc;
    if ((rc = wf_upload_real(&s->zc, zc.data(), zc.size()))) return rc;
    if ((rc = wf_upload_real(&s->x, P->x, Nx))) return rc;
    if ((rc = wf_upload_real(&s->y, P->y, Ny))) return rc;
    /* masks: the host arrays are indexed (i, j) with j fastest; the device
     * tables are indexed col = i + Nx j */
    std::vector<int> cut(s->plane), nzy(s->plane);
    std::vector<double> topo(s->plane);
    for (int i = 0; i < Nx; i++)
        for (int j = 0; j < Ny; j++) {
            cut[i + (long)Nx * j] = P->cut_nodes[(long)j + (long)Ny * i];
            nzy[i + (long)Nx * j] = P->Nz_Y[(long)j + (long)Ny * i];
            topo[i + (long)Nx * j] = P->topography[(long)j + (long)Ny * i];
        }
    if ((rc = wf_upload_real(&s->topo, topo.data(), s->plane))) return rc;
    if ((rc = wf_upload(&s->cut, cut.data(), s->plane))) return rc;
    if ((rc = wf_upload(&s->nzy, nzy.data(), s->plane))) return rc;
    /* the fuel box of the checkpoint reports (src/cu/functions.cu:94-96) */
    std::vector<int> in_box(s->plane);
    for (int i = 0; i < Nx; i++)
        for (int j = 0; j < Ny; j++)
            in_box[i + (long)Nx * j] = P->Y0_x_start <= P->x[i] && P->x[i] <= P->Y0_x_end &&
                                       P->Y0_y_start <= P->y[j] && P->y[j] <= P->Y0_y_end;
    if ((rc = wf_upload(&s->in_box, in_box.data(), s->plane))) return rc;
    WF_HIP(hipMalloc((void **)&s->rep_part, sizeof(double) * WF_REP_N * WF_REP_BLOCKS));
    WF_HIP(hipMalloc((void **)&s->rep_nan, sizeof(unsigned long long)));

    WfConst &c = s->c;
    memset(&c, 0, sizeof(c));
    c.Nx = Nx;
    c.Ny = Ny;
    c.Nz = Nz;
    c.Nzm = Nzm;
    c.plane = s->plane;
    c.N = s->N;
    c.dx = P->dx;
    c.dy = P->dy;
    c.dt = P->dt;
    c.mu = P->mu;
    c.kT = P->k;
    c.Y_f = P->Y_f;
    c.H_C = P->H_C;
    c.A = P->A;
    c.T_act = P->T_act;
    c.T_pc = P->T_pc;
    c.h_c = P->h_c;
    c.alpha_s = P->alpha_s;
    c.sigma_s = P->sigma_s;
    c.T_inf = P->T_inf;
    c.c_p = P->c_p;
    c.rho_inf = P->rho_inf;
    c.C_d = P->C_d;
    c.g = P->g;
    c.delta = P->delta;
    c.Pr = P->Pr;
    c.T_min = P->T_min;
    c.T_max = P->T_max;
    c.Y_min = P->Y_min;
    c.Y_max = P->Y_max;
    c.u_dead = P->u_dead_nodes;
    c.v_dead = P->v_dead_nodes;
    c.w_dead = P->w_dead_nodes;
    c.T_dead = P->T_dead_nodes;
    c.Y_dead = P->Y_dead_nodes;
    c.temperature_convection = P->temperature_convection;
    c.suth_mu = P->sutherland_viscosity;
    c.suth_k = P->sutherland_conductivity;
    c.variable_density = P->variable_density;
    c.fd_z = P->velocity_correction_fd;
    c.exchange_on = (P->alpha_s * P->sigma_s != 0.0);
    c.z = s->z;
    c.cd2 = s->cd2;
    c.delta_k = s->delta_k;
    c.zc = s->zc;
    c.inv2dx = 1.0 / (2 * P->dx);
    c.inv2dy = 1.0 / (2 * P->dy);
    c.invdx2 = 1.0 / (P->dx * P->dx);
    c.invdy2 = 1.0 / (P->dy * P->dy);
    c.inv_cp = 1.0 / P->c_p;
    c.inv_Trho = 1.0 / (P->T_inf * P->rho_inf);
    c.inv_mu = 1.0 / P->mu;
    c.inv_Pr = 1.0 / P->Pr;
    c.topo = s->topo;
    c.cut = s->cut;
    c.nzy = s->nzy;

    /* pressure solve tables (src/cu/pressure.cu:356-390) */
    WfSpectral &sp = s->sp;
    memset(&sp, 0, sizeof(sp));
    sp.nx = Nx - 1;
    sp.ny = Ny - 1;
    sp.nz = Nz - 1;
    sp.hx = sp.nx / 2 + 1;
    sp.ldj = (sp.ny + 7) & ~7;
    sp.fx_pairs = wf_pairs_for(sp.nx);
    sp.fy_cols = wf_f2_n1(sp.ny) ? wf_f2_nseq(sp.ny) : WF_FY_COLS;
    sp.ngroups = ((sp.ny + 1) / 2 + sp.fx_pairs - 1) / sp.fx_pairs;
    sp.npmax = sp.ngroups * sp.nz + 1;
#if !WF_MIXED
    sp.pl = wf_pl_takes(sp.nx, sp.ny, sp.nz, &sp.pl_nt) ? 1 : 0;
#endif
    sp.pl_ld = (sp.ny + 15) & ~15;
    sp.pl_groups = (sp.ny + WF_PL_ROWS - 1) / WF_PL_ROWS;
    if (sp.pl) sp.npmax = sp.pl_groups * sp.nz + 1;
    int radx[WF_MAX_RADICES], rady[WF_MAX_RADICES];
    if (wf_factor(sp.nx, radx) < 0 || wf_factor(sp.ny, rady) < 0)
        return wf_fail(WF_E_ARG, "transform length has too many factors");
    if ((rc = wf_upload(&s->radx, radx, WF_MAX_RADICES))) return rc;
    if ((rc = wf_upload(&s->rady, rady, WF_MAX_RADICES))) return rc;
    std::vector<double2> twx(sp.nx), twy(sp.ny);
    for (int e = 0; e < sp.nx; e++) {
        double ang = 2.0 * M_PI * (double)e / (double)sp.nx;
        twx[e] = make_double2(cos(ang), -sin(ang));
    }
    for (int e = 0; e < sp.ny; e++) {
        double ang = 2.0 * M_PI * (double)e / (double)sp.ny;
        twy[e] = make_double2(cos(ang), -sin(ang));
    }
    if ((rc = wf_upload_real2(&s->twx, twx))) return rc;
    if ((rc = wf_upload_real2(&s->twy, twy))) return rc;
    std::vector<double> kx2(sp.hx), ky2(sp.ny);
    for (int r = 0; r < sp.hx; r++) kx2[r] = P->kx[r] * P->kx[r];
    for (int q = 0; q < sp.ny; q++) ky2[q] = P->ky[q] * P->ky[q];
    if ((rc = wf_upload_real(&s->kx2, kx2.data(), sp.hx))) return rc;
    if ((rc = wf_upload_real(&s->ky2, ky2.data(), sp.ny))) return rc;
    /* padded to the longest chunk of k_thomas, whose rows above the top are x = y / u */
    const size_t npad = (sp.nz + 15) & ~15;
    std::vector<double> ta(npad, 0.0), tc(npad, 0.0), beta(npad, 1.0);
    for (int k = 0; k < Nz - 2; k++) {
        double dz_k = z[k + 1] - z[k], dz_kp1 = z[k + 2] - z[k + 1];
        ta[k] = 2 / (dz_k * (dz_k + dz_kp1));
        if (k > 0) {
            double dz_km1 = z[k] - z[k - 1];
            tc[k] = 2 / (dz_k * (dz_km1 + dz_k));
            beta[k] = 2 / (dz_km1 * dz_k);
        }
    }
    beta[Nz - 2] = 2 / ((z[Nz - 2] - z[Nz - 3]) * (z[Nz - 1] - z[Nz - 2])); /* beta_top */
    if ((rc = wf_upload_real(&s->ta, ta.data(), npad))) return rc;
    if ((rc = wf_upload_real(&s->tc, tc.data(), tc.size()))) return rc;
    if ((rc = wf_upload_real(&s->beta, beta.data(), npad))) return rc;
#if WF_MIXED
    if ((rc = wf_upload(&s->kx2d, kx2.data(), sp.hx))) return rc;
    if ((rc = wf_upload(&s->ky2d, ky2.data(), sp.ny))) return rc;
    if ((rc = wf_upload(&s->tad, ta.data(), npad))) return rc;
    if ((rc = wf_upload(&s->tcd, tc.data(), tc.size()))) return rc;
    if ((rc = wf_upload(&s->betad, beta.data(), npad))) return rc;
    /* the systems solved in FP64: kx index < low_kx and ky index within
     * low_ky of 0 or ny (WF_MIXED_LOW_KX / WF_MIXED_LOW_KY override 4, 4) */
    const char *ekx = getenv("WF_MIXED_LOW_KX"), *eky = getenv("WF_MIXED_LOW_KY");
    sp.low_kx = std::max(0, std::min(ekx ? atoi(ekx) : 4, sp.hx));
    sp.low_ky = eky ? atoi(eky) : 4;
#else
    sp.low_kx = 0;
    sp.low_ky = 0;
#endif
    double dz0 = z[1] - z[0], dz1 = z[2] - z[1];
    double dzNm2 = z[Nz - 2] - z[Nz - 3], dzNm1 = z[Nz - 1] - z[Nz - 2];
    sp.dz0 = dz0;
    sp.c0a = (dz0 + dz1) / (dz0 * dz1);
    sp.c0b = 1 / dz1;
    sp.b0 = -1.0 / dz0;
    sp.beta_top = 2 / (dzNm2 * dzNm1);
    sp.top_div = 2 / (dzNm1 * (dzNm2 + dzNm1));
    /* 4 levels per half-wave chunk (k_thomas_h) up to 128 levels, else whole-wave chunks of 8 or 16 */
    sp.thomas_lc = (WF_THOMAS_HALF && sp.nz <= 4 * 2 * WF_THOMAS_MAX_CHUNKS) ? 4
                   : (sp.nz <= 8 * WF_THOMAS_MAX_CHUNKS)                       ? 8
                                                                               : 16;
    if (sp.pl) {
        const int len[2] = {sp.nx, sp.ny};
        std::vector<double> tab;
        size_t at[5] = {0, 0, 0, 0, 0};
#if !WF_MIXED
        for (int q = 0; q < 4; q++) { /* forward and inverse tables in x, then in y */
            std::vector<double> fwd, inv;
            wf_pl_matrix(len[q / 2], fwd, inv);
            const std::vector<double> &t = (q & 1) ? inv : fwd;
            tab.insert(tab.end(), t.begin(), t.end());
            at[q + 1] = tab.size();
        }
#endif
        if ((rc = wf_upload_real(&s->pl_tab, tab.data(), tab.size()))) return rc;
        sp.pl_fx = s->pl_tab + at[0];
        sp.pl_ix = s->pl_tab + at[1];
        sp.pl_fy = s->pl_tab + at[2];
        sp.pl_iy = s->pl_tab + at[3];
        WF_HIP(hipMalloc((void **)&s->U, sizeof(wf_real) * (size_t)sp.nx * sp.nz * sp.pl_ld));
        const size_t piv = (size_t)sp.hx * ((sp.nz + 15) & ~15) * (sp.ny / 2 + 1);
        WF_HIP(hipMalloc((void **)&s->pl_piv, sizeof(wf_real) * 2 * piv));
        sp.U = s->U;
        sp.pl_l = s->pl_piv;
        sp.pl_ru = s->pl_piv + piv;
    } else {
        const long nspec = (long)sp.nz * sp.hx * sp.ldj;
        const int nchunks = (sp.nz + sp.thomas_lc - 1) / sp.thomas_lc;
        WF_HIP(hipMalloc((void **)&s->F, sizeof(wf_real2) * nspec));
        WF_HIP(hipMemset(s->F, 0, sizeof(wf_real2) * nspec));
        WF_HIP(hipMalloc((void **)&s->Ptop, sizeof(wf_real2) * (long)sp.hx * sp.ldj));
        WF_HIP(hipMemset(s->Ptop, 0, sizeof(wf_real2) * (long)sp.hx * sp.ldj));
        WF_HIP(hipMalloc((void **)&s->UB, sizeof(double) * (long)nchunks * sp.hx * sp.ldj));
        WF_HIP(hipMemset(s->UB, 0, sizeof(double) * (long)nchunks * sp.hx * sp.ldj));
    }
    WF_HIP(hipMalloc((void **)&s->pmax, sizeof(double) * 2 * sp.npmax));
    WF_HIP(hipMemset(s->pmax, 0, sizeof(double) * 2 * sp.npmax));
#if WF_MIXED
    /* the FP32 iteration also stops once max|dp| <= rtol max|p|
     * (WF_MIXED_PRESSURE_RTOL overrides the default) */
    const char *ert = getenv("WF_MIXED_PRESSURE_RTOL");
    s->press_rtol = ert ? atof(ert) : WF_MIXED_PRESSURE_RTOL;
#else
    s->press_rtol = 0.0;
#endif
    sp.F = s->F;
    sp.Ptop = s->Ptop;
    sp.A = s->A;
    sp.UB = s->UB;
    sp.pmax = s->pmax;
    sp.kx2 = s->kx2;
    sp.ky2 = s->ky2;
    sp.ta = s->ta;
    sp.tc = s->tc;
    sp.beta = s->beta;
#if WF_MIXED
    sp.kx2d = s->kx2d;
    sp.ky2d = s->ky2d;
    sp.tad = s->tad;
    sp.tcd = s->tcd;
    sp.betad = s->betad;
#else
    sp.kx2d = s->kx2;
    sp.ky2d = s->ky2;
    sp.tad = s->ta;
    sp.tcd = s->tc;
    sp.betad = s->beta;
#endif
    sp.twx = s->twx;
    sp.twy = s->twy;
    sp.radx = s->radx;
    sp.rady = s->rady;
    sp.rho = s->rho;
    sp.ctl = s->ctl;
    sp.hflag = s->hflag_dev;
#if !WF_MIXED
    if (sp.pl) WF_HIP(wf_pl_prepare(sp, s->stream));
#endif
    if (!sp.pl) WF_HIP(wf_launch_pivots(sp, s->UB, s->stream));
    WF_HIP(hipStreamSynchronize(s->stream));
    for (int q = 0; q < 2 * WF_MAX_EVENTS; q++) WF_HIP(hipEventCreate(&s->ev[q]));
    return WF_OK;
}

int create(const Parameters *parameters, Solver **out) {
    if (parameters == NULL || out == NULL) return wf_fail(WF_E_ARG, "null argument");
    Solver *s = (Solver *)calloc(1, sizeof(Solver));
    if (s == NULL) return wf_fail(WF_E_ALLOC, "out of host memory");
    int rc = wf_create_impl(s, parameters);
    if (rc != WF_OK) {
        char keep[512];
        snprintf(keep, sizeof(keep), "%s", wf_error_message());
        destroy(s);
        wf_error_restore(keep);
        *out = NULL;
        return rc;
    }
    *out = s;
    return WF_OK;
}

int destroy(Solver *s) {
    if (s == NULL) return WF_OK;
    if (s->stream) (void)hipStreamSynchronize(s->stream);
    for (int q = 0; q < 4; q++) (void)hipFree(s->state[q]);
    void *bufs[] = {s->zc, s->derived, s->p, s->A, s->UB, s->pmax, s->F, s->Ptop, s->z, s->cd2, s->delta_k,
                    s->cl_prm, s->cl_frag, s->clq_count, s->clq_node, s->clq_x, s->clq_rho, s->topo, s->kx2, s->ky2, s->ta,
                    s->tc, s->beta, s->x, s->y, s->cut, s->nzy, s->radx, s->rady, s->twx, s->twy, s->scratch,
                    s->Tsrc, s->rho, s->ctl, s->kx2d, s->ky2d, s->tad, s->tcd, s->betad,
                    s->in_box, s->rep_part, s->rep_nan, s->U, s->pl_tab, s->pl_piv};
    for (size_t q = 0; q < sizeof(bufs) / sizeof(bufs[0]); q++)
        if (bufs[q]) (void)hipFree(bufs[q]);
    for (int q = 0; q < 2 * WF_MAX_EVENTS; q++)
        if (s->ev[q]) (void)hipEventDestroy(s->ev[q]);
    if (s->ck_stream) (void)hipStreamSynchronize(s->ck_stream);
    if (s->ck_dev) (void)hipFree(s->ck_dev);
    if (s->ck_host) (void)hipHostFree(s->ck_host);
    if (s->ck_conv) (void)hipEventDestroy(s->ck_conv);
    if (s->ck_done) (void)hipEventDestroy(s->ck_done);
    if (s->ck_stream) (void)hipStreamDestroy(s->ck_stream);
    if (s->hflag) (void)hipHostFree(s->hflag);
    if (s->stream) (void)hipStreamDestroy(s->stream);
    free(s);
    return WF_OK;
}

/* ------------------------------------------------------ layout transfers ---- */

/* host reference-layout state vector (FP64) -> device internal-layout buffer */
static int wf_put_state(Solver *s, const double *y_host, char *dst) {
    const Parameters &P = s->P;
    const WfState d = wf_view(s, dst);
    wf_real *f4[4] = {d.u, d.v, d.w, d.T};
    WF_HIP(hipMemcpyAsync(s->scratch, y_host, sizeof(double) * s->S, hipMemcpyHostToDevice, s->stream));
    for (int f = 0; f < 4; f++)
        WF_HIP(wf_launch_to_internal(s->scratch + f * s->N, f4[f], P.Nx, P.Ny, P.Nz, s->stream));
    WF_HIP(wf_launch_to_internal(s->scratch + 4 * s->N, d.Y, P.Nx, P.Ny, P.Nz_Y_max, s->stream));
    return WF_OK;
}

static int wf_get_state_buf(Solver *s, char *src, double *y_host) {
    const Parameters &P = s->P;
    const WfState v = wf_view(s, src);
    const wf_real *f4[4] = {v.u, v.v, v.w, v.T};
    for (int f = 0; f < 4; f++)
        WF_HIP(wf_launch_to_reference(f4[f], s->scratch + f * s->N, P.Nx, P.Ny, P.Nz, s->stream));
    WF_HIP(wf_launch_to_reference((const double *)v.Y, s->scratch + 4 * s->N, P.Nx, P.Ny, P.Nz_Y_max, s->stream));
    WF_HIP(hipMemcpyAsync(y_host, s->scratch, sizeof(double) * s->S, hipMemcpyDeviceToHost, s->stream));
    WF_HIP(hipStreamSynchronize(s->stream));
    return WF_OK;
}

static int wf_put_field(Solver *s, const double *f_host, wf_real *dst) {
    const Parameters &P = s->P;
    WF_HIP(hipMemcpyAsync(s->scratch, f_host, sizeof(double) * s->N, hipMemcpyHostToDevice, s->stream));
    WF_HIP(wf_launch_to_internal(s->scratch, dst, P.Nx, P.Ny, P.Nz, s->stream));
    return WF_OK;
}

static int wf_get_field(Solver *s, const wf_real *src, double *f_host) {
    const Parameters &P = s->P;
    WF_HIP(wf_launch_to_reference(src, s->scratch, P.Nx, P.Ny, P.Nz, s->stream));
    WF_HIP(hipMemcpyAsync(f_host, s->scratch, sizeof(double) * s->N, hipMemcpyDeviceToHost, s->stream));
    WF_HIP(hipStreamSynchronize(s->stream));
    return WF_OK;
}

/* spectrum of the top pressure plane (fixed for the whole run: the solve never
 * writes the unique nodes of k = Nz-1) */
static int wf_top_spectrum(Solver *s) {
    if (s->sp.pl) return WF_OK; /* its right-hand side reads the plane itself */
    WfState none = {nullptr, nullptr, nullptr, nullptr, nullptr};
    WF_HIP(wf_launch_pressure_rhs_fx(s->c, s->sp, none, none, s->p, WF_F_TOP, 0.0, 0.0, -1, 0, s->stream));
    WF_HIP(wf_launch_fy(s->sp, s->Ptop, 0, 0, 1, -1, 0, s->stream));
    return WF_OK;
}

int set_state(Solver *s, const double *y_n, const double *p) {
    if (s == NULL || y_n == NULL || p == NULL) return wf_fail(WF_E_ARG, "null argument");
    int rc;
    if ((rc = wf_put_state(s, y_n, s->state[s->i_yn]))) return rc;
    if ((rc = wf_put_field(s, p, s->p))) return rc;
    if (!s->have_Tsrc) {
        WF_HIP(hipMemcpyAsync(s->Tsrc, wf_view(s, s->state[s->i_yn]).T, sizeof(wf_real) * s->N,
                              hipMemcpyDeviceToDevice, s->stream));
        s->have_Tsrc = 1;
    }
    if ((rc = wf_top_spectrum(s))) return rc;
    WF_HIP(hipStreamSynchronize(s->stream));
    return WF_OK;
}

int get_state(Solver *s, double *y_n, double *p) {
    if (s == NULL) return wf_fail(WF_E_ARG, "null argument");
    int rc;
    if (y_n && (rc = wf_get_state_buf(s, s->state[s->i_yn], y_n))) return rc;
    if (p && (rc = wf_get_field(s, s->p, p))) return rc;
    return WF_OK;
}

/* --------------------------------------------------------------- pieces ---- */

/* Phi of one stage in `mode`: one pass that evaluates the derived fields on
 * the chip (with the learned closure, after the derived pass's mu-only form
 * and the network pass, which leave mu_sgs in memory); with WF_STAGE_FORM=split,
 * the derived pass on X writing every derived field to memory, then the
 * stage pass. */
static int wf_stage(Solver *s, char *X, char *out, int mode, double a) {
    WfState xs = wf_view(s, X), yn = wf_view(s, s->state[s->i_yn]), acc = wf_view(s, s->state[s->i_acc]);
    WfState o = wf_view(s, out);
    WfDerived D = wf_derived_view(s);
    const WfClosure cl{s->cl_prm, s->cl_frag, s->cl_inplace_min};
    unsigned *cnt = s->clq_count + (s->clq_parity ? WF_CLQ_R * WF_CLQ_STRIDE : 0);
    unsigned *nxt = s->clq_count + (s->clq_parity ? 0 : WF_CLQ_R * WF_CLQ_STRIDE);
    const WfClosureQueue cq{cnt, nxt, s->clq_node, s->clq_x, s->clq_rho, s->clq_cap};
    const bool clo = s->closure_on != 0;
    if (!s->stage_split) {
        if (clo) {
            WF_LAUNCH(s, WF_K_DERIVED, wf_launch_derived(s->c, xs, D, &cl, &cq, s->stream, true));
            s->clq_parity ^= 1;
        }
        if (s->stage_shape < 0 && mode == WF_MODE_MID) s->stage_shape = 0; /* not repeatable: acc += 2 k */
        if (s->stage_shape < 0) {
            /* tile-shape tuning at the first stage: each shape's stage tiles
             * three times on this stage's operands (every shape writes the
             * same values, and a stage other than MID writes the same values
             * however often it runs), the fastest kept */
            hipEvent_t e0, e1;
            WF_HIP(hipEventCreate(&e0));
            WF_HIP(hipEventCreate(&e1));
            float best = 1e30f;
            for (int shp = 0; shp < WF_STAGE_SHAPES; shp++) {
                WF_HIP(wf_launch_stage_fd(s->c, xs, D, yn, acc, o, mode, a, shp, clo, s->stream));
                WF_HIP(hipEventRecord(e0, s->stream));
                for (int r = 0; r < 3; r++)
                    WF_HIP(wf_launch_stage_fd_only(s->c, xs, D, yn, acc, o, mode, a, shp, clo, s->stream));
                WF_HIP(hipEventRecord(e1, s->stream));
                WF_HIP(hipEventSynchronize(e1));
                float ms = 0.0f;
                WF_HIP(hipEventElapsedTime(&ms, e0, e1));
                s->stage_ms[shp] = ms / 3.0f;
                if (ms < best) {
                    best = ms;
                    s->stage_shape = shp;
                }
            }
            (void)hipEventDestroy(e0);
            (void)hipEventDestroy(e1);
        }
        WF_LAUNCH(s, WF_K_STAGE, wf_launch_stage_fd(s->c, xs, D, yn, acc, o, mode, a, s->stage_shape, clo, s->stream));
        return WF_OK;
    }
    WF_LAUNCH(s, WF_K_DERIVED, wf_launch_derived(s->c, xs, D, clo ? &cl : nullptr, &cq, s->stream));
    s->clq_parity ^= clo ? 1 : 0;
    WF_LAUNCH(s, WF_K_STAGE, wf_launch_stage(s->c, xs, D, yn, acc, o, mode, a, clo, s->stream));
    return WF_OK;
}

/* RK stages of src/cu/solver.cu:59-93: y_n -> y* in state[i_x1]. */
static int wf_integrate(Solver *s) {
    double dt = s->P.dt;
    char *yn = s->state[s->i_yn], *x0 = s->state[s->i_x0], *x1 = s->state[s->i_x1];
    int rc;
    if (s->method == 2) {
        if ((rc = wf_stage(s, yn, x0, WF_MODE_FIRST, dt * 0.5))) return rc;
        if ((rc = wf_stage(s, x0, x1, WF_MODE_MID, dt * 0.5))) return rc;
        if ((rc = wf_stage(s, x1, x0, WF_MODE_MID, dt))) return rc;
        if ((rc = wf_stage(s, x0, x1, WF_MODE_LAST, dt / 6))) return rc;
    } else if (s->method == 1) {
        if ((rc = wf_stage(s, yn, x0, WF_MODE_FIRST, dt))) return rc;
        if ((rc = wf_stage(s, x0, x1, WF_MODE_LAST, 0.5 * dt))) return rc;
    } else if (s->method == 0) {
        if ((rc = wf_stage(s, yn, x1, WF_MODE_EULER, dt))) return rc;
    } else {
        return wf_fail(WF_E_METHOD, "Time integration method not found.");
    }
    return WF_OK;
}

/* Pressure solve of src/cu/pressure.cu:506-606 for y* = Ys, y_n = Yn.  The
 * solves are queued without host synchronisation; the check of each (done
 * beside the next one's first pass) tests convergence on the device, turns the
 * remaining kernels into no-ops and writes the flag, the solve count and the
 * error to mapped host memory.  The host keeps at most WF_LOOKAHEAD solves
 * queued ahead of the checked ones, stops queueing once the flag is set, takes
 * the results from it and goes on queueing the step behind the no-ops.
 * Three: the one that runs, the next, and one more for the lag of the count
 * (a solve is counted by the first pass of the next).  64x64x32 mixed, one
 * step: 424 us with six ahead, a copy of the results and a wait for the stream
 * behind them; 397 with six and the results in the flag; 378 with three (379
 * with two, which in FP64 starves the device: 845 us against 825). */
#define WF_LOOKAHEAD 3
static int wf_max_iter(const Parameters &P) { return (P.variable_density == 0) ? 1 : P.pressure_solver_iter; }

/* control reset and rho^n of a solve (launches only: capturable) */
static int wf_pressure_begin(Solver *s, const WfState &yn) {
    WF_LAUNCH(s, WF_K_OTHER, wf_launch_iter_reset(s->ctl, s->stream));
    if (wf_max_iter(s->P) > 0 && s->P.variable_density)
        WF_LAUNCH(s, WF_K_OTHER, wf_launch_density(s->c, yn.T, s->rho, s->stream));
    return WF_OK;
}

/* solve m of the iteration (launches only).  Its first pass checks the
 * convergence of solve m - 1 when check is set; the last solve queued (last)
 * is checked by a launch of its own. */
static int wf_pressure_one(Solver *s, const WfState &ys, const WfState &yn, int m, int max_iter, bool check,
                           bool last) {
    const Parameters &P = s->P;
    const long sstride = (long)s->sp.hx * s->sp.ldj;
    const int form = (m > 0) ? WF_F_ITER : (P.variable_density ? WF_F_FIRST : WF_F_CONST);
    const int chk = check ? m - 1 : -1;
#if !WF_MIXED
    if (s->sp.pl) {
        WF_LAUNCH(s, WF_K_PRHS,
                  wf_launch_pl_rhs(s->c, s->sp, ys, yn, s->p, form, P.pressure_solver_tol, s->press_rtol, chk,
                                   max_iter, s->stream));
        WF_LAUNCH(s, WF_K_THOMAS, wf_launch_pl_solve(s->sp, s->stream));
        WF_LAUNCH(s, WF_K_PINV, wf_launch_pl_inv(s->c, s->sp, s->p, s->stream));
    } else
#endif
    {
        WF_LAUNCH(s, WF_K_PRHS,
                  wf_launch_pressure_rhs_fx(s->c, s->sp, ys, yn, s->p, form, P.pressure_solver_tol, s->press_rtol,
                                            chk, max_iter, s->stream));
        WF_LAUNCH(s, WF_K_PFY, wf_launch_fy(s->sp, s->F, sstride, 1, s->sp.nz - 1, -1, 1, s->stream));
        WF_LAUNCH(s, WF_K_THOMAS, wf_launch_thomas(s->sp, s->stream));
        WF_LAUNCH(s, WF_K_PFY, wf_launch_fy(s->sp, s->F, sstride, 0, s->sp.nz, +1, 1, s->stream));
        WF_LAUNCH(s, WF_K_PINV, wf_launch_inverse_fx(s->c, s->sp, s->p, s->stream));
    }
    if (last)
        WF_LAUNCH(s, WF_K_OTHER,
                  wf_launch_iter_check(s->sp, P.pressure_solver_tol, s->press_rtol, m, max_iter, s->stream));
    return WF_OK;
}

/* solves m0, m0+1, ... until the device flags convergence (or max_iter),
 * then the solve's counters */
static int wf_pressure_rest(Solver *s, const WfState &ys, const WfState &yn, int m0) {
    const int max_iter = wf_max_iter(s->P);
    if (max_iter <= 0) {
        s->last_err = 0.0;
        s->last_iters = 0;
        return WF_OK;
    }
    volatile WfHostFlag *hf = s->hflag;
    int rc, m = m0;
    /* the stream's state while the flag is not set */
    const auto drained = [&](bool *empty) -> int {
        for (int spin = 0; spin < 64 && !hf->done; spin++) __builtin_ia32_pause();
        const hipError_t e = hipStreamQuery(s->stream);
        *empty = e == hipSuccess;
        if (e != hipSuccess && e != hipErrorNotReady) return wf_fail(WF_E_DEVICE, "pressure solve: %s", hipGetErrorString(e));
        return WF_OK;
    };
    while (m < max_iter && !(m > 0 && hf->done)) {
        /* the solves before m0 have been checked */
        if ((rc = wf_pressure_one(s, ys, yn, m, max_iter, m > m0, m + 1 >= max_iter))) return rc;
        m++;
        /* wait until the device is within WF_LOOKAHEAD solves; if the stream
         * drains without the count advancing, keep queueing */
        bool empty = false;
        while (m < max_iter && !empty && !hf->done && m - hf->solves >= WF_LOOKAHEAD)
            if ((rc = drained(&empty))) return rc;
    }
    for (bool empty = false; !hf->done;) {
        if (empty) return wf_fail(WF_E_DEVICE, "pressure solve: the iteration ended without its result");
        if ((rc = drained(&empty))) return rc;
    }
    s->press_solves += hf->solves;
    if (s->P.variable_density == 0) {
        s->last_err = 0.0;
        s->last_iters = 0;
    } else {
        s->last_err = hf->err;
        s->last_iters = hf->iters;
    }
    return WF_OK;
}

static int wf_pressure_solve(Solver *s, char *Ys_buf, char *Yn_buf) {
    const WfState ys = wf_view(s, Ys_buf), yn = wf_view(s, Yn_buf);
    memset(s->hflag, 0, sizeof(WfHostFlag));
    int rc = wf_pressure_begin(s, yn);
    if (rc) return rc;
    return wf_pressure_rest(s, ys, yn, 0);
}

static WfSource wf_source(Solver *s, int n) {
    const Parameters &P = s->P;
    WfSource src;
    memset(&src, 0, sizeof(src));
    double t_n = P.t[n];
    if (!(t_n <= P.t_source_end)) return src;
    if (P.t_source_start <= 0) {
        src.mode = s->have_Tsrc ? 1 : 0;
        src.T_src = s->Tsrc;
        return src;
    }
    src.mode = 2;
    src.shape = (strcmp(P.T_source_shape, "gaussian") == 0) ? 1 : (strcmp(P.T_source_shape, "parallelepiped") == 0 ? 2 : 0);
    src.scale = (t_n <= P.t_source_start) ? t_n / P.t_source_start : 1.0;
    src.T_inf = P.T_inf;
    src.T_source = P.T_source;
    src.xc = P.TS_x_center;
    src.yc = P.TS_y_center;
    src.zc = P.TS_z_center;
    src.sx = P.TS_length;
    src.sy = P.TS_width;
    src.sz = P.TS_height;
    src.x0 = P.TS_x_start;
    src.x1 = P.TS_x_end;
    src.y0 = P.TS_y_start;
    src.y1 = P.TS_y_end;
    src.z0 = P.TS_z_start;
    src.z1 = P.TS_z_end;
    src.x = s->x;
    src.y = s->y;
    return src;
}

int step(Solver *s, int step0, int n_steps) {
    if (s == NULL) return wf_fail(WF_E_ARG, "null solver");
    if (s->method < 0) return wf_fail(WF_E_METHOD, "Time integration method not found.");
    if (step0 < 1 || step0 + n_steps - 1 > s->P.Nt)
        return wf_fail(WF_E_ARG, "steps %d..%d outside 1..Nt=%d", step0, step0 + n_steps - 1, s->P.Nt);
    int rc;
    for (int n = step0; n < step0 + n_steps; n++) {
        if ((rc = wf_integrate(s))) return rc;
        char *ys = s->state[s->i_x1], *yn = s->state[s->i_yn], *out = s->state[s->i_x0];
        if ((rc = wf_pressure_solve(s, ys, yn))) return rc;
        WfSource src = wf_source(s, n);
        WF_LAUNCH(s, WF_K_PROJECT,
                  wf_launch_project(s->c, wf_view(s, ys), wf_view(s, yn), s->p, wf_view(s, out), src, s->stream));
        /* y_n <- y_{n+1} by rotating buffer roles */
        int old_yn = s->i_yn;
        s->i_yn = s->i_x0;
        s->i_x0 = old_yn;
        s->steps++;
        if ((rc = wf_prof_collect(s))) return rc;
    }
    WF_HIP(hipStreamSynchronize(s->stream));
    return WF_OK;
}

int phi(Solver *s, const double *R_old, double *R_new) {
    if (s == NULL || R_old == NULL || R_new == NULL) return wf_fail(WF_E_ARG, "null argument");
    int rc;
    char *x0 = s->state[s->i_x0], *x1 = s->state[s->i_x1];
    if ((rc = wf_put_state(s, R_old, x0))) return rc;
    if ((rc = wf_stage(s, x0, x1, WF_MODE_PHI, 0.0))) return rc;
    if ((rc = wf_get_state_buf(s, x1, R_new))) return rc;
    return wf_prof_collect(s);
}

int pressure(Solver *s, const double *y_np1, const double *y_n, double *p, double *error,
                                  int *iterations) {
    if (s == NULL || y_np1 == NULL || y_n == NULL || p == NULL) return wf_fail(WF_E_ARG, "null argument");
    int rc;
    char *x1 = s->state[s->i_x1], *yn = s->state[s->i_yn];
    if ((rc = wf_put_state(s, y_np1, x1))) return rc;
    if ((rc = wf_put_state(s, y_n, yn))) return rc;
    if ((rc = wf_put_field(s, p, s->p))) return rc;
    if ((rc = wf_top_spectrum(s))) return rc;
    if ((rc = wf_pressure_solve(s, x1, yn))) return rc;
    if ((rc = wf_get_field(s, s->p, p))) return rc;
    if (error) *error = s->last_err;
    if (iterations) *iterations = s->last_iters;
    return wf_prof_collect(s);
}

int project(Solver *s, double *y_np1, const double *y_n, const double *p, int n) {
    if (s == NULL || y_np1 == NULL || y_n == NULL || p == NULL) return wf_fail(WF_E_ARG, "null argument");
    if (n < 0 || n > s->P.Nt) return wf_fail(WF_E_ARG, "step %d outside 0..Nt", n);
    int rc;
    char *x1 = s->state[s->i_x1], *yn = s->state[s->i_yn], *x0 = s->state[s->i_x0];
    if ((rc = wf_put_state(s, y_np1, x1))) return rc;
    if ((rc = wf_put_state(s, y_n, yn))) return rc;
    if ((rc = wf_put_field(s, p, s->p))) return rc;
    WfSource src = wf_source(s, n);
    WF_LAUNCH(s, WF_K_PROJECT,
              wf_launch_project(s->c, wf_view(s, x1), wf_view(s, yn), s->p, wf_view(s, x0), src, s->stream));
    if ((rc = wf_get_state_buf(s, x0, y_np1))) return rc;
    return wf_prof_collect(s);
}

int stats(const Solver *s, long *pressure_iterations, long *steps, double *last_error) {
    if (s == NULL) return wf_fail(WF_E_ARG, "null solver");
    if (pressure_iterations) *pressure_iterations = s->press_solves;
    if (steps) *steps = s->steps;
    if (last_error) *last_error = s->last_err;
    return WF_OK;
}

int profile(Solver *s, int enable) {
    if (s == NULL) return wf_fail(WF_E_ARG, "null solver");
    s->profiling = enable ? 1 : 0;
    s->n_ev = 0;
    for (int q = 0; q < WF_K_COUNT; q++) {
        s->k_ms[q] = 0.0;
        s->k_count[q] = 0;
    }
    return WF_OK;
}

int kernel_times(const Solver *s, int kind, double *total_ms, long *launches) {
    if (s == NULL || kind < 0 || kind >= WF_K_COUNT) return wf_fail(WF_E_ARG, "bad argument");
    if (total_ms) *total_ms = s->k_ms[kind];
    if (launches) *launches = s->k_count[kind];
    return WF_OK;
}

/* Asynchronous checkpoint of the current state: its conversion to the
 * reference layout is queued on the compute stream (so later steps cannot
 * overwrite it first), its download on a copy stream into pinned host memory.
 * The caller continues stepping; checkpoint_wait returns the host copy once it
 * has landed.  A checkpoint waits for the previous one's download. */
int checkpoint_begin(Solver *s) {
    if (s == NULL) return wf_fail(WF_E_ARG, "null solver");
    const Parameters &P = s->P;
    const size_t count = (size_t)(s->S + s->N);
    if (s->ck_dev == NULL) {
        WF_HIP(hipMalloc((void **)&s->ck_dev, sizeof(double) * count));
        WF_HIP(hipHostMalloc((void **)&s->ck_host, sizeof(double) * count, hipHostMallocDefault));
        WF_HIP(hipStreamCreate(&s->ck_stream));
        WF_HIP(hipEventCreateWithFlags(&s->ck_conv, hipEventDisableTiming));
        WF_HIP(hipEventCreateWithFlags(&s->ck_done, hipEventDisableTiming));
    }
    if (s->ck_pending) WF_HIP(hipStreamWaitEvent(s->stream, s->ck_done, 0));
    const WfState v = wf_view(s, s->state[s->i_yn]);
    const wf_real *f4[4] = {v.u, v.v, v.w, v.T};
    for (int f = 0; f < 4; f++)
        WF_HIP(wf_launch_to_reference(f4[f], s->ck_dev + f * s->N, P.Nx, P.Ny, P.Nz, s->stream));
    WF_HIP(wf_launch_to_reference((const double *)v.Y, s->ck_dev + 4 * s->N, P.Nx, P.Ny, P.Nz_Y_max, s->stream));
    WF_HIP(wf_launch_to_reference((const wf_real *)s->p, s->ck_dev + s->S, P.Nx, P.Ny, P.Nz, s->stream));
    WF_HIP(hipEventRecord(s->ck_conv, s->stream));
    WF_HIP(hipStreamWaitEvent(s->ck_stream, s->ck_conv, 0));
    WF_HIP(hipMemcpyAsync(s->ck_host, s->ck_dev, sizeof(double) * count, hipMemcpyDeviceToHost, s->ck_stream));
    WF_HIP(hipEventRecord(s->ck_done, s->ck_stream));
    s->ck_pending = 1;
    return WF_OK;
}

int checkpoint_wait(Solver *s, const double **y, const double **p) {
    if (s == NULL || y == NULL || p == NULL) return wf_fail(WF_E_ARG, "null argument");
    if (!s->ck_pending) return wf_fail(WF_E_ARG, "no checkpoint was started");
    WF_HIP(hipEventSynchronize(s->ck_done));
    *y = s->ck_host;
    *p = s->ck_host + s->S;
    return WF_OK;
}

/* Report values from the reduced partials r[WF_REP_N] (maxima of |u|, |v|,
 * |w|; T range; Y range; sums of the kinetic energy, burned columns, fuel
 * columns, learned nodes) and the first-NaN slot. */
static void wf_reports_finish(const Parameters &P, const double *r, unsigned long long first, double *out,
                              long *nan_index) {
    out[WF_REPORT_CFL] = P.dt * (r[0] / P.dx + r[1] / P.dy + r[2] / P.dz);
    out[WF_REPORT_T_MIN] = r[3];
    out[WF_REPORT_T_MAX] = r[4];
    out[WF_REPORT_Y_MIN] = r[5];
    out[WF_REPORT_Y_MAX] = r[6];
    out[WF_REPORT_KINETIC_ENERGY] = r[7] / ((double)(P.Nx - 1) * (P.Ny - 1) * (P.Nz - 2));
    out[WF_REPORT_BURNED] = (r[9] > 0.0) ? r[8] / r[9] : 0.0;
    out[WF_REPORT_LEARNED] = r[10] / ((double)(P.Nx - 1) * (P.Ny - 1) * (P.Nz - 2));
    *nan_index = (first == ~0ull) ? -1 : (long)first;
}

static int wf_reports_blocks(const Solver *s) {
    return (int)((s->N + 255) / 256 < WF_REP_BLOCKS ? (s->N + 255) / 256 : WF_REP_BLOCKS);
}

/* Checkpoint reports of the current state (src/cu/functions.cu:82-185) from
 * one device reduction: the host reduces the per-workgroup partials. */
int reports(Solver *s, double *out, long *nan_index) {
    if (s == NULL || out == NULL || nan_index == NULL) return wf_fail(WF_E_ARG, "null argument");
    const WfState x = wf_view(s, s->state[s->i_yn]);
    const int nb = wf_reports_blocks(s);
    WF_HIP(hipMemsetAsync(s->rep_nan, 0xff, sizeof(unsigned long long), s->stream));
    WF_HIP(wf_launch_reports(s->c, x, s->derived, s->in_box, s->rep_part, nb, s->rep_nan, s->stream));
    std::vector<double> part((size_t)nb * WF_REP_N);
    unsigned long long first = 0;
    WF_HIP(hipMemcpyAsync(part.data(), s->rep_part, sizeof(double) * part.size(), hipMemcpyDeviceToHost, s->stream));
    WF_HIP(hipMemcpyAsync(&first, s->rep_nan, sizeof(first), hipMemcpyDeviceToHost, s->stream));
    WF_HIP(hipStreamSynchronize(s->stream));
    /* the reference's initial values (src/cu/functions.cu:86-88) */
    double r[WF_REP_N] = {0.0, 0.0, 0.0, 1e9, -1e9, 0.0, -1e9, 0.0, 0.0, 0.0, 0.0};
    for (int b = 0; b < nb; b++) {
        const double *v = &part[(size_t)b * WF_REP_N];
        for (int f = 0; f < WF_REP_N; f++) {
            if (f <= 2 || f == 4 || f == 6)
                r[f] = (v[f] > r[f]) ? v[f] : r[f];
            else if (f == 3 || f == 5)
                r[f] = (v[f] < r[f]) ? v[f] : r[f];
            else
                r[f] += v[f];
        }
    }
    wf_reports_finish(s->P, r, first, out, nan_index);
    return WF_OK;
}

/* The same reports with no allocation: the partials, their reduction and the
 * first-NaN slot live in the library's static device scratch (wf_noalloc.hip),
 * reduced on the device in the host reduction's order, so the values equal
 * those of reports() bit for bit. */
int reports_noalloc(Solver *s, double *out, long *nan_index) {
    if (s == NULL || out == NULL || nan_index == NULL) return wf_fail(WF_E_ARG, "null argument");
    const int nb = wf_reports_blocks(s);
    if (nb > WF_REP_BLOCKS) return wf_fail(WF_E_ARG, "reports: %d partial rows exceed the scratch's %d", nb, WF_REP_BLOCKS);
    double *base = nullptr;
    WF_HIP(wf_noalloc_scratch(s->device, &base));
    unsigned long long *nanp = (unsigned long long *)(base + WF_NA_NAN);
    const WfState x = wf_view(s, s->state[s->i_yn]);
    WF_HIP(wf_launch_fill_u64(nanp, ~0ull, s->stream));
    WF_HIP(wf_launch_reports(s->c, x, s->derived, s->in_box, base, nb, nanp, s->stream));
    WF_HIP(wf_launch_reports_final(base, nb, base + WF_NA_FINAL, s->stream));
    double r[WF_REP_N];
    unsigned long long first = 0;
    WF_HIP(hipMemcpyAsync(r, base + WF_NA_FINAL, sizeof(r), hipMemcpyDeviceToHost, s->stream));
    WF_HIP(hipMemcpyAsync(&first, nanp, sizeof(first), hipMemcpyDeviceToHost, s->stream));
    WF_HIP(hipStreamSynchronize(s->stream));
    wf_reports_finish(s->P, r, first, out, nan_index);
    return WF_OK;
}

/* last pressure-iteration count and error, for the step-loop driver */
int last_pressure(const Solver *s, double *error, int *iterations) {
    if (s == NULL) return wf_fail(WF_E_ARG, "null solver");
    if (error) *error = s->last_err;
    if (iterations) *iterations = s->last_iters;
    return WF_OK;
}

/* ------------------------------------------------------- learned closure ---- */

int set_closure(Solver *s, const float *params, long n) {
    if (s == NULL) return wf_fail(WF_E_ARG, "null solver");
    WF_HIP(hipStreamSynchronize(s->stream));
    void *old[] = {s->cl_prm, s->cl_frag, s->clq_count, s->clq_node, s->clq_x, s->clq_rho};
    for (size_t q = 0; q < sizeof(old) / sizeof(old[0]); q++)
        if (old[q]) WF_HIP(hipFree(old[q]));
    s->cl_prm = NULL;
    s->cl_frag = NULL;
    s->clq_count = s->clq_node = NULL;
    s->clq_x = NULL;
    s->clq_rho = NULL;
    s->closure_on = 0;
    if (params == NULL) return WF_OK;
    int rc = wf_closure_upload(params, n, &s->cl_prm, (void **)&s->cl_frag);
    if (rc) return rc;
    /* the queue: WF_CLQ_R regions, each 64 entries per derived-pass
     * wavefront it serves */
    const size_t waves = (size_t)wf_tile_count(s->c) * WF_TILE_Y;
    s->clq_cap = (unsigned)((waves + WF_CLQ_R - 1) / WF_CLQ_R * 64);
    const size_t E = (size_t)WF_CLQ_R * s->clq_cap;
    if (hipMalloc((void **)&s->clq_count, 2 * WF_CLQ_R * WF_CLQ_STRIDE * sizeof(unsigned)) != hipSuccess ||
        hipMemsetAsync(s->clq_count, 0, 2 * WF_CLQ_R * WF_CLQ_STRIDE * sizeof(unsigned), s->stream) != hipSuccess ||
        hipMalloc((void **)&s->clq_node, E * sizeof(unsigned)) != hipSuccess ||
        hipMalloc((void **)&s->clq_x, 2 * E * sizeof(wf_bf16x8)) != hipSuccess ||
        hipMalloc((void **)&s->clq_rho, E * sizeof(wf_real)) != hipSuccess) {
        (void)hipGetLastError();
        rc = wf_fail(WF_E_DEVICE, "closure: out of device memory for the %zu-entry queue", E);
        (void)set_closure(s, NULL, 0);
        return rc;
    }
    s->clq_parity = 0;
    s->closure_on = 1;
    return WF_OK;
}


/* ------------------------------------------------------------- ensembles ---- */

/* the control blocks of n solvers gathered into one array (one download) */
__global__ void k_ctl_gather(WfIterCtl *const *src, WfIterCtl *dst, int n) {
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m < n) dst[m] = *src[m];
}

/* One RK stage of a step: input and output buffer roles (0 y_n, 1 x0, 2 x1),
 * the combination written, and the step's coefficient (the expressions of
 * wf_integrate, so the members' arithmetic equals their solo runs'). */
struct WfStageDef {
    int x, out, mode;
};
static int wf_stage_defs(int method, WfStageDef d[4]) {
    if (method == 2) {
        d[0] = {0, 1, WF_MODE_FIRST};
        d[1] = {1, 2, WF_MODE_MID};
        d[2] = {2, 1, WF_MODE_MID};
        d[3] = {1, 2, WF_MODE_LAST};
        return 4;
    }
    if (method == 1) {
        d[0] = {0, 1, WF_MODE_FIRST};
        d[1] = {1, 2, WF_MODE_LAST};
        return 2;
    }
    d[0] = {0, 2, WF_MODE_EULER};
    return 1;
}
static double wf_stage_coef(int method, int st, double dt) {
    if (method == 2) return (st == 0 || st == 1) ? dt * 0.5 : (st == 2) ? dt : dt / 6;
    if (method == 1) return (st == 0) ? dt : 0.5 * dt;
    return dt;
}

/* Members advance in lockstep, each with its own buffers, tables and pressure
 * control, on one shared stream.  A step is: the RK stages of all members in
 * one launch per pass (wf_launch_stage_batch: u_tau, the stage with the
 * derived fields on the chip, column completion); the first `budget` solves of
 * each member's pressure iteration (the device stops a converged member's
 * kernels); these two parts are one captured graph per buffer parity.  Then,
 * for a member whose iteration has not converged within the budget, its
 * further solves as in its solo run, and each member's projection. */
/* streams the members' pressure solves are spread over (the hardware
 * queues a process gets by default) */
#define WF_ENS_SIDE 4
struct Ensemble {
    int n, nst, method, budget, use_graph;
    Solver **m;
    hipStream_t stream;
    hipStream_t *own;      /* the members' own streams, restored at destroy */
    WfBatchStage *bs;      /* [2 parities][nst][n] */
    int *first;            /* [WF_BATCH_PASSES][n + 1] */
    int items[WF_BATCH_PASSES];
    WfIterCtl **ctl_ptr;   /* the members' control blocks */
    WfIterCtl *ctl_all;    /* gathered at the end of the graph */
    WfIterCtl *ctl_host;
    WfBatchShape shape;
    int tuned;
    double tune_ms[3];     /* chosen u_tau, stage, column pass times (ms, one stage) */
    hipGraphExec_t exec[2];
    int parity;
    /* the members' pressure solves in the graph run on nside streams forked
     * from and joined back into `stream` (member i on side[i % nside]) */
    int nside;
    hipStream_t side[WF_ENS_SIDE];
    hipEvent_t fork, join[WF_ENS_SIDE];
    /* size classes of the pressure solves: class q holds the members
     * cls_mem[cls_first[q] .. cls_first[q + 1]), whose operands press[par]
     * lists in that order (device, [2 parities][n]); a class of two or more
     * members runs each pressure pass as one launch (batch_press) */
    int ncls, batch_press;
    int *cls_first, *cls_mem;
    WfPressItem *press;
};

static int ens_free(Ensemble *e) {
    if (e == NULL) return WF_OK;
    if (e->stream) (void)hipStreamSynchronize(e->stream);
    for (int q = 0; q < 2; q++)
        if (e->exec[q]) (void)hipGraphExecDestroy(e->exec[q]);
    if (e->m) {
        for (int i = 0; i < e->n; i++) {
            if (e->m[i] == NULL) continue;
            if (e->own) e->m[i]->stream = e->own[i];
            destroy(e->m[i]);
        }
    }
    free(e->cls_first);
    free(e->cls_mem);
    void *bufs[] = {e->bs, e->first, e->ctl_ptr, e->ctl_all, e->press};
    for (size_t q = 0; q < sizeof(bufs) / sizeof(bufs[0]); q++)
        if (bufs[q]) (void)hipFree(bufs[q]);
    if (e->ctl_host) (void)hipHostFree(e->ctl_host);
    for (int k = 0; k < WF_ENS_SIDE; k++) {
        if (e->side[k]) (void)hipStreamDestroy(e->side[k]);
        if (e->join[k]) (void)hipEventDestroy(e->join[k]);
    }
    if (e->fork) (void)hipEventDestroy(e->fork);
    if (e->stream) (void)hipStreamDestroy(e->stream);
    free(e->m);
    free(e->own);
    free(e);
    return WF_OK;
}

int ens_destroy(Ensemble *e) { return ens_free(e); }

/* Members a and b launch identical pressure grids and take their solves under
 * the same rule: same grid, density form and iteration limit. */
static bool ens_same_class(const Solver *a, const Solver *b) {
    const WfSpectral &x = a->sp, &y = b->sp;
    return a->c.Nx == b->c.Nx && a->c.Ny == b->c.Ny && a->c.Nz == b->c.Nz && a->c.N == b->c.N &&
           a->P.variable_density == b->P.variable_density && wf_max_iter(a->P) == wf_max_iter(b->P) &&
           x.nx == y.nx && x.ny == y.ny && x.nz == y.nz && x.hx == y.hx && x.ldj == y.ldj &&
           x.fx_pairs == y.fx_pairs && x.fy_cols == y.fy_cols && x.ngroups == y.ngroups && x.npmax == y.npmax &&
           x.thomas_lc == y.thomas_lc && x.pl == y.pl && x.pl_nt == y.pl_nt;
}

/* Size classes (in order of first appearance) and the pressure operand
 * tables of both parities. */
static int ens_classes(Ensemble *e) {
    const int n = e->n;
    e->cls_first = (int *)calloc((size_t)n + 1, sizeof(int));
    e->cls_mem = (int *)calloc((size_t)n, sizeof(int));
    if (e->cls_first == NULL || e->cls_mem == NULL) return wf_fail(WF_E_ALLOC, "out of host memory");
    std::vector<int> cls(n, -1);
    int ncls = 0, at = 0;
    for (int i = 0; i < n; i++) {
        if (cls[i] >= 0) continue;
        e->cls_first[ncls] = at;
        /* a class is the z extent of its launches: at most 65535 members */
        for (int j = i; j < n; j++)
            if (cls[j] < 0 && at - e->cls_first[ncls] < 65535 && ens_same_class(e->m[i], e->m[j])) {
                cls[j] = ncls;
                e->cls_mem[at++] = j;
            }
        ncls++;
    }
    e->cls_first[ncls] = at;
    e->ncls = ncls;
    const char *bp = getenv("WF_ENS_BATCH_PRESSURE");
    e->batch_press = (bp != NULL) ? (atoi(bp) != 0) : 1;
    std::vector<WfPressItem> tab((size_t)2 * n);
    for (int par = 0; par < 2; par++)
        for (int a = 0; a < n; a++) {
            Solver *s = e->m[e->cls_mem[a]];
            WfPressItem &it = tab[(size_t)par * n + a];
            memset(&it, 0, sizeof(it));
            it.c = s->c;
            it.sp = s->sp;
            it.ys = wf_view(s, s->state[2]);
            it.yn = wf_view(s, s->state[par ? 1 : 0]);
            it.p = s->p;
            it.rho = s->rho;
            it.tol = s->P.pressure_solver_tol;
            it.rtol = s->press_rtol;
            it.max_iter = wf_max_iter(s->P);
        }
    WF_HIP(hipMalloc((void **)&e->press, sizeof(WfPressItem) * tab.size()));
    WF_HIP(hipMemcpy(e->press, tab.data(), sizeof(WfPressItem) * tab.size(), hipMemcpyHostToDevice));
    return WF_OK;
}

static int ens_create_impl(Ensemble *e, const Parameters *const *P, int n, int budget, int use_graph) {
    int rc;
    e->n = n;
    e->budget = budget;
    e->use_graph = use_graph;
    e->m = (Solver **)calloc((size_t)n, sizeof(Solver *));
    e->own = (hipStream_t *)calloc((size_t)n, sizeof(hipStream_t));
    if (e->m == NULL || e->own == NULL) return wf_fail(WF_E_ALLOC, "out of host memory");
    for (int i = 0; i < n; i++) {
        if (P[i] == NULL) return wf_fail(WF_E_ARG, "ensemble member %d has no parameters", i);
        if ((rc = create(P[i], &e->m[i]))) return rc;
        if (e->m[i]->method < 0) return wf_fail(WF_E_METHOD, "Time integration method not found.");
        if (i > 0 && e->m[i]->method != e->m[0]->method)
            return wf_fail(WF_E_ARG, "ensemble members must share one time-integration method");
    }
    e->method = e->m[0]->method;
    WfStageDef def[4];
    e->nst = wf_stage_defs(e->method, def);
    WF_HIP(hipStreamCreate(&e->stream));
    for (int i = 0; i < n; i++) {
        e->own[i] = e->m[i]->stream;
        e->m[i]->stream = e->stream;
    }
    {
        const char *ns = getenv("WF_ENS_STREAMS");
        e->nside = (ns != NULL) ? atoi(ns) : WF_ENS_SIDE;
        e->nside = (e->nside < 1) ? 1 : (e->nside > WF_ENS_SIDE) ? WF_ENS_SIDE : e->nside;
        if (e->nside > n) e->nside = n;
    }
    if (e->nside > 1) {
        WF_HIP(hipEventCreateWithFlags(&e->fork, hipEventDisableTiming));
        for (int k = 0; k < e->nside; k++) {
            WF_HIP(hipStreamCreate(&e->side[k]));
            WF_HIP(hipEventCreateWithFlags(&e->join[k], hipEventDisableTiming));
        }
    }
    /* per parity, stage and member: the batched stage operands */
    std::vector<WfBatchStage> bs((size_t)2 * e->nst * n);
    for (int par = 0; par < 2; par++)
        for (int st = 0; st < e->nst; st++)
            for (int i = 0; i < n; i++) {
                Solver *s = e->m[i];
                /* buffer roles of parity par: y_n, x0, x1, acc */
                char *role[3] = {s->state[par ? 1 : 0], s->state[par ? 0 : 1], s->state[2]};
                WfBatchStage &b = bs[((size_t)par * e->nst + st) * n + i];
                memset(&b, 0, sizeof(b));
                b.c = s->c;
                b.X = wf_view(s, role[def[st].x]);
                b.out = wf_view(s, role[def[st].out]);
                b.Yn = wf_view(s, role[0]);
                b.acc = wf_view(s, s->state[3]);
                b.D = wf_derived_view(s);
                b.mode = def[st].mode;
                b.a = wf_stage_coef(e->method, st, s->P.dt);
            }
    WF_HIP(hipMalloc((void **)&e->bs, sizeof(WfBatchStage) * bs.size()));
    WF_HIP(hipMemcpy(e->bs, bs.data(), sizeof(WfBatchStage) * bs.size(), hipMemcpyHostToDevice));
    std::vector<int> first((size_t)WF_BATCH_PASSES * (n + 1), 0);
    for (int i = 0; i < n; i++) {
        int it[WF_BATCH_PASSES];
        wf_batch_items(e->m[i]->c, it);
        for (int q = 0; q < WF_BATCH_PASSES; q++) {
            const long next = (long)first[(size_t)q * (n + 1) + i] + it[q];
            if (next > (1L << 30)) return wf_fail(WF_E_ARG, "ensemble too large: %ld work items in one pass", next);
            first[(size_t)q * (n + 1) + i + 1] = (int)next;
        }
    }
    for (int q = 0; q < WF_BATCH_PASSES; q++) e->items[q] = first[(size_t)q * (n + 1) + n];
    WF_HIP(hipMalloc((void **)&e->first, sizeof(int) * first.size()));
    WF_HIP(hipMemcpy(e->first, first.data(), sizeof(int) * first.size(), hipMemcpyHostToDevice));
    std::vector<WfIterCtl *> cp(n);
    for (int i = 0; i < n; i++) cp[i] = e->m[i]->ctl;
    WF_HIP(hipMalloc((void **)&e->ctl_ptr, sizeof(WfIterCtl *) * n));
    WF_HIP(hipMemcpy(e->ctl_ptr, cp.data(), sizeof(WfIterCtl *) * n, hipMemcpyHostToDevice));
    WF_HIP(hipMalloc((void **)&e->ctl_all, sizeof(WfIterCtl) * n));
    WF_HIP(hipHostMalloc((void **)&e->ctl_host, sizeof(WfIterCtl) * n, hipHostMallocDefault));
    /* untuned default: the solo launches' shapes (32 x 8 tiles, one workgroup
     * per item), compiled for the exchange term and Sutherland laws when a
     * member uses them */
    e->shape.shape = 0;
    e->shape.general = 0;
    for (int i = 0; i < n; i++) {
        const WfConst &c = e->m[i]->c;
        if (c.exchange_on || c.suth_mu == 1 || c.suth_k == 1) e->shape.general = 1;
    }
    e->shape.grid[0] = e->items[0];
    e->shape.grid[1] = -e->items[1];
    e->shape.grid[2] = e->items[WF_BATCH_SHAPES + 1];
    return ens_classes(e);
}

int ens_create(const Parameters *const *P, int n, int budget, int use_graph, Ensemble **out) {
    if (P == NULL || out == NULL || n < 1) return wf_fail(WF_E_ARG, "bad ensemble arguments");
    if (budget < 1) return wf_fail(WF_E_ARG, "pressure-solve budget must be at least 1 (got %d)", budget);
    Ensemble *e = (Ensemble *)calloc(1, sizeof(Ensemble));
    if (e == NULL) return wf_fail(WF_E_ALLOC, "out of host memory");
    int rc = ens_create_impl(e, P, n, budget, use_graph);
    if (rc != WF_OK) {
        char keep[512];
        snprintf(keep, sizeof(keep), "%s", wf_error_message());
        ens_free(e);
        wf_error_restore(keep);
        *out = NULL;
        return rc;
    }
    *out = e;
    return WF_OK;
}

static int ens_member(Ensemble *e, int i, Solver **s) {
    if (e == NULL) return wf_fail(WF_E_ARG, "null ensemble");
    if (i < 0 || i >= e->n) return wf_fail(WF_E_ARG, "member %d outside 0..%d", i, e->n - 1);
    *s = e->m[i];
    return WF_OK;
}

int ens_set_state(Ensemble *e, int i, const double *y_n, const double *p) {
    Solver *s;
    int rc = ens_member(e, i, &s);
    if (rc) return rc;
    /* the members' roles rotate in lockstep: parity 1 has y_n in buffer 1 */
    if (s->i_yn != (e->parity ? 1 : 0)) return wf_fail(WF_E_ARG, "member %d out of step with the ensemble", i);
    return set_state(s, y_n, p);
}

int ens_get_state(Ensemble *e, int i, double *y_n, double *p) {
    Solver *s;
    int rc = ens_member(e, i, &s);
    if (rc) return rc;
    return get_state(s, y_n, p);
}

int ens_stats(Ensemble *e, int i, long *pressure_solves, long *steps) {
    Solver *s;
    int rc = ens_member(e, i, &s);
    if (rc) return rc;
    return stats(s, pressure_solves, steps, NULL);
}

/* The captured pressure solves of size class q on stream st: the launches of
 * wf_pressure_begin and of the first `budget` wf_pressure_one calls, each as
 * one launch for all the class's members. */
static int ens_pressure_class(Ensemble *e, int par, int q, hipStream_t st) {
    const int a0 = e->cls_first[q], nm = e->cls_first[q + 1] - a0;
    const Solver *s0 = e->m[e->cls_mem[a0]];
    const WfSpectral &sp = s0->sp;
    const WfPressItem *tab = e->press + (size_t)par * e->n + a0;
    const int max_iter = wf_max_iter(s0->P);
    WF_HIP(wf_launch_iter_reset_batch(tab, nm, st));
    if (max_iter > 0 && s0->P.variable_density) WF_HIP(wf_launch_density_batch(s0->c, tab, nm, st));
    const long sstride = (long)sp.hx * sp.ldj;
    for (int m = 0; m < e->budget && m < max_iter; m++) {
        const int form = (m > 0) ? WF_F_ITER : (s0->P.variable_density ? WF_F_FIRST : WF_F_CONST);
#if !WF_MIXED
        if (sp.pl) {
            WF_HIP(wf_launch_pl_rhs_batch(sp, tab, nm, form, m - 1, st));
            WF_HIP(wf_launch_pl_solve_batch(sp, tab, nm, st));
            WF_HIP(wf_launch_pl_inv_batch(sp, tab, nm, st));
        } else
#endif
        {
            WF_HIP(wf_launch_pressure_rhs_fx_batch(sp, tab, nm, form, m - 1, st));
            WF_HIP(wf_launch_fy_batch(sp, tab, nm, sstride, 1, sp.nz - 1, -1, 1, st));
            WF_HIP(wf_launch_thomas_batch(sp, tab, nm, st));
            WF_HIP(wf_launch_fy_batch(sp, tab, nm, sstride, 0, sp.nz, +1, 1, st));
            WF_HIP(wf_launch_inverse_fx_batch(sp, tab, nm, st));
        }
        if (m + 1 >= e->budget || m + 1 >= max_iter) WF_HIP(wf_launch_iter_check_batch(tab, nm, m, st));
    }
    return WF_OK;
}

/* the captured part of a step of parity par: RK stages, then the first
 * `budget` solves of every member (per size class) */
static int ens_enqueue(Ensemble *e, int par) {
    for (int st = 0; st < e->nst; st++)
        WF_HIP(wf_launch_stage_batch(e->bs + (size_t)(par * e->nst + st) * e->n, e->first, e->n, e->shape, e->stream));
    const int K = e->nside;
    if (K > 1) {
        WF_HIP(hipEventRecord(e->fork, e->stream));
        for (int k = 0; k < K; k++) WF_HIP(hipStreamWaitEvent(e->side[k], e->fork, 0));
    }
    int rc = WF_OK, unit = 0;
    for (int q = 0; q < e->ncls && rc == WF_OK; q++) {
        const int a0 = e->cls_first[q], nm = e->cls_first[q + 1] - a0;
        if (nm >= 2 && e->batch_press) {
            rc = ens_pressure_class(e, par, q, (K > 1) ? e->side[unit++ % K] : e->stream);
            continue;
        }
        for (int a = a0; a < a0 + nm && rc == WF_OK; a++) {
            Solver *s = e->m[e->cls_mem[a]];
            s->stream = (K > 1) ? e->side[unit++ % K] : e->stream;
            const WfState ys = wf_view(s, s->state[2]), yn = wf_view(s, s->state[par ? 1 : 0]);
            if ((rc = wf_pressure_begin(s, yn))) break;
            const int max_iter = wf_max_iter(s->P);
            for (int m = 0; m < e->budget && m < max_iter; m++)
                if ((rc = wf_pressure_one(s, ys, yn, m, max_iter, m > 0, m + 1 >= e->budget || m + 1 >= max_iter)))
                    break;
        }
    }
    for (int i = 0; i < e->n; i++) e->m[i]->stream = e->stream;
    if (K > 1) {
        /* joined also after a failed launch, so that a capture can end */
        for (int k = 0; k < K; k++) {
            WF_HIP(hipEventRecord(e->join[k], e->side[k]));
            WF_HIP(hipStreamWaitEvent(e->stream, e->join[k], 0));
        }
    }
    if (rc) return rc;
    hipLaunchKernelGGL(k_ctl_gather, dim3((e->n + 63) / 64), dim3(64), 0, e->stream, e->ctl_ptr, e->ctl_all, e->n);
    WF_HIP(hipGetLastError());
    WF_HIP(hipMemcpyAsync(e->ctl_host, e->ctl_all, sizeof(WfIterCtl) * e->n, hipMemcpyDeviceToHost, e->stream));
    return WF_OK;
}

/* Launch-shape autotuner: each batched pass of the first stage (y_n -> x0,
 * which leaves y_n intact) timed for every candidate (stage tile shape and
 * grid), three launches each, on the members' current states; the fastest
 * candidate of each pass is kept.  Every candidate evaluates each node with
 * the same arithmetic, so the choice does not change the results. */
/* In the stage pass, a candidate replaces the one kept so far only when it
 * is faster by more than 2 %: the first candidate is the default shape (32x8
 * tiles, one workgroup per tile), the shapes' times at the first stage often
 * lie within the timing noise of one another, and there the default has
 * measured the faster step. */
#define WF_TUNE_MARGIN 0.98
static int ens_tune(Ensemble *e) {
    hipEvent_t a, b;
    WF_HIP(hipEventCreate(&a));
    WF_HIP(hipEventCreate(&b));
    const WfBatchStage *B = e->bs + (size_t)(e->parity * e->nst) * e->n;
    auto time3 = [&](auto launch, double *ms) -> int {
        WF_HIP(launch());
        WF_HIP(hipEventRecord(a, e->stream));
        for (int r = 0; r < 3; r++) WF_HIP(launch());
        WF_HIP(hipEventRecord(b, e->stream));
        WF_HIP(hipEventSynchronize(b));
        float t = 0.0f;
        WF_HIP(hipEventElapsedTime(&t, a, b));
        *ms = (double)t / 3.0;
        return WF_OK;
    };
    int rc;
    WfBatchShape sh = e->shape, best = e->shape;
    double best_ms = 1e30, ms;
    /* u_tau pass: one workgroup per item or a fixed grid of 1024 */
    const int ucand[2] = {e->items[0], 1024};
    for (int g = 0; g < 2; g++) {
        if (g > 0 && ucand[g] >= e->items[0]) continue;
        sh.grid[0] = ucand[g];
        if ((rc = time3([&] { return wf_launch_utau_batch(B, e->first, e->n, sh, e->stream); }, &ms))) return rc;
        if (ms < best_ms) {
            best_ms = ms;
            best.grid[0] = ucand[g];
        }
    }
    e->tune_ms[0] = best_ms;
    sh = best;
    WF_HIP(wf_launch_utau_batch(B, e->first, e->n, sh, e->stream));
    /* stage pass: tile shape x (one workgroup per tile, or a fixed grid of
     * 2048 / 1024 looping over the tiles) */
    best_ms = 1e30;
    for (int d = 0; d < WF_BATCH_SHAPES; d++) {
        const int ns = e->items[1 + d];
        const int scand[3] = {-ns, 2048, 1024};
        for (int g = 0; g < 3; g++) {
            if (g > 0 && scand[g] >= ns) continue;
            sh.shape = d;
            sh.grid[1] = scand[g];
            if ((rc = time3([&] { return wf_launch_stage_only_batch(B, e->first, e->n, sh, e->stream); }, &ms)))
                return rc;
            if (ms < best_ms * WF_TUNE_MARGIN) {
                best_ms = ms;
                best.shape = d;
                best.grid[1] = scand[g];
            }
        }
    }
    e->tune_ms[1] = best_ms;
    sh = best;
    /* column pass */
    const int nc = e->items[WF_BATCH_SHAPES + 1];
    const int ccand[2] = {nc, 1024};
    best_ms = 1e30;
    for (int g = 0; g < 2; g++) {
        if (g > 0 && ccand[g] >= nc) continue;
        sh.grid[2] = ccand[g];
        if ((rc = time3([&] { return wf_launch_columns_batch(B, e->first, e->n, sh, e->stream); }, &ms))) return rc;
        if (ms < best_ms) {
            best_ms = ms;
            best.grid[2] = ccand[g];
        }
    }
    e->tune_ms[2] = best_ms;
    e->shape = best;
    e->tuned = 1;
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    return WF_OK;
}

int ens_tuning(const Ensemble *e, int *shape, int *grid, double *ms) {
    if (e == NULL) return wf_fail(WF_E_ARG, "null ensemble");
    if (shape) *shape = e->shape.shape;
    for (int q = 0; q < 3; q++) {
        if (grid) grid[q] = e->shape.grid[q];
        if (ms) ms[q] = e->tune_ms[q];
    }
    return WF_OK;
}

int ens_step(Ensemble *e, int step0, int n_steps) {
    if (e == NULL) return wf_fail(WF_E_ARG, "null ensemble");
    for (int i = 0; i < e->n; i++)
        if (step0 < 1 || step0 + n_steps - 1 > e->m[i]->P.Nt)
            return wf_fail(WF_E_ARG, "member %d: steps %d..%d outside 1..Nt=%d", i, step0, step0 + n_steps - 1,
                           e->m[i]->P.Nt);
    int rc;
    if (!e->tuned && (rc = ens_tune(e))) return rc;
    for (int n = step0; n < step0 + n_steps; n++) {
        const int par = e->parity;
        for (int i = 0; i < e->n; i++) {
            memset(e->m[i]->hflag, 0, sizeof(WfHostFlag));
        }
        if (e->use_graph) {
            if (!e->exec[par]) {
                hipGraph_t g;
                WF_HIP(hipStreamBeginCapture(e->stream, hipStreamCaptureModeThreadLocal));
                rc = ens_enqueue(e, par);
                hipGraph_t gdone = NULL;
                const hipError_t ce = hipStreamEndCapture(e->stream, &gdone);
                if (rc) return rc;
                if (ce != hipSuccess) return wf_fail(WF_E_DEVICE, "step capture: %s", hipGetErrorString(ce));
                g = gdone;
                const hipError_t ie = hipGraphInstantiate(&e->exec[par], g, NULL, NULL, 0);
                (void)hipGraphDestroy(g);
                if (ie != hipSuccess) return wf_fail(WF_E_DEVICE, "step graph: %s", hipGetErrorString(ie));
            }
            WF_HIP(hipGraphLaunch(e->exec[par], e->stream));
        } else if ((rc = ens_enqueue(e, par))) {
            return rc;
        }
        WF_HIP(hipStreamSynchronize(e->stream));
        /* the rest of the step per member (further solves past the budget,
         * projection) on the side streams, joined into `stream` afterwards */
        const int K = e->nside;
        for (int i = 0; i < e->n && rc == WF_OK; i++) {
            Solver *s = e->m[i];
            s->stream = (K > 1) ? e->side[i % K] : e->stream;
            const WfState ys = wf_view(s, s->state[2]), yn = wf_view(s, s->state[s->i_yn]);
            const int max_iter = wf_max_iter(s->P);
            if (max_iter > 0 && !s->hflag->done && e->budget < max_iter) {
                /* not converged within the budget: the further solves of its solo run */
                if ((rc = wf_pressure_rest(s, ys, yn, e->budget))) break;
            } else if (max_iter > 0) {
                const WfIterCtl &ctl = e->ctl_host[i];
                s->press_solves += ctl.solves;
                s->last_err = (s->P.variable_density == 0) ? 0.0 : ctl.err;
                s->last_iters = (s->P.variable_density == 0) ? 0 : ctl.iters;
            } else {
                s->last_err = 0.0;
                s->last_iters = 0;
            }
            const WfSource src = wf_source(s, n);
            const hipError_t pe = wf_launch_project(s->c, ys, yn, s->p, wf_view(s, s->state[s->i_x0]), src, s->stream);
            if (pe != hipSuccess) {
                rc = wf_fail(WF_E_DEVICE, "projection: %s", hipGetErrorString(pe));
                break;
            }
            const int old_yn = s->i_yn;
            s->i_yn = s->i_x0;
            s->i_x0 = old_yn;
            s->steps++;
        }
        for (int i = 0; i < e->n; i++) e->m[i]->stream = e->stream;
        if (K > 1) {
            for (int k = 0; k < K; k++) {
                WF_HIP(hipEventRecord(e->join[k], e->side[k]));
                WF_HIP(hipStreamWaitEvent(e->stream, e->join[k], 0));
            }
        }
        if (rc) return rc;
        e->parity ^= 1;
    }
    WF_HIP(hipStreamSynchronize(e->stream));
    return WF_OK;
}

}  // namespace WF_NS
