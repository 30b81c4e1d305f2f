/*
 * wf_closure_train.hip -- training of the learned subgrid closure on the GPU
 * with the network's own BF16 MFMA forward and backward kernels (FP32
 * accumulation), Adam on FP32 master weights.  No counterpart in the
 * reference.
 *
 * Loss over a batch of rows r with inputs f_r and target viscosity nu_r:
 *   L = w sum_r (softplus(z_r) - nu_r / out_scale)^2,   w = 1 / batch.
 * Rounding points (restated by the oracle's oracle_closure_gradient): the
 * forward of wf_closure.h (bf16 inputs, weights and activations); then
 *   dz  = 2 w (yhat - t) sigmoid(z)                          FP32
 *   dh2 = dz bf16(w3) gelu'(h2);  dh1 = (W2^T bf16(dh2)) gelu'(h1)
 *   dW2 = sum bf16(dh2) a1^T,  dW1 = sum bf16(dh1) x^T       MFMA, samples as K
 *   db2, db1, dw3, db3 from the FP32 deltas                  VALU
 * The weight gradients are straight-through: the bf16 rounding of the
 * weights counts as the identity.
 *
 * Gradient kernel: each pass of a workgroup takes 32 rows, in two 16-row
 * tiles for the forward products and as the K dimension of the
 * weight-gradient products; each of its four wavefronts owns 16 of the 64
 * hidden units.  Per-workgroup partial sums are reduced in a fixed order, so a
 * gradient is deterministic.
 */
#include <math.h>
#include <stdint.h>
#include <string.h>
#include <vector>
#include "../../../include/wildfires.h"
#include "wf_closure.h"
#include "wf_kernels.h"

using namespace WF_NS; /* compiled once, in the FP64 namespace */

#define WF_CLT_NP (WF_CL_NPARAMS + 1) /* gradient entries + the loss */
#define WF_CLT_MAXWG 1024

/* per-workgroup LDS of the trainer: activations and deltas of 32 rows in row
 * ([row][unit]) and transposed ([unit][row]) order, bf16 */
struct __attribute__((aligned(16))) WfClTrainLds {
    __bf16 a1s[32 * 64], a1t[64 * 32], a2s[32 * 64];
    __bf16 dh2s[32 * 64], dh2t[64 * 32], dh1t[64 * 32];
    __bf16 xt[16 * 32];
    float dz[32];
};

__device__ __forceinline__ float wf_cl_gelu_d(float h) {
    const float s = 1.0f / (1.0f + expf(-1.702f * h));
    return s + 1.702f * h * s * (1.0f - s);
}

/* trainable entries of the parameter block */
__host__ __device__ __forceinline__ bool wf_cl_trainable(int q) { return q >= WF_CL_W1 && q <= WF_CL_B3; }

/* x: rows of 16 bf16 (12 normalised inputs, 4 zeros); t: targets nu / out_scale.
 * Rows [off, off + cnt); part: per workgroup WF_CLT_NP partial sums.
 * A batch of 8192 rows is one pass of 256 workgroups, so the kernel is as long
 * as the chain of one pass: four exponentials and divisions per row and hidden
 * unit.  With one wavefront per pass that chain covered all 64 units (22 us;
 * 12 us with four wavefronts of 16 units each). */
__global__ __launch_bounds__(256) void k_cl_grad(WfClosure cl, const wf_bf16x8 *w2bt, const __bf16 *x, const float *t,
                                                 long off, long cnt, float w, float *part) {
    __shared__ WfClTrainLds L;
    const int l = threadIdx.x & 63, lr = l & 15, lg = l >> 4;
    const int nt = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); /* the wavefront's units 16 nt .. 16 nt + 15 */
    const int n = nt * 16 + lr;
    const float *prm = cl.prm;
    const wf_bf16x8 *W1 = cl.frag + WF_CL_FRAG_W1, *W2 = cl.frag + WF_CL_FRAG_W2, *W3 = cl.frag + WF_CL_FRAG_W3;
    const wf_bf16x8 w1 = W1[nt * 64 + l], w2a = W2[(nt * 2) * 64 + l], w2b = W2[(nt * 2 + 1) * 64 + l];
    const wf_bf16x8 w3a = W3[l], w3c = W3[64 + l], wta = w2bt[(nt * 2) * 64 + l], wtb = w2bt[(nt * 2 + 1) * 64 + l];
    const float b1 = prm[WF_CL_B1 + n], b2 = prm[WF_CL_B2 + n], b3 = prm[WF_CL_B3];
    const float w3b = (float)(__bf16)prm[WF_CL_W3 + n];
    wf_f32x4 gW2[4], gW1 = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int b = 0; b < 4; b++) gW2[b] = wf_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    float gw3 = 0.0f, gb2 = 0.0f, gb1 = 0.0f, gb3 = 0.0f, loss = 0.0f;
    const long ngroups = (cnt + 31) / 32;
    for (long grp = blockIdx.x; grp < ngroups; grp += gridDim.x) {
        const long base = off + grp * 32;
        const long last = off + cnt - 1;
        /* forward */
        wf_f32x4 h1[2], h2[2];
#pragma unroll
        for (int mt = 0; mt < 2; mt++) {
            long row = base + mt * 16 + lr;
            row = (row <= last) ? row : last;
            wf_bf16x8 a = {};
            if (lg < 2) a = *(const wf_bf16x8 *)&x[row * 16 + 8 * lg];
#pragma unroll
            for (int j = 0; j < 8; j++)
                if (nt == 0 && lg < 2) L.xt[(8 * lg + j) * 32 + mt * 16 + lr] = a[j];
            const wf_f32x4 d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, w1, wf_f32x4{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                h1[mt][r] = d[r] + b1;
                const __bf16 v = (__bf16)wf_cl_gelu(h1[mt][r]);
                const int s = mt * 16 + 4 * lg + r;
                L.a1s[s * 64 + n] = v;
                L.a1t[n * 32 + s] = v;
            }
        }
        __syncthreads();
#pragma unroll
        for (int mt = 0; mt < 2; mt++) {
            const wf_bf16x8 aa = *(const wf_bf16x8 *)&L.a1s[(mt * 16 + lr) * 64 + 8 * lg];
            const wf_bf16x8 ab = *(const wf_bf16x8 *)&L.a1s[(mt * 16 + lr) * 64 + 32 + 8 * lg];
            wf_f32x4 d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(aa, w2a, wf_f32x4{0, 0, 0, 0}, 0, 0, 0);
            d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ab, w2b, d, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                h2[mt][r] = d[r] + b2;
                L.a2s[(mt * 16 + 4 * lg + r) * 64 + n] = (__bf16)wf_cl_gelu(h2[mt][r]);
            }
        }
        __syncthreads();
        if (nt == 0) {
#pragma unroll
            for (int mt = 0; mt < 2; mt++) {
                const wf_bf16x8 aa = *(const wf_bf16x8 *)&L.a2s[(mt * 16 + lr) * 64 + 8 * lg];
                const wf_bf16x8 ab = *(const wf_bf16x8 *)&L.a2s[(mt * 16 + lr) * 64 + 32 + 8 * lg];
                wf_f32x4 z = __builtin_amdgcn_mfma_f32_16x16x32_bf16(aa, w3a, wf_f32x4{0, 0, 0, 0}, 0, 0, 0);
                z = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ab, w3c, z, 0, 0, 0);
                if (lr == 0) {
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int s = mt * 16 + 4 * lg + r;
                        const long row = base + s;
                        const float zv = z[r] + b3;
                        const float e = (row <= last) ? wf_cl_softplus(zv) - t[row] : 0.0f;
                        loss += w * e * e;
                        const float dz = 2.0f * w * e * (1.0f / (1.0f + expf(-zv)));
                        gb3 += dz;
                        L.dz[s] = dz;
                    }
                }
            }
        }
        /* gelu' of both layers does not wait for dz */
        float g1[2][4], g2[2][4];
#pragma unroll
        for (int mt = 0; mt < 2; mt++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                g1[mt][r] = wf_cl_gelu_d(h1[mt][r]);
                g2[mt][r] = wf_cl_gelu_d(h2[mt][r]);
            }
        __syncthreads();
        /* backward: output layer and second hidden layer */
#pragma unroll
        for (int mt = 0; mt < 2; mt++) {
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int s = mt * 16 + 4 * lg + r;
                const float dz = L.dz[s];
                gw3 += dz * (float)L.a2s[s * 64 + n];
                const float d = dz * w3b * g2[mt][r];
                gb2 += d;
                const __bf16 db = (__bf16)d;
                L.dh2s[s * 64 + n] = db;
                L.dh2t[n * 32 + s] = db;
            }
        }
        __syncthreads();
        /* dW2 += bf16(dh2)^T a1 over the 32 rows (the wavefront's 16 rows of dW2) */
        {
            const wf_bf16x8 A = *(const wf_bf16x8 *)&L.dh2t[n * 32 + 8 * lg];
#pragma unroll
            for (int ki = 0; ki < 4; ki++) {
                const wf_bf16x8 B = *(const wf_bf16x8 *)&L.a1t[(ki * 16 + lr) * 32 + 8 * lg];
                gW2[ki] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A, B, gW2[ki], 0, 0, 0);
            }
        }
        /* da1 = bf16(dh2) W2, then dh1 */
#pragma unroll
        for (int mt = 0; mt < 2; mt++) {
            const wf_bf16x8 Aa = *(const wf_bf16x8 *)&L.dh2s[(mt * 16 + lr) * 64 + 8 * lg];
            const wf_bf16x8 Ab = *(const wf_bf16x8 *)&L.dh2s[(mt * 16 + lr) * 64 + 32 + 8 * lg];
            wf_f32x4 d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(Aa, wta, wf_f32x4{0, 0, 0, 0}, 0, 0, 0);
            d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(Ab, wtb, d, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int s = mt * 16 + 4 * lg + r;
                const float dh = d[r] * g1[mt][r];
                gb1 += dh;
                L.dh1t[n * 32 + s] = (__bf16)dh;
            }
        }
        wf_cl_wave_sync(); /* dh1t: a wavefront reads the rows that it wrote */
        /* dW1 += bf16(dh1)^T x over the 32 rows (input columns 12..15 are zero) */
        {
            const wf_bf16x8 B = *(const wf_bf16x8 *)&L.xt[lr * 32 + 8 * lg];
            const wf_bf16x8 A = *(const wf_bf16x8 *)&L.dh1t[n * 32 + 8 * lg];
            gW1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A, B, gW1, 0, 0, 0);
        }
        __syncthreads(); /* this pass's LDS reads are done before the next pass writes */
    }
    /* partial sums of this workgroup */
    float *P = part + (long)blockIdx.x * WF_CLT_NP;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int m = nt * 16 + 4 * lg + r;
#pragma unroll
        for (int ki = 0; ki < 4; ki++) P[WF_CL_W2 + m * 64 + ki * 16 + lr] = gW2[ki][r];
        if (lr < WF_CL_NIN) P[WF_CL_W1 + m * WF_CL_NIN + lr] = gW1[r];
    }
    gw3 += __shfl_xor(gw3, 16, 64);
    gw3 += __shfl_xor(gw3, 32, 64);
    gb2 += __shfl_xor(gb2, 16, 64);
    gb2 += __shfl_xor(gb2, 32, 64);
    gb1 += __shfl_xor(gb1, 16, 64);
    gb1 += __shfl_xor(gb1, 32, 64);
    if (lg == 0) {
        P[WF_CL_W3 + n] = gw3;
        P[WF_CL_B2 + n] = gb2;
        P[WF_CL_B1 + n] = gb1;
    }
    for (int o = 32; o > 0; o >>= 1) {
        gb3 += __shfl_xor(gb3, o, 64);
        loss += __shfl_xor(loss, o, 64);
    }
    if (threadIdx.x == 0) {
        P[WF_CL_B3] = gb3;
        P[WF_CL_NPARAMS] = loss;
    }
}

/* Places of parameter q in the MFMA operands: the forward set of wf_closure.h
 * and W2 for the da1 product (B[k = n][col = k_in] = W2[n][k_in], 4 column
 * tiles x 2 K-steps), each an element of an operand of 8. */
__device__ __forceinline__ void wf_cl_place(int q, float v, __bf16 *frag, __bf16 *w2bt) {
    const __bf16 b = (__bf16)v;
    if (q >= WF_CL_W1 && q < WF_CL_B1) {
        const int n = (q - WF_CL_W1) / WF_CL_NIN, k = (q - WF_CL_W1) % WF_CL_NIN;
        frag[(WF_CL_FRAG_W1 + (n >> 4) * 64 + (k >> 3) * 16 + (n & 15)) * 8 + (k & 7)] = b;
    } else if (q >= WF_CL_W2 && q < WF_CL_B2) {
        const int n = (q - WF_CL_W2) >> 6, k = (q - WF_CL_W2) & 63;
        frag[(WF_CL_FRAG_W2 + ((n >> 4) * 2 + (k >> 5)) * 64 + ((k & 31) >> 3) * 16 + (n & 15)) * 8 + (k & 7)] = b;
        w2bt[(((k >> 4) * 2 + (n >> 5)) * 64 + ((n & 31) >> 3) * 16 + (k & 15)) * 8 + (n & 7)] = b;
    } else if (q >= WF_CL_W3 && q < WF_CL_B3) {
        const int k = q - WF_CL_W3;
        frag[(WF_CL_FRAG_W3 + (k >> 5) * 64 + ((k & 31) >> 3) * 16) * 8 + (k & 7)] = b;
    }
}
/* the operands of an initial block (their other entries are 0) */
__global__ void k_cl_place(const float *prm, __bf16 *frag, __bf16 *w2bt) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q < WF_CL_NPARAMS) wf_cl_place(q, prm[q], frag, w2bt);
}

/* grad[q] = sum over the nwg partials (trainable entries and the loss; 0
 * elsewhere), in order.  Then, for a training step (step >= 1), Adam on the
 * trainable entries (bias-corrected) and their places in the MFMA operands.
 * One wavefront per workgroup, 64 partials of each entry in flight: the sum is
 * a chain of additions, but its loads are independent (one load at a time in
 * 20 workgroups took 58 us for 256 partials; with the update and the
 * operands as launches of their own a step of 8192 rows took 90 us, now 20). */
#define WF_CLT_RED 64
__global__ __launch_bounds__(64) void k_cl_update(const float *part, int nwg, float *grad, float *prm, float *m,
                                                  float *v, __bf16 *frag, __bf16 *w2bt, float lr, float b1, float b2,
                                                  float eps, int step) {
    const int q = blockIdx.x * 64 + threadIdx.x;
    if (q >= WF_CLT_NP) return;
    float s = 0.0f;
    if (wf_cl_trainable(q) || q == WF_CL_NPARAMS) {
        for (int b0 = 0; b0 < nwg; b0 += WF_CLT_RED) {
            float a[WF_CLT_RED];
#pragma unroll
            for (int u = 0; u < WF_CLT_RED; u++) a[u] = part[(long)min(b0 + u, nwg - 1) * WF_CLT_NP + q];
            if (b0 + WF_CLT_RED <= nwg) {
#pragma unroll
                for (int u = 0; u < WF_CLT_RED; u++) s += a[u];
            } else {
#pragma unroll
                for (int u = 0; u < WF_CLT_RED; u++)
                    if (b0 + u < nwg) s += a[u];
            }
        }
    }
    grad[q] = s;
    if (step < 1 || q >= WF_CL_NPARAMS || !wf_cl_trainable(q)) return;
    const float mq = b1 * m[q] + (1.0f - b1) * s;
    const float vq = b2 * v[q] + (1.0f - b2) * s * s;
    m[q] = mq;
    v[q] = vq;
    const float mh = mq / (1.0f - powf(b1, (float)step)), vh = vq / (1.0f - powf(b2, (float)step));
    const float pq = prm[q] - lr * mh / (sqrtf(vh) + eps);
    prm[q] = pq;
    wf_cl_place(q, pq, frag, w2bt);
}

/* ---------------------------------------------------------------- C-ABI ---- */

struct wf_closure_trainer {
    long n;
    float *prm, *m, *v, *part, *grad;
    wf_bf16x8 *frag, *w2bt;
    __bf16 *x;
    float *t;
    int step;
};

#define WF_CLT_HIP(call)                                                                         \
    do {                                                                                         \
        hipError_t e_ = (call);                                                                  \
        if (e_ != hipSuccess) return wf_set_error(WF_E_DEVICE, hipGetErrorString(e_));           \
    } while (0)

/* one gradient over rows [off, off + cnt) with weight w into T->grad and, for
 * training step `step` (0: none), the Adam step with it */
static int wf_clt_grad(wf_closure_trainer *T, long off, long cnt, float w, float lr, int step) {
    const long groups = (cnt + 31) / 32;
    const int nwg = (int)((groups < WF_CLT_MAXWG) ? groups : WF_CLT_MAXWG);
    hipLaunchKernelGGL(k_cl_grad, dim3(nwg), dim3(256), 0, 0, WfClosure{T->prm, T->frag}, T->w2bt, T->x, T->t, off,
                       cnt, w, T->part);
    WF_CLT_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_cl_update, dim3((WF_CLT_NP + 63) / 64), dim3(64), 0, 0, T->part, nwg, T->grad, T->prm, T->m,
                       T->v, (__bf16 *)T->frag, (__bf16 *)T->w2bt, lr, 0.9f, 0.999f, 1e-8f, step);
    WF_CLT_HIP(hipGetLastError());
    return WF_OK;
}

extern "C" int wf_closure_trainer_destroy(wf_closure_trainer *T) {
    if (T == NULL) return WF_OK;
    (void)hipDeviceSynchronize();
    void *b[] = {T->prm, T->m, T->v, T->part, T->grad, T->frag, T->w2bt, T->x, T->t};
    for (void *p : b)
        if (p) (void)hipFree(p);
    free(T);
    return WF_OK;
}

extern "C" int wf_closure_trainer_create(const float *params, long nparams, const double *features,
                                         const double *nu_target, long n, wf_closure_trainer **out) {
    if (out == NULL || params == NULL || features == NULL || nu_target == NULL || n <= 0)
        return wf_set_error(WF_E_ARG, "closure trainer: null argument or empty data");
    *out = NULL;
    if (nparams != WF_CL_NPARAMS) return wf_set_error(WF_E_ARG, "closure trainer: wrong parameter count");
    for (long q = 0; q < nparams; q++)
        if (!isfinite(params[q])) return wf_set_error(WF_E_ARG, "closure trainer: parameter not finite");
    if (!(params[WF_CL_SCALE] > 0.0f)) return wf_set_error(WF_E_ARG, "closure trainer: out_scale must be positive");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return wf_set_error(WF_E_DEVICE, "no HIP device");
    WF_CLT_HIP(hipSetDevice(0));
    /* normalised bf16 inputs (the rounding of wf_cl_inputs) and targets */
    std::vector<uint16_t> xb((size_t)n * 16, 0);
    std::vector<float> tb(n);
    for (long r = 0; r < n; r++) {
        for (int i = 0; i < WF_CL_NIN; i++) {
            const double f = features[r * WF_CL_NIN + i];
            xb[(size_t)r * 16 + i] =
                wf_bf16_bits((float)((f - (double)params[WF_CL_MEAN + i]) * (double)params[WF_CL_ISTD + i]));
        }
        tb[r] = (float)(nu_target[r] / (double)params[WF_CL_SCALE]);
    }
    wf_closure_trainer *T = (wf_closure_trainer *)calloc(1, sizeof(wf_closure_trainer));
    if (T == NULL) return wf_set_error(WF_E_ALLOC, "closure trainer: host allocation");
    T->n = n;
    hipError_t e = hipMalloc((void **)&T->prm, sizeof(float) * WF_CL_NPARAMS);
    if (e == hipSuccess) e = hipMalloc((void **)&T->m, sizeof(float) * WF_CL_NPARAMS);
    if (e == hipSuccess) e = hipMalloc((void **)&T->v, sizeof(float) * WF_CL_NPARAMS);
    if (e == hipSuccess) e = hipMalloc((void **)&T->part, sizeof(float) * WF_CLT_NP * WF_CLT_MAXWG);
    if (e == hipSuccess) e = hipMalloc((void **)&T->grad, sizeof(float) * WF_CLT_NP);
    if (e == hipSuccess) e = hipMalloc((void **)&T->frag, sizeof(wf_bf16x8) * WF_CL_NFRAG);
    if (e == hipSuccess) e = hipMalloc((void **)&T->w2bt, sizeof(wf_bf16x8) * 8 * 64);
    if (e == hipSuccess) e = hipMalloc((void **)&T->x, sizeof(uint16_t) * 16 * (size_t)n);
    if (e == hipSuccess) e = hipMalloc((void **)&T->t, sizeof(float) * n);
    if (e == hipSuccess) e = hipMemcpy(T->prm, params, sizeof(float) * WF_CL_NPARAMS, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemset(T->m, 0, sizeof(float) * WF_CL_NPARAMS);
    if (e == hipSuccess) e = hipMemset(T->v, 0, sizeof(float) * WF_CL_NPARAMS);
    if (e == hipSuccess) e = hipMemset(T->frag, 0, sizeof(wf_bf16x8) * WF_CL_NFRAG);
    if (e == hipSuccess) e = hipMemset(T->w2bt, 0, sizeof(wf_bf16x8) * 8 * 64);
    if (e == hipSuccess) e = hipMemcpy(T->x, xb.data(), sizeof(uint16_t) * 16 * (size_t)n, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(T->t, tb.data(), sizeof(float) * n, hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        wf_closure_trainer_destroy(T);
        return wf_set_error(WF_E_DEVICE, hipGetErrorString(e));
    }
    hipLaunchKernelGGL(k_cl_place, dim3((WF_CL_NPARAMS + 63) / 64), dim3(64), 0, 0, T->prm, (__bf16 *)T->frag,
                       (__bf16 *)T->w2bt);
    e = hipGetLastError();
    if (e != hipSuccess) {
        wf_closure_trainer_destroy(T);
        return wf_set_error(WF_E_DEVICE, hipGetErrorString(e));
    }
    *out = T;
    return WF_OK;
}

extern "C" int wf_closure_trainer_gradient(wf_closure_trainer *T, long offset, long count, double weight,
                                           float *grad, double *loss) {
    if (T == NULL || grad == NULL || loss == NULL || offset < 0 || count <= 0 || offset + count > T->n)
        return wf_set_error(WF_E_ARG, "closure trainer: bad row range");
    int rc = wf_clt_grad(T, offset, count, (float)weight, 0.0f, 0);
    if (rc) return rc;
    std::vector<float> g(WF_CLT_NP);
    WF_CLT_HIP(hipMemcpy(g.data(), T->grad, sizeof(float) * WF_CLT_NP, hipMemcpyDeviceToHost));
    memcpy(grad, g.data(), sizeof(float) * WF_CL_NPARAMS);
    *loss = g[WF_CL_NPARAMS];
    return WF_OK;
}

extern "C" int wf_closure_trainer_train(wf_closure_trainer *T, int steps, long batch, double lr, double *last_loss) {
    if (T == NULL || steps < 0 || batch <= 0 || batch > T->n || !(lr > 0.0))
        return wf_set_error(WF_E_ARG, "closure trainer: bad training arguments");
    long off = ((long)T->step * batch) % T->n;
    for (int s = 0; s < steps; s++) {
        if (off + batch > T->n) off = 0;
        int rc = wf_clt_grad(T, off, batch, 1.0f / (float)batch, (float)lr, T->step + 1);
        if (rc) return rc;
        T->step++;
        off += batch;
    }
    if (last_loss) {
        float L = 0.0f;
        WF_CLT_HIP(hipMemcpy(&L, T->grad + WF_CL_NPARAMS, sizeof(float), hipMemcpyDeviceToHost));
        *last_loss = L;
    } else {
        WF_CLT_HIP(hipDeviceSynchronize());
    }
    return WF_OK;
}

extern "C" int wf_closure_trainer_params(wf_closure_trainer *T, float *params) {
    if (T == NULL || params == NULL) return wf_set_error(WF_E_ARG, "closure trainer: null argument");
    WF_CLT_HIP(hipMemcpy(params, T->prm, sizeof(float) * WF_CL_NPARAMS, hipMemcpyDeviceToHost));
    return WF_OK;
}
