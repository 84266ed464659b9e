// mi_gp.hip -- the Gaussian-process negative log marginal likelihood and its
// gradient over the tile kernels (no counterpart in the reference):
//
//   nll  = 1/2 a^T a + sum_i log L_ii + N/2 log 2 pi,   K = L L^T, a = L^{-1} y
//   dnll/dK = the reverse of the factorization applied to
//             Lbar = -tril(alpha a^T) + diag(1 / L_ii),  alpha = L^{-T} a
//
// K and its gradient are dense row-major arrays (the lower triangle of a
// row-major array is the upper triangle of the same memory read column-major,
// which is what the staging kernels take); each call enqueues everything on
// the context's streams and waits once.  Against the factorization, torch's
// triangular solve and its backward, and copies between the layouts by torch
// indexing (N = 8192, NB = 512, FP64, forward and backward with the kernel
// matrix): 33.6 -> 19.8 ms; N = 1024, NB = 256, FP32: 1.9 -> 1.4 ms.
#include "mi_common.hpp"
#include "dplasma_mi.h"

using namespace mi;

namespace {

constexpr int UPPER = 121, LOWER = 122;

// out[0] = sum log L_ii, out[1] = sum a_i^2, in FP64; one workgroup, a fixed
// order of summation.  A chain of N / 1024 cache misses and one tree: 5 us at
// N = 1024, too little to be worth a second launch.
template <class T>
__global__ __launch_bounds__(1024) void k_gp_value(const T *__restrict__ Lt, int N, int NB, int MT,
                                                   const T *__restrict__ a, double *__restrict__ out)
{
    __shared__ double sl[1024], sa[1024];
    double l = 0.0, q = 0.0;
    for (int i = threadIdx.x; i < N; i += 1024) {
        const int k = i / NB, r = i - k * NB;
        l += log((double)Lt[tile_index(MT, k, k) * (int64_t)NB * NB + (int64_t)r * NB + r]);
        q += (double)a[i] * (double)a[i];
    }
    sl[threadIdx.x] = l;
    sa[threadIdx.x] = q;
    for (int h = 512; h > 0; h >>= 1) {
        __syncthreads();
        if (threadIdx.x < h) {
            sl[threadIdx.x] += sl[threadIdx.x + h];
            sa[threadIdx.x] += sa[threadIdx.x + h];
        }
    }
    if (threadIdx.x == 0) {
        out[0] = sl[0];
        out[1] = sa[0];
    }
}

// Lbar of the likelihood in packed lower tiles, times *scale: workgroup
// (tile, group of 8 columns); zero above the diagonal and beyond N.  Bound by
// its stores: 66 us for the 285 MB of N = 8192, FP64.
template <class T>
__global__ __launch_bounds__(256) void k_gp_seed(const T *__restrict__ Lt, int N, int NB, int MT,
                                                 const T *__restrict__ a, const T *__restrict__ alpha,
                                                 const T *__restrict__ scale, T *__restrict__ G)
{
    int t = blockIdx.x, n = 0;
    while (t >= MT - n) { t -= MT - n; n++; }
    const int m = n + t;
    const T g = *scale;
    const int64_t base = (int64_t)blockIdx.x * NB * NB;
    for (int c = 8 * blockIdx.y; c < min(NB, 8 * (int)blockIdx.y + 8); c++) {
        const int j = n * NB + c;
        const T aj = g * (j < N ? a[j] : T(0));
        for (int r = threadIdx.x; r < NB; r += 256) {
            const int i = m * NB + r;
            T v = T(0);
            if (i < N && j < N && i >= j) {
                v = -alpha[i] * aj;
                if (i == j) v += g / Lt[base + (int64_t)c * NB + r];
            }
            G[base + (int64_t)c * NB + r] = v;
        }
    }
}

int check(const char *f, int N, int NB, int ld)
{
    if (N < 1 || ld < N) { set_error("%s: bad sizes N=%d ld=%d", f, N, ld); return -2; }
    // the tile sizes of the wavefront solve
    if (NB <= 0 || NB % 32 || NB > 960) { set_error("%s: NB=%d must be a multiple of 32, at most 960", f, NB); return -2; }
    return 0;
}

// trans: 111 / 112; x in place
template <class T> int solve(Ctx *c, int trans, int N, int NB, const T *dT, T *x)
{
    int rc;
    hipStream_t s = c->s_main;
    T *W = (T *)ws_get(c, WS_TRSM, trsm_ws_elems(N, NB) * sizeof(T));
    if (!W) return -3;
    if ((rc = trsm_begin(c, s))) return rc;
    if ((rc = trsm_prepare<T>(c, s, 0, N, NB, dT, W))) return rc;
    return trsm_enqueue<T>(c, s, trans, N, NB, dT, W, 1, x, N);
}

// the span between the context's events, for mi_last_span_ms
int span(Ctx *c)
{
    float ms = 0.f;
    MI_CHECK(hipEventElapsedTime(&ms, c->t0, c->t1));
    c->last_ms = ms;
    return 0;
}

template <class T>
int enqueue_nll(Ctx *c, int N, int NB, const T *dK, int ldk, T *dT, T *dy, double *dout, int *h_info)
{
    int rc;
    const int MT = (N + NB - 1) / NB;
    hipStream_t s = c->s_main;
    if ((rc = sym_stage_enqueue<T>(c, s, true, UPPER, N, NB, dT, const_cast<T *>(dK), ldk))) return rc;
    if ((rc = potrf_enqueue<T>(c, N, NB, dT))) return rc;
    // a failed factorization is noticed after the wait; what follows it then
    // works on numbers nobody reads
    if ((rc = solve<T>(c, 111, N, NB, dT, dy))) return rc;
    MI_LAUNCH(c, s, "gp_value", 0.0, 0.0, (k_gp_value<T><<<1, 1024, 0, s>>>(dT, N, NB, MT, dy, dout)));
    MI_CHECK(hipMemcpyAsync(h_info, c->d_info, sizeof(int), hipMemcpyDeviceToHost, s));
    return 0;
}

template <class T>
int gp_nll(mi_ctx_t *c, int N, int NB, const T *dK, int ldk, T *dT, T *dy, double *dout, int *info)
{
    *info = 0;
    int rc = check("mi_gp_nll", N, NB, ldk), h_info = 0;
    if (rc || (rc = potrf_check<T>(NB))) return rc;      // before anything is written
    rc = enqueue_nll<T>(c, N, NB, dK, ldk, dT, dy, dout, &h_info);
    // the wait comes first also after an error: the caller may free its arrays
    const int rs = mi_synchronize(c);
    if (rc || rs) return rc ? rc : rs;
    *info = h_info;
    if ((rc = span(c))) return rc;                 // the factorization's, between its own events
    return h_info ? 0 : trsm_status(c);
}

template <class T>
int enqueue_grad(Ctx *c, int N, int NB, const T *dT, const T *da, T *dalpha, const T *dscale, T *dG, T *dK, int ldk)
{
    int rc;
    const int MT = (N + NB - 1) / NB;
    hipStream_t s = c->s_main;
    MI_CHECK(hipMemcpyAsync(dalpha, da, (size_t)N * sizeof(T), hipMemcpyDeviceToDevice, s));
    if ((rc = solve<T>(c, 112, N, NB, dT, dalpha))) return rc;
    const dim3 grid((unsigned)((int64_t)MT * (MT + 1) / 2), (unsigned)((NB + 7) / 8));
    MI_LAUNCH(c, s, "gp_seed", 0.0, (double)MT * (MT + 1) / 2 * NB * NB * sizeof(T),
              (k_gp_seed<T><<<grid, 256, 0, s>>>(dT, N, NB, MT, da, dalpha, dscale, dG)));
    MI_CHECK(hipEventRecord(c->t0, s));
    if ((rc = adjoint_enqueue<T>(c, N, NB, dT, dG))) return rc;
    MI_CHECK(hipEventRecord(c->t1, s));
    // the symmetric gradient: both triangles from the lower tiles
    if ((rc = sym_stage_enqueue<T>(c, s, false, UPPER, N, NB, dG, dK, ldk))) return rc;
    return sym_stage_enqueue<T>(c, s, false, LOWER, N, NB, dG, dK, ldk);
}

template <class T>
int gp_nll_grad(mi_ctx_t *c, int N, int NB, const T *dT, const T *da, T *dalpha, const T *dscale, T *dG, T *dK, int ldk)
{
    int rc = check("mi_gp_nll_grad", N, NB, ldk);
    if (rc) return rc;
    rc = enqueue_grad<T>(c, N, NB, dT, da, dalpha, dscale, dG, dK, ldk);
    const int rs = mi_synchronize(c);
    if (rc || rs) return rc ? rc : rs;
    if ((rc = span(c))) return rc;
    return trsm_status(c);
}

}  // namespace

extern "C" {

int mi_dgp_nll(mi_ctx_t *c, int N, int NB, const double *dK, int ldk, double *dT, double *dy, double *dout, int *info)
{
    return gp_nll<double>(c, N, NB, dK, ldk, dT, dy, dout, info);
}

int mi_sgp_nll(mi_ctx_t *c, int N, int NB, const float *dK, int ldk, float *dT, float *dy, double *dout, int *info)
{
    return gp_nll<float>(c, N, NB, dK, ldk, dT, dy, dout, info);
}

int mi_dgp_nll_grad(mi_ctx_t *c, int N, int NB, const double *dT, const double *da, double *dalpha,
                    const double *dscale, double *dG, double *dK, int ldk)
{
    return gp_nll_grad<double>(c, N, NB, dT, da, dalpha, dscale, dG, dK, ldk);
}

int mi_sgp_nll_grad(mi_ctx_t *c, int N, int NB, const float *dT, const float *da, float *dalpha, const float *dscale,
                    float *dG, float *dK, int ldk)
{
    return gp_nll_grad<float>(c, N, NB, dT, da, dalpha, dscale, dG, dK, ldk);
}

}  // extern "C"
