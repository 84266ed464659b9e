// mi_batched.hip -- many independent SPD systems of uneven sizes, factored
// and solved in persistent launches (the largest class captured in a hipGraph
// for replay).
//
// No counterpart in the reference (its batching growth path: each matrix
// is dplasma_dposv, src/zposv_wrapper.c:63-113, on one tile; the per-matrix
// semantics are LAPACK dpotrf/dpotrs as in src/cores/core_zpotrf.c:68-74:
// info = first column whose pivot is not positive, 1-based, and the matrix
// is left partly factored).
//
// Layout: matrix i is n_i x n_i column-major (lda = n_i) at element offset
// sum_{j<i} n_j^2 of one buffer; its right-hand side (NRHS = 1) at offset
// sum_{j<i} n_j of another.  n_i <= 1024.
//
// A workgroup takes matrices from a queue (one atomic counter) in decreasing
// size order (longest first, which bounds the imbalance by the last small
// matrices) and factors one matrix with all its NW waves, left-looking over
// panels of 16 NW columns, on 16 x 16 blocks in the accumulator layout of
// mi_panel.hpp:
//   1. the panel's diagonal block rows (one a wave) lose the products with
//      every column to the left, then diag_factor factors the block and leaves
//      the images of -L and W in LDS;
//   2. the other block rows, RT a wave at a time, do the same product and are
//      solved against these images, in registers from load to store.
// In these products a wave's own rows are MFMA operands straight from memory;
// the panel's rows are staged through LDS for all waves.
// The right-hand side is carried along like one more row below the matrix (y,
// kept in LDS), so the forward solve comes with the factorization; the
// backward solve then goes through the panels from the last.
// Three instances: matrices above 128 (panels of 128), those of at most 128
// and of at most 64 (one panel, and more workgroups per CU).
//
// Measured (512 matrices of one order with solve, FP64 / FP32 ms; in brackets
// 64- or 128-wide panels of 32-column blocks from memory, factored by
// v_readlane broadcasts, and a separate solve): n = 1024 5.16 / 2.55 (9.11 /
// 4.69), 512 0.96 / 0.47 (2.02 / 1.02), 256 0.25 / 0.12 (0.53 / 0.31), 128
// 0.084 / 0.045 (0.150 / 0.116), 32 0.028 / 0.023 (0.042 / 0.038); 4096 of
// 32..1024 14.2 / 6.8 (26.0 / 13.7).  Bound at n = 1024 by the products to the
// left (4.2 us a stage of a full pass, 3.4 us of it MFMA; half-empty last
// passes), below 256 by the chain of pivots (diag_factor).
#include <algorithm>
#include <numeric>
#include <vector>

#include "mi_common.hpp"
#include "mi_panel.hpp"
#include "dplasma_mi.h"

using namespace mi;

namespace {

constexpr int BMAX = 1024;        // largest matrix order of a batch
constexpr int BKC = 16;           // columns to the left per stage

template <class T, int NW, bool MULTI> struct BShared {
    static constexpr int PW = DB * NW;                   // panel columns
    static constexpr int WP = DIAG_WP;
    T img[NW * (NW - 1) / 2][OPI];                       // -L(i, j), i > j, of the current panel
    T w[NW][DB * WP];                                    // W_p, image column t at t WP
    DiagLds<T> ds;
    T bs[MULTI ? 2 : 1][MULTI ? BKC : 1][PW + 128 / sizeof(T)];   // staged rows of the panel, [k][row]
    T ys[MULTI ? BMAX : PW];                             // y, then x
    T ts[PW];                                            // right-hand side of a panel's solve
    T red[4][MULTI ? PW : 1];                            // partial sums
    int idx;
};

// v summed over each row of 16 lanes, in every lane of the row
template <class T> __device__ __forceinline__ T row_sum(T v)
{
    v += row_rotate<8>(v);
    v += row_rotate<4>(v);
    v += row_rotate<2>(v);
    v += row_rotate<1>(v);
    return v;
}

template <class T, int NW, int RT, bool MULTI> struct Batch {
    typedef typename MF<T>::v4 V4;
    typedef BShared<T, NW, MULTI> SH;
    static constexpr int PW = SH::PW;
    SH &sh;
    int lane, wave, fr, fk;

    __device__ __forceinline__ explicit Batch(SH &s) : sh(s) { refresh(); }
    // The lane's coordinates, opaque to the compiler from here on: what it
    // derives from them (addresses, conditions per block) is computed where it
    // is used instead of being held across the caller's loops.
    __device__ __forceinline__ void refresh()
    {
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        lane = tid & 63;
        wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        asm volatile("" : "+s"(wave));
        fr = lane & 15;
        fk = lane >> 4;
    }
    __device__ __forceinline__ T *limg(int i, int j) { return sh.img[i * (i - 1) / 2 + j]; }
    __device__ __forceinline__ V4 get_w(int p)
    {
        V4 w;
#pragma unroll
        for (int q = 0; q < 4; q++) w[q] = sh.w[p][(4 * q + fk) * SH::WP + fr];
        return w;
    }
    // x[c] = W(c, fr) of block p, in the lanes of the first row
    __device__ __forceinline__ void put_w(int p, const T *x)
    {
        const int t = sizeof(T) == 8 ? fr : 4 * (fr & 3) + (fr >> 2);
        if (fk == 0) {
#pragma unroll
            for (int c = 0; c < DB; c++) sh.w[p][t * SH::WP + c] = x[c];
        }
    }
    __device__ __forceinline__ static V4 mul(const V4 &a, const V4 &b, V4 c)
    {
#pragma unroll
        for (int s = 0; s < 4; s++) c = MF<T>::mfma(a[s], b[s], c);
        return c;
    }
    __device__ __forceinline__ V4 get(const T *img)
    {
        V4 v;
#pragma unroll
        for (int q = 0; q < 4; q++) v[q] = img[64 * q + lane];
        return v;
    }
    // X = C L^{-T} for one block row, against the panel's images; put(b, X_b)
    template <int BI, class PUT> __device__ __forceinline__ void solve_strip(V4 (&acc)[NW], int nbc, PUT &&put)
    {
        if constexpr (BI < NW) {
            if (BI < nbc) {
                __builtin_amdgcn_sched_barrier(0);
                acc[BI] = mul(get_w(BI), acc[BI], V4{T(0), T(0), T(0), T(0)});
#pragma unroll
                for (int b2 = BI + 1; b2 < NW; b2++) acc[b2] = mul(get(limg(b2, BI)), acc[BI], acc[b2]);
                put(BI, acc[BI]);
                solve_strip<BI + 1>(acc, nbc, put);
            }
        }
    }

    // One pass over the block rows base, base + 1, .. (NW RA of them, below
    // nrb) of the panel at p0: load, update by the columns to the left (UPD),
    // solve against the panel's images (SOLVE), store.  The pass over the
    // diagonal block's rows (no solve) stores their lower part, and updates
    // the right-hand side's row into sh.ts when b.
    template <int RA, bool UPD, bool SOLVE>
    __device__ __forceinline__ void pass(T *__restrict__ A, int n, const T *__restrict__ b, int p0, int base, int nrb)
    {
        const int lda = n;                                   // n <= 1024: 32-bit offsets
        const int ncol = min(PW, n - p0), nbc = (ncol + DB - 1) / DB;
        refresh();
        V4 acc[RA][NW];
        const T *src[RA];                                    // this lane's row, clamped
#pragma unroll
        for (int t = 0; t < RA; t++) {
            src[t] = A + min(p0 + DB * (base + NW * t + wave) + fr, n - 1);
#pragma unroll
            for (int j = 0; j < NW; j++)
#pragma unroll
                for (int q = 0; q < 4; q++) acc[t][j][q] = src[t][min(p0 + DB * j + MF<T>::row(q, fk), n - 1) * lda];
        }
        if constexpr (UPD) left_update<RA, !SOLVE>(A, lda, n, p0, base + wave < nrb, acc, src, b);
        auto put = [&](int rb, int j, const V4 &v) {
            const int r = p0 + DB * rb + fr;
            if (r < n) {
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int c = p0 + DB * j + MF<T>::row(q, fk);
                    if (c < n && (SOLVE || r >= c)) A[c * lda + r] = v[q];
                }
            }
        };
        if constexpr (!SOLVE) {
            if (wave < nrb) {
#pragma unroll
                for (int j = 0; j < NW; j++)
                    if (j <= wave) put(wave, j, acc[0][j]);
            }
        } else {
#pragma unroll
            for (int t = 0; t < RA; t++) {
                const int rb = base + NW * t + wave;
                if (rb < nrb) solve_strip<0>(acc[t], nbc, [&](int j, const V4 &v) { put(rb, j, v); });
            }
        }
    }

    // y(p0 ..) = (b - L(p0.., 0:p0) y) L^{-T}: the right-hand side's row against
    // the panel's images, by the calling wave; t: its values so far
    __device__ __forceinline__ void solve_row(const T *t, int n, int p0)
    {
        const int ncol = min(PW, n - p0), nbc = (ncol + DB - 1) / DB;
        V4 acc[NW];
#pragma unroll
        for (int j = 0; j < NW; j++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                // columns past n count as zero
                const int c = DB * j + MF<T>::row(q, fk);
                acc[j][q] = c < ncol ? t[min(c, ncol - 1)] : T(0);
            }
        solve_strip<0>(acc, nbc, [&](int j, const V4 &v) {
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int c = p0 + DB * j + MF<T>::row(q, fk);
                if (fr == 0 && c < n) sh.ys[c] = v[q];
            }
        });
    }

    // factor; y = L^{-1} b into sh.ys when b; 0 or the first bad column
    __device__ __forceinline__ int factor(T *__restrict__ A, int n, const T *__restrict__ b)
    {
        for (int p0 = 0; p0 < n; p0 += PW) {
            const int nrb = (n - p0 + DB - 1) / DB;          // block rows
            if constexpr (MULTI) {
                if (p0 > 0) {
                    pass<1, true, false>(A, n, b, p0, 0, nrb);
                    __syncthreads();
                }
            }
            const int f = diag_factor<T, NW, NW>(
                A + (int64_t)p0 * n + p0, min(PW, n - p0), n, sh.ds, [&](int i, int j) { return limg(i, j); },
                [&](int p) { return sh.w[p]; });
            if (f) return p0 + f;
            if constexpr (MULTI) {
                int base = NW;
                if (p0 == 0) {
                    for (; base < nrb; base += NW) pass<1, false, true>(A, n, b, p0, base, nrb);
                } else {
                    for (; base + NW < nrb; base += NW * RT) pass<RT, true, true>(A, n, b, p0, base, nrb);
                    if (base < nrb) pass<1, true, true>(A, n, b, p0, base, nrb);
                }
            }
            // (the wave that has the fewest rows in the last pass)
            if (b && wave == NW - 1) solve_row(p0 > 0 ? sh.ts : b + p0, n, p0);
            __syncthreads();
        }
        return 0;
    }

    // acc -= L(rows, 0:p0) L(p0.., 0:p0)^T; on: this wave has rows.  ROW: also
    // sh.ts = b(p0..) - L(p0.., 0:p0) y, from the staged rows.
    // One step ahead: the loads of the next stage are in flight while a stage
    // is multiplied; in FP64 with one block row a wave (half the products, and
    // one workgroup a CU) two.
    template <int RA, bool ROW>
    __device__ __forceinline__ void left_update(const T *__restrict__ A, int lda, int n, int p0, bool on,
                                                V4 (&acc)[RA][NW], const T *const (&src)[RA], const T *__restrict__ b)
    {
        constexpr int EPT = PW * BKC / (64 * NW);            // staged elements of a thread
        constexpr int KS = 64 * NW / PW;                     // columns staged at a time
        constexpr int D = RA == 1 && sizeof(T) == 8 ? 2 : 1; // stages ahead
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));                        // offsets recomputed here, not held by the caller
        const int sc = tid % PW, sk = tid / PW;              // row of the panel, first column
        const T *bp = A + min(p0 + sc, n - 1);
        const int nst = p0 / BKC;                            // a multiple of PW / BKC
        T rb[D][EPT], a[D + 1][RA][4], dot = T(0);
        auto load_b = [&](int st, T *x) {
#pragma unroll
            for (int e = 0; e < EPT; e++) x[e] = bp[(st * BKC + sk + e * KS) * lda];
        };
        auto store_b = [&](int buf, const T *x) {
#pragma unroll
            for (int e = 0; e < EPT; e++) sh.bs[buf][sk + e * KS][sc] = x[e];
        };
        auto load_a = [&](int st, T (*x)[4]) {
#pragma unroll
            for (int t = 0; t < RA; t++)
#pragma unroll
                for (int s = 0; s < 4; s++) x[t][s] = src[t][(st * BKC + 4 * s + fk) * lda];
        };
        load_b(0, rb[0]);
        load_a(0, a[0]);
        if constexpr (D > 1) {
            if (nst > 1) load_a(1, a[1]);
        }
        store_b(0, rb[0]);
        if constexpr (D > 1) {
            if (nst > 1) load_b(1, rb[1]);
        }
        __syncthreads();
        // stage st from LDS half st % 2 and operand set st % (D + 1); stage
        // st + D is loaded meanwhile
        auto stage = [&](int st, auto ub, auto ua) {
            constexpr int buf = decltype(ub)::value, set = decltype(ua)::value;
            if (st + D < nst) {
                load_b(st + D, rb[(buf + D) % D]);
                if (on) load_a(st + D, a[(set + D) % (D + 1)]);
            }
            if (on) {
#pragma unroll
                for (int s = 0; s < 4; s++) {
                    T bf[NW];
#pragma unroll
                    for (int j = 0; j < NW; j++) bf[j] = sh.bs[buf][4 * s + fk][DB * j + fr];
#pragma unroll
                    for (int j = 0; j < NW; j++)
#pragma unroll
                        for (int t = 0; t < RA; t++) acc[t][j] = MF<T>::mfma(bf[j], -a[set][t][s], acc[t][j]);
                }
            }
            if (ROW && b) {
#pragma unroll
                for (int e = 0; e < EPT; e++)
                    dot += sh.bs[buf][sk + e * KS][sc] * sh.ys[st * BKC + sk + e * KS];
            }
            if (st + 1 < nst) store_b(buf ^ 1, rb[(buf + 1) % D]);
            __syncthreads();
        };
        typedef std::integral_constant<int, 0> I0;
        typedef std::integral_constant<int, 1> I1;
        typedef std::integral_constant<int, 2> I2;
        if constexpr (D == 1) {
            for (int st = 0; st < nst; st += 2) {
                stage(st, I0(), I0());
                stage(st + 1, I1(), I1());
            }
        } else {
            for (int st = 0; st < nst;) {
                stage(st++, I0(), I0());
                stage(st++, I1(), I1());
                if (st >= nst) break;
                stage(st++, I0(), I2());
                stage(st++, I1(), I0());
                if (st >= nst) break;
                stage(st++, I0(), I1());
                stage(st++, I1(), I2());
            }
        }
        if (ROW && b) {
            sh.red[sk][sc] = dot;
            __syncthreads();
            if (sk == 0) {
                T t = p0 + sc < n ? b[p0 + sc] : T(0);
#pragma unroll
                for (int e = 0; e < KS; e++) t -= sh.red[e][sc];
                sh.ts[sc] = t;
            }
        }
    }

    // images of -L and W of the panel at p0 (ncol == PW), from memory
    __device__ __forceinline__ void load_images(const T *__restrict__ A, int lda, int p0)
    {
        for (int u = wave; u < NW * (NW - 1) / 2; u += NW) {
            int i = 1, j = u;
            while (j >= i) { j -= i; i++; }
            T *img = limg(i, j);
#pragma unroll
            for (int s = 0; s < 4; s++)
                img[64 * s + lane] = -A[(p0 + DB * j + MF<T>::row(s, fk)) * lda + p0 + DB * i + fr];
        }
        T v[DB], x[DB];
        T d = T(1);
        const int c0 = p0 + DB * wave;
#pragma unroll
        for (int c = 0; c < DB; c++) {
            v[c] = A[(c0 + c) * lda + c0 + fr];
            x[c] = fr == c ? T(1) : T(0);
            d = fr == c ? v[c] : d;
        }
        invert_rows(v, x, T(1) / d, std::make_integer_sequence<int, DB>());
        put_w(wave, x);
    }

    // x = L^{-T} y, y and x in sh.ys; the last panel's images are in LDS
    __device__ __forceinline__ void backward(const T *__restrict__ A, int n)
    {
        const int lda = n, last = (n - 1) / PW * PW;
        for (int p0 = last; p0 >= 0; p0 -= PW) {
            refresh();
            const int ncol = min(PW, n - p0), nbc = (ncol + DB - 1) / DB;
            if (MULTI && p0 < last) {
                load_images(A, lda, p0);
                // t = y - L(p0 + PW.., panel)^T x: wave w the columns of block w
                const T *Lc = A + (int64_t)(p0 + DB * wave) * lda;
                T s[DB];
#pragma unroll
                for (int c = 0; c < DB; c++) s[c] = T(0);
                for (int r = p0 + PW; r < n; r += 64) {
                    const int rr = min(r + lane, n - 1);
                    const T xr = r + lane < n ? sh.ys[rr] : T(0);
                    T l[DB];
#pragma unroll
                    for (int c = 0; c < DB; c++) l[c] = Lc[c * lda + rr];
#pragma unroll
                    for (int c = 0; c < DB; c++) s[c] += l[c] * xr;
                }
                T mine = T(0);
#pragma unroll
                for (int c = 0; c < DB; c++) {
                    T t = row_sum(s[c]);
                    t += __shfl_xor(t, 16);
                    t += __shfl_xor(t, 32);
                    mine = fr == c ? t : mine;
                }
                if (fk == 0) sh.ts[DB * wave + fr] = sh.ys[p0 + DB * wave + fr] - mine;
                __syncthreads();
            }
            const T *t0 = MULTI && p0 < last ? sh.ts : sh.ys + p0;
            if (wave == 0) {
                // x_p = W_p^T (t_p - sum_{i > p} L(i, p)^T x_i): lane (fr, fk)
                // holds element fr of a block in every fk
                T xb[NW];
#pragma unroll
                for (int i = 0; i < NW; i++) xb[i] = T(0);
#pragma unroll
                for (int p = NW - 1; p >= 0; p--) {
                    if (p >= nbc) continue;
                    asm volatile("" : "+v"(lane), "+v"(fr), "+v"(fk));
                    T s[4] = {T(0), T(0), T(0), T(0)};       // column row(q, fk)
#pragma unroll
                    for (int i = p + 1; i < NW; i++)
                        if (i < nbc) {
                            const V4 l = get(limg(i, p));
#pragma unroll
                            for (int q = 0; q < 4; q++) s[q] += l[q] * xb[i];
                        }
                    const V4 w = get_w(p);                   // W(fr, row(q, fk))
                    T tv = T(0);
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        s[q] = row_sum(s[q]);
                        // column fr of the block from the lanes that hold it
                        const T o = __shfl(s[q], MF<T>::lane_of(fr));
                        tv = MF<T>::slice_of(fr) == q ? o : tv;
                    }
                    tv += DB * p + fr < ncol ? t0[DB * p + fr] : T(0);
                    T xv = T(0);
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const T o = __shfl(row_sum(w[q] * tv), MF<T>::lane_of(fr));
                        xv = MF<T>::slice_of(fr) == q ? o : xv;
                    }
                    xb[p] = xv;
                    if (fk == 0 && DB * p + fr < ncol) sh.ys[p0 + DB * p + fr] = xv;
                }
            }
            __syncthreads();
        }
    }
};

template <class T, int NW, int RT, bool MULTI, int OCC>
__global__ __launch_bounds__(64 * NW, OCC) void k_posv_batched(int count, const int *__restrict__ order,
                                                              const int *__restrict__ nsz,
                                                              const int64_t *__restrict__ aoff,
                                                              const int64_t *__restrict__ boff, T *__restrict__ A,
                                                              T *__restrict__ B, int *__restrict__ info,
                                                              int *__restrict__ counter)
{
    __shared__ __align__(16) BShared<T, NW, MULTI> sh;
    Batch<T, NW, RT, MULTI> bt(sh);
    for (;;) {
        if (threadIdx.x == 0) {
            sh.idx = atomicAdd(counter, 1);
            sh.ds.fail = 0;
        }
        __syncthreads();
        const int q = sh.idx;
        if (q >= count) {
            // every workgroup takes one number past the end, the last of them
            // the one below, and leaves the queue as it was found: empty
            if (threadIdx.x == 0 && q == count + (int)gridDim.x - 1) atomicExch(counter, 0);
            break;
        }
        const int m = order[q];
        const int n = nsz[m];
        T *Am = A + aoff[m];
        T *b = B ? B + boff[m] : nullptr;
        const int f = bt.factor(Am, n, b);
        if (threadIdx.x == 0) info[m] = f;
        if (f == 0 && b) {
            bt.backward(Am, n);
            for (int i = threadIdx.x; i < n; i += 64 * NW) b[i] = sh.ys[i];
        }
        __syncthreads();
    }
}

// Size classes of the queue (largest first): above 128, at most 128, at most 64.
constexpr int BATCH_CLASSES = 3;

}  // namespace

// ---------------------------------------------------------------------------
struct mi_batch_s {
    mi_ctx_t *ctx = nullptr;
    int count = 0;
    std::vector<int> n;
    int64_t a_elems = 0, b_elems = 0;
    int *d_n = nullptr, *d_order = nullptr, *d_info = nullptr;
    int *d_counter = nullptr;                      // of the classes' queues, behind d_order
    int64_t *d_aoff = nullptr, *d_boff = nullptr;
    int first[BATCH_CLASSES + 1] = {0, 0, 0, 0};   // queue positions where the classes begin
    int nsplit = 128, wg_per_cu = 2, cus = 0;      // (nsplit: kept for mi_batch_get_shape only)
    hipEvent_t t2 = nullptr;                       // end of the smaller classes (plans of several classes)
    // captured graph of the largest class, of the last (A, B, type, grid) it ran on
    hipGraphExec_t exec = nullptr;
    hipGraph_t graph = nullptr;
    const void *g_a = nullptr, *g_b = nullptr;
    int g_type = -1, g_wg = -1;
    double last_ms = 0.0;
};

namespace {

void batch_drop_graph(mi_batch_t *p)
{
    if (p->exec) (void)hipGraphExecDestroy(p->exec);
    if (p->graph) (void)hipGraphDestroy(p->graph);
    p->exec = nullptr;
    p->graph = nullptr;
}

// One class: count matrices from queue position q0, at most `wgs` workgroups.
template <class T> int batch_launch(mi_batch_t *p, int cls, int q0, int count, int wgs, T *dA, T *dB, hipStream_t s)
{
    if (count <= 0) return 0;
    const unsigned grid = (unsigned)std::max(1, std::min(count, wgs));
    const int *order = p->d_order + q0;
    int *counter = p->d_counter + cls;
    constexpr bool f64 = sizeof(T) == 8;
    if (cls == 0)
        k_posv_batched<T, 8, 2, true, f64 ? 2 : 4><<<grid, 512, 0, s>>>(count, order, p->d_n, p->d_aoff, p->d_boff, dA,
                                                                        dB, p->d_info, counter);
    else if (cls == 1)
        k_posv_batched<T, 8, 1, false, f64 ? 2 : 4><<<grid, 512, 0, s>>>(count, order, p->d_n, p->d_aoff, p->d_boff, dA, dB,
                                                               p->d_info, counter);
    else
        k_posv_batched<T, 4, 1, false, f64 ? 3 : 4><<<grid, 256, 0, s>>>(count, order, p->d_n, p->d_aoff, p->d_boff, dA, dB,
                                                               p->d_info, counter);
    MI_CHECK(hipGetLastError());
    return 0;
}

int batch_class(int n) { return n > 128 ? 0 : n > 64 ? 1 : 2; }

// All matrices of a class
template <class T> int batch_launch_class(mi_batch_t *p, int cls, T *dA, T *dB, hipStream_t s)
{
    return batch_launch<T>(p, cls, p->first[cls], p->first[cls + 1] - p->first[cls],
                           (cls == 2 ? 2 : 1) * p->wg_per_cu * p->cus, dA, dB, s);
}

// the same kernel launched once per matrix (one workgroup each), in queue
// order: the launch-loop baseline of the persistent launch
template <class T>
int batch_run_loop(mi_batch_t *p, T *dA, T *dB)
{
    mi_ctx_t *c = p->ctx;
    hipStream_t s = c->s_main;
    int rc;
    if (p->count == 0) return 0;
    MI_CHECK(hipEventRecord(c->t0, s));
    for (int q = 0; q < p->count; q++) {
        const int cls = q < p->first[1] ? 0 : q < p->first[2] ? 1 : 2;
        if ((rc = batch_launch<T>(p, cls, q, 1, 1, dA, dB, s))) return rc;
    }
    MI_CHECK(hipEventRecord(c->t1, s));
    if ((rc = mi_synchronize(c))) return rc;
    float ms = 0.f;
    MI_CHECK(hipEventElapsedTime(&ms, c->t0, c->t1));
    p->last_ms = ms;
    c->last_ms = ms;
    return 0;
}

// The largest class on the main stream, as a graph when use_graph, and the
// classes below it beside it on the second stream: a class of a few hundred
// matrices is one wave of workgroups, each as long as its matrix.  Both
// streams are idle when a call begins and waited for before it returns, so
// nothing but the host's wait joins them.  (As a branch of one graph, with
// events between the streams and a kernel that resets the queues, a replay
// took 5 - 25 us longer, and the first call of a plan, or with new arrays,
// another 70 us for the instantiation: 64 FP32 systems of 1 .. 100 120 and 57 us
// a first and a later call, now 58 and 51; 1000 of 8 .. 200 201 and 132, now 117
// and 110.  One class after the other: 100 FP64 systems of 1 .. 200 186 us, now
// 109.)
template <class T> int batch_enqueue(mi_batch_t *p, T *dA, T *dB, int use_graph)
{
    mi_ctx_t *c = p->ctx;
    hipStream_t s = c->s_main;
    const int type = sizeof(T) == 8 ? 0 : 1;
    int big = 0, rc;
    while (p->first[big + 1] == 0) big++;
    MI_CHECK(hipEventRecord(c->t0, s));
    if (!use_graph) {
        if ((rc = batch_launch_class<T>(p, big, dA, dB, s))) return rc;
    } else {
        if (!p->exec || p->g_a != dA || p->g_b != dB || p->g_type != type || p->g_wg != p->wg_per_cu) {
            batch_drop_graph(p);
            MI_CHECK(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
            rc = batch_launch_class<T>(p, big, dA, dB, s);
            hipGraph_t g = nullptr;
            hipError_t e = hipStreamEndCapture(s, &g);
            if (rc) { if (g) (void)hipGraphDestroy(g); return rc; }
            MI_CHECK(e);
            p->graph = g;
            MI_CHECK(hipGraphInstantiate(&p->exec, g, nullptr, nullptr, 0));
            p->g_a = dA;
            p->g_b = dB;
            p->g_type = type;
            p->g_wg = p->wg_per_cu;
        }
        MI_CHECK(hipGraphLaunch(p->exec, s));
    }
    MI_CHECK(hipEventRecord(c->t1, s));
    if (!p->t2) return 0;                          // one class
    for (int cls = big + 1; cls < BATCH_CLASSES; cls++)
        if ((rc = batch_launch_class<T>(p, cls, dA, dB, c->s_panel))) return rc;
    MI_CHECK(hipEventRecord(p->t2, c->s_panel));
    return 0;
}

template <class T>
int batch_run(mi_batch_t *p, T *dA, T *dB, int use_graph)
{
    mi_ctx_t *c = p->ctx;
    if (p->count == 0) return 0;
    const int rc = batch_enqueue<T>(p, dA, dB, use_graph);
    // the wait comes first also after an error: the caller may free its arrays
    const int rs = mi_synchronize(c);
    if (rc || rs) return rc ? rc : rs;
    float ms = 0.f, ms2 = 0.f;
    MI_CHECK(hipEventElapsedTime(&ms, c->t0, c->t1));
    if (p->t2) MI_CHECK(hipEventElapsedTime(&ms2, c->t0, p->t2));
    p->last_ms = std::max(ms, ms2);
    c->last_ms = p->last_ms;
    return 0;
}

template <class T>
int batch_autotune(mi_batch_t *p, const T *dA0, const T *dB0, T *dA, T *dB, int *choice)
{
    mi_ctx_t *c = p->ctx;
    double best = 1e300;
    int bw = p->wg_per_cu, bk = 0;
    for (int w = 1; w <= 2; w++) {
        p->wg_per_cu = w;
        double t = 0.0;
        for (int rep = 0; rep < 2; rep++) {         // the first run warms up
            MI_CHECK(hipMemcpyAsync(dA, dA0, (size_t)p->a_elems * sizeof(T), hipMemcpyDeviceToDevice, c->s_main));
            if (dB) MI_CHECK(hipMemcpyAsync(dB, dB0, (size_t)p->b_elems * sizeof(T), hipMemcpyDeviceToDevice, c->s_main));
            MI_CHECK(hipStreamSynchronize(c->s_main));
            int rc = batch_run<T>(p, dA, dB, 0);
            if (rc) return rc;
            t = p->last_ms;
        }
        if (t < best) { best = t; bw = w; bk = w - 1; }
    }
    p->wg_per_cu = bw;
    if (choice) *choice = bk;
    return 0;
}

uint64_t sm64(uint64_t x)
{
    uint64_t z = x + 0x9E3779B97F4A7C15ULL;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}

}  // namespace

extern "C" {

int mi_batch_sizes(uint64_t seed, int count, int lo, int hi, int *n)
{
    if (count < 0 || lo < 1 || hi < lo) { set_error("bad arguments"); return -2; }
    for (int i = 0; i < count; i++)
        n[i] = lo + (int)(sm64(seed + (uint64_t)i * 0x9E3779B97F4A7C15ULL) % (uint64_t)(hi - lo + 1));
    return 0;
}

int mi_batch_create(mi_ctx_t *c, int count, const int *n, mi_batch_t **plan)
{
    *plan = nullptr;
    if (count < 0) { set_error("bad count"); return -2; }
    for (int i = 0; i < count; i++)
        if (n[i] < 1 || n[i] > BMAX) { set_error("matrix %d: order %d outside [1, %d]", i, n[i], BMAX); return -2; }
    mi_batch_t *p = new mi_batch_t();
    p->ctx = c;
    p->count = count;
    p->n.assign(n, n + count);
    std::vector<int64_t> ao(count), bo(count);
    for (int i = 0; i < count; i++) {
        ao[i] = p->a_elems;
        bo[i] = p->b_elems;
        p->a_elems += (int64_t)n[i] * n[i];
        p->b_elems += n[i];
    }
    std::vector<int> order(count);
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return n[a] > n[b]; });
    for (int cls = 1; cls <= BATCH_CLASSES; cls++) {
        int q = p->first[cls - 1];
        while (q < count && batch_class(n[order[q]]) < cls) q++;
        p->first[cls] = q;
    }
    int dev = 0;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&p->cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (p->cus <= 0) p->cus = 256;
    const size_t m = std::max(1, count);
    hipError_t e = hipSuccess;
    if (e == hipSuccess) e = hipMalloc(&p->d_n, m * sizeof(int));
    if (e == hipSuccess) e = hipMalloc(&p->d_order, (count + BATCH_CLASSES) * sizeof(int));
    if (e == hipSuccess) e = hipMalloc(&p->d_info, m * sizeof(int));
    if (e == hipSuccess) e = hipMalloc(&p->d_aoff, m * sizeof(int64_t));
    if (e == hipSuccess) e = hipMalloc(&p->d_boff, m * sizeof(int64_t));
    int classes = 0;
    for (int cls = 0; cls < BATCH_CLASSES; cls++) classes += p->first[cls + 1] > p->first[cls];
    if (e == hipSuccess && classes > 1) e = hipEventCreate(&p->t2);
    if (e == hipSuccess && count) e = hipMemcpy(p->d_n, n, count * sizeof(int), hipMemcpyHostToDevice);
    order.resize(count + BATCH_CLASSES, 0);          // the queues' counters behind it, at 0
    p->d_counter = p->d_order + count;
    if (e == hipSuccess)
        e = hipMemcpy(p->d_order, order.data(), order.size() * sizeof(int), hipMemcpyHostToDevice);
    if (e == hipSuccess && count) e = hipMemcpy(p->d_aoff, ao.data(), count * sizeof(int64_t), hipMemcpyHostToDevice);
    if (e == hipSuccess && count) e = hipMemcpy(p->d_boff, bo.data(), count * sizeof(int64_t), hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        set_error("mi_batch_create: %s", hipGetErrorString(e));
        mi_batch_destroy(p);
        return -1000 - (int)e;
    }
    *plan = p;
    return 0;
}

int mi_batch_destroy(mi_batch_t *p)
{
    if (!p) return 0;
    batch_drop_graph(p);
    if (p->t2) (void)hipEventDestroy(p->t2);
    (void)hipFree(p->d_n);
    (void)hipFree(p->d_order);
    (void)hipFree(p->d_info);
    (void)hipFree(p->d_aoff);
    (void)hipFree(p->d_boff);
    delete p;
    return 0;
}

int mi_batch_extent(const mi_batch_t *p, int64_t *a_elems, int64_t *b_elems)
{
    *a_elems = p->a_elems;
    *b_elems = p->b_elems;
    return 0;
}

int mi_batch_set_shape(mi_batch_t *p, int nsplit, int wg_per_cu)
{
    if (wg_per_cu < 1 || wg_per_cu > 2) { set_error("workgroups per CU must be 1 or 2"); return -2; }
    p->nsplit = nsplit;
    p->wg_per_cu = wg_per_cu;
    return 0;
}

int mi_batch_get_shape(const mi_batch_t *p, int *nsplit, int *wg_per_cu)
{
    *nsplit = p->nsplit;
    *wg_per_cu = p->wg_per_cu;
    return 0;
}

int mi_dposv_batched(mi_batch_t *p, double *dA, double *dB, int use_graph)
{
    return batch_run<double>(p, dA, dB, use_graph);
}

int mi_sposv_batched(mi_batch_t *p, float *dA, float *dB, int use_graph)
{
    return batch_run<float>(p, dA, dB, use_graph);
}

int mi_dposv_batched_loop(mi_batch_t *p, double *dA, double *dB)
{
    return batch_run_loop<double>(p, dA, dB);
}

int mi_sposv_batched_loop(mi_batch_t *p, float *dA, float *dB)
{
    return batch_run_loop<float>(p, dA, dB);
}

int mi_batch_info(const mi_batch_t *p, int *info)
{
    if (p->count) MI_CHECK(hipMemcpy(info, p->d_info, p->count * sizeof(int), hipMemcpyDeviceToHost));
    return 0;
}

int mi_batch_last_ms(const mi_batch_t *p, double *ms)
{
    *ms = p->last_ms;
    return 0;
}

int mi_dbatch_autotune(mi_batch_t *p, const double *dA0, const double *dB0, double *dA, double *dB, int *choice)
{
    return batch_autotune<double>(p, dA0, dB0, dA, dB, choice);
}

int mi_sbatch_autotune(mi_batch_t *p, const float *dA0, const float *dB0, float *dA, float *dB, int *choice)
{
    return batch_autotune<float>(p, dA0, dB0, dA, dB, choice);
}

}  // extern "C"
