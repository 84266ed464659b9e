// mi_potrf.hip -- tile Cholesky (lower) on gfx950, tiles resident in HBM.
//
// The four task classes of src/zpotrf_L.jdf become, per step k:
//   the panel (mi_panel.hpp)  POTRF(k)       :91-208   and TRSM(m,k), m > k
//                             :214-343: tile column k, 128 columns at a time
//   k_update_*                SYRK(k,m) and   :349-633  C(m,n) -= A(m,k) A(n,k)^T
//                             GEMM(m,n,k)               for every trailing tile
//                             in a column range; SYRK is the m == n case
//                             restricted to the lower triangle.
// The host loop runs the panel of step k+1 on a second stream as soon as
// column k+1 has received its step-k update, so it overlaps the rest of the
// step-k trailing update (look-ahead).
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <type_traits>
#include "mi_common.hpp"
#include "mi_panel.hpp"
#include "mi_update.hpp"
#include "dplasma_mi.h"

using namespace mi;

namespace {

constexpr int PJB = 32;            // panel width inside the diagonal factorization
constexpr int POTRF_THREADS = 512;

// ---------------------------------------------------------------------------
// POTRF(k): factor the n x n diagonal tile A (ld) in place, lower.
// LDS holds the current panel P (rows j0..n-1, PJB columns) column-major with
// row stride RC.  Winv receives, for every 32-column block cb, the inverse of
// the lower-triangular 32x32 diagonal block, column-major 32x32 at
// Winv + cb*1024 (identity-padded past n).
__global__ __launch_bounds__(POTRF_THREADS) void k_potrf_diag(double *__restrict__ A, int n, int ld,
                                                             int RC, int info_base,
                                                             int *__restrict__ d_info,
                                                             double *__restrict__ Winv)
{
    extern __shared__ double smem[];
    double *P = smem;                    // PJB * RC
    double *Wl = smem + PJB * RC;        // 32 x 32 inverse being built
    __shared__ int s_fail;
    const int tid = threadIdx.x, nthr = blockDim.x;
    if (tid == 0) s_fail = 0;
    __syncthreads();

    for (int j0 = 0; j0 < n; j0 += PJB) {
        const int jw = min(PJB, n - j0);
        const int R = n - j0;
        for (int idx = tid; idx < PJB * R; idx += nthr) {
            int c = idx / R, r = idx - c * R;
            P[c * RC + r] = (c < jw) ? A[(int64_t)(j0 + c) * ld + j0 + r] : 0.0;
        }
        __syncthreads();

        // unblocked Cholesky of the jw x jw diagonal block by wave 0 (lane = row)
        if (tid < 64) {
            const int lane = tid;
            for (int c = 0; c < jw; c++) {
                double d = P[c * RC + c];
                if (!(d > 0.0)) {
                    if (lane == 0) s_fail = j0 + c + 1;
                    break;
                }
                d = sqrt(d);
                double lr = 0.0;
                if (lane > c && lane < jw) {
                    lr = P[c * RC + lane] / d;
                    P[c * RC + lane] = lr;
                }
                if (lane == c) P[c * RC + c] = d;
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                if (lane > c && lane < jw)
                    for (int c2 = c + 1; c2 <= lane; c2++) P[c2 * RC + lane] -= lr * P[c * RC + c2];
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            }
        }
        __syncthreads();
        if (s_fail) break;

        // inverse of the diagonal block: lane j < 32 solves L w = e_j
        if (tid < 32) {
            const int j = tid;
            double w[PJB];
#pragma unroll
            for (int i = 0; i < PJB; i++) w[i] = 0.0;
#pragma unroll
            for (int i = 0; i < PJB; i++) {
                if (i < jw) {
                    double s = (i == j) ? 1.0 : 0.0;
#pragma unroll
                    for (int p = 0; p < PJB; p++)
                        if (p < i) s -= P[p * RC + i] * w[p];
                    w[i] = (i >= j) ? s / P[i * RC + i] : 0.0;
                } else {
                    w[i] = (i == j) ? 1.0 : 0.0;
                }
            }
#pragma unroll
            for (int i = 0; i < PJB; i++) Wl[j * 32 + i] = w[i];
        }
        __syncthreads();
        for (int idx = tid; idx < 1024; idx += nthr) Winv[(j0 / PJB) * 1024 + idx] = Wl[idx];

        // panel rows below the diagonal block: x = b L11^{-T}, i.e. x = b W^T
        for (int r = jw + tid; r < R; r += nthr) {
            double b[PJB];
#pragma unroll
            for (int c = 0; c < PJB; c++) b[c] = P[c * RC + r];
#pragma unroll
            for (int c = 0; c < PJB; c++) {
                double s = 0.0;
#pragma unroll
                for (int p = 0; p < PJB; p++)
                    if (p <= c) s += b[p] * Wl[p * 32 + c];
                P[c * RC + r] = (c < jw) ? s : 0.0;
            }
        }
        __syncthreads();
        for (int idx = tid; idx < jw * R; idx += nthr) {
            int c = idx / R, r = idx - c * R;
            if (r >= c) A[(int64_t)(j0 + c) * ld + j0 + r] = P[c * RC + r];
        }

        // trailing update inside the tile: A22 -= P2 P2^T (lower), 4x4 per thread
        const int M2 = R - jw;
        if (M2 > 0) {
            const int T4 = (M2 + 3) >> 2;
            const int ntile = T4 * (T4 + 1) / 2;
            for (int t = tid; t < ntile; t += nthr) {
                int ti = (int)((sqrt(8.0 * t + 1.0) - 1.0) * 0.5);
                while ((ti + 1) * (ti + 2) / 2 <= t) ti++;
                while (ti * (ti + 1) / 2 > t) ti--;
                const int tj = t - ti * (ti + 1) / 2;
                const int r0 = jw + 4 * ti, c0 = jw + 4 * tj;
                double acc[4][4];
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int j = 0; j < 4; j++) acc[i][j] = 0.0;
                for (int p = 0; p < jw; p++) {
                    const double *pc = P + p * RC;
                    double a[4], bb[4];
#pragma unroll
                    for (int i = 0; i < 4; i++) { a[i] = pc[r0 + i]; bb[i] = pc[c0 + i]; }
#pragma unroll
                    for (int i = 0; i < 4; i++)
#pragma unroll
                        for (int j = 0; j < 4; j++) acc[i][j] += a[i] * bb[j];
                }
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const int cc = c0 + j;
                    if (cc >= R) continue;
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const int rr = r0 + i;
                        if (rr < R && rr >= cc) A[(int64_t)(j0 + cc) * ld + j0 + rr] -= acc[i][j];
                    }
                }
            }
        }
        __syncthreads();
    }
    if (tid == 0 && s_fail) atomicCAS(d_info, 0, info_base + s_fail);
}

// ---------------------------------------------------------------------------
// TRSM(m,k) for m = k+1 .. MT-1: C <- C L^{-T}.  Grid: (MT-k-1) tiles x
// ceil(rows/64) strips.  L = diagonal tile (ld NB), Winv = its 32x32
// diagonal-block inverses.  256 threads: row = t % 64, column group g = t / 64
// owns 8 of the 32 columns of the current block.
constexpr int TRSM_ROWS = 64;
__global__ __launch_bounds__(256) void k_trsm_panel(double *__restrict__ T, int N, int NB, int MT, int k,
                                                   const double *__restrict__ Winv, int m0)
{
    __shared__ double Xs[32][TRSM_ROWS + 1];   // X chunk, [p][row]
    __shared__ double Ls[32][33];              // L chunk, [p][col]
    __shared__ double Ys[TRSM_ROWS][33];       // block right-hand side [row][col]
    __shared__ double Ws[32][33];              // inverse of the diagonal block [col][row]
    const int tid = threadIdx.x;
    const int row = tid & 63, g = tid >> 6;
    const int strips = (NB + TRSM_ROWS - 1) / TRSM_ROWS;
    const int m = m0 + blockIdx.x / strips;
    const int strip = blockIdx.x % strips;
    const int rows_m = tile_rows(N, NB, MT, m);
    const int r0 = strip * TRSM_ROWS;
    if (r0 >= rows_m) return;
    const int rv = min(TRSM_ROWS, rows_m - r0);
    double *C = T + tile_index(MT, m, k) * (int64_t)NB * NB + r0;     // strip origin
    const double *L = T + tile_index(MT, k, k) * (int64_t)NB * NB;

    for (int c0 = 0; c0 < NB; c0 += 32) {
        const int cw = min(32, NB - c0);
        double acc[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int c = g * 8 + j;
            acc[j] = (row < rv && c < cw) ? C[(int64_t)(c0 + c) * NB + row] : 0.0;
        }
        for (int p0 = 0; p0 < c0; p0 += 32) {
            __syncthreads();
            for (int idx = tid; idx < 32 * TRSM_ROWS; idx += 256) {
                int p = idx / TRSM_ROWS, r = idx % TRSM_ROWS;
                Xs[p][r] = (r < rv) ? C[(int64_t)(p0 + p) * NB + r] : 0.0;
            }
            for (int idx = tid; idx < 32 * 32; idx += 256) {
                int p = idx / 32, c = idx % 32;
                Ls[p][c] = (c < cw) ? L[(int64_t)(p0 + p) * NB + c0 + c] : 0.0;
            }
            __syncthreads();
#pragma unroll 8
            for (int p = 0; p < 32; p++) {
                const double x = Xs[p][row];
#pragma unroll
                for (int j = 0; j < 8; j++) acc[j] -= x * Ls[p][g * 8 + j];
            }
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 8; j++) Ys[row][g * 8 + j] = acc[j];
        for (int idx = tid; idx < 1024; idx += 256) {
            int col = idx / 32, r = idx % 32;
            Ws[col][r] = Winv[(c0 / 32) * 1024 + idx];   // W(r, col)
        }
        __syncthreads();
        // X(row, c) = sum_{p<=c} Y(row, p) W(c, p)
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int c = g * 8 + j;
            double s = 0.0;
            for (int p = 0; p <= c; p++) s += Ys[row][p] * Ws[p][c];
            if (row < rv && c < cw) C[(int64_t)(c0 + c) * NB + row] = s;
        }
    }
}

// ---------------------------------------------------------------------------
// Trailing update on MFMA: C(m,n) -= A(m,k) A(n,k)^T for tile columns n in
// [n_begin, n_end), rows m in [n, MT).  One workgroup = one BMX x BMX block of
// one tile.
constexpr int BM = 128, BK = 16;

// workgroup L of an update launch -> tile (m, n) and its 128x128 block
// (bm, bn); tiles enumerated column by column from column n_begin, whose
// first m_off tiles (rows n_begin .. n_begin+m_off-1) are skipped; the grid
// size decides how many tiles a launch covers
__device__ inline void decode_block(int L, int nsub, int n_begin, int m_off, int MT, int *m, int *n,
                                    int *bm, int *bn)
{
    const int per_tile = nsub * nsub;
    int t = L / per_tile;
    const int s = L - t * per_tile;
    int nn = n_begin, m0 = n_begin + m_off;
    while (t >= MT - m0) { t -= MT - m0; nn++; m0 = nn; }
    *n = nn;
    *m = m0 + t;
    *bm = s / nsub;
    *bn = s - (*bm) * nsub;
}

// One block of 32 WR rows and columns by WR x 2 waves: C(r_base.., c_base..) -= A(r_base.., 0:K)
// B(c_base.., 0:K)^T, all of them column-major with leading dimension NB;
// rows_m / cols_n bound the rows of A and C / the rows of B and columns of C;
// diag: only row >= column.  For tiles that update_block_lds does not take:
// any leading dimension, K and alignment.
//
// Loads are unconditional, from addresses clamped into the tile: rows past
// the matrix only reach parts of C that are not stored, and both operands are
// zeroed past K (0 times an infinity would not be 0).  Operands wait in registers RING stages ahead, so that a short K (a
// tile of 93 columns is six stages) is not a chain of memory latencies; C is
// loaded with the first of them and waits in registers.  PAIR: even NB and
// aligned pairs of rows, two a load.
// dpotrf N = 378, NB = 93: 13.2 us a launch with masked loads one stage ahead
// and C loaded at the end, 9.5 us with this (6.4 in blocks of 32); N = 3900, NB =
// 367 2.09 -> 1.83 ms in FP64, 1.66 -> 1.33 ms in FP32.
//
// The products add up from zero and meet C once: as the MFMAs' start, C would
// round at its own size every four columns (factor of N = 513, NB = 130 with a
// dominant diagonal, error in units of the type's eps: FP64 4.6 against 2.3,
// FP32 7.3 against 2.6).
constexpr int RING = 3;
template <class T, bool PAIR, int WR>
__device__ __forceinline__ void update_block(const T *Ap, const T *Bp, T *Cp, int NB, int K, int rows_m, int cols_n,
                                             int r_base, int c_base, bool diag)
{
    constexpr int BMX = 32 * WR, WC = 2;
    // rows padded by 128 bytes: the four lane groups of a fragment read (k
    // rows 4s + l/16) then fall on alternating halves of the LDS banks
    constexpr int LP = BMX + 128 / (int)sizeof(T);
    constexpr int NT = 64 * WR * WC;                  // threads
    __shared__ T As[2][BK][LP];
    __shared__ T Bs[2][BK][LP];
    typedef typename MF<T>::v4 V4;
    typedef typename MF<T>::v2 V2;
    constexpr int HR = BMX / WR, HC = BMX / WC;       // rows / columns per wave
    constexpr int TR = HR / 16, TC = HC / 16;         // 16x16 MFMA tiles per wave
    constexpr int W = PAIR ? 2 : 1;                   // rows of a load
    typedef T VW __attribute__((ext_vector_type(W)));
    constexpr int SP = BK * BMX / W / NT;             // loads per thread, operand and stage
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave / WC, wn = wave % WC;
    const int fr = lane & 15, fk = lane >> 4;

    // load e = tid + NT i of a stage: k row kk, rows r .. r + W - 1
    constexpr int LR = BMX / W;
    const int kk0 = tid / LR, r = (tid % LR) * W;     // kk = kk0 + (NT / LR) i
    const int last_a = PAIR ? (rows_m - 1) & ~1 : rows_m - 1, last_b = PAIR ? (cols_n - 1) & ~1 : cols_n - 1;
    const T *ap = Ap + min(r_base + r, last_a), *bp = Bp + min(c_base + r, last_b);
    VW ra[RING][SP], rb[RING][SP];
    auto gload = [&](VW (&xa)[SP], VW (&xb)[SP], int st) {
#pragma unroll
        for (int i = 0; i < SP; i++) {
            const int64_t o = (int64_t)min(st * BK + kk0 + (NT / LR) * i, K - 1) * NB;
            xa[i] = *(const VW *)(ap + o);
            xb[i] = *(const VW *)(bp + o);
        }
    };
    auto lstore = [&](const VW (&xa)[SP], const VW (&xb)[SP], int st) {
#pragma unroll
        for (int i = 0; i < SP; i++) {
            const int kk = kk0 + (NT / LR) * i;
            const bool in = st * BK + kk < K;
            *(VW *)&As[st & 1][kk][r] = in ? -xa[i] : VW(T(0));      // -A: the MFMA accumulates -A B^T
            *(VW *)&Bs[st & 1][kk][r] = in ? xb[i] : VW(T(0));
        }
    };
    const int nstage = (K + BK - 1) / BK;
#pragma unroll
    for (int u = 0; u < RING; u++) gload(ra[u], rb[u], u);

    // MFMA row tiles 0 and 1 of a wave interleave their rows: row i of tile t
    // is row 2i + t of the wave's rows.  Fed (B, A), element q of lane l holds
    // row 2 (l % 16) + t and column row(q, l / 16) of each 16x16 tile.
    V4 acc[TR][TC], cv[TR][TC];
    const int row0 = r_base + wm * HR + 2 * fr, col0 = c_base + wn * HC;
    const int cr = min(row0, last_a);
#pragma unroll
    for (int j = 0; j < TC; j++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const T *c = &Cp[(int64_t)min(col0 + j * 16 + MF<T>::row(q, fk), cols_n - 1) * NB + cr];
            if constexpr (PAIR) {
                const V2 v = *(const V2 *)c;
                cv[0][j][q] = v.x;
                cv[1][j][q] = v.y;
            } else {
                cv[0][j][q] = c[0];
                cv[1][j][q] = c[cr + 1 < rows_m ? 1 : 0];
            }
        }
#pragma unroll
    for (int i = 0; i < TR; i++)
#pragma unroll
        for (int j = 0; j < TC; j++) acc[i][j] = V4{T(0), T(0), T(0), T(0)};
    auto stage = [&](VW (&xa)[SP], VW (&xb)[SP], int st) {
        // one barrier a stage: a wave that stores stage st has passed the
        // barrier of stage st - 1, which no wave reaches before it is done
        // with stage st - 2
        lstore(xa, xb, st);
        __syncthreads();
        gload(xa, xb, st + RING);
#pragma unroll
        for (int kq = 0; kq < BK / 4; kq++) {
            T b[TC];
            const V2 v = *(const V2 *)&As[st & 1][kq * 4 + fk][wm * HR + 2 * fr];
            const T a[TR] = {v.x, v.y};
#pragma unroll
            for (int j = 0; j < TC; j++) b[j] = Bs[st & 1][kq * 4 + fk][wn * HC + j * 16 + fr];
#pragma unroll
            for (int i = 0; i < TR; i++)
#pragma unroll
                for (int j = 0; j < TC; j++) acc[i][j] = MF<T>::mfma(b[j], a[i], acc[i][j]);   // C^T: lanes walk rows
        }
    };
    for (int st = 0; st < nstage; st += RING) {
#pragma unroll
        for (int u = 0; u < RING; u++)
            if (st + u < nstage) stage(ra[u], rb[u], st + u);
    }

#pragma unroll
    for (int j = 0; j < TC; j++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int col = col0 + j * 16 + MF<T>::row(q, fk);
#pragma unroll
            for (int t = 0; t < TR; t++) {
                const int rr = row0 + t;
                if (rr < rows_m && col < cols_n && (!diag || rr >= col))
                    Cp[(int64_t)col * NB + rr] = cv[t][j][q] + acc[t][j][q];
            }
        }
}

// workgroup id -> position in the launch's list of blocks: consecutive ids
// land on different XCDs (round-robin), so each XCD is given a contiguous
// range of blocks; the blocks of one tile then share their A/B panels in
// that XCD's L2
__device__ __forceinline__ int xcd_block()
{
    const int G = gridDim.x, bid = blockIdx.x;
    const int G8 = (G / 8) * 8;
    return (bid < G8) ? (bid % 8) * (G8 / 8) + bid / 8 : bid;
}

// The whole tiles' update, and inside tile column k, after its columns c0 ..
// c0 + w - 1 are solved, that of the columns from c0 + w on (K = w): X the
// solved rows of each tile, X_k those of tile (k, k).  Of the latter's blocks
// the first g0 block rows are those of tile (k, k) below c0 + w (lower part),
// then gr block rows of each tile m0, m0 + 1, ...; nc blocks a block row.
struct UpdArgs {
    int N, NB, MT, k;
    int n_begin, m_off, nsub;                      // whole tiles
    int c0, w, g0, gr, nc, m0;                     // panel (w > 0)
    int prio;                                      // wave priority (on the chain of panels: above the bulk)
};
// Workgroup -> block; false: nothing to do.
__device__ __forceinline__ bool update_decode(const UpdArgs &u, int BMX, int *m, int *n, int *r_base, int *c_base,
                                              int *rows_m, int *cols_n, bool *diag)
{
    const int L = xcd_block();
    if (u.w > 0) {
        const int rb = L / u.nc, bn = L - rb * u.nc;
        const bool own = rb < u.g0;
        if (own && rb < bn) return false;
        *m = own ? u.k : u.m0 + (rb - u.g0) / u.gr;
        *n = u.k;
        *r_base = own ? u.c0 + u.w + BMX * rb : BMX * ((rb - u.g0) % u.gr);
        *c_base = u.c0 + u.w + BMX * bn;
        *diag = own && rb == bn;
    } else {
        int bm, bn;
        decode_block(L, u.nsub, u.n_begin, u.m_off, u.MT, m, n, &bm, &bn);
        if (*m == *n && bm < bn) return false;     // strictly upper blocks of a diagonal tile
        *r_base = bm * BMX;
        *c_base = bn * BMX;
        *diag = *m == *n && bm == bn;
    }
    *rows_m = tile_rows(u.N, u.NB, u.MT, *m);
    *cols_n = tile_rows(u.N, u.NB, u.MT, *n);
    return *r_base < *rows_m && *c_base < *cols_n;
}

// operands staged through registers: any leading dimension and alignment
template <class T, bool PAIR, int WR>
__global__ __launch_bounds__(128 * WR, 2) void k_update_mfma(T *__restrict__ Tt, UpdArgs u)
{
    int m, n, r_base, c_base, rows_m, cols_n;
    bool diag;
    if (u.prio) __builtin_amdgcn_s_setprio(2);
    if (!update_decode(u, 32 * WR, &m, &n, &r_base, &c_base, &rows_m, &cols_n, &diag)) return;
    const int64_t sz = (int64_t)u.NB * u.NB, off = (int64_t)u.c0 * u.NB;
    update_block<T, PAIR, WR>(Tt + tile_index(u.MT, m, u.k) * sz + off, Tt + tile_index(u.MT, n, u.k) * sz + off,
                          Tt + tile_index(u.MT, m, n) * sz, u.NB, u.w > 0 ? u.w : u.NB, rows_m, cols_n, r_base, c_base,
                          diag);
}

// operands straight into LDS (mi_update.hpp)
template <class S, class T, int OCC>
__global__ __launch_bounds__(S::NT, OCC) void k_update_lds(T *__restrict__ Tt, UpdArgs u)
{
    __shared__ __align__(1024) unsigned char lds[S::LDS];
    int m, n, r_base, c_base, rows_m, cols_n;
    bool diag;
    if (u.prio) __builtin_amdgcn_s_setprio(2);
    if (!update_decode(u, S::BM, &m, &n, &r_base, &c_base, &rows_m, &cols_n, &diag)) return;
    const int64_t sz = (int64_t)u.NB * u.NB, off = (int64_t)u.c0 * u.NB;
    update_block_lds<S, T>(lds, Tt + tile_index(u.MT, m, u.k) * sz + off, Tt + tile_index(u.MT, n, u.k) * sz + off,
                           Tt + tile_index(u.MT, m, n) * sz, u.NB, u.w > 0 ? u.w : u.NB, rows_m, cols_n, r_base,
                           c_base, diag);
}
// Shapes, by the step-0 update of N = 32768, NB = 512 (1953 tiles) alone, all
// with the C vectors taken in over the last stages (over the first: as fast or
// 0.5% faster in a factorization; register-staged before: FP64 64.8 TF, FP32
// 121 TF; a library product of 16384 reaches 74 and 153 TF):
//   FP64  2 x 4 waves, BK 16 x 2: 69.7 TF; BK 8 x 4: 68.1; 2 x 2 waves, BK 8
//         x 4: 68.2
//   FP32  2 x 2 waves, BK 16 x 4: 130 TF; x 3 and three workgroups a CU: 123;
//         BK 16 x 2 and four: 120; BK 32 x 2: 126
// and of N = 4096, NB = 256 (64 x 64 blocks, 37.3 / 58.5 TF before): BK 16 x
// 3: 41.3 / 62.6 TF, x 4: 39.6 / 61.2, BK 8 x 8: 38.3 / 60.9.
//
// A launch of at most 256 blocks of 64 x 64 leaves CUs idle and the others on
// a chain of K / 16 stages: 32 x 32 blocks instead (dpotrf N = 4096, NB = 256
// 1.67 -> 1.57 ms; posv N = 6000, NB = 512 4.20 -> 4.07 ms; 128 blocks 1.57 and
// 4.15, 600 1.56 and 3.98, but FP32 N = 3200 2.41 -> 2.43 from 400 on).
constexpr int64_t TINY_BLOCKS = 256;
template <class T> struct UpdShapes;
template <> struct UpdShapes<double> {
    typedef UpdShape<double, 128, 2, 4, 16, 2, 2, 2> big;
    typedef UpdShape<double, 64, 2, 2, 16, 3, 2, 2> small;
    typedef UpdShape<double, 32, 2, 2, 32, 3, 1, 2> tiny;
    static constexpr int occ = 4;
};
template <> struct UpdShapes<float> {
    typedef UpdShape<float, 128, 2, 2, 16, 4, 4, 4> big;
    typedef UpdShape<float, 64, 2, 2, 16, 3, 2, 2> small;
    typedef UpdShape<float, 32, 2, 2, 32, 3, 1, 2> tiny;
    static constexpr int occ = 2;
};

// ---------------------------------------------------------------------------
// FP32 trailing update on BF16 MFMA with a two-term split of both operands
// (v_mfma_f32_16x16x32_bf16, FP32 accumulation): with a = ah + al, ah =
// bf16(a), al = bf16(a - ah), each product is taken as
//     al bh + ah bl + ah bh            (the al bl term, ~2^-16 relative, dropped)
// so the update carries about 16 significant bits per operand instead of 8,
// at three BF16 MFMAs per product.  Used by the mixed-precision solve, whose
// FP64 refinement recovers the rest.  Work decomposition, XCD grouping
// and SYRK masking as k_update_mfma, C as the MFMAs' start; K in chunks of
// 32, split once per workgroup while staged into LDS as [row][k] bf16 rows
// (row pitch 40 bf16 = 80 B: 16-byte aligned fragment reads, spread banks).
// MFMA operand layout: A(i, k) and B(k, j) for lane l in i (resp. j) = l % 16,
// k = 8 (l / 16) + e, e < 8; result element q at row 4 (l / 16) + q.
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf4 __attribute__((ext_vector_type(4)));
constexpr int XK = 32, XS = XK + 8;

// Epilogue of the BF16-split updates: the TI x 4 accumulator tiles of a wave
// (rows r0 + 16 i + 4 fk + q, columns c0 + 16 j + fr) stored as C (pre:
// C was the MFMA's start; 16-byte stores of four rows) or added to C with
// the tile and lower-triangle masks (diag: a diagonal block).
template <int TI>
__device__ inline void bf16x3_store(float *Cp, int NB, const fx4 (&acc)[TI][4], int r0, int c0, int fr, int fk,
                                    bool pre, int rows_m, int cols_n, bool diag)
{
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int row = r0 + i * 16 + 4 * fk, col = c0 + j * 16 + fr;
            float *c = &Cp[(int64_t)col * NB + row];
            if (pre) {
                *(fx4 *)c = acc[i][j];
            } else {
#pragma unroll
                for (int q = 0; q < 4; q++)
                    if (row + q < rows_m && col < cols_n && (!diag || row + q >= col)) c[q] += acc[i][j][q];
            }
        }
}

__global__ __launch_bounds__(256, 2) void k_update_bf16x3(float *__restrict__ Tt, int N, int NB, int MT, int k,
                                                         int n_begin, int m_off, int nsub)
{
    __shared__ __align__(16) __bf16 Ah[BM * XS];
    __shared__ __align__(16) __bf16 Al[BM * XS];
    __shared__ __align__(16) __bf16 Bh[BM * XS];
    __shared__ __align__(16) __bf16 Bl[BM * XS];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int G = gridDim.x, bid = blockIdx.x;
    const int G8 = (G / 8) * 8;
    const int L = (bid < G8) ? (bid % 8) * (G8 / 8) + bid / 8 : bid;
    int m, n, bm, bn;
    decode_block(L, nsub, n_begin, m_off, MT, &m, &n, &bm, &bn);
    if (m == n && bm < bn) return;
    const int rows_m = tile_rows(N, NB, MT, m);
    const int cols_n = tile_rows(N, NB, MT, n);
    const int r_base = bm * BM, c_base = bn * BM;
    if (r_base >= rows_m || c_base >= cols_n) return;
    const bool full = (r_base + BM <= rows_m) && (c_base + BM <= cols_n) && (NB % XK == 0);
    const float *Ap = Tt + tile_index(MT, m, k) * (int64_t)NB * NB;
    const float *Bp = Tt + tile_index(MT, n, k) * (int64_t)NB * NB;
    float *Cp = Tt + tile_index(MT, m, n) * (int64_t)NB * NB;
    const int fr = lane & 15, fk = lane >> 4;

    // element q of acc[i][j] in lane (fr, fk): C(row 4 fk + q of row tile i,
    // column fr of column tile j), four consecutive rows of one column
    fx4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = fx4{0.f, 0.f, 0.f, 0.f};
    const bool pre = full && !((m == n) && (bm == bn));
    if (pre) {
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 4; j++)
                acc[i][j] = *(const fx4 *)&Cp[(int64_t)(c_base + wn * 64 + j * 16 + fr) * NB + r_base + wm * 64 +
                                              i * 16 + 4 * fk];
    }

    // staging: thread (rq, kq) = (tid % 32, tid / 32) holds rows rq + 32 i
    // (i < 4) at k = k0 + 4 kq + u (u < 4) of both operands
    const int rq = tid & 31, kq = tid >> 5;
    float ra[4][4], rb[4][4];                    // [i][u]
    auto gload = [&](int k0) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int kg = k0 + 4 * kq + u;
            const float *ac = Ap + (int64_t)kg * NB + r_base + rq;
            const float *bc = Bp + (int64_t)kg * NB + c_base + rq;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                if (full) {
                    ra[i][u] = ac[32 * i];
                    rb[i][u] = bc[32 * i];
                } else {
                    const bool kin = kg < NB;
                    ra[i][u] = (kin && r_base + rq + 32 * i < rows_m) ? ac[32 * i] : 0.f;
                    rb[i][u] = (kin && c_base + rq + 32 * i < cols_n) ? bc[32 * i] : 0.f;
                }
            }
        }
    };
    auto split_store = [&](__bf16 *H, __bf16 *Lo, const float (&v)[4], int row, float sign) {
        bf4 h, l;
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const float x = sign * v[u];
            const __bf16 xh = (__bf16)x;
            h[u] = xh;
            l[u] = (__bf16)(x - (float)xh);
        }
        *(bf4 *)&H[row * XS + 4 * kq] = h;
        *(bf4 *)&Lo[row * XS + 4 * kq] = l;
    };
    auto lstore = [&]() {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            split_store(Ah, Al, ra[i], rq + 32 * i, -1.f);   // -A: the MFMA accumulates C - A B^T
            split_store(Bh, Bl, rb[i], rq + 32 * i, 1.f);
        }
    };

    const int nstage = (NB + XK - 1) / XK;
    gload(0);
    for (int st = 0; st < nstage; st++) {
        lstore();
        __syncthreads();
        if (st + 1 < nstage) gload((st + 1) * XK);
        bf8 ah[4], al[4], bh[4], bl[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int row = wm * 64 + i * 16 + fr;
            ah[i] = *(const bf8 *)&Ah[row * XS + 8 * fk];
            al[i] = *(const bf8 *)&Al[row * XS + 8 * fk];
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int row = wn * 64 + j * 16 + fr;
            bh[j] = *(const bf8 *)&Bh[row * XS + 8 * fk];
            bl[j] = *(const bf8 *)&Bl[row * XS + 8 * fk];
        }
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[i], bh[j], acc[i][j], 0, 0, 0);
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[i], bl[j], acc[i][j], 0, 0, 0);
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[i], bh[j], acc[i][j], 0, 0, 0);
            }
        __syncthreads();
    }
    bf16x3_store(Cp, NB, acc, r_base + wm * 64, c_base + wn * 64, fr, fk, pre, rows_m, cols_n, (m == n) && (bm == bn));
}

// ---------------------------------------------------------------------------
// The BF16 two-term split of panel column k, once per step instead of once
// per workgroup and K chunk of the update: tile (m, k), m >= m0, is written
// to P as its hi and lo BF16 images (NB x NB each; rows past the tile's
// last row are zero) in chunk-major order [k / 32][row][k % 32], so that
// the update's staging of one 32-wide K chunk of 128 rows reads 8 KB of
// consecutive bytes (whole cache lines) and does no conversion work.  One
// workgroup per 64 x 64 block of a tile, transposed through LDS.
constexpr int SPT = 64;
__global__ __launch_bounds__(256) void k_split_panel(const float *__restrict__ Tt, int N, int NB, int MT, int k,
                                                     int m0, __bf16 *__restrict__ P)
{
    __shared__ float sb[SPT][SPT + 1];
    const int nb = (NB + SPT - 1) / SPT;
    const int per = nb * nb;
    const int t = blockIdx.x / per, s = blockIdx.x - t * per;
    const int m = m0 + t;
    const int bk = s / nb, br = s - bk * nb;       // block of K columns, block of rows
    const int rows = tile_rows(N, NB, MT, m);
    const float *A = Tt + tile_index(MT, m, k) * (int64_t)NB * NB;
    __bf16 *H = P + (int64_t)t * 2 * NB * NB;
    __bf16 *Lo = H + (int64_t)NB * NB;
    const int tid = threadIdx.x;
    for (int e = tid; e < SPT * SPT; e += 256) {   // coalesced along the rows of a column
        const int j = e / SPT, i = e % SPT;
        const int kk = bk * SPT + j, r = br * SPT + i;
        sb[j][i] = (kk < NB && r < rows) ? A[(int64_t)kk * NB + r] : 0.f;
    }
    __syncthreads();
    for (int e = tid; e < SPT * SPT / 2; e += 256) {   // pairs of K, coalesced along a row
        const int i = e / (SPT / 2), j = 2 * (e % (SPT / 2));
        const int kk = bk * SPT + j, r = br * SPT + i;
        if (r < NB && kk < NB) {                   // NB is even here (a multiple of 32)
            const float x0 = sb[j][i], x1 = sb[j + 1][i];
            const __bf16 h0 = (__bf16)x0, h1 = (__bf16)x1;
            typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
            const int64_t o = ((int64_t)(kk / XK) * NB + r) * XK + kk % XK;
            *(bf2 *)&H[o] = bf2{h0, h1};
            *(bf2 *)&Lo[o] = bf2{(__bf16)(x0 - (float)h0), (__bf16)(x1 - (float)h1)};
        }
    }
}

// k_update_bf16x3 on the split panel P (tiles m0.. of column k, as written
// by k_split_panel; NB a multiple of 32).  The A halves are negated on
// their way into LDS (a sign-bit flip: the split of -a is minus the split
// of a), so the MFMAs see exactly the operands of k_update_bf16x3 and the
// result is the same bit for bit.  Staging: thread t holds rows t / 4 and
// t / 4 + 64 at K offset 8 (t % 4) of the four images (A hi, A lo, B hi,
// B lo), for two chunks ahead (two register sets: two waves per SIMD, the
// loads of a chunk in flight over two chunks of MFMA work).  LDS rows are 64 bytes (four 16-byte chunks of eight K values),
// chunk c of row r stored at position c ^ sw(r), sw(r) = ((r >> 1) & 3) ^
// ((r >> 3) & 1): a fragment read (16 rows at one chunk) and a staging
// store (4 rows x 4 chunks) then touch distinct banks in each pass, with
// 32 banks (8 lanes a pass) and with 64 (16 lanes a pass).
__global__ __launch_bounds__(256, 2) void k_update_bf16x3p(float *__restrict__ Tt, int N, int NB, int MT, int k,
                                                          int n_begin, int m_off, int nsub,
                                                          const __bf16 *__restrict__ P, int m0)
{
    __shared__ __align__(16) __bf16 Ah[BM * XK];
    __shared__ __align__(16) __bf16 Al[BM * XK];
    __shared__ __align__(16) __bf16 Bh[BM * XK];
    __shared__ __align__(16) __bf16 Bl[BM * XK];
    auto lds = [](int r, int c) { return r * XK + 8 * (c ^ (((r >> 1) & 3) ^ ((r >> 3) & 1))); };
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int G = gridDim.x, bid = blockIdx.x;
    const int G8 = (G / 8) * 8;
    const int L = (bid < G8) ? (bid % 8) * (G8 / 8) + bid / 8 : bid;
    int m, n, bm, bn;
    decode_block(L, nsub, n_begin, m_off, MT, &m, &n, &bm, &bn);
    if (m == n && bm < bn) return;
    const int rows_m = tile_rows(N, NB, MT, m);
    const int cols_n = tile_rows(N, NB, MT, n);
    const int r_base = bm * BM, c_base = bn * BM;
    if (r_base >= rows_m || c_base >= cols_n) return;
    const bool full = (r_base + BM <= rows_m) && (c_base + BM <= cols_n);
    const int64_t img = (int64_t)NB * NB;
    const __bf16 *AH = P + (int64_t)(m - m0) * 2 * img + (int64_t)r_base * XK;
    const __bf16 *BH = P + (int64_t)(n - m0) * 2 * img + (int64_t)c_base * XK;
    float *Cp = Tt + tile_index(MT, m, n) * (int64_t)NB * NB;
    const int fr = lane & 15, fk = lane >> 4;

    fx4 acc[4][4];                               // as in k_update_bf16x3
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = fx4{0.f, 0.f, 0.f, 0.f};
    const bool pre = full && !((m == n) && (bm == bn));
    if (pre) {
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 4; j++)
                acc[i][j] = *(const fx4 *)&Cp[(int64_t)(c_base + wn * 64 + j * 16 + fr) * NB + r_base + wm * 64 +
                                              i * 16 + 4 * fk];
    }

    typedef unsigned int u4 __attribute__((ext_vector_type(4)));
    auto neg = [](bf8 v) -> bf8 { return __builtin_bit_cast(bf8, __builtin_bit_cast(u4, v) ^ 0x80008000u); };
    const int rq = tid >> 2, kq = tid & 3;
    typedef bf8 Stage[2][4];                     // [row half][A hi, A lo, B hi, B lo]
    Stage sa, sb;
    auto gload = [&](Stage &x, int k0) {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int row = rq + 64 * i;
            const int64_t o = ((int64_t)(k0 / XK) * NB + row) * XK + 8 * kq;
            const bool ain = full || r_base + row < rows_m;
            const bool bin = full || c_base + row < cols_n;
            const bf8 z = bf8{};
            x[i][0] = ain ? *(const bf8 *)(AH + o) : z;
            x[i][1] = ain ? *(const bf8 *)(AH + img + o) : z;
            x[i][2] = bin ? *(const bf8 *)(BH + o) : z;
            x[i][3] = bin ? *(const bf8 *)(BH + img + o) : z;
        }
    };
    auto lstore = [&](const Stage &x) {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int o = lds(rq + 64 * i, kq);
            *(bf8 *)&Ah[o] = neg(x[i][0]);             // -A: the MFMA accumulates C - A B^T
            *(bf8 *)&Al[o] = neg(x[i][1]);
            *(bf8 *)&Bh[o] = x[i][2];
            *(bf8 *)&Bl[o] = x[i][3];
        }
    };
    auto compute = [&]() {
        bf8 ah[4], al[4], bh[4], bl[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int o = lds(wm * 64 + i * 16 + fr, fk);
            ah[i] = *(const bf8 *)&Ah[o];
            al[i] = *(const bf8 *)&Al[o];
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int o = lds(wn * 64 + j * 16 + fr, fk);
            bh[j] = *(const bf8 *)&Bh[o];
            bl[j] = *(const bf8 *)&Bl[o];
        }
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[i], bh[j], acc[i][j], 0, 0, 0);
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[i], bl[j], acc[i][j], 0, 0, 0);
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[i], bh[j], acc[i][j], 0, 0, 0);
            }
    };

    // chunks in pairs: the loads of chunk c + 2 are issued while chunk c
    // is computed (NB / 32 chunks; an odd count ends with a single one)
    const int nstage = NB / XK;
    gload(sa, 0);
    if (nstage > 1) gload(sb, XK);
    for (int st = 0; st < nstage; st += 2) {
        lstore(sa);
        __syncthreads();
        if (st + 2 < nstage) gload(sa, (st + 2) * XK);
        compute();
        __syncthreads();
        if (st + 1 < nstage) {
            lstore(sb);
            __syncthreads();
            if (st + 3 < nstage) gload(sb, (st + 3) * XK);
            compute();
            __syncthreads();
        }
    }

    bf16x3_store(Cp, NB, acc, r_base + wm * 64, c_base + wn * 64, fr, fk, pre, rows_m, cols_n, (m == n) && (bm == bn));
}

// k_update_bf16x3p with 256 x 256 blocks (NB a multiple of 256): half the
// panel operand traffic per flop.  Eight waves as a 2 x 4 grid of 128 x 64;
// the four images' K chunks go straight into LDS by global_load_lds_dwordx4
// (no staging registers), double-buffered in 128 KB (one workgroup per CU).
// A direct load cannot negate, so the B fragments are negated in registers
// instead: (-b) a is the same exact BF16 product as b (-a), so the MFMAs
// sum the same values and the result is that of k_update_bf16x3p bit for
// bit.  Lane l of a wave's load of 16 rows lands at LDS offset 16 l (row
// 16 g + l / 4, slot l % 4), so it fetches K chunk (l % 4) ^ sw(row) of
// that row.  Rows up to r_base + 255 lie inside the NB-row tile image,
// zero past the tile's last row, so no load needs a guard.
typedef __attribute__((address_space(3))) void *lds_ptr;
constexpr int WB = 256;
__global__ __launch_bounds__(512, 1) void k_update_bf16x3w(float *__restrict__ Tt, int N, int NB, int MT, int k,
                                                          int n_begin, int m_off, int nsub,
                                                          const __bf16 *__restrict__ P, int m0)
{
    __shared__ __align__(16) __bf16 S[2][4][WB * XK];     // [buffer][A hi, A lo, B hi, B lo]
    auto sw = [](int r) { return ((r >> 1) & 3) ^ ((r >> 3) & 1); };
    auto lds = [&](int r, int c) { return r * XK + 8 * (c ^ sw(r)); };
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 2, wn = wave & 3;
    const int G = gridDim.x, bid = blockIdx.x;
    const int G8 = (G / 8) * 8;
    const int L = (bid < G8) ? (bid % 8) * (G8 / 8) + bid / 8 : bid;
    int m, n, bm, bn;
    decode_block(L, nsub, n_begin, m_off, MT, &m, &n, &bm, &bn);
    if (m == n && bm < bn) return;
    const int rows_m = tile_rows(N, NB, MT, m);
    const int cols_n = tile_rows(N, NB, MT, n);
    const int r_base = bm * WB, c_base = bn * WB;
    if (r_base >= rows_m || c_base >= cols_n) return;
    const int64_t img = (int64_t)NB * NB;
    const __bf16 *AH = P + (int64_t)(m - m0) * 2 * img + (int64_t)r_base * XK;
    const __bf16 *BH = P + (int64_t)(n - m0) * 2 * img + (int64_t)c_base * XK;
    float *Cp = Tt + tile_index(MT, m, n) * (int64_t)NB * NB;
    const int fr = lane & 15, fk = lane >> 4;

    // Each wave's 128 x 64 lies inside one 128 x 128 block (pr, pc) of
    // k_update_bf16x3p, and takes the path that kernel takes there (C as
    // the MFMA's start, or C += the products), so that both round alike.
    const int pr = r_base + wm * 128, pc = c_base + (wn >> 1) * 128;
    const bool pre = pr + 128 <= rows_m && pc + 128 <= cols_n && !(m == n && pr <= pc);
    fx4 acc[8][4];
#pragma unroll
    for (int i = 0; i < 8; i++)
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int q = 0; q < 4; q++)
                acc[i][j][q] = 0.f;
    if (pre) {
#pragma unroll
        for (int i = 0; i < 8; i++)
#pragma unroll
            for (int j = 0; j < 4; j++)
                acc[i][j] = *(const fx4 *)&Cp[(int64_t)(c_base + wn * 64 + j * 16 + fr) * NB + pr + i * 16 + 4 * fk];
    }
    typedef unsigned int u4 __attribute__((ext_vector_type(4)));
    auto neg = [](bf8 v) -> bf8 { return __builtin_bit_cast(bf8, __builtin_bit_cast(u4, v) ^ 0x80008000u); };
    // wave w fetches rows 32 w .. 32 w + 31 of the four images
    auto dload = [&](int buf, int k0) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int R = wave * 32 + 16 * h, lr = R + (lane >> 2);
            const int lc = (lane & 3) ^ sw(lr);
            const int64_t o = ((int64_t)(k0 / XK) * NB + lr) * XK + 8 * lc;
            __builtin_amdgcn_global_load_lds(AH + o, (lds_ptr)&S[buf][0][R * XK], 16, 0, 0);
            __builtin_amdgcn_global_load_lds(AH + img + o, (lds_ptr)&S[buf][1][R * XK], 16, 0, 0);
            __builtin_amdgcn_global_load_lds(BH + o, (lds_ptr)&S[buf][2][R * XK], 16, 0, 0);
            __builtin_amdgcn_global_load_lds(BH + img + o, (lds_ptr)&S[buf][3][R * XK], 16, 0, 0);
        }
    };
    const int nstage = NB / XK;
    dload(0, 0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    for (int st = 0; st < nstage; st++) {
        const int b = st & 1;
        if (st + 1 < nstage) dload(b ^ 1, (st + 1) * XK);   // into the buffer read at step st - 1
        bf8 bh[4], bl[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int o = lds(wn * 64 + j * 16 + fr, fk);
            bh[j] = neg(*(const bf8 *)&S[b][2][o]);          // -B: the MFMA accumulates C - A B^T
            bl[j] = neg(*(const bf8 *)&S[b][3][o]);
        }
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int o = lds(wm * 128 + i * 16 + fr, fk);
            const bf8 ah = *(const bf8 *)&S[b][0][o], al = *(const bf8 *)&S[b][1][o];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bh[j], acc[i][j], 0, 0, 0);
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bl[j], acc[i][j], 0, 0, 0);
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bh[j], acc[i][j], 0, 0, 0);
            }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // this wave's loads of step st + 1
        __syncthreads();                                      // everyone's, and buffer b read
    }

    bf16x3_store(Cp, NB, acc, pr, c_base + wn * 64, fr, fk, pre, rows_m, cols_n, m == n);
}

// ---------------------------------------------------------------------------
// The same trailing update on the FP64 VALU (engine 0; the MFMA kernel
// above is the default: with two resident waves per SIMD both reach about
// the same FP64 rate on gfx950, and the MFMA kernel needs fewer registers
// per flop).  Work decomposition as k_update_mfma (one
// 128x128 block of one tile per workgroup, XCD-grouped); thread (tx, ty) =
// (t % 16, t / 16) keeps the 8x8 block of rows {32g + 2tx + i} and columns
// {32h + 2ty + j} (g, h < 4, i, j < 2) in registers.  Every k step reads
// four 16-byte A pairs (16 distinct per wave, contiguous: no bank conflict)
// and four B pairs (4 distinct per wave: broadcast) for 64 FMAs.

__global__ __launch_bounds__(256) void k_update_valu(double *__restrict__ T, int N, int NB, int MT, int k,
                                                    int n_begin, int m_off, int nsub)
{
    __shared__ double As[2][BK][BM];
    __shared__ double Bs[2][BK][BM];
    const int tid = threadIdx.x;
    const int tx = tid & 15, ty = tid >> 4;
    const int G = gridDim.x, bid = blockIdx.x;
    const int G8 = (G / 8) * 8;
    const int L = (bid < G8) ? (bid % 8) * (G8 / 8) + bid / 8 : bid;
    int m, n, bm, bn;
    decode_block(L, nsub, n_begin, m_off, MT, &m, &n, &bm, &bn);
    if (m == n && bm < bn) return;
    const int rows_m = tile_rows(N, NB, MT, m);
    const int cols_n = tile_rows(N, NB, MT, n);
    const int r_base = bm * BM, c_base = bn * BM;
    if (r_base >= rows_m || c_base >= cols_n) return;
    const bool full = (r_base + BM <= rows_m) && (c_base + BM <= cols_n) && (NB % BK == 0) && !(NB & 1);

    const double *Ap = T + tile_index(MT, m, k) * (int64_t)NB * NB;
    const double *Bp = T + tile_index(MT, n, k) * (int64_t)NB * NB;
    double *Cp = T + tile_index(MT, m, n) * (int64_t)NB * NB;

    double acc[8][8];
#pragma unroll
    for (int i = 0; i < 8; i++)
#pragma unroll
        for (int j = 0; j < 8; j++) acc[i][j] = 0.0;

    double2 ra[4], rb[4];
    auto gload = [&](int k0) {
        if (full) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int e = tid + 256 * i;
                const int kk = e >> 6, r = (e & 63) * 2;
                ra[i] = *(const double2 *)(Ap + (int64_t)(k0 + kk) * NB + r_base + r);
                rb[i] = *(const double2 *)(Bp + (int64_t)(k0 + kk) * NB + c_base + r);
            }
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int e = tid + 256 * i;
                const int kk = e >> 6, r = (e & 63) * 2;
                const int kg = k0 + kk;
                double a0 = 0.0, a1 = 0.0, b0 = 0.0, b1 = 0.0;
                if (kg < NB) {
                    const double *ac = Ap + (int64_t)kg * NB;
                    const double *bc = Bp + (int64_t)kg * NB;
                    if (r_base + r < rows_m) a0 = ac[r_base + r];
                    if (r_base + r + 1 < rows_m) a1 = ac[r_base + r + 1];
                    if (c_base + r < cols_n) b0 = bc[c_base + r];
                    if (c_base + r + 1 < cols_n) b1 = bc[c_base + r + 1];
                }
                ra[i] = make_double2(a0, a1);
                rb[i] = make_double2(b0, b1);
            }
        }
    };
    auto lstore = [&](int buf) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int e = tid + 256 * i;
            const int kk = e >> 6, r = (e & 63) * 2;
            *(double2 *)&As[buf][kk][r] = ra[i];
            *(double2 *)&Bs[buf][kk][r] = rb[i];
        }
    };

    const int nstage = (NB + BK - 1) / BK;
    gload(0);
    lstore(0);
    __syncthreads();
    for (int st = 0; st < nstage; st++) {
        const int buf = st & 1;
        if (st + 1 < nstage) gload((st + 1) * BK);
#pragma unroll 2
        for (int kk = 0; kk < BK; kk++) {
            double a[8], b[8];
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const double2 va = *(const double2 *)&As[buf][kk][32 * g + 2 * tx];
                const double2 vb = *(const double2 *)&Bs[buf][kk][32 * g + 2 * ty];
                a[2 * g] = va.x;
                a[2 * g + 1] = va.y;
                b[2 * g] = vb.x;
                b[2 * g + 1] = vb.y;
            }
#pragma unroll
            for (int i = 0; i < 8; i++)
#pragma unroll
                for (int j = 0; j < 8; j++) acc[i][j] = fma(a[i], b[j], acc[i][j]);
        }
        if (st + 1 < nstage) lstore(buf ^ 1);
        __syncthreads();
    }

    const bool diag = (m == n) && (bm == bn);
#pragma unroll
    for (int h = 0; h < 4; h++)
#pragma unroll
        for (int jj = 0; jj < 2; jj++) {
            const int col = c_base + 32 * h + 2 * ty + jj;
            double *cc = Cp + (int64_t)col * NB;
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const int row = r_base + 32 * g + 2 * tx;
                if (full && !diag) {
                    double2 c = *(double2 *)(cc + row);
                    c.x -= acc[2 * g][2 * h + jj];
                    c.y -= acc[2 * g + 1][2 * h + jj];
                    *(double2 *)(cc + row) = c;
                } else if (col < cols_n) {
#pragma unroll
                    for (int i = 0; i < 2; i++) {
                        const int rr = row + i;
                        if (rr < rows_m && (!diag || rr >= col)) cc[rr] -= acc[2 * g + i][2 * h + jj];
                    }
                }
            }
        }
}

__global__ void k_fill_int(int *p, int v, int n)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// ---------------------------------------------------------------------------
// panel engine: 0 = VALU diagonal factor / solve (FP64 only), 1 = MFMA panel updates (default)
int g_panel_kernel = 1;
// trailing-update engine: 0 = FP64 VALU, 1 = MFMA (default)
int g_update_kernel = -1;
// FP32 trailing update of mi_spotrf_tiles and the FP32 step launches: 0 =
// FP32 MFMA (default), 1 = BF16 MFMA, two-term split (the mixed solve passes
// its choice as an argument instead)
int g_supdate = 0;
// BF16-split updates of the main stream: 1 = panel column split once per
// step (k_split_panel + k_update_bf16x3p, default), 0 = split by every
// workgroup (k_update_bf16x3)
int g_bf16_panel_split = 1;

// profiler names per precision
template <class T> struct KN;
// (update: launches on the main stream, which never overlap one another;
// update_la: the look-ahead column updates on the panel stream)
template <> struct KN<double> {
    static constexpr const char *potrf = "dpotrf_potrf_diag";
    static constexpr const char *trsm = "dpotrf_trsm_panel";
    static constexpr const char *update = "dpotrf_update";
    static constexpr const char *update_la = "dpotrf_update_la";
    static constexpr const char *panel_update = "dpotrf_panel_update";
};
template <> struct KN<float> {
    static constexpr const char *potrf = "spotrf_potrf_diag";
    static constexpr const char *trsm = "spotrf_trsm_panel";
    static constexpr const char *update = "spotrf_update";
    static constexpr const char *update_la = "spotrf_update_la";
    static constexpr const char *panel_update = "spotrf_panel_update";
    static constexpr const char *update_bf16 = "spotrf_update_bf16x3";
    static constexpr const char *update_bf16_la = "spotrf_update_bf16x3_la";
    static constexpr const char *split_panel = "spotrf_split_panel";
};

template <class T> bool valu_panel() { return std::is_same<T, double>::value && g_panel_kernel == 0; }

// Launch the update blocks of u (K contraction columns) with the block side
// that suits the launch; grid(bm) sets u for blocks of bm and returns their
// number.
template <class T, class G>
int launch_update_blocks(Ctx *c, hipStream_t s, const char *name, double fl, double by, T *dT, UpdArgs &u, int K,
                         const G &grid)
{
    typedef typename UpdShapes<T>::big Big;
    typedef typename UpdShapes<T>::small Small;
    typedef typename UpdShapes<T>::tiny Tiny;
    constexpr int occ = UpdShapes<T>::occ;
    // A launch of fewer than two 128 x 128 blocks per CU leaves the chip
    // idle: 64 x 64 blocks give four times the workgroups at a quarter of
    // the chain.  Where 128 does not divide the tile, blocks of 128 work for
    // padding, and their ragged parts are the slow ones (step-0 update of N =
    // 16000, us, 128 / 64: FP64 NB = 320 1798 / 1254, 192 1530 / 868, 336 1734
    // / 1696; FP32 NB = 64 1712 / 306, 160 1422 / 623, 240 924 / 698; where it
    // does, NB = 256 992 / 1020 and 563 / 593).
    int64_t g = grid(Big::BM);
    const bool big = g >= 512 && u.NB % Big::BM == 0 && update_lds_ok<Big>(dT, u.NB, K);
    if (!big) g = grid(Small::BM);
    // Tiles of 65 .. 127: most of a tile is ragged blocks of 64, the slow ones
    // through LDS, so through registers, in blocks of 32 where those pad less
    // (up to 96), but for few blocks of a tile that 32 divides (step-0 update of
    // N = 16000, us, LDS blocks of 64 / this: FP64 NB = 80 1690 / 1099, 96 1370 /
    // 982, 112 1072 / 1064; FP32 770 / 787, 608 / 600, 522 / 537.  dpotrf, ms:
    // 113.4 / 74.6, 73.3 / 52.0, 55.6 / 50.7; spotrf 52.4 / 52.1, 36.3 / 34.7,
    // 28.7 / 28.5).
    const bool ragged = u.NB > 64 && u.NB < 128;
    const bool few = !big && (g <= TINY_BLOCKS || (ragged && u.NB <= 96));
    const bool tiny = few && g <= TINY_BLOCKS && (!ragged || u.NB % 32 == 0) && update_lds_ok<Tiny>(dT, u.NB, K);
    const bool small = !tiny && !ragged && update_lds_ok<Small>(dT, u.NB, K);
    if (tiny || (few && !small)) g = grid(32);
    if (g > 0x7fffffff) { set_error("update grid too large"); return -3; }
    if (g <= 0) return 0;
    if (big)
        MI_LAUNCH(c, s, name, fl, by, (k_update_lds<Big, T, occ><<<(unsigned)g, Big::NT, 0, s>>>(dT, u)));
    else if (tiny)
        MI_LAUNCH(c, s, name, fl, by, (k_update_lds<Tiny, T, 3><<<(unsigned)g, Tiny::NT, 0, s>>>(dT, u)));
    else if (small)
        MI_LAUNCH(c, s, name, fl, by, (k_update_lds<Small, T, 2><<<(unsigned)g, Small::NT, 0, s>>>(dT, u)));
    else {
        const bool pair = u.NB % 2 == 0 && ((uintptr_t)dT & (2 * sizeof(T) - 1)) == 0;
        if (few && pair)
            MI_LAUNCH(c, s, name, fl, by, (k_update_mfma<T, true, 1><<<(unsigned)g, 128, 0, s>>>(dT, u)));
        else if (few)
            MI_LAUNCH(c, s, name, fl, by, (k_update_mfma<T, false, 1><<<(unsigned)g, 128, 0, s>>>(dT, u)));
        else if (pair)
            MI_LAUNCH(c, s, name, fl, by, (k_update_mfma<T, true, 2><<<(unsigned)g, 256, 0, s>>>(dT, u)));
        else
            MI_LAUNCH(c, s, name, fl, by, (k_update_mfma<T, false, 2><<<(unsigned)g, 256, 0, s>>>(dT, u)));
    }
    return 0;
}

// Largest diagonal tile (or sub-tile, where hmb re-tiles it) that the entry
// points take: what one workgroup's LDS held when a whole tile was factored
// there.  The panel kernels need no such limit; larger tiles stay refused.
template <class T> constexpr int diag_limit() { return sizeof(T) == 8 ? 560 : 1200; }
constexpr int VALU_DIAG_LIMIT = 604;               // k_potrf_diag: the tile's block column in 160 KB of LDS

template <class T> int check_diag(int n)
{
    if (n > (valu_panel<T>() ? VALU_DIAG_LIMIT : diag_limit<T>())) {
        set_error("tile size %d exceeds the limit of the diagonal factorization (%d)", n,
                  valu_panel<T>() ? VALU_DIAG_LIMIT : diag_limit<T>());
        return -4;
    }
    return 0;
}

// Panel engine 0 (FP64, tiles that fit its LDS): POTRF(k), then TRSM(m, k)
// for the ntile tiles from m0, one launch each.
int launch_panel_valu(Ctx *c, hipStream_t s, double *dT, int N, int NB, int MT, int k, double *Winv, bool diag, int m0,
                      int ntile)
{
    const int n = tile_rows(N, NB, MT, k);
    if (diag) {
        const int RC = ((n + 3) & ~3) + 4, lds = (PJB * RC + 1024) * (int)sizeof(double);
        if (lds > 65536)
            MI_CHECK(hipFuncSetAttribute((const void *)k_potrf_diag, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
        double *A = dT + tile_index(MT, k, k) * (int64_t)NB * NB;
        MI_LAUNCH(c, s, KN<double>::potrf, (double)n * n * n / 3.0, 16.0 * n * n,
                  k_potrf_diag<<<1, POTRF_THREADS, lds, s>>>(A, n, NB, RC, k * NB, c->d_info, Winv));
    }
    if (ntile > 0) {
        double fl = 0.0;
        for (int m = m0; m < m0 + ntile; m++) fl += (double)tile_rows(N, NB, MT, m) * NB * NB;
        const int strips = (NB + TRSM_ROWS - 1) / TRSM_ROWS;
        MI_LAUNCH(c, s, KN<double>::trsm, fl, fl / NB * 2.0 * sizeof(double),
                  k_trsm_panel<<<ntile * strips, 256, 0, s>>>(dT, N, NB, MT, k, Winv, m0));
    }
    return 0;
}

// Panel of step k on s: POTRF(k) when diag, and TRSM(m, k) of the ntile tiles
// m0, m0 + 1, ... (rows of the tile column), sub-column by sub-column of sb
// columns (a multiple of 32, at most SB): factor its diagonal block, solve
// the rows below, update the tile column's remaining columns.  ws: the
// operand images, (NB / 16) OPB elements, written when diag and read again by
// a call without it.
//
// Why sub-columns of 128: the diagonal block is one workgroup's chain of
// pivots, everything else spreads over the chip, and a launch behind another
// on one stream costs well under a microsecond.
template <class T>
int launch_panel(Ctx *c, hipStream_t s, T *dT, int N, int NB, int MT, int k, T *ws, int sb, bool diag, int m0,
                 int ntile)
{
    const int n = tile_rows(N, NB, MT, k);
    if constexpr (std::is_same<T, double>::value)
        if (valu_panel<T>() && n <= VALU_DIAG_LIMIT)
            return launch_panel_valu(c, s, dT, N, NB, MT, k, ws, diag, m0, ntile);
    double below = 0.0;                            // rows of the other tiles
    for (int m = m0; m < m0 + ntile; m++) below += tile_rows(N, NB, MT, m);
    T *A = dT + tile_index(MT, k, k) * (int64_t)NB * NB;
    for (int c0 = 0; c0 < n; c0 += sb) {
        const int w = std::min(sb, n - c0), c1 = c0 + w;
        T *op = ws + (int64_t)(c0 / DB) * OPB;
        if (diag)
            MI_LAUNCH(c, s, KN<T>::potrf, (double)w * w * w / 3.0, 2.0 * w * w * sizeof(T),
                      k_diag_factor<T><<<1, 512, 0, s>>>(A + (int64_t)c0 * NB + c0, w, NB, k * NB + c0, c->d_info, op));
        const double rows = below + (diag ? n - c1 : 0);
        const int g0 = diag ? (n - c1 + 63) / 64 : 0, gt = (NB + 63) / 64;
        if (g0 + gt * ntile > 0)
            MI_LAUNCH(c, s, KN<T>::trsm, rows * w * w, 2.0 * rows * w * sizeof(T),
                      k_panel_solve<T><<<g0 + gt * ntile, 256, 0, s>>>(dT, N, NB, MT, k, c0, w, op, g0, gt, m0));
        if (c1 >= n || (!diag && ntile <= 0)) continue;
        const double fl = 2.0 * below * w * (n - c1) + (diag ? (double)w * (n - c1) * (n - c1 + 1.0) : 0.0);
        const double by = (below + (diag ? 0.5 * (n - c1) : 0.0)) * (2.0 * (n - c1) + w) * sizeof(T);
        UpdArgs u{N, NB, MT, k, 0, 0, 0, c0, w, 0, 0, 0, m0, 1};
        auto grid = [&](int bm) -> int64_t {
            u.g0 = diag ? (n - c1 + bm - 1) / bm : 0;
            u.gr = (NB + bm - 1) / bm;
            u.nc = (n - c1 + bm - 1) / bm;
            return ((int64_t)u.g0 + (int64_t)u.gr * ntile) * u.nc;
        };
        int rc = launch_update_blocks<T>(c, s, KN<T>::panel_update, fl, by, dT, u, w, grid);
        if (rc) return rc;
    }
    return 0;
}

// Trailing update of step k over a run of tiles: column n_begin from row
// n_begin + m_off down, then whole columns, ntiles tiles in all (ntiles < 0:
// through the last column).
template <class T>
int launch_update_run(Ctx *c, hipStream_t s, T *dT, int N, int NB, int MT, int k, int n_begin,
                      int m_off, int64_t ntiles, bool bf16_split, bool la = false,
                      const __bf16 *split = nullptr, int split_m0 = 0)
{
    if (n_begin >= MT || n_begin + m_off >= MT) return 0;
    int64_t avail = MT - n_begin - m_off;
    for (int n = n_begin + 1; n < MT; n++) avail += MT - n;
    if (ntiles < 0 || ntiles > avail) ntiles = avail;
    if (ntiles <= 0) return 0;
    int nsub = (NB + BM - 1) / BM;
    int64_t grid = ntiles * nsub * nsub;
    if (g_update_kernel < 0) {
        const char *e = getenv("DPLASMA_MI_UPDATE");
        g_update_kernel = (e && !strcmp(e, "valu")) ? 0 : 1;
    }
    const bool valu = std::is_same<T, double>::value && g_update_kernel == 0;
    const bool bf16 = std::is_same<T, float>::value && bf16_split;
    if (grid > 0x7fffffff) { set_error("update grid too large"); return -3; }
    // algorithmic flops / bytes of the covered tiles: each C tile read and
    // written once, each panel tile (m, k) the launch needs read once
    double fl = 0.0, by = 0.0;
    int64_t left = ntiles;
    int m_lo = MT;
    for (int n = n_begin; n < MT && left > 0; n++)
        for (int m = (n == n_begin ? n + m_off : n); m < MT && left > 0; m++, left--) {
            const double tm = tile_rows(N, NB, MT, m);
            fl += (m == n) ? (double)NB * tm * (tm + 1.0) : 2.0 * tm * NB * NB;
            by += 2.0 * tm * NB * sizeof(T);
            m_lo = std::min(m_lo, n);
        }
    for (int m = m_lo; m < MT; m++) by += (double)tile_rows(N, NB, MT, m) * NB * sizeof(T);
    if (valu)
        MI_LAUNCH(c, s, "dpotrf_update_valu", fl, by,
                  k_update_valu<<<(unsigned)grid, 256, 0, s>>>((double *)dT, N, NB, MT, k, n_begin, m_off,
                                                               nsub));
    else if (bf16 && split && NB % WB == 0 && ntiles * (NB / WB) * (NB / WB) >= 2 * 256)
        // 256 x 256 blocks once the launch fills the chip twice over (one
        // workgroup per CU)
        MI_LAUNCH(c, s, la ? KN<float>::update_bf16_la : KN<float>::update_bf16, fl, by,
                  k_update_bf16x3w<<<(unsigned)(ntiles * (NB / WB) * (NB / WB)), 512, 0, s>>>(
                      (float *)dT, N, NB, MT, k, n_begin, m_off, NB / WB, split, split_m0));
    else if (bf16 && split)
        MI_LAUNCH(c, s, la ? KN<float>::update_bf16_la : KN<float>::update_bf16, fl, by,
                  k_update_bf16x3p<<<(unsigned)grid, 256, 0, s>>>((float *)dT, N, NB, MT, k, n_begin, m_off,
                                                                  nsub, split, split_m0));
    else if (bf16)
        MI_LAUNCH(c, s, la ? KN<float>::update_bf16_la : KN<float>::update_bf16, fl, by,
                  k_update_bf16x3<<<(unsigned)grid, 256, 0, s>>>((float *)dT, N, NB, MT, k, n_begin, m_off,
                                                                 nsub));
    else {
        UpdArgs u{N, NB, MT, k, n_begin, m_off, 0, 0, 0, 0, 0, 0, 0, la ? 1 : 0};
        return launch_update_blocks<T>(c, s, la ? KN<T>::update_la : KN<T>::update, fl, by, dT, u, NB, [&](int bm) {
            u.nsub = (NB + bm - 1) / bm;
            return ntiles * u.nsub * u.nsub;
        });
    }
    return 0;
}

template <class T>
int launch_update(Ctx *c, hipStream_t s, T *dT, int N, int NB, int MT, int k, int n_begin, int n_end,
                  bool bf16_split, bool la = false, const __bf16 *split = nullptr, int split_m0 = 0)
{
    if (n_begin >= n_end) return 0;
    int64_t ntiles = 0;
    for (int n = n_begin; n < n_end; n++) ntiles += MT - n;
    return launch_update_run<T>(c, s, dT, N, NB, MT, k, n_begin, 0, ntiles, bf16_split, la, split, split_m0);
}

// BF16 split of the panel tiles (m, k), m >= m0, into P (k_split_panel)
int launch_split_panel(Ctx *c, hipStream_t s, const float *dT, int N, int NB, int MT, int k, int m0, __bf16 *P)
{
    if (m0 >= MT) return 0;
    const int nb = (NB + SPT - 1) / SPT;
    const int64_t grid = (int64_t)(MT - m0) * nb * nb;
    double by = 0.0;
    for (int m = m0; m < MT; m++) by += (double)tile_rows(N, NB, MT, m) * NB * sizeof(float) + 2.0 * NB * NB * 2;
    MI_LAUNCH(c, s, KN<float>::split_panel, 0.0, by,
              k_split_panel<<<(unsigned)grid, 256, 0, s>>>(dT, N, NB, MT, k, m0, P));
    return 0;
}

// Elements of the operand images handed from POTRF(k) to TRSM(k), two steps
// in flight (the VALU panel's 32 x 32 inverses need a quarter of that).
constexpr size_t potrf_ws_elems(int NB) { return (size_t)2 * ((NB + DB - 1) / DB) * OPB; }

// Whole factorization of the packed lower tiles dT (N, NB), resident, with a
// two-step look-ahead over two streams (src/zpotrf_L.jdf's priorities give
// the panel the critical path):
//   panel stream, step k:  [wait: column k+1 updated by step k-1]
//                          column k+1 updated by step k (SYRK + GEMMs)
//                          -> event for the main stream,
//                          POTRF(k+1), TRSM(k+1)
//   main stream, step k:   [wait: column k+1 updated by step k]
//                          column k+2 updated by step k  -> event for the panel,
//                          columns k+3.. updated by step k (the bulk)
// The bulk starts after column k+1 and not beside it: that column is on the
// chain and takes 16 us alone, 37 us next to the bulk (N = 4096, NB = 256).
//
// Once a whole update is at most ONE_STREAM_WORK multiply-adds (FP64; twice
// that in FP32), about 100 us, it is one launch on the chain: no event (each
// about 10 us on the GPU and 4 us of host time), no column of its own before
// the rest.  A factorization that starts there uses the main stream only.
// Both together: dpotrf N = 378, NB = 93 260 -> 218 us; N = 4096, NB = 256
// 1.86 -> 1.77 ms; FP32 N = 10000, NB = 512 5.71 -> 5.37 ms (with the waves'
// priorities below).  Half or twice the limit: within 1%, four times it FP32
// N = 10000 5.7 ms.
// The waves of the chain's kernels run at a higher priority than the bulk's,
// which share their SIMDs (FP32 N = 10000 5.66 -> 5.45 ms).
// Every tile gets its updates in step order and no two launches touch the
// same tile at once; the panel chain waits for one column of the bulk of
// step k-1, not for all of it.
// bf16_split: FP32 trailing updates on BF16 MFMA with the two-term split.
// ws: potrf_ws_elems(NB) elements of workspace, or nullptr for the context's.
// ring: cross-stream dependencies use the context's fixed ring of events
// (created with the context) instead of its growing pool; every event is
// waited on within three records of being recorded, far inside the ring.
// hmb: the caller's sub-tile size of the diagonal factor (src/zpotrf_L.jdf:
// 168-192 re-tiles POTRF(k) with smallnb); the panel's sub-columns are no
// wider than that (rounded down to a multiple of 32, at least 32).  0: SB.
// The entry points without one use NB / 2 for NB >= 512 (a multiple of 64),
// which only matters for the tile sizes they take.
constexpr double ONE_STREAM_WORK = 2147483648.0;
constexpr int half_tile_hmb(int NB) { return (NB >= 512 && NB % 64 == 0) ? NB / 2 : 0; }

template <class T>
int potrf_tiles(Ctx *c, int N, int NB, T *dT, int *info, bool bf16_split, T *ws, bool ring = false, int hmb = 0,
                bool wait = true)
{
    *info = 0;
    if (N < 0 || NB <= 0) { set_error("bad sizes N=%d NB=%d", N, NB); return -2; }
    if (N == 0) return 0;
    const int MT = (N + NB - 1) / NB;
    int rc;
    const size_t wsz = potrf_ws_elems(NB) / 2;      // elements per step
    if (!ws && !(ws = (T *)ws_get(c, WS_POTRF_WINV, potrf_ws_elems(NB) * sizeof(T)))) return -3;
    c->ev_next = 0;
    size_t ring_next = 0;
    auto ev = [&]() -> hipEvent_t { return ring ? c->ev_ring[ring_next++ % c->ev_ring.size()] : next_event(c); };
    if (hmb > 0) hmb = std::max(32, hmb & ~31);
    if ((rc = check_diag<T>(hmb > 0 ? std::min(hmb, NB) : NB))) return rc;
    const int sb = hmb > 0 ? std::min(hmb, SB) : SB;
    // FP32 factor with BF16 updates: the main stream splits each panel
    // column once (tiles k+2.. of column k; its launches run in order, so one
    // image serves every step)
    __bf16 *split = nullptr;
    if (std::is_same<T, float>::value && bf16_split && g_bf16_panel_split && NB % XK == 0 && MT > 2) {
        split = (__bf16 *)ws_get(c, WS_BF16_PANEL, (size_t)(MT - 2) * 2 * NB * NB * sizeof(__bf16));
        if (!split) return -3;
    }
    // steps from k1 on run on one stream
    int k1 = 0;
    const double one = 0.5 * NB * NB * NB * sizeof(T) / 8;
    while (k1 < MT - 1 && (MT - k1 - 1.0) * (MT - k1) * one > ONE_STREAM_WORK) k1++;
    const hipStream_t sp = k1 > 0 ? c->s_panel : c->s_main;
    auto panel = [&](int k) -> int {
        return launch_panel<T>(c, sp, dT, N, NB, MT, k, ws + (k & 1) * wsz, sb, true, k + 1, MT - k - 1);
    };
    auto pass = [&](hipEvent_t e, hipStream_t from, hipStream_t to) -> int {
        MI_CHECK(hipEventRecord(e, from));
        MI_CHECK(hipStreamWaitEvent(to, e, 0));
        return 0;
    };

    MI_CHECK(hipEventRecord(c->t0, c->s_main));
    k_fill_int<<<1, 64, 0, c->s_main>>>(c->d_info, 0, 1);
    if (sp != c->s_main && (rc = pass(ev(), c->s_main, sp))) return rc;

    if ((rc = panel(0))) return rc;
    hipEvent_t col_ready = nullptr;                // column k+1 updated by step k-1

    for (int k = 0; k < MT - 1; k++) {
        if (k >= k1) {
            if (k == k1 && k > 0 && (rc = pass(ev(), c->s_main, sp))) return rc;
            if ((rc = launch_update<T>(c, sp, dT, N, NB, MT, k, k + 1, MT, bf16_split, true))) return rc;
            if ((rc = panel(k + 1))) return rc;
            continue;
        }
        // panel stream: column k+1 by step k, then the next panel; main
        // stream, once column k+1 is done: the look-ahead column k+2, then
        // the bulk of step k
        if (col_ready) MI_CHECK(hipStreamWaitEvent(sp, col_ready, 0));
        if ((rc = launch_update<T>(c, sp, dT, N, NB, MT, k, k + 1, k + 2, bf16_split, true))) return rc;
        if ((rc = pass(ev(), sp, c->s_main))) return rc;
        if ((rc = panel(k + 1))) return rc;
        col_ready = nullptr;
        const __bf16 *im = (split && k + 2 < MT) ? split : nullptr;
        if (im && (rc = launch_split_panel(c, c->s_main, (const float *)dT, N, NB, MT, k, k + 2, split))) return rc;
        if (k + 2 < MT) {
            if ((rc = launch_update<T>(c, c->s_main, dT, N, NB, MT, k, k + 2, k + 3, bf16_split, false, im, k + 2)))
                return rc;
            col_ready = ev();
            MI_CHECK(hipEventRecord(col_ready, c->s_main));
        }
        if ((rc = launch_update<T>(c, c->s_main, dT, N, NB, MT, k, k + 3, MT, bf16_split, false, im, k + 2)))
            return rc;
    }
    if (sp != c->s_main && (rc = pass(ev(), sp, c->s_main))) return rc;
    MI_CHECK(hipEventRecord(c->t1, c->s_main));
    if (!wait) return 0;                           // info stays in d_info[0]
    int h_info = 0;
    MI_CHECK(hipMemcpyAsync(&h_info, c->d_info, sizeof(int), hipMemcpyDeviceToHost, c->s_main));
    if ((rc = mi_synchronize(static_cast<mi_ctx_t *>(c)))) return rc;
    float ms = 0.f;
    MI_CHECK(hipEventElapsedTime(&ms, c->t0, c->t1));
    c->last_ms = ms;
    *info = h_info;
    return 0;
}

// single task-class launches, blocking (tests)
template <class T>
int step_potrf(mi_ctx_t *c, int N, int NB, T *dT, int k, int *info)
{
    if (N <= 0) { *info = 0; return 0; }
    const int MT = (N + NB - 1) / NB;
    int rc = check_diag<T>(NB);
    if (rc) return rc;
    T *ws = (T *)ws_get(c, WS_POTRF_WINV, potrf_ws_elems(NB) * sizeof(T));
    if (!ws) return -3;
    k_fill_int<<<1, 64, 0, c->s_main>>>(c->d_info, 0, 1);
    if ((rc = launch_panel<T>(c, c->s_main, dT, N, NB, MT, k, ws, SB, true, k + 1, 0))) return rc;
    MI_CHECK(hipMemcpyAsync(info, c->d_info, sizeof(int), hipMemcpyDeviceToHost, c->s_main));
    return mi_synchronize(c);
}

template <class T>
int step_trsm(mi_ctx_t *c, int N, int NB, T *dT, int k)
{
    // the operand images come from the POTRF launch of the same k
    const int MT = (N + NB - 1) / NB;
    T *ws = (T *)c->ws[WS_POTRF_WINV].p;
    if (!ws || c->ws[WS_POTRF_WINV].bytes < potrf_ws_elems(NB) * sizeof(T)) {
        set_error("the panel solve of step k needs the POTRF launch of step k first");
        return -2;
    }
    int rc = launch_panel<T>(c, c->s_main, dT, N, NB, MT, k, ws, SB, false, k + 1, MT - k - 1);
    if (rc) return rc;
    return mi_synchronize(c);
}

template <class T>
int step_update(mi_ctx_t *c, int N, int NB, T *dT, int k, int n_begin, int n_end)
{
    const int MT = (N + NB - 1) / NB;
    if (k < 0 || n_begin <= k || n_end > MT) { set_error("bad update range"); return -2; }
    int rc = launch_update<T>(c, c->s_main, dT, N, NB, MT, k, n_begin, n_end, g_supdate == 1);
    if (rc) return rc;
    return mi_synchronize(c);
}

}  // namespace

namespace mi {

// Single tile tasks on the packed lower image, enqueued on s (the bodies of
// the four task classes of src/zpotrf_L.jdf:91-633, one tile each).
int task_prepare_fp64(int NB) { return check_diag<double>(NB); }
int task_potrf_fp64(Ctx *c, hipStream_t s, double *dT, int N, int NB, int k, double *Winv)
{
    return launch_panel<double>(c, s, dT, N, NB, (N + NB - 1) / NB, k, Winv, SB, true, k + 1, 0);
}
int task_trsm_fp64(Ctx *c, hipStream_t s, double *dT, int N, int NB, int m, int k, double *Winv)
{
    return launch_panel<double>(c, s, dT, N, NB, (N + NB - 1) / NB, k, Winv, SB, false, m, 1);
}
// tile (m, n), m >= n > k: A(m, n) -= A(m, k) A(n, k)^T (SYRK when m == n)
int task_update_fp64(Ctx *c, hipStream_t s, double *dT, int N, int NB, int m, int n, int k)
{
    return launch_update_run<double>(c, s, dT, N, NB, (N + NB - 1) / NB, k, n, m - n, 1, false);
}
size_t task_winv_elems(int NB) { return potrf_ws_elems(NB) / 2; }

template <> int potrf_check<double>(int NB)
{
    const int hmb = half_tile_hmb(NB);
    return check_diag<double>(hmb > 0 ? hmb : NB);
}
template <> int potrf_check<float>(int NB)
{
    const int hmb = g_supdate == 1 ? half_tile_hmb(NB) : 0;
    return check_diag<float>(hmb > 0 ? hmb : NB);
}
template <> int potrf_enqueue<double>(Ctx *c, int N, int NB, double *dT)
{
    int info;
    return potrf_tiles<double>(c, N, NB, dT, &info, false, nullptr, false, half_tile_hmb(NB), false);
}
template <> int potrf_enqueue<float>(Ctx *c, int N, int NB, float *dT)
{
    int info;
    return spotrf_tiles_split(c, N, NB, dT, &info, g_supdate == 1, false);
}

int spotrf_tiles_split(Ctx *c, int N, int NB, float *dT, int *info, bool bf16_split, bool wait)
{
    return potrf_tiles<float>(c, N, NB, dT, info, bf16_split, nullptr, false, bf16_split ? half_tile_hmb(NB) : 0,
                              wait);
}
}  // namespace mi

// ---------------------------------------------------------------------------
// Allocation-free FP64 factorization (mi_dpotrf_tiles_noalloc).  Its only
// scratch memory, the operand images that a panel's diagonal factor hands to
// its row solve, two steps in flight, lives in this file-scope device array
// instead of context workspaces: one copy per GPU, held until the process
// ends, shared by every call on that GPU.  Images are written before they
// are read, so nothing has to be cleared between calls.  On the host the array's name is only a stand-in: host code uses
// the device address that noalloc_setup reads once per device.
namespace {
constexpr int NOALLOC_MAX_NB = 1024;
constexpr int NOALLOC_MAX_DEV = 64;
__device__ __align__(256) double scratch[potrf_ws_elems(NOALLOC_MAX_NB)];                 // 2 MiB

std::mutex g_noalloc_mu;
bool g_noalloc_done[NOALLOC_MAX_DEV];
hipError_t g_noalloc_err[NOALLOC_MAX_DEV];
double *g_noalloc_ptr[NOALLOC_MAX_DEV];
}  // namespace

namespace mi {
// Called by mi_ctx_create with `device` current: the device address of
// `scratch` on that GPU, read once per device and kept.
void noalloc_setup(int device)
{
    if (device < 0 || device >= NOALLOC_MAX_DEV) return;
    std::lock_guard<std::mutex> g(g_noalloc_mu);
    if (g_noalloc_done[device]) return;
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) (void)hipGetLastError();
    g_noalloc_err[device] = e;
    g_noalloc_ptr[device] = e == hipSuccess ? static_cast<double *>(p) : nullptr;
    g_noalloc_done[device] = true;
}
}  // namespace mi

extern "C" {

int mi_set_panel_engine(int which)
{
    if (which != 0 && which != 1) { set_error("panel engine must be 0 (VALU) or 1 (MFMA)"); return -2; }
    g_panel_kernel = which;
    return 0;
}

int mi_set_spotrf_update(int which)
{
    if (which != 0 && which != 1) { set_error("FP32 update must be 0 (FP32 MFMA) or 1 (BF16 split)"); return -2; }
    g_supdate = which;
    return 0;
}

int mi_set_bf16_panel_split(int which)
{
    if (which != 0 && which != 1) { set_error("BF16 panel split must be 0 (per workgroup) or 1 (once per step)"); return -2; }
    g_bf16_panel_split = which;
    return 0;
}

int mi_set_update_engine(int which)
{
    if (which != 0 && which != 1) { set_error("update engine must be 0 (VALU) or 1 (MFMA)"); return -2; }
    g_update_kernel = which;
    return 0;
}

int mi_dpotrf_step_potrf(mi_ctx_t *c, int N, int NB, double *dT, int k, int *info)
{
    return step_potrf<double>(c, N, NB, dT, k, info);
}

int mi_dpotrf_step_trsm(mi_ctx_t *c, int N, int NB, double *dT, int k)
{
    return step_trsm<double>(c, N, NB, dT, k);
}

int mi_dpotrf_step_update(mi_ctx_t *c, int N, int NB, double *dT, int k, int n_begin, int n_end)
{
    return step_update<double>(c, N, NB, dT, k, n_begin, n_end);
}

int mi_spotrf_step_potrf(mi_ctx_t *c, int N, int NB, float *dT, int k, int *info)
{
    return step_potrf<float>(c, N, NB, dT, k, info);
}

int mi_spotrf_step_trsm(mi_ctx_t *c, int N, int NB, float *dT, int k)
{
    return step_trsm<float>(c, N, NB, dT, k);
}

int mi_spotrf_step_update(mi_ctx_t *c, int N, int NB, float *dT, int k, int n_begin, int n_end)
{
    return step_update<float>(c, N, NB, dT, k, n_begin, n_end);
}

int mi_dpotrf_tiles(mi_ctx_t *c, int N, int NB, double *dT, int *info)
{
    return potrf_tiles<double>(c, N, NB, dT, info, false, nullptr, false, half_tile_hmb(NB));
}

int mi_dpotrf_tiles_rec(mi_ctx_t *c, int N, int NB, double *dT, int hmb, int *info)
{
    if (hmb <= 0) { *info = 0; set_error("mi_dpotrf_tiles_rec: hmb=%d must be positive", hmb); return -2; }
    return potrf_tiles<double>(c, N, NB, dT, info, false, nullptr, false, hmb);
}

int mi_dpotrf_tiles_noalloc(mi_ctx_t *c, int N, int NB, double *dT, int *info)
{
    *info = 0;
    if (N < 0 || NB <= 0) { set_error("mi_dpotrf_tiles_noalloc: bad sizes N=%d NB=%d", N, NB); return -2; }
    if (NB > NOALLOC_MAX_NB) {
        set_error("mi_dpotrf_tiles_noalloc: NB=%d exceeds the limit of its fixed scratch (NB <= %d)", NB,
                  NOALLOC_MAX_NB);
        return -2;
    }
    double *ptr = nullptr;
    hipError_t e = hipErrorInvalidDevice;
    if (c->device >= 0 && c->device < NOALLOC_MAX_DEV) {
        std::lock_guard<std::mutex> g(g_noalloc_mu);
        if (g_noalloc_done[c->device]) {
            ptr = g_noalloc_ptr[c->device];
            e = g_noalloc_err[c->device];
        }
    }
    if (!ptr) {
        set_error("mi_dpotrf_tiles_noalloc: no scratch address for device %d (%s)", c->device,
                  hipGetErrorString(e));
        return -1;
    }
    // the context's fixed event ring instead of its event pool, which grows
    // on demand; the profiler creates events on demand, so it is off for
    // this call
    const bool prof = c->prof;
    c->prof = false;
    const int rc = potrf_tiles<double>(c, N, NB, dT, info, false, ptr, true, half_tile_hmb(NB));
    c->prof = prof;
    return rc;
}

int mi_spotrf_tiles(mi_ctx_t *c, int N, int NB, float *dT, int *info)
{
    return spotrf_tiles_split(c, N, NB, dT, info, g_supdate == 1);
}

}  // extern "C"
