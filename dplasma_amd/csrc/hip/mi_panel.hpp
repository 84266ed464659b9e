// mi_panel.hpp -- the panel of the tile Cholesky (POTRF(k) and TRSM(m,k) of
// src/zpotrf_L.jdf:91-343), factored in sub-columns of SB columns:
//   k_diag_factor   one workgroup: the w x w diagonal block of sub-column j
//   k_panel_solve   X = C L_jj^{-T} for every row below it, 16 rows a wave
//   k_update_*      the remaining columns of the tile column -= X X_k^T
// (mi_potrf.hip launches them).  Everything works on 16 x 16 blocks held in
// the accumulator layout of the 16x16x4 MFMA fed (B, A): element q of lane
// l = 16 fk + fr is C(row fr, column row(q, fk)).  The same registers are,
// element s for K slice s, the B operand of a product that contracts over
// those columns (slice s then holds columns row(s, fk)), and likewise the A
// operand X(fr, row(s, fk)); so a block passes from one product to the next
// without leaving the registers, and blocks that other waves need travel as
// [s][lane] images of 64 consecutive elements (no bank conflicts, whole
// lines).
#pragma once
#include <utility>
#include "mi_common.hpp"

namespace mi {

constexpr int SB = 128;               // columns of a sub-column
constexpr int DB = 16;                // block side
constexpr int DBN = SB / DB;          // blocks a side, at most
// Operand images that k_diag_factor leaves for k_panel_solve, per 16-column
// block b of a tile: W_b = L_bb^{-1}, then -L(b + i, b), i = 1 .. (blocks
// left in its sub-column): DBN images of 256 elements, [lane][s] (16-byte
// pieces per lane).
constexpr int OPI = DB * DB;
constexpr int OPB = DBN * OPI;

// ------------------------------------------------------- cross-lane helpers
// value of lane C of each row of 16 lanes
template <int C> __device__ __forceinline__ double row_bcast(double v)
{
    return __longlong_as_double(
        __builtin_amdgcn_update_dpp((long long)0, __double_as_longlong(v), 0x150 + C, 0xf, 0xf, true));
}
template <int C> __device__ __forceinline__ float row_bcast(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + C, 0xf, 0xf, true));
}

// value rotated by C lanes within each row of 16 (row_ror)
template <int C> __device__ __forceinline__ float row_rotate(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + C, 0xf, 0xf, true));
}
template <int C> __device__ __forceinline__ double row_rotate(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, 0x120 + C, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x120 + C, 0xf, 0xf, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// a[C + i] -= row_bcast<C + i>(m) * f, i < K (K <= 8): one DPP FMA each (the
// compiler does not fold a broadcast into the FP64 FMA).  The two wait
// states that a DPP read needs after m was written are inside the block.
#define MI_F(op, i) "v_fmac_" op "_dpp %[a" #i "], -%[m], %[f] row_newbcast:%[c" #i "] row_mask:0xf bank_mask:0xf\n\t"
#define MI_A(i) [a##i] "+&v"(a[C + i])
#define MI_C(i) [c##i] "n"(C + i)
#define MI_FMAC(op, n)                                                        \
    if constexpr (K == n)                                                     \
    asm("s_nop 1\n\t" MI_F##n(op) : MI_A##n : [m] "v"(m), [f] "v"(f), MI_C##n)
#define MI_F1(op) MI_F(op, 0)
#define MI_F2(op) MI_F1(op) MI_F(op, 1)
#define MI_F3(op) MI_F2(op) MI_F(op, 2)
#define MI_F4(op) MI_F3(op) MI_F(op, 3)
#define MI_F5(op) MI_F4(op) MI_F(op, 4)
#define MI_F6(op) MI_F5(op) MI_F(op, 5)
#define MI_F7(op) MI_F6(op) MI_F(op, 6)
#define MI_F8(op) MI_F7(op) MI_F(op, 7)
#define MI_A1 MI_A(0)
#define MI_A2 MI_A1, MI_A(1)
#define MI_A3 MI_A2, MI_A(2)
#define MI_A4 MI_A3, MI_A(3)
#define MI_A5 MI_A4, MI_A(4)
#define MI_A6 MI_A5, MI_A(5)
#define MI_A7 MI_A6, MI_A(6)
#define MI_A8 MI_A7, MI_A(7)
#define MI_C1 MI_C(0)
#define MI_C2 MI_C1, MI_C(1)
#define MI_C3 MI_C2, MI_C(2)
#define MI_C4 MI_C3, MI_C(3)
#define MI_C5 MI_C4, MI_C(4)
#define MI_C6 MI_C5, MI_C(5)
#define MI_C7 MI_C6, MI_C(6)
#define MI_C8 MI_C7, MI_C(7)
template <int C, int K> __device__ __forceinline__ void fmac_bcast(double *a, double m, double f)
{
    MI_FMAC("f64", 1); MI_FMAC("f64", 2); MI_FMAC("f64", 3); MI_FMAC("f64", 4);
    MI_FMAC("f64", 5); MI_FMAC("f64", 6); MI_FMAC("f64", 7); MI_FMAC("f64", 8);
}
template <int C, int K> __device__ __forceinline__ void fmac_bcast(float *a, float m, float f)
{
    MI_FMAC("f32", 1); MI_FMAC("f32", 2); MI_FMAC("f32", 3); MI_FMAC("f32", 4);
    MI_FMAC("f32", 5); MI_FMAC("f32", 6); MI_FMAC("f32", 7); MI_FMAC("f32", 8);
}
#undef MI_FMAC

// a[c] -= row_bcast<c>(m) * f for C <= c < 16
template <int C, class T> __device__ __forceinline__ void fmac_rest(T *a, T m, T f)
{
    if constexpr (C < DB) {
        constexpr int K = DB - C < 8 ? DB - C : 8;
        fmac_bcast<C, K>(a, m, f);
        fmac_rest<C + K>(a, m, f);
    }
}

// The sweep over a 16 x 16 block, four copies of it side by side in the rows
// of 16 lanes: lane fr holds row fr of D in v[] and row fr of the identity in
// x[].  Column c: l[c] becomes L(fr, c) (l may be v), x[c] becomes W(c, fr)
// (W = L^{-1}); v and x lose the multiple of the column.  Entries above the
// diagonal hold arbitrary values throughout and never reach another lane.
//
// A lone wave issues one instruction every four cycles and waits out every
// dependent one, so the order of the instructions is the sweep's time.  It
// is laid down here, at compile time: the chain from pivot to pivot (broadcast,
// reciprocal root, its correction, the scaled column, the next pivot) with
// the FMAs of earlier columns in its gaps, those on v first, those on x
// behind them as far as they fill gaps; what is left of x comes last.  Alone
// on its SIMD a sweep takes 2340 cycles (FP64; 389 instructions, 16 of them
// the 16-cycle root) and 2090 (FP32).  The root's correction is one
// third-order step in FP64 (v_rsq_f64 is good to about 2^-26) and one Newton
// step in FP32; a pivot <= 0, infinite or NaN (in FP32 also a denormal, which
// v_rsq_f32 takes for zero) comes out as NaN.
//
// The instructions are volatile, so that this order stays; the two wait
// states between a write and its read by DPP, and the one after a root, are
// part of the plan and not the compiler's to insert.
enum SweepOp { S_BCAST, S_RSQ, S_T, S_E, S_U, S_W, S_RD, S_COL, S_PIVOT, S_V, S_XS, S_X, S_NOP };
struct SweepStep { int op, c, j; };
struct SweepPlan {
    SweepStep step[512] = {};
    int n = 0;
};
constexpr SweepPlan sweep_plan(bool f64)
{
    SweepPlan p{};
    SweepStep vq[128] = {}, xq[160] = {};              // FMAs on v and x in their order
    int vn = 0, v0 = 0, xn = 0, x0 = 0;
    int col = -8;                                      // place of the latest S_COL, and its column
    int colc = -1;
    auto put = [&](int op, int c, int j) {
        p.step[p.n].op = op;
        p.step[p.n].c = c;
        p.step[p.n].j = j;
        p.n++;
    };
    // one FMA if there is one; a lane broadcast must not read a register
    // that one of the two instructions before it wrote
    auto fill = [&]() -> bool {
        const bool fresh = p.n - col <= 2;
        if (v0 < vn && !(fresh && vq[v0].c == colc)) {
            put(S_V, vq[v0].c, vq[v0].j);
            v0++;
            return true;
        }
        if (x0 < xn && !(xq[x0].op == S_X && fresh && xq[x0].c == colc)) {
            put(xq[x0].op, xq[x0].c, xq[x0].j);
            x0++;
            return true;
        }
        return false;
    };
    auto gap = [&](int want, int need) {
        for (int i = 0; i < want; i++)
            if (!fill() && i < need) put(S_NOP, 0, 0);
    };
    put(S_NOP, 0, 0);
    put(S_NOP, 0, 0);
    for (int c = 0; c < DB; c++) {
        put(S_BCAST, c, 0);
        gap(1, 0);
        put(S_RSQ, c, 0);
        gap(4, 1);
        put(S_T, c, 0);
        gap(2, 0);
        put(S_E, c, 0);
        gap(1, 0);
        put(S_U, c, 0);
        if (f64) put(S_W, c, 0);
        gap(1, 0);
        put(S_RD, c, 0);
        xq[xn].op = S_XS;
        xq[xn].c = c;
        xn++;
        gap(1, 0);
        while (v0 < vn && vq[v0].j <= c + 1) fill();   // what the next pivot still lacks
        put(S_COL, c, 0);
        col = p.n - 1;
        colc = c;
        for (int j = c + 2; j < DB; j++) {
            vq[vn].c = c;
            vq[vn].j = j;
            vn++;
        }
        for (int j = c + 1; j < DB; j++) {
            xq[xn].op = S_X;
            xq[xn].c = c;
            xq[xn].j = j;
            xn++;
        }
        if (c + 1 < DB) {
            gap(2, 2);
            put(S_PIVOT, c, c + 1);
            gap(4, 2);
        }
    }
    gap(2, 2);
    while (fill()) {}
    return p;
}
// Wait states: two instructions between a write of v[c] and its read by DPP,
// one between a root and its first use.
constexpr bool sweep_plan_ok(const SweepPlan &p)
{
    int wrote[DB] = {}, root = -1;
    for (int i = 0; i < DB; i++) wrote[i] = -1;
    for (int i = 0; i < p.n; i++) {
        const SweepStep &t = p.step[i];
        if ((t.op == S_BCAST || t.op == S_PIVOT || t.op == S_V || t.op == S_X) && i - wrote[t.c] < 3) return false;
        if (t.op == S_T && i - root < 2) return false;
        if (t.op == S_RSQ) root = i;
        if (t.op == S_COL) wrote[t.c] = i;
        if (t.op == S_PIVOT || t.op == S_V) wrote[t.j] = i;
    }
    return true;
}
template <class T> struct SweepPlanOf {
    static constexpr SweepPlan plan = sweep_plan(sizeof(T) == 8);
    static_assert(sweep_plan_ok(plan), "wait states of the sweep");
};
template <class T> struct SweepTmp { T p, t, e, u, w, rd[DB]; };

#define MI_SW(f64, f32, ...)                                                       \
    do {                                                                           \
        if constexpr (sizeof(T) == 8) asm volatile(f64 __VA_ARGS__);               \
        else asm volatile(f32 __VA_ARGS__);                                        \
    } while (0)
template <class T, int I> __device__ __forceinline__ void sweep_step(T *v, T *x, T *l, SweepTmp<T> &t)
{
    constexpr SweepStep s = SweepPlanOf<T>::plan.step[I];
    constexpr int c = s.c, j = s.j;
    if constexpr (s.op == S_NOP) asm volatile("s_nop 0");
    else if constexpr (s.op == S_BCAST)
        MI_SW("v_mov_b64_dpp %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf",
              "v_mov_b32_dpp %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf", : "=v"(t.p) : "v"(v[c]), "n"(c));
    else if constexpr (s.op == S_RSQ) MI_SW("v_rsq_f64 %0, %1", "v_rsq_f32 %0, %1", : "=v"(t.rd[c]) : "v"(t.p));
    else if constexpr (s.op == S_T)
        MI_SW("v_mul_f64 %0, -%1, %2", "v_mul_f32 %0, -%1, %2", : "=v"(t.t) : "v"(t.p), "v"(t.rd[c]));
    else if constexpr (s.op == S_E)
        MI_SW("v_fma_f64 %0, %1, %2, 1.0", "v_fma_f32 %0, %1, %2, 1.0", : "=v"(t.e) : "v"(t.t), "v"(t.rd[c]));
    else if constexpr (s.op == S_U)
        MI_SW("v_mul_f64 %0, %1, %2", "v_mul_f32 %0, %1, %2", : "=v"(t.u) : "v"(t.rd[c]), "v"(t.e));
    else if constexpr (s.op == S_W) asm volatile("v_fma_f64 %0, %1, %2, 0.5" : "=v"(t.w) : "v"(t.e), "s"(T(0.375)));
    else if constexpr (s.op == S_RD) {
        if constexpr (sizeof(T) == 8) asm volatile("v_fmac_f64 %0, %1, %2" : "+v"(t.rd[c]) : "v"(t.u), "v"(t.w));
        else asm volatile("v_fma_f32 %0, %1, 0.5, %0" : "+v"(t.rd[c]) : "v"(t.u));
    } else if constexpr (s.op == S_COL)
        MI_SW("v_mul_f64 %0, %1, %2", "v_mul_f32 %0, %1, %2", : "=v"(l[c]) : "v"(v[c]), "v"(t.rd[c]));
    else if constexpr (s.op == S_XS)
        MI_SW("v_mul_f64 %0, %0, %1", "v_mul_f32 %0, %0, %1", : "+v"(x[c]) : "v"(t.rd[c]));
    else if constexpr (s.op == S_X)
        MI_SW("v_fmac_f64_dpp %0, -%1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf",
              "v_fmac_f32_dpp %0, -%1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf",
              : "+v"(x[j]) : "v"(l[c]), "v"(x[c]), "n"(j));
    else
        MI_SW("v_fmac_f64_dpp %0, -%1, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf",
              "v_fmac_f32_dpp %0, -%1, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf",
              : "+v"(v[j]) : "v"(l[c]), "n"(j));
}
#undef MI_SW
template <class T, int... I>
__device__ __forceinline__ void sweep_steps(T *v, T *x, T *l, SweepTmp<T> &t, std::integer_sequence<int, I...>)
{
    (sweep_step<T, I>(v, x, l, t), ...);
}
// True when a pivot was not an ordinary positive number: its NaN reciprocal
// root reaches every later column.
template <class T> __device__ __forceinline__ bool sweep_fast(T *v, T *x, T *l)
{
    SweepTmp<T> t;
    sweep_steps(v, x, l, t, std::make_integer_sequence<int, SweepPlanOf<T>::plan.n>());
    return t.rd[DB - 1] != t.rd[DB - 1];
}

// The sweep's L(c, c) is the pivot times its reciprocal root: two roundings
// and the root's own error, up to 1.1 ulp.  So the pivots, which lane c is left
// with in v[c], go along to the wave that stores L, and it makes the rounded
// root of them, off the chain of pivots (batched factor of order 5, FP64,
// error in eps: 0.89 without, 0.52 with; N = 500, NB = 48 1.01 and 0.91).
template <class T> __device__ __forceinline__ T pivot_of(const T *v, int fr)
{
    T p = v[0];
#pragma unroll
    for (int c = 1; c < DB; c++) {
        T a = v[c];
        asm("" : "+v"(a));                                  // a select of values, not of addresses
        p = fr == c ? a : p;
    }
    return p;
}
// sqrt(p) from d within a few ulp of it; d where p is NaN
__device__ __forceinline__ double root_of(double d, double p)
{
    const double s = fma(fma(-d, d, p), 0.5 * __builtin_amdgcn_rcp(d), d);
    return s == s ? s : d;
}
__device__ __forceinline__ float root_of(float d, float p)
{
    const float s = fmaf(fmaf(-d, d, p), 0.5f * __builtin_amdgcn_rcpf(d), d);
    return s == s ? s : d;
}

// The same sweep with square root and division, for blocks with a pivot that
// is not positive, infinite, NaN or denormal; the first non-positive (or
// NaN) pivot's column goes to *fail (0: none) and counts as 1 from there on.
template <int C, class T> __device__ __forceinline__ void sweep_column_exact(T *v, T *x, int fr, int *fail)
{
    T d0 = row_bcast<C>(v[C]);
    const bool ok = d0 > T(0);
    if (!ok && !*fail) *fail = C + 1;
    d0 = ok ? d0 : T(1);
    const T d = sqrt(d0), rd = T(1) / d;
    const T m = v[C] * rd;
    x[C] = x[C] * rd;
    fmac_rest<C + 1>(v, m, m);
    fmac_rest<C + 1>(x, m, x[C]);
    v[C] = fr == C ? d : m;
}
template <class T, int... C>
__device__ __forceinline__ void sweep_exact(T *v, T *x, int fr, int *fail, std::integer_sequence<int, C...>)
{
    (sweep_column_exact<C>(v, x, fr, fail), ...);
}

// x := W = L^{-1} by rows as in the sweep: v holds L (lane fr: row fr), rd the
// reciprocal of L(fr, fr), x the identity on entry.
template <int C, class T> __device__ __forceinline__ void invert_column(T *v, T *x, T rd)
{
    x[C] = x[C] * row_bcast<C>(rd);
    fmac_rest<C + 1>(x, v[C], x[C]);
}
template <class T, int... C>
__device__ __forceinline__ void invert_rows(T *v, T *x, T rd, std::integer_sequence<int, C...>)
{
    (invert_column<C>(v, x, rd), ...);
}

// ---------------------------------------------------------------------------
// Cholesky factor of the n x n (n <= 16 NBK) block A (column-major, ld),
// lower, in place: right-looking over 16-column blocks, by the NW waves of a
// workgroup; the 16 x 16 blocks below the first diagonal block live in the
// registers of waves 1.. (dealt out column by column) from load to store.
//   wave 0   factors D_p (sweep above), publishes W_p, forms X(p+1, p) =
//            C W_p^T and the next diagonal block D_{p+1} -= X X^T itself,
//   others   meanwhile apply step p - 1 to their blocks, hand C(p+1, p)
//            and D_{p+1} to wave 0 through LDS, and after W_p is there form
//            the rest of block column p.
// Two barriers a step.  Every block is updated in step order whatever the
// timing.  The last wave stores what wave 0 leaves in LDS.  Bound by wave
// 0's chain: 16 dependent pivots (reciprocal square root with one correction
// step, then a DPP FMA into the next pivot), then eight MFMAs and the
// hand-offs.
// xl(i, p): LDS image ([s][lane]) of -X(i, p), valid until step p + 1 is
// over; wl(p): W_p in LDS, image column t at t DIAG_WP, valid as long (both
// may keep all steps).  Returns the 1-based column of the first pivot
// that is not positive, or 0, to every wave (ds.fail is 0 on entry and
// ordered before this by a barrier).
constexpr int DIAG_WP = DB + 2;                             // distinct banks for the writer of W
template <class T> struct DiagLds {
    T hc[OPI], hd[OPI];                                     // C(p+1, p) and D_{p+1} for wave 0
    __align__(16) T ll[2][DB][DIAG_WP];                     // L_pp, [column][row], and behind each column its pivot
    __align__(16) T dl[DB][DIAG_WP];                        // D, [row][column]
    int fail;
};
template <class T, int NW, int NBK, class XL, class WL>
__device__ __forceinline__ int diag_factor(T *__restrict__ A, int n, int ld, DiagLds<T> &ds, XL &&xl, WL &&wl)
{
    typedef typename MF<T>::v4 V4;
    // worker waves; of eight, wave 4 is none: it shares the SIMD of wave 0,
    // where every MFMA would hold up the sweep
    constexpr bool APART = NW == 8;
    constexpr int NK = APART ? NW - 2 : NW - 1;
    constexpr int NBLK = NBK * (NBK + 1) / 2 - 1;           // blocks besides (0, 0)
    constexpr int SLOTS = (NBLK + NK - 1) / NK;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fr = lane & 15, fk = lane >> 4;
    const int nb = (n + DB - 1) / DB;

    // element (r, c) of A; past n the identity, so that a ragged block
    // factors like a whole one
    auto elem = [&](int r, int c) -> T {
        const T a = A[(int64_t)min(c, n - 1) * ld + min(r, n - 1)];
        return r < n && c < n ? a : (r == c ? T(1) : T(0));
    };
    auto store = [&](int i, int j, const V4 &b) {           // block (i, j), below the diagonal
        const int r = DB * i + fr;
        if (r < n) {
#pragma unroll
            for (int q = 0; q < 4; q++) A[(int64_t)(DB * j + MF<T>::row(q, fk)) * ld + r] = b[q];
        }
    };
    auto put = [&](T *img, const V4 &b) {
#pragma unroll
        for (int q = 0; q < 4; q++) img[64 * q + lane] = b[q];
    };
    auto get = [&](const T *img) -> V4 {
        V4 b;
#pragma unroll
        for (int q = 0; q < 4; q++) b[q] = img[64 * q + lane];
        return b;
    };
    auto get_w = [&](int p) -> V4 {
        const T *w = wl(p);
        V4 b;
#pragma unroll
        for (int q = 0; q < 4; q++) b[q] = w[(4 * q + fk) * DIAG_WP + fr];
        return b;
    };
    // C + M_j X_i^T, M_j = -X_j; both as operand images
    auto prod = [&](V4 c, const V4 &mj, const V4 &xi) -> V4 {
#pragma unroll
        for (int s = 0; s < 4; s++) c = MF<T>::mfma(mj[s], xi[s], c);
        return c;
    };
    auto solve = [&](const V4 &w, const V4 &c) -> V4 {       // C W^T
        V4 xx = {T(0), T(0), T(0), T(0)};
#pragma unroll
        for (int s = 0; s < 4; s++) xx = MF<T>::mfma(w[s], c[s], xx);
        return xx;
    };

    // Both roles run the same barriers: one before the loop's second half
    // (W_p, C(p+1, p) and D_{p+1} are in LDS) and one after it (X(., p) is).
    if (wave == 0) {
        __builtin_amdgcn_s_setprio(3);                      // it shares its SIMD with other waves
        T v[DB], x[DB], l[DB];
#pragma unroll
        for (int c = 0; c < DB; c++) {
            v[c] = elem(fr, c);
            if (fk == 0) ds.dl[fr][c] = v[c];
        }
        for (int p = 0; p < nb; p++) {
#pragma unroll
            for (int c = 0; c < DB; c++) x[c] = fr == c ? T(1) : T(0);
            if (__any(sweep_fast(v, x, l))) {
                int fail = 0;
#pragma unroll
                for (int c = 0; c < DB; c++) {
                    v[c] = ds.dl[fr][c];
                    x[c] = fr == c ? T(1) : T(0);
                }
                sweep_exact(v, x, fr, &fail, std::make_integer_sequence<int, DB>());
                if (fail && lane == 0) ds.fail = DB * p + fail;
#pragma unroll
                for (int c = 0; c < DB; c++) {
                    l[c] = v[c];
                    v[c] = T(NAN);                          // no pivot: l is rounded as it is
                }
            }
            // W(c, fr) = x[c] as the A operand of W C^T: slice s, lane 16 fk +
            // i holds W(i, row(s, fk)), so column fr is image column t
            if (fk == 0) {
                T *w = wl(p) + (sizeof(T) == 8 ? fr : 4 * (fr & 3) + (fr >> 2)) * DIAG_WP;
#pragma unroll
                for (int c = 0; c < DB; c++) w[c] = x[c];
            } else if (fk == 1) {
#pragma unroll
                for (int c = 0; c < DB; c++) ds.ll[p & 1][c][fr] = l[c];
            }
            __syncthreads();
            if (ds.fail) break;
            auto leave_pivots = [&]() {
                const T piv = pivot_of(v, fr);
                if (fk == 0) ds.ll[p & 1][fr][DB] = piv;
            };
            if (p + 1 == nb) {
                leave_pivots();
            } else {
                const V4 d0 = get(ds.hd);
                const V4 xx = solve(get_w(p), get(ds.hc));
                leave_pivots();                             // beside the products
                put(xl(p + 1, p), -xx);
                const V4 d = prod(d0, -xx, xx);
#pragma unroll
                for (int q = 0; q < 4; q++) ds.dl[fr][MF<T>::row(q, fk)] = d[q];
            }
            __syncthreads();
            if (p + 1 < nb) {
#pragma unroll
                for (int c = 0; c < DB; c++) v[c] = ds.dl[fr][c];
            }
        }
        __builtin_amdgcn_s_setprio(0);
    } else {
        // slot u: block t = wave + NK u of the list (0,0) (1,0) .. (NBK-1,0)
        // (1,1) (2,1) .. ; bi, bj are wave-uniform, bj = -1 where there is none
        const int worker = !APART || wave < 4 ? wave : wave == 4 ? NBK * NBK : wave - 1;
        V4 blk[SLOTS];
        int bi[SLOTS], bj[SLOTS];
#pragma unroll
        for (int u = 0; u < SLOTS; u++) {
            int t = worker + NK * u, j = 0;
            while (j < NBK && t >= NBK - j) { t -= NBK - j; j++; }
            bj[u] = j < NBK && j + t < nb ? j : -1;
            bi[u] = j + t;
            if (bj[u] >= 0) {
#pragma unroll
                for (int q = 0; q < 4; q++) blk[u][q] = elem(DB * bi[u] + fr, DB * j + MF<T>::row(q, fk));
            }
        }
#pragma unroll
        for (int u = 0; u < SLOTS; u++)
            if (bj[u] >= 0 && bi[u] == 1) put(bj[u] == 0 ? ds.hc : ds.hd, blk[u]);
        for (int p = 0; p < nb; p++) {
            if (p > 0) {
                // step p - 1 on the blocks of columns >= p (wave 0 did (p, p));
                // the two blocks that wave 0 needs next go to LDS
#pragma unroll
                for (int u = 0; u < SLOTS; u++)
                    if (bj[u] >= p && bi[u] > p) {
                        blk[u] = prod(blk[u], get(xl(bj[u], p - 1)), -get(xl(bi[u], p - 1)));
                        if (bi[u] == p + 1) put(bj[u] == p ? ds.hc : ds.hd, blk[u]);
                    }
            }
            __syncthreads();
            if (ds.fail) break;
            const V4 w = get_w(p);
#pragma unroll
            for (int u = 0; u < SLOTS; u++)
                if (bj[u] == p && bi[u] > p + 1) {
                    blk[u] = solve(w, blk[u]);
                    put(xl(bi[u], p), -blk[u]);
                }
            __syncthreads();
#pragma unroll
            for (int u = 0; u < SLOTS; u++)
                if (bj[u] == p && bi[u] > p + 1) store(bi[u], p, blk[u]);
            // what wave 0 left: L_pp and X(p + 1, p)
            if (wave == (APART ? 4 : NK)) {
                if (p + 1 < nb) store(p + 1, p, -get(xl(p + 1, p)));
                const T root = root_of(ds.ll[p & 1][fr][fr], ds.ll[p & 1][fr][DB]);
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const int c = 4 * u + fk;
                    const T a = ds.ll[p & 1][c][fr];
                    if (c <= fr && DB * p + fr < n) A[(int64_t)(DB * p + c) * ld + DB * p + fr] = c == fr ? root : a;
                }
            }
        }
    }
    return __builtin_amdgcn_readfirstlane(ds.fail);
}

// The diagonal block of a sub-column: n <= 128, one workgroup of eight waves.
// op: the operand images for k_panel_solve (see OPB); info = info_base + j of
// the first non-positive pivot j (1-based), as CORE_dpotrf reports it.
//
// As diag_factor, but laid out for the shortest chain, since nothing else of
// a panel runs beside it.  The four rows of 16 lanes of a sweep hold the same
// D and different blocks in x: what becomes W = L^{-1} for the identity
// becomes X = C L^{-T} for the rows of a block C below.  Waves 0 and 1 sweep
// D_p together with the identity and all blocks C(i, p):
//   wave 0   I, C(p+1, p) .. C(p+3, p), then D_{p+1} -= X X^T,
//   wave 1   C(p+4, p) .. C(p+7, p).
// Nothing is solved through W, and one exchange through LDS hands X(., p) to
//   waves 2, 3, 6, 7 (the other two SIMDs): C(i, p+1) -= X(i, p) X(p+1, p)^T
//            for the next sweep, then, while it runs, the rest of the blocks,
//            which they hold in registers;
//   waves 4, 5 (beside the sweeping waves, without products): the stores.
// An MFMA on a sweeping wave's SIMD would hold it up: FP64 products and FP64
// FMAs share their units.
// A block's rows travel as rows of 16 elements, XP apart.
//
// n = 128, FP64, cycles a 16-column step (clock reads included): sweep 2450,
// X out and barrier 440, D_{p+1} beside C(., p+1) 1000 - 1600, rows read back
// 440.  With the solve through W on wave 0's chain and products on its SIMD:
// 3100 - 3900 + 750 + 1500 + 400.  In a factorization 20.5 -> 17.7 us
// (N = 4096, NB = 256), 14.0 -> 12.2 us for 93 columns; FP32 14.2 -> 13.1 us
// (N = 3200, NB = 320); 0.2 - 0.6 us of it are the rounded roots of the pivots.
template <class T>
__global__ __launch_bounds__(512, sizeof(T) == 8 ? 2 : 4) void k_diag_factor(T *__restrict__ A, int n, int ld, int info_base,
                                                       int *__restrict__ d_info, T *__restrict__ op)
{
    typedef typename MF<T>::v4 V4;
    constexpr int XP = DIAG_WP, XS = DB * XP;
    // FP32: 31 KB, what two workgroups of the trailing update leave of a CU
    __shared__ __align__(16) T xr[2][DBN][XS];             // by p & 1: X(i, p), W_p (by columns) for i = 0
    __shared__ __align__(16) T cr[DBN][XS];                // C(i, p + 1) for the sweep
    __shared__ __align__(16) T ll1[XS];                    // L_pp of odd p (even p: cr[0]); behind each row its pivot
    __shared__ __align__(16) T dl[XS];                     // D_{p+1}
    __shared__ T hd[OPI];                                  // D_{p+1} before step p, [s][lane]
    __shared__ int fail;
    __builtin_amdgcn_s_setprio(2);
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fr = lane & 15, fk = lane >> 4;
    const int nb = (n + DB - 1) / DB;
    if (threadIdx.x == 0) fail = 0;

    // element (r, c) of A; past n the identity, so that a ragged block
    // factors like a whole one
    auto elem = [&](int r, int c) -> T {
        const T a = A[(int64_t)min(c, n - 1) * ld + min(r, n - 1)];
        return r < n && c < n ? a : (r == c ? T(1) : T(0));
    };
    auto row_out = [&](T *img, const T *v) {               // row fr of a block
#pragma unroll
        for (int c = 0; c < DB; c++) img[fr * XP + c] = v[c];
    };
    auto row_in = [&](const T *img, T *v) {
#pragma unroll
        for (int c = 0; c < DB; c++) v[c] = img[fr * XP + c];
    };
    // operand / accumulator registers of a block kept by rows
    auto get = [&](const T *img) -> V4 {
        V4 b;
#pragma unroll
        for (int q = 0; q < 4; q++) b[q] = img[fr * XP + MF<T>::row(q, fk)];
        return b;
    };
    auto put = [&](T *img, const V4 &b) {
#pragma unroll
        for (int q = 0; q < 4; q++) img[fr * XP + MF<T>::row(q, fk)] = b[q];
    };
    auto prod = [&](V4 c, const V4 &xj, const V4 &xi) -> V4 {    // C - X_i X_j^T
#pragma unroll
        for (int s = 0; s < 4; s++) c = MF<T>::mfma(-xj[s], xi[s], c);
        return c;
    };

    // every role runs the same two barriers a step
    if (wave < 2) {
        __builtin_amdgcn_s_setprio(3);
        T v[DB], x[DB], l[DB];
        const int g = 4 * wave + fk;                       // block p + g of the step; 0: the identity
        auto unit = [&]() {
#pragma unroll
            for (int c = 0; c < DB; c++) x[c] = fr == c ? T(1) : T(0);
        };
#pragma unroll
        for (int c = 0; c < DB; c++) v[c] = elem(fr, c);
        if (fk == 0) row_out(dl, v);                       // by both waves, the same values
        if (g == 0) {
            unit();
        } else if (g < nb) {
#pragma unroll
            for (int c = 0; c < DB; c++) x[c] = elem(DB * g + fr, c);
            row_out(cr[g], x);
        } else {
            unit();
        }
        for (int p = 0; p < nb; p++) {
            const bool mine = p + g < nb;
            if (__any(sweep_fast(v, x, l))) {
                int f = 0;
                row_in(dl, v);
                if (g > 0 && mine) row_in(cr[p + g], x);
                else unit();
                sweep_exact(v, x, fr, &f, std::make_integer_sequence<int, DB>());
                if (f && tid == 0) fail = DB * p + f;
#pragma unroll
                for (int c = 0; c < DB; c++) {
                    l[c] = v[c];
                    v[c] = T(NAN);                          // no pivot: l is rounded as it is
                }
            }
            if (mine) row_out(xr[p & 1][g == 0 ? 0 : p + g], x);
            __syncthreads();
            if (fail) break;
            if (wave == 1) {
                T *ll = p & 1 ? ll1 : cr[0];
                const T piv = pivot_of(v, fr);
                if (fk == 0) {
                    row_out(ll, l);
                    ll[fr * XP + DB] = piv;
                }
            } else if (p + 1 < nb) {
                V4 d0;
#pragma unroll
                for (int q = 0; q < 4; q++) d0[q] = hd[64 * q + lane];
                const V4 xx = get(xr[p & 1][p + 1]);
                put(dl, prod(d0, xx, xx));
            }
            __syncthreads();
            if (p + 1 < nb) {
                row_in(dl, v);
                if (g > 0 && p + 1 + g < nb) row_in(cr[p + 1 + g], x);
                else unit();
            }
        }
    } else if ((wave & 3) >= 2) {
        // slot u: block t = worker + 4 u of the list (1,1) (2,1) .. (7,1) (2,2)
        // (3,2) .. ; bi, bj are wave-uniform, bj = -1 where there is none
        constexpr int NK = 4, SLOTS = (DBN * (DBN - 1) / 2 + NK - 1) / NK;
        const int worker = (wave & 1) + 2 * (wave >> 2);
        int at[4];
#pragma unroll
        for (int q = 0; q < 4; q++) at[q] = MF<T>::row(q, fk) * ld + fr;
        V4 blk[SLOTS];
        int bi[SLOTS], bj[SLOTS];
#pragma unroll
        for (int u = 0; u < SLOTS; u++) {
            int t = worker + NK * u, j = 1;
            while (j < DBN && t >= DBN - j) { t -= DBN - j; j++; }
            bj[u] = j < DBN && j + t < nb ? j : -1;
            bi[u] = j + t;
            if (bj[u] >= 0) {
                const T *b = A + (int64_t)DB * j * ld + DB * bi[u];
                if (DB * bi[u] + DB <= n) {
#pragma unroll
                    for (int q = 0; q < 4; q++) blk[u][q] = b[at[q]];
                } else {
#pragma unroll
                    for (int q = 0; q < 4; q++) blk[u][q] = elem(DB * bi[u] + fr, DB * j + MF<T>::row(q, fk));
                }
            }
        }
        auto put_d = [&](const V4 &b) {
#pragma unroll
            for (int q = 0; q < 4; q++) hd[64 * q + lane] = b[q];
        };
        if (bj[0] == 1 && bi[0] == 1) put_d(blk[0]);
        for (int p = 0; p < nb; p++) {
            const T (*xp)[XS] = xr[p & 1];
            __syncthreads();
            if (fail) break;
#pragma unroll
            for (int u = 0; u < SLOTS; u++)
                if (bj[u] == p + 1 && bi[u] > p + 1) put(cr[bi[u]], prod(blk[u], get(xp[p + 1]), get(xp[bi[u]])));
            __syncthreads();
#pragma unroll
            for (int u = 0; u < SLOTS; u++)
                if (bj[u] > p + 1) {
                    blk[u] = prod(blk[u], get(xp[bj[u]]), get(xp[bi[u]]));
                    if (bj[u] == p + 2 && bi[u] == p + 2) put_d(blk[u]);
                }
        }
    } else {
        for (int p = 0; p < nb; p++) {
            __syncthreads();
            if (fail) break;
            __syncthreads();
            for (int i = p + 1 + (wave & 1); i < nb; i += 2) {
                const V4 b = get(xr[p & 1][i]);
                const int r = DB * i + fr;
                if (r < n) {
#pragma unroll
                    for (int q = 0; q < 4; q++) A[(int64_t)(DB * p + MF<T>::row(q, fk)) * ld + r] = b[q];
                }
                *(V4 *)(op + (int64_t)p * OPB + (i - p) * OPI + 4 * lane) = -b;
            }
            if (wave == 4) {
                V4 w;
#pragma unroll
                for (int q = 0; q < 4; q++) w[q] = xr[p & 1][0][MF<T>::row(q, fk) * XP + fr];
                *(V4 *)(op + (int64_t)p * OPB + 4 * lane) = w;
            } else {
                const T *row = (p & 1 ? ll1 : cr[0]) + fr * XP, root = root_of(row[fr], row[DB]);
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const int c = 4 * u + fk;
                    if (c <= fr && DB * p + fr < n)
                        A[(int64_t)(DB * p + c) * ld + DB * p + fr] = c == fr ? root : row[c];
                }
            }
        }
    }
    if (tid == 0 && fail) atomicCAS(d_info, 0, info_base + fail);
}

// ---------------------------------------------------------------------------
// X = C L^{-T} for the rows below the diagonal block of a sub-column: columns
// c0 .. c0 + w - 1 of tile column k, rows c0 + w.. of tile (k, k) (the first
// g0 workgroups) and all rows of the tiles m0, m0 + 1, ... (gt workgroups a
// tile).  A wave takes 16 rows with all w columns in registers (nbw =
// ceil(w / 16) blocks): per 16-column block one product with W_b, then the
// update of the later blocks; nothing passes between waves.  The operand
// images of block column b + 1 and block b + AHEAD of C are in flight while
// block column b is multiplied; the four waves of a workgroup read the same
// images at about the same time.  144 MFMAs a wave at w = 128; blocks past nbw
// multiply what the unused images hold and are dropped.
//
// The products for a block add up from zero and meet C once.  With C as their
// start every four columns round at the size of C: entries below the diagonal
// tiles of a factor of N = 378, NB = 93 with a dominant diagonal are then off
// by 2.7 eps (FP64; FP32 2.8) instead of 1.8 (1.9), for 1.3% less time at N =
// 4096, NB = 256 in FP64 and 0.3% in FP32.
//
// Bound by the latency of the first loads and of eight dependent products
// (FP64, 13 us at 1000 rows; its 144 MFMAs of 64 cycles are 3.8 us).
// Staging the images in LDS instead took 16-18 us a launch.
template <class T>
__global__ __launch_bounds__(256, 2) void k_panel_solve(T *__restrict__ Tt, int N, int NB, int MT, int k, int c0,
                                                       int w, const T *__restrict__ op, int g0, int gt, int m0)
{
    typedef typename MF<T>::v4 V4;
    __builtin_amdgcn_s_setprio(2);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int fr = lane & 15, fk = lane >> 4;
    const int g = blockIdx.x;
    const int m = g < g0 ? k : m0 + (g - g0) / gt;
    const int r0 = (g < g0 ? c0 + w + 64 * g : 64 * ((g - g0) % gt)) + 16 * wave;
    const int rows = tile_rows(N, NB, MT, m);
    if (r0 >= rows) return;
    T *C = Tt + tile_index(MT, m, k) * (int64_t)NB * NB + (int64_t)c0 * NB;
    const int nbw = (w + DB - 1) / DB;

    V4 img[2][DBN];
    auto load = [&](V4 *im, int b) {
        const V4 *src = (const V4 *)(op + (int64_t)b * OPB) + lane;
#pragma unroll
        for (int i = 0; i < DBN; i++)
            if (b + i < DBN) im[i] = src[64 * i];
    };
    load(img[0], 0);
    const int r = r0 + fr, rc = min(r, rows - 1);
    constexpr int AHEAD = DBN / 2;                          // blocks of C
    V4 acc[DBN], cv[DBN];                                   // products of the blocks solved so far, C
    auto load_c = [&](int b) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int c = DB * b + MF<T>::row(q, fk);
            cv[b][q] = C[(int64_t)min(c, w - 1) * NB + rc];
        }
    };
#pragma unroll
    for (int b = 0; b < AHEAD; b++) load_c(b);
#pragma unroll
    for (int b = 0; b < DBN; b++) acc[b] = V4{T(0), T(0), T(0), T(0)};
#pragma unroll
    for (int b = 0; b < DBN; b++) {
        if (b < nbw) {
            __builtin_amdgcn_sched_barrier(0);              // no image further ahead than this
            if (b + 1 < nbw) load(img[(b + 1) & 1], b + 1);
            if (b + AHEAD < DBN) load_c(b + AHEAD);
            const V4 *im = img[b & 1];
            V4 cc;
#pragma unroll
            for (int q = 0; q < 4; q++) cc[q] = (DB * b + MF<T>::row(q, fk) < w ? cv[b][q] : T(0)) + acc[b][q];
            V4 xx = {T(0), T(0), T(0), T(0)};
#pragma unroll
            for (int s = 0; s < 4; s++) xx = MF<T>::mfma(im[0][s], cc[s], xx);
#pragma unroll
            for (int s = 0; s < 4; s++)
#pragma unroll
                for (int b2 = b + 1; b2 < DBN; b2++)
                    acc[b2] = MF<T>::mfma(im[b2 - b][s], xx[s], acc[b2]);
            if (r < rows) {
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int c = DB * b + MF<T>::row(q, fk);
                    if (c < w) C[(int64_t)c * NB + r] = xx[q];
                }
            }
        }
    }
}

}  // namespace mi
