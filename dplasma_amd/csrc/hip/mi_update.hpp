// mi_update.hpp -- one block of a tile update C -= A B^T on the 16x16x4 MFMA,
// its operands streamed straight into LDS.
#pragma once
#include <type_traits>
#include <utility>
#include "mi_common.hpp"

namespace mi {

typedef __attribute__((address_space(3))) void *lds_void;

// Every load of this wave but the last n and every LDS read done, then the
// workgroup's barrier.
template <int N> __device__ __forceinline__ void wait_barrier()
{
    __builtin_amdgcn_sched_barrier(0);             // no product of the stage before moves past this
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
    __builtin_amdgcn_sched_barrier(0);
}

template <class S, int... I, class F>
__device__ __forceinline__ void update_tail(std::integer_sequence<int, I...>, F &&f)
{
    (f(std::integral_constant<int, I>()), ...);
}

// Shape of a block: BM x BM of C by WR x WC waves, K in stages of BK columns,
// ST stages of LDS (one being read, the others in flight).  V consecutive
// rows of an operand column form one LDS read: the MFMA tiles 0 .. V-1 of a
// group interleave their rows (row i of tile t is row V i + t of the group),
// so a lane holds V consecutive rows of C.  CPS such vectors of C come in a
// stage at the start.
template <class T, int BM_, int WR_, int WC_, int BK_, int ST_, int V_, int CPS_> struct UpdShape {
    static constexpr int BM = BM_, WR = WR_, WC = WC_, BK = BK_, ST = ST_, V = V_, CPS = CPS_;
    static constexpr int NW = WR * WC, NT = 64 * NW;
    static constexpr int HR = BM / WR, HC = BM / WC;          // rows / columns of a wave
    static constexpr int TR = HR / 16, TC = HC / 16;          // MFMA tiles of a wave
    static constexpr int RB = BM * (int)sizeof(T);            // bytes of an operand column in LDS
    static constexpr int OPBYTES = BK * RB;                   // an operand's stage
    static constexpr int NI = 2 * OPBYTES / 1024 / NW;        // 1 KB loads of a wave and stage
    static constexpr int LDS = 2 * OPBYTES * ST;
    static constexpr int CPI = 1024 / RB;                     // operand columns per load
    static constexpr int NC = TR / V * TC * 4 / CPS;          // stages that take in CPS vectors of C
    // 8-byte reads: a quarter wave covers half the banks, so odd columns are
    // stored with their 128-byte halves swapped
    static constexpr bool SWZ = V * sizeof(T) == 8;
    static_assert(TR % V == 0 && TC % V == 0 && NI * NW * 1024 == 2 * OPBYTES && RB <= 1024, "block shape");
};

// C(r_base.., c_base..) -= A(r_base.., 0:K) B(c_base.., 0:K)^T, column-major
// with leading dimension NB (update_lds_ok: columns 16-byte aligned, K a
// multiple of BK and at least NC BK); rows_m / cols_n bound the valid rows and columns of C; the
// rows past them that a block still reads are those of the last NB - V.., and
// only reach parts of C that are not stored.  diag: only row >= column.
template <class S, class T>
__device__ __forceinline__ void update_block_lds(unsigned char *lds, const T *Ap, const T *Bp, T *Cp, int NB, int K,
                                                 int rows_m, int cols_n, int r_base, int c_base, bool diag)
{
    typedef typename MF<T>::v4 V4;
    typedef T vec __attribute__((ext_vector_type(S::V)));
    constexpr int V = S::V, ST = S::ST;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / S::WC, wn = wave % S::WC;
    const int fr = lane & 15, fk = lane >> 4;

    // load i of this wave: LDS piece wave + NW i of the stage (A's pieces,
    // then B's); a piece holds CPI consecutive operand columns
    constexpr int LPR = S::RB / 16;                           // lanes a column
    const int lcol = lane / LPR, lrow = (lane % LPR) * (16 / (int)sizeof(T));
    const T *src[S::NI];
#pragma unroll
    for (int i = 0; i < S::NI; i++) {
        const int piece = wave + S::NW * i;
        const bool isb = piece * 1024 >= S::OPBYTES;
        const int col = (piece - (isb ? S::OPBYTES / 1024 : 0)) * S::CPI + lcol;
        const int row = S::SWZ ? lrow ^ ((col & 1) * (128 / (int)sizeof(T))) : lrow;
        const int g = min((isb ? c_base : r_base) + row, NB - 16 / (int)sizeof(T));
        src[i] = (isb ? Bp : Ap) + (int64_t)col * NB + g;
    }
    auto issue = [&](int slot) {
#pragma unroll
        for (int i = 0; i < S::NI; i++) {
            __builtin_amdgcn_global_load_lds(src[i], (lds_void)(lds + slot * 2 * S::OPBYTES + (wave + S::NW * i) * 1024),
                                             16, 0, 0);
            src[i] += (int64_t)S::BK * NB;
        }
    };

    const int nst = K / S::BK;
#pragma unroll
    for (int s = 0; s < ST - 1; s++)
        if (s < nst) issue(s);

    V4 acc[S::TR][S::TC];                                     // A B^T - C
#pragma unroll
    for (int i = 0; i < S::TR; i++)
#pragma unroll
        for (int j = 0; j < S::TC; j++) acc[i][j] = V4{T(0), T(0), T(0), T(0)};
    const int row0 = r_base + wm * S::HR + V * fr, col0 = c_base + wn * S::HC;
    const bool whole = r_base + S::BM <= rows_m && c_base + S::BM <= cols_n && !diag;
    // C vector t of a lane: rows row0 + 16 V p .. + V - 1 of one column; a
    // lane's base plus an offset that is the same for all lanes
    T *cbase = Cp + (int64_t)(col0 + V * MF<T>::row(0, fk)) * NB + row0;
    auto cvec = [&](int t) -> vec * {
        const int p = t / (4 * S::TC), j = t / 4 % S::TC, q = t % 4;
        return (vec *)(cbase + (int64_t)(16 * V * (j / V) + V * MF<T>::row(q, 0) + j % V) * NB + 16 * V * p);
    };
    auto sub = [&](int t, const vec &c) {
        const int p = t / (4 * S::TC), j = t / 4 % S::TC, q = t % 4;
#pragma unroll
        for (int e = 0; e < V; e++) acc[V * p + e][j][q] -= c[e];
    };

    auto compute = [&](int slot) {
        const unsigned char *a0 = lds + slot * 2 * S::OPBYTES, *b0 = a0 + S::OPBYTES;
#pragma unroll
        for (int kq = 0; kq < S::BK / 4; kq++) {
            const int k = 4 * kq + fk;
            const int sw = S::SWZ ? (fk & 1) * 128 : 0;
            T a[S::TR], b[S::TC];
#pragma unroll
            for (int p = 0; p < S::TR / V; p++) {
                const vec x = *(const vec *)(a0 + k * S::RB + (((wm * S::HR + 16 * V * p + V * fr) * (int)sizeof(T)) ^ sw));
#pragma unroll
                for (int t = 0; t < V; t++) a[V * p + t] = x[t];
            }
#pragma unroll
            for (int p = 0; p < S::TC / V; p++) {
                const vec x = *(const vec *)(b0 + k * S::RB + (((wn * S::HC + 16 * V * p + V * fr) * (int)sizeof(T)) ^ sw));
#pragma unroll
                for (int t = 0; t < V; t++) b[V * p + t] = x[t];
            }
#pragma unroll
            for (int i = 0; i < S::TR; i++)
#pragma unroll
                for (int j = 0; j < S::TC; j++) acc[i][j] = MF<T>::mfma(b[j], a[i], acc[i][j]);
        }
    };
    // C of a whole block comes in CPS vectors a stage over the first NC stages,
    // so that its traffic spreads over the products instead of standing before
    // them.  (Over the last stages it is as fast, but then the products add up
    // from zero: the matrix cores' rounding has a small bias, and where C and
    // the sum nearly cancel everywhere, as for strongly correlated covariances,
    // every element of the residual A - L L^T gets the same sign.  FP32
    // likelihood gradient at N = 8192: error 1.1e-3 with C last, 3.5e-4 so; FP64
    // 1.9e-12 and 0.9e-12.)
    const bool early = whole && nst >= S::NC;
    int slot = 0, first = 0;
    auto next = [&](int s) {
        if (s + ST - 1 < nst) issue(slot == 0 ? ST - 1 : slot - 1);
    };
    if (early) {
        vec c[2][S::CPS];
        update_tail<S>(std::make_integer_sequence<int, S::NC>(), [&](auto tt) {
            constexpr int t = decltype(tt)::value, left = S::NC - 1 - t;
            // younger than stage t: at least the later stages' loads and the C
            // loads of the ST - 2 stages before this one
            wait_barrier<S::NI * (left < ST - 2 ? left : ST - 2) + S::CPS * (t < ST - 2 ? t : ST - 2)>();
            next(t);
#pragma unroll
            for (int e = 0; e < S::CPS; e++) c[t & 1][e] = *cvec(S::CPS * t + e);
            compute(slot);
            slot = slot == ST - 1 ? 0 : slot + 1;
            if constexpr (t > 0) {
#pragma unroll
                for (int e = 0; e < S::CPS; e++) sub(S::CPS * (t - 1) + e, c[(t - 1) & 1][e]);
            }
        });
#pragma unroll
        for (int e = 0; e < S::CPS; e++) sub(S::CPS * (S::NC - 1) + e, c[(S::NC - 1) & 1][e]);
        first = S::NC;
    }
    for (int s = first; s < nst; s++) {
        // stage s landed, and every wave is done with stage s - 1
        if (s + ST - 2 < nst) wait_barrier<S::NI * (ST - 2)>();
        else wait_barrier<0>();
        next(s);
        compute(slot);
        slot = slot == ST - 1 ? 0 : slot + 1;
    }

    if (early) {
#pragma unroll
        for (int t = 0; t < S::NC * S::CPS; t++) {
            const int p = t / (4 * S::TC), j = t / 4 % S::TC, q = t % 4;
            vec v;
#pragma unroll
            for (int e = 0; e < V; e++) v[e] = -acc[V * p + e][j][q];
            *cvec(t) = v;
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < S::TR; i++)
#pragma unroll
        for (int j = 0; j < S::TC; j++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int row = row0 + 16 * V * (i / V) + i % V;
                const int col = col0 + 16 * V * (j / V) + V * MF<T>::row(q, fk) + j % V;
                if (row < rows_m && col < cols_n && (!diag || row >= col)) Cp[(int64_t)col * NB + row] -= acc[i][j][q];
            }
}

// Whether update_block_lds can run on tiles at `base` with leading dimension
// NB and K columns: whole 16-byte pieces of every column, whole stages, and
// enough of them to take C in.
template <class S, class T> inline bool update_lds_ok(const T *base, int NB, int K)
{
    return ((uintptr_t)base & 15) == 0 && (NB * sizeof(T)) % 16 == 0 && K % S::BK == 0 && K >= S::NC * S::BK;
}

}  // namespace mi
